// Set-up calls over the stand-in runtime of engine_host.cpp (compiled with its
// main, its hipMemcpy and its slice-loop launcher renamed): the copies that a
// set-up makes besides its data, and the tables that the one-launch slice loop
// gets after each order of set-up calls.  Prints one line per failed
// expectation; exit status 0 without any.
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstring>
#include <vector>
#include "jms_hip.h"
#include "jms_kernels.h"

static int bad = 0;
#define EXPECT(c) do { if (!(c)) { ++bad; printf("line %d: %s\n", __LINE__, #c); } } while (0)

static int copies = 0, loops = 0;
static std::vector<jms::GrpPlane> table;

extern "C" hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  ++copies;
  memmove(d, s, n);
  return hipSuccess;
}
namespace jms {
bool loop_ok(int, int, int) { return true; }
hipError_t launch_loop(int, int, int, const LoopArgs& a, bool, hipStream_t) {
  ++loops;
  table.assign(a.pl, a.pl + a.nslc + 1);
  return hipSuccess;
}
}  // namespace jms

int main() {
  const int n = 16;
  std::vector<float> a(2 * n * n * 4, 1.f);
  const std::vector<int> var(8, 0);
  jms_hip_engine* e = nullptr;
  EXPECT(jms_hip_create(&e) == 0);
  std::vector<int> obj, det;
  int npro = 0;
  auto gratings = [&](const std::vector<int>& nvar) {
    EXPECT(jms_hip_setup_gratings(e, n, n, (int)nvar.size(), nvar.data()) == 0);
    for (int i = 0; i < (int)nvar.size(); ++i) EXPECT(jms_hip_upload_gratings(e, i, nvar[i], a.data()) == 0);
  };
  auto propagators = [&](const std::vector<int>& idx) {
    npro = 2;
    EXPECT(jms_hip_setup_propagators(e, npro, (int)idx.size(), idx.data()) == 0);
    for (int i = 0; i < npro; ++i) EXPECT(jms_hip_upload_propagator(e, i, a.data()) == 0);
  };
  auto objects = [&](const std::vector<int>& o) {
    obj = o;
    EXPECT(jms_hip_setup_objects(e, (int)o.size(), o.data()) == 0);
  };
  auto detection = [&](const std::vector<int>& d, int ndet) {
    det = d;
    EXPECT(jms_hip_setup_detection(e, 2, d.data(), ndet, JMS_HIP_DETECT_INTEGRATED) == 0);
    for (int i = 0; i < ndet; ++i) EXPECT(jms_hip_upload_detector(e, i, a.data(), 0, nullptr) == 0);
  };
  // the table of a run: offsets of the gratings, which propagator, the sums
  auto run = [&](const std::vector<int>& nvar, const std::vector<int>& idx, int ndet, bool staged = false) {
    const float zero = 0.f, one = 1.f;
    loops = 0;
    if (staged) {
      EXPECT(jms_hip_stage_scan(e, 1, &zero, &zero, nullptr, 1, &one, var.data()) == 0);
      EXPECT(jms_hip_run_staged(e, 0, 1, 0) == 0);
    } else {
      EXPECT(jms_hip_wave_set(e, a.data()) == 0);
      EXPECT(jms_hip_multislice(e, 0, var.data(), 1.f, 0) == 0);
    }
    EXPECT(loops == 1 && table.size() == obj.size() + 1);
    std::vector<long long> off(1, 0);
    for (int v : nvar) off.push_back(off.back() + (long long)v * n * n);
    const char* p0 = nullptr;  // propagator 0
    for (size_t p = 0; p < obj.size(); ++p) {
      const int js = obj[p] % (int)nvar.size();
      EXPECT(table[p].slc_off == off[js]);
      const char* q = (const char*)table[p].pro_t - (size_t)idx[js] * n * n * 8;
      EXPECT(!p0 || q == p0);
      p0 = q;
    }
    for (size_t p = 0; p <= obj.size(); ++p) EXPECT(table[p].part_off == (det[p] < 0 ? -1 : (long long)det[p] * ndet));
  };
  auto all = [&](const std::vector<int>& nvar, const std::vector<int>& idx, const std::vector<int>& o,
                 const std::vector<int>& d, int ndet) {
    EXPECT(jms_hip_set_grid(e, n, n, 1.f, 1.f, 0.0025f) == 0);
    gratings(nvar), propagators(idx), objects(o), detection(d, ndet);
    EXPECT(jms_hip_set_probe(e, a.data()) == 0);
  };
  // twiddles, gratings, both copies of each propagator and detector, the probe
  auto data = [&](int nslc, int ndet) { return 2 + nslc + 2 * npro + 2 * ndet + 1; };
  all({2, 1}, {0, 1}, {0, 1, 0}, {-1, 0, -1, 1}, 3);
  run({2, 1}, {0, 1}, 3);
  copies = 0;
  all({2, 1}, {0, 1}, {0, 1, 0}, {-1, 0, -1, 1}, 3);  // the same again: its data and nothing else
  if (copies != data(2, 3)) printf("%d copies for %d\n", copies, data(2, 3));
  EXPECT(copies == data(2, 3));
  run({2, 1}, {0, 1}, 3);
  copies = 0;
  all({1, 3}, {1, 0}, {1, 0, 1, 0}, {0, -1, -1, -1, 1}, 1);  // another: the tables once
  if (copies > data(2, 1) + 2) printf("%d copies for %d\n", copies, data(2, 1) + 2);
  EXPECT(copies <= data(2, 1) + 2);
  run({1, 3}, {1, 0}, 1);
  // parts of the set-up, the rest as it was
  gratings({3, 1});
  run({3, 1}, {1, 0}, 1);
  propagators({0, 1});
  run({3, 1}, {0, 1}, 1);
  objects({0, 0, 1, 1});
  run({3, 1}, {0, 1}, 1);
  detection({-1, 1, -1, -1, 0}, 2);
  run({3, 1}, {0, 1}, 2);
  for (bool staged : {false, true}) {
    gratings({1, 1}), objects({1, 1, 1, staged});
    run({1, 1}, {0, 1}, 2, staged);
  }
  jms_hip_destroy(e);
  return bad ? 1 : 0;
}
