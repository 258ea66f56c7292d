// The allocation-free batch entry over the stand-in runtime of engine_host.cpp
// (compiled with its main renamed): no allocation on the host either.  Prints
// one line per failed expectation; exit status 0 without any.
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>
#include "jms_hip.h"

static long allocs = 0;
void* operator new(std::size_t n) {
  ++allocs;
  if (void* p = malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, std::size_t) noexcept { free(p); }

static int bad = 0;
#define EXPECT(c) do { if (!(c)) { ++bad; printf("line %d: %s\n", __LINE__, #c); } } while (0)

int main() {
  const int n = 16, S = 3, one = 1, zero = 0, obj[S] = {0, 0, 0}, det[S + 1] = {-1, 0, -1, 1};
  std::vector<float> a(2 * n * n, 1.f), waves(2 * n * n * 2), res(2 * 2);
  const std::vector<int> var(2 * S, 0);
  const float ppar[8] = {}, weight = 1.f;
  jms_hip_engine* e = nullptr;
  EXPECT(jms_hip_create(&e) == 0);
  EXPECT(jms_hip_set_grid(e, n, n, 1.f, 1.f, 0.0025f) == 0);
  EXPECT(jms_hip_setup_gratings(e, n, n, 1, &one) == 0);
  EXPECT(jms_hip_upload_gratings(e, 0, 1, a.data()) == 0);
  EXPECT(jms_hip_setup_propagators(e, 1, 1, &zero) == 0);
  EXPECT(jms_hip_upload_propagator(e, 0, a.data()) == 0);
  EXPECT(jms_hip_setup_objects(e, S, obj) == 0);
  EXPECT(jms_hip_setup_detection(e, 2, det, 1, JMS_HIP_DETECT_INTEGRATED) == 0);
  EXPECT(jms_hip_upload_detector(e, 0, a.data(), 0, nullptr) == 0);
  EXPECT(jms_hip_set_probe(e, a.data()) == 0);
  for (int islc0 = 0; islc0 <= S; ++islc0) {
    allocs = 0;
    EXPECT(jms_hip_run_batch_noalloc(e, islc0, 2, waves.data(), ppar, var.data(), 2, 1, &weight, res.data()) == 0);
    if (allocs) printf("%ld host allocations from plane %d on\n", allocs, islc0);
    EXPECT(allocs == 0);
  }
  jms_hip_destroy(e);
  return bad ? 1 : 0;
}
