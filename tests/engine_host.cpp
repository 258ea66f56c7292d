// The engine's host code (csrc/jms_engine.cpp) over a HIP runtime and launchers
// made here for the CPU: device memory is host memory, and an asynchronous copy
// reads its source only when its stream is waited for, as late as a device may.
// Prints one line per failed expectation; exit status 0 without any.
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>
#include "jms_hip.h"
#include "jms_kernels.h"

static int bad = 0;
#define EXPECT(c) do { if (!(c)) { ++bad; printf("line %d: %s\n", __LINE__, #c); } } while (0)

struct Copy { void* d; const void* s; size_t n; };
static std::vector<Copy> pending;
static int col_calls = 0, col_fails_at = -1, combine_fails = 0, fft_fails = 0;
static bool freed_in_use = false;

static void drain() {
  for (auto& c : pending) memmove(c.d, c.s, c.n);
  pending.clear();
}

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { *p = calloc(1, n ? n : 1); return hipSuccess; }
hipError_t hipFree(void* p) { drain(); free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) {
  if (!pending.empty()) freed_in_use = true;
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memmove(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  pending.push_back({d, s, n});
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { drain(); return hipSuccess; }
hipError_t hipDeviceSynchronize() { drain(); return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error made by the test"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)1; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
}

namespace jms {
static const hipError_t kFail = hipErrorLaunchFailure, kOk = hipSuccess;
bool size_supported(int n) { return n == 16; }
bool grp_supported(int, int) { return false; }
bool panel_ok(int, int) { return false; }
bool lat_ok(int, int, int) { return true; }
bool loop_ok(int, int, int) { return false; }
int col_tiles(int, int nx, Tile) { return (nx + 7) / 8; }
BandHost band_of(int, int, int, int, int, int, Tile) { return BandHost(); }
BandHost loop_band(int, int, int, int, int, int) { return BandHost(); }
hipError_t scratch_address(int, float** p) { static float s[16]; *p = s; return kOk; }
hipError_t launch_loop(int, int, int, const LoopArgs&, bool, hipStream_t) { return kFail; }
hipError_t launch_fft2d(int, int, int, float2*, int, const float2*, const float2*, hipStream_t) { return kFail; }
hipError_t launch_probe(float2*, double*, const ProbeArgsHost&, hipStream_t) { return kFail; }
hipError_t launch_col_fft(int, int, int, float2*, int, const float2*, hipStream_t) { return fft_fails ? kFail : kOk; }
hipError_t launch_combine(const float*, int, int, int, int, int, const float*, float*, int, float*, hipStream_t) {
  return combine_fails ? kFail : kOk;
}
hipError_t launch_col_pass(int, int, bool, bool, const ColArgsHost&, hipStream_t) {
  return col_calls++ == col_fails_at ? kFail : kOk;
}
hipError_t launch_row_pass(int, int, int, float2*, long long, const float2*, long long, long long, const int*, int, int,
                           const float2*, const RowChanHost&, int, bool, const BandHost&, Shape, hipStream_t) {
  return kOk;
}
hipError_t launch_ff_gratings(float2*, int, int, int, const float2*, const FFAtom*, const int*, float, float, float,
                              int, float, float, int, float, float, const float2*, const float2*, hipStream_t) {
  return kFail;
}
hipError_t launch_offset_wave(float2*, const float2*, int, int, float, float, float, float, float, const float*, int,
                              int, hipStream_t) {
  return kOk;
}
hipError_t launch_col_pass_grp(int, int, int, bool, bool, bool, long long, const float2*, const GrpArgs&, bool,
                               const BandHost&, hipStream_t) {
  return kFail;
}
hipError_t launch_row_pass_grp(int, int, int, long long, long long, const float2*, const GrpArgs&, bool,
                               const BandHost&, hipStream_t) {
  return kFail;
}
hipError_t launch_zero_partial(float*, long long, long long, int, int, hipStream_t) { return kOk; }
hipError_t launch_gauss_gratings(float2*, int, int, int, double, double, double, double, double, const GaussAtom*,
                                 const int*, const int*, hipStream_t) {
  return kFail;
}
}  // namespace jms

int main() {
  const int n = 16;
  std::vector<float> a(2 * n * n, 1.f);
  jms_hip_engine* e = nullptr;
  EXPECT(jms_hip_create(&e) == 0);
  EXPECT(jms_hip_set_grid(e, n, n, 1.f, 1.f, 0.0025f) == 0);
  const int one = 1, zero = 0;
  EXPECT(jms_hip_setup_gratings(e, n, n, 1, &one) == 0);
  EXPECT(jms_hip_upload_gratings(e, 0, 1, a.data()) == 0);
  EXPECT(jms_hip_setup_propagators(e, 1, 1, &zero) == 0);
  EXPECT(jms_hip_upload_propagator(e, 0, a.data()) == 0);
  auto slices = [&](int S) {
    std::vector<int> obj(S, 0), det(S + 1, -1);
    det[S] = 0;
    EXPECT(jms_hip_setup_objects(e, S, obj.data()) == 0);
    EXPECT(jms_hip_setup_detection(e, 1, det.data(), 1, JMS_HIP_DETECT_INTEGRATED | JMS_HIP_DETECT_IMAGE) == 0);
    EXPECT(jms_hip_upload_detector(e, 0, a.data(), 0, nullptr) == 0);
  };
  slices(2);
  EXPECT(jms_hip_wave_set(e, a.data()) == 0);
  std::vector<int> var(64, 0);
  // a run that fails after its upload has waited for it when it returns: the
  // next one writes the pinned buffer anew, or frees it for a larger one
  struct { int col, combine, fft; } at[] = {{0, 0, 0}, {1, 0, 0}, {2, 0, 0}, {-1, 1, 0}, {-1, 0, 1}};
  int S = 2;
  for (auto& f : at) {
    col_calls = 0;
    col_fails_at = f.col;
    combine_fails = f.combine;
    fft_fails = f.fft;
    EXPECT(jms_hip_multislice(e, 0, var.data(), 1.f, 0) != 0);
    if (!pending.empty()) printf("copies in flight after the failure at column pass %d, combine %d, transform %d\n", f.col, f.combine, f.fft);
    EXPECT(pending.empty());
    col_fails_at = -1;
    combine_fails = fft_fails = 0;
    slices(S += 7);  // a longer variant sequence: a larger buffer
    EXPECT(jms_hip_multislice(e, 0, var.data(), 1.f, 0) == 0);
    EXPECT(!freed_in_use);
  }
  jms_hip_destroy(e);
  return bad ? 1 : 0;
}
