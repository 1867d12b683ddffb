// RHS of a device-resident state without any device allocation
// (gocfd_euler2d_rhs_noalloc, include/gocfd_euler2d.h), for callers that
// cannot allocate: code under HIP graph capture, serving loops, harnesses
// that forbid hipMalloc. The tile-layout staging of the input state and of
// the RHS lives in one file-scope device array, `scratch`, of fixed size;
// each device that loads the library holds its own copy until the process
// ends, and every call on that device shares it.
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>

#include "euler2d_handle.hpp"

namespace {

// 32 MiB per device: the input state and the RHS, Kp * 4 NpInt doubles each
// (K up to about 34,900 triangles at N=4, 87,300 at N=2)
constexpr size_t kScratchBytes = size_t(32) << 20;
constexpr size_t kScratchVals = kScratchBytes / sizeof(double);

__device__ __align__(256) double scratch[kScratchVals];

// Device address of `scratch` on each device, resolved once per device with
// that device current. The array's host-side name is not a device address:
// host code uses these pointers only.
constexpr int kMaxDevices = 64;
double *g_scratch[kMaxDevices] = {};
std::mutex g_scratch_mu;

}  // namespace

namespace gocfd {
namespace capi {

void noalloc_setup(int device) {
  if (device < 0 || device >= kMaxDevices)
    throw SetupError(GOCFD_ERR_DEVICE, "device ordinal " + std::to_string(device) + " beyond the scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch[device]) return;
  int cur = -1;
  HIPCHECK(hipGetDevice(&cur));
  if (cur != device) throw SetupError(GOCFD_ERR_DEVICE, "scratch set-up needs its device current");
  void *p = nullptr;
  HIPCHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  if (!p) throw SetupError(GOCFD_ERR_DEVICE, "hipGetSymbolAddress gave no address for the scratch array");
  g_scratch[device] = static_cast<double *>(p);
}

}  // namespace capi
}  // namespace gocfd

extern "C" int gocfd_euler2d_rhs_noalloc(gocfd_euler2d *h, const double *Q, double t, double *RHS, void *stream) {
  GUARD_BEGIN
  if (!h || !Q || !RHS) return fail(GOCFD_ERR_ARG, "null argument");
  NEED_DEVICE(h);
  const size_t vals = size_t(h->L.Kp) * h->NV;
  if (2 * vals > kScratchVals)
    return fail(GOCFD_ERR_ARG, "rhs_noalloc: this mesh and order need " + std::to_string(2 * vals * sizeof(double)) +
                                   " bytes of scratch; the maximum is " + std::to_string(kScratchBytes) +
                                   " (use gocfd_euler2d_rhs)");
  HIPCHECK(hipSetDevice(h->device));
  noalloc_setup(h->device);  // done at create; a no-op here
  double *in = g_scratch[h->device], *out = in + vals;
  hipStream_t s = stream ? static_cast<hipStream_t>(stream) : h->stream;
  const int NpInt = h->d.ops.NpInt;
  dev::StageArgs a = h->rhs_args(in, t, out, s, Q);
  h->launch_one_stage(a, s);
  if (h->shock) {  // the vertex buffers this evaluation used must be clear for the next stage
    HIPCHECK(dev::launch_fill_u64(h->sigV.p, h->sigV.n, 0ull, s));
    HIPCHECK(dev::launch_fill_u64(h->epsV.p, h->epsV.n, 0ull, s));
  }
  HIPCHECK(dev::launch_scatter_state(out, h->perm.p, h->L.K, NpInt, true, RHS, s));
  if (!stream) HIPCHECK(hipStreamSynchronize(s));
  return GOCFD_OK;
  GUARD_END
}
