// Internal helpers shared by the C-ABI translation units (single solver and
// batched ensemble): error state, HIP checks, device buffers, freestream and
// initial states.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "dfr_setup.hpp"
#include "gocfd_euler2d.h"
#include "kernels.hpp"

namespace gocfd {
namespace capi {

int fail(int code, const std::string &msg);
const char *last_error();

// (an error is taken off the runtime's record: the next call's launch checks
// would report it again)
#define HIPCHECK(expr)                                                                     \
  do {                                                                                     \
    hipError_t e_ = (expr);                                                                \
    if (e_ != hipSuccess) {                                                                \
      (void)hipGetLastError();                                                             \
      throw ::gocfd::SetupError(GOCFD_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    }                                                                                      \
  } while (0)

#define GUARD_BEGIN try {
#define GUARD_END                                                                        \
  }                                                                                      \
  catch (const ::gocfd::SetupError &e) { return ::gocfd::capi::fail(e.code, e.what()); } \
  catch (const std::exception &e) { return ::gocfd::capi::fail(GOCFD_ERR_ARG, e.what()); }

template <class T>
struct DevBuf {
  T *p = nullptr;
  size_t n = 0;
  DevBuf() = default;
  DevBuf(const DevBuf &) = delete;
  DevBuf &operator=(const DevBuf &) = delete;
  void alloc(size_t count) {
    free();
    if (count == 0) count = 1;
    HIPCHECK(hipMalloc(&p, count * sizeof(T)));
    n = count;
  }
  void upload(const std::vector<T> &v) {
    alloc(v.size());
    if (!v.empty()) HIPCHECK(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  }
  void free() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  ~DevBuf() { free(); }
};

// At least count values; false when the device has no memory for them (the
// buffer is then empty, and the error is taken off the runtime's record)
template <class T>
bool grow(DevBuf<T> &b, size_t count) {
  if (b.n >= count) return true;
  b.free();
  const hipError_t e = hipMalloc(&b.p, count * sizeof(T));
  if (e == hipErrorOutOfMemory) {
    b.p = nullptr;
    (void)hipGetLastError();
    return false;
  }
  HIPCHECK(e);
  b.n = count;
  return true;
}

// A host array of doubles on the device in the stage kernel's arithmetic
// type: FP32 for the FP32-bulk precision from N=2 on, else FP64
struct StageTypeBuf {
  DevBuf<double> d;
  DevBuf<float> f;
  void upload(const std::vector<double> &v, int prec, int N) {
    if (prec != 0 && N >= 2) f.upload(std::vector<float>(v.begin(), v.end()));
    else d.upload(v);
  }
  const void *ptr() const { return f.p ? static_cast<const void *>(f.p) : static_cast<const void *>(d.p); }
};

// The stage states q1..q4 of a solver or group, one allocation
struct StageStates {
  DevBuf<unsigned char> mem;
  // nval values of ssize bytes each (4 or 8) per state
  void alloc(size_t nval, size_t ssize, void *q[5]) {
    mem.alloc(4 * nval * ssize);
    for (int s = 1; s < 5; ++s) q[s] = mem.p + size_t(s - 1) * nval * ssize;
  }
  // Between calls nothing lives in them (a step's first stage writes q1 before
  // anything reads it), so state transfers use them: 16 nval bytes or more for
  // a state's 8 nval
  double *staging() const { return reinterpret_cast<double *>(mem.p); }
};

// Host states in the reference layout [4][NpInt][K] to and from the device's
// tile layout (or element-major, tiled = false). The re-layout runs on the device: the host only
// copies, through device memory of the caller's (stage, the state's size) and,
// for states up to kPin bytes, one pinned host buffer. (On the host the
// strided re-layout took 14 ms into and 18 ms out of the device at 80,000
// triangles, order 4, 38 MB; the copies alone take 1.3 and 3.7 ms. A
// pageable copy of 256 KB took 115 us where the pinned one and its host copy
// take 14; from 4 MB on the pageable copy is as fast.) The pinned buffer is
// allocated at the first transfer, once, for the largest state that the owner
// will move through it (fit): grown state by state it took nine allocations in
// the first read of 24 cases, 10 ms. One transfer at a time: calls on one
// handle are not re-entrant, and every entry point waits for its stream before
// it returns.
struct HostIo {
  static constexpr size_t kPin = size_t(4) << 20;
  double *pin = nullptr;
  size_t npin = 0;
  dev::Ctl *ctl = nullptr;  // behind the buffer, in the same pinned allocation
  HostIo() = default;
  HostIo(const HostIo &) = delete;
  HostIo &operator=(const HostIo &) = delete;
  ~HostIo() { if (pin) (void)hipHostFree(pin); }
  static size_t bytes_of(int K, int NpInt) { return size_t(K) * 4 * NpInt * sizeof(double); }
  // States of K elements will be moved (all owners call it before the first transfer)
  void fit(int K, int NpInt) {
    const size_t bytes = bytes_of(K, NpInt);
    if (bytes <= kPin) npin = std::max(npin, bytes);
  }
  void reserve() {
    if (pin) return;
    HIPCHECK(hipHostMalloc(reinterpret_cast<void **>(&pin), npin + sizeof(dev::Ctl), hipHostMallocDefault));
    ctl = reinterpret_cast<dev::Ctl *>(reinterpret_cast<char *>(pin) + npin);
  }
  // Q is free again on return; the re-layout may still run on the stream
  void put(const double *Q, const int *perm, int K, int Kp, int NpInt, bool tiled, bool inert, double *stage, double *dst,
           hipStream_t s) {
    const size_t bytes = bytes_of(K, NpInt);
    reserve();
    if (bytes <= npin) {
      std::memcpy(pin, Q, bytes);
      HIPCHECK(hipMemcpyAsync(stage, pin, bytes, hipMemcpyHostToDevice, s));
    } else {
      HIPCHECK(hipMemcpyAsync(stage, Q, bytes, hipMemcpyHostToDevice, s));
      HIPCHECK(hipStreamSynchronize(s));
    }
    HIPCHECK(dev::launch_gather_state(stage, perm, K, Kp, NpInt, tiled, inert, dst, s));
  }
  // Returns when Q is written
  void get(const double *src, const int *perm, int K, int NpInt, bool tiled, double *stage, double *Q, hipStream_t s) {
    const size_t bytes = bytes_of(K, NpInt);
    reserve();
    HIPCHECK(dev::launch_scatter_state(src, perm, K, NpInt, tiled, stage, s));
    HIPCHECK(hipMemcpyAsync(bytes <= npin ? pin : Q, stage, bytes, hipMemcpyDeviceToHost, s));
    HIPCHECK(hipStreamSynchronize(s));
    if (bytes <= npin) std::memcpy(Q, pin, bytes);
  }
};

// Freestream (model_problems/Euler2D/fluids.go:245-273)
struct FreeStream {
  double gamma = 1.4, minf = 0, alpha = 0, q[4] = {1, 0, 0, 0}, pinf = 0, cinf = 0;
  void from_qinf(double g, const double qq[4]) {
    gamma = g;
    for (int i = 0; i < 4; ++i) q[i] = qq[i];
    const double oorho = 1. / q[0], u = q[1] * oorho, v = q[2] * oorho;
    pinf = (g - 1.) * (q[3] - 0.5 * q[0] * (u * u + v * v));
    cinf = std::sqrt(std::fabs(g * pinf * oorho));
  }
  void from_mach(double M, double g, double a) {
    const double ooggm1 = 1. / (g * (g - 1.));
    const double qq[4] = {1, M * std::cos(a * M_PI / 180.), M * std::sin(a * M_PI / 180.), ooggm1 + 0.5 * M * M};
    from_qinf(g, qq);
    minf = M;
    alpha = a;
  }
};

// The far-field states of a case: FSFar (NewEuler, euler.go:70) and the
// FSIn / FSOut of the shock tube (euler.go:742-743), which equal FSFar in
// the other cases
struct CaseStreams {
  FreeStream far, in, out;
};

// Parameter checks shared by every solver kind; returns GOCFD_OK or an error
int validate_params(const gocfd_params *p);

// InitializeSolution (euler.go:728-794): the freestreams, the initial state
// Q0 [4][NpInt][K] in the reference layout, and the IVortex boundary
// conversion of Wall edges (initialization.go:61-83).
void init_case(Discretisation &d, const gocfd_params &p, CaseStreams &fs, std::vector<double> &Q0);

// Device checks: gfx950 and enough LDS for the stage kernel
void check_device(int device, size_t lds_bytes);

// Physics constants of a case for the kernels
bool general_gamma(const dev::Phys &ph);  // a far-field state whose gamma is not 1.4
dev::Phys phys_of(const CaseStreams &fs, const gocfd_params &p);

// Tile layout (dev::state_at) of a reference-layout state, padding elements
// set to the inert state (host side: an ensemble's initial states)
void fill_tiles(const DeviceLayout &L, int NpInt, const double *Q, double *h);

}  // namespace capi
}  // namespace gocfd

// The opaque mesh handle of the C ABI
struct gocfd_mesh {
  gocfd::Mesh m;
};
