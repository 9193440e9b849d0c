// Shared helpers for the tt-atom MI355X (gfx950) kernels: status codes, the thread-local error
// message behind tta_last_error(), launch checks and small device utilities.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

namespace tta {

// Thread-local last-error text; every extern "C" entry point returns 0 on success and a
// non-zero status after writing a message here.
void set_error(const char* fmt, ...);

enum Status : int {
  kOk = 0,
  kBadArgument = 1,
  kLaunchFailed = 2,
  kUnsupported = 3,
};

}  // namespace tta

#define TTA_CHECK_ARG(cond, ...)                 \
  do {                                           \
    if (!(cond)) {                               \
      tta::set_error(__VA_ARGS__);               \
      return tta::kBadArgument;                  \
    }                                            \
  } while (0)

#define TTA_CHECK_LAUNCH(name)                                                   \
  do {                                                                           \
    hipError_t _e = hipGetLastError();                                           \
    if (_e != hipSuccess) {                                                      \
      tta::set_error("%s: launch failed: %s", name, hipGetErrorString(_e));      \
      return tta::kLaunchFailed;                                                 \
    }                                                                            \
  } while (0)

// ---------------------------------------------------------------------------- device helpers
__device__ __forceinline__ float tta_sigmoid(float x) { return 1.0f / (1.0f + __expf(-x)); }

// Sigmoid and SiLU for the force path, whose parity tolerance is tight, in a third fewer
// vector instructions (26 for 38) than 1 / (1 + expf(-x)) with a divide takes: the epilogues of the hidden-layer products
// evaluate them per output, and their vector instructions were as many as the k loop's.  With
// e = exp(-|x|) in (0, 1] nothing overflows and sigmoid(x) = (x < 0 ? e : 1) / (1 + e).  e is the
// hardware's 2^p at p = -|x| log2(e), times 1 + the rounding error of p (two fused steps; NaN at
// infinite x, where the fminf keeps it harmless), and the quotient n r with the hardware
// reciprocal r gets one correction step by its own residual.  SiLU puts x into the numerator, one
// rounding fewer than x sigmoid(x).  Relative 2-norm error against fp64 over x ~ N(0, 1) / N(0, 3)
// / U(-20, 20), previous form -> this one: sigmoid 3.89e-8 / 3.79e-8 / 3.45e-8 -> 3.79e-8 /
// 3.78e-8 / 3.45e-8, SiLU 4.48e-8 / 4.57e-8 / 3.35e-8 -> 4.05e-8 / 4.21e-8 / 3.31e-8, its
// derivative 4.68e-8 / 9.33e-8 / 3.20e-7 -> 4.59e-8 / 9.32e-8 / 3.20e-7.  (U(-80, 0), which no
// activation here reaches: SiLU 4.75e-8 -> 5.58e-8, the other two lower.  Below x = -87.3 the
// results are zero; the sigmoid there is denormal.)  Measured (us): 196,555 x 1024 x 1024 with
// the SiLU-gradient epilogue 1336 -> 1326, with the two-output one 1374 -> 1360; an Orb layer of
// 30,011 edges 2805 -> 2671, its reduced-precision edge encoder 650 -> 617.
__device__ __forceinline__ void tta_exp_parts(float x, float& e, float& d, float& r) {
  const float a = fabsf(x), log2e = 1.44269502f;
  const float p = -a * log2e;
  float c = fmaf(-a, log2e, -p);       // rounding error of p,
  c = fmaf(-a, 1.92596299e-8f, c);     // and of log2e
  c = fminf(c * 0.693147182f, 1e-4f);
  e = __builtin_amdgcn_exp2f(p);
  e = fmaf(e, c, e);
  d = 1.0f + e;
  r = __builtin_amdgcn_rcpf(d);
}
__device__ __forceinline__ float tta_sigmoid_acc(float x) {
  float e, d, r;
  tta_exp_parts(x, e, d, r);
  const float n = x < 0.f ? e : 1.0f, q = n * r;
  return fmaf(fmaf(-d, q, n), r, q);
}
__device__ __forceinline__ float tta_silu(float x) {
  float e, d, r;
  tta_exp_parts(x, e, d, r);
  const float n = x < 0.f ? x * e : x, q = n * r;
  return fmaf(fminf(fmaf(-d, q, n), 3e38f), r, q);  // (fminf: the residual of x = inf is NaN)
}
// d silu / dx = s (1 + x (1 - s))
__device__ __forceinline__ float tta_silu_grad(float x) {
  float s = tta_sigmoid_acc(x);
  return s * (1.0f + x * (1.0f - s));
}

// Butterfly sum over `width` consecutive lanes (width a power of two <= 64).
__device__ __forceinline__ float tta_group_sum(float v, int width) {
  for (int o = width >> 1; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

static inline unsigned tta_blocks(int64_t n, int per) {
  return (unsigned)((n + per - 1) / per);
}
