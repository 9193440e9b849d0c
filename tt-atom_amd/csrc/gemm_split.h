// Shared pieces of the split-plane GEMM kernels (gemm_bf16.hip, gemm_small.hip, gemm_wide.hip): the
// plane formats and their products, the splits of an fp32 operand, and the epilogue of a tile staged in LDS.  The
// modes, the packed layout of B and the scaling of mode 16 are described in gemm_bf16.hip.
#pragma once

#include "gemm_common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

namespace tta_gemm {

template <int MODE>
struct Split;
template <>
struct Split<1> {
  static constexpr int NA = 1, NB = 1, NP = 1;
  static constexpr bool F16 = false;
  static constexpr int pa[1] = {0};
  static constexpr int pb[1] = {0};
};
template <>
struct Split<3> {
  static constexpr int NA = 2, NB = 2, NP = 3;
  static constexpr bool F16 = false;
  static constexpr int pa[3] = {0, 1, 0};
  static constexpr int pb[3] = {1, 0, 0};
};
template <>
struct Split<6> {
  // smallest terms first
  static constexpr int NA = 3, NB = 3, NP = 6;
  static constexpr bool F16 = false;
  static constexpr int pa[6] = {1, 0, 2, 0, 1, 0};
  static constexpr int pb[6] = {1, 2, 0, 1, 0, 0};
};
template <>
struct Split<16> {
  static constexpr int NA = 2, NB = 2, NP = 3;
  static constexpr bool F16 = true;
  static constexpr int pa[3] = {1, 0, 0};
  static constexpr int pb[3] = {0, 1, 0};
};

// Fragment element type per plane format, and the 32x32x16 MFMA on it.
template <bool F16>
struct Frag {
  typedef bf16x8 T;
};
template <>
struct Frag<true> {
  typedef f16x8 T;
};
__device__ __forceinline__ floatx16 mfma32(bf16x8 a, bf16x8 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ floatx16 mfma32(f16x8 a, f16x8 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// mode 16 scaling: a B column's values are multiplied by 2^-(e - kTop), e the frexp exponent of
// its max |value| (max < 2^e), so they land below 2^kTop; an A row's shift follows the rule in the
// header.  kNoExp marks an A row with no nonzero value yet.
constexpr int kTop = 11, kNoExp = -100000;

constexpr int BN = 128, BK = 32;
constexpr int NF = (BN / 32) * 2;  // B fragments per plane per k-step: n32 tiles x k16 halves

__device__ __forceinline__ float epi_one(const GemmArgs& p, float v, int row, int col) {
  if (p.bias) v += p.bias[col];
  if (p.P)
    v += p.P[(int64_t)p.idx0[row] * p.ldp + col] + p.P[(int64_t)p.idx1[row] * p.ldp + p.off1 + col];
  const int64_t off = (int64_t)row * p.ldc + col;
  if (p.epi == EPI_SILU) v = tta_silu(v);
  if (p.epi == EPI_SIGMOID) v = tta_sigmoid_acc(v);
  if (p.epi == EPI_ACCUM) v += p.C[off];
  if (p.epi == EPI_PRE_SILU) p.C2[off] = tta_silu(v);
  if (p.epi == EPI_SILU_GRAD) v = v * tta_silu_grad(p.aux[off]);
  return v;
}

// Rows [row0, row0 + rows) of a 4 CG-column output tile staged in LDS (row stride ldt floats).
// Thread t owns float4 column group t % CG and rows t / CG, t / CG + nth / CG, ...: the bias,
// the column checks and the lane's column offset are set once, and the epilogue type is a
// template parameter, so a row costs one LDS read, one address add and one 16-byte store.
// vec_ok (host-checked 16-byte alignment of every operand row) selects the float4 path; full
// (the tile lies inside M x N) drops the bounds checks.
// Split-K: rows [row0, row0 + rows) of a staged tile, as they are, into the chunk's partial W
// (row-major, row stride N, 16-byte aligned base); the reduction applies bias and epilogue.
__device__ __forceinline__ void partial_rows(float* W, int M, int N, const float* Ct, int ldt,
                                             int rows, int row0, int n0, int t, int nth) {
  const int c4 = t & 31, rstep = nth >> 5;
  const int col = n0 + 4 * c4;
  if (col >= N) return;
  for (int rr = t >> 5; rr < rows; rr += rstep) {
    const int row = row0 + rr;
    if (row >= M) break;
    const floatx4 a = *reinterpret_cast<const floatx4*>(Ct + rr * ldt + 4 * c4);
    float* w = W + (int64_t)row * N + col;
    if (N % 4 == 0 && col + 3 < N) {
      *reinterpret_cast<floatx4*>(w) = a;
    } else {
      for (int e = 0; e < 4 && col + e < N; ++e) w[e] = a[e];
    }
  }
}

// EPI_GATE / EPI_GATE_BWD (ge, gc0: the launch's gate operands and the product's first
// coefficient) take the float4 path only (the host requires their alignments); a thread's four
// columns lie in one coefficient (H % 4 == 0).
template <int EPI, bool BATCH, int CG = 32>
__device__ __forceinline__ void epilogue_rows(const GemmArgs& p, const float* Ct, int ldt,
                                              int rows, int row0, int n0, int t, int nth,
                                              bool vec_ok, bool full,
                                              const GateEpi* ge = nullptr, int gc0 = 0) {
  constexpr bool GATE = EPI == EPI_GATE || EPI == EPI_GATE_BWD;
  const int c4 = t & (CG - 1), rstep = nth / CG;
  const int col = n0 + 4 * c4;
  if (vec_ok && (full || col + 3 < p.N)) {
    const floatx4 bv = p.bias ? *reinterpret_cast<const floatx4*>(p.bias + col)
                              : floatx4{0.f, 0.f, 0.f, 0.f};
    const bool gather = p.P != nullptr;
    // gate: coefficient gc of this thread's columns, their channel gh, gating column gcol
    int gc = 0, gh = 0, gcol = 0;
    if constexpr (GATE) {
      gc = gate_coef(*ge, gc0, col);
      gh = col - (gc - gc0) * ge->H;
      gcol = gc > 0 ? gate_gcol(*ge, gc, gh) : 0;
    }
    // gate epilogue of one float4: coefficient 0 stores its pre-activation and takes SiLU (the
    // backward: is multiplied by silu' of the stored x0 values gv), the others are scaled by their
    // gating sigmoids gv
    auto gate4 = [&](floatx4& v, const floatx4& gv, int row) {
      if (gc > 0) {
        v = v * gv;
      } else if constexpr (EPI == EPI_GATE) {
        __builtin_nontemporal_store(v, reinterpret_cast<floatx4*>(ge->x0 + (int64_t)row * ge->ldx0 + gh));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = tta_silu(v[e]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] * tta_silu_grad(gv[e]);
      }
    };
    // the gate operand of one float4 of row `row`: its sigmoids, or (backward, coefficient 0) x0
    auto gload = [&](int row) -> floatx4 {
      if (gc > 0)
        return *reinterpret_cast<const floatx4*>(ge->sig + (int64_t)row * ge->ldg + gcol);
      if constexpr (EPI == EPI_GATE_BWD)
        return *reinterpret_cast<const floatx4*>(ge->x0 + (int64_t)row * ge->ldx0 + gh);
      return floatx4{0.f, 0.f, 0.f, 0.f};
    };
    constexpr bool LOADS = EPI == EPI_ACCUM || EPI == EPI_SILU_GRAD || GATE;
    constexpr int RB = 8;
    if (BATCH && full && (LOADS || gather) && rows % (RB * rstep) == 0) {
      // An epilogue that reads memory (the accumulated C, the SiLU argument, the gathered rows;
      // BATCH: the callers whose register budget has room for it)
      // issues a batch of RB rows' loads -- the gather indices first, then the rows they name --
      // before it uses any, so their latencies overlap instead of adding up row by row.
#pragma unroll 1
      for (int rb = t / CG; rb < rows; rb += RB * rstep) {
        int i0[RB], i1[RB];
        floatx4 ex[RB], pv[RB];
#pragma unroll
        for (int i = 0; i < RB; ++i) {
          const int row = row0 + rb + i * rstep;
          if (gather) {
            i0[i] = p.idx0[row];
            i1[i] = p.idx1[row];
          }
          if constexpr (EPI == EPI_ACCUM)
            ex[i] = *reinterpret_cast<const floatx4*>(p.C + (int64_t)row * p.ldc + col);
          if constexpr (EPI == EPI_SILU_GRAD)
            ex[i] = *reinterpret_cast<const floatx4*>(p.aux + (int64_t)row * p.ldc + col);
          if constexpr (GATE) ex[i] = gload(row);
        }
        if (gather) {
#pragma unroll
          for (int i = 0; i < RB; ++i)
            pv[i] = *reinterpret_cast<const floatx4*>(p.P + (int64_t)i0[i] * p.ldp + col) +
                    *reinterpret_cast<const floatx4*>(p.P + (int64_t)i1[i] * p.ldp + p.off1 + col);
        }
#pragma unroll
        for (int i = 0; i < RB; ++i) {
          const int rr = rb + i * rstep, row = row0 + rr;
          floatx4 v = *reinterpret_cast<const floatx4*>(Ct + rr * ldt + 4 * c4) + bv;
          const int64_t off = (int64_t)row * p.ldc + col;
          if (gather) v += pv[i];
          if constexpr (EPI == EPI_ACCUM) v += ex[i];
          if constexpr (GATE) gate4(v, ex[i], row);
          if constexpr (EPI == EPI_SIGMOID) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = tta_sigmoid_acc(v[e]);
          }
          if constexpr (EPI == EPI_SILU || EPI == EPI_PRE_SILU || EPI == EPI_SILU_GRAD) {
            floatx4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e)
              w[e] = EPI == EPI_SILU_GRAD ? v[e] * tta_silu_grad(ex[i][e]) : tta_silu(v[e]);
            if constexpr (EPI == EPI_PRE_SILU)
              __builtin_nontemporal_store(w, reinterpret_cast<floatx4*>(p.C2 + off));
            else
              v = w;
          }
          __builtin_nontemporal_store(v, reinterpret_cast<floatx4*>(p.C + off));
        }
      }
      return;
    }
#pragma unroll 4
    for (int rr = t / CG; rr < rows; rr += rstep) {
      const int row = row0 + rr;
      if (!full && row >= p.M) break;
      floatx4 v = *reinterpret_cast<const floatx4*>(Ct + rr * ldt + 4 * c4) + bv;
      const int64_t off = (int64_t)row * p.ldc + col;
      if (gather)
        v += *reinterpret_cast<const floatx4*>(p.P + (int64_t)p.idx0[row] * p.ldp + col) +
             *reinterpret_cast<const floatx4*>(p.P + (int64_t)p.idx1[row] * p.ldp + p.off1 + col);
      if constexpr (EPI == EPI_ACCUM) v += *reinterpret_cast<const floatx4*>(p.C + off);
      if constexpr (GATE) gate4(v, gload(row), row);
      if constexpr (EPI == EPI_SIGMOID) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = tta_sigmoid_acc(v[e]);
      }
      if constexpr (EPI == EPI_SILU || EPI == EPI_PRE_SILU || EPI == EPI_SILU_GRAD) {
        floatx4 w;
        if constexpr (EPI == EPI_SILU_GRAD) {
          const floatx4 x = *reinterpret_cast<const floatx4*>(p.aux + off);
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = v[e] * tta_silu_grad(x[e]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = tta_silu(v[e]);
        }
        if constexpr (EPI == EPI_PRE_SILU)
          __builtin_nontemporal_store(w, reinterpret_cast<floatx4*>(p.C2 + off));
        else
          v = w;
      }
      // streaming stores: the outputs (hundreds of MB on edge-level shapes) would otherwise
      // evict the A row panels that the other column tiles are still re-reading from L2
      // (+15-17 % on the write-heavy short-K shapes)
      __builtin_nontemporal_store(v, reinterpret_cast<floatx4*>(p.C + off));
    }
  } else if constexpr (!GATE) {
    for (int rr = t / CG; rr < rows; rr += rstep) {
      const int row = row0 + rr;
      if (row >= p.M) break;
      const floatx4 a = *reinterpret_cast<const floatx4*>(Ct + rr * ldt + 4 * c4);
      for (int e = 0; e < 4 && col + e < p.N; ++e)
        p.C[(int64_t)row * p.ldc + col + e] = epi_one(p, a[e], row, col + e);
    }
  }
}

// Split 8 fp32 values into NPL bf16 planes (round-to-nearest residuals), pairs at a time.
template <int NPL>
__device__ __forceinline__ void split8(const floatx4& x0, const floatx4& x1, bf16x8 (&out)[NPL]) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 h2 __attribute__((ext_vector_type(2)));
  f2 r[4] = {f2{x0[0], x0[1]}, f2{x0[2], x0[3]}, f2{x1[0], x1[1]}, f2{x1[2], x1[3]}};
#pragma unroll
  for (int q = 0; q < NPL; ++q) {
    h2 h[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      h[i] = __builtin_convertvector(r[i], h2);
      if (q + 1 < NPL) r[i] = r[i] - __builtin_convertvector(h[i], f2);
    }
    out[q] = bf16x8{h[0][0], h[0][1], h[1][0], h[1][1], h[2][0], h[2][1], h[3][0], h[3][1]};
  }
}

// x - (fp16 half 0 / half 1 of hpair) in one v_fma_mix_f32, which reads the fp16 operand in
// place (op_sel_hi marks source 0 as fp16, op_sel picks its half): no conversion back to fp32.
__device__ __forceinline__ float resid_lo(float x, unsigned hpair) {
  float r;
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(hpair), "v"(x));
  return r;
}
__device__ __forceinline__ float resid_hi(float x, unsigned hpair) {
  float r;
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
      : "=v"(r)
      : "v"(hpair), "v"(x));
  return r;
}

// max(|a|, |b|, c) and max(a, b, c) in one v_max3_f32 (abs as source modifiers; fmaxf would
// add a canonicalising max per operand).  Only the exponent of the result is used.
__device__ __forceinline__ float max3_abs(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, |%1|, |%2|, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// Split 8 fp32 values, scaled by 2^-sh, into two fp16 planes (round-to-nearest residuals).
template <int NPL>
__device__ __forceinline__ void split8_f16(const floatx4& x0, const floatx4& x1, int sh,
                                           f16x8 (&out)[NPL]) {
  static_assert(NPL == 2, "two fp16 planes");
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  f2 r[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    r[i] = f2{__builtin_amdgcn_ldexpf(x0[2 * i], -sh), __builtin_amdgcn_ldexpf(x0[2 * i + 1], -sh)};
    r[i + 2] =
        f2{__builtin_amdgcn_ldexpf(x1[2 * i], -sh), __builtin_amdgcn_ldexpf(x1[2 * i + 1], -sh)};
  }
  h2 h[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    h[i] = __builtin_convertvector(r[i], h2);
    const unsigned hp = __builtin_bit_cast(unsigned, h[i]);
    l[i] = __builtin_convertvector(f2{resid_lo(r[i][0], hp), resid_hi(r[i][1], hp)}, h2);
  }
  out[0] = f16x8{h[0][0], h[0][1], h[1][0], h[1][1], h[2][0], h[2][1], h[3][0], h[3][1]};
  out[1] = f16x8{l[0][0], l[0][1], l[1][0], l[1][1], l[2][0], l[2][1], l[3][0], l[3][1]};
}

// Mode 16's row scaling for a wavefront of TI row blocks x TJ column blocks (the rule: header of
// gemm_bf16.hip): er[i] is the shift E of the lane's A row l32 of row block i, whose values enter
// the planes multiplied by 2^-E (lanes l and l + 32 hold the same row and agree); accumulator
// element r of a 32 x 32 block belongs to row acc_row(r, lh) of the block, whose shift lane
// acc_row(r, lh) holds.
__device__ __forceinline__ int acc_row(int r, int lh) { return 8 * (r >> 2) + 4 * lh + (r & 3); }

template <int TI, int TJ, bool F16>
struct RowScale {
  int er[TI];
  bool unscaled = true;  // wave-uniform: E is 0 or unset on every row (the common case)
  __device__ __forceinline__ RowScale() {
#pragma unroll
    for (int i = 0; i < TI; ++i) er[i] = kNoExp;
  }
  // the shift check of one 32-wide k slab (both of its halves); returns whether a shift changed
  // (the accumulators were rescaled)
  __device__ __forceinline__ bool check(const floatx4 (&x0)[TI][2], const floatx4 (&x1)[TI][2],
                                        floatx16 (&acc)[TI][TJ], int lh) {
    if constexpr (F16) {
      int en[TI];
      bool grow = false;
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        float m = 0.f;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) m = max3_abs(x0[i][c][e], x1[i][c][e], m);
        // the row's other 16 values of this k slab are in lane l ^ 32: v_permlane32_swap trades
        // the upper half of one register with the lower half of another, so with m in both, one
        // of them ends up holding the partner's m in every lane (a permute through LDS would wait
        // on the fragment reads in flight).  s_nop 1: the two wait states the swap needs after
        // the VALU writes of its operands.
        {
          float u = m, w = m;
          asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(u), "+v"(w));
          m = max3(m, u, w);
        }
        const int e = m > 0.f ? __builtin_amdgcn_frexp_expf(m) : kNoExp;
        // values below 2^e reach 2^(e - E): a new shift once that passes 2^15, and for the row's
        // first nonzero slab (E = kNoExp); the new shift is never below the old one
        const bool g = e != kNoExp && e - er[i] > 15;
        en[i] = g ? ((e >= 0 && e <= 15) ? 0 : e - kTop) : er[i];
        grow |= g;
      }
      if (__any(grow)) {  // rare: a row's first nonzero k slab, or a much larger value
#pragma unroll
        for (int i = 0; i < TI; ++i) {
          const int d = er[i] - en[i];  // <= 0; the sentinel's huge d zeroes an all-zero acc
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int dr = __shfl(d, acc_row(r, lh));
#pragma unroll
            for (int j = 0; j < TJ; ++j) acc[i][j][r] = __builtin_amdgcn_ldexpf(acc[i][j][r], dr);
          }
          er[i] = en[i];
        }
        unscaled = all_unscaled();
        return true;
      }
    }
    return false;
  }
  // Whether every row of the wavefront has a shift, 0; while that holds a slab needs a new shift only
  // where a value reaches 2^15, which each lane can tell of its own values (overflows): no exchange
  // with the lane that holds the row's other half.
  __device__ __forceinline__ bool all_zero() const {
    bool z = true;
#pragma unroll
    for (int i = 0; i < TI; ++i) z &= er[i] == 0;
    return __all(z);
  }
  __device__ __forceinline__ bool overflows(const floatx4 (&x0)[TI][2],
                                            const floatx4 (&x1)[TI][2]) const {
    if constexpr (!F16) return false;
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) m = max3_abs(x0[i][c][e], x1[i][c][e], m);
    return __any(!(m < 32768.f));
  }
  __device__ __forceinline__ bool all_unscaled() const {
    bool u = true;
#pragma unroll
    for (int i = 0; i < TI; ++i) u &= er[i] == 0 || er[i] == kNoExp;
    return __all(u);
  }
  // undo the scales: acc * 2^(E[row] + F[col]), fc[j] the exponent F of the lane's column l32 of
  // column block j
  __device__ __forceinline__ void undo(floatx16 (&acc)[TI][TJ], const int (&fc)[TJ], int lh) const {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int rs = __shfl(er[i], acc_row(r, lh));
#pragma unroll
        for (int j = 0; j < TJ; ++j)
          acc[i][j][r] = __builtin_amdgcn_ldexpf(acc[i][j][r], rs + fc[j]);
      }
  }
};

// A (fp32) tile row: 8 chunks of 16 B per 32-wide k slab, chunk c of row r stored at c ^ aswz(r):
// 16 consecutive rows at one logical chunk then cover all 64 banks.
__device__ __forceinline__ int aswz(int row) { return (row >> 1) & 7; }

// The small-launch kernel (gemm_small.hip): the wavefronts that share a product's K there, 0 for a
// product that does not run there, and its launch for n products of one such number.
int small_waves(const GemmArgs& p);
int launch_small(GemmGroup& g, int n, int waves, int mode, hipStream_t s);

// The 128 x 256 kernel (gemm_wide.hip); cap: most blocks per product (persistent tiles).
bool wide_ok(const GemmGroup& g, int n, int mode, int cap);
int launch_wide(GemmGroup& g, int n, int mode, int cap, hipStream_t s);

}  // namespace tta_gemm
