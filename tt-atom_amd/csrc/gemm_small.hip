// Split-plane GEMM for products too small to fill the GPU with 128 x 128 tiles (the wider linears
// of small systems and mid-size node batches; their narrow ones keep fp32 operands, gemm.hip): the
// products, arithmetic and epilogues of gemm_bf16.hip, K split over the wavefronts of one
// workgroup.
//
// A launch of few tiles is bound by the serial chain of a tile's k steps, not by the matrix cores:
// the tiled kernel's workgroup waits out a copy round trip and a barrier per 32-wide slab, and
// cutting K over workgroups instead sends every partial product through memory and a second
// launch.  Here a workgroup owns a small tile (32 or 64 on a side) and its NW wavefronts take
// consecutive ranges of K slabs (the whole tile over K / NW each), with no barrier in the k loop: a
// wavefront loads its A rows coalesced into registers, DEPTH slabs ahead, turns them through its
// own LDS area into MFMA fragments (LDS operations of one wavefront stay in order), and takes the
// packed B fragments straight to registers.  The partial tiles then meet in LDS, are added in
// wavefront order (fixed, so results repeat) and go through the shared epilogue.  Tiles are walked column-major inside each
// XCD's contiguous range, so that an XCD reads its own columns of the weight once.
#include "gemm_split.h"

#include <algorithm>

namespace {

using namespace tta_gemm;

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Output tile 32 TI x 32 TJ, NW wavefronts over K, DEPTH slabs in flight per wavefront.
template <int MODE, int TI, int TJ, int NW, int DEPTH>
__global__ __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) void gemm_small_kernel(GemmGroup g) {
  typedef Split<MODE> S;
  typedef typename Frag<S::F16>::T V8;
  constexpr int NA = S::NA, NB = S::NB, SM = 32 * TI, SN = 32 * TJ;
  constexpr int SLDT = SN + 8;           // row stride (floats) of a partial tile in LDS
  constexpr int ACH = TI * 4;            // 16-byte A loads per lane and slab
  static_assert(SM * 32 <= SM * SLDT, "the A slab lies in the wavefront's partial tile");
  __shared__ uint4 smem[NW * SM * SLDT / 4];

  const GemmArgs& p = g.p[blockIdx.z];
  const int NT32 = g.NT32[blockIdx.z], K = p.K;
  const int tm = (p.M + SM - 1) / SM, ntiles = tm * ((p.N + SN - 1) / SN);
  const int per_xcd = (ntiles + 7) / 8, idx = (int)blockIdx.x / 8;
  const int tile = ((int)blockIdx.x % 8) * per_xcd + idx;
  if (idx >= per_xcd || tile >= ntiles) return;
  const int m0 = (tile % tm) * SM, n0 = (tile / tm) * SN;
  const int t = threadIdx.x, lane = t & 63, l32 = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nk = (K + BK - 1) / BK, per = (nk + NW - 1) / NW;
  const int s0 = min(wave * per, nk), s1 = min(s0 + per, nk);

  floatx16 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  RowScale<TI, TJ, S::F16> rs;

  // A: load h of a slab covers rows 8 h .. 8 h + 7, eight lanes (128 bytes) a row; rows past M and
  // columns past K get an offset past the buffer's end and read as zero.  B: 1 KB fragments.
  // The per-lane offsets are fixed and the rest of an address is scalar (host-checked below 2^31).
  const int ar = lane >> 3, ac = lane & 7, ld4 = (int)p.lda * 4, rows_left = p.M - m0;
  const int avo = ar * ld4 + 16 * ac, bvo = lane * 16;
  const __amdgpu_buffer_rsrc_t arsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(p.A + (int64_t)m0 * p.lda), (short)0, 0x7ffffffe, 0x00020000);
  const __amdgpu_buffer_rsrc_t brsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.B), (short)0, 0x7ffffffe, 0x00020000);
  u32x4 pa[DEPTH][ACH], pb[DEPTH][TJ][2][NB];
  auto load = [&](int kt, u32x4 (&a)[ACH], u32x4 (&b)[TJ][2][NB]) {
    const int left = kt * BK + 4 * ac < K ? rows_left : 0;  // rows this lane's column reads
#pragma unroll
    for (int h = 0; h < ACH; ++h) {
      const int vo = 8 * h + ar < left ? avo : (int)0x7fffffff;
      a[h] = __builtin_amdgcn_raw_buffer_load_b128(arsrc, vo, 8 * h * ld4 + kt * BK * 4, 0);
    }
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int q = 0; q < NB; ++q)
          b[j][ks][q] = __builtin_amdgcn_raw_buffer_load_b128(
              brsrc, bvo, ((kt * NB + q) * NT32 + n0 / 32 + j) * 2048 + ks * 1024, 0);
  };
  uint4* As = smem + wave * (SM * SLDT / 4);
  // The products of one slab.  All but the leading ones (a0 b0) are summed by themselves and enter
  // the accumulator together, once per slab: every rounding of the accumulator costs half an ulp of
  // the whole sum, and a wavefront's share of K is up to twice the split-K form's chunk.  Relative
  // 2-norm error in mode 16, one chain -> this (split-K form, fp32 kernel): 576 x 1024 x 1024 1.96e-7 ->
  // 1.47e-7 (1.57e-7, 5.7e-7), 514 x 640 x 768 1.75e-7 -> 1.36e-7 (1.54e-7, 5.0e-7), 300 x 1024 x 256
  // 1.23e-7 -> 1.10e-7 (1.48e-7, 2.9e-7); 12.7 -> 13.2 us at 576 x 1024 x 1024
  auto mm = [&](const floatx4 (&x)[2][TI][2], const u32x4 (&b)[TJ][2][NB], bool scaled) {
    V8 av[2][TI][NA];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        if constexpr (S::F16)
          split8_f16<NA>(x[ks][i][0], x[ks][i][1], scaled ? rs.er[i] : 0, av[ks][i]);
        else
          split8<NA>(x[ks][i][0], x[ks][i][1], av[ks][i]);
      }
    auto prod = [&](int i, int j, int ks, int q, const floatx16& c) {
      return mfma32(av[ks][i][S::pa[q]], __builtin_bit_cast(V8, b[j][ks][S::pb[q]]), c);
    };
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        floatx16 lo;
#pragma unroll
        for (int r = 0; r < 16; ++r) lo[r] = 0.f;
#pragma unroll
        for (int q = 0; q + 1 < S::NP; ++q)
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) lo = prod(i, j, ks, q, lo);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) acc[i][j] = prod(i, j, ks, S::NP - 1, acc[i][j]);
        if constexpr (S::NP > 1) acc[i][j] += lo;
      }
  };
  // (the LDS area passes values between lanes of the wavefront, whose LDS operations run in program
  // order: the wave barriers only keep the compiler from moving them across each other)
  auto compute = [&](const u32x4 (&a)[ACH], const u32x4 (&b)[TJ][2][NB]) {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int h = 0; h < ACH; ++h) {
      const int row = 8 * h + ar;
      As[row * 8 + (ac ^ aswz(row))] = __builtin_bit_cast(uint4, a[h]);
    }
    __builtin_amdgcn_wave_barrier();
    floatx4 x[2][TI][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const int row = i * 32 + l32, c0 = 4 * ks + 2 * lh;
        x[ks][i][0] = __builtin_bit_cast(floatx4, As[row * 8 + (c0 ^ aswz(row))]);
        x[ks][i][1] = __builtin_bit_cast(floatx4, As[row * 8 + ((c0 + 1) ^ aswz(row))]);
      }
    rs.check(x[0], x[1], acc, lh);
    if (!S::F16 || rs.unscaled)
      mm(x, b, false);
    else
      mm(x, b, true);
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (s0 + d < s1) load(s0 + d, pa[d], pb[d]);
  for (int s = s0; s < s1; s += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (s + d < s1) {
        compute(pa[d], pb[d]);
        if (s + d + DEPTH < s1) load(s + d + DEPTH, pa[d], pb[d]);
      }
    }
  }

  // undo the scales, then the wavefront's partial tile to LDS
  float* Ct = reinterpret_cast<float*>(As);
  if constexpr (S::F16) {
    const int* Fc = reinterpret_cast<const int*>(static_cast<const uint4*>(p.B) +
                                                 (int64_t)nk * NB * NT32 * 128);
    int fc[TJ];
#pragma unroll
    for (int j = 0; j < TJ; ++j) fc[j] = Fc[n0 + j * 32 + l32];
    rs.undo(acc, fc, lh);
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        Ct[(i * 32 + acc_row(r, lh)) * SLDT + j * 32 + l32] = acc[i][j][r];
  __syncthreads();
  // sum of the partials in wavefront order, left in the first one's place by the thread that
  // takes the element through the epilogue
  float* C0 = reinterpret_cast<float*>(smem);
  constexpr int CG = SN / 4;
  for (int row = t / CG; row < SM; row += 64 * NW / CG) {
    floatx4* c = reinterpret_cast<floatx4*>(C0 + row * SLDT + 4 * (t % CG));
    floatx4 v = c[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += c[w * (SM * SLDT / 4)];
    c[0] = v;
  }
  const bool vec_ok = g.vec[blockIdx.z] != 0, full = m0 + SM <= p.M && n0 + SN <= p.N;
  constexpr int NTH = 64 * NW;
  switch (p.epi) {
    case EPI_SILU:
      epilogue_rows<EPI_SILU, false, CG>(p, C0, SLDT, SM, m0, n0, t, NTH, vec_ok, full);
      break;
    case EPI_ACCUM:
      epilogue_rows<EPI_ACCUM, false, CG>(p, C0, SLDT, SM, m0, n0, t, NTH, vec_ok, full);
      break;
    case EPI_PRE_SILU:
      epilogue_rows<EPI_PRE_SILU, false, CG>(p, C0, SLDT, SM, m0, n0, t, NTH, vec_ok, full);
      break;
    case EPI_SILU_GRAD:
      epilogue_rows<EPI_SILU_GRAD, false, CG>(p, C0, SLDT, SM, m0, n0, t, NTH, vec_ok, full);
      break;
    case EPI_SIGMOID:
      epilogue_rows<EPI_SIGMOID, false, CG>(p, C0, SLDT, SM, m0, n0, t, NTH, vec_ok, full);
      break;
    case EPI_GATE:
      epilogue_rows<EPI_GATE, false, CG>(p, C0, SLDT, SM, m0, n0, t, NTH, vec_ok, full, &g.gate,
                                         g.gc0[blockIdx.z]);
      break;
    case EPI_GATE_BWD:
      epilogue_rows<EPI_GATE_BWD, false, CG>(p, C0, SLDT, SM, m0, n0, t, NTH, vec_ok, full,
                                             &g.gate, g.gc0[blockIdx.z]);
      break;
    default:
      epilogue_rows<EPI_STORE, false, CG>(p, C0, SLDT, SM, m0, n0, t, NTH, vec_ok, full);
  }
}

// Which products run here, and on how many wavefronts, is a rule on the product's own rows, columns
// and K (small_waves), so that its k sums, and its bits, do not depend on what else is in its
// launch: eight wavefronts share K up to 256 rows and past 1024 columns of K (shares of 256 at most
// up to K = 2048), four otherwise.  The tile is the launch's (every tile adds an element's products
// in one order): a compute unit holds one workgroup of eight wavefronts or two of four, and the
// tile is the smallest one (the shortest chain of k steps) whose workgroups are still one round, or
// 64 x 64.  Measured per launch with one chain of additions per accumulator, 3 to 4 % faster than now
// (us; the split-K launch pair or fp32 kernel that ran before, then 32 x 32 / 32 x 64 / 64 x 64
// tiles, then the tiled kernel): eight wavefronts, 72 x 1024 x 1024: 11.7; 7.3, 8.0, 11.1; 26.6.
// Four: 433 x 1024 x 1024: 20.2; 11.0, 10.3, 13.6; 28.1 (eight: 14.4, 9.1, 12.0).  576 x 1024 x
// 1024: 24.0; 16.3, 12.2, 13.9; 28.2.  1937 x 1024 x 1024: 77.6; 47.3, 29.4, 22.8; 30.2.  2500 x
// 1024 x 1024 (640 tiles of 64 x 64): 89.8; 56.5, 39.2, 34.2; 31.1.  4000 x 1024 x 1024: 64 x 64
// tiles 47, tiled 34; 4000 x 4096 x 1024: 175, 117.  From 4096 rows on callers split a convolution's
// columns over launches and expect the same bits: no small tile.
enum SmallTile { k32x32, k32x64, k64x64 };

SmallTile small_tile(const GemmGroup& g, int n, int waves) {
  auto blocks = [&](int sm, int sn) {
    int64_t b = 0;
    for (int i = 0; i < n; ++i) b += (int64_t)tta_blocks(g.p[i].M, sm) * tta_blocks(g.p[i].N, sn);
    return b;
  };
  if (blocks(32, 32) <= 256) return k32x32;
  if (blocks(32, 64) <= (waves == 8 ? 256 : 512)) return k32x64;
  return k64x64;
}

template <int MODE, int TI, int TJ, int NW, int DEPTH>
void launch_tile(const GemmGroup& g, int n, hipStream_t s) {
  int64_t grid = 0;
  for (int i = 0; i < n; ++i) {
    const int64_t tiles =
        (int64_t)tta_blocks(g.p[i].M, 32 * TI) * tta_blocks(g.p[i].N, 32 * TJ);
    grid = std::max<int64_t>(grid, (tiles + 7) / 8 * 8);
  }
  hipLaunchKernelGGL((gemm_small_kernel<MODE, TI, TJ, NW, DEPTH>),
                     dim3((unsigned)grid, 1, (unsigned)n), dim3(64 * NW), 0, s, g);
}

template <int MODE, int NW>
void launch_waves(const GemmGroup& g, int n, hipStream_t s) {
  // slabs in flight: what 256 registers hold beside the accumulators and fragments
  constexpr int D = Split<MODE>::NB > 2 ? 1 : 2;
  switch (small_tile(g, n, NW)) {
    case k32x32: launch_tile<MODE, 1, 1, NW, 2 * D>(g, n, s); break;
    case k32x64: launch_tile<MODE, 1, 2, NW, D>(g, n, s); break;
    default: launch_tile<MODE, 2, 2, NW, 1>(g, n, s); break;
  }
}

template <int MODE>
void launch_mode_small(const GemmGroup& g, int n, int waves, hipStream_t s) {
  if (waves == 8)
    launch_waves<MODE, 8>(g, n, s);
  else
    launch_waves<MODE, 4>(g, n, s);
}

}  // namespace

namespace tta_gemm {

int small_waves(const GemmArgs& p) {
  if (p.M >= 4096 || (int64_t)tta_blocks(p.M, 64) * tta_blocks(p.N, 64) > 512) return 0;
  return p.M <= 256 || p.K > 1024 ? 8 : 4;
}

int launch_small(GemmGroup& g, int n, int waves, int mode, hipStream_t s) {
  switch (mode) {
    case 1: launch_mode_small<1>(g, n, waves, s); break;
    case 3: launch_mode_small<3>(g, n, waves, s); break;
    case 16: launch_mode_small<16>(g, n, waves, s); break;
    default: launch_mode_small<6>(g, n, waves, s); break;
  }
  TTA_CHECK_LAUNCH("tta_gemm_bf16x");
  return tta::kOk;
}

}  // namespace tta_gemm
