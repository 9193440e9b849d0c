// Split-plane GEMM for launches that fill the GPU: 128 x 256 tiles (products, arithmetic, scaling
// rule and epilogues of gemm_bf16.hip).
//
// The 128 x 128 kernel moves 32 KB from L2 to LDS and splits 128 x 32 A values for every 24 matrix
// instructions of a wavefront; here a wavefront's tile is 32 x 256, so each split A value feeds
// eight column blocks instead of four and a step's copies bring 24 KB for as many instructions.
// Two workgroups still share a compute unit, so that one's epilogue overlaps the other's k loop: a
// stage holds a 16-wide k step (24 KB) and three stages take 72 KB.  Step s multiplies the B of stage
// s while it reads and splits the A rows of stage s + 1; its copies bring the B of stage s + 2 into
// the place that step s - 1 left and the A of stage s + 3 into its own (its A rows were read a
// step ago), after the barrier that retires both, so a copy has a whole step to land.  The A rows
// run one step further ahead because mode 16 checks a row's shift once per 32-wide slab, on both of
// its halves, before it splits the first: the same shifts, and so the same bits, as the 128 x 128
// kernel's.  In mode 1 a stage is 16 KB and a step a third as long: five stages, and a copy has
// three steps.  A last column tile of 128 columns runs the same loop with four column blocks.
#include "gemm_split.h"

#include <algorithm>
#include <type_traits>

typedef __attribute__((address_space(3))) void* lds_ptr;

namespace {

using namespace tta_gemm;

constexpr int WM = 128, WN = 256, WK = 16, WTH = 256;  // tile, k step, threads
constexpr int NT = WN / 32;                            // 32-column blocks per tile

// 16-byte chunk c (of 4) of A row r in a stage, stored at c ^ wswz(r): 16 rows at one chunk cover
// all banks
__device__ __forceinline__ int wswz(int row) { return (row >> 2) & 3; }

template <int MODE>
__global__ __launch_bounds__(WTH, 2) void gemm_wide_kernel(GemmGroup g) {
  typedef Split<MODE> S;
  typedef typename Frag<S::F16>::T V8;
  constexpr int NA = S::NA, NB = S::NB;
  constexpr int A_CH = WM * 4, B_CH = NB * NT * 64, STG = A_CH + B_CH;  // 16-byte chunks
  constexpr int APT = A_CH / WTH, BPT = B_CH / WTH;
  constexpr int LDT = BN + 8;  // epilogue staging: 128 columns at a time
  constexpr int NST = MODE == 1 ? 5 : 3, NIF = APT + BPT;  // stages; copies per stage and thread
  constexpr int SMEM = NST * STG > WM * LDT / 4 ? NST * STG : WM * LDT / 4;
  __shared__ uint4 smem[SMEM];

  const GemmArgs& p = g.p[blockIdx.z];
  const int K = p.K, NT32 = g.NT32[blockIdx.z];
  const bool vec_ok = g.vec[blockIdx.z] != 0;
  const int t = threadIdx.x, lane = t & 63, l32 = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int tn = (p.N + WN - 1) / WN, ntiles = tn * ((p.M + WM - 1) / WM);
  // persistent tiles, an XCD's contiguous row-major range per block group (gemm_bf16.hip)
  const int gb = min(((ntiles + 7) / 8) * 8, g.cap);
  if ((int)blockIdx.x >= gb) return;
  const int per_xcd = (ntiles + 7) / 8, stride = gb / 8;
  const int t_end = min(((int)blockIdx.x % 8 + 1) * per_xcd, ntiles);
  int tile = ((int)blockIdx.x % 8) * per_xcd + (int)blockIdx.x / 8;
  if (tile >= t_end) return;

  // copies: per-lane byte offsets fixed for a tile, the k step in the scalar offset; rows past M and
  // column blocks past the packed weight get an offset past the buffer's end (copied as zeros)
  const __amdgpu_buffer_rsrc_t brsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.B), (short)0, 0x7ffffffe, 0x00020000);
  const int bstep = NB * NT32 * 2048;  // bytes of one packed 32-wide k slab
  int m0 = 0, n0 = 0;
  __amdgpu_buffer_rsrc_t arsrc;
  int avo[APT], bvo[BPT];
  auto set_tile = [&](int tl) {
    n0 = (tl % tn) * WN;
    m0 = (tl / tn) * WM;
    arsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.A + (int64_t)m0 * p.lda),
                                              (short)0, 0x7ffffffe, 0x00020000);
#pragma unroll
    for (int h = 0; h < APT; ++h) {
      const int L = t + WTH * h, r = L >> 2;
      avo[h] = r < p.M - m0 ? (r * (int)p.lda + 4 * ((L & 3) ^ wswz(r))) * 4 : (int)0x7fffffff;
    }
#pragma unroll
    for (int h = 0; h < BPT; ++h) {
      const int c = t + WTH * h, pl = c / (NT * 64), n32 = n0 / 32 + (c / 64) % NT;
      bvo[h] = n32 < NT32 ? (pl * NT32 + n32) * 2048 + (c % 64) * 16 : (int)0x7fffffff;
    }
  };
  auto issueA = [&](int s, int stg) {
    uint4* base = smem + stg * STG + 64 * wave;
#pragma unroll
    for (int h = 0; h < APT; ++h) {
      const int vo = avo[h];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(arsrc, (lds_ptr)(base + WTH * h), 16, vo, s * WK * 4,
                                               0, 0);
    }
  };
  auto issueB = [&](int s, int stg) {
    uint4* base = smem + stg * STG + 64 * wave;
#pragma unroll
    for (int h = 0; h < BPT; ++h) {
      const int vo = bvo[h];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(brsrc, (lds_ptr)(base + A_CH + WTH * h), 16, vo,
                                               (s >> 1) * bstep + (s & 1) * 1024, 0, 0);
    }
  };

  floatx16 acc[1][NT];
  const int rbase = wave * 32, row = rbase + l32;
  // this lane's eight k values of its row in a stage
  auto rdA = [&](int stg, floatx4 (&x)[1][2]) {
    const uint4* As = smem + stg * STG + row * 4;
    x[0][0] = __builtin_bit_cast(floatx4, As[(2 * lh) ^ wswz(row)]);
    x[0][1] = __builtin_bit_cast(floatx4, As[(2 * lh + 1) ^ wswz(row)]);
  };
  RowScale<1, NT, S::F16> rs;
  auto split = [&](const floatx4 (&x)[1][2], int sh, V8 (&a)[NA]) {
    if constexpr (S::F16)
      split8_f16<NA>(x[0][0], x[0][1], sh, a);
    else
      split8<NA>(x[0][0], x[0][1], a);
  };
  // the packed B fragments of column block pair (j, j + 1), and their products, smallest terms first
  auto rdB = [&](int stg, int j, V8 (&b)[2][NB]) {
    const uint4* Bs = smem + stg * STG + A_CH;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < NB; ++q)
        b[i][q] = __builtin_bit_cast(V8, Bs[(q * NT + j + i) * 64 + lane]);
  };
  auto mm = [&](const V8 (&a)[NA], const V8 (&b)[2][NB], int j) {
#pragma unroll
    for (int q = 0; q < S::NP; ++q)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        acc[0][j + i] = mfma32(a[S::pa[q]], b[i][S::pb[q]], acc[0][j + i]);
  };
  const int nks = K / WK;
  const int* Fc = reinterpret_cast<const int*>(static_cast<const uint4*>(p.B) +
                                               (int64_t)(K / BK) * NB * NT32 * 128);

  // the k loop over the first TJ column blocks.  A pair's fragments are read one pair ahead (the first
  // pair of a step during the last of the step before: its stage landed a barrier earlier); the
  // scheduling barriers keep the reads there
  auto next = [](int v) { return v == NST - 1 ? 0 : v + 1; };
  auto prev = [](int v) { return v == 0 ? NST - 1 : v - 1; };
  auto loop = [&](auto tj) {
    constexpr int TJ = decltype(tj)::value;
    floatx4 x[1][2], y[1][2];
    V8 a[NA], b[2][2][NB];
    rdA(0, x);
    rdA(1, y);
    rdB(0, 0, b[0]);
    rs.check(x, y, acc, lh);
    split(x, S::F16 && !rs.unscaled ? rs.er[0] : 0, a);
    int s = 0, stg = 0;
    // one step's copies, reads and products.  ODD: the next step opens a 32-wide slab, whose two
    // halves of A rows end up in x and y; the other steps take y into x.  FAST: the next step's rows
    // split for shift 0 in na and, ODD, the largest magnitude of this lane's in x and y in big
    V8 na[NA];
    float big = 0.f;
    auto take = [&](const floatx4 (&v)[1][2]) {
      big = max3_abs(v[0][0][0], v[0][0][1], big);
      big = max3_abs(v[0][0][2], v[0][0][3], big);
      big = max3_abs(v[0][1][0], v[0][1][1], big);
      big = max3_abs(v[0][1][2], v[0][1][3], big);
    };
    auto step = [&](auto fast, auto odd) {
      constexpr bool LOOK = S::F16 && decltype(fast)::value && decltype(odd)::value;
      const int s1 = next(stg);
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NST - 3) * NIF) : "memory");
      issueB(min(s + NST - 1, nks - 1), prev(stg));
      issueA(min(s + NST, nks - 1), stg);
      if constexpr (decltype(odd)::value) {
        rdA(s1, x);
      } else {
        x[0][0] = y[0][0];
        x[0][1] = y[0][1];
      }
#pragma unroll
      for (int j = 0; j < TJ; j += 2) {
        if (j + 2 < TJ)
          rdB(stg, j + 2, b[(j / 2 + 1) & 1]);
        else
          rdB(s1, 0, b[(j / 2 + 1) & 1]);
        if (decltype(odd)::value && j == TJ - 2) rdA(next(s1), y);
        __builtin_amdgcn_sched_barrier(0);
        mm(a, b[(j / 2) & 1], j);
        if (decltype(fast)::value && j == TJ - 4) {
          split(x, 0, na);
          if constexpr (LOOK) {
            big = 0.f;
            take(x);
          }
        }
      }
      if constexpr (LOOK) take(y);
      stg = s1;
      ++s;
    };
    using std::false_type;
    using std::true_type;
    auto keep = [&]() {
#pragma unroll
      for (int q = 0; q < NA; ++q) a[q] = na[q];
    };
    // (K is a multiple of 32: an even number of steps.)  Every row's shift 0: no branch between the
    // multiplications and the next split, and a new shift is needed only where a value reaches
    // 2^15, which each lane can tell of its own
    if (!S::F16 || rs.all_zero()) {
      while (s < nks) {
        step(true_type{}, false_type{});
        keep();
        step(true_type{}, true_type{});
        keep();
        if (S::F16 && __any(!(big < 32768.f))) {
          rdA(stg, x);
          rs.check(x, y, acc, lh);
          split(x, rs.er[0], a);
          if (!rs.unscaled) break;
        }
      }
    }
    while (s < nks) {
      step(false_type{}, false_type{});
      split(x, S::F16 && !rs.unscaled ? rs.er[0] : 0, a);
      step(false_type{}, true_type{});
      rs.check(x, y, acc, lh);
      split(x, S::F16 && !rs.unscaled ? rs.er[0] : 0, a);
    }
  };

  set_tile(tile);
  issueA(0, 0);
  issueB(0, 0);
  for (;;) {
    const int cm0 = m0, cn0 = n0;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][j][r] = 0.f;
    rs = RowScale<1, NT, S::F16>();
    issueA(min(1, nks - 1), 1);
#pragma unroll
    for (int q = 1; q < NST - 1; ++q) {
      issueB(min(q, nks - 1), q);
      issueA(min(q + 1, nks - 1), q + 1);
    }
    // stage 0 and the A rows of stage 1 landed (with everything issued before them); the later
    // copies may still be in flight
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NST - 2) * NIF) : "memory");
    const bool whole = cn0 + BN < p.N;  // more than 128 columns in this tile
    if (whole)
      loop(std::integral_constant<int, NT>{});
    else
      loop(std::integral_constant<int, NT / 2>{});
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if constexpr (S::F16) {
      int fc[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) fc[j] = Fc[min(cn0 + j * 32, NT32 * 32 - 32) + l32];
      rs.undo(acc, fc, lh);
    }
    float* Ct = reinterpret_cast<float*>(smem);
    const bool mfull = cm0 + WM <= p.M;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // 128 columns at a time, the rows' loads batched in mode 1 too (232 registers: 30,011 x 1024 x
      // 1024 with the SiLU-gradient epilogue 113 -> 102 us, 60,000 rows 293 -> 243, when it was made;
      // the 128 x 128 kernel in mode 1 loses 3-8 % on its other epilogues with the registers that
      // takes)
      if (h == 1 && !whole) break;
#pragma unroll
      for (int j = 0; j < NT / 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          Ct[(rbase + acc_row(r, lh)) * LDT + j * 32 + l32] = acc[0][h * (NT / 2) + j][r];
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      const int c0 = cn0 + h * BN;
      const bool full = mfull && c0 + BN <= p.N;
      switch (p.epi) {
        case EPI_SILU:
          epilogue_rows<EPI_SILU, true>(p, Ct, LDT, WM, cm0, c0, t, WTH, vec_ok, full);
          break;
        case EPI_ACCUM:
          epilogue_rows<EPI_ACCUM, true>(p, Ct, LDT, WM, cm0, c0, t, WTH, vec_ok, full);
          break;
        case EPI_PRE_SILU:
          epilogue_rows<EPI_PRE_SILU, true>(p, Ct, LDT, WM, cm0, c0, t, WTH, vec_ok, full);
          break;
        case EPI_SILU_GRAD:
          epilogue_rows<EPI_SILU_GRAD, true>(p, Ct, LDT, WM, cm0, c0, t, WTH, vec_ok, full);
          break;
        case EPI_SIGMOID:
          epilogue_rows<EPI_SIGMOID, true>(p, Ct, LDT, WM, cm0, c0, t, WTH, vec_ok, full);
          break;
        case EPI_GATE:
          epilogue_rows<EPI_GATE, true>(p, Ct, LDT, WM, cm0, c0, t, WTH, vec_ok, full, &g.gate,
                                          g.gc0[blockIdx.z]);
          break;
        case EPI_GATE_BWD:
          epilogue_rows<EPI_GATE_BWD, true>(p, Ct, LDT, WM, cm0, c0, t, WTH, vec_ok, full,
                                              &g.gate, g.gc0[blockIdx.z]);
          break;
        default:
          epilogue_rows<EPI_STORE, true>(p, Ct, LDT, WM, cm0, c0, t, WTH, vec_ok, full);
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    tile += stride;
    if (tile >= t_end) break;
    set_tile(tile);
    issueA(0, 0);
    issueB(0, 0);
  }
}

}  // namespace

namespace tta_gemm {

// Whether a launch takes the wide tile: mode 16 or 1, whole 32-wide k slabs, at least one whole
// column tile per product.  Mode 16 also needs 3072 k columns of tiles per resident workgroup: from
// there on the uneven last round of the larger tiles costs at most 1 %, below it decides by how
// that round happens to fill.  And where a product's last column tile is at most half full, an
// average K of at least 512 (the half tile's prologue and epilogue are not halved): conv-2 group
// (384 x 384, 512 x 512, 256 x 256) of 110,000 / 150,000 / 204,800 rows 476 -> 484 / 549 -> 561 / 745
// -> 748 us, its 384 columns alone 238 -> 261 at 204,800 rows; 640 columns at K = 768 683 -> 650.
// Measured, 128 x 128 -> 128 x 256 (us; M x N x K, k columns): 196,555
// x 1024 x 1024 (12,288) with the two-output epilogue 1460 -> 1350, with the SiLU-gradient one 1432
// -> 1337; 61,440 rows, conv-1 group (4560) 461 -> 438, its adjoint (4200) 484 -> 470; 90,000 x 640
// x 768 (3168) 285 -> 286; 50,000 x 1024 x 1024 (3128) 362 -> 341; 196,555 x 1024 x 256 (3072) 559 ->
// 546, x 256 x 1024 (3072) 339 -> 320.  Below the line, 45,000 x 1024 x 1024 (2816) 314 -> 316,
// 180,000 x 256 x 1024 (2814) 315 -> 307, 80,000 x 640 x 768 (2812) 246 -> 262, 40,000 x 1024 x 1024
// (2504) 297 -> 267, conv-2 group of 80,000 rows (2500) 288 -> 299 and of 61,440 (1920) 219 -> 231,
// 61,440 x 640 x 768 (2160) 198 -> 195, 10,150 x 1024 x 1024 (640) 86 -> 97.
//
// Mode 1 has a third of the products per copied byte, so its gain hangs on whole rounds of
// resident workgroups rather than on the work in all: it takes the wide tile where that makes
// five rounds or fewer out of eight of the 128 x 128 kernel's, at an average K of at least 384.
// Measured, 128 x 128 -> 128 x 256 (us): 30,011 x 1024 x 1024 (4 rounds -> 2) with the two-output
// epilogue 135 -> 112, with the SiLU-gradient one 170 -> 135; 61,440 rows (8 -> 4), conv-1 group
// 303 -> 260, its adjoint 346 -> 285; 12,000 x 768 x 640 (2 -> 1) 38 -> 31.  Below the line the gain
// is 0 to 7 %: 20,000 x 1024 x 512 (3 -> 2) 46 -> 44, 8,000 x 1024 x 1024 (1 -> 1) 29 -> 28, 30,011 x
// 256 x 1024 (1 -> 1) 28.5 -> 28.5, 60,000 x 1024 at K = 256 / 128 (8 -> 4) 81 -> 77 / 63 -> 60.
// (Drawn when those were losses of 5 to 20 %, before the epilogue's loads went out in batches.)
bool wide_ok(const GemmGroup& g, int n, int mode, int cap) {
  if (mode != 16 && mode != 1) return false;
  int64_t cols = 0, wide = 0, tiles = 0;
  bool half = false;
  for (int i = 0; i < n; ++i) {
    const GemmArgs& p = g.p[i];
    if (p.K % BK != 0 || p.K < 2 * BK || p.N < WN) return false;
    const int64_t rows = tta_blocks(p.M, WM), w = rows * tta_blocks(p.N, WN);
    wide += w;
    tiles += rows * tta_blocks(p.N, BN);
    cols += w * p.K;
    half = half || (p.N % WN > 0 && p.N % WN <= BN);
  }
  if (mode == 16) return cols >= (int64_t)3072 * cap && (!half || cols >= 512 * wide);
  const auto rounds = [&](int64_t c) { return (c + cap - 1) / cap; };
  return cols >= 384 * wide && 5 * rounds(tiles) >= 8 * rounds(wide);
}

int launch_wide(GemmGroup& g, int n, int mode, int cap, hipStream_t s) {
  int64_t grid = 0;
  g.cap = cap;
  for (int i = 0; i < n; ++i) {
    const int64_t ntiles = (int64_t)tta_blocks(g.p[i].N, WN) * tta_blocks(g.p[i].M, WM);
    if (ntiles > (1ll << 30)) {
      tta::set_error("tta_gemm_bf16x: grid too large");
      return tta::kBadArgument;
    }
    grid = std::max(grid, std::min<int64_t>(((ntiles + 7) / 8) * 8, g.cap));
  }
  const auto kern = mode == 1 ? gemm_wide_kernel<1> : gemm_wide_kernel<16>;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid, 1, (unsigned)n), dim3(WTH), 0, s, g);
  TTA_CHECK_LAUNCH("tta_gemm_bf16x");
  return tta::kOk;
}

}  // namespace tta_gemm
