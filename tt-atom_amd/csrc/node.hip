// Fused node-level kernels of the eSCN-MD step (uma-s-1: spectral feed-forward), one launch per
// stage instead of a chain of small ones:
//
//   k_spectral_block_fwd   x2 = x1 + SpectralAtomwise(RMSNormSH_2(x1))          (model.py:158-172,
//                          norm.py:93-111, spectral.py:146-188), optionally followed by the next
//                          RMSNormSH (the next block's norm_1 with the system embedding added to
//                          coefficient 0, or the final norm): 6 launches -> 1 per block
//   k_spectral_block_bwd   the reverse: the next norm's backward plus the residual adjoint, then
//                          the spectral FF and norm_2 backward (forces.py:49-98, 258-346) plus the
//                          residual: 6 -> 1 per block
//   k_energy_head_fwd      per-node energy MLP on coefficient 0 (model.py:223-235)
//   k_energy_head_bwd      its adjoint seeded with dE/dnode_e = 1 (forces.py:438-461)
//
// A spectral workgroup owns T = 2, 4, 8 or 16 nodes.  Their rows live in LDS grouped by degree
// (Pack<T>: the (2 l + 1) T rows of degree l, padded to whole 16-row tiles; row stride C + 4 floats:
// the 16 rows of an MFMA A fragment then fall in distinct banks), and every product is a matrix
// product of one degree's rows with that degree's weight on the fp32 matrix cores
// (v_mfma_f32_16x16x4_f32), the weight read from global memory (shared by every workgroup, it
// stays in L2).  Lane l supplies A[l%16][l/16] and B[l/16][l%16]; the result D[4*(l/16)+r][l%16]
// lands in accumulator element r.  Each wave owns whole 16-column output tiles for every row, so
// the gate's per-degree sums over coefficients stay inside a wavefront.  Per-node norms run one
// wavefront per node (64 lanes x 2 channels).  The energy head's workgroups own NT = 16 nodes (one
// row each).
//
// What bounds a spectral block: up to a few thousand nodes the chain inside one workgroup (load,
// norm, three products that each stream a weight, norm), not a rate of the chip.  Nine 16-node
// tiles cost 9 x 128 MFMAs per product and wavefront however few nodes they hold; packed by degree,
// two nodes take 3 tiles, four 4, eight 6.  T is the smallest with one workgroup per compute unit
// (pick_nodes), and each product's first weights are loaded a phase ahead.  Per launch, forward /
// backward, one coefficient per 16-row tile -> packed: 24 nodes 42.4 / 43.3 -> 22.8 / 26.3 us; 256
// nodes 44.8 / 44.4 -> 24.0 / 27.1; 1000 nodes 45.4 / 49.1 -> 29.9 / 35.4; 2048 nodes 49.7 / 52.6 ->
// 40.4 / 44.2.
//
// Requirements (checked on the host): C and H multiples of 16, at most 128; lmax = 2.
#include "common.h"

#include <atomic>

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int NT = 16;        // nodes per energy-head workgroup, rows of an MFMA tile
constexpr int NW = 8;         // waves per workgroup
constexpr int NTH = 64 * NW;
constexpr int CMAX = 128;     // largest C / H
constexpr int LDP = CMAX + 4; // LDS row stride (floats) of the [coef][node][channel] buffer
static_assert(CMAX / 16 <= NW, "one output column tile per wave");

__device__ __forceinline__ int ndeg(int j) { return j == 0 ? 0 : (j < 4 ? 1 : 2); }
__device__ __forceinline__ float nbdw(int j) {
  const int l = ndeg(j);
  return (float)(1.0 / (2 * l + 1) / 3.0);
}
__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Rows of T nodes grouped by degree: tiles [first(l), first(l + 1)) of 16 rows hold degree l, its
// coefficient m (c = l^2 + m) of node n in row m T + n.  T divides 16, so row 4 q + e of any tile is
// a row of node (4 q + e) % T.
template <int T>
struct Pack {
  static_assert(16 % T == 0, "");
  static constexpr int T1 = (3 * T + 15) / 16, T2 = (5 * T + 15) / 16, TILES = 1 + T1 + T2;
  static __device__ constexpr int first(int l) { return l == 0 ? 0 : l == 1 ? 1 : 1 + T1; }
  static __device__ constexpr int deg(int tile) { return tile < 1 ? 0 : tile < 1 + T1 ? 1 : 2; }
  static __device__ __forceinline__ int row(int c, int n) {
    const int l = ndeg(c);
    return 16 * first(l) + (c - l * l) * T + n;
  }
  // coefficient of row 4 q + e of a tile, and whether the row is one (not padding)
  static __device__ __forceinline__ int coef(int tile, int qe) {
    const int l = deg(tile);
    return l * l + ((tile - first(l)) * 16 + qe) / T;
  }
  static __device__ __forceinline__ bool used(int tile, int qe) {
    const int l = deg(tile);
    return ((tile - first(l)) * 16 + qe) / T < 2 * l + 1;
  }
};
// a * b, rounded: never contracted into an addition
__device__ __forceinline__ float rounded_product(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}

// A degree's sum over its 2 l + 1 coefficients m of one node and column, p_0 .. p_2l, as
// ((p_0 + p_4) + p_1) + (p_2 + p_3) for every T, so that a node's bits do not depend on how many
// nodes share the launch.  v: this lane's rows of the degree's tiles (zero in padding rows), row
// 4 q + e of tile i in v[i][e]: coefficient 16 / T i + (4 q + e) / T of node (4 q + e) % T.  s[e] is
// complete in the lane whose row 4 q + e is below T.
template <int T, int NT_>
__device__ __forceinline__ void degree_sum(const float (&v)[NT_][4], float (&s)[4]) {
  constexpr int E = T < 4 ? T : 4;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    if (T == 16) {
      const float a = NT_ > 3 ? v[0][e] + v[NT_ - 1][e] : v[0][e];
      const float b = NT_ > 3 ? v[2][e] + v[NT_ > 3 ? 3 : 0][e] : v[2][e];
      s[e] = (a + v[1][e]) + b;
    } else if (T == 8) {  // lanes q, q + 2: even and odd coefficients
      const float a = NT_ > 2 ? v[0][e] + v[NT_ - 1][e] : v[0][e];
      const float o0 = __shfl_xor(v[0][e], 32), o1 = __shfl_xor(v[1][e], 32);
      s[e] = (a + o0) + (v[1][e] + o1);
    } else if (T == 4) {  // lane q: coefficients q and q + 4
      float a = NT_ > 1 ? v[0][e] + v[NT_ - 1][e] : v[0][e];
      a += __shfl_xor(a, 16);
      s[e] = a + __shfl_xor(a, 32);
    } else {  // T = 2, lane q: coefficients 2 q (rows e) and 2 q + 1 (rows e + 2)
      float a = v[0][e] + __shfl_xor(v[0][e], 32);
      a += v[0][e + 2];
      s[e] = a + __shfl_xor(a, 16);
    }
  }
}

// one row tile with the degree 0 weight (the scalar products)
struct Scalar {
  static constexpr int TILES = 1;
  static __device__ constexpr int deg(int) { return 0; }
};

// LDS row of (coefficient c, local node n)
template <int T>
__device__ __forceinline__ float* lrow(float* buf, int c, int n) {
  return buf + Pack<T>::row(c, n) * LDP;
}

// One product acc[i][jj] += X tile i (16 x K, LDS rows at stride ldx) @ W[deg(i)] (K x ncol,
// row-major at ldw, per-degree stride dstride) for JT 16-column tiles per wave: tile
// (wave + NW jj) % (ncol / 16) at column offset jj cstep.  (A wave whose tile is past the last one,
// narrow layers only, recomputes a valid tile and its caller discards the result, so the inner
// loop has no branches.)  K runs in chunks of 16: in MFMA step s of a chunk, slot q (= lane / 16) of
// both operands is k = k0 + 4 q + s, so a lane reads its A values of a chunk as one float4 from
// LDS.  The B values arrive D chunks at a time (K a multiple of 16 D), two groups in flight; they do
// not depend on the rows, so start() is called a phase ahead (before a norm, a gate or a barrier)
// and the product finds its first groups landed.
template <class P, int D, int JT>
struct Product {
  static constexpr int NC = P::TILES, NL = NC > 1 ? 3 : 1, G = 16 * D;
  const float* W;
  int ldw, K;
  unsigned off[NL][JT];  // 32-bit element offsets from the (wave-uniform) weight base
  float b0[D][4][NL][JT], b1[D][4][NL][JT];

  __device__ __forceinline__ void load(float (&b)[D][4][NL][JT], int k0) const {
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int l = 0; l < NL; ++l)
#pragma unroll
          for (int jj = 0; jj < JT; ++jj)
            b[d][s][l][jj] = W[off[l][jj] + (unsigned)((k0 + 16 * d + s) * ldw)];
  }
  __device__ __forceinline__ void start(const float* __restrict__ W_, int64_t dstride, int ldw_,
                                        int K_, int ncol, int cstep, int wave, int lane) {
    W = W_;
    ldw = ldw_;
    K = K_;
    const int ntile = ncol / 16;
#pragma unroll
    for (int l = 0; l < NL; ++l)
#pragma unroll
      for (int jj = 0; jj < JT; ++jj)
        off[l][jj] = (unsigned)(l * dstride + jj * cstep + (wave % ntile) * 16 + (lane & 15) +
                                4 * (lane >> 4) * ldw);
    load(b0, 0);
    if (G < K) load(b1, G);
  }
  __device__ __forceinline__ void mul(const float (&b)[D][4][NL][JT], const float* xr, int ldx,
                                      int g0, floatx4 (&acc)[NC][JT]) const {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      floatx4 a[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c)
        a[c] = *reinterpret_cast<const floatx4*>(xr + c * 16 * ldx + g0 + 16 * d);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int jj = 0; jj < JT; ++jj)
            acc[c][jj] = mfma4(a[c][s], b[d][s][P::deg(c)][jj], acc[c][jj]);
    }
  }
  __device__ __forceinline__ void run(const float* X, int ldx, int lane, floatx4 (&acc)[NC][JT]) {
    const float* xr = X + (lane & 15) * ldx + 4 * (lane >> 4);
    for (int g0 = 0; g0 < K; g0 += 2 * G) {
      mul(b0, xr, ldx, g0, acc);
      if (g0 + 2 * G < K) load(b0, g0 + 2 * G);
      if (g0 + G >= K) break;
      mul(b1, xr, ldx, g0 + G, acc);
      if (g0 + 3 * G < K) load(b1, g0 + 3 * G);
    }
  }
};

template <int NC, int JT>
__device__ __forceinline__ void zero_acc(floatx4 (&acc)[NC][JT]) {
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int jj = 0; jj < JT; ++jj) acc[c][jj] = floatx4{0.f, 0.f, 0.f, 0.f};
}

// RMSNormSH forward of one node's 9 x C rows (norm.py:93-111): centre coefficient 0 over the
// channels, ms = mean_c sum_j bdw_j xc_j^2, inv = rsqrt(ms + eps), y = xc * inv * aw[l(j)],
// y[0] += ab (+ add0).  xr(j) / yr(j): the node's input and output rows.  One wavefront; lane
// handles channels lane, lane + 64.
template <class XR, class YR>
__device__ __forceinline__ float rms_fwd_node(XR xr, YR yr, const float* __restrict__ aw,
                                              const float* __restrict__ ab,
                                              const float* __restrict__ add0row, int C,
                                              int lane, float eps) {
  float s0 = 0.f;
  for (int c = lane; c < C; c += 64) s0 += xr(0)[c];
  const float mu = tta_group_sum(s0, 64) / C;
  float ms = 0.f;
  for (int c = lane; c < C; c += 64) {
    float sc = 0.f;
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      const float v = j == 0 ? xr(0)[c] - mu : xr(j)[c];
      sc += v * v * nbdw(j);
    }
    ms += sc;
  }
  ms = tta_group_sum(ms, 64) / C;
  const float inv = 1.0f / sqrtf(ms + eps);
  for (int c = lane; c < C; c += 64) {
    float v[9];
#pragma unroll
    for (int j = 0; j < 9; ++j) v[j] = j == 0 ? xr(0)[c] - mu : xr(j)[c];
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      float o = v[j] * (inv * aw[ndeg(j) * C + c]);
      if (j == 0) {
        o = o + ab[c];
        if (add0row) o = o + add0row[c];
      }
      yr(j)[c] = o;
    }
  }
  return inv;
}

// RMSNormSH backward of one node (forces.py:73-98): gx = g inv aw + xc bdw gms 2/C, minus the
// channel mean on coefficient 0.  gv(j, hh) / xv(j, hh) give the adjoint and the input of
// coefficient j at channel lane + 64 hh (registers or LDS, as the caller holds them); the
// results for those channels are returned in out[9][2].  The sums run over the lane's channels
// in order, then across the wavefront.  The fused steps are spelled out: which of two products the
// compiler contracts into their sum differs between the numbers of nodes per workgroup.
template <class GV, class XV>
__device__ __forceinline__ void rms_bwd_vals(GV gv, XV xv, const float* __restrict__ aw,
                                             float inv, int C, int lane, float (&out)[9][2]) {
#pragma clang fp contract(off)
  float s0 = 0.f;
#pragma unroll
  for (int hh = 0; hh < 2; ++hh)
    if (lane + 64 * hh < C) s0 += xv(0, hh);
  const float mu = tta_group_sum(s0, 64) / C;
  float ginv = 0.f;
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
    const int c = lane + 64 * hh;
    if (c >= C) continue;
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      const float v = j == 0 ? xv(0, hh) - mu : xv(j, hh);
      ginv = fmaf(gv(j, hh) * v, aw[ndeg(j) * C + c], ginv);
    }
  }
  ginv = tta_group_sum(ginv, 64);
  const float gms = ginv * (inv * inv * inv) * -0.5f;
  float s1 = 0.f;
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
    const int c = lane + 64 * hh;
    if (c >= C) continue;
    const float v = xv(0, hh) - mu;
    s1 += fmaf(gv(0, hh), inv * aw[c], v * nbdw(0) * gms * (2.0f / C));
  }
  const float m0 = tta_group_sum(s1, 64) / C;
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
    const int c = lane + 64 * hh;
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      float gx = 0.f;
      if (c < C) {
        const float v = j == 0 ? xv(0, hh) - mu : xv(j, hh);
        gx = fmaf(gv(j, hh), inv * aw[ndeg(j) * C + c], v * nbdw(j) * gms * (2.0f / C));
        if (j == 0) gx -= m0;
      }
      out[j][hh] = gx;
    }
  }
}

// T nodes of a [N, 9, C] tensor into the Pack<T> LDS rows, one wavefront per (node, coefficient)
// row (wave-uniform indices, no per-element division); rows of absent nodes are zero.  (Padding
// rows are left as they are: a row of an MFMA operand reaches only its own output row.)
template <int T>
struct NodeRows {
  static constexpr int RPW = (9 * T + NW - 1) / NW;  // rows per wave
  float v[RPW][2];
  __device__ __forceinline__ void load(const float* __restrict__ x, int64_t n0, int nv, int C,
                                       int wave, int lane) {
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const int rc = wave + NW * i, rr = rc / 9, c = rc - 9 * rr;
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int ch = lane + 64 * hh;
        v[i][hh] = (rr < nv && ch < C) ? x[((n0 + rr) * 9 + c) * C + ch] : 0.f;
      }
    }
  }
  __device__ __forceinline__ void store(float* buf, int C, int wave, int lane) const {
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const int rc = wave + NW * i, rr = rc / 9, c = rc - 9 * rr;
      if (rr >= T) continue;
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int ch = lane + 64 * hh;
        if (ch < C) lrow<T>(buf, c, rr)[ch] = v[i][hh];
      }
    }
  }
};

struct SpecFwdArgs {
  const float* x1;                        // [N, 9, C] block state after the edgewise residual
  const float *aw2, *ab2;                 // norm_2 [3, C], [C]
  const float *ws_t, *bs;                 // scalar MLP [C, 2H], [2H]
  const float *w1t, *b1;                  // SO3_Linear_1 per degree [3, C, H], bias [H] (l = 0)
  const float *w2t, *b2;                  // SO3_Linear_2 per degree [3, H, C], bias [C] (l = 0)
  float *inv2, *a_s, *h;                  // saved: [N], [N, 2H] (pre-SiLU), [N, 9, H] (pre-gate)
  float* x2;                              // [N, 9, C] = x1 + FF
  const float *awn, *abn, *add0;          // next norm (may be null): [3, C], [C], [N, C] or null
  float *yn, *invn;                       // next norm output [N, 9, C], [N]
  int64_t N;
  int C, H;
  float eps;
};

template <int T, int D>
__global__ __launch_bounds__(NTH, 1) void k_spectral_block_fwd(SpecFwdArgs p) {
  typedef Pack<T> P;
  __shared__ float buf[P::TILES * 16 * LDP];
  __shared__ float gat[T * (2 * CMAX + 4)];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int C = p.C, H = p.H, LH = 2 * H, ldg = 2 * CMAX + 4;
  const int64_t n0 = (int64_t)blockIdx.x * T;
  const int nv = (int)min((int64_t)T, p.N - n0);
  const int r = lane & 15, q = lane >> 4;
  const bool hok = wave < H / 16, cok = wave < C / 16;  // this wave owns a column tile
  const int col = wave * 16 + r;
  // 1. x1 rows -> LDS (rows of absent nodes zero)
  NodeRows<T> rows;
  rows.load(p.x1, n0, nv, C, wave, lane);
  Product<Scalar, D, 2> scal;
  scal.start(p.ws_t, 0, LH, C, H, H, wave, lane);
  Product<P, D, 1> lin;
  lin.start(p.w1t, (int64_t)C * H, H, C, H, 0, wave, lane);
  rows.store(buf, C, wave, lane);
  __syncthreads();
  // 2. norm_2 in place, one wave per node
  for (int rr = wave; rr < nv; rr += NW) {
    auto row = [&](int j) { return lrow<T>(buf, j, rr); };
    const float inv = rms_fwd_node(row, row, p.aw2, p.ab2, nullptr, C, lane, p.eps);
    if (lane == 0) p.inv2[n0 + rr] = inv;
  }
  __syncthreads();
  // 3. scalar MLP on coefficient 0: a_s = n2_0 @ ws_t + bs (saved), gating = silu(a_s) -> LDS; this
  //    wave's column tile of both H halves
  floatx4 as[1][2];
  zero_acc(as);
  scal.run(buf, LDP, lane, as);
  // 4. h = n2 @ w1t[l] (+ b1 on coefficient 0)
  floatx4 acc[P::TILES][1];
  zero_acc(acc);
  lin.run(buf, LDP, lane, acc);
  lin.start(p.w2t, (int64_t)H * C, C, H, C, 0, wave, lane);
  if (hok) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const float bias = p.bs[half * H + col];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 4 * q + e;
        const float a = as[0][half][e] + bias;
        if (row < nv) p.a_s[(n0 + row) * LH + half * H + col] = a;
        if (row < T) gat[row * ldg + half * H + col] = tta_silu(a);
      }
    }
  }
  __syncthreads();  // every wave is done reading n2; gating is complete
  // 5. h saved; gout = gate(h) -> LDS (natural order: l = 1 rows gate block 0, l = 2 block 1);
  //    the gate values sigmoid(gating) once per (node, degree, channel)
  if (hok) {
    float sig[2][4];
#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        sig[l][e] = tta_sigmoid_acc(gat[(4 * q + e) % T * ldg + l * H + col]);
    const float b1 = p.b1[col];
#pragma unroll
    for (int i = 0; i < P::TILES; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = (4 * q + e) % T;
        const float v = acc[i][0][e] + (i == 0 ? b1 : 0.f);
        if (n < nv && P::used(i, 4 * q + e))
          p.h[((n0 + n) * 9 + P::coef(i, 4 * q + e)) * H + col] = v;
        const float g = i == 0 ? tta_silu(v) : v * sig[P::deg(i) == 2][e];
        buf[(16 * i + 4 * q + e) * LDP + col] = g;
      }
  }
  // the residual's x1 values, for step 6: they arrive during the product
  float xr[P::TILES][4];
#pragma unroll
  for (int i = 0; i < P::TILES; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int n = (4 * q + e) % T;
      xr[i][e] = cok && n < nv && P::used(i, 4 * q + e)
                     ? p.x1[((n0 + n) * 9 + P::coef(i, 4 * q + e)) * C + col]
                     : 0.f;
    }
  __syncthreads();
  // 6. out = x1 + gout @ w2t[l] (+ b2 on coefficient 0)
  zero_acc(acc);
  lin.run(buf, LDP, lane, acc);
  if (p.awn) __syncthreads();  // the next norm reuses the buffer for x2
  if (cok) {
    const float b2 = p.b2[col];
#pragma unroll
    for (int i = 0; i < P::TILES; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = (4 * q + e) % T;
        const float v = acc[i][0][e] + (i == 0 ? b2 : 0.f) + xr[i][e];
        if (n < nv && P::used(i, 4 * q + e))
          p.x2[((n0 + n) * 9 + P::coef(i, 4 * q + e)) * C + col] = v;
        if (p.awn) buf[(16 * i + 4 * q + e) * LDP + col] = v;
      }
  }
  if (!p.awn) return;
  __syncthreads();
  // 7. the next RMSNormSH on x2 (coefficient 0 + the system embedding when given)
  for (int rr = wave; rr < nv; rr += NW) {
    const int64_t n = n0 + rr;
    const float inv = rms_fwd_node([&](int j) { return lrow<T>(buf, j, rr); },
                                   [&](int j) { return p.yn + (n * 9 + j) * C; }, p.awn, p.abn,
                                   p.add0 ? p.add0 + n * C : nullptr, C, lane, p.eps);
    if (lane == 0) p.invn[n] = inv;
  }
}

struct SpecBwdArgs {
  const float *g_n, *x2, *awn, *invn;     // next norm: output adjoint, input, weight, inv
  const float* res;                       // residual adjoint added to g_x2 (may be null)
  const float *x1, *aw2, *inv2, *a_s, *h; // this block's saved forward terms
  const float *w1, *w2, *ws;              // per degree [3, H, C], [3, C, H]; scalar [2H, C]
  float* g_x1;                            // [N, 9, C]
  int64_t N;
  int C, H;
};

template <int T, int D>
__global__ __launch_bounds__(NTH, 1) void k_spectral_block_bwd(SpecBwdArgs p) {
  typedef Pack<T> P;
  constexpr int NS = (T + NW - 1) / NW;   // nodes per wave in the per-node phases
  __shared__ float buf[P::TILES * 16 * LDP];
  __shared__ float gas[NT * (2 * CMAX + 4)];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int C = p.C, H = p.H, LH = 2 * H, ldg = 2 * CMAX + 4;
  const int64_t n0 = (int64_t)blockIdx.x * T;
  const int nv = (int)min((int64_t)T, p.N - n0);
  const int r = lane & 15, q = lane >> 4;
  const bool hok = wave < H / 16, cok = wave < C / 16;  // this wave owns a column tile
  const int col = wave * 16 + r;
  // 1. g_x2 = next-norm backward (+ res), one wave per node; kept in registers for step 5 and
  //    written to LDS as the FF's output adjoint (absent nodes: zero rows).  The x2 tile comes
  //    into LDS by coalesced rows; each wave's g_n values (its nodes wave + NW s, channels
  //    lane + 64 hh) go straight to registers, all loads in flight together.
  float gx2[NS][9][2];
  // values of a [N, 9, C] tensor at this wave's nodes and channels (0 outside)
  auto node_vals = [&](const float* __restrict__ x, float (&v)[NS][9][2]) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const int rr = wave + NW * s, c = lane + 64 * hh;
        const bool in = rr < nv && c < C;
#pragma unroll
        for (int j = 0; j < 9; ++j) v[s][j][hh] = in ? x[((n0 + rr) * 9 + j) * C + c] : 0.f;
      }
  };
  {
    NodeRows<T> rows;
    rows.load(p.x2, n0, nv, C, wave, lane);
    node_vals(p.g_n, gx2);
    rows.store(buf, C, wave, lane);
  }
  Product<P, D, 1> lin;
  lin.start(p.w2, (int64_t)C * H, H, C, H, 0, wave, lane);
  __syncthreads();
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int rr = wave + NW * s;
    if (rr >= nv) {
      // an absent node's rows stay zero (its x2 rows were zero-filled above)
      continue;
    }
    float o[9][2];
    rms_bwd_vals([&](int j, int hh) { return gx2[s][j][hh]; },
                 [&](int j, int hh) { return lrow<T>(buf, j, rr)[lane + 64 * hh]; }, p.awn,
                 p.invn[n0 + rr], C, lane, o);
    const int64_t n = n0 + rr;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int c = lane + 64 * hh;
#pragma unroll
      for (int j = 0; j < 9; ++j) {
        gx2[s][j][hh] = o[j][hh] + ((p.res && c < C) ? p.res[(n * 9 + j) * C + c] : 0.f);
        if (c < C) lrow<T>(buf, j, rr)[c] = gx2[s][j][hh];   // this wave's own node rows
      }
    }
  }
  // this lane's saved forward values for step 3; they arrive during the product where its registers
  // leave room for them (T < 16)
  float hs[P::TILES][4], as[2][4];
  auto saved_vals = [&]() {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int nd = (4 * q + e) % T;
      const int64_t n = n0 + nd;
      const bool in = hok && nd < nv;
#pragma unroll
      for (int i = 0; i < P::TILES; ++i)
        hs[i][e] = in && P::used(i, 4 * q + e)
                       ? p.h[(n * 9 + P::coef(i, 4 * q + e)) * H + col]
                       : 0.f;
      as[0][e] = in ? p.a_s[n * LH + col] : 0.f;
      as[1][e] = in ? p.a_s[n * LH + H + col] : 0.f;
    }
  };
  if (T < 16) saved_vals();
  __syncthreads();
  // 2. g_gout = g_x2 @ w2[l]  ([C, H] per degree)
  floatx4 acc[P::TILES][1];
  zero_acc(acc);
  lin.run(buf, LDP, lane, acc);
  if (T == 16) saved_vals();
  lin.start(p.w1, (int64_t)H * C, C, H, C, 0, wave, lane);
  Product<Scalar, D, 1> scal;
  if (T < 16) scal.start(p.ws, 0, C, LH, C, 0, wave, lane);
  // 3. gate backward: g_h0 = g_gout0 silu'(h0); g_h_c = g_gout_c sig(gating); the degree sums
  //    sum_{c in l} g_gout_c h_c (this wave holds every row of its columns: degree_sum) give
  //    g_a_s = sum * sig'(gating) * silu'(a_s)
  __syncthreads();  // every wave is done reading g_x2
  if (hok) {
    float v1[P::T1][4], v2[P::T2][4], sum[2][4], sg[2][4];  // the degrees' terms, their sums
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sg[0][e] = tta_sigmoid_acc(tta_silu(as[0][e]));
      sg[1][e] = tta_sigmoid_acc(tta_silu(as[1][e]));
#pragma unroll
      for (int i = 0; i < P::TILES; ++i) {
        const float hv = hs[i][e], gg = acc[i][0][e];
        float gh;
        if (P::deg(i) == 0) {
          gh = gg * tta_silu_grad(hv);
        } else {
          const int l = P::deg(i) - 1;
          gh = gg * sg[l][e];
          const float pr = P::used(i, 4 * q + e) ? rounded_product(gg, hv) : 0.f;
          if (l == 0)
            v1[i - 1][e] = pr;
          else
            v2[i - 1 - P::T1][e] = pr;
        }
        buf[(16 * i + 4 * q + e) * LDP + col] = gh;
      }
    }
    degree_sum<T>(v1, sum[0]);
    degree_sum<T>(v2, sum[1]);
#pragma unroll
    for (int l = 0; l < 2; ++l) {
#pragma unroll
      for (int e = 0; e < (T < 4 ? T : 4); ++e) {
        if (4 * q + e < T)
          gas[(4 * q + e) * ldg + l * H + col] =
              sum[l][e] * sg[l][e] * (1.f - sg[l][e]) * tta_silu_grad(as[l][e]);
      }
    }
  }
  // the x1 values step 5 needs: they arrive during the products
  float x1v[NS][9][2];
  node_vals(p.x1, x1v);
  __syncthreads();
  // 4. g_n2 = g_h @ w1[l] ([H, C] per degree); coefficient 0 also + g_a_s @ ws ([2H, C]), the gas
  //    rows (stride ldg) as the A operand
  zero_acc(acc);
  lin.run(buf, LDP, lane, acc);
  {
    floatx4 acc0[1][1];
    zero_acc(acc0);
    if (T == 16) scal.start(p.ws, 0, C, LH, C, 0, wave, lane);
    scal.run(gas, ldg, lane, acc0);
    acc[0][0] += acc0[0][0];
  }
  __syncthreads();  // every wave is done reading g_h
  if (cok) {
#pragma unroll
    for (int i = 0; i < P::TILES; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) buf[(16 * i + 4 * q + e) * LDP + col] = acc[i][0][e];
  }
  __syncthreads();
  // 5. g_x1 = norm_2 backward of g_n2 (LDS) with x1 from the registers loaded before step 4,
  //    plus g_x2
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int rr = wave + NW * s;
    if (rr >= nv) continue;
    const int64_t n = n0 + rr;
    float gx[9][2];
    rms_bwd_vals([&](int j, int hh) { return lrow<T>(buf, j, rr)[lane + 64 * hh]; },
                 [&](int j, int hh) { return x1v[s][j][hh]; }, p.aw2, p.inv2[n], C, lane, gx);
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int c = lane + 64 * hh;
      if (c >= C) continue;
#pragma unroll
      for (int j = 0; j < 9; ++j) p.g_x1[(n * 9 + j) * C + c] = gx[j][hh] + gx2[s][j][hh];
    }
  }
}

// acc += X (16 rows, LDS stride LDP) @ W (K x ncol, row-major at ldw), one column tile per wave
__device__ __forceinline__ void scalar_product(const float* X, int K, const float* __restrict__ W,
                                               int ldw, int ncol, int wave, int lane,
                                               floatx4 (&acc)[1][1]) {
  if (K % 64 == 0) {
    Product<Scalar, 4, 1> m;
    m.start(W, 0, ldw, K, ncol, 0, wave, lane);
    m.run(X, LDP, lane, acc);
  } else {
    Product<Scalar, 1, 1> m;
    m.start(W, 0, ldw, K, ncol, 0, wave, lane);
    m.run(X, LDP, lane, acc);
  }
}

struct HeadArgs {
  const float* ne;                        // final-norm output [N, 9, C] (coefficient 0 read)
  const float *w0t, *b0, *w1t, *b1, *w2, *b2;  // [C, H], [H], [H, H], [H], [H] (output row), [1]
  const float *w0, *w1;                   // backward: [H, C], [H, H] (torch [out, in])
  float *a1, *a2, *node_e;                // saved pre-activations [N, H] x 2, energies [N]
  float* g_ne;                            // backward output [N, 9, C]
  int64_t N;
  int C, H;
  int npb;                                // nodes per workgroup, NT or NT / 2 (rows past it zero)
};

// Per-node energy MLP on coefficient 0: a1 = ne0 @ w0t + b0, s1 = silu(a1), a2 = s1 @ w1t + b1,
// s2 = silu(a2), e = s2 . w2 + b2.
__global__ __launch_bounds__(NTH, 1) void k_energy_head_fwd(HeadArgs p) {
  __shared__ float buf[NT * LDP];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int C = p.C, H = p.H;
  const int64_t n0 = (int64_t)blockIdx.x * p.npb;
  const int nv = (int)min((int64_t)p.npb, p.N - n0);
  for (int rr = wave; rr < NT; rr += NW)
    for (int ch = lane; ch < C; ch += 64)
      buf[rr * LDP + ch] = rr < nv ? p.ne[(n0 + rr) * 9 * C + ch] : 0.f;
  __syncthreads();
  const int r = lane & 15, q = lane >> 4;
  floatx4 acc[1][1];
  zero_acc(acc);
  scalar_product(buf, C, p.w0t, H, H, wave, lane, acc);
  __syncthreads();
  if (wave < H / 16) {
    const int col = wave * 16 + r;
    const float bias = p.b0[col];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 4 * q + e;
      const float a = acc[0][0][e] + bias;
      if (row < nv) p.a1[(n0 + row) * H + col] = a;
      buf[row * LDP + col] = tta_silu(a);
    }
  }
  __syncthreads();
  zero_acc(acc);
  scalar_product(buf, H, p.w1t, H, H, wave, lane, acc);
  __syncthreads();
  if (wave < H / 16) {
    const int col = wave * 16 + r;
    const float bias = p.b1[col];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 4 * q + e;
      const float a = acc[0][0][e] + bias;
      if (row < nv) p.a2[(n0 + row) * H + col] = a;
      buf[row * LDP + col] = tta_silu(a);
    }
  }
  __syncthreads();
  // e = s2 . w2 + b2: one wave per node, channels in order within each lane, then a butterfly
  for (int rr = wave; rr < nv; rr += NW) {
    float s = 0.f;
    for (int c = lane; c < H; c += 64) s += buf[rr * LDP + c] * p.w2[c];
    s = tta_group_sum(s, 64);
    if (lane == 0) p.node_e[n0 + rr] = s + p.b2[0];
  }
}

// dE/dnode_e = 1: g_a2 = w2 silu'(a2); g_a1 = (g_a2 @ w1) silu'(a1); g_ne0 = g_a1 @ w0; the
// other coefficients of g_ne are zero.
__global__ __launch_bounds__(NTH, 1) void k_energy_head_bwd(HeadArgs p) {
  __shared__ float buf[NT * LDP];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int C = p.C, H = p.H;
  const int64_t n0 = (int64_t)blockIdx.x * p.npb;
  const int nv = (int)min((int64_t)p.npb, p.N - n0);
  for (int rr = wave; rr < NT; rr += NW)
    for (int ch = lane; ch < H; ch += 64)
      buf[rr * LDP + ch] = rr < nv ? p.w2[ch] * tta_silu_grad(p.a2[(n0 + rr) * H + ch]) : 0.f;
  __syncthreads();
  const int r = lane & 15, q = lane >> 4;
  floatx4 acc[1][1];
  zero_acc(acc);
  scalar_product(buf, H, p.w1, H, H, wave, lane, acc);
  __syncthreads();
  if (wave < H / 16) {
    const int col = wave * 16 + r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 4 * q + e;
      buf[row * LDP + col] =
          row < nv ? acc[0][0][e] * tta_silu_grad(p.a1[(n0 + row) * H + col]) : 0.f;
    }
  }
  __syncthreads();
  zero_acc(acc);
  scalar_product(buf, H, p.w0, C, C, wave, lane, acc);
  if (wave < C / 16) {
    const int col = wave * 16 + r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 4 * q + e;
      if (row < nv) p.g_ne[(n0 + row) * 9 * C + col] = acc[0][0][e];
    }
  }
  for (int rr = wave; rr < nv; rr += NW)
    for (int k = lane; k < 8 * C; k += 64) p.g_ne[(n0 + rr) * 9 * C + C + k] = 0.f;
}

bool node_dims_ok(int64_t N, int C, int H) {
  return N >= 0 && N < (1ll << 31) / 9 / 128 && C >= 16 && C <= CMAX && C % 16 == 0 &&
         H >= 16 && H <= CMAX && H % 16 == 0;
}

}  // namespace

static int compute_units() {
  // queried once per device; atomics, since host threads calling the library at the same time may
  // both fill an entry (with the same value)
  static std::atomic<int> cus_of[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  int cus = cus_of[dev].load(std::memory_order_relaxed);
  if (cus == 0) {
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
      cus = 256;
    cus_of[dev].store(cus, std::memory_order_relaxed);
  }
  return cus;
}

// Nodes per energy-head workgroup: NT, or NT / 2 when NT-node workgroups would not cover the
// compute units (the MFMA tile keeps NT rows, those past the workgroup's nodes zero; the per-node
// phases halve and twice as many units work).
static int head_nodes(int64_t N) { return (N + NT - 1) / NT < compute_units() ? NT / 2 : NT; }

// Nodes per spectral workgroup: the fewest with at most one workgroup per compute unit.
static int pick_nodes(int64_t N) {
  for (int T = 2; T < 16; T *= 2)
    if ((N + T - 1) / T <= compute_units()) return T;
  return 16;
}

template <class Args>
static void launch_nodes(void (*kernel)(Args), int T, const Args& p, hipStream_t stream) {
  hipLaunchKernelGGL(kernel, dim3(tta_blocks(p.N, T)), dim3(NTH), 0, stream, p);
}

// The variant for p.N nodes; two chunks per weight group (Product's D) where the tiles of T nodes
// leave the registers for it, one at T = 16 and for widths that are no multiple of 32.
#define LAUNCH_SPECTRAL(kernel, p, stream)                                                        \
  do {                                                                                            \
    const int T_ = pick_nodes((p).N);                                                             \
    const bool d2_ = (p).C % 32 == 0 && (p).H % 32 == 0;                                          \
    if (T_ == 2)                                                                                  \
      d2_ ? launch_nodes(kernel<2, 2>, 2, p, stream) : launch_nodes(kernel<2, 1>, 2, p, stream);  \
    else if (T_ == 4)                                                                             \
      d2_ ? launch_nodes(kernel<4, 2>, 4, p, stream) : launch_nodes(kernel<4, 1>, 4, p, stream);  \
    else if (T_ == 8)                                                                             \
      d2_ ? launch_nodes(kernel<8, 2>, 8, p, stream) : launch_nodes(kernel<8, 1>, 8, p, stream);  \
    else                                                                                          \
      launch_nodes(kernel<16, 1>, 16, p, stream);                                                 \
  } while (0)

extern "C" int tta_spectral_block_fwd(const float* x1, const float* aw2, const float* ab2,
                                      const float* ws_t, const float* bs, const float* w1t,
                                      const float* b1, const float* w2t, const float* b2,
                                      float* inv2, float* a_s, float* h, float* x2,
                                      const float* awn, const float* abn, const float* add0,
                                      float* yn, float* invn, int64_t N, int64_t C, int64_t H,
                                      float eps, hipStream_t stream) {
  TTA_CHECK_ARG(node_dims_ok(N, (int)C, (int)H),
                "tta_spectral_block_fwd: need C, H multiples of 16 in [16, 128] (got N=%lld C=%lld "
                "H=%lld)", (long long)N, (long long)C, (long long)H);
  TTA_CHECK_ARG(x1 && aw2 && ab2 && ws_t && bs && w1t && b1 && w2t && b2 && inv2 && a_s && h &&
                    x2,
                "tta_spectral_block_fwd: null pointer");
  TTA_CHECK_ARG(!awn || (abn && yn && invn), "tta_spectral_block_fwd: incomplete next norm");
  if (N == 0) return tta::kOk;
  SpecFwdArgs p{x1, aw2, ab2, ws_t, bs, w1t, b1, w2t, b2, inv2, a_s, h, x2,
                awn, abn, add0, yn, invn, N, (int)C, (int)H, eps};
  LAUNCH_SPECTRAL(k_spectral_block_fwd, p, stream);
  TTA_CHECK_LAUNCH("tta_spectral_block_fwd");
  return tta::kOk;
}

extern "C" int tta_spectral_block_bwd(const float* g_n, const float* x2, const float* awn,
                                      const float* invn, const float* res, const float* x1,
                                      const float* aw2, const float* inv2, const float* a_s,
                                      const float* h, const float* w1, const float* w2,
                                      const float* ws, float* g_x1, int64_t N, int64_t C,
                                      int64_t H, hipStream_t stream) {
  TTA_CHECK_ARG(node_dims_ok(N, (int)C, (int)H),
                "tta_spectral_block_bwd: need C, H multiples of 16 in [16, 128] (got N=%lld C=%lld "
                "H=%lld)", (long long)N, (long long)C, (long long)H);
  TTA_CHECK_ARG(g_n && x2 && awn && invn && x1 && aw2 && inv2 && a_s && h && w1 && w2 && ws &&
                    g_x1,
                "tta_spectral_block_bwd: null pointer");
  if (N == 0) return tta::kOk;
  SpecBwdArgs p{g_n, x2, awn, invn, res, x1, aw2, inv2, a_s, h, w1, w2, ws, g_x1, N, (int)C,
                (int)H};
  LAUNCH_SPECTRAL(k_spectral_block_bwd, p, stream);
  TTA_CHECK_LAUNCH("tta_spectral_block_bwd");
  return tta::kOk;
}

extern "C" int tta_energy_head_fwd(const float* ne, const float* w0t, const float* b0,
                                   const float* w1t, const float* b1, const float* w2,
                                   const float* b2, float* a1, float* a2, float* node_e,
                                   int64_t N, int64_t C, int64_t H, hipStream_t stream) {
  TTA_CHECK_ARG(node_dims_ok(N, (int)C, (int)H),
                "tta_energy_head_fwd: need C, H multiples of 16 in [16, 128]");
  TTA_CHECK_ARG(ne && w0t && b0 && w1t && b1 && w2 && b2 && a1 && a2 && node_e,
                "tta_energy_head_fwd: null pointer");
  if (N == 0) return tta::kOk;
  HeadArgs p{ne, w0t, b0, w1t, b1, w2, b2, nullptr, nullptr, a1, a2, node_e, nullptr, N, (int)C,
             (int)H, head_nodes(N)};
  hipLaunchKernelGGL(k_energy_head_fwd, dim3(tta_blocks(N, p.npb)), dim3(NTH), 0, stream, p);
  TTA_CHECK_LAUNCH("tta_energy_head_fwd");
  return tta::kOk;
}

extern "C" int tta_energy_head_bwd(const float* a1, const float* a2, const float* w0,
                                   const float* w1, const float* w2, float* g_ne, int64_t N,
                                   int64_t C, int64_t H, hipStream_t stream) {
  TTA_CHECK_ARG(node_dims_ok(N, (int)C, (int)H),
                "tta_energy_head_bwd: need C, H multiples of 16 in [16, 128]");
  TTA_CHECK_ARG(a1 && a2 && w0 && w1 && w2 && g_ne, "tta_energy_head_bwd: null pointer");
  if (N == 0) return tta::kOk;
  HeadArgs p{nullptr, nullptr, nullptr, nullptr, nullptr, w2, nullptr, w0, w1,
             const_cast<float*>(a1), const_cast<float*>(a2), nullptr, g_ne, N, (int)C, (int)H,
             head_nodes(N)};
  hipLaunchKernelGGL(k_energy_head_bwd, dim3(tta_blocks(N, p.npb)), dim3(NTH), 0, stream, p);
  TTA_CHECK_LAUNCH("tta_energy_head_bwd");
  return tta::kOk;
}
