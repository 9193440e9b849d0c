// Per-op entry points of the reference's rotation and scatter modules, for callers that drive the
// eSCN-MD blocks op by op instead of through the fused step:
//  * a rotation by a per-edge matrix with a fixed sparsity pattern (rotation.py:211-260): the
//    pattern's nnz structural nonzeros (i_k, j_k) are shared by all edges, their values are the
//    packed coefficients coef[e, k];
//  * the edge -> node sum over a fixed-width gather table (scatter.py:62-89).
// The fused step uses the specialised kernels of rotate.hip instead; these serve any pattern
// (rectangular, any lmax), any channel count and the reference's table layout.
#include "common.h"

#include <algorithm>

typedef float floatx4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kMaxNnz = 512, kMaxRows = 64, kMaxBlocks = 255;

// A pattern grouped by output block: the terms of output block r are q in [ptr[r], ptr[r+1]),
// each coefficient column (low half of term[q]) times input block (high half) (kernel arguments:
// read-only, uniform).
struct RotPattern {
  uint16_t ptr[kMaxRows + 1];
  uint32_t term[kMaxNnz];
};

// out[e, r, w] = sum_q coef[e, k_q] x[e, blk_q, w] over the terms of block r, in pattern order.
// One thread per output element; consecutive threads take consecutive channels.  The general
// form: any W, any alignment, any number of blocks (the tiled form below takes the others).
__global__ __launch_bounds__(256) void k_rotate_pattern(const float* __restrict__ x,
                                                        const float* __restrict__ coef,
                                                        float* __restrict__ out, int64_t E,
                                                        int n_in, int n_out, int W, int nnz,
                                                        RotPattern pat) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per_edge = (int64_t)n_out * W;
  if (gid >= E * per_edge) return;
  const int64_t e = gid / per_edge;
  const int rw = (int)(gid - e * per_edge);
  const int r = rw / W, w = rw - r * W;
  const float* xe = x + e * (int64_t)n_in * W + w;
  const float* ce = coef + e * (int64_t)nnz;
  float acc = 0.f;
  for (int q = pat.ptr[r]; q < pat.ptr[r + 1]; ++q)
    acc += ce[pat.term[q] & 0xffffu] * xe[(pat.term[q] >> 16) * W];
  out[gid] = acc;
}

// The same for rows of float4s (W % 4 == 0, 16-byte aligned): a workgroup copies the rows and
// coefficients of EB consecutive edges to LDS, each once and coalesced, and a thread forms all
// output blocks of one float4 column of one edge.  Bound by HBM (each input and output byte
// crosses it once); the element-per-thread form read every input block once per term through the
// cache (about four times over for an lmax = 2 rotation) with a 64-bit division per element.
// E = 20,011, nine blocks of 128 channels, 35 terms (187 MB): 153-168 -> 37 us (5.0 TB/s).
__global__ __launch_bounds__(256) void k_rotate_pattern_tiled(const float* __restrict__ x,
                                                              const float* __restrict__ coef,
                                                              float* __restrict__ out, int64_t E,
                                                              int n_in, int n_out, int W4, int nnz,
                                                              int EB, RotPattern pat) {
  extern __shared__ __align__(16) float lds[];
  floatx4* xs = reinterpret_cast<floatx4*>(lds);  // [EB][n_in][W4]
  float* cs = lds + (int64_t)4 * EB * n_in * W4;  // [EB][nnz]
  const int t = threadIdx.x;
  const int64_t e0 = (int64_t)blockIdx.x * EB;
  const int ne = (int)min((int64_t)EB, E - e0);
  const floatx4* xg = reinterpret_cast<const floatx4*>(x) + e0 * n_in * W4;
  const float* cg = coef + e0 * nnz;
  for (int i = t; i < ne * n_in * W4; i += 256) xs[i] = __builtin_nontemporal_load(xg + i);
  for (int i = t; i < ne * nnz; i += 256) cs[i] = cg[i];
  __syncthreads();
  floatx4* og = reinterpret_cast<floatx4*>(out) + e0 * n_out * W4;
  for (int item = t; item < ne * W4; item += 256) {
    const int e = item / W4, c = item - e * W4;
    const floatx4* xe = xs + e * n_in * W4 + c;
    const float* ce = cs + e * nnz;
    for (int r = 0; r < n_out; ++r) {
      floatx4 acc = {0.f, 0.f, 0.f, 0.f};
      const int q1 = pat.ptr[r + 1];
#pragma unroll 4
      for (int q = pat.ptr[r]; q < q1; ++q) {
        const uint32_t w = pat.term[q];
        acc += ce[w & 0xffffu] * xe[(w >> 16) * W4];
      }
      __builtin_nontemporal_store(acc, og + (e * n_out + r) * W4 + c);
    }
  }
}

// gc[e, k] = sum_w g_out[e, i_k, w] x_in[e, j_k, w]: one wavefront per (edge, nonzero), lanes
// striding over the channels, then a fixed butterfly (deterministic).  The general form.
struct GcPattern {
  uint8_t i[kMaxNnz];
  uint8_t j[kMaxNnz];
};

__global__ __launch_bounds__(256) void k_rotate_pattern_gc(const float* __restrict__ g_out,
                                                           const float* __restrict__ x_in,
                                                           float* __restrict__ gc, int64_t E,
                                                           int n_in, int n_out, int W, int nnz,
                                                           GcPattern pat) {
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (wave >= E * nnz) return;
  const int64_t e = wave / nnz;
  const int k = (int)(wave - e * nnz);
  const float* go = g_out + (e * n_out + pat.i[k]) * (int64_t)W;
  const float* xi = x_in + (e * n_in + pat.j[k]) * (int64_t)W;
  float acc = 0.f;
  for (int w = lane; w < W; w += 64) acc += go[w] * xi[w];
  acc = tta_group_sum(acc, 64);
  if (lane == 0) gc[wave] = acc;
}

// The same for rows of float4s: a workgroup copies the rows of EB consecutive edges to LDS (row
// stride W + 4 floats, so that the nine rows a wavefront reads at one column fall on different
// banks) and four lanes share one (edge, nonzero), float4s c, c + 4, ... of the channels each; the
// four components and the four lanes are added pairwise, so the longest chain of additions is
// W / 16.  The wavefront-per-nonzero form fetched both rows again for every nonzero.  E = 20,011,
// nine blocks of 128 channels, 35 nonzeros (187 MB): 152 -> 47 us (4.0 TB/s).
__global__ __launch_bounds__(256) void k_rotate_pattern_gc_tiled(
    const float* __restrict__ g_out, const float* __restrict__ x_in, float* __restrict__ gc,
    int64_t E, int n_in, int n_out, int W4, int nnz, int EB, GcPattern pat) {
  extern __shared__ __align__(16) float lds[];
  const int LD = W4 + 1;                          // row stride in float4s
  floatx4* gs = reinterpret_cast<floatx4*>(lds);  // [EB][n_out][LD]
  floatx4* xs = gs + EB * n_out * LD;             // [EB][n_in][LD]
  const int t = threadIdx.x;
  const int64_t e0 = (int64_t)blockIdx.x * EB;
  const int ne = (int)min((int64_t)EB, E - e0);
  const floatx4* gg = reinterpret_cast<const floatx4*>(g_out) + e0 * n_out * W4;
  const floatx4* xg = reinterpret_cast<const floatx4*>(x_in) + e0 * n_in * W4;
  for (int i = t; i < ne * n_out * W4; i += 256)
    gs[i + i / W4] = __builtin_nontemporal_load(gg + i);
  for (int i = t; i < ne * n_in * W4; i += 256)
    xs[i + i / W4] = __builtin_nontemporal_load(xg + i);
  __syncthreads();
  const int part = t & 3;
  for (int item = t >> 2; item < ne * nnz; item += 64) {
    const int e = item / nnz, k = item - e * nnz;
    const floatx4* a = gs + (e * n_out + pat.i[k]) * LD;
    const floatx4* b = xs + (e * n_in + pat.j[k]) * LD;
    floatx4 s = {0.f, 0.f, 0.f, 0.f};
    for (int c = part; c < W4; c += 4) s += a[c] * b[c];
    float v = (s[0] + s[1]) + (s[2] + s[3]);
    v += __shfl_xor(v, 1);  // the four lanes of an item run the same iterations
    v += __shfl_xor(v, 2);
    if (part == 0) gc[e0 * nnz + item] = v;
  }
}

// out[n, w] = sum_d msg[g, w] for g = gather[n * Dmax + d], d = 0 .. Dmax - 1 in order; an index
// outside [0, n_msg) (the table's sentinel: the zero row appended to the messages) adds nothing.
// V channels per thread (4: W % 4 == 0 and 16-byte aligned rows).  Bound by the gathered rows;
// eight table entries and then the eight rows they name are in flight at once (a sentinel reads
// row 0 and adds nothing), where one entry and its row at a time left a chain of two memory
// latencies per entry.  1000 nodes, 20,011 rows of 1152: 65 -> 25 us (3.9 TB/s).
template <int V>
__global__ __launch_bounds__(256) void k_segment_sum_table(const float* __restrict__ msg,
                                                           const int* __restrict__ gather,
                                                           float* __restrict__ out, int64_t N,
                                                           int Dmax, int WV, int64_t n_msg) {
  typedef float vec __attribute__((ext_vector_type(V)));
  constexpr int B = 8;
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= N * WV) return;
  const int64_t n = gid / WV;
  const int w = (int)(gid - n * WV);
  const int* gr = gather + n * Dmax;
  const vec* m = reinterpret_cast<const vec*>(msg) + w;
  vec acc;
#pragma unroll
  for (int e = 0; e < V; ++e) acc[e] = 0.f;
  if (n_msg > 0) {
    for (int d0 = 0; d0 < Dmax; d0 += B) {
      int g[B];
      vec v[B];
#pragma unroll
      for (int i = 0; i < B; ++i) g[i] = d0 + i < Dmax ? gr[d0 + i] : -1;
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const bool ok = g[i] >= 0 && g[i] < n_msg;
        v[i] = m[(ok ? (int64_t)g[i] : 0) * WV];
      }
#pragma unroll
      for (int i = 0; i < B; ++i)
        if (g[i] >= 0 && g[i] < n_msg) acc += v[i];
    }
  }
  *(reinterpret_cast<vec*>(out) + gid) = acc;
}

// Edges per workgroup of the tiled forms: what 38 KB of LDS hold, at most 64, so that four
// workgroups share a compute unit; one edge whose rows take more gets a workgroup of its own (two
// per compute unit) up to 64 KB; 0: past that, the general form.
int tile_edges(int64_t floats_per_edge) {
  const int64_t bytes = 4 * floats_per_edge;
  if (bytes > 65536) return 0;
  return (int)std::max<int64_t>(1, std::min<int64_t>(64, 38912 / bytes));
}

bool rows_of_float4(int64_t W, const void* a, const void* b) {
  return W % 4 == 0 && (uintptr_t)a % 16 == 0 && (uintptr_t)b % 16 == 0;
}

}  // namespace

extern "C" int tta_rotate_pattern(const float* x, const float* coef, float* out, int64_t E,
                                  int64_t n_in, int64_t n_out, int64_t W, int64_t nnz,
                                  const int* ptr, const int* k, const int* blk,
                                  hipStream_t stream) {
  TTA_CHECK_ARG(E >= 0 && W > 0 && n_in > 0 && n_in <= kMaxBlocks && n_out > 0 &&
                    n_out <= kMaxRows && nnz >= 0 && nnz <= kMaxNnz,
                "tta_rotate_pattern: sizes out of range (n_in <= %d, n_out <= %d, nnz <= %d)",
                kMaxBlocks, kMaxRows, kMaxNnz);
  TTA_CHECK_ARG(E * n_out * W < ((int64_t)1 << 40) && n_in * W < (1 << 30),
                "tta_rotate_pattern: tensor too large");
  TTA_CHECK_ARG(ptr && (nnz == 0 || (k && blk)), "tta_rotate_pattern: null pattern");
  RotPattern pat{};
  TTA_CHECK_ARG(ptr[0] == 0 && ptr[n_out] == nnz, "tta_rotate_pattern: ptr must run 0 .. nnz");
  for (int64_t r = 0; r <= n_out; ++r) {
    TTA_CHECK_ARG(r == 0 || ptr[r] >= ptr[r - 1], "tta_rotate_pattern: ptr must not decrease");
    pat.ptr[r] = (uint16_t)ptr[r];
  }
  for (int64_t q = 0; q < nnz; ++q) {
    TTA_CHECK_ARG(k[q] >= 0 && k[q] < nnz && blk[q] >= 0 && blk[q] < n_in,
                  "tta_rotate_pattern: term %lld out of range", (long long)q);
    pat.term[q] = (uint32_t)k[q] | ((uint32_t)blk[q] << 16);
  }
  if (E == 0) return tta::kOk;
  TTA_CHECK_ARG(x && out && (coef || nnz == 0), "tta_rotate_pattern: null pointer");
  const int EB = rows_of_float4(W, x, out) ? tile_edges(n_in * W + nnz) : 0;
  if (EB > 0)
    hipLaunchKernelGGL(k_rotate_pattern_tiled, dim3(tta_blocks(E, EB)), dim3(256),
                       (size_t)EB * (n_in * W + nnz) * sizeof(float), stream, x, coef, out, E,
                       (int)n_in, (int)n_out, (int)(W / 4), (int)nnz, EB, pat);
  else
    hipLaunchKernelGGL(k_rotate_pattern, dim3(tta_blocks(E * n_out * W, 256)), dim3(256), 0,
                       stream, x, coef, out, E, (int)n_in, (int)n_out, (int)W, (int)nnz, pat);
  TTA_CHECK_LAUNCH("tta_rotate_pattern");
  return tta::kOk;
}

extern "C" int tta_rotate_pattern_gc(const float* g_out, const float* x_in, float* gc, int64_t E,
                                     int64_t n_in, int64_t n_out, int64_t W, int64_t nnz,
                                     const int* ii, const int* jj, hipStream_t stream) {
  TTA_CHECK_ARG(E >= 0 && W > 0 && n_in > 0 && n_in <= kMaxBlocks && n_out > 0 &&
                    n_out <= kMaxBlocks && nnz >= 0 && nnz <= kMaxNnz,
                "tta_rotate_pattern_gc: sizes out of range (n_in, n_out <= %d, nnz <= %d)",
                kMaxBlocks, kMaxNnz);
  TTA_CHECK_ARG(E * nnz < ((int64_t)1 << 34) && (int64_t)n_in * W < (1 << 30) &&
                    (int64_t)n_out * W < (1 << 30),
                "tta_rotate_pattern_gc: tensor too large");
  TTA_CHECK_ARG(nnz == 0 || (ii && jj), "tta_rotate_pattern_gc: null pattern");
  GcPattern pat{};
  for (int64_t q = 0; q < nnz; ++q) {
    TTA_CHECK_ARG(ii[q] >= 0 && ii[q] < n_out && jj[q] >= 0 && jj[q] < n_in,
                  "tta_rotate_pattern_gc: nonzero %lld out of range", (long long)q);
    pat.i[q] = (uint8_t)ii[q];
    pat.j[q] = (uint8_t)jj[q];
  }
  if (E == 0 || nnz == 0) return tta::kOk;
  TTA_CHECK_ARG(g_out && x_in && gc, "tta_rotate_pattern_gc: null pointer");
  const int64_t tile = (n_in + n_out) * (W + 4);
  const int EB = rows_of_float4(W, g_out, x_in) ? tile_edges(tile) : 0;
  if (EB > 0)
    hipLaunchKernelGGL(k_rotate_pattern_gc_tiled, dim3(tta_blocks(E, EB)), dim3(256),
                       (size_t)EB * tile * sizeof(float), stream, g_out, x_in, gc, E, (int)n_in,
                       (int)n_out, (int)(W / 4), (int)nnz, EB, pat);
  else
    hipLaunchKernelGGL(k_rotate_pattern_gc, dim3(tta_blocks(E * nnz * 64, 256)), dim3(256), 0,
                       stream, g_out, x_in, gc, E, (int)n_in, (int)n_out, (int)W, (int)nnz, pat);
  TTA_CHECK_LAUNCH("tta_rotate_pattern_gc");
  return tta::kOk;
}

extern "C" int tta_segment_sum_table(const float* msg, const int* gather, float* out,
                                     int64_t n_msg, int64_t N, int64_t Dmax, int64_t W,
                                     hipStream_t stream) {
  TTA_CHECK_ARG(n_msg >= 0 && N >= 0 && Dmax >= 0 && W > 0 && Dmax < (1 << 20) &&
                    W < (1 << 24) && n_msg < ((int64_t)1 << 31),
                "tta_segment_sum_table: sizes out of range");
  TTA_CHECK_ARG(N * W < ((int64_t)1 << 40), "tta_segment_sum_table: tensor too large");
  if (N == 0) return tta::kOk;
  TTA_CHECK_ARG(out && (Dmax == 0 || gather) && (n_msg == 0 || msg),
                "tta_segment_sum_table: null pointer");
  if (rows_of_float4(W, msg, out))
    hipLaunchKernelGGL(k_segment_sum_table<4>, dim3(tta_blocks(N * W / 4, 256)), dim3(256), 0,
                       stream, msg, gather, out, N, (int)Dmax, (int)(W / 4), n_msg);
  else
    hipLaunchKernelGGL(k_segment_sum_table<1>, dim3(tta_blocks(N * W, 256)), dim3(256), 0, stream,
                       msg, gather, out, N, (int)Dmax, (int)W, n_msg);
  TTA_CHECK_LAUNCH("tta_segment_sum_table");
  return tta::kOk;
}
