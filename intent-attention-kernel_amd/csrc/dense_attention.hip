// Dense softmax attention of the reference's dense_attention() in float32, for gfx950.
//
// Reference semantics (src/intent_attention/reference.py:16-45):
//   scores = (q . k^T) * scale
//   causal, no positions:   scores += triu(-inf, diagonal=1)   (query i sees keys j <= i)
//   causal, kv positions:   scores[i, j] = -inf where i < original_kv_positions[j]
//   mask:                   scores += mask                      (an additive mask; bool adds 1.0)
//   out = softmax(scores) . v
// A row whose scores are all -inf is NaN (softmax of -inf everywhere), as in
// torch; an empty key set gives zeros (torch's matmul over an empty dim).
//
// The reference runs these as torch.matmul / softmax in the input dtype. Here
// every product and sum is float32 over float32, float16 or bfloat16 inputs,
// and the output is rounded once to the input dtype.
//
// Calls with several query rows per batch entry run on the matrix cores
// (dense_matrix.h: causal prefill of 32 heads x 2,048 rows x 128 in float16
// 10.8 ms -> 0.082 ms, 128 rows x 3,072 keys x 64 in float32, 8 heads, 274 -> 21 us);
// what follows is the rows form, for the rest.
//
// Selected tokens (kv_index) are read where they lie: the gathered K and V of 3,072 of
// 4,096 tokens x 8 heads x 64 in float32 took two launches of 9 us and a pass over both,
// the index costs the kernels that read it no time that shows (blocks through
// semantic_block_attention 170 -> 50 us with the index uploaded without a wait); the
// others are compiled without it (dense_row).
//
// Work split. A (batch, query) row's keys go to `splits` workgroups of
// consecutive key ranges (`chunk` keys each); splits > 1 only when the caller
// gives a workspace and there are few rows with 256 keys or more (decode shapes),
// and a second kernel then merges the partials (max, denominator, context)
// by log-sum-exp. A workgroup has WAVES waves (16 when the grid is short, so
// it still has many key rows in flight); wave w takes KEYS consecutive keys
// per step. It loads the K and V rows of all of them first, then reduces the
// KEYS wave-wide dot products together, so one step costs about one memory
// round trip. Lane l holds dims l, l + 64, ... of q and of the context: a key
// or value row is one coalesced load per 64 dims, its row address a scalar.
// Each wave keeps a running max, denominator and context; the waves merge
// through the LDS at the end.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>
#include <type_traits>

#include "iak.h"
#include "iak_device.h"

namespace iak {

namespace {

// the split over keys: rows with at least SPLIT_MIN_KEYS keys, ranges of at
// least RANGE_MIN_KEYS keys
#ifndef SPLIT_MIN_KEYS
#define SPLIT_MIN_KEYS 256
#endif
#ifndef RANGE_MIN_KEYS
#define RANGE_MIN_KEYS 64
#endif
// workgroups the split aims at
#ifndef SPLIT_TARGET_WGS
#define SPLIT_TARGET_WGS 256
#endif

// element types: float, _Float16, and bfloat16 held as its 16 bits
struct bf16_bits { uint16_t b; };

__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(_Float16 x) { return (float)x; }
__device__ __forceinline__ float to_f32(bf16_bits x) { return __builtin_bit_cast(float, (uint32_t)x.b << 16); }
__device__ __forceinline__ float to_f32(uint8_t x) { return x ? 1.f : 0.f; }   // bool mask: adds 1.0

template <typename T>
__device__ __forceinline__ float load_t(const void* p, int64_t i) {
  return to_f32(reinterpret_cast<const T*>(p)[i]);
}

template <typename T>
__device__ __forceinline__ void store_t(void* p, int64_t i, float x) {
  if constexpr (sizeof(T) == 4) {
    reinterpret_cast<float*>(p)[i] = x;
  } else if constexpr (__is_same(T, _Float16)) {
    reinterpret_cast<_Float16*>(p)[i] = (_Float16)x;
  } else {
    // bfloat16, round to nearest even (NaN kept quiet)
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    const uint32_t r = (u & 0x7fffffffu) > 0x7f800000u ? (u | 0x00400000u) : u + 0x7fffu + ((u >> 16) & 1u);
    reinterpret_cast<uint16_t*>(p)[i] = (uint16_t)(r >> 16);
  }
}

// the entry point's arguments, and the rows of k and v that are its keys (or null: key j is row j)
struct DenseArgs : iak_dense_attention_args {
  const int64_t* kv_index;
};

// the mask values of keys j0 .. j0 + KEYS - 1 of one query row (indices
// clamped to the range's last key `last`)
template <typename M, int KEYS>
__device__ __forceinline__ void step_mask(const iak_dense_attention_args& a, int64_t mb, int j0, int last,
                                          float* madd) {
#pragma unroll
  for (int u = 0; u < KEYS; ++u) {
    const int jc = j0 + u < last ? j0 + u : last;
    madd[u] = load_t<M>(a.mask, mb + (int64_t)jc * a.mask_stride_k);
  }
}

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

// Sum over the 64 lanes, the same bits in every lane: each step adds two
// values that the partner lane adds in the other order (lane ^ 1 and lane ^ 2
// by quad permutes; then, with a quad's four lanes equal, the quads two and
// one places round the row of 16 by row rotates; then rows through the lane
// swaps), so every lane forms the same sums.
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp<0xB1>(v);    // quad_perm [1, 0, 3, 2]
  v += dpp<0x4E>(v);    // quad_perm [2, 3, 0, 1]
  v += dpp<0x128>(v);   // row_ror:8
  v += dpp<0x124>(v);   // row_ror:4
  return xsum16_32(v);
}

struct DenseSplit {
  int splits;   // workgroups per row
  int chunk;    // keys per workgroup (the last may have fewer)
  float* ws;    // splits > 1: [rows * splits] max, [rows * splits] denominator, [rows * splits, v_dim] context
};

// T: element type of q, k, v and out; NPL: dims per lane (head_dim and v_dim
// are at most 64 * NPL); KEYS keys per wave and step; WAVES waves per workgroup.
// `item` = row * splits + split, row = b * q_len + i; `items` of them in all.
// INDEX: whether kv_index is given, or ANY_INDEX (a test of it per step cost the others 5 %: 512 rows x 4,096
// keys x 128 in float16 229 / 241 us; between the loads, 1,024 rows x 1,000 keys x
// 1,000 457 / 830 us)
constexpr int ANY_INDEX = 2;
template <typename T, int NPL, int KEYS, int WAVES, int INDEX, typename Args>
__device__ __forceinline__ void dense_row(const Args& a, const DenseSplit& sp, int64_t item, int64_t items) {
  __shared__ float part_acc[WAVES][64 * NPL];
  __shared__ float part_m[WAVES], part_l[WAVES];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t row = item / sp.splits;
  const int split = (int)(item - row * sp.splits);
  const int64_t b = row / a.q_len;
  const int i = (int)(row - b * a.q_len);
  const int lo = split * sp.chunk;
  const int hi = a.kv_len - lo < sp.chunk ? a.kv_len : lo + sp.chunk;   // keys lo .. hi - 1
  const float NEG_INF = -__builtin_inff();

  // this lane's dims, clamped into the row (the values past the width are zeroed)
  int dk[NPL], dv[NPL];
  bool okk[NPL], okv[NPL];
  float q[NPL], acc[NPL];
  const T* qrow = reinterpret_cast<const T*>(a.q) + b * a.q_stride_b + (int64_t)i * a.q_stride_t;
#pragma unroll
  for (int jj = 0; jj < NPL; ++jj) {
    const int d = lane + 64 * jj;
    okk[jj] = d < a.head_dim;
    okv[jj] = d < a.v_dim;
    dk[jj] = okk[jj] ? d : a.head_dim - 1;
    dv[jj] = okv[jj] ? d : a.v_dim - 1;
    const float qx = to_f32(qrow[dk[jj]]);
    q[jj] = okk[jj] ? qx : 0.f;
    acc[jj] = 0.f;
  }
  const T* kbase = reinterpret_cast<const T*>(a.k) + b * a.k_stride_b;
  const T* vbase = reinterpret_cast<const T*>(a.v) + b * a.v_stride_b;
  const int64_t mb = b * a.mask_stride_b + (int64_t)i * a.mask_stride_q;
  float m = NEG_INF, l = 0.f;
  // The K and V rows of a step's KEYS keys, loaded unconditionally at clamped
  // indices (a key past the range reads the range's last key; the values are
  // zeroed at use), so no load waits behind a branch. The loop is pipelined:
  // the next step's rows are in flight while this step's are reduced.
  float kn[KEYS][NPL], vn[KEYS][NPL];
  auto load_step = [&](int j0) {
#pragma unroll
    for (int u = 0; u < KEYS; ++u) {
      const int jc = j0 + u < hi ? j0 + u : hi - 1;
      int64_t at = jc;   // wave-uniform
      if constexpr (INDEX == 1) at = a.kv_index[jc];
      else if constexpr (INDEX == ANY_INDEX) at = a.kv_index ? a.kv_index[jc] : jc;
      const T* kr = kbase + at * a.k_stride_t;
      const T* vr = vbase + at * a.v_stride_t;
#pragma unroll
      for (int jj = 0; jj < NPL; ++jj) {
        kn[u][jj] = to_f32(kr[dk[jj]]);
        vn[u][jj] = to_f32(vr[dv[jj]]);
      }
    }
  };
  if (lo + KEYS * w < hi) load_step(lo + KEYS * w);
  for (int j0 = lo + KEYS * w; j0 < hi; j0 += KEYS * WAVES) {
    float kv[KEYS][NPL], vv[KEYS][NPL];
#pragma unroll
    for (int u = 0; u < KEYS; ++u) {
      const bool key = j0 + u < hi;   // wave-uniform
#pragma unroll
      for (int jj = 0; jj < NPL; ++jj) {
        kv[u][jj] = key && okk[jj] ? kn[u][jj] : 0.f;
        vv[u][jj] = key && okv[jj] ? vn[u][jj] : 0.f;
      }
    }
    // the next step's rows (clamped into the range on the last step)
    load_step(j0 + KEYS * WAVES < hi ? j0 + KEYS * WAVES : j0);
    float s[KEYS];
#pragma unroll
    for (int u = 0; u < KEYS; ++u) {
      float t = 0.f;
#pragma unroll
      for (int jj = 0; jj < NPL; ++jj) t = __builtin_fmaf(q[jj], kv[u][jj], t);
      s[u] = t;
    }
#pragma unroll
    for (int u = 0; u < KEYS; ++u) s[u] = wave_sum(s[u]);
    // the step's mask values and key positions, each set under one uniform branch
    float madd[KEYS];
    bool hidden[KEYS];
#pragma unroll
    for (int u = 0; u < KEYS; ++u) {
      madd[u] = 0.f;
      hidden[u] = false;
    }
    if (a.mask) {
      if (a.mask_dtype == IAK_MASK_BOOL) step_mask<uint8_t, KEYS>(a, mb, j0, hi - 1, madd);
      else if (a.mask_dtype == IAK_DTYPE_F32) step_mask<float, KEYS>(a, mb, j0, hi - 1, madd);
      else if (a.mask_dtype == IAK_DTYPE_F16) step_mask<_Float16, KEYS>(a, mb, j0, hi - 1, madd);
      else step_mask<bf16_bits, KEYS>(a, mb, j0, hi - 1, madd);
    }
    if (a.causal == IAK_CAUSAL_POSITIONS) {
#pragma unroll
      for (int u = 0; u < KEYS; ++u) {
        const int jc = j0 + u < hi ? j0 + u : hi - 1;
        hidden[u] = (int64_t)i < a.kv_positions[jc];   // masked_fill(-inf)
      }
    }
    float smax = NEG_INF;
#pragma unroll
    for (int u = 0; u < KEYS; ++u) {
      const int j = j0 + u;
      float x = s[u] * a.sm_scale;
      if (a.causal == IAK_CAUSAL_TRIU && j > i) x += NEG_INF;   // scores + triu(-inf, diagonal=1)
      if (hidden[u]) x = NEG_INF;
      x += madd[u];
      if (j >= hi) x = NEG_INF;                     // not a key of this range: no mass
      s[u] = x;
      smax = fmaxf(smax, x);
    }
    const float mn = fmaxf(m, smax);
    if (mn > m) {   // wave-uniform
      const float alpha = expf(m - mn);   // 0 while nothing was seen (m = -inf)
      l *= alpha;
#pragma unroll
      for (int jj = 0; jj < NPL; ++jj) acc[jj] *= alpha;
      m = mn;
    }
#pragma unroll
    for (int u = 0; u < KEYS; ++u) {
      // -inf scores (masked keys and the keys past the range) take no mass,
      // also when m is -inf; NaN scores poison l, as in softmax
      const float e = s[u] == NEG_INF ? 0.f : expf(s[u] - m);
      l += e;
#pragma unroll
      for (int jj = 0; jj < NPL; ++jj) acc[jj] = __builtin_fmaf(e, vv[u][jj], acc[jj]);
    }
  }

  if (lane == 0) {
    part_m[w] = m;
    part_l[w] = l;
  }
#pragma unroll
  for (int jj = 0; jj < NPL; ++jj) part_acc[w][lane + 64 * jj] = acc[jj];
  __syncthreads();
  float M = NEG_INF;
#pragma unroll
  for (int k = 0; k < WAVES; ++k) M = fmaxf(M, part_m[k]);
  float wt[WAVES], L = 0.f;
#pragma unroll
  for (int k = 0; k < WAVES; ++k) {
    wt[k] = part_m[k] == NEG_INF ? 0.f : expf(part_m[k] - M);   // 0 for a wave that saw no mass
    L += wt[k] * part_l[k];
  }
  if (sp.splits > 1) {
    // this range's partial: max, denominator and unnormalised context
    if (threadIdx.x == 0) {
      sp.ws[item] = M;
      sp.ws[items + item] = L;
    }
    float* wacc = sp.ws + 2 * items + item * a.v_dim;
    for (int d = threadIdx.x; d < a.v_dim; d += 64 * WAVES) {
      float A = 0.f;
#pragma unroll
      for (int k = 0; k < WAVES; ++k) A = __builtin_fmaf(wt[k], part_acc[k][d], A);
      wacc[d] = A;
    }
    return;
  }
  // all scores -inf: softmax is NaN everywhere; no keys at all: zeros
  const float empty = a.kv_len > 0 ? __builtin_nanf("") : 0.f;
  const int64_t ooff = b * a.out_stride_b + (int64_t)i * a.out_stride_t;
  for (int d = threadIdx.x; d < a.v_dim; d += 64 * WAVES) {
    float A = 0.f;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) A = __builtin_fmaf(wt[k], part_acc[k][d], A);
    store_t<T>(a.out, ooff + d, M == NEG_INF ? empty : A / L);
  }
}

template <typename T, int NPL, int KEYS, int WAVES, int INDEX>
__global__ __launch_bounds__(64 * WAVES) void dense_attention_kernel(
    const std::conditional_t<INDEX == 0, iak_dense_attention_args, DenseArgs> a, const DenseSplit sp) {
  dense_row<T, NPL, KEYS, WAVES, INDEX>(a, sp, blockIdx.x, gridDim.x);
}

#include "dense_matrix.h"

constexpr int MERGE_THREADS = 256;
constexpr int MAX_SPLITS = 1024;

// block-wide max / sum over MERGE_THREADS threads (the result in every thread)
template <bool MAX>
__device__ __forceinline__ float block_reduce(float v, float* red) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float o = __shfl_xor(v, off, 64);
    v = MAX ? fmaxf(v, o) : v + o;
  }
  __syncthreads();   // red[] free from an earlier reduction
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = red[0];
#pragma unroll
  for (int k = 1; k < MERGE_THREADS / 64; ++k) v = MAX ? fmaxf(v, red[k]) : v + red[k];
  return v;
}

// One workgroup per row: the log-sum-exp merge of the row's `splits` partials
// (splits <= MAX_SPLITS). The split weights go to the LDS; each context dim is
// then summed over the splits by G thread groups (G = 256 / dims rounded up to
// 64), each over every G-th split, with eight independent loads in flight.
// accoff: where the contexts lie in ws; log2: the maxima are in the exp2 domain.
// FLAGS: the partials come from dense_matrix_kernel with key-tile flags; a row of a
// flagged batch entry is computed again from its inputs.
template <typename T, bool FLAGS>
__global__ __launch_bounds__(MERGE_THREADS) void dense_merge_kernel(const DenseArgs a,
                                                                    const DenseSplit sp, const MatrixPlan mp,
                                                                    int64_t accoff, int log2) {
  __shared__ float wt[MAX_SPLITS];
  __shared__ float red[MERGE_THREADS / 64];
  __shared__ float part[MERGE_THREADS];
  const int64_t row = blockIdx.x;
  const int64_t b = row / a.q_len;
  const int i = (int)(row - b * a.q_len);
  if constexpr (FLAGS) {
    if (mx_flagged(mp, b)) {
      dense_row<T, MX_MAX_DIM / 64, 2, MERGE_THREADS / 64, ANY_INDEX>(a, DenseSplit{1, a.kv_len, nullptr}, row, 0);
      return;
    }
  }
  const int S = sp.splits;
  const int64_t n = (int64_t)gridDim.x * S;
  const float* wm = sp.ws + row * S;
  const float* wl = sp.ws + n + row * S;
  const float* wacc = sp.ws + accoff + row * S * a.v_dim;
  const float NEG_INF = -__builtin_inff();
  float mx = NEG_INF;
  for (int s = threadIdx.x; s < S; s += MERGE_THREADS) mx = fmaxf(mx, wm[s]);
  const float M = block_reduce<true>(mx, red);
  float ls = 0.f;
  for (int s = threadIdx.x; s < S; s += MERGE_THREADS) {
    // 0 for a range that saw no mass
    const float w = wm[s] == NEG_INF ? 0.f : (log2 ? __builtin_amdgcn_exp2f(wm[s] - M) : expf(wm[s] - M));
    wt[s] = w;
    ls += w * wl[s];
  }
  const float L = block_reduce<false>(ls, red);   // its barriers also publish wt[]
  const int dims = (a.v_dim + 63) & ~63;          // v_dim rounded up to 64
  const int G = dims >= MERGE_THREADS ? 1 : MERGE_THREADS / dims;
  const int g = threadIdx.x / dims, dl = threadIdx.x - g * dims;
  const int64_t ooff = b * a.out_stride_b + (int64_t)i * a.out_stride_t;
  for (int d0 = 0; d0 < a.v_dim; d0 += MERGE_THREADS) {
    const int d = d0 + (G > 1 ? dl : threadIdx.x);
    const int dc = d < a.v_dim ? d : a.v_dim - 1;
    float A = 0.f;
    if (g < G) {
      int s = g;
      for (; s + 7 * G < S; s += 8 * G) {
        float x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = wacc[(int64_t)(s + u * G) * a.v_dim + dc];
#pragma unroll
        for (int u = 0; u < 8; ++u) A = __builtin_fmaf(wt[s + u * G], x[u], A);
      }
      for (; s < S; s += G) A = __builtin_fmaf(wt[s], wacc[(int64_t)s * a.v_dim + dc], A);
    }
    if (G > 1) {
      // the G groups' sums of one dim: group 0 adds them in group order
      part[threadIdx.x] = A;
      __syncthreads();
      if (g == 0) {
        for (int k = 1; k < G; ++k) A += part[k * dims + dl];
      }
      __syncthreads();
      if (g != 0) continue;
    }
    // kv_len > 0 here: every score -inf gives NaN
    if (d < a.v_dim) store_t<T>(a.out, ooff + d, M == NEG_INF ? __builtin_nanf("") : A / L);
  }
}

// MAXW: the most waves per workgroup whose registers and LDS fit (16 waves of
// a 1,024-thread workgroup get 128 VGPRs each)
template <typename T, int NPL, int KEYS, int MAXW, int INDEX>
void launch_items(const DenseArgs& a, const DenseSplit& sp, int64_t items, hipStream_t stream) {
  // waves per workgroup: about 4,096 waves in the grid (16 per CU), between 4 and MAXW
  const int64_t want = (4096 + items - 1) / items;
  const dim3 grid((unsigned)items);
  if (MAXW >= 16 && want >= 16)
    hipLaunchKernelGGL((dense_attention_kernel<T, NPL, KEYS, MAXW >= 16 ? 16 : 4, INDEX>), grid, dim3(1024), 0,
                       stream, a, sp);
  else if (want >= 8)
    hipLaunchKernelGGL((dense_attention_kernel<T, NPL, KEYS, 8, INDEX>), grid, dim3(512), 0, stream, a, sp);
  else
    hipLaunchKernelGGL((dense_attention_kernel<T, NPL, KEYS, 4, INDEX>), grid, dim3(256), 0, stream, a, sp);
}

template <typename T, int INDEX>
void launch_rows(const DenseArgs& a, const DenseSplit& sp, hipStream_t stream) {
  const int64_t rows = (int64_t)a.batch * a.q_len;
  const int64_t items = rows * sp.splits;
  const int width = a.head_dim > a.v_dim ? a.head_dim : a.v_dim;
  const int npl = (width + 63) / 64;
  // keys per step: 2 * KEYS * NPL registers of K and V in flight per lane
  if (npl <= 1) launch_items<T, 1, 8, 16, INDEX>(a, sp, items, stream);
  else if (npl <= 2) launch_items<T, 2, 8, 16, INDEX>(a, sp, items, stream);
  else if (npl <= 4) launch_items<T, 4, 4, 16, INDEX>(a, sp, items, stream);
  else if (npl <= 8) launch_items<T, 8, 4, 8, INDEX>(a, sp, items, stream);
  else launch_items<T, 16, 2, 8, INDEX>(a, sp, items, stream);
  if (sp.splits > 1)
    hipLaunchKernelGGL((dense_merge_kernel<T, false>), dim3((unsigned)rows), dim3(MERGE_THREADS), 0, stream, a, sp,
                       MatrixPlan{}, 2 * items, 0);
}

// Splits per row: rows with SPLIT_MIN_KEYS keys or more on a short grid (fewer
// than 512 rows) go over about SPLIT_TARGET_WGS workgroups in ranges of at
// least RANGE_MIN_KEYS keys
// (at most MAX_SPLITS ranges).
DenseSplit split_plan(const DenseArgs& a) {
  DenseSplit sp{1, a.kv_len, nullptr};
  const int64_t rows = (int64_t)a.batch * a.q_len;
  if (rows <= 0 || rows >= 512 || a.kv_len < SPLIT_MIN_KEYS) return sp;
  int64_t s = (SPLIT_TARGET_WGS + rows - 1) / rows;
  const int64_t by_keys = a.kv_len / RANGE_MIN_KEYS;
  if (s > by_keys) s = by_keys;
  if (s > MAX_SPLITS) s = MAX_SPLITS;   // the merge holds the split weights in the LDS
  if (s <= 1) return sp;
  const int64_t chunk = ((int64_t)a.kv_len + s - 1) / s;
  sp.splits = (int)(((int64_t)a.kv_len + chunk - 1) / chunk);
  sp.chunk = (int)chunk;
  return sp;
}

// ---- the matrix-core form: which calls take it, and its plan ----

// From this many (query, key) pairs on, and from this many query rows per batch
// entry, the matrix form is the faster one (10 calls in a graph, us, rows form
// against this one; 16-bit: 32 x 64 keys x 16 rows = 32,768 pairs 8.0 / 8.2 and
// x 32 rows 10.5 / 8.3; 8 x 512 x 8 rows = 32,768 12.8 / 11.1; 8 x 4,096 x 2
// rows 17.7 / 14.4; 32 x 4,096 x 32 rows 347 / 21; float32: 32 x 512 x 3 rows =
// 49,152 22.9 / 18.3; 1 x 2,048 x 16 rows = 32,768 14.0 / 17.1; 8 x 4,096 x 2
// rows 18.2 / 19.9). One query row keeps the rows form: equal at best.
#ifndef MX_MIN_PAIRS
#define MX_MIN_PAIRS 32768
#define MX_MIN_PAIRS_F32 49152
#define MX_MIN_ROWS 2
#define MX_MIN_ROWS_F32 3
#endif

// The float32 matrix instructions run at the rate of the row form's arithmetic, on 32
// query rows at a time: where the keys are split (two launches) or the workgroups come
// in two turns, the row form keeps calls of up to this many pairs if it takes one launch
// itself (us per call among others, and waited for, row form / this one: 16 x 16 rows x 400 keys x 128 = 102,400
// 19.7 / 24.1 and 42.8 / 43.9, 16 x 32 x 256 x 64 = 131,072 19.4 / 23.5 and 40.6 / 39.3, 300 x
// 3 x 128 x 128 = 115,200 25.4 / 30.0; 16 x 32 x 400 x 64 = 204,800 22.2 / 24.1 and 46.8 / 39.7,
// 100 x 16 x 256 x 64 38.5 / 23.6).
#ifndef MX_TWO_TURN_PAIRS_F32
#define MX_TWO_TURN_PAIRS_F32 131072
#endif

// 128 query rows by four waves over 64 keys, or by eight over 128: a step of one wave per
// SIMD takes 3 us, of two (two workgroups on a CU, or the eight waves of one) 2.2 us for
// each 64 keys, the one's matrix work under the other's softmax. Up to one workgroup per
// CU the eight waves are the only way to two (float16, 16 heads x 2,048 x 128: 100 ->
// 72 us; 32 heads, two workgroups per CU: 138 / 144). A causal grid is bound by its
// longest tiles, which run alone when the short ones have ended; eight waves halve them
// (32 heads x 2,048 x 128: 98 -> 82 us, 3 x 4,096 x 128: 135 -> 100, 32 x 4,096 x
// 128, 1,024 workgroups: 282 / 297).
#ifndef MX_WIDE_WGS
#define MX_WIDE_WGS 256
#define MX_WIDE_WGS_CAUSAL 512
#endif

// scores that go through masks or positions
bool general(const DenseArgs& a) { return a.mask || a.causal == IAK_CAUSAL_POSITIONS; }

struct MatrixShape {
  int dp;       // dims, padded
  int qw, kw;   // waves over query rows and over keys
  int bkw;      // keys per wave and tile
};

// causal tiles past the diagonal are not visited
bool causal_skip(const DenseArgs& a) { return a.causal == IAK_CAUSAL_TRIU && !a.mask && a.sm_scale <= 1.f; }

MatrixShape matrix_shape(const DenseArgs& a) {
  const int width = a.head_dim > a.v_dim ? a.head_dim : a.v_dim;
  MatrixShape s{64, 4, 1, 64};
  const bool f32 = a.dtype == IAK_DTYPE_F32;
  s.dp = width <= 64 ? 64 : (width <= 96 && !f32) ? 96 : width <= 128 || f32 ? 128 : width <= 192 ? 192 : 256;
  if (f32) s.bkw = 32;
  // few query rows: the four waves share out the keys instead
  if (a.q_len <= 32 && s.dp <= 128) s.qw = 1, s.kw = 4, s.bkw = 32;
  else if (a.q_len <= 64 && s.dp <= 128) s.qw = 2, s.kw = 2, s.bkw = 32;
  else if (!f32 && s.dp <= 128 && a.kv_len > 128 &&
           (int64_t)a.batch * ((a.q_len + 127) / 128) <= (causal_skip(a) ? MX_WIDE_WGS_CAUSAL : MX_WIDE_WGS)) s.kw = 2;
  return s;
}

// Keys of a wave times dims up to which the keys are not split: the merge is a second
// launch, 5 us of a short call, and costs more than it saves. us per call among others, and
// waited for, all keys in one workgroup / split, float16: 16 x 16 rows x 400 keys x 128 =
// 16,384 19.3 / 24.0 and 40.8 / 39.3, 16 x 16 x 1,000 x 64 = 16,384 19.0 / 23.9 and 41.3 /
// 38.0, 8 x 64 x 600 x 64 = 20,480 19.3 / 24.2 and 43.0 / 39.1, 4 x 128 x 400 x 128 = 32,768
// 23.0 / 24.1 and 47.3 / 43.2 (the row form 22 to 31 and 47 to 55); float32: 16 x 32 x 256 x
// 64 = 4,096 19.0 / 23.7, x 400 = 8,192 22.2 / 23.7; float16 with a mask: 16 x 16 x 333 x
// 80 = 9,216 31.9 / 36.5, 32 x 2 x 1,024 x 64 = 16,384 38 to 44 / 36.5.
#ifndef MX_SHORT
#define MX_SHORT 16384
#define MX_SHORT_MASK 12288
#define MX_SHORT_F32 6144
#endif
bool matrix_short(const DenseArgs& a, const MatrixShape& s) {
  const int64_t bk = s.kw * s.bkw;
  return s.dp <= 128 && ((int64_t)a.kv_len + bk - 1) / bk * s.bkw * s.dp <=
         (a.dtype == IAK_DTYPE_F32 ? MX_SHORT_F32 : general(a) ? MX_SHORT_MASK : MX_SHORT);
}

// 16-byte pieces of whole elements on every operand, at most 256 dims
bool matrix_applies(const DenseArgs& a) {
  const int es = a.dtype == IAK_DTYPE_F32 ? 4 : 2, vec = 16 / es;
  const double pairs = (double)a.batch * a.q_len * a.kv_len;
  if (a.q_len < (es == 4 ? MX_MIN_ROWS_F32 : MX_MIN_ROWS) || pairs < (es == 4 ? MX_MIN_PAIRS_F32 : MX_MIN_PAIRS)) return false;
  const int most = es == 4 ? MX_MAX_DIM_F32 : MX_MAX_DIM;
  if (a.head_dim > most || a.v_dim > most || a.head_dim % vec || a.v_dim % vec) return false;
  if (!(a.sm_scale > 0.f) || !std::isfinite(a.sm_scale)) return false;
  const uintptr_t at = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k) |
                       reinterpret_cast<uintptr_t>(a.v);
  if ((at & 15u) || (reinterpret_cast<uintptr_t>(a.out) & (4 * es - 1))) return false;
  const int64_t row_strides = a.q_stride_t | a.k_stride_t | a.v_stride_t;
  const int64_t batch_strides = a.batch > 1 ? (a.q_stride_b | a.k_stride_b | a.v_stride_b) : 0;
  if ((row_strides | batch_strides) & (vec - 1)) return false;
  if ((a.out_stride_t | (a.batch > 1 ? a.out_stride_b : 0)) & 3) return false;
  if (es == 4 && pairs <= MX_TWO_TURN_PAIRS_F32 && split_plan(a).splits == 1) {
    const MatrixShape s = matrix_shape(a);
    const int64_t wgs = (int64_t)a.batch * ((a.q_len + 32 * s.qw - 1) / (32 * s.qw));
    const bool one_turn = wgs <= (s.dp > 64 ? 256 : 512);
    if (!matrix_short(a, s) || !one_turn) return false;
  }
  return true;
}

// query tiles of 32 * qw rows; on short grids the keys go over about 256
// workgroups in ranges of whole tiles
MatrixPlan matrix_plan(const DenseArgs& a, const MatrixShape& s) {
  MatrixPlan mp{};
  const int64_t bq = 32 * s.qw, bk = s.kw * s.bkw;
  mp.nq = (int)((a.q_len + bq - 1) / bq);
  mp.nt = (int)((a.kv_len + bk - 1) / bk);
  mp.waves = s.qw * s.kw;
  const int64_t wgs = (int64_t)a.batch * mp.nq;
  int64_t n = wgs > 0 && wgs < SPLIT_TARGET_WGS ? SPLIT_TARGET_WGS / wgs : 1;
  const bool is_short = matrix_short(a, s);
  if (is_short) n = 1;
  if (n > mp.nt) n = mp.nt;
  if (n > MAX_SPLITS) n = MAX_SPLITS;
  const int64_t per = ((int64_t)mp.nt + n - 1) / n;   // tiles per range
  mp.splits = (int)((mp.nt + per - 1) / per);
  mp.chunk = mp.splits > 1 ? (int)(per * bk) : a.kv_len;
  mp.accoff = (2 * (int64_t)a.batch * a.q_len * mp.splits + 3) / 4 * 4;
  mp.again = is_short && a.dtype != IAK_DTYPE_F32;
  mp.skip = !is_short && causal_skip(a);
  return mp;
}

// key-tile flags are needed where tiles are skipped, or a weight is split and not looked after
// in the kernel
bool matrix_flags(const DenseArgs& a, const MatrixPlan& mp) {
  return mp.skip || (a.dtype != IAK_DTYPE_F32 && !mp.again);
}

size_t matrix_partial_bytes(const DenseArgs& a, const MatrixPlan& mp) {
  if (mp.splits <= 1) return 0;
  return ((size_t)mp.accoff + (size_t)a.batch * a.q_len * mp.splits * (size_t)a.v_dim) * sizeof(float);
}

size_t matrix_workspace(const DenseArgs& a) {
  const MatrixPlan mp = matrix_plan(a, matrix_shape(a));
  const size_t flags = matrix_flags(a, mp) ? (size_t)a.batch * mp.nt * mp.waves * sizeof(int32_t) : 0;
  const size_t total = matrix_partial_bytes(a, mp) + flags;
  return total ? total : IAK_DENSE_NO_SCRATCH;   // a workspace at all says that the form may run
}

template <typename T, int DP, int QW, int KW, int BKW, bool GEN>
void launch_matrix_gen(const DenseArgs& a, const MatrixPlan& mp, hipStream_t stream) {
  const dim3 grid((unsigned)((int64_t)a.batch * mp.nq * mp.splits)), block(64 * QW * KW);
  if constexpr (sizeof(T) == 2 && DP <= 128) {
    if (mp.again) {
      hipLaunchKernelGGL((dense_short_kernel<T, DP, QW, KW, BKW, GEN>), grid, block, 0, stream, a, mp);
      return;
    }
  }
  hipLaunchKernelGGL((dense_matrix_kernel<T, DP, QW, KW, BKW, GEN>), grid, block, 0, stream, a, mp);
}

template <typename T, int DP, int QW, int KW, int BKW>
void launch_matrix_cfg(const DenseArgs& a, const MatrixPlan& mp, hipStream_t stream) {
  if (general(a)) launch_matrix_gen<T, DP, QW, KW, BKW, true>(a, mp, stream);
  else launch_matrix_gen<T, DP, QW, KW, BKW, false>(a, mp, stream);
}

template <typename T, int DP>
void launch_matrix_dims(const DenseArgs& a, const MatrixShape& s, const MatrixPlan& mp,
                        hipStream_t stream) {
  constexpr int BKW = sizeof(T) == 4 ? 32 : 64;
  if constexpr (DP <= 128) {
    if constexpr (sizeof(T) == 2) {
      if (s.qw == 4 && s.kw == 2) return launch_matrix_cfg<T, DP, 4, 2, 64>(a, mp, stream);
    }
    if (s.kw == 4) return launch_matrix_cfg<T, DP, 1, 4, 32>(a, mp, stream);
    if (s.kw == 2) return launch_matrix_cfg<T, DP, 2, 2, 32>(a, mp, stream);
  }
  launch_matrix_cfg<T, DP, 4, 1, BKW>(a, mp, stream);
}

template <typename T>
void launch_matrix(const DenseArgs& a, void* workspace, hipStream_t stream) {
  const MatrixShape s = matrix_shape(a);
  MatrixPlan mp = matrix_plan(a, s);
  mp.ws = static_cast<float*>(workspace);
  const bool flags = matrix_flags(a, mp);
  if (flags) mp.flags = reinterpret_cast<int32_t*>(static_cast<char*>(workspace) + matrix_partial_bytes(a, mp));
  if (s.dp == 64) launch_matrix_dims<T, 64>(a, s, mp, stream);
  else if (s.dp == 128) launch_matrix_dims<T, 128>(a, s, mp, stream);
  if constexpr (sizeof(T) == 2) {
    if (s.dp == 96) launch_matrix_dims<T, 96>(a, s, mp, stream);
    else if (s.dp == 192) launch_matrix_dims<T, 192>(a, s, mp, stream);
    else if (s.dp == 256) launch_matrix_dims<T, 256>(a, s, mp, stream);
  }
  const int64_t rows = (int64_t)a.batch * a.q_len;
  if (mp.splits > 1) {
    const DenseSplit sp{mp.splits, mp.chunk, mp.ws};
    const int log2 = general(a) ? 0 : 1;
    if (flags)
      hipLaunchKernelGGL((dense_merge_kernel<T, true>), dim3((unsigned)rows), dim3(MERGE_THREADS), 0, stream, a, sp, mp,
                         mp.accoff, log2);
    else
      hipLaunchKernelGGL((dense_merge_kernel<T, false>), dim3((unsigned)rows), dim3(MERGE_THREADS), 0, stream, a, sp, mp,
                         mp.accoff, log2);
  } else if (flags) {
    const int64_t per = a.batch < 256 ? (256 + a.batch - 1) / a.batch : 1;
    hipLaunchKernelGGL(dense_fixup_kernel<T>, dim3((unsigned)(a.batch * per)), dim3(256), 0, stream, a, mp);
  }
}

template <typename T>
void launch_typed(const DenseArgs& a, void* workspace, hipStream_t stream) {
  if (workspace && matrix_applies(a)) return launch_matrix<T>(a, workspace, stream);
  DenseSplit sp = split_plan(a);
  if (!workspace) sp = DenseSplit{1, a.kv_len, nullptr};
  sp.ws = static_cast<float*>(workspace);
  if (a.kv_index) launch_rows<T, 1>(a, sp, stream);
  else launch_rows<T, 0>(a, sp, stream);
}

}  // namespace

// One object per element type (the Makefile compiles this file three times, side by side).
#if defined(IAK_DENSE_F16)
hipError_t launch_dense_f16(const iak_dense_attention_args& args, const int64_t* kv_index, void* workspace,
                            hipStream_t stream) {
  launch_typed<_Float16>(DenseArgs{args, kv_index}, workspace, stream);
  return hipGetLastError();
}
#elif defined(IAK_DENSE_BF16)
hipError_t launch_dense_bf16(const iak_dense_attention_args& args, const int64_t* kv_index, void* workspace,
                             hipStream_t stream) {
  launch_typed<bf16_bits>(DenseArgs{args, kv_index}, workspace, stream);
  return hipGetLastError();
}
#else
hipError_t launch_dense_f16(const iak_dense_attention_args& args, const int64_t* kv_index, void* workspace,
                            hipStream_t stream);
hipError_t launch_dense_bf16(const iak_dense_attention_args& args, const int64_t* kv_index, void* workspace,
                             hipStream_t stream);

size_t dense_attention_workspace(const iak_dense_attention_args& args) {
  const DenseArgs a{args, nullptr};   // the keys' rows change no size
  if (matrix_applies(a)) return matrix_workspace(a);
  const DenseSplit sp = split_plan(a);
  return sp.splits <= 1 ? 0 : (size_t)a.batch * a.q_len * sp.splits * (2 + (size_t)a.v_dim) * sizeof(float);
}

hipError_t launch_dense_attention(const iak_dense_attention_args& args, const int64_t* kv_index, void* workspace,
                                  hipStream_t stream) {
  if (args.dtype == IAK_DTYPE_F16) return launch_dense_f16(args, kv_index, workspace, stream);
  if (args.dtype == IAK_DTYPE_BF16) return launch_dense_bf16(args, kv_index, workspace, stream);
  launch_typed<float>(DenseArgs{args, kv_index}, workspace, stream);
  return hipGetLastError();
}
#endif

}  // namespace iak
