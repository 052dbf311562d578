// Latent context of the reference's MLA decode API in float32, for gfx950.
//
// Reference semantics: the Triton kernel and CPU path of mla_decode_triton
// (src/intent_attention/triton_mla_decode.py:47-107 and _mla_decode_cpu
// :155-186): each (batch, query position) row attends to the latent rows of
// the pages its page table lists -- page p is rows p*page_size ..
// (p+1)*page_size - 1 of C [rows, d_c], the last page of C possibly shorter --
// with scores (q . c) * sm_scale in float32, an online softmax, and context =
// sum(p c) / sum(p); zeros when no row is visited. The projection by W_VO
// that follows is mla_project.h's kernel, or torch's GEMM (see there).
//
// This is the reference API's arithmetic, not the serving path: the MFMA
// kernel of mla_decode.hip computes over paged f16 / FP8 / INT8 pools with f16
// operands, while this kernel keeps every product and sum in float32 over
// float32, float16 or bfloat16 inputs, any page size and any latent width up
// to 1,024 in one launch.
//
// Keys. The listed pages' rows form one key sequence: key j is row
// page_ids[j / page_size] * page_size + j % page_size of C (the division by a
// multiply-high and one correction, its magic number from the host); a key
// past the end of C (the last page's missing rows) takes no mass. A latent row
// is both the key and the value of its token, so it is loaded once.
//
// Calls with several query rows run on the matrix cores (mla_rows_matrix.h); what
// follows is the rows form, for the rest.
//
// Work split. Every query row attends to the same latent rows, so a
// workgroup takes four query rows once there are four (each latent row it
// loads serves all of them). A row group's keys go to `splits` workgroups of
// consecutive key ranges; splits > 1 only when the caller gives a workspace
// and there are fewer than 512 row groups with at least 256 keys, and a
// second kernel merges each row's ranges' (max, denominator, context) by
// log-sum-exp. A workgroup has WAVES waves (16 when the grid is short); wave w
// takes KEYS consecutive keys per step, loads their latent rows first
// (unconditionally, at clamped indices, the values of keys past the range
// zeroed at use) with the next step's rows in flight while this step's dot
// products are reduced (a DPP + lane-swap wave sum with the same bits in every
// lane). Lane l holds dims l, l + 64, ... of q and of the context. Each wave
// keeps a running max, denominator and context per row; the waves merge
// through the LDS.

#include <hip/hip_runtime.h>
#include <stdint.h>

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

struct bf16_bits { uint16_t b; };

__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(_Float16 x) { return (float)x; }
__device__ __forceinline__ float to_f32(bf16_bits x) { return __builtin_bit_cast(float, (uint32_t)x.b << 16); }

__device__ __forceinline__ float load_q(const void* p, int64_t i, int dtype) {
  if (dtype == IAK_DTYPE_F32) return reinterpret_cast<const float*>(p)[i];
  if (dtype == IAK_DTYPE_F16) return (float)reinterpret_cast<const _Float16*>(p)[i];
  return to_f32(reinterpret_cast<const bf16_bits*>(p)[i]);
}

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

// Sum over the 64 lanes, the same bits in every lane: each step adds two
// values that the partner lane adds in the other order (lane ^ 1 and lane ^ 2
// by quad permutes; then, with a quad's four lanes equal, the quads two and
// one places round the row of 16 by row rotates; then rows through the lane
// swaps).
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp<0xB1>(v);    // quad_perm [1, 0, 3, 2]
  v += dpp<0x4E>(v);    // quad_perm [2, 3, 0, 1]
  v += dpp<0x128>(v);   // row_ror:8
  v += dpp<0x124>(v);   // row_ror:4
  return xsum16_32(v);
}

struct RowSplit {
  int splits;        // workgroups per row group
  int chunk;         // keys per workgroup (the last may have fewer)
  int nkeys;         // num_selected * page_size
  uint32_t magic;    // floor(2^32 / page_size), or 2^32 - 1 for page_size 1
  int rows_per_wg;   // query rows per workgroup (1 or 4; RX_ROWS: the matrix form)
  float* ws;         // splits > 1: [n] max, [n] denominator, [n, d_c] context, n = rows * splits
  int64_t accoff;    // offset of the contexts in ws (floats)
  int log2;          // the maxima are in the exp2 domain
};

// The C row of key j: outside [0, num_rows) for a key past the end of C or of
// an invalid page id (the host rejects those; the kernel gives them no mass).
__device__ __forceinline__ int64_t key_row(const iak_mla_rows_args& a, const RowSplit& sp, uint32_t j) {
  uint32_t q = __umulhi(j, sp.magic);   // floor(j / page_size) or one less
  uint32_t r = j - q * (uint32_t)a.page_size;
  if (r >= (uint32_t)a.page_size) {
    ++q;
    r -= (uint32_t)a.page_size;
  }
  return (int64_t)a.page_ids[q] * a.page_size + r;
}

// T: latent element type; NPL: dims per lane (d_c <= 64 * NPL); KEYS keys per
// wave and step; WAVES waves per workgroup; R query rows per workgroup (every
// row attends to the same latent rows, so each loaded row serves all R)
template <typename T, int NPL, int KEYS, int WAVES, int R>
__global__ __launch_bounds__(64 * WAVES) void mla_rows_kernel(const iak_mla_rows_args a, const RowSplit sp) {
  __shared__ float part_acc[WAVES][R][64 * NPL];
  __shared__ float part_m[WAVES][R], part_l[WAVES][R];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t nrows = (int64_t)a.batch * a.q_len;
  const int64_t item = blockIdx.x;   // group * splits + split; rows R * group .. R * group + R - 1
  const int64_t group = item / sp.splits;
  const int split = (int)(item - group * sp.splits);
  const int dc = a.latent_dim;
  const int lo = split * sp.chunk;
  const int hi = sp.nkeys - lo < sp.chunk ? sp.nkeys : lo + sp.chunk;   // keys lo .. hi - 1
  const float NEG_INF = -__builtin_inff();

  int dd[NPL];
  bool ok[NPL];
#pragma unroll
  for (int jj = 0; jj < NPL; ++jj) {
    const int d = lane + 64 * jj;
    ok[jj] = d < dc;
    dd[jj] = ok[jj] ? d : dc - 1;
  }
  float q[R][NPL], acc[R][NPL], m[R], l[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t row = group * R + r;
    const int64_t rowc = row < nrows ? row : nrows - 1;   // a row past the end repeats the last (not written)
    const int64_t b = rowc / a.q_len;
    const int t = (int)(rowc - b * a.q_len);
    const int64_t qoff = b * a.q_stride_b + (int64_t)t * a.q_stride_t;
#pragma unroll
    for (int jj = 0; jj < NPL; ++jj) {
      const float qx = load_q(a.q, qoff + dd[jj], a.q_dtype);
      q[r][jj] = ok[jj] ? qx : 0.f;
      acc[r][jj] = 0.f;
    }
    m[r] = NEG_INF;
    l[r] = 0.f;
  }
  const T* lat = reinterpret_cast<const T*>(a.latents);
  // a step's latent rows, loaded at clamped indices (a key past the range
  // reads the range's last key, a row outside C its first or last row)
  float cn[KEYS][NPL];
  int64_t rows_n[KEYS];
  auto load_step = [&](int j0) {
#pragma unroll
    for (int u = 0; u < KEYS; ++u) {
      const int jc = j0 + u < hi ? j0 + u : hi - 1;
      const int64_t r = key_row(a, sp, (uint32_t)jc);
      rows_n[u] = r;
      const int64_t rc = r < 0 ? 0 : (r < a.num_rows ? r : a.num_rows - 1);
      const T* cr = lat + rc * a.latent_stride;
#pragma unroll
      for (int jj = 0; jj < NPL; ++jj) cn[u][jj] = to_f32(cr[dd[jj]]);
    }
  };
  if (lo + KEYS * w < hi) load_step(lo + KEYS * w);
  for (int j0 = lo + KEYS * w; j0 < hi; j0 += KEYS * WAVES) {
    float cv[KEYS][NPL];
    bool live[KEYS];
#pragma unroll
    for (int u = 0; u < KEYS; ++u) {
      live[u] = j0 + u < hi && rows_n[u] >= 0 && rows_n[u] < a.num_rows;   // wave-uniform
#pragma unroll
      for (int jj = 0; jj < NPL; ++jj) cv[u][jj] = live[u] && ok[jj] ? cn[u][jj] : 0.f;
    }
    // the next step's rows (clamped into the range on the last step)
    load_step(j0 + KEYS * WAVES < hi ? j0 + KEYS * WAVES : j0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float s[KEYS];
#pragma unroll
      for (int u = 0; u < KEYS; ++u) {
        float x = 0.f;
#pragma unroll
        for (int jj = 0; jj < NPL; ++jj) x = __builtin_fmaf(q[r][jj], cv[u][jj], x);
        s[u] = x;
      }
      float smax = NEG_INF;
#pragma unroll
      for (int u = 0; u < KEYS; ++u) {
        const float x = wave_sum(s[u]) * a.sm_scale;
        s[u] = live[u] ? x : NEG_INF;
        smax = fmaxf(smax, s[u]);
      }
      const float mn = fmaxf(m[r], smax);
      if (mn > m[r]) {   // wave-uniform
        const float alpha = expf(m[r] - mn);   // 0 while nothing was seen (m = -inf)
        l[r] *= alpha;
#pragma unroll
        for (int jj = 0; jj < NPL; ++jj) acc[r][jj] *= alpha;
        m[r] = mn;
      }
#pragma unroll
      for (int u = 0; u < KEYS; ++u) {
        const float e = s[u] == NEG_INF ? 0.f : expf(s[u] - m[r]);   // keys that are not rows take no mass
        l[r] += e;
#pragma unroll
        for (int jj = 0; jj < NPL; ++jj) acc[r][jj] = __builtin_fmaf(e, cv[u][jj], acc[r][jj]);
      }
    }
  }

#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (lane == 0) {
      part_m[w][r] = m[r];
      part_l[w][r] = l[r];
    }
#pragma unroll
    for (int jj = 0; jj < NPL; ++jj) part_acc[w][r][lane + 64 * jj] = acc[r][jj];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t row = group * R + r;
    if (row >= nrows) break;   // workgroup-uniform
    float M = NEG_INF;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) M = fmaxf(M, part_m[k][r]);
    float wt[WAVES], L = 0.f;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) {
      wt[k] = part_m[k][r] == NEG_INF ? 0.f : expf(part_m[k][r] - M);   // 0 for a wave that saw no row
      L += wt[k] * part_l[k][r];
    }
    if (sp.splits > 1) {
      // this range's partial of the row: max, denominator and unnormalised context
      const int64_t n = nrows * sp.splits;
      const int64_t slot = row * sp.splits + split;
      if (threadIdx.x == 0) {
        sp.ws[slot] = M;
        sp.ws[n + slot] = L;
      }
      float* wacc = sp.ws + sp.accoff + slot * dc;
      for (int d = threadIdx.x; d < dc; d += 64 * WAVES) {
        float A = 0.f;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) A = __builtin_fmaf(wt[k], part_acc[k][r][d], A);
        wacc[d] = A;
      }
    } else {
      float* out = a.context + row * dc;
      for (int d = threadIdx.x; d < dc; d += 64 * WAVES) {
        float A = 0.f;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) A = __builtin_fmaf(wt[k], part_acc[k][r][d], A);
        out[d] = L > 0.f ? A / L : 0.f;   // zeros when no row was visited
      }
    }
  }
}

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

// The log-sum-exp merge of a row's `splits` partials (splits <= MAX_SPLITS): one
// workgroup per row and 64 dims, wave w over every fourth split with eight loads
// in flight; the split weights are in the LDS, the waves meet there too. (One
// workgroup per row left 32 rows on 32 CUs: 256 splits x 576 dims 8.5 us.)
__global__ __launch_bounds__(MERGE_THREADS) void mla_rows_merge_kernel(const iak_mla_rows_args a,
                                                                       const RowSplit sp) {
  constexpr int WAVES = MERGE_THREADS / 64;
  __shared__ float wt[MAX_SPLITS];
  __shared__ float red[WAVES];
  __shared__ float part[WAVES][64];
  const int64_t row = blockIdx.x;
  const int S = sp.splits, dc = a.latent_dim;
  const int64_t n = (int64_t)gridDim.x * S;
  const float* wm = sp.ws + row * S;
  const float* wl = sp.ws + n + row * S;
  const float NEG_INF = -__builtin_inff();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int d = blockIdx.y * 64 + lane, dcl = d < dc ? d : dc - 1;
  const float* wacc = sp.ws + sp.accoff + row * S * dc + dcl;
  float mx = NEG_INF;
  for (int s = threadIdx.x; s < S; s += MERGE_THREADS) mx = fmaxf(mx, wm[s]);
  const float M = block_reduce<true>(mx, red);
  float ls = 0.f;
  for (int s = threadIdx.x; s < S; s += MERGE_THREADS) {
    // 0 for a range that visited no row
    const float x = wm[s] == NEG_INF ? 0.f : (sp.log2 ? __builtin_amdgcn_exp2f(wm[s] - M) : expf(wm[s] - M));
    wt[s] = x;
    ls += x * wl[s];
  }
  const float L = block_reduce<false>(ls, red);   // its barriers also publish wt[]
  float A = 0.f;
  int s = w;
  for (; s + 7 * WAVES < S; s += 8 * WAVES) {
    float x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = wacc[(int64_t)(s + u * WAVES) * dc];
#pragma unroll
    for (int u = 0; u < 8; ++u) A = __builtin_fmaf(wt[s + u * WAVES], x[u], A);
  }
  for (; s < S; s += WAVES) A = __builtin_fmaf(wt[s], wacc[(int64_t)s * dc], A);
  part[w][lane] = A;
  __syncthreads();
  if (w == 0 && d < dc) {
    A = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    a.context[row * dc + d] = L > 0.f ? A / L : 0.f;
  }
}

#include "mla_rows_matrix.h"
#include "mla_project.h"

// MAXW: the most waves per workgroup whose registers and LDS fit
template <typename T, int NPL, int KEYS, int MAXW, int R>
void launch_items(const iak_mla_rows_args& a, const RowSplit& sp, int64_t items, hipStream_t stream) {
  // waves per workgroup: about 4,096 waves in the grid (16 per CU), between 4 and MAXW
  const int64_t want = (4096 + items - 1) / items;
  const dim3 grid((unsigned)items);
  if (MAXW >= 16 && want >= 16)
    hipLaunchKernelGGL((mla_rows_kernel<T, NPL, KEYS, MAXW >= 16 ? 16 : 4, R>), grid, dim3(1024), 0, stream, a, sp);
  else if (want >= 8)
    hipLaunchKernelGGL((mla_rows_kernel<T, NPL, KEYS, 8, R>), grid, dim3(512), 0, stream, a, sp);
  else
    hipLaunchKernelGGL((mla_rows_kernel<T, NPL, KEYS, 4, R>), grid, dim3(256), 0, stream, a, sp);
}

template <typename T, int R>
void launch_rows(const iak_mla_rows_args& a, const RowSplit& sp, hipStream_t stream) {
  const int64_t rows = (int64_t)a.batch * a.q_len;
  const int64_t items = (rows + R - 1) / R * sp.splits;
  const int npl = (a.latent_dim + 63) / 64;
  // per lane: R * NPL query and context values, KEYS * NPL latent values in flight (twice, pipelined)
  if (npl <= 1) launch_items<T, 1, 8, 16, R>(a, sp, items, stream);
  else if (npl <= 2) launch_items<T, 2, 8, 16, R>(a, sp, items, stream);
  else if (npl <= 4) launch_items<T, 4, (R > 1 ? 4 : 8), (R > 1 ? 8 : 16), R>(a, sp, items, stream);
  else if (npl <= 9) launch_items<T, 9, (R > 1 ? 2 : 4), 8, R>(a, sp, items, stream);
  else launch_items<T, 16, 2, (R > 1 ? 4 : 8), R>(a, sp, items, stream);
}

template <typename T>
void launch_typed(const iak_mla_rows_args& a, const RowSplit& sp, hipStream_t stream) {
  const int64_t rows = (int64_t)a.batch * a.q_len;
  if (sp.rows_per_wg == RX_ROWS) {
    const dim3 grid((unsigned)((rows + RX_ROWS - 1) / RX_ROWS * sp.splits));
    const int nd = rx_dim_tiles(a.latent_dim), waves = (a.latent_dim + 32 * nd - 1) / (32 * nd);
    const dim3 block(64 * waves);
    if (nd == 1 && waves <= 4) hipLaunchKernelGGL((mla_rows_matrix_kernel<T, 1, 4>), grid, block, 0, stream, a, sp);
    else if (nd == 1) hipLaunchKernelGGL((mla_rows_matrix_kernel<T, 1, 8>), grid, block, 0, stream, a, sp);
    else if (nd == 2) hipLaunchKernelGGL((mla_rows_matrix_kernel<T, 2, 8>), grid, block, 0, stream, a, sp);
    else hipLaunchKernelGGL((mla_rows_matrix_kernel<T, 3, 8>), grid, block, 0, stream, a, sp);
  } else if (sp.rows_per_wg == 4) {
    launch_rows<T, 4>(a, sp, stream);
  } else {
    launch_rows<T, 1>(a, sp, stream);
  }
  if (sp.splits > 1)
    hipLaunchKernelGGL(mla_rows_merge_kernel, dim3((unsigned)rows, (unsigned)((a.latent_dim + 63) / 64)),
                       dim3(MERGE_THREADS), 0, stream, a, sp);
}

// Splits per row group: with fewer than 512 groups and SPLIT_MIN_KEYS keys or
// more, a group's keys go over about SPLIT_TARGET_WGS workgroups in ranges of
// at least RANGE_MIN_KEYS keys
// (at most MAX_SPLITS ranges). Four rows per workgroup when that still gives
// 128 workgroups or more, one otherwise (few rows over few keys keep their
// parallelism).
RowSplit plan_for(const iak_mla_rows_args& a, int R) {
  const int64_t nkeys = (int64_t)a.num_selected * a.page_size;
  RowSplit sp{1, (int)nkeys, (int)nkeys, 0u, R, nullptr, 0, 0};
  sp.magic = a.page_size == 1 ? 0xFFFFFFFFu : (uint32_t)((1ull << 32) / (uint64_t)a.page_size);
  const int64_t rows = (int64_t)a.batch * a.q_len;
  const int64_t groups = (rows + R - 1) / R;
  if (rows <= 0 || groups >= 512 || nkeys < SPLIT_MIN_KEYS) return sp;
  int64_t s = (SPLIT_TARGET_WGS + groups - 1) / groups;
  const int64_t by_keys = nkeys / RANGE_MIN_KEYS;
  if (s > by_keys) s = by_keys;
  if (s > MAX_SPLITS) s = MAX_SPLITS;   // the merge holds the split weights in the LDS
  if (s <= 1) return sp;
  const int64_t chunk = (nkeys + s - 1) / s;
  sp.splits = (int)((nkeys + chunk - 1) / chunk);
  sp.chunk = (int)chunk;
  sp.accoff = 2 * rows * sp.splits;
  return sp;
}

// From this many query rows and (row, key) pairs on the matrix form is the faster
// one, by the 32-dim tiles a wave of it holds (its chain grows with them). Both
// forms, us per call (float16 latents, 30 calls): 128 dims 4 x 8,192 22.5 / 12.3,
// 16 x 2,048 21.9 / 10.0; 512 dims 32 x 512 = 16,384 12.9 / 16.7, 16 x 2,048 =
// 32,768 21.1 / 16.6, 4 x 8,192 21.9 / 18.9; 576 dims 8 x 8,192 = 65,536 22.9 /
// 25.0, 64 x 2,048 30.4 / 25.0, 16 x 8,192 = 131,072 29.7 / 26.5, 32 x 8,192
// 43.8 / 28.9 (52 before the merge went over the dims as well).
#ifndef RX_MIN_ROWS
#define RX_MIN_ROWS 4
#endif
#ifdef RX_MIN_PAIRS
constexpr double rx_min_pairs(int) { return RX_MIN_PAIRS; }
#else
constexpr double rx_min_pairs(int nd) { return nd == 1 ? 2048 : nd == 2 ? 32768 : 131072; }
#endif

// whole 16-byte pieces of every latent row, at most 768 dims
bool matrix_applies(const iak_mla_rows_args& a) {
  const int vec = a.latent_dtype == IAK_DTYPE_F32 ? 4 : 8;
  const int64_t rows = (int64_t)a.batch * a.q_len, nkeys = (int64_t)a.num_selected * a.page_size;
  return rows >= RX_MIN_ROWS && nkeys > 0 && (double)rows * nkeys >= rx_min_pairs(rx_dim_tiles(a.latent_dim)) && a.num_rows > 0 &&
         rx_dim_tiles(a.latent_dim) <= RX_MAX_ND && a.latent_dim % vec == 0 && a.sm_scale > 0.f &&
         !((reinterpret_cast<uintptr_t>(a.latents) | reinterpret_cast<uintptr_t>(a.context)) & 15u) &&
         a.latent_stride % vec == 0;
}

// 32 query rows per workgroup, the keys over about 256 workgroups in ranges of
// whole 32-key tiles
RowSplit matrix_plan(const iak_mla_rows_args& a) {
  const int64_t nkeys = (int64_t)a.num_selected * a.page_size, rows = (int64_t)a.batch * a.q_len;
  RowSplit sp{1, (int)nkeys, (int)nkeys, 0u, RX_ROWS, nullptr, 0, 1};
  sp.magic = a.page_size == 1 ? 0xFFFFFFFFu : (uint32_t)((1ull << 32) / (uint64_t)a.page_size);
  const int64_t groups = (rows + RX_ROWS - 1) / RX_ROWS, tiles = (nkeys + RX_KEYS - 1) / RX_KEYS;
  int64_t s = groups < SPLIT_TARGET_WGS ? SPLIT_TARGET_WGS / groups : 1;
  if (s > tiles) s = tiles;
  if (s > MAX_SPLITS) s = MAX_SPLITS;
  if (s <= 1) return sp;
  const int64_t per = (tiles + s - 1) / s;
  sp.splits = (int)((tiles + per - 1) / per);
  sp.chunk = sp.splits > 1 ? (int)(per * RX_KEYS) : (int)nkeys;
  sp.accoff = (2 * rows * sp.splits + 3) / 4 * 4;
  return sp;
}

// Without a workspace nothing is split; few query rows then leave most of the chip idle, and the
// rows form, with its workgroup per row or four, is the one that uses more of it (float16
// latents, us: 32 rows x 8,192 keys x 576 986, this form 2,514; 2,000 x 1,024 x 576 266 / 317).
RowSplit split_plan(const iak_mla_rows_args& a, bool workspace) {
  if (matrix_applies(a)) {
    const RowSplit sp = matrix_plan(a);
    if (workspace || sp.splits == 1) return sp;
  }
  const int64_t rows = (int64_t)a.batch * a.q_len;
  if (rows >= 4) {
    const RowSplit sp4 = plan_for(a, 4);
    if ((rows + 3) / 4 * sp4.splits >= 128) return sp4;
  }
  return plan_for(a, 1);
}

}  // namespace

size_t mla_rows_workspace(const iak_mla_rows_args& a) {
  const RowSplit sp = split_plan(a, true);
  if (sp.splits <= 1) return 0;
  return ((size_t)sp.accoff + (size_t)a.batch * a.q_len * sp.splits * (size_t)a.latent_dim) * sizeof(float);
}

hipError_t launch_mla_rows(const iak_mla_rows_args& a, void* workspace, hipStream_t stream) {
  RowSplit sp = split_plan(a, workspace != nullptr);
  if (!workspace) sp.splits = 1, sp.chunk = sp.nkeys;
  sp.ws = static_cast<float*>(workspace);
  if (a.latent_dtype == IAK_DTYPE_F32) launch_typed<float>(a, sp, stream);
  else if (a.latent_dtype == IAK_DTYPE_F16) launch_typed<_Float16>(a, sp, stream);
  else launch_typed<bf16_bits>(a, sp, stream);
  return hipGetLastError();
}

hipError_t launch_mla_project(const iak_mla_project_args& a, hipStream_t stream) {
  const dim3 grid((unsigned)(a.d_out / PJ_COLS), (unsigned)((a.rows + PJ_ROWS - 1) / PJ_ROWS)), block(64 * PJ_WAVES);
  if (a.w_dtype == IAK_DTYPE_F32) hipLaunchKernelGGL(mla_project_kernel<float>, grid, block, 0, stream, a);
  else if (a.w_dtype == IAK_DTYPE_F16) hipLaunchKernelGGL(mla_project_kernel<_Float16>, grid, block, 0, stream, a);
  else hipLaunchKernelGGL(mla_project_kernel<bf16_bits>, grid, block, 0, stream, a);
  return hipGetLastError();
}

}  // namespace iak
