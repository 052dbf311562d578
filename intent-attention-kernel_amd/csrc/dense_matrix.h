// Tiled dense attention on the matrix cores: the form of dense_attention.hip
// for several query rows per batch entry. Included by that file only.
//
// A workgroup of QW x KW (four or eight) waves takes QW x 32 query rows of one
// batch entry and walks key tiles of KW x BKW keys; wave (qw, kw) owns 32 query
// rows and the kw-th BKW keys of every tile (KW > 1 keeps the waves busy when
// there are few query rows, and puts two on a SIMD when there are few workgroups;
// the waves' partial results meet in the LDS at the end).
// K and V tiles go through registers into the LDS as they lie in memory, the
// next tile's loads in flight while this tile is computed.
//   scores  S^T[32 keys x 32 rows] = K . Q^T: A operand K[key = lane % 32], B
//           operand Q[row = lane % 32], both 16-byte pieces 2s + h of a row
//           (h = lane / 32). The result leaves 16 keys of one query row in a
//           lane: keys 8 (r / 4) + 4 h + r % 4.
//   softmax per lane over its keys, one lane swap with lane ^ 32 for the other
//           half; the running max moves only when a tile exceeds it by more
//           than 2^8 (float16 2^3, float32 at once), so the accumulators are rarely
//           rescaled.
//   values  O^T[32 dims x 32 rows] += V^T . P^T: P is the score result as it
//           lies in the registers, V^T comes out of the [key][dim] tile
//           (16-bit: the transposing read ds_read_b64_tr_b16).
// Arithmetic. Every product is exact or float32 and every sum is float32.
// float16 / bfloat16 inputs: Q.K products are exact on the 16-bit matrix
// instructions; the float32 weights are split into 16-bit parts whose sum
// carries 22 bits or more (float16: two parts of p * 2^12, to 2^-37 of the row's
// largest weight; bfloat16: three), one matrix instruction per part. float32 inputs: v_mfma_f32_32x32x2_f32.
//
// Non-finite and large values come out as in the plain sum. Four shortcuts would answer
// differently for them: a split weight times an infinite V (inf * 0 in the low part);
// the keys past a range's last one, which fill up its last tile with weight 0 (0 * inf);
// the lagging maximum, whose weights of up to 2^8 take a large finite V over the
// range; and causal tiles past the diagonal, which are not visited (a NaN or an
// overflowing score there makes its row NaN, an infinite V a zero weight's
// product NaN).
//   float32 rows, and 16-bit ones of short calls (dense_short_kernel): V of the keys past
//           the range is zeros, and the maximum does not lag (float16: by 2^3, its V cannot
//           overflow). A workgroup of a short call whose rows end in a sum that is not
//           finite walks its keys once more, with 1 for every weight above 0: the sums
//           are infinite or NaN where the plain ones are, and those are written.
//   the others, and every call with tiles that are not visited: each key tile is checked
//           once, by one of the workgroups that loads it, and its flag (K and V below
//           2^59 or not) goes to the workspace; the kernel that follows (the merge,
//           or dense_fixup_kernel) recomputes every row of a flagged batch entry
//           with dense_row.
// A short call is a fifth shorter without that second launch (16 heads x 32 rows x 256 keys
// x 64 in float16 24 us, now 19, the row form 18.6); in a long one the second walk's
// registers cost as much (32 heads x 2,048 rows x 128, causal: 82 / 87 us).
#ifndef IAK_DENSE_MATRIX_H
#define IAK_DENSE_MATRIX_H

typedef float f16v __attribute__((ext_vector_type(16)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

constexpr int MX_MAX_DIM = 256;      // 16-bit inputs
constexpr int MX_MAX_DIM_F32 = 128;  // float32: Q, scores and context of wider rows spill
constexpr float LOG2E = 1.44269504088896340736f;
constexpr float LARGE = 1e5f;   // scores (exp2 domain) whose rounding reaches 2^-8

struct MatrixPlan {
  int splits;      // key ranges per (batch entry, query tile)
  int chunk;       // keys per range, whole tiles
  int nq;          // query tiles per batch entry
  int nt;          // key tiles per batch entry
  int skip;        // causal: tiles past the diagonal are not visited
  int again;       // 16-bit: the kernel with the second walk
  int64_t accoff;  // offset of the partial contexts in ws (floats)
  float* ws;       // splits > 1: the partials
  int waves;       // waves of a workgroup
  int32_t* flags;  // [batch][nt][waves], or null (nothing to check)
};

template <typename T> struct MxElem;   // operand vector of 16 bytes, matrix product, parts of a weight
template <> struct MxElem<_Float16> {
  typedef h8 vec;
  static constexpr int PARTS = 2;
  static __device__ __forceinline__ f16v mfma(vec a, vec b, f16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};
template <> struct MxElem<bf16_bits> {
  typedef b8 vec;
  static constexpr int PARTS = 3;
  static __device__ __forceinline__ f16v mfma(vec a, vec b, f16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct MxElem<float> {
  typedef f4 vec;
  static constexpr int PARTS = 1;
};

// any of a 16-byte piece's values at or above 2^59 in magnitude (float16: not finite):
// below that, a score of 256 dims cannot overflow
template <typename T> __device__ __forceinline__ bool mx_large(u4 x) {
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (sizeof(T) == 4) {
      bad |= (x[i] & 0x7FFFFFFFu) >= ((127u + 59u) << 23);
    } else {
      constexpr uint32_t lim = __is_same(T, _Float16) ? 0x7C00u : ((127u + 59u) << 7);
      bad |= (x[i] & 0x7FFFu) >= lim || ((x[i] >> 16) & 0x7FFFu) >= lim;
    }
  }
  return bad;
}

// v as it is rounded: not contracted into the sum that follows
__device__ __forceinline__ float rounded(float v) {
  asm volatile("" : "+v"(v));
  return v;
}

// The 16-bit part of two weights, packed; x0 and x1 keep what it leaves out
// (`rest`), exactly.
template <typename T> __device__ __forceinline__ uint32_t mx_take_part(float& x0, float& x1, bool rest) {
  typedef float f2v __attribute__((ext_vector_type(2)));
  uint32_t p;
  if constexpr (__is_same(T, _Float16)) {
    p = bits(__builtin_convertvector((f2v{x0, x1}), h2));
    if (rest) {   // x - part as one mixed-precision fma each
      asm("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel_hi:[1,0,0]" : "+v"(x0) : "v"(p));
      asm("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(x1) : "v"(p));
    }
  } else {
    typedef __bf16 b2v __attribute__((ext_vector_type(2)));
    p = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2v{x0, x1}), b2v));
    if (rest) {
      x0 -= u2f(p << 16);
      x1 -= u2f(p & 0xFFFF0000u);
    }
  }
  return p;
}

// max / sum of a value over lanes l and l ^ 32 (see xmax16_32 for the asm block)
__device__ __forceinline__ float xmax32(float v) {
  float t;
  asm volatile("v_mov_b32 %1, %0\n\ts_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_max_f32 %0, %0, %1"
               : "+v"(v), "=&v"(t));
  return v;
}
__device__ __forceinline__ float xsum32(float v) {
  float t;
  asm volatile("v_mov_b32 %1, %0\n\ts_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_add_f32 %0, %0, %1"
               : "+v"(v), "=&v"(t));
  return v;
}

// LDS position (16-byte pieces) of piece c of row r, rows of RB bytes. K: the 16
// lanes that read one piece of 16 rows touch every bank group once. V, 16-bit:
// a transposing read's four rows x 64 bytes spread over the banks; float32:
// rows r and r + 4 of one read lie in different halves.
template <int RB> __device__ __forceinline__ int k_piece(int r, int c) {
  constexpr int P = RB % 256 == 0 ? 1 : (RB % 128 == 0 ? 2 : 4);   // rows until the bank offset repeats
  return c ^ ((r / P) & (16 / P - 1));
}
template <int RB, int ES> __device__ __forceinline__ int v_piece(int r, int c) {
  if constexpr (ES == 4) return c ^ (8 * ((r >> 2) & 1));
  constexpr int P = RB % 256 == 0 ? 1 : (RB % 128 == 0 ? 2 : 4);
  return c ^ (4 * ((r / P) & (4 / P - 1)));
}

// float32 scores of 32 keys x 32 rows over the pieces 2c + h, c = C0 .. C0 + N - 1
// (`kt` + `koff`: the lane's piece h in the LDS). Chains of 8 dims are added pairwise,
// which keeps the rounding error of dense_row's wave-wide tree sum; one chain
// over 128 dims has twice it.
template <int C0, int N, int NQ>
__device__ __forceinline__ f16v mx_score_tree(const char* kt, int koff, const f4 (&q)[NQ]) {
  if constexpr (N == 1) {
    f16v s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
    const f4 kf = *reinterpret_cast<const f4*>(kt + (koff ^ (32 * C0)));
#pragma unroll
    for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], q[C0][e], s, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);   // one chain after the other: interleaved, they spill
    return s;
  } else {
    constexpr int H = N / 2;
    const f16v x = mx_score_tree<C0, H, NQ>(kt, koff, q);
    return x + mx_score_tree<C0 + H, N - H, NQ>(kt, koff, q);
  }
}

template <typename T, int DP, int QW, int KW, int BKW, bool GEN> struct MxCfg {
  static_assert((QW * KW == 4 || QW * KW == 8) && BKW % 32 == 0 && DP % 32 == 0, "whole 32 x 32 tiles");
  static constexpr int THREADS = 64 * QW * KW;
  static constexpr int ES = sizeof(T);
  static constexpr int RB = DP * ES;               // LDS row bytes
  static constexpr int CH = RB / 16;               // 16-byte pieces per row
  static constexpr int EPC = 16 / ES;              // elements per piece
  static constexpr int BQ = 32 * QW, BK = KW * BKW;
  static constexpr int TILE = BK * RB;             // bytes of a K (or V) tile
  // float32 tiles: K and V of the next tile go through the same registers, one
  // behind the other (K while the scores are computed, V behind the values),
  // into the one buffer; a tile's 64 to 128 matrix instructions of 64 cycles
  // cover the loads. 16-bit tiles: both at once, two buffers where they fit.
  static constexpr bool STAGED = ES == 4;
  static constexpr int NB = !STAGED && 4 * TILE <= 131072 ? 2 : 1;
  // one wave per query group: each wave loads the keys it computes and no other,
  // so the waves need no barrier
  static constexpr bool PRIV = QW == 1;
  static constexpr int LDS = NB * 2 * TILE;
  static constexpr int NCH = BK * CH / THREADS; // pieces per thread and tile
  static constexpr int NSB = BKW / 32, NDV = DP / 32;
  static_assert(BK * CH % THREADS == 0, "whole pieces per thread");
  static_assert(KW == 1 || KW * 32 * QW * DP * 4 <= LDS, "the waves' contexts meet in the tile buffers");
};

template <typename T, int DP, int QW, int KW, int BKW, bool GEN>
__global__ __launch_bounds__(64 * QW * KW, (sizeof(T) == 2 ? DP <= 128 && QW == 4 : DP <= 64) ? 2 : 1)
void dense_matrix_kernel(const DenseArgs a, const MatrixPlan mp) {
  constexpr bool AGAIN = false, PLAIN = false;
  __shared__ u4 mx_lds[MxCfg<T, DP, QW, KW, BKW, GEN>::LDS / 16];
  char* const lds = reinterpret_cast<char*>(mx_lds);
  __shared__ float red_m[KW > 1 ? KW : 1][32 * QW], red_l[KW > 1 ? KW : 1][32 * QW];
#define MX_DONE return
#include "dense_walk.h"
#undef MX_DONE
}

// A walk over the keys in the kernel of short calls; whether this lane's sums are not all finite.
// PLAIN: the second walk, with 1 for every weight above 0, in one part.
template <typename T, int DP, int QW, int KW, int BKW, bool GEN, bool PLAIN>
__device__ __forceinline__ bool mx_walk(const DenseArgs& a, const MatrixPlan& mp, char* const lds,
                                        float (*red_m)[32 * QW], float (*red_l)[32 * QW]) {
  constexpr bool AGAIN = true;
#define MX_DONE return again
#include "dense_walk.h"
#undef MX_DONE
  return again;
}

template <typename T, int DP, int QW, int KW, int BKW, bool GEN>
__global__ __launch_bounds__(64 * QW * KW, DP <= 128 && QW == 4 ? 2 : 1)
void dense_short_kernel(const DenseArgs a, const MatrixPlan mp) {
  __shared__ u4 mx_lds[MxCfg<T, DP, QW, KW, BKW, GEN>::LDS / 16];
  char* const lds = reinterpret_cast<char*>(mx_lds);
  __shared__ float red_m[KW > 1 ? KW : 1][32 * QW], red_l[KW > 1 ? KW : 1][32 * QW];
  const bool again = mx_walk<T, DP, QW, KW, BKW, GEN, false>(a, mp, lds, red_m, red_l);
  if (__syncthreads_or(again)) mx_walk<T, DP, QW, KW, BKW, GEN, true>(a, mp, lds, red_m, red_l);
}

// whether any key tile of batch entry b is flagged (workgroup-uniform)
__device__ __forceinline__ bool mx_flagged(const MatrixPlan& mp, int64_t b) {
  int any = 0;
  const int32_t* f = mp.flags + b * mp.nt * mp.waves;
  for (int64_t i = threadIdx.x; i < (int64_t)mp.nt * mp.waves; i += blockDim.x) any |= f[i];
  return __syncthreads_or(any) != 0;
}

// Workgroup g: batch entry g % batch, every (grid / batch)-th of its rows, and
// only if one of its key tiles is flagged.
template <typename T>
__global__ __launch_bounds__(256) void dense_fixup_kernel(const DenseArgs a, const MatrixPlan mp) {
  const int64_t b = blockIdx.x % (unsigned)a.batch, first = blockIdx.x / (unsigned)a.batch;
  if (!mx_flagged(mp, b)) return;
  for (int64_t i = first; i < a.q_len; i += gridDim.x / (unsigned)a.batch) {
    dense_row<T, MX_MAX_DIM / 64, 2, 4, ANY_INDEX>(a, DenseSplit{1, a.kv_len, nullptr}, b * a.q_len + i, 0);
    __syncthreads();   // its LDS is free for the next row
  }
}

#endif
