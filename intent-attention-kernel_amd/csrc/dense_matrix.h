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
//           than 2^8, so the accumulators are rarely rescaled.
//   values  O^T[32 dims x 32 rows] += V^T . P^T: P is the score result as it
//           lies in the registers, V^T comes out of the [key][dim] tile
//           (16-bit: the transposing read ds_read_b64_tr_b16).
// Arithmetic. Every product is exact or float32 and every sum is float32.
// float16 / bfloat16 inputs: Q.K products are exact on the 16-bit matrix
// instructions; the float32 weights are split into 16-bit parts whose sum
// carries 22 bits or more (float16: two parts of p * 2^7, bfloat16: three),
// one matrix instruction per part. float32 inputs: v_mfma_f32_32x32x2_f32.
//
// Non-finite and large values. Four shortcuts would answer differently from the plain
// sum for them: a split weight times an infinite V (inf * 0 in the low part); the
// rows that fill up a range's last tile, which repeat its last key with weight 0
// (0 * inf); the lagging maximum, whose weights of up to 2^8 overflow on a finite V; and
// causal tiles past the diagonal, which are not visited (a NaN or an
// overflowing score there makes its row NaN, an infinite V a zero weight's
// product NaN). Each key tile is therefore checked once, by one of the
// workgroups that loads it, and its flag (K and V below 2^59 or not) goes to the
// workspace; the kernel that follows (the merge, or dense_fixup_kernel)
// recomputes every row of a flagged batch entry with dense_row.
#ifndef IAK_DENSE_MATRIX_H
#define IAK_DENSE_MATRIX_H

typedef float f16v __attribute__((ext_vector_type(16)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

constexpr int MX_MAX_DIM = 256;      // 16-bit inputs
constexpr int MX_MAX_DIM_F32 = 128;  // float32: Q, scores and context of wider rows spill
constexpr float LOG2E = 1.44269504088896340736f;
// float16 weights are kept as p * 2^MX_P_EXP (<= 2^15): the low part's
// subnormal step is then 2^-31 of the row's largest weight
constexpr float MX_P_EXP = 7.0f;
constexpr float LARGE = 1e5f;   // scores (exp2 domain) whose rounding reaches 2^-8

struct MatrixPlan {
  int splits;      // key ranges per (batch entry, query tile)
  int chunk;       // keys per range, whole tiles
  int nq;          // query tiles per batch entry
  int nt;          // key tiles per batch entry
  int skip;        // causal: tiles past the diagonal are not visited
  int64_t accoff;  // offset of the partial contexts in ws (floats)
  float* ws;       // splits > 1: the partials
  int waves;       // waves of a workgroup
  int32_t* flags;  // [batch][nt][waves]
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
  using C = MxCfg<T, DP, QW, KW, BKW, GEN>;
  using E = MxElem<T>;
  using vec = typename E::vec;
  constexpr bool F32 = sizeof(T) == 4;
  constexpr int BK = C::BK, RB = C::RB, CH = C::CH, NCH = C::NCH, NSB = C::NSB, NDV = C::NDV;
  constexpr int PARTS = E::PARTS;
  __shared__ u4 mx_lds[C::LDS / 16];
  char* const lds = reinterpret_cast<char*>(mx_lds);
  __shared__ float red_m[KW > 1 ? KW : 1][C::BQ], red_l[KW > 1 ? KW : 1][C::BQ];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qw = w % QW, kw = w / QW;
  const int l32 = lane & 31, h = lane >> 5;
  const float NEG_INF = -__builtin_inff();

  // work item: the query tiles over one range of keys (a group) on one XCD
  int b, split, qt;
  {
    const unsigned n = gridDim.x, xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3;
    const unsigned per = n >> 3, rem = n & 7u, nq = (unsigned)mp.nq, groups = n / nq;
    unsigned bs;
    if (mp.skip && (groups & 7u) == 0) {
      // causal: the XCD's groups side by side, the longest query tiles first (32 heads x
      // 4,096 rows x 128: 278 us; one group after the other 349); on a grid of
      // two four-wave workgroups per CU, resident at once, the second half from the
      // shortest, so each CU's two are about as long together
      const unsigned gpx = groups >> 3, half = (nq + 1) / 2 * gpx;
      qt = (int)(QW * KW == 4 && n <= 512 && slot >= half ? (slot - half) / gpx : nq - 1 - slot / gpx);
      bs = xcd * gpx + slot % gpx;
    } else {
      const unsigned item = xcd * per + (xcd < rem ? xcd : rem) + slot;
      bs = item / nq;
      qt = (int)(item - bs * nq);
      if (mp.skip) qt = (int)nq - 1 - qt;
    }
    split = (int)(bs % (unsigned)mp.splits);
    b = (int)(bs / (unsigned)mp.splits);
  }
  const int q0 = qt * C::BQ;
  const int lo = split * mp.chunk;
  const int hi = a.kv_len - lo < mp.chunk ? a.kv_len : lo + mp.chunk;
  const int row = q0 + 32 * qw + l32;                       // this lane's query row
  const int rowc = row < a.q_len ? row : a.q_len - 1;

  // Q of the lane's row: pieces 2s + h
  vec q[CH / 2];
  bool qlarge = false;
  {
    const T* qrow = reinterpret_cast<const T*>(a.q) + (int64_t)b * a.q_stride_b + (int64_t)rowc * a.q_stride_t;
#pragma unroll
    for (int s = 0; s < CH / 2; ++s) {
      const int c = 2 * s + h;
      u4 x = u4{0u, 0u, 0u, 0u};
      if (c * C::EPC < a.head_dim) x = *reinterpret_cast<const u4*>(qrow + c * C::EPC);
      if constexpr (!__is_same(T, _Float16)) qlarge |= mx_large<T>(x);
      q[s] = __builtin_bit_cast(vec, x);
    }
  }
  bool skip = mp.skip != 0;
  // a query at or above 2^59 could overflow against a skipped key: visit them all
  if constexpr (!__is_same(T, _Float16))
    if (skip) skip = __syncthreads_or(qlarge) == 0;
  const int klim = skip && q0 + C::BQ < hi ? q0 + C::BQ : hi;
  const int tiles = klim > lo ? (klim - lo + BK - 1) / BK : 0;

  const T* kbase = reinterpret_cast<const T*>(a.k) + (int64_t)b * a.k_stride_b;
  const T* vbase = reinterpret_cast<const T*>(a.v) + (int64_t)b * a.v_stride_b;
  u4 kr[NCH], vr[C::STAGED ? 1 : NCH];
  // piece i of the thread: row and position in the tile
  auto piece = [&](int i, int& r, int& c) {
    const int f = (C::PRIV ? lane : tid) + (C::PRIV ? 64 : C::THREADS) * i;
    r = f / CH;
    c = f - r * CH;
    if (C::PRIV) r += kw * BKW;
  };
  // K and V rows of the pieces of tile t (rows past the range repeat its last key),
  // looked up one tile ahead where the keys are an index
  int at[NCH];
  auto look_up = [&](int t) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      int r, c;
      piece(i, r, c);
      const int j0 = lo + t * BK + r, j = j0 < hi ? j0 : hi - 1;
      at[i] = a.kv_index ? (int)a.kv_index[j] : j;
    }
  };
  // the pieces of the tile looked up last (dims past the width are zero)
  auto load_pieces = [&](u4* x, const T* base, int64_t stride, int width) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      int r, c;
      piece(i, r, c);
      x[i] = u4{0u, 0u, 0u, 0u};
      if (c * C::EPC < width) x[i] = *reinterpret_cast<const u4*>(base + (int64_t)at[i] * stride + c * C::EPC);
    }
  };
  auto load_k = [&]() { load_pieces(kr, kbase, a.k_stride_t, a.head_dim); };
  auto load_v = [&]() { load_pieces(C::STAGED ? kr : vr, vbase, a.v_stride_t, a.v_dim); };
  auto large = [&](const u4* x) {
    bool bad = false;
#pragma unroll
    for (int i = 0; i < NCH; ++i) bad |= mx_large<T>(x[i]);
    return bad;
  };
  // the flag of tile t of this range, by the workgroup whose turn it is (checks)
  auto put_flag = [&](int t, bool bad) {
    const bool any = __builtin_amdgcn_ballot_w64(bad) != 0;
    if (lane == 0) mp.flags[((int64_t)b * mp.nt + lo / BK + t) * (QW * KW) + w] = any ? 1 : 0;
  };
  auto checks = [&](int t) {
    const int g = lo / BK + t;
    if (!mp.skip) return g % mp.nq == qt;
    const int64_t own = (int64_t)g * BK / C::BQ;      // the first query tile that visits it
    return own == qt;
  };
  auto store_k = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      int r, c;
      piece(i, r, c);
      *reinterpret_cast<u4*>(lds + buf * 2 * C::TILE + r * RB + 16 * k_piece<RB>(r, c)) = kr[i];
    }
  };
  auto store_v = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      int r, c;
      piece(i, r, c);
      *reinterpret_cast<u4*>(lds + buf * 2 * C::TILE + C::TILE + r * RB + 16 * v_piece<RB, C::ES>(r, c)) =
          C::STAGED ? kr[i] : vr[C::STAGED ? 0 : i];
    }
  };
  // LDS writes before, reads behind (and the other way round)
  auto sync = [&]() {
    if constexpr (C::PRIV) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    else __syncthreads();
  };

  f16v acc[NDV];
#pragma unroll
  for (int d = 0; d < NDV; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[d][r] = 0.f;
  // running max (GEN: of the scores, else of the scores times sm_scale log2 e,
  // less PEXP) and this lane's part of the denominator
  float m = NEG_INF, l = 0.f;
  const float cmul = a.sm_scale * LOG2E;
  constexpr float PEXP = F32 ? 0.f : MX_P_EXP;

  f16v s[NSB];
  // the wave's first key of tile t, and whether its rows see any of its keys (wave-uniform)
  auto first_key = [&](int t) { return lo + t * BK + kw * BKW; };
  auto seen = [&](int t) { return first_key(t) < hi && !(skip && first_key(t) > q0 + 32 * qw + 31); };

  auto scores = [&](int t, int buf) {
    const char* kt = lds + buf * 2 * C::TILE + kw * BKW * RB;
    // the lane's byte offsets, opaque to the compiler: the offsets of the single
    // pieces follow by one xor or add each, where hoisting them all out of the
    // loop spilled up to 150 registers
    int krow = l32 * RB, koff = 16 * k_piece<RB>(l32, h);
    asm volatile("" : "+v"(krow), "+v"(koff));
    if constexpr (F32) {
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb) s[sb] = mx_score_tree<0, CH / 2>(kt + 32 * sb * RB + krow, koff, q);
    } else {
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[sb][r] = 0.f;
#pragma unroll
      for (int c = 0; c < CH / 2; ++c)
#pragma unroll
        for (int sb = 0; sb < NSB; ++sb) {
          // BKW and 32 are multiples of 16, so the swizzle of row 32 sb + l32 is that of l32
          const vec kf = *reinterpret_cast<const vec*>(kt + 32 * sb * RB + krow + (koff ^ (32 * c)));
          s[sb] = E::mfma(kf, q[c], s[sb]);
        }
    }
  };

  auto values = [&](int t, int buf) {
    const int key0 = first_key(t);
    const char* vt = lds + buf * 2 * C::TILE + C::TILE + kw * BKW * RB;
    int vrow = 4 * h * RB, voff = 4 * l32;   // opaque, as in scores
    if constexpr (!F32) {
      const int r = (lane & 15) >> 2;
      vrow += r * RB;
      voff = 16 * v_piece<RB, 2>(r, 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) + 8 * (lane & 1);
    }
    asm volatile("" : "+v"(vrow), "+v"(voff));
    // masks: key of s[sb][r] is key0 + 32 sb + 8 (r / 4) + 4 h + r % 4
    if constexpr (GEN) {
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int j = key0 + 32 * sb + 8 * (r >> 2) + 4 * h + (r & 3);
          const int jc = j < hi ? j : hi - 1;
          float x = s[sb][r] * a.sm_scale;
          if (a.causal == IAK_CAUSAL_TRIU && j > row) x += NEG_INF;
          if (a.causal == IAK_CAUSAL_POSITIONS && (int64_t)row < a.kv_positions[jc]) x = NEG_INF;
          if (a.mask) {
            const int64_t mi = (int64_t)b * a.mask_stride_b + (int64_t)rowc * a.mask_stride_q + (int64_t)jc * a.mask_stride_k;
            if (a.mask_dtype == IAK_MASK_BOOL) x += load_t<uint8_t>(a.mask, mi);
            else if (a.mask_dtype == IAK_DTYPE_F32) x += load_t<float>(a.mask, mi);
            else if (a.mask_dtype == IAK_DTYPE_F16) x += load_t<_Float16>(a.mask, mi);
            else x += load_t<bf16_bits>(a.mask, mi);
          }
          s[sb][r] = j < hi ? rounded(x) : NEG_INF;
        }
    } else {
      if (a.causal == IAK_CAUSAL_TRIU && key0 + BKW - 1 > q0 + 32 * qw) {
#pragma unroll
        for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (key0 + 32 * sb + 8 * (r >> 2) + 4 * h + (r & 3) > row) s[sb][r] += NEG_INF;
      }
      if (key0 + BKW > hi) {
#pragma unroll
        for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (key0 + 32 * sb + 8 * (r >> 2) + 4 * h + (r & 3) >= hi) s[sb][r] = NEG_INF;
      }
    }
    float mx = s[0][0];
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[sb][r]);
    mx = xmax32(mx);
    float cur = mx;
    if constexpr (!GEN) {
      const float x = mx * cmul;
      cur = fabsf(x) > LARGE ? x : x - PEXP;
    }
    const bool grow = cur > m + (GEN ? RESCALE_SLACK / LOG2E : RESCALE_SLACK);
    if (__builtin_amdgcn_ballot_w64(grow)) {
      const float alpha = grow ? __builtin_amdgcn_exp2f(GEN ? (m - cur) * LOG2E : m - cur) : 1.f;   // 0 at first (m = -inf)
      l *= alpha;
#pragma unroll
      for (int d = 0; d < NDV; ++d) acc[d] *= alpha;
      if (grow) m = cur;
    }
    // weights p * 2^PEXP; a row that has seen nothing but -inf keeps them 0
    const float ref = m == NEG_INF ? 0.f : m;
    // one fma per score, except where the product's own rounding is no longer
    // small beside 1: there the largest score has to give exactly 2^0
    const bool large = !GEN && __builtin_amdgcn_ballot_w64(fabsf(ref) > LARGE) != 0;
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if constexpr (GEN) s[sb][r] = __builtin_fmaf(s[sb][r] - ref, LOG2E, PEXP);
        else if (large) s[sb][r] = rounded(s[sb][r] * cmul) - ref;
        else s[sb][r] = __builtin_fmaf(s[sb][r], cmul, -ref);
        s[sb][r] = __builtin_amdgcn_exp2f(s[sb][r]);
      }
    float ls = 0.f;
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int r = 0; r < 16; r += 4) ls += (s[sb][r] + s[sb][r + 1]) + (s[sb][r + 2] + s[sb][r + 3]);
    l += ls;

    if constexpr (F32) {
      // a tile's products are summed in four chains of 8 keys and then added to
      // the context: short chains, as above
#pragma unroll
      for (int d = 0; d < NDV; ++d) {
#pragma unroll
        for (int sb = 0; sb < NSB; ++sb) {
          f16v o[4];
#pragma unroll
          for (int r = 0; r < 16; ++r) o[0][r] = o[1][r] = o[2][r] = o[3][r] = 0.f;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            // rows 8 (r / 4) + 4 h + r % 4 (+ 32 sb): bit 2 of the row is h, so the
            // 128-byte groups d and d ^ 1 change places for h = 1
            const int r = (i >> 2) + 4 * (i & 3);
            const float vf = *reinterpret_cast<const float*>(vt + (32 * sb + 8 * (r >> 2) + (r & 3)) * RB + 128 * d +
                                                             vrow + (voff + (d & 1 ? -128 * h : 128 * h)));
            o[i & 3] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf, s[sb][r], o[i & 3], 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
          acc[d] += (o[0] + o[1]) + (o[2] + o[3]);
        }
      }
    } else {
      typedef short s4v __attribute__((ext_vector_type(4)));
      typedef __attribute__((address_space(3))) s4v lds_s4;
#pragma unroll
      for (int kk = 0; kk < BKW / 16; ++kk) {
        // the 16 keys of this step: elements 0..7 of the B operand are
        // s[kk / 2][8 (kk % 2) + 0..7]
        uint32_t pw[PARTS][4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float x0 = s[kk >> 1][8 * (kk & 1) + 2 * e], x1 = s[kk >> 1][8 * (kk & 1) + 2 * e + 1];
#pragma unroll
          for (int pz = 0; pz < PARTS; ++pz) pw[pz][e] = mx_take_part<T>(x0, x1, pz + 1 < PARTS);
        }
#pragma unroll
        for (int d = 0; d < NDV; ++d) {
          // V^T: dims 32 d + lane % 32 of keys 16 kk + 4 h + 0..3 and + 8
          const int off = 16 * kk * RB + vrow + (voff ^ (64 * d));
          const s4v lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(vt + off));
          const s4v hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(vt + off + 8 * RB));
          const vec vf = __builtin_bit_cast(vec, __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
          for (int pz = 0; pz < PARTS; ++pz)
            acc[d] = E::mfma(vf, __builtin_bit_cast(vec, (u4{pw[pz][0], pw[pz][1], pw[pz][2], pw[pz][3]})), acc[d]);
        }
      }
    }
  };

  if constexpr (C::STAGED) {
    bool bad = false;
    if (tiles > 0) {
      look_up(0);
      load_k();
      bad = checks(0) && large(kr);
      store_k(0);
      load_v();
      if (tiles > 1) look_up(1);
      if (checks(0)) put_flag(0, bad || large(kr));
      store_v(0);
    }
    for (int t = 0; t < tiles; ++t) {
      const bool more = t + 1 < tiles;
      sync();   // tile t is in place
      if (more) load_k();
      if (seen(t)) scores(t, 0);
      sync();   // its keys are read
      if (more) {
        bad = checks(t + 1) && large(kr);
        store_k(0);
        load_v();
        if (t + 2 < tiles) look_up(t + 2);
      }
      if (seen(t)) values(t, 0);
      sync();   // its values are read
      if (more) {
        if (checks(t + 1)) put_flag(t + 1, bad || large(kr));
        store_v(0);
      }
    }
  } else {
    if (tiles > 0) {
      look_up(0);
      load_k();
      load_v();
      if (tiles > 1) look_up(1);
      if (checks(0)) put_flag(0, large(kr) || large(vr));
      store_k(0);
      store_v(0);
    }
    for (int t = 0; t < tiles; ++t) {
      const bool more = t + 1 < tiles;
      const int buf = C::NB == 2 ? t & 1 : 0, next = C::NB == 2 ? buf ^ 1 : 0;
      sync();   // tile t is in place; with two buffers, the other one is free
      if (more) {
        load_k();
        load_v();
        if (t + 2 < tiles) look_up(t + 2);
      }
      if (seen(t)) {
        scores(t, buf);
        values(t, buf);
      }
      if (C::NB == 1) sync();   // every reader of tile t is done
      if (more) {
        if (checks(t + 1)) put_flag(t + 1, large(kr) || large(vr));
        store_k(next);
        store_v(next);
      }
    }
  }
  // key tiles that no query tile visits (keys past the last row's diagonal): checked here
  if (mp.skip) {
    const int all = hi > lo ? (hi - lo + BK - 1) / BK : 0;
    for (int t = 0; t < all; ++t) {
      const int64_t g = lo / BK + t;
      if (g * BK / C::BQ >= mp.nq && g % mp.nq == qt) {
        look_up(t);
        load_k();
        bool bad = large(kr);
        load_v();
        if constexpr (C::STAGED) bad |= large(kr);
        else bad |= large(vr);
        put_flag(t, bad);
      }
    }
  }

  l = xsum32(l);
  const bool ok4 = row < a.q_len;
  const int64_t item = ((int64_t)b * a.q_len + row) * mp.splits + split;
  const int64_t items = (int64_t)a.batch * a.q_len * mp.splits;
  // four consecutive dims d0 .. d0 + 3 of query row `r` (item `it`): the output, or the range's partial
  auto put4 = [&](int r, int64_t it, int d0, f4 v, float mm, float inv) {
    if (d0 >= a.v_dim) return;
    if (mp.splits > 1) {
      *reinterpret_cast<f4*>(mp.ws + mp.accoff + it * a.v_dim + d0) = v;
      return;
    }
    T* o = reinterpret_cast<T*>(a.out) + (int64_t)b * a.out_stride_b + (int64_t)r * a.out_stride_t + d0;
    const float nan = __builtin_nanf("");
    // every score -inf: NaN, as softmax gives
    if constexpr (F32) {
      f4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = mm == NEG_INF ? nan : v[e] / inv;
      *reinterpret_cast<f4*>(o) = y;
    } else {
      uint16_t y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) store_t<T>(y, e, mm == NEG_INF ? nan : v[e] * inv);
      *reinterpret_cast<u2*>(o) = u2{(uint32_t)y[0] | ((uint32_t)y[1] << 16), (uint32_t)y[2] | ((uint32_t)y[3] << 16)};
    }
  };
  if constexpr (KW == 1) {
    if (!ok4) return;
    if (mp.splits > 1 && h == 0) {
      mp.ws[item] = m;
      mp.ws[items + item] = l;
    }
    const float inv = F32 ? l : 1.0f / l;
#pragma unroll
    for (int d = 0; d < NDV; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        put4(row, item, 32 * d + 8 * g + 4 * h, f4{acc[d][4 * g], acc[d][4 * g + 1], acc[d][4 * g + 2], acc[d][4 * g + 3]},
             m, inv);
  } else {
    // the KW key groups of a query row meet in the tile buffers, [kw][qw][dim][row]
    __syncthreads();
    float* red = reinterpret_cast<float*>(lds);
    if (h == 0) {
      red_m[kw][32 * qw + l32] = m;
      red_l[kw][32 * qw + l32] = l;
    }
    float* mine = red + (kw * QW + qw) * 32 * DP;
#pragma unroll
    for (int d = 0; d < NDV; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) mine[(32 * d + 8 * (r >> 2) + 4 * h + (r & 3)) * 32 + l32] = acc[d][r];
    __syncthreads();
    // thread: row tid % BQ, every (THREADS / BQ)-th group of four dims
    const int rq = tid % C::BQ, g0 = tid / C::BQ;
    const int r = q0 + rq;
    if (r >= a.q_len) return;
    float M = NEG_INF;
#pragma unroll
    for (int k = 0; k < KW; ++k) M = fmaxf(M, red_m[k][rq]);
    float wt[KW], L = 0.f;
#pragma unroll
    for (int k = 0; k < KW; ++k) {
      const float mk = red_m[k][rq];
      wt[k] = mk == NEG_INF ? 0.f : __builtin_amdgcn_exp2f(GEN ? (mk - M) * LOG2E : mk - M);
      L += wt[k] * red_l[k][rq];
    }
    const int64_t it = ((int64_t)b * a.q_len + r) * mp.splits + split;
    if (mp.splits > 1 && g0 == 0) {
      mp.ws[it] = M;
      mp.ws[items + it] = L;
    }
    const float inv = F32 ? L : 1.0f / L;
    for (int g = g0; g < DP / 4; g += C::THREADS / C::BQ) {
      f4 v = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < KW; ++k) {
        const float* src = red + (k * QW + rq / 32) * 32 * DP + (4 * g) * 32 + (rq & 31);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(wt[k], src[32 * e], v[e]);
      }
      put4(r, it, 4 * g, v, M, inv);
    }
  }
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
    dense_row_any<T, MX_MAX_DIM / 64, 2, 4>(a, b * a.q_len + i);
    __syncthreads();   // its LDS is free for the next row
  }
}

#endif
