// The float32 latent context on the matrix cores: the form of mla_rows.hip for
// several query rows. Included by that file only.
//
// A workgroup takes 32 query rows and a range of keys, 32 at a time, with up to
// eight waves of DW = 32 ND latent dims each (six of 96 at 576): wave w owns dims
// w DW .. + DW - 1 of every row, both as key and as value, so it loads, converts to
// float32 and keeps in the LDS only its own part of the 32 latent rows. Per tile:
//   scores  each wave sums q . c over its dims, S^T[32 keys x 32 rows] on
//           v_mfma_f32_32x32x2_f32 in chains of 8 dims added pairwise; the
//           partial scores meet in the LDS and every wave adds them in the same
//           order;
//   softmax per lane (query row = lane % 32, 16 keys), in every wave alike;
//   values  O^T[32 dims x 32 rows] += C^T . P^T for the wave's dims: P is the
//           score result as it lies in the registers.
// Every product and sum is float32; each key's row is read once for 32 query rows.
// Bound: 576 matrix instructions of 64 cycles per tile at 576 dims (3.8 us for one
// tile per CU), behind a chain of launch, page ids, latents and the partials' merge.
// The rows form reads each latent row for four query rows and sums every score
// across the 64 lanes; 32 rows x 8,192 keys x 576 (float16 latents) took it 44 us,
// this form see mla_rows.hip.
#ifndef IAK_MLA_ROWS_MATRIX_H
#define IAK_MLA_ROWS_MATRIX_H

typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int RX_ROWS = 32, RX_KEYS = 32, RX_WAVES = 8, RX_MAX_ND = 3;
// 32-dim tiles per wave: the fewest that up to eight waves cover the latents with.
// (Four waves of 160 dims: 512 keys x 576 20 us, mostly the latency of one wave's
// chain; nine of 64: one SIMD with three waves has too few registers.)
inline int rx_dim_tiles(int dc) { return (dc + 32 * RX_WAVES - 1) / (32 * RX_WAVES); }
constexpr float RX_LOG2E = 1.44269504088896340736f;

__device__ __forceinline__ float rx_max32(float v) {   // over lanes l and l ^ 32 (see xmax16_32)
  float t;
  asm volatile("v_mov_b32 %1, %0\n\ts_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_max_f32 %0, %0, %1"
               : "+v"(v), "=&v"(t));
  return v;
}
__device__ __forceinline__ float rx_sum32(float v) {
  float t;
  asm volatile("v_mov_b32 %1, %0\n\ts_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_add_f32 %0, %0, %1"
               : "+v"(v), "=&v"(t));
  return v;
}

// LDS position of 16-byte piece c of key row r (rows of RB bytes): the lanes that
// read one piece of 16 rows touch every bank group once
template <int RB> __device__ __forceinline__ int rx_piece(int r, int c) {
  constexpr int P = RB % 256 == 0 ? 1 : 2;   // rows until the bank offset repeats
  static_assert(RB % 128 == 0, "whole 32-dim tiles");
  return c ^ ((r / P) & (16 / P - 1));
}

// scores of 32 keys x 32 rows over the pieces 2c + h, c = C0 .. C0 + N - 1 (N
// even): chains of 8 dims added pairwise, two chains in step so that one's
// matrix instructions fill the other's latency
template <int C0, int N, int NQ>
__device__ __forceinline__ f16v rx_score_tree(const char* kt, int koff, const f4 (&q)[NQ]) {
  static_assert(N % 2 == 0, "pairs of chains");
  if constexpr (N == 2) {
    f16v s[2];
    f4 kf[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[i][r] = 0.f;
      kf[i] = *reinterpret_cast<const f4*>(kt + (koff ^ (32 * (C0 + i))));
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < 2; ++i) s[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[i][e], q[C0 + i][e], s[i], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0x100);   // one pair after the other (interleaved, they spill); LDS reads may move up
    return s[0] + s[1];
  } else {
    constexpr int H = N / 4 * 2;
    const f16v x = rx_score_tree<C0, H, NQ>(kt, koff, q);
    return x + rx_score_tree<C0 + H, N - H, NQ>(kt, koff, q);
  }
}

template <typename T, int ND, int WAVES>   // WAVES: at most that many per workgroup
__global__ __launch_bounds__(64 * WAVES, 1) void mla_rows_matrix_kernel(const iak_mla_rows_args a, const RowSplit sp) {
  constexpr int DW = 32 * ND, RB = 4 * DW;
  constexpr int EPC = 16 / (int)sizeof(T);          // latents per 16-byte piece
  constexpr int PPK = DW / EPC;                     // pieces of a key in the wave's part
  constexpr int NCH = RX_KEYS * PPK / 64;           // pieces per lane and tile
  static_assert(RX_KEYS * PPK % 64 == 0, "whole pieces per lane");
  __shared__ __attribute__((aligned(16))) char tile_lds[WAVES][RX_KEYS * RB];   // read in 16-byte pieces
  __shared__ float part_s[WAVES][16][64];
  const int nw = blockDim.x >> 6;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  const float NEG_INF = -__builtin_inff();
  const int64_t nrows = (int64_t)a.batch * a.q_len;
  const int dc = a.latent_dim;
  const int64_t group = blockIdx.x / (unsigned)sp.splits;
  const int split = (int)(blockIdx.x - group * sp.splits);
  const int lo = split * sp.chunk;
  const int hi = sp.nkeys - lo < sp.chunk ? sp.nkeys : lo + sp.chunk;
  const int tiles = (hi - lo + RX_KEYS - 1) / RX_KEYS;
  const int d0 = w * DW;                            // the wave's first dim
  char* const tile = tile_lds[w];

  const T* lat = reinterpret_cast<const T*>(a.latents);
  u4 cr[NCH];
  uint32_t live = 0;   // bit k: key k of the loaded tile is a row of the latents
  // Lane l looks up key l % 32 of a tile, one tile ahead of its loads: its row
  // (clamped into the latents) and whether it is one.
  int64_t src = 0;
  auto look_up = [&](int t) {
    const int j = lo + t * RX_KEYS + l32;
    src = key_row(a, sp, (uint32_t)(j < hi ? j : hi - 1));
    if (j >= hi) src = -1;
  };
  // The pieces of tile t (looked up before), all loads unconditional at clamped
  // addresses: behind a branch each they waited for one another.
  auto load_tile = [&](int t) {
    live = (uint32_t)__builtin_amdgcn_ballot_w64(src >= 0 && src < a.num_rows);
    const int64_t off = (src < 0 ? 0 : (src < a.num_rows ? src : a.num_rows - 1)) * a.latent_stride;
    if (t + 1 < tiles) look_up(t + 1);
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int f = lane + 64 * i, r = f / PPK, c = f - r * PPK;
      const int d = d0 + c * EPC;
      cr[i] = *reinterpret_cast<const u4*>(lat + __shfl(off, r, 64) + (d < dc ? d : 0));
    }
  };
  // a key that is no row of the latents holds zeros: it takes no mass, and its
  // value adds none
  auto store_tile = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int f = lane + 64 * i, r = f / PPK, c = f - r * PPK;
      const u4 x = ((live >> r) & 1u) && d0 + c * EPC < dc ? cr[i] : u4{0u, 0u, 0u, 0u};   // dims past the width too
      if constexpr (sizeof(T) == 4) {
        *reinterpret_cast<u4*>(tile + r * RB + 16 * rx_piece<RB>(r, c)) = x;
      } else {
        f4 y[2];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint16_t v = (uint16_t)(x[e >> 1] >> (16 * (e & 1)));
          y[e >> 2][e & 3] = to_f32(__builtin_bit_cast(T, v));
        }
        *reinterpret_cast<f4*>(tile + r * RB + 16 * rx_piece<RB>(r, 2 * c)) = y[0];
        *reinterpret_cast<f4*>(tile + r * RB + 16 * rx_piece<RB>(r, 2 * c + 1)) = y[1];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };

  f16v acc[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[d][r] = 0.f;
  float m = NEG_INF, l = 0.f;   // running max of the scores times sm_scale log2 e
  const float cmul = a.sm_scale * RX_LOG2E;

  look_up(0);
  load_tile(0);
  // Q of the lane's row, pieces 2c + h of the wave's dims, by way of the wave's tile
  // buffer: four dims a lane, the loads of a batch in flight together (straight
  // into the operand registers each waited for the last)
  f4 q[DW / 8];
  {
    // whole: rows whose groups of four dims are aligned vectors
    auto load_all = [&](auto type, auto whole) {
      using Q = decltype(type);
      typedef uint32_t qv __attribute__((ext_vector_type(sizeof(Q))));   // four elements
      const Q* qp = reinterpret_cast<const Q*>(a.q);
      constexpr int QN = RX_ROWS * DW / 4 / 64, QB = QN;
      static_assert(QN % QB == 0, "whole batches");
      for (int i0 = 0; i0 < QN; i0 += QB) {
        float y[QB][4];
#pragma unroll
        for (int i = 0; i < QB; ++i) {
          const int f = lane + 64 * (i0 + i), r = f / (DW / 4), c = f - r * (DW / 4), d = d0 + 4 * c;
          const int64_t row = group * RX_ROWS + r, rowc = row < nrows ? row : nrows - 1;
          const int64_t b = rowc / a.q_len;
          const Q* src = qp + b * a.q_stride_b + (rowc - b * a.q_len) * a.q_stride_t;
          if constexpr (decltype(whole)::value) {
            const qv x = *reinterpret_cast<const qv*>(src + (d < dc ? d : 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if constexpr (sizeof(Q) == 4) y[i][e] = u2f(x[e]);
              else y[i][e] = to_f32(__builtin_bit_cast(Q, (uint16_t)(x[e >> 1] >> (16 * (e & 1)))));
            }
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) y[i][e] = to_f32(src[d + e < dc ? d + e : dc - 1]);
          }
        }
#pragma unroll
        for (int i = 0; i < QB; ++i) {
          const int f = lane + 64 * (i0 + i), r = f / (DW / 4), c = f - r * (DW / 4), d = d0 + 4 * c;
          *reinterpret_cast<f4*>(tile + r * RB + 16 * rx_piece<RB>(r, c)) =
              f4{d < dc ? y[i][0] : 0.f, d + 1 < dc ? y[i][1] : 0.f, d + 2 < dc ? y[i][2] : 0.f, d + 3 < dc ? y[i][3] : 0.f};
        }
      }
    };
    const int es = a.q_dtype == IAK_DTYPE_F32 ? 4 : 2;
    const bool whole = dc % 4 == 0 && ((a.q_stride_b | a.q_stride_t) & 3) == 0 &&
                       (reinterpret_cast<uintptr_t>(a.q) & (4 * es - 1)) == 0;
    if (a.q_dtype == IAK_DTYPE_F32) whole ? load_all(float{}, std::true_type{}) : load_all(float{}, std::false_type{});
    else if (a.q_dtype == IAK_DTYPE_F16) whole ? load_all(_Float16{}, std::true_type{}) : load_all(_Float16{}, std::false_type{});
    else whole ? load_all(bf16_bits{}, std::true_type{}) : load_all(bf16_bits{}, std::false_type{});
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int c = 0; c < DW / 8; ++c)
      q[c] = *reinterpret_cast<const f4*>(tile + l32 * RB + 16 * rx_piece<RB>(l32, 2 * c + h));
  }

  for (int t = 0; t < tiles; ++t) {
    store_tile();
    const uint32_t seen = live >> (4 * h);   // key of s[r]: 8 (r / 4) + 4 h + r % 4
    int krow = l32 * RB, koff = 16 * rx_piece<RB>(l32, h);
    asm volatile("" : "+v"(krow), "+v"(koff));   // single offsets by one xor, not hoisted
    f16v s = rx_score_tree<0, DW / 8>(tile + krow, koff, q);
#pragma unroll
    for (int r = 0; r < 16; ++r) part_s[w][r][lane] = s[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = part_s[0][r][lane] + (nw > 1 ? part_s[1][r][lane] : 0.f);
    for (int k = 2; k < nw; k += 2)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[r] += part_s[k][r][lane] + (k + 1 < nw ? part_s[k + 1][r][lane] : 0.f);
    if (t + 1 < tiles) {
      __syncthreads();   // read before the next tile's are written
      load_tile(t + 1);  // in flight behind the values (behind the scores too, it spilled)
    }
    float mx = NEG_INF;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = (seen >> (8 * (r >> 2) + (r & 3))) & 1u ? s[r] * cmul : NEG_INF;
      mx = fmaxf(mx, s[r]);
    }
    mx = rx_max32(mx);
    // the maximum does not lag: a weight above 1 would take a large latent that the scores
    // do not see (its query dim 0) over the range
    const bool grow = mx > m;
    if (__builtin_amdgcn_ballot_w64(grow)) {
      const float alpha = grow ? __builtin_amdgcn_exp2f(m - mx) : 1.f;   // 0 at first (m = -inf)
      l *= alpha;
#pragma unroll
      for (int d = 0; d < ND; ++d) acc[d] *= alpha;
      if (grow) m = mx;
    }
    const float ref = m == NEG_INF ? 0.f : m;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float x = s[r];
      asm volatile("" : "+v"(x));   // the rounded product, as the max has it
      s[r] = __builtin_amdgcn_exp2f(x - ref);
    }
    l += ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7])) +
         (((s[8] + s[9]) + (s[10] + s[11])) + ((s[12] + s[13]) + (s[14] + s[15])));

    // the lane's four offsets within a 128-byte group (rx_piece of rows 8 x + 4 h + y)
    int voff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int x = RB % 256 == 0 ? 4 * h + i : 4 * (i >> 1) + 2 * h + (i & 1);
      voff[i] = 16 * ((l32 >> 2) ^ x) + 4 * (l32 & 3) + 4 * h * RB;
    }
    asm volatile("" : "+v"(voff[0]), "+v"(voff[1]), "+v"(voff[2]), "+v"(voff[3]));
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      f16v o[2];
#pragma unroll
      for (int r = 0; r < 16; ++r) o[0][r] = o[1][r] = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int r = (i >> 1) + 8 * (i & 1), x = r >> 2, y = r & 3;
        const int grp = RB % 256 == 0 ? d ^ (x & 1) : d;
        const int at = RB % 256 == 0 ? voff[y] : voff[2 * (x & 1) + (y >> 1)];
        const float vf = *reinterpret_cast<const float*>(tile + (8 * x + y) * RB + 128 * grp + at);
        o[i & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf, s[r], o[i & 1], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0x100);
      acc[d] += o[0] + o[1];
    }
  }

  l = rx_sum32(l);
  const int64_t row = group * RX_ROWS + l32;
  const int64_t n = nrows * sp.splits, slot = row * sp.splits + split;
  if (sp.splits > 1 && w == 0 && h == 0 && row < nrows) {
    sp.ws[slot] = m;
    sp.ws[n + slot] = l;
  }
  // through the tile buffer once more, so that each row's part leaves in whole
  // lines (16-byte pieces of 32 rows at a time took 9 of 25 us, 256 ranges x 576 dims)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f4 v = f4{acc[d][4 * g], acc[d][4 * g + 1], acc[d][4 * g + 2], acc[d][4 * g + 3]};
      if (sp.splits == 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = l > 0.f ? v[e] / l : 0.f;   // zeros when no row was visited
      *reinterpret_cast<f4*>(tile + l32 * RB + 16 * rx_piece<RB>(l32, 8 * d + 2 * g + h)) = v;
    }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  float* dst = sp.splits > 1 ? sp.ws + sp.accoff + split * dc : a.context;
#pragma unroll
  for (int i = 0; i < RX_ROWS * DW / 4 / 64; ++i) {
    const int f = lane + 64 * i, r = f / (DW / 4), c = f - r * (DW / 4), dim = d0 + 4 * c;
    const f4 v = *reinterpret_cast<const f4*>(tile + r * RB + 16 * rx_piece<RB>(r, c));
    if (dim < dc && group * RX_ROWS + r < nrows)
      *reinterpret_cast<f4*>(dst + (group * RX_ROWS + r) * sp.splits * dc + dim) = v;
  }
}

#endif
