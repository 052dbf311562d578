// MLA latent decode for few heads (a model's heads shared over several GPUs, say):
// the form of mla_decode.hip whose waves share out pages instead of heads.
// Included by that file only.
//
// One workgroup of four waves, one per SIMD, reduces one split for 16 heads; wave
// w takes every fourth page of it end to end, with its own running softmax and
// its own context for all value dims (128 registers at 512), so the waves meet
// only once, at the end, in the LDS. (The 128-head form gives 16 heads to each of
// eight waves that all walk the same pages: with 16 heads seven of them work on
// padding.) With 16 heads a latent byte takes 60 (FP8) or 30 (float16) operations:
// the bound is HBM, and below some 100 MB the chain of launch, table, tags, first
// page and merge (8 x 300 pages of float16, 16 heads: 24.6 -> 20 us, 44 MB; 32 x 512
// pages, 302 MB: 99 -> 78 with the merge).
//   Pages  go from HBM straight into the wave's two LDS slots (global_load_lds),
//          the next one behind the page at hand. A float16 page is its own operand
//          tile: lane addresses permute the 16-byte pieces of a row on the way in, so
//          that the score reads (one piece of 16 rows) and the transposing value
//          reads (32 bytes of 16 rows) spread over the banks as padding would. An FP8 /
//          INT8 page lands in the upper half of its slot and is converted over the
//          whole slot by the wave, through registers.
//   Math   as in mla_decode.hip: scores S^T[16 tok x 16 heads] on 16x16x32, online
//          softmax with the value exponent, values O[16 heads x 16 dims] += P . C on
//          16x16x16 (P is the score result as it lies).
#ifndef IAK_MLA_FEW_H
#define IAK_MLA_FEW_H

constexpr int FEW_WAVES = 4, FEW_HEADS = 16;

template <int DQK, int DV> struct Few {
  static constexpr int RB = 2 * DQK;             // tile row bytes
  static constexpr int CH = RB / 16;             // 16-byte pieces per row
  static constexpr int PAGE8 = PS * DQK, SLOT = 2 * PAGE8;
  static constexpr int N16 = SLOT / 1024, N8 = PAGE8 / 1024;   // 1 KB copies per page
  static constexpr int KSTEPS = DQK / 32, NDB = DV / 16;
  static constexpr int ROWS_PER_BANKS = RB % 256 == 0 ? 1 : 2;
  // piece c of token row r lies at piece c ^ swz(r)
  static __device__ __forceinline__ int swz(int r) { return (r / ROWS_PER_BANKS) & (16 / ROWS_PER_BANKS - 1); }
  static_assert(RB % 128 == 0 && PAGE8 % 1024 == 0 && DV <= DQK, "unsupported MLA shape");
};

// one 1 KB copy, lane i's 16 bytes from `src` to dst + 16 i (see mla_dma_page)
__device__ __forceinline__ void few_copy(const uint8_t* src, uint8_t* dst) {
  typedef __attribute__((address_space(3))) uint8_t lds_u8;
  const uint32_t at = (uint32_t)(uintptr_t)(lds_u8*)dst;
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "{m0}"(at) : "memory");
}

template <int DQK, int DV>
__device__ __forceinline__ void few_dma(uint8_t* slot, const MArgs& a, int pid, int tag, int lane) {
  using C = Few<DQK, DV>;
  if (tag == IAK_TAG_FP16) {
    const uint8_t* base = reinterpret_cast<const uint8_t*>(a.c16) + (int64_t)pid * C::SLOT;
#pragma unroll
    for (int i = 0; i < C::N16; ++i) {
      const int p = 64 * i + lane, r = p / C::CH, c = p - r * C::CH;
      few_copy(base + r * C::RB + 16 * (c ^ C::swz(r)), slot + 1024 * i);
    }
  } else {
    const uint8_t* base =
        reinterpret_cast<const uint8_t*>(tag == IAK_TAG_FP8 ? a.c8f : a.c8i) + (int64_t)pid * C::PAGE8;
#pragma unroll
    for (int i = 0; i < C::N8; ++i) few_copy(base + 1024 * i + 16 * lane, slot + C::PAGE8 + 1024 * i);
  }
}

// a one-byte page from the upper half of its slot to the float16 tile over all of it
template <int DQK, int DV> __device__ __forceinline__ void few_convert(uint8_t* slot, int tag, int lane) {
  using C = Few<DQK, DV>;
  u4 x[C::N8];
#pragma unroll
  for (int i = 0; i < C::N8; ++i) x[i] = *reinterpret_cast<const u4*>(slot + C::PAGE8 + 1024 * i + 16 * lane);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // all read before any is overwritten
#pragma unroll
  for (int i = 0; i < C::N8; ++i) {
    const int p = 1024 * i + 16 * lane, r = p / DQK, c = (p - r * DQK) / 8;   // 16 codes: pieces c and c + 1
    uint32_t o[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (tag == IAK_TAG_FP8) fp8x4_to_f16(x[i][k], o[2 * k], o[2 * k + 1]);
      else i8x4_to_f16(x[i][k], o[2 * k], o[2 * k + 1]);
    }
    uint8_t* row = slot + r * C::RB;
    *reinterpret_cast<u4*>(row + 16 * (c ^ C::swz(r))) = u4{o[0], o[1], o[2], o[3]};
    *reinterpret_cast<u4*>(row + 16 * ((c + 1) ^ C::swz(r))) = u4{o[4], o[5], o[6], o[7]};
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

template <int DQK, int DV>
__global__ __launch_bounds__(64 * FEW_WAVES, 1) void mla_few_heads_kernel(const MArgs a) {
  using C = Few<DQK, DV>;
  __shared__ __attribute__((aligned(16))) uint8_t ring[FEW_WAVES][2][C::SLOT];
  __shared__ float red_m[FEW_WAVES][FEW_HEADS], red_l[FEW_WAVES][FEW_HEADS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int b = blockIdx.x / a.splits, split = blockIdx.x - b * a.splits;
  const int start = split * a.chunk;
  const int h0 = blockIdx.y * FEW_HEADS, head = h0 + c;

  const int limit = a.valid ? __builtin_amdgcn_readfirstlane(a.valid[b]) : 0x7FFFFFFF;
  const MlaPages meta = mla_page_meta(a, b, start, lane, limit);
  const MlaPages meta2 = mla_page_meta(a, b, start, lane + 64, limit);
  uint64_t rem = __builtin_amdgcn_ballot_w64(meta.pid >= 0), rem2 = __builtin_amdgcn_ballot_w64(meta2.pid >= 0);
  const int np = __builtin_popcountll(rem) + __builtin_popcountll(rem2);
  auto next_page = [&]() {   // entry index of the next live page (0 past the end)
    if (rem) return take(rem);
    if (rem2) return 64 + take(rem2);
    return 0;
  };
  auto pick = [&](int v, int v2, int idx) {
    const int x = __builtin_amdgcn_readlane(v, idx & 63), x2 = __builtin_amdgcn_readlane(v2, idx & 63);
    return idx >= 64 ? x2 : x;
  };
  auto page_pid = [&](int idx) { return pick(meta.pid, meta2.pid, idx); };
  auto page_tag = [&](int idx) { return pick(meta.tag, meta2.tag, idx); };
  auto page_scale = [&](int idx) {
    return u2f((uint32_t)pick((int)f2u(meta.scale), (int)f2u(meta2.scale), idx));
  };
  const int mine = np > w ? (np - w + FEW_WAVES - 1) / FEW_WAVES : 0;   // pages of this wave
  int cur = 0;
  for (int k = 0; k <= w; ++k) cur = next_page();
  if (mine > 0) few_dma<DQK, DV>(ring[w][0], a, page_pid(cur), page_tag(cur), lane);

  // Q of the lane's head, rounded to f16: dims 32i + 8g .. +7
  h8 q[C::KSTEPS];
  {
    const bool live = head < a.H;
    const int64_t off = (int64_t)b * a.qsb + (int64_t)(live ? head : 0) * a.qsh + 8 * g;
    if (a.q_dtype == IAK_DTYPE_F32) {
#pragma unroll
      for (int i = 0; i < C::KSTEPS; ++i) {
        const f4* p = reinterpret_cast<const f4*>(reinterpret_cast<const float*>(a.q) + off + 32 * i);
        const f4 x0 = p[0], x1 = p[1];
#pragma unroll
        for (int e = 0; e < 4; ++e) { q[i][e] = (_Float16)x0[e]; q[i][4 + e] = (_Float16)x1[e]; }
      }
    } else if (a.q_dtype == IAK_DTYPE_F16) {
#pragma unroll
      for (int i = 0; i < C::KSTEPS; ++i)
        q[i] = *reinterpret_cast<const h8*>(reinterpret_cast<const _Float16*>(a.q) + off + 32 * i);
    } else {
#pragma unroll
      for (int i = 0; i < C::KSTEPS; ++i) {
        const u4 x = *reinterpret_cast<const u4*>(reinterpret_cast<const uint16_t*>(a.q) + off + 32 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          q[i][2 * e] = (_Float16)u2f(x[e] << 16);
          q[i][2 * e + 1] = (_Float16)u2f(x[e] & 0xFFFF0000u);
        }
      }
    }
    if (!live)
#pragma unroll
      for (int i = 0; i < C::KSTEPS; ++i) q[i] = h8{0, 0, 0, 0, 0, 0, 0, 0};
  }

  float m = -__builtin_inff(), l = 0.f;
  int E = 0;               // value exponent (wave-uniform): the value sum is acc * 2^E
  f4 acc[C::NDB];          // tile db: rows = heads 4g .. 4g+3, column = value dim 16 db + c
#pragma unroll
  for (int db = 0; db < C::NDB; ++db) acc[db] = f4{0.f, 0.f, 0.f, 0.f};
  // the lane's part of the operand reads: score row c, piece g (the swizzle acts on
  // the low bits of a piece, pieces 4i change the others too: one xor each); value
  // row 4g + c / 4, eight bytes (VOFF / 4 + c % 4)
  const int vrow = 4 * g + (c >> 2), vp = (a.VOFF >> 2) + (c & 3);

  for (int t = 0; t < mine; ++t) {
    uint8_t* slot = ring[w][t & 1];
    const int tag = page_tag(cur);
    const bool more = t + 1 < mine;
    int nx = cur;
    if (more) {
      for (int k = 0; k < FEW_WAVES; ++k) nx = next_page();
      const int ntag = page_tag(nx);
      // the other slot's last reads fed matrix instructions already issued
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      few_dma<DQK, DV>(ring[w][(t + 1) & 1], a, page_pid(nx), ntag, lane);
      if (ntag == IAK_TAG_FP16) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(C::N16) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(C::N8) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    if (tag != IAK_TAG_FP16) few_convert<DQK, DV>(slot, tag, lane);

    // ---- scores: two chains ----
    f4 s = f4{0.f, 0.f, 0.f, 0.f}, s1 = s;
    const uint8_t* krow = slot + c * C::RB;
#pragma unroll
    for (int i = 0; i < C::KSTEPS; ++i) {
      const h8 kf = *reinterpret_cast<const h8*>(krow + 16 * ((4 * i + g) ^ C::swz(c)));
      if (i & 1) s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, q[i], s1, 0, 0, 0);
      else s = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, q[i], s, 0, 0, 0);
    }
    s += s1;
    // ---- softmax over the page's 16 tokens ----
    const float ps = page_scale(cur);
    s *= a.score_mult * ps;
    const int64_t end = (int64_t)(start + cur + 1) * PS;
    if (end > limit) {
      const int64_t lim = (int64_t)limit - (end - PS) - 4 * g;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r >= lim) s[r] = -__builtin_inff();
    }
    const float pm = xmax16_32(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])));
    const bool grow = pm > m + RESCALE_SLACK;
    float al = 1.0f;
    if (grow) {
      al = __builtin_amdgcn_exp2f(m - pm);   // 0 on the first page (m = -inf)
      m = pm;
    }
    const int e = scale_exp(ps);
    const bool emove = e > E + EXP_WINDOW || e < E - EXP_WINDOW;
    const float efac = emove ? pow2f(E - e) : 1.0f;
    if (emove) E = e;
    const float vm = pow2f(-E);
    f4 p;
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f(s[r] - m);
    l = l * al + ((p[0] + p[1]) + (p[2] + p[3]));
    h4 pa;
#pragma unroll
    for (int r = 0; r < 4; ++r) pa[r] = (_Float16)(p[r] * (ps * vm));
    if (__builtin_amdgcn_ballot_w64(grow) != 0 || emove) {
      f4 ar;
#pragma unroll
      for (int r = 0; r < 4; ++r) ar[r] = __shfl(al, 4 * g + r, 64) * efac;
#pragma unroll
      for (int db = 0; db < C::NDB; ++db) acc[db] *= ar;
    }
    // ---- values ----
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s4 lds_s4;
    const uint8_t* vr = slot + vrow * C::RB + 8 * (vp & 1);
#pragma unroll
    for (int db = 0; db < C::NDB; ++db) {
      const uint8_t* at = vr + 16 * ((2 * db + (vp >> 1)) ^ C::swz(vrow));
      const h4 vf = __builtin_bit_cast(h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(at)));
      acc[db] = __builtin_amdgcn_mfma_f32_16x16x16f16(pa, vf, acc[db], 0, 0, 0);
    }
    cur = nx;
  }

  // ---- the four waves' contexts meet in the ring, [wave][head][dim] ----
  const float ls = xsum16_32(l);
  if (g == 0) {
    red_m[w][c] = m;
    red_l[w][c] = ls;
  }
  __syncthreads();   // every wave is past its last page: the ring is free
  float* red = reinterpret_cast<float*>(&ring[0][0][0]);
  const float vscale = pow2f(E);
#pragma unroll
  for (int db = 0; db < C::NDB; ++db)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[(w * FEW_HEADS + 4 * g + r) * DV + 16 * db + c] = acc[db][r] * vscale;
  __syncthreads();
  // thread: four dims of one head at a time
  for (int i = tid; i < FEW_HEADS * DV / 4; i += 64 * FEW_WAVES) {
    const int hl = i / (DV / 4), d = 4 * (i - hl * (DV / 4)), h = h0 + hl;
    if (h >= a.H) break;   // heads ascend with i
    float M = -__builtin_inff();
#pragma unroll
    for (int k = 0; k < FEW_WAVES; ++k) M = fmaxf(M, red_m[k][hl]);
    float L = 0.f;
    f4 v = f4{0.f, 0.f, 0.f, 0.f};
    if (M > -__builtin_inff()) {
#pragma unroll
      for (int k = 0; k < FEW_WAVES; ++k) {
        const float wt = __builtin_amdgcn_exp2f(red_m[k][hl] - M);   // 0 for a wave without a page (m = -inf)
        L += wt * red_l[k][hl];
        v += wt * *reinterpret_cast<const f4*>(red + (k * FEW_HEADS + hl) * DV + d);
      }
    }
    const float inv = L > 0.f ? 1.0f / L : 0.0f;
    if (a.splits == 1) {
      const int64_t o = (int64_t)b * a.osb + (int64_t)h * a.osh + d;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (a.out_dtype == IAK_DTYPE_F32) reinterpret_cast<float*>(a.out)[o + e] = v[e] * inv;
        else if (a.out_dtype == IAK_DTYPE_F16) reinterpret_cast<_Float16*>(a.out)[o + e] = (_Float16)(v[e] * inv);
        else reinterpret_cast<__bf16*>(a.out)[o + e] = (__bf16)(v[e] * inv);
      }
      continue;
    }
    const int64_t at = ((int64_t)b * a.splits + split) * a.H + h;
    if (d == 0) {
      a.ws_m[at] = M;
      a.ws_l[at] = L;
    }
    if (a.acc16) {
      h4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = (_Float16)(v[e] * inv);
      *reinterpret_cast<h4*>(reinterpret_cast<_Float16*>(a.ws_acc) + at * DV + d) = y;
    } else {
      *reinterpret_cast<f4*>(a.ws_acc + at * DV + d) = v;
    }
  }
}

#endif
