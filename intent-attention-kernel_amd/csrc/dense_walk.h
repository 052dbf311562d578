// The body of dense_matrix_kernel and of mx_walk, included by dense_matrix.h in both: inlined from a
// function, the compiler schedules the tile loop otherwise (32 heads x 2,048 rows x
// 128, causal, 84 / 88 us; 40 x 2,048 x 64 78 / 84).
  using C = MxCfg<T, DP, QW, KW, BKW, GEN>;
  using E = MxElem<T>;
  using vec = typename E::vec;
  constexpr bool F32 = sizeof(T) == 4;
  constexpr int BK = C::BK, RB = C::RB, CH = C::CH, NCH = C::NCH, NSB = C::NSB, NDV = C::NDV;
  constexpr int PARTS = PLAIN ? 1 : E::PARTS;
  // Weights are kept as p * 2^PEXP; the running maximum lags by up to SLACK (exp2 domain).
  // float16: 2^12 and 2^3, together the 2^15 that fits: a weight is off by at most half the
  // smallest subnormal step, 2^-37 of the row's largest weight; 2^7 and 2^8, 2^-32, left
  // six bits to a weight of 2^-25. (Causal, 32 x 2,048 x 128, us per call: a lag of 2^8 81.3,
  // of 2^3 82.1, none 83.6.)
  constexpr bool F16 = __is_same(T, _Float16), LAGS = !F32 && !F16 && !AGAIN;
  constexpr float PEXP = F16 ? 12.f : LAGS ? 7.f : 0.f, SLACK = F16 ? 3.f : LAGS ? RESCALE_SLACK : 0.f;
  int tid = threadIdx.x;
  // (AGAIN: what both walks work out from the lane's place would be held in registers from
  // the first to the second)
  if constexpr (AGAIN) asm volatile("" : "+v"(tid));
  const int lane = tid & 63;
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
    if (AGAIN || !mp.flags) return false;
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
  auto store_v = [&](int buf, int t) {   // tile t's
    if ((F32 || AGAIN) && lo + (t + 1) * BK > hi) {   // the rows past the range are zeros
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        int r, c;
        piece(i, r, c);
        if (lo + t * BK + r >= hi) (C::STAGED ? kr[i] : vr[C::STAGED ? 0 : i]) = u4{0u, 0u, 0u, 0u};
      }
    }
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
      cur = fabsf(x) > 0x1p23f ? x : x - PEXP;   // up to there the difference is exact
    }
    const bool grow = cur > m + (GEN ? SLACK / LOG2E : SLACK);
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
    if constexpr (PLAIN) {
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[sb][r] = s[sb][r] > 0.f ? 1.f : s[sb][r];
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
      store_v(0, 0);
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
        store_v(0, t + 1);
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
      store_v(0, 0);
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
        store_v(next, t + 1);
      }
    }
  }
  // key tiles that no query tile visits (keys past the last row's diagonal): checked here
  if (mp.flags && mp.skip) {
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
  [[maybe_unused]] bool again = false;   // AGAIN: a sum is not finite
  if constexpr (AGAIN && !PLAIN) {
    float x = 0.f;
#pragma unroll
    for (int d = 0; d < NDV; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) x = __builtin_fmaf(acc[d][r], 0.f, x);
    again = x != x;
  }
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
    if constexpr (PLAIN) {   // only what is not finite
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (!(fabsf(v[e]) < __builtin_inff())) store_t<T>(o, e, v[e]);
      return;
    }
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
    if (!ok4) MX_DONE;
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
    if (r >= a.q_len) MX_DONE;
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
