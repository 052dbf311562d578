// The MLA output projection context . W_VO for a decode step's few rows, in float32:
// out[row, n] = sum over k of context[row, k] w[k, n]. Included by mla_rows.hip only.
//
// W is read once, as it is stored, by workgroups of 32 columns and eight waves; wave
// w takes every eighth group of eight k (a group is four v_mfma_f32_32x32x2_f32: half
// h of the wave holds k = 8 g + 4 h + e in instruction e), and the waves' sums meet in
// the LDS, added pairwise. Every product is a float32 product and every sum float32.
// Bound: the chain of launch, W's first line and the waves' meeting; W is 4.7 MB at
// 576 x 4,096 in float16, 1 us at the rate of HBM. 32 rows x 576 x 4,096, us per call:
// W to float32 and a library GEMM 24.7 to 35, this 7.0 (the kernel's trace, which includes its
// start, 8.9); 128 rows 24.7 / 11.0; 32 rows x 128 x 1,024 23.1 / 3.8. Error against float64 4.3e-7 -> 1.6e-7 (the waves' short chains).
#ifndef IAK_MLA_PROJECT_H
#define IAK_MLA_PROJECT_H

constexpr int PJ_WAVES = 8, PJ_COLS = 32, PJ_ROWS = 32;
constexpr int PJ_BATCH = 5;   // groups whose loads are in flight together

template <typename T>
__global__ __launch_bounds__(64 * PJ_WAVES) void mla_project_kernel(const iak_mla_project_args a) {
  __shared__ float part[PJ_WAVES][16][64];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  const int n0 = blockIdx.x * PJ_COLS, r0 = blockIdx.y * PJ_ROWS;
  const int row = r0 + l32 < a.rows ? r0 + l32 : a.rows - 1;
  const float* x = a.context + (int64_t)row * a.latent_dim + 4 * h;
  const T* wp = reinterpret_cast<const T*>(a.w) + n0 + l32;
  const int groups = a.latent_dim / 8;

  f16v acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  for (int g0 = w; g0 < groups; g0 += PJ_WAVES * PJ_BATCH) {
    f4 xa[PJ_BATCH];
    T wb[PJ_BATCH][4];
#pragma unroll
    for (int i = 0; i < PJ_BATCH; ++i) {
      const int g = g0 + PJ_WAVES * i < groups ? g0 + PJ_WAVES * i : g0;   // past the end: loaded, not used
      xa[i] = *reinterpret_cast<const f4*>(x + 8 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) wb[i][e] = wp[(int64_t)(8 * g + 4 * h + e) * a.w_stride];
    }
#pragma unroll
    for (int i = 0; i < PJ_BATCH; ++i)
      if (g0 + PJ_WAVES * i < groups)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc = __builtin_amdgcn_mfma_f32_32x32x2f32(xa[i][e], to_f32(wb[i][e]), acc, 0, 0, 0);
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) part[w][r][lane] = acc[r];
  __syncthreads();
  // register r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32
#pragma unroll
  for (int i = 0; i < 16 / PJ_WAVES; ++i) {
    const int r = w + PJ_WAVES * i;
    const float y = ((part[0][r][lane] + part[1][r][lane]) + (part[2][r][lane] + part[3][r][lane])) +
                    ((part[4][r][lane] + part[5][r][lane]) + (part[6][r][lane] + part[7][r][lane]));
    const int ro = r0 + 8 * (r >> 2) + 4 * h + (r & 3);
    if (ro >= a.rows) continue;
    const int64_t at = (int64_t)ro * a.d_out + n0 + l32;
    if (a.out_dtype == IAK_DTYPE_F32) reinterpret_cast<float*>(a.out)[at] = y;
    else if (a.out_dtype == IAK_DTYPE_F16) reinterpret_cast<_Float16*>(a.out)[at] = (_Float16)y;
    else reinterpret_cast<__bf16*>(a.out)[at] = (__bf16)y;
  }
}

#endif
