// Products of a step of few rows over bf16 weights: C[b][m][n] (+)= sum_k A[b][m][k] W[b][n][k], up to 32 rows of A (bf16 or fp32; any number over up to
// 64 columns), fp32 sums; the form that vlm_linear_any takes for them.
//
// The weights are read once and bound it, so the launch is laid out for them: a workgroup owns R <= 16 weight rows (x NT) with their whole K - a
// compute unit draws about 25 GB/s whatever its waves do, so narrow outputs take R = N / 256 and fill the chip with tiles whose other MFMA rows
// repeat the last one - and its waves interleave the 64-wide pieces of K, U pieces in flight each.  A lane holds 16 neighbouring k of weight row
// lane % 16 and of activation row lane % 16 (k in the same order in both, which is all the product needs), so four lanes read 128 contiguous
// bytes of a row.  bf16 rows on v_mfma_f32_16x16x32_bf16, fp32 rows on v_mfma_f32_16x16x4_f32 with the weights widened.  The waves' tiles meet in
// LDS and are added up in a fixed order.
#include "common.hpp"
#include "internal.h"
#include "../../include/vlm_hip.h"
#include "recurrence_finish.hpp"

namespace {

struct RowsArgs {
  const void* A;
  const bf16_t* W;
  void* C;
  int M, N, K, R, accumulate;
  long lda, ldw, ldc, sA, sW, sC;
};

template <typename TA, typename TC, int MT, int NT, int U, bool TURNS = false>
__global__ __launch_bounds__(256) void linear_rows_mfma_kernel(RowsArgs p) {
  constexpr int PITCH = 20, WAVES = 4, AV = sizeof(TA) == 2 ? 2 : 4, PER = 16 / AV;          // 16-byte pieces of a lane's 16 activations
  __shared__ __align__(16) float red[WAVES][NT * MT][16 * PITCH];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r16 = lane & 15, g = lane >> 4;
  const int R = p.R, K = p.K, n0 = blockIdx.x * R * NT, cols = min(R * NT, p.N - n0), m0 = blockIdx.z * 16 * MT, M = p.M - m0;
  const TA* A = (const TA*)p.A + blockIdx.y * p.sA + m0 * p.lda;
  const bf16_t* W = p.W + blockIdx.y * p.sW;
  f32x4_t acc[NT][MT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const bf16_t* w[NT];
  const TA* a[MT];
#pragma unroll
  for (int j = 0; j < NT; ++j) w[j] = W + (long)min(n0 + j * R + min(r16, R - 1), p.N - 1) * p.ldw;
#pragma unroll
  for (int i = 0; i < MT; ++i) a[i] = A + (long)min(16 * i + r16, M - 1) * p.lda;
  const int chunks = (K + 63) / 64;
  for (int c0 = wave; c0 < chunks; c0 += U * WAVES) {
    u32x4_t wv[U][NT][2], av[U][MT][AV];
    const auto load = [&](int u, bool inside) {
      const int k0 = (c0 + u * WAVES) * 64 + 16 * g;
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int k = inside ? k0 + 8 * x : min(k0 + 8 * x, K - 8);
#pragma unroll
        for (int j = 0; j < NT; ++j) wv[u][j][x] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(w[j] + k));
      }
#pragma unroll
      for (int x = 0; x < AV; ++x) {
        const int k = inside ? k0 + PER * x : min(k0 + PER * x, K - PER);
#pragma unroll
        for (int i = 0; i < MT; ++i) av[u][i][x] = *reinterpret_cast<const u32x4_t*>(a[i] + k);
      }
    };
    if ((c0 + (U - 1) * WAVES + 1) * 64 <= K) {
#pragma unroll
      for (int u = 0; u < U; ++u) load(u, true);
    } else {                                                         // the last pieces: zeros past K
#pragma unroll
      for (int u = 0; u < U; ++u) load(u, false);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const u32x4_t none = {0u, 0u, 0u, 0u};
        const int k0 = (c0 + u * WAVES) * 64 + 16 * g;
#pragma unroll
        for (int x = 0; x < 2; ++x)
          if (k0 + 8 * x >= K)
#pragma unroll
            for (int j = 0; j < NT; ++j) wv[u][j][x] = none;
#pragma unroll
        for (int x = 0; x < AV; ++x)
          if (k0 + PER * x >= K)
#pragma unroll
            for (int i = 0; i < MT; ++i) av[u][i][x] = none;
      }
    }
    // short chains on the matrix unit, added up by rounding additions: long ones round worse (router logits of 8 rows, K = 1536: relative error
    // 1.3e-7 in one chain a wave, 7e-8 so).  TURNS, fp32 results of up to 8 rows: the U pieces of a turn are added to each other first, which is as close as
    // vlm_linear_rows_bf16w or closer (K = 4096 / 17920: 9.5e-8 / 1.67e-7 one by one, 7.95e-8 / 1.07e-7 so, 8.3e-8 / 1.30e-7 there)
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t turn[NT][MT];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          f32x4_t t[4] = {zero, zero, zero, zero};
          if constexpr (sizeof(TA) == 2) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
              t[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wv[u][j][x]), __builtin_bit_cast(bf16x8_t, av[u][i][x]), zero, 0, 0, 0);
            t[0] += t[1];
          } else {
#pragma unroll
            for (int y = 0; y < 16; ++y) {
              const unsigned q = wv[u][j][y / 8][y % 8 / 2], z = av[u][i][y / 4][y % 4];
              t[y % 4] = __builtin_amdgcn_mfma_f32_16x16x4f32(y & 1 ? bf_hi(q) : bf_lo(q), __builtin_bit_cast(float, z), t[y % 4], 0, 0, 0);
            }
            t[0] = (t[0] + t[1]) + (t[2] + t[3]);
          }
          if constexpr (TURNS) {
            turn[j][i] = u ? turn[j][i] + t[0] : t[0];
            if (u == U - 1) acc[j][i] += turn[j][i];
          } else {
            acc[j][i] += t[0];
          }
        }
  }
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) *reinterpret_cast<f32x4_t*>(&red[wave][j * MT + i][r16 * PITCH + 4 * g]) = acc[j][i];
  __syncthreads();
  TC* C = (TC*)p.C + blockIdx.y * p.sC + m0 * p.ldc;
  for (int i = tid; i < NT * MT * 256; i += 256) {
    const int tile = i >> 8, m = (tile % MT) * 16 + ((i >> 4) & 15), n = i & 15, at = ((i >> 4) & 15) * PITCH + n;
    const int c = (tile / MT) * R + n;
    if (m >= M || n >= R || c >= cols) continue;
    const float v = (red[0][tile][at] + red[1][tile][at]) + (red[2][tile][at] + red[3][tile][at]);
    TC* out = C + (long)m * p.ldc + n0 + c;
    st_f(out, p.accumulate ? ld_f(out) + v : v);
  }
}

// R and NT (microseconds inside a graph, N x K, 8 bf16 rows): 1536 x 1536 R 6 NT 1 4.5, R 16 NT 1 8; 3584 x 3584 R 14 NT 1 8.8; from 4096 columns
// on two tiles a wave share the activations: 4616 x 1536 R 10 NT 2 6.1, R 16 NT 1 7.6; 4608 x 3584 10.5 and 12.2.  Eight or sixteen waves instead
// of four: 1536 x 8960 13.1 and 14.5 instead of 11.8.
// Maps: as many workgroups a map as leave no compute unit two of them (us, 16 rows, 12 maps
// [512, 128]: 264 workgroups of R 12 4.4, 240 of R 13 3.6; 9 rows, 28 maps [256, 192]: 308 of R 12 5.4, 252 of R 15 3.9).
template <typename TA, typename TC>
void launch_rows(RowsArgs a, int batch, hipStream_t st) {
  const int nt = (long)a.N * batch <= 4096 ? 1 : 2, per = std::max(1, 256 / batch) * nt;
  a.R = std::min(16, (a.N + per - 1) / per);
  const dim3 grid((a.N + a.R * nt - 1) / (a.R * nt), batch), block(256);
  constexpr bool f = sizeof(TA) == 4;
  if constexpr (!f && sizeof(TC) == 4)
    if (a.M <= 8) {
      if (nt == 1) hipLaunchKernelGGL((linear_rows_mfma_kernel<TA, TC, 1, 1, 4, true>), grid, block, 0, st, a);
      else hipLaunchKernelGGL((linear_rows_mfma_kernel<TA, TC, 1, 2, 3, true>), grid, block, 0, st, a);
      return;
    }
  if (a.M > 32) {                                                    // (few columns: blocks of 16 rows fill the chip)
    a.R = std::min(16, a.N);
    hipLaunchKernelGGL((linear_rows_mfma_kernel<TA, TC, 1, 1, f ? 3 : 4>), dim3((a.N + a.R - 1) / a.R, batch, (a.M + 15) / 16), block, 0, st, a);
  } else if (a.M <= 16) {
    if (nt == 1) hipLaunchKernelGGL((linear_rows_mfma_kernel<TA, TC, 1, 1, f ? 3 : 4>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((linear_rows_mfma_kernel<TA, TC, 1, 2, f ? 2 : 3>), grid, block, 0, st, a);
  } else {
    if (nt == 1) hipLaunchKernelGGL((linear_rows_mfma_kernel<TA, TC, 2, 1, f ? 2 : 3>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((linear_rows_mfma_kernel<TA, TC, 2, 2, f ? 1 : 2>), grid, block, 0, st, a);
  }
}

}  // namespace

VLM_INTERNAL int vlm_linear_rows_mfma_try(const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc, int a_f32, int c_f32,
                                          int batch, long sA, long sW, long sC, int accumulate, void* stream) {
  // where the line lies: wider outputs fill the chip with whole tiles (9000 x 3584, 8 rows: 17.7 us on the GEMM's, 25.7 here), a longer K is better split
  // over workgroups (1536 x 8960, 16 rows: 12.6 and 15.2); many narrow maps of up to 8 rows are cheap here (28 of [512, 128]: 12.9 -> 4.6)
  // fp32 sums onto a stream keep the long K here up to 8 rows: the split form hands over bf16 (1536 x 21696, 2 / 4 / 8 rows: 26 / 26 / 32; vlm_linear_rows_bf16w
  // 48 / 76 / 140)
  // two or three fp32 rows over a short K are cheaper a wave a column (2 rows, [2048, K], K = 64 / 256 / 384: 3.1 / 3.7 / 4.2, here 3.5 / 3.9 / 3.8; 3 rows,
  // [1024, 64]: 3.3, 3.7)
  if (a_f32 && (M == 2 ? K <= 256 : M == 3 && K <= 64)) return -1;
  const int va = a_f32 ? 4 : 8;
  // more rows over few columns, as blocks of 16: router logits [8, 1536] of 2048 rows 29 -> 7.5 us
  if (M > 32 ? N > 64 || batch > 1 || M > 65535 * 16 : false) return -1;
  const bool fits = (long)N * batch <= 8192 || (M <= 8 && (long)N * batch * K <= 4 << 20);
  if (!fits || (K > 4096 && !(accumulate && !a_f32 && M <= 8)) || K % 8 || lda % va || sA % va || ldw % 8 || sW % 8 || (((uintptr_t)A | (uintptr_t)W) & 15)) return -1;
  const RowsArgs a{A, (const bf16_t*)W, C, M, N, K, 0, accumulate, lda, ldw, ldc, sA, sW, sC};
  hipStream_t st = (hipStream_t)stream;
  if (a_f32) c_f32 ? launch_rows<float, float>(a, batch, st) : launch_rows<float, bf16_t>(a, batch, st);
  else c_f32 ? launch_rows<bf16_t, float>(a, batch, st) : launch_rows<bf16_t, bf16_t>(a, batch, st);
  VLM_CHECK_LAUNCH();
  return VLM_OK;
}
