// Generic strided, batched linear layer for the shapes and number formats the MFMA GEMMs (gemm_bf16.hip) do not take:
//
//     C[b][m][n] (+)= sum_k A[b][m][k] * W[b][n][k]          b < batch, any M, N, K, any leading dimension
//
// A, W and C are each bf16 or fp32 (codes 0 / 1).  A product with an fp32 operand is fp32 throughout, on v_mfma_f32_16x16x4_f32 (linear_f32_ranges_kernel and
// linear_f32_tiles_kernel: an output is eight chains over fixed pieces of k, added in a fixed order).  With all three in fp32 - the true 32-bit product of
// the float32 serving mode - that holds for every number of rows, so a row of C depends on nothing but its own row of A: the result of a token is the same
// bits whatever else is in the batch and however a prompt was cut into steps.  With bf16 weights the number of rows chooses the kernel (few rows:
// linear_rows_kernel and linear_rows_mfma.hip), and with it the order of the sums.  fp32 C and `accumulate` add a projection straight onto an fp32
// residual stream.
//
// bf16 A and W with aligned rows and more than 8 rows of A take the bf16 matrix cores (linear_any_mfma_kernel: fp32 sums in blocks of 32 k).
//
// Per-head projections of one tensor (latent attention's absorbed key / value maps) run as `batch` with element strides between heads.
#include "common.hpp"
#include "internal.h"
#include "../../include/vlm_hip.h"

namespace {

template <typename T> __device__ __forceinline__ float ld_f(const T* p);
template <> __device__ __forceinline__ float ld_f<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float ld_f<bf16_t>(const bf16_t* p) { return bf2f(*p); }
template <typename T> __device__ __forceinline__ void st_f(T* p, float v);
template <> __device__ __forceinline__ void st_f<float>(float* p, float v) { *p = v; }
template <> __device__ __forceinline__ void st_f<bf16_t>(bf16_t* p, float v) { *p = f2bf(v); }

// Products with an fp32 operand.  What bounds them: the fp32 matrix rate (154 TFLOP/s reached by a large library product here) for prompts (70-90 reached here), the
// weights' way from memory for a few rows.  k is cut into slabs of 32 and the slabs into eight ranges; a range is one chain of products, the
// eight sums s0 .. s7 are added as (((s0 + s1) + s2) + s3) + (((s4 + s5) + s6) + s7).  Two kernels compute just that, so that the choice between
// them may depend on the number of rows: linear_f32_ranges_kernel gives each range a wave (few tiles: eight waves per tile stream the
// operands), linear_f32_tiles_kernel runs them one after the other on tiles that share operands through LDS.
// In a slab lane (row, g) of an operand holds k = 8 g .. 8 g + 7 of its row, whole 16-byte pieces in both formats; product e takes element e
// of every lane.
constexpr int FW = 8, FS = 32;             // ranges, k per slab

typedef __attribute__((ext_vector_type(8))) float f32x8_t;
template <typename T> struct PieceOf { typedef f32x8_t type; };          // eight k of a lane
template <> struct PieceOf<bf16_t> { typedef u32x4_t type; };
template <typename T> using Piece = typename PieceOf<T>::type;
__device__ __forceinline__ float elem(const f32x8_t& v, int e) { return v[e]; }
__device__ __forceinline__ float elem(const u32x4_t& v, int e) {
  const unsigned u = v[e >> 1];
  return e & 1 ? bf_hi(u) : bf_lo(u);
}
__device__ __forceinline__ f32x8_t join(f32x4_t lo, f32x4_t hi) { return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7); }
// (a vector type of an element's alignment: rows that are not whole aligned pieces are read in 16-byte accesses all the same)
typedef f32x4_t f32x4_at4_t __attribute__((aligned(4)));
typedef u32x4_t u32x4_at2_t __attribute__((aligned(2)));
template <typename T, bool VEC>
__device__ __forceinline__ Piece<T> piece(const T* p, int left) {          // left: elements before K
  if constexpr (VEC) {
    if constexpr (sizeof(T) == 4) return join(*reinterpret_cast<const f32x4_t*>(p), *reinterpret_cast<const f32x4_t*>(p + 4));
    else return *reinterpret_cast<const u32x4_t*>(p);
  } else if constexpr (sizeof(T) == 4) {
    if (left >= 8) return join(*reinterpret_cast<const f32x4_at4_t*>(p), *reinterpret_cast<const f32x4_at4_t*>(p + 4));
    f32x8_t r;
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = j < left ? p[j] : 0.f;
    return r;
  } else {
    if (left >= 8) return *reinterpret_cast<const u32x4_at2_t*>(p);
    u32x4_t r;
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = (2 * j < left ? (unsigned)p[2 * j] : 0u) | (2 * j + 1 < left ? (unsigned)p[2 * j + 1] << 16 : 0u);
    return r;
  }
}
// the 16 bytes of a piece that begin at p (fp32: half of one)
template <typename T>
__device__ __forceinline__ u32x4_t bytes16(const T* p, int left) {
  if constexpr (sizeof(T) == 4) {
    if (left >= 4) return __builtin_bit_cast(u32x4_t, (f32x4_t)*reinterpret_cast<const f32x4_at4_t*>(p));
    f32x4_t r;
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = j < left ? p[j] : 0.f;
    return __builtin_bit_cast(u32x4_t, r);
  } else {
    return piece<T, false>(p, left);
  }
}
__device__ __forceinline__ f32x4_t mfma_f32(float w, float a, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(w, a, c, 0, 0, 0); }

// consecutive workgroups go to the eight XCDs in turn: one XCD walks a run of tiles, all row tiles of a column tile after each other, so that a
// weight row is read into one L2
__device__ __forceinline__ bool tile_of(int mtiles, int ntiles, int& mt, int& nt) {
  const int id = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  nt = id / mtiles;
  mt = id % mtiles;
  return nt < ntiles;
}

// a workgroup: one tile of MI x NJ products, wave c is range c.  VEC: rows in whole aligned 16-byte pieces (else element by element)
template <typename TA, typename TW, typename TC, int MI, int NJ, bool VEC>
__global__ __launch_bounds__(64 * FW) void linear_f32_ranges_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C, int M, int N,
                                                                    int K, long lda, long ldw, long ldc, long sA, long sW, long sC, int accumulate,
                                                                    int mtiles, int ntiles) {
  constexpr int TM = 16 * MI, TN = 16 * NJ;
  __shared__ __align__(16) float part[FW][16][TN + 4];
  int mt, nt;
  if (!tile_of(mtiles, ntiles, mt, nt)) return;          // (whole workgroups)
  const int m0 = mt * TM, n0 = nt * TN;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  A += (long)blockIdx.z * sA;
  W += (long)blockIdx.z * sW;
  C += (long)blockIdx.z * sC;
  const TA* ar[MI];
  const TW* wr[NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i) ar[i] = A + (long)min(m0 + 16 * i + r16, M - 1) * lda + 8 * g;
#pragma unroll
  for (int j = 0; j < NJ; ++j) wr[j] = W + (long)min(n0 + 16 * j + r16, N - 1) * ldw + 8 * g;
  f32x4_t acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  constexpr int P = MI * NJ == 1 ? 6 : MI * NJ == 4 ? 4 : 3;          // slabs in flight
  Piece<TA> a[P][MI];
  Piece<TW> w[P][NJ];
  const int slabs = (K + FS - 1) / FS, range = (slabs + FW - 1) / FW, live = (slabs + range - 1) / range;
  const int s0 = wave * range, s1 = min(s0 + range, K / FS);           // whole slabs of this wave
  const auto load = [&](int b, int s) {
    const int k = min(s, s1 - 1) * FS;
#pragma unroll
    for (int i = 0; i < MI; ++i) a[b][i] = piece<TA, VEC>(ar[i] + k, 8);
#pragma unroll
    for (int j = 0; j < NJ; ++j) w[b][j] = piece<TW, VEC>(wr[j] + k, 8);
  };
  const auto multiply = [&](int b) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = mfma_f32(elem(w[b][j], e), elem(a[b][i], e), acc[i][j]);
  };
  if (s0 < s1) {
#pragma unroll
    for (int u = 0; u < P; ++u) load(u, s0 + u);
    int s = s0;
    for (; s + P <= s1; s += P) {
#pragma unroll
      for (int u = 0; u < P; ++u) {
        multiply(u);
        load(u, s + u + P);
      }
    }
#pragma unroll
    for (int u = 0; u < P; ++u)
      if (s + u < s1) multiply(u);
  }
  if (K % FS && wave == live - 1) {                      // the last, shorter slab: zeros past K
    const int k = K / FS * FS;
#pragma unroll
    for (int i = 0; i < MI; ++i) a[0][i] = piece<TA, false>(ar[i] + k, K - k - 8 * g);
#pragma unroll
    for (int j = 0; j < NJ; ++j) w[0][j] = piece<TW, false>(wr[j] + k, K - k - 8 * g);
    multiply(0);
  }
  // 16 rows at a time: every wave's sums to LDS, added up by the lane that stores the output
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    if (i) __syncthreads();
    if (wave < live)
#pragma unroll
      for (int j = 0; j < NJ; ++j) *reinterpret_cast<f32x4_t*>(&part[wave][r16][16 * j + 4 * g]) = acc[i][j];
    __syncthreads();
#pragma unroll
    for (int o = threadIdx.x; o < 16 * TN; o += 64 * FW) {
      const int m = m0 + 16 * i + o / TN, n = n0 + o % TN;
      if (m >= M || n >= N) continue;
      float t[2] = {0.f, 0.f};
#pragma unroll
      for (int c = 0; c < FW; ++c)
        if (c < live) t[c / 4] += part[c][o / TN][o % TN];
      const float v = t[0] + t[1];
      TC* c = C + (long)m * ldc + n;
      st_f(c, accumulate ? ld_f(c) + v : v);
    }
  }
}

// a workgroup: one tile of 2 MI x 2 NJ products on two groups of 2 x 2 waves, group q runs ranges 4 q .. 4 q + 3 over its own stages of LDS.
// A slab arrives in LDS by 16-byte direct loads in the operand order (16 rows x 64 lanes per load), so that an operand is one linear read;
// ST slabs are resident, ST - 2 in flight under the products.  VEC: rows in whole aligned 16-byte pieces; others pass through registers, the next slab's
// loads under this one's products (ST = 2).
template <typename TA, typename TW, typename TC, int MI, int NJ, int ST, bool VEC>
__global__ __launch_bounds__(512) void linear_f32_tiles_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C, int M, int N, int K,
                                                               long lda, long ldw, long ldc, long sA, long sW, long sC, int accumulate, int mtiles,
                                                               int ntiles) {
  constexpr int TM = 32 * MI, TN = 32 * NJ;
  constexpr int HA = sizeof(TA) / 2, HW = sizeof(TW) / 2;              // loads per 16 rows of a slab
  constexpr int LA = TM / 16 * HA, LW = TN / 16 * HW, L = LA + LW, PER = (L + 3) / 4;
  extern __shared__ __align__(16) char smem[];                         // [2 groups][ST][L][64 lanes][16 bytes]
  int mt, nt;
  if (!tile_of(mtiles, ntiles, mt, nt)) return;          // (whole workgroups)
  const int m0 = mt * TM, n0 = nt * TN;
  const int q = threadIdx.x >> 8, wave = (threadIdx.x >> 6) & 3, lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int wm = (wave & 1) * MI, wn = (wave >> 1) * NJ;               // first 16-row blocks of this wave's products
  A += (long)blockIdx.z * sA;
  W += (long)blockIdx.z * sW;
  C += (long)blockIdx.z * sC;
  char* base = smem + (size_t)q * ST * L * 1024;
  const char* src[PER];                                                // this wave's loads of a slab: wave, wave + 4, ... (the last one again past L)
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int t = min(wave + 4 * u, L - 1);
    if (t < LA) src[u] = reinterpret_cast<const char*>(A + (long)min(m0 + t / HA * 16 + r16, M - 1) * lda + 8 * g + 4 * (t % HA));
    else src[u] = reinterpret_cast<const char*>(W + (long)min(n0 + (t - LA) / HW * 16 + r16, N - 1) * ldw + 8 * g + 4 * ((t - LA) % HW));
  }
  const int slabs = (K + FS - 1) / FS, range = (slabs + FW - 1) / FW;
  const int s0 = min(q * 4 * range, slabs), s1 = min(s0 + 4 * range, slabs), cnt = s1 - s0, steps = min(4 * range, slabs);
  u32x4_t held[PER];
  const auto fetch = [&](int s) {                                      // this wave's pieces of slab s to registers, zeros past K
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int t = min(wave + 4 * u, L - 1);
      const int half = t < LA ? t % HA : (t - LA) % HW, left = K - s * FS - 8 * g - 4 * half;
      held[u] = t < LA ? bytes16(reinterpret_cast<const TA*>(src[u]) + (size_t)s * FS, left) : bytes16(reinterpret_cast<const TW*>(src[u]) + (size_t)s * FS, left);
    }
  };
  const auto put = [&](char* dst) {
#pragma unroll
    for (int u = 0; u < PER; ++u) *reinterpret_cast<u32x4_t*>(dst + min(wave + 4 * u, L - 1) * 1024 + lane * 16) = held[u];
  };
  const auto issue = [&](int i) {                                      // slab s0 + i
    const int s = s0 + i;
    char* dst = base + (size_t)(i % ST) * L * 1024;
    if ((s + 1) * FS <= K) {
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int t = min(wave + 4 * u, L - 1);
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[u] + (size_t)s * FS * (t < LA ? sizeof(TA) : sizeof(TW))),
                                         (__attribute__((address_space(3))) void*)(dst + t * 1024), 16, 0, 0);
      }
    } else {                                                           // the last, shorter slab
      fetch(s);
      put(dst);
    }
  };
  f32x4_t acc[MI][NJ], tot[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = tot[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if constexpr (VEC) {
#pragma unroll
    for (int i = 0; i < ST - 1; ++i)
      if (i < cnt) issue(i);
  } else if (cnt > 0) {
    fetch(s0);
    put(base);
  }
  int in_range = 0;
  for (int i = 0; i < steps; ++i) {
    if (VEC && i + ST - 2 < cnt) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((ST - 2) * PER) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                                      // slab i is there for every wave, and everybody is done with slab i - 1
    if constexpr (VEC) {
      if (i + ST - 1 < cnt) issue(i + ST - 1);
    } else {
      if (i + 1 < cnt) fetch(s0 + i + 1);                              // (in flight under the products)
    }
    if (i < cnt) {
      const char* st = base + (size_t)(i % ST) * L * 1024 + lane * 16;
      Piece<TA> a[MI];
      Piece<TW> w[NJ];
#pragma unroll
      for (int k = 0; k < MI; ++k) {
        const char* p = st + (wm + k) * HA * 1024;
        if constexpr (HA == 2) a[k] = join(*reinterpret_cast<const f32x4_t*>(p), *reinterpret_cast<const f32x4_t*>(p + 1024));
        else a[k] = *reinterpret_cast<const u32x4_t*>(p);
      }
#pragma unroll
      for (int k = 0; k < NJ; ++k) {
        const char* p = st + (LA + (wn + k) * HW) * 1024;
        if constexpr (HW == 2) w[k] = join(*reinterpret_cast<const f32x4_t*>(p), *reinterpret_cast<const f32x4_t*>(p + 1024));
        else w[k] = *reinterpret_cast<const u32x4_t*>(p);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int x = 0; x < MI; ++x)
#pragma unroll
          for (int y = 0; y < NJ; ++y) acc[x][y] = mfma_f32(elem(w[y], e), elem(a[x], e), acc[x][y]);
      if (++in_range == range || i + 1 == cnt) {
        in_range = 0;
#pragma unroll
        for (int x = 0; x < MI; ++x)
#pragma unroll
          for (int y = 0; y < NJ; ++y) {
            tot[x][y] += acc[x][y];
            acc[x][y] = f32x4_t{0.f, 0.f, 0.f, 0.f};
          }
      }
    }
    if (!VEC && i + 1 < cnt) put(base + (size_t)((i + 1) % ST) * L * 1024);
  }
  // the second group's sums through LDS (the stages' place)
  __syncthreads();
  f32x4_t* sum = reinterpret_cast<f32x4_t*>(smem);
  if (q == 1)
#pragma unroll
    for (int x = 0; x < MI; ++x)
#pragma unroll
      for (int y = 0; y < NJ; ++y) sum[((wave * MI + x) * NJ + y) * 64 + lane] = tot[x][y];
  __syncthreads();
  if (q == 1) return;
#pragma unroll
  for (int x = 0; x < MI; ++x) {
    const int m = m0 + (wm + x) * 16 + r16;
    if (m >= M) continue;
#pragma unroll
    for (int y = 0; y < NJ; ++y) {
      const f32x4_t v = tot[x][y] + sum[((wave * MI + x) * NJ + y) * 64 + lane];
      const int n = n0 + (wn + y) * 16 + 4 * g;
      TC* c = C + (long)m * ldc + n;
      if (n + 4 <= N && !accumulate && (((uintptr_t)c) & (4 * sizeof(TC) - 1)) == 0) {
        if constexpr (sizeof(TC) == 4) *reinterpret_cast<f32x4_t*>(c) = v;
        else *reinterpret_cast<uint2*>(c) = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) st_f(c + r, accumulate ? ld_f(c + r) + v[r] : v[r]);
      }
    }
  }
}

template <typename TA, typename TW, typename TC>
int launch_f32(const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc, int batch, long sA, long sW, long sC,
               int accumulate, hipStream_t st) {
  constexpr int VA = 16 / sizeof(TA), VW = 16 / sizeof(TW);
  const bool vec = lda % VA == 0 && ldw % VW == 0 && sA % VA == 0 && sW % VW == 0 && (((uintptr_t)A | (uintptr_t)W) & 15) == 0;
  const auto tiles = [&](int tm, int tn) { return (long)((M + tm - 1) / tm) * ((N + tn - 1) / tn) * batch; };
#define GO(KERNEL, TM, TN, LDS)                                                                                                     \
  do {                                                                                                                              \
    const long mt = (M + (TM) - 1) / (TM), nt = (N + (TN) - 1) / (TN), blocks = (nt * mt + 7) / 8 * 8;                                       \
    if (blocks > 0x7fffffffL) return VLM_ERR_SHAPE;                                                                                 \
    hipLaunchKernelGGL(KERNEL, dim3((unsigned)blocks, 1, batch), dim3(512), LDS, st, (const TA*)A, (const TW*)W, (TC*)C, M, N, K, lda, ldw, ldc, sA, sW, \
                       sC, accumulate, (int)mt, (int)nt);                                                                           \
  } while (0)
#define RANGES(MI, NJ, VEC) GO((linear_f32_ranges_kernel<TA, TW, TC, MI, NJ, VEC>), 16 * MI, 16 * NJ, 0)
#define TILES(MI, NJ, ST, VEC)                                                                                                      \
  do {                                                                                                                              \
    constexpr int stages = VEC ? ST : 2, lds = 2 * stages * (2 * MI * (int)sizeof(TA) / 2 + 2 * NJ * (int)sizeof(TW) / 2) * 1024;   \
    const hipError_t e = hipFuncSetAttribute((const void*)linear_f32_tiles_kernel<TA, TW, TC, MI, NJ, stages, VEC>,                 \
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);                                      \
    if (e != hipSuccess) return VLM_ERR_HIP + (int)e;                                                                               \
    GO((linear_f32_tiles_kernel<TA, TW, TC, MI, NJ, stages, VEC>), 32 * MI, 32 * NJ, lds);                                          \
  } while (0)
  // Where the lines lie (us of one call; the kernel of scalar FMAs that stood here | ranges 16 x 16 | tiles 32 x 64 | 64 x 64 | 64 x 128):
  //   301 rows, W [26304, 1536] fp32            881 | 1272 | 410 | 357 | 351        1 row, the same W              185 |  51 |  48 |  74 |  69
  //   301 rows, W [1536, 21696] fp32           1921 |  627 | 315 | 490 | 863        1 row, the same W             1457 |  53 | 274 | 459 | 823
  //   400 rows, W [41000, 3584] fp32           3987 | 3910 | 1626 | 1488 | 1335     2048 rows, W [1536, 1536]      333 | 510 | 149 | 123 | 142
  //   301 rows, 12 maps [512, 128] fp32          25 |   89 |  17 |  13 |  20        2048 rows, 12 maps [128, 512] bf16  110 | 191 | 43 | 39 | 50
  //   2048 rows, W [64, 1536] bf16               95 |   19 |  23 |  37 |  64  (ranges 32 x 32: 14)
  // a wide tile reads its operands less often, a narrow one leaves fewer compute units without work.
  // Rows that are not whole aligned pieces come through registers (scalar FMAs | ranges 32 x 32, as all of them ran | tiles 32 x 64 | 64 x 64 | 64 x 128):
  //   301 rows, W [1536, 1537] fp32            119 |  40 |  29 |  44 |  75          2048 rows, W [6144, 1539] bf16     757 | 863 | 690 | 398 | 444
  //   301 rows, W [26304, 1537] fp32           849 | 570 | 335 | 311 | 348          2048 rows, 12 maps [512, 129]      109 | 242 |  76 |  65 |  71
  //   1 row, W [1536, 21699] fp32             2027 | 152 | 299 | 457 | 845  (ranges 16 x 16: 50)
#define BY(KIND, ...) do { if (vec) KIND(__VA_ARGS__, true); else KIND(__VA_ARGS__, false); } while (0)
  if (vec && M > 32 && tiles(64, 128) >= 768) TILES(2, 4, 3, true);
  else if (M > 32 && tiles(64, 64) >= 448) BY(TILES, 2, 2, 3);
  else if (tiles(32, 64) >= 160) BY(TILES, 1, 2, 4);
  else if (M > 16 && tiles(32, 32) >= 128) BY(RANGES, 2, 2);
  else BY(RANGES, 1, 1);
#undef BY
#undef TILES
#undef RANGES
#undef GO
  VLM_CHECK_LAUNCH();
  return VLM_OK;
}

// few rows (decode steps): the weights are the traffic, so W is read ONCE for all rows.  One wave per output column, lanes
// across k (coalesced), up to 8 row accumulators per lane, xor-butterfly sum: a fixed order, so a row's result is still a
// function of that row alone.  Sum order differs from the tiles' (rounding only); not used when everything is fp32.
template <typename TA, typename TW, typename TC>
__global__ __launch_bounds__(256) void linear_rows_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C,
                                                          int M, int N, int K, long lda, long ldw, long ldc, long sA, long sW,
                                                          long sC, int accumulate) {
  const int b = blockIdx.z;
  A += (long)b * sA;
  W += (long)b * sW;
  C += (long)b * sC;
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (n >= N) return;                                     // (whole waves leave together: n is uniform per wave)
  const TW* w = W + (long)n * ldw;
  float acc[8] = {};
  for (int k = lane; k < K; k += 64) {
    const float wv = ld_f(w + k);
#pragma unroll
    for (int m = 0; m < 8; ++m)
      if (m < M) acc[m] = fmaf(ld_f(A + (long)m * lda + k), wv, acc[m]);
  }
#pragma unroll
  for (int m = 0; m < 8; ++m) {
    if (m >= M) break;
    float v = acc[m];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if (lane == 0) {
      TC* c = C + (long)m * ldc + n;
      st_f(c, accumulate ? ld_f(c) + v : v);
    }
  }
}

// the same for bf16 weights whose rows are 16-byte aligned with K a multiple of 8: every lane reads 8 weights per load
// (16 bytes, non-temporal: a decode step reads each weight once).  Two ways to skip weights that cannot matter, both exact:
//   * a lane whose 8 activations are zero in EVERY row does not load its 8 weights (the down projection of stacked experts:
//     the experts no row of the step chose are exact zeros in the activations);
//   * skip_gate != nullptr: output columns [skip_col0, skip_col0 + E * ff) belong to E stacked experts of ff columns each;
//     a column whose expert has a zero gate in every row is written as 0 without reading its weights (the up projection).
template <typename TA, typename TC>
__global__ __launch_bounds__(256) void linear_rows_vec_kernel(const TA* __restrict__ A, const bf16_t* __restrict__ W, TC* __restrict__ C,
                                                              int M, int N, int K, long lda, long ldw, long ldc, int accumulate,
                                                              const float* __restrict__ skip_gate, int skip_col0, int E, int ff) {
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (n >= N) return;
  if (skip_gate && n >= skip_col0 && n < skip_col0 + E * ff) {
    const int e = (n - skip_col0) / ff;
    bool any = false;
    for (int m = 0; m < M; ++m) any |= skip_gate[(long)m * E + e] != 0.f;
    if (!any) {                                          // (wave-uniform)
      if (lane < M && !accumulate) st_f(C + (long)lane * ldc + n, 0.f);
      return;
    }
  }
  const bf16_t* w = W + (long)n * ldw;
  float acc[8] = {};
  for (int k = lane * 8; k < K; k += 512) {
    float a[8][8];
    bool nz = false;
#pragma unroll
    for (int m = 0; m < 8; ++m)
      if (m < M) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          a[m][j] = ld_f(A + (long)m * lda + k + j);
          nz |= a[m][j] != 0.f;
        }
      }
    if (!nz) continue;
    const uint4 wv = nt_load16(w + k);
    const float wf[8] = {bf_lo(wv.x), bf_hi(wv.x), bf_lo(wv.y), bf_hi(wv.y), bf_lo(wv.z), bf_hi(wv.z), bf_lo(wv.w), bf_hi(wv.w)};
#pragma unroll
    for (int m = 0; m < 8; ++m)
      if (m < M) {
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[m] = fmaf(a[m][j], wf[j], acc[m]);
      }
  }
#pragma unroll
  for (int m = 0; m < 8; ++m) {
    if (m >= M) break;
    float v = acc[m];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if (lane == 0) {
      TC* c = C + (long)m * ldc + n;
      st_f(c, accumulate ? ld_f(c) + v : v);
    }
  }
}

// The same for bf16 activations: the rows are staged in LDS once per workgroup, so that whether a lane's activations are zero is known without
// a trip to memory and a wave has the loads of NB pieces of R weight rows in flight at once; products on v_dot2_f32_bf16.
template <typename TC, int MB, int R, int NB>
__global__ __launch_bounds__(256) void linear_rows_stream_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, TC* __restrict__ C, int M,
                                                                 int N, int K, long lda, long ldw, long ldc, int accumulate,
                                                                 const float* __restrict__ skip_gate, int skip_col0, int E, int ff) {
  extern __shared__ __align__(16) unsigned as[];         // [MB][K / 2] (rows past M: not read)
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  const int tid = threadIdx.x, lane = tid & 63, K2 = K / 2;
  const int n0 = (blockIdx.x * 4 + (tid >> 6)) * R;
  bool dead[R];                                          // (wave-uniform)
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int n = n0 + r;
    dead[r] = n >= N;
    if (skip_gate && n >= skip_col0 && n < skip_col0 + E * ff) {
      const int e = (n - skip_col0) / ff;
      bool any = false;
      for (int m = 0; m < M; ++m) any |= skip_gate[(long)m * E + e] != 0.f;
      dead[r] |= !any;
    }
  }
#pragma unroll
  for (int m = 0; m < MB; ++m)
    if (m < M)
      for (int i = tid; i < K / 8; i += 256)
        reinterpret_cast<uint4*>(as + m * K2)[i] = *reinterpret_cast<const uint4*>(A + (long)m * lda + 8 * i);
  __syncthreads();
  const bf16_t* w[R];
#pragma unroll
  for (int r = 0; r < R; ++r) w[r] = W + (long)min(n0 + r, N - 1) * ldw;
  bool all = true;
#pragma unroll
  for (int r = 0; r < R; ++r) all &= dead[r];
  float acc[R][MB] = {};
  if (!all) {
    for (int k0 = lane * 8; k0 < K; k0 += 512 * NB) {
      u32x4_t wv[NB][R];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int k = k0 + 512 * b;
        unsigned nz = 0u;
        if (k < K) {
#pragma unroll
          for (int m = 0; m < MB; ++m)
            if (m < M) {
              const uint4 a = *reinterpret_cast<const uint4*>(as + m * K2 + k / 2);
              nz |= (a.x | a.y | a.z | a.w) & 0x7fff7fffu;
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          wv[b][r] = u32x4_t{0u, 0u, 0u, 0u};
          if (nz && !dead[r]) wv[b][r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(w[r] + k));
        }
      }
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int k = min(k0 + 512 * b, K - 8);
#pragma unroll
        for (int m = 0; m < MB; ++m)
          if (m < M) {
            const u32x4_t a = *reinterpret_cast<const u32x4_t*>(as + m * K2 + k / 2);
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const unsigned x = a[i], y = wv[b][r][i];          // (scalars first: a bit cast of a vector element reads element 0)
                acc[r][m] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2, x), __builtin_bit_cast(bf2, y), acc[r][m], false);
              }
          }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (n0 + r >= N) break;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      if (m >= M) break;
      const float v = wave_sum(acc[r][m]);
      if (lane == 0) {
        TC* c = C + (long)m * ldc + n0 + r;
        st_f(c, accumulate ? ld_f(c) + v : v);
      }
    }
  }
}

template <typename TC>
int launch_stream(const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc, int accumulate, const void* skip_gate,
                  int skip_col0, int E, int ff, hipStream_t st) {
  const int MB = M <= 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : 8;
  const size_t lds = (size_t)MB * K * sizeof(bf16_t);
  const int R = N <= 4096 ? 1 : 2;
  const dim3 grid((N + 4 * R - 1) / (4 * R));
#define GO(MBV, RV, NBV)                                                                                                            \
  do {                                                                                                                              \
    if (lds > 48 * 1024) {                                                                                                          \
      hipError_t e = hipFuncSetAttribute((const void*)linear_rows_stream_kernel<TC, MBV, RV, NBV>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
      if (e != hipSuccess) return VLM_ERR_HIP + (int)e;                                                                             \
    }                                                                                                                               \
    hipLaunchKernelGGL((linear_rows_stream_kernel<TC, MBV, RV, NBV>), grid, dim3(256), lds, st, (const bf16_t*)A, (const bf16_t*)W, (TC*)C, M, N, K, \
                       lda, ldw, ldc, accumulate, (const float*)skip_gate, skip_col0, E, ff);                                       \
  } while (0)
#define GO2(MBV, NBV) do { if (R == 1) GO(MBV, 1, NBV); else GO(MBV, 2, NBV); } while (0)
  if (MB == 1) GO2(1, 4); else if (MB == 2) GO2(2, 4); else if (MB == 4) GO2(4, 4); else GO2(8, 4);
#undef GO2
#undef GO
  VLM_CHECK_LAUNCH();
  return VLM_OK;
}

// bf16 operands of more than 8 rows whose rows come in whole 16-byte pieces, on v_mfma_f32_16x16x32_bf16 with fp32 sums: per-head maps as
// batch and products with fp32 results (the GEMMs of gemm_bf16.hip write bf16).  A wave owns 32 rows of A x 64 rows of W, a workgroup
// 64 x 128; operands come straight from global memory in the operand layout (the W rows of a tile are shared through the caches), the W rows
// dealt out so that a lane ends with 16 neighbouring outputs of one row.
template <typename TC>
__global__ __launch_bounds__(256) void linear_any_mfma_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, TC* __restrict__ C, int M,
                                                              int N, int K, long lda, long ldw, long ldc, long sA, long sW, long sC,
                                                              int accumulate) {
  typedef __attribute__((ext_vector_type(8))) __bf16 bf8;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  const int m0 = blockIdx.y * 64 + (wave & 1) * 32, n0 = blockIdx.x * 128 + (wave >> 1) * 64;
  if (m0 >= M || n0 >= N) return;
  A += (long)blockIdx.z * sA;
  W += (long)blockIdx.z * sW;
  C += (long)blockIdx.z * sC;
  const bf16_t *ar[2], *wr[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) ar[i] = A + (long)min(m0 + 16 * i + r16, M - 1) * lda + 8 * g;
#pragma unroll
  for (int j = 0; j < 4; ++j) wr[j] = W + (long)min(n0 + (r16 >> 2) * 16 + 4 * j + (r16 & 3), N - 1) * ldw + 8 * g;   // (operand row 4 g + r of product j)
  f32x4_t acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int K32 = K & ~31;
#pragma unroll 4
  for (int k = 0; k < K32; k += 32) {
    bf8 a[2], w[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) a[i] = *reinterpret_cast<const bf8*>(ar[i] + k);
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = *reinterpret_cast<const bf8*>(wr[j] + k);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], a[i], acc[i][j], 0, 0, 0);
  }
  if (K32 < K) {
    const u32x4_t none = {0u, 0u, 0u, 0u};
    bf8 a[2], w[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) a[i] = __builtin_bit_cast(bf8, none);
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = __builtin_bit_cast(bf8, none);
    if (K32 + 8 * g < K) {
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = *reinterpret_cast<const bf8*>(ar[i] + K32);
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = *reinterpret_cast<const bf8*>(wr[j] + K32);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], a[i], acc[i][j], 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m0 + 16 * i + r16;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + 16 * g + 4 * j;                 // (a lane's four products: 16 neighbouring columns)
      TC* c = C + (long)m * ldc + n;
      if (n + 4 <= N && !accumulate && (((uintptr_t)c) & (4 * sizeof(TC) - 1)) == 0) {
        if constexpr (sizeof(TC) == 4) *reinterpret_cast<float4*>(c) = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
        else *reinterpret_cast<uint2*>(c) = make_uint2(pack_bf2(acc[i][j][0], acc[i][j][1]), pack_bf2(acc[i][j][2], acc[i][j][3]));
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) st_f(c + r, accumulate ? ld_f(c + r) + acc[i][j][r] : acc[i][j][r]);
      }
    }
  }
}

template <typename TA, typename TW, typename TC>
int launch(const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc, int batch, long sA, long sW,
           long sC, int accumulate, hipStream_t st) {
  // all-fp32 operands (the float32 serving mode) always take launch_f32: one summation order for every row count, so a
  // token's result is the same bits in a prompt, in a portion and decoded alone
  constexpr bool all_f32 = sizeof(TA) == 4 && sizeof(TW) == 4 && sizeof(TC) == 4;
  if constexpr (sizeof(TW) == 2) {
    // a few rows (inside a graph, us): 12 maps [512, 128] to fp32, 8 rows 7.8 -> 3.9; 12 maps [128, 512] of fp32 rows, 2 / 3 / 16 rows 5.6 / 6.4 / 6.3 ->
    // 4.2 / 4.3 / 5.2, one row 4.3 -> 4.8; [8, 1536] to fp32, 9 / 32 rows 12.3 / 15.6 -> 3.9 / 5.1.  Up to 8 fp32 rows with fp32 results stay on the
    // kernel below, whose sums are a little closer (relative error 7.5e-8 and 8.8e-8 at K = 200).
    if (M >= 2 && !(sizeof(TA) == 4 && sizeof(TC) == 4 && M <= 8)) {
      const int rc = vlm_linear_rows_mfma_try(A, W, C, M, N, K, lda, ldw, ldc, sizeof(TA) == 4, sizeof(TC) == 4, batch, sA, sW, sC, accumulate, st);
      if (rc >= 0) return rc;
    }
  }
  if constexpr (sizeof(TA) == 2 && sizeof(TW) == 2) {
    if (M > 8 && K % 8 == 0 && lda % 8 == 0 && ldw % 8 == 0 && sA % 8 == 0 && sW % 8 == 0 && (((uintptr_t)A | (uintptr_t)W) & 15) == 0) {
      dim3 grid((N + 127) / 128, (M + 63) / 64, batch);
      hipLaunchKernelGGL((linear_any_mfma_kernel<TC>), grid, dim3(256), 0, st, (const bf16_t*)A, (const bf16_t*)W, (TC*)C, M, N, K, lda, ldw, ldc,
                         sA, sW, sC, accumulate);
      VLM_CHECK_LAUNCH();
      return VLM_OK;
    }
  }
  if (M <= 8 && !all_f32) {
    dim3 grid((N + 3) / 4, 1, batch);
    hipLaunchKernelGGL((linear_rows_kernel<TA, TW, TC>), grid, dim3(256), 0, st, (const TA*)A, (const TW*)W, (TC*)C, M, N, K, lda,
                       ldw, ldc, sA, sW, sC, accumulate);
    VLM_CHECK_LAUNCH();
    return VLM_OK;
  }
  return launch_f32<TA, TW, TC>(A, W, C, M, N, K, lda, ldw, ldc, batch, sA, sW, sC, accumulate, st);
}

}  // namespace

// decode-step form with the expert-column skip (see linear_rows_vec_kernel); M <= 8, bf16 weights, K % 8 == 0
extern "C" int vlm_linear_rows_bf16w(const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc, int a_f32,
                                     int c_f32, int accumulate, const void* skip_gate, int skip_col0, int E, int ff, void* stream) {
  if (!A || !W || !C || M <= 0 || M > 8 || N <= 0 || K <= 0 || lda < K || ldw < K || ldc < N) return VLM_ERR_ARG;
  if (accumulate && !c_f32) return VLM_ERR_ARG;
  if (skip_gate && (E <= 0 || ff <= 0 || skip_col0 < 0 || skip_col0 + (long)E * ff > N)) return VLM_ERR_ARG;
  if (K % 8 || ldw % 8 || ((uintptr_t)W & 15)) return VLM_ERR_SHAPE;
  hipStream_t st = (hipStream_t)stream;
  const int MB = M <= 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : 8;
  if (!a_f32 && lda % 8 == 0 && ((uintptr_t)A & 15) == 0 && (size_t)MB * K * sizeof(bf16_t) <= 80 * 1024)
    return c_f32 ? launch_stream<float>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, skip_gate, skip_col0, E, ff, st)
                 : launch_stream<bf16_t>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, skip_gate, skip_col0, E, ff, st);
  dim3 grid((N + 3) / 4);
#define GO(TA, TC)                                                                                                              \
  hipLaunchKernelGGL((linear_rows_vec_kernel<TA, TC>), grid, dim3(256), 0, st, (const TA*)A, (const bf16_t*)W, (TC*)C, M, N, K, lda, \
                     ldw, ldc, accumulate, (const float*)skip_gate, skip_col0, E, ff)
  if (a_f32) {
    if (c_f32) GO(float, float); else GO(float, bf16_t);
  } else {
    if (c_f32) GO(bf16_t, float); else GO(bf16_t, bf16_t);
  }
#undef GO
  VLM_CHECK_LAUNCH();
  return VLM_OK;
}

extern "C" int vlm_linear_any(const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc, int a_f32,
                              int w_f32, int c_f32, int batch, long strideA, long strideW, long strideC, int accumulate,
                              void* stream) {
  if (!A || !W || !C || M < 0 || N <= 0 || K <= 0 || batch <= 0 || lda < K || ldw < K || ldc < N) return VLM_ERR_ARG;
  if (accumulate && !c_f32) return VLM_ERR_ARG;
  if (M == 0) return VLM_OK;
  if (M > 65535 * 64 || batch > 65535) return VLM_ERR_SHAPE;
  hipStream_t st = (hipStream_t)stream;
  const int code = (a_f32 ? 4 : 0) | (w_f32 ? 2 : 0) | (c_f32 ? 1 : 0);
#define GO(TA, TW, TC) return launch<TA, TW, TC>(A, W, C, M, N, K, lda, ldw, ldc, batch, strideA, strideW, strideC, accumulate, st)
  switch (code) {
    case 0: GO(bf16_t, bf16_t, bf16_t);
    case 1: GO(bf16_t, bf16_t, float);
    case 2: GO(bf16_t, float, bf16_t);
    case 3: GO(bf16_t, float, float);
    case 4: GO(float, bf16_t, bf16_t);
    case 5: GO(float, bf16_t, float);
    case 6: GO(float, float, bf16_t);
    default: GO(float, float, float);
  }
#undef GO
}
