// Latent attention (see latent_attn.hip: absorbed form, ONE cached row [c (R) | kr (Dr)] per token, scores over R + Dr, values = c) on the
// bf16 matrix cores, for bf16 or fp32 queries and bf16 pools whose rows come in whole 16-byte pieces (R % 8 == 0, Dr % 8 == 0; R <= 512,
// R + Dr <= 576).
//
//     s_hj = scale * (q_h . row_j)        o_h = sum_j exp(s_hj) c_j / (exp(sink_h) + sum_j exp(s_hj)) (* sigmoid(gate_h))
//     j visible from i  <=>  0 <= i - j < window  (window <= 0: every j <= i); no sink: without the first term of the denominator
//
// Scores are fp32 sums, the softmax runs in fp32, and its weights enter the product with the values as two bf16 values each ((p_hi + p_lo) c),
// so nothing of a score or a weight is rounded to 8 bits.  fp32 queries (and read-outs) enter as three bf16 values each, and so do the weights:
// three times 8 bits are the 24 of an fp32 number, a cached bf16 value is one, so every product is exact and the sums are the fp32 sums
// of the former scalar kernel in another order.  Layout of the transposed products: attn_mfma.hpp.
//
//   blocks (prompt)  workgroup = up to 16 consecutive tokens of one sequence x 4 heads, one head per wave.  A wave keeps its 16 query
//                    columns in registers (operand layout) and the whole read-out of R columns; the key tile - one page of 64 rows,
//                    which all heads share - goes through LDS in two buffers, the next page's loads in flight while this one is
//                    used, one barrier per tile.  The same LDS rows serve as keys (16 bytes of one row per lane) and as values
//                    (8 columns of 8 keys per lane, interleaved in registers).  No exchange between the waves.
//                    fp32 queries, R = 512, Dr = 64, 12 heads, 2048 causal keys: 2923 -> 323 us (scalar kernel of latent_attn.hip -> here, bf16
//                    queries 150 us); 28 heads, 1500 tokens, window 1024: 2574 -> 339 us; 40 tokens: 30 -> 22 us.  Bound by the matrix
//                    products and the two reads of a page from LDS per head, one wave per SIMD (the queries' parts alone are 216 registers).
//   rows (decode)    workgroup = one token x up to 16 heads, one page at a time through LDS: the waves share the page's keys for the scores,
//                    exchange them, and share the value columns for the read-out; `nsplit` workgroups take turns over the pages, a second
//                    kernel merges their results.  fp32 queries: 8 rows of 12 heads over 700 keys 45 -> 20 us, one row over 16384 keys
//                    1476 -> 41 us.  Over 20 keys the scalar kernel is ahead (7.3 | 16.1 us, R = 128 5.2 | 9.3; 512 keys 34 | 16 and 14 | 9.6):
//                    contexts that are known to stay short keep it (ROW_KEYS of ops.py).
#include "common.hpp"
#include "../../include/vlm_hip.h"
#include "recurrence_finish.hpp"
#include "attn_mfma.hpp"

namespace {

constexpr int PAGE = 64, QC = 16;
constexpr float LOG2E = 1.4426950408889634f;

// a key tile in LDS: rows of 32 NKS columns (zeros behind R + Dr) at an odd number of 16-byte pieces, so that the same piece of 16 neighbouring
// rows sits in different banks; one more piece behind the tile takes the stores of lanes without a piece
template <int NKS> struct Tile {
  static constexpr int PITCH = 8 * ((4 * NKS) | 1), SIZE = PAGE * PITCH + 8;
};

// bf16 values per query number and per softmax weight
template <typename TQ> constexpr int NQ = sizeof(TQ) == 4 ? 3 : 1;
template <typename TQ> constexpr int NP = sizeof(TQ) == 4 ? 3 : 2;

// 8 fp32 values as N bf16 operands, the leading one first
template <int N> __device__ __forceinline__ void split_parts(const float* f, bf8* o) {
  float r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = f[i];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    u32x4_t w;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned p = pack_bf2(r[2 * i], r[2 * i + 1]);
      w[i] = p;
      r[2 * i] -= bf_lo(p);
      r[2 * i + 1] -= bf_hi(p);
    }
    o[n] = __builtin_bit_cast(bf8, w);
  }
}

// 16 query columns as operands: lane (r16, g) holds dimensions 32 s + 8 g .. + 8 of column r16
template <int NKS> __device__ __forceinline__ void load_queries(const bf16_t* qrow, bool live, int Dk, int g, bf8 (*q)[1]) {
#pragma unroll
  for (int s = 0; s < NKS; ++s) {
    const int d = 32 * s + 8 * g;
    q[s][0] = zero8();
    if (live && d < Dk) q[s][0] = *reinterpret_cast<const bf8*>(qrow + d);
  }
}
// (fp32: cut, not rounded, so that the largest numbers stay finite; an infinity is its leading part alone)
template <int NKS> __device__ __forceinline__ void load_queries(const float* qrow, bool live, int Dk, int g, bf8 (*q)[3]) {
#pragma unroll
  for (int s = 0; s < NKS; ++s) {
    const int d = 32 * s + 8 * g;
    float f[8] = {};
    if (live && d < Dk) {
      const float4 a = *reinterpret_cast<const float4*>(qrow + d), b = *reinterpret_cast<const float4*>(qrow + d + 4);
      f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
    }
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      u32x4_t w;
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = __builtin_amdgcn_perm(__float_as_uint(f[2 * i + 1]), __float_as_uint(f[2 * i]), 0x07060302u);
      q[s][n] = __builtin_bit_cast(bf8, w);
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = fabsf(f[i]) < INFINITY ? f[i] - __uint_as_float(__float_as_uint(f[i]) & 0xffff0000u) : 0.f;
    }
  }
}

// copies of a page's rows into a tile by 256 threads: this thread's pieces are tid, tid + 256, ... (a page's rows are contiguous in memory);
// rows past the last key repeat its last piece (they are masked); the first `skip` rows of a page, which no query sees, are zeros: a zero weight
// would hand on what is not finite there
template <int NKS> struct Stager {
  static constexpr int PARTS = NKS % 3 == 0 ? 3 : 2, HALF = NKS / PARTS;          // a page goes through the registers in parts
  int loff[NKS], pieces, D8;
  u32x4_t st[HALF];
  __device__ __forceinline__ void init(bf16_t* tiles, int ntiles, int Dk, int tid) {
    D8 = Dk / 8;
    pieces = PAGE * D8;
#pragma unroll
    for (int i = 0; i < NKS; ++i) {
      const int idx = tid + 256 * i;
      loff[i] = idx < pieces ? (idx / D8) * Tile<NKS>::PITCH + (idx % D8) * 8 : PAGE * Tile<NKS>::PITCH;
    }
    const int pad = 4 * NKS - D8;                        // pieces of zeros behind every row
    for (int i = tid; i < ntiles * PAGE * pad; i += 256) {
      const int row = (i / pad) % PAGE;
      *reinterpret_cast<u32x4_t*>(tiles + (i / (pad * PAGE)) * Tile<NKS>::SIZE + row * Tile<NKS>::PITCH + (D8 + i % pad) * 8) = u32x4_t{0u, 0u, 0u, 0u};
    }
  }
  template <int H> __device__ __forceinline__ void load(const bf16_t* page, int keys, int tid, int skip = 0) {
    const u32x4_t* src = reinterpret_cast<const u32x4_t*>(page);
    const int have = min(pieces, keys * D8) - 1;
#pragma unroll
    for (int i = 0; i < HALF; ++i) st[i] = src[min(tid + 256 * (H * HALF + i), have)];
    if (skip > 0)
#pragma unroll
      for (int i = 0; i < HALF; ++i)
        if (tid + 256 * (H * HALF + i) < skip * D8) st[i] = u32x4_t{0u, 0u, 0u, 0u};
  }
  template <int H> __device__ __forceinline__ void store(bf16_t* tile) {
#pragma unroll
    for (int i = 0; i < HALF; ++i) *reinterpret_cast<u32x4_t*>(tile + loff[H * HALF + i]) = st[i];
  }
};

// softmax update of one query column over N scores per lane (scores in log2 units); returns the factor of what was summed before
template <int N>
__device__ __forceinline__ float softmax_update(float* pr, float& mrun, float& lrun) {
  float mx = pr[0];
#pragma unroll
  for (int i = 1; i < N; ++i) mx = fmaxf(mx, pr[i]);
  mx = col4_max(mx);
  const float m_new = fmaxf(mrun, mx), ms = m_new == -INFINITY ? 0.f : m_new;
  const float al = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(mrun - ms);
  mrun = m_new;
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    pr[i] = __builtin_amdgcn_exp2f(pr[i] - ms);
    sum += pr[i];
  }
  lrun = fmaf(lrun, al, sum);
  return al;
}

// O^T += V^T P^T for 32 keys and 128 value columns: rows of this lane's 8 keys, 8 columns each (16 bytes); the weights' last part first
template <int N>
__device__ __forceinline__ void accumulate128(const u32x4_t* v, const bf8* pw, f32x4_t* acc) {
  bf8 vt[8];
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    u32x4_t t;
#pragma unroll
    for (int i = 0; i < 4; ++i) t[i] = pair_cols(v[2 * i][b / 2], v[2 * i + 1][b / 2], b & 1);
    vt[b] = __builtin_bit_cast(bf8, t);
    acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vt[b], pw[N - 1], acc[b], 0, 0, 0);
  }
#pragma unroll
  for (int n = N - 2; n >= 0; --n)
#pragma unroll
    for (int b = 0; b < 8; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vt[b], pw[n], acc[b], 0, 0, 0);
  // the interleaving of the next column runs beside a product
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);     // VALU
    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);     // MFMA
  }
  __builtin_amdgcn_sched_group_barrier(0x8, 8 * (N - 1), 0);
}
// eight neighbouring columns of a read-out
__device__ __forceinline__ void store8(bf16_t* o, const f32x4_t* acc, int r, float f) {
  *reinterpret_cast<uint4*>(o) = make_uint4(pack_bf2(acc[0][r] * f, acc[1][r] * f), pack_bf2(acc[2][r] * f, acc[3][r] * f),
                                            pack_bf2(acc[4][r] * f, acc[5][r] * f), pack_bf2(acc[6][r] * f, acc[7][r] * f));
}
__device__ __forceinline__ void store8(float* o, const f32x4_t* acc, int r, float f) {
  *reinterpret_cast<float4*>(o) = make_float4(acc[0][r] * f, acc[1][r] * f, acc[2][r] * f, acc[3][r] * f);
  *reinterpret_cast<float4*>(o + 4) = make_float4(acc[4][r] * f, acc[5][r] * f, acc[6][r] * f, acc[7][r] * f);
}
// this lane's pieces of 8 keys (the contraction order of 32 keys from row `key0` on) at the columns from `cols` on
__device__ __forceinline__ void load_values(const bf16_t* tile, int pitch, int key0, int cols, int r16, int g, u32x4_t* v) {
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const u32x4_t*>(tile + (key0 + 16 * (i / 4) + 4 * g + i % 4) * pitch + cols + r16 * 8);
}

__device__ __forceinline__ float head_gate(const vlm_latent_mfma_args& p, long tok, int h) {
  return p.gate ? 1.f / (1.f + expf(-bf2f(((const bf16_t*)p.gate)[tok * p.ldgate + h]))) : 1.f;
}

// NKS: 32-dimension steps of the scores, NVC: 128-column chunks of the values
template <typename TQ, int NKS, int NVC>
__global__ __launch_bounds__(256, 1) void latent_block_mfma_kernel(vlm_latent_mfma_args p) {
  constexpr int KP = Tile<NKS>::PITCH, TS = Tile<NKS>::SIZE;
  extern __shared__ __align__(16) bf16_t tile[];         // [2][TS]
  const int R = p.R, Dk = p.R + p.Dr;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
  const int blk = gridDim.y - 1 - blockIdx.y;            // (the blocks of a prompt's end have the most keys: they start first)
  const int t0 = p.qb_start[blk], nq = p.qb_count[blk], h = blockIdx.x * 4 + wave;
  const bool live = h < p.H;                             // (a wave without a head still helps with the loads)
  const int* bt = p.block_table + (long)p.tok_seq[t0] * p.max_pages;
  const int pos0 = p.tok_pos[t0], last = pos0 + nq - 1, mypos = r16 < nq ? pos0 + r16 : -1, window = p.window;
  const float sc = p.scale * LOG2E;
  const bf16_t* pool = (const bf16_t*)p.pool;
  const int oldest = window > 0 ? max(0, pos0 - window + 1) : 0, first = oldest / PAGE, tiles = last / PAGE + 1;
  Stager<NKS> sg;
  sg.init(tile, 2, Dk, tid);
  sg.template load<0>(pool + (long)bt[first] * PAGE * Dk, last - first * PAGE + 1, tid, oldest % PAGE);
  bf8 q[NKS][NQ<TQ>];
  load_queries<NKS>((const TQ*)p.q + ((long)(t0 + r16) * p.H + h) * Dk, live && r16 < nq, Dk, g, q);
  f32x4_t acc[NVC][8];
#pragma unroll
  for (int c = 0; c < NVC; ++c)
#pragma unroll
    for (int b = 0; b < 8; ++b) acc[c][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float mrun = -INFINITY, lrun = 0.f;
  sg.template store<0>(tile);
  sg.template load<1>(pool + (long)bt[first] * PAGE * Dk, last - first * PAGE + 1, tid, oldest % PAGE);
  sg.template store<1>(tile);
  if constexpr (Stager<NKS>::PARTS > 2) {
    sg.template load<2>(pool + (long)bt[first] * PAGE * Dk, last - first * PAGE + 1, tid, oldest % PAGE);
    sg.template store<2>(tile);
  }
  for (int j = first; j < tiles; ++j) {
    const bf16_t* cur = tile + ((j - first) & 1) * TS;
    bf16_t* nxt = tile + ((j + 1 - first) & 1) * TS;
    const bool more = j + 1 < tiles;
    const bf16_t* npage = pool + (long)bt[more ? j + 1 : j] * PAGE * Dk;
    const int nkeys = last - (j + 1) * PAGE + 1;
    __syncthreads();                                     // the tile is written, and everybody is through with the other buffer
    if (more) sg.template load<0>(npage, nkeys, tid);
    // scores: KB k steps of the four 16-key groups per batch (a key is used NQ times), the next batch's reads ahead of this one's products
    constexpr int KB = NQ<TQ> == 1 ? 2 : 1;
    f32x4_t s[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) s[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    bf8 ka[2][4 * KB];
    auto keys = [&](int b, bf8* k) {
#pragma unroll
      for (int i = 0; i < 4 * KB; ++i) k[i] = *reinterpret_cast<const bf8*>(cur + (16 * (i & 3) + r16) * KP + 32 * (KB * b + i / 4) + 8 * g);
    };
    keys(0, ka[0]);
#pragma unroll
    for (int b = 0; b < NKS / KB; ++b) {
      if (b + 1 < NKS / KB) keys(b + 1, ka[(b + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = NQ<TQ> - 1; n >= 0; --n)
#pragma unroll
        for (int i = 0; i < 4 * KB; ++i) s[i & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[b & 1][i], q[KB * b + i / 4][n], s[i & 3], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    u32x4_t v[2][8];
    load_values(cur, KP, 0, 0, r16, g, v[0]);            // (in flight during the softmax)
    __builtin_amdgcn_sched_barrier(0);
    const int lo = j * PAGE;
    float pr[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) pr[i] = s[i / 4][i % 4] * sc;
    if (!(lo + PAGE - 1 <= pos0 && (window <= 0 || last - lo < window))) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int dist = mypos - (lo + 16 * (i / 4) + 4 * g + i % 4);
        if (!(dist >= 0 && (window <= 0 || dist < window))) pr[i] = -INFINITY;
      }
    }
    const float al = softmax_update<16>(pr, mrun, lrun);
    if (__any(al != 1.f)) {
#pragma unroll
      for (int c = 0; c < NVC; ++c)
#pragma unroll
        for (int b = 0; b < 8; ++b) acc[c][b] *= al;
    }
    if (more) {
      sg.template store<0>(nxt);
      sg.template load<1>(npage, nkeys, tid);
    }
    bf8 pw[2][NP<TQ>];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) split_parts<NP<TQ>>(pr + 8 * kk, pw[kk]);
#pragma unroll
    for (int i = 0; i < 2 * NVC; ++i) {                  // 32 keys x 128 columns at a time, the next piece's reads ahead
      if (i + 1 < 2 * NVC) load_values(cur, KP, 32 * ((i + 1) / NVC), 128 * ((i + 1) % NVC), r16, g, v[(i + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      accumulate128<NP<TQ>>(v[i & 1], pw[i / NVC], acc[i % NVC]);
      __builtin_amdgcn_sched_barrier(0);
      if (Stager<NKS>::PARTS > 2 && i == NVC - 1 && more) {
        sg.template store<1>(nxt);
        sg.template load<Stager<NKS>::PARTS - 1>(npage, nkeys, tid);
      }
    }
    if (more) sg.template store<Stager<NKS>::PARTS - 1>(nxt);
  }
  float l = col4_sum(lrun);
  const float ms = mrun == -INFINITY ? 0.f : mrun;
  if (!live || r16 >= nq) return;
  if (p.sink) l += __builtin_amdgcn_exp2f(p.sink[h] * LOG2E - ms);
  const float f = (l > 0.f ? 1.f / l : 0.f) * head_gate(p, t0 + r16, h);
  TQ* out = (TQ*)p.out + ((long)(t0 + r16) * p.H + h) * R;
#pragma unroll
  for (int c = 0; c < NVC; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int col = 128 * c + (4 * g + r) * 8;
      if (col < R) store8(out + col, acc[c], r, f);
    }
}

template <typename TQ, int NKS, int NVC>
__global__ __launch_bounds__(256) void latent_rows_mfma_kernel(vlm_latent_mfma_args p) {
  constexpr int KP = Tile<NKS>::PITCH, TS = Tile<NKS>::SIZE, SP = QC + 1;
  extern __shared__ __align__(16) bf16_t tile[];         // [TS], then scores fp32 [64 keys][SP]
  float* sl = reinterpret_cast<float*>(tile + TS);
  const int R = p.R, Dk = p.R + p.Dr;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
  const int t = blockIdx.x, h0 = blockIdx.y * QC, ncol = min(QC, p.H - h0), z = blockIdx.z;
  const int* bt = p.block_table + (long)p.tok_seq[t] * p.max_pages;
  const int pos = p.tok_pos[t], window = p.window;
  const int oldest = window > 0 ? max(0, pos - window + 1) : 0, first = oldest / PAGE, tiles = pos / PAGE + 1;
  const bool split = gridDim.z > 1;
  const float sc = p.scale * LOG2E;
  float* part = p.part + (((long)z * p.H + h0 + r16) * gridDim.x + t) * (R + 2);        // of this lane's column
  if (first + z >= tiles) {                              // no keys for this workgroup: only the marks of an empty part (uniform)
    if (tid < ncol) {
      part[R] = -INFINITY;
      part[R + 1] = 0.f;
    }
    return;
  }
  const bf16_t* pool = (const bf16_t*)p.pool;
  Stager<NKS> sg;
  sg.init(tile, 1, Dk, tid);
  bf8 q[NKS][NQ<TQ>];
  load_queries<NKS>((const TQ*)p.q + ((long)t * p.H + h0 + r16) * Dk, r16 < ncol, Dk, g, q);
  f32x4_t acc[8];
#pragma unroll
  for (int b = 0; b < 8; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float mrun = -INFINITY, lrun = 0.f;
  for (int j = first + z; j < tiles; j += gridDim.z) {
    const bf16_t* page = pool + (long)bt[j] * PAGE * Dk;
    u32x4_t st[NKS];                                     // (the whole page in flight at once)
    const u32x4_t* src = reinterpret_cast<const u32x4_t*>(page);
    const int skip = (oldest - j * PAGE) * sg.D8, have = min(sg.pieces, (pos - j * PAGE + 1) * sg.D8) - 1;
#pragma unroll
    for (int i = 0; i < NKS; ++i) st[i] = src[min(tid + 256 * i, have)];
    if (skip > 0)
#pragma unroll
      for (int i = 0; i < NKS; ++i)
        if (tid + 256 * i < skip) st[i] = u32x4_t{0u, 0u, 0u, 0u};
    __syncthreads();                                     // (everybody is through with the previous page and its scores)
#pragma unroll
    for (int i = 0; i < NKS; ++i) *reinterpret_cast<u32x4_t*>(tile + sg.loff[i]) = st[i];
    __syncthreads();
    f32x4_t s = {0.f, 0.f, 0.f, 0.f}, s1 = s, s2 = s;    // keys 16 wave + 4 g + r of the page: leading parts in two chains, the rest in a third
#pragma unroll
    for (int k = 0; k < NKS; ++k) {
      const bf8 key = *reinterpret_cast<const bf8*>(tile + (16 * wave + r16) * KP + 32 * k + 8 * g);
#pragma unroll
      for (int n = NQ<TQ> - 1; n > 0; --n) s2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(key, q[k][n], s2, 0, 0, 0);
      f32x4_t& lead = NQ<TQ> > 1 && k & 1 ? s1 : s;
      lead = __builtin_amdgcn_mfma_f32_16x16x32_bf16(key, q[k][0], lead, 0, 0, 0);
    }
    if constexpr (NQ<TQ> > 1) s = (s + s1) + s2;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = 16 * wave + 4 * g + r, dist = pos - (j * PAGE + key);
      sl[key * SP + r16] = dist >= 0 && (window <= 0 || dist < window) ? s[r] * sc : -INFINITY;
    }
    __syncthreads();
    float pr[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) pr[i] = sl[(16 * (i / 4) + 4 * g + i % 4) * SP + r16];
    const float al = softmax_update<16>(pr, mrun, lrun); // (the same in every wave)
    if (wave < NVC) {
#pragma unroll
      for (int b = 0; b < 8; ++b) acc[b] *= al;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        bf8 pw[NP<TQ>];
        split_parts<NP<TQ>>(pr + 8 * kk, pw);
        u32x4_t v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const u32x4_t*>(tile + (32 * kk + 16 * (i / 4) + 4 * g + i % 4) * KP + 128 * wave + r16 * 8);
        accumulate128<NP<TQ>>(v, pw, acc);
      }
    }
  }
  float l = col4_sum(lrun);
  if (r16 >= ncol) return;
  const int h = h0 + r16;
  const float ms = mrun == -INFINITY ? 0.f : mrun;
  if (split) {
    if (wave == 0 && g == 0) {
      part[R] = mrun;
      part[R + 1] = l;
    }
  } else if (p.sink) {
    l += __builtin_amdgcn_exp2f(p.sink[h] * LOG2E - ms);
  }
  if (wave >= NVC) return;
  const float f = split ? 1.f : (l > 0.f ? 1.f / l : 0.f) * head_gate(p, t, h);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int col = 128 * wave + (4 * g + r) * 8;
    if (col >= R) continue;
    if (split) {                                         // (R is even and a part's rows are R + 2 long: 8-byte aligned)
#pragma unroll
      for (int b = 0; b < 8; b += 2) *reinterpret_cast<float2*>(part + col + b) = make_float2(acc[b][r], acc[b + 1][r]);
    } else {
      store8((TQ*)p.out + ((long)t * p.H + h) * R + col, acc, r, f);
    }
  }
}

// merge of the splits' partial results: grid (rows, H, chunks of 256 columns).  part: [split][H][rows][R sums | maximum | sum]; the splits
// that had keys come first
template <typename TQ>
__global__ __launch_bounds__(256) void latent_merge_kernel(vlm_latent_mfma_args p, int nsplit) {
  const long t = blockIdx.x;
  const int h = blockIdx.y, lane = threadIdx.x & 63, R = p.R;
  const long step = (long)p.H * gridDim.x * (R + 2);
  const float* q = p.part + ((long)h * gridDim.x + t) * (R + 2);
  const float M_mine = lane < nsplit ? q[lane * step + R] : -INFINITY, l_mine = lane < nsplit ? q[lane * step + R + 1] : 0.f;
  const float M = wave_max(M_mine), ms = M == -INFINITY ? 0.f : M;
  const float f_mine = __builtin_amdgcn_exp2f(M_mine - ms);
  float l = wave_sum(l_mine * f_mine);
  if (p.sink) l += __builtin_amdgcn_exp2f(p.sink[h] * LOG2E - ms);
  const float inv = (l > 0.f ? 1.f / l : 0.f) * head_gate(p, t, h);
  const int n = __popcll(__ballot(M_mine != -INFINITY));
  const int c = min(blockIdx.z * 256 + (int)threadIdx.x, R - 1);          // (whole waves: the shuffles below need every lane)
  float a = 0.f;
  for (int z0 = 0; z0 < n; z0 += 8) {                    // eight loads in flight; splits past the last one count for nothing
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = q[min(z0 + i, n - 1) * step + c];
#pragma unroll
    for (int i = 0; i < 8; ++i) a = fmaf(__shfl(f_mine, min(z0 + i, 63)) * (z0 + i < n ? 1.f : 0.f), v[i], a);
  }
  if (blockIdx.z * 256 + (int)threadIdx.x < R) {
    TQ* o = (TQ*)p.out + (t * p.H + h) * R + c;
    if constexpr (sizeof(TQ) == 4) *o = a * inv;
    else *o = f2bf(a * inv);
  }
}

bool bad(const vlm_latent_mfma_args* a) {
  return !a || !a->q || !a->pool || !a->tok_seq || !a->tok_pos || !a->block_table || !a->out || a->max_pages <= 0 || a->H <= 0 || a->R <= 0 || a->Dr < 0 ||
         (a->gate && a->ldgate < a->H);
}
bool shape_ok(const vlm_latent_mfma_args* a) {
  return a->R % 8 == 0 && a->Dr % 8 == 0 && a->R <= 512 && a->R + a->Dr <= 576 && a->H <= 65535 &&
         (((uintptr_t)a->q | (uintptr_t)a->pool | (uintptr_t)a->out) & 15) == 0;
}

}  // namespace

#define LATENT_SIZES(GO)                                                        \
  do {                                                                          \
    const int Dk = a->R + a->Dr;                                                \
    if (a->R <= 128 && Dk <= 192) GO(6, 1);                                     \
    else if (a->R <= 256 && Dk <= 320) GO(10, 2);                               \
    else GO(18, 4);                                                             \
  } while (0)
#define LDS_LIMIT(K, BYTES)                                                     \
  do {                                                                          \
    if ((BYTES) > 48 * 1024) {                                                  \
      hipError_t e = hipFuncSetAttribute((const void*)(K), hipFuncAttributeMaxDynamicSharedMemorySize, (int)(BYTES)); \
      if (e != hipSuccess) return VLM_ERR_HIP + (int)e;                         \
    }                                                                           \
  } while (0)

namespace {

template <typename TQ>
int blocks_form(const vlm_latent_mfma_args* a, int nblocks, hipStream_t stream) {
  if (bad(a) || !a->qb_start || !a->qb_count || nblocks < 0) return VLM_ERR_ARG;
  if (!shape_ok(a)) return VLM_ERR_SHAPE;
  if (nblocks == 0) return VLM_OK;
  if (nblocks > 65535) return VLM_ERR_SHAPE;
  const dim3 grid((a->H + 3) / 4, nblocks);
#define GO(NKS, NVC)                                                                                                        \
  do {                                                                                                                      \
    constexpr size_t lds = (size_t)2 * Tile<NKS>::SIZE * sizeof(bf16_t);                                                    \
    LDS_LIMIT((latent_block_mfma_kernel<TQ, NKS, NVC>), lds);                                                               \
    hipLaunchKernelGGL((latent_block_mfma_kernel<TQ, NKS, NVC>), grid, dim3(256), lds, stream, *a);                         \
  } while (0)
  LATENT_SIZES(GO);
#undef GO
  VLM_CHECK_LAUNCH();
  return VLM_OK;
}

template <typename TQ>
int rows_form(const vlm_latent_mfma_args* a, int rows, hipStream_t stream) {
  if (bad(a) || rows < 0 || a->nsplit < 0 || a->nsplit > 64 || (a->nsplit > 1 && !a->part)) return VLM_ERR_ARG;
  if (!shape_ok(a)) return VLM_ERR_SHAPE;
  if (rows == 0) return VLM_OK;
  const int nsplit = a->nsplit > 1 ? a->nsplit : 1;
  const dim3 grid(rows, (a->H + QC - 1) / QC, nsplit);
#define GO(NKS, NVC)                                                                                                        \
  do {                                                                                                                      \
    constexpr size_t lds = (size_t)Tile<NKS>::SIZE * sizeof(bf16_t) + PAGE * (QC + 1) * sizeof(float);                      \
    LDS_LIMIT((latent_rows_mfma_kernel<TQ, NKS, NVC>), lds);                                                                \
    hipLaunchKernelGGL((latent_rows_mfma_kernel<TQ, NKS, NVC>), grid, dim3(256), lds, stream, *a);                          \
  } while (0)
  LATENT_SIZES(GO);
#undef GO
  VLM_CHECK_LAUNCH();
  if (nsplit > 1) {
    hipLaunchKernelGGL((latent_merge_kernel<TQ>), dim3(rows, a->H, (a->R + 255) / 256), dim3(256), 0, stream, *a, nsplit);
    VLM_CHECK_LAUNCH();
  }
  return VLM_OK;
}

}  // namespace

extern "C" int vlm_latent_attn_mfma_blocks(const vlm_latent_mfma_args* a, int nblocks, void* stream) {
  return blocks_form<bf16_t>(a, nblocks, (hipStream_t)stream);
}
extern "C" int vlm_latent_attn_mfma_rows(const vlm_latent_mfma_args* a, int rows, void* stream) {
  return rows_form<bf16_t>(a, rows, (hipStream_t)stream);
}
extern "C" int vlm_latent_attn_mfma_f32(const vlm_latent_mfma_args* a, int nblocks, int rows, void* stream) {
  if (nblocks != 0 && rows != 0) return VLM_ERR_ARG;
  return rows ? rows_form<float>(a, rows, (hipStream_t)stream) : blocks_form<float>(a, nblocks, (hipStream_t)stream);
}
