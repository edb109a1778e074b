// Chunk-parallel form of two of the matrix-state recurrences of linear_recurrence.hip: fixed decay
//
//     S_t = a S_(t-1) + k_t v_t^T      o_t = S_t^T q_t          S: [D, Dv] per head, q / k / v optionally through silu, q / k optionally rotated
//
// and exponential gates (S_t = a_t S_(t-1) + b_t k_t v_t^T with the running maximum m_t and the normaliser n_t as one more column),
// for segments of more than max_len tokens (shorter ones stay with the token-by-token kernel).  A segment is cut into chunks of
// CH = 64 tokens counted from its first one; with S_0 the state a chunk starts from and i, j = 0 .. n - 1 its tokens
//
//     o_i = a^(i + 1) S_0^T q_i + sum_(j <= i) a^(i - j) (q_i . k_j) v_j        S_n = a^n S_0 + U,   U = sum_j a^(n - 1 - j) k_j v_j^T
//
// With gates the powers of a become exponentials of differences: F_i the sum of the log forget gates from the chunk's first token to i, i_j the
// log input gates, m_i the running maximum,
//
//     weight of (i, j) = exp(F_i - F_j + i_j - m_i)     of S_0 = exp(F_i + m_(before the chunk) - m_i)     never above 1
//
// F and these differences are kept in fp64 (a handful of numbers per token; fp32 sums of large gates would cost the small differences their digits).
//
//   chunk_rotate_kernel   q and k rotated and scaled once, fp32      -> workspace [2][token][H][D]        (rotated heads)
//   gate_scan_kernel      F, i, m of every token                     -> workspace, mtok                   (gated heads)
//   chunk_update_kernel   U of every chunk, all chunks at once       -> workspace [chunk][H][D][Dv] (| [D] of the normaliser)
//   chunk_scan_kernel     the recurrence over chunks, one lane per state entry: the workspace's U becomes the chunk's S_0, the
//                         slot's state moves to the segment's end
//   chunk_output_kernel   o of every chunk, all chunks at once       -> raw [token][H][Dv] fp32
// All products run on the fp32 matrix cores (v_mfma_f32_16x16x4_f32: fp32 operands, products and sums), straight from global memory
// into the operand layout - a lane's rows / columns of a tile are consecutive in memory, so the loads are 8 to 32 bytes wide and
// neither kernel needs LDS or a barrier.  In the output kernel the scores come out as S^T = K Q^T, keys 4 g + r of a tile in register
// r of lane group g, which is the operand layout of the product with V when step r contracts the keys 4 g + r.
// 2048 tokens of 12 heads of 128 (bf16): rotated fixed decay 1844 us token by token -> 128 us (rotate 26, update 26, scan 11, output 41, norm 15, 10
// of launches), gated 1730 + 125 of maxima -> 144 us (gates 14, update 37, scan 19, output 56, norm 17).  A serial chain before, now bound by the
// fp32 products' operands from the caches.
// Chunks are numbered over all long segments of the step; a launch covers the chunks [c0, c0 + nc) the workspace has room for, and
// windows of chunks follow each other on the stream (the slot's state carries a segment from one window to the next).
#include "common.hpp"
#include "../../include/vlm_hip.h"
#include "recurrence_finish.hpp"
#include "chunk_recurrence.hpp"

namespace {

constexpr int CH = VLM_CHUNK;

__device__ __forceinline__ float silu_f(float x) { return x * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x)); }

// a^n for n >= 0, exact for n = 0 and a = 0
struct Power {
  float l2;                      // log2 |a|
  unsigned sign;                 // the sign bit of a
};
__device__ __forceinline__ Power power_of(float a) { return Power{__builtin_amdgcn_logf(fabsf(a)), __float_as_uint(a) & 0x80000000u}; }
__device__ __forceinline__ float powi(Power a, int n) {
  const float r = n == 0 ? 1.f : __builtin_amdgcn_exp2f(a.l2 * (float)n);
  return __uint_as_float(__float_as_uint(r) ^ (n & 1 ? a.sign : 0u));
}

// N consecutive values of a row, the first `have` of which exist
template <int N> __device__ __forceinline__ void row_vals(const bf16_t* p, int have, bool vec, float* f) {
  if (vec && have >= N && N >= 4) {
#pragma unroll
    for (int i = 0; i < N / 4; ++i) {
      const uint2 a = reinterpret_cast<const uint2*>(p)[i];
      f[4 * i] = bf_lo(a.x); f[4 * i + 1] = bf_hi(a.x); f[4 * i + 2] = bf_lo(a.y); f[4 * i + 3] = bf_hi(a.y);
    }
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) f[i] = i < have ? bf2f(p[i]) : 0.f;
  }
}
template <int N> __device__ __forceinline__ void row_vals(const float* p, int have, bool vec, float* f) {
  if (vec && have >= N && N >= 4) {
#pragma unroll
    for (int i = 0; i < N / 4; ++i) {
      const float4 a = reinterpret_cast<const float4*>(p)[i];
      f[4 * i] = a.x; f[4 * i + 1] = a.y; f[4 * i + 2] = a.z; f[4 * i + 3] = a.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) f[i] = i < have ? p[i] : 0.f;
  }
}

// what the gated form knows of every (token, head)
struct GateRows {
  const double* F;               // [token][H]
  const float* ig;               // [token][H]
};
__device__ __forceinline__ float exp_d(double x) { return expf((float)x); }

// the segment and the first token of global chunk number c (false: the step has fewer chunks)
__device__ __forceinline__ bool find_chunk(const vlm_recurrence_args& p, int nseg, int max_len, int c, int& t0, int& n, int& seg) {
  for (int s = 0; s < nseg; ++s) {
    const int b = p.seg_start[s], len = p.seg_start[s + 1] - b;
    if (len <= max_len) continue;
    const int k = (len + CH - 1) / CH;
    if (c < k) {
      seg = s;
      t0 = b + c * CH;
      n = min(CH, len - c * CH);
      return true;
    }
    c -= k;
  }
  return false;
}

// grid (chunks, H, ceil(super tiles / 4)), 4 waves: a wave owns 64 x 64 entries of U.  Row block rb of the super tile holds rows
// 4 r16 + rb, so one load of four consecutive values feeds four row blocks (columns alike)
template <typename TK, typename T, bool GATED>
__global__ __launch_bounds__(256) void chunk_update_kernel(vlm_recurrence_args p, GateRows gr, int nseg, int max_len, int c0, float* __restrict__ ws) {
  const int h = blockIdx.y, lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4, D = p.D, Dv = p.Dv;
  const int st = blockIdx.z * 4 + (threadIdx.x >> 6), sc = (Dv + 63) / 64;
  if (st >= ((D + 63) / 64) * sc) return;
  int t0, n, seg;
  if (!find_chunk(p, nseg, max_len, c0 + blockIdx.x, t0, n, seg)) return;
  const int d0 = (st / sc) * 64 + 4 * r16, v0 = (st % sc) * 64 + 4 * r16;
  const TK* k = (const TK*)p.k + (long)h * D + d0;
  const T* v = (const T*)p.v + (long)h * Dv + v0;
  const bool kvec = ((uintptr_t)p.k % (4 * sizeof(TK))) == 0 && p.ldk % 4 == 0 && D % 4 == 0;
  const bool vvec = ((uintptr_t)p.v % (4 * sizeof(T))) == 0 && p.ldv % 4 == 0 && Dv % 4 == 0;
  const Power pw = power_of(GATED ? 0.f : p.decay[h]);
  double Fm = 0.;                                                        // (gated) F - m at the chunk's last token
  if constexpr (GATED) Fm = gr.F[(long)(t0 + n - 1) * p.H + h] - (double)p.mtok[(long)(t0 + n - 1) * p.H + h];
  float nacc[4] = {};                                                    // (gated) the normaliser's entries of this lane's rows
  f32x4_t acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
  for (int j0 = 0; j0 < n; j0 += 4) {
    const int j = j0 + g;
    const bool live = j < n;
    const long tok = t0 + (live ? j : 0);
    float kv[4], vv[4];
    row_vals<4>(k + tok * p.ldk, live ? D - d0 : 0, kvec, kv);
    row_vals<4>(v + tok * p.ldv, live ? Dv - v0 : 0, vvec, vv);
    float w = 0.f;
    if (live) w = (GATED ? exp_d(Fm - gr.F[tok * p.H + h] + (double)gr.ig[tok * p.H + h]) : powi(pw, n - 1 - j)) * p.kscale;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      kv[i] = (p.k_act ? silu_f(kv[i]) : kv[i]) * w;
      vv[i] = p.v_act ? silu_f(vv[i]) : vv[i];
      nacc[i] += kv[i];
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[a], vv[b], acc[a][b], 0, 0, 0);
  }
  // tile (a, b): row 4 (4 g + r) + a, column 4 r16 + b of the super tile
  float* U = ws + ((long)blockIdx.x * p.H + h) * (long)D * (Dv + GATED);
  const bool uvec = Dv % 4 == 0 && (((uintptr_t)U) & 15) == 0;          // (with a normaliser column a chunk's piece may begin anywhere)
  if constexpr (GATED) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = col4_sum(nacc[i]);
      if (st % sc == 0 && g == 0 && d0 + i < D) U[(long)D * Dv + d0 + i] = x;
    }
  }
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = (st / sc) * 64 + 4 * (4 * g + r) + a;
      if (d >= D) continue;
      float* u = U + (long)d * Dv + v0;
      if (uvec) {
        if (v0 < Dv) *reinterpret_cast<float4*>(u) = make_float4(acc[a][0][r], acc[a][1][r], acc[a][2][r], acc[a][3][r]);
      } else {
#pragma unroll
        for (int b = 0; b < 4; ++b)
          if (v0 + b < Dv) u[b] = acc[a][b][r];
      }
    }
}

// grid (state entries / 256, nseg)
template <bool GATED>
__global__ __launch_bounds__(256) void chunk_scan_kernel(vlm_recurrence_args p, GateRows gr, int nseg, int max_len, int c0, int nc, float* __restrict__ ws) {
  const int seg = blockIdx.y;
  const int b = p.seg_start[seg], len = p.seg_start[seg + 1] - b;
  if (len <= max_len) return;
  int before = 0;                                                        // chunks of the long segments ahead of this one
  for (int s = 0; s < seg; ++s) {
    const int l = p.seg_start[s + 1] - p.seg_start[s];
    if (l > max_len) before += (l + CH - 1) / CH;
  }
  const int chunks = (len + CH - 1) / CH;
  const int lo = max(0, c0 - before), hi = min(chunks, c0 + nc - before);  // the segment's chunks inside the window
  if (lo >= hi) return;
  const long E = (long)p.D * (p.Dv + GATED), HE = (long)p.H * E, e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= HE) return;
  const int h = (int)(e / E);
  // the workspace keeps the normaliser behind the other columns, the slot as the last of every row
  long se = e;
  if constexpr (GATED) {
    const long i = e % E, DDv = (long)p.D * p.Dv;
    se = h * E + (i < DDv ? i / p.Dv * (p.Dv + 1) + i % p.Dv : (i - DDv) * (p.Dv + 1) + p.Dv);
  }
  float* S = p.state + (long)p.seg_slot[seg] * HE + se;
  float s = (lo > 0 || p.seg_pos0[seg] > 0) ? *S : 0.f;
  float* w = ws + (long)(before + lo - c0) * HE + e;
  int c = lo;
  if constexpr (GATED) {
    float m = lo > 0 ? p.mtok[(long)(b + lo * CH - 1) * p.H + h] : p.mprev[(long)seg * p.H + h];
    for (; c < hi; c += 4) {                                             // four chunks' loads in flight
      float u[4], f[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int x = min(c + i, hi - 1);
        const long tok = b + min((x + 1) * CH, len) - 1;
        const float m1 = p.mtok[tok * p.H + h];
        u[i] = w[(long)(x - lo) * HE];
        f[i] = exp_d(gr.F[tok * p.H + h] + (double)m - (double)m1);
        m = m1;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (c + i >= hi) break;
        w[(long)(c + i - lo) * HE] = s;
        s = fmaf(f[i], s, u[i]);
      }
    }
    *S = s;
    return;
  }
  const Power pw = power_of(p.decay[h]);
  const float full = powi(pw, CH);
  for (; c + 4 < hi; c += 4, w += 4 * HE) {                              // whole chunks, four loads in flight
    float u[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = w[i * HE];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[i * HE] = s;
      s = fmaf(full, s, u[i]);
    }
  }
  for (; c < hi; ++c, w += HE) {
    const float u = *w;
    *w = s;
    s = fmaf(c + 1 < chunks ? full : powi(pw, len - c * CH), s, u);
  }
  *S = s;
}

// grid (chunks, H, value column tiles of 16 NB), 4 waves: wave w owns tokens 16 w .. 16 w + 15 of the chunk
template <typename TK, typename T, int NB, bool GATED>
__global__ __launch_bounds__(256) void chunk_output_kernel(vlm_recurrence_args p, GateRows gr, int nseg, int max_len, int c0, const float* __restrict__ ws) {
  const int h = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4, D = p.D, Dv = p.Dv;
  int t0, n, seg;
  if (!find_chunk(p, nseg, max_len, c0 + blockIdx.x, t0, n, seg)) return;
  const int i = wave * 16 + r16;                                         // this lane's query
  if (wave * 16 >= n) return;
  const int vcol = blockIdx.z * 16 * NB + r16 * NB, vhave = Dv - vcol;
  const TK* qp = (const TK*)p.q + (long)(t0 + min(i, n - 1)) * p.ldq + (long)h * D;
  const TK* kp = (const TK*)p.k + (long)t0 * p.ldk + (long)h * D;
  const T* vp = (const T*)p.v + (long)t0 * p.ldv + (long)h * Dv + vcol;
  const bool qvec = ((uintptr_t)p.q % (4 * sizeof(TK))) == 0 && p.ldq % 4 == 0 && D % 4 == 0;
  const bool kvec = ((uintptr_t)p.k % (4 * sizeof(TK))) == 0 && p.ldk % 4 == 0 && D % 4 == 0;
  const bool vvec = ((uintptr_t)p.v % (4 * sizeof(T))) == 0 && p.ldv % 4 == 0 && Dv % 4 == 0;
  const float* S0 = ws + ((long)blockIdx.x * p.H + h) * (long)D * (Dv + GATED);
  const float* S = S0 + vcol;
  const bool svec = Dv % 4 == 0 && (((uintptr_t)S0) & 15) == 0;
  const Power pw = power_of(GATED ? 0.f : p.decay[h]);
  const long ti = (long)(t0 + min(i, n - 1)) * p.H + h;
  double Fm = 0.;                                                        // (gated) F - m of this lane's query
  float nq = 0.f, mine = 0.f;                                            // (gated) normaliser . q: the chunk's start, its tokens
  if constexpr (GATED) Fm = gr.F[ti] - (double)p.mtok[ti];
  f32x4_t acc[NB], s[4];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < 4; ++t) s[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int c = 0; c < D; c += 16) {
    const int d = c + 4 * g;
    float q[4];
    row_vals<4>(qp + d, D - d, qvec, q);
#pragma unroll
    for (int x = 0; x < 4; ++x) q[x] = (p.q_act ? silu_f(q[x]) : q[x]) * p.qscale;
    // scores against the key tiles up to the wave's own
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (t > wave) break;
      float k[4];
      row_vals<4>(kp + (long)min(t * 16 + r16, n - 1) * p.ldk + d, D - d, kvec, k);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        k[x] = (p.k_act ? silu_f(k[x]) : k[x]) * p.kscale;
        s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[x], q[x], s[t], 0, 0, 0);
      }
    }
    // the state the chunk starts from
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      float sv[NB];
      row_vals<NB>(S + (long)min(d + x, D - 1) * Dv, d + x < D ? vhave : 0, svec, sv);
      if constexpr (GATED) nq = fmaf(S0[(long)D * Dv + min(d + x, D - 1)], d + x < D ? q[x] : 0.f, nq);
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(sv[b], q[x], acc[b], 0, 0, 0);
    }
  }
  float ai;
  if constexpr (GATED) {
    const int first = p.seg_start[seg];
    ai = exp_d(Fm + (double)(t0 > first ? p.mtok[(long)(t0 - 1) * p.H + h] : p.mprev[(long)seg * p.H + h]));
  } else {
    ai = powi(pw, i + 1);
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] *= ai;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (t > wave) break;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = t * 16 + 4 * g + r;
      float pr = 0.f;                                                    // (tokens past the chunk's end are later than every real query)
      if (j <= i) {
        if constexpr (GATED) {
          const long tj = (long)(t0 + min(j, n - 1)) * p.H + h;
          pr = s[t][r] * exp_d(Fm - gr.F[tj] + (double)gr.ig[tj]);
        } else {
          pr = s[t][r] * powi(pw, i - j);
        }
      }
      mine += pr;
      float v[NB];
      row_vals<NB>(vp + (long)min(j, n - 1) * p.ldv, vhave, vvec, v);
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(p.v_act ? silu_f(v[b]) : v[b], pr, acc[b], 0, 0, 0);
    }
  }
  float odd = 0.f;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int x = 0; x < 4; ++x) odd = fmaf(acc[b][x], 0.f, odd);
  if constexpr (GATED) nq = fmaf(col4_sum(nq), ai, col4_sum(mine));
  if (i >= n) return;
  // block b, register r of lane group g: column (4 g + r) NB + b of the tile
  float* o = p.raw + ((long)(t0 + i) * p.H + h) * (Dv + GATED);
  if (GATED && blockIdx.z == 0 && g == 0) o[Dv] = nq;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int c = blockIdx.z * 16 * NB + (4 * g + r) * NB;
    if (!GATED && NB % 4 == 0 && Dv % 4 == 0) {
#pragma unroll
      for (int b = 0; b < NB; b += 4)
        if (c + b < Dv) *reinterpret_cast<float4*>(o + c + b) = make_float4(acc[b][r], acc[(b + 1) % NB][r], acc[(b + 2) % NB][r], acc[(b + 3) % NB][r]);
    } else {
#pragma unroll
      for (int b = 0; b < NB; ++b)
        if (c + b < Dv) o[c + b] = acc[b][r];
    }
  }
  if (!__any(odd != 0.f)) return;
  // a value that is not finite met the zero weights of the queries before it in the last tile: these tokens' read-outs once more, without such products
  const int first = blockIdx.z * 16 * NB + 4 * g * NB, last = min(first + 4 * NB, Dv);
  const auto value = [](const auto* x, int act, float scale) {
    float f;
    row_vals<1>(x, 1, false, &f);
    return (act ? silu_f(f) : f) * scale;
  };
#pragma unroll 1
  for (int c = first; c < last; ++c) {
    float x = 0.f;
#pragma unroll 1
    for (int d = 0; d < D; ++d) x = fmaf(S0[(long)d * Dv + c], value(qp + d, p.q_act, p.qscale), x);
    o[c] = x * ai;
  }
#pragma unroll 1
  for (int j = 0; j <= i; ++j) {
    float x = 0.f;
#pragma unroll 1
    for (int d = 0; d < D; ++d) x = fmaf(value(kp + (long)j * p.ldk + d, p.k_act, p.kscale), value(qp + d, p.q_act, p.qscale), x);
    const long tj = (long)(t0 + j) * p.H + h;
    x *= GATED ? exp_d(Fm - gr.F[tj] + (double)gr.ig[tj]) : powi(pw, i - j);
#pragma unroll 1
    for (int c = first; c < last; ++c) o[c] = fmaf(x, value((const T*)p.v + (long)(t0 + j) * p.ldv + (long)h * Dv + c, p.v_act, 1.f), o[c]);
  }
}

// q and k of the long segments' tokens, rotated (rotate-half pairs on the first rot_dims dimensions) and scaled: grid (tokens, 2), out [2][token][H][D]
template <typename T>
__global__ __launch_bounds__(256) void chunk_rotate_kernel(vlm_recurrence_args p, int nseg, int max_len, int ntok, float* __restrict__ out) {
  const int t = blockIdx.x, H = p.H, D = p.D, half = p.rot_dims / 2;
  int seg = 0;
  while (seg + 1 < nseg && p.seg_start[seg + 1] <= t) ++seg;
  if (p.seg_start[seg + 1] - p.seg_start[seg] <= max_len) return;
  const float pos = (float)(p.seg_pos0[seg] + t - p.seg_start[seg]);
  const T* src = blockIdx.y ? (const T*)p.k + (long)t * p.ldk : (const T*)p.q + (long)t * p.ldq;
  float* dst = out + ((long)blockIdx.y * ntok + t) * H * D;
  const float scale = blockIdx.y ? p.kscale : p.qscale;
  for (int x = threadIdx.x; x < H * D; x += 256) {
    const int i = x % D, base = x - i;
    float v = ld_f(src + x);
    if (i < p.rot_dims) {
      const int j = i < half ? i : i - half;
      float sn, cs;
      sincosf(pos * p.inv_freq[j], &sn, &cs);
      const float o = ld_f(src + base + (i < half ? i + half : j));
      v = i < half ? v * cs - o * sn : v * cs + o * sn;
    }
    dst[x] = v * scale;
  }
}

__device__ __forceinline__ float logsigmoid_f(float x) { return fminf(x, 0.f) - log1pf(expf(-fabsf(x))); }
__device__ __forceinline__ double shfl_up_d(double v, int n, double none) {
  const double o = __shfl_up(v, n);
  return (int)(threadIdx.x & 63) >= n ? o : none;
}

// gates of the long segments: grid (nseg, H), 16 waves, one chunk per wave and turn.  With F_t the sum of f from the chunk's first token and M the
// largest i_j - F_j so far, m_t = F_t + max(m before the chunk, M); the chunks of a turn are strung together by one lane.
template <typename T>
__global__ __launch_bounds__(1024) void gate_scan_kernel(vlm_recurrence_args p, int max_len, double* __restrict__ F, float* __restrict__ ig) {
  __shared__ double end[16], top[16], start[17];
  const int seg = blockIdx.x, h = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b = p.seg_start[seg], len = p.seg_start[seg + 1] - b;
  if (len <= max_len) return;
  float* ms = p.mstate + (long)p.seg_slot[seg] * p.H + h;
  if (threadIdx.x == 0) {
    const float m = p.seg_pos0[seg] > 0 ? *ms : 0.f;
    p.mprev[(long)seg * p.H + h] = m;
    start[0] = (double)m;
  }
  const float bi = ld_f((const T*)p.ib + h), bf = ld_f((const T*)p.fb + h);
  for (int c0 = 0; c0 * CH < len; c0 += 16) {
    const int t = (c0 + wave) * CH + lane;
    const bool live = t < len;
    const long tok = b + min(t, len - 1);
    const float iv = p.cap * tanhf((ld_f((const T*)p.ipre + tok * p.ldi + h) + bi) / p.cap);
    double f = (double)logsigmoid_f(p.cap * tanhf((ld_f((const T*)p.fpre + tok * p.ldf + h) + bf) / p.cap));
    if (!live) f = 0.;
#pragma unroll
    for (int n = 1; n < 64; n <<= 1) f += shfl_up_d(f, n, 0.);
    double M = live ? (double)iv - f : -INFINITY;
#pragma unroll
    for (int n = 1; n < 64; n <<= 1) M = fmax(M, shfl_up_d(M, n, -INFINITY));
    if (lane == 63) {
      end[wave] = f;
      top[wave] = M;
    }
    __syncthreads();
    if (threadIdx.x == 0)                                                // (a slot past the last chunk: F = 0, no maximum - m goes through)
      for (int w = 0; w < 16; ++w) start[w + 1] = (double)(float)(end[w] + fmax(start[w], top[w]));
    __syncthreads();
    const float m = (float)(f + fmax(start[wave], M));
    if (live) {
      p.mtok[tok * p.H + h] = m;
      F[tok * p.H + h] = f;
      ig[tok * p.H + h] = iv;
      if (t == len - 1) *ms = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) start[0] = start[16];
    __syncthreads();
  }
}

template <typename TK, typename T, bool GATED>
int run_windows(const vlm_recurrence_args& a, const GateRows& gr, int nseg, int ntok, int max_len, float* ws, long ws_floats, hipStream_t st) {
  const long HE = (long)a.H * a.D * (a.Dv + GATED);
  const int total = ntok / CH + nseg;                                    // at most this many chunks
  const long room = ws_floats / HE;
  if (room < 1) return VLM_ERR_ARG;
  const int win = (int)(room < total ? room : total);
  const int tiles = ((a.D + 63) / 64) * ((a.Dv + 63) / 64);
  const int NB = a.Dv <= 16 ? 1 : a.Dv <= 64 ? 4 : 8, vt = (a.Dv + 16 * NB - 1) / (16 * NB);
  if ((HE + 255) / 256 > 0x7fffffffL || nseg > 65535) return VLM_ERR_SHAPE;
  for (int c0 = 0; c0 < total; c0 += win) {
    const int nc = total - c0 < win ? total - c0 : win;
    hipLaunchKernelGGL((chunk_update_kernel<TK, T, GATED>), dim3(nc, a.H, (tiles + 3) / 4), dim3(256), 0, st, a, gr, nseg, max_len, c0, ws);
    VLM_CHECK_LAUNCH();
    hipLaunchKernelGGL((chunk_scan_kernel<GATED>), dim3((unsigned)((HE + 255) / 256), nseg), dim3(256), 0, st, a, gr, nseg, max_len, c0, nc, ws);
    VLM_CHECK_LAUNCH();
    const dim3 grid(nc, a.H, vt);
    if (NB == 1) hipLaunchKernelGGL((chunk_output_kernel<TK, T, 1, GATED>), grid, dim3(256), 0, st, a, gr, nseg, max_len, c0, ws);
    else if (NB == 4) hipLaunchKernelGGL((chunk_output_kernel<TK, T, 4, GATED>), grid, dim3(256), 0, st, a, gr, nseg, max_len, c0, ws);
    else hipLaunchKernelGGL((chunk_output_kernel<TK, T, 8, GATED>), grid, dim3(256), 0, st, a, gr, nseg, max_len, c0, ws);
    VLM_CHECK_LAUNCH();
  }
  return VLM_OK;
}

template <typename T>
int run_chunks(const vlm_recurrence_args& a, int nseg, int ntok, int max_len, hipStream_t st) {
  const long prep = vlm_chunk_prep_floats(&a, ntok);
  float* ws = a.ws + prep;
  const long left = a.ws_floats - prep;
  if (a.gated == 1) {
    double* F = reinterpret_cast<double*>(a.ws);
    float* ig = a.ws + 2 * (long)ntok * a.H;
    hipLaunchKernelGGL((gate_scan_kernel<T>), dim3(nseg, a.H), dim3(1024), 0, st, a, max_len, F, ig);
    VLM_CHECK_LAUNCH();
    vlm_recurrence_args b = a;
    b.q_act = 0;                                                         // (an activation of q belongs to the other recurrences)
    return run_windows<T, T, true>(b, GateRows{F, ig}, nseg, ntok, max_len, ws, left, st);
  }
  if (a.rot_dims) {
    hipLaunchKernelGGL((chunk_rotate_kernel<T>), dim3(ntok, 2), dim3(256), 0, st, a, nseg, max_len, ntok, a.ws);
    VLM_CHECK_LAUNCH();
    vlm_recurrence_args b = a;
    b.q = a.ws;
    b.k = a.ws + (long)ntok * a.H * a.D;
    b.ldq = b.ldk = (long)a.H * a.D;
    b.qscale = b.kscale = 1.f;
    return run_windows<float, T, false>(b, GateRows{}, nseg, ntok, max_len, ws, left, st);
  }
  return run_windows<T, T, false>(a, GateRows{}, nseg, ntok, max_len, ws, left, st);
}

}  // namespace

int vlm_chunk_recurrence(const vlm_recurrence_args* a, int nseg, int ntok, int max_len, int dtype, hipStream_t st) {
  return dtype ? run_chunks<float>(*a, nseg, ntok, max_len, st) : run_chunks<bf16_t>(*a, nseg, ntok, max_len, st);
}
