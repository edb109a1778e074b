// Delta-rule recurrences: matrix states S [D, Dv] per head (fp32, one per sequence slot) whose update READS the old state
// before it writes - the new association k -> v replaces what the state returned for that key instead of adding to it.
//
//   * gated (mode 0): one decay g_t and one write strength beta_t per head and token
//         S' = g_t S_(t-1)        u_t = beta_t (v_t - S'^T k_t)        S_t = S' + k_t u_t^T        o_t = S_t^T q_t
//     q and k are unit vectors per head (x / sqrt(sum x^2 + 1e-6), q times D^-1/2) of short causal convolutions (silu) of
//     the projections; q / k heads may be shared by groups of value heads.
//   * general (mode 1): a decay w_t and a removal rate a_t per key channel, unit key u_t = k_t / sqrt(sum k_t^2 + 1e-6)
//         S_t = diag(w_t) S_(t-1) - (a_t * u_t) (u_t^T S_(t-1)) + k_t v_t^T                        o_t = S_t^T r_t
//     both correction terms read S_(t-1).
//
// The work is split into a PREPARE pass (everything per token that does not depend on the state: convolutions, unit norms,
// gates, decays - evaluated in fp32, written as fp32 rows), the SCAN (sequential in the tokens of a segment, same arithmetic
// wherever a prompt was cut) and the finish pass shared with linear_recurrence.hip (per-head unit RMS, weight, output gate).
// A segment is a run of consecutive tokens of one sequence: the state (and the convolution's last taps - 1 inputs) comes from
// the sequence's slot - or is zero when the segment starts at position 0, so a slot that is used again needs no clearing -
// and goes back there.
//
// Scan work split: a state column's rows lie in the registers of 8 / 16 / 32 neighbouring lanes, workgroup = (segment, head, tile of columns) of four
// waves; heads up to 1024 wide.  What bounds a long segment is the chain of one token - a dot product with the state, its sum over the lanes, the
// update - times the tokens, so the rows are spread thin (768 waves for 12 heads of 128, where 16 rows a lane on 8 lanes, one sum after the other
// and tokens staged behind a barrier took 1159 us for 1500 tokens in the general form and 831 us in the gated one: now 265 and 240), the sum of a
// read-out runs beside the next token's, and the tokens' vectors arrive in LDS by direct loads two blocks ahead.
#include "common.hpp"
#include "../../include/vlm_hip.h"
#include "recurrence_finish.hpp"

namespace {

__device__ __forceinline__ float sigmoid_f(float x) { return 1.f / (1.f + expf(-x)); }
__device__ __forceinline__ float softplus_f(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }
__device__ __forceinline__ float silu_f(float x) { return x * sigmoid_f(x); }

__device__ __forceinline__ int segment_of(const int* __restrict__ seg_start, int nseg, int t) {
  int lo = 0, hi = nseg;                 // largest s with seg_start[s] <= t
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (seg_start[mid] <= t) lo = mid; else hi = mid;
  }
  return lo;
}

// ---------------------------------------------------------------------------------------------------------------- prepare
// general form: grid (tokens, heads), one wave.  lw = W2 tanh(low) + w0 is the small second map of the decay (rank R).
template <typename T>
__global__ __launch_bounds__(64) void delta_prep_general_kernel(vlm_delta_prep_general_args p) {
  extern __shared__ float smem[];        // [R] tanh of the low-rank decay input
  const long t = blockIdx.x;
  const int h = blockIdx.y, lane = threadIdx.x, D = p.D, HD = p.H * p.D;
  const T* low = (const T*)p.low + t * p.ld_low;
  for (int j = lane; j < p.R; j += 64) smem[j] = tanhf(ld_f(low + j));
  __syncthreads();
  const T* kr = (const T*)p.k + t * p.ld + (long)h * D;
  float ss = 0.f;
  for (int i = lane; i < D; i += 64) {
    const float kv = ld_f(kr + i);
    ss += kv * kv;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  const float rn = 1.0f / sqrtf(ss + 1e-6f);
  const long o0 = t * HD + (long)h * D;
  for (int i = lane; i < D; i += 64) {
    const int c = h * D + i;
    const float kv = ld_f(kr + i), u = kv * rn;
    float lw = ld_f((const T*)p.w0 + c);
    const T* w2 = (const T*)p.w2 + (long)c * p.R;
    for (int j = 0; j < p.R; ++j) lw = fmaf(ld_f(w2 + j), smem[j], lw);
    const float a = sigmoid_f(ld_f((const T*)p.a + t * p.ld + c) + ld_f((const T*)p.a_bias + c));
    p.q[o0 + i] = ld_f((const T*)p.r + t * p.ld + c);
    p.kw[o0 + i] = kv;
    p.kr[o0 + i] = u;
    p.v[o0 + i] = ld_f((const T*)p.v_in + t * p.ld + c);
    p.w[o0 + i] = expf(-0.6065306597126334f * sigmoid_f(lw));      // exp(-1/2) = 0.60653...
    p.b[o0 + i] = a * u;
  }
}

// gated form: grid (tokens), 256 lanes.  Channels: q [KH * D] | k [KH * D] | v [H * Dv]; conv weights [channels][taps] with
// the current token's tap last; conv state fp32 [slot][taps - 1][channels] = the inputs at the taps - 1 positions before the
// segment (positions below 0 count as zeros whatever the slot holds).
template <typename T>
__global__ __launch_bounds__(256) void delta_prep_gated_kernel(vlm_delta_prep_gated_args p, int nseg) {
  extern __shared__ float y[];           // [channels] conv + silu
  const int t = blockIdx.x, tid = threadIdx.x;
  const int KD = p.KH * p.D, HV = p.H * p.Dv, Cn = 2 * KD + HV, taps = p.taps;
  const int seg = segment_of(p.seg_start, nseg, t);
  const int t0 = p.seg_start[seg], pos0 = p.seg_pos0[seg], pos = pos0 + (t - t0);
  const float* cs = p.conv_state + (long)p.seg_slot[seg] * (taps - 1) * Cn;
  for (int c = tid; c < Cn; c += 256) {
    const T* src;
    const T* cw;
    int cc;
    if (c < KD) { src = (const T*)p.q_in; cw = (const T*)p.q_conv; cc = c; }
    else if (c < 2 * KD) { src = (const T*)p.k_in; cw = (const T*)p.k_conv; cc = c - KD; }
    else { src = (const T*)p.v_in; cw = (const T*)p.v_conv; cc = c - 2 * KD; }
    float acc = 0.f;
    for (int j = 0; j < taps; ++j) {     // tap j sits taps - 1 - j tokens back
      const int pp = pos - (taps - 1) + j;
      float x = 0.f;
      if (pp >= pos0) x = ld_f(src + (long)(t0 + (pp - pos0)) * p.ld + cc);
      else if (pp >= 0) x = cs[(long)(taps - 1 - (pos0 - pp)) * Cn + c];
      acc = fmaf(ld_f(cw + (long)cc * taps + j), x, acc);
    }
    y[c] = silu_f(acc);
  }
  __syncthreads();
  const int wave = tid >> 6, lane = tid & 63;
  for (int hh = wave; hh < 2 * p.KH; hh += 4) {          // unit vectors: q heads then k heads
    const float* src = y + (long)hh * p.D;
    float ss = 0.f;
    for (int i = lane; i < p.D; i += 64) ss += src[i] * src[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
    const float rn = 1.0f / sqrtf(ss + 1e-6f);
    const bool isq = hh < p.KH;
    float* dst = (isq ? p.q : p.k) + (long)t * KD + (long)(isq ? hh : hh - p.KH) * p.D;
    const float sc = isq ? p.qscale : 1.f;
    for (int i = lane; i < p.D; i += 64) dst[i] = src[i] * rn * sc;
  }
  for (int c = tid; c < HV; c += 256) p.v[(long)t * HV + c] = y[2 * KD + c];
  for (int h = tid; h < p.H; h += 256) {
    p.beta[(long)t * p.H + h] = sigmoid_f(ld_f((const T*)p.b_in + (long)t * p.ld + h));
    const float dt = softplus_f(ld_f((const T*)p.a_in + (long)t * p.ld + h) + ld_f((const T*)p.dt_bias + h));
    p.g[(long)t * p.H + h] = expf(-expf(ld_f((const T*)p.A_log + h)) * dt);
  }
}

// the slot's last taps - 1 inputs after the segment: grid (segments), lanes over channels.  Entry j holds the input at
// position end - (taps - 1) + j; for a segment shorter than taps - 1 the older entries move down (entry j reads old entry
// j + n, ascending j: read before overwritten).
template <typename T>
__global__ __launch_bounds__(256) void delta_conv_state_kernel(vlm_delta_prep_gated_args p) {
  const int seg = blockIdx.x;
  const int KD = p.KH * p.D, HV = p.H * p.Dv, Cn = 2 * KD + HV, taps = p.taps;
  const int t0 = p.seg_start[seg], n = p.seg_start[seg + 1] - t0, pos0 = p.seg_pos0[seg];
  float* cs = p.conv_state + (long)p.seg_slot[seg] * (taps - 1) * Cn;
  for (int c = blockIdx.y * 256 + threadIdx.x; c < Cn; c += gridDim.y * 256) {
    const T* src;
    int cc;
    if (c < KD) { src = (const T*)p.q_in; cc = c; }
    else if (c < 2 * KD) { src = (const T*)p.k_in; cc = c - KD; }
    else { src = (const T*)p.v_in; cc = c - 2 * KD; }
    for (int j = 0; j < taps - 1; ++j) {
      const int pp = pos0 + n - (taps - 1) + j;
      float x = 0.f;
      if (pp >= pos0) x = ld_f(src + (long)(t0 + (pp - pos0)) * p.ld + cc);
      else if (pp >= 0) x = cs[(long)(j + n) * Cn + c];
      cs[(long)j * Cn + c] = x;
    }
  }
}

// ------------------------------------------------------------------------------------------------------------------- scan
// The order of a dot product over a state column's rows is the same for every spread of the rows over lanes: two chains over four rows, then a binary
// tree over the fours - inside a lane first, then over the lanes.
template <int DR> __device__ __forceinline__ float row_dot(const float* s, const f32x4_t* m) {
  if constexpr (DR == 4) return fmaf(s[2], m[0][2], s[0] * m[0][0]) + fmaf(s[3], m[0][3], s[1] * m[0][1]);
  else return row_dot<DR / 2>(s, m) + row_dot<DR / 2>(s + DR / 2, m + DR / 8);
}

// sums over the RG lanes of a state column, in every one of them
template <int RG, int NC> __device__ __forceinline__ void group_sum(float (&v)[NC]) {
#pragma unroll
  for (int c = 0; c < NC; ++c) v[c] += vlm_dpp<0xB1, 0xf>(0.f, v[c]);      // quad_perm [1,0,3,2]
#pragma unroll
  for (int c = 0; c < NC; ++c) v[c] += vlm_dpp<0x4E, 0xf>(0.f, v[c]);      // quad_perm [2,3,0,1]
#pragma unroll
  for (int c = 0; c < NC; ++c) v[c] += vlm_dpp<0x141, 0xf>(0.f, v[c]);     // row_half_mirror: the other quad of eight lanes
  if constexpr (RG >= 16)
#pragma unroll
    for (int c = 0; c < NC; ++c) v[c] += vlm_dpp<0x140, 0xf>(0.f, v[c]);   // row_mirror: the other eight of sixteen
  if constexpr (RG >= 32)
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float a, b;
      vlm_xor16_pair(v[c], a, b);
      v[c] = a + b;
    }
}

// 16 / 4 bytes from every lane's address to LDS, lane i's at dst + 16 / 4 * i bytes
__device__ __forceinline__ void direct_load16(const float* src, float* dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}
__device__ __forceinline__ void direct_load4(const float* src, float* dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)dst, 4, 0, 0);
}

// lane = (column group lane / RG of the wave's 64 / RG, row group rg = lane % RG): rows [DR rg, DR rg + DR) of NC neighbouring state columns in
// registers.  A token's vectors in LDS: [vector][token of the block][RG * DR], a lane reads its own rows, four at a time; a lane's fours lie RG fours apart, so that
// neighbouring lanes read neighbouring 16 bytes (as the rows come, lanes of 8 to 32 rows met in the same banks: general form, 4 x 30 tokens of 2 heads of 1024,
// 96 us instead of 42).  WHOLE: D == RG * DR, the vectors' rows in whole aligned 16-byte pieces, and state rows in pieces of NC; FOURS: such vectors alone
// (general form, D = 100, 700 + 700 tokens of 12 heads: 163 us, element by element 358); ANY: element by element.  Zeros past D.
template <int DR, int RG, int NC, bool GENERAL> struct ScanShape {
  static constexpr int DP = RG * DR, NV = GENERAL ? 5 : 2;
  static constexpr int TB = DP > 128 ? 1024 / DP : NC == 1 || DP <= 32 ? 8 : 4, NBUF = 3;                // tokens per block, blocks resident
  static constexpr int VECS = NV * TB * DP, LOADS = VECS / 256, PER = (LOADS + 3) / 4;         // floats; direct loads of the workgroup and of a wave
  static constexpr int BLOCK = (VECS + TB * 256 / RG * NC + (GENERAL ? 0 : 2 * TB) + 3) / 4 * 4;
  static_assert(TB * DP % 256 == 0, "a direct load is 256 floats of one vector");
};

enum { ANY, FOURS, WHOLE };
template <int DR, int RG, int NC, bool GENERAL, int MODE>
__global__ __launch_bounds__(256) void delta_scan_kernel(vlm_delta_rule_args p) {
  extern __shared__ __align__(16) float smem[];
  using SS = ScanShape<DR, RG, NC, GENERAL>;
  constexpr int DP = SS::DP, TB = SS::TB, NBUF = SS::NBUF, VECS = SS::VECS, PER = SS::PER, BLOCK = SS::BLOCK;
  constexpr int CT = 256 / RG * NC, VL = (TB * CT + 255) / 256;
  constexpr int ISSUED = PER + VL + (GENERAL ? 0 : 1);               // direct loads of a wave and block
  const int seg = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * CT;
  const int D = p.D, Dv = p.Dv;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int rg = lane & (RG - 1), cl = (wave * (64 / RG) + lane / RG) * NC, col = c0 + cl, row0 = rg * DR;
  const int kh = h / (p.H / p.KH);
  const int t_begin = p.seg_start[seg], t_end = p.seg_start[seg + 1], blocks = (t_end - t_begin + TB - 1) / TB;
  const int slot = p.seg_slot[seg], pos0 = p.seg_pos0[seg];
  const auto vec = [&](int n) { return n == 0 ? p.kw : n == 1 || !GENERAL ? p.q : n == 2 ? p.kr : n == 3 ? p.w : p.b; };
  float* S = p.state + ((long)slot * p.H + h) * (long)D * Dv;
  float s[NC][DR];
  if constexpr (MODE == WHOLE) {
    typedef float pc_t __attribute__((ext_vector_type(NC)));
#pragma unroll
    for (int r = 0; r < DR; ++r) {
      pc_t x = {};
      if (pos0 > 0 && col < Dv) x = *reinterpret_cast<const pc_t*>(S + (long)(row0 + r) * Dv + col);
#pragma unroll
      for (int c = 0; c < NC; ++c) s[c][r] = x[c];
    }
  } else {
#pragma unroll
    for (int r = 0; r < DR; ++r)
#pragma unroll
      for (int c = 0; c < NC; ++c) s[c][r] = (pos0 > 0 && row0 + r < D && col + c < Dv) ? S[(long)(row0 + r) * Dv + col + c] : 0.f;
  }
  const auto row_of = [](int e) { return (e / 4 % RG * (DR / 4) + e / 4 / RG) * 4 + e % 4; };          // of element e of a vector in LDS
  const float* src[PER];                                             // where this lane's direct loads start
  if constexpr (MODE != ANY)
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int l = min(wave + 4 * u, SS::LOADS - 1);
      src[u] = vec(l / (TB * DP / 256)) + (long)kh * D + row_of((l * 256 + lane * 4) % DP);
    }
  const float* vsrc = p.v + (long)h * Dv;
  const float* gsrc = GENERAL ? nullptr : (lane & 1 ? p.beta : p.g) + h;
  const auto issue = [&](int i) {                                    // block i into its buffer (tokens past the end: the last one again)
    float* buf = smem + (i % NBUF) * BLOCK;
    const int t0 = t_begin + i * TB;
    if constexpr (MODE != ANY) {
#pragma unroll
      for (int u = 0; u < PER; ++u) {                                // (every load has a row below D, its first: none is left out by a wave)
        const int l = min(wave + 4 * u, SS::LOADS - 1), e = l * 256 + lane * 4, t = e / DP % TB;
        if (MODE == WHOLE || row_of(e % DP) < D) direct_load16(src[u] + (long)min(t0 + t, t_end - 1) * p.ldk, buf + l * 256);
      }
    } else {
#pragma unroll 4
      for (int base = wave * 64; base < VECS; base += 256) {
        const int f = base + lane, t = f / DP % TB, row = row_of(f % DP);
        if (row < D) direct_load4(vec(base / (TB * DP)) + (long)min(t0 + t, t_end - 1) * p.ldk + (long)kh * D + row, buf + base);
      }
    }
#pragma unroll
    for (int u = 0; u < VL; ++u) {
      const int base = ((wave + 4 * u) * 64) % (TB * CT < 64 ? 64 : TB * CT), f = base + lane;
      if (f < TB * CT) direct_load4(vsrc + (long)min(t0 + f / CT, t_end - 1) * p.ldv + min(c0 + f % CT, Dv - 1), buf + VECS + base);
    }
    if constexpr (!GENERAL)
      if (lane < 2 * TB) direct_load4(gsrc + (long)min(t0 + lane / 2, t_end - 1) * p.H, buf + VECS + TB * CT);
  };
  if constexpr (MODE != WHOLE) {
    for (int f = tid; f < NBUF * BLOCK; f += 256) smem[f] = 0.f;     // (rows past D stay zero)
    __syncthreads();
  }
  if (blocks > 0) issue(0);
  if (MODE != ANY && blocks > 1) issue(1);
  // (the state has to be waited for here: inside the loop that wait would be for the direct loads too)
#pragma unroll
  for (int r = 0; r < DR; ++r)
#pragma unroll
    for (int c = 0; c < NC; ++c) asm volatile("" : "+v"(s[c][r]));
  struct Token { f32x4_t k[DR / 4], q[DR / 4], u[DR / 4], w[DR / 4], b[DR / 4]; float v[NC], g, beta; };
  for (int i = 0; i < blocks; ++i) {
    if constexpr (MODE != ANY) {
      // (stores of read-outs may be among what is waited for; direct loads return in order)
      if (i + 1 < blocks) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(ISSUED) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();                                  // block i is there for every wave, and everybody is done with block i - 1
      if (i + 2 < blocks) issue(i + 2);
    } else {                                                         // (how many loads a wave has issued depends on D: all of them are waited for)
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      if (i + 1 < blocks) issue(i + 1);
    }
    const float* buf = smem + (i % NBUF) * BLOCK;
    const int t0 = t_begin + i * TB, nb = min(TB, t_end - t0);
    float mine[NC] = {};                                             // the read-outs of token rg of the block
    const auto load = [&](int t) {
      Token x;
      const f32x4_t* row = reinterpret_cast<const f32x4_t*>(buf + t * DP) + rg;
      constexpr int V = TB * DP / 4;
#pragma unroll
      for (int r = 0; r < DR / 4; ++r) {
        if constexpr (GENERAL) {
          x.u[r] = row[RG * r + 2 * V];
          x.w[r] = row[RG * r + 3 * V];
          x.b[r] = row[RG * r + 4 * V];
        }
        x.k[r] = row[RG * r];
        x.q[r] = row[RG * r + V];
      }
      if constexpr (!GENERAL) {
        x.g = buf[VECS + TB * CT + 2 * t];
        x.beta = buf[VECS + TB * CT + 2 * t + 1];
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) x.v[c] = buf[VECS + t * CT + cl + c];
      return x;
    };
    // one token; its read-out's partial sums stay in sum[NC ..] and are added up over the lanes together with the next token's dot products, whose
    // chain is what takes the time (a chain of its own for them: 1500 tokens 353 us)
    float sum[2 * NC];
    const auto token = [&](const Token& x, int t) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        if constexpr (!GENERAL)
#pragma unroll
          for (int r = 0; r < DR; ++r) s[c][r] *= x.g;
        sum[c] = row_dot<DR>(s[c], GENERAL ? x.u : x.k);
        if constexpr (GENERAL)
#pragma unroll
          for (int r = 0; r < DR; ++r) s[c][r] *= x.w[r / 4][r % 4];
      }
      group_sum<RG, 2 * NC>(sum);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        mine[c] = rg == t - 1 ? sum[NC + c] : mine[c];
        const float y = GENERAL ? x.v[c] : x.beta * (x.v[c] - sum[c]);
#pragma unroll
        for (int r = 0; r < DR; ++r) {
          if constexpr (GENERAL) s[c][r] = fmaf(-x.b[r / 4][r % 4], sum[c], s[c][r]);
          s[c][r] = fmaf(x.k[r / 4][r % 4], y, s[c][r]);
        }
        sum[NC + c] = row_dot<DR>(s[c], x.q);
      }
    };
#pragma unroll
    for (int c = 0; c < NC; ++c) sum[NC + c] = 0.f;
    if (nb == TB) {
      Token x = load(0);
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        const Token y = x;
        if (t + 1 < TB) x = load(t + 1);
        __builtin_amdgcn_sched_barrier(0);                           // (the next token's reads stay in front of this one's chain)
        token(y, t);
      }
    } else {
#pragma unroll 1
      for (int t = 0; t < nb; ++t) token(load(t), t);
    }
    float last[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) last[c] = sum[NC + c];
    group_sum<RG, NC>(last);
#pragma unroll
    for (int c = 0; c < NC; ++c) mine[c] = rg == nb - 1 ? last[c] : mine[c];
    if (rg < nb) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (col + c < Dv) p.raw[((long)(t0 + rg) * p.H + h) * Dv + col + c] = mine[c];
    }
  }
#pragma unroll
  for (int r = 0; r < DR; ++r) {
    if constexpr (MODE == WHOLE) {
      typedef float pc_t __attribute__((ext_vector_type(NC)));
      pc_t x;
#pragma unroll
      for (int c = 0; c < NC; ++c) x[c] = s[c][r];
      if (col < Dv) *reinterpret_cast<pc_t*>(S + (long)(row0 + r) * Dv + col) = x;
    } else {
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (row0 + r < D && col + c < Dv) S[(long)(row0 + r) * Dv + col + c] = s[c][r];
    }
  }
}

template <int DR, int RG, int NC, bool GENERAL>
int launch_scan(const vlm_delta_rule_args& a, int nseg, hipStream_t st) {
  using SS = ScanShape<DR, RG, NC, GENERAL>;
  constexpr int CT = 256 / RG * NC;
  constexpr size_t lds = (size_t)SS::NBUF * SS::BLOCK * sizeof(float);
  const uintptr_t ptrs = (uintptr_t)a.kw | (uintptr_t)a.q | (uintptr_t)a.state | (GENERAL ? (uintptr_t)a.kr | (uintptr_t)a.w | (uintptr_t)a.b : 0);
  const bool fours = a.D % 4 == 0 && a.ldk % 4 == 0 && ptrs % 16 == 0;           // the vectors' rows in whole aligned 16-byte pieces
  const bool whole = fours && a.D == SS::DP && a.Dv % NC == 0;
  const dim3 grid(nseg, a.H, (a.Dv + CT - 1) / CT), block(256);
  static_assert(lds <= 64 * 1024, "");
  if (whole) hipLaunchKernelGGL((delta_scan_kernel<DR, RG, NC, GENERAL, WHOLE>), grid, block, lds, st, a);
  else if (fours) hipLaunchKernelGGL((delta_scan_kernel<DR, RG, NC, GENERAL, FOURS>), grid, block, lds, st, a);
  else hipLaunchKernelGGL((delta_scan_kernel<DR, RG, NC, GENERAL, ANY>), grid, block, lds, st, a);
  VLM_CHECK_LAUNCH();
  return VLM_OK;
}

// Which spread of the state (rows a lane, lanes a column, columns a lane; the results are the same bits in all of them).  Heads of 128: (4, 32, 1) keeps a token's
// chain shortest: 1500 tokens of 12 heads 265 us (general) and 240 us (gated), against 354 and 286 with (8, 16, 1), 409 and 380 with (4, 32, 2).  Segments of a few
// tokens move more state than they compute and take pieces of 32 bytes of a state row a wave: 32 sequences of one token, 28 heads: (4, 32, 4) 30 us,
// (4, 32, 1) 85.  With more workgroups than are resident at once the work counts, not the chain: fewer lanes save on sums over them, and the general form reads
// five vectors a token from LDS and shares them between columns.  us, sequences x tokens x heads (`groups`); "before": 16 rows a lane on 8 lanes, tokens behind a barrier:
//   gated 128    3 (1100 + 333 + 70) x 28 (1344)  before 625  (8, 16, 1) 232  (16, 8, 1) 310    4 x 200 x 28 (1792)   132   91   85     16 x 100 x 28 (7168)  153  153  136
//                32 x 40 x 12 (6144)                      59              60              54    16 x 60 x 12 (3072)    53   50   44     32 x 20 x 28 (14336)   76   75   75
//   general 128  3 (1100 + 333 + 70) x 28         before 868  (4, 32, 2) 355  (8, 16, 2) 445    4 x 200 x 28          174  141  126     16 x 100 x 28         221  234  186
//                32 x 40 x 12                             92              85              73    16 x 60 x 12           67   68   59     32 x 20 x 28          103  106   86
//   gated 64     3 (1100 + 333 + 70) x 28 (672)   before 452  (4, 16, 1) 155  (8, 8, 1) 189     8 x 300 x 28 (1792)   140   96   84     32 x 20 x 28 (7168)    32   35   28
//   gated 256    3 (1100 + 333 + 70) x 14 (1344)  before 1007 (8, 32, 1) 407  (16, 16, 1) 408   8 x 300 x 14 (3584)   387  454  362     16 x 100 x 14 (7168)  254  327  265
//                                                             (16, 16, 2) 572                                              424                                        248
//   general 256  3 (1100 + 333 + 70) x 14         before 1483 (8, 32, 2) 667  (16, 16, 2) 735   8 x 300 x 14          930  607  587     32 x 40 x 6 (6144)    148  159  134
// (A step whose sequences differ much in length waits for the longest one's chain, which the shapes for many workgroups lengthen: the host knows only how many
// tokens there are.)
template <bool GENERAL>
int run_scan(const vlm_delta_rule_args& a, int nseg, int ntok, hipStream_t st) {
  const bool few = ntok <= 16L * nseg;
  const long groups = (long)nseg * a.H * ((a.Dv + 7) / 8);           // workgroups of eight columns
  if (a.D <= 32) return launch_scan<4, 8, 1, GENERAL>(a, nseg, st);
  if (a.D <= 64) {
    if (few) return launch_scan<4, 16, 2, GENERAL>(a, nseg, st);
    return groups > 2048 ? launch_scan<8, 8, 1, GENERAL>(a, nseg, st) : launch_scan<4, 16, 1, GENERAL>(a, nseg, st);
  }
  if (a.D <= 128) {
    if (few) return launch_scan<4, 32, 4, GENERAL>(a, nseg, st);
    if (groups <= 1024) return launch_scan<4, 32, 1, GENERAL>(a, nseg, st);
    if constexpr (GENERAL) return groups > 2048 ? launch_scan<8, 16, 2, true>(a, nseg, st) : launch_scan<4, 32, 2, true>(a, nseg, st);
    else return groups > 4096 ? launch_scan<16, 8, 1, false>(a, nseg, st) : launch_scan<8, 16, 1, false>(a, nseg, st);
  }
  if (a.D <= 256) {
    if (few) return launch_scan<8, 32, 4, GENERAL>(a, nseg, st);
    if (groups <= (GENERAL ? 512 : 1024)) return launch_scan<8, 32, 1, GENERAL>(a, nseg, st);
    if (groups > (GENERAL ? 2048 : 4096)) return launch_scan<16, 16, 2, GENERAL>(a, nseg, st);
    if constexpr (GENERAL) return launch_scan<8, 32, 2, true>(a, nseg, st);
    else return launch_scan<16, 16, 1, false>(a, nseg, st);
  }
  if (a.D <= 512) return few ? launch_scan<16, 32, 2, GENERAL>(a, nseg, st) : launch_scan<16, 32, 1, GENERAL>(a, nseg, st);
  if (a.D <= 1024) return few ? launch_scan<32, 32, 2, GENERAL>(a, nseg, st) : launch_scan<32, 32, 1, GENERAL>(a, nseg, st);
  return VLM_ERR_SHAPE;
}

}  // namespace

extern "C" int vlm_delta_prep_general(const vlm_delta_prep_general_args* a, int ntok, int dtype, void* stream) {
  if (!a || ntok < 0) return VLM_ERR_ARG;
  if (!a->r || !a->k || !a->v_in || !a->a || !a->a_bias || !a->low || !a->w2 || !a->w0 || !a->q || !a->kw || !a->kr || !a->v || !a->w ||
      !a->b || a->H <= 0 || a->D <= 0 || a->R <= 0 || a->ld < (long)a->H * a->D || a->ld_low < a->R)
    return VLM_ERR_ARG;
  if (ntok == 0) return VLM_OK;
  if (a->H > 65535 || a->R > 8192) return VLM_ERR_SHAPE;
  hipStream_t st = (hipStream_t)stream;
  const size_t lds = (size_t)a->R * sizeof(float);
  if (dtype) hipLaunchKernelGGL(delta_prep_general_kernel<float>, dim3(ntok, a->H), dim3(64), lds, st, *a);
  else hipLaunchKernelGGL(delta_prep_general_kernel<bf16_t>, dim3(ntok, a->H), dim3(64), lds, st, *a);
  VLM_CHECK_LAUNCH();
  return VLM_OK;
}

extern "C" int vlm_delta_prep_gated(const vlm_delta_prep_gated_args* a, int nseg, int ntok, int dtype, void* stream) {
  if (!a || nseg < 0 || ntok < 0) return VLM_ERR_ARG;
  if (!a->q_in || !a->k_in || !a->v_in || !a->q_conv || !a->k_conv || !a->v_conv || !a->b_in || !a->a_in || !a->A_log || !a->dt_bias ||
      !a->q || !a->k || !a->v || !a->beta || !a->g || !a->seg_start || !a->seg_slot || !a->seg_pos0 || a->H <= 0 || a->KH <= 0 ||
      a->H % a->KH || a->D <= 0 || a->Dv <= 0 || a->taps < 1 || (a->taps > 1 && !a->conv_state))
    return VLM_ERR_ARG;
  if (nseg == 0 || ntok == 0) return VLM_OK;
  const long Cn = 2L * a->KH * a->D + (long)a->H * a->Dv;
  if (Cn * sizeof(float) > 48 * 1024) return VLM_ERR_SHAPE;
  hipStream_t st = (hipStream_t)stream;
  const size_t lds = (size_t)Cn * sizeof(float);
  const unsigned cy = (unsigned)((Cn + 255) / 256 < 64 ? (Cn + 255) / 256 : 64);
  if (dtype) {
    hipLaunchKernelGGL(delta_prep_gated_kernel<float>, dim3(ntok), dim3(256), lds, st, *a, nseg);
    VLM_CHECK_LAUNCH();
    if (a->taps > 1) hipLaunchKernelGGL(delta_conv_state_kernel<float>, dim3(nseg, cy), dim3(256), 0, st, *a);
  } else {
    hipLaunchKernelGGL(delta_prep_gated_kernel<bf16_t>, dim3(ntok), dim3(256), lds, st, *a, nseg);
    VLM_CHECK_LAUNCH();
    if (a->taps > 1) hipLaunchKernelGGL(delta_conv_state_kernel<bf16_t>, dim3(nseg, cy), dim3(256), 0, st, *a);
  }
  VLM_CHECK_LAUNCH();
  return VLM_OK;
}

extern "C" int vlm_delta_rule(const vlm_delta_rule_args* a, int nseg, int ntok, int dtype, void* stream) {
  if (!a || nseg < 0 || ntok < 0) return VLM_ERR_ARG;
  if (!a->q || !a->kw || !a->v || !a->state || !a->raw || !a->gate || !a->out || !a->seg_start || !a->seg_slot || !a->seg_pos0)
    return VLM_ERR_ARG;
  if (a->H <= 0 || a->KH <= 0 || a->H % a->KH || a->D <= 0 || a->Dv <= 0) return VLM_ERR_ARG;
  if (a->mode == 1 ? (!a->kr || !a->w || !a->b) : (a->mode != 0 || !a->beta || !a->g)) return VLM_ERR_ARG;
  if (a->ldk < (long)a->KH * a->D || a->ldv < (long)a->H * a->Dv || a->ldg < (long)a->H * a->Dv || a->ldo < (long)a->H * a->Dv)
    return VLM_ERR_ARG;
  if (nseg == 0 || ntok == 0) return VLM_OK;
  if (nseg > 65535 * 16 || a->H > 65535) return VLM_ERR_SHAPE;
  hipStream_t st = (hipStream_t)stream;
  const int rc = a->mode == 1 ? run_scan<true>(*a, nseg, ntok, st) : run_scan<false>(*a, nseg, ntok, st);
  if (rc != VLM_OK) return rc;
  if (dtype)
    hipLaunchKernelGGL((recurrence_finish_kernel<float, false>), dim3(ntok, a->H), dim3(64), 0, st, a->raw, a->H, a->Dv,
                       (const float*)nullptr, a->eps, (const float*)a->gate, a->ldg, (const float*)a->normw, a->gate_act,
                       (float*)a->out, a->ldo);
  else
    hipLaunchKernelGGL((recurrence_finish_kernel<bf16_t, false>), dim3(ntok, a->H), dim3(64), 0, st, a->raw, a->H, a->Dv,
                       (const float*)nullptr, a->eps, (const bf16_t*)a->gate, a->ldg, (const bf16_t*)a->normw, a->gate_act,
                       (bf16_t*)a->out, a->ldo);
  VLM_CHECK_LAUNCH();
  return VLM_OK;
}
