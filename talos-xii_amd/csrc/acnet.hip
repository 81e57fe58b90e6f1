// acnet.hip -- the reference actor-critic's PPO minibatch in one kernel (and one reduction).
//
// The network the reference trains (ActorCritic::new, src/ppo.rs:254-258; LuckTransformer::new,
// src/transformer.rs:48-69) is small: 44 k parameters, 6 k multiply-adds a token and 40 k a sample
// in the forward. As separate products its minibatch was 30 launches of mostly latency, and at
// 4096 x 16 tokens most of the time went into writing and reading the per-token activations and
// into attention rows that the loss never reads (only each sample's last token reaches the heads).
//
// Here a 512-thread workgroup takes up to 8 samples (at most 128 tokens), keeps every activation in
// LDS and walks the whole graph: embedding, RMSNorm, latent and rotary keys of every token, the
// last token's query, its attention in absorbed form (score = (W_uk_h q_c) . c_j + q_r . k_rj,
// o_h = (sum_j p_j c_j) W_uv_h: no key or value rows are formed), output projection, MLP, final
// norm, out_proj, heads, the clipped loss in f64, and back. Nothing per token or per sample is
// written to memory. The products run on v_mfma_f32_16x16x4f32: token products with 16 tokens as
// the tile rows (a wave a tile), sample products with the 8 samples as half a tile, the weight
// gradients with tokens or samples as k into accumulators that stay in registers over all of the
// workgroup's samples (at most 512 tokens or 256 samples: minibatch_grid); the gains' and the heads'
// gradients add in f64. At the end a workgroup writes its parameter gradients once as a partial
// row; acnet_reduce_kernel adds the rows in a fixed order in f64.
//
// Bound by the latency of its 28 dependent phases (LDS round trips and barriers, one workgroup per
// CU: 160 KB of LDS; about 93 k cycles a group of 8 samples x 16 tokens, the matrix pipe busy for a
// third of them; 256 samples leave three quarters of the CUs idle), then by the partial rows
// (181 KB a workgroup). One MI355X, minibatch forward + backward: 4096 x 16 tokens 849 -> 87 us,
// 256 ragged samples of up to 16 tokens 411 -> 39 us.
#include "acnet.hpp"

#include <algorithm>
#include <type_traits>

#include "plans.hpp"
#include "rowtile.hpp"

namespace talos {
namespace {

constexpr int D = 64, H = 4, LT = 32, RD = 16, HD = 16, VD = 16, F = 128, IN = 8;
constexpr int NK = LT + H * RD;  // a token's latent and rotary key columns
constexpr int T = 128;           // tokens of a workgroup's group of samples, at most
constexpr int GS = 8;            // samples of a group, at most
constexpr int NTHR = 512, NWV = NTHR / 64;
constexpr int MAXA = 8;
static_assert(MAXA == 8, "the loss sums over the first 8 lanes");
static_assert(NWV == GS && D == 64, "row phases: a wave a sample, a lane a feature");
static_assert(HD == 16 && VD == 16 && RD == 16 && LT == 32 && F == 16 * NWV, "tile counts");

// offsets of the flat parameters (talos_ppo_cfg's order)
constexpr int oWE = 0, oBE = oWE + IN * D, oG1 = oBE + D, oWDKV = oG1 + D, oWUK = oWDKV + D * LT,
              oWUV = oWUK + LT * D, oWQ = oWUV + LT * D, oWKR = oWQ + D * D, oWQR = oWKR + D * D, oWO = oWQR + D * D,
              oG2 = oWO + D * D, oW1 = oG2 + D, oB1 = oW1 + D * F, oW2 = oB1 + F, oB2 = oW2 + F * D, oGF = oB2 + D,
              oWOUT = oGF + D, oBOUT = oWOUT + D * D, oWA = oBOUT + D;
constexpr int kStats = 5;  // loss, kl, policy, value, entropy sums (ppo_heads_kernel's)

// LDS row pitches in floats. 68 and 100: float4 reads of 16 rows fall on 16 distinct bank groups,
// and rows 4 apart (the k order of the gradient products) are 16 banks apart.
constexpr int LX = D + 4, LC = NK + 4, LW = NK + 4, LS = IN + 1, LR = D + 4, LF = F + 4, LQ = 2 * D + 4;
constexpr int HP = LT + 4, LH = H * HP;  // per-head rows of 32

struct Smem {
  float W[D * LW];                  // [W_dkv | W_kr]
  float X[T * LX];                  // xn, later dL/dxn and dL/dh0
  float C[T * LC];                  // [c | k_r], later their gradients
  float St[T * LS];                 // states | 1
  float P[T * H], S[T * H], rs[T];  // probabilities, dL/dscore, rstd
  float We[(IN + 1) * D], g1[D];    // (row IN of We: its bias)
  float Q[GS * LQ];                 // [q_c | q_r]
  float QA[GS * LH];                // W_uk_h q_c; later the query path's dL/dxn
  float Z[GS * LH];                 // sum_j p_j c_j
  float xl[GS * LR], o[GS * LR], h2[GS * LR], n2[GS * LR];
  float last[GS * LR], ln[GS * LR], po[GS * LR], gpo[GS * LR];
  float u[GS * LF], a[GS * LF];
  float dz[GS * 16];     // dL/dlogits (columns 0 .. 7) | dL/dvalue (column 8) of each sample
  double st[GS * kStats];  // loss statistics of the waves' samples
  int len[GS], lrow[GS];
  float r2[GS], rf[GS];
};
static_assert(sizeof(Smem) <= 163840, "one workgroup's LDS");
static_assert(GS * LH <= 3 * GS * LR, "DQA overlays xl, o, h2");
static_assert(GS * LQ <= 2 * GS * LR, "DQ overlays po, gpo");
static_assert(GS * LH <= 2 * GS * LF, "DZ overlays u, a");
static_assert(T * H == GS * D, "S holds a row of D for each sample until the scores' gradients");
static_assert(2 * D <= LH, "the two halves of the query path's dL/dxn fit a QA row");

struct KArgs {
  int B, S, G, ngroups, A, relu;
  float eps, scale, clip_eps, cv, ce;
  int vec;  // 16-byte states rows
  int pitch, dpitch;  // floats and doubles of a partial row
  AcNetCall c;
  float* part;        // [workgroups][pitch], at the parameters' offsets
  double* dpart;      // [workgroups][dpitch]: dg1 | dg2 | dgf | the heads
  double* stat_part;  // [workgroups][kStats]
};
typedef double doublex4 __attribute__((ext_vector_type(4)));

// the lane's weights of a 16-column tile, column n: k = k0 + 16 g + 4 kq + u
template <int K, bool TRANS>
__device__ __forceinline__ void load_w(float (&w)[K / 4], const float* W, int ldw, int n, int kq, int k0 = 0) {
#pragma unroll
  for (int g = 0; g < K / 16; ++g)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = k0 + 16 * g + 4 * kq + u;
      w[4 * g + u] = W[TRANS ? n * ldw + k : k * ldw + n];
    }
}
// the 16-row tile of the GS sample rows X (rows past GS repeat) times the lane's weights
template <int K>
__device__ __forceinline__ rt_floatx4 mm_rows(const float* xrow, int kq, const float (&w)[K / 4]) {
  rt_floatx4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int g = 0; g < K / 16; ++g) {
    const float4 x = *reinterpret_cast<const float4*>(xrow + 16 * g + 4 * kq);
    rt_floatx4& acc = (g & 1) ? a1 : a0;
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x.x, w[4 * g], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y, w[4 * g + 1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x.z, w[4 * g + 2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w, w[4 * g + 3], acc, 0, 0, 0);
  }
  return a0 + a1;
}
// acc += X^T G over the GS samples: X, G point at the lane's column, rows ldx / ldg apart
__device__ __forceinline__ void mm_grad(rt_floatx4& acc, int kq, const float* X, int ldx, const float* G, int ldg) {
#pragma unroll
  for (int s = 0; s < GS / 4; ++s)
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(X[(4 * s + kq) * ldx], G[(4 * s + kq) * ldg], acc, 0, 0, 0);
}
// the lane's four rows of a sample tile: rows 4 kq + r < GS sit in the first two lane quarters
template <class Out>
__device__ __forceinline__ void put_rows(int kq, const rt_floatx4& v, Out out) {
  if (kq < GS / 4) {
#pragma unroll
    for (int r = 0; r < 4; ++r) out(4 * kq + r, v[r]);
  }
}
// orders LDS accesses of one wave's lanes (data shared inside the wave only)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}
// v of lane l (wave-uniform)
__device__ __forceinline__ float from_lane(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double from_lane(double v, int l) {
  const int2 x = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_readlane(x.x, l), __builtin_amdgcn_readlane(x.y, l)));
}
// the sum over the wave, in every lane: DPP moves inside 16 lanes and four lane reads instead of
// six dependent LDS-path shuffles
__device__ __forceinline__ float wave_total(float v) {
  v = group_sum<16>(v);
  return (from_lane(v, 0) + from_lane(v, 16)) + (from_lane(v, 32) + from_lane(v, 48));
}
// the sum / largest over aligned groups of 8 lanes in f64
template <int CTRL>
__device__ __forceinline__ double dpp64(double v) {
  const int2 x = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_update_dpp(0, x.x, CTRL, 0xF, 0xF, false),
                                              __builtin_amdgcn_update_dpp(0, x.y, CTRL, 0xF, 0xF, false)));
}
__device__ __forceinline__ double group8_sum(double v) {
  v += dpp64<0xB1>(v);
  v += dpp64<0x4E>(v);
  return v + dpp64<0x141>(v);
}
__device__ __forceinline__ double group8_max(double v) {
  v = fmax(v, dpp64<0xB1>(v));
  v = fmax(v, dpp64<0x4E>(v));
  return fmax(v, dpp64<0x141>(v));
}
// the neighbour lane's value (lane ^ 1)
__device__ __forceinline__ float pair_lane(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
}
__device__ __forceinline__ float group16_max(float v) {
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

template <bool BWD>
__global__ __launch_bounds__(NTHR) __attribute__((amdgpu_waves_per_eu(2, 2))) void acnet_kernel(KArgs k) {
  __shared__ __align__(16) Smem sm;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, i = lane & 15, kq = lane >> 4;
  const int S = k.S, A = k.A;
  const float* P = k.c.params;
  float* const DZ = sm.u;    // [GS][LH] after the tail
  float* const DQA = sm.xl;  // [GS][LH]
  float* const DQ = sm.po;   // [GS][LQ]: [dL/dq_c | dL/dq_r before its rotation]

  {
    constexpr int PER = D * NK / NTHR;
    float v[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {  // (NTHR / NK is no whole number: a thread's elements in any row)
      const int e = tid + q * NTHR, r = e / NK, c = e % NK;
      v[q] = P[c < LT ? oWDKV + r * LT + c : oWKR + r * D + c - LT];
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = tid + q * NTHR;
      sm.W[(e / NK) * LW + e % NK] = v[q];
    }
  }
  sm.We[tid] = P[oWE + tid];  // IN * D = NTHR
  if (tid < D) sm.We[IN * D + tid] = P[oBE + tid];
  if (tid < D) sm.g1[tid] = P[oG1 + tid];
  static_assert(IN * D == NTHR, "one embedding weight a thread");

  // gradient accumulators (tile t of a matrix on wave t % 8 unless said otherwise)
  const rt_floatx4 z4 = {0.f, 0.f, 0.f, 0.f};
  rt_floatx4 gK[3], gQ[4], gUK = z4, gUV = z4, gE = z4, gOut[2], gW2[4], gW1[4], gWo[2];
  float about = 0.f, ab2 = 0.f, ab1 = 0.f;
  // the gains' and the heads' gradients add in f64, as their kernels in the separate products do
  doublex4 gH = {0.0, 0.0, 0.0, 0.0};
  double ag1 = 0.0, agf = 0.0, ag2 = 0.0, abh = 0.0;
  if constexpr (BWD) {
#pragma unroll
    for (int q = 0; q < 3; ++q) gK[q] = z4;
#pragma unroll
    for (int q = 0; q < 4; ++q) gQ[q] = gW2[q] = gW1[q] = z4;
#pragma unroll
    for (int q = 0; q < 2; ++q) gOut[q] = gWo[q] = z4;
    for (int e = tid; e < GS * kStats; e += NTHR) sm.st[e] = 0.0;
  }
  // h0 = [states | 1] [We; be] of a 16-token tile, columns 16 c + i
  auto embed = [&](int tile, int i, int kq, rt_floatx4 (&h)[D / 16]) {
#pragma unroll
    for (int c = 0; c < D / 16; ++c) h[c] = z4;
#pragma unroll
    for (int s = 0; s < (IN + 4) / 4; ++s) {
      const int f = 4 * s + kq;  // (rows past the ones are zero on both sides)
      const float x = f <= IN ? sm.St[(16 * tile + i) * LS + f] : 0.f;
#pragma unroll
      for (int c = 0; c < D / 16; ++c)
        h[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, f <= IN ? sm.We[f * D + 16 * c + i] : 0.f, h[c], 0, 0, 0);
    }
  };
  lds_barrier();

  for (int grp = blockIdx.x; grp < k.ngroups; grp += gridDim.x) {
    // the weights of a pass are loaded a phase ahead of their use. The compiler must not see that
    // they and the lane's addresses are the same in every pass: it would keep all of them in
    // registers over the loop and spill 600 of them.
    int zero = 0;
    asm volatile("" : "+s"(zero));
    const float* P = k.c.params + zero;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, kq = lane >> 4;
    const int n4 = (w & 3) * 16 + i, kh = w >> 2;  // column of a 64-wide product, half of its k
    const int hd2 = w >> 1, hf = w & 1;            // head and half of a [heads x 32] product
    const int t4 = tid >> 2, part = tid & 3;       // token phases: four threads a token
    const int b0 = grp * k.G, ns = min(k.G, k.B - b0), nt = ns * S;
    const int ntile = (nt + 15) >> 4;                               // token tiles
    const int wpt = 4 * ntile <= NWV ? 4 : 2 * ntile <= NWV ? 2 : 1;  // waves a token tile
    float wq[16], wuk[4], wuv[8];
    load_w<64, false>(wq, P + (w < 4 ? oWQ : oWQR), D, n4, kq);
    // ---- embedding and RMSNorm1 of every token (tokens past nt: zero states, no weight anywhere)
    if (tid < GS) {
      int L = 0;
      if (tid < ns) {
        L = k.c.lens ? k.c.lens[b0 + tid] : S;
        L = L < 1 ? 1 : (L > S ? S : L);
      }
      sm.len[tid] = L;
      sm.lrow[tid] = L > 0 ? tid * S + L - 1 : 0;  // (samples past ns: any row that is written)
    }
    {
      float st[IN];
#pragma unroll
      for (int f = 0; f < IN; ++f) st[f] = 0.f;
      if (t4 < nt) {
        const float* src = k.c.states + ((long long)b0 * S + t4) * IN;
        if (k.vec) {
          const float4 x = *reinterpret_cast<const float4*>(src), y = *reinterpret_cast<const float4*>(src + 4);
          st[0] = x.x; st[1] = x.y; st[2] = x.z; st[3] = x.w;
          st[4] = y.x; st[5] = y.y; st[6] = y.z; st[7] = y.w;
        } else {
#pragma unroll
          for (int f = 0; f < IN; ++f) st[f] = src[f];
        }
      }
#pragma unroll
      for (int f = 0; f < IN; ++f)
        if ((f >> 1) == part) sm.St[t4 * LS + f] = st[f];
      if (part == 0) sm.St[t4 * LS + IN] = t4 < nt ? 1.f : 0.f;
    }
    lds_barrier();
    if (w < ntile) {
      rt_floatx4 h[D / 16];
      embed(w, i, kq, h);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < D / 16; ++c) ss = fmaf(h[c][r], h[c][r], ss);
        // rows past nt are zeros: rstd 0 there, as 1 / sqrt(0 + eps) is infinite for eps = 0 and the
        // products over whole tiles would take 0 * inf into every gradient of the token weights
        const int t = 16 * w + 4 * kq + r;
        const float rs0 = 1.0f / sqrtf(group_sum<16>(ss) / (float)D + k.eps), rs = t < nt ? rs0 : 0.f;
        if (i == 0) sm.rs[t] = rs;
#pragma unroll
        for (int c = 0; c < D / 16; ++c) sm.X[t * LX + 16 * c + i] = h[c][r] * rs * sm.g1[16 * c + i];
      }
    }
    lds_barrier();
    load_w<16, true>(wuk, P + oWUK + hd2 * HD, D, hf * 16 + i, kq);
    // ---- [c | k_r] of every token (RoPE on k_r), the last tokens' h0 and queries
    // one, two or four waves a token tile
    auto keys = [&](int tile, int c0, auto nc) {
      constexpr int NC = decltype(nc)::value;
      float cs[4], sn[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int pos = (16 * tile + 4 * kq + r) % S;
        cs[r] = k.c.rcos[pos * (RD / 2) + (i >> 1)];
        sn[r] = k.c.rsin[pos * (RD / 2) + (i >> 1)];
      }
      rt_floatx4 acc[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[c] = z4;
#pragma unroll
      for (int g = 0; g < D / 16; ++g) {
        const float4 x = *reinterpret_cast<const float4*>(sm.X + (16 * tile + i) * LX + 16 * g + 4 * kq);
        const float xv[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float* wr = sm.W + (16 * g + 4 * kq + u) * LW + 16 * c0 + i;
#pragma unroll
          for (int c = 0; c < NC; ++c)
            acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[u], wr[16 * c], acc[c], 0, 0, 0);
        }
      }
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = acc[c][r];
          if (c0 + c >= LT / 16) {  // (uniform) the pair (2j, 2j + 1) sits in neighbouring lanes
            const float other = pair_lane(v);
            v = (i & 1) ? fmaf(other, sn[r], v * cs[r]) : fmaf(v, cs[r], -other * sn[r]);
          }
          sm.C[(16 * tile + 4 * kq + r) * LC + 16 * (c0 + c) + i] = v;
        }
    };
    if (wpt == 1) {
      if (w < ntile) keys(w, 0, std::integral_constant<int, NK / 16>{});
    } else if (wpt == 2) {
      if (w < 2 * ntile) keys(w >> 1, 3 * (w & 1), std::integral_constant<int, 3>{});
    } else if (w < 4 * ntile && (w & 3) < 3) {
      keys(w >> 2, 2 * (w & 3), std::integral_constant<int, 2>{});
    }
    {
      float v = sm.We[IN * D + lane];
      const float* st = sm.St + sm.lrow[w] * LS;
#pragma unroll
      for (int f = 0; f < IN; ++f) v = fmaf(st[f], sm.We[f * D + lane], v);
      sm.xl[w * LR + lane] = v;
      rt_floatx4 q = mm_rows<64>(sm.X + sm.lrow[i & 7] * LX, kq, wq);
      if (w >= 4) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int pos = max(sm.len[(4 * kq + r) & 7], 1) - 1;
          const float cs = k.c.rcos[pos * (RD / 2) + (i >> 1)], sn = k.c.rsin[pos * (RD / 2) + (i >> 1)];
          const float other = pair_lane(q[r]);
          q[r] = (i & 1) ? fmaf(other, sn, q[r] * cs) : fmaf(q[r], cs, -other * sn);
        }
      }
      put_rows(kq, q, [&](int e, float x) { sm.Q[e * LQ + 16 * w + i] = x; });
    }
    lds_barrier();
    // ---- absorbed queries W_uk_h q_c
    put_rows(kq, mm_rows<16>(sm.Q + (i & 7) * LQ + hd2 * HD, kq, wuk),
             [&](int e, float x) { sm.QA[e * LH + hd2 * HP + hf * 16 + i] = x; });
    lds_barrier();
    // ---- scores: a thread a (token, head)
    const int te = min(t4 / S, GS - 1);  // the token's sample
    const bool tin = t4 < nt && t4 - te * S < sm.len[te];
    {
      const float* qa = sm.QA + te * LH + part * HP;
      const float* qr = sm.Q + te * LQ + D + part * RD;
      const float* c = sm.C + t4 * LC;
      float s0 = 0.f, s1 = 0.f;
      if (tin) {
#pragma unroll
        for (int q = 0; q < LT / 4; ++q) {
          const float4 x = *reinterpret_cast<const float4*>(qa + 4 * q), y = *reinterpret_cast<const float4*>(c + 4 * q);
          s0 = fmaf(x.x, y.x, fmaf(x.y, y.y, fmaf(x.z, y.z, fmaf(x.w, y.w, s0))));
        }
#pragma unroll
        for (int q = 0; q < RD / 4; ++q) {
          const float4 x = *reinterpret_cast<const float4*>(qr + 4 * q),
                       y = *reinterpret_cast<const float4*>(c + LT + part * RD + 4 * q);
          s1 = fmaf(x.x, y.x, fmaf(x.y, y.y, fmaf(x.z, y.z, fmaf(x.w, y.w, s1))));
        }
      }
      sm.P[t4 * H + part] = tin ? (s0 + s1) * k.scale : 0.f;
    }
    load_w<32, false>(wuv, P + oWUV + (w & 3) * VD, D, i, kq);
    float wo[8];
    load_w<32, false>(wo, P + oWO, D, n4, kq, 32 * kh);
    lds_barrier();
    // ---- softmax and z_h = sum_j p_j c_j: wave w sample w, 16 lanes a head
    const int slen = sm.len[w], srow = w * S;
    {
      float m = -INFINITY;
#pragma unroll 1
      for (int j = i; j < slen; j += 16) m = fmaxf(m, sm.P[(srow + j) * H + kq]);
      m = group16_max(m);
      float sum = 0.f;
#pragma unroll 1
      for (int j = i; j < slen; j += 16) sum += expf(sm.P[(srow + j) * H + kq] - m);
      sum = group_sum<16>(sum);
      const float inv = 1.0f / sum;
#pragma unroll 1
      for (int j = i; j < slen; j += 16) sm.P[(srow + j) * H + kq] = expf(sm.P[(srow + j) * H + kq] - m) * inv;
      wave_sync();
      float za = 0.f, zb = 0.f;
#pragma unroll 4
      for (int j = 0; j < slen; ++j) {
        const float p = sm.P[(srow + j) * H + kq];
        const float2 c = *reinterpret_cast<const float2*>(sm.C + (srow + j) * LC + 2 * i);
        za = fmaf(p, c.x, za);
        zb = fmaf(p, c.y, zb);
      }
      *reinterpret_cast<float2*>(sm.Z + w * LH + kq * HP + 2 * i) = make_float2(za, zb);
    }
    lds_barrier();
    // ---- o_h = z_h W_uv_h
    if (w < 4)
      put_rows(kq, mm_rows<32>(sm.Z + (i & 7) * LH + w * HP, kq, wuv), [&](int e, float x) { sm.o[e * LR + n4] = x; });
    const float g2 = P[oG2 + lane];
    float w1[16];
    load_w<64, false>(w1, P + oW1, F, 16 * w + i, kq);
    lds_barrier();
    // ---- h2 = x + o Wo (the two halves of k on wave pairs, added in the row phase), RMSNorm2
    {
      float* dst = kh ? sm.n2 : sm.h2;
      put_rows(kq, mm_rows<32>(sm.o + (i & 7) * LR + 32 * kh, kq, wo), [&](int e, float x) { dst[e * LR + n4] = x; });
    }
    lds_barrier();
    {
      const float x = sm.h2[w * LR + lane] + sm.n2[w * LR + lane] + sm.xl[w * LR + lane];
      const float r = 1.0f / sqrtf(wave_total(x * x) / (float)D + k.eps);
      sm.h2[w * LR + lane] = x;
      sm.n2[w * LR + lane] = x * r * g2;
      if (lane == 0) sm.r2[w] = r;
    }
    const float b1 = P[oB1 + 16 * w + i];
    float w2[16];
    load_w<64, false>(w2, P + oW2, D, n4, kq, 64 * kh);
    lds_barrier();
    // ---- a = act(xn2 W1 + b1); u = gelu' or the pre-activation
    put_rows(kq, mm_rows<64>(sm.n2 + (i & 7) * LR, kq, w1), [&](int e, float x) {
      const float v = x + b1;
      float act, aux;
      if (k.relu) {
        aux = v;
        act = fmaxf(v, 0.f);
      } else {
        act = gelu_fd(v, &aux);
      }
      sm.a[e * LF + 16 * w + i] = act;
      sm.u[e * LF + 16 * w + i] = aux;
    });
    const float gf = P[oGF + lane], b2 = P[oB2 + lane];
    float wout[8];
    load_w<32, false>(wout, P + oWOUT, D, n4, kq, 32 * kh);
    lds_barrier();
    // ---- last = h2 + a W2 + b2, the final norm
    {
      float* dst = kh ? sm.po : sm.last;
      put_rows(kq, mm_rows<64>(sm.a + (i & 7) * LF + 64 * kh, kq, w2), [&](int e, float x) { dst[e * LR + n4] = x; });
    }
    lds_barrier();
    {
      const float x = (sm.last[w * LR + lane] + sm.po[w * LR + lane] + b2) + sm.h2[w * LR + lane];
      const float r = 1.0f / sqrtf(wave_total(x * x) / (float)D + k.eps);
      sm.last[w * LR + lane] = x;
      sm.ln[w * LR + lane] = x * r * gf;
      if (lane == 0) sm.rf[w] = r;
    }
    lds_barrier();
    // ---- out_proj
    {
      float* dst = kh ? sm.gpo : sm.po;
      put_rows(kq, mm_rows<32>(sm.ln + (i & 7) * LR + 32 * kh, kq, wout), [&](int e, float x) { dst[e * LR + n4] = x; });
    }
    float wa[MAXA];
#pragma unroll
    for (int q = 0; q < MAXA; ++q) wa[q] = q < A ? P[oWA + lane * A + q] : 0.f;
    const float bout = P[oBOUT + lane], ba = lane < A ? P[oWA + D * A + lane] : 0.f, wc = P[oWA + D * A + A + lane],
                bc = P[oWA + D * A + A + D];
    float woutT[8], w2T[16];
    if constexpr (BWD) load_w<32, true>(woutT, P + oWOUT, D, n4, kq, 32 * kh);
    lds_barrier();
    // ---- heads and the clipped loss (ppo_heads_kernel's arithmetic): wave w sample w
    {
      const float pr = sm.po[w * LR + lane] + sm.gpo[w * LR + lane] + bout;
      float zk = 0.f;
#pragma unroll
      for (int q = 0; q < MAXA; ++q) {
        if (q < A) {
          const float t = wave_total(pr * wa[q]);
          if (lane == q) zk = t + ba;
        }
      }
      const float vf = wave_total(pr * wc) + bc;
      const int b = b0 + w;
      if constexpr (!BWD) {
        if (w < ns) {
          if (k.c.logits && lane < A) k.c.logits[(long long)b * A + lane] = zk;
          if (k.c.values && lane == 0) k.c.values[b] = vf;
        }
      } else {
        float dzf = 0.f, dvf = 0.f;
        if (w < ns) {  // wave-uniform
          const bool own = lane < A;
          double* st = sm.st + w * kStats;
          const double value = (double)vf;
          double mx = own ? (double)zk : -INFINITY;
          mx = group8_max(mx);  // (lanes past the first 8 hold nothing the loss reads)
          const double se = group8_sum(own ? exp((double)zk - mx) : 0.0);
          const double lse = log(se) + mx;
          const double lpk = (double)zk - lse, pk = own ? exp(lpk) : 0.0;
          const double ent = -group8_sum(own ? pk * lpk : 0.0);
          const int act = k.c.actions[b];
          if (act < 0 || act >= A) {
            if (lane == 0) st[0] = NAN;  // (the reference panics) no gradient from this sample
          } else {
            const double invB = 1.0 / (double)k.B;
            const double log_ratio = from_lane(lpk, act) - (double)k.c.old_logp[b];
            const double ratio = exp(log_ratio);
            const double ad = k.c.adv[b];
            const double lo = 1.0 - (double)k.clip_eps, hi = 1.0 + (double)k.clip_eps;
            const double s1 = ratio * ad, s2 = fmin(fmax(ratio, lo), hi) * ad;
            double pol, gr;
            if (s1 < s2) {
              pol = s1;
              gr = ad;
            } else {
              pol = s2;
              gr = (ratio >= lo && ratio <= hi) ? ad : 0.0;
            }
            const double vd = value - (double)k.c.ret[b];
            if (lane == 0) {
              st[0] += -pol + (double)k.cv * vd * vd - (double)k.ce * ent;
              st[1] += (ratio - 1.0) - log_ratio;
              st[2] += pol;
              st[3] += vd * vd;
              st[4] += ent;
            }
            if (own)
              dzf = (float)((-gr * ratio * ((lane == act ? 1.0 : 0.0) - pk) + (double)k.ce * pk * (lpk + ent)) * invB);
            dvf = (float)(2.0 * (double)k.cv * vd * invB);
          }
        }
        float g = dvf * wc;
#pragma unroll
        for (int q = 0; q < MAXA; ++q)
          if (q < A) g += from_lane(dzf, q) * wa[q];
        // the heads' weight gradients are a product like the others: rows pout, columns dz | dvalue
        sm.po[w * LR + lane] = pr;
        const float dzv = lane < MAXA ? dzf : lane == MAXA ? dvf : 0.f;
        if (lane < 16) sm.dz[w * 16 + lane] = dzv;
        abh += (double)dzv;
        about += g;
        sm.gpo[w * LR + lane] = g;
      }
    }
    if constexpr (BWD) {
      load_w<64, true>(w2T, P + oW2, D, 16 * w + i, kq);
      lds_barrier();
      // ---- dL/dlastn = g_pout Wout^T; dWout and the heads' weight gradients
      {
        float* dst = kh ? sm.xl : sm.S;
        const int ld = kh ? LR : D;
        put_rows(kq, mm_rows<32>(sm.gpo + (i & 7) * LR + 32 * kh, kq, woutT), [&](int e, float x) { dst[e * ld + n4] = x; });
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int t = w + 8 * q;
          mm_grad(gOut[q], kq, sm.ln + 16 * (t >> 2) + i, LR, sm.gpo + 16 * (t & 3) + i, LR);
        }
        if (w < 4) {
#pragma unroll
          for (int s = 0; s < GS / 4; ++s)
            gH = __builtin_amdgcn_mfma_f64_16x16x4f64((double)sm.po[(4 * s + kq) * LR + 16 * w + i],
                                                      (double)sm.dz[(4 * s + kq) * 16 + i], gH, 0, 0, 0);
        }
      }
      lds_barrier();
      // ---- the final norm's backward
      {
        const float dy = sm.S[w * D + lane] + sm.xl[w * LR + lane], r = sm.rf[w];
        const float xh = sm.last[w * LR + lane] * r;
        const float md = wave_total(dy * gf * xh) * (1.0f / (float)D);
        const float g = r * (dy * gf - xh * md);
        agf += (double)(dy * xh);
        ab2 += g;
        sm.last[w * LR + lane] = g;
      }
      float w1T[16];
      load_w<64, true>(w1T, P + oW1, F, n4, kq, 64 * kh);
      lds_barrier();
      // ---- g_u = (g_last W2^T) act'; dW2
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int t = w + 8 * q;
        mm_grad(gW2[q], kq, sm.a + 16 * (t >> 2) + i, LF, sm.last + 16 * (t & 3) + i, LR);
      }
      put_rows(kq, mm_rows<64>(sm.last + (i & 7) * LR, kq, w2T), [&](int e, float x) {
        const float aux = sm.u[e * LF + 16 * w + i];
        const float g = k.relu ? (aux > 0.f ? x : 0.f) : x * aux;
        ab1 += g;
        sm.u[e * LF + 16 * w + i] = g;
      });
      float woT[8];
      load_w<32, true>(woT, P + oWO, D, n4, kq, 32 * kh);
      lds_barrier();
      // ---- dL/dxn2 = g_u W1^T; dW1
      {
        float* dst = kh ? sm.xl : sm.po;
        put_rows(kq, mm_rows<64>(sm.u + (i & 7) * LF + 64 * kh, kq, w1T), [&](int e, float x) { dst[e * LR + n4] = x; });
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int t = w + 8 * q;
          mm_grad(gW1[q], kq, sm.n2 + 16 * (t >> 3) + i, LR, sm.u + 16 * (t & 7) + i, LF);
        }
      }
      lds_barrier();
      // ---- RMSNorm2's backward with the residual gradient: g_h2
      {
        const float dy = sm.po[w * LR + lane] + sm.xl[w * LR + lane], r = sm.r2[w];
        const float xh = sm.h2[w * LR + lane] * r;
        const float md = wave_total(dy * g2 * xh) * (1.0f / (float)D);
        ag2 += (double)(dy * xh);
        sm.last[w * LR + lane] += r * (dy * g2 - xh * md);
      }
      float wuvT[4];
      load_w<16, true>(wuvT, P + oWUV + hd2 * VD, D, hf * 16 + i, kq);
      lds_barrier();
      // ---- g_o = g_h2 Wo^T (its two halves of k in ln and n2); dWo
      {
        float* dst = kh ? sm.n2 : sm.ln;
        put_rows(kq, mm_rows<32>(sm.last + (i & 7) * LR + 32 * kh, kq, woT), [&](int e, float x) { dst[e * LR + n4] = x; });
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int t = w + 8 * q;
          mm_grad(gWo[q], kq, sm.o + 16 * (t >> 2) + i, LR, sm.last + 16 * (t & 3) + i, LR);
        }
      }
      lds_barrier();
      // ---- the halves added; dL/dz_h = W_uv_h g_o; dW_uv
      sm.ln[w * LR + lane] += sm.n2[w * LR + lane];
      lds_barrier();
      put_rows(kq, mm_rows<16>(sm.ln + (i & 7) * LR + hd2 * VD, kq, wuvT),
               [&](int e, float x) { DZ[e * LH + hd2 * HP + hf * 16 + i] = x; });
      mm_grad(gUV, kq, sm.Z + hd2 * HP + hf * 16 + i, LH, sm.ln + hd2 * VD + i, LR);
      float wukN[8];
      load_w<32, false>(wukN, P + oWUK + (w & 3) * HD, D, i, kq);
      lds_barrier();
      // ---- dL/dp of every (token, head)
      {
        const float* dz = DZ + te * LH + part * HP;
        const float* c = sm.C + t4 * LC;
        float s0 = 0.f;
        if (tin) {
#pragma unroll
          for (int q = 0; q < LT / 4; ++q) {
            const float4 x = *reinterpret_cast<const float4*>(dz + 4 * q), y = *reinterpret_cast<const float4*>(c + 4 * q);
            s0 = fmaf(x.x, y.x, fmaf(x.y, y.y, fmaf(x.z, y.z, fmaf(x.w, y.w, s0))));
          }
        }
        sm.S[t4 * H + part] = s0;
      }
      lds_barrier();
      // ---- dL/dscore, and the query's gradients: wave w sample w
      {
        float dot = 0.f;
#pragma unroll 1
        for (int j = i; j < slen; j += 16) dot = fmaf(sm.P[(srow + j) * H + kq], sm.S[(srow + j) * H + kq], dot);
        dot = group_sum<16>(dot);
#pragma unroll 1
        for (int j = i; j < slen; j += 16) {
          const int e = (srow + j) * H + kq;
          sm.S[e] = sm.P[e] * (sm.S[e] - dot) * k.scale;
        }
        wave_sync();
        float qa = 0.f, qb = 0.f, qr = 0.f;
#pragma unroll 4
        for (int j = 0; j < slen; ++j) {
          const float ds = sm.S[(srow + j) * H + kq];
          const float* c = sm.C + (srow + j) * LC;
          const float2 cc = *reinterpret_cast<const float2*>(c + 2 * i);
          qa = fmaf(ds, cc.x, qa);
          qb = fmaf(ds, cc.y, qb);
          qr = fmaf(ds, c[LT + kq * RD + i], qr);
        }
        *reinterpret_cast<float2*>(DQA + w * LH + kq * HP + 2 * i) = make_float2(qa, qb);
        const int pos = max(slen, 1) - 1;
        const float cs = k.c.rcos[pos * (RD / 2) + (i >> 1)], sn = k.c.rsin[pos * (RD / 2) + (i >> 1)];
        const float other = pair_lane(qr);
        DQ[w * LQ + D + kq * RD + i] = (i & 1) ? fmaf(qr, cs, -other * sn) : fmaf(qr, cs, other * sn);
      }
      float wqT[16];
      load_w<64, true>(wqT, P + (kh ? oWQR : oWQ), D, n4, kq);
      lds_barrier();
      // ---- dL/dq_c = dqa_h W_uk_h; [dL/dc | dL/dk_r before its rotation] over [c | k_r]
      if (w < 4)
        put_rows(kq, mm_rows<32>(DQA + (i & 7) * LH + w * HP, kq, wukN), [&](int e, float x) { DQ[e * LQ + 16 * w + i] = x; });
      if (t4 < 16 * ntile) {
        const float4 ds = *reinterpret_cast<const float4*>(sm.S + t4 * H), p = *reinterpret_cast<const float4*>(sm.P + t4 * H);
        const float dsv[4] = {ds.x, ds.y, ds.z, ds.w}, pv[4] = {p.x, p.y, p.z, p.w};
        float dc[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) dc[q] = 0.f;
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const float4 x = *reinterpret_cast<const float4*>(sm.QA + te * LH + h * HP + 8 * part + 4 * q),
                         y = *reinterpret_cast<const float4*>(DZ + te * LH + h * HP + 8 * part + 4 * q);
            dc[4 * q] = fmaf(dsv[h], x.x, fmaf(pv[h], y.x, dc[4 * q]));
            dc[4 * q + 1] = fmaf(dsv[h], x.y, fmaf(pv[h], y.y, dc[4 * q + 1]));
            dc[4 * q + 2] = fmaf(dsv[h], x.z, fmaf(pv[h], y.z, dc[4 * q + 2]));
            dc[4 * q + 3] = fmaf(dsv[h], x.w, fmaf(pv[h], y.w, dc[4 * q + 3]));
          }
        float* c = sm.C + t4 * LC;
        *reinterpret_cast<float4*>(c + 8 * part) = make_float4(dc[0], dc[1], dc[2], dc[3]);
        *reinterpret_cast<float4*>(c + 8 * part + 4) = make_float4(dc[4], dc[5], dc[6], dc[7]);
        const float dsh = dsv[part];
        const int pos = t4 % S;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4 x = *reinterpret_cast<const float4*>(sm.Q + te * LQ + D + part * RD + 4 * q);
          const float c0 = k.c.rcos[pos * (RD / 2) + 2 * q], s0 = k.c.rsin[pos * (RD / 2) + 2 * q];
          const float c1 = k.c.rcos[pos * (RD / 2) + 2 * q + 1], s1 = k.c.rsin[pos * (RD / 2) + 2 * q + 1];
          const float x0 = dsh * x.x, x1 = dsh * x.y, x2 = dsh * x.z, x3 = dsh * x.w;
          *reinterpret_cast<float4*>(c + LT + part * RD + 4 * q) =
              make_float4(fmaf(x0, c0, x1 * s0), fmaf(x1, c0, -x0 * s0), fmaf(x2, c1, x3 * s1), fmaf(x3, c1, -x2 * s1));
        }
      }
      lds_barrier();
      // ---- dW_dkv | dW_kr over the tokens (k order 16 b + 4 kq + s: conflict-free rows), dW_q |
      // dW_qr and dW_uk over the samples, and the query path's dL/dxn of the last tokens
      {  // tiles (w / 2, 3 (w % 2) + 0 .. 2)
        const float* x = sm.X + (4 * kq) * LX + 16 * (w >> 1) + i;
        const float* c = sm.C + (4 * kq) * LC + 48 * (w & 1) + i;
#pragma unroll 2
        for (int b = 0; b < ntile; ++b, x += 16 * LX, c += 16 * LC)
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int q = 0; q < 3; ++q)
              gK[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[s * LX], c[s * LC + 16 * q], gK[q], 0, 0, 0);
      }
      {
        float xl[4][2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const float* x = sm.X + sm.lrow[4 * s + kq] * LX + i;
#pragma unroll
          for (int q = 0; q < 4; ++q) xl[q][s] = x[16 * q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)  // rows 16 q .., columns 16 w ..
#pragma unroll
          for (int s = 0; s < 2; ++s)
            gQ[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(xl[q][s], DQ[(4 * s + kq) * LQ + 16 * w + i], gQ[q], 0, 0, 0);
      }
      mm_grad(gUK, kq, DQA + hd2 * HP + hf * 16 + i, LH, sm.Q + hd2 * HD + i, LQ);
      put_rows(kq, mm_rows<64>(DQ + (i & 7) * LQ + D * kh, kq, wqT), [&](int e, float x) { sm.QA[e * LH + D * kh + n4] = x; });
      lds_barrier();
      // ---- dL/dxn of the wave's 16 tokens and, on the accumulators, RMSNorm1's backward: dL/dh0 over
      // xn, the gain gradient's terms over the spent C rows
      if (w < ntile) {
        rt_floatx4 acc[D / 16], h[D / 16];
#pragma unroll
        for (int c = 0; c < D / 16; ++c) acc[c] = z4;
#pragma unroll
        for (int g = 0; g < NK / 16; ++g) {
          const float4 x = *reinterpret_cast<const float4*>(sm.C + (16 * w + i) * LC + 16 * g + 4 * kq);
          float4 b[D / 16];
#pragma unroll
          for (int c = 0; c < D / 16; ++c)
            b[c] = *reinterpret_cast<const float4*>(sm.W + (16 * c + i) * LW + 16 * g + 4 * kq);
#pragma unroll
          for (int c = 0; c < D / 16; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.x, b[c].x, acc[c], 0, 0, 0);
#pragma unroll
          for (int c = 0; c < D / 16; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y, b[c].y, acc[c], 0, 0, 0);
#pragma unroll
          for (int c = 0; c < D / 16; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.z, b[c].z, acc[c], 0, 0, 0);
#pragma unroll
          for (int c = 0; c < D / 16; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w, b[c].w, acc[c], 0, 0, 0);
        }
        embed(w, i, kq, h);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = 16 * w + 4 * kq + r, e = min(t / S, GS - 1);
          const bool is_last = t < nt && t == sm.lrow[e];
          const float rs = sm.rs[t];
          float dy[D / 16], xh[D / 16], dot = 0.f;
#pragma unroll
          for (int c = 0; c < D / 16; ++c) {
            const int f = 16 * c + i;
            dy[c] = acc[c][r];
            if (is_last) dy[c] += sm.QA[e * LH + f] + sm.QA[e * LH + D + f];
            xh[c] = h[c][r] * rs;
            sm.C[t * LC + f] = dy[c] * xh[c];
            dy[c] *= sm.g1[f];
            dot = fmaf(dy[c], xh[c], dot);
          }
          const float md = group_sum<16>(dot) * (1.0f / (float)D);
#pragma unroll
          for (int c = 0; c < D / 16; ++c) {
            const int f = 16 * c + i;
            float o = rs * (dy[c] - xh[c] * md);
            if (is_last) o += sm.last[e * LR + f];
            sm.X[t * LX + f] = o;
          }
        }
      }
      lds_barrier();
      // ---- dWe and dbe (the states' column of ones) as rows 0 .. 8 of a tile, dg1 as the sums over
      // each tile's 16 tokens (every row of g1t) added in f64; tokens of alternate tiles on the wave pairs
      for (int b = kh; b < ntile; b += 2) {
        rt_floatx4 g1t = z4;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int tok = 16 * b + 4 * kq + s;
          const float x = i <= IN ? sm.St[tok * LS + i] : 0.f;
          gE = __builtin_amdgcn_mfma_f32_16x16x4f32(x, sm.X[tok * LX + n4], gE, 0, 0, 0);
          g1t = __builtin_amdgcn_mfma_f32_16x16x4f32(1.f, sm.C[tok * LC + n4], g1t, 0, 0, 0);
        }
        ag1 += (double)g1t[0];
      }
    }
    lds_barrier();  // the next group's phases write what these read
  }
  if constexpr (BWD) {
    // ---- this workgroup's partial row
    const int n4 = (w & 3) * 16 + i, kh = w >> 2, hd2 = w >> 1, hf = w & 1;
    float* G = k.part + (long long)blockIdx.x * k.pitch;
    double* GD = k.dpart + (long long)blockIdx.x * k.dpitch;
    auto tile = [&](const rt_floatx4& v, int off, int ld, int m, int n) {
#pragma unroll
      for (int r = 0; r < 4; ++r) G[off + (16 * m + 4 * kq + r) * ld + 16 * n + i] = v[r];
    };
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int t = 3 * w + q, m = t / 6, n = t % 6;
      if (n < LT / 16)
        tile(gK[q], oWDKV, LT, m, n);
      else
        tile(gK[q], oWKR, D, m, n - LT / 16);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      tile(gQ[q], w < 4 ? oWQ : oWQR, D, q, w & 3);
      const int t = w + 8 * q;
      tile(gW2[q], oW2, D, t >> 2, t & 3);
      tile(gW1[q], oW1, F, t >> 3, t & 7);
    }
    tile(gUK, oWUK, D, hf, hd2);
    tile(gUV, oWUV, D, hf, hd2);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int t = w + 8 * q;
      tile(gOut[q], oWOUT, D, t >> 2, t & 3);
      tile(gWo[q], oWO, D, t >> 2, t & 3);
    }
    ab1 += __shfl_xor(ab1, 16, 64);  // (lane quarters 2 and 3 hold zeros)
    if (kq == 0) G[oB1 + 16 * w + i] = ab1;
    if (w < 4) {  // (register r of an f64 tile is row 4 r + kq)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int f = 16 * w + 4 * r + kq;
        if (i < A) GD[3 * D + f * A + i] = gH[r];
        if (i == MAXA) GD[3 * D + D * A + A + f] = gH[r];
      }
    }
    // sums over the waves (samples) through LDS, in f64, the two halves of the embedding's tile and of dg1
    double* R = reinterpret_cast<double*>(sm.C);           // [8 waves][5][64]
    float* E = sm.X;                                       // [2][16][64]
    double* E1 = reinterpret_cast<double*>(sm.X + 2 * 1024);  // [2][64]
    {
      double* r = R + w * 320 + lane;
      r[0] = agf;
      r[64] = ag2;
      r[128] = abh;
      r[192] = (double)about;
      r[256] = (double)ab2;
#pragma unroll
      for (int q = 0; q < 4; ++q) E[kh * 1024 + (4 * kq + q) * 64 + n4] = gE[q];
      if (kq == 0) E1[kh * 64 + n4] = ag1;
    }
    lds_barrier();
    if (tid < 320) {
      const int row = tid >> 6;
      double s = 0.0;
#pragma unroll
      for (int q = 0; q < NWV; ++q) s += R[q * 320 + tid];
      if (row < 2) GD[(row == 0 ? 2 * D : D) + lane] = s;
      else if (row > 2) G[(row == 3 ? oBOUT : oB2) + lane] = (float)s;
      else if (lane < A) GD[3 * D + D * A + lane] = s;
      else if (lane == MAXA) GD[3 * D + D * A + A + D] = s;
    }
    if (tid < D) GD[tid] = E1[tid] + E1[D + tid];
    for (int e = tid; e < (IN + 1) * D; e += NTHR) G[oWE + e] = E[e] + E[1024 + e];  // be follows we
    if (tid < kStats) {
      double s = 0.0;
#pragma unroll
      for (int q = 0; q < NWV; ++q) s += sm.st[q * kStats + tid];
      k.stat_part[blockIdx.x * kStats + tid] = s;
    }
  }
}

// dparams[e] = the workgroups' partial rows (f64 for the gains and the heads, fp32 for the rest)
// added in a fixed order in f64: 64 consecutive elements a workgroup, wave w the rows w, w + 4, ...
// in four accumulators; the last workgroup adds the loss statistics.
template <class V>
__device__ __forceinline__ double column_sum(int nwg, int w, const V* __restrict__ q, long long pitch) {
  const long long st = 4 * pitch;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  int g = w;
  q += w * pitch;
  for (; g + 12 < nwg; g += 16, q += 4 * st) {
    const V a = q[0], b = q[st], c = q[2 * st], d = q[3 * st];
    s0 += (double)a;
    s1 += (double)b;
    s2 += (double)c;
    s3 += (double)d;
  }
  for (; g < nwg; g += 4, q += st) s0 += (double)q[0];
  return (s0 + s1) + (s2 + s3);
}
__global__ __launch_bounds__(256) void acnet_reduce_kernel(int nwg, int nparams, int pitch, int dpitch, int B,
                                                           const float* __restrict__ part,
                                                           const double* __restrict__ dpart,
                                                           const double* __restrict__ stat_part,
                                                           float* __restrict__ dparams, float* __restrict__ loss,
                                                           double* __restrict__ stats, int stats_acc) {
  __shared__ double red[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (blockIdx.x == gridDim.x - 1) {
    // statistic w (and 4 by wave 0): its partials over the lanes, then across them
    for (int q = w; q < kStats; q += 4) {
      double s = 0.0;
      for (int g = lane; g < nwg; g += 64) s += stat_part[g * kStats + q];
      s = wave_sum(s);
      if (lane == 0) {
        if (q == 0) {
          if (loss) loss[0] = (float)(s / (double)B);
          if (stats) stats[4] = (stats_acc ? stats[4] : 0.0) + (double)B;
        } else if (stats) {
          stats[q - 1] = (stats_acc ? stats[q - 1] : 0.0) + s;
        }
      }
    }
    return;
  }
  // (the f64 sections start and end at multiples of 64)
  const int e0 = blockIdx.x * 64, e = e0 + lane;
  const int d0 = e0 == oG1 ? 0 : e0 == oG2 ? D : e0 == oGF ? 2 * D : e0 >= oWA ? 3 * D + e0 - oWA : -1;
  double sum = 0.0;
  if (e < nparams) sum = d0 < 0 ? column_sum(nwg, w, part + e, pitch) : column_sum(nwg, w, dpart + d0 + lane, dpitch);
  red[w][lane] = sum;
  __syncthreads();
  if (w == 0 && e < nparams) dparams[e] = (float)((red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]));
}

static_assert(oG1 % 64 == 0 && oG2 % 64 == 0 && oGF % 64 == 0 && oWA % 64 == 0 && D == 64, "acnet_reduce_kernel's sections");
constexpr int kPitch = oWA;  // a row's floats: the parameters before the heads
int dpart_pitch(int A) { return 3 * D + D * A + A + D + 1; }
size_t row_bytes(int A) { return (kStats + dpart_pitch(A)) * sizeof(double) + kPitch * sizeof(float); }

// Samples a workgroup takes at a time: as many as its 128 tokens hold (at most 8), fewer where the
// batch would then leave more than three quarters of the CUs without work. (Not all the way down
// to one sample a workgroup: every workgroup writes a whole partial row, and a group's time hardly
// depends on its samples. 256 samples of 16 tokens: 64 workgroups of 4 write 11 MB and take 39 us,
// 128 of 2 wrote 23 MB in 6 us of the 47 they took.)
int group_size(const talos_ppo_cfg& c, int n, int num_cu) {
  const int most = std::min(GS, T / c.seq);
  return std::max(1, std::min(most, n / std::max(1, num_cu / 4)));
}

// Workgroups (and partial rows) of a minibatch: one a CU, more where the fp32 accumulators of a
// workgroup would then run over more than 512 tokens or 256 samples (the runs of the separate
// products' split weight gradients and row chunks, whose partials are added in f64 as these are).
// A later round of workgroups takes what the earlier one left: nothing else changes, and a row
// more is 181 KB written for at least 170 us of work.
unsigned minibatch_grid(int ngroups, int group_tokens, int num_cu) {
  const int run = std::max(1, std::min(256 / GS, 512 / group_tokens));
  const long long rounds = ceil_div((size_t)ngroups, (size_t)run * num_cu);
  return (unsigned)std::min<long long>(ngroups, rounds * num_cu);
}

KArgs make_args(const talos_ppo_cfg& c, int num_cu, const AcNetCall& a, bool backward, unsigned* grid) {
  KArgs k{};
  k.B = a.n;
  k.S = c.seq;
  k.G = group_size(c, a.n, num_cu);
  k.ngroups = (int)ceil_div((size_t)a.n, k.G);
  k.A = c.n_actions;
  k.relu = c.activation != TALOS_ACT_GELU;
  k.eps = c.eps;
  k.scale = 1.0f / sqrtf((float)(HD + RD));
  k.clip_eps = c.clip_eps;
  k.cv = c.value_coef;
  k.ce = c.entropy_coef;
  k.vec = (reinterpret_cast<uintptr_t>(a.states) & 15) == 0;
  k.pitch = kPitch;
  k.dpitch = dpart_pitch(c.n_actions);
  k.c = a;
  *grid = backward ? minibatch_grid(k.ngroups, k.G * k.S, num_cu) : (unsigned)std::min(k.ngroups, num_cu);
  return k;
}

double flops_of(const talos_ppo_cfg& c, int n) {
  const double tok = (double)n * c.seq;
  return 2.0 * (tok * (IN * D + D * NK + 2.0 * H * (LT + RD)) + (double)n * (2.0 * D * D + 4.0 * D * D + 2.0 * D * F));
}

}  // namespace

bool acnet_supported(const talos_ppo_cfg& c) {
  return c.in_dim == IN && c.d_model == D && c.n_layers == 1 && c.n_heads == H && c.head_dim == HD && c.ffn_dim == F &&
         c.attention == TALOS_ATTN_MLA && c.kv_latent == LT && c.rope_dim == RD && c.v_dim == VD &&
         c.n_actions >= 1 && c.n_actions <= MAXA && c.seq >= 1 && c.seq <= T;
}

size_t acnet_ws_bytes(const talos_ppo_cfg& c, int num_cu) {
  // (a call of fewer samples has fewer rows: its groups are whole ones, or no more than CUs)
  const int most = std::min(GS, T / c.seq);
  const size_t rows = std::max((unsigned)num_cu, minibatch_grid((int)ceil_div((size_t)c.batch, most), most * c.seq, num_cu));
  return rows * row_bytes(c.n_actions);
}

int acnet_forward_launch(const talos_ppo_cfg& c, int num_cu, const AcNetCall& a, hipStream_t s) {
  unsigned grid;
  const KArgs k = make_args(c, num_cu, a, false, &grid);
  ProfScope ps(s, "acnet_kernel<false>", flops_of(c, a.n), 4.0 * a.n * (c.seq * IN + c.n_actions + 1.0));
  hipLaunchKernelGGL(acnet_kernel<false>, dim3(grid), dim3(NTHR), 0, s, k);
  return launch_status("acnet_kernel");
}

int acnet_minibatch_launch(const talos_ppo_cfg& c, int num_cu, const AcNetCall& a, hipStream_t s) {
  unsigned grid;
  KArgs k = make_args(c, num_cu, a, true, &grid);
  k.stat_part = a.ws;
  k.dpart = k.stat_part + (size_t)grid * kStats;
  k.part = reinterpret_cast<float*>(k.dpart + (size_t)grid * k.dpitch);
  const int np = oWA + D * c.n_actions + c.n_actions + D + 1;
  {
    ProfScope ps(s, "acnet_kernel<true>", 3.0 * flops_of(c, a.n), 4.0 * a.n * c.seq * IN + (double)grid * row_bytes(c.n_actions));
    hipLaunchKernelGGL(acnet_kernel<true>, dim3(grid), dim3(NTHR), 0, s, k);
    if (int rc = launch_status("acnet_kernel")) return rc;
  }
  ProfScope ps(s, "acnet_reduce_kernel", 0.0, (double)grid * row_bytes(c.n_actions) + 4.0 * np);
  hipLaunchKernelGGL(acnet_reduce_kernel, dim3(ceil_div((size_t)np, 64) + 1), dim3(256), 0, s, (int)grid, np, k.pitch,
                     k.dpitch, a.n, k.part, k.dpart, k.stat_part, a.dparams, a.loss, a.stats, a.stats_acc);
  return launch_status("acnet_reduce_kernel");
}

}  // namespace talos
