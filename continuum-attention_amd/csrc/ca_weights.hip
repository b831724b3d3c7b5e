// Weight-materialising CA kernels: exact weights W (and their score VJP) from
// a materialised block of scores.  These are the row kernels behind the
// reference's ext.forward(scores, start) -> [W, stats] and
// ext.backward_fused(scores, gw, start) -> [W, dS]
// (cuda/continuum_attention.py:136-163, 230-293, 538-554, 578-590), used for
// weight-level diagnostics and for continuous_attention_weights(logits)
// (architecture.py:65-105) on the GPU.  The fused operator kernels never
// materialise W; these do, so they are HBM-bound row passes.
//
// Layout: scores, grad_weights, weights and grad_scores are [rows][K] fp32,
// rows = BH * Q, row r is query start + (r % Q) of slice r / Q and sees keys
// 0 .. start + r % Q (the host checks start + Q <= K).  stats is
// [rows][2] = (row max m, 1/Z) in natural units, as the reference's.
//
// One wave per row, four rows per 256-thread work group.  Rows of 65 to 2048
// keys run in ca_weights_reg_kernel (below), others here: lane l of step t
// owns key j = 64 t + l and evaluates the segment (j, j+1) once: its left
// share stays with key j and its right share moves to key j+1 with one lane
// shift.  Scores are read coalesced; neighbours come from lane shuffles (the
// next step's first score is prefetched for lane 63).  Three passes over the
// row (max; Z and, for the VJP, sum_j w_j gw_j; weights / gradients), so the
// row is read from HBM once and re-read from cache.
#include "ca_common.h"
#include "ca_kernels.h"

namespace ca {

namespace {

// Score (or weight gradient) of key j, or `fill` past the visible prefix.
// Invisible scores read as the row max, so every exponent stays finite; their
// terms are masked.
__device__ __forceinline__ float load_or(const float* p, int j, int n, float fill) {
  return j < n ? p[j] : fill;
}

}  // namespace

template <bool kBwd>
__global__ __launch_bounds__(256) void ca_weights_rows_kernel(
    const float* __restrict__ scores, const float* __restrict__ gw, float* __restrict__ W,
    float* __restrict__ dS, float* __restrict__ stats, int rows, int Q, int K, int start) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;  // whole wave; no work-group barrier below
  const int query = start + row % Q;
  const int nvis = query + 1;  // keys 0 .. query
  const size_t off = (size_t)row * K;
  const float* s = scores + off;
  const float* g = kBwd ? gw + off : nullptr;

  // pass 1: row max over the visible keys
  float m = kNegBig;
  for (int j = lane; j < nvis; j += 64) m = fmaxf(m, s[j]);
  m = wave_max(m);

  // Segment (j, j+1) of one step: shares L (to j) and R (to j+1), and the
  // endpoint weights p_j, p_{j+1}.
  auto step_shares = [&](int j0, float cur, float nxt, float& pl, float& L, float& R) {
    const int j = j0 + lane;
    float sr = __shfl_down(cur, 1);
    const float first_next = __shfl(nxt, 0);
    if (lane == 63) sr = first_next;
    pl = fast_exp2((cur - m) * kLog2e);
    const float pr = fast_exp2((sr - m) * kLog2e);
    seg_shares_x(sr - cur, pl, pr, L, R);
    const bool seg_vis = j + 1 < nvis;
    L = seg_vis ? L : 0.f;
    R = seg_vis ? R : 0.f;
  };

  // pass 2: Z = sum_j w_j and (VJP) P = sum_j w_j gw_j
  float z = 0.f, pg = 0.f;
  {
    float cur = load_or(s, lane, nvis, m);
    float carry = 0.f;  // right share arriving at key j0 from segment (j0-1, j0)
    for (int j0 = 0; j0 < nvis; j0 += 64) {
      const int j = j0 + lane;
      const float nxt = load_or(s, j + 64, nvis, m);
      float pl, L, R;
      step_shares(j0, cur, nxt, pl, L, R);
      float rin = __shfl_up(R, 1);
      const float last_r = __shfl(R, 63);
      if (lane == 0) rin = carry;
      carry = last_r;
      float w = L + rin + ((j == 0) ? 0.5f * pl : 0.f) + ((j == query) ? 0.5f * pl : 0.f);
      w = (j < nvis) ? w : 0.f;
      z += w;
      if (kBwd) pg = fmaf(w, load_or(g, j, nvis, 0.f), pg);
      cur = nxt;
    }
  }
  z = wave_sum(z);
  const float inv_z = 1.0f / z;
  const float dmean = kBwd ? wave_sum(pg) * inv_z : 0.f;  // D = sum_j W_j gw_j

  // pass 3: normalised weights and (VJP) dS
  {
    float cur = load_or(s, lane, nvis, m);
    float gcur = kBwd ? (load_or(g, lane, nvis, 0.f) - dmean) * inv_z : 0.f;
    float carry = 0.f, dcarry = 0.f;
    for (int j0 = 0; j0 < nvis; j0 += 64) {
      const int j = j0 + lane;
      const float nxt = load_or(s, j + 64, nvis, m);
      float pl, L, R;
      if (!kBwd) {
        step_shares(j0, cur, nxt, pl, L, R);
      } else {
        // centred, 1/Z-scaled weight gradient of the right key
        const float gnxt = (load_or(g, j + 64, nvis, 0.f) - dmean) * inv_z;
        float gr = __shfl_down(gcur, 1);
        const float gfirst = __shfl(gnxt, 0);
        if (lane == 63) gr = gfirst;
        float sr = __shfl_down(cur, 1);
        const float first_next = __shfl(nxt, 0);
        if (lane == 63) sr = first_next;
        pl = fast_exp2((cur - m) * kLog2e);
        const float pr = fast_exp2((sr - m) * kLog2e);
        float dL, dR;
        seg_shares_grad_x(sr - cur, pl, pr, gcur, gr, L, R, dL, dR);
        const bool seg_vis = j + 1 < nvis;
        L = seg_vis ? L : 0.f;
        R = seg_vis ? R : 0.f;
        dL = seg_vis ? dL : 0.f;
        dR = seg_vis ? dR : 0.f;
        float din = __shfl_up(dR, 1);
        const float last_d = __shfl(dR, 63);
        if (lane == 0) din = dcarry;
        dcarry = last_d;
        const float caps = ((j == 0) ? 0.5f : 0.f) + ((j == query) ? 0.5f : 0.f);
        const float ds = fmaf(caps * pl, gcur, dL + din);
        if (j < nvis) dS[off + j] = ds;
        gcur = gnxt;
      }
      float rin = __shfl_up(R, 1);
      const float last_r = __shfl(R, 63);
      if (lane == 0) rin = carry;
      carry = last_r;
      const float w = L + rin + ((j == 0) ? 0.5f * pl : 0.f) + ((j == query) ? 0.5f * pl : 0.f);
      if (j < nvis && W) W[off + j] = w * inv_z;
      cur = nxt;
    }
  }
  // future keys: exact zeros
  for (int j = nvis + lane; j < K; j += 64) {
    if (W) W[off + j] = 0.f;
    if (kBwd) dS[off + j] = 0.f;
  }
  if (!kBwd && lane == 0) {
    stats[2 * (size_t)row + 0] = m;
    stats[2 * (size_t)row + 1] = inv_z;
  }
}

// Rows of up to 2048 keys, held in registers: the row is read once, every
// segment is evaluated once, and W (and dS) is written once.  Lane l of chunk
// c holds keys 256c + 4l .. +3, so loads and stores are 16 bytes per lane (VEC:
// rows 16-byte aligned) and three of four segments join keys of one lane.
// The score gradient is linear in the weight gradient g, and a constant g has
// gradient g w_j: with g taken relative to the row's plain mean (so that
// the terms stay small), dS_j = (dS_j(g) - D w_j) / Z needs no second
// evaluation once Z and D = sum_j w_j g_j / Z are known.
// Memory-bound: at 64 score matrices of [512, 512] the three-pass kernel above
// takes 41.5 us forward and 51.9 us backward (HIP events, with their overhead:
// 48.5 and 60.0), this one 26.0 and 35.5 (100 and 134 MB: 3.9 and 3.8 TB/s);
// rows 16-byte misaligned (K = 1023) 42.6 -> 34.3 and 53.9 -> 40.2 us.  Rows
// of at most kRowShort keys, which would leave three quarters of the lanes
// idle, stay with the three-pass kernel (one key per lane; at 256 matrices of
// [64, 64] backward 12.2 against 14.1 us), and so do rows past 2048 keys.  From
// 65 keys on, where the three-pass kernel needs a second step, this one is the
// faster: 2^26 scores in rows of 65 keys 391 / 489 -> 374 / 481 us (three-pass /
// this one, forward / backward), 96 keys 310 / 389 -> 265 / 322, 128 keys
// 296 / 391 -> 208 / 255, 2048 keys 176 / 241 -> 76 / 114.
constexpr int kRowRegChunk = 256;
constexpr int kRowShort = 64;
template <bool kBwd, int NC, bool VEC>
__global__ __launch_bounds__(256) void ca_weights_reg_kernel(
    const float* __restrict__ scores, const float* __restrict__ gw, float* __restrict__ W,
    float* __restrict__ dS, float* __restrict__ stats, int rows, int Q, int K, int start) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;  // whole wave; no work-group barrier below
  const int query = start + row % Q;
  const size_t off = (size_t)row * K;

  // visible values of keys j0 .. j0 + 3 (invisible ones: 0)
  auto load4 = [&](const float* base, int j0, float (&v)[4]) {
    if (VEC) {
      f32x4 t = {0.f, 0.f, 0.f, 0.f};
      if (j0 <= query) t = *reinterpret_cast<const f32x4*>(base + off + j0);  // K % 4 == 0
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = j0 + e <= query ? t[e] : 0.f;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = j0 + e <= query ? base[off + j0 + e] : 0.f;
    }
  };
  auto store4 = [&](float* base, int j0, const float (&v)[4]) {
    if (VEC) {
      if (j0 < K) *reinterpret_cast<f32x4*>(base + off + j0) = f32x4{v[0], v[1], v[2], v[3]};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (j0 + e < K) base[off + j0 + e] = v[e];
    }
  };

  float x[NC][4], g[kBwd ? NC : 1][4];
  float m = kNegBig, gsum = 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int j0 = kRowRegChunk * c + 4 * lane;
    load4(scores, j0, x[c]);
    if (kBwd) load4(gw, j0, g[c]);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int j0 = kRowRegChunk * c + 4 * lane;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (j0 + e <= query) m = fmaxf(m, x[c][e]);
      if (kBwd) gsum += g[c][e];
    }
  }
  m = wave_max(m);
  const float gref = kBwd ? wave_sum(gsum) / (float)(query + 1) : 0.f;

  // 4 w (over x) and, for the VJP, 4 dS of g - gref (over g); z = 4 Z
  float z = 0.f, pg = 0.f, carry = 0.f, dcarry = 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (kRowRegChunk * c > query) break;  // the whole wave: no visible key here
    const int j0 = kRowRegChunk * c + 4 * lane;
    // this lane's four scores, then the next key's
    float s[5], gg[5], p[5];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[e] = j0 + e <= query ? x[c][e] : m;
      p[e] = fast_exp2((s[e] - m) * kLog2e);
      if (kBwd) gg[e] = j0 + e <= query ? g[c][e] - gref : 0.f;
    }
    float s_next = m, g_next = 0.f;  // first key of the next chunk
    if (c + 1 < NC) {
      const int jn = kRowRegChunk * (c + 1);
      const float t = __shfl(x[c + 1][0], 0);
      s_next = jn <= query ? t : m;
      if (kBwd) {
        const float u = __shfl(g[c + 1][0], 0);
        g_next = jn <= query ? u - gref : 0.f;
      }
    }
    s[4] = __shfl_down(s[0], 1);
    if (lane == 63) s[4] = s_next;
    p[4] = fast_exp2((s[4] - m) * kLog2e);
    if (kBwd) {
      gg[4] = __shfl_down(gg[0], 1);
      if (lane == 63) gg[4] = g_next;
    }
    float L[4], R[4], dL[4], dR[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool vis = j0 + e < query;  // segment (j, j+1): its right key is visible
      if (kBwd) {
        seg_shares_grad_h(0.5f * (s[e + 1] - s[e]), p[e], p[e + 1], gg[e], gg[e + 1], L[e], R[e],
                          dL[e], dR[e]);
        dL[e] = vis ? dL[e] : 0.f;
        dR[e] = vis ? dR[e] : 0.f;
      } else {
        seg_shares_h(0.5f * (s[e + 1] - s[e]), p[e], p[e + 1], L[e], R[e]);
      }
      L[e] = vis ? L[e] : 0.f;
      R[e] = vis ? R[e] : 0.f;
    }
    float rin = __shfl_up(R[3], 1);
    const float rlast = __shfl(R[3], 63);
    if (lane == 0) rin = carry;
    carry = rlast;
    float din = 0.f;
    if (kBwd) {
      din = __shfl_up(dR[3], 1);
      const float dlast = __shfl(dR[3], 63);
      if (lane == 0) din = dcarry;
      dcarry = dlast;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int j = j0 + e;
      const float cap = ((j == 0) ? 2.0f : 0.f) + ((j == query) ? 2.0f : 0.f);
      float w = L[e] + (e ? R[e - 1] : rin) + cap * p[e];
      w = j <= query ? w : 0.f;
      z += w;
      x[c][e] = w;
      if (kBwd) {
        pg = fmaf(w, gg[e], pg);
        const float ds = fmaf(cap * p[e], gg[e], dL[e] + (e ? dR[e - 1] : din));
        g[c][e] = j <= query ? ds : 0.f;
      }
    }
  }
  z = wave_sum(z);
  const float inv_z = 1.0f / z;
  const float dmean = kBwd ? wave_sum(pg) * inv_z : 0.f;  // relative to gref

  // normalised weights and gradients; future keys: exact zeros
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int j0 = kRowRegChunk * c + 4 * lane;
    float w[4], d[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool vis = j0 + e <= query;
      w[e] = vis ? x[c][e] * inv_z : 0.f;
      if (kBwd) d[e] = vis ? fmaf(-dmean, x[c][e], g[c][e]) * inv_z : 0.f;
    }
    if (W) store4(W, j0, w);
    if (kBwd) store4(dS, j0, d);
  }
  if (!kBwd && lane == 0) {
    stats[2 * (size_t)row + 0] = m;
    stats[2 * (size_t)row + 1] = 4.0f * inv_z;
  }
}

namespace {

// The register kernel for rows it holds (NC chunks of 256 keys), else the
// three-pass kernel.  16-byte accesses need rows and bases 16-byte aligned.
template <bool kBwd>
hipError_t launch_rows(const float* scores, const float* gw, float* W, float* dS, float* stats,
                       int BH, int Q, int K, int start, hipStream_t stream) {
  const int rows = BH * Q;
  const dim3 grid((rows + 3) / 4), block(256);
  auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  const bool vec = K % 4 == 0 && al(scores) && al(gw) && al(W) && al(dS);
#define CA_ROWS_REG(NC)                                                                        \
  if (K <= NC * kRowRegChunk) {                                                                \
    if (vec)                                                                                   \
      hipLaunchKernelGGL((ca_weights_reg_kernel<kBwd, NC, true>), grid, block, 0, stream, scores, gw, \
                         W, dS, stats, rows, Q, K, start);                                     \
    else                                                                                       \
      hipLaunchKernelGGL((ca_weights_reg_kernel<kBwd, NC, false>), grid, block, 0, stream, scores, \
                         gw, W, dS, stats, rows, Q, K, start);                                 \
    return hipGetLastError();                                                                  \
  }
  if (K > kRowShort) {
    CA_ROWS_REG(1)
    CA_ROWS_REG(2)
    CA_ROWS_REG(4)
    CA_ROWS_REG(8)
  }
#undef CA_ROWS_REG
  hipLaunchKernelGGL(ca_weights_rows_kernel<kBwd>, grid, block, 0, stream, scores, gw, W, dS, stats,
                     rows, Q, K, start);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_weights(const float* scores, float* weights, float* stats, int BH, int Q, int K,
                          int start, hipStream_t stream) {
  return launch_rows<false>(scores, nullptr, weights, nullptr, stats, BH, Q, K, start, stream);
}

hipError_t launch_weights_bwd(const float* scores, const float* grad_weights, float* weights,
                              float* grad_scores, int BH, int Q, int K, int start,
                              hipStream_t stream) {
  return launch_rows<true>(scores, grad_weights, weights, grad_scores, nullptr, BH, Q, K, start,
                           stream);
}

}  // namespace ca
