// S2 centroid scoring + S3 budget selection, S3c causal snapshot, and S4 the
// reverse index with the work list of the KV-outer prefill, for gfx950.
//
// Reference behaviour (pfnet-research/semantic-block-sparse-attention):
//   fused_select.py:1062-1247  _flat_scores_qtiled_kernel (score, LSE, mixture prob)
//   fused_select.py:604-646    _streaming_select_kernel RESIDENT (bisection, bitmask, qmask)
//   fused_select.py:806-919    theta_select_bitmask_flat (the contract)
//   fused_prefill.py:126-135   CausalSnapshot.advance
//   kv_outer.py:41-173, 254-329 build_reverse_index
#include "sbsa_common.h"

#include <type_traits>

namespace {

// ------------------------------------------------------------- S2 + S3 -----
// One block = QT queries x one KV head.  Rows of the score GEMM are
// (query, component) pairs, R = QT * G of them; the four waves split the
// clusters.  Scores live in LDS; each wave then selects for its queries.
// Bound by the chains of a wave's selection (reductions over the lanes, the bisection's
// ballots and counts), not by memory or the matrix units, so the row softmax is taken by
// the query's own wave, all components' reductions side by side, and its weights stay in
// registers: no second walk of the table and no block barrier before the selection.  One
// MI355X, a call with its bitmask fill: C = 256, 8192 queries of 16 heads on 4, D = 256
// 158 -> 117 us, C = 128 97 -> 76 us, C = 512 (8192 queries, 8 heads on 1, D = 128)
// 127 -> 87 us, C = 1024 (2048 queries, 4 on 4, D = 256) 91 -> 78 us.
struct SelectArgs {
  const bf16_t* vectors;   // [Q, Hq, D] routing vectors
  int64_t v_sq, v_sh;      // element strides
  const float* logmix;     // [Q, Hq] or null (uniform: 0)
  const bf16_t* codebooks; // [Hkv, 2, C, D/2]
  const int32_t* sizes;    // sizes[b * s_nb + h * s_h + c]
  int64_t s_nb, s_h;
  int32_t* bitmask;        // [NB, Hkv, C/32] (atomic OR) or null
  int32_t* qmask;          // [Q, Hkv, C/32] or null
  int32_t* counts;         // [Q, Hkv] or null
  int32_t* tokens;         // [Q, Hkv] or null
  float* prob_out;         // [Q, Hkv, C] or null
  float* theta_out;        // [Q, Hkv] or null
  int Q, Hq, Hkv, C, G, g_union, iters, sink;
  float inv_temp, beta, target;
};

// NK: clusters per lane at most; EXACT: C is 64 NK (64, 128, 256, 512, 1024), so that
// the loops over a lane's clusters are straight-line code.
template <int D, int NK, bool EXACT>
__global__ __launch_bounds__(256) void score_select_kernel(SelectArgs a, int R) {
  constexpr int KS = D / 32;
  constexpr int LDQ = D + 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16_t* sq = reinterpret_cast<bf16_t*>(smem);                      // [R][LDQ]
  float* ssc = reinterpret_cast<float*>(smem + (size_t)R * LDQ * 2);  // [R][C+1]
  const int C = EXACT ? 64 * NK : a.C, G = a.G;
  const int LDS_C = C + 1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int h = blockIdx.y;
  const int QT = R / G;
  const int q0 = blockIdx.x * QT;
  const int half = D / 2;

  // Q tile -> LDS (rows r = query*G + component)
  for (int e = threadIdx.x; e < R * (D / 8); e += 256) {
    int r = e / (D / 8), ch = e % (D / 8);
    int q = q0 + r / G, t = r % G;
    u32x4_t v = u32x4_t{0, 0, 0, 0};
    if (q < a.Q)
      v = *reinterpret_cast<const u32x4_t*>(a.vectors + (int64_t)q * a.v_sq + (int64_t)(h * G + t) * a.v_sh + ch * 8);
    *reinterpret_cast<u32x4_t*>(&sq[r * LDQ + ch * 8]) = v;
  }
  __syncthreads();

  // scores: each wave takes C/4 clusters (a multiple of 16); its rows' operands stay in
  // registers over the clusters when they fit (R <= 32)
  const int cols_per_wave = C / 4;
  const bf16_t* cb = a.codebooks + (int64_t)h * 2 * C * half;
  constexpr int RB = 2;
  u32x4_t aop[RB][KS];
  auto load_a = [&](int rb, u32x4_t (&v)[KS]) {
#pragma unroll
    for (int s = 0; s < KS; ++s)
      v[s] = *reinterpret_cast<const u32x4_t*>(&sq[(rb * 16 + (lane & 15)) * LDQ + s * 32 + (lane >> 4) * 8]);
  };
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) load_a(min(rb, R / 16 - 1), aop[rb]);
  for (int cbk = 0; cbk < cols_per_wave / 16; ++cbk) {
    const int col0 = wave * cols_per_wave + cbk * 16;
    const int cc = col0 + (lane & 15);
    u32x4_t bop[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      int d = s * 32 + (lane >> 4) * 8;
      int part = d / half;
      bop[s] = *reinterpret_cast<const u32x4_t*>(cb + ((int64_t)part * C + cc) * half + (d - part * half));
    }
    auto score = [&](int rb, const u32x4_t (&v)[KS]) {
      f32x4_t acc = f32x4_t{0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < KS; ++s) acc = mfma16x16x32(as_bf16x8(v[s]), as_bf16x8(bop[s]), acc);
#pragma unroll
      for (int i = 0; i < 4; ++i) ssc[(rb * 16 + (lane >> 4) * 4 + i) * LDS_C + cc] = acc[i] * a.inv_temp;
    };
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
      if (rb < R / 16) score(rb, aop[rb]);
    for (int rb = RB; rb < R / 16; ++rb) {
      u32x4_t v[KS];
      load_a(rb, v);
      score(rb, v);
    }
  }
  __syncthreads();

  // per row (query, component): lse over C, then each cluster's w = exp(s - lse +
  // logmix) (base-2 hardware exp/log: about 1 ulp, far below the selection's near-tie
  // margin).  The rows r0, r0 + step, .. of a call are taken together, so that their
  // reductions overlap; v holds the lane's clusters, scores in and weights out.
  constexpr float LOG2E = 1.4426950408889634f;
  auto softmax_rows = [&](auto rows, int r0, int step, auto& v) {
    constexpr int N = decltype(rows)::value;
    float m[N], l[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float* row = ssc + (r0 + step * i) * LDS_C;
      m[i] = -INFINITY;
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        v[i][k] = (64 * k < C) ? row[lane + 64 * k] : -INFINITY;
        m[i] = fmaxf(m[i], v[i][k]);
      }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) m[i] = wave_max_dpp(m[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      l[i] = 0.f;
#pragma unroll
      for (int k = 0; k < NK; ++k)
        if (64 * k < C) l[i] += __builtin_amdgcn_exp2f((v[i][k] - m[i]) * LOG2E);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) l[i] = wave_sum_dpp(l[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = r0 + step * i, q = q0 + r / G, t = r % G;
      float lm = 0.f;
      if (a.logmix && q < a.Q) lm = a.logmix[(int64_t)q * a.Hq + h * G + t];
      // log2 of exp(lm) / (sum exp(s))
      const float off2 = (lm - m[i]) * LOG2E - __builtin_amdgcn_logf(l[i]);
#pragma unroll
      for (int k = 0; k < NK; ++k) v[i][k] = __builtin_amdgcn_exp2f(__builtin_fmaf(v[i][k], LOG2E, off2));
    }
  };
  // up to four components, the wave of a query takes their softmax itself (below);
  // with more, the weights go back into the table first
  if (G > 4) {
    for (int r = wave; r < R; r += 4) {
      float v[1][NK];
      softmax_rows(std::integral_constant<int, 1>(), r, 0, v);
#pragma unroll
      for (int k = 0; k < NK; ++k)
        if (64 * k < C) ssc[r * LDS_C + lane + 64 * k] = v[0][k];
    }
    __syncthreads();
  }

  // selection, one wave per query; lane holds clusters lane + 64k
  const int W = C / 32;
  const float NEG = -3.4e38f, POS = 3.4e38f;
  for (int qi = wave; qi < QT; qi += 4) {
    const int q = q0 + qi;
    if (q >= a.Q) break;
    const int b = q / a.g_union;
    const int32_t* sz = a.sizes + (int64_t)b * a.s_nb + (int64_t)h * a.s_h;
    float score[NK], size[NK];
    float real_size[NK];
    int size_i[NK];
    const int nk = C / 64;
    float hi = -INFINITY, lo = INFINITY;
    int live_total = 0;      // token counts: sizes sum to at most the prompt length
    // each cluster's weight: the components' sum, in component order
    float pw[NK];
    auto weights = [&](auto g) {
      float w[g.value][NK];
      softmax_rows(g, qi * G, 1, w);
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        pw[k] = 0.f;
#pragma unroll
        for (int t = 0; t < g.value; ++t) pw[k] += w[t][k];
      }
    };
    if (G == 4) {
      weights(std::integral_constant<int, 4>());
    } else if (G == 2) {
      weights(std::integral_constant<int, 2>());
    } else if (G == 1) {
      weights(std::integral_constant<int, 1>());
    } else {
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        pw[k] = 0.f;
        if (64 * k < C)
          for (int t = 0; t < G; ++t) pw[k] += ssc[(qi * G + t) * LDS_C + lane + 64 * k];
      }
    }
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      score[k] = NEG;
      size[k] = 0.f;
      size_i[k] = 0;
      real_size[k] = 0.f;
      if (k < nk) {
        int c = lane + 64 * k;
        const float p = pw[k];
        if (a.prob_out) a.prob_out[((int64_t)q * a.Hkv + h) * C + c] = p;
        float rs = (float)sz[c];
        float s = (a.sink > 0 && c == 0) ? 0.f : rs;  // the sink is hidden from the search
        real_size[k] = rs;
        size[k] = s;
        size_i[k] = (int)s;
        bool live = s > 0.f;
        constexpr float LN2 = 0.69314718055994531f;
        float sc = __builtin_amdgcn_logf(fmaxf(p, 1e-38f)) * LN2;
        if (a.beta != 0.f) sc = sc - a.beta * (__builtin_amdgcn_logf(1.0f + s) * LN2);
        sc = live ? sc : NEG;
        score[k] = sc;
        hi = fmaxf(hi, sc);
        lo = fminf(lo, live ? sc : POS);
        if (live) live_total += (int)s;
      }
    }
    hi = wave_max_dpp(hi) + 1e-6f;
    lo = wave_min_dpp(lo) - 1e-6f;
    lo = fminf(lo, hi - 1e-5f);
    live_total = wave_sum_i32_dpp(live_total);
    float budget = a.target;
    if (a.sink > 0) budget = fmaxf(a.target - (float)a.sink, 0.f);
    const bool all_fit = (float)live_total < budget;
    const int bud_i = budget_count(budget);
    // two bisection steps per round: the first step's mid and both possible
    // second mids are counted together (the same fp32 mids as one step at a time).
    // Once a mid has failed, the count reaches the budget at lo and not at hi; with
    // one score left in [lo, hi), a mid between them reaches it exactly when it is
    // not above that score, and the remaining steps need no counts.
    bool failed = false;
    for (int it = 0; it < a.iters; it += 2) {
      if (failed && it % 4 == 0) {
        int inside = 0;
        float last = NEG;
#pragma unroll
        for (int k = 0; k < NK; ++k) {
          const bool in = score[k] >= lo && score[k] < hi;
          inside += __popcll(__ballot(in));
          last = in ? score[k] : last;
        }
        if (inside == 1) {
          last = wave_max_dpp(last);
          for (int j = it; j < a.iters; ++j) {
            const float mid = (lo + hi) * 0.5f;
            if (mid <= last) lo = mid;
            else hi = mid;
          }
          break;
        }
      }
      const float m0 = (lo + hi) * 0.5f;
      const float m1 = (m0 + hi) * 0.5f;     // second mid if m0 reaches the budget
      const float m2 = (lo + m0) * 0.5f;     // second mid otherwise
      int c0 = 0, c1 = 0, c2 = 0;
#pragma unroll
      for (int k = 0; k < NK; ++k) {         // size_i[k] is 0 past the C clusters
        c0 += score[k] >= m0 ? size_i[k] : 0;
        c1 += score[k] >= m1 ? size_i[k] : 0;
        c2 += score[k] >= m2 ? size_i[k] : 0;
      }
      wave_sum3_i32_swap(c0, c1, c2);
      if (c0 >= bud_i) {
        lo = m0;
        if (it + 1 < a.iters) {
          if (c1 >= bud_i) lo = m1;
          else hi = m1, failed = true;
        }
      } else {
        hi = m0;
        failed = true;
        if (it + 1 < a.iters) {
          if (c2 >= bud_i) lo = m2;
          else hi = m2;
        }
      }
    }
    const float theta = all_fit ? NEG : lo;
    int nsel = 0;
    int ntok = 0;
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      if (k < nk) {
        int c = lane + 64 * k;
        bool sel = (size[k] > 0.f && score[k] >= theta) || (a.sink > 0 && c == 0 && real_size[k] > 0.f);
        nsel += sel ? 1 : 0;
        ntok += sel ? (int)real_size[k] : 0;
        uint64_t ball = __ballot(sel);
        if (lane < 2) {
          uint32_t word = (uint32_t)(ball >> (32 * lane));
          int wi = 2 * k + lane;
          if (a.qmask) a.qmask[((int64_t)q * a.Hkv + h) * W + wi] = (int32_t)word;
          if (a.bitmask && word) atomicOr((unsigned int*)&a.bitmask[((int64_t)b * a.Hkv + h) * W + wi], word);
        }
      }
    }
    nsel = wave_sum_i32_dpp(nsel);
    ntok = wave_sum_i32_dpp(ntok);
    if (lane == 0) {
      if (a.counts) a.counts[(int64_t)q * a.Hkv + h] = nsel;
      if (a.tokens) a.tokens[(int64_t)q * a.Hkv + h] = (int32_t)ntok;
      if (a.theta_out) a.theta_out[(int64_t)q * a.Hkv + h] = theta;
    }
  }
}

// Several chunks of one prompt in one launch: blockIdx.y is the chunk, whose
// queries follow the earlier chunks' (chunk_q each, the last one what is left of
// total_q).  Strides are in elements; zero strides and one chunk are a single call.
struct ChunkBatch {
  int chunk_q = 0, total_q = 0;
  int64_t sizes = 0, limit = 0, rev = 0, qvals = 0, items = 0;
  __device__ int queries(int q) const { return chunk_q ? min(chunk_q, total_q - (int)blockIdx.y * chunk_q) : q; }
};

// ---------------------------------------------------------------- S3c ------
// |{keys of cluster c with position < limit}|: the run is position-sorted.
__global__ void causal_sizes_kernel(const int32_t* __restrict__ posting, int64_t width,
                                    const int32_t* __restrict__ indptr,
                                    const int32_t* __restrict__ sizes, int hkv, int C,
                                    int64_t limit, int32_t* __restrict__ out, ChunkBatch cb) {
  limit += blockIdx.y * cb.limit;
  out += blockIdx.y * cb.sizes;
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= hkv * C) return;
  int h = e / C, c = e % C;
  const int32_t* run = posting + (int64_t)h * width + indptr[h * (C + 1) + c];
  int lo = 0, hi = sizes[e];
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    if ((int64_t)run[mid] < limit) lo = mid + 1;
    else hi = mid;
  }
  out[e] = lo;
}

// ----------------------------------------------------------------- S4 ------
// Per (head, cluster): the queries whose qmask has the cluster (and the
// cluster has visible rows), in query order.  Pass 0 counts, pass 1 fills
// qvals[rev_indptr + rank] and qrank[q, h, c] = rank.
__global__ __launch_bounds__(256) void rev_pass_kernel(int pass, const int32_t* __restrict__ qmask,
                                                       int Q, int hkv, int C,
                                                       const int32_t* __restrict__ nvis,
                                                       int32_t* __restrict__ rev_counts,
                                                       const int32_t* __restrict__ rev_indptr,
                                                       int32_t* __restrict__ qvals,
                                                       int32_t* __restrict__ qrank) {
  __shared__ int wcnt[4];
  const int hc = blockIdx.x;
  const int h = hc / C, c = hc % C;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int W = C / 32;
  const bool live = nvis[hc] > 0;
  int run = 0;
  const int base_out = (pass == 1) ? rev_indptr[hc] : 0;
  for (int q0 = 0; q0 < Q; q0 += 256) {
    int q = q0 + threadIdx.x;
    bool bit = false;
    if (live && q < Q) bit = (qmask[((int64_t)q * hkv + h) * W + (c >> 5)] >> (c & 31)) & 1;
    uint64_t ball = __ballot(bit);
    if (lane == 0) wcnt[wave] = __popcll(ball);
    __syncthreads();
    int off = run;
    for (int w = 0; w < wave; ++w) off += wcnt[w];
    int before = __popcll(ball & ((lane == 0) ? 0ull : (~0ull >> (64 - lane))));
    if (pass == 1 && bit) {
      int rank = off + before;
      qvals[base_out + rank] = q;
      qrank[((int64_t)q * hkv + h) * C + c] = rank;
    }
    run += wcnt[0] + wcnt[1] + wcnt[2] + wcnt[3];
    __syncthreads();
  }
  if (pass == 0 && threadIdx.x == 0) rev_counts[hc] = run;
}

// The same in segments of REV_SEG queries, given scratch for a count per (segment,
// head, cluster): a block takes one head's clusters over one segment and reads each
// mask word once, where rev_pass_kernel's block walks all queries for one cluster (32
// blocks re-read each word).  Pass 0 counts per segment; the scan below turns the
// counts into each segment's first rank; pass 1 writes the lists.  One MI355X, 8192
// queries, 4 heads, 128 clusters: 2 x 25 -> 6.6 + 22.1 us for the two passes.
constexpr int REV_SEG = 256;

__global__ __launch_bounds__(REV_SEG) void rev_segment_kernel(int pass, const int32_t* __restrict__ qmask, int Q,
                                                              int hkv, int C, const int32_t* __restrict__ nvis,
                                                              int32_t* __restrict__ seg,
                                                              const int32_t* __restrict__ rev_indptr,
                                                              int32_t* __restrict__ qvals,
                                                              int32_t* __restrict__ qrank, ChunkBatch cb) {
  extern __shared__ int s_count[];     // [4 waves][C]: this wave's entries, then its first rank
  const int h = blockIdx.z;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int W = C / 32;
  Q = cb.queries(Q);
  qmask += (int64_t)blockIdx.y * cb.chunk_q * hkv * W;
  nvis += blockIdx.y * cb.sizes + h * C;
  seg += blockIdx.y * cb.qvals + ((int64_t)blockIdx.x * hkv + h) * C;
  rev_indptr += blockIdx.y * cb.rev + h * C;
  qvals += blockIdx.y * cb.qvals;
  qrank += (int64_t)blockIdx.y * cb.chunk_q * hkv * C;
  const int q = blockIdx.x * REV_SEG + threadIdx.x;
  const int32_t* words = qmask + ((int64_t)q * hkv + h) * W;
  auto live_word = [&](int w) -> uint32_t {
    const uint32_t live = (uint32_t)__ballot(lane < 32 && nvis[w * 32 + (lane & 31)] > 0);
    return q < Q ? (uint32_t)words[w] & live : 0u;
  };
  int* mine = s_count + wave * C;
  for (int w = 0; w < W; ++w) {
    const uint32_t m = live_word(w);
    int n = 0;
#pragma unroll
    for (int b = 0; b < 32; ++b) {
      const int k = __popcll(__ballot((m >> b) & 1u));
      if (lane == b) n = k;
    }
    if (lane < 32) mine[w * 32 + lane] = n;
  }
  __syncthreads();
  if (pass == 0) {
    for (int c = threadIdx.x; c < C; c += REV_SEG)
      seg[c] = s_count[c] + s_count[C + c] + s_count[2 * C + c] + s_count[3 * C + c];
    return;
  }
  for (int c = threadIdx.x; c < C; c += REV_SEG) {
    int rank = seg[c];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int n = s_count[v * C + c];
      s_count[v * C + c] = rank;
      rank += n;
    }
  }
  __syncthreads();
  const uint64_t below = (1ull << lane) - 1;
  for (int w = 0; w < W; ++w) {
    const uint32_t m = live_word(w);
#pragma unroll 4
    for (int b = 0; b < 32; ++b) {
      const uint64_t ball = __ballot((m >> b) & 1u);
      if ((m >> b) & 1u) {
        const int c = w * 32 + b;
        const int rank = mine[c] + __popcll(ball & below);
        qvals[rev_indptr[c] + rank] = q;
        qrank[((int64_t)q * hkv + h) * C + c] = rank;
      }
    }
  }
}

// The segments' counts of each (head, cluster) into first ranks, their sum into
// counts, then the exclusive scan of the sums (one block per chunk).
__global__ __launch_bounds__(1024) void rev_segment_scan_kernel(int32_t* __restrict__ seg, int Q, int n,
                                                                int32_t* __restrict__ counts,
                                                                int32_t* __restrict__ indptr,
                                                                int64_t* __restrict__ nnz, ChunkBatch cb) {
  seg += blockIdx.y * cb.qvals;
  counts += blockIdx.y * cb.sizes;
  indptr += blockIdx.y * cb.rev;
  const int segments = (cb.queries(Q) + REV_SEG - 1) / REV_SEG;
  __shared__ int wsum[16];
  __shared__ int carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int base = 0; base < n; base += 1024) {
    const int i = base + threadIdx.x;
    int v = 0;
    if (i < n) {
      for (int k0 = 0; k0 < segments; k0 += 8) {
        int at[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) at[k] = k0 + k < segments ? seg[(int64_t)(k0 + k) * n + i] : 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          if (k0 + k < segments) seg[(int64_t)(k0 + k) * n + i] = v;
          v += at[k];
        }
      }
      counts[i] = v;
    }
    const int incl = wave_incl_scan(v);
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int off = carry;
    for (int w = 0; w < wave; ++w) off += wsum[w];
    if (i < n) indptr[i] = off + incl - v;
    __syncthreads();
    if (threadIdx.x == 1023) carry = off + incl;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    indptr[n] = carry;
    nnz[blockIdx.y] = carry;
  }
}

// Exclusive scan of the Hkv*C counts (one block), total into rev_indptr[n].
__global__ __launch_bounds__(1024) void rev_scan_kernel(const int32_t* __restrict__ counts, int n,
                                                        int32_t* __restrict__ indptr,
                                                        int64_t* __restrict__ nnz) {
  __shared__ int wsum[16];
  __shared__ int carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int base = 0; base < n; base += 1024) {
    int i = base + threadIdx.x;
    int v = (i < n) ? counts[i] : 0;
    int incl = wave_incl_scan(v);
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int off = carry;
    for (int w = 0; w < wave; ++w) off += wsum[w];
    if (i < n) indptr[i] = off + incl - v;
    __syncthreads();
    if (threadIdx.x == 1023) carry = off + incl;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    indptr[n] = carry;
    *nnz = carry;
  }
}

// Work list of the KV-outer body, one segment per XCD so that the items that
// read the same K/V (the query tiles of one KV head's window, the query tiles
// of one cluster) run on one XCD and share its L2.  Items within a segment:
// local-window items first (longest first), then cluster items, longest
// cluster first (visible rows descending, ties in (head, cluster) order), so
// that the items claimed last, when the queues run dry, are the shortest.  Item = {head, cluster or -1, first query slot, query
// count}.  queue = {n[8], off[8], counter[8]}; the counters are zeroed here.
// One block: per-XCD counts, each source's first item (one pass of eight
// per-segment wave scans over each round of 1024 sources), then one thread
// per source writes its items (a window tile, or the query tiles of one
// (head, cluster)).
__device__ __forceinline__ int local_xcd(int h, int tile, int hkv) {
  const int per = hkv >= 8 ? 1 : 8 / hkv;      // XCDs per KV head
  return ((h * per) + (tile % per)) & 7;
}
__device__ __forceinline__ int cluster_xcd(int h, int c, int C) { return (h * C + c) & 7; }

struct ItemSource {
  int x, n, h, c, qb, qn;
};

// order: cluster sources by enumeration position e' = 8 r + x, the source of
// rank r in segment x (every segment's sources keep their segment)
__device__ __forceinline__ ItemSource item_source(const int32_t* rev_counts, const int* order, int s,
                                                  int nloc, int hkv, int C, int Qc, int QT) {
  ItemSource r;
  const int nl = nloc * hkv;
  if (s < nl) {
    const int k = s / hkv, tile = nloc - 1 - k;
    r.h = s % hkv;
    r.c = -1;
    r.qb = tile * QT;
    r.qn = min(QT, Qc - r.qb);
    r.n = 1;
    r.x = local_xcd(r.h, tile, hkv);
  } else {
    const int e = order[s - nl];
    r.h = e / C;
    r.c = e % C;
    r.qb = 0;
    r.qn = rev_counts[e];
    r.n = (r.qn + QT - 1) / QT;
    r.x = cluster_xcd(r.h, r.c, C);
  }
  return r;
}

// queue[QUEUE_OVERFLOW]: 1 when the chunk's partial entries pass the partial
// buffer's capacity (the list is then empty)
constexpr int QUEUE_OVERFLOW = 24;
constexpr int QUEUE_INTS = 32;

__global__ __launch_bounds__(1024) void build_items_kernel(const int32_t* __restrict__ rev_counts,
                                                           int hkv, int C, int Qc, int QT,
                                                           int has_local, const int32_t* __restrict__ indptr,
                                                           const int32_t* __restrict__ nvis,
                                                           const int32_t* __restrict__ rev_indptr,
                                                           PrefillItem* __restrict__ items,
                                                           int32_t* __restrict__ queue,
                                                           int64_t cap, int64_t partials_cap,
                                                           int64_t last_partials_cap, ChunkBatch cb) {
  Qc = cb.queries(Qc);
  rev_counts += blockIdx.y * cb.sizes;
  nvis += blockIdx.y * cb.sizes;
  rev_indptr += blockIdx.y * cb.rev;
  items += blockIdx.y * cb.items;
  queue += blockIdx.y * QUEUE_INTS;
  if (blockIdx.y == gridDim.y - 1) partials_cap = last_partials_cap;
  extern __shared__ int s_first[];     // [nsrc] first item of each source, then
                                       // [hkv C] sort keys and [hkv C] source order
  __shared__ int cnt[8];
  __shared__ int base[8];
  __shared__ int wsum[16][8];
  const int nloc = has_local ? (Qc + QT - 1) / QT : 0;
  const int ncl = hkv * C;
  const int nsrc = nloc * hkv + ncl;
  int* s_key = s_first + nsrc;
  int* s_order = s_key + ncl;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (threadIdx.x < 8) cnt[threadIdx.x] = 0;
  // cluster sources ranked within their segment (e & 7) by visible rows,
  // descending; sources without queries last
  for (int e = threadIdx.x; e < ncl; e += 1024) s_key[e] = rev_counts[e] > 0 ? nvis[e] : -1;
  __syncthreads();
  for (int e = threadIdx.x; e < ncl; e += 1024) {
    const int k = s_key[e];
    int rank = 0;
    for (int e2 = e & 7; e2 < ncl; e2 += 8) {
      const int k2 = s_key[e2];
      rank += (k2 > k || (k2 == k && e2 < e)) ? 1 : 0;
    }
    s_order[8 * rank + (e & 7)] = e;
  }
  __syncthreads();
  for (int s = threadIdx.x; s < nsrc; s += 1024) {
    const ItemSource si = item_source(rev_counts, s_order, s, nloc, hkv, C, Qc, QT);
    if (si.n) atomicAdd(&cnt[si.x], si.n);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int run = 0;
    for (int x = 0; x < 8; ++x) {
      base[x] = run;        // the segment's offset, then its running fill
      run += cnt[x];
    }
  }
  __syncthreads();
  // a chunk whose partial entries (rev_indptr[hkv C]) pass the partial
  // buffer's capacity gets an empty list and the overflow flag: nothing of it
  // is written, and the caller runs it again with a buffer of its exact size
  const bool overflow = partials_cap > 0 && (int64_t)rev_indptr[ncl] > partials_cap;
  if (threadIdx.x < 8) {
    const int x = threadIdx.x;
    const int64_t end = min((int64_t)base[x] + cnt[x], cap);
    queue[x] = overflow ? 0 : (int32_t)max((int64_t)0, end - base[x]);   // n
    queue[8 + x] = base[x];                              // offset
    queue[16 + x] = 0;                                   // counter
    if (x == 0) queue[QUEUE_OVERFLOW] = overflow ? 1 : 0;
  }
  if (overflow) return;
  // each source's first item: the segment's fill plus the items of the
  // segment's earlier sources, by one scan per segment over each round of
  // 1024 sources (sources keep their order within a segment)
  for (int r0 = 0; r0 < nsrc; r0 += 1024) {
    const int s = r0 + threadIdx.x;
    int n = 0, x = 0;
    if (s < nsrc) {
      const ItemSource si = item_source(rev_counts, s_order, s, nloc, hkv, C, Qc, QT);
      n = si.n;
      x = si.x;
    }
    int mine = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int incl = wave_incl_scan_dpp(x == k ? n : 0);
      if (x == k) mine = incl - n;
      if (lane == 63) wsum[wave][k] = incl;
    }
    __syncthreads();
    if (n) {
      int o = base[x] + mine;
      for (int w = 0; w < wave; ++w) o += wsum[w][x];
      s_first[s] = o;
    }
    __syncthreads();
    if (threadIdx.x < 8) {
      int t = 0;
      for (int w = 0; w < 16; ++w) t += wsum[w][threadIdx.x];
      base[threadIdx.x] += t;
    }
    __syncthreads();
  }
  // expansion: a thread per window tile, then a wave per cluster source (its lanes
  // write the items side by side), or eight lanes where a cluster has few items (494
  // queries of 16 heads on 4: the kernel takes 24 us with a wave each, 10 with a
  // thread each, which at 8192 queries takes twice the wave form's 43)
  for (int s = threadIdx.x; s < nloc * hkv; s += 1024) {
    const ItemSource si = item_source(rev_counts, s_order, s, nloc, hkv, C, Qc, QT);
    if (s_first[s] < cap) items[s_first[s]] = PrefillItem{si.h, si.c, si.qb, si.qn, 0, 0, 0, 0};
  }
  const int gl = (Qc + QT - 1) / QT > 64 ? 64 : 8, sub = threadIdx.x & (gl - 1);
  for (int s = nloc * hkv + threadIdx.x / gl; s < nsrc; s += 1024 / gl) {
    const ItemSource si = item_source(rev_counts, s_order, s, nloc, hkv, C, Qc, QT);
    if (!si.n) continue;
    const int64_t f0 = s_first[s];
    const int e = si.h * C + si.c;
    const int nk = nvis[e], ent = rev_indptr[e], row = indptr[si.h * (C + 1) + si.c];
    for (int j = sub; j < si.n; j += gl)
      if (f0 + j < cap) items[f0 + j] = PrefillItem{si.h, si.c, j * QT, min(QT, si.qn - j * QT), nk, ent + j * QT, row, 0};
  }
}


int64_t rev_scratch(int num_queries, int ncl) { return (int64_t)((num_queries + REV_SEG - 1) / REV_SEG) * ncl; }

// With scratch: the segment kernels (any number of chunks); without: a block per
// (head, cluster) over all queries (one chunk).
void launch_reverse_index(const int32_t* qmask, int num_queries, int hkv, int C, const int32_t* nvis,
                          int32_t* rev_counts, int32_t* rev_indptr, int64_t* nnz, int32_t* qvals, int32_t* qrank,
                          int32_t* scratch, int chunks, const ChunkBatch& cb, hipStream_t stream) {
  const int n = hkv * C;
  if (scratch && num_queries > 0) {
    const dim3 grid((num_queries + REV_SEG - 1) / REV_SEG, chunks, hkv);
    const size_t lds = (size_t)4 * C * sizeof(int);
    hipLaunchKernelGGL(rev_segment_kernel, grid, dim3(REV_SEG), lds, stream, 0, qmask, num_queries, hkv, C, nvis,
                       scratch, rev_indptr, qvals, qrank, cb);
    hipLaunchKernelGGL(rev_segment_scan_kernel, dim3(1, chunks), dim3(1024), 0, stream, scratch, num_queries, n,
                       rev_counts, rev_indptr, nnz, cb);
    hipLaunchKernelGGL(rev_segment_kernel, grid, dim3(REV_SEG), lds, stream, 1, qmask, num_queries, hkv, C, nvis,
                       scratch, rev_indptr, qvals, qrank, cb);
    return;
  }
  hipLaunchKernelGGL(rev_pass_kernel, dim3(n), dim3(256), 0, stream, 0, qmask, num_queries, hkv, C, nvis,
                     rev_counts, rev_indptr, qvals, qrank);
  hipLaunchKernelGGL(rev_scan_kernel, dim3(1), dim3(1024), 0, stream, rev_counts, n, rev_indptr, nnz);
  hipLaunchKernelGGL(rev_pass_kernel, dim3(n), dim3(256), 0, stream, 1, qmask, num_queries, hkv, C, nvis,
                     rev_counts, rev_indptr, qvals, qrank);
}

// The builder keeps each source's first item, and the cluster sources' keys and order, in LDS.
constexpr int64_t ITEMS_LDS_BYTES = 150 * 1024;

int launch_items(const int32_t* rev_counts, int hkv, int C, int num_queries, int queries_per_item, int has_local,
                 const int32_t* indptr, const int32_t* nvis, const int32_t* rev_indptr, void* items,
                 int64_t items_cap, int64_t partials_cap, int64_t last_partials_cap, int32_t* queue, int chunks,
                 const ChunkBatch& cb, hipStream_t stream) {
  const int nloc = has_local ? (num_queries + queries_per_item - 1) / queries_per_item : 0;
  const int64_t lds = ((int64_t)nloc * hkv + 3 * (int64_t)hkv * C) * 4;
  if (lds > ITEMS_LDS_BYTES) return SBSA_ERR_UNSUPPORTED;
  static int64_t configured = 0;
  if (lds > configured) {
    if (hipFuncSetAttribute((const void*)build_items_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds) != hipSuccess)
      return SBSA_ERR_UNSUPPORTED;
    configured = lds;
  }
  hipLaunchKernelGGL(build_items_kernel, dim3(1, chunks), dim3(1024), lds, stream, rev_counts, hkv, C, num_queries,
                     queries_per_item, has_local, indptr, nvis, rev_indptr, (PrefillItem*)items, queue, items_cap,
                     partials_cap, last_partials_cap, cb);
  return SBSA_OK;
}

}  // namespace

// One instantiation per bound on the clusters a lane holds (C <= 64 NK).
template <int D, int NK>
int launch_select_nk(const SelectArgs& a, dim3 grid, size_t lds, int R, hipStream_t stream) {
  auto kernel = a.C == 64 * NK ? score_select_kernel<D, NK, true> : score_select_kernel<D, NK, false>;
  if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)lds) != hipSuccess)
    return SBSA_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(kernel, grid, dim3(256), lds, stream, a, R);
  return SBSA_OK;
}
template <int D>
int launch_select(const SelectArgs& a, dim3 grid, size_t lds, int R, hipStream_t stream) {
  const int nk = a.C / 64;
  if (nk <= 1) return launch_select_nk<D, 1>(a, grid, lds, R, stream);
  if (nk <= 2) return launch_select_nk<D, 2>(a, grid, lds, R, stream);
  if (nk <= 4) return launch_select_nk<D, 4>(a, grid, lds, R, stream);
  if (nk <= 8) return launch_select_nk<D, 8>(a, grid, lds, R, stream);
  return launch_select_nk<D, 16>(a, grid, lds, R, stream);
}

extern "C" {

int sbsa_score_select(const void* vectors, int64_t v_sq, int64_t v_sh, const float* logmix,
                      const void* codebooks, const int32_t* sizes, int64_t s_nb, int64_t s_h,
                      int num_queries, int num_q_heads, int num_kv_heads, int num_clusters,
                      int dim, int g_union, float inv_temperature, float beta,
                      float target_tokens, int iters, int sink_tokens, int32_t* bitmask,
                      int32_t* qmask, int32_t* counts, int32_t* tokens, float* prob_out,
                      float* theta_out, hipStream_t stream) {
  if (!vectors || !codebooks || !sizes || num_queries < 0 || num_kv_heads < 1) return SBSA_ERR_ARG;
  if (num_q_heads % num_kv_heads || g_union < 1 || iters < 0) return SBSA_ERR_ARG;
  if (v_sh % 8 || v_sq % 8) return SBSA_ERR_ARG;
  const int G = num_q_heads / num_kv_heads;
  const int C = num_clusters;
  if (C % 64 || C > 1024 || C < 64) return SBSA_ERR_UNSUPPORTED;
  if (G != 1 && G != 2 && G != 4 && G != 8 && G != 16) return SBSA_ERR_UNSUPPORTED;
  if (num_queries == 0) return SBSA_OK;
  // rows (query, component) per block: 32 keep a block's LDS near 50 KB at
  // C <= 256, so three blocks share a CU and hide each other's reduction
  // chains (C = 256, 8192 queries, with the softmax through the table: 373 us with
  // 64 rows, 173 us with 32, 205 with 16)
  int R = (C <= 256) ? 32 : (C <= 512 ? 32 : 16);
  if (R < G) R = G;
  if (R % 16) R = 16;
  SelectArgs a;
  a.vectors = (const bf16_t*)vectors;
  a.v_sq = v_sq;
  a.v_sh = v_sh;
  a.logmix = logmix;
  a.codebooks = (const bf16_t*)codebooks;
  a.sizes = sizes;
  a.s_nb = s_nb;
  a.s_h = s_h;
  a.bitmask = bitmask;
  a.qmask = qmask;
  a.counts = counts;
  a.tokens = tokens;
  a.prob_out = prob_out;
  a.theta_out = theta_out;
  a.Q = num_queries;
  a.Hq = num_q_heads;
  a.Hkv = num_kv_heads;
  a.C = C;
  a.G = G;
  a.g_union = g_union;
  a.iters = iters;
  a.sink = sink_tokens;
  a.inv_temp = inv_temperature;
  a.beta = beta;
  a.target = target_tokens;
  const int QT = R / G;
  dim3 grid((num_queries + QT - 1) / QT, num_kv_heads);
  size_t lds = (size_t)R * (dim + 8) * 2 + (size_t)R * (C + 1) * 4;
  if (lds > 160 * 1024) return SBSA_ERR_UNSUPPORTED;
  int rc = SBSA_ERR_UNSUPPORTED;
  switch (dim) {
    case 64: rc = launch_select<64>(a, grid, lds, R, stream); break;
    case 128: rc = launch_select<128>(a, grid, lds, R, stream); break;
    case 256: rc = launch_select<256>(a, grid, lds, R, stream); break;
    default: break;
  }
  if (rc) return rc;
  SBSA_CHECK_LAUNCH();
  return SBSA_OK;
}

int sbsa_causal_sizes(const int32_t* posting, int64_t width, const int32_t* indptr,
                      const int32_t* sizes, int num_kv_heads, int num_clusters,
                      int64_t pos_limit, int32_t* out, hipStream_t stream) {
  if (!posting || !indptr || !sizes || !out || num_kv_heads < 1 || num_clusters < 1) return SBSA_ERR_ARG;
  int n = num_kv_heads * num_clusters;
  hipLaunchKernelGGL(causal_sizes_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, posting,
                     width, indptr, sizes, num_kv_heads, num_clusters, pos_limit, out, ChunkBatch{});
  SBSA_CHECK_LAUNCH();
  return SBSA_OK;
}

int64_t sbsa_reverse_index_ints(int num_queries, int num_kv_heads, int num_clusters) {
  if (num_queries < 0 || num_kv_heads < 1 || num_clusters < 1) return 0;
  const int64_t ncl = (int64_t)num_kv_heads * num_clusters;
  return num_queries * ncl + rev_scratch(num_queries, (int)ncl);
}

int sbsa_reverse_index(const int32_t* qmask, int num_queries, int num_kv_heads, int num_clusters,
                       const int32_t* nvis, int32_t* rev_counts, int32_t* rev_indptr,
                       int64_t* nnz, int32_t* qvals, int64_t qvals_cap, int32_t* qrank,
                       hipStream_t stream) {
  if (!qmask || !nvis || !rev_counts || !rev_indptr || !nnz || !qvals || !qrank) return SBSA_ERR_ARG;
  if (num_clusters % 32 || num_clusters < 32 || num_queries < 0) return SBSA_ERR_ARG;
  int64_t bound = (int64_t)num_queries * num_kv_heads * num_clusters;
  if (qvals_cap < bound) return SBSA_ERR_CAPACITY;
  // room past the lists holds the segments' counts
  int32_t* scratch =
      qvals_cap >= bound + rev_scratch(num_queries, num_kv_heads * num_clusters) ? qvals + bound : nullptr;
  launch_reverse_index(qmask, num_queries, num_kv_heads, num_clusters, nvis, rev_counts, rev_indptr, nnz, qvals,
                       qrank, scratch, 1, ChunkBatch{}, stream);
  SBSA_CHECK_LAUNCH();
  return SBSA_OK;
}

int64_t sbsa_prefill_items_bound(int64_t nnz, int num_queries, int num_kv_heads, int num_clusters,
                                 int queries_per_item) {
  int64_t qt = queries_per_item;
  return (int64_t)num_kv_heads * ((num_queries + qt - 1) / qt) +
         (int64_t)num_kv_heads * num_clusters + (nnz + qt - 1) / qt;
}

int64_t sbsa_prefill_items_max_queries(int num_kv_heads, int num_clusters, int queries_per_item) {
  if (num_kv_heads < 1 || num_clusters < 1 || queries_per_item < 1) return 0;
  const int64_t tiles = (ITEMS_LDS_BYTES / 4 - 3 * (int64_t)num_kv_heads * num_clusters) / num_kv_heads;
  return tiles > 0 ? tiles * queries_per_item : 0;
}

int sbsa_prefill_items(const int32_t* rev_counts, int num_kv_heads, int num_clusters,
                       int num_queries, int queries_per_item, int has_local,
                       const int32_t* indptr, const int32_t* nvis, const int32_t* rev_indptr,
                       void* items, int64_t items_cap, int64_t partials_cap, int32_t* queue,
                       hipStream_t stream) {
  if (!rev_counts || !items || !queue || queries_per_item < 1) return SBSA_ERR_ARG;
  if (!indptr || !nvis || !rev_indptr) return SBSA_ERR_ARG;
  const int rc = launch_items(rev_counts, num_kv_heads, num_clusters, num_queries, queries_per_item, has_local, indptr,
                              nvis, rev_indptr, items, items_cap, partials_cap, partials_cap, queue, 1, ChunkBatch{},
                              stream);
  if (rc) return rc;
  SBSA_CHECK_LAUNCH();
  return SBSA_OK;
}

int sbsa_plan_chunks(const void* vectors, int64_t v_sq, int64_t v_sh, const void* codebooks, const int32_t* posting,
                     int64_t width, const int32_t* indptr, const int32_t* sizes, int64_t first_pos, int num_queries,
                     int chunk_queries, int num_q_heads, int num_kv_heads, int num_clusters, int dim,
                     float inv_temperature, float beta, float target_tokens, int iters, int queries_per_item,
                     int32_t* causal_sizes, int32_t* tokens, float* theta_out, int32_t* qmask, int32_t* rev_counts,
                     int32_t* rev_indptr, int64_t* nnz, int32_t* qvals, int32_t* qrank, void* items, int64_t items_cap,
                     int64_t partials_cap, int64_t last_partials_cap, int32_t* queues, hipStream_t stream) {
  if (!posting || !indptr || !sizes || !causal_sizes || !qmask || !rev_counts || !rev_indptr || !nnz || !qvals ||
      !qrank || !items || !queues)
    return SBSA_ERR_ARG;
  if (num_queries < 1 || chunk_queries < 1 || num_kv_heads < 1 || num_clusters < 64 || num_clusters % 64 ||
      queries_per_item < 1)
    return SBSA_ERR_ARG;
  const int chunks = (num_queries + chunk_queries - 1) / chunk_queries;
  const int ncl = num_kv_heads * num_clusters;
  ChunkBatch cb;
  cb.chunk_q = chunk_queries;
  cb.total_q = num_queries;
  cb.limit = chunk_queries;
  cb.sizes = ncl;
  cb.rev = ncl + 1;
  const int64_t lists = (int64_t)chunk_queries * ncl;
  cb.qvals = lists + rev_scratch(chunk_queries, ncl);
  cb.items = items_cap;
  hipLaunchKernelGGL(causal_sizes_kernel, dim3((ncl + 255) / 256, chunks), dim3(256), 0, stream, posting, width, indptr,
                     sizes, num_kv_heads, num_clusters, first_pos, causal_sizes, cb);
  int rc = sbsa_score_select(vectors, v_sq, v_sh, nullptr, codebooks, causal_sizes, ncl, num_clusters, num_queries,
                             num_q_heads, num_kv_heads, num_clusters, dim, chunk_queries, inv_temperature, beta,
                             target_tokens, iters, 0, nullptr, qmask, nullptr, tokens, nullptr, theta_out, stream);
  if (rc) return rc;
  launch_reverse_index(qmask, chunk_queries, num_kv_heads, num_clusters, causal_sizes, rev_counts, rev_indptr, nnz,
                       qvals, qrank, qvals + lists, chunks, cb, stream);
  rc = launch_items(rev_counts, num_kv_heads, num_clusters, chunk_queries, queries_per_item, 1, indptr, causal_sizes,
                    rev_indptr, items, items_cap, partials_cap, last_partials_cap, queues, chunks, cb, stream);
  if (rc) return rc;
  SBSA_CHECK_LAUNCH();
  return SBSA_OK;
}

}  // extern "C"
