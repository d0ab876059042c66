// S5 KV-outer sparse prefill attention and S6 log-sum-exp combine for gfx950.
//
// Reference behaviour (pfnet-research/semantic-block-sparse-attention):
//   kv_outer.py:482-816        kv_outer_attention: one FA3 varlen call per
//                              (cluster, KV head) over its visible rows, whose
//                              query rows are the queries that selected it
//                              (Q heads folded into rows), plus an exactly
//                              causal FA3 call over the chunk's own window
//   fused_prefill.py:155-189   dense causal attention for the early chunks
//   kv_outer.py:370-428        _combine_grouped_kernel (query-major LSE fold)
//
// Design (MI355X): one persistent kernel walks a work list of items.  An item
// is (KV head, cluster or the local window, a tile of 128/G queries); its
// 128 (query, head) rows run against the cluster's contiguous packed run (or
// the prompt-order window, causally masked) in 32-key tiles.  Both GEMMs are
// on bf16 MFMA 32x32x16 in the transposed form S^T = K Q^T, O^T = V^T P^T,
// so the softmax probabilities come out of the first MFMA already in the
// B-operand layout of the second and never pass through LDS.
#include "sbsa_common.h"

namespace {

struct AttnArgs {
  const bf16_t* q;          // [Qc, Hq, D] chunk queries
  int64_t q_sq, q_sh;
  const bf16_t* packed;     // [2, Lp, Hkv, D] cluster-ordered K/V
  int64_t packed_len;
  const bf16_t* korig;      // prompt-order keys from position wstart: k[pos - wstart, h, :]
  const bf16_t* vorig;      // prompt-order values, same rows
  int64_t o_st, o_sh;       // their token / head strides (elements)
  const int32_t* indptr;    // [Hkv, C+1] packed run starts
  const int32_t* nvis;      // [Hkv, C] visible rows per cluster
  const int32_t* rev_indptr;// [Hkv*C + 1]
  const int32_t* qvals;     // [nnz] query slots per (head, cluster)
  const PrefillItem* items;
  int32_t* queue;           // n[8], offset[8], counter[8]: one work queue per XCD
  bf16_t* part_o;           // [nnz, G, D]
  float* part_lse;          // [nnz, G]
  bf16_t* local_o;          // [Qc, Hq, D] strided
  int64_t lo_sq, lo_sh;
  float* local_lse;         // [Qc, Hq] or null
  int Hkv, C, Hq;
  int Qc;                   // queries of the chunk
  int64_t chunk_start, wstart;
  float scale_log2;         // sm_scale * log2(e)
#ifdef SBSA_ATTN_PROBE
  int probe_slot;
#endif
};

#ifdef SBSA_ATTN_PROBE
// timing probe (a build flag, not in the product): per launch slot and block,
// the wall clock at each item start, tagged with the item
struct ProbeRec { uint64_t t; int idx, ntiles, qn, c; };
constexpr int PROBE_SLOTS = 32, PROBE_BLOCKS = 256, PROBE_RECS = 640;
__device__ ProbeRec g_attn_probe[PROBE_SLOTS][PROBE_BLOCKS][PROBE_RECS];
__device__ __forceinline__ void probe_mark(const AttnArgs& a, int& k, int idx, int nt, int qn, int c) {
  if (threadIdx.x == 0 && a.probe_slot < PROBE_SLOTS && blockIdx.x < PROBE_BLOCKS && k < PROBE_RECS) {
    ProbeRec r;
    r.t = __builtin_amdgcn_s_memrealtime();
    r.idx = idx; r.ntiles = nt; r.qn = qn; r.c = c;
    g_attn_probe[a.probe_slot][blockIdx.x][k] = r;
  }
  ++k;
}
#define PROBE(...) probe_mark(a, probe_k, __VA_ARGS__)
#else
#define PROBE(...) ((void)0)
#endif

constexpr int KT = 32;                  // keys per tile
constexpr int PREFILL_ROWS = 128;       // (query, head) rows per work item: 32 per wave
// Probabilities are taken against a reference maximum per row and may reach
// 2^OVERFLOW_LOG2 (well inside fp32 and bf16 range) before an item is redone.
constexpr float OVERFLOW_LOG2 = 64.0f;
constexpr int BUFFER_CONFIG = 0x00020000;   // raw buffer resource, 32-bit data format
// an offset past every range a store uses here (ranges stay below 2^31 bytes,
// so adding the access size cannot wrap): such a store is dropped
constexpr int OUT_OF_RANGE = (int)0x80000000u;

typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;

__device__ __forceinline__ const bf16_t* uniform_ptr(const bf16_t* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const bf16_t*)(((uint64_t)hi << 32) | lo);
}

// One 16-byte-per-lane buffer load straight into LDS (lane l writes bytes
// 16 l .. 16 l + 15 past lds_addr).  Issued from inline assembly so that the
// compiler does not track it: it would otherwise make every later LDS read
// wait for the load (it cannot tell that the read is from another buffer).
// The kernel waits for these loads itself (s_waitcnt vmcnt) before the
// barrier that publishes a tile.  M0 holds the LDS base, as the instruction
// requires; nothing else in the kernel uses M0.
__device__ __forceinline__ void lds_dma16(u32x4_t rsrc, uint32_t lds_addr, uint32_t voffset) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :
               : "s"(lds_addr), "v"(voffset), "s"(rsrc)
               : "memory", "m0");
}

// The same for one dword per lane (lane l writes bytes 4 l .. 4 l + 3).
__device__ __forceinline__ void lds_dma4(u32x4_t rsrc, uint32_t lds_addr, uint32_t voffset) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, 0 offen lds"
               :
               : "s"(lds_addr), "v"(voffset), "s"(rsrc)
               : "memory", "m0");
}

// v + (or max with) the same value of lane l ^ 32, in every lane: one swap of
// the lane halves instead of an LDS permute
__device__ __forceinline__ float halves_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float halves_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ __forceinline__ f32x16_t mfma32x32x16(bf16x8_t a, bf16x8_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// LDS tile layout: K and V rows of D bf16, row-major, 16-byte chunks of row r
// permuted by an XOR so that the operand reads of one LDS cycle (256 bytes,
// the 64 banks) hit distinct banks:
//   K: chunk ^ (r % 16)     16 lanes read 16 bytes of 16 different rows
//   V: chunk ^ 4 (r % 4)    32 lanes read 8 bytes of 4 rows, 64 bytes each
// Tiles are filled straight from global memory by buffer loads into LDS
// (lane l writes slot l of a 1 KB run; rows past the item's last key are
// outside the buffer's range and read as zero).
template <int D>
struct AttnTileShape {
  static constexpr int CH = D / 8;                    // 16-byte chunks per row
  static constexpr int ROW_BYTES = D * 2;
  static constexpr int TILE_BYTES = KT * ROW_BYTES;   // one of K or V
  static constexpr size_t LDS_BYTES = 4 * (size_t)TILE_BYTES;   // K, K, V, V tiles
  static constexpr int ROWS_PER_INST = 64 / CH;       // rows one wave instruction covers
  static constexpr int INSTS = KT / ROWS_PER_INST;    // instructions per K (or V) tile
  static constexpr int PER_WAVE = INSTS / 4;
};

// Both GEMMs on bf16 MFMA 32x32x16 in the transposed form: S^T = K Q^T
// (32 keys x 32 rows per tile) and O^T += V^T P^T (32 dims x 32 rows).  Lane
// l holds row l % 32 of the wave's 32 (query, head) rows; in S^T it holds keys
// 8 (i / 4) + 4 (l / 32) + i % 4, i < 16, which are exactly the B operand
// P^T of the two 16-key steps of O^T (keys {0-3, 8-11 | 4-7, 12-15} and
// {16-19, 24-27 | 20-23, 28-31}), so the probabilities never leave the lane.
// This form holds one block per compute unit and stays at 64 KB of LDS and
// under 384 registers per lane, so that the index build's kernels fit beside it
// on the same compute units (the layer's dense chunks run beside the build).
template <int D, int G>
__global__ __launch_bounds__(256, 1) void attn_items_kernel(AttnArgs a) {
  using S = AttnTileShape<D>;
  constexpr int KS = D / 16;        // 16-dim steps of S^T
  constexpr int DT = D / 32;        // 32-dim tiles of O^T
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_attn[];
  __shared__ int s_items[2];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // uniform: scalar LDS bases
  const int l32 = lane & 31, g = lane >> 5;
  const float NEG_INF = -INFINITY;
  // blocks are dispatched round-robin over the 8 XCDs: take work from this
  // XCD's queue, then steal from the others
  const int home = blockIdx.x & 7;
  int probe = 0;

  // --- per-lane address bases (fixed for the kernel) ---------------------
  // loads: instruction m of this wave covers rows r0 + 4 m RPI; their row % 4
  // is r0 % 4, their row % 16 alternates with m when 4 RPI == 8
  const int r0 = wave * S::ROWS_PER_INST + lane / S::CH;
  const int cpos = lane % S::CH;
  uint32_t kslot[2], vslot;
  kslot[0] = (uint32_t)((cpos ^ (r0 & 15)) * 16);
  kslot[1] = (uint32_t)((cpos ^ ((r0 + 4 * S::ROWS_PER_INST) & 15)) * 16);
  vslot = (uint32_t)((cpos ^ ((r0 & 3) << 2)) * 16);
  // K operand (A of S^T): row l32, chunk (2 s + g) ^ (l32 % 16); for s < 8 the
  // chunk stays below 16, past it the XOR keeps the +16 (256 bytes)
  int kbase[8];
#pragma unroll
  for (int s8 = 0; s8 < 8; ++s8) kbase[s8] = l32 * S::ROW_BYTES + 16 * ((2 * s8 + g) ^ (l32 & 15));
  // V^T operand (A of O^T, transposing reads): the 16-lane group (g, hh)
  // covers dims dt*32 + hh*16 .. +16 of rows K0..K0+3 with K0 = 16 m + 4 g
  // (+8 for the second read); lane i of the group reads row K0 + i/4, dims
  // 4 (i % 4).., chunk (4 dt + 2 hh + (i % 4)/2) ^ 4 (i / 4)
  const int i16 = lane & 15, hh = (lane >> 4) & 1;
  int vbase[4];
#pragma unroll
  for (int d4 = 0; d4 < 4; ++d4)
    vbase[d4] = (4 * g + (i16 >> 2)) * S::ROW_BYTES + 16 * (4 * (d4 ^ (i16 >> 2)) + 2 * hh + ((i16 & 3) >> 1)) +
                8 * (i16 & 1);

  // LDS: K tiles in buffers 0/1, V tiles in buffers 2/3
  auto kbuf_at = [&](int i) { return smem_attn + i * S::TILE_BYTES; };
  auto vbuf_at = [&](int i) { return smem_attn + (2 + i) * S::TILE_BYTES; };

  // Thread 0 claims work one item ahead: the atomic for the following claim
  // is issued when a claim resolves, so its latency hides behind an item's
  // work.  Items are used one further ahead: when an item starts, the next
  // one is claimed and its record is loaded, and once the item's first tiles
  // are in, wave 0 loads the next item's query slots straight into LDS.  An
  // item then starts with all of its addresses known, and its Q loads and
  // first tile loads share one round trip.
  // the queues' sizes and offsets are read once, into LDS
  __shared__ int s_queue[16];
  if (threadIdx.x < 16) s_queue[threadIdx.x] = a.queue[threadIdx.x];
  __syncthreads();
  // The first 2 B positions of each segment (B = blocks per segment) are
  // paired statically: the block of rank i in its segment takes positions i
  // and 2 B - 1 - i.  Segments start with their longest items, so a pair
  // (long, short) evens out the blocks' first shares, which would otherwise
  // go by the order of the first atomic claims.  The later positions are
  // claimed through the segment's counter; a segment of no more than 2 B items has none,
  // and its counter is not touched (see attn_pair_kernel).
  const int nstat = (gridDim.x % 8 == 0) ? 2 * (int)(gridDim.x / 8) : 0;
  const int srank = (int)(blockIdx.x >> 3);
  int pend = 0, nclaims = 0;
  auto request = [&]() {
    while (probe < 8 && s_queue[(home + probe) & 7] <= nstat) ++probe;
    if (probe < 8) pend = atomicAdd(&a.queue[16 + ((home + probe) & 7)], 1);
  };
  if (threadIdx.x == 0) request();
  // thread 0 only: the next item of this block's queue (stealing from the
  // other XCDs' queues once it is empty), -1 when every queue is
  auto claim = [&]() -> int {
    while (nclaims < 2 && nstat > 0) {
      const int pos = nclaims++ == 0 ? srank : nstat - 1 - srank;
      if (pos < s_queue[home]) return s_queue[8 + home] + pos;
    }
    while (probe < 8) {
      const int x = (home + probe) & 7, pos = nstat + pend;
      const bool got = pos < s_queue[x];
      if (!got) ++probe;
      request();
      if (got) return s_queue[8 + x] + pos;
    }
    return -1;
  };
  // Claims run two items ahead through two LDS slots, so reading one needs no
  // barrier: when an item starts, the next item's index (slot of parity i + 1)
  // was written when the previous item started, and every item's steps end
  // with barriers; thread 0 then writes the index after next into the slot
  // the current item's index came from, which every thread read one item ago.
  int parity = 0;
  auto next_index = [&]() -> int {
    const int v = __builtin_amdgcn_readfirstlane(s_items[parity ^ 1]);   // uniform: scalar loads below
    if (threadIdx.x == 0) s_items[parity] = v >= 0 ? claim() : -1;
    parity ^= 1;
    return v;
  };
  // this lane's Q row R = wave*32 + l32 is (query slot R / G, head R % G)
  const int row_i = (wave * 32 + l32) / G, row_j = (wave * 32 + l32) % G;
  // a cluster item's query slots, qvals[entry0 ..][0 .. qn), into s_qslots
  // (wave 0; slots past qn read as 0 and are not used)
  __shared__ int s_qslots[PREFILL_ROWS];
  auto fetch_slots = [&](const PrefillItem& r) {
    const int c = __builtin_amdgcn_readfirstlane(r.c);
    if (wave != 0 || c < 0) return;
    const int qn = __builtin_amdgcn_readfirstlane(r.qn);
    const uint64_t b = (uint64_t)(a.qvals + __builtin_amdgcn_readfirstlane(r.entry0));
    u32x4_t rsrc;
    rsrc.x = __builtin_amdgcn_readfirstlane((uint32_t)b);
    rsrc.y = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) & 0xffffu;
    rsrc.z = (uint32_t)qn * 4u;
    rsrc.w = (uint32_t)BUFFER_CONFIG;
    const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void_t*)s_qslots);
#pragma unroll
    for (int k = 0; k < PREFILL_ROWS / G; k += 64) lds_dma4(rsrc, dst + 4 * k, (uint32_t)(lane + k) * 4u);
  };
  // direct loads of the K (or V) rows of tile t into an LDS buffer; rows
  // past the item's last key are outside the buffer range and read as 0
  auto issue = [&](const bf16_t* base, uint32_t rs_bytes, int nkeys, int t, unsigned char* dst_tile, bool is_k) {
    const int t0 = t * KT;
    const int valid = __builtin_amdgcn_readfirstlane((int)((uint32_t)(nkeys - t0) * rs_bytes));
    const uint64_t b = (uint64_t)((const unsigned char*)base + (uint64_t)t0 * rs_bytes);
    u32x4_t rsrc;     // raw buffer resource: base, stride 0, valid bytes, config
    rsrc.x = __builtin_amdgcn_readfirstlane((uint32_t)b);
    rsrc.y = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) & 0xffffu;
    rsrc.z = (uint32_t)valid;
    rsrc.w = (uint32_t)BUFFER_CONFIG;
    const uint32_t dst = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(lds_void_t*)(dst_tile + wave * 1024));
    const uint32_t kvoff = (uint32_t)r0 * rs_bytes;
#pragma unroll
    for (int m = 0; m < S::PER_WAVE; ++m) {
      const uint32_t roff = kvoff + (uint32_t)(m * 4 * S::ROWS_PER_INST) * rs_bytes;
      const uint32_t slot = is_k ? kslot[m & 1] : vslot;
      lds_dma16(rsrc, dst + m * 4096, roff + slot);
    }
  };

  // The item being started: its fields (uniform), this lane's query (-1 past
  // the item's queries; a cluster item's slots were loaded into LDS during the
  // previous item), its Q rows in registers and its first tiles in flight.
  // An item is started as soon as the previous one no longer needs its Q
  // registers and tile buffers, so these loads run under that item's
  // epilogue.  Q^T (B of S^T): lane holds row R -> (slot row_i, head row_j),
  // dims 16 s + 8 g .. +8.  Rows past the item's queries take query slot 0's
  // values: they are computed like any row and never stored.
  int b_h = 0, b_c = 0, b_qb = 0, b_qn = 0, b_nkeys = 0, b_qidx = -1;
  int64_t b_entry0 = 0;
  const bf16_t* b_kp = nullptr;
  const bf16_t* b_vp = nullptr;
  uint32_t b_rsb = 0;
  u32x4_t qr[KS];
  auto begin = [&](const PrefillItem& r) {
    b_h = __builtin_amdgcn_readfirstlane(r.h);
    b_c = __builtin_amdgcn_readfirstlane(r.c);
    b_qb = __builtin_amdgcn_readfirstlane(r.qb);
    b_qn = __builtin_amdgcn_readfirstlane(r.qn);
    b_entry0 = __builtin_amdgcn_readfirstlane(r.entry0);
    const bool local = b_c < 0;
    const int64_t row0 = __builtin_amdgcn_readfirstlane(r.row0);
    int nkeys = local ? (int)(a.chunk_start + b_qb + b_qn - a.wstart) : __builtin_amdgcn_readfirstlane(r.nkeys);
    // an item without keys runs one fully masked tile: its output is 0 and its
    // LSE -inf, and its step publishes the next item's slots like any other
    b_nkeys = max(__builtin_amdgcn_readfirstlane(nkeys), 0);
    const bf16_t* kp;
    const bf16_t* vp;
    int64_t rs;
    if (local) {
      kp = a.korig + (int64_t)b_h * a.o_sh;   // row 0 is position wstart
      vp = a.vorig + (int64_t)b_h * a.o_sh;
      rs = a.o_st;
    } else {
      kp = a.packed + row0 * a.Hkv * D + (int64_t)b_h * D;
      vp = kp + a.packed_len * a.Hkv * D;
      rs = (int64_t)a.Hkv * D;
    }
    // uniform values (scalar registers): the buffer resources built from them
    // need no per-lane loop
    b_kp = uniform_ptr(kp);
    b_vp = uniform_ptr(vp);
    b_rsb = (uint32_t)__builtin_amdgcn_readfirstlane((int)(rs * 2));
    b_qidx = row_i >= b_qn ? -1 : (local ? b_qb + row_i : s_qslots[row_i]);
    const bf16_t* src = a.q + (int64_t)max(b_qidx, 0) * a.q_sq + (int64_t)(b_h * G + row_j) * a.q_sh + g * 8;
#pragma unroll
    for (int s = 0; s < KS; ++s) qr[s] = *reinterpret_cast<const u32x4_t*>(src + s * 16);
    issue(b_kp, b_rsb, b_nkeys, 0, kbuf_at(0), true);
    issue(b_vp, b_rsb, b_nkeys, 0, vbuf_at(0), false);
    if (b_nkeys > KT) issue(b_kp, b_rsb, b_nkeys, 1, kbuf_at(1), true);
  };

  PrefillItem rec{};
  if (threadIdx.x == 0) {
    s_items[0] = claim();
    s_items[1] = s_items[0] >= 0 ? claim() : -1;
  }
  __syncthreads();
  int idx = __builtin_amdgcn_readfirstlane(s_items[0]);
  if (idx >= 0) {
    rec = a.items[idx];
    fetch_slots(rec);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    begin(rec);
  }
  int idx_n = -1;
#ifdef SBSA_ATTN_PROBE
  int probe_k = 0;
#endif
  PROBE(-2, 0, 0, 0);
  for (; idx >= 0; idx = idx_n) {
    // this item, as begin() left it
    const int h = __builtin_amdgcn_readfirstlane(b_h), c = __builtin_amdgcn_readfirstlane(b_c);
    const int qb = __builtin_amdgcn_readfirstlane(b_qb), qn = __builtin_amdgcn_readfirstlane(b_qn);
    const int64_t entry0 = b_entry0;
    const int nkeys = __builtin_amdgcn_readfirstlane(b_nkeys);
    const bf16_t* const kp = b_kp;
    const bf16_t* const vp = b_vp;
    const uint32_t rs_bytes = b_rsb;
    const int qidx_r = b_qidx;
    const bool local = c < 0;
    const int ntiles = max(1, (nkeys + KT - 1) / KT);
    PROBE(idx, ntiles, qn, c);
    idx_n = next_index();
    if (idx_n >= 0) rec = a.items[idx_n];
    // once, after this item's first tiles are in (every wave has read its
    // slot by then); the next item's first step publishes it
    bool prefetched = false;
    auto prefetch_queries = [&]() {
      if (idx_n >= 0 && !prefetched) fetch_slots(rec);
      prefetched = true;
    };
    const int qlim = local ? (int)(a.chunk_start + qidx_r - a.wstart) : 0x7fffffff;
    // the last key any row of this wave may see, and the last key every row
    // sees (no limit inside a cluster item)
    int wave_lim = 0x7fffffff, wave_min = 0x7fffffff;
    if (local) {
      wave_lim = qlim;
      wave_min = qidx_r >= 0 ? qlim : 0x7fffffff;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        wave_lim = max(wave_lim, __shfl_xor(wave_lim, o, 64));
        wave_min = min(wave_min, __shfl_xor(wave_min, o, 64));
      }
      wave_lim = __builtin_amdgcn_readfirstlane(wave_lim);
      wave_min = __builtin_amdgcn_readfirstlane(wave_min);
    }

    // S^T = K Q^T for one tile; K fragments are read KA_AHEAD ahead
    constexpr int KA_AHEAD = 3;
    auto kread = [&](const unsigned char* sK, int s) -> u32x4_t {
      return *reinterpret_cast<const u32x4_t*>(sK + kbase[s & 7] + 256 * (s >> 3));
    };
    auto gemm_s_body = [&](f32x16_t& sacc, const unsigned char* sK) {
#pragma unroll
      for (int e = 0; e < 16; ++e) sacc[e] = 0.f;
      u32x4_t ka[KA_AHEAD];
#pragma unroll
      for (int f = 0; f < KA_AHEAD; ++f) ka[f] = kread(sK, f);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4_t cur = ka[s % KA_AHEAD];
        if (s + KA_AHEAD < KS) ka[s % KA_AHEAD] = kread(sK, s + KA_AHEAD);
        sacc = mfma32x32x16(as_bf16x8(cur), as_bf16x8(qr[s]), sacc);
      }
    };
    auto gemm_s = [&](f32x16_t& sacc, const unsigned char* sK) {
      gemm_s_body(sacc, sK);
      __builtin_amdgcn_sched_group_barrier(0x100, KA_AHEAD, 0);
#pragma unroll
      for (int f = 0; f < KS - KA_AHEAD; ++f) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, KA_AHEAD, 0);
    };

    // masking of tile t (only tiles that cross the item's end or a row's
    // causal limit) and this lane's running maximum of the raw scores
    float lmax_all = NEG_INF;
    auto mask_track = [&](f32x16_t& sacc, int t) {
      const int t0 = t * KT;
      if (t0 + KT > nkeys || t0 + KT - 1 > wave_min) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = t0 + 8 * (e >> 2) + 4 * g + (e & 3);
          if (!(key < nkeys && key <= qlim)) sacc[e] = NEG_INF;
        }
      }
#pragma unroll
      for (int e = 0; e < 16; e += 4)
        lmax_all = fmaxf(lmax_all, fmaxf(fmaxf(sacc[e], sacc[e + 1]), fmaxf(sacc[e + 2], sacc[e + 3])));
    };

    // the masking alone, for the passes that do not track the maximum
    auto mask_only = [&](f32x16_t& sacc, int t) {
      const int t0 = t * KT;
      if (t0 + KT > nkeys || t0 + KT - 1 > wave_min) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = t0 + 8 * (e >> 2) + 4 * g + (e & 3);
          if (!(key < nkeys && key <= qlim)) sacc[e] = NEG_INF;
        }
      }
    };

    // probabilities exp2(s - m) of a tile against the row's reference maximum
    // as the B operands of the two 16-key steps of O^T
    float m_ref = 0.f, l_part = 0.f;
    auto exp_pack = [&](f32x16_t& sacc, u32x4_t (&pb)[2]) {
      float sum = 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[e], a.scale_log2, -m_ref));
        sacc[e] = p;
        sum += p;
      }
      l_part += sum;
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        pb[m].x = pack2bf(sacc[8 * m + 0], sacc[8 * m + 1]);
        pb[m].y = pack2bf(sacc[8 * m + 2], sacc[8 * m + 3]);
        pb[m].z = pack2bf(sacc[8 * m + 4], sacc[8 * m + 5]);
        pb[m].w = pack2bf(sacc[8 * m + 6], sacc[8 * m + 7]);
      }
    };

    // O^T += V^T P^T: two transposing reads per 32-dim x 16-key fragment,
    // VA_AHEAD fragments ahead of the MFMAs
    f32x16_t o[DT];
    auto gemm_pv = [&](const u32x4_t (&pb)[2], const unsigned char* sV) {
      constexpr int NF = DT * 2;          // fragments (m, dt), m-major
      constexpr int VA_AHEAD = 4;
      u32x4_t va[VA_AHEAD];
      auto vread = [&](int f) -> u32x4_t {
        const int m = f / DT, dt = f % DT;
        const unsigned char* p = sV + vbase[dt & 3] + 256 * (dt >> 2) + 16 * m * S::ROW_BYTES;
        s16x4_t part[2];
        part[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)p);
        part[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(p + 8 * S::ROW_BYTES));
        u32x4_t r;
        __builtin_memcpy(&r, part, 16);
        return r;
      };
#pragma unroll
      for (int f = 0; f < VA_AHEAD; ++f) va[f] = vread(f);
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const u32x4_t cur = va[f % VA_AHEAD];
        if (f + VA_AHEAD < NF) va[f % VA_AHEAD] = vread(f + VA_AHEAD);
        const int m = f / DT, dt = f % DT;
        o[dt] = mfma32x32x16(as_bf16x8(cur), as_bf16x8(pb[m]), o[dt]);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * VA_AHEAD, 0);
#pragma unroll
      for (int f = 0; f < NF - VA_AHEAD; ++f) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, VA_AHEAD, 0);
    };

    // One step: S(t+1) on the MFMA units while the VALU turns S(t) into
    // probabilities, then O += V(t) P(t).  K(t+2) and V(t+1) stream into the
    // buffers that K(t) and V(t-1) left.  Two forms: the steady one, for
    // tiles whose successor some row of the wave still sees, is straight-line
    // code the scheduler can interleave; the general one handles the wave's
    // last active tile and the tiles past every row of the wave, whose loads
    // the wave still issues for the others.
    auto issue_next = [&](int t) {
      if (t + 2 < ntiles) issue(kp, rs_bytes, nkeys, t + 2, kbuf_at(t & 1), true);
      if (t + 1 < ntiles) issue(vp, rs_bytes, nkeys, t + 1, vbuf_at((t + 1) & 1), false);
    };
    auto finish_step = [&]() {
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    };
    auto step_full = [&](int t, f32x16_t& cur, f32x16_t& nxt) {
      issue_next(t);
      mask_only(cur, t);
      u32x4_t pb[2];
      gemm_s_body(nxt, kbuf_at((t + 1) & 1));
      exp_pack(cur, pb);
      // the VALU work of exp_pack between the MFMAs of S(t+1)
      __builtin_amdgcn_sched_group_barrier(0x100, KA_AHEAD, 0);
#pragma unroll
      for (int f = 0; f < KS - KA_AHEAD; ++f) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
      }
#pragma unroll
      for (int f = 0; f < KA_AHEAD; ++f) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
      }
      gemm_pv(pb, vbuf_at(t & 1));
      finish_step();
    };
    // the general form, for the tiles around a wave's last active one; with
    // sweep set it only tracks the rows' maxima (no probabilities, no O)
    auto step = [&](int t, f32x16_t& cur, f32x16_t& nxt, bool sweep) {
      issue_next(t);
      const bool act = t * KT <= wave_lim;
      const bool act_n = t + 1 < ntiles && (t + 1) * KT <= wave_lim;
      u32x4_t pb[2];
      if (act) {
        if (sweep) mask_track(cur, t);
        else mask_only(cur, t);
      }
      if (act_n) gemm_s(nxt, kbuf_at((t + 1) & 1));
      if (act && !sweep) {
        exp_pack(cur, pb);
        gemm_pv(pb, vbuf_at(t & 1));
      }
      finish_step();
    };

    // Each row's probabilities are taken against a reference maximum fixed
    // from the first tile; no accumulator is rescaled in the loop.  If a row's
    // sum of probabilities passes 2^OVERFLOW_LOG2 (which any probability past
    // that bound would cause; a probability up to it is safe in fp32 and
    // bf16), the item is redone: a sweep over the tiles finds the rows' true
    // maxima, and the last pass takes them as reference.
    for (int pass = 0; pass < 3; ++pass) {
      const bool sweep = pass == 1;
      if (pass > 0) {           // pass 0's first tiles were issued by begin()
        issue(kp, rs_bytes, nkeys, 0, kbuf_at(0), true);
        issue(vp, rs_bytes, nkeys, 0, vbuf_at(0), false);
        if (ntiles > 1) issue(kp, rs_bytes, nkeys, 1, kbuf_at(1), true);
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[dt][e] = 0.f;
      l_part = 0.f;
      lmax_all = NEG_INF;
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      prefetch_queries();
      f32x16_t sA, sB;
      gemm_s(sA, kbuf_at(0));
      mask_track(sA, 0);
      if (pass == 0) {
        // reference maximum: the row's maximum over the first tile (key 0 of
        // an item is visible to every row, so it is finite)
        const float mx = halves_max(lmax_all);
        m_ref = (mx == NEG_INF) ? 0.f : mx * a.scale_log2;
      }
      int t = 0;
      if (!sweep) {
        // tiles 0..t_last hold keys some row of this wave may see; the steady
        // loop runs while the next tile is active too
        const int t_last = min(ntiles - 1, wave_lim / KT);
        for (; t + 2 <= t_last; t += 2) {
          step_full(t, sA, sB);
          step_full(t + 1, sB, sA);
        }
      }
      for (; t < ntiles; t += 2) {
        step(t, sA, sB, sweep);
        if (t + 1 < ntiles) step(t + 1, sB, sA, sweep);
      }
      if (pass == 0) {
        const float l = halves_sum(l_part);
        const bool over = !(l <= __builtin_exp2f(OVERFLOW_LOG2));
        if (!__syncthreads_or(over ? 1 : 0)) break;
      } else if (sweep) {
        const float mx = halves_max(lmax_all);
        m_ref = (mx == NEG_INF) ? 0.f : mx * a.scale_log2;
      }
    }

    // epilogue: normalise, then write the partial (or the local window) and
    // its LSE.  The rows go through this wave's own 32-row slice of the idle
    // tile buffers, so that every store is 16 bytes per lane and whole rows per instruction: the item's
    // rows are contiguous in part_o, and the G heads of a query are
    // contiguous in the window output.
    {
      const float l = halves_sum(l_part);
      const float inv = (l > 0.f) ? 1.0f / l : 0.f;
      if (qidx_r >= 0 && g == 0) {
        const float lse = (l > 0.f) ? (m_ref + log2f(l)) * 0.69314718055994531f : NEG_INF;
        float* ldst = local ? (a.local_lse ? a.local_lse + (int64_t)qidx_r * a.Hq + h * G + row_j : nullptr)
                            : a.part_lse + (entry0 + row_i) * G + row_j;
        if (ldst) *ldst = lse;
      }
      // 16-byte chunk c of row r sits at chunk c ^ (r % 32) of the row.  Lane
      // (l32, g) holds dims 32 dt + 8 q4 + 4 g .. +3; a swap between the lane
      // halves (lanes l and l + 32) gives lane g = 0 all 8 dims of chunk
      // 4 dt + 2 p and lane g = 1 those of chunk 4 dt + 2 p + 1 (q4 = 2 p, 2 p + 1),
      // so each lane writes whole 16-byte chunks
      unsigned char* stage = smem_attn + wave * 32 * S::ROW_BYTES;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int qa = 2 * p, qb2 = 2 * p + 1;
          const uint32_t a0 = pack2bf(o[dt][4 * qa + 0] * inv, o[dt][4 * qa + 1] * inv);
          const uint32_t a1 = pack2bf(o[dt][4 * qa + 2] * inv, o[dt][4 * qa + 3] * inv);
          const uint32_t b0 = pack2bf(o[dt][4 * qb2 + 0] * inv, o[dt][4 * qb2 + 1] * inv);
          const uint32_t b1 = pack2bf(o[dt][4 * qb2 + 2] * inv, o[dt][4 * qb2 + 3] * inv);
          // lanes < 32 keep their q4 = 2p pair and take the upper lanes' one;
          // lanes >= 32 take the lower lanes' q4 = 2p + 1 pair and keep theirs
          const auto s0 = __builtin_amdgcn_permlane32_swap(a0, b0, false, false);
          const auto s1 = __builtin_amdgcn_permlane32_swap(a1, b1, false, false);
          u32x4_t w;
          w.x = s0[0];
          w.y = s1[0];
          w.z = s0[1];
          w.w = s1[1];
          const int c = (4 * dt + 2 * p + g) ^ (l32 & (S::CH - 1));
          *reinterpret_cast<u32x4_t*>(stage + l32 * S::ROW_BYTES + 16 * c) = w;
        }
      // the wave's lanes hand their rows to each other through the staging
      // slice (in order on the GPU, where a wave's LDS operations run in issue
      // order; the barrier keeps the compiler from moving them)
      __builtin_amdgcn_wave_barrier();
      // read back whole rows (instruction m covers rows ROWS_PER_INST m ..),
      // reads first, then the stores, so no store waits on a single read
      constexpr int NR = 32 / S::ROWS_PER_INST;
      const int c16 = lane % S::CH;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        u32x4_t rows[NR / 2];
#pragma unroll
        for (int mm = 0; mm < NR / 2; ++mm) {
          const int m = half * (NR / 2) + mm;
          const int r = m * S::ROWS_PER_INST + lane / S::CH;
          rows[mm] = *reinterpret_cast<const u32x4_t*>(stage + r * S::ROW_BYTES + 16 * (c16 ^ (r & (S::CH - 1))));
        }
#pragma unroll
        for (int mm = 0; mm < NR / 2; ++mm) {
          const int m = half * (NR / 2) + mm;
          const int RR = wave * 32 + m * S::ROWS_PER_INST + lane / S::CH;
          const int i = RR / G, j = RR % G;
          // read once, later, by the combine: non-temporal, kept out of the way
          // of the K/V in L2
          bf16_t* dst = local ? a.local_o + (int64_t)(qb + i) * a.lo_sq + (int64_t)(h * G + j) * a.lo_sh
                              : a.part_o + ((entry0 + i) * G + j) * D;
          if (i < qn) __builtin_nontemporal_store(rows[mm], reinterpret_cast<u32x4_t*>(dst + 8 * c16));
        }
      }
    }
    if (idx_n >= 0) {
      __syncthreads();          // every wave is done with its staging rows
      begin(rec);
    }
  }
  PROBE(-3, 0, 0, 0);
}


// The form with two blocks per compute unit: 256 registers per lane and 64 KB
// of LDS (D = 256), so a second block's matrix work covers the LDS latency, the
// exponentials and the item boundaries of the first.  What differs from the
// form above:
// - no software pipeline inside a wave: S^T of tile t, its probabilities, then
//   O^T += V^T P^T, with the loads of tile t + 1 in flight over the whole step
//   (they are issued behind the step's one barrier and awaited at its end);
// - the waves run the matrix parts at a raised wave priority, so that one
//   block's exponentials and addresses fill the other's matrix time;
// - an item's end: the next item's first tiles are issued, the first half of
//   each row is staged (in the tile buffers those loads leave alone) and stored,
//   the next item's Q rows are loaded into the registers that half held, and the
//   second half follows; the first wait leaves its stores in flight;
// - nothing that only the boundary uses lives across the tile loop (the lane
//   number is made opaque there): a spilled register's reload would wait for
//   every load and store in flight.
// Bound by the matrix cores at the clock that the chip holds under this load: by the
// counters they are busy 78-79 % of the cycles of a dense chunk (D = 256, 1024 items),
// the LDS index unit 39 %; 46-57 % in sparse chunks, whose items are 7-17 tiles long
// (item ends, and the last items alone on their units).  One MI355X, same inputs, former form -> this one: a
// dense chunk of 8192 queries at 24576, 3564 -> 2967 us (1080 -> 1297 TFLOP/s;
// an 8192^3 bf16 matrix product reaches 1313 there); a sparse chunk of 8192 at
// 114688 (980K entries), 2328 -> 1846 us (750 -> 946 TFLOP/s); D = 128, a sparse
// chunk of 3001 at 40009 with 16 heads on 8, 396 -> 348 us.
template <int D, int G>
__global__ __launch_bounds__(256, 2) void attn_pair_kernel(AttnArgs a) {
  using S = AttnTileShape<D>;
  constexpr int KS = D / 16;        // 16-dim steps of S^T
  constexpr int DT = D / 32;        // 32-dim tiles of O^T
  constexpr int SC = D / 16;        // 16-byte chunks of half a row (the epilogue stages half rows)
  constexpr int HROWS = 64 / SC;    // half rows one store instruction covers
  constexpr int HSTORES = 32 / HROWS;   // row stores of half an epilogue, per wave
  static_assert(HSTORES <= 63, "vmcnt range");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_attn[];
  __shared__ int s_items[2];
  __shared__ int s_queue[16];
  __shared__ int s_over[2];
  __shared__ int s_qslots[PREFILL_ROWS];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const float NEG_INF = -INFINITY;
  const int home = blockIdx.x & 7;
  int probe = 0;

  // per-lane addresses, as in the form above; the XORs of a step's or a tile's
  // number are applied at the read
  const int r0 = wave * S::ROWS_PER_INST + lane / S::CH;
  const int cpos = lane % S::CH;
  const uint32_t kslot0 = (uint32_t)((cpos ^ (r0 & 15)) * 16);
  const uint32_t kslot1 = (uint32_t)((cpos ^ ((r0 + 4 * S::ROWS_PER_INST) & 15)) * 16);
  const uint32_t vslot = (uint32_t)((cpos ^ ((r0 & 3) << 2)) * 16);
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void_t*)smem_attn);
  // K operand: row l32, chunk (2 s + g) ^ (l32 % 16) = (g ^ l32 % 16) ^ 2 s
  const int kb = l32 * S::ROW_BYTES;
  const int kx = 16 * (g ^ (l32 & 15));
  // V^T operand: vbase[d] of the form above is vb + (vx ^ 64 d)
  const int i16 = lane & 15, hh = (lane >> 4) & 1;
  const int vb = 2 * S::TILE_BYTES + (4 * g + (i16 >> 2)) * S::ROW_BYTES + 32 * hh + 16 * ((i16 & 3) >> 1) +
                 8 * (i16 & 1);
  const int vx = 64 * (i16 >> 2);

  if (threadIdx.x < 16) s_queue[threadIdx.x] = a.queue[threadIdx.x];
  if (threadIdx.x < 2) s_over[threadIdx.x] = 0;
  // Thread 0 claims work two items ahead.  The first 2 B positions of this XCD's
  // segment (B = blocks per XCD) are paired statically, a long item with a short
  // one; later positions come from the segment's counter, and from the other
  // segments' once it is empty.  The counter's atomic is issued at an item's end
  // and read after the next item's first tile, when every load has landed.  A segment
  // without later positions is passed by: in a call of few items, 512 blocks asking
  // eight counters each were 46 us of atomics on the same lines (90 ns per block).
  const int nstat = (gridDim.x % 8 == 0) ? 2 * (int)(gridDim.x / 8) : 0;
  int pend = -1, nclaims = 0;
  auto request = [&]() {
    if (threadIdx.x == 0 && pend < 0 && probe < 8 && s_queue[(home + probe) & 7] > nstat)
      pend = atomicAdd(&a.queue[16 + ((home + probe) & 7)], 1);
  };
  auto claim = [&]() -> int {
    while (nclaims < 2 && nstat > 0) {
      const int srank = (int)(blockIdx.x >> 3);
      const int pos = nclaims++ == 0 ? srank : nstat - 1 - srank;
      if (pos < s_queue[home]) return s_queue[8 + home] + pos;
    }
    for (; probe < 8; ++probe) {
      const int x = (home + probe) & 7;
      if (s_queue[x] <= nstat) continue;
      if (pend < 0) pend = atomicAdd(&a.queue[16 + x], 1);
      const int pos = nstat + pend;
      pend = -1;
      if (pos < s_queue[x]) return s_queue[8 + x] + pos;
    }
    return -1;
  };
  // An item's record, one field per lane: field f of the record is lane f's
  int recv = 0;
  auto field = [&](int f) -> int { return __builtin_amdgcn_readlane(recv, f); };
  auto load_record = [&](int idx) {
    int ln = lane;                       // opaque: its address is not kept across the tile loop
    asm volatile("" : "+v"(ln));
    recv = reinterpret_cast<const int*>(a.items + max(idx, 0))[ln & 7];
  };
  // a cluster item's query slots straight into LDS (wave 0)
  auto fetch_slots = [&]() {
    if (wave != 0 || field(1) < 0) return;
    const uint64_t b = (uint64_t)(a.qvals + field(5));
    u32x4_t rsrc;
    rsrc.x = __builtin_amdgcn_readfirstlane((uint32_t)b);
    rsrc.y = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) & 0xffffu;
    rsrc.z = (uint32_t)field(3) * 4u;
    rsrc.w = (uint32_t)BUFFER_CONFIG;
    const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void_t*)s_qslots);
#pragma unroll
    for (int k = 0; k < PREFILL_ROWS / G; k += 64) lds_dma4(rsrc, dst + 4 * k, (uint32_t)(lane + k) * 4u);
  };

  // the item being run
  int i_h = 0, i_c = 0, i_qb = 0, i_qn = 0, i_nkeys = 0, i_entry0 = 0;
  int qlim = 0;             // this lane's row: the last key it sees
  uint64_t kp = 0, vp = 0;  // its first K and V rows
  uint32_t rsb = 0;         // bytes from row to row
  u32x4_t qr[KS];
  // loads of tile t's K (or V) rows straight into LDS: the resource starts at
  // the tile and ends with the item's last key (rows past it read as zero)
  auto issue = [&](uint64_t base, int t, uint32_t dst, bool is_k) {
    const uint32_t t0 = (uint32_t)(t * KT);
    const uint64_t b = base + (uint64_t)t0 * rsb;
    u32x4_t rs;
    rs.x = __builtin_amdgcn_readfirstlane((uint32_t)b);
    rs.y = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) & 0xffffu;
    rs.z = ((uint32_t)i_nkeys - t0) * rsb;
    rs.w = (uint32_t)BUFFER_CONFIG;
    int row = r0;                        // opaque: eight offsets are not kept across the tile loop
    asm volatile("" : "+v"(row));
    const uint32_t off = (uint32_t)row * rsb, step = 4 * S::ROWS_PER_INST * rsb;
#pragma unroll
    for (int m = 0; m < S::PER_WAVE; ++m)
      lds_dma16(rs, dst + wave * 1024 + m * 4096, off + m * step + (is_k ? (m & 1 ? kslot1 : kslot0) : vslot));
  };
  // the item whose record is in recv: its fields, and its first tiles' loads
  auto begin = [&]() {
    i_h = field(0);
    i_c = field(1);
    i_qb = field(2);
    i_qn = field(3);
    i_entry0 = field(5);
    const bool local = i_c < 0;
    i_nkeys = max(local ? (int)(a.chunk_start + i_qb + i_qn - a.wstart) : field(4), 0);
    const bf16_t *k, *v;
    if (local) {
      k = a.korig + (int64_t)i_h * a.o_sh;
      v = a.vorig + (int64_t)i_h * a.o_sh;
      rsb = (uint32_t)(a.o_st * 2);
    } else {
      k = a.packed + ((int64_t)field(6) * a.Hkv + i_h) * D;
      v = k + a.packed_len * a.Hkv * D;
      rsb = (uint32_t)(a.Hkv * D * 2);
    }
    kp = (uint64_t)uniform_ptr(k);
    vp = (uint64_t)uniform_ptr(v);
    issue(kp, 0, lds0, true);
    issue(vp, 0, lds0 + 2 * S::TILE_BYTES, false);
  };
  // its queries (-1 past the item's; a cluster item's slots are in LDS), their
  // Q rows and this lane's causal limit.  Rows past the item's queries take
  // query 0's values: they are computed like any row and never stored.
  auto load_q = [&]() {
    int ln = lane;                       // opaque: its addresses are not kept across the tile loop
    asm volatile("" : "+v"(ln));
    const int R = wave * 32 + (ln & 31);
    const int row_i = R / G, row_j = R % G, g = ln >> 5;
    const bool local = i_c < 0;
    const int qidx = row_i >= i_qn ? -1 : (local ? i_qb + row_i : s_qslots[row_i]);
    qlim = local ? (qidx < 0 ? -1 : (int)(a.chunk_start - a.wstart) + qidx) : 0x7fffffff;
    const bf16_t* src = a.q + (int64_t)max(qidx, 0) * a.q_sq + (int64_t)(i_h * G + row_j) * a.q_sh + g * 8;
#pragma unroll
    for (int s = 0; s < KS; ++s) qr[s] = *reinterpret_cast<const u32x4_t*>(src + s * 16);
  };

  __syncthreads();
  int parity = 0, over_slot = 0;
  if (threadIdx.x == 0) {
    s_items[0] = claim();
    s_items[1] = s_items[0] >= 0 ? claim() : -1;
    request();
  }
  __syncthreads();
  {
    const int idx = __builtin_amdgcn_readfirstlane(s_items[0]);
    if (idx < 0) return;
    load_record(idx);
  }
  fetch_slots();
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  begin();
  load_q();
  int idx_n = __builtin_amdgcn_readfirstlane(s_items[1]);   // the next item
  bool after_stores = false;
  for (;;) {
    const bool local = i_c < 0;
    const int ntiles = max(1, (i_nkeys + KT - 1) / KT);
    // the last key every row of this wave sees (its first query's in the window)
    const int first_row = wave * 32 / G;
    const int wave_min = local && first_row < i_qn ? (int)(a.chunk_start - a.wstart) + i_qb + first_row : 0x7fffffff;
    const int full_end = min(i_nkeys - 1, wave_min);   // tiles up to this key need no mask
    float m_ref = 0.f, l_part = 0.f;
    f32x16_t o[DT];
    for (int pass = 0; pass < 3; ++pass) {
      const bool sweep = pass == 1;
      if (pass > 0) {
        int z = 0;             // opaque: the rare pass's addresses are not kept
        asm volatile("" : "+s"(z));
        issue(kp, z, lds0, true);
        issue(vp, z, lds0 + 2 * S::TILE_BYTES, false);
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[dt][e] = 0.f;
      l_part = 0.f;
      float lmax = NEG_INF;
      if (after_stores)
        __builtin_amdgcn_s_waitcnt((HSTORES & 15) | ((HSTORES >> 4) << 14) | (7 << 4));
      else
        __builtin_amdgcn_s_waitcnt(0);
      after_stores = false;
      for (int t = 0; t < ntiles; ++t) {
        __syncthreads();
        const uint32_t nb = ((t + 1) & 1) * S::TILE_BYTES;
        if (t + 1 < ntiles) {
          issue(kp, t + 1, lds0 + nb, true);
          issue(vp, t + 1, lds0 + 2 * S::TILE_BYTES + nb, false);
        }
        const bool first = pass == 0 && t == 0;
        if (first) {
          // every wave is past the previous item's overflow flag
          load_record(idx_n);
          if (threadIdx.x == 0) s_over[over_slot ^ 1] = 0;
        }
        const int cb = (t & 1) * S::TILE_BYTES;
        __builtin_amdgcn_s_setprio(1);
        f32x16_t sacc;
#pragma unroll
        for (int e = 0; e < 16; ++e) sacc[e] = 0.f;
        {
          constexpr int KA = 3;
          const int kc = kb + cb;
          auto kread = [&](int s) -> u32x4_t {
            return *reinterpret_cast<const u32x4_t*>(smem_attn + kc + (kx ^ (32 * (s & 7))) + 256 * (s >> 3));
          };
          u32x4_t ka[KA];
#pragma unroll
          for (int f = 0; f < KA; ++f) ka[f] = kread(f);
#pragma unroll
          for (int s = 0; s < KS; ++s) {
            const u32x4_t cur = ka[s % KA];
            if (s + KA < KS) ka[s % KA] = kread(s + KA);
            sacc = mfma32x32x16(as_bf16x8(cur), as_bf16x8(qr[s]), sacc);
          }
          __builtin_amdgcn_sched_group_barrier(0x100, KA, 0);
#pragma unroll
          for (int f = 0; f < KS - KA; ++f) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          }
          __builtin_amdgcn_sched_group_barrier(0x008, KA, 0);
        }
        __builtin_amdgcn_s_setprio(0);
        if (t * KT + KT - 1 > full_end) {
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int key = t * KT + 8 * (e >> 2) + 4 * g + (e & 3);
            if (!(key < i_nkeys && key <= qlim)) sacc[e] = NEG_INF;
          }
        }
        if (sweep || first) {
#pragma unroll
          for (int e = 0; e < 16; e += 4)
            lmax = fmaxf(lmax, fmaxf(fmaxf(sacc[e], sacc[e + 1]), fmaxf(sacc[e + 2], sacc[e + 3])));
          if (!sweep) {
            const float mx = halves_max(lmax);
            m_ref = (mx == NEG_INF) ? 0.f : mx * a.scale_log2;
          }
        }
        if (!sweep) {
          u32x4_t pb[2];
          float sum = 0.f;
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[e], a.scale_log2, -m_ref));
            sacc[e] = p;
            sum += p;
          }
          l_part += sum;
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            pb[m].x = pack2bf(sacc[8 * m + 0], sacc[8 * m + 1]);
            pb[m].y = pack2bf(sacc[8 * m + 2], sacc[8 * m + 3]);
            pb[m].z = pack2bf(sacc[8 * m + 4], sacc[8 * m + 5]);
            pb[m].w = pack2bf(sacc[8 * m + 6], sacc[8 * m + 7]);
          }
          __builtin_amdgcn_s_setprio(1);
          constexpr int NF = DT * 2;
          constexpr int VA = 4;
          const int vc = vb + cb;
          u32x4_t va[VA];
          auto vread = [&](int f) -> u32x4_t {
            const int m = f / DT, dt = f % DT;
            const unsigned char* p = smem_attn + vc + (vx ^ (64 * (dt & 3))) + 256 * (dt >> 2) + 16 * m * S::ROW_BYTES;
            s16x4_t part[2];
            part[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)p);
            part[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(p + 8 * S::ROW_BYTES));
            u32x4_t r;
            __builtin_memcpy(&r, part, 16);
            return r;
          };
#pragma unroll
          for (int f = 0; f < VA; ++f) va[f] = vread(f);
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            const u32x4_t cur = va[f % VA];
            if (f + VA < NF) va[f % VA] = vread(f + VA);
            o[f % DT] = mfma32x32x16(as_bf16x8(cur), as_bf16x8(pb[f / DT]), o[f % DT]);
          }
          __builtin_amdgcn_sched_group_barrier(0x100, 2 * VA, 0);
#pragma unroll
          for (int f = 0; f < NF - VA; ++f) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
          }
          __builtin_amdgcn_sched_group_barrier(0x008, VA, 0);
        }
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_s_waitcnt(0);     // this wave's share of the next tile has landed
        if (first && idx_n >= 0) {
          // the next item's record is here: its query slots, and the claim of the item after it
          fetch_slots();
          if (threadIdx.x == 0) s_items[parity] = claim();
          if (ntiles == 1) __builtin_amdgcn_s_waitcnt(0);
        }
      }
      if (pass == 0) {
        const float l = halves_sum(l_part);
        const bool over = !(l <= __builtin_exp2f(OVERFLOW_LOG2));
        if (__ballot(over) && lane == 0) s_over[over_slot] = 1;
        __syncthreads();
        if (!__builtin_amdgcn_readfirstlane(s_over[over_slot])) break;
      } else if (sweep) {
        const float mx = halves_max(lmax);
        m_ref = (mx == NEG_INF) ? 0.f : mx * a.scale_log2;
        __syncthreads();
      } else {
        __syncthreads();
      }
    }

    // what the epilogue needs of this item, then the next item's first tiles
    // (into K 0 and V 0: every wave is done with the tile buffers)
    const int e_h = i_h, e_c = i_c, e_qb = i_qb, e_qn = i_qn, e_entry0 = i_entry0;
    const bool more = idx_n >= 0;
    over_slot ^= 1;
    if (more) {
      begin();
      idx_n = __builtin_amdgcn_readfirstlane(s_items[parity]);
      parity ^= 1;
    }
    {
      int ln = lane;                     // opaque, as in load_q
      asm volatile("" : "+v"(ln));
      const int l32 = ln & 31, g = ln >> 5, lane = ln;
      const int row_i = (wave * 32 + l32) / G, row_j = (wave * 32 + l32) % G;
      const bool loc = e_c < 0;
      const float l = halves_sum(l_part);
      const float inv = (l > 0.f) ? 1.0f / l : 0.f;
      {
        const float lse = (l > 0.f) ? (m_ref + log2f(l)) * 0.69314718055994531f : NEG_INF;
        const float* lbase;
        int lbytes, loff;
        if (loc) {
          lbase = a.local_lse ? a.local_lse : reinterpret_cast<const float*>(a.q);
          lbytes = a.local_lse ? a.Qc * a.Hq * 4 : 0;
          loff = ((e_qb + row_i) * a.Hq + e_h * G + row_j) * 4;
        } else {
          lbase = a.part_lse + (int64_t)e_entry0 * G;
          lbytes = e_qn * G * 4;
          loff = (row_i * G + row_j) * 4;
        }
        const __amdgpu_buffer_rsrc_t lrsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void*)uniform_ptr(reinterpret_cast<const bf16_t*>(lbase)), 0, lbytes, BUFFER_CONFIG);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(lse), lrsrc,
                                              (row_i < e_qn && g == 0) ? loff : OUT_OF_RANGE, 0, 0);
      }
      // half rows through this wave's slice of K 1 and V 1: 16-byte chunk c of
      // row r at c ^ (r % SC), whole chunks from a swap of the lane halves (as in
      // the form above), then whole row halves per store.  Every lane issues every
      // store, a lane without a row past the range, where it is dropped: the
      // next item's first wait counts them.
      unsigned char* stage = smem_attn + S::TILE_BYTES * ((wave >> 1) ? 3 : 1) + (wave & 1) * (S::TILE_BYTES / 2);
      const bf16_t* obase = loc ? a.local_o + (int64_t)e_qb * a.lo_sq + (int64_t)(e_h * G) * a.lo_sh
                                : a.part_o + (int64_t)e_entry0 * G * D;
      const int64_t obytes = loc ? ((int64_t)(e_qn - 1) * a.lo_sq + (int64_t)(G - 1) * a.lo_sh + D) * 2
                                 : (int64_t)e_qn * G * D * 2;
      const __amdgpu_buffer_rsrc_t orsrc =
          __builtin_amdgcn_make_buffer_rsrc((void*)uniform_ptr(obase), 0, (int)obytes, BUFFER_CONFIG);
      const uint32_t osq = loc ? (uint32_t)(a.lo_sq * 2) : G * D * 2, osh = loc ? (uint32_t)(a.lo_sh * 2) : D * 2;
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
        for (int dd = 0; dd < DT / 2; ++dd)
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            const int dt = hf * (DT / 2) + dd;
            const int qa = 2 * p, qb2 = 2 * p + 1;
            const uint32_t a0 = pack2bf(o[dt][4 * qa + 0] * inv, o[dt][4 * qa + 1] * inv);
            const uint32_t a1 = pack2bf(o[dt][4 * qa + 2] * inv, o[dt][4 * qa + 3] * inv);
            const uint32_t b0 = pack2bf(o[dt][4 * qb2 + 0] * inv, o[dt][4 * qb2 + 1] * inv);
            const uint32_t b1 = pack2bf(o[dt][4 * qb2 + 2] * inv, o[dt][4 * qb2 + 3] * inv);
            const auto s0 = __builtin_amdgcn_permlane32_swap(a0, b0, false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(a1, b1, false, false);
            u32x4_t w;
            w.x = s0[0];
            w.y = s1[0];
            w.z = s0[1];
            w.w = s1[1];
            const int c = (4 * dd + 2 * p + g) ^ (l32 & (SC - 1));
            *reinterpret_cast<u32x4_t*>(stage + l32 * D + 16 * c) = w;
          }
        __builtin_amdgcn_wave_barrier();
        u32x4_t rows[HSTORES];
#pragma unroll
        for (int m = 0; m < HSTORES; ++m) {
          const int r = m * HROWS + lane / SC;
          rows[m] = *reinterpret_cast<const u32x4_t*>(stage + r * D + 16 * ((lane % SC) ^ (r & (SC - 1))));
        }
#pragma unroll
        for (int m = 0; m < HSTORES; ++m) {
          const int RR = wave * 32 + m * HROWS + lane / SC;
          const int i = RR / G, j = RR % G;
          const uint32_t off = (uint32_t)i * osq + (uint32_t)j * osh + hf * D + 16 * (lane % SC);
          __builtin_amdgcn_raw_buffer_store_b128(rows[m], orsrc, i < e_qn ? (int)off : OUT_OF_RANGE, 0, 2);
        }
        __builtin_amdgcn_wave_barrier();
        if (hf == 0) {
          // between the halves, when half of O's registers are free: the next item's Q rows,
          // and the counter's atomic for the item after the next two
          __builtin_amdgcn_sched_barrier(0);
          asm volatile("" ::: "memory");
          if (more) {
            request();
            load_q();
          }
          asm volatile("" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (!more) break;
    after_stores = true;
  }
}


// S6: per (query, KV head), one wave.  The reference folds the query's
// partials into the window's result one cluster at a time (online
// log-sum-exp, cluster order).  Here the wave first lists the query's entries
// (lanes test 64 clusters at once), takes the maximum of all the LSEs, and then
// sums exp(lse - max)-weighted partials with four entries' loads in flight, so
// no load waits on the previous fold.  The result is the same merge, rounded
// once instead of per step.  Each lane owns E = G*D/64 consecutive values of
// one head.
constexpr int COMBINE_MAX_LIST = 1024;   // entries per (query, head): at most C

template <int E>
__device__ __forceinline__ void load_bf16_row(const bf16_t* src, float (&v)[E]) {
  if constexpr (E % 8 == 0) {
#pragma unroll
    for (int k = 0; k < E / 8; ++k) {
      const u32x4_t w = *reinterpret_cast<const u32x4_t*>(src + 8 * k);
      const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        v[8 * k + 2 * t] = __uint_as_float(ww[t] << 16);
        v[8 * k + 2 * t + 1] = __uint_as_float(ww[t] & 0xffff0000u);
      }
    }
  } else {
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = bf2f(src[e]);
  }
}

template <int D, int G>
__global__ __launch_bounds__(256) void combine_kernel(
    const int32_t* __restrict__ qmask, const int32_t* __restrict__ nvis,
    const int32_t* __restrict__ rev_indptr, const int32_t* __restrict__ qrank,
    const bf16_t* __restrict__ part_o, const float* __restrict__ part_lse,
    const bf16_t* __restrict__ local_o, int64_t lo_sq, int64_t lo_sh,
    const float* __restrict__ local_lse, bf16_t* __restrict__ out, int64_t out_sq, int64_t out_sh,
    float* __restrict__ out_lse, int Qc, int Hkv, int C, const int32_t* __restrict__ skip) {
  constexpr int E = G * D / 64;
  if (skip && *skip) return;   // the chunk's partials passed their buffer: it runs again
  static_assert(E >= 1 && D % E == 0, "lane share");
  __shared__ int s_list[4][COMBINE_MAX_LIST];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t gw = (int64_t)blockIdx.x * 4 + wave;
  if (gw >= (int64_t)Qc * Hkv) return;
  const int qi = (int)(gw / Hkv), h = (int)(gw % Hkv);
  const int j = (lane * E) / D, d0 = (lane * E) % D;
  const int Hq = Hkv * G;
  int* list = s_list[wave];

  // the query's entries, in cluster order
  const int32_t* qm = qmask + ((int64_t)qi * Hkv + h) * (C / 32);
  const int32_t* qr = qrank + ((int64_t)qi * Hkv + h) * C;
  const uint64_t below = (1ull << lane) - 1;
  int n = 0;
  for (int c0 = 0; c0 < C; c0 += 64) {
    const int c = c0 + lane;
    bool sel = false;
    int entry = 0;
    if (c < C && (((uint32_t)qm[c >> 5] >> (c & 31)) & 1u) && nvis[h * C + c] > 0) {
      sel = true;
      entry = rev_indptr[h * C + c] + qr[c];
    }
    const uint64_t m = __ballot(sel);
    if (sel) list[n + __popcll(m & below)] = entry;
    n += __popcll(m);
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  // the largest LSE: the window's and every partial's
  const float lse_w = local_lse[(int64_t)qi * Hq + h * G + j];
  float mx = lse_w;
  for (int k = 0; k < n; k += 4) {
    float l4[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) l4[u] = k + u < n ? part_lse[(int64_t)list[k + u] * G + j] : -INFINITY;
#pragma unroll
    for (int u = 0; u < 4; ++u) mx = fmaxf(mx, l4[u]);
  }

  float acc[E];
  float den;
  {
    float v[E];
    load_bf16_row<E>(local_o + (int64_t)qi * lo_sq + (int64_t)(h * G + j) * lo_sh + d0, v);
    den = expf(lse_w - mx);
#pragma unroll
    for (int e = 0; e < E; ++e) acc[e] = v[e] * den;
  }
  for (int k = 0; k < n; k += 4) {
    float v[4][E], wt[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool ok = k + u < n;
      const int64_t entry = ok ? list[k + u] : 0;
      wt[u] = ok ? part_lse[entry * G + j] : -INFINITY;
      if (ok) load_bf16_row<E>(part_o + (entry * G + j) * D + d0, v[u]);
      else
#pragma unroll
        for (int e = 0; e < E; ++e) v[u][e] = 0.f;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float w = expf(wt[u] - mx);
      den += w;
#pragma unroll
      for (int e = 0; e < E; ++e) acc[e] = fmaf(v[u][e], w, acc[e]);
    }
  }
  const float inv = 1.0f / fmaxf(den, 1e-30f);
  bf16_t* dst = out + (int64_t)qi * out_sq + (int64_t)(h * G + j) * out_sh + d0;
  if constexpr (E % 8 == 0) {
#pragma unroll
    for (int k = 0; k < E / 8; ++k) {
      u32x4_t w;
      w.x = pack2bf(acc[8 * k + 0] * inv, acc[8 * k + 1] * inv);
      w.y = pack2bf(acc[8 * k + 2] * inv, acc[8 * k + 3] * inv);
      w.z = pack2bf(acc[8 * k + 4] * inv, acc[8 * k + 5] * inv);
      w.w = pack2bf(acc[8 * k + 6] * inv, acc[8 * k + 7] * inv);
      __builtin_nontemporal_store(w, reinterpret_cast<u32x4_t*>(dst + 8 * k));
    }
  } else {
#pragma unroll
    for (int e = 0; e < E; ++e) dst[e] = f2bf(acc[e] * inv);
  }
  if (out_lse && (lane * E) % D == 0) out_lse[(int64_t)qi * Hq + h * G + j] = mx + logf(den);
}

int compute_units() {
  static int units = 0;
  if (!units) {
    int dev = 0, cus = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    units = cus > 0 ? cus : 256;
  }
  return units;
}

// Launches one of the two forms with a grid that fills the GPU (or the caller's).
using AttnKernel = void (*)(AttnArgs);
template <int D>
int launch_attn_kernel(AttnKernel kernel, int& auto_grid, const AttnArgs& a, int grid, hipStream_t stream) {
  const size_t lds = AttnTileShape<D>::LDS_BYTES;
  if (!auto_grid) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return SBSA_ERR_UNSUPPORTED;
    int occ = 0;
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, (const void*)kernel, 256, lds);
    auto_grid = compute_units() * (occ > 0 ? occ : 1);
  }
  hipLaunchKernelGGL(kernel, dim3(grid > 0 ? grid : auto_grid), dim3(256), lds, stream, a);
  return SBSA_OK;
}

// Which form.  A caller that asks for room for other streams' kernels (grid < 0) gets the
// one-block form, which leaves registers and LDS on every compute unit: the layer asks for
// it for the dense chunks that run beside its index build (the other form holds every
// register, so the build would follow it: prefill of 32768 5.5 ms with the one-block dense
// chunks, 6.8 with these; of 131072 42.1 and 42.7).  An explicit grid gets the two-block form.
// Otherwise (grid 0) by how much the second block of a compute unit has to do, one item
// alone being quicker in the one-block form.  Attention alone, one MI355X, one-block against
// two-block us, by the chunk's window items (T) and the 256 compute units (U):
//   D = 128 with 4 or 8 heads per KV head: two blocks of the one-block form share a unit (its
//     253 registers; 258 and 264 with 1 and 2 heads), and it is the quicker at every size:
//     dense T 88 / 512 / 1024: 177 / 355 / 1455 and 244 / 383 / 1505, sparse, 46 chunks of
//     200 to 8192 queries: 0.67 to 1.01 of the two-block form's time.
//   D = 128 with 1 or 2 heads: two-block from T = 5/4 U.  Dense T 256 / 320 / 376 / 512 / 1024:
//     512 / 358 / 347 / 866 / 1734 and 727 / 358 / 313 / 798 / 1446; sparse T 256: 211-712 and
//     260-960 (one chunk of three 447 and 390), T 376 / 512 / 1024: 391 / 435 / 1654 and
//     348 / 372 / 1194.
//   D = 256 dense: two-block once a unit has a second item.  T 188 / 256 / 264 / 1024: 313 / 344 /
//     531 / 2972 and 362 / 385 / 388 / 2569.
//   D = 256 sparse: with few queries a launch ends with its longest cluster items, alone on
//     their units, so the clusters' mean length up to the window counts as well.  111 chunks of
//     200 to 8192 queries, 8K to 390K positions: with 4 or 8 heads per KV head (more items of a
//     cluster for the same queries) two-block from T = U + 1 or up to a length of 256, mean 1.04 of
//     the better form's time (by T alone 1.06; one-block always 1.11; from T = U/2 1.02, but
//     single chunks then lose much: 1115 queries at 90000 453 -> 533 us); with 1 or 2 heads by T
//     alone, 1.01 (with the length 1.05).
// A window's rows whose output offsets pass 31 bits go to the one-block form too.
template <int D, int G>
int launch_attn(const AttnArgs& a, int grid, hipStream_t stream) {
  static int pair_grid = 0, items_grid = 0;
  const int64_t window_out = ((int64_t)(PREFILL_ROWS / G - 1) * a.lo_sq + (int64_t)(G - 1) * a.lo_sh + D) * 2;
  const bool offsets_fit = window_out < INT32_MAX && (int64_t)a.Qc * a.Hq * 4 < INT32_MAX;
  const int64_t tiles = (a.Qc + PREFILL_ROWS / G - 1) / (PREFILL_ROWS / G) * (int64_t)a.Hkv;
  const int64_t units = compute_units();
  bool two_blocks = tiles > units;
  if (D == 128) two_blocks = G <= 2 && 4 * tiles >= 5 * units;
  if (D == 256 && G >= 4 && a.nvis) two_blocks = tiles > units || a.wstart <= (int64_t)a.C * 256;
  const bool pair = grid > 0 || (grid == 0 && two_blocks);
  if (pair && offsets_fit) return launch_attn_kernel<D>(attn_pair_kernel<D, G>, pair_grid, a, grid, stream);
  return launch_attn_kernel<D>(attn_items_kernel<D, G>, items_grid, a, grid, stream);
}

template <int D, int G>
int launch_combine(const int32_t* qmask, const int32_t* nvis, const int32_t* rev_indptr,
                   const int32_t* qrank, const bf16_t* part_o, const float* part_lse,
                   const bf16_t* local_o, int64_t lo_sq, int64_t lo_sh, const float* local_lse,
                   bf16_t* out, int64_t out_sq, int64_t out_sh, float* out_lse, int Qc, int Hkv,
                   int C, const int32_t* skip, hipStream_t stream) {
  int64_t waves = (int64_t)Qc * Hkv;
  hipLaunchKernelGGL((combine_kernel<D, G>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0,
                     stream, qmask, nvis, rev_indptr, qrank, part_o, part_lse, local_o, lo_sq,
                     lo_sh, local_lse, out, out_sq, out_sh, out_lse, Qc, Hkv, C, skip);
  return SBSA_OK;
}

#define SBSA_DISPATCH_DG(D_, G_, FN, ...)                            \
  do {                                                               \
    if (D_ == 128 && G_ == 1) return FN<128, 1>(__VA_ARGS__);        \
    if (D_ == 128 && G_ == 2) return FN<128, 2>(__VA_ARGS__);        \
    if (D_ == 128 && G_ == 4) return FN<128, 4>(__VA_ARGS__);        \
    if (D_ == 128 && G_ == 8) return FN<128, 8>(__VA_ARGS__);        \
    if (D_ == 256 && G_ == 1) return FN<256, 1>(__VA_ARGS__);        \
    if (D_ == 256 && G_ == 2) return FN<256, 2>(__VA_ARGS__);        \
    if (D_ == 256 && G_ == 4) return FN<256, 4>(__VA_ARGS__);        \
    if (D_ == 256 && G_ == 8) return FN<256, 8>(__VA_ARGS__);        \
    return SBSA_ERR_UNSUPPORTED;                                     \
  } while (0)

int attn_dispatch(int D, int G, const AttnArgs& a, int grid, hipStream_t stream) {
  SBSA_DISPATCH_DG(D, G, launch_attn, a, grid, stream);
}

int combine_dispatch(int D, int G, const int32_t* qmask, const int32_t* nvis,
                     const int32_t* rev_indptr, const int32_t* qrank, const bf16_t* part_o,
                     const float* part_lse, const bf16_t* local_o, int64_t lo_sq, int64_t lo_sh,
                     const float* local_lse, bf16_t* out, int64_t out_sq, int64_t out_sh,
                     float* out_lse, int Qc, int Hkv, int C, const int32_t* skip,
                     hipStream_t stream) {
  SBSA_DISPATCH_DG(D, G, launch_combine, qmask, nvis, rev_indptr, qrank, part_o, part_lse, local_o,
                   lo_sq, lo_sh, local_lse, out, out_sq, out_sh, out_lse, Qc, Hkv, C, skip, stream);
}

}  // namespace

extern "C" {

#ifdef SBSA_ATTN_PROBE
int sbsa_probe_read(void* host, size_t bytes) {
  if (bytes > sizeof(g_attn_probe)) bytes = sizeof(g_attn_probe);
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(g_attn_probe), bytes, 0, hipMemcpyDeviceToHost) == hipSuccess ? 0 : 3;
}
#endif

int sbsa_prefill_item_rows(void) { return PREFILL_ROWS; }

int sbsa_prefill_attend(const void* q, int64_t q_sq, int64_t q_sh, int num_queries,
                        int num_q_heads, int num_kv_heads, int dim, const void* packed,
                        int64_t packed_len, const void* k_orig, const void* v_orig, int64_t o_st,
                        int64_t o_sh, const int32_t* indptr, const int32_t* nvis, int num_clusters,
                        const int32_t* rev_indptr, const int32_t* qvals, const void* items,
                        int32_t* queue, void* part_o, float* part_lse,
                        void* local_o, int64_t lo_sq, int64_t lo_sh, float* local_lse,
                        int64_t chunk_start, int64_t wstart, float sm_scale, int grid,
                        hipStream_t stream) {
  if (!q || !k_orig || !v_orig || !items || !queue || !local_o) return SBSA_ERR_ARG;
  if (num_kv_heads < 1 || num_q_heads % num_kv_heads) return SBSA_ERR_ARG;
  if (q_sq % 8 || q_sh % 8 || o_st % 8 || o_sh % 8 || lo_sq % 4 || lo_sh % 4) return SBSA_ERR_ARG;
  if (chunk_start < wstart || wstart < 0) return SBSA_ERR_ARG;
  // The tile loads address K/V through raw buffer resources whose range (the rows
  // left from a tile's first row, in bytes) is 32-bit: the longest row range a work
  // item can read, the window from wstart to the chunk's last query or a whole packed
  // run, must stay below 4 GiB.
  const int64_t window_bytes = (chunk_start + num_queries - wstart) * o_st * 2;
  const int64_t packed_bytes = packed ? packed_len * num_kv_heads * (int64_t)dim * 2 : 0;
  if (window_bytes >= (int64_t(1) << 32) || packed_bytes >= (int64_t(1) << 32))
    return SBSA_ERR_UNSUPPORTED;
  AttnArgs a;
  a.q = (const bf16_t*)q;
  a.q_sq = q_sq;
  a.q_sh = q_sh;
  a.packed = (const bf16_t*)packed;
  a.packed_len = packed_len;
  a.korig = (const bf16_t*)k_orig;
  a.vorig = (const bf16_t*)v_orig;
  a.o_st = o_st;
  a.o_sh = o_sh;
  a.indptr = indptr;
  a.nvis = nvis;
  a.rev_indptr = rev_indptr;
  a.qvals = qvals;
  a.items = (const PrefillItem*)items;
  a.queue = queue;
  a.part_o = (bf16_t*)part_o;
  a.part_lse = part_lse;
  a.local_o = (bf16_t*)local_o;
  a.lo_sq = lo_sq;
  a.lo_sh = lo_sh;
  a.local_lse = local_lse;
  a.Hkv = num_kv_heads;
  a.C = num_clusters;
  a.Hq = num_q_heads;
  a.Qc = num_queries;
  a.chunk_start = chunk_start;
  a.wstart = wstart;
  a.scale_log2 = sm_scale * 1.4426950408889634f;
#ifdef SBSA_ATTN_PROBE
  static int probe_next = 0;
  a.probe_slot = probe_next++;
#endif
  int rc = attn_dispatch(dim, num_q_heads / num_kv_heads, a, grid, stream);
  if (rc) return rc;
  SBSA_CHECK_LAUNCH();
  return SBSA_OK;
}

int sbsa_prefill_combine(const int32_t* qmask, const int32_t* nvis, const int32_t* rev_indptr,
                         const int32_t* qrank, const void* part_o, const float* part_lse,
                         const void* local_o, int64_t lo_sq, int64_t lo_sh, const float* local_lse,
                         void* out, int64_t out_sq, int64_t out_sh, float* out_lse,
                         int num_queries, int num_q_heads, int num_kv_heads, int dim,
                         int num_clusters, const int32_t* skip, hipStream_t stream) {
  if (!qmask || !nvis || !rev_indptr || !qrank || !local_o || !local_lse || !out) return SBSA_ERR_ARG;
  if (num_kv_heads < 1 || num_q_heads % num_kv_heads || num_clusters % 32) return SBSA_ERR_ARG;
  if (num_clusters > COMBINE_MAX_LIST) return SBSA_ERR_UNSUPPORTED;
  // rows are read and written in 16-byte pieces when a lane's share of a head is a
  // multiple of 8 values: every row start must then be 16-byte aligned
  if ((num_q_heads / num_kv_heads) * dim % 512 == 0 &&
      (out_sq % 8 || out_sh % 8 || lo_sq % 8 || lo_sh % 8 || ((uintptr_t)out & 15) ||
       ((uintptr_t)local_o & 15)))
    return SBSA_ERR_ARG;
  if (num_queries == 0) return SBSA_OK;
  int rc = combine_dispatch(dim, num_q_heads / num_kv_heads, qmask, nvis, rev_indptr, qrank,
                            (const bf16_t*)part_o, part_lse, (const bf16_t*)local_o, lo_sq, lo_sh,
                            local_lse, (bf16_t*)out, out_sq, out_sh, out_lse, num_queries,
                            num_kv_heads, num_clusters, skip, stream);
  if (rc) return rc;
  SBSA_CHECK_LAUNCH();
  return SBSA_OK;
}

}  // extern "C"
