// Paged quantized-KV decode attention on gfx950 (one query token per sequence, GQA).
//
// Cache layout (this build's; the reference has no quantized-KV decode kernel -- its nearest relative is the paged
// fp8 gather + blockwise attention with log-sum-exp merge of xpu/exl3xpu/fp8kv_prefill.py:73-117):
//   k_cache, v_cache: 8-bit int8 [pages][Hkv][16][D], or 4-bit packed uint8 [pages][Hkv][16][D/2] (element 2i in
//                     the low nibble, 2i+1 in the high nibble, two's complement);
//   k_scale, v_scale: fp16 [pages][Hkv]; value = code * scale;
//   page_table int32 [B][max_pages]; seq_lens int32 [B]; q fp16 [B][Hq][D]; out fp16 [B][Hq][D]; D = 128.
//   Query head h reads KV head h / (Hq / Hkv).
//
// kv_decode_kernel: grid (chunks of pages, Hkv, sequences), W = 8 (or 4) waves.  Wave w takes pages w, w+W, ...
// of its workgroup's chunk, with the next page's codes in flight while it works on the current one, and keeps an
// online softmax for the G = Hq/Hkv query heads (G <= 16; MFMA columns G..15 are idle).  Per 16-token page --
// exactly one 16-wide MFMA block, so the page's two scales are wave-uniform:
//   S^T = K Q^T     4 x MFMA 16x16x32 f16.  A = the page's 16 keys (lane: key l%16, 32 dims), B = Q^T (lane: query
//                   l%16, the same 32 dims in the same order; loaded once).  C lane: query l%16, keys 4(l/16)..+3;
//   P^T             that C layout is already the B operand of the next MFMA; P' = p * v_scale rounded to fp16;
//   O^T += V^T P^T  8 x MFMA 16x16x16 f16.  A = V^T (lane: dim 8(l%16) + db for block db, keys 4(l/16)..+3): the
//                   lane loads 8 bytes of each of its 4 keys and transposes the 4 x 4 byte blocks with v_perm.
//                   C lane: dims 32(l/16) .. +31 of query l%16 over the 8 blocks.
// Codes become fp16 without conversions: code + bias (bias 128 / 8, one xor) as the low byte (nibble) under 0x64 is
// the fp16 1024 + bias + code.  V: one packed fp16 subtract of 1024 + bias leaves the code exactly (integers of
// magnitude <= 128 are exact in fp16) before it is accumulated.  K: the MFMA takes the biased codes and the page's
// logits subtract (1024 + bias) * sum(q) -- a per-page correction, never accumulated across pages.  The W waves
// merge their (m, l, O) in LDS; the workgroup writes its chunk's partial state and kv_merge_kernel combines the
// chunks by log-sum-exp, in chunk order (deterministic).  Logits are kept in the base-2 domain (scale * log2 e).
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <cstdlib>

#include "exl3_api.hpp"
#include "exl3_device.hpp"

namespace exl3 {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef uint32_t kv_u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t kv_u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kKvWaves = 8;     // waves per decode workgroup (4 when the LDS merge of 8 would not fit 64 KB)
constexpr int kMergeWaves = 4;  // waves per kv_merge_kernel workgroup
constexpr int kHeadDim = 128;
constexpr int kPage = 16;
constexpr int kMaxGroup = 16;

// 4 biased code bytes -> 4 fp16 (1024 + byte - sub); the fp16 subtract is exact for the code range
__device__ __forceinline__ half4_t codes_f16(uint32_t u, _Float16 sub) {
  const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, u, 0x05010400u);  // bytes: u0, 0x64, u1, 0x64
  const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, u, 0x05030402u);  // bytes: u2, 0x64, u3, 0x64
  return __builtin_bit_cast(half4_t, kv_u32x2_t{lo, hi}) - half4_t{sub, sub, sub, sub};
}

// 4 x 4 byte transpose: in[i] holds bytes 0..3 of row i; out[j] holds byte j of rows 0..3 (row order)
__device__ __forceinline__ void transpose4x4(const uint32_t in[4], uint32_t out[4]) {
  const uint32_t a = __builtin_amdgcn_perm(in[1], in[0], 0x05010400u);  // r0b0 r1b0 r0b1 r1b1
  const uint32_t b = __builtin_amdgcn_perm(in[3], in[2], 0x05010400u);  // r2b0 r3b0 r2b1 r3b1
  const uint32_t c = __builtin_amdgcn_perm(in[1], in[0], 0x07030602u);  // r0b2 r1b2 r0b3 r1b3
  const uint32_t d = __builtin_amdgcn_perm(in[3], in[2], 0x07030602u);  // r2b2 r3b2 r2b3 r3b3
  out[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);
  out[1] = __builtin_amdgcn_perm(b, a, 0x07060302u);
  out[2] = __builtin_amdgcn_perm(d, c, 0x05040100u);
  out[3] = __builtin_amdgcn_perm(d, c, 0x07060302u);
}

// reductions over the 4 lanes l, l^16, l^32, l^48 (the 16 keys of a page for one query): v_permlane16_swap and
// v_permlane32_swap with both operands x return (x of row r, x of row r^1) and (x of half h, x of half h^1)
__device__ __forceinline__ float max_over_groups(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum_over_groups(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Keeps the loads above it issued here: otherwise they are free to sink to their first use, which turns the
// next-page prefetch into a load-and-wait.  Registers are not touched, so no wait is implied.  (The cache pointers
// carry no __restrict__: loads of restrict read-only memory count as invariant and would cross the fence.)
__device__ __forceinline__ void issue_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);  // and no instruction that waits on older loads is scheduled above them
}

// The codes one lane needs from one (page, kv head) block, and the block's scales.
template <int BITS>
struct KvRegs {
  static constexpr int ROW = BITS == 8 ? kHeadDim : kHeadDim / 2;  // bytes per token row
  static constexpr int KW = BITS == 8 ? 8 : 4;                      // K dwords per lane
  static constexpr int VW = BITS == 8 ? 8 : 4;                      // V dwords per lane
  uint32_t k[KW], v[VW];
  uint32_t ksw, vsw;  // the block's two fp16 scales, each zero-extended in a register of its own

  // lane (n, g): K row n, bytes [ROW/4 * g, +ROW/4); V rows 4g .. 4g+3, bytes [ROW/16 * n, +ROW/16)
  __device__ __forceinline__ void load(const uint8_t* kblk, const uint8_t* vblk, const uint16_t* ksc,
                                       const uint16_t* vsc, size_t bi, int n, int g) {
    // The scales first, each zero-extended into a 32-bit register that nothing copies or packs before the scales are
    // used: packed as fp16 halves of one register (a copy that must wait for both loads), and issued as the page's
    // youngest loads, their wait covered every load in flight.
    ksw = ksc[bi];
    vsw = vsc[bi];
    const kv_u32x4_t* kp = reinterpret_cast<const kv_u32x4_t*>(kblk + n * ROW + (ROW / 4) * g);
    if constexpr (BITS == 8) {
      const kv_u32x4_t a = kp[0], b = kp[1];
      k[0] = a.x, k[1] = a.y, k[2] = a.z, k[3] = a.w, k[4] = b.x, k[5] = b.y, k[6] = b.z, k[7] = b.w;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const kv_u32x2_t t = *reinterpret_cast<const kv_u32x2_t*>(vblk + (4 * g + i) * ROW + 8 * n);
        v[i] = t.x, v[4 + i] = t.y;
      }
    } else {
      const kv_u32x4_t a = kp[0];
      k[0] = a.x, k[1] = a.y, k[2] = a.z, k[3] = a.w;
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = *reinterpret_cast<const uint32_t*>(vblk + (4 * g + i) * ROW + 4 * n);
    }
  }
  __device__ __forceinline__ _Float16 kscale() const { return __builtin_bit_cast(_Float16, (uint16_t)ksw); }
  __device__ __forceinline__ _Float16 vscale() const { return __builtin_bit_cast(_Float16, (uint16_t)vsw); }

  // K fragment c, biased: 1024 + bias + code (bias 128 / 8; removed after the MFMA, per page, from the query sums).
  // Dims of lane group g, in the order the Q fragment uses: 8 bits, dwords 2c, 2c+1 = dims 32g + 8c + 0..7;
  // 4 bits, dword c = dims 32g + 8c + 0..7 as nibbles 0..7, taken in pairs (s, s+4) straight into fp16 halves.
  __device__ __forceinline__ half8_t kfrag(int c) const {
    if constexpr (BITS == 8) {
      const uint32_t x = k[2 * c] ^ 0x80808080u, y = k[2 * c + 1] ^ 0x80808080u;
      return __builtin_bit_cast(half8_t, kv_u32x4_t{__builtin_amdgcn_perm(0x64646464u, x, 0x05010400u),
                                                     __builtin_amdgcn_perm(0x64646464u, x, 0x05030402u),
                                                     __builtin_amdgcn_perm(0x64646464u, y, 0x05010400u),
                                                     __builtin_amdgcn_perm(0x64646464u, y, 0x05030402u)});
    } else {
      const uint32_t x = k[c];
      return __builtin_bit_cast(half8_t, kv_u32x4_t{(x & 0x000F000Fu) ^ 0x64086408u, ((x >> 4) & 0x000F000Fu) ^ 0x64086408u,
                                                     ((x >> 8) & 0x000F000Fu) ^ 0x64086408u,
                                                     ((x >> 12) & 0x000F000Fu) ^ 0x64086408u});
    }
  }

  // V^T fragments: vt[db] = the 4 keys' biased codes at dim 8n + db
  __device__ __forceinline__ void vtrans(uint32_t vt[8]) const {
    if constexpr (BITS == 8) {
      uint32_t lo[4] = {v[0] ^ 0x80808080u, v[1] ^ 0x80808080u, v[2] ^ 0x80808080u, v[3] ^ 0x80808080u};
      uint32_t hi[4] = {v[4] ^ 0x80808080u, v[5] ^ 0x80808080u, v[6] ^ 0x80808080u, v[7] ^ 0x80808080u};
      transpose4x4(lo, vt);
      transpose4x4(hi, vt + 4);
    } else {
      uint32_t tb[4];
      transpose4x4(v, tb);  // tb[j]: byte j (dims 8n + 2j, 8n + 2j + 1) of the 4 keys
#pragma unroll
      for (int j = 0; j < 4; j++) {
        vt[2 * j] = (tb[j] & 0x0F0F0F0Fu) ^ 0x08080808u;
        vt[2 * j + 1] = ((tb[j] >> 4) & 0x0F0F0F0Fu) ^ 0x08080808u;
      }
    }
  }
};

template <int BITS>
struct KvState {
  float m = -INFINITY, l = 0.f;  // running max (base 2) and sum for query n
  float4_t o[8];

  // One page: logits in base 2 are (S - kbias * qsum) * k_scale * qk_scale.  The reference max m moves only when a
  // page max passes it by more than 4 (then every p <= 16, and P' = p * v_scale stays far inside fp16), so O and l
  // are rarely rescaled; (m, l, O) stay consistent for the merges either way.
  __device__ __forceinline__ void process(const KvRegs<BITS>& r, const half8_t qf[4], float qsum, int key0, int L,
                                          float qk_scale, int g) {
    constexpr float kBias = BITS == 8 ? 1152.0f : 1032.0f;
    float4_t st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; c++) st = __builtin_amdgcn_mfma_f32_16x16x32_f16(r.kfrag(c), qf[c], st, 0, 0, 0);
    const float sc = (float)r.kscale() * qk_scale;
    const float off = -kBias * qsum * sc;
    float sv[4];
#pragma unroll
    for (int i = 0; i < 4; i++) sv[i] = __builtin_fmaf(st[i], sc, off);
    if (key0 + kPage > L) {  // the sequence ends inside this page
#pragma unroll
      for (int i = 0; i < 4; i++) sv[i] = key0 + 4 * g + i < L ? sv[i] : -INFINITY;
    }
    const float pm = max_over_groups(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3])));
    if (__builtin_amdgcn_ballot_w64(pm > m + 4.f)) {
      const float m_new = fmaxf(m, pm);
      const float alpha = __builtin_amdgcn_exp2f(m - m_new);  // 0 on the first page (m = -inf)
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int db = 0; db < 8; db++) o[db] *= alpha;
    }
    const float vs = (float)r.vscale();
    float psum = 0.f;
    half4_t pf;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float p = __builtin_amdgcn_exp2f(sv[i] - m);
      psum += p;
      pf[i] = (_Float16)(p * vs);
    }
    l += sum_over_groups(psum);
    uint32_t vt[8];
    r.vtrans(vt);
#pragma unroll
    for (int db = 0; db < 8; db++)
      o[db] = __builtin_amdgcn_mfma_f32_16x16x16f16(codes_f16(vt[db], (_Float16)kBias), pf, o[db], 0, 0, 0);
  }
};

// ---- split of a batch over the workgroups ----------------------------------------------------------------------------
// The host knows the page table's width but not the lengths.  Chunks of a fixed share of the table leave most
// workgroups idle on a ragged batch (or a table wider than its sequences): the longest sequence's chunks set the time.
// So for up to 64 sequences every wave reads all lengths (one per lane) and derives the same plan: chunks of up to
// `cp` pages, cp the batch's pages over the number of workgroups aimed at, so that a long sequence takes many chunks
// and a short one a single chunk, which writes its output directly.  Measured against the fixed plan (a step of two
// calls, 40 / 8 heads): 16 sequences of 256 .. 4096 tokens in an 8k table, 8 bits 71.4 -> 49.1 us; 7 sequences of
// 4681 .. 32768 tokens, 4 bits 117-129 -> 76.6 us.
// Where the fixed plan's longest chunk is no longer than that (sequences that fill their table, or lie close together),
// the fixed plan stands: 26 sequences of 8 heads, 53-100 % of 7072 tokens, 8 bits 57.9 us by it, 63.7 split by lengths; 16
// full sequences of 4k 26.6 -> 26.0, one of 4224 tokens 10.2 -> 8.7.  Having read the lengths costs 0.3-0.7 us per call
// then (decode and merge; a kernel that does not read them takes 25.4 and 8.3).
struct KvSplit {
  int batch, max_tokens;
  int target, slots;        // by lengths: aiming at `target` chunks per kv head, room for `slots` partial states per
                            // (kv head, query head)
  float inv_target, inv_slots, inv_heads;
  float worth;              // by lengths where worth * the longest chunk of the fixed plan exceeds the chunks by length
  int chunk_pages, chunks;  // the fixed plan: `chunks` chunks of chunk_pages pages per sequence
};

__device__ __forceinline__ int wave_scan(int v) {  // inclusive prefix sum over the 64 lanes
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);   // row_shr:1, 2, 4, 8: inside each row of 16
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
  return v;
}
__device__ __forceinline__ int wave_total(int v) { return __builtin_amdgcn_readlane(wave_scan(v), 63); }

// The plan of a batch of up to 64 sequences, one per lane: its length, pages, chunks, and the inclusive prefix sums of
// the chunks (low half) and of the partial states, the chunks of split sequences (high half; both stay below 2^15).
// Chunk counts come from an approximate reciprocal: one more chunk than needed only leaves the last one short or empty,
// and the pages per chunk (kv_per) are exact in the count.
struct KvBatch {
  int len, pages, chunks, sums;
};

// Pages per chunk of a sequence of `pages` pages in `chunks` chunks, a multiple of `waves`
__device__ __forceinline__ int kv_per(int pages, int chunks, int waves) {
  return (int)(((unsigned)(pages + chunks - 1) / (unsigned)chunks + waves - 1) & -(unsigned)waves);
}

// The plan by lengths; false: the fixed plan (only len and pages are set)
__device__ __forceinline__ bool kv_batch(const KvSplit& s, const int* __restrict__ seq_lens, int waves, KvBatch& k) {
  const int lane = threadIdx.x & 63;
  asm volatile("" ::"s"(s.batch), "s"(s.max_tokens), "s"(s.target), "s"(s.slots), "s"(s.inv_target), "s"(s.inv_slots),
               "s"(s.worth), "s"(s.chunks), "s"(s.chunk_pages), "s"(s.inv_heads), "s"(seq_lens));
  k.len = max(min(seq_lens[min(lane, s.batch - 1)], s.max_tokens), 0);
  k.len = lane < s.batch ? k.len : 0;
  k.pages = (k.len + kPage - 1) / kPage;
  const float np = (float)k.pages;
  auto chunks_of = [&](int cp) { return (int)__builtin_ceilf(np * __builtin_amdgcn_rcpf((float)cp)); };
  auto both = [](int c) { return c > 1 ? c * 0x10001 : c; };
  auto up = [&](float pages) { return (int)(((unsigned)(int)pages + waves) & -(unsigned)waves); };  // above `pages`
  // one sequence: every lane takes lane 0's value for the sum over the lanes
  auto scan = [&](int v) { return s.batch == 1 ? __builtin_amdgcn_readfirstlane(v) : wave_scan(v); };
  auto total_of = [&](int sums) { return __builtin_amdgcn_readlane(sums, 63); };
  const float total = (float)total_of(scan(k.pages));
  // the fixed plan's longest chunk, as it weighs, against an equal share of the batch
  const float longest = (float)min(k.pages, s.chunk_pages) * s.worth;
  auto any = [](bool b) { return __builtin_amdgcn_ballot_w64(b) != 0; };
  if (!any(longest > total * fmaxf(s.inv_target, s.inv_slots))) return false;
  const int live = __builtin_popcountll(__builtin_amdgcn_ballot_w64(k.pages > 0));
  // Chunks of an equal share of the batch, if that gives no more chunks than workgroups aimed at (one per CU: a CU
  // with two takes twice as long) and the partial states fit.  Each sequence's last chunk is short, so a ragged batch
  // needs longer ones: a share that leaves half or three quarters of a chunk per sequence is tried next, a whole one
  // always does.  With more sequences than that the share stands, unless the partial states don't fit; chunks of
  // three times the mean over the slots always fit (fewer than 2 n / cp + 1 chunks in a split sequence of n pages).
  const bool crowded = 2 * live > s.target;
  auto fits = [&](int sums) { return (sums >> 16) <= s.slots && (crowded || (sums & 0xFFFF) <= s.target); };
  const int share = up(__builtin_fmaf(total, s.inv_target, -0.5f));
  int cp = share;
  k.chunks = chunks_of(cp);
  k.sums = scan(both(k.chunks));
  if (!fits(total_of(k.sums))) {
    const float room = (float)max(min(s.target, s.slots) - live, 1);  // chunks left when each sequence wastes one
    auto leaving = [&](float part) { return up(total * __builtin_amdgcn_rcpf(__builtin_fmaf(part, (float)live, room))); };
    const int half = crowded ? share + share / 2 : leaving(0.5f), most = crowded ? 2 * share : leaving(0.25f);
    const int last = crowded ? up(fmaxf(3.f * total * s.inv_slots, 2.f * share)) : leaving(0.f);
    const int b = wave_total(both(chunks_of(half))), c = wave_total(both(chunks_of(most)));
    cp = fits(b) ? half : fits(c) ? most : last;
    k.chunks = chunks_of(cp);
    k.sums = wave_scan(both(k.chunks));
  }
  // With a CU for every workgroup of the fixed plan, chunks by lengths may still come out as long (unless every sequence
  // ends in its first chunk there, whose state would take the merge's detour).  Four workgroups of 4 waves share a CU:
  // there it also counts that chunks by lengths lie side by side in the grid, with no empty workgroups between them (20
  // sequences of 305-6094 tokens, 1 kv head, 8 bits: 510 chunks of 8 pages in both plans, 19.4 us fixed, 16.5 by lengths).
  return waves == 4 || s.slots > s.target || any(longest > (float)cp) || !any(k.pages > s.chunk_pages);
}

// A workgroup's chunk: pages [p0, p1) of sequence b of length len; slot: its partial state, -1 when it is the whole
// sequence; b = -1 past the last chunk.
struct KvChunk {
  int hk, b, len, p0, p1, slot;
};

// The fixed plan's workgroups are (chunk, kv head, sequence).
__device__ __forceinline__ KvChunk kv_fixed_chunk(const KvSplit& s, int len) {
  const int i = blockIdx.x, b = blockIdx.z;
  return KvChunk{(int)blockIdx.y, b, len, i * s.chunk_pages, (i + 1) * s.chunk_pages,
                 s.chunks > 1 ? b * s.chunks + i : -1};
}

// By lengths the kv head is the fast index of a workgroup's linear id and the chunk's number the slow one: workgroups
// past the last chunk then come last and take no CU from a chunk (with the chunk fast, 16 x 4k 26 -> 37 us).
__device__ __forceinline__ KvChunk kv_chunk_by_length(const KvSplit& s, int Hkv, int waves, const KvBatch& k) {
  const int id = blockIdx.x + s.chunks * (blockIdx.y + Hkv * blockIdx.z);
  const int index = __builtin_amdgcn_readfirstlane((int)(((float)id + 0.5f) * s.inv_heads));  // id / Hkv
  if (index >= (__builtin_amdgcn_readlane(k.sums, 63) & 0xFFFF)) return KvChunk{0, -1, 0, 0, 0, -1};
  const int at = __builtin_popcountll(__builtin_amdgcn_ballot_w64((k.sums & 0xFFFF) <= index));
  const int pages = __builtin_amdgcn_readlane(k.pages, at), chunks = __builtin_amdgcn_readlane(k.chunks, at);
  const int sums = __builtin_amdgcn_readlane(k.sums, at);
  const int c = index - ((sums & 0xFFFF) - chunks);
  const int per = chunks == 1 ? pages : kv_per(pages, chunks, waves);
  return KvChunk{id - index * Hkv, at, __builtin_amdgcn_readlane(k.len, at), c * per, (c + 1) * per,
                 chunks > 1 ? (sums >> 16) - chunks + c : -1};
}

template <int BITS, int DEPTH, int WAVES, bool BY_LENGTH>
__global__ __launch_bounds__(WAVES * 64) void kv_decode_kernel(
    const _Float16* __restrict__ q, const uint8_t* kc, const uint8_t* vc, const uint16_t* ksc, const uint16_t* vsc,
    int num_pages,
    const int* __restrict__ page_table, int max_pages, const int* __restrict__ seq_lens, int Hq, int Hkv,
    float qk_scale, KvSplit split, float* __restrict__ part_o, float* __restrict__ part_ml,
    _Float16* __restrict__ out) {
  constexpr int ROW = KvRegs<BITS>::ROW;
  extern __shared__ float red[];  // [WAVES][G][D + 1] then [WAVES][G][2]
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  KvChunk ch;
  if constexpr (BY_LENGTH) {
    KvBatch k;
    if (kv_batch(split, seq_lens, WAVES, k)) {
      ch = kv_chunk_by_length(split, Hkv, WAVES, k);
      if (ch.b < 0) return;
    } else {
      if ((int)blockIdx.z >= split.batch) return;
      ch = kv_fixed_chunk(split, __builtin_amdgcn_readlane(k.len, blockIdx.z));
    }
  } else {
    ch = kv_fixed_chunk(split, min(seq_lens[blockIdx.z], split.max_tokens));
  }
  const int hk = ch.hk, b = ch.b, L = ch.len;
  const int G = Hq / Hkv;
  const int l = threadIdx.x & 63;
  const int n = l & 15, g = l >> 4;

  // Q^T fragment of query n (zero for n >= G), dims in K-fragment order; qsum = sum of its 128 dims
  half8_t qf[4];
  float qpart = 0.f;
  {
    const _Float16* qrow = q + ((size_t)b * Hq + hk * G + min(n, G - 1)) * kHeadDim + 32 * g;
    const _Float16 live = n < G ? (_Float16)1.0f : (_Float16)0.0f;
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int d = BITS == 8 ? 8 * c + e : 8 * c + (e >> 1) + 4 * (e & 1);
        qf[c][e] = qrow[d] * live;
        qpart += (float)qf[c][e];
      }
  }
  const float qsum = sum_over_groups(qpart);

  KvState<BITS> s;
#pragma unroll
  for (int db = 0; db < 8; db++) s.o[db] = float4_t{0.f, 0.f, 0.f, 0.f};

  // this wave's pages: logical pages p0 + w, p0 + w + WAVES, ... below min(chunk end, pages of the sequence)
  const int p0 = ch.p0;
  const int p_end = min(ch.p1, (L + kPage - 1) / kPage);
  const int* ptab = page_table + (size_t)b * max_pages;
  const size_t blk_bytes = (size_t)kPage * ROW;
  int lp = p0 + w;
  if (lp < p_end) {
    // DEPTH register sets rotate: DEPTH - 1 pages are in flight while one is worked on.  The trip is unrolled over
    // the sets so each keeps its registers (no copies that would wait on their loads).  Loads past the wave's last
    // page repeat that page.  Out-of-range page ids are clamped into the cache (never dereferenced outside it).
    KvRegs<BITS> r[DEPTH];
    auto page_of = [&](int p) { return (size_t)min(max(ptab[p], 0), num_pages - 1) * Hkv + hk; };
    auto load = [&](KvRegs<BITS>& dst, int p) {
      const size_t bi = page_of(min(p, p_end - 1));
      dst.load(kc + bi * blk_bytes, vc + bi * blk_bytes, ksc, vsc, bi, n, g);
    };
#pragma unroll
    for (int j = 0; j < DEPTH - 1; j++) load(r[j], lp + j * WAVES);
    bool more = true;
    while (more) {
#pragma unroll
      for (int j = 0; j < DEPTH; j++) {
        if (more) {
          load(r[(j + DEPTH - 1) % DEPTH], lp + (DEPTH - 1) * WAVES);
          issue_fence();
          s.process(r[j], qf, qsum, lp * kPage, L, qk_scale, g);
          lp += WAVES;
          more = lp < p_end;
        }
      }
    }
  }

  // merge the waves; lane (n, g) holds dims 32g + 8i + db (i < 4, db < 8) of query n
  float* red_o = red;
  float* red_ml = red + WAVES * G * (kHeadDim + 1);
  if (n < G) {
    float* dst = red_o + (w * G + n) * (kHeadDim + 1) + 32 * g;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int db = 0; db < 8; db++) dst[8 * i + db] = s.o[db][i];
    if (g == 0) {
      red_ml[(w * G + n) * 2] = s.m;
      red_ml[(w * G + n) * 2 + 1] = s.l;
    }
  }
  __syncthreads();
  const int tq = threadIdx.x >> 4, td = (threadIdx.x & 15) * 8;  // query tq, dims td .. td+7
  if (tq >= G) return;
  float mx = -INFINITY;
#pragma unroll
  for (int ww = 0; ww < WAVES; ww++) mx = fmaxf(mx, red_ml[(ww * G + tq) * 2]);
  float lsum = 0.f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ww = 0; ww < WAVES; ww++) {
    const float mw = red_ml[(ww * G + tq) * 2];
    const float f = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - mx);
    lsum += red_ml[(ww * G + tq) * 2 + 1] * f;
    const float* src = red_o + (ww * G + tq) * (kHeadDim + 1) + td;
#pragma unroll
    for (int e = 0; e < 8; e++) acc[e] += src[e] * f;
  }
  if (ch.slot < 0) {  // the whole sequence: its state is the result
    half8_t h;
#pragma unroll
    for (int e = 0; e < 8; e++) h[e] = (_Float16)(lsum > 0.f ? acc[e] / lsum : 0.f);
    *reinterpret_cast<half8_t*>(out + ((size_t)b * Hq + hk * G + tq) * kHeadDim + td) = h;
    return;
  }
  const size_t slot = ((size_t)ch.slot * Hkv + hk) * G + tq;
  float4_t* po = reinterpret_cast<float4_t*>(part_o + slot * kHeadDim + td);
  po[0] = float4_t{acc[0], acc[1], acc[2], acc[3]};
  po[1] = float4_t{acc[4], acc[5], acc[6], acc[7]};
  if (td == 0) {
    part_ml[slot * 2] = mx;
    part_ml[slot * 2 + 1] = lsum;
  }
}

// out[b][h] = sum_c 2^(m_c - M) O_c / sum_c 2^(m_c - M) l_c.  One workgroup per query head; wave w folds chunks
// w, w+4, ... into a running (M, L, O) (lane: dims 2l, 2l+1), then the 4 waves combine in LDS.  Fixed order.
// A sequence of one chunk has its output already; an empty sequence gets zeros.
template <bool BY_LENGTH>
__global__ __launch_bounds__(kMergeWaves * 64) void kv_merge_kernel(const float* __restrict__ part_o,
                                                       const float* __restrict__ part_ml, int Hq, int Hkv,
                                                       const int* __restrict__ seq_lens, KvSplit split, int waves,
                                                       _Float16* __restrict__ out) {
  __shared__ float sm_ml[kMergeWaves][2];
  __shared__ float sm_o[kMergeWaves][kHeadDim];
  const int h = blockIdx.x, b = blockIdx.y;
  const int G = Hq / Hkv, hk = h / G, q = h - hk * G;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
  int chunks = split.chunks, state0 = b * split.chunks;  // the sequence's chunks, and its first partial state
  if constexpr (BY_LENGTH) {
    KvBatch k;
    if (kv_batch(split, seq_lens, waves, k)) {
      chunks = __builtin_amdgcn_readlane(k.chunks, b);
      state0 = (__builtin_amdgcn_readlane(k.sums, b) >> 16) - chunks;
    }
    if (chunks == 1) return;
  }
  float M = -INFINITY, L = 0.f, a0 = 0.f, a1 = 0.f;
#pragma unroll 4
  for (int c = w; c < chunks; c += kMergeWaves) {
    const size_t slot = ((size_t)(state0 + c) * Hkv + hk) * G + q;
    const float mc = part_ml[slot * 2], lc = part_ml[slot * 2 + 1];
    const float2 oc = *reinterpret_cast<const float2*>(part_o + slot * kHeadDim + 2 * l);
    const float mn = fmaxf(M, mc);
    // equal maxima scale by 1 (also covers -inf == -inf: an empty chunk has l = 0, O = 0)
    const float fa = M == mn ? 1.f : __builtin_amdgcn_exp2f(M - mn);
    const float fc = mc == mn ? 1.f : __builtin_amdgcn_exp2f(mc - mn);
    L = L * fa + lc * fc;
    a0 = a0 * fa + oc.x * fc;
    a1 = a1 * fa + oc.y * fc;
    M = mn;
  }
  if (l == 0) {
    sm_ml[w][0] = M;
    sm_ml[w][1] = L;
  }
  sm_o[w][2 * l] = a0;
  sm_o[w][2 * l + 1] = a1;
  __syncthreads();
  if (threadIdx.x >= kHeadDim) return;
  const int d = threadIdx.x;
  float mx = -INFINITY;
#pragma unroll
  for (int ww = 0; ww < kMergeWaves; ww++) mx = fmaxf(mx, sm_ml[ww][0]);
  float lsum = 0.f, acc = 0.f;
#pragma unroll
  for (int ww = 0; ww < kMergeWaves; ww++) {
    const float f = sm_ml[ww][0] == mx ? 1.f : __builtin_amdgcn_exp2f(sm_ml[ww][0] - mx);
    lsum += sm_ml[ww][1] * f;
    acc += sm_o[ww][d] * f;
  }
  out[((size_t)b * Hq + h) * kHeadDim + d] = (_Float16)(lsum > 0.f ? acc / lsum : 0.f);
}

// Workgroup shape, and the fixed plan's pages per workgroup (it sizes the workspace for the split by lengths too).
// 8 waves per workgroup and chunks that fill the GPU about one workgroup
// per CU (256) deep; groups whose 8-wave LDS merge would pass 64 KB take 4 waves and about 1024 workgroups.  Fewer
// chunks mean fewer partial states to write and merge: at 16 sequences x 8 kv heads, 2 chunks of 8 waves measured 3 %
// faster (8-bit) than 8 chunks of 4 waves, and 4 chunks of 8 waves or 2 of 16 no faster than 2 of 8.  chunk_pages is
// a multiple of the wave count.
struct KvPlan {
  int waves, chunk_pages, chunks;
};
// EXL3_KV_WAVES (4 or 8) and EXL3_KV_TARGET_WGS override the plan for measurements; read once per process, so the
// workspace size and the launch always follow the same plan.
static int kv_target(int waves) {
  static const int env_target = [] {
    const char* e = getenv("EXL3_KV_TARGET_WGS");
    return e ? std::max(1, atoi(e)) : 0;
  }();
  return env_target ? env_target : waves == 8 ? 256 : 1024;
}
static KvPlan kv_plan(int batch, int num_kv_heads, int group, int max_pages) {
  static const int env_waves = [] {
    const char* e = getenv("EXL3_KV_WAVES");
    return e && atoi(e) == 4 ? 4 : kKvWaves;
  }();
  int waves = env_waves;
  if ((size_t)waves * group * (kHeadDim + 1 + 2) * sizeof(float) > 65536) waves = 4;
  const int target = kv_target(waves);
  const long pairs = (long)batch * num_kv_heads;
  const long chunks = std::max(1L, std::min((long)(max_pages + waves - 1) / waves, (target + pairs - 1) / pairs));
  int cp = (int)((max_pages + chunks - 1) / chunks);
  cp = (cp + waves - 1) / waves * waves;
  return KvPlan{waves, cp, (max_pages + cp - 1) / cp};
}

}  // namespace exl3

using namespace exl3;

extern "C" size_t exl3_kv_decode_workspace_bytes(int batch, int num_q_heads, int num_kv_heads, int max_pages) {
  if (batch <= 0 || num_kv_heads <= 0 || num_q_heads < num_kv_heads || max_pages <= 0) return 0;
  const int G = num_q_heads / num_kv_heads;
  const KvPlan plan = kv_plan(batch, num_kv_heads, G, max_pages);
  const size_t slots = (size_t)batch * num_kv_heads * plan.chunks * G;
  return slots * (kHeadDim + 2) * sizeof(float);
}

extern "C" int exl3_kv_decode_attention(const void* q, const void* k_cache, const void* v_cache, const void* k_scale,
                                        const void* v_scale, int num_pages, const void* page_table, int max_pages,
                                        const void* seq_lens, int batch, int num_q_heads, int num_kv_heads,
                                        int head_dim, int page_size, int bits, float sm_scale, void* out,
                                        void* workspace, size_t workspace_bytes, void* stream) {
  EXL3_CHECK_ARG((batch == 0 || (q && page_table && seq_lens && out)) && k_cache && v_cache && k_scale && v_scale,
                 "exl3_kv_decode_attention: null pointer");
  EXL3_CHECK_ARG(head_dim == kHeadDim && page_size == kPage,
                 "exl3_kv_decode_attention: head_dim = %d, page_size = %d (supported: 128, 16)", head_dim, page_size);
  EXL3_CHECK_ARG(bits == 4 || bits == 8, "exl3_kv_decode_attention: bits = %d (4 or 8)", bits);
  EXL3_CHECK_ARG(batch >= 0 && num_pages >= 1 && max_pages >= 1 && num_kv_heads >= 1 &&
                     num_q_heads % num_kv_heads == 0 && num_q_heads / num_kv_heads >= 1 &&
                     num_q_heads / num_kv_heads <= kMaxGroup,
                 "exl3_kv_decode_attention: batch = %d, pages = %d, max_pages = %d, heads %d / %d (group <= 16)",
                 batch, num_pages, max_pages, num_q_heads, num_kv_heads);
  if (batch == 0) return EXL3_OK;
  const size_t need = exl3_kv_decode_workspace_bytes(batch, num_q_heads, num_kv_heads, max_pages);
  EXL3_CHECK_ARG(workspace && workspace_bytes >= need, "exl3_kv_decode_attention: workspace %zu bytes, need %zu",
                 workspace_bytes, need);
  const int G = num_q_heads / num_kv_heads;
  const KvPlan plan = kv_plan(batch, num_kv_heads, G, max_pages);
  const int chunks = plan.chunks;
  float* part_o = static_cast<float*>(workspace);
  float* part_ml = part_o + (size_t)batch * num_kv_heads * chunks * G * kHeadDim;
  const float qk_scale = sm_scale * 1.4426950408889634f;  // logits in base 2
  const size_t lds = (size_t)plan.waves * G * (kHeadDim + 1 + 2) * sizeof(float);
  hipStream_t st = as_stream(stream);
  // The split by lengths, with the merge launch, for up to 64 sequences, unless the fixed plan's chunks are one page per
  // wave, or one chunk per sequence needs no merge and either the table is short (16 pages per wave) or the pairs fill
  // the GPU twice.
  const int target = (kv_target(plan.waves) + num_kv_heads - 1) / num_kv_heads, slots = batch * chunks;
  const bool by_length = batch <= 64 && plan.chunk_pages > plan.waves &&
                         !(chunks == 1 && (max_pages <= 16 * plan.waves || (long)batch * num_kv_heads >= 512));
  // How the fixed plan's longest chunk weighs, fitted at 330 random batches: with a CU for every workgroup of it, chunks by
  // lengths have to be shorter by a seventh (8 sequences, 8 heads, 88 pages for 96: 17.3 us by the fixed plan, 20.2 by
  // lengths); where some CUs work on two they win also when longer (14 sequences, 8 heads, 336 workgroups of up to 248
  // pages, share 276: 66 and 53 us); with more than half as many sequences as aimed at both plans have such CUs.
  const float worth = slots <= target ? 0.87f : 2 * batch <= target ? 1.6f : 1.1f;
  const KvSplit split{batch,           max_pages * kPage,   target, slots,            1.0f / target,
                      1.0f / slots,    1.0f / num_kv_heads, worth,  plan.chunk_pages, chunks};
  // by lengths: at most `slots` chunks of split sequences, and one for every other sequence
  const dim3 grid(chunks, num_kv_heads, by_length ? batch + (batch + chunks - 1) / chunks : batch);
  auto qp = static_cast<const _Float16*>(q);
  auto kp = static_cast<const uint8_t*>(k_cache);
  auto vp = static_cast<const uint8_t*>(v_cache);
  auto ksp = static_cast<const uint16_t*>(k_scale);  // fp16 bits
  auto vsp = static_cast<const uint16_t*>(v_scale);
  auto pt = static_cast<const int*>(page_table);
  auto sl = static_cast<const int*>(seq_lens);
  static const int depth = [] {  // register page sets per wave (prefetch distance + 1); deeper sets measured no faster
    const char* e = getenv("EXL3_KV_DEPTH");
    return e ? std::min(5, std::max(2, atoi(e))) : 2;
  }();
  using Kern = decltype(&kv_decode_kernel<8, 2, 4, false>);
#define EXL3_KV_DEPTHS(B, W, S) \
  {kv_decode_kernel<B, 2, W, S>, kv_decode_kernel<B, 3, W, S>, kv_decode_kernel<B, 4, W, S>, kv_decode_kernel<B, 5, W, S>}
#define EXL3_KV_SPLITS(B, W) {EXL3_KV_DEPTHS(B, W, false), EXL3_KV_DEPTHS(B, W, true)}
  static const Kern table[2][2][2][4] = {{EXL3_KV_SPLITS(4, 4), EXL3_KV_SPLITS(8, 4)},
                                         {EXL3_KV_SPLITS(4, 8), EXL3_KV_SPLITS(8, 8)}};
#undef EXL3_KV_SPLITS
#undef EXL3_KV_DEPTHS
  table[plan.waves == 8][bits == 8][by_length][depth - 2]<<<grid, plan.waves * 64, lds, st>>>(
      qp, kp, vp, ksp, vsp, num_pages, pt, max_pages, sl, num_q_heads, num_kv_heads, qk_scale, split,
      part_o, part_ml, static_cast<_Float16*>(out));
  EXL3_CHECK_LAUNCH();
  if (by_length || chunks > 1) {
    auto merge = by_length ? kv_merge_kernel<true> : kv_merge_kernel<false>;
    merge<<<dim3(num_q_heads, batch), kMergeWaves * 64, 0, st>>>(part_o, part_ml, num_q_heads, num_kv_heads, sl, split, plan.waves,
                                              static_cast<_Float16*>(out));
    EXL3_CHECK_LAUNCH();
  }
  return EXL3_OK;
}
