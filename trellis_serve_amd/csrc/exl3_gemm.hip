// EXL3 prefill: fused decode-GEMM on gfx950 MFMA (v_mfma_f32_16x16x32_f16), y = Had(xh @ W_inner) * svh.
//
// Reference semantics: the reference's prefill is decode-to-HBM + cuBLAS between its rotation launches
// (cuda/src/sglang_exl3/runtime/ops.py:36-59); the fused Marlin path serves < 256 rows
// (exl3_marlin_template.h).  Here the weights are decoded into registers inside the GEMM and never reach HBM.
//
// Operands
//   A: xh in "fragment order", k-step major: the rotated activations with k permuted inside every 32-wide block so
//      that the 8 halves one MFMA lane needs are contiguous, and the blocks of one k-step stored together:
//      xh_f[b][m][8q + 4tr + e] = xh[m][32b + 16tr + r(q, e)], r(q, e) = 2q + (e & 1) + 8(e >> 1) (written by
//      rotate_rows_kernel).  One k-step of 256 rows is one contiguous 16 KB run: the GEMM's loads use whole lines.
//   B: the trellis.  A k-step covers 32 rows = 2 tile rows.  The lane-geometry decode of exl3_device.hpp gives lane
//      (c, j) of a tile the 4 weights of column c at rows r(j, 0..3); tile row tr of the k-step supplies halves
//      4tr..4tr+3 of the lane's 8-half B fragment.  A and B then agree on the k order of every MFMA.
//
// Tiling: workgroup 16 MI rows (64 to 256) x 256 columns (two output rotation blocks; a shard of an odd number of
// 128-column blocks ends in a half tile), 8 waves.  Wave w owns 32 columns of every row: it decodes their weights into
// registers, each once, and multiplies them (the MFMA's A operand) with the A fragments of all rows from LDS.  No
// decoded weight goes through LDS and only the A pieces are shared between waves.  One workgroup per CU (two at 64
// rows).  Against wave tiles of 128 x 64 with the decoded weights in LDS (two waves per weight, a barrier that the
// step's first LDS reads wait behind): 5120 -> 16384 at 4096 rows, one k-step 1.05 -> 0.96 us, a tile's epilogue 22 ->
// 6 us; 729-745 -> 641-676 us in all (636 with the k-steps in pairs).
//
// What bounds it: issue.  Per k-step and wave of a 256-row tile 32 MFMAs (512 cycles) and 71 VALU of decode (284),
// two waves per SIMD.  Counters at 2048 rows of 5120 -> 17408: matrix core 50 % busy, VALU 42 % (MFMA issue included),
// 31 % of the matrix core's cycles beside a VALU instruction, at 1.9 GHz.  The two waves of a SIMD take decode and
// multiply in opposite order (2-3 %); forced bursts, a deeper fragment window (8) and an explicit MFMA / VALU interleave
// were slower.
//
// Work decomposition (1-D grid of work items, dispatched in order): tiles are numbered column block fastest, so
// consecutive workgroups share their A rows in L2.  When the tile count is not a multiple of the machine's
// workgroup slots, the last partial round and one full round before it (stream-K tiles) are shared out as equal runs
// of k-steps over one workgroup per slot: a run crosses tile boundaries, so every workgroup finishes after the same
// number of k-steps.  The stream-K workgroups are dispatched first, then one workgroup per remaining whole tile.  A
// run's first and last segments can cover part of a tile: such a segment stores its fp32 accumulators as a partial,
// and the last of the tile's workgroups to arrive (a per-tile counter in the workspace's counter region) sums the
// tile's partials in workgroup order (deterministic, independent of arrival order), then runs the same epilogue as a
// whole tile and resets the counter.  When whole rounds would finish sooner, every tile is a whole-tile item.
//
// Pipeline: direct-to-LDS 16-byte buffer loads (no VGPR staging) into two 4-slot rings, one for A (a piece is a row
// block of 64 lanes x 16 B: a lane's 16 bytes land exactly where its MFMA fragment lives) and one, private to each
// wave, for the trellis bits.  The compiler does not order LDS-DMA writes before LDS reads, so the waits are explicit
// (vmcnt); one barrier per k-step publishes the A pieces of the NEXT step, so that a wave's fragment reads run ahead
// across the barrier.
#include <stdlib.h>

#include <algorithm>

#include "exl3_api.hpp"
#include "exl3_device.hpp"
#include "exl3_tile.hpp"

namespace exl3 {


constexpr int kCoherentStore = 1 << 4;             // buffer cache policy sc1: device-scope coherent access
constexpr int kPastEnd = 0x7FFFFFF0;               // a buffer offset past every partial
constexpr size_t gemm_partial_bytes(int MI) { return (size_t)MI * 16 * kBN * 4; }  // one fp32 partial tile

struct GemmShards {
  const uint32_t* trellis[EXL3_MAX_SHARDS];
  const uint16_t* svh[EXL3_MAX_SHARDS];
  const uint16_t* xh[EXL3_MAX_SHARDS];  // per-shard rotated activations, fragment order, k-step major
  int tn[EXL3_MAX_SHARDS];              // tile columns of the shard
  int layout[EXL3_MAX_SHARDS];          // EXL3_LAYOUT_STORED / EXL3_LAYOUT_BLOCKS
  int col0[EXL3_MAX_SHARDS];            // first output column of the shard
  int ct0[EXL3_MAX_SHARDS + 1];         // first 256-column tile of the shard (cumulative); ct0[count] = total
  int count;
};

// The work decomposition of one launch (see the header comment).
struct GemmPlan {
  int nct;         // 256-column tiles per row block
  int sk_tiles;    // tiles 0 .. sk_tiles-1 are shared out by runs of k-steps among the stream-K workgroups
  int groups;      // stream-K workgroups: grid items 0 .. groups-1; items groups.. are whole tiles sk_tiles..
  int ksteps;      // k / 32
  float* partial;  // [groups][2 segments][8 waves][MI][2][64 lanes] float4: a workgroup's first / last segment
  int* counters;   // [sk_tiles], zero between calls
};

// Stream-K: workgroup g owns the global k-steps [sk_start(g), sk_start(g + 1)) of the sk_tiles * ksteps steps (tile t
// holds steps t * ksteps ..); sk_owner(q) is the workgroup whose run holds step q.
__host__ __device__ __forceinline__ int64_t sk_start(const GemmPlan& p, int g) {
  return (int64_t)p.sk_tiles * p.ksteps * g / p.groups;
}
__host__ __device__ __forceinline__ int sk_owner(const GemmPlan& p, int64_t q) {
  const int64_t W = (int64_t)p.sk_tiles * p.ksteps;
  return (int)(((q + 1) * p.groups + W - 1) / W) - 1;
}

// lds_barrier() (exl3_device.hpp) between k-steps: the direct-to-LDS writes are waited for explicitly (waitcnt_vm)
// before each barrier.

// per-shard input scales of one prefill call (the rotation runs every shard in one launch)
struct ShardSuh {
  const uint16_t* suh[EXL3_MAX_SHARDS];
};

// Shard s of a rotation unit and its suh (a select over the few shards keeps the pointer in scalar registers)
__device__ __forceinline__ const uint16_t* unit_suh(const ShardSuh& su_all, int s) {
  return s == 0 ? su_all.suh[0] : s == 1 ? su_all.suh[1] : s == 2 ? su_all.suh[2] : su_all.suh[3];
}

// The activations of every shard in fragment order, k-step major (see the header comment): xh_f[s][kt][row][32].  One
// wave per (16 rows, 128-block): it loads the block once as MFMA fragments and, per shard, multiplies by suh (fp16
// product), rotates by MFMA and stores whole fragments, 1 KB per k-step.  The butterfly on 16 lanes per row that this
// replaces took 130 VALU instructions and 8-byte stores per row and block: 4096 rows, 2 shards of k = 5120 49 us against
// 28 (126 MB; at a large copy's rate 25).  ROT = false: the fp16 rows as given, only put in fragment order (the
// rotation-free GEMM of exl3_gemm_rotated).  gridDim.z: shards over workgroups (few rows), else all in one wave.
template <bool X_BF16, bool ROT>
__global__ __launch_bounds__(256) void rotate_rows_kernel(const uint16_t* __restrict__ x, int rows, int k,
                                                          ShardSuh su_all, int shards, uint16_t* __restrict__ xh) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, c = l & 15, j = l >> 4;
  const int row0 = (blockIdx.x * 4 + w) * 16, b = blockIdx.y;
  if (row0 >= rows) return;  // wave-uniform
  const int row = row0 + c, from = row < rows ? row : rows - 1;
  uint16_t* dst = xh + ((size_t)(b * 4) * rows + row) * 32 + 8 * j;
  if constexpr (!ROT) {
    // slot 8 j + 4 tr + e of a 32-block holds position 16 tr + 2 j + (e & 1) + 8 (e >> 1)
    const uint16_t* xr = x + (size_t)from * k + b * 128 + 2 * j;
    u32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int q = 0; q < 4; q++) v[u][q] = *reinterpret_cast<const uint32_t*>(xr + 32 * u + 8 * q);
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (row < rows) *reinterpret_cast<u32x4*>(dst + (size_t)u * rows * 32) = v[u];
  } else {
    half8_t xv[4];
    load_row_frags<X_BF16>(x + (size_t)from * k + b * 128 + 8 * j, xv);
    const HadFrags had = had_frags_act(l);
    const int s0 = gridDim.z > 1 ? blockIdx.z : 0, s1 = gridDim.z > 1 ? s0 + 1 : shards;
    for (int s = s0; s < s1; s++) {
      const uint16_t* suh = unit_suh(su_all, s) + b * 128 + 8 * j;
      half8_t in[4];
#pragma unroll
      for (int kb = 0; kb < 4; kb++) in[kb] = times8(xv[kb], suh + 32 * kb);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const half8_t o = had_pair(had, in, u);
        if (row < rows) *reinterpret_cast<half8_t*>(dst + (size_t)s * rows * k + (size_t)u * rows * 32) = o;
      }
    }
  }
}

// One segment of work: k-steps [kt0, kt1) of tile `tile`.  seg < 0: the whole tile, straight to the epilogue;
// seg = 0 / 1: a stream-K segment at the start / end of workgroup `item`'s run, stored as that partial slot; the
// last of the tile's workgroups to arrive sums every partial of the tile in workgroup order and runs the epilogue.
template <int K, int CB, int MI>
__device__ __forceinline__ void gemm_segment(const GemmShards& sa, const GemmPlan& plan, int M, int k,
                                             void* __restrict__ y, int y_bf16, int n_total, int rotate_out,
                                             uint8_t* lds, int item, int tile, int kt0, int kt1, int seg) {
  constexpr int kRows = 16 * MI;
  constexpr int PIECES = (MI + kGemmWaves - 1) / kGemmWaves;  // A pieces (16 rows) a wave loads per k-step
  uint8_t* a_ring = lds;                            // [kARing][MI row blocks][64 lanes][8 halves]
  uint8_t* bits_ring = lds + kARing * MI * 1024;    // [kBitsRing][8 waves][64 lanes][16 B]

  const int ct = tile % plan.nct, mblk = tile / plan.nct;
  int s = 0;
#pragma unroll
  for (int i = 1; i < EXL3_MAX_SHARDS; i++)
    if (i < sa.count && ct >= sa.ct0[i]) s = i;
  const int tn = sa.tn[s];
  const int tc0 = (ct - sa.ct0[s]) * 16;  // first tile column of this tile in the shard
  const int ntc = min(16, tn - tc0);      // tile columns present: 16, or 8 at the end of a shard of odd 128-blocks
  const int col0 = sa.col0[s] + tc0 * 16;  // first output column
  const int row0 = mblk * kRows;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63;
  const int c = l & 15, j = l >> 4;
  const bool mfma_wave = 2 * w < ntc;  // wave-uniform: its 32 columns exist

  // B: wave w loads and decodes its own two tile columns 2w, 2w + 1 (both tile rows of the k-step); past the end of a
  // half tile it re-reads the tile's first columns (in range, never stored)
  const int tile_bytes = 32 * K;
  const int row_bytes = tn * tile_bytes;
  const __amdgpu_buffer_rsrc_t brsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)sa.trellis[s], (short)0, (k >> 4) * row_bytes, 0x00020000);
  // STORED: the two columns are adjacent in their tile row; BLOCKS: the tiles of a column are adjacent, the columns 8
  // tiles apart inside the unit of the column block
  const bool blocks = sa.layout[s] == EXL3_LAYOUT_BLOCKS;
  const BitsLane bl = bits_lane<K>(l);
  const int bj = tc0 + (mfma_wave ? 2 * w : 0) + bl.col;
  const int bgoff = (blocks ? ((bj >> 3) * (k >> 7) * 64 + (bj & 7) * 8 + bl.row) * tile_bytes
                            : bl.row * row_bytes + bj * tile_bytes) + bl.piece * 16;

  // A: lane l of a piece = row (l % 16) of the row block, k-chunk l / 16.  Rows past M re-read row M-1 (finite, only
  // feeds discarded C rows).
  ActLoads<PIECES> act;
  act.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)sa.xh[s], (short)0, M * k * 2, 0x00020000);
  act.step = M * kBK * 2;
  act.stage = MI * 1024;
#pragma unroll
  for (int q = 0; q < PIECES; q++) {
    const int p = PIECES * w + q, piece = p < MI ? p : p % MI;  // fewer pieces than waves: some are loaded twice
    const int row = row0 + piece * 16 + c;
    act.src[q] = ((row < M ? row : M - 1) * 32 + j * 8) * 2;
    act.dst[q] = piece * 1024;
  }

  const int nk = kt1 - kt0;  // >= 1
  float4_t acc[MI][2];
#pragma unroll
  for (int mi = 0; mi < MI; mi++)
#pragma unroll
    for (int jj = 0; jj < 2; jj++) acc[mi][jj] = float4_t{0.f, 0.f, 0.f, 0.f};

  tile_multiply<K, CB, MI, PIECES>(
      a_ring, act, 0, bits_ring + w * 1024, brsrc, bgoff,
      [&](int kt) { return blocks ? ((kt >> 2) * 64 + (kt & 3) * 2) * tile_bytes : 2 * kt * row_bytes; }, kt0, nk,
      (w & 4) != 0, l, acc);

  // ---- stream-K segment: store the partial (16-byte stores with device-scope coherence: the reader may sit on
  // another XCD, whose L2 is not this one's); the tile's last workgroup to arrive sums all of the tile's partials in
  // workgroup order (deterministic, independent of arrival order)
  if (seg >= 0) {
    __shared__ int last_flag;
    constexpr int kWaveBytes = MI * 2 * 64 * 16;  // a wave's share of a partial tile
    const __amdgpu_buffer_rsrc_t prsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)plan.partial, (short)0, plan.groups * 2 * kGemmWaves * kWaveBytes, 0x00020000);
    auto slot_off = [&](int g, int sl) { return ((g * 2 + sl) * kGemmWaves + w) * kWaveBytes + l * 16; };
    // only the 16-row blocks that hold output rows (rows >= M and columns past a half tile are never stored): the
    // others' offsets lie past the buffer, where stores are dropped and loads give zeros without a request, so that
    // no access is conditional and all are in flight together
    const int live_rows = mfma_wave ? M - row0 : 0;  // wave-uniform
    auto off = [&](int base, int mi, int jj) { return mi * 16 < live_rows ? base + (mi * 2 + jj) * 64 * 16 : kPastEnd; };
    const int mine = slot_off(item, seg);
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
      for (int jj = 0; jj < 2; jj++)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[mi][jj]), prsrc, off(mine, mi, jj), 0,
                                               kCoherentStore);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));  // this thread's partial stores are at the coherence point
    __syncthreads();
    const int64_t q0 = (int64_t)tile * plan.ksteps;
    const int g_first = sk_owner(plan, q0), g_last = sk_owner(plan, q0 + plan.ksteps - 1);
    if (tid == 0) {
      const int prev = __hip_atomic_fetch_add(&plan.counters[tile], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last_flag = prev == g_last - g_first;
    }
    __syncthreads();
    if (!last_flag) return;
    // the sum runs in workgroup order from g_first; when this workgroup is g_first (the usual last arrival: the
    // tile is the end of its run) its registers are that first term, bit for bit what it stored
    int g = g_first;
    if (item == g_first) {
      g++;
    } else {
#pragma unroll
      for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int jj = 0; jj < 2; jj++) acc[mi][jj] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
    for (; g <= g_last; g++) {
      const int src = slot_off(g, sk_start(plan, g) >= q0 ? 0 : 1);  // the tile is g's first segment or its last
      constexpr int kBatch = MI < 8 ? MI : 8;
#pragma unroll
      for (int m0 = 0; m0 < MI; m0 += kBatch) {
        u32x4 v[kBatch][2];
#pragma unroll
        for (int q = 0; q < kBatch; q++)
          if (m0 + q < MI)
#pragma unroll
            for (int jj = 0; jj < 2; jj++)
              v[q][jj] = __builtin_amdgcn_raw_buffer_load_b128(prsrc, off(src, m0 + q, jj), 0, kCoherentStore);
#pragma unroll
        for (int q = 0; q < kBatch; q++)
          if (m0 + q < MI)
#pragma unroll
            for (int jj = 0; jj < 2; jj++) acc[m0 + q][jj] += __builtin_bit_cast(float4_t, v[q][jj]);
      }
    }
    if (tid == 0) __hip_atomic_store(&plan.counters[tile], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // ---- epilogue: the fp16 C tile (rounded once from fp32) goes to LDS, 4 columns of a row per 8-byte write; then each
  // wave rotates its share of the (16-row, 128-column) blocks by MFMA and stores them (rotate_out), or stores the rows
  // as they are.
  _Float16* cl = reinterpret_cast<_Float16*>(lds);
  if (mfma_wave) tile_to_lds<MI>(cl, acc, w, l);
  __syncthreads();
  const HadFrags had = had_frags_rows(l);
  for (int p = w; p < MI * 2; p += kGemmWaves) {
    const int mi = p >> 1, h = p & 1;
    const int m = row0 + mi * 16 + c;
    if (8 * h >= ntc || row0 + mi * 16 >= M) continue;  // wave-uniform
    const half8_t* src = reinterpret_cast<const half8_t*>(cl + (mi * 16 + c) * kCStride + h * 128 + 8 * j);
    half8_t cf[4];
#pragma unroll
    for (int kb = 0; kb < 4; kb++) cf[kb] = src[kb * 4];
    const int col = col0 + h * 128 + 8 * j;
    uint16_t* yr = static_cast<uint16_t*>(y) + (size_t)(m < M ? m : M - 1) * n_total + col;
    const half8_t* sv8 = reinterpret_cast<const half8_t*>(sa.svh[s] + (col - sa.col0[s]));
#pragma unroll
    for (int u = 0; u < 4; u++) {
      half8_t o = cf[u];
      if (rotate_out) {
        o = had_pair(had, cf, u);
        const half8_t sv = sv8[u * 4];
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = o[e] * sv[e];
      }
      if (m < M) {
        if (y_bf16) {
          u32x4 ob;
#pragma unroll
          for (int e = 0; e < 4; e++)
            ob[e] = (uint32_t)f32_to_bf16((float)o[2 * e]) | ((uint32_t)f32_to_bf16((float)o[2 * e + 1]) << 16);
          *reinterpret_cast<u32x4*>(yr + 32 * u) = ob;
        } else {
          *reinterpret_cast<half8_t*>(yr + 32 * u) = o;
        }
      }
    }
  }
  __syncthreads();  // the C tile in LDS is read before the next segment's loads overwrite it
}

// Grid: the stream-K workgroups first (each walks the segments of its run of k-steps), then one workgroup per
// remaining whole tile.
template <int K, int CB, int MI>
__global__ __launch_bounds__(kGemmThreads, MI <= 4 ? 4 : 2) void gemm_kernel(GemmShards sa, GemmPlan plan, int M, int k,
                                                             void* __restrict__ y, int y_bf16, int n_total,
                                                             int rotate_out) {
  extern __shared__ __align__(16) uint8_t lds[];
  const int item = blockIdx.x;
  int64_t q, b;  // global k-steps left
  if (item >= plan.groups) {
    q = (int64_t)(plan.sk_tiles + (item - plan.groups)) * plan.ksteps;
    b = q + plan.ksteps;
  } else {
    q = sk_start(plan, item);
    b = sk_start(plan, item + 1);
  }
  const int64_t a = q;
  while (q < b) {
    const int t = (int)(q / plan.ksteps);
    const int64_t q0 = (int64_t)t * plan.ksteps;
    const int kt0 = (int)(q - q0), kt1 = (int)(b - q0 < plan.ksteps ? b - q0 : plan.ksteps);
    const bool whole = kt0 == 0 && kt1 == plan.ksteps;
    gemm_segment<K, CB, MI>(sa, plan, M, k, y, y_bf16, n_total, rotate_out, lds, item, t, kt0, kt1,
                            whole ? -1 : (q == a ? 0 : 1));
    q = q0 + kt1;
  }
}

#define EXL3_GEMM_DISPATCH(K_, CB_, ...)                                  \
  [&]() -> bool {                                                         \
    switch (K_ * 4 + CB_) {                                               \
      EXL3_GCASE(2, __VA_ARGS__) EXL3_GCASE(3, __VA_ARGS__)               \
      EXL3_GCASE(4, __VA_ARGS__) EXL3_GCASE(5, __VA_ARGS__)               \
      EXL3_GCASE(6, __VA_ARGS__) EXL3_GCASE(8, __VA_ARGS__)               \
      default: return false;                                              \
    }                                                                     \
  }()
#define EXL3_GCASE(KV, ...)                                                            \
  case KV * 4 + 0: { constexpr int kK = KV, kCB = 0; __VA_ARGS__; return true; }      \
  case KV * 4 + 1: { constexpr int kK = KV, kCB = 1; __VA_ARGS__; return true; }      \
  case KV * 4 + 2: { constexpr int kK = KV, kCB = 2; __VA_ARGS__; return true; }



// Workgroups that run at once, counted as one per CU (a 256-row tile takes 135 KB of LDS), per device, queried once.
static int gemm_slots() {
  static int slots[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (slots[dev] == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    slots[dev] = cus;
  }
  return slots[dev];
}

struct GemmLayout {
  int mi, nct, sk_tiles, groups, ksteps, tiles;
  size_t xh_bytes, partial_off, total;
};

// 256-column tiles never straddle shards (each shard reads its own rotated activations): a shard of an odd number
// of 128-column blocks ends in a half tile
static int gemm_col_tiles(const int* shard_n, int nshards) {  // tiles of 256 columns over all shards
  int t = 0;
  for (int s = 0; s < nshards; s++) t += (shard_n[s] / 128 + 1) / 2;
  return t;
}

// The decomposition of `tiles` tiles of `ksteps` k-steps over the machine's slots: whole tiles in rounds, except the
// last (partial) round plus one full round before it (when there is one), which are shared out by runs of k-steps over
// one workgroup per slot (stream-K): every workgroup then finishes after the same number of k-steps, 1 to 2 tiles'
// worth, and writes at most two partial tiles.  A run keeps >= 8 k-steps so the pipeline start-up stays small against
// its work.  Whole rounds only, when they are sooner.  us: the estimated time, from the step time of the tile height
// and what the partials cost it (store, the last arrival's reload of every partial at one CU's bandwidth), fitted at
// 33-1500 rows of the four 27B layers (K = 3; within ~10 %).
struct GemmShape {
  int mi;          // 16-row blocks per tile
  double step_us;  // one k-step of one workgroup per CU
  double sk_us;    // stream-K: partials, and the tile's epilogue
};
constexpr GemmShape kGemmShapes[] = {{4, 0.42, 20}, {8, 0.62, 24}, {12, 0.78, 32}, {16, 0.95, 42}};
constexpr double kEpilogueUs = 8;

static double gemm_share(const GemmShape& shape, int slots, int tiles, int ksteps, int* sk_tiles, int* groups) {
  const int rounds = tiles / slots, rem = tiles - rounds * slots;
  const double tile_us = ksteps * shape.step_us + kEpilogueUs;
  const double whole = (rounds + (rem > 0)) * tile_us;
  *sk_tiles = *groups = 0;
  if (rem == 0) return whole;
  const int sk = rounds >= 1 ? rem + slots : rem;
  const int g = (int)std::max<int64_t>(1, std::min<int64_t>(slots, (int64_t)sk * ksteps / 8));
  const double shared = (tiles - sk) / slots * tile_us + (double)sk * ksteps / g * shape.step_us + shape.sk_us;
  if (shared >= whole) return whole;
  *sk_tiles = sk;
  *groups = g;
  return shared;
}

// The tile height with the least estimated time: few rows (or a remainder of few rows) waste less of a low tile and
// write smaller partials, many rows share each decoded weight in a high one.  Measured against 256-row tiles alone (us,
// K = 3): 80 rows gate/up 99 -> 74, down 82 -> 58; 256 rows q/k/v 88 -> 61, o 76 -> 48; 700 rows q/k/v 117 -> 95.
static GemmLayout gemm_layout(int slots, int rows, int k, int nct, int nshards) {
  GemmLayout L{};
  L.nct = nct;
  L.ksteps = k / kBK;
  double best = 0;
  for (const GemmShape& shape : kGemmShapes) {
    const int tiles = (rows + 16 * shape.mi - 1) / (16 * shape.mi) * nct;
    int sk, groups;
    const double us = gemm_share(shape, slots, tiles, L.ksteps, &sk, &groups);
    if (L.mi == 0 || us < best) {
      best = us;
      L.mi = shape.mi;
      L.tiles = tiles;
      L.sk_tiles = sk;
      L.groups = groups;
    }
  }
  // [counter region (fixed place and size)][rotated activations][partials: 2 per stream-K workgroup]
  L.xh_bytes = ((size_t)nshards * rows * k * 2 + 255) & ~(size_t)255;
  L.partial_off = kCounterBytes + L.xh_bytes;
  L.total = L.partial_off + (size_t)L.groups * 2 * gemm_partial_bytes(L.mi);
  return L;
}

// One workspace for every call of up to `rows` rows: a layout's own need goes down where whole rounds or lower tiles need
// fewer partials.  Tiles are multiples of 64 rows, so up to 1024 rows every layout is looked at (2 us); past that the
// bound is each height's most stream-K workgroups (gemm_share), which grows with the rows: at most 134 MB of partials.
static size_t gemm_most_bytes(int slots, int rows, int k, int nct, int nshards) {
  constexpr int kLooked = 1024;
  size_t most = 0;
  for (int r = std::min(rows, 64);; r = std::min(rows, r + 64)) {
    most = std::max(most, gemm_layout(slots, r, k, nct, nshards).total);
    if (r == rows || r >= kLooked) break;
  }
  if (rows > kLooked) {
    size_t partials = 0;
    for (const GemmShape& shape : kGemmShapes) {
      const int64_t tiles = (rows + 16 * (int64_t)shape.mi - 1) / (16 * shape.mi) * nct;
      const int64_t groups = std::min<int64_t>(slots, std::min<int64_t>(tiles, 2 * slots) * (k / kBK) / 8);
      partials = std::max(partials, (size_t)std::max<int64_t>(1, groups) * 2 * gemm_partial_bytes(shape.mi));
    }
    most = std::max(most, gemm_layout(slots, rows, k, nct, nshards).partial_off + partials);
  }
  return most;
}

}  // namespace exl3

using namespace exl3;

extern "C" size_t exl3_prefill_workspace_bytes(int rows, int k, int n_total, int nshards) {
  if (rows <= 0 || k <= 0 || k % 128 || n_total <= 0 || n_total % 128 || nshards < 1 || nshards > EXL3_MAX_SHARDS)
    return 0;
  // the column-tile count depends on how n_total splits into shards (a shard of an odd number of 128-column blocks
  // ends in a half tile): take the largest need over every possible count
  const int slots = gemm_slots();
  size_t need = 0;
  for (int nct = (n_total / 128 + 1) / 2; nct <= (n_total / 128 + nshards) / 2; nct++)
    need = std::max(need, gemm_most_bytes(slots, rows, k, nct, nshards));
  return need;
}

namespace exl3 {

// The input pass (rotation of every shard in fragment order, or with ROT = false the rows as given in fragment order)
// and the decode-GEMM launch of one call; sa holds the shards, its xh pointers into the workspace.
template <bool ROT>
static int launch_prefill(const void* x, bool x_bf16, int rows, int k, GemmShards& sa, const ShardSuh& su,
                          const int* shard_n, int K, int codebook, void* y, bool y_bf16, void* workspace,
                          size_t workspace_bytes, hipStream_t st, const char* what) {
  const int nshards = sa.count;
  const GemmLayout L = gemm_layout(gemm_slots(), rows, k, gemm_col_tiles(shard_n, nshards), nshards);
  EXL3_CHECK_ARG(workspace && workspace_bytes >= L.total, "%s: workspace %zu bytes, need %zu", what,
                 workspace_bytes, L.total);
  EXL3_CHECK_ARG(L.sk_tiles <= kMaxCounters, "%s: %d stream-K tiles exceed the counter region", what, L.sk_tiles);
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  uint16_t* xh = reinterpret_cast<uint16_t*>(ws + kCounterBytes);
  for (int s = 0; s < nshards; s++) sa.xh[s] = xh + (size_t)s * rows * k;
  GemmPlan plan{L.nct, L.sk_tiles, L.groups, L.ksteps, reinterpret_cast<float*>(ws + L.partial_off),
                reinterpret_cast<int*>(ws)};
  int n_total = 0;
  for (int s = 0; s < nshards; s++) n_total += shard_n[s];
  // the input pass: every shard in one launch
  const dim3 hgrid((unsigned)((rows + 63) / 64), (unsigned)(k / 128), ROT && rows < 1024 ? (unsigned)nshards : 1u);
  const uint16_t* xr = static_cast<const uint16_t*>(x);
  if (x_bf16)
    rotate_rows_kernel<true, ROT><<<hgrid, 256, 0, st>>>(xr, rows, k, su, nshards, xh);
  else
    rotate_rows_kernel<false, ROT><<<hgrid, 256, 0, st>>>(xr, rows, k, su, nshards, xh);
  EXL3_CHECK_LAUNCH();
  const dim3 grid((unsigned)(L.groups + L.tiles - L.sk_tiles));
  bool ok;
#define EXL3_GEMM_LAUNCH(MI_)                                                                                   \
  ok = EXL3_GEMM_DISPATCH(K, codebook, gemm_kernel<kK, kCB, MI_><<<grid, kGemmThreads, tile_lds(MI_, MI_), st>>>( \
                                          sa, plan, rows, k, y, y_bf16 ? 1 : 0, n_total, ROT ? 1 : 0))
  if (L.mi == 4)
    EXL3_GEMM_LAUNCH(4);
  else if (L.mi == 12)
    EXL3_GEMM_LAUNCH(12);
  else if (L.mi == 8)
    EXL3_GEMM_LAUNCH(8);
  else
    EXL3_GEMM_LAUNCH(16);
#undef EXL3_GEMM_LAUNCH
  if (!ok) return set_error(EXL3_ERR_INVALID, "%s: unsupported K/codebook", what);
  EXL3_CHECK_LAUNCH();
  return EXL3_OK;
}

}  // namespace exl3

using namespace exl3;

extern "C" int exl3_linear_prefill(const void* x, int x_bf16, int rows, int k, const exl3_shard* shards_host,
                                   int nshards, int K, int codebook, void* y, int y_bf16, void* workspace,
                                   size_t workspace_bytes, void* stream) {
  EXL3_CHECK_ARG((rows == 0 || (x && y)) && shards_host, "exl3_linear_prefill: null pointer");
  EXL3_CHECK_ARG(valid_bits(K) && valid_cb(codebook), "exl3_linear_prefill: K = %d / codebook = %d", K, codebook);
  EXL3_CHECK_ARG(rows >= 0 && k > 0 && k % 128 == 0, "exl3_linear_prefill: rows = %d, k = %d", rows, k);
  EXL3_CHECK_ARG(nshards >= 1 && nshards <= EXL3_MAX_SHARDS, "exl3_linear_prefill: nshards = %d", nshards);
  if (rows == 0) return EXL3_OK;
  EXL3_CHECK_ARG((int64_t)rows * k * 2 <= INT32_MAX, "exl3_linear_prefill: rows * k too large for one launch");
  GemmShards sa{};
  ShardSuh su{};
  int col = 0, ctl = 0;
  int shard_n[EXL3_MAX_SHARDS];
  for (int s = 0; s < nshards; s++) {
    const exl3_shard& sh = shards_host[s];
    EXL3_CHECK_ARG(sh.trellis && sh.suh && sh.svh, "shard %d: null tensor pointer", s);
    EXL3_CHECK_ARG(sh.n > 0 && sh.n % 128 == 0, "shard %d: n = %d is not a positive multiple of 128", s, sh.n);
    EXL3_CHECK_ARG((int64_t)k * sh.n * K / 8 <= INT32_MAX, "shard %d: trellis exceeds the 2 GiB buffer range", s);
    sa.trellis[s] = static_cast<const uint32_t*>(sh.trellis);
    sa.svh[s] = static_cast<const uint16_t*>(sh.svh);
    su.suh[s] = static_cast<const uint16_t*>(sh.suh);
    sa.tn[s] = sh.n / 16;
    EXL3_CHECK_ARG(sh.layout == EXL3_LAYOUT_STORED || sh.layout == EXL3_LAYOUT_BLOCKS, "shard %d: layout %d", s,
                   sh.layout);
    sa.layout[s] = sh.layout;
    sa.col0[s] = col;
    sa.ct0[s] = ctl;
    shard_n[s] = sh.n;
    col += sh.n;
    ctl += (sh.n / 128 + 1) / 2;
  }
  sa.ct0[nshards] = ctl;
  sa.count = nshards;
  return launch_prefill<true>(x, x_bf16 != 0, rows, k, sa, su, shard_n, K, codebook, y, y_bf16 != 0, workspace,
                              workspace_bytes, as_stream(stream), "exl3_linear_prefill");
}

namespace exl3 {

size_t linear_gemm_workspace_bytes(int rows, int k, int n_total) {
  return exl3_prefill_workspace_bytes(rows, k, n_total, EXL3_MAX_SHARDS);
}

size_t prefill_plain_workspace_bytes(int rows, int k, int n) {
  const int nct = (n / 128 + 1) / 2;
  return gemm_most_bytes(gemm_slots(), rows, k, nct, 1);
}

// exl3_gemm_rotated from kPrefillRows rows: the rows as given (fp16, already in the rotated basis), no output
// rotation, so one-hot rows read W_inner back through the decode-GEMM bit for bit
int prefill_plain_gemm(const void* xh, int rows, int k, const void* trellis, int n, int K, int codebook, void* out,
                       void* workspace, size_t workspace_bytes, hipStream_t st) {
  EXL3_CHECK_ARG((int64_t)rows * k * 2 <= INT32_MAX, "exl3_gemm_rotated: rows * k too large for one launch");
  GemmShards sa{};
  sa.trellis[0] = static_cast<const uint32_t*>(trellis);
  sa.tn[0] = n / 16;
  sa.ct0[1] = (n / 128 + 1) / 2;
  sa.count = 1;
  const ShardSuh su{};
  const int shard_n[1] = {n};
  return launch_prefill<false>(xh, false, rows, k, sa, su, shard_n, K, codebook, out, false, workspace,
                               workspace_bytes, st, "exl3_gemm_rotated");
}

}  // namespace exl3
