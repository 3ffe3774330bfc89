// EXL3 MoE layer for many tokens on gfx950: the slots sorted by expert, and one decode-GEMM tile per (up to 64 or 128
// slots of an expert, 256 columns) on the core of the dense prefill (exl3_tile.hpp).
//
// Launches: moe_sort_kernel (routing) -> moe_gemm_in_kernel (rotated gate and up inputs) -> moe_gate_up_kernel -> moe_
// down_kernel -> the combine of exl3_moe.hip.  The same arithmetic and rounding points as the expert GEMVs there:
//   g, u = fp16 outputs (fp16 of the fp32 sum, rotation, * svh), a = fp16(silu(g) * u) in fp32, * suh_down, rotation
//   (the down inputs), d = fp16 outputs of down (cuda/csrc/exl3_marlin_moe.cu:210-292).
//
// What bounds it: as the dense decode-GEMM, issue (the decode of an expert's weights once per tile, and its MFMAs).  The
// expert GEMVs decode the weights once per 64 slots too, but each wave reads every activation fragment from LDS for 16
// columns, and a workgroup waits for each 256 rows of k of its activations (one workgroup per CU at 64 slots per pass):
// 128 experts, top-8, 2048 / 768 at 2048 tokens, gate|up and down 875 + 456 us (kernel trace)
// against 245 + 137 here.  Counters: at 256 tokens (about 16 slots per expert) gate/up VALU 63 %, matrix core 15 %; at
// 2048 45 % and 25 % with 6 waves per CU.
#include <algorithm>

#include "exl3_moe_gemm.hpp"
#include "exl3_tile.hpp"

namespace exl3 {

constexpr int kSortThreads = 1024;

// The weights' row of global expert e in the launch's class, or -1
__device__ __forceinline__ int moe_row(const MoeGemmArgs& a, int e) {
  if (a.emap == nullptr) return e;
  const int el = a.emap[e];
  return el < a.E_local ? el : -1;
}

// Routing by one workgroup: the slots of each expert (ids outside [0, E) dropped) as a run of `sorted`, runs in
// ascending expert order, and each run cut into equal tiles of at most tile_rows slots (a multiple of 16).  A slot's
// place inside its run follows the LDS atomics; no result depends on it (every slot is its own row of the GEMMs).
__global__ __launch_bounds__(kSortThreads) void moe_sort_kernel(MoeGemmArgs a) {
  __shared__ int cnt[1024], pos[1024], tile[1024];
  const int t = threadIdx.x;
  cnt[t] = 0;
  __syncthreads();
  constexpr int kBatch = 8;  // ids loaded together
  for (int s0 = t; s0 < a.slots; s0 += kSortThreads * kBatch) {
    int ev[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; i++) ev[i] = s0 + kSortThreads * i < a.slots ? a.topk_ids[s0 + kSortThreads * i] : -1;
#pragma unroll
    for (int i = 0; i < kBatch; i++)
      if (ev[i] >= 0 && ev[i] < a.E) atomicAdd(&cnt[ev[i]], 1);
  }
  __syncthreads();
  const int n = cnt[t], nt = (n + a.tile_rows - 1) / a.tile_rows;
  pos[t] = n;
  tile[t] = nt;
  __syncthreads();
  for (int d = 1; d < kSortThreads; d <<= 1) {  // inclusive scans
    const int p = t >= d ? pos[t - d] : 0, q = t >= d ? tile[t - d] : 0;
    __syncthreads();
    pos[t] += p;
    tile[t] += q;
    __syncthreads();
  }
  const int p0 = pos[t] - n, t0 = tile[t] - nt;
  if (t == kSortThreads - 1) {
    a.totals[0] = pos[t];
    a.totals[1] = tile[t];
  }
  __syncthreads();
  cnt[t] = p0;  // the next free place of the expert's run
  if (nt > 0) {
    const int rows = ((n + nt - 1) / nt + 15) / 16 * 16;
    for (int i = 0; i < nt; i++) {
      const int r0 = i * rows, left = n - r0;
      a.tiles[t0 + i] = MoeTile{t, p0 + r0, left < 0 ? 0 : left < rows ? left : rows, 0};
    }
  }
  __syncthreads();
  for (int s0 = t; s0 < a.slots; s0 += kSortThreads * kBatch) {
    int ev[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; i++) ev[i] = s0 + kSortThreads * i < a.slots ? a.topk_ids[s0 + kSortThreads * i] : -1;
#pragma unroll
    for (int i = 0; i < kBatch; i++)
      if (ev[i] >= 0 && ev[i] < a.E) a.sorted[atomicAdd(&cnt[ev[i]], 1)] = int2{s0 + kSortThreads * i, ev[i]};
  }
}

// The rotated gate and up inputs of every routed slot of the class by sorted position, in fragment order: one wave per
// (16 positions, 128-block), both projections from one load of x (2048 tokens: 51 us with the butterfly on 16 lanes per
// row, 39 so; 134 MB written).
template <bool X_BF16>
__global__ __launch_bounds__(256) void moe_gemm_in_kernel(MoeGemmArgs a, const uint16_t* __restrict__ x) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, c = l & 15, j = l >> 4;
  const int pos0 = (blockIdx.x * 4 + w) * 16, b = blockIdx.y, total = a.totals[0];
  if (pos0 >= total) return;  // wave-uniform
  const int pos = pos0 + c;
  const int2 at = a.sorted[pos < total ? pos : total - 1];
  const int el = moe_row(a, at.y);  // -1: another class's row, read as expert 0's and not stored
  const size_t kk = b * 128 + 8 * j, e0 = (size_t)(el < 0 ? 0 : el) * a.H;
  half8_t xv[4];
  load_row_frags<X_BF16>(x + (size_t)(at.x / a.top_k) * a.H + kk, xv);
  const HadFrags had = had_frags_act(l);
#pragma unroll
  for (int s = 0; s < 2; s++) {
    half8_t in[4];
#pragma unroll
    for (int kb = 0; kb < 4; kb++) in[kb] = times8(xv[kb], a.suh[s] + e0 + kk + 32 * kb);
    uint16_t* dst = a.pre_in + ((size_t)(s * (a.H >> 5) + b * 4) * a.slots + pos) * 32 + 8 * j;
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const half8_t o = had_pair(had, in, u);
      if (pos < total && el >= 0) *reinterpret_cast<half8_t*>(dst + (size_t)u * a.slots * 32) = o;
    }
  }
}

// The tile and column block of a workgroup.  Workgroup ids that agree mod 8 run on one XCD: all column blocks of a tile
// get such ids, so the tile's activations come into one XCD's L2 once (any other assignment is only slower).
struct MoeWork {
  int tile, cb;
};
__device__ __forceinline__ MoeWork moe_work(int id, int ncb) {
  const int r = id >> 3, q = r / ncb;
  return MoeWork{q * 8 + (id & 7), r - q * ncb};
}

// acc = the tile's product for a wave's 32 columns, on 16 MI rows.  AP: pieces per stage (MI, or 2 MI with gate and up
// inputs); part: the wave's projection (its fragments' place in the stage).
template <int K, int CB, int MI, int AP>
__device__ __forceinline__ void moe_multiply(const MoeGemmArgs& a, const uint16_t* pre, int k, const MoeTile& tile,
                                             const uint32_t* trellis, int tn, int tc, int part, uint8_t* lds, int w,
                                             int l, float4_t (&acc)[MI][2]) {
  constexpr int PIECES = (AP + kGemmWaves - 1) / kGemmWaves;
  const int c = l & 15, j = l >> 4;
  ActLoads<PIECES> act;
  const int steps = k / kBK;
  act.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)pre, (short)0, (int)((size_t)(AP / MI) * k * a.slots * 2), 0x00020000);
  act.step = a.slots * kBK * 2;
  act.stage = AP * 1024;
#pragma unroll
  for (int q = 0; q < PIECES; q++) {
    const int p = PIECES * w + q, piece = p < AP ? p : p % AP;
    const int r = (piece % MI) * 16 + c, row = r < tile.rows ? r : tile.rows - 1;
    act.src[q] = (((piece / MI) * steps * a.slots + tile.pos0 + row) * 32 + j * 8) * 2;
    act.dst[q] = piece * 1024;
  }
  const int tile_bytes = 32 * K, row_bytes = tn * tile_bytes;
  const __amdgpu_buffer_rsrc_t brsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)trellis, (short)0, (k >> 4) * row_bytes, 0x00020000);
  const BitsLane bl = bits_lane<K>(l);
  const int bgoff = bl.row * row_bytes + (tc + bl.col) * tile_bytes + bl.piece * 16;
#pragma unroll
  for (int mi = 0; mi < MI; mi++)
#pragma unroll
    for (int jj = 0; jj < 2; jj++) acc[mi][jj] = float4_t{0.f, 0.f, 0.f, 0.f};
  tile_multiply<K, CB, MI, PIECES>(
      lds, act, part * MI * 1024, lds + kARing * AP * 1024 + w * 1024, brsrc, bgoff,
      [&](int kt) { return 2 * kt * row_bytes; }, 0, steps, (w & 4) != 0, l, acc);
}

// 128 columns of gate (waves 0-3) and the same of up (waves 4-7), then per 16-row block in one wave: both output
// rotations, the GLU, * suh_down and its rotation, whose results are whole fragments of the down inputs.  The rotated
// blocks stay in registers between the two rotations: a lane's 8 results of pair u are its fragment of the next product.
template <int K, int CB, int MI>
__device__ __forceinline__ void moe_gate_up_tile(const MoeGemmArgs& a, const MoeTile& tile, int el, int cb,
                                                 uint8_t* lds) {
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
  const int c = l & 15, j = l >> 4;
  const int tn = a.I / 16, part = w >> 2;
  const size_t mat_dwords = (size_t)(a.H / 16) * tn * 8 * K;
  const uint32_t* trellis = (part ? a.tr[1] : a.tr[0]) + el * mat_dwords;
  float4_t acc[MI][2];
  moe_multiply<K, CB, MI, 2 * MI>(a, a.pre_in, a.H, tile, trellis, tn, cb * 8 + 2 * (w & 3), part, lds, w, l, acc);
  _Float16* cl = reinterpret_cast<_Float16*>(lds);
  tile_to_lds<MI>(cl, acc, w, l);
  __syncthreads();
  const HadFrags rows = had_frags_rows(l), frag = had_frags_act(l);
  const int kk = cb * 128 + 8 * j;
  const uint16_t* svg = a.svh[0] + (size_t)el * a.I + kk;
  const uint16_t* svu = a.svh[1] + (size_t)el * a.I + kk;
  const uint16_t* su = a.suh[2] + (size_t)el * a.I + kk;
  for (int mi = w; mi < MI && mi * 16 < tile.rows; mi += kGemmWaves) {
    const half8_t* src = reinterpret_cast<const half8_t*>(cl + (mi * 16 + c) * kCStride + 8 * j);
    half8_t gf[4], uf[4], in[4];
#pragma unroll
    for (int kb = 0; kb < 4; kb++) {
      gf[kb] = src[kb * 4];
      uf[kb] = src[16 + kb * 4];
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const half8_t gv = times8(had_pair(rows, gf, u), svg + 32 * u), uv = times8(had_pair(rows, uf, u), svu + 32 * u);
      half8_t av;
#pragma unroll
      for (int e = 0; e < 8; e++) av[e] = f16_of_f32(silu32((float)gv[e]) * (float)uv[e]);
      in[u] = times8(av, su + 32 * u);
    }
    const int r = mi * 16 + c;
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const half8_t o = had_pair(frag, in, u);
      if (r < tile.rows)
        *reinterpret_cast<half8_t*>(a.pre_dn + ((size_t)(cb * 4 + u) * a.slots + tile.pos0 + r) * 32 + 8 * j) = o;
    }
  }
}

// 256 columns of down (128 at the end of an odd count), rotated, * svh, one row per slot
template <int K, int CB, int MI>
__device__ __forceinline__ void moe_down_tile(const MoeGemmArgs& a, const MoeTile& tile, int el, int cb, uint8_t* lds) {
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
  const int c = l & 15, j = l >> 4;
  const int tn = a.H / 16, ntc = tn - cb * 16;  // tile columns left: 8, or 16 and more
  const bool live = 2 * w < ntc;                // the wave's 32 columns exist (else it re-reads the tile's first)
  const size_t mat_dwords = (size_t)(a.I / 16) * tn * 8 * K;
  float4_t acc[MI][2];
  moe_multiply<K, CB, MI, MI>(a, a.pre_dn, a.I, tile, a.tr[2] + el * mat_dwords, tn, cb * 16 + (live ? 2 * w : 0), 0,
                              lds, w, l, acc);
  _Float16* cl = reinterpret_cast<_Float16*>(lds);
  if (live) tile_to_lds<MI>(cl, acc, w, l);
  __syncthreads();
  const HadFrags rows = had_frags_rows(l);
  for (int p = w; p < MI * 2; p += kGemmWaves) {
    const int mi = p >> 1, h = p & 1, r = mi * 16 + c;
    if (8 * h >= ntc || mi * 16 >= tile.rows) continue;  // wave-uniform
    const half8_t* src = reinterpret_cast<const half8_t*>(cl + (mi * 16 + c) * kCStride + h * 128 + 8 * j);
    half8_t cf[4];
#pragma unroll
    for (int kb = 0; kb < 4; kb++) cf[kb] = src[kb * 4];
    const int col = cb * 256 + h * 128 + 8 * j;
    const int slot = a.sorted[tile.pos0 + (r < tile.rows ? r : tile.rows - 1)].x;
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const half8_t o = times8(had_pair(rows, cf, u), a.svh[2] + (size_t)el * a.H + col + 32 * u);
      if (r < tile.rows) *reinterpret_cast<half8_t*>(a.dn + (size_t)slot * a.H + col + 32 * u) = o;
    }
  }
}

// A tile of at most 64 slots takes the 64-row code also where tiles go up to 128, and one of at most 32 the 32-row code
// where there are more workgroups than CUs, which then share issue slots (128 experts, top-8, 256 tokens: 161.6 -> 145.1
// us; 2048 tokens 407 -> 404).  With at most one workgroup per CU a step's latency sets the time, and less work per step
// only hides less of it (16 experts, 61 tokens, two layers: 142.5 us at 64 rows, 144.5 at 32).  64-row kernels are held
// to 128 VGPRs: two workgroups per CU.
template <int K, int CB, int PHASE, int MI>
__global__ __launch_bounds__(kGemmThreads, MI == 4 ? 4 : 2) void moe_gemm_kernel(MoeGemmArgs a) {
  extern __shared__ __align__(16) uint8_t lds[];
  const int ncb = PHASE ? (a.H + 255) / 256 : a.I / 128, tiles = a.totals[1];
  const MoeWork wk = moe_work(blockIdx.x, ncb);
  if (wk.tile >= tiles) return;
  const MoeTile tile = a.tiles[wk.tile];
  const int el = moe_row(a, tile.expert);
  if (el < 0 || tile.rows <= 0) return;
  const bool low = tile.rows <= 32 && tiles * ncb > 256;  // workgroup-uniform
  if constexpr (PHASE == 0) {
    if (low)
      moe_gate_up_tile<K, CB, 2>(a, tile, el, wk.cb, lds);
    else if (MI == 4 || tile.rows <= 64)
      moe_gate_up_tile<K, CB, 4>(a, tile, el, wk.cb, lds);
    else
      moe_gate_up_tile<K, CB, MI>(a, tile, el, wk.cb, lds);
  } else {
    if (low)
      moe_down_tile<K, CB, 2>(a, tile, el, wk.cb, lds);
    else if (MI == 4 || tile.rows <= 64)
      moe_down_tile<K, CB, 4>(a, tile, el, wk.cb, lds);
    else
      moe_down_tile<K, CB, MI>(a, tile, el, wk.cb, lds);
  }
}

int moe_gemm_route(const MoeGemmArgs& a, hipStream_t st) {
  moe_sort_kernel<<<1, kSortThreads, 0, st>>>(a);
  EXL3_CHECK_LAUNCH();
  return EXL3_OK;
}

int moe_gemm_inputs(const MoeGemmArgs& a, const void* x, bool x_bf16, hipStream_t st) {
  const dim3 grid((unsigned)((a.slots + 63) / 64), (unsigned)(a.H / 128));
  if (x_bf16)
    moe_gemm_in_kernel<true><<<grid, 256, 0, st>>>(a, static_cast<const uint16_t*>(x));
  else
    moe_gemm_in_kernel<false><<<grid, 256, 0, st>>>(a, static_cast<const uint16_t*>(x));
  EXL3_CHECK_LAUNCH();
  return EXL3_OK;
}

template <int PHASE>
static int launch(const MoeGemmArgs& a, int K, int codebook, hipStream_t st) {
  const int ncb = PHASE ? (a.H + 255) / 256 : a.I / 128;
  const int tiles = (moe_gemm_max_tiles(a.slots, a.E, a.tile_rows) + 7) / 8 * 8;
  const dim3 grid((unsigned)(tiles * ncb));
  const int pieces = PHASE ? a.tile_rows / 16 : a.tile_rows / 8;
#define EXL3_MG(KV, CV)                                                                                             \
  case KV * 4 + CV:                                                                                                 \
    if (a.tile_rows == 64)                                                                                          \
      moe_gemm_kernel<KV, CV, PHASE, 4><<<grid, kGemmThreads, tile_lds(4, pieces), st>>>(a);                       \
    else                                                                                                            \
      moe_gemm_kernel<KV, CV, PHASE, 8><<<grid, kGemmThreads, tile_lds(8, pieces), st>>>(a);                       \
    break;
#define EXL3_MGK(KV) EXL3_MG(KV, 0) EXL3_MG(KV, 1) EXL3_MG(KV, 2)
  switch (K * 4 + codebook) {
    EXL3_MGK(2) EXL3_MGK(3) EXL3_MGK(4) EXL3_MGK(5) EXL3_MGK(6) EXL3_MGK(8)
    default:
      return set_error(EXL3_ERR_INVALID, "moe: unsupported K = %d / codebook = %d", K, codebook);
  }
#undef EXL3_MGK
#undef EXL3_MG
  EXL3_CHECK_LAUNCH();
  return EXL3_OK;
}

int moe_gemm_gate_up(const MoeGemmArgs& a, int K, int codebook, hipStream_t st) { return launch<0>(a, K, codebook, st); }
int moe_gemm_down(const MoeGemmArgs& a, int K, int codebook, hipStream_t st) { return launch<1>(a, K, codebook, st); }

}  // namespace exl3
