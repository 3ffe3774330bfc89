// The decode-and-multiply core of the decode-GEMMs (dense prefill, MoE experts) on gfx950, and their rotation by MFMA.
//
// A workgroup of 8 waves multiplies a tile of 16 MI rows by 256 columns, 32 columns per wave.  A k-step covers 32 rows
// of the weights = 2 tile rows.  Wave w decodes the weights of its own two tile columns into registers, each once, and
// multiplies them (the MFMA's A operand) with the activation fragments of all rows from LDS (its B operand): no decoded
// weight goes through LDS, only the activations are shared between waves, and a lane's accumulator holds 4 consecutive
// columns of one row.
#pragma once
#include <type_traits>

#include "exl3_device.hpp"

namespace exl3 {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// 8 fp16 (or raw 16-bit) values by two 8-byte loads: the tensors need no more alignment
__device__ __forceinline__ u32x4 load8(const uint16_t* p) {
  const u32x2 a = *reinterpret_cast<const u32x2*>(p), b = *reinterpret_cast<const u32x2*>(p + 4);
  return u32x4{a.x, a.y, b.x, b.y};
}

__device__ __forceinline__ half8_t times8(half8_t v, const uint16_t* p) {
  const half8_t s = __builtin_bit_cast(half8_t, load8(p));
#pragma unroll
  for (int e = 0; e < 8; e++) v[e] = (_Float16)(v[e] * s[e]);
  return v;
}

// A row's 128 values as MFMA fragments: v[kb] = values 32 kb ..+7 from p (the lane's 8 l / 16 included), bf16 rounded to
// fp16
template <bool X_BF16>
__device__ __forceinline__ void load_row_frags(const uint16_t* p, half8_t (&v)[4]) {
  u32x4 raw[4];
#pragma unroll
  for (int kb = 0; kb < 4; kb++) raw[kb] = load8(p + 32 * kb);
#pragma unroll
  for (int kb = 0; kb < 4; kb++) {
    v[kb] = __builtin_bit_cast(half8_t, raw[kb]);
    if constexpr (X_BF16)
#pragma unroll
      for (int e = 0; e < 8; e++)
        v[kb][e] = (_Float16)bf16_to_f32((uint16_t)((e & 1) ? raw[kb][e >> 1] >> 16 : raw[kb][e >> 1] & 0xFFFF));
  }
}

constexpr int kBN = 256, kBK = 32;
constexpr int kGemmWaves = 8, kGemmThreads = kGemmWaves * 64;
constexpr int kARing = 4, kBitsRing = 4;           // ring slots (powers of two)
constexpr int kWindow = 4;                         // A fragments a wave holds ahead of their MFMAs (at most MI)
constexpr int kBitsStage = kGemmWaves * 64 * 16;   // 8 KB: per wave 64 lanes x 16 B (its 4 tiles of a k-step)
constexpr int kCStride = kBN + 8;                  // epilogue fp16 C tile row stride (halves)
// LDS of a tile of 16 MI rows whose k-step stages hold `pieces` 1 KB activation pieces: the rings, or the C tile
__host__ __device__ constexpr int tile_lds(int MI, int pieces) {
  const int rings = kARing * pieces * 1024 + kBitsRing * kBitsStage, c = MI * 16 * kCStride * 2;
  return rings > c ? rings : c;
}

template <int K>
__host__ __device__ constexpr int gemm_chunks() { return 4 * 32 * K / 16; }  // 16-byte pieces of a wave's 4 tiles

// The lane's place in its wave's trellis loads: stage order [tile row][column][32K bytes], 16 bytes per lane (lanes past
// the 4 tiles repeat the last piece)
struct BitsLane {
  int row, col, piece;
};
template <int K>
__device__ __forceinline__ BitsLane bits_lane(int l) {
  constexpr int CHUNKS = gemm_chunks<K>();
  static_assert(CHUNKS <= 64, "one gather per wave per k-step");
  const int L = l < CHUNKS ? l : CHUNKS - 1;
  return BitsLane{L / (4 * K), L % (4 * K) / (2 * K), L % (2 * K)};
}

// Activations of a workgroup: per k-step stage, 1 KB pieces of 16 rows x 32 k in fragment order (a lane's 16 bytes are
// its MFMA fragment of row l % 16, k-chunk l / 16); this wave loads PIECES of them: `src` the lane's byte offset of a
// piece (+ k-step * step bytes), `dst` the piece's place in the stage.
template <int PIECES>
struct ActLoads {
  __amdgpu_buffer_rsrc_t rsrc;
  int src[PIECES], dst[PIECES];
  int step, stage;
};

// acc[mi][jj][r] += C[16 mi + l % 16][32 w + 16 jj + 4 (l / 16) + r] over k-steps [kt0, kt0 + nk).  frags: byte offset of
// the wave's row blocks inside a stage (1 KB each); bits_ring: the wave's first slot; boff(kt): byte offset of k-step kt
// in the trellis.  multiply_first: the order of a step's halves (the two waves of a SIMD, w and w + 4, take opposite
// ones).
//
// Loads come in bundles: bundle b = the activations of step b + the trellis bits of step b + 1 (PIECES + 1 loads per
// wave; past the end, steps clamp to the last one: in range, never used), issued three steps ahead of the activations'
// use and complete two steps later, one step before it: the barrier of step i publishes the activations of step i + 1,
// so a wave reads its next fragments before the step's last MFMAs and no step starts with an LDS round trip.  (boff gets
// clamped steps: lambdas here call no device-only function, whose host-side instantiation would otherwise suppress
// the kernel's host stub.)
template <int K, int CB, int MI, int PIECES, typename BitsOffset>
__device__ __forceinline__ void tile_multiply(uint8_t* a_ring, const ActLoads<PIECES>& act, int frags_at,
                                              uint8_t* bits_ring, __amdgpu_buffer_rsrc_t brsrc, int bgoff,
                                              BitsOffset boff, int kt0, int nk, bool multiply_first, int l,
                                              float4_t (&acc)[MI][2]) {
  constexpr int WINDOW = MI < kWindow ? MI : kWindow;
  const LaneGeo g = lane_geo<K>(l & 15, l >> 4);
  auto issue_a = [&](int i, int kt) {
    uint8_t* st = a_ring + (i & (kARing - 1)) * act.stage;
#pragma unroll
    for (int q = 0; q < PIECES; q++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(act.rsrc, (__attribute__((address_space(3))) void*)(st + act.dst[q]), 16,
                                               act.src[q], kt * act.step, 0, 0);
  };
  auto issue_bits = [&](int i, int kt) {
    uint8_t* st = bits_ring + (i & (kBitsRing - 1)) * kBitsStage;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(brsrc, (__attribute__((address_space(3))) void*)st, 16, bgoff, boff(kt), 0,
                                             0);
  };
  // this wave's trellis words of step i: [column][tile row][word]
  auto read_bits = [&](int i, uint32_t (&bw)[2][2][2]) {
    const uint32_t* tw = reinterpret_cast<const uint32_t*>(bits_ring + (i & (kBitsRing - 1)) * kBitsStage);
#pragma unroll
    for (int tr = 0; tr < 2; tr++)
#pragma unroll
      for (int jj = 0; jj < 2; jj++) {
        bw[jj][tr][0] = tw[(tr * 2 + jj) * 8 * K + g.dw0];
        bw[jj][tr][1] = tw[(tr * 2 + jj) * 8 * K + g.dw1];
      }
  };
  auto frags = [&](int i) {
    return reinterpret_cast<const half8_t*>(a_ring + (i & (kARing - 1)) * act.stage + frags_at) + l;
  };

  auto last = [&](int i) { return kt0 + (i < nk ? i : nk - 1); };
  issue_bits(0, kt0);
#pragma unroll
  for (int i = 0; i < 3; i++) {
    issue_a(i, last(i));
    issue_bits(i + 1, last(i + 1));
  }
  half8_t bcur[2], bnext[2], av[WINDOW];
  uint32_t bw[2][2][2];
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * (PIECES + 1)));  // bundle 0 in (bundles 1 and 2 may be in flight)
  lds_barrier();
  read_bits(0, bw);
#pragma unroll
  for (int jj = 0; jj < 2; jj++)
    bcur[jj] = decode_two_groups<K, CB>(bw[jj][0][0], bw[jj][0][1], bw[jj][1][0], bw[jj][1][1], g);
  read_bits(1, bw);
#pragma unroll
  for (int q = 0; q < WINDOW; q++) av[q] = frags(0)[q * 64];

  // step i: the weights `cur` of the step, `next` those of step i + 1, decoded here from the words in bw, which then
  // take step i + 2's
  auto step = [&](auto multiply_first, int i, const half8_t (&cur)[2], half8_t (&next)[2]) {
    // bundle i + 1 in; bundle i + 2 may still be in flight.  The barrier publishes the A of step i + 1 and retires
    // every read of step i - 1 (consumed by MFMAs issued before it), freeing its slot.
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(PIECES + 1));
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    issue_a(i + 3, last(i + 3));
    issue_bits(i + 4, last(i + 4));
    const half8_t *af = frags(i), *an = frags(i + 1);
    auto decode = [&]() {
#pragma unroll
      for (int jj = 0; jj < 2; jj++)
        next[jj] = decode_two_groups<K, CB>(bw[jj][0][0], bw[jj][0][1], bw[jj][1][0], bw[jj][1][1], g);
      read_bits(i + 2, bw);
    };
    auto multiply = [&]() {
#pragma unroll
      for (int mi = 0; mi < MI; mi++) {
        const half8_t a = av[mi % WINDOW];
        av[mi % WINDOW] = mi + WINDOW < MI ? af[(mi + WINDOW) * 64] : an[(mi + WINDOW - MI) * 64];
#pragma unroll
        for (int jj = 0; jj < 2; jj++)
          acc[mi][jj] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cur[jj], a, acc[mi][jj], 0, 0, 0);
      }
    };
    // the two waves of a SIMD (w and w + 4) take the step's halves in opposite order
    if constexpr (decltype(multiply_first)::value) {
      multiply();
      decode();
    } else {
      decode();
      multiply();
    }
  };
  auto steps = [&](auto multiply_first) {  // in pairs, so that the weights change registers without copies
    int i = 0;
    for (; i + 2 <= nk; i += 2) {
      step(multiply_first, i, bcur, bnext);
      step(multiply_first, i + 1, bnext, bcur);
    }
    if (i < nk) step(multiply_first, i, bcur, bnext);
  };
  if (MI >= 8 && multiply_first)
    steps(std::integral_constant<bool, (MI >= 8)>{});
  else
    steps(std::false_type{});
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));  // drain the trailing re-reads of every wave before LDS is reused
  __syncthreads();
}

// The wave's accumulators as fp16 (rounded once) into the C tile, 4 columns of a row per 8-byte write
template <int MI>
__device__ __forceinline__ void tile_to_lds(_Float16* cl, const float4_t (&acc)[MI][2], int w, int l) {
  const int c = l & 15, j = l >> 4;
#pragma unroll
  for (int mi = 0; mi < MI; mi++)
#pragma unroll
    for (int jj = 0; jj < 2; jj++) {
      const float4_t v = acc[mi][jj];
      *reinterpret_cast<half4_t*>(cl + (mi * 16 + c) * kCStride + w * 32 + jj * 16 + 4 * j) =
          half4_t{(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
    }
}

// Rotation by MFMA: y^T = H C^T of a 16-row x 128-column block, H the +-1 Hadamard matrix (exact in fp16; products and
// sums in fp32).  in[kb]: the lane's fragment C[l % 16][32 kb + 8 (l / 16) ..+7]; the results of the MFMA pair t = 2u,
// 2u + 1 are y[l % 16][n(t, 4 (l / 16) + r)].  The order n of H's rows decides where a lane's results lie; the sign of
// H[n][k] splits into a part of the lane and e (the fragment f0), one of t & 1 (f1 against f0) and one of (u, kb).
struct HadFrags {
  half8_t f0, f1;
};
// n(t, i) = 32 u + 8 (i / 4) + 4 (t & 1) + i % 4: a lane's 8 results of a pair are the consecutive columns
// 32 u + 8 (l / 16) ..+7
__device__ __forceinline__ HadFrags had_frags_rows(int l) {
  const int i = l & 15, j = l >> 4;
  HadFrags f;
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const int odd = __builtin_popcount(((i & 3) & (e & 3)) | (((i >> 2) & j) << 2)) & 1;
    f.f0[e] = odd ? (_Float16)-1.0f : (_Float16)1.0f;
    f.f1[e] = (e & 4) ? -f.f0[e] : f.f0[e];
  }
  return f;
}
// n(t, i) = 32 u + 16 (t & 1) + 2 (i / 4) + i % 2 + 8 (i / 2 % 2): the 8 results are the lane's 16 bytes of the next
// product's activation fragment (k-chunk l / 16)
__device__ __forceinline__ HadFrags had_frags_act(int l) {
  const int i = l & 15, j = l >> 4;
  HadFrags f;
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const int odd = __builtin_popcount((i & e & 1) | (((i >> 2) & (e >> 1)) << 1) | (((i >> 1) & j & 1) << 3)) & 1;
    f.f0[e] = odd ? (_Float16)-1.0f : (_Float16)1.0f;
    f.f1[e] = (j & 2) ? -f.f0[e] : f.f0[e];
  }
  return f;
}
// The pair u's 8 results, * 1/sqrt(128), each rounded to fp16
__device__ __forceinline__ half8_t had_pair(const HadFrags& f, const half8_t (&in)[4], int u) {
  half8_t o;
#pragma unroll
  for (int v = 0; v < 2; v++) {
    float4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < 4; kb++) {
      const half8_t hf = v ? f.f1 : f.f0;
      d = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_popcount(u & kb) & 1 ? -hf : hf, in[kb], d, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) o[4 * v + r] = had_scale_f16(d[r]);
  }
  return o;
}

}  // namespace exl3
