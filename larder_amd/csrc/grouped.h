// What the grouped GEMM kernels share (grouped.hip: Q4_0 / Q4_K and f16 weights; grouped_any.hip: the block types
// decoded from registers): tile sizes and the work list, the LDS layout of A rows, the epilogue, and the global -> LDS
// copies.
#pragma once
#include <type_traits>

#include "lmoe_common.h"

namespace lmoe {

template <int N>
using IC = std::integral_constant<int, N>;

// f(IC<0>), f(IC<1>), ..., f(IC<N - 1>): a loop whose index is a compile-time constant in the body
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (I < N) {
    f(IC<I>{});
    static_for<I + 1, N>(f);
  }
}

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int GM = 128;  // rows a tile (the grouping kernel's bm)
constexpr int GN = 256;  // weight rows a tile (gate/up: 128 gate + 128 up features; down: 256 outputs)
constexpr int GK = 64;   // K a step (one 64-weight unit of every weight row)
constexpr int kThreads = 256;
constexpr int kTileMask = (1 << 20) - 1;

enum { MODE_GATE_UP = 0, MODE_DOWN = 1 };

// 16-byte chunk c (0..7) of A row r in a stage: rows are 128 bytes, chunks XOR-swizzled by the row's low 3 bits
__device__ __forceinline__ int achunk(int r, int c) { return r * 8 + (c ^ (r & 7)); }


// two f16 (1024 + byte) from a word's bytes: {b0, b1} or {b2, b3}
__device__ __forceinline__ uint32_t magic_pair(uint32_t nib, uint32_t sel) {
  return __builtin_amdgcn_perm(0x64646464u, nib, sel);
}
constexpr uint32_t kSel01 = 0x04010400u, kSel23 = 0x04030402u;

// Bytes 0, 1 (HI false) or 2, 3 of a word of nibbles (0 .. 15 a byte) as f16, exactly: read as fp8 (E4M3), 0 .. 7 are the
// subnormals n 2^-9 and 8 .. 15 the first binade (8 + m) 2^-9, so the conversion scaled by 2^9 gives the nibble. One
// instruction (4 cycles a SIMD, like each of the byte permute and the packed subtraction that it stands for).
template <bool HI>
__device__ __forceinline__ h2_t nibbles_f16(uint32_t v) {
  return __builtin_bit_cast(h2_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(v, 512.0f, HI));
}

// An MFMA lane's 8 f16 weights from its nibble word x (low nibbles: K positions 0-3 of the lane group, high
// nibbles: 4-7), one rounding a weight. Q4_0: w = ((1024 + q) - 1032) d, d = the selected half of sw. (fma(q, d, -8 d)
// on nibbles_f16 takes 4 instructions a word fewer and 0.8 % off a layer of 8,192 tokens, but its -8 d overflows f16 from
// |d| = 8192 on, where (q - 8) d may still fit.) Q4_K: sw = {f16(d sc), f16(dmin m)}, w = fma(q, d sc, -dmin m).
template <int TB>
__device__ __forceinline__ half8 decode8(uint32_t x, uint32_t sw, int half) {
  const uint32_t lo = x & 0x0F0F0F0Fu, hi = (x >> 4) & 0x0F0F0F0Fu;
  uint32_t o[4];
  if (TB == LMOE_Q4_0) {
    const _Float16 d = __builtin_bit_cast(h2_t, sw)[half];
    const uint32_t p[4] = {magic_pair(lo, kSel01), magic_pair(lo, kSel23), magic_pair(hi, kSel01), magic_pair(hi, kSel23)};
    const h2_t bias = {_Float16(1032.0f), _Float16(1032.0f)}, scale = {d, d};
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(h2_t, p[i]) - bias) * scale);
  } else {
    const h2_t q[4] = {nibbles_f16<false>(lo), nibbles_f16<true>(lo), nibbles_f16<false>(hi), nibbles_f16<true>(hi)};
    const h2_t v = __builtin_bit_cast(h2_t, sw), scale = {v[0], v[0]}, add = {-v[1], -v[1]};
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(q[i], scale, add));
  }
  return __builtin_bit_cast(half8, u32x4{o[0], o[1], o[2], o[3]});
}

// Tile bookkeeping shared by both kernels
struct Tile {
  int e, nt, row0, rows, kpart;
};

// XCD-aware remap: workgroup `wid` runs on XCD wid % 8; XCD x gets logical work [start_x, start_x + count_x).
// Returns false for workgroups past the device-side work count.
// ksplit > 1: each (tile, n-tile) is worked by ksplit workgroups, one a slice of K (t->kpart), next to each other
// in the logical order.
template <int GMT = GM>
__device__ __forceinline__ bool tile_of(const uint32_t *offsets, const uint32_t *tiles, const uint32_t *n_tiles,
                                        int n_ntile, Tile *t, int ksplit = 1) {
  const uint32_t W = n_tiles[0] * uint32_t(n_ntile) * uint32_t(ksplit);
  const uint32_t wid = blockIdx.x;
  if (wid >= W) return false;
  const uint32_t q8 = W >> 3, r8 = W & 7, xcd = wid & 7;
  const uint32_t logical0 = xcd * q8 + min(xcd, r8) + (wid >> 3);
  t->kpart = int(logical0 % uint32_t(ksplit));
  const uint32_t logical = logical0 / uint32_t(ksplit);
  const uint32_t tile = tiles[logical / uint32_t(n_ntile)];
  t->nt = int(logical % uint32_t(n_ntile));
  t->e = int(tile >> 20);
  t->row0 = int(offsets[t->e]) + int(tile & kTileMask) * GMT;
  t->rows = min(GMT, int(offsets[t->e + 1]) - t->row0);
  return true;
}

// Tile features of a wavefront's 4 fragments: gate/up: gate 32 w + 16 nb (nb < 2), up 128 + 32 w + 16 (nb - 2)
// (the same intermediate features); down: 64 w + 16 nb
template <int MODE>
__device__ __forceinline__ int frag_feature(int wave, int nb) {
  return MODE == MODE_GATE_UP ? (nb < 2 ? 32 * wave + 16 * nb : GN / 2 + 32 * wave + 16 * (nb - 2))
                              : 64 * wave + 16 * nb;
}

// Two f16 of a, b packed in one word
__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
  return __builtin_bit_cast(uint32_t, h2_t{_Float16(a), _Float16(b)});
}

// Two bf16 of a, b packed in one word (round to nearest even)
__device__ __forceinline__ uint32_t pack_bf2(float a, float b) {
  typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
  typedef float f2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2_t{a, b}, bf2_t));
}

// acc[nb][mb][r] = D[tile feature frag_feature(nb) + 4 g + r][tile row 16 mb + fr]. Every store is 16 bytes:
//   * gate/up: h (f16, K order) = silu(gate) * up. A lane's features 4g..4g+3 of fragments 0 and 1 (32 w + 4g.. and
//     32 w + 16 + 4g.. of the n-tile) sit at K-order positions 8g..8g+3 and 8g+4..8g+7 of their 32-block: one store;
//   * down, 16-bit: fragments nb and nb + 1 meet through one permlane16 swap a word: lane group g then holds 8
//     consecutive features, of fragment nb + (g & 1), from 8 (g >> 1) on, so a row's 32 features of the pair go out
//     as one 64-byte run; f32: each fragment's 4 features as they are.
// Down rows go to row p of out (grouped order), or with `order` to row order[p] (the caller's order; a zero is stored as
// +0, also where a negative sum rounds to it in f16, as a sum over one row's output in out's dtype would give it).
// Called by every lane of the workgroup (the swaps read the lanes 16 away); rows past the tile's end store nothing.
template <int MODE, bool ROWS, int MB>
__device__ __forceinline__ void store_tile_as(f32x4 (&acc)[4][MB], const Tile &t, int wave, int fr, int g, void *out,
                                              int ldo, int odt, const uint32_t *order) {
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int m = 16 * mb + fr;
    const bool ok = m < t.rows;
    size_t row = size_t(t.row0 + (ok ? m : 0));
    if (ROWS) {
      row = order[row];
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) acc[nb][mb] += 0.0f;
    }
    const size_t o = row * ldo;
    if (MODE == MODE_GATE_UP) {
      uint32_t v[4];
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 2; ++r)
          v[2 * nb + r] = pack_h2(silu_mul_h(acc[nb][mb][2 * r], acc[nb + 2][mb][2 * r]),
                                  silu_mul_h(acc[nb][mb][2 * r + 1], acc[nb + 2][mb][2 * r + 1]));
      const int n0 = t.nt * (GN / 2) + frag_feature<MODE>(wave, 0);  // a multiple of 32
      if (ok) *reinterpret_cast<u32x4 *>(static_cast<_Float16 *>(out) + o + n0 + 8 * g) = u32x4{v[0], v[1], v[2], v[3]};
    } else if (odt == LMOE_F32) {
      if (ok) {
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
          *reinterpret_cast<f32x4 *>(static_cast<float *>(out) + o + t.nt * GN + frag_feature<MODE>(wave, nb) +
                                     4 * g) = acc[nb][mb];
      }
    } else {
      auto pack = [&](float a, float b) {
        if (ROWS && odt == LMOE_BF16) return pack_bf2(a, b);
        h2_t v = {_Float16(a), _Float16(b)};
        if (ROWS) v += h2_t{_Float16(0.0f), _Float16(0.0f)};
        return __builtin_bit_cast(uint32_t, v);
      };
#pragma unroll
      for (int pr = 0; pr < 2; ++pr) {
        const int nb = 2 * pr;
        const auto s0 = __builtin_amdgcn_permlane16_swap(pack(acc[nb][mb][0], acc[nb][mb][1]),
                                                         pack(acc[nb + 1][mb][0], acc[nb + 1][mb][1]), false, false);
        const auto s1 = __builtin_amdgcn_permlane16_swap(pack(acc[nb][mb][2], acc[nb][mb][3]),
                                                         pack(acc[nb + 1][mb][2], acc[nb + 1][mb][3]), false, false);
        const uint32_t a0 = s0[0], b0 = s0[1], a1 = s1[0], b1 = s1[1];
        const int n = t.nt * GN + frag_feature<MODE>(wave, nb + (g & 1)) + 8 * (g >> 1);
        if (ok) *reinterpret_cast<u32x4 *>(static_cast<uint16_t *>(out) + o + n) = u32x4{a0, a1, b0, b1};
      }
    }
  }
}

template <int MODE, int MB = 8>
__device__ __forceinline__ void store_tile(f32x4 (&acc)[4][MB], const Tile &t, int wave, int fr, int g, void *out,
                                           int ldo, int odt, const uint32_t *order) {
  if (MODE == MODE_DOWN && order)  // uniform: one test a tile (tests a row block cost prompts 1-2%)
    store_tile_as<MODE, true>(acc, t, wave, fr, g, out, ldo, odt, order);
  else
    store_tile_as<MODE, false>(acc, t, wave, fr, g, out, ldo, odt, order);
}

// The GEMMs that decode Q4_1 / Q8_0 / Q5_K / Q6_K (grouped_any.hip), shape checks included. mode gate/up: n_rows = I, a
// gathered through order; down: n_rows = H, order the output rows (nullptr: grouped order).
int grouped_any(const char *fn, int mode, const void *a, long long a_rows, int topk, const uint32_t *order,
                const uint32_t *offsets, const uint32_t *tiles, const uint32_t *n_tiles, int max_tiles, int bm,
                const uint8_t *w0, const uint8_t *w1, int type, int n_experts, int K, int n_rows, void *out, int odt,
                hipStream_t st);

// A wavefront-uniform pointer held in scalar registers (the copy instructions take their base there)
template <typename P>
__device__ __forceinline__ P *uniform(P *p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(v)), hi = __builtin_amdgcn_readfirstlane(uint32_t(v >> 32));
  return reinterpret_cast<P *>((uint64_t(hi) << 32) | lo);
}

// One wavefront-wide global -> LDS copy: lane l's `BYTES` (4 or 16) at base + voff land at LDS address
// lds + l * BYTES (global_load_lds_dwordx3 would also step 16 bytes a lane). M0 carries the LDS address; nothing
// else in these kernels uses M0.
template <int BYTES>
__device__ __forceinline__ void dma(const void *base_any, uint32_t voff, uint32_t lds) {
  const void *base = uniform(base_any);
  if (BYTES == 16)
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(lds) : "memory");
  else
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(base), "s"(lds) : "memory");
}

// The A copies of a tile whose rows end early: copy i of wavefront w (D copies a wavefront a step) moves tile rows
// [8 (D w + i), +8); bit i of the mask says whether any of them is a row of the tile. A copy of rows past the end
// becomes a 4-byte copy of one address into the same place (the rows' LDS bytes are never stored: their output
// rows are masked), so every wavefront still issues the same number of copies a step and the counted waits hold,
// while the padding rows of a short group (~40 rows in a 64-row tile, ~5 in a 32-row one) cost no A bytes.
template <int D>
__device__ __forceinline__ uint32_t a_live_mask(int wave, int rows) {
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < D; ++i) m |= (8 * (D * wave + i) < rows ? 1u : 0u) << i;
  return __builtin_amdgcn_readfirstlane(m);
}

__device__ __forceinline__ void dma_a(const _Float16 *ab, uint32_t off, uint32_t lds, uint32_t live) {
  if (live)
    dma<16>(ab, off, lds);
  else
    dma<4>(ab, 0u, lds);
}

// A barrier that publishes this wavefront's LDS writes and lets other wavefronts overwrite what it has read: its own LDS
// operations are waited for first (issued is not done: another SIMD's read can pass a write still queued), with compiler
// memory fences on both sides. __syncthreads' release fence would also wait for every copy in flight, including the ones
// meant to stay in flight.
__device__ __forceinline__ void barrier_lds() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// s_waitcnt on the vector-memory counter only (the copies this wavefront issued), N outstanding at most
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

}  // namespace lmoe
