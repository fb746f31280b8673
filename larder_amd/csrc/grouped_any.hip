// Grouped expert GEMMs that decode the block types without a Q4 kernel (Q4_1, Q8_0, Q5_K, Q6_K) inside the GEMM, in
// place of dequantizing every expert to f16 in HBM first (the reference's own dense path: gguf_experts.py:698-722,
// DEQ_SRC :529-539).
//
// Tiles, work list, wavefront split (4 wavefronts, each all tile rows x 64 weight rows), MFMA fragments, K order and
// epilogue are k_grouped_f16w's (grouped.hip), and each weight is rounded to f16 as lmoe_dequant_gemm_f16 rounds it, so
// the results are that kernel's on the dequantized weights, bit for bit. What differs is how weights reach the MFMA:
//   * a step is 128 of K: four 32-wide MFMA slices, four 32-weight blocks or half a super-block of every row. A
//     wavefront loads its own 64 rows' bytes into registers two steps ahead, neighbouring lanes on neighbouring bytes of
//     a row, and writes them to its own part of LDS at their step's start: no barrier waits for weights, and only A has
//     two stages;
//   * a lane then reads the words of its 8 weights a slice and decodes them in registers;
//   * a tile is 64 rows: two steps of weights in flight beside 64 accumulators take all 256 VGPRs (32-40 spilled for Q8_0,
//     20 for Q5_K, 3-7 for Q6_K, none for Q4_1; the reloads stand outside the K loops). A 128-row tile of the grouping is
//     worked as two, each decoding every weight.
// Bound: LDS reads and the decode's vector work (15 instructions for 8 weights at Q8_0, ~25 at Q6_K, beside one MFMA for
// each 16 rows) at many rows an expert, the weights' latency at few. Measured on one box, us for gate/up and down
// (dequantizing each matrix to f16, 140-158 us each, plus the f16-weight GEMMs -> this kernel):
//   Q8_0, 3,001 rows, 60 experts of 2048 x 1408          283 + 139 and 142 + 93 -> 127 and 71
//   Q6_K, 16,384 rows, 128 experts of 2048 x 768         316 + 215 and 158 + 138 -> 278 and 161
//   Q8_0 / Q6_K, 65,536 rows, the same experts           853 / 886 and 539 / 548 -> 695 / 795 and 485 / 481
// Past some 500 (Q6_K) to 1,200 (Q8_0) rows an expert the copy is the faster way again, since it is made once and a block
// is decoded once a tile (262,144 rows, the same experts, Q6_K: 2,350 and 1,325 against 3,043 and 1,736); the caller picks.
// Loads with each lane on the row its MFMA operand wants (and 4 x 4 word transposes between lane groups in place of LDS)
// took 221 and 87 us at the first line: neighbouring lanes then look up a cache line each. One step of weights ahead
// instead of two: 130 and 74, Q4_1 101 and 58 against 91 and 53.
#include "grouped.h"

namespace lmoe {

typedef uint32_t u32x4h __attribute__((ext_vector_type(4), aligned(2)));  // 16 bytes at any 2-byte aligned address
typedef uint32_t u32x2h __attribute__((ext_vector_type(2), aligned(2)));

__device__ __forceinline__ half8 half8_of(const uint32_t *o) {
  return __builtin_bit_cast(half8, u32x4{o[0], o[1], o[2], o[3]});
}

// The bytes of a and b as f16 pairs 1024 + byte
__device__ __forceinline__ void byte_pairs(uint32_t a, uint32_t b, h2_t *p) {
  p[0] = __builtin_bit_cast(h2_t, magic_pair(a, kSel01));
  p[1] = __builtin_bit_cast(h2_t, magic_pair(a, kSel23));
  p[2] = __builtin_bit_cast(h2_t, magic_pair(b, kSel01));
  p[3] = __builtin_bit_cast(h2_t, magic_pair(b, kSel23));
}

// f16(q s + c) for the 4 bytes q of a (s[0], c[0]) and of b (s[1], c[1]), given as f16 1024 + q pairs with c less 1024 s,
// where the result is exact in float32: one instruction a weight. A half-register write needs a wait state before its
// register is read: the low halves go first, and s_nop stands after the last.
__device__ __forceinline__ half8 fma_pairs_exact(const h2_t *q, const float *s, const float *c) {
  uint32_t o[4];
  asm("v_fma_mixlo_f16 %0, %4, %8, %10 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixlo_f16 %1, %5, %8, %10 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixlo_f16 %2, %6, %9, %11 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixlo_f16 %3, %7, %9, %11 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %0, %4, %8, %10 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %1, %5, %8, %10 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %2, %6, %9, %11 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %3, %7, %9, %11 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "s_nop 1"
      : "=&v"(o[0]), "=&v"(o[1]), "=&v"(o[2]), "=&v"(o[3])
      : "v"(__builtin_bit_cast(uint32_t, q[0])), "v"(__builtin_bit_cast(uint32_t, q[1])),
        "v"(__builtin_bit_cast(uint32_t, q[2])), "v"(__builtin_bit_cast(uint32_t, q[3])), "v"(s[0]), "v"(s[1]),
        "v"(c[0]), "v"(c[1]));
  return half8_of(o);
}

// f16(float32(q s + c)) for the 4 bytes q of a (s[0], c[0]) and of b (s[1], c[1]): the product is exact, the sum rounds to
// float32, then to f16 (lmoe_dequant's steps; v_fma_mixlo_f16 would round once, which differs in about one weight of 10
// million).
__device__ __forceinline__ half8 fma_bytes(uint32_t a, uint32_t b, const float *s, const float *c) {
  half8 w;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float v = fmaf(float(((i < 4 ? a : b) >> (8 * (i & 3))) & 0xffu), s[i >> 2], c[i >> 2]);
    asm("" : "+v"(v));  // keeps the sum and its conversion apart
    w[i] = _Float16(v);
  }
  return w;
}

constexpr int AK = 128;  // K a step

// What a row's step takes from memory and where it lies in the row's LDS record: up to three runs of n 16-byte granules
// (n a power of two; from byte g of the block, + h a half of the super-block; at byte l of the record), then 8 bytes and
// 2 bytes where the type has them. step: bytes from one step (super-block types: two) to the next. pitch: bytes a
// record; over 64 banks its multiples of 4 dwords keep the 16 rows x 4 words that a fragment reads apart.
struct Run {
  int n, g, h, l;
};
struct Rec {
  Run run[3], t8, t2;
  int step, pitch;
};
constexpr Rec rec_of(int t) {
  switch (t) {
    case LMOE_Q4_1: return {{{4, 0, 0, 0}, {1, 64, 0, 64}, {}}, {}, {}, 80, 80};
    case LMOE_Q8_0: return {{{8, 0, 0, 0}, {}, {}}, {1, 128, 0, 128}, {}, 136, 144};
    case LMOE_Q5_K: return {{{4, 48, 64, 48}, {2, 16, 0, 16}, {1, 0, 0, 0}}, {}, {}, 176, 112};
    default: return {{{4, 0, 64, 0}, {2, 128, 32, 64}, {}}, {1, 192, 8, 96}, {1, 208, 0, 104}, 210, 112};  // Q6_K
  }
}
constexpr bool super_block(int t) { return t == LMOE_Q5_K || t == LMOE_Q6_K; }

// The words a lane reads of its row's record (rec; g: its lane group) for one fragment and step, and its 8 weights of
// slice j. H: the half of the super-block.
template <int T, int H> struct Frag;

__device__ __forceinline__ uint32_t lds32(const uint8_t *p) { return *reinterpret_cast<const uint32_t *>(p); }
__device__ __forceinline__ uint32_t lds16(const uint8_t *p) { return *reinterpret_cast<const uint16_t *>(p); }

template <int H> struct Frag<LMOE_Q8_0, H> {  // four 34-byte blocks: those of even slices start at a word, odd ones 2 past
  const uint8_t *r;
  int g;
  __device__ __forceinline__ Frag(const uint8_t *rec, int g_) : r(rec), g(g_) {}
  __device__ __forceinline__ half8 weights(int j) const {  // q d, one f16 rounding of the exact product
    const uint8_t *b = r + 34 * j;
    uint32_t lo, hi;
    if (j & 1) {
      lo = lds32(b + 2 + 4 * g);
      hi = lds32(b + 18 + 4 * g);
    } else {
      lo = __builtin_amdgcn_alignbyte(lds32(b + 4 + 4 * g), lds32(b + 4 * g), 2);
      hi = __builtin_amdgcn_alignbyte(lds32(b + 20 + 4 * g), lds32(b + 16 + 4 * g), 2);
    }
    h2_t p[4];
    byte_pairs(lo ^ 0x80808080u, hi ^ 0x80808080u, p);
    const _Float16 d = __builtin_bit_cast(_Float16, uint16_t(lds16(b)));
    const h2_t bias = {_Float16(1152.0f), _Float16(1152.0f)}, s = {d, d};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = __builtin_bit_cast(uint32_t, (p[i] - bias) * s);
    return half8_of(o);
  }
};

template <int H> struct Frag<LMOE_Q4_1, H> {
  const uint8_t *r;
  int g;
  __device__ __forceinline__ Frag(const uint8_t *rec, int g_) : r(rec), g(g_) {}
  __device__ __forceinline__ half8 weights(int j) const {  // f16(q d + m)
    const uint32_t dm = lds32(r + 20 * j), q = lds32(r + 20 * j + 4 + 4 * g);
    const float s[2] = {half_lo(dm), half_lo(dm)}, c[2] = {half_hi(dm), half_hi(dm)};
    return fma_bytes(opaque(q & 0x0F0F0F0Fu), opaque((q >> 4) & 0x0F0F0F0Fu), s, c);
  }
};

template <int H> struct Frag<LMOE_Q5_K, H> {  // header 16, qh 32, the half's qs 64
  const uint8_t *r;
  int g;
  uint32_t hb[2];
  u32x4 hdr;
  __device__ __forceinline__ Frag(const uint8_t *rec, int g_) : r(rec + 48 + 4 * g_), g(g_) {
    hdr = *reinterpret_cast<const u32x4 *>(rec);
    hb[0] = lds32(rec + 16 + 4 * g_);
    hb[1] = lds32(rec + 32 + 4 * g_);
  }
  __device__ __forceinline__ half8 weights(int j) const {  // f16((d sc) q - dmin m), sub-block 4 H + j
    const int sb = 4 * H + j;
    uint32_t v[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      v[i] = ((lds32(r + 32 * (j >> 1) + 16 * i) >> (4 * (j & 1))) & 0x0F0F0F0Fu) |
             (((hb[i] >> sb) & 0x01010101u) << 4);
    float sc, mn;
    k4_scale_min(hdr[1], hdr[2], hdr[3], sb, &sc, &mn);
    const float d1 = half_lo(hdr[0]) * sc, m1 = -(half_hi(hdr[0]) * mn);
    const float s[2] = {d1, d1}, c[2] = {m1, m1};
    return fma_bytes(opaque(v[0]), opaque(v[1]), s, c);
  }
};

template <int H> struct Frag<LMOE_Q6_K, H> {  // the half's ql 64, qh 32, scales 8, then d
  const uint8_t *r;
  uint32_t hb[2], sc[2];
  float d;
  __device__ __forceinline__ Frag(const uint8_t *rec, int g) : r(rec + 4 * g) {
    hb[0] = lds32(r + 64);
    hb[1] = lds32(r + 80);
    sc[0] = lds32(rec + 96);
    sc[1] = lds32(rec + 100);
    d = half_lo(lds16(rec + 104));
  }
  __device__ __forceinline__ half8 weights(int j) const {  // f16((d sc) (q - 32)): weights 128 H + 32 j ..
    uint32_t v[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      v[i] = ((lds32(r + 32 * (j & 1) + 16 * i) >> (4 * (j >> 1))) & 0x0F0F0F0Fu) |
             (((hb[i] >> (2 * j)) & 0x03030303u) << 4);
    const uint32_t sw = sc[j >> 1] >> (16 * (j & 1));
    const float s[2] = {d * float(int(int8_t(uint8_t(sw)))), d * float(int(int8_t(uint8_t(sw >> 8))))};
    // (1024 + q) s - 1056 s: 1056 s (24 bits) and the result (24 bits) are exact in float32, so only f16 rounds
    const float c[2] = {-1056.0f * s[0], -1056.0f * s[1]};
    h2_t p[4];
    byte_pairs(v[0], v[1], p);
    return fma_pairs_exact(p, s, c);
  }
};

// Grid as the other grouped GEMMs' (n_ntile times the tile bound, times two with BM = 128: a 128-row tile is worked as
// two of 64 rows next to each other in the logical order, its second half left out where the group ends before it).
// Host guarantees: K % 128 == 0 (256 for super-block types), A and one expert's weights under 4 GiB.
template <int T, int MODE, int BM>
__global__ void __launch_bounds__(kThreads, 2)
k_grouped_any(const _Float16 *a_src, int topk, const uint32_t *order, const uint32_t *offsets, const uint32_t *tiles,
              const uint32_t *n_tiles, int n_ntile, const uint8_t *w0, const uint8_t *w1, int K, int n_rows,
              uint32_t row_bytes, void *out, int ldo, int odt) {
  constexpr int MT = 64, MB = MT / 16, HALF = MT * 128, STAGE = 2 * HALF, D = MT * 128 / 1024 / 4, SUB = BM / MT;
  constexpr Rec R = rec_of(T);
  constexpr int N0 = R.run[0].n, N1 = R.run[1].n, NG = N0 + N1 + R.run[2].n, NP = NG + R.t8.n + R.t2.n;
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * STAGE + 4 * 64 * R.pitch];
  Tile t;
  if (!tile_of<BM>(offsets, tiles, n_tiles, n_ntile * SUB, &t)) return;
  if (SUB == 2) {
    const int half = t.nt & 1;
    t.nt >>= 1;
    t.row0 += MT * half;
    t.rows = min(MT, t.rows - MT * half);
    if (t.rows <= 0) return;  // uniform across the workgroup
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, g = lane >> 4;
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(lds));

  // A: granule q = 64 (D w + i) + lane of a 64-wide half holds chunk (q % 8) ^ (r & 7) of tile row r = q / 8
  uint32_t a_off[D];
#pragma unroll
  for (int i = 0; i < D; ++i) {
    const int q = 64 * (D * wave + i) + lane, r = q >> 3, c = (q & 7) ^ (r & 7);
    const int p = t.row0 + (r < t.rows ? r : 0);
    const uint32_t row = MODE == MODE_GATE_UP ? order[p] / uint32_t(topk) : uint32_t(p);
    a_off[i] = row * uint32_t(K) * 2u + 16u * uint32_t(c);
  }
  const uint32_t a_live = a_live_mask<D>(wave, t.rows);
  const int nk = K / AK;
  auto issue_a = [&](int kk) __attribute__((always_inline)) {  // step kk's A into stage kk % 2
    const uint32_t st = lds0 + uint32_t(kk & 1) * STAGE;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < D; ++i)
        dma_a(a_src + size_t(kk) * AK + 64 * h, a_off[i],
              __builtin_amdgcn_readfirstlane(st + h * HALF + 1024u * uint32_t(D * wave + i)), (a_live >> i) & 1);
  };

  // The wavefront's 64 weight rows: row 16 nb + fr of its records is fragment nb's row fr (gate/up: 32 gate rows, then
  // the same 32 up rows). Granule q = 64 i + lane of a run of n is granule q % n of row q / n: a wavefront-uniform row
  // base and one offset a lane for the run (n > 1); with n = 1, and for the 8- and 2-byte pieces, row lane's pointer.
  uint8_t *rec = lds + 2 * STAGE + wave * 64 * R.pitch;
  const size_t ebytes = size_t(__builtin_amdgcn_readfirstlane(t.e)) * n_rows * row_bytes;
  const uint8_t *wbase[2];
  if (MODE == MODE_GATE_UP) {
    wbase[0] = w0 + ebytes + size_t(t.nt * (GN / 2) + 32 * wave) * row_bytes;
    wbase[1] = w1 + ebytes + size_t(t.nt * (GN / 2) + 32 * wave) * row_bytes;
  } else {
    wbase[0] = w0 + ebytes + size_t(t.nt * GN + 64 * wave) * row_bytes;
    wbase[1] = wbase[0] + size_t(32) * row_bytes;
  }
  const uint8_t *row_src = (lane < 32 ? wbase[0] : wbase[1]) + uint32_t(lane & 31) * row_bytes;
  uint32_t run_off[3];
  int run_dst[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    constexpr Rec RR = rec_of(T);
    const int n = RR.run[k].n > 0 ? RR.run[k].n : 1;
    run_off[k] = uint32_t(lane / n) * row_bytes + uint32_t(16 * (lane % n));
    run_dst[k] = (lane / n) * RR.pitch + RR.run[k].l + 16 * (lane % n);
  }
  struct Raw {
    u32x4 q[NG];
    u32x2 t8;
    uint32_t t2;
  };
  auto issue_w = [&](Raw &raw, auto hc, size_t at) __attribute__((always_inline)) {  // half H of the blocks `at` bytes into the rows
    constexpr int H = decltype(hc)::value;
    static_for<0, NG>([&](auto ic) {
      constexpr int j = decltype(ic)::value, k = j < N0 ? 0 : j < N0 + N1 ? 1 : 2, i = j - (k > 0 ? N0 : 0) - (k > 1 ? N1 : 0);
      constexpr int n = R.run[k].n, r0 = 64 / n * i, o = R.run[k].g + H * R.run[k].h;
      if constexpr (n == 1)
        raw.q[j] = *reinterpret_cast<const u32x4h *>(row_src + at + o);
      else
        raw.q[j] = *reinterpret_cast<const u32x4h *>(wbase[r0 / 32] + (at + o + uint32_t(r0 % 32) * row_bytes) + run_off[k]);
    });
    if constexpr (R.t8.n > 0) raw.t8 = *reinterpret_cast<const u32x2h *>(row_src + at + R.t8.g + H * R.t8.h);
    if constexpr (R.t2.n > 0) raw.t2 = *reinterpret_cast<const uint16_t *>(row_src + at + R.t2.g);
  };
  auto put_w = [&](const Raw &raw) __attribute__((always_inline)) {
    static_for<0, NG>([&](auto ic) {
      constexpr int j = decltype(ic)::value, k = j < N0 ? 0 : j < N0 + N1 ? 1 : 2, i = j - (k > 0 ? N0 : 0) - (k > 1 ? N1 : 0);
      *reinterpret_cast<u32x4 *>(rec + run_dst[k] + 64 / R.run[k].n * i * R.pitch) = raw.q[j];
    });
    if constexpr (R.t8.n > 0) *reinterpret_cast<u32x2 *>(rec + lane * R.pitch + R.t8.l) = raw.t8;
    if constexpr (R.t2.n > 0) *reinterpret_cast<uint32_t *>(rec + lane * R.pitch + R.t2.l) = raw.t2;
  };

  f32x4 acc[4][MB];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // Step kk: its A rows (issued a step ago) and its weights (two steps ago) are waited for, the weights go to the
  // wavefront's records, the barrier publishes the A stage and frees the other one, the next step's A and the weights of
  // the one after go out, and this step multiplies. The copy counter counts in issue order, and the newest NP loads are
  // the next step's weights.
  auto step = [&](int kk, Raw &raw, auto hc, auto mbc) __attribute__((always_inline)) {
    constexpr int H = decltype(hc)::value, MBN = decltype(mbc)::value;
    wait_vm<NP>();
    put_w(raw);
    barrier_lds();
    if (kk + 1 < nk) issue_a(kk + 1);
    // past the end the last steps' weights are asked for again: a branch here costs copies of every loaded register
    const int k2 = min(kk + 2, nk - 1);
    issue_w(raw, hc, size_t(super_block(T) ? k2 >> 1 : k2) * R.step);
    const uint8_t *st = lds + (kk & 1) * STAGE;
    const uint8_t *my = rec + fr * R.pitch;
    const Frag<T, H> w[4] = {{my, g}, {my + 16 * R.pitch, g}, {my + 32 * R.pitch, g}, {my + 48 * R.pitch, g}};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32x4 *as = reinterpret_cast<const u32x4 *>(st + (j >> 1) * HALF);
      half8 xf[MBN];
#pragma unroll
      for (int mb = 0; mb < MBN; ++mb)
        xf[mb] = __builtin_bit_cast(half8, as[achunk(16 * mb + fr, 4 * (j & 1) + g)]);
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        const half8 wf = w[nb].weights(j);
#pragma unroll
        for (int mb = 0; mb < MBN; ++mb)
          acc[nb][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf, xf[mb], acc[nb][mb], 0, 0, 0);
      }
    }
  };
  Raw ra, rb;
  constexpr int H1 = super_block(T) ? 1 : 0;
  issue_w(ra, IC<0>{}, 0);
  issue_a(0);
  issue_w(rb, IC<H1>{}, size_t(super_block(T) ? 0 : min(1, nk - 1)) * R.step);
  auto run = [&](auto mbc) {
    int kk = 0;
    for (; kk + 1 < nk; kk += 2) {  // two steps a turn, one buffer of weights each
      step(kk, ra, IC<0>{}, mbc);
      step(kk + 1, rb, IC<H1>{}, mbc);
    }
    if (!super_block(T) && kk < nk) step(kk, ra, IC<0>{}, mbc);
  };
  switch ((t.rows + 15) / 16) {  // uniform across the workgroup
    case 1: run(IC<1>{}); break;
    case 2: run(IC<2>{}); break;
    case 3: run(IC<3>{}); break;
    default: run(IC<4>{}); break;
  }
  store_tile<MODE, MB>(acc, t, wave, fr, g, out, ldo, odt, order);
}

// Shape checks and the launch that lmoe_grouped_gate_up_any, lmoe_grouped_down_any and lmoe_grouped_down_rows share. mode
// gate/up: n_rows = I; down: n_rows = H.
int grouped_any(const char *fn, int mode, const void *a, long long a_rows, int topk, const uint32_t *order,
                const uint32_t *offsets, const uint32_t *tiles, const uint32_t *n_tiles, int max_tiles, int bm,
                const uint8_t *w0, const uint8_t *w1, int type, int n_experts, int K, int n_rows, void *out, int odt,
                hipStream_t st) {
  LMOE_REQUIRE(type == LMOE_Q4_1 || type == LMOE_Q8_0 || type == LMOE_Q5_K || type == LMOE_Q6_K, LMOE_ETYPE,
               "%s: ggml type %d is not supported (Q4_1 = 3, Q8_0 = 8, Q5_K = 13, Q6_K = 14)", fn, type);
  LMOE_REQUIRE(bm == GM || bm == 64, LMOE_ESHAPE, "%s: tile rows %d (128 or 64)", fn, bm);
  LMOE_REQUIRE(topk > 0 && n_experts > 0 && max_tiles >= 0, LMOE_ESHAPE, "%s: bad shape", fn);
  const int kmul = super_block(type) ? 256 : AK, nt = mode == MODE_GATE_UP ? GN / 2 : GN;
  LMOE_REQUIRE(K > 0 && K % kmul == 0, LMOE_ESHAPE, "%s: row length %d is not a multiple of %d", fn, K, kmul);
  LMOE_REQUIRE(n_rows > 0 && n_rows % nt == 0, LMOE_ESHAPE, "%s: %d rows are not a multiple of %d", fn, n_rows, nt);
  if (a_rows == 0 || max_tiles == 0) return 0;
  LMOE_REQUIRE(a && offsets && tiles && n_tiles && w0 && out && (mode == MODE_DOWN || (order && w1)), LMOE_EINVAL,
               "%s: null pointer", fn);
  LMOE_REQUIRE(aligned16(a) && aligned16(out), LMOE_EALIGN, "%s: activations and output must be 16-byte aligned", fn);
  const uintptr_t wal = type == LMOE_Q5_K ? 16 : type == LMOE_Q4_1 ? 4 : 2;  // as lmoe_dequant_gemm_f16 takes them
  LMOE_REQUIRE((reinterpret_cast<uintptr_t>(w0) | reinterpret_cast<uintptr_t>(w1)) % wal == 0, LMOE_EALIGN,
               "%s: ggml type %d weights must be %d-byte aligned", fn, type, int(wal));
  const long long row_bytes = (long long)(K / (super_block(type) ? 256 : AK)) * rec_of(type).step;
  LMOE_REQUIRE(a_rows * K * 2 <= 0xFFFFFFFFll && n_rows * row_bytes <= 0xFFFFFFFFll, LMOE_ESHAPE,
               "%s: the activations or one expert's weights exceed 4 GiB", fn);
  const int n_ntile = n_rows / nt;
  const long long grid = (long long)n_ntile * max_tiles * (bm / 64);
  LMOE_REQUIRE(grid < (1ll << 31), LMOE_ESHAPE, "%s: %lld workgroups", fn, grid);
  const int ldo = n_rows;
  auto go = [&](auto kern) {
    launch(kern, dim3(unsigned(grid)), dim3(kThreads), 0, st, static_cast<const _Float16 *>(a), topk, order, offsets,
           tiles, n_tiles, n_ntile, w0, w1, K, n_rows, uint32_t(row_bytes), out, ldo, odt);
  };
  auto pick = [&](auto tc) {
    constexpr int T = decltype(tc)::value;
    if (mode == MODE_GATE_UP)
      bm == 64 ? go(k_grouped_any<T, MODE_GATE_UP, 64>) : go(k_grouped_any<T, MODE_GATE_UP, 128>);
    else
      bm == 64 ? go(k_grouped_any<T, MODE_DOWN, 64>) : go(k_grouped_any<T, MODE_DOWN, 128>);
  };
  switch (type) {
    case LMOE_Q4_1: pick(IC<LMOE_Q4_1>{}); break;
    case LMOE_Q8_0: pick(IC<LMOE_Q8_0>{}); break;
    case LMOE_Q5_K: pick(IC<LMOE_Q5_K>{}); break;
    default: pick(IC<LMOE_Q6_K>{}); break;
  }
  LMOE_LAUNCHED(fn);
  return 0;
}

}  // namespace lmoe

using namespace lmoe;

extern "C" int lmoe_grouped_gate_up_any(const void *x, int xdtype, int T, int topk, const uint32_t *order,
                                        const uint32_t *offsets, const uint32_t *tiles, const uint32_t *n_tiles,
                                        int max_tiles, int bm, const uint8_t *wg, const uint8_t *wu, int type,
                                        int n_experts, int H, int I, void *h, void *stream) {
  const char *fn = "lmoe_grouped_gate_up_any";
  LMOE_REQUIRE(xdtype == LMOE_F16, LMOE_EINVAL,
               "%s: x must be float16 in the GEMM K order here (convert once with lmoe_to_gemm_f16)", fn);
  LMOE_REQUIRE(T >= 0, LMOE_ESHAPE, "%s: bad shape", fn);
  return grouped_any(fn, MODE_GATE_UP, x, T, topk, order, offsets, tiles, n_tiles, max_tiles, bm, wg, wu, type,
                     n_experts, H, I, h, LMOE_F16, (hipStream_t)stream);
}

extern "C" int lmoe_grouped_down_any(const void *h, int R, const uint32_t *offsets, const uint32_t *tiles,
                                     const uint32_t *n_tiles, int max_tiles, int bm, const uint8_t *wd, int type,
                                     int n_experts, int I, int H, void *y, int ydtype, void *stream) {
  const char *fn = "lmoe_grouped_down_any";
  LMOE_REQUIRE(ydtype == LMOE_F16 || ydtype == LMOE_F32, LMOE_EINVAL, "%s: y must be float16 or float32", fn);
  LMOE_REQUIRE(R >= 0, LMOE_ESHAPE, "%s: bad shape", fn);
  return grouped_any(fn, MODE_DOWN, h, R, 1, nullptr, offsets, tiles, n_tiles, max_tiles, bm, wd, nullptr, type,
                     n_experts, I, H, y, ydtype, (hipStream_t)stream);
}
