// The trunk's 4-bit affine matmul of T bf16 rows: the reference's route_cuda.qmv_rows (route_cuda.py:460-541),
// which gives every row the bits of MLX 0.32.4's one-row qmv kernel while reading the weights once for all rows.
//
// Weights in MLX's affine 4-bit layout: w uint32 [N][K / 8] (element j of a word at bits 4j), scales and biases
// bf16 [N][K / G]; weight = q s + b. The arithmetic, kept step for step so the output bits match:
//   * a row is worked by 32 lanes; lane l takes elements idx = base + 16 l .. idx + 15, base = 0, 512, ...;
//   * its 16 weights in bf16: bf16(bf16(q s) + b);
//   * 16 bf16 accumulators a row of x, slot e = element idx + e, each step one bf16 fused multiply-add;
//   * the 16 slots summed in float32 in slot order, the xor butterfly 16, 8, 4, 2, 1 in float32, bf16 out.
// On gfx950 a 64-lane wavefront works two output rows, one a 32-lane half, so each half is exactly the reference's
// warp and the butterfly stays inside the half (shuffles of width 32).
//
// bf16 arithmetic runs in float32 with gfx950's v_cvt_pk_bf16_f32 (round to nearest even) for each rounding; with 0 as its
// low operand the result is the rounded value as a float32 already, no unpacking. Products of two bf16 values are exact
// in float32; the sum of two bf16 values is exact unless their exponents are more than 16 apart, where the small one
// cannot reach a bf16 rounding boundary. gfx950 has no bf16 fused multiply-add: see fma_bf16_odd.
//
// VALU-bound (one product is 11-12 instructions, 5 of them the fused multiply-add's, against 0.56 bytes of weights).
// Measured on one box, us, with the exact error of a nearest-rounded float32 sum recovered (TwoSum) and moved off the
// bf16 midpoints (15 instructions) -> rounded to odd: 2048 -> 248,320 1 row 263 -> 157, 2048 -> 8192 1 row 12.2 -> 7.9,
// 5 rows 37.6 -> 19.1, 2048 -> 512 5 rows 15.1 -> 8.7. Eight elements a mode change instead of sixteen: 566 against 495
// at 248,320 x 5 rows, 173 against 166 at 1.
#include <type_traits>

#include "lmoe_common.h"

namespace lmoe {

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// v rounded to bf16 (nearest even), as float32
__device__ __forceinline__ float bf16r(float v) {
  return __uint_as_float(__builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{0.0f, v}, bf16x2_t)));
}

// a[i] <- x[i] w[i] + a[i] rounded to odd in float32 (the float32 neighbour of the exact value whose last bit is set,
// unless the value is a float32 itself): a value whose rounding to bf16 is the one rounding of the exact value, since
// only a value that is exactly halfway between two bf16 values ends in 0x8000. The exact value lies between the fused
// multiply-add rounded down (MODE's round field = 2) and rounded up (1), which are equal or neighbours; the odd one is
// picked bit by bit. One asm block, so that no other rounding instruction can come between the mode changes (a is written
// before the last x and w are read, so no input may share its registers); the
// smallest exact zero keeps the sign that rounding to nearest gives it (rounded up's +0, unless both are -0).
__device__ __forceinline__ void fma_bf16_odd(float (&a)[16], const float *x, const float *w) {
  float t[16];
  asm("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 2\n\t"
      "v_fma_f32 %16, %32, %48, %0\n\t"
      "v_fma_f32 %17, %33, %49, %1\n\t"
      "v_fma_f32 %18, %34, %50, %2\n\t"
      "v_fma_f32 %19, %35, %51, %3\n\t"
      "v_fma_f32 %20, %36, %52, %4\n\t"
      "v_fma_f32 %21, %37, %53, %5\n\t"
      "v_fma_f32 %22, %38, %54, %6\n\t"
      "v_fma_f32 %23, %39, %55, %7\n\t"
      "v_fma_f32 %24, %40, %56, %8\n\t"
      "v_fma_f32 %25, %41, %57, %9\n\t"
      "v_fma_f32 %26, %42, %58, %10\n\t"
      "v_fma_f32 %27, %43, %59, %11\n\t"
      "v_fma_f32 %28, %44, %60, %12\n\t"
      "v_fma_f32 %29, %45, %61, %13\n\t"
      "v_fma_f32 %30, %46, %62, %14\n\t"
      "v_fma_f32 %31, %47, %63, %15\n\t"
      "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 1\n\t"
      "v_fma_f32 %0, %32, %48, %0\n\t"
      "v_fma_f32 %1, %33, %49, %1\n\t"
      "v_fma_f32 %2, %34, %50, %2\n\t"
      "v_fma_f32 %3, %35, %51, %3\n\t"
      "v_fma_f32 %4, %36, %52, %4\n\t"
      "v_fma_f32 %5, %37, %53, %5\n\t"
      "v_fma_f32 %6, %38, %54, %6\n\t"
      "v_fma_f32 %7, %39, %55, %7\n\t"
      "v_fma_f32 %8, %40, %56, %8\n\t"
      "v_fma_f32 %9, %41, %57, %9\n\t"
      "v_fma_f32 %10, %42, %58, %10\n\t"
      "v_fma_f32 %11, %43, %59, %11\n\t"
      "v_fma_f32 %12, %44, %60, %12\n\t"
      "v_fma_f32 %13, %45, %61, %13\n\t"
      "v_fma_f32 %14, %46, %62, %14\n\t"
      "v_fma_f32 %15, %47, %63, %15\n\t"
      "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0"
      : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5]), "+&v"(a[6]), "+&v"(a[7]),
        "+&v"(a[8]), "+&v"(a[9]), "+&v"(a[10]), "+&v"(a[11]), "+&v"(a[12]), "+&v"(a[13]), "+&v"(a[14]), "+&v"(a[15]),
        "=&v"(t[0]), "=&v"(t[1]), "=&v"(t[2]), "=&v"(t[3]), "=&v"(t[4]), "=&v"(t[5]), "=&v"(t[6]), "=&v"(t[7]),
        "=&v"(t[8]), "=&v"(t[9]), "=&v"(t[10]), "=&v"(t[11]), "=&v"(t[12]), "=&v"(t[13]), "=&v"(t[14]),
        "=&v"(t[15])
      : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]), "v"(x[6]), "v"(x[7]), "v"(x[8]),
        "v"(x[9]), "v"(x[10]), "v"(x[11]), "v"(x[12]), "v"(x[13]), "v"(x[14]), "v"(x[15]), "v"(w[0]), "v"(w[1]),
        "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]), "v"(w[10]),
        "v"(w[11]), "v"(w[12]), "v"(w[13]), "v"(w[14]), "v"(w[15]));
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int odd = __builtin_amdgcn_sbfe(__float_as_int(t[i]), 0, 1);  // all ones where rounded down is odd
    asm("v_bfi_b32 %0, %1, %2, %0" : "+v"(a[i]) : "v"(odd), "v"(t[i]));
  }
}

// sum[r] = row r of x [NR][K] bf16 times one weight row (wr, sr, br), by the 32 lanes l of a half-wavefront, in every lane.
// K % 16 == 0, G % 16 == 0, K % G == 0.
template <int NR>
__device__ __forceinline__ void qmv_dot(const uint16_t *x, const uint32_t *wr, const uint16_t *sr, const uint16_t *br, int K,
                                        int G, int l, float (&sum)[NR]) {
  float acc[NR][16];
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[r][e] = 0.0f;
  // the lane's group: one division, then whole groups a 512-element step where G divides 512 (a division a step is 15 of
  // a step's ~205 vector instructions)
  const int gstep = 512 % G == 0 ? 512 / G : 0;
  int grp = 16 * l / G;
  for (int idx = 16 * l; idx < K; idx += 512, grp = gstep ? grp + gstep : idx / G) {
    const u32x2_t wv = *reinterpret_cast<const u32x2_t *>(wr + (idx >> 3));
    const float s = bf16_to_f32(sr[grp]), b = bf16_to_f32(br[grp]);
    float wd[16];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t lo = opaque(wv[h] & 0x0F0F0F0Fu), hi = opaque((wv[h] >> 4) & 0x0F0F0F0Fu);
#pragma unroll
      for (int p = 0; p < 8; ++p) {
        const float m = bf16r(float(((p & 1 ? hi : lo) >> (8 * (p >> 1))) & 0xffu) * s);  // the product is exact
        wd[8 * h + p] = bf16r(m + b);  // exact, or too far from a rounding boundary to matter
      }
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const u32x4 *xp = reinterpret_cast<const u32x4 *>(x + size_t(r) * K + idx);
      float xf[16];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4 xs = xp[h];
#pragma unroll
        for (int p = 0; p < 8; ++p) xf[8 * h + p] = __uint_as_float(p & 1 ? xs[p >> 1] & 0xffff0000u : xs[p >> 1] << 16);
      }
      fma_bf16_odd(acc[r], xf, wd);
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[r][e] = bf16r(acc[r][e]);
    }
  }
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    float s = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) s += acc[r][e];
#pragma unroll
    for (int m = 16; m > 0; m >>= 1) s += __shfl_xor(s, m, 32);
    sum[r] = s;
  }
}

// Grid ceil(N / 8), 256 threads: wavefront w's lanes 0-31 work output row 8 bx + 2 w, lanes 32-63 the next one.
// x [NR][K] bf16, out [NR][N] bf16.
template <int NR>
__global__ void __launch_bounds__(256) k_qmv_rows(const uint16_t *x, const uint32_t *w, const uint16_t *scales,
                                                  const uint16_t *biases, int N, int K, int G, uint16_t *out) {
  const int lane = threadIdx.x & 63, l = lane & 31;
  const int row = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 2 + (lane >> 5);
  const int rr = row < N ? row : N - 1;  // a half past N works the last row again and stores nothing
  float s[NR];
  qmv_dot<NR>(x, w + size_t(rr) * (K / 8), scales + size_t(rr) * (K / G), biases + size_t(rr) * (K / G), K, G, l, s);
  if (l == 0 && row < N) {
#pragma unroll
    for (int r = 0; r < NR; ++r) out[size_t(r) * N + row] = f32_to_bf16(s[r]);
  }
}

// out [NR][N] bf16 = bf16(silu(g) u), g and u the bf16 products of two weights of one shape: grid ceil(N / 4), wavefront w's
// lanes 0-31 work row 4 bx + w of the first weight, lanes 32-63 that row of the second (k_qmv_rows twice and
// k_swiglu_bf16 in one launch, the same bits: at one token each of the three is a launch's latency).
template <int NR>
__global__ void __launch_bounds__(256) k_qmv_swiglu(const uint16_t *x, const uint32_t *wg, const uint16_t *sg,
                                                    const uint16_t *bg, const uint32_t *wu, const uint16_t *su,
                                                    const uint16_t *bu, int N, int K, int G, uint16_t *out) {
  const int lane = threadIdx.x & 63, l = lane & 31;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= N) return;  // uniform across the wavefront
  const bool up = lane >= 32;
  const size_t gi = size_t(row) * (K / G);
  float s[NR];
  qmv_dot<NR>(x, (up ? wu : wg) + size_t(row) * (K / 8), (up ? su : sg) + gi, (up ? bu : bg) + gi, K, G, l, s);
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const float u = __shfl(s[r], 32);
    if (lane == 0) out[size_t(r) * N + row] = f32_to_bf16(silu_mul(bf16r(s[r]), bf16r(u)));
  }
}

// out = bf16(silu(g) u) for bf16 g, u: one rounding of the float32 value (the shared expert's SwiGLU between its
// qmv_rows projections).
__global__ void __launch_bounds__(256) k_swiglu_bf16(const uint16_t *g, const uint16_t *u, long long n,
                                                     uint16_t *out) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  out[i] = f32_to_bf16(silu_mul(bf16_to_f32(g[i]), bf16_to_f32(u[i])));
}

}  // namespace lmoe

using namespace lmoe;

extern "C" int lmoe_swiglu_bf16(const void *g, const void *u, long long n, void *out, void *stream) {
  const char *fn = "lmoe_swiglu_bf16";
  LMOE_REQUIRE(n >= 0, LMOE_ESHAPE, "%s: bad size", fn);
  if (n == 0) return 0;
  LMOE_REQUIRE(g && u && out, LMOE_EINVAL, "%s: null pointer", fn);
  launch(k_swiglu_bf16, dim3(unsigned((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
         static_cast<const uint16_t *>(g), static_cast<const uint16_t *>(u), n, static_cast<uint16_t *>(out));
  LMOE_LAUNCHED(fn);
  return 0;
}

// The checks and the passes over x both products share: at most 8 rows a launch (their accumulators stay in registers);
// rows 8.. in a second pass over the weights, which changes no bit (each row's arithmetic is its own). go(NR, first row).
template <typename F>
static int qmv_passes(const char *fn, const void *x, int T, const void *w, int N, int K, int group_size, F &&go) {
  LMOE_REQUIRE(T >= 0, LMOE_ESHAPE, "%s: %d rows", fn, T);
  LMOE_REQUIRE(N > 0 && K > 0 && K % 16 == 0 && group_size > 0 && group_size % 16 == 0 && K % group_size == 0,
               LMOE_ESHAPE, "%s: K %d and group size %d must be multiples of 16, K of the group size", fn, K,
               group_size);
  if (T == 0) return 0;
  LMOE_REQUIRE(x && w, LMOE_EINVAL, "%s: null pointer", fn);
  LMOE_REQUIRE(aligned16(x) && (reinterpret_cast<uintptr_t>(w) & 7u) == 0, LMOE_EALIGN,
               "%s: x must be 16-byte aligned, w 8-byte aligned", fn);
  for (int r0 = 0; r0 < T; r0 += 8) {
    switch (T - r0 < 8 ? T - r0 : 8) {
      case 1: go(std::integral_constant<int, 1>{}, r0); break;
      case 2: go(std::integral_constant<int, 2>{}, r0); break;
      case 3: go(std::integral_constant<int, 3>{}, r0); break;
      case 4: go(std::integral_constant<int, 4>{}, r0); break;
      case 5: go(std::integral_constant<int, 5>{}, r0); break;
      case 6: go(std::integral_constant<int, 6>{}, r0); break;
      case 7: go(std::integral_constant<int, 7>{}, r0); break;
      default: go(std::integral_constant<int, 8>{}, r0); break;
    }
    LMOE_LAUNCHED(fn);
  }
  return 0;
}

extern "C" int lmoe_qmv_rows(const void *x, int T, const uint32_t *w, const void *scales, const void *biases, int N,
                             int K, int group_size, void *out, void *stream) {
  const char *fn = "lmoe_qmv_rows";
  LMOE_REQUIRE(T <= 0 || (scales && biases && out), LMOE_EINVAL, "%s: null pointer", fn);
  return qmv_passes(fn, x, T, w, N, K, group_size, [&](auto nr, int r0) {
    launch(k_qmv_rows<decltype(nr)::value>, dim3(unsigned((N + 7) / 8)), dim3(256), 0, (hipStream_t)stream,
           static_cast<const uint16_t *>(x) + size_t(r0) * K, w, static_cast<const uint16_t *>(scales),
           static_cast<const uint16_t *>(biases), N, K, group_size, static_cast<uint16_t *>(out) + size_t(r0) * N);
  });
}

extern "C" int lmoe_qmv_swiglu_rows(const void *x, int T, const uint32_t *wg, const void *scales_g, const void *biases_g,
                                    const uint32_t *wu, const void *scales_u, const void *biases_u, int N, int K,
                                    int group_size, void *out, void *stream) {
  const char *fn = "lmoe_qmv_swiglu_rows";
  LMOE_REQUIRE(T <= 0 || (scales_g && biases_g && wu && scales_u && biases_u && out), LMOE_EINVAL, "%s: null pointer", fn);
  LMOE_REQUIRE(T <= 0 || (reinterpret_cast<uintptr_t>(wu) & 7u) == 0, LMOE_EALIGN, "%s: w must be 8-byte aligned", fn);
  return qmv_passes(fn, x, T, wg, N, K, group_size, [&](auto nr, int r0) {
    launch(k_qmv_swiglu<decltype(nr)::value>, dim3(unsigned((N + 3) / 4)), dim3(256), 0, (hipStream_t)stream,
           static_cast<const uint16_t *>(x) + size_t(r0) * K, wg, static_cast<const uint16_t *>(scales_g),
           static_cast<const uint16_t *>(biases_g), wu, static_cast<const uint16_t *>(scales_u),
           static_cast<const uint16_t *>(biases_u), N, K, group_size, static_cast<uint16_t *>(out) + size_t(r0) * N);
  });
}
