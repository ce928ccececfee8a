// Complex GEMM on the gfx950 matrix cores for fp16, bf16, fp32 and fp8
// (e4m3/e5m2) input with fp32 accumulation, and for 1-bit input (+-1 values on
// the fp4 instruction, exact integer sums; kernels/gemm_kernel_int1.cu:64-356).
//
// Stands in for the reference's wmma_complex_gemm_basic / wmma_complex_gemm_opt
// (kernels/gemm_kernel_float.cu:35-181, :186-355) and its epilogue helpers
// (kernels/matrix_operations.h:38-178). The math is the same four real
// products per complex product (gemm_kernel_float.cu:293-303); everything
// else is laid out for 64-wide wavefronts:
//
//  * One persistent block owns a sequence of BX x BY patches of C and walks K in
//    tiles of 64 bytes per row. Tiles go global -> LDS directly
//    (global_load_lds_dwordx4) through a ring of LDS slots, two iterations ahead
//    of the math: for the tiled (opt) layout, for planar (basic) rows and for the
//    pipeline's interleaved rows, of any length from 16 bytes on and at any address.
//    Only shorter planar rows, and 1-bit ones that are not whole aligned 16-byte
//    chunks (both without a tiled copy), are staged through registers by kernels
//    whose element-wise loads do their bounds checks and zero fill.
//  * LDS rows are 64 bytes with the 16-byte chunk index XORed by a function of
//    the row that suits the fragment shape of the MFMA in use (measured free of
//    bank conflicts; see complex_gemm_mfma_dtl).
//  * 16-bit input: 16x16x32 MFMA; 32-bit input: every value split into three
//    bf16 for the 32x32x16 one (fp32 products to fp32 accuracy); fp8: the
//    32x32x64 f8f6f4 MFMA, which runs at twice the rate of the legacy fp8
//    instruction; 1-bit input: the same instruction on fp4 +-1 values expanded
//    from the packed words in registers.
//  * The four products of a complex MAC reuse the same fragments; the minus
//    sign of Re -= Xi*Yi is a sign-bit flip of the Yi fragment registers.
//  * Workgroup ids are remapped so that consecutive tiles land on the same
//    XCD (shared L2), in groups that reuse both operands.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>
#include <utility>

#include "gemm_device.h"

namespace ccglib_amd {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef int int8_t_ __attribute__((ext_vector_type(8)));
typedef unsigned short ushort4_t __attribute__((ext_vector_type(4)));

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>), in this order.
template <int... Is, class F>
__device__ __forceinline__ void static_for_each(std::integer_sequence<int, Is...>, F &&f) {
  (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_each(std::make_integer_sequence<int, N>{}, f);
}

// K tiles consumed by one MFMA: one for 16-bit input (16x16x32), two for fp8
// (16x16x128: 32 bytes per lane, 16 from each of two K tiles).
template <int DT> struct DtypeTraits {
  static constexpr int kTilesPerMfma = (DT == kFloat8e4m3 || DT == kFloat8e5m2) ? 2 : 1;
  static constexpr int kElemBytes = (DT == kFloat8e4m3 || DT == kFloat8e5m2) ? 1
                                    : (DT == kFloat32)                       ? 4
                                                                             : 2;
  static constexpr unsigned kSignMask = (DT == kFloat8e4m3 || DT == kFloat8e5m2) ? 0x80808080u
                                        : (DT == kFloat32)                         ? 0x80000000u
                                                                                   : 0x80008000u;
};

template <int DT> struct Fragment {
  int4_t v[DtypeTraits<DT>::kTilesPerMfma];
};

template <int DT>
__device__ __forceinline__ float4_t mfma(const Fragment<DT> &a, const Fragment<DT> &b,
                                         float4_t acc) {
  if constexpr (DT == kFloat16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(
        __builtin_bit_cast(half8_t, a.v[0]), __builtin_bit_cast(half8_t, b.v[0]), acc, 0, 0, 0);
  } else if constexpr (DT == kBfloat16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
        __builtin_bit_cast(bf16x8_t, a.v[0]), __builtin_bit_cast(bf16x8_t, b.v[0]), acc, 0, 0, 0);
  } else if constexpr (DT == kFloat32) {
    // fp32 input (true fp32 products, no tf32 on this part): a lane's 16-byte
    // chunk is four K values; 16x16x4 takes one value per lane, and which K a
    // lane supplies does not matter as long as both operands agree.
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      // (copies first: a bit cast applied to a vector element expression
      // directly reads element 0 whatever the index)
      const int ae = a.v[0][e], be = b.v[0][e];
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, ae),
                                                 __builtin_bit_cast(float, be), acc, 0, 0, 0);
    }
    return acc;
  } else {
    int8_t_ av, bv;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      av[i] = a.v[0][i];
      av[4 + i] = a.v[1][i];
      bv[i] = b.v[0][i];
      bv[4 + i] = b.v[1][i];
    }
    // format code 0 = e4m3, 1 = e5m2; scale exponent 127 = 2^0
    constexpr int fmt = (DT == kFloat8e4m3) ? 0 : 1;
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, acc, fmt, fmt, 0, 0x7f, 0,
                                                            0x7f);
  }
}

template <int DT>
__device__ __forceinline__ Fragment<DT> negate(const Fragment<DT> &f) {
  Fragment<DT> r;
#pragma unroll
  for (int t = 0; t < DtypeTraits<DT>::kTilesPerMfma; ++t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      r.v[t][i] = f.v[t][i] ^ (int)DtypeTraits<DT>::kSignMask;
    }
  }
  return r;
}

// The 32-row MFMAs. A lane holds 32 bytes of one row of the K tile (two
// 16-byte chunks) and 16 accumulators per 32x32 tile. fp8 (32x32x64) eats the
// whole 64-byte row in one instruction, 16-bit input (32x32x16) takes one
// chunk per instruction. One wave alone keeps the MFMA pipe full with these,
// which the 16-row shapes do not on this part (measured 58 % for 16x16x32),
// so the second wave of a SIMD covers the other's LDS and barrier waits.
typedef float float16_t_ __attribute__((ext_vector_type(16)));
struct Fragment32 {
  int4_t v[2];
};

template <int DT>
__device__ __forceinline__ float16_t_ mfma32(const Fragment32 &a, const Fragment32 &b,
                                             float16_t_ acc) {
  if constexpr (DT == kFloat16) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a.v[u]),
                                                   __builtin_bit_cast(half8_t, b.v[u]), acc, 0, 0, 0);
    }
    return acc;
  } else if constexpr (DT == kBfloat16) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a.v[u]),
                                                    __builtin_bit_cast(bf16x8_t, b.v[u]), acc, 0, 0, 0);
    }
    return acc;
  } else {
    int8_t_ av, bv;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      av[i] = a.v[0][i];
      av[4 + i] = a.v[1][i];
      bv[i] = b.v[0][i];
      bv[4 + i] = b.v[1][i];
    }
    constexpr int fmt = (DT == kFloat8e4m3) ? 0 : 1;
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, acc, fmt, fmt, 0, 0x7f, 0,
                                                           0x7f);
  }
}

// Accumulator of one MFMA tile and how the output is spread over a wave, for
// both MFMA shapes (MS = 16 or 32 rows) and for the 16-row shape with the
// operand roles exchanged (kAcc16T: X is the MFMA "B" operand and tile i of a
// wave holds the columns x = 4 (lane % 16) + i, see complex_gemm_mfma_dtl).
// A lane holds "pieces" of four consecutive x (the contiguous C axis) at one y:
//   MS 16:   piece (jj, ii) at x = 16 ii + 4 (lane / 16), y = 16 jj + lane % 16
//   MS 32:   piece (jj, ii) at x = 32 (ii / 4) + 8 (ii % 4) + 4 (lane / 32), y = 32 jj + lane % 32
//   kAcc16T: piece (jj, ii) at x = 4 (lane % 16), y = 16 jj + 4 (lane / 16) + ii; its four
//            elements are register ii of the four tiles of tile row jj
constexpr int kAcc16T = 116;
template <int MS> struct AccType { using type = float4_t; };
template <> struct AccType<32> { using type = float16_t_; };

template <int MS> __device__ __forceinline__ unsigned piece_x(int ii, int lane) {
  if constexpr (MS == kAcc16T) return (lane & 15) * 4;
  return MS == 16 ? ii * 16 + (lane >> 4) * 4 : (ii >> 2) * 32 + (ii & 3) * 8 + (lane >> 5) * 4;
}
template <int MS> __device__ __forceinline__ unsigned piece_y(int jj, int ii, int lane) {
  if constexpr (MS == kAcc16T) return jj * 16 + (lane >> 4) * 4 + ii;
  return MS == 16 ? jj * 16 + (lane & 15) : jj * 32 + (lane & 31);
}
// (TILE0: kAcc16T only, the first of the four tiles when a wave's tile rows hold more)
template <int MS, int TILE0 = 0, typename Acc>
__device__ __forceinline__ float piece_elem(const Acc &acc, int jj, int ii, int e) {
  if constexpr (MS == kAcc16T) {
    return acc[jj][TILE0 + e][ii];
  } else if constexpr (MS == 16) {
    return acc[jj][ii][e];
  } else {
    return acc[jj][ii >> 2][(ii & 3) * 4 + e];
  }
}

template <int TOUT> struct OutType;
template <> struct OutType<kFloat32> { using type = float; };
template <> struct OutType<kFloat16> { using type = _Float16; };
template <> struct OutType<kBfloat16> { using type = __bf16; };
template <> struct OutType<kInt32> { using type = int; };

// One K tile (or two for fp8) of math for a wave: reads its X and Y fragments
// from the LDS slot(s) and issues the four real products of the complex MAC.
// slot[u] points at the K tile u of this MFMA step: [X re][X im][Y re][Y im].
template <int DT, int BX, int BY, int TX, int TY, typename Mid>
__device__ __forceinline__ void mma_step(const char *const (&slot)[DtypeTraits<DT>::kTilesPerMfma],
                                         int x_frag_off, int y_frag_off,
                                         float4_t (&acc_re)[TY][TX], float4_t (&acc_im)[TY][TX],
                                         Mid &&mid) {
  constexpr int KPM = DtypeTraits<DT>::kTilesPerMfma;
  Fragment<DT> xr[TX], xi[TX];
#pragma unroll
  for (int i = 0; i < TX; ++i) {
#pragma unroll
    for (int u = 0; u < KPM; ++u) {
      const char *p = slot[u] + x_frag_off + i * 16 * kTileRowBytes;
      xr[i].v[u] = *reinterpret_cast<const int4_t *>(p);
      xi[i].v[u] = *reinterpret_cast<const int4_t *>(p + BX * kTileRowBytes);
    }
  }
#pragma unroll
  for (int j = 0; j < TY; ++j) {
    Fragment<DT> yr, yi;
#pragma unroll
    for (int u = 0; u < KPM; ++u) {
      const char *p = slot[u] + y_frag_off + j * 16 * kTileRowBytes;
      yr.v[u] = *reinterpret_cast<const int4_t *>(p);
      yi.v[u] = *reinterpret_cast<const int4_t *>(p + BY * kTileRowBytes);
    }
    const Fragment<DT> yin = negate<DT>(yi);
#pragma unroll
    for (int i = 0; i < TX; ++i) acc_re[j][i] = mfma<DT>(xr[i], yr, acc_re[j][i]);
#pragma unroll
    for (int i = 0; i < TX; ++i) acc_im[j][i] = mfma<DT>(xr[i], yi, acc_im[j][i]);
#pragma unroll
    for (int i = 0; i < TX; ++i) acc_re[j][i] = mfma<DT>(xi[i], yin, acc_re[j][i]);
#pragma unroll
    for (int i = 0; i < TX; ++i) acc_im[j][i] = mfma<DT>(xi[i], yr, acc_im[j][i]);
    if (j == 0) mid();
  }
}

// The same step with every LDS read placed by hand, for one K tile per MFMA and
// a 4 x 4 wave tile. Right after the barrier all waves of the block want their
// fragments at once and the LDS serves them one read at a time; if a wave asks
// for all ten fragments of the first tile row before its first MFMA, the matrix
// cores wait for the whole queue. Here a wave reads what its first MFMA needs,
// keeps about three reads in flight ahead of their use, and fetches the Y
// fragments of the next tile row during the current one.
// xo[i] is the lane's offset of the X fragment of tile i. XT: the operand roles
// of the MFMA are exchanged (Y supplies the instruction's "A" rows, X its "B"
// columns), which transposes what a lane holds of every 16 x 16 tile.
// FIRST: the first K tile of a C tile; the sums start from zero.
// xa[i] / ya: the lane's LDS address of the X fragment of tile i / of the Y
// fragment of tile row 0 in the current slots. late(): called among the MFMAs
// of the last tile row, for whatever the next iteration needs computed (its
// addresses, the slot numbers): work placed there is hidden behind MFMAs, work
// left between the last MFMA and the barrier is not.
template <int DT, int BX, int BY, bool XT, bool FIRST, typename Mid, typename Late>
__device__ __forceinline__ void mma_step_ordered(const unsigned (&xa)[4], unsigned ya,
                                                 float4_t (&acc_re)[4][4], float4_t (&acc_im)[4][4],
                                                 Mid &&mid, Late &&late) {
  static_assert(DtypeTraits<DT>::kTilesPerMfma == 1, "one K tile per MFMA");
  // (LDS addresses as 32-bit numbers: the read's address register is the number itself)
  typedef __attribute__((address_space(3))) const int4_t lds_int4_t;
  auto rd = [](unsigned address) {
    Fragment<DT> f;
    f.v[0] = *reinterpret_cast<lds_int4_t *>(address);
    return f;
  };
  auto mm = [](const Fragment<DT> &x, const Fragment<DT> &y, float4_t acc) {
    return XT ? mfma<DT>(y, x, acc) : mfma<DT>(x, y, acc);
  };
  auto c0 = [](const float4_t &acc) { return FIRST ? float4_t{0.f, 0.f, 0.f, 0.f} : acc; };
  constexpr int ROW16 = 16 * kTileRowBytes, XP = BX * kTileRowBytes, YP = BY * kTileRowBytes;
#define CCGLIB_PIN __builtin_amdgcn_sched_barrier(0)
  Fragment<DT> xr[4], xi[4], yr, yi, yin, yr_next, yi_next;
  yr = rd(ya);
  xr[0] = rd(xa[0]);
  xr[1] = rd(xa[1]);
  xr[2] = rd(xa[2]);
  CCGLIB_PIN;
  acc_re[0][0] = mm(xr[0], yr, c0(acc_re[0][0]));
  xr[3] = rd(xa[3]);
  CCGLIB_PIN;
  acc_re[0][1] = mm(xr[1], yr, c0(acc_re[0][1]));
  yi = rd(ya + YP);
  CCGLIB_PIN;
  acc_re[0][2] = mm(xr[2], yr, c0(acc_re[0][2]));
  xi[0] = rd(xa[0] + XP);
  CCGLIB_PIN;
  acc_re[0][3] = mm(xr[3], yr, c0(acc_re[0][3]));
  xi[1] = rd(xa[1] + XP);
  CCGLIB_PIN;
  acc_im[0][0] = mm(xr[0], yi, c0(acc_im[0][0]));
  xi[2] = rd(xa[2] + XP);
  CCGLIB_PIN;
  acc_im[0][1] = mm(xr[1], yi, c0(acc_im[0][1]));
  xi[3] = rd(xa[3] + XP);
  CCGLIB_PIN;
  acc_im[0][2] = mm(xr[2], yi, c0(acc_im[0][2]));
  yin = negate<DT>(yi);
  CCGLIB_PIN;
  acc_im[0][3] = mm(xr[3], yi, c0(acc_im[0][3]));
  yr_next = rd(ya + ROW16);
  CCGLIB_PIN;
  acc_re[0][0] = mm(xi[0], yin, acc_re[0][0]);
  yi_next = rd(ya + YP + ROW16);
  CCGLIB_PIN;
  acc_im[0][0] = mm(xi[0], yr, acc_im[0][0]);
#pragma unroll
  for (int i = 1; i < 4; ++i) {
    acc_re[0][i] = mm(xi[i], yin, acc_re[0][i]);
    acc_im[0][i] = mm(xi[i], yr, acc_im[0][i]);
  }
  CCGLIB_PIN;
  mid();
  CCGLIB_PIN;
#pragma unroll
  for (int j = 1; j < 4; ++j) {
    yr = yr_next;
    yi = yi_next;
    yin = negate<DT>(yi);
    CCGLIB_PIN;
    // from one MFMA to the next only one of the two operands changes (measured 1-2 %
    // faster on random data than four MFMAs per Y fragment in a row: the part is
    // power limited, and this order toggles fewer operand bits)
    acc_re[j][0] = mm(xr[0], yr, c0(acc_re[j][0]));
    acc_im[j][0] = mm(xr[0], yi, c0(acc_im[j][0]));
    acc_im[j][1] = mm(xr[1], yi, c0(acc_im[j][1]));
    acc_re[j][1] = mm(xr[1], yr, c0(acc_re[j][1]));
    if (j < 3) yr_next = rd(ya + (j + 1) * ROW16);
    CCGLIB_PIN;
    acc_re[j][2] = mm(xr[2], yr, c0(acc_re[j][2]));
    acc_im[j][2] = mm(xr[2], yi, c0(acc_im[j][2]));
    acc_im[j][3] = mm(xr[3], yi, c0(acc_im[j][3]));
    acc_re[j][3] = mm(xr[3], yr, c0(acc_re[j][3]));
    if (j < 3) yi_next = rd(ya + YP + (j + 1) * ROW16);
    CCGLIB_PIN;
    if (j == 3) {
      late();
      CCGLIB_PIN;
    }
    acc_im[j][0] = mm(xi[0], yr, acc_im[j][0]);
    acc_re[j][0] = mm(xi[0], yin, acc_re[j][0]);
    acc_re[j][1] = mm(xi[1], yin, acc_re[j][1]);
    acc_im[j][1] = mm(xi[1], yr, acc_im[j][1]);
    acc_im[j][2] = mm(xi[2], yr, acc_im[j][2]);
    acc_re[j][2] = mm(xi[2], yin, acc_re[j][2]);
    acc_re[j][3] = mm(xi[3], yin, acc_re[j][3]);
    acc_im[j][3] = mm(xi[3], yr, acc_im[j][3]);
    CCGLIB_PIN;
  }
#undef CCGLIB_PIN
}

// The same on the 32-row MFMAs: TX x TY tiles of 32x32, one K tile per step.
// off[0] and off[1] are the lane's two 16-byte chunks of its row.
template <int DT, int BX, int BY, int TX, int TY, typename Mid>
__device__ __forceinline__ void mma_step32(const char *slot, const int (&x_off)[2],
                                           const int (&y_off)[2], float16_t_ (&acc_re)[TY][TX],
                                           float16_t_ (&acc_im)[TY][TX], Mid &&mid) {
  constexpr int D = TX > TY ? TX : TY;
  Fragment32 xr[TX], xi[TX], yr[TY], yi[TY], yin[TY];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    if (d < TX) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const char *p = slot + x_off[u] + d * 32 * kTileRowBytes;
        xr[d].v[u] = *reinterpret_cast<const int4_t *>(p);
        xi[d].v[u] = *reinterpret_cast<const int4_t *>(p + BX * kTileRowBytes);
      }
    }
    if (d < TY) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const char *p = slot + y_off[u] + d * 32 * kTileRowBytes;
        yr[d].v[u] = *reinterpret_cast<const int4_t *>(p);
        yi[d].v[u] = *reinterpret_cast<const int4_t *>(p + BY * kTileRowBytes);
      }
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d) {
    __builtin_amdgcn_sched_barrier(0);
    if (d < TY) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int w = 0; w < 4; ++w) yin[d].v[u][w] = yi[d].v[u][w] ^ (int)DtypeTraits<DT>::kSignMask;
      }
    }
    int ti[TX + TY], tj[TX + TY], n = 0;
    if (d < TX) {
#pragma unroll
      for (int j = 0; j < d && j < TY; ++j) ti[n] = d, tj[n] = j, ++n;
    }
    if (d < TY) {
#pragma unroll
      for (int i = 0; i <= d && i < TX; ++i) ti[n] = i, tj[n] = d, ++n;
    }
#pragma unroll
    for (int t = 0; t < n; ++t)
      acc_re[tj[t]][ti[t]] = mfma32<DT>(xr[ti[t]], yr[tj[t]], acc_re[tj[t]][ti[t]]);
#pragma unroll
    for (int t = 0; t < n; ++t)
      acc_im[tj[t]][ti[t]] = mfma32<DT>(xr[ti[t]], yi[tj[t]], acc_im[tj[t]][ti[t]]);
#pragma unroll
    for (int t = 0; t < n; ++t)
      acc_re[tj[t]][ti[t]] = mfma32<DT>(xi[ti[t]], yin[tj[t]], acc_re[tj[t]][ti[t]]);
#pragma unroll
    for (int t = 0; t < n; ++t)
      acc_im[tj[t]][ti[t]] = mfma32<DT>(xi[ti[t]], yr[tj[t]], acc_im[tj[t]][ti[t]]);
    if (d == 0) {
      __builtin_amdgcn_sched_barrier(0);
      mid();
    }
  }
  __builtin_amdgcn_sched_barrier(0);
}

// The 32-row step for a 2 x 2 wave tile with the LDS reads in order of need
// (see mma_step_ordered): two 16-byte reads per fragment.
template <int DT, int BX, int BY, typename Mid>
__device__ __forceinline__ void mma_step32_ordered(const char *slot, const int (&x_off)[2],
                                                   const int (&y_off)[2], float16_t_ (&acc_re)[2][2],
                                                   float16_t_ (&acc_im)[2][2], Mid &&mid) {
  auto rd = [&](const int (&off)[2], int extra) {
    Fragment32 f;
    f.v[0] = *reinterpret_cast<const int4_t *>(slot + off[0] + extra);
    f.v[1] = *reinterpret_cast<const int4_t *>(slot + off[1] + extra);
    return f;
  };
  auto neg = [](const Fragment32 &f) {
    Fragment32 r;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int w = 0; w < 4; ++w) r.v[u][w] = f.v[u][w] ^ (int)DtypeTraits<DT>::kSignMask;
    }
    return r;
  };
  constexpr int ROW32 = 32 * kTileRowBytes, XP = BX * kTileRowBytes, YP = BY * kTileRowBytes;
#define CCGLIB_PIN __builtin_amdgcn_sched_barrier(0)
  Fragment32 x0r, x0i, x1r, x1i, y0r, y0i, y0n, y1r, y1i, y1n;
  y0r = rd(y_off, 0);
  x0r = rd(x_off, 0);
  y0i = rd(y_off, YP);
  CCGLIB_PIN;
  acc_re[0][0] = mfma32<DT>(x0r, y0r, acc_re[0][0]);
  x0i = rd(x_off, XP);
  CCGLIB_PIN;
  acc_im[0][0] = mfma32<DT>(x0r, y0i, acc_im[0][0]);
  y0n = neg(y0i);
  x1r = rd(x_off, ROW32);
  CCGLIB_PIN;
  acc_re[0][0] = mfma32<DT>(x0i, y0n, acc_re[0][0]);
  x1i = rd(x_off, XP + ROW32);
  CCGLIB_PIN;
  acc_im[0][0] = mfma32<DT>(x0i, y0r, acc_im[0][0]);
  CCGLIB_PIN;
  mid();
  CCGLIB_PIN;
  acc_re[0][1] = mfma32<DT>(x1r, y0r, acc_re[0][1]);
  y1r = rd(y_off, ROW32);
  CCGLIB_PIN;
  acc_im[0][1] = mfma32<DT>(x1r, y0i, acc_im[0][1]);
  y1i = rd(y_off, YP + ROW32);
  CCGLIB_PIN;
  acc_re[0][1] = mfma32<DT>(x1i, y0n, acc_re[0][1]);
  acc_im[0][1] = mfma32<DT>(x1i, y0r, acc_im[0][1]);
  CCGLIB_PIN;
  acc_re[1][0] = mfma32<DT>(x0r, y1r, acc_re[1][0]);
  acc_im[1][0] = mfma32<DT>(x0r, y1i, acc_im[1][0]);
  y1n = neg(y1i);
  CCGLIB_PIN;
  acc_re[1][0] = mfma32<DT>(x0i, y1n, acc_re[1][0]);
  acc_im[1][0] = mfma32<DT>(x0i, y1r, acc_im[1][0]);
  acc_re[1][1] = mfma32<DT>(x1r, y1r, acc_re[1][1]);
  acc_im[1][1] = mfma32<DT>(x1r, y1i, acc_im[1][1]);
  acc_re[1][1] = mfma32<DT>(x1i, y1n, acc_re[1][1]);
  acc_im[1][1] = mfma32<DT>(x1i, y1r, acc_im[1][1]);
  CCGLIB_PIN;
#undef CCGLIB_PIN
}

// 1-bit samples, multiplied on the fp4 MFMA straight from the packed words.
// A 64-byte row of a slot holds 512 samples; a lane reads its two 16-byte
// chunks of a row as for the other 32-row MFMAs, and each of the eight words
// it then holds feeds one 32x32x64 MFMA (64 samples of K: 32 from each half of
// the wave). A word becomes the MFMA's four operand registers with seven
// vector-ALU instructions: nibble i of register j is 0x2 | bit (4 i + j) << 3,
// i.e. fp4 +1.0 for a 0 bit and -1.0 for a 1 bit. Which sample lands in which
// K position of the instruction does not matter as long as X and Y agree, and
// neither does the sign convention (bit 1 = +1 in src/reference/GEMM.cpp:131-200):
// negating X and Y together leaves every product as it is. The expansion of the
// fragment that is needed two to four MFMAs later is placed behind each MFMA,
// in whose shadow the vector ALU is otherwise idle; the MFMAs are issued so
// that only one operand changes from one to the next.
// Samples past K (zero bits in both operands, which the tiled layout and the
// zero tile guarantee) add 0 to every real and +2 to every imaginary sum; the
// epilogue takes that off (KernelArgs::im_excess), which is the reference's
// K_PADDING correction (kernels/gemm_kernel_int1.cu:64-196).
__device__ __forceinline__ int4_t expand_bits(int word) {
  const unsigned w = (unsigned)word;
  int4_t o;
  // (a & b) | c in one instruction (truth table 0xEA)
  o[0] = (int)__builtin_amdgcn_bitop3_b32(w << 3, 0x88888888u, 0x22222222u, 0xEA);
  o[1] = (int)__builtin_amdgcn_bitop3_b32(w << 2, 0x88888888u, 0x22222222u, 0xEA);
  o[2] = (int)__builtin_amdgcn_bitop3_b32(w << 1, 0x88888888u, 0x22222222u, 0xEA);
  o[3] = (int)__builtin_amdgcn_bitop3_b32(w, 0x88888888u, 0x22222222u, 0xEA);
  return o;
}

__device__ __forceinline__ float16_t_ mfma_fp4(const int4_t &a, const int4_t &b, float16_t_ acc) {
  // format code 4 = fp4 (only the low four registers are read); scale 2^0
  const int8_t_ av = {a[0], a[1], a[2], a[3], 0, 0, 0, 0};
  const int8_t_ bv = {b[0], b[1], b[2], b[3], 0, 0, 0, 0};
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, acc, 4, 4, 0, 0x7f, 0, 0x7f);
}

template <int BX, int BY, typename Mid>
__device__ __forceinline__ void mma_step32_bits(const char *slot, const int (&x_off)[2],
                                                const int (&y_off)[2], float16_t_ (&acc_re)[2][2],
                                                float16_t_ (&acc_im)[2][2], Mid &&mid) {
  constexpr int ROW32 = 32 * kTileRowBytes, XP = BX * kTileRowBytes, YP = BY * kTileRowBytes;
  // fragments: 0 x0r, 1 x0i, 2 x1r, 3 x1i, 4 y0r, 5 y0i, 6 y1r, 7 y1i
  enum { X0R, X0I, X1R, X1I, Y0R, Y0I, Y1R, Y1I };
  int4_t raw[8];    // the chunk (four words, one per MFMA step) in use
  auto rd = [&](int f, int u) {
    const int off = (f < 4 ? x_off[u] : y_off[u]) + ((f & 1) ? (f < 4 ? XP : YP) : 0) +
                    ((f & 2) ? ROW32 : 0);
    raw[f] = *reinterpret_cast<const int4_t *>(slot + off);
  };
  auto neg = [](const int4_t &f) {
    int4_t r;
#pragma unroll
    for (int w = 0; w < 4; ++w) r[w] = f[w] ^ (int)0x88888888u;
    return r;
  };
#define CCGLIB_PIN __builtin_amdgcn_sched_barrier(0)
  // in order of first use
  rd(X0R, 0);
  rd(Y0R, 0);
  rd(Y0I, 0);
  rd(Y1I, 0);
  rd(Y1R, 0);
  rd(X1R, 0);
  rd(X1I, 0);
  rd(X0I, 0);
  CCGLIB_PIN;
  int4_t x0r = expand_bits(raw[X0R][0]), y0r = expand_bits(raw[Y0R][0]),
         y0i = expand_bits(raw[Y0I][0]);
  int4_t x0i, x1r, x1i, y1r, y1i, y0n, y1n, x0r_next, y0r_next, y0i_next;
  CCGLIB_PIN;
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int w = s & 3;
    // after a chunk's last word has been taken, the next chunk of the row is read
    // into the same registers (its first word is needed sixteen MFMAs later)
    const bool reload = (s == 3);
    const bool reload_next = (s == 2);   // for the fragments expanded one step ahead
    acc_re[0][0] = mfma_fp4(x0r, y0r, acc_re[0][0]);
    y1i = expand_bits(raw[Y1I][w]);
    if (reload) rd(Y1I, 1);
    CCGLIB_PIN;
    acc_im[0][0] = mfma_fp4(x0r, y0i, acc_im[0][0]);
    y1r = expand_bits(raw[Y1R][w]);
    if (reload) rd(Y1R, 1);
    CCGLIB_PIN;
    acc_im[1][0] = mfma_fp4(x0r, y1i, acc_im[1][0]);
    x1r = expand_bits(raw[X1R][w]);
    if (reload) rd(X1R, 1);
    CCGLIB_PIN;
    acc_re[1][0] = mfma_fp4(x0r, y1r, acc_re[1][0]);
    x1i = expand_bits(raw[X1I][w]);
    if (reload) rd(X1I, 1);
    CCGLIB_PIN;
    if (s == 0) {
      mid();
      CCGLIB_PIN;
    }
    acc_re[1][1] = mfma_fp4(x1r, y1r, acc_re[1][1]);
    y0n = neg(y0i);
    CCGLIB_PIN;
    acc_im[1][1] = mfma_fp4(x1r, y1i, acc_im[1][1]);
    y1n = neg(y1i);
    CCGLIB_PIN;
    acc_im[0][1] = mfma_fp4(x1r, y0i, acc_im[0][1]);
    x0i = expand_bits(raw[X0I][w]);
    if (reload) rd(X0I, 1);
    CCGLIB_PIN;
    acc_re[0][1] = mfma_fp4(x1r, y0r, acc_re[0][1]);
    CCGLIB_PIN;
    acc_im[0][1] = mfma_fp4(x1i, y0r, acc_im[0][1]);
    CCGLIB_PIN;
    acc_re[0][1] = mfma_fp4(x1i, y0n, acc_re[0][1]);
    if (s < 7) x0r_next = expand_bits(raw[X0R][(s + 1) & 3]);
    if (reload_next) rd(X0R, 1);
    CCGLIB_PIN;
    acc_re[1][1] = mfma_fp4(x1i, y1n, acc_re[1][1]);
    if (s < 7) y0r_next = expand_bits(raw[Y0R][(s + 1) & 3]);
    if (reload_next) rd(Y0R, 1);
    CCGLIB_PIN;
    acc_im[1][1] = mfma_fp4(x1i, y1r, acc_im[1][1]);
    if (s < 7) y0i_next = expand_bits(raw[Y0I][(s + 1) & 3]);
    if (reload_next) rd(Y0I, 1);
    CCGLIB_PIN;
    acc_im[1][0] = mfma_fp4(x0i, y1r, acc_im[1][0]);
    acc_re[1][0] = mfma_fp4(x0i, y1n, acc_re[1][0]);
    acc_re[0][0] = mfma_fp4(x0i, y0n, acc_re[0][0]);
    acc_im[0][0] = mfma_fp4(x0i, y0r, acc_im[0][0]);
    CCGLIB_PIN;
    if (s < 7) {
      x0r = x0r_next;
      y0r = y0r_next;
      y0i = y0i_next;
    }
  }
#undef CCGLIB_PIN
}

// The same for interleaved operands (rows of (re, im) pairs, as the caller's
// buffers hold them). With K running over the 2K real numbers of a row,
//   Re = sum X~ . Y1,  Y1 = (yr, -yi, ...)   and   Im = sum X~ . Y2,  Y2 = (yi, yr, ...)
// so the raw X fragment is used as it is and both Y variants come from the raw
// Y fragment in registers: a sign flip of the odd elements and a swap inside
// each pair. Two MFMAs per fragment pair over half as many complex values:
// the same MFMA and LDS work per complex MAC as with planar operands.
template <int DT, int BX, int BY, int TX, int TY, typename Mid>
__device__ __forceinline__ void mma_step_interleaved(const char *slot, const int (&x_off)[2],
                                                     const int (&y_off)[2],
                                                     float4_t (&acc_re)[TY][TX],
                                                     float4_t (&acc_im)[TY][TX], Mid &&mid) {
  // The slot holds 128 bytes of every row; x_off / y_off are the lane's two
  // 16-byte chunks of its row. fp8 takes both in one MFMA, 16-bit input one
  // per MFMA (two passes over the slot).
  constexpr int KPM = DtypeTraits<DT>::kTilesPerMfma;
  constexpr int PASSES = 2 / KPM;
  constexpr bool kBytes = DtypeTraits<DT>::kElemBytes == 1;
#pragma unroll
  for (int h = 0; h < PASSES; ++h) {
    Fragment<DT> x[TX];
#pragma unroll
    for (int i = 0; i < TX; ++i) {
#pragma unroll
      for (int u = 0; u < KPM; ++u) {
        x[i].v[u] = *reinterpret_cast<const int4_t *>(slot + x_off[h * KPM + u] + i * 16 * 128);
      }
    }
#pragma unroll
    for (int j = 0; j < TY; ++j) {
      Fragment<DT> y1, y2;
#pragma unroll
      for (int u = 0; u < KPM; ++u) {
        const int4_t raw =
            *reinterpret_cast<const int4_t *>(slot + y_off[h * KPM + u] + j * 16 * 128);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const unsigned v = (unsigned)raw[w];
          y1.v[u][w] = (int)(v ^ (kBytes ? 0x80008000u : 0x80000000u));
          y2.v[u][w] = kBytes ? (int)__builtin_amdgcn_perm(v, v, 0x02030001u)
                              : (int)__builtin_amdgcn_alignbit(v, v, 16);
        }
      }
#pragma unroll
      for (int i = 0; i < TX; ++i) acc_re[j][i] = mfma<DT>(x[i], y1, acc_re[j][i]);
#pragma unroll
      for (int i = 0; i < TX; ++i) acc_im[j][i] = mfma<DT>(x[i], y2, acc_im[j][i]);
      if (h == 0 && j == 0) mid();
    }
  }
}

// The interleaved step for 16-bit input and a 4 x 4 wave tile with every LDS
// read and every derived fragment placed by hand (see mma_step_ordered). The
// slot is walked as eight tile rows (two halves of K x four rows of Y). The raw
// Y fragment of a row is read two rows ahead; its two variants are computed
// during the previous row, two instructions behind each of that row's last
// four MFMAs, where they issue in the shadow of the matrix instruction instead
// of holding up the next row; the X fragments of the second half are fetched
// during rows 2 and 3.
template <int DT, int BX, int BY, typename Mid>
__device__ __forceinline__ void mma_step_interleaved_ordered(const char *slot, const int (&x_off)[2],
                                                             const int (&y_off)[2],
                                                             float4_t (&acc_re)[4][4],
                                                             float4_t (&acc_im)[4][4], Mid &&mid) {
  static_assert(DtypeTraits<DT>::kTilesPerMfma == 1 && DtypeTraits<DT>::kElemBytes == 2,
                "16-bit input");
  auto rd = [&](int off) {
    Fragment<DT> f;
    f.v[0] = *reinterpret_cast<const int4_t *>(slot + off);
    return f;
  };
  // words w0, w0 + 1 of (yr, -yi, ...) and of (yi, yr, ...) from the raw (yr, yi, ...).
  // The empty asm statement takes the result where it is computed: without it,
  // arithmetic whose result is first used in the next row is sunk there before
  // the instructions are scheduled. (The arithmetic itself stays ordinary code,
  // so the compiler keeps track of the wait states the MFMAs need.)
  auto flip2 = [](Fragment<DT> &f, const Fragment<DT> &raw, int w0) {
#pragma unroll
    for (int w = w0; w < w0 + 2; ++w) {
      int o = (int)((unsigned)raw.v[0][w] ^ 0x80000000u);
      asm volatile("" : "+v"(o));
      f.v[0][w] = o;
    }
  };
  auto swap2 = [](Fragment<DT> &f, const Fragment<DT> &raw, int w0) {
#pragma unroll
    for (int w = w0; w < w0 + 2; ++w) {
      const unsigned v = (unsigned)raw.v[0][w];
      int o = (int)__builtin_amdgcn_alignbit(v, v, 16);
      asm volatile("" : "+v"(o));
      f.v[0][w] = o;
    }
  };
  constexpr int ROW16 = 16 * 128;
  auto y_row_off = [&](int r) { return y_off[r >> 2] + (r & 3) * ROW16; };
#define CCGLIB_PIN __builtin_amdgcn_sched_barrier(0)
  Fragment<DT> xa[4], xb[4], raw[2], y1, y2, y1n, y2n;
  raw[0] = rd(y_row_off(0));
  xa[0] = rd(x_off[0]);
  xa[1] = rd(x_off[0] + ROW16);
  raw[1] = rd(y_row_off(1));
  xa[2] = rd(x_off[0] + 2 * ROW16);
  CCGLIB_PIN;
  flip2(y1, raw[0], 0);
  flip2(y1, raw[0], 2);
  swap2(y2, raw[0], 0);
  swap2(y2, raw[0], 2);
  CCGLIB_PIN;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int j = r & 3;
    Fragment<DT>(&x)[4] = r < 4 ? xa : xb;
    const Fragment<DT> &next_raw = raw[(r + 1) & 1];
    acc_re[j][0] = mfma<DT>(x[0], y1, acc_re[j][0]);
    if (r == 0) xa[3] = rd(x_off[0] + 3 * ROW16);
    if (r + 2 < 8) raw[r & 1] = rd(y_row_off(r + 2));   // this row's raw fragment is used up
    CCGLIB_PIN;
    acc_im[j][0] = mfma<DT>(x[0], y2, acc_im[j][0]);
    if (r == 2 || r == 3) xb[2 * (r - 2)] = rd(x_off[1] + 2 * (r - 2) * ROW16);
    CCGLIB_PIN;
    // (from one MFMA to the next only one of the two operands changes)
    acc_im[j][1] = mfma<DT>(x[1], y2, acc_im[j][1]);
    if (r == 2 || r == 3) xb[2 * (r - 2) + 1] = rd(x_off[1] + (2 * (r - 2) + 1) * ROW16);
    CCGLIB_PIN;
    acc_re[j][1] = mfma<DT>(x[1], y1, acc_re[j][1]);
    CCGLIB_PIN;
    acc_re[j][2] = mfma<DT>(x[2], y1, acc_re[j][2]);
    if (r + 1 < 8) flip2(y1n, next_raw, 0);
    CCGLIB_PIN;
    acc_im[j][2] = mfma<DT>(x[2], y2, acc_im[j][2]);
    if (r + 1 < 8) flip2(y1n, next_raw, 2);
    CCGLIB_PIN;
    acc_im[j][3] = mfma<DT>(x[3], y2, acc_im[j][3]);
    if (r + 1 < 8) swap2(y2n, next_raw, 0);
    CCGLIB_PIN;
    acc_re[j][3] = mfma<DT>(x[3], y1, acc_re[j][3]);
    if (r + 1 < 8) swap2(y2n, next_raw, 2);
    CCGLIB_PIN;
    if (r == 0) {
      mid();
      CCGLIB_PIN;
    }
    y1 = y1n;
    y2 = y2n;
  }
#undef CCGLIB_PIN
}

// Interleaved 8-bit operands on the 32-row MFMA: a 2 x 2 wave tile of 32 x 32
// tiles; the slot holds 128 bytes (64 (re, im) pairs) of every row, walked in two
// halves of 64 bytes, one MFMA step each. off[h][u] are the lane's two 16-byte
// chunks of its row in half h. As for 16-bit input the raw X fragment is used
// as it is and both Y variants come from the raw Y fragment: a sign flip of the
// odd bytes and a swap inside each byte pair. LDS reads are placed by hand, a
// fragment being fetched about four MFMAs (of 32 cycles) ahead of its use.
template <int DT, int BX, int BY, typename Mid>
__device__ __forceinline__ void mma_step32_interleaved(const char *slot, const int (&x_off)[2][2],
                                                       const int (&y_off)[2][2],
                                                       float16_t_ (&acc_re)[2][2],
                                                       float16_t_ (&acc_im)[2][2], Mid &&mid) {
  static_assert(DtypeTraits<DT>::kElemBytes == 1, "8-bit input");
  auto rd = [&](const int (&off)[2], int extra) {
    Fragment32 f;
    f.v[0] = *reinterpret_cast<const int4_t *>(slot + off[0] + extra);
    f.v[1] = *reinterpret_cast<const int4_t *>(slot + off[1] + extra);
    return f;
  };
  auto flip = [](const Fragment32 &raw) {      // (yr, -yi, ...)
    Fragment32 f;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int w = 0; w < 4; ++w) f.v[u][w] = (int)((unsigned)raw.v[u][w] ^ 0x80008000u);
    }
    return f;
  };
  auto swap = [](const Fragment32 &raw) {      // (yi, yr, ...)
    Fragment32 f;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const unsigned v = (unsigned)raw.v[u][w];
        f.v[u][w] = (int)__builtin_amdgcn_perm(v, v, 0x02030001u);
      }
    }
    return f;
  };
  constexpr int ROW32 = 32 * 128;
#define CCGLIB_PIN __builtin_amdgcn_sched_barrier(0)
  Fragment32 x0, x1, raw0, raw1, ya, yb;
  raw0 = rd(y_off[0], 0);
  x0 = rd(x_off[0], 0);
  x1 = rd(x_off[0], ROW32);
  CCGLIB_PIN;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    ya = flip(raw0);
    yb = swap(raw0);
    CCGLIB_PIN;
    acc_re[0][0] = mfma32<DT>(x0, ya, acc_re[0][0]);
    raw1 = rd(y_off[h], ROW32);
    CCGLIB_PIN;
    acc_im[0][0] = mfma32<DT>(x0, yb, acc_im[0][0]);
    CCGLIB_PIN;
    if (h == 0) {
      mid();
      CCGLIB_PIN;
    }
    acc_re[0][1] = mfma32<DT>(x1, ya, acc_re[0][1]);
    if (h == 0) raw0 = rd(y_off[1], 0);
    CCGLIB_PIN;
    acc_im[0][1] = mfma32<DT>(x1, yb, acc_im[0][1]);
    ya = flip(raw1);
    yb = swap(raw1);
    CCGLIB_PIN;
    acc_re[1][0] = mfma32<DT>(x0, ya, acc_re[1][0]);
    acc_im[1][0] = mfma32<DT>(x0, yb, acc_im[1][0]);
    if (h == 0) x0 = rd(x_off[1], 0);
    CCGLIB_PIN;
    acc_re[1][1] = mfma32<DT>(x1, ya, acc_re[1][1]);
    acc_im[1][1] = mfma32<DT>(x1, yb, acc_im[1][1]);
    if (h == 0) x1 = rd(x_off[1], ROW32);
    CCGLIB_PIN;
  }
#undef CCGLIB_PIN
}

// The K tile of a wave of 32 x 32 in a 64 x 64 block (2 x 2 MFMA tiles of 16 x 16, or one of 32 x 32):
// eight 16-byte fragments, read from the slot in one iteration and multiplied in the next, while
// those of the next K tile are read. A lone wave of a SIMD, which is what a small problem
// has, would otherwise wait for its reads in every iteration (bf16 planar rows, 256^3
// 6.45 -> 6.27 us, B=4 48x64x1600 19.0 -> 17.9; the loop then runs at the rate at which the copies of
// half cache lines are issued, and a deeper ring is slower: 9 slots 7.2 and 21.2 us).
struct SmallTile {
  int4_t x[4], y[4];
};
// x[2 i + p]: 16-row MFMA: fragment i, plane p (pairs: half p of the 128 bytes); 32-row MFMA: chunk i
// of plane p (pairs: chunk i of half p). The same for y.
__device__ __forceinline__ void read_small_tile(const char *slot, const int (&x_off)[2][2], const int (&y_off)[2][2],
                                                SmallTile &t) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      t.x[2 * i + p] = *reinterpret_cast<const int4_t *>(slot + x_off[p][i]);
      t.y[2 * i + p] = *reinterpret_cast<const int4_t *>(slot + y_off[p][i]);
    }
  }
}
// For every sum the order of the steps for larger wave tiles.
template <int DT, bool IL, typename Mid>
__device__ __forceinline__ void mma_small_tile(const SmallTile &t, float4_t (&acc_re)[2][2], float4_t (&acc_im)[2][2],
                                               Mid &&mid) {
  auto frag = [](const int4_t &v) {
    Fragment<DT> f;
    f.v[0] = v;
    return f;
  };
  if constexpr (IL) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        Fragment<DT> y1, y2;   // (yr, -yi, ...), (yi, yr, ...)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const unsigned v = (unsigned)t.y[2 * j + h][w];
          y1.v[0][w] = (int)(v ^ 0x80000000u);
          y2.v[0][w] = (int)__builtin_amdgcn_alignbit(v, v, 16);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) acc_re[j][i] = mfma<DT>(frag(t.x[2 * i + h]), y1, acc_re[j][i]);
#pragma unroll
        for (int i = 0; i < 2; ++i) acc_im[j][i] = mfma<DT>(frag(t.x[2 * i + h]), y2, acc_im[j][i]);
        if (h == 0 && j == 0) mid();
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const Fragment<DT> yr = frag(t.y[2 * j]), yi = frag(t.y[2 * j + 1]), yin = negate<DT>(yi);
#pragma unroll
      for (int i = 0; i < 2; ++i) acc_re[j][i] = mfma<DT>(frag(t.x[2 * i]), yr, acc_re[j][i]);
#pragma unroll
      for (int i = 0; i < 2; ++i) acc_im[j][i] = mfma<DT>(frag(t.x[2 * i]), yi, acc_im[j][i]);
#pragma unroll
      for (int i = 0; i < 2; ++i) acc_re[j][i] = mfma<DT>(frag(t.x[2 * i + 1]), yin, acc_re[j][i]);
#pragma unroll
      for (int i = 0; i < 2; ++i) acc_im[j][i] = mfma<DT>(frag(t.x[2 * i + 1]), yr, acc_im[j][i]);
      if (j == 0) mid();
    }
  }
}
template <int DT, bool IL, typename Mid>
__device__ __forceinline__ void mma_small_tile(const SmallTile &t, float16_t_ (&acc_re)[1][1],
                                               float16_t_ (&acc_im)[1][1], Mid &&mid) {
  if constexpr (DT == kInt1) {
    // (every word is expanded for a single tile: the vector ALU has about as much to do as the
    // matrix cores)
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int u = 2 * (s >> 2), w = s & 3;
      const int4_t x0 = expand_bits(t.x[u][w]), x1 = expand_bits(t.x[u + 1][w]);
      const int4_t y0 = expand_bits(t.y[u][w]), y1 = expand_bits(t.y[u + 1][w]);
      int4_t y1n;
#pragma unroll
      for (int e = 0; e < 4; ++e) y1n[e] = y1[e] ^ (int)0x88888888u;
      acc_re[0][0] = mfma_fp4(x0, y0, acc_re[0][0]);
      acc_im[0][0] = mfma_fp4(x0, y1, acc_im[0][0]);
      acc_re[0][0] = mfma_fp4(x1, y1n, acc_re[0][0]);
      acc_im[0][0] = mfma_fp4(x1, y0, acc_im[0][0]);
      if (s == 0) mid();
    }
  } else if constexpr (IL) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      Fragment32 x{{t.x[h], t.x[2 + h]}}, ya, yb;   // (yr, -yi, ...), (yi, yr, ...)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const unsigned v = (unsigned)t.y[2 * u + h][w];
          ya.v[u][w] = (int)(v ^ 0x80008000u);
          yb.v[u][w] = (int)__builtin_amdgcn_perm(v, v, 0x02030001u);
        }
      }
      acc_re[0][0] = mfma32<DT>(x, ya, acc_re[0][0]);
      acc_im[0][0] = mfma32<DT>(x, yb, acc_im[0][0]);
      if (h == 0) mid();
    }
  } else {
    const Fragment32 xr{{t.x[0], t.x[2]}}, xi{{t.x[1], t.x[3]}}, yr{{t.y[0], t.y[2]}}, yi{{t.y[1], t.y[3]}};
    Fragment32 yin;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int w = 0; w < 4; ++w) yin.v[u][w] = yi.v[u][w] ^ (int)DtypeTraits<DT>::kSignMask;
    }
    acc_re[0][0] = mfma32<DT>(xr, yr, acc_re[0][0]);
    acc_im[0][0] = mfma32<DT>(xr, yi, acc_im[0][0]);
    mid();
    acc_re[0][0] = mfma32<DT>(xi, yin, acc_re[0][0]);
    acc_im[0][0] = mfma32<DT>(xi, yr, acc_im[0][0]);
  }
}

// 32-bit input on the bf16 instruction. x = h + m + l, each of the three a bf16 (8 of the 24
// significant bits; what rounding to nearest takes too much or too little the next
// part gives back), and of the nine products of two such sums all but l * l, which lies below
// 2^-33 of the largest, are added up. The product h * h, which has 16 bits, goes into one
// accumulator, the seven others into a second one, of 2^-8 of its size; the two are added when K is
// through. So nothing of a single product is lost but in that last addition, as on the fp32
// instructions, and the large sum is rounded twice per 16 values of K and part. (In one accumulator,
// and with six products, every small product rounds the whole sum - and the instruction drops what of a
// smaller sum lies below half a unit of its largest product: one product of two numbers was off by
// up to 1.4 units in the last place.) N(0, 1) operands, relative error of the result against 64
// bits, fp32 instructions and these: K = 1 3.1e-8, 2.6e-8; K = 32 1.4e-7, 4.9e-8; K = 1000
// 8.0e-7, 2.7e-7; K = 8192 2.3e-6, 8.3e-7; a single product 0.5 units in the last place either way.
// Eight 32x32x16 instructions take the time of half of the fp32 ones they stand for (2.5 PFLOP/s
// dense against 0.157). Planar pipelines, fp32 instructions, these, and one accumulator with six products,
// in us: 4096x4096x512 496, 421, 316; 8192x8192x1024 3740, 3250, 2400; B=2 1000^3 134, 128, 111.
//   Both operands are scaled by 2^24 first and the result by 2^-48, so that no part of a
// small number falls below the range of a bf16: the split is exact for every magnitude up to 2^104.
// What the instructions cannot do is an infinity, a NaN or a larger number (their parts are
// infinite or NaN) or a sum beyond 2^80: the accumulators are then not finite, and the wave computes
// its tile again with the fp32 instructions (recompute_f32) - unless those sums are NaN because of
// a NaN in their rows, such as marks a flagged sample, for which it only looks through the rows
// (only_nan_rows). Planar rows, 4096x4096x512 and B=2 1000^3, in us: finite 428, 124; a NaN in every row of X 531,
// 151 (computed again 1029, 288); an infinity in every row 1015, 279; the fp32 instructions 498, 134 at
// any values.
//   The splitting, 13 vector instructions for two elements, runs in every wave that reads an
// element (split tiles would take half as much LDS again) and in the shadow of the matrix
// instructions: those of a K tile are issued while the next one is split (see
// mma_step32_split).
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;
struct SplitF32 {
  int4_t h, m, l;
};
// Step s of 4 of the splitting of 8 values (x holds what is left to split). A step's
// instructions are independent of each other but for pairs of them: a chain of 13 for one
// pair of values after the other leaves the vector ALU waiting for its own results.
__device__ __forceinline__ void split_step(float (&x)[8], SplitF32 &o, int s) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  auto pack = [&](int4_t &p) {   // (round to nearest even)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = __builtin_bit_cast(int, __builtin_convertvector((float2_t{x[2 * i], x[2 * i + 1]}), bf16x2_t));
    }
  };
  auto subtract = [&](const int4_t &p) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned v = (unsigned)p[i];
      x[2 * i] -= __builtin_bit_cast(float, v << 16);
      x[2 * i + 1] -= __builtin_bit_cast(float, v & 0xffff0000u);
    }
  };
  if (s == 0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] *= kSplitScale;
    pack(o.h);
  } else if (s == 1) {
    subtract(o.h);
  } else if (s == 2) {
    pack(o.m);
    subtract(o.m);
  } else {
    pack(o.l);
  }
}
// products 0 to 7: l h, l m, m l, m m, m h, h l, h m, and h h, which goes into an accumulator of its own
constexpr int kSplitProducts = 8;
template <int P> __device__ __forceinline__ const int4_t &split_x(const SplitF32 &x) {
  return P < 2 ? x.l : P < 5 ? x.m : x.h;
}
template <int P>
__device__ __forceinline__ float16_t_ mfma_split(const int4_t &a, const SplitF32 &y, float16_t_ acc) {
  const int4_t &b = P == 2 || P == 5 ? y.l : P == 1 || P == 3 || P == 6 ? y.m : y.h;
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), acc, 0, 0, 0);
}
struct SplitPair {   // (re, im) fragments of 32 rows
  SplitF32 re, im;
};
struct SplitSum {    // of the products h h; of the others
  float16_t_ large, small;
};

// The 32 instructions of one 32 x 32 tile and K tile, in turn for its two parts (one that adds
// to the result of the one before waits for it); behind(n) is issued behind the n-th.
template <class F>
__device__ __forceinline__ void mma_split_tile(const SplitPair &x, const SplitPair &y, SplitSum &re, SplitSum &im,
                                               F &&behind) {
#define CCGLIB_PIN __builtin_amdgcn_sched_barrier(0)
  auto sum = [](SplitSum &s, auto product) -> float16_t_ & {
    return decltype(product)::value == kSplitProducts - 1 ? s.large : s.small;
  };
  static_for<kSplitProducts>([&](auto product) {
    constexpr int P = decltype(product)::value;
    const int4_t &a = split_x<P>(x.re);
    sum(re, product) = mfma_split<P>(a, y.re, sum(re, product));
    behind(2 * P);
    CCGLIB_PIN;
    sum(im, product) = mfma_split<P>(a, y.im, sum(im, product));
    behind(2 * P + 1);
    CCGLIB_PIN;
  });
  int4_t minus;
  static_for<kSplitProducts>([&](auto product) {
    constexpr int P = decltype(product)::value, N = 2 * kSplitProducts;
    const int4_t &a = split_x<P>(x.im);
    if constexpr (P == 0 || P == 2 || P == 5) {   // (the first product of a part of x)
#pragma unroll
      for (int i = 0; i < 4; ++i) minus[i] = a[i] ^ (int)0x80008000u;
    }
    sum(im, product) = mfma_split<P>(a, y.re, sum(im, product));
    behind(N + 2 * P);
    CCGLIB_PIN;
    sum(re, product) = mfma_split<P>(minus, y.im, sum(re, product));
    behind(N + 2 * P + 1);
    CCGLIB_PIN;
  });
#undef CCGLIB_PIN
}

// What a wave carries from one K iteration to the next: the split fragments of the last K
// tile, and its sums.
template <int TX> struct SplitState {
  SplitPair x[TX], y;
  SplitSum re[TX], im[TX];
};

// One K iteration of a wave with TX tiles of 32 x 32 side by side (1 or 2): reads the K tile
// of `slot` and splits it, a fragment at a time, behind the instructions of one tile, those
// of the K tile before among them (FIRST: there is none); its last tile's instructions
// follow in the next iteration, or in mma_split_last.
// A lane's 8 values of a row are its two 16-byte chunks (of either plane), or every other
// word of its four (IL: 128 bytes of pairs, off[2 h + u]).
template <int BX, int BY, int TX, bool IL, bool FIRST, typename Mid>
__device__ __forceinline__ void mma_step32_split(const char *slot, const int (&x_off)[4], const int (&y_off)[4],
                                                 SplitState<TX> &st, Mid &&mid) {
  static_assert(TX == 1 || TX == 2, "1 x 1 or 2 x 1 tiles");
  constexpr int ROW32 = 32 * (IL ? 128 : kTileRowBytes);
  struct Raw {
    float re[8], im[8];
  };
  auto rd = [&](const int (&off)[4], int extra, int plane_bytes) {
    Raw r;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const char *p = slot + (IL ? off[u] : off[u & 1] + (u >> 1) * plane_bytes) + extra;
      const float4_t v = *reinterpret_cast<const float4_t *>(p);
      if constexpr (IL) {
        r.re[2 * u] = v[0], r.re[2 * u + 1] = v[2], r.im[2 * u] = v[1], r.im[2 * u + 1] = v[3];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) (u < 2 ? r.re : r.im)[4 * (u & 1) + e] = v[e];
      }
    }
    return r;
  };
  auto rd_x = [&](int i) { return rd(x_off, i * ROW32, BX * kTileRowBytes); };
  auto rd_y = [&] { return rd(y_off, 0, BY * kTileRowBytes); };
  // step s of 8: the real part, then the imaginary one
  auto split = [](Raw &r, SplitPair &o, int s) {
    split_step(s < 4 ? r.re : r.im, s < 4 ? o.re : o.im, s & 3);
  };
  auto split_now = [&](Raw r, SplitPair &o) {
#pragma unroll
    for (int s = 0; s < 8; ++s) split(r, o, s);
    __builtin_amdgcn_sched_barrier(0);
  };
  // the split's eight steps behind instructions n0, n0 + 1, n0 + 3, n0 + 4, n0 + 6, ...
  auto split_behind = [&](Raw &r, SplitPair &o, int n, int n0) {
    if (n >= n0 && n < n0 + 12 && (n - n0) % 3 < 2) split(r, o, (n - n0) / 3 * 2 + (n - n0) % 3);
  };
  // (the raw values of a read are there by the time of the fourth instruction after it)
  SplitPair x_next, y_next;
  Raw raw = rd_x(0);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (FIRST) {
    split_now(raw, x_next);
    mid();
    split_now(rd_y(), y_next);
  } else {
    mma_split_tile(st.x[TX - 1], st.y, st.re[TX - 1], st.im[TX - 1], [&](int n) {
      if (n == 2) mid();
      split_behind(raw, x_next, n, 4);
      if (n == 16) raw = rd_y();
      split_behind(raw, y_next, n, 20);
    });
  }
  st.x[0] = x_next;
  st.y = y_next;
  if constexpr (TX == 2) {
    raw = rd_x(1);
    __builtin_amdgcn_sched_barrier(0);
    mma_split_tile(st.x[0], st.y, st.re[0], st.im[0], [&](int n) { split_behind(raw, st.x[1], n, 5); });
  }
}
// What is left after the last K iteration, and the sums as they belong into C; false where the
// wave has one that is not finite.
template <int TX>
__device__ __forceinline__ bool mma_split_last(SplitState<TX> &st, float16_t_ (&acc_re)[1][TX],
                                               float16_t_ (&acc_im)[1][TX]) {
  mma_split_tile(st.x[TX - 1], st.y, st.re[TX - 1], st.im[TX - 1], [](int) {});
  float check = 0.f;   // not zero as soon as one of the sums is not finite
#pragma unroll
  for (int i = 0; i < TX; ++i) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      acc_re[0][i][e] = (st.re[i].large[e] + st.re[i].small[e]) * kSplitUnscale;
      acc_im[0][i][e] = (st.im[i].large[e] + st.im[i].small[e]) * kSplitUnscale;
      check = __builtin_fmaf(acc_re[0][i][e], 0.f, check);
      check = __builtin_fmaf(acc_im[0][i][e], 0.f, check);
    }
  }
  if (__builtin_expect(!__any(check != 0.f), 1)) return true;
  // (an infinity's small products are NaN, the large ones infinite as a rule)
#pragma unroll
  for (int i = 0; i < TX; ++i) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      if (__builtin_isinf(st.re[i].large[e])) acc_re[0][i][e] = st.re[i].large[e];
      if (__builtin_isinf(st.im[i].large[e])) acc_im[0][i][e] = st.im[i].large[e];
    }
  }
  return false;
}

// Wide accesses to C at an address that is aligned to its elements only: rows of any
// length start anywhere, and global memory takes any alignment on this target. Element
// by element, every store instruction touches 64 lines for 4 bytes each: B=16 255x128x256
// bf16 with beta and rows of 255 took 30.2 us instead of 17.2, B=16 300x3001x577 fp16 to
// (re, im) rows of 3001 pairs 158.5 instead of 144.7 (with its transposes). (1-bit C is
// stored like this, but with beta still read element by element.)
typedef float4_t float4_any_t __attribute__((aligned(4)));
typedef int4_t int4_any_t __attribute__((aligned(2)));
typedef ushort4_t ushort4_any_t __attribute__((aligned(2)));
// A piece of C in an epilogue that writes whole cache lines at once. PAST (past_caches): a C of
// 256 MiB or more is not kept: what the caches would make room for by and by, whole lines in some other order,
// goes out as it comes. Us without and with it: B=16 2048x2048x1024 e4m3 282, 259; B=64 1024x1024x512 fp16 309, 259; B=32
// 1024x1024x512 e4m3 pairs 102, 84; with K = 8192 nothing. Of a smaller C the next kernel loses more than this one gains
// (kPastCachesBytes), and rows that share lines (B=176 629x4330x512 e4m3 1626, 3044) only cost.
// Four stores at a time: with the choice at every store planar C of 8 bits that does not take it was 1 to 2 %
// slower; with an epilogue each the 1-bit kernels spill.
template <typename Piece, bool PAST, typename Value>
__device__ __forceinline__ void store_c(void *at, const Value &v) {
  if constexpr (PAST) {
    // (the empty statements keep the compiler from making one ordinary store of the two)
    asm volatile("");
    __builtin_nontemporal_store((Piece)v, reinterpret_cast<Piece *>(at));
    asm volatile("");
  } else {
    *reinterpret_cast<Piece *>(at) = v;
  }
}
template <typename Store> __device__ __forceinline__ void store_four(bool past, Store &&store) {
  if (past) {
    static_for<4>([&](auto n) { store(n, std::true_type{}); });
  } else {
    static_for<4>([&](auto n) { store(n, std::false_type{}); });
  }
}

// The whole pieces of C of a wave tile, read before the sums are there (store_wave_tile): four real and four imaginary
// elements of planar C, eight as they lie of interleaved C.
struct NoPieces {};
template <int TOUT, int TX, int TY, int MS> struct CPieces {
  static constexpr int kPerRow = MS == 32 ? TX * 4 : TX;
  typename OutType<TOUT>::type v[TY][kPerRow][8];

  __device__ __forceinline__ void load(const KernelArgs &args, unsigned b, unsigned x_wave, unsigned y_wave, int lane) {
    using Tout = typename OutType<TOUT>::type;
    typedef Tout Vec4 __attribute__((ext_vector_type(4)));
    typedef Vec4 Piece __attribute__((aligned(sizeof(Tout))));
    const unsigned nx = args.nx, ny = args.ny;
    const Tout *cbase = reinterpret_cast<const Tout *>(args.c) + (size_t)b * 2 * nx * ny;
#pragma unroll
    for (int j = 0; j < TY; ++j) {
#pragma unroll
      for (int i = 0; i < kPerRow; ++i) {
        const unsigned y = y_wave + piece_y<MS>(j, i, lane), x = x_wave + piece_x<MS>(i, lane);
        if (y >= ny || x + 4 > nx) continue;
        const Tout *first = args.c_interleaved ? cbase + ((size_t)y * nx + x) * 2 : cbase + (size_t)y * nx + x;
        const Tout *second = args.c_interleaved ? first + 4 : first + (size_t)nx * ny;
        const Piece p = *reinterpret_cast<const Piece *>(first), q = *reinterpret_cast<const Piece *>(second);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][i][e] = p[e], v[j][i][4 + e] = q[e];
      }
    }
  }
};

// Epilogue of one wave: alpha * acc + beta * C, conversion, bounds-checked
// store, piece by piece (four consecutive elements of the contiguous C axis).
// pieces: the whole pieces of C if they have been read already (CPieces).
template <int TOUT, int TX, int TY, int MS = 16, int TILE0 = 0, typename Acc, typename Pieces = NoPieces>
__device__ __forceinline__ void store_wave_tile(const KernelArgs &args, unsigned b, unsigned x_wave,
                                                unsigned y_wave, int lane, const Acc &acc_re,
                                                const Acc &acc_im, const Pieces &pieces = {}) {
  constexpr bool READ = !std::is_same<Pieces, NoPieces>::value;
  // TX, TY count MFMA tiles; pieces per tile row: 1 (MS 16) or 4 (MS 32)
  constexpr int NPX = MS == 32 ? TX * 4 : TX;
  using Tout = typename OutType<TOUT>::type;
  const unsigned nx = args.nx, ny = args.ny;
  const bool have_alpha = args.have_alpha, have_beta = args.have_beta;
  const float ar = args.alpha_re, ai = args.alpha_im, br = args.beta_re, bi = args.beta_im;
  Tout *cbase = reinterpret_cast<Tout *>(args.c) + (size_t)b * 2 * nx * ny;
#pragma unroll
  for (int j = 0; j < TY; ++j) {
#pragma unroll
    for (int i = 0; i < NPX; ++i) {
      const unsigned y = y_wave + piece_y<MS>(j, i, lane);
      const unsigned x = x_wave + piece_x<MS>(i, lane);
      if (y >= ny || x >= nx) continue;
      float re[4], im[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        re[e] = piece_elem<MS, TILE0>(acc_re, j, i, e);
        im[e] = piece_elem<MS, TILE0>(acc_im, j, i, e);
        if (have_alpha) {
          const float r0 = re[e];
          re[e] = alpha_times_re(ar, ai, r0, im[e]);
          im[e] = alpha_times_im(ar, ai, r0, im[e]);
        }
      }
      const bool full = x + 4 <= nx;
      if (!args.c_interleaved) {
        Tout *pr = cbase + (size_t)y * nx + x;
        Tout *pi = pr + (size_t)nx * ny;
        if (have_beta) {
          // (whole pieces: C comes in with one wide load per plane)
          Tout cr4[4], ci4[4];
          if constexpr (READ) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              cr4[e] = pieces.v[j][i][e];
              ci4[e] = pieces.v[j][i][4 + e];
            }
          } else if (full) {
            typedef Tout Vec __attribute__((ext_vector_type(4)));
            typedef Vec Piece __attribute__((aligned(sizeof(Tout))));
            const Piece vr = *reinterpret_cast<const Piece *>(pr), vi = *reinterpret_cast<const Piece *>(pi);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              cr4[e] = vr[e];
              ci4[e] = vi[e];
            }
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (full || x + e < nx) {
              const float cr = full ? (float)cr4[e] : (float)pr[e];
              const float ci = full ? (float)ci4[e] : (float)pi[e];
              re[e] += br * cr - bi * ci;
              im[e] += bi * cr + br * ci;
            }
          }
        }
        if (full) {
          if constexpr (TOUT == kFloat32) {
            *reinterpret_cast<float4_any_t *>(pr) = float4_t{re[0], re[1], re[2], re[3]};
            *reinterpret_cast<float4_any_t *>(pi) = float4_t{im[0], im[1], im[2], im[3]};
          } else {
            Tout r4[4] = {(Tout)re[0], (Tout)re[1], (Tout)re[2], (Tout)re[3]};
            Tout i4[4] = {(Tout)im[0], (Tout)im[1], (Tout)im[2], (Tout)im[3]};
            *reinterpret_cast<ushort4_any_t *>(pr) = __builtin_bit_cast(ushort4_t, r4);
            *reinterpret_cast<ushort4_any_t *>(pi) = __builtin_bit_cast(ushort4_t, i4);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (x + e < nx) {
              pr[e] = (Tout)re[e];
              pi[e] = (Tout)im[e];
            }
          }
        }
      } else {
        Tout *p = cbase + ((size_t)y * nx + x) * 2;
        if (have_beta) {
          Tout c8[8];
          if constexpr (READ) {
#pragma unroll
            for (int e = 0; e < 8; ++e) c8[e] = pieces.v[j][i][e];
          } else if (full) {
            typedef Tout Vec __attribute__((ext_vector_type(8)));
            typedef Vec Piece __attribute__((aligned(sizeof(Tout))));
            const Piece v = *reinterpret_cast<const Piece *>(p);
#pragma unroll
            for (int e = 0; e < 8; ++e) c8[e] = v[e];
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (full || x + e < nx) {
              const float cr = full ? (float)c8[2 * e] : (float)p[2 * e];
              const float ci = full ? (float)c8[2 * e + 1] : (float)p[2 * e + 1];
              re[e] += br * cr - bi * ci;
              im[e] += bi * cr + br * ci;
            }
          }
        }
        if (full) {
          if constexpr (TOUT == kFloat32) {
            reinterpret_cast<float4_any_t *>(p)[0] = float4_t{re[0], im[0], re[1], im[1]};
            reinterpret_cast<float4_any_t *>(p)[1] = float4_t{re[2], im[2], re[3], im[3]};
          } else {
            Tout v8[8] = {(Tout)re[0], (Tout)im[0], (Tout)re[1], (Tout)im[1],
                          (Tout)re[2], (Tout)im[2], (Tout)re[3], (Tout)im[3]};
            *reinterpret_cast<int4_any_t *>(p) = __builtin_bit_cast(int4_t, v8);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (x + e < nx) {
              p[2 * e] = (Tout)re[e];
              p[2 * e + 1] = (Tout)im[e];
            }
          }
        }
      }
    }
  }
}

// One row of a 32-bit operand in global memory, four values of K at a time.
template <int LOADER> struct RowF32 {
  static constexpr bool kPairs = (LOADER == kLoadInterleavedVec || LOADER == kLoadInterleavedRagged);
  static constexpr unsigned kStep = LOADER == kLoadTiled ? kTileBytes : kPairs ? 128 : kTileRowBytes;
  const char *p;    // K tile 0
  size_t second;    // from the real values to the imaginary ones (pairs: to the second two)
  unsigned k;       // values in whole K tiles, and all
  unsigned k_all;

  // `rows` of them from `base` on; one past the end is read as the last one
  __device__ RowF32(const KernelArgs &args, const char *base, unsigned rows, unsigned row) {
    if constexpr (LOADER == kLoadTiled) {
      rows = (rows + kTileRows - 1) / kTileRows * kTileRows;
    }
    row = row < rows ? row : rows - 1;
    k_all = args.k;
    if constexpr (LOADER == kLoadTiled) {
      p = base + (size_t)(row / kTileRows) * args.k_tiles * kTileBytes + row % kTileRows * kTileRowBytes;
      second = kTilePlaneBytes;
      k = k_all = args.k_tiles * 16;
    } else {
      p = base + (size_t)row * (kPairs ? 2 : 1) * args.row_stride_bytes;
      second = kPairs ? 16 : (size_t)rows * args.row_stride_bytes;
      k = k_all / 16 * 16;
    }
  }
  // values 4 c ... of K tile kt, of which the row has all sixteen
  __device__ void get(unsigned kt, int c, float4_t &re, float4_t &im) const {
    const char *q = p + (size_t)kt * kStep + c * (kPairs ? 32 : 16);
    const float4_t u = *reinterpret_cast<const float4_any_t *>(q);
    const float4_t v = *reinterpret_cast<const float4_any_t *>(q + second);
    if constexpr (kPairs) {
      re = float4_t{u[0], u[2], v[0], v[2]};
      im = float4_t{u[1], u[3], v[1], v[3]};
    } else {
      re = u;
      im = v;
    }
  }
  // ... and of the last K tile, which it has in part
  __device__ void get_end(int c, float4_t &re, float4_t &im) const {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const unsigned at = k + 4 * c + e;
      const float *q = reinterpret_cast<const float *>(p) + (kPairs ? 2 * (size_t)at : (size_t)at);
      re[e] = at < k_all ? q[0] : 0.f;
      im[e] = at < k_all ? q[kPairs ? 1 : second / 4] : 0.f;
    }
  }
};

// The lane, counted where this is called: what follows from it is then worked out there as well, and
// not before the K loop, across which no register is left to keep it.
__device__ __forceinline__ int lane_here() {
  unsigned none = 0;
  asm volatile("" : "+s"(none));
  return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, none));
}

// Which of 16 rows of an operand from row0 on hold a NaN (a bit each), read by the wave until all of
// `wanted` have been found to.
template <int LOADER>
__device__ __forceinline__ unsigned nan_rows(const KernelArgs &args, const char *base, unsigned rows, unsigned row0,
                                             int lane, unsigned wanted) {
  const RowF32<LOADER> row(args, base, rows, row0 + (lane >> 2));
  const bool mine = (wanted >> (lane >> 2)) & 1;
  bool nan = false;
  float4_t re, im;
  auto look = [&] {
#pragma unroll
    for (int e = 0; e < 4; ++e) nan |= __builtin_isunordered(re[e], im[e]);
  };
  auto of_row = [&] { return ((__ballot(nan) >> (lane & ~3)) & 15) != 0; };
  for (unsigned kt = 0; kt < row.k / 16 && __any(mine && !of_row()); kt += 8) {
    float4_t r8[8], i8[8];   // (sixteen loads under way at a time)
#pragma unroll
    for (unsigned u = 0; u < 8; ++u) row.get(kt + u < row.k / 16 ? kt + u : kt, lane & 3, r8[u], i8[u]);
#pragma unroll
    for (unsigned u = 0; u < 8; ++u) {
      re = r8[u];
      im = i8[u];
      look();
    }
  }
  if (row.k < row.k_all) {
    row.get_end(lane & 3, re, im);
    look();
  }
  const unsigned long long found = __ballot(of_row());
  unsigned bits = 0;
#pragma unroll
  for (int r = 0; r < 16; ++r) bits |= (unsigned)((found >> (4 * r)) & 1) << r;
  return bits;
}

// Whether all sums of a wave's tile (32-bit input, TX MFMA tiles side by side) that are not finite are
// those of a row with a NaN. They are NaN then, in the split sums as on the fp32 instructions. (A sum that
// is infinite is not, and the rows need no look.)
template <int LOADER, int TX>
__device__ __forceinline__ bool only_nan_rows(const KernelArgs &args, unsigned b, unsigned x_wave, unsigned y_wave,
                                              int lane, const float16_t_ (&acc_re)[1][TX],
                                              const float16_t_ (&acc_im)[1][TX]) {
  const char *x = args.x + (size_t)b * args.x_batch_bytes, *y = args.y + (size_t)b * args.y_batch_bytes;
  const bool y_inside = y_wave + (lane & 31) < args.ny;
  unsigned bad[TX];   // bit e: element e of a tile (x = 8 (e / 4) + 4 (lane / 32) + e % 4) is not finite
  bool infinite = false;
#pragma unroll
  for (int i = 0; i < TX; ++i) {
    bad[i] = 0;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const unsigned at = x_wave + 32 * i + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
      const float re = acc_re[0][i][e], im = acc_im[0][i][e];
      const bool finite = __builtin_isfinite(re) && __builtin_isfinite(im), inside = y_inside && at < args.nx;
      bad[i] |= (unsigned)(!finite && inside) << e;
      infinite |= inside && (__builtin_isinf(re) || __builtin_isinf(im));
    }
  }
  if (__any(infinite)) return false;
  // rows of X without a finite sum
#pragma unroll
  for (int i = 0; i < TX; ++i) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (!__any((bad[i] >> (8 * h)) & 0xff)) continue;
      unsigned wanted = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const unsigned long long none = __ballot(((bad[i] >> (8 * h + e)) & 1) || !y_inside);
        const int bit = 8 * (e >> 2) + (e & 3);
        wanted |= (unsigned)((unsigned)none == ~0u) << bit | (unsigned)((unsigned)(none >> 32) == ~0u) << (bit + 4);
      }
      if (wanted == 0) continue;
      const unsigned nan = nan_rows<LOADER>(args, x, args.nx, x_wave + 32 * i + 16 * h, lane, wanted);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const unsigned mine = (nan >> (8 * (e >> 2) + 4 * (lane >> 5) + (e & 3))) & 1;
        bad[i] &= ~(mine << (8 * h + e));
      }
    }
  }
  auto left = [&] {
    unsigned any = 0;
#pragma unroll
    for (int i = 0; i < TX; ++i) any |= bad[i];
    return any != 0;
  };
  // rows of Y with one that is not explained yet
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const unsigned long long m = __ballot(left());
    const unsigned wanted = ((unsigned)(m | (m >> 32)) >> (16 * h)) & 0xffff;
    if (wanted == 0) continue;
    const unsigned nan = nan_rows<LOADER>(args, y, args.ny, y_wave + 16 * h, lane, wanted);
    if (((lane >> 4) & 1) == h && ((nan >> (lane & 15)) & 1)) {
#pragma unroll
      for (int i = 0; i < TX; ++i) bad[i] = 0;
    }
  }
  return !__any(left());
}

// A wave's tile of 32-bit input on the fp32 instructions, straight from global memory, one
// 32 x 32 tile at a time: for tiles whose split sums are not finite for another reason than a NaN
// among the operands (mma_step32_split).
template <int TOUT, int LOADER, int TX, int TY>
__device__ __forceinline__ void recompute_f32(const KernelArgs &args, unsigned b, unsigned x_wave,
                                              unsigned y_wave, int lane) {
  struct Four {
    float4_t xr, xi, yr, yi;
  };
  for (int t = 0; t < TX * TY; ++t) {
    const unsigned x0 = x_wave + 32 * (t % TX), y0 = y_wave + 32 * (t / TX);
    const RowF32<LOADER> x(args, args.x + (size_t)b * args.x_batch_bytes, args.nx, x0 + (lane & 31));
    const RowF32<LOADER> y(args, args.y + (size_t)b * args.y_batch_bytes, args.ny, y0 + (lane & 31));
    float16_t_ re[1][1], im[1][1];
    re[0][0] = 0.f;
    im[0][0] = 0.f;
    auto multiply = [&](const Four &f) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        re[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(f.xr[e], f.yr[e], re[0][0], 0, 0, 0);
        im[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(f.xr[e], f.yi[e], im[0][0], 0, 0, 0);
        re[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(f.xi[e], -f.yi[e], re[0][0], 0, 0, 0);
        im[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(f.xi[e], f.yr[e], im[0][0], 0, 0, 0);
      }
    };
    // (half a K tile is read while the one before is multiplied)
    auto get = [&](unsigned half) {
      Four f;
      x.get(half >> 1, (lane >> 5) + 2 * (half & 1), f.xr, f.xi);
      y.get(half >> 1, (lane >> 5) + 2 * (half & 1), f.yr, f.yi);
      return f;
    };
    const unsigned halves = x.k / 8;
    if (halves != 0) {
      Four now = get(0);
#pragma unroll 1
      for (unsigned n = 1; n < halves; ++n) {
        const Four next = get(n);
        multiply(now);
        now = next;
      }
      multiply(now);
    }
    if (x.k < x.k_all) {
#pragma unroll 1
      for (int s = 0; s < 2; ++s) {
        Four f;
        x.get_end((lane >> 5) + 2 * s, f.xr, f.xi);
        y.get_end((lane >> 5) + 2 * s, f.yr, f.yi);
        multiply(f);
      }
    }
    store_wave_tile<TOUT, 1, 1, 32>(args, b, x0, y0, lane, re, im);
  }
}

// Epilogue of the 1-bit GEMM on the MFMA path: the accumulators hold exact
// integers (sums of +-1 products); alpha and beta are truncated to integers and
// everything wraps modulo 2^32, as in the popcount kernel.
template <int TX, int TY, int MS, typename Acc>
__device__ __forceinline__ void store_wave_tile_int32(const KernelArgs &args, unsigned b,
                                                      unsigned x_wave, unsigned y_wave, int lane,
                                                      const Acc &acc_re, const Acc &acc_im) {
  constexpr int NPX = MS == 32 ? TX * 4 : TX;
  const unsigned nx = args.nx, ny = args.ny;
  const unsigned ar = (unsigned)(int)args.alpha_re, ai = (unsigned)(int)args.alpha_im;
  const unsigned br = (unsigned)(int)args.beta_re, bi = (unsigned)(int)args.beta_im;
  const bool have_beta = args.have_beta;
  unsigned *cbase = reinterpret_cast<unsigned *>(args.c) + (size_t)b * 2 * nx * ny;
#pragma unroll
  for (int j = 0; j < TY; ++j) {
#pragma unroll
    for (int i = 0; i < NPX; ++i) {
      const unsigned y = y_wave + piece_y<MS>(j, i, lane);
      const unsigned x = x_wave + piece_x<MS>(i, lane);
      if (y >= ny || x >= nx) continue;
      unsigned re[4], im[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned sr = (unsigned)(int)piece_elem<MS>(acc_re, j, i, e);
        const unsigned si = (unsigned)(int)piece_elem<MS>(acc_im, j, i, e) - args.im_excess;
        re[e] = ar * sr - ai * si;
        im[e] = ai * sr + ar * si;
      }
      const bool full = x + 4 <= nx;
      if (!args.c_interleaved) {
        unsigned *pr = cbase + (size_t)y * nx + x, *pi = pr + (size_t)nx * ny;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (have_beta && x + e < nx) {
            const unsigned cr = pr[e], ci = pi[e];
            re[e] += br * cr - bi * ci;
            im[e] += bi * cr + br * ci;
          }
        }
        if (full) {
          *reinterpret_cast<int4_any_t *>(pr) = int4_t{(int)re[0], (int)re[1], (int)re[2], (int)re[3]};
          *reinterpret_cast<int4_any_t *>(pi) = int4_t{(int)im[0], (int)im[1], (int)im[2], (int)im[3]};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (x + e < nx) {
              pr[e] = re[e];
              pi[e] = im[e];
            }
          }
        }
      } else {
        unsigned *p = cbase + ((size_t)y * nx + x) * 2;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (have_beta && x + e < nx) {
            const unsigned cr = p[2 * e], ci = p[2 * e + 1];
            re[e] += br * cr - bi * ci;
            im[e] += bi * cr + br * ci;
          }
        }
        if (full) {
          reinterpret_cast<int4_any_t *>(p)[0] = int4_t{(int)re[0], (int)im[0], (int)re[1], (int)im[1]};
          reinterpret_cast<int4_any_t *>(p)[1] = int4_t{(int)re[2], (int)im[2], (int)re[3], (int)im[3]};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (x + e < nx) {
              p[2 * e] = re[e];
              p[2 * e + 1] = im[e];
            }
          }
        }
      }
    }
  }
}

// Epilogue of the exchanged-roles layout (kAcc16T) for the common case (planar
// C, beta = 0, wave tile entirely inside C): register e of
// the four tiles of a tile row are four consecutive x, so a lane writes 16 bytes
// (8 for fp16 / bf16 C) and a store instruction four whole 256-byte row segments,
// straight from the accumulators.
template <int TOUT, int TY>
__device__ __forceinline__ void store_wave_tile_rows(const KernelArgs &args, unsigned b,
                                                     unsigned x_wave, unsigned y_wave, int lane,
                                                     float4_t (&acc_re)[TY][4],
                                                     float4_t (&acc_im)[TY][4]) {
  using Tout = typename OutType<TOUT>::type;
  const unsigned nx = args.nx, ny = args.ny;
  const bool past = TOUT == kFloat32 && past_caches(args);
  const bool have_alpha = args.have_alpha;
  const float ar = args.alpha_re, ai = args.alpha_im;
  Tout *out = reinterpret_cast<Tout *>(args.c) + (size_t)b * 2 * nx * ny +
              (size_t)(y_wave + (lane >> 4) * 4) * nx + x_wave + (lane & 15) * 4;
#pragma unroll
  for (int plane = 0; plane < 2; ++plane) {
#pragma unroll
    for (int j = 0; j < TY; ++j) {
      store_four(past, [&](auto n, auto past_them) {
        constexpr int e = n;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float re = acc_re[j][i][e], im = acc_im[j][i][e];
          v[i] = plane == 0 ? (have_alpha ? alpha_times_re(ar, ai, re, im) : re)
                            : (have_alpha ? alpha_times_im(ar, ai, re, im) : im);
        }
        Tout *p = out + (size_t)plane * nx * ny + (size_t)(j * 16 + e) * nx;
        if constexpr (TOUT == kFloat32) {
          store_c<float4_any_t, decltype(past_them)::value>(p, float4_t{v[0], v[1], v[2], v[3]});
        } else {
          Tout t[4] = {(Tout)v[0], (Tout)v[1], (Tout)v[2], (Tout)v[3]};
          *reinterpret_cast<ushort4_any_t *>(p) = __builtin_bit_cast(ushort4_t, t);
        }
      });
    }
  }
}

// Epilogue through LDS for the common case (planar fp32 C, beta = 0, wave tile
// entirely inside C, 64 columns wide): the accumulators of 16 rows are written
// to a wave-private LDS patch and read back row-wise, so that every store
// instruction writes four contiguous 256-byte row segments instead of sixteen
// 64-byte ones. `patch` is 16 rows of 272 bytes (the 16-byte pad keeps both
// the column-wise writes and the row-wise reads free of bank conflicts).
constexpr int kStagePatchBytes = 16 * 272;

template <int TX, int TY>
__device__ __forceinline__ void store_wave_tile_staged(const KernelArgs &args, unsigned b,
                                                       unsigned x_wave, unsigned y_wave, int lane,
                                                       char *patch, float4_t (&acc_re)[TY][TX],
                                                       float4_t (&acc_im)[TY][TX]) {
  static_assert(TX == 4, "patch rows hold 64 columns");
  const unsigned nx = args.nx, ny = args.ny;
  const bool past = past_caches(args);
  const bool have_alpha = args.have_alpha;
  const float ar = args.alpha_re, ai = args.alpha_im;
  float *cbase = reinterpret_cast<float *>(args.c) + (size_t)b * 2 * nx * ny;
  char *wr = patch + (lane & 15) * 272 + (lane >> 4) * 16;   // [y = lane%16][x = (lane/16)*4 ..]
  const char *rd = patch + (lane >> 4) * 272 + (lane & 15) * 16;  // [row lane/16][x = (lane%16)*4 ..]
  float *out = cbase + (size_t)(y_wave + (lane >> 4)) * nx + x_wave + (lane & 15) * 4;
#pragma unroll
  for (int plane = 0; plane < 2; ++plane) {
#pragma unroll
    for (int j = 0; j < TY; ++j) {
#pragma unroll
      for (int i = 0; i < TX; ++i) {
        float4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float re = acc_re[j][i][e], im = acc_im[j][i][e];
          v[e] = plane == 0 ? (have_alpha ? alpha_times_re(ar, ai, re, im) : re)
                            : (have_alpha ? alpha_times_im(ar, ai, re, im) : im);
        }
        *reinterpret_cast<float4_t *>(wr + i * 64) = v;
      }
      store_four(past, [&](auto n, auto past_them) {
        constexpr int r = n;
        const float4_t v = *reinterpret_cast<const float4_t *>(rd + r * 4 * 272);
        store_c<float4_any_t, decltype(past_them)::value>(
            out + (size_t)plane * nx * ny + (size_t)(j * 16 + r * 4) * nx, v);
      });
    }
  }
}

// The same for planar fp16 / bf16 C: a tile row of 16 x 64 values is 16 rows of
// 128 bytes (stride 144 in the patch: conflict-free 8-byte writes down a column,
// 16-byte aligned reads along a row); every store instruction writes eight whole
// 128-byte row segments instead of sixteen 32-byte pieces.
template <int TOUT, int TX, int TY>
__device__ __forceinline__ void store_wave_tile_staged_narrow(const KernelArgs &args, unsigned b,
                                                              unsigned x_wave, unsigned y_wave,
                                                              int lane, char *patch,
                                                              float4_t (&acc_re)[TY][TX],
                                                              float4_t (&acc_im)[TY][TX]) {
  static_assert(TX == 4, "patch rows hold 64 columns");
  using Tout = typename OutType<TOUT>::type;
  const unsigned nx = args.nx, ny = args.ny;
  const bool have_alpha = args.have_alpha;
  const float ar = args.alpha_re, ai = args.alpha_im;
  Tout *cbase = reinterpret_cast<Tout *>(args.c) + (size_t)b * 2 * nx * ny;
  char *wr = patch + (lane & 15) * 144 + (lane >> 4) * 8;        // [y = lane%16][x = (lane/16)*4 ..]
  const char *rd = patch + (lane >> 3) * 144 + (lane & 7) * 16;  // [row lane/8][x = (lane%8)*8 ..]
  Tout *out = cbase + (size_t)(y_wave + (lane >> 3)) * nx + x_wave + (lane & 7) * 8;
#pragma unroll
  for (int plane = 0; plane < 2; ++plane) {
#pragma unroll
    for (int j = 0; j < TY; ++j) {
#pragma unroll
      for (int i = 0; i < TX; ++i) {
        Tout v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float re = acc_re[j][i][e], im = acc_im[j][i][e];
          v[e] = (Tout)(plane == 0 ? (have_alpha ? alpha_times_re(ar, ai, re, im) : re)
                                   : (have_alpha ? alpha_times_im(ar, ai, re, im) : im));
        }
        *reinterpret_cast<ushort4_t *>(wr + i * 32) = __builtin_bit_cast(ushort4_t, v);
      }
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int4_t v = *reinterpret_cast<const int4_t *>(rd + r * 8 * 144);
        *reinterpret_cast<int4_any_t *>(out + (size_t)plane * nx * ny +
                                        (size_t)(j * 16 + r * 8) * nx) = v;
      }
    }
  }
}

// The same for interleaved fp32 C: 16 rows of 32 (re, im) pairs at a time (half
// the width of the wave tile, again 256 bytes per row) go through the patch.
template <int TX, int TY>
__device__ __forceinline__ void store_wave_tile_staged_il(const KernelArgs &args, unsigned b,
                                                          unsigned x_wave, unsigned y_wave, int lane,
                                                          char *patch, float4_t (&acc_re)[TY][TX],
                                                          float4_t (&acc_im)[TY][TX]) {
  static_assert(TX == 4, "two halves of 32 columns");
  const unsigned nx = args.nx, ny = args.ny;
  const bool have_alpha = args.have_alpha;
  const float ar = args.alpha_re, ai = args.alpha_im;
  float *cbase = reinterpret_cast<float *>(args.c) + (size_t)b * 2 * nx * ny;
  char *wr = patch + (lane & 15) * 272 + (lane >> 4) * 32;   // [y = lane%16][pair (lane/16)*4 ..]
  const char *rd = patch + (lane >> 4) * 272 + (lane & 15) * 16;  // [row lane/16][pairs 2 (lane%16) ..]
  float *out = cbase + ((size_t)(y_wave + (lane >> 4)) * nx + x_wave) * 2 + (lane & 15) * 4;
#pragma unroll
  for (int j = 0; j < TY; ++j) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 2 * h; i < 2 * h + 2; ++i) {
        float re[4], im[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float r0 = acc_re[j][i][e], i0 = acc_im[j][i][e];
          re[e] = have_alpha ? alpha_times_re(ar, ai, r0, i0) : r0;
          im[e] = have_alpha ? alpha_times_im(ar, ai, r0, i0) : i0;
        }
        char *w = wr + (i - 2 * h) * 128;
        *reinterpret_cast<float4_t *>(w) = float4_t{re[0], im[0], re[1], im[1]};
        *reinterpret_cast<float4_t *>(w + 16) = float4_t{re[2], im[2], re[3], im[3]};
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float4_t v = *reinterpret_cast<const float4_t *>(rd + r * 4 * 272);
        *reinterpret_cast<float4_any_t *>(out + ((size_t)(j * 16 + r * 4) * nx + h * 32) * 2) = v;
      }
    }
  }
}

// The same for the 32-row MFMA layout: one 32 x 32 tile at a time goes through
// a patch of 32 rows of 144 bytes (128 + 16 of padding), and every store
// instruction writes eight whole 128-byte row segments.
constexpr int kStagePatch32Bytes = 32 * 144;

template <int TX, int TY, bool INT = false>
__device__ __forceinline__ void store_wave_tile_staged32(const KernelArgs &args, unsigned b,
                                                         unsigned x_wave, unsigned y_wave, int lane,
                                                         char *patch, float16_t_ (&acc_re)[TY][TX],
                                                         float16_t_ (&acc_im)[TY][TX]) {
  const unsigned nx = args.nx, ny = args.ny;
  const bool past = past_caches(args);
  const bool have_alpha = args.have_alpha;
  const float ar = args.alpha_re, ai = args.alpha_im;
  float *cbase = reinterpret_cast<float *>(args.c) + (size_t)b * 2 * nx * ny;
  char *wr = patch + (lane & 31) * 144 + (lane >> 5) * 16;        // [y = lane%32][x = 8k + 4 (lane/32) ..]
  const char *rd = patch + (lane >> 3) * 144 + (lane & 7) * 16;   // [row lane/8 (+8q)][x = 4 (lane%8) ..]
  float *out = cbase + (size_t)(y_wave + (lane >> 3)) * nx + x_wave + (lane & 7) * 4;
#pragma unroll
  for (int plane = 0; plane < 2; ++plane) {
#pragma unroll
    for (int j = 0; j < TY; ++j) {
#pragma unroll
      for (int i = 0; i < TX; ++i) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float re = acc_re[j][i][4 * k + e], im = acc_im[j][i][4 * k + e];
            if constexpr (INT) {
              // exact integers; alpha truncated, arithmetic modulo 2^32
              const unsigned sr = (unsigned)(int)re, si = (unsigned)(int)im - args.im_excess;
              const unsigned iar = (unsigned)(int)ar, iai = (unsigned)(int)ai;
              const unsigned o = plane == 0 ? iar * sr - iai * si : iai * sr + iar * si;
              v[e] = __builtin_bit_cast(float, o);
            } else {
              v[e] = plane == 0 ? (have_alpha ? alpha_times_re(ar, ai, re, im) : re)
                                : (have_alpha ? alpha_times_im(ar, ai, re, im) : im);
            }
          }
          *reinterpret_cast<float4_t *>(wr + k * 32) = v;
        }
        store_four(past, [&](auto n, auto past_them) {
          constexpr int q = n;
          const float4_t v = *reinterpret_cast<const float4_t *>(rd + q * 8 * 144);
          store_c<float4_any_t, decltype(past_them)::value>(
              out + (size_t)plane * nx * ny + (size_t)(j * 32 + q * 8) * nx + i * 32, v);
        });
      }
    }
  }
}

// The same for 32-bit input, whose blocks have 4 KiB of a slot for each wave: no padding, the 16-byte
// chunks of the patch's 128-byte rows are XORed with the row (both ways free of bank conflicts). Planar C: a 32 x 32
// tile at a time; (re, im) pairs: half of one. A store instruction writes eight whole lines instead of
// 32 pieces of 32 or 64 bytes, us before and after: one K tile to planar C, 4096x4096x16 40.0, 37.5 (planar rows 41.2,
// 37.9); rows of C that start anywhere, 4001x3999x16 to pairs 46.3, 39.8, x64 81, 75. (Whole lines of
// pairs at longer K: between 2 % faster and 5 % slower, B=64 512x512x64 70.2, 74.5.)
constexpr int kStagePatchF32Bytes = 32 * 128;

template <int TX>
__device__ __forceinline__ void store_wave_tile_staged_f32(const KernelArgs &args, unsigned b, unsigned x_wave,
                                                           unsigned y_wave, int lane, char *patch,
                                                           const float16_t_ (&acc_re)[1][TX],
                                                           const float16_t_ (&acc_im)[1][TX]) {
  const unsigned nx = args.nx, ny = args.ny;
  const bool have_alpha = args.have_alpha;
  const float ar = args.alpha_re, ai = args.alpha_im;
  float *cbase = reinterpret_cast<float *>(args.c) + (size_t)b * 2 * nx * ny;
  auto write = [&](int chunk, float4_t v) {   // (row lane % 32 of the tile)
    *reinterpret_cast<float4_t *>(patch + (lane & 31) * 128 + (chunk ^ (lane & 7)) * 16) = v;
  };
  // rows lane / 8 + 8 q
  const char *rd = patch + (lane >> 3) * 128 + ((lane & 7) ^ (lane >> 3)) * 16;
  auto store = [&](float *out, size_t stride) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4_t v = *reinterpret_cast<const float4_t *>(rd + q * 8 * 128);
      *reinterpret_cast<float4_any_t *>(out + (size_t)(q * 8) * stride) = v;
    }
  };
  auto re_of = [&](int i, int e) {
    const float re = acc_re[0][i][e], im = acc_im[0][i][e];
    return have_alpha ? alpha_times_re(ar, ai, re, im) : re;
  };
  auto im_of = [&](int i, int e) {
    const float re = acc_re[0][i][e], im = acc_im[0][i][e];
    return have_alpha ? alpha_times_im(ar, ai, re, im) : im;
  };
  const size_t row = (size_t)(y_wave + (lane >> 3)) * nx + x_wave;
  if (args.c_interleaved) {
    float *out = cbase + 2 * row + (lane & 7) * 4;
#pragma unroll
    for (int i = 0; i < TX; ++i) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int e = 8 * h + 4 * k, chunk = 4 * k + 2 * (lane >> 5);
          write(chunk, float4_t{re_of(i, e), im_of(i, e), re_of(i, e + 1), im_of(i, e + 1)});
          write(chunk + 1, float4_t{re_of(i, e + 2), im_of(i, e + 2), re_of(i, e + 3), im_of(i, e + 3)});
        }
        store(out + 2 * (32 * i + 16 * h), 2 * (size_t)nx);
      }
    }
  } else {
    float *out = cbase + row + (lane & 7) * 4;
#pragma unroll
    for (int plane = 0; plane < 2; ++plane) {
#pragma unroll
      for (int i = 0; i < TX; ++i) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = plane == 0 ? re_of(i, 4 * k + e) : im_of(i, 4 * k + e);
          write(2 * k + (lane >> 5), v);
        }
        store(out + (size_t)plane * nx * ny + 32 * i, nx);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Register-staged kernel: global -> registers -> LDS, two LDS stages. Used for
// planar (basic) input whose rows are shorter than 16 bytes: its element-wise
// loads do the bounds checks and the zero fill.
// ---------------------------------------------------------------------------
template <int DT, int TOUT, int BX, int BY, int WX, int WY, int KT, int LOADER, int WAVES_PER_EU>
__global__ __launch_bounds__(64 * (BX / WX) * (BY / WY), WAVES_PER_EU) void complex_gemm_mfma(
    const KernelArgs args) {
  constexpr int NWX = BX / WX, NWY = BY / WY;
  constexpr int NTHREADS = 64 * NWX * NWY;
  constexpr int TX = WX / 16, TY = WY / 16;
  constexpr int KPM = DtypeTraits<DT>::kTilesPerMfma;
  constexpr int EB = DtypeTraits<DT>::kElemBytes;
  static_assert(KT % KPM == 0, "stage must hold whole MFMAs");
  constexpr int X_KTILE_BYTES = 2 * BX * kTileRowBytes;
  constexpr int Y_KTILE_BYTES = 2 * BY * kTileRowBytes;
  constexpr int KTILE_BYTES = X_KTILE_BYTES + Y_KTILE_BYTES;
  constexpr int STAGE_BYTES = KT * KTILE_BYTES;
  constexpr int X_CHUNKS = KT * 2 * BX * 4;
  constexpr int Y_CHUNKS = KT * 2 * BY * 4;
  static_assert(X_CHUNKS % NTHREADS == 0 && Y_CHUNKS % NTHREADS == 0, "chunks per thread");
  constexpr int CX = X_CHUNKS / NTHREADS, CY = Y_CHUNKS / NTHREADS;

  extern __shared__ __attribute__((aligned(16))) char lds[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wx = wave % NWX, wy = wave / NWX;

  const TileCoord tc = tile_coord(args, blockIdx.x);
  const unsigned b = tc.b, block_x = tc.block_x, block_y = tc.block_y;

  OperandView xv{args.x + (size_t)b * args.x_batch_bytes, args.nx, args.x_tiles, block_x * BX};
  OperandView yv{args.y + (size_t)b * args.y_batch_bytes, args.ny, args.y_tiles, block_y * BY};
  const unsigned k_tiles = args.k_tiles;
  const unsigned k_bytes = args.k_bytes;

  int4_t xs[CX], ys[CY];
  auto fetch = [&](unsigned kt0) {
#pragma unroll
    for (int i = 0; i < CX; ++i) {
      const int gidx = tid + i * NTHREADS;
      const int kk = gidx / (2 * BX * 4), rem = gidx % (2 * BX * 4);
      xs[i] = load_chunk<EB, LOADER>(xv, kt0 + kk, k_tiles, k_bytes, rem / (BX * 4),
                                     (rem / 4) % BX, rem % 4);
    }
#pragma unroll
    for (int i = 0; i < CY; ++i) {
      const int gidx = tid + i * NTHREADS;
      const int kk = gidx / (2 * BY * 4), rem = gidx % (2 * BY * 4);
      ys[i] = load_chunk<EB, LOADER>(yv, kt0 + kk, k_tiles, k_bytes, rem / (BY * 4),
                                     (rem / 4) % BY, rem % 4);
    }
  };
  auto stash = [&](int stage) {
    char *s = lds + stage * STAGE_BYTES;
#pragma unroll
    for (int i = 0; i < CX; ++i) {
      const int gidx = tid + i * NTHREADS;
      const int kk = gidx / (2 * BX * 4), rem = gidx % (2 * BX * 4);
      const int plane = rem / (BX * 4), row = (rem / 4) % BX, c = rem % 4;
      *reinterpret_cast<int4_t *>(s + kk * KTILE_BYTES + plane * BX * kTileRowBytes +
                                  swizzled_row_offset(row, c)) = xs[i];
    }
#pragma unroll
    for (int i = 0; i < CY; ++i) {
      const int gidx = tid + i * NTHREADS;
      const int kk = gidx / (2 * BY * 4), rem = gidx % (2 * BY * 4);
      const int plane = rem / (BY * 4), row = (rem / 4) % BY, c = rem % 4;
      *reinterpret_cast<int4_t *>(s + kk * KTILE_BYTES + X_KTILE_BYTES +
                                  plane * BY * kTileRowBytes + swizzled_row_offset(row, c)) =
          ys[i];
    }
  };

  float4_t acc_re[TY][TX], acc_im[TY][TX];
#pragma unroll
  for (int j = 0; j < TY; ++j) {
#pragma unroll
    for (int i = 0; i < TX; ++i) {
      acc_re[j][i] = float4_t{0.f, 0.f, 0.f, 0.f};
      acc_im[j][i] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
  }

  const int lane_off = swizzled_row_offset(lane & 15, lane >> 4);
  const int x_frag_off = (wx * WX) * kTileRowBytes + lane_off;
  const int y_frag_off = X_KTILE_BYTES + (wy * WY) * kTileRowBytes + lane_off;

  auto compute = [&](int stage) {
    const char *s = lds + stage * STAGE_BYTES;
#pragma unroll
    for (int kk = 0; kk < KT; kk += KPM) {
      const char *slot[KPM];
#pragma unroll
      for (int u = 0; u < KPM; ++u) slot[u] = s + (kk + u) * KTILE_BYTES;
      mma_step<DT, BX, BY, TX, TY>(slot, x_frag_off, y_frag_off, acc_re, acc_im, [] {});
    }
  };

  const unsigned stages = (k_tiles + KT - 1) / KT;
  fetch(0);
  stash(0);
  if (stages > 1) fetch(KT);
  __syncthreads();
  for (unsigned s = 0; s < stages; ++s) {
    const int cur = s & 1;
    if (s + 1 < stages) stash(cur ^ 1);
    if (s + 2 < stages) fetch((s + 2) * KT);
    compute(cur);
    __syncthreads();
  }

  store_wave_tile<TOUT, TX, TY>(args, b, block_x * BX + wx * WX, block_y * BY + wy * WY, lane,
                                acc_re, acc_im);
}

// ---------------------------------------------------------------------------
// Direct-to-LDS kernel for the tiled (opt) layout, and for planar input with
// 16-byte aligned rows (where each lane brings its own address instead of an
// offset into a contiguous tile). Operand tiles of the tiled layout are
// contiguous 16 KiB blocks; the copy into LDS needs no registers: every wave issues
// global_load_lds_dwordx4, each of which moves 16 rows x 64 bytes (1 KiB)
// straight into LDS. The hardware writes lane L's 16 bytes at LDS offset
// base + 16 L; the XOR swizzle of the LDS layout is obtained by letting lane L
// fetch the chunk that belongs there (a permutation inside each 64-byte row,
// so the global access stays fully coalesced).
//
// LDS is a ring of SLOTS K tiles (X and Y may have rings of different depth).
// Iteration i waits for its own tile with s_waitcnt vmcnt(n) - n being the
// loads issued for later iterations - then passes one barrier, issues the loads
// SLOTS - 1 iterations ahead into the slot that the previous iteration just
// released (after its first group of MFMAs), and does the math.
//
// Blocks are persistent: each walks a sequence of C tiles, and the copy simply
// runs on into the next C tile, so its first K tiles are in flight while the
// current tile's results are stored, and those stores drain under the next
// tile's math. Loads past the end of K (rows whose last K tile is partial) or
// past the last C tile are pointed at a zero tile, which keeps the number of
// outstanding loads the same in every iteration.
// ---------------------------------------------------------------------------
__device__ __attribute__((aligned(256))) char g_zero_tile[kTileBytes];

// READS: the wave's reads of LDS are waited for as well (their slot is refilled behind the barrier).
template <int N, bool READS = false> __device__ __forceinline__ void wait_vmcnt_then_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  if constexpr (READS) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
  }
}

// Both copy helpers write m0 (the LDS base of the copy) and say so in their
// clobber lists, so that the compiler never assumes a value it put there
// survives them; clang warns about any mention of m0 there, which is the point.
// The compiler does not look into an asm statement for the wait states its
// instructions need after what it placed in front of it: the scalar base of the
// first helper may have come out of a vector register right before (a spilled
// scalar register read back with v_readlane), and a vector memory instruction
// may read such a register five wait states later at the earliest. The helper
// therefore hands the base on through a scalar move: the scalar ALU may read the
// register at once, and what it writes the memory instruction may read at once.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_1k_to_lds(const char *base, unsigned lane_offset,
                                               unsigned lds_address) {
  unsigned long long base_here;
  asm volatile(
      "s_mov_b64 %0, %3\n\t"
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %2, %0"
      : "=&s"(base_here)
      : "s"(lds_address), "v"(lane_offset), "s"(base)
      : "memory", "m0");
}

// Same, with a full address per lane (planar layout: the 16 rows of a row block
// are not contiguous in memory).
__device__ __forceinline__ void load_1k_to_lds_by_lane(const char *lane_address,
                                                       unsigned lds_address) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off"
      :
      : "s"(lds_address), "v"(lane_address)
      : "memory", "m0");
}
#pragma clang diagnostic pop

#include "gemm_mfma_wide.h"

template <int DT, int TOUT, int BX, int BY, int WX, int WY, int SLOTS, int WAVES_PER_EU, int LOADER,
          int MS, bool XT, int XSLOTS, bool SKIP>
__global__ __launch_bounds__(64 * (BX / WX) * (BY / WY), WAVES_PER_EU) void complex_gemm_mfma_dtl(
    const KernelArgs args) {
  constexpr int NWX = BX / WX, NWY = BY / WY, NW = NWX * NWY;
  constexpr int TX = WX / MS, TY = WY / MS;          // MFMA tiles of a wave
  static_assert(MS == 32 || DtypeTraits<DT>::kTilesPerMfma == 1,
                "one K tile per iteration: fp8 input runs on the 32-row MFMA here");
  constexpr int KPM = 1;
  // interleaved operands: one plane of (re, im) rows
  // (their slots hold 128 bytes of every row, fetched as whole cache lines)
  constexpr bool IL = (LOADER == kLoadInterleavedVec || LOADER == kLoadInterleavedRagged);
  static_assert(MS == 16 || !IL || DtypeTraits<DT>::kElemBytes != 2,
                "interleaved operands on the 32-row MFMAs: 8- and 32-bit input");
  // rows that are no whole aligned 16-byte chunks, see chunk_source and settle_row_ends
  constexpr bool RAGGED = (LOADER == kLoadPlanarRagged || LOADER == kLoadInterleavedRagged);
  constexpr int PLANES = IL ? 1 : 2;
  constexpr int RB = IL ? 128 : kTileRowBytes;      // bytes of a row in one slot
  constexpr int RPB = 1024 / RB;                    // rows moved by one 1 KiB copy instruction
  constexpr int CPR = RB / 16;                      // 16-byte chunks per row
  constexpr int X_BYTES = PLANES * BX * RB, Y_BYTES = PLANES * BY * RB;
  constexpr int SLOT_BYTES = X_BYTES + Y_BYTES;
  // 1 KiB row blocks (16 rows x 64 bytes or 8 x 128) of the X and the Y part of a K tile
  constexpr int X_ROW_BLOCKS = X_BYTES / 1024, Y_ROW_BLOCKS = Y_BYTES / 1024;
  static_assert(X_ROW_BLOCKS % NW == 0 && Y_ROW_BLOCKS % NW == 0,
                "row blocks must divide evenly over the waves");
  constexpr int XL = X_ROW_BLOCKS / NW, YL = Y_ROW_BLOCKS / NW;   // loads per wave per K tile
  constexpr int LPW = XL + YL;
  // XT: the X fragments feed the "B" side of the 16-row MFMA and tile i of a wave
  // holds the columns x = 4 (lane % 16) + i of its 64, so that a lane ends up with
  // 16 consecutive bytes of four C rows per register index and the C stores need no
  // regrouping through LDS. For that, the rows of every 16-row block of X sit in
  // LDS in the order [4 a + (i ^ a)] <- row 4 a + i, with their 16-byte chunks XORed
  // with 3 (block & 1): fragment reads of rows 4 r + i are then free of bank
  // conflicts (measured), and a copy instruction still moves the contiguous 1 KiB.
  static_assert(!XT || (MS == 16 && TX == 4 && TY == 4 && !IL && WX == 64 && NW % 2 == 0 &&
                        (BX / 16) % 2 == 0),
                "exchanged roles: 16-row MFMA, 4 x 4 tiles per wave");
  // The ring. SLOTS K tiles of Y and XSLOTS >= SLOTS K tiles of X: X tiles are
  // requested XLEAD iterations before their use, Y tiles YLEAD iterations. With
  // equal counts a slot is [X | Y] as one piece of LDS; with more X slots the
  // two rings lie one after the other (X is then the operand to make the narrower
  // one: more of its K tiles fit, and a longer wait for memory is covered).
  static_assert(SLOTS >= 2 && XSLOTS >= SLOTS, "ring must hold at least two iterations");
  constexpr bool SPLIT = XSLOTS != SLOTS;
  constexpr int XLEAD = XSLOTS - 1, YLEAD = SLOTS - 1;
  // The counter of outstanding copies retires in order. In every iteration a wave
  // requests its Y blocks first and then its X blocks; the K tile of iteration k is
  // complete when nothing older than the last request for it is outstanding, which
  // leaves the requests of the YLEAD - 1 iterations since, and the X blocks that
  // followed Y(k) in its own iteration when X runs further ahead.
  constexpr int kOutstandingOk = (XLEAD > YLEAD ? XL : 0) + (YLEAD - 1) * LPW;
  static_assert(kOutstandingOk < 64, "vmcnt range");
  auto x_slot_off = [](unsigned s) { return SPLIT ? s * X_BYTES : s * SLOT_BYTES; };
  auto y_slot_off = [](unsigned s) {
    return SPLIT ? XSLOTS * X_BYTES + s * Y_BYTES : s * SLOT_BYTES + X_BYTES;
  };

  constexpr bool SMALL = BX == 64 && BY == 64 && DT != kFloat32;   // (see SmallTile)
  static_assert(!SMALL || TX * MS == 32, "waves of 32 x 32");

  extern __shared__ __attribute__((aligned(1024))) char lds[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wx = wave % NWX, wy = wave / NWX;
  // slots along K (the host counts 64-byte pieces of a row)
  const unsigned k_tiles = IL ? (args.k_tiles + 1) / 2 : args.k_tiles;
  const unsigned total = args.blocks_x * args.blocks_y * args.batch;
  // bytes of one operand row in memory (planar: one plane's row)
  const unsigned row_bytes = IL ? 2 * args.k_bytes : args.k_bytes;
  // ... and the distance between rows (larger when the launch covers a piece of K)
  const unsigned row_stride = IL ? 2 * args.row_stride_bytes : args.row_stride_bytes;

  // ---- this wave's share of the copy: XL + YL row blocks of every K tile --
  // Row block q of an operand's part of a K tile: re plane, im plane, 16 rows
  // each. What depends on the lane (its row and swizzled chunk inside the row
  // block) is the same for every C tile; the wave-uniform tile pointers are set
  // per C tile.
  const unsigned lane_off = (lane >> 2) * kTileRowBytes +
                            (((lane & 3) ^ (MS == 32 ? (lane >> 4) & 3 : (lane >> 3) & 3)) * 16);
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char *)lds;
  const int r = lane / CPR;                                   // row inside the row block
  // chunk that belongs at lane*16: the XOR pattern that makes the fragment
  // reads of the MFMA shape in use free of bank conflicts (measured)
  // (interleaved rows on the 32-row MFMAs: XOR with (row >> 1) & 7, which also
  // depends on the parity of the 8-row row block, see c_of below)
  const int c = (lane % CPR) ^ (IL ? r & 7 : MS == 32 ? (r >> 2) & 3 : (r >> 1) & 3);
  auto c_of = [&](int rb) {   // chunk this lane fetches for row block rb of an operand
    return (IL && MS == 32) ? ((lane % CPR) ^ (((rb & 1) << 2) | ((r >> 1) & 3))) : c;
  };
  // (XT) row and chunk this lane fetches of an X row block (a wave's X row blocks
  // all have the parity of the wave number)
  const int xt_row = 4 * (lane >> 4) + (((lane >> 2) & 3) ^ (lane >> 4));
  const int xt_chunk = (lane & 3) ^ (3 * (wave & 1));
  const unsigned lane_off_x = XT ? xt_row * kTileRowBytes + xt_chunk * 16 : lane_off;

  // One operand's side of the copy: where its next K tile comes from. The copy
  // walks the same sequence of C tiles as the math, X ahead of Y when its ring
  // is deeper; past the last C tile it re-reads the last one (never used).
  struct Stream {
    unsigned tile, kt;          // C tile and K tile of the request issued last
  };
  Stream xs{blockIdx.x, 0}, ys{blockIdx.x, 0};
  unsigned x_tile_off[XL], y_tile_off[YL];   // wave-uniform: the row block inside its operand tile
  unsigned x_lds[XL], y_lds[YL];             // wave-uniform: LDS byte address inside slot 0 of the ring
  const char *x_src[XL], *y_src[YL];         // wave-uniform: K tile 0 of the operand tile (tiled layout)
  // rows in place: this lane's chunk of K tile 0. The second half of a wave's row blocks are the
  // imaginary planes of the first half's rows (x_plane, y_plane bytes away).
  constexpr int XLS = IL || LOADER == kLoadTiled ? XL : XL / 2, YLS = IL || LOADER == kLoadTiled ? YL : YL / 2;
  static_assert(IL || ((BX / RPB) % NW == 0 && (BY / RPB) % NW == 0), "planes split a wave's row blocks evenly");
  const char *x_lane_src[XLS], *y_lane_src[YLS];
  const size_t x_plane = (size_t)args.nx * row_stride, y_plane = (size_t)args.ny * row_stride;
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int q = i * NW + wave, plane = q / (BX / RPB), rb = q % (BX / RPB);
    x_tile_off[i] = plane * kTilePlaneBytes + ((rb * RPB) % kTileRows) * kTileRowBytes;
    x_lds[i] = lds_base + x_slot_off(0) + q * 1024;
  }
#pragma unroll
  for (int i = 0; i < YL; ++i) {
    const int q = i * NW + wave, plane = q / (BY / RPB), rb = q % (BY / RPB);
    y_tile_off[i] = plane * kTilePlaneBytes + ((rb * RPB) % kTileRows) * kTileRowBytes;
    y_lds[i] = lds_base + y_slot_off(0) + q * 1024;
  }
  // Points one side of the copy at the operand tile of a C tile.
  auto point_x = [&](const TileCoord &tc) {
    const char *op = args.x + (size_t)tc.b * args.x_batch_bytes;
#pragma unroll
    for (int i = 0; i < XLS; ++i) {
      const int q = i * NW + wave, rb = q % (BX / RPB);
      const unsigned row0 = tc.block_x * BX + rb * RPB;
      if constexpr (LOADER == kLoadTiled) {
        unsigned tile = row0 / kTileRows;
        tile = tile < args.x_tiles ? tile : args.x_tiles - 1;   // rows past the end: never stored
        x_src[i] = op + (size_t)tile * args.k_tile_stride * kTileBytes;
        // (a block lower than an operand tile starts inside it)
        if constexpr (BX < kTileRows) x_src[i] += (tc.block_x * BX) % kTileRows * kTileRowBytes;
      } else {
        unsigned row = row0 + (XT ? xt_row : r);
        row = row < args.nx ? row : args.nx - 1;   // likewise
        x_lane_src[i] = op + (size_t)row * row_stride + (XT ? xt_chunk : c_of(rb)) * 16;
      }
    }
  };
  auto point_y = [&](const TileCoord &tc) {
    const char *op = args.y + (size_t)tc.b * args.y_batch_bytes;
#pragma unroll
    for (int i = 0; i < YLS; ++i) {
      const int q = i * NW + wave, rb = q % (BY / RPB);
      const unsigned row0 = tc.block_y * BY + rb * RPB;
      if constexpr (LOADER == kLoadTiled) {
        unsigned tile = row0 / kTileRows;
        tile = tile < args.y_tiles ? tile : args.y_tiles - 1;
        y_src[i] = op + (size_t)tile * args.k_tile_stride * kTileBytes;
        // (a block lower than an operand tile starts inside it)
        if constexpr (BY < kTileRows) y_src[i] += (tc.block_y * BY) % kTileRows * kTileRowBytes;
      } else {
        unsigned row = row0 + r;
        row = row < args.ny ? row : args.ny - 1;
        y_lane_src[i] = op + (size_t)row * row_stride + c_of(rb) * 16;
      }
    }
  };
  // Where a lane's chunk of K tile kt comes from when it lies at `src` in K tile 0 of its row
  // (of the plane `plane` bytes away).
  // Rows of whole chunks: it is either inside K or reads zeros. Ragged rows: the chunk
  // that holds the end of the row is fetched as the last 16 bytes of the row instead
  // (nothing outside the row is touched): its elements lie at the chunk's end and
  // in front of them, once more, some that the chunk before holds, until
  // settle_row_ends puts them right.
  auto chunk_source = [&](const char *src, unsigned kt, int chunk, size_t plane) {
    // (the end of a chunk may lie 4 GiB behind the row's start, and its 32-bit offset be 0)
    const unsigned start = kt * RB + chunk * 16;
    plane += (size_t)kt * RB;
    if constexpr (RAGGED) {
      const unsigned left = row_bytes - start;
      return start < row_bytes ? src + plane - (left < 16 ? 16 - left : 0) : g_zero_tile + lane * 16;
    } else {
      // (by its last byte: with `start` the compiler puts the copies of 16-bit pairs in front of
      // the products, B=3 22x512x608 10.3 -> 10.9 us)
      return start + 15 < row_bytes ? src + plane : g_zero_tile + lane * 16;
    }
  };
  // issue_*: straight-line code (it is placed between MFMAs, and a branch there
  // would let the compiler sink those MFMAs below it); advance_*: the
  // bookkeeping, with the branches of the tile change.
  auto issue_x = [&](unsigned slot) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const unsigned dst = x_lds[i] + (x_slot_off(slot) - x_slot_off(0));
      if constexpr (LOADER == kLoadTiled) {
        load_1k_to_lds(x_src[i] + (size_t)xs.kt * kTileBytes + x_tile_off[i], lane_off_x, dst);
      } else {
        const int q = i * NW + wave, rb = q % (BX / RPB);
        load_1k_to_lds_by_lane(
            chunk_source(x_lane_src[i % XLS], xs.kt, XT ? xt_chunk : c_of(rb), i < XLS ? 0 : x_plane), dst);
      }
    }
  };
  auto issue_y = [&](unsigned slot) {
#pragma unroll
    for (int i = 0; i < YL; ++i) {
      const unsigned dst = y_lds[i] + (y_slot_off(slot) - y_slot_off(0));
      if constexpr (LOADER == kLoadTiled) {
        load_1k_to_lds(y_src[i] + (size_t)ys.kt * kTileBytes + y_tile_off[i], lane_off, dst);
      } else {
        const int q = i * NW + wave, rb = q % (BY / RPB);
        load_1k_to_lds_by_lane(chunk_source(y_lane_src[i % YLS], ys.kt, c_of(rb), i < YLS ? 0 : y_plane), dst);
      }
    }
  };
  auto advance_x = [&] {
    if (++xs.kt == k_tiles) {
      xs.kt = 0;
      xs.tile += gridDim.x;
      if (xs.tile < total) point_x(tile_coord(args, xs.tile));
    }
  };
  auto advance_y = [&] {
    if (++ys.kt == k_tiles) {
      ys.kt = 0;
      ys.tile += gridDim.x;
      if (ys.tile < total) point_y(tile_coord(args, ys.tile));
    }
  };
  // both, with one look at the coordinates (X and Y walk together unless their rings differ)
  auto advance = [&] {
    if constexpr (SPLIT) {
      advance_y();
      advance_x();
    } else if (++xs.kt == k_tiles) {
      xs.kt = ys.kt = 0;
      xs.tile = ys.tile = xs.tile + gridDim.x;
      if (xs.tile < total) {
        const TileCoord tc = tile_coord(args, xs.tile);
        point_y(tc);
        point_x(tc);
      }
    } else {
      ys.kt = xs.kt;
    }
  };

  // (RAGGED) Shifts the last elements of every row of both operands, which lie at the end of
  // the row's last chunk, to its front and clears the rest: the slots then hold what the
  // tiled layout holds. Once per C tile, between the barrier that says that its last K
  // tile has landed and a second one.
  auto settle_row_ends = [&](unsigned x_in, unsigned y_in) {
    const unsigned shift = 8 * (16 - row_bytes % 16), chunk = row_bytes / 16 % CPR;
    for (unsigned t = threadIdx.x; t < (unsigned)(PLANES * (BX + BY)); t += 64 * NW) {
      const bool of_y = t >= (unsigned)(PLANES * BX);
      const unsigned row = of_y ? t - PLANES * BX : t;   // (row of LDS; planes follow each other)
      // the chunk's place: the swizzles of the copies above
      const unsigned at = IL ? (MS == 32 ? (((row >> 3) & 1) << 2) | ((row >> 1) & 3) : row & 7)
                          : XT && !of_y ? 3 * ((row >> 4) & 1)
                          : MS == 32    ? (row >> 2) & 3
                                        : (row >> 1) & 3;
      typedef unsigned long long ulong2_t __attribute__((ext_vector_type(2)));
      ulong2_t *p = reinterpret_cast<ulong2_t *>(lds + (of_y ? y_slot_off(y_in) : x_slot_off(x_in)) +
                                                 row * RB + (chunk ^ at) * 16);
      const ulong2_t v = *p;
      *p = shift >= 64 ? ulong2_t{v[1] >> (shift - 64), 0ull}
                       : ulong2_t{(v[0] >> shift) | (v[1] << (64 - shift)), v[1] >> shift};
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

  const int frag_lane_off = swizzled_row_offset(lane & 15, lane >> 4);
  const int x_frag_off = (wx * WX) * kTileRowBytes + frag_lane_off;
  const int y_frag_off = X_BYTES + (wy * WY) * kTileRowBytes + frag_lane_off;
  int xo[4];   // X fragment of tile i (16-row MFMA)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r16 = lane & 15, g = lane >> 4;
    xo[i] = XT ? (wx * WX + 4 * r16 + (i ^ (r16 & 3))) * kTileRowBytes +
                     ((g ^ (3 * ((r16 >> 2) & 1))) * 16)
               : x_frag_off + i * 16 * kTileRowBytes;
  }
  // 32-row MFMA: row lane % 32, chunks lane / 32 and lane / 32 + 2 (any split
  // of K over the lanes is fine as long as X and Y use the same one)
  const int row32 = lane & 31, sw32 = (row32 >> 2) & 3;
  const int frag32_off[2] = {row32 * kTileRowBytes + (((lane >> 5) ^ sw32) * 16),
                             row32 * kTileRowBytes + ((((lane >> 5) | 2) ^ sw32) * 16)};
  const int x32_off[2] = {(wx * WX) * kTileRowBytes + frag32_off[0],
                          (wx * WX) * kTileRowBytes + frag32_off[1]};
  const int y32_off[2] = {X_BYTES + (wy * WY) * kTileRowBytes + frag32_off[0],
                          X_BYTES + (wy * WY) * kTileRowBytes + frag32_off[1]};
  // interleaved rows of 128 bytes: row lane % 16, chunks lane / 16 and lane / 16 + 4
  const int il_row = lane & 15;
  const int il_off[2] = {il_row * 128 + (((lane >> 4) ^ (il_row & 7)) * 16),
                         il_row * 128 + ((((lane >> 4) | 4) ^ (il_row & 7)) * 16)};
  const int xil_off[2] = {(wx * WX) * 128 + il_off[0], (wx * WX) * 128 + il_off[1]};
  const int yil_off[2] = {X_BYTES + (wy * WY) * 128 + il_off[0],
                          X_BYTES + (wy * WY) * 128 + il_off[1]};
  // interleaved rows on the 32-row MFMAs: row lane % 32, half h of the 128 bytes, chunks
  // 4 h + 2 (lane / 32) and the next one
  int xil32_off[2][2], yil32_off[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int row = lane & 31, chunk = 4 * h + 2 * (lane >> 5) + u;
      const int off = row * 128 + ((chunk ^ ((row >> 1) & 7)) * 16);
      xil32_off[h][u] = (wx * WX) * 128 + off;
      yil32_off[h][u] = X_BYTES + (wy * WY) * 128 + off;
    }
  }
  // (64 x 64 blocks) the lane's fragments, see SmallTile: [plane or half][fragment or chunk]
  int small_x[2][2], small_y[2][2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      small_x[p][i] = IL ? (MS == 32 ? xil32_off[p][i] : xil_off[p] + i * 16 * 128)
                         : (MS == 32 ? x32_off[i] : x_frag_off + i * 16 * kTileRowBytes) + p * BX * kTileRowBytes;
      small_y[p][i] = IL ? (MS == 32 ? yil32_off[p][i] : yil_off[p] + i * 16 * 128)
                         : (MS == 32 ? y32_off[i] : y_frag_off + i * 16 * kTileRowBytes) + p * BY * kTileRowBytes;
    }
  }
  // (32-bit input) the lane's four chunks, see mma_step32_split
  const int x_split_off[4] = {IL ? xil32_off[0][0] : x32_off[0], IL ? xil32_off[0][1] : x32_off[1],
                              xil32_off[1][0], xil32_off[1][1]};
  const int y_split_off[4] = {IL ? yil32_off[0][0] : y32_off[0], IL ? yil32_off[0][1] : y32_off[1],
                              yil32_off[1][0], yil32_off[1][1]};
  // wide stores through LDS: no beta term (interleaved C only with the 16-row layout)
  const bool staged_ok = (MS == 16 || !args.c_interleaved) && !args.have_beta;

  // ---- pipeline ----------------------------------------------------------
  {
    const TileCoord tc = tile_coord(args, blockIdx.x);
    point_x(tc);
    point_y(tc);
  }
  // The bookkeeping of the copy (advance, which branches) is done at the top of
  // an iteration for the copies issued inside it, so that nothing but
  // straight-line code follows the barrier. Before the first iteration: the
  // requests that iterations -XLEAD .. -1 would have made, in their order (as a loop: written
  // out, they are most of the code that a block fetches on the way to its first product;
  // with one look at the coordinates instead of two 64x64x32 4.66 -> 4.23 us, 256^3 7.05 -> 6.45).
  if constexpr (SPLIT) {
#pragma unroll
    for (int t = -XLEAD; t < 0; ++t) {
      if (t + YLEAD >= 0) {
        if (t + YLEAD > 0) advance_y();
        issue_y(t + YLEAD);
      }
      if (t + XLEAD > 0) advance_x();
      issue_x(t + XLEAD);
    }
  } else {
#pragma unroll 1
    for (unsigned t = 0; t < (unsigned)XLEAD; ++t) {
      if (t > 0) advance();
      issue_y(t);
      issue_x(t);
    }
  }
  unsigned x_slot = 0, y_slot = 0;         // slots of the current iteration
  // (hand-ordered 16-row step) the lane's fragment addresses in the current slots
  unsigned xa[4], ya = lds_base + y_slot_off(0) + (y_frag_off - X_BYTES);
#pragma unroll
  for (int i = 0; i < 4; ++i) xa[i] = lds_base + x_slot_off(0) + xo[i];
  const unsigned iters = k_tiles;
  for (unsigned vt = blockIdx.x; vt < total; vt += gridDim.x) {
    // (SKIP) A wave whose part of the block lies beyond C leaves the matrix cores to the wave next to it on the SIMD (a
    // block of 128 rows of which 64 exist has one of each two); idle_waves_pay says when.
    bool inside = true;
    if constexpr (SKIP) {
      const TileCoord tc = tile_coord(args, vt);
      inside = tc.block_x * BX + wx * WX < args.nx && tc.block_y * BY + wy * WY < args.ny;
    }
    typename AccType<MS>::type acc_re[TY][TX], acc_im[TY][TX];
    SplitState<DT == kFloat32 ? TX : 1> split;   // (32-bit input)
    SmallTile small;                             // (64 x 64 blocks)
    // (the hand-ordered step of the 16-row MFMAs starts its first iteration from zero itself)
    constexpr bool kStepClears = !IL && DT != kInt1 && MS == 16 && TX == 4 && TY == 4;
    static_assert(!SPLIT || kStepClears, "separate X and Y rings: hand-ordered 16-row step only");
    if constexpr (DT == kFloat32) {
#pragma unroll
      for (int i = 0; i < TX; ++i) {
        split.re[i] = SplitSum{0.f, 0.f};
        split.im[i] = SplitSum{0.f, 0.f};
      }
    } else if constexpr (!kStepClears) {
#pragma unroll
      for (int j = 0; j < TY; ++j) {
#pragma unroll
        for (int i = 0; i < TX; ++i) {
          acc_re[j][i] = 0.f;
          acc_im[j][i] = 0.f;
        }
      }
    }
    // One K iteration; `first` says at compile time that it is a C tile's first one (kCarries:
    // kernels that multiply a K tile while they read the next one).
    // (math: whether the wave has elements of C to compute)
    auto iteration = [&](unsigned it, auto first, auto math) __attribute__((always_inline)) {
      advance();
      // After the first C tile, the K tiles of the first YLEAD iterations were
      // already waited for before the previous epilogue (see below), so these
      // iterations only need the barrier; waiting on the counter here would
      // wait for the previous tile's C stores, which are younger than them.
      if (vt != blockIdx.x && it < (unsigned)YLEAD) {
        if constexpr (SMALL) {
          asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        } else {
          asm volatile("s_barrier" ::: "memory");
        }
      } else {
        wait_vmcnt_then_barrier<kOutstandingOk, SMALL>();
      }
      if constexpr (RAGGED) {
        if (it + 1 == iters && row_bytes % 16 != 0) settle_row_ends(x_slot, y_slot);
      }
      // The slots of the previous iteration are free now: refill them with the
      // K tiles that are XLEAD / YLEAD iterations ahead (of this C tile or the
      // next). The copy instructions go out after the first group of MFMAs: right
      // after the barrier every wave of the block would otherwise be busy with
      // their address arithmetic and the matrix cores would have nothing to do.
      auto refill_slots = [&] {
        unsigned x_refill = x_slot + XLEAD, y_refill = y_slot + YLEAD;
        x_refill = x_refill >= XSLOTS ? x_refill - XSLOTS : x_refill;
        y_refill = y_refill >= SLOTS ? y_refill - SLOTS : y_refill;
        issue_y(y_refill);
        issue_x(x_refill);
      };
      const unsigned x_next = x_slot + 1 == XSLOTS ? 0 : x_slot + 1;
      const unsigned y_next = y_slot + 1 == SLOTS ? 0 : y_slot + 1;
      if constexpr (kStepClears) {
        // (the first iteration of a C tile starts its sums from zero instead of
        // from accumulators that would have to be cleared first; the fragment
        // addresses of the next iteration are worked out among the last MFMAs
        // of this one, so that only the wait and the barrier stand between two
        // iterations' MFMAs)
        // (no fragment is read after the step calls this, so it overwrites in place)
        auto next_addresses = [&] {
#pragma unroll
          for (int i = 0; i < 4; ++i) xa[i] = lds_base + x_slot_off(x_next) + xo[i];
          ya = lds_base + y_slot_off(y_next) + (y_frag_off - X_BYTES);
        };
        if constexpr (!decltype(math)::value) {
          refill_slots();
          next_addresses();
        } else if (it == 0) {
          mma_step_ordered<DT, BX, BY, XT, true>(xa, ya, acc_re, acc_im, refill_slots,
                                                 next_addresses);
        } else {
          mma_step_ordered<DT, BX, BY, XT, false>(xa, ya, acc_re, acc_im, refill_slots,
                                                  next_addresses);
        }
      } else {
        const char *slot_ptr = lds + x_slot_off(x_slot);
        if constexpr (!decltype(math)::value) {
          refill_slots();
        } else if constexpr (SMALL) {
          SmallTile next;
          read_small_tile(slot_ptr, small_x, small_y, next);
          if constexpr (decltype(first)::value) {
            refill_slots();
          } else {
            mma_small_tile<DT, IL>(small, acc_re, acc_im, refill_slots);
          }
          small = next;
        } else if constexpr (DT == kFloat32) {
          static_assert(MS == 32 && TY == 1, "32-bit input: 32-row MFMA, tiles side by side");
          mma_step32_split<BX, BY, TX, IL, decltype(first)::value>(slot_ptr, x_split_off, y_split_off, split,
                                                                   refill_slots);
        } else if constexpr (IL && MS == 32) {
          static_assert(TX == 2 && TY == 2, "2 x 2 tiles of 32 x 32 per wave");
          mma_step32_interleaved<DT, BX, BY>(slot_ptr, xil32_off, yil32_off, acc_re, acc_im,
                                             refill_slots);
        } else if constexpr (IL && DtypeTraits<DT>::kElemBytes == 2 && TX == 4 && TY == 4) {
          mma_step_interleaved_ordered<DT, BX, BY>(slot_ptr, xil_off, yil_off, acc_re, acc_im,
                                                   refill_slots);
        } else if constexpr (IL) {
          mma_step_interleaved<DT, BX, BY, TX, TY>(slot_ptr, xil_off, yil_off, acc_re, acc_im,
                                                   refill_slots);
        } else {
          const char *tile[KPM] = {slot_ptr};
          if constexpr (DT == kInt1) {
            static_assert(MS == 32 && TX == 2 && TY == 2, "2 x 2 tiles of 32 x 32 per wave");
            mma_step32_bits<BX, BY>(tile[0], x32_off, y32_off, acc_re, acc_im, refill_slots);
          } else if constexpr (MS == 32 && TX == 2 && TY == 2) {
            mma_step32_ordered<DT, BX, BY>(tile[0], x32_off, y32_off, acc_re, acc_im, refill_slots);
          } else if constexpr (MS == 32) {
            mma_step32<DT, BX, BY, TX, TY>(tile[0], x32_off, y32_off, acc_re, acc_im, refill_slots);
          } else {
            mma_step<DT, BX, BY, TX, TY>(tile, x_frag_off, y_frag_off, acc_re, acc_im, refill_slots);
          }
        }
      }
      x_slot = x_next;
      y_slot = y_next;
    };
    unsigned it = 0;
    constexpr bool kCarries = SMALL || DT == kFloat32;
    const std::true_type yes{};
    const std::false_type no{};
    if constexpr (kCarries) iteration(it++, yes, yes);
    if (!SKIP || inside) {
      for (; it < iters; ++it) iteration(it, no, yes);
    } else if constexpr (SKIP) {
#pragma unroll 1
      for (; it < iters; ++it) iteration(it, no, no);
    }
    if constexpr (SMALL) mma_small_tile<DT, IL>(small, acc_re, acc_im, [] {});
    // The stores below are not waited for here: they drain while the next C
    // tile is being computed. The counter cannot tell loads from stores, so
    // the next tile's first K tiles, which are already on their way, are waited
    // for now; the first wait that has to include the stores then comes YLEAD
    // iterations into the next tile. (64 x 64 blocks: the wave's reads of the last slot may still be
    // under way; the next tile's first barrier, behind which the slot is refilled, waits for them,
    // and no epilogue of theirs uses LDS.)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const TileCoord tc = tile_coord(args, vt);
    const unsigned x_wave = tc.block_x * BX + wx * WX, y_wave = tc.block_y * BY + wy * WY;
    bool redo = false;   // (32-bit input) this wave's tile is computed again
    if constexpr (DT == kFloat32) {
      redo = !mma_split_last(split, acc_re, acc_im);
      if (__builtin_expect(redo, 0)) {
        redo = !only_nan_rows<LOADER, TX>(args, tc.b, x_wave, y_wave, lane_here(), acc_re, acc_im);
      }
    }
    bool staged = false;
    if constexpr (XT) {
      // the accumulators already hold whole row segments
      if (staged_ok && !args.c_interleaved && x_wave + WX <= args.nx && y_wave + WY <= args.ny) {
        store_wave_tile_rows<TOUT, TY>(args, tc.b, x_wave, y_wave, lane, acc_re, acc_im);
      } else {
        store_wave_tile<TOUT, TX, TY, kAcc16T>(args, tc.b, x_wave, y_wave, lane, acc_re, acc_im);
      }
      staged = true;
    }
    if constexpr (!XT && MS == 16 && TOUT == kFloat32 && TX == 4 &&
                  !SPLIT && NW * kStagePatchBytes <= SLOT_BYTES) {
      if (staged_ok) {
        // The slot consumed last is free until the next refill, but other waves
        // may still be reading it: one barrier, then every wave uses its own
        // patch of it. (Uniform per block, so the barrier is safe.)
        // ([X | Y] slots here: the rings are one)
        unsigned free_slot = y_slot + YLEAD;
        free_slot = free_slot >= SLOTS ? free_slot - SLOTS : free_slot;
        asm volatile("s_barrier" ::: "memory");
        if (x_wave + WX <= args.nx && y_wave + WY <= args.ny) {
          char *patch = lds + free_slot * SLOT_BYTES + wave * kStagePatchBytes;
          if (args.c_interleaved) {
            store_wave_tile_staged_il<TX, TY>(args, tc.b, x_wave, y_wave, lane, patch, acc_re, acc_im);
          } else {
            store_wave_tile_staged<TX, TY>(args, tc.b, x_wave, y_wave, lane, patch, acc_re, acc_im);
          }
          staged = true;
        }
      }
    }
    if constexpr (!XT && MS == 16 && (TOUT == kFloat16 || TOUT == kBfloat16) && TX == 4 &&
                  !SPLIT && NW * kStagePatchBytes <= SLOT_BYTES) {
      if (staged_ok && !args.c_interleaved) {
        // ([X | Y] slots here: the rings are one)
        unsigned free_slot = y_slot + YLEAD;
        free_slot = free_slot >= SLOTS ? free_slot - SLOTS : free_slot;
        asm volatile("s_barrier" ::: "memory");
        if (x_wave + WX <= args.nx && y_wave + WY <= args.ny) {
          store_wave_tile_staged_narrow<TOUT, TX, TY>(
              args, tc.b, x_wave, y_wave, lane,
              lds + free_slot * SLOT_BYTES + wave * kStagePatchBytes, acc_re, acc_im);
          staged = true;
        }
      }
    }
    if constexpr (DT == kFloat32 && TOUT == kFloat32) {
      static_assert(!SPLIT && NW * kStagePatchF32Bytes <= SLOT_BYTES, "a patch for each wave in one slot");
      if (!args.have_beta) {
        unsigned free_slot = y_slot + YLEAD;
        free_slot = free_slot >= SLOTS ? free_slot - SLOTS : free_slot;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (!redo && x_wave + WX <= args.nx && y_wave + WY <= args.ny) {
          store_wave_tile_staged_f32<TX>(args, tc.b, x_wave, y_wave, lane_here(),
                                         lds + free_slot * SLOT_BYTES + wave * kStagePatchF32Bytes, acc_re, acc_im);
          staged = true;
        }
      }
    } else if constexpr (MS == 32 && (TOUT == kFloat32 || TOUT == kInt32) &&
                         !SPLIT && NW * kStagePatch32Bytes <= SLOT_BYTES) {
      if (staged_ok) {
        // ([X | Y] slots here: the rings are one)
        unsigned free_slot = y_slot + YLEAD;
        free_slot = free_slot >= SLOTS ? free_slot - SLOTS : free_slot;
        asm volatile("s_barrier" ::: "memory");
        if (x_wave + WX <= args.nx && y_wave + WY <= args.ny) {
          store_wave_tile_staged32<TX, TY, TOUT == kInt32>(args, tc.b, x_wave, y_wave, lane,
                                           lds + free_slot * SLOT_BYTES + wave * kStagePatch32Bytes,
                                           acc_re, acc_im);
          staged = true;
        }
      }
    }
    if constexpr (DT == kFloat32) {
      if (__builtin_expect(redo, 0)) {
        recompute_f32<TOUT, LOADER, TX, TY>(args, tc.b, x_wave, y_wave, lane_here());
        // (its loads and stores are not among those that the next tile's waits count)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        staged = true;
      }
    }
    if (!staged) {
      if constexpr (TOUT == kInt32) {
        store_wave_tile_int32<TX, TY, MS>(args, tc.b, x_wave, y_wave, lane, acc_re, acc_im);
      } else if constexpr (DT == kFloat32) {
        // (one MFMA tile after the other: the addresses of both at once do not fit the registers)
        const int at = lane_here();
#pragma unroll
        for (int t = 0; t < TX * TY; ++t) {
          const float16_t_ re[1][1] = {{acc_re[t / TX][t % TX]}}, im[1][1] = {{acc_im[t / TX][t % TX]}};
          store_wave_tile<TOUT, 1, 1, MS>(args, tc.b, x_wave + 32 * (t % TX), y_wave + 32 * (t / TX), at, re, im);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        store_wave_tile<TOUT, TX, TY, MS>(args, tc.b, x_wave, y_wave, lane, acc_re, acc_im);
      }
    }
  }
  // nothing may still be writing into LDS when the block gives it back
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

#include "gemm_mfma_wave.h"

inline hipError_t check_grid(size_t total) {
  return total > 0x7fffffffu ? hipErrorInvalidValue : hipSuccess;
}

// LDS beyond 64 KiB has to be requested once per kernel and device. `done`
// is the caller's per-kernel record (one flag per device ordinal).
constexpr int kMaxDevices = 64;
template <typename Kernel>
hipError_t allow_lds(Kernel kernel, int bytes, std::atomic<bool> (&done)[kMaxDevices]) {
  if (bytes <= 64 * 1024) return hipSuccess;
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev)) return e;
  const bool tracked = dev >= 0 && dev < kMaxDevices;
  if (tracked && done[dev].load(std::memory_order_acquire)) return hipSuccess;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e == hipSuccess && tracked) done[dev].store(true, std::memory_order_release);
  return e;
}

template <int DT, int TOUT, int BX, int BY, int WX, int WY, int KT, int LOADER, int WPE>
hipError_t launch_config(const GemmParams &p, hipStream_t stream) {
  constexpr int NTHREADS = 64 * (BX / WX) * (BY / WY);
  constexpr int LDS_BYTES = 2 * KT * 2 * (BX + BY) * kTileRowBytes;
  const KernelArgs a = make_kernel_args(p, BX, BY);
  const size_t total = (size_t)a.blocks_x * a.blocks_y * p.batch;
  if (total == 0) return hipSuccess;
  if (hipError_t e = check_grid(total)) return e;
  auto kernel = complex_gemm_mfma<DT, TOUT, BX, BY, WX, WY, KT, LOADER, WPE>;
  static std::atomic<bool> lds_allowed[kMaxDevices];
  if (hipError_t e = allow_lds(kernel, LDS_BYTES, lds_allowed)) return e;
  hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(NTHREADS), LDS_BYTES, stream, a);
  return hipGetLastError();
}

// Number of compute units of the current device (queried once).
inline int compute_units() {
  static const int n = [] {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0) {
      cus = 256;
    }
    return cus;
  }();
  return n;
}

template <int DT, int TOUT, int BX, int BY, int WX, int WY, int SLOTS, int WPE,
          int LOADER = kLoadTiled, int MS = 16, bool XT = false, int XSLOTS = SLOTS, bool SKIP = false>
hipError_t launch_dtl(const GemmParams &p, hipStream_t stream) {
  constexpr int NTHREADS = 64 * (BX / WX) * (BY / WY);
  constexpr int LDS_BYTES = 2 * (XSLOTS * BX + SLOTS * BY) * kTileRowBytes;
  constexpr int kLdsPerCu = 160 * 1024;
  constexpr int BLOCKS_PER_CU = (kLdsPerCu / LDS_BYTES) < (WPE * 256 / NTHREADS)
                                    ? (kLdsPerCu / LDS_BYTES)
                                    : (WPE * 256 / NTHREADS);
  static_assert(BLOCKS_PER_CU >= 1, "configuration does not fit a CU");
  const KernelArgs a = make_kernel_args(p, BX, BY);
  const size_t total = (size_t)a.blocks_x * a.blocks_y * p.batch;
  if (total == 0) return hipSuccess;
  if (hipError_t e = check_grid(total)) return e;
  auto kernel = complex_gemm_mfma_dtl<DT, TOUT, BX, BY, WX, WY, SLOTS, WPE, LOADER, MS, XT, XSLOTS, SKIP>;
  static std::atomic<bool> lds_allowed[kMaxDevices];
  if (hipError_t e = allow_lds(kernel, LDS_BYTES, lds_allowed)) return e;
  // persistent blocks: as many as are resident at once, each walking C tiles
  // with a stride of the grid size (a multiple of the XCD count)
  const size_t resident = (size_t)compute_units() * BLOCKS_PER_CU / kNumXcd * kNumXcd;
  const unsigned grid = (unsigned)(total < resident ? total : resident);
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(NTHREADS), LDS_BYTES, stream, a);
  return hipGetLastError();
}

// Whether waves that have nothing of C to compute should leave their products out (SKIP of complex_gemm_mfma_dtl; 16-bit
// input on 256 x 128 and 128 x 128 blocks). Looking for them takes every wave about 0.25 us a tile, and the loop on (re, im)
// pairs 2 to 4 % besides, so it pays where the units that finish last have such waves and a tile is long enough. Time without
// and with it, 2500 problems that have some (geometric means):
//   a unit each, all blocks          up to 4 pieces of K 0.94 to 0.98 (pairs the least), 5 to 8 1.01 to 1.05 (pairs 1.00), from 33 on 1.08 to 1.11
//   a unit each, some of the blocks  0.94 to 0.96 up to 4 pieces, 0.95 (pairs) to 1.01 beyond
//   more blocks than units           fewer than 0.3 of them 0.97 to 1.00; beyond, up to 4 pieces 0.95 to 0.99, then on planar rows and
//                                    tiles 1.01 to 1.08 (all of them: to 1.16), pairs 0.99 at 0.3 * 8 pieces, 1.02 at 0.3 * 32 and 0.8 * 4
// (8- and 1-bit input: B=16 4096x4096x8192, where no wave is idle, 0.8 % slower with the test in the kernel.)
template <int BX, int BY, int WX, int WY>
bool idle_waves_pay(const GemmParams &p) {
  const double pieces = (double)(p.input_interleaved ? (p.k_tiles + 1) / 2 : p.k_tiles);
  const size_t across = ceil_div(p.nx, BX), down = ceil_div(p.ny, BY);
  if (!across || !down) return false;
  const bool idle_x = (p.nx - 1) % BX + 1 <= BX - WX, idle_y = (p.ny - 1) % BY + 1 <= BY - WY;
  // share of the blocks that have idle waves
  const double share = 1.0 - (1.0 - (idle_x ? 1.0 / (double)across : 0.0)) * (1.0 - (idle_y ? 1.0 / (double)down : 0.0));
  if ((size_t)p.batch * across * down <= (size_t)compute_units()) {
    return share == 1.0 && pieces >= (p.input_interleaved ? 8.0 : 5.0);
  }
  return pieces >= 5.0 && share >= 0.3 && share * pieces >= (p.input_interleaved ? 5.0 : 1.5);
}
template <int DT, int TOUT, int BX, int BY, int WX, int WY, int SLOTS, int WPE, int LOADER, int MS = 16, bool XT = false>
hipError_t launch_block(const GemmParams &p, hipStream_t stream) {
  if constexpr (DtypeTraits<DT>::kElemBytes == 2 && DT != kInt1 && BX * BY > 64 * 64) {
    if (idle_waves_pay<BX, BY, WX, WY>(p)) {
      return launch_dtl<DT, TOUT, BX, BY, WX, WY, SLOTS, WPE, LOADER, MS, XT, SLOTS, true>(p, stream);
    }
  }
  return launch_dtl<DT, TOUT, BX, BY, WX, WY, SLOTS, WPE, LOADER, MS, XT>(p, stream);
}

template <int DT, int TOUT, int LOADER, int TX, int TY, int SPLIT = 1>
hipError_t launch_wave(const GemmParams &p, hipStream_t stream) {
  const KernelArgs a = make_kernel_args(p, 16 * TX, 16 * TY);
  const size_t total = (size_t)a.blocks_x * a.blocks_y * p.batch;
  if (total == 0) return hipSuccess;
  if (hipError_t e = check_grid(total)) return e;
  auto kernel = complex_gemm_mfma_wave<DT, TOUT, LOADER, TX, TY, SPLIT>;
  static std::atomic<bool> lds_allowed[kMaxDevices];
  if (hipError_t e = allow_lds(kernel, SPLIT * kWaveLdsBytes, lds_allowed)) return e;
  hipLaunchKernelGGL(kernel, dim3((unsigned)total), dim3(64 * SPLIT), SPLIT * kWaveLdsBytes, stream, a);
  return hipGetLastError();
}

// How the 192 x 256 kernel covers the width of C: tiles of 192 columns, the last of
// which may hang over the edge, or - where 64 divides the width - full tiles
// followed by short ones of 128 columns, which take two thirds of the matrix
// instructions: as many as make the width come out even (4096 = 20 x 192 + 2 x 128),
// or three more for two full ones less as long as that shortens the work of the
// block that finishes last (8192 = 32 x 192 + 16 x 128: with 32 rows of tiles every
// one of 256 blocks gets 4 full and 2 short tiles, 5 1/3 full tiles' worth, where
// 42 x 192 + 128 would give 64 of them 6 full tiles). The short tiles are the last
// ones in the kernel's numbering; `rounds` is that longest block's work in full
// tiles, with a charge for the change of kind.
struct WideTiling {
  unsigned full_x, short_x, grid;
  double rounds;
};
// (the tuner switches the short tiles off for a row of its table)
static bool g_wide_short_tiles = true;
inline WideTiling wide_tiling(const GemmParams &p) {
  const size_t resident = (size_t)compute_units() / kNumXcd * kNumXcd;
  const size_t rows = ceil_div((size_t)p.ny, (size_t)kWideBY) * p.batch;
  WideTiling best;
  best.full_x = (unsigned)ceil_div((size_t)p.nx, (size_t)kWideBX);
  best.short_x = 0;
  const size_t plain_total = best.full_x * rows;
  best.grid = (unsigned)(plain_total < resident ? plain_total : resident);
  best.rounds = best.grid ? (double)ceil_div(plain_total, (size_t)best.grid) : 0.0;
  const size_t units = p.nx / 64;
  if (!g_wide_short_tiles || p.nx % 64 != 0 || plain_total == 0) return best;
  const double short_work = (double)kWideShortBX / kWideBX, change = 0.05;
  for (size_t n_short = units % 3 == 0 ? 3 : units % 3 == 2 ? 1 : 2; 3 + 2 * n_short <= units; n_short += 3) {
    WideTiling mixed;
    mixed.full_x = (unsigned)((units - 2 * n_short) / 3);
    mixed.short_x = (unsigned)n_short;
    const size_t full_total = mixed.full_x * rows, total = full_total + n_short * rows;
    mixed.grid = (unsigned)(total < resident ? total : resident);
    // block i computes the tiles i, i + grid, ...
    mixed.rounds = 0.0;
    for (size_t i = 0; i < mixed.grid; ++i) {
      const size_t mine = (total - i + mixed.grid - 1) / mixed.grid;
      const size_t full = i < full_total ? (full_total - i + mixed.grid - 1) / mixed.grid : 0;
      const double work =
          (double)full + short_work * (double)(mine - full) + (full > 0 && mine > full ? change : 0.0);
      mixed.rounds = work > mixed.rounds ? work : mixed.rounds;
    }
    if (mixed.rounds < best.rounds - 1e-9) best = mixed;
  }
  return best;
}

// The 192 x 256 block of gemm_mfma_wide.h (16-bit input; tiled layout, or IL: the
// pipeline's interleaved rows): one persistent block per compute unit.
template <int DT, int TOUT, bool IL = false>
hipError_t launch_wide(const GemmParams &p, hipStream_t stream) {
  KernelArgs a = make_kernel_args(p, kWideBX, kWideBY);
  const WideTiling tiling = wide_tiling(p);
  a.blocks_x = tiling.full_x;
  a.short_x = tiling.short_x;
  const size_t total = (size_t)(a.blocks_x + a.short_x) * a.blocks_y * p.batch;
  if (total == 0) return hipSuccess;
  if (hipError_t e = check_grid(total)) return e;
  const unsigned grid = tiling.grid;
  if (p.have_alpha) {
    auto kernel = complex_gemm_mfma_wide<DT, TOUT, IL, true>;
    static std::atomic<bool> lds_allowed[kMaxDevices];
    if (hipError_t e = allow_lds(kernel, kWideLdsBytes, lds_allowed)) return e;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), kWideLdsBytes, stream, a);
  } else {
    auto kernel = complex_gemm_mfma_wide<DT, TOUT, IL, false>;
    static std::atomic<bool> lds_allowed[kMaxDevices];
    if (hipError_t e = allow_lds(kernel, kWideLdsBytes, lds_allowed)) return e;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), kWideLdsBytes, stream, a);
  }
  return hipGetLastError();
}

// Which block shape of complex_gemm_mfma_dtl a problem gets: the one whose busiest compute
// unit finishes first, by
//   tiles of a unit * area of a tile * cost * (64-byte pieces of K + what a tile costs besides),
// with the costs relative to 256 x 128, where a tile costs as much as 10 pieces of K besides
// its K loop (ring fill, stores). The smaller a block, the more of the chip a small
// problem fills and the less it computes beyond the edges of C, but the more bytes it
// moves per flop. Times with 256 x 128, 128 x 128 and 64 x 64 blocks in us, on operands that no cache
// held (profiles/gemm_block_choice.txt):
//   too few tiles for the larger blocks, 16 bits on tiles 256^3:  14.8, 12.2, 6.4;  32 bits B=2 1000^3:  (none), 166, 117;
//     8 bits 1024^3:  24.2, 21.7, 10.5;  1 bit 64x64x65536:  526, 308, 115
//   every unit busy, 16 bits on planar rows, B=157 192x604x3680:  735, 757, 1021; B=167 800x184x2064:  553, 642, 863
//     32 bits, which a smaller wave tile splits more often, 4096x4096x512:  (none), 416, 480
//     8 bits on tiles, 4096x4096x512:  46, 45, 65
//     1 bit, whose words a wave with one tile expands for half as many products, 3452x1504x32256:
//       271, 288, 313
// Two blocks share a unit with 64 x 64 tiles and with 128 x 128 tiles (of 16-bit input: those of four waves), and
// a last tile that has the unit to itself leaves it idle for a part of the time: `lone` of a tile.
// With beta the epilogue reads C first, which costs the larger tiles more (8 bits on planar
// rows, B=11 456x1542x192: 97, 84, 47), and pairs of C with beta are read and stored piece by piece by all of them (B=43 144x1024x32
// fp16 pairs 40.2, 36.3, 27.3).
//   128 x 128 blocks of 16-bit input have eight waves and a ring of four slots while every block has a unit to itself, which
// keeps more on its way; beyond, four waves of 64 x 64 and two slots, of which
// two share a unit: one stores C or waits while the other multiplies, the fragments are read once for twice as many
// products, and C is stored in whole row segments. In us, planar rows unless said, 8 and 4 waves (256 x 128 blocks):
// B=67 384x3136x328 439, 330 (328); B=300 512x512x128 211, 126 (137); B=100 320x320x256 pairs 47, 41 (51). With beta, which
// takes the four waves' registers while C is read, eight may be the faster ones there too (B=60 1536x128x80 fp16 planar 41.8, 51.3;
// 750 such problems 0.97 times on planar rows of K up to 300, 1.03 to 1.12 elsewhere), which have constants of their own for it.
//   The constants are fitted, for each type and operand layout, to the times of all three shapes over
// 30000 problems of random sizes, 40 % of them on operands that no cache held
// (python -m ccglib_amd.tuning.block_choice times such problems); those of 8-bit tiles
// to 1900, of 32-bit input to 1200 further ones, timed since those kernels last changed. Those of 16-bit input: to the choice among the
// shapes in 8600 problems on cold operands, 40 % of them of K up to 128 (the least sum of what a choice loses against the fastest shape
// and, counted twice, against the choice from before there were blocks of four waves). On a third kept out of the fit it is
// 0.4 % (tiles), 0.7 % (planar rows) and 0.6 % (pairs) behind the fastest of the shapes on average.
enum BlockShape { k256x128, k128x128, k64x64 };
struct BlockChoice {
  BlockShape shape;
  double time;   // in units of one element of C in a 256 x 128 tile
  bool eight_waves;   // (16-bit input, 128 x 128)
};
struct BlockCosts {
  double cost_128, cost_64;   // per element of C and piece of K, of 256 x 128's
  double tile_128, tile_64;   // what a tile costs besides its K loop, in pieces of K
  double lone_128, lone_64;   // what a tile without a neighbour costs more, of a tile
  double beta_256, beta_128, beta_64;   // added to the tile's cost with beta
  // 16-bit input: the same of 128 x 128 blocks of eight waves, and what beta adds if C holds pairs (256 x 128 and four waves; eight)
  double cost_8w = 0.0, tile_8w = 0.0, beta_8w = 0.0, pairs_beta = 0.0, pairs_beta_8w = 0.0;
};
inline BlockCosts block_costs(const GemmParams &p) {
  if (p.type_in == kInt1) return {1.04, 1.44, 8.8, 9.0, 0.11, 0.0, 0.0, 0.0, 0.0};
  // (32-bit input has no 256 x 128 block: relative to 128 x 128)
  if (p.type_in == kFloat32) return {1.0, 1.24, 6.0, 5.0, 0.0, 0.0, 0.0, 4.0, 2.0};
  const bool planar = p.variant == kBasic && !p.input_interleaved;
  if (bits_of(p.type_in) == 8) {
    if (p.input_interleaved) return {1.04, 1.87, 9.3, 7.0, 0.3, 0.1, 13.0, 10.0, 1.0};
    if (planar) return {1.30, 2.54, 7.6, 7.9, 0.3, 0.1, 13.0, 10.0, 1.0};
    return {1.05, 1.61, 9.2, 9.4, 0.3, 0.11, 13.0, 10.0, 1.0};
  }
  if (p.input_interleaved) {
    return {1.06, 1.85, 9.07, 8.55, 0.34, 0.43, 19.94, 18.45, 10.0, 1.27, 11.81, 12.36, 3.44, 1.27};
  }
  if (planar) return {1.16, 2.51, 7.86, 6.97, 0.48, 0.26, 10.09, 11.93, 2.61, 1.29, 11.73, 3.88, 4.3, 1.6};
  return {1.08, 1.85, 8.72, 8.86, 0.44, 0.60, 15.85, 15.28, 6.62, 1.30, 7.48, 12.97, 5.24, 1.91};
}
inline BlockChoice block_choice(const GemmParams &p) {
  const size_t units = (size_t)compute_units();
  BlockCosts costs = block_costs(p);
  const bool bits16 = bits_of(p.type_in) == 16;
  // (pieces of a plane's row: an interleaved row holds both planes)
  const double pieces = (double)(p.input_interleaved ? (p.k_tiles + 1) / 2 : p.k_tiles);
  if (p.c_interleaved) {
    costs.beta_256 += costs.pairs_beta;
    costs.beta_128 += costs.pairs_beta;
    costs.beta_8w += costs.pairs_beta_8w;
  }
  const double large = pieces + 10.0 + (p.have_beta ? costs.beta_256 : 0.0);
  auto time = [&](size_t bx, size_t by, double cost, double tile, double lone, double beta) {
    const size_t tiles = (size_t)p.batch * ceil_div((size_t)p.nx, bx) * ceil_div((size_t)p.ny, by);
    const size_t mine = ceil_div(tiles, units);
    return ((double)mine + (mine % 2 ? lone : 0.0)) * (double)(bx * by) * cost *
           (pieces + tile + (p.have_beta ? beta : 0.0)) / large;
  };
  const bool no_256 = p.type_in == kFloat32;
  const double t256 = no_256 ? HUGE_VAL : time(256, 128, 1.0, 10.0, 0.0, costs.beta_256);
  // (a large C whose rows share cache lines, which the narrower blocks write in more parts: B=173 1728x1656x64 fp16
  // 1030 us on 256 x 128 blocks, 1357 on these)
  const size_t c_bytes = (size_t)2 * p.batch * p.nx * p.ny * bits_of(p.type_out) / 8;
  const bool shared_lines = bits16 && c_bytes >= ((size_t)256 << 20) &&
                            (size_t)p.nx * (p.c_interleaved ? 2 : 1) * bits_of(p.type_out) / 8 % 128 != 0;
  if (shared_lines) costs.tile_128 += 4.0;
  const bool few = (size_t)p.batch * ceil_div(p.nx, 128) * ceil_div(p.ny, 128) <= units;
  const double t4w = bits16 && few ? HUGE_VAL
                                   : time(128, 128, costs.cost_128, costs.tile_128, costs.lone_128, costs.beta_128);
  const double t8w = bits16 && (few || p.have_beta) ? time(128, 128, costs.cost_8w, costs.tile_8w, 0.0, costs.beta_8w)
                                                    : HUGE_VAL;
  const bool eight = t8w < t4w;
  const double t128 = eight ? t8w : t4w;
  const double t64 = time(64, 64, costs.cost_64, costs.tile_64, costs.lone_64, costs.beta_64);
  if (p.block_tile == 1 && !no_256) return {k256x128, t256, false};
  if (p.block_tile == 1 || p.block_tile == 2) return {k128x128, t128, eight};
  if (p.block_tile >= 4) return {k64x64, t64, false};   // (5 to 7: waves, where there are such kernels)
  if (t256 <= t128 && t256 <= t64) return {k256x128, t256, false};
  return t128 <= t64 ? BlockChoice{k128x128, t128, eight} : BlockChoice{k64x64, t64, false};
}

// Whether the 192 x 256 block of gemm_mfma_wide.h can compute this problem (what
// its stores and its K loop assume), and whether it pays: per flop it measured
// about 7 % faster than the 256 x 128 block once every compute unit is busy
// (B=64 512x4096x576: 0.519 against 0.558 ms), but its tiles are 1.5 times as
// large, so more of the last round of tiles can stay empty - which the short
// tiles of wide_tiling even out where the width allows (8192^3: 5 1/3 tiles for
// every block, 2.75 against 2.78 ms).
inline bool wide_tiles_apply(const GemmParams &p) {
  if (p.c_interleaved || p.have_beta || (uintptr_t)p.c % 16 != 0 ||
      p.nx % 64 != 0 || p.ny % 64 != 0 || p.k_in_memory) {
    return false;
  }
  if (p.input_interleaved) {
    // rows of whole 128-byte pieces (32 complex values), at least two of them; a
    // lane's offset inside a copy of 8 rows is a 32-bit number
    const size_t row_bytes = (size_t)2 * p.k * bits_of(p.type_in) / 8;
    return bits_of(p.type_in) == 16 && row_bytes % 128 == 0 && row_bytes >= 256 &&
           row_bytes < ((size_t)1 << 28) && (uintptr_t)p.x % 16 == 0 && (uintptr_t)p.y % 16 == 0;
  }
  return p.variant == kOpt && p.k_tiles >= 2;
}
inline bool wide_tiles_pay(const GemmParams &p) {
  if (p.block_tile != 0) return p.block_tile == 3;
  return wide_tiling(p).rounds * (kWideBX * kWideBY) < 1.075 * block_choice(p).time;
}

// Which tile the waves of complex_gemm_mfma_wave take, if that kernel is the faster one: the least of, in us,
//   fixed + max(K tiles * alone, K tiles * crowded * n / units, operand MB * bytes) + tile * n / units
// over 64 x 64 blocks and the wave tiles, with n blocks or waves: `alone` is what a K tile takes
// with a unit to itself, `crowded` with others next to it, `tile` what a tile costs besides. Waves: `alone` grows by `second` for every
// further wave of the busiest unit (330 waves on 256 units take as long as 512 where the copies of one wave do not fill the time; a
// wave keeps 32 KiB on its way where a block keeps 80, so that operands that no cache holds come in more slowly: B=197 24x49x2992
// planar fp16 62 us on waves, 46 on blocks). The constants are
// fitted, for each type and operand layout, to the choice among the shapes (what it loses against the fastest one, twice what it loses
// against 64 x 64 blocks alone, and a little of the errors of the times themselves): 10700 problems of 16 bits and 4100 of 8, a fifth of
// them on operands that the caches hold, 1890 of 1 bit, all of which have 64 x 64 blocks by block_choice.
// On those kept out of the fit the choice was behind the fastest shape by 0.3 % (tiles), 0.5 % (pairs) and 1.0 % (planar rows; 1.9 % with the
// constants before) for 16 bits, 0.1 to 0.4 % for 8, 3 to 4 % for 1 bit (waves that do not share K would serve more rounds), and in front of 64 x 64
// blocks by 1.33 to 1.50 times (16 bits), 1.15 to 1.23 (8 bits), 1.21 to 1.31 (1 bit). More waves than there are SIMDs are left to the
// blocks: the fifth wave of a unit has to share one (B=213 32x192x3184 on planar rows, 1278 waves: 179 us on blocks, 261 on waves).
enum WaveShape { kNoWaves, kWaves32x32, kWaves32x16, kWaves16x16 };
struct WaveCosts {
  double fixed, alone, crowded, tile, second;
};
struct WaveTable {
  WaveCosts shape[4];   // 64 x 64 blocks, then as WaveShape
  double beta;          // blocks: they only request C behind the last product
  double block_bytes, wave_bytes;   // us per MB of A and B ...
  double cached_mb = 0.0;           // ... beyond these, which the caches may hold
};
inline const WaveTable &wave_costs(const GemmParams &p) {
  static constexpr WaveCosts none = {0.0, 0.0, 0.0, 0.0, 0.0};
  static constexpr WaveTable bits16_tiled = {{{4.016, 0.295, 0.376, 1.653, 0.000}, {3.304, 0.200, 0.070, 0.437, 0.338},
      {3.316, 0.147, 0.079, 0.009, 0.356}, {2.493, 0.097, 0.060, 0.062, 0.393}}, 1.114, 0.133, 0.090, 32.0};
  static constexpr WaveTable bits16_planar = {{{4.059, 0.432, 0.470, 2.137, 0.000}, {3.899, 0.226, 0.223, 0.293, 0.660},
      {2.865, 0.200, 0.180, 0.093, 0.411}, {2.660, 0.127, 0.097, 0.077, 0.268}}, 0.845, 0.316, 0.453, 32.0};
  static constexpr WaveTable bits16_pairs = {{{4.010, 0.359, 0.476, 2.376, 0.000}, {3.246, 0.288, 0.182, 0.369, 0.253},
      {3.060, 0.187, 0.106, 0.025, 0.381}, {2.581, 0.111, 0.085, 0.015, 0.445}}, 1.766, 0.195, 0.129, 32.0};
  static constexpr WaveTable bits8_tiled = {{{3.670, 0.306, 0.387, 2.100, 0.000}, {3.195, 0.202, 0.136, 0.410, 0.229}, none, none},
      1.888, 0.146, 0.166};
  static constexpr WaveTable bits8_planar = {{{3.851, 0.504, 0.709, 2.196, 0.000}, {3.569, 0.236, 0.266, 0.127, 0.825}, none, none},
      2.029, 0.236, 0.336};
  static constexpr WaveTable bits8_pairs = {{{4.097, 0.391, 0.431, 1.849, 0.000}, {4.204, 0.240, 0.189, 0.043, 0.578}, none, none},
      1.750, 0.285, 0.308};
  // (1 bit: `fixed` and `alone` of a tile shared by four waves, `tile` of a launch, see wave_choice)
  static constexpr WaveTable int1_tiled = {{{3.738, 1.079, 1.353, 1.857, 0.0}, {4.653, 1.026, 0.0, -1.454, 0.0}, none, none},
      0.0, 0.212, 0.271};
  static constexpr WaveTable int1_planar = {{{6.040, 0.947, 0.938, 1.252, 0.0}, {3.101, 1.079, 0.0, 2.437, 0.0}, none, none},
      0.0, 0.268, 0.214};
  const bool tiled = p.variant == kOpt && !p.input_interleaved;
  if (p.type_in == kInt1) return tiled ? int1_tiled : int1_planar;
  if (bits_of(p.type_in) == 8) return p.input_interleaved ? bits8_pairs : tiled ? bits8_tiled : bits8_planar;
  return p.input_interleaved ? bits16_pairs : tiled ? bits16_tiled : bits16_planar;
}
inline WaveShape wave_choice(const GemmParams &p) {
  const bool bits16 = bits_of(p.type_in) == 16;
  if (p.type_in == kFloat32 || (p.block_tile != 0 && p.block_tile < 5)) return kNoWaves;
  if (p.variant != kOpt || p.input_interleaved) {
    // rows in place: a lane's place among 32 rows is a 32-bit number, and its chunk never longer than the row
    const size_t k_mem = p.k_in_memory ? p.k_in_memory : p.k, planes = p.input_interleaved ? 2 : 1;
    if (planes * k_mem * bits_of(p.type_in) / 8 >= ((size_t)1 << 26) ||
        planes * p.k * bits_of(p.type_in) / 8 < 16) {
      return kNoWaves;
    }
  }
  if (p.block_tile >= 5) return p.block_tile == 5 || !bits16 ? kWaves32x32 : p.block_tile == 6 ? kWaves32x16 : kWaves16x16;
  if (block_choice(p).shape != k64x64) return kNoWaves;
  const WaveTable &table = wave_costs(p);
  const WaveCosts *costs = table.shape;
  const double k_tiles = (double)(p.input_interleaved ? (p.k_tiles + 1) / 2 : p.k_tiles);
  const double units = (double)compute_units();
  // Ragged rows of many K tiles that go through the transposes by default have their waves on the tiles behind them. Where an
  // option has them read in place nevertheless they stay on blocks, with which the break-even points of rows_in_place_pay were
  // measured and which its tests hold it to (fp16 64x320x6598: transposes and waves 30.6 us, in place on blocks 68, on
  // waves 22.5). Rows that are read in place by default: fp16 planar B=55 32x16x7026 93 us on blocks, 24 on waves.
  const bool ragged = (p.variant != kOpt || p.input_interleaved) && p.type_in != kInt1 &&
                      (p.input_interleaved ? 2 : 1) * (size_t)p.k * bits_of(p.type_in) / 8 % 16 != 0;
  if (ragged && k_tiles > 64.0 && !p.in_place_pays) return kNoWaves;
  const double operand_mb = std::max(0.0, 1e-6 * 2.0 * (double)p.batch * ((double)p.nx + (double)p.ny) * (double)p.k *
                                                  bits_of(p.type_in) / 8 - table.cached_mb);
  auto time = [&](int shape, unsigned x, unsigned y) {
    const WaveCosts &c = costs[shape];
    const double n = (double)p.batch * (double)ceil_div(p.nx, x) * (double)ceil_div(p.ny, y) / units;
    if (shape != 0 && n > kWavesPerUnit) return HUGE_VAL;
    const double alone = c.alone * (1.0 + c.second * (std::ceil(n) - 1.0));
    const double beta = shape == 0 && p.have_beta ? table.beta : 0.0;
    const double bytes = operand_mb * (shape != 0 ? table.wave_bytes : table.block_bytes);
    return c.fixed + beta + std::max(bytes, k_tiles * std::max(alone, c.crowded * n)) + c.tile * n;
  };
  if (p.type_in == kInt1) {
    // The four SIMDs of a unit share the K tiles of one tile of C, a unit's tiles one after the other: us on 64 x 64 blocks and
    // like this, 512x512 (a tile a unit) K=2048 7.8, 4.9; K=32768 59.7, 19.2; B=20 128x128 (some units two) K=8192
    // 18.4, 13.9; K=32768 60.3, 33.7; 768x1024 (three) K=8192 19.0, 20.2; K=32768 60.9, 49.4; B=5 1064x128 (three) K=9600 planar 23.8, 30.1.
    const double rounds = std::ceil((double)p.batch * (double)ceil_div(p.nx, 32) * (double)ceil_div(p.ny, 32) / units);
    const double waves = costs[1].tile + std::max(rounds * (costs[1].fixed + costs[1].alone * std::ceil(k_tiles / 4.0)),
                                                 operand_mb * table.wave_bytes);
    return rounds <= 3.0 && waves < time(0, 64, 64) ? kWaves32x32 : kNoWaves;
  }
  double best = time(0, 64, 64);
  WaveShape shape = kNoWaves;
  auto try_shape = [&](WaveShape s, unsigned x, unsigned y) {
    const double t = time(s, x, y);
    if (t < best) best = t, shape = s;
  };
  try_shape(kWaves32x32, 32, 32);
  if (bits16) {
    try_shape(kWaves32x16, 32, 16);
    try_shape(kWaves16x16, 16, 16);
  }
  return shape;
}
// Whether four waves share the K tiles of a tile of C (1-bit input, see wave_choice; a single K tile is not shared out).
inline bool waves_share_k(const GemmParams &p) {
  const size_t tiles = (size_t)p.batch * ceil_div(p.nx, 32) * ceil_div(p.ny, 32);
  return p.type_in == kInt1 && p.k_tiles > 1 && tiles <= 3 * (size_t)compute_units();
}
template <int DT, int TOUT>
hipError_t launch_waves(const GemmParams &p, WaveShape shape, hipStream_t stream) {
  auto launch = [&](auto loader) {
    constexpr int L = decltype(loader)::value;
    if constexpr (DT == kFloat16 || DT == kBfloat16) {
      if (shape == kWaves16x16) return launch_wave<DT, TOUT, L, 1, 1>(p, stream);
      if (shape == kWaves32x16) return launch_wave<DT, TOUT, L, 2, 1>(p, stream);
    }
    if constexpr (DT == kInt1) {
      if (waves_share_k(p)) return launch_wave<DT, TOUT, L, 2, 2, 4>(p, stream);
    }
    return launch_wave<DT, TOUT, L, 2, 2>(p, stream);
  };
  if constexpr (DT != kInt1) {
    if (p.input_interleaved) return launch(std::integral_constant<int, kLoadInterleavedRagged>{});
  }
  if (p.variant == kOpt) return launch(std::integral_constant<int, kLoadTiled>{});
  return launch(std::integral_constant<int, kLoadPlanarRagged>{});
}

// 128 x 128 blocks (16-bit input: of eight or four waves, see block_choice).
template <int DT, int TOUT, int LOADER>
hipError_t launch_128x128(const GemmParams &p, hipStream_t stream) {
  if constexpr (DtypeTraits<DT>::kElemBytes == 2 && DT != kInt1) {
    if (block_choice(p).eight_waves) return launch_block<DT, TOUT, 128, 128, 64, 32, 4, 2, LOADER, 16>(p, stream);
    if constexpr (LOADER != kLoadInterleavedVec && LOADER != kLoadInterleavedRagged) {
      // (exchanged roles for planar C; pairs are regrouped through LDS)
      if (!p.c_interleaved) return launch_block<DT, TOUT, 128, 128, 64, 64, 2, 2, LOADER, 16, true>(p, stream);
    }
    return launch_block<DT, TOUT, 128, 128, 64, 64, 2, 2, LOADER, 16>(p, stream);
  } else {
    return launch_block<DT, TOUT, 128, 128, 64, 64, 2, 2, LOADER, 32>(p, stream);
  }
}

template <int DT, int TOUT>
hipError_t launch_typed(const GemmParams &p, hipStream_t stream) {
  if constexpr (DT != kFloat32) {
    const WaveShape waves = wave_choice(p);
    if (waves != kNoWaves) return launch_waves<DT, TOUT>(p, waves, stream);
  }
  constexpr int KPM = DtypeTraits<DT>::kTilesPerMfma;
  const size_t k_bytes = (size_t)p.k * bits_of(p.type_in) / 8;
  // planar rows made of whole, aligned 16-byte chunks are copied straight into LDS,
  // other rows from 16 bytes on by the ragged loader; what is left goes through the
  // register-staged kernel
  const bool planar_direct = (p.variant == kBasic) && (k_bytes >= 16) && (k_bytes % 16 == 0) &&
                             ((uintptr_t)p.x % 16 == 0) && ((uintptr_t)p.y % 16 == 0);
  const BlockShape shape = block_choice(p).shape;
  constexpr bool BITS16 = DtypeTraits<DT>::kElemBytes == 2;
  constexpr int MS = BITS16 ? 16 : 32;
  if constexpr (DT == kFloat32) {
    // 128 x 128 blocks of 8 waves of 64 x 32, 4-slot ring; 64 x 64 of 4 waves of 32 x 32, 5-slot
    // ring, two blocks a unit. The more a wave computes the fewer elements it splits per matrix
    // instruction: planar pipeline of 8192x8192x1024 3250 and 3900 us. (A wave of 64 x 64, which 256 x 128 blocks
    // have, would need 256 registers for its sums alone.)
    auto launch = [&](auto loader) {
      constexpr int L = decltype(loader)::value;
      if (shape == k64x64) return launch_dtl<DT, TOUT, 64, 64, 32, 32, 5, 2, L, 32>(p, stream);
      return launch_block<DT, TOUT, 128, 128, 64, 32, 4, 2, L, 32>(p, stream);
    };
    const bool aligned = (uintptr_t)p.x % 16 == 0 && (uintptr_t)p.y % 16 == 0;
    if (p.input_interleaved) {
      if (2 * k_bytes < 16) return hipErrorInvalidValue;
      return aligned && 2 * k_bytes % 16 == 0 ? launch(std::integral_constant<int, kLoadInterleavedVec>{})
                                              : launch(std::integral_constant<int, kLoadInterleavedRagged>{});
    }
    if (p.variant == kOpt) return launch(std::integral_constant<int, kLoadTiled>{});
    if (planar_direct) return launch(std::integral_constant<int, kLoadPlanarVec>{});
    if (k_bytes >= 16) return launch(std::integral_constant<int, kLoadPlanarRagged>{});
  }
  else if (p.input_interleaved) {
    // raw (re, im) rows straight from the caller: the host side only takes this
    // path for rows of at least 16 bytes
    const bool ragged = 2 * k_bytes % 16 != 0 || (uintptr_t)p.x % 16 != 0 || (uintptr_t)p.y % 16 != 0;
    if (ragged && 2 * k_bytes < 16) return hipErrorInvalidValue;
    if (ragged) {
      if (shape == k64x64) return launch_dtl<DT, TOUT, 64, 64, 32, 32, 5, 2, kLoadInterleavedRagged, MS>(p, stream);
      if (shape == k128x128) return launch_128x128<DT, TOUT, kLoadInterleavedRagged>(p, stream);
      return launch_block<DT, TOUT, 256, 128, 64, 64, 3, 2, kLoadInterleavedRagged, MS>(p, stream);
    } else if constexpr (BITS16) {
      if (wide_tiles_apply(p) && wide_tiles_pay(p)) return launch_wide<DT, TOUT, true>(p, stream);
      if (shape == k64x64) return launch_dtl<DT, TOUT, 64, 64, 32, 32, 5, 2, kLoadInterleavedVec>(p, stream);
      if (shape == k128x128) return launch_128x128<DT, TOUT, kLoadInterleavedVec>(p, stream);
      return launch_block<DT, TOUT, 256, 128, 64, 64, 3, 2, kLoadInterleavedVec>(p, stream);
    } else {
      if (shape == k64x64) {
        return launch_dtl<DT, TOUT, 64, 64, 32, 32, 5, 2, kLoadInterleavedVec, 32>(p, stream);
      }
      if (shape == k128x128) return launch_128x128<DT, TOUT, kLoadInterleavedVec>(p, stream);
      return launch_block<DT, TOUT, 256, 128, 64, 64, 3, 2, kLoadInterleavedVec, 32>(p, stream);
    }
  }
  else if (p.variant == kOpt || planar_direct) {
    if constexpr (BITS16) {
      // 16-bit input, tiled operands, planar C without beta: 192 x 256 block, 4 waves
      // of 192 x 64 (one per SIMD), where that pays
      if (wide_tiles_apply(p) && wide_tiles_pay(p)) return launch_wide<DT, TOUT>(p, stream);
    }
    if constexpr (BITS16) {
      // 16-bit input: 256 x 128 block, 8 waves of 64 x 64 (two per SIMD), 3-slot ring.
      // Interleaved fp32 C: in the exchanged-roles layout a lane's (re, im) pairs of
      // a row lie 32 bytes apart, so every store instruction would write half
      // cache lines; the other layout regroups the tile through LDS into whole
      // rows of pairs (measured 5 % faster at B=64 512x4096x576).
      if constexpr (TOUT == kFloat32) {
        if (p.variant == kOpt && p.c_interleaved && shape == k256x128) {
          return launch_block<DT, TOUT, 256, 128, 64, 64, 3, 2, kLoadTiled, 16, false>(p, stream);
        }
      }
      // problems too small to give every compute unit a 256 x 128 tile: 128 x 128
      // blocks (launch_128x128), or 64 x 64 blocks, 4 waves of 32 x 32,
      // 5-slot ring, two blocks a unit
      if (shape == k64x64) {
        return p.variant == kOpt
                   ? launch_dtl<DT, TOUT, 64, 64, 32, 32, 5, 2, kLoadTiled, 16>(p, stream)
                   : launch_dtl<DT, TOUT, 64, 64, 32, 32, 5, 2, kLoadPlanarVec, 16>(p, stream);
      }
      if (shape == k128x128) {
        return p.variant == kOpt ? launch_128x128<DT, TOUT, kLoadTiled>(p, stream)
                                 : launch_128x128<DT, TOUT, kLoadPlanarVec>(p, stream);
      }
      return p.variant == kOpt
                 ? launch_block<DT, TOUT, 256, 128, 64, 64, 3, 2, kLoadTiled, 16, true>(p, stream)
                 : launch_block<DT, TOUT, 256, 128, 64, 64, 3, 2, kLoadPlanarVec, 16, true>(p, stream);
    } else {
      // fp8: the 32x32x64 MFMA takes one K tile per instruction, which lets the
      // same block shape and ring as for 16-bit input fit into LDS
      // (small problems: 128 x 128 blocks, 4 waves of 64 x 64, or 64 x 64 blocks, 4 waves
      // of 32 x 32; two blocks a unit)
      if (shape == k64x64) {
        return p.variant == kOpt
                   ? launch_dtl<DT, TOUT, 64, 64, 32, 32, 5, 2, kLoadTiled, 32>(p, stream)
                   : launch_dtl<DT, TOUT, 64, 64, 32, 32, 5, 2, kLoadPlanarVec, 32>(p, stream);
      }
      if (shape == k128x128) {
        return p.variant == kOpt ? launch_128x128<DT, TOUT, kLoadTiled>(p, stream)
                                 : launch_128x128<DT, TOUT, kLoadPlanarVec>(p, stream);
      }
      return p.variant == kOpt
                 ? launch_block<DT, TOUT, 256, 128, 64, 64, 3, 2, kLoadTiled, 32>(p, stream)
                 : launch_block<DT, TOUT, 256, 128, 64, 64, 3, 2, kLoadPlanarVec, 32>(p, stream);
    }
  }
  else if (k_bytes >= 16) {
    if (shape == k64x64) return launch_dtl<DT, TOUT, 64, 64, 32, 32, 5, 2, kLoadPlanarRagged, MS>(p, stream);
    if (shape == k128x128) return launch_128x128<DT, TOUT, kLoadPlanarRagged>(p, stream);
    return launch_block<DT, TOUT, 256, 128, 64, 64, 3, 2, kLoadPlanarRagged, MS, BITS16>(p, stream);
  }
  // fp8 stages are twice as large (two K tiles per MFMA): one wave per SIMD
  // with the full register file
  constexpr int WPE = (KPM == 2) ? 1 : 2;
  return launch_config<DT, TOUT, 128, 128, 64, 64, KPM, kLoadPlanarElem, WPE>(p, stream);
}

}  // namespace

// The instantiations are spread over several translation units so that they
// compile in parallel: gemm_mfma_<part>.hip define CCGLIB_GEMM_MFMA_PART and
// include this file (1 fp16, 2 bf16, 3 fp32, 4 fp8, 5 1-bit input; 0 the
// dispatch below). Included without the macro (the tuning program), the file
// holds everything.
#ifndef CCGLIB_GEMM_MFMA_PART
#define CCGLIB_GEMM_MFMA_PART -1
#endif
#define CCGLIB_GEMM_MFMA_HAS(part) (CCGLIB_GEMM_MFMA_PART == -1 || CCGLIB_GEMM_MFMA_PART == (part))

hipError_t launch_gemm_mfma_f16(const GemmParams &p, hipStream_t stream);
hipError_t launch_gemm_mfma_bf16(const GemmParams &p, hipStream_t stream);
hipError_t launch_gemm_mfma_f32(const GemmParams &p, hipStream_t stream);
hipError_t launch_gemm_mfma_fp8(const GemmParams &p, hipStream_t stream);
hipError_t launch_gemm_mfma_int1(const GemmParams &p, hipStream_t stream);

#if CCGLIB_GEMM_MFMA_HAS(1)
hipError_t launch_gemm_mfma_f16(const GemmParams &p, hipStream_t stream) {
  if (p.type_out == kFloat32) return launch_typed<kFloat16, kFloat32>(p, stream);
  if (p.type_out == kFloat16) return launch_typed<kFloat16, kFloat16>(p, stream);
  return hipErrorInvalidValue;
}
#endif

#if CCGLIB_GEMM_MFMA_HAS(2)
hipError_t launch_gemm_mfma_bf16(const GemmParams &p, hipStream_t stream) {
  if (p.type_out == kFloat32) return launch_typed<kBfloat16, kFloat32>(p, stream);
  if (p.type_out == kBfloat16) return launch_typed<kBfloat16, kBfloat16>(p, stream);
  return hipErrorInvalidValue;
}
#endif

#if CCGLIB_GEMM_MFMA_HAS(3)
hipError_t launch_gemm_mfma_f32(const GemmParams &p, hipStream_t stream) {
  if (p.type_out == kFloat32) return launch_typed<kFloat32, kFloat32>(p, stream);
  if (p.type_out == kFloat16) return launch_typed<kFloat32, kFloat16>(p, stream);
  if (p.type_out == kBfloat16) return launch_typed<kFloat32, kBfloat16>(p, stream);
  return hipErrorInvalidValue;
}
#endif

#if CCGLIB_GEMM_MFMA_HAS(4)
hipError_t launch_gemm_mfma_fp8(const GemmParams &p, hipStream_t stream) {
  if (p.type_out != kFloat32) return hipErrorInvalidValue;
  return p.type_in == kFloat8e4m3 ? launch_typed<kFloat8e4m3, kFloat32>(p, stream)
                                  : launch_typed<kFloat8e5m2, kFloat32>(p, stream);
}
#endif

#if CCGLIB_GEMM_MFMA_HAS(5)
hipError_t launch_gemm_mfma_int1(const GemmParams &p, hipStream_t stream) {
  // packed 1-bit samples expanded in registers; the caller has checked that
  // planar rows are whole aligned 16-byte chunks and that K fits fp32 sums
  if (p.type_out != kInt32 || p.input_interleaved) return hipErrorInvalidValue;
  const WaveShape waves = wave_choice(p);
  if (waves != kNoWaves) return launch_waves<kInt1, kInt32>(p, waves, stream);
  const BlockShape shape = block_choice(p).shape;
  if (shape == k64x64) {
    return p.variant == kOpt
               ? launch_dtl<kInt1, kInt32, 64, 64, 32, 32, 5, 2, kLoadTiled, 32>(p, stream)
               : launch_dtl<kInt1, kInt32, 64, 64, 32, 32, 5, 2, kLoadPlanarVec, 32>(p, stream);
  }
  if (shape == k128x128) {
    return p.variant == kOpt
               ? launch_dtl<kInt1, kInt32, 128, 128, 64, 64, 2, 2, kLoadTiled, 32>(p, stream)
               : launch_dtl<kInt1, kInt32, 128, 128, 64, 64, 2, 2, kLoadPlanarVec, 32>(p, stream);
  }
  return p.variant == kOpt
             ? launch_dtl<kInt1, kInt32, 256, 128, 64, 64, 3, 2, kLoadTiled, 32>(p, stream)
             : launch_dtl<kInt1, kInt32, 256, 128, 64, 64, 3, 2, kLoadPlanarVec, 32>(p, stream);
}
#endif

#if CCGLIB_GEMM_MFMA_HAS(0)
// Which kernel launch_gemm_mfma starts for these parameters (the decisions of
// launch_typed, in words).
const char *describe_gemm_mfma(const GemmParams &p) {
  const bool bits16 = p.type_in == kFloat16 || p.type_in == kBfloat16;
  const bool int1 = p.type_in == kInt1;
  const size_t k_bytes = (size_t)p.k * bits_of(p.type_in) / 8;
  const bool planar_direct = (p.variant == kBasic) && (k_bytes >= 16) && (k_bytes % 16 == 0) &&
                             ((uintptr_t)p.x % 16 == 0) && ((uintptr_t)p.y % 16 == 0);
  const BlockChoice choice = block_choice(p);
  const BlockShape shape = choice.shape;
  const WaveShape waves = wave_choice(p);
  if (waves != kNoWaves) {
    // (a wave's tile, and the region of C whose waves are numbered consecutively)
    const bool pairs = p.input_interleaved, tiled = p.variant == kOpt && !pairs;
    auto by_layout = [&](const char *t, const char *i, const char *r) { return tiled ? t : pairs ? i : r; };
    if (waves == kWaves16x16) {
      return by_layout("complex_gemm_mfma_wave, 16x16 a wave, 16 waves to 64x64, tiled operands",
                       "complex_gemm_mfma_wave, 16x16 a wave, 16 waves to 64x64, interleaved rows",
                       "complex_gemm_mfma_wave, 16x16 a wave, 16 waves to 64x64, planar rows");
    }
    if (waves == kWaves32x16) {
      return by_layout("complex_gemm_mfma_wave, 32x16 a wave, 8 waves to 64x64, tiled operands",
                       "complex_gemm_mfma_wave, 32x16 a wave, 8 waves to 64x64, interleaved rows",
                       "complex_gemm_mfma_wave, 32x16 a wave, 8 waves to 64x64, planar rows");
    }
    if (waves_share_k(p)) {
      return tiled ? "complex_gemm_mfma_wave, 32x32 by four waves along K, 4 tiles to 64x64, tiled operands"
                   : "complex_gemm_mfma_wave, 32x32 by four waves along K, 4 tiles to 64x64, planar rows";
    }
    return by_layout("complex_gemm_mfma_wave, 32x32 a wave, 4 waves to 64x64, tiled operands",
                     "complex_gemm_mfma_wave, 32x32 a wave, 4 waves to 64x64, interleaved rows",
                     "complex_gemm_mfma_wave, 32x32 a wave, 4 waves to 64x64, planar rows");
  }
  auto name = [&](const char *large, const char *middle, const char *eight, const char *small) {
    return shape == k256x128 ? large : shape == k64x64 ? small : choice.eight_waves ? eight : middle;
  };
  if (p.input_interleaved) {
    if (bits16 && wide_tiles_apply(p) && wide_tiles_pay(p)) {
      return "complex_gemm_mfma_wide, 192x256 block, one wave per SIMD, interleaved rows";
    }
    if (2 * k_bytes % 16 != 0 || (uintptr_t)p.x % 16 != 0 || (uintptr_t)p.y % 16 != 0) {
      return name("complex_gemm_mfma_dtl, 256x128 block, ragged interleaved rows",
                  "complex_gemm_mfma_dtl, 128x128 block, ragged interleaved rows",
                  "complex_gemm_mfma_dtl, 128x128 block of eight waves, ragged interleaved rows",
                  "complex_gemm_mfma_dtl, 64x64 block, ragged interleaved rows");
    }
    return name("complex_gemm_mfma_dtl, 256x128 block, interleaved rows",
                "complex_gemm_mfma_dtl, 128x128 block, interleaved rows",
                "complex_gemm_mfma_dtl, 128x128 block of eight waves, interleaved rows",
                "complex_gemm_mfma_dtl, 64x64 block, interleaved rows");
  }
  if (p.variant == kOpt || planar_direct || int1) {
    if (bits16 && wide_tiles_apply(p) && wide_tiles_pay(p)) {
      return "complex_gemm_mfma_wide, 192x256 block, one wave per SIMD";
    }
    if (p.variant == kOpt) {
      return name("complex_gemm_mfma_dtl, 256x128 block, tiled operands",
                  "complex_gemm_mfma_dtl, 128x128 block, tiled operands",
                  "complex_gemm_mfma_dtl, 128x128 block of eight waves, tiled operands",
                  "complex_gemm_mfma_dtl, 64x64 block, tiled operands");
    }
    return name("complex_gemm_mfma_dtl, 256x128 block, planar rows",
                "complex_gemm_mfma_dtl, 128x128 block, planar rows",
                "complex_gemm_mfma_dtl, 128x128 block of eight waves, planar rows",
                "complex_gemm_mfma_dtl, 64x64 block, planar rows");
  }
  if (k_bytes >= 16) {
    return name("complex_gemm_mfma_dtl, 256x128 block, ragged planar rows",
                "complex_gemm_mfma_dtl, 128x128 block, ragged planar rows",
                "complex_gemm_mfma_dtl, 128x128 block of eight waves, ragged planar rows",
                "complex_gemm_mfma_dtl, 64x64 block, ragged planar rows");
  }
  return "complex_gemm_mfma, 128x128 block, planar rows through registers";
}

hipError_t launch_gemm_mfma(const GemmParams &p, hipStream_t stream) {
  switch (p.type_in) {
    case kFloat16: return launch_gemm_mfma_f16(p, stream);
    case kBfloat16: return launch_gemm_mfma_bf16(p, stream);
    case kFloat32: return launch_gemm_mfma_f32(p, stream);
    case kFloat8e4m3:
    case kFloat8e5m2: return launch_gemm_mfma_fp8(p, stream);
    case kInt1: return launch_gemm_mfma_int1(p, stream);
    default: return hipErrorInvalidValue;
  }
}
#endif

}  // namespace ccglib_amd
