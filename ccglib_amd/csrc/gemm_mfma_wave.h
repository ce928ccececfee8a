// Complex GEMM for problems too small to fill the chip with 64 x 64 blocks. Included by gemm_mfma.hip.
//
// Every wave is a block of its own and computes 16 x 16, 32 x 16 or (all types) 32 x 32 elements of C, on
// operands that it copies itself into a ring of K tiles in LDS that nobody else uses: it waits for its own
// copies and reads only, and no barrier stands between two K tiles. What a 64 x 64 block spends per
// K tile when it has a compute unit to itself, 0.28 us (16-bit rows of 64 bytes), is not the copies (16 KiB
// at 64 bytes a clock would take 0.11) but the chain of waiting for them, the barrier, the fragment
// reads and the products; a wave of 16 x 16 spends 0.07 us, which is what the four copies
// of a single wave take (one per 45 clocks), and sixteen of them share the work of such a block
// over as many units. Planar fp16 rows, 64 x 64 blocks and 32 x 32, 32 x 16, 16 x 16 waves, in us:
//   256x256x256     6.4, 4.9, 4.3, 3.8      256x256x2048    22.1, 18.4, 12.0, 8.6
//   512x1024x512    9.1, 7.2, 7.3, 8.5      1024x1024x2048  23.5, 29.2, 52.7, 56.2
// The smaller the tile the more bytes a product takes, so that each has its range (wave_choice).
//   The fragments could be loaded straight into registers as well, but the lanes of an MFMA fragment lie in
// 16 or 32 different rows, and an access of 64 lanes in 64 different places takes 64 clocks where one in
// whole 64-byte pieces takes 16: 256x256x4096 16.2 us for 16 x 16 tiles like that, 15.0 as it is here, and
// 57 against 23 with four waves a unit.
#ifndef CCGLIB_AMD_GEMM_MFMA_WAVE_H_
#define CCGLIB_AMD_GEMM_MFMA_WAVE_H_

// The fragments of one K tile of a wave of 16 TX x 16 TY: entries [2 i + p] as in SmallTile.
template <int TX, int TY> struct WaveTile {
  int4_t x[2 * TX], y[2 * TY];
};

// The products of one K tile, for every sum in the order of the larger blocks' steps; behind(n) is issued
// behind the n-th of kWaveProducts<DT, TX, TY> matrix instructions.
template <int DT, int TX, int TY>
constexpr int kWaveProducts = DT == kFloat16 || DT == kBfloat16 ? 4 * TX * TY : DT == kInt1 ? 32 : 4;
#define CCGLIB_PIN __builtin_amdgcn_sched_barrier(0)
template <int DT, bool IL, int TX, int TY, typename Behind>
__device__ __forceinline__ void mma_wave_tile(const WaveTile<TX, TY> &t, float4_t (&acc_re)[TY][TX],
                                              float4_t (&acc_im)[TY][TX],
                                              Behind &&behind) {
  auto frag = [](const int4_t &v) {
    Fragment<DT> f;
    f.v[0] = v;
    return f;
  };
  Fragment<DT> ya[TY][2], yb[TY][2];   // what x of plane or half p is multiplied with for re and for im
#pragma unroll
  for (int j = 0; j < TY; ++j) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      if constexpr (IL) {   // (yr, -yi, ...), (yi, yr, ...)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const unsigned v = (unsigned)t.y[2 * j + p][w];
          ya[j][p].v[0][w] = (int)(v ^ 0x80000000u);
          yb[j][p].v[0][w] = (int)__builtin_amdgcn_alignbit(v, v, 16);
        }
      } else {              // re: xr yr, xi (-yi); im: xr yi, xi yr
        ya[j][p] = p == 0 ? frag(t.y[2 * j]) : negate<DT>(frag(t.y[2 * j + 1]));
        yb[j][p] = frag(t.y[2 * j + 1 - p]);
      }
    }
  }
  static_for<4 * TX * TY>([&](auto n) {
    constexpr int p = n / (2 * TX * TY), j = n / (2 * TX) % TY, i = n / 2 % TX;
    if constexpr (n % 2 == 0) {
      acc_re[j][i] = mfma<DT>(frag(t.x[2 * i + p]), ya[j][p], acc_re[j][i]);
    } else {
      acc_im[j][i] = mfma<DT>(frag(t.x[2 * i + p]), yb[j][p], acc_im[j][i]);
    }
    behind((int)n);
    CCGLIB_PIN;
  });
}
template <int DT, bool IL, typename Behind>
__device__ __forceinline__ void mma_wave_tile(const WaveTile<2, 2> &t, float16_t_ (&acc_re)[1][1],
                                              float16_t_ (&acc_im)[1][1], Behind &&behind) {
  if constexpr (DT == kInt1) {
    static_for<8>([&](auto s) {
      constexpr int u = 2 * (s >> 2), w = s & 3;
      const int4_t x0 = expand_bits(t.x[u][w]), x1 = expand_bits(t.x[u + 1][w]);
      const int4_t y0 = expand_bits(t.y[u][w]), y1 = expand_bits(t.y[u + 1][w]);
      int4_t y1n;
#pragma unroll
      for (int e = 0; e < 4; ++e) y1n[e] = y1[e] ^ (int)0x88888888u;
      acc_re[0][0] = mfma_fp4(x0, y0, acc_re[0][0]);
      behind(4 * s);
      acc_im[0][0] = mfma_fp4(x0, y1, acc_im[0][0]);
      behind(4 * s + 1);
      acc_re[0][0] = mfma_fp4(x1, y1n, acc_re[0][0]);
      behind(4 * s + 2);
      acc_im[0][0] = mfma_fp4(x1, y0, acc_im[0][0]);
      behind(4 * s + 3);
    });
  } else {
    Fragment32 x[2], ya[2], yb[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        x[p].v[u] = t.x[2 * u + p];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if constexpr (IL) {   // (yr, -yi, ...), (yi, yr, ...)
            const unsigned v = (unsigned)t.y[2 * u + p][w];
            ya[p].v[u][w] = (int)(v ^ 0x80008000u);
            yb[p].v[u][w] = (int)__builtin_amdgcn_perm(v, v, 0x02030001u);
          } else {
            ya[p].v[u][w] = t.y[2 * u + p][w] ^ (p ? (int)DtypeTraits<DT>::kSignMask : 0);
            yb[p].v[u][w] = t.y[2 * u + 1 - p][w];
          }
        }
      }
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      acc_re[0][0] = mfma32<DT>(x[p], ya[p], acc_re[0][0]);
      behind(2 * p);
      CCGLIB_PIN;
      acc_im[0][0] = mfma32<DT>(x[p], yb[p], acc_im[0][0]);
      behind(2 * p + 1);
      CCGLIB_PIN;
    }
  }
}
#undef CCGLIB_PIN

// LDS of a wave: seven K tiles of 16 x 16 or three of 32 x 32 are on their way while one is
// multiplied, and the waves of four SIMDs fit a unit.
constexpr int kWaveLdsBytes = 32 * 1024, kWavesPerUnit = 4;
constexpr int wave_ring(int tx, int ty) { return kWaveLdsBytes / (2048 * (tx + ty)); }   // K tiles of the ring

// (LOADER: tiled, or rows in place of any length from 16 bytes on, at any address)
// SPLIT > 1 (1-bit input, whose sums are exact in any order): a block is SPLIT waves, which share the K tiles of one tile of
// C out among them, one after the other, and add their sums up in LDS.
template <int DT, int TOUT, int LOADER, int TX, int TY, int SPLIT = 1>
__global__ __launch_bounds__(64 * SPLIT, 1) void complex_gemm_mfma_wave(const KernelArgs args) {
  static_assert(SPLIT == 1 || DT == kInt1, "sums in another order: whole numbers only");
  static_assert(LOADER == kLoadTiled || LOADER == kLoadPlanarRagged || LOADER == kLoadInterleavedRagged, "");
  constexpr bool IL = LOADER == kLoadInterleavedRagged, TILED = LOADER == kLoadTiled;
  constexpr bool BITS16 = DT == kFloat16 || DT == kBfloat16;
  constexpr int MS = BITS16 ? 16 : 32;
  static_assert(BITS16 || (TX == 2 && TY == 2), "waves lower than 32: 16-bit input");
  constexpr int WX = 16 * TX, WY = 16 * TY, NX = WX / MS, NY = WY / MS;   // the tile, MFMA tiles of it
  constexpr int PLANES = IL ? 1 : 2;
  constexpr int RB = IL ? 128 : kTileRowBytes;   // bytes of a row in one K tile
  constexpr int RPB = 1024 / RB, CPR = RB / 16;  // rows and chunks a row of one copy instruction
  constexpr int RING = wave_ring(TX, TY);
  constexpr int X_BYTES = PLANES * WX * RB, SLOT_BYTES = X_BYTES + PLANES * WY * RB;
  constexpr int XC = X_BYTES / 1024, COPIES = SLOT_BYTES / 1024;   // copy instructions of X, of a K tile
  static_assert(SLOT_BYTES * RING <= kWaveLdsBytes && COPIES * (RING - 1) < 64, "ring, vmcnt range");

  extern __shared__ __attribute__((aligned(1024))) char block_lds[];
  const int lane = threadIdx.x & 63;
  const unsigned part = SPLIT == 1 ? 0 : (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char *lds = block_lds + part * kWaveLdsBytes;
  // (the waves of a 64 x 64 region of C have consecutive numbers, so that they share an L2)
  const TileCoord tc = tile_coord<64 / WY>(args, blockIdx.x);
  const unsigned x0 = tc.block_x * WX, y0 = tc.block_y * WY;

  // ---- copy ----
  const unsigned row_bytes = IL ? 2 * args.k_bytes : args.k_bytes;
  const unsigned row_stride = TILED ? kTileRowBytes : (IL ? 2 : 1) * args.row_stride_bytes;
  const unsigned k_step = TILED ? kTileBytes : RB;
  const unsigned all_k_tiles = TILED ? args.k_tiles : (row_bytes + RB - 1) / RB;
  // this wave's K tiles: part, part + SPLIT, ...
  const unsigned k_tiles = SPLIT == 1 ? all_k_tiles : part < all_k_tiles ? (all_k_tiles - part + SPLIT - 1) / SPLIT : 0;
  const bool partial = !TILED && row_bytes % RB != 0 && (SPLIT == 1 || (all_k_tiles - 1) % SPLIT == part);
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char *)lds;
  const int r = lane / CPR;
  // chunk that this lane fetches of row RPB * rb + r (see the swizzles of complex_gemm_mfma_dtl)
  auto chunk_of = [&](int rb) {
    const int at = IL ? (MS == 32 ? (((rb & 1) << 2) | ((r >> 1) & 3)) : r & 7) : MS == 32 ? (r >> 2) & 3 : (r >> 1) & 3;
    return (unsigned)((lane % CPR) ^ at);
  };
  const char *base[2][2];            // wave-uniform: row 0 of the wave's rows of X and of Y, by plane
  unsigned at[COPIES];               // the lane's chunk of each copy of a K tile, X first
  unsigned last[COPIES];             // ... of the last, partial one, from K tile 0 on
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    const unsigned rows = side ? args.ny : args.nx, row0 = side ? y0 : x0;
    const char *op = (side ? args.y : args.x) + (size_t)tc.b * (side ? args.y_batch_bytes : args.x_batch_bytes);
    if constexpr (TILED) {
      base[side][0] = op + (size_t)(row0 / kTileRows) * args.k_tile_stride * kTileBytes +
                      (row0 % kTileRows) * kTileRowBytes;
      base[side][1] = base[side][0] + kTilePlaneBytes;
    } else {
      base[side][0] = op + (size_t)row0 * row_stride;
      base[side][1] = IL ? base[side][0] : base[side][0] + (size_t)rows * row_stride;
    }
    const int per_plane = (side ? WY : WX) / RPB;
#pragma unroll
    for (int q = 0; q < (side ? COPIES - XC : XC); ++q) {
      const int n = side ? XC + q : q, rb = q % per_plane;
      const unsigned want = RPB * rb + r;   // (rows past the end: never stored)
      const unsigned most = TILED ? want : rows - 1 - row0;
      const unsigned row = (want < most ? want : most) * row_stride;
      at[n] = row + chunk_of(rb) * 16;
      if constexpr (!TILED) {
        const unsigned start = (all_k_tiles - 1) * RB + chunk_of(rb) * 16;
        last[n] = row + (start < row_bytes - 16 ? start : row_bytes - 16);
      }
    }
  }
  // The wave's K tile kt into slot `slot`, instruction n of COPIES. The chunks of a row's last, partial K tile (`end`)
  // come as the 16 bytes that end with them or with the row, whichever comes first (nothing outside
  // the row is read).
  auto copy_one = [&](unsigned kt, unsigned slot, int n, auto end) {
    const int side = n >= XC, q = side ? n - XC : n, plane = q / ((side ? WY : WX) / RPB);
    load_1k_to_lds(decltype(end)::value ? base[side][plane] : base[side][plane] + (size_t)(kt * SPLIT + part) * k_step,
                   decltype(end)::value ? last[n] : at[n], lds_base + slot * SLOT_BYTES + n * 1024);
  };
  auto copy = [&](unsigned kt, unsigned slot, auto end) {
#pragma unroll
    for (int n = 0; n < COPIES; ++n) copy_one(kt, slot, n, end);
  };

  // ---- fragments ----
  // entry [2 i + p]: 16-row MFMA: row 16 i + lane % 16, chunk lane / 16 of plane p (pairs: of half p);
  // 32-row MFMA: row lane % 32, chunk lane / 32 + 2 i of plane p (pairs: 4 p + 2 (lane / 32) + i)
  const int fr = lane % MS, g = lane / MS;
  auto frag_chunk = [&](int i, int p) { return MS == 16 ? (IL ? g + 4 * p : g) : (IL ? 4 * p + 2 * g + i : g + 2 * i); };
  auto frag_off = [&](int i, int p, int plane_bytes) {
    const int sw = IL ? (MS == 32 ? (fr >> 1) & 7 : fr & 7) : MS == 32 ? (fr >> 2) & 3 : (fr >> 1) & 3;
    return (IL ? 0 : p * plane_bytes) + (fr + (MS == 16 ? 16 * i : 0)) * RB + ((frag_chunk(i, p) ^ sw) * 16);
  };
  using Tile = WaveTile<TX, TY>;
  auto read = [&](Tile &t, unsigned slot) {
    const char *from = lds + slot * SLOT_BYTES;
#pragma unroll
    for (int n = 0; n < 2 * TX; ++n) {
      t.x[n] = *reinterpret_cast<const int4_t *>(from + frag_off(n / 2, n % 2, WX * RB));
    }
#pragma unroll
    for (int n = 0; n < 2 * TY; ++n) {
      t.y[n] = *reinterpret_cast<const int4_t *>(from + X_BYTES + frag_off(n / 2, n % 2, WY * RB));
    }
  };
  // (the last, partial K tile) chunks shifted into place, zeros behind the row's end
  auto settle = [&](Tile &t) {
    typedef unsigned long long ulong2_t __attribute__((ext_vector_type(2)));
    auto shifted = [&](int4_t &v, int n) {
      const unsigned start = (all_k_tiles - 1) * RB + frag_chunk(n / 2, n % 2) * 16;
      const unsigned shift = start < row_bytes - 16 ? 0 : (start - (row_bytes - 16)) * 8;
      const ulong2_t u = __builtin_bit_cast(ulong2_t, v);
      ulong2_t o = u;
      if (shift >= 128) {
        o = ulong2_t{0ull, 0ull};
      } else if (shift >= 64) {
        o = ulong2_t{u[1] >> (shift - 64), 0ull};
      } else if (shift > 0) {
        o = ulong2_t{(u[0] >> shift) | (u[1] << (64 - shift)), u[1] >> shift};
      }
      v = __builtin_bit_cast(int4_t, o);
    };
#pragma unroll
    for (int n = 0; n < 2 * TX; ++n) shifted(t.x[n], n);
#pragma unroll
    for (int n = 0; n < 2 * TY; ++n) shifted(t.y[n], n);
  };

  typename AccType<MS>::type acc_re[NY][NX], acc_im[NY][NX];
#pragma unroll
  for (int j = 0; j < NY; ++j) {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      acc_re[j][i] = 0.f;
      acc_im[j][i] = 0.f;
    }
  }

  // C is on its way before the copies are (which are counted from here on), not only when the sums are there: B=16 255x128x256
  // bf16 with beta 7.70 -> 7.19 us.
  constexpr bool FLOAT_C = TOUT != kInt32;
  CPieces<FLOAT_C ? TOUT : kFloat32, NX, NY, MS> c_pieces;
  if (FLOAT_C && args.have_beta) c_pieces.load(args, tc.b, x0, y0, lane);

  const std::true_type end{};
  const std::false_type whole{};
  const unsigned k_whole = k_tiles - (partial ? 1 : 0);
  const unsigned first = k_whole < (unsigned)RING ? k_whole : RING;
#pragma unroll 1
  for (unsigned t = 0; t < first; ++t) copy(t, t, whole);
  if (partial && k_tiles <= (unsigned)RING) copy(k_whole, k_whole, end);
  if (k_tiles > (unsigned)RING) {
    Tile tiles[2];
    unsigned kt = 0, slot = 0;   // K tile that is multiplied, its slot
    // K tiles with a full ring behind them: while tile kt is multiplied, from `now`, the fragments of tile
    // kt + 1 are read into `next`, and its slot (whose reads have landed) is filled again
    auto step = [&](const Tile &now, Tile &next, auto end) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(COPIES * (RING - 2)) : "memory");
      const unsigned refill = slot;
      slot = slot + 1 == RING ? 0 : slot + 1;
      read(next, slot);
      mma_wave_tile<DT, IL>(now, acc_re, acc_im, [&](int n) {
        constexpr int PRODUCTS = kWaveProducts<DT, TX, TY>;
#pragma unroll
        for (int c = 0; c < COPIES; ++c) {
          if (c * PRODUCTS / (COPIES) == n) copy_one(kt + RING, refill, c, end);
        }
      });
      ++kt;
    };
    // `now` holds a tile, and RING - 1 further ones are on their way
    auto rest = [&](Tile &a, Tile &b) {
      static_for<RING>([&](auto n) {
        constexpr int left = RING - 1 - n;   // tiles behind this one
        Tile &now = n % 2 ? b : a, &next = n % 2 ? a : b;
        if constexpr (left > 0) {
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COPIES * (left - 1)) : "memory");
          slot = slot + 1 == RING ? 0 : slot + 1;
          read(next, slot);
        }
        if (left == 0 && partial) settle(now);
        mma_wave_tile<DT, IL>(now, acc_re, acc_im, [](int) {});
      });
    };
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COPIES * (RING - 1)) : "memory");
    read(tiles[0], 0);
#pragma unroll 1
    for (; kt + RING + 1 < k_whole;) {
      step(tiles[0], tiles[1], whole);
      step(tiles[1], tiles[0], whole);
    }
    // (at most one more whole tile to copy, and the partial one)
    if (kt + RING < k_whole) {
      step(tiles[0], tiles[1], whole);
      tiles[0] = tiles[1];
    }
    if (partial) {
      step(tiles[0], tiles[1], end);
      tiles[0] = tiles[1];
    }
    rest(tiles[0], tiles[1]);
  } else {
    static_for<RING>([&](auto n) {
      constexpr int left = RING - 1 - n;
      if ((unsigned)left < k_tiles) {
        Tile now;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COPIES * left) : "memory");
        read(now, k_tiles - 1 - left);
        if (left == 0 && partial) settle(now);
        mma_wave_tile<DT, IL>(now, acc_re, acc_im, [](int) {});
      }
    });
  }
  if constexpr (SPLIT > 1) {
    // The first wave's registers take the sums of the others, through the LDS of their rings (whose reads
    // have landed: their last products are in the sums).
    float *sums = reinterpret_cast<float *>(lds);
    if (part > 0) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        sums[e * 64 + lane] = acc_re[0][0][e];
        sums[(16 + e) * 64 + lane] = acc_im[0][0][e];
      }
    }
    __syncthreads();
    if (part > 0) return;
#pragma unroll
    for (int s = 1; s < SPLIT; ++s) {
      const float *other = reinterpret_cast<const float *>(block_lds + s * kWaveLdsBytes);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        acc_re[0][0][e] += other[e * 64 + lane];
        acc_im[0][0][e] += other[(16 + e) * 64 + lane];
      }
    }
  }
  if constexpr (TOUT == kInt32) {
    store_wave_tile_int32<NX, NY, MS>(args, tc.b, x0, y0, lane, acc_re, acc_im);
  } else {
    store_wave_tile<TOUT, NX, NY, MS>(args, tc.b, x0, y0, lane, acc_re, acc_im, c_pieces);
  }
}

#endif  // CCGLIB_AMD_GEMM_MFMA_WAVE_H_
