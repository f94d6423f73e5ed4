// Dense 16-bit linear layers for many activation rows on gfx950:
//   y[M, N] = x[M, K] * W[N, K]^T (+ bias) (+ residual),   W row-major bf16 / fp16
// and the gate|up projection of a SwiGLU MLP with the activation in its output stage: the target's projections over a
// large draft tree (1 + 48 * 6 = 289 rows in configs/exp_offloading/subspec_sd_qwen_7b.yaml:16-19, through
// ClassicSDGeneratorBase._tree_decoding, specdecodes/models/generators/classic_sd.py:75-109) and over a prefill.
//
// A workgroup of eight wavefronts multiplies a BM x BN tile (BM activation rows, BN weight rows) with
// v_mfma_f32_16x16x32, the WEIGHT rows as A operand and the activation rows as B operand: both are k-contiguous 16-byte
// pieces of row-major rows, and a lane ends up with four consecutive output columns of one row.  K advances in chunks of
// 64: both operands' chunks are copied straight into LDS rings as whole 128-byte lines (global_load_lds_dwordx4, a
// request moves 8 rows; 16-byte piece p of row r sits at p ^ (r / 2) % 8, conflict-free for the operand reads).
//
// What bounds it (measured on the gate|up projection of a 7B layer, 37888 x 3584):
// * Issue.  A compute unit copies 64 bytes per cycle from the L2 and reads 256 bytes per cycle from LDS, both less than
//   the products of a 256 x 256 tile take, but copies, operand reads and products of a wavefront are issued in order: with
//   the copies in a block behind the barrier and the reads in front of the products, a chunk of that tile cost 3500
//   cycles against 2048 of products.  Here copies and reads are issued BETWEEN the products (a read or a copy every few of
//   them, the operands one 32-k step ahead), and the last chunk is peeled so that no branch sits between products.
// * Distance.  Vector memory returns in order, so an activation chunk requested behind a weight chunk waits for it: with two
//   slots of each ring every chunk waits for a request to HBM (2500 cycles and more).  Three slots of both (256 x 160 at 256
//   rows: 83 -> 73 us), or three of weights and two of activations with the weights requested half a chunk later (256 x 256,
//   2048 rows: 490 -> 441 us), are what LDS holds.  Chunks of 32 k in twice as many slots lose (half-line requests).
// * Output.  A workgroup has its compute unit to itself, so nothing runs beside its output stage: with a division per element and the
//   bias looked up for every 16 rows it took 24 of 449 us at 2048 rows and 4 of 88 at 289 (activation included).
// * Weights from HBM (289 rows; the same with every weight request answered by the L2: 69 instead of 88 us, without any copy 61, without
//   waits for them 81 to 88): requests return in order, and those that wait for HBM hold back the activations behind them.  Neither
//   the order of the chunks, nor 256-byte requests, nor weights laid out tile by tile change that.
// 2048 rows: 405 to 435 us = 1.28 to 1.37 PFLOP/s with the activation included (library GEMM alone: 520 us; an 8192^3 product
// reaches 1.38 PFLOP/s on this card), 289 rows: 84 to 86 us (dense_wide_kernel: 106), 128 rows: 57 us = 4.8 TB/s of weights.
#include "dma.h"
#include <algorithm>
#include <type_traits>

namespace subspec {

typedef float tl_v4f __attribute__((ext_vector_type(4)));
typedef uint32_t tl_u4 __attribute__((ext_vector_type(4)));
typedef uint32_t tl_u2 __attribute__((ext_vector_type(2)));
typedef __bf16 tl_v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 tl_v8h __attribute__((ext_vector_type(8)));

template <int DT>
__device__ __forceinline__ tl_v4f tl_mfma(tl_u4 a, tl_u4 b, tl_v4f c) {
  if constexpr (DT == SUBSPEC_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(tl_v8bf, a), __builtin_bit_cast(tl_v8bf, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(tl_v8h, a), __builtin_bit_cast(tl_v8h, b), c, 0, 0, 0);
}
struct TileParams {
  const uint16_t* x; const uint16_t* w; const uint16_t* bias; const uint16_t* residual; uint16_t* y; float* partial;
  int M, K; int64_t N;               // N: rows of w (SILU: 2 F)
  int tiles_m, tiles_n, splits, chunks_per_split;
  int64_t col0;                      // output column at which the first of the tiles_n tiles begins
};

// LDS of a tile shape: the rings, reused by the output stage
template <int GM, int GN, int GK, int TA, int TB, int SW, int SX, bool SILU>
constexpr int tile_lds() {
  const int rings = SW * GN * TA * 16 * 128 + SX * GM * TB * 16 * 128;
  const int out = GM * GN * GK * 16 * (TA * (SILU ? 16 : 32) + 16), red = GK > 1 ? GM * GN * TA * TB * 1024 : 0;
  return std::max(rings, std::max(out, red));
}

// workgroup `id` of the tiles that p describes
template <int DT, int GM, int GN, int GK, int TA, int TB, int SW, int SX, bool NT, bool SILU>
__device__ __forceinline__ void dense_tile(const TileParams& p, uint8_t* const lds, const int id) {
  constexpr int kWaves = GM * GN * GK;
  constexpr int BM = GM * TB * 16, BN = GN * TA * 16;
  constexpr int kWSlots = BN / 8, kXSlots = BM / 8;                        // 1 KB requests per chunk ...
  constexpr int RW = (kWSlots + kWaves - 1) / kWaves, RX = (kXSlots + kWaves - 1) / kWaves;   // ... of one wavefront
  constexpr uint32_t kWStride = BN * 128, kXStride = BM * 128, kXRing = SW * kWStride;
  constexpr int kOutRow = TA * (SILU ? 16 : 32) + 16;                     // bytes of a parked output row
  static_assert(tile_lds<GM, GN, GK, TA, TB, SW, SX, SILU>() <= 160 * 1024, "LDS");
  static_assert(GK <= 2 && SX >= 2 && (SW == SX || (SW == SX + 1 && GK == 1)) , "k groups, ring depths");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 15, c = lane >> 4;
  const int M = p.M, K = p.K;

  // XCD-aware order: consecutive ids go to different XCDs; each XCD takes a contiguous run of the tile list, rows fastest
  const int total = p.tiles_m * p.tiles_n * p.splits;
  const int xcd = id & 7, per = total >> 3, rem = total & 7;
  // The quotients are pinned to scalar registers: the compiler divides in the vector ALU and would keep the tile's origin, and
  // with it the base address of every copy, in vector registers.  A copy's scalar base then comes out of a vector instruction
  // one to four instructions ahead of it, where the architecture asks for five wait states -- which the compiler inserts in front
  // of its own memory instructions, not in front of assembly text.
  const int lin = xcd * per + min(xcd, rem) + (id >> 3);
  int cell = lin / p.tiles_m;
  asm volatile("" : "+s"(cell));
  int ks = cell / p.tiles_n;
  asm volatile("" : "+s"(ks));
  const int tm = lin - cell * p.tiles_m, tn = cell - ks * p.tiles_n;
  const int m0 = tm * BM;
  const int64_t n0 = p.col0 + (int64_t)tn * (SILU ? BN / 2 : BN);         // SILU: first output column
  const int64_t F = p.N >> 1;
  const int n_chunks = K >> 6;
  const int st0 = ks * p.chunks_per_split, nst = min(n_chunks, st0 + p.chunks_per_split) - st0;

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  // ---- copies: request = 8 rows x 128 bytes; lane -> row lane / 8, position lane % 8 holding piece position ^ (row / 2) % 8
  uint32_t woff[RW], wdst[RW], xoff[RX], xdst[RX];
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int slot = (i * kWaves + wave) % kWSlots;                       // surplus requests repeat earlier ones
    const int r = slot * 8 + (lane >> 3);
    const int pc = (lane & 7) ^ ((r >> 1) & 7);
    int64_t row;
    if constexpr (SILU) {
      const int q = r & 15, f_in = (r >> 4) * 8 + (q >> 2) * 2 + (q & 1);
      row = min(n0 + f_in, F - 1) - n0 + ((q >> 1) & 1) * F;
    } else {
      row = min(n0 + r, p.N - 1) - n0;
    }
    woff[i] = (uint32_t)(row * K * 2 + pc * 16);
    wdst[i] = lds0 + slot * 1024;
  }
#pragma unroll
  for (int i = 0; i < RX; ++i) {
    const int slot = (i * kWaves + wave) % kXSlots;
    const int r = slot * 8 + (lane >> 3);
    const int pc = (lane & 7) ^ ((r >> 1) & 7);
    xoff[i] = (uint32_t)((min(m0 + r, M - 1) - m0) * K * 2 + pc * 16);
    xdst[i] = lds0 + kXRing + slot * 1024;
  }
  const uint8_t* const wbase = (const uint8_t*)(p.w + n0 * K) + (int64_t)st0 * 128;
  const uint8_t* const xbase = (const uint8_t*)(p.x + (int64_t)m0 * K) + (int64_t)st0 * 128;
  // source of chunk s (relative to st0; beyond the last one: the last one again, into a slot nobody reads any more)
  auto chunk_src = [&](const uint8_t* base, int s) { return uniform_ptr(base + (int64_t)min(s, nst - 1) * 128); };
  auto copy_w = [&](int i, const uint8_t* src, uint32_t slot_off) {
    dma16<NT>(__builtin_amdgcn_readfirstlane(wdst[i] + slot_off), woff[i], src);
  };
  auto copy_x = [&](int i, const uint8_t* src, uint32_t slot_off) {
    dma16<false>(__builtin_amdgcn_readfirstlane(xdst[i] + slot_off), xoff[i], src);
  };
  auto fill_w = [&](int s) {
#pragma unroll
    for (int i = 0; i < RW; ++i) copy_w(i, chunk_src(wbase, s), s * kWStride);
  };
  auto fill_x = [&](int s) {
#pragma unroll
    for (int i = 0; i < RX; ++i) copy_x(i, chunk_src(xbase, s), s * kXStride);
  };
  // Order of a wavefront's requests, here and in the loop (they return in order): two slots each: X(c), W(c), ...;
  // three and more: the weights of a chunk half a chunk later than its activations; one weight slot more than
  // activation slots: W(c + 1) behind X(c).
  constexpr bool kWLate = GK == 1 && SW > 2;                               // weights are requested in step 0 of the next chunk
  if constexpr (SW > SX) {
#pragma unroll
    for (int s = 0; s < SX; ++s) { fill_w(s); fill_x(s); }
  } else {
#pragma unroll
    for (int s = 0; s < SX; ++s) {
      fill_x(s);
      if (!kWLate || s < SX - 1) fill_w(s);
    }
  }
  constexpr int kFirstWait = SW > SX ? (SX - 1) * (RX + RW) : kWLate ? (SX - 2) * (RX + RW) + RX : (SX - 1) * (RX + RW);
  constexpr int kWait = SW > SX ? (SX - 1) * RW + (SX - 2) * RX : (SX - 2) * (RX + RW);
  static_assert(kFirstWait < 64, "request counter");

  const int kg = wave / (GM * GN), wmn = wave % (GM * GN), wm = wmn % GM, wn = wmn / GM;
  tl_v4f acc[TA][TB];
#pragma unroll
  for (int i = 0; i < TA; ++i)
#pragma unroll
    for (int k = 0; k < TB; ++k) acc[i][k] = tl_v4f{0.f, 0.f, 0.f, 0.f};
  uint32_t opoff[2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
    opoff[s] = (uint32_t)ln * 128 + ((uint32_t)(4 * (GK == 2 ? kg : s) + c) ^ (uint32_t)((ln >> 1) & 7)) * 16;
  const uint32_t wop = wn * TA * 2048, xop = kXRing + wm * TB * 2048;

  tl_u4 a0[TA], b0[TB], a1[TA], b1[TB];
  int wslot = 0, xslot = 0;                                               // slots of the chunk being multiplied
  // One 32-k step of this wavefront: TB groups of TA products; between the groups, so that they are issued while the
  // matrix core works: the operands of the next step (from wsrc / xsrc) and this wavefront's copies into freed slots.
  auto step = [&](tl_u4 (&A)[TA], tl_u4 (&B)[TB], tl_u4 (&An)[TA], tl_u4 (&Bn)[TB], auto read_c, auto cx_c, auto cw_c,
                  const uint8_t* wsrc, const uint8_t* xsrc, const uint8_t* xg, uint32_t xo, const uint8_t* wg, uint32_t wo)
                  __attribute__((always_inline)) {
    constexpr bool kRead = decltype(read_c)::value, kCx = decltype(cx_c)::value, kCw = decltype(cw_c)::value;
    constexpr int kReads = TA + TB, kReadGroups = TB >= 4 ? TB * 3 / 4 : TB, D = (kCx ? RX : 0) + (kCw ? RW : 0);
#pragma unroll
    for (int k = 0; k < TB; ++k) {
      if constexpr (D > 0) {
#pragma unroll
        for (int d = k * D / TB; d < (k + 1) * D / TB; ++d) {
          if (kCx && d < RX) copy_x(d, xg, xo);
          else copy_w(d - (kCx ? RX : 0), wg, wo);
        }
      }
      if constexpr (kRead) {
        if (k < kReadGroups) {
#pragma unroll
          for (int r = k * kReads / kReadGroups; r < (k + 1) * kReads / kReadGroups; ++r) {
            if (r < TA) An[r] = *(const tl_u4*)(wsrc + r * 2048);
            else Bn[r - TA] = *(const tl_u4*)(xsrc + (r - TA) * 2048);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < TA; ++i) acc[i][k] = tl_mfma<DT>(A[i], B[k], acc[i][k]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto sync = [&](auto wait_c) __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    wait_vmcnt<decltype(wait_c)::value>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  const uint8_t* const wop_p = lds + wop;
  const uint8_t* const xop_p = lds + xop;
  sync(std::integral_constant<int, kFirstWait>{});
#pragma unroll
  for (int i = 0; i < TA; ++i) a0[i] = *(const tl_u4*)(wop_p + opoff[0] + i * 2048);
#pragma unroll
  for (int k = 0; k < TB; ++k) b0[k] = *(const tl_u4*)(xop_p + opoff[0] + k * 2048);
  // the last chunk is peeled off: a branch inside the loop would make the accumulators cross basic blocks
  auto advance = [&]() __attribute__((always_inline)) {
    wslot = wslot + 1 == SW ? 0 : wslot + 1;
    xslot = xslot + 1 == SX ? 0 : xslot + 1;
  };
  auto last_step = [&](tl_u4 (&A)[TA], tl_u4 (&B)[TB]) __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    step(A, B, A, B, no, no, no, nullptr, nullptr, nullptr, 0u, nullptr, 0u);
  };
  if constexpr (GK == 1) {
    for (int it = 0; it < nst - 1; ++it) {
      const uint32_t wcur = wslot * kWStride, xcur = xslot * kXStride;
      const int wprev = wslot == 0 ? SW - 1 : wslot - 1;
      step(a0, b0, a1, b1, yes, no, std::integral_constant<bool, kWLate>{}, wop_p + wcur + opoff[1], xop_p + xcur + opoff[1],
           nullptr, 0u, kWLate ? chunk_src(wbase, it - 1 + SW) : nullptr, wprev * kWStride);
      advance();
      sync(std::integral_constant<int, kWait>{});
      step(a1, b1, a0, b0, yes, yes, std::integral_constant<bool, !kWLate>{}, wop_p + wslot * kWStride + opoff[0],
           xop_p + xslot * kXStride + opoff[0], chunk_src(xbase, it + SX), xcur, kWLate ? nullptr : chunk_src(wbase, it + SW), wcur);
    }
    step(a0, b0, a1, b1, yes, no, no, wop_p + wslot * kWStride + opoff[1], xop_p + xslot * kXStride + opoff[1], nullptr, 0u, nullptr, 0u);
    last_step(a1, b1);
  } else {
    // two wavefront groups share a chunk: group g multiplies its 16-byte pieces 4 g .. 4 g + 3 (32 of the 64 k)
    auto half = [&](tl_u4 (&A)[TA], tl_u4 (&B)[TB], tl_u4 (&An)[TA], tl_u4 (&Bn)[TB], int it) __attribute__((always_inline)) {
      const uint32_t wcur = wslot * kWStride, xcur = xslot * kXStride;
      advance();
      sync(std::integral_constant<int, kWait>{});
      step(A, B, An, Bn, yes, yes, yes, wop_p + wslot * kWStride + opoff[0], xop_p + xslot * kXStride + opoff[0],
           chunk_src(xbase, it + SX), xcur, chunk_src(wbase, it + SW), wcur);
    };
    int it = 0;
    for (; it + 2 < nst; it += 2) {
      half(a0, b0, a1, b1, it);
      half(a1, b1, a0, b0, it + 1);
    }
    if (it + 1 < nst) {
      half(a0, b0, a1, b1, it);
      last_step(a1, b1);
    } else {
      last_step(a0, b0);
    }
  }
  // every copy into the rings has landed and every wavefront is done reading them: the space is reused below
  wait_vmcnt<0>();
  __syncthreads();

  if constexpr (GK == 2) {
    tl_v4f* red = (tl_v4f*)lds + (wmn * TA * TB) * 64 + lane;
    if (kg == 1) {
#pragma unroll
      for (int i = 0; i < TA; ++i)
#pragma unroll
        for (int k = 0; k < TB; ++k) red[(i * TB + k) * 64] = acc[i][k];
    }
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int i = 0; i < TA; ++i)
#pragma unroll
      for (int k = 0; k < TB; ++k) {
        const tl_v4f o = red[(i * TB + k) * 64];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][k][r] += o[r];
      }
  }

  // ---- output.  acc[i][k][r]: row m0 + (wm TB + k) 16 + ln, column (wn TA + i) 16 + 4 c + r of the tile
  if (!SILU && p.splits > 1) {
#pragma unroll
    for (int k = 0; k < TB; ++k) {
      const int m = m0 + (wm * TB + k) * 16 + ln;
      if (m >= M) continue;
      float* row = p.partial + ((int64_t)ks * M + m) * p.N;
#pragma unroll
      for (int i = 0; i < TA; ++i) {
        const int64_t n = n0 + (wn * TA + i) * 16 + 4 * c;
        if (n < p.N) *(float4*)(row + n) = make_float4(acc[i][k][0], acc[i][k][1], acc[i][k][2], acc[i][k][3]);
      }
    }
    return;
  }
  // 16 rows at a time through a wavefront-private LDS block, so that rows leave as 16-byte pieces of whole segments.  Each of a
  // lane's 16 to 100 outputs costs the compute unit eight cycles per instruction while its matrix cores are idle: biases, bounds
  // and addresses that do not depend on the 16 rows are worked out in front of them, and pairs share their conversions.
  constexpr int kCols = SILU ? TA * 8 : TA * 16;                           // output columns of this wavefront
  constexpr int kPieces = kCols / 8, kRounds = (16 * kPieces + 63) / 64;
  // (two k groups: the block lies in the part of the exchange that only this wavefront reads)
  static_assert(GK == 1 || TA * TB * 1024 >= 16 * kOutRow, "output block inside the exchange");
  uint8_t* const mine = lds + (GK == 2 ? wmn * TA * TB * 1024 : wmn * 16 * kOutRow);
  const int64_t ncol0 = n0 + (int64_t)wn * kCols, ncols = SILU ? F : p.N;
  float bias[TA][4];                                                       // of acc[i][.][r]
#pragma unroll
  for (int i = 0; i < TA; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) bias[i][r] = 0.f;
  if (p.bias) {
#pragma unroll
    for (int i = 0; i < TA; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t n = SILU ? n0 + (wn * TA + i) * 8 + 2 * c + (r & 1) : n0 + (wn * TA + i) * 16 + 4 * c + r;
        if (n < ncols) bias[i][r] = Elem<DT>::load(p.bias, SILU && r >= 2 ? F + n : n);
      }
  }
  const uint8_t* from[kRounds];                                            // this lane's pieces of the block ...
  int64_t to[kRounds];                                                     // ... and of the first 16 rows
  int row[kRounds];                                                        // their rows; none: M
#pragma unroll
  for (int q = 0; q < kRounds; ++q) {
    const int pi = q * 64 + lane, r = pi / kPieces, piece = pi % kPieces;
    from[q] = mine + r * kOutRow + piece * 16;
    row[q] = r < 16 && ncol0 + piece * 8 < ncols ? m0 + wm * TB * 16 + r : M;
    to[q] = (int64_t)(m0 + wm * TB * 16 + r) * ncols + ncol0 + piece * 8;
  }
#pragma unroll
  for (int k = 0; k < TB; ++k) {
#pragma unroll
    for (int i = 0; i < TA; ++i) {
      const float v0 = acc[i][k][0] + bias[i][0], v1 = acc[i][k][1] + bias[i][1];
      const float v2 = acc[i][k][2] + bias[i][2], v3 = acc[i][k][3] + bias[i][3];
      const uint32_t lo = pack2<DT>(v0, v1), hi = pack2<DT>(v2, v3);
      if constexpr (SILU) {
        float gate[2], up[2];
        unpack2<DT>(lo, gate);
        unpack2<DT>(hi, up);
        unpack2<DT>(pack2<DT>(silu(gate[0]), silu(gate[1])), gate);
        *(uint32_t*)(mine + ln * kOutRow + i * 16 + c * 4) = pack2<DT>(gate[0] * up[0], gate[1] * up[1]);
      } else {
        *(tl_u2*)(mine + ln * kOutRow + i * 32 + c * 8) = tl_u2{lo, hi};
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < kRounds; ++q) {
      if (row[q] + k * 16 < M) {
        const int64_t at = to[q] + (int64_t)(k * 16) * ncols;
        dec_u4 v = *(const dec_u4*)from[q];
        if (p.residual) {
          float a[8], b[8];
          unpack8<DT>(v, a);
          unpack8<DT>(*(const dec_u4*)(p.residual + at), b);
#pragma unroll
          for (int j = 0; j < 8; ++j) a[j] += b[j];
          v = pack8<DT>(a);
        }
        *(dec_u4*)(p.y + at) = v;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

template <int DT, int GM, int GN, int GK, int TA, int TB, int SW, int SX, bool NT, bool SILU>
__global__ __launch_bounds__(GM * GN * GK * 64) void dense_tile_kernel(TileParams p) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[tile_lds<GM, GN, GK, TA, TB, SW, SX, SILU>()];
  dense_tile<DT, GM, GN, GK, TA, TB, SW, SX, NT, SILU>(p, lds, blockIdx.x);
}

// ------------------------------------------------------------------ launch shapes
// Tile shapes and what a chunk of one takes when the chip is full of them (us, measured on the projections of a 7B layer:
// 4608 / 3584 / 37888 x 3584 and 3584 x 18944 at 65 to 2048 rows).  The shapes of 160 columns cut 37888 rows into 237
// workgroups, one per compute unit; those that serve up to 192 rows request their weights as streaming data while one row tile
// holds all rows, and a weight is read once (128 rows 58.5 -> 53.8 us).  Several row tiles share a weight through the L2, which
// streaming defeats: 11264 x 2048 with the activation at 289 rows, 24 layers, 2.83 -> 2.73 ms without it.
#define SUBSPEC_TILE_SHAPES(X)                      \
  X(0, 2, 4, 1, 4, 8, 3, 2, false, 1.55f)           \
  X(1, 4, 2, 1, 5, 5, 3, 2, false, 1.48f)           \
  X(2, 4, 2, 1, 5, 4, 3, 3, false, 1.10f)           \
  X(3, 4, 2, 1, 5, 3, 4, 3, true, 0.925f)           \
  X(4, 4, 2, 1, 5, 2, 4, 4, true, 0.83f)            \
  X(5, 4, 2, 1, 4, 4, 3, 3, false, 0.90f)           \
  X(6, 2, 4, 1, 4, 4, 3, 3, false, 0.93f)           \
  X(7, 4, 2, 1, 4, 2, 4, 4, false, 0.65f)           \
  X(8, 2, 2, 2, 2, 4, 6, 6, false, 0.40f)
struct TileShape { int bm, bn; float chunk_us; };
static constexpr TileShape kShapes[] = {
#define X(ID, GM, GN, GK, TA, TB, SW, SX, NT, US) {GM * TB * 16, GN * TA * 16, US},
    SUBSPEC_TILE_SHAPES(X)
#undef X
};
constexpr int kNumShapes = sizeof(kShapes) / sizeof(kShapes[0]);
constexpr int kTileMaxSplits = 8;

struct TilePlan {
  int shape, tiles_m, tiles_n, splits, chunks_per_split;
  int tail, tail_tiles_m, tail_tiles_n;                                    // shape of the last columns; none: -1
  float us;
};
// Cheapest (shape, number of K ranges) under: 5.5 us for launch, first chunks and output; rounds of 256 workgroups, one
// per compute unit, of chunk_us per chunk; never less than the weights take from HBM at 6 TB/s; fp32 partials written
// and read back at 4.5 TB/s.  Alone, over the four projections of three layer widths and 65 to 2048 rows (216 sizes), the choice
// takes 1.02 times the best shape's time in the mean, 1.14 at worst at the widths of a 7B layer and 1.33 elsewhere (2048 x 2048 at
// 512 rows, whose K ranges save less than their sum costs).  Constants fitted to those times (1.009, 1.12) lost up to 7 % in
// whole layers, where the sums of the q|k|v and o projections are the next kernel's.  (5.5 TB/s here kept 3584 x 18944 at 95 to
// 128 rows on a shape 14 % slower: 45.2 against 39.5 us at 128; 0.95 us for shape 3 kept 37888 x 3584 with the activation at 321
// to 384 on one 7 % slower: 119 against 112 us at 384.)
// gate|up over several rounds of 256 x 256 tiles: the rounds that fill the chip, and what is left of the columns in the same launch in
// smaller tiles that fill it once more (a last round of the large ones keeps most of the matrix cores idle).  3 us for the second
// set of first chunks.  Over 19 row counts from 300 to 2048 at 37888 x 3584, 28672 x 4096 and 11264 x 2048 this takes a tail at 18
// sizes and is ahead of the best single shape at all of them, by 3 to 11 %: 37888 x 3584 with 1000 rows 238 -> 224 us, 1792 415 ->
// 381, 2048 434 -> 422; 28672 x 4096 with 600 rows 164 -> 148, 2048 382 -> 364; 11264 x 2048 with 1900 rows 91 -> 83.  At three
// sizes that it leaves alone a tail would have been 2 to 5 % faster (28672 x 4096 with 1700 and 1792 rows), elsewhere slower.
#define SUBSPEC_TILE_TAILS(X) X(2) X(4) X(5)
static void with_tail(TilePlan& best, int64_t M, int64_t N, int64_t K) {
  const int chunks = (int)(K / 64);
  const int64_t F = N / 2, tm = (M + kShapes[0].bm - 1) / kShapes[0].bm, tn = (F + kShapes[0].bn / 2 - 1) / (kShapes[0].bn / 2);
  const int64_t rounds = tm * tn / 256, main_n = rounds * 256 / tm, left = F - main_n * (kShapes[0].bn / 2);
  const float hbm_us = 8.f + (float)N * (float)K * 2.f / 6.0e6f;           // as in tile_plan
  if (rounds == 0 || left <= 0) return;
  auto consider = [&](int i) {
    const int64_t tail_m = (M + kShapes[i].bm - 1) / kShapes[i].bm, tail_n = (left + kShapes[i].bn / 2 - 1) / (kShapes[i].bn / 2);
    const float us = std::max(hbm_us, 5.5f + 3.f + (float)chunks * ((float)rounds * kShapes[0].chunk_us +
                                                                    (float)((tail_m * tail_n + 255) / 256) * kShapes[i].chunk_us));
    if (us < best.us) best = TilePlan{0, (int)tm, (int)main_n, 1, chunks, i, (int)tail_m, (int)tail_n, us};
  };
#define X(ID) consider(ID);
  SUBSPEC_TILE_TAILS(X)
#undef X
}

static TilePlan tile_plan(int64_t M, int64_t N, int64_t K, bool silu) {
  TilePlan best{};
  best.us = 1e30f;
  const int chunks = (int)(K / 64);
  const float hbm_us = 8.f + (float)N * (float)K * 2.f / 6.0e6f;
  for (int i = 0; i < kNumShapes; ++i) {
    const int64_t tm = (M + kShapes[i].bm - 1) / kShapes[i].bm, cols = silu ? N / 2 : N, bn = silu ? kShapes[i].bn / 2 : kShapes[i].bn;
    const int64_t tn = (cols + bn - 1) / bn;
    for (int s = 1; s <= (silu ? 1 : kTileMaxSplits); ++s) {
      const int cps = (chunks + s - 1) / s;
      if (s > 1 && (cps < 8 || (chunks + cps - 1) / cps != s)) continue;
      const int64_t rounds = (tm * tn * s + 255) / 256;
      float us = std::max(5.5f + (float)rounds * (float)cps * kShapes[i].chunk_us, hbm_us);
      if (s > 1) us += 1.f + 2.f * (float)s * (float)M * (float)N * 4.f / 4.5e6f;
      if (us < best.us) best = TilePlan{i, (int)tm, (int)tn, s, cps, -1, 0, 0, us};
    }
  }
  return best;
}

// Two shapes in one launch (SwiGLU): workgroups below `first` take the tiles of p, the others those of `tail`.
template <int DT, int TAIL>
__global__ __launch_bounds__(512) void dense_tile_pair_kernel(TileParams p, TileParams tail, int first) {
#define X(ID, GM, GN, GK, TA, TB, SW, SX, NT, US) ID == TAIL ? tile_lds<GM, GN, GK, TA, TB, SW, SX, true>() :
  constexpr int kTailLds = SUBSPEC_TILE_SHAPES(X) 0;
#undef X
#define X(ID, GM, GN, GK, TA, TB, SW, SX, NT, US) ID == 0 ? tile_lds<GM, GN, GK, TA, TB, SW, SX, true>() :
  constexpr int kMainLds = SUBSPEC_TILE_SHAPES(X) 0;
#undef X
  __shared__ __attribute__((aligned(16))) uint8_t lds[std::max(kMainLds, kTailLds)];
  const int id = blockIdx.x;
#define X(ID, GM, GN, GK, TA, TB, SW, SX, NT, US)                                                                      \
  if constexpr (ID == 0) {                                                                                             \
    if (id < first) return dense_tile<DT, GM, GN, GK, TA, TB, SW, SX, false, true>(p, lds, id);                        \
  } else if constexpr (ID == TAIL) {                                                                                   \
    return dense_tile<DT, GM, GN, GK, TA, TB, SW, SX, false, true>(tail, lds, id - first);                             \
  }
  SUBSPEC_TILE_SHAPES(X)
#undef X
}

template <int DT, bool SILU>
static void launch_tile(TileParams p, const TilePlan& pl, hipStream_t st) {
  p.tiles_m = pl.tiles_m;
  p.tiles_n = pl.tiles_n;
  p.splits = pl.splits;
  p.chunks_per_split = pl.chunks_per_split;
  const dim3 grid((unsigned)((int64_t)pl.tiles_m * pl.tiles_n * pl.splits));
  if constexpr (SILU) {
    if (pl.tail >= 0) {
      TileParams t = p;
      t.tiles_m = pl.tail_tiles_m;
      t.tiles_n = pl.tail_tiles_n;
      t.col0 = (int64_t)pl.tiles_n * (kShapes[0].bn / 2);
      const dim3 both(grid.x + (unsigned)(pl.tail_tiles_m * pl.tail_tiles_n));
      switch (pl.tail) {
#define X(ID) case ID: hipLaunchKernelGGL((dense_tile_pair_kernel<DT, ID>), both, dim3(512), 0, st, p, t, (int)grid.x); break;
        SUBSPEC_TILE_TAILS(X)
#undef X
      }
      return;
    }
  }
  switch (pl.shape) {
#define X(ID, GM, GN, GK, TA, TB, SW, SX, NT, US)                                                                       \
  case ID:                                                                                                              \
    if (NT && pl.tiles_m == 1)                                                                                          \
      hipLaunchKernelGGL((dense_tile_kernel<DT, GM, GN, GK, TA, TB, SW, SX, NT, SILU>), grid, dim3(512), 0, st, p);     \
    else                                                                                                                \
      hipLaunchKernelGGL((dense_tile_kernel<DT, GM, GN, GK, TA, TB, SW, SX, false, SILU>), grid, dim3(512), 0, st, p);  \
    break;
    SUBSPEC_TILE_SHAPES(X)
#undef X
  }
}

// More than 64 rows: below, dense_wide_kernel with its four weight slots is level or ahead (64 rows: q|k|v and o together
// 23.3 against 22.8 us here, gate|up 50.3 against 53.4, down 33 against 36 us with their reductions).  16-byte stores of
// whole output pieces; 32-bit offsets inside a tile (a SwiGLU tile spans gate and up rows).
bool tile_applies(int64_t M, int64_t N, int64_t K, bool silu, const void* y, const void* residual) {
  return M > 64 && N % (silu ? 32 : 16) == 0 && K % 64 == 0 && (uintptr_t)y % 16 == 0 && (uintptr_t)residual % 16 == 0 &&
         (silu ? N / 2 + 512 : 512) * K * 2 < ((int64_t)1 << 31) && M < (1 << 24) && N < ((int64_t)1 << 31);
}

size_t tile_workspace(int64_t M, int64_t N, int64_t K) {
  const TilePlan pl = tile_plan(M, N, K, false);
  return pl.splits > 1 ? (size_t)pl.splits * M * N * sizeof(float) : 0;
}

int tile_linear(const void* x, const void* w, const void* bias, const void* residual, void* y, int dtype, int64_t M, int64_t N,
                int64_t K, void* workspace, hipStream_t st, int* splits) {
  const TilePlan pl = tile_plan(M, N, K, false);
  const TileParams p{(const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)bias, (const uint16_t*)residual, (uint16_t*)y,
                     (float*)workspace, (int)M, (int)K, N, 0, 0, 0, 0, 0};
  *splits = pl.splits;
  DominantKernelTimer timer(st);
  if (dtype == SUBSPEC_BF16) launch_tile<SUBSPEC_BF16, false>(p, pl, st);
  else launch_tile<SUBSPEC_F16, false>(p, pl, st);
  return SUBSPEC_OK;
}

int tile_gate_up_silu(const void* x, const void* w, const void* bias, void* act, int dtype, int64_t M, int64_t N, int64_t K,
                      hipStream_t st) {
  TilePlan pl = tile_plan(M, N, K, true);
  with_tail(pl, M, N, K);
  const TileParams p{(const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)bias, nullptr, (uint16_t*)act, nullptr,
                     (int)M, (int)K, N, 0, 0, 0, 0, 0};
  DominantKernelTimer timer(st);
  if (dtype == SUBSPEC_BF16) launch_tile<SUBSPEC_BF16, true>(p, pl, st);
  else launch_tile<SUBSPEC_F16, true>(p, pl, st);
  SUBSPEC_CHECK_HIP(hipGetLastError());
  return SUBSPEC_OK;
}

}  // namespace subspec

extern "C" int subspec_dense_tile_plan(int64_t M, int64_t N, int64_t K, int gate_up, int32_t* plan) {
  using namespace subspec;
  if (!plan || M <= 0 || N <= 0 || K <= 0) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "dense_tile_plan: null pointer or empty size");
  if (!tile_applies(M, N, K, gate_up != 0, nullptr, nullptr))
    SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "dense_tile_plan: M=%lld N=%lld K=%lld outside the tiled kernel's range", (long long)M, (long long)N,
                 (long long)K);
  const TilePlan pl = tile_plan(M, N, K, gate_up != 0);
  plan[0] = pl.shape; plan[1] = pl.tiles_m; plan[2] = pl.tiles_n; plan[3] = pl.splits;
  return SUBSPEC_OK;
}

extern "C" int subspec_dense_tile_tail(int64_t M, int64_t N, int64_t K, int32_t* tail) {
  using namespace subspec;
  int32_t plan[4];
  if (!tail) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "dense_tile_tail: null pointer");
  const int code = subspec_dense_tile_plan(M, N, K, 1, plan);
  if (code != SUBSPEC_OK) return code;
  TilePlan pl = tile_plan(M, N, K, true);
  with_tail(pl, M, N, K);
  tail[0] = pl.tail; tail[1] = pl.tail_tiles_m; tail[2] = pl.tail_tiles_n; tail[3] = pl.tail < 0 ? 0 : pl.tiles_n * (kShapes[0].bn / 2);
  return SUBSPEC_OK;
}
