// int4 linear layers (layout and arithmetic: int4.hip) for 33 to 64 activation rows on gfx950: the draft's forward over a whole
// 64-node window, as post-speculation runs it (SubSpecSDGeneratorBase, specdecodes/models/generators/subspec_sd_v2.py:32-55).
//
// What bounds it.  A 16 x 64 weight block is 576 bytes of codes and scales, the activations of its 64 k are 8 KB: wavefronts
// that fetch activations for themselves (int4_gemm_kernel, one or two tiles each) move eight times more of those than of
// weights.  Here a workgroup of eight wavefronts shares them: 256 k at a time, 4 groups, activations and weights are copied
// straight into LDS rings; wavefront (h, kg) multiplies tiles h TA .. h TA + TA - 1 with group kg of each chunk, so an operand
// read of 8 KB feeds TA tiles and the four partial sums meet once, at the end.  Requests return in order, so wavefronts 0..3
// copy activations (from the L2, a chunk or two ahead) and 4..7 weights (from HBM, three to seven chunks ahead): neither waits
// behind the other.  A wavefront's requests, operand reads and the scaling of the previous 16 rows are issued between products.
// What remains is the vector ALU: a block is about 50 vector instructions (dequantization; scale and zero point in fp32) and eight
// products, and a wavefront of five tiles issues 268 of the one and 48 of the other per chunk.  They overlap only where they
// stand next to each other in the code: the scaling of 16 rows sits between the two products of a tile of the next 16 (pinned
// there: left to itself the compiler sinks it behind all products, which then wait for each other in pairs), the next chunk's
// codes are dequantized behind the last product of their tile.  37888 x 3584 with the activation, 64 rows: 37.7 -> 34.5 us,
// 3584 x 18944 29.2 -> 28.0; of the 3.2 us, 1.8 is the order and the rest one v_and_or_b32 a code pair instead of two instructions.
#include "dma.h"
#include <algorithm>

namespace subspec {

typedef float it_v4f __attribute__((ext_vector_type(4)));
typedef uint32_t it_u4 __attribute__((ext_vector_type(4)));
typedef uint32_t it_u2 __attribute__((ext_vector_type(2)));
typedef __bf16 it_v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 it_v8h __attribute__((ext_vector_type(8)));

template <int DT>
__device__ __forceinline__ it_v4f it_mfma(it_u4 a, it_u4 b, it_v4f c) {
  if constexpr (DT == SUBSPEC_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(it_v8bf, a), __builtin_bit_cast(it_v8bf, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(it_v8h, a), __builtin_bit_cast(it_v8h, b), c, 0, 0, 0);
}

struct Int4TileParams {
  const uint8_t* x; const uint8_t* wq; const uint8_t* sz; const uint16_t* bias; const uint16_t* residual; uint16_t* y;
  float* partial;
  int M, K; int64_t N;               // N: weight rows (SILU: 2 F, gate rows first)
  int units;                         // workgroups along N
  int splits, chunks_per_split;
};

// SX / SW: slots of the activation and the weight ring
template <int DT, int TA, int SX, int SW, bool SILU>
__global__ __launch_bounds__(512) void int4_tile_kernel(Int4TileParams p) {
  constexpr int kTiles = 2 * TA;
  constexpr uint32_t kXSlot = 32768, kCodes = kTiles * 2048, kSzReq = (kTiles + 3) / 4, kWSlot = kCodes + kSzReq * 1024;
  constexpr uint32_t kWRing = SX * kXSlot;
  constexpr int kWReq = kTiles * 2 + kSzReq;                              // 1 KB requests of a chunk's weights
  constexpr int RX = 8, RW = (kWReq + 3) / 4, R = RX;  // ... of one wavefront
  constexpr int kRingBytes = kWRing + SW * kWSlot, kRedBytes = 2 * 4 * 3 * TA * 1024, kSiluBytes = SILU ? 4 * TA * 1024 : 0;
  constexpr int kLds = kRingBytes > kRedBytes + kSiluBytes ? kRingBytes : kRedBytes + kSiluBytes;
  static_assert(kLds <= 160 * 1024 && SX >= 2 && SW >= 2 && SW >= SX && RW <= RX && (SW - 1) * RW < 64, "LDS, request counter");
  __shared__ __attribute__((aligned(16))) uint8_t lds[kLds];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 15, c = lane >> 4;
  const int kg = wave & 3, h = wave >> 2;
  const int M = p.M, K = p.K, G = K >> 6;
  const int n_tiles = (int)(p.N >> 4), half = n_tiles >> 1;
  const int unit = blockIdx.x % p.units, ks = blockIdx.x / p.units;
  const int st0 = ks * p.chunks_per_split, nst = min(G >> 2, st0 + p.chunks_per_split) - st0;
  // tile tt of the workgroup; tiles past the end repeat the last one and are not stored
  auto tile_of = [&](int tt) {
    if constexpr (SILU) return min(unit * TA + tt % TA, half - 1) + (tt / TA) * half;
    else return min(unit * kTiles + tt, n_tiles - 1);
  };

  // ---- copies.  Wavefronts 0..3: activations, group `kg` of a chunk, request i = rows 8 i .. 8 i + 7; 16-byte piece q of row
  // r sits at q ^ (r / 2) % 8.  Wavefronts 4..7: codes (a request = two groups of one tile) and scales (256 bytes = four groups
  // of four tiles); surplus requests repeat the last one.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const bool xrole = h == 0;
  uint32_t off[R], dst[R];
  bool scales[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    scales[i] = false;
    if (xrole) {
      const int ii = min(i, RX - 1), r = ii * 8 + (lane >> 3), q = (lane & 7) ^ ((r >> 1) & 7);
      off[i] = (uint32_t)(min(r, M - 1) * K * 2 + kg * 128 + q * 16);
      dst[i] = lds0 + kg * 8192 + ii * 1024;
    } else {
      const int q = min(i * 4 + kg, kWReq - 1);
      if (q < kTiles * 2) {
        off[i] = (uint32_t)tile_of(q >> 1) * (uint32_t)(G * 512) + (q & 1) * 1024 + lane * 16;
        dst[i] = lds0 + kWRing + q * 1024;
      } else {
        const int tt = min((q - kTiles * 2) * 4 + (lane >> 4), kTiles - 1);
        off[i] = (uint32_t)tile_of(tt) * (uint32_t)(G * 64) + (lane & 15) * 16;
        dst[i] = lds0 + kWRing + kCodes + (q - kTiles * 2) * 1024;
        scales[i] = true;
      }
    }
  }
  const uint8_t* const main0 = uniform_ptr(xrole ? p.x + (int64_t)st0 * 512 : p.wq + (int64_t)st0 * 2048);
  const uint8_t* const scale0 = uniform_ptr(p.sz + (int64_t)st0 * 256);
  const int main_step = xrole ? 512 : 2048;
  const uint32_t slot_bytes = xrole ? kXSlot : kWSlot;
  const int slots = xrole ? SX : SW;
  // request i of chunk s (past the last chunk: the last one again, into a slot nobody reads any more)
  auto copy = [&](int i, int s, uint32_t slot) __attribute__((always_inline)) {
    const int64_t cs = min(s, nst - 1);
    const uint8_t* src = uniform_ptr(scales[i] ? scale0 + cs * 256 : main0 + cs * main_step);
    const uint32_t to = __builtin_amdgcn_readfirstlane(dst[i] + slot * slot_bytes);
    dma16<false>(to, off[i], src);
  };
  for (int s = 0; s < slots; ++s)
#pragma unroll
    for (int i = 0; i < R; ++i) if (i < RW || xrole) copy(i, s, s);

  it_v4f acc[TA][4];
#pragma unroll
  for (int t = 0; t < TA; ++t)
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) acc[t][mt] = it_v4f{0.f, 0.f, 0.f, 0.f};
  const uint32_t sw = (ln >> 1) & 7;
  const uint8_t* const xop0 = lds + kg * 8192 + ln * 128 + ((2 * c) ^ sw) * 16;
  const uint8_t* const xop1 = lds + kg * 8192 + ln * 128 + ((2 * c + 1) ^ sw) * 16;
  const uint8_t* const wop = lds + kWRing + h * TA * 2048 + kg * 512 + lane * 8;
  const uint8_t* const sop = lds + kWRing + kCodes + h * TA * 256 + kg * 64 + ln * 4;
  // both constants of ((w >> s) & mask) | magic as values the compiler cannot see through, in registers: one v_and_or_b32 (an and
  // and an or with literals otherwise)
  uint32_t kmask = 0x000f000fu, kmagic = DT == SUBSPEC_BF16 ? 0x43004300u : 0x64006400u;
  asm volatile("" : "+s"(kmask), "+v"(kmagic));
  constexpr float kOffset = DT == SUBSPEC_BF16 ? 128.f : 1024.f;
  const uint32_t one2 = DT == SUBSPEC_BF16 ? 0x3f803f80u : 0x3c003c00u;
  const it_u4 ones = it_u4{one2, one2, one2, one2};

  int xs = 0, ws = 0;                                                     // slots of the chunk being multiplied
  it_u2 w[TA];
  uint32_t sz[TA];
  it_u4 x[4][2];
  auto read_w = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < TA; ++t) {
      w[t] = *(const it_u2*)(wop + slot * kWSlot + t * 2048);
      sz[t] = *(const uint32_t*)(sop + slot * kWSlot + t * 256);
    }
  };
  auto read_x = [&](int mt, int slot) __attribute__((always_inline)) {
    x[mt][0] = *(const it_u4*)(xop0 + slot * kXSlot + mt * 2048);
    x[mt][1] = *(const it_u4*)(xop1 + slot * kXSlot + mt * 2048);
  };
  auto sync = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                    // the chunk's operands are in registers
    if (xrole) wait_vmcnt<(SX - 2) * RX>(); else wait_vmcnt<(SW - 2) * RW>();  // the next one has landed
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  if (xrole) wait_vmcnt<(SX - 1) * RX>(); else wait_vmcnt<(SW - 1) * RW>();
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  it_u4 b[TA][2];
  float sc[TA], szo[TA];                                                  // of the chunk whose products were scaled last
  uint32_t szc[TA];                                                       // (scale, zero) words of the chunk being multiplied
  it_v4f raw[2][TA], xsum[2];
  auto dequantize = [&](int t) __attribute__((always_inline)) {
    auto pair = [&](uint32_t v, int sh) { return ((v >> sh) & kmask) | kmagic; };
    const uint32_t w0 = w[t].x, w1 = w[t].y;
    b[t][0] = it_u4{pair(w0, 0), pair(w0, 4), pair(w0, 8), pair(w0, 12)};
    b[t][1] = it_u4{pair(w1, 0), pair(w1, 4), pair(w1, 8), pair(w1, 12)};
  };
  auto scale_tile = [&](int mt, int t) __attribute__((always_inline)) {
#pragma unroll
    for (int rr = 0; rr < 4; ++rr)
      acc[t][mt][rr] = fmaf(sc[t], raw[mt & 1][t][rr], fmaf(szo[t], xsum[mt & 1][rr], acc[t][mt][rr]));
    asm volatile("" : "+v"(acc[t][mt][0]), "+v"(acc[t][mt][1]), "+v"(acc[t][mt][2]), "+v"(acc[t][mt][3]));   // (pinned here)
  };
  read_w(0);
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) read_x(mt, 0);
#pragma unroll
  for (int t = 0; t < TA; ++t) {
    dequantize(t);
    sc[t] = szo[t] = 0.f;
    raw[1][t] = it_v4f{0.f, 0.f, 0.f, 0.f};
  }
  xsum[1] = it_v4f{0.f, 0.f, 0.f, 0.f};
  for (int it = 0; it < nst; ++it) {
    sync();
    const int xn = xs + 1 == SX ? 0 : xs + 1, wn = ws + 1 == SW ? 0 : ws + 1;
    const uint32_t from = xrole ? xs : ws;
#pragma unroll
    for (int t = 0; t < TA; ++t) szc[t] = sz[t];
    read_w(wn);
    // 16 rows at a time; behind their products, so that they are issued while the matrix core works: the scaling of the 16 rows
    // before (of the last 16 of the chunk before, first), the next chunk's operands of these rows, early the copies into the slots
    // that this chunk has left, and at the end, tile by tile behind its last product, the next chunk's codes.  Nothing but the
    // barrier stands between two chunks' products: the two wavefronts of a SIMD run in step, so what one does alone both do.
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
      for (int i = mt * R / 2; i < min((mt + 1) * R / 2, R); ++i) if (i < RW || xrole) copy(i, it + slots, from);
      it_v4f (&r)[TA] = raw[mt & 1];
      xsum[mt & 1] = it_mfma<DT>(x[mt][0], ones, it_v4f{0.f, 0.f, 0.f, 0.f});   // the group's activation sums, rows 4 c + rr
#pragma unroll
      for (int t = 0; t < TA; ++t) {
        r[t] = it_mfma<DT>(x[mt][0], b[t][0], it_v4f{0.f, 0.f, 0.f, 0.f});
        if (t == 0) xsum[mt & 1] = it_mfma<DT>(x[mt][1], ones, xsum[mt & 1]);
        __builtin_amdgcn_sched_barrier(0);
        scale_tile((mt + 3) & 3, t);
        if (mt == 0) {
          sc[t] = f16_bits_to_float(szc[t] & 0xffffu);
          szo[t] = -sc[t] * (f16_bits_to_float(szc[t] >> 16) + kOffset);
          asm volatile("" : "+v"(sc[t]), "+v"(szo[t]));
        }
        __builtin_amdgcn_sched_barrier(0);
        r[t] = it_mfma<DT>(x[mt][1], b[t][1], r[t]);
        if (mt == 3) {
          dequantize(t);
#pragma unroll
          for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(b[t][0][e]), "+v"(b[t][1][e]));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      read_x(mt, xn);
    }
    xs = xn;
    ws = wn;
  }
#pragma unroll
  for (int t = 0; t < TA; ++t) scale_tile(3, t);
  // every copy has landed and every wavefront is done reading the rings: the space is reused
  wait_vmcnt<0>();
  __syncthreads();

  // ---- wavefront (h, kg) sums the four k groups of rows 16 kg .. 16 kg + 15, in group order
  it_v4f own[TA];
  {
    it_v4f* const red = (it_v4f*)lds + (h * 12 * TA) * 64 + lane;         // [h][source kg][slot][t]
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      if (mt == kg) {
#pragma unroll
        for (int t = 0; t < TA; ++t) own[t] = acc[t][mt];
      } else {
#pragma unroll
        for (int t = 0; t < TA; ++t) red[((kg * 3 + ((mt - kg - 1) & 3)) * TA + t) * 64] = acc[t][mt];
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TA; ++t) {
      it_v4f v = it_v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const it_v4f o = q == kg ? own[t] : red[((q * 3 + ((kg - q - 1) & 3)) * TA + t) * 64];
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) v[rr] += o[rr];
      }
      own[t] = v;
    }
  }
  // ---- output: own[t][rr] is row 16 kg + 4 c + rr, column ln of tile t
  const int m0 = 16 * kg + 4 * c;
  if constexpr (SILU) {
    it_v4f* const ex = (it_v4f*)(lds + kRedBytes) + kg * TA * 64 + lane;
    const int64_t F = p.N >> 1;
    auto rounded = [&](int t) {
      const int64_t n = (int64_t)tile_of(h * TA + t) * 16 + ln;
      const float b = p.bias ? Elem<DT>::load(p.bias, n) : 0.f;
      return it_v4f{Elem<DT>::round(own[t][0] + b), Elem<DT>::round(own[t][1] + b), Elem<DT>::round(own[t][2] + b),
                    Elem<DT>::round(own[t][3] + b)};
    };
    if (h == 1) {
#pragma unroll
      for (int t = 0; t < TA; ++t) ex[t * 64] = rounded(t);
    }
    __syncthreads();
    if (h == 1) return;
#pragma unroll
    for (int t = 0; t < TA; ++t) {
      if (unit * TA + t >= half) break;
      const it_v4f gate = rounded(t), up = ex[t * 64];
      const int64_t f = (int64_t)(unit * TA + t) * 16 + ln;
#pragma unroll
      for (int rr = 0; rr < 4; ++rr)
        if (m0 + rr < M) Elem<DT>::store(p.y, (m0 + rr) * F + f, Elem<DT>::round(silu(gate[rr])) * up[rr]);
    }
  } else {
#pragma unroll
    for (int t = 0; t < TA; ++t) {
      const int tile = unit * kTiles + h * TA + t;
      if (tile >= n_tiles) break;
      const int64_t n = (int64_t)tile * 16 + ln;
      const float b = p.bias && p.splits == 1 ? Elem<DT>::load(p.bias, n) : 0.f;
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        if (m0 + rr >= M) continue;
        if (p.splits > 1) p.partial[((int64_t)ks * M + m0 + rr) * p.N + n] = own[t][rr];
        else store_linear_out<DT>(p.y, (m0 + rr) * p.N + n, own[t][rr] + b, p.residual);
      }
    }
  }
}

// ------------------------------------------------------------------ launch shapes
// Tiles of a wavefront, ring slots, and what a chunk takes with the chip full (us; see int4_tile_plan).
#define SUBSPEC_INT4_TILE_SHAPES(X) \
  X(0, 5, 2, 4, 2.10f)              \
  X(1, 2, 3, 6, 1.05f)              \
  X(2, 1, 3, 8, 0.60f)
struct Int4TileShape { int ta; float chunk_us; };
static constexpr Int4TileShape kInt4Shapes[] = {
#define X(ID, TA, SX, SW, US) {TA, US},
    SUBSPEC_INT4_TILE_SHAPES(X)
#undef X
};
struct Int4TilePlan { int shape, units, splits, chunks_per_split; float us; };
// Cheapest (shape, number of K ranges): 4 us for the launch, rounds of one workgroup per compute unit with 2 us for first chunks
// and output; the sum over the ranges 2 us (a launch, or part of the consumer's), 0.2 per range and its fp32 partials at
// 4.5 TB/s.  Fitted to the times of every shape at 78 matrices (512 to 37888 rows of 512 to 18944, weights from HBM) and 33, 48
// and 64 activation rows, on the kernel as it was before the scaling stood between the products: the choice, int4_gemm_kernel included
// (below), took 1.006 times the best one's time in the mean then, 1.11 at worst (4608 x 3584 shape 2 12.7 us, 3584 x 18944 shape 0 in
// eleven ranges 27.7, 37888 x 3584 with the activation shape 0 36.0).  Shape 0 is 4 to 8 % faster since, the others are level; the
// constants have not been fitted again, so matrices near a line may be a few percent from their best choice.
// gate|up never takes shape 2: one pair per workgroup is int4_gemm_kernel's case, several rounds of it lose to shape 1 or 0.
static Int4TilePlan int4_tile_plan(int64_t M, int64_t N, int64_t K, bool silu) {
  Int4TilePlan best{};
  best.us = 1e30f;
  const int chunks = (int)(K / 256);
  const int64_t cols = silu ? N / 32 : N / 16;
  for (int i = 0; i < (silu ? 2 : 3); ++i) {
    const int per = silu ? kInt4Shapes[i].ta : 2 * kInt4Shapes[i].ta;
    const int units = (int)((cols + per - 1) / per);
    for (int s = 1; s <= (silu ? 1 : 16); ++s) {
      const int cps = (chunks + s - 1) / s;
      if ((chunks + cps - 1) / cps != s) continue;
      const int64_t rounds = ((int64_t)units * s + 255) / 256;
      float us = 4.f + (float)rounds * (2.f + (float)cps * kInt4Shapes[i].chunk_us);
      if (s > 1) us += 2.f + 0.2f * (float)s + 2.f * (float)s * (float)M * (float)N * 4.f / 4.5e6f;
      if (us < best.us) best = Int4TilePlan{i, units, s, cps, us};
    }
  }
  return best;
}
// int4_gemm_kernel at the same row counts: rounds of one gate|up pair per workgroup and compute unit; a linear layer of up to 256
// 16-row tiles and K in one range (beyond those it is 0 to 60 % behind at every size measured).
static float int4_gemm_us(int64_t M, int64_t N, int64_t K, bool silu) {
  const int64_t units = silu ? N / 32 : N / 16, groups = K / 64, rounds = (units + 255) / 256;
  if (silu) return 2.5f + (float)rounds * (1.7f + 0.125f * (float)groups) * (rounds > 1 ? 1.f + 0.005f * (float)(M - 48) : 1.f);
  return units <= 256 && groups < 112 ? 2.7f + 0.135f * (float)groups : 1e30f;
}

// Where sharing the activations pays, by the two estimates.  Few tiles of a short K are better off with a workgroup each, which
// is done before the rings have filled: 3584 x 3584 10.2 us in int4_gemm_kernel against 12.7, 2048 x 2048 7.3 against 9.0,
// 4096 x 4096 11.5 against 13.2.  With more, 4608 x 3584 15.2 against 13.3, 3584 x 18944 41 against 27, 37888 x 3584 with the
// activation 46 against 36.
bool int4_tile_applies(int64_t M, int64_t N, int64_t K, bool silu) {
  return M > 32 && M <= 64 && K % 256 == 0 && N % (silu ? 32 : 16) == 0 && int4_tile_plan(M, N, K, silu).us < int4_gemm_us(M, N, K, silu);
}

size_t int4_tile_workspace(int64_t M, int64_t N, int64_t K) {
  const Int4TilePlan pl = int4_tile_plan(M, N, K, false);
  return pl.splits > 1 ? (size_t)pl.splits * M * N * sizeof(float) : 0;
}

template <int DT, bool SILU>
static void launch_int4_tile(Int4TileParams p, const Int4TilePlan& pl, hipStream_t st) {
  p.units = pl.units;
  p.splits = pl.splits;
  p.chunks_per_split = pl.chunks_per_split;
  const dim3 grid((unsigned)(pl.units * pl.splits));
  DominantKernelTimer timer(st);
  switch (pl.shape) {
#define X(ID, TA, SX, SW, US)                                                                           \
  case ID:                                                                                              \
    if constexpr (!SILU || ID < 2)                                                                      \
      hipLaunchKernelGGL((int4_tile_kernel<DT, TA, SX, SW, SILU>), grid, dim3(512), 0, st, p);          \
    break;
    SUBSPEC_INT4_TILE_SHAPES(X)
#undef X
  }
}

int int4_tile_linear(const void* x, const void* wq, const void* sz, const void* bias, const void* residual, void* y, int dtype,
                     int64_t M, int64_t N, int64_t K, bool silu, void* workspace, hipStream_t st) {
  const Int4TilePlan pl = int4_tile_plan(M, N, K, silu);
  const Int4TileParams p{(const uint8_t*)x, (const uint8_t*)wq, (const uint8_t*)sz, (const uint16_t*)bias, (const uint16_t*)residual,
                         (uint16_t*)y, (float*)workspace, (int)M, (int)K, N, 0, 0, 0};
  if (dtype == SUBSPEC_BF16) {
    if (silu) launch_int4_tile<SUBSPEC_BF16, true>(p, pl, st); else launch_int4_tile<SUBSPEC_BF16, false>(p, pl, st);
  } else {
    if (silu) launch_int4_tile<SUBSPEC_F16, true>(p, pl, st); else launch_int4_tile<SUBSPEC_F16, false>(p, pl, st);
  }
  return pl.splits;
}

}  // namespace subspec

extern "C" int subspec_int4_tile_plan(int64_t M, int64_t N, int64_t K, int gate_up, int32_t* plan) {
  using namespace subspec;
  if (!plan || M <= 0 || N <= 0 || K <= 0) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "int4_tile_plan: null pointer or empty size");
  if (!int4_tile_applies(M, N, K, gate_up != 0))
    SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "int4_tile_plan: M=%lld N=%lld K=%lld take another kernel", (long long)M, (long long)N, (long long)K);
  const Int4TilePlan pl = int4_tile_plan(M, N, K, gate_up != 0);
  plan[0] = pl.shape; plan[1] = pl.units; plan[2] = pl.splits;
  return SUBSPEC_OK;
}
