// One decoder layer over the tree rows, launched from one host call: the substitute draft's int4
// layer, and the target's layer with dense 16-bit projections (same sequence, see the end).
//
// The reference runs the draft as a HuggingFace Qwen2 / Llama decoder layer whose seven projections
// were replaced by HQQ int4 linears (specdecodes/helpers/recipes/subspec/hqq_4bit_postspec.py:17-58)
// and hides the per-module launch cost behind torch.compile / captured graphs
// (specdecodes/models/draft_models/classic_sd.py:85-118 for the step it repeats per tree level).
// Here the layer is a fixed sequence of launches issued by native code on the caller's stream:
//   h      = rmsnorm(x) * w_in
//   qkv    = int4(h) + bias                     [M, (Hq + 2 Hkv) D]
//   q, K/V = rope(qkv), K and V rows written into the static cache at cache_rows
//   a      = tree attention(q, cache)           [M, Hq D]
//   x     += int4(a)                            (o_proj; the add is fused into the next rmsnorm)
//   h      = rmsnorm(x) * w_post
//   act    = silu(gate) * up,  gate|up = int4(h)
//   x     += int4(act)                          (down_proj; the add is fused into its output stage)
// Rounding follows the eager torch layer: every intermediate tensor is rounded to the activation
// dtype where torch would materialise it (normalised activations before the weight product, the
// two rotary products and their sum, silu before the product with `up`, both residual sums).
//
// The target model's layer in the tree-decoding forward (HF Qwen2DecoderLayer under
// ClassicSDGeneratorBase._tree_decoding, specdecodes/models/generators/classic_sd.py:75-109) is the
// same sequence with dense 16-bit projections (dense.hip) in place of the int4 ones.  A chunk of a prompt (generators/base.py:204-263)
// is that sequence with causal attention and any number of rows.
#include "common.h"
#include <algorithm>

namespace subspec {

// x[m] (+= delta[m], rounded, written back) ; y[m] = w * round(x * rsqrt(mean(x^2) + eps))
// One workgroup per row; H % 8 == 0, P 16-byte pieces per thread cover H <= THREADS * 8 * P.
// splits > 0: delta is not a 16-bit tensor yet but `splits` fp32 partial sums [splits][rows][H] of a projection whose K
// was split over workgroups; they are summed in split order and rounded here (what the projection's own reduction
// launch would have stored), which saves that launch.
// A launch of this size is a chain of memory round trips and nothing else, so there are as few as can be before the sum of squares:
// one for the row, the gain and the first four partials together, one more for every further four.  In the
// target's forward over 64 rows, with the partials of the o projection: 5.4 us with the gain behind the sum and the partials one
// after the other, 4.9 now (289 rows 6.0, with six partials of the down projection as well 7.5); an empty launch takes 3.0.
// Few rows take as many threads as there are pieces (64 rows, 3584 wide: 2.6 us with 512 threads, 2.8 with 256 and two pieces each).  Where
// that leaves threads without a piece, from 512 rows on the loads of all workgroups count: small ones, and no more pieces than the
// row has.  2048 rows, bf16, 512 threads with one or four pieces -> this: 896 wide 4.6 -> 3.6 us, 4104 8.9 -> 6.9, 5120 9.2 -> 7.6, 6144
// 10.0 -> 8.4 (256 threads and up to eight pieces, a test around each, before the loads moved up: 4.3, 7.7, 8.8, 10.3); 4096 wide,
// 256 threads and two pieces, 6.9 -> 6.8 alone and level in a forward, stays at 512.
constexpr int kNormMaxHidden = 16384;
template <int DT, bool kAdd, int THREADS, int P>
__global__ __launch_bounds__(THREADS) void add_rmsnorm_kernel(uint16_t* __restrict__ x, const uint16_t* __restrict__ delta,
                                                                   const uint16_t* __restrict__ w, uint16_t* __restrict__ y,
                                                                   int H, float eps, const float* __restrict__ partial,
                                                                   int splits) {
  __shared__ float scratch[THREADS / kWave];
  const int m = blockIdx.x, tid = threadIdx.x, pieces = H / 8;
  dec_u4* xr = (dec_u4*)(x + (int64_t)m * H);
  dec_u4 xv[P], gain[P];
  float v[P][8];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int i = min(p * THREADS + tid, pieces - 1);
    xv[p] = xr[i];
    gain[p] = ((const dec_u4*)w)[i];
  }
  if constexpr (kAdd) {
    if (splits > 0) {
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int j = 0; j < 8; ++j) v[p][j] = 0.f;
      for (int s0 = 0; s0 < splits; s0 += 4) {
        float4 q[P][4][2];
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const int i = min(p * THREADS + tid, pieces - 1);
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            const float4* pp = (const float4*)(partial + ((int64_t)min(s0 + s, splits - 1) * gridDim.x + m) * H) + 2 * i;
            q[p][s][0] = pp[0];
            q[p][s][1] = pp[1];
          }
        }
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
          for (int s = 0; s < 4; ++s)
            if (s0 + s < splits) {
              const float4 a = q[p][s][0], b = q[p][s][1];
              v[p][0] += a.x; v[p][1] += a.y; v[p][2] += a.z; v[p][3] += a.w;
              v[p][4] += b.x; v[p][5] += b.y; v[p][6] += b.z; v[p][7] += b.w;
            }
      }
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int j = 0; j < 8; ++j) v[p][j] = Elem<DT>::round(v[p][j]);
    } else {
#pragma unroll
      for (int p = 0; p < P; ++p) unpack8<DT>(((const dec_u4*)(delta + (int64_t)m * H))[min(p * THREADS + tid, pieces - 1)], v[p]);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int i = p * THREADS + tid;
    float xf[8];
    unpack8<DT>(xv[p], xf);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[p][j] = kAdd ? Elem<DT>::round(xf[j] + v[p][j]) : xf[j];
      // an fp16 value is taken as a float from here on: both forms of the kernel then compile to the same products (left to itself
      // the compiler folds the widening into mixed-precision ones in one of them, which round once instead of twice)
      if constexpr (DT == SUBSPEC_F16) asm volatile("" : "+v"(v[p][j]));
    }
    if (i < pieces) {
      if constexpr (kAdd) xr[i] = pack8<DT>(v[p]);
#pragma unroll
      for (int j = 0; j < 8; ++j) ss = fmaf(v[p][j], v[p][j], ss);
    }
  }
  const float tot = block_sum<THREADS>(ss, scratch);
  const float r = rsqrtf(tot / (float)H + eps);
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int i = p * THREADS + tid;
    if (i < pieces) {
      float wv[8], o[8];
      unpack8<DT>(gain[p], wv);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = wv[j] * Elem<DT>::round(v[p][j] * r);
      ((dec_u4*)(y + (int64_t)m * H))[i] = pack8<DT>(o);
    }
  }
}
// delta null and splits 0: a plain RMSNorm (x is only read)
template <int DT>
static void launch_norm(uint16_t* x, const uint16_t* delta, const void* w, uint16_t* y, int64_t rows, int H, float eps,
                        const float* partial, int splits, hipStream_t st) {
  auto launch = [&](auto threads, auto p) {
    constexpr int kThreads = decltype(threads)::value, kP = decltype(p)::value;
    if (delta || splits > 0)
      hipLaunchKernelGGL((add_rmsnorm_kernel<DT, true, kThreads, kP>), dim3((unsigned)rows), dim3(kThreads), 0, st, x, delta,
                         (const uint16_t*)w, y, H, eps, partial, splits);
    else
      hipLaunchKernelGGL((add_rmsnorm_kernel<DT, false, kThreads, kP>), dim3((unsigned)rows), dim3(kThreads), 0, st, x, delta,
                         (const uint16_t*)w, y, H, eps, partial, splits);
  };
#define SUBSPEC_NORM(THREADS, P) launch(std::integral_constant<int, THREADS>{}, std::integral_constant<int, P>{})
  if (H <= 2048) SUBSPEC_NORM(256, 1);
  else if (H <= 4096) SUBSPEC_NORM(512, 1);
  else if (H <= 8192 && rows >= 512) {
    if (H <= 6144) SUBSPEC_NORM(256, 3);
    else SUBSPEC_NORM(256, 4);
  }
  else if (H <= 8192) SUBSPEC_NORM(512, 2);
  else if (H <= 12288) SUBSPEC_NORM(512, 3);
  else SUBSPEC_NORM(512, 4);
#undef SUBSPEC_NORM
}

// act[m, f] = round(silu(gate)) * up with gate = gu[m, f], up = gu[m, F + f]
template <int DT>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ gu, uint16_t* __restrict__ act, int F,
                                                       int64_t pieces) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= pieces) return;
  const int per_row = F / 8;
  const int64_t m = i / per_row;
  const int p = (int)(i % per_row);
  float g[8], u[8];
  unpack8<DT>(((const dec_u4*)(gu + m * 2 * F))[p], g);
  unpack8<DT>(((const dec_u4*)(gu + m * 2 * F + F))[p], u);
#pragma unroll
  for (int j = 0; j < 8; ++j) g[j] = Elem<DT>::round(silu(g[j])) * u[j];
  ((dec_u4*)(act + m * F))[p] = pack8<DT>(g);
}

// Rotary embedding (rotate-half form, angle = position * theta^(-2i/D)) of the q and k heads of
// qkv [M, (Hq + 2 Hkv) * D]; q goes to q_out [Hq, M, D], k and v to rows cache_rows[m] of the
// layer's [Hkv, S, D] caches (D = 128).
// splits > 0: qkv is still `splits` fp32 partial sums [splits][M][(Hq + 2 Hkv) * D] of the projection (K split over
// workgroups) and `bias` its bias; sum, bias and the rounding to the activation dtype happen here instead of in a
// reduction launch of their own.
// A thread takes dims i, i + 1 and their partners D/2 further, 32 lanes a head, eight heads a workgroup; blockIdx.y strides over
// the groups of eight, so that many rows evaluate their angles once per thread and not once per head.  Bound by launch and round
// trips up to a few hundred rows (64: 4.8 -> 4.7 us, 256: 7.4 -> 6.2 against one wavefront per (row, head)), then by its 38 MB and
// the angles: a workgroup that takes a whole row evaluates each once and requests five groups of heads at a time.
// 2048 rows of 36 heads 19.7 -> 11.8 us against a wavefront per (row, head), 13.3 -> 10.0 with both of these.
constexpr int kRopeHeads = 8;
template <int DT>
__global__ __launch_bounds__(32 * kRopeHeads) void rope_write_kernel(const uint16_t* __restrict__ qkv, const int32_t* __restrict__ positions,
                                                                     const int32_t* __restrict__ cache_rows, uint16_t* __restrict__ q_out,
                                                                     KvRowMap kv, int M, int Hq, int Hkv, float log2_theta,
                                                                     const float* __restrict__ inv_freq_table,
                                                                     const float* __restrict__ partial, int splits,
                                                                     const uint16_t* __restrict__ bias) {
  constexpr int D = 128, half = D / 2;
  const int m = blockIdx.x, i = 2 * (threadIdx.x & 31), heads = Hq + 2 * Hkv;
  const int64_t width = (int64_t)heads * D;
  const int pos = positions[m], cache_row = cache_rows[m];
  // the caller's table (the values its other code paths use, so that both write identical rows), else theta^(-2i/D)
  auto frequency = [&](int d) { return inv_freq_table ? inv_freq_table[d] : exp2f(-(float)(2 * d) / (float)D * log2_theta); };
  auto angle = [&](float freq, float* sine, float* cosine) {
    sincosf((float)pos * freq, sine, cosine);
    *cosine = Elem<DT>::round(*cosine);
    *sine = Elem<DT>::round(*sine);
  };
  float c[2], s[2];
  auto rotate_and_store = [&](int hh, float (&lo)[2], float (&hi)[2]) {
    uint16_t* dst;
    if (hh < Hq) {
      dst = q_out + ((int64_t)hh * M + m) * D;
    } else {
      // a row outside the layer's cache is dropped: a bad rows tensor must not write beyond the cache
      uint16_t *kp, *vp;
      if (!kv_row_ptrs(kv, (hh - Hq) % Hkv, cache_row, &kp, &vp)) return;
      dst = hh < Hq + Hkv ? kp : vp;
    }
    if (hh < Hq + Hkv) {                                  // value heads are copied
      // t * cos + rotate_half(t) * sin, each product and the sum rounded like the eager tensor ops
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float a = lo[e], b = hi[e];
        lo[e] = Elem<DT>::round(a * c[e]) + Elem<DT>::round(-b * s[e]);
        hi[e] = Elem<DT>::round(b * c[e]) + Elem<DT>::round(a * s[e]);
      }
    }
    *(uint32_t*)(dst + i) = pack2<DT>(lo[0], lo[1]);
    *(uint32_t*)(dst + i + half) = pack2<DT>(hi[0], hi[1]);
  };
  if (splits == 0 && gridDim.y == 1) {
    // all heads of a row: five groups' elements are requested before the first is used, and an angle is evaluated once
    __shared__ float sine[half], cosine[half];
    constexpr int kBatch = 5;
    const uint16_t* const src = qkv + (int64_t)m * width + i;
    const int group = threadIdx.x >> 5, dim = threadIdx.x & (half - 1);
    const float freq = frequency(dim);
    bool first = true;
    for (int h0 = 0; h0 < heads; h0 += kBatch * kRopeHeads) {              // (uniform: a barrier in the first round)
      uint32_t raw[kBatch][2];
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        const uint16_t* const head = src + (int64_t)min(h0 + k * kRopeHeads + group, heads - 1) * D;
        raw[k][0] = *(const uint32_t*)head;
        raw[k][1] = *(const uint32_t*)(head + half);
      }
      if (first) {
        first = false;
        if (threadIdx.x < half) angle(freq, &sine[dim], &cosine[dim]);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 2; ++e) { s[e] = sine[i + e]; c[e] = cosine[i + e]; }
      }
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        const int hh = h0 + k * kRopeHeads + group;
        if (hh >= heads) break;
        float lo[2], hi[2];
        unpack2<DT>(raw[k][0], lo);
        unpack2<DT>(raw[k][1], hi);
        rotate_and_store(hh, lo, hi);
      }
    }
    return;
  }
  float freq[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) freq[e] = frequency(i + e);
  bool angles = false;
  for (int hh = blockIdx.y * kRopeHeads + (threadIdx.x >> 5); hh < heads; hh += gridDim.y * kRopeHeads) {
    const int64_t col = (int64_t)hh * D + i;
    // the head's elements (or its first four partials) are requested, the angles evaluated while they travel
    uint32_t raw[2] = {0, 0};
    float bl[2] = {0.f, 0.f}, bh[2] = {0.f, 0.f};
    dec_f2 a[4], b[4];
    auto request = [&](int s0) {
#pragma unroll
      for (int sp = 0; sp < 4; ++sp) {
        const float* pp = partial + ((int64_t)min(s0 + sp, splits - 1) * M + m) * width + col;
        a[sp] = *(const dec_f2*)pp;
        b[sp] = *(const dec_f2*)(pp + half);
      }
    };
    if (splits > 0) {
      request(0);
      if (bias) {                                       // (element loads: the bias may lie at any even address)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          bl[e] = Elem<DT>::load(bias, col + e);
          bh[e] = Elem<DT>::load(bias, col + half + e);
        }
      }
    } else {
      const uint16_t* src = qkv + (int64_t)m * width + col;
      raw[0] = *(const uint32_t*)src;
      raw[1] = *(const uint32_t*)(src + half);
    }
    if (!angles) {
      angles = true;
#pragma unroll
      for (int e = 0; e < 2; ++e) angle(freq[e], &s[e], &c[e]);
    }
    float lo[2], hi[2];
    if (splits > 0) {
      lo[0] = lo[1] = hi[0] = hi[1] = 0.f;
      for (int s0 = 0;;) {
#pragma unroll
        for (int sp = 0; sp < 4; ++sp)
          if (s0 + sp < splits) { lo[0] += a[sp][0]; lo[1] += a[sp][1]; hi[0] += b[sp][0]; hi[1] += b[sp][1]; }
        if ((s0 += 4) >= splits) break;
        request(s0);
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        lo[e] = Elem<DT>::round(lo[e] + bl[e]);
        hi[e] = Elem<DT>::round(hi[e] + bh[e]);
      }
    } else {
      unpack2<DT>(raw[0], lo);
      unpack2<DT>(raw[1], hi);
    }
    rotate_and_store(hh, lo, hi);
  }
}

// Rows 0 .. rows - 1 of a paged layer as contiguous [Hkv, rows, 128] K and V: a prefill's attention reads every row many
// times, so one copy (4 MB at 2048 rows of four heads) lets it run on the contiguous kernel, with the contiguous cache's bits.
__global__ __launch_bounds__(256) void gather_pages_kernel(KvRowMap kv, int64_t rows, dec_u4* __restrict__ k_out,
                                                           dec_u4* __restrict__ v_out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;               // 16-byte piece i % 16 of (row, head)
  const int64_t row = i / (16 * kv.hkv);
  if (row >= rows) return;
  const int piece = (int)(i & 15), head = (int)(i / 16 % kv.hkv);
  uint16_t *k, *v;
  if (!kv_row_ptrs(kv, head, row, &k, &v)) return;
  const int64_t o = ((int64_t)head * rows + row) * 16 + piece;
  k_out[o] = ((const dec_u4*)k)[piece];
  v_out[o] = ((const dec_u4*)v)[piece];
}

// rows of one call: the int4 stack serves draft levels and post-verify windows, the dense stack also whole large trees
constexpr int kInt4LayerMaxRows = 64, kDenseLayerMaxRows = 384, kPrefillMaxRows = 65536;
struct LayerPlan {
  size_t h, qkv, q, a, o, gu, act, kv, sub, sub_bytes, total;
};
static LayerPlan layer_plan(const subspec_decoder_layer_dims& s, bool causal = false) {
  LayerPlan p;
  const size_t es = 2, M = (size_t)s.n_rows, H = (size_t)s.hidden, Q = (size_t)s.n_q_heads * s.head_dim,
               KV = (size_t)s.n_kv_heads * s.head_dim, F = (size_t)s.intermediate;
  size_t off = 0;
  auto take = [&](size_t bytes) { size_t o = off; off += align_up(bytes, 256); return o; };
  p.h = take(M * H * es);
  p.qkv = take(M * (Q + 2 * KV) * es);
  p.q = take(M * Q * es);
  p.a = take(M * Q * es);
  p.o = take(M * H * es);
  // (a prefill's gate|up projection always ends in the activation)
  p.gu = take(causal ? 0 : M * 2 * F * es);
  p.act = take(M * F * es);
  p.kv = take(causal && s.page_indices ? 2 * KV * (size_t)(s.prefix_len + s.n_rows) * es : 0);
  size_t sub = 256;
  if (!causal && s.n_rows <= kInt4LayerMaxRows) {                 // wider windows are dense only
    sub = std::max(sub, subspec_int4_linear_workspace(s.n_rows, Q + 2 * KV, H));
    sub = std::max(sub, subspec_int4_linear_workspace(s.n_rows, H, Q));
    sub = std::max(sub, subspec_int4_linear_workspace(s.n_rows, 2 * F, H));
    sub = std::max(sub, subspec_int4_linear_workspace(s.n_rows, H, F));
  }
  sub = std::max(sub, subspec_dense_linear_workspace(s.n_rows, Q + 2 * KV, H));
  sub = std::max(sub, subspec_dense_linear_workspace(s.n_rows, H, Q));
  if (!causal) sub = std::max(sub, subspec_dense_linear_workspace(s.n_rows, 2 * F, H));
  sub = std::max(sub, subspec_dense_linear_workspace(s.n_rows, H, F));
  if (causal) sub = std::max(sub, causal_attention_workspace(s.n_q_heads, s.n_kv_heads, s.n_rows, s.prefix_len));
  else sub = std::max(sub, subspec_tree_attention_workspace(1, s.n_q_heads, s.n_kv_heads, s.n_rows, s.prefix_len, s.n_tree_slots));
  p.sub_bytes = align_up(sub, 256);
  p.sub = take(p.sub_bytes);
  p.total = off;
  return p;
}

static int check_dims(const subspec_decoder_layer_dims* s, int max_rows) {
  if (!s) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: null dims");
  if (s->dtype != SUBSPEC_BF16 && s->dtype != SUBSPEC_F16)
    SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: dtype %d not supported (bf16 / fp16 only)", s->dtype);
  if (s->n_rows < 1 || s->n_rows > max_rows)
    SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "decoder_layer: n_rows=%lld outside 1..%d", (long long)s->n_rows, max_rows);
  if (s->head_dim != 128) SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "decoder_layer: head_dim=%lld (built for 128)", (long long)s->head_dim);
  if (s->hidden <= 0 || s->hidden % 64 != 0 || s->hidden > kNormMaxHidden)
    SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "decoder_layer: hidden=%lld must be a multiple of 64 and at most %d", (long long)s->hidden,
                 kNormMaxHidden);
  if (s->intermediate <= 0 || s->intermediate % 64 != 0)
    SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: intermediate=%lld must be a multiple of 64", (long long)s->intermediate);
  if (s->n_q_heads <= 0 || s->n_kv_heads <= 0 || s->n_q_heads % s->n_kv_heads != 0)
    SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: %lld query heads over %lld kv heads", (long long)s->n_q_heads, (long long)s->n_kv_heads);
  if (s->n_tree_slots < 1 || s->n_tree_slots > SUBSPEC_MAX_TREE_NODES || s->prefix_len < 0 || s->prefix_len + s->n_tree_slots > s->kv_seq_stride)
    SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: prefix_len=%lld, n_tree_slots=%lld do not fit a cache of %lld rows",
                 (long long)s->prefix_len, (long long)s->n_tree_slots, (long long)s->kv_seq_stride);
  if (!(s->rope_theta > 1.f) || !(s->rms_eps > 0.f)) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: rope_theta / rms_eps out of range");
  if (s->page_indices) {
    if (s->page_len <= 0 || (s->page_len & (s->page_len - 1)) != 0 || s->page_len > 4096)
      SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "decoder_layer: page_len=%lld must be a power of two up to 4096", (long long)s->page_len);
    if (s->n_pages <= 0 || s->max_pages < s->n_pages || s->max_pages > 0x7fffffff)
      SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: n_pages=%lld max_pages=%lld", (long long)s->n_pages, (long long)s->max_pages);
    if (s->kv_seq_stride != s->n_pages * s->page_len)
      SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: kv_seq_stride=%lld must equal n_pages * page_len = %lld for a paged cache",
                   (long long)s->kv_seq_stride, (long long)(s->n_pages * s->page_len));
  }
  return SUBSPEC_OK;
}

// The four projections of a layer in either storage: int4 codes + (scale, zero) words, or a dense
// row-major 16-bit matrix (then the second pointer is unused).
struct Projection { const void* w; const void* sz; };
struct LayerWeights {
  const void *input_norm, *post_norm, *qkv_bias;
  Projection qkv, o, gate_up, down;
  bool dense;
};
static LayerWeights layer_weights(const subspec_decoder_layer_weights& s) {
  return {s.input_norm, s.post_norm, s.qkv_bias, {s.qkv_wq, s.qkv_sz}, {s.o_wq, s.o_sz}, {s.gate_up_wq, s.gate_up_sz},
          {s.down_wq, s.down_sz}, false};
}
static LayerWeights layer_weights(const subspec_dense_layer_weights& s) {
  return {s.input_norm, s.post_norm, s.qkv_bias, {s.qkv_w, nullptr}, {s.o_w, nullptr}, {s.gate_up_w, nullptr}, {s.down_w, nullptr}, true};
}
// int4 layers of up to 32 rows: norms and rotary are prologues and output stages of the projections
static bool int4_norm_prologue(const subspec_decoder_layer_dims& s, bool dense) {
  return !dense && s.n_rows <= 32 &&
         subspec_int4_linear_workspace(s.n_rows, (s.n_q_heads + 2 * s.n_kv_heads) * s.head_dim, s.hidden) == 256;
}
static int project(const LayerWeights& w, const Projection& p, const void* x, const void* bias, const void* residual, void* y,
                   int dtype, int64_t M, int64_t N, int64_t K, void* sub, size_t sub_bytes, hipStream_t st,
                   int* pending_splits = nullptr) {
  if (pending_splits) *pending_splits = 1;
  if (w.dense) return dense_linear_ex(x, p.w, bias, residual, y, dtype, M, N, K, sub, sub_bytes, st, pending_splits);
  return int4_linear_ex(x, (const uint32_t*)p.w, (const uint32_t*)p.sz, bias, residual, y, dtype, M, N, K, 64, sub, sub_bytes, st, pending_splits);
}

// What a layer of a stack takes over from the one before it and leaves to the next: the down projection's residual sum, the
// reduction of its fp32 partials and the NEXT RMSNorm are one launch (add_rmsnorm_kernel) instead of two, so a layer of a stack
// ends with its successor's normalized input.  64 dense rows: 4.7 + 4.8 -> 4.9 us a layer, 2048 rows 20.2 + 7.8 -> 11.4.  The
// same sums in the same order, the same bits.
struct StackLink {
  bool h_ready = false;               // the workspace's h holds this layer's normalized input already
  const uint16_t* next_norm = nullptr;   // gain of the next RMSNorm, or null: x alone is wanted
  uint16_t* h_next = nullptr;         // where its output goes; null: the workspace's h
};
template <int DT>
static int run_layer(const subspec_decoder_layer_dims& s, const LayerWeights& w, uint16_t* x,
                     const int32_t* positions, const int32_t* cache_rows, const uint64_t* anc_bits, uint16_t* k_cache,
                     uint16_t* v_cache, char* ws, hipStream_t st, bool causal = false, StackLink link = {}) {
  const LayerPlan p = layer_plan(s, causal);
  const int M = (int)s.n_rows, H = (int)s.hidden, Hq = (int)s.n_q_heads, Hkv = (int)s.n_kv_heads, D = (int)s.head_dim,
            F = (int)s.intermediate;
  const int64_t Q = (int64_t)Hq * D, KV = (int64_t)Hkv * D;
  uint16_t *h = (uint16_t*)(ws + p.h), *qkv = (uint16_t*)(ws + p.qkv), *q = (uint16_t*)(ws + p.q), *a = (uint16_t*)(ws + p.a),
           *o = (uint16_t*)(ws + p.o), *gu = (uint16_t*)(ws + p.gu), *act = (uint16_t*)(ws + p.act);
  void* sub = ws + p.sub;
  const KvPages pages{s.page_indices, s.n_pages, s.max_pages, s.page_len};
  const KvPages* pg = s.page_indices ? &pages : nullptr;
  const KvRowMap kv = make_kv_row_map(k_cache, v_cache, s.kv_seq_stride, Hkv, pg);
  int rc;
  // int4 stack, a level of at most 32 rows: five launches per layer (six with a split-K down projection, seven when
  // the keys are split) -- both norms are prologues of the projections that consume them, rotary + cache write is the
  // output stage of q|k|v, the attention block's residual add the output stage of o_proj
  const bool fused = int4_norm_prologue(s, w.dense);
  if (fused) {
    if ((rc = int4_qkv_rope_ex(x, (const uint32_t*)w.qkv.w, (const uint32_t*)w.qkv.sz, w.qkv_bias, DT, M, H, w.input_norm, s.rms_eps,
                               positions, cache_rows, q, kv, Hq, s.rope_theta, s.rope_inv_freq, st)))
      return rc;
  } else {
    if (!link.h_ready)
      launch_norm<DT>(x, nullptr, w.input_norm, h, M, H, s.rms_eps, nullptr, 0, st);
    // projections whose K is split leave the sum of their partials to the kernel that reads them next
    int pending = 0;
    if ((rc = project(w, w.qkv, h, w.qkv_bias, nullptr, qkv, DT, M, Q + 2 * KV, H, sub, p.sub_bytes, st, &pending))) return rc;
    // few rows: a workgroup per eight heads; from 512 rows a workgroup per row fills the chip and walks all heads
    const int head_groups = (Hq + 2 * Hkv + kRopeHeads - 1) / kRopeHeads;
    hipLaunchKernelGGL((rope_write_kernel<DT>), dim3(M, M >= 512 ? 1 : head_groups), dim3(32 * kRopeHeads), 0, st, qkv, positions,
                       cache_rows, q, kv, M, Hq, Hkv, log2f(s.rope_theta), s.rope_inv_freq, (const float*)sub,
                       pending > 1 ? pending : 0, (const uint16_t*)w.qkv_bias);
  }
  if (causal) {
    const int64_t rows = s.prefix_len + M;
    const uint16_t *kk = k_cache, *vv = v_cache;
    if (pg) {
      kk = (const uint16_t*)(ws + p.kv);
      vv = kk + KV * rows;
      const int64_t pieces = rows * KV / 8;
      hipLaunchKernelGGL(gather_pages_kernel, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, st, kv, rows, (dec_u4*)kk, (dec_u4*)vv);
    }
    if ((rc = causal_attention(q, kk, vv, a, DT, Hq, Hkv, M, pg ? rows : s.kv_seq_stride, s.prefix_len, 1.f / sqrtf((float)D), sub, st)))
      return rc;
  } else if ((rc = tree_attention_ex(q, k_cache, v_cache, a, DT, Hq, Hkv, M, s.n_tree_slots, s.kv_seq_stride, s.prefix_len,
                              s.prefix_len_dev, pg, anc_bits, 1.f / sqrtf((float)D), sub, p.sub_bytes, st)))
    return rc;
  if (fused) {
    // x = round(round(o_proj(a)) + x), then RMSNorm inside the gate|up projection
    if ((rc = project(w, w.o, a, nullptr, x, x, DT, M, H, Q, sub, p.sub_bytes, st))) return rc;
    if ((rc = int4_gate_up_silu_ex(x, (const uint32_t*)w.gate_up.w, (const uint32_t*)w.gate_up.sz, nullptr, act, DT, M,
                                   2 * (int64_t)F, H, w.post_norm, s.rms_eps, st)))
      return rc;
  } else {
  int pending = 0;
  if ((rc = project(w, w.o, a, nullptr, nullptr, o, DT, M, H, Q, sub, p.sub_bytes, st, &pending))) return rc;
  launch_norm<DT>(x, o, w.post_norm, h, M, H, s.rms_eps, (const float*)sub, pending > 1 ? pending : 0, st);
  if (!w.dense) {
    // the activation sits in the output stage of the gate|up projection
    if ((rc = int4_gate_up_silu_ex(h, (const uint32_t*)w.gate_up.w, (const uint32_t*)w.gate_up.sz, nullptr, act, DT, M,
                                   2 * (int64_t)F, H, nullptr, 0.f, st)))
      return rc;
  } else if (M > 32 || 4 * (int64_t)F * H < ((int64_t)1 << 31)) {   // (up to 32 rows the pair kernel addresses the matrix through one 2 GiB descriptor)
    if ((rc = dense_gate_up_silu_ex(h, w.gate_up.w, nullptr, act, DT, M, 2 * (int64_t)F, H, st))) return rc;
  } else {
    if ((rc = project(w, w.gate_up, h, nullptr, nullptr, gu, DT, M, 2 * (int64_t)F, H, sub, p.sub_bytes, st))) return rc;
    const int64_t act_pieces = (int64_t)M * F / 8;
    hipLaunchKernelGGL((silu_mul_kernel<DT>), dim3((unsigned)((act_pieces + 255) / 256)), dim3(256), 0, st, gu, act, F, act_pieces);
  }
  }
  // down projection with the residual add in its output stage: x = round(round(down(act)) + x)
  int down_splits = 0;
  if ((rc = project(w, w.down, act, nullptr, x, x, DT, M, H, F, sub, p.sub_bytes, st, link.next_norm ? &down_splits : nullptr))) return rc;
  if (link.next_norm) {
    uint16_t* hn = link.h_next ? link.h_next : h;
    launch_norm<DT>(x, nullptr, link.next_norm, hn, M, H, s.rms_eps, (const float*)sub, down_splits > 1 ? down_splits : 0, st);
  }
  SUBSPEC_CHECK_HIP(hipGetLastError());
  return SUBSPEC_OK;
}

// The layers of a stack one after the other; h_out (with final_norm): RMSNorm of the last layer's output
template <int DT, typename Weights>
static int run_stack(const subspec_decoder_layer_dims& s, const Weights* layers, int64_t n_layers, uint16_t* x,
                     const int32_t* positions, const int32_t* cache_rows, const uint64_t* anc_bits, void* const* k_caches,
                     void* const* v_caches, const void* final_norm, void* h_out, char* ws, hipStream_t st, bool causal) {
  StackLink link;
  for (int64_t i = 0; i < n_layers; ++i) {
    const LayerWeights w = layer_weights(layers[i]);
    const bool last = i + 1 == n_layers;
    // (an int4 layer of up to 32 rows has its norm inside the q|k|v projection: it only takes a final norm behind the stack)
    const bool own_norm = int4_norm_prologue(s, w.dense);
    link.next_norm = last ? (const uint16_t*)final_norm : own_norm ? nullptr : (const uint16_t*)layer_weights(layers[i + 1]).input_norm;
    link.h_next = last ? (uint16_t*)h_out : nullptr;
    const int rc = run_layer<DT>(s, w, x, positions, cache_rows, anc_bits, (uint16_t*)k_caches[i],
                                 v_caches ? (uint16_t*)v_caches[i] : nullptr, ws, st, causal, link);
    if (rc != SUBSPEC_OK) return rc;
    link.h_ready = link.next_norm != nullptr;
  }
  return SUBSPEC_OK;
}

}  // namespace subspec

using namespace subspec;

extern "C" int subspec_rms_norm(const void* x, const void* weight, void* y, int dtype, int64_t rows, int64_t hidden,
                                float eps, void* stream) {
  if (dtype != SUBSPEC_BF16 && dtype != SUBSPEC_F16) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "rms_norm: dtype %d not supported (bf16 / fp16)", dtype);
  if (!x || !weight || !y) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "rms_norm: null pointer argument");
  if (rows <= 0 || rows > 0x7fffffff) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "rms_norm: rows=%lld", (long long)rows);
  if (hidden <= 0 || hidden % 8 != 0 || hidden > kNormMaxHidden)
    SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "rms_norm: hidden=%lld must be a multiple of 8 and at most %d", (long long)hidden,
                 kNormMaxHidden);
  if (!(eps > 0.f)) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "rms_norm: eps out of range");
  if ((uintptr_t)x % 16 || (uintptr_t)weight % 16 || (uintptr_t)y % 16) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "rms_norm: pointers must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  // the kernel only writes x when it also adds: here it reads it
  if (dtype == SUBSPEC_BF16) launch_norm<SUBSPEC_BF16>((uint16_t*)x, nullptr, weight, (uint16_t*)y, rows, (int)hidden, eps, nullptr, 0, st);
  else launch_norm<SUBSPEC_F16>((uint16_t*)x, nullptr, weight, (uint16_t*)y, rows, (int)hidden, eps, nullptr, 0, st);
  SUBSPEC_CHECK_HIP(hipGetLastError());
  return SUBSPEC_OK;
}

extern "C" size_t subspec_int4_decoder_layer_workspace(const subspec_decoder_layer_dims* dims) {
  if (!dims || check_dims(dims, kDenseLayerMaxRows) != SUBSPEC_OK) return 0;
  return layer_plan(*dims).total;
}

// what holds for a whole call, and (check_layer) for each of its layers
static int check_layer_call(const subspec_decoder_layer_dims* dims, bool dense, void* x, const int32_t* positions,
                            const int32_t* cache_rows, const uint64_t* anc_bits, void* workspace, size_t workspace_bytes) {
  const int rc = check_dims(dims, dense ? kDenseLayerMaxRows : kInt4LayerMaxRows);
  if (rc != SUBSPEC_OK) return rc;
  // the wide dense kernels take weight rows in tiles of 32
  if (dims->n_rows > 64 && ((dims->n_q_heads + 2 * dims->n_kv_heads) * dims->head_dim % 32 != 0 || dims->hidden % 32 != 0))
    SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "decoder_layer: more than 64 rows need projection widths that are multiples of 32");
  if (!x || !positions || !cache_rows || !anc_bits) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: null pointer argument");
  if ((uintptr_t)x % 16) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: x, norm weights and caches must be 16-byte aligned");
  const size_t need = layer_plan(*dims).total;
  if (!workspace || workspace_bytes < need)
    SUBSPEC_FAIL(SUBSPEC_ERR_WORKSPACE, "decoder_layer: workspace of %zu bytes is smaller than the %zu required", workspace_bytes, need);
  if ((uintptr_t)workspace % 256) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: workspace must be 256-byte aligned");
  return SUBSPEC_OK;
}
static int check_layer(const char* what, const subspec_decoder_layer_dims* dims, const LayerWeights& w, void* k_cache, void* v_cache) {
  if (!k_cache || (!v_cache && !dims->page_indices)) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "%s: null pointer argument", what);
  if (!w.input_norm || !w.post_norm || !w.qkv.w || !w.o.w || !w.gate_up.w || !w.down.w ||
      (!w.dense && (!w.qkv.sz || !w.o.sz || !w.gate_up.sz || !w.down.sz)))
    SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "%s: null weight pointer", what);
  if ((uintptr_t)w.input_norm % 16 || (uintptr_t)w.post_norm % 16 || (uintptr_t)k_cache % 16 || (uintptr_t)v_cache % 16)
    SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "%s: x, norm weights and caches must be 16-byte aligned", what);
  // what the projections would refuse in the middle of a stack
  for (const Projection& p : {w.qkv, w.o, w.gate_up, w.down})
    if ((uintptr_t)p.w % 16 || (!w.dense && (uintptr_t)p.sz % 16))
      SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "%s: projection weights must be 16-byte aligned", what);
  return SUBSPEC_OK;
}

static int decoder_layer_entry(const subspec_decoder_layer_dims* dims, const LayerWeights& w, void* x, const int32_t* positions,
                               const int32_t* cache_rows, const uint64_t* anc_bits, void* k_cache, void* v_cache,
                               void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_layer_call(dims, w.dense, x, positions, cache_rows, anc_bits, workspace, workspace_bytes);
  if (rc == SUBSPEC_OK) rc = check_layer("decoder_layer", dims, w, k_cache, v_cache);
  if (rc != SUBSPEC_OK) return rc;
  if (dims->dtype == SUBSPEC_BF16)
    return run_layer<SUBSPEC_BF16>(*dims, w, (uint16_t*)x, positions, cache_rows, anc_bits, (uint16_t*)k_cache, (uint16_t*)v_cache,
                                   (char*)workspace, (hipStream_t)stream);
  return run_layer<SUBSPEC_F16>(*dims, w, (uint16_t*)x, positions, cache_rows, anc_bits, (uint16_t*)k_cache, (uint16_t*)v_cache,
                                (char*)workspace, (hipStream_t)stream);
}

extern "C" int subspec_int4_decoder_layer(const subspec_decoder_layer_dims* dims, const subspec_decoder_layer_weights* weights,
                                          void* x, const int32_t* positions, const int32_t* cache_rows,
                                          const uint64_t* anc_bits, void* k_cache, void* v_cache, void* workspace,
                                          size_t workspace_bytes, void* stream) {
  if (!weights) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: null weights");
  return decoder_layer_entry(dims, layer_weights(*weights), x, positions, cache_rows, anc_bits, k_cache, v_cache, workspace, workspace_bytes, stream);
}

extern "C" int subspec_dense_decoder_layer(const subspec_decoder_layer_dims* dims, const subspec_dense_layer_weights* weights,
                                           void* x, const int32_t* positions, const int32_t* cache_rows,
                                           const uint64_t* anc_bits, void* k_cache, void* v_cache, void* workspace,
                                           size_t workspace_bytes, void* stream) {
  if (!weights) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_layer: null weights");
  return decoder_layer_entry(dims, layer_weights(*weights), x, positions, cache_rows, anc_bits, k_cache, v_cache, workspace,
                             workspace_bytes, stream);
}

static int check_stack_args(const void* weights, int64_t n_layers, void* const* k_caches, const void* final_norm, const void* h_out) {
  if (!weights || !k_caches || n_layers < 1) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_stack: null pointer argument or no layers");
  if (!final_norm != !h_out || (uintptr_t)final_norm % 16 || (uintptr_t)h_out % 16)
    SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "decoder_stack: final_norm and h_out go together and are 16-byte aligned");
  return SUBSPEC_OK;
}

template <typename Weights>
static int decoder_stack_entry(const subspec_decoder_layer_dims* dims, const Weights* weights, int64_t n_layers, void* x,
                               const int32_t* positions, const int32_t* cache_rows, const uint64_t* anc_bits,
                               void* const* k_caches, void* const* v_caches, const void* final_norm, void* h_out,
                               void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_stack_args(weights, n_layers, k_caches, final_norm, h_out);
  if (rc == SUBSPEC_OK)
    rc = check_layer_call(dims, layer_weights(weights[0]).dense, x, positions, cache_rows, anc_bits, workspace, workspace_bytes);
  if (rc != SUBSPEC_OK) return rc;
  for (int64_t i = 0; i < n_layers; ++i)      // every layer is checked before the first one runs
    if ((rc = check_layer("decoder_layer", dims, layer_weights(weights[i]), k_caches[i], v_caches ? v_caches[i] : nullptr))) return rc;
  if (dims->dtype == SUBSPEC_BF16)
    return run_stack<SUBSPEC_BF16>(*dims, weights, n_layers, (uint16_t*)x, positions, cache_rows, anc_bits, k_caches, v_caches,
                                   final_norm, h_out, (char*)workspace, (hipStream_t)stream, false);
  return run_stack<SUBSPEC_F16>(*dims, weights, n_layers, (uint16_t*)x, positions, cache_rows, anc_bits, k_caches, v_caches,
                                final_norm, h_out, (char*)workspace, (hipStream_t)stream, false);
}

extern "C" int subspec_int4_decoder_stack(const subspec_decoder_layer_dims* dims, const subspec_decoder_layer_weights* weights,
                                          int64_t n_layers, void* x, const int32_t* positions, const int32_t* cache_rows,
                                          const uint64_t* anc_bits, void* const* k_caches, void* const* v_caches,
                                          const void* final_norm, void* h_out, void* workspace, size_t workspace_bytes,
                                          void* stream) {
  return decoder_stack_entry(dims, weights, n_layers, x, positions, cache_rows, anc_bits, k_caches, v_caches, final_norm, h_out,
                             workspace, workspace_bytes, stream);
}

extern "C" int subspec_dense_decoder_stack(const subspec_decoder_layer_dims* dims, const subspec_dense_layer_weights* weights,
                                           int64_t n_layers, void* x, const int32_t* positions, const int32_t* cache_rows,
                                           const uint64_t* anc_bits, void* const* k_caches, void* const* v_caches,
                                           const void* final_norm, void* h_out, void* workspace, size_t workspace_bytes,
                                           void* stream) {
  return decoder_stack_entry(dims, weights, n_layers, x, positions, cache_rows, anc_bits, k_caches, v_caches, final_norm, h_out,
                             workspace, workspace_bytes, stream);
}

// A prefill takes dense layers whose projections the kernels above cover at its number of rows
static int check_prefill(const subspec_decoder_layer_dims* s) {
  if (!s) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "prefill_layer: null dims");
  subspec_decoder_layer_dims d = *s;
  d.n_tree_slots = 1;                                 // (no tree: the rows of the call bound the cache below)
  const int rc = check_dims(&d, kPrefillMaxRows);
  if (rc != SUBSPEC_OK) return rc;
  if (s->prefix_len + s->n_rows > s->kv_seq_stride)
    SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "prefill_layer: prefix_len=%lld + n_rows=%lld exceed a cache of %lld rows", (long long)s->prefix_len,
                 (long long)s->n_rows, (long long)s->kv_seq_stride);
  if (s->prefix_len_dev) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "prefill_layer: no device-side prefix length");
  const int64_t M = s->n_rows, H = s->hidden, F = s->intermediate, Q = s->n_q_heads * s->head_dim, KV = s->n_kv_heads * s->head_dim;
  if (std::max(std::max(H, F), Q) > 65536)
    SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "prefill_layer: a projection longer than 65536");
  // up to 64 rows: kernels with a 2 GiB descriptor range
  if (M <= 64 && std::max(2 * F * H, (Q + 2 * KV) * H) >= ((int64_t)1 << 30))
    SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "prefill_layer: up to 64 rows take matrices below 2 GiB");
  if (M > 64 && !(tile_applies(M, Q + 2 * KV, H, false, nullptr, nullptr) && tile_applies(M, H, Q, false, nullptr, nullptr) &&
                  tile_applies(M, 2 * F, H, true, nullptr, nullptr) && tile_applies(M, H, F, false, nullptr, nullptr)))
    SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "prefill_layer: projection sizes outside the tiled kernel's range");
  if ((Q + 2 * KV) / s->head_dim > 65535 || s->n_q_heads * ((M + 63) / 64) * 2 > 0x7fffff)
    SUBSPEC_FAIL(SUBSPEC_ERR_LIMIT, "prefill_layer: %lld heads over %lld rows", (long long)s->n_q_heads, (long long)M);
  return SUBSPEC_OK;
}

extern "C" size_t subspec_prefill_layer_workspace(const subspec_decoder_layer_dims* dims) {
  return check_prefill(dims) == SUBSPEC_OK ? layer_plan(*dims, true).total : 0;
}

extern "C" int subspec_prefill_stack(const subspec_decoder_layer_dims* dims, const subspec_dense_layer_weights* weights,
                                     int64_t n_layers, void* x, const int32_t* positions, const int32_t* cache_rows,
                                     void* const* k_caches, void* const* v_caches, const void* final_norm, void* h_out,
                                     void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_prefill(dims);
  if (rc == SUBSPEC_OK) rc = check_stack_args(weights, n_layers, k_caches, final_norm, h_out);
  if (rc != SUBSPEC_OK) return rc;
  if (!x || !positions || !cache_rows) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "prefill_layer: null pointer argument");
  if ((uintptr_t)x % 16) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "prefill_layer: x, norm weights and caches must be 16-byte aligned");
  for (int64_t i = 0; i < n_layers; ++i)
    if ((rc = check_layer("prefill_layer", dims, layer_weights(weights[i]), k_caches[i], v_caches ? v_caches[i] : nullptr))) return rc;
  const size_t need = layer_plan(*dims, true).total;
  if (!workspace || workspace_bytes < need)
    SUBSPEC_FAIL(SUBSPEC_ERR_WORKSPACE, "prefill_layer: workspace of %zu bytes is smaller than the %zu required", workspace_bytes, need);
  if ((uintptr_t)workspace % 256) SUBSPEC_FAIL(SUBSPEC_ERR_ARG, "prefill_layer: workspace must be 256-byte aligned");
  if (dims->dtype == SUBSPEC_BF16)
    return run_stack<SUBSPEC_BF16>(*dims, weights, n_layers, (uint16_t*)x, positions, cache_rows, nullptr, k_caches, v_caches,
                                   final_norm, h_out, (char*)workspace, (hipStream_t)stream, true);
  return run_stack<SUBSPEC_F16>(*dims, weights, n_layers, (uint16_t*)x, positions, cache_rows, nullptr, k_caches, v_caches,
                                final_norm, h_out, (char*)workspace, (hipStream_t)stream, true);
}

extern "C" int subspec_prefill_layer(const subspec_decoder_layer_dims* dims, const subspec_dense_layer_weights* weights, void* x,
                                     const int32_t* positions, const int32_t* cache_rows, void* k_cache, void* v_cache,
                                     void* workspace, size_t workspace_bytes, void* stream) {
  return subspec_prefill_stack(dims, weights, 1, x, positions, cache_rows, &k_cache, v_cache ? &v_cache : nullptr, nullptr, nullptr,
                               workspace, workspace_bytes, stream);
}
