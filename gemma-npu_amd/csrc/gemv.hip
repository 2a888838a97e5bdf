// Weight-only int8 GEMV / skinny GEMM for decode and the LM head.
//
// y[m, n] = bf16( (sum_k x[m,k] * w[n,k]) * s[n] ),  x bf16 [M<=16, K], w int8 [N, K] row-major,
// s bf16 or fp32 [N]: the contract of torch._weight_int8pack_mm as the reference calls it
// (gemma_npu.py:155-156, decode linears gemma_npu.py:120-121, Int8Head gemma_npu.py:159-172).
//
// The weight is streamed once from HBM with 16-byte loads; each byte is widened to bf16 (exact:
// |w| <= 128) and multiplied on the bf16 MFMA (v_mfma_f32_16x16x32_bf16, fp32 accumulate), with
// the M <= 16 activation rows as the MFMA's other operand.  A wave covers TPW 16-row n-tiles, so each activation fragment it loads serves
// TPW weight fragments; for shapes with few n-tiles, `split` waves of a workgroup share one
// n-tile's K range (k-blocks of 64 dealt round-robin) and their partial sums are added in LDS in
// fixed wave order, so the result is deterministic.
#include "w8a8_common.h"

namespace w8a8 {

struct GemvParams {
  const uint16_t* x; int64_t ldx;  // bf16 [M, K]
  const int8_t* w; int64_t ldw;    // int8 [N, K]
  const void* s; int s_f32;        // [N] scales, bf16 (0) or fp32 (1)
  uint16_t* y; int64_t ldy;        // bf16 [M, N]
  uint32_t x_bytes, w_bytes;
  int M, N, K, KB;                 // KB = ceil(K / 64)
  int split;                       // waves per group of n-tiles, each taking every split-th k-block
  int units, gpb;                  // one row: units of weight rows, and those of one workgroup
  // Activation epilogue (ACT template argument): 1, GELU pair: the weight is [gate; up] stacked
  // (N = 2I, I a multiple of 16) and y [M, I] = bf16(bf16(gelu_tanh(g)) * u) with g, u the bf16
  // outputs of the gate and up rows; 2, GELU times a multiplier: y = bf16(bf16(gelu_tanh(g)) * mul)
  // with mul bf16 [M, N] (ld = ldm).
  const uint16_t* mul; int64_t ldm;
  int half_tiles;                  // ACT 1: I / 16, the up rows' first tile
  // Row prologue (PRO template argument, M = 1): the activation row is not read from x but made by
  // every workgroup from the previous step's output, as w8a8_rms_residual_norm_bf16 (norm2 set) or
  // w8a8_rms_residual_bf16 (norm2 clear) would make it in a launch of its own:
  //   h = bf16(res + bf16(rms(pro_y) * w1)) [then bf16(h * scalar)],  x = norm2 ? bf16(rms(h) * w2) : h
  // (no res: h = bf16(rms(pro_y) * w1)).  Workgroup 0 stores h when pro_h is set.
  const uint16_t* pro_y; const uint16_t* pro_res; const uint16_t* pro_w1; const uint16_t* pro_scalar;
  const uint16_t* pro_w2; uint16_t* pro_h;
  float pro_eps; int pro_norm2;
  // Attention-merge prologue (PRO == 4, M = 1): the activation row is one token's decode attention
  // output [H * D], merged from the split-key kernel's chunk partials (part_o [KV][nchunk_grid][G][D],
  // part_ml [KV][nchunk_grid][G][2]) as attn_decode_merge_kernel merges them, for at most
  // DEC_MERGE_IN_GEMV_CHUNKS chunks; the live chunks follow from the position in device memory.
  const float* m_po; const float* m_ml; const int* m_pos;
  int m_window, m_nchunk_grid, m_G, m_D, m_chunk; float m_c;
};

// The longest activation row that the one-row kernels hold in LDS (24 KiB).
constexpr int GEMV_ROW_MAX = 12288;
// Heads that the merge prologue makes chunk weights for: H * D <= 4096 at head_dim 128.
constexpr int MERGE_HEADS = 32;

// The merge prologue.  For at most 16 chunks attn_decode_merge_kernel's sums reduce to fixed orders,
// taken here: per head, its chunk weights w_c = exp2(M_c c - M c) and the weighted l over a 16-leaf
// tree (t + 8, t + 4, t + 2, t + 1), made once per workgroup by one thread per head into mw
// [MERGE_HEADS][17] (w_0 .. w_15, then 1 / l); per element, the chunks in order, each term
// fma(w_c, o_c, 0), a +0 after them when fewer than 16 are live (the merge kernel's empty parts).
// Each thread makes elements e, e + 1 of the row (one head, columns d, d + 1); the partials of its
// first pair are fetched before the weights are made.
__device__ __forceinline__ void gemv_attn_merge_row(const GemvParams& p, uint16_t* xs, float* mw) {
  constexpr int NC = DEC_MERGE_IN_GEMV_CHUNKS;
  const int pos = *p.m_pos;
  const int H = p.K / p.m_D;
  auto head_base = [&](int h) { return int64_t(h / p.m_G) * p.m_nchunk_grid * p.m_G + h % p.m_G; };
  // this thread's first pair: its partials now
  int e = 2 * int(threadIdx.x);
  v2f oc[NC];
  auto fetch = [&](int e) {
    const int h = e / p.m_D, d = e % p.m_D;
    const int64_t hb = head_base(h);
#pragma unroll
    for (int c = 0; c < NC; ++c)
      oc[c] = (c < p.m_nchunk_grid && e < p.K)
                  ? *reinterpret_cast<const v2f*>(p.m_po + (hb + int64_t(c) * p.m_G) * p.m_D + d)
                  : v2f{0.0f, 0.0f};
  };
  // The loads cover every chunk the grid has, so none waits for the position; chunks that are not
  // live yet (their partials hold old values) are left out afterwards.
  fetch(e);
  v2f ml[NC];
  const int hw = min(int(threadIdx.x), H - 1);
  if (int(threadIdx.x) < H) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
      ml[c] = c < p.m_nchunk_grid ? *reinterpret_cast<const v2f*>(p.m_ml + (head_base(hw) + int64_t(c) * p.m_G) * 2)
                                  : v2f{0.0f, 0.0f};
  }
  const int klo = p.m_window > 0 ? max(0, pos - p.m_window + 1) : 0;
  const int nchunk = max(0, min((pos - klo) / p.m_chunk + 1, p.m_nchunk_grid));
  if (int(threadIdx.x) < H) {
    const int h = int(threadIdx.x);
    float mc[NC], lc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      mc[c] = c < nchunk ? ml[c][0] : -__builtin_inff();
      lc[c] = c < nchunk ? ml[c][1] : 0.0f;
    }
    float M = -__builtin_inff();
#pragma unroll
    for (int c = 0; c < NC; ++c) M = fmaxf(M, mc[c]);
    const float ms = M == -__builtin_inff() ? 0.0f : M * p.m_c;
    float v[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const float w = c < nchunk ? __builtin_amdgcn_exp2f(__builtin_fmaf(mc[c], p.m_c, -ms)) : 0.0f;
      mw[h * (NC + 1) + c] = w;
      v[c] = c < nchunk ? __builtin_fmaf(w, lc[c], 0.0f) : 0.0f;
    }
#pragma unroll
    for (int s = 8; s > 0; s >>= 1)
#pragma unroll
      for (int t = 0; t < s; ++t) v[t] = v[t] + v[t + s];
    mw[h * (NC + 1) + NC] = v[0] > 0.0f ? 1.0f / v[0] : 0.0f;
  }
  __syncthreads();
  for (; e < p.K; e += 2 * int(blockDim.x)) {
    if (e != 2 * int(threadIdx.x)) fetch(e);
    const float* wh = mw + (e / p.m_D) * (NC + 1);
    float a0 = 0.0f, a1 = 0.0f;
    if (nchunk > 0) {
      a0 = __builtin_fmaf(wh[0], oc[0][0], 0.0f);
      a1 = __builtin_fmaf(wh[0], oc[0][1], 0.0f);
    }
#pragma unroll
    for (int c = 1; c < NC; ++c)
      if (c < nchunk) {
        a0 = a0 + __builtin_fmaf(wh[c], oc[c][0], 0.0f);
        a1 = a1 + __builtin_fmaf(wh[c], oc[c][1], 0.0f);
      }
    if (nchunk < NC) {
      a0 = a0 + 0.0f;
      a1 = a1 + 0.0f;
    }
    const float inv = wh[NC];
    *reinterpret_cast<uint32_t*>(xs + e) = pack_bf16x2(a0 * inv, a1 * inv);
  }
}

// The row prologue, in the arithmetic and order of the row kernel's one-wave rows (row_chain_kernel
// with 64 threads, rowops.hip): lane t holds chunks c < CH of 8 elements at k = 8 * (64 c + t); the
// sums of squares are added chunk by chunk, element by element, then across the wave by
// wave_sum_dpp (chunks past K hold zeros, which change no sum).  It is latency, not throughput, that it costs: every workgroup makes the row again
// while its weights are in flight.  So CH waves share it: each takes the sums over the whole row (a
// multiply and an add per element) but the element-wise work, with its roundings, of chunk `wave`
// only, and the chunks of h meet in LDS.  One wave doing all of it took the gate/up GEMV (K=1536,
// N=12288) 3.9 us more than the plain GEMV's 6.65; see the figures at gemv1_launch.  Its operands
// are fetched first (load), before the kernel issues its weight loads, so the arithmetic waits for
// them alone; the row goes to xs [CH * 512] bf16 (zeros from K on), by way of hs [CH * 512].
template <int CH>
struct RowIn {
  v4u y[CH], own, res, w1, w2;
  uint16_t scalar;

  __device__ __forceinline__ void load(const GemvParams& p, int wave) {
    const int t = threadIdx.x & 63;
    const v4u one = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};  // bf16 1.0 x 8
    const v4u zero = {0u, 0u, 0u, 0u};
    scalar = p.pro_scalar ? *p.pro_scalar : uint16_t(0x3f80);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int k = 8 * (64 * c + t);
      y[c] = k < p.K ? *reinterpret_cast<const v4u*>(p.pro_y + k) : zero;
    }
    const int k = 8 * (64 * wave + t);
    const bool in = k < p.K;
    own = in ? *reinterpret_cast<const v4u*>(p.pro_y + k) : zero;
    res = (in && p.pro_res) ? *reinterpret_cast<const v4u*>(p.pro_res + k) : zero;
    w1 = (in && p.pro_w1) ? *reinterpret_cast<const v4u*>(p.pro_w1 + k) : one;
    w2 = (in && p.pro_norm2 && p.pro_w2) ? *reinterpret_cast<const v4u*>(p.pro_w2 + k) : one;
  }

  // 1 / rms over the row whose chunks are in `c`.
  __device__ __forceinline__ static float inv_rms(const v4u (&c)[CH], const GemvParams& p) {
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      float v[8];
      unpack8(c[i], v);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
    }
    ss = wave_sum_dpp(ss);
    return 1.0f / sqrtf(ss / float(p.K) + p.pro_eps);
  }

  // This wave's chunk of h (wave < CH).
  __device__ __forceinline__ v4u make_h(const GemvParams& p) const {
    const float r = inv_rms(y, p);
    const float scl = bf16_to_f32(scalar);
    float v[8], rv[8], wv[8];
    unpack8(own, v);
    unpack8(res, rv);
    unpack8(w1, wv);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float n = v[i] * r;
      if (p.pro_w1) n = n * wv[i];
      v[i] = p.pro_res ? round_bf16(rv[i] + round_bf16(n)) : round_bf16(n);
      if (p.pro_scalar) v[i] = round_bf16(v[i] * scl);
    }
    return pack8(v);
  }

  // Called by every wave of the workgroup; the row is whole in xs after the caller's barrier.
  __device__ __forceinline__ void make(const GemvParams& p, int wave, uint16_t* xs, uint16_t* hs) {
    const int t = threadIdx.x & 63;
    const int k = 8 * (64 * wave + t);
    v4u h = {0u, 0u, 0u, 0u};
    if (wave < CH) {
      h = make_h(p);
      if (k >= p.K) h = v4u{0u, 0u, 0u, 0u};
      if (p.pro_h && blockIdx.x == 0 && k < p.K) *reinterpret_cast<v4u*>(p.pro_h + k) = h;
      *reinterpret_cast<v4u*>((p.pro_norm2 ? hs : xs) + k) = h;
    }
    if (!p.pro_norm2) return;
    __syncthreads();
    if (wave < CH) {
      v4u hc[CH];
#pragma unroll
      for (int c = 0; c < CH; ++c) hc[c] = *reinterpret_cast<const v4u*>(hs + 8 * (64 * c + t));
      const float r2 = inv_rms(hc, p);
      float v[8], wv[8];
      unpack8(h, v);
      unpack8(w2, wv);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float n = v[i] * r2;
        if (p.pro_w2) n = n * wv[i];
        v[i] = round_bf16(n);
      }
      *reinterpret_cast<v4u*>(xs + k) = k < p.K ? pack8(v) : v4u{0u, 0u, 0u, 0u};
    }
  }
};

// Widen 8 signed bytes (two dwords) to 8 bf16 values, exactly: a sign-extending conversion per byte and
// one packed conversion (nothing to round: |w| <= 128) per pair.
__device__ __forceinline__ v8bf widen8(uint32_t lo, uint32_t hi) {
  v4u r;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t d = i ? hi : lo;
    r[2 * i] = pack_bf16x2(float(int8_t(d & 0xff)), float(int8_t((d >> 8) & 0xff)));
    r[2 * i + 1] = pack_bf16x2(float(int8_t((d >> 16) & 0xff)), float(int8_t(d >> 24)));
  }
  return __builtin_bit_cast(v8bf, r);
}

// k-block of 64 on the MFMA: 16 weight rows' bytes against the activation columns, added to acc.
__device__ __forceinline__ v4f mma_block(v4i w, v4i xa, v4i xb, v4f acc) {
  const v8bf wa = widen8(uint32_t(w[0]), uint32_t(w[1]));
  const v8bf wb = widen8(uint32_t(w[2]), uint32_t(w[3]));
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa, __builtin_bit_cast(v8bf, xa), acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb, __builtin_bit_cast(v8bf, xb), acc, 0, 0, 0);
}

// 16 weight bytes; the packed stream with the streaming (sc0 nt) policy.
template <bool PACKED>
__device__ __forceinline__ v4i load_weight(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, PACKED ? 3 : 0));
}

// The epilogue's operands of one lane: for T tiles `tstep` columns apart, the scales of columns n0 ..
// n0+3, and for ACT 2 row m's multipliers.  load() only asks for them, kept in bounds without a
// branch or a conversion per element (either would wait for the element before the next is asked
// for: 3 us of the gate/up GEMV); scale() and mul() convert.  Columns past N are not stored.
template <int T, int ACT>
struct GemvScales {
  uint32_t s[T][4], m[4];

  __device__ __forceinline__ void load(const GemvParams& p, int row, int n0, int tstep) {
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.s, uint32_t(p.N) * (p.s_f32 ? 4u : 2u));
    if (p.s_f32) {
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          s[t][r] = __builtin_amdgcn_raw_buffer_load_b32(rs, uint32_t(n0 + t * tstep + r) * 4u, 0, 0);
    } else {
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          s[t][r] = __builtin_amdgcn_raw_buffer_load_b16(rs, uint32_t(n0 + t * tstep + r) * 2u, 0, 0);
    }
    if constexpr (ACT == 2) {
      // rows have a 64-bit base each (ldm may be any stride); the last row and column stand for those past
      // them, whose results are not stored
      const uint16_t* const mr = p.mul + int64_t(min(row, p.M - 1)) * p.ldm;
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] = mr[min(n0 + r, p.N - 1)];
    }
  }
  __device__ __forceinline__ float scale(const GemvParams& p, int t, int r) const {
    return __uint_as_float(p.s_f32 ? s[t][r] : s[t][r] << 16);
  }
  __device__ __forceinline__ float mul(int r) const { return __uint_as_float(m[r] << 16); }
};

__device__ __forceinline__ void store4(uint16_t* dst, const float (&o)[4], int n0, int n_end) {
  if (n0 + 3 < n_end && ((reinterpret_cast<uintptr_t>(dst) & 7) == 0)) {
    *reinterpret_cast<v2u*>(dst) = v2u{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n0 + r < n_end) dst[r] = f32_to_bf16(o[r]);
  }
}

// Row m, columns n0 .. n0+3 of tile t: y = bf16(acc * s).
template <int T>
__device__ __forceinline__ void store_plain(const GemvParams& p, const GemvScales<T, 0>& sc, int t, v4f acc, int m,
                                            int n0) {
  float o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = acc[r] * sc.scale(p, t, r);
  store4(p.y + int64_t(m) * p.ldy + n0, o, n0, p.N);
}

// The bf16 GEMV outputs, then the activation with the row kernel's roundings: a, b the gate and up
// sums (ACT 1), or a the gate's alone (ACT 2).
template <int ACT, int T>
__device__ __forceinline__ void store_act(const GemvParams& p, const GemvScales<T, ACT>& sc, v4f a, v4f b, int m, int n0) {
  float o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float g = round_bf16(a[r] * sc.scale(p, 0, r));
    const float u = ACT == 1 ? round_bf16(b[r] * sc.scale(p, T - 1, r)) : sc.mul(r);
    o[r] = round_bf16(gelu_tanh_f32(g)) * u;
  }
  store4(p.y + int64_t(m) * p.ldy + n0, o, n0, ACT == 1 ? p.half_tiles * 16 : p.N);
}

// ---- 2..16 rows, and the LM head's many tiles ---------------------------------------------------
// A wave multiplies TPW n-tiles of 16 weight rows against the M <= 16 activation rows: per k-block
// of 64 it loads the activation fragment once and TPW weight fragments, and issues 2*TPW MFMAs.
// With split > 1 the waves of a group take interleaved k-blocks and their partial sums are added
// in LDS in wave order (deterministic).
//
// PACKED: the weight is in the GEMV fragment layout (pack_gemv_weight_kernel): fragment (t, kb) =
// 1 KiB at (t * KB + kb) * 1024 whose byte 16*l + b is W[16t + l%16][64kb + 16(l/16) + b], the
// bytes lane l feeds the MFMA.  Every weight load is then one contiguous KiB of whole cache
// lines, which the stream reads with the streaming (sc0 nt) policy: measured on MI355X for the
// LM head (K=1536, N=262144), 6.2 TB/s against 5.0 TB/s for the row-major weight, where each load
// takes 64-byte pieces of 16 rows.  Row-major weights keep the default policy (a streamed half
// line would be fetched twice).
template <int TPW, int U, bool PACKED, int NWB, int ACT = 0>
__global__ __launch_bounds__(NWB * 64) void gemv_kernel(GemvParams p) {
  static_assert(ACT != 1 || TPW == 2, "a GELU pair is one gate and one up tile per wave");
  __shared__ v4f red[NWB][TPW][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  // 8 and 16 waves always share one tile group (gemv_launch_few)
  const int split = NWB >= 8 ? NWB : p.split;
  const int group_in_block = wave / split;
  const int ks = wave % split;
  const int groups_per_block = NWB / split;
  const int group = blockIdx.x * groups_per_block + group_in_block;
  // ACT 1: group g multiplies gate tile g and up tile g + half_tiles
  const int tile0 = ACT == 1 ? group : group * TPW;
  const int tstride = ACT == 1 ? p.half_tiles : 1;
  const int ntiles = (p.N + 15) >> 4;
  const bool active = ACT == 1 ? tile0 < p.half_tiles : tile0 < ntiles;

  const __amdgpu_buffer_rsrc_t rw = make_rsrc(p.w, p.w_bytes);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, p.x_bytes);
  const int kc = (lane >> 4) * 16;           // this lane's 16-byte chunk inside each 64-wide k-block
  const int mrow = lane & 15;                // activation row this lane supplies
  // acc[t] of lane l holds row m = l % 16, columns (tile0 + t * tstride)*16 + ncol .. +3
  const int ncol = 4 * (lane >> 4);
  GemvScales<TPW, ACT> sc;
  // few tiles: the epilogue's operands come with the weights, not a round trip after them
  if (split > 1 && ks == 0 && active) sc.load(p, mrow, tile0 * 16 + ncol, tstride * 16);

  // Weight rows past N and activation rows past M start at or past the buffer ends and read 0.
  uint32_t wbase[TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t)
    wbase[t] = PACKED ? uint32_t(tile0 + t * tstride) * uint32_t(p.KB) * 1024u + uint32_t(lane) * 16u
                      : uint32_t((tile0 + t * tstride) * 16 + (lane & 15)) * uint32_t(p.ldw) + uint32_t(kc);
  constexpr uint32_t W_KB = PACKED ? 1024u : 64u;  // weight bytes between k-blocks
  const uint32_t xbase = (uint32_t(mrow) * uint32_t(p.ldx) + uint32_t(kc)) * 2u;

  v4f acc[TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
  if (active) {
    const int stride = split * U;
    for (int kb0 = ks; kb0 < p.KB; kb0 += stride) {
      v4i wv[U][TPW], xa[U], xb[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int kb = kb0 + u * split;
        if (kb < p.KB && kb * 64 + kc < p.K) {
          xa[u] = buf_load16(rx, xbase + uint32_t(kb) * 128u);
          xb[u] = buf_load16(rx, xbase + uint32_t(kb) * 128u + 16u);
#pragma unroll
          for (int t = 0; t < TPW; ++t) wv[u][t] = load_weight<PACKED>(rw, wbase[t] + uint32_t(kb) * W_KB);
        } else {
          xa[u] = v4i{0, 0, 0, 0};
          xb[u] = v4i{0, 0, 0, 0};
#pragma unroll
          for (int t = 0; t < TPW; ++t) wv[u][t] = v4i{0, 0, 0, 0};
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < TPW; ++t) acc[t] = mma_block(wv[u][t], xa[u], xb[u], acc[t]);
    }
  }

  const int m = lane & 15;
  if (split > 1) {
    // only the lanes of the M rows hold sums that are used
    if (m < p.M) {
#pragma unroll
      for (int t = 0; t < TPW; ++t) red[wave][t][lane] = acc[t];
    }
    __syncthreads();
    if (ks != 0) return;
    if (m < p.M) {
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        acc[t] = red[wave][t][lane];
        if constexpr (NWB >= 8) {
          v4f part[NWB];
#pragma unroll
          for (int q = 1; q < NWB; ++q) part[q] = red[q][t][lane];
#pragma unroll
          for (int q = 1; q < NWB; ++q) acc[t] += part[q];
        } else {
          for (int q = 1; q < split; ++q) acc[t] += red[wave + q][t][lane];
        }
      }
    }
  }
  if (!active || m >= p.M) return;
  if (split == 1) sc.load(p, mrow, tile0 * 16 + ncol, tstride * 16);
  if constexpr (ACT != 0) {
    store_act<ACT>(p, sc, acc[0], acc[TPW - 1], m, tile0 * 16 + ncol);
  } else {
#pragma unroll
    for (int t = 0; t < TPW; ++t) store_plain(p, sc, t, acc[t], m, (tile0 + t) * 16 + ncol);
  }
}

// ---- one row -------------------------------------------------------------------------------------
// The decode step's linears (M = 1, 3-38 MB of weights).  They are bound by how many memory round
// trips stand behind one another and by the busiest CU, not by HBM: a weight that lies in the cache
// costs nearly what a cold one does.  So
//  * everything the kernel will need is asked for at its start: the epilogue's scales and multiplier,
//    the row's operands, then up to U fragments of weights per wave, all in flight while the row is
//    made in LDS (PRO 3: the residual stream's norm, a row of 3 * 512; 4: the attention merge; 5:
//    copied from x);
//  * the tiles are dealt in units, `gpb` groups of `split` waves to a workgroup (gemv1_plan), and a
//    wave multiplies no fragment past K: widening a KiB of bytes takes a SIMD about 100 clocks.
// For the same reason a weight with few tiles (N = 1536: 96 of 16 rows on 256 CUs) is dealt in halves
// (wide down 12288 x 1536: 9.6 us in whole tiles, 6.8 in halves): with HALF a unit is 8 weight rows, and a fragment load takes them from two
// k-blocks at once: lane l holds row l % 8 of the unit, of k-block 2 q + (l % 16 >= 8) for pair q,
// bytes 16 (l / 16).  The MFMA's column 0 gets the activations of the even k-block and column 1
// those of the odd one, so the sums of rows 0..7 of column 0 and rows 8..15 of column 1 are the
// unit's two partial sums.  Without HALF, a GELU pair (ACT 1) is 8 gate rows and the same 8 up rows in
// one tile, from the two fragments that hold them.
// The order of every sum is that of gemv_kernel for the same (N, K), so a row gives the same bits alone
// and among 2..16, and so do the plain GEMV, the activations and the prologues: few_tile_split partial
// sums, number v over the k-blocks v, v + parts, .., added in order.  A wave makes the R numbered ks and
// ks + split in turn (parts = R * split), or with HALF, R = 1, the two numbered 2 ks and 2 ks + 1.
template <int U, bool PACKED, int ACT, int PRO, bool HALF, int R>
__global__ __launch_bounds__(PRO == 4 ? 1024 : 768) void gemv1_kernel(GemvParams p) {
  constexpr bool NORM = PRO <= 3;                  // PRO chunks of 512 (K <= 1536)
  constexpr int XS = PRO == 5 ? GEMV_ROW_MAX : PRO == 4 ? 4096 : PRO * 512;
  constexpr int TPW = ACT == 1 && HALF ? 2 : 1;    // HALF pairs: the gate rows' and the up rows' fragments
  constexpr bool SPLIT_ROWS = HALF || ACT == 1;    // a unit is 8 output columns
  constexpr bool PAIR = ACT == 1 && !HALF;         // gate and up rows in one fragment
  static_assert(!HALF || R == 1, "HALF's two sums are two columns of one accumulator");
  static_assert(R == 1 || U % 2 == 0 || U <= 3, "a wave's steps alternate; odd U only where one round is all");
  __shared__ v4f red[32][TPW][4];                  // per partial sum of the workgroup: rows 4j .. 4j+3 of its tile
  __shared__ __attribute__((aligned(16))) uint16_t xs[XS + 16];               // the row, and a piece of zeros
  __shared__ __attribute__((aligned(16))) uint16_t hs[NORM ? PRO * 512 : 8];  // NORM: the first norm's row
  __shared__ float mw[PRO == 4 ? MERGE_HEADS * (DEC_MERGE_IN_GEMV_CHUNKS + 1) : 1];  // PRO 4: chunk weights
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int split = p.split;
  const int gib = wave / split, ks = wave % split;
  const int unit = int(blockIdx.x) * p.gpb + gib;
  const int parts = (HALF ? 2 : R) * split;  // partial sums of a unit
  const bool active = gib < p.gpb && unit < p.units;
  const int i = lane & 15, j = lane >> 4;  // fragment row and 16-byte chunk

  const __amdgpu_buffer_rsrc_t rw = make_rsrc(p.w, p.w_bytes);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, p.x_bytes);
  constexpr uint32_t PAST = 0x80000000u;  // an offset past every buffer here: reads zero

  RowIn<NORM ? PRO : 1> row;
  if constexpr (NORM) {
    if (wave < PRO) row.load(p, wave);
  }
  // The epilogue runs on the group's first wave, lanes 16 j: columns n0 .. n0+3.
  const int n0 = SPLIT_ROWS ? unit * 8 + 4 * j : unit * 16 + 4 * j;
  GemvScales<ACT == 1 ? 2 : 1, ACT> sc;
  if (ks == 0 && active) sc.load(p, i, n0, p.half_tiles * 16);

  // Byte offset of this lane's piece of fragment t at k-block 0, and k-blocks between fragments.
  const int sub = SPLIT_ROWS ? 8 * (unit & 1) + (i & 7) : i;  // row inside its 16-row tile
  uint32_t wbase[TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    int tile = SPLIT_ROWS ? unit >> 1 : unit;
    if (PAIR && i >= 8) tile += p.half_tiles;
    if (TPW == 2 && t == 1) tile += p.half_tiles;
    wbase[t] = PACKED ? uint32_t(tile) * uint32_t(p.KB) * 1024u + uint32_t(j * 16 + sub) * 16u
                      : uint32_t(tile * 16 + sub) * uint32_t(p.ldw) + uint32_t(j * 16);
  }
  constexpr uint32_t W_KB = PACKED ? 1024u : 64u;  // weight bytes between k-blocks
  const int nstep = HALF ? (p.KB + 1) >> 1 : p.KB;   // steps over K: pairs of k-blocks with HALF
  const int hi = HALF ? i >> 3 : 0;                  // this lane's weight k-block within its pair
  auto load_w = [&](int st, v4i (&w)[TPW]) {
    const int kb = HALF ? 2 * st + hi : st;
    const bool ok = active && kb < p.KB && kb * 64 + j * 16 < p.K;
#pragma unroll
    for (int t = 0; t < TPW; ++t) w[t] = load_weight<PACKED>(rw, ok ? wbase[t] + uint32_t(kb) * W_KB : PAST);
  };

  const int row_end = (HALF ? (p.KB + 1) & ~1 : p.KB) * 64;  // the row's elements that are read
  if (threadIdx.x < 2) *reinterpret_cast<v4i*>(xs + XS + 8 * threadIdx.x) = v4i{0, 0, 0, 0};
  v4i wv[U][TPW];
  if constexpr (PRO == 5) {
    // The row's pieces of 8 are asked for before the weights, two per thread: a row of up to 8192 elements
    // at eight waves, 4096 at four.  What a longer one has past that is copied first, in a loop that waits for
    // each piece before any weight is asked for.
    const int k0 = int(threadIdx.x) * 8, nt8 = int(blockDim.x) * 8, k1 = k0 + nt8;
    for (int k = k1 + nt8; k < row_end; k += nt8)
      *reinterpret_cast<v4i*>(xs + k) = buf_load16(rx, k < p.K ? uint32_t(k) * 2u : PAST);
    const v4i x0 = buf_load16(rx, k0 < p.K ? uint32_t(k0) * 2u : PAST);
    const v4i x1 = buf_load16(rx, k1 < p.K ? uint32_t(k1) * 2u : PAST);
#pragma unroll
    for (int u = 0; u < U; ++u) load_w(ks + u * split, wv[u]);
    if (k0 < row_end) *reinterpret_cast<v4i*>(xs + k0) = x0;
    if (k1 < row_end) *reinterpret_cast<v4i*>(xs + k1) = x1;
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u) load_w(ks + u * split, wv[u]);
    if constexpr (PRO == 4)
      gemv_attn_merge_row(p, xs, mw);
    else
      row.make(p, wave, xs, hs);
  }
  __syncthreads();

  // This lane's piece of the row for step st: activation column 0 takes it (with HALF column 0 the even
  // k-blocks and column 1 the odd ones), the others read a piece of zeros, so that the reads take no
  // branch and stand ahead of the MFMAs.  The row is zero from K up to the next k-block (with HALF, the
  // next pair).
  const bool column = i < (HALF ? 2 : 1);
  const uint16_t* const xbase = column ? xs + (HALF ? i * 64 : 0) + j * 16 : xs + XS;
  const int xstep = column ? (HALF ? 128 : 64) : 0;
  v4f acc[R][TPW];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int t = 0; t < TPW; ++t) acc[r][t] = v4f{0.f, 0.f, 0.f, 0.f};
  for (int st0 = ks; st0 < nstep; st0 += split * U) {
    if (st0 != ks) {
#pragma unroll
      for (int u = 0; u < U; ++u) load_w(st0 + u * split, wv[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int st = st0 + u * split;
      if (st >= nstep) break;
      const uint16_t* xv = xbase + st * xstep;
      const v4i xa = *reinterpret_cast<const v4i*>(xv), xb = *reinterpret_cast<const v4i*>(xv + 8);
#pragma unroll
      for (int t = 0; t < TPW; ++t) acc[u % R][t] = mma_block(wv[u][t], xa, xb, acc[u % R][t]);
    }
  }

  // Partials: lane 16 j + c holds rows 4j .. 4j+3 of column c; HALF's rows 8.. of column 1 are rows 0..
  // of the odd k-blocks.
  if (active && i == (HALF && j >= 2 ? 1 : 0)) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        if constexpr (HALF) red[2 * wave + (j >> 1)][t][j & 1] = acc[r][t];
        else red[gib * parts + ks + r * split][t][j] = acc[r][t];
      }
  }
  __syncthreads();
  if (ks != 0 || !active) return;
  // Lanes 16 j add the unit's partials of rows 4j .. in order; in a PAIR lanes 0 and 16 then take their
  // columns' up sums, rows 8.., from lanes 32 and 48.
  v4f sum[TPW], other[TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    // eight at a time, read without a branch; those past the unit are another's and left out
    v4f part[8], more[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) part[q] = red[(gib * parts + q) & 31][t][j];
    if constexpr (HALF || R == 2) {
#pragma unroll
      for (int q = 0; q < 8; ++q) more[q] = red[(gib * parts + 8 + q) & 31][t][j];
    }
    sum[t] = part[0];
#pragma unroll
    for (int q = 1; q < 8; ++q) {
      const v4f s = sum[t] + part[q];
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[t][r] = q < parts ? s[r] : sum[t][r];
    }
    if ((HALF || R == 2) && parts == 16) {
#pragma unroll
      for (int q = 0; q < 8; ++q) sum[t] += more[q];
    }
    if constexpr (PAIR) {
#pragma unroll
      for (int r = 0; r < 4; ++r) other[t][r] = __shfl_xor(sum[t][r], 32, 64);
    }
  }
  if (i != 0 || (SPLIT_ROWS && j >= 2)) return;
  if constexpr (ACT == 0)
    store_plain(p, sc, 0, sum[0], 0, n0);
  else
    store_act<ACT>(p, sc, sum[0], PAIR ? other[0] : sum[TPW - 1], 0, n0);
}

// Row-major int8 W [N, K] (ld = ldw) -> GEMV fragment layout, one thread per 16-byte piece;
// rows past N and k past K are zero.
__global__ __launch_bounds__(256) void pack_gemv_weight_kernel(const int8_t* __restrict__ w, int64_t ldw, int N, int K,
                                                               int KB, int64_t npieces, int8_t* __restrict__ out) {
  const int64_t c = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (c >= npieces) return;
  const int lane = int(c & 63);
  const int64_t f = c >> 6;
  const int t = int(f / KB), kb = int(f % KB);
  const int row = 16 * t + (lane & 15);
  const int k = 64 * kb + 16 * (lane >> 4);
  v4u v = {0u, 0u, 0u, 0u};
  if (row < N && k < K) v = *reinterpret_cast<const v4u*>(w + int64_t(row) * ldw + k);
  *reinterpret_cast<v4u*>(out + c * 16) = v;
}

static int gemv_cu_count() {
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) !=
                                                hipSuccess || n <= 0)
      n = 256;
    return n;
  }();
  return cus;
}

// Waves of a workgroup sharing one n-tile's K range on the few-tile shapes: doubled up to 16 while
// the chip holds fewer than ~4096 waves and each wave keeps two k-blocks, but not to 16 (1024-thread
// workgroups, one per CU) when there are more tiles than CUs: those would run in two rounds, where 8
// (two workgroups per CU) runs in one (the full-attention qkv, N = 5120: 12.5 -> 7.5 us).
static int few_tile_split(int64_t ntiles, int KB) {
  int split = 1;
  while (split < 16 && ntiles * split < 4096 && split * 2 <= KB) split *= 2;
  if (split == 16 && ntiles > gemv_cu_count()) split = 8;
  return split;
}

// The few-tile launch of what gemv1_takes leaves: per tile group `split` waves, NWB = split for 8 and 16.
template <bool PACKED, int TPW, int ACT>
static void gemv_launch_few(const GemvParams& p, int64_t groups, hipStream_t stream) {
  const int per_wave = (p.KB + p.split - 1) / p.split;
  if (p.split <= 4) {
    const int gpb = 4 / p.split;
    gemv_kernel<TPW, 4, PACKED, 4, ACT><<<unsigned((groups + gpb - 1) / gpb), 256, 0, stream>>>(p);
  } else if (p.split == 8) {
    gemv_kernel<TPW, 4, PACKED, 8, ACT><<<unsigned(groups), 512, 0, stream>>>(p);
  } else if (per_wave > 4 && per_wave <= 6) {
    // five or six k-blocks per wave (the down projection, K=6144): all of them in one round
    // trip instead of two
    gemv_kernel<TPW, 6, PACKED, 16, ACT><<<unsigned(groups), 1024, 0, stream>>>(p);
  } else {
    gemv_kernel<TPW, 4, PACKED, 16, ACT><<<unsigned(groups), 1024, 0, stream>>>(p);
  }
}

// One row: HALF where the 16-row tiles would leave half of the CUs without one.  A unit's few_tile_split
// partial sums are shared by up to 8 waves while a CU has one unit (HALF, or N <= 4096 on 256 CUs), by
// up to 4 from two units per CU on: the waves of a CU then stand evenly on its four SIMDs (3 or 6 waves per
// unit cost the gate/up GEMV 1-2 us more), and more waves only cost barriers (down 6144 x 1536 in halves:
// 16 waves 5.5 us, 8 waves 4.7, 6 waves 5.5).  The partial sums depend on (N, K) alone; the units per
// workgroup, which change no sum, are one, or with a row to make (the norm, the merge) up to twelve waves'
// worth, so that the row is made less often (gate/up 1536 x 12288: 8.4 us with one, 7.5 with three), eight
// waves' from 2048 tiles on, where a CU has several such workgroups anyway (33000 x 256 with its norm 6.1 ->
// 5.9 us, 65504 x 128 7.7 -> 7.35; 20000 x 128 with GELU 4.8 with twelve, 5.3 with eight).
// Sets units, split and gpb; the kernel's R, or 0 for HALF.
static int gemv1_plan(GemvParams& p, bool make_row) {
  const int cus = gemv_cu_count();
  const int ntiles = (p.N + 15) / 16;
  const bool half = 2 * ntiles <= cus;
  const int per_cu = half ? 1 : (ntiles + cus - 1) / cus;
  const int parts = few_tile_split(ntiles, p.KB);  // a power of two, above 8 only at one unit per CU
  p.units = half ? (p.N + 7) / 8 : ntiles;
  p.split = half ? max(parts / 2, 1) : min(per_cu == 1 ? 8 : 4, parts);
  p.gpb = make_row ? min(per_cu, (per_cu < 8 ? 12 : 8) / p.split) : 1;
  return half ? 0 : parts / p.split;
}

// Whether a call takes the one-row kernel: its row fits in LDS, and its tiles are few.  From 2048 tiles
// on a tile has one or two partial sums, and a workgroup of as many waves copying the row into LDS again
// costs more than it saves: N x K 50000 x 64 6.0 us here, 3.8 in gemv_kernel; 33000 x 256 5.1 and 4.4;
// 32768 x 1536 12.5 and 12.0; 65000 x 1536 the same.  Below, 20000 x 64 3.1 us here, 3.5 there before.
static bool gemv1_takes(const GemvParams& p) {
  return p.M == 1 && p.KB * 64 <= GEMV_ROW_MAX && (int64_t(p.N) + 15) / 16 < 2048;
}

// U fragments in flight per wave: all of a wave's share in one round where the registers allow it (seven or
// eight steps in one round of 8 rather than 12: 4096 x 4096 6.4 -> 6.1 us, row-major 7.4 -> 7.0, N = 16384,
// K = 2048 9.6 -> 8.5).  With the norm six at most, whose 80 registers let two workgroups of twelve waves
// stand on a CU, and four from 2048 tiles on (one or two waves per unit: N x K 32768 x 1536 18.2 us in rounds
// of 12 fragments, 14.2 in rounds of 6, 11.6 in rounds of 4 with eight waves; 40000 x 1024 11.8 -> 11.1).
// MI355X, weights cold, a chain of launches replayed from a graph (a chain of empty ones takes 1.9 us
// each), us per launch, before (one tile per workgroup of 8 or 16 waves, the row made by one wave, the
// scales fetched after the sums) -> now: o 2048 x 1536 4.5 -> 3.3, 4096 x 1536 5.5 -> 4.0; qkv 1536 x
// 2560 with its norm 6.3 -> 4.4; gate/up with norm and GELU 1536 x 12288 10.5 -> 6.9, x 24576 13.8 ->
// 10.6; down 6144 x 1536 7.0 -> 4.7, 12288 x 1536 10.5 -> 6.8; per-layer gate 1536 x 256 with norm
// 6.3 -> 4.4, projection 256 x 1536 3.3 -> 2.8.  (gate/up x 12288 and x 24576: 0.7 and 1.2 more before the
// packed widening and the branch-free row reads.  x 24576 needs its 80 registers, two workgroups of 12
// waves per CU: 13.0 at 85.)
template <bool PACKED, int ACT, int PRO>
static void gemv1_launch(const GemvParams& p0, hipStream_t stream) {
  GemvParams p = p0;
  // ACT 1 deals the same number of units of 8 gate and 8 up rows as the plain launch of N has
  // tiles, so its sums are made in the same order
  const int R = gemv1_plan(p, PRO != 5);
  const bool half = R == 0;
  // The merge reads every chunk's partials (64 KiB at 8 chunks of 8 heads of 256): both halves of a tile in
  // one workgroup make the row half as often (o projection 2048 x 1536, 8 chunks: 8.1 -> 7.3 us).
  if (PRO == 4 && half) p.gpb = 2;
  if (ACT == 1 && half) p.units = (p.N / 2 + 7) / 8;
  const int waves = max(p.gpb * p.split, PRO <= 3 ? PRO : 1);  // the norm's chunks each need a wave
  const dim3 grid(unsigned((p.units + p.gpb - 1) / p.gpb)), block(unsigned(waves * 64));
  const int steps = half ? (p.KB + 1) / 2 : p.KB;
  const int per_wave = (steps + p.split - 1) / p.split;
#define W8A8_GEMV1_WHOLE(U)                                                                      \
  do {                                                                                           \
    if (R == 2) gemv1_kernel<U, PACKED, ACT, PRO, false, 2><<<grid, block, 0, stream>>>(p);      \
    else gemv1_kernel<U, PACKED, ACT, PRO, false, 1><<<grid, block, 0, stream>>>(p);             \
  } while (0)
#define W8A8_GEMV1(U)                                                                            \
  do {                                                                                           \
    if (half) gemv1_kernel<U, PACKED, ACT, PRO, true, 1><<<grid, block, 0, stream>>>(p);         \
    else W8A8_GEMV1_WHOLE(U);                                                                    \
  } while (0)
  if (per_wave <= 1) W8A8_GEMV1(1);
  else if (per_wave <= 2) W8A8_GEMV1(2);
  else if (per_wave <= 3) W8A8_GEMV1(3);
  else if (per_wave <= 4 || (ACT == 1 && half) || (PRO <= 3 && p.split < 4)) W8A8_GEMV1(4);
  else if (per_wave <= 6 || half || PRO != 5) W8A8_GEMV1(6);
  else if (per_wave <= 8) W8A8_GEMV1_WHOLE(8);
  else W8A8_GEMV1_WHOLE(PRO != 5 ? 8 : 12);
#undef W8A8_GEMV1
#undef W8A8_GEMV1_WHOLE
}

template <bool PACKED>
static void gemv_launch(const GemvParams& p0, hipStream_t stream) {
  GemvParams p = p0;
  if (gemv1_takes(p)) return gemv1_launch<PACKED, 0, 5>(p, stream);
  const int64_t ntiles = (p.N + 15) / 16;
  if (ntiles >= 4096) {
    // Many n-tiles (the LM head): each activation fragment serves two (M <= 8) or four
    // weight tiles per wave.
    p.split = 1;
    if (p.M <= 8) {
      const int64_t groups = (ntiles + 1) / 2;
      gemv_kernel<2, 4, PACKED, 4><<<unsigned((groups + 3) / 4), 256, 0, stream>>>(p);
    } else {
      const int64_t groups = (ntiles + 3) / 4;
      gemv_kernel<4, 2, PACKED, 4><<<unsigned((groups + 3) / 4), 256, 0, stream>>>(p);
    }
    return;
  }
  // Few n-tiles (the per-layer decode shapes: 96-768 tiles): one tile per group of `split`
  // waves that share its K range, up to 16 waves of one workgroup, aiming for ~4096 waves over
  // the chip's 1024 SIMDs, each with at least two k-blocks.
  p.split = few_tile_split(ntiles, p.KB);
  gemv_launch_few<PACKED, 1, 0>(p, ntiles, stream);
}

// The packed few-tile launch with an activation epilogue: ACT 1 over I / 16 gate/up tile pairs (two
// tiles per wave), ACT 2 over the N / 16 tiles.  The split is the plain launch's for the whole N, so
// every tile's sum is added in the same order and the result is the plain GEMV's, bit for bit,
// before the activation.
template <int ACT>
static void gemv_launch_act(const GemvParams& p0, hipStream_t stream) {
  GemvParams p = p0;
  if (gemv1_takes(p)) return gemv1_launch<true, ACT, 5>(p, stream);
  const int64_t ntiles = (p.N + 15) / 16;
  p.split = few_tile_split(ntiles, p.KB);
  gemv_launch_few<true, ACT == 1 ? 2 : 1, ACT>(p, ACT == 1 ? p.half_tiles : ntiles, stream);
}

}  // namespace w8a8

using namespace w8a8;

extern "C" int64_t w8a8_gemv_packed_bytes(int64_t N, int64_t K) {
  if (N < 1 || K < 1 || N > INT32_MAX || K > INT32_MAX) return -1;
  return (N + 15) / 16 * ((K + 63) / 64) * 1024;
}

extern "C" int w8a8_pack_gemv_weight(const int8_t* w, int64_t ldw, int64_t N, int64_t K, int8_t* packed,
                                     hipStream_t stream) {
  if (!w || !packed) return fail(W8A8_EINVAL, "pack_gemv_weight: null pointer");
  if (N < 1 || K < 16 || ldw < K) return fail(W8A8_EINVAL, "pack_gemv_weight: bad shape N=%lld K=%lld ldw=%lld",
                                              (long long)N, (long long)K, (long long)ldw);
  if (K % 16 != 0) return fail(W8A8_ENOTSUP, "pack_gemv_weight: K=%lld must be a multiple of 16", (long long)K);
  if (ldw % 16 != 0 || (uintptr_t)w % 16 != 0 || (uintptr_t)packed % 16 != 0)
    return fail(W8A8_EALIGN, "pack_gemv_weight: w rows and packed must be 16-byte aligned");
  const int64_t bytes = w8a8_gemv_packed_bytes(N, K);
  if (bytes < 0 || bytes > INT32_MAX + 1ll) return fail(W8A8_ENOTSUP, "pack_gemv_weight: packed weight above 2 GiB");
  const int64_t pieces = bytes / 16;
  pack_gemv_weight_kernel<<<unsigned((pieces + 255) / 256), 256, 0, stream>>>(w, ldw, int(N), int(K),
                                                                            int((K + 63) / 64), pieces, packed);
  return check_launch("pack_gemv_weight");
}

extern "C" int w8a8_gemv_packed_bf16(const uint16_t* x, int64_t ldx, int64_t M, const int8_t* packed, int64_t N,
                                     int64_t K, const void* scales, int scale_is_f32, uint16_t* y, int64_t ldy,
                                     hipStream_t stream) {
  if (!x || !packed || !scales || !y) return fail(W8A8_EINVAL, "gemv_packed: null pointer");
  if (M < 1 || M > 16) return fail(W8A8_EINVAL, "gemv_packed: M=%lld, the GEMV takes 1..16 rows", (long long)M);
  if (N < 1 || K < 16) return fail(W8A8_EINVAL, "gemv_packed: bad shape N=%lld K=%lld", (long long)N, (long long)K);
  if (K % 16 != 0) return fail(W8A8_ENOTSUP, "gemv_packed: K=%lld must be a multiple of 16", (long long)K);
  if (ldx < K || ldy < N) return fail(W8A8_EINVAL, "gemv_packed: leading dimension too small");
  if (ldx % 8 != 0 || (uintptr_t)x % 16 != 0 || (uintptr_t)packed % 16 != 0)
    return fail(W8A8_EALIGN, "gemv_packed: x rows and the packed weight must be 16-byte aligned");
  const int64_t wb = w8a8_gemv_packed_bytes(N, K);
  const int64_t xb = ((M - 1) * ldx + K) * 2;
  if (wb > INT32_MAX || xb > INT32_MAX) return fail(W8A8_ENOTSUP, "gemv_packed: operands above 2 GiB");
  GemvParams p;
  p.x = x; p.ldx = ldx; p.w = packed; p.ldw = 0; p.s = scales; p.s_f32 = scale_is_f32 ? 1 : 0;
  p.y = y; p.ldy = ldy; p.x_bytes = uint32_t(xb); p.w_bytes = uint32_t(wb);
  p.M = int(M); p.N = int(N); p.K = int(K); p.KB = int((K + 63) / 64);
  gemv_launch<true>(p, stream);
  return check_launch("gemv_packed_bf16");
}

extern "C" int w8a8_gemv_packed_act_bf16(const uint16_t* x, int64_t ldx, int64_t M, const int8_t* packed, int64_t N,
                                         int64_t K, const void* scales, int scale_is_f32, int act, const uint16_t* mul,
                                         int64_t ldm, uint16_t* y, int64_t ldy, hipStream_t stream) {
  if (!x || !packed || !scales || !y || (act == 2 && !mul)) return fail(W8A8_EINVAL, "gemv_packed_act: null pointer");
  if (act != 1 && act != 2) return fail(W8A8_EINVAL, "gemv_packed_act: act %d (1: GELU pair, 2: GELU times mul)", act);
  if (M < 1 || M > 16) return fail(W8A8_EINVAL, "gemv_packed_act: M=%lld, the GEMV takes 1..16 rows", (long long)M);
  if (N < 1 || K < 16) return fail(W8A8_EINVAL, "gemv_packed_act: bad shape N=%lld K=%lld", (long long)N, (long long)K);
  if (K % 16 != 0) return fail(W8A8_ENOTSUP, "gemv_packed_act: K=%lld must be a multiple of 16", (long long)K);
  if (act == 1 && N % 32 != 0)
    return fail(W8A8_ENOTSUP, "gemv_packed_act: a GELU pair needs N = 2I with I a multiple of 16, got N=%lld",
                (long long)N);
  const int64_t nout = act == 1 ? N / 2 : N;
  if ((N + 15) / 16 >= 4096) return fail(W8A8_ENOTSUP, "gemv_packed_act: N=%lld above the few-tile shapes", (long long)N);
  if (ldx < K || ldy < nout || (act == 2 && ldm < N)) return fail(W8A8_EINVAL, "gemv_packed_act: leading dimension too small");
  if (ldx % 8 != 0 || (uintptr_t)x % 16 != 0 || (uintptr_t)packed % 16 != 0)
    return fail(W8A8_EALIGN, "gemv_packed_act: x rows and the packed weight must be 16-byte aligned");
  const int64_t wb = w8a8_gemv_packed_bytes(N, K);
  const int64_t xb = ((M - 1) * ldx + K) * 2;
  if (wb > INT32_MAX || xb > INT32_MAX) return fail(W8A8_ENOTSUP, "gemv_packed_act: operands above 2 GiB");
  GemvParams p{};
  p.x = x; p.ldx = ldx; p.w = packed; p.ldw = 0; p.s = scales; p.s_f32 = scale_is_f32 ? 1 : 0;
  p.y = y; p.ldy = ldy; p.x_bytes = uint32_t(xb); p.w_bytes = uint32_t(wb);
  p.M = int(M); p.N = int(N); p.K = int(K); p.KB = int((K + 63) / 64);
  p.mul = mul; p.ldm = ldm; p.half_tiles = int(N / 32);
  if (act == 1)
    gemv_launch_act<1>(p, stream);
  else
    gemv_launch_act<2>(p, stream);
  return check_launch("gemv_packed_act_bf16");
}

static bool overlaps(const void* a, int64_t abytes, const void* b, int64_t bbytes) {
  if (!a || !b) return false;
  const uintptr_t a0 = reinterpret_cast<uintptr_t>(a), b0 = reinterpret_cast<uintptr_t>(b);
  return a0 < b0 + uintptr_t(bbytes) && b0 < a0 + uintptr_t(abytes);
}

extern "C" int w8a8_gemv_packed_norm_bf16(const uint16_t* y, const uint16_t* res, const uint16_t* w1,
                                          const uint16_t* scalar, int norm2, const uint16_t* w2, float eps, uint16_t* h,
                                          const int8_t* packed, int64_t N, int64_t K, const void* scales,
                                          int scale_is_f32, int act, const uint16_t* mul, uint16_t* out,
                                          hipStream_t stream) {
  const char* what = "gemv_packed_norm";
  if (!y || !packed || !scales || !out || (act == 2 && !mul)) return fail(W8A8_EINVAL, "%s: null pointer", what);
  if (act < 0 || act > 2) return fail(W8A8_EINVAL, "%s: act %d (0: none, 1: GELU pair, 2: GELU times mul)", what, act);
  if (N < 1 || K < 16) return fail(W8A8_EINVAL, "%s: bad shape N=%lld K=%lld", what, (long long)N, (long long)K);
  if (K % 16 != 0) return fail(W8A8_ENOTSUP, "%s: K=%lld must be a multiple of 16", what, (long long)K);
  if (K > 1536) return fail(W8A8_ENOTSUP, "%s: K=%lld above the prologue's row of 1536", what, (long long)K);
  if ((N + 15) / 16 >= 4096) return fail(W8A8_ENOTSUP, "%s: N=%lld above the few-tile shapes", what, (long long)N);
  if (act == 1 && N % 32 != 0)
    return fail(W8A8_ENOTSUP, "%s: a GELU pair needs N = 2I with I a multiple of 16, got N=%lld", what, (long long)N);
  for (const void* q : {static_cast<const void*>(y), static_cast<const void*>(res), static_cast<const void*>(w1),
                        static_cast<const void*>(w2), static_cast<const void*>(h), static_cast<const void*>(packed)})
    if ((reinterpret_cast<uintptr_t>(q) & 15) != 0)
      return fail(W8A8_EALIGN, "%s: the rows, norm weights and packed weight must be 16-byte aligned", what);
  const int64_t nout = act == 1 ? N / 2 : N;
  const int64_t rb = K * 2, ob = nout * 2;
  // every workgroup reads y and res while workgroup 0 writes h and all of them write out
  if (overlaps(h, rb, y, rb) || overlaps(h, rb, res, rb) || overlaps(h, rb, out, ob))
    return fail(W8A8_EINVAL, "%s: h must not overlap y, res or out", what);
  if (overlaps(out, ob, y, rb) || overlaps(out, ob, res, rb) || (act == 2 && overlaps(out, ob, mul, N * 2)))
    return fail(W8A8_EINVAL, "%s: out must not overlap y, res or mul", what);
  const int64_t wb = w8a8_gemv_packed_bytes(N, K);
  if (wb > INT32_MAX) return fail(W8A8_ENOTSUP, "%s: packed weight above 2 GiB", what);
  GemvParams p{};
  p.x = nullptr; p.ldx = K; p.w = packed; p.ldw = 0; p.s = scales; p.s_f32 = scale_is_f32 ? 1 : 0;
  p.y = out; p.ldy = nout; p.x_bytes = 0; p.w_bytes = uint32_t(wb);
  p.M = 1; p.N = int(N); p.K = int(K); p.KB = int((K + 63) / 64);
  p.mul = mul; p.ldm = N; p.half_tiles = int(N / 32);
  p.pro_y = y; p.pro_res = res; p.pro_w1 = w1; p.pro_scalar = scalar; p.pro_w2 = w2; p.pro_h = h;
  p.pro_eps = eps; p.pro_norm2 = norm2 ? 1 : 0;
  if (act == 0) gemv1_launch<true, 0, 3>(p, stream);
  else if (act == 1) gemv1_launch<true, 1, 3>(p, stream);
  else gemv1_launch<true, 2, 3>(p, stream);
  return check_launch("gemv_packed_norm_bf16");
}

extern "C" int w8a8_gemv_packed_attn_merge_bf16(const void* workspace, const int32_t* q_pos, int64_t H, int64_t KV,
                                                int64_t Tk, int64_t D, int64_t window, float scale,
                                                const int8_t* packed, int64_t N, const void* scales, int scale_is_f32,
                                                uint16_t* out, hipStream_t stream) {
  const char* what = "gemv_packed_attn_merge";
  if (!workspace || !q_pos || !packed || !scales || !out) return fail(W8A8_EINVAL, "%s: null pointer", what);
  if (H < 1 || KV < 1 || H % KV != 0 || H / KV > 16)
    return fail(W8A8_EINVAL, "%s: H=%lld KV=%lld (H a multiple of KV, at most 16 per KV head)", what, (long long)H,
                (long long)KV);
  if (D != 128 && D != 256 && D != 512) return fail(W8A8_ENOTSUP, "%s: head_dim %lld", what, (long long)D);
  if (Tk < 1 || Tk > INT32_MAX || window < 0 || window > INT32_MAX)
    return fail(W8A8_EINVAL, "%s: Tk=%lld window=%lld", what, (long long)Tk, (long long)window);
  const int nchunk_grid = decode_grid_chunks(D, Tk, window);
  if (nchunk_grid > DEC_MERGE_IN_GEMV_CHUNKS)
    return fail(W8A8_ENOTSUP, "%s: %d key chunks (at most %d)", what, nchunk_grid, DEC_MERGE_IN_GEMV_CHUNKS);
  const int64_t K = H * D;
  if (K > 4096) return fail(W8A8_ENOTSUP, "%s: H * D = %lld above 4096", what, (long long)K);
  if (N < 1 || (N + 15) / 16 >= 4096) return fail(W8A8_ENOTSUP, "%s: N=%lld outside the few-tile shapes", what, (long long)N);
  if (!(scale > 0.0f) || scale == __builtin_inff()) return fail(W8A8_EINVAL, "%s: scale must be positive", what);
  if ((uintptr_t)workspace % 16 || (uintptr_t)packed % 16 || (uintptr_t)q_pos % 4)
    return fail(W8A8_EALIGN, "%s: workspace and packed 16-byte aligned, q_pos 4-byte aligned", what);
  const int64_t wb = w8a8_gemv_packed_bytes(N, K);
  if (wb > INT32_MAX) return fail(W8A8_ENOTSUP, "%s: packed weight above 2 GiB", what);
  GemvParams p{};
  p.x = nullptr; p.ldx = K; p.w = packed; p.ldw = 0; p.s = scales; p.s_f32 = scale_is_f32 ? 1 : 0;
  p.y = out; p.ldy = N; p.x_bytes = 0; p.w_bytes = uint32_t(wb);
  p.M = 1; p.N = int(N); p.K = int(K); p.KB = int((K + 63) / 64);
  const int G = int(H / KV);
  p.m_po = static_cast<const float*>(workspace);
  p.m_ml = p.m_po + int64_t(KV) * nchunk_grid * G * D;
  p.m_pos = q_pos; p.m_window = int(window); p.m_nchunk_grid = nchunk_grid; p.m_G = G; p.m_D = int(D);
  p.m_chunk = dec_chunk(int(D));
  p.m_c = scale * 1.4426950408889634f;  // the attention's exp2 factor, computed as it computes it
  gemv1_launch<true, 0, 4>(p, stream);
  return check_launch("gemv_packed_attn_merge_bf16");
}

extern "C" int w8a8_gemv_bf16(const uint16_t* x, int64_t ldx, int64_t M, const int8_t* w, int64_t ldw, int64_t N,
                              int64_t K, const void* scales, int scale_is_f32, uint16_t* y, int64_t ldy,
                              hipStream_t stream) {
  if (!x || !w || !scales || !y) return fail(W8A8_EINVAL, "gemv: null pointer");
  if (M < 1 || M > 16) return fail(W8A8_EINVAL, "gemv: M=%lld, the GEMV takes 1..16 rows", (long long)M);
  if (N < 1 || K < 16) return fail(W8A8_EINVAL, "gemv: bad shape N=%lld K=%lld", (long long)N, (long long)K);
  if (K % 16 != 0) return fail(W8A8_ENOTSUP, "gemv: K=%lld must be a multiple of 16", (long long)K);
  if (ldx < K || ldw < K || ldy < N) return fail(W8A8_EINVAL, "gemv: leading dimension too small");
  if (ldx % 8 != 0 || ldw % 16 != 0 || (uintptr_t)x % 16 != 0 || (uintptr_t)w % 16 != 0)
    return fail(W8A8_EALIGN, "gemv: x and w rows must be 16-byte aligned (ldx %% 8, ldw %% 16)");
  const int64_t wb = (N - 1) * ldw + K;
  const int64_t xb = ((M - 1) * ldx + K) * 2;
  if (wb > INT32_MAX || xb > INT32_MAX) return fail(W8A8_ENOTSUP, "gemv: operands above 2 GiB");
  GemvParams p;
  p.x = x; p.ldx = ldx; p.w = w; p.ldw = ldw; p.s = scales; p.s_f32 = scale_is_f32 ? 1 : 0;
  p.y = y; p.ldy = ldy; p.x_bytes = uint32_t(xb); p.w_bytes = uint32_t(wb);
  p.M = int(M); p.N = int(N); p.K = int(K); p.KB = int((K + 63) / 64);
  gemv_launch<false>(p, stream);
  return check_launch("gemv_bf16");
}
