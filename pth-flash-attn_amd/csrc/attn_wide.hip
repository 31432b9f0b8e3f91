// attn_wide.hip -- the gfx950 wide-block kernel: prefill launches at head size
// D = 64, 128 or 256 on paged cell caches (block size a multiple of 16), with
// or without split partials.
//
// A work-group takes a block of 32 query rows per wave (256 rows at D = 64
// and 128, 128 rows at D = 256) of one request and one KV head, and all its
// waves share one stream of keys: each step loads 8 keys per wave, converts
// them once (K to the query's 16-bit type, V to bf16, both exact for int8)
// and every wave multiplies its rows with all of them. The unit kernels, which
// these launches ran on before, pass over the keys once per 16 rows and
// convert them each time.
//
// Layout. v_mfma_f32_32x32x16 with the keys (or the output columns) on M and
// the wave's 32 query rows on N, so a lane owns one row: lane l holds row
// l % 32, and of a 32-key score tile the keys 8 b + 4 (l / 32) + i (b, i < 4).
// These are the B operand of the PV product as they are, if its A operand
// takes V in the same key order: ds_read_b64_tr_b16 gives each lane one
// column of four consecutive keys from a row-major V, so V needs no
// transposition when it is written. Row paddings (K 16, V 32 bytes) spread
// both reads over the LDS banks (b128 reads 2.3 ns each with eight waves
// against 26.8 without, transposing reads 1.7 against 3.4).
//
// Numerics. As the unit kernels of attn_fwd.hip: P is a bf16 hi + lo pair (16
// significant bits at any size), a row's reference max moves when a score
// exceeds it by more than kRescaleSlack. Here it is a whole number, so that
// every rescale factor is a power of two and the pending P of the previous
// step is rescaled without rounding. An fp16 query takes K in fp16 (one product
// instead of the unit kernels' two). A key whose p is 0, masked or more than
// 2^126 below the row's largest, adds nothing whatever its V scale.
//
// Pipeline. Step k multiplies K(k) with Q, then runs softmax(k) while the
// matrix unit works on P(k - 1) V(k - 1), which is independent of it: a step
// has about as much vector as matrix work. V is therefore kept one step
// longer than K (three V buffers, two K buffers). Loads go to registers one
// step ahead of their conversion.
//
// Bound: issue. A 32x32x16 product occupies its SIMD's vector issue for 16 of
// its 32 cycles (measured with independent fmas beside it), so per step and
// wave at D = 128 the 48 products, ~330 vector instructions and 32 exp2 take
// at least 2,220 cycles, two waves per SIMD 4,440; a step takes ~6,100, at
// 1.84 GHz. Measured, this kernel alone (D = 128: 16q / 4kv, a chunk of 2,011
// tokens at 6,101 of a prefix, fp16; D = 64: 32q / 8kv, chunks of 1,108 and 1,389
// tokens at 7,548 and 4,187; D = 256: 12q / 2kv, 2,048 tokens at 4,099):
//                   D = 128    D = 64   D = 256
//   unit kernels     460 us  2,091 us    375 us
//   this             201       270       246
// Tried on a version with P in fp16 (195 us; D = 64 303 us for the whole call):
//   64 rows per wave, one wave per SIMD, half the LDS reads  206 us     348 us
//   cache bytes direct to a ring in LDS, 2-4 steps ahead     202 us     314 us
//   one softmax part forced after each product               206 us     314 us
//   waves 4-7 half a step behind waves 0-3                  (spills)    347 us
// P in fp16 has 22 bits near a row's largest p, but a floor: weights 2^18 and more
// below the largest lost bits or vanished from the output while l counted them
// (measured: up to a quarter of an element's sum of p |v|, 3e-3 of it on a long
// context with one large V scale).

#include "attn_device.h"

namespace pa {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef int16_t i16x4 __attribute__((ext_vector_type(4)));

constexpr int kWideRows = 32;  // rows per wave
template <int D>
struct WideDim {
  // D = 256 keeps 128 output and 64 query registers per lane: one wave per
  // SIMD, all 512 registers. Smaller heads run two.
  static constexpr int kWaves = D == 256 ? 4 : 8;
  static constexpr int kPerSimd = D == 256 ? 1 : 2;
  static constexpr int kThreads = 64 * kWaves;
  static constexpr int kBlock = kWideRows * kWaves;  // rows per block
  static constexpr int kStep = 8 * kWaves;           // keys per step
  static constexpr int kTiles = kStep / 32;          // 32-key score tiles per step
  static constexpr int kSub = kStep / 16;            // 16-key PV products per step
  static constexpr int kQ = D / 16;                  // Q operands (16 columns each)
  static constexpr int kO = D / 32;                  // output tiles (32 columns each)
  static constexpr int kAhead = 4;                   // K operands read ahead
  static constexpr int kLaneBytes = D / 8;           // cache bytes per lane, step and stream
  static constexpr int kKRow = 2 * D + 16;           // LDS bytes per key row
  static constexpr int kVRow = 2 * D + 32;
  static constexpr int kKBuf = kStep * kKRow;
  static constexpr int kVBuf = kStep * kVRow;
  static constexpr int kSBuf = 8 * kStep;            // K scales, then V scales
  static constexpr int kVBase = 2 * kKBuf;
  static constexpr int kSBase = kVBase + 3 * kVBuf;
  static constexpr int kLds = kSBase + 2 * kSBuf;
  static_assert(kLds <= 160 * 1024, "wide-block LDS");
};

__device__ __forceinline__ int sgpr(int x) { return __builtin_amdgcn_readfirstlane(x); }

// One run of keys of one row block: what a work-group computes at a time.
struct Segment {
  RowTile t;
  int kvh;
  int lo, hi;   // keys the segment reads: [lo, hi)
  int s, live;  // split index and the stream's splits
};

// The segments of one work-group. num_splits > 1: the chunk-stream partition
// of attn_geometry.h over the row blocks (a stream per block and KV head).
// num_splits == 1: whole blocks, the last token blocks of a request (the
// longest key ranges) first, dealt in rounds of W in alternating order.
template <bool kWindow, bool kStream>
struct WideWalk {
  StreamCursor sc;
  StreamDesc d;
  int64_t pos = 0, stop = 0, per = 1;
  int r0 = -64, u0 = 0, u1 = 0, incl = 0, round = 0;

  __device__ __forceinline__ void init(const AttnParams& p, int lane) {
    if constexpr (kStream) {
      d = StreamDesc{p.qsl, p.seq_lens, p.num_reqs, p.blk_tok, kWindow ? p.window : 0,
                     kWindow ? p.causal : 1, p.num_kv_heads, static_cast<int32_t>(gridDim.x),
                     p.num_splits};
      int64_t total;
      per = stream_per_cursor(d, lane, total, sc);
      pos = static_cast<int64_t>(blockIdx.x) * per + kStreamStartPositions;
      stop = pos + per < total ? pos + per : total;
    }
  }

  __device__ __forceinline__ bool next(const AttnParams& p, int lane, Segment& g) {
    const int window = kWindow ? p.window : 0;
    const bool causal = kWindow ? (p.causal != 0) : true;
    int c_lo = 0, c_hi = 0x7fffffff;
    if constexpr (kStream) {
      while (true) {
        if (pos >= stop) return false;
        StreamPos sp;
        if (!stream_locate(d, sc, pos, lane, sp)) return false;
        const int64_t cs = sp.c0 + kStreamStartPositions;
        const int c0 = pos > cs ? static_cast<int>(pos - cs) : 0;
        const int64_t end = cs + sp.n < stop ? cs + sp.n : stop;
        const int c1 = static_cast<int>(end - cs);
        pos = end > pos ? end : pos + 1;
        // A row without any visible key (n == 0) has no position, so it is
        // never a segment here: it has none to read and its rows are none.
        if (c1 <= c0) continue;
        int first;
        stream_splits(sp.c0, sp.n, per, first, g.live);
        g.s = static_cast<int>(blockIdx.x) - first;
        g.t = sp.t;
        g.kvh = sp.hg;
        c_lo = sp.cb + kChunkTokens * c0;
        c_hi = sp.cb + kChunkTokens * c1;
        break;
      }
    } else {
      const int W = gridDim.x;
      const int u = round * W + ((round & 1) ? W - 1 - static_cast<int>(blockIdx.x)
                                             : static_cast<int>(blockIdx.x));
      ++round;
      while (u >= u1) {
        r0 += 64;
        u0 = u1;
        if (r0 >= p.num_reqs) return false;
        const int r = r0 + lane;
        const int units = r < p.num_reqs ? request_row_tiles(p.qsl[r + 1] - p.qsl[r], p.blk_tok) *
                                               p.num_kv_heads
                                         : 0;
        incl = wave_scan32(units);
        u1 = u0 + __builtin_amdgcn_readlane(incl, 63);
      }
      const int local = u - u0;
      const int j = static_cast<int>(__popcll(__ballot(incl <= local)));
      const int req = r0 + j;
      const int u_loc = local - (j > 0 ? __builtin_amdgcn_readlane(incl, j - 1) : 0);
      const int q_start = ld_ro(p.qsl, req);
      const int q_len = ld_ro(p.qsl, req + 1) - q_start;
      const int seq_len = ld_ro(p.seq_lens, req);
      const int nb = request_row_tiles(q_len, p.blk_tok);
      const int jb = u_loc / p.num_kv_heads;
      g.t = request_tile(req, q_start, q_len, seq_len, p.blk_tok, nb - 1 - jb);
      g.kvh = u_loc - jb * p.num_kv_heads;
      g.s = 0;
      g.live = 1;
    }
    const int lo = range_begin(g.t, window), hi = range_end(g.t, window, causal);
    g.lo = c_lo > lo ? c_lo : lo;
    g.hi = c_hi < hi ? c_hi : hi;
    g.t.req = sgpr(g.t.req);
    g.t.tok_begin = sgpr(g.t.tok_begin);
    g.t.num_tok = sgpr(g.t.num_tok);
    g.t.q_len = sgpr(g.t.q_len);
    g.t.seq_len = sgpr(g.t.seq_len);
    g.t.q_start = sgpr(g.t.q_start);
    g.kvh = sgpr(g.kvh);
    g.lo = sgpr(g.lo);
    g.hi = sgpr(g.hi);
    g.s = sgpr(g.s);
    g.live = sgpr(g.live);
    return true;
  }
};

// A lane's row of a 32-row group of the block.
struct WideLanes {
  bool vrow;
  int head;
  int64_t qtok;
  int lo, hi;  // the row's visible keys [lo, hi] of the segment
};

// The wave's mask bounds: every row of it sees all keys of [lo_max, hi_min].
struct WideBounds {
  int lo_max, hi_min;
};

template <bool kWindow>
__device__ __forceinline__ WideLanes wide_lanes(const AttnParams& p, const Segment& g, int row0,
                                                int lane) {
  const int window = kWindow ? p.window : 0;
  const bool causal = kWindow ? (p.causal != 0) : true;
  const int rows = g.t.num_tok * p.group;
  WideLanes L;
  const int row = row0 + (lane & 31);
  L.vrow = row < rows;
  const int rr = L.vrow ? row : 0;
  const int tok = static_cast<int>(p.g_div.div(static_cast<uint32_t>(rr)));
  L.head = g.kvh * p.group + (rr - tok * p.group);
  L.qtok = static_cast<int64_t>(g.t.q_start) + g.t.tok_begin + tok;
  // Only the segment's keys: a step reaches past its ends.
  L.lo = max(key_lo(g.t, g.t.tok_begin + tok, window), g.lo);
  L.hi = min(key_hi(g.t, g.t.tok_begin + tok, window, causal), g.hi - 1);
  return L;
}

template <bool kWindow>
__device__ __forceinline__ WideBounds wide_bounds(const AttnParams& p, const Segment& g, int row0,
                                                  int n) {
  const int window = kWindow ? p.window : 0;
  const bool causal = kWindow ? (p.causal != 0) : true;
  const int rows = g.t.num_tok * p.group;
  const int last = row0 + n < rows ? row0 + n - 1 : rows - 1;
  const int tok_first = static_cast<int>(p.g_div.div(static_cast<uint32_t>(row0)));
  const int tok_last = static_cast<int>(p.g_div.div(static_cast<uint32_t>(last)));
  WideBounds b;
  b.lo_max = max(key_lo(g.t, g.t.tok_begin + tok_last, window), g.lo);
  b.hi_min = min(key_hi(g.t, g.t.tok_begin + tok_first, window, causal), g.hi - 1);
  return b;
}

// The wave's 8 keys of a step lie in one 16-key group of one page. Its block
// ids come from a register that holds 64 consecutive entries of the request's
// block-table row (lane l: entry win + l), the next 64 loaded when it comes
// into use: a lane read per step, no load to wait for.
struct PageWindow {
  const int32_t* row;
  int win, last;  // first entry of `cur`; the row's last entry a load may read
  int cur, nxt;
};

__device__ __forceinline__ int window_load(const PageWindow& w, int first, int lane) {
  const int e = first + lane;
  return w.row[e < w.last ? e : w.last];
}

// Moves the window on to the one of block blk, if it is the next. The new
// entries are waited for here, once in 64 blocks: left in flight, every step
// would wait for them.
__device__ __forceinline__ void page_window(PageWindow& w, int blk, int lane) {
  if (blk - w.win < 64) return;
  w.win += 64;
  w.cur = w.nxt;
  w.nxt = window_load(w, w.win + 64, lane);
  asm volatile("s_waitcnt vmcnt(0)" : "+v"(w.nxt));
}

// One step's cache bytes of a lane: key 8 wave + lane / 8 of the step, bytes
// [(lane % 8) D / 8, + D / 8) of its K and V rows; and the scale of key
// 8 wave + lane % 8 (lanes with lane & 8: the V scale, else the K scale).
template <int D>
struct WideRaw {
  uint32_t k[WideDim<D>::kLaneBytes / 4], v[WideDim<D>::kLaneBytes / 4];
  float s;
};

template <int N>
__device__ __forceinline__ void wide_words(const char* src, uint32_t (&w)[N]) {
  if constexpr (N == 2) {
    const u32x2 x = *reinterpret_cast<const u32x2_a4*>(src);
    w[0] = x[0];
    w[1] = x[1];
  } else {
#pragma unroll
    for (int i = 0; i < N; i += 4) {
      const u32x4 x = *reinterpret_cast<const u32x4_a4*>(src + 4 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) w[i + j] = x[j];
    }
  }
}

struct WideOffsets {
  uint32_t kv, s;  // lane offsets from the wave's 16-key group
};

// The 16-key group that the wave loads for the step at key c: its block and
// first slot. Groups past the segment's last key (last16) read that key's
// group again (their scales are staged as 0).
struct KeyGroup {
  int blk, slot0;
};

__device__ __forceinline__ KeyGroup key_group(const AttnParams& p, int c, int wave, int last16) {
  int k16 = (c + 8 * wave) & ~15;
  k16 = k16 < last16 ? k16 : last16;
  KeyGroup g;
  // Blocks of at least 16 keys: never the division by one.
  g.blk = static_cast<int>(mulhi32(static_cast<uint32_t>(k16), p.bs_div.mul) >> p.bs_div.shift);
  g.slot0 = k16 - g.blk * static_cast<int>(p.bs_div.d);
  return g;
}

template <int D>
__device__ __forceinline__ void wide_load(const AttnParams& p, const PageWindow& w,
                                          const WideOffsets& o, const KeyGroup& g,
                                          WideRaw<D>& r) {
  const int page = __builtin_amdgcn_readlane(w.cur, g.blk - w.win);
  const char* base = p.cell_base +
                     static_cast<uint64_t>(static_cast<uint32_t>(page)) * p.cell_block +
                     static_cast<uint32_t>(g.slot0) * p.cell_slot;
  wide_words(base + p.cell_off[0] + o.kv, r.k);
  wide_words(base + p.cell_off[1] + o.kv, r.v);
  r.s = *reinterpret_cast<const float*>(base + o.s);
}

// Four int8 -> four fp16 (exact).
__device__ __forceinline__ u32x2 i8x4_to_f16(uint32_t w) {
  u32x2 r;
  r[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(i8_to_f32(w, 0), i8_to_f32(w, 1)));
  r[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(i8_to_f32(w, 2), i8_to_f32(w, 3)));
  return r;
}

__device__ __forceinline__ u32x2 i8x4_to_bf16(uint32_t w) {
  u32x2 r;
  r[0] = __builtin_bit_cast(uint32_t, pack_bf16(i8_to_f32(w, 0), i8_to_f32(w, 1)));
  r[1] = __builtin_bit_cast(uint32_t, pack_bf16(i8_to_f32(w, 2), i8_to_f32(w, 3)));
  return r;
}

// Converts word pair i of a step's bytes (the K words, then the V words) and
// writes it row-major: K as the query's 16-bit type, V as bf16.
template <int D, bool kF16Q>
__device__ __forceinline__ void wide_stage_pair(const WideRaw<D>& r, int i, char* kdst,
                                                char* vdst) {
  constexpr int kHalf = WideDim<D>::kLaneBytes / 8;
  const bool is_v = i >= kHalf;
  const int w = 2 * (is_v ? i - kHalf : i);
  const uint32_t w0 = is_v ? r.v[w] : r.k[w], w1 = is_v ? r.v[w + 1] : r.k[w + 1];
  const u32x2 a = kF16Q && !is_v ? i8x4_to_f16(w0) : i8x4_to_bf16(w0);
  const u32x2 b = kF16Q && !is_v ? i8x4_to_f16(w1) : i8x4_to_bf16(w1);
  *reinterpret_cast<u32x4*>((is_v ? vdst : kdst) + 8 * w) = (u32x4){a[0], a[1], b[0], b[1]};
}

// All of a step, with its scales: the K scale times scale * log2 e, the V
// scale; 0 for a key outside the segment (its cache bytes may be any bits).
template <int D, bool kF16Q>
__device__ __forceinline__ void wide_stage(const WideRaw<D>& r, char* kdst, char* vdst, char* sdst,
                                           bool live_key, float smul) {
#pragma unroll
  for (int i = 0; i < WideDim<D>::kLaneBytes / 4; ++i) wide_stage_pair<D, kF16Q>(r, i, kdst, vdst);
  *reinterpret_cast<float*>(sdst) = live_key ? r.s * smul : 0.0f;
}

template <bool kF16Q>
__device__ __forceinline__ f32x16 wide_qk(const u32x4& k, const u32x4& q, f32x16 c) {
  if constexpr (kF16Q)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, k),
                                                  __builtin_bit_cast(f16x8, q), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, k),
                                                   __builtin_bit_cast(bf16x8, q), c, 0, 0, 0);
}

// A row with a non-finite fp16 query element gets a NaN one, so that all its
// scores are NaN, as in the unit kernels (their hi + lo pair of an infinity is
// inf, NaN): an infinity alone would give keys with a negative byte there the
// score -inf, and drop them.
template <int N>
__device__ __forceinline__ void query_non_finite(u32x4 (&q)[N]) {
  uint32_t any = 0;  // bit 15 of a half: the sum of a half with an exponent of all ones
#pragma unroll
  for (int j = 0; j < N; ++j)
#pragma unroll
    for (int w = 0; w < 4; ++w) any |= (q[j][w] & 0x7fff7fffu) + 0x04000400u;
  if (any & 0x80008000u) q[0][0] |= 0x7fff7fffu;
}

// Column l % 32 of four consecutive keys of a row-major bf16 V (see above).
__device__ __forceinline__ bf16x4 v_column(const char* a) {
  return __builtin_bit_cast(
      bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                 (i16x4 __attribute__((address_space(3)))*)(const_cast<char*>(a))));
}

// V operand of output tile j and sub-product s: 32 columns of 16 keys, from
// the V buffer whose lane address is `v`.
template <int D>
__device__ __forceinline__ bf16x8 v_operand(const char* v, int s, int j) {
  constexpr int kVRow = WideDim<D>::kVRow;
  const bf16x4 x = v_column(v + (16 * s) * kVRow + 64 * j);
  const bf16x4 y = v_column(v + (16 * s + 8) * kVRow + 64 * j);
  return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Online-softmax state of a lane's row (the two lanes of a row hold the same
// m and thr, and each its own part of l).
template <int D>
struct WideState {
  f32x16 o[WideDim<D>::kO];
  bf16x8 ph[WideDim<D>::kSub], pl[WideDim<D>::kSub];  // P of the previous step
  float m;    // reference max (log2 units, a whole number); 0 before the first key
  float thr;  // the row's m moves when a score minus m exceeds this (rescale_threshold)
  float l;
};

// O *= alpha. With one wave per SIMD, O lives in accumulation registers, which
// the vector unit cannot use: said in the operand constraints, since
// otherwise the compiler moves all of O to vector registers at the top of
// every step, for this rare branch. (The products that wrote O were issued
// before the Q K products whose scores are known here.)
template <int D>
__device__ __forceinline__ void wide_scale_o(WideState<D>& st, float alpha) {
  if constexpr (WideDim<D>::kPerSimd == 1) {
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int j = 0; j < WideDim<D>::kO; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float x = st.o[j][i], tmp;
        asm volatile(
            "v_accvgpr_read_b32 %1, %0\n\t"
            "s_nop 1\n\t"
            "v_mul_f32 %1, %1, %2\n\t"
            "s_nop 1\n\t"
            "v_accvgpr_write_b32 %0, %1"
            : "+a"(x), "=&v"(tmp)
            : "v"(alpha));
        st.o[j][i] = x;
      }
    asm volatile("s_nop 15" ::: "memory");
  } else {
#pragma unroll
    for (int j = 0; j < WideDim<D>::kO; ++j) st.o[j] *= alpha;
  }
}

// P *= alpha, a power of two: exact.
__device__ __forceinline__ bf16x8 scale_p(bf16x8 p, float alpha) {
  const u32x4 w = __builtin_bit_cast(u32x4, p);
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = __builtin_bit_cast(float, w[i] << 16) * alpha;
    const float b = __builtin_bit_cast(float, w[i] & 0xffff0000u) * alpha;
    r[i] = __builtin_bit_cast(uint32_t, pack_bf16(a, b));
  }
  return __builtin_bit_cast(bf16x8, r);
}

template <int D>
__device__ __forceinline__ void wide_grow(WideState<D>& st, float lane_mx, float& shift) {
  const SwapPair sw = swap_halves(lane_mx);
  const float mx = max_raw(sw.a, sw.b);
  const bool grow = mx > st.thr;
  shift = grow ? ceilf(mx) : 0.0f;
  // A row's first visible key: nothing accumulated, any factor.
  const float alpha =
      grow && st.thr == kRescaleSlack ? __builtin_amdgcn_exp2f(-shift) : 1.0f;
  st.l *= alpha;
  wide_scale_o(st, alpha);
#pragma unroll
  for (int s = 0; s < WideDim<D>::kSub; ++s) {
    st.ph[s] = scale_p(st.ph[s], alpha);
    st.pl[s] = scale_p(st.pl[s], alpha);
  }
  st.m += shift;
  st.thr = grow ? kRescaleSlack : st.thr;
}

// v_mul_legacy_f32 (no builtin): a product in which 0 times anything is 0. The p
// of a masked key is 0, and its V scale may be any bits, also infinite or NaN.
extern "C" __device__ float mul_legacy(float a, float b) __asm("llvm.amdgcn.fmul.legacy");

// Two P V weights -> bf16 hi + lo. x - hi is exact, and one instruction: a dot
// product with a pair that picks the element. The pairs are kept in registers:
// as a constant, {-1, 0} becomes the instruction's inline -1.0, whose bits are
// those of the fp32 value, {0, -1}.
struct Picks {
  uint32_t first = 0x0000bf80u, second = 0xbf800000u;  // bf16 {-1, 0}, {0, -1}
  __device__ __forceinline__ void keep() { asm volatile("" : "+s"(first), "+s"(second)); }
};
struct PPair {
  bf16x2 hi, lo;
};
__device__ __forceinline__ PPair p_pair(const Picks& k, float x, float y) {
  PPair r;
  r.hi = pack_bf16(x, y);
  r.lo = pack_bf16(
      __builtin_amdgcn_fdot2_f32_bf16(r.hi, __builtin_bit_cast(bf16x2, k.first), x, false),
      __builtin_amdgcn_fdot2_f32_bf16(r.hi, __builtin_bit_cast(bf16x2, k.second), y, false));
  return r;
}

// O += P V of 16 keys: sub-product s of the step whose V rows are at `v`
// (the lane's address).
template <int D>
__device__ __forceinline__ void wide_pv(WideState<D>& st, const char* v, int s) {
  constexpr int kO = WideDim<D>::kO;
  bf16x8 a[kO];
#pragma unroll
  for (int j = 0; j < kO; ++j) a[j] = v_operand<D>(v, s, j);
#pragma unroll
  for (int j = 0; j < kO; ++j)
    st.o[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[j], st.ph[s], st.o[j], 0, 0, 0);
#pragma unroll
  for (int j = 0; j < kO; ++j)
    st.o[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[j], st.pl[s], st.o[j], 0, 0, 0);
}

// Stores of a finished segment: out, or the split's partial.
template <int D>
__device__ __forceinline__ void wide_store(const AttnParams& p, const Segment& g,
                                           const WideLanes& L, const WideState<D>& st, int lane) {
  constexpr int kO = WideDim<D>::kO;
  const int h = lane >> 5;
  const SwapPair ls = swap_halves(st.l);
  const float l_tot = ls.a + ls.b;
  const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
  const float lse2 = l_tot > 0.0f ? st.m + __builtin_amdgcn_logf(l_tot) : kNegInf;
  const int64_t head = L.head;
  if (writes_marker(p, g.s, g.live) && L.vrow) {
    char* lse_row = reinterpret_cast<char*>(p.ws_lse) + L.qtok * p.s_wl_tok + head * p.s_wl_head;
    *reinterpret_cast<uint32_t*>(lse_row + static_cast<int64_t>(p.num_splits - 1) * p.s_wl_split) =
        kSplitMarker | static_cast<uint32_t>(g.live);
  }
  const bool part = !direct_out(p, g.live);
  if (part || p.out_dtype == PTH_ATTN_F32) {
    if (!L.vrow) return;
    char* dst = part ? reinterpret_cast<char*>(p.ws_o) + g.s * p.s_wo_split + L.qtok * p.s_wo_tok +
                           head * p.s_wo_head
                     : p.out + L.qtok * p.s_out_tok + head * p.s_out_head;
#pragma unroll
    for (int j = 0; j < kO; ++j)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        *reinterpret_cast<f32x4*>(dst + 4 * (32 * j + 8 * b + 4 * h)) =
            (f32x4){st.o[j][4 * b] * inv, st.o[j][4 * b + 1] * inv, st.o[j][4 * b + 2] * inv,
                    st.o[j][4 * b + 3] * inv};
    if (part) {
      char* lse_row = reinterpret_cast<char*>(p.ws_lse) + L.qtok * p.s_wl_tok + head * p.s_wl_head;
      *reinterpret_cast<float*>(lse_row + g.s * p.s_wl_split) = lse2;
      return;
    }
  } else {
    // The two lanes of a row hold columns 8 b + 4 h ..: swapping halves
    // between b and b + 1 gives each lane 8 consecutive columns, 16 bytes.
    char* dst = p.out + L.qtok * p.s_out_tok + head * p.s_out_head;
    const bool bf = p.out_dtype == PTH_ATTN_BF16;
#pragma unroll
    for (int j = 0; j < kO; ++j)
#pragma unroll
      for (int b = 0; b < 4; b += 2) {
        uint32_t x[2], y[2];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          const float x0 = st.o[j][4 * b + 2 * w] * inv, x1 = st.o[j][4 * b + 2 * w + 1] * inv;
          const float y0 = st.o[j][4 * b + 4 + 2 * w] * inv,
                      y1 = st.o[j][4 * b + 5 + 2 * w] * inv;
          const uint32_t xb = __builtin_bit_cast(uint32_t, pack_bf16(x0, x1));
          const uint32_t yb = __builtin_bit_cast(uint32_t, pack_bf16(y0, y1));
          const uint32_t xh = __builtin_bit_cast(
              uint32_t, (f16x2){static_cast<_Float16>(x0), static_cast<_Float16>(x1)});
          const uint32_t yh = __builtin_bit_cast(
              uint32_t, (f16x2){static_cast<_Float16>(y0), static_cast<_Float16>(y1)});
          auto sw = __builtin_amdgcn_permlane32_swap(bf ? xb : xh, bf ? yb : yh, false, false);
          const uint32_t s0 = sw[0], s1 = sw[1];
          x[w] = s0;
          y[w] = s1;
        }
        if (L.vrow)
          *reinterpret_cast<u32x4*>(dst + 2 * (32 * j + 8 * b + 8 * h)) =
              (u32x4){x[0], x[1], y[0], y[1]};
      }
    if (!L.vrow) return;
  }
  if (p.lse_out != nullptr) {
    float* lo_ptr = reinterpret_cast<float*>(reinterpret_cast<char*>(p.lse_out) +
                                             L.qtok * p.s_lo_tok + head * p.s_lo_head);
    *lo_ptr = lse2 * 0.69314718055994530942f;
  }
}

template <int D, bool kWindow, bool kStream, bool kF16Q>
__global__ __launch_bounds__(WideDim<D>::kThreads)
    __attribute__((amdgpu_waves_per_eu(WideDim<D>::kPerSimd, WideDim<D>::kPerSimd)))
void attn_fwd_wide(const AttnParams p) {
  using W = WideDim<D>;
  __shared__ __attribute__((aligned(16))) char lds[W::kLds];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5;

  // The first step of a segment multiplies its zero P with the V buffer
  // "before" it: finite bytes, zero until a step has written the buffer.
  for (int i = static_cast<int>(threadIdx.x) * 16; i < 3 * W::kVBuf; i += W::kThreads * 16)
    *reinterpret_cast<u32x4*>(lds + W::kVBase + i) = (u32x4){0u, 0u, 0u, 0u};

  const int key8 = 8 * wave + (lane >> 3);  // the lane's key of a step
  char* const k_dst = lds + key8 * W::kKRow + (lane & 7) * (2 * W::kLaneBytes);
  char* const v_dst = lds + W::kVBase + key8 * W::kVRow + (lane & 7) * (2 * W::kLaneBytes);
  const int s_key = 8 * wave + (lane & 7);  // the lane's scale
  char* const s_dst = lds + W::kSBase + ((lane & 8) ? 4 * W::kStep : 0) + 4 * s_key;
  const float smul = (lane & 8) ? 1.0f : p.scale_log2;
  const char* const k_src = lds + (lane & 31) * W::kKRow + 16 * h;
  const char* const v_src = lds + W::kVBase + (4 * h + ((lane & 15) >> 2)) * W::kVRow +
                            32 * ((lane >> 4) & 1) + 8 * (lane & 3);
  const char* const s_src = lds + W::kSBase + 16 * h;

  Picks picks;
  picks.keep();
  WideWalk<kWindow, kStream> walk;
  walk.init(p, lane);
  Segment g;
  while (walk.next(p, lane, g)) {
    const int row0 = kWideRows * wave;
    const bool has_rows = row0 < g.t.num_tok * p.group;
    const WideLanes L = wide_lanes<kWindow>(p, g, row0, lane);
    const WideBounds wb = wide_bounds<kWindow>(p, g, has_rows ? row0 : 0, kWideRows);
    WideState<D> st;
#pragma unroll
    for (int j = 0; j < W::kO; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) st.o[j][e] = 0.0f;
#pragma unroll
    for (int s = 0; s < W::kSub; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) st.ph[s][e] = st.pl[s][e] = static_cast<__bf16>(0.0f);
    st.m = 0.0f;
    st.thr = rescale_threshold(true);
    st.l = 0.0f;

    const int c0 = g.lo & ~15;
    const int n = g.hi > c0 ? (g.hi - c0 + W::kStep - 1) / W::kStep : 0;
    if (n > 0) {
      const int last16 = (g.hi - 1) & ~15;
      PageWindow pw;
      pw.row = p.block_table + static_cast<int64_t>(g.t.req) * p.bt_stride;
      pw.win = static_cast<int>(p.bs_div.div(static_cast<uint32_t>(c0)));
      pw.last = static_cast<int>(p.bs_div.div(static_cast<uint32_t>(g.hi - 1)));
      pw.cur = window_load(pw, pw.win, lane);
      pw.nxt = window_load(pw, pw.win + 64, lane);
      u32x4 q[W::kQ];
      {
        const char* qrow = p.q + L.qtok * p.s_q_tok + static_cast<int64_t>(L.head) * p.s_q_head;
#pragma unroll
        for (int j = 0; j < W::kQ; ++j) {
          q[j] = *reinterpret_cast<const u32x4*>(qrow + 32 * j + 16 * h);
          if (!L.vrow) q[j] = (u32x4){0u, 0u, 0u, 0u};
        }
        if constexpr (kF16Q) query_non_finite(q);
      }
      WideOffsets wo;
      const uint32_t cell_head = static_cast<uint32_t>(g.kvh) * p.cell_head;
      wo.kv = (8u * (wave & 1) + (lane >> 3)) * p.cell_slot + cell_head +
              (lane & 7) * static_cast<uint32_t>(W::kLaneBytes);
      wo.s = (8u * (wave & 1) + (lane & 7)) * p.cell_slot + cell_head +
             ((lane & 8) ? p.cell_off[3] : p.cell_off[2]);
      WideRaw<D> raw;
      wide_load<D>(p, pw, wo, key_group(p, c0, wave, last16), raw);
      __syncthreads();  // the previous segment's reads of the buffers are done
      wide_stage<D, kF16Q>(raw, k_dst, v_dst, s_dst,
                           c0 + s_key >= g.lo && c0 + s_key < g.hi, smul);
      wide_load<D>(p, pw, wo, key_group(p, c0 + W::kStep, wave, last16), raw);
      int kb = 0, vb = 0, vprev = 2 * W::kVBuf;  // LDS offsets of K(k), V(k), V(k - 1)
      int sb = 0;
      // A wave without rows (a short block) only stages its share.
      for (int k = has_rows ? n : 0; k < n; ++k) {
        const int c = c0 + W::kStep * k;
        __syncthreads();
        const KeyGroup kg = key_group(p, c + 2 * W::kStep, wave, last16);
        page_window(pw, kg.blk, lane);
        kb = W::kKBuf - kb;
        sb = W::kSBuf - sb;
        vb = vb == 2 * W::kVBuf ? 0 : vb + W::kVBuf;
        wide_stage<D, kF16Q>(raw, k_dst + kb, v_dst + vb, s_dst + sb, c + W::kStep + s_key < g.hi,
                             smul);
        wide_load<D>(p, pw, wo, kg, raw);
      }
      for (int k = has_rows ? 0 : n; k < n; ++k) {
        const int c = c0 + W::kStep * k;
        const int kn = W::kKBuf - kb, sn = W::kSBuf - sb;
        const int vn = vb == 2 * W::kVBuf ? 0 : vb + W::kVBuf;
        // K(k), V(k) and the scales are complete in LDS; every wave is done
        // with K(k - 1) and V(k - 2), whose buffers step k + 1 takes.
        __syncthreads();
        const KeyGroup kg = key_group(p, c + 2 * W::kStep, wave, last16);  // of step k + 2
        page_window(pw, kg.blk, lane);
        // K Q^T: operands read kAhead ahead of their use, the tiles in turn,
        // and step k + 1 converted into the other buffers between the
        // products. The scheduling barriers keep this order: the compiler's
        // own puts each read right before its product and waits for it.
        constexpr int kProducts = W::kTiles * W::kQ;
        constexpr int kAhead = W::kAhead;
        auto k_read = [&](int i) {
          return *reinterpret_cast<const u32x4*>(k_src + kb + 32 * (i % W::kTiles) * W::kKRow +
                                                 32 * (i / W::kTiles));
        };
        const bool live_key = c + W::kStep + s_key < g.hi;
        f32x16 acc[W::kTiles];
#pragma unroll
        for (int t = 0; t < W::kTiles; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[t][e] = 0.0f;
        u32x4 kk[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) kk[i] = k_read(i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kProducts; ++i) {
          acc[i % W::kTiles] = wide_qk<kF16Q>(kk[i % kAhead], q[i / W::kTiles], acc[i % W::kTiles]);
          if (i + kAhead < kProducts) kk[i % kAhead] = k_read(i + kAhead);
          constexpr int kPairs = W::kLaneBytes / 4;  // word pairs of K and V together
          constexpr int kEvery = kProducts / kPairs;
          if (i % kEvery == kEvery - 1)
            wide_stage_pair<D, kF16Q>(raw, i / kEvery, k_dst + kn, v_dst + vn);
          if (i == kProducts - 1)
            *reinterpret_cast<float*>(s_dst + sn) = live_key ? raw.s * smul : 0.0f;
          __builtin_amdgcn_sched_barrier(0);
        }
        wide_load<D>(p, pw, wo, kg, raw);
        // Scores minus m, masked.
        float t[W::kTiles][16];
#pragma unroll
        for (int tt = 0; tt < W::kTiles; ++tt)
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const f32x4 ks = *reinterpret_cast<const f32x4*>(s_src + sb + 128 * tt + 32 * b);
#pragma unroll
            for (int e = 0; e < 4; ++e)
              t[tt][4 * b + e] = fmaf(acc[tt][4 * b + e], ks[e], -st.m);
          }
        if (c < wb.lo_max || c + W::kStep - 1 > wb.hi_min) {
#pragma unroll
          for (int tt = 0; tt < W::kTiles; ++tt)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const int key = c + 32 * tt + 8 * (e >> 2) + 4 * h + (e & 3);
              if (key < L.lo || key > L.hi) t[tt][e] = kNegInf;
            }
        }
        float mx;
        {
          float a[4 * W::kTiles];
#pragma unroll
          for (int tt = 0; tt < W::kTiles; ++tt)
#pragma unroll
            for (int b = 0; b < 4; ++b)
              a[4 * tt + b] = max_raw(max3_raw(t[tt][4 * b], t[tt][4 * b + 1], t[tt][4 * b + 2]),
                                      t[tt][4 * b + 3]);
          mx = max_raw(max3_raw(a[0], a[1], a[2]), a[3]);
          if constexpr (W::kTiles == 2)
            mx = max3_raw(mx, max_raw(a[4], a[5]), max_raw(a[6], a[7]));
        }
        if (__ballot(mx > st.thr) != 0) {
          float shift;
          wide_grow<D>(st, mx, shift);
#pragma unroll
          for (int tt = 0; tt < W::kTiles; ++tt)
#pragma unroll
            for (int e = 0; e < 16; ++e) t[tt][e] -= shift;
        }
        // softmax(k), 8 scores per lane at a time, beside P(k - 1) V(k - 1). The
        // step's p are summed before l takes them: added to l one by one, a long
        // tail of small p would be rounded to l's last place each time.
        float l_step = 0.0f;
#pragma unroll
        for (int s = 0; s < W::kSub; ++s) {
          wide_pv<D>(st, v_src + vprev, s);
          bf16x8 ph, pl;
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            const f32x4 vs =
                *reinterpret_cast<const f32x4*>(s_src + sb + 4 * W::kStep + 64 * s + 32 * b);
            float pv[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float pe = __builtin_amdgcn_exp2f(t[s >> 1][8 * (s & 1) + 4 * b + e]);
              l_step = s + b + e == 0 ? pe : l_step + pe;
              pv[e] = mul_legacy(pe, vs[e]);
            }
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
              const PPair pp = p_pair(picks, pv[e], pv[e + 1]);
              ph[4 * b + e] = pp.hi[0];
              ph[4 * b + e + 1] = pp.hi[1];
              pl[4 * b + e] = pp.lo[0];
              pl[4 * b + e + 1] = pp.lo[1];
            }
          }
          st.ph[s] = ph;
          st.pl[s] = pl;
        }
        st.l += l_step;
        kb = kn;
        sb = sn;
        vprev = vb;
        vb = vn;
      }
      if (has_rows) {  // the last step's P V
#pragma unroll
        for (int s = 0; s < W::kSub; ++s) wide_pv<D>(st, v_src + vprev, s);
      }
    }
    if (has_rows) wide_store<D>(p, g, L, st, lane);
  }
}

template <int D, bool kWindow, bool kStream>
hipError_t launch_wide(const AttnParams& p, dim3 grid, bool q_f16, hipStream_t stream) {
  const dim3 block(WideDim<D>::kThreads);
  if (q_f16)
    hipLaunchKernelGGL((attn_fwd_wide<D, kWindow, kStream, true>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((attn_fwd_wide<D, kWindow, kStream, false>), grid, block, 0, stream, p);
  return hipGetLastError();
}

}  // namespace

int32_t wide_block_tokens(int32_t head_size, int32_t group) {
  const int32_t rows = head_size == 256 ? WideDim<256>::kBlock : WideDim<128>::kBlock;
  return rows / group;
}

hipError_t launch_wide_kernel(const AttnParams& p, dim3 grid, bool windowed, bool q_f16,
                              int head_size, hipStream_t stream) {
  const bool split = p.num_splits > 1;
  note_kernel("attn_fwd_wide");
  if (head_size == 64)
    return split ? launch_wide<64, false, true>(p, grid, q_f16, stream)
                 : launch_wide<64, false, false>(p, grid, q_f16, stream);
  if (head_size == 256)
    return split ? launch_wide<256, false, true>(p, grid, q_f16, stream)
                 : launch_wide<256, false, false>(p, grid, q_f16, stream);
  if (!split) return hipErrorInvalidValue;  // the row-block kernel's launches
  return windowed ? launch_wide<128, true, true>(p, grid, q_f16, stream)
                  : launch_wide<128, false, true>(p, grid, q_f16, stream);
}

}  // namespace pa
