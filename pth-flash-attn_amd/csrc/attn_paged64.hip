// attn_paged64.hip -- the unit kernels at head size D = 64 on paged cell caches
// (block size a multiple of 16): decode and verify launches. Same work
// decomposition, MFMA layout and numerics as attn_fwd.hip at D = 64
// (HeadDim<64>); what differs from attn_fwd_generic, which looks every key up
// in the block table on its own, is how keys reach the wave: 64 keys at a
// time, with the loads of the next 64 in flight while the wave computes two
// 32-key chunks out of LDS. A 64-key step of D = 64 has the bytes of a 32-key
// chunk of D = 128, which is what the D = 128 kernels keep in flight.
//
//  * attn_fwd_pagerows64 (the vLLM NHD cell of 8 KV heads, work-groups whose
//    8 waves are the 8 heads of the same keys): the work-group loads whole
//    slot rows (8 cells of 136 bytes), every cache line by one wave only, into
//    a shared double-buffered LDS step, one barrier per step (as
//    attn_fwd_pagerows);
//  * attn_fwd_staged64 (any other cell cache): each wave loads its own head's
//    rows into its own LDS slot (as attn_fwd_staged).
//
// Bound: HBM and issue together. Page rows, 48 requests of up to 16k keys
// (440 MB of cells, 32 query heads): 248 us by the register-load kernel, 95
// here with the combine (4.8 TB/s in the kernel; 109 if staged per wave,
// whose waves share cache lines); vector and matrix issue take 63% of the
// launch. A second set of staging registers (loads two steps ahead) measured
// 3 us more, so the loads are early enough. One request of 1k keys: 9.2 us by
// either kernel, start to end. Staged: the same requests with 4 KV heads 154
// -> 81, HND with 8 220 -> 93, four verify tokens against 128k keys of 4 heads
// 47 -> 28.

#include "attn_device.h"

namespace pa {
namespace {

constexpr int kStep64 = 64;          // keys per step
constexpr int kGroups64 = kStep64 / 16;

// Pages and first slots of a step's four 16-key groups (scalar loads of the
// block table; a group outside the unit's keys reads page 0 and is masked).
struct StepPages {
  int32_t page[kGroups64], slot0[kGroups64];
};

__device__ __forceinline__ StepPages step_pages(const AttnParams& p, const Unit& U, int c) {
  const int64_t bt0 = static_cast<int64_t>(U.t.req) * p.bt_stride;
  c = __builtin_amdgcn_readfirstlane(c);
  StepPages sp;
#pragma unroll
  for (int i = 0; i < kGroups64; ++i) {
    const int c16 = c + 16 * i;
    sp.page[i] = 0;
    sp.slot0[i] = 0;
    if (c16 < U.ld_hi && c16 + 16 > U.ld_lo) {
      const int blk = static_cast<int>(p.bs_div.div(c16));
      sp.slot0[i] = c16 - blk * static_cast<int>(p.bs_div.d);
      sp.page[i] = ld_ro(p.block_table, bt0 + blk);
    }
  }
  return sp;
}

__device__ __forceinline__ void step_bases(const AttnParams& p, const StepPages& sp,
                                           const char* (&base)[kGroups64]) {
#pragma unroll
  for (int i = 0; i < kGroups64; ++i)
    base[i] = p.cell_base +
              static_cast<uint64_t>(static_cast<uint32_t>(sp.page[i])) * p.cell_block +
              static_cast<uint32_t>(sp.slot0[i]) * p.cell_slot;
}

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Every field of a unit is wave-uniform: said, so that they stay scalar.
__device__ __forceinline__ void make_uniform(Unit& U) {
  U.t.req = uni(U.t.req);
  U.t.tok_begin = uni(U.t.tok_begin);
  U.t.num_tok = uni(U.t.num_tok);
  U.t.q_len = uni(U.t.q_len);
  U.t.seq_len = uni(U.t.seq_len);
  U.t.q_start = uni(U.t.q_start);
  U.s = uni(U.s);
  U.live = uni(U.live);
  U.kvh = uni(U.kvh);
  U.rg = uni(U.rg);
  U.rows = uni(U.rows);
  U.row0 = uni(U.row0);
  U.has_rows = uni(U.has_rows ? 1 : 0) != 0;
  U.ld_lo = uni(U.ld_lo);
  U.ld_hi = uni(U.ld_hi);
  U.c_begin = uni(U.c_begin);
  U.n_chunks = uni(U.n_chunks);
  U.w_lo_max = uni(U.w_lo_max);
  U.w_hi_min = uni(U.w_hi_min);
}

template <bool kStream>
__device__ __forceinline__ bool next_live_unit(const AttnParams& p, Work<false, kStream>& work,
                                               int lane, Unit& U, Lanes& L) {
  while (work.next(p, lane, U)) {
    make_uniform(U);
    if (!U.has_rows) continue;
    L = unit_lanes<false>(p, U, lane);
    if (U.n_chunks == 0) {  // no key of these rows in this split
      StateT<64> empty;
      state_reset(empty);
      epilogue(p, U, L, empty);
      continue;
    }
    return true;
  }
  return false;
}

// The operands of a 32-key chunk in registers (the layout of HeadDim<64>):
// K bytes [16 g, 16 g + 16) of keys r and 16 + r, V bytes [4 r, 4 r + 4) of
// keys tv(e), one scale.
struct Chunk64 {
  u32x4 k[2];
  uint32_t v[8];
  float s;
};

struct Chunk64Ops {
  const Chunk64& ch;
  __device__ __forceinline__ float sc() const { return ch.s; }
  __device__ __forceinline__ bf16x8 k(int sub, int j) const {
    return j == 0 ? i8x8_to_bf16(ch.k[sub][0], ch.k[sub][1])
                  : i8x8_to_bf16(ch.k[sub][2], ch.k[sub][3]);
  }
  __device__ __forceinline__ bf16x8 v(int j) const {
    bf16x2 pr[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      pr[e] = pack_bf16(i8_to_f32(ch.v[2 * e], j), i8_to_f32(ch.v[2 * e + 1], j));
    return (bf16x8){pr[0][0], pr[0][1], pr[1][0], pr[1][1], pr[2][0], pr[2][1], pr[3][0], pr[3][1]};
  }
};

// ---------------------------------------------------------------------------
// Page rows: a slot row is the 8 heads' 136-byte cells, 1088 contiguous
// bytes. The work-group's 512 lanes split a step's 4,352 16-byte pieces:
// pieces L + 512 j, and the last 256 of them to the first 256 lanes. Rows are
// padded to kRowPad64 bytes in LDS: 16 keys' K pieces (8-byte reads, stride 20
// banks) and the V words of keys 4 apart (stride 16 banks) then touch
// distinct banks.
constexpr int kRow64 = 1088;
constexpr int kRowPad64 = kRow64 + 16;
constexpr int kRowPieces64 = kRow64 / 16;          // 68
constexpr int kGroupPieces64 = 16 * kRowPieces64;  // 1088
constexpr int kRowBuf64 = kStep64 * kRowPad64;
static_assert(kGroups64 * kGroupPieces64 == 8 * 512 + 256, "pieces of a step");

struct Row64Staged {
  u32x4 piece[9];
};

// Group of piece i: constant over a lane's piece j but where a group ends
// within the 512 pieces.
__device__ __forceinline__ int piece_group(int i) {
  return (i >= kGroupPieces64 ? 1 : 0) + (i >= 2 * kGroupPieces64 ? 1 : 0) +
         (i >= 3 * kGroupPieces64 ? 1 : 0);
}

// Non-temporal: every line is fetched by one wave and never again in the
// launch (see attn_fwd_pagerows).
__device__ __forceinline__ void rows64_load(const AttnParams& p, const StepPages& sp, int L,
                                            Row64Staged& S) {
  const char* base[kGroups64];
  step_bases(p, sp, base);
#pragma unroll
  for (int j = 0; j < 9; ++j) {
    const int i = L + 512 * j;
    const int lo = piece_group(512 * j), hi = piece_group(512 * j + 511);
    const char* b = lo == hi || i < hi * kGroupPieces64 ? base[lo] : base[hi];
    const int w = i - piece_group(i) * kGroupPieces64;
    if (j < 8 || L < 256) S.piece[j] = ld_nt<u32x4>(b + 16 * w);
  }
}

__device__ __forceinline__ void rows64_write(char* buf, int L, const Row64Staged& S) {
#pragma unroll
  for (int j = 0; j < 9; ++j) {
    const int i = L + 512 * j;  // key i / 68 of the step (groups are whole rows)
    const int key = i / kRowPieces64;
    if (j < 8 || L < 256)
      *reinterpret_cast<u32x4*>(buf + key * kRowPad64 + 16 * (i - key * kRowPieces64)) = S.piece[j];
  }
}

// The wave's operands of the chunk whose rows start at `buf`, KV head `head`.
__device__ __forceinline__ void rows64_read(const char* buf, const AttnParams& p, int head,
                                            int lane, Chunk64& ch) {
  const int r16 = lane & 15, g = lane >> 4;
  const char* cell = buf + head * 136;
#pragma unroll
  for (int sub = 0; sub < 2; ++sub) {
    const char* kr = cell + (16 * sub + r16) * kRowPad64 + p.cell_off[0] + 16 * g;
    const u32x2_a4 a = *reinterpret_cast<const u32x2_a4*>(kr);
    const u32x2_a4 b = *reinterpret_cast<const u32x2_a4*>(kr + 8);
    ch.k[sub] = (u32x4){a[0], a[1], b[0], b[1]};
  }
#pragma unroll
  for (int e = 0; e < 8; ++e)
    ch.v[e] = *reinterpret_cast<const uint32_t*>(
        cell + (16 * (e >> 2) + 4 * g + (e & 3)) * kRowPad64 + p.cell_off[1] + 4 * r16);
  const int e = r16 & 7;
  ch.s = *reinterpret_cast<const float*>(cell + (16 * (e >> 2) + 4 * g + (e & 3)) * kRowPad64 +
                                         (r16 < 8 ? p.cell_off[2] : p.cell_off[3]));
}

template <bool kStream, bool kF16Q>
__global__ __launch_bounds__(kFwdWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_fwd_pagerows64(const AttnParams p_arg) {
  __shared__ __attribute__((aligned(16))) char lds_rows[2 * kRowBuf64];
  const int lane = threadIdx.x & 63;
  const AttnParams p = params_in_registers(p_arg, lane);
  const int L = threadIdx.x;
  const float scl = scale_factor(lane & 15, p.scale_log2);
  Work<false, kStream> work;
  work.init(p, lane);
  Unit U;
  Lanes Ls;
  int it = 0;  // steps of the work-group (buffer parity)
  // Every wave of the work-group walks the same units (the 8 KV heads of the
  // same keys), so they all meet the same barriers.
  while (next_live_unit(p, work, lane, U, Ls)) {
    const int n = (U.n_chunks + 1) / 2;
    Row64Staged S;
    StepPages sp = step_pages(p, U, U.c_begin);
    rows64_load(p, sp, L, S);
    bf16x8 qb[HeadDim<64>::kQK], qlo[HeadDim<64>::kQK];
    load_q<kF16Q, 64>(p, Ls, qb, qlo);
    if (n > 1) sp = step_pages(p, U, U.c_begin + kStep64);
    StateT<64> st;
    state_reset(st);
    for (int k = 0; k < n; ++k, ++it) {
      char* buf = lds_rows + (it & 1) * kRowBuf64;
      // The buffer was last read two steps ago; every wave has passed the
      // barrier after that read.
      rows64_write(buf, L, S);
      if (k + 1 < n) {
        rows64_load(p, sp, L, S);
        if (k + 2 < n) sp = step_pages(p, U, U.c_begin + kStep64 * (k + 2));
      }
      __syncthreads();  // the step's rows are in the buffer
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (2 * k + h >= U.n_chunks) break;
        Chunk64 ch;
        rows64_read(buf + 32 * h * kRowPad64, p, U.kvh, lane, ch);
        compute_chunk_t<64, kF16Q>(U, Ls, U.c_begin + kStep64 * k + 32 * h, Chunk64Ops{ch}, qb, qlo,
                                   scl, st);
      }
    }
    epilogue(p, U, Ls, st);
  }
}

// ---------------------------------------------------------------------------
// Per-wave staging: lane (t, c) = (lane / 4, lane % 4) loads 16-byte piece c of
// K and V of key t of each 16-key group (16 whole 64-byte rows per
// instruction) and the two scales of key `lane` of the step. In the wave's LDS
// slot, piece c of K row key is at c ^ (key / 4 % 4), so 16 keys' reads of one
// piece touch all banks; V rows have a row's gap after every four, so the
// words of keys 4 apart do.
constexpr int kSlot64V = kStep64 * 64;
constexpr int kSlot64S = kSlot64V + kStep64 * 80;
constexpr int kSlot64 = kSlot64S + kStep64 * 8;

struct Wave64Staged {
  u32x4 k[kGroups64], v[kGroups64];
  float ks, vs;
};

struct Wave64Offsets {
  uint32_t k, s;  // lane offsets of K piece c of key t, and of a key's K scale
};

__device__ __forceinline__ Wave64Offsets wave64_offsets(const AttnParams& p, int kvh, int lane) {
  const uint32_t head = static_cast<uint32_t>(kvh) * p.cell_head;
  Wave64Offsets o;
  o.k = static_cast<uint32_t>(lane >> 2) * p.cell_slot + head + 16u * (lane & 3) + p.cell_off[0];
  o.s = static_cast<uint32_t>(lane & 15) * p.cell_slot + head + p.cell_off[2];
  return o;
}

__device__ __forceinline__ void wave64_load(const AttnParams& p, const StepPages& sp,
                                            const Wave64Offsets& o, int lane, Wave64Staged& S) {
  const char* base[kGroups64];
  step_bases(p, sp, base);
  const int64_t kv = static_cast<int64_t>(p.cell_off[1]) - p.cell_off[0];  // K row -> V row
#pragma unroll
  for (int i = 0; i < kGroups64; ++i) {
    S.k[i] = *reinterpret_cast<const u32x4_a4*>(base[i] + o.k);
    S.v[i] = *reinterpret_cast<const u32x4_a4*>(base[i] + o.k + kv);
  }
  const char* lo = lane & 16 ? base[1] : base[0];
  const char* hi = lane & 16 ? base[3] : base[2];
  const char* sb = (lane & 32 ? hi : lo) + o.s;
  S.ks = *reinterpret_cast<const float*>(sb);
  S.vs = *reinterpret_cast<const float*>(sb + (static_cast<int64_t>(p.cell_off[3]) - p.cell_off[2]));
}

__device__ __forceinline__ void wave64_write(char* slot, int lane, const Wave64Staged& S) {
  const int t = lane >> 2, c = lane & 3;
#pragma unroll
  for (int i = 0; i < kGroups64; ++i) {
    const int key = 16 * i + t;
    *reinterpret_cast<u32x4*>(slot + 64 * key + 16 * (c ^ ((t >> 2) & 3))) = S.k[i];
    *reinterpret_cast<u32x4*>(slot + kSlot64V + 64 * (key + (key >> 2)) + 16 * c) = S.v[i];
  }
  *reinterpret_cast<float*>(slot + kSlot64S + 4 * lane) = S.ks;
  *reinterpret_cast<float*>(slot + kSlot64S + 4 * kStep64 + 4 * lane) = S.vs;
}

// Operands of chunk h (0, 1) of the step in the slot.
__device__ __forceinline__ void wave64_read(const char* slot, int h, int lane, Chunk64& ch) {
  const int r16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int sub = 0; sub < 2; ++sub)
    ch.k[sub] = *reinterpret_cast<const u32x4*>(slot + 64 * (32 * h + 16 * sub + r16) +
                                                16 * (g ^ (r16 >> 2)));
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int key = 32 * h + 16 * (e >> 2) + 4 * g + (e & 3);
    ch.v[e] =
        *reinterpret_cast<const uint32_t*>(slot + kSlot64V + 64 * (key + (key >> 2)) + 4 * r16);
  }
  const int e = r16 & 7;
  ch.s = *reinterpret_cast<const float*>(slot + kSlot64S + (r16 < 8 ? 0 : 4 * kStep64) +
                                         4 * (32 * h + 16 * (e >> 2) + 4 * g + (e & 3)));
}

template <bool kStream, bool kF16Q>
__global__ __launch_bounds__(kFwdWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_fwd_staged64(const AttnParams p_arg) {
  __shared__ __attribute__((aligned(16))) char lds_all[kFwdWaves * kSlot64];
  const int lane = threadIdx.x & 63;
  const AttnParams p = params_in_registers(p_arg, lane);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char* slot = lds_all + wave * kSlot64;
  const float scl = scale_factor(lane & 15, p.scale_log2);
  Work<false, kStream> work;
  work.init(p, lane);
  Unit U;
  Lanes L;
  while (next_live_unit(p, work, lane, U, L)) {
    const int n = (U.n_chunks + 1) / 2;
    const Wave64Offsets o = wave64_offsets(p, U.kvh, lane);
    Wave64Staged S;
    StepPages sp = step_pages(p, U, U.c_begin);
    wave64_load(p, sp, o, lane, S);
    bf16x8 qb[HeadDim<64>::kQK], qlo[HeadDim<64>::kQK];
    load_q<kF16Q, 64>(p, L, qb, qlo);
    if (n > 1) sp = step_pages(p, U, U.c_begin + kStep64);
    StateT<64> st;
    state_reset(st);
    for (int k = 0; k < n; ++k) {
      wave64_write(slot, lane, S);
      if (k + 1 < n) {
        wave64_load(p, sp, o, lane, S);
        if (k + 2 < n) sp = step_pages(p, U, U.c_begin + kStep64 * (k + 2));
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (2 * k + h >= U.n_chunks) break;
        Chunk64 ch;
        wave64_read(slot, h, lane, ch);
        compute_chunk_t<64, kF16Q>(U, L, U.c_begin + kStep64 * k + 32 * h, Chunk64Ops{ch}, qb, qlo,
                                   scl, st);
      }
    }
    epilogue(p, U, L, st);
  }
}

}  // namespace

hipError_t launch_paged64_kernel(const AttnParams& p, dim3 grid, bool q_f16, hipStream_t stream) {
  const bool st = p.num_splits > 1;
  note_kernel(p.page_rows ? "attn_fwd_pagerows64" : "attn_fwd_staged64");
  const dim3 block(kFwdWaves * 64);
#define PA_LAUNCH(K, St, F) hipLaunchKernelGGL((K<St, F>), grid, block, 0, stream, p)
  if (p.page_rows) {
    if (st && q_f16) PA_LAUNCH(attn_fwd_pagerows64, true, true);
    else if (st) PA_LAUNCH(attn_fwd_pagerows64, true, false);
    else if (q_f16) PA_LAUNCH(attn_fwd_pagerows64, false, true);
    else PA_LAUNCH(attn_fwd_pagerows64, false, false);
  } else {
    if (st && q_f16) PA_LAUNCH(attn_fwd_staged64, true, true);
    else if (st) PA_LAUNCH(attn_fwd_staged64, true, false);
    else if (q_f16) PA_LAUNCH(attn_fwd_staged64, false, true);
    else PA_LAUNCH(attn_fwd_staged64, false, false);
  }
#undef PA_LAUNCH
  return hipGetLastError();
}

}  // namespace pa
