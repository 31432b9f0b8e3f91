// attn_writer.hip -- the gfx950 int8 per-token-head cache writer: vLLM's
// reshape_and_cache for the int8_per_token_head cache (the reference relies
// on vLLM's Triton writer, mirrored by python/pth_testing/reference.py:76-103;
// no counterpart in the reference's ABI).
//
// The K row and the V row of D values of a (token, KV head) each get their
// fp32 absmax, scale = max(absmax / 127, 1e-6), inverse 1 / scale
// (both correctly rounded fp32 divisions), and q = trunc(clamp(x * inv +-
// 0.5, -128, 127)) with every step a separate fp32 operation (contraction
// off), so the bytes equal the writer's.
//
// Rows on 16-byte addresses, cells on 4-byte addresses, fewer than 2^31 slots
// and items: write_kv_int8_wide, D / 8 lanes per (token, head), each with one
// 16-byte load (two of fp32) and one 8-byte store of eight values a row, the
// absmax by lane moves within the row's lanes. Anything else: write_kv_int8,
// one wave per (token, head), lane l with the D / 64 values from l D / 64 on.
//
// Bound: HBM. 8,192 tokens of 8 heads of 128 in bf16 (51 MB, 11 us at the rate
// of a copy): 34 us by the narrow kernel, whose loads and stores were 4 and 2
// bytes a lane and whose maxima were six LDS round trips; 11.6 here (4.4 TB/s).

#include <hip/hip_runtime.h>

#include <cmath>
#include <string>

#include "attn_stream.h"

namespace pa {
namespace {

struct WriteParams {
  const char* key;
  const char* value;
  int64_t s_k_tok, s_k_head, s_v_tok, s_v_head;
  int32_t kv_dtype;
  int32_t num_tokens;
  int32_t num_kv_heads;
  const int64_t* slot_mapping;
  CacheStream k, v, ks, vs;
  int32_t block_size;
  int64_t num_slots;  // num_blocks * block_size
  Div32 bs_div, heads_div;  // of the wide kernel
};

__device__ __forceinline__ float load_elem(const char* p, int32_t dtype) {
  if (dtype == PTH_ATTN_F32) return *reinterpret_cast<const float*>(p);
  if (dtype == PTH_ATTN_F16) return static_cast<float>(*reinterpret_cast<const _Float16*>(p));
  return static_cast<float>(*reinterpret_cast<const __bf16*>(p));
}

__device__ __forceinline__ float wave_absmax(float x) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) x = fmaxf(x, __shfl_xor(x, d));
  return x;
}

// One row of D values (lane's NC at x) -> int8 at dst, scale at sdst.
template <int NC>
__device__ __forceinline__ void quantize_row(const float (&x)[NC], char* dst, float* sdst,
                                             int lane) {
#pragma clang fp contract(off)
  float a = 0.0f;
#pragma unroll
  for (int i = 0; i < NC; ++i) a = fmaxf(a, fabsf(x[i]));
  const float amax = wave_absmax(a);
  float s = amax / 127.0f;
  if (!(s >= 1e-6f)) s = 1e-6f;
  const float inv = 1.0f / s;
  int8_t q[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    float v = x[i] * inv;
    v = v >= 0.0f ? v + 0.5f : v - 0.5f;
    v = v < -128.0f ? -128.0f : v;
    v = v > 127.0f ? 127.0f : v;
    q[i] = static_cast<int8_t>(v);  // truncates toward zero
  }
#pragma unroll
  for (int i = 0; i < NC; ++i) dst[NC * lane + i] = static_cast<char>(q[i]);
  if (lane == 0) *sdst = s;
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x2 u32x2_a4 __attribute__((aligned(4)));

// Eight consecutive elements of a row.
template <int kType>
struct Eight {
  u32x4 w[kType == PTH_ATTN_F32 ? 2 : 1];
  __device__ __forceinline__ void load(const char* p) {
    w[0] = *reinterpret_cast<const u32x4*>(p);
    if constexpr (kType == PTH_ATTN_F32) w[1] = *reinterpret_cast<const u32x4*>(p + 16);
  }
  __device__ __forceinline__ float at(int i) const {
    if constexpr (kType == PTH_ATTN_F32) {
      const uint32_t x = w[i >> 2][i & 3];  // a value: a cast of the element reads element 0
      return __builtin_bit_cast(float, x);
    } else {
      const uint16_t h = static_cast<uint16_t>(w[0][i >> 1] >> (16 * (i & 1)));
      if constexpr (kType == PTH_ATTN_F16)
        return static_cast<float>(__builtin_bit_cast(_Float16, h));
      else return static_cast<float>(__builtin_bit_cast(__bf16, h));
    }
  }
};

// The lane's eight values of a row -> 8 bytes at dst, the row's scale at sdst.
template <int kLanes, int kType>
__device__ __forceinline__ void quantize_eight(const Eight<kType>& e, char* dst, float* sdst,
                                               bool first, bool live) {
#pragma clang fp contract(off)
  float x[8], a = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    x[i] = e.at(i);
    a = fmaxf(a, fabsf(x[i]));
  }
  const float amax = lanes_max<kLanes>(a);
  float s = amax / 127.0f;
  if (!(s >= 1e-6f)) s = 1e-6f;
  const float inv = 1.0f / s;
  u32x2 q = {0u, 0u};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float v = x[i] * inv;
    v = v >= 0.0f ? v + 0.5f : v - 0.5f;
    v = v < -128.0f ? -128.0f : v;
    v = v > 127.0f ? 127.0f : v;
    const int b = static_cast<int>(v);  // truncates toward zero; in [-128, 127]
    q[i >> 2] |= (static_cast<uint32_t>(b) & 0xffu) << (8 * (i & 3));
  }
  if (!live) return;
  *reinterpret_cast<u32x2_a4*>(dst) = q;
  if (first) *sdst = s;
}

template <int D, int kType>
__global__ __launch_bounds__(256) void write_kv_int8_wide(const WriteParams w) {
  constexpr int kLanes = D / 8;  // lanes per row
  constexpr int kElt = kType == PTH_ATTN_F32 ? 4 : 2;
  const uint32_t item = blockIdx.x * (256u / kLanes) + threadIdx.x / kLanes;
  const int l = threadIdx.x % kLanes;
  const uint32_t items =
      static_cast<uint32_t>(w.num_tokens) * static_cast<uint32_t>(w.num_kv_heads);
  if (item >= items) return;  // a row's lanes together
  const uint32_t tok = w.heads_div.div(item);
  const uint32_t head = item - tok * static_cast<uint32_t>(w.num_kv_heads);
  const int64_t slot = w.slot_mapping[tok];
  Eight<kType> k, v;
  k.load(w.key + static_cast<int64_t>(tok) * w.s_k_tok + static_cast<int64_t>(head) * w.s_k_head +
         8 * kElt * l);
  v.load(w.value + static_cast<int64_t>(tok) * w.s_v_tok + static_cast<int64_t>(head) * w.s_v_head +
         8 * kElt * l);
  const bool live = slot >= 0 && slot < w.num_slots;  // else a padding token
  const uint32_t at = live ? static_cast<uint32_t>(slot) : 0u;
  const uint32_t page = w.bs_div.div(at);
  const uint32_t in_page = at - page * static_cast<uint32_t>(w.block_size);
  auto cell = [&](const CacheStream& s) {
    return const_cast<char*>(s.base) + static_cast<int64_t>(page) * s.s_block +
           static_cast<int64_t>(in_page) * s.s_slot + static_cast<int64_t>(head) * s.s_head;
  };
  quantize_eight<kLanes, kType>(k, cell(w.k) + 8 * l, reinterpret_cast<float*>(cell(w.ks)),
                                l == 0, live);
  quantize_eight<kLanes, kType>(v, cell(w.v) + 8 * l, reinterpret_cast<float*>(cell(w.vs)),
                                l == 0, live);
}

template <int D>
__global__ __launch_bounds__(256) void write_kv_int8(const WriteParams w) {
  constexpr int NC = D / 64;
  const int lane = threadIdx.x & 63;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int64_t tok = item / w.num_kv_heads;
  const int head = static_cast<int>(item - tok * w.num_kv_heads);
  if (tok >= w.num_tokens) return;
  const int64_t slot = w.slot_mapping[tok];
  if (slot < 0 || slot >= w.num_slots) return;  // padding token (or out of the cache)
  const int64_t page = slot / w.block_size;
  const int64_t in_page = slot - page * w.block_size;
  float xk[NC], xv[NC];
  const int elt = w.kv_dtype == PTH_ATTN_F32 ? 4 : 2;
  const char* kr = w.key + tok * w.s_k_tok + static_cast<int64_t>(head) * w.s_k_head;
  const char* vr = w.value + tok * w.s_v_tok + static_cast<int64_t>(head) * w.s_v_head;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    xk[i] = load_elem(kr + static_cast<int64_t>(elt) * (NC * lane + i), w.kv_dtype);
    xv[i] = load_elem(vr + static_cast<int64_t>(elt) * (NC * lane + i), w.kv_dtype);
  }
  auto cell = [&](const CacheStream& s) {
    return const_cast<char*>(s.base) + page * s.s_block + in_page * s.s_slot +
           static_cast<int64_t>(head) * s.s_head;
  };
  quantize_row<NC>(xk, cell(w.k), reinterpret_cast<float*>(cell(w.ks)), lane);
  quantize_row<NC>(xv, cell(w.v), reinterpret_cast<float*>(cell(w.vs)), lane);
}

CacheStream stream_of(const PthAttnStream& s) {
  return CacheStream{static_cast<const char*>(s.data), s.stride_block, s.stride_slot,
                     s.stride_head};
}

}  // namespace

int32_t launch_write_kv(const PthAttnWriteArgs& a, hipStream_t stream) {
  clear_error();
  PA_REQUIRE(a.abi_version == PTH_ATTN_ABI_VERSION,
             "abi_version " + std::to_string(a.abi_version) + " != library ABI " +
                 std::to_string(PTH_ATTN_ABI_VERSION));
  PA_REQUIRE(a.struct_bytes == static_cast<int32_t>(sizeof(PthAttnWriteArgs)),
             "struct_bytes " + std::to_string(a.struct_bytes) + " != sizeof(PthAttnWriteArgs) " +
                 std::to_string(sizeof(PthAttnWriteArgs)));
  PA_REQUIRE(a.head_size == 64 || a.head_size == 128 || a.head_size == 256,
             "head_size must be 64, 128 or 256");
  PA_REQUIRE(a.kv_dtype == PTH_ATTN_F32 || a.kv_dtype == PTH_ATTN_F16 ||
                 a.kv_dtype == PTH_ATTN_BF16,
             "kv_dtype must be PTH_ATTN_F32, PTH_ATTN_F16 or PTH_ATTN_BF16");
  PA_REQUIRE(a.num_tokens >= 0 && a.num_kv_heads >= 1 && a.block_size >= 1 &&
                 a.num_blocks >= 1,
             "num_tokens >= 0, num_kv_heads, block_size and num_blocks >= 1");
  PA_REQUIRE(a.key && a.value && a.slot_mapping && a.k_cache.data && a.v_cache.data &&
                 a.k_scale.data && a.v_scale.data,
             "key, value, slot_mapping and the four cache streams must be non-NULL");
  const int64_t elt = a.kv_dtype == PTH_ATTN_F32 ? 4 : 2;
  PA_REQUIRE(reinterpret_cast<uintptr_t>(a.key) % elt == 0 &&
                 reinterpret_cast<uintptr_t>(a.value) % elt == 0 &&
                 a.key_stride_token % elt == 0 && a.key_stride_head % elt == 0 &&
                 a.value_stride_token % elt == 0 && a.value_stride_head % elt == 0,
             "key and value must be aligned to their element");
  PA_REQUIRE(reinterpret_cast<uintptr_t>(a.k_scale.data) % 4 == 0 &&
                 reinterpret_cast<uintptr_t>(a.v_scale.data) % 4 == 0 &&
                 a.k_scale.stride_slot % 4 == 0 && a.k_scale.stride_head % 4 == 0 &&
                 a.k_scale.stride_block % 4 == 0 && a.v_scale.stride_slot % 4 == 0 &&
                 a.v_scale.stride_head % 4 == 0 && a.v_scale.stride_block % 4 == 0,
             "the scale streams must be 4-B aligned");
  if (a.num_tokens == 0) return PTH_ATTN_OK;
  WriteParams w{};
  w.key = static_cast<const char*>(a.key);
  w.value = static_cast<const char*>(a.value);
  w.s_k_tok = a.key_stride_token;
  w.s_k_head = a.key_stride_head;
  w.s_v_tok = a.value_stride_token;
  w.s_v_head = a.value_stride_head;
  w.kv_dtype = a.kv_dtype;
  w.num_tokens = a.num_tokens;
  w.num_kv_heads = a.num_kv_heads;
  w.slot_mapping = a.slot_mapping;
  w.k = stream_of(a.k_cache);
  w.v = stream_of(a.v_cache);
  w.ks = stream_of(a.k_scale);
  w.vs = stream_of(a.v_scale);
  w.block_size = a.block_size;
  w.num_slots = static_cast<int64_t>(a.num_blocks) * a.block_size;
  const int64_t items = static_cast<int64_t>(a.num_tokens) * a.num_kv_heads;
  const auto rows16 = [](const void* p, int64_t tok, int64_t head) {
    return reinterpret_cast<uintptr_t>(p) % 16 == 0 && tok % 16 == 0 && head % 16 == 0;
  };
  const auto cells4 = [](const CacheStream& s) {
    return reinterpret_cast<uintptr_t>(s.base) % 4 == 0 && s.s_block % 4 == 0 &&
           s.s_slot % 4 == 0 && s.s_head % 4 == 0;
  };
  const bool wide = rows16(w.key, w.s_k_tok, w.s_k_head) &&
                    rows16(w.value, w.s_v_tok, w.s_v_head) && cells4(w.k) && cells4(w.v) &&
                    items < 0x7fffffff && w.num_slots < 0x7fffffff;
  if (wide) {
    w.bs_div = Div32::make(static_cast<uint32_t>(a.block_size));
    w.heads_div = Div32::make(static_cast<uint32_t>(a.num_kv_heads));
    const int per = 256 / (a.head_size / 8);  // items of a work-group
    const dim3 grid(static_cast<unsigned>((items + per - 1) / per)), block(256);
#define PA_WRITE(D, T) hipLaunchKernelGGL((write_kv_int8_wide<D, T>), grid, block, 0, stream, w)
#define PA_WRITE_D(D)                                          \
  do {                                                         \
    if (a.kv_dtype == PTH_ATTN_F32) PA_WRITE(D, PTH_ATTN_F32); \
    else if (a.kv_dtype == PTH_ATTN_F16) PA_WRITE(D, PTH_ATTN_F16); \
    else PA_WRITE(D, PTH_ATTN_BF16);                           \
  } while (0)
    switch (a.head_size) {
      case 64: PA_WRITE_D(64); break;
      case 256: PA_WRITE_D(256); break;
      default: PA_WRITE_D(128);
    }
#undef PA_WRITE_D
#undef PA_WRITE
  } else {
    const dim3 grid(static_cast<unsigned>((items + 3) / 4)), block(256);
    switch (a.head_size) {
      case 64: hipLaunchKernelGGL(write_kv_int8<64>, grid, block, 0, stream, w); break;
      case 256: hipLaunchKernelGGL(write_kv_int8<256>, grid, block, 0, stream, w); break;
      default: hipLaunchKernelGGL(write_kv_int8<128>, grid, block, 0, stream, w);
    }
  }
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess)
    return fail(PTH_ATTN_ECUDA, std::string("cache writer launch: ") + hipGetErrorString(err));
  return PTH_ATTN_OK;
}

}  // namespace pa

extern "C" {

int32_t pth_attn_write_args_bytes(void) {
  return static_cast<int32_t>(sizeof(PthAttnWriteArgs));
}

int32_t pth_attn_write_kv(const PthAttnWriteArgs* args, void* stream) {
  if (args == nullptr) return pa::fail(PTH_ATTN_EINVAL, "args is NULL");
  return pa::launch_write_kv(*args, static_cast<hipStream_t>(stream));
}

}  // extern "C"
