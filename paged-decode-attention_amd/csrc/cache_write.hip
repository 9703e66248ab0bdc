// Paged KV-cache write for MI355X (gfx950): this decode step's K and V rows
// scattered into the NHD pages at slot_mapping, quantised to the cache dtype.
//
// Replaces the KV write that precedes the decode in the reference's vLLM
// path (`reshape_and_cache_flash`, integration/vllm_backend.py:117-122) for
// caches in this library's formats, with the quantisation semantics of
// pagedattn/cache.py:33-48:
//   fp16      copy (bf16 rows into a bf16 cache: copy too)
//   fp8_e5m2  round-to-nearest-even of the fp16 bit pattern to its high byte
//             (e5m2 shares fp16's exponent); overflow rounds to inf and NaN
//             stays NaN, as torch's cast does
//   int8      amax over head_dim (clamped to 1e-6), scale = amax / 127 rounded
//             to the scale type, q = round_half_even(x / scale) clamped to
//             +-127. Bytes and scales are those of fp32 IEEE division, as
//             torch's: amax / 127 is a product corrected by its remainder,
//             x / scale a product with the reciprocal, and the division itself
//             in lanes where the two could round to different integers
//
// One (token, kv_head) row per D/8 lanes, 16 bytes (8 fp16) per lane; the
// int8 row maximum is a DPP reduction inside those lanes. A workgroup holds
// whole tokens (or, above 256 lanes a token, a 256-lane part of one), so a
// lane finds its token and head without an integer division; K, V and the
// slot are loaded together, before anything waits.
//
// What bounds it: HBM (read and write) for large writes, the launch and one
// round trip for a decode step's. The form with two 64-bit divisions a lane, K
// and V one after the other and ~15 VALU instructions per int8 element was
// bound by issue. The bytes go out with non-temporal stores (16,384 fp16 rows
// 28.9 us without); the rows come in with plain loads, since the projection
// that made them has just left them in a cache (non-temporal loads: 2-6% faster
// on rows from HBM, up to 8% slower on cached ones). Graph-timed at the
// Llama-3-8B shape (8 kv heads, head_dim 128), before -> after:
//   16,384 tokens: fp16 29.1 -> 25.0 us, fp8 25.2 -> 20.7, int8 with fp32
//     scales 32.1 -> 22.4 (4.6 TB/s; a large device copy runs at 4.7);
//   64 tokens: fp16 2.42 -> 2.29, fp8 3.20 -> 2.33, int8 3.89 -> 2.90 (an empty
//     kernel in a graph takes 1.6).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pa_errors.h"
#include "pagedattn.h"

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

struct WParams {
  const uint8_t *key;
  const uint8_t *value;
  uint8_t *kc;
  uint8_t *vc;
  uint8_t *ks;
  uint8_t *vs;
  const int64_t *slots;
  uint32_t tokens;
  uint32_t lanes;      // lanes of one token: num_kv_heads * head_dim / 8
  uint32_t tpb;        // tokens per group of 256 lanes (1 when a token takes several groups)
  uint32_t parts;      // groups per token (1 when a group holds whole tokens)
  uint32_t groups;     // all groups; workgroup i takes groups i, i + grid, ...
  uint32_t grid;       // workgroups (gridDim.x would be read from the hidden arguments, cold)
  uint32_t inv_lanes;  // ceil(2^16 / lanes): x / lanes = x * inv_lanes >> 16 for x < 256, lanes <= 256
  int32_t block_size;
  int32_t log2_block;  // -1: block_size is not a power of two
  int64_t max_slot;        // num_blocks * block_size
  int64_t skt, skh, svt, svh;  // bytes
  int64_t scn, sct, sch;       // bytes
  int64_t ssn, sst;            // bytes
};

// Index times stride, added to base: 32 x 32 -> 64 bits (one v_mad_u64_u32) or
// 64-bit throughout.
template <bool WIDE>
__device__ __forceinline__ uint64_t at(uint64_t base, uint64_t index, int64_t stride) {
  if constexpr (WIDE) return base + index * (uint64_t)stride;
  return base + (uint64_t)(uint32_t)index * (uint32_t)stride;
}

constexpr int64_t kMaxGrid = 1 << 14;  // workgroups of a launch; more groups than that loop

// fp16 bit pattern -> e5m2 byte, round to nearest even on the dropped byte.
__device__ __forceinline__ uint32_t half_to_e5m2(uint32_t h) {
  const uint32_t sign = (h >> 8) & 0x80u;
  const uint32_t mag = h & 0x7fffu;
  if (mag > 0x7c00u) return sign | 0x7fu;  // NaN
  return sign | ((mag + 0x7fu + ((mag >> 8) & 1u)) >> 8);
}

// Two fp16 patterns, rounded so that bytes 1 and 3 are their e5m2 bytes: the
// same sum as half_to_e5m2 on 16-bit halves (for anything but NaN it cannot
// carry out of the magnitude, so the sign stays).
__device__ __forceinline__ uint32_t round_halves_e5m2(uint32_t w) {
  const u16x2 h = __builtin_bit_cast(u16x2, w);
  const u16x2 odd = __builtin_bit_cast(u16x2, (w >> 8) & 0x00010001u);
  return __builtin_bit_cast(uint32_t, h + u16x2{0x7f, 0x7f} + odd);
}

__device__ __forceinline__ float half_bits_to_float(uint32_t h) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}

// x combined by max with the value of the lane that DPP control CTRL names (the
// lanes of a row are all active), on the bits of non-negative floats, which
// order as integers do: one v_max_u32 each.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_max(uint32_t x) {
  const uint32_t y = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
  return x > y ? x : y;
}

// Maximum of a non-negative float over the LANES (4, 8, 16 or 32) neighbouring lanes of a row.
template <int LANES>
__device__ __forceinline__ float row_max(float f) {
  uint32_t x = __builtin_bit_cast(uint32_t, f);
  x = dpp_max<0xB1>(x);                              // quad_perm 1,0,3,2
  x = dpp_max<0x4E>(x);                              // quad_perm 2,3,0,1
  if constexpr (LANES >= 8) x = dpp_max<0x141>(x);   // row_half_mirror: the other quad of 8
  if constexpr (LANES >= 16) x = dpp_max<0x140>(x);  // row_mirror: the other 8 of 16
  f = __builtin_bit_cast(float, x);
  if constexpr (LANES >= 32) f = fmaxf(f, __shfl_xor(f, 16));
  return f;
}

// 16 bytes of fp16 -> 8 e5m2 bytes.
__device__ __forceinline__ u32x2 to_e5m2(u32x4 w) {
  // a NaN anywhere in the lane (its magnitude above infinity's) takes the
  // form that tests each value
  u16x2 m = __builtin_bit_cast(u16x2, w.x & 0x7fff7fffu);
  m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, w.y & 0x7fff7fffu));
  m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, w.z & 0x7fff7fffu));
  m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, w.w & 0x7fff7fffu));
  if (__builtin_expect(m[0] > 0x7c00u || m[1] > 0x7c00u, 0)) {
    uint32_t b[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) b[i] = half_to_e5m2(i & 1 ? w[i / 2] >> 16 : w[i / 2] & 0xffffu);
    return u32x2{b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24),
                 b[4] | (b[5] << 8) | (b[6] << 16) | (b[7] << 24)};
  }
  // v_perm: bytes 1, 3 of the first word, then of the second
  return u32x2{__builtin_amdgcn_perm(round_halves_e5m2(w.y), round_halves_e5m2(w.x), 0x07050301u),
               __builtin_amdgcn_perm(round_halves_e5m2(w.w), round_halves_e5m2(w.z), 0x07050301u)};
}

// a / 127 correctly rounded, for a = |fp16| or 1e-6f (every such value is
// checked against the division in tests/test_cache_write_math.py): the product
// with 1/127 corrected once by its exact remainder; infinity as it is.
__device__ __forceinline__ float div127(float a) {
  constexpr float kInv = 1.0f / 127.0f;
  const float q = a * kInv;
  return a < __builtin_inff() ? __builtin_fmaf(__builtin_fmaf(-q, 127.0f, a), kInv, q) : a;
}

// 16 bytes of fp16 -> 8 int8 bytes and the row's scale.
template <int SC, int LANES>
__device__ __forceinline__ u32x2 to_int8(u32x4 w, float &scale) {
  float x[8];
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    x[i] = half_bits_to_float(i & 1 ? w[i / 2] >> 16 : w[i / 2] & 0xffffu);
    // (emits nothing: keeps the products below from becoming v_fma_mix, which
    // takes the fp16 value itself at half the rate)
    asm("" : "+v"(x[i]));
    amax = fmaxf(amax, fabsf(x[i]));
  }
  amax = fmaxf(row_max<LANES>(amax), 1e-6f);
  scale = div127(amax);
  if constexpr (SC == PA_SCALE_FP16) scale = (float)(_Float16)scale;
  // round_half_even(x / scale) with the IEEE quotient's rounding: x times the
  // scale's reciprocal (v_rcp_f32, 1 ulp) is within 2 * 2^-23 of x / scale,
  // relatively, so for a quotient up to 127.5 the two round to different
  // integers only within 2^-15 of a half-integer. x * inv + 1.5 * 2^23 rounds
  // the product to an integer, half to even, and leaves it in the low mantissa
  // byte. A lane takes the division form when an element is within 2^-14 of a
  // half-integer, when one is NaN (__builtin_elementwise_maximum hands it on),
  // or when the row's largest quotient is 127.4 or more (infinities, and fp16
  // scales that rounded far down or to zero).
  const float inv = __builtin_amdgcn_rcpf(scale);
  constexpr float kMagic = 12582912.0f;
  uint32_t t[8];
  float off = __builtin_elementwise_maximum(__builtin_fmaf(amax, inv, -126.9f), 0.0f);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float r = __builtin_fmaf(x[i], inv, kMagic);
    t[i] = __builtin_bit_cast(uint32_t, r);
    off = __builtin_elementwise_maximum(off, fabsf(__builtin_fmaf(x[i], inv, kMagic - r)));
  }
  if (__builtin_expect(!(off < 0.5f - 0x1p-14f), 0)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float r = rintf(x[i] / scale);
      // a zero row with fp16 scales underflows the scale to 0: 0/0 is NaN,
      // which the reference's cast to int8 stores as 0
      const float q = (r != r) ? 0.f : fminf(fmaxf(r, -127.f), 127.f);
      t[i] = (uint32_t)(int32_t)q;
    }
  }
  // the low bytes, four to a word
  const uint32_t a = __builtin_amdgcn_perm(t[1], t[0], 0x0c0c0400u), b = __builtin_amdgcn_perm(t[3], t[2], 0x04000c0cu);
  const uint32_t c = __builtin_amdgcn_perm(t[5], t[4], 0x0c0c0400u), d = __builtin_amdgcn_perm(t[7], t[6], 0x04000c0cu);
  return u32x2{a | b, c | d};
}

// WIDE: some stride is 4 GiB or more, or block_size is not a power of two (64-bit
// products and divisions); otherwise strides and block ids fit 32 bits.
template <int KV, int SC, int D, bool WIDE>
__global__ void __launch_bounds__(256) cache_write_kernel(const WParams p) {
  constexpr int kLanesPerRow = D / 8;  // 8 fp16 (16 bytes) per lane
  const uint32_t tid = threadIdx.x;
  // The grid has at most p.groups workgroups, so the first pass needs no test:
  // one would wait for its argument (cold on an eager launch) before the others
  // are loaded.
  uint32_t g = blockIdx.x;
  do {
    uint32_t t, lane;  // token, lane in the token
    if (p.lanes <= 256) {
      const uint32_t tb = tid * p.inv_lanes >> 16;
      if (tb >= p.tpb) return;
      t = g * p.tpb + tb;
      lane = tid - tb * p.lanes;
    } else {
      t = g / p.parts;
      lane = (g % p.parts) * 256u + tid;
    }
    // (all these tests are uniform over a row's lanes)
    if (lane >= p.lanes || t >= p.tokens) continue;
    const uint32_t h = lane / kLanesPerRow, piece = lane % kLanesPerRow;

    const int64_t slot = p.slots[t];
    u32x4 w[2];
    w[0] = *reinterpret_cast<const u32x4 *>(
        p.key + at<WIDE>(at<WIDE>(piece * 16, h, p.skh), t, p.skt));
    w[1] = *reinterpret_cast<const u32x4 *>(
        p.value + at<WIDE>(at<WIDE>(piece * 16, h, p.svh), t, p.svt));
    // both rows are in flight with the slot: without this (it emits nothing)
    // the compiler moves their loads behind the slot's arrival
    asm volatile("" : : "v"(w[0]), "v"(w[1]));
    if (slot < 0 || slot >= p.max_slot) continue;
    uint64_t blk, off;
    if constexpr (WIDE) {
      blk = (uint64_t)slot / (uint32_t)p.block_size;
      off = (uint64_t)slot % (uint32_t)p.block_size;
    } else {
      blk = (uint64_t)slot >> p.log2_block;
      off = (uint32_t)slot & (uint32_t)(p.block_size - 1);
    }
    constexpr int kPiece = (KV == PA_KV_FP16 || KV == PA_KV_BF16) ? 16 : 8;  // bytes a lane stores
    const uint64_t cbase = at<WIDE>(at<WIDE>(at<WIDE>(piece * kPiece, h, p.sch), off, p.sct), blk, p.scn);

#pragma unroll
    for (int which = 0; which < 2; ++which) {
      uint8_t *dst = (which ? p.vc : p.kc) + cbase;
      if constexpr (KV == PA_KV_FP16 || KV == PA_KV_BF16) {
        __builtin_nontemporal_store(w[which], reinterpret_cast<u32x4 *>(dst));
      } else if constexpr (KV == PA_KV_FP8_E5M2) {
        __builtin_nontemporal_store(to_e5m2(w[which]), reinterpret_cast<u32x2 *>(dst));
      } else {
        float scale;
        __builtin_nontemporal_store(to_int8<SC, kLanesPerRow>(w[which], scale), reinterpret_cast<u32x2 *>(dst));
        if (piece == 0) {
          uint8_t *s = (which ? p.vs : p.ks) + at<WIDE>(at<WIDE>(0, off, p.sst), blk, p.ssn);
          if constexpr (SC == PA_SCALE_FP16) {
            reinterpret_cast<_Float16 *>(s)[h] = (_Float16)scale;
          } else {
            reinterpret_cast<float *>(s)[h] = scale;
          }
        }
      }
    }
  } while ((g += p.grid) < p.groups);
}

template <int KV, int SC, int D>
void launch_d(const WParams &p, dim3 grid, hipStream_t st) {
  const int64_t big = int64_t(1) << 32;
  const bool wide = p.log2_block < 0 || p.skt >= big || p.skh >= big || p.svt >= big || p.svh >= big ||
                    p.scn >= big || p.sct >= big || p.sch >= big || p.ssn >= big || p.sst >= big;
  if (wide)
    hipLaunchKernelGGL((cache_write_kernel<KV, SC, D, true>), grid, dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((cache_write_kernel<KV, SC, D, false>), grid, dim3(256), 0, st, p);
}

template <int KV, int SC>
hipError_t launch_w(const WParams &p, int d, dim3 grid, hipStream_t st) {
  switch (d) {
    case 32: launch_d<KV, SC, 32>(p, grid, st); break;
    case 64: launch_d<KV, SC, 64>(p, grid, st); break;
    case 128: launch_d<KV, SC, 128>(p, grid, st); break;
    default: launch_d<KV, SC, 256>(p, grid, st); break;
  }
  return hipGetLastError();
}

}  // namespace

extern "C" int pa_cache_write(const pa_cache_write_args *a, void *stream) {
  if (a == nullptr) return pa_fail(PA_ERR_INVALID, "args is NULL");
  if (a->num_tokens < 0) return pa_fail(PA_ERR_INVALID, "num_tokens %d < 0", a->num_tokens);
  if (!a->key || !a->value || !a->k_cache || !a->v_cache || !a->slot_mapping)
    return pa_fail(PA_ERR_INVALID, "key, value, k_cache, v_cache and slot_mapping must be non-NULL");
  if (a->num_kv_heads <= 0 || a->block_size <= 0 || a->num_blocks <= 0)
    return pa_fail(PA_ERR_INVALID, "num_kv_heads %d, block_size %d and num_blocks %d must be positive",
                   a->num_kv_heads, a->block_size, a->num_blocks);
  if (a->head_dim != 32 && a->head_dim != 64 && a->head_dim != 128 && a->head_dim != 256)
    return pa_fail(PA_ERR_UNSUPPORTED, "head_dim %d not in (32, 64, 128, 256)", a->head_dim);
  if (a->kv_dtype != PA_KV_FP16 && a->kv_dtype != PA_KV_FP8_E5M2 && a->kv_dtype != PA_KV_INT8 &&
      a->kv_dtype != PA_KV_BF16)
    return pa_fail(PA_ERR_INVALID, "kv_dtype %d unknown", a->kv_dtype);
  const int64_t strides[] = {a->stride_kt, a->stride_kh, a->stride_vt, a->stride_vh,
                             a->stride_cn, a->stride_ct, a->stride_ch};
  for (int64_t s : strides)
    if (s < 0) return pa_fail(PA_ERR_INVALID, "strides must be non-negative");
  const int elem = (a->kv_dtype == PA_KV_FP16 || a->kv_dtype == PA_KV_BF16) ? 2 : 1;
  const int piece = 8 * elem;  // bytes a lane stores
  if (!pa_aligned(a->key, 16) || !pa_aligned(a->value, 16) || (a->stride_kt * 2) % 16 ||
      (a->stride_kh * 2) % 16 || (a->stride_vt * 2) % 16 || (a->stride_vh * 2) % 16)
    return pa_fail(PA_ERR_INVALID, "key/value and their strides must be 16-byte aligned");
  if (!pa_aligned(a->k_cache, piece) || !pa_aligned(a->v_cache, piece) ||
      (a->stride_cn * elem) % piece || (a->stride_ct * elem) % piece || (a->stride_ch * elem) % piece)
    return pa_fail(PA_ERR_INVALID, "k_cache/v_cache and their strides must be %d-byte aligned", piece);
  int sb = 0;
  if (a->kv_dtype == PA_KV_INT8) {
    if (a->scale_dtype != PA_SCALE_FP16 && a->scale_dtype != PA_SCALE_FP32)
      return pa_fail(PA_ERR_INVALID, "int8 KV needs scale_dtype fp16 or fp32, got %d", a->scale_dtype);
    if (!a->k_scale || !a->v_scale) return pa_fail(PA_ERR_INVALID, "int8 KV needs k_scale and v_scale");
    if (a->stride_sn < 0 || a->stride_st < 0) return pa_fail(PA_ERR_INVALID, "scale strides must be non-negative");
    sb = a->scale_dtype == PA_SCALE_FP32 ? 4 : 2;
    if (!pa_aligned(a->k_scale, sb) || !pa_aligned(a->v_scale, sb))
      return pa_fail(PA_ERR_INVALID, "scale pointers must be %d-byte aligned", sb);
  } else if (a->scale_dtype != PA_SCALE_NONE) {
    return pa_fail(PA_ERR_INVALID, "scale_dtype must be PA_SCALE_NONE for kv_dtype %d", a->kv_dtype);
  }
  const int64_t rows = (int64_t)a->num_tokens * a->num_kv_heads;
  const int64_t lanes = (int64_t)a->num_kv_heads * (a->head_dim / 8);  // of one token
  const bool whole = lanes <= 256;  // a group holds whole tokens
  const uint32_t tpb = whole ? 256u / (uint32_t)lanes : 1u;
  const int64_t parts = whole ? 1 : (lanes + 255) >> 8;
  const int64_t groups = whole ? ((uint32_t)a->num_tokens + tpb - 1) / tpb : a->num_tokens * parts;
  if (lanes > 0xffffff00u || groups > 0x7fffffff)
    return pa_fail(PA_ERR_UNSUPPORTED, "too many rows (%lld)", (long long)rows);
  if (rows == 0) return pa_ok();

  WParams p;
  p.key = static_cast<const uint8_t *>(a->key);
  p.value = static_cast<const uint8_t *>(a->value);
  p.kc = static_cast<uint8_t *>(a->k_cache);
  p.vc = static_cast<uint8_t *>(a->v_cache);
  p.ks = static_cast<uint8_t *>(a->k_scale);
  p.vs = static_cast<uint8_t *>(a->v_scale);
  p.slots = a->slot_mapping;
  p.tokens = (uint32_t)a->num_tokens;
  p.lanes = (uint32_t)lanes;
  p.tpb = tpb;
  p.parts = (uint32_t)parts;
  p.groups = (uint32_t)groups;
  p.inv_lanes = whole ? (65536u + (uint32_t)lanes - 1) / (uint32_t)lanes : 0;
  p.block_size = a->block_size;
  p.log2_block = (a->block_size & (a->block_size - 1)) == 0 ? __builtin_ctz(a->block_size) : -1;
  p.max_slot = (int64_t)a->num_blocks * a->block_size;
  p.skt = a->stride_kt * 2;
  p.skh = a->stride_kh * 2;
  p.svt = a->stride_vt * 2;
  p.svh = a->stride_vh * 2;
  p.scn = a->stride_cn * elem;
  p.sct = a->stride_ct * elem;
  p.sch = a->stride_ch * elem;
  p.ssn = a->stride_sn * sb;
  p.sst = a->stride_st * sb;
  p.grid = (uint32_t)(groups < kMaxGrid ? groups : kMaxGrid);
  const dim3 grid(p.grid);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int d = a->head_dim;
  hipError_t e;
  if (a->kv_dtype == PA_KV_FP16) e = launch_w<PA_KV_FP16, PA_SCALE_NONE>(p, d, grid, st);
  else if (a->kv_dtype == PA_KV_BF16) e = launch_w<PA_KV_BF16, PA_SCALE_NONE>(p, d, grid, st);
  else if (a->kv_dtype == PA_KV_FP8_E5M2) e = launch_w<PA_KV_FP8_E5M2, PA_SCALE_NONE>(p, d, grid, st);
  else if (a->scale_dtype == PA_SCALE_FP32) e = launch_w<PA_KV_INT8, PA_SCALE_FP32>(p, d, grid, st);
  else e = launch_w<PA_KV_INT8, PA_SCALE_FP16>(p, d, grid, st);
  if (e != hipSuccess) return pa_fail(PA_ERR_HIP, "cache write launch failed: %s", hipGetErrorString(e));
  return pa_ok();
}
