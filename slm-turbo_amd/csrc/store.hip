// Quantize-on-write store into the packed per-token 4-bit paged cache.
//
// Same arithmetic as the reference's kv_quantize_store_kernel
// (kernels/kv_dequant_kernels.cuh:816-919), laid out for CDNA4: 8 dims per lane, so
// a (token, kv head) row is 8 lanes at head_dim 64 and 16 at 80 and 128 (6 of them
// idle at 80), and a wave takes 8 or 4 rows.  K and V are one 16-byte load and one
// 4-byte store each per lane; minima and maxima go over packed fp16 pairs and DPP
// within the row's lanes.  Every fp32 operation is rounded separately (contraction
// off) so codes and fp16 rulers are bit-exact with the reference.
//
// Long prompts move each byte once (7001 tokens, 8 KV heads of 128 dims: 28.5 MB read and
// 7.2 MB written by the counters, in 10.2 us), and what bounds them is the launch and each
// wave's one chain of load, reduction and store, not the memory: rotating over 430 MB of
// buffers, so that all of it comes from HBM, takes 6 % longer than passes over one set,
// which the Infinity Cache holds.  2 dims per lane, a wave per row, byte stores and the
// compiler's division took 23.1 us.
#include "slmt_internal.h"

namespace slmt {

namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ f16x2 pair_min(f16x2 a, f16x2 b) { return __builtin_elementwise_min(a, b); }
__device__ __forceinline__ f16x2 pair_max(f16x2 a, f16x2 b) { return __builtin_elementwise_max(a, b); }
template <int CTRL>
__device__ __forceinline__ f16x2 pair_dpp(f16x2 h) {
  return __builtin_bit_cast(f16x2, dpp_u<CTRL>(__builtin_bit_cast(uint32_t, h)));
}

// Eight fp16 values from an address that is a multiple of 4 only (the hardware
// takes 16-byte loads there).
struct Eight {
  f16x2 h[4];
};
__device__ __forceinline__ Eight load_eight(const uint16_t* p) {
  Eight v;
  __builtin_memcpy(&v, __builtin_assume_aligned(p, 4), 16);
  return v;
}

// Ruler of a row spread over LANES lanes: minimum and step (1 where the range is 0
// or no number).  NaNs are passed over; a row of nothing else has the minimum
// infinity at head_dim 64 and 80 (`seed`) and NaN at 128.
template <int LANES, bool SEED>
__device__ __forceinline__ void row_ruler(const Eight& x, float& mn, float& step) {
#pragma clang fp contract(off)
  f16x2 lo = pair_min(pair_min(x.h[0], x.h[1]), pair_min(x.h[2], x.h[3]));
  f16x2 hi = pair_max(pair_max(x.h[0], x.h[1]), pair_max(x.h[2], x.h[3]));
  lo = pair_min(lo, pair_dpp<DPP_QUAD_XOR1>(lo));
  hi = pair_max(hi, pair_dpp<DPP_QUAD_XOR1>(hi));
  lo = pair_min(lo, pair_dpp<DPP_QUAD_XOR2>(lo));
  hi = pair_max(hi, pair_dpp<DPP_QUAD_XOR2>(hi));
  if (LANES == 8) {
    lo = pair_min(lo, pair_dpp<DPP_ROW_HALF_MIRROR>(lo));
    hi = pair_max(hi, pair_dpp<DPP_ROW_HALF_MIRROR>(hi));
  } else {
    lo = pair_min(lo, pair_dpp<DPP_ROW_ROR4>(lo));
    hi = pair_max(hi, pair_dpp<DPP_ROW_ROR4>(hi));
    lo = pair_min(lo, pair_dpp<DPP_ROW_ROR8>(lo));
    hi = pair_max(hi, pair_dpp<DPP_ROW_ROR8>(hi));
  }
  mn = fminf((float)lo[0], (float)lo[1]);
  float mx = fmaxf((float)hi[0], (float)hi[1]);
  if (SEED) {
    mn = fminf(mn, INFINITY);
    mx = fmaxf(mx, -INFINITY);
  }
  step = (mx - mn) / 15.0f;
  if (!(step > 0.0f)) step = 1.0f;
}

// Codes (int)((x - mn) / step + 0.5) of eight values, two a byte.  The quotient is
// correctly rounded as a division's: r is 1 / step correctly rounded, the first
// residual step leaves less than an ulp of error and the second, from there, the
// rounded quotient (Markstein).  Nothing under- or overflows: x - mn is 0 or at
// least 2^-24, and step lies in [2^-24 / 15, 8734].  Half the compiler's division.
// Infinite steps and NaNs, which the division takes to 0 or NaN, come out NaN, and
// NaN is code 0; a number's quotient is at most 15 (1 + 2^-22) and needs no clamp.
__device__ __forceinline__ uint32_t codes(const Eight& x, float mn, float step, float r) {
#pragma clang fp contract(off)
  uint32_t out = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float a = (float)x.h[i >> 1][i & 1] - mn;
    float q = a * r;
    q = __builtin_fmaf(__builtin_fmaf(-q, step, a), r, q);
    q = __builtin_fmaf(__builtin_fmaf(-q, step, a), r, q);
    out |= (uint32_t)fmaxf(q + 0.5f, 0.0f) << (4 * i);
  }
  return out;
}

template <int D>
__global__ void __launch_bounds__(kThreads)
quantize_store_kernel(const uint16_t* __restrict__ key, int64_t key_stride,
                      const uint16_t* __restrict__ value, int64_t value_stride,
                      uint8_t* __restrict__ cache, int64_t num_slots,
                      const int64_t* __restrict__ slot_mapping, uint32_t rows, uint32_t KV) {
  constexpr int SLOT = D + 8, HALF = D / 2;
  constexpr int LANES = D == 64 ? 8 : 16;
  const int lane = threadIdx.x & (LANES - 1);
  const uint32_t row = blockIdx.x * (kThreads / LANES) + threadIdx.x / LANES;
  const uint32_t rw = min(row, rows - 1);             // lanes past the end repeat the last row and store nothing
  const uint32_t t = rw / KV, h = rw - t * KV;
  // The row is quantized whether or not its slot is valid and only the stores
  // test it: with an early exit on the slot the row's K/V loads were issued
  // after the slot's had returned, two dependent round trips per call.
  const int64_t slot = slot_mapping[t];
  const int d0 = 8 * min(lane, D / 8 - 1);            // idle lanes re-read the row's last dims
  const Eight k = load_eight(key + t * key_stride + (int64_t)h * D + d0);
  const Eight v = load_eight(value + t * value_stride + (int64_t)h * D + d0);
  float kmin, kstep, vmin, vstep;
  row_ruler<LANES, D != 128>(k, kmin, kstep);
  row_ruler<LANES, D != 128>(v, vmin, vstep);
  const uint32_t kc = codes(k, kmin, kstep, 1.0f / kstep);
  const uint32_t vc = codes(v, vmin, vstep, 1.0f / vstep);

  // padding token / out of range: no store
  if (row >= rows || slot < 0 || slot >= num_slots) return;
  uint8_t* dst = cache + (slot * KV + h) * (int64_t)SLOT;
  if (lane < D / 8) {
    *reinterpret_cast<uint32_t*>(dst + 4 * lane) = kc;
    *reinterpret_cast<uint32_t*>(dst + HALF + 4 * lane) = vc;
  }
  if (lane == 0) {
    const uint32_t r0 = (uint32_t)f2h(kmin) | ((uint32_t)f2h(kstep) << 16);
    const uint32_t r1 = (uint32_t)f2h(vmin) | ((uint32_t)f2h(vstep) << 16);
    *reinterpret_cast<uint2*>(dst + D) = make_uint2(r0, r1);   // slot base is 8-byte aligned
  }
}

}  // namespace

int launch_quantize_store(const void* key, int64_t key_stride, const void* value,
                          int64_t value_stride, void* cache, int64_t num_slots,
                          const int64_t* slot_mapping, int64_t N, int KV, int D,
                          hipStream_t stream) {
  if (N == 0) return SLMT_OK;
  // (row numbers are 32-bit: 2^32 rows of K alone would not fit the device)
  const int64_t rows = N * KV, per_block = kThreads / (D == 64 ? 8 : 16);
  const int64_t blocks = (rows + per_block - 1) / per_block;
  if (rows >= (int64_t(1) << 32) - kThreads || blocks > 0x7fffffffLL)
    return fail(SLMT_ERR_UNSUPPORTED, "store: too many tokens for one launch");
  const dim3 grid((unsigned)blocks), block(kThreads);
  auto k = reinterpret_cast<const uint16_t*>(key);
  auto v = reinterpret_cast<const uint16_t*>(value);
  auto c = reinterpret_cast<uint8_t*>(cache);
  switch (D) {
    case 64:
      hipLaunchKernelGGL(quantize_store_kernel<64>, grid, block, 0, stream, k, key_stride, v,
                         value_stride, c, num_slots, slot_mapping, (uint32_t)rows, (uint32_t)KV);
      break;
    case 80:
      hipLaunchKernelGGL(quantize_store_kernel<80>, grid, block, 0, stream, k, key_stride, v,
                         value_stride, c, num_slots, slot_mapping, (uint32_t)rows, (uint32_t)KV);
      break;
    case 128:
      hipLaunchKernelGGL(quantize_store_kernel<128>, grid, block, 0, stream, k, key_stride, v,
                         value_stride, c, num_slots, slot_mapping, (uint32_t)rows, (uint32_t)KV);
      break;
    default:
      return fail(SLMT_ERR_INVALID, "store: head_dim must be 64/80/128, got " + std::to_string(D));
  }
  return check_launch("store");
}

}  // namespace slmt
