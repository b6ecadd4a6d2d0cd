// Per-channel asymmetric 4-bit quantizer of the standalone path, on the GPU.
//
// The reference runs this as host-side torch code on fp16 tensors
// (compute_scale_zero / quantize_tensor, kernels/benchmark/benchmark.py:26-56):
// every op produces an fp16 result, i.e. it is evaluated in fp32 and rounded
// to nearest-even fp16.  fp32 carries >= 2*11+2 significand bits, so
// fp16(fp32(a op b)) is the correctly rounded fp16 result and this kernel
// reproduces torch's bytes exactly.  Reductions follow torch.min/torch.max
// (a NaN anywhere in a channel makes the channel's min/max NaN).
//
// A channel's ruler needs every row before any row can be quantized.  Up to
// kMaxRows rows a workgroup holds all of them, for 8 channels of one KV head, in
// registers: memory is read once and one launch does it all.  Longer sequences
// take three: every chunk's minima and maxima, the rulers, the codes.  K and V go
// through one launch together.
#include "slmt_internal.h"

#include <algorithm>

namespace slmt {

namespace {

constexpr int kRegThreads = 1024;
constexpr int kRegPasses = 8;    // rows each thread holds at most
constexpr int64_t kMaxRows = kRegThreads * kRegPasses;
constexpr int kMaxChunks = 64;   // chunks of a long sequence
constexpr int kChunkRows = 64;   // their smallest size (8 rows' codes hold a chunk's minima and maxima)
constexpr int kRowPasses = 4;    // rows per thread of the codes kernel
constexpr int kXcds = 8;

// torch.min / torch.max of pairs: a NaN operand gives NaN (v_pk_minimum3_f16)
__device__ __forceinline__ f16x2 pk_min(f16x2 a, f16x2 b) { return __builtin_elementwise_minimum(a, b); }
__device__ __forceinline__ f16x2 pk_max(f16x2 a, f16x2 b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ f16x2 as_pair(uint32_t w) { return __builtin_bit_cast(f16x2, w); }
__device__ __forceinline__ uint32_t as_word(f16x2 h) { return __builtin_bit_cast(uint32_t, h); }

__device__ __forceinline__ float r16(float x) { return h2f(f2h(x)); }  // round to fp16

// Eight fp16 values, from an address that is a multiple of 2 or 4 only (the
// hardware takes 16-byte loads there).
struct Half8 {
  f16x2 h[4];
};
template <int ALIGN = 4>
__device__ __forceinline__ Half8 load8(const uint16_t* p) {
  Half8 v;
  __builtin_memcpy(&v, __builtin_assume_aligned(p, ALIGN), 16);
  return v;
}

// Minima and maxima of 8 channels.
struct Range8 {
  f16x2 mn[4], mx[4];
  __device__ __forceinline__ void set(const Half8& v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) mn[i] = mx[i] = v.h[i];
  }
  __device__ __forceinline__ void add(const Half8& v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      mn[i] = pk_min(mn[i], v.h[i]);
      mx[i] = pk_max(mx[i], v.h[i]);
    }
  }
};

// A ruler pair and the scale's reciprocal, of 8 channels.
struct Rulers8 {
  float sc[8], rc[8];
  f16x2 zp[4];
  __device__ __forceinline__ void set(const Half8& scale, const Half8& zero) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      sc[i] = (float)scale.h[i >> 1][i & 1];
      rc[i] = __builtin_amdgcn_rcpf(sc[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) zp[i] = zero.h[i];
  }
};

// x / sc rounded to fp16, for fp16 x and sc: one residual step on x * rcp(sc)
// leaves the fp32 quotient within an ulp (2^-23), and exact where it is a number of
// 12 bits.  A quotient of two 11-bit significands that is not itself the middle
// between two fp16 numbers lies at least 2^-23 of its size from every such middle, so
// it rounds to the same fp16 as the exact quotient does (all 2^32 pairs were
// compared).  v_div_fixup gives the quotients of 0, infinities and NaN.  The
// compiler's correctly rounded division took twice the instructions.
__device__ __forceinline__ _Float16 quotient(float x, float sc, float rc) {
#pragma clang fp contract(off)
  const float q0 = x * rc;
  const float q1 = __builtin_fmaf(__builtin_fmaf(-q0, sc, x), rc, q0);
  return (_Float16)__builtin_amdgcn_div_fixupf(q1, sc, x);
}

// q = clamp(round(x / scale) + zero, 0, 15), an fp16 result after each op; NaN
// codes (a scale that underflowed) are 0: max(NaN, 0) is 0.  Eight dims, four bytes.
__device__ __forceinline__ uint32_t codes8(const Half8& x, const Rulers8& r) {
#pragma clang fp contract(off)
  uint32_t out = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f16x2 q;
    q[0] = quotient((float)x.h[i][0], r.sc[2 * i], r.rc[2 * i]);
    q[1] = quotient((float)x.h[i][1], r.sc[2 * i + 1], r.rc[2 * i + 1]);
    q = __builtin_elementwise_roundeven(q) + r.zp[i];
    q = __builtin_elementwise_max(q, (f16x2)(_Float16)0.0f);
    q = __builtin_elementwise_min(q, (f16x2)(_Float16)15.0f);
    // 1024 + n has the bits 0x6400 | n (a fractional zero point: truncated)
    const uint32_t w = as_word(__builtin_elementwise_trunc(q) + (f16x2)(_Float16)1024.0f) & 0x000F000Fu;
    out |= ((w | (w >> 12)) & 0xFFu) << (8 * i);
  }
  return out;
}

// scale = (max - min) / 15 ; zero = 0 - round(min / scale), clamped (fp16 after each op)
__device__ __forceinline__ void ruler(_Float16 lo, _Float16 hi, uint16_t& scale, uint16_t& zero) {
#pragma clang fp contract(off)
  float mn = (float)lo, mx = (float)hi;
  mn = mn != mn ? __builtin_nanf("") : mn;
  mx = mx != mx ? __builtin_nanf("") : mx;
  const float scale_raw = r16(r16(mx - mn) / 15.0f);
  const float zero_raw = r16(0.0f - __builtin_rintf(r16(mn / scale_raw)));
  const bool is_const = (mx == mn);
  const float zp = is_const ? 0.0f : zero_raw;
  scale = f2h(is_const ? 1.0f : scale_raw);
  zero = f2h(zp != zp ? zp : fminf(fmaxf(zp, 0.0f), 15.0f));   // torch.clamp keeps NaN
}

// The tensors of one call, at most two of the same shape.
struct Tensors {
  const uint16_t* x[2];
  uint8_t* packed[2];
  uint16_t *scale[2], *zero[2];
};

template <int CTRL>
__device__ __forceinline__ f16x2 dpp_pair(f16x2 h) { return as_pair(dpp_u<CTRL>(as_word(h))); }

// Rows in registers, one thread per row and 8 channels; a thread's rows are
// blockDim apart, past the end the last row again.  The 16-byte pieces of a row go
// to workgroups of the same XCD (workgroups go round the XCDs in turn), whose L2
// then reads a row's lines once and puts its codes together.  Against one workgroup
// per KV head and 64 channels that walked the rows twice, 4 waves at a time, us of
// kernels for K and V: 4 KV heads, 64 dims, 1500 tokens 2 x 87 -> 6.1; 8 KV heads,
// 128 dims, 4000 tokens 2 x 380 -> 14.3 (with 16 channels per workgroup, rows over
// every XCD and the compiler's division 12.2 and 27.8).  What bounds it is one
// round trip, the reductions and the conversions of the few CUs that it uses.
template <int RPT>
__global__ void __launch_bounds__(kRegThreads) quantize_rows_kernel(const Tensors t, int KV, int nt, int S, int D) {
  __shared__ uint32_t s_mn[kRegThreads / 64][4], s_mx[kRegThreads / 64][4];
  __shared__ uint16_t s_ruler[2][8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, NT = blockDim.x;
  const int slices = D / 8;
  const int p = blockIdx.x % kXcds + kXcds * (blockIdx.x / (kXcds * slices));   // (tensor, KV head)
  if (p >= KV * nt) return;
  const int slice = blockIdx.x / kXcds % slices, tz = p / KV, kv = p - tz * KV;
  const uint16_t* base = t.x[tz] + (int64_t)kv * S * D + 8 * slice;

  Half8 v[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) v[i] = load8(base + (int64_t)min(tid + i * NT, S - 1) * D);
  Range8 r;
  r.set(v[0]);
#pragma unroll
  for (int i = 1; i < RPT; ++i) r.add(v[i]);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    f16x2 a = r.mn[c], b = r.mx[c];
    a = pk_min(a, dpp_pair<DPP_QUAD_XOR1>(a));
    b = pk_max(b, dpp_pair<DPP_QUAD_XOR1>(b));
    a = pk_min(a, dpp_pair<DPP_QUAD_XOR2>(a));
    b = pk_max(b, dpp_pair<DPP_QUAD_XOR2>(b));
    a = pk_min(a, dpp_pair<DPP_ROW_ROR4>(a));
    b = pk_max(b, dpp_pair<DPP_ROW_ROR4>(b));
    a = pk_min(a, dpp_pair<DPP_ROW_ROR8>(a));
    b = pk_max(b, dpp_pair<DPP_ROW_ROR8>(b));
    auto a16 = __builtin_amdgcn_permlane16_swap(as_word(a), as_word(a), false, false);
    auto b16 = __builtin_amdgcn_permlane16_swap(as_word(b), as_word(b), false, false);
    a = pk_min(as_pair(a16[0]), as_pair(a16[1]));
    b = pk_max(as_pair(b16[0]), as_pair(b16[1]));
    auto a32 = __builtin_amdgcn_permlane32_swap(as_word(a), as_word(a), false, false);
    auto b32 = __builtin_amdgcn_permlane32_swap(as_word(b), as_word(b), false, false);
    a = pk_min(as_pair(a32[0]), as_pair(a32[1]));
    b = pk_max(as_pair(b32[0]), as_pair(b32[1]));
    if (lane == 0) {
      s_mn[wave][c] = as_word(a);
      s_mx[wave][c] = as_word(b);
    }
  }
  __syncthreads();
  if (tid < 8) {
    f16x2 a = as_pair(s_mn[0][tid >> 1]), b = as_pair(s_mx[0][tid >> 1]);
    for (int w = 1; w < NT / 64; ++w) {
      a = pk_min(a, as_pair(s_mn[w][tid >> 1]));
      b = pk_max(b, as_pair(s_mx[w][tid >> 1]));
    }
    uint16_t scale, zero;
    ruler(tid & 1 ? a[1] : a[0], tid & 1 ? b[1] : b[0], scale, zero);
    s_ruler[0][tid] = scale;
    s_ruler[1][tid] = zero;
    const int64_t o = (int64_t)kv * D + 8 * slice + tid;
    t.scale[tz][o] = scale;
    t.zero[tz][o] = zero;
  }
  __syncthreads();
  Rulers8 ru;
  ru.set(load8<2>(s_ruler[0]), load8<2>(s_ruler[1]));
  uint8_t* out = t.packed[tz] + (int64_t)kv * S * (D / 2) + 4 * slice;
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int row = tid + i * NT;
    if (row < S) {
      const uint32_t q = codes8(v[i], ru);
      __builtin_memcpy(out + (int64_t)row * (D / 2), &q, 4);
    }
  }
}

// Long sequences (8 KV heads, 128 dims, 100000 tokens, K and V, 410 MB in and 102 out:
// 70.6 + 4.6 + 89.9 us, the first kernel's bytes at 5.8 TB/s; 30 ms before): chunk c of n is rows [c S / n, (c + 1) S / n).  Its minima and
// maxima (fp16, exact; a pair of channels' minima, then their maxima) are left at
// the start of the chunk's own codes, which the last of the three launches
// overwrites.
__device__ __forceinline__ int64_t chunk_row(int c, int S, int n) { return (int64_t)c * S / n; }

__global__ void __launch_bounds__(256) chunk_range_kernel(const Tensors t, int S, int D) {
  __shared__ uint32_t s_mn[4][256], s_mx[4][256];
  const int tid = threadIdx.x, kv = blockIdx.y, tz = blockIdx.z;
  const int tpr = D / 8, rows = 256 / tpr;             // threads per row, rows per pass
  const int64_t lo = chunk_row(blockIdx.x, S, gridDim.x), hi = chunk_row(blockIdx.x + 1, S, gridDim.x);
  const int rr = tid / tpr, j = tid - rr * tpr;
  const uint16_t* base = t.x[tz] + (int64_t)kv * S * D + 8 * j;
  Range8 r;
  r.set(load8(base + min(lo + rr, hi - 1) * D));
  for (int64_t row = lo + rr; row < hi; row += 4 * rows) {
    Half8 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = load8(base + min(row + i * rows, hi - 1) * D);   // past the end: a row again
#pragma unroll
    for (int i = 0; i < 4; ++i) r.add(v[i]);
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    s_mn[c][tid] = as_word(r.mn[c]);
    s_mx[c][tid] = as_word(r.mx[c]);
  }
  __syncthreads();
  if (tid < D / 2) {
    const int c = tid & 3, t0 = tid >> 2;
    f16x2 a = as_pair(s_mn[c][t0]), b = as_pair(s_mx[c][t0]);
    for (int k = 1; k < rows; ++k) {
      a = pk_min(a, as_pair(s_mn[c][k * tpr + t0]));
      b = pk_max(b, as_pair(s_mx[c][k * tpr + t0]));
    }
    const uint32_t w[2] = {as_word(a), as_word(b)};
    __builtin_memcpy(t.packed[tz] + ((int64_t)kv * S + lo) * (D / 2) + 8 * tid, w, 8);
  }
}

// One workgroup per tensor and KV head; wave w takes chunks w, w + 16, ... of n.
__global__ void __launch_bounds__(1024) chunk_ruler_kernel(const Tensors t, int S, int D, int n) {
  __shared__ uint2 s_r[16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, kv = blockIdx.x, tz = blockIdx.y;
  const int pair = min(lane, D / 2 - 1);
  uint2 w[kMaxChunks / 16];
#pragma unroll
  for (int i = 0; i < kMaxChunks / 16; ++i) {
    const int c = min(wave + 16 * i, n - 1);
    __builtin_memcpy(&w[i], t.packed[tz] + ((int64_t)kv * S + chunk_row(c, S, n)) * (D / 2) + 8 * pair, 8);
  }
  f16x2 a = as_pair(w[0].x), b = as_pair(w[0].y);
#pragma unroll
  for (int i = 1; i < kMaxChunks / 16; ++i) {
    a = pk_min(a, as_pair(w[i].x));
    b = pk_max(b, as_pair(w[i].y));
  }
  s_r[wave][lane] = make_uint2(as_word(a), as_word(b));
  __syncthreads();
  if (wave > 0 || lane >= D / 2) return;
  for (int k = 1; k < 16; ++k) {
    a = pk_min(a, as_pair(s_r[k][lane].x));
    b = pk_max(b, as_pair(s_r[k][lane].y));
  }
#pragma unroll
  for (int e = 0; e < 2; ++e)
    ruler(a[e], b[e], t.scale[tz][(int64_t)kv * D + 2 * lane + e], t.zero[tz][(int64_t)kv * D + 2 * lane + e]);
}

// Codes with the rulers given: the append with frozen rulers (quantize_tensor of
// the reference, kernels/benchmark/benchmark.py:45-56) and the last launch of a
// long sequence.  A thread takes 8 dims of kRowPasses rows: 16-byte loads, 4-byte
// stores, the rulers' reciprocals once.
__global__ void __launch_bounds__(256)
quantize_rulers_kernel(const Tensors t, int64_t x_head_stride, int64_t x_seq_stride, int S, int D,
                       int64_t out_head_stride, int64_t out_seq_stride) {
  const int kv = blockIdx.y, tz = blockIdx.z;
  const int tpr = D / 8, rows = 256 / tpr;
  const int rr = threadIdx.x / tpr, j = threadIdx.x - rr * tpr;
  const int64_t row0 = (int64_t)blockIdx.x * rows * kRowPasses + rr;
  if (rr >= rows || row0 >= S) return;
  const uint16_t* x = t.x[tz] + kv * x_head_stride + 8 * j;
  Half8 v[kRowPasses];
#pragma unroll
  for (int i = 0; i < kRowPasses; ++i) v[i] = load8(x + min(row0 + i * rows, (int64_t)S - 1) * x_seq_stride);
  Rulers8 ru;
  ru.set(load8<2>(t.scale[tz] + (int64_t)kv * D + 8 * j), load8<2>(t.zero[tz] + (int64_t)kv * D + 8 * j));
  uint8_t* out = t.packed[tz] + kv * out_head_stride + 4 * j;
#pragma unroll
  for (int i = 0; i < kRowPasses; ++i) {
    const int64_t row = row0 + i * rows;
    if (row < S) {
      const uint32_t q = codes8(v[i], ru);
      __builtin_memcpy(out + row * out_seq_stride, &q, 4);
    }
  }
}

int launch_rulers(const Tensors& t, int nt, int64_t x_head_stride, int64_t x_seq_stride, int KV, int S, int D,
                  int64_t out_head_stride, int64_t out_seq_stride, hipStream_t stream) {
  const int rows = 256 / (D / 8) * kRowPasses;
  hipLaunchKernelGGL(quantize_rulers_kernel, dim3((S + rows - 1) / rows, KV, nt), dim3(256), 0, stream, t,
                     x_head_stride, x_seq_stride, S, D, out_head_stride, out_seq_stride);
  return check_launch("quantize_tensor");
}

}  // namespace

int launch_quantize_rulers(const void* x, int64_t x_head_stride, int64_t x_seq_stride, int KV, int S, int D,
                           const void* scale, const void* zero, void* packed, int64_t out_head_stride,
                           int64_t out_seq_stride, hipStream_t stream) {
  if (KV == 0 || S == 0) return SLMT_OK;
  if (((int64_t)S * (D / 2) + 255) / 256 > 0x7fffffffLL || KV > 65535)
    return fail(SLMT_ERR_UNSUPPORTED, "quantize_tensor: too large for one launch");
  Tensors t{};
  t.x[0] = reinterpret_cast<const uint16_t*>(x);
  t.scale[0] = const_cast<uint16_t*>(reinterpret_cast<const uint16_t*>(scale));   // read only
  t.zero[0] = const_cast<uint16_t*>(reinterpret_cast<const uint16_t*>(zero));
  t.packed[0] = reinterpret_cast<uint8_t*>(packed);
  return launch_rulers(t, 1, x_head_stride, x_seq_stride, KV, S, D, out_head_stride, out_seq_stride, stream);
}

int launch_quantize_per_channel(int nt, const void* const* x, int KV, int S, int D, void* const* packed,
                                void* const* scale, void* const* zero, hipStream_t stream) {
  if (KV == 0) return SLMT_OK;
  Tensors t{};
  for (int i = 0; i < nt; ++i) {
    t.x[i] = reinterpret_cast<const uint16_t*>(x[i]);
    t.packed[i] = reinterpret_cast<uint8_t*>(packed[i]);
    t.scale[i] = reinterpret_cast<uint16_t*>(scale[i]);
    t.zero[i] = reinterpret_cast<uint16_t*>(zero[i]);
  }
  const int kvs = 65535;   // KV heads per launch (grid y)
  for (int kv0 = 0; kv0 < KV; kv0 += kvs) {
    const int n = std::min(kvs, KV - kv0);
    if (S <= kMaxRows) {
      const int threads = std::min(kRegThreads, (S + 63) & ~63);
      const int rpt = (S + threads - 1) / threads;
      const dim3 grid(kXcds * (D / 8) * ((n * nt + kXcds - 1) / kXcds)), block(threads);
      if (rpt <= 1) hipLaunchKernelGGL(quantize_rows_kernel<1>, grid, block, 0, stream, t, n, nt, S, D);
      else if (rpt <= 2) hipLaunchKernelGGL(quantize_rows_kernel<2>, grid, block, 0, stream, t, n, nt, S, D);
      else if (rpt <= 4) hipLaunchKernelGGL(quantize_rows_kernel<4>, grid, block, 0, stream, t, n, nt, S, D);
      else hipLaunchKernelGGL(quantize_rows_kernel<kRegPasses>, grid, block, 0, stream, t, n, nt, S, D);
    } else {
      const int chunks = std::max(1, std::min({kMaxChunks, 1024 / (n * nt), S / kChunkRows}));
      hipLaunchKernelGGL(chunk_range_kernel, dim3(chunks, n, nt), dim3(256), 0, stream, t, S, D);
      hipLaunchKernelGGL(chunk_ruler_kernel, dim3(n, nt), dim3(1024), 0, stream, t, S, D, chunks);
      if (int rc = launch_rulers(t, nt, (int64_t)S * D, D, n, S, D, (int64_t)S * (D / 2), D / 2, stream)) return rc;
    }
    if (int rc = check_launch("quantize_per_channel")) return rc;
    for (int i = 0; i < nt; ++i) {
      t.x[i] += (int64_t)n * S * D;
      t.packed[i] += (int64_t)n * S * (D / 2);
      t.scale[i] += (int64_t)n * D;
      t.zero[i] += (int64_t)n * D;
    }
  }
  return SLMT_OK;
}

}  // namespace slmt
