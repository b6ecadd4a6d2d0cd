// Chunked prefill over the packed per-token 4-bit paged cache on the matrix cores,
// head_dim 64, 80 and 128, any number of query heads per KV head: every query token
// of a serving step attends to its request's cached tokens up to its own position
// (the reference leaves continuation unsupported, adapters/vllm_adapter.py:238-239).
//
// A workgroup takes 64 query columns of one request and KV head, column = (token,
// query head of the KV head), 16 per wave, and walks the 64-key tiles that they can
// see.  As in the per-channel prefill everything is transposed, so a lane owns one
// query column from the scores to the output:
//   S^T = K Q^T,  P^T = exp2(S^T - m),  O^T += V^T P^T    (v_mfma_f32_16x16x32_f16)
// and the tiles are converted once per workgroup into a 2-stage LDS ring, K as
// [key][dim] and V^T as [dim][key] fp16 rows (prefill_mfma.hip has the layouts'
// reasons); a tile's codes are in registers two tiles ahead and its block-table
// entries three.
//
// Exactness: codes enter as (n - 8) 2^-9, the query as it is; both are fp16 numbers and
// their products exact, so a score is kstep (q . (n - 8)) + (kmin + 8 kstep) sum(q)
// with fp32 sums (log2(e) / sqrt(D) folded into the staged rulers).  Weights
// p * vstep enter as an fp16 number and the fp16 remainder in units of 2^-11, two
// products into two accumulators, ~22 bits; sum(p) and sum(p (vmin + 8 vstep)) stay
// in fp32.
//
// Long contexts are split into parts of about `split_tiles` tiles (blockIdx.z), which
// write (m, l, o) partials; merge_kernel, next on the stream, joins them.
//
// Bound by vector-instruction issue, 330 per wave and tile, half of them the softmax.
// Every query token as a sequence of its own in the batched decode, the path before,
// read the cache once per token.  us per step with the store: 500 tokens on 1393 of
// context beside 12 decodes, 32 q / 4 KV heads, 64 dims, 106 -> 44.  Two column sets
// per wave, which halve the staging per column, measured no faster (36 to 45 us for the
// kernel against 38): fewer waves are left to fill the issue slots.
#include "slmt_internal.h"

#include <algorithm>
#include <type_traits>

namespace slmt {
namespace chunk {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int BM = 64;             // query columns per workgroup
constexpr int BN = 64;             // keys per tile
constexpr float kMargin = 4.0f;    // the weights' reference lies this far (base 2) above the largest score

template <int D>
struct Geo {
  static constexpr int QB = (D + 31) / 32;   // 32-dim blocks of QK
  static constexpr int KROW = QB * 64 + 32;
  static constexpr int VROW = BN * 2 + 32;
  static constexpr int KBYTES = BN * KROW;
  static constexpr int ROFF = KBYTES + D * VROW;   // the keys' K rulers, 8 bytes each, then their V rulers
  static constexpr int STAGE = ROFF + BN * 16;
  static constexpr int LDS = 2 * STAGE;
  static constexpr int KW = D / 64;
  static constexpr int VW = D / 64;
  static constexpr bool X = D == 80;         // 16 dims more: 2 bytes of K, 1 of V per key and thread
};

// Position of key k of a tile in a V^T row (see prefill_mfma.hip).
__device__ __forceinline__ int vpos(int k) { return (k & 32) | ((k & 12) << 1) | ((k & 16) >> 2) | (k & 3); }

// Codes n of a pair (bits 0-3 and 16-19; as fp16 numbers n 2^-24) to (n - 8) 2^-9: one
// exact packed fma; kCode makes up for the 2^-9.
constexpr float kCode = 512.0f;
__device__ __forceinline__ uint32_t centred(uint32_t w) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(half2v, w),
                                                                half2v{(_Float16)0x1p15f, (_Float16)0x1p15f},
                                                                half2v{(_Float16)-0x1p-6f, (_Float16)-0x1p-6f}));
}
// of the low nibbles of byte i of a and b
__device__ __forceinline__ uint32_t nib_pair(uint32_t a, uint32_t b, int i) {
  return centred(__builtin_amdgcn_perm(b, a, 0x0C000C00u | ((4u + i) << 16) | (uint32_t)i));
}

// A workgroup's place: request, its tokens and this block's columns.
struct Item {
  int req, block;      // req < 0: none
  int start, qlen;     // the request's first token and its tokens within the step
  int shift;           // keys that the request's first token sees, minus 1
};

// Item x of the step: the requests' blocks of BM columns, one request after another.
// Uniform over the wave.
__device__ __forceinline__ Item find_item(const ChunkParams& p, int x) {
  const int lane = threadIdx.x & 63;
  int base = 0;
  for (int r0 = 0; r0 < p.R; r0 += 64) {
    const int r = min(r0 + lane, p.R - 1);
    const int q0 = p.query_start[r], q1 = p.query_start[r + 1], len = p.seq_lens[r];
    const int first = r ? q0 : 0;
    const int n = r0 + lane < p.R ? max(0, min(q1, p.N) - first) : 0;
    const int blocks = (n * p.G + BM - 1) / BM;
    int incl = blocks;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    const uint64_t hit = __builtin_amdgcn_ballot_w64(base + incl > x);
    if (hit) {
      const int l = __builtin_ctzll(hit);
      Item it;
      it.req = r0 + l;
      it.block = x - base - (__builtin_amdgcn_readlane(incl, l) - __builtin_amdgcn_readlane(blocks, l));
      it.start = __builtin_amdgcn_readlane(first, l);
      it.qlen = __builtin_amdgcn_readlane(n, l);
      // token i of the request sits at len - (q1 - q0) + (start + i - q0)
      it.shift = __builtin_amdgcn_readlane(len - (q1 - q0) + (first - q0), l);
      return it;
    }
    base += __builtin_amdgcn_readlane(incl, 63);
  }
  Item none{};
  none.req = -1;
  return none;
}
// Tiles that the block's last column sees.
__device__ __forceinline__ int item_tiles(const ChunkParams& p, const Item& it, int& kend) {
  const int last = (min(it.qlen * p.G, (it.block + 1) * BM) - 1) / p.G;
  kend = max(0, it.shift + last + 1);
  return (kend + BN - 1) / BN;
}
// Parts that its keys are split into, of as many tiles each (give or take one).
__device__ __forceinline__ int item_parts(const ChunkParams& p, int tiles) {
  return max(1, min(p.nsplit, (tiles + p.split_tiles - 1) / p.split_tiles));
}

template <int D>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 64 ? 3 : 2))) chunk_kernel(const ChunkParams p) {
  using GG = Geo<D>;
  constexpr int QB = GG::QB, SLOT = D + 8;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kv = blockIdx.y, part = blockIdx.z;
  const Item it = find_item(p, blockIdx.x);
  if (it.req < 0) return;
  int kend;
  const int tiles = item_tiles(p, it, kend), parts = item_parts(p, tiles);
  if (part >= parts) return;
  const int t0 = (int)((int64_t)part * tiles / parts), t1 = (int)((int64_t)(part + 1) * tiles / parts);

  // ---- the lane's column
  const int col = lane & 15, grp = lane >> 4;
  const int ncols = it.qlen * p.G;
  const int c0 = it.block * BM + 16 * w;                     // the wave's first column
  const int flat = min(c0 + col, ncols - 1);                 // columns past the end repeat the last one
  const int tok = flat / p.G, head = kv * p.G + flat - tok * p.G;
  const int lim = it.shift + tok + 1;                        // keys the column sees
  const bool live = c0 < ncols;
  const int lim_lo = __builtin_amdgcn_readfirstlane(lim), lim_hi = __builtin_amdgcn_readlane(lim, 15);
  half8 qh[QB];
  float qsum = 0.f;
  {
    const uint16_t* qrow = p.q + (int64_t)(it.start + tok) * p.q_seq_stride + (int64_t)head * p.q_head_stride;
#pragma unroll
    for (int j = 0; j < QB; ++j) qh[j] = *reinterpret_cast<const half8*>(qrow + min(32 * j + 8 * grp, D - 8));
#pragma unroll
    for (int j = 0; j < QB; ++j) {
      if (32 * j + 8 * grp >= D) qh[j] = half8{};            // head_dim 80, past its dims
#pragma unroll
      for (int e = 0; e < 8; ++e) qsum += (float)qh[j][e];
    }
    float a, b;
    swap16(qsum, a, b);
    qsum = a + b;
    swap32(qsum, a, b);
    qsum = a + b;
  }

  // ---- staging roles, as in prefill_mfma.hip
  const int kk = (tid & 15) + 16 * w, ku = (tid >> 4) & 3;   // K: key and quarter of its dims
  const int vk = lane & 31, vb = 2 * w + (lane >> 5);        // V: key pair and byte group
  const int vcol = 2 * vpos(2 * vk);
  const int esh = p.bt64 ? 3 : 2;
  const uint8_t* const table = reinterpret_cast<const uint8_t*>(p.block_tables) + (((int64_t)it.req * p.bt_stride) << esh);
  const uint32_t row_bytes = p.KV * SLOT, blk_bytes = row_bytes << p.block_shift;   // (the host checks that it fits)
  const int in_block = (1 << p.block_shift) - 1;
  struct Entries {
    uint32_t k, v;
  };
  // block-table entries of tile t's keys (low 32 bits; past the end the last key's)
  auto entries = [&](int t) -> Entries {
    const int key = min(t * BN + kk, kend - 1), k0 = min(t * BN + 2 * vk, kend - 1);
    return {*reinterpret_cast<const uint32_t*>(table + ((uint32_t)(key >> p.block_shift) << esh)),
            *reinterpret_cast<const uint32_t*>(table + ((uint32_t)(k0 >> p.block_shift) << esh))};
  };
  // A block holds 16 tokens or more, so a key pair lies in one, and a tile's first
  // key plus the lane's place in the tile never leaves it: slots past the sequence's
  // end are read where they are, and masked.
  const uint32_t koff = (uint32_t)(kk & in_block) * row_bytes + kv * SLOT;
  const uint32_t voff = (uint32_t)(2 * vk & in_block) * row_bytes + kv * SLOT + D / 2;
  uint2 kx[2][GG::KW], rl[2];
  uint32_t vx[2][GG::VW][2];
  uint32_t kxx[2], vxx[2][2];        // head_dim 80: the codes past dim 63
  auto load = [&](int t, const Entries& e, auto slot) {
    constexpr int sl = decltype(slot)::value;
    const uint8_t* const base = p.cache + (uint64_t)(uint32_t)(t * BN & in_block) * row_bytes;
    const uint8_t* const ks = base + ((uint64_t)e.k * blk_bytes + koff);
#pragma unroll
    for (int i = 0; i < GG::KW; ++i) kx[sl][i] = *reinterpret_cast<const uint2*>(ks + 8 * (GG::KW * ku + i));
    rl[sl] = *reinterpret_cast<const uint2*>(ks + D);
    const uint8_t* const v0 = base + ((uint64_t)e.v * blk_bytes + voff);
    const uint8_t* const v1 = v0 + row_bytes;
#pragma unroll
    for (int r = 0; r < GG::VW; ++r) {
      vx[sl][r][0] = *reinterpret_cast<const uint32_t*>(v0 + 4 * vb + 32 * r);
      vx[sl][r][1] = *reinterpret_cast<const uint32_t*>(v1 + 4 * vb + 32 * r);
    }
    if constexpr (GG::X) {
      kxx[sl] = *reinterpret_cast<const uint16_t*>(ks + 32 + 2 * ku);
      vxx[sl][0] = v0[32 + vb];
      vxx[sl][1] = v1[32 + vb];
    }
  };
  constexpr float kC = 1.4426950408889634f / (D == 64 ? 8.0f : D == 80 ? 8.94427190999916f : 11.313708498984761f);
  auto store = [&](auto slot) {
    constexpr int sl = decltype(slot)::value;
    uint8_t* Ks = smem + sl * GG::STAGE;
    uint8_t* Vs = Ks + GG::KBYTES;
    uint32_t kw[8 * GG::KW];
#pragma unroll
    for (int i = 0; i < GG::KW; ++i) {
      const uint32_t ws2[2] = {kx[sl][i].x, kx[sl][i].y};
#pragma unroll
      for (int hw = 0; hw < 2; ++hw) {
        const uint32_t lo = ws2[hw] & 0x0F0F0F0Fu, hi = (ws2[hw] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
        for (int b = 0; b < 4; ++b) kw[8 * i + 4 * hw + b] = nib_pair(lo, hi, b);
      }
    }
    uint4* kd = reinterpret_cast<uint4*>(Ks + kk * GG::KROW + ku * 32 * GG::KW);
#pragma unroll
    for (int i = 0; i < 2 * GG::KW; ++i) kd[i] = make_uint4(kw[4 * i], kw[4 * i + 1], kw[4 * i + 2], kw[4 * i + 3]);
    if (ku == 0) {
      const float kmin = h2f((uint16_t)(rl[sl].x & 0xffffu)), kstep = h2f((uint16_t)(rl[sl].x >> 16));
      const float vmin = h2f((uint16_t)(rl[sl].y & 0xffffu)), vstep = h2f((uint16_t)(rl[sl].y >> 16));
      *reinterpret_cast<float2*>(Ks + GG::ROFF + 8 * kk) = make_float2(__builtin_fmaf(8.0f, kstep, kmin) * kC, kstep * (kC * kCode));
      *reinterpret_cast<float2*>(Ks + GG::ROFF + 8 * (BN + kk)) = make_float2(__builtin_fmaf(8.0f, vstep, vmin), vstep);
    }
    if constexpr (GG::X) {
      const uint32_t lo = kxx[sl] & 0x0F0Fu, hi = (kxx[sl] >> 4) & 0x0F0Fu;
      *reinterpret_cast<uint2*>(Ks + kk * GG::KROW + 128 + 8 * ku) = make_uint2(nib_pair(lo, hi, 0), nib_pair(lo, hi, 1));
      const uint32_t b2 = vxx[sl][0] | (vxx[sl][1] << 16);
      *reinterpret_cast<uint32_t*>(Vs + (64 + 2 * vb) * GG::VROW + vcol) = centred(b2 & 0x000F000Fu);
      *reinterpret_cast<uint32_t*>(Vs + (65 + 2 * vb) * GG::VROW + vcol) = centred((b2 >> 4) & 0x000F000Fu);
    }
#pragma unroll
    for (int r = 0; r < GG::VW; ++r) {
      const uint32_t lo0 = vx[sl][r][0] & 0x0F0F0F0Fu, hi0 = (vx[sl][r][0] >> 4) & 0x0F0F0F0Fu;
      const uint32_t lo1 = vx[sl][r][1] & 0x0F0F0F0Fu, hi1 = (vx[sl][r][1] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int d = 8 * (vb + 8 * r) + 2 * b;
        *reinterpret_cast<uint32_t*>(Vs + d * GG::VROW + vcol) = nib_pair(lo0, lo1, b);
        *reinterpret_cast<uint32_t*>(Vs + (d + 1) * GG::VROW + vcol) = nib_pair(hi0, hi1, b);
      }
    }
  };

  floatx4 o[D / 16], ol[D / 16];     // sums of the weights' products and of their remainders'
#pragma unroll
  for (int c = 0; c < D / 16; ++c) o[c] = ol[c] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, msub = 0.f;   // the weights' reference; what is subtracted (0 while it is -inf)
  float l = 0.f, vt = 0.f;

  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  if constexpr (GG::X) {             // the K rows' dims 80 .. 95, in both stages
    if (tid < 128) {
      uint4* z = reinterpret_cast<uint4*>(smem + (tid >> 6) * GG::STAGE + (tid & 63) * GG::KROW + 160);
      z[0] = z[1] = make_uint4(0, 0, 0, 0);
    }
  }
  Entries en{};
  if (t0 < t1) {
    const Entries e0 = entries(t0), e1 = entries(min(t0 + 1, t1 - 1));
    en = entries(min(t0 + 2, t1 - 1));
    load(t0, e0, S0{});
    load(min(t0 + 1, t1 - 1), e1, S1{});
    store(S0{});
  }
  __syncthreads();
  auto iteration = [&](int t, auto slot) {
    constexpr int sl = decltype(slot)::value;
    using Next = std::integral_constant<int, sl ^ 1>;
    const Entries e3 = entries(min(t + 3, t1 - 1));
    load(min(t + 2, t1 - 1), en, slot);
    en = e3;
    const int kt0 = t * BN;
    if (live && kt0 < lim_hi) {      // uniform over the wave
      const uint8_t* Ks = smem + sl * GG::STAGE;
      const uint8_t* Vs = Ks + GG::KBYTES;
      half8 ka[4][QB];
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int j = 0; j < QB; ++j)
          ka[n][j] = *reinterpret_cast<const half8*>(Ks + (16 * n + col) * GG::KROW + (32 * j + 8 * grp) * 2);
      floatx4 s[4];
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        s[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka[n][0], qh[0], floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int j = 1; j < QB; ++j) s[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka[n][j], qh[j], s[n], 0, 0, 0);
      }
      float tmax = -INFINITY;
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const float4* kr = reinterpret_cast<const float4*>(Ks + GG::ROFF + 8 * (16 * n + 4 * grp));
        const float4 k01 = kr[0], k23 = kr[1];
        s[n][0] = __builtin_fmaf(s[n][0], k01.y, __builtin_fmaf(qsum, k01.x, -msub));
        s[n][1] = __builtin_fmaf(s[n][1], k01.w, __builtin_fmaf(qsum, k01.z, -msub));
        s[n][2] = __builtin_fmaf(s[n][2], k23.y, __builtin_fmaf(qsum, k23.x, -msub));
        s[n][3] = __builtin_fmaf(s[n][3], k23.w, __builtin_fmaf(qsum, k23.z, -msub));
      }
      const bool whole = kt0 + BN <= lim_lo;
      if (!whole) {                  // keys past a column's position: weight 0
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int i = 0; i < 4; ++i) s[n][i] = kt0 + 16 * n + 4 * grp + i < lim ? s[n][i] : -INFINITY;
      }
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) tmax = fmaxf(tmax, s[n][i]);
      // (scores are relative to msub)
      if (__builtin_amdgcn_ballot_w64(tmax > (m == -INFINITY ? -INFINITY : 0.f))) {
        float a, b;                  // over the four lane groups that hold the column
        swap16(tmax, a, b);
        tmax = fmaxf(a, b);
        swap32(tmax, a, b);
        tmax = fmaxf(a, b);
        const bool grow = tmax > (m == -INFINITY ? -INFINITY : 0.f);
        const float up = grow ? tmax + kMargin : 0.f;
        const float alpha = !grow ? 1.f : m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(-up);
        msub += up;
        m = grow ? msub : m;
        l *= alpha;
        vt *= alpha;
#pragma unroll
        for (int c = 0; c < D / 16; ++c) {
          o[c] *= alpha;
          ol[c] *= alpha;
        }
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int i = 0; i < 4; ++i) s[n][i] -= up;
      }
      half4 ph[4], pl[4];
      auto weights = [&](auto all) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          const float4* vr = reinterpret_cast<const float4*>(Ks + GG::ROFF + 8 * (BN + 16 * n + 4 * grp));
          const float4 v01 = vr[0], v23 = vr[1];
          float vmin[4] = {v01.x, v01.z, v23.x, v23.z}, vstep[4] = {v01.y, v01.w, v23.y, v23.w};
          if constexpr (!decltype(all)::value) {   // (nor may the rulers of keys past a position reach the sums)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const bool ok = kt0 + 16 * n + 4 * grp + i < lim;
              vmin[i] = ok ? vmin[i] : 0.f;
              vstep[i] = ok ? vstep[i] : 0.f;
            }
          }
#pragma unroll
          for (int i = 0; i < 4; i += 2) {
            float pr[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              pr[e] = __builtin_amdgcn_exp2f(s[n][i + e]);
              l += pr[e];
              vt = __builtin_fmaf(pr[e], vmin[i + e], vt);
            }
            // One rounding of the weight for both uses: through the empty asm, since the
            // compiler rounds product and conversion at once for one and apart for the
            // other, and where those differ the remainder is off by an fp16 ulp.
            uint32_t hw = __builtin_bit_cast(uint32_t, half2v{(_Float16)(pr[0] * vstep[i]), (_Float16)(pr[1] * vstep[i + 1])});
            asm("" : "+v"(hw));
            const half2v h2 = __builtin_bit_cast(half2v, hw);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              ph[n][i + e] = h2[e];
              pl[n][i + e] = (_Float16)(__builtin_fmaf(pr[e], vstep[i + e], -(float)h2[e]) * 2048.0f);
            }
          }
        }
      };
      if (whole) weights(std::true_type{});
      else weights(std::false_type{});
      half8 va[D / 16][2];
#pragma unroll
      for (int c = 0; c < D / 16; ++c)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
          va[c][hh] = *reinterpret_cast<const half8*>(Vs + (16 * c + col) * GG::VROW + (32 * hh + 8 * grp) * 2);
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const half8 bh = __builtin_shufflevector(ph[2 * hh], ph[2 * hh + 1], 0, 1, 2, 3, 4, 5, 6, 7);
        const half8 bl = __builtin_shufflevector(pl[2 * hh], pl[2 * hh + 1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int c = 0; c < D / 16; ++c) {
          o[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[c][hh], bh, o[c], 0, 0, 0);
          ol[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[c][hh], bl, ol[c], 0, 0, 0);
        }
      }
    }
    if (t + 1 < t1) store(Next{});
    __syncthreads();
  };
  for (int t = t0; t < t1; t += 2) {
    iteration(t, S0{});
    if (t + 1 < t1) iteration(t + 1, S1{});
  }

  if (!live) return;
  float a, b;
  swap16(l, a, b);
  l = a + b;
  swap32(l, a, b);
  l = a + b;
  swap16(vt, a, b);
  vt = a + b;
  swap32(vt, a, b);
  vt = a + b;
  if (c0 + col >= ncols) return;
  if (parts == 1) {
    const float rl1 = 1.0f / l;
    const int64_t at = (int64_t)(it.start + tok) * p.out_seq_stride + (int64_t)head * p.out_head_stride + 4 * grp;
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = lim > 0 ? __builtin_fmaf(__builtin_fmaf(ol[c][i], 0x1p-11f, o[c][i]), kCode, vt) * rl1 : 0.f;
      if (p.out_f16)
        *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(p.out) + at + 16 * c) =
            make_uint2((uint32_t)f2h(v[0]) | ((uint32_t)f2h(v[1]) << 16), (uint32_t)f2h(v[2]) | ((uint32_t)f2h(v[3]) << 16));
      else
        *reinterpret_cast<float4*>(reinterpret_cast<float*>(p.out) + at + 16 * c) = make_float4(v[0], v[1], v[2], v[3]);
    }
  } else {
    const int64_t row = (((int64_t)blockIdx.x * p.KV + kv) * p.nsplit + part) * BM + 16 * w + col;
#pragma unroll
    for (int c = 0; c < D / 16; ++c)
      *reinterpret_cast<float4*>(p.part_o + row * D + 16 * c + 4 * grp) =
          make_float4(__builtin_fmaf(__builtin_fmaf(ol[c][0], 0x1p-11f, o[c][0]), kCode, vt), __builtin_fmaf(__builtin_fmaf(ol[c][1], 0x1p-11f, o[c][1]), kCode, vt),
                      __builtin_fmaf(__builtin_fmaf(ol[c][2], 0x1p-11f, o[c][2]), kCode, vt), __builtin_fmaf(__builtin_fmaf(ol[c][3], 0x1p-11f, o[c][3]), kCode, vt));
    if (grp == 0) *reinterpret_cast<float2*>(p.part_ml + row * 2) = make_float2(m, l);
  }
}

// Joins the parts of split items: a quarter of the item's columns per workgroup,
// four dims per thread and step.
template <int D>
__global__ void __launch_bounds__(256) merge_kernel(const ChunkParams p) {
  const Item it = find_item(p, blockIdx.x);
  if (it.req < 0) return;
  int kend;
  const int tiles = item_tiles(p, it, kend), parts = item_parts(p, tiles);
  if (parts == 1) return;
  const int kv = blockIdx.y;
  constexpr int C = BM / 4, Q = D / 4;
  for (int e = threadIdx.x; e < C * Q; e += 256) {
    const int c = blockIdx.z * C + e / Q, d = (e % Q) * 4;
    const int flat = it.block * BM + c;
    if (flat >= it.qlen * p.G) return;
    const int tok = flat / p.G, head = kv * p.G + flat - tok * p.G;
    const int64_t row = ((int64_t)blockIdx.x * p.KV + kv) * p.nsplit * BM + c;
    float M = -INFINITY;
    for (int s = 0; s < parts; ++s) M = fmaxf(M, p.part_ml[(row + (int64_t)s * BM) * 2]);
    float L = 0.f, v[4] = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < parts; ++s) {
      const float2 ml = *reinterpret_cast<const float2*>(p.part_ml + (row + (int64_t)s * BM) * 2);
      const float4 o = *reinterpret_cast<const float4*>(p.part_o + (row + (int64_t)s * BM) * D + d);
      const float f = ml.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml.x - M);   // no key of the part: 0
      L = __builtin_fmaf(f, ml.y, L);
      v[0] = __builtin_fmaf(f, o.x, v[0]);
      v[1] = __builtin_fmaf(f, o.y, v[1]);
      v[2] = __builtin_fmaf(f, o.z, v[2]);
      v[3] = __builtin_fmaf(f, o.w, v[3]);
    }
    const float rL = 1.0f / L;
    const bool sees = it.shift + tok + 1 > 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = sees ? v[i] * rL : 0.f;
    const int64_t at = (int64_t)(it.start + tok) * p.out_seq_stride + (int64_t)head * p.out_head_stride + d;
    if (p.out_f16)
      *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(p.out) + at) =
          make_uint2((uint32_t)f2h(v[0]) | ((uint32_t)f2h(v[1]) << 16), (uint32_t)f2h(v[2]) | ((uint32_t)f2h(v[3]) << 16));
    else
      *reinterpret_cast<float4*>(reinterpret_cast<float*>(p.out) + at) = make_float4(v[0], v[1], v[2], v[3]);
  }
}

// Blocks of BM columns that N tokens of R requests fill at most.
int64_t items(int64_t N, int R, int G) { return N * G / BM + std::min<int64_t>(R, N); }

struct Split {
  int n, tiles;
};
// Parts that the keys are split into.  The workgroups run in rounds of as many as the
// CUs hold (three by LDS at head_dim 64, else two by registers; a full round leaves
// some waiting, so an eighth less).  A round takes a part's tiles and about three tiles'
// time before its first (the item's place, its block-table entries, its first codes,
// each after the other); a workgroup's partials and their merge cost a ninetieth of a
// tile's time on the whole chip.  Mostly within 15 % of the best of 1 to 32 parts for 1
// to 64 requests of 600 to 32000 tokens; us, one part, the rule's and the best: 500 tokens on
// 2000, 32 q / 4 KV heads, 64 dims 52.5, 41.3, 39.7; 512 on 32000, 32 / 8 heads, 128
// dims 1110, 585, 579.
// The partials are memory that the caller has to find in the middle of a step (they are
// allocated with the call), so a split has to give a twentieth at least and its partials
// stay within kPartBytes: by the time alone 8192 tokens of 4 requests at 131072 keys, 64 /
// 8 heads of 128 dims, took 783 MiB for 2.5 %, and of 8 requests at 16384, 32 / 8 heads,
// 264 MiB to be slower (4371 us, 4283 in one part).
constexpr int64_t kPartBytes = int64_t(128) << 20;
int64_t part_bytes(int64_t N, int R, int G, int KV, int D) { return items(N, R, G) * KV * BM * (D + 2) * 4; }

Split split_of(int64_t N, int R, int G, int KV, int D, int max_seq_len) {
  // (about as many workgroups as the requests fill: their last blocks are half full)
  const int64_t wgs = std::max<int64_t>(1, std::max<int64_t>(std::min<int64_t>(R, N), N * G / BM + R / 2) * KV);
  const int cus = device_cu_count();
  const int64_t slots = (int64_t)(cus > 0 ? cus : 256) * (D == 64 ? 21 : 14) / 8;   // (sizes asked for without a device: the MI355X)
  const int64_t part = std::max<int64_t>(1, part_bytes(N, R, G, KV, D));
  const int tiles = std::max(1, (int)(((int64_t)std::max(max_seq_len, 1) + BN - 1) / BN));
  const int most = (int)std::min<int64_t>(std::min(32, std::max(1, tiles / 2)), kPartBytes / part);
  int best = 1;
  int64_t one = 0, least = 0;
  for (int n = 1; n <= std::max(1, most); ++n) {
    const int64_t time = ((wgs * n + slots - 1) / slots) * ((tiles + n - 1) / n + 3) + (n > 1 ? wgs * n / 90 : 0);
    if (n == 1) one = least = time;
    if (time < least && 20 * time <= 19 * one) {
      least = time;
      best = n;
    }
  }
  return {best, (tiles + best - 1) / best};
}

template <int D>
int launch(const ChunkParams& p, int64_t nitems, hipStream_t stream) {
  static const bool lds_ok = [] {   // above 64 KB of LDS (head_dim 128) needs the attribute
    return hipFuncSetAttribute(reinterpret_cast<const void*>(chunk_kernel<D>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, Geo<D>::LDS) == hipSuccess;
  }();
  if (!lds_ok) return fail(SLMT_ERR_HIP, "chunk: could not grant the kernel its LDS");
  hipLaunchKernelGGL((chunk_kernel<D>), dim3((unsigned)nitems, p.KV, p.nsplit), dim3(256), Geo<D>::LDS, stream, p);
  if (int rc = check_launch("chunk")) return rc;
  if (p.nsplit == 1) return SLMT_OK;
  hipLaunchKernelGGL((merge_kernel<D>), dim3((unsigned)nitems, p.KV, 4), dim3(256), 0, stream, p);
  return check_launch("chunk merge");
}

}  // namespace chunk

int64_t chunk_workspace_bytes(int64_t N, int R, int H, int KV, int D, int max_seq_len) {
  const chunk::Split sp = chunk::split_of(N, R, H / KV, KV, D, max_seq_len);
  if (sp.n == 1) return 0;
  return chunk::part_bytes(N, R, H / KV, KV, D) * sp.n;
}

int launch_chunk(int D, ChunkParams& p, int max_seq_len, void* workspace, int64_t ws_bytes, hipStream_t stream) {
  const int64_t n = chunk::items(p.N, p.R, p.G);
  if (((int64_t)p.KV * (D + 8)) << p.block_shift >= (int64_t(1) << 31))
    return fail(SLMT_ERR_UNSUPPORTED, "chunk: a cache block of 2 GiB or more");
  if (n > 0x7fffffff || p.KV > 65535) return fail(SLMT_ERR_UNSUPPORTED, "chunk: too many query blocks for one launch");
  const chunk::Split sp = chunk::split_of(p.N, p.R, p.G, p.KV, D, max_seq_len);
  p.nsplit = sp.n;
  p.split_tiles = sp.tiles;
  if (sp.n > 1) {
    const int64_t need = chunk_workspace_bytes(p.N, p.R, p.G * p.KV, p.KV, D, max_seq_len);
    if (workspace == nullptr || ws_bytes < need)
      return fail(SLMT_ERR_INVALID, "chunk: workspace of " + std::to_string(need) + " bytes required, got " + std::to_string(ws_bytes));
    if (reinterpret_cast<uintptr_t>(workspace) & 15)
      return fail(SLMT_ERR_INVALID, "chunk: the workspace must be 16-byte aligned");
    p.part_o = reinterpret_cast<float*>(workspace);
    p.part_ml = p.part_o + n * p.KV * sp.n * chunk::BM * D;
  }
  if (D == 64) return chunk::launch<64>(p, n, stream);
  if (D == 80) return chunk::launch<80>(p, n, stream);
  return chunk::launch<128>(p, n, stream);
}

}  // namespace slmt
