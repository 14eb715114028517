// Causal prefill attention (declarations in prefill.hpp): scores, row
// statistics, then P.V with the probabilities formed on the way in.
//
// Reference semantics: encodeMaterializedPrefillBf16 (src/model/block_attn.zig:500-631),
// prefill_softmax_scaled_masked_bf16 (shaders/attention.metal:1463-1523),
// sigmoid_mul_pair_inplace_bf16 (shaders/elementwise.metal:88-99): bf16 scores,
// scale after the rounding, the row sum over 256 strided partial sums and a
// halving tree, bf16 probabilities, the gate after the bf16 context.
#include "attention.hpp"
#include "gemm_dev.hpp"
#include "prefill.hpp"

namespace {

using namespace prg;

constexpr float kLog2e = 1.4426950408889634f;
constexpr uint32_t kTileCols = 64;                     // cache slots per tile
constexpr uint32_t kRowBytes = kAttnHeadDim * 2;       // one K row or query row
constexpr int kScoreTokens = 32;                       // x 4 q heads = 128 rows per block
constexpr int kPvTokens = 16;                          // x 4 q heads = 64 rows per block
constexpr int kPvThreads = 512;                        // 4 consumer and 4 producer waves
static_assert(kAttnGroup == 4 && kAttnHeadDim == 256, "lane layouts");

__device__ inline uint32_t lds_addr(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const uint8_t*)p));
}
__device__ inline uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline uint32_t clamp_bytes(uint64_t n) { return n < 0xffffffffull ? static_cast<uint32_t>(n) : 0xffffffffu; }

// scores[z][h * T + t][c] = bf16(q . k_c). Block = 32 tokens of the four q
// heads of kv head z (wave = head) over `seg` tiles of 64 slots; the query
// fragments stay in registers and the K tiles come straight into two LDS
// buffers, so a tile is read from L2 once per 128 rows. Tiles past every row's
// last visible slot are skipped. K is the A operand, so a lane holds four
// consecutive columns of one row; they leave through a wave's own LDS rows as
// 128-byte row segments. Same products and k order per score as a 16x16x32
// tiling with the operands exchanged. Bound by the score writes (2.8 TB/s at a
// long context; matrix cores 30% busy). 1600 tokens 47 -> 25 us, 1021 tokens
// after 15003 357 -> 180-196 us (a 128 x 128 GEMM before).
__global__ __launch_bounds__(256) void attn_prefill_scores_kernel(const uint16_t* __restrict__ q,
                                                                  const uint16_t* __restrict__ cache_k,
                                                                  uint16_t* __restrict__ scores, uint32_t T,
                                                                  uint32_t prefix, uint32_t stride, uint32_t ld,
                                                                  uint32_t seg) {
  __shared__ __attribute__((aligned(1024))) uint4 sK[2][kTileCols][32];
  __shared__ uint4 sS[4][32][8];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = uniform(tid >> 6);
  const int fr = lane & 15, fc = lane >> 4;
  const uint32_t z = blockIdx.z, t0 = blockIdx.x * kScoreTokens;
  const uint32_t t_last = min(T - 1, t0 + kScoreTokens - 1);
  const uint32_t tiles = (prefix + t_last) / kTileCols + 1;
  const uint32_t first = blockIdx.y * seg, last = min(tiles, first + seg);
  if (first >= last) return;

  // Queries: 32 rows of this wave's head into sK (free until the first tile),
  // 16-byte chunk c of row r at c ^ (r & 15); rows past T read as zero.
  const uint32_t lr = lane >> 5, lp = lane & 31;
  {
    const uint32_t head = z * kAttnGroup + wave;
    const uint64_t row_bytes = static_cast<uint64_t>(kAttnQHeads) * kRowBytes;
    const __amdgpu_buffer_rsrc_t rq = buffer_rsrc(q + (static_cast<uint64_t>(t0) * kAttnQHeads + head) * kAttnHeadDim,
                                                  static_cast<uint32_t>((t_last - t0) * row_bytes + kRowBytes));
    const uint32_t base = lds_addr(sK) + wave * 32 * kRowBytes;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t r = 2 * i + lr;
      lds_load16(rq, uniform(base + i * 1024), static_cast<uint32_t>(r * row_bytes) + (lp ^ (r & 15)) * 16, 0);
    }
  }
  PRG_WAIT_VMCNT(0);
  __syncthreads();
  bf16x8 qf[2][8];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      qf[x][i] = __builtin_bit_cast(bf16x8, (&sK[0][0][0])[(wave * 32 + 16 * x + fr) * 32 + ((4 * i + fc) ^ fr)]);
  __syncthreads();

  // K tile: 64 rows of 512 bytes; wave w copies rows 16 w .. +15. Rows past
  // the cache read as zero; rows past the prompt give columns nobody reads.
  auto issue = [&](uint32_t tile, uint32_t buf) {
    const uint32_t c0 = tile * kTileCols;
    const __amdgpu_buffer_rsrc_t rk =
        buffer_rsrc(cache_k + (static_cast<uint64_t>(z) * stride + c0) * kAttnHeadDim, min(kTileCols, stride - c0) * kRowBytes);
    const uint32_t base = lds_addr(&sK[0][0][0]) + (buf * kTileCols + 16 * wave) * kRowBytes;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t r = 2 * i + lr;
      lds_load16(rk, uniform(base + i * 1024), (16 * wave + r) * kRowBytes + (lp ^ r) * 16, 0);
    }
  };
  issue(first, 0);
  PRG_WAIT_VMCNT(0);
  __syncthreads();
  uint16_t* srow = scores + (static_cast<uint64_t>(z) * kAttnGroup + wave) * T * ld;
  for (uint32_t tile = first; tile < last; ++tile) {
    const uint32_t buf = (tile - first) & 1;
    issue(tile + 1 < last ? tile + 1 : tile, buf ^ 1);  // the last copy is never read
    f32x4 acc[2][4];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[x][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      bf16x8 kf[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) kf[j] = __builtin_bit_cast(bf16x8, sK[buf][16 * j + fr][(4 * i + fc) ^ fr]);
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[x][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[j], qf[x][i], acc[x][j], 0, 0, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 16, 0);
    // lane: row 16 x + fr, columns 16 j + 4 fc .. +3
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t ch = (2 * j + (fc >> 1)) ^ (fr & 7);
        *(reinterpret_cast<uint2*>(&sS[wave][16 * x + fr][ch]) + (fc & 1)) =
            make_uint2(pack_bf16(acc[x][j][0], acc[x][j][1]), pack_bf16(acc[x][j][2], acc[x][j][3]));
      }
    PRG_WAIT_VMCNT(0);  // the next tile has landed (and the previous tile's stores)
    // The wave's lanes exchange the tile through its own rows of sS: in order in
    // the LDS pipe, and kept so by the compiler.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t r = 8 * i + (lane >> 3), ch = lane & 7;
      const uint4 v = sS[wave][r][ch ^ (r & 7)];
      if (t0 + r < T)
        *reinterpret_cast<uint4*>(srow + static_cast<uint64_t>(t0 + r) * ld + tile * kTileCols + 8 * ch) = v;
    }
    __syncthreads();
  }
  PRG_WAIT_VMCNT(0);
}

// e^(x - m) as the reference forms it (x's scaling and the difference may be one
// fma, the same value for a power of two such as the model's 1/16) on v_exp_f32:
// results below 2^-126 come out as zero. The row sums take it as it is: they are
// at least 1, the term of the maximum. Probabilities below 2^-126 exist in bf16
// and count where the values are large: prob_small.
__device__ inline float prob_exp(float x, float m) {
  return __builtin_amdgcn_exp2f(__fmul_rn(__fsub_rn(x, m), kLog2e));
}
// e^(x - m) / sum with subnormal exponentials and quotients.
__device__ inline float prob_small(float x, float m, float sum) {
  return exp2f(__fmul_rn(__fsub_rn(x, m), kLog2e)) / sum;
}
constexpr float kProbSmall = 0x1p-100f;

// stats[row] = (max, sum of e^(x - max)) over the visible columns of a score
// row, x = float(score) * scale. One wave per row; lane l holds columns
// 256 n + 4 l .. +3, i.e. the reference's 256 strided partial sums 4 l .. 4 l + 3
// (each summed in column order), which then combine in its halving tree's
// pairs: t with t + 128 is lane l with l + 32, t + 64 lane l + 16, and so on
// down to the lane's own four. The first NG groups stay in registers (packed:
// their f32 values took 256 registers and a wave per SIMD, 260 us) between the
// two passes; later ones are read again. Bound by reading the scores once
// (3.2 TB/s at a long context); the NG groups are loaded whatever the row's length,
// so a cold prompt reads the masked half of its rows too (82 MB at 1600 tokens).
// 1600 tokens 16 us, 1021 after 15003 160-179 us, where the softmax that rewrote
// the row took 49 and 727 us.
template <int NG>
__global__ __launch_bounds__(256) void attn_prefill_stats_kernel(const uint16_t* __restrict__ scores,
                                                                 float2* __restrict__ stats, uint32_t ld, uint32_t T,
                                                                 uint32_t rows, uint32_t prefix, float scale) {
  const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
  if (row >= rows) return;  // whole wave: no barrier below
  const uint16_t* s = scores + static_cast<uint64_t>(row) * ld;
  const uint32_t vis = prefix + row % T;
  const uint32_t groups = vis / 256 + 1, full = (vis + 1) / 256;  // groups with any / only visible columns
  auto load = [&](uint32_t n) -> uint2 {  // ld % 64 == 0; columns past the row's end repeat its last four
    return *reinterpret_cast<const uint2*>(s + min(256 * n + 4 * l, ld - 4));
  };
  auto value = [&](const uint2& v, int e) {
    const uint32_t w = e < 2 ? v.x : v.y;
    return __fmul_rn((e & 1) ? bf_hi(w) : bf_lo(w), scale);
  };
  uint2 held[NG];
#pragma unroll
  for (int n = 0; n < NG; ++n) held[n] = load(n);
  float m = -INFINITY;
  auto take_max = [&](const uint2& v, uint32_t n) {
    if (n < full) {
#pragma unroll
      for (int e = 0; e < 4; ++e) m = fmaxf(m, value(v, e));
    } else if (n < groups) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (256 * n + 4 * l + e <= vis) m = fmaxf(m, value(v, e));
    }
  };
#pragma unroll
  for (int n = 0; n < NG; ++n) take_max(held[n], n);
  for (uint32_t n = NG; n < groups; ++n) take_max(load(n), n);
  m = wave_max(m);
  // keep the scores packed between the passes (not their 128 f32 values)
#pragma unroll
  for (int n = 0; n < NG; ++n) asm("" : "+v"(held[n].x), "+v"(held[n].y));
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
  auto take_sum = [&](const uint2& v, uint32_t n) {
    if (n < full) {
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] = __fadd_rn(sum[e], prob_exp(value(v, e), m));
    } else if (n < groups) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p = prob_exp(value(v, e), m);
        sum[e] = __fadd_rn(sum[e], 256 * n + 4 * l + e <= vis ? p : 0.0f);
      }
    }
  };
#pragma unroll
  for (int n = 0; n < NG; ++n) take_sum(held[n], n);
  for (uint32_t n = NG; n < groups; ++n) take_sum(load(n), n);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float a = sum[e], b = a;
    swap32(a, b);
    a = __fadd_rn(a, b);  // t and t + 128
    b = a;
    swap16(a, b);
    a = __fadd_rn(a, b);  // (t, t + 128) and (t + 64, t + 192)
    a = __fadd_rn(a, dpp_f<0x108>(a));  // t + 32: row_shl:8
    a = __fadd_rn(a, dpp_f<0x104>(a));  // t + 16
    a = __fadd_rn(a, dpp_f<0x102>(a));  // t + 8
    sum[e] = __fadd_rn(a, dpp_f<0x101>(a));  // t + 4
  }
  const float total = __fadd_rn(__fadd_rn(sum[0], sum[2]), __fadd_rn(sum[1], sum[3]));
  if (l == 0) stats[row] = make_float2(m, total == 0.0f ? 1.0f : total);
}

// out = bf16(bf16(P.V) * sigmoid(gate)), P = bf16(e^(x - max) / sum). Block =
// 16 tokens of the four q heads of kv head z (64 rows) x 256 / DS value dims,
// tiles of 64 slots, one barrier per tile. Loads return in order within a
// wave, so the two streams have waves of their own: four producer waves keep
// kAhead tiles of scores in flight (HBM), turn the next tile's into
// probabilities (two rows per thread, their statistics in registers) and write
// them to LDS; four consumer waves (2 x 32 rows, 2 x half of the dims) copy the V
// tiles straight to LDS kBufs - 1 tiles ahead and run the matrix instructions,
// in slot order from 0, so a row's bits do not depend on the chunk it is
// computed in. A tile takes about 2000 clocks (counters, long context): a producer
// wave's ~240 VALU operations take 960, the matrix cores are busy for 510 and LDS
// reads and stores for 380 beside the V copies; behind one barrier per tile they
// mostly follow one another.
// 1600 tokens 57 -> 46 us, 1021 after 15003 323 -> 250-290 us (a GEMM over
// stored probabilities before).
template <int DS>
__global__ __launch_bounds__(kPvThreads) void attn_prefill_pv_kernel(const uint16_t* __restrict__ scores,
                                                                     const float2* __restrict__ stats,
                                                                     const uint16_t* __restrict__ cache_v,
                                                                     const uint16_t* __restrict__ gate,
                                                                     uint16_t* __restrict__ out, uint32_t T,
                                                                     uint32_t prefix, uint32_t stride, uint32_t ld,
                                                                     float scale) {
  constexpr int kDims = kAttnHeadDim / DS, DB = kDims / 32;  // dims per block, 16-dim blocks per consumer wave
  constexpr int kCopies = kDims / 32;                        // V copies per consumer wave and tile
  constexpr int kBufs = 4, kAhead = 4;
  __shared__ __attribute__((aligned(1024))) uint4 sV[kBufs][kDims][8];
  __shared__ uint4 sP[2][64][8];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = uniform(tid >> 6);
  const uint32_t z = blockIdx.y, d0 = blockIdx.z * kDims;
  const uint32_t t0 = (gridDim.x - 1 - blockIdx.x) * kPvTokens;  // the longest rows first
  const uint32_t t_last = min(T - 1, t0 + kPvTokens - 1);
  const uint32_t L = prefix + T, tiles = (prefix + t_last) / kTileCols + 1;
  auto clampt = [&](uint32_t k) { return k < tiles ? k : tiles - 1; };

  if (wave >= 4) {
    // thread -> rows pr, pr + 32 (head row / 16, token t0 + row % 16), columns 8 pc .. +7
    const uint32_t pr = (tid & 255) >> 3, pc = tid & 7;
    const uint16_t* sp[2];
    float pm[2], pd[2], pinv[2];
    uint32_t pvis[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t r = pr + 32 * i, t = min(T - 1, t0 + (r & 15));
      const uint64_t row = (static_cast<uint64_t>(z) * kAttnGroup + (r >> 4)) * T + t;
      sp[i] = scores + row * ld + 8 * pc;
      const float2 st = stats[row];
      pm[i] = st.x;
      pd[i] = st.y;
      pinv[i] = 1.0f / st.y;
      pvis[i] = prefix + t;
    }
    uint4 ss[kAhead][2];
    auto load_s = [&](int set, uint32_t tile) {
#pragma unroll
      for (int i = 0; i < 2; ++i) ss[set][i] = *reinterpret_cast<const uint4*>(sp[i] + tile * kTileCols);
    };
    // A tile's probabilities, on straight-line code to the LDS store; where an
    // exponential or the quotient's residual may underflow (a score 69 or more
    // under the maximum) the plain division writes them again. A branch before
    // the store keeps one row's chain from overlapping the other's (9 tokens after
    // 15000: 165 us). Blocks with a part of the value dims are bound by this chain,
    // so there the columns past a row's token are zeroed the same way, in the one or
    // two tiles that have any: 141 us, against 147 with the masks in line and 143
    // with them and without the test for small exponentials. Blocks with all dims
    // lose by that (512 after 4000: 111 -> 115 us) and mask in line; the test costs
    // them 0-1% (1600 tokens 97.1 -> 97.2 us, 1021 after 15003 571 -> 579).
    auto probs = [&](int set, uint32_t tile) {
      const uint32_t c0 = tile * kTileCols + 8 * pc;
      auto score = [&](int i, int e) {
        const uint32_t w = (&ss[set][i].x)[e >> 1];
        return __fmul_rn((e & 1) ? bf_hi(w) : bf_lo(w), scale);
      };
      auto pack = [](const float* p) {
        return make_uint4(pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3]), pack_bf16(p[4], p[5]), pack_bf16(p[6], p[7]));
      };
      auto put = [&](int i, uint4 v, bool mask) {
        const uint32_t r = pr + 32 * i;
        if (mask) {
          uint32_t* w = &v.x;
#pragma unroll
          for (uint32_t e = 0; e < 4; ++e)
            w[e] &= (c0 + 2 * e <= pvis[i] ? 0xffffu : 0u) | (c0 + 2 * e + 1 <= pvis[i] ? 0xffff0000u : 0u);
        }
        sP[tile & 1][r][pc ^ (r & 7)] = v;
      };
      uint4 v[2];
      float least = 1.0f;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float ex = prob_exp(score(i, e), pm[i]);
          least = fminf(least, ex);
          // ex / sum: the quotient by the rounded reciprocal and one residual step
          // (Markstein). The residual is exact from kProbSmall up; 4e8 random pairs
          // of ex in [2^-100, 1] and sums to 2^17 gave the rounded quotient each time
          const float qt = __fmul_rn(ex, pinv[i]);
          p[e] = __fmaf_rn(__fmaf_rn(-qt, pd[i], ex), pinv[i], qt);
          if (DS == 1) p[e] = c0 + e <= pvis[i] ? p[e] : 0.0f;
        }
        v[i] = pack(p);
        put(i, v[i], false);
      }
      const bool small = least < kProbSmall;
      // the tile past the last goes into a buffer nobody reads
      const bool diag = DS != 1 && tile < tiles && tile * kTileCols + kTileCols - 1 > prefix + t0;
      if (__builtin_expect(small | diag, 0)) {
        if (diag) {
#pragma unroll
          for (int i = 0; i < 2; ++i) put(i, v[i], true);
        }
        if (small) {
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            float p[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) p[e] = prob_small(score(i, e), pm[i], pd[i]);
            put(i, pack(p), true);
          }
        }
      }
    };
#pragma unroll
    for (int k = 0; k < kAhead; ++k) load_s(k, clampt(k));
    probs(0, 0);
    load_s(0, clampt(kAhead));
    __syncthreads();
    // Straight-line rounds of kAhead tiles; the tile past the last goes into
    // the buffer nobody reads again.
    uint32_t k = 0;
    for (; k + kAhead <= tiles; k += kAhead) {
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        probs((u + 1) % kAhead, k + u + 1);
        load_s((u + 1) % kAhead, clampt(k + u + 1 + kAhead));
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      if (k + u >= tiles) break;
      probs((u + 1) % kAhead, k + u + 1);
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
    }
    return;
  }

  const int wm = wave >> 1, wn = wave & 1;
  const int fr = lane & 15, fc = lane >> 4;
  // V tile: kDims rows of 128 bytes, chunk c of row d at c ^ (d & 7); one copy
  // takes 8 rows. Slots past the cache row's end belong to the next row (or
  // read as zero): like every slot in [L, ..) they are masked below.
  const uint16_t* vbase = cache_v + (static_cast<uint64_t>(z) * kAttnHeadDim + d0) * stride;
  const uint32_t voff = (lane >> 3) * stride * 2 + ((lane & 7) ^ (lane >> 3)) * 16;
  auto issue = [&](uint32_t tile, uint32_t buf) {
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
      const uint32_t d = (wave * kCopies + i) * 8;
      const uint64_t first = static_cast<uint64_t>(d) * stride + tile * kTileCols;
      const __amdgpu_buffer_rsrc_t rv =
          buffer_rsrc(vbase + first, clamp_bytes((static_cast<uint64_t>(kDims) * stride - first) * 2));
      lds_load16(rv, uniform(lds_addr(&sV[0][0][0]) + (buf * kDims + d) * 128), voff, 0);
    }
  };
  f32x4 acc[2][DB];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int j = 0; j < DB; ++j) acc[x][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto consume = [&](uint32_t tile, uint32_t buf, bool tail) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      bf16x8 pf[2], vf[DB];
#pragma unroll
      for (int x = 0; x < 2; ++x) pf[x] = __builtin_bit_cast(bf16x8, sP[tile & 1][32 * wm + 16 * x + fr][(4 * i + fc) ^ (fr & 7)]);
#pragma unroll
      for (int j = 0; j < DB; ++j) {
        uint4 v = sV[buf][wn * (kDims / 2) + 16 * j + fr][(4 * i + fc) ^ (fr & 7)];
        if (tail) {  // slots from L on may hold anything: zero them
          const uint32_t c0 = tile * kTileCols + 8 * (4 * i + fc);
          uint32_t* w = &v.x;
#pragma unroll
          for (uint32_t e = 0; e < 4; ++e)
            w[e] &= (c0 + 2 * e < L ? 0xffffu : 0u) | (c0 + 2 * e + 1 < L ? 0xffff0000u : 0u);
        }
        vf[j] = __builtin_bit_cast(bf16x8, v);
      }
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int j = 0; j < DB; ++j) acc[x][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf[x], vf[j], acc[x][j], 0, 0, 0);
    }
  };
#pragma unroll
  for (int i = 0; i < kBufs - 1; ++i) issue(clampt(i), i);
  PRG_WAIT_VMCNT(kCopies * (kBufs - 2));
  __syncthreads();
  for (uint32_t k = 0; k < tiles; ++k) {
    issue(clampt(k + kBufs - 1), (k + kBufs - 1) % kBufs);  // the buffer tile k - 1 was read from
    if ((k + 1) * kTileCols > L)
      consume(k, k % kBufs, true);
    else
      consume(k, k % kBufs, false);
    PRG_WAIT_VMCNT(kCopies * (kBufs - 2));  // tile k + 1 has landed
    __syncthreads();
  }
  PRG_WAIT_VMCNT(0);

  // lane: rows 32 wm + 16 x + 4 fc + r, dims 16 j + fr of the wave's half
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const uint32_t h = z * kAttnGroup + 2 * wm + x;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t t = t0 + 4 * fc + r;
      if (t >= T) continue;
      const uint64_t o = (static_cast<uint64_t>(t) * kAttnQHeads + h) * kAttnHeadDim + d0 + wn * (kDims / 2) + fr;
#pragma unroll
      for (int j = 0; j < DB; ++j) out[o + 16 * j] = f2bf(round_bf(acc[x][j][r]) * sigmoid(bf2f(gate[o + 16 * j])));
    }
  }
}

}  // namespace

namespace prg {

// Per row: ld scores, then (max, sum) of every row as float2 behind the score block.
size_t attn_prefill_scores_elems(uint32_t T, uint32_t prefix) {
  const size_t L = static_cast<size_t>(prefix) + T, ld = (L + 63) / 64 * 64;
  return static_cast<size_t>(kAttnQHeads) * T * (ld + kAttnStatElems);
}

int launch_attn_prefill(hipStream_t s, const uint16_t* q, const uint16_t* cache_k, const uint16_t* cache_v,
                        const uint16_t* gate, uint16_t* out, uint16_t* scores, size_t scores_cap, uint32_t T,
                        uint32_t prefix, uint32_t stride, float scale) {
  // scores_cap: bf16 elements the workspace holds
  if (attn_prefill_scores_elems(T, prefix) > scores_cap)
    return set_error(PRG_ERR_INVALID_ARG, "attention prefill: %u tokens after %u need %zu score elements, %zu held",
                     T, prefix, attn_prefill_scores_elems(T, prefix), scores_cap);
  for (const void* p : {static_cast<const void*>(q), static_cast<const void*>(cache_k),
                        static_cast<const void*>(cache_v), static_cast<const void*>(scores)})
    PRG_CHECK_ARG(reinterpret_cast<uintptr_t>(p) % 16 == 0, "attn_prefill: q, the caches and scores must be 16-byte aligned");
  const uint32_t L = prefix + T, ld = (L + 63) / 64 * 64, rows = kAttnQHeads * T;
  float2* stats = reinterpret_cast<float2*>(scores + static_cast<size_t>(rows) * ld);
  const uint32_t tiles = ld / kTileCols, gx = (T + kScoreTokens - 1) / kScoreTokens;
  // 64-slot tiles per block: more amortise the block's query load, fewer fill
  // the chip (two blocks per CU) on short prompts
  const uint64_t work = static_cast<uint64_t>(gx) * kAttnKvHeads * tiles;
  const uint32_t seg = static_cast<uint32_t>(work < 2048 ? 2 : work > 16384 ? 16 : work / 1024);
  hipLaunchKernelGGL(attn_prefill_scores_kernel, dim3(gx, (tiles + seg - 1) / seg, kAttnKvHeads), dim3(256), 0, s, q,
                     cache_k, scores, T, prefix, stride, ld, seg);
  PRG_CHECK_LAUNCH("attn_prefill.scores");
  const dim3 sgrid((rows + 3) / 4);
  if (L <= 2048)
    hipLaunchKernelGGL(attn_prefill_stats_kernel<8>, sgrid, dim3(256), 0, s, scores, stats, ld, T, rows, prefix, scale);
  else if (L <= 6144)
    hipLaunchKernelGGL(attn_prefill_stats_kernel<24>, sgrid, dim3(256), 0, s, scores, stats, ld, T, rows, prefix, scale);
  else
    hipLaunchKernelGGL(attn_prefill_stats_kernel<64>, sgrid, dim3(256), 0, s, scores, stats, ld, T, rows, prefix, scale);
  PRG_CHECK_LAUNCH("attn_prefill.stats");
  const uint32_t px = (T + kPvTokens - 1) / kPvTokens;
  // Few row blocks leave CUs idle: split the value dims over 2 or 4 blocks,
  // each forming the probabilities again. Whole op, 1 / 2 / 4 splits: 2048
  // tokens after 2048 307 / 316 / 377 us; 600 after 3000 121 / 126 / 142;
  // 300 after 0 34 / 30 / 32; 100 after 4001 88 / 70 / 65; 9 after 15000
  // 231 / 173 / 148.
  const int ds = px >= 32 ? 1 : px >= 16 ? 2 : 4;
  const dim3 grid(px, kAttnKvHeads, ds);
  if (ds == 1)
    hipLaunchKernelGGL(attn_prefill_pv_kernel<1>, grid, dim3(kPvThreads), 0, s, scores, stats, cache_v, gate, out, T, prefix, stride, ld, scale);
  else if (ds == 2)
    hipLaunchKernelGGL(attn_prefill_pv_kernel<2>, grid, dim3(kPvThreads), 0, s, scores, stats, cache_v, gate, out, T, prefix, stride, ld, scale);
  else
    hipLaunchKernelGGL(attn_prefill_pv_kernel<4>, grid, dim3(kPvThreads), 0, s, scores, stats, cache_v, gate, out, T, prefix, stride, ld, scale);
  PRG_CHECK_LAUNCH("attn_prefill.values");
  return PRG_OK;
}

}  // namespace prg
