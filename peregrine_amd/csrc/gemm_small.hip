// Prompt GEMM for few activation rows (a chat turn, the tail chunk of a
// prompt): declarations in gemm.hpp, the large-M kernels in gemm.hip.
#include "gemm.hpp"
#include "gemm_dev.hpp"

namespace {

using namespace prg;

constexpr int kSmallThreads = 512;  // 4 consumer waves, 4 producer waves

// Q4 GEMM for few activation rows. The 192 / 256-row kernel computes a whole
// row tile whatever M is and covers N = 4096 with 32 blocks, so at 43 rows a
// K = 12288 projection took 162 us for 28 MB of weights. Here a block takes 16
// TN weight rows (one block per CU at N = 4096, TN = 1) and up to 64 MW
// activation rows, and its waves are split by role, because loads return in
// order within a wave and the weights must be fetched much further ahead (HBM)
// than the activations (L2):
//   - four producer waves keep D stages of KC k of packed weights in flight in
//     registers, dequantise one stage ahead (dequant_word, the values of every
//     other prompt GEMM) and write it to LDS in matrix-operand order;
//   - four consumer waves own 16 (MW = 2: 32) activation rows each, copied
//     straight to LDS R - 1 stages ahead in whole 128-byte lines (a lane per
//     row, as the matrix operand wants it, is one 16-byte request per lane and
//     ran at a quarter of this rate), and run the matrix instructions.
// One barrier per stage. Per output element the instructions are those of
// gemm_q4_kernel in the same k order (16x16x32 blocks of k 32 i .. +31, one
// accumulator), so a row has the same bits whichever kernel a call takes.
// What bounds it (gate/up at 43 rows, counters): a stage takes about 2200 clocks,
// of which a producer wave issues VALU operations for 880 (dequantisation, about
// 31 per 8 values), LDS is busy for 960 (every consumer wave reads all of the
// dequantised weights) and the matrix cores for 380. Behind one barrier per stage
// they follow one another instead of overlapping, on 192 of 256 CUs. Measured at 43
// rows (us, before -> now, 4.5 Q4 bits from HBM): gate/up 12288 x 2 x 4096
// 57 -> 33; down 4096 x 12288 162 -> 28; 12288 x 4096 55 -> 21; 4096 x 4096
// 54 -> 13.
// TN: 16-row weight tiles per block; MW: 16-row activation blocks per consumer
// wave; KC: k per stage; D: weight stages in flight; R: activation stages.
template <int EPI, int TN, int MW, int KC, int D, int R>
__global__ __launch_bounds__(kSmallThreads) void gemm_small_kernel(const GemmArgs g) {
  constexpr bool kPair = EPI == kGemmSiluPair;
  static_assert(!kPair || TN % 2 == 0, "gate and up tiles come in pairs");
  static_assert(KC == 256 || KC == 128, "k per stage");
  constexpr int kTileN = 16 * (kPair ? TN / 2 : TN);  // output columns per block
  constexpr int KS = KC / 32;                         // matrix instructions per stage along k
  constexpr int kSwz = 16 / KS;
  constexpr int kUnits = TN * 16 * KS;                // 16-byte weight units per stage
  constexpr int UPT = kUnits >= 256 ? kUnits / 256 : 1;
  constexpr int WPU = kUnits >= 256 ? 4 : 2;          // words of a unit one producer thread takes
  static_assert(kUnits == 128 || kUnits % 256 == 0, "units per producer thread");
  constexpr int kChunks = KC / 8;                     // 16-byte chunks of an activation row per stage
  // weight fragments of a stage in matrix-operand order [k step][tile][lane], lane j of a
  // 16-lane group at j ^ (k step * kSwz), so that the writes of 16 lanes (16 / KS rows of KS
  // k steps each in the MLX layout) cover all banks; activations [wave][16-row block][stage][row][chunk],
  // chunk c of row r at c ^ r
  __shared__ __attribute__((aligned(1024))) uint4 sA[4][MW][R][16][kChunks];
  __shared__ uint4 sB[2][KS][TN][kWave];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t tiles_m = (g.M + 64 * MW - 1) / (64 * MW);
  uint32_t tm, tn;
  {
    const uint32_t T = gridDim.x, b = blockIdx.x, x = b % 8, q = T / 8, r = T % 8;
    const uint32_t L = x * q + (x < r ? x : r) + b / 8;
    tm = L % tiles_m;
    tn = L / tiles_m;
  }
  uint32_t seg = 0;
  if constexpr (!kPair) {
#pragma unroll
    for (int i = 1; i < kGemmMaxSegs; ++i)
      if (i < static_cast<int>(g.nq) && tn >= g.q[i].tile0) seg = i;
  }
  const uint32_t N = g.q[seg].n, K = g.K, stages = K / KC;
  const uint32_t m0 = tm * 64 * MW, n0 = (tn - g.q[seg].tile0) * kTileN;
  auto clampk = [&](uint32_t k) { return k < stages ? k : stages - 1; };

  if (wave >= 4) {
    // ------------------------------------------------ producers ----
    const int p = tid - 256;
    __amdgpu_buffer_rsrc_t wr[UPT], sr[UPT], br[UPT];
    uint32_t wo[UPT], mo[UPT];
    uint32_t dst[UPT];  // uint4 index of the unit's first word in a stage
#pragma unroll
    for (int i = 0; i < UPT; ++i) {
      const uint32_t u = WPU == 2 ? p >> 1 : p + 256 * i, h = WPU == 2 ? p & 1 : 0;
      const uint32_t t = __builtin_amdgcn_readfirstlane(u / (16 * KS));  // a wave's units lie in one tile
      const uint32_t q = u % KS, j = (u / KS) & 15;  // k step of the stage and row: memory order
      const GemmQ4& Q = g.q[kPair ? (t >= TN / 2 ? 1 : 0) : seg];
      const uint32_t n = n0 + 16 * (kPair ? t % (TN / 2) : t) + j;
      const uint32_t row = n < N ? n : N - 1;  // rows past N are computed, never stored
      const uint32_t wbytes = static_cast<uint32_t>(static_cast<uint64_t>(N) * K / 2);
      wr[i] = buffer_rsrc(Q.w, wbytes);
      sr[i] = buffer_rsrc(Q.s, wbytes / 16);
      br[i] = buffer_rsrc(Q.b, wbytes / 16);
      wo[i] = row * (K / 2) + 16 * q + 8 * h;
      mo[i] = (row * (K / 64) + (q >> 1)) * 2;
      dst[i] = (q * TN + t) * kWave + (j ^ (q * kSwz)) + 32 * h;
    }
    constexpr uint32_t kWStep = KC / 2, kMStep = KC / 32;  // bytes per stage
    uint32_t w[D][UPT][WPU];
    uint32_t sc[D][UPT], bi[D][UPT];
    auto load = [&](int r, uint32_t ks) {
#pragma unroll
      for (int i = 0; i < UPT; ++i) {
        if constexpr (WPU == 4) {
          const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(wr[i], wo[i], ks * kWStep, 0);
          w[r][i][0] = v.x; w[r][i][1] = v.y; w[r][i][2] = v.z; w[r][i][3] = v.w;
        } else {
          const auto v = __builtin_amdgcn_raw_buffer_load_b64(wr[i], wo[i], ks * kWStep, 0);
          w[r][i][0] = v[0]; w[r][i][1] = v[1];
        }
        sc[r][i] = static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(sr[i], mo[i], ks * kMStep, 0));
        bi[r][i] = static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(br[i], mo[i], ks * kMStep, 0));
      }
    };
    auto produce = [&](int r, uint32_t buf) {
      uint4* base = &sB[buf][0][0][0];
#pragma unroll
      for (int i = 0; i < UPT; ++i) {
        const float s = bf_lo(sc[r][i]), b = bf_lo(bi[r][i]);
#pragma unroll
        for (int k = 0; k < WPU; ++k) base[dst[i] + 16 * k] = dequant_word(w[r][i][k], s, b);
      }
    };
#pragma unroll
    for (int r = 0; r < D; ++r) load(r, clampk(r));
    produce(0, 0);
    load(0, clampk(D));
    __syncthreads();
    // Straight-line rounds of D stages: a branch between a load and its use
    // would make the compiler wait for every newer load too. The last round's
    // extra stage lands in the buffer nobody reads any more.
    uint32_t s = 0;
    for (; s + D <= stages; s += D) {
#pragma unroll
      for (int u = 0; u < D; ++u) {
        produce((u + 1) % D, (s + u + 1) & 1);
        load((u + 1) % D, clampk(s + u + 1 + D));
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);  // a later stage's dequantisation stays in its stage
      }
    }
#pragma unroll
    for (int u = 0; u < D; ++u) {
      if (s + u >= stages) break;
      produce((u + 1) % D, (s + u + 1) & 1);
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
    }
    return;
  }

  // -------------------------------------------------- consumers ----
  // Wave w owns 16-row blocks w and w + 4 (MW = 2) of the tile's rows, copied
  // straight into its own part of LDS: lane l of instruction i takes position
  // l % kChunks of row l / kChunks + i * (64 / kChunks). Rows past M read as
  // zero (their offset fails the buffer's range check).
  const int ml = lane & 15, c = lane >> 4;
  constexpr int kRowsPer = 64 / kChunks, kLoads = 16 / kRowsPer;
  const __amdgpu_buffer_rsrc_t ra = buffer_rsrc(g.a, static_cast<uint32_t>(static_cast<uint64_t>(g.M) * g.lda * 2));
  bool act[MW];
  uint32_t va[MW][kLoads];
#pragma unroll
  for (int x = 0; x < MW; ++x) {
    act[x] = m0 + 16 * (wave + 4 * x) < g.M;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const uint32_t r = lane / kChunks + i * kRowsPer, ch = (lane % kChunks) ^ r;
      va[x][i] = static_cast<uint32_t>(((m0 + 16 * (wave + 4 * x) + r) * g.lda + 8 * ch) * 2);
    }
  }
  const bool both = MW == 2 && act[MW - 1];
  const uint32_t lbase = static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)&sA[wave][0][0][0][0]));
  auto issue = [&](uint32_t ks, uint32_t slot) {
#pragma unroll
    for (int x = 0; x < MW; ++x) {
      if (!act[x]) continue;
#pragma unroll
      for (int i = 0; i < kLoads; ++i)
        lds_load16(ra, __builtin_amdgcn_readfirstlane(lbase + ((x * R + slot) * 16 * kChunks + 64 * i) * 16), va[x][i],
                   __builtin_amdgcn_readfirstlane(ks * KC * 2));
    }
  };
  // all but this wave's newest R - 2 stages have landed
  auto wait_next = [&]() {
    if (both)
      PRG_WAIT_VMCNT(2 * kLoads * (R - 2));
    else
      PRG_WAIT_VMCNT(kLoads * (R - 2));
  };
  f32x4 acc[MW][TN];
#pragma unroll
  for (int x = 0; x < MW; ++x)
#pragma unroll
    for (int t = 0; t < TN; ++t) acc[x][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < R - 1; ++r) issue(clampk(r), r);
  wait_next();
  __syncthreads();
  uint32_t slot = 0;
  for (uint32_t s = 0; s < stages; ++s) {
    // into the slot that stage s - 1 read, released by the last barrier
    issue(clampk(s + R - 1), slot == 0 ? R - 1 : slot - 1);
    if (act[0]) {
      const uint4* B = &sB[s & 1][0][0][0];
      const uint4* A = &sA[wave][0][0][0][0] + slot * 16 * kChunks + ml * kChunks;
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        bf16x8 a[MW], b[TN];
#pragma unroll
        for (int x = 0; x < MW; ++x) a[x] = __builtin_bit_cast(bf16x8, A[x * R * 16 * kChunks + ((4 * i + c) ^ ml)]);
#pragma unroll
        for (int t = 0; t < TN; ++t) b[t] = __builtin_bit_cast(bf16x8, B[(i * TN + t) * kWave + ((ml ^ (i * kSwz)) + 16 * c)]);
#pragma unroll
        for (int x = 0; x < MW; ++x)
#pragma unroll
          for (int t = 0; t < TN; ++t) acc[x][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[x], b[t], acc[x][t], 0, 0, 0);
      }
      // fragments are read two k steps ahead of their matrix instructions
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * (MW + TN), 0);
#pragma unroll
      for (int i = 0; i < KS - 2; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, MW * TN, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, MW + TN, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 2 * MW * TN, 0);
    }
    wait_next();
    __syncthreads();
    slot = slot + 1 == R ? 0 : slot + 1;
  }
  PRG_WAIT_VMCNT(0);

  // Epilogue: lane holds rows 4 (lane / 16) + r, column lane % 16 of each block.
  uint16_t* C = g.q[seg].c;
#pragma unroll
  for (int x = 0; x < MW; ++x) {
    if (!act[x]) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t m = m0 + 16 * (wave + 4 * x) + 4 * c + r;
      if (m >= g.M) continue;
      uint16_t* out = C + static_cast<uint64_t>(m) * N;
      if constexpr (kPair) {
#pragma unroll
        for (int t = 0; t < TN / 2; ++t) {
          const uint32_t n = n0 + 16 * t + ml;
          if (n >= N) continue;
          const float gate = round_bf(acc[x][t][r]), up = round_bf(acc[x][t + TN / 2][r]);
          out[n] = f2bf(silu(gate) * up);
        }
      } else {
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          const uint32_t n = n0 + 16 * t + ml;
          if (n >= N) continue;
          const float v = acc[x][t][r];
          if constexpr (EPI == kGemmResidual)
            out[n] = f2bf(round_bf(v) + bf2f(g.res[static_cast<uint64_t>(m) * N + n]));
          else
            out[n] = f2bf(v);
        }
      }
    }
  }
}

template <int EPI, int TN, int MW, int KC, int D, int R>
int launch_small(hipStream_t s, GemmArgs g, const char* name) {
  constexpr uint32_t kTileN = 16 * (EPI == kGemmSiluPair ? TN / 2 : TN);
  uint32_t tiles_n = 0;
  for (uint32_t i = 0; i < (EPI == kGemmSiluPair ? 1 : g.nq); ++i) {
    g.q[i].tile0 = tiles_n;
    tiles_n += (g.q[i].n + kTileN - 1) / kTileN;
  }
  const uint32_t blocks = tiles_n * ((g.M + 64 * MW - 1) / (64 * MW));
  hipLaunchKernelGGL((gemm_small_kernel<EPI, TN, MW, KC, D, R>), dim3(blocks), dim3(kSmallThreads), 0, s, g);
  PRG_CHECK_LAUNCH(name);
  return PRG_OK;
}

template <int EPI, int TN>
int launch_small_rows(hipStream_t s, const GemmArgs& g, int mw, const char* name) {
  if constexpr (TN == 1) {
    if (mw == 1) return launch_small<EPI, 1, 1, 256, 8, 4>(s, g, name);
    return launch_small<EPI, 1, 2, 256, 8, 2>(s, g, name);
  } else if constexpr (TN == 2) {
    if (mw == 1) return launch_small<EPI, 2, 1, 256, 8, 3>(s, g, name);
    return launch_small<EPI, 2, 2, 256, 8, 2>(s, g, name);
  } else {
    if (mw == 1) return launch_small<EPI, TN, 1, 128, 32 / TN, 3>(s, g, name);
    return launch_small<EPI, TN, 2, 128, 32 / TN, 3>(s, g, name);
  }
}

// Cost of a round of blocks in units of gemm_q4_kernel rows (0.255 us at
// K = 4096), from launches of 192 to 256 blocks over rotating weights: with up to
// 64 activation rows 16 / 32 / 64 / 128 weight rows per block take 13 / 14 / 20 /
// 34 us; with up to 128, 18.4 / 20 / 35 / 46 us. {1, 2} and {2, 2} are the pick
// only where the column tiles leave the others a nearly empty round: 384 rows x
// 1360 outputs 18.4 us against 20.9 of {4, 1}, 322 x 2720 20.1 against 26.4 of
// {4, 2}. A pair form {4, 2} gained nothing on two rounds of {4, 1} (322 x 2720:
// 13.5 against 12.6 us at K = 1024, 35.0 / 34.0 at 4096, 90.6 / 90.9 at 12288).
struct SmallVariant {
  int tn, mw;
  uint32_t cost;
};
constexpr SmallVariant kSmallPlain[] = {{1, 1, 51}, {2, 1, 55}, {4, 1, 75}, {1, 2, 72}, {2, 2, 80}, {4, 2, 133}};
constexpr SmallVariant kSmallPair[] = {{4, 1, 75}, {8, 1, 130}, {8, 2, 175}};

}  // namespace

namespace prg {

GemmSmallPick gemm_small_pick(const GemmArgs& g, int epi, uint32_t cus) {
  GemmSmallPick best;
  if (g.K % 256 != 0) return best;
  const bool pair = epi == kGemmSiluPair;
  auto consider = [&](const SmallVariant& v) {
    const uint32_t cols = 16 * (pair ? v.tn / 2 : v.tn), rows = 64 * v.mw;
    uint64_t blocks = 0;
    for (uint32_t i = 0; i < (pair ? 1 : g.nq); ++i) blocks += (g.q[i].n + cols - 1) / cols;
    blocks *= (g.M + rows - 1) / rows;
    const uint64_t c = (blocks + cus - 1) / cus * v.cost;
    if (c < best.cost) best = {v.tn, v.mw, c};
  };
  if (pair)
    for (const SmallVariant& v : kSmallPair) consider(v);
  else
    for (const SmallVariant& v : kSmallPlain) consider(v);
  return best;
}

int launch_gemm_small(hipStream_t s, const GemmArgs& g, int epi, const GemmSmallPick& v, const char* name) {
  if (epi == kGemmSiluPair) {
    if (v.tn == 4) return launch_small<kGemmSiluPair, 4, 1, 128, 8, 3>(s, g, name);
    return launch_small_rows<kGemmSiluPair, 8>(s, g, v.mw, name);
  }
  if (epi == kGemmResidual) {
    if (v.tn == 1) return launch_small_rows<kGemmResidual, 1>(s, g, v.mw, name);
    if (v.tn == 2) return launch_small_rows<kGemmResidual, 2>(s, g, v.mw, name);
    return launch_small_rows<kGemmResidual, 4>(s, g, v.mw, name);
  }
  if (v.tn == 1) return launch_small_rows<kGemmStore, 1>(s, g, v.mw, name);
  if (v.tn == 2) return launch_small_rows<kGemmStore, 2>(s, g, v.mw, name);
  return launch_small_rows<kGemmStore, 4>(s, g, v.mw, name);
}

}  // namespace prg
