// Products of 65 to about 700 rows (16-bit types, both operands K-contiguous) whose output tiles are to be cut to the chip: one round of
// workgroups, each a rectangle of up to 256 rows by up to 192 columns over the whole of K.
#include <algorithm>
#include <type_traits>

#include "gemm.hpp"

namespace amd {

// What bounds these products is what a compute unit takes in through its L1: 118 KB/us of lines that L2 holds, 45 KB/us out of HBM, and
// at most 60 of a mixture, because lines return in order and the activations' wait behind the weights'. This kernel takes in 46 (gated 203 x 22016 x
// 4096: 2.5 MB a unit in 53.7 us) to 50 (300 x 12288 x 4096): little more than what HBM alone gives. Every byte less counts, and
// every unit at work: 256 rectangles of 112 x 96 take in 1.6 MB each where 192 tiles of 128 x 128 take 2.1.
//   * 8 waves: two k-steps of 32 x two row halves x two column halves of the tile, two waves on a SIMD. A stage is 64 columns
//     of K; fragments of stage t + 1 are read while those of stage t are multiplied, one barrier a stage.
//   * Waves 0 and 1 copy weights, waves 2 - 7 activations, straight into two LDS rings of their own depths: loads return to
//     a wave in the order it issued them.
//   * The two k-steps' sums meet in LDS; each wave finishes half of its fragment rows.
//   * Tried: four waves with twice the columns (203 x 12288 x 4096 43 us against 37), four that multiply and four that copy (36.5,
//     but 256 registers hold no more than 128 x 96), all copies at a stage's start, deeper rings (the same).
constexpr int kStreamBK = 64;

// LDS rings of an output tile of 32 TM rows by 32 TN columns, in stages: what of 160 KiB the activations leave goes to the weights.
constexpr int streamStagesA(int tm, int tn) { return tm <= 4 ? (tn <= 4 ? 5 : 4) : tm <= 6 ? (tn >= 6 ? 3 : 4) : tm == 7 && tn <= 3 ? 4 : 3; }
constexpr int streamStagesB(int tm, int tn) { return std::min((160 - streamStagesA(tm, tn) * tm * 4) / (tn * 4), 8); }

template <int N>
__device__ __forceinline__ void waitLoads() {  // all but the N youngest loads of this wave have landed, and its LDS reads are done
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | (N >> 4) << 14);
}

template <typename T, int TM, int TN>
__global__ __launch_bounds__(512) void gemmWeightStreamKernel(WeightStreamArgs g) {
  typedef typename Vec16<T>::type Frag;
  typedef T T4 __attribute__((ext_vector_type(4)));
  constexpr int SA = streamStagesA(TM, TN), SB = streamStagesB(TM, TN);
  constexpr int BM = 32 * TM, BN = 32 * TN;
  constexpr unsigned kStageA = BM * 128, kStageB = BN * 128;  // bytes
  constexpr int kCopiesA = BM / 8, kCopiesB = BN / 8;         // copy instructions (8 rows x 128 bytes) of a stage
  constexpr int kShareA = (kCopiesA + 5) / 6, kShareB = kCopiesB / 2, kMost = kShareA > kShareB ? kShareA : kShareB;  // of a wave: two copy weights, six activations
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 15, kq = lane >> 4;
  const int ks = wave & 1, mh = (wave >> 1) & 1, nh = wave >> 2;  // this wave multiplies k-step ks of every stage, rows 16 TM mh ... of the tile
  int tm, tn;
  {
    const int total = gridDim.x, pid = blockIdx.x, xcd = pid & 7, idx = pid >> 3, q = total >> 3, r = total & 7;
    const int logical = xcd * q + min(xcd, r) + idx;
    tm = logical % g.tilesM, tn = logical / g.tilesM;
  }
  const int rowFirst = tm * g.rowsPerWg, rowEnd = min(g.M, rowFirst + g.rowsPerWg);
  const int firstTile = tn * g.tilesPerWg, nTiles = min(g.tilesPerWg, g.tilesN - firstTile);  // column tiles of 16
  const int nK = g.K / kStreamBK;
  // The weight row in row r of the tile's column block j. With a gate a block holds 8 channels: their gate rows, then their up rows.
  auto weightRow = [&](int j, int r) {
    const int t = firstTile + j;
    if (!g.siluMul) return t * 16 + r;
    const int channel = t * 8 + (r & 7);
    return (channel >> 5) * 64 + (channel & 31) + (r >> 3) * 32;
  };
  auto descriptor = [](const void* base, int64_t bytes) {
    const uint64_t p = reinterpret_cast<uint64_t>(base);
    u32x4 d = {(uint32_t)p, (uint32_t)(p >> 32) & 0xffffu, (uint32_t)bytes, 0x00020000u};
    return d;
  };
  const bool copiesB = wave < 2;
  const u32x4 rs = copiesB ? descriptor(g.B, ((int64_t)(g.N - 1) * g.ldb + g.K) * (int64_t)sizeof(T))
                           : descriptor(g.A, ((int64_t)(g.M - 1) * g.lda + g.K) * (int64_t)sizeof(T));
  const int first = copiesB ? wave : wave - 2, step = copiesB ? 2 : 6;
  int voff[kMost];
#pragma unroll
  for (int i = 0; i < kMost; ++i) {
    // (the waves that copy activations take every sixth piece; one that is past the last repeats the wave's own last, so that all have as many)
    const int at = first + step * min(i, copiesB ? kShareB - 1 : (kCopiesA - 1 - first) / 6);
    const int row = 8 * at + (lane >> 3), piece = ((lane & 7) ^ ((row >> 1) & 7)) * 8;
    // rows that are not there: an offset past the end of the descriptor, which reads as zeros without traffic
    if (copiesB)
      voff[i] = (row >> 4) < nTiles ? (int)(((int64_t)weightRow(row >> 4, row & 15) * g.ldb + piece) * (int64_t)sizeof(T)) : (int)0x80000000u;
    else
      voff[i] = rowFirst + row < rowEnd ? (int)(((int64_t)(rowFirst + row) * g.lda + piece) * (int64_t)sizeof(T)) : (int)0x80000000u;
  }
  const unsigned ldsBase = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem;
  const int kx = ((4 * ks + kq) ^ ((frow >> 1) & 7)) * 16;
  const unsigned aLane = (unsigned)((mh * TM * 16 + frow) * 128 + kx), bLane = SA * kStageA + (unsigned)((nh * TN * 16 + frow) * 128 + kx);
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  Frag fa[2][TM], fb[2][TN];

  auto multiply = [&](auto weights) {  // weights: what this wave copies
    constexpr bool kB = decltype(weights)::value;
    constexpr int S = kB ? SB : SA, COPIES = kB ? kShareB : kShareA;
    constexpr unsigned kStage = kB ? kStageB : kStageA;
    const unsigned ringBase = ldsBase + (kB ? SA * kStageA : 0u) + (unsigned)first * 1024u, ringEnd = ringBase + S * kStage;
    const int lastPiece = kB ? kShareB - 1 : (kCopiesA - 1 - first) / 6;
    unsigned fill = ringBase;                       // the ring place that the next copies go to
    int soff = 0;                                   // and the bytes into a row that they come from
    auto copyPart = [&](int from, int to) {
      const int at = __builtin_amdgcn_readfirstlane(soff);
#pragma unroll
      for (int i = from; i < to; ++i)
        if (i < COPIES) {
          const unsigned dst = fill + (unsigned)(min(i, lastPiece) * step) * 1024u;
          if constexpr (kB) loadToLds16Stream(rs, voff[i], at, dst);
          else loadToLds16(rs, voff[i], at, dst);
        }
    };
    auto copied = [&] {
      fill = fill + kStage == ringEnd ? ringBase : fill + kStage;
      soff += 128;
    };
    // all but the youngest `left` stages that this wave asked for have landed
    auto waitStages = [&](int left) {
      staticFor<S>([&](auto l) {
        if (left == decltype(l)::value) waitLoads<COPIES * decltype(l)::value>();
      });
    };
    unsigned readA = aLane, readB = bLane;  // where this lane's fragments of the stage that is read next lie
    auto readPart = [&](int buf, int from, int to) {
#pragma unroll
      for (int x = from; x < to; ++x) {
        if (x < TN) fb[buf][x] = *reinterpret_cast<const Frag*>(smem + readB + x * 2048);
        else if (x < TN + TM) fa[buf][x - TN] = *reinterpret_cast<const Frag*>(smem + readA + (x - TN) * 2048);
      }
    };
    int placeA = 0, placeB = 0;
    auto nextRead = [&] {
      const bool endA = ++placeA == SA, endB = ++placeB == SB;
      placeA = endA ? 0 : placeA, placeB = endB ? 0 : placeB;
      readA += endA ? kStageA * (1u - SA) : kStageA, readB += endB ? kStageB * (1u - SB) : kStageB;
    };
    for (int t = 0; t < S && t < nK; ++t) copyPart(0, COPIES), copied();
    waitStages(min(nK, S) - 1);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    readPart(0, 0, TM + TN), nextRead();
    // Stage t out of registers, stage t + 1 into registers, stage t + S out of memory. Past the barrier stage t + 1 is in LDS,
    // and every wave has its fragments of stage t: its place is free.
    auto products = [&](auto parity, auto copies) {
      constexpr int cur = decltype(parity)::value;
      constexpr int reads = (TM + TN + TN - 1) / TN, loads = (COPIES + TN - 1) / TN;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        readPart(cur ^ 1, j * reads, std::min((j + 1) * reads, TM + TN));
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[i][j] = MfmaOp16<T>::run(fb[cur][j], fa[cur][i], acc[i][j]);
        if constexpr (decltype(copies)::value) copyPart(j * loads, (j + 1) * loads);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (decltype(copies)::value) copied();
      nextRead();
    };
    using Even = std::integral_constant<int, 0>;
    using Odd = std::integral_constant<int, 1>;
    auto steady = [&](auto parity) {
      waitLoads<COPIES * (S - 2)>();
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      products(parity, std::true_type{});
    };
    int t = 0;
    for (; t + 2 + S <= nK; t += 2) {
      steady(Even{});
      steady(Odd{});
    }
    auto last = [&](auto parity) {
      waitStages(max(0, min(nK - 2 - t, S - 2)));
      __builtin_amdgcn_s_waitcnt(0xc07f);  // (the fragments of stage t)
      __builtin_amdgcn_s_barrier();
      if (t + S < nK) copyPart(0, COPIES), copied();
      __builtin_amdgcn_sched_barrier(0);
      products(parity, std::false_type{});  // (past the last stage: fragments that nothing multiplies)
      ++t;
    };
    while (t < nK) {
      last(Even{});
      if (t < nK) last(Odd{});
    }
  };
  if (copiesB) multiply(std::true_type{});
  else multiply(std::false_type{});
  __syncthreads();  // the rings are done with
  // The two k-steps' sums of a row half meet in LDS: wave ks = 0 finishes the first H fragment rows, ks = 1 the others.
  constexpr int H = (TM + 1) / 2;
  f32x4* const box = reinterpret_cast<f32x4*>(smem) + (mh + 2 * nh) * TM * TN * 64 + lane;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      if ((i < H) != (ks == 0)) box[(i * TN + j) * 64] = acc[i][j];
  const int row0 = rowFirst + mh * TM * 16 + frow;
  constexpr int kOutside = (int)0x80000000u;
  __syncthreads();
  const int tile0 = firstTile + nh * TN, tilesHere = nTiles - nh * TN;
  auto finish = [&](auto from, auto to) {
    constexpr int I0 = decltype(from)::value, I1 = decltype(to)::value;
    const int outCols = g.siluMul ? g.N / 2 : g.N;
    const __amdgpu_buffer_rsrc_t rsOut = __builtin_amdgcn_make_buffer_rsrc(g.out, 0, (int)(((int64_t)(g.M - 1) * g.ldo + outCols) * (int64_t)sizeof(T)), 0x00020000);
    auto put = [&](int i, bool there, int col, const f32x4& v) {
      const T4 o = {static_cast<T>(v[0]), static_cast<T>(v[1]), static_cast<T>(v[2]), static_cast<T>(v[3])};
      const int row = row0 + i * 16;
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, o), rsOut, row < rowEnd && there ? (int)(((int64_t)row * g.ldo + col) * (int64_t)sizeof(T)) : kOutside, 0, 0);
    };
    if (g.siluMul) {
      // gate columns are in lanes 0 - 31, the up columns of the same channels in lanes 32 - 63
#pragma unroll
      for (int i = I0; i < I1; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const f32x4 gate = acc[i][j] + box[(i * TN + j) * 64];
          f32x4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = gate[r] * __builtin_amdgcn_rcpf(1.f + __expf(-gate[r])) * __shfl_xor(gate[r], 32, 64);
          put(i, j < tilesHere && kq < 2, (tile0 + j) * 8 + kq * 4, v);
        }
      return;
    }
    float bias[TN][4];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      T4 b4 = {T(0.f), T(0.f), T(0.f), T(0.f)};
      if (g.bias && j < tilesHere) b4 = *reinterpret_cast<const T4*>(static_cast<const T*>(g.bias) + (tile0 + j) * 16 + kq * 4);
#pragma unroll
      for (int r = 0; r < 4; ++r) bias[j][r] = static_cast<float>(b4[r]);
    }
    if (g.rotCols > 0) {
      // adjacent columns are a pair: two pairs a lane, whose angles are two consecutive table entries of the lane's row
      const int half = g.rotHeadDim >> 1, tsz = g.rotTableF32 ? 4 : (int)sizeof(T);
      const int bytes = (int)((int64_t)g.rotTableRows * half * tsz);
      const __amdgpu_buffer_rsrc_t rsCos = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(g.rotCos), 0, bytes, 0x00020000);
      const __amdgpu_buffer_rsrc_t rsSin = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(g.rotSin), 0, bytes, 0x00020000);
      typedef T T2 __attribute__((ext_vector_type(2)));
      auto entries = [&](const __amdgpu_buffer_rsrc_t& r, int off, float (&f)[2]) {
        if (g.rotTableF32) {
          const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
          f[0] = __uint_as_float(v[0]), f[1] = __uint_as_float(v[1]);
        } else {
          const T2 v = __builtin_bit_cast(T2, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
          f[0] = static_cast<float>(v[0]), f[1] = static_cast<float>(v[1]);
        }
      };
      float cs[I1 - I0][TN][2], sn[I1 - I0][TN][2];
#pragma unroll
      for (int i = I0; i < I1; ++i) {
        const int row = row0 + i * 16, tableRow = row % g.rotTableRows;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int col = (tile0 + j) * 16 + kq * 4;
          const int off = row < rowEnd && j < tilesHere && col < g.rotCols ? (tableRow * half + ((col % g.rotHeadDim) >> 1)) * tsz : kOutside;
          entries(rsCos, off, cs[i - I0][j]), entries(rsSin, off, sn[i - I0][j]);
        }
      }
#pragma unroll
      for (int i = I0; i < I1; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          f32x4 v = acc[i][j] + box[(i * TN + j) * 64];
          const int col = (tile0 + j) * 16 + kq * 4;
          const bool rot = col < g.rotCols;
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] += bias[j][r];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const float c = rot ? cs[i - I0][j][e] : 1.f, s = rot ? sn[i - I0][j][e] * g.rotSinSign : 0.f;
            const float x = v[2 * e], y = v[2 * e + 1];
            if (rot) v[2 * e] = x * c - y * s, v[2 * e + 1] = x * s + y * c;
          }
          put(i, j < tilesHere, col, v);
        }
      return;
    }
    u32x2 add[I1 - I0][TN];
    if (g.Cin) {
      const __amdgpu_buffer_rsrc_t rsC = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(g.Cin), 0, (int)(((int64_t)(g.M - 1) * g.sCm + g.N) * (int64_t)sizeof(T)), 0x00020000);
#pragma unroll
      for (int i = I0; i < I1; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int row = row0 + i * 16, col = (tile0 + j) * 16 + kq * 4;
          add[i - I0][j] = __builtin_amdgcn_raw_buffer_load_b64(rsC, row < rowEnd && j < tilesHere ? (int)(((int64_t)row * g.sCm + col) * (int64_t)sizeof(T)) : kOutside, 0, 0);
        }
    }
#pragma unroll
    for (int i = I0; i < I1; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        f32x4 v = acc[i][j] + box[(i * TN + j) * 64];
        T4 c4;
        if (g.Cin) c4 = __builtin_bit_cast(T4, add[i - I0][j]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[r] = v[r] * g.alpha + bias[j][r];
          if (g.Cin) v[r] += g.beta * static_cast<float>(c4[r]);
        }
        put(i, j < tilesHere, (tile0 + j) * 16 + kq * 4, v);
      }
  };
  if (ks == 0) finish(std::integral_constant<int, 0>{}, std::integral_constant<int, H>{});
  else finish(std::integral_constant<int, H>{}, std::integral_constant<int, TM>{});
}

template <typename T, int TM, int TN>
static diopiError_t launchTile(hipStream_t stream, const WeightStreamArgs& g) {
  constexpr int ring = streamStagesA(TM, TN) * TM * 4096 + streamStagesB(TM, TN) * TN * 4096, sums = 4 * TM * TN * 1024;
  constexpr int lds = ring > sums ? ring : sums;
  static_assert(lds <= 160 * 1024 && streamStagesB(TM, TN) >= 3 && (streamStagesB(TM, TN) - 1) * 2 * TN < 64, "LDS of a compute unit, loads of a wave");
  AMD_HIP(allowDynamicLds(reinterpret_cast<const void*>(&gemmWeightStreamKernel<T, TM, TN>), lds));
  hipLaunchKernelGGL((gemmWeightStreamKernel<T, TM, TN>), dim3((unsigned)(g.tilesM * ceilDiv(g.tilesN, g.tilesPerWg))), dim3(512), lds, stream, g);
  AMD_LAUNCH_CHECK();
  return diopiSuccess;
}

template <typename T, int TM>
static diopiError_t launchRows(hipStream_t stream, const WeightStreamArgs& g) {
  if constexpr (TM < 8) {  // (240 rows by two column tiles never are the best cut for 256 units)
    if (g.tilesPerWg <= 2) return launchTile<T, TM, 1>(stream, g);
  }
  if (g.tilesPerWg <= 4) return launchTile<T, TM, 2>(stream, g);
  if (g.tilesPerWg <= 6) return launchTile<T, TM, 3>(stream, g);
  if constexpr (TM <= 5) {
    if (g.tilesPerWg > 8) return launchTile<T, TM, 6>(stream, g);
  }
  return launchTile<T, TM, 4>(stream, g);
}

template <typename T>
static diopiError_t launchType(hipStream_t stream, const WeightStreamArgs& g) {
  switch (std::max(4, (g.rowsPerWg + 31) / 32)) {
    case 4: return launchRows<T, 4>(stream, g);
    case 5: return launchRows<T, 5>(stream, g);
    case 6: return launchRows<T, 6>(stream, g);
    case 7: return launchRows<T, 7>(stream, g);
    default: return launchRows<T, 8>(stream, g);
  }
}

// The cut with the least estimated time, at most one workgroup for a unit (0: there is none). In us, fitted to 500 products of
// 65 to 700 rows (19 weights of 2 to 180 MB out of memory), each within 12 %, 4 % on average: a stage takes 0.077, 0.86 ns a row, 60 ns a pair
// of column tiles and 0.25 ns for each row of each pair; weights 28 ns a MB, 50 where no two workgroups share any; results 390 ns a MB;
// the launch, the first stages and the epilogue 3.9.
float weightStreamPlan(int64_t m, int64_t n, int64_t k, WeightStreamArgs* g) {
  const int64_t units = computeUnits() / 8 * 8;
  float best = 0.f;
  if (n % 16 != 0 || k % kStreamBK != 0 || k < 16 * kStreamBK) return best;  // (shorter K was not measured)
  for (int64_t tilesM = 1; tilesM <= 8; ++tilesM) {
    const int64_t rows = ceilDiv(ceilDiv(m, tilesM), (int64_t)16) * 16, colWgs = units / tilesM;
    if (rows > 256 || (tilesM > 1 && rows < 64) || rows * (tilesM - 1) >= m) continue;
    const int64_t tiles = std::max<int64_t>(ceilDiv(n / 16, colWgs), 2);
    if (tiles > (rows <= 160 ? 12 : 8)) continue;
    const float r = (float)rows, pairs = (float)ceilDiv(tiles, (int64_t)2);
    const float us = 3.9f + (float)(k / kStreamBK) * (0.077f + 0.00086f * r + (0.0595f + 0.00025f * r) * pairs) +
                     (tilesM == 1 ? 0.1e-6f : 0.055e-6f) * (float)(n * k) + (g->siluMul ? 0.39e-6f : 0.78e-6f) * (float)(m * n);
    if (best != 0.f && us >= best) continue;
    best = us;
    g->tilesM = (int)tilesM, g->rowsPerWg = (int)rows, g->tilesN = (int)(n / 16), g->tilesPerWg = (int)tiles;
  }
  return best;
}

diopiError_t launchWeightStream(hipStream_t stream, diopiDtype_t dtype, const WeightStreamArgs& g) {
  AMD_CHECK(g.tilesM >= 1 && g.rowsPerWg >= 1 && g.rowsPerWg <= 256 && (int64_t)g.tilesM * g.rowsPerWg >= g.M && g.tilesN * 16 == g.N && g.K % kStreamBK == 0 &&
                g.K >= kStreamBK && g.tilesPerWg >= 1 && g.tilesPerWg <= (g.rowsPerWg <= 160 ? 12 : 8),
            "weight stream: %d rows in %d, %d column tiles in %d", g.M, g.rowsPerWg, g.tilesN, g.tilesPerWg);
  return dtype == diopi_dtype_bfloat16 ? launchType<bf16_t>(stream, g) : launchType<half_t>(stream, g);
}

}  // namespace amd
