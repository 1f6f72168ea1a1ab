// Decode-sized products (at most 64 rows) with few output columns for each compute unit: the o and down projections, stacked
// QKV projections with grouped K/V heads, in 16-bit and int8 weights.
#include <algorithm>
#include <type_traits>

#include "gemm.hpp"

namespace amd {

// A workgroup owns at most 16 NT columns for the whole of K, so that there are no partial products and no reduction launch.
//   * What bounds it is the bytes a unit has under way: HBM answers after about a microsecond, so 256 units need some 30 KB each
//     to reach its rate. With 16 to 32 weight rows per workgroup that takes long pieces of a row: a stage is 512 columns (1 KiB
//     of a 16-bit row, one copy instruction), and 3 or 4 of them are in the LDS ring. From 33 rows on (and from 17 with two
//     column tiles of 16 bits) it is 256 columns, as the activations' ring has to fit too.
//   * Waves 0 - 3 copy weights, waves 4 - 7 activations: loads return to a wave in the order it issued them, so one that
//     copied both could not keep weights out of HBM further ahead than activations out of L2. One barrier a stage publishes both.
//   * Wave w multiplies the w-th eighth of every stage's columns; the eight shares meet in LDS at the end.
//   * 16-byte pieces are XOR-swizzled by row on the global side, so that the fragment reads are free of bank conflicts.
//   * Workgroup b starts its walk over K at stage b / 8 + 4 (b % 8): the workgroups of an XCD (every eighth) read the activations,
//     and rows of a power of two bytes, at different columns, so that the requests of a moment fall on all channels of its
//     L2. With 13 b, whose every eighth value repeats a few columns, 8192 x 8192 took 25.6 us at one row instead of 24.0, with a
//     common start 30.2.
//   * Columns past the end of K, rows past M and weight rows past the workgroup's share get an offset past the end of the
//     buffer descriptor: they read as zeros without traffic.
constexpr int kNarrowBK = 512;
// Ring places, of weights and of activations. More are slower here as in the other streaming kernels (a unit has at most some 45 KB
// out of HBM under way: copies past that hold up the waves that issue them). us at one row, places 5 + 4 -> 4 + 3 (16-bit, one
// column tile) 4096 x 4096 8.73 -> 8.35; int8, 8 + 4 -> 4 + 4, 4096 x 11008 11.60 -> 10.85; int8, two tiles, 6 + 4 -> 3 + 3, 8192 x 8192
// 13.9 -> 12.65. Fewer lose: 16-bit 3 + 3 4096 x 11008 16.75 -> 22.7, two tiles 3 + 2 5120 x 13824 24.2 -> 27.6.
constexpr int narrowStagesW(int tiles) { return tiles == 1 ? 4 : 3; }
constexpr int narrowStagesX(bool int8, int tiles, int bk) { return int8 && tiles == 1 && bk == kNarrowBK ? 4 : 3; }

// The stage of K that a workgroup which starts its walk at stage `start` visits c-th. Past the end, where copies fetch nothing, the last
// one again: the range check of a buffer load subtracts its scalar offset from the size, so that offset stays inside the rows.
__host__ __device__ constexpr int narrowStage(int c, int start, int stages) {
  const int at = (c < stages ? c : stages - 1) + start;
  return at >= stages ? at - stages : at;
}

template <typename T, bool W8, int G, int NT, int BK>
__global__ __launch_bounds__(512) void narrowStreamKernel(NarrowStreamArgs a) {
  typedef typename Vec16<T>::type Frag;
  constexpr int kSize = W8 ? 1 : 2, KS = BK / 256;                   // bytes of a weight; 32-wide k-steps of a wave and stage
  constexpr int WST = narrowStagesW(NT), XST = narrowStagesX(W8, NT, BK);    // ring places
  constexpr int kRowBytes = BK * kSize, kLanes = kRowBytes / 16;     // of a weight row's stage, and the lanes that copy it
  constexpr int kRows = 64 / kLanes;                                 // weight rows of a copy instruction (1 KiB)
  static_assert(16 * NT / kRows % 4 == 0, "four waves copy as many pieces each");
  constexpr int WIPW = 16 * NT / kRows / 4, XIPW = 4 * G * BK / 512, IPW = WIPW > XIPW ? WIPW : XIPW;  // copy instructions of a wave and stage
  constexpr unsigned WBUF = 16 * NT * kRowBytes, XBUF = 32 * G * BK;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* const sw = smem;
  char* const sx = smem + WST * WBUF;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kgrp = lane >> 4;
  const int n0 = blockIdx.x * a.colsPerWg, nCols = min(a.colsPerWg, a.N - n0);
  const int nStages = (a.K + BK - 1) / BK, rest = a.K - (nStages - 1) * BK;  // columns of the last stage
  const int kStart = (int)(((blockIdx.x >> 3) + 4u * (blockIdx.x & 7)) % (unsigned)nStages);
  auto descriptor = [](const void* base, int64_t bytes) {
    const uint64_t p = reinterpret_cast<uint64_t>(base);
    u32x4 d = {(uint32_t)p, (uint32_t)(p >> 32) & 0xffffu, (uint32_t)bytes, 0x00020000u};
    return d;
  };
  // The sums of (row group gi, column tile j, register r) are finished by wave (4 (NT gi + j) + r) % 8: what its lanes need of the epilogue is
  // requested now, as bits (a conversion here would wait for the answer before the first copy goes out).
  constexpr int ITEMS = (4 * G * NT + 7) / 8;
  constexpr bool kHalfIsBf16 = std::is_same<T, bf16_t>::value;
  const int tDtype = kHalfIsBf16 ? diopi_dtype_bfloat16 : diopi_dtype_float16;
  uint32_t scale[ITEMS], bias[ITEMS], add[ITEMS], cs[ITEMS], sn[ITEMS];
  auto bits = [](const void* base, int64_t at, int dtype) -> uint32_t {
    return dtype == diopi_dtype_float32 ? reinterpret_cast<const uint32_t*>(base)[at] : reinterpret_cast<const uint16_t*>(base)[at];
  };
  auto value = [](uint32_t v, int dtype) {
    return dtype == diopi_dtype_float32 ? __uint_as_float(v) : dtype == diopi_dtype_bfloat16 ? __uint_as_float(v << 16)
                                        : static_cast<float>(__builtin_bit_cast(half_t, (uint16_t)v));
  };
  const int rotDtype = a.rotTableF32 ? (int)diopi_dtype_float32 : tDtype;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int item = wave + 8 * i, lc = (item >> 2) % NT * 16 + r16, row = (item >> 2) / NT * 16 + kgrp * 4 + (item & 3), col = n0 + lc;
    scale[i] = bias[i] = add[i] = cs[i] = sn[i] = 0;
    if (item < 4 * G * NT && lc < nCols && row < a.M) {
      if (a.scale) scale[i] = bits(a.scale, col, a.scaleDtype);
      if (a.bias) bias[i] = bits(a.bias, col, a.biasDtype);
      if (a.Cin) add[i] = bits(a.Cin, (int64_t)row * a.sCm + (int64_t)col * a.sCn, tDtype);
      if (col < a.rotCols) {
        const int64_t at = (int64_t)(row % a.rotTableRows) * (a.rotHeadDim >> 1) + ((col % a.rotHeadDim) >> 1);
        cs[i] = bits(a.rotCos, at, rotDtype), sn[i] = bits(a.rotSin, at, rotDtype);
      }
    }
  }
  const bool copiesW = wave < 4;
  const int ci = wave & 3;
  const u32x4 rs = copiesW ? descriptor(a.B, ((int64_t)(a.N - 1) * a.ldb + a.K) * kSize) : descriptor(a.A, ((int64_t)(a.M - 1) * a.lda + a.K) * 2);
  // copy instruction q = ci + 4 i: kRows weight rows or one activation row; a lane owns a physical piece and fetches the
  // logical one that the swizzle puts there
  unsigned voff[IPW];
  int pieceCol[IPW];  // the first column of this lane's piece in a stage
#pragma unroll
  for (int i = 0; i < IPW; ++i) {
    const int q = ci + 4 * i;
    if (copiesW) {
      const int row = kRows * q + lane / kLanes, piece = (lane % kLanes) ^ (row & 15);
      pieceCol[i] = piece * (16 / kSize);
      voff[i] = row < nCols ? (unsigned)((int64_t)(n0 + row) * a.ldb * kSize + piece * 16) : 0x80000000u;
    } else {
      constexpr int kXLanes = BK / 8;
      const int row = 64 / kXLanes * q + lane / kXLanes, piece = (lane % kXLanes) ^ (row & 15);
      pieceCol[i] = piece * 8;
      voff[i] = row < a.M ? (unsigned)((int64_t)row * a.lda * 2 + piece * 16) : 0x80000000u;
    }
  }
  const unsigned ldsBase = (unsigned)(size_t)(__attribute__((address_space(3))) char*)(copiesW ? sw : sx) + (unsigned)ci * 1024u;
  auto copyStage = [&](auto weights, int c, int place) {
    constexpr bool kW = decltype(weights)::value;
    const int cc = narrowStage(c, kStart, nStages);
    const int from = cc * BK * (kW ? kSize : 2);
    const unsigned to = ldsBase + (unsigned)place * (kW ? WBUF : XBUF);
    // (of a stage past the end no column is there: the copies count as the others do, and fetch nothing)
    const int columns = c >= nStages ? 0 : cc == nStages - 1 ? rest : BK;
    auto copy = [&](auto whole) {
#pragma unroll
      for (int i = 0; i < (kW ? WIPW : XIPW); ++i) {
        const int v = decltype(whole)::value || pieceCol[i] < columns ? (int)voff[i] : (int)0x80000000u;
        if constexpr (kW) loadToLds16Stream(rs, v, from, to + (unsigned)i * 4096u);
        else loadToLds16(rs, v, from, to + (unsigned)i * 4096u);
      }
    };
    if (columns == BK) copy(std::true_type{});
    else copy(std::false_type{});
  };
  f32x4 acc[G][NT];
#pragma unroll
  for (int gi = 0; gi < G; ++gi)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[gi][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // This wave's fragments, columns 32 KS w of a stage on: of k-step s = KS w + t piece 4 s + kgrp of both operands; int8: 8 KS
  // weights at 8 KS (4 w + kgrp), which meet the activations of the same columns.
  unsigned xAt[KS], wAt[KS];
#pragma unroll
  for (int t = 0; t < KS; ++t) {
    const int px = W8 ? KS * (4 * wave + kgrp) + t : 4 * (KS * wave + t) + kgrp, w8 = 8 * KS * (4 * wave + kgrp);
    xAt[t] = WST * WBUF + (unsigned)(r16 * BK * 2 + ((px ^ r16) << 4));
    wAt[t] = W8 ? (unsigned)(r16 * kRowBytes + (((w8 >> 4) ^ r16) << 4) + (w8 & 8)) : (unsigned)(r16 * kRowBytes + ((px ^ r16) << 4));
  }
  typedef typename std::conditional<W8 && KS == 1, u32x2, u32x4>::type Weights;
  Frag x[G][KS];
  Weights q[NT][W8 ? 1 : KS];
  auto fetch = [&](unsigned placeW, unsigned placeX) {
#pragma unroll
    for (int gi = 0; gi < G; ++gi)
#pragma unroll
      for (int t = 0; t < KS; ++t) x[gi][t] = *reinterpret_cast<const Frag*>(smem + xAt[t] + placeX * XBUF + gi * 32 * BK);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int t = 0; t < (W8 ? 1 : KS); ++t) q[j][t] = *reinterpret_cast<const Weights*>(smem + wAt[t] + placeW * WBUF + j * 16 * kRowBytes);
  };
  auto multiply = [&] {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      Frag w[KS];
#pragma unroll
      for (int t = 0; t < KS; ++t) {
        if constexpr (W8) w[t] = int8Fragment<T>(q[j][0][2 * t], q[j][0][2 * t + 1]);
        else w[t] = __builtin_bit_cast(Frag, q[j][t]);
      }
#pragma unroll
      for (int gi = 0; gi < G; ++gi)
#pragma unroll
        for (int t = 0; t < KS; ++t) acc[gi][j] = MfmaOp16<T>::run(x[gi][t], w[t], acc[gi][j]);
    }
  };
  auto walk = [&](auto weights) {
    constexpr bool kW = decltype(weights)::value;
    constexpr int ST = kW ? WST : XST;
#pragma unroll
    for (int c = 0; c < ST - 1; ++c) copyStage(weights, c, c);
    unsigned placeW = 0, placeX = 0, fill = ST - 1;
    for (int c = 0; c < nStages; ++c) {
      // This wave's copies of stage c have landed (behind them ST - 2 stages are under way); past the barrier both operands
      // of it are in LDS, and every wave has left the place of stage c - 1.
      constexpr int n = (ST - 2) * (kW ? WIPW : XIPW);
      __builtin_amdgcn_s_waitcnt(0x0070 | (n & 15) | ((n >> 4) << 14));
      __builtin_amdgcn_s_barrier();
      fetch(placeW, placeX);  // (answered while the copies go out)
      copyStage(weights, c + ST - 1, (int)fill);
      multiply();
      placeW = placeW + 1 == WST ? 0 : placeW + 1, placeX = placeX + 1 == XST ? 0 : placeX + 1, fill = fill + 1 == ST ? 0 : fill + 1;
    }
  };
  if (copiesW) walk(std::true_type{});
  else walk(std::false_type{});
  __builtin_amdgcn_s_waitcnt(0x0070);  // (the copies of stages past the end)
  __syncthreads();
  float* const sums = reinterpret_cast<float*>(smem);  // [8 waves][G][NT][4][64]
#pragma unroll
  for (int gi = 0; gi < G; ++gi)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) sums[(((wave * G + gi) * NT + j) * 4 + r) * 64 + lane] = acc[gi][j][r];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int item = wave + 8 * i, lc = (item >> 2) % NT * 16 + r16, row = (item >> 2) / NT * 16 + kgrp * 4 + (item & 3), col = n0 + lc;
    if (item >= 4 * G * NT) break;  // wave-uniform
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) v += sums[(w * G * NT * 4 + item) * 64 + lane];
    v = v * (a.scale ? value(scale[i], a.scaleDtype) : a.alpha);
    if (a.bias) v += value(bias[i], a.biasDtype);
    if (a.Cin) v += a.beta * value(add[i], tDtype);
    if (a.rotCols > 0) {
      // adjacent columns are a pair and sit in adjacent lanes (the shares are even): every lane takes part in the exchange
      const float other = __shfl_xor(v, 1, 64), c = value(cs[i], rotDtype), s = value(sn[i], rotDtype) * a.rotSinSign;
      if (col < a.rotCols) v = (col & 1) ? other * s + v * c : v * c - other * s;
    }
    if (lc < nCols && row < a.M) reinterpret_cast<T*>(a.out)[(int64_t)row * a.ldo + col] = static_cast<T>(v);
  }
}

template <typename T, bool W8, int G, int NT, int BK = kNarrowBK>
static diopiError_t launchTiles(hipStream_t stream, const NarrowStreamArgs& a) {
  constexpr int lds = std::max(narrowStagesW(NT) * 16 * NT * BK * (W8 ? 1 : 2) + narrowStagesX(W8, NT, BK) * 32 * G * BK, 8 * G * NT * 1024);
  static_assert(lds <= 160 * 1024, "LDS of a compute unit");
  AMD_HIP(allowDynamicLds(reinterpret_cast<const void*>(&narrowStreamKernel<T, W8, G, NT, BK>), lds));
  hipLaunchKernelGGL((narrowStreamKernel<T, W8, G, NT, BK>), dim3((unsigned)ceilDiv(a.N, a.colsPerWg)), dim3(512), lds, stream, a);
  AMD_LAUNCH_CHECK();
  return diopiSuccess;
}

template <typename T, bool W8, int G>
static diopiError_t launchManyRows(hipStream_t stream, const NarrowStreamArgs& a) {
  return a.colsPerWg <= 16 ? launchTiles<T, W8, G, 1, 256>(stream, a) : launchTiles<T, W8, G, 2, 256>(stream, a);
}

template <typename T>
static diopiError_t launchType(hipStream_t stream, const NarrowStreamArgs& a) {
  const int tiles = (a.colsPerWg + 15) / 16;
  if (a.M > 48) return a.int8B ? launchManyRows<T, true, 4>(stream, a) : launchManyRows<T, false, 4>(stream, a);
  if (a.M > 32) return a.int8B ? launchManyRows<T, true, 3>(stream, a) : launchManyRows<T, false, 3>(stream, a);
  if (a.int8B) {
    if (a.M > 16) return tiles == 1 ? launchTiles<T, true, 2, 1>(stream, a) : launchTiles<T, true, 2, 2>(stream, a);
    return tiles == 1 ? launchTiles<T, true, 1, 1>(stream, a) : tiles == 2 ? launchTiles<T, true, 1, 2>(stream, a) : launchTiles<T, true, 1, 3>(stream, a);
  }
  if (a.M > 16) return tiles == 1 ? launchTiles<T, false, 2, 1>(stream, a) : launchTiles<T, false, 2, 2, 256>(stream, a);
  return tiles == 1 ? launchTiles<T, false, 1, 1>(stream, a) : launchTiles<T, false, 1, 2>(stream, a);
}

// Where this kernel is the faster one, from both sides timed over 40 weights of 256 to 16384 rows at 1 to 64 activation rows, with
// the weights out of memory (us, kernels of gemm.hip or weight_only_int8.hip -> this one):
//   16-bit, 1 / 4 / 16 / 32 rows: 4096 x 4096 8.9 -> 8.4, 9.8 -> 8.6, 10.7 -> 8.8, 12.6 -> 9.8; 5120 x 5120 14.2 -> 11.7 at one row; 4096 x 11008
//     (two K slices and their reduction) 19.4 -> 16.7, 20.2 -> 18.5 at 16 rows; 6144 x 4096 13.0 -> 11.2; 8192 x 28672 73.1 -> 72.4
//   int8: 4096 x 4096 7.8 -> 6.2, 8.6 -> 6.3, 10.9 -> 7.0, 12.1 -> 8.8; 4096 x 11008 13.9 -> 10.8 at one row; 8192 x 8192 17.3 -> 12.8; 4096 x
//     6144 15.3 -> 8.7 at 16 rows; 4096 x 4160, which only the one-output-a-lane kernel took, 580 -> 7.1
//   33 / 64 rows: 16-bit 4096 x 4096 14.3 -> 11.0, 16.5 -> 13.2; 6144 x 4096 15.8 -> 13.6, 18.6 -> 16.2; 8192 x 8192 26.9 -> 24.1, 32.7 -> 27.5; int8
//     4096 x 4096 13.3 -> 10.1, 14.4 -> 12.3; 6144 x 4096 16.5 -> 11.5, 17.5 -> 14.5; 8192 x 4096 17.7 -> 11.8, 18.9 -> 14.9
// The others stay where they were:
//   * more columns for a unit than 32 (16-bit) or 48 (int8): there whole K in shorter stages streams as well (int8 16384 x 4096
//     13.4 against 14.4, 16-bit 10240 x 8192 the same); from 17 rows on 32, as far as the rings go;
//   * one or two rows of a small weight, all latency (16-bit 2048 x 2048 4.9 against 5.3, int8 2560 x 2560 4.6 against 4.9);
//   * up to four rows of a 16-bit weight with K no longer than its 7168 and more columns (8192 x 8192 23.0 against 24.0);
//   * int8 with two or three column tiles and a K of fewer than four stages (8192 x 1024 4.5 against 5.2);
//   * many rows with a long K, where a unit takes in more of the activations than of its weights and K slices, which divide
//     them, win: 17 rows, 16-bit 4096 x 11008 20.2 against 20.6, int8 5120 x 13824 19.2 against 21.0; 16 rows, int8 8192 x 28672
//     41.0 against 42.2 (8192 x 16384 29.3 -> 23.6); 64 rows, 16-bit 4096 x 8192 20.8 against 21.8, 1024 x 4096 10.1 against 11.8, int8
//     4096 x 8192 19.0 against 20.6, 2048 x 8192 15.1 against 19.3 (1024 x 4096 11.8 -> 11.3). The 16-bit line below K = 4096, from 760
//     products: 33 to 64 rows x 64 to 1024, whose four slices are one round of the chip, K = 3328 0.97 to 1.03 of the slices' time, 3456 up
//     to 1.06, 3968 1.03 to 1.16 (64 x 512 x 3968 10.1 against 11.3); 64 x 1280 x 3584 15.2 -> 11.0, 64 x 2048 x 3968 13.7 -> 12.4.
bool narrowStreamPays(const NarrowStreamArgs& a) {
  const int64_t size = a.int8B ? 1 : 2, weights = (int64_t)a.N * a.K;
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (a.M < 1 || a.M > 64 || a.N < 1 || a.K < 16 || a.K % (16 / size) != 0 || !al16(a.A) || !al16(a.B) || a.lda % 8 != 0 || a.ldb * size % 16 != 0 ||
      ((int64_t)(a.N - 1) * a.ldb + a.K) * size >= ((int64_t)1 << 31) || ((int64_t)(a.M - 1) * a.lda + a.K) * 2 >= ((int64_t)1 << 31))
    return false;
  const int64_t cols = ceilDiv(a.N, (int64_t)computeUnits());
  if (a.M > 32) {
    if (cols > 32) return false;
    if (2 * (int64_t)a.K <= 3 * (int64_t)a.N) return true;
    if (a.int8B) return a.K <= 4096;
    // (the other form: four slices of up to 1024 columns, eight steps of 128, in pieces of 8 results, and a rotation in a pass of its own)
    const bool slicesFit = a.rotCols == 0 && !a.noSlices && ceilDiv(a.N, 16) * 4 <= computeUnits() && a.N >= 16 && a.N % 8 == 0 && a.K % 128 == 0;
    return a.K < 4096 && !(a.K > 3328 && slicesFit);
  }
  if (a.int8B) {
    if (cols > (a.M > 16 ? 32 : 48) || (cols > 16 && a.K < 4 * kNarrowBK)) return false;
    if (a.M > 16) return a.K <= 8192 || a.K <= 2 * (int64_t)a.N;
    return !(a.M <= 2 && weights <= ((int64_t)1 << 23)) && !(a.M > 12 && weights > ((int64_t)3 << 26));
  }
  if (a.M > 16) return cols <= 32 && a.K <= 8192;
  return cols <= 32 && !(a.M <= 2 && weights <= ((int64_t)1 << 22)) && !(a.M <= 4 && cols > 28 && a.K <= a.N);
}

diopiError_t launchNarrowStream(hipStream_t stream, diopiDtype_t dtype, NarrowStreamArgs a) {
  AMD_CHECK(narrowStreamPays(a), "narrow stream: %d x %d x %d", a.M, a.N, a.K);
  a.colsPerWg = (int)ceilDiv(a.N, (int64_t)computeUnits());
  if (a.rotCols > 0) a.colsPerWg = (a.colsPerWg + 1) & ~1;  // the two columns of a rotary pair stay together
  return dtype == diopi_dtype_bfloat16 ? launchType<bf16_t>(stream, a) : launchType<half_t>(stream, a);
}

}  // namespace amd
