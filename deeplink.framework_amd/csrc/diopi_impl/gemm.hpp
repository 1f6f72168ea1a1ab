// Internal GEMM interface shared by the dense (diopiMm/Bmm/Matmul/Addmm/Baddbmm/Linear)
// entry points. One problem description, two engines:
//   * the MFMA engine (bf16/fp16, fp32 accumulate) for K-contiguous operands,
//   * a strided fp32-accumulate FMA engine for everything else (fp32, odd shapes).
#pragma once

#include "common.hpp"

namespace amd {

// out[b, m, n] = alpha * sum_k A[b, m, k] * B[b, n, k]  +  beta * Cin[b, m, n]  +  bias[n]
// All strides in elements. B is described in [N, K] orientation whatever its storage order.
struct GemmProblem {
  diopiDtype_t dtype = diopi_dtype_unsupported;  // A, B, out (and Cin/bias) element type
  int64_t batch = 1, M = 0, N = 0, K = 0;
  const void* A = nullptr;
  int64_t sAb = 0, sAm = 0, sAk = 0;
  const void* B = nullptr;
  int64_t sBb = 0, sBn = 0, sBk = 0;
  void* out = nullptr;
  int64_t sOb = 0, sOm = 0;  // out: n-contiguous
  const void* Cin = nullptr;
  int64_t sCb = 0, sCm = 0, sCn = 0;
  const void* bias = nullptr;
  float alpha = 1.f, beta = 0.f;
  // out[m, n] = alpha * sum * colScale[n] + colBias[n], one rounding: N values each of their own dtype (fp16 / bf16 /
  // fp32), colBias optional. Only for problems gemmAppliesColumnScale accepts (no addend, no `bias`).
  const void* colScale = nullptr;
  diopiDtype_t colScaleDtype = diopi_dtype_float32;
  const void* colBias = nullptr;
  diopiDtype_t colBiasDtype = diopi_dtype_float32;
  // B holds int8 (strides in bytes, rows at multiples of 16), converted to `dtype` on the way into the product; with colScale only.
  bool int8B = false;
  // Workspace for K slices of 256 x 256 tiles, held once it is settled that the product takes that form (reserveTail in
  // gemm.hip). Not for callers to set.
  void* tailSlots = nullptr;
};

diopiError_t runGemm(diopiContextHandle_t ctx, hipStream_t stream, GemmProblem p);

#ifdef __HIPCC__
// v_mfma_f32_16x16x32: lane l feeds row (l & 15), K elements [8 * (l >> 4), +8) of both operands and
// receives D[4 * (l >> 4) + r][l & 15], r = 0..3. The large-tile kernel passes the weight fragment
// first, so D is the transposed block and a lane holds four consecutive columns of output row (l & 15).
template <typename T>
struct MfmaOp16;
template <>
struct MfmaOp16<bf16_t> {
  static __device__ __forceinline__ f32x4 run(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct MfmaOp16<half_t> {
  static __device__ __forceinline__ f32x4 run(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// The four int8 of one dword as floats: one SDWA conversion per byte (left to itself the compiler shifts
// bytes 1 and 3 into place first, two more VALU instructions per dword in a loop that has no slack).
__device__ __forceinline__ void cvt4(uint32_t w, float& f0, float& f1, float& f2, float& f3) {
  asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(f0) : "v"(w));
  asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(f1) : "v"(w));
  asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(f2) : "v"(w));
  asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(f3) : "v"(w));
}

// converts 8 consecutive int8 (two dwords) to an MFMA operand fragment
template <typename T>
__device__ __forceinline__ typename Vec16<T>::type int8Fragment(uint32_t lo, uint32_t hi) {
  float f[8];
  cvt4(lo, f[0], f[1], f[2], f[3]);
  cvt4(hi, f[4], f[5], f[6], f[7]);
  typename Vec16<T>::type r;
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = static_cast<T>(f[j]);
  return r;
}
#endif

// narrow_stream.hip: products of at most 64 rows whose columns are few for each compute unit.
// out[m, n] = (alpha, or scale[n]) * sum + bias[n] + beta * Cin[m, n], then the interleaved rotary embedding on the leading rotCols columns.
struct NarrowStreamArgs {
  const void* A = nullptr;
  const void* B = nullptr;  // of the type of A, or int8
  void* out = nullptr;
  const void* Cin = nullptr;
  const void* scale = nullptr;
  const void* bias = nullptr;
  int64_t lda = 0, ldb = 0, ldo = 0, sCm = 0, sCn = 0;
  int M = 0, N = 0, K = 0;
  bool int8B = false;
  int scaleDtype = 0, biasDtype = 0;
  float alpha = 1.f, beta = 0.f;
  const void* rotCos = nullptr;
  const void* rotSin = nullptr;
  int rotCols = 0, rotHeadDim = 2, rotTableRows = 1;
  bool rotTableF32 = false;
  float rotSinSign = 1.f;
  int colsPerWg = 0;
  bool noSlices = false;  // K slices, the faster form of some, have no workspace
};
bool narrowStreamPays(const NarrowStreamArgs& a);
diopiError_t launchNarrowStream(hipStream_t stream, diopiDtype_t dtype, NarrowStreamArgs a);

// Whether runGemm would send p to the kernel whose epilogue can multiply every column by a scale of its own (the
// 4-wave large-tile kernel): the caller sets colScale only then, and applies the scale in a pass of its own otherwise.
// What it settles and reserves for that stays in *p, which then goes to runGemm.
bool gemmAppliesColumnScale(diopiContextHandle_t ctx, hipStream_t stream, GemmProblem* p);

// gemm_weight_stream.hip: 16-bit products in one round of workgroups, each a rectangle of the output over the whole of K.
// A and B K-contiguous with 16-byte rows and less than 2 GiB each; out, Cin (n-contiguous) and bias in 8-byte pieces.
struct WeightStreamArgs {
  const void* A = nullptr;
  const void* B = nullptr;
  void* out = nullptr;
  const void* Cin = nullptr;
  const void* bias = nullptr;
  int64_t lda = 0, ldb = 0, ldo = 0, sCm = 0;
  int M = 0, N = 0, K = 0;
  float alpha = 1.f, beta = 0.f;
  int tilesM = 1, rowsPerWg = 0;   // workgroups along the rows, and the rows of one
  int tilesN = 0, tilesPerWg = 0;  // column tiles of 16, in all and of a workgroup
  bool siluMul = false;  // every 64 columns are 32 gate and 32 up columns; out (N / 2 wide) = silu(gate) * up
  // the interleaved rotary embedding on the leading rotCols columns
  const void* rotCos = nullptr;
  const void* rotSin = nullptr;
  int rotCols = 0, rotHeadDim = 2, rotTableRows = 1;
  bool rotTableF32 = false;
  float rotSinSign = 1.f;
};
// The estimated time (us) of the best cut, which is left in *g; 0 where there is none.
float weightStreamPlan(int64_t m, int64_t n, int64_t k, WeightStreamArgs* g);
diopiError_t launchWeightStream(hipStream_t stream, diopiDtype_t dtype, const WeightStreamArgs& g);

// diopiRotaryEmbedding on views (rotary_kv.hip): out and x of shape [..., heads, head_dim], strided views allowed.
diopiError_t runRotary(diopiContextHandle_t ctx, hipStream_t stream, const TensorView& out, const TensorView& x,
                       const TensorView& cosT, const TensorView& sinT, bool conj, bool interleaved);

// dst[b, c, r] = src[b, r, c] for 2-byte or 4-byte elements (64 x 64 tiles through LDS): src is [rows, cols] with the
// element strides given, dst dense [cols, rows] per batch.
diopiError_t transposeCopy(hipStream_t stream, void* dst, const void* src, int itemsize, int64_t batch, int64_t rows,
                           int64_t cols, int64_t sRow, int64_t sCol, int64_t sBatch);

}  // namespace amd
