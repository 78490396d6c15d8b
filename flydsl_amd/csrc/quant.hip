// Quantization entry points: rows (a scale per row) and blocks of 128 (declarations: include/flygemm.h).
//
// A source of its own, so that these kernels' addresses do not follow the GEMM kernels' sizes: behind
// them in one source, the same instructions 0x1100 bytes further on made an 8-token fp8 MoE layer (7168 x
// 256, 256 experts) 0.4-0.5 us slower (76.2 -> 76.7), other shifts 0.1-0.4; here it is at 75.8 again.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/flygemm.h"
#include "abi_error.h"
#include "quant_rows.h"

using namespace flygemm;

namespace {

typedef void (*QuantFn)(QuantArgs);

// A quant launch: kernel, rows per workgroup and threads
struct QuantLaunch {
  QuantFn fn;
  int rows, threads;
};

// Short rows: the lanes of one wave per row.  Else one workgroup per row, in registers for rows of
// up to 1, 2, 4 or 8 slices, streaming beyond (quant_rows.h has the rules' figures).
template <int IN, int OUT, int MODE>
QuantLaunch quant_fn(int M, int N) {
#define SHORT(LPR, VPT) \
  if (N <= LPR * 8 * VPT) return QuantLaunch{quant_short_rows_kernel<IN, OUT, MODE, LPR, VPT>, 256 / LPR, 256};
  SHORT(8, 1) SHORT(16, 1) SHORT(32, 1) SHORT(64, 1)
  if (M >= kQuantManyRows) {
    SHORT(64, 2) SHORT(64, 4)
  }
#undef SHORT
  auto pick = [&](auto nt) -> QuantLaunch {
    constexpr int NT = decltype(nt)::value;
    const int nslices = (N + NT * 8 - 1) / (NT * 8);
    QuantFn fn = nslices <= 1   ? quant_rows_kernel<IN, OUT, MODE, 1, NT>
                 : nslices <= 2 ? quant_rows_kernel<IN, OUT, MODE, 2, NT>
                 : nslices <= 4 ? quant_rows_kernel<IN, OUT, MODE, 4, NT>
                 : nslices <= 8 ? quant_rows_kernel<IN, OUT, MODE, 8, NT>
                                : quant_rows_kernel<IN, OUT, MODE, 0, NT>;
    return QuantLaunch{fn, 1, NT};
  };
  if (N >= kQuantWideN || (M <= kQuantFewRows && N > 256 * 8)) return pick(std::integral_constant<int, 512>{});
  return pick(std::integral_constant<int, 256>{});
}

template <int IN>
QuantLaunch quant_fn_in(int out_dtype, int mode, int M, int N) {
  if (out_dtype == QOUT_FP8)
    return mode == QMODE_DIV_NEAREST ? quant_fn<IN, QOUT_FP8, QMODE_DIV_NEAREST>(M, N) : QuantLaunch{nullptr, 0, 0};
  if (mode == QMODE_RECIP_TRUNC) return quant_fn<IN, QOUT_INT8, QMODE_RECIP_TRUNC>(M, N);
  if (mode == QMODE_DIV_TRUNC) return quant_fn<IN, QOUT_INT8, QMODE_DIV_TRUNC>(M, N);
  if (mode == QMODE_DIV_NEAREST) return quant_fn<IN, QOUT_INT8, QMODE_DIV_NEAREST>(M, N);
  return QuantLaunch{nullptr, 0, 0};
}

}  // namespace

extern "C" {

int flygemm_quant_rows(void* out, float* scales, const void* in, int32_t M, int32_t N, int32_t in_dtype,
                       int32_t out_dtype, int32_t mode, void* stream) {
  if (M < 0 || N <= 0) return fail(hipErrorInvalidValue, "invalid sizes M=%d N=%d", M, N);
  if (N % 8 != 0) return fail(hipErrorInvalidValue, "N=%d must be a multiple of 8 (16-byte row vectors)", N);
  if (in_dtype < FLYGEMM_QIN_F16 || in_dtype > FLYGEMM_QIN_F32)
    return fail(hipErrorInvalidValue, "quant in_dtype %d not supported", in_dtype);
  if (out_dtype != FLYGEMM_QOUT_FP8 && out_dtype != FLYGEMM_QOUT_INT8)
    return fail(hipErrorInvalidValue, "quant out_dtype %d not supported", out_dtype);
  if (mode < FLYGEMM_QMODE_RECIP_TRUNC || mode > FLYGEMM_QMODE_DIV_NEAREST)
    return fail(hipErrorInvalidValue, "quant mode %d not supported", mode);
  if (out_dtype == FLYGEMM_QOUT_FP8 && mode != FLYGEMM_QMODE_DIV_NEAREST)
    return fail(hipErrorInvalidValue, "fp8 output rounds to nearest: mode must be FLYGEMM_QMODE_DIV_NEAREST");
  const int esz = in_dtype == FLYGEMM_QIN_F32 ? 4 : 2;
  if ((long)M * N * esz >= (1L << 40)) return fail(hipErrorInvalidValue, "input too large (M=%d N=%d)", M, N);
  if (M == 0) return 0;
  if (!out || !scales || !in) return fail(hipErrorInvalidValue, "null pointer");
  if (((uintptr_t)in & 15) || ((uintptr_t)out & 7) || ((uintptr_t)scales & 3))
    return fail(hipErrorInvalidValue, "misaligned pointer (input needs 16-byte, output 8-byte alignment)");
  const QuantLaunch q = in_dtype == FLYGEMM_QIN_F16    ? quant_fn_in<QIN_F16>(out_dtype, mode, M, N)
                        : in_dtype == FLYGEMM_QIN_BF16 ? quant_fn_in<QIN_BF16>(out_dtype, mode, M, N)
                                                       : quant_fn_in<QIN_F32>(out_dtype, mode, M, N);
  if (!q.fn) return fail(hipErrorInvalidValue, "unsupported quant combination");
  QuantArgs args{out, scales, in, M, N};
  hipLaunchKernelGGL(q.fn, dim3((unsigned)(((long)M + q.rows - 1) / q.rows)), dim3(q.threads), 0, (hipStream_t)stream, args);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(e, "launch of quant_rows failed: %s", hipGetErrorString(e));
  return 0;
}

int flygemm_quant_blocks(void* out, float* scales, const void* in, int64_t blocks, int32_t in_dtype, float qmax,
                         void* stream) {
  if (blocks < 0 || blocks >= (1L << 35)) return fail(hipErrorInvalidValue, "invalid block count %ld", (long)blocks);
  if (in_dtype < FLYGEMM_QIN_F16 || in_dtype > FLYGEMM_QIN_F32)
    return fail(hipErrorInvalidValue, "quant in_dtype %d not supported", in_dtype);
  if (blocks == 0) return 0;
  if (!out || !scales || !in) return fail(hipErrorInvalidValue, "null pointer");
  if (((uintptr_t)in & 15) || ((uintptr_t)out & 7) || ((uintptr_t)scales & 3))
    return fail(hipErrorInvalidValue, "misaligned pointer (input needs 16-byte, output 8-byte alignment)");
  BlockQuantArgs args{out, scales, in, blocks, 1.f / qmax};
  auto fn = in_dtype == FLYGEMM_QIN_F16    ? quant_blocks_kernel<QIN_F16>
            : in_dtype == FLYGEMM_QIN_BF16 ? quant_blocks_kernel<QIN_BF16>
                                           : quant_blocks_kernel<QIN_F32>;
  hipLaunchKernelGGL(fn, dim3((unsigned)((blocks + 15) / 16)), dim3(256), 0, (hipStream_t)stream, args);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(e, "launch of quant_blocks failed: %s", hipGetErrorString(e));
  return 0;
}

}  // extern "C"
