// Per-row (per-token) quantization of activations on the device: the step that produces
// a GEMM's A operand and its per-token scale.
//
//   amax[m]  = max_n |x[m][n]|                      (fp32)
//   scale[m] = amax[m] / qmax, or 1 where that is 0  (qmax = 127 for int8, 448 for fp8)
//   q[m][n]  = cast(x[m][n] / scale[m])  or  cast(x[m][n] * (1 / scale[m]))
//
// Two reference formulations, selected by `mode`:
//  * QMODE_RECIP_TRUNC -- the reference's device kernel (tests/kernels/test_quant.py:81-265):
//    fp16 in, int8 out, q = fptosi(x * (1/scale)) (truncation toward zero, :223-238).
//  * QMODE_DIV_TRUNC / QMODE_DIV_NEAREST -- the reference's host quantizer pertoken_quant
//    (tests/utils.py:29-73): NaN -> 0 and +-inf -> +-qmax first (:50-55), then
//    q = (x / scale).to(dtype) (:71), which truncates for int8 (DIV_TRUNC); DIV_NEAREST
//    rounds half to even instead (and clamps to +-127), the int8 rule of the benchmark
//    workloads.  fp8 (e4m3fn) always rounds to nearest even, as torch's cast does.
//
// Short rows (kQuantManyRows): 8 to 64 lanes of one wave per row, each with up to four 8-element
// vectors, so a workgroup takes 4 to 32 rows and no barrier is needed.  Else one workgroup per row; each thread owns 8 consecutive elements per (8 * NT)-element slice, and rows of up to
// VPT slices stay in registers between the max pass and the quantize pass, so HBM is read once
// (VPT == 0: streaming variant, which re-reads the row from L2).  Loads (16-byte vectors) and
// stores (8 bytes) are non-temporal; consecutive lanes touch consecutive addresses in every
// instruction.
//
// What bounds it: HBM for many rows, once the arithmetic is kept small enough to hide behind it
// (the operators above taken literally are about 30 vector instructions per element), and the
// latency of load, row maximum and store for few rows.  So
//   * the row maximum is taken over the inputs' bits: |x| orders like its bits as an unsigned
//     number, two 16-bit inputs per instruction.  A maximum at or past infinity's bits says that the
//     thread holds NaN or infinity, and only then are its inputs scrubbed one by one;
//   * x / scale is formed from the correctly rounded reciprocal r = 1/scale: q = x*r, then twice
//     q += fma(-q, scale, x) * r.  The first step brings q within one unit in the last place of
//     the quotient, and from there the second rounds it correctly (Markstein, "Computation of
//     elementary functions on the IBM RISC System/6000 processor", 1990, theorem on division), so it
//     equals the division bit for bit at 5 instructions in place of 10 and a quarter-rate
//     reciprocal.  It needs the residuals to be exact: rows with a scale outside [2^-90, 2^90]
//     divide; smaller inputs of the other rows round to zero either way.
// Together 8192 x 7168 bf16 -> fp8 takes 30.9 us (5.7 TB/s) against 39.0 with the divisions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace flygemm {

enum QuantIn : int { QIN_F16 = 0, QIN_BF16 = 1, QIN_F32 = 2 };
enum QuantOut : int { QOUT_FP8 = 0, QOUT_INT8 = 1 };
enum QuantMode : int { QMODE_RECIP_TRUNC = 0, QMODE_DIV_TRUNC = 1, QMODE_DIV_NEAREST = 2 };

struct QuantArgs {
  void* out;          // [M][N] int8 or fp8 codes
  float* scales;      // [M]
  const void* in;     // [M][N] fp16 / bf16 / fp32
  int M, N;
};

// Threads of the one-row workgroups: 512 for rows of at least kQuantWideN elements, and for up to
// kQuantFewRows rows of more than one slice of 256 threads (fewer vectors one after another in a thread;
// with one slice the other threads only wait: 512 x 1024 fp16 -> int8 2.56 us with 512, 2.36 with 256), else 256.  Graph-timed on MI355X,
// bf16 -> fp8, 256 / 512 / 1024 threads: 1 x 7168 2.97 / 2.40 / 2.59 us, 512 x 7168 4.64 / 4.39 / 4.62,
// 1024 x 7168 6.19 / 5.83, 2048 x 7168 10.28 / 10.24 / 12.41, 8192 x 7168 30.9 / 32.7 / 41.4,
// 4096 x 8192 20.2 / 19.5 / 22.9.
constexpr int kQuantWideN = 8192;
constexpr int kQuantFewRows = 1024;
// Lanes-per-row kernel: every row of up to 512 elements, and rows of up to 2048 when there are at
// least kQuantManyRows.  Against one row per 256-thread workgroup: 65536 x 256 13.2 us against 53.7
// (7/8 of the threads idle), 64 x 256 2.20 against 2.64, 4096 x 768 4.27 against 5.55, 4096 x 2048
// 6.83 against 7.17; with fewer rows of over 512 elements the four vectors of a lane are a longer
// chain: 2048 x 2048 4.97 against 4.47, 1 x 2048 2.76 against 1.95.
constexpr int kQuantManyRows = 4096;

typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef int i32x2q __attribute__((ext_vector_type(2)));

typedef uint32_t u32x4q __attribute__((ext_vector_type(4)));

// 8 consecutive 16-bit inputs (one 16-byte vector, element order) as fp32
template <int IN>
__device__ __forceinline__ f32x8 cvt8_16(u32x4q w) {
  static_assert(IN == QIN_F16 || IN == QIN_BF16, "16-bit inputs");
  f32x8 v;
  const uint32_t words[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint16_t h0 = (uint16_t)(words[i] & 0xFFFFu), h1 = (uint16_t)(words[i] >> 16);
    if constexpr (IN == QIN_F16) {
      v[2 * i] = (float)__builtin_bit_cast(_Float16, h0);
      v[2 * i + 1] = (float)__builtin_bit_cast(_Float16, h1);
    } else {
      v[2 * i] = __builtin_bit_cast(float, (uint32_t)h0 << 16);
      v[2 * i + 1] = __builtin_bit_cast(float, (uint32_t)h1 << 16);
    }
  }
  return v;
}

typedef uint16_t u16x2q __attribute__((ext_vector_type(2)));

// 8 consecutive inputs as loaded, and what is taken from them
template <int IN>
struct Raw8 {
  u32x4q w;
  __device__ __forceinline__ void load(const void* row_base, int col) {
    w = __builtin_nontemporal_load((const u32x4q*)((const uint16_t*)row_base + col));
  }
  __device__ __forceinline__ f32x8 value() const { return cvt8_16<IN>(w); }
  // running maximum of |x| as bits, one in each half of the word
  __device__ __forceinline__ uint32_t max_bits(uint32_t m) const {
    u16x2q r = __builtin_bit_cast(u16x2q, m);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      r = __builtin_elementwise_max(r, __builtin_bit_cast(u16x2q, w[i] & 0x7FFF7FFFu));
    return __builtin_bit_cast(uint32_t, r);
  }
  static __device__ __forceinline__ uint32_t fold(uint32_t m) { return max(m & 0xFFFFu, m >> 16); }
  static constexpr uint32_t kInf = IN == QIN_F16 ? 0x7C00u : 0x7F80u;
  static __device__ __forceinline__ float abs_value(uint32_t bits) {
    if constexpr (IN == QIN_F16)
      return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
    else
      return __builtin_bit_cast(float, bits << 16);
  }
};

template <>
struct Raw8<QIN_F32> {
  u32x4q lo, hi;
  __device__ __forceinline__ void load(const void* row_base, int col) {
    const u32x4q* p = (const u32x4q*)((const float*)row_base + col);
    lo = __builtin_nontemporal_load(p);
    hi = __builtin_nontemporal_load(p + 1);
  }
  __device__ __forceinline__ f32x8 value() const {
    f32x8 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t a = lo[i], b = hi[i];
      v[i] = __builtin_bit_cast(float, a);
      v[4 + i] = __builtin_bit_cast(float, b);
    }
    return v;
  }
  __device__ __forceinline__ uint32_t max_bits(uint32_t m) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) m = max(max(m, lo[i] & 0x7FFFFFFFu), hi[i] & 0x7FFFFFFFu);
    return m;
  }
  static __device__ __forceinline__ uint32_t fold(uint32_t m) { return m; }
  static constexpr uint32_t kInf = 0x7F800000u;
  static __device__ __forceinline__ float abs_value(uint32_t bits) { return __builtin_bit_cast(float, bits); }
};

// pertoken_quant's nan_to_num(nan=0, posinf=qmax, neginf=-qmax)
__device__ __forceinline__ float scrub(float x, float qmax) {
  if (__builtin_isnan(x)) return 0.f;
  if (__builtin_isinf(x)) return x > 0.f ? qmax : -qmax;
  return x;
}

// the host quantizer's modes scrub NaN / inf before the scale is taken (see scrub)
template <int MODE>
__device__ __forceinline__ f32x8 prepare8(f32x8 v, float qmax) {
  if constexpr (MODE != QMODE_RECIP_TRUNC) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = scrub(v[i], qmax);
  }
  return v;
}

__device__ __forceinline__ float absmax8(const f32x8& v) {
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) m = __builtin_fmaxf(m, __builtin_fabsf(v[i]));
  return m;
}

// x / scale, correctly rounded (see the head of this file)
__device__ __forceinline__ float div_by(float x, float scale, float inv_scale) {
  float q = x * inv_scale;
  q = __builtin_fmaf(__builtin_fmaf(-q, scale, x), inv_scale, q);
  return __builtin_fmaf(__builtin_fmaf(-q, scale, x), inv_scale, q);
}

// the scales whose quotients div_by gives
__device__ __forceinline__ bool div_by_ok(float scale) { return scale >= 0x1p-90f && scale <= 0x1p90f; }

// 8 quantized codes packed little-endian into two dwords; fast: div_by_ok(scale), the same for
// every lane of a row
template <int OUT, int MODE>
__device__ __forceinline__ uint2 quant8(const f32x8& v, float scale, float inv_scale, bool fast) {
  float y[8];
  // the quotient (or product) is rounded to fp32 before the cast, as in the reference
  if (MODE == QMODE_RECIP_TRUNC) {
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = v[i] * inv_scale;
  } else if (fast) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      y[i] = div_by(v[i], scale, inv_scale);
      if constexpr (OUT == QOUT_FP8) y[i] = __builtin_copysignf(y[i], v[i]);   // -0 stays -0
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = v[i] / scale;
  }
  uint32_t w[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(y[4 * h + i]));
    if constexpr (OUT == QOUT_FP8) {
      // hardware fp32 -> OCP e4m3fn conversion, round to nearest even
      int p = __builtin_amdgcn_cvt_pk_fp8_f32(y[4 * h], y[4 * h + 1], 0, false);
      p = __builtin_amdgcn_cvt_pk_fp8_f32(y[4 * h + 2], y[4 * h + 3], p, true);
      w[h] = (uint32_t)p;
    } else {
      uint32_t packed = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int q;
        if constexpr (MODE == QMODE_DIV_NEAREST)
          q = (int)__builtin_rintf(__builtin_fminf(__builtin_fmaxf(y[4 * h + i], -127.f), 127.f));
        else
          q = (int)y[4 * h + i];  // truncation toward zero; |y| <= 127 * (1 + 2^-22) by construction
        packed |= ((uint32_t)q & 0xFFu) << (8 * i);
      }
      w[h] = packed;
    }
  }
  return make_uint2(w[0], w[1]);
}

// 8 output bytes, non-temporal (measured 3-7% faster than plain stores on MI355X)
__device__ __forceinline__ void store8(uint8_t* dst, uint2 v) {
  __builtin_nontemporal_store(__builtin_bit_cast(i32x2q, v), (i32x2q*)dst);
}

// maximum over groups of LANES consecutive lanes
template <int LANES>
__device__ __forceinline__ float lanes_max(float v) {
#pragma unroll
  for (int off = LANES / 2; off >= 1; off >>= 1) v = __builtin_fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// amax of a thread's vectors from the maximum of their bits; `dirty` when they hold NaN or
// infinity (as many of them as `have(s)` says), which are then looked at one by one
template <int IN, int MODE, int VPT, typename Have>
__device__ __forceinline__ float thread_amax(const Raw8<IN> (&raw)[VPT], uint32_t mb, float qmax, Have have, bool& dirty) {
  mb = Raw8<IN>::fold(mb);
  dirty = mb >= Raw8<IN>::kInf;
  if (!dirty) return Raw8<IN>::abs_value(mb);
  float m = 0.f;
#pragma unroll
  for (int s = 0; s < VPT; ++s)
    if (have(s)) m = __builtin_fmaxf(m, absmax8(prepare8<MODE>(raw[s].value(), qmax)));
  return m;
}

// Rows of up to LPR * 8 * VPT elements: LPR lanes per row, 4 waves per workgroup.
template <int IN, int OUT, int MODE, int LPR, int VPT>
__global__ void __launch_bounds__(256) quant_short_rows_kernel(QuantArgs p) {
  constexpr int ESZ = (IN == QIN_F32) ? 4 : 2;
  constexpr float QMAX = (OUT == QOUT_FP8) ? 448.f : 127.f;
  const int N = p.N, lane = threadIdx.x % LPR;
  const long row = (long)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  if (row >= p.M) return;   // whole groups of LPR lanes
  const void* rin = (const uint8_t*)p.in + (size_t)row * N * ESZ;
  uint8_t* rout = (uint8_t*)p.out + (size_t)row * N;
  auto col = [&](int s) { return (s * LPR + lane) * 8; };
  auto have = [&](int s) { return col(s) < N; };
  Raw8<IN> raw[VPT];
  uint32_t mb = 0;
#pragma unroll
  for (int s = 0; s < VPT; ++s)
    if (have(s)) raw[s].load(rin, col(s));
#pragma unroll
  for (int s = 0; s < VPT; ++s)
    if (have(s)) mb = raw[s].max_bits(mb);
  bool dirty;
  const float m = lanes_max<LPR>(thread_amax<IN, MODE>(raw, mb, QMAX, have, dirty));
  float scale = m / QMAX;
  if (scale == 0.f) scale = 1.f;
  const float inv_scale = 1.f / scale;
  if (lane == 0) p.scales[row] = scale;
  const bool fast = div_by_ok(scale);
#pragma unroll
  for (int s = 0; s < VPT; ++s) {
    if (!have(s)) continue;
    f32x8 v = raw[s].value();
    if (dirty) v = prepare8<MODE>(v, QMAX);
    store8(rout + col(s), quant8<OUT, MODE>(v, scale, inv_scale, fast));
  }
}

template <int IN, int OUT, int MODE, int VPT, int NT>
__global__ void __launch_bounds__(NT) quant_rows_kernel(QuantArgs p) {
  constexpr int kQuantSlice = NT * 8;  // elements per workgroup pass
  constexpr int ESZ = (IN == QIN_F32) ? 4 : 2;
  constexpr float QMAX = (OUT == QOUT_FP8) ? 448.f : 127.f;
  const int row = blockIdx.x;
  const int N = p.N;
  const int tid = threadIdx.x;
  const void* rin = (const uint8_t*)p.in + (size_t)row * N * ESZ;
  uint8_t* rout = (uint8_t*)p.out + (size_t)row * N;
  const int nslices = (N + kQuantSlice - 1) / kQuantSlice;
  auto have = [&](int s) { return s * kQuantSlice + tid * 8 < N; };

  // ---- pass 1: row amax (inputs kept in registers when the row fits) ----
  Raw8<IN> raw[VPT > 0 ? VPT : 1];
  float m = 0.f;
  bool dirty = false;
  if constexpr (VPT > 0) {
    uint32_t mb = 0;
#pragma unroll
    for (int s = 0; s < VPT; ++s)
      if (have(s)) raw[s].load(rin, s * kQuantSlice + tid * 8);
#pragma unroll
    for (int s = 0; s < VPT; ++s)
      if (have(s)) mb = raw[s].max_bits(mb);
    m = thread_amax<IN, MODE>(raw, mb, QMAX, have, dirty);
  } else {
    for (int s = 0; s < nslices; ++s) {
      if (!have(s)) continue;
      raw[0].load(rin, s * kQuantSlice + tid * 8);
      bool d;
      m = __builtin_fmaxf(m, thread_amax<IN, MODE>(raw, raw[0].max_bits(0), QMAX, [](int) { return true; }, d));
      dirty |= d;
    }
  }
  __shared__ float red[NT / 64];
  m = lanes_max<64>(m);
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
  m = red[0];
#pragma unroll
  for (int w = 1; w < NT / 64; ++w) m = __builtin_fmaxf(m, red[w]);

  float scale = m / QMAX;
  if (scale == 0.f) scale = 1.f;
  const float inv_scale = 1.f / scale;
  if (tid == 0) p.scales[row] = scale;
  const bool fast = div_by_ok(scale);

  // ---- pass 2: quantize and store 8 codes (8 bytes) per thread per slice ----
  auto emit = [&](const Raw8<IN>& r, int s) {
    f32x8 v = r.value();
    if (dirty) v = prepare8<MODE>(v, QMAX);
    store8(rout + s * kQuantSlice + tid * 8, quant8<OUT, MODE>(v, scale, inv_scale, fast));
  };
  if constexpr (VPT > 0) {
#pragma unroll
    for (int s = 0; s < VPT; ++s)
      if (have(s)) emit(raw[s], s);
  } else {
    for (int s = 0; s < nslices; ++s) {
      if (!have(s)) continue;
      raw[0].load(rin, s * kQuantSlice + tid * 8);
      emit(raw[0], s);
    }
  }
}

// One scale per 128 consecutive elements of a row (blockscale activations), fp8 codes:
//   scale = amax * inv_qmax (1 where that is 0), code = e4m3fn(x / scale),
// the arithmetic of torch's operators on the GPU, where a division by a constant is a product
// with its reciprocal, amax passes NaN on, and the cast keeps NaN's sign.
// 16 lanes per block of 128, each with 8 elements; bound by HBM for many blocks and by its launch
// for few (torch.float16, back-to-back calls from Python: 1024 x 7168 14.9 us against 58.5
// for the operators, 65536 x 256 14.1 against 104).
struct BlockQuantArgs {
  void* out;        // [blocks][128] fp8 codes
  float* scales;    // [blocks]
  const void* in;   // [blocks][128]
  long blocks;
  float inv_qmax;
};

template <int IN>
__global__ void __launch_bounds__(256) quant_blocks_kernel(BlockQuantArgs p) {
  constexpr int ESZ = (IN == QIN_F32) ? 4 : 2;
  const int lane = threadIdx.x % 16;
  const long blk = (long)blockIdx.x * 16 + threadIdx.x / 16;
  if (blk >= p.blocks) return;   // whole groups of 16 lanes
  Raw8<IN> raw;
  raw.load((const uint8_t*)p.in + (size_t)blk * 128 * ESZ, lane * 8);
  uint32_t mb = Raw8<IN>::fold(raw.max_bits(0));
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1) mb = max(mb, (uint32_t)__shfl_xor((int)mb, off, 64));
  const bool finite = mb < Raw8<IN>::kInf;
  float scale = Raw8<IN>::abs_value(mb) * p.inv_qmax;
  if (scale == 0.f) scale = 1.f;
  const f32x8 v = raw.value();
  if (mb > Raw8<IN>::kInf) {   // NaN: the block's first one
    uint32_t first = 0;
    bool nan = false;
#pragma unroll
    for (int i = 7; i >= 0; --i) {
      const float x = v[i];
      if (x != x) {
        nan = true;
        first = __builtin_bit_cast(uint32_t, x);
      }
    }
    const uint64_t m = (__builtin_amdgcn_ballot_w64(nan) >> (threadIdx.x & 48)) & 0xFFFFu;
    first = (uint32_t)__shfl((int)first, (threadIdx.x & 48) + __builtin_ctzll(m), 64);
    scale = __builtin_bit_cast(float, first | 0x00400000u);   // quiet, its payload kept
  }
  if (lane == 0) p.scales[blk] = scale;
  uint2 c = quant8<QOUT_FP8, QMODE_DIV_NEAREST>(v, scale, 1.f / scale, div_by_ok(scale));
  if (!finite) {
    uint32_t w[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float y = v[i] / scale;
      const uint32_t b = __builtin_bit_cast(uint32_t, y);
      const uint32_t code = (b >> 24 & 0x80u) | (y != y ? 0x7Fu : 0u);   // finite / infinite = 0
      w[i / 4] |= code << (8 * (i % 4));
    }
    c = make_uint2(w[0], w[1]);
  }
  store8((uint8_t*)p.out + (size_t)blk * 128 + lane * 8, c);
}

}  // namespace flygemm
