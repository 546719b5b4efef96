// Per-row activation quantiser: the producer of the indexer's low-precision q / k.
//
//   amax  = max(max_j |x[r, j]|, 1e-4)
//   scale = amax / QMAX                       (round_scale: 2^ceil(log2(amax / QMAX)))
//   y     = cvt(clamp(x / scale, -QMAX, QMAX))
//
// QMAX = 127 with round-half-to-even to int8 (examples/deepseek_v4/act_quant.py:33-92 kernel,
// :118-142 golden), or 448 with round-to-nearest-even to OCP fp8 e4m3fn (the same recipe for
// the fp8 indexer inputs).  HBM bound: (input bytes + 1) per element, plus 4 B of scale per row.
//
// Aligned rows of up to 2048 16-byte chunks (act_quant_rows_kernel): a row is held in the registers
// of a group of lanes, as many as it has chunks (up to the wave), so the 256-byte rows of a 128-wide
// head fill the wave four at a time and are read once: 262144 bf16 rows of 128 take 17.4 us (5.8 TB/s)
// against 84.2 with a wave per row, where 16 of 64 lanes loaded; 4681 rows of 7168 23.7 against 31.6.  Other rows (act_quant_kernel): one wave per
// row, a pass for the absolute maximum and a pass that scales, converts and stores.
#include "common.hpp"

namespace dsa {

enum QuantIn : int { kQInBf16 = 1, kQInFp16 = 2, kQInFp32 = 3 };
enum QuantOut : int { kQOutFp8 = 0, kQOutInt8 = 4 };

template <int kIn>
struct QIn;
template <> struct QIn<kQInBf16> {
  typedef uint16_t T;
  static __device__ __forceinline__ float f(T v) { return __uint_as_float((uint32_t)v << 16); }
};
template <> struct QIn<kQInFp16> {
  typedef uint16_t T;
  static __device__ __forceinline__ float f(T v) { return (float)__builtin_bit_cast(_Float16, v); }
};
template <> struct QIn<kQInFp32> {
  typedef float T;
  static __device__ __forceinline__ float f(T v) { return v; }
};

// 2^ceil(log2(v)) for a positive normal v, from its bits (exponent + 1 unless the
// mantissa is zero): act_quant.py:96-109.
__device__ __forceinline__ float pow2_ceil(float v) {
  const uint32_t b = __float_as_uint(v);
  const int e = (int)((b >> 23) & 0xff) - 127 + ((b & 0x7fffff) ? 1 : 0);
  return __uint_as_float((uint32_t)(e + 127) << 23);
}

// One value to the output type: int8 after round-half-even, fp8 e4m3fn by the
// hardware conversion (round to nearest even; the input is already within +-448).
template <int kOut>
__device__ __forceinline__ uint8_t quant_one(float v) {
  if constexpr (kOut == kQOutInt8) {
    return (uint8_t)(int8_t)(int)__builtin_rintf(v);
  } else {
    return (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(v, 0.f, 0, false) & 0xff);
  }
}

// Every row starts on 16 bytes of input and on the output's store width, and holds whole 16-byte chunks.
template <class T>
__host__ __device__ __forceinline__ bool quant_aligned(const void* x, int n, const void* y) {
  return ((n * (int64_t)sizeof(T)) & 15) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0 &&
         (reinterpret_cast<uintptr_t>(y) & 7) == 0;
}

// Lanes of a row group reduce among themselves.
template <int kL>
__device__ __forceinline__ float group_max(float v) {
#pragma unroll
  for (int o = kL / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
  return v;
}

// x / s for |x| <= s * QMAX, equal to the IEEE quotient after the conversion: with r = 1 / s
// correctly rounded, q = fma(-fma(x r, s, -x), r, x r) is the correctly rounded quotient (P.
// Markstein, "Computation of elementary functions on the IBM RISC System/6000 processor", IBM J.
// Res. Dev. 34(1), 1990), 3 operations against the ~10 of a general divide (the divides of a
// 262144 x 128 call cost about as much as its memory traffic).  The residual is inexact only for
// |x| < 2^-100, whose quotient (s >= 2^-23) converts to zero either way; an infinite s (r = 0) is
// left to the general divide by the caller.
__device__ __forceinline__ float div_by(float x, float s, float r) {
  const float q = x * r;
  return fmaf(-fmaf(q, s, -x), r, q);  // the signs keep x = -0 negative
}

// Four values to the output type, packed in order.
template <int kOut>
__device__ __forceinline__ uint32_t quant_four(const float (&v)[4]) {
  constexpr float kQMax = kOut == kQOutInt8 ? 127.f : 448.f;
  float c[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) c[i] = fminf(fmaxf(v[i], -kQMax), kQMax);
  if constexpr (kOut == kQOutInt8) {
    uint32_t w = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) w |= ((uint32_t)(int)__builtin_rintf(c[i]) & 0xffu) << (8 * i);
    return w;
  } else {
    const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(c[0], c[1], 0, false);
    return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c[2], c[3], lo, true);
  }
}

// kL lanes hold a row of nv 16-byte chunks, chunk l + kL * i in lane l; each group takes kR rows,
// whose loads all go out before the first is used.
template <int kIn, int kOut, int kL, int kC, int kR>
__global__ __launch_bounds__(256) void act_quant_rows_kernel(const void* __restrict__ xv, int64_t rows, int nv,
                                                             uint8_t* __restrict__ y, float* __restrict__ scales,
                                                             int round_scale) {
  typedef typename QIn<kIn>::T T;
  constexpr int kVec = 16 / sizeof(T);
  constexpr int kGroups = 256 / kL;
  constexpr float kQMax = kOut == kQOutInt8 ? 127.f : 448.f;
  const int l = threadIdx.x & (kL - 1);
  const int64_t r0 = (int64_t)blockIdx.x * (kGroups * kR) + threadIdx.x / kL;
  u32x4 w[kR][kC];
#pragma unroll
  for (int j = 0; j < kR; ++j) {
    const int64_t r = r0 + j * kGroups;
#pragma unroll
    for (int i = 0; i < kC; ++i) {
      const int c = l + kL * i;
      w[j][i] = u32x4{0, 0, 0, 0};
      if (r < rows && c < nv) w[j][i] = static_cast<const u32x4*>(xv)[r * nv + c];
    }
  }
#pragma unroll
  for (int j = 0; j < kR; ++j) {
    const int64_t r = r0 + j * kGroups;
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < kC; ++i) {
      T e[kVec];
      __builtin_memcpy(e, &w[j][i], 16);
#pragma unroll
      for (int k = 0; k < kVec; ++k) amax = fmaxf(amax, fabsf(QIn<kIn>::f(e[k])));
    }
    amax = fmaxf(group_max<kL>(amax), 1e-4f);
    float scale = amax / kQMax;
    if (round_scale) scale = pow2_ceil(scale);
    if (r >= rows) continue;
    if (l == 0) scales[r] = scale;
    const bool finite = scale < __builtin_huge_valf();
    const float rs = 1.f / scale;
#pragma unroll
    for (int i = 0; i < kC; ++i) {
      const int c = l + kL * i;
      if (c >= nv) break;
      T e[kVec];
      __builtin_memcpy(e, &w[j][i], 16);
      uint32_t out[kVec / 4];
#pragma unroll
      for (int k = 0; k < kVec; k += 4) {
        float v[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const float x = QIn<kIn>::f(e[k + m]);
          v[m] = finite ? div_by(x, scale, rs) : x / scale;
        }
        out[k / 4] = quant_four<kOut>(v);
      }
      if constexpr (kVec == 8) {
        reinterpret_cast<u32x2*>(y)[r * nv + c] = u32x2{out[0], out[1]};
      } else {
        reinterpret_cast<uint32_t*>(y)[r * nv + c] = out[0];
      }
    }
  }
}

template <int kIn, int kOut>
__global__ __launch_bounds__(256) void act_quant_kernel(const void* __restrict__ xv, int64_t rows, int n,
                                                        uint8_t* __restrict__ y, float* __restrict__ scales,
                                                        int round_scale) {
  typedef typename QIn<kIn>::T T;
  constexpr int kVec = 16 / sizeof(T);  // elements per 16-byte load
  constexpr float kQMax = kOut == kQOutInt8 ? 127.f : 448.f;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t r = (int64_t)blockIdx.x * (256 / kWave) + threadIdx.x / kWave;
  if (r >= rows) return;
  const T* x = static_cast<const T*>(xv) + r * n;
  uint8_t* yr = y + r * n;
  // 16-byte row loads (and 8- / 4-byte stores) when every row starts aligned.
  const int nv = quant_aligned<T>(xv, n, y) ? n / kVec : 0;  // whole 16-byte chunks

  float amax = 0.f;
  for (int c = lane; c < nv; c += kWave) {
    const u32x4 w = *reinterpret_cast<const u32x4*>(x + (int64_t)c * kVec);
    const T* e = reinterpret_cast<const T*>(&w);
#pragma unroll
    for (int i = 0; i < kVec; ++i) amax = fmaxf(amax, fabsf(QIn<kIn>::f(e[i])));
  }
  for (int j = nv * kVec + lane; j < n; j += kWave) amax = fmaxf(amax, fabsf(QIn<kIn>::f(x[j])));
  amax = wave_max(amax);
  amax = fmaxf(amax, 1e-4f);
  float scale = amax / kQMax;
  if (round_scale) scale = pow2_ceil(scale);
  if (lane == 0) scales[r] = scale;

  for (int c = lane; c < nv; c += kWave) {
    const u32x4 w = *reinterpret_cast<const u32x4*>(x + (int64_t)c * kVec);
    const T* e = reinterpret_cast<const T*>(&w);
    uint8_t q[kVec];
#pragma unroll
    for (int i = 0; i < kVec; ++i) q[i] = quant_one<kOut>(fminf(fmaxf(QIn<kIn>::f(e[i]) / scale, -kQMax), kQMax));
    if constexpr (kVec == 8) {
      *reinterpret_cast<uint2*>(yr + (int64_t)c * kVec) = *reinterpret_cast<const uint2*>(q);
    } else {
      *reinterpret_cast<uint32_t*>(yr + (int64_t)c * kVec) = *reinterpret_cast<const uint32_t*>(q);
    }
  }
  for (int j = nv * kVec + lane; j < n; j += kWave)
    yr[j] = quant_one<kOut>(fminf(fmaxf(QIn<kIn>::f(x[j]) / scale, -kQMax), kQMax));
}

template <int kIn, int kOut, int kL, int kC, int kR>
static void launch_quant_rows(const void* x, int64_t rows, int nv, uint8_t* y, float* scales, int round_scale,
                              hipStream_t stream) {
  constexpr int64_t kPerBlock = (256 / kL) * kR;
  const dim3 grid((unsigned)((rows + kPerBlock - 1) / kPerBlock)), block(256);
  hipLaunchKernelGGL((act_quant_rows_kernel<kIn, kOut, kL, kC, kR>), grid, block, 0, stream, x, rows, nv, y, scales,
                     round_scale);
}

// Rows of up to one chunk per lane: two rows per lane group (twice the loads in flight) where 4096
// workgroups are left, one otherwise.  262144 bf16 rows of 128: 18.3 us with one, 17.6 with two, 20.5
// with four; 32768 rows: 4.1, 4.3 and 5.2.
constexpr int kRowsPerGroup = 2;

template <int kIn, int kOut, int kL>
static void launch_quant_short(const void* x, int64_t rows, int nv, uint8_t* y, float* scales, int round_scale,
                               hipStream_t stream) {
  if (rows * kL >= (int64_t)4096 * 256 * kRowsPerGroup)
    launch_quant_rows<kIn, kOut, kL, 1, kRowsPerGroup>(x, rows, nv, y, scales, round_scale, stream);
  else
    launch_quant_rows<kIn, kOut, kL, 1, 1>(x, rows, nv, y, scales, round_scale, stream);
}

template <int kIn, int kOut>
static hipError_t launch_quant(const void* x, int64_t rows, int n, uint8_t* y, float* scales, int round_scale,
                               hipStream_t stream) {
  typedef typename QIn<kIn>::T T;
  constexpr int kVec = 16 / sizeof(T);
  const int64_t nv = quant_aligned<T>(x, n, y) ? n / kVec : 0;
  if (nv == 0 || nv > 2048) {
    const dim3 grid((unsigned)((rows + 3) / 4)), block(256);
    hipLaunchKernelGGL((act_quant_kernel<kIn, kOut>), grid, block, 0, stream, x, rows, n, y, scales, round_scale);
  } else if (nv <= 8) {
    launch_quant_short<kIn, kOut, 8>(x, rows, (int)nv, y, scales, round_scale, stream);
  } else if (nv <= 16) {
    launch_quant_short<kIn, kOut, 16>(x, rows, (int)nv, y, scales, round_scale, stream);
  } else if (nv <= 32) {
    launch_quant_short<kIn, kOut, 32>(x, rows, (int)nv, y, scales, round_scale, stream);
  } else if (nv <= 64) {
    launch_quant_short<kIn, kOut, 64>(x, rows, (int)nv, y, scales, round_scale, stream);
  } else if (nv <= 128) {
    launch_quant_rows<kIn, kOut, 64, 2, 1>(x, rows, (int)nv, y, scales, round_scale, stream);
  } else if (nv <= 256) {
    launch_quant_rows<kIn, kOut, 64, 4, 1>(x, rows, (int)nv, y, scales, round_scale, stream);
  } else if (nv <= 512) {
    launch_quant_rows<kIn, kOut, 64, 8, 1>(x, rows, (int)nv, y, scales, round_scale, stream);
  } else if (nv <= 1024) {
    launch_quant_rows<kIn, kOut, 64, 16, 1>(x, rows, (int)nv, y, scales, round_scale, stream);
  } else {
    launch_quant_rows<kIn, kOut, 64, 32, 1>(x, rows, (int)nv, y, scales, round_scale, stream);
  }
  return hipGetLastError();
}

template <int kIn>
static hipError_t launch_quant_in(int out_kind, const void* x, int64_t rows, int n, uint8_t* y, float* scales,
                                  int round_scale, hipStream_t stream) {
  return out_kind == kQOutInt8 ? launch_quant<kIn, kQOutInt8>(x, rows, n, y, scales, round_scale, stream)
                               : launch_quant<kIn, kQOutFp8>(x, rows, n, y, scales, round_scale, stream);
}

// Caller validated: in_kind in {bf16, fp16, fp32}, out_kind in {fp8, int8}, rows * n < 2^62, n < 2^31.
hipError_t launch_act_quant(int in_kind, const void* x, int64_t rows, int64_t n, int out_kind, void* y,
                            float* scales, int round_scale, hipStream_t stream) {
  if (rows == 0 || n == 0) return hipSuccess;
  uint8_t* yb = static_cast<uint8_t*>(y);
  switch (in_kind) {
    case kQInBf16: return launch_quant_in<kQInBf16>(out_kind, x, rows, (int)n, yb, scales, round_scale, stream);
    case kQInFp16: return launch_quant_in<kQInFp16>(out_kind, x, rows, (int)n, yb, scales, round_scale, stream);
    case kQInFp32: return launch_quant_in<kQInFp32>(out_kind, x, rows, (int)n, yb, scales, round_scale, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace dsa
