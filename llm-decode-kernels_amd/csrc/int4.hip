// int4 weight format on the GPU: pack, unpack, RTN quantize and the bit-exact dequantizer.
//
// Format (kernels/quant.py:3-10 of the reference): qweight int32 [K/8, N]; nibble i (bits
// 4i..4i+3) of word [r, n] is q[8r+i, n]; scales/zeros [K/G, N]; w = (q - z) * s.
#include "ldk_common.h"

namespace {

// ------------------------------------------------------------------------------ pack / unpack

// One thread per packed word [r, n]; consecutive threads take consecutive n (coalesced).
// The sum of q << 4i is taken modulo 2^32 and reinterpreted as int32, which is what
// quant.py:24-28 computes in int64 for any integer input (for 0..15 it is a plain OR).
__global__ void int4_pack_kernel(const int32_t* __restrict__ q, uint32_t* __restrict__ packed,
                                 int64_t R, int64_t N) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= R * N) return;
  const int64_t r = i / N, n = i - r * N;
  const int32_t* src = q + (8 * r) * N + n;
  uint32_t acc = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) acc += (uint32_t)src[k * N] << (4 * k);
  packed[i] = acc;
}

// q[8r+k, n] = (packed[r, n] >> 4k) & 0xF (quant.py:31-35).
__global__ void int4_unpack_kernel(const uint32_t* __restrict__ packed, int32_t* __restrict__ q,
                                   int64_t R, int64_t N) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= R * N) return;
  const int64_t r = i / N, n = i - r * N;
  const uint32_t w = packed[i];
  int32_t* dst = q + (8 * r) * N + n;
#pragma unroll
  for (int k = 0; k < 8; ++k) dst[k * N] = (int32_t)((w >> (4 * k)) & 0xFu);
}

// ------------------------------------------------------------------------------ RTN quantizer

template <typename T>
__device__ __forceinline__ float load_f32(const T* p);
template <>
__device__ __forceinline__ float load_f32<half_t>(const half_t* p) { return (float)*p; }
template <>
__device__ __forceinline__ float load_f32<float>(const float* p) { return *p; }
template <>
__device__ __forceinline__ float load_f32<uint16_t>(const uint16_t* p) {  // bf16 bits
  return __builtin_bit_cast(float, (uint32_t)*p << 16);
}

// float32 -> storage type with round-to-nearest-even (the `.to(dtype)` of quant.py:49).
template <typename T>
__device__ __forceinline__ T store_cast(float v);
template <>
__device__ __forceinline__ half_t store_cast<half_t>(float v) { return (half_t)v; }
template <>
__device__ __forceinline__ float store_cast<float>(float v) { return v; }
template <>
__device__ __forceinline__ uint16_t store_cast<uint16_t>(float v) {
  uint32_t u = __builtin_bit_cast(uint32_t, v);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);  // quiet NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// One thread per (group g, column n), consecutive threads on consecutive n so that the packed
// words, scales and zeros are written coalesced. Each thread reads its group's G contiguous
// weights of row n twice (min/max pass, then quantize pass; the second pass hits in cache).
//
// The arithmetic is the float32 sequence of quant.py:42-47, each step one IEEE operation:
// scale = max((wmax - wmin) / 15, 1e-6); zero = clamp(rint(-wmin / scale), 0, 15);
// q = clamp(rint(w / scale + zero), 0, 15). Division is correctly rounded (the library is built
// with -fhip-fp32-correctly-rounded-divide-sqrt) and rint rounds half to even like torch.round.
template <typename T>
__global__ void quantize_rtn_kernel(const T* __restrict__ w, uint32_t* __restrict__ qweight,
                                    T* __restrict__ scales, T* __restrict__ zeros, int64_t N,
                                    int64_t K, int G) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t ng = K / G;
  if (i >= ng * N) return;
  const int64_t g = i / N, n = i - g * N;
  const T* src = w + n * K + g * G;
  float wmin = load_f32(src), wmax = wmin;
  for (int k = 1; k < G; ++k) {
    const float v = load_f32(src + k);
    wmin = fminf(wmin, v);
    wmax = fmaxf(wmax, v);
  }
  const float scale = fmaxf((wmax - wmin) / 15.0f, 1e-6f);
  // Compare-select clamp keeps a -0.0 from rint, as torch's CPU clamp and numpy's clip do.
  float zero = rintf(-wmin / scale);
  zero = zero < 0.0f ? 0.0f : zero;
  zero = zero > 15.0f ? 15.0f : zero;
  uint32_t* dst = qweight + (g * (G / 8)) * N + n;
  for (int r = 0; r < G / 8; ++r) {
    uint32_t word = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float v = load_f32(src + 8 * r + k);
      const float q = fminf(fmaxf(rintf(v / scale + zero), 0.0f), 15.0f);
      word |= (uint32_t)q << (4 * k);
    }
    dst[(int64_t)r * N] = word;
  }
  scales[i] = store_cast<T>(scale);
  zeros[i] = store_cast<T>(zero);
}

// The same quantizer with the weights read once and in whole lines, for groups of 8 * LPG weights
// (LPG = 4 .. 64, a power of two) and 16-byte aligned weights. A workgroup takes one group of 64
// columns: LPG lanes hold a column's group, 8 weights (one packed word) each, and meet for its
// minimum and maximum through DPP (min and max do not depend on the order). The words are turned
// through LDS, so a packed row is stored as 256 contiguous bytes. The arithmetic per weight is the
// kernel above's. Bound by the vector instructions, the quotient per weight above all (85% busy). On
// 14336 x 4096 fp16 (149 MB) the one-thread-per-group kernel took 968 us (each lane walking its own
// 256-byte run, twice); this 38, 3.9 TB/s (51 us with the IEEE division per weight).
constexpr int kQCols = 64;

template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return ldk::u2f(__builtin_amdgcn_update_dpp(0u, ldk::f2u(v), CTRL, 0xf, 0xf, false));
}
// min and max over aligned runs of LPG lanes, in every lane
template <int LPG>
__device__ __forceinline__ void run_min_max(float& lo, float& hi) {
  auto meet = [&](float a, float b) {
    lo = fminf(lo, a);
    hi = fmaxf(hi, b);
  };
  meet(dpp_mov<0xB1>(lo), dpp_mov<0xB1>(hi));                          // quad_perm: lane ^ 1
  meet(dpp_mov<0x4E>(lo), dpp_mov<0x4E>(hi));                          // quad_perm: lane ^ 2
  if constexpr (LPG >= 8) meet(dpp_mov<0x141>(lo), dpp_mov<0x141>(hi));   // half-row mirror: the other quad
  if constexpr (LPG >= 16) meet(dpp_mov<0x140>(lo), dpp_mov<0x140>(hi));  // row mirror: the other half-row
  if constexpr (LPG >= 32) {
    const auto a = __builtin_amdgcn_permlane16_swap(ldk::f2u(lo), ldk::f2u(lo), false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(ldk::f2u(hi), ldk::f2u(hi), false, false);
    lo = fminf(ldk::u2f(a[0]), ldk::u2f(a[1]));
    hi = fmaxf(ldk::u2f(b[0]), ldk::u2f(b[1]));
  }
  if constexpr (LPG >= 64) {
    const auto a = __builtin_amdgcn_permlane32_swap(ldk::f2u(lo), ldk::f2u(lo), false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(ldk::f2u(hi), ldk::f2u(hi), false, false);
    lo = fminf(ldk::u2f(a[0]), ldk::u2f(a[1]));
    hi = fmaxf(ldk::u2f(b[0]), ldk::u2f(b[1]));
  }
}

template <typename T, int LPG>
__global__ __launch_bounds__(256) void quantize_rtn_tile_kernel(const T* __restrict__ w, uint32_t* __restrict__ qweight,
                                                                T* __restrict__ scales, T* __restrict__ zeros, int64_t N,
                                                                int64_t K) {
  typedef T tv_t __attribute__((ext_vector_type(8)));
  constexpr int CPP = 256 / LPG;                       // columns per pass of the workgroup
  constexpr int P = kQCols / CPP > 0 ? kQCols / CPP : 1;  // passes
  static_assert(P * CPP == kQCols, "whole passes");
  __shared__ uint32_t words[LPG][kQCols + 1];
  __shared__ float sc[kQCols], zr[kQCols];
  const int tid = threadIdx.x, r = tid % LPG;
  const int64_t ng = K / (8 * LPG);
  const int64_t g = blockIdx.x % ng, n0 = blockIdx.x / ng * kQCols;
  tv_t v[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {  // columns past N read the last one again; they store nothing
    const int64_t n = min(n0 + p * CPP + tid / LPG, N - 1);
    v[p] = *reinterpret_cast<const tv_t*>(w + n * K + (g * LPG + r) * 8);
  }
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int c = p * CPP + tid / LPG;
    float f[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const T e = v[p][k];
      f[k] = load_f32(&e);
    }
    float wmin = f[0], wmax = f[0];
#pragma unroll
    for (int k = 1; k < 8; ++k) {
      wmin = fminf(wmin, f[k]);
      wmax = fmaxf(wmax, f[k]);
    }
    run_min_max<LPG>(wmin, wmax);
    const float scale = fmaxf((wmax - wmin) / 15.0f, 1e-6f);
    float zero = rintf(-wmin / scale);
    zero = zero < 0.0f ? 0.0f : zero;
    zero = zero > 15.0f ? 15.0f : zero;
    // w / scale: with y the rounded reciprocal, each fma pair takes the quotient one Newton step
    // nearer, and the second rounds it correctly (P. Markstein, IBM J. Res. Dev. 34, 1990) while
    // nothing overflows or loses bits to underflow: 5 operations instead of the division's 11.
    // Quotients small enough to underflow in the residual round to the same integer. Groups out
    // of that range (infinities among them) divide.
    const float y = 1.0f / scale;
    uint32_t word = 0;
    auto put = [&](int k, float quot) __attribute__((always_inline)) {
      const float q = fminf(fmaxf(rintf(quot + zero), 0.0f), 15.0f);
      word |= (uint32_t)q << (4 * k);
    };
    if (__all(scale < 1e30f && fmaxf(fabsf(wmin), fabsf(wmax)) * y < 1e37f)) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float q = f[k] * y;
        q = __builtin_fmaf(__builtin_fmaf(-scale, q, f[k]), y, q);
        put(k, __builtin_fmaf(__builtin_fmaf(-scale, q, f[k]), y, q));
      }
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) put(k, f[k] / scale);
    }
    words[r][c] = word;
    if (r == 0) {
      sc[c] = scale;
      zr[c] = zero;
    }
  }
  __syncthreads();
  const int c = tid & (kQCols - 1);
  if (n0 + c >= N) return;
  for (int q = tid / kQCols; q < LPG; q += 256 / kQCols) qweight[(g * LPG + q) * N + n0 + c] = words[q][c];
  if (tid < kQCols) {
    scales[g * N + n0 + c] = store_cast<T>(sc[c]);
    zeros[g * N + n0 + c] = store_cast<T>(zr[c]);
  }
}

// ---------------------------------------------------------------------------------- dequant

// out [N, K] fp16 = (q - z) * s, one fp16 rounding (reference.py:27-36). A workgroup takes 16 packed
// rows of 64 columns: it reads whole 256-byte runs of each packed row, and turns the decoded
// 16-byte pieces through LDS (column c's piece r at slot r ^ (c % 16), so neither side has bank
// conflicts beyond the 16-byte accesses' own), so every output row is stored as 256 contiguous
// bytes. At the copy's rate on 14336 x 4096 (149 MB): 26 us, 5.8 TB/s, where reading one word per lane
// down a column took 45; under 1M weights that, without the LDS round, was 0.2-0.5 us faster (512 x 256
// 2.4 against 2.9 us).
constexpr int kDRows = 16, kDCols = 64;

__global__ __launch_bounds__(256) void w4a16_dequant_kernel(const uint32_t* __restrict__ qw,
                                                            const half_t* __restrict__ sc,
                                                            const half_t* __restrict__ zr,
                                                            half_t* __restrict__ out, int64_t N,
                                                            int64_t K, int gshift_rows) {
  __shared__ __align__(16) half8_t tile[kDCols][kDRows];
  const int64_t R = K / 8, rt = (R + kDRows - 1) / kDRows;
  const int64_t t = ldk::tile_index(), r0 = t % rt * kDRows, n0 = t / rt * kDCols;
  if (n0 >= N) return;  // uniform
  const int tid = threadIdx.x, c = tid & (kDCols - 1);
  const int64_t nc = min(n0 + c, N - 1);  // columns and rows past the end repeat the last ones
  uint32_t word[4];
  half_t s[4], z[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t r = min(r0 + tid / kDCols + 4 * i, R - 1), g = r >> gshift_rows;
    word[i] = qw[r * N + nc];
    s[i] = sc[g * N + nc];
    z[i] = zr[g * N + nc];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = tid / kDCols + 4 * i;
    half8_t v;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const half_t q = (half_t)(float)((word[i] >> (4 * k)) & 0xFu);
      v[k] = (half_t)(q - z[i]) * s[i];
    }
    tile[c][r ^ (c & (kDRows - 1))] = v;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int col = tid / kDRows + 16 * i, r = tid & (kDRows - 1);
    if (n0 + col < N && r0 + r < R)
      *reinterpret_cast<half8_t*>(out + (n0 + col) * K + 8 * (r0 + r)) = tile[col][r ^ (col & (kDRows - 1))];
  }
}

inline int blocks_for(int64_t n, int threads) { return (int)((n + threads - 1) / threads); }

int log2_exact(int64_t v) {
  if (v <= 0 || (v & (v - 1))) return -1;
  int s = 0;
  while ((int64_t(1) << s) < v) ++s;
  return s;
}

// Launches the tiled quantizer for group sizes 32 .. 512 (powers of two), 16-byte aligned weights and
// fewer than 2^24 tiles (a launch holds fewer than 2^32 threads per grid dimension), else the
// one-thread-per-group one.
template <typename T>
void launch_quantize(const T* w, uint32_t* qweight, T* scales, T* zeros, int64_t N, int64_t K, int G, hipStream_t s) {
  const int64_t tiles = (K / G) * ((N + kQCols - 1) / kQCols);
  auto tiled = [&](auto kernel) { kernel<<<(unsigned)tiles, 256, 0, s>>>(w, qweight, scales, zeros, N, K); };
  if (ldk::aligned(w, 16) && tiles < (int64_t(1) << 24)) {
    switch (G) {
      case 32: return tiled(quantize_rtn_tile_kernel<T, 4>);
      case 64: return tiled(quantize_rtn_tile_kernel<T, 8>);
      case 128: return tiled(quantize_rtn_tile_kernel<T, 16>);
      case 256: return tiled(quantize_rtn_tile_kernel<T, 32>);
      case 512: return tiled(quantize_rtn_tile_kernel<T, 64>);
    }
  }
  quantize_rtn_kernel<T><<<blocks_for((K / G) * N, 256), 256, 0, s>>>(w, qweight, scales, zeros, N, K, G);
}

}  // namespace

extern "C" int ldk_int4_pack(const int32_t* q, int32_t* packed, int64_t K, int64_t N, void* stream) {
  if (!q || !packed) return ldk::fail(LDK_ERR_INVALID, "int4_pack: null pointer");
  if (K <= 0 || N <= 0 || K % 8) return ldk::fail(LDK_ERR_INVALID, "int4_pack: K=%lld must be a positive multiple of 8, N=%lld > 0", (long long)K, (long long)N);
  const int64_t R = K / 8;
  if (R * N > (int64_t)INT32_MAX * 256) return ldk::fail(LDK_ERR_UNSUPPORTED, "int4_pack: too large");
  (void)hipGetLastError();
  int4_pack_kernel<<<blocks_for(R * N, 256), 256, 0, (hipStream_t)stream>>>(q, (uint32_t*)packed, R, N);
  return ldk::check_launch("int4_pack");
}

extern "C" int ldk_int4_unpack(const int32_t* packed, int32_t* q, int64_t K, int64_t N, void* stream) {
  if (!q || !packed) return ldk::fail(LDK_ERR_INVALID, "int4_unpack: null pointer");
  if (K <= 0 || N <= 0 || K % 8) return ldk::fail(LDK_ERR_INVALID, "int4_unpack: K=%lld must be a positive multiple of 8, N=%lld > 0", (long long)K, (long long)N);
  const int64_t R = K / 8;
  (void)hipGetLastError();
  int4_unpack_kernel<<<blocks_for(R * N, 256), 256, 0, (hipStream_t)stream>>>((const uint32_t*)packed, q, R, N);
  return ldk::check_launch("int4_unpack");
}

extern "C" int ldk_quantize_rtn(const void* w, int dtype, int32_t* qweight, void* scales, void* zeros,
                                int64_t N, int64_t K, int group_size, void* stream) {
  if (!w || !qweight || !scales || !zeros) return ldk::fail(LDK_ERR_INVALID, "quantize_rtn: null pointer");
  if (N <= 0 || K <= 0 || group_size <= 0 || group_size % 8 || K % group_size)
    return ldk::fail(LDK_ERR_INVALID, "quantize_rtn: K=%lld must be a multiple of group_size=%d, which must be a multiple of 8", (long long)K, group_size);
  hipStream_t s = (hipStream_t)stream;
  (void)hipGetLastError();
  switch (dtype) {
    case LDK_F16:
      launch_quantize((const half_t*)w, (uint32_t*)qweight, (half_t*)scales, (half_t*)zeros, N, K, group_size, s);
      break;
    case LDK_BF16:
      launch_quantize((const uint16_t*)w, (uint32_t*)qweight, (uint16_t*)scales, (uint16_t*)zeros, N, K, group_size, s);
      break;
    case LDK_F32:
      launch_quantize((const float*)w, (uint32_t*)qweight, (float*)scales, (float*)zeros, N, K, group_size, s);
      break;
    default:
      return ldk::fail(LDK_ERR_INVALID, "quantize_rtn: unknown dtype %d", dtype);
  }
  return ldk::check_launch("quantize_rtn");
}

extern "C" int ldk_w4a16_dequant(const int32_t* qweight, const void* scales, const void* zeros, void* out,
                                 int64_t N, int64_t K, int group_size, void* stream) {
  if (!qweight || !scales || !zeros || !out) return ldk::fail(LDK_ERR_INVALID, "w4a16_dequant: null pointer");
  const int gsh = log2_exact(group_size);
  if (N <= 0 || K <= 0 || K % 8 || gsh < 3 || K % group_size)
    return ldk::fail(LDK_ERR_INVALID, "w4a16_dequant: need K %% 8 == 0, group_size a power of two >= 8 dividing K (K=%lld, group_size=%d)", (long long)K, group_size);
  if (!ldk::aligned(out, 16)) return ldk::fail(LDK_ERR_ALIGN, "w4a16_dequant: out must be 16-byte aligned");
  const int64_t tiles = ((N + kDCols - 1) / kDCols) * ((K / 8 + kDRows - 1) / kDRows);
  if (!ldk::tiles_fit(tiles)) return ldk::fail(LDK_ERR_UNSUPPORTED, "w4a16_dequant: too large");
  (void)hipGetLastError();
  w4a16_dequant_kernel<<<ldk::tile_grid(tiles), 256, 0, (hipStream_t)stream>>>(
      (const uint32_t*)qweight, (const half_t*)scales, (const half_t*)zeros, (half_t*)out, N, K, gsh - 3);
  return ldk::check_launch("w4a16_dequant");
}
