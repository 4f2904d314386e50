// fp32 products on the fp16 matrix pipe, three instructions per product, for long convolutions (included by convmm.hip).
//
// A float x is taken times a power of two 2^e and written as h + l / 2^12 with h = fp16(x 2^e) and l = fp16 of 2^12 times
// what h leaves (after Ootomo and Yokota, "Recovering single precision accuracy from Tensor Cores while surpassing the FP32
// theoretical peak performance", IJHPCA 36, 2022). For |x 2^e| from 2^-14 to 2^15 that is x to one unit in its last place: the
// remainder has up to 12 significant bits and a sign, l keeps 11 bits. The product of two floats is
// h h' + (h l' + l h') / 2^12; what is left out, l l' / 2^24, is 2^-22 of the product at the very most, so a product is held to
// 2^-21 of itself at worst. hh' and the two small products are summed in fp32 accumulators of their own. Either split costs 6e-8 of the result's norm, which a fourth
// product (l l') does not change (8.6e-8 at 48 terms with three and with four), so short sums are left to the six products
// of bf16 parts (convmm.hip), whose error starts at 4e-8 but grows with the root of the number of terms. The GEMM of
// conv_halves.h therefore also moves the sum of the large products to a third accumulator every kFoldTerms terms, so that a sum
// of 2304 terms is rounded some 25 times at its full size and not 144 times (a product of fp16 parts has 22 bits, so, unlike
// one of bf16 parts, it is rounded with every addition), and the weight gradient takes shorter partial sums. Error against 64 bits,
// normally distributed terms, K = 1152 / 2304 / 8192: 1.2e-7 / 1.3e-7 / 1.4e-7 in conv_halves.h; six bf16 products 2.0e-7 / 2.9e-7 /
// 5.7e-7; the fp32 instruction three times that. Sums are given to these kernels where their error is no larger than that of the
// others for operands half of which are zero, too (convmm.hip: convHalves, convGradWeight).
//
// The exponent e comes from the largest finite element of what shares one - an image, a weight row, the images of a partial
// weight gradient - so nothing overflows; and the parts are only used where the smallest non-zero element of it, times 2^e, is
// 2^-14 or more too (fitsHalves: within 2^28 of the largest). What spans more goes to the six products of bf16 parts, which
// are exact for elements of every size. Either kernel family looks both numbers up (rangesKernel: a pass of its own over the
// operands) before it starts. Sums that are not finite are computed again with the fp32 instruction.
#pragma once

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));

constexpr int kMaxSlots = 64;          // slices of an image

// x: the largest finite |x|, as its bits; y: the smallest non-zero |x|, as its bits less one (all ones: there is none)
__device__ __forceinline__ uint2 noRange() { return make_uint2(0u, 0xffffffffu); }
__device__ __forceinline__ uint2 joinRanges(uint2 a, uint2 b) { return make_uint2(max(a.x, b.x), min(a.y, b.y)); }
__device__ __forceinline__ uint2 addToRange(uint2 r, float x) {
  const unsigned u = __float_as_uint(x) & 0x7fffffffu;
  return make_uint2(u < 0x7f800000u ? max(r.x, u) : r.x, min(r.y, u - 1u));
}
// of `lanes` neighbouring lanes (a power of two)
__device__ __forceinline__ uint2 lanesRange(uint2 r, int lanes) {
  for (int d = lanes >> 1; d > 0; d >>= 1)
    r = joinRanges(r, make_uint2((unsigned)__shfl_xor((int)r.x, d), (unsigned)__shfl_xor((int)r.y, d)));
  return r;
}
__device__ __forceinline__ uint2 blockRange(uint2 r, uint2 *red) {
  r = lanesRange(r, dev::kWave);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = r;
  __syncthreads();
  return joinRanges(joinRanges(red[0], red[1]), joinRanges(red[2], red[3]));
}
// e with 2^14 <= |x| 2^e < 2^15 for the largest |x| (its bits; a subnormal one counts as 2^-127)
__device__ __forceinline__ int exponentFor(unsigned mostBits) { return mostBits ? 14 + 127 - (int)(mostBits >> 23) : 0; }
__device__ __forceinline__ bool fitsHalves(uint2 r, int e) {
  return r.y == 0xffffffffu || __builtin_amdgcn_ldexpf(__uint_as_float(r.y + 1u), e) >= 0x1p-14f;
}

// rows[row] = range of a weight row (the first workgroups: the longest), slots[image * nSlots + slice] = range of a slice of the
// image. Bound by memory: the split behind it finds what still fits the Infinity Cache there.
struct RangeArgs {
  const float *x;          // images of perImg floats, nSlots slices of perSlice each
  uint2 *slots;
  long perImg;
  int perSlice, nSlots;
  bool vec;                // perImg % 4 == 0, perSlice % 4 == 0, aligned base
  const float *w;          // element (row, channel, tap) at row * rs + channel * cs + tap
  uint2 *rows;
  int M, rs, cs, C, taps;
};
__global__ void __launch_bounds__(dev::kBlock) rangesKernel(RangeArgs a) {
  __shared__ uint2 red[4];
  uint2 r = noRange();
  const int t = threadIdx.x;
  if ((int)blockIdx.x < a.M) {
    const float *src = a.w + (long)blockIdx.x * a.rs;
    const int n = a.C * a.taps;
    for (int i0 = t; i0 < n; i0 += 8 * dev::kBlock) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {  // (elements past the last repeat it)
        const int i = min(i0 + u * dev::kBlock, n - 1), c = i / a.taps;
        v[u] = src[(long)c * a.cs + (i - c * a.taps)];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) r = addToRange(r, v[u]);
    }
    r = blockRange(r, red);
    if (t == 0) a.rows[blockIdx.x] = r;
    return;
  }
  const int slot = blockIdx.x - a.M, img = slot / a.nSlots, slice = slot - img * a.nSlots;
  const long b = (long)slice * a.perSlice, e = min(a.perImg, b + a.perSlice);
  const float *src = a.x + img * a.perImg;
  if (a.vec) {
    const float4 *s4 = reinterpret_cast<const float4 *>(src);
    auto add = [&](const float4 &v) { r = addToRange(addToRange(addToRange(addToRange(r, v.x), v.y), v.z), v.w); };
    long i = (b >> 2) + t;
    for (; i + 3 * dev::kBlock < e >> 2; i += 4 * dev::kBlock) {
      float4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = s4[i + u * dev::kBlock];
#pragma unroll
      for (int u = 0; u < 4; ++u) add(v[u]);
    }
    for (; i < e >> 2; i += dev::kBlock) add(s4[i]);
  } else {
    for (long i = b + t; i < e; i += dev::kBlock) r = addToRange(r, src[i]);
  }
  r = blockRange(r, red);
  if (t == 0) a.slots[slot] = r;
}

// y0, y1: already scaled
__device__ __forceinline__ void splitHalves(float y0, float y1, unsigned &h, unsigned &l) {
  const f32x2 r = {y0, y1};
  const half2v p = __builtin_convertvector(r, half2v);
  const f32x2 q = {__builtin_fmaf(-(float)p.x, 4096.f, r.x * 4096.f), __builtin_fmaf(-(float)p.y, 4096.f, r.y * 4096.f)};
  h = __builtin_bit_cast(unsigned, p);
  l = __builtin_bit_cast(unsigned, __builtin_convertvector(q, half2v));
}

__device__ __forceinline__ half8v asHalf(u32x4 v) { return __builtin_bit_cast(half8v, v); }

// One k-step of 16 of one wave on parts (h, l) as mfmaSplit.
template <int TI, int TJ>
__device__ __forceinline__ void mfmaHalves(const u32x4 (&a)[2][TI], const u32x4 (&b)[2][TJ], float16v (&hi)[TI][TJ],
                                           float16v (&lo)[TI][TJ]) {
  auto all = [&](int sa, int sb, float16v (&acc)[TI][TJ]) {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(asHalf(a[sa][i]), asHalf(b[sb][j]), acc[i][j], 0, 0, 0);
  };
  all(0, 0, hi);
  all(0, 1, lo);
  all(1, 0, lo);
}
// A block's sums without their scale; returns (to the whole wave) whether one is not finite.
__device__ __forceinline__ bool finishHalves(float16v &acc, const float16v &lo, int e) {
  float bad = 0.f;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const float s = acc[v] + lo[v] * 0x1p-12f;
    bad = __builtin_fmaf(s, 0.f, bad);
    acc[v] = __builtin_amdgcn_ldexpf(s, e);
  }
  return __any(bad != bad);
}

// Scales of the two operands of a split of a weight gradient over images [n0, n1), from the ranges of gyN and xN slices of
// every image. fits: the fp16 parts hold all of their elements.
struct HalvesScale {
  float gy, x;
  int gyExp, xExp;
  bool fits;
};
__device__ __forceinline__ HalvesScale halvesScale(const uint2 *gySlots, int gyN, const uint2 *xSlots, int xN, int n0, int n1) {
  __shared__ uint2 red[2][4];
  auto range = [&](const uint2 *slots, int n, uint2 *r4) {
    uint2 r = noRange();
    for (long i = (long)n0 * n + threadIdx.x; i < (long)n1 * n; i += dev::kBlock) r = joinRanges(r, slots[i]);
    r = blockRange(r, r4);
    return make_uint2(__builtin_amdgcn_readfirstlane(r.x), __builtin_amdgcn_readfirstlane(r.y));
  };
  const uint2 a = range(gySlots, gyN, red[0]), b = range(xSlots, xN, red[1]);
  HalvesScale s{};
  s.gyExp = min(exponentFor(a.x), 127), s.xExp = min(exponentFor(b.x), 127);
  s.gy = __uint_as_float((unsigned)(s.gyExp + 127) << 23), s.x = __uint_as_float((unsigned)(s.xExp + 127) << 23);  // (-113 <= e <= 127)
  s.fits = fitsHalves(a, s.gyExp) && fitsHalves(b, s.xExp);
  return s;
}
