// SpatialConvolutionMM for gfx950: implicit im2col GEMM on the matrix cores, fp32 in and out.
//
// The reference loops over the batch and per image launches im2col, an SGEMM
// and (for the bias) a k=1 SGEMM, writing a (Cin*kH*kW) x (oH*oW) column
// buffer to memory and reading it back
// (lib/THCUNN/generic/SpatialConvolutionMM.cu:129-194, 272-308, 396-470).
// Here each entry point is one batched GEMM over the whole mini-batch. Most kernels
// multiply fp32 operands as products of three bf16 parts each, accumulated in fp32
// (v_mfma_f32_32x32x16_bf16; "fp32 products on the bf16 matrix pipe" below), long forward and
// gradInput passes as three products of fp16 parts (conv_halves.h); the 1x1 kernel of 32 planes, the
// few-plane gradInput and the general fallbacks use the fp32 matrix instruction.
//   updateOutput       C[o][n,l]  = bias[o] + sum_k W[o][k] * col[k][n,l]
//                      col is never stored: the B-tile loader gathers it from a
//                      zero-bordered copy of the input on the fly (implicit im2col)
//   accGradParameters  gW[o][k]  += scale * sum_{n,l} gy[n][o][l] * col[k][n,l]
//                      split over groups of positions; partial products go to the
//                      caller's `columns` scratch and are folded in a fixed
//                      order (deterministic, no atomics); gradBias rides along
//                      where the fold can take it, else it is a pass of its own
//   updateGradInput    stride 1: the forward kernels on gradOutput with flipped
//                      weights; other strides: the same phase by phase; what neither
//                      takes: gradCol[k][n,l] = sum_o W[o][k] * gy[n][o][l] for a group of
//                      images into `gradColumns`, then the col2im gather of
//                      lib/THCUNN/im2col.h:63-102 over the group.
#include <atomic>
#include <climits>
#include <cstring>
#include <map>
#include <mutex>
#include <numeric>
#include <type_traits>

#include "device_utils.h"
#include "launch_utils.h"
#include "thc_internal.h"

using namespace thc;

namespace {

typedef float float16v __attribute__((ext_vector_type(16)));

constexpr int BM = 128, BN = 128, BK = 16;
constexpr int PITCH = 132;  // 8 * PITCH % 64 == 32: the two k-halves of a transposing store hit disjoint banks

struct ConvGeom {
  int N, Cin, Cout, H, W, oH, oW;
  int kH, kW, dH, dW, padH, padW;
  int dilH, dilW;  // tap spacing (1 = ordinary convolution)
  int K;  // Cin * kH * kW
  int L;  // oH * oW
};

enum GemmMode { kForward = 0, kGradCol = 1, kGradWeight = 2 };

struct GemmArgs {
  const float *a;   // forward: W (Cout x K); gradCol: W; gradWeight: gy
  const float *b;   // forward: x; gradCol: gy; gradWeight: x
  float *c;         // forward: out; gradCol: gradCol of the group; gradWeight: partials
  const float *bias;
  int M, Ncols, R;  // GEMM extents: C is M x Ncols, reduction length R (per split)
  int n0;           // first image of the group (gradCol) / reduction tiles (of BK positions) per split (gradWeight)
  int nImages;      // images covered by this launch
  int mTiles;
  bool vecA;        // A rows may be fetched with 16-byte loads (extent % 4 == 0, aligned base)
};

// Decomposition of a flat output position lg = n*L + oh*oW + ow.
struct Pos {
  int n, oh, ow;
};

// ---- the MFMA core: one 128x128 tile, 4 waves of 64x64 -----------------------
__device__ __forceinline__ void mfmaTile(const float (*As)[PITCH], const float (*Bs)[PITCH], float16v (&acc)[2][2],
                                         int wm, int wn, int lane) {
  const int kk = lane >> 5, idx = lane & 31;
#pragma unroll
  for (int k = 0; k < BK; k += 2) {
    float a0 = As[k + kk][wm * 64 + idx], a1 = As[k + kk][wm * 64 + 32 + idx];
    float b0 = Bs[k + kk][wn * 64 + idx], b1 = Bs[k + kk][wn * 64 + 32 + idx];
    acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b1, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b0, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, acc[1][1], 0, 0, 0);
  }
}

// Element (r, col) of the implicit im2col matrix for image base xb:
// x[c][oh*dH - padH + kh][ow*dW - padW + kw] or 0 (lib/THCUNN/im2col.h:24-36).
__device__ __forceinline__ float gatherCol(const float *__restrict__ xb, const ConvGeom &g, int c, int kh, int kw,
                                           int ih0, int iw0) {
  int ih = ih0 + kh * g.dilH, iw = iw0 + kw * g.dilW;
  return (ih >= 0 && ih < g.H && iw >= 0 && iw < g.W) ? xb[((long)c * g.H + ih) * g.W + iw] : 0.f;
}

template <int MODE>
__global__ void __launch_bounds__(dev::kBlock)
convGemmKernel(GemmArgs p, ConvGeom g) {
  __shared__ float As[2][BK][PITCH];
  __shared__ float Bs[2][BK][PITCH];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int mTile = blockIdx.x % p.mTiles, nTile = blockIdx.x / p.mTiles;
  const int m0 = mTile * BM, j0 = nTile * BN;
  const int split = blockIdx.y;
  const int KK = g.kH * g.kW;

  float16v acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  float ra[8], rb[8];

  // ---- per-thread loader state ------------------------------------------------
  // "col-major" mapping: one tile column, 8 consecutive reduction rows
  const int colA = t & 127, rowA8 = (t >> 7) * 8;
  // "row-major" mapping: one tile row/column pair (t >> 1), 8 consecutive reduction elements
  const int rowT = t >> 1, redT8 = (t & 1) * 8;

  // forward / gradCol: B column = output position lg (fixed per thread)
  Pos bp = {0, 0, 0};
  bool bValid = false;
  const float *bBase = nullptr;
  int ih0 = 0, iw0 = 0;
  if (MODE == kForward || MODE == kGradCol) {
    long lg = (long)j0 + colA;
    bValid = lg < (long)p.Ncols;
    if (bValid) {
      bp.n = (int)(lg / g.L);
      int l = (int)(lg - (long)bp.n * g.L);
      bp.oh = l / g.oW;
      bp.ow = l - bp.oh * g.oW;
      if (MODE == kForward) {
        bBase = p.b + (long)(p.n0 + bp.n) * g.Cin * g.H * g.W;
        ih0 = bp.oh * g.dH - g.padH;
        iw0 = bp.ow * g.dW - g.padW;
      } else {
        bBase = p.b + (long)(p.n0 + bp.n) * g.Cout * g.L + l;  // + o * L
      }
    }
  }
  // gradWeight: B column = k index (c, kh, kw), 16-lane groups walk consecutive positions
  const int gwR = t & 15, gwJ = t >> 4;  // reduction row within the tile, first of 8 columns (stride 16)
  // gradWeight: split `split` reduces positions [rBegin, rEnd) of the N*L positions of the batch
  const long rBegin = (MODE == kGradWeight) ? (long)split * p.n0 * BK : 0;
  const long rEnd = (MODE == kGradWeight) ? min(rBegin + (long)p.n0 * BK, (long)p.nImages * g.L) : (long)p.R;
  const int nkt = (int)((rEnd - rBegin + BK - 1) / BK);

  auto loadTiles = [&](int kt) {
    const int r0 = kt * BK;
    if (MODE == kForward) {
      // A: W[o][k], k contiguous
      {
        int o = m0 + rowT, k = r0 + redT8;
        const float *src = p.a + (long)o * g.K + k;
        bool rowOk = o < p.M;
        if (p.vecA && rowOk && k + 8 <= g.K) {
          float4 v0 = reinterpret_cast<const float4 *>(src)[0], v1 = reinterpret_cast<const float4 *>(src)[1];
          ra[0] = v0.x, ra[1] = v0.y, ra[2] = v0.z, ra[3] = v0.w;
          ra[4] = v1.x, ra[5] = v1.y, ra[6] = v1.z, ra[7] = v1.w;
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) ra[i] = (rowOk && k + i < g.K) ? src[i] : 0.f;
        }
      }
      // B: implicit im2col, rows k = r0 + rowA8 + i
      {
        int k = r0 + rowA8;
        int c = k / KK, rem = k - c * KK;
        int kh = rem / g.kW, kw = rem - kh * g.kW;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          rb[i] = (bValid && k + i < g.K) ? gatherCol(bBase, g, c, kh, kw, ih0, iw0) : 0.f;
          if (++kw == g.kW) {
            kw = 0;
            if (++kh == g.kH) {
              kh = 0;
              ++c;
            }
          }
        }
      }
    } else if (MODE == kGradCol) {
      // A[m = k][r = o] = W[o][k]: contiguous along m
      {
        int k = m0 + colA;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          int o = r0 + rowA8 + i;
          ra[i] = (k < p.M && o < p.R) ? p.a[(long)o * g.K + k] : 0.f;
        }
      }
      // B[r = o][lg] = gy[n][o][l]
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        int o = r0 + rowA8 + i;
        rb[i] = (bValid && o < p.R) ? bBase[(long)o * g.L] : 0.f;
      }
    } else {
      // gradWeight. A[m = o][r = (n,l)] = gy[n][o][l]: contiguous along r inside an image
      {
        int o = m0 + rowT;
        long r = rBegin + r0 + redT8;
        bool rowOk = o < p.M;
        int n = (int)(r / g.L);
        int l = (int)(r - (long)n * g.L);
        if (p.vecA && rowOk && r + 8 <= rEnd) {
          // with L % 4 == 0 a group of 4 never straddles an image
          const float *s0 = p.a + ((long)n * g.Cout + o) * g.L + l;
          float4 v0 = *reinterpret_cast<const float4 *>(s0);
          int l2 = l + 4, n2 = n;
          if (l2 >= g.L) {
            l2 -= g.L;
            ++n2;
          }
          const float *s1 = p.a + ((long)n2 * g.Cout + o) * g.L + l2;
          float4 v1 = *reinterpret_cast<const float4 *>(s1);
          ra[0] = v0.x, ra[1] = v0.y, ra[2] = v0.z, ra[3] = v0.w;
          ra[4] = v1.x, ra[5] = v1.y, ra[6] = v1.z, ra[7] = v1.w;
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            ra[i] = (rowOk && r + i < rEnd) ? p.a[((long)n * g.Cout + o) * g.L + l] : 0.f;
            if (++l == g.L) {
              l = 0;
              ++n;
            }
          }
        }
      }
      // B[r = (n,l)][j = k] = col[k][n,l]; lanes 0..15 of a group walk consecutive l
      {
        long r = rBegin + r0 + gwR;
        bool rOk = r < rEnd;
        int n = rOk ? (int)(r / g.L) : 0;
        int l = rOk ? (int)(r - (long)n * g.L) : 0;
        int oh = l / g.oW, ow = l - oh * g.oW;
        const float *xb = p.b + (long)n * g.Cin * g.H * g.W;
        int ih0g = oh * g.dH - g.padH, iw0g = ow * g.dW - g.padW;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          int k = j0 + gwJ + 16 * i;
          float v = 0.f;
          if (rOk && k < p.Ncols) {
            int c = k / KK, rem = k - c * KK;
            int kh = rem / g.kW, kw = rem - kh * g.kW;
            v = gatherCol(xb, g, c, kh, kw, ih0g, iw0g);
          }
          rb[i] = v;
        }
      }
    }
  };

  auto storeTiles = [&](int buf) {
    if (MODE == kForward) {
#pragma unroll
      for (int i = 0; i < 8; ++i) As[buf][redT8 + i][rowT] = ra[i];
#pragma unroll
      for (int i = 0; i < 8; ++i) Bs[buf][rowA8 + i][colA] = rb[i];
    } else if (MODE == kGradCol) {
#pragma unroll
      for (int i = 0; i < 8; ++i) As[buf][rowA8 + i][colA] = ra[i];
#pragma unroll
      for (int i = 0; i < 8; ++i) Bs[buf][rowA8 + i][colA] = rb[i];
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) As[buf][redT8 + i][rowT] = ra[i];
#pragma unroll
      for (int i = 0; i < 8; ++i) Bs[buf][gwR][gwJ + 16 * i] = rb[i];
    }
  };

  if (nkt > 0) {
    loadTiles(0);
    storeTiles(0);
  }
  __syncthreads();
  for (int kt = 0; kt < nkt; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nkt) loadTiles(kt + 1);
    mfmaTile(As[buf], Bs[buf], acc, wm, wn, lane);
    if (kt + 1 < nkt) storeTiles(buf ^ 1);
    __syncthreads();
  }

  // ---- epilogue ----------------------------------------------------------------
  // 32x32 accumulator layout: lane holds column (lane & 31) and rows
  // 8*(v/4) + 4*(lane/32) + v%4, v = 0..15.
  const int colInTile = lane & 31, rowHalf = (lane >> 5) * 4;
#pragma unroll
  for (int tj = 0; tj < 2; ++tj) {
    const long col = (long)j0 + wn * 64 + tj * 32 + colInTile;
    if (col >= p.Ncols) continue;
    long cOff;  // offset of (row 0, col) and row stride
    long rowStride;
    if (MODE == kForward) {
      int n = (int)(col / g.L);
      int l = (int)(col - (long)n * g.L);
      cOff = (long)(p.n0 + n) * g.Cout * g.L + l;
      rowStride = g.L;
    } else if (MODE == kGradCol) {
      int n = (int)(col / g.L);
      int l = (int)(col - (long)n * g.L);
      cOff = (long)n * g.K * g.L + l;
      rowStride = g.L;
    } else {
      cOff = (long)split * p.M * p.Ncols + col;
      rowStride = p.Ncols;
    }
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        int row = m0 + wm * 64 + ti * 32 + 8 * (v >> 2) + rowHalf + (v & 3);
        if (row < p.M) {
          float val = acc[ti][tj][v];
          if (MODE == kForward && p.bias) val += p.bias[row];
          p.c[cOff + (long)row * rowStride] = val;
        }
      }
    }
  }
}

// ---- forward implicit GEMM, second generation ---------------------------------
// Same 128x128x16 tiling as convGemmKernel<kForward>, with the two costs that
// kept the MFMA pipe at ~40 % removed:
//  * operands sit in LDS as float4 groups of 4 consecutive k
//    (As[kg][row], Bs[kg][col]); a lane fetches the operands of four MFMAs with
//    one ds_read_b128 and the loaders store with ds_write_b128. Lane group
//    g = lane / 32 of super-step s consumes k-group 2s + g, i.e. MFMA j contracts
//    k = 8s + j (g = 0) with k = 8s + 4 + j (g = 1) - any pairing is valid as long
//    as A and B agree.
//  * the im2col gather is a buffer load: the image base is a scalar resource,
//    the lane's position (n, oh, ow) is a fixed 32-bit byte offset, and the tap
//    (c, kh, kw) of each k is wave-uniform, so it lives in scalar registers.
//    A tap outside the image gets an out-of-range offset, for which the buffer
//    unit returns 0 - the zero padding costs no branch.
constexpr int FPITCH = BM + 8;  // float4 per k-group row: +8 keeps the 2 k-groups a lane pair writes in disjoint banks

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

struct FwdArgs {
  const float *w;     // (M x K) row-major
  const float *x;     // images n0 .. n0 + nImages - 1 of (N, Cin, H, W)
  float *out;         // element (n, row, oh, ow) at out[n * outImg + row * outRow + oh * outSH + ow * outSW]
  long outImg;        // dense output (nImages, M, oH, oW): M * L, L, oW, 1
  int outRow, outSH, outSW;
  // != 0 (outSW == 2, outSH == 2 * row length): every element is the top-left corner of a 2 x 2 block of out
  // whose other three elements get the bias (or 0) - the gradInput of a 1x1 convolution with stride 2
  int dilate;
  const float *bias;  // M or null
  int M, Ncols;       // Ncols = nImages * L
  int mTiles;
  int bm, bn;         // rows and columns of an output tile (tileShape)
  int xBytes;         // bytes of the nImages input images (< 2^31)
  int wBytes;         // padded kernel: bytes of the weights (< 2^31)
  int kReal;          // padded kernel: k of the convolution itself; from there to K the weights are zero and the taps any valid ones
  bool vecA;
  // tail launch: tiles tile0 .. are each reduced by nSplit workgroups over ktPerSplit k-tiles;
  // their 128x128 partial tiles go to `partial` and fwdTailFixupKernel folds them
  int tile0, nSplit, ktPerSplit;
  // padded kernel, one launch for both: workgroups 0 .. full - 1 reduce tiles 0 .. full - 1 over all of K,
  // workgroup full + split * tail + i reduces split `split` of tile tile0 + i (tile0 = full)
  int full, tail;
  float *partial;
  int relu;           // != 0: the stored value is v > 0 ? v : 0 (Threshold(0, 0) applied to the output)
  // padded kernel: the output spans fewer than 2^31 bytes (outBytes) - whole row tiles are then stored with a
  // per-lane column offset and a scalar row offset, no address arithmetic on the vector ALU
  int outBytes;       // 0: not applicable
  unsigned magicL, magicOW;  // reciprocals of L and oW (dev::magicOf), 0: divide
  const int *taps;    // padded kernel: byte offset of tap (c, kh, kw) inside a (zero-padded) image, per k
  int tapStride;      // > 0 (1x1 windows): tap k sits at byte offset k * tapStride, no table is read
};

// Epilogue shared by the forward kernels: a lane holds column (lane & 31) and rows
// 8*(v/4) + 4*(lane/32) + v%4 of each 32x32 accumulator tile. Split workgroups store their
// partial tile, the others add the bias and store to out(n, row, l).
// biasLds: the tile's bias values in LDS (index = row - m0, zeros where there is no bias or row), or null.
// column (n, l) -> (n, oh, ow): through the reciprocals when the launch provides them
__device__ __forceinline__ void splitColumn(const FwdArgs &p, const ConvGeom &g, unsigned col, int &n, int &oh, int &ow) {
  n = p.magicL ? dev::fastDiv((int)col, p.magicL) : (int)(col / (unsigned)g.L);
  const int l = (int)col - n * g.L;
  oh = p.magicOW ? dev::fastDiv(l, p.magicOW) : l / g.oW;
  ow = l - oh * g.oW;
}

// biasDone: the accumulators started from the bias (whole tiles of the padded kernel)
template <int TBN = BN, int TI = 2, int TJ = 2>
__device__ __forceinline__ void fwdEpilogue(const FwdArgs &p, const ConvGeom &g, const float16v (&acc)[TI][TJ], int bx,
                                            int by, int m0, int j0, int wm, int wn, int grp, int idx,
                                            const float *biasLds = nullptr, int toPartial = -1, bool biasDone = false) {
  const int rowHalf = grp * 4;
  if (toPartial < 0 ? p.nSplit > 1 : toPartial != 0) {
    float *dst = p.partial + ((long)bx * p.nSplit + by) * (BM * BN);  // (no tile shape holds more than BM * BN elements)
#pragma unroll
    for (int tj = 0; tj < TJ; ++tj)
#pragma unroll
      for (int ti = 0; ti < TI; ++ti)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          dst[(wm * 64 + ti * 32 + 8 * (v >> 2) + rowHalf + (v & 3)) * TBN + wn * 32 * TJ + tj * 32 + idx] = acc[ti][tj][v];
    return;
  }
  if (biasDone && p.outBytes > 0 && m0 + wm * 64 + TI * 32 <= p.M) {
    // every row of the wave exists: 64 stores of (per-lane column offset, scalar row offset); a column past the
    // batch is an offset out of range
    const __amdgpu_buffer_rsrc_t orr = dev::makeRsrc(p.out, p.outBytes);
    const int rowBase = __builtin_amdgcn_readfirstlane(m0 + wm * 64);
#pragma unroll
    for (int tj = 0; tj < TJ; ++tj) {
      const unsigned col = (unsigned)j0 + wn * 32 * TJ + tj * 32 + idx;
      int n, oh, ow;
      splitColumn(p, g, min(col, (unsigned)p.Ncols - 1), n, oh, ow);
      const int voff = col < (unsigned)p.Ncols
                           ? (int)(((long)n * p.outImg + (long)oh * p.outSH + ow * p.outSW + (long)rowHalf * p.outRow) * 4)
                           : dev::kBufOob;
#pragma unroll
      for (int ti = 0; ti < TI; ++ti)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          float o = acc[ti][tj][v];
          if (p.relu) o = o > 0.f ? o : 0.f;
          const int soff = (rowBase + ti * 32 + 8 * (v >> 2) + (v & 3)) * p.outRow * 4;
          if (p.dilate) {
            // the element and its right neighbour, then the two below: 8-byte stores, a wave covers whole rows
            const float z = biasLds ? biasLds[wm * 64 + ti * 32 + 8 * (v >> 2) + rowHalf + (v & 3)] : 0.f;
            const u32x2 top = {__float_as_uint(o), __float_as_uint(z)}, bottom = {__float_as_uint(z), __float_as_uint(z)};
            const int below = col < (unsigned)p.Ncols ? voff + (p.outSH >> 1) * 4 : dev::kBufOob;
            __builtin_amdgcn_raw_buffer_store_b64(top, orr, voff, soff, 0);
            __builtin_amdgcn_raw_buffer_store_b64(bottom, orr, below, soff, 0);
          } else {
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o), orr, voff, soff, 0);
          }
        }
    }
    return;
  }
  auto store = [&](auto withBias) {
    constexpr bool BIAS = decltype(withBias)::value;
    // the lane's 32 bias values first: a load between the stores would wait for each store before it
    // (the compiler must assume that out and bias overlap)
    float bv[TI][16];
    if (BIAS) {
#pragma unroll
      for (int ti = 0; ti < TI; ++ti)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (biasLds) {  // 4 consecutive rows: one 16-byte LDS read
            const float4 b4 = *reinterpret_cast<const float4 *>(biasLds + wm * 64 + ti * 32 + 8 * q + rowHalf);
            bv[ti][4 * q] = b4.x, bv[ti][4 * q + 1] = b4.y, bv[ti][4 * q + 2] = b4.z, bv[ti][4 * q + 3] = b4.w;
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int row = m0 + wm * 64 + ti * 32 + 8 * q + rowHalf + r;
              bv[ti][4 * q + r] = row < p.M ? p.bias[row] : 0.f;
            }
          }
        }
    }
#pragma unroll
    for (int tj = 0; tj < TJ; ++tj) {
      const unsigned col = (unsigned)j0 + wn * 32 * TJ + tj * 32 + idx;  // Ncols < 2^31
      if (col >= (unsigned)p.Ncols) continue;
      int n, oh, ow;
      splitColumn(p, g, col, n, oh, ow);
      float *dst = p.out + (long)n * p.outImg + (long)oh * p.outSH + ow * p.outSW;
#pragma unroll
      for (int ti = 0; ti < TI; ++ti)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int row = m0 + wm * 64 + ti * 32 + 8 * (v >> 2) + rowHalf + (v & 3);
          float o = BIAS ? acc[ti][tj][v] + bv[ti][v] : acc[ti][tj][v];
          if (p.relu) o = o > 0.f ? o : 0.f;
          if (row < p.M) {
            float *q = dst + (long)row * p.outRow;
            q[0] = o;
            if (p.dilate) {
              const float z = p.bias ? p.bias[row] : 0.f;
              q[1] = z, q[p.outSH >> 1] = z, q[(p.outSH >> 1) + 1] = z;
            }
          }
        }
    }
  };
  if (p.bias && !biasDone)
    store(std::true_type{});
  else
    store(std::false_type{});
}

// taps[k] = ((c*H + kh*dilH)*W + kw*dilW) * 4 for k = (c*kH + kh)*kW + kw; g is the geometry of the padded images.
// Entries beyond Cin*kH*kW (rows padded to a multiple of BK, spare entries) point at the position's own
// first element: valid memory, and their weights are zero or they are never used. (If that element is not finite its
// product with a zero weight is NaN, and the second pass over such a block leaves these k out: FwdArgs::kReal.)
// byte offset of tap k = (c, kh, kw) inside a (zero-bordered) image of g.H x g.W; 0 beyond the last tap
__device__ __forceinline__ int tapOffset(int k, const ConvGeom &g) {
  const int KK = g.kH * g.kW;
  const int c = k / KK, rem = k - c * KK;
  const int kh = rem / g.kW, kw = rem - kh * g.kW;
  return c < g.Cin ? ((c * g.H + kh * g.dilH) * g.W + kw * g.dilW) * 4 : 0;
}

__global__ void __launch_bounds__(dev::kBlock)
buildTapTableKernel(int *taps, int entries, ConvGeom g) {
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < entries; k += gridDim.x * blockDim.x) taps[k] = tapOffset(k, g);
}

// wp(rows x Kp) = w(rows x K) with zeros in columns K .. Kp-1
__global__ void __launch_bounds__(dev::kBlock)
padRowsKernel(const float *__restrict__ w, float *__restrict__ wp, int rows, int K, int Kp) {
  const long total = (long)rows * Kp;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const int k = (int)(i % Kp);
    const long r = i / Kp;
    wp[i] = k < K ? w[r * K + k] : 0.f;
  }
}

// Wf[c][(o, kh', kw')] = W[o][(c, kH-1-kh', kW-1-kw')]: with these weights the stride-1 gradInput is a plain forward
// convolution of gradOutput (padding k-1-pad). The job rides along with the bordered copy of gradOutput (a few more
// workgroups of that launch) instead of costing a launch of its own: both are short, and their latencies would add.
__global__ void flipWeightKernel(const float *__restrict__ w, float *__restrict__ wf, int Cout, int Cin, int kH, int kW);
struct FlipJob {
  const float *w;
  float *wf;
  int Cout, Cin, kH, kW;
};
constexpr int kFlipBlocks = 4096;  // a lane per element up to a million weights: a lane that walks several is bound by their latencies
__device__ __forceinline__ void flipWeights(const FlipJob &f, int block, int blocks) {
  const int KK = f.kH * f.kW;
  const long total = (long)f.Cout * f.Cin * KK;
  for (long i = (long)block * dev::kBlock + threadIdx.x; i < total; i += (long)blocks * dev::kBlock) {
    const int t = (int)(i % KK);
    const long r = i / KK;
    const int o = (int)(r % f.Cout), c = (int)(r / f.Cout);
    f.wf[i] = f.w[((long)o * f.Cin + c) * KK + (KK - 1 - t)];
  }
}

// xp(nc, Hp, Wp) = x(nc, H, W) at row padTop, column padLeft inside zeros, for any plane size and count: a workgroup
// writes one run of 1024 U floats of the destination with 16-byte stores, wherever planes begin and end in it. One
// scalar division per workgroup locates the run; inside it a lane's offsets are small, so the reciprocal divisions
// are exact (a dividend below d + the run with d below the run; a larger d is passed at most once). The four elements of
// a group are found by stepping. Bound by memory: 6144 planes 71 x 71 -> 75 x 75 (262 MB) 103 us with a lane per
// element and a workgroup per 256 elements of a plane, 48 us (5.4 TB/s) in this form.
// U = 1: runs of 1024 for destinations that would leave CUs without one of 4096 (64 planes 33 x 33: 4.2 us with U = 4, 2.9 so).
template <int U>
__global__ void __launch_bounds__(dev::kBlock)
padPlanesRunKernel(const float *__restrict__ x, float *__restrict__ xp, int H, int W, int padTop, int padLeft, int Hp, int Wp,
                   long total, int copyBlocks, bool vec, int *taps, int tapEntries, ConvGeom tg, int tapBlocks, FlipJob flip) {
  if ((int)blockIdx.x >= copyBlocks + tapBlocks) {  // the weights of the convolution that follows, flipped
    flipWeights(flip, blockIdx.x - copyBlocks - tapBlocks, gridDim.x - copyBlocks - tapBlocks);
    return;
  }
  if ((int)blockIdx.x >= copyBlocks) {              // its tap table
    for (int k = (blockIdx.x - copyBlocks) * dev::kBlock + threadIdx.x; k < tapEntries; k += tapBlocks * dev::kBlock)
      taps[k] = tapOffset(k, tg);
    return;
  }
  constexpr int kPadRun = 4 * U * dev::kBlock;
  const int plane = Hp * Wp;
  const unsigned magicPlane = dev::magicOf(plane), magicW = dev::magicOf(Wp);
  const long e0 = (long)blockIdx.x * kPadRun;
  const long pl0 = e0 / plane;
  const int r0 = (int)(e0 - pl0 * plane), h0 = r0 / Wp, c0 = r0 - h0 * Wp;
  const float *src = x + pl0 * H * W;
  float v[U][4];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int o = (u * dev::kBlock + threadIdx.x) * 4;
    const int r = r0 + o;
    int pl = plane < kPadRun ? dev::fastDiv(r, magicPlane) : r >= plane;
    const int j = pl ? r - pl * plane : c0 + o;
    int hp = Wp < kPadRun ? dev::fastDiv(j, magicW) : j >= Wp;
    int wp = j - hp * Wp;
    if (!pl) hp += h0;
    const int left = (int)min(total - e0, (long)kPadRun) - o;  // elements of the destination from here on
    int h = hp - padTop, w = wp - padLeft, at = (pl * H + h) * W + w;  // (spans less than a run past a plane: an int)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[u][k] = (((unsigned)h < (unsigned)H) & ((unsigned)w < (unsigned)W) & (k < left)) ? src[at] : 0.f;
      ++w, ++at;
      if (w == Wp - padLeft) {
        w = -padLeft, ++h, at += W - Wp;
        if (h == Hp - padTop) h = -padTop, at += (H - Hp) * W;
      }
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const long e = e0 + (u * dev::kBlock + threadIdx.x) * 4;
    if (vec && e + 4 <= total) {
      *reinterpret_cast<float4 *>(xp + e) = make_float4(v[u][0], v[u][1], v[u][2], v[u][3]);
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (e + k < total) xp[e + k] = v[u][k];
    }
  }
}

// The copy of padPlanesFlatKernel for planes of a multiple of 4 floats: workgroups 0 .. copyBlocks - 1 of a launch, a
// lane per 16-byte group of the bordered planes.
__device__ __forceinline__ void padFlatVecBody(const float *__restrict__ x, float *__restrict__ xp, int H, int W, int padTop,
                                               int padLeft, int Hp, int Wp, long total4, int copyBlocks) {
  const int plane4 = (Hp * Wp) >> 2;
  const unsigned magicPlane = dev::magicOf(plane4), magicW = dev::magicOf(Wp);
  for (long i = (long)blockIdx.x * dev::kBlock + threadIdx.x; i < total4; i += (long)copyBlocks * dev::kBlock) {
    const int pl = dev::fastDiv((int)i, magicPlane), j = ((int)i - pl * plane4) * 4;
    const float *src = x + (long)pl * H * W;
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int hp = dev::fastDiv(j + k, magicW), wp = j + k - hp * Wp;
      const int h = hp - padTop, w = wp - padLeft;
      v[k] = (((unsigned)h < (unsigned)H) & ((unsigned)w < (unsigned)W)) ? src[h * W + w] : 0.f;
    }
    reinterpret_cast<float4 *>(xp)[i] = make_float4(v[0], v[1], v[2], v[3]);
  }
}

// The bordered copy for small planes (7x7 ... 28x28 stages): a lane per 16-byte group of the whole destination. Workgroups
// past copyBlocks build the tap table, those behind them flip the weights.
// ANY: planes of any size (9x9 = a bordered 7x7 plane): a group may straddle two planes and the last elements of
// the destination may not fill a group.
template <bool ANY>
__global__ void __launch_bounds__(dev::kBlock)
padPlanesFlatKernel(const float *__restrict__ x, float *__restrict__ xp, int H, int W, int padTop, int padLeft, int Hp, int Wp,
                    long total4, int copyBlocks, int *taps, int tapEntries, ConvGeom tg, int tapBlocks, FlipJob flip) {
  if ((int)blockIdx.x >= copyBlocks + tapBlocks) {  // the weights of the convolution that follows, flipped
    flipWeights(flip, blockIdx.x - copyBlocks - tapBlocks, gridDim.x - copyBlocks - tapBlocks);
    return;
  }
  if ((int)blockIdx.x >= copyBlocks) {
    for (int k = (blockIdx.x - copyBlocks) * dev::kBlock + threadIdx.x; k < tapEntries; k += tapBlocks * dev::kBlock)
      taps[k] = tapOffset(k, tg);
    return;
  }
  if (ANY) {
    // total4 counts elements here
    const int plane = Hp * Wp;
    const unsigned magicPlane = dev::magicOf(plane), magicW = dev::magicOf(Wp);
    auto fetch = [&](unsigned e) {
      const int pl = dev::fastDiv((int)e, magicPlane), j = (int)e - pl * plane;
      const int hp = dev::fastDiv(j, magicW), wp = j - hp * Wp;
      const int h = hp - padTop, w = wp - padLeft;
      return (((unsigned)h < (unsigned)H) & ((unsigned)w < (unsigned)W)) ? x[(long)pl * H * W + h * W + w] : 0.f;
    };
    const long groups = (total4 + 3) >> 2;
    for (long i = (long)blockIdx.x * dev::kBlock + threadIdx.x; i < groups; i += (long)copyBlocks * dev::kBlock) {
      const unsigned e = (unsigned)(i * 4);
      if (e + 4 <= (unsigned long)total4) {
        reinterpret_cast<float4 *>(xp)[i] = make_float4(fetch(e), fetch(e + 1), fetch(e + 2), fetch(e + 3));
      } else {
        for (unsigned q = e; q < (unsigned long)total4; ++q) xp[q] = fetch(q);
      }
    }
    return;
  }
  padFlatVecBody(x, xp, H, W, padTop, padLeft, Hp, Wp, total4, copyBlocks);
}

int residentSlots(const void *kernel);

// taps != nullptr: the same launch also builds the tap table (tapEntries entries) of geometry tg
// flip != nullptr: and flips the weights of *flip
void launchPadPlanes(hipStream_t s, const float *x, float *xp, long planes, int H, int W, int padTop, int padLeft, int Hp,
                     int Wp, int *taps = nullptr, int tapEntries = 0, const ConvGeom *tg = nullptr, const FlipJob *flip = nullptr) {
  const int plane = Hp * Wp;
  const FlipJob fj = flip ? *flip : FlipJob{};
  const int flipBlocks = flip ? (int)std::min<long>(kFlipBlocks, ((long)fj.Cout * fj.Cin * fj.kH * fj.kW + dev::kBlock - 1) / dev::kBlock) : 0;
  if (launch::ceilDiv(plane, dev::kBlock) > 65535) error("SpatialConvolutionMM: image plane too large");
  const int tapBlocks = taps ? std::max(1, std::min(16, launch::ceilDiv(tapEntries, dev::kBlock))) : 0;
  const ConvGeom g = tg ? *tg : ConvGeom{};
  const long total4 = planes * (plane / 4);
  // (the reciprocal division of a group index by the groups per plane is exact while index * divisor < 2^32)
  if (plane % 4 == 0 && plane < 4096 && launch::aligned16(xp) && total4 * (plane / 4) < 0xffffffffL) {
    const int copyBlocks = (int)std::min<long>((total4 + dev::kBlock - 1) / dev::kBlock, 16384);
    padPlanesFlatKernel<false><<<copyBlocks + tapBlocks + flipBlocks, dev::kBlock, 0, s>>>(
        x, xp, H, W, padTop, padLeft, Hp, Wp, total4, copyBlocks, taps, tapEntries, g, tapBlocks, fj);
  } else if (plane < 1024 && launch::aligned16(xp) && planes * plane * (long)plane < 0xffffffffL) {
    // small planes of any size (a bordered 7x7 or 13x13 plane): a workgroup per plane would leave most of its lanes idle
    const long total = planes * plane;
    const int copyBlocks = (int)std::min<long>(((total + 3) / 4 + dev::kBlock - 1) / dev::kBlock, 16384);
    padPlanesFlatKernel<true><<<copyBlocks + tapBlocks + flipBlocks, dev::kBlock, 0, s>>>(
        x, xp, H, W, padTop, padLeft, Hp, Wp, total, copyBlocks, taps, tapEntries, g, tapBlocks, fj);
  } else {
    const long total = planes * plane;
    const int run = total <= 4096L * residentSlots(nullptr) ? 1024 : 4096;
    const long copyBlocks = (total + run - 1) / run;
    if (copyBlocks + tapBlocks + flipBlocks > 0x7fffffffL) error("SpatialConvolutionMM: batch too large");
    (run == 1024 ? padPlanesRunKernel<1> : padPlanesRunKernel<4>)<<<(unsigned)copyBlocks + tapBlocks + flipBlocks, dev::kBlock, 0, s>>>(
        x, xp, H, W, padTop, padLeft, Hp, Wp, total, (int)copyBlocks, launch::aligned16(xp), taps, tapEntries, g, tapBlocks, fj);
  }
  THC_HIP_CHECK(hipGetLastError());
}
inline void launchPadPlanes(hipStream_t s, const float *x, float *xp, long planes, int H, int W, int padH, int padW,
                            int *taps = nullptr, int tapEntries = 0, const ConvGeom *tg = nullptr, const FlipJob *flip = nullptr) {
  launchPadPlanes(s, x, xp, planes, H, W, padH, padW, H + 2 * padH, W + 2 * padW, taps, tapEntries, tg, flip);
}

// ---- gradInput by output phase ------------------------------------------------------------------
// gi[h] receives gy[oh] * w[kh] where h + pad = oh * stride + kh * dil. For the positions
// h = ph + stride * i of one phase only the taps with kh * dil = ph + pad (mod stride) contribute,
// they form an arithmetic sequence kh = k0 + a * kStep, and tap a reads gy row i + q0 - a * qStep:
// per phase a stride-1 convolution of gy with a sub-kernel, written to a strided sub-grid of gi.
struct PhaseAxis {
  int n;                // gi positions of the phase along the axis
  int k0, kStep, nk;    // contributing taps
  int q0, qStep;        // gy index of tap a at position i: i + q0 - a * qStep
};
struct Phase {
  PhaseAxis h, w;
  int h0, w0;           // first gi row / column of the phase
  int K, Kp;            // Cout * h.nk * w.nk, rounded up to a positive multiple of BK
  int tapOfs;           // ints from the start of the tap tables
  long wOfs;            // floats from the start of the phase weights
};
constexpr int kMaxPhases = 16;
struct PhaseSet {
  Phase ph[kMaxPhases];
  int count;
};

// Phase weights Wp(Cin x Kp): Wp[c][(o, a, b)] = w[o][c][h.k0 + a*h.kStep][w.k0 + b*w.kStep], zero from K to Kp, and the
// tap table of each phase: entry k = (o, a, b) is the byte offset of gy element (o, q0h - a*qStepH, q0w - b*qStepW) of
// the bordered image, 0 from K on.
// grid = (chunks of a weight row, Cin + 1, phases): blocks with blockIdx.y == Cin write the tap table.
// (bx of gx, by, bz) = the workgroup's position in that grid
__device__ __forceinline__ void phaseSetupBody(const float *__restrict__ w, float *__restrict__ dst, int *__restrict__ taps,
                                               const PhaseSet &set, int Cin, int kH, int kW, int Hp, int Wp, int top, int left,
                                               int bx, int gx, int by, int bz) {
  const Phase &P = set.ph[bz];
  const int tp = P.h.nk * P.w.nk;
  const unsigned magicTp = dev::magicOf(tp), magicNk = dev::magicOf(P.w.nk);
  const int c = by;
  if (c == Cin) {
    const int entries = P.Kp + 2 * BK;
    int *d = taps + P.tapOfs;
    for (int k = bx * dev::kBlock + threadIdx.x; k < entries; k += gx * dev::kBlock) {
      int v = 0;
      if (k < P.K) {
        const int o = dev::fastDiv(k, magicTp), r = k - o * tp;
        const int a = dev::fastDiv(r, magicNk), b = r - a * P.w.nk;
        v = ((o * Hp + top + P.h.q0 - a * P.h.qStep) * Wp + left + P.w.q0 - b * P.w.qStep) * 4;
      }
      d[k] = v;
    }
    return;
  }
  float *d = dst + P.wOfs + (long)c * P.Kp;
  const long oStride = (long)Cin * kH * kW;
  const float *src = w + ((long)c * kH + P.h.k0) * kW + P.w.k0;
  for (int k = bx * dev::kBlock + threadIdx.x; k < P.Kp; k += gx * dev::kBlock) {
    float v = 0.f;
    if (k < P.K) {
      const int o = dev::fastDiv(k, magicTp), r = k - o * tp;
      const int a = dev::fastDiv(r, magicNk), b = r - a * P.w.nk;
      v = src[o * oStride + (a * P.h.kStep) * kW + b * P.w.kStep];
    }
    d[k] = v;
  }
}

__global__ void __launch_bounds__(dev::kBlock)
phaseSetupKernel(const float *__restrict__ w, float *__restrict__ dst, int *__restrict__ taps, PhaseSet set, int Cin, int kH,
                 int kW, int Hp, int Wp, int top, int left) {
  phaseSetupBody(w, dst, taps, set, Cin, kH, kW, Hp, Wp, top, left, blockIdx.x, gridDim.x, blockIdx.y, blockIdx.z);
}

// The bordered copy of gradOutput and the phase set-up in one launch (both are short: as two launches their latencies
// add): workgroups 0 .. copyBlocks - 1 copy (planes of a multiple of 4 floats), the others are the set-up's grid
// (chunks, Cin + 1, phases) laid out flat.
__global__ void __launch_bounds__(dev::kBlock)
padPlanesPhaseSetupKernel(const float *__restrict__ x, float *__restrict__ xp, int H, int W, int Hp, int Wp, int top, int left,
                          long total4, int copyBlocks, const float *__restrict__ w, float *__restrict__ dst,
                          int *__restrict__ taps, PhaseSet set, int Cin, int kH, int kW, int chunks) {
  if ((int)blockIdx.x < copyBlocks) {
    padFlatVecBody(x, xp, H, W, top, left, Hp, Wp, total4, copyBlocks);
    return;
  }
  const int l = blockIdx.x - copyBlocks;
  const int r = l / chunks, bx = l - r * chunks;
  const int bz = r / (Cin + 1), by = r - bz * (Cin + 1);
  phaseSetupBody(w, dst, taps, set, Cin, kH, kW, Hp, Wp, top, left, bx, chunks, by, bz);
}

// Generic forward kernel: any K, any alignment; taps and bounds resolved in the loop.
__global__ void __launch_bounds__(dev::kBlock)
convFwdImplicitKernel(FwdArgs p, ConvGeom g) {
  __shared__ float4 As[2][BK / 4][FPITCH];
  __shared__ float4 Bs[2][BK / 4][FPITCH];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int tileIdx = p.tile0 + blockIdx.x;
  const int mTile = tileIdx % p.mTiles, nTile = tileIdx / p.mTiles;
  const int m0 = mTile * BM, j0 = nTile * BN;
  const int KK = g.kH * g.kW;

  float16v acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // A loader: row (t >> 1), k = 8 * (t & 1) .. + 7
  const int rowA = t >> 1, kA = (t & 1) * 8;
  const bool rowOk = m0 + rowA < p.M;
  const float *aSrc = p.w + (long)(m0 + rowA) * g.K + kA;
  // B loader: column (t & 127) = one output position, k = 8 * (t >> 7) .. + 7 (wave-uniform)
  const int colB = t & 127;
  const int kB = __builtin_amdgcn_readfirstlane((t >> 7) * 8);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, p.xBytes, 0x00020000);
  const int kOob = 0x7fffffff;  // beyond num_records: the load returns 0
  int ih0 = 0, iw0 = 0, posOff = kOob;
  {
    long lg = (long)j0 + colB;
    if (lg < (long)p.Ncols) {
      int n = (int)(lg / g.L);
      int l = (int)(lg - (long)n * g.L);
      int oh = l / g.oW, ow = l - oh * g.oW;
      ih0 = oh * g.dH - g.padH;
      iw0 = ow * g.dW - g.padW;
      posOff = ((n * g.Cin * g.H + ih0) * g.W + iw0) * 4;  // may be "negative": only used when the tap is inside
    } else {
      ih0 = -(1 << 28);  // every tap fails the bounds test
    }
  }

  float4 ra0, ra1, rb0, rb1;
  const int nktAll = (g.K + BK - 1) / BK;
  const int ktBegin = blockIdx.y * p.ktPerSplit;
  const int nkt = min(nktAll, ktBegin + p.ktPerSplit);  // this workgroup reduces k-tiles [ktBegin, nkt)

  auto loadTiles = [&](int kt) {
    const int k0 = kt * BK;
    // ---- A
    if (p.vecA && rowOk && k0 + kA + 8 <= g.K) {
      ra0 = reinterpret_cast<const float4 *>(aSrc + k0)[0];
      ra1 = reinterpret_cast<const float4 *>(aSrc + k0)[1];
    } else {
      float tmp[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) tmp[i] = (rowOk && k0 + kA + i < g.K) ? aSrc[k0 + i] : 0.f;
      ra0 = make_float4(tmp[0], tmp[1], tmp[2], tmp[3]);
      ra1 = make_float4(tmp[4], tmp[5], tmp[6], tmp[7]);
    }
    // ---- B: scalar walk over the 8 taps of this wave
    int k = k0 + kB;  // scalar
    int c = k / KK, rem = k - c * KK;
    int kh = rem / g.kW, kw = rem - kh * g.kW;
    float tmp[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int ih = ih0 + kh * g.dilH, iw = iw0 + kw * g.dilW;
      const bool ok = (unsigned)ih < (unsigned)g.H && (unsigned)iw < (unsigned)g.W && (k + i) < g.K;
      const int soff = ((c * g.H + kh * g.dilH) * g.W + kw * g.dilW) * 4;  // scalar
      const int off = ok ? posOff + soff : kOob;
      tmp[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, off, 0, 0));
      if (++kw == g.kW) {
        kw = 0;
        if (++kh == g.kH) {
          kh = 0;
          ++c;
        }
      }
    }
    rb0 = make_float4(tmp[0], tmp[1], tmp[2], tmp[3]);
    rb1 = make_float4(tmp[4], tmp[5], tmp[6], tmp[7]);
  };
  auto storeTiles = [&](int buf) {
    As[buf][(t & 1) * 2][rowA] = ra0;
    As[buf][(t & 1) * 2 + 1][rowA] = ra1;
    Bs[buf][(t >> 7) * 2][colB] = rb0;
    Bs[buf][(t >> 7) * 2 + 1][colB] = rb1;
  };

  loadTiles(ktBegin);
  storeTiles(ktBegin & 1);
  __syncthreads();
  const int grp = lane >> 5, idx = lane & 31;
  for (int kt = ktBegin; kt < nkt; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nkt) loadTiles(kt + 1);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const float4 a0 = As[buf][2 * s + grp][wm * 64 + idx], a1 = As[buf][2 * s + grp][wm * 64 + 32 + idx];
      const float4 b0 = Bs[buf][2 * s + grp][wn * 64 + idx], b1 = Bs[buf][2 * s + grp][wn * 64 + 32 + idx];
      const float av0[4] = {a0.x, a0.y, a0.z, a0.w}, av1[4] = {a1.x, a1.y, a1.z, a1.w};
      const float bv0[4] = {b0.x, b0.y, b0.z, b0.w}, bv1[4] = {b1.x, b1.y, b1.z, b1.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(av0[j], bv0[j], acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(av0[j], bv1[j], acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(av1[j], bv0[j], acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(av1[j], bv1[j], acc[1][1], 0, 0, 0);
      }
    }
    if (kt + 1 < nkt) storeTiles(buf ^ 1);
    __syncthreads();
  }
  fwdEpilogue(p, g, acc, blockIdx.x, blockIdx.y, m0, j0, wm, wn, grp, idx);
}

// ---- fp32 products on the bf16 matrix pipe ------------------------------------------------------
// A float is the exact sum of three bf16 values h + m + l (8 significant bits each, every remainder exact), and the
// product of two bf16 values is exact in fp32. x * w is computed as the six products hh + hm + mh + mm + hl + lh; the
// three left out (ml, lm, ll) are below 2^-26 of x * w, a quarter of what rounding the product to fp32 would cost. The
// large products (hh) and the five small ones are summed in accumulators of their own, so a k-step of 16 rounds the
// large sum once where the fp32 instruction rounds it 16 times: against a 64-bit sum the error over K = 128 / 2304 /
// 8192 normally distributed terms is 6.4e-8 / 2.9e-7 / 5.8e-7 of the result's norm, with v_mfma_f32_32x32x2_f32
// 2.0e-7 / 8.6e-7 / 1.6e-6 (one-signed, badly scaled and 1e-30-sized terms: the same ratio or better).
// The matrix pipe runs bf16 at 16 times its fp32 rate, so six products cost 6/16 of the fp32 instruction's time
// (measured on registers alone: 300 TFLOP/s of fp32 products, held back by power, against 138 - 150).
// The bf16 instruction reads subnormal parts as zero, and the last part of a float reaches 2^-23 below it. Every operand is
// therefore multiplied by 2^24 as it is split: its parts are multiples of 2^-149 * 2^24 = 2^-125 then, none of them
// subnormal, so the sums are as exact for the smallest floats as for any other, whatever the other operand is. The sums
// carry 2^48, which is taken out of them at the end (their own underflow lies at 2^-174, below the smallest float). One
// more multiplication per element: 256 -> 256 planes 3x3 at 28 x 28, N = 64, forward + backward 977 -> 990 us; 64-row tiles,
// with half the products per element, 20.7 -> 21.6 us (64 -> 64 3x3 on 56 x 56, N = 8). (Taking the remainders with
// v_dot2c_f32_bf16, nine instructions a pair instead of thirteen, is exact too but does not run at the full rate: 1101 us.)
// An operand that is not finite or reaches 2^104, and a sum that reaches 2^80, make a block's results infinite or NaN; the
// kernels then compute that block of 32 x 32 again with the fp32 instruction, so infinities, NaNs, overflows and numbers
// of that size come out as they did.
// (Splitting a float into bf16 parts: Henry, Tang, Heinecke, "Leveraging the bfloat16 artificial intelligence
// datatype for higher-precision computations", ARITH 2019.)
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr float kSplitScale = 0x1p24f;       // of each operand
constexpr float kSumScale = 0x1p48f;         // of their products

// two neighbouring k -> the packed pairs of the three parts of kSplitScale times them
__device__ __forceinline__ void splitPair(unsigned x0, unsigned x1, unsigned &h, unsigned &m, unsigned &l) {
  f32x2 r = {__uint_as_float(x0) * kSplitScale, __uint_as_float(x1) * kSplitScale};
  h = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
  r = f32x2{r.x - __uint_as_float(h << 16), r.y - __uint_as_float(h & 0xffff0000u)};
  m = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
  r = f32x2{r.x - __uint_as_float(m << 16), r.y - __uint_as_float(m & 0xffff0000u)};
  l = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
}

// A block's sums from the large and the small products, without their scale. Returns (to the whole wave) whether one of
// them is not finite, so that the block has to be computed again.
__device__ __forceinline__ bool finishSums(float16v &acc, const float16v &lo) {
  float bad = 0.f;        // NaN as soon as one sum is not finite
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    acc[v] = (acc[v] + lo[v]) * (1.f / kSumScale);
    bad = __builtin_fmaf(acc[v], 0.f, bad);
  }
  return __any(bad != bad);
}

__device__ __forceinline__ bf16x8 asBf16(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// One k-step of 16 of one wave: TI x TJ blocks of 32 x 32. a[s][i], b[s][j]: part s (h, m, l) of the lane's 8
// k (k-group lane / 32) of row / column lane % 32 of a block.
template <int TI, int TJ>
__device__ __forceinline__ void mfmaSplit(const u32x4 (&a)[3][TI], const u32x4 (&b)[3][TJ], float16v (&hi)[TI][TJ],
                                          float16v (&lo)[TI][TJ]) {
  auto all = [&](int sa, int sb, float16v (&acc)[TI][TJ]) {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(asBf16(a[sa][i]), asBf16(b[sb][j]), acc[i][j], 0, 0, 0);
  };
  all(0, 0, hi);
  all(0, 1, lo);
  all(1, 0, lo);
  all(1, 1, lo);
  all(0, 2, lo);
  all(2, 0, lo);
}

// The products of a block with the fp32 instruction, added to c: `steps` times 16 terms, of which fetch(step, a, b) brings the
// lane's 8 of either operand (lanes 0-31 and 32-63 hold different terms, a and b the same ones). Operands come straight
// from memory, those of the next step under the current one's instructions. 256 -> 256 planes 3x3 at 28 x 28, N = 64,
// forward + backward, ordinary data 1050 us: with one infinity in x 1375, all of x NaN 2760, sums of 1e26 1806 (a load of 8
// terms waited for at a time: 2230, 5285 and 2834; fp32 instructions alone, on any data: 1360).
template <class Fetch>
__device__ __forceinline__ float16v fp32Block(float16v c, int steps, Fetch fetch) {
  float na[8], nb[8];
  if (steps > 0) fetch(0, na, nb);
#pragma unroll 1
  for (int s = 0; s < steps; ++s) {
    float a[8], b[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = na[u], b[u] = nb[u];
    if (s + 1 < steps) fetch(s + 1, na, nb);
#pragma unroll
    for (int u = 0; u < 8; ++u) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u], b[u], c, 0, 0, 0);
  }
  return c;
}
__device__ __forceinline__ void put4(float *dst, u32x4 v) {
  const unsigned x = v.x, y = v.y, z = v.z, w = v.w;
  dst[0] = __uint_as_float(x), dst[1] = __uint_as_float(y), dst[2] = __uint_as_float(z), dst[3] = __uint_as_float(w);
}

// Forward kernel for images that carry their zero border in memory (padH = padW = 0 in g,
// K % BK == 0, 16-byte loadable weight rows), on split operands (see above). Tiles come from memory as fp32 and are
// split by the lane that fetched them, on the way into LDS:
//  * a lane's output position is a fixed byte offset in a VGPR, the tap (c, kh, kw) of each k
//    is a byte offset read from a table with scalar loads and handed to the buffer load as its
//    scalar offset; every tap of every position is inside the padded image - no bounds test
//  * weight rows are addressed as fixed VGPR offset + scalar k offset
//  * the loop is unrolled over the two LDS buffers, so every LDS address is base + immediate
//  * a k-step of a wave is 24 matrix instructions of 32 cycles, 104 vector-ALU instructions that split the next
//    tile (between the matrix instructions: leaving out all but the scaling gained 5 %), 12 LDS reads and 6 LDS writes
// What bounds it: two workgroups per CU (128 accumulator registers per lane) keep the matrix pipe 53 % busy at a
// clock that power has pulled down to about 2 GHz. 256 -> 256 planes 3x3 at 28 x 28, N = 64 (59.2 GFLOP):
// 430 us with v_mfma_f32_32x32x2_f32, 315 us (188 TFLOP/s) on the parts.
// Rows past M and columns past the batch are clamped to valid ones and dropped in the epilogue.
// (bx, by): position among the tiles that start at tile0, and split; whole: the workgroup reduces all of K of tile bx and
// writes the output itself, else it leaves a partial tile. LINEAR: 1x1 windows - the tap offsets are an arithmetic sequence,
// computed by the scalar unit instead of read from the table.
// WM = 2: 128 x 128 tiles, the four waves as 2 x 2, 64 x 64 each. For row counts that would leave much of a 128-row tile
// empty (tileShape) the four waves sit side by side: WM = 1: 64 x 128 tiles, 64 x 32 a wave; WM = 3: 96 x 128, 96 x 32;
// WM = 0: 32 x 256, 32 x 64. WM = 1 keeps three workgroups on a CU; with 64 x 256 tiles (64 x 64 a wave, two workgroups)
// 64 -> 64 3x3 on 56x56 took, at N = 8 / 16 / 32, 33.7 / 49.0 / 65.9 us, with these 32.5 / 42.1 / 61.6; 3 -> 64 7x7 stride 2 on
// 224x224, N = 32: 83.9 and 75.0; 256 -> 64 1x1 on 56x56, N = 8: 21.0 and 12.5. (Both before operands were scaled as they are
// split, which costs 3 - 6 % here: 14.3 us now for the last kernel, 70 for the 7x7 one.)
template <int WM, bool LINEAR = false>
__device__ __forceinline__ void fwdPaddedBody(const FwdArgs &p, const ConvGeom &g, int bx, int by, bool whole) {
  constexpr int TBM = WM == 0 ? 32 : WM == 2 ? 128 : WM == 3 ? 96 : 64, TBN = WM == 0 ? 256 : 128;
  constexpr int TI = WM == 0 ? 1 : WM == 3 ? 3 : 2, TJ = WM == 1 || WM == 3 ? 1 : 2;  // 32 x 32 blocks of a wave
  constexpr int NA = WM == 2 || WM == 3 ? 2 : 1;         // 16-byte groups of weights a lane loads per k-tile
  constexpr int AP = TBM + 8, BP = TBN + 8;   // 16-byte groups (8 k of one part) per k-group row
  constexpr int NB = WM == 0 ? 16 : 8;        // image elements a lane gathers per k-tile
  __shared__ u32x4 As[2][3][2][AP];           // [buffer][part][k-group of 8][row]
  __shared__ u32x4 Bs[2][3][2][BP];
  __shared__ __attribute__((aligned(16))) float biasS[TBM];  // the tile's bias values: the epilogue reads them from here
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = WM == 2 ? wave >> 1 : 0, wn = WM == 2 ? wave & 1 : wave;
  const int tileIdx = whole ? bx : p.tile0 + bx;
  const int mTile = tileIdx % p.mTiles, nTile = tileIdx / p.mTiles;
  const int m0 = mTile * TBM, j0 = nTile * TBN;
  if (t < TBM) biasS[t] = p.bias && m0 + t < p.M ? p.bias[m0 + t] : 0.f;  // visible after the first barrier

  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void *)p.w, 0, p.wBytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, p.xBytes, 0x00020000);
  // weights: WM = 2 - a lane loads 8 consecutive k of row t / 2; WM = 1 - 4 consecutive k of row t / 4;
  //          WM = 0 - the same of row (t / 4) % 32: both halves of the workgroup fetch and park the same values
  //          WM = 3 - 4 consecutive k of row t / 4, and of row 64 + (t / 4) % 32 (both halves the same)
  // image:   a lane gathers 8 taps of column t % 128; WM = 0 - all 16 taps of column t
  const int rowA = WM == 2 ? t >> 1 : WM == 0 ? (t >> 2) & 31 : t >> 2;
  const int rowA2 = 64 + ((t >> 2) & 31);  // WM = 3
  const int kA = WM == 2 ? (t & 1) * 8 : (t & 3) * 4;
  const int colB = WM == 0 ? t : t & 127;
  const int kgB = WM == 0 ? 0 : t >> 7;
  const int aOff = (min(m0 + rowA, p.M - 1) * g.K + kA) * 4;
  const int aOff2 = WM == 3 ? (min(m0 + rowA2, p.M - 1) * g.K + kA) * 4 : aOff + 16;  // the second group
  const int kB = __builtin_amdgcn_readfirstlane(kgB * 8);
  auto columnOffset = [&](unsigned col) {
    int n, oh, ow;
    splitColumn(p, g, min(col, (unsigned)p.Ncols - 1), n, oh, ow);  // Ncols < 2^31
    return ((n * g.Cin * g.H + oh * g.dH) * g.W + ow * g.dW) * 4;
  };
  const int posOff = columnOffset((unsigned)j0 + colB);
  const int ktBegin = by * p.ktPerSplit;  // by == 0 for whole tiles
  const int nkt = whole ? g.K / BK : min(g.K / BK, ktBegin + p.ktPerSplit);  // this workgroup reduces k-tiles [ktBegin, nkt)

  u32x4 ra[NA];
  unsigned rb[NB];
  // The tap offsets of a wave and k-tile are fetched with scalar loads one tile ahead of their use,
  // so that no wave waits on the scalar cache inside the loop (the table has spare entries at its end).
  const int4 *tapBase = reinterpret_cast<const int4 *>(p.taps + kB);
  int4 e[NB / 4];
  auto loadTaps = [&](int kt) {
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
      if (LINEAR) {
        const int b = __builtin_amdgcn_readfirstlane((int)((unsigned)(kt * BK + kB + 4 * i) * (unsigned)p.tapStride));
        e[i] = make_int4(b, b + p.tapStride, b + 2 * p.tapStride, b + 3 * p.tapStride);
      } else {
        e[i] = tapBase[kt * (BK / 4) + i];
      }
    }
  };
  auto loadTiles = [&](int kt) {
    const int k0 = __builtin_amdgcn_readfirstlane(kt * BK);
#pragma unroll
    for (int i = 0; i < NA; ++i) ra[i] = __builtin_amdgcn_raw_buffer_load_b128(wr, i ? aOff2 : aOff, k0 * 4, 0);
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
      rb[4 * i + 0] = __builtin_amdgcn_raw_buffer_load_b32(xr, posOff, e[i].x, 0);
      rb[4 * i + 1] = __builtin_amdgcn_raw_buffer_load_b32(xr, posOff, e[i].y, 0);
      rb[4 * i + 2] = __builtin_amdgcn_raw_buffer_load_b32(xr, posOff, e[i].z, 0);
      rb[4 * i + 3] = __builtin_amdgcn_raw_buffer_load_b32(xr, posOff, e[i].w, 0);
    }
  };
  constexpr int PA = 2 * AP, PB = 2 * BP;    // 16-byte groups of one part in one buffer
  constexpr int BUFA = 3 * PA, BUFB = 3 * PB;  // of one buffer
  u32x4 *aDst = &As[0][0][kA >> 3][rowA];
  u32x4 *bDst = &Bs[0][0][kgB][colB];
  auto storeTiles = [&](auto bufc) {
    constexpr int b = decltype(bufc)::value;
    if constexpr (WM == 2) {
      unsigned h[4], m[4], l[4];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        splitPair(ra[i].x, ra[i].y, h[2 * i], m[2 * i], l[2 * i]);
        splitPair(ra[i].z, ra[i].w, h[2 * i + 1], m[2 * i + 1], l[2 * i + 1]);
      }
      aDst[b * BUFA] = u32x4{h[0], h[1], h[2], h[3]};
      aDst[b * BUFA + PA] = u32x4{m[0], m[1], m[2], m[3]};
      aDst[b * BUFA + 2 * PA] = u32x4{l[0], l[1], l[2], l[3]};
    } else {  // 4 k: half of a group
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        unsigned h[2], m[2], l[2];
        splitPair(ra[i].x, ra[i].y, h[0], m[0], l[0]);
        splitPair(ra[i].z, ra[i].w, h[1], m[1], l[1]);
        u32x2 *d = reinterpret_cast<u32x2 *>(aDst + b * BUFA + (i ? rowA2 - rowA : 0)) + ((kA >> 2) & 1);
        d[0] = u32x2{h[0], h[1]};
        d[2 * PA] = u32x2{m[0], m[1]};
        d[4 * PA] = u32x2{l[0], l[1]};
      }
    }
#pragma unroll
    for (int q = 0; q < NB / 8; ++q) {
      unsigned h[4], m[4], l[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) splitPair(rb[8 * q + 2 * i], rb[8 * q + 2 * i + 1], h[i], m[i], l[i]);
      bDst[b * BUFB + q * BP] = u32x4{h[0], h[1], h[2], h[3]};
      bDst[b * BUFB + PB + q * BP] = u32x4{m[0], m[1], m[2], m[3]};
      bDst[b * BUFB + 2 * PB + q * BP] = u32x4{l[0], l[1], l[2], l[3]};
    }
  };
  const int grp = lane >> 5, idx = lane & 31;
  const u32x4 *aSrc = &As[0][0][grp][wm * 64 + idx];
  const u32x4 *bSrc = &Bs[0][0][grp][wn * 32 * TJ + idx];
  using Buf0 = std::integral_constant<int, 0>;
  using Buf1 = std::integral_constant<int, 1>;

  float16v acc[TI][TJ], lo[TI][TJ];

  // Software pipeline. While tile kt is multiplied out of one LDS buffer, tile kt + 1 waits in registers - it is
  // split and parked in the other buffer under the matrix instructions - and tile kt + 2 is requested from memory.
  auto step = [&](auto cur, auto nxt, int kt, bool store, bool load) {
    constexpr int C = decltype(cur)::value;
    u32x4 a[3][TI], b[3][TJ];
#pragma unroll
    for (int s = 0; s < 3; ++s) {
#pragma unroll
      for (int i = 0; i < TI; ++i) a[s][i] = aSrc[C * BUFA + s * PA + 32 * i];
#pragma unroll
      for (int j = 0; j < TJ; ++j) b[s][j] = bSrc[C * BUFB + s * PB + 32 * j];
    }
    if (store) storeTiles(nxt);
    if (load) {
      loadTiles(kt + 2);
      loadTaps(kt + 3);
    }
    mfmaSplit(a, b, acc, lo);
    __syncthreads();
  };

  loadTaps(ktBegin);
  loadTiles(ktBegin);
  loadTaps(ktBegin + 1);
  storeTiles(Buf0{});
  if (ktBegin + 1 < nkt) {
    loadTiles(ktBegin + 1);
    loadTaps(ktBegin + 2);
  }
  __syncthreads();
  // the accumulators of a whole tile start from the bias (in LDS since the barrier): no addition in the epilogue
  auto biasBlock = [&](int i) {
    float16v v;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float4 b4 = make_float4(0.f, 0.f, 0.f, 0.f);
      if (whole) b4 = *reinterpret_cast<const float4 *>(biasS + wm * 64 + i * 32 + 8 * q + grp * 4);
      v[4 * q] = b4.x, v[4 * q + 1] = b4.y, v[4 * q + 2] = b4.z, v[4 * q + 3] = b4.w;
    }
    return v;
  };
#pragma unroll
  for (int i = 0; i < TI; ++i) {
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      acc[i][j] = biasBlock(i);
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] *= kSumScale, lo[i][j][v] = 0.f;
    }
  }
  int kt = ktBegin;
  for (; kt + 3 < nkt; kt += 2) {  // tile kt sits in buffer 0, tile kt + 1 in registers
    step(Buf0{}, Buf1{}, kt, true, true);
    step(Buf1{}, Buf0{}, kt + 1, true, true);
  }
  // one to three tiles left
  step(Buf0{}, Buf1{}, kt, kt + 1 < nkt, kt + 2 < nkt);
  if (kt + 1 < nkt) step(Buf1{}, Buf0{}, kt + 1, kt + 2 < nkt, false);
  if (kt + 2 < nkt) step(Buf0{}, Buf1{}, kt + 2, false, false);

#pragma unroll
  for (int j = 0; j < TJ; ++j)
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      if (!finishSums(acc[i][j], lo[i][j])) continue;
      // the block again in fp32, operands straight from memory
      const int cOff = columnOffset((unsigned)j0 + wn * 32 * TJ + j * 32 + idx);
      const int rOff = min(m0 + wm * 64 + i * 32 + idx, p.M - 1) * g.K * 4;
      const int4 *tp = LINEAR ? nullptr : reinterpret_cast<const int4 *>(p.taps + ktBegin * BK + 8 * grp);
      int4 t0{}, t1{};  // the lane's taps of the next step (the table has two spare k-tiles)
      if (!LINEAR) t0 = tp[0], t1 = tp[1];
      acc[i][j] = fp32Block(biasBlock(i), nkt - ktBegin, [&](int s, float (&a)[8], float (&b)[8]) {
        const int k = (ktBegin + s) * BK + 8 * grp;
        const int tap[8] = {t0.x, t0.y, t0.z, t0.w, t1.x, t1.y, t1.z, t1.w};
        put4(a, __builtin_amdgcn_raw_buffer_load_b128(wr, rOff + k * 4, 0, 0));
        put4(a + 4, __builtin_amdgcn_raw_buffer_load_b128(wr, rOff + k * 4 + 16, 0, 0));
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          b[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(xr, cOff + (LINEAR ? (k + e) * p.tapStride : tap[e]), 0, 0));
          if (k + e >= p.kReal) b[e] = 0.f;  // (times a weight of zero an infinity there would be NaN)
        }
        if (!LINEAR) tp += BK / 4, t0 = tp[0], t1 = tp[1];
      });
    }
  fwdEpilogue<TBN, TI, TJ>(p, g, acc, bx, by, m0, j0, wm, wn, grp, idx, biasS, whole ? 0 : 1, whole);
}

// Forward kernel for short calls (planDirect): a workgroup computes a tile of 32 T x 32 T, its four waves a quarter of
// K each, folded through LDS at the end; both operands go from memory straight into the registers that the matrix
// instructions read (no LDS, no barrier in the loop). So a short call fills the chip without partial tiles in memory and
// a second launch. Bound by latency: the loads of D k-steps are in flight, then by the weight loads (a 16-byte load of
// 32 rows touches 64 cache lines). Lanes 0-31 work on the first half of the input planes, lanes 32-63 on the second half
// (the order of a sum's terms is free), so that a tap's offset is the same for the whole wave: a scalar.
// Needs whole k-steps: K % 16 == 0 and Cin even. Operands as in the padded kernel (images with their border, 16-byte
// loadable weight rows, tap table); the grid is the number of tiles.
template <int T, bool LINEAR>
__global__ void __launch_bounds__(dev::kBlock, T == 2 ? 2 : 3)
convFwdDirectKernel(FwdArgs p, ConvGeom g) {
  constexpr int TI = T, TJ = T;                            // blocks of 32 x 32
  constexpr int D = T == 1 ? 4 : 2;                        // k-steps in flight
  constexpr int RQ = TI * TJ * 4;                          // groups of 4 accumulator registers
  __shared__ float4 red[4][RQ][dev::kWave];
  const int lane = threadIdx.x & 63, slice = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = lane >> 5, idx = lane & 31;
  const int tile = dev::xcdRemap(blockIdx.x, gridDim.x);    // (neighbours share columns: same XCD, same L2)
  const int nTile = tile / p.mTiles, mTile = tile - nTile * p.mTiles;
  const int m0 = mTile * 32 * TI, j0 = nTile * 32 * TJ;

  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void *)p.w, 0, p.wBytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, p.xBytes, 0x00020000);
  const int halfK = g.K >> 1, halfX = (g.Cin >> 1) * g.H * g.W * 4;
  int rowOff[TI], posOff[TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i) rowOff[i] = (min(m0 + i * 32 + idx, p.M - 1) * g.K + grp * halfK) * 4;
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    int n, oh, ow;
    splitColumn(p, g, min((unsigned)(j0 + j * 32 + idx), (unsigned)p.Ncols - 1), n, oh, ow);
    posOff[j] = ((n * g.Cin * g.H + oh * g.dH) * g.W + ow * g.dW) * 4 + grp * halfX;
  }
  const int steps = halfK >> 3, perSlice = (steps + 3) / 4;
  const int s0 = slice * perSlice, s1 = min(steps, s0 + perSlice);

  u32x4 ra[D][TI][2];
  unsigned rb[D][TJ][8];
  int4 t0, t1;                                             // the taps of the next step to be loaded
  auto loadTaps = [&](int step) {
    if (LINEAR) return;
    const int4 *tp = reinterpret_cast<const int4 *>(p.taps + min(step, steps - 1) * 8);
    t0 = tp[0], t1 = tp[1];
  };
  auto load = [&](auto dc, int step) {
    constexpr int d = decltype(dc)::value;
    // (steps past the slice: empty resources, everything reads as 0)
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void *)p.w, 0, step < s1 ? p.wBytes : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, step < s1 ? p.xBytes : 0, 0x00020000);
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int q = 0; q < 2; ++q) ra[d][i][q] = __builtin_amdgcn_raw_buffer_load_b128(wr, rowOff[i] + 16 * q, step * 32, 0);
    const int tap[8] = {t0.x, t0.y, t0.z, t0.w, t1.x, t1.y, t1.z, t1.w};
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        rb[d][j][e] = __builtin_amdgcn_raw_buffer_load_b32(xr, posOff[j], LINEAR ? (step * 8 + e) * p.tapStride : tap[e], 0);
    loadTaps(step + 1);
  };
  float16v acc[TI][TJ], lo[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = lo[i][j][v] = 0.f;
  auto split8 = [](const unsigned (&v)[8], u32x4 &h, u32x4 &m, u32x4 &l) {
    unsigned ph[4], pm[4], pl[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) splitPair(v[2 * q], v[2 * q + 1], ph[q], pm[q], pl[q]);
    h = u32x4{ph[0], ph[1], ph[2], ph[3]}, m = u32x4{pm[0], pm[1], pm[2], pm[3]}, l = u32x4{pl[0], pl[1], pl[2], pl[3]};
  };
  auto step = [&](auto dc, int next) {
    constexpr int d = decltype(dc)::value;
    u32x4 a[3][TI], b[3][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      const unsigned v[8] = {ra[d][i][0].x, ra[d][i][0].y, ra[d][i][0].z, ra[d][i][0].w,
                             ra[d][i][1].x, ra[d][i][1].y, ra[d][i][1].z, ra[d][i][1].w};
      split8(v, a[0][i], a[1][i], a[2][i]);
    }
#pragma unroll
    for (int j = 0; j < TJ; ++j) split8(rb[d][j], b[0][j], b[1][j], b[2][j]);
    // (fences: left alone the scheduler gathers the loads of several steps in front of one wait)
    __builtin_amdgcn_sched_barrier(0);
    load(dc, next);
    __builtin_amdgcn_sched_barrier(0);
    mfmaSplit(a, b, acc, lo);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto each = [](auto f) {
    f(std::integral_constant<int, 0>{});
    f(std::integral_constant<int, 1>{});
    if constexpr (D == 4) f(std::integral_constant<int, 2>{}), f(std::integral_constant<int, 3>{});
  };
  if (s0 < s1) {
    loadTaps(s0);
    each([&](auto dc) { load(dc, s0 + decltype(dc)::value); });
#pragma unroll 1
    for (int k = s0; k < s1; k += D) each([&](auto dc) { step(dc, k + D + decltype(dc)::value); });
  }
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      if (!finishSums(acc[i][j], lo[i][j])) continue;
      // the block over the slice again in fp32
      acc[i][j] = fp32Block(float16v{}, s1 - s0, [&](int s, float (&a)[8], float (&b)[8]) {
        const int k = (s0 + s) * 8;
        put4(a, __builtin_amdgcn_raw_buffer_load_b128(wr, rowOff[i], k * 4, 0));
        put4(a + 4, __builtin_amdgcn_raw_buffer_load_b128(wr, rowOff[i] + 16, k * 4, 0));
#pragma unroll
        for (int e = 0; e < 8; ++e)
          b[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(xr, posOff[j], LINEAR ? (k + e) * p.tapStride : p.taps[k + e], 0));
      });
    }

  // rows 8 * (r % 4) + 4 * (lane / 32) .. + 3 of block (r / 4 / TJ, r / 4 % TJ) at column lane % 32
  auto finish = [&](int r, float4 v) {
    const int row = m0 + r / (4 * TJ) * 32 + 8 * (r & 3) + 4 * grp;
    const unsigned col = (unsigned)j0 + (r >> 2) % TJ * 32 + idx;
    if (col >= (unsigned)p.Ncols) return;
    int n, oh, ow;
    splitColumn(p, g, col, n, oh, ow);
    float *dst = p.out + (long)n * p.outImg + (long)oh * p.outSH + ow * p.outSW + (long)row * p.outRow;
    const float vals[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (row + e < p.M) {
        float o = vals[e] + (p.bias ? p.bias[row + e] : 0.f);
        if (p.relu) o = o > 0.f ? o : 0.f;
        dst[(long)e * p.outRow] = o;
      }
  };
#pragma unroll
  for (int r = 0; r < RQ; ++r) {
    const float16v &c = acc[r / (4 * TJ)][(r >> 2) % TJ];
    red[slice][r][lane] = make_float4(c[4 * (r & 3)], c[4 * (r & 3) + 1], c[4 * (r & 3) + 2], c[4 * (r & 3) + 3]);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < RQ / 4; ++u) {  // each wave folds and stores a quarter
    const int r = slice * (RQ / 4) + u;
    float4 v = red[0][r][lane];
#pragma unroll
    for (int q = 1; q < 4; ++q) {
      const float4 w = red[q][r][lane];
      v.x += w.x, v.y += w.y, v.z += w.z, v.w += w.w;
    }
    finish(r, v);
  }
}

template <int WM, bool LINEAR = false>
__global__ void __launch_bounds__(dev::kBlock, WM == 1 ? 3 : 2)
convFwdPaddedKernel(FwdArgs p, ConvGeom g) {
  int bx = blockIdx.x, by = 0;
  const bool whole = bx < p.full;
  if (!whole) {
    const int u = bx - p.full;
    by = u / p.tail;
    bx = u - by * p.tail;
  }
  fwdPaddedBody<WM, LINEAR>(p, g, bx, by, whole);
}

// Several independent GEMMs of the same tile shape in one launch (the phases of a strided gradInput). An item's
// first p.full tiles are reduced by one workgroup each, its other p.tail tiles by p.nSplit workgroups. One flat
// grid: the whole tiles of all items in item order, then the splits of all items (split-major within an item) -
// the splits fill the slots that the last whole tiles free.
struct FwdBatchItem {
  FwdArgs p;
  ConvGeom g;
  int wholeEnd, splitEnd;  // running totals of p.full and of p.tail * p.nSplit up to and including this item
};
constexpr int kMaxBatch = 16;
struct FwdBatch {
  FwdBatchItem item[kMaxBatch];
  int count, wholeTotal;
};
static_assert(sizeof(FwdBatch) <= 4096, "kernel arguments are limited to 4 KB");

template <int WM>
__global__ void __launch_bounds__(dev::kBlock, WM == 1 ? 3 : 2)
convFwdPaddedBatchKernel(FwdBatch b) {
  int bx = blockIdx.x, by = 0, i = 0;
  const bool whole = bx < b.wholeTotal;
  if (whole) {
    while (i + 1 < b.count && bx >= b.item[i].wholeEnd) ++i;
    bx -= i > 0 ? b.item[i - 1].wholeEnd : 0;
  } else {
    bx -= b.wholeTotal;
    while (i + 1 < b.count && bx >= b.item[i].splitEnd) ++i;
    bx -= i > 0 ? b.item[i - 1].splitEnd : 0;
    const int tail = b.item[i].p.tail;
    by = bx / tail;
    bx -= by * tail;
  }
  fwdPaddedBody<WM>(b.item[i].p, b.item[i].g, bx, by, whole);
}

// 16-byte load of data that is read exactly once (non-temporal hint: it does not displace what the caches hold)
__device__ __forceinline__ float4 loadOnce4(const float4 *p) {
  typedef float f32x4v __attribute__((ext_vector_type(4)));
  const f32x4v v = __builtin_nontemporal_load(reinterpret_cast<const f32x4v *>(p));
  return make_float4(v.x, v.y, v.z, v.w);
}

// out tile = bias + sum over the nSplit partial tiles (ascending split order).
// grid = (tail tiles, BM*BN / 1024): a workgroup folds 1024 consecutive tile elements, 4 per lane.
__device__ __forceinline__ void fwdTailFixupBody(const FwdArgs &p, const ConvGeom &g) {
  const int tileIdx = p.tile0 + blockIdx.x;
  const int mTile = tileIdx % p.mTiles, nTile = tileIdx / p.mTiles;
  const float *src = p.partial + (long)blockIdx.x * p.nSplit * (BM * BN);
  const int e = (blockIdx.y * dev::kBlock + threadIdx.x) * 4;  // tile width % 4 == 0: the 4 elements share a row
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  // the partials are requested eight (then four) at a time and added in ascending split order: one memory round trip
  // per batch instead of one per split, the same sum bit for bit
  int sp = 0;
  auto batch = [&](auto nc) {
    constexpr int NQ = decltype(nc)::value;
    float4 q[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) q[i] = loadOnce4(reinterpret_cast<const float4 *>(src + (long)(sp + i) * (BM * BN) + e));
#pragma unroll
    for (int i = 0; i < NQ; ++i) v.x += q[i].x, v.y += q[i].y, v.z += q[i].z, v.w += q[i].w;
    sp += NQ;
  };
  while (sp + 8 <= p.nSplit) batch(std::integral_constant<int, 8>{});
  if (sp + 4 <= p.nSplit) batch(std::integral_constant<int, 4>{});
  while (sp < p.nSplit) batch(std::integral_constant<int, 1>{});
  const int r = e / p.bn, c = e - r * p.bn;
  const int row = mTile * p.bm + r;
  if (r >= p.bm || row >= p.M) return;  // 32 x 256 tiles fill half of a partial
  const float b = p.bias ? p.bias[row] : 0.f;
  float vals[4] = {v.x + b, v.y + b, v.z + b, v.w + b};
  if (p.relu) {
#pragma unroll
    for (int i = 0; i < 4; ++i) vals[i] = vals[i] > 0.f ? vals[i] : 0.f;
  }
  // (n, oh, ow) of the first of the four columns by one division (through the reciprocals when the launch provides
  // them), the others by stepping
  const long col0 = (long)nTile * p.bn + c;
  if (col0 >= p.Ncols) return;
  int n, oh, ow;
  if (col0 + 3 < 0x7fffffffL) {
    splitColumn(p, g, (unsigned)col0, n, oh, ow);
  } else {
    n = (int)(col0 / g.L);
    const int l = (int)(col0 - (long)n * g.L);
    oh = l / g.oW, ow = l - oh * g.oW;
  }
  if (p.dilate) {
    // four neighbouring columns of one output row: their 2 x 2 blocks are 8 consecutive floats of two rows of out
    float *q = p.out + (long)n * p.outImg + (long)row * p.outRow + (long)oh * p.outSH + ow * 2;
    if (col0 + 3 < p.Ncols && ow + 3 < g.oW && ((uintptr_t)q & 15) == 0 && (p.outSH & 7) == 0) {
      float4 *top = reinterpret_cast<float4 *>(q), *bottom = reinterpret_cast<float4 *>(q + (p.outSH >> 1));
      top[0] = make_float4(vals[0], b, vals[1], b), top[1] = make_float4(vals[2], b, vals[3], b);
      bottom[0] = bottom[1] = make_float4(b, b, b, b);
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (col0 + i >= p.Ncols) break;
    float *q = p.out + (long)n * p.outImg + (long)row * p.outRow + (long)oh * p.outSH + ow * p.outSW;
    if (p.dilate) {  // the block's rows start on 8-byte boundaries (even extents, 8-byte aligned tensor)
      *reinterpret_cast<float2 *>(q) = make_float2(vals[i], b);
      *reinterpret_cast<float2 *>(q + (p.outSH >> 1)) = make_float2(b, b);
    } else {
      q[0] = vals[i];
    }
    if (++ow == g.oW) {
      ow = 0;
      if (++oh == g.oH) oh = 0, ++n;
    }
  }
}

__global__ void __launch_bounds__(dev::kBlock)
fwdTailFixupKernel(FwdArgs p, ConvGeom g) {
  fwdTailFixupBody(p, g);
}

// the fold for the split tiles of a batch; grid = (most split tiles of an item, BM*BN / 1024, items)
__global__ void __launch_bounds__(dev::kBlock)
fwdTailFixupBatchKernel(FwdBatch b) {
  const FwdBatchItem &it = b.item[blockIdx.z];
  if ((int)blockIdx.x >= it.p.tail) return;
  fwdTailFixupBody(it.p, it.g);
}

#include "half_parts.h"

// ---- weight gradient, second generation ------------------------------------------
// partial[split][o][k] = sum over the split's positions r = (n, l) of gy[n][o][l] * col[k][n,l].
// Same MFMA core and float4 operand layout as the forward kernels, with the reduction
// running over positions: 4 consecutive l of one gradOutput row are already a float4
// in memory (L % 4 == 0), so the A tile goes from 16-byte buffer loads to
// ds_write_b128 without a transpose. For the B tile a lane owns one position of the
// k-tile and 8 columns k; the columns never change, so their tap offsets are resolved
// once into registers, the images carry their zero border in memory (no bounds test)
// and a gather costs one add per element on top of one position update per k-tile.
// 16 consecutive lanes gather 16 consecutive positions (64-byte runs of x).
// L16: L % 16 == 0 - a k-tile never crosses an image, so the gradOutput offsets are a
// fixed VGPR part plus a scalar part.
constexpr int kSmallPositions = 64;  // positions of a k-tile of the small tiles (BK of the large ones)
struct GradWeightArgs {
  const float *gy;  // (N, M, L)
  const float *x;   // (N, Cin, H, W) of g: images with their zero border
  float *partial;   // (splits, M, Ncols)
  float *biasPartial;  // (splits, M) row sums of gy per split, or null: the bias gradient comes out of the same pass
  int M, Ncols;     // Cout, K
  int mTiles, nTiles;
  int totalKt, ktPerSplit;  // k-tiles of BK (small tiles: kSmallPositions) positions over the N*L positions; per split
  int gyBytes, xBytes;      // < 2^31
  unsigned magicOW;
  unsigned magicKK, magicKW;  // reciprocals of kH * kW and kW (dev::magicOf)
  int Lvalid;               // positions of an image (g.L may count the padding of the gradOutput rows)
  const uint2 *gySlots, *xSlots;  // HALVES: ranges of gyNSlots / xNSlots slices of every image (rangesKernel)
  int gyNSlots, xNSlots;
};

// Small gradWeights (first layers, narrow 1x1 convolutions), where the large tiles would spend most of their
// multiplications on padding: tiles of 32 TI x 32 TJ. A k-tile is 64 positions, every wave multiplies 16 of them with the
// whole tile, and the four sums are added through LDS at the end. Split operands as in the large tiles. Loads: 16 lanes
// fetch 256 consecutive bytes of a gradOutput row with 16-byte loads; a wave gathers one column of the image at 64
// consecutive positions, the tap being a scalar, and transposes 4 x 4 elements inside quads so that LDS holds whole groups
// of positions. One LDS buffer and registers for the next k-tile: two to four workgroups per CU cover the barriers.
// Bound by the vector ALU (24 elements split per lane against 12 matrix instructions of a wave for 64 x 32).
template <int TI, int TJ>
__global__ void __launch_bounds__(dev::kBlock, TI * TJ >= 4 ? 2 : 3)
convGradWeightSmallKernel(GradWeightArgs p, ConvGeom g) {
  constexpr int TBM = 32 * TI, TBN = 32 * TJ, KP = kSmallPositions;
  constexpr int AP = TBM + 4, BP = TBN + 4;   // a row of 16-byte groups; +4: the 8 position groups of a store spread over the banks
  constexpr int NA = TBM / 16, NC = TBN / 4;  // 16-byte gradOutput loads and gathered columns of a lane per k-tile
  constexpr int RQ = TI * TJ * 4;             // groups of 4 accumulator registers
  constexpr int TILE = 3 * 8 * (AP + BP), FOLD = 4 * RQ * dev::kWave;
  __shared__ u32x4 lds[TILE > FOLD ? TILE : FOLD];  // [part][group of 8 positions][row], then [..][column]; at the end the sums
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int tilesPerSplit = p.mTiles * p.nTiles;
  const int bid = dev::xcdRemap(blockIdx.x, gridDim.x);  // the tiles of one split are neighbours: same XCD, same L2
  const int split = bid / tilesPerSplit, tileIdx = bid - split * tilesPerSplit;
  const int mTile = tileIdx % p.mTiles, nTile = tileIdx / p.mTiles;
  const int m0 = mTile * TBM, j0 = nTile * TBN;
  const int ktBegin = split * p.ktPerSplit;
  const int ktEnd = min(p.totalKt, ktBegin + p.ktPerSplit);

  // (n, l) of a position; positions past the batch have n == N
  auto locate = [&](unsigned r, int &n, int &l) {
    n = min((int)(r / (unsigned)g.L), g.N), l = (int)(r - (unsigned)n * (unsigned)g.L);
  };
  auto advance = [&](int &n, int &l) {
    for (l += KP; l >= g.L && n < g.N; ++n) l -= g.L;
  };
  // ---- gradOutput: rows (t >> 4) + 16 i, positions 4 * (t & 15) .. + 3 of the k-tile
  const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc((void *)p.gy, 0, p.gyBytes, 0x00020000);
  const int imgStrideA = p.M * g.L * 4;
  int rowOffA[NA], nA, lA;
#pragma unroll
  for (int i = 0; i < NA; ++i) rowOffA[i] = min(m0 + (t >> 4) + 16 * i, p.M - 1) * g.L * 4;  // rows past M: dropped in the end
  locate((unsigned)ktBegin * KP + (t & 15) * 4, nA, lA);
  // ---- image: position `lane` of the k-tile, columns NC * wave .. + NC - 1
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, p.xBytes, 0x00020000);
  auto columnOffset = [&](int col) {  // byte offset of a column's tap; columns past K are dropped in the end
    const int k = min(col, p.Ncols - 1), KK = g.kH * g.kW;
    const int c = dev::fastDiv(k, p.magicKK), rem = k - c * KK;
    const int kh = dev::fastDiv(rem, p.magicKW), kw = rem - kh * g.kW;
    return ((c * g.H + kh * g.dilH) * g.W + kw * g.dilW) * 4;
  };
  int tap[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) tap[i] = __builtin_amdgcn_readfirstlane(columnOffset(j0 + wave * NC + i));
  const int imgStrideB = g.Cin * g.H * g.W * 4;
  int nB, lB;
  locate((unsigned)ktBegin * KP + lane, nB, lB);
  // byte offset of a position; past the batch, and past the image's last position (gradOutput rows padded to a multiple
  // of 4, zeros there): out of range, reads as 0
  auto positionOffset = [&](int n, int l) {
    const int oh = dev::fastDiv(l, p.magicOW), ow = l - oh * g.oW;
    return n < g.N && l < p.Lvalid ? n * imgStrideB + (oh * g.dH * g.W + ow * g.dW) * 4 : 0x7fffffff;
  };

  u32x4 ra[NA];
  unsigned rb[NC];
  auto loadTiles = [&]() {
    const int offA = nA < g.N ? nA * imgStrideA + lA * 4 : 0x7fffffff;
#pragma unroll
    for (int i = 0; i < NA; ++i)
      ra[i] = __builtin_amdgcn_raw_buffer_load_b128(gr, (int)((unsigned)offA + (unsigned)rowOffA[i]), 0, 0);
    const int offB = positionOffset(nB, lB);
#pragma unroll
    for (int i = 0; i < NC; ++i) rb[i] = __builtin_amdgcn_raw_buffer_load_b32(xr, offB, tap[i], 0);
    advance(nA, lA);
    advance(nB, lB);
  };
  u32x2 *aDst = reinterpret_cast<u32x2 *>(lds + ((t & 15) >> 1) * AP + (t >> 4)) + (t & 1);
  u32x2 *bDst = reinterpret_cast<u32x2 *>(lds + 24 * AP + (lane >> 3) * BP + wave * NC + (lane & 3)) + ((lane >> 2) & 1);
  const bool rowSums = nTile == 0 && p.biasPartial != nullptr;  // the bias gradient rides along
  float rowSum[NA] = {};
  auto split4 = [](const u32x4 &v, u32x2 (&part)[3]) {
    unsigned h[2], m[2], l[2];
    splitPair(v.x, v.y, h[0], m[0], l[0]);
    splitPair(v.z, v.w, h[1], m[1], l[1]);
    part[0] = u32x2{h[0], h[1]}, part[1] = u32x2{m[0], m[1]}, part[2] = u32x2{l[0], l[1]};
  };
  auto storeTiles = [&]() {
    u32x2 part[3];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      split4(ra[i], part);
#pragma unroll
      for (int s = 0; s < 3; ++s) aDst[2 * (s * 8 * AP + 16 * i)] = part[s];
      if (rowSums) {
        const unsigned ex = ra[i].x, ey = ra[i].y, ez = ra[i].z, ew = ra[i].w;
        rowSum[i] += (__uint_as_float(ex) + __uint_as_float(ey)) + (__uint_as_float(ez) + __uint_as_float(ew));
      }
    }
#pragma unroll
    for (int i = 0; i < NC / 4; ++i) {
      split4(dev::quadTranspose(rb[4 * i], rb[4 * i + 1], rb[4 * i + 2], rb[4 * i + 3]), part);
#pragma unroll
      for (int s = 0; s < 3; ++s) bDst[2 * (s * 8 * BP + 4 * i)] = part[s];
    }
  };
  const int grp = lane >> 5, idx = lane & 31;
  const u32x4 *aSrc = lds + (2 * wave + grp) * AP + idx, *bSrc = lds + 24 * AP + (2 * wave + grp) * BP + idx;

  float16v acc[TI][TJ], lo[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = lo[i][j][v] = 0.f;
  loadTiles();
#pragma unroll 1
  for (int kt = ktBegin; kt < ktEnd; ++kt) {
    storeTiles();
    __syncthreads();
    u32x4 a[3][TI], b[3][TJ];
#pragma unroll
    for (int s = 0; s < 3; ++s) {
#pragma unroll
      for (int i = 0; i < TI; ++i) a[s][i] = aSrc[s * 8 * AP + 32 * i];
#pragma unroll
      for (int j = 0; j < TJ; ++j) b[s][j] = bSrc[s * 8 * BP + 32 * j];
    }
    loadTiles();  // (one k-tile past the end at the last: inside the tensors or out of range)
    mfmaSplit(a, b, acc, lo);
    __syncthreads();
  }

#pragma unroll
  for (int j = 0; j < TJ; ++j)
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      if (!finishSums(acc[i][j], lo[i][j])) continue;
      // the block over the wave's positions again with the fp32 instruction, straight from memory
      const unsigned off = (unsigned)columnOffset(j0 + j * 32 + idx);
      const unsigned rOff = (unsigned)(min(m0 + i * 32 + idx, p.M - 1) * g.L * 4);
      acc[i][j] = fp32Block(float16v{}, ktEnd - ktBegin, [&](int s, float (&a)[8], float (&b)[8]) {
#pragma unroll
        for (int q = 0; q < 8; q += 4) {  // 4 positions of one image
          int n, l;
          locate((unsigned)(ktBegin + s) * KP + wave * 16 + 8 * grp + q, n, l);
          const unsigned at = n < g.N ? (unsigned)(n * imgStrideA + l * 4) : 0x7fffffffu;
          put4(a + q, __builtin_amdgcn_raw_buffer_load_b128(gr, (int)(at + rOff), 0, 0));
#pragma unroll
          for (int e = 0; e < 4; ++e)
            b[q + e] = __uint_as_float(
                __builtin_amdgcn_raw_buffer_load_b32(xr, (int)((unsigned)positionOffset(n, l + e) + off), 0, 0));
        }
      });
    }

  // the four waves' sums; lane holds column (lane & 31), rows 8 * (v / 4) + 4 * (lane / 32) + v % 4 of each block
  float4 *fold = reinterpret_cast<float4 *>(lds);
#pragma unroll
  for (int r = 0; r < RQ; ++r) {
    const float16v &c = acc[r / (4 * TJ)][(r >> 2) % TJ];
    fold[(wave * RQ + r) * dev::kWave + lane] = make_float4(c[4 * (r & 3)], c[4 * (r & 3) + 1], c[4 * (r & 3) + 2], c[4 * (r & 3) + 3]);
  }
  __syncthreads();
  float *dst = p.partial + (long)split * p.M * p.Ncols;
#pragma unroll
  for (int u = 0; u < RQ / 4; ++u) {  // each wave folds and stores a quarter
    const int r = wave * (RQ / 4) + u;
    float4 v = fold[r * dev::kWave + lane];
#pragma unroll
    for (int q = 1; q < 4; ++q) {
      const float4 w = fold[(q * RQ + r) * dev::kWave + lane];
      v.x += w.x, v.y += w.y, v.z += w.z, v.w += w.w;
    }
    const int row = m0 + r / (4 * TJ) * 32 + 8 * (r & 3) + 4 * grp, col = j0 + (r >> 2) % TJ * 32 + idx;
    const float vals[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (row + e < p.M && col < p.Ncols) dst[(long)(row + e) * p.Ncols + col] = vals[e];
  }
  if (rowSums) {
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      float v = rowSum[i];  // the 16 lanes that loaded parts of a row
      v = dev::dppAdd<0xB1>(v), v = dev::dppAdd<0x4E>(v), v = dev::dppAdd<0x141>(v), v = dev::dppAdd<0x140>(v);
      const int row = m0 + (t >> 4) + 16 * i;
      if ((t & 15) == 0 && row < p.M) p.biasPartial[(long)split * p.M + row] = v;
    }
  }
}

// The large tiles on split operands (fp32 products on the bf16 matrix pipe, see the forward kernel): a matrix
// instruction consumes 8 consecutive positions per lane, so the operands of a k-tile sit in LDS as 16-byte groups of
// 8 positions, one array per part. Both loaders hand over 4 consecutive positions of a row or column at a time:
//  * gradOutput: 16-byte loads, as they are in memory
//  * image, B4: 4 consecutive positions of a column are 4 consecutive floats (unit stride along the row, and the 4
//    positions never straddle two output rows - or the rows follow each other without a gap): 16-byte loads
//  * image, else: a lane owns one position of the k-tile and gathers groups of 4 neighbouring columns (16 lanes read
//    16 consecutive positions, 64-byte runs); the 4 lanes of a quad then transpose their 4 x 4 elements through DPP
// WM = 2: 128 x 128 tiles of gradWeight (Cout x K), WM = 1: 64 x 256 tiles; a wave multiplies 64 x 64 either way.
// A block whose sums are not all finite is computed again with the fp32 instruction, straight from memory.
// HALVES: for long reductions. A split whose images are held by two fp16 parts (half_parts.h), scaled by the largest element
// of either operand among them, takes these and three products, any other split the three bf16 parts; five times as many
// splits keep the sums as exact as six products do (there is no register left to fold them as conv_halves.h does). Whole pass,
// ranges (20 us) and a longer fold (18) included, us: 256 x 2304 over 64 x 28 x 28 positions 339 -> 272 (395 where no split can).
// What bounds it: as the forward kernel, two workgroups per CU and a clock that power pulls down. Against the fp32
// instruction: 256 x 2304 over 64 x 28 x 28 positions (59.2 GFLOP) 519 -> 334 us; 192 x 720 over 32 x 71 x 71 (64 x 256
// tiles, gathers transposed) 462 -> 342 us; 256 x 2048, stride 2, over 64 x 14 x 14 142 -> 99 us.
// NP: parts; split: of the reduction; sc: scale of the fp16 parts (NP = 2).
template <int WM, int NP>
struct GradWeightLds {
  static constexpr int AP = 64 * WM + 8, BP = 256 / WM + 8;  // 16-byte groups (8 positions of one part) per position-group row
  u32x4 a[2][NP][2][AP];                        // [buffer][part][group of 8 positions][row]
  u32x4 b[2][NP][2][BP];
};
template <bool L16, int WM, bool B4, int NP>
__device__ __forceinline__ void gradWeightSplitBody(const GradWeightArgs &p, const ConvGeom &g, int split, int tileIdx,
                                                    GradWeightLds<WM, NP> &lds, const HalvesScale &sc) {
  constexpr int TBM = 64 * WM, TBN = 256 / WM;
  constexpr int AP = GradWeightLds<WM, NP>::AP, BP = GradWeightLds<WM, NP>::BP;
  constexpr int NQ = TBN / 64;                  // groups of 4 positions a lane parks per k-tile
  constexpr int NT = B4 ? NQ : 4 * NQ;          // columns a lane fetches
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = WM == 2 ? wave >> 1 : 0, wn = WM == 2 ? wave & 1 : wave;
  const int mTile = tileIdx % p.mTiles, nTile = tileIdx / p.mTiles;
  const int m0 = mTile * TBM, j0 = nTile * TBN;
  const int ktBegin = split * p.ktPerSplit;
  const int ktEnd = min(p.totalKt, ktBegin + p.ktPerSplit);
  const int kOob = 0x7fffffff;

  // ---- gradOutput. WM = 2: row t >> 1, positions 8 * (t & 1) .. + 7 of the k-tile; WM = 1: row t >> 2, positions
  //      4 * (t & 3) .. + 3
  const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc((void *)p.gy, 0, p.gyBytes, 0x00020000);
  const int rowA = WM == 2 ? t >> 1 : t >> 2;
  const int pgA = WM == 2 ? (t & 1) * 2 : t & 3;  // first group of 4 positions of the lane
  const int rowOffA = min(m0 + rowA, p.M - 1) * g.L * 4;  // rows past M are clamped and dropped in the epilogue
  const int imgStrideA = p.M * g.L * 4;
  int nA, lA;  // L16: scalar image and position of the k-tile; else: of this lane's first group
  {
    const unsigned r = (unsigned)ktBegin * BK + (L16 ? 0 : pgA * 4);  // N * L < 2^31
    nA = (int)(r / (unsigned)g.L);
    lA = (int)(r - (unsigned)nA * (unsigned)g.L);
  }
  // ---- image. B4: positions 4 * (t & 3) .. + 3, columns (t >> 2) + 64 i;
  //             else position t & 15, columns 4 * (t >> 4) + 64 i .. + 3
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, p.xBytes, 0x00020000);
  const int rB = B4 ? (t & 3) * 4 : t & 15;
  auto columnOffset = [&](int col) {  // byte offset of a column's tap; columns past K are dropped in the epilogue
    const int k = min(col, p.Ncols - 1), KK = g.kH * g.kW;
    const int c = dev::fastDiv(k, p.magicKK), rem = k - c * KK;
    const int kh = dev::fastDiv(rem, p.magicKW), kw = rem - kh * g.kW;
    return ((c * g.H + kh * g.dilH) * g.W + kw * g.dilW) * 4;
  };
  int tapOff[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) tapOff[i] = columnOffset(j0 + (B4 ? (t >> 2) + 64 * i : (t >> 4) * 4 + 64 * (i >> 2) + (i & 3)));
  const int imgStrideB = g.Cin * g.H * g.W * 4;
  const int rowStepB = g.dH * g.W * 4, colStepB = g.dW * 4;
  int lB, nOffB;  // position inside the image, byte offset of the image (>= xBytes past the batch: loads return 0)
  {
    const unsigned r = (unsigned)ktBegin * BK + rB;
    const int n = (int)(r / (unsigned)g.L);
    lB = (int)(r - (unsigned)n * (unsigned)g.L);
    nOffB = n * imgStrideB;
  }
  // byte offset of position l of the image at nOff (positions behind the image's last one exist when the gradOutput
  // rows were padded to a multiple of 4: zeros in gradOutput, and out of range here, which reads as 0 too)
  auto positionOffset = [&](int l, int nOff) {
    const int oh = dev::fastDiv(l, p.magicOW), ow = l - oh * g.oW;
    return l < p.Lvalid ? nOff + oh * rowStepB + ow * colStepB : kOob;
  };

  u32x4 ra[WM];
  u32x4 rb[NQ];                 // B4: 4 positions of a column
  unsigned re[B4 ? 1 : NT];     // else: one position of each column
  // loads the k-tile the position counters stand on, then advances them by BK (L >= BK: one wrap at most)
  auto loadTiles = [&]() {
    if constexpr (L16) {
      // N*L is a multiple of BK here, so every k-tile lies inside the batch (the scalar offset is not range-checked)
      const int so = __builtin_amdgcn_readfirstlane(nA * imgStrideA + lA * 4);
#pragma unroll
      for (int i = 0; i < WM; ++i) ra[i] = __builtin_amdgcn_raw_buffer_load_b128(gr, rowOffA + pgA * 16 + 16 * i, so, 0);
    } else {
      ra[0] = __builtin_amdgcn_raw_buffer_load_b128(gr, nA < g.N ? nA * imgStrideA + rowOffA + lA * 4 : kOob, 0, 0);
      if constexpr (WM == 2) {
        int n1 = nA, l1 = lA + 4;
        if (l1 >= g.L) l1 -= g.L, ++n1;
        ra[1] = __builtin_amdgcn_raw_buffer_load_b128(gr, n1 < g.N ? n1 * imgStrideA + rowOffA + l1 * 4 : kOob, 0, 0);
      }
    }
    lA += BK;
    if (lA >= g.L) lA -= g.L, ++nA;
    const unsigned posOff = (unsigned)positionOffset(lB, nOffB);
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      if constexpr (B4)
        rb[i] = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)(posOff + (unsigned)tapOff[i]), 0, 0);
      else
        re[i] = __builtin_amdgcn_raw_buffer_load_b32(xr, (int)(posOff + (unsigned)tapOff[i]), 0, 0);
    }
    lB += BK;
    if (lB >= g.L) lB -= g.L, nOffB += imgStrideB;
  };
  constexpr int PA = 2 * AP, PB = 2 * BP;      // 16-byte groups of one part in one buffer
  constexpr int BUFA = NP * PA, BUFB = NP * PB;  // of one buffer
  u32x4 *aDst = &lds.a[0][0][pgA >> 1][rowA];
  const int pgB = B4 ? t & 3 : (t & 15) >> 2, colB = B4 ? t >> 2 : (t >> 4) * 4 + (t & 3);
  u32x2 *bDst = reinterpret_cast<u32x2 *>(&lds.b[0][0][pgB >> 1][colB]) + (pgB & 1);
  // The workgroups of the first column tile also sum the gradOutput elements they pass on (each element of a
  // row is loaded by exactly one lane of exactly one of them): the bias gradient without a second pass over gy.
  const bool rowSums = nTile == 0 && p.biasPartial != nullptr;
  float rowSum = 0.f;
  auto split4 = [](const u32x4 &v, u32x2 (&part)[NP], float scale) {  // scale: of fp16 parts
    unsigned h[2], m[2], l[2];
    if constexpr (NP == 2) {
      const unsigned ux = v.x, uy = v.y, uz = v.z, uw = v.w;
      const float x = __uint_as_float(ux), y = __uint_as_float(uy), z = __uint_as_float(uz), w = __uint_as_float(uw);
      splitHalves(x * scale, y * scale, h[0], m[0]);
      splitHalves(z * scale, w * scale, h[1], m[1]);
      part[0] = u32x2{h[0], h[1]}, part[1] = u32x2{m[0], m[1]};
    } else {
      splitPair(v.x, v.y, h[0], m[0], l[0]);
      splitPair(v.z, v.w, h[1], m[1], l[1]);
      part[0] = u32x2{h[0], h[1]}, part[1] = u32x2{m[0], m[1]}, part[2] = u32x2{l[0], l[1]};
    }
  };
  auto storeTiles = [&](auto bufc) {
    constexpr int buf = decltype(bufc)::value;
    u32x2 pa[WM][NP];
#pragma unroll
    for (int i = 0; i < WM; ++i) split4(ra[i], pa[i], sc.gy);
#pragma unroll
    for (int s = 0; s < NP; ++s) {
      if constexpr (WM == 2)
        aDst[buf * BUFA + s * PA] = u32x4{pa[0][s].x, pa[0][s].y, pa[1][s].x, pa[1][s].y};
      else
        (reinterpret_cast<u32x2 *>(aDst + buf * BUFA + s * PA))[pgA & 1] = pa[0][s];
    }
    if (rowSums) {
#pragma unroll
      for (int i = 0; i < WM; ++i) {
        // (element by element: a bit cast applied to a vector element expression reads element 0 here)
        const unsigned ex = ra[i].x, ey = ra[i].y, ez = ra[i].z, ew = ra[i].w;
        rowSum += (__uint_as_float(ex) + __uint_as_float(ey)) + (__uint_as_float(ez) + __uint_as_float(ew));
      }
    }
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      if constexpr (!B4) rb[i] = dev::quadTranspose(re[4 * i], re[4 * i + 1], re[4 * i + 2], re[4 * i + 3]);
      u32x2 pb[NP];
      split4(rb[i], pb, sc.x);
#pragma unroll
      for (int s = 0; s < NP; ++s) bDst[2 * (buf * BUFB + s * PB + 64 * i)] = pb[s];
    }
  };
  const int grp = lane >> 5, idx = lane & 31;
  const u32x4 *aSrc = &lds.a[0][0][grp][wm * 64 + idx];
  const u32x4 *bSrc = &lds.b[0][0][grp][wn * 64 + idx];
  using Buf0 = std::integral_constant<int, 0>;
  using Buf1 = std::integral_constant<int, 1>;

  float16v acc[2][2], lo[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = lo[i][j][v] = 0.f;

  // same software pipeline as the forward kernel: tile kt in LDS, kt + 1 in registers, kt + 2 requested
  auto step = [&](auto cur, auto nxt, bool store, bool load) {
    constexpr int C = decltype(cur)::value;
    u32x4 a[NP][2], b[NP][2];
#pragma unroll
    for (int s = 0; s < NP; ++s) {
#pragma unroll
      for (int i = 0; i < 2; ++i) a[s][i] = aSrc[C * BUFA + s * PA + 32 * i];
#pragma unroll
      for (int j = 0; j < 2; ++j) b[s][j] = bSrc[C * BUFB + s * PB + 32 * j];
    }
    if (store) storeTiles(nxt);
    if (load) loadTiles();
    if constexpr (NP == 2)
      mfmaHalves(a, b, acc, lo);
    else
      mfmaSplit(a, b, acc, lo);
    __syncthreads();
  };
  if (ktBegin < ktEnd) {
    loadTiles();
    storeTiles(Buf0{});
    if (ktBegin + 1 < ktEnd) loadTiles();
    __syncthreads();
    int kt = ktBegin;
    for (; kt + 3 < ktEnd; kt += 2) {  // tile kt sits in buffer 0, tile kt + 1 in registers
      step(Buf0{}, Buf1{}, true, true);
      step(Buf1{}, Buf0{}, true, true);
    }
    // one to three tiles left
    step(Buf0{}, Buf1{}, kt + 1 < ktEnd, kt + 2 < ktEnd);
    if (kt + 1 < ktEnd) step(Buf1{}, Buf0{}, kt + 2 < ktEnd, false);
    if (kt + 2 < ktEnd) step(Buf0{}, Buf1{}, false, false);
  }

#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if constexpr (NP == 2) {
        if (!finishHalves(acc[i][j], lo[i][j], -(sc.gyExp + sc.xExp))) continue;
      } else {
        if (!finishSums(acc[i][j], lo[i][j])) continue;
      }
      // the block again with the fp32 instruction, straight from memory
      const unsigned tap = (unsigned)columnOffset(j0 + wn * 64 + j * 32 + idx);
      const int rOff = min(m0 + wm * 64 + i * 32 + idx, p.M - 1) * g.L * 4;
      acc[i][j] = fp32Block(float16v{}, ktEnd - ktBegin, [&](int s, float (&a)[8], float (&b)[8]) {
#pragma unroll
        for (int q = 0; q < 8; q += 4) {  // 4 positions of one image
          const unsigned r = (unsigned)(ktBegin + s) * BK + 8 * grp + q;
          const int n = (int)(r / (unsigned)g.L), l = (int)(r - (unsigned)n * (unsigned)g.L);
          put4(a + q, __builtin_amdgcn_raw_buffer_load_b128(gr, n < g.N ? n * imgStrideA + rOff + l * 4 : kOob, 0, 0));
#pragma unroll
          for (int e = 0; e < 4; ++e)
            b[q + e] = __uint_as_float(
                __builtin_amdgcn_raw_buffer_load_b32(xr, (int)((unsigned)positionOffset(l + e, n * imgStrideB) + tap), 0, 0));
        }
      });
    }

  // lane holds column (lane & 31), rows 8*(v/4) + 4*(lane/32) + v%4 of each 32x32 tile
  float *dst = p.partial + (long)split * p.M * p.Ncols;
#pragma unroll
  for (int tj = 0; tj < 2; ++tj) {
    const int col = j0 + wn * 64 + tj * 32 + idx;
    if (col >= p.Ncols) continue;
#pragma unroll
    for (int ti = 0; ti < 2; ++ti)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = m0 + wm * 64 + ti * 32 + 8 * (v >> 2) + grp * 4 + (v & 3);
        if (row < p.M) dst[(long)row * p.Ncols + col] = acc[ti][tj][v];
      }
  }
  if (rowSums) {
    // the 2 (WM = 2) or 4 (WM = 1) lanes that loaded parts of a row are neighbours inside a quad
    rowSum = dev::dppAdd<0xB1>(rowSum);
    if (WM == 1) rowSum = dev::dppAdd<0x4E>(rowSum);
    if ((t & (WM == 2 ? 1 : 3)) == 0 && m0 + rowA < p.M) p.biasPartial[(long)split * p.M + m0 + rowA] = rowSum;
  }
}

template <bool L16, int WM, bool B4, bool HALVES>
__global__ void __launch_bounds__(dev::kBlock, 2)
convGradWeightSplitKernel(GradWeightArgs p, ConvGeom g) {
  // workgroups that reduce the same positions (one split) are neighbours in the remapped order: same XCD, same L2
  const int tilesPerSplit = p.mTiles * p.nTiles;
  const int bid = dev::xcdRemap(blockIdx.x, gridDim.x);
  const int split = bid / tilesPerSplit, tileIdx = bid - split * tilesPerSplit;
  if constexpr (HALVES) {
    __shared__ union {
      GradWeightLds<WM, 2> two;
      GradWeightLds<WM, 3> three;
    } lds;
    const long r0 = (long)split * p.ktPerSplit * BK, r1 = min((long)p.totalKt, (long)(split + 1) * p.ktPerSplit) * BK;
    const int n0 = (int)(r0 / g.L), n1 = min(g.N, (int)((r1 - 1) / g.L) + 1);
    const HalvesScale sc = halvesScale(p.gySlots, p.gyNSlots, p.xSlots, p.xNSlots, n0, n1);
    if (sc.fits)
      gradWeightSplitBody<L16, WM, B4, 2>(p, g, split, tileIdx, lds.two, sc);
    else
      gradWeightSplitBody<L16, WM, B4, 3>(p, g, split, tileIdx, lds.three, sc);
  } else {
    __shared__ GradWeightLds<WM, 3> lds;
    gradWeightSplitBody<L16, WM, B4, 3>(p, g, split, tileIdx, lds, HalvesScale{});
  }
}

// gW[i] += scale * sum_s partial[s][i] in a fixed association: a workgroup owns 64 consecutive float4
// of gW; its 4 lane groups each sum the splits s = group, group + 4, ... with 4 independent
// accumulators (16 16-byte loads in flight per lane), then the groups are added in order through
// LDS. With few elements and hundreds of splits (1x1 convolutions) a one-lane-per-element loop is
// latency bound; this form keeps enough bytes in flight to run at memory speed.
// Blocks past the last float4 of gW do the same for the bias partials (biasPartial(splits, M), M % 4 == 0), when given.
// E: float4 of gW a workgroup owns (64, 16 or 4); its 256 / E lane groups share the splits. Small
// gradWeights with thousands of splits take small E: more workgroups, more loads in flight.
template <int E>
__global__ void __launch_bounds__(dev::kBlock)
foldPartials4Kernel(const float *__restrict__ partial, float *__restrict__ dst, long count4, int splits, float scale,
                    const float *__restrict__ biasPartial, float *__restrict__ gradBias, int M, int gwBlocks) {
  constexpr int G = dev::kBlock / E;
  __shared__ float4 part[G][E];
  int blk = blockIdx.x;
  if (blk >= gwBlocks) blk -= gwBlocks, partial = biasPartial, dst = gradBias, count4 = M >> 2;
  const int e = threadIdx.x % E, grp = threadIdx.x / E;
  const long i = (long)blk * E + e;
  float4 a[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) a[u] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (i < count4) {
    const float4 *p = reinterpret_cast<const float4 *>(partial) + i;
    int s = grp;
    for (; s + 3 * G < splits; s += 4 * G) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float4 v = loadOnce4(p + (long)(s + G * u) * count4);  // the partials' only reader
        a[u].x += v.x, a[u].y += v.y, a[u].z += v.z, a[u].w += v.w;
      }
    }
    for (; s < splits; s += G) {
      const float4 v = loadOnce4(p + (long)s * count4);
      a[0].x += v.x, a[0].y += v.y, a[0].z += v.z, a[0].w += v.w;
    }
  }
  part[grp][e] = make_float4((a[0].x + a[1].x) + (a[2].x + a[3].x), (a[0].y + a[1].y) + (a[2].y + a[3].y),
                             (a[0].z + a[1].z) + (a[2].z + a[3].z), (a[0].w + a[1].w) + (a[2].w + a[3].w));
  __syncthreads();
  if (grp == 0 && i < count4) {
    float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
    for (int q = 0; q < G; q += 4) {
      const float4 p0 = part[q][e], p1 = part[q + 1][e], p2 = part[q + 2][e], p3 = part[q + 3][e];
      t.x += (p0.x + p1.x) + (p2.x + p3.x), t.y += (p0.y + p1.y) + (p2.y + p3.y);
      t.z += (p0.z + p1.z) + (p2.z + p3.z), t.w += (p0.w + p1.w) + (p2.w + p3.w);
    }
    float4 d = reinterpret_cast<float4 *>(dst)[i];
    d.x += scale * t.x, d.y += scale * t.y, d.z += scale * t.z, d.w += scale * t.w;
    reinterpret_cast<float4 *>(dst)[i] = d;
  }
}

// the same for any count / alignment: gW[i] += scale * sum_s partial[s][i], s ascending
__global__ void __launch_bounds__(dev::kBlock)
foldPartialsKernel(const float *__restrict__ partial, float *__restrict__ dst, long count, int splits, float scale) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (long)gridDim.x * blockDim.x) {
    float s = 0.f;
    for (int k = 0; k < splits; ++k) s += partial[(long)k * count + i];
    dst[i] += scale * s;
  }
}

// gradBias[o] += scale * sum_{n,l} gy[n][o][l]   (lib/THCUNN/generic/SpatialConvolutionMM.cu:440-455)
// One 1024-lane workgroup per output plane o streams its N runs of L floats.
constexpr int kBiasBlock = 1024;
template <bool VEC>
__global__ void __launch_bounds__(kBiasBlock)
gradBiasKernel(const float *__restrict__ gy, float *__restrict__ gradBias, int N, int Cout, int L, float scale) {
  __shared__ float red[kBiasBlock / dev::kWave];
  const int o = blockIdx.x;
  float acc = 0.f;
  if (VEC) {
    const int L4 = L >> 2;
    const int total4 = N * L4;
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
    for (int i = threadIdx.x; i < total4; i += kBiasBlock) {
      int n = i / L4, l4 = i - n * L4;
      float4 v = *reinterpret_cast<const float4 *>(gy + ((long)n * Cout + o) * L + (l4 << 2));
      a0 += v.x, a1 += v.y, a2 += v.z, a3 += v.w;
    }
    acc = (a0 + a1) + (a2 + a3);
  } else {
    const long total = (long)N * L;
    for (long i = threadIdx.x; i < total; i += kBiasBlock) {
      int n = (int)(i / L);
      int l = (int)(i - (long)n * L);
      acc += gy[((long)n * Cout + o) * L + l];
    }
  }
  acc = dev::waveSum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.f;
    for (int w = 0; w < kBiasBlock / dev::kWave; ++w) s += red[w];
    gradBias[o] += scale * s;
  }
}

// wt[k][o] = w[o][k] for w (rows x cols)
__global__ void __launch_bounds__(dev::kBlock)
transposeKernel(const float *__restrict__ w, float *__restrict__ wt, int rows, int cols) {
  const long total = (long)rows * cols;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const int o = (int)(i % rows);
    const long k = i / rows;
    wt[i] = w[(long)o * cols + k];
  }
}

// Wf[c][(o, kh', kw')] = W[o][(c, kH-1-kh', kW-1-kw')]: with these weights the
// stride-1 gradInput is a plain forward convolution of gradOutput (padding k-1-pad).
__global__ void __launch_bounds__(dev::kBlock)
flipWeightKernel(const float *__restrict__ w, float *__restrict__ wf, int Cout, int Cin, int kH, int kW) {
  const int KK = kH * kW;
  const long total = (long)Cout * Cin * KK;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    int t = (int)(i % KK);
    long r = i / KK;
    int o = (int)(r % Cout);
    int c = (int)(r / Cout);
    wf[i] = w[((long)o * Cin + c) * KK + (KK - 1 - t)];
  }
}

// ---- im2col / col2im (lib/THCUNN/im2col.h) -----------------------------------
// One lane per column entry; consecutive lanes write consecutive addresses.
__global__ void __launch_bounds__(dev::kBlock)
im2colKernel(const float *__restrict__ im, float *__restrict__ col, int nImg, int C, int H, int W, int kH, int kW,
             int padH, int padW, int dH, int dW, int dilH, int dilW, int oH, int oW) {
  const long L = (long)oH * oW;
  const long perImg = (long)C * kH * kW * L;
  const long total = perImg * nImg;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    long n = i / perImg;
    long r = i - n * perImg;
    int ow = (int)(r % oW);
    r /= oW;
    int oh = (int)(r % oH);
    r /= oH;
    int kw = (int)(r % kW);
    r /= kW;
    int kh = (int)(r % kH);
    int c = (int)(r / kH);
    int h = oh * dH - padH + kh * dilH, w = ow * dW - padW + kw * dilW;
    col[i] = (h >= 0 && w >= 0 && h < H && w < W) ? im[((n * C + c) * H + h) * W + w] : 0.f;
  }
}

// One lane per image pixel gathers every column entry that maps onto it
// (lib/THCUNN/im2col.h:63-102); float accumulation in the reference's order.
__global__ void __launch_bounds__(dev::kBlock)
col2imKernel(const float *__restrict__ col, float *__restrict__ im, int nImg, int C, int H, int W, int kH, int kW,
             int padH, int padW, int dH, int dW, int dilH, int dilW, int oH, int oW, const float *__restrict__ bias) {
  const long total = (long)nImg * C * H * W;
  const int extW = (kW - 1) * dilW + 1, extH = (kH - 1) * dilH + 1;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    int w_im = (int)(i % W) + padW;
    int h_im = (int)((i / W) % H) + padH;
    long nc = i / ((long)W * H);  // n * C + c
    int ws = (w_im < extW) ? 0 : (w_im - extW) / dW + 1;
    int we = min(w_im / dW + 1, oW);
    int hs = (h_im < extH) ? 0 : (h_im - extH) / dH + 1;
    int he = min(h_im / dH + 1, oH);
    float val = bias ? bias[(int)(nc % C)] : 0.f;  // per-plane bias of the transposed convolution, else 0
    for (int hc = hs; hc < he; ++hc)
      for (int wc = ws; wc < we; ++wc) {
        int hk = h_im - hc * dH, wk = w_im - wc * dW;
        if (hk % dilH == 0 && wk % dilW == 0) {
          hk /= dilH;
          wk /= dilW;
          val += col[(((nc * kH + hk) * kW + wk) * oH + hc) * oW + wc];
        }
      }
    im[i] = val;
  }
}

#include "conv_pointwise.h"
#include "conv_pointwise_split.h"
#include "conv_fewplanes.h"
#include "conv_halves.h"

// ---- host side -----------------------------------------------------------------
struct ConvCall {
  ConvGeom g;
  bool batch;
};

ConvGeom makeGeom(int N, int Cin, int Cout, int H, int W, int oH, int oW, int kH, int kW, int dH, int dW, int padH,
                  int padW, int dilH, int dilW) {
  ConvGeom g{};
  g.N = N, g.Cin = Cin, g.Cout = Cout, g.H = H, g.W = W, g.oH = oH, g.oW = oW;
  g.kH = kH, g.kW = kW, g.dH = dH, g.dW = dW, g.padH = padH, g.padW = padW, g.dilH = dilH, g.dilW = dilW;
  g.K = g.Cin * kH * kW;
  g.L = g.oH * g.oW;
  if ((long)g.Cin * g.H * g.W >= 0x7fffffffL || (long)g.Cout * g.L >= 0x7fffffffL || (long)g.K * g.L >= 0x7fffffffL * 8L)
    error("spatial convolution: image too large");
  return g;
}

// Shape rules of lib/THCUNN/generic/SpatialConvolutionMM.cu:5-56 (kConvMM: `weight` 2-D
// (Cout, Cin*kH*kW) or 4-D) and of generic/SpatialDilatedConvolution.cu:5-67 (kDilated: 4-D weight,
// dilation > 0); only the extents of `weight` are read here.
enum ConvFlavor { kConvMM, kDilated };
ConvCall convSetup(THCudaTensor *input, THCudaTensor *gradOutput, THCudaTensor *weight, THCudaTensor *bias,
                   const char *weightName, int kH, int kW, int dH, int dW, int padH, int padW, int dilH = 1,
                   int dilW = 1, ConvFlavor flavor = kConvMM) {
  THC_ARG_CHECK(input && weight, 2, "input and weight tensors expected");
  if (flavor == kDilated)
    THC_ARG_CHECK(weight->nDimension == 4, 4,
                  "4D weight tensor (nOutputPlane,nInputPlane,kH,kW) expected, but got: %s",
                  sizeDesc(erase(weight)).c_str());
  else
    THC_ARG_CHECK(isContiguous(erase(weight)), 4, "%s tensor has to be contiguous", weightName);
  THC_ARG_CHECK(kW > 0 && kH > 0, 9, "kernel size should be greater than zero, but got kH: %d kW: %d", kH, kW);
  THC_ARG_CHECK(dW > 0 && dH > 0, 11, "stride should be greater than zero, but got dH: %d dW: %d", dH, dW);
  if (flavor == kDilated)
    THC_ARG_CHECK(isContiguous(erase(weight)), 4, "%s tensor has to be contiguous", weightName);
  THC_ARG_CHECK(!bias || isContiguous(erase(bias)), 5, "bias tensor has to be contiguous");
  if (flavor == kDilated)
    THC_ARG_CHECK(dilW > 0 && dilH > 0, 14, "dilation should be greater than 0, but got dilationH: %d dilationW: %d",
                  dilH, dilW);
  else
    THC_ARG_CHECK(weight->nDimension == 2 || weight->nDimension == 4, 5,
                  "2D or 4D weight tensor expected, but got: %s", sizeDesc(erase(weight)).c_str());
  long nOutputPlane = weight->size[0];
  long wcols = weight->nDimension == 2 ? weight->size[1] : weight->size[1] * weight->size[2] * weight->size[3];
  if (bias) checkDimSize(erase(bias), "bias", 1, 0, nOutputPlane);
  int ndim = input->nDimension;
  int dimf = 0, dimh = 1, dimw = 2;
  if (ndim == 4) {
    dimf++;
    dimh++;
    dimw++;
  }
  THC_ARG_CHECK(ndim == 3 || ndim == 4, 2, "3D or 4D input tensor expected but got: %s",
                sizeDesc(erase(input)).c_str());
  long nInputPlane = flavor == kDilated ? weight->size[1] : wcols / (kH * kW);
  long inputHeight = input->size[dimh], inputWidth = input->size[dimw];
  long outputHeight = (inputHeight + 2 * padH - (dilH * (kH - 1) + 1)) / dH + 1;
  long outputWidth = (inputWidth + 2 * padW - (dilW * (kW - 1) + 1)) / dW + 1;
  if (outputWidth < 1 || outputHeight < 1)
    error("Given input size: (%ld x %ld x %ld). Calculated output size: (%ld x %ld x %ld). Output size is too small",
          nInputPlane, inputHeight, inputWidth, nOutputPlane, outputHeight, outputWidth);
  checkDimSize(erase(input), "input", ndim, dimf, nInputPlane);
  if (gradOutput) {
    checkDimSize(erase(gradOutput), "gradOutput", ndim, dimf, nOutputPlane);
    checkDimSize(erase(gradOutput), "gradOutput", ndim, dimh, outputHeight);
    checkDimSize(erase(gradOutput), "gradOutput", ndim, dimw, outputWidth);
    if (ndim == 4 && gradOutput->size[0] != input->size[0])
      error("input and gradOutput batch sizes do not match: input %s, gradOutput %s", sizeDesc(erase(input)).c_str(),
            sizeDesc(erase(gradOutput)).c_str());
  }
  if (wcols != nInputPlane * kH * kW)
    error("%s of shape %s does not match a %d x %d kernel", weightName, sizeDesc(erase(weight)).c_str(), kH, kW);
  ConvCall call;
  call.batch = ndim == 4;
  call.g = makeGeom(call.batch ? (int)input->size[0] : 1, (int)nInputPlane, (int)nOutputPlane, (int)inputHeight,
                    (int)inputWidth, (int)outputHeight, (int)outputWidth, kH, kW, dH, dW, padH, padW, dilH, dilW);
  return call;
}

inline unsigned tiles(long n, int b) { return (unsigned)((n + b - 1) / b); }

// Workgroups of `kernel` (256 lanes, static LDS) the whole device holds at once.
// kernel == nullptr: the number of CUs.
int residentSlots(const void *kernel) {
  static std::mutex mu;
  static std::map<std::pair<int, const void *>, int> cache;  // per (device, kernel)
  int dev = 0, cus = 0, perCu = 1;
  THC_HIP_CHECK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  auto it = cache.find({dev, kernel});
  if (it != cache.end()) return it->second;
  THC_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  if (kernel) THC_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, kernel, dev::kBlock, 0));
  int v = std::max(1, cus) * std::max(1, perCu);
  cache[{dev, kernel}] = v;
  return v;
}

// Test switch: "1" routes the forward pass (and the stride-1 gradInput that
// reuses it) through the first-generation kernels.
bool forceGeneric() { return g_switches.convGeneric == 1; }

// Plan of one implicit-GEMM forward launch. The 128x128 tiles are dealt to the
// CUs in rounds; a last partial round would leave most CUs idle while a few
// finish one more tile, so the tiles of that round are instead split along K
// over all CUs (partials in scratch, folded by fwdTailFixupKernel in a fixed order).
// Whole tiles and splits are workgroups of one launch: the splits take the slots
// that the last whole tiles free.
struct FwdPlan {
  int bm, bn;          // tile shape: 128 x 128, or one that wastes fewer rows (tileShape; padded kernel only)
  int direct;          // != 0: convFwdDirectKernel, tiles of 32 * direct rows and columns
  int mTiles, total, full, tail, nSplit, ktPerSplit;
  int tapEntries;      // > 0: the padded kernel applies; entries of the tap table at the start of the scratch
  long paddedFloats;   // floats of the zero-bordered copy of the images (0: no border needed, or generic kernel)
  long weightFloats;   // floats of the copy of the weights with rows padded to a multiple of BK (0: not needed)
  long scratchFloats;  // tap table, tail partials, padded images
};
// Shape of the output tiles for M rows (others: the padded kernel's shapes beside 128 x 128 may be used).
// tiles64, kTiles64: the output in 64 x 128 tiles, and the k-tiles of all of them together.
void tileShape(int M, bool others, long tiles64, long kTiles64, int &bm, int &bn) {
  const long r128 = tiles(M, BM) * (long)BM, r64 = tiles(M, 64) * 64L, r96 = tiles(M, 96) * 96L, r32 = tiles(M, 32) * 32L;
  bm = BM, bn = BN;
  if (!others) return;
  // Short calls - one round of 64 x 128 tiles with short sums, or little work altogether - are bound by the start and end of
  // a workgroup, which the 64 x 128 shape has the shortest of. us, 64 rows / 96 (72 -> 96 rows): 3136 positions, 4 k-tiles 7.1 /
  // 8.9; 12544, 12: 12.3 / 16.5; 2178, 21: 16.5 / 17.7; beyond: 50176, 4: 15.9 / 12.9; 3362, 54: 24.8 / 22.6. 64 rows / 32 (16
  // rows): 3136, 6: 7.6 / 9.7; 12544, 12: 12.9 / 12.5; beyond: 200704, 2: 15.7 / 13.8; 9600, 29 (32 rows): 21.4 / 19.4.
  const bool brief = (tiles64 <= residentSlots(nullptr) && kTiles64 / 12 <= tiles64) || kTiles64 < 1200;
  if (brief && M <= 96) {
    bm = 64;
    return;
  }
  // 96 x 128 where that pads a sixth fewer rows (65 ... 96 rows; its waves read LDS a third more often per product): 80 rows,
  // 3x3 of 192 planes over 32 x 71 x 71 positions 455 us in 32-row tiles, 348 in 96; 288 rows of 128 planes 24.6 in 64, 26.2
  if (r96 * 6 < std::min(r64, r128) * 5)
    bm = 96;
  else if (r32 * 4 <= r64 * 3)  // 32 rows: a wave issues half the matrix instructions per element it gathers
    bm = 32, bn = 256;
  else if (r64 < r128)  // (128 rows or more: 128 x 128 is better, 256 -> 256 3x3 on 28x28, N = 64: 334 against 357 us)
    bm = 64;
}

// Tiles of an M x Ncols output reduced over nkt k-tiles; wideOk: tileShape has its choice.
// over: what a workgroup costs beside its k-tiles, in k-tiles; brief: short calls have a shape of their own.
void planTiles(FwdPlan &pl, int M, long Ncols, int nkt, bool wideOk, double over = 4.0, bool brief = true) {
  const long tiles64 = tiles(M, 64) * (long)tiles(Ncols, 128);
  tileShape(M, wideOk, brief ? tiles64 : LONG_MAX, brief ? tiles64 * nkt : LONG_MAX, pl.bm, pl.bn);
  pl.mTiles = (int)tiles(M, pl.bm);
  pl.total = pl.mTiles * (int)tiles(Ncols, pl.bn);
  const int cus = residentSlots(nullptr);
  // Which tiles to split along K, and how finely: the workgroups go to the CUs in launch order (up to three
  // share a CU), so a CU's time is the sum over what it is dealt. In units of one k-tile of one workgroup alone
  // on its CU: a workgroup costs its k-tiles + 4 (prologue, epilogue), a split tile 0.006 more per partial
  // (written, then read by the fold), and a CU that only ever holds one workgroup runs at 0.85 of the rate (0.75 with 64-row tiles)
  // (nothing covers its barriers) - constants fitted to measured sweeps over S on 14x14 ... 56x56 layers.
  // Candidates: no split; the last, partial round split S ways; every tile split S ways (S <= 16, >= 4 k-tiles
  // per split). E.g. 196 tiles on 256 CUs: 5 splits (980 workgroups, 4 per CU at most) beat 2 (392: 136 CUs
  // carry two halves, 120 one) by 15 %; 136 tiles left over after a full round: 3 splits, not 1.
  const int maxS = std::max(1, std::min(nkt / 4, 16));
  const int q = pl.total / cus, r = pl.total % cus;
  const double lone = pl.bm == 64 ? 0.75 : 0.85;
  auto perWg = [&](int S) { return (double)launch::ceilDiv(nkt, S) + over; };
  // a split has to promise 5 % before it is taken: the model is coarse and the fold is one more launch
  double best = 0.95 * launch::ceilDiv(pl.total, cus) * perWg(1) / (pl.total <= cus ? lone : 1.0);
  int nSplit = 1;
  pl.tail = 0;
  for (int S = 2; S <= maxS; ++S) {
    if (launch::ceilDiv(nkt, launch::ceilDiv(nkt, S)) != S) continue;  // the same pieces as a smaller S
    if (q > 0 && r > 0) {
      const double t = q * perWg(1) + launch::ceilDiv(r * S, cus) * perWg(S) + 0.006 * r * S;
      if (t < best) best = t, nSplit = S, pl.tail = r;
    }
    if (pl.total <= 2 * cus) {
      const int n = launch::ceilDiv(pl.total * S, cus);
      const double t = n * perWg(S) / (n == 1 ? lone : 1.0) + 0.006 * pl.total * S;
      if (t < best) best = t, nSplit = S, pl.tail = pl.total;
    }
  }
  pl.full = pl.total - pl.tail;
  pl.ktPerSplit = launch::ceilDiv(nkt, nSplit);
  pl.nSplit = launch::ceilDiv(nkt, pl.ktPerSplit);
}
inline long partialFloats(const FwdPlan &pl) { return pl.tail ? (long)pl.tail * pl.nSplit * BM * BN : 0; }

// Whether a short call runs on convFwdDirectKernel: one launch, against workgroup tiles that would leave CUs idle or
// have K split over workgroups, with partial tiles in memory and a second launch that folds them. Both times in us, without
// the copies that both need, fitted to 320 calls of 1x1 ... 5x5 windows, strides 1, 2 and 4, up to 4 GFLOP (taking the estimated
// better one costs 0.5 % over the better one). E.g. (tiled / direct): 512 -> 512 1x1 on 14x14, N = 1: 9.8 / 6.3; 256 -> 256 1x1 on
// 14x14, N = 8: 12.8 / 7.7; 128 -> 128 3x3 on 28x28, N = 2: 20.4 / 14.6; 256 -> 64 1x1 on 56x56, N = 8: 12.5 / 15.6; 128 -> 512 1x1
// on 28x28, N = 8: 13.7 / 20.7; 256 -> 32 1x1 on 28x28, N = 48: 21.5 / 19.2. With a stride the lanes' loads touch more cache lines:
// 64 -> 620 4x4 stride 4, 160 positions: 20.6 / 32.0.
// 32 x 32 tiles while those are few, then 64 x 64 (fewer loads per product; the line between them: 64 -> 64 3x3 on
// 56x56, N = 4, 784 tiles of 32 x 32: 23.9 / 20.0; 256 -> 256 1x1 on 14x14, N = 8, 392 tiles: 7.7 / 9.8), which 32 rows cannot
// fill (the last call above with 64 x 64: 25.5).
void planDirect(FwdPlan &pl, int M, long Ncols, int nkt, bool window, bool strided) {
  const int force = g_switches.convDirect;
  if (force == 0) return;
  const long tiles32 = (long)tiles(M, 32) * tiles(Ncols, 32);
  const bool small = tiles32 <= 512 || M <= 32;
  if (force < 0) {
    if (pl.total >= residentSlots(nullptr)) return;  // a workgroup tile for every CU: the tiled kernel is better at any size
    const double tiled = pl.tail > 0 ? (pl.bm == BM ? 6.3 : 4.6) + 0.85 * pl.ktPerSplit + 0.025 * pl.tail * pl.nSplit
                         : pl.bm == BM ? 4.7 + 1.15 * pl.ktPerSplit
                                       : 3.4 + 0.66 * pl.ktPerSplit;
    const double perStep = !small ? 0.25 : strided ? 0.13 : window ? 0.11 : 0.08;   // bound by latency
    const double perTile = !small ? 0.4e-3 : strided ? 0.72e-3 : 0.45e-3;           // bound by loads
    const double direct = 4.3 + 0.002 * tiles32 + std::max(perStep * nkt, perTile * tiles32 * nkt);
    if (direct >= tiled) return;
  }
  pl.direct = force > 0 ? force : small ? 1 : 2;
  pl.bm = pl.bn = 32 * pl.direct;
  pl.mTiles = (int)tiles(M, pl.bm);
  pl.total = pl.full = pl.mTiles * (int)tiles(Ncols, pl.bn);
  pl.tail = 0, pl.nSplit = 1, pl.ktPerSplit = nkt;
}

// wAligned: the weights start on a 16-byte boundary (else the padded kernel works on an aligned copy)
FwdPlan planFwdImplicit(int M, int nImages, const ConvGeom &g, bool wAligned = true, bool direct = true) {
  FwdPlan pl{};
  const int nkt = launch::ceilDiv(g.K, BK);
  const long padded = (long)nImages * g.Cin * (g.H + 2 * g.padH) * (g.W + 2 * g.padW);
  // K that is not a multiple of BK (first layers: Cin = 3) runs on the same kernel with the weight rows
  // copied into rows of Kp = nkt * BK floats, zero beyond K
  const int Kp = nkt * BK;
  const bool fast = !forceGeneric() && padded * 4 < 0x7fffffffL && (long)M * Kp * 4 < 0x7fffffffL;
  planTiles(pl, M, (long)nImages * g.L, nkt, fast);
  if (fast && direct && g.K % BK == 0 && g.Cin % 2 == 0) planDirect(pl, M, (long)nImages * g.L, nkt, g.kH * g.kW > 1, g.dW > 1);
  pl.tapEntries = fast ? Kp + 2 * BK : 0;  // spare entries: the kernel reads tap offsets up to two k-tiles ahead
  pl.paddedFloats = fast && (g.padH > 0 || g.padW > 0) ? padded : 0;
  pl.weightFloats = fast && (Kp != g.K || !wAligned) ? (long)M * Kp : 0;
  pl.scratchFloats = pl.tapEntries + partialFloats(pl) + (pl.paddedFloats + 3) / 4 * 4 + pl.weightFloats;
  return pl;
}

// The launches of one planned forward GEMM: full rounds, then the K-split tail and its fold. `p` carries the
// operands, the output addressing, M, Ncols and the byte sizes; gk is the geometry the kernels see.
void launchFwdKernels(hipStream_t s, const FwdPlan &pl, FwdArgs p, float *partial, const ConvGeom &gk, bool fast) {
  p.mTiles = pl.mTiles;
  p.bm = pl.bm, p.bn = pl.bn;
  p.full = pl.full, p.tail = pl.tail;
  if (pl.direct) {
    if (pl.direct == 1 && p.tapStride > 0)
      convFwdDirectKernel<1, true><<<pl.total, dev::kBlock, 0, s>>>(p, gk);
    else if (pl.direct == 1)
      convFwdDirectKernel<1, false><<<pl.total, dev::kBlock, 0, s>>>(p, gk);
    else if (p.tapStride > 0)
      convFwdDirectKernel<2, true><<<pl.total, dev::kBlock, 0, s>>>(p, gk);
    else
      convFwdDirectKernel<2, false><<<pl.total, dev::kBlock, 0, s>>>(p, gk);
    THC_HIP_CHECK(hipGetLastError());
    return;
  }
  if (fast) {
    // one launch: the tiles reduced by one workgroup first, then the splits of the tail tiles, which fill
    // the slots that the last whole tiles leave
    p.tile0 = pl.full;
    p.nSplit = pl.tail > 0 ? pl.nSplit : 1;
    p.ktPerSplit = pl.tail > 0 ? pl.ktPerSplit : launch::ceilDiv(gk.K, BK);
    p.partial = partial;
    const dim3 grid(pl.full + pl.tail * p.nSplit);
    if (p.tapStride > 0) {
      if (pl.bm == 32)
        convFwdPaddedKernel<0, true><<<grid, dev::kBlock, 0, s>>>(p, gk);
      else if (pl.bm == 64)
        convFwdPaddedKernel<1, true><<<grid, dev::kBlock, 0, s>>>(p, gk);
      else if (pl.bm == 96)
        convFwdPaddedKernel<3, true><<<grid, dev::kBlock, 0, s>>>(p, gk);
      else
        convFwdPaddedKernel<2, true><<<grid, dev::kBlock, 0, s>>>(p, gk);
    } else if (pl.bm == 32) {
      convFwdPaddedKernel<0><<<grid, dev::kBlock, 0, s>>>(p, gk);
    } else if (pl.bm == 64) {
      convFwdPaddedKernel<1><<<grid, dev::kBlock, 0, s>>>(p, gk);
    } else if (pl.bm == 96) {
      convFwdPaddedKernel<3><<<grid, dev::kBlock, 0, s>>>(p, gk);
    } else {
      convFwdPaddedKernel<2><<<grid, dev::kBlock, 0, s>>>(p, gk);
    }
    THC_HIP_CHECK(hipGetLastError());
    if (pl.tail > 0) {
      fwdTailFixupKernel<<<dim3(pl.tail, BM * BN / (4 * dev::kBlock)), dev::kBlock, 0, s>>>(p, gk);
      THC_HIP_CHECK(hipGetLastError());
    }
    return;
  }
  p.tile0 = 0;
  p.nSplit = 1;
  p.ktPerSplit = launch::ceilDiv(gk.K, BK);
  if (pl.full > 0) {
    convFwdImplicitKernel<<<dim3(pl.full), dev::kBlock, 0, s>>>(p, gk);
    THC_HIP_CHECK(hipGetLastError());
  }
  if (pl.tail > 0) {
    p.tile0 = pl.full;
    p.ktPerSplit = pl.ktPerSplit;
    p.nSplit = pl.nSplit;
    p.partial = partial;
    convFwdImplicitKernel<<<dim3(pl.tail, pl.nSplit), dev::kBlock, 0, s>>>(p, gk);
    THC_HIP_CHECK(hipGetLastError());
    fwdTailFixupKernel<<<dim3(pl.tail, BM * BN / (4 * dev::kBlock)), dev::kBlock, 0, s>>>(p, gk);
    THC_HIP_CHECK(hipGetLastError());
  }
}

// out(nImages, M, L) = bias + W(M x K) * im2col(x); `scratch` holds plan.scratchFloats floats
// Where the output elements go when not into a dense (nImages, M, oH, oW) tensor.
struct OutMap {
  long outImg;
  int outRow, outSH, outSW;
  int dilate;  // FwdArgs::dilate
};

void launchFwdImplicit(hipStream_t s, const FwdPlan &pl, float *scratch, const float *w, const float *x, float *out,
                       const float *bias, int M, int nImages, const ConvGeom &g, bool relu = false,
                       const OutMap *om = nullptr, const FlipJob *flip = nullptr) {
  const bool fast = pl.tapEntries > 0;
  if (flip && !(fast && pl.paddedFloats > 0)) {  // no bordered copy to ride along with
    flipWeightKernel<<<launch::directGrid((long)flip->Cout * flip->Cin * flip->kH * flip->kW, dev::kBlock), dev::kBlock, 0, s>>>(
        flip->w, flip->wf, flip->Cout, flip->Cin, flip->kH, flip->kW);
    THC_HIP_CHECK(hipGetLastError());
    flip = nullptr;
  }
  if (fast && !(launch::aligned16(scratch) && (pl.weightFloats > 0 || launch::aligned16(w))))
    error("SpatialConvolutionMM: internal error, convolution scratch or weights not 16-byte aligned");
  float *partial = scratch + pl.tapEntries;
  ConvGeom gk = g;  // geometry the kernel sees
  FwdArgs p{};
  p.x = x;
  if (fast) {
    gk.H = g.H + 2 * g.padH, gk.W = g.W + 2 * g.padW, gk.padH = gk.padW = 0;
    float *xp = partial + partialFloats(pl);
    // 1x1 windows over a whole number of k-tiles: tap k is plane k of the image, no table needed
    const bool linear = g.kH == 1 && g.kW == 1 && g.K % BK == 0;
    if (pl.paddedFloats > 0) {  // the copy into the bordered layout builds the tap table on the side
      launchPadPlanes(s, x, xp, (long)nImages * g.Cin, g.H, g.W, g.padH, g.padW, linear ? nullptr : reinterpret_cast<int *>(scratch),
                      pl.tapEntries, &gk, flip);
      p.x = xp;
    }
    if (linear) {
      p.tapStride = gk.H * gk.W * (int)sizeof(float);
    } else if (pl.paddedFloats <= 0) {
      buildTapTableKernel<<<launch::directGrid(pl.tapEntries, dev::kBlock), dev::kBlock, 0, s>>>(
          reinterpret_cast<int *>(scratch), pl.tapEntries, gk);
      THC_HIP_CHECK(hipGetLastError());
    }
    if (pl.weightFloats > 0) {
      float *wp = xp + (pl.paddedFloats + 3) / 4 * 4;
      gk.K = (int)(pl.weightFloats / M);
      padRowsKernel<<<launch::directGrid(pl.weightFloats, dev::kBlock), dev::kBlock, 0, s>>>(w, wp, M, g.K, gk.K);
      THC_HIP_CHECK(hipGetLastError());
      w = wp;
    }
  }
  p.taps = reinterpret_cast<const int *>(scratch);
  p.w = w;
  p.out = out;
  p.bias = bias;
  p.relu = relu ? 1 : 0;
  p.M = M;
  p.Ncols = nImages * g.L;
  p.outImg = (long)M * g.L, p.outRow = g.L, p.outSH = g.oW, p.outSW = 1;
  if (om) p.outImg = om->outImg, p.outRow = om->outRow, p.outSH = om->outSH, p.outSW = om->outSW, p.dilate = om->dilate;
  if (fast) {
    const long span = ((long)(nImages - 1) * p.outImg + (long)(M - 1) * p.outRow + (long)(g.oH - 1) * p.outSH +
                       (long)(g.oW - 1) * p.outSW + 1 + (p.dilate ? p.outSH / 2 + 1 : 0)) * 4;
    p.outBytes = span < 0x7fffffffL ? (int)span : 0;
    // (the reciprocal division is exact while dividend * divisor < 2^32)
    p.magicL = (long)p.Ncols * g.L < 0xffffffffL ? dev::magicOf(g.L) : 0;
    p.magicOW = (long)g.L * g.oW < 0xffffffffL ? dev::magicOf(g.oW) : 0;
  }
  p.xBytes = (int)((long)nImages * gk.Cin * gk.H * gk.W * sizeof(float));
  p.wBytes = (int)((long)M * gk.K * sizeof(float));
  p.kReal = g.K;
  p.vecA = (gk.K % 4 == 0) && launch::aligned16(w);
  launchFwdKernels(s, pl, p, partial, gk, fast);
}

// Scratch of `floats` floats: the caller's buffer tensor (resized) or a stream-ordered temporary.
float *scratchFloats(THCState *state, THCudaTensor *buffer, long floats, Temp &tmp, const char *name) {
  if (floats <= 0) return nullptr;
  if (buffer) {
    resize(state, buffer, {floats});
    if (!isContiguous(erase(buffer))) error("%s tensor has to be contiguous", name);
    if (launch::aligned16(data(buffer))) return data(buffer);
    // a buffer tensor at an odd storage offset: its contents are unspecified anyway, work in a temporary
  }
  tmp = Temp(state->stream, (size_t)floats * sizeof(float));
  return (float *)tmp.get();
}

// Terms that one accumulator of a planned forward pass sums, the mean over the output.
double termsOf(const FwdPlan &pl, int K) {
  if (pl.direct) return K / 4;  // the four waves of a workgroup
  return ((double)pl.full * K + (double)pl.tail * std::min(K, pl.ktPerSplit * BK)) / std::max(1, pl.total);
}

// ---- pointwise forward -------------------------------------------------------------------------
// Launch shape of convPointwiseKernel for M rows: blocks of 32 rows per wave, waves along the rows. One workgroup of 8 waves
// per CU; a chunk of positions is 64 KB of x, two of them in LDS (32 -> 64 at 112 x 112, N = 64, 44.9 us). Outputs of 32 rows or
// fewer are left to the tiled GEMM, which measured faster.
struct PwShape {
  int mr, wr;
};
bool pwShape(int M, PwShape *sh) {
  if (M >= 256)
    *sh = {2, 4};  // 256 rows per workgroup
  else if (M > 64)
    *sh = {1, 4};  // 128 rows, two waves along the positions
  else if (M > 32)
    *sh = {1, 2};  // 64 rows, four waves along the positions
  else
    return false;
  return true;
}

template <int MR, int WR>
void launchPointwise(hipStream_t s, PwArgs p, int device, bool relu, bool transW) {
  constexpr int lds = kPwLdsFloats * (int)sizeof(float);
  const int form = transW ? 2 : relu ? 1 : 0;
  auto kernel = transW ? convPointwiseKernel<MR, WR, false, true>
                : relu ? convPointwiseKernel<MR, WR, true, false>
                       : convPointwiseKernel<MR, WR, false, false>;
  static std::atomic<bool> raised[3][64];  // once per kernel instance and device: allow more than 64 KB of dynamic LDS
  if (!raised[form][device].load()) {
    THC_HIP_CHECK(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    raised[form][device].store(true);
  }
  const int rowBlocks = launch::ceilDiv(p.M, 32 * MR * WR);
  // one workgroup per CU, shared between the row blocks; each streams a run of column tiles
  int slots = std::max(1, residentSlots(nullptr) / rowBlocks);
  if (g_switches.convPointwise > 1) slots = std::min(slots, g_switches.convPointwise);  // tests: long runs of tiles per workgroup
  p.tilesPerWg = launch::ceilDiv(p.nTiles, std::min(slots, p.nTiles));
  kernel<<<dim3(launch::ceilDiv(p.nTiles, p.tilesPerWg), rowBlocks), 64 * kPwWaves, lds, s>>>(p);
  THC_HIP_CHECK(hipGetLastError());
}

// out(N, M, L) = bias + W(M x K) x(N, K, L) on the weight-stationary kernel; false: the shape is not one of its.
// Whether the library may give the caller's buffer the size it needs.
bool growable(const THCudaTensor *buffer) {
  const Storage *s = buffer ? erase(buffer)->storage : nullptr;
  return buffer && (!s || ((s->flag & TH_STORAGE_RESIZABLE) && !s->allocator));
}
// Whether the buffer (null: a temporary) can have that many floats: a kernel that needs more scratch than the one it replaces
// is not a reason to refuse a fixed buffer, nor to allocate while a graph is being captured.
bool roomFor(THCState *state, const THCudaTensor *buffer, long floats) {
  if (!buffer || numel(erase(buffer)) >= floats) return true;
  if (!growable(buffer)) return false;
  const Storage *s = erase(buffer)->storage;
  return (s && s->size - erase(buffer)->storageOffset >= floats) || !capturing(state);
}

template <int K, int WR, int KW>
void launchPointwiseSplit(hipStream_t s, PwArgs p, bool relu, bool transW) {
  using S = PsShape<K, WR, KW>;
  auto kernel = transW ? convPointwiseSplitKernel<K, WR, KW, false, true>
                : relu ? convPointwiseSplitKernel<K, WR, KW, true, false>
                       : convPointwiseSplitKernel<K, WR, KW, false, false>;
  const int rowBlocks = launch::ceilDiv(p.M, S::ROWS);
  p.nTiles = launch::ceilDiv(p.P, S::TP);
  int slots = std::max(1, residentSlots((const void *)kernel) / rowBlocks);  // two or three workgroups a CU
  if (g_switches.convPointwise > 1) slots = std::min(slots, g_switches.convPointwise);  // tests: long runs of tiles per workgroup
  p.tilesPerWg = launch::ceilDiv(p.nTiles, std::min(slots, p.nTiles));
  kernel<<<dim3(launch::ceilDiv(p.nTiles, p.tilesPerWg), rowBlocks), dev::kBlock, 0, s>>>(p);
  THC_HIP_CHECK(hipGetLastError());
}

// transW: w holds (K x M) and its transpose is what multiplies (the gradInput pass hands over the layer's weights).
// scratchBuf: the buffer that the other kernels would take their scratch from (this one needs none).
bool convPointwise(THCState *state, const ConvGeom &g, const float *x, const float *w, const float *bias, float *out,
                   const THCudaTensor *scratchBuf, bool relu = false, bool transW = false) {
  if (forceGeneric() || g_switches.convPointwise == 0) return false;
  if (g.kH != 1 || g.kW != 1 || g.dH != 1 || g.dW != 1 || g.padH != 0 || g.padW != 0) return false;
  const long P = (long)g.N * g.L;
  PwShape sh;
  if (g.K != 32 && g.K != 64 && g.K != 128 && g.K != 256) return false;
  if (g.L % 4 != 0 || g.Cout % 8 != 0 || P < 32 || !pwShape(g.Cout, &sh)) return false;
  if ((long)g.Cout * g.K * 4 >= 0x7fffffffL) return false;
  // 256 planes: outputs of up to 128 rows, transposed up to 256 (every 64 rows read all of x again), and not where the other kernels
  // split K four ways or more, which is faster and more exact. us, those / this one: 256 -> 64 forward, 8 x 56 x 56 16.1 / 14.6;
  // 256 -> 512, 8 x 28 x 28 21.3 / 22.5; gradInput of 64 -> 256, 8 x 56 x 56 18.8 / 13.2, 32 x 56 x 56 39.6 / 36.4.
  if (g.K == 256 && (g.Cout > (transW ? 256 : 128) || termsOf(planFwdImplicit(g.Cout, g.N, g), g.K) < 128)) return false;
  // The shortest forward calls (an image or two of 14x14 and smaller planes) go to the direct kernel; those with the
  // transposed weights stay (direct needs a launch that transposes). us, this one / direct: 128 -> 256, 2 x 14 x 14 7.0 / 6.6.
  // So do wide outputs where direct splits short sums. 32 planes: the 256-row shape has a long start; up to 560 million
  // products the other kernels are better (32 -> 512, 31360 positions 25.6 / 21.2, gradInput 25.5 / 23.4; 37632: 25.6 / 26.5,
  // 25.5 / 29.1). (Calls whose buffer has a fixed size, or none, stay: they need no scratch here.)
  if (g_switches.convPointwise == 1 && g_switches.convDirect < 0 && growable(scratchBuf)) {
    if (!transW && P <= 512) return false;
    if (g.K == 32 && sh.mr == 2 && P >= 1024 && P * g.Cout * g.K < 560000000L) return false;
    if (g.K == 64 && sh.mr == 2 && P >= 1024 && termsOf(planFwdImplicit(g.Cout, g.N, g), g.K) < 64) return false;
  }
  if (!launch::aligned16(x) || !launch::aligned16(w) || !launch::aligned16(out)) return false;
  // 32-bit byte offsets into x and out; the reciprocal division of a position by L is exact while P * L < 2^32
  if (P * g.K * 4 >= 0x7fffffffL || P * g.Cout * 4 >= 0x7fffffffL || P * g.L >= 0xffffffffL) return false;
  int device = 0;
  THC_HIP_CHECK(hipGetDevice(&device));
  if (device < 0 || device >= 64) return false;
  PwArgs p{};
  p.w = w, p.x = x, p.out = out, p.bias = bias;
  p.M = g.Cout, p.L = g.L, p.P = (int)P;
  p.nTiles = (int)((P + 31) / 32);
  p.magicL = dev::magicOf(g.L);
  p.xBytes = (int)(P * g.K * 4), p.outBytes = (int)(P * g.Cout * 4);
  hipStream_t s = state->stream;
  auto split = [&](auto kc) {
    constexpr int KK = decltype(kc)::value;
    if (g.Cout <= 64)
      launchPointwiseSplit<KK, 2, 1>(s, p, relu, transW);
    else
      launchPointwiseSplit<KK, 4, 1>(s, p, relu, transW);
    return true;
  };
  if (g.K == 64) return split(std::integral_constant<int, 64>{});
  if (g.K == 128) return split(std::integral_constant<int, 128>{});
  if (g.K == 256) return launchPointwiseSplit<256, 2, 2>(s, p, relu, transW), true;
  if (sh.mr == 2)
    launchPointwise<2, 4>(s, p, device, relu, transW);
  else if (sh.wr == 4)
    launchPointwise<1, 4>(s, p, device, relu, transW);
  else
    launchPointwise<1, 2>(s, p, device, relu, transW);
  return true;
}

// ---- long convolutions on half-precision parts (conv_halves.h) ----------------------------------
// For the passes with sums long enough that these parts are no less exact than the kernels above and enough work to pay for
// the two launches that take the ranges of the operands and split them.
struct HalvesGemm {        // one GEMM: output positions nH x nW, its window, and where its elements go
  int nH, nW, dH, dW;
  SplitAxis h, v;
  long outOfs;
  int outSH, outSW;
};

// out(images, M, ...) = bias + the GEMMs of `gemm` over x(N, C, H, W); false: not a call for these kernels.
// oldTerms(): terms that one accumulator of the other kernels would sum (the mean over the output); asked last, it plans a pass.
template <class Terms>
bool convHalves(THCState *state, int N, int C, int H, int W, int M, const float *x, const float *w, int rs, int cs, int kW, long wFloats,
                const HalvesGemm *gemm, int count, Terms oldTerms, float *out, long outImg, int outRow, const float *bias,
                THCudaTensor *scratchBuf, const char *bufName, bool relu) {
  const int force = g_switches.convHalves;
  if (forceGeneric() || force == 0 || count < 1 || count > kMaxHalvesJobs || N < 1 || (force < 0 && C < 16)) return false;
  const int groups = launch::ceilDiv(C, kHalvesGroup);
  int lowH = 0, highH = H - 1, lowW = 0, highW = W - 1;  // rows and columns the windows touch
  long maxL = 1, minPositions = LONG_MAX;  // positions in steps of one
  double products = 0;
  long maxTaps = 0;
  for (int i = 0; i < count; ++i) {
    const HalvesGemm &G = gemm[i];
    const long taps = (long)G.h.n * G.v.n;
    if (taps < 1 || G.nH < 1 || G.nW < 1) return false;
    // items (group, tap) are taken apart by dev::fastDiv: exact while their number, with what fills the last stages, times taps < 2^32
    if (C * taps > (1 << 20) || (groups * taps + 8L * kStageItems) * taps >= 1L << 32) return false;
    maxTaps = std::max(maxTaps, taps);
    auto span = [](const SplitAxis &a, int n, int stride, int &low, int &high) {
      const int first = a.q0, last = a.q0 - (a.n - 1) * a.qStep;
      low = std::min(low, std::min(first, last)), high = std::max(high, (n - 1) * stride + std::max(first, last));
    };
    span(G.h, G.nH, G.dH, lowH, highH);
    span(G.v, G.nW, G.dW, lowW, highW);
    maxL = std::max(maxL, (long)G.nH * G.nW);
    minPositions = std::min(minPositions, (long)G.nH * G.nW * G.dH * G.dW);
    products += (double)N * G.nH * G.nW * M * C * taps;
  }
  const long Hp = (long)highH + 1 - lowH, Wp = (long)highW + 1 - lowW;
  const long imgBytes = Hp * Wp * groups * kHalvesGroup * 4, xImgBytes = (long)C * H * W * 4;
  if (imgBytes >= (1L << 30) || Hp * Wp * Wp >= 0xffffffffL || wFloats * 4 >= 0x7fffffffL || (long)C * H * W >= 0x7fffffffL) return false;
  // Fast enough: the products take about half the time (9 us less for 10^9 of them, on 98 layers of 100 at least 6; least with 2x2
  // windows and few output planes), the ranges and the split read the images twice and write them once (the bordered copy of the
  // other kernels, where there is a border, does a third of that less), the weights are read twice and written in both forms by
  // one workgroup a row, and there is a launch more. Of 15000 random passes the ones taken need 0.4 to 1.11 of the time of the other
  // kernels, one in a thousand more than all of it; with 7.5 us in the place of 6 the worst needed 1.28 (N = 5, 471 -> 44 2x2
  // on 75x85: 92 us on the others, 117 on these). E.g. (us, others / these) N = 64, 256 -> 256 3x3 on 28x28 332 / 199; left: N = 58,
  // 223 -> 54 3x3 stride 2 on 64x26 59 / 84; N = 9, 361 -> 156 7x7 on 26x9 70 / 76. 1x1 windows use every element once
  // (N = 32, 708 -> 272 on 26x62 163 / 187). Phases are not split along K: they have to fill the chip (gradInput, N = 14, 120 -> 311
  // 7x7 stride 2 on 26x42 106 / 142).
  const double moved = (double)N * C * H * W * (Hp * Wp != (long)H * W ? 4 : 12) + 48.0 * wFloats;
  if (force < 0 && (groups * kHalvesGroup * 4 > 5 * C || products * 6e-9 < 6.0 + moved / 6e6 || (count == 1 && maxTaps == 1))) return false;
  // Precise enough: the error of these kernels hardly grows with the number of terms (1.2e-7 of the result's norm at 600
  // terms, 1.3e-7 at 5000, 1.4e-7 at 10000), that of the other ones with the square root of those that one accumulator gets
  // and that are not zero (K split over workgroups or waves gives each fewer, and so does a border). With both operands half zeros,
  // as behind a ReLU, it is 1.04e-7 at 600 terms, 1.07e-7 at 700, 1.2e-7 at 850 and 1.4e-7 at 1500 (normal operands 1.3e-7 at
  // 560, 2.9e-7 at 2304). Over 7000 random passes, ordinary and masked, the error is at most 0.98 times that of the other kernels
  // (with K / 36 in the place of K / 24 1.015 times on 54 x 24 x 10, 426 -> 140 5x5); of 13 x 61 x 76, 76 -> 32 5x5, input masked, it is
  // 0.94 to 1.03 times by the seed, 0.97 in the middle.
  const double inside = std::min(1.0, (double)H * W / minPositions);  // share of a window's taps on the image, about
  if (force < 0 && (C * maxTaps * inside < 850 || oldTerms() * inside < 850 + C * maxTaps * inside / 24.0)) return false;
  if (N * maxL > 0x7fffffffL / 2 || N * std::max(imgBytes, xImgBytes) > (1L << 31) - 1 - 4096) return false;

  // scratch: ranges and forms of images and rows, items, split weights, split images, partial tiles
  long at = 0;
  auto take = [&](long bytes) {
    const long o = at;
    at += (bytes + 255) / 256 * 256;
    return o;
  };
  int bm = 0, bn = 0;
  FwdPlan pl[kMaxHalvesJobs];
  long partial[kMaxHalvesJobs], items[kMaxHalvesJobs], rowForm[kMaxHalvesJobs], split[kMaxHalvesJobs], split3[kMaxHalvesJobs];
  int itemsPad[kMaxHalvesJobs], rows = 0;
  const int chunks = launch::ceilDiv((int)(Hp * Wp), kSplitRun * dev::kBlock);
  // slices of an image that rangesKernel reads, a power of two: enough workgroups to fill the chip, at least 4096 floats each
  const long perImg = (long)C * H * W;
  int nSlots = 1;
  while (nSlots < kMaxSlots && 2 * nSlots <= perImg / 4096 && nSlots < launch::ceilDiv(2048, N)) nSlots *= 2;
  const long slots = take((long)N * nSlots * sizeof(uint2)), imgForm = take((long)N * 4), rowRanges = take(M * (long)sizeof(uint2));
  long minL = LONG_MAX;
  for (int i = 0; i < count; ++i) {
    const HalvesGemm &G = gemm[i];
    itemsPad[i] = launch::roundUp(groups * G.h.n * G.v.n, kStageItems);
    pl[i] = FwdPlan{};
    planTiles(pl[i], M, (long)N * G.nH * G.nW, itemsPad[i] / kStageItems, true, 5.0, false);
    bm = pl[i].bm, bn = pl[i].bn;
    rows = launch::roundUp(M, bm);
    const long splitBytes = (long)rows * itemsPad[i] * 32;
    if (splitBytes / 2 * 3 >= 0x7fffffffL) return false;
    items[i] = take(2 * (itemsPad[i] + 4 * kStageItems) * 4L), rowForm[i] = take(rows * 4L);
    split[i] = take(splitBytes), split3[i] = take(splitBytes / 2 * 3);
    minL = std::min(minL, (long)G.nH * G.nW);
  }
  const int reach = (int)((bn - 2) / minL) + 1;  // images of a tile lie at most that far from each other
  if ((reach + 1) * (imgBytes / 2 * 3) >= 0x7fffffffL) return false;
  const long images = take(N * imgBytes), images3 = take(N * (imgBytes / 2 * 3));
  // several GEMMs (phases) in one launch: their tiles fill each other's last rounds, no tile is split
  if (count > 1) {
    int total = 0;
    for (int i = 0; i < count; ++i) {
      pl[i].tail = 0, pl[i].full = pl[i].total, pl[i].nSplit = 1, pl[i].ktPerSplit = itemsPad[i] / kStageItems;
      total += pl[i].total;
    }
    if (force < 0 && total < residentSlots(nullptr)) return false;
  }
  for (int i = 0; i < count; ++i) partial[i] = take(partialFloats(pl[i]) * 4);
  if (!roomFor(state, scratchBuf, at / 4)) return false;

  Temp tmp;
  char *buf = reinterpret_cast<char *>(scratchFloats(state, scratchBuf, at / 4, tmp, bufName));
  hipStream_t s = state->stream;
  RangeArgs ra{};
  ra.x = x, ra.slots = (uint2 *)(buf + slots), ra.perImg = perImg, ra.perSlice = (int)((perImg + nSlots - 1) / nSlots + 3) / 4 * 4;
  ra.nSlots = nSlots, ra.vec = perImg % 4 == 0 && launch::aligned16(x);
  ra.w = w, ra.rows = (uint2 *)(buf + rowRanges), ra.M = M, ra.rs = rs, ra.cs = cs, ra.C = C, ra.taps = std::min(rs, cs);
  rangesKernel<<<(unsigned)(M + N * nSlots), dev::kBlock, 0, s>>>(ra);
  THC_HIP_CHECK(hipGetLastError());
  SplitJobs J{};
  SplitImages &I = J.im;
  I.x = x, I.dst = (u32x4 *)(buf + images), I.dst3 = (u32x4 *)(buf + images3), I.slots = (uint2 *)(buf + slots);
  I.forms = (int *)(buf + imgForm);
  I.nSlots = nSlots, I.N = N, I.C = C, I.H = H, I.W = W, I.top = -lowH, I.left = -lowW, I.Hp = (int)Hp, I.Wp = (int)Wp;
  I.groups = groups, I.chunks = chunks, I.reach = reach, I.blocks = N * groups * chunks, I.magicW = dev::magicOf((int)Wp);
  J.count = count;
  long blocks = I.blocks;
  HalvesBatch<kMaxHalvesJobs> batch{};
  FwdBatch foldBatch{};
  int wholeTotal = 0, splitTotal = 0, maxTail = 0;
  for (int i = 0; i < count; ++i) {
    const HalvesGemm &G = gemm[i];
    SplitRows &R = J.rows[i];
    R.w = w, R.dst = (u32x4 *)(buf + split[i]), R.dst3 = (u32x4 *)(buf + split3[i]);
    R.ranges = (uint2 *)(buf + rowRanges), R.forms = (int *)(buf + rowForm[i]);
    R.items = (int *)(buf + items[i]), R.items3 = R.items + itemsPad[i] + 4 * kStageItems;
    R.rs = rs, R.cs = cs, R.kW = kW, R.M = M, R.rows = rows, R.C = C, R.tileRows = bm, R.itemsPad = itemsPad[i];
    R.h = G.h, R.v = G.v;
    blocks += rows + 1;
    HalvesItem &it = batch.item[i];
    HalvesArgs &q = it.q;
    q.a = R.dst, q.b = I.dst, q.a3 = R.dst3, q.b3 = I.dst3, q.items = R.items, q.items3 = R.items3;
    q.rowForm = R.forms, q.imgForm = I.forms, q.imgBytes = imgBytes, q.planeBytes = (int)(Hp * Wp * 16);
    q.nItems = groups * G.h.n * G.v.n, q.itemsPad = itemsPad[i];
    q.w = w, q.x = x, q.wBytes = (int)(wFloats * 4), q.xBytes = (int)(N * xImgBytes);
    q.rs = rs, q.cs = cs, q.kW = kW, q.C = C, q.H = H, q.W = W, q.h = G.h, q.v = G.v;
    q.magicT = dev::magicOf(G.h.n * G.v.n), q.magicV = dev::magicOf(G.v.n);
    ConvGeom &gk = it.g;
    gk.N = N, gk.Cin = C, gk.Cout = M, gk.H = (int)Hp, gk.W = (int)Wp, gk.oH = G.nH, gk.oW = G.nW;
    gk.kH = G.h.n, gk.kW = G.v.n, gk.dH = G.dH, gk.dW = G.dW, gk.dilH = gk.dilW = 1;
    gk.K = itemsPad[i] * kHalvesGroup, gk.L = G.nH * G.nW;
    FwdArgs &a = it.p;
    a.bias = bias, a.relu = relu ? 1 : 0;
    a.M = M, a.Ncols = N * gk.L;
    a.out = out + G.outOfs;
    a.outImg = outImg, a.outRow = outRow, a.outSH = G.outSH, a.outSW = G.outSW;
    const long spanBytes = ((long)(N - 1) * outImg + (long)(M - 1) * outRow + (long)(G.nH - 1) * G.outSH + (long)(G.nW - 1) * G.outSW + 1) * 4;
    a.outBytes = spanBytes < 0x7fffffffL ? (int)spanBytes : 0;
    a.magicL = (long)a.Ncols * gk.L < 0xffffffffL ? dev::magicOf(gk.L) : 0;
    a.magicOW = (long)gk.L * gk.oW < 0xffffffffL ? dev::magicOf(gk.oW) : 0;
    a.mTiles = pl[i].mTiles, a.bm = bm, a.bn = bn;
    a.full = pl[i].full, a.tail = pl[i].tail, a.tile0 = pl[i].full;
    a.nSplit = a.tail > 0 ? pl[i].nSplit : 1;
    a.ktPerSplit = a.tail > 0 ? pl[i].ktPerSplit : itemsPad[i] / kStageItems;
    a.partial = (float *)(buf + partial[i]);
    wholeTotal += a.full, splitTotal += a.tail * a.nSplit;
    it.wholeEnd = wholeTotal, it.splitEnd = splitTotal;
    maxTail = std::max(maxTail, a.tail);
    foldBatch.item[i].p = a, foldBatch.item[i].g = gk;
  }
  batch.count = foldBatch.count = count, batch.wholeTotal = wholeTotal;
  splitOperandsKernel<<<(unsigned)blocks, dev::kBlock, 0, s>>>(J);
  THC_HIP_CHECK(hipGetLastError());
  const dim3 grid(wholeTotal + splitTotal);
  auto launchShape = [&](auto wr, auto wc, auto ti, auto tj) {
    constexpr int A = decltype(wr)::value, B = decltype(wc)::value, I2 = decltype(ti)::value, J2 = decltype(tj)::value;
    if (count == 1) {
      HalvesBatch<1> one{};
      one.item[0] = batch.item[0], one.count = 1, one.wholeTotal = wholeTotal;
      convHalvesKernel<1, A, B, I2, J2><<<grid, dev::kBlock, 0, s>>>(one);
    } else {
      convHalvesKernel<kMaxHalvesJobs, A, B, I2, J2><<<grid, dev::kBlock, 0, s>>>(batch);
    }
  };
  using N1 = std::integral_constant<int, 1>;
  using N2 = std::integral_constant<int, 2>;
  using N3 = std::integral_constant<int, 3>;
  using N4 = std::integral_constant<int, 4>;
  if (bm == 32)
    launchShape(N1{}, N4{}, N1{}, N2{});
  else if (bm == 64)
    launchShape(N1{}, N4{}, N2{}, N1{});
  else if (bm == 96)
    launchShape(N1{}, N4{}, N3{}, N1{});
  else
    launchShape(N2{}, N2{}, N2{}, N2{});
  THC_HIP_CHECK(hipGetLastError());
  if (maxTail > 0) {
    fwdTailFixupBatchKernel<<<dim3(maxTail, BM * BN / (4 * dev::kBlock), count), dev::kBlock, 0, s>>>(foldBatch);
    THC_HIP_CHECK(hipGetLastError());
  }
  return true;
}

bool convHalvesForward(THCState *state, const ConvGeom &g, const float *x, const float *w, const float *bias, float *out,
                       THCudaTensor *scratchBuf, const char *bufName, bool relu) {
  HalvesGemm G{};
  G.nH = g.oH, G.nW = g.oW, G.dH = g.dH, G.dW = g.dW;
  G.h = SplitAxis{g.kH, 0, 1, -g.padH, -g.dilH}, G.v = SplitAxis{g.kW, 0, 1, -g.padW, -g.dilW};
  G.outSH = g.oW, G.outSW = 1;
  if ((long)g.Cout * g.K >= 0x7fffffffL / 4) return false;
  return convHalves(state, g.N, g.Cin, g.H, g.W, g.Cout, x, w, g.K, g.kH * g.kW, g.kW, (long)g.Cout * g.K, &G, 1,
                    [&] { return termsOf(planFwdImplicit(g.Cout, g.N, g), g.K); }, out, (long)g.Cout * g.L,
                    g.L, bias, scratchBuf, bufName, relu);
}

// ---- the three passes on raw device pointers -------------------------------------------------
// `scratchBuf` is the caller's buffer tensor (columns / gradColumns) or null; its contents are
// unspecified afterwards.

// out(N, Cout, oH, oW) = bias + conv(x(N, Cin, H, W), w(Cout, K))
// relu: out = Threshold(0, 0) of that, applied as the values are stored
void convForward(THCState *state, const ConvGeom &g, const float *x, const float *w, const float *bias, float *out,
                 THCudaTensor *scratchBuf, const char *bufName, bool relu = false) {
  if ((long)g.N * g.Cout == 0) return;
  if (convPointwise(state, g, x, w, bias, out, scratchBuf, relu)) return;
  if (convHalvesForward(state, g, x, w, bias, out, scratchBuf, bufName, relu)) return;
  hipStream_t s = state->stream;
  // images per launch so that the flat column index n*L + l fits an int
  int group = (int)std::min<long>(g.N, std::max<long>(1, 0x7fffffffL / 2 / g.L));
  const long imgBytes = (long)g.Cin * (g.H + 2 * g.padH) * (g.W + 2 * g.padW) * sizeof(float);  // with its zero border
  const bool implicit2 = !forceGeneric() && imgBytes < (1L << 30);
  if (implicit2) group = (int)std::min<long>(group, std::max<long>(1, ((1L << 31) - 1 - 4096) / imgBytes));
  if (implicit2) {
    FwdPlan pl = planFwdImplicit(g.Cout, std::min(group, g.N), g, launch::aligned16(w));
    long need = pl.scratchFloats;  // the last, smaller group may split differently
    if (g.N % group != 0) need = std::max(need, planFwdImplicit(g.Cout, g.N % group, g, launch::aligned16(w)).scratchFloats);
    Temp tmp;
    float *scratch = scratchFloats(state, scratchBuf, need, tmp, bufName);
    for (int n0 = 0; n0 < g.N; n0 += group) {
      int cnt = std::min(group, g.N - n0);
      if (cnt != std::min(group, g.N)) pl = planFwdImplicit(g.Cout, cnt, g, launch::aligned16(w));
      launchFwdImplicit(s, pl, scratch, w, x + (long)n0 * g.Cin * g.H * g.W, out + (long)n0 * g.Cout * g.L, bias, g.Cout,
                        cnt, g, relu);
    }
    return;
  }
  for (int n0 = 0; n0 < g.N; n0 += group) {
    int cnt = std::min(group, g.N - n0);
    GemmArgs p{};
    p.a = w;
    p.b = x;
    p.c = out;
    p.bias = bias;
    p.M = g.Cout;
    p.Ncols = cnt * g.L;
    p.R = g.K;
    p.n0 = n0;
    p.nImages = cnt;
    p.mTiles = (int)tiles(p.M, BM);
    p.vecA = (g.K % 4 == 0) && launch::aligned16(p.a);
    dim3 grid(p.mTiles * tiles(p.Ncols, BN), 1);
    convGemmKernel<kForward><<<grid, dev::kBlock, 0, s>>>(p, g);
    THC_HIP_CHECK(hipGetLastError());
  }
  if (relu) reluInPlace(s, out, (long)g.N * g.Cout * g.L);  // the first-generation kernel has no such epilogue
}

// Taps and gy indices of phase ph along one axis (see PhaseAxis).
PhaseAxis phaseAxis(int ph, int size, int pad, int k, int dil, int stride) {
  PhaseAxis a{};
  a.n = ph < size ? (size - ph + stride - 1) / stride : 0;
  const int d = std::gcd(dil, stride);
  a.kStep = stride / d, a.qStep = dil / d;
  for (int kk = 0; kk < std::min(k, a.kStep); ++kk) {  // kk * dil = ph + pad (mod stride) has period stride / d in kk
    const int v = ph + pad - kk * dil;
    if (((v % stride) + stride) % stride == 0) {
      a.k0 = kk, a.nk = (k - 1 - kk) / a.kStep + 1, a.q0 = v / stride;
      break;
    }
  }
  return a;
}

// gi by phases of the stride (one phase at stride 1) on the same kernels
bool convHalvesGradInput(THCState *state, const ConvGeom &g, const float *gy, const float *w, float *gi, THCudaTensor *scratchBuf,
                         const char *bufName, const float *bias) {
  if ((long)g.dH * g.dW > kMaxHalvesJobs || (long)g.Cout * g.K >= 0x7fffffffL / 4) return false;
  HalvesGemm G[kMaxHalvesJobs] = {};
  int count = 0;
  for (int ph = 0; ph < g.dH; ++ph)
    for (int pw = 0; pw < g.dW; ++pw) {
      const PhaseAxis h = phaseAxis(ph, g.H, g.padH, g.kH, g.dilH, g.dH), v = phaseAxis(pw, g.W, g.padW, g.kW, g.dilW, g.dW);
      if (h.n == 0 || v.n == 0) continue;
      HalvesGemm &q = G[count++];
      q.nH = h.n, q.nW = v.n, q.dH = q.dW = 1;
      q.h = SplitAxis{h.nk, h.k0, h.kStep, h.q0, h.qStep}, q.v = SplitAxis{v.nk, v.k0, v.kStep, v.q0, v.qStep};
      q.outOfs = (long)ph * g.W + pw, q.outSH = g.dH * g.W, q.outSW = g.dW;
    }
  // the terms of an accumulator of the other route: of the forward kernels at stride 1, else of the phases, which are split
  // so that every workgroup gets about the same number of k-tiles
  auto oldTerms = [&]() {
    if (g.dH == 1 && g.dW == 1) {
      ConvGeom t = g;
      t.Cin = g.Cout, t.Cout = g.Cin, t.H = g.oH, t.W = g.oW, t.oH = g.H, t.oW = g.W;
      t.padH = t.padW = 0, t.K = g.Cout * g.kH * g.kW, t.L = g.H * g.W;
      return termsOf(planFwdImplicit(t.Cout, t.N, t), t.K);
    }
    int bm, bn;
    tileShape(g.Cin, true, LONG_MAX, LONG_MAX, bm, bn);
    long units = 0;
    for (int i = 0; i < count; ++i)
      units += (long)tiles(g.Cin, bm) * tiles((long)g.N * G[i].nH * G[i].nW, bn) * launch::ceilDiv(g.Cout * G[i].h.n * G[i].v.n, BK);
    const long target = std::max<long>(4, units / (2L * residentSlots(nullptr)));
    double terms = 0, positions = 0;
    for (int i = 0; i < count; ++i) {
      const int nkt = launch::ceilDiv(g.Cout * G[i].h.n * G[i].v.n, BK);
      const long parts = std::max<long>(1, std::min<long>(nkt / 4, (nkt + target / 2) / target));
      terms += (double)G[i].nH * G[i].nW * nkt * BK / parts, positions += (double)G[i].nH * G[i].nW;
    }
    return terms / std::max(1.0, positions);
  };
  // heaviest phase first: its workgroups are dispatched first
  std::stable_sort(G, G + count, [](const HalvesGemm &a, const HalvesGemm &b) { return a.h.n * a.v.n > b.h.n * b.v.n; });
  return convHalves(state, g.N, g.Cout, g.oH, g.oW, g.Cin, gy, w, g.kH * g.kW, g.K, g.kW, (long)g.Cout * g.K, G, count, oldTerms, gi,
                    (long)g.Cin * g.H * g.W, g.H * g.W, bias, scratchBuf, bufName, false);
}

// gradInput (and the transposed convolution's forward pass) for any stride, padding and dilation:
// per phase of gi a stride-1 convolution of the zero-bordered gradOutput with the phase's sub-kernel,
// on the forward kernels. No gradient columns reach memory and no multiply is spent on the zeros a
// strided convolution's transpose is full of. Returns false when the geometry is outside the 32-bit
// offsets of those kernels (the caller then takes the column path).
bool gradInputByPhase(THCState *state, const ConvGeom &g, const float *gy, const float *w, float *gi,
                      THCudaTensor *scratchBuf, const char *bufName, const float *bias) {
  if ((long)g.dH * g.dW > kMaxPhases) return false;
  hipStream_t s = state->stream;
  PhaseSet set{};
  int lowH = 0, highH = g.oH - 1, lowW = 0, highW = g.oW - 1;  // gy rows / columns the phases touch
  long wTotal = 0, tapTotal = 0, maxL = 1;
  for (int ph = 0; ph < g.dH; ++ph)
    for (int pw = 0; pw < g.dW; ++pw) {
      Phase P{};
      P.h = phaseAxis(ph, g.H, g.padH, g.kH, g.dilH, g.dH);
      P.w = phaseAxis(pw, g.W, g.padW, g.kW, g.dilW, g.dW);
      if (P.h.n == 0 || P.w.n == 0) continue;
      P.h0 = ph, P.w0 = pw;
      const long K = (long)g.Cout * P.h.nk * P.w.nk;
      if (K >= 0x7fffffffL / 8) return false;
      P.K = (int)K;
      P.Kp = std::max(BK, launch::ceilDiv(P.K, BK) * BK);
      if (P.K > 0) {
        lowH = std::min(lowH, P.h.q0 - (P.h.nk - 1) * P.h.qStep), highH = std::max(highH, P.h.n - 1 + P.h.q0);
        lowW = std::min(lowW, P.w.q0 - (P.w.nk - 1) * P.w.qStep), highW = std::max(highW, P.w.n - 1 + P.w.q0);
      }
      maxL = std::max(maxL, (long)P.h.n * P.w.n);
      set.ph[set.count++] = P;
    }
  if (set.count == 0) return true;  // gi has no elements
  // heaviest phase first: its workgroups are dispatched first
  std::stable_sort(set.ph, set.ph + set.count, [](const Phase &a, const Phase &b) { return a.Kp > b.Kp; });
  for (int i = 0; i < set.count; ++i) {
    Phase &P = set.ph[i];
    P.tapOfs = (int)tapTotal, tapTotal += P.Kp + 2 * BK;
    P.wOfs = wTotal, wTotal += (long)g.Cin * P.Kp;
  }
  const int top = -lowH, left = -lowW;
  const long Hp = (long)highH + 1 + top, Wp = (long)highW + 1 + left;
  const long imgFloats = (long)g.Cout * Hp * Wp;
  if (imgFloats * 4 >= (1L << 30) || wTotal * 4 >= 0x7fffffffL || tapTotal >= 0x7fffffffL / 8 ||
      launch::ceilDiv(Hp * Wp, (long)dev::kBlock) > 65535)
    return false;
  const bool copy = top > 0 || left > 0 || Hp != g.oH || Wp != g.oW || !launch::aligned16(gy);
  int group = (int)std::min<long>(g.N, std::max<long>(1, 0x7fffffffL / 2 / maxL));
  group = (int)std::min<long>(group, std::max<long>(1, ((1L << 31) - 1 - 4096) / (imgFloats * 4)));

  // All phases of a group of images run as one batched launch. The phases differ in K; the heavier ones are
  // split along K so that a workgroup reduces about the same number of k-tiles whatever its phase and the
  // grid holds about two workgroups per CU. Split phases leave partial tiles for the batched fold.
  int bm, bn;
  long tiles64 = 0, kTiles64 = 0;  // (up to 32 rows: the splits below make up for few tiles better than 64-row tiles do, so those
  for (int i = 0; i < set.count && g.Cin > 32; ++i) {  // never count as a short call: 192 -> 8 4x4 stride 4, N = 33: 20.6 against 26.3 us)
    const long t = tiles(g.Cin, 64) * (long)tiles((long)std::min(group, g.N) * set.ph[i].h.n * set.ph[i].w.n, 128);
    tiles64 += t, kTiles64 += t * (set.ph[i].Kp / BK);
  }
  tileShape(g.Cin, true, tiles64, g.Cin > 32 ? kTiles64 : LONG_MAX, bm, bn);
  const int mTiles = (int)tiles(g.Cin, bm);
  struct Split {
    int tiles, tail, nSplit, ktPerSplit;  // the last `tail` of the item's tiles are split nSplit ways
    long partialOfs;
  } split[kMaxPhases];
  long partialTotal = 0;
  auto planAll = [&](int cnt) {
    const int cus = residentSlots(nullptr);
    long units = 0, wgs = 0;
    for (int i = 0; i < set.count; ++i) {
      const Phase &P = set.ph[i];
      split[i].tiles = mTiles * (int)tiles((long)cnt * P.h.n * P.w.n, bn);
      units += (long)split[i].tiles * (P.Kp / BK);
    }
    const long target = std::max<long>(4, units / (2L * cus));  // k-tiles per workgroup
    bool anySplit = false;
    for (int i = 0; i < set.count; ++i) {
      const int nkt = set.ph[i].Kp / BK;
      const int n = (int)std::max<long>(1, std::min<long>(nkt / 4, (nkt + target / 2) / target));
      split[i].ktPerSplit = launch::ceilDiv(nkt, n);
      split[i].nSplit = launch::ceilDiv(nkt, split[i].ktPerSplit);
      split[i].tail = split[i].nSplit > 1 ? split[i].tiles : 0;
      anySplit = anySplit || split[i].nSplit > 1;
      wgs += split[i].tiles;
    }
    // No phase is heavy enough to be split by that rule, and the whole tiles fill the CUs once or more with a
    // partial round left over (4 equal phases of a 4x4 stride-2 layer: 392 tiles on 256 CUs): the tiles of that
    // last round - the end of the launch order - are split along K like the tail of a single forward pass
    // (planTiles: same cost model, the k-tiles of the heaviest phase in the tail), where that pays for the fold: its
    // stores are every other float of a row, 17 us for 408 partial tiles. (256 -> 128 4x4 stride 2 on 14x14, N = 64,
    // forward + backward: 336 us with the last round split three ways, 328 with whole tiles, two to a CU.)
    const int q = (int)(wgs / cus), r = (int)(wgs % cus);
    if (!anySplit && q > 0 && r > 0) {
      int first = set.count - 1;  // first item with tiles in the tail
      for (int left = r; first > 0 && left > split[first].tiles; --first) left -= split[first].tiles;
      const int nktTail = set.ph[first].Kp / BK, nktHead = set.ph[0].Kp / BK;
      auto perWg = [&](int nkt, int S) { return (double)launch::ceilDiv(nkt, S) + 4.0; };
      double best = 0.95 * (q + 1) * perWg(nktHead, 1);
      int S = 1;
      for (int c = 2; c <= std::max(1, std::min(nktTail / 4, 16)); ++c) {
        if (launch::ceilDiv(nktTail, launch::ceilDiv(nktTail, c)) != c) continue;
        const double t = q * perWg(nktHead, 1) + launch::ceilDiv(r * c, cus) * perWg(nktTail, c) + 0.05 * r * c;
        if (t < best) best = t, S = c;
      }
      if (S > 1) {
        int left = r;
        for (int i = set.count - 1; i >= 0 && left > 0; --i) {
          const int nkt = set.ph[i].Kp / BK;
          split[i].tail = std::min(left, split[i].tiles);
          left -= split[i].tail;
          split[i].ktPerSplit = launch::ceilDiv(nkt, std::min(S, std::max(1, nkt / 4)));
          split[i].nSplit = launch::ceilDiv(nkt, split[i].ktPerSplit);
          if (split[i].nSplit <= 1) split[i].tail = 0;
        }
      }
    }
    long total = 0;
    for (int i = 0; i < set.count; ++i) {
      split[i].partialOfs = total;
      total += (long)split[i].tail * split[i].nSplit * BM * BN;
    }
    partialTotal = std::max(partialTotal, total);
  };
  if (g.N % group != 0) planAll(g.N % group);  // the last, smaller group may split differently
  planAll(std::min(group, g.N));
  const long paddedFloats = copy ? (group * imgFloats + 3) / 4 * 4 : 0;
  Temp tmp;
  float *buf = scratchFloats(state, scratchBuf, tapTotal + wTotal + partialTotal + paddedFloats, tmp, bufName);
  int *taps = reinterpret_cast<int *>(buf);
  float *wph = buf + tapTotal;
  float *partial = wph + wTotal;
  float *gyp = partial + partialTotal;
  int maxKp = 0;
  for (int i = 0; i < set.count; ++i) maxKp = std::max(maxKp, set.ph[i].Kp);
  if (g.Cin + 1 > 65535) return false;
  const int chunks = std::max(1, std::min(8, launch::ceilDiv(maxKp + 2 * BK, 4 * dev::kBlock)));
  // the set-up rides along with the first group's bordered copy when that copy has the flat 16-byte form
  const long plane = Hp * Wp, firstTotal4 = (long)std::min(group, g.N) * g.Cout * (plane / 4);
  const long setupBlocks = (long)chunks * (g.Cin + 1) * set.count;
  const bool together = copy && plane % 4 == 0 && plane < 4096 && launch::aligned16(gyp) &&
                        firstTotal4 * (plane / 4) < 0xffffffffL && setupBlocks < (1L << 24);
  if (!together) {
    phaseSetupKernel<<<dim3(chunks, g.Cin + 1, set.count), dev::kBlock, 0, s>>>(w, wph, taps, set, g.Cin, g.kH, g.kW, (int)Hp,
                                                                              (int)Wp, top, left);
    THC_HIP_CHECK(hipGetLastError());
  }
  for (int n0 = 0; n0 < g.N; n0 += group) {
    const int cnt = std::min(group, g.N - n0);
    if (cnt != std::min(group, g.N)) planAll(cnt);
    const float *src = gy + (long)n0 * g.Cout * g.L;
    if (copy && together && n0 == 0) {
      const int copyBlocks = (int)std::min<long>((firstTotal4 + dev::kBlock - 1) / dev::kBlock, 16384);
      padPlanesPhaseSetupKernel<<<(unsigned)(copyBlocks + setupBlocks), dev::kBlock, 0, s>>>(
          src, gyp, g.oH, g.oW, (int)Hp, (int)Wp, top, left, firstTotal4, copyBlocks, w, wph, taps, set, g.Cin, g.kH, g.kW, chunks);
      THC_HIP_CHECK(hipGetLastError());
      src = gyp;
    } else if (copy) {
      launchPadPlanes(s, src, gyp, (long)cnt * g.Cout, g.oH, g.oW, top, left, (int)Hp, (int)Wp);
      src = gyp;
    }
    FwdBatch batch{};
    batch.count = set.count;
    int maxTail = 0, wholeTotal = 0, splitTotal = 0;
    for (int i = 0; i < set.count; ++i) {
      const Phase &P = set.ph[i];
      FwdBatchItem &it = batch.item[i];
      ConvGeom &gk = it.g;  // what the forward kernel sees: a stride-1 pass over the bordered gy
      gk.N = cnt, gk.Cin = g.Cout, gk.Cout = g.Cin;
      gk.H = (int)Hp, gk.W = (int)Wp, gk.oH = P.h.n, gk.oW = P.w.n;
      gk.kH = gk.kW = gk.dH = gk.dW = gk.dilH = gk.dilW = 1;
      gk.K = P.Kp, gk.L = P.h.n * P.w.n;
      FwdArgs &a = it.p;
      a.w = wph + P.wOfs;
      a.x = src;
      a.taps = taps + P.tapOfs;
      a.bias = bias;
      a.M = g.Cin;
      a.Ncols = cnt * gk.L;
      a.out = gi + (long)n0 * g.Cin * g.H * g.W + (long)P.h0 * g.W + P.w0;
      a.outImg = (long)g.Cin * g.H * g.W, a.outRow = g.H * g.W, a.outSH = g.dH * g.W, a.outSW = g.dW;
      {
        const long span = ((long)(cnt - 1) * a.outImg + (long)(g.Cin - 1) * a.outRow + (long)(P.h.n - 1) * a.outSH +
                           (long)(P.w.n - 1) * a.outSW + 1) * 4;
        a.outBytes = span < 0x7fffffffL ? (int)span : 0;
        a.magicL = (long)a.Ncols * gk.L < 0xffffffffL ? dev::magicOf(gk.L) : 0;
        a.magicOW = (long)gk.L * gk.oW < 0xffffffffL ? dev::magicOf(gk.oW) : 0;
      }
      a.xBytes = (int)(cnt * imgFloats * 4);
      a.wBytes = (int)((long)g.Cin * P.Kp * 4);
      a.kReal = P.K;
      a.vecA = true;
      a.mTiles = mTiles, a.bm = bm, a.bn = bn;
      a.tail = split[i].tail, a.full = split[i].tiles - split[i].tail;
      a.tile0 = a.full;
      a.nSplit = a.tail > 0 ? split[i].nSplit : 1;
      a.ktPerSplit = a.tail > 0 ? split[i].ktPerSplit : P.Kp / BK;
      a.partial = partial + split[i].partialOfs;
      wholeTotal += a.full, splitTotal += a.tail * a.nSplit;
      it.wholeEnd = wholeTotal, it.splitEnd = splitTotal;
      maxTail = std::max(maxTail, a.tail);
    }
    batch.wholeTotal = wholeTotal;
    const dim3 grid(wholeTotal + splitTotal);
    if (bm == 32)
      convFwdPaddedBatchKernel<0><<<grid, dev::kBlock, 0, s>>>(batch);
    else if (bm == 64)
      convFwdPaddedBatchKernel<1><<<grid, dev::kBlock, 0, s>>>(batch);
    else if (bm == 96)
      convFwdPaddedBatchKernel<3><<<grid, dev::kBlock, 0, s>>>(batch);
    else
      convFwdPaddedBatchKernel<2><<<grid, dev::kBlock, 0, s>>>(batch);
    THC_HIP_CHECK(hipGetLastError());
    if (maxTail > 0) {
      fwdTailFixupBatchKernel<<<dim3(maxTail, BM * BN / (4 * dev::kBlock), set.count), dev::kBlock, 0, s>>>(batch);
      THC_HIP_CHECK(hipGetLastError());
    }
  }
  return true;
}

// ---- gradInput with one to four input planes (conv_fewplanes.h) ----
template <int S, int T, int KC, int PADC>
void launchFewPlanes(hipStream_t s, FpArgs a, const FpTaps &tp, const ConvGeom &g) {
  using Sh = FpShape<S, T, KC, PADC>;
  const int PR = (g.H + S - 1) / S, PC = (g.W + S - 1) / S;  // phase positions per image
  a.tilesR = (int)tiles(PR, 4 * T), a.tilesC = (int)tiles(PC, 16);
  a.magicTiles = dev::magicOf(a.tilesR * a.tilesC), a.magicTilesC = dev::magicOf(a.tilesC);
  const int RR = Sh::CT ? Sh::RR : a.RR;
  const int KKP = (g.kH * g.kW + 3) / 4 * 4;
  convFewPlanesGradInputKernel<S, T, KC, PADC>
      <<<g.N * a.tilesR * a.tilesC, 64 * kFpWaves, Sh::ldsBytes(RR, KKP), s>>>(a, tp);
  THC_HIP_CHECK(hipGetLastError());
}

// false: not a shape for this kernel (the caller goes on to the other routes)
bool convFewPlanesGradInput(THCState *state, const ConvGeom &g, const float *gy, const float *w, float *gi,
                            const float *bias, bool runtimeOnly) {
  const int S = g.dH;
  if (g.Cin > 4 || g.dilH != 1 || g.dilW != 1 || g.dH != g.dW || S > 4 || g.padH < 0 || g.padW < 0) return false;
  if ((long)g.Cout * g.L * 4 >= (1L << 31) || (long)g.Cin * g.H * g.W * 4 >= (1L << 31) || (long)g.Cout * g.K * 4 >= (1L << 31))
    return false;
  FpArgs a{};
  FpTaps tp{};
  a.gy = gy, a.w = w, a.bias = bias, a.gi = gi;
  a.Cin = g.Cin, a.Cout = g.Cout, a.H = g.H, a.W = g.W, a.oH = g.oH, a.oW = g.oW, a.kH = g.kH, a.kW = g.kW;
  a.magicCK = dev::magicOf(g.Cin * g.kH * g.kW), a.magicKK = dev::magicOf(g.kH * g.kW);
  const int PR = (g.H + S - 1) / S, PC = (g.W + S - 1) / S;
  const int Tg = S <= 2 ? 4 : S == 3 ? 2 : 1;  // rows per lane of the run-time variant
  {  // block numbering: n * tiles + tile must divide back exactly
    const long tl = tiles(PR, 4) * tiles(PC, 16);  // at most this many blocks per image (T >= 1)
    if ((long)g.N * tl >= (1L << 31) || (double)g.N * tl * tl >= 4294967296.0) return false;
  }
  hipStream_t s = state->stream;
  const bool square = g.kH == g.kW && g.padH == g.padW;
  const int k = g.kH, pad = g.padH;
  if (square && !runtimeOnly) {
#define FEW_PLANES_SHAPE(S_, T_, K_, P_)                  \
  if (S == S_ && k == K_ && pad == P_) {                  \
    launchFewPlanes<S_, T_, K_, P_>(s, a, tp, g);         \
    return true;                                          \
  }
    FEW_PLANES_SHAPE(2, 4, 7, 3)   // 7x7 stride 2: the first layer of ResNet / Inception-v1
    FEW_PLANES_SHAPE(2, 4, 3, 1)   // 3x3 stride 2: MobileNet
    FEW_PLANES_SHAPE(2, 4, 3, 0)   // 3x3 stride 2, unpadded: Inception-v3
    FEW_PLANES_SHAPE(1, 8, 3, 1)   // 3x3: VGG
    FEW_PLANES_SHAPE(1, 8, 5, 2)   // 5x5
    FEW_PLANES_SHAPE(2, 4, 4, 1)   // 4x4 stride 2: the transposed convolutions of a generator
    FEW_PLANES_SHAPE(4, 2, 11, 2)  // 11x11 stride 4: AlexNet
#undef FEW_PLANES_SHAPE
  }
  // any other kernel size / padding: tap loops with run-time bounds
  if (g.kH * g.kW > kFpMaxTaps) return false;
  auto fill = [&](FpDim &d, int kk, int pd) {
    d.lo = fpLo(pd, S, kk), d.hi = fpHi(pd, S, kk);
    for (int ph = 0; ph < S; ++ph) d.rem[ph] = fpRem(ph, pd, S), d.q0[ph] = fpQ0(ph, pd, S), d.taps[ph] = fpTaps(ph, pd, S, kk);
  };
  fill(a.dh, g.kH, g.padH);
  fill(a.dw, g.kW, g.padW);
  a.RR = 4 * Tg + a.dh.hi - a.dh.lo, a.CC = 16 + a.dw.hi - a.dw.lo;
  a.magicCC = dev::magicOf(a.CC);
  const int pitch = Tg == 4 ? 28 : Tg == 2 ? 24 : 48;
  if (a.CC > pitch || a.RR * a.CC > 64 * kFpMaxLoads || 2 * g.Cin * g.kH * g.kW > 64 * kFpMaxWLoads ||
      a.RR * pitch >= 65536)
    return false;
  int cnt = 0;
  for (int ph = 0; ph < S; ++ph)
    for (int pw = 0; pw < S; ++pw) {
      tp.first[ph * S + pw] = cnt;
      for (int ta = 0; ta < a.dh.taps[ph]; ++ta)
        for (int tb = 0; tb < a.dw.taps[pw]; ++tb) {
          const unsigned tap = (a.dh.rem[ph] + ta * S) * g.kW + a.dw.rem[pw] + tb * S;
          const unsigned off = (a.dh.q0[ph] - ta - a.dh.lo) * pitch + (a.dw.q0[pw] - tb - a.dw.lo);
          tp.e[cnt++] = tap | off << 16;
        }
    }
  for (int q = S * S; q <= 16; ++q) tp.first[q] = cnt;
  switch (S) {
    case 1: launchFewPlanes<1, 4, 0, 0>(s, a, tp, g); break;
    case 2: launchFewPlanes<2, 4, 0, 0>(s, a, tp, g); break;
    case 3: launchFewPlanes<3, 2, 0, 0>(s, a, tp, g); break;
    default: launchFewPlanes<4, 1, 0, 0>(s, a, tp, g); break;
  }
  return true;
}

// gi(N, Cin, H, W) = conv^T(gy(N, Cout, oH, oW), w(Cout, K))
// + bias[c] per plane of gi when bias != null (the transposed convolution's forward pass)
void convGradInput(THCState *state, const ConvGeom &g, const float *gy, const float *w, float *gi,
                   THCudaTensor *scratchBuf, const char *bufName, const float *bias = nullptr) {
  if ((long)g.N * g.Cin == 0) return;
  hipStream_t s = state->stream;
  // Stride 1: gradInput is a forward convolution of gradOutput with the flipped,
  // transposed weights and padding dil*(k-1)-pad, so it runs on the implicit-GEMM
  // forward kernel and no gradient columns ever reach memory.
  const int tpH = g.dilH * (g.kH - 1) - g.padH, tpW = g.dilW * (g.kW - 1) - g.padW;
  const long goImgBytes = (long)g.Cout * (g.oH + 2 * std::max(tpH, 0)) * (g.oW + 2 * std::max(tpW, 0)) * sizeof(float);  // with its zero border
  // (with stride 1 the extents correspond exactly unless a transposed convolution asks for output padding)
  const bool exact = g.H == g.oH + 2 * tpH - g.dilH * (g.kH - 1) && g.W == g.oW + 2 * tpW - g.dilW * (g.kW - 1);
  // (one to four input planes - the first layer of a network - would fill a sixteenth of the 64-row tiles of that
  // GEMM: 1.08 ms for 3 -> 64 planes 3x3 at 224x224, N = 32; the column GEMM below has K = Cin * kH * kW rows)
  const bool sliver = g.Cin <= 4 && g.kH * g.kW > 1;
  const int route = g_switches.convGradInput;  // 1: phases, 2: columns, 3: few-plane kernel with run-time tap loops
  if (g.Cin <= 4 && (g.kH * g.kW > 1 || g.dH > 1 || g.dW > 1) && !forceGeneric() && (route == 0 || route == 3) &&
      convFewPlanesGradInput(state, g, gy, w, gi, bias, route == 3))
    return;
  // 1x1 window, stride 2, no padding, even extents (the shortcut and reduction layers of a residual network):
  // gradInput is W^T gradOutput at the even positions and the bias (or 0) everywhere else. One pointwise pass of
  // the forward kernels over gradOutput whose epilogue writes each element's whole 2 x 2 block - contiguous
  // 8-byte stores - instead of four phases that each write every other element of every other row.
  if (g.kH == 1 && g.kW == 1 && g.dH == 2 && g.dW == 2 && g.padH == 0 && g.padW == 0 && g.H == 2 * g.oH && g.W == 2 * g.oW &&
      route == 0 && !forceGeneric() && ((uintptr_t)gi & 7) == 0 && (long)g.Cout * g.oH * g.oW * 4 < (1L << 30) &&
      (long)g.Cout * g.K < 0x7fffffffL / 4) {
    ConvGeom t = g;
    t.Cin = g.Cout, t.Cout = g.Cin;
    t.H = t.oH = g.oH, t.W = t.oW = g.oW;
    t.dH = t.dW = 1;
    t.K = g.Cout;
    t.L = g.oH * g.oW;
    OutMap om{(long)g.Cin * g.H * g.W, g.H * g.W, 2 * g.W, 2, 1};
    int group = (int)std::min<long>(g.N, std::max<long>(1, 0x7fffffffL / 2 / t.L));
    group = (int)std::min<long>(group, std::max<long>(1, ((1L << 31) - 1 - 4096) / ((long)g.Cout * t.L * 4)));
    FwdPlan pl = planFwdImplicit(t.Cout, std::min(group, g.N), t, true, false);
    long need = pl.scratchFloats;
    if (g.N % group != 0) need = std::max(need, planFwdImplicit(t.Cout, g.N % group, t, true, false).scratchFloats);
    const long wfFloats = ((long)g.Cout * g.K + 3) / 4 * 4;
    Temp tmp;
    float *buf = scratchFloats(state, scratchBuf, wfFloats + need, tmp, bufName);
    flipWeightKernel<<<launch::directGrid((long)g.Cout * g.K, dev::kBlock), dev::kBlock, 0, s>>>(w, buf, g.Cout, g.Cin, 1, 1);
    THC_HIP_CHECK(hipGetLastError());
    for (int n0 = 0; n0 < g.N; n0 += group) {
      int cnt = std::min(group, g.N - n0);
      if (cnt != std::min(group, g.N)) pl = planFwdImplicit(t.Cout, cnt, t, true, false);
      launchFwdImplicit(s, pl, buf + wfFloats, buf, gy + (long)n0 * g.Cout * g.L, gi + (long)n0 * g.Cin * g.H * g.W, bias,
                        t.Cout, cnt, t, false, &om);
    }
    return;
  }
  if (!sliver && route == 0 && !(g.kH == 1 && g.kW == 1) && convHalvesGradInput(state, g, gy, w, gi, scratchBuf, bufName, bias)) return;
  if (g.dH == 1 && g.dW == 1 && tpH >= 0 && tpW >= 0 && exact && !sliver && !forceGeneric() && goImgBytes < (1L << 30) &&
      (long)g.Cout * g.K < 0x7fffffffL / 4) {
    ConvGeom t = g;  // the transposed problem
    t.Cin = g.Cout, t.Cout = g.Cin;
    t.H = g.oH, t.W = g.oW, t.oH = g.H, t.oW = g.W;
    t.padH = tpH, t.padW = tpW;
    t.K = g.Cout * g.kH * g.kW;
    t.L = g.H * g.W;
    int group = (int)std::min<long>(g.N, std::max<long>(1, 0x7fffffffL / 2 / t.L));
    group = (int)std::min<long>(group, std::max<long>(1, ((1L << 31) - 1 - 4096) / goImgBytes));
    FwdPlan pl = planFwdImplicit(t.Cout, std::min(group, g.N), t);
    long need = pl.scratchFloats;
    if (g.N % group != 0) need = std::max(need, planFwdImplicit(t.Cout, g.N % group, t).scratchFloats);
    // 1x1: gradInput = W^T gradOutput, a pointwise pass itself, which reads the weights as they are
    if (convPointwise(state, t, gy, w, bias, gi, scratchBuf, false, true)) return;
    const long wfFloats = ((long)g.Cout * g.K + 3) / 4 * 4;
    Temp tmp;
    float *buf = scratchFloats(state, scratchBuf, wfFloats + need, tmp, bufName);
    const FlipJob flip{w, buf, g.Cout, g.Cin, g.kH, g.kW};  // done by the first group's bordered copy, or by a launch of its own
    for (int n0 = 0; n0 < g.N; n0 += group) {
      int cnt = std::min(group, g.N - n0);
      if (cnt != std::min(group, g.N)) pl = planFwdImplicit(t.Cout, cnt, t);
      launchFwdImplicit(s, pl, buf + wfFloats, buf, gy + (long)n0 * g.Cout * g.L, gi + (long)n0 * g.Cin * g.H * g.W,
                        bias, t.Cout, cnt, t, false, nullptr, n0 == 0 ? &flip : nullptr);
    }
    return;
  }
  // Every other geometry goes phase by phase (with 32-row tiles that measured faster than the gradient columns
  // below down to 8 input planes: 8 -> 16 3x3 stride 2 at 128x128, N = 32: 37 against 62 us); the columns remain for
  // what that route refuses and for the test switch THCUNN_CONV_GRADINPUT = "columns".
  const bool tryPhases = route != 2;
  if (!forceGeneric() && tryPhases && gradInputByPhase(state, g, gy, w, gi, scratchBuf, bufName, bias)) return;
  // Gradient columns of a group of images at a time (<= 128 MB so the buffer stays cache resident), then
  // the col2im gather. gradCol[n][k][l] = sum_o W[o][k] * gy[n][o][l] is itself a 1x1 convolution of gy
  // with the transposed weights, so it runs on the forward kernels as well.
  const long perImg = (long)g.K * g.L;
  int group = (int)std::max<long>(1, std::min<long>(g.N, (128L << 20) / 4 / perImg));
  group = (int)std::min<long>(group, std::max<long>(1, 0x7fffffffL / 2 / g.L));
  const long gyImgBytes = (long)g.Cout * g.L * sizeof(float);
  const bool viaForward = !forceGeneric() && gyImgBytes < (1L << 30) && (long)g.Cout * g.K < 0x7fffffffL / 4;
  if (viaForward) group = (int)std::min<long>(group, std::max<long>(1, ((1L << 31) - 1 - 4096) / gyImgBytes));
  ConvGeom q{};  // the 1x1 convolution: (N, Cout, oH, oW) -> (N, K, oH, oW)
  q.N = g.N, q.Cin = g.Cout, q.Cout = g.K, q.H = q.oH = g.oH, q.W = q.oW = g.oW;
  q.kH = q.kW = q.dH = q.dW = q.dilH = q.dilW = 1;
  q.K = g.Cout, q.L = g.L;
  FwdPlan pl{};
  long wtFloats = 0;
  if (viaForward) {
    pl = planFwdImplicit(q.Cout, std::min(group, g.N), q);
    wtFloats = ((long)g.Cout * g.K + 3) / 4 * 4;
  }
  long need = pl.scratchFloats;
  if (viaForward && g.N % group != 0) need = std::max(need, planFwdImplicit(q.Cout, g.N % group, q).scratchFloats);
  const long fwdFloats = (need + 3) / 4 * 4;
  Temp tmp;
  float *buf = scratchFloats(state, scratchBuf, wtFloats + fwdFloats + (long)group * perImg, tmp, bufName);
  float *gcol = buf + wtFloats + fwdFloats;
  if (viaForward) {
    transposeKernel<<<launch::directGrid((long)g.Cout * g.K, dev::kBlock), dev::kBlock, 0, s>>>(w, buf, g.Cout, g.K);
    THC_HIP_CHECK(hipGetLastError());
  }
  for (int n0 = 0; n0 < g.N; n0 += group) {
    int cnt = std::min(group, g.N - n0);
    if (viaForward) {
      if (cnt != std::min(group, g.N)) pl = planFwdImplicit(q.Cout, cnt, q);
      launchFwdImplicit(s, pl, buf + wtFloats, buf, gy + (long)n0 * g.Cout * g.L, gcol, nullptr, q.Cout, cnt, q);
    } else {
      GemmArgs p{};
      p.a = w;
      p.b = gy;
      p.c = gcol;
      p.M = g.K;
      p.Ncols = cnt * g.L;
      p.R = g.Cout;
      p.n0 = n0;
      p.nImages = cnt;
      p.mTiles = (int)tiles(p.M, BM);
      dim3 grid(p.mTiles * tiles(p.Ncols, BN), 1);
      convGemmKernel<kGradCol><<<grid, dev::kBlock, 0, s>>>(p, g);
      THC_HIP_CHECK(hipGetLastError());
    }
    long total = (long)cnt * g.Cin * g.H * g.W;
    col2imKernel<<<launch::directGrid(total, dev::kBlock), dev::kBlock, 0, s>>>(
        gcol, gi + (long)n0 * g.Cin * g.H * g.W, cnt, g.Cin, g.H, g.W, g.kH, g.kW, g.padH, g.padW, g.dH, g.dW, g.dilH,
        g.dilW, g.oH, g.oW, bias);
    THC_HIP_CHECK(hipGetLastError());
  }
}

// gB[o] += scale * sum_{n,l} gy[n][o][l] over a (N, C, L) tensor
void convGradBias(hipStream_t s, const float *gy, float *gB, int N, int C, int L, float scale) {
  if ((long)N * C * L == 0) return;
  if (L % 4 == 0 && launch::aligned16(gy) && (long)N * (L / 4) < 0x7fffffffL)
    gradBiasKernel<true><<<C, kBiasBlock, 0, s>>>(gy, gB, N, C, L, scale);
  else
    gradBiasKernel<false><<<C, kBiasBlock, 0, s>>>(gy, gB, N, C, L, scale);
  THC_HIP_CHECK(hipGetLastError());
}

// gW(Cout, K) += scale * sum_n gy_n(Cout x L) * im2col(x_n)^T
// gB(Cout) += scale * sum_{n,l} gy when gB is given (the bias gradient of the ordinary convolution)
void convGradWeight(THCState *state, const ConvGeom &g, const float *x, const float *gy, float *gW,
                    THCudaTensor *scratchBuf, float scale, float *gB = nullptr) {
  if ((long)g.N * g.Cout * g.K == 0) return;
  hipStream_t s = state->stream;

  // Split the reduction over the N*L positions so that the grid fills the
  // resident workgroup slots of the chip exactly once: with fewer, fatter
  // splits some CUs would carry one workgroup more than others for the whole
  // kernel.
  // The second-generation kernel loads 4 consecutive positions of a gradOutput row as one 16-byte group. Rows
  // whose length is not a multiple of 4 (7x7, 13x13, 27x27 ... planes) or that start off a 16-byte boundary are
  // first copied into rows padded with zeros to a multiple of 4: the added positions contribute nothing (on the image's
  // side they are out of range, which reads as 0 too).
  const int Lp = launch::roundUp(g.L, 4);
  const bool padGy = !forceGeneric() && (g.L % 4 != 0 || !launch::aligned16(gy)) && Lp >= BK;
  const int Lk = padGy ? Lp : g.L;  // positions per image as the kernel sees them
  if ((long)g.N * Lk >= 0x7fffffffL) error("spatial convolution: batch too large");
  const int HpX = g.H + 2 * g.padH;
  // second-generation kernel: gradOutput rows loadable as float4 groups, 32-bit byte offsets into both operands
  const bool bordered = g.padH > 0 || g.padW > 0;
  const long gyBytes = (long)g.N * g.Cout * Lk * 4;
  const long xpFloats = (long)g.N * g.Cin * HpX * (g.W + 2 * g.padW);
  const long gypFloats = padGy ? (long)g.N * g.Cout * Lp : 0;
  const bool fast = !forceGeneric() && Lk % 4 == 0 && Lk >= BK && (padGy || launch::aligned16(gy)) &&
                    gyBytes < 0x7fffffffL && xpFloats * 4 < 0x7fffffffL - 65536 && (long)Lk * g.oW < 0x7fffffffL;
  const bool l16 = Lk % BK == 0;
  // tile shape: 64 x 256 where it covers gradWeight (Cout x K) with less padding than 128 x 128
  const bool wide = fast && tiles(g.Cout, 64) * 64 * tiles(g.K, 256) * 256 < tiles(g.Cout, BM) * BM * tiles(g.K, BN) * BN;
  // 16-byte gathers of the image: unit stride along a row, and groups of 4 positions that stay inside an output row
  // (or output rows that follow each other in the image without a gap: kW = 1, no padding, unit stride down too)
  const bool b4 = fast && !padGy && g.dW == 1 && (g.oW % 4 == 0 || (g.dH == 1 && g.W + 2 * g.padW == g.oW));
  // Small tiles (32 x 32 blocks: 1x1, 1x2, 2x1, 2x2) where the large shapes would mostly multiply padding. The shape is
  // the one with the least tiles x cost of a tile per position, in proportion to measured times: 64 x 147 over
  // 32 x 112 x 112 positions, stride 2 (us, without the bordered copy): 10 tiles of 1x1 105, 6 of 1x2 107, 5 of 2x1 83,
  // 3 of 2x2 80, one of 64 x 256 86; 64 x 576 over 32 x 56 x 56, stride 1: 86, 72, 72, 56, 51 (16-byte gathers). The
  // first took 116 with the fp32 instruction (2x1), the second 81 (128 x 128). (All of the split ones are 2 - 3 % longer now
  // that operands are scaled as they are split: the 2x2 kernel of the first 98 -> 100 us in a whole pass.)
  struct Shape {
    int ti, tj, cost;
  };
  static const Shape kSmall[] = {{2, 2, 85}, {1, 2, 55}, {2, 1, 53}, {1, 1, 33}};
  const int bigCost = b4 ? 240 : 270;  // a 128 x 128 or 64 x 256 tile
  long bestCost = std::min(tiles(g.Cout, 64) * tiles(g.K, 256), tiles(g.Cout, BM) * tiles(g.K, BN)) * (long)bigCost;
  int tI = 0, tJ = 0;
  if (fast)
    for (const Shape &sh : kSmall) {
      const long c = (long)tiles(g.Cout, 32 * sh.ti) * tiles(g.K, 32 * sh.tj) * sh.cost;
      if (c < bestCost) bestCost = c, tI = sh.ti, tJ = sh.tj;
    }
  // Short reductions: up to 16 blocks of 32 x 32 x 64 positions per CU, every larger tile leaves CUs idle, and its start and
  // end (16 KB of sums per block folded through LDS) are most of the time. us, the shape by cost / 1x1: 136 x 64 over 64
  // positions 10.4 / 7.5; 64 x 64 over 6480 13.0 / 9.8; 456 x 200 over 484 18.2 / 12.4; 144 x 432 over 2312 (10 per CU) 24.2 /
  // 20.5; 240 x 2600 over 486 (20 per CU) 26.9 / 27.1; 368 x 288 over 5184 (34 per CU) 33.1 / 32.9.
  if (fast && tiles(g.Cout, 32) * tiles(g.K, 32) * (long)launch::ceilDiv(g.N * Lk, kSmallPositions) <= 16L * residentSlots(nullptr))
    tI = tJ = 1;
  const bool tiny = tI > 0;
  const int mT = (int)tiles(g.Cout, tiny ? 32 * tI : wide ? 64 : BM), nT = (int)tiles(g.K, tiny ? 32 * tJ : wide ? 256 : BN);
  struct Kernel {
    const void *fn;
    void (*launch)(dim3, hipStream_t, const GradWeightArgs &, const ConvGeom &);
  };
  auto smallKernel = [](auto tic, auto tjc) {
    constexpr int I = decltype(tic)::value, J = decltype(tjc)::value;
    return Kernel{(const void *)convGradWeightSmallKernel<I, J>,
                  [](dim3 grid, hipStream_t st, const GradWeightArgs &q, const ConvGeom &gk) {
                    convGradWeightSmallKernel<I, J><<<grid, dev::kBlock, 0, st>>>(q, gk);
                  }};
  };
  auto pickSmall = [&]() {
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    if (tI == 1 && tJ == 1) return smallKernel(I1{}, I1{});
    if (tI == 1 && tJ == 2) return smallKernel(I1{}, I2{});
    if (tI == 2 && tJ == 1) return smallKernel(I2{}, I1{});
    return smallKernel(I2{}, I2{});
  };
  bool halves = false;
  auto bigKernel = [&halves](auto l16c, auto wmc, auto b4c) {
    constexpr bool L = decltype(l16c)::value, B = decltype(b4c)::value;
    constexpr int W = decltype(wmc)::value;
    if (halves)
      return Kernel{(const void *)convGradWeightSplitKernel<L, W, B, true>,
                    [](dim3 grid, hipStream_t st, const GradWeightArgs &q, const ConvGeom &gk) {
                      convGradWeightSplitKernel<L, W, B, true><<<grid, dev::kBlock, 0, st>>>(q, gk);
                    }};
    return Kernel{(const void *)convGradWeightSplitKernel<L, W, B, false>,
                  [](dim3 grid, hipStream_t st, const GradWeightArgs &q, const ConvGeom &gk) {
                    convGradWeightSplitKernel<L, W, B, false><<<grid, dev::kBlock, 0, st>>>(q, gk);
                  }};
  };
  auto pickBig = [&](auto l16c, auto wmc) { return b4 ? bigKernel(l16c, wmc, std::true_type{}) : bigKernel(l16c, wmc, std::false_type{}); };
  auto pickBigW = [&](auto l16c) {
    return wide ? pickBig(l16c, std::integral_constant<int, 1>{}) : pickBig(l16c, std::integral_constant<int, 2>{});
  };
  auto pick = [&]() { return tiny ? pickSmall() : l16 ? pickBigW(std::true_type{}) : pickBigW(std::false_type{}); };
  Kernel gw = pick();
  const void *kern = fast ? gw.fn : (const void *)convGemmKernel<kGradWeight>;
  const int ktPositions = tiny ? kSmallPositions : BK;
  const int totalKt = launch::ceilDiv(g.N * Lk, ktPositions);
  // Every split leaves a partial copy of gradWeight (64 KB per large tile) for the fold. The registers hold two workgroups
  // of the large tiles on a CU, three or four of the small ones, which stream: as many as fit, to have enough loads in
  // flight; two where gradWeight is one or two tiles and the partials are most of the traffic. A split should keep at
  // least about 20 k-tiles of 16 positions (short reductions at 14x14 and 7x7: with 8 k-tiles per split the partial
  // copies and the pipeline fill cost more than another workgroup per CU gains).
  int perCu = mT * nT <= 2 ? 2 : tiny ? 4 : 3;  // (the large tiles' limit comes from the resident slots)
  auto splitsAt = [&](int wgPerCu) {
    const int slots = std::min(residentSlots(kern), residentSlots(nullptr) * wgPerCu);
    return std::max(1, std::min(totalKt, slots / (mT * nT)));
  };
  while (perCu > 1 && totalKt / splitsAt(perCu) < 20 * BK / ktPositions) --perCu;
  int splits = splitsAt(perCu);
  // slices of an image that rangesKernel reads: about 1024 workgroups, at least 4096 floats each
  auto slices = [&](long perImg) { return (int)std::max<long>(1, std::min<long>(perImg / 4096, launch::ceilDiv(1024, g.N))); };
  const int gySlots = slices((long)g.Cout * g.L), xSlots = slices((long)g.Cin * g.H * g.W);
  const long rangeFloats = 2L * g.N * (gySlots + xSlots);
  const long count = (long)g.Cout * g.K;
  const bool fold4 = count % 4 == 0 && launch::aligned16(gW);
  // Long reductions on half-precision parts, with five times the splits. That keeps their error no larger than that of six products
  // from about 2800 positions a split of those on, with both operands half zeros, too (as behind a ReLU; a bf16 product adds
  // without rounding, so six products are the better the fewer of the terms count): 3600 positions 2.0e-7 against 3.0e-7 with
  // the input half zeros, 1.9e-7 against 2.15e-7 with both; and where the fold does not add all splits one after the other.
  // Fast enough: the products take 4.5 us less for 10^9 of them (3.4 / 2.2 where the image is gathered element by element, with a
  // stride), the ranges read both tensors and the splits leave more partials; where no split can take fp16 parts only that is left.
  const int perSplitSix = launch::ceilDiv(totalKt, splits) * BK;
  const long moreSplits = std::min(totalKt, 5 * splits);
  const double moved = 4.0 * g.N * ((double)g.Cin * g.H * g.W + (double)g.Cout * g.L) + 8.0 * (moreSplits - splits) * count;
  const bool pays = fold4 && perSplitSix >= 2800 && (double)g.N * g.L * count * (b4 ? 4.5e-9 : g.dW == 1 ? 3.4e-9 : 2.2e-9) >= 1.5 * (3.0 + moved / 6e6);
  // (They need more scratch: not with a buffer that cannot grow.)
  if (fast && !tiny && g_switches.convHalves != 0 && (pays || g_switches.convHalves == 1) &&
      (!scratchBuf || (growable(scratchBuf) && roomFor(state, scratchBuf, moreSplits * (count + g.Cout) + xpFloats + gypFloats +
                                                                          rangeFloats + 16)))) {
    halves = true;
    gw = pick();
    kern = gw.fn;
    splits = (int)moreSplits;
  }
  const int perSplit = launch::ceilDiv(totalKt, splits);
  splits = launch::ceilDiv(totalKt, perSplit);
  // scratch: the splits' partial products, then (second-generation kernel) the images with their zero border
  const long partialFloats = (splits * count + 3) / 4 * 4;
  // the bias gradient rides along when the fold below has the 16-byte form; else it is a pass of its own
  const bool fusedBias = gB && fast && fold4 && g.Cout % 4 == 0 && launch::aligned16(gB);
  const long biasFloats = fusedBias ? ((long)splits * g.Cout + 3) / 4 * 4 : 0;
  Temp tmp;
  const long xpScratch = fast && bordered ? (xpFloats + 3) / 4 * 4 : 0;
  const long slotFloats = halves ? rangeFloats : 0;
  float *partial = scratchFloats(state, scratchBuf, partialFloats + biasFloats + xpScratch + (fast ? (gypFloats + 3) / 4 * 4 : 0) + slotFloats, tmp,
                                 "columns");
  float *biasPartial = fusedBias ? partial + partialFloats : nullptr;
  if (fast) {
    ConvGeom gk = g;
    const float *xk = x, *gyk = gy;
    if (bordered) {
      float *xp = partial + partialFloats + biasFloats;
      launchPadPlanes(s, x, xp, (long)g.N * g.Cin, g.H, g.W, g.padH, g.padW, HpX, g.W + 2 * g.padW);
      gk.H = HpX, gk.W = g.W + 2 * g.padW, gk.padH = gk.padW = 0;
      xk = xp;
    }
    if (padGy) {  // rows of L floats -> rows of Lp floats, zeros behind
      float *gyp = partial + partialFloats + biasFloats + xpScratch;
      launchPadPlanes(s, gy, gyp, (long)g.N * g.Cout, 1, g.L, 0, 0, 1, Lp);
      gk.L = Lp;
      gyk = gyp;
    }
    GradWeightArgs q{};
    q.gy = gyk;
    q.x = xk;
    q.partial = partial;
    q.biasPartial = biasPartial;
    q.M = g.Cout;
    q.Ncols = g.K;
    q.mTiles = mT;
    q.nTiles = nT;
    q.totalKt = totalKt;
    q.ktPerSplit = perSplit;
    q.gyBytes = (int)gyBytes;
    q.xBytes = (int)(xpFloats * 4);
    q.magicOW = dev::magicOf(g.oW);
    q.magicKK = dev::magicOf(g.kH * g.kW), q.magicKW = dev::magicOf(g.kW);
    q.Lvalid = g.L;
    if (halves) {
      uint2 *slots = reinterpret_cast<uint2 *>(partial + partialFloats + biasFloats + xpScratch + (gypFloats + 3) / 4 * 4);
      auto ranges = [&](const float *t, long perImg, int nSlots, uint2 *dst) {
        RangeArgs ra{};
        ra.x = t, ra.slots = dst, ra.perImg = perImg, ra.perSlice = (int)((perImg + nSlots - 1) / nSlots + 3) / 4 * 4, ra.nSlots = nSlots;
        ra.vec = perImg % 4 == 0 && launch::aligned16(t);
        rangesKernel<<<(unsigned)(g.N * nSlots), dev::kBlock, 0, s>>>(ra);
        THC_HIP_CHECK(hipGetLastError());
        return dst;
      };
      q.gyNSlots = gySlots, q.gySlots = ranges(gy, (long)g.Cout * g.L, gySlots, slots);
      q.xNSlots = xSlots, q.xSlots = ranges(x, (long)g.Cin * g.H * g.W, xSlots, slots + (long)g.N * gySlots);
    }
    gw.launch(dim3(mT * nT * splits), s, q, gk);
  } else {
    GemmArgs p{};
    p.a = gy;
    p.b = x;
    p.c = partial;
    p.M = g.Cout;
    p.Ncols = g.K;
    p.R = 0;
    p.n0 = perSplit;
    p.nImages = g.N;
    p.mTiles = mT;
    p.vecA = (g.L % 4 == 0) && launch::aligned16(p.a);
    dim3 grid(mT * nT, splits);
    convGemmKernel<kGradWeight><<<grid, dev::kBlock, 0, s>>>(p, g);
  }
  THC_HIP_CHECK(hipGetLastError());
  if (fold4) {  // (the scratch starts on a 16-byte boundary)
    // elements per workgroup: the fewest (most lane groups over the splits) that still give 128 workgroups
    const int E = count / 4 >= 128 * 64 ? 64 : count / 4 >= 128 * 16 ? 16 : 4;
    const int gwBlocks = (int)((count / 4 + E - 1) / E);
    const int biasBlocks = fusedBias ? launch::ceilDiv(g.Cout / 4, E) : 0;
    if (E == 64)
      foldPartials4Kernel<64><<<gwBlocks + biasBlocks, dev::kBlock, 0, s>>>(partial, gW, count / 4, splits, scale, biasPartial,
                                                                           gB, g.Cout, gwBlocks);
    else if (E == 16)
      foldPartials4Kernel<16><<<gwBlocks + biasBlocks, dev::kBlock, 0, s>>>(partial, gW, count / 4, splits, scale, biasPartial,
                                                                           gB, g.Cout, gwBlocks);
    else
      foldPartials4Kernel<4><<<gwBlocks + biasBlocks, dev::kBlock, 0, s>>>(partial, gW, count / 4, splits, scale, biasPartial,
                                                                          gB, g.Cout, gwBlocks);
  } else {
    foldPartialsKernel<<<launch::directGrid(count, dev::kBlock), dev::kBlock, 0, s>>>(partial, gW, count, splits, scale);
  }
  THC_HIP_CHECK(hipGetLastError());
  if (gB && !fusedBias) convGradBias(s, gy, gB, g.N, g.Cout, g.L, scale);
}

// ---- entry-point bodies shared by SpatialConvolutionMM and SpatialDilatedConvolution --------
void convUpdateOutput(THCState *state, THCudaTensor *input, THCudaTensor *output, THCudaTensor *weight,
                      THCudaTensor *bias, THCudaTensor *columns, int kW, int kH, int dW, int dH, int padW, int padH,
                      int dilW, int dilH, ConvFlavor flavor, bool relu = false) {
  THC_ARG_CHECK(output != nullptr, 3, "output tensor expected");
  ConvCall call = convSetup(input, nullptr, weight, bias, "weight", kH, kW, dH, dW, padH, padW, dilH, dilW, flavor);
  ConvGeom &g = call.g;
  Contiguous in(state, input);
  if (call.batch)
    resize(state, output, {g.N, g.Cout, g.oH, g.oW});
  else
    resize(state, output, {g.Cout, g.oH, g.oW});
  if (!isContiguous(erase(output))) error("output tensor has to be contiguous");
  convForward(state, g, in.ptr(), data(weight), bias ? data(bias) : nullptr, data(output), columns, "columns", relu);
}

void convUpdateGradInput(THCState *state, THCudaTensor *input, THCudaTensor *gradOutput, THCudaTensor *gradInput,
                         THCudaTensor *weight, THCudaTensor *gradColumns, int kW, int kH, int dW, int dH, int padW,
                         int padH, int dilW, int dilH, ConvFlavor flavor) {
  THC_ARG_CHECK(gradOutput != nullptr, 3, "gradOutput tensor expected");
  THC_ARG_CHECK(gradInput != nullptr, 4, "gradInput tensor expected");
  ConvCall call = convSetup(input, gradOutput, weight, nullptr, "weight", kH, kW, dH, dW, padH, padW, dilH, dilW, flavor);
  ConvGeom &g = call.g;
  Contiguous go(state, gradOutput);
  if (call.batch)
    resize(state, gradInput, {g.N, g.Cin, g.H, g.W});
  else
    resize(state, gradInput, {g.Cin, g.H, g.W});
  if (!isContiguous(erase(gradInput))) error("gradInput tensor has to be contiguous");
  convGradInput(state, g, go.ptr(), data(weight), data(gradInput), gradColumns, "gradColumns");
}

void convAccGradParameters(THCState *state, THCudaTensor *input, THCudaTensor *gradOutput, THCudaTensor *gradWeight,
                           THCudaTensor *gradBias, THCudaTensor *columns, int kW, int kH, int dW, int dH, int padW,
                           int padH, int dilW, int dilH, float scale, ConvFlavor flavor) {
  THC_ARG_CHECK(gradOutput != nullptr, 3, "gradOutput tensor expected");
  THC_ARG_CHECK(gradWeight != nullptr, 4, "gradWeight tensor expected");
  ConvCall call = convSetup(input, gradOutput, gradWeight, gradBias, "weight", kH, kW,
                            dH, dW, padH, padW, dilH, dilW, flavor);
  ConvGeom &g = call.g;
  Contiguous in(state, input);
  Contiguous go(state, gradOutput);
  convGradWeight(state, g, in.ptr(), go.ptr(), data(gradWeight), columns, scale, gradBias ? data(gradBias) : nullptr);
}

// ---- transposed ("full") convolution -----------------------------------------------------------
// SpatialFull(Dilated)Convolution maps the (N, Cin, H, W) input to (N, Cout, oH, oW) with
// oH = (H-1)*dH - 2*padH + dilH*(kH-1) + 1 + adjH; its weight is (Cin, Cout, kH, kW). It is the
// ordinary convolution C with input (N, Cout, oH, oW), output (N, Cin, H, W) and weight
// (Cin, Cout*kH*kW) run backwards: updateOutput = C's gradInput pass (+ bias), updateGradInput =
// C's forward pass, accGradParameters = C's weight-gradient pass with the roles of input and
// gradOutput swapped (lib/THCUNN/generic/SpatialFullDilatedConvolution.cu:141-165, 268-298, 385-414).
// The geometry returned here is C's.
ConvCall fullSetup(THCudaTensor *input, THCudaTensor *gradOutput, THCudaTensor *weight, THCudaTensor *bias, int kH,
                   int kW, int dH, int dW, int padH, int padW, int dilH, int dilW, int adjH, int adjW) {
  // lib/THCUNN/generic/SpatialFullDilatedConvolution.cu:5-66
  THC_ARG_CHECK(input && weight, 2, "input and weight tensors expected");
  THC_ARG_CHECK(kW > 0 && kH > 0, 9, "kernel size should be greater than zero, but got kH: %d kW: %d", kH, kW);
  THC_ARG_CHECK(dW > 0 && dH > 0, 11, "stride should be greater than zero, but got dH: %d dW: %d", dH, dW);
  THC_ARG_CHECK(dilW > 0 && dilH > 0, 15, "dilation should be greater than zero, but got dilationH: %d, dilationW: %d",
                dilH, dilW);
  THC_ARG_CHECK((adjW < dW || adjW < dilW) && (adjH < dH || adjH < dilH), 15,
                "output padding must be smaller than either stride or dilation, but got adjH: %d adjW: %d dH: %d dW: %d "
                "dilationH: %d dilationW: %d",
                adjH, adjW, dH, dW, dilH, dilW);
  THC_ARG_CHECK(isContiguous(erase(weight)), 4, "weight tensor has to be contiguous");
  THC_ARG_CHECK(!bias || isContiguous(erase(bias)), 5, "bias tensor has to be contiguous");
  THC_ARG_CHECK(weight->nDimension == 2 || weight->nDimension == 4, 5, "2D or 4D weight tensor expected, but got: %s",
                sizeDesc(erase(weight)).c_str());
  if (bias) checkDimSize(erase(bias), "bias", 1, 0, weight->size[1]);
  int ndim = input->nDimension;
  int dimf = 0, dimh = 1, dimw = 2;
  if (ndim == 4) {
    dimf++;
    dimh++;
    dimw++;
  }
  THC_ARG_CHECK(ndim == 3 || ndim == 4, 2, "3D or 4D input tensor expected but got: %s",
                sizeDesc(erase(input)).c_str());
  if (weight->nDimension != 4) error("transposed convolution: 4D weight tensor (nInputPlane,nOutputPlane,kH,kW) expected");
  long nInputPlane = weight->size[0], nOutputPlane = weight->size[1];
  long inputHeight = input->size[dimh], inputWidth = input->size[dimw];
  long outputHeight = (inputHeight - 1) * dH - 2 * padH + (dilH * (kH - 1) + 1) + adjH;
  long outputWidth = (inputWidth - 1) * dW - 2 * padW + (dilW * (kW - 1) + 1) + adjW;
  if (outputWidth < 1 || outputHeight < 1)
    error("Given input size: (%ld x %ld x %ld). Calculated output size: (%ld x %ld x %ld). Output size is too small",
          nInputPlane, inputHeight, inputWidth, nOutputPlane, outputHeight, outputWidth);
  checkDimSize(erase(input), "input", ndim, dimf, nInputPlane);
  if (gradOutput) {
    checkDimSize(erase(gradOutput), "gradOutput", ndim, dimf, nOutputPlane);
    checkDimSize(erase(gradOutput), "gradOutput", ndim, dimh, outputHeight);
    checkDimSize(erase(gradOutput), "gradOutput", ndim, dimw, outputWidth);
    if (ndim == 4 && gradOutput->size[0] != input->size[0])
      error("input and gradOutput batch sizes do not match: input %s, gradOutput %s", sizeDesc(erase(input)).c_str(),
            sizeDesc(erase(gradOutput)).c_str());
  }
  if (weight->size[2] != kH || weight->size[3] != kW)
    error("weight of shape %s does not match a %d x %d kernel", sizeDesc(erase(weight)).c_str(), kH, kW);
  ConvCall call;
  call.batch = ndim == 4;
  call.g = makeGeom(call.batch ? (int)input->size[0] : 1, (int)nOutputPlane, (int)nInputPlane, (int)outputHeight,
                    (int)outputWidth, (int)inputHeight, (int)inputWidth, kH, kW, dH, dW, padH, padW, dilH, dilW);
  return call;
}

void fullUpdateOutput(THCState *state, THCudaTensor *input, THCudaTensor *output, THCudaTensor *weight,
                      THCudaTensor *bias, THCudaTensor *columns, int kW, int kH, int dW, int dH, int padW, int padH,
                      int dilW, int dilH, int adjW, int adjH) {
  THC_ARG_CHECK(output != nullptr, 3, "output tensor expected");
  ConvCall call = fullSetup(input, nullptr, weight, bias, kH, kW, dH, dW, padH, padW, dilH, dilW, adjH, adjW);
  ConvGeom &g = call.g;
  Contiguous in(state, input);
  if (call.batch)
    resize(state, output, {g.N, g.Cin, g.H, g.W});
  else
    resize(state, output, {g.Cin, g.H, g.W});
  if (!isContiguous(erase(output))) error("output tensor has to be contiguous");
  convGradInput(state, g, in.ptr(), data(weight), data(output), columns, "columns", bias ? data(bias) : nullptr);
}

void fullUpdateGradInput(THCState *state, THCudaTensor *input, THCudaTensor *gradOutput, THCudaTensor *gradInput,
                         THCudaTensor *weight, THCudaTensor *gradColumns, int kW, int kH, int dW, int dH, int padW,
                         int padH, int dilW, int dilH, int adjW, int adjH) {
  THC_ARG_CHECK(gradOutput != nullptr, 3, "gradOutput tensor expected");
  THC_ARG_CHECK(gradInput != nullptr, 4, "gradInput tensor expected");
  ConvCall call = fullSetup(input, gradOutput, weight, nullptr, kH, kW, dH, dW, padH, padW, dilH, dilW, adjH, adjW);
  ConvGeom &g = call.g;
  Contiguous go(state, gradOutput);
  if (call.batch)
    resize(state, gradInput, {g.N, g.Cout, g.oH, g.oW});
  else
    resize(state, gradInput, {g.Cout, g.oH, g.oW});
  if (!isContiguous(erase(gradInput))) error("gradInput tensor has to be contiguous");
  convForward(state, g, go.ptr(), data(weight), nullptr, data(gradInput), gradColumns, "gradColumns");
}

void fullAccGradParameters(THCState *state, THCudaTensor *input, THCudaTensor *gradOutput, THCudaTensor *gradWeight,
                           THCudaTensor *gradBias, THCudaTensor *columns, int kW, int kH, int dW, int dH, int padW,
                           int padH, int dilW, int dilH, int adjW, int adjH, float scale) {
  THC_ARG_CHECK(gradOutput != nullptr, 3, "gradOutput tensor expected");
  THC_ARG_CHECK(gradWeight != nullptr, 4, "gradWeight tensor expected");
  ConvCall call = fullSetup(input, gradOutput, gradWeight, gradBias, kH, kW, dH, dW, padH, padW, dilH, dilW, adjH, adjW);
  ConvGeom &g = call.g;
  Contiguous in(state, input);
  Contiguous go(state, gradOutput);
  convGradWeight(state, g, go.ptr(), in.ptr(), data(gradWeight), columns, scale);
  if (gradBias) convGradBias(state->stream, go.ptr(), data(gradBias), g.N, g.Cin, g.H * g.W, scale);
}

}  // namespace

extern "C" {

void THNN_CudaSpatialConvolutionMM_updateOutput(THCState *state, THCudaTensor *input, THCudaTensor *output,
                                                THCudaTensor *weight, THCudaTensor *bias, THCudaTensor *columns,
                                                THCudaTensor *ones, int kW, int kH, int dW, int dH, int padW,
                                                int padH) {
  THNN_ENTER
  (void)ones;  // never read; `columns` is used (and resized) only as scratch
  convUpdateOutput(state, input, output, weight, bias, columns, kW, kH, dW, dH, padW, padH, 1, 1, kConvMM);
  THNN_LEAVE
}

// No counterpart in the reference (include/THCUNN_fused.h): SpatialConvolutionMM_updateOutput followed by
// Threshold_updateOutput(0, 0), the clamp applied as the convolution stores its values.
void THNN_CudaSpatialConvolutionMMReLU_updateOutput(THCState *state, THCudaTensor *input, THCudaTensor *output,
                                                    THCudaTensor *weight, THCudaTensor *bias, THCudaTensor *columns,
                                                    THCudaTensor *ones, int kW, int kH, int dW, int dH, int padW,
                                                    int padH) {
  THNN_ENTER
  (void)ones;
  convUpdateOutput(state, input, output, weight, bias, columns, kW, kH, dW, dH, padW, padH, 1, 1, kConvMM, true);
  THNN_LEAVE
}

void THNN_CudaSpatialConvolutionMM_updateGradInput(THCState *state, THCudaTensor *input, THCudaTensor *gradOutput,
                                                   THCudaTensor *gradInput, THCudaTensor *weight,
                                                   THCudaTensor *gradColumns, THCudaTensor *ones, int kW, int kH,
                                                   int dW, int dH, int padW, int padH) {
  THNN_ENTER
  (void)ones;
  convUpdateGradInput(state, input, gradOutput, gradInput, weight, gradColumns, kW, kH, dW, dH, padW, padH, 1, 1, kConvMM);
  THNN_LEAVE
}

void THNN_CudaSpatialConvolutionMM_accGradParameters(THCState *state, THCudaTensor *input, THCudaTensor *gradOutput,
                                                     THCudaTensor *gradWeight, THCudaTensor *gradBias,
                                                     THCudaTensor *columns, THCudaTensor *ones, int kW, int kH,
                                                     int dW, int dH, int padW, int padH, float scale) {
  THNN_ENTER
  (void)ones;
  convAccGradParameters(state, input, gradOutput, gradWeight, gradBias, columns, kW, kH, dW, dH, padW, padH, 1, 1, scale,
                        kConvMM);
  THNN_LEAVE
}

// SpatialDilatedConvolution (lib/THCUNN/generic/SpatialDilatedConvolution.cu:69-190, 192-293, 295-432):
// the same three GEMMs with taps dilationH/W apart.
void THNN_CudaSpatialDilatedConvolution_updateOutput(THCState *state, THCudaTensor *input, THCudaTensor *output,
                                                     THCudaTensor *weight, THCudaTensor *bias, THCudaTensor *columns,
                                                     THCudaTensor *ones, int kW, int kH, int dW, int dH, int padW,
                                                     int padH, int dilationW, int dilationH) {
  THNN_ENTER
  (void)ones;
  convUpdateOutput(state, input, output, weight, bias, columns, kW, kH, dW, dH, padW, padH, dilationW, dilationH,
                   kDilated);
  THNN_LEAVE
}

void THNN_CudaSpatialDilatedConvolution_updateGradInput(THCState *state, THCudaTensor *input,
                                                        THCudaTensor *gradOutput, THCudaTensor *gradInput,
                                                        THCudaTensor *weight, THCudaTensor *gradColumns, int kW,
                                                        int kH, int dW, int dH, int padW, int padH, int dilationW,
                                                        int dilationH) {
  THNN_ENTER
  convUpdateGradInput(state, input, gradOutput, gradInput, weight, gradColumns, kW, kH, dW, dH, padW, padH, dilationW,
                      dilationH, kDilated);
  THNN_LEAVE
}

void THNN_CudaSpatialDilatedConvolution_accGradParameters(THCState *state, THCudaTensor *input,
                                                          THCudaTensor *gradOutput, THCudaTensor *gradWeight,
                                                          THCudaTensor *gradBias, THCudaTensor *columns,
                                                          THCudaTensor *ones, int kW, int kH, int dW, int dH,
                                                          int padW, int padH, int dilationW, int dilationH,
                                                          float scale) {
  THNN_ENTER
  (void)ones;
  convAccGradParameters(state, input, gradOutput, gradWeight, gradBias, columns, kW, kH, dW, dH, padW, padH, dilationW,
                        dilationH, scale, kDilated);
  THNN_LEAVE
}

// SpatialFullDilatedConvolution / SpatialFullConvolution
// (lib/THCUNN/generic/SpatialFullDilatedConvolution.cu:68-204, 206-312, 314-465; generic/SpatialFullConvolution.cu:5-59)
void THNN_CudaSpatialFullDilatedConvolution_updateOutput(THCState *state, THCudaTensor *input, THCudaTensor *output,
                                                         THCudaTensor *weight, THCudaTensor *bias,
                                                         THCudaTensor *columns, THCudaTensor *ones, int kW, int kH,
                                                         int dW, int dH, int padW, int padH, int dilationW,
                                                         int dilationH, int adjW, int adjH) {
  THNN_ENTER
  (void)ones;
  fullUpdateOutput(state, input, output, weight, bias, columns, kW, kH, dW, dH, padW, padH, dilationW, dilationH, adjW,
                   adjH);
  THNN_LEAVE
}

void THNN_CudaSpatialFullDilatedConvolution_updateGradInput(THCState *state, THCudaTensor *input,
                                                            THCudaTensor *gradOutput, THCudaTensor *gradInput,
                                                            THCudaTensor *weight, THCudaTensor *gradColumns, int kW,
                                                            int kH, int dW, int dH, int padW, int padH,
                                                            int dilationW, int dilationH, int adjW, int adjH) {
  THNN_ENTER
  fullUpdateGradInput(state, input, gradOutput, gradInput, weight, gradColumns, kW, kH, dW, dH, padW, padH, dilationW,
                      dilationH, adjW, adjH);
  THNN_LEAVE
}

void THNN_CudaSpatialFullDilatedConvolution_accGradParameters(THCState *state, THCudaTensor *input,
                                                              THCudaTensor *gradOutput, THCudaTensor *gradWeight,
                                                              THCudaTensor *gradBias, THCudaTensor *columns,
                                                              THCudaTensor *ones, int kW, int kH, int dW, int dH,
                                                              int padW, int padH, int dilationW, int dilationH,
                                                              int adjW, int adjH, float scale) {
  THNN_ENTER
  (void)ones;
  fullAccGradParameters(state, input, gradOutput, gradWeight, gradBias, columns, kW, kH, dW, dH, padW, padH, dilationW,
                        dilationH, adjW, adjH, scale);
  THNN_LEAVE
}

void THNN_CudaSpatialFullConvolution_updateOutput(THCState *state, THCudaTensor *input, THCudaTensor *output,
                                                  THCudaTensor *weight, THCudaTensor *bias, THCudaTensor *columns,
                                                  THCudaTensor *ones, int kW, int kH, int dW, int dH, int padW,
                                                  int padH, int adjW, int adjH) {
  THNN_ENTER
  (void)ones;
  fullUpdateOutput(state, input, output, weight, bias, columns, kW, kH, dW, dH, padW, padH, 1, 1, adjW, adjH);
  THNN_LEAVE
}

void THNN_CudaSpatialFullConvolution_updateGradInput(THCState *state, THCudaTensor *input, THCudaTensor *gradOutput,
                                                     THCudaTensor *gradInput, THCudaTensor *weight,
                                                     THCudaTensor *gradColumns, int kW, int kH, int dW, int dH,
                                                     int padW, int padH, int adjW, int adjH) {
  THNN_ENTER
  fullUpdateGradInput(state, input, gradOutput, gradInput, weight, gradColumns, kW, kH, dW, dH, padW, padH, 1, 1, adjW,
                      adjH);
  THNN_LEAVE
}

void THNN_CudaSpatialFullConvolution_accGradParameters(THCState *state, THCudaTensor *input, THCudaTensor *gradOutput,
                                                       THCudaTensor *gradWeight, THCudaTensor *gradBias,
                                                       THCudaTensor *columns, THCudaTensor *ones, int kW, int kH,
                                                       int dW, int dH, int padW, int padH, int adjW, int adjH,
                                                       float scale) {
  THNN_ENTER
  (void)ones;
  fullAccGradParameters(state, input, gradOutput, gradWeight, gradBias, columns, kW, kH, dW, dH, padW, padH, 1, 1, adjW,
                        adjH, scale);
  THNN_LEAVE
}

// Stand-alone im2col / col2im over a batch of images with the semantics of
// lib/THCUNN/im2col.h:40-61 and :104-121 (the reference keeps them as C++
// templates inside the library; they are exported here so that their parity
// can be checked on their own).
void THNN_Cuda_im2col(THCState *state, const float *im, int nImages, int channels, int height, int width, int kH,
                      int kW, int padH, int padW, int dH, int dW, int dilH, int dilW, float *col) {
  THNN_ENTER
  int oH = (height + 2 * padH - (dilH * (kH - 1) + 1)) / dH + 1;
  int oW = (width + 2 * padW - (dilW * (kW - 1) + 1)) / dW + 1;
  long total = (long)nImages * channels * kH * kW * oH * oW;
  if (total <= 0) return;
  im2colKernel<<<launch::directGrid(total, dev::kBlock), dev::kBlock, 0, state->stream>>>(
      im, col, nImages, channels, height, width, kH, kW, padH, padW, dH, dW, dilH, dilW, oH, oW);
  THC_HIP_CHECK(hipGetLastError());
  THNN_LEAVE
}

void THNN_Cuda_col2im(THCState *state, const float *col, int nImages, int channels, int height, int width, int kH,
                      int kW, int padH, int padW, int dH, int dW, int dilH, int dilW, float *im) {
  THNN_ENTER
  int oH = (height + 2 * padH - (dilH * (kH - 1) + 1)) / dH + 1;
  int oW = (width + 2 * padW - (dilW * (kW - 1) + 1)) / dW + 1;
  long total = (long)nImages * channels * height * width;
  if (total <= 0) return;
  col2imKernel<<<launch::directGrid(total, dev::kBlock), dev::kBlock, 0, state->stream>>>(
      col, im, nImages, channels, height, width, kH, kW, padH, padW, dH, dW, dilH, dilW, oH, oW, nullptr);
  THC_HIP_CHECK(hipGetLastError());
  THNN_LEAVE
}

}  // extern "C"
