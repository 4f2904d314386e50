// Backward pass of BatchNormalization in training with a team of workgroups per channel (included by batchnorm.hip).
//
// A channel that does not fit the registers of one compute unit used to be read twice (sums, then gradInput). Here the channel
// is cut into pieces, one workgroup each: it loads its piece once into registers, publishes the piece's two sums, waits for
// those of the others, merges all of them in the same order and writes its results. Every byte crosses HBM once. Bound by memory; 64 x 112 x 112, N = 32 (with ReLU): 85.2 -> 63.1 us (53 at the rate of a large copy).
// Two workgroups of 121 registers share a compute unit, so that one loads while the other waits or stores.
// (The forward pass stays with the kernels it had: the sign of a normalised element within rounding of zero decides a fused
// ReLU's gradient, so its statistics keep their order of summation.)
//
// The sums travel as 64-bit values (number, tag of the launch), so that a slot proves itself and no fence is needed. The tag is
// the host's (taggedScratch): no slot of the scratch holds it when the launch begins.
//
// The wait is bounded: pieces start in the order of their numbers and a team is far smaller than what the chip holds, so the
// others are running or done; should one not answer in time (another program's kernels hold the compute units), the
// waiting workgroup computes that piece's sums itself, from memory and with the same operations, and gets the same
// numbers. That needs the inputs intact: calls that write over their input take the other kernels.
#pragma once

constexpr int kTeamLanes = 512;
constexpr int kTeamWaves = kTeamLanes / dev::kWave;
constexpr int kTeamMax = 256;            // pieces of a channel
constexpr int kTeamChannels = 2048;      // a call has at most

// The scratch: per channel two slots a piece, on cache lines of the channel's own.
__host__ __device__ constexpr size_t teamStride(int pieces) { return (pieces * 16 + 127) / 128 * 128; }
struct TeamArgs {
  char *block;
  __device__ unsigned long *slots(int ch) const { return reinterpret_cast<unsigned long *>(block + ch * teamStride(pieces)); }
  unsigned tag;
  int pieces, units;                     // of a channel; units of a piece
  int spin;                              // polls before a workgroup helps itself
  int N, C, L;
};

// Walks the units base + lane, base + lane + kTeamLanes, ... of a channel (numbered n-major over its N planes of L / V units)
// as byte offsets from the channel's first plane; cf. ResWalker.
template <int V>
struct TeamWalker {
  int off, l, stepOff, stepL, Lu, wrapOff;
  __device__ TeamWalker(const TeamArgs &a, int base) : Lu(a.L / V) {
    int i = base + (int)threadIdx.x;
    __asm__ volatile("" : "+v"(i));      // every walk derives its offsets anew instead of keeping a register per step
    const int n = i / Lu;
    l = i - n * Lu;
    const int stepN = kTeamLanes / Lu;
    stepL = kTeamLanes - stepN * Lu;
    off = (n * a.C * a.L + l * V) * 4;
    stepOff = (stepN * a.C * a.L + stepL * V) * 4;
    wrapOff = (a.C * a.L - a.L) * 4;
  }
  __device__ void next() {
    off += stepOff, l += stepL;
    if (l >= Lu) l -= Lu, off += wrapOff;
  }
};

template <int V>
struct TeamUnit {
  float v[V];
};
template <int V>
__device__ __forceinline__ TeamUnit<V> teamLoad(__amdgpu_buffer_rsrc_t r, int off) {
  TeamUnit<V> u;
  if constexpr (V == 4) {
    const float4 q = dev::bufLoadStream4(r, off);
    u.v[0] = q.x, u.v[1] = q.y, u.v[2] = q.z, u.v[3] = q.w;
  } else {
    u.v[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 2));
  }
  return u;
}
template <int V>
__device__ __forceinline__ void teamStore(__amdgpu_buffer_rsrc_t r, int off, const TeamUnit<V> &u) {
  if constexpr (V == 4)
    dev::bufStoreStream4(r, off, make_float4(u.v[0], u.v[1], u.v[2], u.v[3]));
  else
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(u.v[0]), r, off, 0, 2);
}

__device__ __forceinline__ float teamSum(float v, float *red) {
  const int lane = threadIdx.x % dev::kWave, wave = threadIdx.x / dev::kWave;
  v = dev::waveSum(v);
  __syncthreads();                       // red may still be read from a previous reduction
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < kTeamWaves; w += 4) s += (red[w] + red[w + 1]) + (red[w + 2] + red[w + 3]);
  return s;
}

struct TeamShared {
  float red[kTeamWaves];
  float stat[kTeamMax][2];
  double out[2];
};

// Publishes (a, b) of piece `piece` and gathers those of all pieces into sh.stat. Returns false when some have not
// come in time: their entries in sh.stat are marked by bit k of `missing`.
__device__ __forceinline__ bool teamExchange(const TeamArgs &t, int ch, int piece, float a, float b, TeamShared &sh, unsigned *missing) {
  if (t.pieces == 1) {
    if (threadIdx.x == 0) sh.stat[0][0] = a, sh.stat[0][1] = b;
    __syncthreads();
    return true;
  }
  unsigned long *slot = t.slots(ch);
  const int k = threadIdx.x;
  const unsigned tag = t.tag;
  if (k < kTeamMax / 32) missing[k] = 0;
  if (k == 0) {
    __hip_atomic_store(slot + 2 * piece, (unsigned long)tag << 32 | __float_as_uint(a), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(slot + 2 * piece + 1, (unsigned long)tag << 32 | __float_as_uint(b), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  bool late = false;
  if (k < t.pieces) {
    float v0 = a, v1 = b;
    if (k != piece) {
      for (int s = 0;; ++s) {
        const unsigned long p = __hip_atomic_load(slot + 2 * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long q = __hip_atomic_load(slot + 2 * k + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((unsigned)(p >> 32) == tag && (unsigned)(q >> 32) == tag) {
          v0 = __uint_as_float((unsigned)p), v1 = __uint_as_float((unsigned)q);
          break;
        }
        if (s >= t.spin) {
          late = true;
          atomicOr(&missing[k >> 5], 1u << (k & 31));
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    sh.stat[k][0] = v0, sh.stat[k][1] = v1;
  }
  return __syncthreads_or(late) == 0;
}

// The backward pass: pieces of up to kTeamLanes * R units of V floats, R per lane, x and gradOutput of each.
template <int V, int R>
__global__ void __launch_bounds__(kTeamLanes, 4)
bnBwdTeam(const float *__restrict__ x, const float *__restrict__ gy, float *__restrict__ gx, float *__restrict__ gradWeight,
          float *__restrict__ gradBias, const float *__restrict__ weight, const float *__restrict__ meanSrc,
          const float *__restrict__ stdSrc, TeamArgs t, float scale, ReluMask rm) {
  __shared__ TeamShared sh;
  __shared__ unsigned missing[kTeamMax / 32];
  const int ch = blockIdx.x / t.pieces, piece = blockIdx.x - ch * t.pieces;
  const float mean = meanSrc[ch], stdVal = stdSrc[ch], weightVal = weight ? weight[ch] : 1.f;
  const ChannelMask m(rm, ch, mean);
  const int total = t.N * (t.L / V);
  const long span = ((long)(t.N - 1) * t.C * t.L + t.L) * 4;
  const __amdgpu_buffer_rsrc_t xr = dev::makeRsrc(x + (long)ch * t.L, span), gr = dev::makeRsrc(gy + (long)ch * t.L, span);
  const __amdgpu_buffer_rsrc_t or_ = dev::makeRsrc(gx ? gx + (long)ch * t.L : x, gx ? span : 0);  // no gx: nothing is stored
  TeamUnit<V> d[R], q[R];
  auto load = [&](int k) {
    TeamWalker<V> wk(t, k * t.units);
    const int n = min(t.units, total - k * t.units);
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int off = u * kTeamLanes + (int)threadIdx.x < n ? wk.off : dev::kBufOob;
      d[u] = teamLoad<V>(gr, off);
      q[u] = teamLoad<V>(xr, off);
      wk.next();
    }
  };
  // (units past the piece have d == 0)
  auto statistics = [&](float &s0, float &s1) {
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int u = 0; u < R; ++u)
#pragma unroll
      for (int e = 0; e < V; ++e) {
        d[u].v[e] = m.apply(d[u].v[e], q[u].v[e]);
        a += d[u].v[e];
        b += d[u].v[e] * (q[u].v[e] - mean);
      }
    s0 = teamSum(a, sh.red), s1 = teamSum(b, sh.red);
  };
  load(piece);
  float s0, s1;
  statistics(s0, s1);
  int late = !teamExchange(t, ch, piece, s0, s1, sh, missing);
  // (opaque: compiled into two copies, with and without an exchange, the kernel keeps x and gradOutput twice and spills)
  asm volatile("" : "+v"(late));
  if (__builtin_amdgcn_readfirstlane(late)) {
#pragma unroll 1
    for (int k = 0; k < t.pieces; ++k)
      if (missing[k >> 5] >> (k & 31) & 1) {
        load(k);
        statistics(s0, s1);
        if (threadIdx.x == 0) sh.stat[k][0] = s0, sh.stat[k][1] = s1;
      }
    load(piece);
#pragma unroll
    for (int u = 0; u < R; ++u)
#pragma unroll
      for (int e = 0; e < V; ++e) d[u].v[e] = m.apply(d[u].v[e], q[u].v[e]);
    __syncthreads();
  }
  if (threadIdx.x < dev::kWave) {
    double a = 0.0, b = 0.0;
    for (int k = threadIdx.x; k < t.pieces; k += dev::kWave) a += sh.stat[k][0], b += sh.stat[k][1];
#pragma unroll
    for (int o = 1; o < dev::kWave; o <<= 1) a += __shfl_xor(a, o), b += __shfl_xor(b, o);
    if (threadIdx.x == 0) sh.out[0] = a, sh.out[1] = b;
  }
  __syncthreads();
  // lib/THCUNN/BatchNormalization.cu:253-282
  const float gradOutputSum = (float)sh.out[0], dotP = (float)sh.out[1], norm = 1.f / ((float)t.N * (float)t.L);
  const float gradMean = gradOutputSum * norm, projScale = dotP * norm * stdVal * stdVal, gradScale = stdVal * weightVal;
  TeamWalker<V> wk(t, piece * t.units);
  const int n = min(t.units, total - piece * t.units);
#pragma unroll
  for (int u = 0; u < R; ++u) {
#pragma unroll
    for (int e = 0; e < V; ++e) d[u].v[e] = (d[u].v[e] - (q[u].v[e] - mean) * projScale - gradMean) * gradScale;
    teamStore<V>(or_, u * kTeamLanes + (int)threadIdx.x < n ? wk.off : dev::kBufOob, d[u]);
    wk.next();
  }
  if (piece == 0 && threadIdx.x == 0) {
    if (gradWeight) gradWeight[ch] += scale * dotP * stdVal;
    if (gradBias) gradBias[ch] += scale * gradOutputSum;
  }
}
