// The engine's steps ahead of its Chebyshev path, for inference on gfx950: the
// input RMSNorm with the mean of its result over the tokens, then the
// complexity gate of that mean and the EMA momentum schedule.
//
// Reference counterpart: sdpc_engine.py:163-209 (torch operations there).
//   xn[b,t,:] = x[b,t,:] / sqrt(mean_d x^2 + eps) * w
//   m[b,:]    = mean_t xn[b,t,:]
//   gate[b]   = sigmoid(W2 silu(W1 m + b1) + b2)       W1 [D/4, D], W2 [1, D/4]
//   tokens   += S;  mu = 0.7 + 0.5 (base - 0.7) (1 + cos(pi clamp(tokens / 1e8, 0, 1)))
//
// Two launches in place of about thirty torch operations, most of them a few
// elements each.  What bounds it: at short sequences the two launches; at
// long ones the norm's bytes (x read, xn written: the column sums ride along
// in registers, where a separate mean read xn again).
#include <algorithm>

#include "osm_device.h"

namespace osm {
namespace {

constexpr int kNormThreads = 512, kNormWaves = kNormThreads / 64;
constexpr int kGateThreads = 1024, kGateWaves = kGateThreads / 64;

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Block (tile, b): rows tile * rows .. of batch row b, one row per wave at a
// time, the next one in flight.  Lane l holds the NV float4 pieces l + 64 v of
// a row.  part[b][tile][d]: the tile's sums of xn over its rows, waves added
// in order.
template <int NV>
__global__ void __launch_bounds__(kNormThreads) engine_norm_kernel(const EngineParams p, int rows) {
  __shared__ f32x4 red[kNormWaves][NV * 64];
  const int tile = blockIdx.x, b = blockIdx.y, wave = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int n4 = p.D / 4;
  const f32x4* const w4 = reinterpret_cast<const f32x4*>(p.norm_w);
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 w[NV], sum[NV], cur[NV], nxt[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    w[v] = l + 64 * v < n4 ? w4[l + 64 * v] : zero;
    sum[v] = zero;
  }
  const int t0 = tile * rows, t1 = min(t0 + rows, p.S);
  auto load = [&](f32x4 (&r)[NV], int t) {
    const f32x4* src = reinterpret_cast<const f32x4*>(p.x + (int64_t)b * p.x_sb + (int64_t)t * p.x_ss);
#pragma unroll
    for (int v = 0; v < NV; ++v) r[v] = l + 64 * v < n4 ? src[l + 64 * v] : zero;
  };
  if (t0 + wave < t1) load(cur, t0 + wave);
  for (int t = t0 + wave; t < t1; t += kNormWaves) {
    if (t + kNormWaves < t1) load(nxt, t + kNormWaves);
    float ss = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i) ss = __builtin_fmaf(cur[v][i], cur[v][i], ss);
    const float rstd = rsqrtf(wave_sum(ss) / (float)p.D + p.eps);
    f32x4* dst = reinterpret_cast<f32x4*>(p.xn + ((int64_t)b * p.S + t) * p.D);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      f32x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = cur[v][i] * rstd * w[v][i];
      if (l + 64 * v < n4) dst[l + 64 * v] = o;
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[v][i] += o[i];
      cur[v] = nxt[v];
    }
  }
#pragma unroll
  for (int v = 0; v < NV; ++v) red[wave][l + 64 * v] = sum[v];
  __syncthreads();
  f32x4* part = reinterpret_cast<f32x4*>(p.part + ((int64_t)b * gridDim.x + tile) * p.D);
  for (int c = threadIdx.x; c < n4; c += kNormThreads) {
    f32x4 s = red[0][c];
#pragma unroll
    for (int q = 1; q < kNormWaves; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] += red[q][c][i];
    part[c] = s;
  }
}

// Block b: the mean of batch row b from its tiles' sums (in a fixed order),
// then the gate.  Block 0 also advances the token count and forms mu.
__global__ void __launch_bounds__(kGateThreads) engine_gate_kernel(const EngineParams p, int n_tiles) {
  __shared__ f32x4 red[kGateThreads];
  __shared__ f32x4 mean4[kEngineMaxD / 4];
  __shared__ float hid[kEngineMaxD / 4];
  const int b = blockIdx.x, tid = threadIdx.x, wave = tid >> 6, l = tid & 63;
  const int n4 = p.D / 4, hidden = p.D / 4;
  if (b == 0 && tid == 0) {
    const long long tokens = *p.tokens + p.S;
    *p.tokens = tokens;
    const float pr = __builtin_fminf(__builtin_fmaxf((float)tokens / 1e8f, 0.0f), 1.0f);
    *p.mu = 0.7f + 0.5f * (*p.ema_base - 0.7f) * (1.0f + cosf(pr * 3.14159265358979323846f));
  }
  // Thread (group g, piece c) adds tiles g, g + G, ..; then the groups in order.
  const f32x4* part = reinterpret_cast<const f32x4*>(p.part + (int64_t)b * n_tiles * p.D);
  const int G = min(kGateThreads / n4, 16), c = tid % n4, g = tid / n4;
  f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
  if (g < G) {
#pragma unroll 8
    for (int t = g; t < n_tiles; t += G) {
      const f32x4 v = part[(int64_t)t * n4 + c];
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] += v[i];
    }
  }
  red[tid] = s;
  __syncthreads();
  if (tid < n4) {
    for (int q = 1; q < G; ++q) {
      const f32x4 v = red[q * n4 + tid];
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] += v[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] /= (float)p.S;
    mean4[tid] = s;
  }
  __syncthreads();
  // Hidden units, four per wave at a time.
  constexpr int U = 4;
  for (int j0 = wave * U; j0 < hidden; j0 += kGateWaves * U) {
    float acc[U];
#pragma unroll
    for (int u = 0; u < U; ++u) acc[u] = 0.0f;
    for (int k = l; k < n4; k += 64) {
      const f32x4 m = mean4[k];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = min(j0 + u, hidden - 1);
        const f32x4 w = reinterpret_cast<const f32x4*>(p.w1 + (int64_t)j * p.D)[k];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[u] = __builtin_fmaf(w[i], m[i], acc[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) acc[u] = wave_sum(acc[u]);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (l == u && j0 + u < hidden) {
        const float a = acc[u] + p.b1[j0 + u];
        hid[j0 + u] = a / (1.0f + expf(-a));
      }
  }
  __syncthreads();
  if (wave == 0) {
    float a = 0.0f;
    for (int j = l; j < hidden; j += 64) a = __builtin_fmaf(p.w2[j], hid[j], a);
    a = wave_sum(a);
    if (l == 0) p.gate[b] = 1.0f / (1.0f + expf(-(a + p.b2[0])));
  }
}

template <int NV>
void launch_norm(const EngineParams& p, int n_tiles, int rows, hipStream_t stream) {
  hipLaunchKernelGGL((engine_norm_kernel<NV>), dim3(n_tiles, p.B), dim3(kNormThreads), 0, stream, p, rows);
}

}  // namespace

// Tiles of a batch row: up to 128, of at least one row per wave.  (64 left the
// norm short of workgroups at B = 1; with 256 the gate kernel's mean, one
// workgroup per batch row, grows longer than the norm.)
int engine_tiles(int64_t S) {
  const int64_t rows = std::max<int64_t>(kNormWaves, (S + 127) / 128);
  return (int)((S + rows - 1) / rows);
}

hipError_t launch_engine(const EngineParams& p, hipStream_t stream) {
  const int n_tiles = engine_tiles(p.S);
  const int rows = (p.S + n_tiles - 1) / n_tiles;
  if (p.D <= 256)
    launch_norm<1>(p, n_tiles, rows, stream);
  else if (p.D <= 512)
    launch_norm<2>(p, n_tiles, rows, stream);
  else
    launch_norm<4>(p, n_tiles, rows, stream);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(engine_gate_kernel, dim3(p.B), dim3(kGateThreads), 0, stream, p, n_tiles);
  return hipGetLastError();
}

}  // namespace osm
