// Backward of the full path for gfx950: dL/dx of every chunk in one launch.
//
// Reference counterpart: FusedChebyRKVv10.backward (sdpc_kernel.py:2436-2515)
// on every chunk of the chunk loop (2574-2606).  Per lane, tokens t of a
// chunk [t0, t1) whose coefficients were c:
//   a[t]     = m[t] (dL/dout[t] + mu a[t+1]),  a = 0 past the chunk,
//              m[t] = [|out[t]| < 1 - 1e-6] on the saved output
//   dL/dx[t] = (1 - mu) a[t] gamma_h (1 - z[t]^2) sum_k k c_k U_{k-1}(u[t]) / (1 + |x[t]|)^2
// with z the forward's saved bf16 z.
//
// The adjoint restarts at every chunk end, so a chunk of a lane-block is one
// workgroup and nothing passes between workgroups: no look-back, no
// workspace.  A workgroup walks its chunk from the end in blocks of G::TILE
// tokens (one block when the chunk fits, the usual case: 256 of 256).
// Thread (token group, lane pair) holds a run of G::R tokens: pass 1 forms
// the run's map of v[t] = mu a[t] (A per lane, as a mask cuts it), the runs
// after it are composed from LDS, pass 2 replays from the true v.
//
// What bounds it: HBM, 18 bytes per element in fp32 (x, dL/dout, out, z
// read, dL/dx written): 5.1 TB/s at B=4 S=4096 D=512, 5.5 at B=8 S=8192, where
// a plain copy reaches 5.0-5.2.  The general backward on chunks as batch rows
// (192-token tiles, so a 256-token chunk left two thirds of its second tile
// empty) took 35 us at the first, plus the copies that laid the rows out.
#include "osm_device.h"

namespace osm {
namespace {

constexpr float kMaskBound = 0.999999f;   // 1 - 1e-6 rounded to fp32, as the reference compares in fp32

// 16 waves on 64 lanes, LPT adjacent lanes per thread, runs of R tokens:
// TILE = 16 LPT R tokens per block.  One workgroup of 1024 threads per CU
// with 16 elements per thread in flight: 29.3 us at B=4 S=4096 D=512 fp32 and
// 110 us at B=8 S=8192, against 35.7 and 132 with 8 waves and twice the run,
// 31.8 and 122 with 8 waves on 32 lanes, 45.8 and 207 at 64 VGPRs (two
// workgroups per CU: every row load waits for the one before).
template <int LPT_, int R_>
struct ChunkGeo {
  static constexpr int LPT = LPT_, R = R_, WAVES = 16, LANES = 64;
  static constexpr int THREADS = WAVES * 64;
  static constexpr int TPR = LANES / LPT;        // threads per row
  static constexpr int NTG = THREADS / TPR;      // token groups (runs) per block
  static constexpr int TILE = NTG * R;
};

struct Rows {
  Rsrc r;
  uint32_t v, s;   // this thread's byte offset, bytes per token
};

// Rows t_blk .. t_end - 1 of a [B,S,D] tensor: stores past t_end are dropped
// and nothing past the last row is read.  A read of a token past t_end gives 0
// where rows lie D or more apart; rows that share memory (dL/dout of a sum
// over tokens has stride 0) give values of earlier tokens there.
template <class G, typename T>
__device__ __forceinline__ Rows chunk_rows(const void* base, int64_t sb, int64_t ss, int b, int t_blk, int t_end,
                                           int D, int tg, int d0) {
  Rows w;
  const char* p = static_cast<const char*>(base) + ((int64_t)b * sb + (int64_t)t_blk * ss) * (int64_t)sizeof(T);
  w.r = make_rsrc(p, ((uint64_t)(t_end - 1 - t_blk) * ss + D) * sizeof(T));
  w.s = (uint32_t)(ss * sizeof(T));
  w.v = d0 < D ? (uint32_t)(((int64_t)tg * G::R * ss + d0) * sizeof(T)) : kOffOOB;
  return w;
}

template <class G, typename T>
__device__ __forceinline__ void load_run(float (&dst)[G::R][G::LPT], const Rows& w) {
  uint32_t so = 0;
#pragma unroll
  for (int r = 0; r < G::R; ++r) {
    BufVec<T, G::LPT>::load(w.r, w.v, so, dst[r]);
    so += w.s;
    asm volatile("" : "+s"(so));   // one SGPR for the offset, not one per row
  }
}

// The saved z of a run, as loaded (two bf16 values, or one, per register).
template <class G>
struct ZRun {
  unsigned q[G::R];
  __device__ __forceinline__ void load(const Rows& w) {
    uint32_t so = 0;
#pragma unroll
    for (int r = 0; r < G::R; ++r) {
      if constexpr (G::LPT == 2)
        q[r] = __builtin_amdgcn_raw_buffer_load_b32(w.r, w.v, so, kNT);
      else
        q[r] = (unsigned)__builtin_amdgcn_raw_buffer_load_b16(w.r, w.v, so, kNT);
      so += w.s;
      asm volatile("" : "+s"(so));
    }
  }
  __device__ __forceinline__ float get(int r, int i) const {
    return __uint_as_float(i == 0 ? q[r] << 16 : q[r] & 0xffff0000u);
  }
};

// Pass 2 over a run, last token first, from v = mu a of the token after it.
// dm: the lane's derivative series (times gamma (1 - mu)): sum dm[j] u^j, or
// sum dm[j] U_j(u) with CHEB.  MASKED: mb bit r set cuts the chain at token r.
template <class G, typename XT, int KP, bool CHEB, bool MASKED>
__device__ __forceinline__ void chunk_pass2(float (&v)[G::LPT], const float (&xv)[G::R][G::LPT],
                                            const float (&gv)[G::R][G::LPT], const ZRun<G>& zv,
                                            const unsigned (&mb)[G::LPT], float mu,
                                            const float (&dm)[G::LPT][KP - 1], const Rows& gx) {
  uint32_t so = (uint32_t)(G::R - 1) * gx.s;
  asm volatile("" : "+s"(so));
#pragma unroll
  for (int r = G::R - 1; r >= 0; --r) {
    float o[G::LPT];
#pragma unroll
    for (int i = 0; i < G::LPT; ++i) {
      float a = gv[r][i] + v[i];
      if constexpr (MASKED) a = ((mb[i] >> r) & 1u) ? 0.0f : a;
      v[i] = mu * a;
      const float x = xv[r][i];
      const float ir = __builtin_amdgcn_rcpf(1.0f + __builtin_fabsf(x));
      const float u = __builtin_copysignf(1.0f - ir, x);
      const float z = zv.get(r, i);
      const float e = a * __builtin_fmaf(-z, z, 1.0f);
      o[i] = e * (CHEB ? clenshaw_u<KP - 1>(u, dm[i]) : horner<KP - 1>(u, dm[i])) * (ir * ir);
    }
    BufVec<XT, G::LPT>::store(gx.r, gx.v, so, o);
    if (r > 0) {
      so -= gx.s;
      asm volatile("" : "+s"(so));
    }
  }
}

// 4 waves per SIMD: at most 128 VGPRs.
template <class G, typename XT, int KP>
__global__ void __launch_bounds__(G::THREADS) __attribute__((amdgpu_waves_per_eu(4)))
v10_bwd_kernel(const V10BwdParams p) {
  constexpr int R = G::R, LPT = G::LPT, NTG = G::NTG, LANES = G::LANES;
  __shared__ float sA[NTG][LANES], sB[NTG][LANES];   // run maps v[run start] = A v[run end + 1] + B
  __shared__ float sdm[KP][LANES];                   // derivative series: row 0 unused
  __shared__ float carry[LANES];                     // v at the start of the block after this one
  __shared__ unsigned big[8];

  // Items (batch row, chunk, lane-block), lane-blocks fastest; the items of
  // one XCD (workgroups go to the 8 XCDs round-robin) are consecutive, so
  // lines that two lane-blocks share are read into one L2.
  const int item = (int)(blockIdx.x & 7u) * p.items_per_xcd + (int)(blockIdx.x >> 3);
  if (item >= p.n_items) return;
  const int lbd = item % p.n_lbd;
  const int row = item / p.n_lbd;
  const int ch = row % p.n_chunks, b = row / p.n_chunks;
  const int t0 = ch * p.chunk, t1 = t0 + min(p.chunk, p.S - t0);
  const int tid = threadIdx.x, lt = tid % G::TPR, tg = tid / G::TPR;
  const int d0 = lbd * LANES + lt * LPT;
  const float mu = p.mu_dev ? *p.mu_dev : p.mu;

  // Coefficient j of lane l: thread (j, l) loads c_j, c_{j+2}, .. here and
  // forms the derivative's coefficient after the bulk loads are issued.
  static_assert(G::THREADS >= KP * LANES, "one thread per coefficient and lane");
  const int cj = __builtin_amdgcn_readfirstlane(tid / LANES), cl = tid % LANES;
  const int cd = lbd * LANES + cl;
  float cm[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  float gamma = 0.0f;
  if (cj < KP && cd < p.D) {
    const int h = cd / p.hd;
    const float* c = p.hist + (((size_t)ch * p.B + b) * p.H + h) * p.K * p.hd + (cd - h * p.hd);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (cj + 2 * i < p.K) cm[i] = c[(size_t)(cj + 2 * i) * p.hd];
    gamma = 0.98f - 0.06f * (float)h / (float)p.H;
  }
  if (tid < LANES) carry[tid] = 0.0f;

  float dm[LPT][KP - 1];
  const int n_blk = (t1 - t0 + G::TILE - 1) / G::TILE;
  for (int blk = n_blk - 1; blk >= 0; --blk) {
    const int t_blk = t0 + blk * G::TILE;
    float gv[R][LPT], xv[R][LPT];
    ZRun<G> zv;
    unsigned mb[LPT];
    float A[LPT], Bv[LPT];
    bool masked = false;
    {
      float ov[R][LPT];
      load_run<G, float>(gv, chunk_rows<G, float>(p.gout, p.go_sb, p.go_ss, b, t_blk, t1, p.D, tg, d0));
      load_run<G, float>(ov, chunk_rows<G, float>(p.out, p.o_sb, p.o_ss, b, t_blk, t1, p.D, tg, d0));
      if (blk == n_blk - 1 && cj < KP) {
        double acc = 0.0;
        switch (cj) {
          case 0: acc = mono_coef<0>(cm); break;
          case 1: acc = mono_coef<1>(cm); break;
          case 2: acc = mono_coef<2>(cm); break;
          case 3: acc = mono_coef<3>(cm); break;
          case 4: acc = mono_coef<4>(cm); break;
          case 5: acc = mono_coef<5>(cm); break;
          case 6: acc = mono_coef<6>(cm); break;
          default: acc = mono_coef<7>(cm); break;
        }
        // kMonoBound's rule, on the monomial coefficients in exp2 units
        const bool over = __ballot(!(__builtin_fabs(acc * (double)(kTwoLog2e * gamma)) <= kMonoBound)) != 0;
        if (cl == 0) big[cj] = over ? 1u : 0u;
        sdm[cj][cl] = (float)((double)cj * acc * (double)gamma * (double)(1.0f - mu));
      }
      // The adjoint is 0 past the chunk's end: where rows of dL/dout share
      // memory, tokens there have read another's row.
      if (p.go_ss < p.D) {
        const int n_valid = t1 - (t_blk + tg * R);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int i = 0; i < LPT; ++i) gv[r][i] = r < n_valid ? gv[r][i] : 0.0f;
      }
      // Pass 1, last token first: the run's map.
#pragma unroll
      for (int i = 0; i < LPT; ++i) {
        mb[i] = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const bool cut = !(__builtin_fabsf(ov[r][i]) < kMaskBound);
          masked |= cut;
          mb[i] |= cut ? 1u << r : 0u;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      Bv[i] = 0.0f;
      A[i] = 1.0f;
    }
    if (!masked) {
#pragma unroll
      for (int r = R - 1; r >= 0; --r)
#pragma unroll
        for (int i = 0; i < LPT; ++i) {
          Bv[i] = mu * (gv[r][i] + Bv[i]);
          A[i] *= mu;
        }
    } else {
#pragma unroll
      for (int r = R - 1; r >= 0; --r)
#pragma unroll
        for (int i = 0; i < LPT; ++i) {
          const float m = ((mb[i] >> r) & 1u) ? 0.0f : mu;
          // (a select, not a product: a cut token's dL/dout may be infinite)
          Bv[i] = ((mb[i] >> r) & 1u) ? 0.0f : mu * (gv[r][i] + Bv[i]);
          A[i] *= m;
        }
    }
    asm volatile("" ::: "memory");   // x and z after the saved output's registers are free
    load_run<G, XT>(xv, chunk_rows<G, XT>(p.x, p.x_sb, p.x_ss, b, t_blk, t1, p.D, tg, d0));
    zv.load(chunk_rows<G, __bf16>(p.z, p.z_sb, p.z_ss, b, t_blk, t1, p.D, tg, d0));
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      sA[tg][lt * LPT + i] = A[i];
      sB[tg][lt * LPT + i] = Bv[i];
    }
    __syncthreads();
    float v[LPT];
#pragma unroll
    for (int i = 0; i < LPT; ++i) v[i] = carry[lt * LPT + i];
    for (int g = NTG - 1; g > tg; --g)
#pragma unroll
      for (int i = 0; i < LPT; ++i) v[i] = __builtin_fmaf(sA[g][lt * LPT + i], v[i], sB[g][lt * LPT + i]);
    if (blk == n_blk - 1) {
#pragma unroll
      for (int j = 1; j < KP; ++j)
#pragma unroll
        for (int i = 0; i < LPT; ++i) dm[i][j - 1] = sdm[j][lt * LPT + i];
    }
    unsigned any = 0;
#pragma unroll
    for (int j = 0; j < KP; ++j) any |= big[j];
    const bool cheb = __builtin_amdgcn_readfirstlane(any) != 0;
    if (cheb && blk == n_blk - 1) {
      // Second-kind coefficients j c_j (T_j' = j U_{j-1}) in place of the
      // monomial ones: large coefficients cancel in the monomial form.
      __syncthreads();
      if (cj < KP) sdm[cj][cl] = (float)((double)cj * (double)cm[0] * (double)gamma * (double)(1.0f - mu));
      __syncthreads();
#pragma unroll
      for (int j = 1; j < KP; ++j)
#pragma unroll
        for (int i = 0; i < LPT; ++i) dm[i][j - 1] = sdm[j][lt * LPT + i];
    }
    const Rows gx = chunk_rows<G, XT>(p.gx, p.gx_sb, p.gx_ss, b, t_blk, t1, p.D, tg, d0);
    if (cheb)
      chunk_pass2<G, XT, KP, true, true>(v, xv, gv, zv, mb, mu, dm, gx);
    else if (masked)
      chunk_pass2<G, XT, KP, false, true>(v, xv, gv, zv, mb, mu, dm, gx);
    else
      chunk_pass2<G, XT, KP, false, false>(v, xv, gv, zv, mb, mu, dm, gx);
    if (blk > 0) {
      __syncthreads();   // every read of the carry and the run maps is done
      if (tg == 0) {
#pragma unroll
        for (int i = 0; i < LPT; ++i) carry[lt * LPT + i] = v[i];
      }
      // (read after the next block's barrier)
    }
  }
}

template <class G, typename XT>
hipError_t launch_g(const V10BwdParams& p, int kpad, hipStream_t stream) {
  const dim3 grid((unsigned)p.items_per_xcd * 8u), block(G::THREADS);
  if (kpad == 4)
    hipLaunchKernelGGL((v10_bwd_kernel<G, XT, 4>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((v10_bwd_kernel<G, XT, 8>), grid, block, 0, stream, p);
  return hipGetLastError();
}

template <typename XT, int LPT>
hipError_t launch_x(const V10BwdParams& p, int kpad, hipStream_t stream) {
  // Shortest block that holds the chunk (longer chunks: 256-token blocks).
  if (p.chunk <= 64) return launch_g<ChunkGeo<LPT, 4 / LPT>, XT>(p, kpad, stream);
  if (p.chunk <= 128) return launch_g<ChunkGeo<LPT, 8 / LPT>, XT>(p, kpad, stream);
  return launch_g<ChunkGeo<LPT, 16 / LPT>, XT>(p, kpad, stream);
}

}  // namespace

int v10_bwd_lanes() { return ChunkGeo<2, 8>::LANES; }

hipError_t launch_v10_bwd(const V10BwdParams& p, int x_dtype, int lpt, int kpad, hipStream_t stream) {
  if (x_dtype == 0) return lpt == 2 ? launch_x<float, 2>(p, kpad, stream) : launch_x<float, 1>(p, kpad, stream);
  return lpt == 2 ? launch_x<__bf16, 2>(p, kpad, stream) : launch_x<__bf16, 1>(p, kpad, stream);
}

}  // namespace osm
