// Fixed-coefficient LUT/Clenshaw forward for gfx950 as a single-pass scan:
// x_norm, tanh_y, the clamped EMA and its final state.
//
// Reference counterpart: _fused_clenshaw_ema_kernel (sdpc_kernel.py:988-1209),
// the arithmetic of which stands at osm_lut_fwd_args in include/osm.h.  Its
// state is clamped to [-1, 1] where it crosses a clamp_tile boundary.  Since
// |tanh_y| < 1, a state inside [-1, 1] stays there under 0 <= mu <= 1, so only
// the first boundary can bind (through ema_init); after it the EMA is affine.
// The tiles are chained by the look-back of osm_chain.h; the tile that holds
// the first boundary publishes its state, clamped there, as a checkpoint, and
// the tiles after it start their group from it.
//
// What bounds it: at large sizes HBM (16 bytes per element: 118 us at B=4
// S=16384 D=512, 4.6 TB/s; the one-workgroup-per-lanes walk of osm_v10.hip
// 234 us), at small ones the VALU work of one tile on one CU (65
// instructions per element) and the launch: 15.5 against 51.4 us at B=2
// S=4096 D=512, 8.0 against 8.7 at B=1 S=384.  The table gathers cost little
// (15.1 us at B=2 S=4096 with the Clenshaw series in their place).
#include "osm_tile.h"
#include "osm_v10_math.h"

namespace osm {
namespace {

// Smallest decay kept for a run or tile: an infinite ema_init stays infinite
// up to the first clamp, as a token-by-token EMA keeps it, where an underflow
// to 0 would make it NaN.  Finite states do not notice 2^-149.
constexpr float kTinyDecay = 1.401298464324817e-45f;

// The clamp of a state; NaN (a look-back wait gave up) stays NaN.
__device__ __forceinline__ float clamp_state(float s) {
  return s == s ? __builtin_amdgcn_fmed3f(s, -1.0f, 1.0f) : s;
}

template <class G, typename XT, int KP, bool LUT, bool SPREAD>
__global__ void __launch_bounds__(G::THREADS) __attribute__((amdgpu_waves_per_eu(4)))
lut_fwd_kernel(const LutScanParams p) {
  constexpr int R = G::R, LPT = G::LPT;
  static_assert(G::LANES == kLanes && 16 % R == 0, "a clamp boundary (a multiple of 16) falls between runs");
  static_assert(G::THREADS >= KP * kLanes, "one thread per coefficient and lane");
  __shared__ ChainLds<G> L;
  __shared__ __attribute__((aligned(16))) float lut[LUT ? 256 : 1][kLutStride];
  __shared__ float cs[KP][kLanes];

  const ThreadPos q = thread_pos<G>();
  const Tags tags = launch_tags(p.hdr);
  TileInfo ti = tile_info<G, SPREAD>(p.order, p.hdr, p.n_lb, p.n_lbd, p.n_tiles, p.wsh);
  if (SPREAD && ti.pad) {
    skip_block(p.hdr, tags, ti);
    return;
  }
  const int t_tile = ti.tile * G::TILE;
  const int d0 = ti.lbd * kLanes + q.lt * LPT;
  const bool lane_ok = d0 < p.D;
  auto head_of = [&](int d) { return (int)((__umulhi((uint32_t)d, p.hd_magic) + (uint32_t)d) >> p.hd_shift); };

  // The table and the coefficients (one value per thread), then the rows.
  if constexpr (LUT) {
    for (int i = q.tid; i < KP * 256; i += G::THREADS) lut[i % 256][i / 256] = p.lut[i];
  }
  {
    const int k = q.tid / kLanes, d = ti.lbd * kLanes + q.tid % kLanes;
    if (k < KP) {
      const int h = d < p.D ? head_of(d) : 0;
      cs[k][q.tid % kLanes] = d < p.D && k < p.K ? p.coeffs[(int64_t)ti.b * p.c_sb + (int64_t)h * p.c_sh +
                                                            (int64_t)k * p.c_sk + (d - h * p.hd)]
                                                 : 0.0f;
    }
  }
  auto rows = [&](const void* base, int64_t sb, int64_t ss, int64_t elem) {
    const char* b = static_cast<const char*>(base) + ((int64_t)ti.b * sb + (int64_t)t_tile * ss) * elem;
    return make_rsrc(b, base ? ((uint64_t)(p.S - 1 - t_tile) * ss + p.D) * elem : 0);   // no buffer: stores dropped
  };
  auto lane_off = [&](int64_t ss, int64_t elem) {
    return lane_ok ? (uint32_t)(((int64_t)q.tg * R * ss + d0) * elem) : kOffOOB;
  };
  float w[R][LPT];
  {
    const Rsrc xr = rows(p.x, p.x_sb, p.x_ss, sizeof(XT));
    const uint32_t vx = lane_off(p.x_ss, sizeof(XT)), sx = (uint32_t)(p.x_ss * sizeof(XT));
    uint32_t so = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      BufVec<XT, LPT>::load(xr, vx, so, w[r]);
      so = next_off(so, sx);
    }
  }
  const float gamma = 0.98f - 0.06f * (float)(lane_ok ? head_of(d0) : 0) / (float)p.H;
  const float mu = p.mu, one_m = 1.0f - mu;
  __syncthreads();
  float c[LPT][KP];
#pragma unroll
  for (int k = 0; k < KP; ++k)
#pragma unroll
    for (int i = 0; i < LPT; ++i) c[i][k] = cs[k][q.lt * LPT + i];

  // Pass 1: x_norm and tanh_y stored, w = (1 - mu) tanh_y in place of x, the
  // run's aggregate from a zero state.
  float Bv[LPT];
#pragma unroll
  for (int i = 0; i < LPT; ++i) Bv[i] = 0.0f;
  {
    const Rsrc nr = rows(p.xnorm, p.xn_sb, p.xn_ss, 4), yr = rows(p.tanhy, p.ty_sb, p.ty_ss, 4);
    const uint32_t vn = lane_off(p.xn_ss, 4), vy = lane_off(p.ty_ss, 4);
    const uint32_t sn = (uint32_t)(p.xn_ss * 4), sy = (uint32_t)(p.ty_ss * 4);
    uint32_t on = 0, oy = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float u[LPT], z[LPT];
#pragma unroll
      for (int i = 0; i < LPT; ++i) {
        const float x = w[r][i];
        float absu, sgn;
        v10_softsign(x, absu, sgn);
        u[i] = sgn * absu;
        float y;
        if constexpr (LUT) {
          const float fidx = absu * 255.0f;
          const int i0 = min((int)fidx, 254);
          const float fr = __builtin_fminf(__builtin_fmaxf(fidx - (float)i0, 0.0f), 1.0f);
          const f32x4* ra = reinterpret_cast<const f32x4*>(&lut[i0][0]);
          const f32x4* rb = reinterpret_cast<const f32x4*>(&lut[i0 + 1][0]);
          // the series at both table points, then one interpolation
          float ae = 0.0f, ao = 0.0f, be = 0.0f, bo = 0.0f;
#pragma unroll
          for (int k4 = 0; k4 < KP / 4; ++k4) {
            const f32x4 ta = ra[k4], tb = rb[k4];
#pragma unroll
            for (int k = 0; k < 4; k += 2) {
              ae = __builtin_fmaf(c[i][4 * k4 + k], ta[k], ae);
              ao = __builtin_fmaf(c[i][4 * k4 + k + 1], ta[k + 1], ao);
              be = __builtin_fmaf(c[i][4 * k4 + k], tb[k], be);
              bo = __builtin_fmaf(c[i][4 * k4 + k + 1], tb[k + 1], bo);
            }
          }
          const float ya = __builtin_fmaf(sgn, ao, ae), yb = __builtin_fmaf(sgn, bo, be);
          y = __builtin_fmaf(fr, yb - ya, ya);
        } else {
          // b_k = 2u b_{k+1} - b_{k+2} + c_k, y = u b_1 - b_2 + c_0
          const float u2 = u[i] + u[i];
          float b1 = c[i][KP - 1], b2 = 0.0f;
#pragma unroll
          for (int k = KP - 2; k >= 1; --k) {
            const float b0 = __builtin_fmaf(u2, b1, c[i][k]) - b2;
            b2 = b1;
            b1 = b0;
          }
          y = __builtin_fmaf(u[i], b1, c[i][0]) - b2;
        }
        const float yc = __builtin_amdgcn_fmed3f(gamma * y, -4.0f, 4.0f);
        const float e2 = __builtin_amdgcn_exp2f(2.0f * kLog2e * yc);
        z[i] = (e2 - 1.0f) * __builtin_amdgcn_rcpf(e2 + 1.0f);
        z[i] = x == x ? z[i] : 0.0f;
        w[r][i] = one_m * z[i];
        Bv[i] = __builtin_fmaf(mu, Bv[i], w[r][i]);
      }
      BufVec<float, LPT>::store(nr, vn, on, u);
      BufVec<float, LPT>::store(yr, vy, oy, z);
      on = next_off(on, sn);
      oy = next_off(oy, sy);
    }
  }
  const unsigned fin_prev = finish_issue(p.hdr, tags.epoch);

  // Chain.  The first clamp boundary (after token clamp_tile - 1) lies in, or
  // at the end of, tile p.clamp_at.
  const LaneSlots ls = lane_slots<G, false>(p.slots, ti, p.n_tiles);
  const bool at_clamp = ti.tile == p.clamp_at;
  const int g_clamp = at_clamp ? (p.clamp_tile - t_tile) / R - 1 : -1;   // the run before the boundary
  const bool ckpt = ti.is_ckpt;
  ti.is_ckpt = ckpt || at_clamp;
  float pA, pB[LPT], aggA, aggB;
  jitter(p.jitter, tags.epoch, 0);
  const float run_A = __builtin_fmaxf(pow_n<R>(mu), kTinyDecay);
  tile_scan<G, false>(L, q, ti, tags, run_A, Bv, pA, pB, aggA, aggB, ls);
  {
    const int dc = ti.lbd * kLanes + carry_lane<G>(q);
    // (past the first clamp no tile uses it.)  A NaN state gives -1 from every
    // clamp, as -inf does, which stands for it here: a NaN carry then comes
    // only from a look-back wait that gave up.
    float init_c = 0.0f;
    if (p.ema_init && ti.tile <= p.clamp_at && q.wave == 0 && dc < p.D) {
      init_c = p.ema_init[(int64_t)ti.b * p.init_sb + dc];
      init_c = init_c == init_c ? init_c : -__builtin_inff();
    }
    const double tile_A64 = __builtin_fmax(pow_n_f64<G::TILE>((double)mu), (double)kTinyDecay);
    const float tile_A = (float)tile_A64;
    LookBack<G, false> lbk;
    look_back_issue<G, false>(lbk, q, ti, ls, p.wsh, ti.tile > p.clamp_at ? p.clamp_at + 1 : 0);
    ti.is_ckpt = ckpt && !at_clamp;   // the clamped tile's state is published below
    jitter(p.jitter, tags.epoch, 1);
    look_back_finish<G, false, false>(lbk, L, q, ti, tags, tile_A, aggB, ls, init_c, tile_A64, p.hdr, p.poll_limit,
                               kTinyDecay);
  }
  finish_complete<SPREAD>(p.hdr, tags.epoch, fin_prev);
  if (at_clamp && !ti.is_last && q.wave == 0) {
    float s = L.carry[q.wl];
    for (int g = 0; g < G::NTG; ++g) {
      s = __builtin_fmaf(L.A[g][q.wl / LPT], s, L.B[g][q.wl]);
      if (g == g_clamp) s = clamp_state(s);
    }
    publish(ls.at(ti.tile, q.wl), tags.pre, s);
  }

  // Pass 2.  Up to the first boundary a run starts from the earlier runs'
  // maps applied one after the other, with the clamp between them.
  float s[LPT];
  bool lost = false;
  if (ti.tile <= p.clamp_at) {
#pragma unroll
    for (int i = 0; i < LPT; ++i) s[i] = L.carry[q.lt * LPT + i];
    for (int g = 0; g < q.tg; ++g)
#pragma unroll
      for (int i = 0; i < LPT; ++i) {
        s[i] = __builtin_fmaf(L.A[g][q.lt], s[i], L.B[g][q.lt * LPT + i]);
        if (g == g_clamp) s[i] = clamp_state(s[i]);
      }
  } else {
#pragma unroll
    for (int i = 0; i < LPT; ++i) s[i] = __builtin_fmaf(pA, L.carry[q.lt * LPT + i], pB[i]);
  }
#pragma unroll
  for (int i = 0; i < LPT; ++i) lost |= s[i] != s[i];
  const Rsrc orr = rows(p.out, p.o_sb, p.o_ss, 4);
  const uint32_t vo = lane_off(p.o_ss, 4), so_step = (uint32_t)(p.o_ss * 4);
  const int r_last = p.S - 1 - (t_tile + q.tg * R);
  float* fin = ti.is_last && p.ema_final && lane_ok && r_last >= 0 && r_last < R
                   ? p.ema_final + (int64_t)ti.b * p.final_sb + d0
                   : nullptr;
  auto replay = [&](auto nan_c) {
    uint32_t so = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float o[LPT];
#pragma unroll
      for (int i = 0; i < LPT; ++i) {
        s[i] = __builtin_fmaf(mu, s[i], w[r][i]);
        o[i] = decltype(nan_c)::value ? clamp_state(s[i]) : __builtin_amdgcn_fmed3f(s[i], -1.0f, 1.0f);
      }
      BufVec<float, LPT>::store(orr, vo, so, o);
      so = next_off(so, so_step);
      if (fin && r == r_last) {
#pragma unroll
        for (int i = 0; i < LPT; ++i) fin[i] = o[i];
      }
    }
  };
  if (lost)
    replay(std::true_type{});
  else
    replay(std::false_type{});
}

template <class G, typename XT, bool LUT, int KP>
hipError_t launch_kp(const LutScanParams& p, hipStream_t stream) {
  with_order(p.order, [&](auto spread) {
    hipLaunchKernelGGL((lut_fwd_kernel<G, XT, KP, LUT, decltype(spread)::value>), dim3(p.order.grid),
                       dim3(G::THREADS), 0, stream, p);
  });
  return hipGetLastError();
}

template <class G, typename XT, bool LUT>
hipError_t launch_g(const LutScanParams& p, int kpad, hipStream_t stream) {
  return kpad == 4 ? launch_kp<G, XT, LUT, 4>(p, stream) : launch_kp<G, XT, LUT, 8>(p, stream);
}

template <typename XT, bool LUT>
hipError_t launch_x(const LutScanParams& p, FwdShape s, int kpad, hipStream_t stream) {
  if (s.lpt == 2)
    return s.tile == LutTile::TILE ? launch_g<LutTile, XT, LUT>(p, kpad, stream)
                                   : launch_g<LutTileSmall, XT, LUT>(p, kpad, stream);
  return s.tile == LutTileGeneric::TILE ? launch_g<LutTileGeneric, XT, LUT>(p, kpad, stream)
                                        : launch_g<LutTileGenericSmall, XT, LUT>(p, kpad, stream);
}

}  // namespace

hipError_t launch_lut_scan(const LutScanParams& p, int x_dtype, bool use_lut, FwdShape s, int kpad,
                           hipStream_t stream) {
  if (x_dtype == 0)
    return use_lut ? launch_x<float, true>(p, s, kpad, stream) : launch_x<float, false>(p, s, kpad, stream);
  return use_lut ? launch_x<__bf16, true>(p, s, kpad, stream) : launch_x<__bf16, false>(p, s, kpad, stream);
}

}  // namespace osm
