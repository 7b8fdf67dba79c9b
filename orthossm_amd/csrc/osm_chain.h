// Tile chaining protocol shared by the fused kernels: tile assignment, the
// token-group scan inside a tile, and the single-pass checkpointed look-back
// that hands each tile its EMA carry-in.
//
// The EMA s[t] = lam[t] s[t-1] + w[t] composes as affine maps f(s) = A s + B.
// A tile's aggregate is (A, B) = composition over its tokens from a zero
// state.  Tiles are grouped in runs of G::CKPT; the carry into tile t of
// group m is
//     carry = f_{t-1}( ... f_{CKPT m}( C_m ) ... )
// where C_m is the state after tile CKPT m - 1 (the checkpoint, ema_init for
// m = 0).  Every tile publishes its aggregate except the last tile of a
// group, which publishes its inclusive state as the next checkpoint.  The
// composition order is fixed, so results do not depend on timing.
//
// A lane-block is G::LANES consecutive lanes of one batch row (64 or 128);
// the look-back works on 64-lane sub-blocks: sub-block sb is served by waves
// sb*WPS .. sb*WPS+WPS-1, each reading WPT predecessor tiles, so that
// CKPT = WPS * WPT (or, where a launch chooses, fewer words: WPS << wsh).
// Look-back words are laid out [lane-block][tile][lane].
//
// Tile order (tile_order, tile_info).  A tile waits on earlier tiles of its
// lane-block, and blocks that wait may fill every place that another launch's
// blocks need, on any XCD.  So an awaited block has to be running already
// whenever the waiting one is:
//   - by index over a multiple of 8 slots: workgroups go to the 8 XCDs
//     round-robin by index and in index order within an XCD, and the tiles of
//     a lane-block are on blocks of one residue mod 8, ascending: those
//     awaited were dispatched to the same XCD before.
//   - by ticket: a block draws its tile from its lane-block's counter when it
//     starts, so those awaited have started, whatever XCD they are on.
//   - with one tile nothing waits.
// (By index over several XCDs holds for one launch alone; two of them could
// wait for each other, each holding the XCD that the other needs.)  The waits
// are bounded (kSpinLimit), so a broken assumption surfaces as a fault flag,
// not a hang.
#pragma once

#include "osm_device.h"
#include "osm_kernels.h"

namespace osm {

template <class G>
struct ChainLds {
  float A[G::NTG][G::TPR];      // token-group aggregate A (one per thread)
  float B[G::NTG][G::LANES];    // token-group aggregate B per lane
  float mA[G::WAVES][kLanes];   // look-back partial maps per wave (lane of its sub-block)
  float mB[G::WAVES][kLanes];
  float carry[G::LANES];        // resolved carry-in of the tile
};

struct TileInfo {
  int tile, lb, b, lbd;
  bool is_last, is_ckpt;
  bool pad;   // no tile: a slot without a lane-block
};

struct Tags {
  unsigned epoch, agg, pre;
};

// Thread coordinates inside the workgroup: wave, lane in wave (wl), thread in
// its row (lt: lanes lt*LPT .. lt*LPT+LPT-1 of the lane-block) and token
// group (tg).
struct ThreadPos {
  int tid, wave, wl, lt, tg;
};

template <class G>
__device__ __forceinline__ ThreadPos thread_pos() {
  ThreadPos q;
  q.tid = threadIdx.x;
  q.wave = q.tid >> 6;
  q.wl = q.tid & 63;
  q.lt = q.wl % G::TPR;
  q.tg = q.wave * G::TGW + q.wl / G::TPR;
  return q;
}

// Lane (within the lane-block) whose look-back words this thread reads, and
// the lane whose carry it resolves (waves < NSUB only).
template <class G>
__device__ __forceinline__ int look_lane(const ThreadPos& q) {
  return (q.wave / G::WPS) * kLanes + q.wl;
}
template <class G>
__device__ __forceinline__ int carry_lane(const ThreadPos& q) {
  return q.wave * kLanes + q.wl;
}

// Launch epoch: constant for the whole launch (the last block bumps it only
// after every block of this launch has read it).
__device__ __forceinline__ Tags launch_tags(unsigned* hdr_words) {
  Tags t;
  t.epoch = __hip_atomic_load(hdr_words, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  t.agg = make_tag(t.epoch, kKindAgg);
  t.pre = make_tag(t.epoch, kKindPre);
  return t;
}

// log2 of the look-back words per thread when a kernel always uses G::WPT.
template <class G>
constexpr int kWordsShift = G::WPT == 1 ? 0 : (G::WPT == 2 ? 1 : (G::WPT == 4 ? 2 : 3));

// The block's tile.  wsh: log2 of the look-back words per thread of this
// launch (at most G::WPT words); checkpoints lie every WPS << wsh tiles.
template <class G, bool SPREAD>
__device__ __forceinline__ TileInfo tile_info(const TileOrder& order, unsigned* hdr_words, int n_lb, int n_lbd,
                                              int n_tiles, int wsh = kWordsShift<G>) {
  TileInfo ti;
  ti.pad = false;
  if constexpr (!SPREAD) {
    const int v = blockIdx.x;
    ti.tile = v / n_lb;
    ti.lb = slot_lane_block(v - ti.tile * n_lb, n_lb);
  } else {
    const TileSlot slot = spread_slot(order, blockIdx.x, n_lb, n_tiles);
    ti.tile = slot.tile;
    ti.lb = slot.lb;
    if (ti.tile < 0 && ti.lb >= 0) {
      __shared__ unsigned drawn;
      if (threadIdx.x == 0)
        drawn = __hip_atomic_fetch_add(&reinterpret_cast<WsHeader*>(hdr_words)->ticket[ti.lb & 7].next, 1u,
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      ti.tile = (int)__builtin_amdgcn_readfirstlane(drawn);
    }
    // (a drawn tile past the last: only where two launches share a workspace)
    ti.pad = ti.lb < 0 || (unsigned)ti.tile >= (unsigned)n_tiles;
  }
  ti.b = SPREAD ? (int)order.by_row.of((unsigned)ti.lb) : ti.lb / n_lbd;
  ti.lbd = ti.lb - ti.b * n_lbd;
  ti.is_last = ti.tile == n_tiles - 1;
  ti.is_ckpt = ((ti.tile + 1) & ((G::WPS << wsh) - 1)) == 0;
  if constexpr (SPREAD) ti.is_ckpt |= order.lead && ti.tile == 0;
  return ti;
}

// Look-back words of one lane-block: [tile][LANES][words].
struct LaneSlots {
  unsigned long long* base;   // tile 0, lane 0 of the lane-block
  size_t tile_stride;         // words per tile
  int words;                  // 1 (B) or 2 (B, A)
  __device__ __forceinline__ unsigned long long* at(int tile, int lane) const {
    return base + (size_t)tile * tile_stride + (size_t)lane * words;
  }
};

template <class G, bool DYN>
__device__ __forceinline__ LaneSlots lane_slots(unsigned long long* slots, const TileInfo& ti, int n_tiles) {
  LaneSlots s;
  s.words = DYN ? 2 : 1;
  s.tile_stride = (size_t)G::LANES * s.words;
  s.base = slots + (size_t)ti.lb * n_tiles * s.tile_stride;
  return s;
}

// Aggregate A of a full tile under a static lambda, lambda^TILE rounded once
// (the producing workgroup publishes only B and uses the same value for its
// checkpoint; an error in A would repeat at every tile of the carry chain).
template <class G>
__device__ __forceinline__ float static_tile_A(float lam) {
  return pow_n<G::TILE>(lam);
}

// Test aid (OSM_FLAG_TIMING_JITTER): the workgroup sleeps 0..15 x ~0.85 us,
// a hash of its index, the launch epoch and `site`, so tiles publish and
// combine in orders the normal schedule rarely produces.  Every wait of the
// look-back is on a word a predecessor publishes without waiting on later
// tiles, so a delay only postpones, and results must not change.
__device__ __forceinline__ void jitter(int on, unsigned epoch, unsigned site) {
  if (!on) return;
  unsigned h = (blockIdx.x * 0x9E3779B1u) ^ (epoch * 0x85EBCA77u) ^ (site * 0xC2B2AE3Du);
  h ^= h >> 15;
  h *= 0x2C1B3C6Du;
  h ^= h >> 12;
  const unsigned n = __builtin_amdgcn_readfirstlane(h & 15u);
  for (unsigned i = 0; i < n; ++i) __builtin_amdgcn_s_sleep(32);
}

// Token-group scan.  In: this thread's run aggregate (A, Bv).  Out: (pA, pB)
// mapping the tile carry to the state before this thread's first token; in
// waves < NSUB, (aggA, aggB) = the tile aggregate of carry_lane(q), which is
// published unless the tile is a checkpoint or the last tile.
template <class G, bool DYN>
__device__ __forceinline__ void tile_scan(ChainLds<G>& L, const ThreadPos& q, const TileInfo& ti, const Tags& tg,
                                          float A, const float (&Bv)[G::LPT], float& pA, float (&pB)[G::LPT],
                                          float& aggA, float& aggB, const LaneSlots& ls) {
  constexpr int LPT = G::LPT;
  L.A[q.tg][q.lt] = A;
#pragma unroll
  for (int i = 0; i < LPT; ++i) L.B[q.tg][q.lt * LPT + i] = Bv[i];
  __syncthreads();
  pA = 1.0f;
#pragma unroll
  for (int i = 0; i < LPT; ++i) pB[i] = 0.0f;
  for (int g = 0; g < q.tg; ++g) {
    const float a = L.A[g][q.lt];
#pragma unroll
    for (int i = 0; i < LPT; ++i) pB[i] = __builtin_fmaf(a, pB[i], L.B[g][q.lt * LPT + i]);
    pA *= a;
  }
  aggA = 1.0f;
  aggB = 0.0f;
  if (q.wave < G::NSUB) {
    const int cl = carry_lane<G>(q);
    for (int g = 0; g < G::NTG; ++g) {
      const float a = L.A[g][cl / LPT];
      aggB = __builtin_fmaf(a, aggB, L.B[g][cl]);
      aggA *= a;
    }
    if (!ti.is_ckpt && !ti.is_last) {
      unsigned long long* mine = ls.at(ti.tile, cl);
      if (DYN) publish(mine + 1, tg.agg, aggA);
      publish(mine, tg.agg, aggB);
    }
  }
}

// Look-back in two halves so that a caller can issue other loads in between:
// look_back_issue reads (without waiting) the words this thread needs;
// look_back_finish waits for the ones not yet published, combines, and
// leaves the carry-in of every lane in L.carry.  Thread (wave, wl) reads
// lane look_lane of WPT predecessor tiles; waves < NSUB also read the
// checkpoint of their carry lane.
template <class G, bool DYN>
struct LookBack {
  unsigned long long vB[G::WPT];
  unsigned long long vA[DYN ? G::WPT : 1];
  unsigned long long vck;
  int beg, end, g0;
};

template <class G, bool DYN>
__device__ __forceinline__ void look_back_issue(LookBack<G, DYN>& st, const ThreadPos& q, const TileInfo& ti,
                                                const LaneSlots& ls, int wsh = kWordsShift<G>, int g0_min = 0) {
  static_assert((G::WPS & (G::WPS - 1)) == 0 && (1 << kWordsShift<G>) == G::WPT, "checkpoint groups are powers of two");
  const int ll = look_lane<G>(q);
  // g0_min: first tile of the group when an extra checkpoint precedes it
  st.g0 = max(ti.tile & ~((G::WPS << wsh) - 1), g0_min);
  // (wave-uniform, so the tests on it below are scalar)
  st.beg = st.g0 + ((__builtin_amdgcn_readfirstlane(q.wave) % G::WPS) << wsh);
  st.end = min(st.beg + (1 << wsh), ti.tile);
#pragma unroll
  for (int i = 0; i < G::WPT; ++i) {
    if (st.beg + i >= st.end) break;
    const unsigned long long* s = ls.at(st.beg + i, ll);
    st.vB[i] = peek(s);
    if constexpr (DYN) st.vA[i] = peek(s + 1);
  }
  st.vck = 0;
  if (q.wave < G::NSUB && st.g0 > 0) st.vck = peek(ls.at(st.g0 - 1, carry_lane<G>(q)));
}

// `a_look` is the full-tile decay static_tile_A of look_lane's static lambda
// (unused when DYN); `init_carry` the initial state of carry_lane (waves <
// NSUB); `limit` the poll limit of await_word.  A wait that gives up yields
// NaN, so the carry (and a checkpoint published from it) is NaN.
// AL: the type in which a thread's words compose; double where a launch may
// choose several per thread (rounded once; in fp32 the longer composition
// raised the error of a long carry chain by half).
// LEAD: the first tile may be a checkpoint (TileOrder::lead).
template <class G, bool DYN, bool LEAD, typename AL>
__device__ __forceinline__ void look_back_finish(LookBack<G, DYN>& st, ChainLds<G>& L, const ThreadPos& q,
                                                 const TileInfo& ti, const Tags& tg, float aggA, float aggB,
                                                 const LaneSlots& ls, float init_carry, AL a_look,
                                                 unsigned* hdr_words, unsigned limit, float min_a = 0.0f) {
  if (ti.tile > 0) {
    const int ll = look_lane<G>(q);
    AL mA = 1, mB = 0;
    if (st.beg < st.end) {
      const AL Afull = DYN ? AL(1) : a_look;
#pragma unroll
      for (int i = 0; i < G::WPT; ++i) {
        if (st.beg + i >= st.end) break;
        const unsigned long long* s = ls.at(st.beg + i, ll);
        const float Bp = await_word(s, st.vB[i], tg.agg, hdr_words, limit);
        AL Ap = Afull;
        if constexpr (DYN) Ap = await_word(s + 1, st.vA[i], tg.agg, hdr_words, limit);
        if constexpr (std::is_same_v<AL, double>)
          mB = __builtin_fma(Ap, mB, (double)Bp);
        else
          mB = __builtin_fmaf(Ap, mB, Bp);
        mA *= Ap;
      }
    }
    // min_a > 0: a composed decay does not underflow to 0 (an infinite state
    // stays infinite)
    L.mA[q.wave][q.wl] = min_a > 0.0f ? __builtin_fmaxf((float)mA, min_a) : (float)mA;
    L.mB[q.wave][q.wl] = (float)mB;
    float ck = init_carry;
    if (q.wave < G::NSUB && st.g0 > 0)
      ck = await_word(ls.at(st.g0 - 1, carry_lane<G>(q)), st.vck, tg.pre, hdr_words, limit);
    __syncthreads();
    if (q.wave < G::NSUB) {
      const int w0 = q.wave * G::WPS;   // the waves that read this sub-block
      float carry = ck;
#pragma unroll
      for (int w = 0; w < G::WPS; ++w) carry = __builtin_fmaf(L.mA[w0 + w][q.wl], carry, L.mB[w0 + w][q.wl]);
      L.carry[carry_lane<G>(q)] = carry;
      if (ti.is_ckpt && !ti.is_last)
        publish(ls.at(ti.tile, carry_lane<G>(q)), tg.pre, __builtin_fmaf(aggA, carry, aggB));
    }
  } else if (q.wave < G::NSUB) {
    L.carry[carry_lane<G>(q)] = init_carry;
    if (LEAD && ti.is_ckpt && !ti.is_last)
      publish(ls.at(0, carry_lane<G>(q)), tg.pre, __builtin_fmaf(aggA, init_carry, aggB));
  }
  __syncthreads();
}

// Counting the blocks of a launch, in two halves: finish_issue counts this
// block (thread 0), finish_complete acts on the count.  The last block of its
// class resets the class counter; the last class bumps the epoch for the next
// launch.  Safe once this block's epoch read (launch_tags) has returned,
// which the increment's data dependency on the epoch enforces: blocks of
// this launch use the epoch they read at their start, so a bump while some
// of them still publish or wait changes nothing for them.  Split so that the
// counter's round trip overlaps the block's work and its result is read
// before the block's bulk stores (loads and stores share one wait counter, so
// reading it after them would wait for every store).
__device__ __forceinline__ unsigned finish_issue(unsigned* hdr_words, unsigned epoch) {
  unsigned prev = 0;
  if (threadIdx.x == 0) {
    WsHeader* hdr = reinterpret_cast<WsHeader*>(hdr_words);
    unsigned one = 1u;
    asm volatile("" : "+v"(one) : "v"(epoch));   // the count depends on the epoch value
    prev = __hip_atomic_fetch_add(&hdr->cls[blockIdx.x & 7u].done, one, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
  }
  return prev;
}

// (SPREAD: and the ticket counters, from which every block has drawn.)
template <bool SPREAD>
__device__ __forceinline__ void finish_complete(unsigned* hdr_words, unsigned epoch, unsigned prev) {
  if (threadIdx.x == 0) {
    WsHeader* hdr = reinterpret_cast<WsHeader*>(hdr_words);
    const unsigned cls = blockIdx.x & 7u;
    const unsigned cls_size = (gridDim.x - cls + 7u) >> 3;
    if (prev == cls_size - 1u) {
      __hip_atomic_store(&hdr->cls[cls].done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const unsigned n_cls = gridDim.x < 8u ? gridDim.x : 8u;
      const unsigned prev_all = __hip_atomic_fetch_add(&hdr->done_all, 1u, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT);
      if (prev_all == n_cls - 1u) {
        __hip_atomic_store(&hdr->done_all, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if constexpr (SPREAD) {
#pragma unroll 1
          for (int i = 0; i < 7; ++i)
            __hip_atomic_store(&hdr->ticket[i].next, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __hip_atomic_store(&hdr->epoch, epoch + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
}

// Both halves at once (blocks without a tile, and the end of a kernel).
template <bool SPREAD>
__device__ __forceinline__ void finish_block(unsigned* hdr_words, unsigned epoch) {
  finish_complete<SPREAD>(hdr_words, epoch, finish_issue(hdr_words, epoch));
}

// A block without a tile.  (Also one whose drawn tile is past the last, which
// takes another launch drawing from the same workspace: a fault of both.)
__device__ __forceinline__ void skip_block(unsigned* hdr_words, const Tags& tg, const TileInfo& ti) {
  if (ti.lb >= 0 && threadIdx.x == 0) raise_fault(hdr_words, fault_tag_of(tg.agg));
  finish_block<true>(hdr_words, tg.epoch);
}

// First tile of the look-back group of a tile after the first: its checkpoint
// is the tile before.
template <bool SPREAD>
__device__ __forceinline__ int group_min(const TileOrder& order, const TileInfo& ti) {
  return SPREAD && order.lead && ti.tile > 0 ? 1 : 0;
}

// Launches a kernel in the version of the launch's tile order: f gets
// std::true_type for a spread order.
template <class F>
void with_order(const TileOrder& o, F f) {
  if (o.spread)
    f(std::true_type{});
  else
    f(std::false_type{});
}

}  // namespace osm
