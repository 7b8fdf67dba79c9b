// Launch parameters, tile geometry and launcher declarations shared by the
// kernel files and the C-ABI layer.  No torch types.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <type_traits>

namespace osm {

// Largest padded coefficient count evaluated in monomial form.  Beyond it
// the monomial coefficients of T_k grow like 2^(k-1) and cancel in fp32, so
// longer series keep their Chebyshev coefficients and use Clenshaw.
constexpr int kMonoMaxK = 8;

// Tile geometry.  A lane-block is LANES (64 or 128) consecutive lanes of one
// batch row; a tile is TILE consecutive tokens of a lane-block and is one
// workgroup.  A thread owns LPT adjacent lanes and a run of R consecutive
// tokens; TPR threads cover the LANES lanes of a row, so one wave instruction
// reads or writes TGW rows x LANES*4 contiguous bytes (fp32).  Token groups
// (runs) are ordered wave-major: tg = wave * TGW + lane_in_wave / TPR.  The
// look-back serves each 64-lane sub-block with WPS waves of WPT words per
// thread, so tiles are grouped in checkpoint runs of WPS * WPT (see osm_chain.h).
template <int LPT_, int WAVES_, int R_, int LANES_ = 64, int WPT_ = 8>
struct TileGeo {
  static constexpr int LPT = LPT_;            // lanes per thread
  static constexpr int WAVES = WAVES_;        // waves per workgroup
  static constexpr int R = R_;                // tokens per thread run
  static constexpr int LANES = LANES_;        // lanes per lane-block
  static constexpr int THREADS = WAVES * 64;
  static constexpr int NSUB = LANES / 64;     // 64-lane look-back sub-blocks
  static constexpr int TPR = LANES / LPT;     // threads per row
  static constexpr int TGW = 64 / TPR;        // token groups per wave
  static constexpr int NTG = WAVES * TGW;     // token groups per tile
  static constexpr int TILE = NTG * R;        // tokens per tile
  static constexpr int WPS = WAVES / NSUB;    // look-back waves per sub-block
  static constexpr int WPT = WPT_;            // look-back words per thread
  static_assert(LANES % 64 == 0 && LANES % LPT == 0 && TPR <= 64 && 64 % TPR == 0, "geometry");
  static_assert(WAVES % NSUB == 0, "look-back waves");
};

// Forward: the run length sets the tile.  Longer runs amortise the per-tile
// scan and look-back over more tokens but give fewer workgroups, so the host
// takes the largest tile that still fills the chip (fwd_geometry).  Dynamic
// lambda keeps a per-token lambda in registers and is limited to the medium
// tile.  Measured on MI355X at B=4 S=16384 D=512 against 128-lane tiles
// with 2 or 4 lanes per thread (256 and 128 tokens) and 64-lane tiles with 4
// lanes per thread: the 64-lane, 2-lane, 512-token tile is fastest.
// The medium, small and one-lane tiles read one or kFwdWords look-back words
// per thread, chosen per launch (look_back_shift in osm_api.hip): every thread
// runs the polling code of each of its words, and on a chip full of tiles one
// is best (dynamic lambda, B=8 S=32768 D=1024: 420 us against 429 with two and
// 449 with eight).  The large tile keeps eight (no difference at B=4 S=16384
// D=512).
constexpr int kFwdWords = 4;
using FwdTileLarge = TileGeo<2, 8, 32>;           // 512 tokens x 64 lanes
// Dynamic lambda at 512 tokens: the per-token lambda lives in LDS (formed
// once per token and head), which leaves the registers for the run; one
// look-back word per thread (two per word pair: A and B).
using FwdTileLargeDyn = TileGeo<2, 8, 32, 64, 1>;
using FwdTileMedium = TileGeo<2, 8, 16, 64, kFwdWords>;   // 256 tokens x 64 lanes
using FwdTileSmall = TileGeo<2, 8, 8, 64, kFwdWords>;     // 128 tokens x 64 lanes
// One lane per thread: any head size, rows aligned to one element, and the
// Chebyshev form of longer series (more than kMonoMaxK coefficients), whose
// coefficients take twice the registers.  Used only where the geometries
// above do not apply.
// (two versions of one shape: with room for kFwdWords words the many-tile
// launches of 2-byte rows lose 1%: bf16 B=3 S=5001 D=400, 12.8 against 12.9 us)
using FwdTileGeneric = TileGeo<1, 8, 16, 64, 1>;             // 128 tokens x 64 lanes
using FwdTileGenericFew = TileGeo<1, 8, 16, 64, kFwdWords>;  // few lane-blocks
constexpr int kMaxTileRows = 512;              // bound on TILE (+1 row read past a tile)

// Geometry of a forward launch.
struct FwdShape {
  int tile;    // tokens per tile
  int lanes;   // lanes per lane-block
  int lpt;     // lanes per thread
};
// `generic`: the one-lane geometry (head size not a multiple of 4, rows not
// on 4-element boundaries, or more than 8 coefficients).
FwdShape fwd_geometry(bool dyn, int64_t B, int64_t D, int64_t S, bool generic);

// TTT: keeps the raw x and w = (1-lam)(1-2r) (r = 1/(1+exp(2 damping p)))
// of every token of the run in registers, u = softsign(x) in LDS, plus 2K
// gradient accumulators per lane: one lane per thread (half the
// accumulators of two).  Measured on MI355X at B=16 S=65536 D=512 (bf16),
// with u in LDS: 24-token runs 1001-1008 us against 1047-1056 with 20, 1025
// with 28 and 1092-1095 with 16 (longer runs amortise the per-thread setup,
// chain, composition and reduction over more tokens; at the 128-VGPR bound
// of two workgroups per CU the compiler spills 19 registers at 24 tokens,
// mostly on the rare slow path, and 40 at 28); 2 lanes x 8 or 16 tokens
// +10-20% (an earlier version).
// One look-back word per thread (checkpoints every 8 tiles): the kernel is
// VALU-bound, and every thread runs the polling code of each of its words
// (at 16-token runs 1147 us with two words against 1254 with eight and 1177
// with four; at 20-token runs one word 1069 against 1086 with two).
using TttTile = TileGeo<1, 8, 24, 64, 1>;   // 192 tokens
// 128-token tiles where the 192-token ones would leave CUs idle and one kernel
// still merges them (kDirectTiles): a tile's VALU work is then a launch's
// latency.  Measured on MI355X, 192 against 128 tokens: 15.0 and 12.3 us at B=1
// S=256 D=512 (16 tiles of 192), 18.1 and 15.1 at B=2 S=2048 (176), 20.0 and
// 21.4 at B=1 S=6000 (47 tiles of 128 a lane-block).  (96 tokens: 11.5, 16.7.)
using TttTileSmall = TileGeo<1, 8, 16, 64, 1>;   // 128 tokens
constexpr int kDirectTiles = 32;                 // tiles of a lane-block merged by one kernel (osm_ttt.hip)
int ttt_tile_tokens(int64_t n_lb, int64_t S);

// Backward: one lane per thread (the clamp mask makes the adjoint map's A
// differ per lane); x and dL/dout of the run stay in registers between the
// passes (plus lambda per token with a dynamic lambda), and the look-back
// reads two words (A, B) per predecessor.  Four look-back words per thread
// (checkpoints every 32 tiles) instead of eight brought the static kernel from
// 101 to 77 VGPRs, three workgroups per CU instead of two: 129 against 141 us
// at B=4 S=16384 D=512 on MI355X; two words (checkpoints every 16 tiles)
// 116.9 against 118.2 us with four.  24-token runs (94 VGPRs, two
// workgroups per CU) 113.8-114.4 against 116.5-116.8 us for 16 tokens; 20
// tokens 114.3, 28 tokens 118.2, 32 tokens 114.2; 8-token runs are slower
// (185 us).
using BwdTile = TileGeo<1, 8, 24, 64, 2>;   // 192 tokens
// More than 8 coefficients (Chebyshev form, kpad 16): 12-token runs; more
// than 16 (kpad 32): 4-token runs, room for 3 x 32 coefficient and gradient
// registers.
using BwdTileCheb = TileGeo<1, 8, 12, 64, 2>;   // 96 tokens
using BwdTileCheb32 = TileGeo<1, 8, 4, 64, 2>;  // 32 tokens
int bwd_tile_tokens(bool dyn, int kpad);

// Upper bound on polls of one look-back word (each poll is a device-scope
// load plus a short sleep: about a second in total).  It only guarantees
// that every wave exits if the dispatch-order assumption of the look-back
// ever failed or two calls overlapped on one workspace.  A launch with
// OSM_FLAG_POLL_LIMIT_ZERO (a test aid) polls no word a second time.
constexpr unsigned kSpinLimit = 1u << 20;

// Workspace: a kHeaderBytes header (launch epoch, fault word, completion
// counters), then the look-back words, then (TTT and backward) per-tile
// partials.
constexpr size_t kHeaderBytes = 2048;
// Header bytes kept when a known workspace changes layout (the launch epoch
// and the fault word; the completion counters from this offset on are
// cleared with the look-back words).
constexpr size_t kHeaderKeepBytes = 64;

// Multiplier and shift that divide by v (1 <= v < 2^31) for dividends
// 0 <= n < 2^31: s = ceil(log2 v), m = floor(2^32 (2^s - v) / v) + 1
// (Granlund and Montgomery, "Division by invariant integers using
// multiplication", 1994, the round-up variant).
inline void div_magic(uint32_t v, uint32_t* magic, int* shift) {
  int s = 0;
  while ((uint64_t(1) << s) < v) ++s;
  *shift = s;
  *magic = (uint32_t)((((uint64_t(1) << s) - v) << 32) / v + 1);
}

__host__ __device__ __forceinline__ unsigned mul_hi(unsigned a, unsigned b) {
  return (unsigned)(((unsigned long long)a * b) >> 32);
}

struct Divisor {
  uint32_t mul;
  int shift;
  __host__ __device__ __forceinline__ unsigned of(unsigned n) const { return (mul_hi(n, mul) + n) >> shift; }
};
inline Divisor divisor(int64_t v) {
  Divisor d;
  div_magic((uint32_t)v, &d.mul, &d.shift);
  return d;
}

// Tile order of a launch with a look-back (see osm_chain.h): which tile of
// which lane-block a block takes.
struct TileOrder {
  unsigned grid;
  bool spread;       // false: block v takes tile v / n_lb of slot v % n_lb
  unsigned ticket;   // spread: 0, or with tickets the share of ticket blocks as a fraction of 2^32
  int n_slots;       // spread, by index: blocks per tile row, a multiple of 8
  bool lead;         // spread: the first tile alone reads the initial state and publishes its own end state
  Divisor by_slots, by_whole, by_rest;   // n_slots; with tickets n_lb / 8 and n_lb % 8
  Divisor by_row;    // spread: lane-blocks of a batch row
};
struct TileSlot {
  int tile;   // >= n_tiles: none; -1: the next of the lane-block, by its ticket counter
  int lb;     // < 0: none
};

// Lane-block of slot s: the slots of one residue mod 8 (an XCD) serve
// consecutive lane-blocks, so the lane-blocks of a batch row share an L2 (they
// read the same lines of g, one value per head per token).  With n_lb = 8 q + r,
// residues below r hold q + 1.
__host__ __device__ __forceinline__ int slot_lane_block(int s, int n_lb) {
  const int c = s & 7, r = n_lb & 7;
  return c * (n_lb >> 3) + (c < r ? c : r) + (s >> 3);
}

// Spread orders.  By index, block v takes tile v / n_slots of slot v %
// n_slots, which is empty where its residue holds no such lane-block.
// With tickets, an XCD walks q whole lane-blocks by index and, spread evenly
// among their tiles, takes its eighth of the tiles of the r others.
__host__ __device__ __forceinline__ TileSlot spread_slot(const TileOrder& o, unsigned block, int n_lb, int n_tiles) {
  const int q = n_lb >> 3, r = n_lb & 7;
  if (!o.ticket) {
    const unsigned tile = o.by_slots.of(block), s = block - tile * (unsigned)o.n_slots;
    const bool held = (int)(s >> 3) < q + ((int)(s & 7u) < r ? 1 : 0);
    return {(int)tile, held ? slot_lane_block((int)s, n_lb) : -1};
  }
  const unsigned c = block & 7u, k = block >> 3;
  const unsigned e = q ? mul_hi(k, o.ticket) : k;   // ticket blocks of this XCD before block k
  if (q && mul_hi(k + 1, o.ticket) == e) {
    const unsigned tile = o.by_whole.of(k - e);
    return {(int)tile, (int)(c * (unsigned)q + (k - e - tile * (unsigned)q))};
  }
  const unsigned t = e * 8u + c;
  return {-1, t < (unsigned)r * (unsigned)n_tiles ? 8 * q + (int)(t - o.by_rest.of(t) * (unsigned)r) : -1};
}

// With n_lb off the multiples of 8, the order by index pads the slots and gives
// some XCDs a lane-block more than others; tickets balance them, but a block
// then waits for an atomic on memory before its first load.  By index where the
// fullest XCD has at most one tile for each of its CUs, or its surplus over the
// mean is at most 12 tiles or a sixteenth of its tiles.  Measured on MI355X, by
// index against tickets (fp32 unless noted):
//   forward B=1 S=4096 D=256 (32 tiles on the fullest XCD) 7.0 and 7.7 us, B=3
//   S=1000 D=400 (24) 6.9 and 7.5, TTT B=1 S=4000 D=256 (32) 15.5 and 16.2;
//   backward B=3 S=5000 D=448 (81, surplus 10) 31.5 and 32.6; forward B=9 S=8192
//   D=448 (128, surplus 2) 46.5 and 52.1;
//   forward B=3 S=5001 D=400 bf16 (120, surplus 15) 13.0 and 12.9, S=20000 fp32
//   52.4 and 49.2, B=5 S=5000 D=320 (160, surplus 35) 16.6 and 14.1, B=1 S=65536
//   D=128 37.9 and 19.7; TTT B=5 S=16384 D=448 bf16 (430, surplus 54) 94.8 and 90.1;
//   backward B=1 S=65536 D=128 91.6 and 46.2; table forward B=3 S=5000 D=448 (120,
//   surplus 15) 29.5 and 27.7.
// One counter for all lane-blocks made the tickets a queue (11 ns each): 21.1 us
// for the bf16 forward above.
//
// state_in_place: the final state may be written to the initial state's memory.
// The tiles of the first look-back group read the initial state when they
// resolve their carry, after they have published, so the last tile may be done
// before them; with `lead` they take the first tile's published state instead.
inline TileOrder tile_order(int64_t n_lb, int64_t n_tiles, int64_t n_lbd, bool state_in_place = false) {
  constexpr int64_t kCusPerXcd = 32;
  TileOrder o{};
  o.grid = (unsigned)(n_lb * n_tiles);
  if (n_tiles == 1 || (n_lb % 8 == 0 && !state_in_place)) return o;
  o.spread = true;
  o.by_row = divisor(n_lbd);
  o.lead = state_in_place;
  const int64_t pad = (n_lb + 7) / 8 * 8, most = pad / 8 * n_tiles, surplus = most - n_lb * n_tiles / 8;
  if (most <= kCusPerXcd || surplus <= 12 || surplus <= most / 16) {
    o.grid = (unsigned)(pad * n_tiles);
    o.n_slots = (int)pad;
    o.by_slots = divisor(pad);
    return o;
  }
  const int64_t q = n_lb / 8, r = n_lb % 8;
  const uint64_t tickets = (uint64_t)(r * n_tiles + 7) / 8, per_xcd = (uint64_t)(q * n_tiles) + tickets;
  o.grid = (unsigned)(8 * per_xcd);
  o.ticket = q ? (unsigned)(((tickets << 32) + per_xcd - 1) / per_xcd) : 1u;
  if (q) o.by_whole = divisor(q);
  o.by_rest = divisor(r);
  return o;
}

struct FwdParams {
  const void* x;
  void* out;
  const float* coeffs;
  const float* damping;
  const float* lam;
  const float* g;
  const float* ema_init;
  float* ema_final;
  unsigned long long* slots;   // look-back words [n_lb][n_tiles][LANES][words]
  unsigned* hdr;               // WsHeader
  float* partials;             // TTT per-tile partials (TTT kernels only)
  float* mono_tab;             // TTT: scaled monomial coefficients [n_lb][KP][64], formed once per launch,
                               // or NULL (each tile forms its own)
  const unsigned* mono_form;   // TTT: [n_lb] 1 where mono_tab holds Chebyshev coefficients instead
  int64_t x_sb, x_ss, o_sb, o_ss;
  int64_t c_sb, c_sh, c_sk;
  int64_t g_sb, g_ss, g_sh;
  int B, S, H, hd, K, D;
  uint32_t hd_magic;           // n / hd = (umulhi(n, hd_magic) + n) >> hd_shift for 0 <= n < 2^31
  int hd_shift;
  int n_lbd;                   // lane-blocks per batch row = ceil(D / LANES)
  int n_lb;                    // B * n_lbd
  TileOrder order;
  int n_tiles;                 // ceil(S / TILE)
  float lam_shift, lam_min, lam_max;
  int clamp_out;
  int nan_zero_u;              // NaN x counts as u = 0 (else z = 0)
  int jitter;                  // OSM_FLAG_TIMING_JITTER: pseudo-random delays (test aid)
  int wsh;                     // log2 of the look-back words per thread (kFwdWords geometries)
  unsigned poll_limit;         // look-back polls before a wait gives up: kSpinLimit, or 0 under
                               // OSM_FLAG_POLL_LIMIT_ZERO (test aid)
  float ttt_scale;             // 2 / (B*(S-1)*D)
  int ttt_target;
};

// Backward launch: the forward's parameters (x, out = the saved forward
// output, coefficients, lambda, shapes, workspace) plus the gradient streams.
struct BwdParams {
  FwdParams f;
  const void* gout;            // dL/dout, dtype of out
  void* gx;                    // dL/dx, dtype of x
  int64_t go_sb, go_ss, gx_sb, gx_ss;
  const float* grad_state;     // dL/d ema_final [B,D] or NULL
  float* grad_init;            // dL/d ema_init [B,D] or NULL
  float* grad_coeffs;          // [B,H,K,hd]
  const void* zs;              // saved z, bf16 [B,S,D], or NULL (recompute)
  int64_t zs_sb, zs_ss;
  int full_jac;                // dL/dx with 1/(1+|x|)^2 everywhere (no 1e-7 cutoff)
};

// Full-path launch (online TTT over chunks with an inline Lion update): one
// workgroup per (batch row, head, group of `lanes` lanes) walks the chunks in
// order.  Needs no workspace.  The chunks of a lane are sequential, so the
// lanes are the only parallelism: 8 lanes per workgroup, or 4 where that
// spreads the work better (v10_lanes).
constexpr int kV10Groups = 64;    // token groups (runs) per 256-token block
constexpr int kV10Run = 4;        // tokens per run
int v10_lanes(int64_t B, int64_t H, int64_t hd);
int v10_fixed_lanes(int64_t B, int64_t H, int64_t hd);
struct V10Params {
  const void* x;
  float* out;
  const float* coeffs;
  const float* momentum;
  float* coeffs_out;
  float* momentum_out;
  const float* lut;            // [8][256] fp32 (LUT mode)
  const float* lion_lambda;    // [H]
  const float* lr_scale;       // [H]
  const float* spectral_scale; // [K]
  const float* gate;           // [B] or NULL
  const float* dyn_lambda;     // [B] or NULL
  void* z_save;                // bf16 [B,S,D] or NULL
  float* coeff_hist;           // [n_chunks][B,H,K,hd] or NULL
  const float* mu_dev;         // device scalar overriding mu, or NULL
  int64_t x_sb, x_ss, o_sb, o_ss, z_sb, z_ss;
  int64_t c_sb, c_sh, c_sk, m_sb, m_sh, m_sk;
  int B, S, H, hd, K, D, chunk, n_lg;
  int lanes;                   // lanes per workgroup (4 or 8; fixed forward 8 or 16)
  float mu, base_lr, beta1, beta2, wd;
};

// The fixed-coefficient forward (osm_cheby_ema_lut_fwd) on the same kernel:
// one chunk of S tokens, no Lion, x as given, EMA from ema_init, out =
// clamp(s) in fp32, the carried state clamped every clamp_tile tokens, and
// optional x_norm, tanh_y and ema_final outputs.  (A separate struct, so the
// full path's kernel arguments stay as they are.)
struct V10FixedParams : V10Params {
  const float* ema_init;       // [B, D] (row stride init_sb) or NULL (0)
  float* ema_final;            // [B, D] (row stride final_sb) or NULL
  float* xnorm;                // [B,S,D] fp32 or NULL
  float* tanhy;                // [B,S,D] fp32 or NULL
  int64_t init_sb, final_sb, xn_sb, xn_ss, ty_sb, ty_ss;
  int clamp_tile;              // tokens between clamps of the carried state
};

// The same forward as a single-pass scan over tiles (osm_lut.hip), chained by
// the look-back: for 0.25 <= mu <= 1 and a caller's workspace.  128-token
// tiles where they give every CU one, else 64 (a tile of 128 tokens holds
// its CU's VALUs ~3.8 us): on MI355X, D=512 K=8, 64 tokens against 128, 9.4 and
// 10.4 us at B=4 S=512 (128 tiles of 128 tokens), 12.0 and 12.1 at B=2 S=2000
// D=400 (224), 21.3 and 15.2 at B=2 S=4096 (512).  One lane per thread where
// rows are off two-element boundaries.
using LutTile = TileGeo<2, 8, 8, 64, kFwdWords>;              // 128 tokens x 64 lanes
using LutTileSmall = TileGeo<2, 8, 4, 64, kFwdWords>;         // 64 tokens
using LutTileGeneric = TileGeo<1, 8, 16, 64, kFwdWords>;      // 128 tokens
using LutTileGenericSmall = TileGeo<1, 8, 8, 64, kFwdWords>;  // 64 tokens
struct LutScanParams : V10FixedParams {
  unsigned long long* slots;   // look-back words [n_lb][n_tiles][64]
  unsigned* hdr;               // WsHeader
  uint32_t hd_magic;           // division by hd (div_magic)
  int hd_shift;
  int n_lbd, n_lb, n_tiles;
  TileOrder order;
  int wsh;                     // log2 of the look-back words per thread
  int clamp_at;                // tile that holds the first clamp boundary
  int jitter;                  // as in FwdParams
  unsigned poll_limit;
};

// Backward of the full path (osm_v10_bwd): dL/dx of every chunk, one
// workgroup per (batch row, chunk, 64-lane lane-block).  Needs no workspace.
struct V10BwdParams {
  const void* x;
  const float* gout;           // dL/dout
  const float* out;            // the saved output (the clamp mask)
  const void* z;               // the saved z, bf16
  const float* hist;           // [n_chunks][B,H,K,hd]
  void* gx;                    // dL/dx, dtype of x
  const float* mu_dev;         // device scalar overriding mu, or NULL
  int64_t x_sb, x_ss, go_sb, go_ss, o_sb, o_ss, z_sb, z_ss, gx_sb, gx_ss;
  int B, S, H, hd, K, D, chunk, n_chunks, n_lbd;
  int n_items;                 // B * n_chunks * n_lbd
  int items_per_xcd;           // ceil(n_items / 8); grid = 8 * items_per_xcd
  float mu;
};

// The engine's input norm, complexity gate and momentum schedule (osm_engine).
constexpr int kEngineMaxD = 1024;   // row length the kernels hold in registers and LDS
struct EngineParams {
  const float* x;
  const float* norm_w;         // [D]
  const float* w1;             // [D/4, D]
  const float* b1;             // [D/4]
  const float* w2;             // [D/4]
  const float* b2;             // [1]
  const float* ema_base;       // scalar
  long long* tokens;           // scalar, advanced by S
  float* xn;                   // [B,S,D] contiguous
  float* gate;                 // [B]
  float* mu;                   // scalar
  float* part;                 // [B][engine_tiles(S)][D]
  int64_t x_sb, x_ss;
  int B, S, D;
  float eps;
};

// Workspace layout helpers (bytes).
size_t slot_words(bool dyn);
size_t fwd_workspace_bytes(int n_lb, int n_tiles, int lanes, bool dyn);
size_t ttt_workspace_bytes(int n_lb, int n_tiles, bool dyn, int K);
size_t bwd_workspace_bytes(int n_lb, int n_tiles, int K);
size_t bwd_slot_bytes(int n_lb, int n_tiles);

// Launchers: return hipSuccess or the launch error.
hipError_t launch_fwd(const FwdParams& p, int x_dtype, int out_dtype, bool dyn, FwdShape shape, int kpad,
                      hipStream_t stream);
hipError_t launch_ttt(const FwdParams& p, float* grad, int x_dtype, int out_dtype, bool dyn, int tile,
                      int kpad, hipStream_t stream);
hipError_t launch_bwd(const BwdParams& p, int x_dtype, int out_dtype, bool dyn, int tile, int kpad,
                      hipStream_t stream);
hipError_t launch_v10(const V10Params& p, int x_dtype, bool use_lut, int kpad, hipStream_t stream);
int v10_bwd_lanes();   // lanes per lane-block of launch_v10_bwd
hipError_t launch_v10_bwd(const V10BwdParams& p, int x_dtype, int lpt, int kpad, hipStream_t stream);
hipError_t launch_v10_fixed(const V10FixedParams& p, int x_dtype, bool use_lut, int kpad, hipStream_t stream);
hipError_t launch_lut_scan(const LutScanParams& p, int x_dtype, bool use_lut, FwdShape s, int kpad,
                           hipStream_t stream);
int engine_tiles(int64_t S);
hipError_t launch_engine(const EngineParams& p, hipStream_t stream);
hipError_t launch_fill_zero(void* ptr, size_t bytes, hipStream_t stream);
hipError_t launch_copy_state(const float* src, float* dst, size_t n, hipStream_t stream);
hipError_t launch_ws_status(void* ws, unsigned* dst, int reset, hipStream_t stream);

}  // namespace osm
