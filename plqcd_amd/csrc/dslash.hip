// Host side of the Wilson hopping matrix: argument checks, dispatch to the
// per-format launchers (kernels in dslash_kernels.h, instantiated once per
// storage precision and link format in dslash_<precision>_l<links>.hip), and the
// process-wide launch shapes with the per-shape cache of the autotuner.
#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>

#include "dslash.h"
#include "reduce.h"

// Built-in launch shapes.
//
// A march kernel's time is rounds x slices: its blocks run in rounds of as
// many as the chip holds at once, and each block takes as many slice times as
// its t-chunk has slices, plus a prologue worth `c` of them.  A last round
// that is nearly empty costs almost as much as a full one, so the t-chunk
// count that fits the rounds matters more than anything else in the shape: at
// 24^3 x 48, F64 with one RHS on 24 x 4 x 2 tiles (192 lanes, one block per
// CU), 16 slices per chunk fill 84 % of one round and take 153 us, 12 need a
// second round and take 223 us.  The cost of a shape is therefore
//
//   lanes of a round x k x (slices + c) x (whole rounds + max(last round's share, f))
//
// and the cheapest shape is taken.  f is the share of a round below which the
// blocks no longer run faster for being fewer (latency), k the kernel's time
// per lane and slice relative to the others, `waves` how many waves of it a
// SIMD's registers hold.  The gather kernel has no chunks and no rounds to
// speak of.  The constants were fitted to timings of every shape of 14 lattices
// from 8^3 x 16 to 32^3 x 64, ten of them with extents that are no powers of
// two (28 x 20 x 36 x 44, 32 x 42 x 24 x 64, 10 x 16 x 14 x 54 and so on), with
// 1, 2 and 3 RHS, and of 6 lattices with 4 and 12 RHS.  The shapes they pick take
// on average 3 to 6 % longer than the fastest one timed, depending on the
// format, and 17 % at most.
namespace {
constexpr int kCus = 256;
constexpr int kPipeRhs = 4;  // right-hand sides from which the pipelined t-march runs (pipe_fits)
struct KernelCost {
   int waves;
   double k, f, c;
   int most = 1 << 30;  // slices per chunk; blocks drift apart over long ones and lose their shared L2 lines
};
struct FormatCost {
   KernelCost march, tile, gather;
};

const FormatCost &one_rhs_cost(int prec, int links)
{
   static const FormatCost f64 = {{1, 1.12, 0.53, 0.54}, {1, 1.0, 0.89, 1.52}, {3, 1.64, 0.07, 0}};
   static const FormatCost f32_18 = {{2, 0.95, 0.33, 0.19}, {1, 1.0, 0.32, 0.60}, {4, 1.90, 0.52, 0}};
   static const FormatCost f32_12 = {{2, 1.07, 0.84, 1.12}, {2, 1.0, 0.95, 1.20}, {4, 1.29, 0.39, 0}};
   static const FormatCost f16 = {{3, 0.83, 0.56, 0.81}, {2, 1.0, 0.78, 1.18}, {5, 1.05, 0.62, 0}};
   return prec == PLQCD_PREC_F64 ? f64 : prec == PLQCD_PREC_F16 ? f16 : links == 18 ? f32_18 : f32_12;
}

const FormatCost &multi_rhs_cost(int prec, int links, int R)  // no tiles
{
   // the t-march (2 and 3 RHS)
   static const FormatCost f64 = {{1, 1.0, 0.91, 0.43, 32}, {}, {3, 1.58, 0.04, 0}};
   static const FormatCost f32_18 = {{2, 1.0, 1.00, 0.43}, {}, {4, 1.31, 0.06, 0}};
   static const FormatCost f32_12 = {{2, 1.0, 1.00, 0.49}, {}, {4, 1.20, 0.09, 0}};
   static const FormatCost f16 = {{3, 1.0, 1.00, 0.65, 8}, {}, {5, 1.28, 0.53, 0}};
   // the pipelined t-march
   static const FormatCost p64 = {{1, 1.0, 0.99, 0.97, 32}, {}, {3, 1.57, 0.37, 0}};
   static const FormatCost p32 = {{2, 1.0, 0.78, 0.80, 32}, {}, {4, 1.49, 0.39, 0}};
   static const FormatCost p16 = {{3, 1.0, 0.92, 0.20, 12}, {}, {5, 1.40, 0.16, 0}};
   if (R < kPipeRhs)
      return prec == PLQCD_PREC_F64 ? f64 : prec == PLQCD_PREC_F16 ? f16 : links == 18 ? f32_18 : f32_12;
   return prec == PLQCD_PREC_F64 ? p64 : prec == PLQCD_PREC_F32 ? p32 : p16;
}

// LDS of a pipelined t-march block (hop_pipe_block): two slices' links
size_t pipe_lds(int prec, int spb)
{
   return size_t(14) * spb * (prec == PLQCD_PREC_F64 ? 144 : prec == PLQCD_PREC_F32 ? 80 : 48);
}

// The patch of gy x gz column blocks (of spb sites each, both parities) that
// an XCD's L2 serves at a time: the least halo per site -- 1 / rows in y and 1
// / planes in z, none over a whole extent -- of the patches with at most as
// many column blocks as an XCD holds and its L2 keeps the slices of (F64 16,
// else 48; 24^3 x 48, 12 RHS: F64 12 blocks 1032 us, 18 1038, 24 1064, 36 1078;
// F32 24 blocks 499 us, 36 494, 48 491; 32^3 x 64 F16 32 blocks 894, 64 909).
void pick_patch(const int L[4], int prec, int spb, HopTuning *t)
{
   const int Lxh = L[0] / 2, nby = Lxh * L[1] / spb, most = prec == PLQCD_PREC_F64 ? 16 : 48;
   t->order = 1;
   t->group = 1;
   if (nby < 1 || Lxh * L[1] % spb) return;
   double best = 1e300;
   for (int gy = 1; gy <= nby && gy <= most; gy++) {
      if (nby % gy) continue;
      for (int gz = 1; gz <= L[2] && gy * gz <= most; gz++) {
         if (L[2] % gz) continue;
         const double halo = (gy < nby ? double(Lxh) / (gy * spb) : 0) + (gz < L[2] ? 1.0 / gz : 0) + 1e-6 * gy * gz;
         if (halo < best) {
            best = halo;
            t->gy = gy;
            t->gz = gz;
         }
      }
   }
   t->order = 2;
   t->group = 2 * t->gy * t->gz;
}

// LDS of a tile block (hop_tile_kernel): two slices of centre spinors, the
// backward t terms and, in F64 blocks of up to 128 lanes, the x links.
size_t tile_lds(int prec, int lanes)
{
   const int block = lanes <= 128 ? 128 : lanes <= 256 ? 256 : 512;
   const size_t sp = prec == PLQCD_PREC_F64 ? 192 : prec == PLQCD_PREC_F32 ? 96 : 52;
   const size_t hv = prec == PLQCD_PREC_F64 ? 96 : prec == PLQCD_PREC_F32 ? 48 : 52;
   return block * (2 * sp + hv + (prec == PLQCD_PREC_F64 && block == 128 ? 144 : 0));
}

double rounds(double blocks, double resident, double f)
{
   const double x = blocks / resident, whole = std::floor(x);
   return whole + (x > whole ? std::max(x - whole, f) : 0.0);
}

struct Pick {
   const int *L;
   HopTuning best{};
   double cost = 1e300;
   // `chunk_blocks` blocks per t-chunk, of `lanes` lanes, `per_cu` on a CU.  Too
   // few lanes for latency to be hidden at all are left out (10 x 16 x 14 x 54,
   // F32: 13000 lanes in tiles 45 us, 60000 untiled 15).
   void march(const KernelCost &c, HopTuning t, double chunk_blocks, int lanes, int per_cu)
   {
      const bool tile = t.ty > 0;
      const double fewest = tile ? 16000 : 8000;
      // the chunk counts that were timed, and one slice per chunk
      for (int n : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 24, 32, 48, 64, L[3]}) {
         const int nt = std::min(n, L[3]), T = (L[3] + nt - 1) / nt;
         if (T > c.most || (T > 1 && chunk_blocks * nt * lanes < fewest) || (T == 1 && tile)) continue;
         const double res = double(kCus) * per_cu;
         t.tmarch = T;
         offer(t, res * lanes * c.k * (T + c.c) * rounds(chunk_blocks * ((L[3] + T - 1) / T), res, c.f));
      }
   }
   void offer(const HopTuning &t, double v)
   {
      if (v < cost * (1 - 1e-9)) {
         cost = v;
         best = t;
      }
   }
};

// The shape for R right-hand sides on the lattice with extents L.
HopTuning pick_shape(const int L[4], int prec, int links, int R, bool solver)
{
   const int Lxh = L[0] / 2, wave = 64;
   const double S = double(Lxh) * L[1] * L[2], Vh = S * L[3];
   const FormatCost &fc = R <= 1 ? one_rhs_cost(prec, links) : multi_rhs_cost(prec, links, R);
   Pick p{L};
   // Each XCD takes a contiguous eighth; with two or three RHS on large
   // t-slices the eighth's slices no longer fit an XCD's L2 and the XCDs sweep
   // the lattice together (mean over the shapes near the best, XCDs together
   // against eighths: 0.97 at 32^3, 1.01 at 38 x 18 x 26 and 24^3, 1.04 and more
   // below).  F64 with two RHS from somewhat larger ones on (us, 32^3 x 64 785
   // and 771, 40^3 x 80 1951 and 1987; three RHS at 32^3 x 64 1129 and 1159); F16,
   // a quarter of the bytes, never (two RHS 190 and 184, at 40^3 x 80 450 and 444;
   // three 279 and 273).
   const bool together = R > 1 && prec != PLQCD_PREC_F16 &&
                         2 * S * (prec == PLQCD_PREC_F64 ? R : 3) >= 3 * 32768;
   for (int block : {64, 128, 256}) {
      if (R <= 1 ? block != 64 : block == 64) continue;
      const int spb = REDUCE_CHUNK * std::max(1, block / (REDUCE_CHUNK * R));
      const int lanes = spb * R, wpb = (lanes + wave - 1) / wave;
      HopTuning t{together ? 2 : 1, together ? 8 : 1, block, 0, 1, 0, 0};
      const double res = double(kCus) * std::max(1, 4 * fc.gather.waves / wpb);
      const double gb = 2 * std::ceil(Vh / spb);
      // of equals, gather blocks of 128 lanes (2 RHS at 8^3 x 16: 8.0 against 10.2
      // us), march blocks of 256
      p.offer(t, std::max(gb / res, fc.gather.f) * res * lanes * fc.gather.k * (block == 256 ? 1 + 1e-6 : 1));
      int per_cu = 4 * fc.march.waves / wpb;
      if (R >= kPipeRhs) {
         // F16 with the solver's epilogues and two links per lane: two waves (pipe_waves)
         if (solver && prec == PLQCD_PREC_F16 && 7 * spb > lanes) per_cu = 4 * 2 / wpb;
         per_cu = std::min<int>(per_cu, 160 * 1024 / pipe_lds(prec, spb));
         pick_patch(L, prec, spb, &t);
      }
      // smaller blocks share each link and halo row among fewer lanes: only
      // where they fit the rounds clearly better
      KernelCost c = fc.march;
      // one RHS in F16: long marches drift apart, the solver's epilogues sooner (us
      // per H with 12, 16, 24 and 96 slices, 48^3 x 96: 529, 538, 544, 566; ms per
      // CG solve with 8, 12, 16 and 32: 26.9, 27.4, 29.4, 35.7 at 32^3 x 64).  Those
      // epilogues also hold fewer waves (6 slices, which would fill three waves
      // best: 28.5) and fill a round sooner (24^3 x 48, 6 and 8 slices: 11.9, 12.7)
      if (R <= 1 && prec == PLQCD_PREC_F16) {
         c.most = solver ? 8 : 16;
         if (solver) {
            per_cu = 4 * 2 / wpb;
            c.f = 0.8;
         }
      }
      if (block == 128) c.k *= R >= kPipeRhs ? 1.1 : 1 + 1e-6;
      p.march(c, t, 2 * std::ceil(S / spb), lanes, std::max(1, per_cu));
   }
   if (R <= 1) {
      // Tiles that fill more than four fifths of 2, 3, 4, 6 or 8 waves (F64 38 x
      // 18 x 26 x 60, 152 of 192 lanes: 274 us, 228 lanes: 250).  Of equally large ones those longer in y,
      // within 1 % of the best turn on average (the other way 5 to 7 % above);
      // except F64 with x rows of 32 sites or more, plain H (401 us for 32 x 1 x 4
      // at 32^3 x 64, 414 for 32 x 4 x 1; its solver epilogues prefer the long
      // one too, 0.0769 against 0.0806 s a solve).
      const bool flat = prec == PLQCD_PREC_F64 && L[0] >= 32 && !solver;
      const int most = prec == PLQCD_PREC_F64 ? 256 : 512;
      for (int i = 1; i <= 8 && i <= L[1] && i * L[0] <= most; i++) {
         for (int k = 1; k <= 8 && k <= L[2] && k * L[0] <= most; k++) {
            const int ty = i, tz = k, lanes = L[0] * ty * tz;
            const bool full = (lanes > 102 && lanes <= 128) || (lanes > 153 && lanes <= 192) ||
                              (lanes > 204 && lanes <= 256) || (lanes > 307 && lanes <= 384) ||
                              (lanes > 409 && lanes <= 512);
            if (L[1] % ty || L[2] % tz || !full || lanes > most) continue;
            if (solver && Lxh * ty % REDUCE_CHUNK) continue;  // the norms' chunks
            const int wpb = (lanes + wave - 1) / wave;
            const int per_cu = std::min(4 * fc.tile.waves / wpb, int(160 * 1024 / tile_lds(prec, lanes)));
            KernelCost c = fc.tile;
            // F64 blocks of up to 128 lanes pass the x links through LDS (32^3 x 64,
            // 32 x 4 x 1 410 us, 32 x 8 x 1 452)
            if (prec == PLQCD_PREC_F64 && lanes > 128) c.k *= 1.03;
            c.k *= 1 + 1e-6 * (flat ? ty : -ty);
            p.march(c, HopTuning{1, 1, 256, 0, 1, ty, tz}, S / (double(Lxh) * ty * tz), lanes, std::max(1, per_cu));
         }
      }
   }
   return p.best;
}
bool g_tuning_set[3] = {false, false, false};  // set by plqcd_hip_hop_tuning

HopTuning headline_shape(int prec)
{
   const int L[4] = {32, 32, 32, 64};
   return pick_shape(L, prec, prec == PLQCD_PREC_F16 ? 12 : 18, 1, false);
}

// Shapes picked so far, by value of what they were picked for.
std::mutex g_shape_mu;
std::map<plqcd::TuneKey, HopTuning> g_shapes;
constexpr size_t kMostShapes = 4096;
}  // namespace

// The one-RHS shapes at 32^3 x 64 of the 18-real (F16: 12-real) formats, per
// precision; plqcd_hip_hop_tuning replaces them.
HopTuning g_tuning[3] = {headline_shape(PLQCD_PREC_F64), headline_shape(PLQCD_PREC_F32),
                         headline_shape(PLQCD_PREC_F16)};

bool plqcd::user_tuning(int prec, HopTuning *t)
{
   if (g_tuning_set[prec]) *t = g_tuning[prec];
   return g_tuning_set[prec];
}

HopTuning plqcd::default_tuning(const int L[4], int prec, int links, int R, bool solver)
{
   if (g_tuning_set[prec]) return g_tuning[prec];
   const TuneKey key{{L[0], L[1], L[2], L[3]}, prec, links, R, solver ? kTuneOpSolver : kTuneOpHop};
   std::lock_guard<std::mutex> lk(g_shape_mu);
   auto it = g_shapes.find(key);
   if (it != g_shapes.end()) return it->second;
   if (g_shapes.size() >= kMostShapes) g_shapes.clear();
   return g_shapes[key] = pick_shape(L, prec, links, R, solver);
}

namespace {
std::mutex g_tune_mu;
std::map<plqcd::TuneKey, HopTuning> g_tune_cache;
}  // namespace

bool plqcd::lookup_tuning(const TuneKey &k, HopTuning *t)
{
   std::lock_guard<std::mutex> lk(g_tune_mu);
   auto it = g_tune_cache.find(k);
   if (it == g_tune_cache.end()) return false;
   *t = it->second;
   return true;
}

void plqcd::store_tuning(const TuneKey &k, const HopTuning &t)
{
   std::lock_guard<std::mutex> lk(g_tune_mu);
   g_tune_cache[k] = t;
}

void plqcd::clear_tuning(const TuneKey *k)
{
   std::lock_guard<std::mutex> lk(g_tune_mu);
   if (k) g_tune_cache.erase(*k);
   else g_tune_cache.clear();
}

extern "C" int plqcd_hip_hop_batch(int n, const plqcd_hip_gauge *const *g, const plqcd_hip_field *const *in,
                                   plqcd_hip_field *const *out, int mode)
{
   plqcd::clear_error();
   if (n < 1 || !g || !in || !out) return plqcd::set_error(1, "hop_batch: bad arguments");
   for (int i = 0; i < n; i++) {
      if (!g[i] || !in[i] || !out[i] || in[i] == out[i] || in[i]->lat != g[i]->lat || out[i]->lat != g[i]->lat ||
          in[i]->nrhs != out[i]->nrhs || in[i]->prec != g[i]->prec || out[i]->prec != g[i]->prec ||
          g[i]->prec != g[0]->prec || g[i]->links != g[0]->links)
         return plqcd::set_error(1, "hop_batch: item %d is inconsistent (all items share precision and link format)", i);
      if (g[i]->lat->stream != g[0]->lat->stream)
         return plqcd::set_error(1, "hop_batch: all lattices must use the same stream (set_stream)");
   }
   if (mode != PLQCD_HOP_COMPAT && mode != PLQCD_HOP_WILSON) return plqcd::set_error(1, "hop_batch: bad mode");
   switch (g[0]->prec * 100 + g[0]->links) {
      case PLQCD_PREC_F64 * 100 + 18: return plqcd::hop_batch_launch<PLQCD_PREC_F64, 18>(n, g, in, out, mode);
      case PLQCD_PREC_F64 * 100 + 12: return plqcd::hop_batch_launch<PLQCD_PREC_F64, 12>(n, g, in, out, mode);
      case PLQCD_PREC_F32 * 100 + 18: return plqcd::hop_batch_launch<PLQCD_PREC_F32, 18>(n, g, in, out, mode);
      case PLQCD_PREC_F32 * 100 + 12: return plqcd::hop_batch_launch<PLQCD_PREC_F32, 12>(n, g, in, out, mode);
      case PLQCD_PREC_F16 * 100 + 12: return plqcd::hop_batch_launch<PLQCD_PREC_F16, 12>(n, g, in, out, mode);
      case PLQCD_PREC_F16 * 100 + 18: return plqcd::hop_batch_launch<PLQCD_PREC_F16, 18>(n, g, in, out, mode);
      default: return plqcd::set_error(1, "hop_batch: unsupported gauge format");
   }
}

HopArgs make_hop_args(const plqcd_hip_lattice *lat, int parity)
{
   HopArgs a{};
   for (int mu = 0; mu < 4; mu++) a.L[mu] = lat->L[mu];
   a.Lxh = lat->Lxh;
   a.Vh = lat->Vh;
   a.nparity = (parity == PLQCD_PARITY_ALL) ? 2 : 1;
   a.parity0 = (parity == PLQCD_PARITY_ODD) ? 1 : 0;
   a.order = 0;
   a.group = 1;
   a.S = lat->Vh / lat->L[3];
   a.nt = 1;
   a.R = 1;
   a.spb = 256;
   return a;
}

int plqcd::dslash(const plqcd_hip_gauge *g, const plqcd_hip_field *in, plqcd_hip_field *out, int parity, int mode,
                  const DslashOp &op)
{
   if (!g || !in || !out) return plqcd::set_error(1, "hop: null argument");
   if (in == out) return plqcd::set_error(1, "hop: in and out must be distinct fields");
   if (in->lat != g->lat || out->lat != g->lat)
      return plqcd::set_error(1, "hop: fields and gauge belong to different lattices");
   if (in->prec != g->prec || (out->prec != g->prec && !op.resid_b))
      return plqcd::set_error(1, "hop: precision mismatch (gauge %d, in %d, out %d)", g->prec, in->prec, out->prec);
   if (in->nrhs != out->nrhs) return plqcd::set_error(1, "hop: RHS count mismatch");
   if (parity < PLQCD_PARITY_EVEN || parity > PLQCD_PARITY_ALL) return plqcd::set_error(1, "hop: bad parity %d", parity);
   if (mode != PLQCD_HOP_COMPAT && mode != PLQCD_HOP_WILSON) return plqcd::set_error(1, "hop: bad mode %d", mode);
   if (op.rlist && (op.nr < 1 || op.nr > in->nrhs))
      return plqcd::set_error(1, "hop: RHS list of %d entries for fields of %d", op.nr, in->nrhs);
   if (!op.rlist && (op.nr < 0 || op.r0 < 0 || (op.nr > 0 && op.r0 + op.nr > in->nrhs)))
      return plqcd::set_error(1, "hop: RHS window %d + %d outside the fields' %d", op.r0, op.nr, in->nrhs);
   if (op.kappa_host && (op.kappa || in->nrhs > kInlineKappa || op.alpha || op.resid_b || op.partial))
      return plqcd::set_error(1, "hop: kappa by value is for up to %d right-hand sides of M and M^+", kInlineKappa);
   if (op.centre) {
      const plqcd_hip_field *c = op.centre;
      if (c->lat != g->lat || c->prec != g->prec || c->nrhs != in->nrhs || c == out || !(op.kappa || op.kappa_host) || op.dag ||
          op.alpha || op.partial || op.resid_b)
         return plqcd::set_error(1, "hop: the centre field must be like in, distinct from out, with kappa and no "
                                    "other epilogue");
   }
   if (op.resid_b) {
      const plqcd_hip_field *b = op.resid_b;
      if (g->prec != PLQCD_PREC_F64 || b->lat != g->lat || b->prec != PLQCD_PREC_F64 || b->nrhs != in->nrhs ||
          b == in || b == out || op.alpha || !op.dag || !op.kappa || !op.partial)
         return plqcd::set_error(1, "hop: the residual epilogue needs an F64 gauge, an F64 b distinct from in and "
                                    "out, M^+, kappa and a norm");
   }
   switch (g->prec * 100 + g->links) {
      case PLQCD_PREC_F64 * 100 + 18: return plqcd::hop_launch<PLQCD_PREC_F64, 18>(g, in, out, parity, mode, op);
      case PLQCD_PREC_F64 * 100 + 12: return plqcd::hop_launch<PLQCD_PREC_F64, 12>(g, in, out, parity, mode, op);
      case PLQCD_PREC_F32 * 100 + 18: return plqcd::hop_launch<PLQCD_PREC_F32, 18>(g, in, out, parity, mode, op);
      case PLQCD_PREC_F32 * 100 + 12: return plqcd::hop_launch<PLQCD_PREC_F32, 12>(g, in, out, parity, mode, op);
      case PLQCD_PREC_F16 * 100 + 12: return plqcd::hop_launch<PLQCD_PREC_F16, 12>(g, in, out, parity, mode, op);
      case PLQCD_PREC_F16 * 100 + 18: return plqcd::hop_launch<PLQCD_PREC_F16, 18>(g, in, out, parity, mode, op);
      default: return plqcd::set_error(1, "hop: unsupported gauge format");
   }
}

extern "C" int plqcd_hip_hop(const plqcd_hip_gauge *g, const plqcd_hip_field *in, plqcd_hip_field *out, int parity,
                             int mode)
{
   return plqcd::dslash(g, in, out, parity, mode, plqcd::DslashOp{});
}

extern "C" int plqcd_hip_hop_tuning(int prec, int order, int group, int block, int tmarch, int rb, int tile_y,
                                    int tile_z)
{
   if (prec < -1 || prec > PLQCD_PREC_F16 || order < 0 || order > 2 || group < 1 || group > 4096 ||
       (block != 64 && block != 128 && block != 256 && block != 512) || tmarch < 0 || tmarch > 4096 ||
       (rb != 1 && rb != 2 && rb != 4) || tile_y < 0 || tile_z < 0 || tile_y > 4096 || tile_z > 4096 ||
       ((tile_y == 0) != (tile_z == 0)))
      return plqcd::set_error(1, "plqcd_hip_hop_tuning: bad parameters (prec %d, order %d, group %d, block %d, "
                                 "tmarch %d, rb %d, tile %d x %d)", prec, order, group, block, tmarch, rb, tile_y, tile_z);
   for (int p = 0; p < 3; p++)
      if (prec < 0 || p == prec) {
         g_tuning[p] = HopTuning{order, group, block, tmarch, rb, tile_y, tile_z};
         g_tuning_set[p] = true;
      }
   return 0;
}

extern "C" int plqcd_hip_hop_tuning_reset(int prec)
{
   if (prec < -1 || prec > PLQCD_PREC_F16) return plqcd::set_error(1, "plqcd_hip_hop_tuning_reset: bad precision");
   for (int p = 0; p < 3; p++)
      if (prec < 0 || p == prec) {
         g_tuning[p] = headline_shape(p);
         g_tuning_set[p] = false;
      }
   return 0;
}

extern "C" int plqcd_hip_hop_get_tuning(int prec, int out[7])
{
   if (prec < 0 || prec > PLQCD_PREC_F16 || !out) return plqcd::set_error(1, "plqcd_hip_hop_get_tuning: bad arguments");
   out[0] = g_tuning[prec].order;
   out[1] = g_tuning[prec].group;
   out[2] = g_tuning[prec].block;
   out[3] = g_tuning[prec].tmarch;
   out[4] = g_tuning[prec].rb;
   out[5] = g_tuning[prec].ty;
   out[6] = g_tuning[prec].tz;
   return 0;
}
