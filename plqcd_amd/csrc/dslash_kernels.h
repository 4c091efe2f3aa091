// The Wilson hopping matrix on gfx950.
//
//   out(x) = sum_mu [ U_mu(x) (1 - gamma_mu) in(x+mu) + U_mu(x-mu)^+ (1 + gamma_mu) in(x-mu) ]
//
// (plqcd.pdf Eq. 2.1; lib/dirac.c:35-408 and :414-791 compute the two parity
// halves of it in four phases over half-spinor scratch fields).  Here it is a
// single gather pass: one thread per output site reads its 8 neighbour
// spinors and 8 links straight from HBM-resident structure-of-arrays fields,
// projects each neighbour to a half-spinor (2 colour vectors) before the SU(3)
// multiply, and writes its output once with a non-temporal store.  There is
// no scratch field, no halo and no MPI: periodic neighbours are computed from
// the site coordinates inside the kernel.
//
// Gamma matrices, projectors and reconstruction are the reference's chiral
// basis (lib/dirac.c:95-114, :163-195, :269-311, :371-398):
//   mu  upper((1-g)f)          upper((1+g)g)           s2 +=            s3 +=
//   0   (f0+f2,   f1+f3)       (g0-g2,   g1-g3)        a0 - b0          a1 - b1
//   1   (f0+i f3, f1+i f2)     (g0-i g3, g1-i g2)      -i a1 + i b1     -i a0 + i b0
//   2   (f0+f3,   f1-f2)       (g0-g3,   g1+g2)        -a1 + b1         a0 - b0
//   3   (f0+i f2, f1-i f3)     (g0-i g2, g1+i g3)      -i a0 + i b0     i a1 - i b1
// with a = U_mu(x) h, b = U_mu(x-mu)^+ k, s0 += a0 + b0, s1 += a1 + b1.
//
// MODE_COMPAT reproduces what the compiled reference outputs: forward terms
// do not reach s2/s3 (dirac.c:373-374 and :756-757 assign the mu=0 backward
// term over them) and odd output sites take their forward links from the even
// site with the same index inside its parity (dirac.c:643-644).
#pragma once

#include <algorithm>
#include <type_traits>
#include <vector>

#include "fields.h"
#include "dslash.h"
#include "reduce.h"

namespace {

constexpr int MODE_COMPAT = PLQCD_HOP_COMPAT;

// Site of thread (parity p, index j inside the parity) and the within-parity
// indices of its 8 neighbours (which all have the other parity).
struct Nbr {
   int up[4], dn[4];
};

__device__ __forceinline__ Nbr neighbours(const HopArgs &a, int p, int j)
{
   const int row = j / a.Lxh;  // row = y + L1*(z + L2*t)
   const int xh = j - row * a.Lxh;
   const int y = row % a.L[1];
   const int zt = row / a.L[1];
   const int z = zt % a.L[2];
   const int t = zt / a.L[2];
   const int x = 2 * xh + ((p + y + z + t) & 1);
   Nbr n;
   const int xp = (x + 1 == a.L[0]) ? 0 : x + 1;
   const int xm = (x == 0) ? a.L[0] - 1 : x - 1;
   n.up[0] = row * a.Lxh + (xp >> 1);
   n.dn[0] = row * a.Lxh + (xm >> 1);
   const int ryp = (y == a.L[1] - 1) ? row - (a.L[1] - 1) : row + 1;
   const int rym = (y == 0) ? row + (a.L[1] - 1) : row - 1;
   const int sz = a.L[1];
   const int rzp = (z == a.L[2] - 1) ? row - (a.L[2] - 1) * sz : row + sz;
   const int rzm = (z == 0) ? row + (a.L[2] - 1) * sz : row - sz;
   const int st = a.L[1] * a.L[2];
   const int rtp = (t == a.L[3] - 1) ? row - (a.L[3] - 1) * st : row + st;
   const int rtm = (t == 0) ? row + (a.L[3] - 1) * st : row - st;
   n.up[1] = ryp * a.Lxh + xh;
   n.dn[1] = rym * a.Lxh + xh;
   n.up[2] = rzp * a.Lxh + xh;
   n.dn[2] = rzm * a.Lxh + xh;
   n.up[3] = rtp * a.Lxh + xh;
   n.dn[3] = rtm * a.Lxh + xh;
   return n;
}

// h = upper((1 - gamma_mu) f): h[0..2] = first colour vector, h[3..5] = second
template <int MU, class C>
__device__ __forceinline__ void proj_minus(const C f[12], C h[6])
{
#pragma unroll
   for (int c = 0; c < 3; c++) {
      if (MU == 0) { h[c] = f[c] + f[6 + c];     h[3 + c] = f[3 + c] + f[9 + c]; }
      if (MU == 1) { h[c] = f[c] + ci(f[9 + c]); h[3 + c] = f[3 + c] + ci(f[6 + c]); }
      if (MU == 2) { h[c] = f[c] + f[9 + c];     h[3 + c] = f[3 + c] - f[6 + c]; }
      if (MU == 3) { h[c] = f[c] + ci(f[6 + c]); h[3 + c] = f[3 + c] - ci(f[9 + c]); }
   }
}
// k = upper((1 + gamma_mu) g)
template <int MU, class C>
__device__ __forceinline__ void proj_plus(const C g[12], C k[6])
{
#pragma unroll
   for (int c = 0; c < 3; c++) {
      if (MU == 0) { k[c] = g[c] - g[6 + c];     k[3 + c] = g[3 + c] - g[9 + c]; }
      if (MU == 1) { k[c] = g[c] - ci(g[9 + c]); k[3 + c] = g[3 + c] - ci(g[6 + c]); }
      if (MU == 2) { k[c] = g[c] - g[9 + c];     k[3 + c] = g[3 + c] + g[6 + c]; }
      if (MU == 3) { k[c] = g[c] - ci(g[6 + c]); k[3 + c] = g[3 + c] + ci(g[9 + c]); }
   }
}
// acc += forward reconstruction of a (lower components only if LOWER)
template <int MU, bool LOWER, class C>
__device__ __forceinline__ void recon_minus(C acc[12], const C a[6])
{
#pragma unroll
   for (int c = 0; c < 3; c++) {
      acc[c] += a[c];
      acc[3 + c] += a[3 + c];
      if (LOWER) {
         if (MU == 0) { acc[6 + c] += a[c];          acc[9 + c] += a[3 + c]; }
         if (MU == 1) { acc[6 + c] -= ci(a[3 + c]); acc[9 + c] -= ci(a[c]); }
         if (MU == 2) { acc[6 + c] -= a[3 + c];     acc[9 + c] += a[c]; }
         if (MU == 3) { acc[6 + c] -= ci(a[c]);     acc[9 + c] += ci(a[3 + c]); }
      }
   }
}
template <int MU, class C>
__device__ __forceinline__ void recon_plus(C acc[12], const C b[6])
{
#pragma unroll
   for (int c = 0; c < 3; c++) {
      acc[c] += b[c];
      acc[3 + c] += b[3 + c];
      if (MU == 0) { acc[6 + c] -= b[c];          acc[9 + c] -= b[3 + c]; }
      if (MU == 1) { acc[6 + c] += ci(b[3 + c]); acc[9 + c] += ci(b[c]); }
      if (MU == 2) { acc[6 + c] += b[3 + c];     acc[9 + c] -= b[c]; }
      if (MU == 3) { acc[6 + c] += ci(b[c]);     acc[9 + c] -= ci(b[3 + c]); }
   }
}

// r = U v for the two colour vectors of a half-spinor
template <class C>
__device__ __forceinline__ void mul_u(const C u[9], const C v[6], C r[6])
{
#pragma unroll
   for (int s = 0; s < 2; s++)
#pragma unroll
      for (int a = 0; a < 3; a++) {
         C t = cmul(u[3 * a], v[3 * s]);
         t = cmadd(u[3 * a + 1], v[3 * s + 1], t);
         r[3 * s + a] = cmadd(u[3 * a + 2], v[3 * s + 2], t);
      }
}
// r = U^+ v
template <class C>
__device__ __forceinline__ void mul_udag(const C u[9], const C v[6], C r[6])
{
#pragma unroll
   for (int s = 0; s < 2; s++)
#pragma unroll
      for (int a = 0; a < 3; a++) {
         C t = cmul(cconj(u[a]), v[3 * s]);
         t = cjmadd(u[3 + a], v[3 * s + 1], t);
         r[3 * s + a] = cjmadd(u[6 + a], v[3 * s + 2], t);
      }
}

// (1 + SIGN gamma_mu) projection and reconstruction, SIGN = -1 or +1
template <int MU, int SIGN, class C>
__device__ __forceinline__ void proj(const C f[12], C h[6])
{
   if (SIGN < 0) proj_minus<MU>(f, h);
   else proj_plus<MU>(f, h);
}
template <int MU, int SIGN, bool LOWER, class C>
__device__ __forceinline__ void recon(C acc[12], const C a[6])
{
   if (SIGN < 0) recon_minus<MU, LOWER>(acc, a);
   else recon_plus<MU>(acc, a);
}

// ---------------------------------------------------------------- terms
//
// term_u:    r = U (1 + SG gamma_mu) f        (a forward term, before recon)
// term_udag: r = U^+ (1 + SG gamma_mu) f      (a backward term)
// accum:     acc += reconstruction of r
// on the held forms of fields.h.  F64 and F32 project, multiply and add in
// the working precision.

template <int MU, int SG, class C>
__device__ __forceinline__ void term_u(const SpinV<C> &f, const LinkV<C> &u, HalfV<C> &r)
{
   C h[6];
   proj<MU, SG>(f.e, h);
   mul_u(u.e, h, r.e);
}
template <int MU, int SG, class C>
__device__ __forceinline__ void term_udag(const SpinV<C> &f, const LinkV<C> &u, HalfV<C> &r)
{
   C h[6];
   proj<MU, SG>(f.e, h);
   mul_udag(u.e, h, r.e);
}
template <int MU, int SG, bool LOWER, class C>
__device__ __forceinline__ void accum(C acc[12], const HalfV<C> &r)
{
   recon<MU, SG, LOWER>(acc, r.e);
}

// F16: the projection adds stored half pairs of one site (one v_pk_add_f16
// per half-spinor component; sign changes and the factor i are operand
// modifiers), the SU(3) multiply is v_dot2_f32_f16 on half pairs with float
// accumulation, and the site scale of the neighbour multiplies the float
// result as it is accumulated (acc += s * r, one fma per real).  Every kernel
// variant uses these functions, so a site's result does not depend on the
// variant.

// X g for X = 0: +1, 1: -1, 2: +i, 3: -i
template <int X>
__device__ __forceinline__ hh2 xmul(hh2 g)
{
   if (X == 0) return g;
   if (X == 1) return -g;
   if (X == 2) return hh2{-g.y, g.x};
   return hh2{g.y, -g.x};
}

// The projection of proj_minus / proj_plus as h[c] = f[c] + X0 f[P0 + c],
// h[3 + c] = f[3 + c] + X1 f[P1 + c]; the lower rows of the reconstruction
// (recon_minus / recon_plus) as acc[6 + c] += Y2 r[S2 + c], acc[9 + c] +=
// Y3 r[S3 + c] (factors coded as in xmul).
template <int MU, int SG>
struct SpinTab {
   static constexpr int P0 = (MU == 0 || MU == 3) ? 6 : 9;
   static constexpr int P1 = 15 - P0;
   static constexpr int X0 = ((MU == 0 || MU == 2) ? 0 : 2) ^ (SG > 0);
   static constexpr int X1 = (MU == 0 ? 0 : MU == 1 ? 2 : MU == 2 ? 1 : 3) ^ (SG > 0);
   static constexpr int S2 = (MU == 0 || MU == 3) ? 0 : 3;
   static constexpr int S3 = 3 - S2;
   static constexpr int Y2 = (MU == 0 ? 0 : MU == 1 ? 3 : MU == 2 ? 1 : 3) ^ (SG > 0);
   static constexpr int Y3 = (MU == 0 ? 0 : MU == 1 ? 3 : MU == 2 ? 0 : 2) ^ (SG > 0);
};

// h = upper((1 + SG gamma_mu) f) in halves, and its swapped pairs (h.im, h.re)
template <int MU, int SG>
__device__ __forceinline__ void proj_h(const SpinH &f, hh2 h[6], hh2 hs[6])
{
   typedef SpinTab<MU, SG> T;
#pragma unroll
   for (int c = 0; c < 3; c++) {
      h[c] = f.h(c) + xmul<T::X0>(f.h(T::P0 + c));
      h[3 + c] = f.h(3 + c) + xmul<T::X1>(f.h(T::P1 + c));
      hs[c] = hswap(h[c]);
      hs[3 + c] = hswap(h[3 + c]);
   }
}

// One colour vector (h, hs = hswap(h)) times U (DAG false) or U^+ (DAG
// true), r = (re, im) of the 3 result colours, as one assembly block of 18
// v_dot2_f32_f16 (see fields.h for why assembly and the closing s_nop):
//   U h:   re_a = sum_b U_ab . (h_b.re, -h_b.im)   im_a = sum_b U_ab . hs_b
//   U^+ h: re_a = sum_b U_ba . h_b                  im_a = sum_b U_ba . (hs_b.re, -hs_b.im)
template <bool DAG>
__device__ __forceinline__ void mat_h(const LinkH &u, const hh2 h[3], const hh2 hs[3], float r[6])
{
   // operands: %0..%5 re0 im0 re1 im1 re2 im2, %6..%14 u_k (k = 3 row + col),
   // %15..%17 h, %18..%20 hs
   if constexpr (!DAG) {
      asm(PLQCD_D2Z("%0", "%6", "%15", PLQCD_NHI)
          PLQCD_D2Z("%1", "%6", "%18", "")
          PLQCD_D2Z("%2", "%9", "%15", PLQCD_NHI)
          PLQCD_D2Z("%3", "%9", "%18", "")
          PLQCD_D2Z("%4", "%12", "%15", PLQCD_NHI)
          PLQCD_D2Z("%5", "%12", "%18", "")
          PLQCD_D2("%0", "%7", "%16", PLQCD_NHI)
          PLQCD_D2("%1", "%7", "%19", "")
          PLQCD_D2("%2", "%10", "%16", PLQCD_NHI)
          PLQCD_D2("%3", "%10", "%19", "")
          PLQCD_D2("%4", "%13", "%16", PLQCD_NHI)
          PLQCD_D2("%5", "%13", "%19", "")
          PLQCD_D2("%0", "%8", "%17", PLQCD_NHI)
          PLQCD_D2("%1", "%8", "%20", "")
          PLQCD_D2("%2", "%11", "%17", PLQCD_NHI)
          PLQCD_D2("%3", "%11", "%20", "")
          PLQCD_D2("%4", "%14", "%17", PLQCD_NHI)
          PLQCD_D2("%5", "%14", "%20", "")
          "s_nop 2"
          : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5])
          : "v"(u.h(0)), "v"(u.h(1)), "v"(u.h(2)), "v"(u.h(3)), "v"(u.h(4)), "v"(u.h(5)), "v"(u.h(6)),
            "v"(u.h(7)), "v"(u.h(8)), "v"(h[0]), "v"(h[1]), "v"(h[2]), "v"(hs[0]), "v"(hs[1]), "v"(hs[2]));
   } else {
      asm(PLQCD_D2Z("%0", "%6", "%15", "")
          PLQCD_D2Z("%1", "%6", "%18", PLQCD_NHI)
          PLQCD_D2Z("%2", "%7", "%15", "")
          PLQCD_D2Z("%3", "%7", "%18", PLQCD_NHI)
          PLQCD_D2Z("%4", "%8", "%15", "")
          PLQCD_D2Z("%5", "%8", "%18", PLQCD_NHI)
          PLQCD_D2("%0", "%9", "%16", "")
          PLQCD_D2("%1", "%9", "%19", PLQCD_NHI)
          PLQCD_D2("%2", "%10", "%16", "")
          PLQCD_D2("%3", "%10", "%19", PLQCD_NHI)
          PLQCD_D2("%4", "%11", "%16", "")
          PLQCD_D2("%5", "%11", "%19", PLQCD_NHI)
          PLQCD_D2("%0", "%12", "%17", "")
          PLQCD_D2("%1", "%12", "%20", PLQCD_NHI)
          PLQCD_D2("%2", "%13", "%17", "")
          PLQCD_D2("%3", "%13", "%20", PLQCD_NHI)
          PLQCD_D2("%4", "%14", "%17", "")
          PLQCD_D2("%5", "%14", "%20", PLQCD_NHI)
          "s_nop 2"
          : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5])
          : "v"(u.h(0)), "v"(u.h(1)), "v"(u.h(2)), "v"(u.h(3)), "v"(u.h(4)), "v"(u.h(5)), "v"(u.h(6)),
            "v"(u.h(7)), "v"(u.h(8)), "v"(h[0]), "v"(h[1]), "v"(h[2]), "v"(hs[0]), "v"(hs[1]), "v"(hs[2]));
   }
}

template <int MU, int SG>
__device__ __forceinline__ void term_u(const SpinH &f, const LinkH &u, HalfH &r)
{
   hh2 h[6], hs[6];
   proj_h<MU, SG>(f, h, hs);
   mat_h<false>(u, h, hs, r.e);
   mat_h<false>(u, h + 3, hs + 3, r.e + 6);
   r.e[12] = f.s();
}

template <int MU, int SG>
__device__ __forceinline__ void term_udag(const SpinH &f, const LinkH &u, HalfH &r)
{
   hh2 h[6], hs[6];
   proj_h<MU, SG>(f, h, hs);
   mat_h<true>(u, h, hs, r.e);
   mat_h<true>(u, h + 3, hs + 3, r.e + 6);
   r.e[12] = f.s();
}

// acc += s * Y (x + i y), Y coded as in xmul
template <int Y>
__device__ __forceinline__ void acc_add(f2 &acc, float s, float x, float y)
{
   if (Y == 0) { acc.x = fma(s, x, acc.x);  acc.y = fma(s, y, acc.y); }
   if (Y == 1) { acc.x = fma(-s, x, acc.x); acc.y = fma(-s, y, acc.y); }
   if (Y == 2) { acc.x = fma(-s, y, acc.x); acc.y = fma(s, x, acc.y); }
   if (Y == 3) { acc.x = fma(s, y, acc.x);  acc.y = fma(-s, x, acc.y); }
}

// recon_minus (SG < 0; lower rows only if LOWER) / recon_plus (SG > 0)
template <int MU, int SG, bool LOWER>
__device__ __forceinline__ void accum(f2 acc[12], const HalfH &r)
{
   typedef SpinTab<MU, SG> T;
   const float s = r.e[12];
#pragma unroll
   for (int c = 0; c < 3; c++) {
      acc_add<0>(acc[c], s, r.e[2 * c], r.e[2 * c + 1]);
      acc_add<0>(acc[3 + c], s, r.e[2 * (3 + c)], r.e[2 * (3 + c) + 1]);
      if (SG > 0 || LOWER) {
         acc_add<T::Y2>(acc[6 + c], s, r.e[2 * (T::S2 + c)], r.e[2 * (T::S2 + c) + 1]);
         acc_add<T::Y3>(acc[9 + c], s, r.e[2 * (T::S3 + c)], r.e[2 * (T::S3 + c) + 1]);
      }
   }
}

// Forward term of direction MU for output site (p, j); jnb = site of x+mu.
// H uses (1 - gamma_mu) forward and (1 + gamma_mu) backward; the adjoint
// H^+ = gamma5 H gamma5 has the signs swapped (gamma5 anticommutes with
// gamma_mu), so DAG only flips the projector signs.
// NT: streaming link loads.
template <int MU, int MODE, bool DAG, bool NT = false, class SIO, class GIO>
__device__ __forceinline__ void hop_fwd(const SIO &in, const GIO &g, int p, int j, int jnb, typename SIO::C acc[12])
{
   constexpr int SG = DAG ? 1 : -1;
   typename SIO::Sp f;
   typename GIO::U u;
   typename SIO::Hv r;
   in.load_sp(1 - p, jnb, f);
   g.template load_u<NT>(MODE == MODE_COMPAT ? 0 : p, MU, j, u);
   term_u<MU, SG>(f, u, r);
   accum<MU, SG, MODE != MODE_COMPAT>(acc, r);
}

// Backward term of direction MU; jnb = site of x-mu (its link U_mu(x-mu) too).
template <int MU, bool DAG, bool NT = false, class SIO, class GIO>
__device__ __forceinline__ void hop_bwd(const SIO &in, const GIO &g, int p, int jnb, typename SIO::C acc[12])
{
   constexpr int SG = DAG ? -1 : 1;
   typename SIO::Sp f;
   typename GIO::U u;
   typename SIO::Hv r;
   in.load_sp(1 - p, jnb, f);
   g.template load_u<NT>(1 - p, MU, jnb, u);
   term_udag<MU, SG>(f, u, r);
   accum<MU, SG, true>(acc, r);
}

template <int MU, int MODE, bool DAG, bool NT = false, class SIO, class GIO>
__device__ __forceinline__ void hop_dir(const SIO &in, const GIO &g, int p, int j, const Nbr &n,
                                        typename SIO::C acc[12])
{
   hop_fwd<MU, MODE, DAG, NT>(in, g, p, j, n.up[MU], acc);
   hop_bwd<MU, DAG, NT>(in, g, p, n.dn[MU], acc);
}

// Maps the hardware block index to a logical tile.  Blocks are handed to
// the 8 XCDs round-robin (block b runs on XCD b % 8), and each XCD has its
// own L2, so the order decides which L2 sees which part of the lattice:
//   order 0: logical = b
//   order 1: XCD k takes the k-th contiguous eighth of the lattice (eighths
//            differ by one block where the block count is no multiple of 8)
//   order 2: the lattice is cut into chunks of 8*group logical blocks; XCD k
//            takes the k-th run of `group` blocks of every chunk, so all XCDs
//            sweep the lattice together and neighbouring tiles share an L2;
//            the blocks after the last whole chunk are split as in order 1
// Both are one-to-one for every block count.
// The output parity alternates between consecutive logical blocks, so a link
// is read as a forward and as a backward link by nearby tiles.
__device__ __forceinline__ int logical_block(const HopArgs &a)
{
   int b = blockIdx.x, nb = gridDim.x, first = 0;
   if (a.order == 0) return b;
   if (a.order == 2) {
      const int G = a.group;
      first = nb - nb % (8 * G);
      if (b < first) {
         const int q = b >> 3;
         return (q / G) * 8 * G + (b & 7) * G + (q % G);
      }
      b -= first;
      nb -= first;
   }
   const int k = b & 7;
   return first + k * (nb >> 3) + min(k, nb & 7) + (b >> 3);
}

// The RHS of the fields that lane-RHS r of a launch handles: r0 + r, or the
// r-th entry of the launch's RHS list.
__device__ __forceinline__ int rhs_of(const HopArgs &a, int r)
{
   return a.rlist ? a.rlist[r] : a.r0 + r;
}

// Operands of the epilogues: the per-RHS step alpha (EPI = 2), the
// right-hand side b (EPI = 3) and the centre field (EPI = 4).
template <class SIO>
struct CgFuse {
   SIO p;  // EPI 3: b; EPI 4: the centre field
   const double *alpha;
   double kappa[plqcd::kInlineKappa];  // EPI 1 and 4 without norm: the RHS's kappa where HopArgs::kappa is null
};

// Epilogue: EPI = 0 stores H in; EPI = 1 stores in(x) - kappa_r * (H in)(x).
// EPI = 2 forms Ap = in(x) - kappa_r * (H in)(x) in registers and applies the
// CG residual update at the site instead of storing it: out -= alpha_r Ap (out
// holds the residual), in the working precision of the kernel (float for
// F32/F16 storage, double for F64).  The iterate's update x += alpha_r p is
// left to the solver's next pass over p.
// EPI = 3 (F64 storage) stores the residual b - Ap, with b in f.p, in the
// precision of `out`, for every RHS of the launch (the reliable update of the
// mixed-precision CG: the true residual goes straight into the low-precision
// iterate's residual; the solver launches it once per run of consecutive
// RHS being updated).  No per-RHS predicate: a data-dependent condition
// around the stores made the compiler keep both paths' values live (280
// registers, one wave per SIMD, against 144 and three waves).
// EPI = 4 is EPI = 1 with the centre taken from another field, f.p: out =
// c(x) - kappa_r * (H in)(x) (the even-odd operator's second half hop, whose
// input lives on the other parity; half-lattice kernel only).
// With NORM the site's |out|^2 joins the deterministic chunk reduction.  `in`
// and `out` are positioned at the RHS `r`, whose kappa and alpha apply.  `pre`,
// when not null, is the site's spinor of b that EPI 3 reads, loaded earlier.
template <int EPI, bool NORM, class SIO, class SO>
__device__ __forceinline__ double epilogue(const SIO &in, const SO &out, const HopArgs &a, int r, int p, int j,
                                           typename SIO::C acc[12], const typename SIO::C *cen, const CgFuse<SIO> &f,
                                           const typename SIO::Sp *pre = nullptr)
{
   typedef typename SIO::real real;
   typedef typename SIO::C C;
   if (EPI >= 1) {
      C c0[12];
      if constexpr (EPI == 4)
         f.p.at_rhs(r).load(p, j, c0);
      else if (cen == nullptr)
         in.load(p, j, c0);
      const real kap = (real)((EPI == 4 || EPI == 1) && !NORM && !a.kappa ? f.kappa[r] : a.kappa[r]);
#pragma unroll
      for (int m = 0; m < 12; m++) acc[m] = cxmky(cen ? cen[m] : c0[m], kap, acc[m]);
   }
   if constexpr (EPI == 3) {
      const SIO b = f.p.at_rhs(r);
      const uint32_t o = b.off(j);
      d2 rs[12];
      C bs[12];
      if (pre) SIO::to_c(*pre, bs);
#pragma unroll
      for (int m = 0; m < 12; m++) {
         const C bm = pre ? bs[m] : ld<C>(b.cbase(p, m), o);
         rs[m] = d2{(double)bm.x - (double)acc[m].x, (double)bm.y - (double)acc[m].y};
      }
      store_d(out, p, j, rs);
      return NORM ? norm2(rs) : 0.0;
   } else if constexpr (EPI == 2) {
      const real al = (real)f.alpha[r];
      C rs[12];
      out.load(p, j, rs);
      double nrm = 0.0;
#pragma unroll
      for (int m = 0; m < 12; m++) {
         rs[m] = C{fma(-al, acc[m].x, rs[m].x), fma(-al, acc[m].y, rs[m].y)};
         nrm = fma((double)rs[m].y, (double)rs[m].y, fma((double)rs[m].x, (double)rs[m].x, nrm));
      }
      out.store(p, j, rs);
      return NORM ? nrm : 0.0;
   } else {
      double nrm = 0.0;
      if (NORM) {
#pragma unroll
         for (int m = 0; m < 12; m++)
            nrm = fma((double)acc[m].y, (double)acc[m].y, fma((double)acc[m].x, (double)acc[m].x, nrm));
      }
      out.store(p, j, acc);
      return nrm;
   }
}

// One block of the gather kernel: logical block `blk` of the launch.
template <int MODE, bool DAG, int EPI, bool NORM, int BLOCK, class SIO, class GIO, class SO>
__device__ __forceinline__ void hop_block(const SIO &in, const SO &out, const GIO &g, const HopArgs &a, int blk,
                                          const CgFuse<SIO> &f)
{
   typedef typename SIO::C C;
   int p;
   if (a.nparity == 2) {
      p = blk & 1;
      blk >>= 1;
   } else {
      p = a.parity0;
   }
   const int r = threadIdx.x % a.R;
   const int js = threadIdx.x / a.R;
   const int rr = rhs_of(a, r);
   const int j = blk * a.spb + js;
   double nrm = 0.0;
   if (js < a.spb && j < a.Vh) {
      const SIO si = in.at_rhs(rr);
      const SO so = out.at_rhs(rr);
      const Nbr n = neighbours(a, p, j);
      C acc[12];
#pragma unroll
      for (int c = 0; c < 12; c++) acc[c] = C{0, 0};
      hop_dir<0, MODE, DAG>(si, g, p, j, n, acc);
      hop_dir<1, MODE, DAG>(si, g, p, j, n, acc);
      hop_dir<2, MODE, DAG>(si, g, p, j, n, acc);
      hop_dir<3, MODE, DAG>(si, g, p, j, n, acc);
      nrm = epilogue<EPI, NORM>(si, so, a, rr, p, j, acc, (const C *)nullptr, f);
   }
   if (NORM) chunk_reduce<BLOCK>(nrm, js, r, a.R, p * a.nchunk + (blk * a.spb + js) / REDUCE_CHUNK,
                                 j - (js & (REDUCE_CHUNK - 1)) < a.Vh, a.partial + (size_t)rr * 2 * a.nchunk);
}

template <int MODE, bool DAG, int EPI, bool NORM, int BLOCK, class SIO, class GIO, class SO>
__global__ __launch_bounds__(BLOCK) void hop_kernel(SIO in, SO out, GIO g, HopArgs a, CgFuse<SIO> f)
{
   if (NORM && a.halt && *a.halt) return;
   hop_block<MODE, DAG, EPI, NORM, BLOCK>(in, out, g, a, logical_block(a), f);
}

// Half-lattice hop (eo or oe; EPI 0 or 4): the gather kernel's sites and order
// of operations, in block orders and with link loads for one parity.
//   It is bound by the bytes its L2s miss: each link is used once, and a
// spinor by eight sites, so what the L2 holds should be spinors.  NT streams
// the links past it; order 3 gives XCD k the k-th eighth of the column blocks
// of a t-slice (a slab in z), swept through all t-slices, so that a spinor's t
// neighbours find it in the L2 too.  us per half, F64: 32^3 x 64 364 -> 316
// (NT; 1.6 GB compulsory, 5.1 TB/s), 28 x 20 x 36 x 44 152 -> 133 (NT), 24^3 x
// 48 with 4 RHS 281 -> 256 (both), with 12 RHS 753 -> 648 (order 3).
template <int MODE, int EPI, bool NT, int BLOCK, class SIO, class GIO>
__global__ __launch_bounds__(BLOCK) void hop_half_kernel(SIO in, SIO out, GIO g, HopArgs a, CgFuse<SIO> f)
{
   typedef typename SIO::C C;
   const int p = a.parity0;
   const int r = threadIdx.x % a.R;
   const int js = threadIdx.x / a.R;
   const int rr = rhs_of(a, r);
   int j, end;  // the lane's site; the first one past its block's t-slice (order 3) or the parity
   if (a.order == 3) {
      const int nbS = (a.S + a.spb - 1) / a.spb;
      const int k = blockIdx.x & 7, i = blockIdx.x >> 3;
      const int n = (nbS >> 3) + (k < (nbS & 7)), first = k * (nbS >> 3) + min(k, nbS & 7);
      const int t = i / n;
      j = t * a.S + (first + i - t * n) * a.spb + js;
      end = t < a.L[3] ? (t + 1) * a.S : 0;
   } else {
      j = logical_block(a) * a.spb + js;
      end = a.Vh;
   }
   if (js >= a.spb || j >= end) return;
   const SIO si = in.at_rhs(rr);
   const Nbr n = neighbours(a, p, j);
   C acc[12];
#pragma unroll
   for (int c = 0; c < 12; c++) acc[c] = C{0, 0};
   hop_dir<0, MODE, false, NT>(si, g, p, j, n, acc);
   hop_dir<1, MODE, false, NT>(si, g, p, j, n, acc);
   hop_dir<2, MODE, false, NT>(si, g, p, j, n, acc);
   hop_dir<3, MODE, false, NT>(si, g, p, j, n, acc);
   epilogue<EPI, false>(si, out.at_rhs(rr), a, rr, p, j, acc, (const C *)nullptr, f);
}

// RHS-blocked gather: each lane handles RB consecutive right-hand sides of
// one site, so a link is loaded (and, with 12-real links, rebuilt) once per
// RB right-hand sides.  Lanes per site G = R / RB.  Every RHS goes through
// the same operation sequence as in hop_block.
template <int MODE, bool DAG, int EPI, bool NORM, int BLOCK, int RB, class SIO, class GIO>
__device__ __forceinline__ void hop_block_rb(const SIO &in, const SIO &out, const GIO &g, const HopArgs &a, int blk,
                                             const CgFuse<SIO> &f)
{
   typedef typename SIO::C C;
   constexpr int SF = DAG ? 1 : -1, SB = -SF;
   int p;
   if (a.nparity == 2) {
      p = blk & 1;
      blk >>= 1;
   } else {
      p = a.parity0;
   }
   const int G = a.R / RB;
   const int gi = threadIdx.x % G;
   const int js = threadIdx.x / G;
   const int j = blk * a.spb + js;
   double nrm[RB];
#pragma unroll
   for (int k = 0; k < RB; k++) nrm[k] = 0.0;
   if (js < a.spb && j < a.Vh) {
      const Nbr n = neighbours(a, p, j);
      C acc[RB][12];
#pragma unroll
      for (int k = 0; k < RB; k++)
#pragma unroll
         for (int c = 0; c < 12; c++) acc[k][c] = C{0, 0};
      const SIO si = in.at_rhs(rhs_of(a, gi * RB));
#define PLQCD_RB_DIR(MU)                                                                      \
   {                                                                                          \
      typename GIO::U u;                                                                      \
      g.load_u(MODE == MODE_COMPAT ? 0 : p, MU, j, u);                                        \
      _Pragma("unroll") for (int k = 0; k < RB; k++)                                          \
      {                                                                                       \
         typename SIO::Sp f;                                                                  \
         typename SIO::Hv r;                                                                  \
         si.at_rhs(rhs_of(a, gi * RB + k)).load_sp(1 - p, n.up[MU], f);                           \
         term_u<MU, SF>(f, u, r);                                                             \
         accum<MU, SF, MODE != MODE_COMPAT>(acc[k], r);                                       \
      }                                                                                       \
      g.load_u(1 - p, MU, n.dn[MU], u);                                                       \
      _Pragma("unroll") for (int k = 0; k < RB; k++)                                          \
      {                                                                                       \
         typename SIO::Sp f;                                                                  \
         typename SIO::Hv r;                                                                  \
         si.at_rhs(rhs_of(a, gi * RB + k)).load_sp(1 - p, n.dn[MU], f);                           \
         term_udag<MU, SB>(f, u, r);                                                          \
         accum<MU, SB, true>(acc[k], r);                                                      \
      }                                                                                       \
   }
      PLQCD_RB_DIR(0)
      PLQCD_RB_DIR(1)
      PLQCD_RB_DIR(2)
      PLQCD_RB_DIR(3)
#undef PLQCD_RB_DIR
#pragma unroll
      for (int k = 0; k < RB; k++)
         nrm[k] = epilogue<EPI, NORM>(in.at_rhs(rhs_of(a, gi * RB + k)), out.at_rhs(rhs_of(a, gi * RB + k)), a,
                                      rhs_of(a, gi * RB + k), p, j, acc[k],
                                      (const C *)nullptr, f);
   }
   if (NORM) {
#pragma unroll
      for (int k = 0; k < RB; k++)
         chunk_reduce<BLOCK>(nrm[k], js, gi, G, p * a.nchunk + (blk * a.spb + js) / REDUCE_CHUNK,
                             j - (js & (REDUCE_CHUNK - 1)) < a.Vh,
                             a.partial + (size_t)(rhs_of(a, gi * RB + k)) * 2 * a.nchunk, k);
   }
}

template <int MODE, bool DAG, int EPI, bool NORM, int BLOCK, int RB, class SIO, class GIO>
__global__ __launch_bounds__(BLOCK) void hop_rb_kernel(SIO in, SIO out, GIO g, HopArgs a, CgFuse<SIO> f)
{
   if (NORM && a.halt && *a.halt) return;
   hop_block_rb<MODE, DAG, EPI, NORM, BLOCK, RB>(in, out, g, a, logical_block(a), f);
}

// First t-slice of t-chunk k of the marching kernels: the time extent is cut
// into a.nt chunks whose lengths differ by at most one slice, so any chunk
// count serves any extent.
__device__ __forceinline__ int chunk_t0(const HopArgs &a, int k)
{
   return (int)((long long)k * a.L[3] / a.nt);
}

// One application of H on each of several independent lattices (each with its
// own gauge field and fields) in a single launch over the concatenated
// logical blocks of the items.
template <class SIO, class GIO>
struct BatchItem {
   SIO in, out;
   GIO g;
   HopArgs a;
   int first;  // first global block of this item
   int nb;     // blocks of this item
};
// A launch takes up to kBatchItems items by value, as a kernel argument (no
// device copy of the list); longer batches take several launches.
constexpr int kBatchItems = 16;
constexpr int kBatchGroup = 8;  // consecutive logical blocks an XCD takes in a ragged batch
template <class SIO, class GIO>
struct BatchList {
   BatchItem<SIO, GIO> it[kBatchItems];
};

// t-march variant (full lattice, either mode): a thread owns one (x,y,z)
// column and walks the consecutive t-slices of one of a.nt balanced chunks of
// the time extent.  Along t each spinor and each U_t
// is loaded once: psi(t+1), read as the forward t-neighbour at step t, is kept
// (it is the centre site of step t+1) and its projection, multiplied by
// U_t(t+1)^+ at step t+1 (that step's forward link), gives the backward
// t-term of step t+2.  The spatial directions read their neighbours from L2
// as the gather kernel does.  The site parity alternates from step to step;
// the index of the site inside its parity advances by S = L0/2*L1*L2 per
// t-slice.  Terms are accumulated in the same order as in hop_kernel.
template <int MODE, bool DAG, int EPI, bool NORM, int BLOCK, class SIO, class GIO, class SO>
__device__ __forceinline__ void hop_tmarch_block(const SIO &in, const SO &out, const GIO &g, const HopArgs &a, int lb,
                                                 const CgFuse<SIO> &fuse)
{
   typedef typename SIO::C C;
   constexpr int SF = DAG ? 1 : -1;  // forward projector sign
   const int S = a.S;
   const int nbS = (S + a.spb - 1) / a.spb;
   const int q = lb & 1;  // parity of the column's first site
   lb >>= 1;
   const int sb = lb % nbS;
   const int chunk = lb / nbS;
   const int r = threadIdx.x % a.R;
   const int js = threadIdx.x / a.R;
   const int rr = rhs_of(a, r);
   const int c = sb * a.spb + js;
   const bool valid = js < a.spb && c < S;  // a batch block may have spare lanes
   const SIO si = in.at_rhs(rr);
   const SO so = out.at_rhs(rr);

   const int t0 = chunk_t0(a, chunk), nts = chunk_t0(a, chunk + 1) - t0;
   const int cc = valid ? c : 0;
   const int row = cc / a.Lxh;  // y + L1*z
   const int xh = cc - row * a.Lxh;
   const int y = row % a.L[1];
   const int z = row / a.L[1];
   const int x = 2 * xh + ((q + y + z + t0) & 1);
   int cu[3], cd[3];
   {
      const int xp = (x + 1 == a.L[0]) ? 0 : x + 1;
      const int xm = (x == 0) ? a.L[0] - 1 : x - 1;
      cu[0] = row * a.Lxh + (xp >> 1);
      cd[0] = row * a.Lxh + (xm >> 1);
      const int ryp = (y == a.L[1] - 1) ? row - (a.L[1] - 1) : row + 1;
      const int rym = (y == 0) ? row + (a.L[1] - 1) : row - 1;
      const int rzp = (z == a.L[2] - 1) ? row - (a.L[2] - 1) * a.L[1] : row + a.L[1];
      const int rzm = (z == 0) ? row + (a.L[2] - 1) * a.L[1] : row - a.L[1];
      cu[1] = ryp * a.Lxh + xh;
      cd[1] = rym * a.Lxh + xh;
      cu[2] = rzp * a.Lxh + xh;
      cd[2] = rzm * a.Lxh + xh;
   }
   const int Lt = a.L[3];
   typedef typename SIO::Sp Sp;
   typedef typename SIO::Hv Hv;
   Sp cen;  // the lane's centre spinor and backward t term live across t-slices
   Hv b;
   // prologue: cen = psi(t0); b = U_t(t0-1)^+ (1 -+ g_t) psi(t0-1)
   if (valid) {
      Sp f;
      typename GIO::U u;
      si.load_sp(q, c + t0 * S, cen);
      const int tm = (t0 == 0 ? Lt : t0) - 1;
      si.load_sp(q ^ 1, c + tm * S, f);
      g.load_u(q ^ 1, 3, c + tm * S, u);
      term_udag<3, -SF>(f, u, b);
   }
   for (int s = 0; s < nts; s++) {
      const int t = t0 + s;
      const int p = q ^ (s & 1);
      const int base = t * S;
      const int j = cc + base;
      double nrm = 0.0;
      if (valid) {
         C acc[12];
#pragma unroll
         for (int m = 0; m < 12; m++) acc[m] = C{0, 0};
         hop_fwd<0, MODE, DAG>(si, g, p, j, cu[0] + base, acc);
         hop_bwd<0, DAG>(si, g, p, cd[0] + base, acc);
         hop_fwd<1, MODE, DAG>(si, g, p, j, cu[1] + base, acc);
         hop_bwd<1, DAG>(si, g, p, cd[1] + base, acc);
         hop_fwd<2, MODE, DAG>(si, g, p, j, cu[2] + base, acc);
         hop_bwd<2, DAG>(si, g, p, cd[2] + base, acc);
         Sp f;
         {
            typename GIO::U u;
            Hv rr;
            const int tp = (t + 1 == Lt) ? 0 : t + 1;
            si.load_sp(p ^ 1, c + tp * S, f);
            // U_t(t) serves this slice's forward and the next slice's
            // backward t term from registers and no other block reads it: a
            // streaming load (FP16 with one RHS 6-9 % faster at 32^3 x 64,
            // 12 RHS under 1 % slower; choosing by R at run time cost the
            // one-RHS kernel its gain).  Compat mode's forward term takes the
            // even site's link with the same index, a second load.
            g.template load_u<true>(p, 3, j, u);
            if constexpr (MODE == MODE_COMPAT) {
               typename GIO::U uf;
               g.load_u(0, 3, j, uf);
               term_u<3, SF>(f, uf, rr);
            } else {
               term_u<3, SF>(f, u, rr);
            }
            accum<3, SF, MODE != MODE_COMPAT>(acc, rr);
            accum<3, -SF, true>(acc, b);
            term_udag<3, -SF>(cen, u, b);
         }
         if (EPI >= 1) {
            C cv[12];
            SIO::to_c(cen, cv);
            nrm = epilogue<EPI, NORM>(si, so, a, rr, p, j, acc, cv, fuse);
         } else {
            nrm = epilogue<EPI, NORM>(si, so, a, rr, p, j, acc, (const C *)nullptr, fuse);
         }
         cen = f;
      }
      if (NORM) chunk_reduce<BLOCK>(nrm, js, r, a.R, p * a.nchunk + (sb * a.spb + js + base) / REDUCE_CHUNK, valid,
                                    a.partial + (size_t)rr * 2 * a.nchunk, s);
   }
}

template <int MODE, bool DAG, int EPI, bool NORM, int BLOCK, class SIO, class GIO, class SO>
__global__ __launch_bounds__(BLOCK) void hop_tmarch_kernel(SIO in, SO out, GIO g, HopArgs a, CgFuse<SIO> fuse)
{
   if (NORM && a.halt && *a.halt) return;
   hop_tmarch_block<MODE, DAG, EPI, NORM, BLOCK>(in, out, g, a, logical_block(a), fuse);
}

// ------------------------------------------------- several right-hand sides
//
// Links of the pipelined t-march, in LDS: slot (buffer, direction, site of the
// block), link_slot bytes each, two buffers.
template <class GIO>
constexpr int link_slot()
{
   return (9 * (int)sizeof(typename GIO::U::E) + 15) / 16 * 16;
}
// Links a site needs per t-slice: forward x y z t, backward x y z (the
// backward t term is formed one slice earlier), and in compat mode the true
// U_t beside the even site's.
template <int MODE>
constexpr int links_per_slice()
{
   return MODE == MODE_COMPAT ? 8 : 7;
}
template <int MODE, class GIO>
constexpr size_t pipe_lds_bytes(int spb)
{
   return (size_t)2 * links_per_slice<MODE>() * spb * link_slot<GIO>();
}

// Computes the accumulators here: without it the compiler moves the products
// of a whole slice down to the stores they end in, behind every load.
template <class C>
__device__ __forceinline__ void pin(C acc[12])
{
   asm volatile("" : "+v"(acc[0].x), "+v"(acc[0].y), "+v"(acc[1].x), "+v"(acc[1].y), "+v"(acc[2].x), "+v"(acc[2].y),
                "+v"(acc[3].x), "+v"(acc[3].y), "+v"(acc[4].x), "+v"(acc[4].y), "+v"(acc[5].x), "+v"(acc[5].y));
   asm volatile("" : "+v"(acc[6].x), "+v"(acc[6].y), "+v"(acc[7].x), "+v"(acc[7].y), "+v"(acc[8].x), "+v"(acc[8].y),
                "+v"(acc[9].x), "+v"(acc[9].y), "+v"(acc[10].x), "+v"(acc[10].y), "+v"(acc[11].x), "+v"(acc[11].y));
}

// Pipelined t-march for several right-hand sides (full lattice, either mode):
// hop_tmarch_kernel's columns, chunks, lanes and order of operations, with the
// loads taken off the lanes' critical path.
//   Links: the R lanes of a site need the same links, so each link of a slice
// is loaded (and, with 12-real links, rebuilt) by one lane of the block, a
// slice ahead, and read by all from LDS; a lane loads NIT links per slice
// instead of 7.
//   Spinors: the neighbours x+ x- y+ y- z+ z- pass through a ring of three
// register sets, so the next two to three are in flight while one is
// multiplied, across the slice boundary too; psi(t+1) and EPI 3's b
// are loaded in the middle of the slice.
// The loads ahead read only `in`, b and links, so any may be issued before the
// slice's barrier.
//   Blocks: with several right-hand sides an XCD's L2 holds the t-slices of
// few columns, and what a block reads beyond them counts, so consecutive
// blocks (the run of one XCD in block order 2) form a patch of gy x gz column
// blocks in y and z (a.gy = 0: no patches).
//   Bound by the bytes its L2s miss.  32^3 x 64, 12 RHS, us per H, against
// hop_tmarch_kernel: F64 4242 -> 3360 (17.3 GB missed, 10.9 GB compulsory,
// 5.2 TB/s), F32 12-real 1753 -> 1590 (8.9 and 5.2 GB, 5.6 TB/s), F16 12-real
// 957 -> 895 (4.5 and 2.8 GB, 5.0 TB/s; vector instructions alone take 500 us).
// 24^3 x 48, 12 RHS, the solver's FP64 operators: M 1497 -> 1127 us, the
// residual of EPI 3 1540 -> 1265 (1924 without b loaded ahead).
// Patches: 24^3 x 48 F64 1127 -> 1032, F32 526 -> 491, F16 303 -> 291.
template <int MODE, bool DAG, int EPI, bool NORM, int BLOCK, int NIT, class SIO, class GIO, class SO>
__device__ __forceinline__ void hop_pipe_block(const SIO &in, const SO &out, const GIO &g, const HopArgs &a, int lb,
                                               const CgFuse<SIO> &fuse)
{
   typedef typename SIO::C C;
   typedef typename SIO::Sp Sp;
   typedef typename SIO::Hv Hv;
   typedef typename GIO::U U;
   constexpr int SF = DAG ? 1 : -1;  // forward projector sign
   constexpr bool compat = MODE == MODE_COMPAT;
   constexpr int NL = links_per_slice<MODE>();
   constexpr int LS = link_slot<GIO>();
   // EPI 3's b is loaded ahead, EPI 2's residual is not: in F16 it costs the
   // third wave (12-RHS CG at 24^3 x 48 91 against 82 ms), in F32 nothing
   // (119.5 against 118.5 ms), in F64 it spills
   constexpr bool PRE = EPI == 3;
   extern __shared__ char lk[];  // [2][NL][spb][LS]
   const int S = a.S;
   const int nbS = (S + a.spb - 1) / a.spb;
   const int q = lb & 1;  // parity of the column's first site
   lb >>= 1;
   int sb = lb % nbS;
   const int chunk = lb / nbS;
   if (a.gy > 0) {
      const int nby = a.Lxh * a.L[1] / a.spb, area = a.gy * a.gz;
      const int patch = sb / area, w = sb - patch * area, py = nby / a.gy;
      sb = (patch % py) * a.gy + w % a.gy + nby * ((patch / py) * a.gz + w / a.gy);
   }
   const int tid = threadIdx.x;
   const int r = tid % a.R;
   const int js = tid / a.R;
   const int rr = rhs_of(a, r);
   const int c = sb * a.spb + js;
   // lanes past the block's sites (a batch block may have some) or past the
   // last column work on site 0 or column 0 and store nothing
   const bool valid = js < a.spb && c < S;
   const int jl = js < a.spb ? js : 0;
   const SIO si = in.at_rhs(rr);
   const SO so = out.at_rhs(rr);
   const int t0 = chunk_t0(a, chunk), nts = chunk_t0(a, chunk + 1) - t0;
   const int Lt = a.L[3];
   const int cc = valid ? c : 0;
   // columns of the x, y, z neighbours (up, down) of column `col`
   auto nbr_cols = [&](int col, int n[6]) {
      const int row = col / a.Lxh;  // y + L1*z
      const int xh = col - row * a.Lxh;
      const int y = row % a.L[1];
      const int z = row / a.L[1];
      const int x = 2 * xh + ((q + y + z + t0) & 1);  // the same at every t-slice
      const int xp = (x + 1 == a.L[0]) ? 0 : x + 1;
      const int xm = (x == 0) ? a.L[0] - 1 : x - 1;
      n[0] = row * a.Lxh + (xp >> 1);
      n[1] = row * a.Lxh + (xm >> 1);
      const int ryp = (y == a.L[1] - 1) ? row - (a.L[1] - 1) : row + 1;
      const int rym = (y == 0) ? row + (a.L[1] - 1) : row - 1;
      const int rzp = (z == a.L[2] - 1) ? row - (a.L[2] - 1) * a.L[1] : row + a.L[1];
      const int rzm = (z == 0) ? row + (a.L[2] - 1) * a.L[1] : row - a.L[1];
      n[2] = ryp * a.Lxh + xh;
      n[3] = rym * a.Lxh + xh;
      n[4] = rzp * a.Lxh + xh;
      n[5] = rzm * a.Lxh + xh;
   };
   int cn[6];
   nbr_cols(cc, cn);
   // the links this lane fetches: slot index, direction, parity relative to
   // the site's (0 the site's, 1 the other; -1: always even) and column
   int lslot[NIT], lmu[NIT], lpar[NIT], lcol[NIT];
#pragma unroll
   for (int i = 0; i < NIT; i++) {
      const int n = tid + i * (int)blockDim.x;
      const int d = n / a.spb, s = n - d * a.spb;
      lslot[i] = n < NL * a.spb ? n : -1;  // a lane without a link loads one all the same
      int ln[6];
      const int col = sb * a.spb + s < S ? sb * a.spb + s : 0;
      nbr_cols(col, ln);
      // slots: 0 x+  1 x-  2 y+  3 y-  4 z+  5 z-  6 U_t  7 (compat) the forward t link
      lmu[i] = d >= 6 ? 3 : d >> 1;
      lpar[i] = d < 6 && (d & 1) ? 1 : (compat && d != 6) ? -1 : 0;
      lcol[i] = d == 1 ? ln[1] : d == 3 ? ln[3] : d == 5 ? ln[5] : col;
   }
   U lr[NIT];
   auto fetch = [&](int i, int s) {  // no condition: it would hold both outcomes' registers
      const int p = q ^ (s & 1);
      const int par = lpar[i] < 0 ? 0 : p ^ lpar[i];
      g.load_raw(par, lmu[i], lcol[i] + (t0 + s) * S, lr[i]);
   };
   auto publish = [&](int i, int s) {
      U u = lr[i];
      GIO::finish(u);
      char *d = lk + ((s & 1) * NL * a.spb + lslot[i]) * LS;
#pragma unroll
      for (int k = 0; k < 9; k++) reinterpret_cast<typename U::E *>(d)[k] = u.e[k];
   };
   auto link = [&](int d, int s, U &u) {
      const char *p = lk + (((s & 1) * NL + d) * a.spb + jl) * LS;
#pragma unroll
      for (int k = 0; k < 9; k++) u.e[k] = reinterpret_cast<const typename U::E *>(p)[k];
   };
   // prologue: the links of the first slice; cen = psi(t0); bt = U_t(t0-1)^+
   // (1 -+ g_t) psi(t0-1); the first three neighbours
#pragma unroll
   for (int i = 0; i < NIT; i++)
      fetch(i, 0);
   Sp cen, nxt, ring[3], pre;
   Hv bt;
   {
      Sp f;
      U u;
      const int tm = (t0 == 0 ? Lt : t0) - 1;
      si.load_sps(q ^ 1, cc + tm * S, f);
      g.load_u(q ^ 1, 3, cc + tm * S, u);
      si.load_sps(q, cc + t0 * S, cen);
#pragma unroll
      for (int n = 0; n < 3; n++) si.load_sps(q ^ 1, cn[n] + t0 * S, ring[n]);
      term_udag<3, -SF>(f, u, bt);
   }
#pragma unroll
   for (int i = 0; i < NIT; i++)
      if (lslot[i] >= 0) publish(i, 0);
   // Norms: a slice's site values are summed (chunk_sum) after the next slice's
   // barrier, which spares one of their own (F32, 12-RHS CG at 24^3 x 48: 118.8
   // -> 116.8 ms).  Not in F16, where the values held longer spill (M 360 -> 395
   // us).
   constexpr bool DEFER = NORM && SIO::NC != 3;
   __shared__ double red[DEFER ? 2 : 1][DEFER ? BLOCK : 1];
   auto sum_chunk = [&](int s) {
      const int chunk = (q ^ (s & 1)) * a.nchunk + (c + (t0 + s) * S) / REDUCE_CHUNK;
      chunk_sum(red[s & 1], js, a.R, chunk, valid, a.partial + (size_t)rr * 2 * a.nchunk);
   };
   for (int s = 0; s < nts; s++) {
      const int t = t0 + s;
      const int p = q ^ (s & 1);
      const int base = t * S;
      const int j = cc + base;
      // what the slice loads ahead is the next slice's, or at the end the
      // slice's own again (unused)
      const int ahead = s + 1 < nts;
      const int pn = ahead ? p : p ^ 1, bn = base + ahead * S;
      // the slice's links are in their buffer, and the other buffer's readers
      // (the previous slice) are done; so are the previous slice's norms
      __syncthreads();
      if (DEFER && s > 0) sum_chunk(s - 1);
#pragma unroll
      for (int i = 0; i < NIT; i++) fetch(i, s + ahead);
      C acc[12];
#pragma unroll
      for (int m = 0; m < 12; m++) acc[m] = C{0, 0};
      // the scheduling barriers keep each load where it is issued, ahead of
      // the products it overlaps
#define PLQCD_PIPE(N, MU)                                                            \
   {                                                                                 \
      U u;                                                                           \
      Hv h;                                                                          \
      link(N, s, u);                                                                 \
      if constexpr ((N & 1) == 0) {                                                  \
         term_u<MU, SF>(ring[N % 3], u, h);                                          \
         accum<MU, SF, !compat>(acc, h);                                             \
      } else {                                                                       \
         term_udag<MU, -SF>(ring[N % 3], u, h);                                      \
         accum<MU, -SF, true>(acc, h);                                               \
      }                                                                              \
      pin(acc);                                                                      \
      __builtin_amdgcn_sched_barrier(0);                                             \
      if (N < 3) si.load_sps(p ^ 1, cn[(N + 3) % 6] + base, ring[N % 3]);             \
      else si.load_sps(pn, cn[(N + 3) % 6] + bn, ring[N % 3]);                        \
   }
      PLQCD_PIPE(0, 0)
      __builtin_amdgcn_sched_barrier(0);
      PLQCD_PIPE(1, 0)
      __builtin_amdgcn_sched_barrier(0);
      PLQCD_PIPE(2, 1)
      {
         const int tp = (t + 1 == Lt) ? 0 : t + 1;
         si.load_sps(p ^ 1, cc + tp * S, nxt);
      }
      __builtin_amdgcn_sched_barrier(0);
      PLQCD_PIPE(3, 1)
      if constexpr (PRE) fuse.p.at_rhs(rr).load_sps(p, j, pre);
      __builtin_amdgcn_sched_barrier(0);
      PLQCD_PIPE(4, 2)
      __builtin_amdgcn_sched_barrier(0);
      PLQCD_PIPE(5, 2)
      __builtin_amdgcn_sched_barrier(0);
#undef PLQCD_PIPE
      {
         U u;
         Hv h;
         link(compat ? 7 : 6, s, u);
         term_u<3, SF>(nxt, u, h);
         accum<3, SF, !compat>(acc, h);
         accum<3, -SF, true>(acc, bt);
         if constexpr (compat) link(6, s, u);
         term_udag<3, -SF>(cen, u, bt);
      }
      double nrm = 0.0;
      if (valid) {
         C cv[12];
         if (EPI >= 1) SIO::to_c(cen, cv);
         nrm = epilogue<EPI, NORM>(si, so, a, rr, p, j, acc, EPI >= 1 ? cv : (const C *)nullptr, fuse,
                                   PRE ? &pre : (const Sp *)nullptr);
      }
      cen = nxt;
#pragma unroll
      for (int i = 0; i < NIT; i++)
         if (lslot[i] >= 0) publish(i, s + 1);
      if (DEFER)
         red[s & 1][tid] = nrm;
      else if (NORM)
         chunk_reduce<BLOCK>(nrm, js, r, a.R, p * a.nchunk + (c + base) / REDUCE_CHUNK, valid,
                             a.partial + (size_t)rr * 2 * a.nchunk, s);
   }
   if (DEFER) {
      __syncthreads();
      sum_chunk(nts - 1);
   }
}

// Waves a SIMD is to hold.  F16 with the solver's epilogues takes 174 to 192
// registers by itself, two waves; held to three it spills 6 to 25 (12 RHS at
// 24^3 x 48: M 375 -> 360 us, M^+ with the update 410 -> 394).  With two links
// per lane and slice (four to six RHS) it would spill 30 to 34, and two waves
// are the faster: a 4-RHS CG 97.3 -> 84.0 ms at 32^3 x 64, 243.9 -> 212.2 at
// 40^3 x 80 (the plain t-march 86.2 and 213.3).
template <class SIO, int EPI, int NIT>
constexpr int pipe_waves()
{
   return std::is_same<typename SIO::real, double>::value ? 1 : SIO::NC == 6 ? 2 : EPI >= 1 && NIT > 1 ? 2 : 3;
}
template <int MODE, bool DAG, int EPI, bool NORM, int BLOCK, int NIT, class SIO, class GIO, class SO>
__global__ __launch_bounds__(BLOCK, (pipe_waves<SIO, EPI, NIT>())) void hop_pipe_kernel(SIO in, SO out, GIO g, HopArgs a, CgFuse<SIO> fuse)
{
   if (NORM && a.halt && *a.halt) return;
   hop_pipe_block<MODE, DAG, EPI, NORM, BLOCK, NIT>(in, out, g, a, logical_block(a), fuse);
}

// Pipelined t-march for one to three right-hand sides, F64 and F32 18-real:
// hop_tmarch_kernel's columns, chunks, lanes and order of operations, with
// every lane's loads (its own links beside the spinors they multiply) issued
// two neighbours ahead, across the slice boundary too.  With 12-real and F16
// links the rebuilding and the arithmetic cover more of the latency and the
// plain t-march holds more waves: it is as fast or up to 6 % faster and stays.
//   us per H with one RHS, untiled t-march and this: F64 16^3 x 32 30.4 and
// 26.3, 24^3 x 48 158.7 and 160.5 (its traffic moves at 4.6 TB/s either way);
// F32 18-real 16^3 x 32 20.9 and 15.8, 20^3 x 40 45.6 and 40.2, 24^3 x 48 87.1
// and 83.1, 32 x 42 x 24 x 64 241.8 and 227.5.
template <class SIO, class GIO>
constexpr bool stream_march()
{
   return std::is_same<typename SIO::real, double>::value || (SIO::NC == 6 && std::is_same<GIO, GaugeIO<PLQCD_PREC_F32, 18>>::value);
}
template <int MODE, bool DAG, int EPI, bool NORM, int BLOCK, class SIO, class GIO, class SO>
__global__ __launch_bounds__(BLOCK) void hop_stream_kernel(SIO in, SO out, GIO g, HopArgs a, CgFuse<SIO> fuse)
{
   if (NORM && a.halt && *a.halt) return;
   typedef typename SIO::C C;
   typedef typename SIO::Sp Sp;
   typedef typename SIO::Hv Hv;
   typedef typename GIO::U U;
   constexpr int SF = DAG ? 1 : -1;
   constexpr bool compat = MODE == MODE_COMPAT;
   constexpr int D = 2;  // neighbours in flight
   const int S = a.S;
   const int nbS = (S + a.spb - 1) / a.spb;
   int lb = logical_block(a);
   const int q = lb & 1;  // parity of the column's first site
   lb >>= 1;
   const int sb = lb % nbS;
   const int chunk = lb / nbS;
   const int tid = threadIdx.x;
   const int r = tid % a.R;
   const int js = tid / a.R;
   const int rr = rhs_of(a, r);
   const int c = sb * a.spb + js;
   const bool valid = c < S;
   const SIO si = in.at_rhs(rr);
   const SO so = out.at_rhs(rr);
   const int t0 = chunk_t0(a, chunk), nts = chunk_t0(a, chunk + 1) - t0;
   const int Lt = a.L[3];
   const int cc = valid ? c : 0;
   const int row = cc / a.Lxh;
   const int xh = cc - row * a.Lxh;
   const int y = row % a.L[1];
   const int z = row / a.L[1];
   const int odd = (q + y + z + t0) & 1;  // the parity of x, the same at every slice
   // x neighbours: for odd x, up is xh + 1 and down xh; for even x, up is xh and down xh - 1
   const int xup = row * a.Lxh + (xh + 1 == a.Lxh ? 0 : xh + 1);
   const int xdn = row * a.Lxh + (xh == 0 ? a.Lxh - 1 : xh - 1);
   int cn[6];
   {
      cn[0] = odd ? xup : cc;
      cn[1] = odd ? cc : xdn;
      const int ryp = (y == a.L[1] - 1) ? row - (a.L[1] - 1) : row + 1;
      const int rym = (y == 0) ? row + (a.L[1] - 1) : row - 1;
      const int rzp = (z == a.L[2] - 1) ? row - (a.L[2] - 1) * a.L[1] : row + a.L[1];
      const int rzm = (z == 0) ? row + (a.L[2] - 1) * a.L[1] : row - a.L[1];
      cn[2] = ryp * a.Lxh + xh;
      cn[3] = rym * a.Lxh + xh;
      cn[4] = rzp * a.Lxh + xh;
      cn[5] = rzm * a.Lxh + xh;
   }
   Sp cen, nxt, ring[D], pre;
   U lring[D], ut;
   Hv bt;
   auto issue = [&](int n, int s) {
      const int p = q ^ (s & 1), base = (t0 + s) * S;
      const int col = cn[n];
      si.load_sps(p ^ 1, col + base, ring[n % D]);
      if (n & 1) g.template load_raw<false, true>(p ^ 1, n >> 1, col + base, lring[n % D]);
      else g.template load_raw<false, true>(compat ? 0 : p, n >> 1, cc + base, lring[n % D]);
   };
   // prologue as in hop_tmarch_block
   {
      const int tm = (t0 == 0 ? Lt : t0) - 1;
      Sp f;
      U u;
      si.load_sps(q ^ 1, cc + tm * S, f);
      g.template load_raw<false, true>(q ^ 1, 3, cc + tm * S, u);
      si.load_sps(q, cc + t0 * S, cen);
#pragma unroll
      for (int n = 0; n < D; n++) issue(n, 0);
      GIO::finish(u);
      term_udag<3, -SF>(f, u, bt);
   }
   for (int s = 0; s < nts; s++) {
      const int t = t0 + s;
      const int p = q ^ (s & 1);
      const int base = t * S;
      const int j = cc + base;
      const int sn = s + 1 < nts ? s + 1 : s;
      C acc[12];
#pragma unroll
      for (int m = 0; m < 12; m++) acc[m] = C{0, 0};
      U ub;
#define PLQCD_PIPE(N, MU)                                                            \
   {                                                                                 \
      U u = lring[N % D];                                                            \
      Hv h;                                                                          \
      GIO::finish(u);                                                                \
      if constexpr ((N & 1) == 0) {                                                  \
         term_u<MU, SF>(ring[N % D], u, h);                                          \
         accum<MU, SF, !compat>(acc, h);                                             \
      } else {                                                                       \
         term_udag<MU, -SF>(ring[N % D], u, h);                                      \
         accum<MU, -SF, true>(acc, h);                                               \
      }                                                                              \
      pin(acc);                                                                      \
      __builtin_amdgcn_sched_barrier(0);                                             \
      if (N < 6 - D) issue(N + D, s);                                                \
      else issue((N + D) % 6, sn);                                                   \
      __builtin_amdgcn_sched_barrier(0);                                             \
   }
      PLQCD_PIPE(0, 0)
      PLQCD_PIPE(1, 0)
      PLQCD_PIPE(2, 1)
      {
         const int tp = (t + 1 == Lt) ? 0 : t + 1;
         si.load_sps(p ^ 1, cc + tp * S, nxt);
         g.template load_raw<true, true>(p, 3, j, ut);  // read by this lane only
         if constexpr (compat) g.template load_raw<false, true>(0, 3, j, ub);
      }
      __builtin_amdgcn_sched_barrier(0);
      PLQCD_PIPE(3, 1)
   
      if constexpr (EPI == 3) fuse.p.at_rhs(rr).load_sps(p, j, pre);
      __builtin_amdgcn_sched_barrier(0);
      PLQCD_PIPE(4, 2)
      PLQCD_PIPE(5, 2)
#undef PLQCD_PIPE
      {
         Hv h;
         GIO::finish(ut);
         if constexpr (compat) GIO::finish(ub);
         if constexpr (compat) term_u<3, SF>(nxt, ub, h);
         else term_u<3, SF>(nxt, ut, h);
         accum<3, SF, !compat>(acc, h);
         accum<3, -SF, true>(acc, bt);
         term_udag<3, -SF>(cen, ut, bt);
      }
      double nrm = 0.0;
      if (valid) {
         C cv[12];
         if (EPI >= 1) SIO::to_c(cen, cv);
         nrm = epilogue<EPI, NORM>(si, so, a, rr, p, j, acc, EPI >= 1 ? cv : (const C *)nullptr, fuse,
                                   EPI == 3 ? &pre : (const Sp *)nullptr);
      }
      cen = nxt;
      if (NORM) chunk_reduce<BLOCK>(nrm, js, r, a.R, p * a.nchunk + (c + base) / REDUCE_CHUNK, valid,
                                    a.partial + (size_t)rr * 2 * a.nchunk, s);
   }
}

// LDS for the links of a pipelined t-march block (of the CU's 160 KiB)
constexpr size_t kPipeLds = 144 * 1024;
// Whether hop_pipe_block runs blocks of `lanes` lanes and spb sites: at most
// 256 lanes, two links per lane and slice (four right-hand sides or more).
template <class GIO>
bool pipe_fits(int mode, int spb, int lanes)
{
   const int nl = mode == MODE_COMPAT ? links_per_slice<MODE_COMPAT>() : links_per_slice<PLQCD_HOP_WILSON>();
   return lanes <= 256 && nl * spb <= 2 * lanes && (size_t)2 * nl * spb * link_slot<GIO>() <= kPipeLds;
}

// One launch over a ragged batch (see BatchItem) of t-march blocks, pipelined
// ones (PIPE) when every item has four right-hand sides or more: 8^3 x 16 +
// 16^3 x 32 + 20^3 x 40 + 24^3 x 48, F32 12-real, 4 RHS 332 -> 313 us.
// Blocks go round-robin to the 8 XCDs; as in block order 2, the XCDs sweep the
// concatenated logical blocks together, XCD k (blockIdx % 8 == k) taking the
// k-th run of kBatchGroup consecutive blocks of every 8 kBatchGroup.  The grid
// is 8 x the blocks an XCD takes, rounded up.
template <int MODE, bool PIPE, int BLOCK, class SIO, class GIO>
__global__ __launch_bounds__(BLOCK) void hop_batch_kernel(const BatchList<SIO, GIO> items, int nitems, int total)
{
   const int i = blockIdx.x >> 3;
   const int b = ((i / kBatchGroup) * 8 + (blockIdx.x & 7)) * kBatchGroup + i % kBatchGroup;
   if (b >= total) return;
   int it = 0;
   while (it + 1 < nitems && b >= items.it[it + 1].first) it++;
   const BatchItem<SIO, GIO> &I = items.it[it];
   if constexpr (PIPE)
      hop_pipe_block<MODE, false, 0, false, BLOCK, 2>(I.in, I.out, I.g, I.a, b - I.first, CgFuse<SIO>{});
   else
      hop_tmarch_block<MODE, false, 0, false, BLOCK>(I.in, I.out, I.g, I.a, b - I.first, CgFuse<SIO>{});
}

// LDS bytes of the tiled kernel for BLOCK lanes: two buffers of centre
// spinors, the backward t terms and, in FP64 blocks of up to 128 lanes, the
// forward x links of a slice (hop_tile_kernel).
template <class S, class G, int BLOCK>
constexpr bool tile_xsh()
{
   return BLOCK <= 128 && std::is_same<typename S::real, double>::value;
}
template <class S, class G, int BLOCK>
constexpr size_t tile_lds_bytes()
{
   return (2 * sizeof(typename S::Sp) + sizeof(typename S::Hv)) * BLOCK +
          (tile_xsh<S, G, BLOCK>() ? 9 * sizeof(typename G::U::E) * BLOCK : 0);
}

// One direction of the tiled kernel: neighbours inside the tile come from the
// LDS slots su / sd (>= 0), the others from memory; same operation sequence
// as hop_fwd + hop_bwd.  With XSH (x direction only) the lane's forward link
// is streamed from memory and published in ux, and the backward link -- the
// forward link of the x - 1 lane, slot sd -- is read from there after a
// barrier; every lane of the block calls this.  In compat mode the forward
// link is the even site's with the same index j (slot sx in the tile): with
// XSH an odd lane reads it from ux after the barrier, otherwise from memory.
// NB: where the neighbours are -- 0 always in the tile (x: whole rows), 2
// never (z with one-plane tiles), 1 either, by lane (slot >= 0: in the tile).
// With NB 1 the compiler merges the two reads into one flat load.
template <int MU, int NB, int MODE, bool DAG, int BLOCK, bool XSH, class SIO, class GIO>
__device__ __forceinline__ void tile_dir(const SIO &in, const GIO &g, const typename SIO::Sp::E (*buf)[BLOCK], int p,
                                         int j, int base, int cu, int cd, int su, int sd, int sx,
                                         typename SIO::C acc[12], typename GIO::U::E (*ux)[BLOCK])
{
   typedef typename SIO::Sp Sp;
   constexpr int SG = DAG ? 1 : -1;
   constexpr bool share = MU == 0 && XSH;
   constexpr bool compat = MODE == MODE_COMPAT;
   Sp f;
   typename GIO::U u;
   typename SIO::Hv r;
   auto nb_load = [&](int slot, int jnb) {
      if (NB == 0 || (NB == 1 && slot >= 0)) {
#pragma unroll
         for (int m = 0; m < Sp::N; m++) f.e[m] = buf[m][slot];
      } else {
         in.load_sp(1 - p, jnb + base, f);
      }
   };
   nb_load(su, cu);
   if constexpr (share) {
      g.template load_u<true>(p, MU, j, u);
#pragma unroll
      for (int k = 0; k < 9; k++) ux[k][threadIdx.x] = u.e[k];
      if constexpr (compat) {
         __syncthreads();
         if (p) {
#pragma unroll
            for (int k = 0; k < 9; k++) u.e[k] = ux[k][sx];
         }
      }
   } else {
      g.load_u(compat ? 0 : p, MU, j, u);
   }
   term_u<MU, SG>(f, u, r);
   accum<MU, SG, !compat>(acc, r);
   nb_load(sd, cd);
   if constexpr (share) {
      if constexpr (!compat) __syncthreads();
#pragma unroll
      for (int k = 0; k < 9; k++) u.e[k] = ux[k][sd];
   } else {
      g.load_u(1 - p, MU, cd + base, u);
   }
   term_udag<MU, -SG>(f, u, r);
   accum<MU, -SG, true>(acc, r);
}

// LDS-tiled t-march (full lattice, one RHS).  A block owns the
// columns of a tile of Lxh x ty x tz (x, y, z) sites -- whole x rows -- for
// both parities: lanes q = 0 and 1 of a column hold its two x-adjacent sites,
// and the block walks the t-slices of one t-chunk.  The centre spinors of a t-slice are in LDS
// (two buffers, one barrier per slice), and the x, y and z
// neighbours inside the tile are read from there; only the tile's y/z halo and
// the t+1 spinor are loaded from memory.  The centre spinor and the backward
// t term stay in LDS rather than in registers.  Links and the t direction are
// handled as in hop_tmarch_kernel, except that FP64 blocks of up to 128 lanes
// pass the x links between the two lanes that use each one through LDS (a
// second barrier per slice).  Terms are accumulated in the order of hop_kernel.
// Compat mode takes the forward links of odd sites from the even site with
// the same index (its t link with a second load, since the true one still
// serves the next slice's backward term).  2 Lxh ty tz <= BLOCK lanes.
template <int MODE, bool DAG, int EPI, bool NORM, int BLOCK, class SIO, class GIO>
__global__ __launch_bounds__(BLOCK) void hop_tile_kernel(SIO in, SIO out, GIO g, HopArgs a, CgFuse<SIO> fuse)
{
   if (NORM && a.halt && *a.halt) return;
   typedef typename SIO::C C;
   const int r0 = rhs_of(a, 0);  // the launch's one RHS
   in = in.at_rhs(r0);
   out = out.at_rhs(r0);
   constexpr int SF = DAG ? 1 : -1;  // forward projector sign
   typedef typename SIO::Sp Sp;
   typedef typename SIO::Hv Hv;
   __shared__ typename Sp::E sm[2][Sp::N][BLOCK];
   __shared__ typename Hv::E sb[Hv::N][BLOCK];  // the lane's backward t term b (read and written by that lane only)
   // x links through LDS in FP64 blocks of two waves: a CU then holds several
   // blocks, and one works while another waits at the extra barrier (FP64
   // 18-real, 32x4x1 tiles at 32^3 x 64: 407 against 427 us).  FP32 tiles ran
   // up to 27 % slower with it (12-real, 32x4x1, 16 slices: 220 against 173 us).
   constexpr bool XSH = tile_xsh<SIO, GIO, BLOCK>();
   constexpr bool SPLIT = std::is_same<typename SIO::real, double>::value;
   __shared__ typename GIO::U::E ux[XSH ? 9 : 1][XSH ? BLOCK : 1];  // the lanes' forward x links of this slice
   typedef typename GIO::U::E(*UxRow)[BLOCK];
   const int S = a.S;
   const int ncol = a.Lxh * a.ty * a.tz;  // columns of the tile, 2 ncol <= BLOCK lanes
   const int nty = a.L[1] / a.ty;
   const int ntile = nty * (a.L[2] / a.tz);
   const int lb = logical_block(a);
   const int tile = lb % ntile;
   const int chunk = lb / ntile;
   const int tid = threadIdx.x;
   const int q = tid >= ncol ? 1 : 0;  // parity of the lane's first site
   const int lc = tid - q * ncol;      // xh + Lxh * (ly + ty * lz)
   const int xh = lc % a.Lxh;
   const int lyz = lc / a.Lxh;
   const int ly = lyz % a.ty, lz = lyz / a.ty;
   const int y0 = (tile % nty) * a.ty, z0 = (tile / nty) * a.tz;
   const int y = y0 + ly, z = z0 + lz;
   const int row = y + a.L[1] * z;
   const int c = row * a.Lxh + xh;
   const int t0 = chunk_t0(a, chunk), nts = chunk_t0(a, chunk + 1) - t0;
   const int x = 2 * xh + ((q + y + z + t0) & 1);  // the same at every t-slice
   const int sx = (1 - q) * ncol + lc;              // the lane with the same index j, other parity
   int cu[3], cd[3], su[3], sd[3];
   {
      const int oth = (1 - q) * ncol;  // lanes of the other parity
      const int xp = (x + 1 == a.L[0]) ? 0 : x + 1;
      const int xm = (x == 0) ? a.L[0] - 1 : x - 1;
      cu[0] = row * a.Lxh + (xp >> 1);
      cd[0] = row * a.Lxh + (xm >> 1);
      su[0] = oth + lc - xh + (xp >> 1);
      sd[0] = oth + lc - xh + (xm >> 1);
      const int yp = (y + 1 == a.L[1]) ? 0 : y + 1;
      const int ym = (y == 0) ? a.L[1] - 1 : y - 1;
      const int zp = (z + 1 == a.L[2]) ? 0 : z + 1;
      const int zm = (z == 0) ? a.L[2] - 1 : z - 1;
      cu[1] = (yp + a.L[1] * z) * a.Lxh + xh;
      cd[1] = (ym + a.L[1] * z) * a.Lxh + xh;
      cu[2] = (y + a.L[1] * zp) * a.Lxh + xh;
      cd[2] = (y + a.L[1] * zm) * a.Lxh + xh;
      const int lyp = yp - y0, lym = ym - y0, lzp = zp - z0, lzm = zm - z0;
      su[1] = (lyp >= 0 && lyp < a.ty) ? oth + xh + a.Lxh * (lyp + a.ty * lz) : -1;
      sd[1] = (lym >= 0 && lym < a.ty) ? oth + xh + a.Lxh * (lym + a.ty * lz) : -1;
      su[2] = (lzp >= 0 && lzp < a.tz) ? oth + xh + a.Lxh * (ly + a.ty * lzp) : -1;
      sd[2] = (lzm >= 0 && lzm < a.tz) ? oth + xh + a.Lxh * (ly + a.ty * lzm) : -1;
   }
   const int Lt = a.L[3];
   // prologue: psi(t0) into the first buffer; b = U_t(t0-1)^+ (1 -+ g_t) psi(t0-1)
   {
      Sp f;
      typename GIO::U u;
      Hv b;
      in.load_sp(q, c + t0 * S, f);
#pragma unroll
      for (int m = 0; m < Sp::N; m++) sm[0][m][tid] = f.e[m];
      const int tm = (t0 == 0 ? Lt : t0) - 1;
      in.load_sp(q ^ 1, c + tm * S, f);
      g.load_u(q ^ 1, 3, c + tm * S, u);
      term_udag<3, -SF>(f, u, b);
#pragma unroll
      for (int m = 0; m < Hv::N; m++) sb[m][tid] = b.e[m];
   }
   for (int s = 0; s < nts; s++) {
      const int t = t0 + s;
      const int p = q ^ (s & 1);
      const int base = t * S;
      const int j = c + base;
      // buf holds the centre spinors of this t-slice; the t+1 spinors go to
      // nxt, whose readers (the previous slice) have all passed this barrier
      typename Sp::E(*buf)[BLOCK] = sm[s & 1];
      typename Sp::E(*nxt)[BLOCK] = sm[(s + 1) & 1];
      __syncthreads();
      C acc[12];
#pragma unroll
      for (int m = 0; m < 12; m++) acc[m] = C{0, 0};
      // the scheduling barriers keep each direction's loads in its own
      // section, which holds the kernel within 256 VGPRs without spills
      // The x neighbours (whole rows) are read from LDS with no test, and in
      // FP64 the z neighbours of one-plane tiles from memory with none: each
      // neighbour read under a per-lane test became one flat load serving
      // both places, waited for with every global load in flight (FP64
      // 12-real 32x1x4 tiles at 32^3 x 64: 333 against 351 us; FP32 18-real
      // 32x8x1: 240 against 245 us with the x test gone, 2.5 % slower with
      // the z one gone too, so FP32 keeps that).
      tile_dir<0, 0, MODE, DAG, BLOCK, XSH>(in, g, buf, p, j, base, cu[0], cd[0], su[0], sd[0], sx, acc, (UxRow)ux);
      __builtin_amdgcn_sched_barrier(0);
      tile_dir<1, 1, MODE, DAG, BLOCK, XSH>(in, g, buf, p, j, base, cu[1], cd[1], su[1], sd[1], sx, acc, (UxRow)ux);
      __builtin_amdgcn_sched_barrier(0);
      if (SPLIT && a.tz == 1)
         tile_dir<2, 2, MODE, DAG, BLOCK, XSH>(in, g, buf, p, j, base, cu[2], cd[2], su[2], sd[2], sx, acc, (UxRow)ux);
      else
         tile_dir<2, 1, MODE, DAG, BLOCK, XSH>(in, g, buf, p, j, base, cu[2], cd[2], su[2], sd[2], sx, acc, (UxRow)ux);
      __builtin_amdgcn_sched_barrier(0);
      {
         Sp f;
         typename GIO::U u;
         Hv rr, b;
         const int tp = (t + 1 == Lt) ? 0 : t + 1;
         in.load_sp(p ^ 1, c + tp * S, f);
#pragma unroll
         for (int m = 0; m < Sp::N; m++) nxt[m][tid] = f.e[m];
         g.template load_u<true>(p, 3, j, u);  // read by this lane only (see hop_tmarch_kernel)
         if constexpr (MODE == MODE_COMPAT) {
            typename GIO::U uf;
            g.load_u(0, 3, j, uf);
            term_u<3, SF>(f, uf, rr);
         } else {
            term_u<3, SF>(f, u, rr);
         }
         accum<3, SF, MODE != MODE_COMPAT>(acc, rr);
#pragma unroll
         for (int m = 0; m < Hv::N; m++) b.e[m] = sb[m][tid];
         accum<3, -SF, true>(acc, b);
#pragma unroll
         for (int m = 0; m < Sp::N; m++) f.e[m] = buf[m][tid];
         term_udag<3, -SF>(f, u, b);
#pragma unroll
         for (int m = 0; m < Hv::N; m++) sb[m][tid] = b.e[m];
      }
      double nrm;
      if (EPI >= 1) {
         Sp cs;
         C cen[12];
#pragma unroll
         for (int m = 0; m < Sp::N; m++) cs.e[m] = buf[m][tid];
         SIO::to_c(cs, cen);
         nrm = epilogue<EPI, NORM>(in, out, a, r0, p, j, acc, cen, fuse);
      } else {
         nrm = epilogue<EPI, NORM>(in, out, a, r0, p, j, acc, (const C *)nullptr, fuse);
      }
      if (NORM)
         chunk_reduce<BLOCK>(nrm, lc, 0, 1, p * a.nchunk + j / REDUCE_CHUNK, true,
                             a.partial + (size_t)r0 * 2 * a.nchunk, s);
   }
}

// kernel variants: gather (1 RHS per lane), t-march, RHS-blocked gather, LDS tile, pipelined t-march, half lattice
enum Variant { V_GATHER = 0, V_MARCH = 1, V_RB2 = 2, V_RB4 = 4, V_TILE = 8, V_PIPE = 16, V_HALF = 32 };

// S: the input field's accessor; SO: the output's (differs only with EPI 3,
// which the tile and RHS-blocked kernels don't have).  Returns 0 when the kernel was enqueued, and
// an error when the variant does not exist for these template arguments (the
// host-side checks of launch_t keep such launches out; this keeps a future
// change from silently launching nothing).
template <int MODE, bool DAG, int EPI, bool NORM, int BLOCK, class S, class G, class SO>
int launch_one(int variant, dim3 grid, dim3 block, hipStream_t st, S si, SO so, G gg, const HopArgs &a,
               const CgFuse<S> &f)
{
   constexpr bool same = std::is_same<S, SO>::value && EPI != 3;  // the tile and RHS-blocked kernels
   if constexpr ((EPI == 0 || EPI == 4) && !DAG && !NORM && same) {
      if (variant == V_HALF) {
         if (a.stream_links)
            hipLaunchKernelGGL((hop_half_kernel<MODE, EPI, true, BLOCK, S, G>), grid, block, 0, st, si, so, gg, a, f);
         else
            hipLaunchKernelGGL((hop_half_kernel<MODE, EPI, false, BLOCK, S, G>), grid, block, 0, st, si, so, gg, a, f);
         return 0;
      }
   }
   if constexpr (EPI == 4) {  // the external-centre epilogue exists for the half-lattice kernel only
      return plqcd::set_error(2, "hop: the external-centre epilogue runs on one parity only (variant %d)", variant);
   } else if (variant == V_PIPE) {
      if constexpr (BLOCK == 256) {
         const size_t lds = pipe_lds_bytes<MODE, G>(a.spb);
         if (links_per_slice<MODE>() * a.spb <= (int)block.x)
            hipLaunchKernelGGL((hop_pipe_kernel<MODE, DAG, EPI, NORM, BLOCK, 1, S, G, SO>), grid, block, lds, st, si, so,
                               gg, a, f);
         else
            hipLaunchKernelGGL((hop_pipe_kernel<MODE, DAG, EPI, NORM, BLOCK, 2, S, G, SO>), grid, block, lds, st, si, so,
                               gg, a, f);
         return 0;
      }
   } else if (variant == V_MARCH) {
      if constexpr (stream_march<S, G>() && BLOCK <= 256)  // blocks of 512 lanes hold too few registers each
         hipLaunchKernelGGL((hop_stream_kernel<MODE, DAG, EPI, NORM, BLOCK, S, G, SO>), grid, block, 0, st, si, so, gg, a,
                            f);
      else
         hipLaunchKernelGGL((hop_tmarch_kernel<MODE, DAG, EPI, NORM, BLOCK, S, G, SO>), grid, block, 0, st, si, so, gg, a,
                            f);
      return 0;
   } else if (variant == V_TILE) {
      // two LDS buffers of BLOCK spinors, BLOCK half-spinors and (FP64 blocks
      // of up to 128 lanes) BLOCK x links must fit the CU's 160 KiB
      if constexpr (same && tile_lds_bytes<S, G, BLOCK>() <= 136 * 1024) {
         hipLaunchKernelGGL((hop_tile_kernel<MODE, DAG, EPI, NORM, BLOCK, S, G>), grid, block, 0, st, si, so, gg, a, f);
         return 0;
      }
   } else if (variant == V_RB2) {
      if constexpr (same) {
         hipLaunchKernelGGL((hop_rb_kernel<MODE, DAG, EPI, NORM, BLOCK, 2, S, G>), grid, block, 0, st, si, so, gg, a, f);
         return 0;
      }
   } else if (variant == V_RB4) {
      if constexpr (same) {
         hipLaunchKernelGGL((hop_rb_kernel<MODE, DAG, EPI, NORM, BLOCK, 4, S, G>), grid, block, 0, st, si, so, gg, a, f);
         return 0;
      }
   } else if (variant == V_GATHER) {
      hipLaunchKernelGGL((hop_kernel<MODE, DAG, EPI, NORM, BLOCK, S, G, SO>), grid, block, 0, st, si, so, gg, a, f);
      return 0;
   }
   return plqcd::set_error(2, "hop: kernel variant %d with %d-lane blocks does not exist for this operation", variant,
                           BLOCK);
}

template <int MODE, bool DAG, int EPI, bool NORM, class S, class G, class SO>
int launch_block(int maxblock, int variant, dim3 grid, dim3 block, hipStream_t st, S si, SO so, G gg,
                 const HopArgs &a, const CgFuse<S> &f = CgFuse<S>{})
{
   if (maxblock <= 128) return launch_one<MODE, DAG, EPI, NORM, 128>(variant, grid, block, st, si, so, gg, a, f);
   if (maxblock <= 256) return launch_one<MODE, DAG, EPI, NORM, 256>(variant, grid, block, st, si, so, gg, a, f);
   return launch_one<MODE, DAG, EPI, NORM, 512>(variant, grid, block, st, si, so, gg, a, f);
}

template <int PREC, int LINKS>
int launch_t(const plqcd_hip_gauge *g, const plqcd_hip_field *in, plqcd_hip_field *out, int parity, int mode,
             const plqcd::DslashOp &op)
{
   const plqcd_hip_lattice *lat = g->lat;
   HopArgs a = make_hop_args(lat, parity);
   typedef SpinorIO<PREC> S;
   typedef GaugeIO<PREC, LINKS> G;
   const S si = spinor_io<PREC>(in);
   const G gg = gauge_io<PREC, LINKS>(g);
   const bool resid = op.resid_b != nullptr;  // EPI 3: out may have another precision
   const bool centre = op.centre != nullptr;  // EPI 4: one parity only
   // lanes: the window of right-hand sides [op.r0, op.r0 + R) of the fields
   const int R = op.nr > 0 ? op.nr : in->nrhs;
   a.r0 = op.nr > 0 && !op.rlist ? op.r0 : 0;
   a.rlist = op.rlist;
   const bool solver = op.kappa || op.kappa_host;  // M or M^+
   HopTuning tu = plqcd::default_tuning(lat->L, PREC, LINKS, R, solver);
   plqcd::lookup_tuning(plqcd::TuneKey{{lat->L[0], lat->L[1], lat->L[2], lat->L[3]}, PREC, LINKS, R,
                                       solver ? plqcd::kTuneOpSolver : plqcd::kTuneOpHop},
                        &tu);
   // RHS per lane (RHS-blocked gather) when it divides R; none for the
   // residual epilogue, and the external-centre one runs the half-lattice kernel only
   const int rb = !resid && !centre && (tu.rb == 2 || tu.rb == 4) && R % tu.rb == 0 ? tu.rb : 1;
   const int lanes = R / rb;  // lanes per site
   // block shape: `lanes` lanes per site and a whole number of reduction chunks
   int target = tu.block;
   if (lanes * REDUCE_CHUNK > target) {
      target = 128;
      while (target < lanes * REDUCE_CHUNK) target *= 2;
   }
   if (target > 512)
      return plqcd::set_error(2, "hop: %d right-hand sides exceed the per-launch limit of %d", R, 512 / REDUCE_CHUNK);
   a.R = R;
   a.spb = REDUCE_CHUNK * (target / (REDUCE_CHUNK * lanes));
   const int threads = lanes * a.spb;
   const int maxblock = threads <= 128 ? 128 : threads <= 256 ? 256 : 512;
   a.kappa = op.kappa;
   a.partial = op.partial;
   a.halt = op.halt;
   a.nchunk = plqcd::reduce_chunks(lat->Vh);
   const bool dag = op.dag != 0;
   const int epi = resid ? 3 : op.alpha ? 2 : op.centre ? 4 : solver ? 1 : 0;
   const bool norm = op.partial != nullptr;
   if ((dag || epi || norm) && mode != PLQCD_HOP_WILSON)
      return plqcd::set_error(2, "hop: M, M^+ and norms need the wilson mode");
   if (epi == 2 && (!dag || !norm || !op.kappa))
      return plqcd::set_error(2, "hop: the CG-update epilogue needs M^+, a norm and kappa");
   if (epi == 4 && (dag || norm || !solver))
      return plqcd::set_error(2, "hop: the external-centre epilogue needs kappa, and no M^+ or norm");
   if (epi == 3 && (PREC != PLQCD_PREC_F64 || !dag || !norm || !op.kappa))
      return plqcd::set_error(2, "hop: the residual epilogue needs F64 storage, M^+, a norm and kappa");
   CgFuse<S> fu{};
   if (op.kappa_host)
      for (int r = 0; r < in->nrhs; r++) fu.kappa[r] = op.kappa_host[r];
   if (epi == 2) {
      fu.alpha = op.alpha;
   } else if (epi == 4) {
      fu.p = spinor_io<PREC>(op.centre);
   } else if (epi == 3) {
      fu.p = spinor_io<PREC>(op.resid_b);
   }
   if (norm && a.nparity != 2) return plqcd::set_error(2, "hop: norms are only fused into full-lattice launches");
   // the t-march kernel serves full-lattice applications (either mode; with a
   // norm, the t-slices hold whole reduction chunks), in t-chunks of at most
   // tmarch slices
   const bool march = !centre && rb == 1 && tu.tmarch > 0 && a.nparity == 2 && (!norm || a.S % REDUCE_CHUNK == 0);
   // the LDS-tiled t-march: one RHS, a tile of whole x rows dividing the y and
   // z extents, 2 Lxh ty tz lanes per block (at most 256 with F64 storage for
   // the LDS), and, with a norm, reduction chunks that do not leave a tile row
   const long long tlanes = 2LL * lat->Lxh * tu.ty * tu.tz;
   const bool tiled = march && !resid && R == 1 && tu.ty > 0 && tu.tz > 0 && lat->L[1] % tu.ty == 0 &&
                      lat->L[2] % tu.tz == 0 && tlanes <= (PREC == PLQCD_PREC_F64 ? 256 : 512) &&
                      (!norm || (lat->Lxh * tu.ty) % REDUCE_CHUNK == 0);
   // the pipelined t-march wherever it fits (four right-hand sides or more)
   const bool pipe = march && !tiled && pipe_fits<G>(mode, a.spb, threads);
   const bool half = a.nparity == 1 && !dag && !norm && rb == 1 && (epi == 0 || epi == 4);
   const int variant = half ? V_HALF : tiled ? V_TILE : pipe ? V_PIPE : march ? V_MARCH : (rb == 2 ? V_RB2 : rb == 4 ? V_RB4 : V_GATHER);
   a.nt = march ? (lat->L[3] + tu.tmarch - 1) / tu.tmarch : 1;
   int nb, nthreads = threads, mblock = pipe ? 256 : maxblock;
   if (tiled) {
      a.ty = tu.ty;
      a.tz = tu.tz;
      nb = (lat->L[1] / tu.ty) * (lat->L[2] / tu.tz) * a.nt;
      nthreads = (int)tlanes;
      mblock = nthreads <= 128 ? 128 : nthreads <= 256 ? 256 : 512;
   } else {
      const int nblk = march ? ((a.S + a.spb - 1) / a.spb) * a.nt : (lat->Vh + a.spb - 1) / a.spb;
      nb = nblk * a.nparity;
   }
   a.order = tu.order;
   a.group = tu.group > 0 ? tu.group : 1;
   if (pipe && tu.gy > 0 && lat->Lxh * lat->L[1] % (a.spb * tu.gy) == 0 && lat->L[2] % tu.gz == 0) {
      a.gy = tu.gy;
      a.gz = tu.gz;
   }
   if (half) {
      // Links stream past the L2s unless the field of links about fits them (32
      // MB together) and is there from the last call, or many RHS share each
      // load: one RHS, us per half without and with, F32 12-real 16^3 x 32 (25
      // MB of links) 8.7 and 10.7, 20^3 x 40 (61 MB) 18.1 and 22.0, 24^3 x 48
      // (127 MB) 42.9 and 40.5; F64 16^3 x 32 (75 MB) 21.2 and 21.4, 20^3 x 40
      // (184 MB) 56.7 and 48.8; F64 24^3 x 48 4 RHS 281 and 268, 6 RHS 392 and
      // 386, 12 RHS 753 and 780.
      a.stream_links = R <= 4 && g->bytes >= size_t(75) << 20;
      // Slabs where t-slices of several RHS crowd each other out: without and
      // with, F64 24^3 x 48 with 4 RHS (a field of 510 MB) 268 and 256, 16^3 x 32
      // with 4 RHS (101 MB) 54 and 59, with 12 RHS (302 MB) 150 and 145; one RHS
      // at 32^3 x 64 (403 MB) 316 and 341.
      HopTuning user{};
      if (!plqcd::user_tuning(PREC, &user)) {
         const int nbS = (a.S + a.spb - 1) / a.spb, most = (nbS + 7) / 8;
         const bool slab = R >= 4 && in->bytes * (double(R) / in->nrhs) >= double(size_t(200) << 20) &&
                           8 * most <= nbS + nbS / 8;  // an XCD's slab at most an eighth larger than the mean
         a.order = slab ? 3 : 1;
         if (slab) nb = 8 * most * lat->L[3];
      }
   }
   const dim3 grid(nb), block(nthreads);
   hipStream_t st = lat->stream;
   int lrc = 0;
   if (epi == 3) {
      if constexpr (PREC == PLQCD_PREC_F64) {
         if (out->prec == PLQCD_PREC_F64)
            lrc = launch_block<PLQCD_HOP_WILSON, true, 3, true>(mblock, variant, grid, block, st, si,
                                                                 spinor_io<PLQCD_PREC_F64>(out), gg, a, fu);
         else if (out->prec == PLQCD_PREC_F32)
            lrc = launch_block<PLQCD_HOP_WILSON, true, 3, true>(mblock, variant, grid, block, st, si,
                                                                 spinor_io<PLQCD_PREC_F32>(out), gg, a, fu);
         else
            lrc = launch_block<PLQCD_HOP_WILSON, true, 3, true>(mblock, variant, grid, block, st, si,
                                                                 spinor_io<PLQCD_PREC_F16>(out), gg, a, fu);
      }
      if (lrc) return lrc;
      PLQCD_HIP_TRY(hipGetLastError());
      return 0;
   }
   const S so = spinor_io<PREC>(out);
   if (mode == PLQCD_HOP_COMPAT) {
      lrc = launch_block<PLQCD_HOP_COMPAT, false, 0, false>(mblock, variant, grid, block, st, si, so, gg, a);
   } else if (!dag) {
      if (epi == 0) lrc = launch_block<PLQCD_HOP_WILSON, false, 0, false>(mblock, variant, grid, block, st, si, so, gg, a);
      else if (epi == 4)
         lrc = launch_block<PLQCD_HOP_WILSON, false, 4, false>(mblock, variant, grid, block, st, si, so, gg, a, fu);
      else if (!norm) lrc = launch_block<PLQCD_HOP_WILSON, false, 1, false>(mblock, variant, grid, block, st, si, so, gg, a, fu);
      else lrc = launch_block<PLQCD_HOP_WILSON, false, 1, true>(mblock, variant, grid, block, st, si, so, gg, a);
   } else {
      if (epi == 0) lrc = launch_block<PLQCD_HOP_WILSON, true, 0, false>(mblock, variant, grid, block, st, si, so, gg, a);
      else if (epi == 2)
         lrc = launch_block<PLQCD_HOP_WILSON, true, 2, true>(mblock, variant, grid, block, st, si, so, gg, a, fu);
      else if (!norm) lrc = launch_block<PLQCD_HOP_WILSON, true, 1, false>(mblock, variant, grid, block, st, si, so, gg, a, fu);
      else lrc = launch_block<PLQCD_HOP_WILSON, true, 1, true>(mblock, variant, grid, block, st, si, so, gg, a);
   }
   if (lrc) return lrc;
   PLQCD_HIP_TRY(hipGetLastError());
   return 0;
}


template <int PREC, int LINKS>
int launch_batch_t(int n, const plqcd_hip_gauge *const *g, const plqcd_hip_field *const *in,
                   plqcd_hip_field *const *out, int mode)
{
   typedef SpinorIO<PREC> S;
   typedef GaugeIO<PREC, LINKS> G;
   static_assert(sizeof(BatchList<S, G>) <= 4096, "kernel argument too large");
   for (int i = 0; i < n; i++)
      if (in[i]->nrhs * REDUCE_CHUNK > 256) return plqcd::set_error(2, "hop_batch: at most 32 right-hand sides per item");
   hipStream_t st = g[0]->lat->stream;
   for (int i0 = 0; i0 < n; i0 += kBatchItems) {
      const int m = std::min(kBatchItems, n - i0);
      // block size: the largest whole number of reduction chunks of sites
      // times the RHS count that fits 256 lanes, maximised over the items (a
      // batch of 12-RHS items runs 192-lane blocks with no idle lane)
      int block = 64;
      for (int i = 0; i < m; i++) {
         const int R = in[i0 + i]->nrhs;
         block = std::max(block, REDUCE_CHUNK * (256 / (REDUCE_CHUNK * R)) * R);
      }
      // t-chunks of 16 (F64) or 8 slices (or as plqcd_hip_hop_tuning asks),
      // shorter ones while the batch has fewer blocks than the chip has places
      int T = PREC == PLQCD_PREC_F64 ? 16 : 8;
      HopTuning user{};
      const bool asked = plqcd::user_tuning(PREC, &user) && user.tmarch > 0;
      if (asked) T = user.tmarch;
      BatchList<S, G> L{};
      int total = 0;
      bool pipe = true;
      size_t lds = 0;
      for (;; T /= 2) {
         total = 0;
         for (int i = 0; i < m; i++) {
            BatchItem<S, G> &I = L.it[i];
            I.in = spinor_io<PREC>(in[i0 + i]);
            I.out = spinor_io<PREC>(out[i0 + i]);
            I.g = gauge_io<PREC, LINKS>(g[i0 + i]);
            const plqcd_hip_lattice *lat = g[i0 + i]->lat;
            I.a = make_hop_args(lat, PLQCD_PARITY_ALL);
            I.a.R = in[i0 + i]->nrhs;
            I.a.spb = REDUCE_CHUNK * (block / (REDUCE_CHUNK * I.a.R));
            I.a.nt = (lat->L[3] + T - 1) / T;
            I.nb = 2 * ((I.a.S + I.a.spb - 1) / I.a.spb) * I.a.nt;
            I.first = total;
            total += I.nb;
            pipe = pipe && pipe_fits<G>(mode, I.a.spb, I.a.R * I.a.spb);
            lds = std::max(lds, mode == PLQCD_HOP_COMPAT ? pipe_lds_bytes<PLQCD_HOP_COMPAT, G>(I.a.spb)
                                                         : pipe_lds_bytes<PLQCD_HOP_WILSON, G>(I.a.spb));
         }
         if (asked || T == 1 || total >= 512) break;
      }
      // one hardware block per logical block (8 XCDs x span, see
      // hop_batch_kernel): the hardware then balances the items' blocks over
      // the CUs.  A persistent grid of occupancy x CUs blocks, each taking a
      // fixed stride of logical blocks, was 2-9 % slower than this at
      // 16^3x32 + 24^3x48 + 32^3x64 with 12 RHS.
      auto go = [&](auto kern) {
         const int span = ((total + 8 * kBatchGroup - 1) / (8 * kBatchGroup)) * kBatchGroup;
         hipLaunchKernelGGL(kern, dim3(8 * span), dim3(block), pipe ? lds : 0, st, L, m, total);
      };
      if (mode == PLQCD_HOP_COMPAT) {
         if (pipe) go(hop_batch_kernel<PLQCD_HOP_COMPAT, true, 256, S, G>);
         else go(hop_batch_kernel<PLQCD_HOP_COMPAT, false, 256, S, G>);
      } else {
         if (pipe) go(hop_batch_kernel<PLQCD_HOP_WILSON, true, 256, S, G>);
         else go(hop_batch_kernel<PLQCD_HOP_WILSON, false, 256, S, G>);
      }
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return plqcd::set_error(10, "hop_batch: %s", hipGetErrorString(e));
   }
   return 0;
}

}  // namespace

// Entry points of one (precision, link format), explicitly instantiated in
// dslash_<precision>_l<links>.hip.
template <int PREC, int LINKS>
int plqcd::hop_launch(const plqcd_hip_gauge *g, const plqcd_hip_field *in, plqcd_hip_field *out, int parity, int mode,
                      const DslashOp &op)
{
   return launch_t<PREC, LINKS>(g, in, out, parity, mode, op);
}

template <int PREC, int LINKS>
int plqcd::hop_batch_launch(int n, const plqcd_hip_gauge *const *g, const plqcd_hip_field *const *in,
                            plqcd_hip_field *const *out, int mode)
{
   return launch_batch_t<PREC, LINKS>(n, g, in, out, mode);
}
