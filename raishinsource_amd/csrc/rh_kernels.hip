// HIP kernels of the RAISHIN GRMHD time step for gfx950 (FP64 path).
//
// Device layout (structure of arrays, i fastest):
//   state planes   A[n*N + c],  c = (i-1) + ni*((j-1) + nj*(k-1)),  n = 0..8
//   fluxes         F[d][n*N + c] holds ww(d,n,i,j,k) = flux at i+1/2 (j+1/2, k+1/2)
//   metric tables  (i,k) planes: the Kerr-Schild metric has no phi dependence,
//                  so each location set is 33 planes of ni*nk values and the
//                  Christoffel symbols 64 planes.
// Each kernel cites the reference routines it restates.
#include <type_traits>
#include "rh_device.hpp"
#include "rh_metric.hpp"
#include "rh_kernels.hpp"

namespace rh {

// Cell and (i,k) indices, thread and workgroup numbers are 32-bit (cells are
// below 2^29): a 64-bit division, four of which decode a thread's (i,j,k),
// takes several times the instructions of a 32-bit one.
RH_DEV unsigned cidx(int i, int j, int k, const Geo& G) {
  const unsigned jr = G.jfix ? 0u : (unsigned)(j - 1);
  return (unsigned)(i - 1) + (unsigned)G.ni * (jr + (unsigned)G.njs * (unsigned)(k - 1));
}
// j range of a box: the stored row of a collapsed model, else [lo, hi]
RH_DEV int jlo(const Geo& G, int lo) { return G.jfix ? G.jfix : lo; }
RH_DEV int jhi(const Geo& G, int hi) { return G.jfix ? G.jfix : hi; }
// strides of a step in j and in k in the stored planes
RH_DEV long long jstride(const Geo& G) { return G.jfix ? 0LL : (long long)G.ni; }
RH_DEV long long kstride(const Geo& G) { return (long long)G.ni * G.njs; }
RH_DEV unsigned q2(int i, int k, const Geo& G) { return (unsigned)(i - 1) + (unsigned)G.ni * (unsigned)(k - 1); }

// 1-based (i,j,k) of linear thread t over a box [lo_a, hi_a] per axis; false if outside.
RH_DEV bool box_index(unsigned t, int ilo, int ihi, int jlo, int jhi, int klo, int khi, int& i, int& j, int& k) {
  if (ihi < ilo || jhi < jlo || khi < klo) return false;
  const unsigned ci = ihi - ilo + 1, cj = jhi - jlo + 1, ck = khi - klo + 1;
  const unsigned r = t / ci, kk = r / cj;
  if (kk >= ck) return false;
  i = ilo + (int)(t - r * ci);
  j = jlo + (int)(r - kk * cj);
  k = klo + (int)kk;
  return true;
}

// Workgroup b is dispatched to XCD b % 8.  Renumbering the workgroups so that
// each XCD takes one contiguous eighth of the launch keeps neighbouring rows
// of a stencil in the same L2.  A bijection on [0, nb), for a launch or a part
// of one that starts at a multiple of 8.
RH_DEV unsigned xcd_renumber(unsigned nb, unsigned b) {
  const unsigned x = b % 8u, idx = b / 8u, q = nb / 8u, r = nb % 8u;
  return x < r ? x * (q + 1) + idx : r * (q + 1) + (x - r) * q + idx;
}
RH_DEV unsigned xcd_block() { return xcd_renumber(gridDim.x, blockIdx.x); }

// As box_index with the j and k axes swapped in the ordering (i fastest, then
// k, then j): consecutive workgroups step along k, the k sweep's stencil axis.
RH_DEV bool box_index_ikj(unsigned t, int ilo, int ihi, int jlo, int jhi, int klo, int khi, int& i, int& j, int& k) {
  return box_index(t, ilo, ihi, klo, khi, jlo, jhi, i, k, j);
}

// Waves along the D axis (D = 2 or 3): a lane's i within a 64-wide chunk
// of the row, consecutive waves on consecutive j (D=2) or k (D=3) rows, so
// the cell's index along D is the same in every lane of a wave.  Covers
// 64*ceil(ci/64)*cj*ck indices; lanes past the row's end return false.
template <int D>
RH_DEV bool box_index_wave(unsigned t, int ilo, int ihi, int jlo, int jhi, int klo, int khi, int& i, int& j,
                           int& k) {
  if (ihi < ilo || jhi < jlo || khi < klo) return false;
  const unsigned ci = ihi - ilo + 1, cj = jhi - jlo + 1, ck = khi - klo + 1;
  const unsigned nic = (ci + 63) / 64, w = t >> 6;
  const unsigned n1 = D == 2 ? cj : ck, n2 = D == 2 ? ck : cj;
  const unsigned r = w / n1, a = w - r * n1, b = r / nic, ic = r - b * nic;
  if (b >= n2) return false;
  j = jlo + (int)(D == 2 ? a : b);
  k = klo + (int)(D == 2 ? b : a);
  i = ilo + (int)(ic * 64 + (t & 63));
  return i <= ihi;
}

// Counter slots (raishin_counters field order).
enum { C_FALLBACK = 0, C_FAIL, C_NEGRHO, C_NEGP, C_VSQGT1, C_DET0, C_WGCARRY, C_ATM, C_PMMSCALE, C_PMMFLOOR,
       C_GUARD, C_NCOUNT };

// Event counts without atomics: each wavefront of a launch owns the row
// cpart[w*C_NCOUNT ..] (w = its index in the model's part of the launch, from
// the workgroup's index blk there); the lowest flagged lane
// adds the wave's popcount.  Launches are stream-ordered, so a row has one
// writer at a time; k_sum_counters folds the rows when counters are read.
// (Device-scope atomics on a few addresses from every wave serialise across
// the XCDs: they cost more than the kernels that raise the events.)
RH_DEV void count_wave(unsigned long long* cpart, unsigned blk, int slot, bool flag,
                       unsigned long long weight = 1) {
  const unsigned long long b = __ballot(flag);
  if (b && (threadIdx.x % warpSize) == (unsigned)(__ffsll((long long)b) - 1)) {
    const unsigned w = (blk * blockDim.x + threadIdx.x) / warpSize;
    cpart[(unsigned long long)w * C_NCOUNT + slot] += (unsigned long long)__popcll(b) * weight;
  }
}

// cnt[s] += sum over rows of cpart[.][s], then the rows are cleared.  One
// workgroup of 1024.
__global__ void __launch_bounds__(1024) k_sum_counters(unsigned long long* __restrict__ cpart, long long rows,
                                                       unsigned long long* __restrict__ cnt) {
  __shared__ unsigned long long part[C_NCOUNT][1024 / 64];
  unsigned long long acc[C_NCOUNT];
#pragma unroll
  for (int s = 0; s < C_NCOUNT; s++) acc[s] = 0;
  for (long long r = threadIdx.x; r < rows; r += blockDim.x)
#pragma unroll
    for (int s = 0; s < C_NCOUNT; s++) {
      acc[s] += cpart[r * C_NCOUNT + s];
      cpart[r * C_NCOUNT + s] = 0;
    }
  const int lane = threadIdx.x % 64, wv = threadIdx.x / 64;
#pragma unroll
  for (int s = 0; s < C_NCOUNT; s++) {
    unsigned long long v = acc[s];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off);
    if (lane == 0) part[s][wv] = v;
  }
  __syncthreads();
  if (threadIdx.x < C_NCOUNT) {
    unsigned long long t = 0;
    for (int q = 0; q < (int)(blockDim.x / 64); q++) t += part[threadIdx.x][q];
    cnt[threadIdx.x] += t;
  }
}

// ------------------------------------------------------------------------
// PPM reconstruction of one cell (rec.f90:1261-2056), direction D.
// Hands each variable's left edge l (uri*r(c-1)) and right edge r (uri*l(c))
// to store(n, l, r), one variable at a time.
// p is the 1-based index of the cell along D; the loads are along stride s.
// dxs[d] holds the dummy dx*b(d) of rec2 (= actual dx*b(d-1), rec.f90:58).
// ------------------------------------------------------------------------
// Shape coefficients of the cell: flattening f2 (rec.f90:1736-1858) and the
// contact-steepening eta of the density (rec.f90:1537-1629).  R is the
// arithmetic type (double: the reference's; float: the mixed-precision form).
// One cell's shock indicator (flaten, rec.f90:1736-1830) from the pressure at
// +-1 and +-2 and the velocity along D at +-1.
template <class R>
RH_DEV R ppm_f1(R pm2, R pm1, R pp1, R pp2, R vm1, R vp1) {
  const R t3a = absr(pp1 - pm1);
  const R t1 = R(1) * fminf_(pp1, pm1) - t3a;
  const R t2 = vp1 - vm1;
  const R omg1 = (t1 < R(0) && t2 < R(0)) ? R(1) : R(0);
  const R t3b = (pp2 - pm2);
  R t4;
  if (t3b == R(0)) t4 = (t3a == R(0)) ? R(-0.52) : R(1.0) - R(0.52);
  else t4 = (t3a / t3b) - R(0.52);
  return fminf_(R(1), omg1 * fmaxf_(R(0), t4 * R(10.0)));
}

// f2 of a cell from the indicators of its neighbours and its own
// (rec.f90:1831-1858).
template <class R>
RH_DEV R ppm_f2(R f1m, R f10, R f1p, R p5m, R p5p) {
  const R f1b = (p5p - p5m < R(0)) ? f1p : f1m;
  return fmaxf_(f10, f1b);
}

// Steepening eta of the density (detect, rec.f90:1537-1629) from the second
// differences of the two neighbouring cells; xm, x0, xp: cell positions.
template <class R>
RH_DEV R ppm_eta(R ddm, R ddp, R um1, R up1, R p5m, R p5p, R xm, R x0, R xp, R gam) {
  const R t1 = ddp * ddm;
  const R t2 = mad_(-R(0.1), fminf_(absr(up1), absr(um1)), absr(up1 - um1));
  R etatil;
  if (t1 >= R(0) && t2 <= R(0)) etatil = R(0);
  else {
    const R t2a = -(ddp - ddm) / (xp - xm);
    const R dl = x0 - xm, dr = xp - x0;
    const R t2b = mad_(dr * dr, dr, dl * dl * dl) / (up1 - um1);
    etatil = t2a * t2b;
  }
  R eta = fmaxf_(R(0), fminf_(R(5.0) * (etatil - R(0.05)), R(1)));
  const R t3 = absr(up1 - um1) / fminf_(up1, um1);
  const R t4 = absr(p5p - p5m) / fminf_(p5p, p5m);
  if (gam * R(1) * t3 < t4) eta = R(0);
  return eta;
}

template <int D, class R>
RH_DEV void ppm_shape(const double* __restrict__ W, long long N, long long c, long long s, int p,
                      const double* __restrict__ dxs, const double* __restrict__ xs, R gam, R& f2_out, R& eta_out) {
  const R dm2 = R(dxs[p - 2]), dm1 = R(dxs[p - 1]), d0 = R(dxs[p]), dp1 = R(dxs[p + 1]), dp2 = R(dxs[p + 2]);
  const int VEL = D;  // velocity component along D is variable D+1 (0-based D)
  const double* P5 = W + 4 * N + c;
  const double* PV = W + (long long)VEL * N + c;
  R f1[3];
#pragma unroll
  for (int q = -1; q <= 1; q++)
    f1[q + 1] = ppm_f1<R>(R(P5[(q - 2) * s]), R(P5[(q - 1) * s]), R(P5[(q + 1) * s]), R(P5[(q + 2) * s]),
                          R(PV[(q - 1) * s]), R(PV[(q + 1) * s]));
  const R p5p = R(P5[s]), p5m = R(P5[-s]);
  f2_out = ppm_f2<R>(f1[0], f1[1], f1[2], p5m, p5p);
  const double* P1 = W + c;
  const R um2 = R(P1[-2 * s]), um1 = R(P1[-s]), u0 = R(P1[0]), up1 = R(P1[s]), up2 = R(P1[2 * s]);
  const R ddm = (R(1) / (dm2 + dm1 + d0)) * ((u0 - um1) / (d0 + dm1) - (um1 - um2) / (dm1 + dm2));
  const R ddp = (R(1) / (d0 + dp1 + dp2)) * ((up2 - up1) / (dp2 + dp1) - (up1 - u0) / (dp1 + d0));
  eta_out = ppm_eta<R>(ddm, ddp, um1, up1, p5m, p5p, R(xs[p - 2]), R(xs[p - 1]), R(xs[p]), gam);
}

// interp's width-only coefficients of a cell at index p (ppm_coefficients on
// the host, same expressions and order): t1a,t1b,t1c of dma at q = p-1, p,
// p+1 (rec.f90:1353-1355) and the four of equation (51) at q+1/2 for q = p
// and p-1 (rec.f90:1427-1436).  The same for every variable: loaded once.
template <class R>
struct PpmCoef {
  R ta[3], tb[3], tc[3];
  R e2[2], e3[2], e4[2], e5[2];
};

template <class R>
RH_DEV void ppm_coef(const double* __restrict__ pc, long long npc, int p, PpmCoef<R>& k) {
#pragma unroll
  for (int o = 0; o < 3; o++) {
    const int q = p - 1 + o;
    k.ta[o] = R(pc[q]); k.tb[o] = R(pc[npc + q]); k.tc[o] = R(pc[2 * npc + q]);
  }
#pragma unroll
  for (int o = 0; o < 2; o++) {
    const int q = p - o;
    k.e2[o] = R(pc[3 * npc + q]); k.e3[o] = R(pc[4 * npc + q]);
    k.e4[o] = R(pc[5 * npc + q]); k.e5[o] = R(pc[6 * npc + q]);
  }
}

// Interface values of variable n of the cell from its 5-point stencil
// u = (u(p-2) .. u(p+2)): interp (rec.f90:1309-1476), steepening of the
// density (rec.f90:1661-1677), flattening and monoto (rec.f90:1887-2056).
// l = uri*r(c-1), r = uri*l(c).
// dma of a cell (rec.f90:1338-1414): the limited slope from its neighbours.
template <int D, class R>
RH_DEV R ppm_dma(R um, R u0, R up, R t1a, R t1b, R t1c) {
  const R sp1 = (up - u0);
  const R sm1 = (u0 - um);
  const R spm1 = sp1 * sm1;
  const R da = t1a * mad_(t1b, sp1, t1c * sm1);
  if (spm1 <= R(0)) return R(0);
  const R t1 = (da < R(0)) ? R(-1) : R(1);
  const R t1d = fminf_(absr(sm1), absr(sp1));
  if (D == 3) return t1 * fminf_(absr(da), t1d);   // rec.f90:1414
  return t1 * fminf_(absr(da), R(2.0) * t1d);
}

// Equation (51) (rec.f90:1427-1476): the value at the face between the cells
// q and q+1, uq + t2 + t3 - e4 dmq1 + e5 dmq with t2 = e2 (uq1 - uq),
// t3 = e3 (uq1 - uq).
template <class R>
RH_DEV R ppm_eq51(R uq, R uq1, R dmq, R dmq1, R e2, R e3, R e4, R e5) {
  const R du = uq1 - uq;
  return mad_(e5, dmq, mad_(-e4, dmq1, mad_(e3, du, mad_(e2, du, uq))));
}

// Flattening and monoto (rec.f90:1887-2056) of a cell's two face values.
template <class R>
RH_DEV void ppm_monoto(R u0, R f2, R& l, R& r) {
  r = mad_(u0, f2, r * (R(1) - f2));
  l = mad_(u0, f2, l * (R(1) - f2));
  if ((r - u0) * (l - u0) >= R(0)) { r = u0; l = u0; }            // equation (73)
  const R t3 = R(6.0) * (r - l) * mad_(-R(0.5), r + l, u0);        // equations (74), (75)
  const R t4 = (r - l) * (r - l);
  if (t3 > t4) l = mad_(R(3.0), u0, -(R(2.0) * r));
  if (-t3 > t4) r = mad_(R(3.0), u0, -(R(2.0) * l));
}

template <int D, class R>
RH_DEV void ppm_var(const R u[5], const PpmCoef<R>& k, int n, R f2, R eta, R& l_out, R& r_out) {
  const R um2 = u[0], um1 = u[1], u0 = u[2], up1 = u[3], up2 = u[4];
  const R dmm1 = ppm_dma<D, R>(um2, um1, u0, k.ta[0], k.tb[0], k.tc[0]);
  const R dm0 = ppm_dma<D, R>(um1, u0, up1, k.ta[1], k.tb[1], k.tc[1]);
  const R dmp1 = ppm_dma<D, R>(u0, up1, up2, k.ta[2], k.tb[2], k.tc[2]);
  R r = ppm_eq51<R>(u0, up1, dm0, dmp1, k.e2[0], k.e3[0], k.e4[0], k.e5[0]);   // value at p+1/2
  R l = ppm_eq51<R>(um1, u0, dmm1, dm0, k.e2[1], k.e3[1], k.e4[1], k.e5[1]);   // value at p-1/2
  if (n == 0) {
    r = mad_(r, R(1) - eta, mad_(-R(0.5), dmp1, up1) * eta);
    l = mad_(l, R(1) - eta, mad_(R(0.5), dmm1, um1) * eta);
  }
  ppm_monoto<R>(u0, f2, l, r);
  l_out = l;
  r_out = r;
}

// ------------------------------------------------------------------------
// PPM face values of every cell once, along D: one thread per cell computes
// f2 and eta, then each variable's edges in turn, writing E indexed by
// interface: planes 0..8 at c-s the left edge of cell c (uri*r(c-1)), planes
// 9..17 at c its right edge (uri*l(c)).  Cells nm0..n-nm0+1 along D, the
// sweep's box across.  R: arithmetic and storage type of the edges.
// ------------------------------------------------------------------------
template <int D, class R>
RH_DEV void b_ppm_edges(const Geo& G, const EdgeArgs& A, unsigned blk) {
  const double* __restrict__ W = A.W;
  const double* __restrict__ dxs = A.dxs;
  const double* __restrict__ xs = A.xs;
  const double* __restrict__ pc = A.pc;
  const double gam = A.gam;
  R* __restrict__ E = (R*)A.E;
  int i, j, k;
  const unsigned t = blk * blockDim.x + threadIdx.x;
  const int hi = G.ni - G.nm0 + (D == 1), hj = jhi(G, G.nj - G.nm0 + (D == 2)), hk = G.nk - G.nm0 + (D == 3);
  const int lj = jlo(G, G.nm0);
  const bool in = (D == 1) ? box_index(t, G.nm0, hi, lj, hj, G.nm0, hk, i, j, k)
                           : box_index_wave<D>(t, G.nm0, hi, lj, hj, G.nm0, hk, i, j, k);
  if (!in) return;
  const long long N = G.N;
  const long long s = (D == 1) ? 1LL : (D == 2) ? jstride(G) : kstride(G);
  const unsigned c = cidx(i, j, k, G);
  // along j and k every lane of a wave has the same index along D: its
  // coefficients and widths are loaded once per wave, into scalar registers
  const int p = (D == 1) ? i : __builtin_amdgcn_readfirstlane((D == 2) ? j : k);
  const long long npc = ((D == 1) ? G.ni : (D == 2) ? G.nj : G.nk) + 2;
  PpmCoef<R> kc;
  ppm_coef<R>(pc, npc, p, kc);
  R f2, eta;
  ppm_shape<D, R>(W, N, c, s, p, dxs, xs, R(gam), f2, eta);
  // one variable at a time, the next variable's stencil loads in flight
  // while the current one is computed
  R cur[5], nxt[5];
#pragma unroll
  for (int o = 0; o < 5; o++) cur[o] = R(W[c + (o - 2) * s]);
#pragma unroll 1
  for (int n = 0; n < 9; n++) {
    if (n < 8) {
      const double* Pn = W + (long long)(n + 1) * N + c;
#pragma unroll
      for (int o = 0; o < 5; o++) nxt[o] = R(Pn[(o - 2) * s]);
    }
    R l, r;
    ppm_var<D, R>(cur, kc, n, f2, eta, l, r);
    E[(long long)n * N + c - s] = l;   // stored at the interface it belongs to (c-1/2)
    E[(long long)(9 + n) * N + c] = r;
#pragma unroll
    for (int o = 0; o < 5; o++) cur[o] = nxt[o];
  }
}

// MC-limited slope of a cell (mclim, rec.f90:208-367, irec=1) from its
// neighbours; im, ip: 1 / (distance to them + 1e-12).
template <class R>
RH_DEV R mc_slope(R um, R u, R up, R im, R ip) {
  const R sp = (up - u) * ip;
  const R sm = (u - um) * im;
  const R tmp = (sp < R(0)) ? R(-1) : R(1);
  return tmp * fmaxf_(R(0), fminf_(fminf_(R(2) * absr(sp), tmp * R(2) * sm), tmp * R(0.5) * (sp + sm)));
}

// Face physics and HLLE of interface c+1/2 along D from its two face states
// (wl: the left cell's right edge, wr: the right cell's left edge):
// caluu3 -> calflx3 -> calcha -> hlle, written to F (and the transverse B
// fluxes to their CTsrc planes).  SAME: the two face states are the same.
template <int D, class R, int ICHA, bool SAME = false, class MT>
RH_DEV void sweep_face(const Geo& G, R* __restrict__ F, R* __restrict__ CTsrc, unsigned c, int i, int j, int k,
                       const MT& M, R gam, const R wl[9], const R wr[9]) {
  const long long N = G.N;
  const R detg = M.detg();
  R Ul[9], Fl[9], vpl, vml;
  {
    PrelT<R> sl;
    prelude(wl, gam, M, sl);
    const R pw = powr(sl.de, gam);
    tmunu_row<R>(sl, 0, detg, pw, Ul);
    tmunu_row<R>(sl, D, detg, pw, Fl);
    face_speed<R, ICHA>(sl, D, gam, M, vpl, vml);
  }
  R Ur[9], Fr[9], vpr = vpl, vmr = vml;
  if constexpr (SAME) {
#pragma unroll
    for (int n = 0; n < 9; n++) { Ur[n] = Ul[n]; Fr[n] = Fl[n]; }
  } else {
    PrelT<R> sr;
    prelude(wr, gam, M, sr);
    const R pw = powr(sr.de, gam);
    tmunu_row<R>(sr, 0, detg, pw, Ur);
    tmunu_row<R>(sr, D, detg, pw, Fr);
    face_speed<R, ICHA>(sr, D, gam, M, vpr, vmr);
  }
  const R cmax = fmaxf_(fmaxf_(R(0), vpr), vpl);
  const R cmin = (D == 3) ? fminf_(fminf_(R(0), vpr), vml)   // calcha.f90:107
                          : fminf_(fminf_(R(0), vmr), vml);
  const unsigned co = c * (unsigned)sizeof(R);
  // transverse B fluxes of this direction and their CTsrc planes
  // (0 ww(2,7) 1 ww(3,7) 2 ww(1,8) 3 ww(3,8) 4 ww(1,9) 5 ww(2,9))
  constexpr int nA = (D == 1) ? 7 : 6, nB = (D == 3) ? 7 : 8;
  constexpr int pA = (D == 1) ? 2 : (D == 2) ? 0 : 1, pB = (D == 1) ? 4 : (D == 2) ? 5 : 3;
  const bool in_ct = i >= G.nm1 && i <= G.ni - G.nm1 && j >= G.nm1 && j <= G.nj - G.nm1 && k >= G.nm1 &&
                     k <= G.nk - G.nm1;
#pragma unroll
  for (int n = 0; n < 9; n++) {
    double o;
    if (cmin > R(0)) o = double(Fl[n]);
    else if (cmin <= R(0) && cmax > R(0)) {
      const R c1 = fmaxf_(absr(cmax), absr(cmin));
      o = double(R(0.5) * mad_(-c1, Ur[n] - Ul[n], Fl[n] + Fr[n]));
    } else if (cmax <= R(0)) o = double(Fr[n]);
    else o = F[(long long)n * N + c];  // unordered (NaN) speeds: hlle keeps ww, then flushes it
    if (absr(o) < 1.0e-40) o = 0.0;
    // the labelled non-reference form: no flux of the normal field component
    // (the induction flux itself is zero; HLLE's dissipation term is what
    // the reference keeps, hll.f90:109-111), so flux-CT keeps div B
    if (n == 5 + D && G.divb0) o = 0.0;
    if (n == nA || n == nB) {
      st_(CTsrc + (long long)(n == nA ? pA : pB) * N, co, R(o));
      if (!in_ct) st_(F + (long long)n * N, co, R(o));  // inside the CT box fluxct writes this slot
    } else {
      st_(F + (long long)n * N, co, R(o));
    }
  }
}

// ------------------------------------------------------------------------
// Direction sweep: reconstruction + face fluxes + wave speeds + HLLE.
// rec2 (rec.f90:2-142) -> caluu3/calflx3* -> calcha (calcha.f90:2-126) -> hlle
// (hll.f90:47-192), fused per interface.  One thread per interface c+1/2.
// ------------------------------------------------------------------------
// F holds ww(D,:,:,:,:) exactly as the reference's array: the last value that
// hlle or ct wrote to each slot.  The two transverse B fluxes of direction D
// also go to their plane of CTsrc (the copies ct.f90:54-67 takes before
// averaging); inside the CT box fluxct then writes F itself.
//
// PPM's face values come from k_ppm_edges (E); MC, MP5 and WENO5 reconstruct
// here.  (MC from its four cells: with the face values of every cell through
// HBM from a kernel of their own, as PPM's, 151x50x83 took 0.195 ms for a
// stage's edges and sweeps, now 0.127.)
template <int D, int IREC, class R, int ICHA, bool MK>
RH_DEV void b_sweep(const Geo& G, const SweepArgs& A, unsigned blk) {
  const double* __restrict__ W = A.W;
  const R* __restrict__ E = (const R*)A.E;
  R* __restrict__ F = (R*)A.F;
  R* __restrict__ CTsrc = (R*)A.CTsrc;
  const R gam = R(A.gam);
  int i, j, k;
  const unsigned t = blk * blockDim.x + threadIdx.x;
  const int lj = jlo(G, G.nm0), hj = jhi(G, G.nj - G.nm0);
  // k sweeps that read a stencil along k (MC, MP5, WENO5) walk k before j so
  // neighbouring workgroups share the stencil planes in L2; with the face
  // values precomputed (PPM) the i,j,k walk keeps each (i,k) metric entry in
  // L2 across the j rows instead.
  constexpr bool kfirst = D == 3 && IREC != 5;
  const bool in = kfirst ? box_index_ikj(t, G.nm0, G.ni - G.nm0, lj, hj, G.nm0, G.nk - G.nm0, i, j, k)
                         : box_index(t, G.nm0, G.ni - G.nm0, lj, hj, G.nm0, G.nk - G.nm0, i, j, k);
  if (!in) return;
  const long long N = G.N;
  const long long s = (D == 1) ? 1LL : (D == 2) ? jstride(G) : kstride(G);
  const unsigned c = cidx(i, j, k, G);
  R wl[9], wr[9];
  if (IREC == 5) {
    // right edge of cell c (uri*l(c)) and left edge of cell c+1 (uri*r(c)),
    // both stored at interface c+1/2's index
#pragma unroll
    for (int n = 0; n < 9; n++) {
      wl[n] = ld_(E + (long long)(9 + n) * N, c * (unsigned)sizeof(R));
      wr[n] = ld_(E + (long long)n * N, c * (unsigned)sizeof(R));
    }
  } else if (IREC == 1) {
    const unsigned c8 = c * 8u;
    const int p = (D == 1) ? i : (D == 2) ? j : k;
    const R small = R(1.0e-12);
    const R xm = R(A.xs[p - 2]), x0 = R(A.xs[p - 1]), x1 = R(A.xs[p]), x2 = R(A.xs[p + 1]), xf = R(A.xa[p - 1]);
    const R i0 = R(1) / (x0 - xm + small), i1 = R(1) / (x1 - x0 + small), i2 = R(1) / (x2 - x1 + small);
#pragma unroll
    for (int n = 0; n < 9; n++) {
      const double* Pn = W + (long long)n * N;
      const R a = R(ld_(Pn - s, c8)), b = R(ld_(Pn, c8)), d = R(ld_(Pn + s, c8)), e = R(ld_(Pn + 2 * s, c8));
      wl[n] = b + mc_slope<R>(a, b, d, i0, i1) * (xf - x0);
      wr[n] = d - mc_slope<R>(b, d, e, i1, i2) * (x1 - xf);
    }
  } else {
    const unsigned c8 = c * 8u;
#pragma unroll
    for (int n = 0; n < 9; n++) {
      const double* Pn = W + (long long)n * N;
      const R a = R(ld_(Pn - 2 * s, c8)), b = R(ld_(Pn - s, c8)), cc = R(ld_(Pn, c8)), d = R(ld_(Pn + s, c8)),
              e = R(ld_(Pn + 2 * s, c8)), f = R(ld_(Pn + 3 * s, c8));
      if (IREC == 6) {
        const R sl[5] = {a, b, cc, d, e};
        const R sr[5] = {b, cc, d, e, f};
        wl[n] = mp5_right<R>(sl);
        wr[n] = mp5_left<R>(sr);
      } else {
        wl[n] = weno_edge<R>(a, b, cc, d, e);
        wr[n] = weno_edge<R>(f, e, d, cc, b);
      }
    }
  }
  const MetOf<MK, R> M(A.metF, G.P2, q2(i, k, G));
  sweep_face<D, R, ICHA>(G, F, CTsrc, c, i, j, k, M, gam, wl, wr);
}

// ------------------------------------------------------------------------
// PPM direction sweep with its face values computed in the same kernel
// (interp, detect, flaten, monoto; rec.f90:1261-2056, then caluu3 -> calflx3
// -> calcha -> hlle), through LDS, so the 18 edge planes never reach HBM.
//
// A workgroup holds a tile of A.tp cells along D by blockDim.x / A.tp lines
// across (D = 1: rows; D = 2, 3: consecutive i, so every load instruction
// reads runs of contiguous values).  Everything that belongs to a cell or to
// a face is computed by one lane and passed to the lanes beside it:
//   1. each cell's limited slope of every variable, its shock indicator f1
//      and its second difference of the density, from its +-1 (+-2) cells;
//   2. the face value of equation (51) between the lane's cell and the next;
//   3. the cell's two face values after steepening, flattening and monoto;
//   4. the interface between the lane's cell and the next: own right edge,
//      the next lane's left edge.
// A tile of tp cells gives tp - 3 interfaces (the first cell lacks the face
// below it, the last two the face above them or above the next cell), so
// tiles overlap by three cells.  The lane's arithmetic is that of
// k_ppm_edges followed by k_sweep on the same values (the pieces above), so
// the fluxes are the same bit for bit; what a cell alone would compute three
// times (slopes, indicators) or twice (face values) is computed once.
// The entropy variable (plane 5) is not reconstructed: no flux reads its
// face value.
//
// D = 0: the j sweep of a collapsed model.  Its one phi row is its own
// neighbour, so every slope is zero, the face values are the cell's own
// (not a number where the cell's value is infinite, as inf - inf makes the
// slopes) and the two sides of each interface are the same state.
// ------------------------------------------------------------------------
constexpr int PS_NV = 8;                                     // reconstructed variables
RH_DEV constexpr int ps_plane(int q) { return q < 5 ? q : q + 1; }

template <int D, class R, int ICHA, bool MK>
RH_DEV void b_psweep(const Geo& G, const PSweepArgs& A, unsigned blk) {
  const int bt = blockDim.x, tid = threadIdx.x;
  const long long N = G.N;
  const double* __restrict__ W = A.W;
  R* __restrict__ F = (R*)A.F;
  R* __restrict__ CTsrc = (R*)A.CTsrc;
  const R gam = R(A.gam);
  const unsigned nif_i = (unsigned)(G.ni - 2 * G.nm0 + 1), nif_k = (unsigned)(G.nk - 2 * G.nm0 + 1);
  const int ihi = G.ni - G.nm0, jl = jlo(G, G.nm0), jh = jhi(G, G.nj - G.nm0);
  if constexpr (D == 0) {
    const unsigned t = (unsigned)blk * (unsigned)bt + (unsigned)tid;
    const unsigned kk = t / nif_i;
    if (kk >= nif_k) return;
    const int i = G.nm0 + (int)(t - kk * nif_i), k = G.nm0 + (int)kk;
    const long long c = cidx(i, jl, k, G);
    R w[9];
#pragma unroll
    for (int n = 0; n < 9; n++) {
      const R u = n == 5 ? R(0) : R(ld_(W + (long long)n * N, c * 8u));
      w[n] = absr(u) == R(__builtin_inf()) ? R(__builtin_nan("")) : u;
    }
    const MetOf<MK, R> M(A.metF, G.P2, q2(i, k, G));
    sweep_face<2, R, ICHA, true>(G, F, CTsrc, c, i, jl, k, M, gam, w, w);
    return;
  }
  extern __shared__ unsigned char rh_dyn_lds[];  // 18 planes of blockDim.x values of R
  R* const L = reinterpret_cast<R*>(rh_dyn_lds) + tid;
  R* const Lv = L + 8 * bt;   // slopes, then left edges (L: cell values, then those of equation (51))
  R* const Ls = L + 16 * bt;  // f1, second difference of the density
  const int TP = A.tp, IPT = TP - 3;
  const int phi = D == 1 ? ihi : D == 2 ? jh : G.nk - G.nm0;
  // place in the tile: pl along D, il across; a step along D is `st` lanes
  const int pl = D == 1 ? tid & ((1 << A.sh) - 1) : tid >> A.sh;
  const int il = D == 1 ? tid >> A.sh : tid & ((1 << A.sh) - 1);
  const int st = D == 1 ? 1 : 1 << A.sh;
  const unsigned b = (unsigned)blk;
  // the lane's cell (p: its index along D); lanes past the last line or the
  // last cell that a needed slope reads (phi + 3, the grid's last but one)
  // are clamped to it and write nothing
  int i, j, k, p;
  bool in;
  if constexpr (D == 1) {
    const unsigned rt = b / (unsigned)A.ndc, dc = b - rt * (unsigned)A.ndc;
    const unsigned cj = (unsigned)(jh - jl + 1), rows = cj * nif_k;
    unsigned row = rt * (unsigned)(bt / TP) + (unsigned)il;
    in = row < rows;
    row = in ? row : rows - 1;
    const unsigned kk = row / cj;
    j = jl + (int)(row - kk * cj);
    k = G.nm0 + (int)kk;
    p = G.nm0 - 1 + (int)dc * IPT + pl;
    in = in && p <= phi;
    if (p > phi + 3) p = phi + 3;
    i = p;
  } else {
    // consecutive workgroups along i (their lines share cache lines); then,
    // along j, the tiles of a k row; along k, the j of one k range, which
    // share that range's face metric
    const int TI = 1 << A.sh;
    const unsigned r = b / (unsigned)A.nig, ig = b - r * (unsigned)A.nig;
    const unsigned nin = D == 2 ? (unsigned)A.ndc : (unsigned)(jh - jl + 1), ro = r / nin, ri = r - ro * nin;
    const unsigned tt = D == 2 ? ro : ri, dc = D == 2 ? ri : ro;
    i = G.nm0 + (int)ig * TI + il;
    in = i <= ihi;
    if (!in) i = ihi;
    p = (D == 2 ? jl : G.nm0) - 1 + (int)dc * IPT + pl;
    in = in && p <= phi;
    if (p > phi + 3) p = phi + 3;
    j = D == 2 ? p : jl + (int)tt;
    k = D == 2 ? G.nm0 + (int)tt : p;
  }
  const long long s = (D == 1) ? 1LL : (D == 2) ? jstride(G) : kstride(G);
  const unsigned c = cidx(i, j, k, G), c8 = c * 8u;
  // the lane's own cell from memory, its neighbours from the lanes beside it
  // (the tile's first and last cells read theirs)
  const int nx = pl < TP - 1 ? st : 0, pv = pl > 0 ? -st : 0;
  R um[PS_NV], u0[PS_NV], up[PS_NV], ue[PS_NV];
#pragma unroll
  for (int q = 0; q < PS_NV; q++) u0[q] = R(ld_(W + (long long)ps_plane(q) * N, c8));
  const bool edge = pl == 0 || pl == TP - 1;
  if (edge) {
    const unsigned e8 = c8 + (pl == 0 ? 0u - (unsigned)s : (unsigned)s) * 8u;
#pragma unroll
    for (int q = 0; q < PS_NV; q++) ue[q] = R(ld_(W + (long long)ps_plane(q) * N, e8));
  }
  // (the cell at phi + 3 has no second neighbour and needs no indicator)
  const R pm2 = R(ld_(W + 4 * N - 2 * s, c8)), pp2 = R(ld_(W + 4 * N, c8 + (unsigned)((p < phi + 3 ? 2 : 1) * s) * 8u));
  const long long npc = ((D == 1) ? G.ni : (D == 2) ? G.nj : G.nk) + 2;
  const double* __restrict__ pc = A.pc + p;
#pragma unroll
  for (int q = 0; q < PS_NV; q++) L[q * bt] = u0[q];
  __syncthreads();  // every thread of the block reaches each of the four
#pragma unroll
  for (int q = 0; q < PS_NV; q++) {
    um[q] = L[q * bt + pv];
    up[q] = L[q * bt + nx];
    if (pl == 0) um[q] = ue[q];
    if (pl == TP - 1) up[q] = ue[q];
  }
  // 1. slopes, shock indicator, second difference of the density
  R dm[PS_NV];
  {
    const R ta = R(pc[0]), tb = R(pc[npc]), tc = R(pc[2 * npc]);
#pragma unroll
    for (int q = 0; q < PS_NV; q++) {
      dm[q] = ppm_dma<D, R>(um[q], u0[q], up[q], ta, tb, tc);
      Lv[q * bt] = dm[q];
    }
    Ls[0] = ppm_f1<R>(pm2, um[4], up[4], pp2, um[D], up[D]);
    const R dl = R(A.dxs[p - 1]), d0 = R(A.dxs[p]), dr = R(A.dxs[p + 1]);
    Ls[bt] = (R(1) / (dl + d0 + dr)) * ((up[0] - u0[0]) / (dr + d0) - (u0[0] - um[0]) / (d0 + dl));
  }
  __syncthreads();
  // 2. face value between this cell and the next
  R V[PS_NV], dmp0 = R(0);
  {
    const R e2 = R(pc[3 * npc]), e3 = R(pc[4 * npc]), e4 = R(pc[5 * npc]), e5 = R(pc[6 * npc]);
#pragma unroll
    for (int q = 0; q < PS_NV; q++) {
      const R dmp = Lv[q * bt + nx];
      if (q == 0) dmp0 = dmp;
      V[q] = ppm_eq51<R>(u0[q], up[q], dm[q], dmp, e2, e3, e4, e5);
      L[q * bt] = V[q];
    }
  }
  const R dmm0 = Lv[pv], f1m = Ls[pv], f10 = Ls[0], f1p = Ls[nx], ddm = Ls[bt + pv], ddp = Ls[bt + nx];
  __syncthreads();
  // 3. the cell's face values: left edges to LDS, right edges kept
  R wl[9], wr[9];
  {
    const R f2 = ppm_f2<R>(f1m, f10, f1p, um[4], up[4]);
    const R eta = ppm_eta<R>(ddm, ddp, um[0], up[0], um[4], up[4], R(A.xs[p - 2]), R(A.xs[p - 1]),
                             R(A.xs[p]), gam);
#pragma unroll
    for (int q = 0; q < PS_NV; q++) {
      R l = L[q * bt + pv], r = V[q];
      if (q == 0) {
        r = mad_(r, R(1) - eta, mad_(-R(0.5), dmp0, up[0]) * eta);
        l = mad_(l, R(1) - eta, mad_(R(0.5), dmm0, um[0]) * eta);
      }
      ppm_monoto<R>(u0[q], f2, l, r);
      Lv[q * bt] = l;
      wl[ps_plane(q)] = r;
    }
  }
  __syncthreads();
  // 4. the interface
  if (in && pl >= 1 && pl <= IPT) {
#pragma unroll
    for (int q = 0; q < PS_NV; q++) wr[ps_plane(q)] = Lv[q * bt + st];
    wl[5] = wr[5] = R(0);
    const MetOf<MK, R> M(A.metF, G.P2, q2(i, k, G));
    sweep_face<D, R, ICHA>(G, F, CTsrc, c, i, j, k, M, gam, wl, wr);
  }
}

// ------------------------------------------------------------------------
// Flux-CT (Toth 2000): fluxct, ct.f90:30-118.  Reads the six transverse B
// fluxes from CTsrc (planes 0 ww(2,7) 1 ww(3,7) 2 ww(1,8) 3 ww(3,8) 4 ww(1,9)
// 5 ww(2,9), as the sweeps left them) and writes the averaged values into
// the flux array in place, like ct.f90:98-109.  FT: the stored type (float
// in the mixed form); the averages are formed in double.
// ------------------------------------------------------------------------
RH_DEV void b_cfl_finish(const CflArgs& A);

template <class FT>
RH_DEV void b_fluxct(const Geo& G, const CtArgs& A, unsigned blk) {
  if (A.fin >= 0 && blk == (unsigned)A.fin) {  // the workgroup that combines the CFL reduction
    b_cfl_finish(A.cfl);
    return;
  }
  const FT* __restrict__ CTsrc = (const FT*)A.CTsrc;
  FT* __restrict__ F1 = (FT*)A.F1;
  FT* __restrict__ F2 = (FT*)A.F2;
  FT* __restrict__ F3 = (FT*)A.F3;
  int i, j, k;
  const unsigned t = blk * blockDim.x + threadIdx.x;
  if (!box_index(t, G.nm1, G.ni - G.nm1, jlo(G, G.nm1), jhi(G, G.nj - G.nm1), G.nm1, G.nk - G.nm1, i, j, k)) return;
  const long long N = G.N;
  const unsigned c = cidx(i, j, k, G);
  const long long si = 1, sj = jstride(G), sk = kstride(G);
  const unsigned co = c * (unsigned)sizeof(FT);
  auto fyx = [&](long long d) { return ld_(CTsrc + 0 * N + d, co); };  // ww(2,7)
  auto fzx = [&](long long d) { return ld_(CTsrc + 1 * N + d, co); };  // ww(3,7)
  auto fxy = [&](long long d) { return ld_(CTsrc + 2 * N + d, co); };  // ww(1,8)
  auto fzy = [&](long long d) { return ld_(CTsrc + 3 * N + d, co); };  // ww(3,8)
  auto fxz = [&](long long d) { return ld_(CTsrc + 4 * N + d, co); };  // ww(1,9)
  auto fyz = [&](long long d) { return ld_(CTsrc + 5 * N + d, co); };  // ww(2,9)
  const double c8 = 1.0 / 8.0;
  // 2.0 * x leads each sum, so every term is added in double
  double v[6];
  v[0] = c8 * (2.0 * fyx(0) + fyx(si) + fyx(-si) - fxy(0) - fxy(sj) - fxy(-si) - fxy(-si + sj));
  v[1] = c8 * (2.0 * fzx(0) + fzx(si) + fzx(-si) - fxz(0) - fxz(sk) - fxz(-si) - fxz(-si + sk));
  v[2] = c8 * (2.0 * fxy(0) + fxy(sj) + fxy(-sj) - fyx(0) - fyx(si) - fyx(-sj) - fyx(si - sj));
  v[3] = c8 * (2.0 * fzy(0) + fzy(sj) + fzy(-sj) - fyz(0) - fyz(sk) - fyz(-sj) - fyz(-sj + sk));
  v[4] = c8 * (2.0 * fxz(0) + fxz(sk) + fxz(-sk) - fzx(0) - fzx(si) - fzx(-sk) - fzx(si - sk));
  v[5] = c8 * (2.0 * fyz(0) + fyz(sk) + fyz(-sk) - fzy(0) - fzy(sj) - fzy(-sk) - fzy(sj - sk));
  st_(F2 + 6 * N, co, FT(v[0]));
  st_(F3 + 6 * N, co, FT(v[1]));
  st_(F1 + 7 * N, co, FT(v[2]));
  st_(F3 + 7 * N, co, FT(v[3]));
  st_(F1 + 8 * N, co, FT(v[4]));
  st_(F2 + 8 * N, co, FT(v[5]));
  // the mixed form keeps the CT update of B in FP64: the update reads these
  // (the float copies above are what a later sweep keeps where its wave
  // speeds are unordered, as ww keeps what ct wrote)
  if (sizeof(FT) == 4 && A.CTd) {
#pragma unroll
    for (int q = 0; q < 6; q++) st_(A.CTd + (long long)q * N, c * 8u, v[q]);
  }
}

// ------------------------------------------------------------------------
// Recovery of primitives, recov1a (recov.f90:578-1228), one interior cell.
// u[9] = stage conserved (after RK + sources); wold = previous primitives
// (initial guess and fallback).  Writes w[9].  The initial W of a cell whose
// quadratic has no non-negative root is inherited from the previous cell in
// the reference's loop order; that cell is flagged in *carry.  s5: whether
// w[5] (a pow) is wanted; 0 otherwise.
// ------------------------------------------------------------------------
// The reference's "goto 95": W times 1.5 or 0.9 until it is admissible.  It may
// never be; the trips are bounded, and true says the bound was hit.  Such a
// cell's W wanders between the two conditions without repeating, so it needs
// all its trips, one dependent chain: they are free of branches, eight between
// two looks at the result (with a branch per condition and trip 320 cycles,
// 13.3 ms for one cell of a strongly magnetised tube, the length of the whole
// launch; now 9.5).  The first trip, which ends it for most cells, is by itself.
RH_DEV bool admissible_w(double& wg, double gf, double drogf, double gam2, double bsq, double qtsq, double qdotn,
                         double qdotbsq) {
  const double b2 = 2.0 * bsq, qb = qtsq - bsq * bsq, bq = 0.5 * bsq + qdotn, q2b = 0.5 * qdotbsq;
  int n = 0;
  auto trip = [&](bool go) {
    const double pp = gam2 * (wg * gf - drogf);
    const double wsq = wg * wg, w3 = wsq * wg;
    const double t3a = w3 * (wg + b2) - qdotbsq * (2.0 * wg + bsq);
    const double t3b = wsq * qb;
    const double t3c = w3 + wsq * (bq - pp) - q2b;
    const bool up = t3a <= t3b;
    go = go && n < 100000 && (up || t3c > 0.0);
    const double next = fabs((up ? 1.5 : (double)0.9f) * wg);
    wg = go ? next : wg;
    n += go;
    return go;
  };
  if (trip(true)) {
    bool go = true;
    while (go) {
#pragma unroll
      for (int q = 0; q < 8; q++) go = trip(go);
    }
  }
  return n >= 100000;
}

struct RecovOut { double w[9]; int fallback, fail, negrho, negp, vsqgt1, det0, guard, indep; };

template <class MT>
RH_DEV void recov_cell(const double u[9], const double wold[9], const MT& M, double gam, double dmin,
                       double pmin, int iter, double x1pow15, double x1pow25, double wg_in, bool s5, bool& carry,
                       RecovOut& o, double& wg_out) {
  const double safty = 1.0e-4, saftybig = 1.0e5, dv = 1.0e-2;
  const double gam1 = gam / (gam - 1.0);
  const double gam2 = 1.0 / gam1;
  o.fallback = o.fail = o.negrho = o.negp = o.vsqgt1 = o.det0 = o.guard = 0;
  double delta = 1.0, deltaend = 1.0e-7;
  int irecov = 0;
  const double alpha1 = M.alpha();
  const double detg1 = M.detg();
  const double dro = alpha1 * u[0] * (1.0 / detg1);
  double qcov[4], qcon[4], bcon[4], bcov[4], oncov[4], oncon[4];
  qcov[0] = alpha1 * (u[4] - u[0]) * (1.0 / detg1);
  qcov[1] = alpha1 * u[1] * (1.0 / detg1);
  qcov[2] = alpha1 * u[2] * (1.0 / detg1);
  qcov[3] = alpha1 * u[3] * (1.0 / detg1);
  const double gss = alpha1 * u[5] * (1.0 / detg1);
  bcon[0] = 0.0;
  bcon[1] = alpha1 * u[6] * (1.0 / detg1);
  bcon[2] = alpha1 * u[7] * (1.0 / detg1);
  bcon[3] = alpha1 * u[8] * (1.0 / detg1);
  double util[4] = {0.0, wold[1], wold[2], wold[3]};
  const double ro1 = wold[0], pp1 = wold[4];
  lower(bcon, bcov, M);
  upper(qcov, qcon, M);
  const double bsq = bcon[1] * bcov[1] + bcon[2] * bcov[2] + bcon[3] * bcov[3];
  const double qdotb = qcov[0] * bcon[0] + qcov[1] * bcon[1] + qcov[2] * bcon[2] + qcov[3] * bcon[3];
  const double qdotbsq = qdotb * qdotb;
  oncov[0] = -1.0 * alpha1; oncov[1] = 0.0; oncov[2] = 0.0; oncov[3] = 0.0;
  upper(oncov, oncon, M);
  const double qdotn = qcon[0] * oncov[0];
  const double qsq = qcov[0] * qcon[0] + qcov[1] * qcon[1] + qcov[2] * qcon[2] + qcov[3] * qcon[3];
  const double qtsq = qsq + (qdotn * qdotn);
  double utsq = 0.0;
#pragma unroll
  for (int m = 1; m <= 3; m++)
#pragma unroll
    for (int n = 1; n <= 3; n++) utsq = utsq + M.g(m, n) * util[m] * util[n];
  if (utsq < 0.0 && fabs(utsq) <= safty) utsq = fabs(utsq);
  if (fabs(utsq) > 1.0e4) utsq = 1.0e4;
  double gfsq = 1.0 + utsq;
  double gf = sqrt(gfsq);
  double vsq = (gfsq - 1.0) * (1.0 / gfsq);
  const double t1a = 4.0 - vsq;
  const double t1b = 4.0 * (bsq + qdotn);
  const double t1c = qtsq + bsq * bsq + 2.0 * bsq * qdotn;
  double t1d = (t1b * t1b) - 4.0 * t1a * t1c;
  if (t1d <= 0.0) t1d = fabs(t1d);
  const double wgp = (-t1b + sqrt(t1d)) * (1.0 / (2.0 * t1a));
  const double wgm = (-t1b - sqrt(t1d)) * (1.0 / (2.0 * t1a));
  double wg = wg_in;
  carry = false;
  // With a NaN among these the result and the final W are NaN whatever W the
  // cell starts from, so an inherited guess cannot change it.
  o.indep = isnan(dro) || isnan(qtsq) || isnan(qdotn) || isnan(qdotbsq) || isnan(bsq);
  if (wgp > 0.0) wg = wgp;
  else if (wgm >= 0.0) wg = wgm;
  else carry = true;
  double pp = 0.0, ro = 0.0;
  // recov.f90:823-850 ("goto 95")
  if (admissible_w(wg, gf, dro * sqrt(gf), gam2, bsq, qtsq, qdotn, qdotbsq)) o.guard = 1;
  double wsq = wg * wg;
  const double xsq = (bsq + wg) * (bsq + wg);
  vsq = fabs((wsq * qtsq + qdotbsq * (bsq + 2.0 * wg)) * (1.0 / (wsq * xsq)));
  if (vsq > 1.0) { o.vsqgt1 = 1; vsq = 1.0 - dv; }
  const double vsqo = vsq;
  double xxn = wg, yyn = vsq, w3, gtmp;
  // 2D Newton-Raphson on (W, v^2): recov.f90:877-960.  Trips after convergence
  // change nothing in the reference, so the loop stops there.  A cell whose
  // iteration never meets the tolerance runs all iter trips in the reference;
  // such an iteration usually falls into a short exact cycle of states.  Once
  // a state repeats (Brent's cycle detection) while the tolerance still fails,
  // every later trip repeats the cycle, so whole periods are skipped (with
  // their det=0 events) and the last trips run as usual: the loop ends in the
  // state, and with the count, of the reference's full run.
  unsigned long long cyx = (unsigned long long)__double_as_longlong(xxn);
  unsigned long long cyy = (unsigned long long)__double_as_longlong(yyn);
  int cy_pow = 1, cy_len = 0, cy_det0 = 0;
  for (int nnn = 1; nnn <= iter; nnn++) {
    if (!(fabs(delta) >= deltaend && irecov == 0)) break;
    if (nnn == iter) { irecov = 1; break; }
    wg = xxn; vsq = yyn;
    wsq = wg * wg; w3 = wsq * wg;
    gtmp = 1.0 - vsq;
    if (gtmp < 0.0 || gtmp < safty) { gtmp = safty; vsq = 1.0 - gtmp; }
    const double ptmp = gam2 * (wg * gtmp - dro * sqrt(gtmp));
    const double f1 = qtsq - vsq * (wg + bsq) * (wg + bsq) + (qdotbsq * (bsq + 2.0 * wg)) * (1.0 / wsq);
    const double g1 = -qdotn - 0.5 * bsq * (1.0 + vsq) + 0.5 * (qdotbsq * (1.0 / wsq)) - wg + ptmp;
    const double dpdw = gam2 * gtmp;
    const double dpdvsq = -gam2 * wg + 0.5 * gam2 * dro * (1.0 / (sqrt(gtmp)));
    const double dfx = -2.0 * (wg + bsq) * (vsq + qdotbsq * (1.0 / w3));
    const double dfy = -((wg + bsq) * (wg + bsq));
    const double dgx = -1.0 - (qdotbsq * (1.0 / w3)) + dpdw;
    const double dgy = -0.5 * bsq + dpdvsq;
    double det = dfx * dgy - dfy * dgx;
    if (det == 0.0) { o.det0 += 1; det = 1.0; }
    const double dx = (-dgy * f1 + dfy * g1) * (1.0 / det);
    const double dy = (dgx * f1 - dfx * g1) * (1.0 / det);
    delta = 0.5 * (fabs(dx) + fabs(dy));
    xxn = wg + dx;
    yyn = vsq + dy;
    if (xxn < 0.0) xxn = fabs(xxn);
    if (xxn > saftybig) xxn = saftybig;
    if (yyn < 0.0) yyn = fabs(yyn);
    if (fabs(yyn) > 1.0) yyn = 1.0 - dv;
    const unsigned long long bx = (unsigned long long)__double_as_longlong(xxn);
    const unsigned long long by = (unsigned long long)__double_as_longlong(yyn);
    cy_len++;
    if (bx == cyx && by == cyy && fabs(delta) >= deltaend) {
      const int periods = (iter - 1 - nnn) / cy_len;
      nnn += periods * cy_len;
      o.det0 += periods * (o.det0 - cy_det0);
      cy_pow = 0x40000000;
    } else if (cy_len == cy_pow) {
      cyx = bx; cyy = by; cy_pow <<= 1; cy_len = 0; cy_det0 = o.det0;
    }
  }
  if (irecov == 0) {
    wg = xxn; vsq = yyn;
    gtmp = 1.0 - vsq;
    if (gtmp < 0.0 || gtmp < safty) { gtmp = safty; vsq = 1.0 - gtmp; }
    gf = 1.0 / sqrt(gtmp);
    ro = dro * (1.0 / gf);
    const double w2 = wg * (gtmp);
    pp = gam2 * (w2 - ro);
    if (ro < 0.0 || pp < 0.0) irecov = 1;
    if (irecov == 0) {
#pragma unroll
      for (int m = 1; m <= 3; m++) {
        const double qt = qcon[m] + oncon[m] * qdotn;
        util[m] = (gf * (1.0 / (wg + bsq))) * (qt + qdotb * bcon[m] * (1.0 / wg));
      }
    }
    wg = xxn;
  }
  if (irecov == 1) {
    // entropy-based 1D inversion on v^2: recov.f90:975-1147
    o.fallback = 1;
    delta = 1.0; deltaend = 1.0e-6; irecov = 0;
    xxn = vsqo;
    // same cycle skipping as the 2D iteration; the state is v^2 alone
    unsigned long long cyv = (unsigned long long)__double_as_longlong(xxn);
    int ey_pow = 1, ey_len = 0;
    for (int nnn = 1; nnn <= iter; nnn++) {
      if (!(fabs(delta) >= deltaend && irecov == 0)) break;
      if (nnn == iter) { irecov = 1; break; }
      vsq = xxn;
      gtmp = 1.0 - vsq;
      if (gtmp < 0.0 || gtmp < safty) { gtmp = safty; vsq = 1.0 - gtmp; }
      gf = 1.0 / sqrt(gtmp);
      gfsq = gf * gf;
      ro = dro * (1.0 / gf);
      pp = (gss / dro) * (pow(ro, gam));
      const double roh = ro + gam1 * pp;
      wg = fabs(gfsq * roh);
      wsq = wg * wg; w3 = wsq * wg;
      const double dgfdvsq = 0.5 * pow(gtmp, -1.5);
      const double dwdvsq = dro * dgfdvsq + gam1 * gss * (pow(dro, gam - 1.0)) * (2.0 - gam) * (pow(gf, 1.0 - gam)) * dgfdvsq;
      const double f = qtsq - vsq * (wg + bsq) * (wg + bsq) + (qdotbsq * (bsq + 2.0 * wg)) / wsq;
      const double a = -((wg + bsq) * (wg + bsq));
      const double b = -2.0 * vsq * (wg + bsq);
      const double cc = -2.0 * qdotbsq * (bsq + 2.0 * wg) * (1.0 / w3);
      const double d = 2.0 * qdotbsq * (1.0 / wsq);
      const double df = a + (b + cc + d) * dwdvsq;
      delta = f / df;
      xxn = vsq - delta;
      if (xxn < 0.0) xxn = fabs(xxn);
      if (fabs(xxn) >= 1.0) xxn = 1.0 - dv;
      const unsigned long long bv = (unsigned long long)__double_as_longlong(xxn);
      ey_len++;
      if (bv == cyv && fabs(delta) >= deltaend) {
        nnn += ((iter - 1 - nnn) / ey_len) * ey_len;
        ey_pow = 0x40000000;
      } else if (ey_len == ey_pow) {
        cyv = bv; ey_pow <<= 1; ey_len = 0;
      }
    }
    if (irecov == 0) {
      vsq = xxn;
      gtmp = 1.0 - vsq;
      if (gtmp < 0.0 || gtmp < safty) gtmp = safty;
      gf = 1.0 / sqrt(gtmp);
      gfsq = gf * gf;
      ro = dro * (1.0 / gf);
      pp = (gss * (1.0 / gf)) * (pow(ro, gam - 1.0));
      const double roh = ro + gam1 * pp;
      if (ro < 0.0) { o.negrho = 1; ro = dmin * x1pow15; }
      if (pp < 0.0) { o.negp = 1; pp = (gam - 1.0) * pmin * x1pow25; }
      wg = fabs(gfsq * roh);
#pragma unroll
      for (int m = 1; m <= 3; m++) {
        const double qt = qcon[m] + oncon[m] * qdotn;
        util[m] = (gf / (wg + bsq)) * (qt + qdotb * bcon[m] * (1.0 / wg));
      }
    }
  }
  if (irecov == 0) {
    o.w[0] = ro; o.w[1] = util[1]; o.w[2] = util[2]; o.w[3] = util[3]; o.w[4] = pp;
    o.w[5] = s5 ? ro * pp / pow(ro, gam - 1.0) : 0.0;
  } else {
    o.fail = 1;
    o.w[0] = ro1; o.w[1] = wold[1]; o.w[2] = wold[2]; o.w[3] = wold[3]; o.w[4] = pp1;
    o.w[5] = s5 ? ro1 * pp1 / pow(ro1, gam) : 0.0;
  }
  o.w[6] = u[6] * (1.0 / detg1);
  o.w[7] = u[7] * (1.0 / detg1);
  o.w[8] = u[8] * (1.0 / detg1);
  wg_out = wg;
}

// ------------------------------------------------------------------------
// Recovery of primitives, recov2 (recov.f90:1919-2454: Mignone & McKinney
// 2007, one Newton-Raphson unknown W' = W - D, gamma-law EoS), one interior
// cell; the same interface as recov_cell.  The initial W of a cell whose
// quadratic has no admissible root is the previous cell's final W.  recov2
// prints "vsq > 1.0" at every trip that clamps v^2; vsqgt1 counts them.
// ------------------------------------------------------------------------
template <class MT>
RH_DEV void recov2_cell(const double u[9], const double wold[9], const MT& M, double gam, double dmin,
                        double pmin, int iter, double x1pow15, double x1pow25, double wg_in, bool s5, bool& carry,
                        RecovOut& o, double& wg_out) {
  const double safty = 1.0e-5, dv = 1.0e-4;
  const double gam1 = gam / (gam - 1.0);
  const double gam2 = 1.0 / gam1;
  o.fallback = o.fail = o.negrho = o.negp = o.vsqgt1 = o.det0 = o.guard = 0;
  double delta = 1.0;
  const double deltaend = 1.0e-8;
  int irecov = 0;
  const double alpha1 = M.alpha();
  const double detg1 = M.detg();
  const double dro = alpha1 * u[0] / detg1;
  double qcov[4], qcon[4], bcon[4], bcov[4], oncov[4], oncon[4];
  qcov[0] = alpha1 * (u[4] - u[0]) * (1.0 / detg1);
  qcov[1] = alpha1 * u[1] * (1.0 / detg1);
  qcov[2] = alpha1 * u[2] * (1.0 / detg1);
  qcov[3] = alpha1 * u[3] * (1.0 / detg1);
  bcon[0] = 0.0;
  bcon[1] = alpha1 * u[6] * (1.0 / detg1);
  bcon[2] = alpha1 * u[7] * (1.0 / detg1);
  bcon[3] = alpha1 * u[8] * (1.0 / detg1);
  double util[4] = {0.0, wold[1], wold[2], wold[3]};
  const double ro1 = wold[0], pp1 = wold[4];
  lower(bcon, bcov, M);
  upper(qcov, qcon, M);
  const double bsq = bcon[1] * bcov[1] + bcon[2] * bcov[2] + bcon[3] * bcov[3];
  const double qdotb = qcov[0] * bcon[0] + qcov[1] * bcon[1] + qcov[2] * bcon[2] + qcov[3] * bcon[3];
  const double qdotbsq = qdotb * qdotb;
  oncov[0] = -1.0 * alpha1; oncov[1] = 0.0; oncov[2] = 0.0; oncov[3] = 0.0;
  upper(oncov, oncon, M);
  const double qdotn = qcon[0] * oncov[0];
  const double qsq = qcov[0] * qcon[0] + qcov[1] * qcon[1] + qcov[2] * qcon[2] + qcov[3] * qcon[3];
  const double qtsq = qsq + (qdotn * qdotn);
  double utsq = 0.0;
#pragma unroll
  for (int m = 1; m <= 3; m++)
#pragma unroll
    for (int n = 1; n <= 3; n++) utsq = utsq + M.g(m, n) * util[m] * util[n];
  if (utsq < 0.0 && fabs(utsq) <= safty) utsq = fabs(utsq);
  if (utsq < 0.0 || fabs(utsq) > 1.0e4) utsq = 1.0e4;
  double gfsq = 1.0 + utsq;
  double gf = sqrt(gfsq);
  double vsq = (gfsq - 1.0) * (1.0 / gfsq);
  const double t1a = 4.0 - vsq;
  const double t1b = 4.0 * (bsq + qdotn);
  const double t1c = qtsq + bsq * bsq + 2.0 * bsq * qdotn;
  double t1d = (t1b * t1b) - 4.0 * t1a * t1c;
  if (t1d <= 0.0) t1d = fabs(t1d);
  const double wgp = (-t1b + sqrt(t1d)) * (1.0 / (2.0 * t1a));
  const double wgm = (-t1b - sqrt(t1d)) * (1.0 / (2.0 * t1a));
  double wg = wg_in;
  carry = false;
  // as in recov_cell: NaN inputs make the result independent of the guess
  o.indep = isnan(dro) || isnan(qtsq) || isnan(qdotn) || isnan(qdotbsq) || isnan(bsq);
  if (wgp > 0.0) wg = wgp;
  else if (wgm >= 0.0) wg = wgm;
  else carry = true;
  double pp = 0.0, ro = 0.0;
  // recov.f90:2150-2172 ("goto 95")
  if (admissible_w(wg, gf, dro * sqrt(gf), gam2, bsq, qtsq, qdotn, qdotbsq)) o.guard = 1;
  double wgd = wg - dro;
  double xxn = wgd;
  // Newton-Raphson on W' (recov.f90:2180-2300); a trip is a function of xxn
  // alone, so a repeated xxn while the tolerance fails is an exact cycle and
  // whole periods are skipped (with their "vsq > 1" events), as in recov_cell.
  unsigned long long cyx = (unsigned long long)__double_as_longlong(xxn);
  int cy_pow = 1, cy_len = 0, cy_vsq = 0;
  for (int nnn = 1; nnn <= iter; nnn++) {
    if (!(fabs(delta) >= deltaend && irecov == 0)) break;
    if (nnn == iter) { irecov = 1; break; }
    wgd = xxn;
    wg = wgd + dro;
    const double wsq = wg * wg;
    const double w3 = wsq * wg;
    const double xsq = (bsq + wg) * (bsq + wg);
    vsq = fabs((wsq * qtsq + qdotbsq * (bsq + 2.0 * wg)) * (1.0 / (wsq * xsq)));
    if (fabs(vsq) > 1.0) { o.vsqgt1 += 1; vsq = 1.0 - dv; }
    if (vsq < 0.0) vsq = fabs(vsq);
    double gtmp = 1.0 - vsq;
    if (gtmp < 0.0 || gtmp < safty) { gtmp = safty; vsq = 1.0 - gtmp; }
    const double usq = (1.0 - gtmp) / (gtmp);
    gf = sqrt(1.0 + usq);
    gfsq = gf * gf;
    ro = dro / gf;
    const double xi = (wg - dro * gf) * (1.0 / gfsq);
    pp = gam2 * xi;
    const double dpdxi = gam2, dpdro = 0.0;
    const double ta = (bsq + wg);
    const double tb = (bsq + wg) * (bsq + wg) * (bsq + wg);
    const double tc = (qtsq == 0.0) ? 0.0 : -2.0 * qtsq * (1.0 / tb);
    const double td = (qdotbsq == 0.0) ? 0.0 : -2.0 * qdotbsq * (3.0 * wg * ta + bsq * bsq) * (1.0 / (tb * w3));
    const double dvdwd = tc + td;
    const double dxidwd = (1.0 / gfsq) - 0.5 * gf * (dro + 2.0 * gf * xi) * dvdwd;
    const double drodwd = -0.5 * dro * gf * dvdwd;
    const double dpdwd = dpdxi * dxidwd + dpdro * drodwd;
    const double t5a = bsq * qtsq - qdotbsq;
    const double t5b = bsq + wgd + dro;
    double t5c = 0.0, t5d = 0.0;
    if (t5a != 0.0) {
      t5c = 0.5 * t5a * (1.0 / (t5b * t5b));
      t5d = t5a * (1.0 / (t5b * t5b * t5b));
    }
    const double f = -(qdotn + dro) - wgd + pp - 0.5 * bsq - t5c;
    const double df = -1.0 + dpdwd + t5d;
    delta = f / df;
    xxn = wgd - delta;
    if (xxn < 0.0) xxn = fabs(xxn);
    if (xxn > 1.0e8) xxn = 1.0e8;
    const unsigned long long bx = (unsigned long long)__double_as_longlong(xxn);
    cy_len++;
    if (bx == cyx && fabs(delta) >= deltaend) {
      const int periods = (iter - 1 - nnn) / cy_len;
      nnn += periods * cy_len;
      o.vsqgt1 += periods * (o.vsqgt1 - cy_vsq);
      cy_pow = 0x40000000;
    } else if (cy_len == cy_pow) {
      cyx = bx; cy_pow <<= 1; cy_len = 0; cy_vsq = o.vsqgt1;
    }
  }
  if (irecov == 0) {
    wgd = xxn;
    wg = wgd + dro;
    const double wsq = wg * wg;
    const double xsq = (bsq + wg) * (bsq + wg);
    vsq = fabs((wsq * qtsq + qdotbsq * (bsq + 2.0 * wg)) * (1.0 / (wsq * xsq)));
    if (vsq < 0.0) vsq = fabs(vsq);
    if (vsq > 1.0) { o.vsqgt1 += 1; vsq = 1.0 - dv; }
    double gtmp = 1.0 - vsq;
    if (gtmp < safty) gtmp = safty;
    const double usq = (1.0 - gtmp) / gtmp;
    gf = sqrt(1.0 + usq);
    gfsq = gf * gf;
    ro = dro / gf;
    const double xi = wg * (1.0 / gfsq) - ro;
    pp = gam2 * xi;
    if (ro < 0.0) { o.negrho = 1; ro = dmin * x1pow15; }
    if (pp < 0.0) { o.negp = 1; pp = pmin * (gam - 1.0) * x1pow25; }
#pragma unroll
    for (int m = 1; m <= 3; m++) {
      const double qt = qcon[m] + oncon[m] * qdotn;
      util[m] = (gf * (1.0 / (wg + bsq))) * (qt + qdotb * bcon[m] * (1.0 / wg));
    }
    o.w[0] = ro; o.w[1] = util[1]; o.w[2] = util[2]; o.w[3] = util[3]; o.w[4] = pp;
    o.w[5] = s5 ? pp / pow(ro, gam - 1.0) : 0.0;
  } else {
    o.fail = 1;
    o.w[0] = ro1; o.w[1] = wold[1]; o.w[2] = wold[2]; o.w[3] = wold[3]; o.w[4] = pp1;
    o.w[5] = s5 ? pp1 / pow(ro1, gam - 1.0) : 0.0;
  }
  o.w[6] = u[6] * (1.0 / detg1);
  o.w[7] = u[7] * (1.0 / detg1);
  o.w[8] = u[8] * (1.0 / detg1);
  wg_out = wg;
}

// one cell of the recovery iwvec selects
template <int IW, class MT>
RH_DEV void recov_any(const double u[9], const double wold[9], const MT& M, double gam, double dmin, double pmin,
                      int iter, double x1pow15, double x1pow25, double wg_in, bool s5, bool& carry, RecovOut& o,
                      double& wg_out) {
  if constexpr (IW == 2) recov2_cell(u, wold, M, gam, dmin, pmin, iter, x1pow15, x1pow25, wg_in, s5, carry, o, wg_out);
  else recov_cell(u, wold, M, gam, dmin, pmin, iter, x1pow15, x1pow25, wg_in, s5, carry, o, wg_out);
}

// ------------------------------------------------------------------------
// Update of one interior cell: flux divergence (with CT'd B fluxes), the
// geometric source (caltenr + calsf, calsf.f90:6-151), the TVD-RK stage
// (rkt.f90:2-180) plus its source add (rkt.f90:183-320), then recov1a.
// STAGE: 1 rk2fst, 2 rk2snd, 3 rk3snd, 4 rk3trd.
// ------------------------------------------------------------------------
// Plane of Gamma^l_{ab} in the Christoffel tables (christ(l,a,b) at l+4a+16b).
// SYM: the tables are bit-for-bit symmetric in (a,b) (checked on the host),
// so (a,b) and (b,a) read one plane and the compiler loads it once.
template <bool SYM>
RH_DEV long long chr_plane(int l, int a, int b) {
  if (SYM && a > b) { const int t = a; a = b; b = t; }
  return (long long)(l + 4 * a + 16 * b);
}

// The cell's index and (i,k) to c, i, k; its stage-start primitives to w; its
// updated conserved variables to put(m, value).
template <int STAGE, bool SYM, class FT, bool MK, int NGF, class Put>
RH_DEV bool rk_cell(const Geo& G, const StageArgs& A, unsigned blk, unsigned& c, int& i, int& k, double w[9], Put&& put) {
  const FT* __restrict__ F1 = (const FT*)A.F1;
  const FT* __restrict__ F2 = (const FT*)A.F2;
  const FT* __restrict__ F3 = (const FT*)A.F3;
  int j;
  const unsigned t = blk * blockDim.x + threadIdx.x;
  if (!box_index(t, G.nm1 + 1, G.ni - G.nm1, jlo(G, G.nm1 + 1), jhi(G, G.nj - G.nm1), G.nm1 + 1, G.nk - G.nm1, i, j,
                 k))
    return false;
  const long long N = G.N;
  c = cidx(i, j, k, G);
  const unsigned c8 = c * 8u;
  const long long sj = jstride(G), sk = kstride(G);
  const double gam = A.gam;
  // dt and dt/dx (main.f90:760-780), recomputed per thread from the CFL minimum
  double dt, a1, a2, a3;
  if (A.ak1) {  // akap*b and dt handed in by the caller (main.f90:760-780 on the host)
    dt = A.dt_host;
    a1 = A.ak1[i - 1]; a2 = A.ak2[j - 1]; a3 = A.ak3[k - 1];
  } else {
    const double dtcfl = __longlong_as_double((long long)A.dtbits[0]);
    dt = A.cfl * dtcfl;
    a1 = dt / A.dx1b[i - 1]; a2 = dt / A.dx2b[j - 1]; a3 = dt / A.dx3b[k - 1];
  }
  const MetOf<MK, double> M(A.metC, G.P2, q2(i, k, G));

#pragma unroll
  for (int n = 0; n < 9; n++) w[n] = ld_(A.W + (long long)n * N, c8);

  // geometric source: sf(2..5) = sqrt(-g) T^m_n Gamma^n_{(1,2,3,0) m}
  double sf[4];
  {
    Prel s;
    prelude(w, gam, M, s);
    double ta = 0.0, tb = 0.0, tc = 0.0, td = 0.0;
    const unsigned q = q2(i, k, G) * 8u;
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const double dl = (m == n) ? 1.0 : 0.0;
        const double tv = (s.roh + s.bbsq) * s.ucon[m] * s.ucov[n] + (s.pr + 0.5 * s.bbsq) * dl - s.bb[m] * s.bbcov[n];
        ta = ta + tv * ld_(A.chr + chr_plane<SYM>(n, 1, m) * G.P2, q);
        tb = tb + tv * ld_(A.chr + chr_plane<SYM>(n, 2, m) * G.P2, q);
        tc = tc + tv * ld_(A.chr + chr_plane<SYM>(n, 3, m) * G.P2, q);
        td = td + tv * ld_(A.chr + chr_plane<SYM>(n, 0, m) * G.P2, q);
      }
    const double dg = M.detg();
    sf[0] = dg * ta; sf[1] = dg * tb; sf[2] = dg * tc; sf[3] = dg * td;
  }

  // transverse-B fluxes from flux-CT's FP64 planes in the mixed form
  // (component m, direction d -> plane; -1: the sweep's own flux)
  constexpr int ctp[3][3] = {{-1, 0, 1}, {2, -1, 3}, {4, 5, -1}};
  const bool ctd = sizeof(FT) == 4 && A.CTd;
  const unsigned cf = c * (unsigned)sizeof(FT);
  auto fl = [&](int m, int d, long long off) -> double {
    const FT* Fd = d == 0 ? F1 : d == 1 ? F2 : F3;
    if (m >= 6 && ctd && ctp[m - 6][d] >= 0) return ld_(A.CTd + (long long)ctp[m - 6][d] * N - off, c8);
    return double(ld_(Fd + (long long)m * N - off, cf));
  };
  // Several variables at a time, their reads in flight together (left to
  // itself the compiler waits for one variable's eight before the next one's):
  // three in FP64 (256x128x128 0.449 -> 0.431 ms, with all nine 0.479; one
  // 128x128 row 11.7 -> 7.8 us); where the fluxes are floats NGF, nine in the
  // update alone (0.401 -> 0.377 ms, with three 0.414) and one in the fused
  // kernel, whose registers more of them would spill (0.432, three 0.613).
  constexpr int NG = sizeof(FT) == 4 ? NGF : 3;
#pragma unroll
  for (int g = 0; g < 9; g += NG) {
    double f[NG][6], ua[NG], ub[NG];
#pragma unroll
    for (int q = 0; q < NG; q++) {
      const int m = g + q;
      f[q][0] = fl(m, 0, 0); f[q][1] = fl(m, 0, 1);
      f[q][2] = fl(m, 1, 0); f[q][3] = fl(m, 1, sj);
      f[q][4] = fl(m, 2, 0); f[q][5] = fl(m, 2, sk);
      ua[q] = ld_(A.Ua + (long long)m * N, c8);
      ub[q] = STAGE == 1 ? 0.0 : ld_(A.Ub + (long long)m * N, c8);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < NG; q++) {
      const int m = g + q;
      const double d1 = f[q][0] - f[q][1], d2 = f[q][2] - f[q][3], d3 = f[q][4] - f[q][5];
      double v;
      if (STAGE == 1) {
        v = ua[q] - a1 * d1 - a2 * d2 - a3 * d3;
      } else if (STAGE == 2) {
        v = (ua[q] + ub[q]) * 0.5 + (-a1 * d1 - a2 * d2 - a3 * d3) * 0.5;
      } else if (STAGE == 3) {
        v = (3.0 * ua[q] + ub[q]) * 0.25 + (-a1 * d1 - a2 * d2 - a3 * d3) * 0.25;
      } else {
        v = (ua[q] + 2.0 * ub[q]) * (double)(1.0f / 3.0f) + (-a1 * d1 - a2 * d2 - a3 * d3) * (double)(2.0f / 3.0f);
      }
      if (m >= 1 && m <= 4) {
        const double sdt = sf[m - 1] * dt;
        if (STAGE == 1) v = v + sdt;
        else if (STAGE == 2) v = v + sdt * 0.5;
        else if (STAGE == 3) v = v + sdt * 0.25;
        else v = v + sdt * (double)(2.0f / 3.0f);
      }
      put(m, v);
    }
  }
  return true;
}

template <int STAGE, bool SYM, class FT, bool MK>
RH_DEV void b_rk(const Geo& G, const StageArgs& A, unsigned blk) {
  unsigned c;
  int i, k;
  double w[9];
  rk_cell<STAGE, SYM, FT, MK, 9>(G, A, blk, c, i, k, w,
                              [&](int m, double v) { st_(A.Ukeep + (long long)m * G.N, c * 8u, v); });
}

// recov1a (recov.f90:578-1228) or recov2 (recov.f90:1919-2454) on every
// interior cell from the stage's RK result; cells whose initial W is
// inherited are flagged for k_recov_carry.
template <int IW, bool MK>
RH_DEV void recov_put(const Geo& G, const StageArgs& A, unsigned blk, unsigned c, int i, int k, const double u[9],
                      const double w[9], bool keep) {
  const long long N = G.N;
  const MetOf<MK, double> M(A.metC, G.P2, q2(i, k, G));
  RecovOut ro;
  bool carry;
  double wgout;
  recov_any<IW>(u, w, M, A.gam, A.dmin, A.pmin, A.iter, A.r15[i - 1], A.r25[i - 1], __builtin_nan(""), A.s5,
                carry, ro, wgout);
  const bool dep = carry && !ro.indep;
#pragma unroll
  for (int n = 0; n < 9; n++) st_(A.Wpre + (long long)n * N, c * 8u, ro.w[n]);
  st_(A.wgout, c * 8u, wgout);
  // a flagged cell's outcome is counted when the fix-up computes it
  count_wave(A.cpart, blk, C_FALLBACK, ro.fallback && !dep);
  count_wave(A.cpart, blk, C_FAIL, ro.fail && !dep);
  count_wave(A.cpart, blk, C_NEGRHO, ro.negrho && !dep);
  count_wave(A.cpart, blk, C_NEGP, ro.negp && !dep);
  count_wave(A.cpart, blk, C_VSQGT1, ro.vsqgt1 && !dep);
  if (ro.vsqgt1 > 1 && !dep) atomicAdd(&A.cnt[C_VSQGT1], (unsigned long long)(ro.vsqgt1 - 1));  // recov2: per trip
  if (ro.det0 && !dep) atomicAdd(&A.cnt[C_DET0], (unsigned long long)ro.det0);  // rare: one event per det=0 trip
  count_wave(A.cpart, blk, C_WGCARRY, carry);
  count_wave(A.cpart, blk, C_GUARD, ro.guard && !dep);
  if (dep) {
    // remember the cell for the in-order resolution
    A.cflag[c] = 1;
    const unsigned long long slot = atomicAdd(&A.carry[0], 1ULL);
    if (slot < (unsigned long long)A.carry_cap) A.carry[1 + slot] = (unsigned long long)c;
    if (keep)
#pragma unroll
      for (int n = 0; n < 9; n++) st_(A.Ukeep + (long long)n * N, c * 8u, u[n]);
  }
}

template <int IW, bool MK>
RH_DEV void b_recov(const Geo& G, const StageArgs& A, unsigned blk) {
  int i, j, k;
  const unsigned t = blk * blockDim.x + threadIdx.x;
  if (!box_index(t, G.nm1 + 1, G.ni - G.nm1, jlo(G, G.nm1 + 1), jhi(G, G.nj - G.nm1), G.nm1 + 1, G.nk - G.nm1, i, j,
                 k))
    return;
  const long long N = G.N;
  const unsigned c = cidx(i, j, k, G);
  double w[9], u[9];
#pragma unroll
  for (int n = 0; n < 9; n++) {
    w[n] = ld_(A.W + (long long)n * N, c * 8u);
    u[n] = ld_((const double*)A.Ukeep + (long long)n * N, c * 8u);
  }
  recov_put<IW, MK>(G, A, blk, c, i, k, u, w, false);
}

// The update and the recovery of a cell in one kernel: the stage's conserved
// variables stay in registers (they are read again only where k_recov_carry
// has the cell, which finds them in Ukeep), and W is read once: 27 planes
// less.  164 VGPRs put it at 3 waves per SIMD, enough for the update's reads
// since they go out in groups: 256x128x128 0.433 + 0.166 -> 0.466 ms, 64^3
// 33 -> 24 us, one 128x128 row 14.2 -> 11.3 us.
template <int STAGE, class FT, int IW>
RH_DEV void b_rkrecov(const Geo& G, const StageArgs& A, unsigned blk) {
  unsigned c;
  int i, k;
  double w[9], u[9];
  if (!rk_cell<STAGE, true, FT, true, 1>(G, A, blk, c, i, k, w, [&](int m, double v) { u[m] = v; })) return;
  recov_put<IW, true>(G, A, blk, c, i, k, u, w, true);
}

// ------------------------------------------------------------------------
// Ghost fill + floors + conserved variables, every cell.
// bnd4 (bnd.f90:4-1059) is composed per cell: the value a ghost holds after
// the periodic pass, then the x1, x2, x3 passes.  Then infchk (bnd.f90:1636),
// atmosphere1a (correction.f90:226), pminmax2b (correction.f90:744) and
// caluu1 (caluu.f90:2).
// ------------------------------------------------------------------------
RH_DEV bool is_ghost(int p, int n, int nm1) { return p <= nm1 || p > n - nm1; }

// p folded into the interior by whole periods (nm1 periods reach past every ghost)
RH_DEV int fold(int p, int n, int nm1) {
  const unsigned Wd = (unsigned)(n - 2 * nm1);
  return nm1 + 1 + (int)((unsigned)(p - (nm1 + 1) + nm1 * (int)Wd) % Wd);
}

// One variable's planes and boundary codes (bc[axis*2+side]) in the ghost fill.
struct BndVar {
  const double* Wpre;   // post-recov interior values
  const double* Wold;   // values before this stage (ghosts not rewritten keep these)
  const double* Wo;     // primitives at the start of the step (fixed-value type 2)
  const int *bc, *bc2;  // its codes bc[axis*2+side], and those of u^1
  long long v2;         // from these planes to those of u^1
};

// value after the periodic pass (bndpefb4)
RH_DEV double bnd_s0(const Geo& G, const BndVar& B, int i, int j, int k) {
  const int nm1 = G.nm1;
  const bool gi = is_ghost(i, G.ni, nm1), gj = is_ghost(j, G.nj, nm1), gk = is_ghost(k, G.nk, nm1);
  const int ng = (int)gi + (int)gj + (int)gk;
  bool inner = ng == 0;
  if (ng == 1) {
    if (gi && (B.bc[0] == 1 || B.bc[1] == 1)) { i = fold(i, G.ni, nm1); inner = true; }
    else if (gj && (B.bc[2] == 1 || B.bc[3] == 1)) { j = fold(j, G.nj, nm1); inner = true; }
    else if (gk && (B.bc[4] == 1 || B.bc[5] == 1)) { k = fold(k, G.nk, nm1); inner = true; }
  }
  return (inner ? B.Wpre : B.Wold)[cidx(i, j, k, G)];
}

// Value at ghost (i,j,k) after the three physical passes.  Each pass maps the
// cell to its source in the previous pass (copy, mirror, with a sign for
// antisymmetric codes) or ends in a constant: walking x3 -> x2 -> x1 and then
// reading the periodic-pass value composes the passes exactly.
RH_DEV double bnd_value(const Geo& G, const BndVar& B, int i, int j, int k) {
  const int nm1 = G.nm1;
  double sgn = 1.0;
  int c[4] = {0, i, j, k};
  const int n[4] = {0, G.ni, G.nj, G.nk};
#pragma unroll
  for (int ax = 3; ax >= 1; ax--) {
    const int p = c[ax];
    if (!is_ghost(p, n[ax], nm1)) continue;
    const bool outer = p > n[ax] - nm1;
    const int type = outer ? B.bc[(ax - 1) * 2 + 1] : B.bc[(ax - 1) * 2];
    if (type == 5) {
      c[ax] = outer ? n[ax] - nm1 : nm1 + 1;
    } else if (type == 12 || type == 14) {
      if (type == 12) sgn = -sgn;
      c[ax] = outer ? 2 * n[ax] - 2 * nm1 + 1 - p : 2 * nm1 - p + 1;
    } else if (type == 13) {
      return sgn * 0.0;
    } else if (type == 2) {
      return sgn * B.Wo[cidx(c[1], c[2], c[3], G)];
    } else if (type == 18) {
      // bnd.f90:598-610 (x1 outer only, u^1 to u^3): no inflow through the outer boundary
      BndVar V = B;
      V.Wpre = B.Wpre + B.v2;
      V.Wold = B.Wold + B.v2;
      V.bc = B.bc2;
      if (bnd_s0(G, V, n[ax] - nm1, c[2], c[3]) < 0.0) return sgn * 0.0;
      c[ax] = n[ax] - nm1;
    }  // 1: periodic, filled by the periodic pass
  }
  return sgn * bnd_s0(G, B, c[1], c[2], c[3]);
}

// 1-based (i,j,k) of the t-th ghost cell: the two theta slabs (all i, j),
// then the two phi slabs (interior k), then the two r slabs (interior j, k).
// A collapsed model stores no phi ghosts: its row's theta and r ghosts.
RH_DEV bool ghost_index(unsigned t, const Geo& G, int& i, int& j, int& k) {
  const unsigned ni = G.ni, nj = G.jfix ? 1u : (unsigned)G.nj, nk = G.nk, g = G.nm1;
  const unsigned jin = G.jfix ? 1u : nj - 2 * g, j0 = G.jfix ? (unsigned)G.jfix - 1u : 0u;
  const unsigned nkS = 2 * g * ni * nj, njS = G.jfix ? 0u : 2 * g * ni * (nk - 2 * g), niS = 2 * g * jin * (nk - 2 * g);
  auto slab = [&](unsigned a, unsigned n) { return (int)(a < g ? a : n - 2 * g + a) + 1; };
  if (t < nkS) {
    const unsigned r = t / ni, kk = r / nj;
    i = (int)(t - r * ni) + 1;
    j = (int)(j0 + r - kk * nj) + 1;
    k = slab(kk, nk);
    return true;
  }
  t -= nkS;
  if (t < njS) {
    const unsigned r = t / ni, kk = r / (2 * g);
    i = (int)(t - r * ni) + 1;
    j = slab(r - kk * 2 * g, nj);
    k = (int)(g + kk) + 1;
    return true;
  }
  t -= njS;
  if (t < niS) {
    const unsigned r = t / (2 * g), kk = r / jin;
    i = slab(t - r * 2 * g, ni);
    j = (int)((G.jfix ? j0 : g) + r - kk * jin) + 1;
    k = (int)(g + kk) + 1;
    return true;
  }
  return false;
}

// Ghost fill of the stage: bnd4 composed per ghost cell, written into the
// ghost slots of the recovered primitives.  bnd_value reads only interior
// cells of that array (and the stage-start values of other ghosts), so the
// writes cannot race with the reads.  A thread takes NV variables of a ghost
// cell, the same ones in its workgroup (A.nbc workgroups per NV variables),
// so their codes are scalars and their reads in flight together: one where
// the launch is then still small (every read's latency counts: one 128x128
// row 4.4 us, with three 6.4 us), three beyond (they share the thread's index
// arithmetic: 256x128x128 0.046 ms, with one 0.048; eight 1024-zone tubes
// 0.054, with one 0.064).  A thread that took the nine in turn waited nine
// times: 13.2 us, 0.054 and 0.062 ms.
template <int NV>
RH_DEV void bnd_cells(const Geo& G, const PostArgs& A, unsigned blk) {
  const int g = (int)(blk / (unsigned)A.nbc);
  int i, j, k;
  if (!ghost_index((blk - (unsigned)g * (unsigned)A.nbc) * blockDim.x + threadIdx.x, G, i, j, k)) return;
  const unsigned c = cidx(i, j, k, G);
  double v[NV];
#pragma unroll
  for (int q = 0; q < NV; q++) {
    const int m = NV * g + q;
    const long long o = (long long)m * G.N;
    int bc[6], bc2[6];
#pragma unroll
    for (int e = 0; e < 6; e++) { bc[e] = A.bc[e * 9 + m]; bc2[e] = A.bc[e * 9 + 1]; }
    v[q] = bnd_value(G, BndVar{A.Wpre + o, A.Wold + o, A.Wo + o, bc, bc2, (1 - m) * G.N}, i, j, k);
  }
#pragma unroll
  for (int q = 0; q < NV; q++) A.Wghost[(long long)(NV * g + q) * G.N + c] = v[q];
}
RH_DEV void b_bnd(const Geo& G, const PostArgs& A, unsigned blk) {
  if (A.nbv == 1) bnd_cells<1>(G, A, blk);
  else bnd_cells<3>(G, A, blk);
}

// infchk + atmosphere1a + pminmax2b + caluu1 on every cell, after k_bnd.
// The metric of cell (i,k) through a pointer the compiler cannot see
// through, so its values are loaded again (from cache) in the next phase
// instead of being held in registers across phases.  k_post's three phases
// each read the 32 metric values; holding them costs two waves per SIMD.
template <bool MK>
RH_DEV MetOf<MK, double> reload_met(const void* metC, const Geo& G, int i, int k) {
  asm volatile("" : "+s"(metC));
  return MetOf<MK, double>(metC, G.P2, q2(i, k, G));
}

template <bool MK>
RH_DEV void b_post(const Geo& G, const PostArgs& A, unsigned blk) {
  const unsigned t = blk * blockDim.x + threadIdx.x;
  int i, j, k;
  if (!box_index(t, 1, G.ni, jlo(G, 1), jhi(G, G.nj), 1, G.nk, i, j, k)) return;
  const long long N = G.N;
  const unsigned c = cidx(i, j, k, G);
  const double gam = A.gam;
  const MetOf<MK, double> M(A.metC, G.P2, q2(i, k, G));
  double w[9];
#pragma unroll
  for (int n = 0; n < 9; n++) w[n] = ld_(A.Wpre + (long long)n * N, c * 8u);
  // infchk, outer radial ghosts (bnd.f90:1740-1819); model 7..20
  if (A.model >= 7 && A.model <= 20 && i > G.ni - G.nm1) {
    const double gfl = calgfl(w[1], w[2], w[3], M);
    double vel[4];
    vel[1] = w[1] * (1.0 / gfl);
    vel[2] = w[2] * (1.0 / gfl);
    vel[3] = w[3] * (1.0 / gfl);
    if (vel[1] < 0.0) {
      vel[1] = M.beta(1) * M.ralpha();
      double vsq = 0.0;
#pragma unroll
      for (int m = 1; m <= 3; m++)
#pragma unroll
        for (int nn = 1; nn <= 3; nn++) vsq = vsq + M.g(m, nn) * vel[m] * vel[nn];
      if (vsq >= 1.0) vsq = 1.0 - 1.0 / (10.0 * 10.0);
      const double g2 = 1.0 / sqrt(1.0 - vsq);
      w[1] = vel[1] * g2; w[2] = vel[2] * g2; w[3] = vel[3] * g2;
    }
  }
  const double demin = A.dmin * A.r15[i - 1];
  const double prmin = (gam - 1.0) * A.pmin * A.r25[i - 1];
  // atmosphere1a (model 7..15): correction.f90:276-393
  bool atm = false;
  if (A.model >= 7 && A.model <= 15) {
    const double dthe = 1.0 * (1.0 + 1.0e-2) * demin;
    const double dthe1 = 1.0 * (1.0 + 1.0e-2) * prmin;
    const double bsq = w[6] * w[6] + w[7] * w[7] + w[8] * w[8];
    if (w[0] < dthe || (w[4] < dthe1 && bsq <= 1.0e-20)) {
      atm = true;
      double vsq = 0.0;
      const double vel[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int m = 1; m <= 3; m++)
#pragma unroll
        for (int nn = 1; nn <= 3; nn++) vsq = vsq + M.g(m, nn) * vel[m] * vel[nn];
      if (vsq >= 1.0) vsq = 1.0 - 1.0 / (10.0 * 10.0);
      const double g2 = 1.0 / sqrt(1.0 - vsq);
      w[0] = demin; w[4] = prmin;
      w[1] = vel[1] * g2; w[2] = vel[2] * g2; w[3] = vel[3] * g2;
    }
    w[5] = 0.0;
  }
  // a collapsed model's cell stands for its nj phi copies, each counted by the reference
  const unsigned long long rows = G.jfix ? (unsigned long long)G.nj : 1ULL;
  count_wave(A.cpart, blk, C_ATM, atm, rows);
  // pminmax2b: correction.f90:808-961
  bool scaled = false, hit = false;
  {
    const auto M = reload_met<MK>(A.metC, G, i, k);
    const double gflmax = 20.0;
    double gfl = calgfl(w[1], w[2], w[3], M);
    double vel[4];
    vel[1] = w[1] * (1.0 / gfl);
    vel[2] = w[2] * (1.0 / gfl);
    vel[3] = w[3] * (1.0 / gfl);
    double vsq = 0.0;
#pragma unroll
    for (int m = 1; m <= 3; m++)
#pragma unroll
      for (int nn = 1; nn <= 3; nn++) vsq = vsq + M.g(m, nn) * vel[m] * vel[nn];
    if (vsq >= 1.0 || gfl > gflmax) vsq = 1.0 - 1.0 / (gflmax * gflmax);
    gfl = 1.0 / sqrt(1.0 - vsq);
    Prel s;
    const double wl[9] = {w[0], vel[1] * gfl, vel[2] * gfl, vel[3] * gfl, w[4], w[5], w[6], w[7], w[8]};
    prelude(wl, gam, M, s);  // gfl, u^mu, b^mu of the limited velocity
    gfl = s.gfl;
    const double bcon1[4] = {0.0, w[6], w[7], w[8]};
    double bcov1[4];
    lower(bcon1, bcov1, M);
    const double bsq = bcon1[1] * bcov1[1] + bcon1[2] * bcov1[2] + bcon1[3] * bcov1[3];
    double de = w[0], pr = w[4];
    int guard = 0;
    for (; guard < 100000; guard++) {
      const double roh = de + (gam / (gam - 1.0)) * pr;
      const double t1a = roh * gfl * gfl - pr;
      const double t1b = fabs((double)0.05f * bsq);
      if (t1a <= t1b) { de = (double)1.05f * de; pr = (double)1.05f * pr; scaled = true; continue; }
      break;
    }
    if (de != w[0]) w[0] = de;
    else if (pr != w[4]) w[4] = pr;
    if (pr < prmin) { w[4] = prmin; hit = true; }
    if (pr > A.pmax) { w[4] = A.pmax; hit = true; }
    if (de < demin) { w[0] = demin; hit = true; }
    const double prro = w[4] * (1.0 / w[0]);
    if (prro > 1.0e6) { w[0] = w[4] / 1.0e6; hit = true; }
    const double bbro = s.bbsq * (1.0 / w[0]);
    const double bbpr = s.bbsq * (1.0 / w[4]);
    if (bbro > 50.0) { w[0] = s.bbsq / 50.0; hit = true; }
    if (bbpr > 2.0e3) { w[4] = s.bbsq / 2.0e3; hit = true; }
  }
  count_wave(A.cpart, blk, C_PMMSCALE, scaled, rows);
  count_wave(A.cpart, blk, C_PMMFLOOR, hit, rows);
#pragma unroll
  for (int n = 0; n < 9; n++) st_(A.Wout + (long long)n * N, c * 8u, w[n]);
  // caluu1 (caluu.f90:2-126): conserved variables of the final primitives
  {
    const auto M = reload_met<MK>(A.metC, G, i, k);
    Prel s2;
    prelude(w, gam, M, s2);
    double u[9];
    tmunu_row(s2, 0, M.detg(), pow(s2.de, gam), u);
#pragma unroll
    for (int n = 0; n < 9; n++) st_(A.Uout + (long long)n * N, c * 8u, u[n]);
  }
}

// ------------------------------------------------------------------------
// CFL: cdtcfl4 (cdtcfl.f90:2-129) with calcha4 centre speeds.
// The reference folds dtcfl = MIN(dtcfl, x) over the cells in (k,j,i) order,
// and MIN(a,b) = a<b?a:b: a NaN element sets the running value to NaN and
// the next element replaces it.  So the result is the minimum over the
// elements after the last NaN (NaN if a NaN is the last element; 1.0 and all
// elements if there is none).  Each workgroup reduces its contiguous range of
// A.per cells, a thread each at a time, to (position of its last NaN, minimum after it)
// with wavefront shuffles; one workgroup then combines their results in order
// and, in a step, advances the time (main.f90:760-781).  (The last workgroup
// to finish doing that in the same launch measured slower: its device-scope
// fence writes the L2 back in every workgroup, 256x128x128 0.135 -> 0.21 ms.)
// Accumulators: 0 dtcfl (three elements per cell: dtx1a, dtx2a, dtx3a),
// 1..3 dtx1..dtx3 (one element per cell).
// ------------------------------------------------------------------------
RH_DEV double wave_min(double v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const double o = __shfl_xor(v, off, 64);
    v = (o < v) ? o : v;  // operands are never NaN here
  }
  return v;
}
RH_DEV int wave_max(int v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const int o = __shfl_xor(v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}

// The four accumulators' values over a workgroup of at most 256 (maximum of
// v, or minimum of m), every thread the same.
RH_DEV void group_max4(int v[4]) {
  __shared__ int part[4][4];
  const int lane = threadIdx.x % 64, wid = threadIdx.x / 64;
  __syncthreads();
#pragma unroll
  for (int a = 0; a < 4; a++) {
    const int w = wave_max(v[a]);
    if (lane == 0) part[wid][a] = w;
  }
  __syncthreads();
#pragma unroll
  for (int a = 0; a < 4; a++) {
    v[a] = part[0][a];
    for (int w = 1; w < (int)(blockDim.x / 64); w++) v[a] = part[w][a] > v[a] ? part[w][a] : v[a];
  }
}
RH_DEV void group_min4(double m[4]) {
  __shared__ double part[4][4];
  const int lane = threadIdx.x % 64, wid = threadIdx.x / 64;
  __syncthreads();
#pragma unroll
  for (int a = 0; a < 4; a++) {
    const double w = wave_min(m[a]);
    if (lane == 0) part[wid][a] = w;
  }
  __syncthreads();
#pragma unroll
  for (int a = 0; a < 4; a++) {
    m[a] = part[0][a];
    for (int w = 1; w < (int)(blockDim.x / 64); w++) m[a] = (part[w][a] < m[a]) ? part[w][a] : m[a];
  }
}

// Signal times of the cell at box position t (dtx1a, dtx2a, dtx3a); infinite
// past the box.
template <int ICHA, bool MK>
RH_DEV bool cfl_cell(const Geo& G, const CflArgs& A, unsigned t, double e[3]) {
  int i, j, k;
  e[0] = e[1] = e[2] = __builtin_inf();
  if (!box_index(t, 2, G.ni - 1, jlo(G, 2), jhi(G, G.nj - 1), 2, G.nk - 1, i, j, k)) return false;
  const long long N = G.N;
  const unsigned c = cidx(i, j, k, G);
  const MetOf<MK, double> M(A.metC, G.P2, q2(i, k, G));
  double w[9];
#pragma unroll
  for (int n = 0; n < 9; n++) w[n] = ld_(A.W + (long long)n * N, c * 8u);
  Prel s;
  prelude(w, A.gam, M, s);
  double vp[4], vm[4];
  centre_speeds<ICHA>(s, A.gam, M, vp, vm);
  const int nmax = G.nm1 * 2 + (G.nm1 - 1);
  const int nd[4] = {0, G.ni, G.nj, G.nk};
  const double dxv[4] = {0.0, A.dx1b[i - 1], A.dx2b[j - 1], A.dx3b[k - 1]};
#pragma unroll
  for (int q = 1; q <= 3; q++) {
    double vf = fmaxf_(fmaxf_(0.0, fabs(vp[q])), fabs(vm[q]));
    if (nd[q] > nmax && vf > 0.0) {
      if (vf > 1.0) vf = 1.0;
      e[q - 1] = fabs(dxv[q] / (vf + 1.0e-12));
    } else {
      e[q - 1] = 1.0e10;
    }
  }
  return true;
}

template <int ICHA, bool MK>
RH_DEV void b_cfl(const Geo& G, const CflArgs& A, unsigned blk) {
  // the workgroup's last NaN per accumulator (positions below 3 * 2^29) and
  // the minimum after it; without a NaN among the cells, a plain minimum
  int L[4] = {-1, -1, -1, -1};
  double mn[4];
#pragma unroll
  for (int a = 0; a < 4; a++) mn[a] = __builtin_inf();
  const unsigned t0 = blk * (unsigned)A.per;
  for (unsigned b = 0; b < (unsigned)A.per; b += blockDim.x) {
    const int t = (int)(t0 + b + threadIdx.x);
    double e[3];
    const bool valid = cfl_cell<ICHA, MK>(G, A, (unsigned)t, e);
    if (__syncthreads_or(valid && (isnan(e[0]) || isnan(e[1]) || isnan(e[2])))) {
      // minima so far count only where this chunk has no NaN of the accumulator
      int last[4] = {-1, -1, -1, -1};
#pragma unroll
      for (int q = 0; q < 3; q++)
        if (valid && isnan(e[q])) { last[0] = 3 * t + q; last[q + 1] = t; }
      group_max4(last);
#pragma unroll
      for (int a = 0; a < 4; a++)
        if (last[a] >= 0) { L[a] = last[a]; mn[a] = __builtin_inf(); }
#pragma unroll
      for (int q = 0; q < 3; q++) {
        if (!valid || isnan(e[q])) continue;
        if (3 * t + q > last[0]) mn[0] = (e[q] < mn[0]) ? e[q] : mn[0];
        if (t > last[q + 1]) mn[q + 1] = (e[q] < mn[q + 1]) ? e[q] : mn[q + 1];
      }
    } else {
#pragma unroll
      for (int q = 0; q < 3; q++) {
        mn[0] = (e[q] < mn[0]) ? e[q] : mn[0];
        mn[q + 1] = (e[q] < mn[q + 1]) ? e[q] : mn[q + 1];
      }
    }
  }
  group_min4(mn);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int a = 0; a < 4; a++) { A.blast[4 * blk + a] = L[a]; A.bmin[4 * blk + a] = mn[a]; }
  }
}

// One workgroup combines the results of A.nblocks workgroups.
RH_DEV void b_cfl_finish(const CflArgs& A) {
  double mn[4];
  // the last NaN lies in the last workgroup that has one; that workgroup's
  // minimum after it and the full minima of every later one make the result
  int B[4] = {-1, -1, -1, -1};
  for (int q = threadIdx.x; q < A.nblocks; q += blockDim.x)
#pragma unroll
    for (int a = 0; a < 4; a++)
      if (A.blast[4 * q + a] >= 0) B[a] = q;
  group_max4(B);
#pragma unroll
  for (int a = 0; a < 4; a++) mn[a] = __builtin_inf();
  for (int q = threadIdx.x; q < A.nblocks; q += blockDim.x)
#pragma unroll
    for (int a = 0; a < 4; a++)
      if (q >= B[a]) { const double v = A.bmin[4 * q + a]; mn[a] = (v < mn[a]) ? v : mn[a]; }
  group_min4(mn);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int a = 0; a < 4; a++) {
      double r;
      if (B[a] < 0) r = fminf_(1.0, mn[a]);                               // no NaN: MIN over 1.0 and all
      else r = (mn[a] == __builtin_inf()) ? __builtin_nan("") : mn[a];  // a trailing NaN stays
      A.dtbits[a] = (unsigned long long)__double_as_longlong(r);
      if (a == 0 && A.tdt) {  // time <- time + cfl*dtcfl; last dt kept
        const double dt = A.cfl * r;
        A.tdt[0] = A.tdt[0] + dt;
        A.tdt[1] = dt;
      }
    }
  }
}

// Resolution of cells whose initial W is inherited from the previous cell in
// the reference's (k,j,i) loop order (recov.f90:815-817 leaves wg unchanged,
// recov.f90:632 starts it at 0).  A flagged cell is computed once its
// predecessor's final W is known.
//
// Chain heads (flagged cells whose predecessor is not flagged, or that open
// the loop) are independent: every workgroup of the launch takes a share of
// them.  The last workgroup to finish (a device-scope counter after a
// device-scope fence) then resolves the remaining links in passes over the
// flagged list, each pass taking the cells whose predecessor is resolved,
// until none is left: a chain of consecutive flagged cells takes one pass
// per link.  A batch runs one workgroup per member, which does both parts.

// Predecessor of interior cell c in (k,j,i) order, -1 for the first cell.
RH_DEV long long carry_pred(const Geo& G, long long c, int& i, int& k) {
  const long long sk = kstride(G);
  i = (int)(c % G.ni) + 1;
  k = (int)(c / sk) + 1;
  const int j = G.jfix ? G.jfix : (int)((c / G.ni) % G.nj) + 1;
  int pi = i - 1, pj = j, pk = k;
  if (pi < G.nm1 + 1) { pi = G.ni - G.nm1; pj = j - 1; if (pj < G.nm1 + 1) { pj = G.nj - G.nm1; pk = k - 1; } }
  return pk >= G.nm1 + 1 ? (long long)cidx(pi, pj, pk, G) : -1LL;
}

template <int IW, bool MK>
RH_DEV void carry_cell(const Geo& G, const FixArgs& A, long long c, int i, int k, double wg_prev) {
  const long long N = G.N;
  const MetOf<MK, double> M(A.metC, G.P2, q2(i, k, G));
  double u[9], w[9];
  for (int m = 0; m < 9; m++) { u[m] = A.Ustage[(long long)m * N + c]; w[m] = A.W[(long long)m * N + c]; }
  RecovOut ro;
  bool carry;
  double wgout;
  recov_any<IW>(u, w, M, A.gam, A.dmin, A.pmin, A.iter, A.r15[i - 1], A.r25[i - 1], wg_prev, A.s5, carry, ro,
                wgout);
  for (int m = 0; m < 9; m++) A.Wpre[(long long)m * N + c] = ro.w[m];
  A.wgout[c] = wgout;
  if (ro.fallback) atomicAdd(&A.cnt[C_FALLBACK], 1ULL);
  if (ro.fail) atomicAdd(&A.cnt[C_FAIL], 1ULL);
  if (ro.negrho) atomicAdd(&A.cnt[C_NEGRHO], 1ULL);
  if (ro.negp) atomicAdd(&A.cnt[C_NEGP], 1ULL);
  if (ro.vsqgt1) atomicAdd(&A.cnt[C_VSQGT1], (unsigned long long)ro.vsqgt1);
  if (ro.det0) atomicAdd(&A.cnt[C_DET0], (unsigned long long)ro.det0);
  if (ro.guard) atomicAdd(&A.cnt[C_GUARD], 1ULL);
}

// grp/ngrp: this workgroup's place among those sharing the chain heads
// (ngrp == 1: the workgroup does everything and needs no counter).
// Pass -1 takes the chain heads (pend 2 = resolved, 1 = waits for its
// predecessor); passes 0, 1, ... (last workgroup) take the links.  One loop
// body, so the recovery is compiled once.
template <int IW, bool MK>
RH_DEV void b_recov_carry(const Geo& G, const FixArgs& A, int grp, int ngrp) {
  __shared__ int s_progress, s_left, s_last;
  unsigned long long n = A.carry[0];
  if (n == 0) return;
  if (n > (unsigned long long)A.carry_cap) n = (unsigned long long)A.carry_cap;
  const unsigned long long* list = A.carry + 1;
  unsigned char* pend = A.pend;
  for (int pass = -1; pass < (1 << 22); pass++) {
    const bool heads = pass < 0;
    if (!heads) {
      if (threadIdx.x == 0) { s_progress = 0; s_left = 0; }
      __syncthreads();
    }
    const unsigned long long e0 = heads ? (unsigned long long)grp * blockDim.x + threadIdx.x : threadIdx.x;
    const unsigned long long es = heads ? (unsigned long long)ngrp * blockDim.x : blockDim.x;
    for (unsigned long long e = e0; e < n; e += es) {
      if (!heads && pend[e] != 1) continue;
      const long long c = (long long)list[e];
      int i, k;
      const long long pc = carry_pred(G, c, i, k);  // -1 only for the first cell, a head
      if (pc >= 0 && A.cflag[pc]) {  // predecessor not resolved yet
        if (heads) pend[e] = 1;
        else s_left = 1;
        continue;
      }
      carry_cell<IW, MK>(G, A, c, i, k, pc >= 0 ? A.wgout[pc] : 0.0);
      pend[e] = 2;
      if (!heads) s_progress = 1;
    }
    if (heads && ngrp > 1) {
      unsigned long long* done = A.carry + 1 + A.carry_cap;
      __threadfence();  // each thread's results visible on the device before the count
      __syncthreads();
      if (threadIdx.x == 0) s_last = atomicAdd(done, 1ULL) == (unsigned long long)(ngrp - 1);
      __syncthreads();
      if (!s_last) return;
      __threadfence();  // every workgroup's results before the links are read
    }
    __syncthreads();
    if (heads && threadIdx.x == 0 && A.carry[0] > (unsigned long long)A.carry_cap) atomicAdd(&A.cnt[C_GUARD], 1ULL);
    for (unsigned long long e = threadIdx.x; e < n; e += blockDim.x)
      if (pend[e] == 2) { pend[e] = 0; A.cflag[list[e]] = 0; }
    __syncthreads();
    if (heads) continue;
    const bool stop = !s_left || !s_progress;  // no progress: nothing can resolve further
    __syncthreads();                            // all have read before the next reset
    if (stop) break;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    A.carry[0] = 0;
    if (ngrp > 1) A.carry[1 + A.carry_cap] = 0;
  }
}

// Set-up tables of an axisymmetric metric (metric 303 or 1) on the device,
// one thread per (i,k): the metric at centres, i-, j- and k-faces (j-face =
// centre, coord.f90:116,121) with sqrt(-g), and the Christoffel symbols.
// tr holds per k the host's sin/cos of the folded theta (clamped): at
// x3(k), x3(k)+1e-5, x3(k)-1e-5 and x3a(k); everything else is arithmetic,
// so the tables equal the host set-up's bit for bit.  *sym is cleared where
// Gamma^l_{ab} != Gamma^l_{ba} (the caller sets it to 1 first).
__global__ void __launch_bounds__(256) k_metric_tables(int ni, int nk, int metric, double akm,
                                                       const double* __restrict__ x1, const double* __restrict__ x1a,
                                                       const double* __restrict__ x3, double ph,
                                                       const double* __restrict__ tr, double* met0, double* met1,
                                                       double* met2, double* met3, double* chr, int* sym) {
  const long long P2 = (long long)ni * nk;
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= P2) return;
  const int i = (int)(q % ni), k = (int)(q / ni);
  const double* T = tr + 8LL * k;
  const double r = x1[i];
  double g[16], h[16];
  auto put = [&](double* met) {
    for (int e = 0; e < 16; e++) { met[e * P2 + q] = g[e]; met[(16 + e) * P2 + q] = h[e]; }
    met[32 * P2 + q] = rhmet::detg(g);
  };
  rhmet::cov(metric, akm, g, r, T[0], T[1]);
  rhmet::con(metric, akm, h, r, T[0], T[1]);
  put(met0);
  put(met2);
  rhmet::cov(metric, akm, g, x1a[i], T[0], T[1]);
  rhmet::con(metric, akm, h, x1a[i], T[0], T[1]);
  put(met1);
  rhmet::cov(metric, akm, g, r, T[6], T[7]);
  rhmet::con(metric, akm, h, r, T[6], T[7]);
  put(met3);
  const rhmet::ThetaTrig tt{T[0], T[1], T[2], T[3], T[4], T[5]};
  double ch[64];
  rhmet::christoffel(metric, akm, r, x3[k], ph, tt, ch);
  bool s = true;
  for (int e = 0; e < 64; e++) chr[e * P2 + q] = ch[e];
  for (int l = 0; l < 4; l++)
    for (int a = 0; a < 4; a++)
      for (int b = a + 1; b < 4; b++)
        s = s && __double_as_longlong(ch[l + 4 * a + 16 * b]) == __double_as_longlong(ch[l + 4 * b + 16 * a]);
  if (!s) atomicAnd(sym, 0);
}

// Compact tables (MetK) of the four locations from the general ones, in
// double and, for the three faces, in float (the derived values formed in
// float from float-rounded entries, as the mixed form forms them), one
// thread per location (blockIdx.y) and (i,k).  *ok is cleared where the metric does not have the
// structure the compact form assumes (the caller sets it to 1 first).
template <class R>
RH_DEV void put_compact(const double* met, long long P2, long long q, R* out, bool centre) {
  const MetG<R> M(met, P2, q);
  auto put = [&](int pl, R v) { out[(long long)pl * P2 + q] = v; };
  put(MK_G00, M.g(0, 0)); put(MK_G01, M.g(0, 1)); put(MK_G02, M.g(0, 2));
  put(MK_G11, M.g(1, 1)); put(MK_G12, M.g(1, 2)); put(MK_G22, M.g(2, 2)); put(MK_G33, M.g(3, 3));
  put(MK_DETG, M.detg()); put(MK_ALPHA, M.alpha()); put(MK_RALPHA, M.ralpha()); put(MK_BETA1, M.beta(1));
  put(MK_GI3_1, M.gi3(1)); put(MK_GI3_2, M.gi3(2)); put(MK_GI3_3, M.gi3(3));
  if (centre) {
    put(MK_GI00, M.gi(0, 0)); put(MK_GI01, M.gi(0, 1)); put(MK_GI11, M.gi(1, 1));
    put(MK_GI12, M.gi(1, 2)); put(MK_GI22, M.gi(2, 2)); put(MK_GI33, M.gi(3, 3));
  }
}

__global__ void __launch_bounds__(256) k_compact_metric(CompactArgs A, long long P2, int* ok) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= P2) return;
  const int a = blockIdx.y;
  const double* met = A.met[a];
  auto bits = [&](int e) { return __double_as_longlong(met[(long long)e * P2 + q]); };
  bool fine = true;
  for (int h = 0; h < 2; h++)
    for (int m = 0; m < 4; m++)
      for (int n = m + 1; n < 4; n++) {
        fine = fine && bits(16 * h + m + 4 * n) == bits(16 * h + n + 4 * m);
        if (n == 3 || (h == 1 && m == 0 && n == 2)) fine = fine && bits(16 * h + m + 4 * n) == 0;
      }
  put_compact<double>(met, P2, q, A.mk[a], a == 0);
  if (a > 0) put_compact<float>(met, P2, q, A.mkf[a - 1], false);
  if (!fine) atomicAnd(ok, 0);
}

hipError_t launch_compact_metric(const CompactArgs& A, long long P2, int* ok, hipStream_t st) {
  if (P2 <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_compact_metric, dim3((unsigned)((P2 + 255) / 256), 4), dim3(256), 0, st, A, P2, ok);
  return hipGetLastError();
}

hipError_t launch_metric_tables(int ni, int nk, int metric, double akm, const double* x1, const double* x1a,
                                const double* x3, double ph, const double* tr, double* const met[4], double* chr,
                                int* sym, hipStream_t st) {
  const long long P2 = (long long)ni * nk;
  if (P2 <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_metric_tables, dim3((unsigned)((P2 + 255) / 256)), dim3(256), 0, st, ni, nk, metric, akm, x1,
                     x1a, x3, ph, tr, met[0], met[1], met[2], met[3], chr, sym);
  return hipGetLastError();
}

// caluu1 (caluu.f90:2-126) on every cell: conserved variables from primitives.
template <bool MK>
__global__ void __launch_bounds__(256) k_caluu1(Geo G, const double* __restrict__ W, const void* __restrict__ metC,
                                                double gam, double* __restrict__ U) {
  const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
  int i, j, k;
  if (!box_index(t, 1, G.ni, jlo(G, 1), jhi(G, G.nj), 1, G.nk, i, j, k)) return;
  const long long N = G.N;
  const unsigned c = cidx(i, j, k, G);
  const MetOf<MK, double> M(metC, G.P2, q2(i, k, G));
  double w[9], u[9];
#pragma unroll
  for (int n = 0; n < 9; n++) w[n] = ld_(W + (long long)n * N, c * 8u);
  Prel s;
  prelude(w, gam, M, s);
  tmunu_row(s, 0, M.detg(), pow(s.de, gam), u);
#pragma unroll
  for (int n = 0; n < 9; n++) st_(U + (long long)n * N, c * 8u, u[n]);
}

// ------------------------------------------------------------------------
// Layout conversion between the reference's (n,i,j,k) arrays and planes.
// ------------------------------------------------------------------------
__global__ void k_aos_to_soa(const double* __restrict__ aos, double* __restrict__ soa, long long N) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= N * 9) return;
  const long long c = t / 9, n = t % 9;
  soa[n * N + c] = aos[t];
}
__global__ void k_soa_to_aos(const double* __restrict__ soa, double* __restrict__ aos, long long N) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= N * 9) return;
  const long long c = t / 9, n = t % 9;
  aos[t] = soa[n * N + c];
}

// ww(3,9,i,j,k) of the reference (d fastest, then n) <-> planes d*9+n.
__global__ void k_ww_to_planes(const double* __restrict__ ww, double* __restrict__ F, long long N) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= N) return;
#pragma unroll
  for (int d = 0; d < 3; d++)
#pragma unroll
    for (int n = 0; n < 9; n++) F[(long long)(d * 9 + n) * N + t] = ww[27 * t + d + 3 * n];
}
// the stored flux planes between the two precision forms
template <class S, class T>
__global__ void k_retype(const S* __restrict__ src, T* __restrict__ dst, long long n) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) dst[t] = T(src[t]);
}
__global__ void k_planes_to_ww(const double* __restrict__ F, double* __restrict__ ww, long long N) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= N) return;
#pragma unroll
  for (int d = 0; d < 3; d++)
#pragma unroll
    for (int n = 0; n < 9; n++) ww[27 * t + d + 3 * n] = F[(long long)(d * 9 + n) * N + t];
}

// ------------------------------------------------------------------------
// Kernels: one model per launch (the workgroups renumbered per XCD where the
// stencil benefits), and the batched twins, where one launch covers the same
// step of many models.  A batched launch reads a table of BatchItem (the
// model's Geo, its arguments, and the first workgroup of its part of the
// grid); each workgroup finds its model by binary search and runs the same
// body with its index inside that model's part.
// ------------------------------------------------------------------------
RH_DEV int batch_find(const BatchItem* __restrict__ it, int n, long long b) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (it[mid].off <= b) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

RH_DEV void b_copy(const CopyArgs& A, unsigned blk) {
  const long long t = (long long)blk * blockDim.x + threadIdx.x;
  if (t < A.n) A.dst[t] = A.src[t];
}

template <int D, class R>
__global__ void __launch_bounds__(256) k_ppm_edges(Geo G, EdgeArgs A) { b_ppm_edges<D, R>(G, A, xcd_block()); }
// the PPM and MC sweeps fit 3 waves per SIMD in FP64 (168 VGPRs) and 5 in
// float (96); MP5 and WENO5 are left to the compiler
template <class R, int IREC>
constexpr int sweep_waves = (IREC == 5 || IREC == 1) ? (sizeof(R) == 4 ? 5 : 3) : 1;
template <int D, int IREC, class R, int ICHA, bool MK>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sweep_waves<R, IREC>)))
k_sweep(Geo G, SweepArgs A) { b_sweep<D, IREC, R, ICHA, MK>(G, A, xcd_block()); }
template <int D, class R, int ICHA, bool MK>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sweep_waves<R, 5>)))
k_psweep(Geo G, PSweepArgs A) { b_psweep<D, R, ICHA, MK>(G, A, xcd_block()); }
// The three sweeps of a stage, and in a step's first stage the CFL reduction
// of the same primitives, in one launch: none reads what another writes.
// COLL: a collapsed model's j sweep.
// Each part starts at a multiple of 8 workgroups (a batch member's does too)
// and is renumbered per XCD by itself.  Against a launch each (and three of
// the CFL reduction's): 64x64 and 128x128 torus 116 -> 78 and 125 -> 84 us a
// step, 64^3 443 -> 371, 96x64x64 593 -> 521, 256x128x128 5880 -> 5800 us;
// without the renumbering 6010 us.
template <class R, int ICHA, bool MK, bool COLL>
RH_DEV void b_psweep3(const Geo& G, const PSweep3Args& A, unsigned blk) {
  auto part = [&](int d, unsigned& b) {
    b = blk - (d ? A.end[d - 1] : 0u);
    if (b >= A.n[d]) return false;  // the filling up to a multiple of 8
    b = xcd_renumber(A.n[d], b);
    return true;
  };
  unsigned b;
  if (blk < A.end[0]) { if (part(0, b)) b_psweep<1, R, ICHA, MK>(G, A.s[0], b); }
  else if (blk < A.end[1]) { if (part(1, b)) b_psweep<COLL ? 0 : 2, R, ICHA, MK>(G, A.s[1], b); }
  else if (blk < A.end[2]) { if (part(2, b)) b_psweep<3, R, ICHA, MK>(G, A.s[2], b); }
  else if (blk - A.end[2] < (unsigned)A.cfl.nblocks) b_cfl<ICHA, MK>(G, A.cfl, blk - A.end[2]);
}
// The same for the other reconstructions (a model alone, compact metric tables).
template <int IREC, class R, int ICHA>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sweep_waves<R, IREC>)))
k_sweep3(Geo G, Sweep3Args A) {
  const unsigned part = blockIdx.x / A.each, b = blockIdx.x - part * A.each;
  if (part >= 3) {
    b_cfl<ICHA, true>(G, A.cfl, blockIdx.x - 3 * A.each);
    return;
  }
  if (b >= A.n) return;
  const unsigned blk = xcd_renumber(A.n, b);
  if (part == 0) b_sweep<1, IREC, R, ICHA, true>(G, A.s[0], blk);
  else if (part == 1) b_sweep<2, IREC, R, ICHA, true>(G, A.s[1], blk);
  else b_sweep<3, IREC, R, ICHA, true>(G, A.s[2], blk);
}
template <class R, int ICHA, bool MK, bool COLL>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sweep_waves<R, 5>)))
k_psweep3(Geo G, PSweep3Args A) { b_psweep3<R, ICHA, MK, COLL>(G, A, blockIdx.x); }
template <class FT>
__global__ void __launch_bounds__(256) k_fluxct(Geo G, CtArgs A) { b_fluxct<FT>(G, A, xcd_block()); }
template <int STAGE, bool SYM, class FT, bool MK>
__global__ void __launch_bounds__(256) k_rk(Geo G, StageArgs A) { b_rk<STAGE, SYM, FT, MK>(G, A, xcd_block()); }
template <int STAGE, class FT, int IW>
__global__ void __launch_bounds__(256) k_rkrecov(Geo G, StageArgs A) { b_rkrecov<STAGE, FT, IW>(G, A, xcd_block()); }
template <int IW, bool MK>
__global__ void __launch_bounds__(256) k_recov(Geo G, StageArgs A) { b_recov<IW, MK>(G, A, xcd_block()); }
template <int IW, bool MK>
__global__ void __launch_bounds__(1024) k_recov_carry(Geo G, FixArgs A) {
  b_recov_carry<IW, MK>(G, A, blockIdx.x, gridDim.x);
}
__global__ void __launch_bounds__(256) k_bnd(Geo G, PostArgs A) { b_bnd(G, A, blockIdx.x); }
template <bool MK>
__global__ void __launch_bounds__(256) k_post(Geo G, PostArgs A) { b_post<MK>(G, A, xcd_block()); }
template <int ICHA, bool MK>
__global__ void __launch_bounds__(256) k_cfl(Geo G, CflArgs A) { b_cfl<ICHA, MK>(G, A, blockIdx.x); }
__global__ void __launch_bounds__(256) k_cfl_finish(CflArgs A) { b_cfl_finish(A); }

// batched twins: BODY(G, A, blk) for the model that owns workgroup blockIdx.x
#define RH_BATCH_PROLOGUE                                  \
  const int q = batch_find(it, n, (long long)blockIdx.x);  \
  const Geo G = it[q].G;                                   \
  const unsigned blk = blockIdx.x - (unsigned)it[q].off;
template <int D, class R>
__global__ void __launch_bounds__(256) kb_ppm_edges(const BatchItem* __restrict__ it, int n) {
  RH_BATCH_PROLOGUE
  const EdgeArgs A = it[q].A.e;
  b_ppm_edges<D, R>(G, A, blk);
}
template <int D, int IREC, class R, int ICHA, bool MK>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sweep_waves<R, IREC>)))
kb_sweep(const BatchItem* __restrict__ it, int n) {
  RH_BATCH_PROLOGUE
  const SweepArgs A = it[q].A.s;
  b_sweep<D, IREC, R, ICHA, MK>(G, A, blk);
}
template <class R, int ICHA, bool MK, bool COLL>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sweep_waves<R, 5>)))
kb_psweep3(const BatchItem* __restrict__ it, int n) {
  RH_BATCH_PROLOGUE
  const PSweep3Args A = it[q].A.ps3;
  b_psweep3<R, ICHA, MK, COLL>(G, A, blk);
}
template <class FT>
__global__ void __launch_bounds__(256) kb_fluxct(const BatchItem* __restrict__ it, int n) {
  RH_BATCH_PROLOGUE
  const CtArgs A = it[q].A.c;
  b_fluxct<FT>(G, A, blk);
}
template <int STAGE, bool SYM, class FT, bool MK>
__global__ void __launch_bounds__(256) kb_rk(const BatchItem* __restrict__ it, int n) {
  RH_BATCH_PROLOGUE
  const StageArgs A = it[q].A.st;
  b_rk<STAGE, SYM, FT, MK>(G, A, blk);
}
template <int STAGE, class FT, int IW>
__global__ void __launch_bounds__(256) kb_rkrecov(const BatchItem* __restrict__ it, int n) {
  RH_BATCH_PROLOGUE
  const StageArgs A = it[q].A.st;
  b_rkrecov<STAGE, FT, IW>(G, A, blk);
}
template <int IW, bool MK>
__global__ void __launch_bounds__(256) kb_recov(const BatchItem* __restrict__ it, int n) {
  RH_BATCH_PROLOGUE
  const StageArgs A = it[q].A.st;
  b_recov<IW, MK>(G, A, blk);
}
__global__ void __launch_bounds__(256) kb_bnd(const BatchItem* __restrict__ it, int n) {
  RH_BATCH_PROLOGUE
  const PostArgs A = it[q].A.p;
  b_bnd(G, A, blk);
}
template <bool MK>
__global__ void __launch_bounds__(256) kb_post(const BatchItem* __restrict__ it, int n) {
  RH_BATCH_PROLOGUE
  const PostArgs A = it[q].A.p;
  b_post<MK>(G, A, blk);
}
template <int ICHA, bool MK>
__global__ void __launch_bounds__(256) kb_cfl(const BatchItem* __restrict__ it, int n) {
  RH_BATCH_PROLOGUE
  const CflArgs A = it[q].A.cf;
  b_cfl<ICHA, MK>(G, A, blk);
}
__global__ void __launch_bounds__(256) kb_copy(const BatchItem* __restrict__ it, int n) {
  RH_BATCH_PROLOGUE
  (void)G;
  const CopyArgs A = it[q].A.cp;
  b_copy(A, blk);
}
#undef RH_BATCH_PROLOGUE
// one workgroup per model
template <int IW, bool MK>
__global__ void __launch_bounds__(1024) kb_recov_carry(const BatchItem* __restrict__ it, int n) {
  if ((int)blockIdx.x >= n) return;
  const Geo G = it[blockIdx.x].G;
  const FixArgs A = it[blockIdx.x].A.fx;
  b_recov_carry<IW, MK>(G, A, 0, 1);
}

__global__ void __launch_bounds__(256) kb_cfl_finish(const BatchItem* __restrict__ it, int n) {
  if ((int)blockIdx.x >= n) return;
  const CflArgs A = it[blockIdx.x].A.cf;
  b_cfl_finish(A);
}

// ------------------------------------------------------------------------
// Launch helpers (host side).  While a recorder is set, each helper appends
// the launch it would make (kind, template variant, workgroups, arguments)
// instead of launching; the batch executor merges the records of many models.
// ------------------------------------------------------------------------
static inline unsigned nblk(long long n, int b) { return (unsigned)((n + b - 1) / b); }
static inline long long box(int lo, int hi) { return hi >= lo ? (long long)(hi - lo + 1) : 0; }
// rows of a box along j: one for a collapsed model (its stored row lies in every box)
static inline long long jbox(const Geo& G, int lo, int hi) { return G.jfix ? 1 : box(lo, hi); }

static thread_local std::vector<LaunchRec>* g_rec = nullptr;

void set_recorder(std::vector<LaunchRec>* r) { g_rec = r; }

static void record(int kind, int variant, int threads, long long nb, const Geo& G, const AnyArgs& A) {
  LaunchRec r;
  r.kind = kind; r.variant = variant; r.threads = threads; r.nb = nb; r.G = G; r.A = A;
  g_rec->push_back(r);
}

bool one_group_per_model(int kind) { return kind == LK_CARRY || kind == LK_CFL_FINISH; }

hipError_t launch_edges(const Geo& G, int dir, const double* W, const double* dxs, const double* xs,
                        const double* pc, double gam, void* E, bool mixed, hipStream_t st) {
  const long long ci = box(G.nm0, G.ni - G.nm0 + (dir == 1));
  // along j and k: whole 64-lane rows (box_index_wave)
  const long long ciw = dir != 1 ? 64 * ((ci + 63) / 64) : ci;
  const long long n = ciw * jbox(G, G.nm0, G.nj - G.nm0 + (dir == 2)) * box(G.nm0, G.nk - G.nm0 + (dir == 3));
  EdgeArgs A{W, dxs, xs, pc, gam, E};
  const int bt = slot_threads(G, TS_EDGES);
  const unsigned nb = nblk(n, bt);
  if (g_rec) {
    AnyArgs a{};
    a.e = A;
    record(LK_EDGES, dir + 4 * (int)mixed, bt, nb, G, a);
    return hipSuccess;
  }
  if (n == 0) return hipSuccess;
#define L(Dd, T) hipLaunchKernelGGL((k_ppm_edges<Dd, T>), dim3(nb), dim3(bt), 0, st, G, A)
#define LD(T) do { if (dir == 1) L(1, T); else if (dir == 2) L(2, T); else L(3, T); } while (0)
  if (mixed) LD(float); else LD(double);
#undef LD
#undef L
  return hipGetLastError();
}

// Whether a stage's sweeps share a launch where nothing keeps them apart.
static bool sweeps_share(const Geo& G, int irec) { return irec == 5 ? !G.ppm_split : G.mk != 0; }

bool sweeps_one_launch(const Geo& G, int irec) { return sweeps_share(G, irec) && (irec == 5 || !g_rec); }

int sweep_threads(const Geo& G, int irec, int dir) {
  return slot_threads(G, sweeps_share(G, irec) ? TS_SWEEP1 : TS_SWEEP1 + dir - 1);
}

void record_no_edges(const Geo& G) {
  if (g_rec) record(LK_EDGES, 0, 256, 0, G, AnyArgs{});
}

// Sweep kernels are instantiated per (direction, reconstruction, arithmetic
// type, wave-speed formula); the variant number packs the four so that batch
// plans group launches of the same kernel:
//   dir + 4*mixed + 8*irec + 64*icha + 256*compact (metric tables).
template <int V> using IC = std::integral_constant<int, V>;
template <class T> struct TypeTag { using type = T; };

static int sweep_variant(int dir, bool mixed, int irec, const Geo& G) {
  return dir + 4 * (int)mixed + 8 * irec + 64 * G.icha + 256 * G.mk;
}

// f(compact metric tables?)
template <class F>
static void with_mk(bool mk, F&& f) {
  if (mk) f(std::true_type{});
  else f(std::false_type{});
}

// f(wave-speed formula, compact metric tables?)
template <class F>
static void with_icha(int icha, bool mk, F&& f) {
  with_mk(mk, [&](auto K) {
    if (icha == 2) f(IC<2>{}, K);
    else if (icha == 1) f(IC<1>{}, K);
    else f(IC<0>{}, K);
  });
}

// f(primitive recovery, compact metric tables?) for a variant iwvec + 4*compact
template <class F>
static void with_recov(int variant, F&& f) {
  with_mk((variant & 4) != 0, [&](auto K) {
    if ((variant & 3) == 2) f(IC<2>{}, K);
    else f(IC<1>{}, K);
  });
}

// f(stage, symmetric Christoffel tables?, stored flux type, compact metric
// tables?) for a variant stage + 8*sym + 16*float + 32*compact
template <class F>
static void with_rk(int variant, F&& f) {
  with_mk((variant & 32) != 0, [&](auto K) {
    with_mk((variant & 8) != 0, [&](auto Y) {
      auto t = [&](auto S) {
        if (variant & 16) f(S, Y, TypeTag<float>{}, K);
        else f(S, Y, TypeTag<double>{}, K);
      };
      switch (variant & 7) {
        case 1: t(IC<1>{}); break;
        case 2: t(IC<2>{}); break;
        case 3: t(IC<3>{}); break;
        default: t(IC<4>{}); break;
      }
    });
  });
}

template <class F>
static void with_sweep(int variant, F&& f) {
  const int d = variant & 3, irec = (variant >> 3) & 7;
  const bool mx = (variant & 4) != 0;
  with_icha((variant >> 6) & 3, (variant & 256) != 0, [&](auto C, auto K) {
    auto t = [&](auto D, auto I) {
      if (mx) f(D, I, TypeTag<float>{}, C, K);
      else f(D, I, TypeTag<double>{}, C, K);
    };
    auto r = [&](auto I) {
      if (d == 1) t(IC<1>{}, I);
      else if (d == 2) t(IC<2>{}, I);
      else t(IC<3>{}, I);
    };
    if (irec == 5) r(IC<5>{});
    else if (irec == 1) r(IC<1>{});
    else if (irec == 6) r(IC<6>{});
    else r(IC<7>{});
  });
}

hipError_t launch_sweep(const Geo& G, int dir, int irec, const SweepArgs& A, bool mixed, hipStream_t st) {
  const long long n = box(G.nm0, G.ni - G.nm0) * jbox(G, G.nm0, G.nj - G.nm0) * box(G.nm0, G.nk - G.nm0);
  const int bt = sweep_threads(G, irec, dir);
  const unsigned nb = nblk(n, bt);
  if (g_rec) {
    AnyArgs a{};
    a.s = A;
    record(LK_SWEEP, sweep_variant(dir, mixed, irec, G), bt, nb, G, a);
    return hipSuccess;
  }
  if (n == 0) return hipSuccess;
  with_sweep(sweep_variant(dir, mixed, irec, G), [&](auto D, auto I, auto T, auto C, auto K) {
    hipLaunchKernelGGL((k_sweep<D.value, I.value, typename decltype(T)::type, C.value, K.value>), dim3(nb), dim3(bt), 0, st,
                       G, A);
  });
  return hipGetLastError();
}

// Fused PPM sweeps: variant as the sweeps' without irec, dir 0
// the j sweep of a collapsed model.
static int psweep_variant(int dir, bool mixed, const Geo& G) { return sweep_variant(dir, mixed, 0, G); }

template <class F>
static void with_psweep(int variant, F&& f) {
  const int d = variant & 3;
  const bool mx = (variant & 4) != 0;
  with_icha((variant >> 6) & 3, (variant & 256) != 0, [&](auto C, auto K) {
    auto t = [&](auto D) {
      if (mx) f(D, TypeTag<float>{}, C, K);
      else f(D, TypeTag<double>{}, C, K);
    };
    if (d == 0) t(IC<0>{});
    else if (d == 1) t(IC<1>{});
    else if (d == 2) t(IC<2>{});
    else t(IC<3>{});
  });
}

// Interfaces of a fused PPM sweep along dir and the lines across it (D = 1:
// rows; D = 2, 3: the i of one transverse index, and those indices).
static void psweep_extent(const Geo& G, int dir, long long& along, long long& lines, long long& across) {
  const long long ni = box(G.nm0, G.ni - G.nm0), nj = jbox(G, G.nm0, G.nj - G.nm0), nk = box(G.nm0, G.nk - G.nm0);
  along = dir == 1 ? ni : dir == 2 ? nj : nk;
  lines = dir == 1 ? nj * nk : ni;
  across = dir == 1 ? 1 : dir == 2 ? nk : nj;
}

// Tile of a fused PPM sweep along dir in workgroups of bt threads: tp cells
// along the axis (3 of them overlap the next tile) by bt / tp lines.
//  D = 1: the whole workgroup along the row, or 16, 32 or 64 cells of several
//  rows, whichever leaves the fewest idle or overlapping lanes.
//  D = 2, 3: a wave holds w cells along the axis by 64 / w consecutive i and
//  the workgroup's waves are stacked along the axis.  As set by the caller
//  (Geo::seg, the tile's cells), else along j the w with the fewest such lanes
//  among 2 to 16, and along k 4, or 8 where that has fewer and still two waves
//  per SIMD (1024 of them): along j a tile's cells share their face metric,
//  along k every (i, k) has its own, read in runs of 64 / w (w 4, 8, 16:
//  256x128x128 0.373, 0.406, 0.370 ms, mixed 0.202, 0.242, 0.250; 64^3, fewer
//  lanes at 8, 28.0, 25.7, 26.1 us; 251x57x77 89, 90, 119 us; one 64x64 row,
//  with half the workgroups at 8, 12.4, 16.7, 13.4 us).  Never below a tile of
//  8 cells, 5 interfaces (64 threads, with a k tile of 4 and one interface:
//  one 128x128 row 76.7 -> 71.8 us a step, 40x24x40 146.7 -> 136.3), unless
//  the axis needs no more (Riemann tubes' four transverse interfaces), and
//  never below the 4 that give an interface.
static int psweep_tp(const Geo& G, int dir, int bt) {
  long long along, lines, across;
  psweep_extent(G, dir, along, lines, across);
  auto lanes = [&](long long tp, long long ti) {
    return ((along + tp - 4) / (tp - 3)) * tp * ((lines + ti - 1) / ti) * ti;
  };
  if (dir == 1) {
    int best = bt;
    for (int tp : {64, 32, 16})
      if (tp < bt && lanes(tp, bt / tp) < lanes(best, bt / best)) best = tp;
    return best;
  }
  const int nw = bt / 64, want = G.seg[dir - 2];
  int w;
  if (want) {  // the tallest tile no taller than that
    for (w = 1; 2 * w * nw <= want;) w *= 2;
  } else if (dir == 2) {
    w = 16;
    for (int q : {8, 4, 2})
      if (q * nw >= 8 && lanes(q * nw, 64 / q) < lanes(w * nw, 64 / w)) w = q;
  } else {
    const long long l4 = lanes(4 * nw, 16), l8 = lanes(8 * nw, 8);
    w = nw == 1 || (l8 < l4 && l8 * across >= 2 * 64 * 1024) ? 8 : 4;
  }
  while (w > 1 && w * nw / 2 >= 4 && w * nw / 2 - 3 >= along) w /= 2;
  while (w * nw < 4) w *= 2;
  return w * nw;
}

// The sweep's tile along j or k as a size that can be asked for: its cells, a
// power of two (three waves make tiles of three quarters of one).
int psweep_segment(const Geo& G, int dir) {
  const int tp = psweep_tp(G, dir, slot_threads(G, TS_SWEEP1));  // fused sweeps share a launch
  int seg = 4;
  while (seg < tp) seg *= 2;
  return seg;
}

// Whether the axis fills three quarters of a tile of seg cells along dir.
bool psweep_fills(const Geo& G, int dir, int seg) {
  long long along, lines, across;
  psweep_extent(G, dir, along, lines, across);
  return 4 * along >= 3 * (seg - 3);
}

size_t psweep_lds_bytes(int threads, bool mixed) { return (size_t)18 * threads * (mixed ? sizeof(float) : sizeof(double)); }

static long long cfl_cells(const Geo& G) {
  return box(2, G.ni - 1) * jbox(G, 2, G.nj - 1) * box(2, G.nk - 1);
}

long long cfl_blocks(const Geo& G) {
  const long long n = cfl_cells(G);
  return n > 0 ? (long long)nblk(n, 256) : 1;
}

long long cfl_slots(const Geo& G) { return std::min<long long>(CFL_GROUPS, std::max(1LL, (cfl_cells(G) + 63) / 64)); }

// Workgroups of bt threads of the CFL reduction (set in A with their cells):
// bt cells each, or more so that there are CFL_GROUPS at most, whose results
// one workgroup reads.
static unsigned cfl_groups(const Geo& G, int bt, CflArgs& A) {
  const long long chunks = std::max(1LL, (cfl_cells(G) + bt - 1) / bt), each = (chunks + CFL_GROUPS - 1) / CFL_GROUPS;
  A.nblocks = (int)((chunks + each - 1) / each);
  A.per = (int)(bt * each);
  return (unsigned)A.nblocks;
}

// Arguments and workgroups (of bt threads) of one fused sweep.
static long long psweep_args(const Geo& G, int dir, int bt, PSweepArgs& A) {
  long long along, lines, across;
  psweep_extent(G, dir, along, lines, across);
  if (dir == 2 && G.jfix) return (lines * across + bt - 1) / bt;  // one stored phi row: its own neighbour
  if (along <= 0 || lines <= 0 || across <= 0) return 0;
  A.tp = psweep_tp(G, dir, bt);
  const int ti = bt / A.tp;
  // log2 of the lanes that vary fastest (D = 1 with the whole workgroup on one row: all)
  const int fast = dir == 1 ? A.tp : ti;
  A.sh = dir == 1 && ti == 1 ? 30 : __builtin_ctz((unsigned)fast);
  A.nig = (int)((lines + ti - 1) / ti);
  A.ndc = (int)((along + A.tp - 4) / (A.tp - 3));
  return (long long)A.nig * A.ndc * across;
}

hipError_t launch_psweep(const Geo& G, int dir, const PSweepArgs& A0, bool mixed, hipStream_t st) {
  const int bt = sweep_threads(G, 5, dir);
  const bool self = dir == 2 && G.jfix;
  PSweepArgs A = A0;
  const unsigned nb = (unsigned)psweep_args(G, dir, bt, A);
  const int variant = psweep_variant(self ? 0 : dir, mixed, G);
  if (nb == 0) return hipSuccess;
  const size_t lds = self ? 0 : psweep_lds_bytes(bt, mixed);
  with_psweep(variant, [&](auto D, auto T, auto C, auto K) {
    hipLaunchKernelGGL((k_psweep<D.value, typename decltype(T)::type, C.value, K.value>), dim3(nb), dim3(bt), lds, st,
                       G, A);
  });
  return hipGetLastError();
}

// variant: (collapsed) + 4*mixed + 64*icha + 256*compact
template <class F>
static void with_psweep3(int variant, F&& f) {
  with_icha((variant >> 6) & 3, (variant & 256) != 0, [&](auto C, auto K) {
    with_mk((variant & 1) != 0, [&](auto L) {
      if (variant & 4) f(TypeTag<float>{}, C, K, L);
      else f(TypeTag<double>{}, C, K, L);
    });
  });
}

hipError_t launch_sweep3(const Geo& G, int irec, const SweepArgs s[3], bool mixed, const CflArgs* cfl,
                         hipStream_t st) {
  const long long n = box(G.nm0, G.ni - G.nm0) * jbox(G, G.nm0, G.nj - G.nm0) * box(G.nm0, G.nk - G.nm0);
  const int bt = slot_threads(G, TS_SWEEP1);
  Sweep3Args A{{s[0], s[1], s[2]}, nblk(n, bt), 0, CflArgs{}};
  A.each = (A.n + 7u) & ~7u;
  if (A.n == 0) A.each = 8;
  unsigned nb = 3 * A.each;
  if (cfl) {
    A.cfl = *cfl;
    nb += cfl_groups(G, bt, A.cfl);
  }
  with_icha(G.icha, true, [&](auto C, auto) {
    auto t = [&](auto I) {
      if (mixed) hipLaunchKernelGGL((k_sweep3<I.value, float, C.value>), dim3(nb), dim3(bt), 0, st, G, A);
      else hipLaunchKernelGGL((k_sweep3<I.value, double, C.value>), dim3(nb), dim3(bt), 0, st, G, A);
    };
    if (irec == 1) t(IC<1>{});
    else if (irec == 6) t(IC<6>{});
    else t(IC<7>{});
  });
  return hipGetLastError();
}

hipError_t launch_psweep3(const Geo& G, const PSweepArgs s[3], bool mixed, const CflArgs* cfl, hipStream_t st) {
  const int bt = slot_threads(G, TS_SWEEP1);
  PSweep3Args A{};
  unsigned nb = 0;
  for (int d = 0; d < 3; d++) {
    A.s[d] = s[d];
    A.n[d] = (unsigned)psweep_args(G, d + 1, bt, A.s[d]);
    nb += (A.n[d] + 7u) & ~7u;
    A.end[d] = nb;
  }
  if (cfl) {
    A.cfl = *cfl;
    nb += (cfl_groups(G, bt, A.cfl) + 7u) & ~7u;
  }
  const int variant = psweep_variant(G.jfix ? 1 : 0, mixed, G);
  if (g_rec) {
    AnyArgs a{};
    a.ps3 = A;
    record(LK_PSWEEP3, variant, bt, nb, G, a);
    return hipSuccess;
  }
  if (nb == 0) return hipSuccess;
  with_psweep3(variant, [&](auto T, auto C, auto K, auto L) {
    hipLaunchKernelGGL((k_psweep3<typename decltype(T)::type, C.value, K.value, L.value>), dim3(nb), dim3(bt),
                       psweep_lds_bytes(bt, mixed), st, G, A);
  });
  return hipGetLastError();
}

hipError_t launch_fluxct(const Geo& G, const void* CTsrc, void* F1, void* F2, void* F3, bool f32, double* CTd,
                         const CflArgs* cfl, hipStream_t st) {
  const long long n = box(G.nm1, G.ni - G.nm1) * jbox(G, G.nm1, G.nj - G.nm1) * box(G.nm1, G.nk - G.nm1);
  CtArgs A{CTsrc, F1, F2, F3, f32 ? CTd : nullptr, -1, CflArgs{}};
  const int bt = slot_threads(G, TS_FLUXCT);
  unsigned nb = nblk(n, bt);
  if (cfl) {  // one more workgroup combines the CFL reduction of launch_psweep3
    A.cfl = *cfl;
    (void)cfl_groups(G, slot_threads(G, TS_SWEEP1), A.cfl);
    A.fin = (int)nb++;
  }
  if (g_rec) { AnyArgs a{}; a.c = A; record(LK_FLUXCT, (int)f32, bt, nb, G, a); return hipSuccess; }
  if (nb == 0) return hipSuccess;
  if (f32) hipLaunchKernelGGL(k_fluxct<float>, dim3(nb), dim3(bt), 0, st, G, A);
  else hipLaunchKernelGGL(k_fluxct<double>, dim3(nb), dim3(bt), 0, st, G, A);
  return hipGetLastError();
}

static int rk_variant(const Geo& G, int stage, const StageArgs& A) {
  return stage + 8 * (int)A.chr_sym + 16 * (int)A.f32flux + 32 * G.mk;
}

hipError_t launch_update(const Geo& G, int stage, const StageArgs& A, hipStream_t st) {
  const long long n = box(G.nm1 + 1, G.ni - G.nm1) * jbox(G, G.nm1 + 1, G.nj - G.nm1) * box(G.nm1 + 1, G.nk - G.nm1);
  const int bt = slot_threads(G, TS_RK);
  const unsigned nb = nblk(n, bt);
  const int variant = rk_variant(G, stage, A);
  if (n == 0) return hipSuccess;
  with_rk(variant, [&](auto S, auto Y, auto T, auto K) {
    hipLaunchKernelGGL((k_rk<S.value, Y.value, typename decltype(T)::type, K.value>), dim3(nb), dim3(bt), 0, st, G, A);
  });
  return hipGetLastError();
}

hipError_t launch_recov(const Geo& G, const StageArgs& A, hipStream_t st) {
  const long long n = box(G.nm1 + 1, G.ni - G.nm1) * jbox(G, G.nm1 + 1, G.nj - G.nm1) * box(G.nm1 + 1, G.nk - G.nm1);
  const int bt = slot_threads(G, TS_RECOV);
  if (n == 0) return hipSuccess;
  with_recov(G.iwvec + 4 * G.mk, [&](auto I, auto K) {
    hipLaunchKernelGGL((k_recov<I.value, K.value>), dim3(nblk(n, bt)), dim3(bt), 0, st, G, A);
  });
  return hipGetLastError();
}

// The fused update and recovery for a variant as launch_update's, plus
// 64*(iwvec == 2); false where it is not built (general metric tables or
// Christoffel symbols that are not symmetric).
template <class F>
static bool with_rkrecov(int variant, F&& f) {
  if ((variant & 40) != 40) return false;
  auto t = [&](auto S) {
    auto w = [&](auto T) {
      if (variant & 64) f(S, T, IC<2>{});
      else f(S, T, IC<1>{});
    };
    if (variant & 16) w(TypeTag<float>{});
    else w(TypeTag<double>{});
  };
  switch (variant & 7) {
    case 1: t(IC<1>{}); break;
    case 2: t(IC<2>{}); break;
    case 3: t(IC<3>{}); break;
    default: t(IC<4>{}); break;
  }
  return true;
}

bool update_recov_one_launch(const Geo& G, bool chr_sym) { return (G.mk && chr_sym) || g_rec; }

hipError_t launch_update_recov(const Geo& G, int stage, const StageArgs& A, hipStream_t st) {
  const long long n = box(G.nm1 + 1, G.ni - G.nm1) * jbox(G, G.nm1 + 1, G.nj - G.nm1) * box(G.nm1 + 1, G.nk - G.nm1);
  const int bt = slot_threads(G, TS_RK);
  const unsigned nb = nblk(n, bt);
  const int variant = rk_variant(G, stage, A) + 64 * (G.iwvec == 2);
  if (g_rec) { AnyArgs a{}; a.st = A; record(LK_RKRECOV, variant, bt, nb, G, a); return hipSuccess; }
  if (n == 0) return hipSuccess;
  const bool built = with_rkrecov(variant, [&](auto S, auto T, auto I) {
    hipLaunchKernelGGL((k_rkrecov<S.value, typename decltype(T)::type, I.value>), dim3(nb), dim3(bt), 0, st, G, A);
  });
  return built ? hipGetLastError() : hipErrorInvalidValue;
}

hipError_t launch_recov_carry(const Geo& G, const FixArgs& A, hipStream_t st) {
  if (g_rec) { AnyArgs a{}; a.fx = A; record(LK_CARRY, G.iwvec + 4 * G.mk, 1024, 1, G, a); return hipSuccess; }
  // workgroups sharing the chain heads: one per 1024 flaggable cells, at most 64
  const int ng = (int)std::min<long long>(64, std::max<long long>(1, (A.carry_cap + 1023) / 1024));
  with_recov(G.iwvec + 4 * G.mk, [&](auto I, auto K) {
    hipLaunchKernelGGL((k_recov_carry<I.value, K.value>), dim3(ng), dim3(1024), 0, st, G, A);
  });
  return hipGetLastError();
}

hipError_t launch_post(const Geo& G, const PostArgs& A0, hipStream_t st) {
  const long long g = G.nm1;
  const long long ng = G.N - (long long)(G.ni - 2 * g) * (G.jfix ? 1 : G.nj - 2 * g) * (G.nk - 2 * g);
  const int bt = slot_threads(G, TS_POST);
  PostArgs A = A0;
  A.nbc = ng > 0 ? (int)nblk(ng, bt) : 0;
  // one variable a thread while that is at most two waves per SIMD (1024 of them)
  A.nbv = 9 * ng <= 2 * 64 * 1024 ? 1 : 3;
  if (g_rec) {
    AnyArgs a{};
    a.p = A;
    record(LK_BND, 0, bt, (9LL / A.nbv) * A.nbc, G, a);
    record(LK_POST, G.mk, bt, nblk(G.N, bt), G, a);
    return hipSuccess;
  }
  if (ng > 0) hipLaunchKernelGGL(k_bnd, dim3((unsigned)(9 / A.nbv * A.nbc)), dim3(bt), 0, st, G, A);
  with_mk(G.mk, [&](auto K) {
    hipLaunchKernelGGL(k_post<K.value>, dim3(nblk(G.N, bt)), dim3(bt), 0, st, G, A);
  });
  return hipGetLastError();
}

hipError_t launch_sum_counters(unsigned long long* cpart, long long rows, unsigned long long* cnt, hipStream_t st) {
  hipLaunchKernelGGL(k_sum_counters, dim3(1), dim3(1024), 0, st, cpart, rows, cnt);
  return hipGetLastError();
}

hipError_t launch_cfl(const Geo& G, const CflArgs& A0, hipStream_t st) {
  CflArgs A = A0;
  const unsigned nb = cfl_groups(G, 256, A);
  if (g_rec) {
    AnyArgs a{};
    a.cf = A;
    record(LK_CFL, G.icha + 4 * G.mk, 256, nb, G, a);
    record(LK_CFL_FINISH, 0, 256, 1, G, a);
    return hipSuccess;
  }
  with_icha(G.icha, G.mk, [&](auto C, auto K) {
    hipLaunchKernelGGL((k_cfl<C.value, K.value>), dim3(nb), dim3(256), 0, st, G, A);
  });
  hipLaunchKernelGGL(k_cfl_finish, dim3(1), dim3(256), 0, st, A);
  return hipGetLastError();
}

hipError_t launch_copy(const Geo& G, double* dst, const double* src, long long n, hipStream_t st) {
  if (g_rec) {
    AnyArgs a{};
    a.cp = CopyArgs{src, dst, n};
    record(LK_COPY, 0, 256, nblk(n, 256), G, a);
    return hipSuccess;
  }
  return hipMemcpyAsync(dst, src, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, st);
}

hipError_t launch_batched(int kind, int variant, int threads, const BatchItem* it, int n, long long total_blocks,
                          hipStream_t st) {
  if (n <= 0 || total_blocks <= 0) return hipSuccess;
  if (total_blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  if (!one_group_per_model(kind) && (threads < 64 || threads > 256 || threads % 64)) return hipErrorInvalidValue;
  const dim3 g((unsigned)total_blocks), b((unsigned)threads);
  switch (kind) {
    case LK_EDGES: {
      const int d = variant & 3;
#define L(Dd, T) hipLaunchKernelGGL((kb_ppm_edges<Dd, T>), g, b, 0, st, it, n)
#define LD(T) do { if (d == 1) L(1, T); else if (d == 2) L(2, T); else L(3, T); } while (0)
      if (variant & 4) LD(float); else LD(double);
#undef LD
#undef L
      break;
    }
    case LK_SWEEP:
      with_sweep(variant, [&](auto D, auto I, auto T, auto C, auto K) {
        hipLaunchKernelGGL((kb_sweep<D.value, I.value, typename decltype(T)::type, C.value, K.value>), g, b, 0, st, it, n);
      });
      break;
    case LK_PSWEEP3:
      with_psweep3(variant, [&](auto T, auto C, auto K, auto L) {
        hipLaunchKernelGGL((kb_psweep3<typename decltype(T)::type, C.value, K.value, L.value>), g, b,
                           psweep_lds_bytes(threads, (variant & 4) != 0), st, it, n);
      });
      break;
    case LK_FLUXCT:
      if (variant == 1) hipLaunchKernelGGL(kb_fluxct<float>, g, b, 0, st, it, n);
      else hipLaunchKernelGGL(kb_fluxct<double>, g, b, 0, st, it, n);
      break;
    case LK_RKRECOV:
      if (with_rkrecov(variant, [&](auto S, auto T, auto I) {
            hipLaunchKernelGGL((kb_rkrecov<S.value, typename decltype(T)::type, I.value>), g, b, 0, st, it, n);
          }))
        break;
      with_rk(variant & 63, [&](auto S, auto Y, auto T, auto K) {
        hipLaunchKernelGGL((kb_rk<S.value, Y.value, typename decltype(T)::type, K.value>), g, b, 0, st, it, n);
      });
      with_recov(((variant & 64) ? 2 : 1) + ((variant & 32) ? 4 : 0), [&](auto I, auto K) {
        hipLaunchKernelGGL((kb_recov<I.value, K.value>), g, b, 0, st, it, n);
      });
      break;
    case LK_BND: hipLaunchKernelGGL(kb_bnd, g, b, 0, st, it, n); break;
    case LK_POST:
      with_mk(variant != 0, [&](auto K) { hipLaunchKernelGGL(kb_post<K.value>, g, b, 0, st, it, n); });
      break;
    case LK_CFL:
      with_icha(variant & 3, (variant & 4) != 0, [&](auto C, auto K) {
        hipLaunchKernelGGL((kb_cfl<C.value, K.value>), g, b, 0, st, it, n);
      });
      break;
    case LK_COPY: hipLaunchKernelGGL(kb_copy, g, b, 0, st, it, n); break;
    case LK_CFL_FINISH: hipLaunchKernelGGL(kb_cfl_finish, dim3(n), dim3(256), 0, st, it, n); break;
    case LK_CARRY:
      with_recov(variant, [&](auto I, auto K) {
        hipLaunchKernelGGL((kb_recov_carry<I.value, K.value>), dim3(n), dim3(1024), 0, st, it, n);
      });
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

__global__ void k_gather_first(const double* const* __restrict__ src, double* __restrict__ dst, int n) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) dst[t] = src[t][0];
}

hipError_t launch_gather_first(const double* const* src, double* dst, int n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_gather_first, dim3(nblk(n, 256)), dim3(256), 0, st, src, dst, n);
  return hipGetLastError();
}

hipError_t launch_caluu1(const Geo& G, const double* W, const void* metC, double gam, double* U, hipStream_t st) {
  if (G.mk) hipLaunchKernelGGL(k_caluu1<true>, dim3(nblk(G.N, 256)), dim3(256), 0, st, G, W, metC, gam, U);
  else hipLaunchKernelGGL(k_caluu1<false>, dim3(nblk(G.N, 256)), dim3(256), 0, st, G, W, metC, gam, U);
  return hipGetLastError();
}

hipError_t launch_aos_to_soa(const double* aos, double* soa, long long N, hipStream_t st) {
  hipLaunchKernelGGL(k_aos_to_soa, dim3(nblk(N * 9, 256)), dim3(256), 0, st, aos, soa, N);
  return hipGetLastError();
}
hipError_t launch_soa_to_aos(const double* soa, double* aos, long long N, hipStream_t st) {
  hipLaunchKernelGGL(k_soa_to_aos, dim3(nblk(N * 9, 256)), dim3(256), 0, st, soa, aos, N);
  return hipGetLastError();
}

hipError_t launch_ww_to_planes(const double* ww, double* F, long long N, hipStream_t st) {
  if (N == 0) return hipSuccess;
  hipLaunchKernelGGL(k_ww_to_planes, dim3(nblk(N, 256)), dim3(256), 0, st, ww, F, N);
  return hipGetLastError();
}
hipError_t launch_planes_to_ww(const double* F, double* ww, long long N, hipStream_t st) {
  if (N == 0) return hipSuccess;
  hipLaunchKernelGGL(k_planes_to_ww, dim3(nblk(N, 256)), dim3(256), 0, st, F, ww, N);
  return hipGetLastError();
}

hipError_t launch_retype(const void* src, void* dst, long long n, bool to_float, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  if (to_float)
    hipLaunchKernelGGL((k_retype<double, float>), dim3(nblk(n, 256)), dim3(256), 0, st, (const double*)src, (float*)dst, n);
  else
    hipLaunchKernelGGL((k_retype<float, double>), dim3(nblk(n, 256)), dim3(256), 0, st, (const float*)src, (double*)dst, n);
  return hipGetLastError();
}

}  // namespace rh
