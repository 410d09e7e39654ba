// ocfd_hybrid.hip -- the nonlinear faces of the hybrid scheme, gathered.
//
// The hybrid scheme (OCFD_Schemes.f90:319-358, OCFD_SetHybrid.f90:2-15)
// reconstructs most faces with the linear UD7L blend and a few with WENO7 or
// WENO5, chosen per face from the sensor Rhybrid that comput_Rhybrid forms
// once per time step.  Computed inside the sweep tiles, the few WENO faces
// leave most lanes of a tile idle; here they are
//   k_hyb_list    listed once per step, per sweep axis (a range of the
//                 list reserved per workgroup, faces in order inside it),
//                 with a face -> slot map for the sweeps;
//   k_weno_faces  computed densely before each stage's sweeps: batches of 64
//                 listed faces on five wavefronts each, split fluxes of the 8
//                 stencil points in LDS, then one characteristic row -- or
//                 component, without projection -- per wavefront, one face
//                 per lane.
// The sweep kernels read the listed faces' fluxes by slot.  Every flux is the
// same expression as in the sweep (flux_charteric,
// OCFD_inviscous_character.f90:190-290; OCFD2d_flux1/2,
// OCFD_inviscous.f90:210-361), so results are unchanged bit for bit.
#include <algorithm>
#include <type_traits>

#include "ocfd_kernels.h"

namespace ocfd {

namespace {

constexpr int FB = 64;           // listed faces of a batch: one per lane
constexpr int NSUB = 3;          // batches a workgroup works on together
constexpr int WNT = NSUB * 5 * FB;  // per batch a wavefront for each characteristic row / component

// A workgroup lists LPT * NT consecutive faces of the axis: scheme index from
// the sensor, the WENO faces appended to the axis list in face order, and the
// face -> slot map.  The list position is reserved with one atomic per
// workgroup; inside it the slots follow the face index.
constexpr int LPT = 16;  // faces per thread
constexpr int LPB = 8;   // of which the sensor values are loaded together
template <int AXIS>
__device__ __forceinline__ void hyb_list_axis(const Block &B, int (&soff)[LPT][NT / 64], int &sbase, const int64_t blk) {
  typedef TileIndex<AXIS> TI;
  const Geom &g = B.g;
  const SchemeParams &S = B.S;
  const int n = g.n(AXIS);
  const int64_t nfa = TI::nfaces(g);
  const int64_t f0 = blk * (NT * LPT) + threadIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned wbits = 0, hbits = 0;  // bit it: face f0 + it * NT is WENO / WENO7-class
#pragma unroll 1
  for (int i0 = 0; i0 < LPT; i0 += LPB) {
    // the sensor values of LPB faces before the first is looked at
    double ra[LPB], rb[LPB];
    int sv[LPB];
#pragma unroll
    for (int q = 0; q < LPB; q++) {
      const int64_t fid = f0 + (int64_t)(i0 + q) * NT;
      int w, c;
      TI::face_of(g, fid < nfa ? fid : nfa - 1, sv[q], w, c);
      const int64_t h = TI::hidx(g, sv[q], w, c);
      ra[q] = B.rhyb[h];
      rb[q] = B.rhyb[h + g.hstride(AXIS)];
    }
#pragma unroll
    for (int q = 0; q < LPB; q++) {
      const int it = i0 + q, s = sv[q];
      // set_hybrid_scheme: the larger sensor value of the two cells of the face
      const int scm = hybrid_index(dmax2(ra[q], rb[q]), S.hyb2, S.hyb3);
      // the characteristic path closes non-periodic block edges with the
      // non-reflecting face whatever the scheme index
      const bool closure = S.is_char && ((S.bidx[AXIS][0] == 1 && S.sb[2 * AXIS] == 0 && s == 0) ||
                                         (S.bidx[AXIS][1] == 1 && S.sb[2 * AXIS + 1] == 0 && s == n));
      const bool weno = f0 + (int64_t)it * NT < nfa && scm >= 2 && !closure;
      if (weno) wbits |= 1u << it;
      if (scm == 3) hbits |= 1u << it;
      const unsigned long long mask = __ballot(weno);
      if (lane == 0) soff[it][wave] = __popcll(mask);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    for (int it = 0; it < LPT; it++)
      for (int q = 0; q < NT / 64; q++) {
        const int c = soff[it][q];
        soff[it][q] = t;
        t += c;
      }
    sbase = t ? atomicAdd(&B.hcount[AXIS], t) : 0;
  }
  __syncthreads();
  const int base = sbase;
  const unsigned long long below = (1ull << lane) - 1ull;
  for (int it = 0; it < LPT; it++) {
    const int64_t fid = f0 + (int64_t)it * NT;
    const bool weno = (wbits >> it) & 1u;
    const unsigned long long mask = __ballot(weno);
    const int slot = base + soff[it][wave] + __popcll(mask & below);
    // the wavefront's 64 faces are one aligned group of the face map
    if (lane == 0 && fid < nfa) {
      B.hbits[AXIS][fid >> 6] = mask;
      B.hgbase[AXIS][fid >> 6] = base + soff[it][wave];
    }
    if (weno) B.hlist[AXIS][slot] = (int)(fid * 2 + ((hbits >> it) & 1u));
  }
}

// the lists of the three axes: workgroups [0, n0) x, [n0, n0 + n1) y, then z
// (256^3 181 us in three launches with one face's loads at a time, 147 now;
// 101 x 75 x 54 34 and 11)
__global__ __launch_bounds__(NT) void k_hyb_list(const Block B, const unsigned n0, const unsigned n1) {
  __shared__ int soff[LPT][NT / 64];
  __shared__ int sbase;
  if (blockIdx.x < n0) hyb_list_axis<0>(B, soff, sbase, blockIdx.x);
  else if (blockIdx.x < n0 + n1) hyb_list_axis<1>(B, soff, sbase, blockIdx.x - n0);
  else hyb_list_axis<2>(B, soff, sbase, blockIdx.x - n0 - n1);
}

// type the split fluxes are held in: the projections are FP64 in both forms, so
// the mixed form's FP32 fluxes are widened once instead of by all five rows
template <bool CHAR, typename RR>
using weno_lds_t = typename std::conditional<CHAR, double, RR>::type;

// Fluxes of the listed faces of one axis: workgroup wg of nwg strides over
// batches of FB faces; the list length is read from the device counter.  RR is
// the real type of the splitting and the WENO reconstruction: double, or float
// in the mixed-precision form, where the characteristic basis and the
// projections onto and back from it stay FP64.  MET as in the sweeps: 0
// closures and metric fields, 1 periodic axis and uniform metrics, 2 also a
// metric vector along the axis' own coordinate.
//
// Of the five wavefronts of a batch, wavefront r works on row (component) r
// of its 64 faces, so the row is the same for all its lanes: its entries of
// the basis are formed by scalar branches, and with MET 2 the two rows of the
// tangential velocities project two components instead of five.  The split
// fluxes lie [component][point][face]: every LDS access is 64 consecutive
// values.  Wavefront r also splits stencil points r and r + 5.  While a batch
// is projected and reconstructed, the primitives of the next one and the list
// entries of the one after are in flight (two dependent loads, about as long
// as the arithmetic of a batch), and a lane keeps its face's coefficients in
// registers to the end: two barriers per batch.  A workgroup takes three
// batches at once: as workgroups of five wavefronts only two fitted a CU (the
// first SIMD takes two of each five), 2.1 wavefronts per SIMD instead of 3.7,
// which was half of the gain.  Bound by instruction issue (VALU 65% busy).  The
// three axes in the former layout (256 lanes on 51 faces, one lane per row:
// every lane formed all rows' entries, three launches) and now: 256^3 FP64,
// 3.9% of the faces listed, 609 and 406 us; mixed (5.7%) 389 and 275; 160^3
// FP64 with metric fields (10%) 428 and 306; 101 x 75 x 54 mixed (28%) 49 and 38.
template <int AXIS, bool CHAR, int MET, typename RR>
__device__ __forceinline__ void weno_faces_axis(const Block &B, weno_lds_t<CHAR, RR> *const sFa, double *const sQa,
                                                double *const sGa,
                                                const int wg, const int nwg) {
  typedef TileIndex<AXIS> TI;
  constexpr int NH = CHAR ? 5 : 10;
  const Geom &g = B.g;
  const SchemeParams &S = B.S;
  const int n = g.n(AXIS);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = wave / 5, row = wave - 5 * sub;
  weno_lds_t<CHAR, RR> *const sF = sFa + sub * (80 * FB);
  double *const sQ = sQa + sub * (CHAR ? 14 * FB : 0), *const sG = sGa + sub * (CHAR ? 5 * FB : 0);
  const int q1 = M_AKX1 + 3 * AXIS;
  const int count = B.hcount[AXIS];
  const int ngroup = (count + NSUB * FB - 1) / (NSUB * FB);  // groups of NSUB batches
  const int *const list = B.hlist[AXIS];
  RR *const out = reinterpret_cast<RR *>(B.wflux[AXIS]);
  const bool sw = S.flux_split == 1;
  const bool unif = MET != 0 || B.M.uniform != 0;
  // groups in one contiguous range per XCD (workgroup b runs on XCD
  // b % NXCD), strided over that XCD's workgroups: list-neighbouring faces,
  // whose y / z stencils share rows, then meet in the same L2
  const int nw = nwg / NXCD, xcd = wg % NXCD;
  const bool split = nwg % NXCD == 0 && nw > 0;
  const int bhi = split ? (int)((int64_t)ngroup * (xcd + 1) / NXCD) : ngroup;
  const int b0 = split ? (int)((int64_t)ngroup * xcd / NXCD) + wg / NXCD : wg;
  const int bstep = split ? nw : nwg;
  if (b0 >= bhi) return;
  const RR *const P[5] = {B.d.as<RR>(), B.u.as<RR>(), B.v.as<RR>(), B.w.as<RR>(), B.T.as<RR>()};
  // entry of this lane in group bt (past the end: the last one again)
  auto entry = [&](int bt) {
    const int f = (bt * NSUB + sub) * FB + lane;
    return list[f < count ? f : count - 1];
  };
  // stencil points row and row + 5 (< 8) of this lane's face
  RR pv[2][5];
  int sn = 0;        // the fetched face's s, and its first stencil point
  int64_t hn = 0;
  const int64_t st = g.hstride(AXIS);
  auto fetch = [&](int code) {
    int w, c;
    TI::face_of(g, code >> 1, sn, w, c);
    const int64_t h0 = hn = TI::hidx(g, sn - 3, w, c);
#pragma unroll
    for (int r = 0; r < 2; r++)
      if (row + 5 * r < 8) {
        const int64_t h = h0 + (row + 5 * r) * st;
#pragma unroll
        for (int q = 0; q < 5; q++) pv[r][q] = P[q][h];
      }
  };
  int code = entry(b0);
  fetch(code);
  int code1 = entry(b0 + bstep < bhi ? b0 + bstep : b0);
  for (int batch = b0; batch < bhi; batch += bstep) {
    const int s = sn;
    // split fluxes at the stencil points (OCFD_inviscous.f90:64-70, split_*)
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const int p = row + 5 * r;
      if (p >= 8) continue;
      const RR dd = pv[r][0], uu = pv[r][1], vv = pv[r][2], ww = pv[r][3], Tt = pv[r][4];
      SplitK<RR> K = split_const<RR>(B, AXIS);
      double A[3] = {0.0, 0.0, 0.0};
      if (!unif) {
        const int64_t h = hn + p * st;
#pragma unroll
        for (int q = 0; q < 3; q++) A[q] = B.M.p[q1 + q][h];
        split_k_metric(RR(A[0]), RR(A[1]), RR(A[2]), sw, K);
      }
      const RR ccr = div_known(RR(sqrt(Tt)), K.ma, K.rma);  // OCFD_inviscous.f90:67, in the splitting's type
      RR fp[5], fm[5];
      if (sw) split_sw<RR>(K, ccr, dd, uu, vv, ww, fp, fm);
      else split_llf<RR>(K, ccr, dd, uu, vv, ww, fp, fm);
#pragma unroll
      for (int m = 0; m < 5; m++) {
        sF[(m * 8 + p) * FB + lane] = fp[m];
        sF[((5 + m) * 8 + p) * FB + lane] = fm[m];
      }
      if (CHAR && (p == 3 || p == 4)) {
        double *const q = sQ + (p - 3) * 7 * FB + lane;
        q[0 * FB] = uu;
        q[1 * FB] = vv;
        q[2 * FB] = ww;
        q[3 * FB] = div_known(sqrt(double(Tt)), B.sk64[AXIS].ma, B.sk64[AXIS].rma);
        if (!unif) {
#pragma unroll
          for (int a = 0; a < 3; a++) q[(4 + a) * FB] = A[a];
        }
      }
    }
    const int f = (batch * NSUB + sub) * FB + lane;
    const int scm = (code & 1) ? 3 : 2;
    code = code1;
    if (batch + bstep < bhi) {
      fetch(code);
      code1 = entry(batch + 2 * bstep < bhi ? batch + 2 * bstep : batch + bstep);
    }
    __syncthreads();
    const auto *const F = sF + lane;
    auto recon_p = [&](const RR *x) {
      if (!CHAR) return MET ? inner_p<SCH_HYBRID>(S, x, scm) : face_p_nonchar<SCH_HYBRID>(S, x, s, n, AXIS, scm);
      return MET ? inner_p<SCH_HYBRID>(S, x, scm) : face_p_char<SCH_HYBRID>(S, x, s, n, AXIS, scm);
    };
    auto recon_m = [&](const RR *x) {
      if (!CHAR) return MET ? inner_m<SCH_HYBRID>(S, x, scm) : face_m_nonchar<SCH_HYBRID>(S, x, s, n, AXIS, scm);
      return MET ? inner_m<SCH_HYBRID>(S, x, scm) : face_m_char<SCH_HYBRID>(S, x, s, n, AXIS, scm);
    };
    if constexpr (!CHAR) {
      // flux+ and flux- of component `row`
      RR x[8];
#pragma unroll
      for (int k = 0; k < 8; k++) x[k] = F[(row * 8 + k) * FB];
      const RR hp = recon_p(x);
#pragma unroll
      for (int k = 0; k < 8; k++) x[k] = F[((5 + row) * 8 + k) * FB];
      const RR hm = recon_m(x);
      if (f < count) {
        out[(int64_t)f * NH + row] = hp;
        out[(int64_t)f * NH + 5 + row] = hm;
      }
      __syncthreads();  // the next batch overwrites the split fluxes
    } else {
      // basis from the face-averaged state (OCFD_inviscous_character.f90:200-236)
      double a[7];
#pragma unroll
      for (int q = 0; q < 7; q++) {
        if (q < 4 || !unif) a[q] = (sQ[q * FB + lane] + sQ[(7 + q) * FB + lane]) * 0.5;
        else a[q] = (B.M.u[q1 + q - 4] + B.M.u[q1 + q - 4]) * 0.5;
      }
      const double gamma = B.P.gamma;
      // row `row` of S (with MET 2 rows 1 and 2 are sr5[0] and sg at component
      // tq) and of S1; a product with an exact 0 or 1 changes no finite sum
      double sr5[5], sb5[5];
      // the tangents' coordinates and signs of an aligned metric vector
      constexpr int IL = AXIS == 0 ? 1 : 0, IM = AXIS == 2 ? 1 : 2;
      constexpr int SL = AXIS == 0 ? 1 : -1, SM = AXIS == 2 ? -1 : 1;
      const bool sparse = MET == 2 && (row == 1 || row == 2);
      const int tq = 1 + (row == 1 ? IL : IM);
      const double sg = row == 1 ? SL : SM;
      if constexpr (MET == 2) {
        const double un = a[AXIS], ul = SL > 0 ? a[IL] : -a[IL], um = SM > 0 ? a[IM] : -a[IM];
        const double V2 = (a[0] * a[0] + a[1] * a[1] + a[2] * a[2]) * 0.5;
        const double KK = ediv(gamma - 1.0, a[3] * a[3]);
        const double KK1 = KK * 0.5;
        if (row == 0) {
          sr5[0] = 1.0 - KK * V2;
          sr5[4] = -KK;
#pragma unroll
          for (int q = 0; q < 3; q++) sr5[1 + q] = KK * a[q];
        } else if (row < 3) {
          sr5[0] = row == 1 ? -ul : -um;
        } else {
          const double X1 = ediv(1.0, 2.0 * a[3]);
          sr5[0] = row == 3 ? KK1 * V2 + X1 * un : KK1 * V2 - X1 * un;
          sr5[4] = KK1;
#pragma unroll
          for (int q = 0; q < 3; q++)
            sr5[1 + q] = q == AXIS ? (row == 3 ? -X1 : X1) - KK1 * a[q] : -(KK1 * a[q]);
        }
        if (row == 0) {
          sb5[0] = sb5[3] = sb5[4] = 1.0;
          sb5[1] = sb5[2] = 0.0;
        } else if (row < 4) {
          const double v = row == 1 ? a[0] : (row == 2 ? a[1] : a[2]);
          sb5[0] = v;
          sb5[1] = row == 1 + IL ? SL : 0.0;
          sb5[2] = row == 1 + IM ? SM : 0.0;
          sb5[3] = row == 1 + AXIS ? v - a[3] : v;
          sb5[4] = row == 1 + AXIS ? v + a[3] : v;
        } else {
          const double H = V2 + ediv(1.0, KK);
          sb5[0] = V2;
          sb5[1] = ul;
          sb5[2] = um;
          sb5[3] = madd(-a[3], un, H);
          sb5[4] = madd(a[3], un, H);
        }
      } else {
        CharBasis Bs;
        if (row == 0) {  // needs no direction
          Bs.u1 = a[0];
          Bs.v1 = a[1];
          Bs.w1 = a[2];
          Bs.V2 = (a[0] * a[0] + a[1] * a[1] + a[2] * a[2]) * 0.5;
          Bs.KK = ediv(gamma - 1.0, a[3] * a[3]);
          char_S_row(Bs, 0, sr5);
          char_S1_row(Bs, 0, sb5);
        } else {
          char_basis(gamma, a[0], a[1], a[2], a[3], a[4], a[5], a[6], Bs);
          char_S_row(Bs, row, sr5);
          char_S1_row(Bs, row, sb5);
        }
      }
      // one flux projected (FP64) and reconstructed (RR) at a time, one
      // component's loads at a time (registers, as in the sweeps).  FP64 path:
      // the reference's two roundings per term; the mixed form fuses them.
      auto acc = [](double x, double y, double z) { return sizeof(RR) == 8 ? madd(x, y, z) : fma(x, y, z); };
      // (points k0 .. k0 + 6: WENO7 of flux + reads 0 .. 6, of flux - 1 .. 7,
      // WENO5 the inner five; outside its stencil, Ka1_H2.. / Ka1_H3.., the
      // closures read 0)
      auto project = [&](int p, const int k0, RR *y) {
        double x[8];
#pragma unroll
        for (int k = k0; k < k0 + 7; k++) x[k] = sr5[0] * double(F[(p * 8 + k) * FB]);
        if (sparse) {
#pragma unroll
          for (int k = k0; k < k0 + 7; k++) x[k] = xmadd(sg, double(F[((p + tq) * 8 + k) * FB]), x[k]);
        } else {
#pragma unroll
          for (int q = 1; q < 5; q++) {
#pragma unroll
            for (int k = k0; k < k0 + 7; k++) asm volatile("" : "+v"(x[k]) : : "memory");
#pragma unroll
            for (int k = k0; k < k0 + 7; k++) x[k] = acc(sr5[q], double(F[((p + q) * 8 + k) * FB]), x[k]);
          }
        }
#pragma unroll
        for (int k = 0; k < 8; k++) {
          const bool in = k >= k0 && k < k0 + 7;
          const bool inner = k > k0 && k < k0 + 6;
          y[k] = in ? RR(x[in ? k : k0]) : RR(0.0);
          if (!MET && in && !inner && scm == 3) y[k] = RR(0.0);
        }
      };
      RR y[8];
      project(0, 0, y);
      const RR hp = recon_p(y);
      __builtin_amdgcn_sched_barrier(0);
      project(5, 1, y);
      const RR hm = recon_m(y);
      sG[row * FB + lane] = double(hp + hm);
      __syncthreads();
      // back to conservative components (S1 * h0): component `row`
      double h0[5];
#pragma unroll
      for (int q = 0; q < 5; q++) h0[q] = sG[q * FB + lane];
      const double hh = madd(sb5[4], h0[4], madd(sb5[3], h0[3], madd(sb5[2], h0[2], madd(sb5[1], h0[1], sb5[0] * h0[0]))));
      if (f < count) out[(int64_t)f * NH + row] = RR(hh);
    }
  }
}

// one axis (AXIS >= 0), or all three in one launch of 3 x nwg workgroups
template <int AXIS, bool CHAR, int MET, typename RR>
__global__ __launch_bounds__(WNT) void k_weno_faces(const Block B, const int nwg) {
  // per batch:
  __shared__ weno_lds_t<CHAR, RR> sF[NSUB * 80 * FB];  // [10 components][8 points][face]
  __shared__ double sQ[CHAR ? NSUB * 14 * FB : 1];  // u, v, w, c, A1..A3 at points s, s+1
  __shared__ double sG[CHAR ? NSUB * 5 * FB : 1];   // characteristic fluxes h0(1:5)
  const int wg = (int)blockIdx.x % nwg;
  const int axis = AXIS >= 0 ? AXIS : (int)blockIdx.x / nwg;
  if (axis == 0) weno_faces_axis<0, CHAR, MET, RR>(B, sF, sQ, sG, wg, nwg);
  else if (axis == 1) weno_faces_axis<1, CHAR, MET, RR>(B, sF, sQ, sG, wg, nwg);
  else weno_faces_axis<2, CHAR, MET, RR>(B, sF, sQ, sG, wg, nwg);
}

template <int AXIS, bool CHAR, int MET, typename RR>
hipError_t weno_launch(const Block &B, hipStream_t st) {
  static DeviceCache cache;
  const Geom &g = B.g;
  int64_t faces = TileIndex<0>::nfaces(g);
  if (AXIS != 0 && TileIndex<1>::nfaces(g) > faces) faces = TileIndex<1>::nfaces(g);
  if (AXIS != 0 && TileIndex<2>::nfaces(g) > faces) faces = TileIndex<2>::nfaces(g);
  // as many workgroups per axis as the device holds at once, so that the batches
  // spread evenly, and no more than the axis can have batches
  const int64_t most = ((faces + NSUB * FB - 1) / (NSUB * FB) + NXCD - 1) / NXCD * NXCD;
  const int nwg = (int)std::min<int64_t>(most, resident_groups(k_weno_faces<AXIS, CHAR, MET, RR>, cache, WNT));
  hipLaunchKernelGGL((k_weno_faces<AXIS, CHAR, MET, RR>), dim3((unsigned)(AXIS >= 0 ? nwg : 3 * nwg)), dim3(WNT), 0,
                     st, B, nwg);
  return hipGetLastError();
}

// FP32 splitting and reconstruction in the mixed-precision form
template <int AXIS, bool CHAR, int MET>
hipError_t weno_prec(const Block &B, hipStream_t st) {
  if (B.prec == OCFD_PREC_MIXED_CODE) return weno_launch<AXIS, CHAR, MET, float>(B, st);
  return weno_launch<AXIS, CHAR, MET, double>(B, st);
}

template <int AXIS>
hipError_t weno_axis(const Block &B, hipStream_t st) {
  if (!(B.S.iperiodic[AXIS] == 1 && B.M.uniform))
    return B.S.is_char ? weno_prec<AXIS, true, 0>(B, st) : weno_prec<AXIS, false, 0>(B, st);
  if (!B.S.is_char) return weno_prec<AXIS, false, 1>(B, st);
  return axis_aligned<AXIS>(B.M) ? weno_prec<AXIS, true, 2>(B, st) : weno_prec<AXIS, true, 1>(B, st);
}

}  // namespace

hipError_t launch_hybrid_lists(const Block &B, hipStream_t st) {
  const Geom &g = B.g;
  constexpr int64_t FPB = NT * LPT;
  const unsigned n0 = (unsigned)((TileIndex<0>::nfaces(g) + FPB - 1) / FPB);
  const unsigned n1 = (unsigned)((TileIndex<1>::nfaces(g) + FPB - 1) / FPB);
  const unsigned n2 = (unsigned)((TileIndex<2>::nfaces(g) + FPB - 1) / FPB);
  hipLaunchKernelGGL(k_hyb_list, dim3(n0 + n1 + n2), dim3(NT), 0, st, B, n0, n1);
  return hipGetLastError();
}

// the listed faces of the three axes: one launch where the axes run the same
// kernel (a block of 64^3 has few batches per axis, and the axes' tails
// overlap), else one per axis
hipError_t launch_weno_faces(const Block &B, hipStream_t st) {
  if (!prims_match(B)) return hipErrorInvalidValue;
  const bool per = B.S.iperiodic[0] == 1 && B.S.iperiodic[1] == 1 && B.S.iperiodic[2] == 1;
  const bool aligned = axis_aligned<0>(B.M) && axis_aligned<1>(B.M) && axis_aligned<2>(B.M);
  if (per && B.M.uniform) {
    if (!B.S.is_char) return weno_prec<-1, false, 1>(B, st);
    if (aligned) return weno_prec<-1, true, 2>(B, st);
  } else if (!B.M.uniform || (B.S.iperiodic[0] != 1 && B.S.iperiodic[1] != 1 && B.S.iperiodic[2] != 1)) {
    return B.S.is_char ? weno_prec<-1, true, 0>(B, st) : weno_prec<-1, false, 0>(B, st);
  }
  hipError_t e = weno_axis<0>(B, st);
  if (e == hipSuccess) e = weno_axis<1>(B, st);
  return e == hipSuccess ? weno_axis<2>(B, st) : e;
}

}  // namespace ocfd
