// ocfd_inviscid_xy.hip -- the x and y sweeps of the hybrid scheme in one march.
//
// Same arithmetic as the two sweeps one after the other (ocfd_sweep.h,
// ocfd_march.h; du_inviscous_Character, OCFD_inviscous_character.f90:3-159):
// du = x part + y part, for the z sweep to add to.
#include <algorithm>

#include "ocfd_kernels.h"

namespace ocfd {

namespace {

constexpr int XYW = 64;  // columns of a wavefront

// v of lane m, in all lanes; v of the lane below, `first` in lane 0
__device__ __forceinline__ float lane_value(float v, int m) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), m));
}
__device__ __forceinline__ double lane_value(double v, int m) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), m),
                          __builtin_amdgcn_readlane(__double2loint(v), m));
}
__device__ __forceinline__ int lane_below(int v, int first) {
  return __builtin_amdgcn_update_dpp(first, v, 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
}
__device__ __forceinline__ float lane_below(float v, float first) {
  return __int_as_float(lane_below(__float_as_int(v), __float_as_int(first)));
}
__device__ __forceinline__ double lane_below(double v, double first) {
  return __hiloint2double(lane_below(__double2hiint(v), __double2hiint(first)),
                          lane_below(__double2loint(v), __double2loint(first)));
}

// a value that is the same in all lanes, in scalar registers
__device__ __forceinline__ float uniform(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ double uniform(double v) { return v; }

// One wavefront marches 64 neighbouring columns of a plane along y.  The split
// y fluxes of the last 8 points of a column are a register queue (as in
// ocfd_march.h); the split x fluxes of a row's 64 points lie in LDS, where each
// lane reads the stencil of its cell's right face.  The 4 points on either
// side of the row are split for 4 rows at a time, one point per lane, and the
// face left of the row by ten lanes, one of its ten sums each; a lane's left
// face is its neighbour's right one.  The x part of a row waits in LDS for
// its y part, which comes 4 rows later.  A workgroup is one wavefront, whose
// LDS accesses are in order: no barriers.
//
// The two sweeps write du, read it back and read the primitives twice: 200
// bytes per cell in FP64, 80 here.  They were bound by memory in FP64 (y 4.5
// TB/s) and by instruction issue in mixed precision (VALU 87% and 69% busy),
// where the march saves their tiles' overlap and index arithmetic.  It is bound
// by the issue of its two wavefronts per SIMD.  The map of the listed WENO
// faces is looked up a row ahead: at the row itself the two dependent loads
// took half the time (mixed 256^3 573 us).  x + y and march, 256^3 with 5.7%
// WENO faces: FP64 802 us and 600, mixed 506 and 285; 512^3 FP64 6150 and 4420.
template <typename R, bool SW>
__global__ __launch_bounds__(XYW) __attribute__((amdgpu_waves_per_eu(2)))
void k_inviscid_xy(const Block B, const int sl) {
  const Geom &g = B.g;
  const SchemeParams &S = B.S;
  constexpr int NP = XYW + 8;
  __shared__ R sRow[10 * NP];        // split x fluxes (+: 0-4, -: 5-9) of the row and its halo points
  __shared__ R sHal[10 * 32];        // those of the halo points of 4 rows
  __shared__ R ring[4 * 5 * XYW];    // x parts of 4 rows
  // FP64 is short of registers (the queue takes 160 of the 256 that two
  // wavefronts per SIMD leave each): the previous y face waits in LDS, the x
  // sums take one sign's stencil at a time, and a listed x face's fluxes are
  // loaded two components ahead instead of at the start of the row
  constexpr bool DP = sizeof(R) == 8;
  __shared__ R sPrev[DP ? 5 * XYW : 1];
  const int l = (int)threadIdx.x;
  const int nxs = (g.nx + XYW - 1) / XYW, nseg = (g.ny + sl - 1) / sl;
  int b = xcd_tile(blockIdx.x, gridDim.x);
  const int x0 = b % nxs * XYW + 1;
  b /= nxs;
  const int s0 = b % nseg * sl + 1, c = b / nseg + 1;
  const int s1 = s0 + sl - 1 < g.ny ? s0 + sl - 1 : g.ny;
  const bool act = x0 + l <= g.nx;
  const R *const pd = B.d.as<R>(), *const pu = B.u.as<R>(), *const pv = B.v.as<R>(), *const pw = B.w.as<R>(),
          *const pT = B.T.as<R>();
  R *const du = reinterpret_cast<R *>(B.du);
  const SplitK<R> KX = split_const<R>(B, 0), KY = split_const<R>(B, 1);
  const R hx = uniform(R(B.P.hinv[0])), hy = uniform(R(B.P.hinv[1]));
  R cf[8];
#pragma unroll
  for (int k = 0; k < 8; k++) cf[k] = uniform(R(S.ud7l[k]));
  auto sum_p = [&](const R *x) {  // ud7lp, ud7lm
    R s = cf[0] * x[0];
#pragma unroll
    for (int k = 1; k < 8; k++) s = madd(cf[k], x[k], s);
    return s;
  };
  auto sum_m = [&](const R *x) {
    R s = cf[0] * x[7];
#pragma unroll
    for (int k = 1; k < 8; k++) s = madd(cf[k], x[7 - k], s);
    return s;
  };
  const int ncell = s1 - s0 + 1, npts = ncell + 8;  // points s0 - 4 .. s1 + 4
  // point at h (uniform) and o bytes (32-bit, per lane)
  auto load = [&](int64_t h, unsigned o, R *q) {
    q[0] = *reinterpret_cast<const R *>(reinterpret_cast<const char *>(pd + h) + o);
    q[1] = *reinterpret_cast<const R *>(reinterpret_cast<const char *>(pu + h) + o);
    q[2] = *reinterpret_cast<const R *>(reinterpret_cast<const char *>(pv + h) + o);
    q[3] = *reinterpret_cast<const R *>(reinterpret_cast<const char *>(pw + h) + o);
    q[4] = *reinterpret_cast<const R *>(reinterpret_cast<const char *>(pT + h) + o);
  };
  auto sound = [&](const R *q) { return div_known(R(sqrt(q[4])), KX.ma, KX.rma); };  // OCFD_inviscous.f90:67
  auto split = [&](const SplitK<R> &K, R cc, const R *q, R *fp, R *fm) {
    if (SW) split_sw<R>(K, cc, q[0], q[1], q[2], q[3], fp, fm);
    else split_llf<R>(K, cc, q[0], q[1], q[2], q[3], fp, fm);
  };
  // columns past the block: the halo points of the last one, then its last
  const unsigned xo = (unsigned)((x0 + l < g.nx + LAP ? x0 + l : g.nx + LAP) - 1) * sizeof(R);
  auto load_row = [&](int p, R *o) { load(g.hi(1, s0 - 4 + (p < npts ? p : npts - 1), c), xo, o); };
  // halo point l % 8 (x0 - 4 .. x0 - 1, x0 + 64 .. x0 + 67) of row l / 8 % 4 of the group
  const int hq = l & 7;
  const int hxi = hq < 4 ? x0 - 4 + hq : (x0 + XYW - 4 + hq < g.nx + LAP ? x0 + XYW - 4 + hq : g.nx + LAP);
  const unsigned ho = (unsigned)(hxi + LAP - 1) * sizeof(R);
  auto load_halo = [&](int base, R *o) {
    const int p = base + ((l >> 3) & 3);
    load(g.hi(1 - LAP, s0 - 4, c), ho + (unsigned)((p < npts ? p : npts - 1) * g.sx) * (unsigned)sizeof(R), o);
  };
  // its place in the row: flux l / 8, and 8 + l / 8 % 2
  const int hd = hq < 4 ? hq : XYW + hq;
  const int hs0 = (l >> 3) * 32 + hq, hs1 = (8 + ((l >> 3) & 1)) * 32 + hq;
  const int hd0 = (l >> 3) * NP + hd, hd1 = (8 + ((l >> 3) & 1)) * NP + hd;
  // the face left of the row: lanes 0-4 its + sums, 5-9 its - sums, whose
  // terms come from the other end of the stencil
  const int lq = l < 10 ? l : 9, dir = lq < 5 ? 1 : -1;
  const int a0 = lq * NP + (lq < 5 ? 0 : 7);

  // face ids (ocfd_create refuses hybrid blocks with 2^30 or more per axis)
  const int sx = x0 + l < g.nx ? x0 + l : g.nx;
  const int yo = act ? x0 + l - 1 : 0;
  auto xfid = [&](int row) { return ((c - 1) * g.ny + (row - 1)) * (g.nx + 1); };
  auto yfid = [&](int f) { return ((c - 1) * (g.ny + 1) + f) * g.nx; };
  // Listed WENO faces (k_weno_faces) replace linear ones: the face map's entry
  // is loaded a row ahead, the fluxes at the start of the row that uses them.
  struct Entry {
    unsigned long long bits;
    int base;
  };
  auto entry = [&](int axis, int fid) { return Entry{B.hbits[axis][fid >> 6], B.hgbase[axis][fid >> 6]}; };
  // (the fluxes of slot 0 for a face that is not listed)
  auto listed = [&](int axis, int fid, const Entry &e, unsigned &at) {
    const int bit = (int)(fid & 63);
    const bool y = ((e.bits >> bit) & 1ull) != 0;
    const unsigned slot = (unsigned)(e.base + __popcll(e.bits & ((1ull << bit) - 1ull)));
    at = y ? slot * 5u : 0u;  // (inviscid_xy_wins bounds it)
    return y;
  };
  const R *const wfx = reinterpret_cast<const R *>(B.wflux[0]), *const wfy = reinterpret_cast<const R *>(B.wflux[1]);
  auto xrow_of = [&](int pi) { return s0 - 4 + (pi < 4 ? 4 : (pi < ncell + 4 ? pi : ncell + 3)); };
  auto yface_of = [&](int pi) { return s0 - 8 + (pi < 7 ? 7 : (pi < npts ? pi : npts - 1)); };

  R qp[8][5], qm[8][5];  // split y fluxes of the last 8 points
  R hprev[DP ? 1 : 5];   // fluxes of the previous y face (DP: sPrev)
  R pr[5];
  load_row(0, pr);
  Entry ey = entry(1, yfid(yface_of(0)) + yo), ex = entry(0, xfid(xrow_of(0)) + sx),
        el = entry(0, xfid(xrow_of(0)) + x0 - 1);
  for (int base = 0; base < npts; base += 8) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
      // (opaque: the addresses of each of the 8 steps kept as induction
      // variables took 90 registers)
      int pi = base + j;
      asm volatile("" : "+s"(pi));
      const bool xrow = pi >= 4 && pi < ncell + 4;
      const int f = s0 - 8 + pi;
      R wy[5], wx[5];
      unsigned fy, fx, fl;
      const bool ly = listed(1, yfid(yface_of(pi)) + yo, ey, fy), lx = listed(0, xfid(xrow_of(pi)) + sx, ex, fx),
                 ll = listed(0, xfid(xrow_of(pi)) + x0 - 1, el, fl);
#pragma unroll
      for (int q = 0; q < 5; q++) {
        wy[q] = wfy[fy + q];
        if (!DP) wx[q] = wfx[fx + q];
      }
      const R wl = wfx[fl + (l < 5 ? l : 4)];
      // ---- split fluxes of the row's points ----
      const R cc = sound(pr);
      split(KY, cc, pr, qp[j], qm[j]);
      if (xrow) {
        R fp[5], fm[5];
        split(KX, cc, pr, fp, fm);
#pragma unroll
        for (int m = 0; m < 5; m++) {
          sRow[m * NP + 4 + l] = fp[m];
          sRow[(5 + m) * NP + 4 + l] = fm[m];
        }
      }
      load_row(pi + 1, pr);
      R ph[5];
      if (j % 4 == 0) load_halo(base + j, ph);
      ey = entry(1, yfid(yface_of(pi + 1)) + yo);
      ex = entry(0, xfid(xrow_of(pi + 1)) + sx);
      const Entry el1 = entry(0, xfid(xrow_of(pi + 1)) + x0 - 1);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_sched_barrier(0);
      // ---- y face f, stencil f-3 .. f+4, and cell f ----
      if (pi >= 7) {
        R hv[5];
#pragma unroll
        for (int m = 0; m < 5; m++) {
          R xp[8], xm[8];
#pragma unroll
          for (int k = 0; k < 8; k++) {
            xp[k] = qp[(j + 1 + k) & 7][m];
            xm[k] = qm[(j + 1 + k) & 7][m];
          }
          const R h1 = sum_p(xp);
          const R h2 = sum_m(xm);
          hv[m] = ly ? wy[m] : h1 + h2;
          asm volatile("" : "+v"(hv[m])::"memory");
        }
        if (pi >= 8 && act && pi - 8 < ncell) {
          R *const dq = du + g.ii(x0, f, c);
#pragma unroll
          for (int m = 0; m < 5; m++) {
            const R below = DP ? sPrev[m * XYW + l] : hprev[DP ? 0 : m];
            (dq + m * g.ni)[l] = ring[((j & 3) * 5 + m) * XYW + l] + (hv[m] - below) * hy;
          }
        }
#pragma unroll
        for (int m = 0; m < 5; m++) {
          if (DP) sPrev[m * XYW + l] = hv[m];
          else hprev[DP ? 0 : m] = hv[m];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (j % 4 == 0) {
        // ---- halo points of this row and the next 3 ----
        R fp[5], fm[5];
        split(KX, sound(ph), ph, fp, fm);
        if (l < 32) {
#pragma unroll
          for (int m = 0; m < 5; m++) {
            sHal[m * 32 + l] = fp[m];
            sHal[(5 + m) * 32 + l] = fm[m];
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
      // ---- x faces and cells of the row ----
      if (DP) {
        asm volatile("" : "+v"(fx)::"memory");
        wx[0] = wfx[fx];
        wx[1] = wfx[fx + 1];
      }
      if (xrow) {
        const R v0 = sHal[hs0 + (j & 3) * 8], v1 = sHal[hs1 + (j & 3) * 8];
        sRow[hd0] = v0;
        sRow[hd1] = v1;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        // the face left of the row: component m in lane m
        R hl;
        {
          R x[8];
#pragma unroll
          for (int k = 0; k < 8; k++) x[k] = sRow[a0 + dir * k];
          const R h1 = sum_p(x), h2 = __shfl(h1, l + 5);
          hl = ll ? wl : h1 + h2;
        }
        // one component's stencil at a time in registers
#pragma unroll
        for (int m = 0; m < 5; m++) {
          if (DP && m < 3) wx[m + 2] = wfx[fx + m + 2];
          R xp[8], xm[8];
#pragma unroll
          for (int k = 0; k < 8; k++) xp[k] = sRow[m * NP + l + 1 + k];
          if (!DP)
#pragma unroll
            for (int k = 0; k < 8; k++) xm[k] = sRow[(5 + m) * NP + l + 1 + k];
          R h1 = sum_p(xp);
          if (DP) {
            asm volatile("" : "+v"(h1)::"memory");
#pragma unroll
            for (int k = 0; k < 8; k++) xm[k] = sRow[(5 + m) * NP + l + 1 + k];
          }
          const R h2 = sum_m(xm);
          const R h = lx ? wx[m] : h1 + h2;
          R part = (h - lane_below(h, lane_value(hl, m))) * hx;
          asm volatile("" : "+v"(part)::"memory");
          ring[((j & 3) * 5 + m) * XYW + l] = part;
        }
      }
      el = el1;
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
}

// Rows of a segment: the march's time is close to the number of rounds of
// resident wavefronts times the rows of a segment (its cells and 8 more, in
// whole groups of 8); `work` gets that product in lanes.  Of equal ones the
// shortest segments (FP64 256^3: 7 segments 600 us, 5 639).
template <typename R, bool SW>
int xy_segment(const Geom &g, int64_t &work) {
  static DeviceCache cache;
  const int64_t slots = resident_groups(k_inviscid_xy<R, SW>, cache, XYW);
  const int64_t cols = (int64_t)((g.nx + XYW - 1) / XYW) * g.nz;
  int best = 0;
  work = INT64_MAX;
  for (int nseg = 1; nseg <= (g.ny + 7) / 8; nseg++) {
    const int sl = (g.ny + nseg - 1) / nseg;
    const int64_t rounds = (cols * ((g.ny + sl - 1) / sl) + slots - 1) / slots;
    const int64_t w = rounds * ((sl + 15) / 8 * 8) * slots * XYW;
    if (w <= work) {
      work = w;
      best = sl;
    }
  }
  return best;
}

template <typename R, bool SW>
hipError_t inviscid_xy_as(const Block &B, hipStream_t st) {
  const Geom &g = B.g;
  int64_t work;
  const int sl = xy_segment<R, SW>(g, work);
  const int64_t waves = (int64_t)((g.nx + XYW - 1) / XYW) * ((g.ny + sl - 1) / sl) * g.nz;
  hipLaunchKernelGGL((k_inviscid_xy<R, SW>), dim3((unsigned)waves), dim3(XYW), 0, st, B, sl);
  return hipGetLastError();
}

}  // namespace

// Two sweeps cost about twice the march's time per lane and row, so the march
// wins where its lanes' rows -- the 8 more of each segment, idle columns and
// unfilled rounds with them -- are less than about twice the cells.  x + y and
// march, us: FP64 128^3 (1.75 rows per cell) 100 and 95, 160^3 (1.79) 219 and
// 189, 200 x 180 x 150 (2.2) 301 and 283, 96^3 (3.1) 50 and 67; mixed precision
// 128^3 (1.5) 66 and 48, 200 x 180 x 150 (1.75) 176 and 134, 100 x 140 x 120
// (2.5) 57 and 60.  Steger-Warming in FP64 needs more registers than there
// are: 256^3 (1.3) 840 and 777, 160^3 219 and 240.
// It addresses the five fluxes of a listed face with 32 bits, so blocks with
// more faces per axis than that reaches (ocfd_create accepts up to 2^30) take
// the two sweeps.
bool inviscid_xy_wins(const Block &B) {
  if (B.S.scheme_invis != SCH_HYBRID || !B.S.is_char || B.S.iperiodic[0] != 1 || B.S.iperiodic[1] != 1 || !B.M.uniform)
    return false;
  if (5 * std::max(TileIndex<0>::nfaces(B.g), TileIndex<1>::nfaces(B.g)) > (int64_t)UINT32_MAX) return false;
  const bool f32 = B.prec == OCFD_PREC_MIXED_CODE, sw = B.S.flux_split == 1;
  int64_t work;
  if (f32) sw ? xy_segment<float, true>(B.g, work) : xy_segment<float, false>(B.g, work);
  else sw ? xy_segment<double, true>(B.g, work) : xy_segment<double, false>(B.g, work);
  return 10 * work < (sw && !f32 ? 17 : 22) * B.g.ni;
}

hipError_t launch_inviscid_xy(const Block &B, hipStream_t st) {
  if (!prims_match(B)) return hipErrorInvalidValue;
  const bool sw = B.S.flux_split == 1;
  if (B.prec == OCFD_PREC_MIXED_CODE)
    return sw ? inviscid_xy_as<float, true>(B, st) : inviscid_xy_as<float, false>(B, st);
  return sw ? inviscid_xy_as<double, true>(B, st) : inviscid_xy_as<double, false>(B, st);
}

}  // namespace ocfd
