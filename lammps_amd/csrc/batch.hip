// batch.hip - forces and force-matching adjoints over many independent
// configurations ("replicas") in single persistent launches (mdx_batch.h).
//
// Layout: all replicas' atoms in one array, sorted by a global bin key
// (replica bin offset + local bin), so replicas stay contiguous and in
// order, and within a replica atoms are bin-sorted.  Each replica has its
// own orthogonal box, periodicity and bin grid (binsize >= cutneigh/2,
// stencil +-2 bins).  Lists are full, row-major, one row per atom; an entry
// holds the neighbour index (bits 0-26) and its periodic image code
// 9(sx+1) + 3(sy+1) + (sz+1) (bits 27-31).  The ghost coordinate is
// x_j + s*prd rounded once, as CommBrick::borders forms it
// (atom_vec_atomic.cpp:290-297): whether a pair lies inside a cutoff is
// decided by the FP64 distance to it, in each atom's row by itself.  Away
// from the cutoff the passes use cheaper separations (kQBand).
//
// Every pair kernel is persistent: block b takes a contiguous chunk of
// atoms (chunks ordered so each XCD gets a contiguous eighth) and loops over
// it in tiles of block/TPA atoms, so one launch covers all replicas
// whatever their sizes, and the grid is a tuning parameter.
//
// Adjoints (reference expressions: pair_lj_cut.cpp:104-112,
// pair_eam.cpp:160-303).  With G_i = dL/dF_i and full-list rows:
//   lj:  dL/deps_ab   += (G_i.del) r^-8 (48 s^12 r^-6 - 24 s^6)
//        dL/dsigma_ab += (G_i.del) r^-8 (576 eps s^11 r^-6 - 144 eps s^5)
//   eam: b = -(G_i.del)/r;  z2r'(r) gets b/r, z2r(r) gets -b/r^2,
//        rhor'(r) gets b (fp_i + fp_j),
//        u_i = sum_j -((G_i - G_j).del)/r rhor'(r)  (= dL/dfp_i, both rows),
//        frho'(rho_i) gets u_i, and v_i = u_i F''(rho_i) reaches rhor(r)
//        through rho_i (second pass).
// The adjoint kernels run FP64 arithmetic whatever the forward precision.
// Gradients are accumulated per spline interval and coefficient (c3..c6:
// the value weights p^3, p^2, p, 1 and derivative weights 3p^2, 2p, 1, 0
// over the knot spacing) in LDS with ds_add_f64, flushed per block and
// summed over blocks in a fixed order; the host maps coefficient gradients
// to knot gradients with the transpose of the spline construction.
#include <hip/hip_ext.h>
#include <hipcub/hipcub.hpp>

#include <cmath>
#include <type_traits>

#include "../../include/mdx_batch.h"
#include "bin_rows.h"
#include "mdx_internal.h"

namespace mdx {
namespace {

constexpr int kS = 2;  // stencil half-width in bins (binsize >= cutneigh / 2)
constexpr int kNT = MDX_NT1 * MDX_NT1;
constexpr int kTabLDS = 6144;  // doubles of spline table staged in LDS at most (48 KB)

struct RepGeom {
  double lo[3], prd[3], bininv[3];
  // 32-bit fixed-point positions of the mixed-precision force passes:
  // q = round((x - lo) * qscale) (mod 2^32 periodic, where the wrapping
  // difference is the minimum-image separation), qstep = prd * 2^-32
  // (periodic) or prd * 2^-30, exact
  double qscale[3], qstep[3];
  double iprd[3];  // 1 / prd in periodic dimensions, 0 in the others
  int nbin[3], periodic[3];
  int bin_off;
};

// Pairs at the cutoff are tested again on the FP64 positions with their image
// (image_rsq).  By the fixed-point separations, those within kQBand of it
// (relative, on rsq).  By the nearest-image separations of the FP64 passes,
// those whose rsq has one of the two upper words h and h + 1 around cutsq,
// h = edge_word(cutsq): at least 2^-21 of it on either side.  So one integer
// difference says inside (negative), edge (0 or 1) or outside.
constexpr double kQBand = 2e-6;
__device__ __forceinline__ int edge_word(double cutsq) {
  return __double2hiint(cutsq) - (static_cast<unsigned>(__double2loint(cutsq)) < 0x80000000u ? 1 : 0);
}

__device__ __forceinline__ int4 quantize_rep(const RepGeom &g, const double4 &p) {
  return make_int4((int)(unsigned)(long long)rint((p.x - g.lo[0]) * g.qscale[0]),
                   (int)(unsigned)(long long)rint((p.y - g.lo[1]) * g.qscale[1]),
                   (int)(unsigned)(long long)rint((p.z - g.lo[2]) * g.qscale[2]), (int)p.w);
}

__device__ __forceinline__ double qsep(int qi, int qj, double step) {
  return (double)(int)((unsigned)qi - (unsigned)qj) * step;
}



// lj/cut tables (ntypes+1)^2: cutsq, lj1..lj4 (init_one), and the
// gradient factors A1 = 48 s^12, A2 = 24 s^6, B1 = 576 eps s^11, B2 = 144 eps s^5
enum { T_CUTSQ = 0, T_LJ1, T_LJ2, T_LJ3, T_LJ4, T_A1, T_A2, T_B1, T_B2, T_N };

struct EamTab {
  int nrho, nr;
  double rdrho, rdr, rhomax, cutsq;
};

struct Tune {
  int block = 0, tpa = 0, grid = 0;  // tpa 0: by default_tune
};

__device__ __forceinline__ int chunk_begin(int n, int apb, int *end) {
  const int G = gridDim.x;
  const int lb = (G % kXCD == 0) ? xcd_block() : blockIdx.x;
  const int tiles = (n + apb - 1) / apb;
  const int per = (tiles + G - 1) / G;
  const int b0 = lb * per * apb;
  *end = min(n, b0 + per * apb);
  return b0;
}

template <int TPA, typename T>
__device__ __forceinline__ T gsum(T v) {
#pragma unroll
  for (int off = TPA / 2; off > 0; off >>= 1) v += __shfl_down(v, off, TPA);
  return v;
}

__device__ __forceinline__ void shift_of(int code, double &sx, double &sy, double &sz) {
  sx = (double)(code / 9 - 1);
  sy = (double)((code / 3) % 3 - 1);
  sz = (double)(code % 3 - 1);
}

// the squared distance from a to the ghost of b under an image code, rounded as
// the reference rounds it (every product and sum)
__device__ __forceinline__ double image_rsq(const double4 &a, const double4 &b, int code, const RepGeom &g) {
#pragma clang fp contract(off)
  double sx, sy, sz;
  shift_of(code, sx, sy, sz);
  const double ex = a.x - (b.x + sx * g.prd[0]), ey = a.y - (b.y + sy * g.prd[1]), ez = a.z - (b.z + sz * g.prd[2]);
  return ex * ex + ey * ey + ez * ez;
}
// the code under which b sees a's image
__device__ __forceinline__ int reverse_code(int code) { return 26 - code; }

__device__ __forceinline__ int local_bin(const RepGeom &g, double x, int d) {
  int c = (int)floor((x - g.lo[d]) * g.bininv[d]);
  return min(max(c, 0), g.nbin[d] - 1);
}

// ---------------------------------------------------------------- build

// caller order: wrap (Domain::pbc), bin key, histogram
__global__ void k_b_load(int n, const double *__restrict__ xin, const int *__restrict__ type,
                         const int *__restrict__ rep_c, const RepGeom *__restrict__ geom, double4 *__restrict__ xw,
                         unsigned *__restrict__ key, int *__restrict__ slot, int *__restrict__ bin_count,
                         int *__restrict__ dflags) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const RepGeom &g = geom[rep_c[c]];
  double v[3];
  for (int d = 0; d < 3; d++) {
    double u = xin[3 * (size_t)c + d];
    const double hi = g.lo[d] + g.prd[d];
    if (g.periodic[d]) {
      if (u < g.lo[d] || u >= hi) {
        u -= floor((u - g.lo[d]) / g.prd[d]) * g.prd[d];
        if (u >= hi) u -= g.prd[d];
        u = fmax(u, g.lo[d]);
      }
    } else if (!(u >= g.lo[d] && u <= hi)) {
      atomicOr(&dflags[4], 1);  // outside a non-periodic box
    }
    if (u != u) atomicOr(&dflags[7], 1);  // no place: the mirror would give it one
    v[d] = u;
  }
  xw[c] = make_double4(v[0], v[1], v[2], (double)type[c]);
  const int bx = local_bin(g, v[0], 0), by = local_bin(g, v[1], 1), bz = local_bin(g, v[2], 2);
  const unsigned k = (unsigned)(g.bin_off + (bz * g.nbin[1] + by) * g.nbin[0] + bx);
  key[c] = k;
  slot[c] = atomicAdd(&bin_count[k], 1);  // arrival order; k_b_rank_permute makes it the caller's
}

// Stable counting sort by bin: each atom to its arrival slot in its bin, then
// to the rank of its caller index among the bin's atoms (a bin holds a few).
__global__ void k_b_scatter(int n, const unsigned *__restrict__ key, const int *__restrict__ slot,
                            const int *__restrict__ bin_start, int *__restrict__ tmp) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < n) tmp[bin_start[key[c]] + slot[c]] = c;
}

__global__ void k_b_rank_permute(int n, const int *__restrict__ tmp, const unsigned *__restrict__ key,
                                 const int *__restrict__ bin_start, const double4 *__restrict__ xw,
                                 const int *__restrict__ rep_c, const RepGeom *__restrict__ geom,
                                 double4 *__restrict__ x, int4 *__restrict__ xq, int *__restrict__ rep,
                                 int *__restrict__ orig, int *__restrict__ inv) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int c = tmp[p];
  const unsigned b = key[c];
  const int s = bin_start[b], e = bin_start[b + 1];
  const double4 q = xw[c];
  const int r = rep_c[c];
  int k = s;
  for (int t = s; t < e; t++) k += tmp[t] < c;
  x[k] = q;
  xq[k] = quantize_rep(geom[r], q);
  rep[k] = r;
  orig[k] = c;
  inv[c] = k;
}

// The list build, 32 lanes per atom: the atom's 25 stencil rows (y, z) in
// parallel, one per lane, each row of bins one contiguous atom range (two
// where it wraps around a periodic x face); a scan over the lanes places the
// rows in the atom's candidate sequence (z, y, x ascending), the lanes write
// the sequence to LDS and test it 32 at a time, four gathers in flight, a
// ballot placing the accepted entries in the row.  Rows and row ends beyond
// the cutoff are skipped (FP32 bin units, margins 1e-3 bin and 1e-4 on the
// squared cutoff).  Q: candidates come from the fixed-point mirror and are
// tested in FP32; one within kBuildBand of the cutoff is re-tested on the
// FP64 positions with its image, so the list is the FP64 test's (the host
// checks that the mirror is fine enough and that no stencil holds an atom
// under two images).  A pair on the cutoff that the rounding of its two ghosts
// puts into one row only is listed in both: the force passes decide each row
// again, the gradient passes need it in the row they take it from.  The one-loop-per-bin build that this replaces read 250
// bin starts per atom one after the other and counted rows in two words by
// atomics: 962 us at 96 x 1,331 atoms, 1.90 ms at 64 x 8,000, 7.32 ms for
// 512 clusters of 1.33 M atoms.
constexpr int kBuildLanes = 32, kBuildU = 4, kBuildBlock = 256, kBuildGrid = 2048;
constexpr int kBuildCand = 384;  // candidates of one atom held in LDS at a time
constexpr double kBuildBand = 2e-6;
constexpr int kRows = 2 * kS + 1;
template <bool Q>
__global__ __launch_bounds__(kBuildBlock, 5) void k_b_build(int n, const double4 *__restrict__ x,
                                                            const int4 *__restrict__ xq, const int *__restrict__ rep,
                                                            const RepGeom *__restrict__ geom,
                                                            const int *__restrict__ bin_start, double cutneighsq,
                                                            float c_lo, float c_hi, float reach, int cap,
                                                            int *__restrict__ nbr, int *__restrict__ numneigh,
                                                            ListSlot *__restrict__ slots) {
  static_assert(kRows * kRows <= kBuildLanes, "one stencil row per lane");
  constexpr int GL = kBuildLanes, NG = kBuildBlock / GL;
  __shared__ int s_cand[NG * kBuildCand];
  __shared__ int s_max[NG], s_sum[NG];
  const int lane = threadIdx.x % GL, grp = threadIdx.x / GL;
  const unsigned long long gmask = 0xffffffffull << ((threadIdx.x & 63) / GL * GL);
  int *const cand = s_cand + grp * kBuildCand;
  const int tiles = (n + NG - 1) / NG, per_xcd = (tiles + kXCD - 1) / kXCD;
  const int xcd = blockIdx.x % kXCD, step = gridDim.x / kXCD;
  const int dz = lane / kRows - kS, dy = lane % kRows - kS;  // this lane's stencil row
  int most = 0, sum = 0;
  for (int tt = blockIdx.x / kXCD; tt < per_xcd; tt += step) {
    const int i = (xcd * per_xcd + tt) * NG + grp;
    const bool live = i < n;
    const int ii = live ? i : 0;
    const double4 xi = x[ii];
    int4 qi = make_int4(0, 0, 0, 0);
    if constexpr (Q) qi = xq[ii];
    const RepGeom &g = geom[rep[ii]];
    const int nbx = g.nbin[0], nby = g.nbin[1], nbz = g.nbin[2];
    const int ix = local_bin(g, xi.x, 0), iy = local_bin(g, xi.y, 1), iz = local_bin(g, xi.z, 2);
    const float tx = (float)((xi.x - g.lo[0]) * g.bininv[0]), ty = (float)((xi.y - g.lo[1]) * g.bininv[1]),
                tz = (float)((xi.z - g.lo[2]) * g.bininv[2]);
    const float q0 = (float)g.qstep[0], q1 = (float)g.qstep[1], q2 = (float)g.qstep[2];
    const int self = i | (13 << MDX_IDX_BITS);
    // the row's pieces in scan order: bins [lo, hi) and the image code
    int lo[2] = {0, 0}, hi[2] = {0, 0}, code[2] = {0, 0};
    const float bsy = (float)g.prd[1] / (float)nby, bsz = (float)g.prd[2] / (float)nbz;
    const float gz = (dz > 0 ? (iz + dz) - tz : dz < 0 ? tz - (iz + dz + 1) : 0.0f) - 1e-3f;
    const float gy = (dy > 0 ? (iy + dy) - ty : dy < 0 ? ty - (iy + dy + 1) : 0.0f) - 1e-3f;
    const float dyz2 = (gz > 0.0f ? gz * gz * bsz * bsz : 0.0f) + (gy > 0.0f ? gy * gy * bsy * bsy : 0.0f);
    int jz = iz + dz, jy = iy + dy;
    const int sz = jz < 0 ? -1 : jz >= nbz ? 1 : 0, sy = jy < 0 ? -1 : jy >= nby ? 1 : 0;
    if (live && lane < kRows * kRows && dyz2 <= reach && (sz == 0 || g.periodic[2]) && (sy == 0 || g.periodic[1])) {
      jz -= sz * nbz;
      jy -= sy * nby;
      const int rowbase = g.bin_off + (jz * nby + jy) * nbx;
      const float wb = sqrtf(reach - dyz2) * (float)g.bininv[0] + 1e-3f;
      int x0, x1;
      row_bins(ix, kS, tx, wb, x0, x1);
      const int cyz = 9 * (0 + 1) + 3 * (sy + 1) + (sz + 1);
      const bool wlo = x0 < 0 && g.periodic[0], whi = x1 >= nbx && g.periodic[0];  // 2 kS <= nbx: not both
      const int p = wlo ? 1 : 0;
      lo[p] = rowbase + max(x0, 0);  // x0 <= ix <= x1: never empty
      hi[p] = rowbase + min(x1, nbx - 1) + 1;
      code[p] = cyz;
      if (wlo) {
        lo[0] = rowbase + x0 + nbx;
        hi[0] = rowbase + nbx;
        code[0] = cyz - 9;
      } else if (whi) {
        lo[1] = rowbase;
        hi[1] = rowbase + (x1 - nbx) + 1;
        code[1] = cyz + 9;
      }
    }
    int jlo[2], len[2];
#pragma unroll
    for (int p = 0; p < 2; p++) {
      jlo[p] = bin_start[lo[p]];
      len[p] = bin_start[hi[p]] - jlo[p];
    }
    const int mine = len[0] + len[1];
    int incl = mine;
#pragma unroll
    for (int off = 1; off < GL; off <<= 1) {
      const int up = __shfl_up(incl, off, GL);
      if (lane >= off) incl += up;
    }
    const int total = __shfl(incl, GL - 1, GL), first = incl - mine;
    int *const row = nbr + (size_t)ii * cap;
    int cnt = 0;
    for (int w = 0; w < total; w += kBuildCand) {
      const int wn = min(total - w, kBuildCand);
      int at = first - w;
#pragma unroll
      for (int p = 0; p < 2; p++) {
        const int t1 = min(len[p], kBuildCand - at);
        const int e0 = jlo[p] | (code[p] << MDX_IDX_BITS);
        for (int t = max(0, -at); t < t1; t++) cand[at + t] = e0 + t;
        at += len[p];
      }
      // a group lies in one wavefront: its writes above precede its reads
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      for (int c0 = lane; c0 - lane < wn; c0 += GL * kBuildU) {
        int e[kBuildU];
        double4 xj[Q ? 1 : kBuildU];
        int4 qj[Q ? kBuildU : 1];
#pragma unroll
        for (int u = 0; u < kBuildU; u++) {
          const int c = c0 + u * GL;
          e[u] = c < wn ? cand[c] : self;  // past the end: the atom itself, rejected below
        }
#pragma unroll
        for (int u = 0; u < kBuildU; u++) {
          if constexpr (Q) qj[u] = gather_q(xq, e[u]);
          else xj[u] = gather_x(x, e[u]);
        }
#pragma unroll
        for (int u = 0; u < kBuildU; u++) {
          bool keep = e[u] != self;
          bool test64 = keep;
          if constexpr (Q) {
            const float dx = (float)(int)((unsigned)qi.x - (unsigned)qj[u].x) * q0;
            const float dy = (float)(int)((unsigned)qi.y - (unsigned)qj[u].y) * q1;
            const float dz = (float)(int)((unsigned)qi.z - (unsigned)qj[u].z) * q2;
            const float rq = dx * dx + dy * dy + dz * dz;
            test64 = keep && rq > c_lo && rq <= c_hi;
            keep = keep && rq <= c_hi;
          }
          if (test64) {
            const int code = (int)((unsigned)e[u] >> MDX_IDX_BITS);
            double4 pi = xi, pj = Q ? xi : xj[Q ? 0 : u];
            if constexpr (Q) {
              pi = x[ii];
              pj = gather_x(x, e[u]);
            }
            const double rsq = image_rsq(pi, pj, code, g);
            keep = rsq < cutneighsq;
            // a pair on the cutoff that the other row holds
            if (!keep && rsq < cutneighsq * (1.0 + kBuildBand)) keep = image_rsq(pj, pi, reverse_code(code), g) < cutneighsq;
          }
          const unsigned long long m = __ballot(keep) & gmask;
          if (keep) {
            const int k = cnt + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
            if (k < cap) row[k] = e[u];
          }
          cnt += __popcll(m);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // read before the next window is written
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if (live && lane == 0) numneigh[i] = cnt;
    most = max(most, cnt);
    sum += cnt;
  }
  if (lane == 0) {
    s_max[grp] = most;
    s_sum[grp] = sum;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long all = 0;
    for (int k = 0; k < NG; k++) {
      most = max(most, s_max[k]);
      all += (unsigned long long)s_sum[k];
    }
    count_rows(slots, most, all);
  }
}

// Results of a force pass: the atom's energy in sorted order (for the replica
// sums), its force straight into the caller's order (f null: not wanted)
struct ForceOut {
  double *e;
  double *f;
  const int *orig;
  __device__ __forceinline__ void store(int i, double fx, double fy, double fz, double energy) const {
    e[i] = energy;
    if (!f) return;
    double *const d = f + 3 * (size_t)orig[i];
    d[0] = fx;
    d[1] = fy;
    d[2] = fz;
  }
};

// ---------------------------------------------------------------- pair helpers

// One lane's four consecutive entries k0 .. k0+3 of a row (rows start 16-B
// aligned; entries past jn are not written and become the atom itself)
__device__ __forceinline__ void row_chunk(const int *__restrict__ row, int k0, int jn, int self, int (&ent)[4]) {
  const int4 e4 = *reinterpret_cast<const int4 *>(row + k0);
  ent[0] = e4.x;
  ent[1] = k0 + 1 < jn ? e4.y : self;
  ent[2] = k0 + 2 < jn ? e4.z : self;
  ent[3] = k0 + 3 < jn ? e4.w : self;
}

// How a lane walks its share of a row.  By chunk: four consecutive entries,
// the chunks lane, lane + TPA, ...  QUAD with four lanes per atom: the four
// chunks of a trip are transposed across the lanes, so gather u of the atom
// covers entries 4u .. 4u+3 of the trip, which share cache lines, instead of
// entries u, 4+u, 8+u, 12+u.  That pays for the passes that gather 64 B per
// pair and wait for L1 (40 line lookups per load instruction, chunk / quad at
// 1,367,136 atoms: eam pass A 412 / 367 us, pass B 186 / 179, FP64 forces 269 /
// 261; lj gradient 101,250 atoms 45.3 / 40.8); the 16-B gathers of mixed
// precision, and more lanes in small batches, lose (101,903: 14.8 / 16.0).
template <int TPA, bool QUAD>
struct RowWalk {
  static constexpr bool kQuad = QUAD && TPA == 4;
  int lane;
  __device__ __forceinline__ int first() const { return kQuad ? 0 : 4 * lane; }
  // the entry that gather u of the trip from k0 covers
  __device__ __forceinline__ int at(int k0, int u) const { return kQuad ? k0 + 4 * u + lane : k0 + u; }
  __device__ __forceinline__ void read(const int *__restrict__ row, int k0, int jn, int self, int (&ent)[4]) const {
    if constexpr (kQuad) {  // trips are group-uniform: the transpose reads all four lanes
      int4 e4 = make_int4(self, self, self, self);
      if (k0 + 4 * lane < jn) e4 = *reinterpret_cast<const int4 *>(row + k0 + 4 * lane);
      ent[0] = e4.x;
      ent[1] = e4.y;
      ent[2] = e4.z;
      ent[3] = e4.w;
      quad_transpose(ent, lane);
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (at(k0, u) >= jn) ent[u] = self;
    } else {
      row_chunk(row, k0, jn, self, ent);
    }
  }
};

// separation of a pair within half the box, in FP64: the nearest image
// (periodic boxes are at least two cutoffs wide, so it is the list's)
__device__ __forceinline__ double nearest(double d, double prd, double iprd) { return fma(-prd, rint(d * iprd), d); }
__device__ __forceinline__ double nearest_rsq(const double4 &a, const double4 &b, const double (&prd)[3],
                                              const double (&iprd)[3], double &dx, double &dy, double &dz) {
  dx = nearest(a.x - b.x, prd[0], iprd[0]);
  dy = nearest(a.y - b.y, prd[1], iprd[1]);
  dz = nearest(a.z - b.z, prd[2], iprd[2]);
  return dx * dx + dy * dy + dz * dz;
}

// A pair that may lie on the cutoff.  There the rounding of the two ghosts can
// put it into one of its rows only: here() and there() decide for the row of
// xi and for that of xj.
struct EdgePair {
  const int i, ent;
  const double4 xi, xj;
  const RepGeom &g;
  double dx, dy, dz, rsq;
  __device__ __forceinline__ bool on_edge(int h) const { return (unsigned)(__double2hiint(rsq) - h) < 2u; }
  __device__ __forceinline__ bool first() const { return (ent & MDX_IDX_MASK) > i; }
  __device__ __forceinline__ bool here(double cutsq) const { return image_rsq(xi, xj, code(), g) < cutsq; }
  __device__ __forceinline__ bool there(double cutsq) const { return image_rsq(xj, xi, reverse_code(code()), g) < cutsq; }
  __device__ __forceinline__ int code() const { return (int)((unsigned)ent >> MDX_IDX_BITS); }
  // (G_i - G_j) . del, each row's share if the pair is inside there
  __device__ __forceinline__ double factor(const double4 &gi, const double4 &gj, double cutsq) const {
    return (here(cutsq) ? gi.x * dx + gi.y * dy + gi.z * dz : 0.0) -
           (there(cutsq) ? gj.x * dx + gj.y * dy + gj.z * dz : 0.0);
  }
};

// The FP64 passes leave a row's pairs on the cutoff's edge for after the loop
// over it: the loop marks the trip (modulo 32) in a lane's mask, and
// marked_trips visits every entry of the lane's marked trips.  In the loop the
// test would hold registers for about one pair in 10^5 (lj gradient, two types:
// 114 to over 128, which spills; eam pass B 76 to 92); for the same reason the
// visit loads all it needs anew, from an index the compiler does not see through.
struct EdgeMarks {
  unsigned trips = 0, least = ~0u;
  // where a pair lies: inside the cutoff for certain?  edge pairs are noted
  __device__ __forceinline__ bool inside(double rsq, int h) {
    const int u = __double2hiint(rsq) - h;
    least = min(least, (unsigned)u);
    return u < 0;
  }
  __device__ __forceinline__ void end_trip(int tpa, int k0) {
    if (least < 2u) {
      trips |= 1u << (k0 / (4 * tpa) % 32);
      least = ~0u;
    }
  }
};
template <int TPA, bool QUAD, typename F>
__device__ __forceinline__ void marked_trips(const RowWalk<TPA, QUAD> &walk, unsigned mask, int i,
                                             const double4 *__restrict__ x, const int *__restrict__ rep,
                                             const RepGeom *__restrict__ geom, const int *__restrict__ nbr,
                                             const int *__restrict__ numneigh, int cap, F &&pair) {
  asm volatile("" : "+v"(i));
  const double4 xi = x[i];
  const RepGeom &g = geom[rep[i]];
  const int *row = nbr + (size_t)i * cap;
  const int jn = numneigh[i];
#pragma unroll 1
  while (mask) {
    const int trip = __ffs(mask) - 1;
    mask &= mask - 1;
#pragma unroll 1
    for (int k0 = walk.first() + trip * 4 * TPA; k0 < jn; k0 += 32 * 4 * TPA)
#pragma unroll 1
      for (int u = 0; u < 4; u++) {
        if (walk.at(k0, u) >= jn) continue;
        const int ent = row[walk.at(k0, u)];
        EdgePair e{i, ent, xi, gather_x(x, ent), g};
        e.rsq = nearest_rsq(e.xi, e.xj, g.prd, g.iprd, e.dx, e.dy, e.dz);
        pair(e);
      }
  }
}

// ---------------------------------------------------------------- lj/cut

// MIXED: neighbours are read from the fixed-point mirror (16 B instead of
// 32, no image decode: the wrapping difference is the minimum-image
// separation), separations rebuilt in FP64, a pair within kQBand of the
// cutoff re-tested on the FP64 positions with its image shift; FP32 pair
// arithmetic, FP64 accumulation.
template <bool MIXED, int TPA>
__global__ __launch_bounds__(1024) void k_b_lj(int n, int nt1, const double4 *__restrict__ x,
                                               const int4 *__restrict__ xq, const int *__restrict__ rep,
                                               const RepGeom *__restrict__ geom, const int *__restrict__ nbr,
                                               const int *__restrict__ numneigh, int cap,
                                               const double *__restrict__ tab, ForceOut out) {
  __shared__ double s_tab[T_N * kNT];
  __shared__ double s_qlo[MIXED ? kNT : 1], s_qhi[MIXED ? kNT : 1];
  __shared__ int s_h[MIXED ? 1 : kNT];
  __shared__ float s_f[MIXED ? 4 * kNT : 1];
  for (int k = threadIdx.x; k < T_N * kNT; k += blockDim.x) s_tab[k] = tab[k];
  if (!MIXED)
    for (int k = threadIdx.x; k < kNT; k += blockDim.x) s_h[k] = edge_word(tab[T_CUTSQ * kNT + k]);
  if (MIXED)
    for (int k = threadIdx.x; k < kNT; k += blockDim.x) {
      s_qlo[k] = tab[T_CUTSQ * kNT + k] * (1.0 - kQBand);
      s_qhi[k] = tab[T_CUTSQ * kNT + k] * (1.0 + kQBand);
      s_f[k] = (float)tab[T_LJ1 * kNT + k];
      s_f[kNT + k] = (float)tab[T_LJ2 * kNT + k];
      s_f[2 * kNT + k] = (float)tab[T_LJ3 * kNT + k];
      s_f[3 * kNT + k] = (float)tab[T_LJ4 * kNT + k];
    }
  __syncthreads();
  const int apb = blockDim.x / TPA;
  int end;
  const int b0 = chunk_begin(n, apb, &end);
  const int lane = threadIdx.x % TPA;
  const RowWalk<TPA, false> walk{lane};
  for (int base = b0; base < end; base += apb) {
    const int i = base + threadIdx.x / TPA;
    if (i >= end) continue;
    const double4 xi = x[i];
    const int ti = (int)xi.w;
    const RepGeom &g = geom[rep[i]];
    const double px = g.prd[0], py = g.prd[1], pz = g.prd[2];
    const int *row = nbr + (size_t)i * cap;
    const int jn = numneigh[i];
    double fx = 0.0, fy = 0.0, fz = 0.0, e = 0.0;
    if constexpr (MIXED) {
      // chunks of four consecutive entries per lane (one 16-B index load,
      // rows start 16-B aligned), then four 16-B gathers in flight
      const int4 qi = xq[i];
      const double q0 = g.qstep[0], q1 = g.qstep[1], q2 = g.qstep[2];
      for (int k0 = walk.first(); k0 < jn; k0 += 4 * TPA) {
        int ent[4];
        int4 qj[4];
        walk.read(row, k0, jn, i, ent);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          qj[u] = gather_q(xq, ent[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          if (walk.at(k0, u) >= jn) continue;
          const double dx = qsep(qi.x, qj[u].x, q0), dy = qsep(qi.y, qj[u].y, q1), dz = qsep(qi.z, qj[u].z, q2);
          const double rsq = dx * dx + dy * dy + dz * dz;
          const int t = ti * nt1 + qj[u].w;
          bool inside = rsq < s_qlo[t];
          if (!inside && rsq < s_qhi[t]) {
            inside = image_rsq(xi, x[ent[u] & MDX_IDX_MASK], (int)((unsigned)ent[u] >> MDX_IDX_BITS), g) <
                     s_tab[T_CUTSQ * kNT + t];
          }
          if (inside) {
            const float r2inv = __builtin_amdgcn_rcpf((float)rsq);
            const float r6inv = r2inv * r2inv * r2inv;
            const double fpair = (double)(r6inv * (s_f[t] * r6inv - s_f[kNT + t]) * r2inv);
            fx += dx * fpair;
            fy += dy * fpair;
            fz += dz * fpair;
            e += 0.5 * (double)(r6inv * (s_f[2 * kNT + t] * r6inv - s_f[3 * kNT + t]));
          }
        }
      }
    } else {
      auto add = [&](int t, double dx, double dy, double dz, double rsq) {
        const double r2inv = 1.0 / rsq;
        const double r6inv = r2inv * r2inv * r2inv;
        const double forcelj = r6inv * (s_tab[T_LJ1 * kNT + t] * r6inv - s_tab[T_LJ2 * kNT + t]);
        const double fpair = forcelj * r2inv;
        fx += dx * fpair;
        fy += dy * fpair;
        fz += dz * fpair;
        e += 0.5 * (r6inv * (s_tab[T_LJ3 * kNT + t] * r6inv - s_tab[T_LJ4 * kNT + t]));
      };
      EdgeMarks marks;
      for (int k0 = walk.first(); k0 < jn; k0 += 4 * TPA) {
        int ent[4];
        double4 xj[4];
        walk.read(row, k0, jn, i, ent);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          xj[u] = gather_x(x, ent[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          if (walk.at(k0, u) >= jn) continue;
          const double dx = nearest(xi.x - xj[u].x, px, g.iprd[0]), dy = nearest(xi.y - xj[u].y, py, g.iprd[1]),
                       dz = nearest(xi.z - xj[u].z, pz, g.iprd[2]);
          const double rsq = dx * dx + dy * dy + dz * dz;
          const int t = ti * nt1 + (int)xj[u].w;
          if (marks.inside(rsq, s_h[t])) add(t, dx, dy, dz, rsq);
        }
        marks.end_trip(TPA, k0);
      }
      if (marks.trips)
        marked_trips(walk, marks.trips, i, x, rep, geom, nbr, numneigh, cap, [&](const EdgePair &p) {
          const int t = ti * nt1 + (int)p.xj.w;
          if (p.on_edge(s_h[t]) && p.here(s_tab[T_CUTSQ * kNT + t])) add(t, p.dx, p.dy, p.dz, p.rsq);
        });
    }
    fx = gsum<TPA>(fx);
    fy = gsum<TPA>(fy);
    fz = gsum<TPA>(fz);
    e = gsum<TPA>(e);
    if (lane == 0) out.store(i, fx, fy, fz, e);
  }
}

// Parameter gradients, FP64.  A pair's gradient factor is the same in both of
// its atoms' rows, so each pair is taken once (entry j > i) with G_i - G_j;
// its sums go to the type pair (lower, higher type).  Per-block partial rows:
// [eps grad | sigma grad], nt1^2 each.
// One or two atom types: the NT(NT+1)/2 type pairs' sums stay in registers
// for the whole launch and are added up once, at its end.
template <int NT, int TPA>
__global__ __launch_bounds__(1024) void k_b_lj_vjp(int n, int nt1, const double4 *__restrict__ x,
                                                   const int *__restrict__ rep, const RepGeom *__restrict__ geom,
                                                   const int *__restrict__ nbr, const int *__restrict__ numneigh,
                                                   int cap, const double *__restrict__ tab,
                                                   const double4 *__restrict__ gin, double *__restrict__ partials) {
  constexpr bool FEW = NT <= 2;
  constexpr int NP = NT * (NT + 1) / 2;
  constexpr int NA = FEW ? NP : NT;  // sums per lane: type pairs, or the partner's types
  __shared__ int s_h[kNT];
  __shared__ double2 s_a[kNT], s_b[kNT];
  __shared__ double s_acc[FEW ? 2 * NP * 16 : 2 * kNT];
  const int cols = nt1 * nt1;
  for (int k = threadIdx.x; k < cols; k += blockDim.x) {
    s_h[k] = edge_word(tab[T_CUTSQ * kNT + k]);
    s_a[k] = make_double2(tab[T_A1 * kNT + k], tab[T_A2 * kNT + k]);
    s_b[k] = make_double2(tab[T_B1 * kNT + k], tab[T_B2 * kNT + k]);
  }
  if (!FEW)
    for (int k = threadIdx.x; k < 2 * kNT; k += blockDim.x) s_acc[k] = 0.0;
  __syncthreads();
  const int apb = blockDim.x / TPA;
  int end;
  const int b0 = chunk_begin(n, apb, &end);
  const int lane = threadIdx.x % TPA;
  const RowWalk<TPA, true> walk{lane};
  double ae[NA] = {}, as[NA] = {};
  for (int base = b0; base < end; base += apb) {
    const int i = base + threadIdx.x / TPA;
    if (i >= end) continue;
    const double4 xi = x[i];
    const double4 gi = gin[i];
    const int ti = (int)xi.w;
    const RepGeom &g = geom[rep[i]];
    const double px = g.prd[0], py = g.prd[1], pz = g.prd[2], ix = g.iprd[0], iy = g.iprd[1], iz = g.iprd[2];
    const int *row = nbr + (size_t)i * cap;
    const int jn = numneigh[i];
    auto add = [&](int tj, double a, double rsq) {  // a: (G_i - G_j) . del
      const int t = ti * nt1 + tj;
      const double r2inv = 1.0 / rsq;
      const double r6inv = r2inv * r2inv * r2inv;
      const double ar8 = a * (r2inv * r6inv);
      const double2 ca = s_a[t], cb = s_b[t];
      const double de = ca.x * r6inv - ca.y, ds = cb.x * r6inv - cb.y;
      const int slot = FEW ? ti + tj - 2 : tj - 1;  // (1,1), (1,2), (2,2), or the partner's type
#pragma unroll
      for (int c = 0; c < NA; c++)
        if (NA == 1 || slot == c) {
          ae[c] += ar8 * de;
          as[c] += ar8 * ds;
        }
    };
    EdgeMarks marks;
    for (int k0 = walk.first(); k0 < jn; k0 += 4 * TPA) {
      int ent[4];
      double4 xj[4], gj[4];
      walk.read(row, k0, jn, i, ent);
      bool any = false;
#pragma unroll
      for (int q = 0; q < 4; q++) any |= (ent[q] & MDX_IDX_MASK) > i;
      if (!any) continue;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        xj[q] = gather_x(x, ent[q]);
        gj[q] = gather_x(gin, ent[q]);
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        if ((ent[q] & MDX_IDX_MASK) <= i) continue;  // the pair's other row, or past the end
        const double dx = nearest(xi.x - xj[q].x, px, ix), dy = nearest(xi.y - xj[q].y, py, iy),
                     dz = nearest(xi.z - xj[q].z, pz, iz);
        const double rsq = dx * dx + dy * dy + dz * dz;
        const int tj = (int)xj[q].w;
        if (marks.inside(rsq, s_h[ti * nt1 + tj]))
          add(tj, (gi.x - gj[q].x) * dx + (gi.y - gj[q].y) * dy + (gi.z - gj[q].z) * dz, rsq);
      }
      marks.end_trip(TPA, k0);
    }
    if (marks.trips)
      marked_trips(walk, marks.trips, i, x, rep, geom, nbr, numneigh, cap, [&](const EdgePair &p) {
        const int tj = (int)p.xj.w, t = ti * nt1 + tj;
        if (p.first() && p.on_edge(s_h[t]))
          add(tj, p.factor(gin[p.i], gather_x(gin, p.ent), tab[T_CUTSQ * kNT + t]), p.rsq);
      });
    if constexpr (!FEW) {
#pragma unroll
      for (int c = 0; c < NA; c++)
        if (c + 1 < nt1) {
          const double se = gsum<TPA>(ae[c]), ss = gsum<TPA>(as[c]);
          if (lane == 0) {
            const int t = min(ti, c + 1) * nt1 + max(ti, c + 1);
            atomicAdd(&s_acc[t], se);
            atomicAdd(&s_acc[kNT + t], ss);
          }
          ae[c] = as[c] = 0.0;
        }
    }
  }
  double *out = partials + (size_t)blockIdx.x * 2 * cols;
  if constexpr (FEW) {
#pragma unroll
    for (int c = 0; c < NP; c++) {
      const double se = gsum<64>(ae[c]), ss = gsum<64>(as[c]);
      if ((threadIdx.x & 63) == 0) {
        s_acc[(2 * c) * 16 + (threadIdx.x >> 6)] = se;
        s_acc[(2 * c + 1) * 16 + (threadIdx.x >> 6)] = ss;
      }
    }
    __syncthreads();
    const int nw = blockDim.x >> 6;
    for (int k = threadIdx.x; k < 2 * cols; k += blockDim.x) {
      const int t = k % cols, lo = t / nt1, hi = t % nt1;
      double v = 0.0;
      if (lo >= 1 && hi >= lo) {
        const double *w = s_acc + (2 * (lo + hi - 2) + (k >= cols ? 1 : 0)) * 16;
        for (int q = 0; q < nw; q++) v += w[q];
      }
      out[k] = v;
    }
  } else {
    __syncthreads();
    for (int k = threadIdx.x; k < 2 * cols; k += blockDim.x) out[k] = s_acc[k < cols ? k : kNT + k - cols];
  }
}

// ---------------------------------------------------------------- eam

// The spline tables of the pair passes: per knot two 4-vectors, {c0,c1,c2,0}
// (derivative) and {c3,c4,c5,c6} (value), so a lookup is one or two vector
// reads.  They are copied to LDS when they fit (kTabLDS), one vector kind
// after the other; persistent grids make that once per workgroup.
template <bool MIXED>
struct Real {
  using T = double;
  using V = double4;
};
template <>
struct Real<true> {
  using T = float;
  using V = float4;
};
struct EamKnots {
  const double4 *rhor_d, *z2r_d;
  const float4 *rhor_f, *z2r_f;
};
template <bool MIXED>
__device__ __forceinline__ const typename Real<MIXED>::V *rhor_knots(const EamKnots &t) {
  if constexpr (MIXED) return t.rhor_f;
  else return t.rhor_d;
}
template <bool MIXED>
__device__ __forceinline__ const typename Real<MIXED>::V *z2r_knots(const EamKnots &t) {
  if constexpr (MIXED) return t.z2r_f;
  else return t.z2r_d;
}

template <typename T>
__device__ __forceinline__ void r_spline(const EamTab &et, T r, int &m, T &p) {
  T pp = r * (T)et.rdr + (T)1;
  m = (int)pp;
  m = min(m, et.nr - 1);
  pp -= (T)m;
  p = pp < (T)1 ? pp : (T)1;
}

// Whether the pair (i, entry) lies inside cutsq, and its separation, from the
// fixed-point mirror.
__device__ __forceinline__ bool eam_inside(const int4 &qi, int i, const double4 *__restrict__ x, const int4 &qj,
                                           const RepGeom &g, int ent, double cutsq, const double (&step)[3],
                                           double &dx, double &dy, double &dz, double &rsq) {
  dx = qsep(qi.x, qj.x, step[0]);
  dy = qsep(qi.y, qj.y, step[1]);
  dz = qsep(qi.z, qj.z, step[2]);
  rsq = dx * dx + dy * dy + dz * dz;
  if (rsq < cutsq * (1.0 - kQBand)) return true;
  if (!(rsq < cutsq * (1.0 + kQBand))) return false;
  return image_rsq(x[i], x[ent & MDX_IDX_MASK], (int)((unsigned)ent >> MDX_IDX_BITS), g) < cutsq;
}

template <bool MIXED, int TPA, bool TL>
__global__ __launch_bounds__(1024) void k_b_eam_rho(int n, const double4 *__restrict__ x,
                                                    const int4 *__restrict__ xq, const int *__restrict__ rep,
                                                    const RepGeom *__restrict__ geom, const int *__restrict__ nbr,
                                                    const int *__restrict__ numneigh, int cap, EamTab et,
                                                    EamKnots knots, const double *__restrict__ frho_d,
                                                    double *__restrict__ rho, double *__restrict__ fp,
                                                    double *__restrict__ eemb) {
  extern __shared__ double4 s_knots[];
  using T = typename Real<MIXED>::T;
  using V = typename Real<MIXED>::V;
  const V *const tab = rhor_knots<MIXED>(knots);
  V *const s_val = reinterpret_cast<V *>(s_knots);
  if constexpr (TL)
    for (int m = threadIdx.x; m <= et.nr; m += blockDim.x) s_val[m] = tab[2 * m + 1];
  __syncthreads();
  const int apb = blockDim.x / TPA;
  int end;
  const int b0 = chunk_begin(n, apb, &end);
  const int lane = threadIdx.x % TPA;
  const RowWalk<TPA, false> walk{lane};
  const int h = edge_word(et.cutsq);
  for (int base = b0; base < end; base += apb) {
    const int i = base + threadIdx.x / TPA;
    if (i >= end) continue;
    double4 xi = make_double4(0.0, 0.0, 0.0, 0.0);
    int4 qi = make_int4(0, 0, 0, 0);
    if constexpr (MIXED) qi = xq[i];
    else xi = x[i];
    const RepGeom &g = geom[rep[i]];
    double step[3], ip[3];
    for (int d = 0; d < 3; d++) {
      step[d] = MIXED ? g.qstep[d] : g.prd[d];
      ip[d] = g.iprd[d];
    }
    const int *row = nbr + (size_t)i * cap;
    const int jn = numneigh[i];
    double acc = 0.0;
    if constexpr (MIXED) {
      for (int k0 = walk.first(); k0 < jn; k0 += 4 * TPA) {
        int ent[4];
        int4 qj[4];
        walk.read(row, k0, jn, i, ent);
#pragma unroll
        for (int u = 0; u < 4; u++) qj[u] = gather_q(xq, ent[u]);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          double dx, dy, dz, rsq;
          if (walk.at(k0, u) < jn && eam_inside(qi, i, x, qj[u], g, ent[u], et.cutsq, step, dx, dy, dz, rsq)) {
            int m;
            T p;
            (void)eam_index_mixed(rsq, et.rdr, et.nr, m, p);
            const V c = TL ? s_val[m] : tab[2 * m + 1];
            acc += (double)(((c.x * p + c.y) * p + c.z) * p + c.w);
          }
        }
      }
    } else {
      auto add = [&](double rsq) {
        int m;
        double p, r, ri;
        sqrt_and_inverse(rsq, r, ri);
        r_spline<double>(et, r, m, p);
        const V c = TL ? s_val[m] : tab[2 * m + 1];
        acc += ((c.x * p + c.y) * p + c.z) * p + c.w;
      };
      EdgeMarks marks;
      for (int k0 = walk.first(); k0 < jn; k0 += 4 * TPA) {
        int ent[4];
        double4 xj[4];
        walk.read(row, k0, jn, i, ent);
#pragma unroll
        for (int u = 0; u < 4; u++) xj[u] = gather_x(x, ent[u]);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          if (walk.at(k0, u) >= jn) continue;
          double dx, dy, dz;
          const double rsq = nearest_rsq(xi, xj[u], step, ip, dx, dy, dz);
          if (marks.inside(rsq, h)) add(rsq);
        }
        marks.end_trip(TPA, k0);
      }
      if (marks.trips)
        marked_trips(walk, marks.trips, i, x, rep, geom, nbr, numneigh, cap, [&](const EdgePair &p) {
          if (p.on_edge(h) && p.here(et.cutsq)) add(p.rsq);
        });
    }
    acc = gsum<TPA>(acc);
    if (lane == 0) {
      // fp pass (pair_eam.cpp:213-228), FP64
      double p = acc * et.rdrho + 1.0;
      int m = (int)p;
      m = max(1, min(m, et.nrho - 1));
      p -= m;
      p = fmin(p, 1.0);
      const double *c = frho_d + m * 7;
      const double fpi = (c[0] * p + c[1]) * p + c[2];
      double phi = ((c[3] * p + c[4]) * p + c[5]) * p + c[6];
      if (acc > et.rhomax) phi += fpi * (acc - et.rhomax);
      rho[i] = acc;
      fp[i] = fpi;
      eemb[i] = phi;
    }
  }
}

template <bool MIXED, int TPA, bool TL>
__global__ __launch_bounds__(1024) void k_b_eam_force(int n, const double4 *__restrict__ x,
                                                      const int4 *__restrict__ xq, const int *__restrict__ rep,
                                                      const RepGeom *__restrict__ geom, const int *__restrict__ nbr,
                                                      const int *__restrict__ numneigh, int cap, EamTab et,
                                                      EamKnots knots, const double *__restrict__ fp,
                                                      const double *__restrict__ eemb, ForceOut out) {
  extern __shared__ double4 s_knots[];
  using T = typename Real<MIXED>::T;
  using V = typename Real<MIXED>::V;
  const V *const rtab = rhor_knots<MIXED>(knots), *const ztab = z2r_knots<MIXED>(knots);
  const int kn = et.nr + 1;
  V *const s_tab = reinterpret_cast<V *>(s_knots);  // rho' | z2' | z2
  if constexpr (TL)
    for (int m = threadIdx.x; m < kn; m += blockDim.x) {
      s_tab[m] = rtab[2 * m];
      s_tab[kn + m] = ztab[2 * m];
      s_tab[2 * kn + m] = ztab[2 * m + 1];
    }
  __syncthreads();
  const int apb = blockDim.x / TPA;
  int end;
  const int b0 = chunk_begin(n, apb, &end);
  const int lane = threadIdx.x % TPA;
  const RowWalk<TPA, !MIXED> walk{lane};
  const int h = edge_word(et.cutsq);
  for (int base = b0; base < end; base += apb) {
    const int i = base + threadIdx.x / TPA;
    if (i >= end) continue;
    double4 xi = make_double4(0.0, 0.0, 0.0, 0.0);
    int4 qi = make_int4(0, 0, 0, 0);
    if constexpr (MIXED) qi = xq[i];
    else xi = x[i];
    const double fpi = fp[i];
    const RepGeom &g = geom[rep[i]];
    double step[3], ip[3];
    for (int d = 0; d < 3; d++) {
      step[d] = MIXED ? g.qstep[d] : g.prd[d];
      ip[d] = g.iprd[d];
    }
    const int *row = nbr + (size_t)i * cap;
    const int jn = numneigh[i];
    double fx = 0.0, fy = 0.0, fz = 0.0, e = 0.0;
    if constexpr (MIXED) {
      for (int k0 = walk.first(); k0 < jn; k0 += 4 * TPA) {
        int ent[4];
        int4 qj[4];
        double fpj[4];
        walk.read(row, k0, jn, i, ent);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          qj[u] = gather_q(xq, ent[u]);
          fpj[u] = gather_d(fp, ent[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          double dx, dy, dz, rsq;
          if (walk.at(k0, u) < jn && eam_inside(qi, i, x, qj[u], g, ent[u], et.cutsq, step, dx, dy, dz, rsq)) {
            int m;
            T p, r, recip;
            r = eam_index_mixed(rsq, et.rdr, et.nr, m, p);
            recip = __builtin_amdgcn_rcpf(r);  // hardware reciprocal, 1 ulp
            const V rd = TL ? s_tab[m] : rtab[2 * m];
            const V zd = TL ? s_tab[kn + m] : ztab[2 * m];
            const V zv = TL ? s_tab[2 * kn + m] : ztab[2 * m + 1];
            const T rhop = (rd.x * p + rd.y) * p + rd.z;
            const T z2p = (zd.x * p + zd.y) * p + zd.z;
            const T z2 = ((zv.x * p + zv.y) * p + zv.z) * p + zv.w;
            const T phi = z2 * recip;
            const T phip = z2p * recip - phi * recip;
            const T psip = (T)fpi * rhop + (T)fpj[u] * rhop + phip;
            const double fpair = (double)(-psip * recip);
            fx += dx * fpair;
            fy += dy * fpair;
            fz += dz * fpair;
            e += 0.5 * (double)phi;
          }
        }
      }
    } else {
      auto add = [&](double fpj, double dx, double dy, double dz, double rsq) {
        int m;
        double p, r, recip;
        sqrt_and_inverse(rsq, r, recip);
        r_spline<double>(et, r, m, p);
        const V rd = TL ? s_tab[m] : rtab[2 * m];
        const V zd = TL ? s_tab[kn + m] : ztab[2 * m];
        const V zv = TL ? s_tab[2 * kn + m] : ztab[2 * m + 1];
        const double rhop = (rd.x * p + rd.y) * p + rd.z;
        const double z2p = (zd.x * p + zd.y) * p + zd.z;
        const double z2 = ((zv.x * p + zv.y) * p + zv.z) * p + zv.w;
        const double phi = z2 * recip;
        const double phip = z2p * recip - phi * recip;
        const double psip = fpi * rhop + fpj * rhop + phip;
        const double fpair = -psip * recip;
        fx += dx * fpair;
        fy += dy * fpair;
        fz += dz * fpair;
        e += 0.5 * phi;
      };
      EdgeMarks marks;
      for (int k0 = walk.first(); k0 < jn; k0 += 4 * TPA) {
        int ent[4];
        double4 xj[4];
        double fpj[4];
        walk.read(row, k0, jn, i, ent);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          xj[u] = gather_x(x, ent[u]);
          fpj[u] = gather_d(fp, ent[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          if (walk.at(k0, u) >= jn) continue;
          double dx, dy, dz;
          const double rsq = nearest_rsq(xi, xj[u], step, ip, dx, dy, dz);
          if (marks.inside(rsq, h)) add(fpj[u], dx, dy, dz, rsq);
        }
        marks.end_trip(TPA, k0);
      }
      if (marks.trips)
        marked_trips(walk, marks.trips, i, x, rep, geom, nbr, numneigh, cap, [&](const EdgePair &p) {
          if (p.on_edge(h) && p.here(et.cutsq)) add(gather_d(fp, p.ent), p.dx, p.dy, p.dz, p.rsq);
        });
    }
    fx = gsum<TPA>(fx);
    fy = gsum<TPA>(fy);
    fz = gsum<TPA>(fz);
    e = gsum<TPA>(e);
    if (lane == 0) out.store(i, fx, fy, fz, e + eemb[i]);
  }
}

// Adjoint passes, FP64.  A pair appears in both of its atoms' rows at one
// distance, so the spline terms are taken once per pair (entry j > i) with
// both rows' factors added: half the LDS atomics, which bound these passes,
// together with their conflicts (a thermalised crystal's distances fall on a
// few knots).  Each workgroup therefore keeps `copies` accumulator sets, one
// per thread modulo copies, coefficient-major (neighbouring knots in
// neighbouring banks).  Row of partials: [frho c3..c6 (nrho+1)*4 | rhor
// (nr+1)*4 | z2r (nr+1)*4] from pass A, rhor alone from pass B.
// The partner's scalar comes with a vector that is gathered anyway: fp in
// dL/dF's fourth component (pass A: read inside the j > i branch it cost a
// memory latency per pair, 367 against 329 us at 1,367,136 atoms), dL/drho
// in that of the positions pass A writes for pass B (179 against 163).
// stride of one accumulator set of `terms` coefficients: offset by 8 doubles
// modulo 32 from copy to copy
__host__ __device__ inline int adj_stride(int terms, int kn) { return (terms * kn + 31) / 32 * 32 + 8; }

template <int TPA, bool TL>
__global__ __launch_bounds__(1024) void k_b_eam_adj_a(int n, const double4 *__restrict__ x,
                                                      const int *__restrict__ rep, const RepGeom *__restrict__ geom,
                                                      const int *__restrict__ nbr, const int *__restrict__ numneigh,
                                                      int cap, EamTab et, const double4 *__restrict__ rhor,
                                                      const double *__restrict__ frho_d, const double *__restrict__ rho,
                                                      const double4 *__restrict__ gin, int copies,
                                                      double4 *__restrict__ vout,
                                                      double *__restrict__ partials) {
  extern __shared__ double4 s_knots[];
  const int kn = et.nr + 1, kf = et.nrho + 1, stride = adj_stride(7, kn);
  double4 *const s_rd = s_knots;  // TL: rho' {c0,c1,c2,0}
  double *const s_gf = reinterpret_cast<double *>(s_knots + (TL ? kn : 0)), *const s_g = s_gf + 3 * kf;
  for (int k = threadIdx.x; k < 3 * kf + copies * stride; k += blockDim.x) s_gf[k] = 0.0;
  if constexpr (TL)
    for (int m = threadIdx.x; m < kn; m += blockDim.x) s_rd[m] = rhor[2 * m];
  __syncthreads();
  double *const mine = s_g + (threadIdx.x % copies) * stride;  // z2r terms t*kn, then rhor terms (4+t)*kn
  const int apb = blockDim.x / TPA;
  int end;
  const int b0 = chunk_begin(n, apb, &end);
  const int lane = threadIdx.x % TPA;
  const RowWalk<TPA, true> walk{lane};
  const double rdr = et.rdr;
  const int h = edge_word(et.cutsq);
  for (int base = b0; base < end; base += apb) {
    const int i = base + threadIdx.x / TPA;
    if (i >= end) continue;
    const double4 xi = x[i];
    const double4 gi = gin[i];
    const RepGeom &g = geom[rep[i]];
    const double px = g.prd[0], py = g.prd[1], pz = g.prd[2], ix = g.iprd[0], iy = g.iprd[1], iz = g.iprd[2];
    const int *row = nbr + (size_t)i * cap;
    const int jn = numneigh[i];
    double u = 0.0;
    auto add = [&](bool once, double gd, double fpsum, double rsq) {  // gd: (G_i - G_j) . del
      double r, ri, p;
      int m;
      sqrt_and_inverse(rsq, r, ri);
      r_spline<double>(et, r, m, p);
      const double4 c = TL ? s_rd[m] : rhor[2 * m];
      const double b = -gd * ri;
      u += b * ((c.x * p + c.y) * p + c.z);
      if (once) {
        const double gz1 = b * ri, gz0 = -gz1 * ri, grp = b * fpsum * rdr, gzr = gz1 * rdr, pp = p * p;
        double *a = mine + m;
        atomicAdd(a, 3.0 * pp * gzr + gz0 * pp * p);
        atomicAdd(a + kn, 2.0 * p * gzr + gz0 * pp);
        atomicAdd(a + 2 * kn, gzr + gz0 * p);
        atomicAdd(a + 3 * kn, gz0);
        atomicAdd(a + 4 * kn, 3.0 * pp * grp);
        atomicAdd(a + 5 * kn, 2.0 * p * grp);
        atomicAdd(a + 6 * kn, grp);
      }
    };
    EdgeMarks marks;
    for (int k0 = walk.first(); k0 < jn; k0 += 4 * TPA) {
      int ent[4];
      double4 xj[4], gj[4];
      walk.read(row, k0, jn, i, ent);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        xj[q] = gather_x(x, ent[q]);
        gj[q] = gather_x(gin, ent[q]);
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        if (walk.at(k0, q) >= jn) continue;
        const double dx = nearest(xi.x - xj[q].x, px, ix), dy = nearest(xi.y - xj[q].y, py, iy),
                     dz = nearest(xi.z - xj[q].z, pz, iz);
        const double rsq = dx * dx + dy * dy + dz * dz;
        if (marks.inside(rsq, h))
          add((ent[q] & MDX_IDX_MASK) > i, (gi.x - gj[q].x) * dx + (gi.y - gj[q].y) * dy + (gi.z - gj[q].z) * dz,
              gi.w + gj[q].w, rsq);
      }
      marks.end_trip(TPA, k0);
    }
    if (marks.trips)
      marked_trips(walk, marks.trips, i, x, rep, geom, nbr, numneigh, cap, [&](const EdgePair &p) {
        if (!p.on_edge(h)) return;
        const double4 ga = gin[p.i], gb = gather_x(gin, p.ent);
        add(p.first(), p.factor(ga, gb, et.cutsq), ga.w + gb.w, p.rsq);
      });
    u = gsum<TPA>(u);
    if (lane == 0) {
      // fp = F'(rho_i): dL/dF'(rho_i) = u, dL/drho_i = u F''(rho_i)
      const double rhoi = rho[i];
      double p = rhoi * et.rdrho + 1.0;
      int m = (int)p;
      m = max(1, min(m, et.nrho - 1));
      p -= m;
      const bool clamped = p > 1.0;
      p = fmin(p, 1.0);
      const double rdrho = et.rdrho;
      atomicAdd(s_gf + m, u * 3.0 * p * p * rdrho);
      atomicAdd(s_gf + kf + m, u * 2.0 * p * rdrho);
      atomicAdd(s_gf + 2 * kf + m, u * rdrho);
      const double *c = frho_d + m * 7;
      const double fpp = clamped ? 0.0 : (2.0 * c[0] * p + c[1]) * rdrho;
      vout[i] = make_double4(xi.x, xi.y, xi.z, u * fpp);
    }
  }
  __syncthreads();
  const int P = 4 * kf + 8 * kn;
  double *out = partials + (size_t)blockIdx.x * P;
  for (int k = threadIdx.x; k < P; k += blockDim.x) {
    double v = 0.0;
    if (k < 4 * kf) {
      if ((k & 3) < 3) v = s_gf[(k & 3) * kf + (k >> 2)];
    } else {
      const int q = k - 4 * kf, z = q >= 4 * kn, m = (z ? q - 4 * kn : q) >> 2, t = q & 3;
      if (z || t < 3)
        for (int c = 0; c < copies; c++) v += s_g[c * stride + (z ? t : 4 + t) * kn + m];
    }
    out[k] = v;
  }
}

template <int TPA>
__global__ __launch_bounds__(1024) void k_b_eam_adj_b(int n, const double4 *__restrict__ xv,
                                                      const int *__restrict__ rep, const RepGeom *__restrict__ geom,
                                                      const int *__restrict__ nbr, const int *__restrict__ numneigh,
                                                      int cap, EamTab et, int copies,
                                                      double *__restrict__ partials) {
  extern __shared__ double4 s_knots[];
  const int kn = et.nr + 1, stride = adj_stride(4, kn);
  double *const s_g = reinterpret_cast<double *>(s_knots);
  for (int k = threadIdx.x; k < copies * stride; k += blockDim.x) s_g[k] = 0.0;
  __syncthreads();
  double *const mine = s_g + (threadIdx.x % copies) * stride;
  const int apb = blockDim.x / TPA;
  int end;
  const int b0 = chunk_begin(n, apb, &end);
  const int lane = threadIdx.x % TPA;
  const RowWalk<TPA, true> walk{lane};
  const int h = edge_word(et.cutsq);
  for (int base = b0; base < end; base += apb) {
    const int i = base + threadIdx.x / TPA;
    if (i >= end) continue;
    const double4 xi = xv[i];
    const RepGeom &g = geom[rep[i]];
    const double px = g.prd[0], py = g.prd[1], pz = g.prd[2], ix = g.iprd[0], iy = g.iprd[1], iz = g.iprd[2];
    const int *row = nbr + (size_t)i * cap;
    const int jn = numneigh[i];
    auto add = [&](double v, double rsq) {  // v: dL/drho of both atoms
      double r, ri, p;
      int m;
      sqrt_and_inverse(rsq, r, ri);
      r_spline<double>(et, r, m, p);
      double *a = mine + m;
      atomicAdd(a, v * p * p * p);
      atomicAdd(a + kn, v * p * p);
      atomicAdd(a + 2 * kn, v * p);
      atomicAdd(a + 3 * kn, v);
    };
    EdgeMarks marks;
    for (int k0 = walk.first(); k0 < jn; k0 += 4 * TPA) {
      int ent[4];
      double4 xj[4];
      walk.read(row, k0, jn, i, ent);
      bool any = false;
#pragma unroll
      for (int q = 0; q < 4; q++) any |= (ent[q] & MDX_IDX_MASK) > i;
      if (!any) continue;
#pragma unroll
      for (int q = 0; q < 4; q++) xj[q] = gather_x(xv, ent[q]);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        if ((ent[q] & MDX_IDX_MASK) <= i) continue;  // the pair's other row, or past the end
        const double dx = nearest(xi.x - xj[q].x, px, ix), dy = nearest(xi.y - xj[q].y, py, iy),
                     dz = nearest(xi.z - xj[q].z, pz, iz);
        const double rsq = dx * dx + dy * dy + dz * dz;
        const double v = xi.w + xj[q].w;
        if (marks.inside(rsq, h) && v != 0.0) add(v, rsq);
      }
      marks.end_trip(TPA, k0);
    }
    if (marks.trips)
      marked_trips(walk, marks.trips, i, xv, rep, geom, nbr, numneigh, cap, [&](const EdgePair &p) {
        if (!p.first() || !p.on_edge(h)) return;
        const double v = (p.here(et.cutsq) ? p.xi.w : 0.0) + (p.there(et.cutsq) ? p.xj.w : 0.0);
        if (v != 0.0) add(v, p.rsq);
      });
  }
  __syncthreads();
  double *out = partials + (size_t)blockIdx.x * 4 * kn;
  for (int k = threadIdx.x; k < 4 * kn; k += blockDim.x) {
    double v = 0.0;
    for (int c = 0; c < copies; c++) v += s_g[c * stride + (k & 3) * kn + (k >> 2)];
    out[k] = v;
  }
}

// ---------------------------------------------------------------- utilities

// Column sums of the per-block partial rows, in two fixed-order passes
// (deterministic): k_b_colsum_chunks sums chunk ry of the rows (rows
// [rows*ry/nchunk, rows*(ry+1)/nchunk)) for 64 columns per block, four row
// lanes per column combined in LDS; k_b_colsum then sums the nchunk chunk
// rows the same way, into mapped host memory.  A second set of rows (partB)
// covers colsB columns from c0B on.
constexpr int kColChunks = 64;
__device__ __forceinline__ void colsum_store(double (&s)[4][64], double acc, int c, int cols, double *out) {
  const int l = threadIdx.x & 63, sub = threadIdx.x >> 6;
  s[sub][l] = acc;
  __syncthreads();
  if (sub == 0 && c < cols) out[c] = ((s[0][l] + s[1][l]) + s[2][l]) + s[3][l];
}
__global__ __launch_bounds__(256) void k_b_colsum_chunks(const double *__restrict__ part, int rows, int cols,
                                                         const double *__restrict__ partB, int rowsB, int c0B,
                                                         int colsB, double *__restrict__ mid) {
  __shared__ double s[4][64];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63), sub = threadIdx.x >> 6;
  const int ry = blockIdx.y, nchunk = gridDim.y;
  double acc = 0.0;
  if (c < cols) {
    const int r0 = (int)((long)rows * ry / nchunk), r1 = (int)((long)rows * (ry + 1) / nchunk);
    for (int r = r0 + sub; r < r1; r += 4) acc += part[(size_t)r * cols + c];
  }
  const int cb = c - c0B;
  if (cb >= 0 && cb < colsB) {
    const int r0 = (int)((long)rowsB * ry / nchunk), r1 = (int)((long)rowsB * (ry + 1) / nchunk);
    for (int r = r0 + sub; r < r1; r += 4) acc += partB[(size_t)r * colsB + cb];
  }
  colsum_store(s, acc, c, cols, mid + (size_t)ry * cols);
}
__global__ __launch_bounds__(256) void k_b_colsum(const double *__restrict__ mid, int rows, int cols,
                                                  double *__restrict__ out) {
  __shared__ double s[4][64];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63);
  double acc = 0.0;
  if (c < cols)
#pragma unroll 4
    for (int r = threadIdx.x >> 6; r < rows; r += 4) acc += mid[(size_t)r * cols + c];
  colsum_store(s, acc, c, cols, out);
}

// per-replica energy: one block per replica, fixed-order tree
__global__ void k_b_rep_energy(const double *__restrict__ e, const int *__restrict__ off, double *__restrict__ out) {
  __shared__ double s[256];
  const int r = blockIdx.x;
  double acc = 0.0;
  for (int i = off[r] + threadIdx.x; i < off[r + 1]; i += 256) acc += e[i];
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (threadIdx.x < h) s[threadIdx.x] += s[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[r] = s[0];
}

__global__ void k_b_gather_s(int n, const int *__restrict__ inv, const double *__restrict__ a, double *__restrict__ out) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < n) out[c] = a[inv[c]];
}

// dL/dF in sorted order, with a per-atom value w (null: 0) beside it
__global__ void k_b_scatter_g(int n, const int *__restrict__ inv, const double *__restrict__ gin,
                              const double *__restrict__ w, double4 *__restrict__ g) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const int i = inv[c];
  g[i] = make_double4(gin[3 * (size_t)c], gin[3 * (size_t)c + 1], gin[3 * (size_t)c + 2], w ? w[i] : 0.0);
}

}  // namespace
}  // namespace mdx

using namespace mdx;

struct mdx_batch {
  int device = 0;
  hipStream_t stream = nullptr;      // where the batch's work goes: own_stream or the caller's
  hipStream_t own_stream = nullptr;  // created with the batch
  int nrep = 0, ntypes = 0, n = 0, precision = MDX_FP64;
  double skin = 0.0;
  std::vector<int> natoms, off;
  std::vector<RepGeom> geom_h;
  RepGeom *geom = nullptr;
  int *off_d = nullptr;
  int total_bins = 0, count_cap = 0, start_cap = 0;  // bins; elements of bin_count, bin_start
  double cutneigh = 0.0;  // of the current bins/list
  bool positions = false, built = false;
  // atoms
  double *xin = nullptr;  // caller order staging [N][3]
  int *type_c = nullptr, *rep_c = nullptr;
  double4 *xw = nullptr, *x = nullptr, *g = nullptr;
  double *eat = nullptr;       // per-atom energies of the last force pass
  double *rep_host = nullptr;  // mapped: replica energies
  int4 *xq = nullptr;  // fixed-point copy of x (mixed-precision force passes)
  int *rep = nullptr, *orig = nullptr, *inv = nullptr;
  unsigned *key = nullptr;
  int *slot = nullptr, *order = nullptr;  // arrival slots; atoms by bin in arrival order
  int *bin_count = nullptr, *bin_start = nullptr;
  char *scan_tmp = nullptr;
  size_t scan_bytes = 0;
  int *nbr = nullptr, *numneigh = nullptr;
  int cap = 0;
  int *dflags = nullptr;       // kFlagWords: [0] max count, [4] outside box, [7] NaN, [8..9] u64 total
  int *flags_host = nullptr;   // mapped copy of the first kFlagInts
  int flag_serial = 0;         // list passes whose flags were asked for (kFlagSerial)
  bool mirror_ok = false;      // the fixed-point mirror can decide the list's candidates
  long total_neighbors = 0;
  int max_neighbors = 0;
  double *staging = nullptr;  // [N][3] output staging
  double *rho = nullptr, *fp = nullptr, *eemb = nullptr;
  double4 *vadj = nullptr;  // positions with dL/drho beside them
  double *partials = nullptr;
  size_t partials_cap = 0;  // doubles
  double *colsum = nullptr;
  size_t colsum_cap = 0;
  double *sums_host = nullptr;  // mapped: the column sums
  size_t sums_cap = 0;
  // pair
  int pair = MDX_PAIR_NONE;
  double *ljtab = nullptr;  // T_N * kNT
  double lj_cutmax = 0.0;
  std::vector<double> lj_tab;  // the table last uploaded (a repeated init uploads nothing)
  EamTab et{};
  double *frho_d = nullptr;
  EamKnots knots{};             // packed rhor and z2r (into knots_d, knots_f)
  double4 *knots_d = nullptr;
  float4 *knots_f = nullptr;
  std::vector<double> eam_knots[3];
  double eam_drho = 0.0, eam_dr = 0.0, eam_cut = 0.0;
  int eam_rho_prec = -1;  // precision of the rho/fp on the device for the current positions and tables (-1: stale)
  // tuning / timing
  Tune tune[MDX_BK_NKIND];
  bool autotune = false;
  bool tuned[MDX_BK_NKIND] = {false};
  double kms[MDX_BK_NKIND] = {0};
  long klaunch[MDX_BK_NKIND] = {0};
  int num_cu = 256;
  // start and stop events of the launches not yet added to kms (read when the
  // times are asked for, or when the ring is full)
  struct Launched {
    hipEvent_t a, b;
    int kind;
  };
  std::vector<Launched> ring;
  size_t pending = 0;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;  // of the launch being queued
  int lds_max = 65536;
};

namespace {

int bfail(hipError_t e, const char *what) { return hip_fail(e, what); }

template <typename P>
int dalloc(P **p, size_t count) {
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  if (count == 0) count = 1;
  hipError_t e = hipMalloc((void **)p, count * sizeof(P));
  return e == hipSuccess ? MDX_OK : bfail(e, "batch allocation");
}

// *p holds at least `count` elements when this returns MDX_OK.  The capacity
// is 0 while there is no array: after a failed allocation the next call tries
// again, whatever it asks for.
template <typename P, typename C>
int grow(P **p, C *cap, size_t count) {
  if (*p && count <= (size_t)*cap) return MDX_OK;
  *cap = 0;
  const int rc = dalloc(p, count);
  if (!rc) *cap = (C)count;
  return rc;
}

bool is_device_ptr(const void *p, int device) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type == hipMemoryTypeDevice && a.device == device;
}

int check_b(mdx_batch *b) {
  if (!b) {
    set_error("null batch");
    return MDX_ERR_ARG;
  }
  hipError_t e = hipSetDevice(b->device);
  return e == hipSuccess ? MDX_OK : bfail(e, "hipSetDevice");
}

// The launch shape of a kernel kind that was neither set nor tuned.  A grid
// of as many workgroups as the chip holds at once (512 threads, two per CU)
// lets each copy its tables to LDS once and loop; four lanes per atom read a
// row in whole 64-B pieces and waste the least.  Small batches take more
// lanes per atom, as one launch is then one chain of loads.  Measured (us):
//   eam 1.37 M atoms, one workgroup of 256 at 8 lanes per tile (the former
//   default) against this: rho 347 / 156, force 538 / 198, FP64 rho 435 / 196,
//   adjoint 525 / 414 and 256 / 188; lj 512,000 atoms: forces 111 / 85 mixed,
//   134 / 118 FP64, gradient 192 / 158
//   at 4 / 16 lanes: eam 3,164 atoms rho 12.7 / 7.9, adjoint 29 / 15.5, 22,401
//   atoms 9.5 / 12.3 and 22.7 / 25.3; lj 21,952 atoms 21.5 / 17.6, 101,250
//   atoms 35 / 46; 16 / 32 lanes: lj 4,000 atoms 10.4 / 9.5
Tune default_tune(const mdx_batch *b, int kind) {
  Tune t;
  const bool lj = kind == MDX_BK_LJ || kind == MDX_BK_LJ_VJP;
  const bool large = b->n > (lj ? 50000 : 10000);
  t.tpa = large ? 4 : lj && b->n <= 10000 ? 32 : 16;
  t.block = large ? 512 : 256;
  t.grid = (large ? 2 : 4) * b->num_cu;
  return t;
}

// the list build's own shape, whatever is set for its kind
Tune build_tune(int n) {
  constexpr int per = kBuildBlock / kBuildLanes;
  Tune t;
  t.block = kBuildBlock;
  t.tpa = kBuildLanes;
  t.grid = std::min(xcd_grid((n + per - 1) / per), kBuildGrid);
  return t;
}

Tune tune_of(const mdx_batch *b, int kind) {
  if (kind == MDX_BK_BUILD) return build_tune(b->n);
  return b->tune[kind].tpa ? b->tune[kind] : default_tune(b, kind);
}

// adds the times of the launches since the last call to kms; waits for them
int resolve_times(mdx_batch *b) {
  if (b->pending == 0) return MDX_OK;
  hipError_t e = hipEventSynchronize(b->ring[b->pending - 1].b);
  if (e != hipSuccess) return bfail(e, "batch kernel");
  for (size_t k = 0; k < b->pending; k++) {
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, b->ring[k].a, b->ring[k].b);
    b->kms[b->ring[k].kind] += ms;
  }
  b->pending = 0;
  return MDX_OK;
}

// A launch whose own start and stop times go to the events b->ev0 and ev1:
// they come with the dispatch, so nothing is queued around it and the host
// does not wait for it (two recorded events and a wait per kernel cost a
// 64 x 8,000 atom loss and gradient about 100 us).
#define BATCH_LAUNCH(KERNEL, G, B, LDS, ...) \
  hipExtLaunchKernelGGL(KERNEL, dim3(G), dim3(B), LDS, b->stream, b->ev0, b->ev1, 0, __VA_ARGS__)

// run one launch of kind `kind` under timing; `launch(tune)` enqueues it.
// With ms_out it is waited for and timed on its own, else it is queued.
constexpr size_t kRing = 64;
template <typename F>
int timed(mdx_batch *b, int kind, const Tune &t, F &&launch, float *ms_out = nullptr) {
  int rc;
  hipError_t e;
  if (b->pending == kRing && (rc = resolve_times(b))) return rc;
  if (b->ring.size() == b->pending) {
    mdx_batch::Launched l{};
    if ((e = hipEventCreate(&l.a)) != hipSuccess) return bfail(e, "batch events");
    if ((e = hipEventCreate(&l.b)) != hipSuccess) {
      (void)hipEventDestroy(l.a);
      return bfail(e, "batch events");
    }
    b->ring.push_back(l);
  }
  mdx_batch::Launched &l = b->ring[b->pending];
  l.kind = kind;
  b->ev0 = l.a;
  b->ev1 = l.b;
  launch(t);
  if ((e = hipGetLastError()) != hipSuccess) return bfail(e, "batch kernel launch");
  if (ms_out) {
    if ((e = hipEventSynchronize(l.b)) != hipSuccess) return bfail(e, "batch kernel");
    (void)hipEventElapsedTime(ms_out, l.a, l.b);
    return MDX_OK;
  }
  b->pending++;
  b->klaunch[kind]++;
  return MDX_OK;
}

int finish(mdx_batch *b, const char *what) {
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(b->stream);
  return e == hipSuccess ? MDX_OK : bfail(e, what);
}

// kernels that flush per-block partial rows cap the grid at kPartialBlocksPerCU per CU
constexpr int kPartialBlocksPerCU = 8;
constexpr size_t kAdjLDS = 20480;  // LDS per workgroup of the eam adjoint with small tables
int persistent_grid(mdx_batch *b, const Tune &t, bool partial_rows = false) {
  const int apb = t.block / t.tpa;
  const long tiles = (b->n + apb - 1) / apb;
  long G = t.grid > 0 ? t.grid : tiles;
  G = std::max<long>(1, std::min<long>(G, tiles));
  if (partial_rows) G = std::min<long>(G, (long)kPartialBlocksPerCU * b->num_cu);
  if (G >= kXCD) G = (G / kXCD) * kXCD;
  return (int)G;
}

// candidates for the autotuner, 2 to 16 lanes per atom: the default first
// where it is one of them (lj above 10,000 atoms, eam always), which the others
// have to beat
std::vector<Tune> candidates(const mdx_batch *b, int kind) {
  std::vector<Tune> v;
  const Tune dflt = default_tune(b, kind);
  if (dflt.tpa <= 16) v.push_back(dflt);
  for (int tpa : {2, 4, 8, 16})
    for (int block : {128, 256, 512})
      for (int per_cu : {2, 4, 8, 0}) {
        Tune t;
        t.tpa = tpa;
        t.block = block;
        t.grid = per_cu ? per_cu * b->num_cu : 0;
        v.push_back(t);
      }
  return v;
}

// runs kind with the current tune, or tunes first when asked; the last run
// uses the chosen shape so its results are the call's results
template <typename F>
int run_kind(mdx_batch *b, int kind, F &&launch) {
  if (b->autotune && !b->tuned[kind]) {
    float best = 1e30f;
    Tune bt = tune_of(b, kind);
    for (const Tune &t : candidates(b, kind)) {
      float ms = 0.0f;
      for (int rep = 0; rep < 2; rep++) {  // second timing counts (warm caches)
        int rc = timed(b, kind, t, launch, &ms);
        if (rc) return rc;
      }
      if (ms < best) {
        best = ms;
        bt = t;
      }
    }
    b->tune[kind] = bt;
    b->tuned[kind] = true;
  }
  return timed(b, kind, tune_of(b, kind), launch);
}

#define TPA_DISPATCH(tpa, CALL)                      \
  switch (tpa) {                                     \
    case 1: { constexpr int TP = 1; CALL; } break;   \
    case 2: { constexpr int TP = 2; CALL; } break;   \
    case 4: { constexpr int TP = 4; CALL; } break;   \
    case 8: { constexpr int TP = 8; CALL; } break;   \
    case 16: { constexpr int TP = 16; CALL; } break; \
    case 32: { constexpr int TP = 32; CALL; } break; \
    default: { constexpr int TP = 64; CALL; } break; \
  }

// column sums of `rows` partial rows (and rowsB rows of colsB columns at partB,
// into the columns from c0B on), left in b->sums_host when this returns
int colsum(mdx_batch *b, int rows, int cols, const double *partB = nullptr, int rowsB = 0, int c0B = 0, int colsB = 0) {
  int rc = grow(&b->colsum, &b->colsum_cap, (size_t)kColChunks * cols);
  if (rc) return rc;
  if ((size_t)cols > b->sums_cap) {
    if (b->sums_host) (void)hipHostFree(b->sums_host);
    b->sums_host = nullptr;
    b->sums_cap = 0;
    hipError_t e = hipHostMalloc(&b->sums_host, sizeof(double) * cols, hipHostMallocCoherent | hipHostMallocMapped);
    if (e != hipSuccess) return bfail(e, "gradient buffer");
    b->sums_cap = cols;
  }
  const int nchunk = std::max(1, std::min(kColChunks, std::max(rows, rowsB)));
  hipLaunchKernelGGL(k_b_colsum_chunks, dim3((cols + 63) / 64, nchunk), dim3(256), 0, b->stream, b->partials, rows,
                     cols, partB, rowsB, c0B, colsB, b->colsum);
  hipLaunchKernelGGL(k_b_colsum, dim3((cols + 63) / 64), dim3(256), 0, b->stream, b->colsum, nchunk, cols,
                     b->sums_host);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(b->stream);
  return e == hipSuccess ? MDX_OK : bfail(e, "gradient reduction");
}

double pair_cutmax(mdx_batch *b) {
  if (b->pair == MDX_PAIR_LJ) return b->lj_cutmax;
  if (b->pair == MDX_PAIR_EAM) return b->eam_cut;
  return 0.0;
}

// bins for cutneigh, then wrap/sort/permute/list
int build(mdx_batch *b) {
  if (!b->positions) {
    set_error("positions not set (mdx_batch_set_positions)");
    return MDX_ERR_ARG;
  }
  const double cutneigh = pair_cutmax(b) + b->skin;
  if (!(cutneigh > 0)) {
    set_error("no pair style set");
    return MDX_ERR_ARG;
  }
  int rc;
  hipError_t e;
  b->built = false;  // a failed build leaves no list
  if (cutneigh != b->cutneigh) {
    b->cutneigh = 0.0;  // until the bins for it are there
    const double binsize = 0.5 * cutneigh;
    long total = 0;
    for (int r = 0; r < b->nrep; r++) {
      RepGeom &g = b->geom_h[r];
      for (int d = 0; d < 3; d++) {
        if (g.periodic[d] && g.prd[d] < 2.0 * cutneigh) {
          set_error("a periodic replica box is shorter than twice the neighbour cutoff");
          return MDX_ERR_ARG;
        }
        int nb = (int)std::floor(g.prd[d] / binsize);
        nb = std::max(1, std::min(nb, 1024));
        g.nbin[d] = nb;
        g.bininv[d] = nb / g.prd[d];
      }
      g.bin_off = (int)total;
      total += (long)g.nbin[0] * g.nbin[1] * g.nbin[2];
      if (total >= (1l << 30)) {
        set_error("too many bins over all replicas");
        return MDX_ERR_ARG;
      }
    }
    b->total_bins = (int)total;
    if ((e = hipMemcpy(b->geom, b->geom_h.data(), sizeof(RepGeom) * b->nrep, hipMemcpyHostToDevice)) != hipSuccess)
      return bfail(e, "replica geometry upload");
    if ((rc = grow(&b->bin_count, &b->count_cap, b->total_bins + 1)) ||
        (rc = grow(&b->bin_start, &b->start_cap, b->total_bins + 1)))
      return rc;
    // list candidates are decided on the mirror where its rounding stays well
    // inside the re-test band and the wrapping difference is a candidate's own
    // image (no atom in a stencil under two images)
    b->mirror_ok = true;
    for (const RepGeom &g : b->geom_h)
      for (int d = 0; d < 3; d++)
        if (2.0 * std::sqrt(3.0) * g.qstep[d] > 5e-7 * cutneigh || (g.periodic[d] && 2 * kS + 1 > g.nbin[d]))
          b->mirror_ok = false;
    size_t need = 0;
    (void)hipcub::DeviceScan::ExclusiveSum(nullptr, need, b->bin_count, b->bin_start, b->total_bins + 1,
                                           b->stream);
    if ((rc = grow(&b->scan_tmp, &b->scan_bytes, need))) return rc;
    b->cutneigh = cutneigh;
  }
  const int n = b->n;
  if ((e = hipMemsetAsync(b->bin_count, 0, sizeof(int) * (b->total_bins + 1), b->stream)) != hipSuccess ||
      (e = hipMemsetAsync(b->dflags, 0, sizeof(int) * kFlagWords, b->stream)) != hipSuccess)
    return bfail(e, "build flags");
  hipLaunchKernelGGL(k_b_load, dim3((n + 255) / 256), dim3(256), 0, b->stream, n, b->xin, b->type_c, b->rep_c,
                     b->geom, b->xw, b->key, b->slot, b->bin_count, b->dflags);
  size_t scb = b->scan_bytes;
  if ((e = hipcub::DeviceScan::ExclusiveSum(b->scan_tmp, scb, b->bin_count, b->bin_start, b->total_bins + 1,
                                            b->stream)) != hipSuccess)
    return bfail(e, "bin scan");
  hipLaunchKernelGGL(k_b_scatter, dim3((n + 255) / 256), dim3(256), 0, b->stream, n, b->key, b->slot, b->bin_start,
                     b->order);
  hipLaunchKernelGGL(k_b_rank_permute, dim3((n + 255) / 256), dim3(256), 0, b->stream, n, b->order, b->key,
                     b->bin_start, b->xw, b->rep_c, b->geom, b->x, b->xq, b->rep, b->orig, b->inv);
  auto alloc_rows = [&](int cap) {  // cap stays 0 without a list
    b->cap = 0;
    rc = dalloc(&b->nbr, (size_t)cap * n);
    if (!rc) b->cap = cap;
    return rc;
  };
  if (b->cap == 0 && alloc_rows(96)) return rc;
  const double cutneighsq = cutneigh * cutneigh;
  const float c_lo = (float)(cutneighsq * (1.0 - kBuildBand)), c_hi = (float)(cutneighsq * (1.0 + kBuildBand)),
              reach = (float)(cutneighsq * (1.0 + 1e-4));
  bool mirror = b->mirror_ok;
  for (int attempt = 0; attempt < 5; attempt++) {
    if (attempt > 0 &&
        (e = hipMemsetAsync(b->dflags + kFlagInts, 0, sizeof(ListSlot) * kListSlots, b->stream)) != hipSuccess)
      return bfail(e, "build flags");
    auto launch = [&](const Tune &t) {
      const int G = t.grid;
      auto go = [&](auto kernel) {
        BATCH_LAUNCH(kernel, G, kBuildBlock, 0, n, b->x, b->xq, b->rep, b->geom, b->bin_start, cutneighsq, c_lo, c_hi,
                     reach, b->cap, b->nbr, b->numneigh, reinterpret_cast<ListSlot *>(b->dflags + kFlagInts));
      };
      if (mirror) go(k_b_build<true>);
      else go(k_b_build<false>);
    };
    if ((rc = timed(b, MDX_BK_BUILD, build_tune(n), launch))) return rc;
    b->flag_serial = b->flag_serial == 0x7fffffff ? 1 : b->flag_serial + 1;
    launch_build_flags(b->stream, b->dflags, b->flags_host, b->flag_serial);
    int fl[kFlagInts], got;
    if ((rc = wait_word(b->stream, b->flags_host + kFlagSerial, b->flag_serial, b->flag_serial, &got))) return rc;
    std::memcpy(fl, b->flags_host, sizeof(fl));
    if (fl[4]) {
      set_error("an atom lies outside its replica's box in a non-periodic dimension");
      return MDX_ERR_ARG;
    }
    if (fl[7] && mirror) {  // a coordinate is not a number: FP64 candidates, which reject its pairs
      mirror = false;
      continue;
    }
    if (fl[0] <= b->cap) {
      unsigned long long tot;
      std::memcpy(&tot, fl + 8, sizeof(tot));
      b->total_neighbors = (long)tot;
      b->max_neighbors = fl[0];
      b->built = true;
      b->eam_rho_prec = -1;
      return MDX_OK;
    }
    if (alloc_rows((fl[0] + 16 + 15) / 16 * 16)) return rc;
  }
  set_error("neighbour list capacity did not converge");
  return MDX_ERR_OVERFLOW;
}

int ensure_built(mdx_batch *b) {
  const double cutneigh = pair_cutmax(b) + b->skin;
  if (b->built && cutneigh == b->cutneigh) return MDX_OK;
  return build(b);
}

// where a force pass writes: the caller's device array, or staging for a host one
ForceOut force_out(mdx_batch *b, double *f) {
  return {b->eat, !f ? nullptr : is_device_ptr(f, b->device) ? f : b->staging, b->orig};
}

// what follows a force pass: replica energies, the copy to a host force array,
// and the wait for both (the list build, when there was one, has waited for its flags)
int force_results(mdx_batch *b, const ForceOut &out, double *f, double *energy) {
  if (energy)
    hipLaunchKernelGGL(k_b_rep_energy, dim3(b->nrep), dim3(256), 0, b->stream, b->eat, b->off_d, b->rep_host);
  if (f && out.f != f) {
    hipError_t e = hipMemcpyAsync(f, out.f, sizeof(double) * 3 * b->n, hipMemcpyDeviceToHost, b->stream);
    if (e != hipSuccess) return bfail(e, "force output");
  }
  int rc = finish(b, "batch forces");
  if (!rc && energy) std::memcpy(energy, b->rep_host, sizeof(double) * b->nrep);
  return rc;
}

int read_g(mdx_batch *b, const double *gf, const double *w = nullptr) {
  const int n = b->n;
  const double *src = gf;
  hipError_t e;
  if (!is_device_ptr(gf, b->device)) {
    if ((e = hipMemcpyAsync(b->staging, gf, sizeof(double) * 3 * n, hipMemcpyHostToDevice, b->stream)) !=
        hipSuccess)
      return bfail(e, "dL/dF upload");
    src = b->staging;
  }
  hipLaunchKernelGGL(k_b_scatter_g, dim3((n + 255) / 256), dim3(256), 0, b->stream, n, b->inv, src, w, b->g);
  return MDX_OK;
}

// transpose of the knot -> (c3..c6) map of the spline construction
// (pair_eam.cpp:723-751): g_knot[k] = sum_m,t gc[m][t] * d coeff_t(m) / d knot_k
void spline_coeffs(int n, const double *f /* [n] */, double *c /* (n+1)*4: c3..c6 */) {
  std::vector<double> c5(n + 1, 0.0);
  auto F = [&](int m) { return f[m - 1]; };
  c5[1] = F(2) - F(1);
  c5[2] = 0.5 * (F(3) - F(1));
  c5[n - 1] = 0.5 * (F(n) - F(n - 2));
  c5[n] = F(n) - F(n - 1);
  for (int m = 3; m <= n - 2; m++) c5[m] = ((F(m - 2) - F(m + 2)) + 8.0 * (F(m + 1) - F(m - 1))) / 12.0;
  for (int t = 0; t < 4 * (n + 1); t++) c[t] = 0.0;
  for (int m = 1; m <= n; m++) {
    c[4 * m + 2] = c5[m];
    c[4 * m + 3] = F(m);
  }
  for (int m = 1; m <= n - 1; m++) {
    c[4 * m + 1] = 3.0 * (F(m + 1) - F(m)) - 2.0 * c5[m] - c5[m + 1];
    c[4 * m + 0] = c5[m] + c5[m + 1] - 2.0 * (F(m + 1) - F(m));
  }
}

// dL/d(knots) from dL/d(c3..c6): the transpose of spline_coeffs, one sweep
void knot_gradient(int n, const double *gc, double *g) {
  std::vector<double> gk(n + 1, 0.0), g5(n + 1, 0.0);  // by knot 1..n: F and c5
  for (int m = 1; m <= n; m++) {
    g5[m] += gc[4 * m + 2];
    gk[m] += gc[4 * m + 3];
  }
  for (int m = 1; m <= n - 1; m++) {
    const double a = gc[4 * m], b = gc[4 * m + 1];
    gk[m + 1] += 3.0 * b - 2.0 * a;
    gk[m] -= 3.0 * b - 2.0 * a;
    g5[m] += a - 2.0 * b;
    g5[m + 1] += a - b;
  }
  gk[2] += g5[1];
  gk[1] -= g5[1];
  gk[3] += 0.5 * g5[2];
  gk[1] -= 0.5 * g5[2];
  gk[n] += 0.5 * g5[n - 1];
  gk[n - 2] -= 0.5 * g5[n - 1];
  gk[n] += g5[n];
  gk[n - 1] -= g5[n];
  for (int m = 3; m <= n - 2; m++) {
    const double q = g5[m] / 12.0;
    gk[m - 2] += q;
    gk[m + 2] -= q;
    gk[m + 1] += 8.0 * q;
    gk[m - 1] -= 8.0 * q;
  }
  for (int k = 0; k < n; k++) g[k] = gk[k + 1];
}

// full 7-coefficient table from knots (host copy uploaded to the device)
void spline7(int n, double delta, const double *f, std::vector<double> &sp) {
  std::vector<double> c(4 * (n + 1));
  spline_coeffs(n, f, c.data());
  sp.assign(7 * (n + 1), 0.0);
  for (int m = 1; m <= n; m++) {
    sp[7 * m + 3] = c[4 * m + 0];
    sp[7 * m + 4] = c[4 * m + 1];
    sp[7 * m + 5] = c[4 * m + 2];
    sp[7 * m + 6] = c[4 * m + 3];
    sp[7 * m + 2] = sp[7 * m + 5] / delta;
    sp[7 * m + 1] = 2.0 * sp[7 * m + 4] / delta;
    sp[7 * m + 0] = 3.0 * sp[7 * m + 3] / delta;
  }
}

int upload(void *dst, const void *src, size_t bytes) {
  hipError_t e = hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
  return e == hipSuccess ? MDX_OK : bfail(e, "table upload");
}

}  // namespace

extern "C" {

int mdx_batch_create(int device, int nrep, const int *natoms, const double *lo, const double *hi,
                     const int *periodic, int ntypes, const int *type, mdx_batch **out) {
  if (!out || nrep <= 0 || !natoms || !lo || !hi || !periodic || !type || ntypes < 1 || ntypes > MDX_MAXT) {
    set_error("mdx_batch_create: invalid arguments (nrep > 0, 1 <= ntypes <= 8)");
    return MDX_ERR_ARG;
  }
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) {
    (void)hipGetLastError();
    set_error("no HIP device available");
    return MDX_ERR_HIP;
  }
  long total = 0;
  for (int r = 0; r < nrep; r++) {
    if (natoms[r] < 0) {
      set_error("negative replica size");
      return MDX_ERR_ARG;
    }
    total += natoms[r];
    for (int d = 0; d < 3; d++)
      if (!(hi[3 * r + d] > lo[3 * r + d])) {
        set_error("empty replica box");
        return MDX_ERR_ARG;
      }
  }
  if (total <= 0 || total >= (1l << MDX_IDX_BITS)) {
    set_error("total atoms must be in [1, 2^27)");
    return MDX_ERR_ARG;
  }
  for (long i = 0; i < total; i++)
    if (type[i] < 1 || type[i] > ntypes) {
      set_error("atom type out of range");
      return MDX_ERR_ARG;
    }
  mdx_batch *b = new mdx_batch();
  b->device = device;
  b->nrep = nrep;
  b->ntypes = ntypes;
  b->n = (int)total;
  b->natoms.assign(natoms, natoms + nrep);
  b->off.assign(nrep + 1, 0);
  for (int r = 0; r < nrep; r++) b->off[r + 1] = b->off[r] + natoms[r];
  b->geom_h.assign(nrep, RepGeom{});
  for (int r = 0; r < nrep; r++)
    for (int d = 0; d < 3; d++) {
      b->geom_h[r].lo[d] = lo[3 * r + d];
      b->geom_h[r].prd[d] = hi[3 * r + d] - lo[3 * r + d];
      b->geom_h[r].periodic[d] = periodic[3 * r + d] ? 1 : 0;
      b->geom_h[r].nbin[d] = 1;
      b->geom_h[r].bininv[d] = 1.0 / b->geom_h[r].prd[d];
      const double span = periodic[3 * r + d] ? 4294967296.0 : 1073741824.0;
      b->geom_h[r].qscale[d] = span / b->geom_h[r].prd[d];
      b->geom_h[r].qstep[d] = b->geom_h[r].prd[d] / span;
      b->geom_h[r].iprd[d] = periodic[3 * r + d] ? 1.0 / b->geom_h[r].prd[d] : 0.0;
    }
  hipError_t e;
  int rc;
  if ((e = hipSetDevice(device)) != hipSuccess || (e = hipStreamCreate(&b->own_stream)) != hipSuccess ||
      (e = hipHostMalloc(&b->flags_host, sizeof(int) * kFlagInts, hipHostMallocCoherent | hipHostMallocMapped)) !=
          hipSuccess ||
      (e = hipHostMalloc(&b->rep_host, sizeof(double) * nrep, hipHostMallocCoherent | hipHostMallocMapped)) !=
          hipSuccess) {
    rc = bfail(e, "batch stream");
    mdx_batch_destroy(b);
    return rc;
  }
  std::memset(b->flags_host, 0, sizeof(int) * kFlagInts);  // no serial yet
  b->stream = b->own_stream;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) == hipSuccess) {
    b->num_cu = prop.multiProcessorCount;
    b->lds_max = (int)prop.sharedMemPerBlock;
  }
  const int n = b->n;
  std::vector<int> rep_c(n);
  for (int r = 0; r < nrep; r++)
    for (int i = b->off[r]; i < b->off[r + 1]; i++) rep_c[i] = r;
  if ((rc = dalloc(&b->geom, nrep)) || (rc = dalloc(&b->off_d, nrep + 1)) || (rc = dalloc(&b->xin, 3 * (size_t)n)) ||
      (rc = dalloc(&b->staging, std::max<size_t>(3 * (size_t)n, nrep))) || (rc = dalloc(&b->type_c, n)) ||
      (rc = dalloc(&b->rep_c, n)) ||
      (rc = dalloc(&b->xw, n)) || (rc = dalloc(&b->x, n)) || (rc = dalloc(&b->xq, n)) || (rc = dalloc(&b->eat, n)) ||
      (rc = dalloc(&b->g, n)) ||
      (rc = dalloc(&b->rep, n)) || (rc = dalloc(&b->orig, n)) || (rc = dalloc(&b->inv, n)) ||
      (rc = dalloc(&b->key, n)) || (rc = dalloc(&b->slot, n)) || (rc = dalloc(&b->order, n)) ||
      (rc = dalloc(&b->numneigh, n)) || (rc = dalloc(&b->dflags, kFlagWords)) ||
      (rc = dalloc(&b->rho, n)) || (rc = dalloc(&b->fp, n)) || (rc = dalloc(&b->eemb, n)) ||
      (rc = dalloc(&b->vadj, n)) || (rc = upload(b->geom, b->geom_h.data(), sizeof(RepGeom) * nrep)) ||
      (rc = upload(b->off_d, b->off.data(), sizeof(int) * (nrep + 1))) ||
      (rc = upload(b->type_c, type, sizeof(int) * n)) || (rc = upload(b->rep_c, rep_c.data(), sizeof(int) * n))) {
    mdx_batch_destroy(b);
    return rc;
  }
  *out = b;
  return MDX_OK;
}

int mdx_batch_destroy(mdx_batch *b) {
  if (!b) return MDX_OK;
  (void)hipSetDevice(b->device);
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  void *ptrs[] = {b->xq, b->geom,    b->off_d,    b->xin,      b->staging,  b->type_c,  b->rep_c,   b->xw,      b->x,
                  b->eat,     b->g,        b->rep,      b->orig,     b->inv,     b->key,     b->slot,    b->order,
                  b->bin_count, b->bin_start, b->scan_tmp, b->nbr,    b->numneigh, b->dflags,
                  b->rho,     b->fp,       b->eemb,     b->vadj,     b->partials, b->colsum,  b->ljtab,   b->frho_d,
                  b->knots_d, b->knots_f};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  if (b->flags_host) (void)hipHostFree(b->flags_host);
  if (b->rep_host) (void)hipHostFree(b->rep_host);
  if (b->sums_host) (void)hipHostFree(b->sums_host);
  for (auto &l : b->ring) {
    (void)hipEventDestroy(l.a);
    (void)hipEventDestroy(l.b);
  }
  if (b->own_stream) {
    (void)hipStreamSynchronize(b->own_stream);
    (void)hipStreamDestroy(b->own_stream);
  }
  delete b;
  return MDX_OK;
}

int mdx_batch_set_stream(mdx_batch *b, int external, void *stream) {
  int rc = check_b(b);
  if (rc) return rc;
  hipError_t e = hipStreamSynchronize(b->stream);  // work already queued finishes where it was queued
  if (e != hipSuccess) return bfail(e, "batch stream switch");
  b->stream = external ? static_cast<hipStream_t>(stream) : b->own_stream;
  return MDX_OK;
}

int mdx_batch_set_positions(mdx_batch *b, const double *x) {
  int rc = check_b(b);
  if (rc) return rc;
  if (!x) {
    set_error("null positions");
    return MDX_ERR_ARG;
  }
  hipError_t e = hipMemcpyAsync(b->xin, x, sizeof(double) * 3 * b->n,
                                is_device_ptr(x, b->device) ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice,
                                b->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(b->stream);
  if (e != hipSuccess) return bfail(e, "positions upload");
  b->positions = true;
  b->built = false;
  b->eam_rho_prec = -1;
  return MDX_OK;
}

int mdx_batch_set_precision(mdx_batch *b, int precision) {
  int rc = check_b(b);
  if (rc) return rc;
  if (precision != MDX_FP64 && precision != MDX_MIXED) {
    set_error("precision must be MDX_FP64 or MDX_MIXED");
    return MDX_ERR_ARG;
  }
  if (precision != b->precision) {
    b->precision = precision;
    b->eam_rho_prec = -1;
    for (int k = 0; k < MDX_BK_NKIND; k++) b->tuned[k] = false;
  }
  return MDX_OK;
}

int mdx_batch_set_skin(mdx_batch *b, double skin) {
  int rc = check_b(b);
  if (rc) return rc;
  if (!(skin >= 0.0)) {
    set_error("skin must be >= 0");
    return MDX_ERR_ARG;
  }
  b->skin = skin;
  return MDX_OK;
}

int mdx_batch_lj_init(mdx_batch *b, const double *eps, const double *sigma, const double *cut) {
  int rc = check_b(b);
  if (rc) return rc;
  if (!eps || !sigma || !cut) {
    set_error("null lj tables");
    return MDX_ERR_ARG;
  }
  const int nt1 = b->ntypes + 1;
  std::vector<double> tab(T_N * kNT, 0.0);
  double cutmax = 0.0;
  for (int i = 1; i < nt1; i++)
    for (int j = 1; j < nt1; j++) {
      const int s = i * nt1 + j;
      const double ep = eps[s], sg = sigma[s], c = cut[s];
      if (!(sg > 0.0) || !(c > 0.0) || !(ep >= 0.0)) {
        set_error("lj tables need eps >= 0, sigma > 0, cut > 0 for every type pair");
        return MDX_ERR_ARG;
      }
      const int t = i * nt1 + j;  // kernel index ti*nt1 + tj
      tab[T_CUTSQ * kNT + t] = c * c;
      tab[T_LJ1 * kNT + t] = 48.0 * ep * std::pow(sg, 12.0);
      tab[T_LJ2 * kNT + t] = 24.0 * ep * std::pow(sg, 6.0);
      tab[T_LJ3 * kNT + t] = 4.0 * ep * std::pow(sg, 12.0);
      tab[T_LJ4 * kNT + t] = 4.0 * ep * std::pow(sg, 6.0);
      tab[T_A1 * kNT + t] = 48.0 * std::pow(sg, 12.0);
      tab[T_A2 * kNT + t] = 24.0 * std::pow(sg, 6.0);
      tab[T_B1 * kNT + t] = 576.0 * ep * std::pow(sg, 11.0);
      tab[T_B2 * kNT + t] = 144.0 * ep * std::pow(sg, 5.0);
      cutmax = std::max(cutmax, c);
    }
  if (b->pair == MDX_PAIR_LJ && b->ljtab && tab == b->lj_tab) return MDX_OK;
  if (!b->ljtab && (rc = dalloc(&b->ljtab, T_N * kNT))) return rc;
  if ((rc = upload(b->ljtab, tab.data(), sizeof(double) * T_N * kNT))) return rc;
  b->lj_tab = tab;
  b->pair = MDX_PAIR_LJ;
  b->lj_cutmax = cutmax;
  return MDX_OK;
}

int mdx_batch_lj_forces(mdx_batch *b, double *f, double *energy) {
  int rc = check_b(b);
  if (rc) return rc;
  if (b->pair != MDX_PAIR_LJ) {
    set_error("lj/cut not initialised (mdx_batch_lj_init)");
    return MDX_ERR_ARG;
  }
  if ((rc = ensure_built(b))) return rc;
  const int nt1 = b->ntypes + 1;
  const bool mixed = b->precision == MDX_MIXED;
  const ForceOut out = force_out(b, f);
  auto launch = [&](const Tune &t) {
    const int G = persistent_grid(b, t);
    if (mixed)
      TPA_DISPATCH(t.tpa, BATCH_LAUNCH((k_b_lj<true, TP>), G, t.block, 0, b->n, nt1, b->x, b->xq, b->rep, b->geom, b->nbr,
                                       b->numneigh, b->cap, b->ljtab, out))
    else
      TPA_DISPATCH(t.tpa, BATCH_LAUNCH((k_b_lj<false, TP>), G, t.block, 0, b->n, nt1, b->x, b->xq, b->rep, b->geom, b->nbr,
                                       b->numneigh, b->cap, b->ljtab, out))
  };
  if ((rc = run_kind(b, MDX_BK_LJ, launch))) return rc;
  return force_results(b, out, f, energy);
}

int mdx_batch_lj_vjp(mdx_batch *b, const double *gf, double *geps, double *gsigma) {
  int rc = check_b(b);
  if (rc) return rc;
  if (b->pair != MDX_PAIR_LJ) {
    set_error("lj/cut not initialised (mdx_batch_lj_init)");
    return MDX_ERR_ARG;
  }
  if (!gf || !geps || !gsigma) {
    set_error("null argument");
    return MDX_ERR_ARG;
  }
  if ((rc = ensure_built(b)) || (rc = read_g(b, gf))) return rc;
  const int nt1 = b->ntypes + 1;
  // the adjoint's per-pair factors (48 s^12 r^-6 - 24 s^6 and the sigma
  // term) cancel near the potential minimum, where FP32 loses ~5e-6
  // relative: the adjoint runs FP64 arithmetic in both precision modes
  int grid_used = 0;
  auto launch = [&](const Tune &t) {
    const int G = persistent_grid(b, t, true);
    grid_used = G;
    auto go = [&](auto nt) {
      TPA_DISPATCH(t.tpa, BATCH_LAUNCH((k_b_lj_vjp<decltype(nt)::value, TP>), G, t.block, 0, b->n, nt1, b->x, b->rep, b->geom, b->nbr, b->numneigh, b->cap,
                                             b->ljtab, b->g, b->partials))
    };
    if (b->ntypes == 1) go(std::integral_constant<int, 1>{});
    else if (b->ntypes == 2) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, MDX_MAXT>{});
  };
  // partial rows for the largest grid any candidate can use
  const long maxgrid = (long)kPartialBlocksPerCU * b->num_cu;
  if ((rc = grow(&b->partials, &b->partials_cap, (size_t)maxgrid * 2 * nt1 * nt1))) return rc;
  if ((rc = run_kind(b, MDX_BK_LJ_VJP, launch))) return rc;
  const int cols = nt1 * nt1;
  if ((rc = colsum(b, grid_used, 2 * cols))) return rc;
  for (int k = 0; k < cols; k++) {
    geps[k] = b->sums_host[k];
    gsigma[k] = b->sums_host[cols + k];
  }
  return MDX_OK;
}

int mdx_batch_eam_init(mdx_batch *b, int nrho, double drho, int nr, double dr, double cut, const double *frho,
                       const double *rhor, const double *z2r) {
  int rc = check_b(b);
  if (rc) return rc;
  if (nrho < 5 || nr < 5 || !(drho > 0) || !(dr > 0) || !(cut > 0) || !frho || !rhor || !z2r) {
    set_error("mdx_batch_eam_init: invalid tables (at least 5 knots, positive spacings and cutoff)");
    return MDX_ERR_ARG;
  }
  if (b->pair == MDX_PAIR_EAM && b->et.nrho == nrho && b->et.nr == nr && b->eam_drho == drho && b->eam_dr == dr &&
      b->eam_cut == cut && std::equal(frho, frho + nrho, b->eam_knots[0].begin()) &&
      std::equal(rhor, rhor + nr, b->eam_knots[1].begin()) && std::equal(z2r, z2r + nr, b->eam_knots[2].begin()))
    return MDX_OK;  // same tables: keep rho/fp of the last forward pass
  std::vector<double> sf, sr, sz;
  spline7(nrho, drho, frho, sf);
  spline7(nr, dr, rhor, sr);
  spline7(nr, dr, z2r, sz);
  // rhor and z2r as two 4-vectors per knot, in both precisions
  const size_t kn = (size_t)nr + 1;
  std::vector<double4> kd(4 * kn);
  std::vector<float4> kf(4 * kn);
  for (size_t q = 0; q < 2 * kn; q++) {
    const double *c = (q < kn ? sr.data() + 7 * q : sz.data() + 7 * (q - kn));
    kd[2 * q] = make_double4(c[0], c[1], c[2], 0.0);
    kd[2 * q + 1] = make_double4(c[3], c[4], c[5], c[6]);
    kf[2 * q] = make_float4((float)c[0], (float)c[1], (float)c[2], 0.0f);
    kf[2 * q + 1] = make_float4((float)c[3], (float)c[4], (float)c[5], (float)c[6]);
  }
  // no pair style until the new tables are on the device
  const bool same_nrho = b->et.nrho == nrho, same_nr = b->et.nr == nr;
  if (b->pair == MDX_PAIR_EAM) b->pair = MDX_PAIR_NONE;
  b->et.nrho = b->et.nr = 0;
  if (!same_nrho && (rc = dalloc(&b->frho_d, sf.size()))) return rc;
  if (!same_nr && ((rc = dalloc(&b->knots_d, kd.size())) || (rc = dalloc(&b->knots_f, kf.size())))) return rc;
  if ((rc = upload(b->frho_d, sf.data(), sizeof(double) * sf.size())) ||
      (rc = upload(b->knots_d, kd.data(), sizeof(double4) * kd.size())) ||
      (rc = upload(b->knots_f, kf.data(), sizeof(float4) * kf.size())))
    return rc;
  b->knots = {b->knots_d, b->knots_d + 2 * kn, b->knots_f, b->knots_f + 2 * kn};
  b->et.nrho = nrho;
  b->et.nr = nr;
  b->et.rdrho = 1.0 / drho;
  b->et.rdr = 1.0 / dr;
  b->et.rhomax = (nrho - 1) * drho;
  b->et.cutsq = cut * cut;
  b->eam_knots[0].assign(frho, frho + nrho);
  b->eam_knots[1].assign(rhor, rhor + nr);
  b->eam_knots[2].assign(z2r, z2r + nr);
  b->eam_drho = drho;
  b->eam_dr = dr;
  b->eam_cut = cut;
  b->pair = MDX_PAIR_EAM;
  b->eam_rho_prec = -1;
  return MDX_OK;
}

namespace {
// rho + fp pass in `precision`, then (with_force) the force pass
int eam_forward(mdx_batch *b, bool with_force, int precision, double *f = nullptr) {
  int rc;
  if ((rc = ensure_built(b))) return rc;
  const bool mixed = precision == MDX_MIXED;
  const size_t vec = (size_t)(b->et.nr + 1) * (mixed ? sizeof(float4) : sizeof(double4));
  const bool lds1 = vec <= (size_t)kTabLDS * 8, lds2 = 3 * vec <= (size_t)kTabLDS * 8;
  // precision and table place as types, threads per atom from the tune
  auto choose = [&](bool lds, auto &&go) {
    if (mixed && lds) go(std::true_type{}, std::true_type{});
    else if (mixed) go(std::true_type{}, std::false_type{});
    else if (lds) go(std::false_type{}, std::true_type{});
    else go(std::false_type{}, std::false_type{});
  };
  auto rho_launch = [&](const Tune &t) {
    const int G = persistent_grid(b, t);
    choose(lds1, [&](auto mx, auto tl) {
      TPA_DISPATCH(t.tpa, BATCH_LAUNCH((k_b_eam_rho<decltype(mx)::value, TP, decltype(tl)::value>), G, t.block,
                                       lds1 ? vec : 0, b->n, b->x, b->xq, b->rep,
                                             b->geom, b->nbr, b->numneigh, b->cap, b->et, b->knots, b->frho_d, b->rho,
                                             b->fp, b->eemb))
    });
  };
  if ((rc = run_kind(b, MDX_BK_EAM_RHO, rho_launch))) return rc;
  b->eam_rho_prec = precision;
  if (!with_force) return MDX_OK;
  const ForceOut out = force_out(b, f);
  auto force_launch = [&](const Tune &t) {
    const int G = persistent_grid(b, t);
    choose(lds2, [&](auto mx, auto tl) {
      TPA_DISPATCH(t.tpa, BATCH_LAUNCH((k_b_eam_force<decltype(mx)::value, TP, decltype(tl)::value>), G, t.block,
                                       lds2 ? 3 * vec : 0, b->n, b->x, b->xq, b->rep,
                                             b->geom, b->nbr, b->numneigh, b->cap, b->et, b->knots, b->fp, b->eemb,
                                             out))
    });
  };
  return run_kind(b, MDX_BK_EAM_FORCE, force_launch);
}
}  // namespace

int mdx_batch_eam_forces(mdx_batch *b, double *f, double *energy, double *rho, double *fp) {
  int rc = check_b(b);
  if (rc) return rc;
  if (b->pair != MDX_PAIR_EAM) {
    set_error("eam not initialised (mdx_batch_eam_init)");
    return MDX_ERR_ARG;
  }
  if ((rc = eam_forward(b, true, b->precision, f))) return rc;
  if ((rc = force_results(b, force_out(b, f), f, energy))) return rc;
  for (int k = 0; k < 2; k++) {
    double *out = k == 0 ? rho : fp;
    if (!out) continue;
    hipLaunchKernelGGL(k_b_gather_s, dim3((b->n + 255) / 256), dim3(256), 0, b->stream, b->n, b->inv,
                       k == 0 ? b->rho : b->fp, b->staging);
    hipError_t e = hipMemcpyAsync(out, b->staging, sizeof(double) * b->n, hipMemcpyDeviceToHost, b->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(b->stream);
    if (e != hipSuccess) return bfail(e, "rho/fp output");
  }
  return MDX_OK;
}

int mdx_batch_eam_vjp(mdx_batch *b, const double *gf, double *g_frho, double *g_rhor, double *g_z2r) {
  int rc = check_b(b);
  if (rc) return rc;
  if (b->pair != MDX_PAIR_EAM) {
    set_error("eam not initialised (mdx_batch_eam_init)");
    return MDX_ERR_ARG;
  }
  if (!gf || !g_frho || !g_rhor || !g_z2r) {
    set_error("null argument");
    return MDX_ERR_ARG;
  }
  if ((rc = ensure_built(b))) return rc;
  // the adjoint uses FP64 rho/fp (a mixed forward's rho moves the frho
  // spline weights by ~1e-5 relative): rerun the rho pass in FP64 if needed
  if (b->eam_rho_prec != MDX_FP64 && (rc = eam_forward(b, false, MDX_FP64))) return rc;
  if ((rc = read_g(b, gf, b->fp))) return rc;
  // FP64 adjoint arithmetic in both precision modes, as for lj/cut
  const int P = 4 * (b->et.nrho + 1) + 8 * (b->et.nr + 1);
  if ((long)sizeof(double) * P > b->lds_max) {
    set_error("eam tables too large for the adjoint's LDS accumulators");
    return MDX_ERR_ARG;
  }
  const int kn = b->et.nr + 1, kf = b->et.nrho + 1;
  // accumulator sets per workgroup: as many of 4, 2, 1 as keep it within an
  // eighth of a CU's LDS (small tables), and rho' beside them if it fits
  const size_t tabA = sizeof(double4) * kn, gfA = sizeof(double) * 3 * kf, setA = sizeof(double) * adj_stride(7, kn),
               setB = sizeof(double) * adj_stride(4, kn);
  int cA = 4, cB = 4;
  while (cA > 1 && gfA + tabA + cA * setA > kAdjLDS) cA /= 2;
  while (cB > 1 && cB * setB > kAdjLDS) cB /= 2;
  const bool tlA = tabA + gfA + cA * setA <= (size_t)b->lds_max;
  const size_t shA = (tlA ? tabA : 0) + gfA + cA * setA, shB = cB * setB;
  const long maxgrid = (long)kPartialBlocksPerCU * b->num_cu;
  if ((rc = grow(&b->partials, &b->partials_cap, (size_t)maxgrid * (P + 4 * kn)))) return rc;
  int gA = 0, gB = 0;
  auto launchA = [&](const Tune &t) {
    const int G = persistent_grid(b, t, true);
    gA = G;
    auto go = [&](auto tl) {
      TPA_DISPATCH(t.tpa, BATCH_LAUNCH((k_b_eam_adj_a<TP, decltype(tl)::value>), G, t.block, shA, b->n, b->x, b->rep, b->geom, b->nbr, b->numneigh, b->cap,
                                             b->et, b->knots.rhor_d, b->frho_d, b->rho, b->g, cA, b->vadj,
                                             b->partials))
    };
    if (tlA) go(std::true_type{});
    else go(std::false_type{});
  };
  if ((rc = run_kind(b, MDX_BK_EAM_ADJ_A, launchA))) return rc;
  double *partB = b->partials + (size_t)gA * P;
  auto launchB = [&](const Tune &t) {
    const int G = persistent_grid(b, t, true);
    gB = G;
    TPA_DISPATCH(t.tpa, BATCH_LAUNCH((k_b_eam_adj_b<TP>), G, t.block, shB, b->n, b->vadj,
                                           b->rep, b->geom, b->nbr, b->numneigh, b->cap, b->et, cB, partB))
  };
  if ((rc = run_kind(b, MDX_BK_EAM_ADJ_B, launchB))) return rc;
  if ((rc = colsum(b, gA, P, partB, gB, 4 * kf, 4 * kn))) return rc;
  knot_gradient(b->et.nrho, b->sums_host, g_frho);
  knot_gradient(b->et.nr, b->sums_host + 4 * kf, g_rhor);
  knot_gradient(b->et.nr, b->sums_host + 4 * kf + 4 * kn, g_z2r);
  return MDX_OK;
}

int mdx_batch_set_launch(mdx_batch *b, int kind, int block, int tpa, int grid) {
  int rc = check_b(b);
  if (rc) return rc;
  if (kind < 0 || kind >= MDX_BK_NKIND || block < 64 || block > 1024 || block % 64 || tpa < 1 || tpa > 64 ||
      (tpa & (tpa - 1)) || grid < 0) {
    set_error("invalid launch shape (block 64..1024 multiple of 64, tpa power of two <= 64, grid >= 0)");
    return MDX_ERR_ARG;
  }
  b->tune[kind].block = block;
  b->tune[kind].tpa = tpa;
  b->tune[kind].grid = grid;
  b->tuned[kind] = true;
  return MDX_OK;
}

int mdx_batch_get_launch(mdx_batch *b, int kind, int *block, int *tpa, int *grid) {
  int rc = check_b(b);
  if (rc) return rc;
  if (kind < 0 || kind >= MDX_BK_NKIND) {
    set_error("invalid kernel kind");
    return MDX_ERR_ARG;
  }
  const Tune t = tune_of(b, kind);
  if (block) *block = t.block;
  if (tpa) *tpa = t.tpa;
  if (grid) *grid = t.grid;
  return MDX_OK;
}

int mdx_batch_autotune(mdx_batch *b, int on) {
  int rc = check_b(b);
  if (rc) return rc;
  b->autotune = on != 0;
  if (b->autotune)
    for (int k = 0; k < MDX_BK_NKIND; k++) b->tuned[k] = false;
  return MDX_OK;
}

int mdx_batch_kernel_time(mdx_batch *b, int kind, double *ms, long *launches) {
  int rc = check_b(b);
  if (rc) return rc;
  if (kind < 0 || kind >= MDX_BK_NKIND) {
    set_error("invalid kernel kind");
    return MDX_ERR_ARG;
  }
  if ((rc = resolve_times(b))) return rc;
  if (ms) *ms = b->kms[kind];
  if (launches) *launches = b->klaunch[kind];
  return MDX_OK;
}

int mdx_batch_neigh_stats(mdx_batch *b, long *total, int *max_per_atom) {
  int rc = check_b(b);
  if (rc) return rc;
  if ((rc = ensure_built(b))) return rc;
  if (total) *total = b->total_neighbors;
  if (max_per_atom) *max_per_atom = b->max_neighbors;
  return MDX_OK;
}

}  // extern "C"
