// pair.hip - lj/cut and eam force kernels for gfx950.
//
// Replaces PairLJCut::compute (src/pair_lj_cut.cpp:68-141) and
// PairEAM::compute (src/MANYBODY/pair_eam.cpp:125-306).  The reference walks
// a half list and scatters f[j] -= ...; here every atom owns its row of a
// full list and only gathers, so forces, energies and virials are written
// once per atom with no atomics and a fixed summation order (deterministic).
// Energy and virial per atom are half of each pair term (pair.cpp:862-901,
// ev_tally_full), and the global sums come from a fixed-order block tree.
//
// Threads per atom (TPA, a template parameter dividing 64): the TPA lanes of
// an atom share its list.  The lj/cut kernels give each lane chunks of four
// consecutive entries (one 16-B index load per chunk; the FP64 kernel with
// four lanes per atom transposes the group's chunks so that one gather
// covers four consecutive entries); the eam kernels take entries lane,
// lane+TPA, ...  Lists hold neighbours in bin-sorted order, so the lanes of
// a group gather nearby atoms and a 64-lane load touches fewer cache lines.
// The TPA partial sums are combined with cross-lane shuffles; lane 0 of the
// group writes the atom.
//
// Precision modes (template MIXED):
//   FP64  : everything in double, as the reference.
//   MIXED : neighbours are read from the 32-bit fixed-point mirror and
//           del = x_i - x_j and rsq are rebuilt in FP64 (a pair within a
//           narrow band of the cutoff is re-tested on the FP64 positions, so
//           the cutoff test is the reference's); the potential arithmetic
//           (1/r^2, r^6, splines) is FP32; forces, energies and virials
//           accumulate in FP64.
//
// EAM: the reference needs rho -> reverse_comm -> fp -> forward_comm ->
// force (pair_eam.cpp:206,232).  With a full list rho_i is complete inside
// one atom's lanes, so the fp pass is fused into the rho kernel and the only
// grid-wide dependency left is fp[j] for the force kernel: two launches.
#include "mdx_internal.h"

namespace mdx {

namespace {

constexpr int kNT2 = MDX_NT1 * MDX_NT1;
constexpr int kUnroll = 4;  // neighbour entries in flight per lane (FP64 gathers)
#ifndef MDX_GATHER_UNROLL_Q
#define MDX_GATHER_UNROLL_Q 4
#endif
// entries in flight per lane for the 16-B fixed-point gathers; a lane's
// entry sequence (lane, lane+TPA, ...) does not depend on it, so neither do
// the results
constexpr int kUnrollQ = MDX_GATHER_UNROLL_Q;

#ifndef MDX_PAIR_MIN_WAVES
#define MDX_PAIR_MIN_WAVES 1
#endif
#define MDX_PAIR_BOUNDS __launch_bounds__(256, MDX_PAIR_MIN_WAVES)
// the FP64 eam kernels with LDS tables run in workgroups of up to 512 threads
#define MDX_EAM_BOUNDS(WIDE) __launch_bounds__((WIDE) ? 512 : 256, MDX_PAIR_MIN_WAVES)

// A lane's share of a row is either strided, entries lane, lane+TPA, ...,
// or chunked, four consecutive entries 4*lane .. 4*lane+3, then
// 4*(lane+TPA) .., one 16-B index load per chunk (rows start 16-B aligned).
// Chunks take 4x fewer index-load requests; measured on MI355X they speed
// up lj/cut (threads per atom 4) by 3-7% and slow the eam kernels (8) by
// 10-15%, so k_lj is chunked and the eam kernels are strided.

#ifndef MDX_TRANS_LJ
#define MDX_TRANS_LJ 1
#endif
constexpr bool kTransLJ = MDX_TRANS_LJ;

#ifndef MDX_STREAM_LIST
#define MDX_STREAM_LIST 0
#endif
// list entries are read once per launch: a streaming (non-temporal) load
// keeps them from evicting the neighbour positions the gathers reuse from L2
__device__ __forceinline__ int list_entry(const int *p) {
  if (MDX_STREAM_LIST) return __builtin_nontemporal_load(p);
  return *p;
}

template <int NV>
__device__ __forceinline__ void block_reduce_store(double (&v)[NV], double *__restrict__ out) {
  __shared__ double s[NV][16];
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int k = 0; k < NV; k++) v[k] += __shfl_down(v[k], off, 64);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < NV; k++) s[k][w] = v[k];
  __syncthreads();
  if (threadIdx.x < NV) {
    const int nw = (blockDim.x + 63) >> 6;
    double acc = 0.0;
    for (int q = 0; q < nw; q++) acc += s[threadIdx.x][q];
    out[(size_t)blockIdx.x * NV + threadIdx.x] = acc;
  }
}

// Which atom and which of its TPA lanes a thread is.  By default a group's
// lanes are neighbours in the wavefront.  ACROSS puts neighbouring atoms in
// neighbouring lanes instead (lane l of a wavefront: atom l mod 64/TPA, share
// l / (64/TPA)): the chunked lj/cut kernel then reads one chunk of 64/TPA
// consecutive atoms as contiguous 16-B pieces, not TPA chunks npad * 16 B
// apart, and the gathers of neighbouring atoms share more cache lines.  The
// kernel waits for L1: 1.09 line lookups per CU and cycle at 2.048 M atoms
// (47 per load instruction; across 0.85 and 34), its vector units 57% busy.  Per step kernel,
// grouped / across: mixed, 4 lanes 2.048 M atoms 287 / 272 us, 256,000 35.1 /
// 32.3; FP64, 8 lanes 32,000 11.0 / 10.2; 16 lanes 8,000 Kob-Andersen 6.37 /
// 6.15.  Four lanes in FP64 keep the group (its transposed chunks are faster:
// 381 against 400 us at 2.048 M).  So do the eam kernels: they read entries,
// not chunks, so the lanes of a group already gather consecutive entries
// (17-21 lookups per instruction; across, 256,000 atoms FP64 145 against 109).
constexpr bool lj_across(bool mixed, int tpa) { return tpa >= (mixed ? 4 : 8); }
// The lj/cut kernel loads a lane's next chunk before it waits for the gathers
// of the current one where a lane has few trips and the kernel is a chain of
// latencies (4,000 atoms, 16 lanes: 4.89 against 5.16 us; 32,000 mixed, 8
// lanes: 7.74 against 7.88).  At 4 lanes the registers cost more (2.048 M
// mixed: 306 against 272).
constexpr bool lj_ahead(int tpa) { return tpa >= 8; }

template <int TPA, bool ACROSS>
__device__ __forceinline__ void group_place(int &i, int &lane) {
  const unsigned t = xcd_block() * blockDim.x + threadIdx.x;  // workgroups are whole wavefronts
  constexpr unsigned A = 64 / TPA;
  i = ACROSS ? (t >> 6) * A + t % A : t / TPA;
  lane = ACROSS ? (t & 63) / A : t % TPA;
}

// sum over the TPA lanes of a group; the result is valid in lane 0
template <int TPA, bool ACROSS = false>
__device__ __forceinline__ double group_sum(double v) {
  constexpr int A = ACROSS ? 64 / TPA : 1;
#pragma unroll
  for (int off = TPA / 2; off > 0; off >>= 1) v += __shfl_down(v, off * A, A > 1 ? 64 : TPA);
  return v;
}

// Mixed precision with four lanes per atom keeps two sets of sums per lane,
// set h holding the lane's trips (eam: entries) of parity h, and adds the
// sets before the lanes: the order of the additions, and so every bit of the
// result, is that of eight lanes per atom.  A mixed trajectory then does not
// depend on which of the two the default launch takes for its size; the
// fixed-point mirror otherwise turns a last-bit difference of a sum into a
// rounding step of a position (about 1e-8 of the box).
__host__ __device__ constexpr bool split_sums(bool mixed, int tpa) { return mixed && tpa == 4; }
template <int NS>
__device__ __forceinline__ double set_sum(const double (&v)[NS]) {
  return NS == 2 ? v[0] + v[NS - 1] : v[0];
}

__device__ __forceinline__ void image_shift(int code, double px, double py, double pz, double &sx, double &sy,
                                            double &sz) {
  sx = ((code % 3) - 1) * px;
  sy = (((code / 3) % 3) - 1) * py;
  sz = ((code / 9) - 1) * pz;
}

// del = x_i - (x_j + image shift), the ghost-image geometry of the reference
__device__ __forceinline__ void pair_delta(const double4 &xi, const double4 &xj, int code, double px, double py,
                                           double pz, double &delx, double &dely, double &delz) {
  double gx = xj.x, gy = xj.y, gz = xj.z;
  if (code != MDX_NOSHIFT) {
    double sx, sy, sz;
    image_shift(code, px, py, pz, sx, sy, sz);
    gx += sx;
    gy += sy;
    gz += sz;
  }
  delx = xi.x - gx;
  dely = xi.y - gy;
  delz = xi.z - gz;
}

// Virial of one full-list entry (the pair's force on i is fpair * del).
// pervir: the per-pair tally of ev_tally (src/pair.cpp:850-855), half of
// del x f per entry, which also gives the per-atom virial.  Otherwise the
// global virial is taken as virial_fdotr_compute does (src/pair.cpp:
// 1402-1450): sum_i x_i f_i, formed once per atom in finish_atom, minus
// half of s x f for every entry whose partner image is shifted by s (the
// ghost atoms' share of the reference's sum over owned and ghost atoms):
// sum_i sum_j del_ij f_ij / 2 with del_ij = x_i - x_j - s_ij and
// f_ji = -f_ij.
__device__ __forceinline__ void virial_entry(double (&w)[6], int pervir, int code, double px, double py, double pz,
                                             double delx, double dely, double delz, double fpair) {
  if (pervir) {
    const double hf = 0.5 * fpair;
    w[0] += delx * delx * hf;
    w[1] += dely * dely * hf;
    w[2] += delz * delz * hf;
    w[3] += delx * dely * hf;
    w[4] += delx * delz * hf;
    w[5] += dely * delz * hf;
  } else if (code != MDX_NOSHIFT) {
    double sx, sy, sz;
    image_shift(code, px, py, pz, sx, sy, sz);
    const double h = -0.5 * fpair;
    w[0] += sx * delx * h;
    w[1] += sy * dely * h;
    w[2] += sz * delz * h;
    w[3] += sx * dely * h;
    w[4] += sx * delz * h;
    w[5] += sy * delz * h;
  }
}

// fix nve for one atom right after its force is complete: final integrate
// of this step, then (ig.next) the initial integrate of the next step into
// ig.xn, with the rebuild trigger.  Same operations and order as
// k_nve_final + k_nve_initial, so fused and unfused trajectories are
// bit-identical.  Returns m*v^2 after the final half-kick (thermo).
// v and xhold (vpre, hpre) are loaded at the start of the force kernel, so
// their latency hides behind the neighbour loop instead of extending it.
__device__ __forceinline__ double integrate_atom(int i, const double4 &xi, double fx, double fy, double fz,
                                                 const IntegArgs &ig, double4 q, const double4 &h) {
#pragma clang fp contract(off)
  const double m = ig.mass[static_cast<int>(xi.w)];
  const double dtfm = ig.dtf / m;
  q.x += dtfm * fx;
  q.y += dtfm * fy;
  q.z += dtfm * fz;
  const double mv2 = (q.x * q.x + q.y * q.y + q.z * q.z) * m;
  if (ig.next) {
    q.x += dtfm * fx;
    q.y += dtfm * fy;
    q.z += dtfm * fz;
    double4 p = xi;
    p.x += ig.dtv * q.x;
    p.y += ig.dtv * q.y;
    p.z += ig.dtv * q.z;
    ig.xn[i] = p;
    if (ig.xqn) ig.xqn[i] = quantize(ig.qs, p);
    if (ig.check) {
      const double dx = p.x - h.x, dy = p.y - h.y, dz = p.z - h.z;
      mark_trigger(dx * dx + dy * dy + dz * dz > ig.triggersq, ig.trig, ig.trig_dev, ig.stamp);
    }
  }
  ig.v[i] = q;
  return mv2;
}

// per-atom results of one group: lane 0 stores (and integrates when fused),
// all lanes join the block sum of {e, virial[6], m v^2}
template <int TPA, bool EV, bool INTEG, bool LATE = false, bool ACROSS = false>
__device__ __forceinline__ void finish_atom(int i, bool owner, const double4 &xi, double fx, double fy,
                                            double fz, double e, double (&w)[6], const IntegArgs &ig,
                                            double4 vpre, double4 hpre, double4 *__restrict__ f,
                                            double *__restrict__ partials) {
  int o = 0;  // caller index: its load overlaps the lane sums
  const bool caller = !INTEG && owner && (ig.out.f || (EV && (ig.out.e || ig.out.v)));
  if (caller) o = ig.out.orig[i];
  fx = group_sum<TPA, ACROSS>(fx);
  fy = group_sum<TPA, ACROSS>(fy);
  fz = group_sum<TPA, ACROSS>(fz);
  if (EV) {
    e = group_sum<TPA, ACROSS>(e);
#pragma unroll
    for (int q = 0; q < 6; q++) w[q] = group_sum<TPA, ACROSS>(w[q]);
  }
  double mv2 = 0.0;
  if (owner) {
    if (!INTEG || EV || ig.write_f) f[i] = make_double4(fx, fy, fz, e);
    if (caller) {
      if (ig.out.f) {
        double *const d = ig.out.f + 3 * (size_t)o;
        d[0] = ig.out.add ? d[0] + fx : fx;
        d[1] = ig.out.add ? d[1] + fy : fy;
        d[2] = ig.out.add ? d[2] + fz : fz;
      }
      if (EV && ig.out.e) ig.out.e[o] = e;
      if (EV && ig.pervir && ig.out.v) {
        double *const d = ig.out.v + 6 * (size_t)o;
#pragma unroll
        for (int q = 0; q < 6; q++) d[q] = w[q];
      }
    }
    if (EV && !ig.pervir) {  // the x_i f_i share of the global virial
      w[0] += xi.x * fx;
      w[1] += xi.y * fy;
      w[2] += xi.z * fz;
      w[3] += xi.x * fy;
      w[4] += xi.x * fz;
      w[5] += xi.y * fz;
    }
    if (INTEG && LATE) {  // v and xhold read here, not held through the neighbour loop
      vpre = ig.v[i];
      if (ig.check) hpre = ig.xhold[i];
    }
    if (INTEG) mv2 = integrate_atom(i, xi, fx, fy, fz, ig, vpre, hpre);
  }
  if (EV) {
    double v[8] = {owner ? e : 0.0,    owner ? w[0] : 0.0, owner ? w[1] : 0.0, owner ? w[2] : 0.0,
                   owner ? w[3] : 0.0, owner ? w[4] : 0.0, owner ? w[5] : 0.0, owner ? mv2 : 0.0};
    block_reduce_store<8>(v, partials);
  }
}

// ------------------------------------------------------------------ LJ
// Q (mixed only): neighbours are read from the 32-bit fixed-point mirror xq
// (16 B instead of 32), their separation rebuilt in FP64 from the wrapping
// integer difference; a pair whose rsq lies within kBand of the cutoff is
// re-tested on the FP64 positions with its image shift, so the cutoff
// decision is the FP64 one (the quantised rsq is within ~1e-7 relative).
constexpr double kBand = 2e-6;

// fused force kernels (lj/cut, eam): read v (and xhold) after the
// neighbour loop instead of before it, so they do not occupy registers
// through the loop
#ifndef MDX_LATE_V
#define MDX_LATE_V 1
#endif
constexpr bool kLateV = MDX_LATE_V;

// ONE: a single atom type, so every pair uses the coefficients of type pair
// (1,1): the table reads are loop-invariant and leave the neighbour loop.
struct LJOne {  // the (1,1) coefficients of a single-type system, as kernel arguments (scalar registers)
  double clo, chi, cut, lj1, lj2, lj3, lj4, off;
  float f1, f2, f3, f4, foff;
};
template <bool MIXED, bool EV, int TPA, bool INTEG, bool Q, bool ONE>
__global__ MDX_PAIR_BOUNDS void k_lj(int n, int npad, int cap, int nt1, double px, double py, double pz,
                                           const double4 *__restrict__ x, const int4 *__restrict__ xq, QScale qs,
                                           const int *__restrict__ nbr, const int *__restrict__ numneigh,
                                           const LJTab *__restrict__ tab, double4 *__restrict__ f,
                                           double *__restrict__ partials, IntegArgs ig,
                                           LJOne one) {
  if constexpr (INTEG) {
    if (gate_closed(ig.gate)) return;
  }
  __shared__ double s_cutsq[kNT2], s_lj1[kNT2], s_lj2[kNT2], s_lj3[kNT2], s_lj4[kNT2], s_off[kNT2];
  __shared__ double s_clo[Q ? kNT2 : 1], s_chi[Q ? kNT2 : 1];
  __shared__ float f_lj1[kNT2], f_lj2[kNT2], f_lj3[kNT2], f_lj4[kNT2], f_off[kNT2];
  const int nt2 = nt1 * nt1;
  for (int q = threadIdx.x; q < nt2; q += blockDim.x) {
    if (Q) {
      s_clo[q] = tab->cutsq[q] * (1.0 - kBand);
      s_chi[q] = tab->cutsq[q] * (1.0 + kBand);
    }
    s_cutsq[q] = tab->cutsq[q];
    s_lj1[q] = tab->lj1[q];
    s_lj2[q] = tab->lj2[q];
    s_lj3[q] = tab->lj3[q];
    s_lj4[q] = tab->lj4[q];
    s_off[q] = tab->offset[q];
    f_lj1[q] = (float)tab->lj1[q];
    f_lj2[q] = (float)tab->lj2[q];
    f_lj3[q] = (float)tab->lj3[q];
    f_lj4[q] = (float)tab->lj4[q];
    f_off[q] = (float)tab->offset[q];
  }
  __syncthreads();
  int i, lane;
  constexpr bool ACROSS = lj_across(MIXED, TPA);
  group_place<TPA, ACROSS>(i, lane);
  // single type: the (1,1) coefficients come as kernel arguments, so they
  // stay in scalar registers for the whole loop (no LDS reads, no vector
  // registers)
  constexpr bool HOIST = ONE;
  const int t11 = nt1 + 1;
  (void)t11;
  const double o_clo = one.clo, o_chi = one.chi, o_cut = one.cut, o_lj1 = one.lj1, o_lj2 = one.lj2;
  const float o_f1 = one.f1, o_f2 = one.f2;
  constexpr int NS = split_sums(MIXED, TPA) ? 2 : 1;
  double fx[NS] = {}, fy[NS] = {}, fz[NS] = {}, e = 0.0;
  double w[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  double4 xi = make_double4(0.0, 0.0, 0.0, 0.0);
  double4 vpre = make_double4(0.0, 0.0, 0.0, 0.0), hpre = vpre;
  if (INTEG && !kLateV && i < n && lane == 0) {
    vpre = ig.v[i];
    if (ig.check) hpre = ig.xhold[i];
  }
  if (i < n) {
    if (!Q) xi = x[i];  // Q reads it where it is used: the re-test, the end
    const int4 qi = Q ? xq[i] : make_int4(0, 0, 0, 0);
    const int row = (Q ? qi.w : static_cast<int>(xi.w)) * nt1;
    const int jn = numneigh[i];
    const int4 *nb4 = reinterpret_cast<const int4 *>(nbr) + i;  // chunk c at nb4[c * npad]
    // UNROLL entries per lane per trip: all index loads, then all gathers,
    // are issued before the first use, so a lane has UNROLL gathers in flight
    constexpr int U = 4;  // entries of a chunk
    const int self = i | (MDX_NOSHIFT << MDX_IDX_BITS);
    // TRANS (four lanes per atom, 32-B FP64 gathers): the group's four
    // chunks are transposed across its lanes, so gather u of the group
    // covers entries 4u .. 4u+3, consecutive entries that share cache lines,
    // instead of entries u, 4+u, 8+u, 12+u.  Trips are group-uniform (the
    // transpose reads all four lanes); the entry of (lane, u) in the trip
    // from k0 is k0 + 4u + lane.  Measured at 2.048 M atoms: FP64 fused
    // kernel 0.395 ms against 0.452; the 16-B fixed-point gathers gain
    // nothing (0.310 against 0.304), so Q keeps the lane's own chunk.
    constexpr bool TRANS = TPA == 4 && kTransLJ && !Q && !ACROSS;
    constexpr bool AHEAD = !TRANS && lj_ahead(TPA);
    int4 pre = make_int4(0, 0, 0, 0);  // AHEAD: the lane's next chunk
    if (AHEAD && 4 * lane < jn) pre = nb4[(size_t)lane * npad];
    for (int kt = TRANS ? 0 : 4 * lane; kt < jn; kt += NS * U * TPA) {
#pragma unroll
      for (int h = 0; h < NS; h++) {  // trip h of NS adds into set h
        const int k0 = kt + h * U * TPA;
        if (h > 0 && k0 >= jn) break;
        int jc[U];
        double4 xj[Q ? 1 : U];
        int4 qj[Q ? U : 1];
        if constexpr (TRANS) {
          int ev[4] = {self, self, self, self};
          if (k0 + 4 * lane < jn) {  // chunks past the row may lie past the list's capacity
            const int4 e4 = nb4[(size_t)((k0 >> 2) + lane) * npad];
            ev[0] = e4.x;
            ev[1] = e4.y;
            ev[2] = e4.z;
            ev[3] = e4.w;
          }
          quad_transpose(ev, lane);
#pragma unroll
          for (int u = 0; u < U; u++) jc[u] = k0 + 4 * u + lane < jn ? ev[u] : self;
        } else {
          const int4 e4 = AHEAD ? pre : nb4[(size_t)(k0 >> 2) * npad];
          const int ev[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
          for (int u = 0; u < U; u++) jc[u] = k0 + u < jn ? ev[u] : self;
          if (AHEAD && k0 + U * TPA < jn) pre = nb4[(size_t)((k0 + U * TPA) >> 2) * npad];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          if (Q) qj[u] = gather_q(xq, jc[u]);
          else xj[Q ? 0 : u] = gather_x(x, jc[u]);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          // entries carry image bits: test the index, not the sign
          if ((TRANS ? k0 + 4 * u + lane : k0 + u) >= jn) continue;
          double delx, dely, delz, rsq;
          int t;
          bool inside;
          if (Q) {
            delx = qdelta(qi.x, qj[u].x, qs.step[0]);
            dely = qdelta(qi.y, qj[u].y, qs.step[1]);
            delz = qdelta(qi.z, qj[u].z, qs.step[2]);
            rsq = delx * delx + dely * dely + delz * delz;
            t = ONE ? nt1 + 1 : row + qj[u].w;
            inside = rsq < (HOIST ? o_clo : s_clo[t]);
            if (!inside && rsq < (HOIST ? o_chi : s_chi[t])) {
              double ex, ey, ez;
              pair_delta(x[i], x[jc[u] & MDX_IDX_MASK], (unsigned)jc[u] >> MDX_IDX_BITS, px, py, pz, ex, ey, ez);
              inside = ex * ex + ey * ey + ez * ez < (HOIST ? o_cut : s_cutsq[t]);
            }
          } else {
            pair_delta(xi, xj[Q ? 0 : u], (unsigned)jc[u] >> MDX_IDX_BITS, px, py, pz, delx, dely, delz);
            rsq = delx * delx + dely * dely + delz * delz;
            t = ONE ? nt1 + 1 : row + static_cast<int>(xj[Q ? 0 : u].w);
            inside = rsq < (HOIST ? o_cut : s_cutsq[t]);
          }
          if (inside) {
            double fpair, evdwl = 0.0;
            if (MIXED) {
              // hardware reciprocal (1 ulp): well inside the FP32 pair-math budget
              const float r2inv = __builtin_amdgcn_rcpf((float)rsq);
              const float r6inv = r2inv * r2inv * r2inv;
              const float forcelj = r6inv * ((HOIST ? o_f1 : f_lj1[t]) * r6inv - (HOIST ? o_f2 : f_lj2[t]));
              fpair = (double)(forcelj * r2inv);
              if (EV)
                evdwl = HOIST ? (double)(r6inv * (one.f3 * r6inv - one.f4) - one.foff)
                              : (double)(r6inv * (f_lj3[t] * r6inv - f_lj4[t]) - f_off[t]);
            } else {
              const double r2inv = 1.0 / rsq;
              const double r6inv = r2inv * r2inv * r2inv;
              const double forcelj = r6inv * ((HOIST ? o_lj1 : s_lj1[t]) * r6inv - (HOIST ? o_lj2 : s_lj2[t]));
              fpair = forcelj * r2inv;
              if (EV)
                evdwl = HOIST ? r6inv * (one.lj3 * r6inv - one.lj4) - one.off
                              : r6inv * (s_lj3[t] * r6inv - s_lj4[t]) - s_off[t];
            }
            fx[h] += delx * fpair;
            fy[h] += dely * fpair;
            fz[h] += delz * fpair;
            if (EV) {
              e += 0.5 * evdwl;
              virial_entry(w, ig.pervir, (unsigned)jc[u] >> MDX_IDX_BITS, px, py, pz, delx, dely, delz, fpair);
            }
          }
        }
      }
    }
  }
  if (Q && i < n && lane == 0) xi = x[i];
  finish_atom<TPA, EV, INTEG, kLateV, ACROSS>(i, i < n && lane == 0, xi, set_sum<NS>(fx), set_sum<NS>(fy),
                                              set_sum<NS>(fz), e, w, ig, vpre, hpre, f, partials);
}

// ------------------------------------------------------------------ EAM
// a pair inside the cutoff, for the FP64/mixed gathers (Q false) or the
// fixed-point gathers with the FP64 re-test near the cutoff (Q true)
template <bool Q>
__device__ __forceinline__ bool pair_inside(const double4 &xi, int i, const int4 &qi, const double4 *__restrict__ x,
                                            int entry, const double4 &xj, const int4 &qj, const QScale &qs,
                                            double px, double py, double pz, double cutsq, double clo, double chi,
                                            double &delx, double &dely, double &delz, double &rsq) {
  if (Q) {
    delx = qdelta(qi.x, qj.x, qs.step[0]);
    dely = qdelta(qi.y, qj.y, qs.step[1]);
    delz = qdelta(qi.z, qj.z, qs.step[2]);
    rsq = delx * delx + dely * dely + delz * delz;
    if (rsq < clo) return true;
    if (!(rsq < chi)) return false;
    double ex, ey, ez;
    pair_delta(x[i], x[entry & MDX_IDX_MASK], (unsigned)entry >> MDX_IDX_BITS, px, py, pz, ex, ey, ez);
    return ex * ex + ey * ey + ez * ez < cutsq;
  }
  pair_delta(xi, xj, (unsigned)entry >> MDX_IDX_BITS, px, py, pz, delx, dely, delz);
  rsq = delx * delx + dely * dely + delz * delz;
  return rsq < cutsq;
}

// TL (one type): the spline knots the kernel reads are copied into LDS first
// (dynamic shared memory), so a lookup is an LDS read instead of a cached
// global gather; same arithmetic.
template <bool MIXED, bool EV, int TPA, bool Q, bool ONE, bool TL>
__global__ MDX_EAM_BOUNDS(TL && !MIXED) void k_eam_rho(int n, int npad, int cap, double px, double py, double pz, EAMArgs a,
                                                const double4 *__restrict__ x, const int4 *__restrict__ xq, QScale qs,
                                                const int *__restrict__ nbr, const int *__restrict__ numneigh,
                                                double *__restrict__ rho_out, double *__restrict__ fp_out,
                                                double *__restrict__ eemb, void *__restrict__ xf, StepGate gate) {
  static_assert(!TL || ONE, "LDS tables hold the one table of a single-type system");
  if (gate_closed(gate)) return;
  // type map in LDS: a kernel-argument array indexed per lane is a memory read
  __shared__ int s_t2r[kNT2];
  extern __shared__ float4 s_eam_tab[];  // TL: c3..c6 of knots 0..nr (FP64: two double2 each)
  [[maybe_unused]] double2 *const s_eam_tab64 = reinterpret_cast<double2 *>(s_eam_tab);
  for (int q = threadIdx.x; q < a.ntypes1 * a.ntypes1; q += blockDim.x) s_t2r[q] = a.type2rhor[q];
  if constexpr (TL) {
    const size_t kn = (size_t)(a.nr + 1), t = a.type2rhor[a.ntypes1 + 1];
    if constexpr (MIXED) {
      for (int m = threadIdx.x; m < (int)kn; m += blockDim.x) s_eam_tab[m] = a.rhor_pf[2 * (t * kn + m) + 1];
    } else {
      const double2 *src = reinterpret_cast<const double2 *>(a.rhor_p + 2 * t * kn);
      for (int q = threadIdx.x; q < 2 * (int)kn; q += blockDim.x) s_eam_tab64[q] = src[4 * (q >> 1) + 2 + (q & 1)];
    }
  }
  __syncthreads();
  const int i = (xcd_block() * blockDim.x + threadIdx.x) / TPA;
  const int lane = threadIdx.x % TPA;
  constexpr int NS = split_sums(MIXED, TPA) ? 2 : 1;
  double rhos[NS] = {};
  int ti = 0;
  double4 xi = make_double4(0.0, 0.0, 0.0, 0.0);
  int4 qi = make_int4(0, 0, 0, 0);
  const double clo = a.clo, chi = a.chi;  // kernel arguments: scalar registers
  if (i < n) {
    if (Q) qi = xq[i];
    else xi = x[i];
    ti = Q ? qi.w : static_cast<int>(xi.w);
    const int jn = numneigh[i];
    constexpr int U = Q ? kUnrollQ : kUnroll;
    constexpr int KS = TPA;  // entry stride within a trip
    const int self = i | (MDX_NOSHIFT << MDX_IDX_BITS);
    for (int k0 = lane; k0 < jn; k0 += U * TPA) {
      int jc[U];
      double4 xj[Q ? 1 : U];
      int4 qj[Q ? U : 1];
#pragma unroll
      for (int u = 0; u < U; u++)
        jc[u] = (k0 + u * KS < jn) ? list_entry(nbr + list_index(i, k0 + u * KS, npad)) : self;
#pragma unroll
      for (int u = 0; u < U; u++) {
        if (Q) qj[u] = gather_q(xq, jc[u]);
        else xj[Q ? 0 : u] = gather_x(x, jc[u]);
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        if (k0 + u * KS >= jn) continue;  // entries carry image bits: test the index, not the sign
        double delx, dely, delz, rsq;
        if (pair_inside<Q>(xi, i, qi, x, jc[u], xj[Q ? 0 : u], qj[Q ? u : 0], qs, px, py, pz, a.cutforcesq, clo, chi,
                           delx, dely, delz, rsq)) {
          const int tj = Q ? qj[Q ? u : 0].w : static_cast<int>(xj[Q ? 0 : u].w);
          if constexpr (TL) {
            int m;
            if constexpr (MIXED) {
              float p;
              (void)eam_index_mixed(rsq, a.rdr, a.nr, m, p);
              rhos[u % NS] += (double)eam_rho_eval(s_eam_tab[m], p);
            } else {
              double p, r, ri;
              sqrt_and_inverse(rsq, r, ri);
              eam_spline_index<double>(r, a.rdr, a.nr, m, p);
              const double2 c0 = s_eam_tab64[2 * m], c1 = s_eam_tab64[2 * m + 1];
              rhos[u % NS] += ((c0.x * p + c0.y) * p + c1.x) * p + c1.y;
            }
          } else {
            rhos[u % NS] += eam_rho_term<MIXED>(a, s_t2r[ONE ? a.ntypes1 + 1 : tj * a.ntypes1 + ti], rsq);
          }
        }
      }
    }
  }
  const double rho = group_sum<TPA>(set_sum<NS>(rhos));
  if (i < n && lane == 0) {
    // fp pass (pair_eam.cpp:213-228), FP64 in both modes: one per atom
    double p = rho * a.rdrho + 1.0;
    int m = static_cast<int>(p);
    m = max(1, min(m, a.nrho - 1));
    p -= m;
    p = fmin(p, 1.0);
    const double *c = a.frho + ((size_t)a.type2frho[ti] * (a.nrho + 1) + m) * 7;
    const double fpi = (c[0] * p + c[1]) * p + c[2];
    rho_out[i] = rho;
    fp_out[i] = fpi;
    // a single type: the force pass gathers the position with fp in the type's
    // place (mixed: rounded as its pair arithmetic rounds it), one load per
    // pair for two.  rho + force, us: 256,000 atoms mixed 82.4 to 79.0, FP64
    // 105 to 99.6; 2,048,000 FP64 909 to 866; 32,000 FP64 23.3 to 22.5
    if constexpr (ONE) {
      if constexpr (Q) static_cast<int4 *>(xf)[i] = make_int4(qi.x, qi.y, qi.z, __float_as_int((float)fpi));
      else static_cast<double4 *>(xf)[i] = make_double4(xi.x, xi.y, xi.z, fpi);
    }
    if (EV) {
      double phi = ((c[3] * p + c[4]) * p + c[5]) * p + c[6];
      if (rho > a.rhomax) phi += fpi * (rho - a.rhomax);
      eemb[i] = phi;
    }
  }
}

template <bool MIXED, bool EV, int TPA, bool INTEG, bool Q, bool ONE, bool TL>
__global__ MDX_EAM_BOUNDS(TL && !MIXED) void k_eam_force(int n, int npad, int cap, double px, double py, double pz,
                                                  EAMArgs a, const double4 *__restrict__ x,
                                                  const int4 *__restrict__ xq, QScale qs,
                                                  const int *__restrict__ nbr, const int *__restrict__ numneigh,
                                                  const double *__restrict__ fp, const double *__restrict__ eemb,
                                                  const void *__restrict__ xf,
                                                  double4 *__restrict__ f, double *__restrict__ partials,
                                                  IntegArgs ig) {
  static_assert(!TL || ONE, "LDS tables hold the one table of a single-type system");
  if constexpr (INTEG) {
    if (gate_closed(ig.gate)) return;
  }
  // type maps in LDS: kernel-argument arrays indexed per lane are memory reads
  __shared__ int s_t2r[kNT2], s_t2z[kNT2];
  // TL: rho' c0..c2, z2' c0..c2 and z2 c3..c6 of knots 0..nr, one after the
  // other (mixed), or as five double2 per knot (FP64)
  extern __shared__ float4 s_eam_tab[];
  [[maybe_unused]] double2 *const s_eam_tab64 = reinterpret_cast<double2 *>(s_eam_tab);
  for (int q = threadIdx.x; q < a.ntypes1 * a.ntypes1; q += blockDim.x) {
    s_t2r[q] = a.type2rhor[q];
    s_t2z[q] = a.type2z2r[q];
  }
  const int kn = a.nr + 1;
  if constexpr (TL) {
    const size_t t = a.type2rhor[a.ntypes1 + 1], z = a.type2z2r[a.ntypes1 + 1];
    for (int m = threadIdx.x; m < kn; m += blockDim.x) {
      if constexpr (MIXED) {
        s_eam_tab[m] = a.rhor_pf[2 * (t * kn + m)];
        s_eam_tab[kn + m] = a.z2r_pf[2 * (z * kn + m)];
        s_eam_tab[2 * kn + m] = a.z2r_pf[2 * (z * kn + m) + 1];
      } else {
        const double4 rd = a.rhor_p[2 * (t * kn + m)], zd = a.z2r_p[2 * (z * kn + m)],
                      zv = a.z2r_p[2 * (z * kn + m) + 1];
        double2 *const d = s_eam_tab64 + 5 * m;
        d[0] = make_double2(rd.x, rd.y);
        d[1] = make_double2(rd.z, zd.x);
        d[2] = make_double2(zd.y, zd.z);
        d[3] = make_double2(zv.x, zv.y);
        d[4] = make_double2(zv.z, zv.w);
      }
    }
  }
  __syncthreads();
  const int i = (xcd_block() * blockDim.x + threadIdx.x) / TPA;
  const int lane = threadIdx.x % TPA;
  constexpr int NS = split_sums(MIXED, TPA) ? 2 : 1;
  double fx[NS] = {}, fy[NS] = {}, fz[NS] = {}, e = 0.0;
  double w[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  double4 xi = make_double4(0.0, 0.0, 0.0, 0.0);
  double4 vpre = make_double4(0.0, 0.0, 0.0, 0.0), hpre = vpre;
  if (INTEG && !kLateV && i < n && lane == 0) {
    vpre = ig.v[i];
    if (ig.check) hpre = ig.xhold[i];
  }
  const double clo = a.clo, chi = a.chi;  // kernel arguments: scalar registers
  if (i < n) {
    if (!Q) xi = x[i];  // Q reads it where it is used: the re-test, the end
    const int4 qi = Q ? xq[i] : make_int4(0, 0, 0, 0);
    const int ti = Q ? qi.w : static_cast<int>(xi.w);
    const double fpi = fp[i];
    const int jn = numneigh[i];
    constexpr int U = Q ? kUnrollQ : kUnroll;
    constexpr int KS = TPA;  // entry stride within a trip
    const int self = i | (MDX_NOSHIFT << MDX_IDX_BITS);
    for (int k0 = lane; k0 < jn; k0 += U * TPA) {
      int jc[U];
      double4 xjv[Q ? 1 : U];
      int4 qjv[Q ? U : 1];
      double fpjv[ONE ? 1 : U];
#pragma unroll
      for (int u = 0; u < U; u++)
        jc[u] = (k0 + u * KS < jn) ? list_entry(nbr + list_index(i, k0 + u * KS, npad)) : self;
#pragma unroll
      for (int u = 0; u < U; u++) {
        if (Q) qjv[u] = gather_q(ONE ? static_cast<const int4 *>(xf) : xq, jc[u]);
        else xjv[Q ? 0 : u] = gather_x(ONE ? static_cast<const double4 *>(xf) : x, jc[u]);
        if (!ONE) fpjv[ONE ? 0 : u] = gather_d(fp, jc[u]);
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
      if (k0 + u * KS >= jn) continue;  // entries carry image bits: test the index, not the sign
      double delx, dely, delz, rsq;
      if (pair_inside<Q>(xi, i, qi, x, jc[u], xjv[Q ? 0 : u], qjv[Q ? u : 0], qs, px, py, pz, a.cutforcesq, clo, chi,
                         delx, dely, delz, rsq)) {
        const double fpj = !ONE ? fpjv[ONE ? 0 : u] : Q ? (double)__int_as_float(qjv[Q ? u : 0].w) : xjv[Q ? 0 : u].w;
        const int tj = Q ? qjv[Q ? u : 0].w : static_cast<int>(xjv[Q ? 0 : u].w);
        const int tij = ONE ? a.ntypes1 + 1 : ti * a.ntypes1 + tj, tji = ONE ? tij : tj * a.ntypes1 + ti;
        double fpair, phi;
        if constexpr (TL) {
          int m;
          if constexpr (MIXED) {
            float p;
            const float r = eam_index_mixed(rsq, a.rdr, a.nr, m, p);
            const float4 ci = s_eam_tab[m];
            eam_pair_eval(ci, ci, s_eam_tab[kn + m], s_eam_tab[2 * kn + m], r, p, fpi, fpj, fpair, phi);
          } else {
            double r, recip, p;
            sqrt_and_inverse(rsq, r, recip);
            eam_spline_index<double>(r, a.rdr, a.nr, m, p);
            const double2 *const d = s_eam_tab64 + 5 * m;
            const double2 d0 = d[0], d1 = d[1], d2 = d[2], d3 = d[3], d4 = d[4];
            const double4 ci = make_double4(d0.x, d0.y, d1.x, 0.0);
            eam_pair_eval64(ci, ci, make_double4(d1.y, d2.x, d2.y, 0.0), make_double4(d3.x, d3.y, d4.x, d4.y), recip,
                            p, fpi, fpj, fpair, phi);
          }
        } else {
          eam_pair_term<MIXED>(a, s_t2r[tij], s_t2r[tji], s_t2z[tij], rsq, fpi, fpj, fpair, phi);
        }
        fx[u % NS] += delx * fpair;
        fy[u % NS] += dely * fpair;
        fz[u % NS] += delz * fpair;
        if (EV) {
          e += 0.5 * phi;
          virial_entry(w, ig.pervir, (unsigned)jc[u] >> MDX_IDX_BITS, px, py, pz, delx, dely, delz, fpair);
        }
      }
      }
    }
    if (EV && lane == 0) e += eemb[i];
  }
  if (Q && i < n && lane == 0) xi = x[i];
  finish_atom<TPA, EV, INTEG, kLateV>(i, i < n && lane == 0, xi, set_sum<NS>(fx), set_sum<NS>(fy), set_sum<NS>(fz), e,
                                      w, ig, vpre, hpre, f, partials);
}

// Resident wavefronts per SIMD of the fused force kernels, held by giving
// each workgroup enough LDS that no more workgroups fit on a CU (160 KiB of
// LDS, four SIMDs).  The FP64 fused lj/cut kernel runs fastest held to 6
// (2.048 M atoms: 386 us at 5, 380 at 6, 389 at 7, 397 at its own 8; 256,000:
// 48.3, 46.5, 46.6, 47.0) once it has two rounds of them; below, the last
// round decides and all that fit run (108,000: 25.8, 26.9, 24.2, 24.6; 157,216:
// 32.0, 32.2, 32.0, 31.9).  The mixed one runs at the 7 that its registers
// allow (272 us; held to 6: 283, to 5: 311).  MDX_PAIR_WAVES sets a cap (0:
// none) on both and on the EAM passes.
constexpr long kChipSimds = 256 * 4;
int pair_wave_cap(int dflt) {
  static const int w = [] {
    const char *s = std::getenv("MDX_PAIR_WAVES");
    return s ? std::atoi(s) : -1;
  }();
  return w >= 0 ? w : dflt;
}

// Dynamic LDS of a launch: `used` bytes, or, under a wave cap, enough that
// the workgroup's whole LDS (the kernel's static LDS, from its attributes,
// plus this) lets at most 4 * cap / (B/64) workgroups share a CU's 160 KiB.
template <auto K>
size_t static_lds() {
  static const size_t v = [] {
    hipFuncAttributes attr{};
    return hipFuncGetAttributes(&attr, reinterpret_cast<const void *>(K)) == hipSuccess ? attr.sharedSizeBytes
                                                                                         : size_t(0);
  }();
  return v;
}

size_t occupancy_lds(size_t stat, int B, size_t used, int dflt) {
  const int w = pair_wave_cap(dflt);
  if (w <= 0) return used;
  const int per_block = (B + 63) / 64;
  const int blocks = std::max(1, 4 * w / per_block);
  const size_t total = ((size_t)(163840 / (blocks + 1)) + 256) & ~(size_t)255;
  return std::max(used, total > stat ? total - stat : 0);
}

template <bool MIXED, bool EV, int TPA, bool INTEG, bool Q, bool ONE>
void launch_lj_t(mdx_ctx *c, int B, const IntegArgs &ig) {
  const int G = xcd_grid(((long)c->n * TPA + B - 1) / B);
  prof_begin(c, INTEG ? MDX_K_FUSED : MDX_K_LJ);
  const int waves = !MIXED && (long)c->n * TPA > 2 * 6 * 64 * kChipSimds ? 6 : 0;
  const size_t lds = INTEG ? occupancy_lds(static_lds<k_lj<MIXED, EV, TPA, INTEG, Q, ONE>>(), B, 0, waves) : 0;
  LJOne one{};
  if (ONE) {
    const LJTab &t = c->lj_host;
    const int q = (c->ntypes + 1) + 1;
    one.clo = t.cutsq[q] * (1.0 - kBand);
    one.chi = t.cutsq[q] * (1.0 + kBand);
    one.cut = t.cutsq[q];
    one.lj1 = t.lj1[q];
    one.lj2 = t.lj2[q];
    one.lj3 = t.lj3[q];
    one.lj4 = t.lj4[q];
    one.off = t.offset[q];
    one.f1 = (float)t.lj1[q];
    one.f2 = (float)t.lj2[q];
    one.f3 = (float)t.lj3[q];
    one.f4 = (float)t.lj4[q];
    one.foff = (float)t.offset[q];
  }
  hipLaunchKernelGGL((k_lj<MIXED, EV, TPA, INTEG, Q, ONE>), dim3(G), dim3(B), lds, c->stream, c->n, c->npad, c->maxneigh,
                     c->ntypes + 1, c->prd[0], c->prd[1], c->prd[2], c->x, c->xq, c->qs, c->nbr, c->numneigh,
                     c->lj_dev, c->f, c->partials, ig, one);
  prof_end(c);
  c->last_grid = G;
}

// knots (nr+1) up to which the single-type tables go to LDS: the force pass
// holds three float4 per knot (48 KiB at this limit), or in FP64 five double2
// (62.5 KiB).  FP64 from LDS against gathers through L1: rho + force 23.1
// against 35.6 us at 32,000 atoms, 106 against 212 at 256,000.
constexpr int kEamLdsKnots = 1024, kEamLdsKnots64 = 800;

template <bool MIXED, bool EV, int TPA, bool INTEG, bool Q, bool ONE, bool TL>
void launch_eam_t(mdx_ctx *c, int B, const IntegArgs &ig) {
  const int G = xcd_grid(((long)c->n * TPA + B - 1) / B);
  const size_t kn = (size_t)c->eam.nr + 1;
  EAMArgs ea = c->eam;
  ea.clo = ea.cutforcesq * (1.0 - kBand);
  ea.chi = ea.cutforcesq * (1.0 + kBand);
  prof_begin(c, MDX_K_EAM_RHO);
  const size_t rho_bytes = TL ? kn * (MIXED ? sizeof(float4) : sizeof(double4)) : 0;
  hipLaunchKernelGGL((k_eam_rho<MIXED, EV, TPA, Q, ONE, TL>), dim3(G), dim3(B),
                     occupancy_lds(static_lds<k_eam_rho<MIXED, EV, TPA, Q, ONE, TL>>(), B, rho_bytes, 0), c->stream,
                     c->n, c->npad, c->maxneigh, c->prd[0], c->prd[1], c->prd[2], ea, c->x, c->xq, c->qs, c->nbr,
                     c->numneigh, c->rho, c->fp, c->eemb, c->xf, INTEG ? ig.gate : StepGate{});
  prof_end(c);
  IntegArgs fi = ig;
  fi.gate.decided = nullptr;  // the density pass has told the host
  prof_begin(c, INTEG ? MDX_K_FUSED : MDX_K_EAM_FORCE);
  const size_t tl_bytes = TL ? kn * (MIXED ? 3 * sizeof(float4) : 5 * sizeof(double2)) : 0;
  const size_t lds =
      INTEG ? occupancy_lds(static_lds<k_eam_force<MIXED, EV, TPA, INTEG, Q, ONE, TL>>(), B, tl_bytes, 0) : tl_bytes;
  hipLaunchKernelGGL((k_eam_force<MIXED, EV, TPA, INTEG, Q, ONE, TL>), dim3(G), dim3(B), lds, c->stream, c->n, c->npad,
                     c->maxneigh, c->prd[0], c->prd[1], c->prd[2], ea, c->x, c->xq, c->qs, c->nbr, c->numneigh, c->fp,
                     c->eemb, c->xf, c->f, c->partials, fi);
  prof_end(c);
  c->last_grid = G;
}

// whether the eam kernels take the LDS tables of a single-type system
bool eam_lds_tables(const mdx_ctx *c, int tpa) {
  return c->ntypes == 1 && (tpa == 4 || tpa == 8 || tpa == 16) &&
         c->eam.nr + 1 <= (c->precision == MDX_MIXED ? kEamLdsKnots : kEamLdsKnots64);
}

template <bool MIXED, bool EV, int TPA, bool INTEG, bool Q>
void launch_lj(mdx_ctx *c, int B, const IntegArgs &ig) {
  if constexpr (TPA == 4 || TPA == 8 || TPA == 16) {
    if (c->ntypes == 1) return launch_lj_t<MIXED, EV, TPA, INTEG, Q, true>(c, B, ig);
  }
  launch_lj_t<MIXED, EV, TPA, INTEG, Q, false>(c, B, ig);
}

template <bool MIXED, bool EV, int TPA, bool INTEG, bool Q>
void launch_eam(mdx_ctx *c, int B, const IntegArgs &ig) {
  if constexpr (TPA == 4 || TPA == 8 || TPA == 16) {
    if (c->ntypes == 1) {
      if (eam_lds_tables(c, TPA)) return launch_eam_t<MIXED, EV, TPA, INTEG, Q, true, true>(c, B, ig);
      return launch_eam_t<MIXED, EV, TPA, INTEG, Q, true, false>(c, B, ig);
    }
  }
  launch_eam_t<MIXED, EV, TPA, INTEG, Q, false, false>(c, B, ig);
}

template <bool MIXED, bool EV, bool INTEG, bool Q>
int dispatch_tpa(mdx_ctx *c, const Launch &l, const IntegArgs &ig) {
  const int B = l.block;
  const bool lj = c->pair_style == MDX_PAIR_LJ;
  switch (l.tpa) {
    case 1: lj ? launch_lj<MIXED, EV, 1, INTEG, Q>(c, B, ig) : launch_eam<MIXED, EV, 1, INTEG, Q>(c, B, ig); break;
    case 2: lj ? launch_lj<MIXED, EV, 2, INTEG, Q>(c, B, ig) : launch_eam<MIXED, EV, 2, INTEG, Q>(c, B, ig); break;
    case 4: lj ? launch_lj<MIXED, EV, 4, INTEG, Q>(c, B, ig) : launch_eam<MIXED, EV, 4, INTEG, Q>(c, B, ig); break;
    case 8: lj ? launch_lj<MIXED, EV, 8, INTEG, Q>(c, B, ig) : launch_eam<MIXED, EV, 8, INTEG, Q>(c, B, ig); break;
    case 16: lj ? launch_lj<MIXED, EV, 16, INTEG, Q>(c, B, ig) : launch_eam<MIXED, EV, 16, INTEG, Q>(c, B, ig); break;
    case 32: lj ? launch_lj<MIXED, EV, 32, INTEG, Q>(c, B, ig) : launch_eam<MIXED, EV, 32, INTEG, Q>(c, B, ig); break;
    default:
      set_error("threads per atom must be one of 1, 2, 4, 8, 16, 32");
      return MDX_ERR_ARG;
  }
  return MDX_OK;
}

template <bool INTEG>
int dispatch_prec(mdx_ctx *c, int ev, const IntegArgs &ig) {
  const Launch l = pair_launch(c);
  if (c->precision == MDX_MIXED) {
    if (c->qpos) {
      int rc = refresh_xq(c);
      if (rc) return rc;
      return ev ? dispatch_tpa<true, true, INTEG, true>(c, l, ig) : dispatch_tpa<true, false, INTEG, true>(c, l, ig);
    }
    return ev ? dispatch_tpa<true, true, INTEG, false>(c, l, ig) : dispatch_tpa<true, false, INTEG, false>(c, l, ig);
  }
  return ev ? dispatch_tpa<false, true, INTEG, false>(c, l, ig) : dispatch_tpa<false, false, INTEG, false>(c, l, ig);
}

}  // namespace

// Launch shape where the caller set none.  Few lanes per atom do the least
// work (fewer partial sums, longer index chunks) and win once they fill the
// chip; below that more lanes per atom shorten the one chain of dependent
// loads that a small launch consists of.  Measured per step kernel (us, lanes
// 4 / 8 / 16 / 32 per atom, FP64):
//   lj/cut            500 atoms  7.9 /  5.3 /  4.7 /  4.4
//                   4,000        7.5 /  5.3 /  4.8 /  5.0
//                  32,000       10.8 / 10.3 / 12.2 / 15.2  (mixed 7.8 / 7.6)
//                  42,592       12.1 / 13.3 / 15.4 / 19.8  (mixed 9.0 / 9.3)
//                 108,000       24.6 / 26.8 / 32.8 / 47    (mixed 17.1 / 19.0)
//               2,048,000        380 /  447 /  591 /  967  (mixed  272 /  329)
//   Kob-Andersen    2,744        9.9 /  6.5 /  5.4 /  4.9
//                   8,000       10.6 /  6.8 /  6.1 /  6.2
//   eam (rho+force)   500       19.3 / 14.6 / 12.2 / 10.5
//                   4,000       19.6 / 14.7 / 12.4 / 12.6
//                  13,500       22.3 / 16.3 / 17.4 / 24.2
//                 108,000         55 /   58 /   89 /  136
// By default mixed precision takes only 8 and 4, which give the same bits
// (split_sums): a mixed trajectory amplifies any other difference to its own
// error.  A shape that is set, or found by the autotuner, may be another.
// Workgroups of one wavefront spread a small launch evenly over the CUs
// (13,500 lj/cut atoms at 8 lanes: 64 threads 14% faster than 256); with 1024 or more
// workgroups of 256 there is nothing to gain.  The single-type eam kernels
// copy their spline tables to LDS once per workgroup, so they keep 256 (mixed,
// 13,500 atoms: 15.9 against 22.1 us), and 512 for the larger FP64 tables
// above 10,000 atoms (32,000: 23.1 against 24.7 us, 665,500: 269 against 283;
// 1024: 283).
Launch pair_launch(const mdx_ctx *c) {
  Launch l = c->launch;
  const bool mixed = c->precision == MDX_MIXED;
  if (!l.tpa) l.tpa = c->n > 40000 ? 4 : c->n > 10000 || mixed ? 8 : c->n > 3000 ? 16 : 32;
  if (!l.block) {
    const bool tables = c->pair_style == MDX_PAIR_EAM && eam_lds_tables(c, l.tpa);
    l.block = tables ? (mixed || c->n <= 10000 ? 256 : 512) : (long)c->n * l.tpa < 1024L * 256 ? 64 : 256;
  }
  // a shape that was set: only the FP64 eam kernels with LDS tables take 512
  if (l.block > 256 && (mixed || c->pair_style != MDX_PAIR_EAM || !eam_lds_tables(c, l.tpa))) l.block = 256;
  return l;
}

// Pair::compute on the device.  With `ig` the force
// kernel also runs fix nve's final integrate of this step and, if ig->next,
// the initial integrate of the next one (positions go to ig->xn).  ev: 0
// forces only, 1 also energy and global virial, 2 also the per-atom virial;
// with ev the reduction's slots are {eng_vdwl, virial[6], sum m v^2 (fused
// only)}.
int pair_compute(mdx_ctx *c, int ev, const IntegArgs *ig, const PairOut *out, bool wait) {
  if (c->n == 0) {  // no atoms: zero energy, virial and kinetic sums
    for (int k = 0; k < MDX_RED_SLOTS; k++) c->red_host[k] = 0.0;
    return MDX_OK;
  }
  if (c->pair_style != MDX_PAIR_LJ && c->pair_style != MDX_PAIR_EAM) {
    set_error("no pair style set");
    return MDX_ERR_ARG;
  }
  int rc;
  const int nslots = 8;
  IntegArgs args = ig ? *ig : IntegArgs{};
  args.pervir = ev >= 2 ? 1 : 0;
  if (out) args.out = *out;
  if (ig) rc = dispatch_prec<true>(c, ev, args);
  else rc = dispatch_prec<false>(c, ev, args);
  if (rc) return rc;
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "pair kernel launch");
  // the per-atom energy in f.w already includes the EAM embedding term
  if (ev) return finish_reduction(c, c->last_grid, nslots, wait);
  return MDX_OK;
}

}  // namespace mdx
