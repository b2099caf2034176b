// integrate.hip - fix nve, the rebuild trigger, reductions and host<->device
// reordering for gfx950.
//
// FixNVE::initial_integrate / final_integrate (src/fix_nve.cpp:65-142) run
// one thread per atom on the FP64 x, v, f; contraction is disabled so the
// updates round exactly as the reference's  v += dtfm*f;  x += dtv*v.
// On steps where Neighbor::decide would call check_distance
// (src/neighbor.cpp:1294-1372) the initial-integrate kernel also tests
// |x - xhold|^2 > (skin/2)^2 and raises a device flag, so the trigger costs
// no extra pass over x.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <limits>
#include <thread>
#include <vector>
#include "mdx_internal.h"
#include "piece_gate.h"

namespace mdx {

namespace {

struct MassTab {
  double m[MDX_NT1];
};

__global__ __launch_bounds__(256) void k_nve_initial(int n, MassTab mt, double dtv, double dtf,
                                                    double4 *__restrict__ x, double4 *__restrict__ v,
                                                    const double4 *__restrict__ f,
                                                    const double4 *__restrict__ xhold, int check,
                                                    double triggersq, int *__restrict__ trig,
                                                    int *__restrict__ trig_dev, int stamp,
                                                    int4 *__restrict__ xq, QScale qs) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double4 p = x[i];
  double4 q = v[i];
  const double4 fi = f[i];
  const double dtfm = dtf / mt.m[static_cast<int>(p.w)];
  q.x += dtfm * fi.x;
  q.y += dtfm * fi.y;
  q.z += dtfm * fi.z;
  p.x += dtv * q.x;
  p.y += dtv * q.y;
  p.z += dtv * q.z;
  x[i] = p;
  v[i] = q;
  if (xq) xq[i] = quantize(qs, p);
  if (check) {
    const double4 h = xhold[i];
    const double dx = p.x - h.x, dy = p.y - h.y, dz = p.z - h.z;
    const double rsq = dx * dx + dy * dy + dz * dz;
    mark_trigger(rsq > triggersq, trig, trig_dev, stamp);
  }
}

__global__ __launch_bounds__(256) void k_nve_final(int n, MassTab mt, double dtf, const double4 *__restrict__ x,
                                                  double4 *__restrict__ v, const double4 *__restrict__ f) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double4 q = v[i];
  const double4 fi = f[i];
  const double dtfm = dtf / mt.m[static_cast<int>(x[i].w)];
  q.x += dtfm * fi.x;
  q.y += dtfm * fi.y;
  q.z += dtfm * fi.z;
  v[i] = q;
}

// sum_i m_i |v_i|^2 (ComputeTemp::compute_scalar, compute_temp.cpp:71-95)
__global__ __launch_bounds__(256) void k_ke(int n, MassTab mt, const double4 *__restrict__ x,
                                           const double4 *__restrict__ v, double *__restrict__ partials) {
  __shared__ double s[16];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double t = 0.0;
  if (i < n) {
    const double4 q = v[i];
    t = (q.x * q.x + q.y * q.y + q.z * q.z) * mt.m[static_cast<int>(x[i].w)];
  }
  for (int off = 32; off > 0; off >>= 1) t += __shfl_down(t, off, 64);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    double acc = 0.0;
    for (int q = 0; q < (int)(blockDim.x + 63) / 64; q++) acc += s[q];
    partials[blockIdx.x] = acc;
  }
}

// Fixed-order reduction of per-block records [nrec][nslots], nslots <=
// MDX_RED_SLOTS: block r sums records [r*per, min((r+1)*per, nrec)) (a
// thread reads whole records start + t, start + t + 256, ..., then a fixed
// tree per slot) into record r of `out`.  One block with per = nrec is the
// whole reduction; many blocks are its first level.
__global__ __launch_bounds__(256) void k_reduce_records(const double *__restrict__ rec, int nrec, int nslots, int per,
                                                       double *__restrict__ out) {
  __shared__ double s[MDX_RED_SLOTS][256];
  double acc[MDX_RED_SLOTS];
#pragma unroll
  for (int k = 0; k < MDX_RED_SLOTS; k++) acc[k] = 0.0;
  const long start = (long)blockIdx.x * per, end = min((long)nrec, start + per);
  for (long b = start + threadIdx.x; b < end; b += 256) {
    const double *r = rec + (size_t)b * nslots;
#pragma unroll
    for (int k = 0; k < MDX_RED_SLOTS; k++)
      if (k < nslots) acc[k] += r[k];
  }
#pragma unroll
  for (int k = 0; k < MDX_RED_SLOTS; k++) s[k][threadIdx.x] = acc[k];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
#pragma unroll
      for (int k = 0; k < MDX_RED_SLOTS; k++) s[k][threadIdx.x] += s[k][threadIdx.x + w];
    __syncthreads();
  }
  if ((int)threadIdx.x < nslots) out[(size_t)blockIdx.x * nslots + threadIdx.x] = s[threadIdx.x][0];
}

// caller-order positions (device or mapped host memory) -> device (sorted)
// order, type kept in w
__global__ void k_scatter_x(int n, const double *__restrict__ hx, const int *__restrict__ orig,
                            double4 *__restrict__ x, int4 *__restrict__ xq, QScale qs) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int o = orig[i];
  double4 p = x[i];
  p.x = hx[3 * o];
  p.y = hx[3 * o + 1];
  p.z = hx[3 * o + 2];
  x[i] = p;
  if (xq) xq[i] = quantize(qs, p);
}

// the caller's arrays as uploaded -> a context's atoms in caller order (v, tag
// may be null: zero velocities, tags 1..n); forces are cleared up to npad
__global__ void k_load_atoms(int n, int npad, const double *__restrict__ hx, const double *__restrict__ hv,
                             const int *__restrict__ type, const int *__restrict__ htag, int img0,
                             double4 *__restrict__ x, double4 *__restrict__ v, double4 *__restrict__ f,
                             int *__restrict__ tag, int *__restrict__ orig, int *__restrict__ inv,
                             int *__restrict__ image) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npad) return;
  f[i] = make_double4(0.0, 0.0, 0.0, 0.0);
  if (i >= n) return;
  const size_t k = 3 * (size_t)i;
  x[i] = make_double4(hx[k], hx[k + 1], hx[k + 2], (double)type[i]);
  v[i] = hv ? make_double4(hv[k], hv[k + 1], hv[k + 2], 0.0) : make_double4(0.0, 0.0, 0.0, 0.0);
  tag[i] = htag ? htag[i] : i + 1;
  orig[i] = i;
  inv[i] = i;
  image[i] = img0;
}

// a context's atoms -> caller-order arrays (device or mapped host memory;
// null: not wanted), the image counts unpacked to three ints
__global__ void k_store_atoms(int n, const int *__restrict__ orig, const double4 *__restrict__ x,
                              const double4 *__restrict__ v, const double4 *__restrict__ f,
                              const int *__restrict__ image, double *__restrict__ ox, double *__restrict__ ov,
                              double *__restrict__ of, int *__restrict__ oi) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t k = 3 * (size_t)orig[i];
  auto put = [k](double *o, const double4 &p) {
    o[k] = p.x;
    o[k + 1] = p.y;
    o[k + 2] = p.z;
  };
  if (ox) put(ox, x[i]);
  if (ov) put(ov, v[i]);
  if (of) put(of, f[i]);
  if (oi) {
    const int im = image[i];
    oi[k] = (im & MDX_IMGMASK) - MDX_IMGMAX;
    oi[k + 1] = ((im >> 10) & MDX_IMGMASK) - MDX_IMGMAX;
    oi[k + 2] = (im >> 20) - MDX_IMGMAX;
  }
}

// fixed-point mirror of all positions (after a change of precision or
// position format)
__global__ void k_quantize(int n, const double4 *__restrict__ x, int4 *__restrict__ xq, QScale qs) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) xq[i] = quantize(qs, x[i]);
}

// device order -> caller order, one value per atom
__global__ void k_gather1(int n, const int *__restrict__ orig, const double *__restrict__ src,
                          double *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[orig[i]] = src[i];
}

// streaming copy of known size (HBM calibration: bytes moved = 2 * bytes)
__global__ __launch_bounds__(256) void k_copy(long n4, const double4 *__restrict__ src,
                                             double4 *__restrict__ dst) {
  const long stride = (long)gridDim.x * blockDim.x;
  for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n4; k += stride) dst[k] = src[k];
}

MassTab mass_tab(const mdx_ctx *c) {
  MassTab t;
  for (int k = 0; k < MDX_NT1; k++) t.m[k] = c->mass[k];
  return t;
}

}  // namespace

int nve_initial(mdx_ctx *c, double dtv, double dtf, int check) {
  if (c->n == 0) return MDX_OK;
  const int B = 256, G = (c->n + B - 1) / B;
  const int stamp = check ? next_trigger_stamp(c) : 0;
  prof_begin(c, MDX_K_NVE_INITIAL);
  hipLaunchKernelGGL(k_nve_initial, dim3(G), dim3(B), 0, c->stream, c->n, mass_tab(c), dtv, dtf, c->x, c->v, c->f,
                     c->xhold, check, c->triggersq, c->trig_host, c->trig_dev, stamp, c->qpos ? c->xq : nullptr, c->qs);
  prof_end(c);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? MDX_OK : hip_fail(e, "nve initial");
}

int nve_final(mdx_ctx *c, double dtf) {
  if (c->n == 0) return MDX_OK;
  const int B = 256, G = (c->n + B - 1) / B;
  prof_begin(c, MDX_K_NVE_FINAL);
  hipLaunchKernelGGL(k_nve_final, dim3(G), dim3(B), 0, c->stream, c->n, mass_tab(c), dtf, c->x, c->v, c->f);
  prof_end(c);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? MDX_OK : hip_fail(e, "nve final");
}

int neigh_check_displacement(mdx_ctx *c, int *flag) {
  hipError_t e = hipStreamSynchronize(c->stream);
  if (e != hipSuccess) return hip_fail(e, "trigger sync");
  *flag = __atomic_load_n(c->trig_host, __ATOMIC_ACQUIRE) == c->trig_stamp ? 1 : 0;
  return MDX_OK;
}

// Sum of the per-block records into red_host (mapped).  Many records (64,000 for the
// fused lj/cut kernel at 2.048 M atoms) are first reduced by up to 1024
// blocks of at least 256 contiguous records each, into the space after the
// records (partials_for holds it), then by one block: the partition depends only on nblocks, so the
// sums are reproducible.
int finish_reduction(mdx_ctx *c, int nblocks, int nslots, bool wait) {
  const int per = std::max(256, (nblocks + 1023) / 1024);
  const int nlev = (nblocks + per - 1) / per;
  if (nblocks > 2 * per) {
    double *lev = c->partials + (size_t)nblocks * nslots;
    hipLaunchKernelGGL(k_reduce_records, dim3(nlev), dim3(256), 0, c->stream, c->partials, nblocks, nslots, per, lev);
    hipLaunchKernelGGL(k_reduce_records, dim3(1), dim3(256), 0, c->stream, lev, nlev, nslots, nlev, c->red_host);
  } else {
    hipLaunchKernelGGL(k_reduce_records, dim3(1), dim3(256), 0, c->stream, c->partials, nblocks, nslots, nblocks,
                       c->red_host);
  }
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && wait) e = hipStreamSynchronize(c->stream);
  return e == hipSuccess ? MDX_OK : hip_fail(e, "reduction");
}

int reduce_ke(mdx_ctx *c) {
  if (c->n == 0) {
    c->red_host[0] = 0.0;
    return MDX_OK;
  }
  const int B = 256, G = (c->n + B - 1) / B;
  hipLaunchKernelGGL(k_ke, dim3(G), dim3(B), 0, c->stream, c->n, mass_tab(c), c->x, c->v, c->partials);
  return finish_reduction(c, G, 1);
}

// ---- transfers between the caller's arrays and the device
//
// Everything goes through the pinned stage in pieces: a piece's DMA overlaps
// the host's copies of its neighbours.  One thread copies about 10 GB/s, well
// under the link's rate, so transfers of 2 MiB and more are split over up to
// eight threads, each taking its slice of every piece.
constexpr size_t kPiece = size_t(2) << 20;
constexpr int kPiecesInFlight = 64;

struct Piece {
  char *host, *dev, *stage;
  size_t len;
  bool add;
};

static std::vector<Piece> pieces_of(const Seg *segs, int nseg, size_t &total) {
  std::vector<Piece> v;
  total = 0;
  for (int s = 0; s < nseg; s++)
    for (size_t off = 0; off < segs[s].bytes; off += kPiece) {
      const size_t len = std::min(kPiece, segs[s].bytes - off);
      v.push_back({(char *)segs[s].host + off, (char *)segs[s].dev + off, nullptr, len, segs[s].add});
      total += len;
    }
  return v;
}

// slice t of nt of `len` bytes, on whole 64-byte lines
static void slice(size_t len, int t, int nt, size_t &a, size_t &b) {
  const size_t per = ((len + nt - 1) / nt + 63) / 64 * 64;
  a = std::min(len, per * t);
  b = std::min(len, a + per);
}

void host_add(double *dst, const double *src, size_t count) {
  for (size_t k = 0; k < count; k++) dst[k] += src[k];
}

// Runs work(t, nt) on nt threads, the caller's among them as t = 0; fewer
// threads than asked for if the system gives no more.
template <typename W>
static void on_threads(size_t bytes, W &&work) {
  const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
  const int want = bytes < kPiece ? 1 : (int)std::min<size_t>(std::min(8u, hw), bytes >> 20);
  std::atomic<int> nt{0};
  std::vector<std::thread> pool;
  try {
    pool.reserve(want);
    for (int t = 1; t < want; t++)
      pool.emplace_back([&nt, &work, t] {
        int n;
        while (!(n = nt.load(std::memory_order_acquire))) std::this_thread::yield();
        work(t, n);
      });
  } catch (...) {
  }
  const int n = (int)pool.size() + 1;
  nt.store(n, std::memory_order_release);
  work(0, n);
  for (auto &th : pool) th.join();
}

int stage_ready(mdx_ctx *c) {
  if (!c->stage_busy) return MDX_OK;
  hipError_t e = hipStreamSynchronize(c->stream);
  if (e != hipSuccess) return hip_fail(e, "staging memory");
  c->stage_busy = false;
  return MDX_OK;
}

// the next pieces that fit the stage, from piece `first` on
static size_t place(mdx_ctx *c, std::vector<Piece> &v, size_t first) {
  const size_t cap = (size_t)(sizeof(double) * kStageDoubles * c->cap_atoms);
  size_t off = 0, k = first;
  for (; k < v.size() && k - first < (size_t)kPiecesInFlight && off + v[k].len <= cap; k++) {
    v[k].stage = (char *)c->host_stage + off;
    off += (v[k].len + 63) / 64 * 64;
  }
  return k;
}

int upload(mdx_ctx *c, const Seg *segs, int nseg) {
  size_t total;
  std::vector<Piece> v = pieces_of(segs, nseg, total);
  hipError_t e = hipSuccess;
  for (size_t first = 0, last; first < v.size(); first = last) {
    int rc = stage_ready(c);
    if (rc) return rc;
    if ((last = place(c, v, first)) == first) {
      set_error("staging memory too small");
      return MDX_ERR_ARG;
    }
    std::vector<std::atomic<int>> done(last - first);
    c->stage_busy = true;
    on_threads(total, [&](int t, int nt) {
      for (size_t k = first; k < last; k++) {
        size_t a, b;
        slice(v[k].len, t, nt, a, b);
        memcpy(v[k].stage + a, v[k].host + a, b - a);
        if (t) {
          done[k - first].fetch_add(1, std::memory_order_release);
        } else {
          while (done[k - first].load(std::memory_order_acquire) < nt - 1) std::this_thread::yield();
          if (e == hipSuccess) e = hipMemcpyAsync(v[k].dev, v[k].stage, v[k].len, hipMemcpyHostToDevice, c->stream);
        }
      }
    });
    if (e != hipSuccess) return hip_fail(e, "upload");
  }
  return MDX_OK;
}

int download(mdx_ctx *c, const Seg *segs, int nseg) {
  size_t total;
  std::vector<Piece> v = pieces_of(segs, nseg, total);
  hipError_t e = hipSuccess;
  for (size_t first = 0, last; first < v.size(); first = last) {
    if ((last = place(c, v, first)) == first) {
      set_error("staging memory too small");
      return MDX_ERR_ARG;
    }
    while (c->stage_ev.size() < last - first) {
      hipEvent_t ev;
      if ((e = hipEventCreateWithFlags(&ev, hipEventDisableTiming)) != hipSuccess) return hip_fail(e, "staging events");
      c->stage_ev.push_back(ev);
    }
    for (size_t k = first; k < last; k++)
      if ((e = hipMemcpyAsync(v[k].stage, v[k].dev, v[k].len, hipMemcpyDeviceToHost, c->stream)) != hipSuccess ||
          (e = hipEventRecord(c->stage_ev[k - first], c->stream)) != hipSuccess) {
        (void)hipStreamSynchronize(c->stream);
        return hip_fail(e, "download");
      }
    constexpr int kFailed = std::numeric_limits<int>::max();
    PieceGate gate;
    on_threads(total, [&](int t, int nt) {
      for (size_t k = first; k < last; k++) {
        const int piece = (int)(k - first);
        if (t == 0) {
          e = hipEventSynchronize(c->stage_ev[piece]);
          gate.raise(e == hipSuccess ? piece + 1 : kFailed);
        }
        if (gate.wait(piece) == kFailed) return;
        size_t a, b;
        slice(v[k].len, t, nt, a, b);
        if (v[k].add)
          host_add(reinterpret_cast<double *>(v[k].host + a), reinterpret_cast<const double *>(v[k].stage + a),
                   (b - a) / sizeof(double));
        else
          memcpy(v[k].host + a, v[k].stage + a, b - a);
      }
    });
    if (e != hipSuccess) return hip_fail(e, "download");
    c->stage_busy = false;  // the stream has passed everything queued before
  }
  return MDX_OK;
}

int scatter_positions(mdx_ctx *c, const double *host_x) {
  const int B = 256, G = (c->n + B - 1) / B;
  const size_t bytes = sizeof(double) * 3 * c->n;
  const double *src = c->dscratch;
  int rc;
  if (c->n <= kIoAtoms) {
    if ((rc = stage_ready(c))) return rc;
    memcpy(c->host_in, host_x, bytes);
    src = c->host_in;
    c->stage_busy = true;
  } else {
    const Seg seg{const_cast<double *>(host_x), c->dscratch, bytes, false};
    if ((rc = upload(c, &seg, 1))) return rc;
  }
  hipLaunchKernelGGL(k_scatter_x, dim3(G), dim3(B), 0, c->stream, c->n, src, c->orig, c->x, c->qpos ? c->xq : nullptr,
                     c->qs);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? MDX_OK : hip_fail(e, "positions scatter");
}

int load_atoms(mdx_ctx *c, const double *x, const double *v, const int *type, const int *tag) {
  const size_t n = (size_t)c->n, n3 = 3 * n;
  Seg segs[4];
  int ns = 0;
  segs[ns++] = {const_cast<double *>(x), c->dscratch, sizeof(double) * n3, false};
  if (v) segs[ns++] = {const_cast<double *>(v), c->dscratch + n3, sizeof(double) * n3, false};
  segs[ns++] = {const_cast<int *>(type), c->bidx, sizeof(int) * n, false};
  if (tag) segs[ns++] = {const_cast<int *>(tag), c->bidx_s, sizeof(int) * n, false};
  int rc = upload(c, segs, ns);
  if (rc) return rc;
  const int img0 = (MDX_IMGMAX << 20) | (MDX_IMGMAX << 10) | MDX_IMGMAX;
  const int B = 256, G = (c->npad + B - 1) / B;
  hipLaunchKernelGGL(k_load_atoms, dim3(G), dim3(B), 0, c->stream, c->n, c->npad, c->dscratch,
                     v ? c->dscratch + n3 : nullptr, c->bidx, tag ? c->bidx_s : nullptr, img0, c->x, c->v, c->f, c->tag,
                     c->orig, c->inv, c->image);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? MDX_OK : hip_fail(e, "atom upload");
}

int store_atoms(mdx_ctx *c, double *x, double *v, double *f, int *image) {
  const size_t n3 = 3 * (size_t)c->n;
  const bool small = c->n <= kIoAtoms;
  // x | v | f | image, in mapped host memory or in two device scratch arrays
  double *dx = small ? c->host_out : c->dscratch, *dv = dx + n3, *df = small ? dv + n3 : c->vatom;
  int *di = reinterpret_cast<int *>(df + n3);
  const int B = 256, G = (c->n + B - 1) / B;
  hipLaunchKernelGGL(k_store_atoms, dim3(G), dim3(B), 0, c->stream, c->n, c->orig, c->x, c->v, c->f, c->image,
                     x ? dx : nullptr, v ? dv : nullptr, f ? df : nullptr, image ? di : nullptr);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "atom download");
  Seg segs[4];
  int ns = 0;
  if (x) segs[ns++] = {x, dx, sizeof(double) * n3, false};
  if (v) segs[ns++] = {v, dv, sizeof(double) * n3, false};
  if (f) segs[ns++] = {f, df, sizeof(double) * n3, false};
  if (image) segs[ns++] = {image, di, sizeof(int) * n3, false};
  if (!small) return download(c, segs, ns);
  if ((e = hipStreamSynchronize(c->stream)) != hipSuccess) return hip_fail(e, "atom download");
  c->stage_busy = false;
  for (int k = 0; k < ns; k++) memcpy(segs[k].host, segs[k].dev, segs[k].bytes);
  return MDX_OK;
}

int refresh_xq(mdx_ctx *c) {
  if (!c->qpos || !c->xq_stale || c->n == 0) return MDX_OK;
  const int B = 256, G = (c->n + B - 1) / B;
  hipLaunchKernelGGL(k_quantize, dim3(G), dim3(B), 0, c->stream, c->n, c->x, c->xq, c->qs);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "fixed-point positions");
  c->xq_stale = false;
  return MDX_OK;
}

int copy_probe(mdx_ctx *c, long nbytes, int iters, double *gbs) {
  const long n4 = nbytes / (long)sizeof(double4);
  if (n4 <= 0 || iters <= 0) {
    set_error("copy probe needs nbytes >= 32 and iters >= 1");
    return MDX_ERR_ARG;
  }
  double4 *a = nullptr, *b = nullptr;
  if (hipMalloc(&a, sizeof(double4) * n4) != hipSuccess || hipMalloc(&b, sizeof(double4) * n4) != hipSuccess) {
    if (a) (void)hipFree(a);
    set_error("Insufficient memory on accelerator (copy probe)");
    return MDX_ERR_NOMEM;
  }
  const int B = 256, G = 256 * 32;  // 32 workgroups per CU on 256 CUs
  hipEvent_t e0 = nullptr, e1 = nullptr;
  float ms = 0.0f;
  hipError_t e = hipMemsetAsync(a, 0, sizeof(double4) * n4, c->stream);
  if (e == hipSuccess) e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_copy, dim3(G), dim3(B), 0, c->stream, n4, a, b);  // warm-up
    e = hipEventRecord(e0, c->stream);
  }
  if (e == hipSuccess) {
    for (int it = 0; it < iters; it++) hipLaunchKernelGGL(k_copy, dim3(G), dim3(B), 0, c->stream, n4, a, b);
    e = hipEventRecord(e1, c->stream);
  }
  if (e == hipSuccess) e = hipEventSynchronize(e1);
  if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  (void)hipFree(a);
  (void)hipFree(b);
  if (e != hipSuccess) return hip_fail(e, "copy probe");
  *gbs = 2.0 * sizeof(double4) * (double)n4 * iters / (ms * 1e-3) / 1e9;
  return MDX_OK;
}

int gather_value(mdx_ctx *c, const double *dev, double *host_out) {
  const int B = 256, G = (c->n + B - 1) / B;
  hipLaunchKernelGGL(k_gather1, dim3(G), dim3(B), 0, c->stream, c->n, c->orig, dev, c->dscratch);
  const Seg seg{host_out, c->dscratch, sizeof(double) * c->n, false};
  return download(c, &seg, 1);
}

}  // namespace mdx
