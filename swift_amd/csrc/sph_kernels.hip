// sph_kernels.hip -- gfx950 kernels of the SPHENIX neighbour pass.
//
// Data layout (HBM, particles sorted by top-level cell):
//   px,py,pz double, vx..h float, tb int8: structure of arrays, read by the
//   per-particle kernels (ghost, extra ghost, end force);
//   DensRec / GradRec / ForceRec: one packed record per particle with the
//   fields a neighbour loop reads from particle j (sph_kernels.h), rebuilt
//   after the stage that changes them.
//
// The neighbour loops are in sph_gather.h (engine) and sph_loops.h (the
// three interaction bodies); this file holds the record builders, the
// per-particle kernels of the ghosts and the launchers.
#include <atomic>
#include "sph_device.h"
#include "sph_kernels.h"
#include "sph_loops.h"
#include "sph_ghost.h"
#include "sph_gather.h"
#include "sph_sparse.h"
#include "sph_tile.h"

using namespace sph;
using namespace sphl;

namespace {

// ------------------------------------------------------ neighbour records --
// Thread = record slot j of a cell-aligned slot range (its particle is the
// field slot soa[j] with two slot orders, in the same cells).
__global__ void k_build_pos(DevParts d, GridDesc g, float pos_eps, int lo,
                            int hi) {
  const int j = lo + blockIdx.x * blockDim.x + threadIdx.x;
  if (j < hi) d.pos[j] = pos_rec(d, g, pos_eps, field_slot(d, j));
}

// Bounding box (non-inhibited particles) and largest search radius of each
// chunk in [c0, c1); an empty chunk gets an inverted box that no test passes.
// A wave takes 64 / C chunks, one lane per particle, and reduces over the C
// lanes of each chunk; the largest radius of the block goes to *hg2_all with
// one atomic per block.
constexpr int kBoundsBlock = 1024;
__global__ __launch_bounds__(kBoundsBlock) void k_chunk_bounds(
    DevParts d, const int *chunk_start, int c0, int c1, int C, double *bbox,
    float *hg2max, unsigned int *hg2_all, GridDesc gd, float pos_eps,
    float4 *fbox) {
  __shared__ float wmax[kBoundsBlock / 64];
  const int lane = threadIdx.x & 63;
  const int wave = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  const int k = c0 + wave * (64 / C) + lane / C;
  const int g = lane % C;
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  float flo[3] = {3e38f, 3e38f, 3e38f}, fhi[3] = {-3e38f, -3e38f, -3e38f};
  float hm = 0.f, fh = -1.f;
  if (k < c1) {
    const int j = chunk_start[k] + g;
    const int i = j < chunk_start[k + 1] ? field_slot(d, j) : 0;
    if (j < chunk_start[k + 1] && d.tb[i] != kBinInhibited) {
      lo[0] = hi[0] = d.px[i];
      lo[1] = hi[1] = d.py[i];
      lo[2] = hi[2] = d.pz[i];
      hm = search_radius2(d.h[i]);
      if (fbox) {
        // the candidate's pre-test record, as k_build_pos forms it
        const PosRec p = pos_rec(d, gd, pos_eps, i);
        flo[0] = fhi[0] = p.x;
        flo[1] = fhi[1] = p.y;
        flo[2] = fhi[2] = p.z;
        fh = p.hg2m;
      }
    }
  }
  for (int off = 1; off < C; off <<= 1) {
    for (int a = 0; a < 3; a++) {
      lo[a] = fmin(lo[a], __shfl_xor(lo[a], off));
      hi[a] = fmax(hi[a], __shfl_xor(hi[a], off));
    }
    hm = fmaxf(hm, __shfl_xor(hm, off));
    if (fbox) {
      for (int a = 0; a < 3; a++) {
        flo[a] = fminf(flo[a], __shfl_xor(flo[a], off));
        fhi[a] = fmaxf(fhi[a], __shfl_xor(fhi[a], off));
      }
      fh = fmaxf(fh, __shfl_xor(fh, off));
    }
  }
  if (k < c1 && g == 0) {
    for (int a = 0; a < 3; a++) {
      bbox[6 * k + a] = lo[a];
      bbox[6 * k + 3 + a] = hi[a];
    }
    hg2max[k] = hm;
    if (fbox) {
      fbox[2 * k] = make_float4(flo[0], flo[1], flo[2], fh);
      fbox[2 * k + 1] = make_float4(fhi[0], fhi[1], fhi[2], 0.f);
    }
  }
  for (int off = 32; off >= C; off >>= 1) hm = fmaxf(hm, __shfl_xor(hm, off));
  if (lane == 0) wmax[threadIdx.x >> 6] = hm;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kBoundsBlock / 64; k++) hm = fmaxf(hm, wmax[k]);
    // positive floats order like their bit patterns
    // a plain read first: only a block that raises the maximum pays an
    // atomic (one per block on one address serialised the whole launch)
    if (__float_as_uint(hm) >
        __hip_atomic_load(hg2_all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(hg2_all, __float_as_uint(hm));
  }
}

// The radius part of k_chunk_bounds for chunks whose positions have not
// moved since their boxes were formed: the largest search radius (and, with
// fbox, the largest widened radius in fbox[2 k].w) of chunks [c0, c1), and
// with pos the widened radius of each member's pre-test record, as
// k_build_pos forms it.
__global__ __launch_bounds__(kBoundsBlock) void k_radius_bounds(
    DevParts d, const int *chunk_start, int c0, int c1, int C, float *hg2max,
    unsigned int *hg2_all, float pos_eps, float4 *fbox, PosRec *pos) {
  __shared__ float wmax[kBoundsBlock / 64];
  const int lane = threadIdx.x & 63;
  const int wave = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  const int k = c0 + wave * (64 / C) + lane / C;
  const int g = lane % C;
  float hm = 0.f, fh = -1.f;
  if (k < c1) {
    const int j = chunk_start[k] + g;
    if (j < chunk_start[k + 1]) {
      const int i = field_slot(d, j);
      const bool inh = d.tb[i] == kBinInhibited;
      if (!inh) {
        hm = search_radius2(d.h[i]);
        fh = pretest_radius2(hm, pos_eps);
      }
      if (pos) pos[j].hg2m = inh ? -1.f : fh;
    }
  }
  for (int off = 1; off < C; off <<= 1) {
    hm = fmaxf(hm, __shfl_xor(hm, off));
    fh = fmaxf(fh, __shfl_xor(fh, off));
  }
  if (k < c1 && g == 0) {
    hg2max[k] = hm;
    if (fbox) fbox[2 * k].w = fh;
  }
  for (int off = 32; off >= C; off >>= 1) hm = fmaxf(hm, __shfl_xor(hm, off));
  if (lane == 0) wmax[threadIdx.x >> 6] = hm;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k2 = 1; k2 < kBoundsBlock / 64; k2++) hm = fmaxf(hm, wmax[k2]);
    // a plain read first: only a block that raises the maximum pays an
    // atomic (one per block on one address serialised the whole launch)
    if (__float_as_uint(hm) >
        __hip_atomic_load(hg2_all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(hg2_all, __float_as_uint(hm));
  }
}

// Records of particles [lo, hi); with max_active_bin >= 0 only of the
// active ones (the others keep theirs), stored one by one.  For all
// particles of the range, each wave stages its 64 records in LDS and writes
// them out as contiguous 16-byte words (a record per lane would scatter
// every store instruction over the wave's whole span).
constexpr int kRecBlock = 256;

// Store words of a record type: 16 bytes, or 8 for records of 8-byte
// multiples.
template <class R>
using RecWord = typename std::conditional<sizeof(R) % 16 == 0, uint4,
                                          uint2>::type;

template <class R>
__device__ __forceinline__ void store_wave_records(R *dst, int i0, int cnt,
                                                   const R &r,
                                                   RecWord<R> *lds) {
  using W = RecWord<R>;
  constexpr int Q = (int)(sizeof(R) / sizeof(W));
  static_assert(sizeof(R) % 8 == 0, "records are whole 8-byte words");
  const int lane = threadIdx.x & 63;
  const W *src = reinterpret_cast<const W *>(&r);
#pragma unroll
  for (int q = 0; q < Q; q++) lds[lane * Q + q] = src[q];
  __syncthreads();
  W *out = reinterpret_cast<W *>(dst + i0);
  const int words = cnt * Q;
  for (int k = lane; k < words; k += 64) out[k] = lds[k];
}

// LDS written by lanes of one wave and read by others of the same wave: no
// block barrier (the waves of a block take different branches here).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class R, class Make>
__device__ __forceinline__ void build_records(const DevParts &d, R *dst,
                                              int lo, int hi, int mab,
                                              const int *list, const int *cnt,
                                              Make make) {
  using W = RecWord<R>;
  constexpr int Q = (int)(sizeof(R) / sizeof(W));
  __shared__ W buf[kRecBlock * sizeof(R) / sizeof(W)];
  if (mab >= 0) {  // uniform; launched with run_blocks(hi - lo, kRecBlock)
    if (list || d.cand) {  // record slots not contiguous: one by one
      auto one = [&](int i, int8_t tb) {
        if (is_active(tb, mab)) dst[rec_slot(d, i)] = make(i);
      };
      if (list)
        for_runs_list(list, cnt, d.tb, one);
      else
        for_runs(lo, hi, d.tb, one);
      return;
    }
    // kRuns runs a grid's width apart; a run whose 64 particles of a wave
    // are all active is staged in the wave's LDS and stored as contiguous
    // words, otherwise the active ones store their records one by one
    const int lane = threadIdx.x & 63;
    W *mine = buf + (threadIdx.x >> 6) * 64 * Q;
    const int base = lo + blockIdx.x * kRecBlock + threadIdx.x;
    const int stride = gridDim.x * kRecBlock;
    int8_t t[kRuns];
#pragma unroll
    for (int u = 0; u < kRuns; u++) {
      const int i = base + u * stride;
      t[u] = i < hi ? d.tb[i] : (int8_t)kBinInhibited;
    }
    for (int u = 0; u < kRuns; u++) {
      const int i = base + u * stride;
      const bool act = i < hi && is_active(t[u], mab);
      if (__ballot(act) == ~0ull) {  // uniform over the wave
        const R r = make(i);
        const W *src = reinterpret_cast<const W *>(&r);
#pragma unroll
        for (int q = 0; q < Q; q++) mine[lane * Q + q] = src[q];
        wave_lds_sync();
        W *out = reinterpret_cast<W *>(dst + (i - lane));
        for (int k = lane; k < 64 * Q; k += 64) out[k] = mine[k];
        wave_lds_sync();  // the next run reuses the wave's LDS
      } else if (act) {
        dst[i] = make(i);
      }
    }
    return;
  }
  // thread = record slot; with two slot orders its particle is the field
  // slot soa[j] (the same cells' slot range), so the stores stay contiguous
  const int j = lo + blockIdx.x * kRecBlock + threadIdx.x;
  R r{};
  if (j < hi) r = make(field_slot(d, j));
  const int w = threadIdx.x >> 6;
  const int i0 = lo + blockIdx.x * kRecBlock + (w << 6);
  store_wave_records(dst, i0, max(0, min(64, hi - i0)), r, buf + w * 64 * Q);
}

__global__ __launch_bounds__(kRecBlock) void k_build_dens_rec(
    DevParts d, int lo, int hi, int mab, const int *list, const int *cnt) {
  build_records(d, d.rd, lo, hi, mab, list, cnt,
                [&](int i) { return dens_rec(d, i); });
}

__global__ __launch_bounds__(kRecBlock) void k_build_grad_rec(
    DevParts d, int lo, int hi, int mab, const int *list, const int *cnt) {
  build_records(d, d.rg, lo, hi, mab, list, cnt,
                [&](int i) { return grad_rec(d, i); });
}

__global__ __launch_bounds__(kRecBlock) void k_build_force_rec(
    DevParts d, int lo, int hi, int mab, const int *list, const int *cnt) {
  build_records(d, d.rf, lo, hi, mab, list, cnt,
                [&](int i) { return force_rec(d, i); });
}

// ------------------------------------------------------ per-particle work --
// hydro_init_part (hydro.h:564-606) for active particles in [lo, hi); also
// resets the ghost bracket.
__global__ void k_init_density(DevParts d, int lo, int hi, int max_active_bin,
                               float h_max, const int *list, const int *cnt,
                               int light) {
  auto body = [&](int i, int8_t tb) {
    const bool act = is_active(tb, max_active_bin);
    d.redo[i] = act ? 1 : 0;
    d.lfb[i] = 0;
    if (!act) return;
    d.left[i] = 0.f;
    d.right[i] = h_max;
    if (light) return;
    d.rho[i] = 0.f;
    d.rho_dh[i] = 0.f;
    d.wc[i] = 0.f;
    d.wc_dh[i] = 0.f;
    d.divv[i] = 0.f;
    d.rotx[i] = 0.f;
    d.roty[i] = 0.f;
    d.rotz[i] = 0.f;
    d.nd[i] = 0;
    d.lapu[i] = 0.f;
  };
  if (list)
    for_runs_list(list, cnt, d.tb, body);
  else
    for_runs(lo, hi, d.tb, body);
}

// One ghost round (runner_do_ghost, runner_ghost.c:1113-1628) for the
// particles flagged in redo[] within [lo, hi): ghost_step on the density
// sums, and either convergence (prepare the gradient loop) or a
// re-initialised particle flagged for another density round.  `relist`
// tells whether the particle's neighbour list no longer covers its new
// search radius (for another round, or for the gradient loop once
// converged).
__device__ bool ghost_one(const DevParts &d, const GhostArgs &ga, int i,
                          bool &relist) {
  GhostState g{d.h[i], d.left[i], d.right[i]};
  DensSums a{d.rho[i], d.rho_dh[i], d.wc[i], d.wc_dh[i],
             d.divv[i], d.rotx[i], d.roty[i], d.rotz[i]};
  const bool again = ghost_step(ga, d.m[i], g, a);
  relist = !ga.lists || !(search_radius2(g.h) <= d.r2b[i]);
  if (again) {
    // Not converged: re-initialise (hydro_init_part) and ask for a rerun.
    d.h[i] = g.h;
    d.left[i] = g.left;
    d.right[i] = g.right;
    d.rho[i] = 0.f;
    d.rho_dh[i] = 0.f;
    d.wc[i] = 0.f;
    d.wc_dh[i] = 0.f;
    d.divv[i] = 0.f;
    d.rotx[i] = 0.f;
    d.roty[i] = 0.f;
    d.rotz[i] = 0.f;
    d.nd[i] = 0;
    return true;
  }
  if (ga.lists) d.lfb[i] = relist ? 1 : 0;
  ghost_finish(d, ga, i, g.h, a);
  return false;
}

// Counts are reduced over the block first: one atomic per block and
// counter keeps the same-address traffic small.  A block covers kRuns runs of
// kGhostBlock particles a grid's width apart (their redo flags loaded
// together); the particles that go again are appended to d.sel in block,
// wave, run, lane order.
constexpr int kGhostBlock = 256;
__global__ __launch_bounds__(kGhostBlock) void k_ghost(
    DevParts d, GhostArgs ga, int lo, int hi, int off, int nt,
    unsigned long long *counters, const int *list, const int *cnt) {
  constexpr int W = kGhostBlock / 64;
  __shared__ int wcnt[3][W];
  __shared__ unsigned long long wwork[W];
  __shared__ int base;
  // run u of this thread: particle slot i0 + u * stride, or with a compact
  // list the particle of list entry k0 + u * stride
  const int i0 = lo + blockIdx.x * kGhostBlock + threadIdx.x;
  const int k0 = blockIdx.x * kGhostBlock + threadIdx.x;
  const int stride = gridDim.x * kGhostBlock;
  const int nl = list ? *cnt : 0;
  int idx[kRuns], redo[kRuns];
  int8_t tb[kRuns];
#pragma unroll
  for (int u = 0; u < kRuns; u++) {
    if (list) {
      const int k = k0 + u * stride;
      idx[u] = k < nl ? list[k] : -1;
    } else {
      // share off of nt of the slots (runner_do_ghost's offset / ntasks)
      const int i = i0 + u * stride;
      idx[u] = (i < hi && (nt == 1 || (i - lo) % nt == off)) ? i : -1;
    }
  }
#pragma unroll
  for (int u = 0; u < kRuns; u++) {
    redo[u] = idx[u] >= 0 ? d.redo[idx[u]] : 0;
    tb[u] = idx[u] >= 0 ? d.tb[idx[u]] : (int8_t)kBinInhibited;
  }
  unsigned int again = 0u, relist = 0u;  // bit u: run u
  // density interactions evaluated for these particles in the last round
  unsigned long long work = 0ull;
#pragma unroll
  for (int u = 0; u < kRuns; u++) {
    // (an inactive particle's flag is not cleared by every pass)
    if (redo[u] && is_active(tb[u], ga.max_active_bin)) {
      const int i = idx[u];
      work += (unsigned long long)d.nd[i];
      bool rl = false;
      if (ghost_one(d, ga, i, rl)) again |= 1u << u;
      if (rl) relist |= 1u << u;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) work += __shfl_xor(work, off);
  int na = 0, nb = 0, nc = 0;
#pragma unroll
  for (int u = 0; u < kRuns; u++) {
    const bool ag = (again >> u) & 1u, rl = (relist >> u) & 1u;
    na += __popcll(__ballot(ag));
    nb += __popcll(__ballot(ag && rl));
    nc += ga.lists ? __popcll(__ballot(!ag && rl)) : 0;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    wcnt[0][w] = na;
    wcnt[1][w] = nb;
    wcnt[2][w] = nc;
    wwork[w] = work;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    unsigned long long t = 0;
    for (int k = 0; k < W; k++) t += (unsigned long long)wcnt[threadIdx.x][k];
    unsigned long long b0 = 0;
    if (t) b0 = atomicAdd(&counters[threadIdx.x], t);
    if (threadIdx.x == 0) base = (int)b0;
  } else if (threadIdx.x == 3) {
    unsigned long long t = 0;
    for (int k = 0; k < W; k++) t += wwork[k];
    if (t) atomicAdd(&counters[3 + blockIdx.x % kGhostWorkSlots], t);
  }
  __syncthreads();
  if (__any(again != 0u)) {
    // append to the compact list of particles for the next round
    int off = base;
    for (int k = 0; k < w; k++) off += wcnt[0][k];
    const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
    for (int u = 0; u < kRuns; u++) {
      const bool ag = (again >> u) & 1u;
      const unsigned long long ba = __ballot(ag);
      if (ag) d.sel[off + __popcll(ba & below)] = idx[u];
      off += __popcll(ba);
    }
  }
}

__global__ void k_fill_f32(float *p, float v, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Clears the image masks, their error word and the cell mask.
__global__ void k_task_clear(unsigned int *images, unsigned char *cmask,
                             int ncells) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c <= ncells) images[c] = 0u;
  if (c < ncells) cmask[c] = 0;
}

// One thread per task {type, ci, cj}: sets the image bits of its directed
// interactions.  A task that swsph_run_tasks refuses sets the error word.
__global__ void k_task_images(const int *__restrict__ tasks, int ntasks,
                              GridDesc grid, int ncells, unsigned int *images,
                              unsigned char *cmask) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= ntasks) return;
  const int type = tasks[3 * n], ci = tasks[3 * n + 1];
  const int cj = type == kTaskSelf ? ci : tasks[3 * n + 2];
  bool ok = ci >= 0 && ci < ncells && cj >= 0 && cj < ncells &&
            (type == kTaskSelf ||
             (type == kTaskPair && ci != cj));
  int o = 0;
  if (ok) {
    int a[3], b[3];
    cell_coords(ci, grid, a[0], a[1], a[2]);
    cell_coords(cj, grid, b[0], b[1], b[2]);
    for (int k = 0; k < 3; k++) {
      int dd = b[k] - a[k];
      dd = dd > 1 ? dd - grid.nc[k] : (dd < -1 ? dd + grid.nc[k] : dd);
      ok = ok && dd >= -1 && dd <= 1;
      o = 3 * o + dd + 1;
    }
  }
  if (ok) {
    const unsigned int bi = 1u << o, bj = 1u << (26 - o);
    ok = !(atomicOr(&images[ci], bi) & bi);
    cmask[ci] = 1;
    if (type == kTaskPair) {
      ok = !(atomicOr(&images[cj], bj) & bj) && ok;
      cmask[cj] = 1;
    }
  }
  if (!ok) atomicOr(&images[ncells], 1u);
}

// runner_do_extra_ghost for the active particles in [lo, hi) or of the list.
__global__ void k_extra_ghost(DevParts d, GhostArgs ga, int lo, int hi,
                              const int *list, const int *cnt) {
  if (ga.stop && *ga.stop != 0ull) return;  // uniform
  auto body = [&](int i, int8_t tb) {
    if (!is_active(tb, ga.max_active_bin)) return;
    extra_ghost_one(d, ga, i, tb, d.vsig[i], d.lapu[i], d.avmax[i]);
  };
  if (list)
    for_runs_list(list, cnt, d.tb, body);
  else
    for_runs(lo, hi, d.tb, body);
}

// runner_do_end_hydro_force for the active particles.
__global__ void k_end_force(DevParts d, int lo, int hi, int max_active_bin,
                            const int *list, const int *cnt,
                            const unsigned long long *stop) {
  if (stop && *stop != 0ull) return;  // uniform
  auto body = [&](int i, int8_t tb) {
    if (is_active(tb, max_active_bin))
      d.hdt[i] = end_force_hdt(d.hdt[i], d.h[i]);
  };
  if (list)
    for_runs_list(list, cnt, d.tb, body);
  else
    for_runs(lo, hi, d.tb, body);
}

__global__ void k_zero_int(int *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

__global__ void k_zero_ghost(unsigned long long *counters) {
  const int k = threadIdx.x;
  if (k < 4) counters[k < 3 ? k : kGhostRounds] = 0ull;
}

__global__ void k_zero_u64(unsigned long long *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0ull;
}

// mask[c] = 1 for the n cells of `cells`, 0 for the others (two launches:
// clear, then set).
__global__ void k_zero_u8(unsigned char *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}
__global__ void k_set_mask(unsigned char *mask, const int *cells, int n) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) mask[cells[k]] = 1;
}

// act[c] = 1 for the cells holding an active particle (cleared before).
__global__ void k_cell_active(DevParts d, int n, int max_active_bin,
                              unsigned char *act) {
  for_runs(0, n, d.tb, [&](int i, int8_t tb) {
    if (is_active(tb, max_active_bin)) act[d.cell[i]] = 1;
  });
}

// inv[perm[s]] = s: device slot of every caller index.
__global__ void k_invert_perm(const int *perm, int *inv, int n) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n) inv[perm[s]] = s;
}

// *moved = 1 when perm is not the identity (flag zeroed first).
__global__ void k_perm_moved(const int *perm, int n, unsigned int *moved) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n && perm[s] != s) *moved = 1u;
}

// Chunk table of capacity C from the cells' slot ranges: chunk ch of cell c
// (cell_chunk[c] <= ch < cell_chunk[c + 1]) starts at slot cell_start[c] +
// C * (ch - cell_chunk[c]); start[nchunks] = n closes the last one.  The
// cell of a chunk is found by bisection over cell_chunk.
__global__ void k_chunk_fill(const int *cell_start, const int *cell_chunk,
                             int ncells, int C, int nchunks, int n,
                             int *start, int *chunk_cell) {
  const int ch = blockIdx.x * blockDim.x + threadIdx.x;
  if (ch > nchunks) return;
  if (ch == nchunks) {
    start[ch] = n;
    return;
  }
  int lo = 0, hi = ncells;  // cell_chunk[lo] <= ch < cell_chunk[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cell_chunk[mid] <= ch)
      lo = mid;
    else
      hi = mid;
  }
  start[ch] = cell_start[lo] + C * (ch - cell_chunk[lo]);
  chunk_cell[ch] = lo;
}

// flag[slot of caller index first + ind[k]] = 1 for k < count; a particle
// whose slot lies outside [lo, hi) (not in the task's cell) is counted in
// *err instead.  The caller checked first + ind[k] against the particle
// count.
__global__ void k_mark_subset(int *flag, const int *inv, long long first,
                              const int *ind, int count, int lo, int hi,
                              unsigned int *err) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= count) return;
  const int s = inv[first + ind[k]];
  if (s >= lo && s < hi)
    flag[s] = 1;
  else
    atomicAdd(err, 1u);
}

// dst[i] = src[i] for the particles i of [lo, hi) with (i - lo) % nt == off,
// 0 for the others: the share of a cell's ghost task `off` of `nt`.
__global__ void k_share_flags(int *dst, const int *src, int lo, int hi,
                              int off, int nt) {
  const int i = lo + blockIdx.x * blockDim.x + threadIdx.x;
  if (i < hi) dst[i] = ((i - lo) % nt == off) ? src[i] : 0;
}

// Sums the per-particle interaction counters of active particles:
// out[0] density, out[1] gradient, out[2] force.  One atomic per block.
__global__ void k_count(DevParts d, int n, int max_active_bin,
                        unsigned long long *out) {
  __shared__ unsigned long long part[3][4];
  unsigned long long a = 0, b = 0, c = 0;
  // kRuns time bins in flight per thread and sweep
  const int stride = gridDim.x * blockDim.x;
  for (int i0 = blockIdx.x * blockDim.x + threadIdx.x; i0 < n;
       i0 += stride * kRuns) {
    int8_t t[kRuns];
#pragma unroll
    for (int u = 0; u < kRuns; u++) {
      const int i = i0 + u * stride;
      t[u] = i < n ? d.tb[i] : kBinInhibited;
    }
#pragma unroll
    for (int u = 0; u < kRuns; u++) {
      const int i = i0 + u * stride;
      if (i < n && is_active(t[u], max_active_bin)) {
        a += (unsigned)d.nd[i];
        b += (unsigned)d.ng[i];
        c += (unsigned)d.nf[i];
      }
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    a += __shfl_down(a, off);
    b += __shfl_down(b, off);
    c += __shfl_down(c, off);
  }
  const int wv = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    part[0][wv] = a;
    part[1][wv] = b;
    part[2][wv] = c;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    unsigned long long s = 0;
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) s += part[threadIdx.x][k];
    atomicAdd(&out[threadIdx.x], s);
  }
}

// Block (x, k) copies 1024 floats of array k as float4 words (the buffers
// are 256-byte aligned; the last partial word element by element).
__global__ __launch_bounds__(256) void k_copy_set(sphk::CopySet cs, int n) {
  const int k = blockIdx.y;
  const int w = blockIdx.x * 256 + threadIdx.x;  // float4 word
  const int i = 4 * w;
  if (i + 3 < n) {
    reinterpret_cast<float4 *>(cs.dst[k])[w] =
        reinterpret_cast<const float4 *>(cs.src[k])[w];
  } else {
    for (int j = i; j < n; j++) cs.dst[k][j] = cs.src[k][j];
  }
}

// Active particles of [0, n) at max_active_bin: one atomic per block.
__global__ void k_count_active(const int8_t *__restrict__ tb, int n,
                               int max_active_bin, unsigned int *out) {
  __shared__ unsigned int part[4];
  unsigned int c = 0;
  const int stride = gridDim.x * blockDim.x;
  for (int i0 = blockIdx.x * blockDim.x + threadIdx.x; i0 < n;
       i0 += stride * kRuns) {
    int8_t t[kRuns];
#pragma unroll
    for (int u = 0; u < kRuns; u++) {
      const int i = i0 + u * stride;
      t[u] = i < n ? tb[i] : kBinInhibited;
    }
#pragma unroll
    for (int u = 0; u < kRuns; u++) c += is_active(t[u], max_active_bin) ? 1u : 0u;
  }
  for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned int t = 0;
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) t += part[k];
    if (t) atomicAdd(out, t);
  }
}

// ------------------------------------------------------------ tile builder --
// The particles a loop processes, compacted in cell order and cut into
// tiles, in three launches: a wave per cell counts its particles, one block
// scans the sums of every kTileWaves cells, and a wave per cell writes its
// part of the list and its tiles; a cell that holds most of its block's slots
// is shared by the block's waves.  Everything stays on the device.  (A scan
// over the particle slots took ten launches and five passes over 4 bytes
// per slot: 35 us of launches on a small box, 150-200 us at 16.8 M slots.)
// Bound by the latency of a wave's dependent loads, 512 slots at a time: with
// one wave for every cell a bundle on 4096 cells, one of 20000 / 100000 / 300000
// particles, took 238 / 727 / 1950 us, shared 130 / 174 / 289; a pass over a
// halo of 69000 in a cell, 1 % active, 2.10 ms, shared 1.71; 27 cells of 16384
// each 194 us, shared in blocks of a cell each 52.  The fill waits for no other
// wave: what precedes a cell in its block, and a part in its cell, comes from
// the count (fill of 144^3 31.8 us with barriers and a second count, 21.9 like
// this; count 18.2 and 22.3).
constexpr int kTileBlock = 64 * kTileWaves;
constexpr int kScanBlock = 1024;
constexpr int kTileShared = 4;  // cells that a block shares, at most

// Exclusive scan of v over a block of kScanBlock threads; *total receives
// the block sum.
__device__ __forceinline__ unsigned long long block_excl_scan(
    unsigned long long v, unsigned long long *wsum, unsigned long long *total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  unsigned long long incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned long long t = __shfl_up(incl, off);
    if (lane >= off) incl += t;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  if (w == 0) {
    const unsigned long long x = lane < kScanBlock / 64 ? wsum[lane] : 0ull;
    unsigned long long xi = x;
#pragma unroll
    for (int off = 1; off < kScanBlock / 64; off <<= 1) {
      const unsigned long long t = __shfl_up(xi, off);
      if (lane >= off) xi += t;
    }
    if (lane < kScanBlock / 64) wsum[lane] = xi - x;
    if (lane == kScanBlock / 64 - 1) wsum[kScanBlock / 64] = xi;
  }
  __syncthreads();
  *total = wsum[kScanBlock / 64];
  return wsum[w] + incl - v;
}

__device__ __forceinline__ bool tile_pred(const DevParts &d, const LoopArgs &la,
                                          int mode, const int *flag, int i,
                                          int8_t tb) {
  if (!is_active(tb, la.max_active_bin)) return false;
  if (mode >= 1 && !flag[i]) return false;
  // mode 2: only particles whose neighbour list does not cover their radius
  if (mode == 2 && search_radius2(d.h[i]) <= d.r2b[i]) return false;
  return true;
}

// The particles of cell c's slots [lo, hi) that the tiles take, 64 at a time
// in slot order: f(field slot, taken).  With two slot orders the slots are
// record slots, so that the particles of a cell that several active time bins
// hold still form tiles in the cell's Morton order; with one active bin both
// orders list them alike.  kRuns runs are loaded together.
template <class F>
__device__ __forceinline__ void for_cell_tiles(const DevParts &d,
                                               const LoopArgs &la, int mode,
                                               const int *flag, int c, int lo,
                                               int hi, F f) {
  if (la.cmask && !la.cmask[c]) return;  // uniform over the wave
  const int lane = threadIdx.x & 63;
  for (int j0 = lo; j0 < hi; j0 += 64 * kRuns) {
    int ii[kRuns];
#pragma unroll
    for (int u = 0; u < kRuns; u++) {
      const int j = j0 + 64 * u + lane;
      ii[u] = j < hi ? field_slot(d, j) : -1;
    }
    int8_t tb[kRuns];
#pragma unroll
    for (int u = 0; u < kRuns; u++) tb[u] = ii[u] >= 0 ? d.tb[ii[u]] : 0;
#pragma unroll
    for (int u = 0; u < kRuns; u++) {
      if (j0 + 64 * u >= hi) break;  // uniform
      f(ii[u], ii[u] >= 0 && tile_pred(d, la, mode, flag, ii[u], tb[u]));
    }
  }
}

// Part w of kTileWaves of the slots [lo, hi), whole runs of 64.
__device__ __forceinline__ int2 cell_part(int lo, int hi, int w) {
  const int part = (hi - lo + 64 * kTileWaves - 1) / (64 * kTileWaves) * 64;
  const int a = min(hi, lo + w * part);
  return make_int2(a, min(hi, a + part));
}
// The counts of the parts of a shared cell whose first slot is lo.
__device__ __forceinline__ int *tile_part(const TileScratch &ts, int lo) {
  return ts.part + lo / kTileOwn * kTileWaves;
}

// The block's CPB cells: at most kTileShared of them, those with more than
// kTileOwn slots and a fifth of the block's, are shared by its waves, the
// others taken by a wave each.  (Shared cells are taken one after the other,
// so more of a size are done sooner by a wave each: 1000 cells of 1024
// particles on average took 107 us with every cell above 1024 shared, 70 like
// this.)
template <int CPB>
__global__ __launch_bounds__(kTileBlock) void k_tile_count(
    DevParts d, LoopArgs la, int mode, const int *flag, int ncells, int C,
    TileScratch ts) {
  __shared__ int sum[CPB];                       // of a cell
  __shared__ int parts[kTileShared][kTileWaves]; // of a shared cell's parts
  const int lane = threadIdx.x & 63, w = uniform((int)(threadIdx.x >> 6));
  const int c0 = blockIdx.x * CPB;
  if (blockIdx.x == 0 && threadIdx.x < 8 * 64) ts.heads[threadIdx.x] = 0;
  // lane q holds the slots of cell c0 + q
  const bool in = lane < CPB && c0 + lane < ncells;
  const int lo = in ? la.cell_start[c0 + lane] : 0;
  const int hi = in ? la.cell_start[c0 + lane + 1] : 0;
  unsigned int shared = 0u;  // bit q: cell c0 + q (the same in every wave)
  if (__any(hi - lo > kTileOwn)) {  // uniform
    int all = hi - lo;
    for (int off = CPB / 2; off > 0; off >>= 1) all += __shfl_xor(all, off);
    shared = (unsigned int)__ballot(
        hi - lo > max(kTileOwn, all / (kTileShared + 1)));
  }
  auto count = [&](int q, int a, int b) -> int {
    int k = 0;
    for_cell_tiles(d, la, mode, flag, c0 + q, a, b,
                   [&](int, bool take) { k += __popcll(__ballot(take)); });
    return k;
  };
  if (w < CPB && c0 + w < ncells && !(shared >> w & 1u)) {
    const int k = count(w, __builtin_amdgcn_readlane(lo, w),
                        __builtin_amdgcn_readlane(hi, w));
    if (lane == 0) sum[w] = k;
  }
  int n = 0;
  for (unsigned int big = shared; big != 0u; big &= big - 1u, n++) {
    const int q = __builtin_ctz(big);
    const int lo_q = __builtin_amdgcn_readlane(lo, q);
    const int2 p = cell_part(lo_q, __builtin_amdgcn_readlane(hi, q), w);
    const int k = count(q, p.x, p.y);
    if (lane == 0) {
      parts[n][w] = k;
      tile_part(ts, lo_q)[w] = k;
    }
  }
  __syncthreads();
  if (w > 0) return;
  unsigned long long v = 0ull;  // of cell c0 + lane
  if (in) {
    int k = 0;
    if (shared >> lane & 1u) {
      const int at = __popc(shared & ((1u << lane) - 1u));
      for (int j = 0; j < kTileWaves; j++) k += parts[at][j];
    } else {
      k = sum[lane];
    }
    v = ((unsigned long long)k << 32) | (unsigned int)((k + C - 1) / C);
    ts.cell[c0 + lane] = v;
  }
  unsigned long long incl = v;
  for (int off = 1; off < CPB; off <<= 1) {
    const unsigned long long t = __shfl_up(incl, off);
    if (lane >= off) incl += t;
  }
  if (in) ts.first[c0 + lane] = incl - v;
  if (lane == CPB - 1) {
    ts.blk[blockIdx.x] = incl;
    ts.big[blockIdx.x] = shared;
  }
}

// One block: exclusive scan of the nb block sums in place; the totals close
// the tables.
__global__ __launch_bounds__(kScanBlock) void k_tile_scan(int nb,
                                                          TileScratch ts) {
  __shared__ unsigned long long wsum[kScanBlock / 64 + 1];
  const int per = (nb + kScanBlock - 1) / kScanBlock;
  const int a = threadIdx.x * per, b = min(nb, a + per);
  unsigned long long sum = 0ull;
  for (int k = a; k < b; k++) sum += ts.blk[k];
  unsigned long long total;
  unsigned long long run = block_excl_scan(sum, wsum, &total);
  for (int k = a; k < b; k++) {
    const unsigned long long v = ts.blk[k];
    ts.blk[k] = run;
    run += v;
  }
  if (threadIdx.x == 0) {
    const int nt = (int)(unsigned int)total;
    *ts.nlist = (int)(total >> 32);
    *ts.ntiles = nt;
    ts.tile_start[nt] = (int)(total >> 32);
  }
}

template <int CPB>
__global__ __launch_bounds__(kTileBlock) void k_tile_fill(
    DevParts d, LoopArgs la, int mode, const int *flag, int ncells, int C,
    TileScratch ts) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c0 = blockIdx.x * CPB;
  const unsigned long long base = ts.blk[blockIdx.x];
  unsigned int big = ts.big[blockIdx.x];
  // the wave's own cell (all loads in flight together)
  const int c = c0 + (w < CPB && c0 + w < ncells ? w : 0);
  const unsigned long long own = ts.cell[c], at0 = base + ts.first[c];
  const int lo = la.cell_start[c], hi = la.cell_start[c + 1];
  // the cell's tiles, by `step` threads of which this is number `me`
  auto tiles = [&](int cell, unsigned long long v, unsigned long long at,
                   int me, int step) {
    const int t0 = (int)(unsigned int)at, l0 = (int)(at >> 32);
    const int nt = (int)(unsigned int)v;
    for (int t = me; t < nt; t += step) {
      ts.tile_start[t0 + t] = l0 + t * C;
      ts.tile_cell[t0 + t] = cell;
    }
  };
  const unsigned long long below = (1ull << lane) - 1ull;
  auto list = [&](int cell, int a, int b, int at) {
    for_cell_tiles(d, la, mode, flag, cell, a, b, [&](int i, bool take) {
      const unsigned long long m = __ballot(take);
      if (take) ts.alist[at + __popcll(m & below)] = i;
      at += __popcll(m);
    });
  };
  if (w < CPB && c0 + w < ncells && !(big >> w & 1u) && own != 0ull) {
    tiles(c, own, at0, lane, 64);
    list(c, lo, hi, (int)(at0 >> 32));
  }
  for (; big != 0u; big &= big - 1u) {
    const int cb = c0 + __builtin_ctz(big);
    const unsigned long long v = ts.cell[cb], b0 = base + ts.first[cb];
    const int lo_b = la.cell_start[cb];
    int before = lane < w ? tile_part(ts, lo_b)[lane] : 0;  // of the list
    tiles(cb, v, b0, (int)threadIdx.x, kTileBlock);
    const int2 p = cell_part(lo_b, la.cell_start[cb + 1], w);
    for (int off = kTileWaves / 2; off > 0; off >>= 1)
      before += __shfl_xor(before, off);
    list(cb, p.x, p.y, (int)(b0 >> 32) + uniform(before));
  }
}

// Tiles with a particle of filt[i] != 0, appended to ids with one atomic
// per wave (grid-stride over the device-side tile count).
__global__ void k_select_tiles(const int *tile_start, const int *alist,
                               const int *ntiles, const int *filt, int *ids,
                               int *nids) {
  const int nt = *ntiles;
  const int lane = threadIdx.x & 63;
  for (int b = blockIdx.x * blockDim.x; b < nt; b += gridDim.x * blockDim.x) {
    const int t = b + threadIdx.x;
    bool any = false;
    if (t < nt) {
      const int e = tile_start[t + 1];
      for (int k = tile_start[t]; k < e && !any; k++) any = filt[alist[k]] != 0;
    }
    const unsigned long long m = __ballot(any);
    int off = 0;
    if (lane == 0 && m) off = atomicAdd(nids, __popcll(m));
    off = __shfl(off, 0);
    if (any)
      ids[off + __popcll(m & ((1ull << lane) - 1ull))] = t;
  }
}

}  // namespace

// --------------------------------------------------------------- launchers --
namespace sphk {

static inline int nblk(int n, int b) { return (n + b - 1) / b; }
// Blocks (one wave each) of the grid that takes the tiles beyond a captured
// grid's reach.
constexpr int kRestBlocks = 2048;

template <class L, bool SUB, int C>
void stencil_c(const DevParts &d, const LoopArgs &la, const ChunkArgs &ca,
               const typename L::Rec *rec, hipStream_t st) {
  const NbrList none{};
  hipLaunchKernelGGL((k_loop_stencil<L, C, SUB, false>),
                     dim3(xcd_blocks(ca.nchunks)), dim3(64 * kWaves), 0, st, d,
                     la, ca, rec, (const PosRec *)d.pos, none);
}

hipError_t launch_build_lists(bool subset, const DevParts &d,
                              const LoopArgs &la, const ChunkArgs &ca,
                              const NbrList &nl, hipStream_t st) {
  if (ca.nchunks <= 0) return hipSuccess;
  if (ca.C != kListChunk) return hipErrorInvalidValue;
  const dim3 grid(xcd_blocks(ca.nchunks)), blk(64 * kWaves);
  if (subset)
    hipLaunchKernelGGL((k_loop_stencil<DensityLoop, kListChunk, true, true>),
                       grid, blk, 0, st, d, la, ca, d.rd,
                       (const PosRec *)d.pos, nl);
  else
    hipLaunchKernelGGL((k_loop_stencil<DensityLoop, kListChunk, false, true>),
                       grid, blk, 0, st, d, la, ca, d.rd,
                       (const PosRec *)d.pos, nl);
  return hipGetLastError();
}

template <class L>
void list_loop(bool compact, const DevParts &d, const LoopArgs &la,
               const ChunkArgs &ca, const NbrList &nl,
               const typename L::Rec *rec, int nsel, hipStream_t st) {
  if (compact) {
    hipLaunchKernelGGL((k_loop_list<L, true>),
                       dim3(nblk(nsel, kListChunk * kWaves)), dim3(64 * kWaves),
                       0, st, d, la, ca, nl, rec, nsel);
  } else {
    hipLaunchKernelGGL((k_loop_list<L, false>), dim3(xcd_blocks(ca.nchunks)),
                       dim3(64 * kWaves), 0, st, d, la, ca, nl, rec, 0);
  }
}

hipError_t launch_list_loop(LoopKind kind, bool compact, const DevParts &d,
                            const LoopArgs &la, const ChunkArgs &ca,
                            const NbrList &nl, int nsel, hipStream_t st) {
  if (compact ? nsel <= 0 : ca.nchunks <= 0) return hipSuccess;
  if (!compact && ca.C != kListChunk) return hipErrorInvalidValue;
  switch (kind) {
    case LoopKind::Density:
      list_loop<DensityLoop>(compact, d, la, ca, nl, d.rd, nsel, st);
      break;
    case LoopKind::Gradient:
      list_loop<GradientLoop>(compact, d, la, ca, nl, d.rg, nsel, st);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_build_tiles(const DevParts &d, const LoopArgs &la, int n,
                              int ncells, int C, int mode, const int *flag,
                              const TileScratch &ts, hipStream_t st) {
  if (n <= 0) {
    hipLaunchKernelGGL(k_zero_int, dim3(8), dim3(64), 0, st, ts.heads, 8 * 64);
    hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, st, ts.ntiles, 1);
    hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, st, ts.nlist, 1);
    return hipGetLastError();
  }
  // A block per cell where nearly all cells are shared and their blocks do
  // not outnumber the work (1000 cells of 1024 particles 70 us by 16 cells in
  // a block, 77 by one; of 4096 103 and 85; 512 cells of 1024 61 and 58).
  const bool wide = n / ncells >= max(kTileWide, 2 * ncells);
  const int nb = wide ? ncells : nblk(ncells, kTileWaves);
  if (wide)
    hipLaunchKernelGGL((k_tile_count<1>), dim3(nb), dim3(kTileBlock), 0, st, d,
                       la, mode, flag, ncells, C, ts);
  else
    hipLaunchKernelGGL((k_tile_count<kTileWaves>), dim3(nb), dim3(kTileBlock),
                       0, st, d, la, mode, flag, ncells, C, ts);
  hipLaunchKernelGGL(k_tile_scan, dim3(1), dim3(kScanBlock), 0, st, nb, ts);
  if (wide)
    hipLaunchKernelGGL((k_tile_fill<1>), dim3(nb), dim3(kTileBlock), 0, st, d,
                       la, mode, flag, ncells, C, ts);
  else
    hipLaunchKernelGGL((k_tile_fill<kTileWaves>), dim3(nb), dim3(kTileBlock),
                       0, st, d, la, mode, flag, ncells, C, ts);
  return hipGetLastError();
}

// Resident grid of a persistent kernel: blocks per CU at full occupancy
// times the CU count (queried once per kernel instance).
template <class L, int CI, int CJ, bool B>
static int resident_blocks() {
  static std::atomic<int> cached{0};
  if (cached.load() == 0) {
    int dev = 0, ncu = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount,
                              dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per, k_loop_queue<L, CI, CJ, B>, 64 * kWaves, 0) != hipSuccess ||
        per <= 0)
      return 0;
    cached.store(ncu * per * kWaves);
  }
  return cached.load();
}

template <class L, int CI, int CJ, bool B>
hipError_t queue_c(const DevParts &d, const LoopArgs &la, const ChunkArgs &ca,
                   const TileArgs &ta, const NbrList &nl,
                   const typename L::Rec *rec, bool persistent, int waves,
                   int max_tiles, bool rest, hipStream_t st) {
  if (!persistent) {
    const int nb = max_tiles > 0 ? xcd_blocks(max_tiles) : 0;
    if (nb > 0)
      hipLaunchKernelGGL((k_loop_tiles<L, CI, CJ, B>), dim3(nb),
                         dim3(64 * kWaves), 0, st, d, la, ca, rec,
                         (const PosRec *)d.pos, nl, ta);
    if (rest)
      hipLaunchKernelGGL((k_loop_tiles_rest<L, CI, CJ, B>), dim3(kRestBlocks),
                         dim3(64), 0, st, d, la, ca, rec,
                         (const PosRec *)d.pos, nl, ta, nb);
    return hipGetLastError();
  }
  auto kern = k_loop_queue<L, CI, CJ, B>;
  if (waves <= 0) waves = resident_blocks<L, CI, CJ, B>();
  if (waves <= 0) return hipErrorInvalidValue;
  // `waves` counts waves; blocks hold kWaves of them
  hipLaunchKernelGGL(kern, dim3((waves + kWaves - 1) / kWaves),
                     dim3(64 * kWaves), 0, st, d, la, ca, rec,
                     (const PosRec *)d.pos, nl, ta);
  return hipGetLastError();
}

// Tile (CI) x chunk (CJ) shapes with kernels of the chunk engine: CJ = CI,
// CJ = CI / 2 for CI = 32 (finer candidate chunks under the same tile; the
// tiles of 16 have their own kernels, launch_tile16), and the narrow tiles
// (4, 16), (4, 32), (8, 16) for sparse activity (a few active particles per
// cell: more candidate streams per particle, fewer idle lanes).
template <class L>
hipError_t queue_any(const DevParts &d, const LoopArgs &la, const ChunkArgs &ca,
                     const TileArgs &ta, const NbrList &nl,
                     const typename L::Rec *rec, int CI, int CJ, bool p,
                     int waves, int mt, bool rest, hipStream_t st) {
  switch (CI * 100 + CJ) {
    case 808: return queue_c<L, 8, 8, false>(d, la, ca, ta, nl, rec, p, waves, mt, rest, st);
    case 3232: return queue_c<L, 32, 32, false>(d, la, ca, ta, nl, rec, p, waves, mt, rest, st);
    case 3216: return queue_c<L, 32, 16, false>(d, la, ca, ta, nl, rec, p, waves, mt, rest, st);
    case 6464: return queue_c<L, 64, 64, false>(d, la, ca, ta, nl, rec, p, waves, mt, rest, st);
    case 416: return queue_c<L, 4, 16, false>(d, la, ca, ta, nl, rec, p, waves, mt, rest, st);
    case 432: return queue_c<L, 4, 32, false>(d, la, ca, ta, nl, rec, p, waves, mt, rest, st);
    case 816: return queue_c<L, 8, 16, false>(d, la, ca, ta, nl, rec, p, waves, mt, rest, st);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_queue(LoopKind kind, bool build_lists, const DevParts &d,
                        const LoopArgs &la, const ChunkArgs &ca,
                        const TileArgs &ta, const NbrList &nl, int CI, int CJ,
                        bool persistent, int waves, int max_tiles, bool rest,
                        hipStream_t st) {
  if (ca.C != CJ) return hipErrorInvalidValue;
  switch (kind) {
    case LoopKind::Density:
      if (build_lists) {
        if (CI != kListChunk || CJ != kListChunk) return hipErrorInvalidValue;
        return queue_c<DensityLoop, kListChunk, kListChunk, true>(
            d, la, ca, ta, nl, d.rd, persistent, waves, max_tiles, rest, st);
      }
      return queue_any<DensityLoop>(d, la, ca, ta, nl, d.rd, CI, CJ,
                                    persistent, waves, max_tiles, rest,
                                    st);
    case LoopKind::Gradient:
      return queue_any<GradientLoop>(d, la, ca, ta, nl, d.rg, CI, CJ,
                                     persistent, waves, max_tiles, rest,
                                    st);
    case LoopKind::Force:
      return queue_any<ForceLoop>(d, la, ca, ta, nl, d.rf, CI, CJ,
                                  persistent, waves, max_tiles, rest,
                                    st);
  }
  return hipErrorInvalidValue;
}

template <class L, int CJ, bool FIN>
static int tile16_resident_blocks() {
  static std::atomic<int> cached{0};
  if (cached.load() == 0) {
    int dev = 0, ncu = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount,
                              dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per, k_tile16_queue<L, CJ, FIN>, 64, 0) != hipSuccess ||
        per <= 0)
      return 0;
    cached.store(ncu * per);
  }
  return cached.load();
}

template <class L, int CJ, bool FIN>
hipError_t tile16_c(const DevParts &d, const LoopArgs &la, const ChunkArgs &ca,
                    const TileArgs &ta, const TileGhost &tg,
                    const typename L::Rec *rec, bool persistent, int waves,
                    int max_tiles, bool rest, hipStream_t st) {
  const PosRec *pos = (const PosRec *)d.pos;
  if (!persistent) {
    const int nb = max_tiles > 0 ? tile16_blocks<L>(max_tiles) : 0;
    if (nb > 0)
      hipLaunchKernelGGL((k_tile16<L, CJ, FIN>), dim3(nb), dim3(64), 0, st, d,
                         la, ca, rec, pos, ta, tg);
    if (rest)
      hipLaunchKernelGGL((k_tile16_rest<L, CJ, FIN>), dim3(kRestBlocks),
                         dim3(64), 0, st, d, la, ca, rec, pos, ta, tg, nb);
    return hipGetLastError();
  }
  if (waves <= 0) waves = tile16_resident_blocks<L, CJ, FIN>();
  if (waves <= 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_tile16_queue<L, CJ, FIN>), dim3(waves), dim3(64), 0,
                     st, d, la, ca, rec, pos, ta, tg);
  return hipGetLastError();
}

template <class L, bool FIN>
hipError_t tile16_any(const DevParts &d, const LoopArgs &la,
                      const ChunkArgs &ca, const TileArgs &ta,
                      const TileGhost &tg, const typename L::Rec *rec, bool p,
                      int waves, int mt, bool rest, hipStream_t st) {
  switch (ca.C) {
    case 8: return tile16_c<L, 8, FIN>(d, la, ca, ta, tg, rec, p, waves, mt, rest, st);
    case 16: return tile16_c<L, 16, FIN>(d, la, ca, ta, tg, rec, p, waves, mt, rest, st);
    case 32: return tile16_c<L, 32, FIN>(d, la, ca, ta, tg, rec, p, waves, mt, rest, st);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_ghost_cell(bool fin, const DevParts &d, const LoopArgs &la,
                             const ChunkArgs &ca, const GhostArgs &ga,
                             int max_iter, unsigned long long *counters,
                             int cell, int nchunks, int off, int nt,
                             hipStream_t st) {
  if (!ca.fbox || ca.C != 16 || (!fin && !la.fresh))
    return hipErrorInvalidValue;
  if (nchunks <= 0) return hipSuccess;
  const TileGhost tg{ga, max_iter, counters,
                     (unsigned int *)(counters + kGhostRounds), 1};
  const PosRec *pos = (const PosRec *)d.pos;
  if (fin)
    hipLaunchKernelGGL((k_ghost_cell<DensityLoop, true>), dim3(nchunks),
                       dim3(64), 0, st, d, la, ca, d.rd, pos, tg, cell, off,
                       nt);
  else
    hipLaunchKernelGGL((k_ghost_cell<DensityLoop, false>), dim3(nchunks),
                       dim3(64), 0, st, d, la, ca, d.rd, pos, tg, cell, off,
                       nt);
  return hipGetLastError();
}

hipError_t launch_tile16(LoopKind kind, bool fin, bool given,
                         const DevParts &d, const LoopArgs &la,
                         const ChunkArgs &ca, const TileArgs &ta,
                         const GhostArgs &ga, int max_iter,
                         unsigned long long *counters, bool persistent,
                         int waves, int max_tiles, bool rest, hipStream_t st) {
  if (!ca.fbox || (fin && !la.fresh) || ta.ids || ta.filt)
    return hipErrorInvalidValue;
  const TileGhost tg{ga, max_iter, counters,
                     (unsigned int *)(counters + kGhostRounds), given ? 1 : 0};
  auto run = [&](auto loop, const auto *rec) {
    using L = decltype(loop);
    return fin ? tile16_any<L, true>(d, la, ca, ta, tg, rec, persistent, waves,
                                     max_tiles, rest, st)
               : tile16_any<L, false>(d, la, ca, ta, tg, rec, persistent,
                                      waves, max_tiles, rest, st);
  };
  switch (kind) {
    case LoopKind::Density: return run(DensityLoop{}, d.rd);
    case LoopKind::Gradient: return run(GradientLoop{}, d.rg);
    case LoopKind::Force: return run(ForceLoop{}, d.rf);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_select_tiles(const TileScratch &ts, const int *filt,
                               int *ids, int *nids, hipStream_t st) {
  hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, st, nids, 1);
  hipLaunchKernelGGL(k_select_tiles, dim3(1024), dim3(256), 0, st,
                     (const int *)ts.tile_start, (const int *)ts.alist,
                     (const int *)ts.ntiles, filt, ids, nids);
  return hipGetLastError();
}

template <class L>
static int sparse_resident_blocks() {
  static std::atomic<int> cached{0};
  if (cached.load() == 0) {
    int dev = 0, ncu = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount,
                              dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_sparse_queue<L>,
                                                     64, 0) != hipSuccess ||
        per <= 0)
      return 0;
    cached.store(ncu * per);
  }
  return cached.load();
}

template <class L>
hipError_t sparse_l(const DevParts &d, const LoopArgs &la, const ChunkArgs &c1,
                    const ChunkArgs &c2, const TileArgs &ta,
                    const typename L::Rec *rec, bool persistent, int waves,
                    int max_tiles, bool rest, hipStream_t st) {
  const PosRec *pos = (const PosRec *)d.pos;
  if (!persistent) {
    const int nb = max_tiles > 0 ? xcd_blocks(max_tiles) : 0;
    if (nb > 0)
      hipLaunchKernelGGL((k_sparse_tiles<L>), dim3(nb), dim3(64), 0, st, d, la,
                         c1, c2, rec, pos, ta);
    if (rest)
      hipLaunchKernelGGL((k_sparse_tiles_rest<L>), dim3(kRestBlocks), dim3(64),
                         0, st, d, la, c1, c2, rec, pos, ta, nb);
    return hipGetLastError();
  }
  if (waves <= 0) waves = sparse_resident_blocks<L>();
  if (waves <= 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_sparse_queue<L>), dim3(waves), dim3(64), 0, st, d, la,
                     c1, c2, rec, pos, ta);
  return hipGetLastError();
}

hipError_t launch_sparse(LoopKind kind, const DevParts &d, const LoopArgs &la,
                         const ChunkArgs &c1, const ChunkArgs &c2,
                         const TileArgs &ta, bool persistent, int waves,
                         int max_tiles, bool rest, hipStream_t st) {
  if (c1.C != kSpC1 || c2.C != kSpC2) return hipErrorInvalidValue;
  switch (kind) {
    case LoopKind::Density:
      return sparse_l<DensityLoop>(d, la, c1, c2, ta, d.rd, persistent, waves,
                                   max_tiles, rest, st);
    case LoopKind::Gradient:
      return sparse_l<GradientLoop>(d, la, c1, c2, ta, d.rg, persistent, waves,
                                    max_tiles, rest, st);
    case LoopKind::Force:
      return sparse_l<ForceLoop>(d, la, c1, c2, ta, d.rf, persistent, waves,
                                 max_tiles, rest, st);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_fill_f32(float *p, float v, int n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_f32, dim3(nblk(n, 256)), dim3(256), 0, st, p, v, n);
  return hipGetLastError();
}

template <class L, bool SUB>
hipError_t stencil_any(const DevParts &d, const LoopArgs &la,
                       const ChunkArgs &ca, const typename L::Rec *rec,
                       hipStream_t st) {
  switch (ca.C) {
    case 8: stencil_c<L, SUB, 8>(d, la, ca, rec, st); break;
    case 16: stencil_c<L, SUB, 16>(d, la, ca, rec, st); break;
    case 32: stencil_c<L, SUB, 32>(d, la, ca, rec, st); break;
    case 64: stencil_c<L, SUB, 64>(d, la, ca, rec, st); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <class L, bool SUB, int C>
void task_c(const DevParts &d, const LoopArgs &la, const ChunkArgs &ca,
            const typename L::Rec *rec, const TaskArgs &ta, int nb,
            hipStream_t st) {
  hipLaunchKernelGGL((k_loop_task<L, C, SUB>), dim3(nb), dim3(64), 0, st, d, la,
                     ca, rec, (const PosRec *)d.pos, ta);
}

template <class L, bool SUB>
hipError_t task_any(const DevParts &d, const LoopArgs &la, const ChunkArgs &ca,
                    const typename L::Rec *rec, const TaskArgs &ta,
                    hipStream_t st) {
  const int nb = ta.ntiles[0] + ta.ntiles[1];
  if (nb <= 0) return hipSuccess;
  switch (ca.C) {
    case 8: task_c<L, SUB, 8>(d, la, ca, rec, ta, nb, st); break;
    case 16:
      if constexpr (SUB)
        task_c<L, SUB, 16>(d, la, ca, rec, ta, nb, st);
      else
        hipLaunchKernelGGL((k_tile16_task<L>), dim3(nb), dim3(64), 0, st, d,
                           la, ca, rec, (const PosRec *)d.pos, ta);
      break;
    case 32: task_c<L, SUB, 32>(d, la, ca, rec, ta, nb, st); break;
    case 64: task_c<L, SUB, 64>(d, la, ca, rec, ta, nb, st); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_stencil(LoopKind kind, bool subset, const DevParts &d,
                          const LoopArgs &la, const ChunkArgs &ca,
                          hipStream_t st) {
  if (ca.nchunks <= 0) return hipSuccess;
  switch (kind) {
    case LoopKind::Density:
      return subset ? stencil_any<DensityLoop, true>(d, la, ca, d.rd, st)
                    : stencil_any<DensityLoop, false>(d, la, ca, d.rd, st);
    case LoopKind::Gradient:
      return subset ? stencil_any<GradientLoop, true>(d, la, ca, d.rg, st)
                    : stencil_any<GradientLoop, false>(d, la, ca, d.rg, st);
    case LoopKind::Force:
      return stencil_any<ForceLoop, false>(d, la, ca, d.rf, st);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_task(LoopKind kind, bool subset, const DevParts &d,
                       const LoopArgs &la, const ChunkArgs &ca,
                       const TaskArgs &ta, hipStream_t st) {
  switch (kind) {
    case LoopKind::Density:
      return subset ? task_any<DensityLoop, true>(d, la, ca, d.rd, ta, st)
                    : task_any<DensityLoop, false>(d, la, ca, d.rd, ta, st);
    case LoopKind::Gradient:
      return task_any<GradientLoop, false>(d, la, ca, d.rg, ta, st);
    case LoopKind::Force:
      return task_any<ForceLoop, false>(d, la, ca, d.rf, ta, st);
  }
  return hipErrorInvalidValue;
}

template <class L>
hipError_t bundle_any(const DevParts &d, const LoopArgs &la,
                      const ChunkArgs &ca, const typename L::Rec *rec,
                      const BundleArgs &ba, hipStream_t st) {
  if (ba.nitems <= 0) return hipSuccess;
  const dim3 g(ba.nitems), b(64);
  const PosRec *p = (const PosRec *)d.pos;
  switch (ca.C) {
    case 8: hipLaunchKernelGGL((k_loop_bundle<L, 8>), g, b, 0, st, d, la, ca, rec, p, ba); break;
    case 16: hipLaunchKernelGGL((k_loop_bundle<L, 16>), g, b, 0, st, d, la, ca, rec, p, ba); break;
    case 32: hipLaunchKernelGGL((k_loop_bundle<L, 32>), g, b, 0, st, d, la, ca, rec, p, ba); break;
    case 64: hipLaunchKernelGGL((k_loop_bundle<L, 64>), g, b, 0, st, d, la, ca, rec, p, ba); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_bundle(LoopKind kind, const DevParts &d, const LoopArgs &la,
                         const ChunkArgs &ca, const BundleArgs &ba,
                         hipStream_t st) {
  switch (kind) {
    case LoopKind::Density:
      return bundle_any<DensityLoop>(d, la, ca, d.rd, ba, st);
    case LoopKind::Gradient:
      return bundle_any<GradientLoop>(d, la, ca, d.rg, ba, st);
    case LoopKind::Force:
      return bundle_any<ForceLoop>(d, la, ca, d.rf, ba, st);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_zero_ghost(unsigned long long *counters, hipStream_t st) {
  hipLaunchKernelGGL(k_zero_ghost, dim3(1), dim3(64), 0, st, counters);
  return hipGetLastError();
}

hipError_t launch_zero_u64(unsigned long long *p, int n, hipStream_t st) {
  hipLaunchKernelGGL(k_zero_u64, dim3(nblk(n, 64)), dim3(64), 0, st, p, n);
  return hipGetLastError();
}

hipError_t launch_cell_mask(unsigned char *mask, int ncells, const int *cells,
                            int n, hipStream_t st) {
  if (ncells > 0)
    hipLaunchKernelGGL(k_zero_u8, dim3(nblk(ncells, 256)), dim3(256), 0, st,
                       mask, ncells);
  if (n > 0)
    hipLaunchKernelGGL(k_set_mask, dim3(nblk(n, 256)), dim3(256), 0, st, mask,
                       cells, n);
  return hipGetLastError();
}

hipError_t launch_cell_active(const DevParts &d, int n, int ncells,
                              int max_active_bin, unsigned char *act,
                              hipStream_t st) {
  if (ncells > 0)
    hipLaunchKernelGGL(k_zero_u8, dim3(nblk(ncells, 256)), dim3(256), 0, st,
                       act, ncells);
  if (n > 0)
    hipLaunchKernelGGL(k_cell_active, dim3(run_blocks(n, 256)), dim3(256), 0,
                       st, d, n, max_active_bin, act);
  return hipGetLastError();
}

hipError_t launch_invert_perm(const int *perm, int *inv, int n,
                              hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_invert_perm, dim3(nblk(n, 256)), dim3(256), 0, st, perm,
                     inv, n);
  return hipGetLastError();
}

hipError_t launch_mark_subset(int *flag, const int *inv, long long first,
                              const int *ind, int count, int lo, int hi,
                              unsigned int *err, hipStream_t st) {
  hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, st, (int *)err, 1);
  if (hi > lo)
    hipLaunchKernelGGL(k_zero_int, dim3(nblk(hi - lo, 256)), dim3(256), 0, st,
                       flag + lo, hi - lo);
  if (count > 0)
    hipLaunchKernelGGL(k_mark_subset, dim3(nblk(count, 256)), dim3(256), 0, st,
                       flag, inv, first, ind, count, lo, hi, err);
  return hipGetLastError();
}

hipError_t launch_share_flags(int *dst, const int *src, int lo, int hi,
                              int off, int nt, hipStream_t st) {
  if (hi <= lo) return hipSuccess;
  hipLaunchKernelGGL(k_share_flags, dim3(nblk(hi - lo, 256)), dim3(256), 0, st,
                     dst, src, lo, hi, off, nt);
  return hipGetLastError();
}

hipError_t launch_perm_moved(const int *perm, int n, unsigned int *moved,
                             hipStream_t st) {
  hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, st, (int *)moved, 1);
  if (n > 0)
    hipLaunchKernelGGL(k_perm_moved, dim3(nblk(n, 256)), dim3(256), 0, st,
                       perm, n, moved);
  return hipGetLastError();
}

hipError_t launch_chunk_fill(const int *cell_start, const int *cell_chunk,
                             int ncells, int C, int nchunks, int n, int *start,
                             int *chunk_cell, hipStream_t st) {
  hipLaunchKernelGGL(k_chunk_fill, dim3(nblk(nchunks + 1, 256)), dim3(256), 0,
                     st, cell_start, cell_chunk, ncells, C, nchunks, n, start,
                     chunk_cell);
  return hipGetLastError();
}

hipError_t launch_zero_u32(unsigned int *p, int n, hipStream_t st) {
  hipLaunchKernelGGL(k_zero_int, dim3(nblk(n, 64)), dim3(64), 0, st, (int *)p,
                     n);
  return hipGetLastError();
}

hipError_t launch_build_pos(const DevParts &d, const GridDesc &g, float pos_eps,
                            int lo, int hi, hipStream_t st) {
  if (hi <= lo) return hipSuccess;
  hipLaunchKernelGGL(k_build_pos, dim3(nblk(hi - lo, 256)), dim3(256), 0, st, d,
                     g, pos_eps, lo, hi);
  return hipGetLastError();
}

hipError_t launch_chunk_bounds(const DevParts &d, const int *chunk_start,
                               int c0, int c1, int C, double *bbox,
                               float *hg2max, unsigned int *hg2_all,
                               hipStream_t st, const GridDesc &g, float pos_eps,
                               float4 *fbox) {
  if (c1 <= c0) return hipSuccess;
  if (C != 8 && C != 16 && C != 32 && C != 64) return hipErrorInvalidValue;
  const int waves = nblk(c1 - c0, 64 / C);
  hipLaunchKernelGGL(k_chunk_bounds, dim3(nblk(waves, kBoundsBlock / 64)),
                     dim3(kBoundsBlock), 0, st, d, chunk_start, c0, c1, C, bbox,
                     hg2max, hg2_all, g, pos_eps, fbox);
  return hipGetLastError();
}

hipError_t launch_radius_bounds(const DevParts &d, const int *chunk_start,
                                int c0, int c1, int C, float *hg2max,
                                unsigned int *hg2_all, float pos_eps,
                                float4 *fbox, bool records, hipStream_t st) {
  if (c1 <= c0) return hipSuccess;
  if (C != 8 && C != 16 && C != 32 && C != 64) return hipErrorInvalidValue;
  const int waves = nblk(c1 - c0, 64 / C);
  hipLaunchKernelGGL(k_radius_bounds, dim3(nblk(waves, kBoundsBlock / 64)),
                     dim3(kBoundsBlock), 0, st, d, chunk_start, c0, c1, C,
                     hg2max, hg2_all, pos_eps, fbox,
                     records ? (PosRec *)d.pos : nullptr);
  return hipGetLastError();
}

hipError_t launch_build_records(LoopKind kind, const DevParts &d, int lo,
                                int hi, hipStream_t st, int max_active_bin,
                                const int *list, const int *cnt) {
  if (max_active_bin < 0) list = cnt = nullptr;  // all records: staged path
  if (hi <= lo) return hipSuccess;
  const int m = max_active_bin;
  // active records: kRuns runs per block; all records: one run, staged
  const dim3 g(m >= 0 ? run_blocks(hi - lo, kRecBlock) : nblk(hi - lo, kRecBlock)),
      b(kRecBlock);
  switch (kind) {
    case LoopKind::Density:
      hipLaunchKernelGGL(k_build_dens_rec, g, b, 0, st, d, lo, hi, m, list, cnt);
      break;
    case LoopKind::Gradient:
      hipLaunchKernelGGL(k_build_grad_rec, g, b, 0, st, d, lo, hi, m, list, cnt);
      break;
    case LoopKind::Force:
      hipLaunchKernelGGL(k_build_force_rec, g, b, 0, st, d, lo, hi, m, list, cnt);
      break;
  }
  return hipGetLastError();
}

hipError_t launch_init_density(const DevParts &d, int lo, int hi,
                               int max_active_bin, float h_max, hipStream_t st,
                               const int *list, const int *cnt, bool light) {
  if (hi <= lo) return hipSuccess;
  hipLaunchKernelGGL(k_init_density, dim3(run_blocks(hi - lo, 256)), dim3(256), 0, st,
                     d, lo, hi, max_active_bin, h_max, list, cnt, light ? 1 : 0);
  return hipGetLastError();
}

hipError_t launch_ghost(const DevParts &d, const GhostArgs &ga, int lo, int hi,
                        unsigned long long *counters, hipStream_t st,
                        const int *list, const int *cnt, int off, int nt) {
  // counters[3] accumulates over the rounds of a pass (zeroed by the pass)
  hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, st, counters, 3);
  if (hi > lo)
    hipLaunchKernelGGL(k_ghost, dim3(run_blocks(hi - lo, kGhostBlock)),
                       dim3(kGhostBlock), 0, st, d, ga, lo, hi, off, nt,
                       counters, list, cnt);
  return hipGetLastError();
}

hipError_t launch_task_images(const int *tasks, int ntasks, GridDesc grid,
                              int ncells, unsigned int *images,
                              unsigned char *cmask, hipStream_t st) {
  hipLaunchKernelGGL(k_task_clear, dim3(nblk(ncells + 1, 256)), dim3(256), 0,
                     st, images, cmask, ncells);
  hipLaunchKernelGGL(k_task_images, dim3(nblk(ntasks, 256)), dim3(256), 0, st,
                     tasks, ntasks, grid, ncells, images, cmask);
  return hipGetLastError();
}

hipError_t launch_extra_ghost(const DevParts &d, const GhostArgs &ga, int lo,
                              int hi, hipStream_t st, const int *list,
                              const int *cnt) {
  if (hi <= lo) return hipSuccess;
  hipLaunchKernelGGL(k_extra_ghost, dim3(run_blocks(hi - lo, 256)), dim3(256), 0, st,
                     d, ga, lo, hi, list, cnt);
  return hipGetLastError();
}

hipError_t launch_end_force(const DevParts &d, int lo, int hi,
                            int max_active_bin, hipStream_t st, const int *list,
                            const int *cnt, const unsigned long long *stop) {
  if (hi <= lo) return hipSuccess;
  hipLaunchKernelGGL(k_end_force, dim3(run_blocks(hi - lo, 256)), dim3(256), 0, st, d,
                     lo, hi, max_active_bin, list, cnt, stop);
  return hipGetLastError();
}

hipError_t launch_copy_set(const CopySet &cs, int n, hipStream_t st) {
  if (n <= 0 || cs.m <= 0) return hipSuccess;
  if (cs.m > kMaxCopies) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_copy_set, dim3(nblk(n, 1024), cs.m), dim3(256), 0, st,
                     cs, n);
  return hipGetLastError();
}

// Blocks of 256 of the counting sweeps: a particle per thread up to 128 blocks,
// then up to kRuns in flight each and at most 1024 blocks.  (Every block ends
// with atomics on the same addresses: with a particle per thread up to 1024
// blocks a count of 262144 / 600000 / 1000000 particles took 30 / 31 / 32 us
// of wall time, 21 / 23 / 26 like this; 256 blocks even, 512 +2-3 us.)
static int count_blocks(int n) {
  const int most = min(nblk(n, 256), 128);
  return min(1024, max(max(1, most), nblk(n, 256 * kRuns)));
}

hipError_t launch_count_active(const DevParts &d, int n, int max_active_bin,
                               unsigned int *out, hipStream_t st) {
  hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(64), 0, st, (int *)out, 1);
  if (n > 0)
    hipLaunchKernelGGL(k_count_active, dim3(count_blocks(n)), dim3(256), 0, st,
                       (const int8_t *)d.tb, n, max_active_bin, out);
  return hipGetLastError();
}

hipError_t launch_count(const DevParts &d, int n, int max_active_bin,
                        unsigned long long *out3, hipStream_t st) {
  hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, st, out3, 3);
  hipLaunchKernelGGL(k_count, dim3(count_blocks(n)), dim3(256), 0, st, d, n,
                     max_active_bin, out3);
  return hipGetLastError();
}

}  // namespace sphk
