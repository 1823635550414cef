// sph_tile.h -- neighbour loops over the work queue's tiles of 16 particles.
//
// One wave64 owns a tile of up to 16 particles of one cell: lane g + 16 s is
// candidate stream s of 4 of particle g, as in the chunk engine
// (sph_gather.h), and visits the same candidates in the same order, so the
// sums are those of that engine bit for bit.  The work between is arranged
// in windows of 2048 candidates (512 rows of 4):
//
//   1. cull: the chunks of the 27 neighbour cells, one per lane, box against
//      the tile's box in FP32 (ChunkArgs::fbox) in the tile frame -- positions
//      relative to the centre of the tile's box; survivors in LDS;
//   2. test: 64 candidates at a time are staged in the tile frame and met
//      with the 16 particles by v_mfma_f32_16x16x4_f32 (see the chunk
//      engine's matrix pre-test); the signs of the results are the hits;
//   3. expand: each lane writes the rows of its hits to its list in LDS;
//   4. walk: each lane takes its hits in turn, the next record's loads in
//      flight while the current one is evaluated (FP64 pair contract, the
//      loop's test, the interaction).
//
// Bound: the walk's gathers and VALU issue together, in waves that run as long
// as their fullest lane (busy share of the cycles, L1 return path / VALU, on
// modulated 97^3 and clustered 144^3: density 0.86-0.92 / 0.78-0.81 and 0.88 /
// 0.95, gradient 0.95 / 0.88 and 0.95 / 0.84, force 0.95 / 0.79 and 0.95 / 0.81).
// A window of 512 rows evens the lanes out better than the chunk engine's
// 128 (modulated 97^3 box: 26 -> 21 iterations per tile at 256 for 13.5 hits
// per lane; 512 rows in lists of 32 against 256 in lists of 44: density -4 %,
// force -5 %, gradient even; wider ones cost more in LDS), the matrix test
// takes 1 instruction per 64 pairs beside the signs (the FP16 rows took 7),
// and the pipelined walk has one load latency per hit instead of three.
//
// With FIN the tiles also finish their particles, which saves the sweeps over
// them that would follow (a launch each and their fields read back): the
// gradient form ends with the extra ghost and the force record, the force
// form with the end of the force loop.
// The density form then iterates the smoothing lengths itself: the wave
// holds the finished sums of its particles after the walk, takes their
// Newton step (sph_ghost.h) and goes on with the particles that are not done
// -- on the same lists while their radius is inside the one the lists were
// made with, else from step 1 -- until all have converged.  That replaces a
// ghost launch, a tile build and a density launch per round.  A step reads 2
// of the 8 sums, and all are needed at the last h only: after the first an
// evaluation takes the 2 (a third of the walk's arithmetic and 16 of the
// record's 40 bytes less) until a particle of the tile is expected to
// converge, its last step (relative: s) making s^2, the order of the next
// one, pass the tolerance; a particle found to have converged before that is
// evaluated once more.
#pragma once

#include "sph_gather.h"
#include "sph_ghost.h"

namespace sphl {

constexpr int kTileRows = 512;    // rows of 4 candidates in a window
constexpr int kTileHits = 32;     // hits of a lane between two walks

// What the finishing forms need beside the loop's arguments.
struct TileGhost {
  GhostArgs ga;
  int max_iter;
  unsigned long long *counters;  // launch_ghost's: [0] not converged,
                                 // [3..] density interactions
  unsigned int *rounds;          // largest number of density evaluations
  // 1: the first evaluation is done already, its raw sums are in the fields
  // (the density tasks or bundles before a ghost task)
  int given;
};

// The particles of a tile: lane g + 16 s of the wave holds the field slot
// and record slot of particle g (act: it takes part); images: the stencil
// images they meet (TileArgs::images).
constexpr unsigned int kAllImages = (1u << 27) - 1u;
struct TileParts {
  int cell;
  unsigned int images;
  bool act;
  int i, ic;
};
__device__ __forceinline__ TileParts queue_parts(const DevParts &d,
                                                 const TileArgs &tq, int tile) {
  const int g = threadIdx.x & 15;
  const int ts = uniform(tq.tile_start[tile]);
  TileParts t;
  t.act = g < uniform(tq.tile_start[tile + 1]) - ts;
  t.cell = uniform(tq.tile_cell[tile]);
  t.images = tq.images ? tq.images[t.cell] : kAllImages;
  t.i = t.act ? tq.alist[ts + g] : 0;
  t.ic = t.act ? rec_slot(d, t.i) : -1;
  return t;
}

template <class L, int CJ>
struct TileLds {
  static constexpr int RPC = CJ / 4;               // rows per chunk
  static constexpr int CHUNKS = kTileRows / RPC;   // chunks of a window
  double fo[27 * 6];    // pair-contract frame {oi, oj} of each neighbour
  double xi[16 * 3];    // the particles' positions (own cell: oi = oj = x_i)
  float qoff[27 * 3];   // neighbour image corners relative to the tile centre
  int qk0[27], qpre[28], qj0[27], qj1[27];
  // staged candidates: rows x, y, z, |x|^2 and (force) |x|^2 - H_j^2
  float tp[L::kSymmetric ? kTpLen : 4 * kTpRow];
  // surviving chunks: (neighbour << 27) | first record slot
  unsigned int surv[CHUNKS + 64];
  unsigned short rows[kTileHits * 64];  // hit k of lane l at 64 k + l
};

// Maximum over the 16 lanes of a row of lanes (lane % 16 varies).
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(
      0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, dpp_f<0x128>(v));  // row_ror:8, 4, 2, 1
  v = fmaxf(v, dpp_f<0x124>(v));
  v = fmaxf(v, dpp_f<0x122>(v));
  return fmaxf(v, dpp_f<0x121>(v));
}
// Largest value of the wave (uniform).
__device__ __forceinline__ int wave_most(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x124, 0xf, 0xf, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x122, 0xf, 0xf, true));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x121, 0xf, 0xf, true));
  return max(max(__builtin_amdgcn_readlane(v, 0),
                 __builtin_amdgcn_readlane(v, 16)),
             max(__builtin_amdgcn_readlane(v, 32),
                 __builtin_amdgcn_readlane(v, 48)));
}
// Marks every field of a loaded record as used here: the wait for its loads
// stands at this point.
__device__ __forceinline__ void arrived(const DensRec &r) {
  asm volatile("" :: "v"(r.x), "v"(r.y), "v"(r.z), "v"(r.vx), "v"(r.vy),
                    "v"(r.vz), "v"(r.m));
}
__device__ __forceinline__ void arrived(const GradRec &r) {
  asm volatile("" :: "v"(r.x), "v"(r.y), "v"(r.z), "v"(r.vx), "v"(r.vy),
                    "v"(r.vz), "v"(r.mrho), "v"(r.u), "v"(r.c),
                    "v"(r.alpha));
}
__device__ __forceinline__ void arrived(const ForceRec &r) {
  asm volatile("" :: "v"(r.x), "v"(r.y), "v"(r.z), "v"(r.hg2), "v"(r.vx),
                    "v"(r.vy), "v"(r.vz), "v"(r.m), "v"(r.inv_m),
                    "v"(r.h_inv));
  asm volatile("" :: "v"(r.rho), "v"(r.inv_rho), "v"(r.pr2), "v"(r.f),
                    "v"(r.bal), "v"(r.c), "v"(r.alpha), "v"(r.P),
                    "v"(r.Pad), "v"(r.u));
  asm volatile("" :: "v"(r.tb));
}
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// n / d for 0 <= n < 2^31 by the host's floor(2^32 / d) (d >= 2): the
// estimate is at most 1 short.
__device__ __forceinline__ int div_magic(int n, int d, unsigned int magic) {
  const int q = (int)__umulhi((unsigned int)n, magic);
  return n - q * d >= d ? q + 1 : q;
}

// One tile; slot spreads the density work over the counters.
template <class L, int CJ, bool FIN>
__device__ __forceinline__ void run_tile(
    const DevParts &d, const LoopArgs &la, const ChunkArgs &ca,
    const typename L::Rec *__restrict__ rec, const PosRec *__restrict__ pos,
    const TileParts &tp, const TileGhost &tg, int slot) {
  using Sh = TileLds<L, CJ>;
  using Rec = typename L::Rec;
  constexpr int RPC = Sh::RPC, CHUNKS = Sh::CHUNKS;
  constexpr int G = 64 / CJ;  // chunks staged together
  constexpr bool ITER = FIN && std::is_same<L, DensityLoop>::value;
  __shared__ Sh sh;
  const int lane = threadIdx.x & 63;
  const int g = lane & 15, s = lane >> 4;
  const int cell_i = tp.cell;
  const bool act = tp.act;
  const int i = tp.i, ic = tp.ic;
  typename L::I st{};
  st.x = st.y = st.z = kFar;
  if (act) L::load_i(d, i, st);

  // The tile's box in its cell's frame, rounded to float (monotone), the
  // tile centre in FP64, and the largest radius.
  const int cyz = div_magic(cell_i, la.grid.nc[2], la.magic[2]);
  const int cz = cell_i - cyz * la.grid.nc[2];
  const int cx = div_magic(cyz, la.grid.nc[1], la.magic[1]);
  const int cy = cyz - cx * la.grid.nc[1];
  const int ci3[3] = {cx, cy, cz};
  double cen[3];
  float half[3];  // half extents, at least those of the particles
  float fi[3];    // the particle in the tile frame
  {
    const double xi[3] = {st.x, st.y, st.z};
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const double corner = (double)ci3[k] * la.w[k];
      const float f = act ? (float)(xi[k] - corner) : -1e30f;
      const float hi = row16_max(f);
      const float lo = -row16_max(act ? -f : -1e30f);
      cen[k] = corner + (double)(0.5f * (lane_value(lo, 0) + lane_value(hi, 0)));
      fi[k] = act ? (float)(xi[k] - cen[k]) : 0.f;
      half[k] = lane_value(row16_max(fabsf(fi[k])), 0);
    }
  }
  const float hg2i = lane_value(row16_max(act ? st.hg2 : 0.f), 0);
  // lengths of the matrix test in units of the largest radius
  const float invR = lane_value(hg2i > 0.f ? 1.f / sqrtf(hg2i) : 1.f, 0);
  const float invR2 = lane_value(invR * invR * kRadUp, 0);
  if (s == 0 && act) {
    sh.xi[3 * g] = st.x;
    sh.xi[3 * g + 1] = st.y;
    sh.xi[3 * g + 2] = st.z;
  }

  // Neighbour table: lane q < 27 describes neighbour q of the stencil.
  int nchq = 0;
  if (lane < 27) {
    const int o = stencil_code(lane);
    const int o3[3] = {o / 9 - 1, (o / 3) % 3 - 1, o % 3 - 1};
    int v[3];
    double t[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      v[k] = ci3[k] + o3[k];
      t[k] = 0.0;
      if (v[k] < 0) {
        v[k] += la.grid.nc[k];
        t[k] = -la.grid.dim[k];
      } else if (v[k] >= la.grid.nc[k]) {
        v[k] -= la.grid.nc[k];
        t[k] = la.grid.dim[k];
      }
      sh.qoff[3 * lane + k] =
          (float)(((double)v[k] * la.w[k] + t[k]) - cen[k]);
    }
    const int cj = (v[0] * la.grid.nc[1] + v[1]) * la.grid.nc[2] + v[2];
    const int k0 = ca.cell_chunk[cj], k1 = ca.cell_chunk[cj + 1];
    sh.qk0[lane] = k0;
    sh.qj0[lane] = la.cell_start[cj];
    sh.qj1[lane] = la.cell_start[cj + 1];
    nchq = tp.images >> o & 1u ? k1 - k0 : 0;
    double fo[6];
    (void)pair_frame(o3, ci3, v, t, la.w, fo);
    for (int k = 0; k < 6; k++) sh.fo[6 * lane + k] = fo[k];
  }
  int incl = nchq;  // inclusive prefix over lanes 0..31
#pragma unroll
  for (int off = 1; off < 32; off <<= 1) {
    const int v = __shfl_up(incl, off);
    if (lane >= off) incl += v;
  }
  if (lane < 27) sh.qpre[lane] = incl - nchq;
  const int total = __builtin_amdgcn_readlane(incl, 26);

  // i side of the matrix test (see the chunk engine)
  const float ux = fi[0] * invR, uy = fi[1] * invR, uz = fi[2] * invR;
  const float isq = fmaf(uz, uz, fmaf(uy, uy, ux * ux)) * kSqLo;
  const float mb =
      s == 3 ? 1.f : (act ? -2.f * (s == 0 ? ux : (s == 1 ? uy : uz)) : 0.f);
  // candidate (row of A) of this lane and its component
  const int am = (lane & 3) * 4 + ((lane >> 2) & 3);
  const int t1 = s * kTpRow + am;
  const int t2 = s == 3 ? kTpRowJ + am : t1;

  typename L::Acc acc;
  int cnt = 0;  // hits in this lane's list
  bool full = true;  // the walk takes all sums (uniform)

  // Step 4: the lists against the exact contract, the next record's loads in
  // flight while the current one is evaluated.  The loop is uniform (to the
  // fullest lane's hits) and its loads unconditional, a lane past its hits
  // reading record 0: with a branch around them, or a register of a record
  // that an untaken branch has not waited for, the compiler's waits for one
  // record also wait for the next, and each hit costs a whole load latency.
  auto walk_as = [&](auto all) {
    constexpr bool ALL = decltype(all)::value;  // else only the step's sums
    auto fetch = [&](int k, unsigned int &info, Rec &r) -> int {
      const bool on = k < cnt;
      // (read by all lanes: no branch)
      const int got = sh.rows[64 * min(k, kTileHits - 1) + lane];
      const int row = on ? got : 0;
      info = sh.surv[row / RPC];
      const int at = (int)(info & kRowMask) + (row % RPC) * 4 + s;
      const int j = on ? at : 0;
      if constexpr (ALL) {
        r = rec[j];
      } else {
        r.x = rec[j].x;
        r.y = rec[j].y;
        r.z = rec[j].z;
      }
      return j;
    };
    auto eval = [&](int k, unsigned int info, const Rec &r, int j) {
      // all of the record has arrived from here on
      if constexpr (ALL)
        arrived(r);
      else
        asm volatile("" :: "v"(r.x), "v"(r.y), "v"(r.z));
      const int q = (int)(info >> 27);
      // own cell: oi = oj = x_i, which gives 0 - (float)(x_j - x_i)
      const double *fo = q ? &sh.fo[6 * q] : &sh.xi[3 * g];
      const double *fj = q ? fo + 3 : fo;
      const float dx = (float)(st.x - fo[0]) - (float)(r.x - fj[0]);
      const float dy = (float)(st.y - fo[1]) - (float)(r.y - fj[1]);
      const float dz = (float)(st.z - fo[2]) - (float)(r.z - fj[2]);
      const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
      // (the matrix test passes the particle itself)
      if (L::test(r2, st, &r) && j != ic && k < cnt) {
        if constexpr (ITER)
          L::interact(r2, dx, dy, dz, st, r, acc, ALL);
        else
          L::interact(r2, dx, dy, dz, st, r, acc);
      }
    };
    const int most = wave_most(cnt);
    if (most == 0) return;  // uniform
    unsigned int n0, n1;
    Rec r0, r1;
    int j0 = fetch(0, n0, r0), j1 = 0;
    int k = 0;
    for (; k + 2 < most; k += 2) {
      j1 = fetch(k + 1, n1, r1);
      eval(k, n0, r0, j0);
      j0 = fetch(k + 2, n0, r0);
      eval(k + 1, n1, r1, j1);
    }
    // one or two are left (no load past the last)
    const bool two = k + 1 < most;
    if (two) j1 = fetch(k + 1, n1, r1);
    eval(k, n0, r0, j0);
    if (two) eval(k + 1, n1, r1, j1);
  };
  auto walk = [&]() {
    if (!ITER || full)
      walk_as(std::true_type{});
    else
      walk_as(std::false_type{});
  };

  // The candidates of a sweep, a window at a time.  pre: the lane's squared
  // pre-test radius (negative: it takes no part); fb: chunks culled so far;
  // ns: survivors in LDS (the first `done` of them walked already).
  float pre = -1.f, maxpre = -1.f;
  int fb = 0, ns = 0, done = 0;
  // Steps 1 to 3: fills the lists from the next window and returns whether
  // candidates are left after it.
  auto window = [&]() -> bool {
    // the survivors past the last window open this one
    if (done > 0) {
      for (int c = done; c < ns; c += 64) {  // uniform
        const unsigned int e = c + lane < ns ? sh.surv[c + lane] : 0u;
        wave_sync();
        if (c + lane < ns) sh.surv[c - done + lane] = e;
        wave_sync();
      }
      ns -= done;
    }
    // 1. cull until the window is full
    while (ns < CHUNKS && fb < total) {
      const int f = fb + lane;
      bool pass = false;
      unsigned int pe = 0u;
      if (f < total) {
        int q = 0;
#pragma unroll
        for (int b = 16; b > 0; b >>= 1)
          if (q + b < 27 && sh.qpre[q + b] <= f) q += b;
        const int kin = f - sh.qpre[q];
        const int kc = sh.qk0[q] + kin;
        const float4 lo = ca.fbox[2 * kc], hi = ca.fbox[2 * kc + 1];
        const float ox = sh.qoff[3 * q], oy = sh.qoff[3 * q + 1],
                    oz = sh.qoff[3 * q + 2];
        const float gx =
            fmaxf(0.f, fmaxf(lo.x + ox - half[0], -half[0] - (hi.x + ox)));
        const float gy =
            fmaxf(0.f, fmaxf(lo.y + oy - half[1], -half[1] - (hi.y + oy)));
        const float gz =
            fmaxf(0.f, fmaxf(lo.z + oz - half[2], -half[2] - (hi.z + oz)));
        const float gap2 = fmaf(gz, gz, fmaf(gy, gy, gx * gx));
        pass = gap2 < (L::kSymmetric ? fmaxf(maxpre, lo.w) : maxpre);
        pe = ((unsigned int)q << 27) | (unsigned int)(sh.qj0[q] + kin * CJ);
      }
      const unsigned long long pm = __ballot(pass);
      if (pass) sh.surv[ns + (int)__popcll(pm & ((1ull << lane) - 1ull))] = pe;
      ns += (int)__popcll(pm);
      fb += 64;
    }
    wave_sync();
    // 2. and 3. test and expand, two groups of 64 candidates at a time
    const int nw = min(ns, CHUNKS);
    const int ng = (nw + G - 1) / G;
    done = nw;
    cnt = 0;
    const float ci = pre >= 0.f ? fmaf(-pre * kRadUp, invR2, isq) : 1e30f;
    const float4v mc = {ci, ci, ci, ci};
    const float cs = pre >= 0.f ? isq : 1e30f;
    const float4v mc2 = {cs, cs, cs, cs};
    // the candidate of this lane in group k: loaded one group ahead
    auto load = [&](int k, int &q) -> PosRec {
      const int c = k * G + lane / CJ;
      PosRec p{0.f, 0.f, 0.f, 0.f};
      q = -1;
      if (c < nw) {
        const unsigned int e = sh.surv[c];
        const int j = (int)(e & kRowMask) + lane % CJ;
        if (j < sh.qj1[e >> 27]) {
          q = (int)(e >> 27);
          p = pos[j];
        }
      }
      return p;
    };
    int q;
    PosRec p = load(0, q);
    for (int k0 = 0; k0 < ng; k0 += 2) {
      unsigned int hits = 0u;
#pragma unroll
      for (int kk = 0; kk < 2; kk++) {
        const int k = k0 + kk;
        if (k >= ng) break;  // uniform
        // past the end of a short chunk: far away
        float vx = 1e15f, vy = 0.f, vz = 0.f, sq = 1e30f, sqj = 1e30f;
        if (q >= 0) {
          vx = (p.x + sh.qoff[3 * q]) * invR;
          vy = (p.y + sh.qoff[3 * q + 1]) * invR;
          vz = (p.z + sh.qoff[3 * q + 2]) * invR;
          sq = fmaf(vz, vz, fmaf(vy, vy, vx * vx)) * kSqLo;
          if (L::kSymmetric) sqj = fmaf(-p.hg2m * kRadUp, invR2, sq);
        }
        if (k + 1 < ng) p = load(k + 1, q);
        sh.tp[lane] = vx;
        sh.tp[kTpRow + lane] = vy;
        sh.tp[2 * kTpRow + lane] = vz;
        sh.tp[3 * kTpRow + lane] = sq;
        if (L::kSymmetric) sh.tp[kTpRowJ + lane] = sqj;
        wave_sync();
        unsigned int w = 0u;  // row 0 in the highest of 16 bits
#pragma unroll
        for (int b = 0; b < 4; b++) {
          float4v dd = __builtin_amdgcn_mfma_f32_16x16x4f32(
              sh.tp[t1 + 16 * b], mb, mc, 0, 0, 0);
          if (L::kSymmetric) {
            const float4v d2 = __builtin_amdgcn_mfma_f32_16x16x4f32(
                sh.tp[t2 + 16 * b], mb, mc2, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; r++)
              dd[r] = __uint_as_float(__float_as_uint(dd[r]) |
                                      __float_as_uint(d2[r]));
          }
#pragma unroll
          for (int r = 0; r < 4; r++)  // append the sign
            w = __builtin_amdgcn_alignbit(w, __float_as_uint(dd[r]), 31);
        }
        wave_sync();
        hits |= (__builtin_bitreverse32(w) >> 16) << (16 * kk);
      }
      // a list that these rows could overfill ends the window before them
      // (they always fit an empty list)
      if (__any(cnt + __popc(hits) > kTileHits)) {  // uniform
        done = k0 * G;
        break;
      }
      while (hits != 0u) {  // rows of these groups: 16 k0 + bit
        const int b = __builtin_ctz(hits);
        hits &= hits - 1u;
        sh.rows[64 * cnt + lane] = (unsigned short)(16 * k0 + b);
        cnt++;
      }
    }
    wave_sync();
    return done < ns || fb < total;
  };
  auto sweep = [&](float radius2) {
    pre = radius2;
    maxpre = lane_value(row16_max(pre), 0);
    fb = ns = done = 0;
  };

  if constexpr (!ITER) {
    L::identity(acc);
    if (act && s == 0) {
      if (la.fresh)
        L::fresh_acc(st, acc);
      else
        L::load_acc(d, i, acc);
    }
    wave_sync();
    sweep(act ? pretest_radius2(st.hg2, la.pos_eps) : -1.f);
    bool more;
    do {
      more = window();
      walk();
      wave_sync();
    } while (more);  // uniform
    L::template combine<4>(acc);
    if (act && s == 0) {
      // (an opaque copy: the addresses of the particle's fields are formed
      // here and not kept in registers across the walks)
      int iw = i;
      asm volatile("" : "+v"(iw));
      if constexpr (FIN && std::is_same<L, GradientLoop>::value) {
        d.vsig[iw] = acc.vsig;
        d.avmax[iw] = acc.avmax;
        d.ng[iw] = acc.n;
        extra_ghost_one(d, tg.ga, iw, d.tb[iw], acc.vsig, acc.lapu, acc.avmax);
      } else {
        if constexpr (FIN && std::is_same<L, ForceLoop>::value)
          acc.hdt = end_force_hdt(acc.hdt, d.h[iw]);
        L::store_acc(d, iw, acc);
      }
    }
  } else {
    // The particle's iteration; every lane of a particle holds its whole
    // sums after the combination and takes the same step.
    GhostState gs{0.f, 0.f, tg.ga.h_max};
    if (act) gs.h = d.h[i];
    bool live = act;
    // pend: converged in an evaluation of the step's sums only; want: the
    // next one should take all
    bool pend = false, want = false;
    float listed = -1.f;  // squared radius that the lists cover
    // the lists hold every hit of the sweep (one window took it all)
    bool whole = false, fresh = true, given = tg.given != 0;
    int work = 0, round = 1;
    L::identity(acc);
    if (given && act) {
      L::load_acc(d, i, acc);
      gs.left = d.left[i];  // as the last ghost or hydro_init_part left them
      gs.right = d.right[i];
    }
    wave_sync();
    for (;;) {  // a window, or a walk over lists that still serve
      bool more = false;
      if (!given && (fresh || !whole)) {  // uniform
        if (fresh) {
          // room for the next steps' growth: the lists cover 1 % more at
          // the first evaluation and 2 % more later (radius)
          listed = st.hg2 * (round == 1 ? 1.0201f : 1.0404f);
          sweep(live ? pretest_radius2(listed, la.pos_eps) : -1.f);
        }
        more = window();
        whole = fresh && !more;
        fresh = false;
      }
      walk();
      wave_sync();
      if (more) continue;  // uniform
      if (!given) {
        if (full)
          L::template combine<4>(acc);
        else
          L::template combine_count<4>(acc);
      }
      given = false;
      if (live) {
        // (an opaque copy: the addresses of the particle's fields are formed
        // here and not kept in registers across the walks)
        int iw = i;
        asm volatile("" : "+v"(iw));
        if (!pend) work += acc.n;
        DensSums a{acc.rho, acc.rho_dh, acc.wc, acc.wc_dh,
                   acc.divv, acc.rx, acc.ry, acc.rz};
        const GhostState old = gs;
        const bool again = ghost_step(tg.ga, d.m[iw], gs, a);
        if (again && round < tg.max_iter) {
          const float rel = gs.h / old.h - 1.f;
          want = rel * rel <= 2.f * tg.ga.eps;
          pend = false;
          st.h_inv = 1.f / gs.h;
          st.hg2 = search_radius2(gs.h);
        } else if (!full && !again) {
          gs = old;
          pend = want = true;
        } else {
          live = false;
          cnt = 0;
          if (s == 0) {
            d.nd[iw] = acc.n;
            if (again) {
              // Not converged: flagged, with the bracket of its new h; the
              // host has the sums at that h formed (FIN = false), from which
              // another ghost goes on.
              d.h[iw] = gs.h;
              d.left[iw] = gs.left;
              d.right[iw] = gs.right;
              d.redo[iw] = 1;
              atomicAdd(&tg.counters[0], 1ull);
            } else {
              ghost_finish(d, tg.ga, iw, gs.h, a);
            }
          }
        }
      }
      if (!__any(live)) break;  // uniform
      L::identity(acc);
      if (__any(live && !pend)) round++;
      full = __any(live && want);
      fresh = !whole || __any(live && !(st.hg2 <= listed));
    }
    // density interactions of the tile, and its rounds
    work = s == 0 ? work : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) work += __shfl_xor(work, off);
    if (lane == 0) {
      atomicAdd(&tg.counters[3 + slot % kGhostWorkSlots],
                (unsigned long long)work);
      // a plain read first: only a wave that raises the maximum pays an
      // atomic
      if ((unsigned int)round >
          __hip_atomic_load(tg.rounds, __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(tg.rounds, (unsigned int)round);
    }
  }
}

// Block -> tile of the grids below.
template <class L>
constexpr bool kTileRuns = !std::is_same<L, DensityLoop>::value;
template <class L>
__host__ __device__ inline int tile16_blocks(int n) {
  return kTileRuns<L> ? xcd_run_blocks(n) : xcd_blocks(n);
}
template <class L>
__device__ __forceinline__ int tile16_item(int b, int w, int n) {
  return kTileRuns<L> ? xcd_run_item(b, w, n) : xcd_item(b, w, n);
}

// One wave per tile over a grid sized for the tile count (see k_loop_tiles).
template <class L, int CJ, bool FIN>
__global__ __launch_bounds__(64, L::kTile16WavesPerSimd) void k_tile16(
    DevParts d, LoopArgs la, ChunkArgs ca,
    const typename L::Rec *__restrict__ rec, const PosRec *__restrict__ pos,
    TileArgs tq, TileGhost tg) {
  const int n = tile_count(tq);
  const int t = tile16_item<L>(blockIdx.x, threadIdx.x >> 6, n);
  if (t >= n) return;  // uniform per wave
  run_tile<L, CJ, FIN>(d, la, ca, rec, pos, queue_parts(d, tq, t), tg, t);
}

// The tiles beyond a grid of b0 blocks (see k_loop_tiles_rest).
template <class L, int CJ, bool FIN>
__global__ __launch_bounds__(64, L::kTile16WavesPerSimd) void k_tile16_rest(
    DevParts d, LoopArgs la, ChunkArgs ca,
    const typename L::Rec *__restrict__ rec, const PosRec *__restrict__ pos,
    TileArgs tq, TileGhost tg, int b0) {
  const int n = tile_count(tq);
  const int nb = tile16_blocks<L>(n);
  for (int b = b0 + (int)blockIdx.x; b < nb; b += (int)gridDim.x) {
    const int t = tile16_item<L>(b, threadIdx.x >> 6, n);
    if (t >= n) continue;  // uniform per wave
    wave_sync();
    run_tile<L, CJ, FIN>(d, la, ca, rec, pos, queue_parts(d, tq, t), tg, t);
  }
}

// Persistent form (see k_loop_queue).
template <class L, int CJ, bool FIN>
__global__ __launch_bounds__(64, L::kTile16WavesPerSimd) void k_tile16_queue(
    DevParts d, LoopArgs la, ChunkArgs ca,
    const typename L::Rec *__restrict__ rec, const PosRec *__restrict__ pos,
    TileArgs tq, TileGhost tg) {
  drain_queue(tq, [&](int t) {
    wave_sync();
    run_tile<L, CJ, FIN>(d, la, ca, rec, pos, queue_parts(d, tq, t), tg, t);
  });
}

// runner_do_ghost on one cell after its density tasks: one wave per chunk of
// 16 of the cell, each taking the chunk's flagged particles of share off of
// nt (slot counted from the cell's first field slot, as k_ghost).  FIN =
// false: only their density sums.
template <class L, bool FIN>
__global__ __launch_bounds__(64, L::kTile16WavesPerSimd) void k_ghost_cell(
    DevParts d, LoopArgs la, ChunkArgs ca,
    const typename L::Rec *__restrict__ rec, const PosRec *__restrict__ pos,
    TileGhost tg, int cell, int off, int nt) {
  const int lo = la.cell_start[cell], hi = la.cell_start[cell + 1];
  TileParts t;
  t.cell = cell;
  t.images = kAllImages;
  t.ic = lo + 16 * (int)blockIdx.x + (int)(threadIdx.x & 15);
  t.i = t.ic < hi ? field_slot(d, t.ic) : 0;
  // (an inactive particle's flag is not cleared by every pass)
  t.act = t.ic < hi && d.redo[t.i] != 0 && (t.i - lo) % nt == off &&
          is_active(d.tb[t.i], la.max_active_bin);
  if (!__any(t.act)) return;  // uniform
  if (!t.act) t.ic = -1;
  run_tile<L, 16, FIN>(d, la, ca, rec, pos, t, tg, (int)blockIdx.x);
}

// A self or pair task on cells in chunks of 16: one wave per chunk of either
// i-cell (as k_loop_task) against the one image of the task.  A task is one
// wave's latency and a launch (1134 tasks on 27 cells of 64: 10.8 -> 10.1 ms
// against the chunk engine).
template <class L>
__global__ __launch_bounds__(64, L::kTile16WavesPerSimd) void k_tile16_task(
    DevParts d, LoopArgs la, ChunkArgs ca,
    const typename L::Rec *__restrict__ rec, const PosRec *__restrict__ pos,
    TaskArgs ta) {
  const bool second = (int)blockIdx.x >= ta.ntiles[0];
  const int b = second ? (int)blockIdx.x - ta.ntiles[0] : (int)blockIdx.x;
  TileParts t;
  t.cell = second ? ta.icell[1] : ta.icell[0];
  t.images = second ? ta.images[1] : ta.images[0];
  t.ic = la.cell_start[t.cell] + 16 * b + (int)(threadIdx.x & 15);
  t.act = t.ic < la.cell_start[t.cell + 1];
  t.i = t.act ? field_slot(d, t.ic) : 0;
  t.act = t.act && is_active(d.tb[t.i], la.max_active_bin);
  if (!__any(t.act)) return;  // uniform
  if (!t.act) t.ic = -1;
  run_tile<L, 16, false>(d, la, ca, rec, pos, t, TileGhost{}, 0);
}

}  // namespace sphl
