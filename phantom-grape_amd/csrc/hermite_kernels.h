// Block-time-step 4th-order Hermite integration on the GPU: the host loop of
// the reference's sample integrator (PG6/banana/banana01.c:120-166,
// hermite.c:39-208, timestep.c:24-92) as device kernels around the GRAPE-6
// force.  A block step needs no host round trip: the step's time, active
// set and launch plan live in device memory (Ctl), so the host only queues
// kernels and reads Ctl back when it wants to know where the run stands.
//
// State (device, FP64, particle order = j address = id): x[n][3], v[n][3],
// a[n][3], j[n][3], pot[n], t[n], dt[n], m[n].  One block step:
//   1. t_next = min_i (t_i + dt_i) from the minima of the step before; predict
//      every j to it; active = { i : t_i + dt_i == t_next }, appended to the
//      active list with their predicted i data (predict_exmotion); the minima
//      of t + dt over the others                           (pg6h_select)
//   2. force, jerk, pot of the active i against all j      (pg6h_force)
//   3. sum of the j-range partials, corrector + new time step, j-memory
//      update, reset of every time at the end of a dtmax window; minima of
//      the new t + dt, whose minimum is the next t_next; step bookkeeping
//                                                          (pg6h_finish)
// The first minima come from pg6h_min_time after the start-up.
// Every FP64 expression is written in the reference's operation order with
// contraction off, so given the same forces the corrected state and the time
// steps equal those of the reference's code bit for bit.  One deviation: the
// reference keeps the jerk in float (PG6/banana/particle.h:17-19); here it
// stays FP64.  The active list is filled by atomics, so its order varies
// from run to run; nothing computed per particle depends on it (each i's
// pair sums run over the j addresses in a fixed order).
#pragma once
#include <hip/hip_runtime.h>
#include <climits>
#include <cmath>
#include "pg6_kernels.h"

namespace pg6h {

// Taylor coefficients as the reference writes them (hermite.c:16-19).
constexpr double kSecond = 5e-1;
constexpr double kThird = 1.666666666666667e-1;
constexpr double kFourth = 4.166666666666667e-2;
constexpr double kFifth = 8.333333333333333e-3;

struct State {
  double *x, *v, *a, *j, *pot, *t, *dt, *m;
};

struct Params {
  double eta_s, eta, dtmax, dtmin;
};

// calc_modulus (timestep.c:176-190): what remains of `num` after removing
// the powers-of-two multiples of `mod` (up to modmax) it is built from; 0 when
// `num` is a multiple of `mod` on the block-time grid.
__host__ __device__ inline double calc_modulus(double num, double mod, double modmax) {
  double tmpmod = modmax;
  while (num > 0.0) {
    while (tmpmod > num) tmpmod *= 0.5;
    if (tmpmod < mod) break;
    num -= tmpmod;
  }
  return num;
}

// dt_startup (timestep.c:24-48), without the reference's exit on failure:
// returns 0 when no admissible step exists (the caller reports it).
__device__ inline double dt_startup(const Params& P, double t_gl, const double* a,
                                    const double* j) {
#pragma clang fp contract(off)
  const double acc = a[0] * a[0] + a[1] * a[1] + a[2] * a[2];
  const double jrk = j[0] * j[0] + j[1] * j[1] + j[2] * j[2];
  const double dtcrit = P.eta_s * sqrt(acc / jrk);
  double dtblock = P.dtmax;
  while (dtblock > dtcrit && dtblock > P.dtmin) dtblock = dtblock * 0.5;
  while (calc_modulus(t_gl, dtblock, P.dtmax) != 0.0) {
    dtblock = dtblock * 0.5;
    if (dtblock < P.dtmin) return 0.0;
  }
  return dtblock;
}

// ---------------------------------------------------------------- control
// Step state in device memory.  No kernel reads what its own other blocks
// write here, so a step needs neither fences nor counted blocks: pg6h_select
// reads the state between the steps and writes the step's own, pg6h_force and
// pg6h_finish read that, and block 0 of pg6h_finish writes the state between
// the steps.  The lengths of the active lists of this step and the next take
// turns (pg6h_finish clears the next one's).
struct Ctl {
  // between the steps: pg6h_finish, and the host between runs
  double t_gl;              // time inside the current window [0, dtmax)
  double t_end;             // a step is taken only while t_mod * dtmax + t_gl < t_end
  long long t_mod;          // completed windows (t = t_mod * dtmax + t_gl)
  long long nsteps;         // particle steps taken
  long long nblocks;        // block steps taken
  int last_nact;            // active particles of the last step taken
  int bad;                  // particles whose step fell below dtmin
  // of the step: pg6h_select
  double tnext;             // min(t + dt)
  int run;                  // 0: the step is past t_end and nothing is done
  int turn;                 // the list length in use
  int nact[2];              // length of the active list being formed
};

// Whether the step being queued is past the end of the run.
__device__ inline bool pg6h_skip(const Ctl* c, double dtmax) {
#pragma clang fp contract(off)
  return (double)c->t_mod * dtmax + c->t_gl >= c->t_end;
}

// Split of the force work of `nact` active particles over all nj
// j-particles: tiles of 64 i times ns j-ranges of jper addresses, one block
// of kForceWaves wavefronts per (tile, range) item; wavefront w of the block
// takes the w-th of kForceWaves equal pieces of the range (a multiple of 16
// addresses, at least min_jper).  About `target` wavefronts of work in all.
constexpr int kForceWaves = 8;
// pg6h_force writes a record of kRec doubles per (range, active slot): ax,
// ay, az, pot, jx, jy, jz and one unused, the eight wavefronts' threads in
// that order.  Range s, slot k: record s * stride + k.
constexpr int kRec = 8;
static_assert(kForceWaves == kRec, "pg6h_force writes one component per thread");

// What the host knows of the split before nact: with up to `tiles` tiles the
// number of ranges is the largest there is, ns of jper addresses.
struct Split {
  int nj, blocks, max_ns, tiles, ns, jper;
};
struct Plan {
  int ntiles, ns, jper, stride;
};

__host__ __device__ inline void pg6h_ranges(int nj, int want, int* ns, int* jper) {
  const int q = 16 * kForceWaves;
  *jper = ((nj + want - 1) / want + q - 1) / q * q;
  *ns = (nj + *jper - 1) / *jper;
}

inline Split pg6h_split(int nj, int target, int min_jper) {
  Split sp;
  sp.nj = nj;
  sp.blocks = target / kForceWaves;
  sp.max_ns = nj / (kForceWaves * min_jper);
  if (sp.max_ns < 1) sp.max_ns = 1;
  // ceil(blocks / tiles) >= max_ns up to this many tiles
  sp.tiles = sp.max_ns > 1 ? (sp.blocks - 1) / (sp.max_ns - 1) : INT_MAX;
  pg6h_ranges(nj, sp.max_ns, &sp.ns, &sp.jper);
  return sp;
}

__device__ inline Plan pg6h_plan(int nact, const Split& sp) {
  Plan p;
  p.ntiles = (nact + 63) / 64;
  p.stride = p.ntiles * 64;
  if (p.ntiles <= sp.tiles) {  // no division on a short step's way
    p.ns = sp.ns;
    p.jper = sp.jper;
  } else {
    pg6h_ranges(sp.nj, (sp.blocks + p.ntiles - 1) / p.ntiles, &p.ns, &p.jper);
  }
  return p;
}

// ---------------------------------------------------------------- next time
// v of the lane that a DPP control names (within its row of 16).
template <int CTRL>
__device__ inline double dpp(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline double readlane(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// Minimum over the wavefront (all lanes active): rotations by 8, 4, 2 and 1
// in the rows, then the four rows.
__device__ inline double wave_min(double v) {
  v = fmin(v, dpp<0x128>(v));
  v = fmin(v, dpp<0x124>(v));
  v = fmin(v, dpp<0x122>(v));
  v = fmin(v, dpp<0x121>(v));
  return fmin(fmin(readlane(v, 0), readlane(v, 16)), fmin(readlane(v, 32), readlane(v, 48)));
}

// t_next = min_i (t_i + dt_i) is the minimum of mins[], one value per
// wavefront of pg6h_finish; without a value 1e300.  This fills it after the
// start-up, with the same grid.
constexpr double kNoTime = 1e300;
__global__ __launch_bounds__(256) void pg6h_min_time(int n, State S, double* __restrict__ mins) {
#pragma clang fp contract(off)
  double v = kNoTime;
  const int i0 = blockIdx.x * blockDim.x + threadIdx.x;
  for (int i = i0; i < n; i += gridDim.x * blockDim.x) v = fmin(v, S.t[i] + S.dt[i]);
  v = wave_min(v);
  if ((threadIdx.x & 63) == 0) mins[i0 / 64] = v;
}

// ---------------------------------------------------------------- selection
// t_next; every j predicted to it (the board's predictor, pg6_predict_j); the
// active particles (t + dt == t_next, global_time of banana01.c /
// timestep.c:81-92) appended to the active list with their i data as
// predict_exmotion (hermite.c:39-62) computes it: FP64 position and
// velocity at t_next, id = address.  rest[block] = the smallest t + dt of the
// block's particles that do not move (kNoTime: none).  Block = 256 threads,
// one particle each.  All loads of a thread are issued before the first wait;
// only the length of the list and what depends on it come after.
__global__ __launch_bounds__(256) void pg6h_select(int n, State S, Params P, Ctl* ctl,
                                                   const double* __restrict__ mins, int nmins,
                                                   pg6::JState js, pg6::JPred jp,
                                                   int* __restrict__ act,
                                                   double* __restrict__ ipos,
                                                   double* __restrict__ ivel,
                                                   int* __restrict__ iid,
                                                   double* __restrict__ rest) {
#pragma clang fp contract(off)
  __shared__ double s_min[4], s_rest[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = i < n;
  const pg6::JRaw raw = pg6::pg6_load_j(i, valid, js);
  double t = 0.0, dts = 0.0, v = kNoTime;
  if (valid) {
    t = S.t[i];
    dts = S.dt[i];
  }
  for (int q = threadIdx.x; q < nmins; q += 256) v = fmin(v, mins[q]);
  if (pg6h_skip(ctl, P.dtmax)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl->run = 0;
    return;
  }
  const int turn = (int)(ctl->nblocks & 1);
  v = wave_min(v);
  if (lane == 0) s_min[wave] = v;
  __syncthreads();
  v = fmin(fmin(s_min[0], s_min[1]), fmin(s_min[2], s_min[3]));
  const double tnext = v < kNoTime ? v : (double)INFINITY;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    ctl->tnext = tnext;
    ctl->turn = turn;
    ctl->run = 1;
  }
  const double tn = valid ? t + dts : kNoTime;
  const bool a = valid && tn == tnext;
  const unsigned long long mask = __ballot(a);
  int base = 0;
  if (lane == 0 && mask != 0ull) base = atomicAdd(&ctl->nact[turn], __popcll(mask));
  double x[3], vel[3], ac[3], j[3];
  if (a)
    for (int d = 0; d < 3; ++d) {
      x[d] = S.x[3 * i + d];
      vel[d] = S.v[3 * i + d];
      ac[d] = S.a[3 * i + d];
      j[d] = S.j[3 * i + d];
    }
  pg6::pg6_predict_j(i, valid, tnext, raw, jp);
  const double r = wave_min(a ? kNoTime : tn);
  if (lane == 0) s_rest[wave] = r;
  base = __builtin_amdgcn_readfirstlane(base);
  if (a) {
    const int k = base + __popcll(mask & ((1ull << lane) - 1ull));
    act[k] = i;
    const double dt = tnext - t;
    const double dt2 = dt * dt;
    const double dt3 = dt * dt2;
    for (int d = 0; d < 3; ++d) {
      ipos[3 * k + d] = x[d] + vel[d] * dt + ac[d] * dt2 * kSecond + j[d] * dt3 * kThird;
      ivel[3 * k + d] = vel[d] + ac[d] * dt + j[d] * dt2 * kSecond;
    }
    iid[k] = i;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    rest[blockIdx.x] = fmin(fmin(s_rest[0], s_rest[1]), fmin(s_rest[2], s_rest[3]));
}

// ---------------------------------------------------------------- force
// pg6::pg6_range_h for a range of at most kStage addresses (one tile of it),
// the same sums: the wavefront's lanes read all records at once into its
// `stage`, where pg6_range_h waits for scalar loads of four records after
// four (a step's force on up to 64 particles of 16384: 4.9 us, so 6.5).  Every
// pair is tested by id, which costs less than the loads and exchanges that
// show where it can be left out.  Longer ranges are bound by the pairs, where
// reading the records from LDS gained nothing.
constexpr int kStage = 32;
__device__ inline pg6::RangeSums short_range(double xi, double yi, double zi, float vxi, float vyi,
                                             float vzi, int idi, float eps2, int j0, int j1,
                                             const pg6::JPred& jp, float4* stage) {
  const int lane = threadIdx.x & 63;
  const float4* rec = jp.rec + 3 * (size_t)j0;
  for (int e = lane; e < 3 * (j1 - j0); e += 64) stage[e] = rec[e];
  const float xih = (float)xi, yih = (float)yi, zih = (float)zi;
  const float xil = (float)(xi - (double)xih);
  const float yil = (float)(yi - (double)yih);
  const float zil = (float)(zi - (double)zih);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  pg6::TileAcc t{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0u};
#pragma unroll 4
  for (int j = 0; j < j1 - j0; ++j) {
    const float4 a = stage[3 * j], b = stage[3 * j + 1], c = stage[3 * j + 2];
    pg6::pg6_pair_h<true, false>(t, (a.x - xih) + (b.x - xil), (a.y - yih) + (b.y - yil),
                                 (a.z - zih) + (b.z - zil), b.w - vxi, c.x - vyi, c.y - vzi, a.w,
                                 eps2, __float_as_int(c.z) == idi, 0u);
  }
  return {(double)t.ax, (double)t.ay, (double)t.az, (double)t.pot,
          (double)t.jx, (double)t.jy, (double)t.jz, 0.f, -1};
}

// Acc, jerk and pot of the active list against all n j-particles with the
// two-float pair loop (pg6::pg6_range_h).  Block = kForceWaves wavefronts;
// blocks walk the (i-tile, j-range) items of pg6h_plan.  The wavefronts'
// sums over their pieces of a range are added in LDS in wavefront order and
// written as one FP64 partial per range.
__global__ __launch_bounds__(64 * kForceWaves) void pg6h_force(
    int n, float eps2, const Ctl* ctl, Split split, const double* __restrict__ ipos,
    const double* __restrict__ ivel, const int* __restrict__ iid, pg6::JPred jp,
    double* __restrict__ part) {
  if (!ctl->run) return;
  const int nact = ctl->turn ? ctl->nact[1] : ctl->nact[0];
  const Plan pl = pg6h_plan(nact, split);
  const int items = pl.ntiles * pl.ns;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int piece = pl.jper / kForceWaves;
  __shared__ double red[7][kForceWaves * 64 + 8];  // the 8 spread the components over the banks
  __shared__ float4 stage[kForceWaves][3 * kStage];
  for (int it = blockIdx.x; it < items; it += gridDim.x) {
    const int sp = pl.ntiles == 1 ? it : it / pl.ntiles, tile = it - sp * pl.ntiles;
    const int i = tile * 64 + lane;
    const int ic = i < nact ? i : nact - 1;  // padding lanes repeat the last slot
    const int j0 = min(n, sp * pl.jper + w * piece), j1 = min(n, j0 + piece);
    const double x = ipos[3 * ic], y = ipos[3 * ic + 1], z = ipos[3 * ic + 2];
    const float vx = (float)ivel[3 * ic], vy = (float)ivel[3 * ic + 1],
                vz = (float)ivel[3 * ic + 2];
    const pg6::RangeSums r =
        piece <= kStage
            ? short_range(x, y, z, vx, vy, vz, iid[ic], eps2, j0, j1, jp, stage[w])
            : pg6::pg6_range_h<false>(x, y, z, vx, vy, vz, iid[ic], eps2, j0, j1, jp);
    red[0][threadIdx.x] = r.ax;
    red[1][threadIdx.x] = r.ay;
    red[2][threadIdx.x] = r.az;
    red[3][threadIdx.x] = r.pot;
    red[4][threadIdx.x] = r.jx;
    red[5][threadIdx.x] = r.jy;
    red[6][threadIdx.x] = r.jz;
    __syncthreads();
    const int slot = threadIdx.x / kRec, c = threadIdx.x % kRec;
    const int k = tile * 64 + slot;
    if (c < 7 && k < nact) {
      double sum = 0.0;
      for (int q = 0; q < kForceWaves; ++q) sum += red[c][q * 64 + slot];
      part[((size_t)sp * pl.stride + k) * kRec + c] = sum;
    }
    __syncthreads();
  }
}

// j-memory record of particle i as set_particle_on_grape / the end of
// integrate_exmotion write it (banana01.c:206-236, hermite.c:244-274):
// acc/2, jerk/6, snap 0.
__device__ inline void store_j(const State& S, int i, pg6::JState js) {
#pragma clang fp contract(off)
  const double over2 = 0.5, over6 = 1.0 / 6.0;
  js.x[i] = S.x[3 * i];
  js.y[i] = S.x[3 * i + 1];
  js.z[i] = S.x[3 * i + 2];
  js.vx[i] = S.v[3 * i];
  js.vy[i] = S.v[3 * i + 1];
  js.vz[i] = S.v[3 * i + 2];
  js.ax[i] = S.a[3 * i] * over2;
  js.ay[i] = S.a[3 * i + 1] * over2;
  js.az[i] = S.a[3 * i + 2] * over2;
  js.kx[i] = S.j[3 * i] * over6;
  js.ky[i] = S.j[3 * i + 1] * over6;
  js.kz[i] = S.j[3 * i + 2] * over6;
  js.m[i] = S.m[i];
  js.t[i] = S.t[i];
  js.idx[i] = i;
}

// ---------------------------------------------------------------- corrector
// What the corrector needs of active slot k = particle i, in lane d of four:
// the axis d (lane 3 repeats the last).
struct Own {
  double a0, j0, x1, v1, t, dts, m;
};

__device__ inline Own load_own(int k, int i, int d, const State& S,
                               const double* __restrict__ ipos, const double* __restrict__ ivel) {
  const size_t e = 3 * (size_t)i + min(d, 2), g = 3 * (size_t)k + min(d, 2);
  return {S.a[e], S.j[e], ipos[g], ivel[g], S.t[i], S.dt[i], S.m[i]};
}

// correct (hermite.c:66-110) and dt_criterion (timestep.c:50-79) for the
// particle i of four lanes, lane d < 3 with its axis and the force a1 and jerk
// j1 along it, lane 3 with a1 = the potential; then the j-memory update.  A
// step that ends the dtmax window stores t = 0 (reset_time, timestep.c:166-174:
// every particle is active then).  Returns the new t + dt.
__device__ inline double correct_quad(const Own& o, int i, int d, double a1, double j1,
                                      const State& S, const Params& P, const pg6::JState& js,
                                      int* bad) {
#pragma clang fp contract(off)
  const double dts = o.dts, a0 = o.a0, j0 = o.j0;
  const double ts = o.t + dts;  // p0.t (hermite.c:154)
  const double dtsinv = 1.0 / dts;
  const double s0 = 2.0 * (-3.0 * (a0 - a1) - (2.0 * j0 + j1) * dts) * dtsinv * dtsinv;
  const double c0 = 6.0 * (2.0 * (a0 - a1) + (j0 + j1) * dts) * dtsinv * dtsinv * dtsinv;
  double x1 = o.x1, v1 = o.v1;
  x1 += s0 * dts * dts * dts * dts * kFourth + c0 * dts * dts * dts * dts * dts * kFifth;
  v1 += s0 * dts * dts * dts * kThird + c0 * dts * dts * dts * dts * kFourth;
  // dt_criterion
  const double s1 = s0 + c0 * dts;
  auto norm = [](double e) {  // of the three axes' values
    const double q = e * e;
    return sqrt(dpp<0x00>(q) + dpp<0x55>(q) + dpp<0xAA>(q));
  };
  const double acc = norm(a1), jrk = norm(j1), snp = norm(s1), crc = norm(c0);
  const double dti = P.eta * sqrt((acc * snp + jrk * jrk) / (jrk * crc + snp * snp));
  double dtn = dts;
  if (dti < dtn) {
    while (dtn > dti && dtn > P.dtmin) dtn = dtn * 0.5;
  } else if (dti > 2.0 * dtn) {
    if (calc_modulus(ts, 2.0 * dtn, P.dtmax) == 0.0) dtn = 2.0 * dtn;
  }
  const double tnew = ts == P.dtmax ? 0.0 : ts;
  const double over2 = 0.5, over6 = 1.0 / 6.0;  // of the j-memory, as store_j
  if (d == 3) {
    if (!(dtn >= P.dtmin)) atomicAdd(bad, 1);
    S.pot[i] = a1;
    S.t[i] = tnew;
    S.dt[i] = dtn;
    js.m[i] = o.m;
    js.t[i] = tnew;
    js.idx[i] = i;
  } else {
    const size_t e = 3 * (size_t)i + d;
    S.x[e] = x1;
    S.v[e] = v1;
    S.a[e] = a1;
    S.j[e] = j1;
    (d == 0 ? js.x : d == 1 ? js.y : js.z)[i] = x1;
    (d == 0 ? js.vx : d == 1 ? js.vy : js.vz)[i] = v1;
    (d == 0 ? js.ax : d == 1 ? js.ay : js.az)[i] = a1 * over2;
    (d == 0 ? js.kx : d == 1 ? js.ky : js.kz)[i] = j1 * over6;
  }
  return tnew + dtn;
}

// Sums each active particle's j-range partials in a fixed order (four lanes
// per particle for up to 16 ranges, one wavefront per particle with a fixed
// butterfly for more), corrects it (correct_quad), and leaves in mins[], one
// value per wavefront, the smallest new t + dt and of rest[nrest]; block 0
// closes the step in Ctl.
//
// Half of the steps of 16384 particles move up to 7, so this is a chain of
// latencies: the list, the particle and its partials in one flight, the sums,
// the corrector with an axis per lane.  No step ends in atomics: the next
// pg6h_select takes the minimum of mins[].  5 us a step, the integration of
// 16384 particles 22 us a step; one lane a particle, each component's partials
// apart, an atomic minimum and a count of the blocks that are done took 10 us
// and 28.
__global__ __launch_bounds__(256) void pg6h_finish(Params P, Ctl* ctl, Split split,
                                                   const int* __restrict__ act, State S,
                                                   const double* __restrict__ ipos,
                                                   const double* __restrict__ ivel,
                                                   const double* __restrict__ part,
                                                   const double* __restrict__ rest, int nrest,
                                                   double* __restrict__ mins, pg6::JState js) {
#pragma clang fp contract(off)
  if (!ctl->run) return;
  const int turn = ctl->turn;
  const int nact = turn ? ctl->nact[1] : ctl->nact[0];
  const int lane = threadIdx.x & 63;
  // the block's wavefronts are those of distant particles: few ones spread over the CUs
  const int w = (threadIdx.x / 64) * gridDim.x + blockIdx.x, nw = 4 * gridDim.x;
  double tmin = kNoTime;
  for (int b = w + nw * lane; b < nrest; b += nw * 64) tmin = fmin(tmin, rest[b]);
  const Plan pl = pg6h_plan(nact, split);
  const int d = lane & 3;
  if (pl.ns <= 16) {
    for (int k = w * 16 + lane / 4; k < nact; k += nw * 16) {
      const int i = act[k];
      const Own o = load_own(k, i, d, S, ipos, ivel);
      double a1 = 0.0, j1 = 0.0;
      for (int sp = 0; sp < pl.ns; ++sp) {
        const double* r = part + ((size_t)sp * pl.stride + k) * kRec + d;
        a1 += r[0];
        j1 += r[4];  // lane 3: unused
      }
      tmin = fmin(tmin, correct_quad(o, i, d, a1, j1, S, P, js, &ctl->bad));
    }
  } else {
    for (int k = w; k < nact; k += nw) {
      const int i = act[k];
      double f[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      for (int sp = lane; sp < pl.ns; sp += 64) {
        const double* r = part + ((size_t)sp * pl.stride + k) * kRec;
        for (int c = 0; c < 7; ++c) f[c] += r[c];
      }
      const Own o = load_own(k, i, d, S, ipos, ivel);
      // Butterfly over the lanes, each half of which goes on with half of
      // the components: component c ends in the lanes 8 c to 8 c + 7.
      for (int h = 4, x = 32; h >= 1; h >>= 1, x >>= 1)
        for (int c = 0; c < h; ++c) {
          const bool up = (lane & x) != 0;
          const double keep = up ? f[c + h] : f[c], give = up ? f[c] : f[c + h];
          f[c] = keep + __shfl_xor(give, x);
        }
      for (int x = 4; x >= 1; x >>= 1) f[0] += __shfl_xor(f[0], x);
      const double a1 = __shfl(f[0], 8 * d), j1 = __shfl(f[0], 8 * (d + 4));
      if (lane < 4) tmin = fmin(tmin, correct_quad(o, i, d, a1, j1, S, P, js, &ctl->bad));
    }
  }
  tmin = wave_min(tmin);
  if (lane == 0) mins[w] = tmin;
  if (blockIdx.x == 0 && threadIdx.x == 192) {
    const double tnext = ctl->tnext;
    ctl->last_nact = nact;
    ctl->nsteps += nact;
    ctl->nblocks += 1;
    if (tnext == P.dtmax) {  // end of a window: every time restarts at 0
      ctl->t_gl = 0.0;
      ctl->t_mod += 1;
    } else {
      ctl->t_gl = tnext;
    }
    ctl->nact[1 - turn] = 0;
  }
}

// startup_sgmotion (hermite.c:114-142) for every particle: forces at t = 0
// (acc1 etc. in particle order), first time steps, j-memory.
__global__ void pg6h_startup(int n, State S, Params P, const double* __restrict__ acc1,
                             const double* __restrict__ jrk1, const double* __restrict__ pot1,
                             pg6::JState js, int* __restrict__ bad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int d = 0; d < 3; ++d) {
    S.a[3 * i + d] = acc1[3 * i + d];
    S.j[3 * i + d] = jrk1[3 * i + d];
  }
  S.pot[i] = pot1[i];
  const double dt = dt_startup(P, S.t[i], S.a + 3 * i, S.j + 3 * i);
  if (!(dt > 0.0)) atomicAdd(bad, 1);
  S.dt[i] = dt > 0.0 ? dt : P.dtmin;
  store_j(S, i, js);
}

// j-memory record of every particle (set_particle_on_grape).
__global__ void pg6h_store_all(int n, State S, pg6::JState js) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) store_j(S, i, js);
}

// Per-block partial sums of m v^2 and m pot, in FP64 (calc_energy.c:8-33).
__global__ void pg6h_energy_part(int n, State S, double* __restrict__ part) {
#pragma clang fp contract(off)
  __shared__ double s[2][256];
  double ek = 0.0, ew = 0.0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    double v2 = S.v[3 * i] * S.v[3 * i];
    v2 += S.v[3 * i + 1] * S.v[3 * i + 1];
    v2 += S.v[3 * i + 2] * S.v[3 * i + 2];
    ek += S.m[i] * v2;
    ew += S.m[i] * S.pot[i];
  }
  s[0][threadIdx.x] = ek;
  s[1][threadIdx.x] = ew;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) {
      s[0][threadIdx.x] += s[0][threadIdx.x + h];
      s[1][threadIdx.x] += s[1][threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s[0][0];
    part[2 * blockIdx.x + 1] = s[1][0];
  }
}

}  // namespace pg6h
