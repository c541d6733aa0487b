// Batched TreePM short-range force: every tree i-group with its j-list in one
// persistent launch.  No counterpart in the reference, whose caller loops over
// groups with g5_set_xmjMC + g5_calculate_force_on_xMC inside an OpenMP loop
// (the pattern of PG5/newton_quad/source.cpp:813-860).
//
// Inputs (device): pos[np] float4 {x*xs, y*xs, z*xs, m} (positions scaled as
// in PG5/table/libpg5/phantom_g5.c:112-128; periodic images are ghost copies
// appended by the caller); optionally pos64[np][3], the same positions in
// FP64 (unscaled), from which each group forms its separations relative to a
// group origin o (its first i-particle): a position enters the pair loop
// through the reference's ingest conversions applied to x - o instead of x
// (i: float(double(float(x - o)) * xs), PG5/table/libpg5/phantom_g5.c:102-104;
// j: float(x - o) * float(xs) in FP32, :116-127), so separations keep their
// digits where |x| >> |dx| (masses still come from pos[].w); per group g an
// i-list
// ilist[ioff[g] .. +icnt[g])
// and a j-list jlist[joff[g] .. +jcnt[g]) (groups may share list ranges), an
// optional processing order (groups by decreasing cost), and a work counter
// that must be 0 at launch.
// Each block repeatedly takes the next group from the counter and stages the
// group's j-list in LDS tiles (gathered through jlist).  The cut-off shape
// comes from the evaluator: the LDS table (treepm_batch_table, bit-identical
// per pair with the drop-in kernel) or the learned MLP (treepm_batch_mlp).
// Results: acc[i][3] FP64 (written, not accumulated) for every listed i.
#pragma once
#include <hip/hip_runtime.h>

#include "mlp_kernels.h"
#include "table_kernels.h"

namespace pgb {

constexpr int kThreads = 256;    // treepm_batch_mlp block
constexpr int kJTile = 256;
constexpr int kTableBlock = 1024;  // treepm_batch_table default block (256, 512 also built)

// Table evaluator: s = 2 + |dx_s|^2, f from the LDS table (linear: the
// reference's {value, slope}; quadratic: {c0, c1, c2, 0}).
struct TableCut {
  const float2* gtab;
  const float4* gquad;
  int ntab, frc_bit;
};

// Group-origin positions (see above).  o: the group's origin in FP64.
struct Origin {
  const double* pos64;  // null: take the scaled float4 positions as they are
  double xs;
  float xsf;  // float(xs)
};

template <bool I>
__device__ inline float4 load_pos(const float4* __restrict__ pos, const Origin& og, int k,
                                  double ox, double oy, double oz) {
  float4 q = pos[k];
  if (og.pos64) {
    const double* p = og.pos64 + 3 * (size_t)k;
    if (I) {
      q.x = (float)((double)(float)(p[0] - ox) * og.xs);
      q.y = (float)((double)(float)(p[1] - oy) * og.xs);
      q.z = (float)((double)(float)(p[2] - oz) * og.xs);
    } else {
      q.x = (float)(p[0] - ox) * og.xsf;
      q.y = (float)(p[1] - oy) * og.xsf;
      q.z = (float)(p[2] - oz) * og.xsf;
    }
  }
  return q;
}

__device__ inline int take_item(int* counter, int* s_item) {
  __syncthreads();
  if (threadIdx.x == 0) *s_item = atomicAdd(counter, 1);
  __syncthreads();
  return *s_item;
}

// Learned cut-off.  Only pairs inside the cut-off are evaluated, 64 at a time
// whatever i-particle they belong to: a wavefront marks the pairs of its 64
// i-particles in reach, queues them in LDS one lane after the other, runs the
// network over the queue with every lane busy, and each lane adds the results
// of its own pairs in j order.
//
// A block's item is a slice of up to 64 i-particles of a group (slices q, q +
// 4, ... for item 4 group + q), its wavefronts taking the units of j in turn:
// unit (tile, g) holds every G-th j of a tile of kJTile, G = 4, 2 or 1 for a
// block of up to 64, 128 or 256 i (kMlpBlockI at a time).  A unit's sum is
// formed in FP32 and folded into FP64.
//
// Clumpy box of 2^18 particles (3.9e8 listed pairs, 70 % inside the cut-off,
// 50 i-particles per group on average): 8.6-9.5 ms with one network pass per
// j for all lanes of a wavefront (9.2e6 passes of 64 pairs, half of them
// empty lanes or pairs out of reach; the queue needs 4.3e6), 5.2 ms with the
// queue and the matrix cores, 3.3-3.5 ms with slices as items: with whole
// groups the largest (256 i) ran on alone after the others.  Four blocks per
// CU would fit the LDS only without the queue; three hold 130 registers.
constexpr int kMlpBlockI = 256;
constexpr int kMlpQueue = 1024;  // queued pairs per wavefront

// Keeps a wavefront's LDS writes before its other lanes' reads.
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__global__ __launch_bounds__(kThreads, 3) void treepm_batch_mlp(
    int ngroups, const int* __restrict__ order, const int* __restrict__ ioff,
    const int* __restrict__ icnt, const int* __restrict__ ilist, const int* __restrict__ joff,
    const int* __restrict__ jcnt, const int* __restrict__ jlist,
    const float4* __restrict__ pos, Origin og, mlp::Cut mc, double ascale,
    double* __restrict__ acc, int* counter) {
  constexpr int kWaves = kThreads / 64;
  __shared__ float4 s_j[kWaves][kJTile], s_i[kWaves][64];
  __shared__ float s_f[kWaves][kMlpQueue];
  __shared__ unsigned short s_pair[kWaves][kMlpQueue];
  __shared__ double s_red[3][kThreads];
  __shared__ int s_item;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  float4* wj = s_j[wave];
  float4* wi = s_i[wave];
  float* qf = s_f[wave];
  unsigned short* qp = s_pair[wave];
  const mlp::WaveNet net = mlp::load_wave_net(mc.w);
  // r2 > 0 and r2 < r_c^2 (or the S2 core's radius^2) as one unsigned
  // comparison of the float bits: 0 wraps round, NaN lies above
  const unsigned rcb = __float_as_uint(mc.rc2) - 1u;
  const unsigned ppb = mc.pp2 > 0.f ? __float_as_uint(mc.pp2) - 1u : 0u;
  for (;;) {
    const int it = take_item(counter, &s_item);
    if (it / 4 >= ngroups) break;
    const int grp = order ? order[it / 4] : it / 4;
    const int i0 = ioff[grp], ni = icnt[grp];
    const int j0 = joff[grp], nj = jcnt[grp];
    if ((it & 3) * 64 >= ni) continue;  // uniform: every thread read the same item
    double ox = 0.0, oy = 0.0, oz = 0.0;
    if (og.pos64) {
      const double* o = og.pos64 + 3 * (size_t)ilist[i0];
      ox = o[0];
      oy = o[1];
      oz = o[2];
    }
    for (int i1 = (it & 3) * 64; i1 < ni; i1 += kMlpBlockI) {
      const int nib = min(kMlpBlockI, ni - i1 / kMlpBlockI * kMlpBlockI);
      const int G = nib <= 64 ? 4 : (nib <= 128 ? 2 : 1);
      const int nl = min(64, ni - i1);  // lanes with an i-particle
      const bool iv = lane < nl;
      const int ii = ilist[i0 + i1 + (iv ? lane : 0)];
      const float4 ip = load_pos<true>(pos, og, ii, ox, oy, oz);
      wi[lane] = ip;
      // so many j at a time that their pairs with nl lanes fit the queue
      const int step = nl <= kMlpQueue / 32 ? 32 : kMlpQueue / 64;
      // 0, or NaN for an i-particle without a finite position
      double ax = (double)(ip.x - ip.x), ay = (double)(ip.y - ip.y), az = (double)(ip.z - ip.z);
      const int units = G * ((nj + kJTile - 1) / kJTile);
      for (int u = wave; u < units; u += kWaves) {
        const int jt = u / G * kJTile, g = u % G;
        const int nt = min(kJTile, nj - jt);
        const int nsub = nt > g ? (nt - g + G - 1) / G : 0;  // j = jt + g + G t
        for (int t = lane; t < nsub; t += 64)
          wj[t] = load_pos<false>(pos, og, jlist[j0 + jt + g + G * t], ox, oy, oz);
        wave_lds_sync();
        float fax = 0.f, fay = 0.f, faz = 0.f;
        // 64 t at a time: the pairs inside the cut-off in t order (pass 0),
        // then the second term of those inside the S2 core (pass 1).  Pairs
        // outside contribute exactly 0, so leaving them out changes no sum.
        for (int c0 = 0; c0 < nsub; c0 += 64) {
          const int cn = min(64, nsub - c0);
          const float4* sj = wj + c0;
          unsigned long long core = 0ull;  // lane's pairs inside the core
#pragma unroll 1
          for (int pass = 0; pass < 2; ++pass) {
            if (pass == 1 && !__builtin_amdgcn_ballot_w64(core != 0ull)) break;
#pragma unroll 1
            for (int s0 = 0; s0 < cn; s0 += step) {
              const int sn = min(step, cn - s0);
              unsigned m = 0u;  // bit t - s0
              if (pass == 0) {
                unsigned in_core = 0u;
#pragma unroll 4
                for (int t = 0; t < sn; ++t) {
                  const float4 q = sj[s0 + t];
                  const float dx = q.x - ip.x;
                  const float dy = q.y - ip.y;
                  const float dz = q.z - ip.z;
                  const float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                  const unsigned b = __float_as_uint(r2) - 1u;
                  m |= b < rcb ? 1u << t : 0u;
                  in_core |= b < ppb ? 1u << t : 0u;
                }
                m = iv ? m : 0u;
                core |= (unsigned long long)(iv ? in_core : 0u) << s0;
              } else {
                m = (unsigned)(core >> s0) & (step == 32 ? ~0u : (1u << step) - 1u);
              }
              // queue slots: an exclusive sum of the lanes' counts, bit by bit
              const int cnt = __popc(m);
              int base = 0, total = 0;
#pragma unroll
              for (int b = 0; b < 6; ++b) {
                const unsigned long long v = __builtin_amdgcn_ballot_w64((cnt >> b) & 1);
                base += (int)__builtin_amdgcn_mbcnt_hi((unsigned)(v >> 32),
                                                       __builtin_amdgcn_mbcnt_lo((unsigned)v, 0u))
                        << b;
                total += __popcll(v) << b;
              }
              int k = base;
              for (unsigned r = m; r != 0u; r &= r - 1u)
                qp[k++] = (unsigned short)(lane << 6 | (s0 + __builtin_ctz(r)));
              wave_lds_sync();
#pragma unroll 1
              for (int r0 = 0; r0 < total; r0 += 64) {
                const int at = min(r0 + lane, total - 1);
                const int code = qp[at];
                const float4 q = sj[code & 63];
                const float4 p = wi[code >> 6];
                const float dx = q.x - p.x;
                const float dy = q.y - p.y;
                const float dz = q.z - p.z;
                const float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                const float rinv = __builtin_amdgcn_rsqf(r2);
                const float r = r2 * rinv;
                const float v = pass == 0 ? mlp::cut_input(mc, r) : r * mc.inv_pp;
                const float y = mlp::eval_wave(net, v);
                qf[at] = pass == 0 ? mlp::cut_main(mc, y, r, r2, rinv) : y * mc.cpp;
              }
              wave_lds_sync();
              k = base;
              for (unsigned r = m; r != 0u; r &= r - 1u) {
                const float4 q = sj[s0 + __builtin_ctz(r)];
                const float f = qf[k++];
                fax = fmaf(f, q.w * (q.x - ip.x), fax);
                fay = fmaf(f, q.w * (q.y - ip.y), fay);
                faz = fmaf(f, q.w * (q.z - ip.z), faz);
              }
              wave_lds_sync();
            }
          }
        }
        ax += (double)fax;
        ay += (double)fay;
        az += (double)faz;
      }
      __syncthreads();
      s_red[0][tid] = ax;
      s_red[1][tid] = ay;
      s_red[2][tid] = az;
      __syncthreads();
      if (tid < nl) {
        for (int q = 1; q < kWaves; ++q) {
          ax += s_red[0][64 * q + tid];
          ay += s_red[1][64 * q + tid];
          az += s_red[2][64 * q + tid];
        }
        acc[3 * (size_t)ii + 0] = ax * ascale;
        acc[3 * (size_t)ii + 1] = ay * ascale;
        acc[3 * (size_t)ii + 2] = az * ascale;
      }
    }
  }
}

// Table cut-off with lanes packed by phases.  Block = BLOCK threads.  A
// group of n <= BLOCK i-particles takes p = BLOCK / n copies of the i-set:
// lane t holds i-particle t % n and walks the j of each LDS tile with
// jj = t / n, t / n + p, ...; the p phase sums of each i are added in phase
// order at the end.  Lanes in use: n p of BLOCK (at least half, usually far
// more), where whole-wavefront i-blocks of 64, 128 or 256 lanes leave the
// rest of a wavefront idle for every group that is not a multiple of 64.
// Groups larger than BLOCK run in passes of BLOCK.  QUAD: the quadratic
// table (one more FMA and a 16-byte LDS read per pair).
template <int BLOCK, bool QUAD>
__global__ __launch_bounds__(BLOCK) void treepm_batch_table(
    int ngroups, const int* __restrict__ order, const int* __restrict__ ioff,
    const int* __restrict__ icnt, const int* __restrict__ ilist, const int* __restrict__ joff,
    const int* __restrict__ jcnt, const int* __restrict__ jlist,
    const float4* __restrict__ pos, Origin og, TableCut tc, double ascale,
    double* __restrict__ acc, int* counter) {
  // linear: {value, slope} per entry; quadratic: {c0, c1} per entry, then c2
  extern __shared__ float4 s_tab4[];
  float2* s_tab = reinterpret_cast<float2*>(s_tab4);
  float* s_c2 = reinterpret_cast<float*>(s_tab + tc.ntab);
  __shared__ float4 s_j[BLOCK];
  __shared__ double s_red[3][BLOCK];
  __shared__ int s_item;
  const int tid = threadIdx.x;
  for (int k = tid; k < tc.ntab; k += BLOCK) {
    if (QUAD) {
      const float4 q = tc.gquad[k];
      s_tab[k] = make_float2(q.x, q.y);
      s_c2[k] = q.z;
    } else {
      s_tab[k] = tc.gtab[k];
    }
  }
  const int shift = 23 - tc.frc_bit;
  const int base = 1 << (30 - shift);
  const float scut = __uint_as_float((1u << 30) | ((unsigned)(tc.ntab - 1) << shift));
  for (;;) {
    const int it = take_item(counter, &s_item);
    if (it >= ngroups) break;
    const int grp = order ? order[it] : it;
    const int i0 = ioff[grp], ni = icnt[grp];
    const int j0 = joff[grp], nj = jcnt[grp];
    double ox = 0.0, oy = 0.0, oz = 0.0;
    if (og.pos64 && ni > 0) {
      const double* o = og.pos64 + 3 * (size_t)ilist[i0];
      ox = o[0];
      oy = o[1];
      oz = o[2];
    }
    for (int ib = 0; ib < ni; ib += BLOCK) {
      const int nib = min(BLOCK, ni - ib);
      const int p = BLOCK / nib;  // phases
      const int il = tid % nib;
      const int phase = tid / nib;
      const bool live = phase < p;
      const int ii = ilist[i0 + ib + il];
      const float4 ip = load_pos<true>(pos, og, ii, ox, oy, oz);
      double ax = 0.0, ay = 0.0, az = 0.0;
      for (int jt = 0; jt < nj; jt += BLOCK) {
        const int nt = min(BLOCK, nj - jt);
        __syncthreads();
        if (tid < nt) s_j[tid] = load_pos<false>(pos, og, jlist[j0 + jt + tid], ox, oy, oz);
        __syncthreads();
        float fax = 0.f, fay = 0.f, faz = 0.f;
        if (live) {
#pragma unroll 4
          for (int jj = phase; jj < nt; jj += p) {
            const float4 q = s_j[jj];
            const float dx = q.x - ip.x;
            const float dy = q.y - ip.y;
            const float dz = q.z - ip.z;
            const float s = fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, 2.0f)));
            const float f = QUAD ? pgt::table_f_quad(s_tab, s_c2, s, scut, shift, base)
                                 : pgt::table_f(s_tab, s, scut, shift, base);
            fax = fmaf(f, q.w * dx, fax);
            fay = fmaf(f, q.w * dy, fay);
            faz = fmaf(f, q.w * dz, faz);
          }
        }
        ax += (double)fax;
        ay += (double)fay;
        az += (double)faz;
      }
      __syncthreads();
      s_red[0][tid] = ax;
      s_red[1][tid] = ay;
      s_red[2][tid] = az;
      __syncthreads();
      if (tid < nib) {
        double sx = 0.0, sy = 0.0, sz = 0.0;
        for (int q = 0; q < p; ++q) {
          sx += s_red[0][q * nib + tid];
          sy += s_red[1][q * nib + tid];
          sz += s_red[2][q * nib + tid];
        }
        acc[3 * (size_t)ii + 0] = sx * ascale;
        acc[3 * (size_t)ii + 1] = sy * ascale;
        acc[3 * (size_t)ii + 2] = sz * ascale;
      }
    }
  }
}

// Clears the work counter (a kernel, not a memset, so it can sit in a graph).
__global__ void zero_counter(int* counter) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *counter = 0;
}

}  // namespace pgb
