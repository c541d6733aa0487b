// Particle-mesh long-range force of the TreePM split on the GPU.
//
// The table force of PG5/table (f = R(r, eps_PP) - R(r, eps_PM),
// PG5/table/libpg5/pg5_table.c:8-34) is the short-range side; this is the
// long-range side, the periodic force of R(r, eps_PM), i.e. of two S2 spheres
// of diameter a = eps_PM (Hockney & Eastwood sec. 8-3), so that PP + PM is
// the S2-softened Newtonian force of the periodic unit box.  Mesh method:
//   1. TSC assignment of the particles' density on an M^3 mesh (mesh points
//      at integer multiples of h = 1/M): the particles are sorted by bricks
//      of 8^3 mesh points, each block sums up to kChunk particles of a brick
//      into the 10^3 points their stencils cover, held in LDS, and adds those
//      to the mesh (where bricks hold few particles, every stencil point goes
//      straight to the mesh).  The sums are 64-bit fixed point
//      (fix_scale): integer addition is associative, so the mesh does not
//      depend on the order in which the atomics land, nor on the order of the
//      particles inside a brick, and the force is the same bit for bit on
//      every run;
//   2. real-to-complex FFT (FP64; hipFFT, but for the transforms along x of
//      meshes of 32 to 256 points that are powers of two: pm_green_x);
//   3. Green's function -4 pi S(k a)^2 / (k^2 W(k)^2), with S the S2 form
//      factor and W the TSC window, times -i k for each axis (spectral
//      gradient), normalised by 1/M^3;
//   4. three complex-to-real FFTs (the same);
//   5. TSC interpolation of the mesh accelerations back to the particles.
// G = 1, uniform neutralising background (k = 0 dropped), as in Ewald
// summation.
#pragma once
#include <hip/hip_runtime.h>

namespace pm {

// x M, rounded.  Every kernel takes a particle's mesh point from this value: its
// brick is the one its stencil lies in, so whether the product is rounded before
// 0.5 is added (at x = -0.5 / M that decides between two points) must not differ
// from kernel to kernel, as it does where the compiler fuses the two.
__device__ inline double mesh_units(double x, int M) {
#pragma clang fp contract(off)
  return x * (double)M;
}

// Nearest mesh point and TSC weights along one axis, u in mesh units.
__device__ inline int tsc(double u, double w[3]) {
  const double g = floor(u + 0.5);
  const double d = u - g;
  w[0] = 0.5 * (0.5 - d) * (0.5 - d);
  w[1] = 0.75 - d * d;
  w[2] = 0.5 * (0.5 + d) * (0.5 + d);
  return (int)g;
}

__device__ inline int wrap(int i, int m) {
  i %= m;
  return i < 0 ? i + m : i;
}

// Nearest mesh point of the position x, wrapped into [0, M).
__device__ inline int nearest(double x, int M) {
  return wrap((int)floor(mesh_units(x, M) + 0.5), M);
}

// Fixed-point scale of the mass assignment.  Every mesh point receives at
// most sum |m| M^3 (TSC weights of a particle sum to 1), so with
// 2^e <= 2^62 / (sum |m| M^3) no point and no partial sum can overflow a
// signed 64-bit integer; one unit is 2^-e, a relative resolution of
// M^3 / 2^62 of the mean density (4.5e-13 at M = 128).
constexpr int kMassBlocks = 256;

// Clears the mesh (nr doubles; nr is even) and the brick counters, and block b
// < kMassBlocks sums |m| over its particles (FP64, fixed order) into
// msum[b].  Grid: at least kMassBlocks blocks of 256.
__global__ __launch_bounds__(256) void pm_begin(size_t nr, double2* __restrict__ rho, int bricks,
                                                int* __restrict__ count, int n,
                                                const double* __restrict__ mass,
                                                double* __restrict__ msum) {
  const size_t step = gridDim.x * (size_t)256, i0 = blockIdx.x * (size_t)256 + threadIdx.x;
  for (size_t i = i0; i < nr / 2; i += step) rho[i] = make_double2(0.0, 0.0);
  for (size_t i = i0; i < (size_t)bricks; i += step) count[i] = 0;
  if (blockIdx.x >= kMassBlocks) return;  // uniform
  __shared__ double s[256];
  double v = 0.0;
  for (int p = blockIdx.x * 256 + threadIdx.x; p < n; p += kMassBlocks * 256) v += fabs(mass[p]);
  s[threadIdx.x] = v;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) s[threadIdx.x] += s[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) msum[blockIdx.x] = s[0];
}

// 2^e from the block sums, added in block order by one thread.
__device__ inline double fix_scale(const double* msum, int M) {
  double sum = 0.0;
  for (int b = 0; b < kMassBlocks; ++b) sum += msum[b];
  const double bound = sum * (double)M * (double)M * (double)M;
  int e = 0;
  if (bound > 0.0) {
    frexp(bound, &e);  // bound < 2^e
    e = 62 - e;
  }
  return ldexp(1.0, e);
}

// ------------------------------------------------------------ brick sort
// The order of the particles matters for speed only (integer sums, one
// result per particle), so a counting sort by brick does: one pass counts and
// keeps each particle's place in its brick, one block scans the counts, one
// pass writes the particles in brick order.  2^20 particles of a clumpy box
// on a 128^3 mesh: 15 + 12 + 27 us, where a library sort of Morton codes took
// 183 us with its key pass and left the positions to be gathered.
constexpr int kBrick = 8;                 // mesh points per brick edge
constexpr int kBox = kBrick + 2;          // with the stencils' reach
constexpr int kBoxCells = kBox * kBox * kBox;
constexpr int kChunk = 512;               // particles per block of a brick
constexpr int kBrickThreads = 256;
constexpr int kCountThreads = 1024;
constexpr int kCountPer = 4;              // particles per thread of the counting pass
constexpr int kLdsBricks = 4096;          // counted in LDS first up to this many bricks

inline int brick_edges(int M) { return (M + kBrick - 1) / kBrick; }

__device__ inline int brick_of(const double* __restrict__ x, int M, int nb) {
  const int gx = nearest(x[0], M), gy = nearest(x[1], M), gz = nearest(x[2], M);
  return (gx / kBrick * nb + gy / kBrick) * nb + gz / kBrick;
}

// place[p] = {brick, index inside it}; count[brick] += its particles.  With
// LDS counters a block claims its share of a brick with one atomic: a clump
// holds thousands of particles of one brick.
template <bool LDS>
__global__ __launch_bounds__(kCountThreads) void pm_count(int n, const double* __restrict__ pos,
                                                          int M, int nb, int* __restrict__ count,
                                                          int2* __restrict__ place) {
  __shared__ int s_cnt[LDS ? kLdsBricks : 1];
  const int bricks = nb * nb * nb;
  const int p0 = blockIdx.x * kCountThreads * kCountPer + threadIdx.x;
  if (LDS) {
    for (int b = threadIdx.x; b < bricks; b += kCountThreads) s_cnt[b] = 0;
    __syncthreads();
  }
  int2 at[kCountPer];
#pragma unroll
  for (int q = 0; q < kCountPer; ++q) {
    const int p = p0 + q * kCountThreads;
    if (p >= n) continue;
    at[q].x = brick_of(pos + 3 * (size_t)p, M, nb);
    at[q].y = atomicAdd(LDS ? &s_cnt[at[q].x] : &count[at[q].x], 1);
  }
  if (LDS) {
    __syncthreads();
    for (int b = threadIdx.x; b < bricks; b += kCountThreads) {
      const int c = s_cnt[b];
      if (c) s_cnt[b] = atomicAdd(&count[b], c);
    }
    __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < kCountPer; ++q) {
    const int p = p0 + q * kCountThreads;
    if (p >= n) continue;
    if (LDS) at[q].y += s_cnt[at[q].x];
    place[p] = at[q];
  }
}

// Chunk of block b: block b runs on XCD b % 8, and each XCD takes one
// contiguous range of chunks, so that neighbouring bricks meet in its L2.
// -1 for the blocks beyond the chunks.
__device__ inline int chunk_of_block(int b, int nchunks) {
  const int x = b % 8, i = b / 8, q = nchunks / 8, r = nchunks % 8;
  if (i >= q + (x < r ? 1 : 0)) return -1;
  return x * q + min(x, r) + i;
}

// A block's work in the assignment and the interpolation: sorted particles
// [k0, k1) of one brick.
struct Chunk {
  int brick, k0, k1, pad;
};

// Sum over the block's 1024 threads, in every thread; s: an int2 per wavefront.
__device__ inline int2 sum1024(int2 v, int2* s) {
  for (int o = 32; o > 0; o >>= 1) {
    v.x += __shfl_xor(v.x, o);
    v.y += __shfl_xor(v.y, o);
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
  __syncthreads();
  v = make_int2(0, 0);
  for (int w = 0; w < 16; ++w) {
    v.x += s[w].x;
    v.y += s[w].y;
  }
  return v;
}

__device__ inline int2 brick_work(int c) { return make_int2(c, (c + kChunk - 1) / kChunk); }

// Particles and chunks of every 1024 bricks, a block each.
__global__ __launch_bounds__(1024) void pm_tile_sums(int bricks, const int* __restrict__ count,
                                                     int2* __restrict__ tiles) {
  __shared__ int2 s_wave[16];
  const int b = blockIdx.x * 1024 + threadIdx.x;
  const int2 v = sum1024(brick_work(b < bricks ? count[b] : 0), s_wave);
  if (threadIdx.x == 0) tiles[blockIdx.x] = v;
}

// scale[0] from the block sums of |m|, start[b] = first sorted particle of brick
// b, the chunks of all bricks and their number.  One block, or (TILES) one per 1024
// bricks, which begins after the tiles before its own: one block takes 13 us
// over the 4096 bricks of a 128^3 mesh, but 426 over the 262144 of 512^3, where the
// two launches take 11.
template <bool TILES>
__global__ __launch_bounds__(1024) void pm_scan(int bricks, const int* __restrict__ count,
                                                const int2* __restrict__ tiles,
                                                int* __restrict__ start,
                                                Chunk* __restrict__ chunks,
                                                int* __restrict__ nchunks,
                                                const double* __restrict__ msum, int M,
                                                double* __restrict__ scale) {
  __shared__ int2 s_wave[16];
  __shared__ double s_mass[kMassBlocks];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int2 run = make_int2(0, 0);  // particles and chunks before this round
  if (!TILES || blockIdx.x == 0) {
    if (tid < kMassBlocks) s_mass[tid] = msum[tid];
    __syncthreads();
    if (tid == 1023) scale[0] = fix_scale(s_mass, M);
  }
  if (TILES) {
    for (int t = tid; t < (int)blockIdx.x; t += 1024) {
      run.x += tiles[t].x;
      run.y += tiles[t].y;
    }
    run = sum1024(run, s_wave);
  }
  for (int b0 = TILES ? blockIdx.x * 1024 : 0; b0 < bricks; b0 += TILES ? bricks : 1024) {
    const int b = b0 + tid;
    const int c = b < bricks ? count[b] : 0;
    const int2 own = brick_work(c);
    int2 v = own;
    for (int o = 1; o < 64; o <<= 1) {
      const int x = __shfl_up(v.x, o), y = __shfl_up(v.y, o);
      if (lane >= o) {
        v.x += x;
        v.y += y;
      }
    }
    __syncthreads();
    if (lane == 63) s_wave[wave] = v;
    __syncthreads();
    int2 all = make_int2(0, 0);
    for (int w = 0; w < 16; ++w) {
      if (w < wave) {
        v.x += s_wave[w].x;
        v.y += s_wave[w].y;
      }
      all.x += s_wave[w].x;
      all.y += s_wave[w].y;
    }
    if (b < bricks) {
      const int k0 = run.x + v.x - own.x, q0 = run.y + v.y - own.y;
      start[b] = k0;
      for (int q = 0; q < own.y; ++q)
        chunks[q0 + q] = Chunk{b, k0 + q * kChunk, k0 + min(c, (q + 1) * kChunk), 0};
    }
    run.x += all.x;
    run.y += all.y;
  }
  if ((!TILES || blockIdx.x == gridDim.x - 1) && tid == 0 && nchunks) *nchunks = run.y;
}

// Sorted copies: index, and position in mesh units with the mass.
__global__ __launch_bounds__(256) void pm_scatter(int n, const double* __restrict__ pos,
                                                  const double* __restrict__ mass, int M,
                                                  const int* __restrict__ start,
                                                  const int2* __restrict__ place,
                                                  int* __restrict__ order,
                                                  double4* __restrict__ part) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  const int2 at = place[p];
  const int k = start[at.x] + at.y;
  order[k] = p;
  part[k] = make_double4(mesh_units(pos[3 * (size_t)p], M), mesh_units(pos[3 * (size_t)p + 1], M),
                         mesh_units(pos[3 * (size_t)p + 2], M), mass[p]);
}

// v[r % 3] for r in [0, 5).
__device__ inline double pick(const double (&v)[3], int r) {
  return r == 0 || r == 3 ? v[0] : (r == 1 || r == 4 ? v[1] : v[2]);
}

// TSC assignment of the sorted particles as fixed-point integers (units of 1
// / scale[0]) into rho (M^3 signed 64-bit integers, two's complement sums
// through unsigned atomics), one chunk per block.  Bound: LDS atomics (27 per
// particle).  Particles of a clump share their mesh points, so each lane
// takes its 27 points in an order of its own (each axis rotated by the
// lane): in the same order all lanes of a wavefront met on one address.
// 2^20-particle clumpy box, 128^3 mesh: 289 us for runs of 128 particles in
// Morton order with a box of run-time size (48 KB of LDS, 3 blocks per CU,
// integer divisions per point), now 59 us.
__global__ __launch_bounds__(kBrickThreads) void pm_assign(
    const int* __restrict__ nchunks, const Chunk* __restrict__ chunks,
    const double4* __restrict__ part, int M, int nb, const double* __restrict__ scale,
    unsigned long long* __restrict__ rho) {
  __shared__ unsigned long long box[kBoxCells];
  const int at = chunk_of_block(blockIdx.x, *nchunks);
  if (at < 0) return;  // uniform
  const Chunk ck = chunks[at];
  const int tid = threadIdx.x;
  for (int t = tid; t < kBoxCells; t += kBrickThreads) box[t] = 0ull;
  // mesh point of box point (0, 0, 0)
  const int ox = ck.brick / (nb * nb) * kBrick - 1, oy = ck.brick / nb % nb * kBrick - 1,
            oz = ck.brick % nb * kBrick - 1;
  const double m3 = (double)M * (double)M * (double)M * scale[0];
  const int ra = tid % 3, rb = tid / 3 % 3, rc = tid / 9 % 3;
  __syncthreads();
  for (int k = ck.k0 + tid; k < ck.k1; k += kBrickThreads) {
    const double4 q = part[k];
    double vx[3], vy[3], vz[3];
    const int gx = wrap(tsc(q.x, vx), M), gy = wrap(tsc(q.y, vy), M), gz = wrap(tsc(q.z, vz), M);
    const int first = ((gx - 1 - ox) * kBox + gy - 1 - oy) * kBox + gz - 1 - oz;
    const double qm = q.w * m3;  // mass / h^3 in fixed-point units
    // the weights in this lane's order
    const double wx[3] = {pick(vx, ra), pick(vx, ra + 1), pick(vx, ra + 2)};
    const double wy[3] = {pick(vy, rb), pick(vy, rb + 1), pick(vy, rb + 2)};
    const double wz[3] = {pick(vz, rc), pick(vz, rc + 1), pick(vz, rc + 2)};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int ia = first + (a + ra < 3 ? a + ra : a + ra - 3) * (kBox * kBox);
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        const int iab = ia + (b + rb < 3 ? b + rb : b + rb - 3) * kBox;
        const double wab = qm * wx[a] * wy[b];
#pragma unroll
        for (int c = 0; c < 3; ++c)
          atomicAdd(&box[iab + (c + rc < 3 ? c + rc : c + rc - 3)],
                    (unsigned long long)llrint(wab * wz[c]));
      }
    }
  }
  __syncthreads();
  for (int t = tid; t < kBoxCells; t += kBrickThreads) {
    const unsigned long long v = box[t];
    if (v == 0ull) continue;
    // a point that a stencil reached is at most one beyond the mesh
    int ix = ox + t / (kBox * kBox), iy = oy + t / kBox % kBox, iz = oz + t % kBox;
    ix += ix < 0 ? M : (ix >= M ? -M : 0);
    iy += iy < 0 ? M : (iy >= M ? -M : 0);
    iz += iz < 0 ? M : (iz >= M ? -M : 0);
    atomicAdd(&rho[((size_t)ix * M + iy) * M + iz], v);
  }
}

// The same without the sort, every stencil point straight to rho: for few
// particles per brick, whose boxes would be mostly empty.
__global__ __launch_bounds__(256) void pm_assign_direct(int n, const double* __restrict__ pos,
                                                        const double* __restrict__ mass, int M,
                                                        const double* __restrict__ scale,
                                                        unsigned long long* __restrict__ rho) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  double wx[3], wy[3], wz[3];
  const int gx = tsc(mesh_units(pos[3 * (size_t)p], M), wx);
  const int gy = tsc(mesh_units(pos[3 * (size_t)p + 1], M), wy);
  const int gz = tsc(mesh_units(pos[3 * (size_t)p + 2], M), wz);
  const double qm = mass[p] * ((double)M * (double)M * (double)M * scale[0]);
  for (int a = 0; a < 3; ++a) {
    const size_t ix = (size_t)wrap(gx + a - 1, M) * M;
    for (int b = 0; b < 3; ++b) {
      const size_t iy = (ix + wrap(gy + b - 1, M)) * M;
      const double wab = qm * wx[a] * wy[b];
      for (int c = 0; c < 3; ++c)
        atomicAdd(&rho[iy + wrap(gz + c - 1, M)], (unsigned long long)llrint(wab * wz[c]));
    }
  }
}

// The fixed-point mesh back to FP64 in place: rho[i] = int64(bits) / scale.
__global__ void pm_fix_to_double(size_t nr, const double* __restrict__ scale, double* rho) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nr) return;
  const long long v = reinterpret_cast<const long long*>(rho)[i];
  rho[i] = (double)v / scale[0];
}

// S2 form factor of a sphere of diameter a at wave number k.
__device__ inline double s2_form(double k, double a) {
  const double u = k * a * 0.5;
  if (u < 1e-3) return 1.0 - u * u / 15.0;
  const double u2 = u * u;
  return 12.0 / (u2 * u2) * (2.0 - 2.0 * cos(u) - u * sin(u));
}

__device__ inline double sinc(double x) { return fabs(x) < 1e-12 ? 1.0 : sin(x) / x; }

// Potential per density of a mode (kx, ky, kz) with window w = sinc sinc sinc,
// scaled by 1/M^3; 0 for the mean and for Nyquist modes (the gradient of one
// has no real counterpart).
__device__ inline double green(int M, double a, double kx, double ky, double kz, double w,
                               bool nyquist) {
  const double k2 = kx * kx + ky * ky + kz * kz;
  if (!(k2 > 0.0) || nyquist) return 0.0;
  const double w3 = w * w * w;
  const double s = s2_form(sqrt(k2), a);
  return -4.0 * 3.14159265358979323846 * s * s / (k2 * w3 * w3) /
         ((double)M * (double)M * (double)M);
}
__device__ inline double wave_number(int i, int M) {
  const double tp = 2.0 * 3.14159265358979323846;
  return tp * (i <= M / 2 - 1 || M == 1 ? i : i - M);
}

// rhok: M x M x (M/2+1) complex (double2); out: 3 such arrays, the
// transformed accelerations of each axis, already scaled by 1/M^3.
__global__ void pm_green(int M, double a, const double2* __restrict__ rhok,
                         double2* __restrict__ fk) {
  const int Mz = M / 2 + 1;
  const size_t nk = (size_t)M * M * Mz;
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nk) return;
  const int iz = (int)(k % Mz);
  const int iy = (int)((k / Mz) % M);
  const int ix = (int)(k / ((size_t)Mz * M));
  const double kv[3] = {wave_number(ix, M), wave_number(iy, M),
                        2.0 * 3.14159265358979323846 * iz};
  const double h2 = 0.5 / M;
  const double g = green(M, a, kv[0], kv[1], kv[2],
                         sinc(kv[0] * h2) * sinc(kv[1] * h2) * sinc(kv[2] * h2),
                         ix == M / 2 || iy == M / 2 || iz == M / 2);
  const double2 r = rhok[k];
  const double pr = r.x * g, pi = r.y * g;  // phi_k
  for (int d = 0; d < 3; ++d)               // -i k phi = (k pi, -k pr)
    fk[d * nk + k] = make_double2(kv[d] * pi, -kv[d] * pr);
}

__device__ inline double2 cadd(double2 a, double2 b) { return {a.x + b.x, a.y + b.y}; }
__device__ inline double2 csub(double2 a, double2 b) { return {a.x - b.x, a.y - b.y}; }
__device__ inline double2 cmul(double2 a, double2 w) {
  return {a.x * w.x - a.y * w.y, a.x * w.y + a.y * w.x};
}

// Forward transform of kCols columns of M = 2^p points, a thread holding the
// points b + k M/4 of one column in v[k], before and after.  Radix-4 passes of
// the self-sorting (Stockham) form: pass s = 1, 4, 16, ... combines the
// points b + k M/4, which every pass reads, and leaves them at q + s (4 p + k)
// with p = b / s, q = b % s; an odd power ends with a radix-2 pass.  s: the
// columns in LDS; tw[j] = exp(-2 pi i j / M).
constexpr int kCols = 8;
template <int M>
__device__ inline void fft_columns(double2 v[4], double2 (*s)[kCols], const double2* tw, int b,
                                   int col) {
#pragma unroll
  for (int st = 1; M / st >= 4; st *= 4) {
    const int p = b / st, q = b % st;
    const double2 ac = cadd(v[0], v[2]), am = csub(v[0], v[2]);
    const double2 bd = cadd(v[1], v[3]), bm = csub(v[1], v[3]);
    const double2 jb = {-bm.y, bm.x};
    v[0] = cadd(ac, bd);
    v[1] = csub(am, jb);
    v[2] = csub(ac, bd);
    v[3] = cadd(am, jb);
    if (M / st == 4) break;  // p = 0: in place, no factors
#pragma unroll
    for (int k = 1; k < 4; ++k) v[k] = cmul(v[k], tw[k * p * st]);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) s[q + st * (4 * p + k)][col] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = s[b + k * (M / 4)][col];
    if (M / st == 8) {
      const double2 a = v[0], c = v[1];
      v[0] = cadd(a, v[2]);
      v[2] = csub(a, v[2]);
      v[1] = cadd(c, v[3]);
      v[3] = csub(c, v[3]);
      break;
    }
  }
}

// pm_green between the two transforms along x: rhok holds the density's
// transforms over (y, z) of each x plane, and fk gets what is left to be
// transformed back over (y, z), so that the modes pass through memory once.
// The y and z components share their transform along x (k_y and k_z do not
// depend on it).  Block = 2 M threads: kCols neighbouring (y, z) columns of M
// points, M/4 threads each.
//
// A mesh of 128^3: 22.8 us, of which 15 would move the 17 MB read and 51 MB
// written at the rate of a copy; the library's passes along x took 13 and
// 25.4, pm_green 22.2 between them.  Bound: memory, with the FP64 functions of
// green() behind it.
template <int M>
__global__ __launch_bounds__(2 * M) void pm_green_x(double a, const double2* __restrict__ twiddle,
                                                    const double2* __restrict__ rhok,
                                                    double2* __restrict__ fk) {
  constexpr int Mz = M / 2 + 1, kStride = M * Mz;
  static_assert(kStride % kCols == 0, "whole blocks of columns");
  __shared__ double2 s[M][kCols];
  __shared__ double2 tw[M];
  __shared__ double s_sinc[M / 2 + 1];
  const int tid = threadIdx.x, col = tid % kCols, b = tid / kCols;
  const int c = blockIdx.x * kCols + col;
  const double2* src = rhok + c;
  double2 v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = src[(size_t)(b + k * (M / 4)) * kStride];
  if (tid < M) tw[tid] = twiddle[tid];
  if (tid <= M / 2) s_sinc[tid] = sinc(2.0 * 3.14159265358979323846 * tid * (0.5 / M));
  __syncthreads();
  fft_columns<M>(v, s, tw, b, col);
  const int iy = c / Mz, iz = c % Mz;
  const double ky = wave_number(iy, M), kz = 2.0 * 3.14159265358979323846 * iz;
  const double wy = s_sinc[iy <= M / 2 ? iy : M - iy], wz = s_sinc[iz];
  double2 fx[4], fp[4];  // real and imaginary parts swapped: the forward transform inverts
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int ix = b + k * (M / 4);
    const double kx = wave_number(ix, M);
    const double g = green(M, a, kx, ky, kz, s_sinc[ix <= M / 2 ? ix : M - ix] * wy * wz,
                           ix == M / 2 || iy == M / 2 || iz == M / 2);
    const double pr = v[k].x * g, pi = v[k].y * g;  // phi_k; -i k phi = (k pi, -k pr)
    fx[k] = make_double2(-kx * pr, kx * pi);
    fp[k] = make_double2(-pr, pi);
  }
  fft_columns<M>(fx, s, tw, b, col);
  fft_columns<M>(fp, s, tw, b, col);
  double2* dst = fk + c;
  constexpr size_t nk = (size_t)M * kStride;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const size_t e = (size_t)(b + k * (M / 4)) * kStride;
    dst[e] = make_double2(fx[k].y, fx[k].x);
    dst[nk + e] = make_double2(ky * fp[k].y, ky * fp[k].x);
    dst[2 * nk + e] = make_double2(kz * fp[k].y, kz * fp[k].x);
  }
}

// TSC interpolation of a chunk of sorted particles: the block loads the
// brick's 10^3 points of the three mesh accelerations into LDS (24 KB) once,
// where every particle gathered its 81 values from memory (206 us for the
// 2^20-particle box; now 63 us with chunks in launch order and 45 us with
// each XCD on a range of its own).  Bound: memory, 150 MB of boxes through L2
// and 24 scattered bytes written per particle.
__global__ __launch_bounds__(kBrickThreads) void pm_interp(
    const int* __restrict__ nchunks, const Chunk* __restrict__ chunks,
    const int* __restrict__ order, const double4* __restrict__ part, int M, int nb,
    const double* __restrict__ f, double* __restrict__ acc) {
  __shared__ double box[3][kBoxCells];
  const int at = chunk_of_block(blockIdx.x, *nchunks);
  if (at < 0) return;  // uniform
  const Chunk ck = chunks[at];
  const int tid = threadIdx.x;
  const size_t nr = (size_t)M * M * M;
  const int ox = ck.brick / (nb * nb) * kBrick - 1, oy = ck.brick / nb % nb * kBrick - 1,
            oz = ck.brick % nb * kBrick - 1;
  for (int t = tid; t < kBoxCells; t += kBrickThreads) {
    int ix = ox + t / (kBox * kBox), iy = oy + t / kBox % kBox, iz = oz + t % kBox;
    // the box of a last, partly filled brick passes the mesh's end by up to 8
    // points (M >= 8)
    auto inside = [M](int i) {
      i += i < 0 ? M : 0;
      i -= i >= M ? M : 0;
      return i >= M ? i - M : i;
    };
    const size_t o = ((size_t)inside(ix) * M + inside(iy)) * M + inside(iz);
    for (int d = 0; d < 3; ++d) box[d][t] = f[d * nr + o];
  }
  __syncthreads();
  for (int k = ck.k0 + tid; k < ck.k1; k += kBrickThreads) {
    const double4 q = part[k];
    double wx[3], wy[3], wz[3];
    const int gx = wrap(tsc(q.x, wx), M), gy = wrap(tsc(q.y, wy), M), gz = wrap(tsc(q.z, wz), M);
    const int first = ((gx - 1 - ox) * kBox + gy - 1 - oy) * kBox + gz - 1 - oz;
    double ax = 0.0, ay = 0.0, az = 0.0;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        const double wab = wx[a] * wy[b];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const int o = first + (a * kBox + b) * kBox + c;
          const double w = wab * wz[c];
          ax += w * box[0][o];
          ay += w * box[1][o];
          az += w * box[2][o];
        }
      }
    const size_t p = (size_t)order[k];
    acc[3 * p] = ax;
    acc[3 * p + 1] = ay;
    acc[3 * p + 2] = az;
  }
}

// The same from memory, for few particles per brick.
__global__ __launch_bounds__(256) void pm_interp_direct(int n, const double* __restrict__ pos,
                                                        int M, const double* __restrict__ f,
                                                        double* __restrict__ acc) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  const size_t nr = (size_t)M * M * M;
  double wx[3], wy[3], wz[3];
  const int gx = tsc(mesh_units(pos[3 * (size_t)p], M), wx);
  const int gy = tsc(mesh_units(pos[3 * (size_t)p + 1], M), wy);
  const int gz = tsc(mesh_units(pos[3 * (size_t)p + 2], M), wz);
  double ax = 0.0, ay = 0.0, az = 0.0;
  for (int a = 0; a < 3; ++a) {
    const size_t ix = (size_t)wrap(gx + a - 1, M) * M;
    for (int b = 0; b < 3; ++b) {
      const size_t iy = (ix + wrap(gy + b - 1, M)) * M;
      const double wab = wx[a] * wy[b];
      for (int c = 0; c < 3; ++c) {
        const size_t o = iy + wrap(gz + c - 1, M);
        const double w = wab * wz[c];
        ax += w * f[o];
        ay += w * f[nr + o];
        az += w * f[2 * nr + o];
      }
    }
  }
  acc[3 * (size_t)p] = ax;
  acc[3 * (size_t)p + 1] = ay;
  acc[3 * (size_t)p + 2] = az;
}

}  // namespace pm
