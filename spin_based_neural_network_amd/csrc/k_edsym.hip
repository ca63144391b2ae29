// k_edsym.hip — Lanczos inside one symmetry sector, and the drivers' start
// vector (src/mps/lanczos.c:160-176, 824-1130; projector
// src/nqs/nqs_symproj.c:786-851).
//
// Where the permutations form a group, the characters are +-1 and multiply
// with it, and the group maps the bond list onto itself, the projector P
// commutes with H and every vector of the projected recurrence satisfies
// v[T(g) s] = chi_g v[s].  Such a vector is one value per orbit of basis
// states; the recurrence runs on these and P, which the general drivers apply
// after every product, has nothing left to do.
//   reps   smallest state of each orbit, by its number of set bits, then ascending
//   code   per basis state: its orbit, bit 31 set where chi = -1; orbits that
//          P removes point at entry R of every vector, which is 0
//   ell    per orbit the codes of the states that H couples the representative
//          to, antiparallel bonds first to last, then flipped sites; used: the
//          most bonds of a wave's 64 orbits (the others' lists end in entry R)
// Sums over basis states are sums over orbits times the orbit's length.
//
// What bounds it: a product reads ell once (4 bytes a listed bond and orbit)
// and gathers one double for each; in the full basis it gathers as often from 2^N
// states, and the projector G times more.  Exchange bonds keep the number of
// set bits, so in this order a stretch of orbits gathers from a window of one
// magnetisation's orbits (24 sites, 8 operations: 2.7 MB at most, of 17);
// consecutive stretches go to one XCD, whose L2 holds its window.
//
// Measured (24 sites, 48 bonds, 8 operations, 60 steps): 145.5 ms in the full
// basis, 15.2 here (17.6 with the orbits in ascending order, 15.9 with the
// parallel bonds in the lists); a step's product and projection took 505 + 1177
// us; making the orbits and couplings 0.8 ms once; the start vector 35 ms on
// the host, 0.19 here.
#include "nqs_kernels.h"

namespace nqs {

namespace {

constexpr int kSymBlocks = 2048;     // fixed grid of the vector kernels
constexpr int kSeedRun = 32;         // start-vector elements a thread makes
constexpr long kStateBlock = 4096;   // states a workgroup of the orbit search takes

__device__ inline double sum256(double v, double* red) {
  const int tid = threadIdx.x;
  red[tid] = v;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w) red[tid] += red[tid + w];
    __syncthreads();
  }
  return red[0];
}

__device__ inline void stage(const EdSym& y, unsigned* tab) {
  const int n = y.G * (y.nc << y.bits);
  for (int e = threadIdx.x; e < n; e += 256) tab[e] = y.tab[e];
  __syncthreads();
}

// T(g) s from the tables of runs of y.bits bits
__device__ inline unsigned image(const EdSym& y, const unsigned* tab, int g, unsigned s) {
  const unsigned* t = tab + ((g * y.nc) << y.bits);
  unsigned r = 0;
  for (int c = 0; c < y.nc; c++)
    r |= t[(c << y.bits) + ((s >> (c * y.bits)) & ((1u << y.bits) - 1u))];
  return r;
}

// value of the state that code c names, in the vector v
__device__ inline double at(const double* __restrict__ v, unsigned c) {
  const double x = v[c & 0x7FFFFFFFu];
  return __hiloint2double(__double2hiint(x) ^ (int)(c & 0x80000000u), __double2loint(x));
}

// flags: one bit a state, set where no image is smaller; counts of them by
// number of set bits [32] per block.  A wave goes on to the next operation only
// while one of its states is left.
__global__ __launch_bounds__(256) void k_eds_flags(EdSym y, long dim, unsigned long long* flags,
                                                   unsigned* counts) {
  extern __shared__ unsigned tab[];
  __shared__ unsigned cnt[32];
  if (threadIdx.x < 32) cnt[threadIdx.x] = 0;
  stage(y, tab);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int i = 0; i < 16; i++) {
    const long s = blockIdx.x * kStateBlock + (wave * 16 + i) * 64 + lane;
    bool rep = s < dim;
    for (int g = 0; g < y.G && __ballot(rep); g++)
      if (rep && image(y, tab, g, (unsigned)s) < (unsigned)s) rep = false;
    const unsigned long long m = __ballot(rep);
    if (lane == 0) flags[blockIdx.x * 64L + wave * 16 + i] = m;
    if (rep) atomicAdd(&cnt[__popc((unsigned)s)], 1u);
  }
  __syncthreads();
  if (threadIdx.x < 32) counts[blockIdx.x * 32L + threadIdx.x] = cnt[threadIdx.x];
}

// reps from the flags; first [block][32]: where a block's states of each number
// of set bits go.  One wave a block, 64 states at a time.
__global__ __launch_bounds__(64) void k_eds_list(const unsigned long long* __restrict__ flags,
                                                 const unsigned* __restrict__ first,
                                                 unsigned* __restrict__ reps) {
  __shared__ unsigned next[32];
  const int lane = threadIdx.x;
  if (lane < 32) next[lane] = first[blockIdx.x * 32L + lane];
  __syncthreads();
  for (int w = 0; w < 64; w++) {
    const unsigned long long m = flags[blockIdx.x * 64L + w];
    const unsigned s = (unsigned)(blockIdx.x * kStateBlock + w * 64 + lane);
    const int base = __popc((unsigned)(s & ~63u)), p = __popc(s);
    for (int q = base; q <= base + 6; q++) {
      const unsigned long long same = __ballot(((m >> lane) & 1ULL) && p == q);
      if (!same) continue;
      const unsigned at = next[q & 31];
      if ((same >> lane) & 1ULL) reps[at + __popcll(same & ((1ULL << lane) - 1ULL))] = s;
      __syncthreads();
      if (lane == 0) next[q & 31] = at + __popcll(same);
      __syncthreads();
    }
  }
}

// the orbit of each representative: codes of its states, its length (0 where
// P removes it: an operation that fixes the state has chi = -1)
__global__ __launch_bounds__(256) void k_eds_orbit(EdSym y, const unsigned* __restrict__ reps, long R,
                                                   unsigned* __restrict__ code,
                                                   double* __restrict__ len) {
  extern __shared__ unsigned tab[];
  stage(y, tab);
  for (long r = blockIdx.x * 256L + threadIdx.x; r < R; r += (long)gridDim.x * 256) {
    const unsigned s = reps[r];
    int fix = 0;
    bool gone = false;
    for (int g = 0; g < y.G; g++)
      if (image(y, tab, g, s) == s) {
        fix++;
        if (y.chi[g] < 0.0) gone = true;
      }
    for (int g = 0; g < y.G; g++)
      code[image(y, tab, g, s)] =
          gone ? (unsigned)R : (unsigned)r | (y.chi[g] < 0.0 ? 0x80000000u : 0u);
    len[r] = gone ? 0.0 : (double)(y.G / fix);
  }
}

// x = (P v) at the representatives (the projector's own sum); partial |P v|^2
__global__ __launch_bounds__(256) void k_eds_restrict(EdSym y, const unsigned* __restrict__ reps,
                                                      long R, const double* __restrict__ v,
                                                      const double* __restrict__ len,
                                                      double* __restrict__ x,
                                                      double* __restrict__ part) {
  extern __shared__ unsigned tab[];
  __shared__ double red[256];
  stage(y, tab);
  const double invG = 1.0 / y.G;
  double acc2 = 0.0;
  for (long r = blockIdx.x * 256L + threadIdx.x; r < R; r += (long)gridDim.x * 256) {
    const unsigned s = reps[r];
    double acc = 0.0;
    for (int g = 0; g < y.G; g++) acc += y.chi[g] * v[image(y, tab, g, s)];
    const double z = len[r] > 0.0 ? acc * invG : 0.0;
    x[r] = z;
    acc2 += len[r] * z * z;
  }
  const double t = sum256(acc2, red);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
  if (blockIdx.x == 0 && threadIdx.x == 0) x[R] = 0.0;
}

// couplings and the diagonal of every representative
__global__ __launch_bounds__(256) void k_eds_ell(EdOp op, const unsigned* __restrict__ reps, long R,
                                                 const unsigned* __restrict__ code,
                                                 unsigned* __restrict__ ell, int* __restrict__ used,
                                                 double* __restrict__ diag) {
  for (long r0 = blockIdx.x * 256L; r0 < R; r0 += (long)gridDim.x * 256) {
    const long r = r0 + threadIdx.x;
    const bool in = r < R;
    const unsigned s = in ? reps[r] : 0u;
    double d = 0.0;
    int n = 0;
    for (int b = 0; b < op.nb; b++) {
      const int u = op.bonds[2 * b], v = op.bonds[2 * b + 1];
      const bool anti = ((s >> u) ^ (s >> v)) & 1u;
      d += anti ? -op.jd : op.jd;
      if (in && anti && op.jo != 0.0) ell[(long)n++ * R + r] = code[s ^ ((1u << u) | (1u << v))];
    }
    int most = n;
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) most = max(most, __shfl_xor(most, m, 64));
    if ((threadIdx.x & 63) == 0) used[r >> 6] = most;
    if (!in) continue;
    for (; n < most; n++) ell[(long)n * R + r] = (unsigned)R;
    diag[r] = d;
    if (op.field != 0.0) {
      unsigned* e = ell + (op.jo != 0.0 ? op.nb : 0) * R + r;
      for (int i = 0; i < op.N; i++, e += R) *e = code[s ^ (1u << i)];
    }
  }
}

// out = H in; partial <in, out>
__global__ __launch_bounds__(256) void k_eds_matvec(const double* __restrict__ in,
                                                    double* __restrict__ out, long R,
                                                    const unsigned* __restrict__ ell,
                                                    const int* __restrict__ used, int nb, double jo,
                                                    int nf, double field,
                                                    const double* __restrict__ diag,
                                                    const double* __restrict__ len,
                                                    double* __restrict__ part) {
  __shared__ double red[256];
  double dot = 0.0;
  // tiles of 256 orbits: an eighth of them, in order, to the blocks of each XCD
  const long T = (R + 255) / 256;
  const int xcds = gridDim.x >= 8 ? 8 : 1, x0 = blockIdx.x % xcds;
  const long end = T * (x0 + 1) / xcds;
  for (long t = T * x0 / xcds + blockIdx.x / xcds; t < end; t += (gridDim.x - x0 + xcds - 1) / xcds) {
    const long r = t * 256 + threadIdx.x;
    if (r >= R) break;
    double off = 0.0;
    auto couple = [&](const unsigned* e, int n, double h) {
      for (int b = 0; b < n; b += 8) {
        unsigned c[8];
        double v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) c[j] = b + j < n ? e[(long)(b + j) * R] : (unsigned)R;
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = at(in, c[j]);
#pragma unroll
        for (int j = 0; j < 8; j++) off += h * v[j];
      }
    };
    if (nb) couple(ell + r, __builtin_amdgcn_readfirstlane(used[r >> 6]), jo);
    if (nf) couple(ell + nb * R + r, nf, field);
    const double x = in[r], z = diag[r] * x + off;
    out[r] = z;
    dot += len[r] * x * z;
  }
  const double t = sum256(dot, red);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
  if (blockIdx.x == 0 && threadIdx.x == 0) out[R] = 0.0;
}

// w -= a[0] v + b u (u may be null); partial |w|^2.  Orbits that P removes
// (length 0) stay 0.
__global__ __launch_bounds__(256) void k_eds_axpy2(double* __restrict__ w, const double* __restrict__ v,
                                                   const double* __restrict__ a,
                                                   const double* __restrict__ u, double b, long R,
                                                   const double* __restrict__ len,
                                                   double* __restrict__ part) {
  __shared__ double red[256];
  const double al = a[0];
  double acc = 0.0;
  for (long r = blockIdx.x * 256L + threadIdx.x; r < R; r += (long)gridDim.x * 256) {
    double x = w[r] - al * v[r];
    if (u) x -= b * u[r];
    const double n = len[r];
    if (n == 0.0) x = 0.0;
    w[r] = x;
    acc += n * x * x;
  }
  const double t = sum256(acc, red);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// y = x / sqrt(n2[0]), n2 read where it was left
__global__ __launch_bounds__(256) void k_eds_unit(const double* __restrict__ x, double* __restrict__ y,
                                                  const double* __restrict__ n2, long R) {
  const double c = 1.0 / sqrt(n2[0]);
  for (long r = blockIdx.x * 256L + threadIdx.x; r < R; r += (long)gridDim.x * 256) y[r] = x[r] * c;
  if (blockIdx.x == 0 && threadIdx.x == 0) y[R] = 0.0;
}

__global__ __launch_bounds__(256) void k_eds_sum(const double* __restrict__ part, int n,
                                                 double* __restrict__ out) {
  __shared__ double red[256];
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) acc += part[i];
  const double t = sum256(acc, red);
  if (threadIdx.x == 0) out[0] = t;
}

__global__ void k_eds_expand(const unsigned* __restrict__ code, const double* __restrict__ v, long dim,
                             double c, double* __restrict__ out) {
  for (long s = blockIdx.x * 256L + threadIdx.x; s < dim; s += (long)gridDim.x * 256)
    out[s] = c * at(v, code[s]);
}

// Start vector: xorshift64 is linear over GF(2), so a thread multiplies the
// seed by the power of its step's matrix that its run starts at (jump[k]: the
// columns of the 2^k-th power) and makes kSeedRun elements one by one.
__global__ __launch_bounds__(256) void k_ed_seed(unsigned long long x0,
                                                 const unsigned long long* __restrict__ jump, int nj,
                                                 long dim, double* __restrict__ v) {
  __shared__ unsigned long long col[32 * 64];
  __shared__ double run[256 * (kSeedRun + 1)];
  for (int e = threadIdx.x; e < nj * 64; e += 256) col[e] = jump[e];
  __syncthreads();
  const long b0 = blockIdx.x * (256L * kSeedRun);
  const unsigned long long s0 = (unsigned long long)b0 + threadIdx.x * kSeedRun;
  unsigned long long x = x0;
  for (int k = 0; k < nj; k++) {
    if (!((s0 >> k) & 1ULL)) continue;
    unsigned long long z = 0;
    for (int i = 0; i < 64; i++) z ^= col[k * 64 + i] & (0ULL - ((x >> i) & 1ULL));
    x = z;
  }
  for (int i = 0; i < kSeedRun; i++) {
    x ^= x << 13;
    x ^= x >> 7;
    x ^= x << 17;
    run[threadIdx.x * (kSeedRun + 1) + i] = (double)(x >> 11) / 9007199254740992.0 - 0.5;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 256 * kSeedRun; e += 256)
    if (b0 + e < dim) v[b0 + e] = run[(e / kSeedRun) * (kSeedRun + 1) + e % kSeedRun];
}

int blocks_of(long n) {
  const long g = (n + 255) / 256;
  return (int)(g < kSymBlocks ? (g > 0 ? g : 1) : kSymBlocks);
}
size_t tab_bytes(const EdSym& y) { return sizeof(unsigned) * (size_t)y.G * (y.nc << y.bits); }

}  // namespace

long ed_state_blocks(long dim) { return (dim + kStateBlock - 1) / kStateBlock; }

int launch_eds_flags(const EdSym& y, long dim, unsigned long long* flags, unsigned* counts,
                     hipStream_t st) {
  KScope ks("ed_orbits", st);
  hipLaunchKernelGGL(k_eds_flags, dim3((unsigned)ed_state_blocks(dim)), dim3(256), tab_bytes(y), st, y,
                     dim, flags, counts);
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

int launch_eds_orbits(const EdSym& y, long dim, const unsigned long long* flags, const unsigned* first,
                      unsigned* reps, long R, unsigned* code, double* len, hipStream_t st) {
  KScope ks("ed_orbits", st);
  hipLaunchKernelGGL(k_eds_list, dim3((unsigned)ed_state_blocks(dim)), dim3(64), 0, st, flags, first,
                     reps);
  hipLaunchKernelGGL(k_eds_orbit, dim3(blocks_of(R)), dim3(256), tab_bytes(y), st, y, reps, R, code, len);
  count_launch(2);
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

int launch_eds_couplings(const EdOp& op, const unsigned* reps, long R, const unsigned* code,
                         unsigned* ell, int* used, double* diag, hipStream_t st) {
  KScope ks("ed_orbits", st);
  hipLaunchKernelGGL(k_eds_ell, dim3(blocks_of(R)), dim3(256), 0, st, op, reps, R, code, ell, used,
                     diag);
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

int launch_eds_restrict(const EdSym& y, const unsigned* reps, long R, const double* v, const double* len,
                        double* x, double* part, double* norm2, hipStream_t st) {
  const int g = blocks_of(R);
  KScope ks("ed_project", st);
  hipLaunchKernelGGL(k_eds_restrict, dim3(g), dim3(256), tab_bytes(y), st, y, reps, R, v, len, x, part);
  hipLaunchKernelGGL(k_eds_sum, dim3(1), dim3(256), 0, st, part, g, norm2);
  count_launch();
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

int launch_eds_matvec(const EdOp& op, const double* in, double* out, long R, const unsigned* ell,
                      const int* used, const double* diag, const double* len, double* part, double* dot, hipStream_t st) {
  const int g = blocks_of(R);
  KScope ks("ed_matvec", st);
  hipLaunchKernelGGL(k_eds_matvec, dim3(g), dim3(256), 0, st, in, out, R, ell, used, op.jo != 0.0 ? op.nb : 0,
                     op.jo, op.field != 0.0 ? op.N : 0, op.field, diag, len, part);
  hipLaunchKernelGGL(k_eds_sum, dim3(1), dim3(256), 0, st, part, g, dot);
  count_launch();
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

int launch_eds_axpy2(double* w, const double* v, const double* a, const double* u, double b, long R,
                     const double* len, double* part, double* norm2, hipStream_t st) {
  const int g = blocks_of(R);
  hipLaunchKernelGGL(k_eds_axpy2, dim3(g), dim3(256), 0, st, w, v, a, u, b, R, len, part);
  hipLaunchKernelGGL(k_eds_sum, dim3(1), dim3(256), 0, st, part, g, norm2);
  count_launch();
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

int launch_eds_unit(const double* x, double* y, const double* n2, long R, hipStream_t st) {
  hipLaunchKernelGGL(k_eds_unit, dim3(blocks_of(R)), dim3(256), 0, st, x, y, n2, R);
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

int launch_eds_expand(const unsigned* code, const double* v, long dim, double c, double* out,
                      hipStream_t st) {
  hipLaunchKernelGGL(k_eds_expand, dim3(blocks_of(dim)), dim3(256), 0, st, code, v, dim, c, out);
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

int launch_ed_seed(unsigned long long x0, const unsigned long long* jump, int nj, long dim, double* v,
                   hipStream_t st) {
  const long per = 256L * kSeedRun;
  hipLaunchKernelGGL(k_ed_seed, dim3((unsigned)((dim + per - 1) / per)), dim3(256), 0, st, x0, jump, nj,
                     dim, v);
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace nqs
