// k_multi.hip — many independent real-RBM CG-SR problems stepped together.
//
// Reference semantics per problem: nqs_sr_step_custom_full with the ansatz's
// own gradient (src/nqs/nqs_optimizer.c:141-241): F_k = <O_k E> - <O_k> <E>,
// CG on (S + eps I) delta = F with S v = O^T (O v) / Ns - <O> mean(O v)
// (qgt_apply, :44-80) and cg_solve's stopping rules (:84-139), then
// theta -= lr delta.
//
// The O matrix is never formed: in the padded (M+1) x (N+1) parameter layout
// an O row is [t_b, 1] (x) [s_b, 1], so
//   (O v)_b     = sum_h [t_b, 1]_h (V [s_b, 1]^T)_h       (Z = V S1^T, row weights u)
//   (O^T w)_hi  = sum_b w_b [t_b, 1]_h [s_b, 1]_i         (G = (T1 w)^T S1)
// on FP64 MFMA, and the last entry of O^T w is sum_b w_b, the mean that the
// QGT needs.  A spin operand is made in registers from its bit.
//
// A CG iteration of a problem is five phases, and the workgroups of the
// problem meet after each:
//   Z     u = O p, split over samples, and over 64-row tiles of p where the
//         workgroups outnumber the 16-sample tiles
//   G     O^T u, split over tiles of 16 hidden units; in a workgroup the waves
//         take slots of the samples (nsplit, in order) and sum them in LDS
//   A p   and partial p.Ap, split over 256-element slices
//   x, r  alpha; x, r, partial r.r
//   p     beta or stop; p
// k_mb_cg runs every iteration of every problem in one cooperative launch, a
// workgroup per CU, each problem on workgroups of its own that meet at a
// counter of its own.  What crosses workgroups (p, u, O^T u, partial sums)
// goes through relaxed agent-scope atomics, past the L2s that the XCDs do not
// share, so no cache is flushed at a meeting: 1.7 us for 8 or 32 workgroups,
// 4.9 us for 256, where a kernel boundary costs about 7 us.  The vectors stay
// in registers; a small problem (own) has them whole in every workgroup and
// meets twice an iteration.  k_mb_phase runs one phase as a launch, with the
// same functions: the same bits.
//
// Measured: 32 chains of 16 to 128 sites, 2048 samples each, 240 us an
// iteration as five launches on 64 x 64 tiles, 110 here (35 us of MFMA time;
// the rest mostly the latency of t, which 32 problems do not leave in the
// L2s); one of 16 sites, 1024 samples: 38 us, now 20.
//
// Every sum has a fixed order that depends on the problem and nsplit alone:
// row weights over hidden units by tiles of 64 rows, in each tile eight
// chains of eight; G over a slot's samples in one fused chain; slots in order;
// vector sums by 256 elements and then 256 strided partials.
#include "nqs_kernels.h"

#include <vector>

namespace nqs {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int CT = 512;              // threads of the CG kernels
constexpr int CW = CT / 64;
constexpr int kZs = 512;             // samples of a workgroup in hand in Z
constexpr int kZb = 128;             // samples of a workgroup of the launch of Z, at most
constexpr int kTiles = 4;            // most site tiles of a wave in G
constexpr int kPairs = 4;            // pairs of slices of a workgroup in hand

enum { F_PREP = 0, F_Z, F_G, F_VEC, F_APPLY, F_CG };
enum { PH_G1 = 0, PH_GE, PH_F, PH_Z, PH_G, PH_AP, PH_XR, PH_P };

template <int FIELD>
__device__ inline int first_blk(const MultiProb& q) {
  return FIELD == F_PREP    ? q.blk_prep
       : FIELD == F_Z     ? q.blk_z
       : FIELD == F_G     ? q.blk_g
       : FIELD == F_VEC   ? q.blk_vec
       : FIELD == F_APPLY ? q.blk_apply
                          : q.blk_cg;
}

// problem owning block `blk` of a launch (largest q with first block <= blk)
template <int FIELD>
__device__ inline int find_prob(const MultiBatch& mb, int blk) {
  int lo = 0, hi = mb.n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (first_blk<FIELD>(mb.probs[mid]) <= blk) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// values that workgroups of one launch exchange
__device__ inline double ld_x(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_x(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// a b rounded: not fused with a sum that it enters
__device__ inline double mul_only(double a, double b) {
  double r = a * b;
  asm volatile("" : "+v"(r));
  return r;
}

// +1.0, or -1.0 where bit 0 of m is set
__device__ inline double spin_of(unsigned m) {
  return __hiloint2double((int)(0x3FF00000u | (m << 31)), 0);
}

// LDS of a workgroup: sums (in hand: also the problem's own p), partials,
// row weights of the samples in hand (finished, and of the tile of 64 rows in
// hand), their spin words; then the rows of p with partial row weights (Z), or
// the partial tiles and each wave's samples (G).
struct Lds {
  double *red, *part, *u, *cur, *v, *up, *tile, *wu;
  unsigned *bits, *wbits;
};
__device__ __host__ inline size_t lds_head(int nw) {
  return kPairs * CT + kMultiMaxPart + 2 * kZs + (size_t)kZs * nw / 2;
}
__device__ inline Lds carve(const MultiProb& q, int hct, double* base) {
  Lds l;
  l.red = base;
  l.part = l.red + kPairs * CT;
  l.u = l.part + kMultiMaxPart;
  l.cur = l.u + kZs;
  l.bits = (unsigned*)(l.cur + kZs);
  l.v = base + lds_head(q.nw);
  l.up = l.v + hct * 16 * q.si;
  l.tile = l.v;
  l.wu = l.tile + CW * kTiles * 256;
  l.wbits = (unsigned*)(l.wu + CW * 64);
  return l;
}

// index of this thread's wave, in a scalar register
__device__ inline int wave_of() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// KE steps (four sites) of two tiles of Z; m: the sample's sites, from lane's on
template <int KE>
__device__ __forceinline__ void row_steps(const double* pa, const double* pb, unsigned m, v4d& z0,
                                          v4d& z1) {
#pragma unroll
  for (int j = 0; j < KE; j++) {
    const double sp = spin_of(m >> (4 * j));
    z0 = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[4 * j], sp, z0, 0, 0, 0);
    z1 = __builtin_amdgcn_mfma_f64_16x16x4f64(pb[4 * j], sp, z1, 0, 0, 0);
  }
}

__device__ __host__ inline int tiles64(int M) { return (M + 64) / 64; }

// ---- Z: row weights u = O p of the samples of 16-sample tiles t0 .. t1 - 1, of
// share `part` of the 64-row tiles ------------------------------------------------
// own: p is l.red.  held: the samples' words are in l.bits from the call before.
// SHARED false: rw.parts is 1 (the code without the shares: 1 % of an iteration).
template <bool SHARED>
__device__ void cg_rows(const MultiProb& q, const Lds& l, const MultiRows& rw, int part, int t0, int t1,
                        bool own, bool held) {
  const int tid = threadIdx.x, wave = wave_of(), lane = tid & 63;
  const int lr = lane & 15, lk = lane >> 4;
  const int M = q.M, N1 = q.N + 1, M1 = M + 1, nw = q.nw, si = q.si;
  const int HT = (M1 + 15) >> 4, KK = (N1 + 3) >> 2;
  int c0 = 0, c1 = HT;   // 16-row tiles c0 .. c1 - 1
  if (SHARED) {
    c0 = tiles64(M) * part / rw.parts * 4;
    c1 = tiles64(M) * (part + 1) / rw.parts * 4;
    if (c1 > HT) c1 = HT;
  }
  const unsigned magic = 0xFFFFFFFFu / (unsigned)N1 + 1;   // f / N1 for f < 2^17
  const int end = t1 * 16 < q.B ? t1 * 16 : q.B;
  for (int g0 = t0 * 16; g0 < end; g0 += kZs) {
    const int ns = end - g0 < kZs ? end - g0 : kZs;
    if (!held) {
      __syncthreads();
      for (int e = tid; e < ns * nw; e += CT) l.bits[e] = q.bits[(long)g0 * nw + e];
    }
    for (int c = c0; c < c1; c += rw.hct) {
      const int nh = c1 - c < rw.hct ? c1 - c : rw.hct, pairs = (nh + 1) >> 1;
      __syncthreads();
      if (rw.hct < c1 - c0 || g0 == t0 * 16) {
        // rows past M and columns past N are zero
        const int r1 = M1 - c * 16 < pairs * 32 ? M1 - c * 16 : pairs * 32;
        for (int e = tid; e < r1 * (si - N1); e += CT) {
          const int h = e / (si - N1);
          l.v[h * si + N1 + e - h * (si - N1)] = 0.0;
        }
        for (int e = r1 * si + tid; e < pairs * 32 * si; e += CT) l.v[e] = 0.0;
        const int f0 = c * 16 * N1, nf = r1 * N1;
        for (int f = tid; f < nf; f += 16 * CT) {
          double x[16];
#pragma unroll
          for (int j = 0; j < 16; j++) {
            const int g = f + j * CT < nf ? f + j * CT : nf - 1;
            x[j] = own ? l.red[f0 + g] : ld_x(q.p + f0 + g);
          }
#pragma unroll
          for (int j = 0; j < 16; j++) {
            const int g = f + j * CT;
            if (g < nf) {
              const int h = __umulhi((unsigned)g, magic);
              l.v[h * si + g - h * N1] = x[j];
            }
          }
        }
      }
      for (int b0 = 0; b0 < ns; b0 += rw.zb) {
        const int nb = ns - b0 < rw.zb ? ns - b0 : rw.zb, nst = (nb + 15) >> 4;
        // an item: 32 rows x 16 samples, two tiles of Z = V S1^T (rows hidden
        // units), weighted by t in a chain of eight as they leave the
        // accumulators; the next item's t is under way meanwhile
        double t[8];
        auto fetch = [&](int it) {
          const int p = it / nst, s = (it - p * nst) * 16 + lr, sc = s < nb ? s : nb - 1;
          const double* __restrict__ tT = q.tT + g0 + b0 + sc;
          const int h0 = (c + 2 * p) * 16 + lk;
#pragma unroll
          for (int j = 0; j < 8; j++) {
            const int h = h0 + 4 * j;
            t[j] = tT[(long)(h < M ? h : M - 1) * q.B];
          }
        };
        if (wave < nst * pairs) fetch(wave);
        __syncthreads();
        for (int it = wave; it < nst * pairs; it += CW) {
          const int p = it / nst, s = (it - p * nst) * 16 + lr, sc = s < nb ? s : nb - 1;
          const unsigned* bw = l.bits + (b0 + sc) * nw;
          const int h0 = (c + 2 * p) * 16 + lk;
          double w[8];
#pragma unroll
          for (int j = 0; j < 8; j++) w[j] = h0 + 4 * j < M ? t[j] : h0 + 4 * j == M ? 1.0 : 0.0;
          if (it + CW < nst * pairs) fetch(it + CW);
          const double* va = l.v + (2 * p * 16 + lr) * si + lk;
          const double* vb = va + 16 * si;
          v4d z0 = {0.0, 0.0, 0.0, 0.0}, z1 = z0;
          for (int k8 = 0; k8 < KK >> 3; k8++)
            row_steps<8>(va + k8 * 32, vb + k8 * 32, bw[k8] >> lk, z0, z1);
          if (KK & 7) {
            const double *pa = va + (KK >> 3) * 32, *pb = vb + (KK >> 3) * 32;
            const unsigned m = bw[KK >> 3] >> lk;
            switch (KK & 7) {
              case 1: row_steps<1>(pa, pb, m, z0, z1); break;
              case 2: row_steps<2>(pa, pb, m, z0, z1); break;
              case 3: row_steps<3>(pa, pb, m, z0, z1); break;
              case 4: row_steps<4>(pa, pb, m, z0, z1); break;
              case 5: row_steps<5>(pa, pb, m, z0, z1); break;
              case 6: row_steps<6>(pa, pb, m, z0, z1); break;
              default: row_steps<7>(pa, pb, m, z0, z1);
            }
          }
          double x = 0.0;
#pragma unroll
          for (int r = 0; r < 4; r++) x = fma(z0[r], w[r], x);
#pragma unroll
          for (int r = 0; r < 4; r++) x = fma(z1[r], w[4 + r], x);
          l.up[(p * 4 + lk) * rw.zb + s] = x;
        }
        __syncthreads();
        // the eight chains of a tile of 64 rows (two pairs) in order, then the tiles
        if (tid < nb) {
          const int s = b0 + tid;
          double cur = l.cur[s], u = l.u[s];
          for (int p = 0; p < pairs; p++) {
            const int g = c / 2 + p;
            if (!(g & 1)) cur = 0.0;
#pragma unroll
            for (int k = 0; k < 4; k++) cur += l.up[(p * 4 + k) * rw.zb + tid];
            if ((g & 1) || 2 * g + 2 >= HT) {
              u = g < 2 ? cur : u + cur;
              if (SHARED && rw.parts > 1) st_x(q.u + (long)(g >> 1) * q.B + g0 + s, cur);
            }
          }
          l.cur[s] = cur;
          l.u[s] = u;
          if ((!SHARED || rw.parts == 1) && c + nh >= HT) st_x(q.u + g0 + s, u);
        }
      }
    }
  }
}

// ---- G: O^T w -------------------------------------------------------------------
// 16 samples of a wave's chain, from the first of y, wu and wbits: NT site
// tiles from tile tl on; y the t of the 16 hidden units as MFMA operands, the
// samples' weights and words (those of tiles tl ..) in LDS
template <int NT>
__device__ __forceinline__ void chain16(const double* y, const double* wu, const unsigned* wbits, int tl,
                                        v4d* acc) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int s = 4 * j + lk;
    const double a = y[j] * wu[s];
    const unsigned n0 = wbits[s], n1 = NT > 1 ? wbits[64 + s] : 0u, n2 = NT > 3 ? wbits[128 + s] : 0u;
    // tile tl + c sits in half (tl + c) & 1 of word (tl + c) / 2
#pragma unroll
    for (int c = 0; c < NT; c++) {
      const int o = (tl & 1) + c;
      const unsigned n = o < 2 ? n0 : o < 4 ? n1 : n2;
      acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, spin_of(n >> ((o & 1) * 16 + lr)), acc[c], 0, 0, 0);
    }
  }
}
// 64 samples, or the `left` of them that there are (up to 15 past it have no
// weight); x is refilled with the next samples' operands g0 .. of nA as it is used
template <int NT>
__device__ __forceinline__ void chain64(double* x, const double* wu, const unsigned* wbits, int tl,
                                        int left, v4d* acc, const double* __restrict__ nA, int g0,
                                        int B4) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (left > 16 * j) chain16<NT>(x + 4 * j, wu + 16 * j, wbits + 16 * j, tl, acc);
#pragma unroll
    for (int i = 4 * j; i < 4 * j + 4; i++) x[i] = nA[(long)(g0 + i < B4 ? g0 + i : B4 - 1) * 64];
  }
}

// Units u0, u0 + us, .. of O^T w into out.  A unit: 16 hidden units by q.nt
// site tiles for each of CW / ws groups of waves, the waves of a group on ws
// slots at a time.  A lane fetches its sample's weight and words for the wave;
// the next 64 samples (slot, unit) are under way while these are used.
// parts: of the row weights (SHARED false: 1)
template <bool SHARED>
__device__ void cg_tiles(const MultiProb& q, const Lds& l, int u0, int us, int units, int mode, int parts,
                         double* out) {
  const int tid = threadIdx.x, wave = wave_of(), lane = tid & 63;
  const int N1 = q.N + 1, M1 = q.M + 1, sts = (N1 + 15) >> 4, nw = q.nw;
  const int ws = q.nsplit < CW ? q.nsplit : CW, tg = CW / ws;
  const int ng = (sts + q.nt * tg - 1) / (q.nt * tg);
  const int sl = wave % ws, grp = wave / ws, B4 = (q.B + 15) / 16 * 4;
  double* wu = l.wu + wave * 64;
  unsigned* wbits = l.wbits + wave * 192;
  const int ne = q.nt * tg * 256;   // elements of a unit, at most kTiles * CT
  double x[16], u = 0.0;
  unsigned m0 = 0, m1 = 0, m2 = 0;
  auto first_tile = [&](int unit) { return (unit % ng * tg + grp) * q.nt; };
  auto operands = [&](int unit) { return q.tA + (long)(unit / ng) * B4 * 64 + lane; };
  auto fetch = [&](int unit, int k0, int sub) {
    const int b0 = (k0 + sl) * q.chunk + sub, end = (k0 + sl + 1) * q.chunk;
    const int b1 = end < q.B ? end : q.B;
    const int s = b0 + lane, sc = s < q.B ? s : q.B - 1;
    double w = mode == PH_G1 ? 1.0 : mode == PH_GE ? q.E[sc] : ld_x(q.u + sc);
    if (SHARED && mode == PH_G && parts > 1) {
      // the 64-row tiles in order, four under way
      const int T = tiles64(q.M);
      for (int k = 1; k < T; k += 4) {
        double y[4];
#pragma unroll
        for (int j = 0; j < 4; j++) y[j] = ld_x(q.u + (long)(k + j < T ? k + j : T - 1) * q.B + sc);
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (k + j < T) w += y[j];
      }
    }
    u = s < b1 ? w : 0.0;
    const int w0 = first_tile(unit) >> 1;
    const unsigned* bw = q.bits + (long)sc * nw;
    m0 = bw[w0 < nw ? w0 : nw - 1];
    m1 = q.nt > 1 ? bw[w0 + 1 < nw ? w0 + 1 : nw - 1] : 0u;
    m2 = q.nt > 3 ? bw[w0 + 2 < nw ? w0 + 2 : nw - 1] : 0u;
  };
  if (u0 >= units) return;
  fetch(u0, 0, 0);
  {
    const double* __restrict__ tA = operands(u0);
    const int g0 = sl * q.chunk / 4;
#pragma unroll
    for (int j = 0; j < 16; j++) x[j] = tA[(long)(g0 + j < B4 ? g0 + j : B4 - 1) * 64];
  }
  for (int unit = u0; unit < units; unit += us) {
    const int tl = first_tile(unit), nt = sts - tl < q.nt ? sts - tl : q.nt;
    double sum[kTiles] = {0.0, 0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < q.nsplit; k0 += ws) {
      v4d acc[kTiles];
#pragma unroll
      for (int c = 0; c < kTiles; c++) acc[c] = (v4d){0.0, 0.0, 0.0, 0.0};
      for (int sub = 0; sub < q.chunk; sub += 64) {
        wu[lane] = u;
        wbits[lane] = m0;
        wbits[64 + lane] = m1;
        wbits[128 + lane] = m2;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int s0 = (k0 + sl) * q.chunk + sub;
        const int left = q.chunk - sub < q.B - s0 ? q.chunk - sub : q.B - s0;
        // the next samples of this slot, of the next slots, of the next unit
        int nu = unit, nk = k0, nsub = sub + 64;
        if (nsub >= q.chunk) {
          nsub = 0;
          nk += ws;
          if (nk >= q.nsplit) {
            nk = 0;
            nu = unit + us < units ? unit + us : unit;
          }
        }
        fetch(nu, nk, nsub);
        const double* __restrict__ nA = operands(nu);
        const int g0 = ((nk + sl) * q.chunk + nsub) / 4;
        if (nt >= 4) chain64<4>(x, wu, wbits, tl, left, acc, nA, g0, B4);
        else if (nt == 3) chain64<3>(x, wu, wbits, tl, left, acc, nA, g0, B4);
        else if (nt == 2) chain64<2>(x, wu, wbits, tl, left, acc, nA, g0, B4);
        else if (nt == 1) chain64<1>(x, wu, wbits, tl, left, acc, nA, g0, B4);
        else chain64<0>(x, wu, wbits, tl, left, acc, nA, g0, B4);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
      __syncthreads();
#pragma unroll
      for (int c = 0; c < kTiles; c++)
        if (c < q.nt) {
          double* d = l.tile + ((grp * q.nt + c) * ws + sl) * 256 + lane;
#pragma unroll
          for (int r = 0; r < 4; r++) d[r * 64] = acc[c][r];
        }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kTiles; i++) {
        const int e = i * CT + tid;
        if (e < ne) {
          const double* d = l.tile + (e >> 8) * ws * 256 + (e & 255);
          if (ws == CW) {
            double v[CW];
#pragma unroll
            for (int k = 0; k < CW; k++) v[k] = d[k * 256];
#pragma unroll
            for (int k = 0; k < CW; k++) sum[i] += v[k];
          } else {
            for (int k = 0; k < ws; k++) sum[i] += d[k * 256];
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kTiles; i++) {
      const int e = i * CT + tid;
      if (e < ne) {
        const int site = (unit % ng * q.nt * tg + (e >> 8)) * 16 + (e & 15);
        const int h = unit / ng * 16 + ((e & 255) >> 4);
        if (site < N1 && h < M1) st_x(out + (long)h * N1 + site, sum[i]);
      }
    }
  }
}
__device__ __host__ inline int tile_units(const MultiProb& q, int nt) {
  const int HT = (q.M + 16) >> 4, sts = (q.N + 16) >> 4;
  const int per = nt * (CW / (q.nsplit < CW ? q.nsplit : CW));
  return HT * ((sts + per - 1) / per);
}

// ---- the vectors -----------------------------------------------------------------
// Elements by 256-element slices, two (a pair) to a workgroup's 512 threads;
// kPairs pairs j0, j0 + js, .. are in hand at a time.
struct Elem {
  double x, r, p, ap, om;
};
struct Pairs {
  int j0, js;
  __device__ int pair(int i) const { return j0 + i * js; }
  __device__ long at(int i) const { return (long)pair(i) * CT + threadIdx.x; }
};
__device__ inline long vec_len(const MultiProb& q) { return (long)(q.M + 1) * (q.N + 1); }

// Partial sums of v over the slices in hand, each by halves (128 apart, 64,
// .. 1), into part (shared: exchanged)
__device__ inline void put_parts(const MultiProb& q, const Pairs& w, const double* v, double* part,
                                 bool shared, double* red) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPairs; i++) red[i * CT + tid] = v[i];
  __syncthreads();
  const double* d = red + wave * 256 + lane;
  double s = (d[0] + d[128]) + (d[64] + d[192]);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
  const int sl = 2 * w.pair(wave >> 1) + (wave & 1);
  if (lane == 0 && sl < q.nvec) {
    if (shared) st_x(part + sl, s);
    else part[sl] = s;
  }
}
static_assert(2 * kPairs == CW, "a slice for each wave");

// their sum to every thread: 256 strided sums, then by halves
__device__ inline double total(const MultiProb& q, const double* part, bool shared, double* red) {
  const int tid = threadIdx.x, lane = tid & 63;
  double v = 0.0;
  if (tid < 256)
    for (int i = tid; i < q.nvec; i += 256) v += shared ? ld_x(part + i) : part[i];
  __syncthreads();
  if (tid < 256) red[tid] = v;
  __syncthreads();
  double s = (red[lane] + red[lane + 128]) + (red[lane + 64] + red[lane + 192]);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
  return s;
}

// Ap = (O^T u)/B - Om mean(u) + eps p, partial p.Ap (nqs_optimizer.c:103-106)
__device__ inline void pairs_ap(const MultiProb& q, const Pairs& w, Elem* st, double* part, bool shared,
                                double* red) {
  const long L = vec_len(q);
  const double inv = 1.0 / (double)q.B, gu = ld_x(q.g + L - 1);
  double g[kPairs], pa[kPairs];
#pragma unroll
  for (int i = 0; i < kPairs; i++) g[i] = ld_x(q.g + (w.at(i) < L ? w.at(i) : L - 1));
  const double mu = mul_only(gu, inv);
#pragma unroll
  for (int i = 0; i < kPairs; i++) {
    const double ap = fma(q.eps, st[i].p, fma(g[i], inv, -mul_only(st[i].om, mu)));
    st[i].ap = w.at(i) < L - 1 ? ap : 0.0;
    pa[i] = w.at(i) < L ? st[i].p * st[i].ap : 0.0;
  }
  put_parts(q, w, pa, part, shared, red);
}

// x += alpha p, r -= alpha Ap, partial r.r (nqs_optimizer.c:113-120)
__device__ inline void pairs_xr(const MultiProb& q, const Pairs& w, Elem* st, double a, double* part,
                                bool shared, double* red) {
  double rr[kPairs];
#pragma unroll
  for (int i = 0; i < kPairs; i++) {
    st[i].x = fma(a, st[i].p, st[i].x);
    st[i].r = fma(-a, st[i].ap, st[i].r);
    rr[i] = w.at(i) < vec_len(q) ? st[i].r * st[i].r : 0.0;
  }
  put_parts(q, w, rr, part, shared, red);
}

__device__ inline void load_pairs(const MultiProb& q, const Pairs& w, Elem* st) {
  const long L = vec_len(q);
#pragma unroll
  for (int i = 0; i < kPairs; i++) {
    const long e = w.at(i) < L ? w.at(i) : L - 1;   // the last element is zero
    st[i] = Elem{q.x[e], q.r[e], ld_x(q.p + e), q.Ap[e], q.Om[e]};
    if (w.at(i) >= L) st[i].om = 0.0;
  }
}

// |r|^2 before iteration it, of the launch sequence's partials
__device__ inline double* part_rr(const MultiProb& q, int it) {
  return q.part + (it < 0 ? 0 : 2 + (it & 1)) * (long)kMultiMaxPart;
}
__device__ inline bool broke(double pAp) { return !(fabs(pAp) >= 1e-30); }

// ---------------------------------------------------------------------------
// spin words [B][nw] (bit set: s = -1); t by hidden unit for Z (tT [M][B]) and,
// with the unit column and zeros to whole tiles, as the A operand of G (tA:
// tile of 16 hidden units, four samples, lane): 64 samples a workgroup
__global__ __launch_bounds__(256) void k_mb_prep(MultiBatch mb) {
  __shared__ double tile[64][33];
  const MultiProb& q = mb.probs[find_prob<F_PREP>(mb, blockIdx.x)];
  const long b0 = (blockIdx.x - q.blk_prep) * 64L;
  const int nb = (int)(q.B - b0 < 64 ? q.B - b0 : 64);
  for (int e = threadIdx.x; e < nb * q.nw; e += 256) {
    const int b = e / q.nw, w = e - b * q.nw;
    const int* s = q.spins + (b0 + b) * q.N;
    unsigned m = 0;
    for (int i = w * 32; i < q.N && i < w * 32 + 32; i++)
      if (s[i] < 0) m |= 1u << (i & 31);
    q.bits[b0 * q.nw + e] = m;
  }
  const int B4 = (q.B + 15) / 16 * 4, j1 = B4 - b0 / 4 < 16 ? B4 - (int)(b0 / 4) : 16;
  for (int e = threadIdx.x; e < (q.M + 16) / 16 * j1 * 64; e += 256) {
    const int lr = e & 15, lk = (e >> 4) & 3, ht = (e >> 6) / j1, j = (e >> 6) - ht * j1;
    const int h = ht * 16 + lr, b = 4 * j + lk;
    const double t = b >= nb || h > q.M ? 0.0 : h == q.M ? 1.0 : q.t[(b0 + b) * q.M + h];
    q.tA[((long)ht * B4 + b0 / 4 + j) * 64 + (e & 63)] = t;
  }
  for (int h0 = 0; h0 < q.M; h0 += 32) {
    __syncthreads();
    for (int e = threadIdx.x; e < 64 * 32; e += 256) {
      const int b = e >> 5, h = h0 + (e & 31);
      if (b < nb && h < q.M) tile[b][e & 31] = q.t[(b0 + b) * q.M + h];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 64 * 32; e += 256) {
      const int h = h0 + (e >> 6), b = e & 63;
      if (b < nb && h < q.M) q.tT[(long)h * q.B + b0 + b] = tile[b][e >> 6];
    }
  }
}

// One phase of every problem as a launch of its own (iteration `it` of the CG
// phases).  A problem's scalars are written by its first block in PH_P; a
// block of that launch that reads `done` after the write has nothing left to do.
__global__ __launch_bounds__(CT) void k_mb_phase(MultiBatch mb, int phase, int it) {
  extern __shared__ double lds[];
  __shared__ int done;   // read once: the whole workgroup takes one branch
  const int blk = blockIdx.x;
  const MultiProb& q = mb.probs[phase == PH_Z ? find_prob<F_Z>(mb, blk)
                                : phase <= PH_GE || phase == PH_G ? find_prob<F_G>(mb, blk)
                                                                  : find_prob<F_VEC>(mb, blk)];
  const Lds l = carve(q, q.solo.hct, lds);
  if (phase <= PH_GE) {
    cg_tiles<false>(q, l, blk - q.blk_g, 1, blk - q.blk_g + 1, phase, 1, phase == PH_G1 ? q.g : q.Ap);
    return;
  }
  const long L = vec_len(q);
  const Pairs w{blk - q.blk_vec, (((q.nvec + 1) >> 1) + kPairs - 1) / kPairs};
  double* red = l.red;
  if (phase == PH_F) {
    // Om = (O^T 1)/B, F = (O^T E)/B - Om <E>; CG start x = 0, r = p = F
    // (cg_solve, nqs_optimizer.c:84-95)
    double ff[kPairs];
#pragma unroll
    for (int i = 0; i < kPairs; i++) {
      const long e = w.at(i);
      ff[i] = 0.0;
      if (e < L) {
        const double inv = 1.0 / (double)q.B;
        const double om = mul_only(q.g[e], inv);
        const double f = e == L - 1 ? 0.0 : fma(q.Ap[e], inv, -mul_only(om, q.stats[0]));
        q.Om[e] = om;
        q.x[e] = 0.0;
        q.r[e] = f;
        q.p[e] = f;
        ff[i] = f * f;
      }
    }
    put_parts(q, w, ff, part_rr(q, -1), true, red);
    if (w.j0 == 0 && threadIdx.x == 0) {
      q.sc->iters = 0;
      q.sc->converged = 0;
      q.sc->breakdown = 0;
      q.sc->done = q.max_it <= 0 ? 1 : 0;
    }
    return;
  }
  if (threadIdx.x == 0) done = q.sc->done;
  __syncthreads();
  if (done) return;
  if (phase == PH_Z) {
    const MultiRows& rw = q.solo;
    const int at = (blk - q.blk_z) / rw.parts, nT = (q.B + 15) / 16, per = rw.samples / 16;
    cg_rows<true>(q, l, rw, blk - q.blk_z - at * rw.parts, at * per, at * per + per < nT ? at * per + per : nT,
            false, false);
    return;
  }
  if (phase == PH_G) {
    cg_tiles<true>(q, l, blk - q.blk_g, 1, blk - q.blk_g + 1, PH_G, q.solo.parts, q.g);
    return;
  }
  Elem st[kPairs];
  load_pairs(q, w, st);
  double* part_pap = q.part + kMultiMaxPart;
  if (phase == PH_AP) {
    pairs_ap(q, w, st, part_pap, true, red);
#pragma unroll
    for (int i = 0; i < kPairs; i++)
      if (w.at(i) < L) q.Ap[w.at(i)] = st[i].ap;
    return;
  }
  const double pAp = total(q, part_pap, true, red), rs = total(q, part_rr(q, it - 1), true, red);
  if (phase == PH_XR) {
    if (broke(pAp)) return;
    pairs_xr(q, w, st, rs / pAp, part_rr(q, it), true, red);
#pragma unroll
    for (int i = 0; i < kPairs; i++)
      if (w.at(i) < L) {
        q.x[w.at(i)] = st[i].x;
        q.r[w.at(i)] = st[i].r;
      }
    return;
  }
  const double rs0 = total(q, part_rr(q, -1), true, red);
  const double rn = broke(pAp) ? rs : total(q, part_rr(q, it), true, red);
  const bool conv = !broke(pAp) && rn <= q.tol * q.tol * rs0;
  if (!broke(pAp) && !conv) {
    const double be = rn / rs;
#pragma unroll
    for (int i = 0; i < kPairs; i++)
      if (w.at(i) < L) q.p[w.at(i)] = fma(be, st[i].p, st[i].r);
  }
  if (w.j0 == 0 && threadIdx.x == 0) {
    CGScalars* sc = q.sc;
    sc->rs0 = rs0;
    sc->pAp = pAp;
    sc->rs_new = rn;
    sc->rs = rn;
    if (broke(pAp)) sc->breakdown = 1;
    else sc->iters = it + 1;
    if (conv) sc->converged = 1;
    if (broke(pAp) || conv || it + 1 >= q.max_it) sc->done = 1;
  }
}

// The problem's nb workgroups meet: every thread's exchanged stores have
// reached the agent's coherence point (the wait), then one arrival; `n` counts
// the meetings.  False when the others do not arrive within `polls` looks
// (seconds): the kernel then ends.
__device__ inline bool meet(const MultiProb& q, unsigned& n, int polls) {
  __shared__ int ok;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (q.nb == 1) return true;
  n++;
  if (threadIdx.x == 0) {
    const unsigned want = n * (unsigned)q.nb;
    __hip_atomic_fetch_add(q.bar, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    int got = 0;
    for (int i = 0; i < polls; i++) {
      if ((int)(__hip_atomic_load(q.bar, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - want) >= 0) {
        got = 1;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    ok = got;
  }
  __syncthreads();
  return ok != 0;
}

// Up to `iters` CG iterations of every problem (matvec_only: O^T O p once,
// which changes nothing that the CG start has set).  Consecutive workgroups of
// a problem sit on one XCD (block b runs on XCD b % 8), where its t stays in
// that XCD's L2.
// SHARED: a problem of the batch has its rows of p in shares.
template <bool SHARED>
__global__ __launch_bounds__(CT) void k_mb_cg(MultiBatch mb, int iters, int matvec_only) {
  extern __shared__ double lds[];
  const int lb = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (lb >= mb.nblk_cg) return;
  const MultiProb& q = mb.probs[find_prob<F_CG>(mb, lb)];
  if (q.max_it <= 0) return;   // nothing to do, and no meeting to pass
  const MultiRows& rw = q.coop;
  const Lds l = carve(q, rw.hct, lds);
  double* red = l.red;
  const int b = lb - q.blk_cg, nb = q.nb, J = (q.nvec + 1) >> 1, tid = threadIdx.x;
  // row weights: share b % parts of the rows of p for the samples of share
  // b / parts (the last workgroups may have neither)
  const int nT = (q.B + 15) / 16, parts = SHARED ? rw.parts : 1, shares = nb / parts, at = b / parts;
  const int t0 = at < shares ? (int)((long)nT * at / shares) : nT;
  const int t1 = at < shares ? (int)((long)nT * (at + 1) / shares) : nT;
  const int units = tile_units(q, q.nt);
  const long L = vec_len(q);
  // every workgroup has the whole vectors, or every js-th pair of slices; in
  // registers (one group) or, past kPairs pairs, in memory
  const bool own = nb > 1 && J <= kPairs, local = own || nb == 1;
  const int j0 = own ? 0 : b, js = own ? 1 : nb;
  const int groups = ((J - j0 + js - 1) / js + kPairs - 1) / kPairs;
  const bool kept = groups <= 1;
  double* pp = local ? l.part : q.part + kMultiMaxPart;
  double* pr = local ? l.part : q.part + 2 * kMultiMaxPart;
  Elem st[kPairs];
  Pairs w{j0, js};
  if (kept) load_pairs(q, w, st);
  unsigned n = 0;
  bool live = true, conv = false, brk = false;
  int it = 0;
  double rs = total(q, q.part, true, red), rs0 = rs, rn = rs, pAp = 0.0;
  if (own) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPairs; i++) red[i * CT + tid] = st[i].p;
  }
  // what only this workgroup has is its own threads' business
  auto pause = [&]() -> bool {
    if (local) {
      __syncthreads();
      return true;
    }
    return meet(q, n, mb.polls);
  };
  const int cap = matvec_only ? 1 : iters < q.max_it ? iters : q.max_it;
  while (it < cap) {
    cg_rows<SHARED>(q, l, rw, b % parts, t0, t1, own, it > 0 && (t1 - t0) * 16 <= kZs);
    if (!(live = meet(q, n, mb.polls))) break;
    cg_tiles<SHARED>(q, l, b, nb, units, PH_G, parts, q.g);
    if (matvec_only) break;
    if (!(live = meet(q, n, mb.polls))) break;
    for (int g = 0; g < groups; g++) {
      w.j0 = j0 + g * kPairs * js;
      if (!kept) load_pairs(q, w, st);
      pairs_ap(q, w, st, pp, !local, red);
      if (!kept) {
#pragma unroll
        for (int i = 0; i < kPairs; i++)
          if (w.at(i) < L) q.Ap[w.at(i)] = st[i].ap;
      }
    }
    if (!(live = pause())) break;
    pAp = total(q, pp, !local, red);
    if (broke(pAp)) {
      brk = true;
      break;
    }
    const double a = rs / pAp;
    for (int g = 0; g < groups; g++) {
      w.j0 = j0 + g * kPairs * js;
      if (!kept) load_pairs(q, w, st);
      pairs_xr(q, w, st, a, pr, !local, red);
      if (!kept) {
#pragma unroll
        for (int i = 0; i < kPairs; i++)
          if (w.at(i) < L) {
            q.x[w.at(i)] = st[i].x;
            q.r[w.at(i)] = st[i].r;
          }
      }
    }
    if (!(live = pause())) break;
    rn = total(q, pr, !local, red);
    it++;
    if (rn <= q.tol * q.tol * rs0) {
      conv = true;
      break;
    }
    const double be = rn / rs;
    rs = rn;
    if (it >= cap) break;
    if (own) __syncthreads();   // the sums in red are read
    for (int g = 0; g < groups; g++) {
      w.j0 = j0 + g * kPairs * js;
      if (!kept) load_pairs(q, w, st);
#pragma unroll
      for (int i = 0; i < kPairs; i++) {
        st[i].p = fma(be, st[i].p, st[i].r);
        if (own) red[i * CT + tid] = st[i].p;
        else if (w.at(i) < L) st_x(q.p + w.at(i), st[i].p);
      }
    }
    if (own) __syncthreads();
    else if (!(live = meet(q, n, mb.polls))) break;
  }
  if (kept && !matvec_only && (!own || b == 0)) {
#pragma unroll
    for (int i = 0; i < kPairs; i++)
      if (w.at(i) < L) q.x[w.at(i)] = st[i].x;
  }
  if (threadIdx.x == 0) {
    if (b == 0 && !matvec_only) {
      CGScalars* sc = q.sc;
      sc->rs0 = rs0;
      sc->pAp = pAp;
      sc->rs_new = rn;
      sc->rs = rn;
      sc->iters = live ? it : -1;
      sc->converged = conv ? 1 : 0;
      sc->breakdown = brk ? 1 : 0;
      sc->done = 1;
    }
    // the last workgroup to leave resets the counters for the next launch:
    // all have passed their last meeting then
    if (__hip_atomic_fetch_add(q.bar + 32, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
        (unsigned)nb - 1u) {
      __hip_atomic_store(q.bar, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(q.bar + 32, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// Block partial -> problem scalar: the block that arrives last among `nblk`
// returns true with the sum of all partials (block order) in `total`.
__device__ inline bool reduce_last(double v, double* red, double* part, unsigned* ticket,
                                   int blk, int nblk, double& total) {
  __shared__ int last;
  const double s = block_sum(v, red);
  if (threadIdx.x == 0) {
    part[blk] = s;
    __threadfence();
    const unsigned t = atomicAdd(ticket, 1u);
    last = (t == (unsigned)nblk - 1u);
  }
  __syncthreads();
  if (!last) return false;
  __threadfence();
  double w = 0.0;
  for (int i = threadIdx.x; i < nblk; i += blockDim.x) w += __builtin_nontemporal_load(&part[i]);
  // fixed assignment of partials to threads and a fixed tree: deterministic
  total = block_sum(w, red);
  if (threadIdx.x == 0) atomicExch(ticket, 0u);
  return true;
}

// theta -= lr delta in the reference layout [a | b | W], |delta|^2; nothing in
// the whole batch when the workgroups of a problem gave up a meeting (iters
// -1): its x may be of different iterations, and a step is taken for all or none
__global__ __launch_bounds__(kMultiVecBlock) void k_mb_apply(MultiBatch mb) {
  __shared__ double red[kMultiVecBlock];
  const int qi = find_prob<F_APPLY>(mb, blockIdx.x);
  const MultiProb& q = mb.probs[qi];
  const int blk = blockIdx.x - q.blk_apply, nblk = q.nvec;
  const int N = q.N, M = q.M, N1 = N + 1, L = (M + 1) * N1;
  const int e = blk * kMultiVecBlock + threadIdx.x;
  int gave_up = 0;
  for (int i = threadIdx.x; i < mb.n; i += kMultiVecBlock) gave_up |= mb.probs[i].sc->iters < 0;
  gave_up = __syncthreads_or(gave_up);
  double xx = 0.0;
  if (e < L - 1 && !gave_up) {
    const int h = e / N1, i = e - h * N1;
    const long k = (h == M) ? i : (i == N ? (long)N + h : (long)N + M + (long)h * N + i);
    const double d = q.x[e];
    q.par[k] += -q.lr * d;
    xx = d * d;
  }
  double tot;
  if (reduce_last(xx, red, q.part, q.ticket, blk, nblk, tot) && threadIdx.x == 0) *q.norm2 = tot;
}

// one thread per problem
__global__ void k_mb_gather(MultiBatch mb, double* out) {
  const int qi = blockIdx.x * blockDim.x + threadIdx.x;
  if (qi >= mb.n) return;
  const MultiProb& q = mb.probs[qi];
  const CGScalars* sc = q.sc;
  unsigned long long a = 0, t = 0;
  for (int c = 0; c < q.C; c++) {
    a += q.acc[c];
    t += q.tot[c];
  }
  double* o = out + (long)qi * kMultiOut;
  o[0] = q.stats[0];
  o[1] = q.stats[1];
  o[2] = *q.norm2;
  o[3] = (double)sc->iters;
  o[4] = (double)sc->converged;
  o[5] = (double)sc->breakdown;
  o[6] = sc->pAp;
  o[7] = sc->rs_new;
  o[8] = sc->rs0;
  o[9] = t ? (double)a / (double)t : 0.0;
  o[10] = q.range_flag ? (double)*q.range_flag : 0.0;
}

constexpr size_t kCgLds = 156 * 1024;   // of the CU's 160 KB: one workgroup per CU

size_t lds_bytes(const MultiProb& q, int hct, int zb) {
  const size_t z = (size_t)hct * 16 * q.si + (size_t)hct * 2 * zb;
  const size_t g = (size_t)CW * (kTiles * 256 + 64 + 96);
  return sizeof(double) * (lds_head(q.nw) + (z > g ? z : g));
}

// Shares of the rows of p on nb workgroups, more than one where these outnumber
// the 16-sample tiles: by samples alone every workgroup reads all of p for 16
// samples that keep one wave in eight busy.  One problem, 50 iterations, by
// samples / shared, ms: N 256, M 256 (66049 parameters), 512 samples 6.4 / 3.5,
// 2048 7.3 / 5.8; N 128, M 128 (16641), 512 2.35 / 2.14, 1024 2.51 / 2.51, 2048
// 2.81 / 3.21; N 64, M 64 (4225), 256 1.63 / 1.78.  So for many parameters, 16
// and more to a sample.
int row_parts(const MultiProb& q, int nb) {
  const int nT = (q.B + 15) / 16, T = tiles64(q.M);
  const long L = (q.M + 1L) * (q.N + 1);
  if (L < 16384 || L < 16L * q.B) return 1;
  const int p = nb / nT;
  return p < 1 ? 1 : p < T ? p : T;
}
static_assert(16384 > kPairs * CT, "a problem that is whole in every workgroup (own) has one part");

// Cycles of a CG iteration of q on nb workgroups of a CU each (FP64 16x16x4
// MFMAs take a SIMD 64): Z by 16-sample tiles, G by units (the site tiles of a
// wave, nt, for the fewest), the meetings and the vector work.
double iter_cost(const MultiProb& q, int nb, int& nt) {
  const int HT = (q.M + 16) / 16, KK = (q.N + 4) / 4, nT = (q.B + 15) / 16;
  const int parts = row_parts(q, nb), per = nb / parts, hp = (tiles64(q.M) + parts - 1) / parts * 4;
  const double z = 16.0 * ((nT + per - 1) / per) * (hp < HT ? hp : HT) * (KK + 4) +
                   (q.M + 1.0) * (q.N + 1.0) / (8 * parts);
  const int ws = q.nsplit < CW ? q.nsplit : CW, rounds = q.nsplit / ws;
  double g = 0.0;
  for (int t = 1; t <= kTiles && t <= kTiles * 2 * ws / CW + 1; t++) {
    // a unit's elements are at most kTiles per thread
    if (t * (CW / ws) > 2 * kTiles) break;
    const int n = (tile_units(q, t) + nb - 1) / nb;
    const double c = n * (2000.0 + rounds * (1200.0 + (q.chunk + 63) / 64 * (600.0 + 2048.0 * t)));
    if (t == 1 || c < g) {
      g = c;
      nt = t;
    }
  }
  const int J = (q.nvec + 1) / 2;
  return z + g + (nb == 1 ? 8000.0 : J <= kPairs ? 16000.0 : 26000.0) + 4000.0 * J / (kPairs * nb);
}

}  // namespace

int multi_words(int N) { return (N + 1 + 31) / 32; }
int multi_parts(int M) { return tiles64(M); }
size_t multi_ta_elems(int B, int M) { return (size_t)((M + 16) / 16) * ((B + 15) / 16 * 4) * 64; }

// nsplit slots of equal runs of samples (multiples of 16)
void multi_shape(MultiProb& q, int nsplit) {
  const int N1 = q.N + 1, M1 = q.M + 1, n4 = (N1 + 3) / 4 * 4;
  q.nsplit = nsplit;
  q.chunk = ((q.B + nsplit - 1) / nsplit + 15) / 16 * 16;
  q.nw = multi_words(q.N);
  q.si = n4 + 2;   // 2 mod 4: the 16 x 2 operands of half a wave fall on 32 bank pairs
  q.nvec = (M1 * N1 + kMultiVecBlock - 1) / kMultiVecBlock;
}

// Hidden tiles of a chunk of p and samples of a pass over it in Z, by what the
// LDS holds for a workgroup's share of the rows (parts) and samples
void shape_rows(const MultiProb& q, MultiRows& w) {
  int HT = (tiles64(q.M) + w.parts - 1) / w.parts * 4;
  if (HT > (q.M + 16) / 16) HT = (q.M + 16) / 16;
  w.zb = w.samples;
  if (w.zb > kZs) w.zb = kZs;
  w.hct = (HT + 1) / 2 * 2;
  while (w.zb > kZb && lds_bytes(q, w.hct < 8 ? w.hct : 8, w.zb) > kCgLds) w.zb -= 16;
  while (w.hct > 2 && lds_bytes(q, w.hct, w.zb) > kCgLds) w.hct -= 2;
  const int nc = (HT + w.hct - 1) / w.hct;   // equal chunks
  w.hct = ((HT + nc - 1) / nc + 1) / 2 * 2;
}

// First blocks of every launch, and the workgroups of the cooperative one:
// every problem gets one; the rest go, to the next count that shortens its
// iteration, to the problem with the longest.
void multi_layout(MultiProb* probs, int n, MultiBatch& mb) {
  int cus = 0, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    cus = 0;
  (void)hipGetLastError();
  size_t lds = 0;
  std::vector<double> cost(n);
  for (int i = 0; i < n; i++) {
    MultiProb& q = probs[i];
    q.nb = 1;
    cost[i] = iter_cost(q, 1, q.nt);
  }
  for (int left = cus - n; left > 0;) {
    int at = 0;
    for (int i = 1; i < n; i++)
      if (cost[i] > cost[at]) at = i;
    MultiProb& q = probs[at];
    int nb = q.nb + 1, nt = 1;
    double c = iter_cost(q, nb, nt);
    while (c >= 0.98 * cost[at] && nb - q.nb <= left) c = iter_cost(q, ++nb, nt);
    if (nb - q.nb > left) break;
    left -= nb - q.nb;
    q.nb = nb;
    q.nt = nt;
    cost[at] = c;
  }
  // the launch of the row weights: 128 samples a workgroup, where that leaves
  // CUs without one shares of the rows, then fewer samples
  long items = 0;
  for (int i = 0; i < n; i++) items += (probs[i].B + kZb - 1) / kZb;
  const int want = items < cus ? (int)((cus + items - 1) / items) : 1;
  int prep = 0, z = 0, g = 0, vec = 0, apply = 0, cg = 0;
  mb.shared = 0;
  for (int i = 0; i < n; i++) {
    MultiProb& q = probs[i];
    const int T = tiles64(q.M);
    q.coop.parts = row_parts(q, q.nb);
    if (q.coop.parts > 1) mb.shared = 1;
    const int shares = q.nb / q.coop.parts;
    q.coop.samples = ((q.B + 15) / 16 + shares - 1) / shares * 16;
    q.solo.parts = want < T ? want : T;
    q.solo.samples = kZb;
    while (q.solo.samples > 32 && q.solo.parts * kZb < want * q.solo.samples) q.solo.samples /= 2;
    shape_rows(q, q.coop);
    shape_rows(q, q.solo);
    for (const MultiRows* w : {&q.coop, &q.solo}) {
      const size_t b = lds_bytes(q, w->hct, w->zb);
      if (b > lds) lds = b;
    }
    q.blk_prep = prep;
    q.blk_z = z;
    q.blk_g = g;
    q.blk_vec = vec;
    q.blk_apply = apply;
    q.blk_cg = cg;
    prep += (q.B + 63) / 64;
    z += (q.B + q.solo.samples - 1) / q.solo.samples * q.solo.parts;
    g += tile_units(q, q.nt);
    vec += ((q.nvec + 1) / 2 + kPairs - 1) / kPairs;
    apply += q.nvec;
    cg += q.nb;
  }
  mb.n = n;
  mb.nblk_prep = prep;
  mb.nblk_z = z;
  mb.nblk_g = g;
  mb.nblk_vec = vec;
  mb.nblk_apply = apply;
  mb.nblk_cg = n <= cus ? cg : 0;   // more problems than CUs: launch by launch
  mb.lds = lds;
}

int launch_multi_prep(const MultiBatch& mb, hipStream_t st) {
  if (mb.n <= 0) return 0;
  KScope ks("multi_prep", st);
  hipLaunchKernelGGL(k_mb_prep, dim3((unsigned)mb.nblk_prep), dim3(256), 0, st, mb);
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

namespace {

int phase(const MultiBatch& mb, int ph, int it, const char* tag, hipStream_t st) {
  static bool set = false;
  if (!set) {
    NQS_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_mb_phase),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)kCgLds));
    set = true;
  }
  const bool g = ph <= PH_GE || ph == PH_G, z = ph == PH_Z;
  KScope ks(tag, st);
  hipLaunchKernelGGL(k_mb_phase, dim3((unsigned)(z ? mb.nblk_z : g ? mb.nblk_g : mb.nblk_vec)), dim3(CT),
                     z || g ? mb.lds : sizeof(double) * kPairs * CT, st, mb, ph, it);
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace

int launch_multi_force(const MultiBatch& mb, hipStream_t st) {
  if (mb.n <= 0) return 0;
  if (phase(mb, PH_G1, 0, "multi_gemm_g", st) || phase(mb, PH_GE, 0, "multi_gemm_g", st) ||
      phase(mb, PH_F, 0, "multi_vec", st))
    return -1;
  return 0;
}

int launch_multi_cg_iter(const MultiBatch& mb, int it, int matvec_only, hipStream_t st) {
  if (mb.n <= 0) return 0;
  if (phase(mb, PH_Z, it, "multi_gemm_z", st) || phase(mb, PH_G, it, "multi_gemm_g", st)) return -1;
  if (matvec_only) return 0;
  if (phase(mb, PH_AP, it, "multi_vec", st) || phase(mb, PH_XR, it, "multi_vec", st) ||
      phase(mb, PH_P, it, "multi_vec", st))
    return -1;
  return 0;
}

int launch_multi_cg_persist(const MultiBatch& mb, int iters, hipStream_t st, int matvec_only) {
  if (mb.n <= 0 || iters <= 0) return 0;
  if (mb.nblk_cg <= 0) {
    fprintf(stderr, "nqs_hip: more problems than CUs for the persistent CG launch\n");
    return -1;
  }
  const void* kernel = mb.shared ? reinterpret_cast<const void*>(k_mb_cg<true>)
                                 : reinterpret_cast<const void*>(k_mb_cg<false>);
  static bool set[2] = {false, false};
  if (!set[mb.shared ? 1 : 0]) {
    NQS_HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kCgLds));
    set[mb.shared ? 1 : 0] = true;
  }
  MultiBatch a = mb;
  void* args[] = {&a, &iters, &matvec_only};
  KScope ks("multi_cg", st);
  // a grid of whole XCD rounds; the workgroups past the last problem return
  const unsigned grid = (unsigned)(mb.nblk_cg + 7) / 8 * 8;
  const hipError_t e = hipLaunchCooperativeKernel(kernel, dim3(grid), dim3(CT), args,
                                                  (unsigned)mb.lds, st);
  count_launch();
  if (e != hipSuccess) {
    (void)hipGetLastError();
    fprintf(stderr, "nqs_hip: persistent CG launch refused (%s)\n", hipGetErrorString(e));
    return -1;
  }
  return 0;
}

int launch_multi_apply(const MultiBatch& mb, hipStream_t st) {
  if (mb.n <= 0) return 0;
  hipLaunchKernelGGL(k_mb_apply, dim3((unsigned)mb.nblk_apply), dim3(kMultiVecBlock), 0, st, mb);
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

int launch_multi_gather(const MultiBatch& mb, double* out, hipStream_t st) {
  if (mb.n <= 0) return 0;
  hipLaunchKernelGGL(k_mb_gather, dim3((unsigned)((mb.n + 63) / 64)), dim3(64), 0, st, mb, out);
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace nqs
