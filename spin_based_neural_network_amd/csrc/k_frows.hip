// k_frows.hip — products with the O rows of an RBM that are never formed:
// u = O v and O^T w from the spins and t = tanh theta, and the CG of the
// (holomorphic) SR step on them (src/nqs/nqs_optimizer.c:44-139, :317-401).
//
// A row is (s, t, t (x) s) for a real RBM; for a complex one
//   R = (s, Re t, Re t (x) s | 0, -Im t, -Im t (x) s),
//   I = (0, Im t, Im t (x) s | s,  Re t,  Re t (x) s)
// (R alone for the real-projected step).  A spin is exactly +-1, so
// (t s) v = t (s v) is one rounding either way, and the kernels below add the
// same terms in the same order as k_rowdot and k_colsum_* do over stored
// rows: lane l of a row's 64 partial sums takes the entries k = l (mod 64) in
// ascending order and the partials meet by halves; a column is summed over
// 128 samples at a time and the chunks in order.  Every result has the bits
// that the stored rows give, which matters where 100 unconverged CG steps
// would amplify another order of sums.
//
// What it replaces: four passes over B x P doubles per CG iteration.  Kagome
// 2x4, complex RBM M = 96, 16384 samples, holomorphic (P = 4848): 0.63 ms of
// kernels per iteration over 2 x 635 MB of rows, 0.089 ms here (row products
// 49 us, column products 22, chunk sums and A p 7.6, the rest of the iteration
// 11); the step 68.3 -> 10.0 ms.  The 318 M fused multiply-adds of a product
// are 8 us at the FP64 rate.
#include <type_traits>

#include "nqs_kernels.h"

namespace nqs {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int kChunk = 128;     // samples of one column partial (as kColChunk)
constexpr int RT = 512;         // threads of k_fr_rowdot: 8 waves x 64 rows
constexpr int kPad = 8;         // lane masks before site 0 and past site N

__device__ inline double flip_sign(double v, bool neg) {
  const int hi = __double2hiint(v);
  return __hiloint2double(neg ? (int)(hi ^ 0x80000000) : hi, __double2loint(v));
}

}  // namespace

// Signs (bit: s = -1) by row, 32 sites a word ([word][Bp], Bp rows a multiple
// of 64), and per 64 rows one lane mask per site (bit l: row l), with room on
// both sides so that eight can be read from 7 before any site on
__global__ __launch_bounds__(64) void k_fr_bits(const int* __restrict__ spins, int B, int N, int Bp,
                                                unsigned* __restrict__ bits,
                                                unsigned long long* __restrict__ lanes) {
  const int b = blockIdx.x * 64 + threadIdx.x;
  const bool in = b < B;
  const int* s = spins + (long)(in ? b : B - 1) * N;
  unsigned long long* lm = lanes + (long)blockIdx.x * (N + 2 * kPad);
  if (threadIdx.x < kPad) lm[threadIdx.x] = lm[kPad + N + threadIdx.x] = 0;
  unsigned w = 0;
  for (int i = 0; i < (N + 32) / 32 * 32; i++) {
    const bool neg = in && i < N && s[i < N ? i : 0] < 0;
    const unsigned long long m = __ballot(neg);
    if (threadIdx.x == 0 && i < N) lm[kPad + i] = m;
    w |= neg ? 1u << (i & 31) : 0u;
    if ((i & 31) == 31) {
      bits[(long)(i >> 5) * Bp + b] = w;
      w = 0;
    }
  }
}

// tT [M][B], and tp [B][hp] with `last` at hidden unit M (the visible row:
// 1 and 0) and zeros past it; t is widened exactly
template <typename R>
__global__ __launch_bounds__(256) void k_fr_factors(const R* __restrict__ t, int B, int M, int hp,
                                                    double last, double* __restrict__ tT,
                                                    double* __restrict__ tp) {
  __shared__ double tile[32][33];
  const int b0 = blockIdx.x * 32, h0 = blockIdx.y * 32;
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
  for (int r = y; r < 32; r += 8) {
    const int b = b0 + r, h = h0 + x;
    if (b < B) {
      const double v = h < M ? (double)t[(long)b * M + h] : h == M ? last : 0.0;
      tile[r][x] = v;
      tp[(long)b * hp + h] = v;
    }
  }
  __syncthreads();
  for (int r = y; r < 32; r += 8) {
    const int h = h0 + r, b = b0 + x;
    if (b < B && h < M) tT[(long)h * B + b] = tile[x][r];
  }
}

__global__ void k_fr_ones(double* __restrict__ x, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) x[i] = 1.0;
}

namespace {

// Eight sums as scalars: an array that loops index is kept as one vector of 16
// registers by the compiler and copied whole at every branch.
struct Acc8 {
  double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0, a4 = 0.0, a5 = 0.0, a6 = 0.0, a7 = 0.0;
  template <int C>
  __device__ __forceinline__ double& at() {
    static_assert(C >= 0 && C < 8, "eight sums");
    if constexpr (C == 0) return a0;
    else if constexpr (C == 1) return a1;
    else if constexpr (C == 2) return a2;
    else if constexpr (C == 3) return a3;
    else if constexpr (C == 4) return a4;
    else if constexpr (C == 5) return a5;
    else if constexpr (C == 6) return a6;
    else return a7;
  }
};
template <typename F>
__device__ __forceinline__ void each8(F f) {
  f(std::integral_constant<int, 0>());
  f(std::integral_constant<int, 1>());
  f(std::integral_constant<int, 2>());
  f(std::integral_constant<int, 3>());
  f(std::integral_constant<int, 4>());
  f(std::integral_constant<int, 5>());
  f(std::integral_constant<int, 6>());
  f(std::integral_constant<int, 7>());
}

// acc += x v and acc -= x v, in place
__device__ __forceinline__ void fma_in(double& acc, double x, double v) {
  asm("v_fmac_f64 %0, %1, %2" : "+v"(acc) : "v"(x), "v"(v));
}
__device__ __forceinline__ void fms_in(double& acc, double x, double v) {
  asm("v_fma_f64 %0, -%1, %2, %0" : "+v"(acc) : "v"(x), "v"(v));
}

// aR, aI += one entry: R and I of plane PL times v, the row's sign in `neg`
template <int KIND, int PL>
__device__ __forceinline__ void row_entry(double tr, double ti, double v, bool neg, double& aR,
                                          double& aI) {
  if (PL == 0 || KIND == 2) {
    const double sr = flip_sign(tr, neg);
    fma_in(PL == 0 ? aR : aI, sr, v);
  }
  if (KIND && (PL == 1 || KIND == 2)) {
    const double si = flip_sign(ti, neg);
    if (PL == 0) fma_in(aI, si, v);
    else fms_in(aR, si, v);
  }
}

// dst[e] = get(e), e < n, over the workgroup: eight loads of a thread in
// flight at a time (one by one, a workgroup's 100 KB of t took 12 us)
template <typename G>
__device__ __forceinline__ void stage(double* dst, int n, G get) {
  for (int e0 = threadIdx.x; e0 < n; e0 += 8 * RT) {
    double x[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int e = e0 + j * RT;
      x[j] = get(e < n ? e : e0);
    }
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (e0 + j * RT < n) dst[e0 + j * RT] = x[j];
  }
}

// One plane of a row product: the partial sums of this wave's residues over
// its entries, in ascending order.  The weights go by segments of `seg`
// entries whose part of v, and unless all of t is `staged` in ts already,
// whose hidden units' t, are staged in LDS.
template <int KIND, int PL>
__device__ __forceinline__ void row_plane(const FactorRows& f, const double* __restrict__ v,
                                          const unsigned long long* __restrict__ lm,
                                          const double* __restrict__ tT,
                                          const double* __restrict__ tiT, int seg, int hseg,
                                          bool staged, int wave, int lane, long row0, double* ts,
                                          Acc8& aR, Acc8& aI) {
  const int N = f.N, M = f.M, B = f.B;
  const int Pr = N + M + M * N, k0 = PL * Pr;
  const long rc = row0 + lane < B ? row0 + lane : B - 1;
  const int wk = 8 * wave;
  double* tis = ts + hseg * 64;
  double* vs = ts + (KIND ? 2 : 1) * hseg * 64;
  // visible: R has s in plane 0, I in plane 1
  if (PL == 0 || KIND == 2) {
#pragma unroll 1
    for (int kb = (k0 & ~63) + wk; kb < k0 + N; kb += 64) {
      each8([&](auto ci) {
        constexpr int c = ci;
        const int k = kb + c;
        if (k >= k0 && k < k0 + N) {
          const double sv = flip_sign(v[k], __builtin_amdgcn_inverse_ballot_w64(lm[k - k0]));
          if (PL == 0) aR.template at<c>() += sv;
          else aI.template at<c>() += sv;
        }
      });
    }
  }
  // hidden biases
#pragma unroll 1
  for (int kb = ((k0 + N) & ~63) + wk; kb < k0 + N + M; kb += 64) {
    each8([&](auto ci) {
      constexpr int c = ci;
      const int k = kb + c;
      if (k >= k0 + N && k < k0 + N + M) {
        const int h = k - k0 - N;
        const long at = (long)h * B + rc;
        const double tr = staged ? ts[h * 64 + lane] : tT[at];
        const double ti = !KIND ? 0.0 : staged ? tis[h * 64 + lane] : tiT[at];
        row_entry<KIND, PL>(tr, ti, v[k], false, aR.template at<c>(), aI.template at<c>());
      }
    });
  }
  // weights: entry w0 + h N + i
  const int w0 = k0 + N + M, w1 = k0 + Pr;
  const int s1 = 64 / N, s2 = 64 - s1 * N;
#pragma unroll 1
  for (int ks = w0 & ~63; ks < w1; ks += seg) {
    const int ka = ks > w0 ? ks : w0, ke = ks + seg < w1 ? ks + seg : w1;
    const int hA = staged ? 0 : (ka - w0) / N;
    __syncthreads();
    stage(vs, ke - ks, [&](int e) { return v[ks + e]; });
    if (!staged) {
      const int n = ((ke - 1 - w0) / N - hA + 1) * 64;
      auto at = [&](int e) {
        const long r = row0 + (e & 63);
        return (long)(hA + (e >> 6)) * B + (r < B ? r : B - 1);
      };
      stage(ts, n, [&](int e) { return tT[at(e)]; });
      if (KIND) stage(tis, n, [&](int e) { return tiT[at(e)]; });
    }
    __syncthreads();
    // A step: the entries kb + c0 .. kb + c1 - 1 of this wave's eight that
    // belong to hidden unit h, sites i ..; the others of the eight take a zero
    // of the vector.  A group that reaches into the next hidden unit is two
    // steps (a branch for them made the compiler copy all sums at its end).
    // The operands of a step are loaded while the step before is summed.
    struct Step {
      int kb, c0, h, i;
    };
    struct Ops {
      double2 v0, v2, v4, v6;                  // the vector at kb ..
      unsigned long long m0, m1, m2, m3, m4, m5, m6, m7;   // lane masks of the sites
      double tr, ti;
    };
    auto load = [&](Step s) {
      const double2* vp = (const double2*)(vs + (s.kb - ks));
      const unsigned long long* mp = lm + (s.i - s.c0);
      const int at = (s.h - hA) * 64 + lane;
      return Ops{vp[0], vp[1], vp[2], vp[3], mp[0], mp[1], mp[2], mp[3],
                 mp[4], mp[5], mp[6], mp[7], ts[at], KIND ? tis[at] : 0.0};
    };
    Step s;
    s.kb = ks + wk;
    if (s.kb + 8 <= ka) s.kb += 64;   // (the eight before the weights begin)
    if (s.kb >= ke) continue;
    s.c0 = ka > s.kb ? ka - s.kb : 0;
    const int e0 = s.kb + s.c0 - w0;
    s.h = __builtin_amdgcn_readfirstlane(e0 / N);
    s.i = __builtin_amdgcn_readfirstlane(e0 - e0 / N * N);
    Ops o = load(s);
#pragma unroll 1
    while (s.kb < ke) {
      int c1 = s.c0 + N - s.i;
      if (c1 > 8) c1 = 8;
      if (c1 > ke - s.kb) c1 = ke - s.kb;
      Step n;
      const bool split = c1 < 8 && s.kb + c1 < ke;   // the rest of the eight is the next unit's
      n.kb = split ? s.kb : s.kb + 64;
      n.c0 = split ? c1 : 0;
      // from (h, i) at c0 on: to c1, or to the next group's first entry
      const int back = s.i - s.c0 + s2;              // site of kb + 64, before wrapping
      int hn = s.h + s1, in = back;
      while (in < 0) {
        in += N;
        hn--;
      }
      while (in >= N) {
        in -= N;
        hn++;
      }
      n.h = split ? s.h + 1 : hn;
      n.i = split ? 0 : in;
      const Ops p = load(n.kb < ke ? n : s);
      const int c0 = s.c0;
      auto pick = [&](int c, double x) { return c >= c0 && c < c1 ? x : 0.0; };
      row_entry<KIND, PL>(o.tr, o.ti, pick(0, o.v0.x), __builtin_amdgcn_inverse_ballot_w64(o.m0), aR.a0, aI.a0);
      row_entry<KIND, PL>(o.tr, o.ti, pick(1, o.v0.y), __builtin_amdgcn_inverse_ballot_w64(o.m1), aR.a1, aI.a1);
      row_entry<KIND, PL>(o.tr, o.ti, pick(2, o.v2.x), __builtin_amdgcn_inverse_ballot_w64(o.m2), aR.a2, aI.a2);
      row_entry<KIND, PL>(o.tr, o.ti, pick(3, o.v2.y), __builtin_amdgcn_inverse_ballot_w64(o.m3), aR.a3, aI.a3);
      row_entry<KIND, PL>(o.tr, o.ti, pick(4, o.v4.x), __builtin_amdgcn_inverse_ballot_w64(o.m4), aR.a4, aI.a4);
      row_entry<KIND, PL>(o.tr, o.ti, pick(5, o.v4.y), __builtin_amdgcn_inverse_ballot_w64(o.m5), aR.a5, aI.a5);
      row_entry<KIND, PL>(o.tr, o.ti, pick(6, o.v6.x), __builtin_amdgcn_inverse_ballot_w64(o.m6), aR.a6, aI.a6);
      row_entry<KIND, PL>(o.tr, o.ti, pick(7, o.v6.y), __builtin_amdgcn_inverse_ballot_w64(o.m7), aR.a7, aI.a7);
      o = p;
      s = n;
    }
  }
}

// the partials of the waves HALF .. 2 HALF - 1 added to those of 0 .. HALF - 1
template <int KIND, int HALF>
__device__ inline void meet(double* lds, int wave, int lane, Acc8& aR, Acc8& aI) {
  __syncthreads();
  if (wave >= HALF && wave < 2 * HALF) {
    double* o = lds + (wave - HALF) * 512 + lane;
    each8([&](auto ci) {
      constexpr int c = ci;
      o[c * 64] = aR.template at<c>();
      if (KIND == 2) o[2048 + c * 64] = aI.template at<c>();
    });
  }
  __syncthreads();
  if (wave < HALF) {
    const double* o = lds + wave * 512 + lane;
    each8([&](auto ci) {
      constexpr int c = ci;
      aR.template at<c>() += o[c * 64];
      if (KIND == 2) aI.template at<c>() += o[2048 + c * 64];
    });
  }
}

}  // namespace

// u1 = R v and (KIND 2) u2 = I v.  A workgroup takes 64 rows, a lane one row;
// wave w holds the partial sums of the residues k = 8w .. 8w + 7 (mod 64).
// The sign of a site is a lane mask in scalar registers; v (one address per
// wave) and t are read from LDS.  Bound by instruction issue: per eight
// entries 59 vector instructions, 32 of them the products and their signs, and
// as many scalar ones, on two waves per SIMD (49 us at the kagome size; 81 us
// with a division and a compare per entry).  KIND: 0 real RBM, 1 complex
// real-projected, 2 holomorphic.
template <int KIND>
__global__ __launch_bounds__(RT) void k_fr_rowdot(FactorRows f, const double* __restrict__ v,
                                                  const unsigned long long* __restrict__ lanes,
                                                  const double* __restrict__ tT,
                                                  const double* __restrict__ tiT, int seg, int hseg,
                                                  double* __restrict__ u1, double* __restrict__ u2,
                                                  const int* __restrict__ skip) {
  extern __shared__ double lds[];
  if (skip && *skip) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long row0 = blockIdx.x * 64L, row = row0 + lane;
  const unsigned long long* __restrict__ lm = lanes + (long)blockIdx.x * (f.N + 2 * kPad) + kPad;
  Acc8 aR, aI;
  const bool staged = hseg >= f.M;   // all of t at once
  if (staged) {
    auto at = [&](int e) {
      const long r = row0 + (e & 63);
      return (long)(e >> 6) * f.B + (r < f.B ? r : f.B - 1);
    };
    stage(lds, f.M * 64, [&](int e) { return tT[at(e)]; });
    if (KIND) stage(lds + hseg * 64, f.M * 64, [&](int e) { return tiT[at(e)]; });
    __syncthreads();
  }
  row_plane<KIND, 0>(f, v, lm, tT, tiT, seg, hseg, staged, wave, lane, row0, lds, aR, aI);
  if (KIND) row_plane<KIND, 1>(f, v, lm, tT, tiT, seg, hseg, staged, wave, lane, row0, lds, aR, aI);
  // the 64 partials of a row, by halves: residues 32, 16 and 8 apart sit in
  // other waves, 4, 2 and 1 apart in this thread
  meet<KIND, 4>(lds, wave, lane, aR, aI);
  meet<KIND, 2>(lds, wave, lane, aR, aI);
  meet<KIND, 1>(lds, wave, lane, aR, aI);
  if (wave == 0 && row < f.B) {
    u1[row] = ((aR.a0 + aR.a4) + (aR.a2 + aR.a6)) + ((aR.a1 + aR.a5) + (aR.a3 + aR.a7));
    if (KIND == 2)
      u2[row] = ((aI.a0 + aI.a4) + (aI.a2 + aI.a6)) + ((aI.a1 + aI.a5) + (aI.a3 + aI.a7));
  }
}

// Column partials of R^T w1 and (KIND 2) I^T w2 over chunk c of 128 samples,
// work[c][R, I][plane][hidden unit, M the visible row][site, N the bias, np
// in all], on FP64 MFMA: v_mfma_f64_16x16x4 adds its four products to the
// accumulator one after the other, each fused (checked bit for bit against
// that chain), so a tile carries the chain over the samples.  A wave takes 16
// hidden units (t as A: 16 consecutive units of 4 samples) and 16 sites (s w
// as B, the sign set per lane), 32 steps of 1, 2 or 4 products, the operands
// of 16 samples in flight ahead (22 us at the kagome size, 1792 waves, against
// 43 us with the chains on the vector unit and the signs on the scalar one).  The last
// workgroups of a launch with means take the sums of w1 and w2 over all
// samples (k_sum's order: 1024 strided partials).
template <int KIND>
__global__ __launch_bounds__(256) void k_fr_colsum(FactorRows f, const double* __restrict__ t,
                                                   const double* __restrict__ ti,
                                                   const unsigned* __restrict__ words,
                                                   const double* __restrict__ w1,
                                                   const double* __restrict__ w2, int ht, int st,
                                                   int hp, int nmain, double* __restrict__ work,
                                                   double* __restrict__ mean1,
                                                   double* __restrict__ mean2,
                                                   const int* __restrict__ skip) {
  if (skip && *skip) return;
  const int N = f.N, M = f.M;
  if ((int)blockIdx.x >= nmain) {
    __shared__ double red[256];
    const bool first = (int)blockIdx.x == nmain;
    const double* w = first ? w1 : w2;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    for (long i = threadIdx.x; i < f.B; i += 1024) {
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (i + 256 * q < f.B) s[q] += w[i + 256 * q];
    }
    // block_sum over 1024 threads: 512 apart, 256 apart, then 256 threads
    s[0] += s[2];
    s[1] += s[3];
    s[0] += s[1];
    const double tot = block_sum(s[0], red);
    if (threadIdx.x == 0) *(first ? mean1 : mean2) = (1.0 / f.B) * tot;
    return;
  }
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int item = blockIdx.x * 4 + (threadIdx.x >> 6), per = ht * st;
  const int c = item / per, g = item - c * per, h0 = g / st * 16, i0 = g % st * 16;
  const long b0 = (long)c * kChunk;
  if (b0 >= f.B) return;
  const int nb = (int)(f.B - b0 < kChunk ? f.B - b0 : kChunk);
  const double* tp = t + b0 * hp + h0 + lr;
  const double* tq = KIND ? ti + b0 * hp + h0 + lr : nullptr;
  const unsigned* bw = words + (long)(i0 >> 5) * f.Bp + b0;
  const int up = 31 - ((i0 & 31) + lr);   // site's bit to the sign position
  v4d r0 = {0.0, 0.0, 0.0, 0.0}, r1 = r0, q0 = r0, q1 = r0;
  // a step: samples b + lk; past the chunk's end both operands are zero
  struct Ops {
    double x, y, a, z;
    unsigned m;
  };
  auto load = [&](int b) {
    const int s = b + lk, sc = s < nb ? s : nb - 1;
    Ops o;
    o.x = tp[(long)sc * hp];
    o.y = KIND ? tq[(long)sc * hp] : 0.0;
    o.a = w1[b0 + sc];
    o.z = KIND == 2 ? w2[b0 + sc] : 0.0;
    o.m = bw[sc];
    return o;
  };
  auto use = [&](int b, Ops o) {
    if (b + lk >= nb) o.x = o.y = o.a = o.z = 0.0;
    const int sg = (int)((o.m << up) & 0x80000000u);
    const double sa = __hiloint2double(__double2hiint(o.a) ^ sg, __double2loint(o.a));
    r0 = __builtin_amdgcn_mfma_f64_16x16x4f64(o.x, sa, r0, 0, 0, 0);
    if (KIND) r1 = __builtin_amdgcn_mfma_f64_16x16x4f64(-o.y, sa, r1, 0, 0, 0);
    if (KIND == 2) {
      const double sz = __hiloint2double(__double2hiint(o.z) ^ sg, __double2loint(o.z));
      q0 = __builtin_amdgcn_mfma_f64_16x16x4f64(o.y, sz, q0, 0, 0, 0);
      q1 = __builtin_amdgcn_mfma_f64_16x16x4f64(o.x, sz, q1, 0, 0, 0);
    }
  };
  Ops o0 = load(0), o1 = load(4), o2 = load(8), o3 = load(12);
  for (int b = 0; b < nb; b += 16) {
    const Ops p0 = load(b + 16), p1 = load(b + 20), p2 = load(b + 24), p3 = load(b + 28);
    use(b, o0);
    use(b + 4, o1);
    use(b + 8, o2);
    use(b + 12, o3);
    o0 = p0;
    o1 = p1;
    o2 = p2;
    o3 = p3;
  }
  const long np = st * 16, plane = (long)(M + 1) * np;
  double* o = work + (long)c * (KIND == 2 ? 4 : KIND ? 2 : 1) * plane + i0 + lr;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int h = h0 + lk + 4 * r;
    if (h <= M) {
      double* at = o + h * np;
      at[0] = r0[r];
      if (KIND) at[plane] = r1[r];
      if (KIND == 2) {
        at[2 * plane] = q0[r];
        at[3 * plane] = q1[r];
      }
    }
  }
}

namespace {

// parameter index of entry e = (hidden unit, site) of a plane of the column
// partials: -1 at the padding
__device__ inline long param_of(const FactorRows& f, int pl, int e, int np) {
  const int h = e / np, i = e - h * np;
  const long Pr = (long)f.N + f.M + (long)f.M * f.N;
  if (h > f.M || i > f.N || (h == f.M && i == f.N)) return -1;
  return pl * Pr + (h == f.M ? i : i == f.N ? f.N + h : (long)f.N + f.M + (long)h * f.N + i);
}

// The chunks of entry e in order: wave 0 sums the R partials of 64 entries,
// wave 1 the I partials; the four waves load 16 chunks each into LDS ahead of
// the chain.
template <int KIND>
__device__ inline double chunk_chain(const FactorRows& f, const double* __restrict__ work, int nch,
                                     int np, int pl, int e, double (*buf)[64][64]) {
  constexpr int nq = KIND == 2 ? 2 : 1, npl = KIND ? 2 : 1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long plane = (long)(f.M + 1) * np;
  const bool in = e < plane;
  double s = 0.0;
  for (int c0 = 0; c0 < nch; c0 += 64) {
    __syncthreads();
    double x[nq][16];
#pragma unroll
    for (int j = 0; j < 16; j++) {
      const int c = c0 + wave * 16 + j;
#pragma unroll
      for (int q = 0; q < nq; q++)
        x[q][j] = in && c < nch ? work[((long)c * nq * npl + q * npl + pl) * plane + e] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < 16; j++)
#pragma unroll
      for (int q = 0; q < nq; q++) buf[q][wave * 16 + j][lane] = x[q][j];
    __syncthreads();
    const int n = nch - c0 < 64 ? nch - c0 : 64;
    if (wave < nq)
      for (int j = 0; j < n; j++) s += buf[wave][j][lane];
  }
  return s;
}

// a b rounded: not fused with a sum that it enters
__device__ inline double mul_only(double a, double b) {
  double r = a * b;
  asm volatile("" : "+v"(r));
  return r;
}

}  // namespace

// out1 = a1 R^T w1, out2 = a2 I^T w2 in the reference layout
template <int KIND>
__global__ __launch_bounds__(256) void k_fr_final(FactorRows f, const double* __restrict__ work,
                                                  int nch, int np, double a1, double a2,
                                                  double* __restrict__ out1,
                                                  double* __restrict__ out2) {
  __shared__ double buf[KIND == 2 ? 2 : 1][64][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int pl = blockIdx.y, e = blockIdx.x * 64 + lane;
  const double s = chunk_chain<KIND>(f, work, nch, np, pl, e, buf);
  const long k = param_of(f, pl, e, np);
  if (k < 0 || wave >= (KIND == 2 ? 2 : 1)) return;
  if (wave == 0) out1[k] = a1 * s;
  else out2[k] = a2 * s;
}

// A p of the QGT: k_qgt_finish on the two sums
template <int KIND>
__global__ __launch_bounds__(256) void k_fr_finish(FactorRows f, const double* __restrict__ work,
                                                   int nch, int np, double* __restrict__ out,
                                                   const double* __restrict__ m1,
                                                   const double* __restrict__ u1,
                                                   const double* __restrict__ m2,
                                                   const double* __restrict__ u2, double scale,
                                                   double eps, const double* __restrict__ v,
                                                   const int* __restrict__ skip) {
  __shared__ double buf[KIND == 2 ? 2 : 1][64][64];
  if (skip && *skip) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int pl = blockIdx.y, e = blockIdx.x * 64 + lane;
  const double s = chunk_chain<KIND>(f, work, nch, np, pl, e, buf);
  double c1 = mul_only(1.0 / f.B, s), c2 = 0.0;
  if (KIND == 2) {
    __syncthreads();
    if (wave == 1) buf[0][0][lane] = c1;
    __syncthreads();
    c2 = buf[0][0][lane];
  }
  const long k = param_of(f, pl, e, np);
  if (k < 0 || wave != 0) return;
  // rounded where k_qgt_finish's code rounds; the holomorphic step of a real
  // RBM (holo: its imaginary rows are zero) subtracts the rounded product too
  const double a = KIND == 2   ? fma(-m2[k], u2[0], (c1 + c2) - mul_only(m1[k], u1[0]))
                   : f.holo ? c1 - mul_only(m1[k], u1[0])
                            : fma(-m1[k], u1[0], c1);
  out[k] = fma(scale, a, mul_only(eps, v[k]));
}

// One CG iteration after A p, on one workgroup: alpha, x, r, the stopping
// rule, p (k_sum's order of sums).  In place of seven dependent launches an
// iteration over stored rows takes 34 us at P = 2208 (40 with them), 49 at 4848
// (50), 65 at 7928 (65), 86 at 11828 (83), 106 at 15728 (98): half of kCgOneBlock
// there.  With the factored products, whose iterations past the end are queued
// and do nothing, seven launches fewer in each of those are worth more: up to
// kCgOneBlock (P = 15728, 32 samples: 2.58 ms a step, 2.76 with the launches).
__global__ __launch_bounds__(1024) void k_cg_rest(CGScalars* sc, double* __restrict__ x,
                                                  double* __restrict__ r, double* __restrict__ p,
                                                  const double* __restrict__ Ap, long P, double tol) {
  __shared__ double red[1024];
  __shared__ double bc;
  if (sc->done) return;
  double s = 0.0;
  for (long i = threadIdx.x; i < P; i += 1024) s += p[i] * Ap[i];
  s = block_sum(s, red);
  if (threadIdx.x == 0) bc = s;
  __syncthreads();
  const double pAp = bc, rs = sc->rs;
  if (!(fabs(pAp) >= 1e-30)) {
    if (threadIdx.x == 0) {
      sc->pAp = pAp;
      sc->breakdown = 1;
      sc->done = 1;
    }
    return;
  }
  const double a = rs / pAp;
  s = 0.0;
  for (long i = threadIdx.x; i < P; i += 1024) {
    x[i] += a * p[i];
    const double rn = r[i] + -a * Ap[i];
    r[i] = rn;
    s += rn * rn;
  }
  s = block_sum(s, red);
  __syncthreads();
  if (threadIdx.x == 0) bc = s;
  __syncthreads();
  const double rn = bc;
  const bool conv = rn <= tol * tol * sc->rs0;
  const double be = rn / rs;
  if (!conv)
    for (long i = threadIdx.x; i < P; i += 1024) p[i] = r[i] + be * p[i];
  __syncthreads();
  if (threadIdx.x == 0) {
    sc->pAp = pAp;
    sc->alpha = a;
    sc->rs_new = rn;
    sc->iters += 1;
    if (conv) {
      sc->converged = 1;
      sc->done = 1;
    } else {
      sc->beta = be;
      sc->rs = rn;
    }
  }
}

int launch_cg_rest(CGScalars* sc, double* x, double* r, double* p, const double* Ap, long P,
                   double tol, hipStream_t st) {
  KScope ks("cg_rest", st);
  hipLaunchKernelGGL(k_cg_rest, dim3(1), dim3(1024), 0, st, sc, x, r, p, Ap, P, tol);
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

namespace {

struct Shape {
  int nch, ht, st, np, hp, seg, hseg;
};

// The row product keeps all of t in LDS where that leaves room for 1024
// entries of v, else the hidden units of as many entries as fit.
Shape shape_of(const FactorRows& f) {
  Shape s;
  s.nch = (f.B + kChunk - 1) / kChunk;
  s.ht = (f.M + 16) / 16;
  s.st = (f.N + 16) / 16;
  s.np = s.st * 16;
  s.hp = frows_hidden(f.M);
  constexpr long cap = 150 * 1024;
  const long tb = (f.kind ? 2 : 1) * 64 * 8;
  const bool all = f.M * tb + 1024 * 8 <= cap;
  auto bytes = [&](int seg) {
    return (long)seg * 8 + (all ? f.M : (seg - 1) / f.N + 2) * tb;
  };
  s.seg = 64;
  while (s.seg < 4096 && s.seg < f.M * f.N + 64 && bytes(s.seg + 64) <= cap) s.seg += 64;
  s.hseg = all ? f.M : (s.seg - 1) / f.N + 2;
  if (s.hseg > f.M) s.hseg = f.M;
  return s;
}

template <int KIND>
int colsum(const FactorRows& f, const Shape& s, const double* w1, const double* w2, double* m1,
           double* m2, const int* skip, hipStream_t st) {
  KScope ks("frows_colsum", st);
  const int nmain = (s.nch * s.ht * s.st + 3) / 4;
  const int extra = m1 ? (KIND == 2 ? 2 : 1) : 0;
  hipLaunchKernelGGL(k_fr_colsum<KIND>, dim3((unsigned)(nmain + extra)), dim3(256), 0, st, f, f.tp,
                     f.tip, f.bits, w1, w2, s.ht, s.st, s.hp, nmain, f.work, m1, m2, skip);
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

template <int KIND>
int rowdot(const FactorRows& f, const Shape& s, const double* v, double* u1, double* u2,
           const int* skip, hipStream_t st) {
  static bool set = false;
  if (!set) {
    NQS_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_fr_rowdot<KIND>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    set = true;
  }
  size_t lds = sizeof(double) * ((size_t)(KIND ? 2 : 1) * s.hseg * 64 + s.seg);
  const size_t red = sizeof(double) * (KIND == 2 ? 64 : 32) * 64;
  if (lds < red) lds = red;
  KScope ks("frows_rowdot", st);
  hipLaunchKernelGGL(k_fr_rowdot<KIND>, dim3((unsigned)((f.B + 63) / 64)), dim3(RT), lds, st, f, v,
                     f.lanes, f.tT, f.tiT, s.seg, s.hseg, u1, u2, skip);
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace

// A row product is one workgroup's pass over the P entries for every 64 rows,
// as long for 64 rows as for 16384; stored rows cost what they weigh, and up to
// 256 MB of them stay in the memory-side cache.  Where N is a multiple of 64 and
// the weights do not begin at a multiple of 8, one wave has all the groups that
// reach into the next hidden unit, and twice the others' steps.  us of a CG
// iteration, factored / stored:
//   R alone    N 16, P 2208, B 80: 39 / 37, 160: 40 / 42
//              N 24, P 4848, B 320: 65 / 57, 1280: 64 / 65, 2560: 65 / 71
//              N 64, P 7928, B 1024: 100 / 83, 2048: 101 / 92, 4096: 102 / 130
//              N 100, P 30500, B 1024: 276 / 224, 2048: 282 / 366
//              N 100, P 81000, B 256: 677 / 483, 512: 688 / 688
// and of a holomorphic step (R and I), where the stored rows' two planes are
// also made first:
//   N 24, P 4848, B 16: 1210 / 1280;  N 36, P 7472, B 16: 1330 / 1500
//   N 64, P 11828, B 16: 1700 / 1340, 64: 2940 / 2800, 80: 3310 / 3340
//   N 64, P 15728, B 16: 1640 / 1540, 32: 2560 / 2640
bool frows_pays(int N, int M, long P, int B, bool cplx, bool holo) {
  const bool uneven = N % 64 == 0 && (N + M) % 8 != 0;
  if (holo) return !cplx || P < 7680 || P > 16384 || B > (uneven && P <= 12288 ? 64 : 16);
  return B > (uneven ? 2560 : 1280) || 2L * B > P - 2048 || 8L * B * P > (256L << 20);
}

size_t frows_work_elems(const FactorRows& f) {
  const Shape s = shape_of(f);
  return (size_t)s.nch * (f.kind == 2 ? 4 : f.kind ? 2 : 1) * (f.M + 1) * s.np;
}
int frows_hidden(int M) { return (M + 32) / 32 * 32; }
int frows_words(int N) { return (N + 32) / 32; }
size_t frows_bits_elems(int B, int N) { return (size_t)(B + 63) / 64 * 64 * frows_words(N); }
size_t frows_lane_elems(int B, int N) { return (size_t)(B + 63) / 64 * (N + 2 * kPad); }

int launch_frows_prep(FactorRows& f, const int* spins, const double* t, const double* ti,
                      const float* t32, const float* ti32, hipStream_t st) {
  const int blocks = (f.B + 63) / 64, hp = frows_hidden(f.M);
  f.Bp = blocks * 64;
  hipLaunchKernelGGL(k_fr_bits, dim3((unsigned)blocks), dim3(64), 0, st, spins, f.B, f.N, f.Bp,
                     f.bits, f.lanes);
  const dim3 g((unsigned)((f.B + 31) / 32), (unsigned)(hp / 32));
  for (int pl = 0; pl < (f.kind ? 2 : 1); pl++) {
    double *o = pl ? f.tiT : f.tT, *p = pl ? f.tip : f.tp;
    const double last = pl ? 0.0 : 1.0;
    if (t32)
      hipLaunchKernelGGL(k_fr_factors<float>, g, dim3(256), 0, st, pl ? ti32 : t32, f.B, f.M, hp,
                         last, o, p);
    else
      hipLaunchKernelGGL(k_fr_factors<double>, g, dim3(256), 0, st, pl ? ti : t, f.B, f.M, hp, last,
                         o, p);
  }
  hipLaunchKernelGGL(k_fr_ones, dim3((unsigned)((f.B + 255) / 256)), dim3(256), 0, st, f.ones, f.B);
  count_launch(f.kind ? 4 : 3);
  NQS_HIP_CHECK(hipGetLastError());
  return 0;
}

int launch_frows_colsum(const FactorRows& f, const double* w1, const double* w2, double a1,
                        double a2, double* out1, double* out2, hipStream_t st) {
  const Shape s = shape_of(f);
  if (!w1) w1 = f.ones;
  if (!w2) w2 = f.ones;
  const dim3 g((unsigned)(((f.M + 1) * s.np + 63) / 64), f.kind ? 2 : 1);
  int rc;
  if (f.kind == 0) {
    rc = colsum<0>(f, s, w1, w2, nullptr, nullptr, nullptr, st);
    hipLaunchKernelGGL(k_fr_final<0>, g, dim3(256), 0, st, f, f.work, s.nch, s.np, a1, a2, out1, out2);
  } else if (f.kind == 1) {
    rc = colsum<1>(f, s, w1, w2, nullptr, nullptr, nullptr, st);
    hipLaunchKernelGGL(k_fr_final<1>, g, dim3(256), 0, st, f, f.work, s.nch, s.np, a1, a2, out1, out2);
  } else {
    rc = colsum<2>(f, s, w1, w2, nullptr, nullptr, nullptr, st);
    hipLaunchKernelGGL(k_fr_final<2>, g, dim3(256), 0, st, f, f.work, s.nch, s.np, a1, a2, out1, out2);
  }
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return rc;
}

int launch_frows_qgt(const FactorRows& f, const double* v, const double* m1, const double* m2,
                     double* u1, double* u2, double* mean1, double* mean2, double scale, double eps,
                     double* out, const int* skip, hipStream_t st) {
  const Shape s = shape_of(f);
  const dim3 g((unsigned)(((f.M + 1) * s.np + 63) / 64), f.kind ? 2 : 1);
  int rc;
  if (f.kind == 0) {
    rc = rowdot<0>(f, s, v, u1, u2, skip, st) || colsum<0>(f, s, u1, u2, mean1, mean2, skip, st);
    hipLaunchKernelGGL(k_fr_finish<0>, g, dim3(256), 0, st, f, f.work, s.nch, s.np, out, m1, mean1, m2,
                       mean2, scale, eps, v, skip);
  } else if (f.kind == 1) {
    rc = rowdot<1>(f, s, v, u1, u2, skip, st) || colsum<1>(f, s, u1, u2, mean1, mean2, skip, st);
    hipLaunchKernelGGL(k_fr_finish<1>, g, dim3(256), 0, st, f, f.work, s.nch, s.np, out, m1, mean1, m2,
                       mean2, scale, eps, v, skip);
  } else {
    rc = rowdot<2>(f, s, v, u1, u2, skip, st) || colsum<2>(f, s, u1, u2, mean1, mean2, skip, st);
    hipLaunchKernelGGL(k_fr_finish<2>, g, dim3(256), 0, st, f, f.work, s.nch, s.np, out, m1, mean1, m2,
                       mean2, scale, eps, v, skip);
  }
  count_launch();
  NQS_HIP_CHECK(hipGetLastError());
  return rc ? -1 : 0;
}

}  // namespace nqs
