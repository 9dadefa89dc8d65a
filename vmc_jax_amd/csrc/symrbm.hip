// Symmetrised RBMs (avgFun_Coefficients_Exp over an RBM, sym_wrapper.py:7-9,
// 66-77) with the orbit resident in one workgroup: log psi, local energies and
// Metropolis chains without materialising the |G| transformed configurations,
// their s' or a launch per proposal.
//
// psi(s) = sum_g b_g psi_net(g s).  Flipping site i flips one site of every row
// g s, so psi(s') / psi(s) = sum_g w_g r_g with w_g = b_g psi_net(g s) / psi(s)
// and r_g the RBM ratio of rbmq.hpp: eight FP64 operations per row, hidden
// unit and flip.  Parameters outside the ratio form's range, and orbits with a
// row that reads a site twice, are evaluated row by row from scratch
// (sym_rows_*).
#include <algorithm>
#include <cmath>
#include <string>

#include "rbmq.hpp"

namespace jv {

int set_lds_limit(const void* fn, size_t bytes);
bool make_rbm_geom(const jv_net* net, RbmGeom& g);
OpDev make_opdev(const jv_optable* op, const double* pref, int L);

namespace {

struct SymGeom {
  int G, cpx;          // orbit elements; complex coefficients or factors
  const int32_t* map;  // [G][L]: j for s_j, -1 - j for 1 - s_j
  const double* fac;   // [G] complex
};

constexpr int SYM_MAX_G = 2048;  // per-row sums of one configuration stay in LDS
constexpr int SYM_T = 256;       // threads of the forward and local-energy workgroups

// Row r of the orbit at site i of configuration s.
__device__ inline int row_spin(const SymGeom& o, int L, const int32_t* s, int r, int i) {
  const int m = o.map[(int64_t)r * L + i];
  return m >= 0 ? (s[m] > 0) : !(s[-1 - m] > 0);
}

// Whether the resident chains and local energies apply: parameters in range,
// and every row a permutation of the sites (they look up where a flipped site
// sits in a row; log psi only reads the rows).
__device__ inline bool sym_ok(const RbmGeom& g, const SymGeom& o, const RbmTab& t, int lane) {
  bool ok = true;
  for (int r = lane; r < o.G; r += WAVE) ok = ok && t.perm[r];
  return __all(ok) && rbmq_ok(g, t, 2, lane);
}

struct quad {
  double v[4];
};
// Four neighbouring doubles (two 16-byte loads; h + 3 < H), or the clamped ones.
__device__ inline quad load4(const double* __restrict__ p, int h, int H) {
  quad q;
  if (h + 4 <= H) {
    q = *(const quad*)(p + h);
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) q.v[k] = p[min(h + k, H - 1)];
  }
  return q;
}
// theta of hidden units h .. h + U - 1 (clamped to H - 1; U = 4 or 1) for one
// row's spins.
template <bool CPX, int U = 4>
__device__ inline void theta_of(const RbmGeom& g, const double* __restrict__ P, const unsigned char* row, int h,
                                cd* th) {
  const double* Wr = P + g.ow;
  const double* Wi = Wr + (int64_t)g.L * g.H;
#pragma unroll
  for (int k = 0; k < U; ++k) {
    const int hc = min(h + k, g.H - 1);
    th[k] = {g.ob >= 0 ? P[g.ob + hc] : 0.0, CPX && g.ob >= 0 ? P[g.ob + g.H + hc] : 0.0};
  }
#pragma unroll(U == 4 ? 4 : 8)
  for (int i = 0; i < g.L; ++i) {
    const double sg = row[i] ? 1.0 : -1.0;
    if constexpr (U == 4) {
      const quad wr = load4(Wr + (int64_t)i * g.H, h, g.H);
      quad wm = wr;
      if (CPX) wm = load4(Wi + (int64_t)i * g.H, h, g.H);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        th[k].re = fma(sg, wr.v[k], th[k].re);
        if (CPX) th[k].im = fma(sg, wm.v[k], th[k].im);
      }
    } else {
      th[0].re = fma(sg, Wr[(int64_t)i * g.H + h], th[0].re);
      if (CPX) th[0].im = fma(sg, Wi[(int64_t)i * g.H + h], th[0].im);
    }
  }
}
template <bool CPX>
__device__ inline void ab_of(cd th, typename num_of<CPX>::type& al, typename num_of<CPX>::type& be, cd& lin,
                             typename num_of<CPX>::type& d) {
  if constexpr (CPX) {
    rbm_ab(th, al, be, lin, d);
  } else {
    double l;
    rbm_ab(th.re, al, be, l, d);
    lin = {l, 0.0};
  }
}
// Visible part of log psi of one row, the sites split over `sl` of SL lanes.
__device__ inline cd visible(const RbmGeom& g, const double* __restrict__ P, const unsigned char* row, int sl, int SL) {
  cd v = {0.0, 0.0};
  if (g.oa >= 0)
    for (int i = sl; i < g.L; i += SL) {
      const double sg = row[i] ? 1.0 : -1.0;
      v.re = fma(sg, P[g.oa + i], v.re);
      v.im = fma(sg, P[g.oa + g.L + i], v.im);
    }
  return v;
}

__device__ inline cd block_sum_cd(cd v, double* red) { return {block_sum(v.re, red), block_sum(v.im, red)}; }
__device__ inline double block_max(double v, double* red) {
  for (int o = WAVE / 2; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  __syncthreads();
  if (threadIdx.x % WAVE == 0) red[threadIdx.x / WAVE] = v;
  __syncthreads();
  double m = red[0];
  for (int i = 1; i < (int)blockDim.x / WAVE; ++i) m = fmax(m, red[i]);
  __syncthreads();
  return m;
}
// log of sum_g b_g e^{x_g} d_g from its shifted sum (jax's logsumexp: a
// negative sum of real terms is NaN).
__device__ inline cd log_of_sum(cd S, double shift, int cpx) {
  if (cpx) return {log(hypot(S.re, S.im)) + shift, atan2(S.im, S.re)};
  return {S.re < 0.0 ? NAN : log(fabs(S.re)) + shift, 0.0};
}

// ------------------------------------------------------------------ log psi
// log psi of the spins s (LDS) by the whole workgroup: SL threads per row, U
// hidden units at a time (sym_lanes).  A row's amplitude is
// e^{lin} prod_h d_h / 2^H with Re lin >= 0 and |d_h| <= 2 (rbm_ab), whatever
// the size of theta: no logarithm per unit and no range to test.  lin, dd: [G];
// rb: [threads / SL][L].  Same value in every thread.
template <bool CPX, int U, int SLC>
__device__ __forceinline__ cd block_logpsi(const RbmGeom& g, const SymGeom& o, const double* __restrict__ P,
                                           const int32_t* s, int SLr, cd* lin, cd* dd, unsigned char* rb, double* red) {
  typedef typename num_of<CPX>::type T;
  const int SL = SLC > 0 ? SLC : SLr;
  const int L = g.L, H = g.H, G = o.G, tid = threadIdx.x, nt = blockDim.x, RC = nt / SL;
  const int r = tid / SL, sl = tid % SL;
  double mx = -INFINITY;
  __syncthreads();  // s is set
  for (int r0 = 0; r0 < G; r0 += RC) {
    if (r < min(RC, G - r0)) {
      unsigned char* row = rb + r * L;  // of this row's threads, all in one wave
      wave_sync();
      for (int i = sl; i < L; i += SL) row[i] = row_spin(o, L, s, r0 + r, i);
      wave_sync();
      cd li = visible(g, P, row, sl, SL);
      T dp;
      set_one(dp);
      for (int h = U * sl; h < H; h += U * SL) {
        cd th[U];
        theta_of<CPX, U>(g, P, row, h, th);
#pragma unroll
        for (int k = 0; k < U; ++k)
          if (h + k < H) {
            T al, be, d;
            cd l;
            ab_of<CPX>(th[k], al, be, l, d);
            li = li + l;
            dp = mulc(dp, d);
          }
      }
      for (int m = 1; m < SL; m *= 2) {
        li = li + shfl_xor(li, m);
        dp = mulc(dp, shfl_xor(dp, m));
      }
      if (sl == 0) {
        lin[r0 + r] = li;
        dd[r0 + r] = to_cd(dp);
      }
      if (o.fac[2 * (r0 + r)] != 0.0 || o.fac[2 * (r0 + r) + 1] != 0.0) mx = fmax(mx, li.re);
    }
  }
  mx = block_max(mx, red);
  if (!isfinite(mx)) mx = 0.0;
  cd S = {0.0, 0.0};
  for (int q = tid; q < G; q += nt) {
    const cd b = {o.fac[2 * q], o.fac[2 * q + 1]};
    if (b.re == 0.0 && b.im == 0.0) continue;
    const double x = fma(-(double)H, LN2, lin[q].re - mx);
    if (o.cpx) S = S + mulc(mulc(cexp({x, lin[q].im}), dd[q]), b);
    else S.re += exp(x) * dd[q].re * b.re;
  }
  return log_of_sum(block_sum_cd(S, red), mx, o.cpx);
}

// Threads per row and hidden units at a time (*four: 4, else 1).  Four units a
// thread share a row's spins and signs; one where rows have fewer than 16 units
// or all rows' units fit one wave.  As many threads as the units fill within
// 256 a configuration: with four per row whatever the group, 64 sites x 200
// units of a two-element group took 1701 us for 4096 samples (165 with 64, 258
// by one wave per materialised row); 512 a configuration: 274 against 188 us
// for 64 elements of 16 sites x 32 units.
int sym_lanes(int G, int H, bool* four) {
  int p2 = 4, sl = 4;
  while (p2 < H && p2 < WAVE) p2 *= 2;
  *four = H >= 16 && (H > WAVE || G * p2 > WAVE);
  while (sl < WAVE && (*four ? 4 * sl : sl) < H && 2 * sl * G <= SYM_T) sl *= 2;
  return sl;
}
size_t sym_rows_lds(const RbmGeom& g, int G, int T, int SL) {
  return 8 * 8 + 32 * (size_t)G + 4 * (size_t)g.L + (size_t)(T / SL) * g.L + 16;
}
// Threads of the workgroup: no more than the rows fill or the LDS takes.
int sym_threads(const RbmGeom& g, int G, int SL) {
  int T = std::min(SYM_T, (G * SL + WAVE - 1) / WAVE * WAVE);
  while (T > WAVE && sym_rows_lds(g, G, T, SL) > 160 * 1024) T -= WAVE;
  return T;
}

// Estimated times in us, for the choice between the forms below and materialised
// rows; they hold within a third over groups of 2 to 160, 8 to 64 sites and 3 to
// 200 units (a real network's units cost half).
//
// log psi resident: loading theta, a step of SL threads times U units per site,
// is a chain of loads; beyond 512 workgroups of 256 threads they queue.
double sym_resident_us(const RbmGeom& g, int G, double n) {
  bool four;
  const int SL = sym_lanes(G, g.H, &four), T = sym_threads(g, G, SL), per = (four ? 4 : 1) * SL;
  const double steps = (double)((G * SL + T - 1) / T) * ((g.H + per - 1) / per);
  return (9.0 + (g.cpx ? 0.26 : 0.13) * g.L * steps) * std::max(1.0, 1.3 * n * T / (512.0 * SYM_T));
}
// ... over materialised rows, a wave each (without the launches).
double sym_materialised_us(const RbmGeom& g, int G, double n) {
  const double chain = (double)g.L * ((g.H + WAVE - 1) / WAVE);
  return 0.16 * chain + (g.cpx ? 1.25e-4 : 0.63e-4) * n * G * chain;
}

// A workgroup per configuration.  FP64 issue (exp and sincos of every theta)
// sets its time: 4096 samples, 16 sites x 32 units, 64 elements: 589 us with
// materialised rows, 188 here (a call and its wait).
template <bool CPX, int U, int SLC>
__global__ void __launch_bounds__(SYM_T, 2) sym_rbm_forward(RbmGeom g, SymGeom o, const double* __restrict__ P, int SL,
                                                            const int32_t* __restrict__ cfg, int64_t n,
                                                            double* __restrict__ out) {
  extern __shared__ double lds[];
  double* red = lds;
  cd* lin = (cd*)(red + 8);  // [G]
  cd* dd = lin + o.G;        // [G]
  int32_t* s = (int32_t*)(dd + o.G);
  unsigned char* rb = (unsigned char*)(s + g.L);
  for (int64_t q = blockIdx.x; q < n; q += gridDim.x) {
    for (int i = threadIdx.x; i < g.L; i += blockDim.x) s[i] = cfg[q * g.L + i];
    const cd lp = block_logpsi<CPX, U, SLC>(g, o, P, s, SL, lin, dd, rb, red);
    if (threadIdx.x == 0) {
      out[2 * q] = lp.re;
      out[2 * q + 1] = lp.im;
    }
  }
}

// ------------------------------------------------------------------ local energies
// A workgroup per configuration.  The orbit in chunks of RC rows: four (eight,
// sixteen) threads per row form alpha, beta and w_g; then lane = row (RC < 64:
// several groups of strings per wave), a wave takes four strings at a time, so
// that one read of (alpha, beta) serves four products, and sums them over its
// rows.  LDS reads (24 bytes per row, unit and string) and FP64 issue bound it.
// LDS of alpha, beta chooses RC: rows of 2 H + 1 entries (an odd number of
// 16-byte units, so rows do not share banks).  TAB: the g table in LDS.
// 4096 samples, 16 sites x 32 units, 64 elements, Ising chain: 17644 us with
// materialised rows (4.5e6 forward passes), 455 us here (716 with 64 rows and
// one workgroup per CU).
template <bool CPX, int RC, bool TAB>
__global__ void __launch_bounds__(SYM_T, 2) sym_rbm_eloc(RbmGeom g, SymGeom o, const double* __restrict__ P,
                                                         OpDev op, RbmTab tab, const int32_t* __restrict__ cfg,
                                                         const double* __restrict__ lps, int64_t n, int nstr,
                                                         const double* __restrict__ part, int K,
                                                         double* __restrict__ out) {
  typedef typename num_of<CPX>::type T;
  extern __shared__ double lds[];
  constexpr int SL = SYM_T / RC, NG = WAVE / RC * (SYM_T / WAVE);  // threads per row; groups of strings at once
  const int L = g.L, H = g.H, G = o.G, tid = threadIdx.x, lane = tid % WAVE;
  const int w = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int stride = 2 * H + 1, gq = (nstr + 3) / 4;
  double* red = lds;
  T* ab = (T*)(red + 8);                  // [RC][2 H + 1]
  T* he = ab + (size_t)RC * stride;       // [H][L][2] if TAB
  cd* wt = (cd*)(he + (TAB ? (size_t)2 * H * L : 0));  // [RC]
  cd* mel = wt + RC;                      // [nstr] matrix elements
  cd* sum = mel + nstr;                   // [4 gq] sums over the orbit
  int32_t* site = (int32_t*)(sum + 4 * gq);  // [4 gq][2] changed sites, negative: none
  int32_t* s = site + 8 * gq;
  unsigned short* inv = (unsigned short*)(s + L);  // [RC][L]: position of a site in the row
  unsigned char* rb = (unsigned char*)(inv + RC * L);  // [RC][L]
  const int nl = tab.lead[0];
  if (!sym_ok(g, o, tab, lane)) {  // sym_rows_eloc's
    if (K > 1)
      for (int64_t q = blockIdx.x * (int64_t)SYM_T + tid; q < 2 * n; q += (int64_t)gridDim.x * SYM_T) {
        double v = 0.0;
        for (int k = 0; k < K; ++k) v += part[2 * n * k + q];
        out[q] = v;
      }
    return;
  }
  if (TAB)
    for (int t = tid; t < 2 * H * L; t += SYM_T) he[t] = ((const T*)tab.he)[t];
  for (int64_t q = blockIdx.x; q < n; q += gridDim.x) {
    const cd lq = {lps[2 * q], lps[2 * q + 1]};
    __syncthreads();
    for (int i = tid; i < L; i += SYM_T) s[i] = cfg[q * L + i];
    __syncthreads();
    // matrix elements; the merged diagonal strings (branch_free.py:483-485)
    cd ds = {0.0, 0.0};
    if (op.num_diag > 1)
      for (int d = tid; d < op.num_diag; d += SYM_T) {
        bool fa, fb;
        ds = ds + string2(op, op.diag[d], s, fa, fb);
      }
    for (int j = tid; j < 4 * gq; j += SYM_T) {
      cd m = {0.0, 0.0};
      int sa = -2, sb = -1;  // -2: no string applies to this sample
      if (j < nl) {
        const int code = tab.lead[1 + j], st = code >> 4, fol = code & 15;
        for (int f = 0; f <= fol; ++f) {
          bool fa, fb;
          const cd mf = string2(op, st + f, s, fa, fb);
          if (!nonzero(mf)) continue;
          m = m + mf;
          const int i0 = min(max(op.idx[(st + f) * op.max_len], 0), L - 1);
          sa = fa ? i0 : -1;
          sb = fb ? min(max(op.idx[(st + f) * op.max_len + 1], 0), L - 1) : -1;
          if (sa < 0) {
            sa = sb;
            sb = -1;
          }
        }
      }
      if (j < nstr) mel[j] = m;
      site[2 * j] = sa;
      site[2 * j + 1] = sb;
      sum[j] = {0.0, 0.0};
    }
    ds = block_sum_cd(ds, red);
    cd base = {0.0, 0.0};  // sum_g w_g (threads that own a row's first slice)
    for (int r0 = 0; r0 < G; r0 += RC) {
      const int nr = min(RC, G - r0);
      __syncthreads();
      for (int t = tid; t < nr * L; t += SYM_T) {
        const int r = t / L, i = t % L, m = o.map[(int64_t)(r0 + r) * L + i];
        rb[t] = m >= 0 ? (s[m] > 0) : !(s[-1 - m] > 0);
        inv[r * L + (m >= 0 ? m : -1 - m)] = (unsigned short)i;
      }
      __syncthreads();
      {
        const int r = tid / SL, sl = tid % SL;
        if (r < nr) {
          const unsigned char* row = rb + r * L;
          cd li = visible(g, P, row, sl, SL);
          T dp;
          set_one(dp);
          for (int h = 4 * sl; h < H; h += 4 * SL) {
            cd th[4];
            theta_of<CPX>(g, P, row, h, th);
#pragma unroll
            for (int k = 0; k < 4; ++k)
              if (h + k < H) {
                T al, be, d;
                cd l;
                ab_of<CPX>(th[k], al, be, l, d);
                li = li + l;
                dp = mulc(dp, d);
                ab[(size_t)r * stride + 2 * (h + k)] = al;
                ab[(size_t)r * stride + 2 * (h + k) + 1] = be;
              }
          }
          for (int m = 1; m < SL; m *= 2) {
            li = li + shfl_xor(li, m);
            dp = mulc(dp, shfl_xor(dp, m));
          }
          if (sl == 0) {
            const cd b = {o.fac[2 * (r0 + r)], o.fac[2 * (r0 + r) + 1]};
            cd x = {0.0, 0.0};
            if (b.re != 0.0 || b.im != 0.0)
              x = mulc(mulc(cexp({fma(-(double)H, LN2, li.re - lq.re), li.im - lq.im}), to_cd(dp)), b);
            wt[r] = x;
            base = base + x;
          }
        }
      }
      __syncthreads();
      // products: row = lane % RC, strings 4 jg .. 4 jg + 3
      const int r = lane % RC;
      const T* arow = ab + (size_t)min(r, nr - 1) * stride;
      const T* tabq = TAB ? (const T*)he : (const T*)tab.he;
      for (int jg = w * (WAVE / RC) + lane / RC; jg < (gq + NG - 1) / NG * NG; jg += NG) {
        const int j4 = 4 * min(jg, gq - 1);
        int at[4], at2[4];
        cd pre[4];
        bool two = false;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          pre[k] = {1.0, 0.0};
          at[k] = at2[k] = -1;
          for (int z = 0; z < 2; ++z) {
            const int si = site[2 * (j4 + k) + z];
            if (si < 0) continue;
            const int rr = min(r, nr - 1), i = inv[rr * L + si], v = rb[rr * L + i];
            const double* pq = tab.site + 8 * (int64_t)i + 2 + 2 * v;
            pre[k] = mulc(pre[k], cd{pq[0], pq[1]});
            (z ? at2[k] : at[k]) = 2 * i + v;
            two = two || z;
          }
        }
        T pr[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) set_one(pr[k]);
        if (__any(two)) {
          for (int h = 0; h < H; ++h) {
            const T a = arow[2 * h], b = arow[2 * h + 1];
            const T* qh = tabq + (size_t)2 * h * L;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              T x = qh[max(at[k], 0)], y = qh[max(at2[k], 0)], one;
              set_one(one);
              y = sel(at2[k] >= 0, y, one);
              pr[k] = mulc(pr[k], fmac(b, mulc(x, y), a));
            }
          }
        } else {
#pragma unroll 2
          for (int h = 0; h < H; ++h) {
            const T a = arow[2 * h], b = arow[2 * h + 1];
            const T* qh = tabq + (size_t)2 * h * L;
#pragma unroll
            for (int k = 0; k < 4; ++k) pr[k] = mulc(pr[k], fmac(b, qh[max(at[k], 0)], a));
          }
        }
        const cd wr = r < nr ? wt[r] : cd{0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          cd z = wr;
          if (at[k] >= 0) z = mulc(mulc(to_cd(pr[k]), pre[k]), wr);
          for (int m = 1; m < RC; m *= 2) z = z + shfl_xor(z, m);
          if (r == 0 && jg < gq) sum[4 * jg + k] = sum[4 * jg + k] + z;
        }
      }
    }
    __syncthreads();
    base = block_sum_cd(base, red);
    // a negative sum of real terms has no logarithm (jax's logsumexp): NaN
    cd acc = {0.0, 0.0};
    for (int j = tid; j < nl; j += SYM_T) {
      if (site[2 * j] == -2) continue;
      const cd m = mel[j];  // 0 where strings cancel; a NaN counts all the same
      acc = acc + (!o.cpx && sum[j].re < 0.0 ? cd{NAN, NAN} : mulc(m, sum[j]));
    }
    if (tid == 0 && nonzero(ds)) acc = acc + (!o.cpx && base.re < 0.0 ? cd{NAN, NAN} : mulc(ds, base));
    acc = block_sum_cd(acc, red);
    if (tid == 0) {
      out[2 * q] = acc.re;
      out[2 * q + 1] = acc.im;
    }
  }
}
size_t sym_eloc_lds(const RbmGeom& g, int RC, bool tabl, int nstr) {
  const size_t cw = 8 * (size_t)rbm_cw(g), gq = (nstr + 3) / 4;
  size_t abb = cw * RC * (2 * g.H + 1);
  abb += tabl ? cw * 2 * g.H * g.L : 0;
  return 64 + abb + 16 * (size_t)RC + 16 * (size_t)nstr + 64 * gq + 32 * gq +
         4 * (size_t)g.L + 3 * (size_t)RC * g.L + 16;
}

// ------------------------------------------------------------------ Metropolis chains
// Moves the power of two of a row's weight into its exponent (0, infinities
// and NaN stay as they are).
__device__ inline void scale_row(cd& wt, int& ex) {
  const double m = fmax(fabs(wt.re), fabs(wt.im));
  if (m > 0.0 && m < INFINITY) {
    int e;
    (void)frexp(m, &e);
    wt = {ldexp(wt.re, -e), ldexp(wt.im, -e)};
    ex += e;
  }
}

// A workgroup per chain (sampler.py:264-367), SL threads per row, HT hidden
// units each: e and alpha live in registers, the spins and the flipped
// position of every row in LDS.  A proposal: one product per row, a sum over
// the orbit (one barrier: the partial sums alternate between two slots), the
// decision, and on acceptance e' = e g and one reciprocal per unit.  Proposals
// use the Philox counters of the other chain kernels.  theta is recomputed at
// emissions at least RBMQ_MC_REFRESH proposals apart.  Registers decide how
// many chains share a CU: beta = e alpha is not kept (three waves per SIMD
// instead of one).
// 1024 chains x 140 proposals, 16 sites x 32 units, 64 elements: 22.0 ms with
// one batched forward per proposal, 1.11 ms here (with beta kept, one workgroup
// per CU, 6 % more); 386 vector instructions per wave and proposal, 38 % of the
// issue cycles, bank conflicts of the table reads 37 % of the time.
template <bool CPX, int HT, int MAXT, bool TAB>
__global__ void __launch_bounds__(MAXT, MAXT == 256 ? 3 : MAXT == 512 ? 2 : 4)
    sym_rbm_mc(RbmGeom g, SymGeom o, const double* __restrict__ P, jv_mc_args a, RbmTab tab, int SL,
               int32_t* __restrict__ walkers, int32_t* __restrict__ configs, int64_t* __restrict__ counters) {
  typedef typename num_of<CPX>::type T;
  extern __shared__ double lds[];
  const int L = g.L, H = g.H, G = o.G, tid = threadIdx.x, nt = blockDim.x, lane = tid % WAVE, nw = nt / WAVE;
  const int chain = blockIdx.x;
  double* red = lds;                     // block reductions; [2][16] complex partial sums of the proposals
  cd* part = (cd*)(red + 16);
  cd* pre = part + 32;                   // [L][2]
  T* me = (T*)(pre + 2 * L);                // [L][2][HP] if TAB, HP odd: rows do not share banks
  const int HP = H | 1;
  int32_t* s = (int32_t*)(me + (TAB ? (size_t)2 * L * HP : 0));
  unsigned short* inv = (unsigned short*)(s + L);  // [G][L]: 2 * position + (row holds the flipped spin)
  unsigned char* rb = (unsigned char*)(inv + (size_t)G * L);  // [G][L] spins of the rows (refresh only)
  if (!sym_ok(g, o, tab, lane)) return;  // sym_rows_mc's
  for (int i = tid; i < L; i += nt) s[i] = walkers[(int64_t)chain * L + i] > 0;
  for (int t = tid; t < 2 * L; t += nt) {
    const double* pq = tab.site + 8 * (int64_t)(t / 2) + 2 + 2 * (t % 2);
    pre[t] = {pq[0], pq[1]};
  }
  if constexpr (TAB)
    for (int t = tid; t < 2 * L * H; t += nt) me[t / H * HP + t % H] = ((const T*)tab.me)[t];
  for (int t = tid; t < G * L; t += nt) {
    const int r = t / L, i = t % L, m = o.map[t];
    inv[r * L + (m >= 0 ? m : -1 - m)] = (unsigned short)(2 * i + (m < 0));
  }
  __syncthreads();
  // the ratio form keeps the spins in every wave's registers too (bit w of lane
  // l: site 64 w + l), so one barrier per proposal suffices
  const int words = (L + WAVE - 1) / WAVE;
  uint32_t sp = 0;
  for (int w = 0; w < words; ++w)
    if (w * WAVE + lane < L && s[w * WAVE + lane]) sp |= 1u << w;
  auto spins_out = [&]() {  // registers -> s (all threads call)
    __syncthreads();
    if (tid < WAVE)
      for (int w = 0; w < words; ++w)
        if (w * WAVE + lane < L) s[w * WAVE + lane] = (sp >> w) & 1;
    __syncthreads();
  };
  const int r = tid / SL, sl = tid % SL, h0 = sl * HT;
  const bool mine = r < G;
  const int rc = min(r, G - 1);
  const cd b = {o.fac[2 * rc], o.fac[2 * rc + 1]};
  T e[HT], al[HT];
  // b_g psi_net(g s) up to a common factor, wt 2^ex (every lane of the row): rows
  // differ by more than the double range, and a row that counts for nothing now
  // may count for everything some flips later
  cd wt = {0.0, 0.0};
  int ex = 0;
  double cur2 = 0.0;    // |sum_g wt|^2
  auto refresh = [&]() __attribute__((always_inline)) {
    __syncthreads();
    for (int t = tid; t < G * L; t += nt) rb[t] = row_spin(o, L, s, t / L, t % L);
    __syncthreads();
    const unsigned char* row = rb + rc * L;
    cd li = visible(g, P, row, sl, SL);
    T dp;
    set_one(dp);
#pragma unroll
    for (int k0 = 0; k0 < HT; k0 += 4) {
      cd th[4];
      theta_of<CPX>(g, P, row, h0 + k0, th);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = k0 + j;
        const bool in = h0 + k < H;
        if constexpr (CPX) e[k] = in ? cexp({-2.0 * th[j].re, -2.0 * th[j].im}) : cd{0.0, 0.0};
        else e[k] = in ? exp(-2.0 * th[j].re) : 0.0;
        al[k] = recip(plus1(e[k]));
        // cosh theta = e^{theta} (1 + e) / 2 with |1 + e| <= 2 on the side where |e| <= 1
        const bool neg = th[j].re < 0.0;
        if (in) {
          li = li + (neg ? cd{-th[j].re, -th[j].im} : th[j]);
          dp = mulc(dp, sel(neg, mulc(e[k], al[k]), al[k]));
        }
      }
    }
    for (int m = 1; m < SL; m *= 2) {
      li = li + shfl_xor(li, m);
      dp = mulc(dp, shfl_xor(dp, m));
    }
    const bool on = mine && (b.re != 0.0 || b.im != 0.0);
    double mx = block_max(on ? li.re : -INFINITY, red);
    if (!isfinite(mx)) mx = 0.0;
    const double x = fma(-(double)H, LN2, li.re - mx), k = on ? rint(x * 1.4426950408889634) : 0.0;
    const double xr = fma(-k, 2.31904681384629955842e-17, fma(-k, 6.93147180559945286227e-01, x));
    wt = on ? mulc(mulc(cexp({xr, li.im}), to_cd(recip(dp))), b) : cd{0.0, 0.0};
    ex = (int)k;
    scale_row(wt, ex);
    const cd S = block_sum_cd(sl == 0 ? cd{ldexp(wt.re, ex), ldexp(wt.im, ex)} : cd{0.0, 0.0}, red);
    cur2 = !o.cpx && S.re < 0.0 ? NAN : norm2(S);
  };
  refresh();
  const int total = a.therm_steps + a.samples_per_chain * a.sweep_steps;
  int dsite = 0;
  double du = 0.0;
  int64_t nacc = 0;
  int since = 0, left = a.therm_steps + a.sweep_steps;
  int64_t row_out = chain;
  for (int step = 0; step < total; ++step) {
    const int k64 = step & 63;
    if (k64 == 0 && step + lane < total)
      mc_draw(a.seed, (uint32_t)(step + lane), (uint32_t)chain, a.call_index, a.stream, L, dsite, du);
    const int site = __builtin_amdgcn_readlane(dsite, k64);
    const double u = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(du), k64),
                                      __builtin_amdgcn_readlane(__double2loint(du), k64));
    const int up = (__builtin_amdgcn_readlane((int)sp, site & 63) >> (site >> 6)) & 1;
    const int iv = inv[rc * L + site], pos = iv >> 1, v = up ^ (iv & 1);
    T en[HT], pr;  // e after the flip; (1 + e') / (1 + e) per unit
    set_one(pr);
    const int at = (2 * pos + v) * (TAB ? HP : H);
#pragma unroll
    for (int k = 0; k < HT; ++k) {
      const int hc = min(h0 + k, H - 1);
      if constexpr (TAB) en[k] = mulc(e[k], me[at + hc]);
      else en[k] = mulc(e[k], ((const T*)tab.me)[at + hc]);
      pr = mulc(pr, mulc(al[k], plus1(en[k])));
    }
    for (int m = 1; m < SL; m *= 2) pr = mulc(pr, shfl_xor(pr, m));
    const cd z = mulc(to_cd(pr), mulc(pre[2 * pos + v], wt));
    const double zr = wave_sum(mine && sl == 0 ? ldexp(z.re, ex) : 0.0);
    const double zi = o.cpx ? wave_sum(mine && sl == 0 ? ldexp(z.im, ex) : 0.0) : 0.0;
    cd* slot = part + 16 * (step & 1);
    if (lane == 0) slot[tid / WAVE] = {zr, zi};
    __syncthreads();
    cd S = slot[0];
    for (int i = 1; i < nw; ++i) S = S + slot[i];
    const double new2 = !o.cpx && S.re < 0.0 ? NAN : norm2(S);
    // random.bernoulli(key, P), sampler.py:336-340
    const bool acc = a.mu == 2.0 ? u * cur2 < new2 : u < exp(a.mu * (0.5 * log(new2) - 0.5 * log(cur2)));
    if (acc) {
#pragma unroll
      for (int k = 0; k < HT; ++k) {  // units beyond H: e = 0 stays 0
        e[k] = en[k];
        al[k] = recip(plus1(en[k]));
      }
      const double sc = new2 > 0.0 ? 1.0 / sqrt(new2) : 1.0;
      wt = {z.re * sc, z.im * sc};
      scale_row(wt, ex);
      cur2 = new2 > 0.0 ? 1.0 : 0.0;
      if (lane == (site & 63)) sp ^= 1u << (site >> 6);
    }
    nacc += acc;
    ++since;
    if (--left == 0) {
      left = a.sweep_steps;
      int32_t* out = configs + row_out * L;
      row_out += a.num_chains;
      spins_out();
      for (int i = tid; i < L; i += nt) out[i] = s[i];
      if (since >= RBMQ_MC_REFRESH) {
        refresh();
        since = 0;
      }
    }
  }
  spins_out();
  for (int i = tid; i < L; i += nt) walkers[(int64_t)chain * L + i] = s[i];
  if (tid == 0) {
    atomicAdd((unsigned long long*)&counters[0], (unsigned long long)total);
    atomicAdd((unsigned long long*)&counters[1], (unsigned long long)nacc);
  }
}
size_t sym_mc_lds(const RbmGeom& g, int G, bool tabl) {
  return 8 * 16 + 16 * 32 + 32 * (size_t)g.L + (tabl ? 8 * (size_t)rbm_cw(g) * 2 * g.L * (g.H | 1) : 0) + 4 * (size_t)g.L +
         3 * (size_t)G * g.L + 16;
}

// ------------------------------------------------------------------ parameters out of range, other maps
// log psi of every configuration from scratch (block_logpsi), one configuration
// or chain per workgroup; these kernels return at once where the resident ones
// above work (and the other way round), so neither carries the other's
// registers.  Against a launch per step over materialised rows (4096 samples or
// 1024 chains x 128 proposals, one |Re W| = 90): 16 x 32, 64 elements E_loc
// 17.8 -> 3.9 ms, chains 20.3 -> 5.3; 64 x 200, two elements 30.1 -> 11.2, 8.9
// -> 4.2.
// Few samples: the strings over gridDim.y workgroups each, whose sums [K][n] the
// launch behind adds up (16 samples of 64 x 200, two elements: 1746 us with one
// workgroup a sample, 238 so; 659 with materialised rows).  Without tables
// (tab.site null) it serves every parameter.
template <bool CPX, int U>
__global__ void __launch_bounds__(SYM_T, 2) sym_rows_eloc(RbmGeom g, SymGeom o, const double* __restrict__ P, OpDev op,
                                                          RbmTab tab, int SL, const int32_t* __restrict__ cfg,
                                                          const double* __restrict__ lps, int64_t n,
                                                          double* __restrict__ out) {
  extern __shared__ double lds[];
  if (tab.site && sym_ok(g, o, tab, threadIdx.x % WAVE)) return;
  out += 2 * n * blockIdx.y;
  double* red = lds;
  cd* lin = (cd*)(red + 8);
  cd* dd = lin + o.G;
  int32_t* s = (int32_t*)(dd + o.G);
  unsigned char* rb = (unsigned char*)(s + g.L);
  for (int64_t q = blockIdx.x; q < n; q += gridDim.x) {
    const int32_t* cq = cfg + q * g.L;
    for (int i = threadIdx.x; i < g.L; i += blockDim.x) s[i] = cq[i];
    cd acc = {0.0, 0.0};
    const cd dsum = diag_sum(op, cq);
    for (int j = blockIdx.y; j < op.num_ops; j += gridDim.y) {
      int sites[MAXLEN], vals[MAXLEN], nch;
      const cd m = merged_m(op, j, apply_string(op, j, cq, sites, vals, nch), dsum);
      if (!nonzero(m)) continue;
      __syncthreads();  // s is set
      if (threadIdx.x == 0)
        for (int k = 0; k < nch; ++k) s[sites[k]] = vals[k];
      const cd lp = block_logpsi<CPX, U, 0>(g, o, P, s, SL, lin, dd, rb, red);
      acc = acc + m * cexp(lp - cd{lps[2 * q], lps[2 * q + 1]});
      if (threadIdx.x == 0)
        for (int k = 0; k < nch; ++k) s[sites[k]] = cq[sites[k]];
    }
    if (threadIdx.x == 0) {
      out[2 * q] = acc.re;
      out[2 * q + 1] = acc.im;
    }
    __syncthreads();
  }
}

template <bool CPX, int U>
__global__ void __launch_bounds__(SYM_T, 2) sym_rows_mc(RbmGeom g, SymGeom o, const double* __restrict__ P, jv_mc_args a,
                                                        RbmTab tab, int SL, int32_t* __restrict__ walkers,
                                                        int32_t* __restrict__ configs, int64_t* __restrict__ counters) {
  extern __shared__ double lds[];
  if (sym_ok(g, o, tab, threadIdx.x % WAVE)) return;
  const int tid = threadIdx.x, nt = blockDim.x, chain = blockIdx.x;
  double* red = lds;
  cd* lin = (cd*)(red + 8);
  cd* dd = lin + o.G;
  int32_t* s = (int32_t*)(dd + o.G);
  unsigned char* rb = (unsigned char*)(s + g.L);
  for (int i = tid; i < g.L; i += nt) s[i] = walkers[(int64_t)chain * g.L + i];
  double lacc = a.mu * block_logpsi<CPX, U, 0>(g, o, P, s, SL, lin, dd, rb, red).re;
  const int total = a.therm_steps + a.samples_per_chain * a.sweep_steps;
  int64_t nacc = 0;
  for (int step = 0; step < total; ++step) {
    int site;
    double u;
    mc_draw(a.seed, (uint32_t)step, (uint32_t)chain, a.call_index, a.stream, g.L, site, u);
    if (tid == 0) s[site] ^= 1;
    const double lnew = a.mu * block_logpsi<CPX, U, 0>(g, o, P, s, SL, lin, dd, rb, red).re;
    const bool acc = u < exp(lnew - lacc);
    if (tid == 0 && !acc) s[site] ^= 1;
    if (acc) lacc = lnew;
    nacc += acc;
    const int k = step + 1 - a.therm_steps;
    if (k > 0 && k % a.sweep_steps == 0) {
      __syncthreads();
      for (int i = tid; i < g.L; i += nt)
        configs[((int64_t)(k / a.sweep_steps - 1) * a.num_chains + chain) * g.L + i] = s[i];
      __syncthreads();
    }
  }
  __syncthreads();
  for (int i = tid; i < g.L; i += nt) walkers[(int64_t)chain * g.L + i] = s[i];
  if (tid == 0) {
    atomicAdd((unsigned long long*)&counters[0], (unsigned long long)total);
    atomicAdd((unsigned long long*)&counters[1], (unsigned long long)nacc);
  }
}

__global__ void __launch_bounds__(SYM_T) sym_add_parts(const double* __restrict__ part, int K, int64_t n,
                                                       double* __restrict__ out) {
  for (int64_t q = blockIdx.x * (int64_t)SYM_T + threadIdx.x; q < 2 * n; q += (int64_t)gridDim.x * SYM_T) {
    double v = 0.0;
    for (int k = 0; k < K; ++k) v += part[2 * n * k + q];
    out[q] = v;
  }
}

__global__ void sym_zero_counters(int64_t* c) {
  if (threadIdx.x < 2) c[threadIdx.x] = 0;
}

bool sym_rbm_geom(const jv_net* net, const jv_orbit* orbit, RbmGeom& g, SymGeom& o) {
  if (orbit->avg != JV_AVG_EXP || !make_rbm_geom(net, g)) return false;
  o.G = orbit->num_elements;
  o.cpx = net->is_complex || orbit->complex_factor;
  o.map = orbit->map;
  o.fac = orbit->factor;
  return o.G <= SYM_MAX_G && g.H <= RBMQ_MAX_H && g.L <= RBM_ORBIT_MAX_L;
}

}  // namespace

// Each returns JV_OK with *done = true when the resident form applies (RBM,
// avgFun_Coefficients_Exp, LDS and registers suffice), else *done = false.
int sym_rbm_forward_launch(const jv_net* net, const double* params, const jv_orbit* orbit, const int32_t* configs,
                           int64_t n, double* logpsi, hipStream_t st, bool* done) {
  *done = false;
  RbmGeom g;
  SymGeom o;
  if (!sym_rbm_geom(net, orbit, g, o)) return JV_OK;
  bool four;
  const int SL = sym_lanes(o.G, g.H, &four), T = sym_threads(g, o.G, SL);
  const size_t lds = sym_rows_lds(g, o.G, T, SL);
  if (lds > 160 * 1024) return JV_OK;
  // few configurations of large orbits: rows over the whole chip (three launches;
  // 16 of 96 elements, 24 x 100: 27 us, resident 92; 256: 156 against 94)
  if (std::max(22.0, 10.0 + sym_materialised_us(g, o.G, (double)n)) < 0.9 * (5.0 + sym_resident_us(g, o.G, (double)n)))
    return JV_OK;
#define JV_SYM_FWD(CPX)                                                                  \
  (four ? (SL == 4 ? sym_rbm_forward<CPX, 4, 4> : sym_rbm_forward<CPX, 4, 0>) : sym_rbm_forward<CPX, 1, 0>)
  const auto fn = g.cpx ? JV_SYM_FWD(true) : JV_SYM_FWD(false);
#undef JV_SYM_FWD
  const int rc = set_lds_limit((const void*)fn, lds);
  if (rc) return rc;
  hipLaunchKernelGGL(fn, dim3((unsigned)std::min<int64_t>(n, 1 << 20)), dim3((unsigned)T), lds, st, g, o, params, SL,
                     configs, n, logpsi);
  JV_LAUNCH_CHECK("sym_rbm_forward");
  *done = true;
  return JV_OK;
}

int sym_rbm_eloc_launch(const jv_net* net, const double* params, const jv_orbit* orbit, const jv_optable* op,
                        const double* prefactor, const int32_t* configs, const double* lps, int64_t n, double* out,
                        hipStream_t st, int slot0, int slot1, bool* done) {
  *done = false;
  RbmGeom g;
  SymGeom o;
  if (!sym_rbm_geom(net, orbit, g, o) || op->max_len > 2 || op->fermi || !prefactor) return JV_OK;
  const OpDev d = make_opdev(op, prefactor, net->num_sites);
  const int nstr = rbmq_strings(d);
  // two workgroups per CU, with the table in LDS if that leaves room for rows,
  // then as many rows as fit; else whatever fits one
  int RC = 0;
  bool tabl = false;
  size_t lds = 0;
  for (int pass = 0; pass < 4 && !RC; ++pass)
    for (int rows : {64, 32, 16}) {
      const bool t = pass == 0 || pass == 2;
      const size_t b = sym_eloc_lds(g, rows, t, nstr);
      if (b > (size_t)(pass < 2 ? 80 : 160) * 1024) continue;
      RC = rows;
      tabl = t;
      lds = b;
      break;
    }
  bool four;
  const int SL = sym_lanes(o.G, g.H, &four), T = sym_threads(g, o.G, SL);
  const size_t rlds = sym_rows_lds(g, o.G, T, SL);
  if (!RC || rlds > 160 * 1024) return JV_OK;
  // Times of the three forms: resident (alpha and beta of all rows once, then a
  // product per string), a log psi per string, materialised s' and rows.
  // 4000 samples, one string: 16 x 32, 64 elements 400 / 156 / 564 us, with 16
  // more 453 / - / 17217; 64 x 200, two elements 2056 / 138 / 257, eight strings
  // 2110 / - / 1797; one sample of 24 x 100, 96 elements 352 / 97 / 38.
  const double steps = (double)((o.G + RC - 1) / RC) *
                       ((tabl && !g.cpx ? 0.3 : 0.47) * g.H + 0.2 * g.L * ((g.H + 4 * (SYM_T / RC) - 1) / (4 * (SYM_T / RC))));
  const double t_res = (18.0 + (g.cpx ? 1.0 : 0.5) * steps) * std::max(1.0, n / (lds > 80 * 1024 ? 340.0 : 512.0));
  const int K = n <= 256 ? std::min(d.num_ops, 512 / (int)n) : 1;
  const int kmax = std::min(d.num_ops, nstr + (d.num_diag > 1));  // strings of a sample with a matrix element
  // (every workgroup sums the diagonal strings and looks at its share of all)
  const double t_rows = 8.0 + (d.num_diag > 1 ? 2.2 * d.num_diag : 0.0) + 0.5 * ((d.num_ops + K - 1) / K) +
                        (kmax + K - 1) / K * sym_resident_us(g, o.G, (double)n * K);
  const double N = (double)n * d.num_ops;
  const double t_mat = 28.0 + 2.5 * std::max(0, d.num_ops - 4) +
                       std::min(sym_materialised_us(g, o.G, N), sym_resident_us(g, o.G, N));
  const bool rows = t_rows < 0.9 * t_res;
  if (t_mat < 0.9 * std::min(t_res, t_rows)) return JV_OK;
  RbmTab tab = {};
  int rc = rows ? JV_OK : build_rbm_tables(g, params, &d, false, true, st, slot0, &tab, o.map, o.G);
  if (rc) return rc;
  const auto rf = g.cpx ? (four ? sym_rows_eloc<true, 4> : sym_rows_eloc<true, 1>)
                        : (four ? sym_rows_eloc<false, 4> : sym_rows_eloc<false, 1>);
  if ((rc = set_lds_limit((const void*)rf, rlds))) return rc;
  double* part = K > 1 ? (double*)capturable_workspace(16 * (size_t)K * n, slot1, st) : out;
  if (!part) return fail(JV_E_NOMEM, "jv_sym_eloc: workspace allocation failed");
  hipLaunchKernelGGL(rf, dim3((unsigned)std::min<int64_t>(n, 512 * SYM_T / T), (unsigned)K), dim3((unsigned)T), rlds, st,
                     g, o, params, d, tab, SL, configs, lps, n, part);
  JV_LAUNCH_CHECK("sym_rows_eloc");
  if (rows) {
    if (K > 1) {
      hipLaunchKernelGGL(sym_add_parts, dim3((unsigned)((2 * n + SYM_T - 1) / SYM_T)), dim3(SYM_T), 0, st, part, K, n, out);
      JV_LAUNCH_CHECK("sym_add_parts");
    }
    *done = true;
    return JV_OK;
  }
#define JV_SYM_ELO(RCv)                                                                           \
  (g.cpx ? (tabl ? sym_rbm_eloc<true, RCv, true> : sym_rbm_eloc<true, RCv, false>)                \
         : (tabl ? sym_rbm_eloc<false, RCv, true> : sym_rbm_eloc<false, RCv, false>))
  const auto fn = RC == 64 ? JV_SYM_ELO(64) : RC == 32 ? JV_SYM_ELO(32) : JV_SYM_ELO(16);
#undef JV_SYM_ELO
  if ((rc = set_lds_limit((const void*)fn, lds))) return rc;
  hipLaunchKernelGGL(fn, dim3((unsigned)std::min<int64_t>(n, 4096)), dim3(SYM_T), lds, st, g, o, params, d, tab, configs,
                     lps, n, nstr, part, K, out);
  JV_LAUNCH_CHECK("sym_rbm_eloc");
  *done = true;
  return JV_OK;
}

int sym_rbm_mc_launch(const jv_net* net, const double* params, const jv_orbit* orbit, const jv_mc_args& a,
                      int32_t* walkers, int32_t* configs, int64_t* counters, hipStream_t st, int slot0, bool* done) {
  *done = false;
  RbmGeom g;
  SymGeom o;
  if (!sym_rbm_geom(net, orbit, g, o) || !rbmq_mc_fits(g)) return JV_OK;
  // hidden units per thread: as many as leave the fewest threads (a power of
  // two of them per row, inside one wave), with registers for 512 threads of
  // eight units or 1024 of four
  int HT = 0, SL = 0;
  for (int ht : {8, 4}) {
    int sl = 1;
    while (sl * ht < g.H) sl *= 2;
    if (!HT && sl <= WAVE && (int64_t)o.G * sl <= (ht == 8 ? 512 : 1024)) {
      HT = ht;
      SL = sl;
    }
  }
  const int64_t most = (1 << 22) - 1;  // workgroups of 1024 threads in a launch (fewer than 2^32 threads)
  if (!HT || a.num_chains > most) return JV_OK;
  const bool tabl = sym_mc_lds(g, o.G, true) <= 64 * 1024;
  const size_t lds = sym_mc_lds(g, o.G, tabl);
  bool four;
  const int rSL = sym_lanes(o.G, g.H, &four), rT = sym_threads(g, o.G, rSL);
  const size_t rlds = sym_rows_lds(g, o.G, rT, rSL);
  if (lds > 160 * 1024 || rlds > 160 * 1024) return JV_OK;
  RbmTab tab;
  int rc = build_rbm_tables(g, params, nullptr, true, false, st, slot0, &tab, o.map, o.G);
  if (rc) return rc;
  const int T = (o.G * SL + WAVE - 1) / WAVE * WAVE;
#define JV_SYM_MC(HTv, Tv)                                                                                \
  (g.cpx ? (tabl ? sym_rbm_mc<true, HTv, Tv, true> : sym_rbm_mc<true, HTv, Tv, false>)                    \
         : (tabl ? sym_rbm_mc<false, HTv, Tv, true> : sym_rbm_mc<false, HTv, Tv, false>))
  const auto fn = HT == 8 ? (T <= 256 ? JV_SYM_MC(8, 256) : JV_SYM_MC(8, 512)) : JV_SYM_MC(4, 1024);
#undef JV_SYM_MC
  rc = set_lds_limit((const void*)fn, lds);
  if (rc) return rc;
  hipLaunchKernelGGL(sym_zero_counters, dim3(1), dim3(64), 0, st, counters);
  JV_LAUNCH_CHECK("sym_zero_counters");
  hipLaunchKernelGGL(fn, dim3((unsigned)a.num_chains), dim3(T), lds, st, g, o, params, a, tab, SL, walkers,
                     configs, counters);
  JV_LAUNCH_CHECK("sym_rbm_mc");
  const auto rf = g.cpx ? (four ? sym_rows_mc<true, 4> : sym_rows_mc<true, 1>)
                        : (four ? sym_rows_mc<false, 4> : sym_rows_mc<false, 1>);
  if ((rc = set_lds_limit((const void*)rf, rlds))) return rc;
  hipLaunchKernelGGL(rf, dim3((unsigned)a.num_chains), dim3((unsigned)rT), rlds, st, g, o, params, a, tab, rSL, walkers,
                     configs, counters);
  JV_LAUNCH_CHECK("sym_rows_mc");
  *done = true;
  return JV_OK;
}

}  // namespace jv
