// RBM amplitude ratios without transcendentals per hidden unit.
//
// With theta_h = b_h + sum_i sigma_i W_ih, alpha_h = 1 / (1 + e^{-2 theta_h})
// and beta_h = 1 - alpha_h = e^{-2 theta_h} alpha_h, flipping the spins of a
// set of sites gives
//   psi(s') / psi(s) = prod_j pre_j prod_h (alpha_h + beta_h prod_j g_jh),
//   g_jh = e^{4 sigma_j W_jh},  pre_j = e^{-2 sigma_j (sum_h W_jh + a_j)},
// (cosh(theta') / cosh(theta) per hidden unit).  g and pre depend on the
// parameters only, so one small launch tabulates them and a ratio costs one
// complex multiply-add and one multiply per hidden unit instead of a complex
// log-cosh (exp, sincos, log1p, atan2).  Both terms of a factor carry full
// relative accuracy, so nothing cancels that does not cancel in cosh(theta').
//
// Range: the routines below are used when |Re theta_h| <= RBMQ_THETA for every
// configuration and sum_h |Re W_ih| + |Re a_i| <= 150 / n for strings of n
// sites (pre_j and the products over units then stay inside the double range);
// the rbmq_*_direct routines serve everything else.  The kernels read the two
// bounds from the table, so no host synchronisation is needed and NaN
// parameters count as out of range.
#pragma once
#include "rbm.hpp"

namespace jv {

constexpr double RBMQ_THETA = 150.0;
// First slots of the tables in stream_workspace, for the local energies and
// the chains (which a step may run on different streams).
constexpr int WS_RBMQ_ELOC = 130, WS_RBMQ_MC = WS_RBMQ_ELOC + WS_STREAMS;
constexpr int RBMQ_MAX_H = 900;  // prod_h (1 + e_h) <= 2^H
constexpr int RBM_ORBIT_MAX_L = 16384;  // sites of an orbit's map (positions in 16 bits)

// Device tables of one parameter vector (and one operator).  Elements of me /
// he are complex for complex networks, real otherwise; index v is the spin
// value (0, 1) of the site before the flip.
struct RbmTab {
  double* me;     // [L][2][H]: g of a flip, for the chains (null: not built)
  double* he;     // [H][L][2]: g of a flip, for the local energies (null: not built)
  double* site;   // [L][8]: |pre|^2 for v = 0, 1; pre for v = 0 (re, im), v = 1; sum_h |Re W_ih| + |Re a_i|
  double* row;    // [H]: |Re b_h| + sum_i |Re W_ih|
  int32_t* lead;  // [0]: count; then 16 * string + followers (strings behind it that flip the same sites)
  int32_t* mark;  // [num_ops]: 1 for merged diagonal strings
  int32_t* perm;  // [orbit elements]: 1 where every site is read once (null: no orbit)
};

__host__ __device__ inline int rbm_cw(const RbmGeom& g) { return g.cpx ? 2 : 1; }
// Doubles of a table set (num_ops = 0: without the operator's lists; G: orbit
// elements to check, 0 without an orbit).
__host__ __device__ inline size_t rbm_tab_doubles(const RbmGeom& g, bool me, bool he, int num_ops, int G = 0) {
  return (size_t)(me + he) * 2 * g.L * g.H * rbm_cw(g) + 8 * (size_t)g.L + g.H + (size_t)num_ops + 1 +
         ((size_t)G + 1) / 2;
}
__host__ __device__ inline RbmTab rbm_tab_at(const RbmGeom& g, double* base, bool me, bool he, int num_ops,
                                             int G = 0) {
  RbmTab t;
  const size_t q = (size_t)2 * g.L * g.H * rbm_cw(g);
  t.me = me ? base : nullptr;
  base += me ? q : 0;
  t.he = he ? base : nullptr;
  base += he ? q : 0;
  t.site = base;
  t.row = base + 8 * (size_t)g.L;
  int32_t* i = (int32_t*)(t.row + g.H);
  t.lead = num_ops > 0 ? i : nullptr;
  t.mark = num_ops > 0 ? i + 1 + num_ops : nullptr;
  t.perm = G > 0 ? i + 2 * ((size_t)num_ops + 1) : nullptr;
  return t;
}
// Workgroups that build a table set: one per site, one per 256 hidden units,
// one for the operator's lists.
__host__ __device__ inline int rbm_tab_blocks(const RbmGeom& g, int num_ops) {
  return g.L + (g.H + 255) / 256 + (num_ops > 0 ? 1 : 0);
}

// Work of workgroup `blk` (256 threads; red: 4 doubles of LDS, wcnt: 4 ints).
__device__ inline void rbm_tab_build(const RbmGeom& g, const double* __restrict__ P, const RbmTab& t,
                                     const OpDev* op, int blk, double* red, int* wcnt) {
  const int tid = threadIdx.x;
  const double* Wr = P + g.ow;
  const double* Wi = P + g.ow + (int64_t)g.L * g.H;
  if (blk < g.L) {
    const int i = blk;
    double sr = 0.0, si = 0.0, sa = 0.0;
    for (int h = tid; h < g.H; h += 256) {
      const double wr = Wr[(int64_t)i * g.H + h], wi = g.cpx ? Wi[(int64_t)i * g.H + h] : 0.0;
      sr += wr;
      si += wi;
      sa += fabs(wr);
      const double up = exp(4.0 * wr), dn = exp(-4.0 * wr);
      if (g.cpx) {
        double s, c;
        sincos(4.0 * wi, &s, &c);
        const cd q1 = {up * c, up * s}, q0 = {dn * c, -(dn * s)};
        if (t.me) {
          ((cd*)t.me)[((int64_t)i * 2 + 0) * g.H + h] = q0;
          ((cd*)t.me)[((int64_t)i * 2 + 1) * g.H + h] = q1;
        }
        if (t.he) {
          ((cd*)t.he)[((int64_t)h * g.L + i) * 2 + 0] = q0;
          ((cd*)t.he)[((int64_t)h * g.L + i) * 2 + 1] = q1;
        }
      } else {
        if (t.me) {
          t.me[((int64_t)i * 2 + 0) * g.H + h] = dn;
          t.me[((int64_t)i * 2 + 1) * g.H + h] = up;
        }
        if (t.he) {
          t.he[((int64_t)h * g.L + i) * 2 + 0] = dn;
          t.he[((int64_t)h * g.L + i) * 2 + 1] = up;
        }
      }
    }
    sr = block_sum(sr, red);
    si = block_sum(si, red);
    sa = block_sum(sa, red);
    if (tid < 2) {
      if (g.oa >= 0) {
        sr += P[g.oa + i];
        si += P[g.oa + g.L + i];
        sa += fabs(P[g.oa + i]);
      }
      const double sg = tid ? 1.0 : -1.0;
      const cd pre = cexp({-2.0 * sg * sr, -2.0 * sg * si});
      double* o = t.site + 8 * (int64_t)i;
      o[tid] = exp(-4.0 * sg * sr);
      o[2 + 2 * tid] = pre.re;
      o[3 + 2 * tid] = pre.im;
      o[6 + tid] = sa;
    }
    return;
  }
  const int nrow = (g.H + 255) / 256;
  if (blk < g.L + nrow) {
    const int h = (blk - g.L) * 256 + tid;
    if (h < g.H) {
      double a = g.ob >= 0 ? fabs(P[g.ob + h]) : 0.0;
      for (int i = 0; i < g.L; ++i) a += fabs(Wr[(int64_t)i * g.H + h]);
      t.row[h] = a;
    }
    return;
  }
  // leaders: runs of consecutive strings with the same sites and maps flip the
  // same spins; the first of every four carries their summed matrix element
  const int n = op->num_ops, ml = op->max_len;
  for (int o = tid; o < n; o += 256) t.mark[o] = 0;
  __syncthreads();
  if (op->num_diag > 1)
    for (int d = tid; d < op->num_diag; d += 256) t.mark[op->diag[d]] = 1;
  __syncthreads();
  auto same = [&](int a, int b) {
    if (t.mark[a] != t.mark[b]) return false;
    for (int k = 0; k < ml; ++k)
      if (op->idx[a * ml + k] != op->idx[b * ml + k] || op->map[2 * (a * ml + k)] != op->map[2 * (b * ml + k)] ||
          op->map[2 * (a * ml + k) + 1] != op->map[2 * (b * ml + k) + 1])
        return false;
    return true;
  };
  int cnt = 0;
  for (int base = 0; base < n; base += 256) {
    const int o = base + tid;
    bool flag = false;
    int fol = 0;
    if (o < n && !t.mark[o]) {
      int pos = 0;
      while (o - pos - 1 >= 0 && same(o, o - pos - 1)) ++pos;
      flag = (pos & 3) == 0;
      if (flag)
        while (fol < 3 && o + fol + 1 < n && same(o, o + fol + 1)) ++fol;
    }
    const uint64_t mask = __ballot(flag);
    const int lane = tid % WAVE, w = tid / WAVE;
    if (lane == 0) wcnt[w] = __popcll(mask);
    __syncthreads();
    int before = 0, tot = 0;
    for (int k = 0; k < 4; ++k) {
      before += k < w ? wcnt[k] : 0;
      tot += wcnt[k];
    }
    if (flag) t.lead[1 + cnt + before + __popcll(mask & ((1ull << lane) - 1ull))] = 16 * o + fol;
    cnt += tot;
    __syncthreads();
  }
  if (tid == 0) t.lead[0] = cnt;
}

int build_rbm_tables(const RbmGeom& g, const double* params, const OpDev* op, bool me, bool he, hipStream_t st,
                     int slot0, RbmTab* out, const int32_t* map = nullptr, int G = 0);

// Whether the products stay in range for strings changing up to `nch` sites
// (same answer in every lane; false for NaN parameters).
__device__ inline bool rbmq_ok(const RbmGeom& g, const RbmTab& t, int nch, int lane) {
  bool ok = true;
  const double lim = 150.0 / nch;
  for (int i = lane; i < g.L; i += WAVE) ok = ok && t.site[8 * (int64_t)i + 6] <= lim;
  for (int h = lane; h < g.H; h += WAVE) ok = ok && t.row[h] <= RBMQ_THETA;
  return __all(ok);
}

// Whether orbit element r reads every site once: perm[r] (workgroup of 256
// threads; bits: one bit per site in LDS).
__device__ inline void rbm_tab_perm(const int32_t* __restrict__ map, int L, int r, int32_t* perm, uint32_t* bits) {
  for (int i = threadIdx.x; i < (L + 31) / 32; i += 256) bits[i] = 0;
  __syncthreads();
  int bad = 0;
  for (int i = threadIdx.x; i < L; i += 256) {
    const int m = map[(int64_t)r * L + i], j = m >= 0 ? m : -1 - m;
    if (j >= L || (atomicOr(&bits[j / 32], 1u << (j % 32)) >> (j % 32) & 1)) bad = 1;
  }
  bad = __syncthreads_or(bad);
  if (threadIdx.x == 0) perm[r] = !bad;
}

// ------------------------------------------------------------------ arithmetic
__device__ inline cd fmac(cd a, cd b, cd c) {
  return {fma(a.re, b.re, fma(-a.im, b.im, c.re)), fma(a.re, b.im, fma(a.im, b.re, c.im))};
}
__device__ inline double fmac(double a, double b, double c) { return fma(a, b, c); }
__device__ inline cd mulc(cd a, cd b) {
  return {fma(a.re, b.re, -(a.im * b.im)), fma(a.re, b.im, a.im * b.re)};
}
__device__ inline double mulc(double a, double b) { return a * b; }
__device__ inline double norm2(cd a) { return fma(a.re, a.re, a.im * a.im); }
__device__ inline double norm2(double a) { return a * a; }
__device__ inline double recip(double d) {
  double q = __builtin_amdgcn_rcp(d);
  q = fma(q, fma(-d, q, 1.0), q);
  return fma(q, fma(-d, q, 1.0), q);
}
__device__ inline cd recip(cd d) {
  const double q = recip(norm2(d));
  return {d.re * q, -(d.im * q)};
}
__device__ inline cd sel(bool c, cd a, cd b) { return {c ? a.re : b.re, c ? a.im : b.im}; }
__device__ inline double sel(bool c, double a, double b) { return c ? a : b; }
__device__ inline cd to_cd(cd a) { return a; }
__device__ inline cd to_cd(double a) { return {a, 0.0}; }
template <bool CPX>
struct num_of { typedef double type; };
template <>
struct num_of<true> { typedef cd type; };
__device__ inline void set_one(cd& a) { a = {1.0, 0.0}; }
__device__ inline void set_one(double& a) { a = 1.0; }
__device__ inline cd plus1(cd a) { return {1.0 + a.re, a.im}; }
__device__ inline double plus1(double a) { return 1.0 + a; }

// Wave-wide product in a fixed order, the value in every lane (wave_sum's lane
// moves with 1 for lanes without a source).
template <int CTRL, int ROWS>
__device__ inline double dpp_shift1(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0x3ff00000, __double2hiint(v), CTRL, ROWS, 0xf, false);
  return __hiloint2double(hi, lo);
}
template <int CTRL, int ROWS>
__device__ inline cd dpp_shift1(cd v) {
  return {dpp_shift1<CTRL, ROWS>(v.re), dpp_shift<CTRL, ROWS>(v.im)};
}
__device__ inline double lane63(double v) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), 63);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), 63);
  return __hiloint2double(hi, lo);
}
__device__ inline cd lane63(cd v) { return {lane63(v.re), lane63(v.im)}; }
template <typename T>
__device__ inline T wave_prod(T v) {
  v = mulc(v, dpp_shift1<0x111, 0xf>(v));
  v = mulc(v, dpp_shift1<0x112, 0xf>(v));
  v = mulc(v, dpp_shift1<0x114, 0xf>(v));
  v = mulc(v, dpp_shift1<0x118, 0xf>(v));
  v = mulc(v, dpp_shift1<0x142, 0xa>(v));
  v = mulc(v, dpp_shift1<0x143, 0xc>(v));
  return lane63(v);
}

__device__ inline double shfl_xor(double v, int m) { return __shfl_xor(v, m); }
__device__ inline cd shfl_xor(cd v, int m) { return {__shfl_xor(v.re, m), __shfl_xor(v.im, m)}; }

// e^{-2 |theta|} side of one hidden unit: alpha, beta; `lin` = theta with the
// sign that makes its real part >= 0 and `d` = 1 + e^{-2 lin}, so that
// cosh(theta) = e^{lin} d / 2.
__device__ inline void rbm_ab(cd th, cd& al, cd& be, cd& lin, cd& d) {
  const bool neg = th.re < 0.0;
  lin = neg ? cd{-th.re, -th.im} : th;
  const cd e = cexp({-2.0 * lin.re, -2.0 * lin.im});
  d = plus1(e);
  const cd inv = recip(d), ei = mulc(e, inv);
  al = sel(neg, ei, inv);
  be = sel(neg, inv, ei);
}
__device__ inline void rbm_ab(double th, double& al, double& be, double& lin, double& d) {
  const bool neg = th < 0.0;
  lin = fabs(th);
  const double e = exp(-2.0 * lin);
  d = 1.0 + e;
  const double inv = recip(d), ei = e * inv;
  al = neg ? ei : inv;
  be = neg ? inv : ei;
}

// ------------------------------------------------------------------ local energies
// A workgroup of four waves evaluates a tile of samples together: eight where
// that leaves four workgroups per CU (n >= 8192: 67 against 81 us with four at
// 16384 samples of 32 sites x 64 units), else four (49.5 against 57.7 us at 3000
// samples of 45 x 90), and two for more than 256 hidden units, whose alpha,
// beta would not fit otherwise.  A sample's result does not depend on it.
constexpr int RBMQ_WAVES = 4;
__host__ __device__ inline int rbmq_tile(const RbmGeom& g, int64_t n) {
  return g.H > 256 ? 2 : (n >= 8192 ? 8 : 4);
}
// Strings of one pass: the smallest power of two >= n, at most a wave.
__host__ __device__ inline int rbmq_jp(int n) {
  int jp = WAVE;
  while (jp > 1 && jp / 2 >= n) jp /= 2;
  return jp;
}
// Few strings on few samples: the log-cosh form's one launch is over before the
// ratio form's table is (one Sx on 1000 samples of 16 x 32: 15.8 against 18.6
// us a call, on 5000 24.9 against 27.2, on 20000 81.8 against 58.5; three on
// 5000 40.1 against 26.2; real 21.6 against 25.4 for one on 5000).  Work is
// counted in strings times units a lane, whose log-cosh costs a complex network
// three times a real one's.  A real network's two-sample tiles do not pay for a
// single string at any size (8 x 300, 100000 samples: 487 against 526 us).
__host__ __device__ inline bool rbmq_eloc_small(const RbmGeom& g, int num_ops, int64_t n) {
  const int64_t w = (int64_t)num_ops * ((g.H + WAVE - 1) / WAVE);
  if (!g.cpx && g.H > 256 && num_ops == 1) return true;
  return w <= (g.cpx ? 3 : 10) && n * w <= (g.cpx ? 6000 : 12000);
}
// LDS doubles of the workgroup, for at most `nstr` strings per sample: alpha,
// beta; psi(s) / e^{lps}; matrix elements and per-wave products of a pass;
// spins; one flag.
__host__ __device__ inline size_t rbmq_eloc_lds_doubles(const RbmGeom& g, int nstr, int64_t n) {
  const size_t S = rbmq_tile(g, n), jp = rbmq_jp(nstr), cw = rbm_cw(g);
  return S * (2 * cw * g.H + 2 + 2 * jp + RBMQ_WAVES * cw * jp + (g.L + 1) / 2) + 2;
}
// ... of any form.
__host__ __device__ inline size_t rbmq_block_lds_doubles(const RbmGeom& g, int nstr, int64_t n) {
  const size_t log_form = (size_t)RBMQ_WAVES * 4 * g.H;
  if (g.H > RBMQ_MAX_H) return log_form;
  const size_t q = rbmq_eloc_lds_doubles(g, nstr, n);
  return q > log_form ? q : log_form;
}

// String o of at most two factors on configuration c: matrix element (unmerged)
// and whether each factor's site ends flipped.
__device__ inline cd string2(const OpDev& op, int o, const int32_t* c, bool& fa, bool& fb) {
  cd m = {op.pref[2 * o], op.pref[2 * o + 1]};
  const int base = o * op.max_len;
  const int i0 = min(max(op.idx[base], 0), op.L - 1);
  const int c0 = min(max(c[i0], 0), 1);
  m = m * cd{op.matel[2 * (2 * base + c0)], op.matel[2 * (2 * base + c0) + 1]};
  const int n0 = min(max(op.map[2 * base + c0], 0), 1);
  fa = n0 != c[i0];
  fb = false;
  if (op.max_len > 1) {
    const int i1 = min(max(op.idx[base + 1], 0), op.L - 1);
    const int c1 = i1 == i0 ? n0 : min(max(c[i1], 0), 1);
    m = m * cd{op.matel[2 * (2 * (base + 1) + c1)], op.matel[2 * (2 * (base + 1) + c1) + 1]};
    const int n1 = min(max(op.map[2 * (base + 1) + c1], 0), 1);
    fb = n1 != c[i1];
    if (i1 == i0) fa = false;  // the site's final value is the second factor's
  }
  return m;
}

// O_loc (base.py:162-192) of samples [0, ns), ns <= S, by one workgroup of
// RBMQ_WAVES waves.  Per string, hidden unit and sample: eight FP64 operations
// and two 16-byte LDS reads (one address per wave: broadcast).  Lanes own
// strings and loop over hidden units, split over the waves and, where strings
// leave lanes free, over lane groups, so a string needs no wave reduction; S
// samples share each read of the g table, which would otherwise be the bound
// (64 KB per sample for 32 sites x 64 units).  Everything else (theta, matrix
// elements, sums over strings) belongs to the wave that owns the sample.  The
// order of every sum and product depends on the sizes only, not on ns or on
// which samples share a workgroup.
// Measured (tables included): 16384 samples of 32 sites x 64 units, Ising
// chain, 2042 -> 65 us; 3000 samples of 45 x 90, XXZ chain (90 two-site
// strings, the X X and Y Y of a bond sharing one ratio), 1430 -> 49 us.  Vector
// issue takes 65 % of the time (3200 instructions per wave and tile), bank
// conflicts 4 %.
// SMALL: strings of at most two factors without Jordan-Wigner signs.
template <bool CPX, bool SMALL, int S>
__device__ inline void rbmq_eloc_tile(const RbmGeom& g, const double* __restrict__ P, const OpDev& op,
                                      const RbmTab& tab, const int32_t* __restrict__ cfg, int ns, int nstr,
                                      const double* __restrict__ lps, double* __restrict__ out, double* lds,
                                      int lane, int w) {
  typedef typename num_of<CPX>::type T;
  constexpr int SPW = (S + RBMQ_WAVES - 1) / RBMQ_WAVES;  // samples owned by a wave: w, w + 4, ...
  const int L = g.L, H = g.H;
  const int nl = tab.lead[0];
  const int jp = rbmq_jp(nstr);  // nstr >= nl: also the LDS layout's
  T* ab = (T*)lds;                              // [sample][h][2]
  cd* amp = (cd*)(ab + (size_t)S * 2 * H);      // [sample]
  cd* mel = amp + S;                            // [sample][jp]
  T* part = (T*)(mel + (size_t)S * jp);         // [wave][sample][jp]
  int32_t* sp = (int32_t*)(part + (size_t)RBMQ_WAVES * S * jp);  // [sample][L]
  int32_t* odd = sp + 2 * (size_t)S * ((L + 1) / 2);
  __syncthreads();  // the previous tile is done
  for (int s = w; s < S; s += RBMQ_WAVES)
    for (int i = lane; i < L; i += WAVE) sp[s * L + i] = cfg[(int64_t)min(s, ns - 1) * L + i];
  if (threadIdx.x == 0) *odd = 0;
  __syncthreads();  // the clear comes before any wave's set in the first pass
  // hidden units of the wave's samples: lane = unit
  const double* Wr = P + g.ow;
  const double* Wi = Wr + (int64_t)L * H;
  cd acc[SPW];
#pragma unroll
  for (int k = 0; k < SPW; ++k) acc[k] = {0.0, 0.0};
  // (S < RBMQ_WAVES: the waves without a sample skip this)
  if (S >= RBMQ_WAVES || w < S) {
    double lin_re[SPW] = {}, lin_im[SPW] = {};
    T dprod[SPW];
#pragma unroll
    for (int k = 0; k < SPW; ++k) set_one(dprod[k]);
    for (int h0 = 0; h0 < H; h0 += WAVE) {
      const int h = h0 + lane, hc = min(h, H - 1);
      cd th[SPW];
      cd b = {0.0, 0.0};
      if (g.ob >= 0) {
        b.re = P[g.ob + hc];
        if (CPX) b.im = P[g.ob + H + hc];
      }
#pragma unroll
      for (int k = 0; k < SPW; ++k) th[k] = b;
      for (int i0 = 0; i0 < L; i0 += WAVE) {
        uint64_t up[SPW];  // bit i: spin i0 + i is up
#pragma unroll
        for (int k = 0; k < SPW; ++k) {
          const int s = min(w + k * RBMQ_WAVES, S - 1);
          up[k] = __ballot(i0 + lane < L && sp[s * L + min(i0 + lane, L - 1)] > 0);
        }
        const int ni = min(WAVE, L - i0);
#pragma unroll 8
        for (int i = 0; i < ni; ++i) {
          const int64_t wi = (int64_t)(i0 + i) * H + hc;
          const double wr = Wr[wi], wm = CPX ? Wi[wi] : 0.0;
#pragma unroll
          for (int k = 0; k < SPW; ++k) {
            const double sg = (up[k] >> i) & 1 ? 1.0 : -1.0;
            th[k].re = fma(sg, wr, th[k].re);
            if (CPX) th[k].im = fma(sg, wm, th[k].im);
          }
        }
      }
      if (h < H) {
#pragma unroll
        for (int k = 0; k < SPW; ++k) {
          const int s = w + k * RBMQ_WAVES;
          T al, be, lin, d;
          if constexpr (CPX) {
            rbm_ab(th[k], al, be, lin, d);
            lin_re[k] += lin.re;
            lin_im[k] += lin.im;
          } else {
            rbm_ab(th[k].re, al, be, lin, d);
            lin_re[k] += lin;
          }
          dprod[k] = mulc(dprod[k], d);
          if (s < S) {
            ab[((size_t)s * H + h) * 2] = al;
            ab[((size_t)s * H + h) * 2 + 1] = be;
          }
        }
      }
    }
    // psi(s) / e^{log psi given by the caller} (base.py:164) and the merged
    // diagonal string (branch_free.py:483-485)
#pragma unroll
    for (int k = 0; k < SPW; ++k) {
      const int s = min(w + k * RBMQ_WAVES, S - 1), sc = min(s, ns - 1);
      double vr = lin_re[k], vi = lin_im[k];
      if (g.oa >= 0) {
        for (int i = lane; i < L; i += WAVE) {
          const double sg = (double)(2 * sp[s * L + i] - 1);
          vr = fma(sg, P[g.oa + i], vr);
          vi = fma(sg, P[g.oa + L + i], vi);
        }
      }
      // explicit fma: H * LN2 hoisted out of a loop over tiles would round differently
      const cd x = {fma(-(double)H, LN2, wave_sum(vr)) - lps[2 * sc], wave_sum(vi) - lps[2 * sc + 1]};
      const cd a = mulc(to_cd(wave_prod(dprod[k])), cexp(x));
      if (lane == 0) amp[s] = a;
      if (op.num_diag > 1) {
        cd ds = {0.0, 0.0};
        for (int d = lane; d < op.num_diag; d += WAVE) {
          if constexpr (SMALL) {
            bool fa, fb;
            ds = ds + string2(op, op.diag[d], sp + s * L, fa, fb);
          } else {
            int sites[MAXLEN], vals[MAXLEN], nch;
            ds = ds + apply_string(op, op.diag[d], sp + s * L, sites, vals, nch);
          }
        }
        ds = {wave_sum(ds.re), wave_sum(ds.im)};
        if (lane == 0 && nonzero(ds)) acc[k] = mulc(ds, a);
      }
    }
  }
  const T* he = (const T*)tab.he;
  const int nsl = RBMQ_WAVES * (WAVE / jp), sl = w * (WAVE / jp) + lane / jp;
  for (int j0 = 0; j0 < nl; j0 += jp) {
    const int j = j0 + lane % jp;
    const bool have = j < nl;
    const int code = have ? tab.lead[1 + j] : 0;
    const int o = code >> 4, fol = code & 15;
    bool general = !SMALL;
    if constexpr (SMALL) {
      // sites whose spin the string can change (identity factors pad shorter strings)
      const int base = o * op.max_len;
      int sa = -1, sb = -1;
      for (int k = 0; k < op.max_len; ++k)
        if (op.map[2 * (base + k)] != 0 || op.map[2 * (base + k) + 1] != 1) {
          const int i = min(max(op.idx[base + k], 0), L - 1);
          if (sa < 0) sa = i;
          else sb = i;
        }
      // matrix elements of the wave's samples (lane groups take one sample each)
      for (int k = lane / jp; k < SPW; k += WAVE / jp) {
        const int s = w + k * RBMQ_WAVES;
        if (s >= S) break;
        const int32_t* c = sp + s * L;
        cd m = {0.0, 0.0};
        if (have)
          for (int f = 0; f <= fol; ++f) {
            bool fa, fb;
            const cd mf = string2(op, o + f, c, fa, fb);
            if (nonzero(mf)) {
              m = m + mf;
              // a changing factor that leaves its site: the general loop below
              // (a padding identity on the changed site reports the change as its own)
              if (sb >= 0 ? !(fa && fb && sa != sb) : sa >= 0 && !(fa || fb)) *odd = 1;
            }
          }
        mel[s * jp + lane % jp] = m;
      }
      __syncthreads();
      general = *odd != 0;
      if (!general) {
        T pr[S];
        bool va[S], vb[S];
        const int la = max(sa, 0), lb = max(sb, 0);
#pragma unroll
        for (int s = 0; s < S; ++s) {
          set_one(pr[s]);
          va[s] = sp[s * L + la] > 0;
          vb[s] = sp[s * L + lb] > 0;
        }
        if (__any(sb >= 0)) {
#pragma unroll 2
          for (int h = sl; h < H; h += nsl) {
            const T* qa = he + ((int64_t)h * L + la) * 2;
            const T* qb = he + ((int64_t)h * L + lb) * 2;
            const T a0 = qa[0], a1 = qa[1];
            T b0 = qb[0], b1 = qb[1], one;
            set_one(one);
            b0 = sel(sb >= 0, b0, one);
            b1 = sel(sb >= 0, b1, one);
#pragma unroll
            for (int s = 0; s < S; ++s) {
              const T* p = ab + ((size_t)s * H + h) * 2;
              pr[s] = mulc(pr[s], fmac(p[1], mulc(sel(va[s], a1, a0), sel(vb[s], b1, b0)), p[0]));
            }
          }
        } else {
#pragma unroll 4
          for (int h = sl; h < H; h += nsl) {
            const T* qa = he + ((int64_t)h * L + la) * 2;
            const T a0 = qa[0], a1 = qa[1];
#pragma unroll
            for (int s = 0; s < S; ++s) {
              const T* p = ab + ((size_t)s * H + h) * 2;
              pr[s] = mulc(pr[s], fmac(p[1], sel(va[s], a1, a0), p[0]));
            }
          }
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
          T r = pr[s];
          for (int off = jp; off < WAVE; off *= 2) r = mulc(r, shfl_xor(r, off));
          if (lane < jp) part[((size_t)w * S + s) * jp + lane] = r;
        }
        __syncthreads();
        // ratios of the wave's samples, summed over strings per lane
#pragma unroll
        for (int k = 0; k < SPW; ++k) {
          const int s = w + k * RBMQ_WAVES;
          if (s < S && lane < jp) {
            const cd m = mel[s * jp + lane];
            // a string that does not apply to this sample adds nothing
            if (have && (m.re != 0.0 || m.im != 0.0)) {
              cd r = {1.0, 0.0};
              if (sa >= 0) {
                T t = part[(size_t)s * jp + lane];
#pragma unroll
                for (int q = 1; q < RBMQ_WAVES; ++q) t = mulc(t, part[((size_t)q * S + s) * jp + lane]);
                const double* pa = tab.site + 8 * (int64_t)sa + 2 + 2 * (int)(sp[s * L + sa] > 0);
                r = mulc(to_cd(t), cd{pa[0], pa[1]});
                if (sb >= 0) {
                  const double* pb = tab.site + 8 * (int64_t)sb + 2 + 2 * (int)(sp[s * L + sb] > 0);
                  r = mulc(r, cd{pb[0], pb[1]});
                }
              }
              acc[k] = acc[k] + mulc(m, mulc(r, amp[s]));
            }
          }
        }
      }
    } else {
      if (j0 == 0) __syncthreads();  // alpha, beta and amp of this wave's samples only: order LDS
    }
    if (general) {
      // any string: sites and matrix element per sample, all hidden units in one lane
#pragma unroll
      for (int k = 0; k < SPW; ++k) {
        const int s = w + k * RBMQ_WAVES;
        if (s < S && have && lane < jp) {
          for (int f = 0; f <= fol; ++f) {
            int sites[MAXLEN], vals[MAXLEN], nch;
            const cd m = apply_string(op, o + f, sp + s * L, sites, vals, nch);
            if (!nonzero(m)) continue;
            T pr;
            set_one(pr);
            for (int h = 0; h < (nch > 0 ? H : 0); ++h) {
              T q;
              set_one(q);
              for (int c = 0; c < nch; ++c)
                q = mulc(q, he[((int64_t)h * L + sites[c]) * 2 + (sp[s * L + sites[c]] > 0)]);
              const T* p = ab + ((size_t)s * H + h) * 2;
              pr = mulc(pr, fmac(p[1], q, p[0]));
            }
            cd r = to_cd(pr);
            for (int c = 0; c < nch; ++c) {
              const double* pa = tab.site + 8 * (int64_t)sites[c] + 2 + 2 * (sp[s * L + sites[c]] > 0);
              r = mulc(r, cd{pa[0], pa[1]});
            }
            acc[k] = acc[k] + mulc(m, mulc(r, amp[s]));
          }
        }
      }
    }
    if (j0 + jp < nl) {
      __syncthreads();
      if (threadIdx.x == 0) *odd = 0;
      __syncthreads();
    }
  }
#pragma unroll
  for (int k = 0; k < SPW; ++k) {
    const int s = w + k * RBMQ_WAVES;
    const double er = wave_sum(acc[k].re), ei = wave_sum(acc[k].im);
    if (lane == 0 && s < ns) {
      out[2 * s] = er;
      out[2 * s + 1] = ei;
    }
  }
}

// theta of unit h for the spins s and its value on the side where Re >= 0;
// d = 1 + e^{-2 lin}, so that cosh(theta) = e^{lin} d / 2.
__device__ inline void rbm_lin(cd th, cd& lin, cd& d) {
  lin = th.re < 0.0 ? cd{-th.re, -th.im} : th;
  d = plus1(cexp({-2.0 * lin.re, -2.0 * lin.im}));
}
__device__ inline void rbm_lin(double th, double& lin, double& d) {
  lin = fabs(th);
  d = 1.0 + exp(-2.0 * lin);
}

// O_loc of one sample by one wave for parameters out of the ratio form's range:
// psi(s') = e^{sum lin'} prod d' per string, an exponential per hidden unit and
// no logarithm (H <= RBMQ_MAX_H keeps the product in range whatever theta).
// 2000 samples of 100 x 200: 3.0 ms with rbm.hpp's log-cosh form inside this
// kernel, whose registers and LDS leave it half the waves, 1.53 so (1.74 in
// eloc_rbm).  th: H complex (real) of LDS.
template <bool CPX>
__device__ inline void rbmq_eloc_direct(const RbmGeom& g, const double* __restrict__ P, const OpDev& op,
                                        const int32_t* c, const double* lps_s, double* out_s, double* lds, int lane) {
  typedef typename num_of<CPX>::type T;
  T* th = (T*)lds;
  const double* Wr = P + g.ow;
  const double* Wi = Wr + (int64_t)g.L * g.H;
  T lin0, prod;
  set_one(prod);
  lin0 = prod - prod;
  wave_sync();  // the previous sample is done
  for (int h = lane; h < g.H; h += WAVE) {
    const cd t = rbm_theta(g, P, c, h);
    T x, lin, d;
    if constexpr (CPX) x = t;
    else x = t.re;
    th[h] = x;
    rbm_lin(x, lin, d);
    lin0 = lin0 + lin;
    prod = mulc(prod, d);
  }
  cd base = to_cd(lin0);
  if (g.oa >= 0)
    for (int i = lane; i < g.L; i += WAVE) {
      const double sg = (double)(2 * c[i] - 1);
      base.re = fma(sg, P[g.oa + i], base.re);
      base.im = fma(sg, P[g.oa + g.L + i], base.im);
    }
  // e^{base} prod d = psi(s) / e^{log psi given by the caller} (base.py:164)
  base = {fma(-(double)g.H, LN2, wave_sum(base.re)) - lps_s[0], wave_sum(base.im) - lps_s[1]};
  const T prod0 = wave_prod(prod);
  wave_sync();
  const cd dsum = diag_sum(op, c);
  cd acc = {0.0, 0.0};
  int sites[MAXLEN], vals[MAXLEN], nch;
  for (int o = 0; o < op.num_ops; ++o) {
    const cd m = merged_m(op, o, apply_string(op, o, c, sites, vals, nch), dsum);
    if (!nonzero(m)) continue;
    cd x = base;
    T dp = prod0;
    if (nch > 0) {
      T dl;
      set_one(dp);
      dl = dp - dp;
      for (int h = lane; h < g.H; h += WAVE) {
        const T t0 = th[h];
        cd t = to_cd(t0);
        for (int j = 0; j < nch; ++j) {
          const double f = 2.0 * (double)(vals[j] - c[sites[j]]);
          const int64_t wi = (int64_t)sites[j] * g.H + h;
          t.re = fma(f, Wr[wi], t.re);
          if (CPX) t.im = fma(f, Wi[wi], t.im);
        }
        T lin, d, l0;
        if constexpr (CPX) {
          rbm_lin(t, lin, d);
          l0 = t0.re < 0.0 ? cd{-t0.re, -t0.im} : t0;
        } else {
          rbm_lin(t.re, lin, d);
          l0 = fabs(t0);
        }
        dl = dl + (lin - l0);
        dp = mulc(dp, d);
      }
      const cd dc = to_cd(dl);
      x.re += wave_sum(dc.re);
      if (CPX) x.im += wave_sum(dc.im);
      dp = wave_prod(dp);
      if (g.oa >= 0)
        for (int j = 0; j < nch; ++j) {
          const double f = 2.0 * (double)(vals[j] - c[sites[j]]);
          x.re = fma(f, P[g.oa + sites[j]], x.re);
          x.im = fma(f, P[g.oa + g.L + sites[j]], x.im);
        }
    }
    acc = acc + mulc(m, mulc(to_cd(dp), cexp(x)));
  }
  if (lane == 0) {
    out_s[0] = acc.re;
    out_s[1] = acc.im;
  }
}

// Samples [s0, s0 + cnt) by one workgroup of RBMQ_WAVES waves, S at a time:
// the ratio form where the parameters' range allows it, string by string
// otherwise (S = 0: rbm.hpp's log-cosh form always).
template <bool CPX, bool SMALL, int S>
__device__ inline void rbmq_eloc_range(const RbmGeom& g, const double* __restrict__ P, const OpDev& op,
                                       const RbmTab& tab, const int32_t* __restrict__ cfg, int64_t s0, int64_t cnt,
                                       int nstr, const double* __restrict__ lps, double* __restrict__ out,
                                       double* lds) {
  const int lane = threadIdx.x % WAVE, w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  if constexpr (S > 0) {
    if (__builtin_expect(rbmq_ok(g, tab, max(2, op.max_len), lane), 1)) {
      for (int64_t k = 0; k < cnt; k += S) {
        const int64_t s = s0 + k;
        rbmq_eloc_tile<CPX, SMALL, S>(g, P, op, tab, cfg + s * g.L, (int)min((int64_t)S, cnt - k), nstr, lps + 2 * s,
                                      out + 2 * s, lds, lane, w);
      }
      return;
    }
    for (int64_t k = w; k < cnt; k += RBMQ_WAVES)
      rbmq_eloc_direct<CPX>(g, P, op, cfg + (s0 + k) * g.L, lps + 2 * (s0 + k), out + 2 * (s0 + k),
                            lds + (size_t)w * rbm_cw(g) * g.H, lane);
    return;
  }
  for (int64_t k = w; k < cnt; k += RBMQ_WAVES)
    eloc_rbm_sample(g, P, op, cfg + (s0 + k) * g.L, lps + 2 * (s0 + k), out + 2 * (s0 + k),
                    (cd*)lds + (size_t)w * 2 * g.H, lane);
}
// Strings that rbmq_eloc_tile may meet per sample (the merged diagonal ones aside).
__host__ __device__ inline int rbmq_strings(const OpDev& op) {
  const int n = op.num_ops - (op.num_diag > 1 ? op.num_diag : 0);
  return n > 1 ? n : 1;
}

// ------------------------------------------------------------------ Metropolis chains
constexpr int RBMQ_MC_MAX_H = 256, RBMQ_MC_MAX_L = 2048;
constexpr int RBMQ_MC_REFRESH = 128;  // proposals after which an emission recomputes theta
__host__ __device__ inline bool rbmq_mc_fits(const RbmGeom& g) {
  return g.H <= RBMQ_MC_MAX_H && g.L <= RBMQ_MC_MAX_L;
}

// Metropolis chain `chain` of MCSampler._get_samples_mcmc / _sweep
// (sampler.py:264-367) by one wavefront, lane = hidden unit (NH units per
// lane, H <= 64 NH); returns the accepted proposals (every lane).  A proposal
// is |psi(s') / psi(s)|^2 = |pre|^2 prod_h |alpha + beta g|^2 against the
// uniform number.  One wave's issue and latency set its time (1024 chains are
// one wave per SIMD): the sites of 64 proposals are drawn at once, so g and pre
// are loaded four proposals ahead (502 us with one ahead), the spins sit in a register per lane
// (bit w of lane l: site 64 w + l), and the accepted state e' = e g, alpha' =
// 1 / (1 + e') is formed beside the wave product, before the decision.
// e = e^{-2 theta} is updated by products (relative error only) and recomputed
// from the weights at emissions at least RBMQ_MC_REFRESH proposals apart.
// 1024 chains x 1312 proposals, 32 sites x 64 units: 2080 us with a complex
// log-cosh per unit and proposal, 428 us here (0.33 us and 64 vector
// instructions per proposal, 38 % of the issue cycles).
template <bool CPX, int NH>
__device__ inline int64_t rbmq_mc_chain(const RbmGeom& g, const double* __restrict__ P, const jv_mc_args& a,
                                        const RbmTab& tab, int32_t* __restrict__ walkers,
                                        int32_t* __restrict__ configs, int chain, int lane) {
  typedef typename num_of<CPX>::type T;
  const int L = g.L, H = g.H, words = (L + WAVE - 1) / WAVE;
  const double* Wr = P + g.ow;
  const double* Wi = Wr + (int64_t)L * H;
  const T* me = (const T*)tab.me;
  uint32_t sp = 0;
  for (int w = 0; w < words; ++w) {
    const int i = w * WAVE + lane;
    if (i < L && walkers[(int64_t)chain * L + i] > 0) sp |= 1u << w;
  }
  T e[NH], al[NH], be[NH];
  auto refresh = [&]() {
    cd th[NH];
#pragma unroll
    for (int c = 0; c < NH; ++c) {
      const int hc = min(c * WAVE + lane, H - 1);
      th[c] = {0.0, 0.0};
      if (g.ob >= 0) {
        th[c].re = P[g.ob + hc];
        if (CPX) th[c].im = P[g.ob + H + hc];
      }
    }
    for (int w = 0; w < words; ++w) {
      const uint64_t up = __ballot((sp >> w) & 1);
      const int ni = min(WAVE, L - w * WAVE);
#pragma unroll 8
      for (int i = 0; i < ni; ++i) {
        const double sg = (up >> i) & 1 ? 1.0 : -1.0;
#pragma unroll
        for (int c = 0; c < NH; ++c) {
          const int64_t wi = (int64_t)(w * WAVE + i) * H + min(c * WAVE + lane, H - 1);
          th[c].re = fma(sg, Wr[wi], th[c].re);
          if (CPX) th[c].im = fma(sg, Wi[wi], th[c].im);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < NH; ++c) {
      const bool in = c * WAVE + lane < H;
      if constexpr (CPX) e[c] = in ? cexp({-2.0 * th[c].re, -2.0 * th[c].im}) : cd{0.0, 0.0};
      else e[c] = in ? exp(-2.0 * th[c].re) : 0.0;
      al[c] = recip(plus1(e[c]));
      be[c] = mulc(e[c], al[c]);
    }
  };
  refresh();
  const int total = a.therm_steps + a.samples_per_chain * a.sweep_steps;
  int dsite = 0;
  double du = 0.0;
  auto batch = [&](int base) {
    if (base + lane < total)
      mc_draw(a.seed, (uint32_t)(base + lane), (uint32_t)chain, a.call_index, a.stream, L, dsite, du);
  };
  // g and |pre|^2 of the next AHEAD proposals, for either spin
  constexpr int AHEAD = NH == 1 ? 4 : 2;
  T q0[AHEAD][NH], q1[AHEAD][NH];
  double p0[AHEAD], p1[AHEAD];
  int sites[AHEAD];
  double us[AHEAD];
  auto fetch = [&](int d, int step) {
    if (step < total && (step & 63) == 0) batch(step);
    const int site = __builtin_amdgcn_readlane(dsite, step & 63);
    sites[d] = site;
    us[d] = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(du), step & 63),
                             __builtin_amdgcn_readlane(__double2loint(du), step & 63));
#pragma unroll
    for (int c = 0; c < NH; ++c) {
      const int64_t at = (int64_t)site * 2 * H + min(c * WAVE + lane, H - 1);
      q0[d][c] = me[at];
      q1[d][c] = me[at + H];
    }
    p0[d] = tab.site[8 * (int64_t)site];
    p1[d] = tab.site[8 * (int64_t)site + 1];
  };
#pragma unroll
  for (int d = 0; d < AHEAD; ++d) fetch(d, d);
  int64_t nacc = 0;
  int since = 0, left = a.therm_steps + a.sweep_steps;
  int64_t row = chain;
  for (int step0 = 0; step0 < total; step0 += AHEAD) {
#pragma unroll
    for (int d = 0; d < AHEAD; ++d) {
      const int step = step0 + d;
      if (step >= total) break;
      const double u = us[d];
      const int wd = sites[d] >> 6, ln = sites[d] & 63;
      const bool up = (__builtin_amdgcn_readlane((int)sp, ln) >> wd) & 1;
      T gq[NH];
#pragma unroll
      for (int c = 0; c < NH; ++c) gq[c] = sel(up, q1[d][c], q0[d][c]);
      const double pre = up ? p1[d] : p0[d];
      fetch(d, step + AHEAD);
      double p = 1.0;
      T en[NH], an[NH], bn[NH];
#pragma unroll
      for (int c = 0; c < NH; ++c) {
        p *= norm2(fmac(be[c], gq[c], al[c]));
        en[c] = mulc(e[c], gq[c]);
        an[c] = recip(plus1(en[c]));
        bn[c] = mulc(en[c], an[c]);
      }
      const double ratio = pre * wave_prod(p);
      // random.bernoulli(key, P), sampler.py:336-340
      const bool acc = a.mu == 2.0 ? u < ratio : u < exp(a.mu * (0.5 * log(ratio)));
      if (acc) {
#pragma unroll
        for (int c = 0; c < NH; ++c) {
          e[c] = en[c];
          al[c] = an[c];
          be[c] = bn[c];
        }
        if (lane == ln) sp ^= 1u << wd;
        ++nacc;
      }
      ++since;
      if (--left == 0) {
        left = a.sweep_steps;
        int32_t* out = configs + row * L;
        row += a.num_chains;
        for (int w = 0; w < words; ++w)
          if (w * WAVE + lane < L) out[w * WAVE + lane] = (sp >> w) & 1;
        if (since >= RBMQ_MC_REFRESH) {
          refresh();
          since = 0;
        }
      }
    }
  }
  for (int w = 0; w < words; ++w)
    if (w * WAVE + lane < L) walkers[(int64_t)chain * L + w * WAVE + lane] = (sp >> w) & 1;
  return nacc;
}

// The chain for parameters out of that range, H <= RBMQ_MC_MAX_H: theta in LDS
// (2 H doubles), |cosh theta|^2 = e^{2 a} q / 4 with a = |Re theta| and
// q = |1 + e^{-2 theta}|^2 in [0, 4], so a proposal costs an exponential and a
// cosine per unit, a sum of a' - a and a product of q', and no logarithm per
// unit.  1024 chains x 320 proposals, 32 x 64: 609 us with rbm.hpp's log-cosh
// form here, 467 so (541 in mc_rbm); 4096 chains, 8 x 8: 2.61 ms, 0.99 (1.54).
template <bool CPX>
__device__ inline int64_t rbmq_mc_direct(const RbmGeom& g, const double* __restrict__ P, const jv_mc_args& a,
                                         int32_t* __restrict__ walkers, int32_t* __restrict__ configs, int chain,
                                         int lane, double* lds) {
  typedef typename num_of<CPX>::type T;
  T* th = (T*)lds;
  int32_t* s = (int32_t*)(lds + rbm_cw(g) * g.H);
  const double* Wr = P + g.ow;
  const double* Wi = Wr + (int64_t)g.L * g.H;
  for (int i = lane; i < g.L; i += WAVE) s[i] = walkers[(int64_t)chain * g.L + i];
  wave_sync();
  auto q_of = [](T t) {
    if constexpr (CPX) {
      const double e = exp(-2.0 * fabs(t.re));
      return 1.0 + fma(2.0 * e, cos(2.0 * t.im), e * e);
    } else {
      const double e = 1.0 + exp(-2.0 * fabs(t));
      return e * e;
    }
  };
  double Q;  // product of q over the units
  auto refresh = [&]() {
    double p = 1.0;
    for (int h = lane; h < g.H; h += WAVE) {
      const cd t = rbm_theta(g, P, s, h);
      if constexpr (CPX) th[h] = t;
      else th[h] = t.re;
      p *= q_of(th[h]);
    }
    Q = wave_prod(p);
  };
  refresh();
  auto moved = [&](int site, double d, int h) {
    const int64_t wi = (int64_t)site * g.H + h;
    if constexpr (CPX) return cd{fma(d, Wr[wi], th[h].re), fma(d, Wi[wi], th[h].im)};
    else return fma(d, Wr[wi], th[h]);
  };
  int64_t nacc = 0;
  const int total = a.therm_steps + a.samples_per_chain * a.sweep_steps;
  for (int step = 0; step < total; ++step) {
    int site;
    double u;
    mc_draw(a.seed, (uint32_t)step, (uint32_t)chain, a.call_index, a.stream, g.L, site, u);
    const double d = -2.0 * (double)(2 * s[site] - 1);
    double dl = 0.0, p = 1.0;
    for (int h = lane; h < g.H; h += WAVE) {
      const T t = moved(site, d, h);
      dl += fabs(to_cd(t).re) - fabs(to_cd(th[h]).re);
      p *= q_of(t);
    }
    dl = wave_sum(dl);
    p = wave_prod(p);
    if (g.oa >= 0) dl = fma(d, P[g.oa + site], dl);
    // random.bernoulli(key, P), sampler.py:336-340
    const bool acc = a.mu == 2.0 ? u < exp(2.0 * dl) * (p / Q) : u < exp(a.mu * fma(0.5, log(p / Q), dl));
    if (acc) {
      for (int h = lane; h < g.H; h += WAVE) th[h] = moved(site, d, h);
      Q = p;
      wave_sync();
      if (lane == 0) s[site] ^= 1;
      ++nacc;
    }
    wave_sync();
    const int k = step + 1 - a.therm_steps;
    if (k > 0 && k % a.sweep_steps == 0) {
      const int64_t t = k / a.sweep_steps - 1;
      int32_t* out = configs + (t * a.num_chains + chain) * g.L;
      for (int i = lane; i < g.L; i += WAVE) out[i] = s[i];
      refresh();
      wave_sync();
    }
  }
  for (int i = lane; i < g.L; i += WAVE) walkers[(int64_t)chain * g.L + i] = s[i];
  return nacc;
}

// The chain in the form the parameters' range allows, sizes as rbmq_mc_fits
// (lds: mc_rbm_lds_doubles(g), used out of range).
template <bool CPX, int NH>
__device__ inline int64_t rbmq_mc(const RbmGeom& g, const double* __restrict__ P, const jv_mc_args& a,
                                  const RbmTab& tab, int32_t* __restrict__ walkers, int32_t* __restrict__ configs,
                                  int chain, int lane, double* lds) {
  if (__builtin_expect(rbmq_ok(g, tab, 2, lane), 1))  // squared moduli: twice the exponent of one flip
    return rbmq_mc_chain<CPX, NH>(g, P, a, tab, walkers, configs, chain, lane);
  return rbmq_mc_direct<CPX>(g, P, a, walkers, configs, chain, lane, lds);
}
// The same for any sizes (the batch's instances differ).
__device__ inline int64_t rbmq_mc_any(const RbmGeom& g, const double* __restrict__ P, const jv_mc_args& a,
                                      const RbmTab& tab, int32_t* __restrict__ walkers, int32_t* __restrict__ configs,
                                      int chain, int lane, double* lds) {
  if (!rbmq_mc_fits(g)) return mc_rbm_chain(g, P, a, walkers, configs, chain, lane, lds);
#define JV_RBMQ_MC(NHv)                                                                        \
  return g.cpx ? rbmq_mc<true, NHv>(g, P, a, tab, walkers, configs, chain, lane, lds)          \
               : rbmq_mc<false, NHv>(g, P, a, tab, walkers, configs, chain, lane, lds)
  if (g.H <= 64) JV_RBMQ_MC(1);
  if (g.H <= 128) JV_RBMQ_MC(2);
  JV_RBMQ_MC(4);
#undef JV_RBMQ_MC
}

}  // namespace jv
