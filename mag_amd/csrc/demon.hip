// demon_microcanonical (field-demon.h:25-126) on the device, in the
// reference's sequential order: links in site-index order, mu inner, two hits
// per link, each accepted hit changing the link before the next link's
// staples are formed. The chain is inherently serial (one demon energy, one
// RNG stream), so one wavefront runs it: the 64 lanes split the 168 staple
// paths of a link (6 plaquette, 18 rectangle, 72 chair, 72 twist; index
// tables of field-staple.h:27-135 with their defects kept), the four sums are
// reduced in a fixed lane order through LDS, and lane 0 makes the proposals
// and the window test. One launch per sweep.
#include <algorithm>
#include <cstring>
#include <vector>

#include "kernels.hpp"
#include "runtime.hpp"

using namespace mag;

namespace {

constexpr int NPATH = 168;  // per direction
constexpr int PLEN = 5;

struct DemonTable {
  // dirs[mu][path][k]: 0..3 forward, 4..7 backward, -1 = end of path
  signed char dirs[4][NPATH][PLEN];
  unsigned char kind[NPATH];  // 0 plaquette, 1 rectangle, 2 chair, 3 twist
};

// Paths of get_staple_dagger (field-hmc.h:226-240), get_rectangular_dagger
// (field-hmc.h:137-201), init_chair_index / init_twist_index
// (field-staple.h:27-135).
void build_table(DemonTable& t) {
  std::memset(t.dirs, -1, sizeof t.dirs);
  const int D = 4;
  for (int mu = 0; mu < 4; ++mu) {
    int n = 0;
    auto put = [&](std::initializer_list<int> d, int kind) {
      int k = 0;
      for (int v : d) t.dirs[mu][n][k++] = (signed char)v;
      t.kind[n] = (unsigned char)kind;
      ++n;
    };
    for (int nu = 0; nu < D; ++nu) {
      if (nu == mu) continue;
      put({nu, mu, nu + D}, 0);
      put({nu + D, mu, nu}, 0);
    }
    for (int nu = 0; nu < D; ++nu) {
      if (nu == mu) continue;
      put({nu, mu, mu, nu + D, mu + D}, 1);
      put({nu + D, mu, mu, nu, mu + D}, 1);
      put({nu, nu, mu, nu + D, nu + D}, 1);
      put({nu + D, nu + D, mu, nu, nu}, 1);
      put({mu + D, nu, mu, mu, nu + D}, 1);
      put({mu + D, nu + D, mu, mu, nu}, 1);
    }
    for (int twist = 0; twist < 2; ++twist)
      for (int nu = 0; nu < D; ++nu) {
        if (nu == mu) continue;
        for (int la = 0; la < D; ++la) {
          if (la == nu || la == mu) continue;
          int b[4][4];
          if (!twist) {
            int c[4][4] = {{nu, la, la + D, nu + D}, {nu, la + D, la + D, nu},
                           {nu + D, la, la, nu + D}, {nu + D, la + D, la, nu}};
            std::memcpy(b, c, sizeof b);
          } else {
            int c[4][4] = {{nu, la, nu + D, la + D}, {nu, la + D, nu + D, la},
                           {nu + D, la, nu, la + D}, {nu + D, la + D, nu, la}};
            std::memcpy(b, c, sizeof b);
          }
          for (int k = 0; k < 4; ++k)
            for (int i = 1; i < 4; ++i) {
              int d[5], m = 0;
              for (int j = 0; j < 4; ++j) {
                if (j == i) d[m++] = mu;
                d[m++] = b[k][j];
              }
              t.dirs[mu][n][0] = (signed char)d[0];
              for (int j = 1; j < 5; ++j) t.dirs[mu][n][j] = (signed char)d[j];
              t.kind[n] = (unsigned char)(2 + twist);
              ++n;
            }
        }
      }
  }
}

struct DemonState {
  double E[4];
  long long acc, rej;
};

__global__ __launch_bounds__(64) void k_demon_sweep(LinkView<double, 18> U, Geom g, const DemonTable* tab,
                                                    DemonState* st, double emax, uint64_t seed, int sweep) {
  __shared__ double part[72][64];
  __shared__ double tot[72];
  const int lane = threadIdx.x;
  double E[4] = {st->E[0], st->E[1], st->E[2], st->E[3]};
  long long acc = st->acc, rej = st->rej;
  for (int s = 0; s < g.V; ++s) {
    const Site p0 = site_of(g, s);
    for (int mu = 0; mu < 4; ++mu) {
      M3<double> sum[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) sum[k] = zero3<double>();
      for (int q = lane; q < NPATH; q += 64) {
        Site y = p0;
        M3<double> m = unit3<double>();
        for (int j = 0; j < PLEN; ++j) {
          const int d = tab->dirs[mu][q][j];
          if (d < 0) break;
          if (d < 4) {
            m = mul(m, U.template load<double>(d, y.s));
            y.s += off_rt(g, y, d, 1);
            y.x[0] = y.s % g.L[0];
            y.x[1] = (y.s / g.S[1]) % g.L[1];
            y.x[2] = (y.s / g.S[2]) % g.L[2];
            y.x[3] = y.s / g.S[3];
          } else {
            y.s += off_rt(g, y, d - 4, -1);
            y.x[0] = y.s % g.L[0];
            y.x[1] = (y.s / g.S[1]) % g.L[1];
            y.x[2] = (y.s / g.S[2]) % g.L[2];
            y.x[3] = y.s / g.S[3];
            m = mul_nd(m, U.template load<double>(d - 4, y.s));
          }
        }
        const int kd = tab->kind[q];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (k == kd) add_to(sum[k], m);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int e = 0; e < 9; ++e) {
          part[k * 18 + 2 * e][lane] = sum[k].e[e].r;
          part[k * 18 + 2 * e + 1][lane] = sum[k].e[e].i;
        }
      __syncthreads();
      for (int comp = lane; comp < 72; comp += 64) {
        double a = 0.;
        for (int l = 0; l < 64; ++l) a += part[comp][l];
        tot[comp] = a;
      }
      __syncthreads();
      if (lane == 0) {
        M3<double> X[4];
        for (int k = 0; k < 4; ++k)
          for (int e = 0; e < 9; ++e) X[k].e[e] = {tot[k * 18 + 2 * e], tot[k * 18 + 2 * e + 1]};
        // plaquette and rectangle sums are used daggered (get_staple_dagger,
        // get_rectangular_dagger); chair and twist undaggered (field-staple.h:149,164)
        X[0] = dag(X[0]);
        X[1] = dag(X[1]);
        M3<double> v = U.template load<double>(mu, s);
        const uint32_t link = (uint32_t)s * 4u + (uint32_t)mu;
        for (int n = 0; n < 2; ++n) {
          const u32x4 w0 = rng_draw(seed, RNG_DEMON, (uint64_t)sweep, link, 3 * n);
          const u32x4 w1 = rng_draw(seed, RNG_DEMON, (uint64_t)sweep, link, 3 * n + 1);
          const u32x4 w2 = rng_draw(seed, RNG_DEMON, (uint64_t)sweep, link, 3 * n + 2);
          // random_su3_from_su2(0.9) (field-matrix.h:36-65)
          const double a0 = 0.9 + (1. - 0.9) * rng_u01(w0.x, w0.y);
          double a1 = -1. + 2. * rng_u01(w0.z, w0.w);
          double a2 = -1. + 2. * rng_u01(w1.x, w1.y);
          double a3 = -1. + 2. * rng_u01(w1.z, w1.w);
          const double nrm = sqrt((1. - a0 * a0) / (a1 * a1 + a2 * a2 + a3 * a3));
          a1 *= nrm;
          a2 *= nrm;
          a3 *= nrm;
          M3<double> m = unit3<double>();
          switch (w2.x % 3) {
            case 0: m(1, 1) = {a0, a3}; m(1, 2) = {a2, a1}; m(2, 1) = {-a2, a1}; m(2, 2) = {a0, -a3}; break;
            case 1: m(0, 0) = {a0, a3}; m(0, 2) = {a2, a1}; m(2, 0) = {-a2, a1}; m(2, 2) = {a0, -a3}; break;
            default: m(0, 0) = {a0, a3}; m(0, 1) = {a2, a1}; m(1, 0) = {-a2, a1}; m(1, 1) = {a0, -a3}; break;
          }
          const M3<double> mv = mul(m, v);
          double dS[4];
          bool ok = true;
          for (int k = 0; k < 4; ++k) {
            dS[k] = -retrace_mul(mv, X[k]) + retrace_mul(v, X[k]);
            ok = ok && (E[k] - dS[k] > -emax) && (E[k] - dS[k] < emax);
          }
          if (ok) {
            v = mv;
            for (int k = 0; k < 4; ++k) E[k] -= dS[k];
            ++acc;
          } else {
            ++rej;
          }
        }
        U.store(mu, s, v);
      }
      // make lane 0's link store visible to every lane's next loads
      __threadfence();
      __syncthreads();
    }
  }
  if (lane == 0) {
    for (int k = 0; k < 4; ++k) st->E[k] = E[k];
    st->acc = acc;
    st->rej = rej;
  }
}

// ------------------------------------------------------------ chair / twist staples
// chair_staple_dagger / twist_staple_dagger (field-staple.h:141-165) for every
// link: S(x, mu) = the sum of the 72 chair (kind 2) or twist (kind 3) path
// products of the table, undaggered as the reference returns it.
__global__ __launch_bounds__(BLOCK) void k_staple_table_sum(LinkView<double, 18> U, Geom g, const DemonTable* tab,
                                                            int kind, LinkView<double, 18> S) {
  const int s = blockIdx.x * BLOCK + threadIdx.x;
  const int mu = blockIdx.y;
  if (s >= g.V) return;
  const Site p0 = site_of(g, s);
  M3<double> acc = zero3<double>();
  for (int q = 0; q < NPATH; ++q) {
    if (tab->kind[q] != kind) continue;
    Site y = p0;
    M3<double> m = unit3<double>();
    for (int j = 0; j < PLEN; ++j) {
      const int d = tab->dirs[mu][q][j];
      if (d < 0) break;
      if (d < 4) {
        m = mul(m, U.template load<double>(d, y.s));
        y.s += off_rt(g, y, d, 1);
      } else {
        y.s += off_rt(g, y, d - 4, -1);
      }
      y.x[0] = y.s % g.L[0];
      y.x[1] = (y.s / g.S[1]) % g.L[1];
      y.x[2] = (y.s / g.S[2]) % g.L[2];
      y.x[3] = y.s / g.S[3];
      if (d >= 4) m = mul_nd(m, U.template load<double>(d - 4, y.s));
    }
    add_to(acc, m);
  }
  S.store(mu, s, acc);
}

// ------------------------------------------------------------ checkerboard demon
// demon_microcanonical with a demon per link (four energies per link, four
// MAG_REAL1 fields), updated in parallel: per direction MU, 128 classes
// (x_MU mod 2, then x_nu mod 4 for the transverse nu in increasing order).
// Every staple path of a link holds its MU-links at offsets with |d_nu| <= 2
// and d_MU in {-1, 0, 1}, so two links of one class never meet in a path:
// the updates of a class commute and each moves its own action change into
// its own demons. The classes are swept in order; two that follow each other
// with no path between them share a launch (demon_launches). Hit counts in
// per-member slots.
struct DemonClassArgs {
  LinkView<double, 18> U;
  Geom g;
  double* E[4];   // per-link demon energies, [mu][site] each
  double* cnt;    // [thread][2]: accept, reject
  double emax;
  uint64_t seed;
  int sweep;
  int cls[2];  // the launch's classes: x_MU parity + 2 (transverse residues, base 4)
  int nthr;    // class members
};

// The classes of a direction in launches of one or two: a class goes into the
// launch after the last earlier class whose links its paths read or that reads
// its links. Only classes that commute change place, so a sweep gives what the
// 128 classes give in order, in 95 launches. That counts where a launch does
// not fill the chip: sweep 4^4 7.2 -> 5.5 ms, 16^4 9.0 -> 6.9, 24^4 22.0 -> 19.9, 32^4
// 52 -> 49.5.
struct DemonLaunches {
  int n;
  int cls[128][2];  // second: -1 where there is none
};
DemonLaunches demon_launches(const DemonTable& t, int mu) {
  // the offsets between links that meet in a path, x_mu modulo 2 and the
  // transverse coordinates modulo 4
  bool meet[2][4][4][4] = {};
  for (int p = 0; p < NPATH; ++p) {
    int y[4] = {0, 0, 0, 0};  // mu first, then the transverse axes in order
    for (int k = 0; k < PLEN && t.dirs[mu][p][k] >= 0; ++k) {
      const int d = t.dirs[mu][p][k] & 3, i = d == mu ? 0 : (d < mu ? d + 1 : d);
      const bool back = t.dirs[mu][p][k] >= 4;
      if (back) --y[i];
      if (d == mu) {
        meet[y[0] & 1][y[1] & 3][y[2] & 3][y[3] & 3] = true;
        meet[-y[0] & 1][-y[1] & 3][-y[2] & 3][-y[3] & 3] = true;
      }
      if (!back) ++y[i];
    }
  }
  DemonLaunches out{};
  int at[128];  // launch of each class
  for (int c = 0; c < 128; ++c) {
    int l = 0;
    for (int e = 0; e < c; ++e)
      if (meet[(c - e) & 1][((c >> 1) - (e >> 1)) & 3][((c >> 3) - (e >> 3)) & 3][((c >> 5) - (e >> 5)) & 3])
        l = std::max(l, at[e] + 1);
    while (l < out.n && out.cls[l][1] >= 0) ++l;  // full
    if (l == out.n) {
      out.cls[l][0] = c;
      out.cls[out.n++][1] = -1;
    } else {
      out.cls[l][1] = c;
    }
    at[c] = l;
  }
  return out;
}

// The staple sums of a member, by signed transverse directions n and l on
// different axes (24 pairs). Writing a path as the directions it steps along,
// with m for +MU:
//   twist   n m l -n -l,  n l m -n -l,  n l -n m -l              every (n, l)
//   chair   n m l l n,    n l m l n,    n l l m n                signs of n, l differ
//           n l m -l -n,  and n m l -l -n, n l -l m -n           signs alike
// (the table's defects kept). The last two step back along a link at once and
// are the plaquette staple n m -n: each staple four times in all. The others
// share factors: with A1 = U_m(x+n) U_l(x+n+m), A2 = U_l(x+n) U_m(x+n+l), both
// from x+n to x+n+l+m, each pair gives
//   twist   U_n [(A1 + A2) U_-n + U_l U_-n U_m] U_-l
//   chair   U_n [(A1 + A2) U_l + U_l U_l U_m] U_n      or      U_n A2 U_-l U_-n
// 13-16 links and about 10 products against 30 links and 24 products path by
// path. The 24 plaquette and rectangle staples go one to each pair.
//
// A block is ten members by four wavefronts, one per choice of signs, so that
// the form and every dagger are the same across a wavefront; a lane is one of
// its six axis pairs of one member, ten neighbouring members side by side.
// The shares are summed in LDS in a fixed order, one kind of sum at a time;
// then four lanes per member, one per kind, make the two hits. What bounds a
// class launch on lattices up to 16^4 (52 blocks) is the latency of one
// wavefront, above that one wavefront per SIMD (460 registers: a lane asks
// for all its links at once; held to two, it spills 856 bytes and takes 1.5
// to 1.9 times as long). Launch of a class: 4^4 77 -> 14 us, 16^4 78 -> 18,
// 24^4 90 -> 43, 32^4 152 -> 103, against eight lanes per member that walked
// the 168 paths one by one.
constexpr int DEMON_MEMBERS = 10, DEMON_PAIRS = 6;
// MAG_DEMON_READ12 = 1: the path links are read as rows 0 and 1 with row 2
// rebuilt (the links stay in SU(3)).
#ifndef MAG_DEMON_READ12
#define MAG_DEMON_READ12 1
#endif

struct DemonPos {
  int x[4], s;
};
// The link of a step along axis k, forward or backward, from y, which moves on.
template <bool BACK>
MAG_D M3<double> demon_step(const DemonClassArgs& A, DemonPos& y, int k) {
  const int s0 = y.s;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (i == k) {
      const int v = y.x[i], L = A.g.L[i];
      const int w = BACK ? (v == 0 ? L - 1 : v - 1) : (v == L - 1 ? 0 : v + 1);
      y.x[i] = w;
      y.s += (w - v) * A.g.S[i];
    }
  const M3<double> m = A.U.template load_su3<double, MAG_DEMON_READ12 != 0>(k, BACK ? y.s : s0);
  return BACK ? dag(m) : m;
}
MAG_D M3<double> mul_su3(const M3<double>& a, const M3<double>& b) {
  M3<double> c = mul_r2(a, b);
  reconstruct_row2(c);
  return c;
}

// One lane's shares: twist, chair (without the plaquette staples) and one
// plaquette or rectangle staple; SN, SL: whether n, l point backward. j = 0 or
// 1 numbers the axis of l; with SL forward j = 0 holds the plaquette staple.
template <int MU, bool SN, bool SL>
MAG_D void demon_shares(const DemonClassArgs& A, const DemonPos& x, int n, int l, int j, M3<double>& tw,
                        M3<double>& ch, M3<double>& pr) {
  DemonPos yn = x;
  const M3<double> Un = demon_step<SN>(A, yn, n);  // x -> x+n
  DemonPos ym = yn, yl = yn;
  const M3<double> m1 = demon_step<false>(A, ym, MU);  // x+n -> x+n+m
  const M3<double> l1 = demon_step<SL>(A, yl, l);      // x+n -> x+n+l
  DemonPos ye = ym, t = yl;
  const M3<double> l2 = demon_step<SL>(A, ye, l);      // x+n+m -> x+n+l+m
  const M3<double> m2 = demon_step<false>(A, t, MU);   // x+n+l -> x+n+l+m
  const M3<double> A2 = mul_su3(l1, m2);
  const M3<double> S = add(mul_su3(m1, l2), A2);
  {
    t = ye;
    M3<double> B = mul(S, demon_step<!SN>(A, t, n));   // -> x+l+m
    DemonPos u = yl;
    M3<double> C = mul_r2(l1, demon_step<!SN>(A, u, n));  // -> x+l
    add_to(B, mul_su3(C, demon_step<false>(A, u, MU)));   // -> x+l+m
    tw = mul(Un, mul(B, demon_step<!SL>(A, t, l)));       // -> x+m
  }
  t = ye;
  if (SN != SL) {
    M3<double> B = mul(S, demon_step<SL>(A, t, l));       // -> x+n+2l+m
    DemonPos u = yl;
    M3<double> C = mul_r2(l1, demon_step<SL>(A, u, l));   // -> x+n+2l
    add_to(B, mul_su3(C, demon_step<false>(A, u, MU)));   // -> x+n+2l+m
    ch = mul(Un, mul(B, demon_step<SN>(A, t, n)));        // -> x+2n+2l+m
  } else {
    M3<double> B = mul_r2(mul_r2(Un, A2), demon_step<!SL>(A, t, l));  // -> x+n+m
    ch = mul_su3(B, demon_step<!SN>(A, t, n));                        // -> x+m
  }
  if (!SL) {
    t = ym;
    M3<double> B = mul_r2(Un, m1);
    if (j == 0) {  // n m -n
      pr = mul_su3(B, demon_step<!SN>(A, t, n));
    } else {  // n m m -n -m
      B = mul_r2(B, demon_step<false>(A, t, MU));
      B = mul_r2(B, demon_step<!SN>(A, t, n));
      pr = mul_su3(B, demon_step<true>(A, t, MU));
    }
  } else if (j == 0) {  // n n m -n -n
    t = yn;
    M3<double> B = mul_r2(Un, demon_step<SN>(A, t, n));
    B = mul_r2(B, demon_step<false>(A, t, MU));
    B = mul_r2(B, demon_step<!SN>(A, t, n));
    pr = mul_su3(B, demon_step<!SN>(A, t, n));
  } else {  // -m n m m -n
    t = x;
    M3<double> B = demon_step<true>(A, t, MU);
    B = mul_r2(B, demon_step<SN>(A, t, n));
    B = mul_r2(B, demon_step<false>(A, t, MU));
    B = mul_r2(B, m1);
    t = ym;
    pr = mul_su3(B, demon_step<!SN>(A, t, n));
  }
}

// Proposal of hit n of link (x, mu): random_su3_from_su2(0.9) (field-matrix.h:36-65).
MAG_D M3<double> demon_proposal(const DemonClassArgs& A, uint32_t link, int n) {
  const u32x4 w0 = rng_draw(A.seed, RNG_DEMON, (uint64_t)A.sweep, link, 3 * n);
  const u32x4 w1 = rng_draw(A.seed, RNG_DEMON, (uint64_t)A.sweep, link, 3 * n + 1);
  const u32x4 w2 = rng_draw(A.seed, RNG_DEMON, (uint64_t)A.sweep, link, 3 * n + 2);
  const double a0 = 0.9 + (1. - 0.9) * rng_u01(w0.x, w0.y);
  double a1 = -1. + 2. * rng_u01(w0.z, w0.w);
  double a2 = -1. + 2. * rng_u01(w1.x, w1.y);
  double a3 = -1. + 2. * rng_u01(w1.z, w1.w);
  const double nrm = sqrt((1. - a0 * a0) / (a1 * a1 + a2 * a2 + a3 * a3));
  a1 *= nrm;
  a2 *= nrm;
  a3 *= nrm;
  M3<double> m = unit3<double>();
  switch (w2.x % 3) {
    case 0: m(1, 1) = {a0, a3}; m(1, 2) = {a2, a1}; m(2, 1) = {-a2, a1}; m(2, 2) = {a0, -a3}; break;
    case 1: m(0, 0) = {a0, a3}; m(0, 2) = {a2, a1}; m(2, 0) = {-a2, a1}; m(2, 2) = {a0, -a3}; break;
    default: m(0, 0) = {a0, a3}; m(0, 1) = {a2, a1}; m(1, 0) = {-a2, a1}; m(1, 1) = {a0, -a3}; break;
  }
  return m;
}

// Member t of a class of direction MU.
template <int MU>
MAG_D DemonPos demon_member(const DemonClassArgs& A, int cls, int t) {
  DemonPos p;
  p.s = 0;
  int c = cls >> 1;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int step = (i == MU) ? 2 : 4, n = A.g.L[i] / step, h = t % n;
    t /= n;
    if (i == MU) {
      p.x[i] = 2 * h + (cls & 1);
    } else {
      p.x[i] = 4 * h + (c & 3);
      c >>= 2;
    }
    p.s += p.x[i] * A.g.S[i];
  }
  return p;
}

template <int MU>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1))) void k_demon_class(DemonClassArgs A) {
  constexpr int NM = DEMON_MEMBERS, NP = DEMON_PAIRS;
  __shared__ double buf[4][NP][NM][18];  // one kind of share at a time
  __shared__ double tot[4][NM][18];      // plaquette, rectangle, chair, twist sums
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  // lanes 60-63 repeat the last pair and write nothing, members past the end the last member
  const int pair = min(lane / NM, NP - 1), mem = lane % NM;
  const int cls = blockIdx.y ? A.cls[1] : A.cls[0];
  const DemonPos x = demon_member<MU>(A, cls, min((int)blockIdx.x * NM + mem, A.nthr - 1));
  const int i = pair >> 1, j = pair & 1;
  const int n = i + (i >= MU ? 1 : 0);  // axis of n; that of l is the j-th of the other two
  int l = 0, seen = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (k != MU && k != n && seen++ == j) l = k;
  M3<double> sh[3];
  switch (wave) {
    case 0: demon_shares<MU, false, false>(A, x, n, l, j, sh[0], sh[1], sh[2]); break;
    case 1: demon_shares<MU, false, true>(A, x, n, l, j, sh[0], sh[1], sh[2]); break;
    case 2: demon_shares<MU, true, false>(A, x, n, l, j, sh[0], sh[1], sh[2]); break;
    default: demon_shares<MU, true, true>(A, x, n, l, j, sh[0], sh[1], sh[2]); break;
  }
  const int e = threadIdx.x % 18, m = threadIdx.x / 18;  // the element that a thread sums
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    if (lane < NP * NM) {
#pragma unroll
      for (int k = 0; k < 9; ++k) {
        buf[wave][pair][mem][2 * k] = sh[r].e[k].r;
        buf[wave][pair][mem][2 * k + 1] = sh[r].e[k].i;
      }
    }
    __syncthreads();
    if (m < NM) {
      double a = 0., b = 0.;
      for (int w = 0; w < 4; ++w)
        for (int q = 0; q < NP; ++q) {
          const double v = buf[w][q][m][e];
          if (r == 2 && (w & 1) == 0 && (q & 1) == 0) b += v;  // plaquette staples
          else a += v;
        }
      if (r == 0) tot[3][m][e] = a;
      if (r == 1) tot[2][m][e] = a;
      if (r == 2) {
        tot[1][m][e] = a;
        tot[0][m][e] = b;
        tot[2][m][e] += 4. * b;
      }
    }
    __syncthreads();
  }
  // the hits: lane 4 m + k holds kind k of member m
  if (wave != 3 || lane >= 4 * NM) return;
  const int hm = lane >> 2, k = lane & 3, t = (int)blockIdx.x * NM + hm;
  if (t >= A.nthr) return;
  const int s = demon_member<MU>(A, cls, t).s;
  const uint32_t link = (uint32_t)s * 4u + (uint32_t)MU;
  M3<double> X;
#pragma unroll
  for (int q = 0; q < 9; ++q) X.e[q] = {tot[k][hm][2 * q], tot[k][hm][2 * q + 1]};
  // plaquette and rectangle sums are used daggered, chair and twist as they are
  if (k < 2) X = dag(X);
  M3<double> v = A.U.template load<double>(MU, s);
  double E = A.E[k][(size_t)MU * A.g.V + s];
  double acc = 0., rej = 0.;
  double old = retrace_mul(v, X);
#pragma unroll 1
  for (int h = 0; h < 2; ++h) {
    const M3<double> mv = mul(demon_proposal(A, link, h), v);
    const double now = retrace_mul(mv, X), dS = old - now;
    const bool ok = (E - dS > -A.emax) && (E - dS < A.emax);
    if (((__ballot(ok) >> (lane & ~3)) & 15) == 15) {
      v = mv;
      old = now;
      E -= dS;
      acc += 1.;
    } else {
      rej += 1.;
    }
  }
  A.E[k][(size_t)MU * A.g.V + s] = E;
  if (k == 0) {
    A.U.template store<double>(MU, s, v);
    double* cnt = A.cnt + 2 * ((size_t)blockIdx.y * A.nthr + t);
    cnt[0] += acc;
    cnt[1] += rej;
  }
}

}  // namespace

extern "C" int mag_demon_microcanonical(mag_field U, int nsweeps, double E_max, uint64_t seed, double E[4],
                                        long acc_rej[2]) {
  if (!U || !E || !acc_rej || nsweeps < 0) return MAG_ERR_ARG;
  mag_ctx c = U->ctx;
  if (U->kind != MAG_LINK18 || U->prec != MAG_F64)
    return fail(c, MAG_ERR_UNSUPPORTED, "the demon runs on FP64 18-real links");
  DemonTable* ht = new DemonTable();
  build_table(*ht);
  DemonTable* dt = nullptr;
  DemonState* ds = nullptr;
  int r = dev_alloc(c, (void**)&dt, sizeof(DemonTable));
  if (!r) r = dev_alloc(c, (void**)&ds, sizeof(DemonState));
  DemonState h{};
  for (int k = 0; k < 4; ++k) h.E[k] = E[k];
  if (!r && (hipMemcpyAsync(dt, ht, sizeof(DemonTable), hipMemcpyHostToDevice, c->stream) != hipSuccess ||
             hipMemcpyAsync(ds, &h, sizeof h, hipMemcpyHostToDevice, c->stream) != hipSuccess))
    r = fail(c, MAG_ERR_DEVICE, "demon upload failed");
  for (int sw = 0; sw < nsweeps && !r; ++sw) {
    KTimer t(c, "demon");
    hipLaunchKernelGGL(k_demon_sweep, dim3(1), dim3(64), 0, c->stream, LinkView<double, 18>{(double*)U->p, U->g.V},
                       U->g, dt, ds, E_max, seed, sw);
    if (hipGetLastError() != hipSuccess) r = fail(c, MAG_ERR_DEVICE, "demon launch failed");
  }
  if (!r && (hipMemcpyAsync(&h, ds, sizeof h, hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
             hipStreamSynchronize(c->stream) != hipSuccess))
    r = fail(c, MAG_ERR_DEVICE, "demon download failed");
  (void)hipStreamSynchronize(c->stream);
  dev_free(c, dt, dt ? sizeof(DemonTable) : 0);
  dev_free(c, ds, ds ? sizeof(DemonState) : 0);
  delete ht;
  if (r) return r;
  for (int k = 0; k < 4; ++k) E[k] = h.E[k];
  acc_rej[0] = (long)h.acc;
  acc_rej[1] = (long)h.rej;
  return MAG_OK;
}

extern "C" int mag_demon_checkerboard(mag_field U, mag_field Ep, mag_field Er, mag_field Ec, mag_field Et, int nsweeps,
                                      double E_max, uint64_t seed, long acc_rej[2]) {
  mag_field Ef[4] = {Ep, Er, Ec, Et};
  if (!U || nsweeps < 0) return MAG_ERR_ARG;
  mag_ctx c = U->ctx;
  if (U->kind != MAG_LINK18 || U->prec != MAG_F64)
    return fail(c, MAG_ERR_UNSUPPORTED, "the demon runs on FP64 18-real links");
  for (int k = 0; k < 4; ++k) {
    if (!Ef[k] || Ef[k]->kind != MAG_REAL1 || Ef[k]->ctx != c)
      return fail(c, MAG_ERR_ARG, "demon energies are four MAG_REAL1 fields of the links' context");
    for (int i = 0; i < 4; ++i)
      if (Ef[k]->dims[i] != U->dims[i]) return fail(c, MAG_ERR_GEOMETRY, "demon fields differ in extents");
  }
  for (int i = 0; i < 4; ++i)
    if (U->g.L[i] % 4) return fail(c, MAG_ERR_GEOMETRY, "the checkerboard demon needs extents that are multiples of 4");
  if (c->rec) return fail(c, MAG_ERR_UNSUPPORTED, "the demon is not recordable");
  const int nthr = U->g.V / 128;
  int r;
  Workspace* ws = workspace(c, U->g, MAG_F64, 18);
  if ((r = ws->need_cnt())) return r;  // V doubles >= 4 per member
  double* cnt = (double*)ws->Cnt;
  if ((r = fill_dev(c, cnt, 0., 4 * nthr))) return r;
  DemonClassArgs A{};
  A.U = LinkView<double, 18>{(double*)U->p, U->g.V};
  A.g = U->g;
  for (int k = 0; k < 4; ++k) A.E[k] = (double*)Ef[k]->p;
  A.cnt = cnt;
  A.emax = E_max;
  A.seed = seed;
  void (*ks[4])(DemonClassArgs) = {k_demon_class<0>, k_demon_class<1>, k_demon_class<2>, k_demon_class<3>};
  A.nthr = nthr;
  DemonTable table;
  build_table(table);
  DemonLaunches dl[4];
  for (int mu = 0; mu < 4; ++mu) dl[mu] = demon_launches(table, mu);
  for (int sw = 0; sw < nsweeps && !r; ++sw) {
    A.sweep = sw;
    for (int mu = 0; mu < 4 && !r; ++mu)
      for (int l = 0; l < dl[mu].n && !r; ++l) {
        A.cls[0] = dl[mu].cls[l][0];
        A.cls[1] = dl[mu].cls[l][1];
        const dim3 grid((nthr + DEMON_MEMBERS - 1) / DEMON_MEMBERS, A.cls[1] < 0 ? 1 : 2);
        KTimer t(c, "demon_checkerboard");
        hipLaunchKernelGGL(ks[mu], grid, dim3(256), 0, c->stream, A);
        if (hipGetLastError() != hipSuccess) r = fail(c, MAG_ERR_DEVICE, "demon launch failed");
      }
  }
  std::vector<double> h((size_t)4 * nthr);
  if (!r && (hipMemcpyAsync(h.data(), cnt, h.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream) !=
                 hipSuccess ||
             hipStreamSynchronize(c->stream) != hipSuccess))
    r = fail(c, MAG_ERR_DEVICE, "demon download failed");
  if (r) return r;
  if (acc_rej) {
    double a = 0., b = 0.;
    for (int t = 0; t < 2 * nthr; ++t) {
      a += h[(size_t)2 * t];
      b += h[(size_t)2 * t + 1];
    }
    acc_rej[0] = (long)a;
    acc_rej[1] = (long)b;
  }
  return MAG_OK;
}

namespace {
int staple_table_field(mag_field S, mag_field U, int kind) {
  if (!S || !U || S->ctx != U->ctx) return MAG_ERR_ARG;
  mag_ctx c = U->ctx;
  if (U->kind != MAG_LINK18 || U->prec != MAG_F64 || S->kind != MAG_LINK18 || S->prec != MAG_F64)
    return fail(c, MAG_ERR_UNSUPPORTED, "chair/twist staples take and give FP64 18-real fields");
  for (int i = 0; i < 4; ++i)
    if (S->dims[i] != U->dims[i]) return fail(c, MAG_ERR_ARG, "chair/twist staples: fields differ in shape");
  if (S->p == U->p) return fail(c, MAG_ERR_ARG, "chair/twist staples: output must not alias the links");
  if (c->rec) return fail(c, MAG_ERR_UNSUPPORTED, "chair/twist staples are not recordable");
  DemonTable* ht = new DemonTable();
  build_table(*ht);
  DemonTable* dt = nullptr;
  int r = dev_alloc(c, (void**)&dt, sizeof(DemonTable));
  if (!r && hipMemcpyAsync(dt, ht, sizeof(DemonTable), hipMemcpyHostToDevice, c->stream) != hipSuccess)
    r = fail(c, MAG_ERR_DEVICE, "staple table upload failed");
  if (!r) {
    KTimer t(c, "staple_table");
    hipLaunchKernelGGL(k_staple_table_sum, grid_links(U->g), dim3(BLOCK), 0, c->stream,
                       LinkView<double, 18>{(double*)U->p, U->g.V}, U->g, (const DemonTable*)dt, kind,
                       LinkView<double, 18>{(double*)S->p, U->g.V});
    if (hipGetLastError() != hipSuccess) r = fail(c, MAG_ERR_DEVICE, "staple table launch failed");
  }
  (void)hipStreamSynchronize(c->stream);
  dev_free(c, dt, dt ? sizeof(DemonTable) : 0);
  delete ht;
  return r;
}
}  // namespace

extern "C" int mag_chair_staple_dagger(mag_field S, mag_field U) { return staple_table_field(S, U, 2); }
extern "C" int mag_twist_staple_dagger(mag_field S, mag_field U) { return staple_table_field(S, U, 3); }
