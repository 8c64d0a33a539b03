// Definitions of Ops<TS, NC>: the launch schedules of the force (thin or
// stout-smeared), link updates, integrators and reductions. Included only by
// the per-format instantiation units (inst_f64.hip, inst_f32.hip).
#pragma once
#include <algorithm>
#include <cmath>

#include "kernels.hpp"
#include "launch.hpp"
#include "runtime.hpp"

// Reals per staged link of the LDS-tiled FP32 Iwasaki top kernel (12 or 20;
// 0: the untiled kernel).
#ifndef MAG_TOP_LDS
#define MAG_TOP_LDS 0
#endif

// FP64 18-real links read as rows 0 and 1 with row 2 rebuilt, a bit per
// kernel: 1 stout forward, 2 stout backward, 4 last backward, 8 link update.
// The rectangle staples of the top kernel and the thin-link force read whole
// links (two rows: 2.16 -> 2.37 ms and 1.88 -> 2.13 ms at 32^4).
#ifndef MAG_FP64_READ12
#define MAG_FP64_READ12 15
#endif

namespace mag {

// whether Ops<TS, NC> reads its links as two rows in those kernels
template <class TS, int NC>
constexpr bool ops_read12(int bit) { return (MAG_FP64_READ12 & bit) != 0 && std::is_same<TS, double>::value && NC == 18; }

// FP64 rectangle staples take the split form (with one exception in
// thin_force). One thread per link
// needs more than 256 VGPRs for them (it spills, or runs one wave per SIMD),
// a plane's share fits; and three wavefronts on the same 64 sites ask L2 for
// a third of the sites at a time. Thin force / top kernel, one thread per
// link -> split: 12^4 59 -> 43 / 72 -> 57 us, 16^4 128 -> 110 / 161 -> 139,
// 24^4 707 -> 569 / 857 -> 691, 32^4 2.17 -> 1.86 / 2.54 -> 2.15 ms.
template <class TS>
constexpr bool split_rectangles() { return std::is_same<TS, double>::value; }

template <class TS, int NC>
LinkView<TS, NC> lview(void* p, const Geom& g) { return LinkView<TS, NC>{(TS*)p, g.V}; }
template <class TS>
AlgView<TS> aview(void* p, const Geom& g) { return AlgView<TS>{(TS*)p, g.V}; }
template <class TS>
MatView<TS> mview(void* p, const Geom& g) { return MatView<TS>{(TS*)p, g.V}; }

template <class TS, int NC>
int Ops<TS, NC>::link_update(mag_ctx c, const Geom& g, void* Uin, void* Uout, void* P, double eps, int mag) {
  UpdateArgs<TS, NC> a{g, lview<TS, NC>(Uin, g), lview<TS, NC>(Uout, g), aview<TS>(P, g), eps, mag};
  constexpr bool R12 = ops_read12<TS, NC>(8);
  return launch(c, "link_update", k_link_update<TS, NC, TS, R12>, k_link_update_b<TS, NC, TS, R12>, grid_links(g), a);
}

// Thin-link force. Constrained runs on small lattices: the links with two
// staple sums have blocks of their own, since with both sums in the stencil
// every wavefront that meets such a link is twice as long (FP64 Iwasaki, mag
// = 2: 4^4 58 -> 22 us, 8^4 61 -> 24, 12^4 107 -> 60; FP32 61 -> 17, 65 -> 18,
// 64 -> 27). On larger lattices that costs little, and those blocks, which
// share no neighbours with the stencil's in flight, cost more: 32^4 2.44 ms in
// one thread per link, 2.86 with them; at 32,768 sites FP64 Wilson 29 -> 25 us (16^3
// x 8; 8 x 14 x 16^2 19 -> 21), Iwasaki 121 -> 77. Block size 1 has no such link and no
// force at all (the classes alone say so: 5 us against 45 at 12^4), and a negative size,
// whose links are never the last of a block, is not one that pair_site lists.
inline bool gather_pairs(const Geom& g, int mag) { return mag >= 2 && g.V <= 32768; }
template <int ACT, class TS, int NC>
int thin_force(mag_ctx c, ForceArgs<TS, NC> fa) {
  const char* name = ACT == ACT_IWASAKI ? "force_iwasaki" : "force_wilson";
  const Geom& g = fa.g;
  if (fa.mag && !gather_pairs(g, fa.mag))
    return launch(c, name, k_gauge_force<ACT, true, TS, NC, TS>, k_gauge_force_b<ACT, true, TS, NC, TS>,
                  grid_stencil(g), fa);
  if (fa.mag) {
    int n = 0;
    for (int mu = 0; mu < 4; ++mu) n = std::max(n, pair_count(g, mu, fa.mag));
    fa.npair = (4 * ((n + 63) / 64) + 7) / 8 * 8;  // the stencil's blocks keep their XCDs
    dim3 grid = grid_split(g);
    grid.x += fa.npair;
    return launch(c, name, k_cons_force<ACT, TS, NC, TS>, k_cons_force_b<ACT, TS, NC, TS>, grid, fa, PLANE_THREADS);
  }
  const Stencil<ForceStencil<ACT, false, TS, NC, TS>> split;
  if constexpr (ACT == ACT_IWASAKI && split_rectangles<TS>()) {
    // 12-real links: one wavefront per SIMD takes 27-28 us up to
    // 16,384 sites; split 24.6 at 12,288, 29.9 at 13,824, 30.9 at 16,384
    if (NC != 12 || g.V <= 12288 || g.V > 16384) return launch_split(c, name, split, g, fa);
    return launch(c, name, k_gauge_force<ACT, false, TS, NC, TS>, k_gauge_force_b<ACT, false, TS, NC, TS>,
                  grid_stencil(g), fa);
  } else {
    return launch_stencil(c, name, k_gauge_force<ACT, false, TS, NC, TS>, k_gauge_force_b<ACT, false, TS, NC, TS>,
                          split, g, fa);
  }
}

// Force of the (possibly smeared) action on U with one of the epilogues
// OUT_F -> F, OUT_PADD -> P += eps F, OUT_UAUX -> Uaux = e^{i eps F} U.
// Thin action: one kernel (k_gauge_force). Smeared action (n levels):
// n forward kernels, the top kernel (action derivative + Lambda of level
// n-1), n-1 backward kernels each fused with the next Lambda step, and the
// last backward kernel fused with the force epilogue.
template <class TS, int NC>
int Ops<TS, NC>::force(mag_ctx c, const Geom& g, void* U, const mag_action& act, int out, void* F, void* P,
                       void* Uaux, double eps, Workspace* ws) {
  int r;
  // constrained runs cannot fuse the auxiliary link update (it needs F(x-mu))
  if (act.mag && out == OUT_UAUX) {
    if ((r = ws->need_md())) return r;
    if ((r = force(c, g, U, act, OUT_F, ws->F, nullptr, nullptr, 0., ws))) return r;
    return link_update(c, g, U, Uaux, ws->F, eps, act.mag);
  }
  ForceArgs<TS, NC> fa{};
  fa.g = g;
  fa.U = lview<TS, NC>(U, g);
  fa.F = aview<TS>(F, g);
  fa.P = aview<TS>(P, g);
  fa.Uaux = lview<TS, NC>(Uaux, g);
  fa.beta = act.beta;
  fa.c1 = act.c1;
  fa.mag = act.mag;
  fa.out = out;
  fa.eps = eps;
  const bool iw = act.type == MAG_IWASAKI;
  if (act.n_stout <= 0) return iw ? thin_force<ACT_IWASAKI>(c, fa) : thin_force<ACT_WILSON>(c, fa);
  const int n = act.n_stout;
  constexpr bool R12 = ops_read12<TS, NC>(1), R12B = ops_read12<TS, NC>(2), R12L = ops_read12<TS, NC>(4);
  if ((r = ws->need_stout(n))) return r;
  // FP64 12-real chains keep the top level U_n as 18 reals (written by the
  // last forward level, read only by the top kernel's staple sum).
  constexpr int NCN = (std::is_same<TS, double>::value && NC == 12) ? 18 : NC;
  if (NCN != NC && (r = ws->need_top18())) return r;
  auto Ulev = [&](int k) { return k == 0 ? U : ws->Us[k - 1]; };
  for (int k = 0; k < n; ++k) {
    if (NCN != NC && k == n - 1) {
      StoutFwdArgs<TS, NC, TS, NCN> fw{g, lview<TS, NC>(Ulev(k), g), aview<TS>(ws->Qs[k], g),
                                       mview<TS>(ws->Cs[k], g), lview<TS, NCN>(ws->Utop, g), act.rho, 1};
      r = launch_stencil(c, "stout_fwd", k_stout_fwd<TS, NC, TS, NCN, TS>, k_stout_fwd_b<TS, NC, TS, NCN, TS>,
                         Stencil<FwdStencil<TS, NC, TS, NCN, TS>>{}, g, fw);
    } else {
      StoutFwdArgs<TS, NC, TS, NC> fw{g, lview<TS, NC>(Ulev(k), g), aview<TS>(ws->Qs[k], g),
                                      mview<TS>(ws->Cs[k], g), lview<TS, NC>(ws->Us[k], g), act.rho, 1};
      r = launch_stencil(c, "stout_fwd", k_stout_fwd<TS, NC, TS, NC, TS, R12>, k_stout_fwd_b<TS, NC, TS, NC, TS, R12>,
                         Stencil<FwdStencil<TS, NC, TS, NC, TS, R12>>{}, g, fw);
    }
    if (r) return r;
  }
  int cur = 0;
  {
    StoutTopArgs<TS, NC, NCN> tp{g,
                                 lview<TS, NCN>(NCN != NC ? ws->Utop : Ulev(n), g),
                                 lview<TS, NC>(Ulev(n - 1), g),
                                 aview<TS>(ws->Qs[n - 1], g),
                                 mview<TS>(ws->Cs[n - 1], g),
                                 aview<TS>(ws->L[cur], g),
                                 mview<TS>(ws->W, g),
                                 act.beta,
                                 act.c1,
                                 act.rho};
    bool tiled = false;  // the LDS-tiled FP32 Iwasaki top kernel, when compiled in and the shape fits
    if constexpr (MAG_TOP_LDS != 0 && std::is_same<TS, float>::value && NC == 12) {
      tiled = iw && top_tile_ok(g);
      if (tiled)
        r = launch(c, "stout_top", k_stout_top_tile<MAG_TOP_LDS>, k_stout_top_tile_b<MAG_TOP_LDS>, grid_stencil(g),
                   tp);
    }
    if (!tiled) {
      const Stencil<TopStencil<ACT_IWASAKI, TS, NC, TS, NCN>> split;
      if (!iw)
        r = launch_stencil(c, "stout_top", k_stout_top<ACT_WILSON, TS, NC, TS, NCN>,
                           k_stout_top_b<ACT_WILSON, TS, NC, TS, NCN>,
                           Stencil<TopStencil<ACT_WILSON, TS, NC, TS, NCN>>{}, g, tp);
      else if constexpr (split_rectangles<TS>())
        r = launch_split(c, "stout_top", split, g, tp);
      else
        r = launch_stencil(c, "stout_top", k_stout_top<ACT_IWASAKI, TS, NC, TS, NCN>,
                           k_stout_top_b<ACT_IWASAKI, TS, NC, TS, NCN>, split, g, tp);
    }
    if (r) return r;
  }
  for (int k = n - 1; k >= 1; --k) {
    StoutBwdArgs<TS, NC> bw{};
    bw.g = g;
    bw.U = lview<TS, NC>(Ulev(k), g);
    bw.L = aview<TS>(ws->L[cur], g);
    bw.W = mview<TS>(ws->W, g);
    bw.Ulo = lview<TS, NC>(Ulev(k - 1), g);
    bw.Qlo = aview<TS>(ws->Qs[k - 1], g);
    bw.Clo = mview<TS>(ws->Cs[k - 1], g);
    bw.Lout = aview<TS>(ws->L[1 - cur], g);
    bw.Wout = mview<TS>(ws->W, g);
    bw.rho = act.rho;
    if ((r = launch_stencil(c, "stout_bwd", k_stout_bwd<false, TS, NC, TS, R12B>,
                            k_stout_bwd_b<false, TS, NC, TS, R12B>, Stencil<BwdStencil<false, TS, NC, TS, R12B>>{}, g, bw)))
      return r;
    cur = 1 - cur;
  }
  StoutBwdArgs<TS, NC> bw{};
  bw.g = g;
  bw.U = lview<TS, NC>(U, g);
  bw.L = aview<TS>(ws->L[cur], g);
  bw.W = mview<TS>(ws->W, g);
  bw.rho = act.rho;
  bw.f = fa;
  if (act.mag) {
    if ((r = ws->need_Z())) return r;
    bw.Zout = mview<TS>(ws->Z, g);
  }
  if ((r = launch_stencil(c, "stout_bwd_force", k_stout_bwd<true, TS, NC, TS, R12L>,
                          k_stout_bwd_b<true, TS, NC, TS, R12L>, Stencil<BwdStencil<true, TS, NC, TS, R12L>>{}, g, bw)))
    return r;
  if (!act.mag) return MAG_OK;
  // constrained: F from the stored Z_0 with the link classes
  void* Fout = (out == OUT_F) ? F : nullptr;
  if (!Fout) {
    if ((r = ws->need_md())) return r;
    Fout = ws->F;
  }
  ForceZArgs<TS, NC> fz{fa, mview<TS>(ws->Z, g)};
  fz.f.F = aview<TS>(Fout, g);
  if ((r = launch(c, "force_from_z", k_force_from_Z<TS, NC, TS>, k_force_from_Z_b<TS, NC, TS>, grid_links(g), fz)))
    return r;
  if (out == OUT_PADD) return mom_update(c, g, std::is_same<TS, double>::value ? MAG_F64 : MAG_F32, P, Fout, eps);
  return MAG_OK;
}

// force_gradient_integrator (field-hmc.h:525-567). The auxiliary field is
// written directly by the first force of each half step (no copy), and the
// second force of each half step updates the momenta in its epilogue.
template <class TS, int NC>
int Ops<TS, NC>::fg(mag_ctx c, const Geom& g, void* U, void* P, const mag_action& act, int steps, double dt,
                    Workspace* ws) {
  int r;
  if ((r = ws->need_md())) return r;
  const double alpha = (3. - std::sqrt(3.)) * dt / 6.;
  const double beta = dt / std::sqrt(3.);
  const double gamma = (2. - std::sqrt(3.)) * dt * dt / 12.;
  if ((r = link_update(c, g, U, U, P, alpha, act.mag))) return r;
  for (int i = 0; i < steps; ++i) {
    for (int half = 0; half < 2; ++half) {
      if ((r = force(c, g, U, act, OUT_UAUX, nullptr, nullptr, ws->Uaux, gamma, ws))) return r;
      if ((r = force(c, g, ws->Uaux, act, OUT_PADD, nullptr, P, nullptr, 0.5 * dt, ws))) return r;
      if (half == 0 && (r = link_update(c, g, U, U, P, beta, act.mag))) return r;
    }
    const double a = (i < steps - 1) ? 2. * alpha : alpha;
    if ((r = link_update(c, g, U, U, P, a, act.mag))) return r;
  }
  return MAG_OK;
}

// leap_frog_integrator (field-hmc.h:569-587).
template <class TS, int NC>
int Ops<TS, NC>::leapfrog(mag_ctx c, const Geom& g, void* U, void* P, const mag_action& act, int steps, double dt,
                          Workspace* ws) {
  int r;
  if ((r = ws->need_md())) return r;
  if ((r = link_update(c, g, U, U, P, dt / 2., act.mag))) return r;
  for (int i = 0; i < steps; ++i) {
    if ((r = force(c, g, U, act, OUT_PADD, nullptr, P, nullptr, dt, ws))) return r;
    const double a = (i < steps - 1) ? dt : dt / 2.;
    if ((r = link_update(c, g, U, U, P, a, act.mag))) return r;
  }
  return MAG_OK;
}

template <class TS, int NC>
int Ops<TS, NC>::action_sums(mag_ctx c, const Geom& g, void* U, bool rect, int slot) {
  const int nb = (g.V + BLOCK - 1) / BLOCK;
  int r;
  if ((r = ensure_part(c, 2 * (size_t)nb))) return r;
  ActionArgs<TS, NC> aa{lview<TS, NC>(U, g), g, c->d_part, rect ? 1 : 0};
  if ((r = launch(c, "action", k_action_partial<TS, NC>, k_action_partial_b<TS, NC>, dim3(nb), aa))) return r;
  if ((r = final_reduce(c, c->d_part, nb, 2, 0, slot))) return r;
  return final_reduce(c, c->d_part + 1, nb, 2, 0, slot + 1);
}

// The Hamiltonian's action on the smeared field: smearing in FP64 from the
// stored links (FP32 or FP64), then the FP64 plaquette/rectangle sums.
template <class TS, int NC>
int Ops<TS, NC>::smeared_action_sums(mag_ctx c, const Geom& g, void* U, double rho, int n, bool rect, int slot) {
  if (n <= 0) return action_sums(c, g, U, rect, slot);
  Workspace* wsd = workspace(c, g, MAG_F64, 18);
  int r;
  if ((r = wsd->need_h(n))) return r;
  for (int k = 0; k < n; ++k) {
    void* dst = wsd->Uh[k & 1];
    if (k == 0) {
      StoutFwdArgs<TS, NC, double, 18> fw{g, lview<TS, NC>(U, g), aview<double>(nullptr, g),
                                          mview<double>(nullptr, g), lview<double, 18>(dst, g), rho, 0};
      r = launch_stencil(c, "stout_fwd_h", k_stout_fwd<TS, NC, double, 18, double>,
                         k_stout_fwd_b<TS, NC, double, 18, double>, Stencil<FwdStencil<TS, NC, double, 18, double>>{}, g, fw);
    } else {
      StoutFwdArgs<double, 18, double, 18> fw{g, lview<double, 18>(wsd->Uh[(k - 1) & 1], g),
                                              aview<double>(nullptr, g), mview<double>(nullptr, g),
                                              lview<double, 18>(dst, g), rho, 0};
      r = launch_stencil(c, "stout_fwd_h", k_stout_fwd<double, 18, double, 18, double>,
                         k_stout_fwd_b<double, 18, double, 18, double>, Stencil<FwdStencil<double, 18, double, 18, double>>{}, g, fw);
    }
    if (r) return r;
  }
  void* top = wsd->Uh[(n - 1) & 1];
  const int nb = (g.V + BLOCK - 1) / BLOCK;
  if ((r = ensure_part(c, 2 * (size_t)nb))) return r;
  ActionArgs<double, 18> aa{lview<double, 18>(top, g), g, c->d_part, rect ? 1 : 0};
  if ((r = launch(c, "action", k_action_partial<double, 18>, k_action_partial_b<double, 18>, dim3(nb), aa))) return r;
  if ((r = final_reduce(c, c->d_part, nb, 2, 0, slot))) return r;
  return final_reduce(c, c->d_part + 1, nb, 2, 0, slot + 1);
}

template <class TS, int NC>
int Ops<TS, NC>::smear(mag_ctx c, const Geom& g, void* Uout, void* U, double rho, int n, Workspace* ws) {
  int r;
  if ((r = ws->need_md())) return r;
  void* src = U;
  for (int k = 0; k < n; ++k) {
    void* dst = (k == n - 1) ? Uout : ((src == ws->Uaux) ? Uout : ws->Uaux);
    if (dst == src) dst = (src == Uout) ? ws->Uaux : Uout;
    StoutFwdArgs<TS, NC, TS, NC> fw{g, lview<TS, NC>(src, g), aview<TS>(nullptr, g), mview<TS>(nullptr, g),
                                    lview<TS, NC>(dst, g), rho, 0};
    if ((r = launch_stencil(c, "stout_fwd", k_stout_fwd<TS, NC, TS, NC, TS>, k_stout_fwd_b<TS, NC, TS, NC, TS>,
                            Stencil<FwdStencil<TS, NC, TS, NC, TS>>{}, g, fw,
                            std::is_same<TS, double>::value ? 8192 : SPLIT_MAX_SITES)))
      return r;
    src = dst;
  }
  if (src != Uout) return copy_dev(c, Uout, src, (size_t)g.V * 4 * NC * sizeof(TS));
  return MAG_OK;
}

template <class TS, int NC>
int Ops<TS, NC>::reunitarize(mag_ctx c, const Geom& g, void* U, int slot) {
  const int nb = (g.V + BLOCK - 1) / BLOCK;
  int r;
  if ((r = ensure_part(c, 4 * (size_t)nb))) return r;
  ReunitArgs<TS, NC> ra{lview<TS, NC>(U, g), g.V, c->d_part};
  if ((r = launch(c, "reunitarize", k_reunitarize<TS, NC>, k_reunitarize_b<TS, NC>, grid_links(g), ra))) return r;
  return final_reduce(c, c->d_part, 4 * nb, 1, 1, slot);
}

template <class TS, int NC>
int Ops<TS, NC>::max_diff(mag_ctx c, const Geom& g, void* A, void* B, int slot) {
  const int nb = (g.V + BLOCK - 1) / BLOCK;
  int r;
  if ((r = ensure_part(c, 4 * (size_t)nb))) return r;
  hipLaunchKernelGGL((k_max_diff<TS, NC>), grid_links(g), dim3(BLOCK), 0, c->stream, lview<TS, NC>(A, g),
                     lview<TS, NC>(B, g), g.V, c->d_part);
  CHECK_LAUNCH(c);
  return final_reduce(c, c->d_part, 4 * nb, 1, 1, slot);
}

template <class TS, int NC>
int Ops<TS, NC>::haar(mag_ctx c, const Geom& g, void* U, uint64_t seed) {
  hipLaunchKernelGGL((k_haar<TS, NC>), grid_links(g), dim3(BLOCK), 0, c->stream, lview<TS, NC>(U, g), g.V, seed);
  CHECK_LAUNCH(c);
  return MAG_OK;
}

template <class TS, int NC>
int Ops<TS, NC>::unit(mag_ctx c, const Geom& g, void* U) {
  hipLaunchKernelGGL((k_unit<TS, NC>), grid_links(g), dim3(BLOCK), 0, c->stream, lview<TS, NC>(U, g), g.V);
  CHECK_LAUNCH(c);
  return MAG_OK;
}

// Whether loops of spatial extents r (ascending) by T go one thread per loop.
// Calls with the sum read back, two wavefronts per loop over one thread per loop:
//   r = 0, T = 1 / 2                   20^4 1.04 / 1.00, 24^3 x 32 1.13 / 1.04, 32^4 1.18 / 1.20
//   FP32 R = T = 1                     24^4 0.97, 24^3 x 32 1.03, 28^4 1.03, 32^4 1.06
//   FP32 (2,0,0) / (1,1,0), T = 1      24^3 x 32 1.00 / 0.94, 32^4 1.01 / 1.02, 48^2 x 16 x 32 1.03 / 1.03
//   FP32 (1,1,1), T = 1 / 2 / 4        28^4 1.00 / 0.97 / 0.93, 32^4 1.12 / 1.09 / 1.05, 16^3 x 64 1.07 / 1.07 / 1.04
//   FP64 12 reals, R = 1 / 2 / 4, T = 1  28^4 0.84 / 0.82 / 0.79, 32^4 1.09 / 1.11 / 1.03
//   FP64 12 reals, (1,1,1), T = 2      32^4 0.89, 48^2 x 16 x 32 1.03, 32^3 x 48 1.07, 32^3 x 64 1.10
// and at 32^4 FP32 R = 4, T = 1 0.97, R = T = 2 0.92, FP64 18 reals R = T = 1 0.85.
template <class TS, int NC>
bool wloop_short(const Geom& g, const int r[3], int nperm, int T) {
  const long len = (long)r[0] + r[1] + r[2];
  const int V = g.V;
  if (len == 0) return T <= 2 && V > WLOOP_ROW_SITES;
  if (NC != 12) return false;
  if (std::is_same<TS, double>::value)
    return (V > 3 << 18 && T == 1 && r[1] == 0) || (V > 5 << 18 && nperm == 1 && len <= 6);
  return (V > 3 << 17 && len == 1 && T == 1) || (V > 3 << 18 && len <= 2 && T == 1) ||
         (len == 3 && nperm == 1 && (V > 3 << 18 || (V > WLOOP_ROW_SITES && g.L[3] > 32)));
}

template <class TS, int NC>
int Ops<TS, NC>::wilson_loop(mag_ctx c, const Geom& g, void* U, const int r3[3], int T, int slot, int* nperm) {
  WloopArgs a{};
  a.g = g;
  a.T = T;
  int rl[3] = {r3[0], r3[1], r3[2]};
  std::sort(rl, rl + 3);
  a.nperm = 0;
  do {
    for (int i = 0; i < 3; ++i) a.r[a.nperm][i] = rl[i];
    a.nperm++;
  } while (std::next_permutation(rl, rl + 3));
  *nperm = a.nperm;
  int r;
  if (wloop_short<TS, NC>(g, rl, a.nperm, T)) {
    const int nb = (g.V + BLOCK - 1) / BLOCK;
    if ((r = ensure_part(c, (size_t)nb))) return r;
    {
      KTimer t(c, "wilson_loop");
      hipLaunchKernelGGL((k_wilson_loop_short<TS, NC>), dim3(nb), dim3(BLOCK), 0, c->stream, lview<TS, NC>(U, g), a,
                         c->d_part);
    }
    CHECK_LAUNCH(c);
    return final_reduce(c, c->d_part, nb, 1, 0, slot);
  }
  const int nb = (g.V + WLOOP_SITES - 1) / WLOOP_SITES;
  // a row of the grid per permutation where the sites alone leave SIMDs idle
  // (R = T = 4: 8^4 15 -> 9 us, 12^4 17 -> 13; 16^4 27 -> 29, 24^3 x 32 186 -> 223)
  a.per = g.V <= WLOOP_ROW_SITES ? 1 : a.nperm;
  const int rows = (a.nperm + a.per - 1) / a.per;
  if ((r = ensure_part(c, (size_t)nb * rows))) return r;
  {
    KTimer t(c, "wilson_loop");
    hipLaunchKernelGGL((k_wilson_loop<TS, NC>), dim3(nb, rows), dim3(BLOCK), 0, c->stream, lview<TS, NC>(U, g), a,
                       c->d_part);
  }
  CHECK_LAUNCH(c);
  return final_reduce(c, c->d_part, nb * rows, 1, 0, slot);
}

}  // namespace mag
