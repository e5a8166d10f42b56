// pf_host_solve.hip -- the aggregation multigrid preconditioner (levels, cycle), the
// pressure projection with its PCG and FP64 refinement loop, and their entry points.
//
// One of the library's host files: pf_api.hip includes them in order into a single
// translation unit together with the kernel files, so every launch is a direct call.

namespace {

// ---- aggregation multigrid preconditioner (pf_mg.hip)

bool mg_cfg_valid(const pf_mg_cfg& q) {
  return q.sweeps >= 1 && q.sweeps <= 16 && q.coarsest_sweeps >= 1 && q.coarsest_sweeps <= 1024 &&
         q.omega > 0.0f && q.omega < 1.0f && q.correction > 0.0f && q.correction < 2.0f &&
         (q.chebyshev_ratio == 0.0f || (q.chebyshev_ratio > 1.0f && q.chebyshev_ratio <= 1000.0f));
}

// the built-in cycle (pf_set_multigrid changes a context's)
const pf_mg_cfg& mg_default_cfg() {
  static const pf_mg_cfg p{2, 32, 0.9f, 1.8f, 6.0f};
  return p;
}

MgLevel mg_level0(const pf_ctx* c) {
  MgLevel L;
  L.d = c->dc;
  L.nx = c->geom.nx; L.ny = c->geom.ny; L.nz = c->geom.nz;
  L.cd = c->cd32; L.cx = c->cx32; L.cy = c->cy32; L.cz = c->cz32; L.inv = c->invd32;
  return L;
}

MgLevel mg_level(const Ctx::MgBuf& b) {
  MgLevel L;
  L.d = b.d;
  L.nx = b.nx; L.ny = b.ny; L.nz = b.nz;
  L.cd = b.cd; L.cx = b.cx; L.cy = b.cy; L.cz = b.cz; L.inv = b.inv;
  return L;
}

// the coarse operators of the assembled system (levels allocated on first use:
// halving down to at most 4 cells a side; a grid of at most 4 cells a side has none)
void mg_free_level(Ctx::MgBuf& b) {
  float** arrs[8] = {&b.cd, &b.cx, &b.cy, &b.cz, &b.inv, &b.x, &b.r, &b.t};
  for (float** a : arrs) dfree(*a);
  for (auto& p : b.h) dfree(p);
  dfree(b.unscale);
}

// every multigrid buffer, or none: a partial allocation is released and the context
// keeps no levels, so a later call starts again from nothing
int mg_alloc(pf_ctx* c) {
  std::vector<Ctx::MgBuf> levels;
  float* t0 = nullptr;
  uint16_t* h[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
  float* mx = nullptr;
  float* unscale = nullptr;
  auto release = [&]() {
    for (auto& b : levels) mg_free_level(b);
    dfree(t0);
    for (auto& p : h) dfree(p);
    dfree(mx);
    dfree(unscale);
  };
  hipError_t e = hipSuccess;
  int nx = c->geom.nx, ny = c->geom.ny, nz = c->geom.nz;
  while (e == hipSuccess && std::max({nx, ny, nz}) > 4) {
    nx = (nx + 1) / 2; ny = (ny + 1) / 2; nz = (nz + 1) / 2;
    Ctx::MgBuf b;
    b.d = make_dims(nx, ny, nz);
    b.nx = nx; b.ny = ny; b.nz = nz;
    const long long n = b.d.nblocks * kBlockVol;
    float** arrs[8] = {&b.cd, &b.cx, &b.cy, &b.cz, &b.inv, &b.x, &b.r, &b.t};
    for (float** a : arrs)
      if (e == hipSuccess) e = dalloc(c, a, n);
    for (auto& p : b.h)
      if (e == hipSuccess) e = dalloc(c, &p, n);
    if (e == hipSuccess) e = dalloc(c, &b.unscale, 2);
    levels.push_back(b);
  }
  const long long n0 = c->dc.nblocks * kBlockVol;
  if (e == hipSuccess) e = dalloc(c, &t0, n0);
  for (auto& p : h)
    if (e == hipSuccess) e = dalloc(c, &p, n0);
  if (e == hipSuccess) e = dalloc(c, &mx, 2 * kMaxPartials);
  if (e == hipSuccess) e = dalloc(c, &unscale, 2);
  if (e != hipSuccess) {
    release();
    return fail(c, PF_ERR_NOMEM, std::string("multigrid levels: ") + hipGetErrorString(e));
  }
  c->mg = std::move(levels);
  c->mg_t0 = t0;
  for (int q = 0; q < 5; ++q) c->mg_h[q] = h[q];
  c->mg_mx = mx;
  c->mg_unscale = unscale;
  return PF_OK;
}

int mg_coarsen_from(pf_ctx* c, MgLevel F, size_t from);

// workgroups of the kernels that build a level: each reader sums one maximum per workgroup
unsigned mg_build_grid(long long cells) { return std::min<unsigned>(grid_for(cells, 256), 1024u); }

// a level's FP16 copy, scaled by the maxima of nmx workgroups in c->mg_mx
void mg_tohalf(pf_ctx* c, const MgLevel& L, uint16_t* const* hb, int nmx, float* unscale) {
  const long long n = L.d.nblocks * kBlockVol;
  _Float16* h[5];
  for (int q = 0; q < 5; ++q) h[q] = reinterpret_cast<_Float16*>(hb[q]);
  hipLaunchKernelGGL(k_mg_tohalf, dim3(mg_build_grid(n)), dim3(256), 0, c->stream, n, L.cd, L.cx, L.cy, L.cz, L.inv,
                     h[0], h[1], h[2], h[3], h[4], c->mg_mx, nmx, unscale);
}

int mg_build(pf_ctx* c) {
  if (!c->mg_t0) {
    int st = mg_alloc(c);
    if (st) return st;
  }
  // level 1's residual is restricted from the FLUID blocks only: the aggregates of the
  // other blocks stay zero through the solve
  if (!c->mg.empty()) HIP_TRY(c, fill_f32(c->stream, c->mg[0].r, 0.f, c->mg[0].d.nblocks * kBlockVol));
  // the FP16 level-0 operator of the row kernels
  {
    const long long n0 = c->dc.nblocks * kBlockVol;
    int nmx = c->mg_mx_n;  // left by the assembly
    if (!nmx) {
      nmx = (int)mg_build_grid(n0);
      hipLaunchKernelGGL(k_mg_absmax, dim3((unsigned)nmx), dim3(256), 0, c->stream, n0, c->cd32, c->cx32, c->cy32,
                         c->cz32, c->invd32, c->mg_mx);
    }
    c->mg_mx_n = 0;  // (the levels below use the array next)
    mg_tohalf(c, mg_level0(c), c->mg_h, nmx, c->mg_unscale);
    LAUNCH_CHECK(c);
  }
  return mg_coarsen_from(c, mg_level0(c), 0);
}

// levels c->mg[from..] by aggregation from F (the level above c->mg[from])
int mg_coarsen_from(pf_ctx* c, MgLevel F, size_t from) {
  for (size_t l = from; l < c->mg.size(); ++l) {
    Ctx::MgBuf& b = c->mg[l];
    const MgLevel Cl = mg_level(b);
    const unsigned g = mg_build_grid(b.d.nblocks * kBlockVol);
    hipLaunchKernelGGL(k_mg_coarsen, dim3(g), dim3(256), 0, c->stream, F, Cl, b.cd, b.cx, b.cy, b.cz, b.inv,
                       c->mg_mx);
    mg_tohalf(c, Cl, b.h, (int)g, b.unscale);
    LAUNCH_CHECK(c);
    F = Cl;
  }
  return PF_OK;
}

// The multires cycle's levels: the block grid (the uniform hierarchy's second level,
// c->mg[1]) from R S P, then the uniform levels below it.  Leaves of level 0..2 only.
int mr_mg_build(pf_ctx* c, const MrRowOp& op) {
  for (size_t a = 0; a < c->mr_leaves.size(); a += 4)
    if (c->mr_leaves[a] > 2)
      return fail(c, PF_ERR_ARG, "the multires multigrid takes leaves of level 0 to 2");
  if (!c->mg_t0) {
    int st = mg_alloc(c);
    if (st) return st;
  }
  if (c->mg.size() < 2) return fail(c, PF_ERR_ARG, "the multires multigrid needs a grid above 8 cells per axis");
  Ctx::MgBuf& b = c->mg[1];
  const long long nl = b.d.nblocks * kBlockVol;
  // block-grid cells of no listed block keep a zero residual through the solve
  HIP_TRY(c, fill_f32(c->stream, b.r, 0.f, nl));
  float** arrs[4] = {&b.cd, &b.cx, &b.cy, &b.cz};
  for (float** q : arrs) HIP_TRY(c, fill_f32(c->stream, *q, 0.f, nl));
  hipLaunchKernelGGL(k_mr_mg_coarse, dim3(grid_for(c->dc.nblocks, 4)), dim3(256), 0, c->stream, op, b.d, b.cd, b.cx,
                     b.cy, b.cz);
  LAUNCH_CHECK(c);
  const unsigned g = mg_build_grid(nl);
  hipLaunchKernelGGL(k_mg_inverse, dim3(g), dim3(256), 0, c->stream, mg_level(b), b.inv, c->mg_mx);
  mg_tohalf(c, mg_level(b), b.h, (int)g, b.unscale);
  LAUNCH_CHECK(c);
  return mg_coarsen_from(c, mg_level(b), 2);
}

// workgroups of the level-0 kernels: a multiple of 8 (the XCD-aware list walk), at
// most 1024 (the partials of r.z)
unsigned mg_grid0n(long long nlist) { return std::min(list_grid(nlist), 1024u); }
unsigned mg_grid0(const pf_ctx* c) { return mg_grid0n(c->npblk); }

// the weights of a smoothing pass's sweeps: all omega, or (a Chebyshev ratio r > 1)
// the reciprocals of the Chebyshev roots of degree nu on [lmax / r, lmax], lmax = 2
// (Gershgorin bound of D^-1 A), which damp that whole interval; the post-pass takes
// them in reverse order (they commute, so the cycle stays symmetric)
std::vector<float> mg_sweep_weights(const pf_ctx* c) {
  const int nu = c->mg_cfg.sweeps;
  const float cheb = c->mg_cfg.chebyshev_ratio;
  std::vector<float> w(nu, c->mg_cfg.omega);
  if (cheb > 1.0f) {
    const double b = 2.0, lo = b / cheb;
    for (int q = 0; q < nu; ++q) {
      const double lam = 0.5 * (b + lo) + 0.5 * (b - lo) * std::cos((2.0 * q + 1.0) * M_PI / (2.0 * nu));
      w[q] = (float)(1.0 / lam);
    }
  }
  return w;
}

// Whether the cycle from level l (1..nl) down runs in k_mg_tail: at least two sweeps (the
// row kernels' FP16 operator), at most a row per thread on level l, and all levels' blocks
// in its LDS.
bool mg_in_tail(const pf_ctx* c, int l) {
  const size_t nl = c->mg.size();
  long long blocks = 0;
  for (size_t q = (size_t)l - 1; q < nl; ++q) blocks += c->mg[q].d.nblocks;
  return c->mg_cfg.sweeps >= 2 && c->mg_cfg.sweeps <= kTailSweeps &&
         c->mg[(size_t)l - 1].d.nblocks * 16 <= kTailThreads && blocks <= kTailBlocks &&
         nl - (size_t)l + 1 <= kTailLevels;
}

float* mg_tail(pf_ctx* c, int l, const int* done, const std::vector<float>& wpre) {
  MgTailArgs a{};
  a.done = done;
  a.n = (int)c->mg.size() - l + 1;
  int off = 0;
  for (int q = 0; q < a.n; ++q) {
    const Ctx::MgBuf& b = c->mg[(size_t)(l - 1 + q)];
    MgTailLevel& L = a.lv[q];
    L.d = b.d;
    L.cd = reinterpret_cast<const _Float16*>(b.h[0]);
    L.cx = reinterpret_cast<const _Float16*>(b.h[1]);
    L.cy = reinterpret_cast<const _Float16*>(b.h[2]);
    L.cz = reinterpret_cast<const _Float16*>(b.h[3]);
    L.inv = reinterpret_cast<const _Float16*>(b.h[4]);
    L.unscale = b.unscale;
    L.rows = (int)b.d.nblocks * 16;
    L.off = off;
    off += L.rows * 4;
  }
  a.last = mg_level(c->mg.back());
  Ctx::MgBuf& top = c->mg[(size_t)l - 1];
  a.r = top.r;
  a.x = top.x;
  a.nu = c->mg_cfg.sweeps;
  for (int q = 0; q < a.nu; ++q) a.w[q] = wpre[(size_t)q];
  a.coarsest_sweeps = c->mg_cfg.coarsest_sweeps;
  a.omega = c->mg_cfg.omega;
  a.omega_c = c->mg_cfg.correction;
  hipLaunchKernelGGL(k_mg_tail, dim3(1), dim3(kTailThreads), 0, c->stream, a);
  return top.x;
}

// coarse levels: level l (1..nl) solves A_l x = r_l from zero (its buffer r holds r_l);
// returns the buffer that holds x.  (Two corrections per level -- a W-cycle -- cost
// more launches than they save iterations at 256^3, and twice the 1.8 over-correction
// stops converging.)
float* mg_coarse(pf_ctx* c, int l, const int* done, const std::vector<float>& wpre) {
  const int nl = (int)c->mg.size();
  const int nu = c->mg_cfg.sweeps;
  if (mg_in_tail(c, l)) return mg_tail(c, l, done, wpre);
  MgWalk wd{nullptr, 0, done};
  Ctx::MgBuf& b = c->mg[(size_t)l - 1];
  const MgLevel L = mg_level(b);
  float* x = b.x;
  float* t = b.t;
  if (l == nl) {
    hipLaunchKernelGGL(k_mg_coarsest, dim3(1), dim3(64), 0, c->stream, done, L, b.r, x, c->mg_cfg.omega,
                       c->mg_cfg.coarsest_sweeps);
    return x;
  }
  if (nu >= 2) {
    // by cell rows, as level 0 (k_mg_row over every block of the slab, the level's
    // FP16 operator): the two first sweeps fused, the restriction, then the
    // prolongation fused with the first post-sweep -- four passes instead of six
    Ctx::MgBuf& nb = c->mg[(size_t)l];
    MgRowArgs ra{};
    ra.list = nullptr;
    ra.nlist = b.d.nblocks;
    ra.done = done;
    ra.d = b.d;
    ra.dc = nb.d;
    ra.cd = reinterpret_cast<const _Float16*>(b.h[0]);
    ra.cx = reinterpret_cast<const _Float16*>(b.h[1]);
    ra.cy = reinterpret_cast<const _Float16*>(b.h[2]);
    ra.cz = reinterpret_cast<const _Float16*>(b.h[3]);
    ra.inv = reinterpret_cast<const _Float16*>(b.h[4]);
    ra.unscale = b.unscale;
    ra.r = b.r;
    ra.omega_c = c->mg_cfg.correction;
    ra.part = nullptr;
    const unsigned gw = list_grid(b.d.nblocks);
    float* cur = nullptr;
    float* nxt = x;
    auto flip = [&]() {
      cur = nxt;
      nxt = (cur == x) ? t : x;
    };
    ra.x = nullptr; ra.out = nxt;
    ra.omega_u = wpre[0];
    ra.omega = wpre[1];
    hipLaunchKernelGGL(k_mg_row<MG_FIRST2>, dim3(gw), dim3(256), 0, c->stream, ra);
    flip();
    for (int s2 = 2; s2 < nu; ++s2) {
      ra.x = cur; ra.out = nxt;
      ra.omega = wpre[(size_t)s2];
      hipLaunchKernelGGL(k_mg_row<MG_SWEEP>, dim3(gw), dim3(256), 0, c->stream, ra);
      flip();
    }
    ra.x = cur; ra.out = nb.r;
    hipLaunchKernelGGL(k_mg_row<MG_RESTRICT>, dim3(gw), dim3(256), 0, c->stream, ra);
    float* below = mg_coarse(c, l + 1, done, wpre);
    ra.x = cur; ra.out = nxt; ra.xc = below;
    ra.omega = wpre[(size_t)(nu - 1)];
    hipLaunchKernelGGL(k_mg_row<MG_PSWEEP>, dim3(gw), dim3(256), 0, c->stream, ra);
    flip();
    for (int s2 = 1; s2 < nu; ++s2) {
      ra.x = cur; ra.out = nxt;
      ra.omega = wpre[(size_t)(nu - 1 - s2)];
      hipLaunchKernelGGL(k_mg_row<MG_SWEEP>, dim3(gw), dim3(256), 0, c->stream, ra);
      flip();
    }
    return cur;
  }
  const unsigned g = std::min<unsigned>(grid_for(b.d.nblocks * kBlockVol, 256), 2048u);
  hipLaunchKernelGGL(k_mg_first, dim3(g), dim3(256), 0, c->stream, wd, L, b.r, x, wpre[0]);
  for (int s2 = 1; s2 < nu; ++s2) {
    hipLaunchKernelGGL(k_mg_sweep, dim3(g), dim3(256), 0, c->stream, wd, L, b.r, x, t, wpre[(size_t)s2], nullptr);
    std::swap(x, t);
  }
  Ctx::MgBuf& nb = c->mg[(size_t)l];
  hipLaunchKernelGGL(k_mg_restrict, dim3(g), dim3(256), 0, c->stream, wd, L, b.r, x, mg_level(nb), nb.r);
  float* below = mg_coarse(c, l + 1, done, wpre);
  hipLaunchKernelGGL(k_mg_prolong, dim3(g), dim3(256), 0, c->stream, wd, L, mg_level(nb), below, x,
                     c->mg_cfg.correction);
  for (int s2 = 0; s2 < nu; ++s2) {
    hipLaunchKernelGGL(k_mg_sweep, dim3(g), dim3(256), 0, c->stream, wd, L, b.r, x, t,
                       wpre[(size_t)(nu - 1 - s2)], nullptr);
    std::swap(x, t);
  }
  return x;
}

// level-1 quantities of one cycle, for training the correction weights: the restricted
// residual y before the scaling and the coarse solution B (S y) before the scaling
struct MgTrace {
  float* y = nullptr;
  float* h = nullptr;
};

// z = V-cycle(r) on the assembled system whose FLUID blocks are list[0..nlist);
// partial r.z (mg_grid0n(nlist) workgroups) in part[2 * kMaxPartials ...]; every
// kernel is skipped while *done
int mg_apply_on(pf_ctx* c, const uint32_t* list, long long nlist, const float* r, float* z, const int* done,
                double* part, const MgTrace* tr) {
  struct {
    int nu, coarsest;
    float omega, correction;
  } const P{c->mg_cfg.sweeps, c->mg_cfg.coarsest_sweeps, c->mg_cfg.omega, c->mg_cfg.correction};
  const int nl = (int)c->mg.size();
  MgWalk w0{list, nlist, done};
  const unsigned g0 = mg_grid0n(nlist);
  // kernels that write no partial may take more workgroups (up to 16 list blocks each)
  const unsigned gw = list_grid(nlist);
  const MgLevel L0 = mg_level0(c);
  double* const rz = part + 2 * kMaxPartials;
  // level 0 by cell rows when the slabs are below 2 GiB and there is a coarse level
  const bool rows = nl > 0 && c->dc.nblocks * kBlockVol * 4 < (1LL << 31);
  MgRowArgs ra{};
  ra.list = list;
  ra.nlist = nlist;
  ra.done = done;
  ra.d = c->dc;
  ra.cd = reinterpret_cast<const _Float16*>(c->mg_h[0]);
  ra.cx = reinterpret_cast<const _Float16*>(c->mg_h[1]);
  ra.cy = reinterpret_cast<const _Float16*>(c->mg_h[2]);
  ra.cz = reinterpret_cast<const _Float16*>(c->mg_h[3]);
  ra.inv = reinterpret_cast<const _Float16*>(c->mg_h[4]);
  ra.unscale = c->mg_unscale;
  ra.r = r;
  ra.omega = P.omega;
  const std::vector<float> wpre = mg_sweep_weights(c);
  auto wpost = [&](int q) { return wpre[(size_t)(P.nu - 1 - q)]; };
  ra.omega_c = P.correction;
  if (nl > 0) ra.dc = c->mg[0].d;
  // the level-0 kernels that write an iterate alternate between the work array and
  // z; the first one is chosen so that the last lands in z
  const int pre = rows ? (P.nu >= 2 ? P.nu - 1 : 1) : P.nu;
  const int writes = pre + P.nu;
  float* cur = nullptr;
  float* nxt = (writes & 1) ? z : c->mg_t0;
  auto flip = [&]() {
    cur = nxt;
    nxt = (cur == z) ? c->mg_t0 : z;
  };
  // pre-smoothing
  if (rows && P.nu >= 2) {
    ra.x = nullptr; ra.out = nxt; ra.part = nullptr;
    ra.omega_u = wpre[0];
    ra.omega = wpre[1];
    hipLaunchKernelGGL(k_mg_row<MG_FIRST2>, dim3(gw), dim3(256), 0, c->stream, ra);
    flip();
    for (int s2 = 2; s2 < P.nu; ++s2) {
      ra.x = cur; ra.out = nxt;
      ra.omega = wpre[(size_t)s2];
      hipLaunchKernelGGL(k_mg_row<MG_SWEEP>, dim3(gw), dim3(256), 0, c->stream, ra);
      flip();
    }
  } else {
    hipLaunchKernelGGL(k_mg_first, dim3(g0), dim3(256), 0, c->stream, w0, L0, r, nxt, wpre[0]);
    flip();
    const int more = nl > 0 ? P.nu - 1 : 2 * P.nu - 1;
    for (int s2 = 0; s2 < more; ++s2) {
      const bool last = nl == 0 && s2 == more - 1;
      const int q = s2 + 1;  // sweep q of pre (q < nu) and post (q - nu) smoothing
      const float om = q < P.nu ? wpre[(size_t)q] : wpost(q - P.nu);
      hipLaunchKernelGGL(k_mg_sweep, dim3(g0), dim3(256), 0, c->stream, w0, L0, r, cur, nxt, om,
                         last ? rz : nullptr);
      flip();
    }
  }
  if (nl == 0) {
    LAUNCH_CHECK(c);
    return PF_OK;
  }
  // restriction to level 1
  if (rows) {
    ra.x = cur; ra.out = c->mg[0].r; ra.part = nullptr;
    hipLaunchKernelGGL(k_mg_row<MG_RESTRICT>, dim3(gw), dim3(256), 0, c->stream, ra);
  } else {
    hipLaunchKernelGGL(k_mg_restrict, dim3(g0), dim3(256), 0, c->stream, w0, L0, r, cur, mg_level(c->mg[0]),
                       c->mg[0].r);
  }
  // per-aggregate correction scaling: S on the restricted residual ...
  const long long n1 = c->mg[0].d.nblocks * kBlockVol;
  if (tr && tr->y)
    HIP_TRY(c, hipMemcpyAsync(tr->y, c->mg[0].r, sizeof(float) * (size_t)n1, hipMemcpyDeviceToDevice, c->stream));
  if (c->mg_cs_active)
    hipLaunchKernelGGL(k_mg_scale, dim3(std::min<unsigned>(grid_for(n1, 256), 2048u)), dim3(256), 0, c->stream, n1,
                       c->mg[0].r, c->mg_cs_active, done);
  float* const res1 = mg_coarse(c, 1, done, wpre);
  if (tr && tr->h)
    HIP_TRY(c, hipMemcpyAsync(tr->h, res1, sizeof(float) * (size_t)n1, hipMemcpyDeviceToDevice, c->stream));
  // ... and on the correction (P S B_1 S P^T stays symmetric)
  if (c->mg_cs_active)
    hipLaunchKernelGGL(k_mg_scale, dim3(std::min<unsigned>(grid_for(n1, 256), 2048u)), dim3(256), 0, c->stream, n1,
                       res1, c->mg_cs_active, done);
  // level 0: prolong and post-smooth, the last sweep into z with the partial r.z
  if (rows) {
    ra.x = cur; ra.out = nxt; ra.xc = res1; ra.part = P.nu == 1 ? rz : nullptr;
    ra.omega = wpost(0);
    hipLaunchKernelGGL(k_mg_row<MG_PSWEEP>, dim3(ra.part ? g0 : gw), dim3(256), 0, c->stream, ra);
    flip();
    for (int s2 = 1; s2 < P.nu; ++s2) {
      ra.x = cur; ra.out = nxt; ra.part = s2 == P.nu - 1 ? rz : nullptr;
      ra.omega = wpost(s2);
      hipLaunchKernelGGL(k_mg_row<MG_SWEEP>, dim3(ra.part ? g0 : gw), dim3(256), 0, c->stream, ra);
      flip();
    }
  } else {
    hipLaunchKernelGGL(k_mg_prolong, dim3(g0), dim3(256), 0, c->stream, w0, L0, mg_level(c->mg[0]), res1, cur,
                       P.correction);
    for (int s2 = 0; s2 < P.nu; ++s2) {
      hipLaunchKernelGGL(k_mg_sweep, dim3(g0), dim3(256), 0, c->stream, w0, L0, r, cur, nxt, wpost(s2),
                         s2 == P.nu - 1 ? rz : nullptr);
      flip();
    }
  }
  LAUNCH_CHECK(c);
  if (cur != z) return fail(c, PF_ERR_STATE, "multigrid: cycle did not end in z");
  return PF_OK;
}

int mg_apply(pf_ctx* c, const float* r, float* z, const int* done, double* part) {
  return mg_apply_on(c, c->pblk, c->npblk, r, z, done, part, nullptr);
}

// the assembled multires operator by cell rows (pf_mr_row.hip)
MrRowOp mr_row_op(const pf_ctx* c) {
  MrRowOp o;
  o.dc = c->dc;
  o.info = c->mr_info;
  o.cd = c->cd32; o.cx = c->cx32; o.cy = c->cy32; o.cz = c->cz32; o.inv = c->invd32;
  o.cs = c->mr_cs;
  return o;
}

// workgroups: four list blocks to a wave, at most 1024 (every workgroup sums that many
// partials of five quantities), a multiple of 8 (one share per XCD)
unsigned cg_grid(long long nlist) {
  return (unsigned)std::clamp<long long>((((nlist + 15) / 16 + 7) / 8) * 8, 8, 1024);
}

// the same without a sum to keep small
unsigned mr_grid_wide(long long nlist) {
  return (unsigned)std::clamp<long long>((((nlist + 15) / 16 + 7) / 8) * 8, 8, 8192);
}

// z = the multires cycle on r over the listed blocks: nu sweeps on S, the block sums of
// the residual onto the block grid, the uniform cycle from there, the prolongation and
// nu sweeps back, the last into z with the partial r.z (cg_grid workgroups) in slot 2 of
// part; skipped while *done
int mr_mg_apply(pf_ctx* c, const MrRowOp& op, const VecArgs& va, const float* r, float* z, const int* done,
                double* part) {
  const int nu = std::max(1, c->mg_cfg.sweeps);
  std::vector<float> wpre = mg_sweep_weights(c);
  wpre.resize((size_t)nu, c->mg_cfg.omega);
  Ctx::MgBuf& b = c->mg[1];
  MrCycleArgs a{};
  a.list = va.list;
  a.nlist = va.nlist;
  a.done = done;
  a.op = op;
  a.dcc = b.d;
  a.r = r;
  a.omega_c = c->mg_cfg.correction;
  const unsigned g = cg_grid(va.nlist), gw = mr_grid_wide(va.nlist);
  // the kernels that write an iterate alternate between the work array and z; the first
  // is chosen so that the last lands in z
  const int writes = (nu >= 2 ? nu - 1 : 1) + nu;
  float* cur = nullptr;
  float* nxt = (writes & 1) ? z : c->mg_t0;
  auto flip = [&]() {
    cur = nxt;
    nxt = (cur == z) ? c->mg_t0 : z;
  };
  a.out = nxt;
  if (nu >= 2) {
    a.omega_u = wpre[0];
    a.omega = wpre[1];
    hipLaunchKernelGGL(k_mr_cycle<MG_FIRST2>, dim3(gw), dim3(256), 0, c->stream, a);
  } else {
    a.omega = wpre[0];
    hipLaunchKernelGGL(k_mr_cycle_first, dim3(gw), dim3(256), 0, c->stream, a);
  }
  flip();
  for (int q = 2; q < nu; ++q) {
    a.x = cur; a.out = nxt;
    a.omega = wpre[(size_t)q];
    hipLaunchKernelGGL(k_mr_cycle<MG_SWEEP>, dim3(gw), dim3(256), 0, c->stream, a);
    flip();
  }
  a.x = cur;
  a.out = b.r;
  hipLaunchKernelGGL(k_mr_cycle<MG_RESTRICT>, dim3(gw), dim3(256), 0, c->stream, a);
  a.xc = mg_coarse(c, 2, done, wpre);
  for (int q = 0; q < nu; ++q) {
    a.x = cur; a.out = nxt;
    a.omega = wpre[(size_t)(nu - 1 - q)];
    a.part = q == nu - 1 ? part + 2 * kMaxPartials : nullptr;
    const dim3 grid(a.part ? g : gw);
    if (q == 0)
      hipLaunchKernelGGL(k_mr_cycle<MG_PSWEEP>, grid, dim3(256), 0, c->stream, a);
    else
      hipLaunchKernelGGL(k_mr_cycle<MG_SWEEP>, grid, dim3(256), 0, c->stream, a);
    flip();
  }
  LAUNCH_CHECK(c);
  if (cur != z) return fail(c, PF_ERR_STATE, "multires multigrid: cycle did not end in z");
  return PF_OK;
}

// ---- the Jacobi PCG in one kernel per iteration (pf_cg.hip)

// what the next launch reads: which scalars, sums (nsums partials of each) and vectors
struct CgState {
  int cur = 0, sums = 0, nsums = 0, par = 0;
  unsigned long long seq = 0;  // launches so far
};

float* cg_r(const pf_ctx* c, int par) { return par ? c->z32 : c->r32; }
float* cg_q(const pf_ctx* c, int par) { return par ? c->cgq : c->Ap; }
float* cg_p(const pf_ctx* c, int par) { return par ? c->pB : c->pA; }
double* cg_sums(const pf_ctx* c, int sums) { return c->partial + sums * CG_SUMS * kMaxPartials; }

CgArgs cg_args(const pf_ctx* c, const CgState& g, const VecArgs& va) {
  CgArgs a{};
  a.dc = c->dc; a.list = va.list; a.nlist = va.nlist;
  a.x = c->x32;
  a.r = cg_r(c, g.par); a.q = cg_q(c, g.par); a.p = cg_p(c, g.par);
  a.rn = cg_r(c, g.par ^ 1); a.qn = cg_q(c, g.par ^ 1); a.pn = cg_p(c, g.par ^ 1);
  a.inv = c->invd32; a.cd = c->cd32; a.cx = c->cx32; a.cy = c->cy32; a.cz = c->cz32;
  a.sums = cg_sums(c, g.sums);
  a.sums_out = cg_sums(c, g.sums ^ 1);
  a.nsums = g.nsums;
  a.in = c->sc + g.cur;
  a.out = c->sc + (g.cur ^ 1);
  a.word = c->cg_word;
  a.seq = g.seq;
  return a;
}

// the FP64 residual into the buffers that the next launch reads, the direction zero
// before the first iteration
int cg_load(pf_ctx* c, CgState& g, VecArgs va, unsigned G, const double* r_src, bool first) {
  va.part = cg_sums(c, g.sums);
  if (c->mr) {
    g.nsums = (int)cg_grid(va.nlist);
    hipLaunchKernelGGL(k_mr_load, dim3((unsigned)g.nsums), dim3(256), 0, c->stream, va, mr_row_op(c), r_src, c->x32,
                       cg_r(c, g.par), first ? cg_p(c, g.par) : nullptr, first ? cg_q(c, g.par) : nullptr, 1);
    LAUNCH_CHECK(c);
    return PF_OK;
  }
  g.nsums = (int)std::min(G, 1024u);
  hipLaunchKernelGGL(k_cg_load, dim3((unsigned)g.nsums), dim3(256), 0, c->stream, va, r_src, c->x32, cg_r(c, g.par),
                     first ? cg_p(c, g.par) : nullptr, first ? cg_q(c, g.par) : nullptr, c->invd32);
  LAUNCH_CHECK(c);
  return PF_OK;
}

int cg_start(pf_ctx* c, CgState& g, const VecArgs& va, unsigned G, const double* r_src, double delta2,
             double tol2_abs, int budget, int between) {
  g.cur = g.par = 0;
  hipLaunchKernelGGL(k_cg_begin, dim3(1), dim3(1), 0, c->stream, c->sc, 1, delta2, tol2_abs, budget, between);
  return cg_load(c, g, va, G, r_src, true);
}

// after a residual replacement (g and sc_host hold the paused state)
int cg_resume(pf_ctx* c, CgState& g, const VecArgs& va, unsigned G) {
  hipLaunchKernelGGL(k_cg_begin, dim3(1), dim3(1), 0, c->stream, c->sc + g.cur, 2, 0.0, 0.0, 0, 0);
  g.par ^= 1;
  return cg_load(c, g, va, G, c->r64, false);
}

// Iterations until the recursion pauses; the state is then in sc_host.  The host follows
// through one word that each launch stores in pinned memory and stays at most `ahead`
// launches in front of it, so no iteration waits for the host and a pause costs at most
// that many launches that return at once.  While residuals are recorded, the stream is
// drained every `ahead` iterations instead and `look` sees the residual.
template <typename Look>
int cg_run(pf_ctx* c, CgState& g, const VecArgs& va, int check, const Look& look) {
  const int ahead = std::clamp(check, 1, 16);
  const unsigned grid = cg_grid(va.nlist);
  volatile unsigned long long* word = c->cg_word;
  *word = 2 * g.seq;  // (the stream is idle: no launch of an earlier segment is left)
  auto fetch = [&]() -> int {
    HIP_TRY(c, hipMemcpyAsync(c->sc_host, c->sc + g.cur, sizeof(SolveScalars), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    // (launches after the pause moved nothing)
    if (c->sc_host->done) g.par = c->sc_host->par;
    return PF_OK;
  };
  for (int launched = 1;; ++launched) {
    ++g.seq;
    const CgArgs a = cg_args(c, g, va);
    const long long ki = kbegin(c, PF_K_PCG_SPMV);
    if (c->mr)
      hipLaunchKernelGGL(k_mr_cg_iter, dim3(grid), dim3(256), 0, c->stream, a, mr_row_op(c));
    else if (grid <= 512)
      hipLaunchKernelGGL(k_cg_iter<true>, dim3(grid), dim3(256), 0, c->stream, a);
    else
      hipLaunchKernelGGL(k_cg_iter<false>, dim3(grid), dim3(256), 0, c->stream, a);
    kend(c, ki);
    LAUNCH_CHECK(c);
    g.cur ^= 1;
    g.sums ^= 1;
    g.par ^= 1;
    g.nsums = (int)grid;
    if (c->snap_cap > 0) {
      if (launched % ahead) continue;
      int st = fetch();
      if (st) return st;
      const SolveScalars& S = *c->sc_host;
      st = look(S.iter, cg_r(c, S.par));
      if (st || S.done) return st;
      continue;
    }
    unsigned long long w = *word;
    for (unsigned spin = 0; !(w & 1) && (w >> 1) + ahead < g.seq; w = *word) {
      // (a launch that failed would never store its word: the stream says so)
      if ((++spin & 0xffff) == 0) {
        const hipError_t e = hipStreamQuery(c->stream);
        if (e != hipSuccess && e != hipErrorNotReady) HIP_TRY(c, e);
        if (e == hipSuccess && (*word >> 1) < g.seq) return fail(c, PF_ERR_HIP, "solver launches left no state");
      }
    }
    if (w & 1) return fetch();
  }
}

// Workgroups of the pin scan: each ends in atomics on the same three words (about 12 ns
// each), and walks its blocks one wait after another, so neither many nor few: 64 blocks
// each, 512 to 2048 of them.  With 512, 1024 and 2048 the scan takes 17, 27 and 27 us at
// 64^3, 39, 39 and 57 at 128^3, 118, 80 and 80 at 192^3, 278, 180 and 126 at 256^3, the
// multires one 2.04, 1.30 and 0.86 ms at 512^3 effective.  (A look at the word before the atomic
// is a read of what other XCDs change: 170 us instead of 126.)
unsigned pin_grid(long long npb) {
  return std::min<unsigned>(list_grid(npb), (unsigned)std::clamp<long long>(npb / 64, 512, 2048) & ~7u);
}

// single: the single-phase unit-density projection (ph unused, cdiv ignored);
// c->mr: the multires finite-volume projection, stopping when
// |rhs - A x|_inf < max(cfg->tol, mr_rel_tol * |rhs|_inf)
int run_project(pf_ctx* c, const pf_phase* ph, double dt, const pf_solve_cfg* cfg, double cdiv,
                pf_solve_stats* out, bool timing, int ev_assemble, int ev_solve, int ev_vel,
                bool single = false, double mr_rel_tol = 0.0) {
  const bool mr = c->mr;
  if (cfg->precond < PF_PRECOND_JACOBI || cfg->precond > PF_PRECOND_MULTIGRID)
    return fail(c, PF_ERR_ARG, "unknown preconditioner");
  pf_solve_stats S;
  std::memset(&S, 0, sizeof(S));
  S.pinned_cell = -1;
  const Geom& g = c->geom;
  const long long nb = c->dc.nblocks;
  // 1. the blocks holding FLUID cells (flags; sorted list below)
  c->mg_mx_n = 0;
  uint8_t* flag8 = reinterpret_cast<uint8_t*>(c->blk_flag32);
  hipLaunchKernelGGL(k_fluid_flags, dim3(grid_for(nb, 4)), dim3(256), 0, c->stream, c->dc, c->marker, flag8);
  LAUNCH_CHECK(c);
  // 2. blocks of the previous solve return to zero; the pressure field is cleared
  if (c->npblk_prev > 0) {
    const bool warm = cfg->warm_start != 0;
    if (warm) {
      hipLaunchKernelGGL(k_warm_save, dim3(grid_for(c->npblk_prev, 4)), dim3(256), 0, c->stream, c->pblk_prev,
                         c->npblk_prev, c->f[F_P], c->x64);
      LAUNCH_CHECK(c);
    }
    ZeroArgs z{};
    z.list = c->pblk_prev;
    z.nlist = c->npblk_prev;
    // Cleared on every block of the previous solve: the pressure and the iteration
    // vectors (with the multigrid work array: its values at cells outside the next
    // system are read, times a zero coupling, by the level-0 sweeps, so none may stay
    // non-finite).  Only on the blocks that leave the system (sparse path): the
    // assembly's outputs, which k_assemble writes on all 64 cells of every listed
    // block, x64 (k_ir_start writes it there) and r64 (written before it is read).
    int nf = 0;
    for (float* p : {c->f[F_P], c->x32, c->r32, c->z32, c->pA, c->pB, c->Ap, c->mg_t0, c->cgq})
      if (p) z.f32[nf++] = p;
    z.nf32_all = nf;
    for (float* p : {c->cd32, c->cx32, c->cy32, c->cz32, c->invd32}) z.f32[nf++] = p;
    z.nf32 = nf;
    double* f64[7] = {c->b64, c->r64, c->cd64, c->cx64, c->cy64, c->cz64, c->x64};
    for (int q = 0; q < 7; ++q) z.f64[q] = f64[q];
    z.nf64 = warm ? 6 : 7;  // a warm start keeps x64 (the saved pressure)
    z.keep = mr ? nullptr : flag8;
    hipLaunchKernelGGL(k_zero_blocks, dim3(grid_for(c->npblk_prev, 4)), dim3(256), 0, c->stream, z);
    LAUNCH_CHECK(c);
  }
  HIP_TRY(c, fill_u8(c->stream, c->act[F_P], 0, nb));
  // 3. the sorted list
  HIP_TRY(c, compact_flags_morton(*c, c->dc, flag8, c->pblk, c->u32_dev + 2));
  HIP_TRY(c, fill_u32(c->stream, c->u32_dev, 0u, 1));
  HIP_TRY(c, fill_u32(c->stream, c->u32_dev + 1, 0xffffffffu, 1));
  HIP_TRY(c, fill_u32(c->stream, c->u32_dev + 4, 0u, 1));
  HIP_TRY(c, hipMemcpyAsync(c->u32_host, c->u32_dev, sizeof(uint32_t) * 4, hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(c, hipStreamSynchronize(c->stream));
  const long long npb = c->u32_host[2];
  c->npblk = npb;
  if (npb == 0) {
    std::swap(c->pblk, c->pblk_prev);
    c->npblk_prev = 0;
    c->npblk = 0;
    S.converged = 1;
    record(c, timing, ev_assemble);
    record(c, timing, ev_solve);
    record(c, timing, ev_vel);
    if (out) *out = S;
    return PF_OK;
  }
  // learned preconditioner: the multigrid cycle with per-aggregate correction weights
  // from the attached network; its tiles and features of this system are built for
  // the solve or for recording training snapshots
  const bool want_learned = cfg->precond == PF_PRECOND_LEARNED;
  if (want_learned && !c->lpc) return fail(c, PF_ERR_STATE, "precond = learned but no network attached (pf_lpc_attach)");
  if (want_learned && mr) return fail(c, PF_ERR_ARG, "the learned preconditioner runs on the sparse path only");
  const bool want_mg = cfg->precond == PF_PRECOND_MULTIGRID;
  const bool lpc_system = c->lpc && (want_learned || c->snap_cap > 0);
  c->tiles_valid = false;
  c->nsnap = 0;
  c->snap_last_iter = -1;
  if (lpc_system) {
    int s2 = lpc_features_alloc(c);
    if (!s2) s2 = lpc_cw_tiles(c, c->pblk, npb);
    if (s2) return s2;
  }
  // From here on these blocks' arrays hold this system, so the next solve clears them,
  // also after an error: a stale coupling in a block outside its list would join a listed
  // neighbour's row.
  struct Listed {
    pf_ctx* c;
    ~Listed() {
      std::swap(c->pblk, c->pblk_prev);
      c->npblk_prev = c->npblk;
    }
  } listed{c};
  ProjArgs pa;
  pa.g = g; pa.dc = c->dc; pa.du = c->du; pa.dv = c->dv; pa.dw = c->dw;
  pa.marker = c->marker; pa.list = c->pblk; pa.nlist = npb;
  const pf_phase unit_phase = {1.0, 1.0, 1.0, 1.0};
  pa.ph = phase_k(single ? &unit_phase : ph);
  pa.scale = dt / (g.dx * g.dx);
  pa.cdiv = single ? 0.0 : cdiv;
  pa.pin = c->u32_dev;
  pa.single = single ? 1 : 0;
  const unsigned G = list_grid(npb);
  const bool refmode = mr && c->mr_cfg && c->mr_cfg->mode == PF_MR_SOLVE_REFERENCE;
  if (mr) {
    c->mr_detail = pf_mr_solve_detail{};
    c->mr_detail.coarse_preconditioner_auto_disable_iteration = -1;
  }
  if (refmode) {
    if (!c->mrf) HIP_TRY(c, dalloc(c, &c->mrf, (long long)kMrfVectors * c->dc.nblocks * kBlockVol));
    if (!c->mr_pin_dev) HIP_TRY(c, dalloc(c, &c->mr_pin_dev, 1));
    if (!c->mr_pin_host) HIP_TRY(c, hipHostMalloc((void**)&c->mr_pin_host, sizeof(long long)));
    HIP_TRY(c, fill_u32(c->stream, reinterpret_cast<uint32_t*>(c->mr_pin_dev), 0xffffffffu, 2));
  }
  if (mr) {
    MrAsm ma{};
    ma.m = mr_grid(c);
    ma.list = c->pblk; ma.nlist = npb;
    ma.ph = phase_k(ph);
    ma.dt = dt; ma.cdiv = cdiv; ma.pin = c->u32_dev;
    ma.u = c->f[F_U]; ma.v = c->f[F_V]; ma.w = c->f[F_W];
    ma.mu = c->f[F_MU]; ma.mv = c->f[F_MV]; ma.mw = c->f[F_MW];
    ma.part = c->partial;
    if (refmode) {
      // the couplings are written per fine face, so the arrays start at zero
      const Dims* fd[3] = {&c->du, &c->dv, &c->dw};
      for (int a = 0; a < 3; ++a) {
        const long long n = fd[a]->nblocks * kBlockVol;
        if (!c->mr_cf64[a]) HIP_TRY(c, dalloc(c, &c->mr_cf64[a], n));
        HIP_TRY(c, fill_f64(c->stream, c->mr_cf64[a], 0.0, n));
        ma.cf64[a] = c->mr_cf64[a];
      }
      ma.b64 = c->b64; ma.cd64 = c->cd64; ma.vol64 = c->mr_vol64;
      const long long ncell = c->dc.nblocks * kBlockVol;
      ma.rref = c->mrf + 12 * ncell;
      ma.dref = c->mrf + 13 * ncell;
      ma.vtrue = c->mrf + 14 * ncell;
      ma.pin_cell = c->mr_pin_dev;
    }
    HIP_TRY(c, fill_u32(c->stream, c->u32_dev + 5, 0u, 1));
    hipLaunchKernelGGL(k_mr_pin, dim3(pin_grid(npb)), dim3(256), 0, c->stream, ma);
    LAUNCH_CHECK(c);
    if (refmode) {
      TIMED(c, PF_K_ASSEMBLE, hipLaunchKernelGGL(k_mr_assemble, dim3(G), dim3(256), 0, c->stream, ma));
    } else {
      MrCellOut mo;
      mo.b64 = c->b64; mo.cd64 = c->cd64; mo.cx64 = c->cx64; mo.cy64 = c->cy64; mo.cz64 = c->cz64;
      mo.vol64 = c->mr_vol64;
      mo.cd32 = c->cd32; mo.cx32 = c->cx32; mo.cy32 = c->cy32; mo.cz32 = c->cz32; mo.inv32 = c->invd32;
      mo.cs = c->mr_cs;
      // (a neighbour outside the list has no couplings)
      HIP_TRY(c, fill_f32(c->stream, reinterpret_cast<float*>(c->mr_cs), 0.f, 4 * c->dc.nblocks));
      TIMED(c, PF_K_ASSEMBLE, hipLaunchKernelGGL(k_mr_assemble_cells, dim3(G), dim3(256), 0, c->stream, ma, mo));
    }
    LAUNCH_CHECK(c);
  } else {
  hipLaunchKernelGGL(k_pin_detect, dim3(pin_grid(npb)), dim3(256), 0, c->stream, pa);
  LAUNCH_CHECK(c);
  AsmOut ao;
  ao.b64 = c->b64; ao.cd64 = c->cd64; ao.cx64 = c->cx64; ao.cy64 = c->cy64; ao.cz64 = c->cz64;
  ao.cd32 = c->cd32; ao.cx32 = c->cx32; ao.cy32 = c->cy32; ao.cz32 = c->cz32; ao.invd32 = c->invd32;
  ao.u = c->f[F_U]; ao.v = c->f[F_V]; ao.w = c->f[F_W];
  ao.mu = c->f[F_MU]; ao.mv = c->f[F_MV]; ao.mw = c->f[F_MW];
  ao.part = c->partial;
  ao.fbeta = lpc_system ? c->fbeta : nullptr;
  ao.fphi = lpc_system ? c->fphi : nullptr;
  // the FP16 scaling of a multigrid build that may follow needs the operator's maxima:
  // the assembly reduces them from the values it writes (cells outside the list are zero)
  const bool want_mx = want_mg || want_learned || lpc_system;
  ao.mx = nullptr;
  if (want_mx) {
    if (!c->mg_t0) {
      int s2 = mg_alloc(c);
      if (s2) return s2;
    }
    ao.mx = c->mg_mx;
  }
  TIMED(c, PF_K_ASSEMBLE, hipLaunchKernelGGL(k_assemble, dim3(G), dim3(256), 0, c->stream, pa, ao));
  LAUNCH_CHECK(c);
  if (want_mx) c->mg_mx_n = (int)G;
  }
  // red[2] = sum b^2; red[3] = max |b| (sparse assembly only)
  hipLaunchKernelGGL(k_reduce_slots, dim3(mr ? 1 : 2), dim3(256), 0, c->stream, c->partial, (int)G, 2u,
                     c->red + 2);
  LAUNCH_CHECK(c);
  record(c, timing, ev_assemble);

  // 4. FP64 iterative refinement around the FP32 Jacobi PCG
  VecArgs va;
  va.dc = c->dc; va.list = c->pblk; va.nlist = npb; va.sc = c->sc; va.part = c->partial;
  hipLaunchKernelGGL(k_ir_start, dim3(G), dim3(256), 0, c->stream, va, c->x64, c->invd32, cfg->warm_start);
  LAUNCH_CHECK(c);
  MrRowOp mop{};
  MrRowOp64 mrow64{};
  MrOp64 mop64{};
  if (mr) {
    mop = mr_row_op(c);
    mrow64.dc = c->dc; mrow64.info = c->mr_info; mrow64.vol = c->mr_vol64;
    mrow64.cd = c->cd64; mrow64.cx = c->cx64; mrow64.cy = c->cy64; mrow64.cz = c->cz64;
    mop64.m = mr_grid(c);
    mop64.cd = c->cd64; mop64.vol = c->mr_vol64;
    for (int a = 0; a < 3; ++a) mop64.cf[a] = c->mr_cf64[a];
  }
  const double* r_src = c->r64;  // the FP64 residual the next (re)start loads
  auto residual = [&]() -> int {
    if (mr && refmode)
      TIMED(c, PF_K_RESIDUAL64,
            hipLaunchKernelGGL(k_mr_residual64, dim3(G), dim3(256), 0, c->stream, va, mop64, c->b64, c->x64, c->r64));
    else if (mr)
      TIMED(c, PF_K_RESIDUAL64,
            hipLaunchKernelGGL(k_mr_residual, dim3(G), dim3(256), 0, c->stream, va, mrow64, c->b64, c->x64, c->r64));
    else
    TIMED(c, PF_K_RESIDUAL64,
          hipLaunchKernelGGL(k_residual64, dim3(G), dim3(256), 0, c->stream, va, c->b64, c->x64, c->r64, c->cd64,
                             c->cx64, c->cy64, c->cz64));
    LAUNCH_CHECK(c);
    hipLaunchKernelGGL(k_reduce_slots, dim3(2), dim3(256), 0, c->stream, c->partial, (int)G, 2u, c->red);
    LAUNCH_CHECK(c);
    r_src = c->r64;
    return read_small(c);
  };
  // From x = 0 (no warm start) the FP64 residual is b itself: its sum of squares and max
  // norm come from the assembly's reduction (the same partition and order, so the same
  // bits), and the first load reads b64 -- no residual pass.
  const bool zero_start = !mr && !cfg->warm_start;
  int st = zero_start ? read_small(c) : residual();
  if (st) return st;
  if (zero_start) r_src = c->b64;
  const double bnorm2 = c->red_host[2];
  double rr = zero_start ? c->red_host[2] : c->red_host[0], rmax = zero_start ? c->red_host[3] : c->red_host[1];
  S.rhs_norm2 = bnorm2;
  S.initial_max_residual = rmax;
  S.pinned = c->u32_host[0] == 0;
  S.pinned_cell = S.pinned ? (int64_t)c->u32_host[1] : -1;
  const int max_iters = std::max(cfg->max_iters, 0);
  const int max_updates = cfg->max_outer > 0 ? cfg->max_outer : 200;
  // (a multigrid iteration costs several products: check at least every 4)
  const int check_base = cfg->check_every > 0 ? cfg->check_every : 8;
  const int check = (want_mg || want_learned) ? std::min(check_base, 4) : check_base;
  const double delta = (cfg->inner_rel_tol > 0 && cfg->inner_rel_tol < 1) ? cfg->inner_rel_tol : 0.1;
  // the multires rule: max(absolute, relative * initial max residual), with x0 = 0
  // (multires_pressure3d.cpp:858-863)
  const double mr_tol = std::max(std::max(0.0, cfg->tol), std::max(0.0, mr_rel_tol) * rmax);
  auto met = [&]() {
    if (mr) return rmax < mr_tol;
    if (cfg->stop_rule == PF_STOP_REL2) return bnorm2 == 0.0 || std::sqrt(rr) <= cfg->tol * std::sqrt(bnorm2);
    return rmax < cfg->tol;
  };
  // FP32 residual level that triggers a (checking) replacement: the target itself
  // (none for the multires rows, whose FP32 residual is scaled by the cell volume)
  const double tol2_abs = mr ? 0.0
                             : (cfg->stop_rule == PF_STOP_REL2 ? cfg->tol * cfg->tol * bnorm2 : cfg->tol * cfg->tol);
  static const bool trace = std::getenv("PF_SOLVE_TRACE") != nullptr;
  // most FP32 iterations between two residual replacements
  constexpr int between = 200;
  int total = 0, outer = 0;
  bool converged = met();
  if (lpc_system) c->tiles_valid = true;
  const long long ncell = c->dc.nblocks * kBlockVol;
  // residual snapshot (training data), at most one per `snap_every` iterations
  auto snapshot = [&](int iter, const float* r32) -> int {
    if (c->snap_cap <= 0 || c->nsnap >= c->snap_cap) return PF_OK;
    if (c->snap_last_iter >= 0 && iter - c->snap_last_iter < c->snap_every) return PF_OK;
    HIP_TRY(c, hipMemcpyAsync(c->snaps + (long long)c->nsnap * ncell, r32, sizeof(float) * (size_t)ncell,
                              hipMemcpyDeviceToDevice, c->stream));
    c->nsnap++;
    c->snap_last_iter = iter;
    return PF_OK;
  };
  // flexible PCG around the multigrid V-cycle, plain or with the network's correction
  // weights (z and partial r.z in slot 2, GT partials)
  bool learned = want_learned || want_mg;
  c->mg_cs_active = c->mg_cs;  // caller-set weights (pf_mg_set_correction_weights) or none
  if (mr && !refmode && c->u32_host[5])
    return fail(c, PF_ERR_STATE, "multires leaves above level 2 hold FLUID cells: the fast solves take levels 0 to 2");
  if (learned) {
    st = mr ? mr_mg_build(c, mop) : mg_build(c);
    if (st) return st;
  }
  if (want_learned && !c->mg.empty()) {
    // the network runs once per solve; the cycle then costs what the plain one does
    long long ki = kbegin(c, PF_K_LPC_APPLY);
    st = lpc_cw_weights(c, false);
    kend(c, ki);
    if (st) return st;
    c->mg_cs_active = c->mg_cs_net;
  }
  const unsigned GT = mr ? cg_grid(npb) : (learned ? mg_grid0(c) : 1u);
  auto papply = [&](const int* done) -> int {
    long long ki = kbegin(c, PF_K_MG_APPLY);
    int s2 = mr ? mr_mg_apply(c, mop, va, c->r32, c->z32, done, c->partial)
                : mg_apply(c, c->r32, c->z32, done, c->partial);
    kend(c, ki);
    return s2;
  };
  int* done_dev = &c->sc->done;
  if (refmode) {
    // the reference's FP64 iteration with its options; x in x64
    HIP_TRY(c, hipMemcpyAsync(c->mr_pin_host, c->mr_pin_dev, sizeof(long long), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    c->mr_detail.reference_order = 1;
    int ri = 0;
    bool rc = false, rb = false;
    st = mr_reference_solve(c, *c->mr_cfg, G, va, mop64, (long long)c->u32_host[4], ri, rc, rb);
    if (st) return st;
    total = ri;
    converged = rc;
    if (rb) S.breakdown = 1;
    st = residual();
    if (st) return st;
    rr = c->red_host[0];
    rmax = c->red_host[1];
  }
  if (!refmode && !converged && max_iters > 0 && std::isfinite(rmax)) {
    // the buffer-addressed kernels take 32-bit byte offsets: arrays below 2 GiB
    const bool spmv_buffers = c->dc.nblocks * kBlockVol * 4 < (1LL << 31);
    CgState cg;
    // The Jacobi iteration as k_cg_iter or k_mr_cg_iter.  k_cg_iter moves 52 B a cell where the
    // separate kernels move 64, but between about 5 and 15 million cells those find part of
    // theirs in the last-level cache.  Separate against one kernel, us an iteration: 160^3 53.8
    // and 48.7, 176^3 67.5 and 69.3, 192^3 96 and 100, 208^3 122 and 130, 240^3 203 and 206, 256^3
    // 250 and 245, 288^3 350 and 342.
    const bool cached = npb > 80000 && npb < 240000;
    bool one_kernel = mr || (spmv_buffers && !cached);
    const unsigned GL = mr ? cg_grid(npb) : G;    // workgroups of the load, one partial each
    // r32 from the FP64 residual, x32 = 0 (and p = 0)
    auto load = [&](const double* src, float* p) {
      if (mr)
        hipLaunchKernelGGL(k_mr_load, dim3(GL), dim3(256), 0, c->stream, va, mop, src, c->x32, c->r32, p,
                           static_cast<float*>(nullptr), 0);
      else
        hipLaunchKernelGGL(k_pcg_load, dim3(GL), dim3(256), 0, c->stream, va, src, c->x32, c->r32, c->z32, p,
                           c->invd32, learned ? 1 : 0);
    };
    // (re)start: r32 from r64, x32 = 0, p = 0, z = M(r)
    auto start = [&](int budget) -> int {
      if (one_kernel && !learned && !c->cgq) {
        const hipError_t e = dalloc(c, &c->cgq, ncell);
        if (mr) HIP_TRY(c, e);
        one_kernel = e == hipSuccess;  // (the separate kernels need no second A p)
      }
      if (one_kernel && !learned) return cg_start(c, cg, va, G, r_src, delta * delta, tol2_abs, budget, between);
      load(r_src, c->pA);
      LAUNCH_CHECK(c);
      if (learned) {
        int s2 = papply(nullptr);
        if (s2) return s2;
        hipLaunchKernelGGL(k_pcg_start_flex, dim3(1), dim3(256), 0, c->stream, c->partial, (int)GL, (int)GT, c->sc,
                           delta * delta, tol2_abs, budget, between);
      } else {
        hipLaunchKernelGGL(k_pcg_start, dim3(1), dim3(256), 0, c->stream, c->partial, (int)G, c->sc, delta * delta,
                           tol2_abs, budget, between);
      }
      LAUNCH_CHECK(c);
      return PF_OK;
    };
    st = start(max_iters);
    if (st) return st;
    st = snapshot(0, c->r32);
    if (st) return st;
    // the two iteration kernels use at most 1024 workgroups, so the per-iteration
    // scalar kernels sum few partials
    const unsigned GS = mr ? cg_grid(npb) : std::min(G, 1024u);
    VecArgs vs = va;
    int iter_before = 0, iter_base = 0;
    double best_rr = rr, prev_rr = rr;
    int no_gain = 0, learned_slow = 0;
    // With a cycle preconditioner an iteration costs ~0.8 ms at 256^3, so iterations
    // queued past the replacement trigger are worth avoiding: the next look at the done
    // flag comes after the predicted number of iterations, from the FP32 residual's
    // observed decay per iteration toward max(tol2 rr_ref, tol2_abs) (1..check)
    const bool predict = want_mg || want_learned;
    int q_next = check;
    double rate = -1.0, rr_last = -1.0;
    int iter_last = 0;
    for (;;) {
      const size_t rec0 = c->krec.size();
      const bool fused = one_kernel && !learned;
      if (fused) {
        st = cg_run(c, cg, va, check, [&](int iter, const float* r) { return snapshot(iter_base + iter, r); });
        if (st) return st;
      }
      for (int q = 0; q < (fused ? 0 : q_next); ++q) {
        if (mr)
          TIMED(c, PF_K_PCG_SPMV,
                hipLaunchKernelGGL(k_mr_spmv, dim3(GS), dim3(256), 0, c->stream, vs, mop, c->z32, c->pA, c->pB, c->Ap));
        else if (spmv_buffers)
        TIMED(c, PF_K_PCG_SPMV,
              hipLaunchKernelGGL(k_pcg_spmv, dim3(GS), dim3(256), 0, c->stream, vs, c->z32, c->pA, c->pB, c->Ap,
                                 c->cd32, c->cx32, c->cy32, c->cz32));
        else
        TIMED(c, PF_K_PCG_SPMV,
              hipLaunchKernelGGL(k_pcg_spmv_gather, dim3(GS), dim3(256), 0, c->stream, vs, c->z32, c->pA, c->pB,
                                 c->Ap, c->cd32, c->cx32, c->cy32, c->cz32));
        hipLaunchKernelGGL(k_pcg_alpha, dim3(1), dim3(256), 0, c->stream, c->partial, (int)GS, c->sc);
        if (learned) {
          if (mr)
            TIMED(c, PF_K_PCG_UPDATE,
                  hipLaunchKernelGGL(k_mr_update, dim3(GS), dim3(256), 0, c->stream, vs, c->mr_info, c->x32, c->r32,
                                     c->z32, c->pA, c->pB, c->Ap));
          else
            TIMED(c, PF_K_PCG_UPDATE,
                  hipLaunchKernelGGL(k_pcg_update_flex, dim3(GS), dim3(256), 0, c->stream, vs, c->x32, c->r32, c->z32,
                                     c->pA, c->pB, c->Ap));
          st = papply(done_dev);
          if (st) return st;
          hipLaunchKernelGGL(k_pcg_beta_flex, dim3(1), dim3(256), 0, c->stream, c->partial, (int)GS, (int)GT, c->sc);
        } else {
          TIMED(c, PF_K_PCG_UPDATE,
                hipLaunchKernelGGL(k_pcg_update, dim3(GS), dim3(256), 0, c->stream, vs, c->x32, c->r32, c->z32, c->pA,
                                   c->pB, c->Ap, c->invd32));
          hipLaunchKernelGGL(k_pcg_beta, dim3(1), dim3(256), 0, c->stream, c->partial, (int)GS, c->sc);
        }
      }
      LAUNCH_CHECK(c);
      if (!fused) {
        HIP_TRY(c, hipMemcpyAsync(c->sc_host, c->sc, sizeof(SolveScalars), hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(c, hipStreamSynchronize(c->stream));
      }
      std::memcpy(c->done_host, &c->sc_host->iter, sizeof(int) * 8);
      // {iter, done, breakdown, stalled, iter_best, max_iter, stall_window, upd}
      // launches after a pause return at once: keep the timings of those that ran
      const int ran = c->done_host[0] - iter_before;
      iter_before = c->done_host[0];
      int kept_s = 0, kept_u = 0, kept_l = 0;
      for (size_t r = rec0; r < c->krec.size(); ++r) {
        int& k = c->krec[r].first;
        if (k == PF_K_PCG_SPMV && kept_s++ >= ran) k = -1;
        if (k == PF_K_PCG_UPDATE && kept_u++ >= ran) k = -1;
        if ((k == PF_K_LPC_APPLY || k == PF_K_MG_APPLY) && kept_l++ >= ran) k = -1;
      }
      if (ran > 0 && !fused) {
        st = snapshot(iter_base + c->done_host[0], c->r32);
        if (st) return st;
      }
      if (!c->done_host[1]) {
        q_next = check;
        if (predict) {
          const SolveScalars& H = *c->sc_host;
          const int it = c->done_host[0];
          if (rr_last > 0.0 && it > iter_last && H.rr > 0.0 && H.rr < rr_last)
            rate = std::pow(H.rr / rr_last, 1.0 / (it - iter_last));
          rr_last = H.rr;
          iter_last = it;
          const double target = std::max(H.tol2 * H.rr_ref, H.tol2_abs);
          if (rate > 0.0 && rate < 1.0 && H.rr > target)
            q_next = std::max(1, std::min(check, (int)std::ceil(std::log(target / H.rr) / std::log(rate) - 1e-9)));
        }
        continue;
      }
      // a new segment follows (residual replacement): it ends after about
      // log(tol2) / log(rate) iterations; its first look measures the decay afresh
      rr_last = -1.0;
      q_next = check;
      if (predict && rate > 0.0 && rate < 1.0 && c->sc_host->tol2 > 0.0 && c->sc_host->tol2 < 1.0)
        q_next = std::max(1, std::min(check, (int)std::ceil(std::log(c->sc_host->tol2) / std::log(rate) - 1e-9)));
      total = iter_base + c->done_host[0];
      const bool breakdown = c->done_host[2] != 0;
      // residual replacement: x64 += x32, r64 = b - A x64 in FP64
      hipLaunchKernelGGL(k_ir_accum, dim3(G), dim3(256), 0, c->stream, va, c->x64, c->x32);
      LAUNCH_CHECK(c);
      st = residual();
      if (st) return st;
      rr = c->red_host[0];
      rmax = c->red_host[1];
      ++outer;
      converged = met();
      if (trace) {
        double s_rr32 = 0.0;
        s_rr32 = c->sc_host->rr;
        std::fprintf(stderr, "[pf solve] update %d iter %d fp32 rel %.3e true rel %.3e max %.3e%s%s\n", outer, total,
                     std::sqrt(s_rr32 / std::max(bnorm2, 1e-300)), std::sqrt(rr / std::max(bnorm2, 1e-300)), rmax,
                     breakdown ? " breakdown" : "", learned ? " (learned)" : "");
      }
      if (rr < best_rr * 0.999) { best_rr = rr; no_gain = 0; } else { ++no_gain; }
      // (no gain over 40 replacements: the solve has stagnated)
      if (converged || total >= max_iters || outer >= max_updates || !std::isfinite(rr) || no_gain >= 40) {
        if (breakdown) S.breakdown = 1;
        break;
      }
      // the learned preconditioner falls back to Jacobi when two replacements in a
      // row gained less than 10% (or the recursion broke down)
      if (learned) {
        learned_slow = (rr > 0.9 * prev_rr || breakdown) ? learned_slow + 1 : 0;
        if (learned_slow >= 2 || breakdown) {
          learned = false;
          S.fallback_used = 1;
          iter_base = total;
          iter_before = 0;
          prev_rr = rr;
          st = start(max_iters - total);
          if (st) return st;
          continue;
        }
      }
      prev_rr = rr;
      // resume from the true residual; after a breakdown restart the direction too
      if (fused) {
        st = breakdown ? start(max_iters - total) : cg_resume(c, cg, va, G);
        if (st) return st;
        if (breakdown) {
          iter_base = total;
          iter_before = 0;
        }
        continue;
      }
      load(c->r64, breakdown ? c->pA : nullptr);
      LAUNCH_CHECK(c);
      if (learned) {
        st = papply(nullptr);
        if (st) return st;
      }
      if (breakdown) {
        if (learned)
          hipLaunchKernelGGL(k_pcg_start_flex, dim3(1), dim3(256), 0, c->stream, c->partial, (int)GL, (int)GT, c->sc,
                             delta * delta, tol2_abs, max_iters - total, between);
        else
          hipLaunchKernelGGL(k_pcg_start, dim3(1), dim3(256), 0, c->stream, c->partial, (int)G, c->sc, delta * delta,
                             tol2_abs, max_iters - total, between);
        iter_base = total;
        iter_before = 0;
      } else if (learned) {
        hipLaunchKernelGGL(k_pcg_resume_flex, dim3(1), dim3(256), 0, c->stream, c->partial, (int)GL, (int)GT, c->sc);
      } else {
        hipLaunchKernelGGL(k_pcg_resume, dim3(1), dim3(256), 0, c->stream, c->partial, (int)G, c->sc);
      }
      LAUNCH_CHECK(c);
    }
  }
  S.iterations = total;
  S.outer_iterations = outer;
  S.converged = converged ? 1 : 0;
  S.final_max_residual = rmax;
  S.true_max_residual = rmax;
  S.true_rel_residual = bnorm2 > 0 ? std::sqrt(rr / bnorm2) : 0.0;
  S.fluid_cells = c->u32_host[4];
  if (mr) S.pinned_cell = S.pinned ? 0 : -1;  // index in the reference's FLUID cell order
  record(c, timing, ev_solve);

  // 5. pressure store and face velocity update
  if (mr) {
    const long long ncell = c->dc.nblocks * kBlockVol;
    hipLaunchKernelGGL(k_mr_store_pressure, dim3(grid_for(ncell, 256)), dim3(256), 0, c->stream, mr_grid(c), c->x64,
                       c->f[F_P], c->mr_pfull, c->act[F_P]);
    const Dims* fd[3] = {&c->du, &c->dv, &c->dw};
    const PhaseK pk = phase_k(ph);
    for (int a = 0; a < 3; ++a)
      TIMED(c, PF_K_VELOCITY,
            hipLaunchKernelGGL(k_mr_velocity, dim3(grid_for(fd[a]->nblocks * kBlockVol, 256)), dim3(256), 0, c->stream,
                               mr_grid(c), a, c->mr_pfull, c->f[F_U + a], c->f[F_MU + a], pk, dt));
    LAUNCH_CHECK(c);
    record(c, timing, ev_vel);
    if (out) *out = S;
    return PF_OK;
  }
  hipLaunchKernelGGL(k_store_pressure, dim3(G), dim3(256), 0, c->stream, va, c->marker, c->x64, c->f[F_P],
                     c->act[F_P]);
  LAUNCH_CHECK(c);
  VelArgs vl;
  vl.g = g; vl.dc = c->dc; vl.df[0] = c->du; vl.df[1] = c->dv; vl.df[2] = c->dw;
  vl.marker = c->marker; vl.p = c->f[F_P];
  for (int ax = 0; ax < 3; ++ax) {
    vl.vel[ax] = c->f[F_U + ax];
    vl.mass[ax] = c->f[F_MU + ax];
    vl.act_vel[ax] = c->act[F_U + ax];
  }
  vl.ph = pa.ph;
  vl.s = dt / g.dx;
  vl.list = c->pblk;
  vl.nlist = npb;
  vl.unit_beta = single ? 1 : 0;
  TIMED(c, PF_K_VELOCITY,
        hipLaunchKernelGGL(k_velocity_update, dim3(grid_for(npb, 4)), dim3(256), 0, c->stream, vl));
  LAUNCH_CHECK(c);
  record(c, timing, ev_vel);
  if (out) *out = S;
  return PF_OK;
}

}  // namespace

extern "C" {

void pf_mg_defaults(pf_mg_cfg* cfg) {
  if (cfg) *cfg = mg_default_cfg();
}

int pf_set_multigrid(pf_ctx* c, const pf_mg_cfg* cfg) {
  if (!c || !cfg) return PF_ERR_ARG;
  if (!mg_cfg_valid(*cfg)) return fail(c, PF_ERR_ARG, "invalid multigrid cycle");
  c->mg_cfg = *cfg;
  return PF_OK;
}

int pf_mg_set_correction_weights(pf_ctx* c, const float* w, int64_t n) {
  if (!c) return PF_ERR_ARG;
  if (!w) {
    dfree(c->mg_cs);
    return PF_OK;
  }
  const int ax = (c->geom.nx + 1) / 2, ay = (c->geom.ny + 1) / 2, az = (c->geom.nz + 1) / 2;
  if (std::max({c->geom.nx, c->geom.ny, c->geom.nz}) <= 4)
    return fail(c, PF_ERR_ARG, "pf_mg_set_correction_weights: the grid has no coarse level");
  if (n != (int64_t)ax * ay * az)
    return fail(c, PF_ERR_ARG, "pf_mg_set_correction_weights: n must be the aggregate count ceil(nx/2)*ceil(ny/2)*ceil(nz/2)");
  const Dims d1 = make_dims(ax, ay, az);
  std::vector<float> s((size_t)(d1.nblocks * kBlockVol), 1.0f);
  for (int k = 0; k < az; ++k)
    for (int j = 0; j < ay; ++j)
      for (int i = 0; i < ax; ++i) {
        const float v = w[i + (int64_t)ax * (j + (int64_t)ay * k)];
        if (!(v > 0.f) || !std::isfinite(v))
          return fail(c, PF_ERR_ARG, "pf_mg_set_correction_weights: weights must be positive and finite");
        s[(size_t)bm_index(d1, i, j, k)] = std::sqrt(v);
      }
  if (!c->mg_cs) HIP_TRY(c, dalloc(c, &c->mg_cs, d1.nblocks * kBlockVol));
  HIP_TRY(c, hipMemcpyAsync(c->mg_cs, s.data(), sizeof(float) * s.size(), hipMemcpyHostToDevice, c->stream));
  HIP_TRY(c, hipStreamSynchronize(c->stream));
  return PF_OK;
}

int pf_get_multigrid(const pf_ctx* c, pf_mg_cfg* cfg) {
  if (!c || !cfg) return PF_ERR_ARG;
  *cfg = c->mg_cfg;
  return PF_OK;
}

int pf_project(pf_ctx* c, const pf_phase* ph, double dt, const pf_solve_cfg* cfg, double div_correction,
               pf_solve_stats* stats) {
  if (!c || !ph || !cfg) return PF_ERR_ARG;
  return run_project(c, ph, dt, cfg, div_correction, stats, false, 0, 0, 0);
}

int pf_project_single(pf_ctx* c, double dt, const pf_solve_cfg* cfg, pf_solve_stats* stats) {
  if (!c || !cfg) return PF_ERR_ARG;
  return run_project(c, nullptr, dt, cfg, 0.0, stats, false, 0, 0, 0, true);
}

}  // extern "C"
