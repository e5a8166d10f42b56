// pf_host_particles.hip -- binning, marking, the P2G splat launches, the face-field pass,
// G2P and advection, and the rho_tilde_0 calibration.
//
// One of the library's host files: pf_api.hip includes them in order into a single
// translation unit together with the kernel files, so every launch is a direct call.

namespace {

int grow_particles(pf_ctx* c, long long n, bool vol) {
  if (n <= c->pcap && (!vol || c->pa.vol)) return PF_OK;
  long long cap = std::max(n, c->pcap);
  PBuf* bufs[2] = {&c->pa, &c->pb};
  for (PBuf* b : bufs) {
    if (n > c->pcap) {
      hipFree(b->x); hipFree(b->y); hipFree(b->z); hipFree(b->u); hipFree(b->v); hipFree(b->w);
      hipFree(b->type); hipFree(b->id); hipFree(b->vol);
      *b = PBuf{};
      HIP_TRY(c, dalloc(c, &b->x, cap)); HIP_TRY(c, dalloc(c, &b->y, cap)); HIP_TRY(c, dalloc(c, &b->z, cap));
      HIP_TRY(c, dalloc(c, &b->u, cap)); HIP_TRY(c, dalloc(c, &b->v, cap)); HIP_TRY(c, dalloc(c, &b->w, cap));
      HIP_TRY(c, dalloc(c, &b->type, cap)); HIP_TRY(c, dalloc(c, &b->id, cap));
    }
    if (vol && !b->vol) HIP_TRY(c, dalloc(c, &b->vol, cap));
  }
  if (n > c->pcap) {
    hipFree(c->rank);
    HIP_TRY(c, dalloc(c, &c->rank, cap));
    c->pcap = cap;
  }
  return PF_OK;
}

// counting sort of particles by block-major cell index
int ensure_binned(pf_ctx* c) {
  if (c->binned) return PF_OK;
  c->mark_order_valid = false;
  const long long ncell = c->dc.nblocks * kBlockVol;
  HIP_TRY(c, fill_u32(c->stream, c->cell_count, 0u, ncell));
  // the cell index in exact FP32 where the origin is 0 and dx a power of two
  const Geom& g = c->geom;
  const float fscale =
      (g.ox == 0.0 && g.oy == 0.0 && g.oz == 0.0 && is_pow2(g.dx)) ? (float)(1.0 / g.dx) : 0.f;
  if (c->np > 0) {
    TIMED(c, PF_K_BIN_COUNT,
          hipLaunchKernelGGL(k_bin_count, dim3(grid_for(c->np, 256)), dim3(256), 0, c->stream, c->np, c->pa,
                             c->geom, c->dc, fscale, c->rank, c->cell_count));
    LAUNCH_CHECK(c);
  }
  HIP_TRY(c, scan_u32(*c, c->cell_count, c->cell_start, ncell));
  if (c->np > 0) {
    TIMED(c, PF_K_BIN_SCATTER,
          hipLaunchKernelGGL(k_bin_scatter, dim3(grid_for(c->np, 256)), dim3(256), 0, c->stream, c->np, c->pa,
                             c->pb, c->has_vol, c->geom, c->dc, fscale, c->rank, c->cell_start));
    LAUNCH_CHECK(c);
    std::swap(c->pa, c->pb);
    // cells of more than kRankMax particles (piles against walls) sorted by caller id,
    // so that P2G walks them in order without a quadratic selection
    const long long cap = c->np / (kRankMax + 1) + 1;
    if (cap > c->crowd_cap) {
      dfree(c->crowd_list);
      HIP_TRY(c, dalloc(c, &c->crowd_list, cap));
      c->crowd_cap = cap;
    }
    HIP_TRY(c, fill_u32(c->stream, c->u32_dev + 16, 0u, 1));
    hipLaunchKernelGGL(k_crowded_cells, dim3(grid_for(ncell, 256)), dim3(256), 0, c->stream, ncell, c->cell_start,
                       (uint32_t)kRankMax, (uint32_t)kSortedMax, c->crowd_list, c->u32_dev + 16, c->crowd_cap);
    hipLaunchKernelGGL(k_sort_crowded, dim3(512), dim3(256), 0, c->stream, c->crowd_list, c->u32_dev + 16,
                       c->cell_start, c->pa, c->has_vol);
    LAUNCH_CHECK(c);
  }
  c->binned = true;
  c->colors_valid = false;
  return PF_OK;
}

// the binned particles' source blocks per colour (large grids' P2G, pf_color_lists)
int ensure_color_lists(pf_ctx* c) {
  int st = ensure_binned(c);
  if (st || c->colors_valid) return st;
  HIP_TRY(c, fill_u32(c->stream, c->color_cnt, 0u, 8));
  hipLaunchKernelGGL(k_color_lists, dim3(grid_for(c->dc.nblocks, 256)), dim3(256), 0, c->stream, c->dc,
                     c->cell_start, c->color_cnt, c->color_list, c->color_cap);
  LAUNCH_CHECK(c);
  c->colors_valid = true;
  return PF_OK;
}

int run_mark(pf_ctx* c) {
  int st = ensure_binned(c);
  if (st) return st;
  hipLaunchKernelGGL(k_mark, dim3(grid_for(c->dc.nblocks, 4)), dim3(256), 0, c->stream, c->dc, c->geom,
                     c->cell_start, c->marker, c->act[F_MK]);
  LAUNCH_CHECK(c);
  c->mark_order_valid = true;
  return PF_OK;
}

int run_face_ops(pf_ctx* c, int ops, float dtg) {
  const Dims* d[3] = {&c->du, &c->dv, &c->dw};
  for (int ax = 0; ax < 3; ++ax) {
    dim3 grid(grid_for(d[ax]->nblocks, 4));
    float* vel = c->f[F_U + ax];
    const float* mass = c->f[F_MU + ax];
    float* sv = c->f[F_SU + ax];
    uint8_t* av = c->act[F_U + ax];
    uint8_t* as = c->act[F_SU + ax];
    long long ki = kbegin(c, PF_K_FACE_OPS);
    if (ax == 0)
      hipLaunchKernelGGL(k_face_ops<0>, grid, dim3(256), 0, c->stream, *d[ax], c->geom, vel, mass, sv, av, as, ops, dtg);
    else if (ax == 1)
      hipLaunchKernelGGL(k_face_ops<1>, grid, dim3(256), 0, c->stream, *d[ax], c->geom, vel, mass, sv, av, as, ops, dtg);
    else
      hipLaunchKernelGGL(k_face_ops<2>, grid, dim3(256), 0, c->stream, *d[ax], c->geom, vel, mass, sv, av, as, ops, dtg);
    kend(c, ki);
    LAUNCH_CHECK(c);
  }
  return PF_OK;
}

// single: the single-phase trilinear unit-mass splat (ph and Vp unused)
// mr: the cubic splat over the enumerated multires faces
int run_p2g_splat(pf_ctx* c, const pf_phase* ph, double Vp, bool single = false, bool mr = false) {
  int st = ensure_binned(c);
  if (st) return st;
  const Dims* d[3] = {&c->du, &c->dv, &c->dw};
  const long long nb = c->dc.nblocks;
  if (nb <= kP2GRegionMost && c->np > 0 && !c->p2g_regions && !c->p2g_no_regions) {
    // (without the memory for them: by colours)
    if (hipMalloc((void**)&c->p2g_regions, (sizeof(float2) * 3 * 256 + 1) * (size_t)nb) != hipSuccess) {
      (void)hipGetLastError();
      c->p2g_regions = nullptr;
      c->p2g_no_regions = true;
    }
  }
  const bool regions = c->p2g_regions && c->np > 0;
  for (int ax = 0; ax < 3 && !regions; ++ax) {
    HIP_TRY(c, fill_f32(c->stream, c->f[F_U + ax], 0.f, d[ax]->nblocks * kBlockVol));
    HIP_TRY(c, fill_f32(c->stream, c->f[F_MU + ax], 0.f, d[ax]->nblocks * kBlockVol));
    HIP_TRY(c, fill_u8(c->stream, c->act[F_U + ax], 0, d[ax]->nblocks));
    HIP_TRY(c, fill_u8(c->stream, c->act[F_MU + ax], 0, d[ax]->nblocks));
  }
  P2GArgs a;
  a.g = c->geom;
  a.dc = c->dc;
  for (int ax = 0; ax < 3; ++ax) {
    a.df[ax] = *d[ax];
    a.mom[ax] = c->f[F_U + ax];
    a.mass[ax] = c->f[F_MU + ax];
    a.act_vel[ax] = c->act[F_U + ax];
    a.act_mass[ax] = c->act[F_MU + ax];
  }
  a.start = c->cell_start;
  a.P = c->pa;
  a.has_vol = c->has_vol;
  a.pow2 = is_pow2(c->geom.dx);
  a.inv_dx = 1.0 / c->geom.dx;
  a.fast32 = a.pow2 && c->geom.ox == 0.0 && c->geom.oy == 0.0 && c->geom.oz == 0.0 &&
             std::max({c->geom.nx, c->geom.ny, c->geom.nz}) < (1 << 22);
  a.inv_dx_f = (float)a.inv_dx;
  for (int ax = 0; ax < 3; ++ax) a.valid[ax] = mr ? c->mr_valid[ax] : nullptr;
  a.mp_l = single ? 1.f : (float)(ph->rho_l * Vp);
  a.mp_g = single ? 1.f : (float)(ph->rho_g * Vp);
  if (c->np == 0) return PF_OK;
  a.regions = c->p2g_regions;
  if (regions) {
    // (how many blocks hold particles is on the device; 8 particles a cell is usual)
    const bool split = p2g_split((uint32_t)std::min<long long>(nb, c->np / 512 + 1));
    const P2GShared sh = p2g_shared_args(a);
    const P2GField f0 = p2g_field_args(a, 0), f1 = p2g_field_args(a, 1), f2 = p2g_field_args(a, 2);
    const dim3 grid((unsigned)nb, split ? 3 : 1);
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(64), 0, c->stream, sh, f0, f1, f2); };
    const long long ki = kbegin(c, PF_K_P2G);
    if (mr)
      a.fast32 ? launch(k_p2g_block<2, true>) : launch(k_p2g_block<2, false>);
    else if (single)
      a.fast32 ? launch(k_p2g_block<1, true>) : launch(k_p2g_block<1, false>);
    else
      a.fast32 ? launch(k_p2g_block<0, true>) : launch(k_p2g_block<0, false>);
    const long long nf = std::max({d[0]->nblocks, d[1]->nblocks, d[2]->nblocks});
    hipLaunchKernelGGL(k_p2g_gather, dim3(grid_for(nf, 4), 3), dim3(256), 0, c->stream, sh, f0, f1, f2);
    kend(c, ki);
    LAUNCH_CHECK(c);
    return PF_OK;
  }
  st = ensure_color_lists(c);
  if (st) return st;
  for (int col = 0; col < 8; ++col) {
    a.list = c->color_list + (long long)col * c->color_cap;
    a.count = c->color_cnt + col;
    // (the list's length is on the device: offer the split by axes where it may be short)
    const dim3 grid((unsigned)std::max<long long>(c->color_cap, 1), c->color_cap <= 2 * kP2GSplitMost ? 3 : 1);
    const P2GShared sh = p2g_shared_args(a);
    const P2GField f0 = p2g_field_args(a, 0), f1 = p2g_field_args(a, 1), f2 = p2g_field_args(a, 2);
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(64), 0, c->stream, sh, f0, f1, f2); };
    const long long ki = kbegin(c, PF_K_P2G);
    if (mr)
      a.fast32 ? launch(k_p2g_color<2, true>) : launch(k_p2g_color<2, false>);
    else if (single)
      a.fast32 ? launch(k_p2g_color<1, true>) : launch(k_p2g_color<1, false>);
    else
      a.fast32 ? launch(k_p2g_color<0, true>) : launch(k_p2g_color<0, false>);
    kend(c, ki);
    LAUNCH_CHECK(c);
  }
  return PF_OK;
}

// Whether an advection without G2P packs the grid's velocity into pairs first.  The packing
// costs three launches (6 us) and 5.7 ps a cell and saves 9 ps a particle in second order, 13 in
// third.  Plain gathers against pairs, in us (second order; third): 32^3 cells x 8 particles 34
// and 39 (37.6; 42), 48^3 x 8 52 and 53 (63; 59), 64^3 x 2 42 and 46 (49; 50), 64^3 x 8 83 and 76
// (105; 91), 96^3 x 1 53 and 61 (65; 66.5), 96^3 x 2 80 and 75 (101; 86), 128^3 x 1 86 and 86 (109;
// 96), 128^3 x 4 250 and 188 (355; 248).
bool advect_in_pairs(long long np, long long cells, int order) {
  return np >= std::max(cells, order == 3 ? 600000 + cells / 5 * 2 : 700000 + cells / 3 * 2);
}

// Room for the velocity pairs of an advection without G2P: the G2P's quads where it has
// allocated them, else arrays of their own (8 B a face).  False without the memory: the plain
// gathers then, the same bits.
bool g2p_pairs(pf_ctx* c, const Dims* const (&fd)[3], float2* (&pair)[3]) {
  if (c->g2p_quad[2]) {
    for (int ax = 0; ax < 3; ++ax) pair[ax] = reinterpret_cast<float2*>(c->g2p_quad[ax]);
    return true;
  }
  for (int ax = 0; ax < 3 && !c->g2p_no_pairs; ++ax) {
    if (!c->g2p_pair[ax]) c->g2p_no_pairs = dalloc(&c->g2p_pair[ax], fd[ax]->nblocks * kBlockVol) != hipSuccess;
    pair[ax] = c->g2p_pair[ax];
  }
  if (c->g2p_no_pairs)
    for (auto& q : c->g2p_pair) dfree(q);
  return !c->g2p_no_pairs;
}

int run_g2p_advect(pf_ctx* c, bool g2p, bool adv, double aL, double aG, double dt, int order) {
  if (c->np == 0) return PF_OK;
  G2PArgs a;
  a.g = c->geom;
  a.df[0] = c->du; a.df[1] = c->dv; a.df[2] = c->dw;
  a.P = c->pa;
  a.n = c->np;
  a.inv_dx = (float)(1.0 / c->geom.dx);
  a.ox = (float)c->geom.ox; a.oy = (float)c->geom.oy; a.oz = (float)c->geom.oz;
  const Geom& g = c->geom;
  a.lo[0] = (float)(g.ox + 0.5 * g.dx); a.hi[0] = (float)(g.ox + (g.nx - 0.5) * g.dx);
  a.lo[1] = (float)(g.oy + 0.5 * g.dx); a.hi[1] = (float)(g.oy + (g.ny - 0.5) * g.dx);
  a.lo[2] = (float)(g.oz + 0.5 * g.dx); a.hi[2] = (float)(g.oz + (g.nz - 0.5) * g.dx);
  a.aL = (float)aL; a.aG = (float)aG; a.dt = (float)dt;
  a.order = order;
  a.do_g2p = g2p; a.do_advect = adv;
  a.esc = c->esc_dev;
  a.vmax_bits = reinterpret_cast<uint32_t*>(c->vmax_dev);
  const Dims* fd[3] = {&c->du, &c->dv, &c->dw};
  float2* pair[3] = {nullptr, nullptr, nullptr};
  const bool pairs = !g2p && advect_in_pairs(c->np, (long long)g.nx * g.ny * g.nz, order) && g2p_pairs(c, fd, pair);
  if (g2p && !c->g2p_quad[2])
    for (auto& q : c->g2p_pair) dfree(q);  // (the quads hold pairs too)
  for (int ax = 0; ax < 3; ++ax) {
    if (g2p && !c->g2p_quad[ax]) HIP_TRY(c, dalloc(c, &c->g2p_quad[ax], fd[ax]->nblocks * kBlockVol));
    a.field[ax] = g2p ? static_cast<const void*>(c->g2p_quad[ax]) : (pairs ? static_cast<const void*>(pair[ax]) : c->f[F_U + ax]);
  }
  // the G2P reduces the max speed of the velocities it writes (the next CFL scan's value)
  if (g2p) HIP_TRY(c, fill_u32(c->stream, reinterpret_cast<uint32_t*>(c->vmax_dev), 0u, 1));
  {
    // (the kernel timer covers the packing and the kernel)
    const long long ki = kbegin(c, PF_K_G2P_ADVECT);
    const unsigned grid = xcd_grid(c->np, 256, 8192);
    for (int ax = 0; ax < 3; ++ax) {
      const dim3 gp(std::min<unsigned>(grid_for(fd[ax]->nblocks * kBlockVol, 256), 8192u));
      if (g2p)
        hipLaunchKernelGGL(k_pack_quad, gp, dim3(256), 0, c->stream, *fd[ax], c->f[F_U + ax], c->f[F_SU + ax],
                           c->g2p_quad[ax]);
      else if (pairs)
        hipLaunchKernelGGL(k_pack_pair, gp, dim3(256), 0, c->stream, *fd[ax], c->f[F_U + ax], pair[ax]);
    }
    if (g2p)
      hipLaunchKernelGGL(k_g2p_advect<float4>, dim3(grid), dim3(256), 0, c->stream, a);
    else if (pairs)
      hipLaunchKernelGGL(k_g2p_advect<float2>, dim3(grid), dim3(256), 0, c->stream, a);
    else
      hipLaunchKernelGGL(k_g2p_advect<float>, dim3(grid), dim3(256), 0, c->stream, a);
    kend(c, ki);
  }
  LAUNCH_CHECK(c);
  if (g2p) c->vmax_valid = true;
  if (adv) c->binned = false;
  return PF_OK;
}

// calibrateRhoTilde0, src/transfer/transfer3d_tp.cpp:29-36: raw u-face mass at
// (4,4,4) of an 8^3 lattice with 8 liquid particles per cell, over rho_l.
double calibrate_host(const pf_phase* pp, double Vp) {
  const int n = 8;
  std::vector<double> M((size_t)(n + 1) * n * n, 0.0);
  const double mp = pp->rho_l * Vp;
  auto kern = [](double d2) {
    double q = d2 / (1.5 * 1.5), t = 1.0 - q;
    return t > 0.0 ? t * t * t : 0.0;
  };
  for (int k = 0; k < n; ++k)
    for (int j = 0; j < n; ++j)
      for (int i = 0; i < n; ++i)
        for (int s = 0; s < 8; ++s) {
          double gx = i + 0.25 + 0.5 * (s & 1), gy = j + 0.25 + 0.5 * ((s >> 1) & 1) - 0.5,
                 gz = k + 0.25 + 0.5 * ((s >> 2) & 1) - 0.5;
          int i0 = (int)std::floor(gx), j0 = (int)std::floor(gy), k0 = (int)std::floor(gz);
          double wsum = 0.0;
          for (int dk = -2; dk <= 3; ++dk)
            for (int dj = -2; dj <= 3; ++dj)
              for (int di = -2; di <= 3; ++di) {
                int ii = i0 + di, jj = j0 + dj, kk = k0 + dk;
                if (ii < 0 || ii >= n + 1 || jj < 0 || jj >= n || kk < 0 || kk >= n) continue;
                double dx = gx - ii, dy = gy - jj, dz = gz - kk;
                wsum += kern(dx * dx + dy * dy + dz * dz);
              }
          if (wsum <= 0.0) continue;
          for (int dk = -2; dk <= 3; ++dk)
            for (int dj = -2; dj <= 3; ++dj)
              for (int di = -2; di <= 3; ++di) {
                int ii = i0 + di, jj = j0 + dj, kk = k0 + dk;
                if (ii < 0 || ii >= n + 1 || jj < 0 || jj >= n || kk < 0 || kk >= n) continue;
                double dx = gx - ii, dy = gy - jj, dz = gz - kk;
                double w = kern(dx * dx + dy * dy + dz * dz) / wsum;
                if (w <= 0.0) continue;
                M[ii + (size_t)(n + 1) * (jj + (size_t)n * kk)] += w * mp;
              }
        }
  double raw = M[4 + (size_t)(n + 1) * (4 + (size_t)n * 4)];
  return raw > 0 ? raw / pp->rho_l : 1.0;
}

}  // namespace
