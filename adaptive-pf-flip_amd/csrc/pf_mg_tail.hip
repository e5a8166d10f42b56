// pf_mg_tail.hip -- the multigrid cycle's small levels in one workgroup.
//
// A level of at most 64 blocks (16^3 cells) is 1024 cell rows or fewer: one row per
// thread of one workgroup.  From the first such level down, the whole cycle -- sweeps,
// restriction, the coarsest level's sweeps, prolongation, sweeps -- runs in one launch
// with the iterates in LDS, instead of four launches a level and one for the coarsest.
//
// What bounds it: a launch of k_mg_row on such a level takes 4.4 to 5 us whatever its
// size (start-up, then one chain of loads), 43 us in all for levels of 16^3, 8^3 and
// 4^3; here a sweep is one LDS round and a barrier, 14.3 us for the three.  The levels
// above keep k_mg_row: a 32^3 level would read its operator through one CU, no faster
// than four launches.  The arithmetic and its order are k_mg_row's and k_mg_coarsest's
// (but for what the compiler contracts).
#include "pf_internal.h"

namespace pf {

constexpr int kTailThreads = 1024;
constexpr int kTailLevels = 8;
constexpr int kTailBlocks = 80;  // blocks of all the tail's levels together (LDS)
constexpr int kTailSweeps = 16;  // pf_mg_cfg.sweeps' limit

struct MgTailLevel {
  Dims d;
  const _Float16 *cd, *cx, *cy, *cz, *inv;
  const float* unscale;
  int rows, off;                 // cell rows; first cell in the LDS arrays
};

struct MgTailArgs {
  const int* done;
  MgTailLevel lv[kTailLevels];   // from the finest; the last is the coarsest level
  int n;
  MgLevel last;                  // the coarsest level in FP32, one block
  const float* r;                // the finest level's residual
  float* x;                      // its correction
  float w[kTailSweeps];          // the sweeps' weights, down
  int nu, coarsest_sweeps;
  float omega, omega_c;
};

// a thread's row: its operator, and where its neighbours lie in the level's LDS array
// (a missing neighbour is the row itself)
struct MgTailRow {
  F4 cd, cx, cy, cz, iv, cym, czm;
  float cxm;
  int own, xp, xm, yp, ym, zp, zm, coarse;  // coarse: the row's first aggregate
};

__device__ inline MgTailRow mg_tail_row(const MgTailLevel& L, const Dims& dc, int t) {
  MgTailRow R;
  const int b = t >> 4, row = t & 15, ly = row & 3, lz = row >> 2;
  int bx, by, bz;
  block_coords(L.d, b, bx, by, bz);
  const int sy = L.d.nbx * kBlockVol, sz = sy * L.d.nby, o = t * 4;
  const bool fxp = bx + 1 < L.d.nbx, fxm = bx > 0, fyp = by + 1 < L.d.nby, fym = by > 0, fzp = bz + 1 < L.d.nbz,
             fzm = bz > 0;
  R.own = o;
  R.xp = fxp ? o + kBlockVol : o + 3;
  R.xm = fxm ? o - kBlockVol + 3 : o;
  R.yp = ly < 3 ? o + 4 : (fyp ? o + sy - 12 : o);
  R.ym = ly > 0 ? o - 4 : (fym ? o - sy + 12 : o);
  R.zp = lz < 3 ? o + 16 : (fzp ? o + sz - 48 : o);
  R.zm = lz > 0 ? o - 16 : (fzm ? o - sz + 48 : o);
  R.coarse = (int)bm_index(dc, 2 * bx, (4 * by + ly) >> 1, (4 * bz + lz) >> 1);
  const float ua = L.unscale[0], ui = L.unscale[1];
  const uint32_t bytes = (uint32_t)L.rows * 8;
  const auto bcd = buf_rsrc(L.cd, bytes), bcx = buf_rsrc(L.cx, bytes), bcy = buf_rsrc(L.cy, bytes),
             bcz = buf_rsrc(L.cz, bytes), bi = buf_rsrc(L.inv, bytes);
  const uint32_t of = (uint32_t)o * 4;
  R.cd = mg_ldh4(bcd, of, ua);
  R.cx = mg_ldh4(bcx, of, ua);
  R.cy = mg_ldh4(bcy, of, ua);
  R.cz = mg_ldh4(bcz, of, ua);
  R.iv = mg_ldh4(bi, of, ui);
  R.cxm = mg_ldh1(bcx, fxm ? (uint32_t)R.xm * 4 : kNoLoad, ua);
  R.cym = mg_ldh4(bcy, ly > 0 || fym ? (uint32_t)R.ym * 4 : kNoLoad, ua);
  R.czm = mg_ldh4(bcz, lz > 0 || fzm ? (uint32_t)R.zm * 4 : kNoLoad, ua);
  return R;
}

__device__ inline F4 mg_tail_ld(const float* p) {
  const float4 q = *reinterpret_cast<const float4*>(p);
  return F4{{q.x, q.y, q.z, q.w}};
}
__device__ inline void mg_tail_st(float* p, const F4& v) {
  *reinterpret_cast<float4*>(p) = make_float4(v.v[0], v.v[1], v.v[2], v.v[3]);
}

// r - A u of the row, u its own cells, X the level's iterate in LDS
__device__ inline F4 mg_tail_residual(const MgTailRow& R, const float* X, const F4& u, const F4& r) {
  const float uxp = X[R.xp], uxm = X[R.xm];
  const F4 yp = mg_tail_ld(X + R.yp), ym = mg_tail_ld(X + R.ym), zp = mg_tail_ld(X + R.zp), zm = mg_tail_ld(X + R.zm);
  F4 out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float uc = u.v[i];
    float ax = R.cd.v[i] * uc;
    ax = fmaf(R.cx.v[i], uc - (i < 3 ? u.v[i + 1] : uxp), ax);
    ax = fmaf(i > 0 ? R.cx.v[i - 1] : R.cxm, uc - (i > 0 ? u.v[i - 1] : uxm), ax);
    ax = fmaf(R.cy.v[i], uc - yp.v[i], ax);
    ax = fmaf(R.cym.v[i], uc - ym.v[i], ax);
    ax = fmaf(R.cz.v[i], uc - zp.v[i], ax);
    ax = fmaf(R.czm.v[i], uc - zm.v[i], ax);
    out.v[i] = r.v[i] - ax;
  }
  return out;
}

__global__ void __launch_bounds__(kTailThreads) k_mg_tail(MgTailArgs a) {
  __shared__ __align__(16) float xs[2][kTailBlocks * kBlockVol], rs[kTailBlocks * kBlockVol];
  if (a.done && *a.done) return;
  const int t = threadIdx.x, last = a.n - 1;
  unsigned parity = 0;  // bit l: which of xs holds level l's iterate
  auto residual_row = [&](int l) {
    return l == 0 ? mg_tail_ld(a.r + 4 * t) : mg_tail_ld(rs + a.lv[l].off + 4 * t);
  };
  // one sweep over level l from its current iterate into the other array
  auto sweep = [&](int l, const MgTailRow& R, const F4& r, F4& u, float w, bool act) {
    const unsigned p = (parity >> l) & 1;
    const float* X = xs[p] + a.lv[l].off;
    if (act) {
      const F4 res = mg_tail_residual(R, X, u, r);
#pragma unroll
      for (int i = 0; i < 4; ++i) u.v[i] = fmaf(w * R.iv.v[i], res.v[i], u.v[i]);
      mg_tail_st(xs[p ^ 1] + a.lv[l].off + R.own, u);
    }
    parity ^= 1u << l;
    __syncthreads();
  };
  for (int l = 0; l < last; ++l) {
    const MgTailLevel& L = a.lv[l];
    const MgTailLevel& C = a.lv[l + 1];
    const bool act = t < L.rows;
    MgTailRow R;
    F4 u, r;
    if (act) {
      R = mg_tail_row(L, C.d, t);
      r = residual_row(l);
#pragma unroll
      for (int i = 0; i < 4; ++i) u.v[i] = a.w[0] * R.iv.v[i] * r.v[i];
      mg_tail_st(xs[0] + L.off + R.own, u);
    }
    // (aggregates without children keep a zero residual)
    for (int q = t; q < C.rows * 4; q += kTailThreads) rs[C.off + q] = 0.f;
    __syncthreads();
    for (int s = 1; s < a.nu; ++s) sweep(l, R, r, u, a.w[s], act);
    if (act) {
      const F4 res = mg_tail_residual(R, xs[(parity >> l) & 1] + L.off, u, r);
      float s0 = (R.iv.v[0] != 0.0f ? res.v[0] : 0.0f) + (R.iv.v[1] != 0.0f ? res.v[1] : 0.0f);
      float s1 = (R.iv.v[2] != 0.0f ? res.v[2] : 0.0f) + (R.iv.v[3] != 0.0f ? res.v[3] : 0.0f);
      s0 += __shfl_xor(s0, 1);
      s1 += __shfl_xor(s1, 1);
      s0 += __shfl_xor(s0, 4);
      s1 += __shfl_xor(s1, 4);
      if ((t & 5) == 0) *reinterpret_cast<float2*>(rs + C.off + R.coarse) = make_float2(s0, s1);
    }
    __syncthreads();
  }
  // the coarsest level: one block, a cell to a lane of the first wave
  if (t < 64) {
    const MgLevel& L = a.last;
    const int i = t & 3, j = (t >> 2) & 3, k = t >> 4;
    const float rc = last == 0 ? a.r[t] : rs[a.lv[last].off + t], inv = L.inv[t], cd = L.cd[t];
    const int di[6] = {1, -1, 4, -4, 16, -16};
    const bool in[6] = {i + 1 < L.nx, i > 0, j + 1 < L.ny, j > 0, k + 1 < L.nz, k > 0};
    const float* cw[3] = {L.cx, L.cy, L.cz};
    float wv[6];
    int nb[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      nb[f] = in[f] ? t + di[f] : t;
      wv[f] = in[f] ? cw[f >> 1][(f & 1) ? nb[f] : t] : 0.0f;
    }
    float xc = a.omega * inv * rc;
    for (int s = 1; s < a.coarsest_sweeps; ++s) {
      float ax = cd * xc;
#pragma unroll
      for (int f = 0; f < 6; ++f) ax = fmaf(wv[f], xc - __shfl(xc, nb[f], 64), ax);
      xc = fmaf(a.omega * inv, rc - ax, xc);
    }
    if (last == 0)
      a.x[t] = xc;
    else
      xs[0][a.lv[last].off + t] = xc;
  }
  __syncthreads();
  for (int l = last - 1; l >= 0; --l) {
    const MgTailLevel& L = a.lv[l];
    const MgTailLevel& C = a.lv[l + 1];
    const bool act = t < L.rows;
    MgTailRow R;
    F4 u, r;
    const unsigned p = (parity >> l) & 1;
    if (act) {
      R = mg_tail_row(L, C.d, t);
      r = residual_row(l);
      u = mg_tail_ld(xs[p] + L.off + R.own);
      const float2 c = *reinterpret_cast<const float2*>(xs[(parity >> (l + 1)) & 1] + C.off + R.coarse);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (R.iv.v[i] != 0.0f) u.v[i] = fmaf(a.omega_c, i < 2 ? c.x : c.y, u.v[i]);
      mg_tail_st(xs[p ^ 1] + L.off + R.own, u);
    }
    parity ^= 1u << l;
    __syncthreads();
    for (int s = 0; s < a.nu; ++s) sweep(l, R, r, u, a.w[a.nu - 1 - s], act);
    if (l == 0 && act) mg_tail_st(a.x + R.own, u);
  }
}

}  // namespace pf
