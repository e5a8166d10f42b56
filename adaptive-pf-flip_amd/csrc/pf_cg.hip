// pf_cg.hip -- the Jacobi PCG iteration in one kernel.
//
// The reference's iteration (sparse_ops3d_tp.cpp:341-364) has two reductions that wait
// on each other: p.Ap before the update, r.z after it, and the direction needs the
// second.  Here a launch forms r, z, p and q = A p from the previous launch's, and the
// sums p.q, r.z, z.q, q.D^-1 q and r.r in the same pass.  The next launch's alpha is
// r.z / p.q as before, and the r.z after its update, which beta needs before r is formed,
// comes from those sums (r' = r - alpha q, but for the rounding of r' to FP32):
//   r'.z' = r.z - 2 alpha z.q + alpha^2 q.D^-1 q
// (in FP64; the next launch sums r'.z' itself, so nothing accumulates).  Recurring q
// instead (Chronopoulos and Gear 1989, s = A r + beta s) drifts: a closed box at a
// residual of 1e-9 then took 1.2 to 1.4 times the iterations, this form the same number.
// q needs p at the neighbours, so a cell on a block face recomputes its neighbours' r, z
// and p from the old r, q and p; r, q, p and the scalars alternate between two copies.
// FP32 vectors, FP64 products and scalars, as the separate kernels.
//
// What bounds it: below about 10^6 cells the chain of latencies in one launch (kernel
// start, the sums, the row's loads, the reduction), above it HBM (52 B/cell).  The
// separate form (SpMV, alpha, update, beta: four launches of 2 to 5 us) took, per
// iteration, 12.6 us at 48^3, 17.7 at 64^3, 33 at 128^3 and 225 to 260 at 256^3; this one
// 6.4, 6.9, 24 and 233.
#include "pf_internal.h"

namespace pf {

struct CgArgs {
  Dims dc;
  const uint32_t* list;
  long long nlist;
  float* x;
  const float *r, *q, *p;       // the last launch's, read
  float *rn, *qn, *pn;          // this one's
  const float *inv, *cd, *cx, *cy, *cz;
  const double* sums;           // the partial sums of r, q, p, nsums <= 1024 in each of CG_SUMS
                                // slots (after a load: r.z and r.r only)
  double* sums_out;
  int nsums;
  const SolveScalars* in;
  SolveScalars* out;
  unsigned long long* word;     // pinned host memory: 2 seq + done
  unsigned long long seq;
};
enum { CG_PQ = 0, CG_RZ, CG_ZQ, CG_QDQ, CG_RR, CG_SUMS };

// A lane's x-row of 4 cells in its block (16 lanes to a block, as k_pcg_spmv) and the
// face rows of the neighbouring blocks it touches: both x ends, and at most one y and
// one z row (a row lies on one y face at most, and on one z face).
struct CgRow {
  uint32_t o, xp, xm, y, z;    // byte offsets, kNoLoad where there is nothing to read
  int ly, lz;
};

__device__ inline CgRow cg_row(const Dims& dc, uint32_t sy, uint32_t sz, uint32_t b, bool valid, int row) {
  CgRow R;
  R.ly = row & 3;
  R.lz = row >> 2;
  int bx, by, bz;
  block_coords(dc, b, bx, by, bz);
  const uint32_t o = valid ? (b * kBlockVol + 4 * row) * 4 : kNoLoad;
  R.o = o;
  R.xp = valid && bx + 1 < dc.nbx ? o + kBlockVol * 4 : kNoLoad;
  R.xm = valid && bx > 0 ? o - kBlockVol * 4 + 12 : kNoLoad;
  R.y = R.z = kNoLoad;
  if (valid && R.ly == 3 && by + 1 < dc.nby) R.y = o + sy - 48;
  if (valid && R.ly == 0 && by > 0) R.y = o - sy + 48;
  if (valid && R.lz == 3 && bz + 1 < dc.nbz) R.z = o + sz - 192;
  if (valid && R.lz == 0 && bz > 0) R.z = o - sz + 192;
  return R;
}

struct CgCoef {
  F4 cd, cx, cy, cz, cyf, czf;  // cyf, czf: the lower y and z face rows' couplings
  float cxm;
};

__device__ inline void cg_coef(__amdgpu_buffer_rsrc_t cd, __amdgpu_buffer_rsrc_t cx, __amdgpu_buffer_rsrc_t cy,
                               __amdgpu_buffer_rsrc_t cz, const CgRow& R, CgCoef& C) {
  C.cd = buf_ld4(cd, R.o);
  C.cx = buf_ld4(cx, R.o);
  C.cy = buf_ld4(cy, R.o);
  C.cz = buf_ld4(cz, R.o);
  C.cxm = buf_ld(cx, R.xm);
  C.cyf = buf_ld4(cy, R.ly == 0 ? R.y : kNoLoad);
  C.czf = buf_ld4(cz, R.lz == 0 ? R.z : kNoLoad);
}

// A u on the row (u: own cells, xp/xm: the cells past its ends, uy/uz: the face rows);
// a missing neighbour stands in as the cell itself, whose term vanishes
__device__ inline F4 cg_stencil(const F4& u, float xp, float xm, const F4& uy, const F4& uz, const CgRow& R,
                                const CgCoef& C, int lane) {
  F4 out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float syp = __shfl(u.v[i], lane + 1, 64), sym = __shfl(u.v[i], lane - 1, 64);
    const float szp = __shfl(u.v[i], lane + 4, 64), szm = __shfl(u.v[i], lane - 4, 64);
    const float scy = __shfl(C.cy.v[i], lane - 1, 64), scz = __shfl(C.cz.v[i], lane - 4, 64);
    const bool hy = R.y != kNoLoad, hz = R.z != kNoLoad;
    const float own = u.v[i];
    const float uxp = i < 3 ? u.v[i + 1] : (R.xp != kNoLoad ? xp : own);
    const float uxm = i > 0 ? u.v[i - 1] : (R.xm != kNoLoad ? xm : own);
    const float cxm = i > 0 ? C.cx.v[i - 1] : C.cxm;
    const float uyp = R.ly < 3 ? syp : (hy ? uy.v[i] : own);
    const float uym = R.ly > 0 ? sym : (hy ? uy.v[i] : own);
    const float cym = R.ly > 0 ? scy : C.cyf.v[i];
    const float uzp = R.lz < 3 ? szp : (hz ? uz.v[i] : own);
    const float uzm = R.lz > 0 ? szm : (hz ? uz.v[i] : own);
    const float czm = R.lz > 0 ? scz : C.czf.v[i];
    float a = C.cd.v[i] * own;
    a = fmaf(C.cx.v[i], own - uxp, a);
    a = fmaf(cxm, own - uxm, a);
    a = fmaf(C.cy.v[i], own - uyp, a);
    a = fmaf(cym, own - uym, a);
    a = fmaf(C.cz.v[i], own - uzp, a);
    a = fmaf(czm, own - uzm, a);
    out.v[i] = a;
  }
  return out;
}

// r = (float)r64, x = 0 (and p = q = 0 before the first iteration), partial r.z and r.r
__global__ void __launch_bounds__(256) k_cg_load(VecArgs a, const double* __restrict__ r64, float* __restrict__ x,
                                                 float* __restrict__ r, float* __restrict__ p, float* __restrict__ q,
                                                 const float* __restrict__ inv) {
  const int lane = threadIdx.x & 63;
  double v[CG_SUMS] = {};
  FOR_LIST_BLOCKS(a, b, lane) {
    const long long c = b * kBlockVol + lane;
    const float rc = (float)r64[c];
    x[c] = 0.f;
    r[c] = rc;
    if (p) p[c] = q[c] = 0.f;
    v[CG_RZ] += (double)rc * (double)(inv[c] * rc);
    v[CG_RR] += (double)rc * (double)rc;
  }
  const bool mx[CG_SUMS] = {};
  block_reduce_store<CG_SUMS>(v, mx, a.part, kMaxPartials);
}

// The state before the first launch of a solve (fresh 1), or after a residual
// replacement (fresh 2): the paused direction was formed from the replaced residual, so
// the recursion steps back to the direction before it, in the other buffers.
__global__ void k_cg_begin(SolveScalars* sc, int fresh, double delta2, double tol2_abs, int max_iter, int between) {
  sc->fresh = fresh;
  sc->done = 0;
  sc->upd = 0;
  if (fresh == 1) {
    sc->rz = 0.0; sc->alpha = 0.0; sc->beta = 0.0; sc->pAp = 0.0;
    sc->tol2 = delta2; sc->tol2_abs = tol2_abs;
    sc->iter = 0; sc->iter_best = 0; sc->max_iter = max_iter; sc->stall_window = between;
    sc->breakdown = 0; sc->stalled = 0; sc->par = 0;
  } else {
    sc->par ^= 1;
  }
}

// The end of the iteration before (as finish_iteration) and this one's alpha and beta
// from the previous launch's sums v; every thread of every workgroup forms the same
// values.  Returns false when the recursion pauses (done is set in S).  S.rz stays the
// r.z of the direction in the other buffers, which a resumed recursion continues.
__device__ inline bool cg_scalars(SolveScalars& S, const double (&v)[CG_SUMS]) {
  const double rz = v[CG_RZ], rr = v[CG_RR];
  S.rr = rr;
  if (S.fresh) {
    S.rr_ref = rr;
    if (S.fresh == 1) S.rr0 = S.rr_best = rr;
    S.iter_best = S.iter;
    S.fresh = 0;
    S.alpha = 0.0;
    S.beta = S.rz != 0.0 ? rz / S.rz : 0.0;
    if (rr == 0.0 || S.iter >= S.max_iter) S.done = 1;
    return !S.done;
  }
  const double pq = v[CG_PQ];
  if (!isfinite(rr) || !isfinite(rz) || !isfinite(pq)) {
    S.breakdown = 1;
    S.done = 1;
    return false;
  }
  // residual replacement when the FP32 residual fell by delta below the largest since the
  // last one, reached the target, ran `stall_window` iterations, or the budget is spent
  // (after one iteration at least: the restart's residual itself stops nothing)
  if (rr > S.rr_ref) S.rr_ref = rr;
  if (S.iter > S.iter_best && (rr <= S.tol2 * S.rr_ref || rr <= S.tol2_abs || S.iter >= S.max_iter ||
                               S.iter - S.iter_best >= S.stall_window)) {
    S.upd = 1;
    S.done = 1;
    return false;
  }
  S.pAp = pq;
  if (!(pq > 0.0)) {
    S.breakdown = 1;
    S.done = 1;
    return false;
  }
  const double alpha = rz / pq;
  const double next = rz - 2.0 * alpha * v[CG_ZQ] + alpha * alpha * v[CG_QDQ];
  S.alpha = alpha;
  S.beta = rz != 0.0 ? next / rz : 0.0;
  S.rz = rz;
  S.iter += 1;
  return true;
}

// the fields that the recursion uses, one by one (a copy of the whole struct goes
// through a private array, which the compiler places in LDS by the workgroup's shape:
// every wave then reads the dispatch packet in host memory first, 10 us a launch)
__device__ inline SolveScalars cg_state(const SolveScalars* s) {
  SolveScalars S;
  S.rz = s->rz; S.alpha = s->alpha; S.beta = s->beta; S.pAp = s->pAp;
  S.rr = s->rr; S.rr0 = s->rr0; S.rr_best = s->rr_best; S.rr_ref = s->rr_ref;
  S.tol2 = s->tol2; S.tol2_abs = s->tol2_abs;
  S.iter = s->iter; S.done = s->done; S.breakdown = s->breakdown; S.iter_best = s->iter_best;
  S.max_iter = s->max_iter; S.stall_window = s->stall_window; S.upd = s->upd; S.fresh = s->fresh; S.par = s->par;
  return S;
}
__device__ inline void cg_publish(const CgArgs& a, const SolveScalars& S) {
  SolveScalars* o = a.out;
  o->rz = S.rz; o->alpha = S.alpha; o->beta = S.beta; o->pAp = S.pAp;
  o->rr = S.rr; o->rr0 = S.rr0; o->rr_best = S.rr_best; o->rr_ref = S.rr_ref;
  o->tol2 = S.tol2; o->tol2_abs = S.tol2_abs;
  o->iter = S.iter; o->done = S.done; o->breakdown = S.breakdown; o->iter_best = S.iter_best;
  o->max_iter = S.max_iter; o->stall_window = S.stall_window; o->upd = S.upd; o->fresh = S.fresh; o->par = S.par;
  __hip_atomic_store(a.word, 2 * a.seq + (S.done ? 1u : 0u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The last launch's partial sums: every one that a thread adds is loaded before any is
// waited for (a load of what other XCDs just wrote takes 1 to 2 us).
__device__ inline void cg_fetch(const CgArgs& a, double (&w)[4][CG_SUMS]) {
  const auto bs = buf_rsrc(a.sums, CG_SUMS * kMaxPartials * 8);
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int k = 0; k < CG_SUMS; ++k) {
      const uint32_t t = threadIdx.x + 256 * j;
      w[j][k] = buf_ld_f64(bs, t < (uint32_t)a.nsums ? (k * kMaxPartials + t) * 8 : kNoLoad);
    }
}

// The sums and the recursion's next scalars in S, published by the first workgroup; false
// when this launch has nothing to do.
__device__ inline bool cg_advance(const CgArgs& a, const double (&w)[4][CG_SUMS], SolveScalars& S,
                                  double (&sh)[4][CG_SUMS]) {
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  if (S.done) {
    if (lead) cg_publish(a, S);
    return false;
  }
  double v[CG_SUMS];
#pragma unroll
  for (int k = 0; k < CG_SUMS; ++k) v[k] = wave_sum((w[0][k] + w[1][k]) + (w[2][k] + w[3][k]));
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < CG_SUMS; ++k) sh[threadIdx.x >> 6][k] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < CG_SUMS; ++k) v[k] = (sh[0][k] + sh[1][k]) + (sh[2][k] + sh[3][k]);
  const bool go = cg_scalars(S, v);
  if (go) S.par ^= 1;
  if (lead) cg_publish(a, S);
  return go;
}

// this launch's partial sums
__device__ inline void cg_store_sums(const CgArgs& a, double (&v)[CG_SUMS], double (&sh)[4][CG_SUMS]) {
#pragma unroll
  for (int k = 0; k < CG_SUMS; ++k) v[k] = wave_sum(v[k]);
  __syncthreads();  // (every wave has read the sums in sh)
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < CG_SUMS; ++k) sh[threadIdx.x >> 6][k] = v[k];
  __syncthreads();
  if (threadIdx.x < CG_SUMS)
    a.sums_out[threadIdx.x * kMaxPartials + blockIdx.x] =
        (sh[0][threadIdx.x] + sh[1][threadIdx.x]) + (sh[2][threadIdx.x] + sh[3][threadIdx.x]);
}

// one row's inputs
struct CgLoads {
  CgRow R;
  CgCoef C;
  F4 r, q, p, inv, x, ry, qy, py, iy, rz, qz, pz, iz;
  float rxp, qxp, pxp, ixp, rxm, qxm, pxm, ixm;
};

// The list goes in slots of four blocks (one per 16 lanes of a wave), each XCD a contiguous
// eighth.
// PRE: a wave's one row loads are issued before the sums are waited for, which hides their
// latency for 170 registers, two workgroups to a CU, instead of 91.  No better once the
// workgroups are not all resident, so up to 512 of them.  Without and with, per iteration of
// whole solves: 64^3 (256 workgroups) 7.6 and 7.4 us, 72^3 (368) 9.3 and 9.5, 80^3 (504) 9.7
// and 9.7, 84^3 (584) 11.1 and 11.8, 96^3 (864) 13.3 and 15.2.
template <bool PRE>
__global__ void __launch_bounds__(256) k_cg_iter(CgArgs a) {
  __shared__ double sh[4][CG_SUMS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double w[4][CG_SUMS];
  cg_fetch(a, w);
  const uint32_t bytes = (uint32_t)(a.dc.nblocks * kBlockVol * 4);
  const uint32_t sy = (uint32_t)a.dc.nbx * kBlockVol * 4, sz = sy * (uint32_t)a.dc.nby;
  const auto br = buf_rsrc(a.r, bytes), bq = buf_rsrc(a.q, bytes), bp = buf_rsrc(a.p, bytes);
  const auto cr = buf_rsrc(a.rn, bytes), cq = buf_rsrc(a.qn, bytes), cp = buf_rsrc(a.pn, bytes);
  const auto bx = buf_rsrc(a.x, bytes), bi = buf_rsrc(a.inv, bytes);
  const auto bcd = buf_rsrc(a.cd, bytes), bcx = buf_rsrc(a.cx, bytes), bcy = buf_rsrc(a.cy, bytes),
             bcz = buf_rsrc(a.cz, bytes);
  const uint32_t seg = (uint32_t)((a.nlist + 7) / 8), s0 = (blockIdx.x & 7) * seg,
                 e = min((uint32_t)a.nlist, s0 + seg), step = (gridDim.x >> 3) * 16;
  uint32_t t0 = s0 + ((blockIdx.x >> 3) * 4 + wave) * 4;
  CgLoads L;
  auto load = [&]() {
    const uint32_t t = t0 + (lane >> 4);
    L.R = cg_row(a.dc, sy, sz, a.list[min(t, e - 1)], t < e, lane & 15);
    const CgRow& R = L.R;
    L.r = buf_ld4(br, R.o); L.q = buf_ld4(bq, R.o); L.p = buf_ld4(bp, R.o);
    L.inv = buf_ld4(bi, R.o); L.x = buf_ld4(bx, R.o);
    L.ry = buf_ld4(br, R.y); L.qy = buf_ld4(bq, R.y); L.py = buf_ld4(bp, R.y); L.iy = buf_ld4(bi, R.y);
    L.rz = buf_ld4(br, R.z); L.qz = buf_ld4(bq, R.z); L.pz = buf_ld4(bp, R.z); L.iz = buf_ld4(bi, R.z);
    L.rxp = buf_ld(br, R.xp); L.qxp = buf_ld(bq, R.xp); L.pxp = buf_ld(bp, R.xp); L.ixp = buf_ld(bi, R.xp);
    L.rxm = buf_ld(br, R.xm); L.qxm = buf_ld(bq, R.xm); L.pxm = buf_ld(bp, R.xm); L.ixm = buf_ld(bi, R.xm);
    cg_coef(bcd, bcx, bcy, bcz, R, L.C);
  };
  if (PRE && t0 < e) load();
  SolveScalars S = cg_state(a.in);
  if (!cg_advance(a, w, S, sh)) return;
  const float alpha = (float)S.alpha, beta = (float)S.beta;
  // the new p of any cell from the old r, q, p (the same arithmetic for a block's own
  // cells and for its neighbours')
  auto direction = [&](float r, float q, float p, float inv) {
    return fmaf(beta, p, inv * fmaf(-alpha, q, r));
  };
  double v[CG_SUMS] = {};
  while (t0 < e) {
    if (!PRE) load();
    F4 pn, rn, xn, py, pz;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      xn.v[i] = fmaf(alpha, L.p.v[i], L.x.v[i]);
      rn.v[i] = fmaf(-alpha, L.q.v[i], L.r.v[i]);
      pn.v[i] = fmaf(beta, L.p.v[i], L.inv.v[i] * rn.v[i]);
      py.v[i] = direction(L.ry.v[i], L.qy.v[i], L.py.v[i], L.iy.v[i]);
      pz.v[i] = direction(L.rz.v[i], L.qz.v[i], L.pz.v[i], L.iz.v[i]);
    }
    const F4 qn = cg_stencil(pn, direction(L.rxp, L.qxp, L.pxp, L.ixp), direction(L.rxm, L.qxm, L.pxm, L.ixm), py, pz,
                             L.R, L.C, lane);
    buf_st4(bx, L.R.o, xn.v);
    buf_st4(cr, L.R.o, rn.v);
    buf_st4(cp, L.R.o, pn.v);
    buf_st4(cq, L.R.o, qn.v);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double rd = rn.v[i], zd = L.inv.v[i] * rn.v[i], qd = qn.v[i];
      v[CG_PQ] += (double)pn.v[i] * qd;
      v[CG_RZ] += rd * zd;
      v[CG_ZQ] += zd * qd;
      v[CG_QDQ] += qd * (double)L.inv.v[i] * qd;
      v[CG_RR] += rd * rd;
    }
    if (PRE) break;  // (up to 512 workgroups a wave has one slot)
    t0 += step;
  }
  cg_store_sums(a, v, sh);
}

}  // namespace pf
