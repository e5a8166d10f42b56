// pf_mr_row.hip -- the multires operator S by cell rows: the fast solves' kernels.
//
// A 4^3 block lies inside one leaf, so its cells all have level L = 0, 1 or 2.  The
// solve's vectors hold a leaf cell's value at every fine cell of it (level 0 and 1), or
// at the block's first entry (level 2: one leaf cell fills the block).  The couplings lie
// at the fine cells as in the uniform operator (cx, cy, cz of the + faces), zero inside a
// leaf cell.  Then S x is the uniform 7-point stencil on the fine grid, summed over each
// leaf cell's fine cells: no level or anchor look-ups, and every level shares a kernel.
// A lane holds one x-row of 4 fine cells (16 lanes to a block, as k_pcg_spmv); a byte per
// block holds its level and which of its six neighbours have level 2.  The Dirichlet
// part cd is at the anchors only and joins the sum.
//
// What bounds it: the rows' loads from L2 and HBM.  The form it replaces went through
// each leaf cell's patches one by one (level byte, face index and anchor of every patch)
// and split the levels over two launches.  On 1.75 million leaf cells of three levels (256^3
// effective, 131,000 blocks) an SpMV took 194 + 30 us and takes 49, a sweep of the cycle
// 150 + 20 and takes 37, an FP64 residual 348 and takes 109.
#include "pf_internal.h"

namespace pf {

constexpr int kMrLevelMask = 3;  // info bits 0-1: level; bits 2-7: +x, -x, +y, -y, +z, -z neighbour has level 2

struct MrRowOp {
  Dims dc;
  const uint8_t* info;
  const float *cd, *cx, *cy, *cz, *inv;
  const float4* cs;  // per block of level 2: the sums of cd, cx, cy and cz (0 in other blocks)
};
struct MrRowOp64 {
  Dims dc;
  const uint8_t* info;
  const double *cd, *cx, *cy, *cz, *vol;
};

template <typename T>
struct Row4 {
  T v[4];
};
__device__ inline Row4<float> mr_ld4(const float* p) {
  const float4 q = *reinterpret_cast<const float4*>(p);
  return {{q.x, q.y, q.z, q.w}};
}
__device__ inline Row4<double> mr_ld4(const double* p) {
  const double2 a = reinterpret_cast<const double2*>(p)[0], b = reinterpret_cast<const double2*>(p)[1];
  return {{a.x, a.y, b.x, b.y}};
}
__device__ inline void mr_st4(float* p, const Row4<float>& v) {
  *reinterpret_cast<float4*>(p) = make_float4(v.v[0], v.v[1], v.v[2], v.v[3]);
}
__device__ inline void mr_st4(double* p, const Row4<double>& v) {
  reinterpret_cast<double2*>(p)[0] = make_double2(v.v[0], v.v[1]);
  reinterpret_cast<double2*>(p)[1] = make_double2(v.v[2], v.v[3]);
}

// A lane's row: cell indices of its values (own, the cells past its x ends, its one y
// and one z face row) and of its couplings.  A missing neighbour is the row itself, with
// a zero coupling; a level-2 neighbour is that block's first entry.
struct MrRow {
  uint32_t own, oc;              // values; couplings (the row itself on every level)
  uint32_t xp, xm, y, z;         // values
  uint32_t cxm, cy, cz;          // the lower neighbours' couplings
  bool hxm, hy, hz;              // ... that exist
  bool sy, sz;                   // the face row's values are one value
  bool pure;                     // a level-2 block among level-2 blocks: one coupling a face
  bool valid;
  int L, ly, lz, row;
  int bx, by, bz;
  float w;                       // share of a leaf cell in one entry of a row
};

__device__ inline MrRow mr_row(const Dims& dc, unsigned f, uint32_t b, bool valid, int row) {
  MrRow R;
  R.valid = valid;
  R.row = row;
  R.ly = row & 3;
  R.lz = row >> 2;
  R.L = (int)(f & kMrLevelMask);
  R.w = !valid ? 0.f : (R.L == 0 ? 1.f : (R.L == 1 ? 0.125f : 0.015625f));
  block_coords(dc, b, R.bx, R.by, R.bz);
  const uint32_t base = b * kBlockVol, sy = (uint32_t)dc.nbx * kBlockVol, sz = sy * (uint32_t)dc.nby;
  R.oc = base + 4 * row;
  R.own = R.L == 2 ? base : R.oc;
  R.xp = R.own;
  R.xm = R.own;
  R.y = R.own;
  R.z = R.own;
  R.cxm = R.cy = R.cz = R.oc;
  if (R.bx + 1 < dc.nbx) R.xp = base + kBlockVol + (f & 4 ? 0 : 4 * row);
  R.hxm = R.bx > 0;
  if (R.hxm) {
    R.cxm = base - kBlockVol + 4 * row + 3;
    R.xm = f & 8 ? base - kBlockVol : R.cxm;
  }
  R.sy = R.sz = R.L == 2;
  R.hy = R.hz = false;
  if (R.ly == 3 && R.by + 1 < dc.nby) {
    R.sy = f & 16;
    R.y = base + sy + (R.sy ? 0 : 16 * R.lz);
  }
  if (R.ly == 0 && R.by > 0) {
    R.hy = true;
    R.sy = f & 32;
    R.cy = base - sy + 16 * R.lz + 12;
    R.y = R.sy ? base - sy : R.cy;
  }
  if (R.lz == 3 && R.bz + 1 < dc.nbz) {
    R.sz = f & 64;
    R.z = base + sz + (R.sz ? 0 : 4 * R.ly);
  }
  if (R.lz == 0 && R.bz > 0) {
    R.hz = true;
    R.sz = f & 128;
    R.cz = base - sz + 48 + 4 * R.ly;
    R.z = R.sz ? base - sz : R.cz;
  }
  R.pure = R.L == 2 && (f & 4 || R.bx + 1 >= dc.nbx) && (f & 8 || R.bx == 0) && (f & 16 || R.by + 1 >= dc.nby) &&
           (f & 32 || R.by == 0) && (f & 64 || R.bz + 1 >= dc.nbz) && (f & 128 || R.bz == 0);
  return R;
}

template <typename T>
__device__ inline Row4<T> mr_splat(Row4<T> r, bool one) {
  if (one) r.v[1] = r.v[2] = r.v[3] = r.v[0];
  return r;
}
template <typename T>
__device__ inline Row4<T> mr_own(const T* __restrict__ a, const MrRow& R) {
  return mr_splat(mr_ld4(a + R.own), R.L == 2);
}
template <typename T>
__device__ inline Row4<T> mr_yrow(const T* __restrict__ a, const MrRow& R) {
  return mr_splat(mr_ld4(a + R.y), R.sy);
}
template <typename T>
__device__ inline Row4<T> mr_zrow(const T* __restrict__ a, const MrRow& R) {
  return mr_splat(mr_ld4(a + R.z), R.sz);
}
// a row's values back to its leaf cells' entries.  The two entries of a level-1 cell in a row
// take the first one's value: the compiler may contract the arithmetic of a row's
// entries differently, and values of one cell that differ by an ulp drift apart over a
// solve (multigrid: 7e-7 of 4 in x64, a flux of 1.6e-5 left in the cells whose residual, formed
// from all the entries, was 1e-12).  The cell's four lanes run the same instructions.
template <typename T>
__device__ inline void mr_put(T* __restrict__ a, const MrRow& R, Row4<T> v) {
  if (!R.valid) return;
  if (R.L == 1) {
    v.v[1] = v.v[0];
    v.v[3] = v.v[2];
  }
  if (R.L < 2)
    mr_st4(a + R.own, v);
  else if (R.row == 0)
    a[R.own] = v.v[0];
}

// the sum of a row's entries over each leaf cell, at every entry of it
template <typename T>
__device__ inline Row4<T> mr_leaf_sum(Row4<T> a, int L) {
  if (!__any(L != 0)) return a;  // (a wave of fine blocks)
  T lo = a.v[0] + a.v[1], hi = a.v[2] + a.v[3], all = lo + hi;
  lo += __shfl_xor(lo, 1, 64);
  hi += __shfl_xor(hi, 1, 64);
  lo += __shfl_xor(lo, 4, 64);
  hi += __shfl_xor(hi, 4, 64);
  all += __shfl_xor(all, 1, 64);
  all += __shfl_xor(all, 2, 64);
  all += __shfl_xor(all, 4, 64);
  all += __shfl_xor(all, 8, 64);
  if (L == 1) return {{lo, lo, hi, hi}};
  if (L == 2) return {{all, all, all, all}};
  return a;
}

// S u at the row's leaf cells: u its own values, uxp and uxm the cells past its ends, uy
// and uz its face rows.  Every lane of the wave calls it.  With SUMS a pure block's rows read
// the sums of its 16 couplings a face (summed in FP64 by the assembly) instead of 1.2 KB of
// couplings: its first row takes the cell's own term and the lower faces, its last row
// the upper y and z faces.  On 256^3 effective (131,000
// blocks of three levels) an SpMV 53 -> 49 us, the cycle's four passes 159 -> 146.  Not in the Jacobi
// iteration, whose small grids wait for latencies: 7.3 -> 7.6 us with them.
template <typename T, bool SUMS, typename Op>
__device__ inline Row4<T> mr_apply(const MrRow& R, const Op& op, const Row4<T>& u, T uxp, T uxm, const Row4<T>& uy,
                                   const Row4<T>& uz) {
  const int lane = threadIdx.x & 63;
  const bool pure = SUMS && R.pure;
  Row4<T> d = {}, c0 = {}, c1 = {}, c2 = {}, y0 = {}, z0 = {};
  T xlo = (T)0;
  if (!pure) {
    d = mr_ld4(op.cd + R.oc);
    c0 = mr_ld4(op.cx + R.oc);
    c1 = mr_ld4(op.cy + R.oc);
    c2 = mr_ld4(op.cz + R.oc);
    y0 = mr_ld4(op.cy + R.cy);
    z0 = mr_ld4(op.cz + R.cz);
    if (R.hxm) xlo = op.cx[R.cxm];
  }
  Row4<T> a = {};
  if constexpr (SUMS) {
    if (pure && (R.row == 0 || R.row == 15)) {
      const float4 q = op.cs[R.own >> 6];
      if (R.row == 0) {
        const float xl = R.hxm ? op.cs[R.xm >> 6].y : 0.f, yl = R.hy ? op.cs[R.y >> 6].z : 0.f,
                    zl = R.hz ? op.cs[R.z >> 6].w : 0.f;
        const float own = u.v[0];
        float s = q.x * own;
        s = fmaf(q.y, own - uxp, s);
        s = fmaf(xl, own - uxm, s);
        s = fmaf(yl, own - uy.v[0], s);
        a.v[0] = fmaf(zl, own - uz.v[0], s);
      } else {
        a.v[0] = fmaf(q.z, u.v[0] - uy.v[0], q.w * (u.v[0] - uz.v[0]));
      }
    }
    if (!__any(!pure)) return mr_leaf_sum(a, R.L);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const T own = u.v[i];
    const T yp = __shfl(own, lane + 1, 64), ym = __shfl(own, lane - 1, 64);
    const T zp = __shfl(own, lane + 4, 64), zm = __shfl(own, lane - 4, 64);
    const T cyl = __shfl(c1.v[i], lane - 1, 64), czl = __shfl(c2.v[i], lane - 4, 64);
    T s = d.v[i] * own;
    s = fma(c0.v[i], own - (i < 3 ? u.v[i + 1] : uxp), s);
    s = fma(i > 0 ? c0.v[i - 1] : xlo, own - (i > 0 ? u.v[i - 1] : uxm), s);
    s = fma(c1.v[i], own - (R.ly < 3 ? yp : uy.v[i]), s);
    s = fma(R.ly > 0 ? cyl : (R.hy ? y0.v[i] : (T)0), own - (R.ly > 0 ? ym : uy.v[i]), s);
    s = fma(c2.v[i], own - (R.lz < 3 ? zp : uz.v[i]), s);
    s = fma(R.lz > 0 ? czl : (R.hz ? z0.v[i] : (T)0), own - (R.lz > 0 ? zm : uz.v[i]), s);
    if (!pure) a.v[i] = s;
  }
  return mr_leaf_sum(a, R.L);
}

// The list in slots of four blocks (one per 16 lanes), each XCD a contiguous eighth.  The
// next slot's info bytes and the one after's list entries load while a slot is worked
// on (list, info and values would be three waits in a row): an update 36.5 ->
// 32.6 us on those blocks.  The Jacobi iteration makes its walk before it waits for the sums,
// so the first slot's list and info load meanwhile: 7.34 -> 7.23 us on 80 x 72 x 80, where
// every wave has one slot.
struct MrWalk {
  const uint32_t* list;
  const uint8_t* info;
  uint32_t t, e, step, b, nb;
  unsigned f, nf;
  __device__ MrWalk(const uint32_t* list_, long long nlist, const uint8_t* info_) : list(list_), info(info_) {
    const uint32_t seg = (uint32_t)((nlist + 7) / 8), s0 = (blockIdx.x & 7) * seg;
    e = min((uint32_t)nlist, s0 + seg);
    t = s0 + ((blockIdx.x >> 3) * 4 + (threadIdx.x >> 6)) * 4;
    step = (gridDim.x >> 3) * 16;
    b = nb = 0;
    f = nf = 0;
    if (t < e) {
      b = at(t);
      nb = at(t + step);
      f = info[b];
    }
  }
  __device__ uint32_t at(uint32_t s) const { return list[min(s + ((threadIdx.x & 63) >> 4), e - 1)]; }
  __device__ bool more() const { return t < e; }
  __device__ bool valid() const { return t + ((threadIdx.x & 63) >> 4) < e; }
  // (call with the slot's b and f taken: prefetches the next)
  __device__ uint32_t ahead() {
    nf = info[nb];
    return at(t + 2 * step);
  }
  __device__ void next(uint32_t nnb) {
    t += step;
    b = nb;
    f = nf;
    nb = nnb;
  }
};
#define FOR_MR_WALK(W, op, R)                                                                    \
  for (uint32_t _nn; (W).more() && ((_nn = (W).ahead()), true); (W).next(_nn))                    \
    if (const MrRow R = mr_row((op).dc, (W).f, (W).b, (W).valid(), threadIdx.x & 15); true)
#define FOR_MR_ROWS(A, op, R)                         \
  MrWalk _walk((A).list, (A).nlist, (op).info);       \
  FOR_MR_WALK(_walk, op, R)

// Levels and neighbours' levels of every block (the whole slab), as info bytes.
__global__ void __launch_bounds__(256) k_mr_info(MrGrid m, uint8_t* __restrict__ info) {
  const long long b = (long long)blockIdx.x * 256 + threadIdx.x;
  if (b >= m.dc.nblocks) return;
  int bx, by, bz;
  block_coords(m.dc, b, bx, by, bz);
  auto level = [&](int x, int y, int z) { return mr_level(m, 4 * x, 4 * y, 4 * z); };
  const int L = level(bx, by, bz);
  unsigned f = L < 0 ? 0u : (unsigned)min(L, 3);
  if (level(bx + 1, by, bz) == 2) f |= 4;
  if (level(bx - 1, by, bz) == 2) f |= 8;
  if (level(bx, by + 1, bz) == 2) f |= 16;
  if (level(bx, by - 1, bz) == 2) f |= 32;
  if (level(bx, by, bz + 1) == 2) f |= 64;
  if (level(bx, by, bz - 1) == 2) f |= 128;
  info[b] = (uint8_t)f;
}

// ---- the PCG around the cycle

// p_new = z + beta p_old, Ap = S p_new, partial p.Ap (k_pcg_spmv's twin)
__global__ void __launch_bounds__(256) k_mr_spmv(VecArgs a, MrRowOp op, const float* __restrict__ z,
                                                 float* __restrict__ pA, float* __restrict__ pB,
                                                 float* __restrict__ Ap) {
  if (a.sc->done) return;
  const bool odd = a.sc->iter & 1;
  const float* __restrict__ pold = odd ? pB : pA;
  float* __restrict__ pnew = odd ? pA : pB;
  const float beta = (float)a.sc->beta;
  double pap = 0.0;
  FOR_MR_ROWS(a, op, R) {
    Row4<float> p = mr_own(pold, R), py = mr_yrow(pold, R), pz = mr_zrow(pold, R);
    const Row4<float> zo = mr_own(z, R), zy = mr_yrow(z, R), zz = mr_zrow(z, R);
    const float xp = fmaf(beta, pold[R.xp], z[R.xp]), xm = fmaf(beta, pold[R.xm], z[R.xm]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p.v[i] = fmaf(beta, p.v[i], zo.v[i]);
      py.v[i] = fmaf(beta, py.v[i], zy.v[i]);
      pz.v[i] = fmaf(beta, pz.v[i], zz.v[i]);
    }
    const Row4<float> ap = mr_apply<float, true>(R, op, p, xp, xm, py, pz);
    mr_put(pnew, R, p);
    mr_put(Ap, R, ap);
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) s += (double)p.v[i] * (double)ap.v[i];
    pap += (double)R.w * s;
  }
  double v[1] = {pap};
  const bool mx[1] = {false};
  block_reduce_store<1>(v, mx, a.part, kMaxPartials);
}

// x += alpha p, r -= alpha Ap; partial r_new . z_old (slot 0) and r.r (slot 1)
__global__ void __launch_bounds__(256) k_mr_update(VecArgs a, const uint8_t* __restrict__ info, float* __restrict__ x,
                                                   float* __restrict__ r, const float* __restrict__ z,
                                                   const float* __restrict__ pA, const float* __restrict__ pB,
                                                   const float* __restrict__ Ap) {
  if (a.sc->done) return;
  const float* __restrict__ p = (a.sc->iter & 1) ? pA : pB;
  const float alpha = (float)a.sc->alpha;
  struct { Dims dc; const uint8_t* info; } const op{a.dc, info};
  double v[2] = {0.0, 0.0};
  FOR_MR_ROWS(a, op, R) {
    Row4<float> xo = mr_own(x, R), ro = mr_own(r, R);
    const Row4<float> po = mr_own(p, R), ao = mr_own(Ap, R), zo = mr_own(z, R);
    double s0 = 0.0, s1 = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      xo.v[i] = fmaf(alpha, po.v[i], xo.v[i]);
      ro.v[i] = fmaf(-alpha, ao.v[i], ro.v[i]);
      s0 += (double)ro.v[i] * (double)zo.v[i];
      s1 += (double)ro.v[i] * (double)ro.v[i];
    }
    mr_put(x, R, xo);
    mr_put(r, R, ro);
    v[0] += (double)R.w * s0;
    v[1] += (double)R.w * s1;
  }
  const bool mx[2] = {false, false};
  block_reduce_store<2>(v, mx, a.part, kMaxPartials);
}

// r = (float)r64, x = 0 and, where given, p = 0 and q = 0; partial r.z with z = D^-1 r
// (slot CG_RZ) and r.r (slot CG_RR) as k_cg_load, or in slots 0 and 1
__global__ void __launch_bounds__(256) k_mr_load(VecArgs a, MrRowOp op, const double* __restrict__ r64,
                                                 float* __restrict__ x, float* __restrict__ r, float* __restrict__ p,
                                                 float* __restrict__ q, int cg) {
  double rz = 0.0, rr = 0.0;
  FOR_MR_ROWS(a, op, R) {
    const Row4<double> rd = mr_own(r64, R);
    const Row4<float> inv = mr_own(op.inv, R);
    Row4<float> rf, zero = {{0.f, 0.f, 0.f, 0.f}};
    double s0 = 0.0, s1 = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      rf.v[i] = (float)rd.v[i];
      s0 += (double)rf.v[i] * (double)(inv.v[i] * rf.v[i]);
      s1 += (double)rf.v[i] * (double)rf.v[i];
    }
    mr_put(r, R, rf);
    mr_put(x, R, zero);
    if (p) mr_put(p, R, zero);
    if (q) mr_put(q, R, zero);
    rz += (double)R.w * s0;
    rr += (double)R.w * s1;
  }
  if (cg) {
    double v[CG_SUMS] = {};
    v[CG_RZ] = rz;
    v[CG_RR] = rr;
    const bool mx[CG_SUMS] = {};
    block_reduce_store<CG_SUMS>(v, mx, a.part, kMaxPartials);
  } else {
    double v[2] = {rz, rr};
    const bool mx[2] = {false, false};
    block_reduce_store<2>(v, mx, a.part, kMaxPartials);
  }
}

// the Jacobi iteration in one kernel (k_cg_iter's twin): 7.2 us on 80 x 72 x 80 with two
// levels, where the six separate kernels took 35
__global__ void __launch_bounds__(256) k_mr_cg_iter(CgArgs a, MrRowOp op) {
  __shared__ double sh[4][CG_SUMS];
  double w[4][CG_SUMS];
  cg_fetch(a, w);
  MrWalk walk(a.list, a.nlist, op.info);
  SolveScalars S = cg_state(a.in);
  if (!cg_advance(a, w, S, sh)) return;
  const float alpha = (float)S.alpha, beta = (float)S.beta;
  auto direction = [&](float r, float q, float p, float inv) {
    return fmaf(beta, p, inv * fmaf(-alpha, q, r));
  };
  double v[CG_SUMS] = {};
  FOR_MR_WALK(walk, op, R) {
    const Row4<float> r = mr_own(a.r, R), q = mr_own(a.q, R), p = mr_own(a.p, R), inv = mr_own(op.inv, R);
    const Row4<float> ry = mr_yrow(a.r, R), qy = mr_yrow(a.q, R), iy = mr_yrow(op.inv, R);
    const Row4<float> rz = mr_zrow(a.r, R), qz = mr_zrow(a.q, R), iz = mr_zrow(op.inv, R);
    Row4<float> py = mr_yrow(a.p, R), pz = mr_zrow(a.p, R), x = mr_own(static_cast<const float*>(a.x), R), pn, rn;
    const float xp = direction(a.r[R.xp], a.q[R.xp], a.p[R.xp], op.inv[R.xp]);
    const float xm = direction(a.r[R.xm], a.q[R.xm], a.p[R.xm], op.inv[R.xm]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x.v[i] = fmaf(alpha, p.v[i], x.v[i]);
      rn.v[i] = fmaf(-alpha, q.v[i], r.v[i]);
      pn.v[i] = fmaf(beta, p.v[i], inv.v[i] * rn.v[i]);
      py.v[i] = direction(ry.v[i], qy.v[i], py.v[i], iy.v[i]);
      pz.v[i] = direction(rz.v[i], qz.v[i], pz.v[i], iz.v[i]);
    }
    const Row4<float> qn = mr_apply<float, false>(R, op, pn, xp, xm, py, pz);
    mr_put(a.x, R, x);
    mr_put(a.rn, R, rn);
    mr_put(a.pn, R, pn);
    mr_put(a.qn, R, qn);
    double s[CG_SUMS] = {};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double rd = rn.v[i], zd = inv.v[i] * rn.v[i], qd = qn.v[i];
      s[CG_PQ] += (double)pn.v[i] * qd;
      s[CG_RZ] += rd * zd;
      s[CG_ZQ] += zd * qd;
      s[CG_QDQ] += qd * (double)inv.v[i] * qd;
      s[CG_RR] += rd * rd;
    }
#pragma unroll
    for (int k = 0; k < CG_SUMS; ++k) v[k] += (double)R.w * s[k];
  }
  cg_store_sums(a, v, sh);
}

// FP64 residual r = V rhs - S x at every entry of the leaf cells; partial r^2 and
// max |r / V| over the leaf cells (V is non-zero at FLUID anchors only)
__global__ void __launch_bounds__(256) k_mr_residual(VecArgs a, MrRowOp64 op, const double* __restrict__ b64,
                                                     const double* __restrict__ x, double* __restrict__ r) {
  double rr = 0.0, rm = 0.0;
  FOR_MR_ROWS(a, op, R) {
    const Row4<double> u = mr_own(x, R), uy = mr_yrow(x, R), uz = mr_zrow(x, R);
    const Row4<double> sx = mr_apply<double, false>(R, op, u, x[R.xp], x[R.xm], uy, uz);
    const Row4<double> vol = mr_ld4(op.vol + R.oc);
    Row4<double> res = mr_leaf_sum(mr_ld4(b64 + R.oc), R.L);
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      res.v[i] -= sx.v[i];
      s += res.v[i] * res.v[i];
      if (R.valid && vol.v[i] != 0.0) rm = fmax(rm, fabs(res.v[i] / vol.v[i]));
    }
    mr_put(r, R, res);
    rr += (double)R.w * s;
  }
  double v[2] = {rr, rm};
  const bool mx[2] = {false, true};
  block_reduce_store<2>(v, mx, a.part, kMaxPartials);
}

// ---- the cycle on S (first coarse level: the block grid)

struct MrCycleArgs {
  const uint32_t* list;
  long long nlist;
  const int* done;
  MrRowOp op;
  Dims dcc;              // the block grid's slab
  const float *r, *x;
  float* out;            // the new iterate, or the block grid's residual
  const float* xc;       // the block grid's correction (PSWEEP)
  float omega, omega_c, omega_u;
  double* part;
};

// the modes are k_mg_row's: FIRST2 two sweeps from zero, SWEEP one, PSWEEP one after
// adding the block's correction, RESTRICT the block sums of the residual; SWEEP and
// PSWEEP add the partial r . out when part is set
template <int MODE>
__global__ void __launch_bounds__(256) k_mr_cycle(MrCycleArgs a) {
  if (a.done && *a.done) return;
  const MrRowOp& op = a.op;
  double rz = 0.0;
  FOR_MR_ROWS(a, op, R) {
    const Row4<float> r = mr_own(a.r, R), inv = mr_own(op.inv, R);
    Row4<float> u, uy, uz;
    float uxp, uxm;
    if (MODE == MG_FIRST2) {
      const Row4<float> ry = mr_yrow(a.r, R), iy = mr_yrow(op.inv, R), rz_ = mr_zrow(a.r, R), iz = mr_zrow(op.inv, R);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        u.v[i] = a.omega_u * inv.v[i] * r.v[i];
        uy.v[i] = a.omega_u * iy.v[i] * ry.v[i];
        uz.v[i] = a.omega_u * iz.v[i] * rz_.v[i];
      }
      uxp = a.omega_u * op.inv[R.xp] * a.r[R.xp];
      uxm = a.omega_u * op.inv[R.xm] * a.r[R.xm];
    } else {
      u = mr_own(a.x, R);
      uy = mr_yrow(a.x, R);
      uz = mr_zrow(a.x, R);
      uxp = a.x[R.xp];
      uxm = a.x[R.xm];
    }
    if (MODE == MG_PSWEEP) {
      // (loads without a branch, in flight with the rest: a missing neighbour takes the
      // block's own correction, times a zero coupling)
      auto corr = [&](int bx, int by, int bz) { return a.omega_c * a.xc[bm_index(a.dcc, bx, by, bz)]; };
      const int ny = R.ly == 3 ? min(R.by + 1, op.dc.nby - 1) : (R.ly == 0 ? max(R.by - 1, 0) : R.by);
      const int nz = R.lz == 3 ? min(R.bz + 1, op.dc.nbz - 1) : (R.lz == 0 ? max(R.bz - 1, 0) : R.bz);
      const float c = corr(R.bx, R.by, R.bz), cy = corr(R.bx, ny, R.bz), cz = corr(R.bx, R.by, nz);
      uxp += corr(min(R.bx + 1, op.dc.nbx - 1), R.by, R.bz);
      uxm += corr(max(R.bx - 1, 0), R.by, R.bz);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (inv.v[i] != 0.f) u.v[i] += c;
        uy.v[i] += cy;
        uz.v[i] += cz;
      }
    }
    const Row4<float> ax = mr_apply<float, true>(R, op, u, uxp, uxm, uy, uz);
    if (MODE == MG_RESTRICT) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) s += r.v[i] - ax.v[i];
      s *= R.w;
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) s += __shfl_xor(s, o, 64);
      if (R.valid && R.row == 0) a.out[bm_index(a.dcc, R.bx, R.by, R.bz)] = s;
    } else {
      Row4<float> o;
      double s = 0.0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        o.v[i] = fmaf(a.omega * inv.v[i], r.v[i] - ax.v[i], u.v[i]);
        s += (double)r.v[i] * (double)o.v[i];
      }
      mr_put(a.out, R, o);
      rz += (double)R.w * s;
    }
  }
  if ((MODE == MG_SWEEP || MODE == MG_PSWEEP) && a.part) {
    double v[1] = {rz};
    const bool mx[1] = {false};
    block_reduce_store<1>(v, mx, a.part, kMaxPartials);
  }
}

// x = omega D^-1 r (one sweep from zero, a cycle of one sweep)
__global__ void __launch_bounds__(256) k_mr_cycle_first(MrCycleArgs a) {
  if (a.done && *a.done) return;
  FOR_MR_ROWS(a, a.op, R) {
    const Row4<float> r = mr_own(a.r, R), inv = mr_own(a.op.inv, R);
    Row4<float> o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o.v[i] = a.omega * inv.v[i] * r.v[i];
    mr_put(a.out, R, o);
  }
}

// R S P on the block grid: one wave per fine block (all blocks), lane = fine cell; the
// face weights are the couplings of the 16 fine cells on the block's + faces
__global__ void __launch_bounds__(256) k_mr_mg_coarse(MrRowOp op, Dims dcc, float* __restrict__ cd,
                                                      float* __restrict__ cx, float* __restrict__ cy,
                                                      float* __restrict__ cz) {
  const long long b = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (b >= op.dc.nblocks) return;  // whole waves
  int bx, by, bz;
  block_coords(op.dc, b, bx, by, bz);
  const long long c = b * kBlockVol + lane;
  float d = op.cd[c];
  float wx = (lane & 3) == 3 ? op.cx[c] : 0.f;
  float wy = ((lane >> 2) & 3) == 3 ? op.cy[c] : 0.f;
  float wz = (lane >> 4) == 3 ? op.cz[c] : 0.f;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    d += __shfl_xor(d, o, 64);
    wx += __shfl_xor(wx, o, 64);
    wy += __shfl_xor(wy, o, 64);
    wz += __shfl_xor(wz, o, 64);
  }
  if (lane == 0) {
    const long long q = bm_index(dcc, bx, by, bz);
    cd[q] = d;
    cx[q] = wx;
    cy[q] = wy;
    cz[q] = wz;
  }
}

// ---- the rows by fine cells (the reference-order solve keeps k_mr_assemble)

struct MrCellOut {
  double *b64, *cd64, *cx64, *cy64, *cz64, *vol64;
  float *cd32, *cx32, *cy32, *cz32, *inv32;
  float4* cs;
};

// sum over the lanes (fine cells of a block) of each leaf cell, L wave-uniform
__device__ inline double mr_lane_sum(double v, int L) {
  for (int bit = 0; bit < min(L, 2); ++bit) {
    v += __shfl_xor(v, 1 << bit, 64);
    v += __shfl_xor(v, 4 << bit, 64);
    v += __shfl_xor(v, 16 << bit, 64);
  }
  return v;
}

// k_mr_assemble's rows, one lane per fine cell: each lane takes the (at most six) patches
// on its own cell's faces and the leaf cell's lanes add up, instead of one lane going
// through a level-2 cell's 96 patches (256^3 effective: 5.8 ms before, 0.57 now).
__global__ void __launch_bounds__(256) k_mr_assemble_cells(MrAsm a, MrCellOut o) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  double bb = 0.0;
  const double dx = a.m.g.dx, area = dx * dx;
  const bool pins = a.pin[0] == 0;
  const uint32_t pin_key = pins ? a.pin[1] : 0xffffffffu;
  FOR_LIST_BLOCKS(a, b, lane) {
    const long long c = b * kBlockVol + lane;
    int bx, by, bz;
    block_coords(a.m.dc, b, bx, by, bz);
    const int i = bx * 4 + (lane & 3), j = by * 4 + ((lane >> 2) & 3), k = bz * 4 + (lane >> 4);
    const int L = mr_level(a.m, bx * 4, by * 4, bz * 4);  // (wave-uniform)
    const int s = 1 << (L < 0 ? 0 : L), mask = s - 1;
    if (L > 2 && lane == 0) a.pin[5] = 1;  // (the host refuses the solve)
    const bool fluid = L >= 0 && i < a.m.g.nx && j < a.m.g.ny && k < a.m.g.nz && a.m.marker[c] == CELL_FLUID;
    const double h = dx * (double)s, V = h * h * h;
    const bool pinned = fluid && pins && mr_order_key(a.m, i & ~mask, j & ~mask, k & ~mask, L) == pin_key;
    double cd = 0.0, diag = 0.0, div = 0.0, cp[3] = {0.0, 0.0, 0.0};
    if (fluid) {
      const int at[3] = {i, j, k};
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        const int axis = q >> 1, up = q & 1;
        // a patch where the face bounds the leaf cell
        if (up ? (at[axis] & mask) != mask : (at[axis] & mask) != 0) continue;
        const int d = up ? 1 : -1;
        const int ni = i + (axis == 0 ? d : 0), nj = j + (axis == 1 ? d : 0), nk = k + (axis == 2 ? d : 0);
        const int mn = mr_marker(a.m, ni, nj, nk);
        if (mn == CELL_SOLID) continue;
        const int Ln = mr_level(a.m, ni, nj, nk), sn = 1 << Ln;
        const double dist = 0.5 * h + 0.5 * (dx * (double)sn);
        const long long fi = bm_index(mr_fdims(a.m, axis), i + (axis == 0 ? up : 0), j + (axis == 1 ? up : 0),
                                      k + (axis == 2 ? up : 0));
        const double cond =
            dist > 0.0 ? a.dt * beta_of_raw((double)mr_face_mass(a, axis, fi), a.ph) * area / dist : 0.0;
        diag += cond;
        const bool coupled = mn == CELL_FLUID && !pinned &&
                             mr_order_key(a.m, ni & ~(sn - 1), nj & ~(sn - 1), nk & ~(sn - 1), Ln) != pin_key;
        if (!coupled) cd += cond;
        if (coupled && up) cp[axis] = cond;
        div += (double)d * (double)mr_face_vel(a, axis, fi) * area / V;
      }
    }
    cd = mr_lane_sum(cd, L);
    diag = mr_lane_sum(diag, L);
    div = mr_lane_sum(div, L);
    const bool anchor = fluid && ((i | j | k) & mask) == 0;
    const double Vp = pinned ? 1.0 : V, rhs = pinned ? 0.0 : -div + a.cdiv;
    if (pinned) cd = diag = 1.0;
    if (L == 2) {
      const double sx = mr_lane_sum(cp[0], 2), sy = mr_lane_sum(cp[1], 2), sz = mr_lane_sum(cp[2], 2);
      if (lane == 0) o.cs[b] = make_float4((float)cd, (float)sx, (float)sy, (float)sz);
    }
    const double bv = anchor ? Vp * rhs : 0.0;
    o.b64[c] = bv;
    o.vol64[c] = anchor ? Vp : 0.0;
    o.cd64[c] = anchor ? cd : 0.0;
    o.cd32[c] = anchor ? (float)cd : 0.f;
    o.cx64[c] = cp[0]; o.cy64[c] = cp[1]; o.cz64[c] = cp[2];
    o.cx32[c] = (float)cp[0]; o.cy32[c] = (float)cp[1]; o.cz32[c] = (float)cp[2];
    // (at every entry of the leaf cell, as the vectors)
    o.inv32[c] = fluid && diag > 0.0 ? (float)(1.0 / diag) : 0.f;
    bb += bv * bv;
  }
  double v[1] = {bb};
  const bool mx[1] = {false};
  block_reduce_store<1>(v, mx, a.part, kMaxPartials);
}

}  // namespace pf
