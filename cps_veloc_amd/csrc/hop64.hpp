// hop64.hpp -- FP64 hop kernels for small lattices.
//
// k_dwf_dslash / k_mobius give a (site, slice) to one thread: at 8^3x8 that is
// one wave on half of the chip's SIMDs, each with a serial chain of 8
// neighbours and about 1500 instructions, and a pass takes 10 us whatever the
// lattice.  Here four threads share a (site, slice):
//   hf = 0 / 1 carries the first / second component of every projected
//     two-spinor (spins 0 and 3, or 1 and 2, of an x- or y-neighbour; 0 and 2,
//     or 1 and 3, of a z- or t-neighbour), half of the neighbour's data;
//   z = 0 / 1 walks the x and y, or the z and t, neighbours.
// Each thread has its four neighbours and the epilogue's operands in flight at
// once (they are issued before the links are staged), so that a pass waits for
// memory twice (table, data) instead of once per neighbour.  After the hop the
// threads trade partial sums through LDS: z = 0 owns spin hf, z = 1 spin
// 2 + hf.
// Measured, FP64 MatPcDagMatPc with an event around each of its five launches
// (each event costs about 3 us): DWF 8^3x8 Ls 8 55.4 -> 45.5 us, Mobius
// 6x10x4x12 Ls 10 67.5 -> 56.3 us, DWF 4^3x8 Ls 8 49.3 -> 37.2 us.  What is left
// of a pass (4-6 us) is its launch, two waits for memory and the store; how
// many neighbours are in flight (1 to 4) makes 2 % of difference.  On larger
// lattices the one-thread form wins: the line is in set_shape64().
#pragma once
#include "dwf_kernels.hpp"

namespace dwfk {

typedef cx<double> c64;

// the three complex components a thread owns after the hop: spin 2 z + hf
struct Own {
  int hf, z;
  __device__ __forceinline__ int comp(int c) const { return 6 * z + 3 * hf + c; }
};
__device__ __forceinline__ void ld_own(const c64* __restrict__ d, int vh, int i, const Own& o,
                                       c64* v) {
#pragma unroll
  for (int c = 0; c < 3; ++c) v[c] = d[(size_t)o.comp(c) * vh + i];
}
__device__ __forceinline__ void st_own(c64* __restrict__ d, int vh, int i, const Own& o,
                                       const c64* v) {
#pragma unroll
  for (int c = 0; c < 3; ++c) d[(size_t)o.comp(c) * vh + i] = v[c];
}
__device__ __forceinline__ double norm_own(const c64* v) {
  double n = 0.0;
#pragma unroll
  for (int c = 0; c < 3; ++c) n += v[c].re * v[c].re + v[c].im * v[c].im;
  return n;
}

// stage_links for these kernels: one thread per (direction, link row, site)
__device__ __forceinline__ void stage_links64(c64* __restrict__ lu, const c64* __restrict__ U,
                                              const Geom& g, int blk, int ns, int nsets,
                                              int p_first) {
  const int tid = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
  const int nthr = blockDim.x * blockDim.y * blockDim.z;
  for (int w = tid; w < nsets * 24 * ns; w += nthr) {
    const int il = w & (ns - 1), q = w / ns, row = q % 3, sd = q / 3, d = sd & 7;
    const int i = blk * ns + il;
    if (i >= g.vh) continue;
    const int p = (p_first + (sd >> 3)) & 1;
    const int nbr = g.nbt[(size_t)(p * 8 + d) * g.vh + i] & 0x7fffffff;
    const int site = d >= 4 ? nbr : i;
    const int par = d >= 4 ? 1 - p : p;  // U_mu(x - mu) lives on the other parity
    const c64* src = U + (size_t)(((d & 3) * 2 + par) * 9 + 3 * row) * g.vh + site;
    c64* dst = lu + (size_t)(sd * ns + il) * 9 + 3 * row;
#pragma unroll
    for (int e = 0; e < 3; ++e) dst[e] = src[(size_t)e * g.vh];
  }
}

// this thread's component of (1 + SG gamma_MU) psi from its two spins; hs is
// +1 for hf = 0 and -1 for hf = 1 (the products with +-1 are exact)
template <int MU, int SG>
__device__ __forceinline__ void project64(const c64* u, const c64* w, c64* h, double hs) {
  const double k = SG * hs;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (MU == 0)
      h[c] = u[c] + sgi<SG>(w[c]);
    else if (MU == 1)
      h[c] = c64{fma(-k, w[c].re, u[c].re), fma(-k, w[c].im, u[c].im)};
    else if (MU == 2)
      h[c] = c64{fma(-k, w[c].im, u[c].re), fma(k, w[c].re, u[c].im)};
    else
      h[c] = u[c] + sgr<SG>(w[c]);
  }
}
// the transported component r into spin hf (au) and the lower spin it feeds:
// 3 - hf from x and y, 2 + hf from z and t (al)
template <int MU, int SG>
__device__ __forceinline__ void reconstruct64(c64* au, c64* al, const c64* r, double hs) {
  const double k = SG * hs;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    au[c] = au[c] + r[c];
    if (MU == 0)
      al[c] = al[c] - sgi<SG>(r[c]);
    else if (MU == 1)
      al[c] = c64{fma(-k, r[c].re, al[c].re), fma(-k, r[c].im, al[c].im)};
    else if (MU == 2)
      al[c] = c64{fma(k, r[c].im, al[c].re), fma(-k, r[c].re, al[c].im)};
    else
      al[c] = al[c] + sgr<SG>(r[c]);
  }
}
template <int MU, int SG, bool FWD>
__device__ __forceinline__ void half_dir64(c64* au, c64* al, const c64* u, const c64* w,
                                           const c64* l, double hs) {
  c64 h[3], r[3];
  project64<MU, SG>(u, w, h, hs);
#pragma unroll
  for (int row = 0; row < 3; ++row)
    r[row] = FWD ? row_dot(l[3 * row], l[3 * row + 1], l[3 * row + 2], h[0], h[1], h[2])
                 : row_dotc(l[row], l[3 + row], l[6 + row], h[0], h[1], h[2]);
  reconstruct64<MU, SG>(au, al, r, hs);
}

// as pin12
__device__ __forceinline__ void pin3(c64* v) {
#pragma unroll
  for (int c = 0; c < 3; ++c) asm volatile("" : "+v"(v[c].re), "+v"(v[c].im));
}

// a thread's four neighbours k: +mu -mu +nu -nu with (mu, nu) = (x, y) for
// z = 0 and (z, t) for z = 1, and the hop's partial sums
struct Hop64 {
  int hf, z;
  double hs;
  c64 u[4][3], w[4][3];  // spin hf and the second spin of the projection
  c64 au[3], al[3];
  // staged slot of neighbour k (stage_links64's direction)
  __device__ __forceinline__ int dir(int k) const { return (k & 1) * 4 + (k >> 1) + 2 * z; }

  // issue the loads of all four (in: the slice; p: output parity; inactive
  // lanes read site 0's neighbours)
  __device__ __forceinline__ void load(const c64* __restrict__ in, const Geom& g, int p, int i) {
    const c64* a = in + (size_t)(3 * hf) * g.vh;
    const c64* b = in + (size_t)(z ? 6 + 3 * hf : 9 - 3 * hf) * g.vh;
    int n[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      n[k] = g.nbt[(size_t)(p * 8 + dir(k)) * g.vh + (i < g.vh ? i : 0)] & 0x7fffffff;
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        u[k][c] = a[(size_t)c * g.vh + n[k]];
        w[k][c] = b[(size_t)c * g.vh + n[k]];
      }
#pragma unroll
    for (int c = 0; c < 3; ++c) au[c] = al[c] = c64{0, 0};
  }
  // neighbour k with its staged link
  template <int DAG>
  __device__ __forceinline__ void add(int k, const c64* l) {
    constexpr int SF = DAG ? 1 : -1;  // forward: 1 - s gamma, s = +1 (dag 0) / -1 (dag 1)
    if (z == 0) {
      if (k == 0) half_dir64<0, SF, true>(au, al, u[0], w[0], l, hs);
      if (k == 1) half_dir64<0, -SF, false>(au, al, u[1], w[1], l, hs);
      if (k == 2) half_dir64<1, SF, true>(au, al, u[2], w[2], l, hs);
      if (k == 3) half_dir64<1, -SF, false>(au, al, u[3], w[3], l, hs);
    } else {
      if (k == 0) half_dir64<2, SF, true>(au, al, u[0], w[0], l, hs);
      if (k == 1) half_dir64<2, -SF, false>(au, al, u[1], w[1], l, hs);
      if (k == 2) half_dir64<3, SF, true>(au, al, u[2], w[2], l, hs);
      if (k == 3) half_dir64<3, -SF, false>(au, al, u[3], w[3], l, hs);
    }
    pin3(au);
    pin3(al);
    __builtin_amdgcn_sched_barrier(0);
  }
  // trade the partial sums through mycol (this (site, slice)'s 12 complex, in
  // the links' LDS): z = 0's al is the partner hf's lower spin, z = 1's au the
  // z = 0 thread's upper spin.  Two barriers.
  __device__ __forceinline__ void finish(c64* v, c64* mycol, const Own& o) const {
    const int to = z ? 3 * hf : 9 - 3 * hf;
    __syncthreads();  // every thread is done with the staged links
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const c64 give{z ? au[c].re : al[c].re, z ? au[c].im : al[c].im};
      v[c] = c64{z ? al[c].re : au[c].re, z ? al[c].im : au[c].im};
      mycol[to + c] = give;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = v[c] + mycol[o.comp(c)];
  }
};

// LDS bytes: staged links of nsets parities; the s-columns that reuse them;
// the (b + c D5) exchange slots behind the links (two neighbours a thread)
__host__ __device__ constexpr size_t lds64_links(int ns, int nsets) {
  return (size_t)nsets * 8 * ns * 9 * 16;
}
__host__ __device__ constexpr size_t lds64_cols(int ns, int ls) {
  return (size_t)ns * (ls * 12 + 1) * 16;
}
__host__ __device__ constexpr size_t lds64_tx(int ns, int ls) {
  return lds64_links(ns, 1) + (size_t)4 * ns * ls * 12 * 16;
}

// Sum of partials that every work-group forms for itself, without a barrier of
// its own: the loads at the kernel's start, a value per wave staged before a
// barrier the kernel has anyway, the total after it.  All work-groups of a
// launch add in one order and get the same bits.
struct PartSum {
  double v = 0.0;
  __device__ __forceinline__ void load(const double* __restrict__ p, int n, int tid, int nthr) {
    for (int k = tid; k < n; k += nthr) v += p[k];
  }
  __device__ __forceinline__ void stage(double* sh, int tid) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if ((tid & 63) == 0) sh[tid >> 6] = v;
  }
  static __device__ __forceinline__ double total(const double* sh, int nthr) {
    double t = 0.0;
    for (int w = 0; w < (nthr + 63) / 64; ++w) t += sh[w];
    return t;
  }
};

// What the last pass of a CG step gets of the scalars: *rr = |r|^2 and the
// partials of <p, A p> (n > 0), of which work-group 0 leaves alpha and the sum
// (host: pinned); or, n == 0, rr[1] = <p, A p>.
struct CgScal64 {
  const double* rr;
  const double* dot;
  int n;
  double *alpha, *host;
};
__device__ __forceinline__ double cg_alpha64(const CgScal64& c, const double* sh, int tid,
                                             int nthr) {
  const double d = c.n ? PartSum::total(sh, nthr) : c.rr[1];
  const double a = d != 0.0 ? c.rr[0] / d : 0.0;
  if (c.n && blockIdx.x == 0 && tid == 0) {
    *c.alpha = a;
    c.host[1] = d;
  }
  return a;
}

// End of a CG step: |r|^2 from its partials into *rr_new and host[0] (pinned),
// and the next direction pn = r + (|r|^2 / *rr_old) p of n components, one a
// thread.  The two sums as launches of their own cost an 8^4 Ls 8 DWF step 5.2
// us and two gaps; inside the last pass (7.5 -> 7.9 us) and here (3.4 -> 3.6 us)
// the step takes 40.3 us instead of 46.1.  Every work-group reads
// all partials, one for each 8 or 4 sites: 256 here, 2048 at the line of
// set_shape64() (Ls 2), and on a larger lattice more than the launch saves.
__global__ void __launch_bounds__(256)
k_cg_end64(c64* __restrict__ pn, const c64* __restrict__ r, const c64* __restrict__ p,
           const double* __restrict__ partial, int np, const double* __restrict__ rr_old,
           double* __restrict__ rr_new, double* __restrict__ host, size_t n) {
  __shared__ double sh[4];
  const int tid = threadIdx.x;
  const size_t e = blockIdx.x * (size_t)256 + tid;
  c64 rv{0, 0}, pv{0, 0};
  if (e < n) {
    rv = r[e];
    pv = p[e];
  }
  const double ro = *rr_old;
  PartSum s;
  s.load(partial, np, tid, 256);
  s.stage(sh, tid);
  __syncthreads();
  const double rr = PartSum::total(sh, 256), b = ro != 0.0 ? rr / ro : 0.0;
  if (e < n) pn[e] = rv + b * pv;
  if (e == 0) {
    *rr_new = rr;
    host[0] = rr;
  }
}

// ---------------------------------------------------------------------------
// DWF (as k_dwf_dslash).  CG: r -= alpha_cg (x0 + alpha D in) instead of `out`.
// ---------------------------------------------------------------------------
template <int DAG, int EPI, bool NORM, bool CG>
__global__ void __launch_bounds__(512)
k_dwf64(c64* __restrict__ out, const c64* __restrict__ in, const c64* __restrict__ U,
        const c64* __restrict__ x0, double* __restrict__ partial, Geom g, int cb_in,
        double two_a5, double nm_two_a5, double alpha, c64* __restrict__ r, CgScal64 cs,
        const double* __restrict__ mass, size_t vs) {
  // batched operator: right-hand side blockIdx.y starts vs components further
  // and has its own mass
  if (mass) {
    const size_t off = blockIdx.y * vs;
    in += off;
    out += off;
    x0 += off;
    nm_two_a5 = -mass[blockIdx.y] * two_a5;
  }
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double sh[16], shd[8];
  const int ns = blockDim.x >> 1, s = threadIdx.y;
  const Own o{(int)threadIdx.x >= ns ? 1 : 0, (int)threadIdx.z};
  const int il = threadIdx.x - o.hf * ns;
  c64* lu = reinterpret_cast<c64*>(smem_raw);  // [2][8][ns][9]
  c64* mycol = lu + il * (g.ls * 12 + 1) + s * 12;
  const int tid = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
  const int nthr = blockDim.x * blockDim.y * blockDim.z;
  const int blk = xcd_block(g.nxcd, g.rev);
  const int i = blk * ns + il;
  const bool act = i < g.vh;
  const size_t slice = (size_t)12 * g.vh;
  Hop64 hop{o.hf, o.z, o.hf ? -1.0 : 1.0};
  hop.load(in + s * slice, g, (1 + cb_in + s) & 1, i);
  // fifth dimension: dag 0 takes the upper spins from s-1 and the lower ones
  // from s+1, dag 1 the reverse
  const bool minus = (o.z == 0) == (DAG == 0);
  const int s5 = minus ? (s > 0 ? s - 1 : g.ls - 1) : (s < g.ls - 1 ? s + 1 : 0);
  const double c5 = (minus ? s > 0 : s < g.ls - 1) ? two_a5 : nm_two_a5;
  c64 f[3], x[3], rv[3];
  if (act) {
    ld_own(in + s5 * slice, g.vh, i, o, f);
    if (EPI == 1) ld_own(x0 + s * slice, g.vh, i, o, x);
    if (CG) ld_own(r + s * slice, g.vh, i, o, rv);
  }
  PartSum dot;
  if (CG) dot.load(cs.dot, cs.n, tid, nthr);
  __builtin_amdgcn_sched_barrier(0);
  stage_links64(lu, U, g, blk, ns, 2, (1 + cb_in) & 1);
  if (CG) dot.stage(shd, tid);
  __syncthreads();
  const double a_cg = CG ? cg_alpha64(cs, shd, tid, nthr) : 0.0;
  const int set = (s & 1) * 8;
#pragma unroll
  for (int k = 0; k < 4; ++k) hop.add<DAG>(k, lu + (size_t)((set + hop.dir(k)) * ns + il) * 9);
  c64 v[3];
  hop.finish(v, mycol, o);
  double nrm = 0.0;
  if (act) {
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = v[c] + c5 * f[c];
    if (EPI == 1) {
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c] = x[c] + alpha * v[c];
      if (NORM) nrm = norm_own(v);
    }
    if (CG) {
#pragma unroll
      for (int c = 0; c < 3; ++c)
        rv[c] = c64{-a_cg * v[c].re + rv[c].re, -a_cg * v[c].im + rv[c].im};
      st_own(r + s * slice, g.vh, i, o, rv);
      nrm = norm_own(rv);
    } else {
      st_own(out + s * slice, g.vh, i, o, v);
    }
  }
  if (NORM || CG) {
    const double t = block_sum(nrm, sh);
    if (threadIdx.x + threadIdx.y + threadIdx.z == 0) partial[blockIdx.x] = t;
  }
}

// ---------------------------------------------------------------------------
// Mobius (as k_mobius; dag 0 without FL_PRE_T trades (b + c D5) through LDS)
// ---------------------------------------------------------------------------
template <int DAG, int EPI, int FL>
__global__ void __launch_bounds__(512)
k_mobius64(c64* __restrict__ out, const c64* __restrict__ in, const c64* __restrict__ psi,
           const c64* __restrict__ U, double* __restrict__ partial, Geom g, int p_out, MobArgs a,
           c64* __restrict__ r, CgScal64 cs) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double sh[16], shd[8];
  const int ns = blockDim.x >> 1, s = threadIdx.y, ls = g.ls;
  const Own o{(int)threadIdx.x >= ns ? 1 : 0, (int)threadIdx.z};
  const int il = threadIdx.x - o.hf * ns;
  const int sst = ls * 12 + 1;
  c64* lu = reinterpret_cast<c64*>(smem_raw);   // [8][ns][9]
  c64* col = reinterpret_cast<c64*>(smem_raw);  // s-columns, once the hop is done
  c64* mysite = col + il * sst;
  c64* mycol = mysite + s * 12;
  const int ct = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
  const int cthr = blockDim.x * blockDim.y * blockDim.z;
  const int blk = xcd_block(g.nxcd, g.rev);
  const int i = blk * ns + il;
  const bool act = i < g.vh;
  const int nvalid = min(ns, g.vh - blk * ns);
  const size_t slice = (size_t)12 * g.vh;
  const int sm = s > 0 ? s - 1 : ls - 1, sp = s < ls - 1 ? s + 1 : 0;
  Hop64 hop{o.hf, o.z, o.hf ? -1.0 : 1.0};
  hop.load(in + s * slice, g, p_out, i);
  c64 w[3], rv[3], v[3];
  if (EPI == EPI_SCHUR && act) ld_own(psi + s * slice, g.vh, i, o, w);
  if ((FL & FL_CG) && act) ld_own(r + s * slice, g.vh, i, o, rv);
  PartSum dot;
  if (FL & FL_CG) dot.load(cs.dot, cs.n, ct, cthr);
  __builtin_amdgcn_sched_barrier(0);
  stage_links64(lu, U, g, blk, ns, 1, p_out);
  if (FL & FL_CG) dot.stage(shd, ct);
  __syncthreads();
  const double a_cg = (FL & FL_CG) ? cg_alpha64(cs, shd, ct, cthr) : 0.0;
  if constexpr (DAG == 0 && !(FL & FL_PRE_T)) {
    // (b + c D5) in of each neighbour: spin hf of slice s - 1 and the second
    // spin (a lower one) of slice s + 1 from those slices' threads, two
    // neighbours at a time (component c of thread t at tx[c * nthr + t])
    c64* tx = reinterpret_cast<c64*>(smem_raw + lds64_links(ns, 1));
    const int nx = 2 * ns, nthr = 2 * nx * ls, t0 = threadIdx.x + nx * ls * o.z;
    const int tid = t0 + nx * s, tp = t0 + nx * sm, tn = t0 + nx * sp;
    const double cm = s > 0 ? a.c : a.mc, cp = s < ls - 1 ? a.c : a.mc;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h) __syncthreads();  // the first pair's readers are done
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          tx[(6 * q + c) * nthr + tid] = hop.u[2 * h + q][c];
          tx[(6 * q + 3 + c) * nthr + tid] = hop.w[2 * h + q][c];
        }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int k = 2 * h + q;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          hop.u[k][c] = a.b * hop.u[k][c] + cm * tx[(6 * q + c) * nthr + tp];
          hop.w[k][c] = a.b * hop.w[k][c] + cp * tx[(6 * q + 3 + c) * nthr + tn];
        }
        hop.add<0>(k, lu + (size_t)(hop.dir(k) * ns + il) * 9);
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) hop.add<DAG>(k, lu + (size_t)(hop.dir(k) * ns + il) * 9);
  }
  hop.finish(v, mycol, o);
  if (DAG == 0 && EPI == EPI_PLAIN) {
    if (act) st_own(out + s * slice, g.vh, i, o, v);
    return;
  }
  // coefficient and source of the fifth-dimension terms at the owned spin
  const bool minus = (o.z == 0) == (DAG == 0);
  const bool wall = minus ? s == 0 : s == ls - 1;
  const c64* side = mysite + (minus ? sm : sp) * 12 + o.comp(0);
  c64* own = mycol + o.comp(0);
  if (DAG == 1) {
    // (b + c D5^dag) on the hop's output
#pragma unroll
    for (int c = 0; c < 3; ++c) own[c] = v[c];
    __syncthreads();
    const double ct = wall ? a.mc : a.c;
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = a.b * v[c] + ct * side[c];
    if (EPI == EPI_PLAIN) {
      if (act) st_own(out + s * slice, g.vh, i, o, v);
      return;
    }
    __syncthreads();
  }
  if (EPI == EPI_SCHUR) {
    // psi + K D5 psi through the s-column, and the hop's term
    if (act)
#pragma unroll
      for (int c = 0; c < 3; ++c) own[c] = w[c];
    __syncthreads();
    double nrm = 0.0;
    if (act) {
      const double ck = wall ? a.mK : a.K;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        w[c] = w[c] + ck * side[c];
        w[c] = w[c] + (DAG ? v[c] : -a.kappa_b * v[c]);
      }
      if (FL & FL_NORM) nrm = norm_own(w);
      if (FL & FL_CG) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
          rv[c] = c64{-a_cg * w[c].re + rv[c].re, -a_cg * w[c].im + rv[c].im};
        st_own(r + s * slice, g.vh, i, o, rv);
        nrm = norm_own(rv);
      } else {
        st_own(out + s * slice, g.vh, i, o, w);
      }
    }
    if (FL & (FL_NORM | FL_CG)) {
      const double t = block_sum(nrm, sh);
      if (threadIdx.x + threadIdx.y + threadIdx.z == 0) partial[blockIdx.x] = t;
    }
    return;
  }
  const double kb = DAG ? -a.kappa_b : a.kappa_b;
#pragma unroll
  for (int c = 0; c < 3; ++c) own[c] = kb * v[c];
  __syncthreads();
  m5inv_columns<DAG>(col, sst, ns, nvalid, ls, a.m5);
  __syncthreads();
  if (act) {
    if (DAG == 0 && (FL & FL_POST_T)) {
      const double ct = wall ? a.mc : a.c;
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c] = a.b * own[c] + ct * side[c];
    } else {
      const double sc = DAG ? a.kappa_b : 1.0;
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c] = sc * own[c];
    }
    st_own(out + s * slice, g.vh, i, o, v);
  }
}

}  // namespace dwfk
