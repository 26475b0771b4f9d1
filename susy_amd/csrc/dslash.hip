// Twisted fermion operator D and D^dagger on the A4* lattice
// (reference: 4d_Q16/susy/utilities.c:141-865), one fused gather-only kernel.
//
// Every thread owns one output matrix (one of the 16 Twist_Fermion components)
// of one site and sums all terms landing on it:
//   site  eta      : DbminusLtoS + detLtoS                 (10 matmuls)
//   link  psi_b    : Dminus + DbplusStoL + detStoL          (10 matmuls)
//   plaq  chi_ab   : Dplus + DbplusPtoP + DbminusPtoP       (10 matmuls)
// so no output is written twice and no atomics are needed.  D^dagger uses
// D^dagger v = -(D v^dagger)^dagger (utilities.c:780-788, 856-864): the
// adjoint is applied on the loads and the stores, in registers.
//
// NCOL <= 4 complex matrix products are VALU FMA chains: an output matrix
// accumulates in registers, the right operand of each product is held in
// registers while the left operand streams element by element.
//
// Memory access goes through raw buffer loads: each field has a 128-bit buffer
// descriptor in SGPRs, a lane supplies only the 32-bit byte offset of its
// site, and the matrix-element offset is a uniform SGPR offset computed on
// the scalar unit.  This keeps address arithmetic out of the VGPR budget, and
// the descriptor's record count bounds every access.
//
// Block mapping is XCD-aware: consecutive hardware block ids are dealt to the
// 8 XCDs round-robin.  The ids are remapped so that each XCD walks one
// contiguous slab of site chunks, all 16 component-blocks of a chunk back to
// back: neighbouring chunks (the z and t neighbours of a site) then share the
// same L2.
#include "dev_buf.h"

#include <mutex>

__constant__ PlaqTerms c_pt;

int dslash_init_tables(const PlaqTerms &pt) {
  HIPCHK(hipMemcpyToSymbol(HIP_SYMBOL(c_pt), &pt, sizeof(PlaqTerms)));
  return 0;
}

// minimum wavefronts per SIMD the register allocator must allow.  From
// U(5) on an FP64 output matrix and its operands exceed 256 registers; at one
// wave per SIMD the allocator keeps the excess in AGPRs instead of spilling
// it to scratch memory.
#ifndef DS_WAVES
#define DS_WAVES (NCOL >= 5 ? 1 : 2)
#endif
#ifndef DS_WAVES64
#define DS_WAVES64 DS_WAVES
#endif
#ifndef DS_WAVES32
#define DS_WAVES32 DS_WAVES
#endif
// dynamic LDS bytes requested per block: caps the blocks resident per CU
// (160 KB of LDS per CU), and with it the sites in flight per XCD, whose
// neighbourhood must fit the XCD's L2.  0 leaves occupancy to registers.
#ifndef DS_OCC_LDS64
#define DS_OCC_LDS64 0
#endif
#ifndef DS_OCC_LDS32
#define DS_OCC_LDS32 0
#endif
// unroll factor of the term loops (a wave can issue the next product's
// loads before the current product's FMAs when registers allow)
#ifndef DS_UNROLL
#define DS_UNROLL 1
#endif
#define DS_STR(x) #x
#define DS_UNROLL_LOOP(n) _Pragma(DS_STR(unroll n))

// cache policy of the output stores: k_dslash's are non-temporal (2), so the
// written lines, which this launch never reads again, do not displace the
// neighbour gathers' source lines in L2 (FP32 CG iteration -0.8%, FP64 -1.8%
// at 12^3x24).  k_dslash_split's are ordinary ones (0): its fields fit L2,
// and the next kernel finds them there (CG iteration, us, non-temporal ->
// ordinary: U(2) 4^4 36.4 -> 31.1, U(3) 4^4 38.0 -> 34.7, U(4) 8^4 FP32 76.7
// -> 75.0).
#define DS_STORE_NT 2
#define DS_STORE_L2 0
// (callers keep the stored values live until the stores have read them:
// hold() after the last store, see st_keep)
template <int POLICY>
__device__ __forceinline__ void bstore(double2 v, Rsrc r, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned, v), r, voff, soff, POLICY);
}
template <int POLICY>
__device__ __forceinline__ void bstore(float2 v, Rsrc r, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(__attribute__((ext_vector_type(2))) unsigned, v), r, voff, soff, POLICY);
}

template <typename R>
__device__ __forceinline__ R bcsign(int t, int dt, int nt, R pbc) {
  int tt = t + dt;
  return (tt < 0 || tt > nt - 1) ? pbc : (R)1;
}

// Pre-pass for the plaquette-determinant terms (doG): per site
//   aux[0] = Tr eta,  aux[1+a] = Tr(U_a^-1 psi_a)
// with eta, psi taken adjointed for D^dagger (utilities.c:793-799, 706-712).
// One thread per site: for lattices whose sites fill the chip.
template <typename R, bool DAG>
__global__ void __launch_bounds__(256)
k_dslash_prep(const typename CT<R>::t *__restrict__ src,
              const typename CT<R>::t *__restrict__ Uinv,
              typename CT<R>::t *__restrict__ aux, int V, const int *__restrict__ skip) {
  typedef typename CT<R>::t C;
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= V || (skip != nullptr && *skip)) return;
  C t[1 + NUMLINK];
  t[0] = mkc<C>(0, 0);
#pragma unroll
  for (int i = 0; i < NCOL; i++) {
    C v = src[(i * NCOL + i) * V + s];
    t[0].x += v.x;
    t[0].y += DAG ? -v.y : v.y;
  }
#pragma unroll
  for (int a = 0; a < NUMLINK; a++) {
    const C *psi = src + (size_t)(1 + a) * NN * V + s;
    const C *ui = Uinv + (size_t)a * NN * V + s;
    C ta = mkc<C>(0, 0);
#pragma unroll
    for (int i = 0; i < NCOL; i++)
#pragma unroll
      for (int j = 0; j < NCOL; j++) {
        C u = ui[(i * NCOL + j) * V];
        C p = DAG ? psi[(i * NCOL + j) * V] : psi[(j * NCOL + i) * V];
        if (DAG) p.y = -p.y;
        ta.x += u.x * p.x - u.y * p.y;
        ta.y += u.x * p.y + u.y * p.x;
      }
    t[1 + a] = ta;
  }
  vm_drain();
#pragma unroll
  for (int a = 0; a <= NUMLINK; a++) st_keep(aux + (size_t)a * V + s, t[a]);
}

// The same values with one thread per site and trace (blockIdx.y): six times
// the waves hide the latency of a thread's loads.  The line lies where both
// take the same time (us, pre-pass and D, k_dslash_prep | this, FP64): U(4)
// 1296 sites 22.4 | 17.6, 8192 54.1 | 50.4, 65536 417.7 | 416.3; U(2) 8192
// 16.8 | 15.6, 65536 95.4 | 96.9; at U(4) 131072 the pre-pass alone 60 | 67.
#define PREP_TRACE_V 65536
template <typename R, bool DAG>
__global__ void __launch_bounds__(256)
k_dslash_prep_trace(const typename CT<R>::t *__restrict__ src,
                    const typename CT<R>::t *__restrict__ Uinv,
                    typename CT<R>::t *__restrict__ aux, int V, const int *__restrict__ skip) {
  typedef typename CT<R>::t C;
  const int s = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y;
  if (s >= V || (skip != nullptr && *skip)) return;
  const C *psi = src + (size_t)k * NN * V + s;
  C t = mkc<C>(0, 0);
  if (k == 0) {
#pragma unroll
    for (int i = 0; i < NCOL; i++) {
      const C v = psi[(i * NCOL + i) * V];
      t.x += v.x;
      t.y += DAG ? -v.y : v.y;
    }
  } else {
    const C *ui = Uinv + (size_t)(k - 1) * NN * V + s;
#pragma unroll
    for (int i = 0; i < NCOL; i++)
#pragma unroll
      for (int j = 0; j < NCOL; j++) {
        C u = ui[(i * NCOL + j) * V];
        C p = DAG ? psi[(i * NCOL + j) * V] : psi[(j * NCOL + i) * V];
        if (DAG) p.y = -p.y;
        t.x += u.x * p.x - u.y * p.y;
        t.y += u.x * p.y + u.y * p.x;
      }
  }
  vm_drain();
  st_keep(aux + (size_t)k * V + s, t);
}

template <typename R> struct DsSites;
template <> struct DsSites<double> {
  static constexpr int n = DS_SITES64, waves = DS_WAVES64;
};
template <> struct DsSites<float> {
  static constexpr int n = DS_SITES32, waves = DS_WAVES32;
};

// EPI = 0: dst = result.  EPI = 1: dst = result + shift * p0, and the block's
// partial sum of Re Tr(p0^dag dst) goes to partial[block].
// With aux_out (D, EPI = 0 only) the blocks of the site and link components
// also store the pre-pass values of D^dagger applied to this output:
// aux_out[0] = Tr(out_0)^*, aux_out[1+a] = Tr(U_a^-1 out_{1+a}^dag).
//
// A block covers ord.sites sites (at most DsSites::n, see ds_sites) of one
// output component.  (Two threads sharing an output matrix: 10-15% slower.)
// What bounds it on large lattices is the operand lines that L1 misses (U(4)
// 16^3x32: 8.6e7 of 128 bytes a launch in FP64, 4.6e7 in FP32; 96 and 65 in
// flight per CU at 480 and 370 cycles each).  The lines that the L2 misses are
// not it alone: tiled orders of a layout of whole matrices halved them without
// a matching gain in time.
template <typename R, bool DAG, int EPI>
__global__ void __launch_bounds__(DsSites<R>::n)
    __attribute__((amdgpu_waves_per_eu(DsSites<R>::waves)))
k_dslash(const typename CT<R>::t *__restrict__ src, typename CT<R>::t *__restrict__ dst,
         const typename CT<R>::t *__restrict__ U, const typename CT<R>::t *__restrict__ Uinv,
         const typename CT<R>::t *__restrict__ pdet, const typename CT<R>::t *__restrict__ aux,
         typename CT<R>::t *__restrict__ aux_out,
         const int *__restrict__ nbr, const int *__restrict__ tco, int V, int nt,
         R pbc, int doG, R G, DsOrder ord,
         const typename CT<R>::t *__restrict__ p0,
         R shift, double *__restrict__ partial, const int *__restrict__ skip) {
  typedef typename CT<R>::t C;
  // a solver that has converged leaves its remaining queued launches idle
  // (the flag is one word read by every thread: the exit is block-uniform)
  if (skip != nullptr && *skip) return;
  const int L = blockIdx.x;
  const int lane = threadIdx.x, sites = ord.sites;
  const int q = L >> 3, comp = q % NTF;       // position in this XCD's queue
  const int qq = q / NTF;                     // chunk position in the queue
  int s;
  const bool live = ord_site(ord, sites, L & 7, qq, lane, V, &s);

  const uint32_t cs = sizeof(C);
  const uint32_t pl = (uint32_t)V * cs;     // one element plane
  const uint32_t Mb = NN * pl;              // one matrix field
  const Rsrc rS = make_rsrc(src, NTF * Mb), rU = make_rsrc(U, NUMLINK * Mb);
  const Rsrc rN = make_rsrc(nbr, (uint32_t)NGATHER * V * 4u);
  auto nb = [&](int g) { return bload_i32(rN, (uint32_t)s * 4u, (uint32_t)g * V * 4u); };
  auto S = [&](int k, int x) { return Opnd{rS, (uint32_t)x * cs, (uint32_t)k * Mb}; };
  auto Ul = [&](int a, int x) { return Opnd{rU, (uint32_t)x * cs, (uint32_t)a * Mb}; };

  // The determinant sums' gathered scalars: 20 (site) or 4 (link) round trips
  // to memory one after the other were up to a third of a wave's time, so
  // their loads go out together.  FP64 from U(4) on has as many lines in flight
  // as a CU keeps (96 at 16^3x32) and loses by it; so does FP32 at U(5), at every
  // size (with the same three waves per SIMD).  us of a CG iteration, in turn | together: U(4) FP32
  // 8^3x16 107 | 99, 12^3x24 462 | 453, 16^4 738 | 730; U(3) FP64 8^3x16 89.3 |
  // 86.5, 16^4 712 | 706; but U(4) FP64 16^4 1337 | 1394, U(5) FP32 4^4 75 | 92,
  // 8^4 125 | 161, 8^3x16 176 | 211, 12^4 438 | 495, 16^4 1333 | 1438.
  constexpr bool det_together = NCOL <= 3 || (sizeof(R) == 4 && NCOL == 4);
  constexpr int det_unroll = det_together ? NUMLINK : 1;
  C acc[NCOL][NCOL];
#pragma unroll
  for (int i = 0; i < NCOL; i++)
#pragma unroll
    for (int k = 0; k < NCOL; k++) acc[i][k] = mkc<C>(0, 0);

  if (live) {
    const int t = tco[s];

    if (comp == 0) {
      // ---- site output: 1/2 sum_a [psi_a(x) Ubar_a(x) - bc(-a) Ubar_a(x-a) psi_a(x-a)]
      DS_UNROLL_LOOP(DS_UNROLL)
      for (int a = 0; a < NUMLINK; a++) {
        const int xm = nb(g_bwd(a));
        mmacc<R, DAG, true>(acc, (R)0.5, S(1 + a, s), Ul(a, s), pl);
        mmacc<R, true, DAG>(acc, (R)-0.5 * bcsign<R>(t, -link_tau(a), nt, pbc), Ul(a, xm),
                            S(1 + a, xm), pl);
      }
      if (doG) {
        // detLtoS: -(i G C2 sqrt(N)/2) sum_{a!=b} plaqdet_ab [T_b(x) + bc(b) T_a(x+b)]
        //          * Lambda_{DIMF-1},  Lambda_{DIMF-1} = i I / sqrt(N)
        const Rsrc rA = make_rsrc(aux, 6 * pl), rP = make_rsrc(pdet, NUMLINK * NUMLINK * pl);
        C sum = mkc<C>(0, 0);
        int xf[NUMLINK];
#pragma unroll
        for (int b = 0; b < NUMLINK; b++)
          if (det_together) xf[b] = nb(g_fwd(b));
        DS_UNROLL_LOOP(det_unroll)
        for (int b = 0; b < NUMLINK; b++) {
          if (det_together && sizeof(R) == 8) __builtin_amdgcn_sched_barrier(0);
          const int xb = det_together ? xf[b] : nb(g_fwd(b));
          const C tb = bload<C>(rA, (uint32_t)s * cs, (1 + b) * pl);
          const R sg = bcsign<R>(t, link_tau(b), nt, pbc);
          DS_UNROLL_LOOP(det_unroll)
          for (int a = 0; a < NUMLINK; a++) {
            if (a == b) continue;
            const C ta = bload<C>(rA, (uint32_t)xb * cs, (1 + a) * pl);
            const C t2 = mkc<C>(tb.x + sg * ta.x, tb.y + sg * ta.y);
            const C pd = bload<C>(rP, (uint32_t)s * cs, (a * NUMLINK + b) * pl);
            sum.x += pd.x * t2.x - pd.y * t2.y;
            sum.y += pd.x * t2.y + pd.y * t2.x;
          }
        }
        // trd = i lg sum; acc -= trd * (i/sqrt N) I = (lg/sqrt N) sum I
        const R f = (R)(0.5 * C2) * G;  // lg / sqrt(N) = G C2 / 2
#pragma unroll
        for (int i = 0; i < NCOL; i++) {
          acc[i][i].x += f * sum.x;
          acc[i][i].y += f * sum.y;
        }
      }
    } else if (comp <= NUMLINK) {
      // ---- link output b
      const int b = comp - 1;
      const int xb = nb(g_fwd(b));
      DS_UNROLL_LOOP(DS_UNROLL)
      for (int a = 0; a < NUMLINK; a++) {
        if (a == b) continue;
        // Dminus: U_a(x+b) chi_ab(x) - bc(-a) chi_ab(x-a) U_a(x-a)
        const int xm = nb(g_bwd(a));
        const R sg = a < b ? (R)1 : (R)-1;   // chi_ab = sg * stored chi_{min,max}
        const int pc = 6 + plaq_idx(a, b);
        mmacc<R, false, DAG>(acc, sg, Ul(a, xb), S(pc, s), pl);
        mmacc<R, DAG, false>(acc, -sg * bcsign<R>(t, -link_tau(a), nt, pbc), S(pc, xm),
                             Ul(a, xm), pl);
      }
      // DbplusStoL: 1/2 [bc(b) eta(x+b) Ubar_b(x) - Ubar_b(x) eta(x)]
      mmacc<R, DAG, true>(acc, (R)0.5 * bcsign<R>(t, link_tau(b), nt, pbc), S(0, xb), Ul(b, s),
                          pl);
      mmacc<R, true, DAG>(acc, (R)-0.5, Ul(b, s), S(0, s), pl);
      if (doG) {
        // detStoL: -G C2/2 U_b^-1(x) sum_{c!=b} [Tr eta(x) plaqdet_cb(x)
        //                                        + bc(-c) Tr eta(x-c) plaqdet_bc(x-c)]
        const Rsrc rA = make_rsrc(aux, 6 * pl), rP = make_rsrc(pdet, NUMLINK * NUMLINK * pl);
        const Rsrc rI = make_rsrc(Uinv, NUMLINK * Mb);
        C sum = mkc<C>(0, 0);
        const C te = bload<C>(rA, (uint32_t)s * cs, 0);
        DS_UNROLL_LOOP(det_unroll)
        for (int n = 0; n < (det_together ? NUMLINK - 1 : NUMLINK); n++) {
          const int c = det_together ? n + (n >= b) : n;
          if (c == b) continue;
          const int xm = nb(g_bwd(c));
          const C p1 = bload<C>(rP, (uint32_t)s * cs, (c * NUMLINK + b) * pl);
          const C p2 = bload<C>(rP, (uint32_t)xm * cs, (b * NUMLINK + c) * pl);
          const C tm = bload<C>(rA, (uint32_t)xm * cs, 0);
          const R sg = bcsign<R>(t, -link_tau(c), nt, pbc);
          sum.x += te.x * p1.x - te.y * p1.y + sg * (tm.x * p2.x - tm.y * p2.y);
          sum.y += te.x * p1.y + te.y * p1.x + sg * (tm.x * p2.y + tm.y * p2.x);
        }
        const R f = (R)(-0.5 * C2) * G;
        const R sr = f * sum.x, si = f * sum.y;
#pragma unroll
        for (int i = 0; i < NCOL; i++)
#pragma unroll
          for (int k = 0; k < NCOL; k++) {
            const C u = bload<C>(rI, (uint32_t)s * cs, b * Mb + (i * NCOL + k) * pl);
            acc[i][k].x += sr * u.x - si * u.y;
            acc[i][k].y += sr * u.y + si * u.x;
          }
      }
    } else {
      // ---- plaquette output (a,b), a<b
      const int p = comp - 1 - NUMLINK;
      const int a = c_pt.a[p], b = c_pt.b[p];
      const int xa = nb(g_fwd(a)), xb = nb(g_fwd(b));
      // Dplus: bc(a) U_a(x) psi_b(x+a) - psi_b(x) U_a(x+b)
      //        - bc(b) U_b(x) psi_a(x+b) + psi_a(x) U_b(x+a)
      mmacc<R, false, DAG>(acc, bcsign<R>(t, link_tau(a), nt, pbc), Ul(a, s), S(1 + b, xa), pl);
      mmacc<R, DAG, false>(acc, (R)-1, S(1 + b, s), Ul(a, xb), pl);
      mmacc<R, false, DAG>(acc, -bcsign<R>(t, link_tau(b), nt, pbc), Ul(b, s), S(1 + a, xb), pl);
      mmacc<R, DAG, false>(acc, (R)1, S(1 + a, s), Ul(b, xa), pl);
      // DbplusPtoP + DbminusPtoP.  Each DbminusPtoP term landing on (a,b)
      // coincides with the DbplusPtoP term of the same c: with (d,e) the
      // other two links, x-d-e = x+a+b+c and x-d-e-c = x+a+b (the five e_a
      // sum to zero), perm(d,e,c,a,b) = perm(a,b,c,d,e), and the temporal
      // offsets agree for the same reason.  The DbplusPtoP terms are applied
      // at double weight (checked term by term when the tables are built).
      DS_UNROLL_LOOP(DS_UNROLL)
      for (int n = 0; n < 3; n++) {
        const int c = c_pt.pp_c[p][n];
        const int pc = 6 + c_pt.pp_de[p][n];
        const int x1 = nb(c_pt.pp_g1[p][n]), x2 = nb(c_pt.pp_g2[p][n]), xmc = nb(g_bwd(c));
        const R tr = (R)(2.0f * c_pt.pp_tr[p][n]);
        mmacc<R, DAG, true>(acc, tr * bcsign<R>(t, c_pt.pp_dt3[p][n], nt, pbc), S(pc, x2),
                            Ul(c, x1), pl);
        mmacc<R, true, DAG>(acc, -tr * bcsign<R>(t, c_pt.pp_dt2[p][n], nt, pbc), Ul(c, xmc),
                            S(pc, x1), pl);
      }
    }
  }

  double dot = 0.0;
  if (live) {
    // ---- epilogue loads (p0 for the DSq epilogue, U^-1 for the D^dagger
    // pre-pass values), all drained before the first store
    const Rsrc rD = make_rsrc(dst, NTF * Mb);
    const bool pre = !DAG && EPI == 0 && aux_out != nullptr && comp <= NUMLINK;
    C q[NCOL][NCOL];
    if (EPI == 1) {
      const Rsrc rQ = make_rsrc(p0, NTF * Mb);
#pragma unroll
      for (int i = 0; i < NCOL; i++)
#pragma unroll
        for (int k = 0; k < NCOL; k++)
          q[i][k] = bload<C>(rQ, (uint32_t)s * cs, comp * Mb + (i * NCOL + k) * pl);
    } else if (pre && comp > 0) {
      const Rsrc rI = make_rsrc(Uinv, NUMLINK * Mb);
#pragma unroll
      for (int i = 0; i < NCOL; i++)
#pragma unroll
        for (int k = 0; k < NCOL; k++)
          q[i][k] = bload<C>(rI, (uint32_t)s * cs, (comp - 1) * Mb + (i * NCOL + k) * pl);
    }
    vm_drain();
    // ---- store (D^dagger: negated adjoint); the stored values stay live
    // until one wait after the last store reports their registers read
    C out[NCOL][NCOL];
#pragma unroll
    for (int i = 0; i < NCOL; i++)
#pragma unroll
      for (int k = 0; k < NCOL; k++) {
        C v = DAG ? mkc<C>(-acc[k][i].x, acc[k][i].y) : acc[i][k];
        const uint32_t so = comp * Mb + (i * NCOL + k) * pl;
        if (EPI == 1) {
          v.x = fma(shift, q[i][k].x, v.x);
          v.y = fma(shift, q[i][k].y, v.y);
          dot += (double)q[i][k].x * (double)v.x + (double)q[i][k].y * (double)v.y;
        }
        bstore<DS_STORE_NT>(v, rD, (uint32_t)s * cs, so);
        out[i][k] = v;
      }
#pragma unroll
    for (int i = 0; i < NCOL; i++)
#pragma unroll
      for (int k = 0; k < NCOL; k++) hold(out[i][k]);
    if (pre) {
      C tr = mkc<C>(0, 0);
      if (comp == 0) {
#pragma unroll
        for (int i = 0; i < NCOL; i++) {
          tr.x += acc[i][i].x;
          tr.y -= acc[i][i].y;
        }
      } else {
#pragma unroll
        for (int i = 0; i < NCOL; i++)
#pragma unroll
          for (int j = 0; j < NCOL; j++) {
            const C u = q[i][j], p = acc[i][j];
            tr.x += u.x * p.x + u.y * p.y;
            tr.y += u.y * p.x - u.x * p.y;
          }
      }
      st_keep(aux_out + (size_t)comp * V + s, tr);
    }
  }
  if (EPI == 1) {
    // deterministic block reduction: wavefront butterfly, then across waves
    for (int off = 32; off > 0; off >>= 1) dot += __shfl_xor(dot, off, 64);
    __shared__ double red[DsSites<R>::n / 64];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = dot;
    __syncthreads();
    if (threadIdx.x == 0) {
      double tsum = 0;
      for (int u = 0; u < sites / 64; u++) tsum += red[u];
      partial[L] = tsum;
    }
  }
}

#define DS_PARTS 5   // waves of k_dslash_split's block
#if NCOL <= 4
// The operator for lattices whose components and sites alone leave the chip
// mostly idle: the ten products of an output matrix are shared by five waves
// (two products each), which meet in LDS.  k_dslash makes them one after the
// other, each behind its own loads, and that chain of memory latencies is
// all its time on a small lattice.
//
// A block is 5 waves on one output component of 64 sites.  Wave w takes, for
// the site, a = w; for link b, the w-th a != b or (w = 4) the StoL pair; for a
// plaquette, one half of Dplus or (w >= 2) one PtoP pair.  The determinant
// terms' sums over neighbours are shared the same way.
//
// What bounds it is still latency: gathered loads, then LDS and two barriers
// (U(4) 6^3x10: 83% L2 hits, 38 lines in flight per CU in FP64 and 22 in FP32 at
// 190-260 cycles each, waves waiting 44% of their time).
// FP32 holds its partial matrices in two rounds of half the LDS and asks for
// five waves per SIMD (U(4) D: four, what its registers allow without
// scratch); FP64 asks for two.  At U(4) its 87 KB of LDS leave a CU one block,
// five waves, whatever its registers, so fewer registers gained nothing there.
// D with its pre-pass, us, FP64 | FP32, k_dslash -> this kernel:
//   U(4) 4^3x8 23.7 -> 10.2 | 19.0 -> 9.4, 6^3x10 27.9 -> 23.3 | 24.9 -> 15.6
//   U(3) 4^3x8 15.5 -> 8.0 | 13.9 -> 7.4, 6^3x10 19.3 -> 15.2 | 18.2 -> 11.3
//   U(2) 4^4 10.2 -> 4.7 | 9.8 -> 4.7, 8^3x16 16.8 -> 14.7 | 16.7 -> 12.6
// INL makes the pre-pass values in this kernel (ds_split_inline).
template <typename R>
constexpr int ds_split_waves(bool dag, bool inl) {
  return sizeof(R) == 8 || inl ? 2 : NCOL == 4 && !dag ? 4 : 5;
}
template <typename R, bool DAG, int EPI, bool INL>
__global__ void __launch_bounds__(64 * DS_PARTS)
    __attribute__((amdgpu_waves_per_eu(ds_split_waves<R>(DAG, INL))))
k_dslash_split(const typename CT<R>::t *__restrict__ src, typename CT<R>::t *__restrict__ dst,
               const typename CT<R>::t *__restrict__ U,
               const typename CT<R>::t *__restrict__ Uinv,
               const typename CT<R>::t *__restrict__ pdet,
               const typename CT<R>::t *__restrict__ aux, typename CT<R>::t *__restrict__ aux_out,
               const int *__restrict__ nbr, const int *__restrict__ tco, int V, int nt, R pbc,
               int doG, R G, DsOrder ord, const typename CT<R>::t *__restrict__ p0, R shift,
               double *__restrict__ partial, const int *__restrict__ skip) {
  typedef typename CT<R>::t C;
  if (skip != nullptr && *skip) return;
  // The partial matrices meet in LDS, ROUNDS times NR elements of them, and
  // the determinant sums beside them
  constexpr int ROUNDS = sizeof(R) == 8 ? 1 : 2, NR = (NN + ROUNDS - 1) / ROUNDS;
  __shared__ C part[DS_PARTS][NR][64], dsum[DS_PARTS][64];
  const int L = blockIdx.x, lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int q = L >> 3, comp = q % NTF, qq = q / NTF;
  int s;   // (a lane without a site computes site 0 again and stores nothing)
  const bool live = ord_site64(ord, L & 7, qq, lane, V, &s);

  const uint32_t cs = sizeof(C);
  const uint32_t pl = (uint32_t)V * cs;     // one element plane
  const uint32_t Mb = NN * pl;              // one matrix field
  const Rsrc rS = make_rsrc(src, NTF * Mb), rU = make_rsrc(U, NUMLINK * Mb);
  const Rsrc rN = make_rsrc(nbr, (uint32_t)NGATHER * V * 4u);
  const Rsrc rA = make_rsrc(aux, 6 * pl), rP = make_rsrc(pdet, NUMLINK * NUMLINK * pl);
  const Rsrc rI = make_rsrc(Uinv, NUMLINK * Mb);
  auto nb = [&](int g) { return bload_i32(rN, (uint32_t)s * 4u, (uint32_t)g * V * 4u); };
  auto S = [&](int k, int x) { return Opnd{rS, (uint32_t)x * cs, (uint32_t)k * Mb}; };
  auto Ul = [&](int a, int x) { return Opnd{rU, (uint32_t)x * cs, (uint32_t)a * Mb}; };
  auto num = [&](Rsrc r, int x, int k) { return bload<C>(r, (uint32_t)x * cs, k * pl); };
  auto madd = [](C &sum, C a, C b, R f) {
    sum.x += f * (a.x * b.x - a.y * b.y);
    sum.y += f * (a.x * b.y + a.y * b.x);
  };

  // The pre-pass values Tr eta and Tr(U_c^-1 psi_c) at site x: read, or made
  // here where the caller gives none, which costs the site component's waves
  // ten more matrices but saves a launch
  auto tr_eta = [&](int x) {
    if (!INL) return num(rA, x, 0);
    C v = mkc<C>(0, 0);
#pragma unroll
    for (int i = 0; i < NCOL; i++) {
      const C e = num(rS, x, i * NCOL + i);
      v.x += e.x;
      v.y += DAG ? -e.y : e.y;
    }
    return v;
  };
  auto tr_psi = [&](int c, int x) {
    if (!INL) return num(rA, x, 1 + c);
    C v = mkc<C>(0, 0);
#pragma unroll
    for (int i = 0; i < NCOL; i++)
#pragma unroll
      for (int k = 0; k < NCOL; k++) {
        C e = num(rS, x, (1 + c) * NN + (DAG ? i * NCOL + k : k * NCOL + i));
        if (DAG) e.y = -e.y;
        madd(v, num(rI, x, c * NN + i * NCOL + k), e, (R)1);
      }
    return v;
  };

  C acc[NCOL][NCOL], sum = mkc<C>(0, 0);
#pragma unroll
  for (int i = 0; i < NCOL; i++)
#pragma unroll
    for (int k = 0; k < NCOL; k++) acc[i][k] = mkc<C>(0, 0);
  const int t = tco[s];
  if (comp == 0) {
    const int a = w, xm = nb(g_bwd(a));
    const int xf = doG ? nb(g_fwd(a)) : s;
    mmacc<R, DAG, true>(acc, (R)0.5, S(1 + a, s), Ul(a, s), pl);
    mmacc<R, true, DAG>(acc, (R)-0.5 * bcsign<R>(t, -link_tau(a), nt, pbc), Ul(a, xm),
                        S(1 + a, xm), pl);
    if (doG) {
      // sum_{c != a} plaqdet_ca(x) [T_a(x) + bc(a) T_c(x+a)]
      const C ta = tr_psi(a, s);
      const R sg = bcsign<R>(t, link_tau(a), nt, pbc);
#pragma unroll
      for (int n = 0; n < NUMLINK - 1; n++) {
        const int c = n + (n >= a);
        const C tc = tr_psi(c, xf);
        madd(sum, num(rP, s, c * NUMLINK + a), mkc<C>(ta.x + sg * tc.x, ta.y + sg * tc.y), (R)1);
      }
    }
  } else if (comp <= NUMLINK) {
    const int b = comp - 1, xb = nb(g_fwd(b));
    if (w < NUMLINK - 1) {
      const int a = w + (w >= b), xm = nb(g_bwd(a)), pc = 6 + plaq_idx(a, b);
      const R sg = a < b ? (R)1 : (R)-1;   // chi_ab = sg * stored chi_{min,max}
      const R bc = bcsign<R>(t, -link_tau(a), nt, pbc);
      mmacc<R, false, DAG>(acc, sg, Ul(a, xb), S(pc, s), pl);
      mmacc<R, DAG, false>(acc, -sg * bc, S(pc, xm), Ul(a, xm), pl);
      if (doG) {
        // Tr eta(x) plaqdet_ab(x) + bc(-a) Tr eta(x-a) plaqdet_ba(x-a)
        madd(sum, tr_eta(s), num(rP, s, a * NUMLINK + b), (R)1);
        madd(sum, tr_eta(xm), num(rP, xm, b * NUMLINK + a), bc);
      }
    } else {
      mmacc<R, DAG, true>(acc, (R)0.5 * bcsign<R>(t, link_tau(b), nt, pbc), S(0, xb), Ul(b, s),
                          pl);
      mmacc<R, true, DAG>(acc, (R)-0.5, Ul(b, s), S(0, s), pl);
    }
  } else {
    const int p = comp - 1 - NUMLINK;
    if (w < 2) {
      // +-[bc(a) U_a(x) psi_b(x+a) + psi_a(x) U_b(x+a)], - with a, b exchanged
      const int a = w ? c_pt.b[p] : c_pt.a[p], b = w ? c_pt.a[p] : c_pt.b[p];
      const int xa = nb(g_fwd(a));
      const R sg = w ? (R)-1 : (R)1;
      mmacc<R, false, DAG>(acc, sg * bcsign<R>(t, link_tau(a), nt, pbc), Ul(a, s),
                           S(1 + b, xa), pl);
      mmacc<R, DAG, false>(acc, sg, S(1 + a, s), Ul(b, xa), pl);
    } else {
      // PtoP at double weight (see k_dslash)
      const int n = w - 2, c = c_pt.pp_c[p][n], pc = 6 + c_pt.pp_de[p][n];
      const int x1 = nb(c_pt.pp_g1[p][n]), x2 = nb(c_pt.pp_g2[p][n]), xmc = nb(g_bwd(c));
      const R tr = (R)(2.0f * c_pt.pp_tr[p][n]);
      mmacc<R, DAG, true>(acc, tr * bcsign<R>(t, c_pt.pp_dt3[p][n], nt, pbc), S(pc, x2),
                          Ul(c, x1), pl);
      mmacc<R, true, DAG>(acc, -tr * bcsign<R>(t, c_pt.pp_dt2[p][n], nt, pbc), Ul(c, xmc),
                          S(pc, x1), pl);
    }
  }
  // ---- the waves share the elements of the sum: of each round's, wave w
  // takes w, w + 5, ...
  constexpr int NE = (NR + DS_PARTS - 1) / DS_PARTS;
  const bool det = doG && comp <= NUMLINK;
  const bool pre = !DAG && EPI == 0 && aux_out != nullptr && comp <= NUMLINK;
  C pq[ROUNDS][NE], u[ROUNDS][NE];
#pragma unroll
  for (int r = 0; r < ROUNDS; r++)
#pragma unroll
    for (int j = 0; j < NE; j++) {
      const int e = min(r * NR + min(w + j * DS_PARTS, NR - 1), NN - 1);
      pq[r][j] = u[r][j] = mkc<C>(0, 0);
      if (EPI == 1)
        pq[r][j] = bload<C>(make_rsrc(p0, NTF * Mb), (uint32_t)s * cs,
                            comp * Mb + (DAG ? (e % NCOL) * NCOL + e / NCOL : e) * pl);
      // element e of U^-1 as the accumulator holds it
      if ((det || pre) && comp > 0)
        u[r][j] = bload<C>(rI, (uint32_t)s * cs, (comp - 1) * Mb + e * pl);
    }
  dsum[w][lane] = sum;
  double dot = 0;
  C tr = mkc<C>(0, 0);
  const Rsrc rD = make_rsrc(dst, NTF * Mb);
#pragma unroll
  for (int r = 0; r < ROUNDS; r++) {
    if (r) __syncthreads();   // the last round's elements have been read
#pragma unroll
    for (int e = 0; e < NR; e++)
      if (r * NR + e < NN) part[w][e][lane] = acc[(r * NR + e) / NCOL][(r * NR + e) % NCOL];
    __syncthreads();
    if (r == 0 && det) {
      sum = mkc<C>(0, 0);
#pragma unroll
      for (int i = 0; i < DS_PARTS; i++) {
        const C v = dsum[i][lane];
        sum.x += v.x;
        sum.y += v.y;
      }
      const R f = (R)(comp == 0 ? 0.5 * C2 : -0.5 * C2) * G;
      sum.x *= f;
      sum.y *= f;
    }
#pragma unroll
    for (int j = 0; j < NE; j++) {
      const int er = w + j * DS_PARTS, e = r * NR + er;
      if (er >= NR || e >= NN) continue;
      C v = mkc<C>(0, 0);
#pragma unroll
      for (int i = 0; i < DS_PARTS; i++) {
        const C x = part[i][er][lane];
        v.x += x.x;
        v.y += x.y;
      }
      const bool diag = e / NCOL == e % NCOL;
      const C ue = u[r][j];
      if (det) {
        if (comp > 0) {
          v.x += sum.x * ue.x - sum.y * ue.y;
          v.y += sum.x * ue.y + sum.y * ue.x;
        } else if (diag) {
          v.x += sum.x;
          v.y += sum.y;
        }
      }
      if (pre) {
        // Tr(out_0)^*, or Tr(U^-1 out^dagger)
        if (comp > 0) {
          tr.x += ue.x * v.x + ue.y * v.y;
          tr.y += ue.y * v.x - ue.x * v.y;
        } else if (diag) {
          tr.x += v.x;
          tr.y -= v.y;
        }
      }
      // D^dagger: element (i,k) of the accumulator is minus the conjugate of
      // element (k,i) of the result
      const int d = DAG ? (e % NCOL) * NCOL + e / NCOL : e;
      if (DAG) v.x = -v.x;
      if (EPI == 1) {
        const C x = pq[r][j];
        v.x = fma(shift, x.x, v.x);
        v.y = fma(shift, x.y, v.y);
        dot += (double)x.x * (double)v.x + (double)x.y * (double)v.y;
      }
      if (live) {
        bstore<DS_STORE_L2>(v, rD, (uint32_t)s * cs, comp * Mb + d * pl);
        hold(v);
      }
    }
  }
  if (pre) {
    __syncthreads();   // the determinant sums have been read
    dsum[w][lane] = tr;
    __syncthreads();
    if (w == 0 && live) {
      tr = mkc<C>(0, 0);
#pragma unroll
      for (int i = 0; i < DS_PARTS; i++) {
        const C v = dsum[i][lane];
        tr.x += v.x;
        tr.y += v.y;
      }
      st_keep(aux_out + (size_t)comp * V + s, tr);
    }
  }
  if (EPI == 1) {
    if (!live) dot = 0;
    for (int off = 32; off > 0; off >>= 1) dot += __shfl_xor(dot, off, 64);
    __shared__ double red[DS_PARTS];
    if (lane == 0) red[w] = dot;
    __syncthreads();
    if (threadIdx.x == 0) {
      double tsum = 0;
      for (int i = 0; i < DS_PARTS; i++) tsum += red[i];
      partial[L] = tsum;
      hold(tsum);
    }
  }
}

// The lattices k_dslash_split is for.  It reads each operand about half as
// often beyond L2 as k_dslash, but keeps fewer loads in flight per wave, so
// k_dslash wins where a launch fills the chip.  Both sides, us of a CG
// iteration, which leaves less of the operands in the caches than an operator
// that is repeated alone, k_dslash | k_dslash_split:
//   U(4) FP64  2160: 74.5 | 64.3    4096: 92.1 | 88.0    8192: 154 | 165
//        FP32  2160: 55.7 | 49.4    3072: 56.8 | 50.8    4096: 63.6 | 64.1
//   U(3) FP64  2160: 46.5 | 44.7    3072: 49.6 | 47.4    4096: 55.1 | 58.6
//        FP32  4096: 43.3 | 40.6    8192: 63.8 | 63.1   16384: 111 | 108
//             32768: 209 | 199     49152: 303 | 299     65536: 404 | 418
//   U(2) FP64  4096: 32.0 | 31.5    6144: 40.9 | 40.0    8192: 48.3 | 49.1
//              9216: 54.2 | 52.6   16384: 82.8 | 80.6   32768: 156 | 148
//             49152: 229 | 231     65536: 294 | 322
//        FP32  2048: 26.0 | 24.2    3072: 28.3 | 27.5    3584: 29.9 | 30.6
//              4096: 29.3 | 31.0    5120: 33.5 | 34.5    6144: 35.2 | 35.9
//              6912: 39.1 | 38.3    8192: 41.5 | 42.3    9216: 45.4 | 44.6
//             16384: 64.7 | 64.1   32768: 111 | 110     65536: 191 | 192
// U(2) FP32 gives the sizes between 3072 and 6144 back to k_dslash; 2% at 6144
// and 8192 (and at 8192 in FP64) are left to this kernel, which is the faster
// one at 6912 and from 9216 on, and alone at 6144 (10.7 us of 11.2).  Between the
// sizes measured on both sides of an upper limit up to 4% are left to k_dslash
// (U(2) 12^3x24 FP64 198 | 192, FP32 136 | 131; U(4) 8^3x12 FP64 124 | 121).
template <typename R>
static bool ds_split(int V) {
  const bool dbl = sizeof(R) == sizeof(double);
  if (NCOL == 2 && !dbl && V > 3072 && V < 6144) return false;
  return V <= (NCOL == 2 || (NCOL == 3 && !dbl) ? 32768 : NCOL == 4 && dbl ? 4096 : 3072);
}

// Where it also makes the pre-pass values itself instead of a launch of their
// own (us of an operator, launch | inside, FP64, FP32): U(2) 256 sites 6.3 | 4.7,
// 6.1 | 4.8; 1296 7.8 | 7.6, 7.3 | 7.1; 2160 9.0 | 8.1, 8.1 | 9.3; 4096 10.3 | 10.7,
// 9.1 | 11.1.  With the larger matrices the ten more products cost more than
// the launch (U(3) 4^4 7.9 | 10.0, U(4) 4^3x8 10.2 | 12.3).
static constexpr bool ds_split_inline(int V) { return NCOL == 2 && V <= 1296; }
#endif  // NCOL <= 4

template <typename R>
static int dslash_launch(susy_ctx *c, const typename CT<R>::t *src,
                         typename CT<R>::t *dst, int sign, const typename CT<R>::t *p0,
                         R shift, double *partial, int *nblocks,
                         const typename CT<R>::t *U, const typename CT<R>::t *Uinv,
                         const typename CT<R>::t *pdet, typename CT<R>::t *aux,
                         const int *skip, typename CT<R>::t *aux_out = nullptr,
                         bool prep = true, bool sampled = true, bool keep_prep = false) {
  if (sign != 1 && sign != -1) {
    set_error("fermion_op: incorrect sign %d", sign);
    return SUSY_E_ARG;
  }
  const int V = c->V;
  if ((size_t)NTF * NN * V * sizeof(typename CT<R>::t) > 0x7fffffffu) {
    set_error("lattice too large for 32-bit buffer offsets (V=%d)", V);
    return SUSY_E_ARG;
  }
  if (sign != 1 || p0 != nullptr || !c->doG) aux_out = nullptr;
#if NCOL <= 4
  const bool split = ds_split<R>(V);
  // (an epilogue's launch has its pre-pass values from D)
  const bool inl = split && c->doG && prep && !keep_prep && p0 == nullptr && ds_split_inline(V);
#else
  const bool split = false, inl = false;
#endif
  if (c->doG && prep && !inl) {
    const int nbp = (V + 255) / 256;
#define PREP_GO(KERNEL, GRID)                                                          \
  do {                                                                                 \
    if (sign == 1)                                                                     \
      hipLaunchKernelGGL((KERNEL<R, false>), GRID, dim3(256), 0, c->s, src, Uinv, aux, \
                         V, skip);                                                     \
    else                                                                               \
      hipLaunchKernelGGL((KERNEL<R, true>), GRID, dim3(256), 0, c->s, src, Uinv, aux,  \
                         V, skip);                                                     \
  } while (0)
    if (V <= PREP_TRACE_V) PREP_GO(k_dslash_prep_trace, dim3(nbp, 1 + NUMLINK));
    else PREP_GO(k_dslash_prep, dim3(nbp));
#undef PREP_GO
    HIPCHK(hipGetLastError());
  }
  DsOrder ord;
  const int sites = split ? 64 : ds_sites(V, DsSites<R>::n);
  const int threads = split ? 64 * DS_PARTS : sites;
  const int nb = ds_grid(V, c->p.nx * c->p.ny * c->p.nz,
                         sizeof(R) == sizeof(float) ? c->site_order32 : c->site_order,
                         sites, &ord);
  if (nblocks) *nblocks = nb;
  R pbc = (R)c->p.PBC, G = (R)c->p.G;
#define DS_ARGS src, dst, U, Uinv, pdet, aux, aux_out, c->d_nbr, c->d_t, V, c->p.nt, pbc, \
                c->doG, G, ord, p0, shift, partial, skip
  // sampled timing covers the plain operator D (sign +1, no epilogue) only
  const int pi = sizeof(R) == sizeof(float) ? 1 : 0;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (sampled && c->prof_every > 0 && sign == 1 && p0 == nullptr &&
      (c->prof_launch[pi]++ % c->prof_every) == 0) {
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    HIPCHK(hipEventRecord(e0, c->s));
  }
  const unsigned lds = sizeof(R) == sizeof(double) ? DS_OCC_LDS64 : DS_OCC_LDS32;
#if NCOL <= 4
#define DS_GO(DAG, EPI)                                                                       \
  do {                                                                                        \
    if (inl)                                                                                  \
      hipLaunchKernelGGL((k_dslash_split<R, DAG, EPI, NCOL == 2 && EPI == 0>), dim3(nb),      \
                         dim3(threads), 0, c->s, DS_ARGS);                                    \
    else if (split)                                                                           \
      hipLaunchKernelGGL((k_dslash_split<R, DAG, EPI, false>), dim3(nb), dim3(threads), 0,    \
                         c->s, DS_ARGS);                                                      \
    else                                                                                      \
      hipLaunchKernelGGL((k_dslash<R, DAG, EPI>), dim3(nb), dim3(threads), lds, c->s, DS_ARGS); \
  } while (0)
#else
#define DS_GO(DAG, EPI) \
  hipLaunchKernelGGL((k_dslash<R, DAG, EPI>), dim3(nb), dim3(threads), lds, c->s, DS_ARGS)
#endif
  if (p0 == nullptr) {
    if (sign == 1) DS_GO(false, 0);
    else DS_GO(true, 0);
  } else {
    if (sign == 1) DS_GO(false, 1);
    else DS_GO(true, 1);
  }
#undef DS_GO
#undef DS_ARGS
  HIPCHK(hipGetLastError());
  if (e0) {
    HIPCHK(hipEventRecord(e1, c->s));
    c->prof_ev[pi].push_back(e0);
    c->prof_ev[pi].push_back(e1);
  }
  return 0;
}

// Sampled timing of the operator kernel on the context's stream: every
// prof_every-th launch of D (sign +1, no epilogue) is bracketed by events.
// prof_every = 0 switches sampling off.
extern "C" int susy_prof_enable(susy_ctx *c, int every) {
  if (!c || every < 0) return SUSY_E_ARG;
  HIPCHK(hipStreamSynchronize(c->s));
  for (int p = 0; p < 2; p++) {
    for (hipEvent_t e : c->prof_ev[p]) (void)hipEventDestroy(e);
    c->prof_ev[p].clear();
    c->prof_launch[p] = 0;
  }
  c->prof_every = every;
  return 0;
}
// Average duration (ms) of the sampled launches and the count of D launches,
// for FP64 (prec 0) or FP32 (prec 1) operator kernels.
extern "C" int susy_prof_read(susy_ctx *c, int prec, double *avg_ms, long *launches,
                              long *sampled) {
  if (!c || prec < 0 || prec > 1) return SUSY_E_ARG;
  HIPCHK(hipStreamSynchronize(c->s));
  double tot = 0;
  size_t n = c->prof_ev[prec].size() / 2;
  for (size_t k = 0; k < n; k++) {
    float ms = 0;
    HIPCHK(hipEventElapsedTime(&ms, c->prof_ev[prec][2 * k], c->prof_ev[prec][2 * k + 1]));
    tot += ms;
  }
  *avg_ms = n ? tot / n : 0.0;
  *launches = c->prof_launch[prec];
  *sampled = (long)n;
  return 0;
}

int dslash64(susy_ctx *c, const double2 *src, double2 *dst, int sign,
             const double2 *p0, double shift, double *partial, int *nblocks, const int *skip) {
  return dslash_launch<double>(c, src, dst, sign, p0, shift, partial, nblocks,
                               c->d_links, c->d_uinv, c->d_pdet, c->d_aux, skip);
}
// dst = D src; with G terms also the traces Tr src_0, Tr(U_a^-1 src_{1+a}) in
// d_aux and Tr(dst_0)^*, Tr(U_a^-1 dst_{1+a}^dag) in d_aux2 (6 planes each)
int dslash64_traces(susy_ctx *c, const double2 *src, double2 *dst) {
  return dslash_launch<double>(c, src, dst, 1, nullptr, 0.0, nullptr, nullptr, c->d_links,
                               c->d_uinv, c->d_pdet, c->d_aux, nullptr, c->d_aux2, true, true,
                               true);
}
int dslash32(susy_ctx *c, const float2 *src, float2 *dst, int sign,
             const float2 *p0, float shift, double *partial, int *nblocks, const int *skip) {
  if (!c->f_fresh) {
    int r = fields_refresh32(c);
    if (r) return r;
  }
  return dslash_launch<float>(c, src, dst, sign, p0, shift, partial, nblocks,
                              c->f_links, c->f_uinv, c->f_pdet, c->f_aux, skip);
}

// dst = D^dagger D src + shift src, tmp = D src, per-block partials of
// Re <src, dst> in partial (the DSq of utilities.c:874-885 with the CG's
// shift).  D stores the D^dagger pre-pass values of its output (aux2), so
// D^dagger runs without its pre-pass.  prep_src = false: the caller has
// already stored the pre-pass values of src in the context's aux buffer.
int dsq_pair64(susy_ctx *c, const double2 *src, double2 *tmp, double2 *dst, double shift,
               double *partial, int *nblocks, const int *skip, bool prep_src) {
  int r = dslash_launch<double>(c, src, tmp, 1, nullptr, 0.0, nullptr, nullptr, c->d_links,
                                c->d_uinv, c->d_pdet, c->d_aux, skip, c->d_aux2, prep_src);
  if (r) return r;
  return dslash_launch<double>(c, tmp, dst, -1, src, shift, partial, nblocks, c->d_links,
                               c->d_uinv, c->d_pdet, c->d_aux2, skip, nullptr, false);
}
int dsq_pair32(susy_ctx *c, const float2 *src, float2 *tmp, float2 *dst, float shift,
               double *partial, int *nblocks, const int *skip, bool prep_src) {
  if (!c->f_fresh) {
    int r = fields_refresh32(c);
    if (r) return r;
  }
  int r = dslash_launch<float>(c, src, tmp, 1, nullptr, 0.f, nullptr, nullptr, c->f_links,
                               c->f_uinv, c->f_pdet, c->f_aux, skip, c->f_aux2, prep_src);
  if (r) return r;
  return dslash_launch<float>(c, tmp, dst, -1, src, shift, partial, nblocks, c->f_links,
                              c->f_uinv, c->f_pdet, c->f_aux2, skip, nullptr, false);
}

// ---------------------------------------------------------------------
// Operator without allocation (susy_fermion_op_noalloc).  Its only scratch
// memory -- the G-term pre-pass values, 6 complex numbers per site -- lives
// in this fixed device array instead of the context's buffer.  Every device
// the library runs on holds one copy until the process ends.  The pre-pass
// writes every value the operator then reads, so nothing in it needs
// clearing between calls; calls that overlap on one device race on it.
#define NOALLOC_SCRATCH_BYTES (16u << 20)
#define NOALLOC_MAX_DEVICES 64
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];
// device address of `scratch` on each device (the name itself is only a
// host-side handle of the symbol)
static void *g_scratch_dev[NOALLOC_MAX_DEVICES];
static std::mutex g_scratch_mu;

// Called by susy_create with the context's device current: looks up that
// device's copy of the array once.
int noalloc_init_device(susy_ctx *c) {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) {
    set_error("device %d beyond the %d the library tracks", dev, NOALLOC_MAX_DEVICES);
    return SUSY_E_STATE;
  }
  c->dev = dev;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void *p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      set_error("hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
      return SUSY_E_HIP;
    }
    g_scratch_dev[dev] = p;
  }
  return 0;
}

extern "C" int susy_fermion_op_noalloc(susy_ctx *c, const double *src, double *dst, int sign) {
  if (!c) return SUSY_E_STATE;
  if (!src || !dst) {
    set_error("susy_fermion_op_noalloc: null field pointer");
    return SUSY_E_ARG;
  }
  if (sign != 1 && sign != -1) {
    set_error("susy_fermion_op_noalloc: incorrect sign %d", sign);
    return SUSY_E_ARG;
  }
  const size_t need = (size_t)6 * c->V * sizeof(double2);
  if (need > NOALLOC_SCRATCH_BYTES) {
    set_error("susy_fermion_op_noalloc: %d sites need %zu bytes of scratch; the fixed "
              "array holds %u (at most %u sites)", c->V, need, NOALLOC_SCRATCH_BYTES,
              (unsigned)(NOALLOC_SCRATCH_BYTES / (6 * sizeof(double2))));
    return SUSY_E_ARG;
  }
  void *aux = g_scratch_dev[c->dev];
  if (!aux) {
    set_error("susy_fermion_op_noalloc: scratch of device %d not set up", c->dev);
    return SUSY_E_STATE;
  }
  int r = dslash_launch<double>(c, (const double2 *)src, (double2 *)dst, sign, nullptr, 0.0,
                                nullptr, nullptr, c->d_links, c->d_uinv, c->d_pdet,
                                (double2 *)aux, nullptr, nullptr, true, false);
  if (r) return r;
  HIPCHK(hipStreamSynchronize(c->s));
  return 0;
}
