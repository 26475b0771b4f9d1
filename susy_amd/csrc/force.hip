// Fermion force (reference: 4d_Q16/susy/update_h.c:272-978).
//
// For each pole n, with sol = psi_n and psol = D psi_n, the force matrix on
// link (x, mu) is assembled by the block that owns (x, mu) from
//   SV    (update_h.c:709-746)   site/link terms
//   VP    (update_h.c:756-894)   link/plaquette terms
//   detF  (update_h.c:477-651)   plaquette-determinant terms (G > 0), both
//                                orientations (update_h.c:899-905)
//   F1Q, F2Q (update_h.c:272-462) Q-closed terms landing on link mu
// and accumulated as F += amp_n f^dag (update_h.c:943-958).  Every term is
// linear in psol, so psol is used unscaled and amp_n scales the sum.
// Finally mom -= eps F (update_h.c:965-969).
#include "dev_buf.h"
#include "dev_mat.h"

__constant__ ForceTerms c_ft;

int force_init_tables(const ForceTerms &ft) {
  HIPCHK(hipMemcpyToSymbol(HIP_SYMBOL(c_ft), &ft, sizeof(ForceTerms)));
  return 0;
}

__device__ __forceinline__ double bcs(int t, int dt, int nt, double pbc) {
  int tt = t + dt;
  return (tt < 0 || tt > nt - 1) ? pbc : 1.0;
}

// F[mu](x) (+)= amp * f_U[mu](x)^dag for one pole.  X accumulates
// f_U[mu](x)^dagger: a term A B of f_U enters as B^dag A^dag.
//
// A block makes one link direction of 64 sites: its four waves share the terms
// (wave w: VP and the determinant sums of the w-th nu != mu, one SV product,
// the Q-closed terms w and w + 4), their sums meet in LDS, and then each wave
// makes a column of X.  One thread per link went through its 32 products and
// the determinant's gathered scalars one after the other, which was all its
// time on small lattices.  On large ones it waits for gathered lines, half of
// which the XCD's L2 misses (U(4) 16^4: 46% hits, 66 lines in flight per CU at
// 465 cycles each, waves waiting 72% of their time): the blocks take the
// operator kernel's order of site chunks, so the neighbourhoods shared by the
// directions and by the next chunks meet in one XCD's L2.  A force with one
// pole (D, this and the update), us: U(4) 4^3x8 166 -> 63, 8^3x16 238 -> 164,
// 16^4 1472 -> 1085; U(3) 4^4 106 -> 48, 16^4 761 -> 603; U(2) 4^4 57 -> 36,
// 16^4 330 -> 233.  Five waves with SV on its own leave three of eight wave
// slots empty (16^4: 1308 at U(4)), one wave a link spills or takes 256
// registers (2355).
// auxS, auxP: Tr sol_site, Tr(U_a^-1 sol_a); Tr psol_site^dag,
// Tr(U_a^-1 psol_a^dag).
// (waves per SIMD: what the registers of two operands and X allow without
// scratch)
#define FR_EU (NCOL >= 5 ? 1 : NCOL == 2 ? 3 : 2)
#define FR_PARTS (NUMLINK - 1)
__global__ void __launch_bounds__(64 * FR_PARTS) __attribute__((amdgpu_waves_per_eu(FR_EU)))
k_force_assemble(const double2 *__restrict__ S, const double2 *__restrict__ P,
                 const double2 *__restrict__ uinv, const double2 *__restrict__ pd,
                 const double2 *__restrict__ auxS, const double2 *__restrict__ auxP,
                 const int *__restrict__ nbr, const int *__restrict__ tco,
                 double2 *__restrict__ F, int V, int nt, double pbc, int doG, double G,
                 double amp, int first, DsOrder ord) {
  constexpr int NH = (NCOL + 1) / 2;   // rows of X in one round of the exchange
  __shared__ double2 part[FR_PARTS][NH * NCOL][64], dets[FR_PARTS][3][64];
  const int L = blockIdx.x, lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int mu = (L >> 3) % NUMLINK;
  int s;   // (a lane without a site computes site 0 and stores nothing)
  const bool live = ord_site64(ord, L & 7, (L >> 3) / NUMLINK, lane, V, &s);
  const uint32_t cs = sizeof(double2), pl = (uint32_t)V * cs, Mb = NN * pl;
  const Rsrc rS = make_rsrc(S, NTF * Mb), rP = make_rsrc(P, NTF * Mb);
  const Rsrc rI = make_rsrc(uinv, NUMLINK * Mb), rF = make_rsrc(F, NUMLINK * Mb);
  auto Sx = [&](int k, int x) { return Opnd{rS, (uint32_t)x * cs, (uint32_t)k * Mb}; };
  auto Px = [&](int k, int x) { return Opnd{rP, (uint32_t)x * cs, (uint32_t)k * Mb}; };
  const int t = tco[s];
  const int xm = nbr[g_fwd(mu) * V + s];
  const double bm = bcs(t, link_tau(mu), nt, pbc);
  Mat X;
  mzero(X);
  double2 z = make_double2(0, 0), w1 = make_double2(0, 0), w2 = make_double2(0, 0);
  {
    // ---- VP: f_U += -bc s_psi_nu(x+mu) p_chi(x) + p_chi(x-nu) s_psi_nu(x-nu)
    //                 + bc p_psi_nu(x+mu) s_chi(x) - s_chi(x-nu) p_psi_nu(x-nu)
    // chi = chi_{mu nu} = sg * stored, p_chi = psol chi^dag, p_psi = psol psi^dag
    const int nu = w + (w >= mu), xn = nbr[g_bwd(nu) * V + s], pc = 6 + plaq_idx(mu, nu);
    const double sg = mu < nu ? 1.0 : -1.0;
    mmacc<double, false, true>(X, -bm * sg, Px(pc, s), Sx(1 + nu, xm), pl);
    mmacc<double, true, false>(X, sg, Sx(1 + nu, xn), Px(pc, xn), pl);
    mmacc<double, true, false>(X, bm * sg, Sx(pc, s), Px(1 + nu, xm), pl);
    mmacc<double, false, true>(X, -sg, Px(1 + nu, xn), Sx(pc, xn), pl);
    // (else the products sink below the determinant's branch, with all their
    // operands in registers)
#pragma unroll
    for (int i = 0; i < NCOL; i++)
#pragma unroll
      for (int j = 0; j < NCOL; j++) asm volatile("" : "+v"(X[i][j].x), "+v"(X[i][j].y));
    if (doG) {
      // determinant terms: X^dag += z U^-1 - U^-1 W U^-1, i.e.
      // X += conj(z) U^-dag - (U^-1 W U^-1)^dag.  call 0: eta = psol_site^dag,
      // psi = sol links; call 1: eta = sol_site, psi = psol links^dag
      const int a = mu, b = nu;
      const int xb = nbr[g_fwd(b) * V + s], xamb = nbr[g_bwd(b) * V + xm];   // x + e_a - e_b
      const int tmb = tco[xn];
      const double2 dba = pd[(b * NUMLINK + a) * V + s], dab = pd[(a * NUMLINK + b) * V + s];
      const double2 dab_m = pd[(a * NUMLINK + b) * V + xn],
                    dba_m = pd[(b * NUMLINK + a) * V + xn];
      const double sa = bcs(t, link_tau(a), nt, pbc), smb = bcs(t, -link_tau(b), nt, pbc);
      const double sb = bcs(t, link_tau(b), nt, pbc), sam = bcs(tmb, link_tau(a), nt, pbc);
#pragma unroll
      for (int call = 0; call < 2; call++) {
        const double2 *te = call == 0 ? auxP : auxS, *T = (call == 0 ? auxS : auxP) + V;
        const double lg = call == 0 ? -0.5 * C2 * G : 0.5 * C2 * G;
        const double2 Ta = T[a * V + s], Tb = T[b * V + s], Tb_xa = T[b * V + xm];
        const double2 Tb_m = T[b * V + xn], Ta_xb = T[a * V + xb], Ta_m = T[a * V + xn];
        const double2 Tb_amb = T[b * V + xamb], e = te[s], em = te[xn];
        const double2 Dba = cmul(e, dba), Dab = cmul(e, dab), Dab_m = cmul(em, dab_m),
                      Dba_m = cmul(em, dba_m);
        const double2 p1 = cmul(Dba, make_double2(Ta.x + sa * Tb_xa.x, Ta.y + sa * Tb_xa.y));
        const double2 p2 = cmul(Dab_m, make_double2(Tb_m.x + smb * Ta.x, Tb_m.y + smb * Ta.y));
        const double2 a1 = cmul(Dab, make_double2(Tb.x + sb * Ta_xb.x, Tb.y + sb * Ta_xb.y));
        const double2 a2 =
            cmul(Dba_m, make_double2(Ta_m.x + sam * Tb_amb.x, Ta_m.y + sam * Tb_amb.y));
        // f_U += (lg plaq) U^-1 + conj(lg adj) U^-1 - (lg inv) U^-1 psi U^-1
        z.x += lg * (p1.x + p2.x) + lg * (a1.x + a2.x);
        z.y += lg * (p1.y + p2.y) - lg * (a1.y + a2.y);
        double2 &wc = call == 0 ? w1 : w2;
        wc.x += lg * (Dba.x + smb * Dab_m.x);
        wc.y += lg * (Dba.y + smb * Dab_m.y);
      }
    }
  }
  // ---- SV: f_U += 1/2 u^dag, so X += 1/2 u with
  // u = bc s_psi(x) p_eta(x+mu) - p_eta(x) s_psi(x) - bc p_psi(x) s_eta(x+mu)
  //     + s_eta(x) p_psi(x),   p_eta = psol_site^dag, p_psi = psol_link^dag
  if (w == 0) mmacc<double, false, true>(X, 0.5 * bm, Sx(1 + mu, s), Px(0, xm), pl);
  else if (w == 1) mmacc<double, true, false>(X, -0.5, Px(0, s), Sx(1 + mu, s), pl);
  else if (w == 2) mmacc<double, true, false>(X, -0.5 * bm, Px(1 + mu, s), Sx(0, xm), pl);
  else mmacc<double, false, true>(X, 0.5, Sx(0, s), Px(1 + mu, s), pl);
  // ---- Q-closed F1Q / F2Q on link c = mu: f_U += -1/2 T^dag, X += -1/2 T.
  // The F2Q term of (a,b,d,e) equals the F1Q term of (d,e,a,b): x-a-b =
  // x+c+d+e, perm(a,b,c,d,e) = perm(d,e,c,a,b) and the two temporal offsets
  // trade places, so the F1Q terms are applied at double weight (checked
  // term by term when the tables are built).
#pragma unroll 1
  for (int n = w; n < 6; n += FR_PARTS) {
    const int ab = 6 + c_ft.ab[mu][n], de = 6 + c_ft.de[mu][n];
    const int xabc = nbr[c_ft.g_abc[mu][n] * V + s];
    const int xmab = nbr[c_ft.g_mab[mu][n] * V + s];
    const double b3 = bcs(t, c_ft.dt3[mu][n], nt, pbc) * bm;
    const double b2 = bcs(t, c_ft.dt2m[mu][n], nt, pbc) * bm;
    const double p1 = c_ft.perm1[mu][n];
    // F1Q: T = p1 b3 Pde^dag(x+a+b+c) Sab(x+c) - p1 b2 Sab(x-a-b) Pde^dag(x+c)
    mmacc<double, true, false>(X, -p1 * b3, Px(de, xabc), Sx(ab, xm), pl);
    mmacc<double, false, true>(X, p1 * b2, Sx(ab, xmab), Px(de, xm), pl);
  }
  // ---- column i of X: F[j][i] (+)= amp (X[j][i] + conj(z u - q)[i][j]) with
  // u = U^-1, q = u W u, W = w1 sol_mu + w2 psol_mu^dag
  auto column = [&](int i, const double2 *x, const Mat Wm) {
    double2 u[NCOL], d[NCOL], f[NCOL];
#pragma unroll
    for (int j = 0; j < NCOL; j++) d[j] = f[j] = make_double2(0, 0);
    if (doG) {
      double2 rr[NCOL];   // row i of u W
#pragma unroll
      for (int l = 0; l < NCOL; l++) {
        u[l] = bload<double2>(rI, (uint32_t)s * cs, mu * Mb + (i * NCOL + l) * pl);
        rr[l] = make_double2(0, 0);
      }
#pragma unroll
      for (int k = 0; k < NCOL; k++)
#pragma unroll
        for (int l = 0; l < NCOL; l++) {
          const double2 v = cmul(u[k], Wm[k][l]);
          rr[l].x += v.x;
          rr[l].y += v.y;
        }
#pragma unroll
      for (int j = 0; j < NCOL; j++) {
        d[j] = cmul(z, u[j]);
#pragma unroll
        for (int l = 0; l < NCOL; l++) {
          const double2 v = cmul(rr[l], bload<double2>(rI, (uint32_t)s * cs,
                                                       mu * Mb + (l * NCOL + j) * pl));
          d[j].x -= v.x;
          d[j].y -= v.y;
        }
      }
    }
    if (!first) {
#pragma unroll
      for (int j = 0; j < NCOL; j++)
        f[j] = bload<double2>(rF, (uint32_t)s * cs, mu * Mb + (j * NCOL + i) * pl);
    }
#pragma unroll
    for (int j = 0; j < NCOL; j++) {
      f[j].x += amp * (x[j].x + d[j].x);
      f[j].y += amp * (x[j].y - d[j].y);
    }
    if (live) {
#pragma unroll
      for (int j = 0; j < NCOL; j++)
        st_keep(F + (size_t)(mu * NN + j * NCOL + i) * V + s, f[j]);
    }
  };
  auto load_W = [&](Mat Wm) {
    const uint32_t o = (1 + mu) * Mb;
#pragma unroll
    for (int i = 0; i < NCOL; i++)
#pragma unroll
      for (int j = 0; j < NCOL; j++) {
        Wm[i][j] = make_double2(0, 0);
        if (!doG) continue;
        const double2 x = bload<double2>(rS, (uint32_t)s * cs, o + (i * NCOL + j) * pl);
        const double2 y = cconjd(bload<double2>(rP, (uint32_t)s * cs, o + (j * NCOL + i) * pl));
        Wm[i][j] = make_double2(w1.x * x.x - w1.y * x.y + w2.x * y.x - w2.y * y.y,
                                w1.x * x.y + w1.y * x.x + w2.x * y.y + w2.y * y.x);
      }
  };
  // ---- the waves meet: rows [0, NH) of X, then the others; wave w takes the
  // columns w, w + 4
  constexpr int NI = (NCOL + FR_PARTS - 1) / FR_PARTS;
  dets[w][0][lane] = z;
  dets[w][1][lane] = w1;
  dets[w][2][lane] = w2;
  double2 x[NI][NCOL];
#pragma unroll
  for (int r = 0; r < 2; r++) {
    if (r) __syncthreads();
#pragma unroll
    for (int j = r * NH; j < min(NCOL, (r + 1) * NH); j++)
#pragma unroll
      for (int i = 0; i < NCOL; i++) part[w][(j - r * NH) * NCOL + i][lane] = X[j][i];
    __syncthreads();
#pragma unroll
    for (int j = r * NH; j < min(NCOL, (r + 1) * NH); j++)
#pragma unroll
      for (int n = 0; n < NI; n++) {
        x[n][j] = make_double2(0, 0);
#pragma unroll
        for (int i = 0; i < FR_PARTS; i++) {
          const double2 v =
              part[i][(j - r * NH) * NCOL + min(w + n * FR_PARTS, NCOL - 1)][lane];
          x[n][j].x += v.x;
          x[n][j].y += v.y;
        }
      }
  }
  if (w >= NCOL) return;
  z = w1 = w2 = make_double2(0, 0);
#pragma unroll
  for (int i = 0; i < FR_PARTS; i++) {
    z.x += dets[i][0][lane].x;
    z.y += dets[i][0][lane].y;
    w1.x += dets[i][1][lane].x;
    w1.y += dets[i][1][lane].y;
    w2.x += dets[i][2][lane].x;
    w2.y += dets[i][2][lane].y;
  }
  Mat Wm;
  load_W(Wm);
#pragma unroll
  for (int n = 0; n < NI; n++)
    if (w + n * FR_PARTS < NCOL) column(w + n * FR_PARTS, x[n], Wm);
}

// mom -= eps F; partial |F|^2
__global__ void __launch_bounds__(FB)
k_force_apply(const double2 *__restrict__ F, double2 *__restrict__ mom, double eps,
              int V, double *__restrict__ partial) {
  int gid = blockIdx.x * blockDim.x + threadIdx.x;
  double nrm = 0;
  if (gid < V * NUMLINK) {
    int mu = gid / V, s = gid - mu * V;
    const size_t M = (size_t)NN * V;
#pragma unroll
    for (int e = 0; e < NN; e++) {
      size_t k = mu * M + (size_t)e * V + s;
      double2 f = F[k], m = mom[k];
      m.x -= eps * f.x;
      m.y -= eps * f.y;
      st_keep(mom + k, m);
      nrm += f.x * f.x + f.y * f.y;
    }
  }
  block_partial(nrm, partial, 0, 0);
}

int fermion_force_dev(susy_ctx *c, double eps, double2 *const *sol, int nsol,
                      const double *amps, double *norm) {
  const int V = c->V;
  double2 *psol = c->d_tmp;
  DsOrder ord;
  const int grid = ds_grid(V, c->p.nx * c->p.ny * c->p.nz, c->site_order, 64, &ord, NUMLINK);
  for (int n = 0; n < nsol; n++) {
    int r = dslash64_traces(c, sol[n], psol);
    if (r) return r;
    hipLaunchKernelGGL(k_force_assemble, dim3(grid), dim3(64 * FR_PARTS), 0, c->s, sol[n], psol,
                       c->d_uinv, c->d_pdet, c->d_aux, c->d_aux2, c->d_nbr, c->d_t, c->d_force,
                       V, c->p.nt, (double)c->p.PBC, c->doG, c->p.G, amps[n], n == 0, ord);
    HIPCHK(hipGetLastError());
  }
  int nb = (V * NUMLINK + FB - 1) / FB;
  hipLaunchKernelGGL(k_force_apply, dim3(nb), dim3(FB), 0, c->s, c->d_force, c->d_mom, eps, V,
                     c->d_part);
  HIPCHK(hipGetLastError());
  int r = reduce_partials(c, c->d_part, nb, 0);
  if (r) return r;
  double sc;
  if ((r = read_scalars(c, &sc, 1))) return r;
  if (norm) *norm = eps * sqrt(sc) / V;
  return 0;
}
