// Device kernels of the FLO-SIC per-Fermi-orbital evaluation, written for gfx950 (64-wide wavefronts).
//
//   k_basis_planes   contracted Cartesian Gaussians and their derivatives on the mesh (gorbdrv.f:18-316);
//                    FOD independent, computed once per system and kept resident in HBM
//   k_prim_coef      FLO coefficients folded onto primitive shells (the ADD/DMAT contraction of
//                    coupot_sic.F:398-482)
//   k_hermite        Hermite expansion of every primitive pair density for every FLO (the COEFICIENT
//                    polynomial set of poisson1.f:295-496, McMurchie-Davidson form), 2 pi/p folded in
//   k_coulomb        exact Gaussian-pair potential at every mesh point for all FLOs at once: Boys
//                    functions by the table/Taylor/asymptote scheme of fffmt3.F/fffmt4.F/fffmtc.F,
//                    Hermite recursion in registers, contraction with the pair coefficients
//   k_xc             spin-polarised LSDA/PBE for rho_up = rho_i, rho_dn = 0 (subvlxc_libxc.F90), total SIC
//                    potential and per-block partial sums of the RESULTS energies (apotnl_sic.F:536-581)
//   k_vab_mfma       V^i_ab = sum_k w phi_a V_i phi_b as an FP64 MFMA GEMM over point slices
#include "flosic_device.h"

namespace flosic {

// value (+ gradient, + Hessian xx,yy,zz,xy,xz,yz) of component IDX times the radial sums
// S0 = sum c e^{-a r^2}, S1 = sum c a e^{-a r^2}, S2 = sum c a^2 e^{-a r^2}
template <int IDX, int ND>
__device__ __forceinline__ void cart_eval(double x, double y, double z, double S0, double S1, double S2,
                                          double *o) {
    constexpr int a = cpow(IDX, 0), b = cpow(IDX, 1), c = cpow(IDX, 2);
    const double px[3] = {1.0, x, x * x}, py[3] = {1.0, y, y * y}, pz[3] = {1.0, z, z * z};
    const double P = px[a] * py[b] * pz[c];
    o[0] = P * S0;
    if constexpr (ND >= 4) {
        const double dPx = a ? a * px[a - 1] * py[b] * pz[c] : 0.0;
        const double dPy = b ? b * px[a] * py[b - 1] * pz[c] : 0.0;
        const double dPz = c ? c * px[a] * py[b] * pz[c - 1] : 0.0;
        o[1] = dPx * S0 - 2.0 * x * P * S1;
        o[2] = dPy * S0 - 2.0 * y * P * S1;
        o[3] = dPz * S0 - 2.0 * z * P * S1;
        if constexpr (ND == 10) {
            const double dPxx = a >= 2 ? a * (a - 1) * py[b] * pz[c] : 0.0;
            const double dPyy = b >= 2 ? b * (b - 1) * px[a] * pz[c] : 0.0;
            const double dPzz = c >= 2 ? c * (c - 1) * px[a] * py[b] : 0.0;
            const double dPxy = (a && b) ? a * b * px[a - 1] * py[b - 1] * pz[c] : 0.0;
            const double dPxz = (a && c) ? a * c * px[a - 1] * py[b] * pz[c - 1] : 0.0;
            const double dPyz = (b && c) ? b * c * px[a] * py[b - 1] * pz[c - 1] : 0.0;
            o[4] = dPxx * S0 - 4.0 * x * dPx * S1 + P * (4.0 * x * x * S2 - 2.0 * S1);
            o[5] = dPyy * S0 - 4.0 * y * dPy * S1 + P * (4.0 * y * y * S2 - 2.0 * S1);
            o[6] = dPzz * S0 - 4.0 * z * dPz * S1 + P * (4.0 * z * z * S2 - 2.0 * S1);
            o[7] = dPxy * S0 - 2.0 * x * dPy * S1 - 2.0 * y * dPx * S1 + 4.0 * x * y * P * S2;
            o[8] = dPxz * S0 - 2.0 * x * dPz * S1 - 2.0 * z * dPx * S1 + 4.0 * x * z * P * S2;
            o[9] = dPyz * S0 - 2.0 * y * dPz * S1 - 2.0 * z * dPy * S1 + 4.0 * y * z * P * S2;
        }
    }
}

// ND = 1, 4 or 10 planes (value, gradient, Hessian); ND = -1: one plane holding the Laplacian
template <typename T, int ND, int L, int M0>
__device__ __forceinline__ void store_comps(double x, double y, double z, double S0, double S1, double S2, T *phi,
                                            int64_t ldphi, int64_t plane, int f0, int stride, int64_t k) {
    if constexpr (M0 < ncart(L)) {
        const int64_t col = (int64_t)(f0 + M0 * stride) * ldphi + k;
        if constexpr (ND == -1) {
            double o[10];
            cart_eval<loff(L) + M0, 10>(x, y, z, S0, S1, S2, o);
            phi[col] = (T)(o[4] + o[5] + o[6]);
        } else if constexpr (ND == -3) {
            double o[4];
            cart_eval<loff(L) + M0, 4>(x, y, z, S0, S1, S2, o);
#pragma unroll
            for (int d = 0; d < 3; ++d) phi[d * plane + col] = (T)o[1 + d];
        } else {
            double o[ND];
            cart_eval<loff(L) + M0, ND>(x, y, z, S0, S1, S2, o);
#pragma unroll
            for (int d = 0; d < ND; ++d) phi[d * plane + col] = (T)o[d];
        }
        store_comps<T, ND, L, M0 + 1>(x, y, z, S0, S1, S2, phi, ldphi, plane, f0, stride, k);
    }
}

// Planes phi[d][mu][k] (leading dimension ldphi >= M, plane = nbas*ldphi).  Thread = point, blockIdx.y = a share of the
// contracted shells; a function screened at a point is stored as zero, so the planes need no clearing beforehand.
// Bound: the stores where points abound, the chain of exponentials of a thread where they do not, so the shells are shared out
// over blocks until there are about 2048 of 256 threads (eight per CU): the chain of a pass over a few FODs ends after
// one shell.  With all shells in one thread, after a fill of the planes: value and gradient at 10 FODs 27 us, at 96
// FODs 240; three gradient planes of 16 atoms' basis on 32 768 points 102 and 39 for the fill.  Now 11, 9 and 51.
template <typename T, int ND>
__global__ void __launch_bounds__(256) k_basis_planes(BasisDev B, const double *__restrict__ X,
                                                      const double *__restrict__ Y, const double *__restrict__ Z,
                                                      int64_t M, T *__restrict__ phi, int64_t ldphi) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= M) return;
    const int s0 = (int)((int64_t)B.ncs * blockIdx.y / gridDim.y), s1 = (int)((int64_t)B.ncs * (blockIdx.y + 1) / gridDim.y);
    const double px = X[k], py = Y[k], pz = Z[k];
    const int64_t plane = (int64_t)B.nbas * ldphi;
    const double geps = exp(-kCutExp);
    for (int a = 0, s = s0; s < s1; ++a) {
        const int se = min(s1, B.atom_cs[a + 1]);
        if (s >= se) continue;
        const double x = px - B.atom_xyz[3 * a], y = py - B.atom_xyz[3 * a + 1], z = pz - B.atom_xyz[3 * a + 2];
        const double r2 = x * x + y * y + z * z;
        const bool in = r2 < B.atom_r2cut[a];
        for (; s < se; ++s) {
            double S0 = 0.0, S1 = 0.0, S2 = 0.0;
            for (int p = in ? B.cs_p0[s] : B.cs_p0[s + 1]; p < B.cs_p0[s + 1]; ++p) {
                const double al = B.prim_alpha[p];
                const double arg = al * r2;
                if (!(arg < kCutExp)) continue;
                const double g = exp(-arg);
                const double cc = B.prim_coef[p];
                if (!(fabs(cc) * g > geps)) continue;
                const double gc = g * cc;
                S0 += gc;
                S1 += gc * al;
                S2 += gc * al * al;
            }
            const int l = B.cs_l[s];
            if (l == 0) store_comps<T, ND, 0, 0>(x, y, z, S0, S1, S2, phi, ldphi, plane, B.cs_f0[s], B.cs_stride[s], k);
            else if (l == 1) store_comps<T, ND, 1, 0>(x, y, z, S0, S1, S2, phi, ldphi, plane, B.cs_f0[s], B.cs_stride[s], k);
            else store_comps<T, ND, 2, 0>(x, y, z, S0, S1, S2, phi, ldphi, plane, B.cs_f0[s], B.cs_stride[s], k);
        }
    }
}

template <typename T>
void launch_basis_planes(const BasisDev &B, const double *x, const double *y, const double *z, int64_t M, int nd,
                         T *phi, int64_t ldphi, hipStream_t s) {
    if (M <= 0 || B.ncs <= 0) return;
    const int64_t nb = (M + 255) / 256;
    const dim3 grid((unsigned)nb, (unsigned)std::min<int64_t>(B.ncs, (2048 + nb - 1) / nb)), blk(256);
    if (nd == 1) hipLaunchKernelGGL((k_basis_planes<T, 1>), grid, blk, 0, s, B, x, y, z, M, phi, ldphi);
    else if (nd == 4) hipLaunchKernelGGL((k_basis_planes<T, 4>), grid, blk, 0, s, B, x, y, z, M, phi, ldphi);
    else if (nd == -1) hipLaunchKernelGGL((k_basis_planes<T, -1>), grid, blk, 0, s, B, x, y, z, M, phi, ldphi);
    else if (nd == -3) hipLaunchKernelGGL((k_basis_planes<T, -3>), grid, blk, 0, s, B, x, y, z, M, phi, ldphi);
    else hipLaunchKernelGGL((k_basis_planes<T, 10>), grid, blk, 0, s, B, x, y, z, M, phi, ldphi);
}
template void launch_basis_planes<double>(const BasisDev &, const double *, const double *, const double *, int64_t,
                                          int, double *, int64_t, hipStream_t);
template void launch_basis_planes<float>(const BasisDev &, const double *, const double *, const double *, int64_t,
                                         int, float *, int64_t, hipStream_t);

// T[f][k] = w_k (a * lap[f][k] + pot[k] * phi[f][k]) over n FLOs, lap the sum of nlap planes of [n][M] (lap may be null:
// T = w * pot * phi, or with pot null: T = w * phi)
__global__ void k_weighted_op(int n, int64_t M, const double *__restrict__ w, const double *__restrict__ pot,
                              const double *__restrict__ phi, const double *__restrict__ lap, int nlap, double a,
                              double *__restrict__ T) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)n * M) return;
    const int64_t k = e % M;
    double v = pot ? pot[k] * phi[e] : phi[e];
    if (lap) {
        double l = lap[e];
        for (int q = 1; q < nlap; ++q) l += lap[(int64_t)q * n * M + e];
        v += a * l;
    }
    T[e] = w[k] * v;
}
void launch_weighted_op(int n, int64_t M, const double *w, const double *pot, const double *phi, const double *lap,
                        int nlap, double a, double *T, hipStream_t s) {
    const int64_t cnt = (int64_t)n * M;
    if (cnt <= 0) return;
    hipLaunchKernelGGL(k_weighted_op, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, s, n, M, w, pot, phi, lap, nlap, a,
                       T);
}

// ---------------------------------------------------------------------------------------------------
// FLO coefficients on primitive shells: dps[(ps*6 + m)*nF + f] = sum_c con_c * cflo[f*ldc + f0 + m*stride + c]
// ---------------------------------------------------------------------------------------------------
__global__ void k_prim_coef(int nps, const int *__restrict__ ps_f0, const int *__restrict__ ps_stride,
                            const int *__restrict__ ps_ncart, const int *__restrict__ ps_c0,
                            const int *__restrict__ ps_nc, const double *__restrict__ ps_coef,
                            const double *__restrict__ cflo, int nF, int ldc, double *__restrict__ dps) {
    const int ps = blockIdx.x;
    const int f0 = ps_f0[ps], st = ps_stride[ps], nc = ps_nc[ps], c0 = ps_c0[ps], nm = ps_ncart[ps];
    for (int f = threadIdx.x; f < nF; f += blockDim.x) {
        for (int m = 0; m < 6; ++m) {
            double s = 0.0;
            if (m < nm)
                for (int c = 0; c < nc; ++c) s += ps_coef[c0 + c] * cflo[(int64_t)f * ldc + f0 + m * st + c];
            dps[((int64_t)ps * 6 + m) * nF + f] = s;
        }
    }
}

void launch_prim_coef(int nps, const int *ps_f0, const int *ps_stride, const int *ps_ncart, const int *ps_c0,
                      const int *ps_nc, const double *ps_coef, const double *cflo, int nF, int ldc, double *dps,
                      hipStream_t s) {
    if (nps <= 0) return;
    hipLaunchKernelGGL(k_prim_coef, dim3(nps), dim3(128), 0, s, nps, ps_f0, ps_stride, ps_ncart, ps_c0, ps_nc,
                       ps_coef, cflo, nF, ldc, dps);
}

// ---------------------------------------------------------------------------------------------------
// Hermite coefficients of every pair for every FLO.  E^{ij}_t along one axis by the McMurchie-Davidson
// recursion; H[row+tuv][f] = sym * 2pi/p * sum_{mu,nu} dA[mu][f] dB[nu][f] Ex Ey Ez
//
// Bound: latency, a few microseconds of work per block at any system size.  One block per group: 27 threads raise the
// E^{ij}_t of one axis and (i, j) in registers; the products Ex Ey Ez of every (component pair, tuv) go to LDS, wave = component
// of the first centre, lane = tuv; then a thread holds one (tuv, FLO) and runs over the component pairs, up to 100, from LDS,
// five loads at a time.  A thread that held all 35 sums of one FLO (indexed at run time, so in scratch memory) left 54 of
// 64 lanes idle at 10 FLOs and took 190 us there (289 groups), 229 at 30 FLOs (1686 groups), 525 at 96 FLOs (15750); with one
// load after the other and the pairs one by one over the waves 27, 82 and 279; now 17, 60 and 262.
// ---------------------------------------------------------------------------------------------------
constexpr int kHermThreads = 256, kHermCols = 64;
__device__ __forceinline__ void e_raise(double (&v)[5], double shift, double inv2p) {
    double o[5];
#pragma unroll
    for (int t = 0; t < 5; ++t) o[t] = v[t];
#pragma unroll
    for (int t = 0; t < 5; ++t) {
        double x = t >= 1 ? inv2p * o[t >= 1 ? t - 1 : 0] : 0.0;
        x += shift * o[t];
        if (t < 4) x += (t + 1) * o[t < 4 ? t + 1 : 4];
        v[t] = x;
    }
}
__global__ void __launch_bounds__(kHermThreads) k_hermite(const PairDev *__restrict__ pairs,
                                                          const double *__restrict__ dps, int nF,
                                                          double *__restrict__ H, int ldh) {
    __shared__ double E[3][3][3][5], C[100 * 35], dA[10][kHermCols], dB[10][kHermCols];
    const PairDev pr = pairs[blockIdx.x];
    const double p = pr.a + pr.b;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (tid < 27) {
        const int d = tid / 9, i = tid / 3 % 3, j = tid % 3;
        const double A = d == 0 ? pr.A[0] : d == 1 ? pr.A[1] : pr.A[2], B = d == 0 ? pr.B[0] : d == 1 ? pr.B[1] : pr.B[2];
        const double P = (pr.a * A + pr.b * B) / p;
        const double xpa = P - A, xpb = P - B, dd = A - B, inv2p = 0.5 / p;
        double v[5] = {exp(-pr.a * pr.b / p * dd * dd), 0.0, 0.0, 0.0, 0.0};
        for (int q = 0; q < j; ++q) e_raise(v, xpb, inv2p);
        for (int q = 0; q < i; ++q) e_raise(v, xpa, inv2p);
#pragma unroll
        for (int t = 0; t < 5; ++t) E[d][i][j][t] = v[t];
    }
    // components of either centre: those of the shells l that it has, as bits of the component index 0..9
    int mA = 0, mB = 0;
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        const int bits = ((1 << ncart(l)) - 1) << loff(l);
        if (l <= pr.lA && pr.psA[l] >= 0) mA |= bits;
        if (l <= pr.lB && pr.psB[l] >= 0) mB |= bits;
    }
    const int nB = __builtin_popcount(mB), nA = __builtin_popcount(mA), nt = ntuv(pr.lA + pr.lB);
    const double fac = pr.sym * 2.0 * M_PI / p;
    __syncthreads();
    {
        // (t, u, v) of entry `lane`: order, then the position in its block: t falls by one after 1, 2, 3, .. entries
        const int ord = lane < 1 ? 0 : lane < 4 ? 1 : lane < 10 ? 2 : lane < 20 ? 3 : 4;
        const int pos = min(lane, 34) - ord * (ord + 1) * (ord + 2) / 6;
        const int uv = pos < 1 ? 0 : pos < 3 ? 1 : pos < 6 ? 2 : pos < 10 ? 3 : 4;
        const int t = ord - uv, v = pos - uv * (uv + 1) / 2, u = uv - v;
        for (int ma = mA, ia = 0; ma; ma &= ma - 1, ++ia) {
            if ((ia & 3) != wave) continue;
            const int a = __builtin_ctz(ma), ax = cpow(a, 0), ay = cpow(a, 1), az = cpow(a, 2);
            double *c = C + ia * nB * nt + lane;
            for (int mb = mB; mb; mb &= mb - 1, c += nt) {
                const int b = __builtin_ctz(mb), bx = cpow(b, 0), by = cpow(b, 1), bz = cpow(b, 2);
                if (lane < nt) *c = E[0][ax][bx][t] * E[1][ay][by][u] * E[2][az][bz][v];
            }
        }
    }
    // columns at a time (of ldh, nF rounded up to 16)
    const int sh = ldh > 32 ? 6 : ldh > 16 ? 5 : 4, cols = 1 << sh;
    for (int f0 = 0; f0 < ldh; f0 += cols) {
        __syncthreads();
        for (int x = tid; x < (nA + nB) << sh; x += kHermThreads) {
            const int f = f0 + (x & (cols - 1)), c = x >> sh;
            const bool isA = c < nA;
            int m = isA ? mA : mB;
            for (int q = isA ? c : c - nA; q > 0; --q) m &= m - 1;
            const int k = __builtin_ctz(m), l = k < loff(1) ? 0 : k < loff(2) ? 1 : 2;
            const int ps = isA ? (l == 0 ? pr.psA[0] : l == 1 ? pr.psA[1] : pr.psA[2])
                               : (l == 0 ? pr.psB[0] : l == 1 ? pr.psB[1] : pr.psB[2]);
            (isA ? dA[c] : dB[c - nA])[x & (cols - 1)] = f < nF ? dps[((int64_t)ps * 6 + k - loff(l)) * nF + f] : 0.0;
        }
        __syncthreads();
        for (int x = tid; x < nt << sh; x += kHermThreads) {
            const int fl = x & (cols - 1), tuv = x >> sh;
            if (f0 + fl >= ldh) continue;
            const double *c = C + tuv;
            double h = 0.0;
            for (int m = 0; m < nA; ++m) {
                const double da = dA[m][fl];
                int n = 0;
                for (; n + 5 <= nB; n += 5, c += 5 * nt) {  // ten of an spd centre: the LDS loads of five go out together
                    double b[5], x[5];
#pragma unroll
                    for (int e = 0; e < 5; ++e) {
                        b[e] = dB[n + e][fl];
                        x[e] = c[e * nt];
                    }
#pragma unroll
                    for (int e = 0; e < 5; ++e) h += da * b[e] * x[e];
                }
                for (; n < nB; ++n, c += nt) h += da * dB[n][fl] * *c;
            }
            H[(int64_t)(pr.row + tuv) * ldh + f0 + fl] = fac * h;
        }
    }
}

void launch_hermite(int ngroup, const PairDev *pairs, const double *dps, int nF, double *H, int ldh, hipStream_t s) {
    if (ngroup <= 0) return;
    hipLaunchKernelGGL(k_hermite, dim3(ngroup), dim3(kHermThreads), 0, s, pairs, dps, nF, H, ldh);
}

template <int L, int CH>
__device__ __forceinline__ void coulomb_segment(int beg, int end, const double4 *__restrict__ pP,
                                                const int *__restrict__ prow, const double *__restrict__ H, int ldh,
                                                int f0, double x, double y, double z, const double *__restrict__ tab,
                                                double *acc) {
    for (int ip = beg; ip < end; ++ip) {
        const double4 P = pP[ip];
        const int row = prow[ip];
        double R[ntuv(L)];
        hermite_R<L>(P.w, P.x - x, P.y - y, P.z - z, tab, R);
        const double *h = H + (int64_t)row * ldh + f0;
#pragma unroll
        for (int t = 0; t < ntuv(L); ++t) {
#pragma unroll
            for (int c = 0; c < CH; ++c) acc[c] = fma(R[t], h[(int64_t)t * ldh + c], acc[c]);
        }
    }
}

// block = 4 wavefronts; wave w of block (bx, by) handles points bx*64 .. +63 and FLO chunk (by*4 + w)
template <int CH>
__global__ void __launch_bounds__(256) k_coulomb(int s0, int s1, int s2, int s3, int s4, int s5,
                                                  const double4 *__restrict__ pP, const int *__restrict__ prow,
                                                  const double *__restrict__ H, int ldh, const double *__restrict__ X,
                                                  const double *__restrict__ Y, const double *__restrict__ Z,
                                                  int64_t M, const double *__restrict__ tab, int nF,
                                                  double *__restrict__ V, int64_t ldv) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int f0 = (blockIdx.y * 4 + wave) * CH;
    if (f0 >= nF) return;
    const int64_t k = (int64_t)blockIdx.x * 64 + lane;
    const bool valid = k < M;
    const double x = valid ? X[k] : 0.0, y = valid ? Y[k] : 0.0, z = valid ? Z[k] : 0.0;
    double acc[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) acc[c] = 0.0;
    coulomb_segment<0, CH>(s0, s1, pP, prow, H, ldh, f0, x, y, z, tab, acc);
    coulomb_segment<1, CH>(s1, s2, pP, prow, H, ldh, f0, x, y, z, tab, acc);
    coulomb_segment<2, CH>(s2, s3, pP, prow, H, ldh, f0, x, y, z, tab, acc);
    coulomb_segment<3, CH>(s3, s4, pP, prow, H, ldh, f0, x, y, z, tab, acc);
    coulomb_segment<4, CH>(s4, s5, pP, prow, H, ldh, f0, x, y, z, tab, acc);
    if (valid) {
#pragma unroll
        for (int c = 0; c < CH; ++c)
            if (f0 + c < nF) V[(int64_t)(f0 + c) * ldv + k] = acc[c];
    }
}

void launch_coulomb(const int *segL, const double4 *pairP, const int *pairRow, const double *H, int ldh,
                    const double *x, const double *y, const double *z, int64_t M, const double *btab, int nF, double *V,
                    int64_t ldv, hipStream_t s) {
    constexpr int CH = 16;
    const int nchunk = (nF + CH - 1) / CH;
    const dim3 grid((unsigned)((M + 63) / 64), (unsigned)((nchunk + 3) / 4)), blk(256);
    hipLaunchKernelGGL((k_coulomb<CH>), grid, blk, 0, s, segL[0], segL[1], segL[2], segL[3], segL[4], segL[5], pairP,
                       pairRow, H, ldh, x, y, z, M, btab, nF, V, ldv);
}

// Column-block widths: by default all FLOs up to 256 columns (ldh is nF rounded up to a multiple of this), in the split-BF16
// form up to 192 and 128 beyond that.  A block takes at most 12 tiles of 16 columns, four column waves of three, whatever
// width is asked for (coulomb_col_blocks).
int coulomb_cols(int nF) { return nF <= 64 ? 64 : nF <= 128 ? 128 : nF <= 192 ? 192 : 256; }
bool coulomb_cols_legal(int nfb, int ldh, bool split) {
    if (nfb != 64 && nfb != 128 && nfb != 192 && nfb != 256) return false;
    if (split && nfb > 192) return false;
    return ldh % nfb == 0;
}
int coulomb_cols_split(int nF) { return nF <= 64 ? 64 : nF <= 128 ? 128 : nF <= 192 ? 192 : 128; }

// ---------------------------------------------------------------------------------------------------
// exchange-correlation for rho_up = rho_i, rho_dn = 0, NSPN = 2 (subvlxc_libxc.F90:197-470)
// ---------------------------------------------------------------------------------------------------
__device__ __forceinline__ void gcor(double A, double A1, double B1, double B2, double B3, double B4, double RS,
                                     double &GG, double &GGRS) {
    const double Q0 = -2 * A * (1.0 + A1 * RS);
    const double RS12 = sqrt(RS);
    const double RS32 = RS12 * RS12 * RS12;
    const double Q1 = 2 * A * (B1 * RS12 + B2 * RS + B3 * RS32 + B4 * RS * RS);
    const double Q2 = log(1.0 + 1.0 / Q1);
    GG = Q0 * Q2;
    const double Q3 = A * (B1 / RS12 + 2 * B2 + 3 * B3 * RS12 + 4 * B4 * RS);
    GGRS = -2 * A * A1 * Q2 - Q0 * Q3 / (Q1 * Q1 + Q1);
}
__device__ __forceinline__ void gcor2(double A, double A1, double B1, double B2, double B3, double B4, double RTRS,
                                      double &GG, double &GGRS) {
    const double Q0 = -2.0 * A * (1.0 + A1 * RTRS * RTRS);
    const double Q1 = 2.0 * A * RTRS * (B1 + RTRS * (B2 + RTRS * (B3 + B4 * RTRS)));
    const double Q2 = log(1.0 + 1.0 / Q1);
    GG = Q0 * Q2;
    const double Q3 = A * (B1 / RTRS + 2.0 * B2 + RTRS * (3.0 * B3 + 4.0 * B4 * RTRS));
    GGRS = -2.0 * A * A1 * Q2 - Q0 * Q3 / (Q1 * (1.0 + Q1));
}

// PW91 exchange (pw91ex.f:7-50)
__device__ __forceinline__ void pw91ex(double DKF, double S, double U, double V, double &EXL, double &EXN,
                                       double &VX) {
    const double A1 = 0.19645, A2 = 0.27430, A3 = 0.15084, A4 = 100.0, AX = -0.238732414, A = 7.7956, B1 = 0.004;
    const double THRD4 = 1.3333333333333333;
    const double FAC = AX * DKF;
    const double S2 = S * S, S3 = S2 * S, S4 = S2 * S2;
    const double AS = A * S;
    const double PA = sqrt(1.0 + AS * AS);
    const double P0 = AS / PA;
    const double P1 = A1 * log(AS + PA);
    const double P2 = A3 * exp(-A4 * S2);
    const double P3 = 1.0 / (1.0 + S * P1 + B1 * S4);
    const double P4 = 1.0 + S * P1 + (A2 - P2) * S2;
    const double F = P3 * P4;
    EXL = FAC;
    EXN = FAC * (F - 1.0);
    const double P5 = B1 * S2 - (A2 - P2);
    const double P6 = S * (P1 + A1 * P0);
    const double P7 = 2 * ((A2 - P2) + A4 * S2 * P2 - 2 * B1 * S2 * F);
    const double FS = P3 * (P3 * P5 * P6 + P7);
    const double P8 = 2 * S * (B1 - A4 * P2);
    const double P9 = P1 + A1 * P0 * (3.0 - P0 * P0);
    const double P10 = 4 * (A4 * S * P2 * (2.0 - A4 * S2) - 2 * B1 * S * F - B1 * S3 * FS);
    const double P11 = P3 * P3 * (P1 + A1 * P0 + 4 * B1 * S3);
    const double FSS = P3 * P3 * (P5 * P9 + P6 * P8) - 2 * P3 * P5 * P6 * P11 + P3 * P10 - P7 * P11;
    VX = FAC * (THRD4 * F - (U - THRD4 * S3) * FSS - V * FS);
}

// PW92 local correlation at zeta = 1 (pw91lc.f:4-43): the spin stiffness (its third interpolation) has the factor 1 - zeta^4,
// and the zeta derivative enters the up-spin potential as -zeta + 1 times itself, so neither is computed
__device__ __forceinline__ void pw91lc_pol(double RS, double &EC, double &VCUP) {
    const double GAMR = 1.92366105, THRD = 0.333333333333;
    const double ZETPR = pow(2.0, THRD);
    const double F = (ZETPR * ZETPR * ZETPR * ZETPR - 2.0) * GAMR;
    double EU, EURS, EP, EPRS;
    gcor(0.0310907, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294, RS, EU, EURS);
    gcor(0.01554535, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517, RS, EP, EPRS);
    EC = EU * (1.0 - F) + EP * F;
    const double ECRS = EURS * (1.0 - F) + EPRS * F;
    VCUP = EC - RS * ECRS * THRD;
}

// PW92 local correlation at general zeta (pw91lc.f:4-43): EC and both spin potentials
__device__ __forceinline__ void pw91lc_gen(double RS, double ZET, double &EC, double &VCUP, double &VCDN) {
    const double GAMR = 1.92366105, FZZR = 0.58482234, THRD = 0.333333333333, THRD4 = 1.333333333333;
    const double ZETPR = pow(1.0 + ZET, THRD), ZETMR = pow(1.0 - ZET, THRD);
    const double F = (ZETPR * ZETPR * ZETPR * ZETPR + ZETMR * ZETMR * ZETMR * ZETMR - 2.0) * GAMR;
    double EU, EURS, EP, EPRS, ALFM, ALFRSM;
    gcor(0.0310907, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294, RS, EU, EURS);
    gcor(0.01554535, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517, RS, EP, EPRS);
    gcor(0.0168869, 0.11125, 10.357, 3.6231, 0.88026, 0.49671, RS, ALFM, ALFRSM);
    const double Z3 = ZET * ZET * ZET, Z4 = Z3 * ZET;
    EC = EU * (1.0 - F * Z4) + EP * F * Z4 - ALFM * F * (1.0 - Z4) * FZZR;
    const double ECRS = EURS * (1.0 - F * Z4) + EPRS * F * Z4 - ALFRSM * F * (1.0 - Z4) * FZZR;
    const double FZ = THRD4 * (ZETPR - ZETMR) * GAMR;
    const double ECZET = 4.0 * Z3 * F * (EP - EU + ALFM * FZZR) + FZ * (Z4 * EP - Z4 * EU - (1.0 - Z4) * ALFM * FZZR);
    const double COMM = EC - RS * ECRS * THRD - ZET * ECZET;
    VCUP = COMM + ECZET;
    VCDN = COMM - ECZET;
}

// PBE exchange (pbeex.f, MODE=1) from the cube root of the density
__device__ __forceinline__ void pbeex(double RHO3, double S, double U, double V, double &EXL, double &EXN,
                                      double &VX) {
    const double THRD4 = 4.0 / 3.0;
    const double AX = -0.738558766382022405884230032680836, UM = 0.2195149727645171, UK = 0.8040, UL = UM / UK;
    const double EXUNIF = AX * RHO3;
    const double S2 = S * S;
    const double P0 = 1.0 + UL * S2;
    const double FXPBE = 1.0 + UK - UK / P0;
    EXL = EXUNIF;
    EXN = EXUNIF * (FXPBE - 1.0);
    const double FS = 2.0 * UK * UL / (P0 * P0);
    const double FSS = -4.0 * UL * S * FS / P0;
    VX = EXUNIF * (THRD4 * FXPBE - (U - THRD4 * S2 * S) * FSS - V * FS);
}

// PBE correlation at zeta = 1, WW = 0 (pbecor.f).  The spin stiffness has the factor 1 - zeta^4, and every zeta derivative
// enters the up-spin potential as -zeta + 1 times itself, so neither is computed
__device__ __forceinline__ void pbecor_pol(double RS, double T, double UU, double VV, double &EC, double &VCUP,
                                           double &H, double &DVCUP) {
    const double THRD2 = 2.0 / 3.0, THRD4 = 4.0 / 3.0;
    const double GAM = 0.5198420997897463295344212145565;
    const double GAMMA = 0.03109069086965489503494086371273, BET = 0.06672455060314922, DELT = BET / GAMMA;
    const double RTRS = sqrt(RS);
    double EU, EURS, EP, EPRS;
    gcor2(0.0310907, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294, RTRS, EU, EURS);
    gcor2(0.01554535, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517, RTRS, EP, EPRS);
    const double F = (pow(2.0, THRD4) - 2.0) / GAM;
    const double ec = EU * (1.0 - F) + EP * F;
    const double ECRS = EURS * (1.0 - F) + EPRS * F;
    EC = ec;
    VCUP = ec - RS * ECRS / 3.0;
    const double G = pow(2.0, THRD2) / 2.0;
    const double G3 = G * G * G;
    const double PON = -ec / (G3 * GAMMA);
    const double B = DELT / (exp(PON) - 1.0);
    const double B2 = B * B, T2 = T * T, T4 = T2 * T2;
    const double Q4 = 1.0 + B * T2;
    const double Q5 = 1.0 + B * T2 + B2 * T4;
    const double h = G3 * (BET / DELT) * log(1.0 + DELT * Q4 * T2 / Q5);
    const double T6 = T4 * T2, RSTHRD = RS / 3.0;
    const double FAC = DELT / B + 1.0;
    const double BEC = B2 * FAC / (BET * G3);
    const double Q8 = Q5 * Q5 + DELT * Q4 * Q5 * T2;
    const double Q9 = 1.0 + 2.0 * B * T2;
    const double HB = -BET * G3 * B * T6 * (2.0 + B * T2) / Q8;
    const double HRS = -RSTHRD * HB * BEC * ECRS;
    const double FACT0 = 2.0 * DELT - 6.0 * B;
    const double FACT1 = Q5 * Q9 + Q4 * Q9 * Q9;
    const double HBT = 2.0 * BET * G3 * T4 * ((Q4 * Q5 * FACT0 - DELT * FACT1) / Q8) / Q8;
    const double HRST = RSTHRD * T2 * HBT * BEC * ECRS;
    const double HT = 2.0 * BET * G3 * Q9 / Q8;
    const double FACT2 = Q4 * Q5 + B * T2 * (Q4 * Q9 + Q5);
    const double FACT3 = 2.0 * B * Q5 * Q9 + DELT * FACT2;
    const double HTT = 4.0 * BET * G3 * T * (2.0 * B / Q8 - (Q9 * FACT3 / Q8) / Q8);
    H = h;
    DVCUP = h + HRS + HRST + T2 * HT / 6.0 + 7.0 * T2 * T * HTT / 6.0 - UU * HTT - VV * HT;
}

// ---------------------------------------------------------------------------------------------------
// Exact partial derivatives of the PBE energy density.  The energy that xc_point integrates depends on the
// orbital density only through rho and g = |grad rho| (U, V, UU, VV enter the potential alone), so
// e(rho, g) = EXL + EXN + ECL + ECN is restated below as one expression and differentiated in forward mode
// (value + derivative along rho + derivative along g, in one evaluation).
// ---------------------------------------------------------------------------------------------------
struct Fwd {
    double v, r, g;
};
__device__ __forceinline__ Fwd operator+(Fwd a, Fwd b) { return {a.v + b.v, a.r + b.r, a.g + b.g}; }
__device__ __forceinline__ Fwd operator-(Fwd a, Fwd b) { return {a.v - b.v, a.r - b.r, a.g - b.g}; }
__device__ __forceinline__ Fwd operator*(Fwd a, Fwd b) {
    return {a.v * b.v, a.r * b.v + a.v * b.r, a.g * b.v + a.v * b.g};
}
__device__ __forceinline__ Fwd operator/(Fwd a, Fwd b) {
    const double q = a.v / b.v, i = 1.0 / b.v;
    return {q, (a.r - q * b.r) * i, (a.g - q * b.g) * i};
}
__device__ __forceinline__ Fwd operator+(double a, Fwd b) { return {a + b.v, b.r, b.g}; }
__device__ __forceinline__ Fwd operator-(double a, Fwd b) { return {a - b.v, -b.r, -b.g}; }
__device__ __forceinline__ Fwd operator*(double a, Fwd b) { return {a * b.v, a * b.r, a * b.g}; }
__device__ __forceinline__ Fwd operator/(double a, Fwd b) {
    const double q = a / b.v, s = -q / b.v;
    return {q, s * b.r, s * b.g};
}
__device__ __forceinline__ Fwd fsqrt(Fwd a) {
    const double s = sqrt(a.v), i = 0.5 / s;
    return {s, i * a.r, i * a.g};
}
__device__ __forceinline__ Fwd flog(Fwd a) {
    const double i = 1.0 / a.v;
    return {log(a.v), i * a.r, i * a.g};
}
__device__ __forceinline__ Fwd fexp(Fwd a) {
    const double e = exp(a.v);
    return {e, e * a.r, e * a.g};
}

// the value part of gcor2 (pbecor.f) in forward mode
__device__ __forceinline__ Fwd gcor2_fwd(double A, double A1, double B1, double B2, double B3, double B4, Fwd RTRS) {
    const Fwd Q0 = -2.0 * A * (1.0 + A1 * (RTRS * RTRS));
    const Fwd Q1 = 2.0 * A * (RTRS * (B1 + RTRS * (B2 + RTRS * (B3 + B4 * RTRS))));
    return Q0 * flog(1.0 + 1.0 / Q1);
}

// cube roots of 2 and of 3 pi^2 (TRPI2 below)
constexpr double kCbrt2 = 1.2599210498948731648, kCbrtTRPI2 = 3.0936677262801359310;

// e(rho, g): PBE exchange of the up spin at D = 2 rho (pbeex.f) + PBE correlation at zeta = 1 (pbecor.f), per
// unit volume, with the same constants as xc_point; rho3 the cube root of rho
__device__ __forceinline__ Fwd pbe_edens(double rhov, double rho3, double gv) {
    const double FRDPI = 1.2732395447351627;
    const double DKF2RS = 1.9191582926775128;
    const double AX = -0.738558766382022405884230032680836, UM = 0.2195149727645171, UK = 0.8040, UL = UM / UK;
    const double GAM = 0.5198420997897463295344212145565;
    const double GAMMA = 0.03109069086965489503494086371273, BET = 0.06672455060314922, DELT = BET / GAMMA;
    const Fwd rho{rhov, 1.0, 0.0}, g{gv, 0.0, 1.0}, c{rho3, rho3 / (3.0 * rhov), 0.0};
    // exchange: S = 2g / (2 kF D)
    const Fwd D = 2.0 * rho;
    const Fwd DKF = (kCbrtTRPI2 * kCbrt2) * c;
    const Fwd S = (2.0 * g) * (0.5 / (DKF * D));
    const Fwd EXUNIF = (AX * kCbrt2) * c;
    const Fwd FX = (1.0 + UK) - UK / (1.0 + UL * (S * S));
    const Fwd ex = 0.5 * ((EXUNIF * FX) * D);
    // correlation: T = g / (2 G ks rho)
    const Fwd DKFc = kCbrtTRPI2 * c;
    const Fwd RS = DKF2RS / DKFc;
    const Fwd RTRS = fsqrt(RS);
    const Fwd EU = gcor2_fwd(0.0310907, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294, RTRS);
    const Fwd EP = gcor2_fwd(0.01554535, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517, RTRS);
    const double F = (pow(2.0, 4.0 / 3.0) - 2.0) / GAM;
    const Fwd ec = (1.0 - F) * EU + F * EP;
    const double G = 0.5 * pow(2.0, 0.6666666666666667), G3 = G * G * G;
    const Fwd DKS = fsqrt(FRDPI * DKFc);
    const Fwd T = g * (0.5 / (G * DKS)) / rho;
    const Fwd B = DELT / (-1.0 + fexp((-1.0 / (G3 * GAMMA)) * ec));
    const Fwd T2 = T * T;
    const Fwd Q4 = 1.0 + B * T2;
    const Fwd Q5 = 1.0 + B * T2 + (B * B) * (T2 * T2);
    const Fwd H = (G3 * (BET / DELT)) * flog(1.0 + DELT * (Q4 * T2) / Q5);
    return ex + rho * (ec + H);
}

// rg: rho, grad(3), Hessian xx,yy,zz,xy,xz,yz of the orbital density; returns v_xc and EXL,EXN,ECL,ECN
// densities per unit weight
// rho3: the cube root of rho
template <int GGA>
__device__ __forceinline__ void xc_point(const double *rg, double rho3, double &vxc, double *e4) {
    const double FRDPI = 1.2732395447351627;
    const double DKF2RS = 1.9191582926775128, EPS = 1.0e-20;
    const double rho = rg[0] < 0.0 ? 0.0 : rg[0];
    e4[0] = e4[1] = e4[2] = e4[3] = 0.0;
    vxc = 0.0;
    if (rho < EPS) return;
    double DG2 = 0.0, DGG = 0.0, DLP = 0.0;
    if (GGA) {
        DG2 = rg[1] * rg[1] + rg[2] * rg[2] + rg[3] * rg[3];
        DGG = rg[4] * rg[1] * rg[1] + rg[5] * rg[2] * rg[2] + rg[6] * rg[3] * rg[3] +
              2 * (rg[7] * rg[1] * rg[2] + rg[8] * rg[1] * rg[3] + rg[9] * rg[2] * rg[3]);
        DLP = rg[4] + rg[5] + rg[6];
    }
    {   // exchange of the up spin at density 2 rho
        const double D = 2.0 * rho;
        if (D > EPS) {
            const double DKF = (kCbrtTRPI2 * kCbrt2) * rho3;
            double S = 0.0, U = 0.0, V = 0.0;
            if (GGA) {
                const double DGRAD = 2.0 * sqrt(DG2);
                const double DLAP = 2.0 * DLP;
                const double REC2 = 0.5 / (DKF * D);
                const double REC1 = REC2 * D;
                const double REC22 = REC2 * REC2;
                S = DGRAD * REC2;
                V = DLAP * REC1 * REC2;
                U = DGRAD > EPS ? 8.0 * DGG * REC1 * REC22 / DGRAD : 0.0;
            }
            double EX, DEX, VX;
            if (GGA) pbeex(kCbrt2 * rho3, S, U, V, EX, DEX, VX);
            else pw91ex(DKF, S, U, V, EX, DEX, VX);
            vxc += VX;
            e4[0] += 0.5 * EX * D;
            e4[1] += 0.5 * DEX * D;
        }
    }
    {   // correlation, zeta = 1
        const double D = rho;
        const double DKF = kCbrtTRPI2 * rho3;
        const double RS = DKF2RS / DKF;
        double EC, VCUP, DEC = 0.0, DVCUP = 0.0;
        if (!GGA) {
            pw91lc_pol(RS, EC, VCUP);
        } else {
            const double DKS = sqrt(FRDPI * DKF);
            const double G = 0.5 * pow(2.0, 0.6666666666666667);
            const double DGRAD = sqrt(DG2);
            const double REC3 = 1.0 / D;
            const double REC1 = 0.5 / (DKS * G);
            const double REC2 = REC1 * REC3;
            const double REC22 = REC2 * REC2;
            const double T = DGRAD * REC2;
            const double VV = DLP * REC1 * REC2;
            const double UU = DGRAD > EPS ? DGG * REC1 * REC22 / DGRAD : 0.0;
            pbecor_pol(RS, T, UU, VV, EC, VCUP, DEC, DVCUP);
        }
        e4[2] += EC * D;
        e4[3] += DEC * D;
        vxc += VCUP + DVCUP;
    }
}

// Bound: the FP64 transcendental functions (a point reads and writes 32 bytes, PBE 144).  All powers of the density come from one
// cube root, rho^(4/3) from it and a logarithm, terms that vanish or cancel at zeta = 1 are left out, and the two
// derivatives of the PBE energy come from one forward-mode pass.  With a pow for each, three interpolations and two
// passes: LSDA 48 FLOs, 1.9e5 points 300 us; PBE 30 FLOs 426 us, 96 FLOs, 3.7e5 points 3.98 ms; now 158, 263 and 2.49.
// thread (k, f); per-block partial sums q: 0 XCH1 1 XCOU 2 XEXX 3 -sum w rho vxc 4 EXL 5 EXN 6 ECL 7 ECN
// 8 sum|V_H|
template <int GGA>
__global__ void __launch_bounds__(256) k_xc(const double *__restrict__ phi, int64_t M, int nF,
                                             const double *__restrict__ VH, int64_t ldvh,
                                             const double *__restrict__ w, double *__restrict__ Vtot,
                                             double *__restrict__ U, double *__restrict__ partial, int nblk,
                                             int blk0, double *__restrict__ Ux) {
    __shared__ double red[9][256];
    const int f = blockIdx.y;
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double q[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) q[i] = 0.0;
    if (k < M) {
        const int64_t plane = (int64_t)nF * M;
        const int64_t off = (int64_t)f * M + k;
        const double ph = phi[off];
        double rg[10];
        rg[0] = ph * ph;
        if (GGA) {
            const double gx = phi[plane + off], gy = phi[2 * plane + off], gz = phi[3 * plane + off];
            rg[1] = 2 * ph * gx;
            rg[2] = 2 * ph * gy;
            rg[3] = 2 * ph * gz;
            rg[4] = 2 * (gx * gx + phi[4 * plane + off] * ph);
            rg[5] = 2 * (gy * gy + phi[5 * plane + off] * ph);
            rg[6] = 2 * (gz * gz + phi[6 * plane + off] * ph);
            rg[7] = 2 * (gx * gy + phi[7 * plane + off] * ph);
            rg[8] = 2 * (gx * gz + phi[8 * plane + off] * ph);
            rg[9] = 2 * (gy * gz + phi[9 * plane + off] * ph);
        }
        double vxc, e4[4];
        const double rho3 = cbrt(rg[0]);
        xc_point<GGA>(rg, rho3, vxc, e4);
        const double wk = w[k];
        const double vh = VH[(int64_t)f * ldvh + k];
        const double vt = vxc + vh;
        Vtot[off] = vt;
        U[off] = wk * vt * ph;
        if (GGA && Ux) {
            // exact mesh derivative of E_xc + the Hartree term: dE/dphi = w[(e_rho + vh) phi + 2 q phi |grad phi|^2],
            // dE/d(grad phi) = w 2 q phi^2 grad phi, q = e_g / g
            double er = 0.0, qg = 0.0, g2phi = 0.0;
            const double rho = rg[0];
            if (rho >= 1.0e-20) {
                const double g = sqrt(rg[1] * rg[1] + rg[2] * rg[2] + rg[3] * rg[3]);
                const Fwd e = pbe_edens(rho, rho3, g);
                er = e.r;
                if (g > 1.0e-30) qg = e.g / g;
            }
            const int64_t plane = (int64_t)nF * M;
            double gp[3];
            for (int d = 0; d < 3; ++d) {
                gp[d] = phi[(1 + d) * plane + off];
                g2phi += gp[d] * gp[d];
            }
            Ux[off] = wk * ((er + vh) * ph + 2.0 * qg * ph * g2phi);
            for (int d = 0; d < 3; ++d) Ux[(1 + d) * plane + off] = wk * 2.0 * qg * ph * ph * gp[d];
        }
        q[0] = wk * rg[0];
        q[1] = wk * rg[0] * vh;
        {   // rho^(4/3) with the exponent in FP32 (4/3 + 4e-8), as rho rho^(1/3) e^z, z = 4e-8 ln rho (|z| < 3e-5 over the
            // normal numbers, so that z^4 / 24 is below 4e-20)
            const double z = rg[0] > 0.0 ? ((double)(4.0f / 3.0f) - 4.0 / 3.0) * log(rg[0]) : 0.0;
            q[2] = wk * (rg[0] * rho3 * (1.0 + z * (1.0 + z * (0.5 + z * (1.0 / 6.0)))));
        }
        q[3] = -wk * rg[0] * vxc;
        q[4] = e4[0] * wk;
        q[5] = e4[1] * wk;
        q[6] = e4[2] * wk;
        q[7] = e4[3] * wk;
        q[8] = fabs(vh);
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) red[i][threadIdx.x] = q[i];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
#pragma unroll
            for (int i = 0; i < 9; ++i) red[i][threadIdx.x] += red[i][threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x < 9)
        partial[((int64_t)f * nblk + blk0 + blockIdx.x) * 9 + threadIdx.x] = red[threadIdx.x][0];
}

void launch_xc(int xc, int nd, const double *phi, int64_t M, int nF, const double *VH, int64_t ldvh,
               const double *w, double *Vtot, double *U, double *partial, int nblk, int blk0, hipStream_t s,
               double *Ux) {
    const dim3 grid((unsigned)((M + 255) / 256), (unsigned)nF), blk(256);
    if (xc == 1)
        hipLaunchKernelGGL((k_xc<1>), grid, blk, 0, s, phi, M, nF, VH, ldvh, w, Vtot, U, partial, nblk, blk0, Ux);
    else
        hipLaunchKernelGGL((k_xc<0>), grid, blk, 0, s, phi, M, nF, VH, ldvh, w, Vtot, U, partial, nblk, blk0,
                           (double *)nullptr);
    (void)nd;
}

// DFT-side LSDA potential of the total spin densities (APOTNL_DFT with NSPN = 2, getvlxc.F ->
// subvlxc_libxc.F90:290-470 on the LDA path): rho_s = sum of the FLO densities of spin s (the FLOs of a spin are an
// orthonormal rotation of its occupied orbitals), V_H = sum of the FLO Hartree potentials (the potential of the total
// density), exchange per spin at 2 rho_s (PW91EX with s = u = v = 0), PW92 correlation at the point's zeta.
// pot[0, M) spin up, pot[ldpot, ldpot + M) spin down = V_H + V_xc,s; partial[block * 5 + q] = block sums of
// {E_x, E_c, E_H = 1/2 w rho V_H, N_up, N_dn} in a fixed order.
__global__ void __launch_bounds__(256) k_dft_lsda(const double *__restrict__ phi, int64_t M, int nup, int nF,
                                                  const double *__restrict__ VH, int64_t ldvh,
                                                  const double *__restrict__ w, double *__restrict__ pot, int64_t ldpot,
                                                  double *__restrict__ partial) {
    const double THIRD = 0.3333333333333333, TRPI2 = 29.6088132032680759, DKF2RS = 1.9191582926775128;
    const double EPS = 1.0e-20;
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double q[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (k < M) {
        double ru = 0.0, rd = 0.0, vh = 0.0;
        for (int f = 0; f < nF; ++f) {
            const double p = phi[(int64_t)f * M + k];
            if (f < nup)
                ru += p * p;
            else
                rd += p * p;
            vh += VH[(int64_t)f * ldvh + k];
        }
        const double D = ru + rd;
        double vxu = 0.0, vxd = 0.0, vcu = 0.0, vcd = 0.0, ex = 0.0, ec = 0.0;
        if (D >= EPS) {
            for (int sp = 0; sp < 2; ++sp) {
                const double Ds = 2.0 * (sp == 0 ? ru : rd);
                if (Ds > EPS) {
                    double EX, DEX, VX;
                    pw91ex(pow(TRPI2 * Ds, THIRD), 0.0, 0.0, 0.0, EX, DEX, VX);
                    (sp == 0 ? vxu : vxd) = VX;
                    ex += 0.5 * EX * Ds;
                }
            }
            double EC;
            pw91lc_gen(DKF2RS / pow(TRPI2 * D, THIRD), (ru - rd) / D, EC, vcu, vcd);
            ec = EC * D;
        }
        pot[k] = vh + vxu + vcu;
        pot[ldpot + k] = vh + vxd + vcd;
        const double wk = w[k];
        q[0] = wk * ex;
        q[1] = wk * ec;
        q[2] = 0.5 * wk * D * vh;
        q[3] = wk * ru;
        q[4] = wk * rd;
    }
    __shared__ double red[5][256];
#pragma unroll
    for (int i = 0; i < 5; ++i) red[i][threadIdx.x] = q[i];
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h)
#pragma unroll
            for (int i = 0; i < 5; ++i) red[i][threadIdx.x] += red[i][threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x < 5) partial[(int64_t)blockIdx.x * 5 + threadIdx.x] = red[threadIdx.x][0];
}

void launch_dft_lsda(const double *phi, int64_t M, int nup, int nF, const double *VH, int64_t ldvh, const double *w,
                     double *pot, int64_t ldpot, double *partial, hipStream_t s) {
    if (M <= 0) return;
    hipLaunchKernelGGL(k_dft_lsda, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, s, phi, M, nup, nF, VH, ldvh, w,
                       pot, ldpot, partial);
}

// PBE correlation at general zeta (pbecor.f, LGGA = LPOT = 1): EC, VCUP, VCDN, H, DVCUP, DVCDN
__device__ __forceinline__ void pbecor_gen(double RS, double ZET, double T, double UU, double VV, double WW, double &EC,
                                           double &VCUP, double &VCDN, double &H, double &DVCUP, double &DVCDN) {
    const double THRD = 1.0 / 3.0, THRD2 = 2.0 * THRD, THRD4 = 4.0 * THRD, SIXTHM = -THRD / 2.0;
    const double GAM = 0.5198420997897463295344212145565, FZZ = 8.0 / (9.0 * GAM);
    const double GAMMA = 0.03109069086965489503494086371273, BET = 0.06672455060314922, DELT = BET / GAMMA;
    const double ETA = 1.0e-12;
    const double RTRS = sqrt(RS);
    double EU, EURS, EP, EPRS, ALFM, ALFRSM;
    gcor2(0.0310907, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294, RTRS, EU, EURS);
    gcor2(0.01554535, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517, RTRS, EP, EPRS);
    gcor2(0.0168869, 0.11125, 10.357, 3.6231, 0.88026, 0.49671, RTRS, ALFM, ALFRSM);
    const double Z3 = ZET * ZET * ZET, Z4 = Z3 * ZET;
    const double F = (pow(1.0 + ZET, THRD4) + pow(1.0 - ZET, THRD4) - 2.0) / GAM;
    const double ec = EU * (1.0 - F * Z4) + EP * F * Z4 - ALFM * F * (1.0 - Z4) / FZZ;
    const double ECRS = EURS * (1.0 - F * Z4) + EPRS * F * Z4 - ALFRSM * F * (1.0 - Z4) / FZZ;
    const double FZ = THRD4 * (pow(1.0 + ZET, THRD) - pow(1.0 - ZET, THRD)) / GAM;
    const double ECZET = 4.0 * Z3 * F * (EP - EU + ALFM / FZZ) + FZ * (Z4 * EP - Z4 * EU - (1.0 - Z4) * ALFM / FZZ);
    const double COMM0 = ec - RS * ECRS / 3.0 - ZET * ECZET;
    EC = ec;
    VCUP = COMM0 + ECZET;
    VCDN = COMM0 - ECZET;
    const double G = (pow(1.0 + ZET, THRD2) + pow(1.0 - ZET, THRD2)) / 2.0;
    const double G3 = G * G * G;
    const double PON = -ec / (G3 * GAMMA);
    const double B = DELT / (exp(PON) - 1.0);
    const double B2 = B * B, T2 = T * T, T4 = T2 * T2;
    const double Q4 = 1.0 + B * T2;
    const double Q5 = 1.0 + B * T2 + B2 * T4;
    const double h = G3 * (BET / DELT) * log(1.0 + DELT * Q4 * T2 / Q5);
    const double G4 = G3 * G, T6 = T4 * T2, RSTHRD = RS / 3.0;
    const double GZ = (pow((1.0 + ZET) * (1.0 + ZET) + ETA, SIXTHM) - pow((1.0 - ZET) * (1.0 - ZET) + ETA, SIXTHM)) / 3.0;
    const double FAC = DELT / B + 1.0;
    const double BG = -3.0 * B2 * ec * FAC / (BET * G4);
    const double BEC = B2 * FAC / (BET * G3);
    const double Q8 = Q5 * Q5 + DELT * Q4 * Q5 * T2;
    const double Q9 = 1.0 + 2.0 * B * T2;
    const double HB = -BET * G3 * B * T6 * (2.0 + B * T2) / Q8;
    const double HRS = -RSTHRD * HB * BEC * ECRS;
    const double FACT0 = 2.0 * DELT - 6.0 * B;
    const double FACT1 = Q5 * Q9 + Q4 * Q9 * Q9;
    const double HBT = 2.0 * BET * G3 * T4 * ((Q4 * Q5 * FACT0 - DELT * FACT1) / Q8) / Q8;
    const double HRST = RSTHRD * T2 * HBT * BEC * ECRS;
    const double HZ = 3.0 * GZ * h / G + HB * (BG * GZ + BEC * ECZET);
    const double HT = 2.0 * BET * G3 * Q9 / Q8;
    const double HZT = 3.0 * GZ * HT / G + HBT * (BG * GZ + BEC * ECZET);
    const double FACT2 = Q4 * Q5 + B * T2 * (Q4 * Q9 + Q5);
    const double FACT3 = 2.0 * B * Q5 * Q9 + DELT * FACT2;
    const double HTT = 4.0 * BET * G3 * T * (2.0 * B / Q8 - (Q9 * FACT3 / Q8) / Q8);
    double comm = h + HRS + HRST + T2 * HT / 6.0 + 7.0 * T2 * T * HTT / 6.0;
    const double PREF = HZ - GZ * T2 * HT / G;
    const double FACT5 = GZ * (2.0 * HT + T * HTT) / G;
    comm = comm - PREF * ZET - UU * HTT - VV * HT - WW * (HZT - FACT5);
    H = h;
    DVCUP = comm + PREF;
    DVCDN = comm - PREF;
}

// |grad|^2, grad.H.grad and the Laplacian of a 10-component density (value, gradient, xx,yy,zz,xy,xz,yz)
__device__ __forceinline__ void gga_invariants(const double *r, double &dg2, double &dgg, double &dlp) {
    dg2 = r[1] * r[1] + r[2] * r[2] + r[3] * r[3];
    dgg = r[4] * r[1] * r[1] + r[5] * r[2] * r[2] + r[6] * r[3] * r[3] +
          2 * (r[7] * r[1] * r[2] + r[8] * r[1] * r[3] + r[9] * r[2] * r[3]);
    dlp = r[4] + r[5] + r[6];
}

// DFT-side PBE potential of the total spin densities (APOTNL_DFT with NSPN = 2 and IGGA = 1: SUBVLXC as the program links it, subvlxc_libxc.F90:197-470; subvlxc.F:138-323 has the same non-libxc branch): per
// point the value, gradient and Hessian of rho_up and rho_dn from the FLO planes (rho = sum phi^2,
// grad rho = 2 sum phi grad phi, H = 2 sum (grad phi grad phi^T + phi H phi)); the total and down densities clipped
// as there; exchange per spin at D = 2 rho_s (PBEEX with s, u, v of 2 rho_s), PBE correlation at the point's zeta with
// t, uu, vv of the total density and the zeta-gradient term ww.  phi: 10 planes of [nF][M]; pot and partial as in
// k_dft_lsda (E_x = EXL + EXN, E_c = ECL + ECN).
__global__ void __launch_bounds__(256) k_dft_gga(const double *__restrict__ phi, int64_t M, int nup, int nF,
                                                 const double *__restrict__ VH, int64_t ldvh,
                                                 const double *__restrict__ w, double *__restrict__ pot, int64_t ldpot,
                                                 double *__restrict__ partial) {
    const double THIRD = 0.3333333333333333, THIRD2 = 0.6666666666666667;
    const double TRPI2 = 29.6088132032680759, FRDPI = 1.2732395447351627, DKF2RS = 1.9191582926775128;
    const double EPS = 1.0e-20;
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double q[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (k < M) {
        const int64_t plane = (int64_t)nF * M;
        double ru[10], rd[10], vh = 0.0;
#pragma unroll
        for (int i = 0; i < 10; ++i) ru[i] = rd[i] = 0.0;
        for (int f = 0; f < nF; ++f) {
            const int64_t off = (int64_t)f * M + k;
            const double ph = phi[off];
            const double gx = phi[plane + off], gy = phi[2 * plane + off], gz = phi[3 * plane + off];
            double *r = f < nup ? ru : rd;
            r[0] += ph * ph;
            r[1] += 2 * ph * gx;
            r[2] += 2 * ph * gy;
            r[3] += 2 * ph * gz;
            r[4] += 2 * (gx * gx + phi[4 * plane + off] * ph);
            r[5] += 2 * (gy * gy + phi[5 * plane + off] * ph);
            r[6] += 2 * (gz * gz + phi[6 * plane + off] * ph);
            r[7] += 2 * (gx * gy + phi[7 * plane + off] * ph);
            r[8] += 2 * (gx * gz + phi[8 * plane + off] * ph);
            r[9] += 2 * (gy * gz + phi[9 * plane + off] * ph);
            vh += VH[(int64_t)f * ldvh + k];
        }
        // RHT(:,1) = total, RHT(:,2) = down, values clipped to [0, total]; the up components are their difference
        double R1[10], R2[10], RU[10];
#pragma unroll
        for (int i = 0; i < 10; ++i) {
            R1[i] = ru[i] + rd[i];
            R2[i] = rd[i];
        }
        if (R1[0] < 0.0) R1[0] = 0.0;
        if (R2[0] < 0.0) R2[0] = 0.0;
        if (R2[0] > R1[0]) R2[0] = R1[0];
#pragma unroll
        for (int i = 0; i < 10; ++i) RU[i] = R1[i] - R2[i];
        const double DEN1 = R1[0], DEN3 = R2[0], DEN2 = DEN1 - DEN3;
        double DG2[3], DGG[3], DLP[3];
        gga_invariants(R1, DG2[0], DGG[0], DLP[0]);
        gga_invariants(RU, DG2[1], DGG[1], DLP[1]);
        gga_invariants(R2, DG2[2], DGG[2], DLP[2]);
        double v[2] = {0.0, 0.0}, ex = 0.0, ec = 0.0;
        if (DEN1 >= EPS) {
            for (int sp = 0; sp < 2; ++sp) {
                const double D = 2.0 * (sp == 0 ? DEN2 : DEN3);
                if (!(D > EPS)) continue;
                const double DKF = pow(TRPI2 * D, THIRD);
                const double DGRAD = 2.0 * sqrt(DG2[sp + 1]), DLAP = 2.0 * DLP[sp + 1];
                const double REC2 = 0.5 / (DKF * D), REC1 = REC2 * D, REC22 = REC2 * REC2;
                const double S = DGRAD * REC2, V = DLAP * REC1 * REC2;
                const double U = DGRAD > EPS ? 8.0 * DGG[sp + 1] * REC1 * REC22 / DGRAD : 0.0;
                double EX, DEX, VX;
                pbeex(pow(D, THIRD), S, U, V, EX, DEX, VX);
                v[sp] += VX;
                ex += 0.5 * (EX + DEX) * D;
            }
            const double D = DEN1, DREC = 1.0 / D, ZET = (DEN2 - DEN3) * DREC;
            const double DKF = pow(TRPI2 * D, THIRD), DKS = sqrt(FRDPI * DKF), RS = DKF2RS / DKF;
            double G = 0.5 * (pow(1.0 + ZET, THIRD2) + pow(1.0 - ZET, THIRD2));
            if (ZET == 1.0 || ZET == -1.0) G = 0.5 * pow(2.0, THIRD2);
            const double DGRAD = sqrt(DG2[0]);
            const double REC3 = DREC, REC1 = 0.5 / (DKS * G), REC2 = REC1 * REC3, REC22 = REC2 * REC2;
            const double T = DGRAD * REC2, VV = DLP[0] * REC1 * REC2;
            const double WW = (D * (DG2[1] - DG2[2]) - (DEN2 - DEN3) * DG2[0]) * REC3 * REC22;
            const double UU = DGRAD > EPS ? DGG[0] * REC1 * REC22 / DGRAD : 0.0;
            double EC, VCUP, VCDN, DEC, DVCUP, DVCDN;
            pbecor_gen(RS, ZET, T, UU, VV, WW, EC, VCUP, VCDN, DEC, DVCUP, DVCDN);
            ec = (EC + DEC) * D;
            v[0] += VCUP + DVCUP;
            v[1] += VCDN + DVCDN;
        }
        pot[k] = vh + v[0];
        pot[ldpot + k] = vh + v[1];
        const double wk = w[k];
        q[0] = wk * ex;
        q[1] = wk * ec;
        q[2] = 0.5 * wk * DEN1 * vh;
        q[3] = wk * DEN2;
        q[4] = wk * DEN3;
    }
    __shared__ double red[5][256];
#pragma unroll
    for (int i = 0; i < 5; ++i) red[i][threadIdx.x] = q[i];
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h)
#pragma unroll
            for (int i = 0; i < 5; ++i) red[i][threadIdx.x] += red[i][threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x < 5) partial[(int64_t)blockIdx.x * 5 + threadIdx.x] = red[threadIdx.x][0];
}

void launch_dft_gga(const double *phi, int64_t M, int nup, int nF, const double *VH, int64_t ldvh, const double *w,
                    double *pot, int64_t ldpot, double *partial, hipStream_t s) {
    if (M <= 0) return;
    hipLaunchKernelGGL(k_dft_gga, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, s, phi, M, nup, nF, VH, ldvh, w,
                       pot, ldpot, partial);
}

// out[q] = sum over b in increasing order of part[b * nq + q]: the host's block-order sum, on one thread (the same
// additions in the same order, so the same bits).
__global__ void k_sum_partials_ordered(const double *__restrict__ part, int nblk, int nq, double *__restrict__ out) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    for (int q = 0; q < nq; ++q) {
        double s = 0.0;
        for (int b = 0; b < nblk; ++b) s += part[(int64_t)b * nq + q];
        out[q] = s;
    }
}
void launch_sum_partials_ordered(const double *part, int nblk, int nq, double *out, hipStream_t s) {
    hipLaunchKernelGGL(k_sum_partials_ordered, dim3(1), dim3(64), 0, s, part, nblk, nq, out);
}

__global__ void k_fill_zero(double *__restrict__ p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0.0;
}
void launch_fill_zero(double *p, size_t n, hipStream_t s) {
    if (n == 0) return;
    const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 8192);
    hipLaunchKernelGGL(k_fill_zero, dim3(blocks), dim3(256), 0, s, p, (int64_t)n);
}

__global__ void k_gather(const double *__restrict__ src, int64_t stride, int n, double *__restrict__ dst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[(int64_t)i * stride];
}
void launch_gather(const double *src, int64_t stride, int n, double *dst, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_gather, dim3((n + 255) / 256), dim3(256), 0, s, src, stride, n, dst);
}

// Deterministic compensated (Neumaier) reduction of per-block partials, out[f][q] = sum_b partial[f][b][q]; with accumulate
// the sum starts from out.  Two shapes:
// k_reduce_partials, few outputs: bound by the latency of the loads, so 16 waves share the partials of 64 outputs (consecutive
// ranges of b, eight loads in flight) and their sums are added in order, compensated again.  One thread per output, one
// load after the other, took 22 us at 90 outputs of 132 partials (10 FLOs, 3.4e4 points), 62 at 30 FLOs (1.2e5 points) and
// 188 at 96 FLOs (3.7e5 points), each an average over the sums of a pass; now 4.2, 6.0 and 14.7.
// k_reduce_many, many outputs (those of V^i_ab, n^3, and of the products over a block of the mesh, with few partials each):
// bound by memory, a thread per output, four loads in flight, no LDS.  16 waves per 64 outputs, most of them without a
// partial, took 117 us at 1.7e6 outputs (n = 120) of 8 partials, here 25 (5.5 TB/s); at 1e6 of 2 57 and 5.6.
// The limit (us, 16 waves and one thread): 2 partials of 1.6e4 outputs 2.8 and 2.7, of 6.4e4 5.2 and 2.4; 8 of 1.6e4 3.0 and
// 2.7, of 6.4e4 5.4 and 3.6; 32 of 6.4e4 6.5 and 6.7, of 2.5e5 26 and 13; 128 of 6.4e4 14 and 27, of 2.5e5 48 and 43; 1024
// of 1.6e4 25 and 180, of 2.5e5 336 and 325: one thread from 2048 outputs per partial or 2^17 outputs on.
constexpr int kRedWaves = 16;
__device__ __forceinline__ void neumaier(double x, double &s, double &c) {
    const double t = s + x;
    c += fabs(s) >= fabs(x) ? (s - t) + x : (x - t) + s;
    s = t;
}
__global__ void __launch_bounds__(256) k_reduce_many(const double *__restrict__ partial, int n, int nblk, int nq,
                                                     double *__restrict__ out, int accumulate) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int f = i / nq;
    const double *p = partial + (int64_t)f * nblk * nq + i - f * nq;
    double s = accumulate ? out[i] : 0.0, c = 0.0;
    for (int b = 0; b < nblk; b += 4, p += (int64_t)4 * nq) {
        double x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (b + j < nblk) x[j] = p[(int64_t)j * nq];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (b + j < nblk) neumaier(x[j], s, c);
    }
    out[i] = s + c;
}
__global__ void __launch_bounds__(64 * kRedWaves) k_reduce_partials(const double *__restrict__ partial, int n, int nblk,
                                                                    int nq, double *__restrict__ out, int accumulate) {
    __shared__ double S[kRedWaves][64], Cs[kRedWaves][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = blockIdx.x * 64 + lane;
    double s = 0.0, c = 0.0;
    if (i < n) {
        const int b0 = (int)((int64_t)nblk * wave / kRedWaves), b1 = (int)((int64_t)nblk * (wave + 1) / kRedWaves);
        const int f = i / nq;
        const double *p = partial + ((int64_t)f * nblk + b0) * nq + i - f * nq;
        int b = b0;
        for (; b + 8 <= b1; b += 8) {
            double x[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = p[(int64_t)j * nq];
            p += (int64_t)8 * nq;
#pragma unroll
            for (int j = 0; j < 8; ++j) neumaier(x[j], s, c);
        }
        for (; b < b1; ++b, p += nq) neumaier(*p, s, c);
    }
    S[wave][lane] = s;
    Cs[wave][lane] = c;
    __syncthreads();
    if (wave == 0 && i < n) {
        s = accumulate ? out[i] : 0.0;
        c = 0.0;
#pragma unroll
        for (int g = 0; g < kRedWaves; ++g) {
            neumaier(S[g][lane], s, c);
            c += Cs[g][lane];
        }
        out[i] = s + c;
    }
}

void launch_reduce_partials(const double *partial, int nF, int nblk, int nq, double *out, hipStream_t s,
                            bool accumulate) {
    const int n = nF * nq;
    if (n <= 0) return;
    if (n >= std::min<int64_t>(1 << 17, (int64_t)2048 * nblk)) {
        hipLaunchKernelGGL(k_reduce_many, dim3((unsigned)(((int64_t)n + 255) / 256)), dim3(256), 0, s, partial, n, nblk, nq, out,
                           accumulate ? 1 : 0);
        return;
    }
    hipLaunchKernelGGL(k_reduce_partials, dim3((n + 63) / 64), dim3(64 * kRedWaves), 0, s, partial, n, nblk, nq, out,
                       accumulate ? 1 : 0);
}

// ---------------------------------------------------------------------------------------------------
// V^i_ab = sum_k Vtot_i(k) [w phi_a phi_b](k): a GEMM over the points with the pair-product operand generated in
// registers.  Block (pair block, point slice, i block): pair block = 8 a x 8 b with a-block <= b-block (V is
// symmetric in a,b; the mirror is stored too), 4 wavefronts, wave w takes a = 8A + 2w + {0,1} and all 8 b, i.e.
// 16 pair columns, against up to 16*NIT i rows.  Points are staged 32 at a time; 16x16x4 FP64 MFMAs, or FP32
// MFMAs (operands rounded to FP32, FP32 accumulation over each 32 staged points, FP64 sums).  Partial sums per
// slice: part[slice][i][b][a].
// ---------------------------------------------------------------------------------------------------
constexpr int kVabKS = 32;

template <typename T, int NIT>
__global__ void __launch_bounds__(256) k_vab_mfma(const double *__restrict__ phi, const double *__restrict__ Vt,
                                                  const double *__restrict__ w, int64_t M, int n, int nb8,
                                                  int64_t kslice, double *__restrict__ part) {
    constexpr int NI = 16 * NIT, LDV = kVabKS + 1;
    using Tr = MfmaTraits<T>;
    __shared__ T Vl[NI * LDV];
    __shared__ double Pa[8 * LDV], Pb[8 * LDV], Wl[kVabKS];
    // pair block index -> (A, B), A <= B, row-major over the upper triangle
    int A = 0, rem = blockIdx.x;
    while (rem >= nb8 - A) {
        rem -= nb8 - A;
        ++A;
    }
    const int B = A + rem;
    const int s = blockIdx.y, i0 = blockIdx.z * NI;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane >> 4, lc = lane & 15;
    const int la = 2 * wave + (lc >> 3), lb = lc & 7;  // this lane's pair inside the 8x8 block
    const int64_t kb = (int64_t)s * kslice, ke = min(M, kb + kslice);
    typename Tr::acc acc[NIT];
    double sum[NIT][4];  // FP32 form: the FP32 accumulators of every 32 staged points are added here
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            acc[it][r] = (T)0;
            sum[it][r] = 0.0;
        }
    // the 32 points of the next step are loaded into registers while the MFMAs consume the current step from LDS
    constexpr int NV = NI * kVabKS / 256, NP = 16 * kVabKS / 256;
    double rv[NV], rp[NP], rw = 0.0;
    auto load = [&](int64_t t0) {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int e = threadIdx.x + 256 * j, i = e / kVabKS, kk = e - i * kVabKS;
            const int64_t k = t0 + kk;
            rv[j] = (i0 + i < n && k < ke) ? Vt[(int64_t)(i0 + i) * M + k] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int e = threadIdx.x + 256 * j, r = e / kVabKS, kk = e - r * kVabKS;
            const int64_t k = t0 + kk;
            const int f = r < 8 ? 8 * A + r : 8 * B + r - 8;
            rp[j] = (f < n && k < ke) ? phi[(int64_t)f * M + k] : 0.0;
        }
        if (threadIdx.x < kVabKS) rw = t0 + threadIdx.x < ke ? w[t0 + threadIdx.x] : 0.0;
    };
    auto store = [&]() {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int e = threadIdx.x + 256 * j, i = e / kVabKS, kk = e - i * kVabKS;
            Vl[i * LDV + kk] = (T)rv[j];
        }
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int e = threadIdx.x + 256 * j, r = e / kVabKS, kk = e - r * kVabKS;
            if (r < 8)
                Pa[r * LDV + kk] = rp[j];
            else
                Pb[(r - 8) * LDV + kk] = rp[j];
        }
        if (threadIdx.x < kVabKS) Wl[threadIdx.x] = rw;
    };
    load(kb);
    store();
    __syncthreads();
    for (int64_t t0 = kb; t0 < ke; t0 += kVabKS) {
        const bool more = t0 + kVabKS < ke;  // uniform over the block
        if (more) load(t0 + kVabKS);
#pragma unroll
        for (int ks = 0; ks < kVabKS; ks += 4) {
            const int kk = ks + lr;
            const T bv = (T)(Wl[kk] * Pa[la * LDV + kk] * Pb[lb * LDV + kk]);
#pragma unroll
            for (int it = 0; it < NIT; ++it) acc[it] = Tr::mma(Vl[(it * 16 + lc) * LDV + kk], bv, acc[it]);
        }
        if (sizeof(T) == 4) {
#pragma unroll
            for (int it = 0; it < NIT; ++it)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    sum[it][r] += (double)acc[it][r];
                    acc[it][r] = (T)0;
                }
        }
        __syncthreads();
        if (more) store();
        __syncthreads();
    }
    const int a = 8 * A + 2 * wave + (lc >> 3), b = 8 * B + (lc & 7);
    if (a >= n || b >= n) return;
    const int64_t nn = (int64_t)n * n, base = (int64_t)s * n * nn;
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = i0 + it * 16 + Tr::row(lr, r);
            if (i >= n) continue;
            const double v = sizeof(T) == 4 ? sum[it][r] : (double)acc[it][r];
            part[base + i * nn + (int64_t)b * n + a] = v;
            if (A != B) part[base + i * nn + (int64_t)a * n + b] = v;
        }
}

// Point slices: at least 64 where they have 1024 points each; for few FLOs, whose pair blocks are few, as many as give 1024
// blocks in all, of at least 256 points (eight staged steps).  With 64 at most, 10 FLOs (one pair block per spin, 3.4e4
// points) took 24 us per spin, 48 FLOs in FP32 (six, 1.9e5 points) 118; now 8.7 and 80.
int vab_slices(int64_t M, int n) {
    int s = 64;
    while (s > 1 && M / s < 1024) --s;
    const int64_t nb8 = (n + 7) / 8, per_slice = nb8 * (nb8 + 1) / 2 * ((n + 127) / 128);
    const int64_t more = std::min<int64_t>(1024 / std::max<int64_t>(1, per_slice), M / 256);
    return (int)std::max<int64_t>(s, more);
}

void launch_vab(const double *phi0, const double *Vtot, const double *w, int64_t M, int n, int nslice, double *part,
                hipStream_t s, bool fp32) {
    if (n <= 0) return;
    const int nb8 = (n + 7) / 8;
    const int64_t kslice = ((M + nslice - 1) / nslice + kVabKS - 1) / kVabKS * kVabKS;
    const int nit = std::min(8, (n + 15) / 16);
    const dim3 grid((unsigned)(nb8 * (nb8 + 1) / 2), (unsigned)nslice, (unsigned)((n + 16 * nit - 1) / (16 * nit)));
#define FLOSIC_VAB(NIT)                                                                                         \
    if (fp32)                                                                                                   \
        hipLaunchKernelGGL((k_vab_mfma<float, NIT>), grid, dim3(256), 0, s, phi0, Vtot, w, M, n, nb8, kslice, part); \
    else                                                                                                        \
        hipLaunchKernelGGL((k_vab_mfma<double, NIT>), grid, dim3(256), 0, s, phi0, Vtot, w, M, n, nb8, kslice, part)
    switch (nit) {
        case 1: FLOSIC_VAB(1); break;
        case 2: FLOSIC_VAB(2); break;
        case 3: FLOSIC_VAB(3); break;
        case 4: FLOSIC_VAB(4); break;
        case 5: FLOSIC_VAB(5); break;
        case 6: FLOSIC_VAB(6); break;
        case 7: FLOSIC_VAB(7); break;
        default: FLOSIC_VAB(8); break;
    }
#undef FLOSIC_VAB
}

// ---------------------------------------------------------------------------------------------------
// host: Boys table (fffmt3.F:24-65): F_19 by its series, downward recursion, F_0..F_7 kept
// ---------------------------------------------------------------------------------------------------
void boys_table(double *tab) {
    // rows 0 .. kBoysRows-1 in FP64, followed by the same table rounded to FP32
    float *tab32 = (float *)(tab + kBoysRows * kBoysCols);
    for (int i = 0; i < kBoysCols; ++i) tab[i] = 1.0 / (2 * (i + 1) - 1);
    for (int L = 2; L <= kBoysRows; ++L) {
        const double T = 1.0e-2 * (L - 1);
        const double X = 2 * T;
        double den = 39.0, term = 1.0 / den, sum = term;
        for (int i = 2; i <= 100; ++i) {
            den += 2.0;
            term = term * X / den;
            sum = sum + term;
            if (term / sum - 1.0e-12 <= 0) break;
        }
        const double ex = exp(-T);
        double G[21];
        G[20] = ex * sum;
        for (int i = 1; i <= 19; ++i) {
            const int kk = 20 - i;
            G[kk] = (X * G[kk + 1] + ex) / (2 * kk - 1);
        }
        for (int i = 0; i < kBoysCols; ++i) tab[(L - 1) * kBoysCols + i] = G[i + 1];
    }
    for (int i = 0; i < kBoysRows * kBoysCols; ++i) tab32[i] = (float)tab[i];
}

}  // namespace flosic
