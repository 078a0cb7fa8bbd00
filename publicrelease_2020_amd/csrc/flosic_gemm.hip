// FP64 MFMA products over the mesh: orbitals on points (points x functions times functions x orbitals) and sums over the
// points (A^T B).  Both have one huge and two small dimensions, which a general library GEMM pads to 64 or 128 columns
// and, for A^T B, spreads over too few blocks.  Operands go from global memory to registers in MFMA operand order, with
// no LDS: a lane loads four consecutive elements (32 bytes) along the contiguous dimension and the four K steps (or the
// four row tiles) that they belong to are numbered so that every lane's four are its own.
#include "flosic_device.h"

namespace flosic {

// four consecutive doubles at any 8-byte aligned address (leading dimensions are mesh sizes, odd ones among them)
typedef double v4du __attribute__((ext_vector_type(4), aligned(8)));
typedef double v2du __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ v2du load2(const double *p) { return *(const __attribute__((address_space(1))) v2du *)p; }
__device__ __forceinline__ v4du load4(const double *p) { return *(const __attribute__((address_space(1))) v4du *)p; }
// the same with every index clamped to [0, n)
__device__ __forceinline__ v4du load4c(const double *p, int64_t i, int64_t n) {
    v4du d;
#pragma unroll
    for (int e = 0; e < 4; ++e) d[e] = gload(p + min(i + e, n - 1));
    return d;
}

// ---------------------------------------------------------------------------------------------------
// phi[d][f][k] = sum_mu planes[d][mu][k] cf[mu + N f], k < m points, f < nc orbitals, d planes (blockIdx.z).
// Wave: 64 points x CB tiles of 16 orbitals; block: 4 waves, the CW = 4 / PW that share 64 points holding different
// orbitals.  Function block of 16: K step s of lane group lr is function 16 b + 4 lr + s; point tile i, row r is point
// 4 r + i.  Bound: 2 m N nc / 77 TFLOP/s of FP64 MFMA or the 8 m N bytes of the planes, whichever is longer (equal
// near 45 orbitals).  Measured against the library's product (128 x 128 tiles): 128 functions x 20 orbitals, 69 773 points
// 62 -> 29 us; 500 x 48, 185 742 0.42 -> 0.22 ms (planes at 3.3 TB/s); 260 x 30, 116 200 points, 10 planes 1.48 -> 0.61;
// 916 x 96, 370 513, 10 planes 13.8 -> 11.4 (57 TFLOP/s); 1720 x 192, 368 437 4.7 -> 4.0 (61 TFLOP/s).
// ---------------------------------------------------------------------------------------------------
template <int CB, bool TAIL>
__device__ __forceinline__ void phi_load(const double *pl, int64_t m, int64_t k, int N, const double *cf, int nc, int f0,
                                         int mu0, int lr, int lc, double (&a)[4][4], double (&b)[CB][4]) {
    const bool whole = mu0 + 16 <= N;  // uniform
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int mu = mu0 + 4 * lr + s;
        const double *row = pl + (int64_t)(whole ? mu : min(mu, N - 1)) * m;
        const v4du x = TAIL ? load4c(row, k, m) : load4(row + k);
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i][s] = x[i];
    }
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        const double *col = cf + (int64_t)min(f0 + 16 * j + lc, nc - 1) * N;
        if (whole) {
            const v4du x = load4(col + mu0 + 4 * lr);
#pragma unroll
            for (int s = 0; s < 4; ++s) b[j][s] = x[s];
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int mu = mu0 + 4 * lr + s;
                const double x = gload(col + min(mu, N - 1));
                b[j][s] = mu < N ? x : 0.0;
            }
        }
    }
}

template <int CB, bool TAIL>
__device__ __forceinline__ void phi_wave(const double *__restrict__ pl, int64_t m, int64_t k0, int N,
                                         const double *__restrict__ cf, int nc, int f0, double *__restrict__ out) {
    const int lane = threadIdx.x & 63, lr = lane >> 4, lc = lane & 15;
    v4d acc[4][CB];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i][j] = (v4d){0.0, 0.0, 0.0, 0.0};
    double a[2][4][4], b[2][CB][4];
    const int64_t k = k0 + 4 * lc;
    phi_load<CB, TAIL>(pl, m, k, N, cf, nc, f0, 0, lr, lc, a[0], b[0]);
    for (int mu0 = 0; mu0 < N; mu0 += 32) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int cur = mu0 + 16 * h;
            if (cur < N) {
                if (cur + 16 < N) phi_load<CB, TAIL>(pl, m, k, N, cf, nc, f0, cur + 16, lr, lc, a[h ^ 1], b[h ^ 1]);
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int j = 0; j < CB; ++j)
                            acc[i][j] = MfmaTraits<double>::mma(a[h][i][s], b[h][j][s], acc[i][j]);
            }
        }
    }
    // register r of tile i: point 4 (lr + 4 r) + i of orbital column lc
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        const int f = f0 + 16 * j + lc;
        if (f < nc) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t p = k0 + 4 * (lr + 4 * r);
                double *o = out + (int64_t)f * m + p;
                if (!TAIL) {
                    v4du x;
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[i] = acc[i][j][r];
                    *(__attribute__((address_space(1))) v4du *)o = x;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (p + i < m) gstore(o + i, acc[i][j][r]);
                }
            }
        }
    }
}

template <int CB>
__global__ void __launch_bounds__(256, 2) k_orbitals(const double *__restrict__ planes, int64_t m, int N,
                                                     const double *__restrict__ cf, int nc, int cw,
                                                     double *__restrict__ phi) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t k0 = ((int64_t)blockIdx.x * (4 / cw) + wave / cw) * 64;
    const int f0 = (blockIdx.y * cw + wave % cw) * 16 * CB;
    if (k0 >= m || f0 >= nc) return;
    const double *pl = planes + (int64_t)blockIdx.z * N * m;
    double *out = phi + (int64_t)blockIdx.z * nc * m;
    if (k0 + 64 <= m) phi_wave<CB, false>(pl, m, k0, N, cf, nc, f0, out);
    else phi_wave<CB, true>(pl, m, k0, N, cf, nc, f0, out);
}

void launch_orbitals(const double *planes, int64_t m, int nd, int N, const double *cf, int nc, double *phi,
                     hipStream_t s) {
    if (m <= 0 || nc <= 0 || nd <= 0) return;
    const int ct = (nc + 15) / 16, ng = (ct + 2) / 3, cb = (ct + ng - 1) / ng;  // ng column groups of cb <= 3 tiles
    const int cw = ng >= 3 ? 4 : ng;
    const int64_t tiles = (m + 63) / 64, pw = 4 / cw;
    const dim3 grid((unsigned)((tiles + pw - 1) / pw), (unsigned)((ng + cw - 1) / cw), (unsigned)nd), blk(256);
    switch (cb) {
        case 1: hipLaunchKernelGGL((k_orbitals<1>), grid, blk, 0, s, planes, m, N, cf, nc, cw, phi); break;
        case 2: hipLaunchKernelGGL((k_orbitals<2>), grid, blk, 0, s, planes, m, N, cf, nc, cw, phi); break;
        default: hipLaunchKernelGGL((k_orbitals<3>), grid, blk, 0, s, planes, m, N, cf, nc, cw, phi); break;
    }
}

// ---------------------------------------------------------------------------------------------------
// part[slice][r + rows c] = sum over the slice's points of A[k + lda r] B[k + ldb c], planes p = slice / nsl of A and B
// (strides sa, sb) one after the other.  Wave: RA row tiles x CB column tiles of 16; the 4 waves of a block take
// quarters of the slice and add up through LDS.  Point block of 16: K steps 0, 1 of lane group lr are points 2 lr and
// 2 lr + 1, steps 2, 3 points 8 + 2 lr and 9 + 2 lr, so that each load takes 64 contiguous bytes of 16 rows.
// Bound: 2 rows n M / 77 TFLOP/s or 8 (rows + n) M bytes.  Blocks go to the 8 XCDs round robin, and a slice's tiles (which
// read the same points) are numbered 8 apart: they meet in one XCD's L2.  Measured with the final sum, against the
// library's product batched over point slices of at least 4096: 12 x 10, 11 640 points 320 -> 19 us; 128 x 20, 69 773
// 236 -> 58 us; 260 x 30 and four 15 x 15 planes per spin, 116 200 2.12 -> 0.45 ms; equal at 500 x 48 (0.27 -> 0.29 ms).
// Which of the two takes a product: tn_by_library.
// ---------------------------------------------------------------------------------------------------
// k: the first of this lane's points (2 lr into the block)
template <int NT, bool TAIL>
__device__ __forceinline__ void tn_load(const double *X, int64_t ld, int nx, int x0, int64_t k, int64_t kend, int64_t M,
                                        bool zero, int lc, double (&v)[NT][4]) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const double *row = X + (int64_t)min(x0 + 16 * t + lc, nx - 1) * ld;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if constexpr (!TAIL) {
                const v2du x = load2(row + k + 8 * h);
                v[t][2 * h] = x[0];
                v[t][2 * h + 1] = x[1];
            } else {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int64_t q = k + 8 * h + e;
                    const double x = gload(row + min(q, M - 1));
                    v[t][2 * h + e] = zero && q >= kend ? 0.0 : x;
                }
            }
        }
    }
}

template <int RA, int CB>
__global__ void __launch_bounds__(256, 2) k_tn(const double *__restrict__ A, int64_t lda, int64_t sa,
                                               const double *__restrict__ B, int64_t ldb, int64_t sb, int rows, int n,
                                               int64_t M, int nsl, int nslices, int rt, int cg,
                                               int64_t per_wave, double *__restrict__ part) {
    __shared__ double red[4][4][256];  // wave, tile of the round, element
    const int lane = threadIdx.x & 63, lr = lane >> 4, lc = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tiles = rt * cg, id = blockIdx.x;
    const int slice = id / (8 * tiles) * 8 + id % 8, tile = id / 8 % tiles;
    if (slice >= nslices) return;
    const int p = slice / nsl;
    const int r0 = tile % rt * 16 * RA, c0 = tile / rt * 16 * CB;
    A += p * sa;
    B += p * sb;
    const int64_t kb = ((int64_t)(slice - p * nsl) * 4 + wave) * per_wave, ke = min(M, kb + per_wave);
    v4d acc[RA][CB];
#pragma unroll
    for (int i = 0; i < RA; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i][j] = (v4d){0.0, 0.0, 0.0, 0.0};
    double a[2][RA][4], b[2][CB][4];
    auto mul = [&](int h) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < RA; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j) acc[i][j] = MfmaTraits<double>::mma(a[h][i][s], b[h][j][s], acc[i][j]);
    };
    auto load = [&](int64_t k, int h) {
        tn_load<RA, false>(A, lda, rows, r0, k + 2 * lr, ke, M, false, lc, a[h]);
        tn_load<CB, false>(B, ldb, n, c0, k + 2 * lr, ke, M, true, lc, b[h]);
    };
    const int64_t kw = kb < ke ? kb + (ke - kb) / 16 * 16 : kb;  // whole blocks of 16 points
    if (kb < kw) load(kb, 0);
    for (int64_t k = kb; k < kw; k += 32) {
        if (k + 16 < kw) load(k + 16, 1);
        mul(0);
        if (k + 16 < kw) {
            if (k + 32 < kw) load(k + 32, 0);
            mul(1);
        }
    }
    if (kw < ke) {  // the last points: rows of B beyond them are zero, rows of A any finite value
        tn_load<RA, true>(A, lda, rows, r0, kw + 2 * lr, ke, M, false, lc, a[0]);
        tn_load<CB, true>(B, ldb, n, c0, kw + 2 * lr, ke, M, true, lc, b[0]);
        mul(0);
    }
    double *out = part + (int64_t)slice * rows * n;
#pragma unroll
    for (int t0 = 0; t0 < RA * CB; t0 += 4) {
        if (t0 > 0) __syncthreads();
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (t0 + t < RA * CB) {
                const int q = t0 + t < RA * CB ? t0 + t : 0;
#pragma unroll
                for (int r = 0; r < 4; ++r) red[wave][t][lc * 16 + lr + 4 * r] = acc[q / CB][q % CB][r];
            }
        __syncthreads();
        const int q = t0 + wave;  // wave w adds up tile t0 + w
        if (q < RA * CB) {
            const int rb = r0 + 16 * (q / CB), cb = c0 + 16 * (q % CB);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int x = e * 64 + lane, r = rb + x % 16, c = cb + x / 16;
                const double v = (red[0][wave][x] + red[1][wave][x]) + (red[2][wave][x] + red[3][wave][x]);
                if (r < rows && c < n) gstore(out + (int64_t)c * rows + r, v);
            }
        }
    }
}

namespace {
struct TnPlan {
    int ra, cb, rt, cg, nsl;
    int64_t per_wave;
};
// Row tiles per wave: four where that still leaves enough waves, fewer for few rows.  Slices: a multiple of 8 (as many on
// every XCD) or at most 3; of those the one with the least rounds of 512 blocks (two per CU) times points per wave, 64 of
// which stand for a round's start and final sum.  (A target of 1024 blocks, rounded up, ran three rounds, the last one
// nearly empty: 1374 x 48, 32 768 points 145 us, now 123; 458 x 24, 185 742 points 187, now 171.)
TnPlan tn_plan(int rows, int n, int64_t M, int nplane) {
    TnPlan p;
    p.ra = rows > 96 ? 4 : rows > 16 ? 2 : 1;
    const int ct = (n + 15) / 16, ng = (ct + 2) / 3;
    p.cb = (ct + ng - 1) / ng;
    p.cg = (ct + p.cb - 1) / p.cb;
    p.rt = (rows + 16 * p.ra - 1) / (16 * p.ra);
    const int64_t smax = std::min<int64_t>(128, std::max<int64_t>(1, (M + 255) / 256));
    int64_t best = -1;
    for (int64_t s = 1; s <= smax; s = s < 3 ? s + 1 : s < 8 ? 8 : s + 8) {
        const int64_t pw = ((M + 4 * s - 1) / (4 * s) + 15) / 16 * 16, nsl = (M + 4 * pw - 1) / (4 * pw);
        const int64_t blocks = (nsl * nplane + 7) / 8 * 8 * p.rt * p.cg, cost = (blocks + 511) / 512 * (pw + 64);
        if (best < 0 || cost < best) {
            best = cost;
            p.per_wave = pw;
            p.nsl = (int)nsl;
        }
    }
    return p;
}
}  // namespace

// The library's LDS-tiled product (batched over point slices) computes whole multiples of 64 columns, k_tn whole multiples of a
// wave's, reading A once for each.  Small products give the library too few tiles: about 230 us at any size.  Library and
// k_tn in us, work in rows x columns x points: 604 x 64, 32768 points (1.3e9) 230 and 78, 65536 (2.5e9) 236 and 139, 370001
// (1.4e10) 664 and 910; 604 x 128, 32768 (2.5e9) 227 and 127, 65536 (5.1e9) 238 and 236; 1208 x 128, 32768 (5.1e9) 235 and
// 234, 120001 (1.9e10) 723 and 816; 1832 x 192, 370001 4266 and 6456: from 5e9 on.  Above 192 columns tall products gain
// earlier: 1208 x 224, 8192 (2.2e9) 231 and 129, 1832 x 224 (3.4e9) 146 and 172, 1832 x 256 (3.8e9) 145 and 201: from 3e9 on.
// Where k_tn pads less (65 to 96 and 129 to 144 columns) it holds out longer: 604 x 96, 120001 (7e9) 474 and 341; 604 x 144,
// 370001 (3.2e10) 1473 and 1243; 1832 x 96, 120001 (2.1e10) 933 and 1075, 370001 (6.5e10) 2758 and 3173: from 3e10 on.
bool tn_by_library(int rows, int n, int64_t M) {
    if (n <= 48) return false;  // one column group: 604 x 48, 370001 points 608 and 587 us
    const TnPlan p = tn_plan(rows, n, M, 1);
    const bool pads_less = 16 * p.cb * p.cg < (n + 63) / 64 * 64;
    return (double)rows * n * (double)M >= (n > 192 ? 3e9 : pads_less ? 3e10 : 5e9);
}

int tn_slices(int rows, int n, int64_t M, int nplane) { return tn_plan(rows, n, M, nplane).nsl * nplane; }

void launch_tn(const double *A, int64_t lda, int64_t sa, const double *B, int64_t ldb, int64_t sb, int rows, int n,
               int64_t M, int nplane, double *part, hipStream_t s) {
    const TnPlan p = tn_plan(rows, n, M, nplane);
    const int nslices = p.nsl * nplane;
    const dim3 grid((unsigned)((nslices + 7) / 8 * 8 * p.rt * p.cg)), blk(256);
#define FLOSIC_TN(RA, CB) \
    hipLaunchKernelGGL((k_tn<RA, CB>), grid, blk, 0, s, A, lda, sa, B, ldb, sb, rows, n, M, p.nsl, nslices, p.rt, p.cg, \
                       p.per_wave, part)
    switch (10 * p.ra + p.cb) {
        case 11: FLOSIC_TN(1, 1); break;
        case 12: FLOSIC_TN(1, 2); break;
        case 13: FLOSIC_TN(1, 3); break;
        case 21: FLOSIC_TN(2, 1); break;
        case 22: FLOSIC_TN(2, 2); break;
        case 23: FLOSIC_TN(2, 3); break;
        case 41: FLOSIC_TN(4, 1); break;
        case 42: FLOSIC_TN(4, 2); break;
        default: FLOSIC_TN(4, 3); break;
    }
#undef FLOSIC_TN
}

}  // namespace flosic
