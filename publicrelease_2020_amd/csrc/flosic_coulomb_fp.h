// FP64 and FP32 MFMA Coulomb kernels (k_coulomb_fp and its batched form), included by one source file per type.
//
// V[f][k] = sum_rows R[k][row] H[row][f]: R_tuv(p, P - r_k) is generated on the fly (Boys functions and Hermite
// recursion), H is the Hermite-coefficient matrix of every exponent-pair group for every FLO in MFMA operand order.
#pragma once
#include "flosic_device.h"

namespace flosic {

// ---------------------------------------------------------------------------------------------------
// FP64 / FP32 Coulomb tile.
//
// Bound.  On gfx950 an FP64 or FP32 MFMA and the VALU instructions of the same SIMD do not overlap (measured: FP64
// MFMAs of one wave beside FP64, FP32 or integer VALU work of another take the sum of both times), so the kernel's
// floor is MFMA time + VALU time: 64 points x 16 columns x 4 rows are 4 MFMAs of 64 (FP64) or 32 (FP32) cycles, and R
// of one (64 points, group) pair is 70-250 VALU instructions.  Everything else has to leave the VALU: R passes from
// "lane = point" to the MFMA's A operand (lane = 16 points x 4 rows) through LDS, H comes straight from L1/L2 in B
// operand order, all loop and address arithmetic is scalar.
//
// Split.  Block = 4 wavefronts on one tile of 64 points = CW column waves x RW = 4 / CW row groups.  A wave holds 64
// points x NT column tiles of 16 FLOs (96 registers of FP64 accumulators at NT = 3, two waves per SIMD), so each B
// operand feeds four MFMAs.  Up to 64 FLOs one wave holds all columns (CW = 1, NT <= 4), makes the R it needs by itself
// and meets the other three, which take other Hermite rows, only in the final sum: no barrier in the loop.  Up to 96
// (192) FLOs CW = 2 (4) waves share the R that each makes a part of, with two barriers per CW units, and hold at most
// three tiles: a fourth would spill beside the shared R's bookkeeping (120 FLOs, 24 241 groups, 308 110 points, FP64:
// two waves of four tiles 271 ms, four waves of two tiles 238 ms).  More FLOs go to further blocks (grid.y).  Only
// column tiles that hold FLOs are computed (16-column granularity).
//
// Measured on synthetic systems (kernel time, against one 16-wave block per tile with dedicated R, copy and consumer
// waves that met at a barrier every 16 or 32 rows, columns padded to 64): FP64 30 FLOs / 116 200 points / 1686 groups
// 7.64 -> 2.24 ms; 48 / 185 742 / 4163 32.6 -> 12.3 ms (59 TFLOP/s, 76% of the 77.5 that FP64 MFMAs alone reach);
// 96 / 370 513 / 15 750 311 -> 173 ms; 192 / 196 174 / 60 795 784 -> 625 ms (82%).  FP32: 3.26 -> 1.21, 13.9 -> 7.1,
// 162 -> 91, 415 -> 338 ms (74% of 158 TFLOP/s).
//
// A unit is a run of groups of one order L that fills whole 4-row K steps: 16 groups of L = 0, 4 of L = 1 (4 K steps),
// 2 of L = 2, 1 of L = 3 (5 K steps), 1 of L = 4 (9 K steps; FP64: in LDS as 5 + 4).  The last unit of an L repeats its last
// group against zero rows of H.  FP32 accumulators go into FP64 sums after every chunk of chunk_units(L) units
// (<= 64 Hermite rows).
// ---------------------------------------------------------------------------------------------------
__host__ __device__ constexpr int unit_groups(int L) { return L == 0 ? 16 : L == 1 ? 4 : L == 2 ? 2 : 1; }
__host__ __device__ constexpr int unit_steps(int L) { return L < 2 ? 4 : L < 4 ? 5 : 9; }
__host__ __device__ constexpr int chunk_units(int L) { return L < 2 ? 4 : L < 4 ? 3 : 1; }
// Hermite rows of a unit in LDS at a time: an L = 4 unit (36) goes whole in FP32, whose accumulation order follows the
// units, and in two parts in FP64
template <typename T>
constexpr int kPartRows = sizeof(T) == 4 ? 36 : 20;
__host__ __device__ inline int seg_units(const FpSegs &s, int L) {
    return (s.g[L + 1] - s.g[L] + unit_groups(L) - 1) / unit_groups(L);
}
__host__ __device__ inline int64_t seg_step0(const FpSegs &s, int L) {  // first K step of the units of order L
    int64_t n = 0;
    for (int l = 0; l < L; ++l) n += (int64_t)seg_units(s, l) * unit_steps(l);
    return n;
}
inline int fp_units(const FpSegs &s) {
    int n = 0;
    for (int l = 0; l < 5; ++l) n += seg_units(s, l);
    return n;
}
// column waves of a block
__host__ __device__ constexpr int fp_col_waves(int nct, int ncb) {
    const int tb = (nct + ncb - 1) / ncb;
    return tb <= 4 ? 1 : tb <= 6 ? 2 : 4;
}

// H in operand order: Hf[(step * nct + ct) * 64 + lane] = H[row 4*step + lane/16][column 16*ct + lane%16] over the
// units' zero-extended rows; one block per unit
template <typename T>
__global__ void k_frag_h(FpSegs seg, const double *__restrict__ H, int ldh, int nF, T *__restrict__ Hf) {
    int u = blockIdx.x, L = 0, hrow = 0;
    for (; L < 4 && u >= seg_units(seg, L); ++L) {
        u -= seg_units(seg, L);
        hrow += (seg.g[L + 1] - seg.g[L]) * ntuv(L);
    }
    const int nt = ntuv(L), ng = min(unit_groups(L), seg.g[L + 1] - seg.g[L] - u * unit_groups(L));
    const int nreal = ng * nt, kr = 4 * unit_steps(L), nct = ldh / 16;
    hrow += u * unit_groups(L) * nt;
    T *dst = Hf + (seg_step0(seg, L) + (int64_t)u * unit_steps(L)) * nct * 64;
    for (int e = threadIdx.x; e < kr * ldh; e += blockDim.x) {
        const int r = e / ldh, f = e - r * ldh;
        const double v = (r < nreal && f < nF) ? H[(int64_t)(hrow + r) * ldh + f] : 0.0;
        dst[((r / 4) * nct + f / 16) * 64 + (r % 4) * 16 + f % 16] = (T)v;
    }
}

// per wave: kPartRows x 64 points of R; in the epilogue one column tile of sums, [column][66 points] in FP64
template <typename T>
struct FpTileLds {
    static constexpr int kWave = (kPartRows<T> * 64 * (int)sizeof(T) > 16 * 66 * 8 ? kPartRows<T> * 64 * (int)sizeof(T) : 16 * 66 * 8);
    __attribute__((aligned(16))) unsigned char raw[4][kWave];
};

template <typename T, int NT>
struct FpAcc {
    typename MfmaTraits<T>::acc a[4][NT];
    double sum[sizeof(T) == 4 ? 4 : 1][NT][4];  // FP32 form
};

// the units of order L that belong to row group rg
template <typename T, int CW, int NT, int L>
__device__ __forceinline__ void fp_segment(const FpSegs &seg, const double4 *__restrict__ pP,
                                           const T *__restrict__ Hf, int nct, int ct0, T *__restrict__ Rg, int cw, int rg,
                                           int lane, double px, double py, double pz, const RType<T> *__restrict__ tab,
                                           FpAcc<T, NT> &A) {
    using C = RType<T>;
    using Tr = MfmaTraits<T>;
    constexpr int G = unit_groups(L), NS = unit_steps(L), CU = chunk_units(L), nt = ntuv(L), RW = 4 / CW;
    constexpr int NH = L == 4 && sizeof(T) == 8 ? 2 : 1;  // parts of a unit in LDS
    constexpr int NR = G * nt;           // rows of a unit (35 of L = 4: a zero row is added)
    // four column tiles: the B operands of an L = 4 unit are not held in registers beside its 35 R values
    constexpr bool HOLD = !(NT == 4 && L == 4);
    constexpr int S0 = NH == 2 ? 5 : NS;  // K steps of part 0; part 1 has NS - S0
    const int nu = seg_units(seg, L);
    if (nu <= 0) return;
    const int nch = (nu + CU - 1) / CU;
    const int u0 = min(nu, nch * rg / RW * CU), u1 = min(nu, nch * (rg + 1) / RW * CU);
    // with shared R every row group runs the same number of stages, so that all waves meet at the barriers
    const int nst = CW == 1 ? u1 - u0 : ((nch + RW - 1) / RW * CU + CW - 1) / CW;
    const int lr = lane >> 4, lc = lane & 15;
    // R row r of point q sits at r * 64 + (q ^ 16 (r & 3)): the four rows of a K step are read from different banks
    int ra[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ra[i] = lr * 64 + ((i ^ lr) << 4) + lc;
    const T *hb = Hf + (seg_step0(seg, L) * nct + ct0) * 64 + lane;
    const int64_t ustride = (int64_t)NS * nct * 64;
    // B operands of one part of a unit; step s of the next part is loaded as soon as step s of this one is used
    T b[S0][NT];
    auto load_b = [&](int s, int u, int h) {
        const T *p = hb + (int64_t)min(u, nu - 1) * ustride + (int64_t)((h * S0 + s) * nct) * 64;
#pragma unroll
        for (int j = 0; j < NT; ++j) b[s][j] = gload(p + j * 64);
    };
    if constexpr (HOLD) {
#pragma unroll
        for (int s = 0; s < S0; ++s) load_b(s, u0, 0);
    }
    for (int st = 0; st < nst; ++st) {
        const int ub = u0 + st * CW, mine = ub + cw;
        C R[NR];
        if (CW == 1 || mine < u1) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const v4d P = cload(reinterpret_cast<const v4d *>(pP + min(seg.g[L] + mine * G + g, seg.g[L + 1] - 1)));
                // lanes past the mesh end compute finite values too: an A row feeds only its own point's output row
                hermite_R<L, C>((C)P.w, (C)(P.x - px), (C)(P.y - py), (C)(P.z - pz), tab, R + g * nt);
            }
        }
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            const int ns = h == 0 ? S0 : NS - S0;
            tile_sync<CW>();  // the last part has been read
#pragma unroll
            for (int r = 0; r < 4 * S0; ++r)
                if (r < 4 * ns) {
                    const int q = 4 * h * S0 + r;
                    Rg[cw * (kPartRows<T> * 64) + r * 64 + (lane ^ ((r & 3) << 4))] = q < NR ? (T)R[q < NR ? q : 0] : (T)0;
                }
            tile_sync<CW>();
            if constexpr (!HOLD) {
                if (h == 0) {
#pragma unroll
                    for (int s = 0; s < S0; ++s) load_b(s, ub, 0);
                }
            }
#pragma unroll
            for (int u = 0; u < CW; ++u) {
                // the part after this one: the next unit, the first unit's second part, or the next stage
                const int un = u + 1 < CW ? ub + u + 1 : h + 1 < NH ? ub : ub + CW;
                const int hn = u + 1 < CW ? h : h + 1 < NH ? h + 1 : 0;
                const int nn = !HOLD && u + 1 == CW && h + 1 == NH ? 0 : hn == 0 ? S0 : NS - S0;
                const T *Ru = Rg + u * (kPartRows<T> * 64);
                const bool on = ub + u < u1;
                if (on) {
#pragma unroll
                    for (int s = 0; s < S0; ++s) {
                        if (s < ns) {
                            T a[4];
#pragma unroll
                            for (int i = 0; i < 4; ++i) a[i] = Ru[s * 256 + ra[i]];
#pragma unroll
                            for (int i = 0; i < 4; ++i)
#pragma unroll
                                for (int j = 0; j < NT; ++j) A.a[i][j] = Tr::mma(a[i], b[s][j], A.a[i][j]);
                        }
                        if (s < nn) load_b(s, un, hn);
                    }
                    if constexpr (sizeof(T) == 4) {
                        if (h + 1 == NH && ((ub + u + 1) % CU == 0 || ub + u + 1 == u1)) {
#pragma unroll
                            for (int i = 0; i < 4; ++i)
#pragma unroll
                                for (int j = 0; j < NT; ++j)
#pragma unroll
                                    for (int r = 0; r < 4; ++r) {
                                        A.sum[i][j][r] += (double)A.a[i][j][r];
                                        A.a[i][j][r] = 0.0f;
                                    }
                        }
                    }
                } else if (CW > 1) {
#pragma unroll
                    for (int s = 0; s < S0; ++s)
                        if (s < nn) load_b(s, un, hn);
                }
            }
        }
    }
}

// the work of one wave: NT column tiles from ct0 on
template <typename T, int CW, int NT>
__device__ __forceinline__ void fp_wave(FpTileLds<T> &lds, const CoulJob<T> &J, const double *__restrict__ tab,
                                        int64_t tile, int wave, int ct0, int ntmax) {
    constexpr int RW = 4 / CW;
    const int lane = threadIdx.x & 63, cw = wave % CW, rg = wave / CW;
    const int64_t k0 = tile * 64;
    const int64_t kl = k0 + lane;
    const bool valid = kl < J.M;
    const double px = valid ? gload(J.X + kl) : 0.0, py = valid ? gload(J.Y + kl) : 0.0, pz = valid ? gload(J.Z + kl) : 0.0;
    const RType<T> *ctab = sizeof(T) == 8 ? (const RType<T> *)tab : (const RType<T> *)(tab + kBoysRows * kBoysCols);
    T *Rg = reinterpret_cast<T *>(lds.raw[rg * CW]);  // the CW waves' R one after the other
    FpAcc<T, NT> A;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                A.a[i][j][r] = (T)0;
                if constexpr (sizeof(T) == 4) A.sum[i][j][r] = 0.0;
            }
    const T *Hf = (const T *)J.H;
    fp_segment<T, CW, NT, 0>(J.seg, J.pP, Hf, J.nct, ct0, Rg, cw, rg, lane, px, py, pz, ctab, A);
    fp_segment<T, CW, NT, 1>(J.seg, J.pP, Hf, J.nct, ct0, Rg, cw, rg, lane, px, py, pz, ctab, A);
    fp_segment<T, CW, NT, 2>(J.seg, J.pP, Hf, J.nct, ct0, Rg, cw, rg, lane, px, py, pz, ctab, A);
    fp_segment<T, CW, NT, 3>(J.seg, J.pP, Hf, J.nct, ct0, Rg, cw, rg, lane, px, py, pz, ctab, A);
    fp_segment<T, CW, NT, 4>(J.seg, J.pP, Hf, J.nct, ct0, Rg, cw, rg, lane, px, py, pz, ctab, A);
    // the row groups' sums of one column tile at a time through LDS: wave (cw, rg) adds and stores 16 / RW columns,
    // 64 points (512 bytes) per store
    const int lr = lane >> 4, lc = lane & 15;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (j >= ntmax) break;
        __syncthreads();
        if (j < NT) {
            double *o = reinterpret_cast<double *>(lds.raw[wave]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int jj = j < NT ? j : 0;
                    double v;
                    if constexpr (sizeof(T) == 4) v = A.sum[i][jj][r];
                    else v = A.a[i][jj][r];
                    o[lc * 66 + i * 16 + MfmaTraits<T>::row(lr, r)] = v;
                }
        }
        __syncthreads();
        if (j < NT) {
#pragma unroll
            for (int q = 0; q < 16 / RW; ++q) {
                const int col = rg * (16 / RW) + q, f = (ct0 + j) * 16 + col;
                double v = reinterpret_cast<const double *>(lds.raw[cw])[col * 66 + lane];
#pragma unroll
                for (int g = 1; g < RW; ++g) v += reinterpret_cast<const double *>(lds.raw[g * CW + cw])[col * 66 + lane];
                if (f < J.nF && valid) gstore(J.V + (int64_t)f * J.ldv + kl, v);
            }
        }
    }
}

// One (64-point tile, column block cb of ncb) of one system's contraction.  The column tiles are shared out evenly over
// the blocks and over a block's column waves; NTLO..NTHI bounds the tiles per wave that this instance is built for.
template <typename T, int CW, int NTLO, int NTHI>
__device__ __forceinline__ void coulomb_tile_fp(FpTileLds<T> &lds, const CoulJob<T> &J, const double *__restrict__ tab,
                                                int64_t tile, int cb) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), cw = wave % CW;
    const int tb0 = J.nct * cb / J.ncb, tb = J.nct * (cb + 1) / J.ncb - tb0;
    const int c0 = tb * cw / CW, nt = tb * (cw + 1) / CW - c0, ntmax = (tb + CW - 1) / CW;
    if constexpr (NTHI >= 4) {
        if (nt == 4) return fp_wave<T, CW, 4>(lds, J, tab, tile, wave, tb0 + c0, ntmax);
    }
    if constexpr (NTLO <= 3 && NTHI >= 3) {
        if (nt == 3) return fp_wave<T, CW, 3>(lds, J, tab, tile, wave, tb0 + c0, ntmax);
    }
    if constexpr (NTLO <= 2 && NTHI >= 2) {
        if (nt == 2) return fp_wave<T, CW, 2>(lds, J, tab, tile, wave, tb0 + c0, ntmax);
    }
    if constexpr (NTLO <= 1) {
        if (nt == 1) return fp_wave<T, CW, 1>(lds, J, tab, tile, wave, tb0 + c0, ntmax);
    }
}

// waves per SIMD that the registers allow without spilling much: 32 accumulator registers per tile (FP32: 48 with the
// FP64 sums), 35 R values and the B operands of a unit; FP64 waves that share R need two more units' bookkeeping
template <typename T, int CW, int NTM>
constexpr int fp_waves_per_simd = NTM > 2 || (CW > 1 && sizeof(T) == 8) ? 2 : 5 - NTM;

// NTM: the most column tiles a wave of this launch holds (the others hold one less)
template <typename T, int CW, int NTM>
__global__ void __launch_bounds__(256, (fp_waves_per_simd<T, CW, NTM>)) k_coulomb_fp(CoulJob<T> J, const double *__restrict__ tab) {
    __shared__ FpTileLds<T> lds;
    static_assert(split_covered(fp_col_waves, 256, CW, (NTM > 1 ? NTM - 1 : 1), NTM, true), "a wave's tiles have no instance");
    coulomb_tile_fp<T, CW, (NTM > 1 ? NTM - 1 : 1), NTM>(lds, J, tab, blockIdx.x, blockIdx.y);
}

template <typename T>
__global__ void __launch_bounds__(256, 2) k_coulomb_fp_batch_all(const CoulJob<T> *__restrict__ jobs,
                                                                 const int64_t *__restrict__ off, int njobs,
                                                                 const double *__restrict__ tab) {
    __shared__ FpTileLds<T> lds;
    int64_t local = 0;
    const int j = job_of_block(off, njobs, (int64_t)blockIdx.x, local);
    const CoulJob<T> J = uniform_job(jobs, j);
    const int64_t tile = local / J.ncb;
    const int cb = (int)(local - tile * J.ncb);
    static_assert(split_covered(fp_col_waves, 256, 1, 1, 4, false) && split_covered(fp_col_waves, 256, 2, 2, 3, false) &&
                      split_covered(fp_col_waves, 256, 4, 1, 3, false), "a wave's tiles have no instance");
    switch (fp_col_waves(J.nct, J.ncb)) {
        case 1: coulomb_tile_fp<T, 1, 1, 4>(lds, J, tab, tile, cb); break;
        case 2: coulomb_tile_fp<T, 2, 2, 3>(lds, J, tab, tile, cb); break;
        default: coulomb_tile_fp<T, 4, 1, 3>(lds, J, tab, tile, cb); break;
    }
}

template <typename T>
void launch_frag_h(const FpSegs &seg, const double *H, int ldh, int nF, T *Hf, hipStream_t s) {
    const int nu = fp_units(seg);
    if (nu <= 0) return;
    hipLaunchKernelGGL((k_frag_h<T>), dim3(nu), dim3(256), 0, s, seg, H, ldh, nF, Hf);
}

template <typename T>
void launch_coulomb_mfma(const FpSegs &seg, const double4 *pairP, const T *Hf, const double *x, const double *y,
                         const double *z, int64_t M, const double *btab, int nF, double *V, int64_t ldv, hipStream_t s,
                         int nfb) {
    if (seg.g[5] <= 0 || M <= 0) return;
    if (nfb <= 0) nfb = coulomb_cols(nF);
    CoulJob<T> J{};
    J.seg = seg;
    J.pP = pairP;
    J.H = Hf;
    J.nct = (nF + 15) / 16;
    J.X = x;
    J.Y = y;
    J.Z = z;
    J.M = M;
    J.nF = nF;
    J.V = V;
    J.ldv = ldv;
    J.ncb = coulomb_col_blocks(nF, nfb);
    const int cw = fp_col_waves(J.nct, J.ncb), tb = (J.nct + J.ncb - 1) / J.ncb, ntm = (tb + cw - 1) / cw;
    const dim3 grid((unsigned)((M + 63) / 64), (unsigned)J.ncb), blk(256);
#define FLOSIC_FP(CW, NTM) hipLaunchKernelGGL((k_coulomb_fp<T, CW, NTM>), grid, blk, 0, s, J, btab)
    switch (10 * cw + ntm) {
        case 11: FLOSIC_FP(1, 1); break;
        case 12: FLOSIC_FP(1, 2); break;
        case 13: FLOSIC_FP(1, 3); break;
        case 14: FLOSIC_FP(1, 4); break;
        case 23: FLOSIC_FP(2, 3); break;
        case 42: FLOSIC_FP(4, 2); break;
        default: FLOSIC_FP(4, 3); break;
    }
#undef FLOSIC_FP
}

template <typename T>
void launch_coulomb_batch_all(const CoulJob<T> *jobs, const int64_t *off, int njobs, int64_t items,
                              const double *btab, hipStream_t s) {
    if (njobs <= 0 || items <= 0) return;
    hipLaunchKernelGGL((k_coulomb_fp_batch_all<T>), dim3((unsigned)items), dim3(256), 0, s, jobs, off, njobs, btab);
}

}  // namespace flosic
