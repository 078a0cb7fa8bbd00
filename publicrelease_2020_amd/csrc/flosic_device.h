// Device code shared by the kernel files: Cartesian and Hermite index tables, Boys functions and Hermite integrals R_tuv,
// typed loads, MFMA wrappers, batch job lookup.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "flosic_internal.h"

namespace flosic {

// ---------------------------------------------------------------------------------------------------
// Cartesian component tables: index 0..9 = s, x, y, z, xx, yy, zz, xy, xz, yz (gorbdrv.f:78-98)
// ---------------------------------------------------------------------------------------------------
__host__ __device__ constexpr int cpow(int idx, int ax) {
    return idx == 0 ? 0
           : idx <= 3 ? (idx - 1 == ax ? 1 : 0)
           : idx <= 6 ? (idx - 4 == ax ? 2 : 0)
           : idx == 7 ? (ax < 2 ? 1 : 0)
           : idx == 8 ? (ax != 1 ? 1 : 0)
                      : (ax > 0 ? 1 : 0);
}
__host__ __device__ constexpr int ncart(int l) { return l == 0 ? 1 : (l == 1 ? 3 : 6); }
__host__ __device__ constexpr int loff(int l) { return l == 0 ? 0 : (l == 1 ? 1 : 4); }

// ---------------------------------------------------------------------------------------------------
// Hermite index tables: entries grouped by total order L' = 0..4; within an order t descending, then u
// descending (t+u+v = L')
// ---------------------------------------------------------------------------------------------------
__host__ __device__ constexpr int ntuv(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }
// Chunk types of the split-BF16 chunk list: L = 0..4 whole groups of that L; L = 5 the first 32 Hermite rows of L = 4
// groups, L = 6 their last 3 rows (a 35-row group would otherwise fill a 64-row chunk with 29 zero rows).  Rows per
// group in the chunk, offset of those rows inside the group's Hermite block, and the group's Hermite order:
__host__ __device__ constexpr int chunk_rpg(int L) { return L == 5 ? 32 : L == 6 ? 3 : ntuv(L); }
__host__ __device__ constexpr int chunk_roff(int L) { return L == 6 ? 32 : 0; }
__host__ __device__ constexpr int chunk_herm(int L) { return L > 4 ? 4 : L; }
__host__ __device__ constexpr int tuv_idx(int t, int u, int v) {
    // position inside order block: enumerate t from L' down, u from L'-t down
    int L = t + u + v;
    int base = L == 0 ? 0 : ntuv(L - 1);
    int pos = 0;
    for (int tt = L; tt > t; --tt) pos += L - tt + 1;
    pos += (L - t) - u;
    return base + pos;
}
__host__ __device__ constexpr int tuv_comp(int i, int which) {
    for (int L = 0; L <= 4; ++L)
        for (int t = L; t >= 0; --t)
            for (int u = L - t; u >= 0; --u) {
                int v = L - t - u;
                if (tuv_idx(t, u, v) == i) return which == 0 ? t : (which == 1 ? u : v);
            }
    return -1;
}

// ---------------------------------------------------------------------------------------------------
// Boys functions F_0..F_TOP (fffmt3.F:66-88): T > 16 one-term asymptote + upward recursion; otherwise
// cubic Taylor of F_TOP about the nearest 0.01 node and downward recursion
// ---------------------------------------------------------------------------------------------------
// Boys F_0..F_TOP of the reference scheme (fffmt3.F): T > 16 one-term asymptote and upward recursion, else the
// cubic Taylor expansion of F_TOP about the nearest table node and downward recursion.  C = double for the FP64
// forms; C = float (table rounded to FP32) where R feeds FP32 or split-BF16 MFMA operands anyway.
// The FP32 branches, with their rounding steps written out (see rterm): far (T > 16) and near, the hardware reciprocal and
// square root (1 ulp) instead of correctly rounded ones, well inside the FP32 R's own rounding
template <int TOP>
__device__ __forceinline__ void boys32_far(float T, float eT, float *F) {
    const float rect1 = 0.5f * __builtin_amdgcn_rcpf(T);
    const float q = __builtin_fmaf(__builtin_amdgcn_sqrtf(T), 1.77245385090551602728f, -eT);
    F[0] = rect1 * q;
    F[1] = rect1 * __builtin_fmaf(rect1, q, -eT);
#pragma unroll
    for (int m = 2; m <= TOP; ++m) F[m] = rect1 * __builtin_fmaf((float)(2 * m - 1), F[m - 1], -eT);
}
template <int TOP>
__device__ __forceinline__ void boys32_near(float T, float eT, const float *__restrict__ tab, float *F) {
    const int it = (int)__builtin_fmaf(100.0f, T, 1.5f);
    const float dt = __builtin_fmaf(1.0e-2f, (float)(it - 1), -T);
    const float *f = tab + (it - 1) * kBoysCols;
    // times the rounded 1/6 (a correctly rounded division costs 10 VALU)
    F[TOP] = __builtin_fmaf(dt, __builtin_fmaf(dt, __builtin_fmaf(f[TOP + 2], 0.5f, dt * (f[TOP + 3] * (1.0f / 6.0f))), f[TOP + 1]),
                            f[TOP]);
    const float rect1 = 2.0f * T;
#pragma unroll
    for (int m = TOP - 1; m >= 0; --m) {
        const float r = __builtin_fmaf(rect1, F[m + 1], eT);
        F[m] = m == 0 ? r : r * (1.0f / (2 * m + 1));
    }
}
template <int TOP, typename C>
__device__ __forceinline__ void boys(C T, C eT, const C *__restrict__ tab, C *F) {
    if constexpr (sizeof(C) == 4) {
        if (T > 16.0f) boys32_far<TOP>(T, eT, F);
        else boys32_near<TOP>(T, eT, tab, F);
    } else if (T > 16.0) {
        // 1/sqrt(T) from the hardware's estimate (relative error below 2^-20) and one third-order step, y (1 + e/2 + 3e^2/8)
        // with e = 1 - T y^2, which leaves e^3; its square, corrected once, is 1/(2T).  With sqrt(pi/4T) 13 VALU instructions,
        // where a correctly rounded division and square root took 30.  F_0 .. F_4 over T = 16 .. 400 against extended
        // precision, mean error in units of 2^-53: 0.59, 0.77, 1.09, 1.42, 1.76 (before 0.75, 1.02, 1.37, 1.72, 2.07)
        double y = __builtin_amdgcn_rsq(T);
        const double e = __builtin_fma(-T * y, y, 1.0);
        y = __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
        double rect1 = 0.5 * y * y;
        rect1 = __builtin_fma(rect1, __builtin_fma(-2.0 * T, rect1, 1.0), rect1);
        F[0] = __builtin_fma(y, 0.88622692545275801365, -rect1 * eT);
#pragma unroll
        for (int m = 1; m <= TOP; ++m) F[m] = rect1 * ((2 * m - 1) * F[m - 1] - eT);
    } else {
        const int it = (int)(100.0 * T + 1.5);
        const double dt = 1.0e-2 * (it - 1) - T;
        const double *f = tab + (it - 1) * kBoysCols;
        // times the rounded 1/6: half an ulp of a term that is below 1e-8 of the sum
        F[TOP] = f[TOP] + dt * (f[TOP + 1] + dt * (f[TOP + 2] * 0.5 + dt * (f[TOP + 3] * (1.0 / 6.0))));
        const double rect1 = 2.0 * T;
#pragma unroll
        for (int m = TOP - 1; m >= 0; --m) {
            const double r = F[m + 1] * rect1 + eT;
            F[m] = (m == 0) ? r : r * (1.0 / (2 * m + 1));
        }
    }
}

// x r0 + c r1.  FP32: with the rounding steps written out, so that every kernel that generates R in FP32 gets the same bits
template <int c, typename C>
__device__ __forceinline__ C rterm(C x, C r0, C r1) {
    if constexpr (sizeof(C) == 4) return c == 1 ? __builtin_fmaf(x, r0, r1) : __builtin_fmaf((float)c, r1, x * r0);
    else return x * r0 + c * r1;
}
// one Hermite step R^{(n)}_I from R^{(n+1)} in place (entries of lower order still hold level n+1)
template <int I, typename C>
__device__ __forceinline__ void rstep(C *R, C X, C Y, C Z) {
    constexpr int t = tuv_comp(I, 0), u = tuv_comp(I, 1), v = tuv_comp(I, 2);
    if constexpr (t > 0) {
        if constexpr (t > 1) R[I] = rterm<t - 1, C>(X, R[tuv_idx(t - 1, u, v)], R[tuv_idx(t - 2, u, v)]);
        else R[I] = X * R[tuv_idx(t - 1, u, v)];
    } else if constexpr (u > 0) {
        if constexpr (u > 1) R[I] = rterm<u - 1, C>(Y, R[tuv_idx(t, u - 1, v)], R[tuv_idx(t, u - 2, v)]);
        else R[I] = Y * R[tuv_idx(t, u - 1, v)];
    } else {
        if constexpr (v > 1) R[I] = rterm<v - 1, C>(Z, R[tuv_idx(t, u, v - 1)], R[tuv_idx(t, u, v - 2)]);
        else R[I] = Z * R[tuv_idx(t, u, v - 1)];
    }
}
template <int I, typename C>
__device__ __forceinline__ void rdown(C *R, C X, C Y, C Z) {
    if constexpr (I >= 1) {
        rstep<I, C>(R, X, Y, Z);
        rdown<I - 1, C>(R, X, Y, Z);
    }
}
template <int L, int N, typename C>
__device__ __forceinline__ void rlevels(C *R, C X, C Y, C Z, const C *F, const C *pw) {
    if constexpr (N >= 0) {
        rdown<ntuv(L - N) - 1, C>(R, X, Y, Z);
        R[0] = pw[N] * F[N];
        rlevels<L, N - 1, C>(R, X, Y, Z, F, pw);
    }
}

// R_tuv(p, P - C) for all t+u+v <= L, TUV order
template <int L, typename C = double>
__device__ __forceinline__ void hermite_R(C p, C X, C Y, C Z, const C *__restrict__ tab, C *R) {
    constexpr int TOP = L < 2 ? 2 : L;
    C T;
    if constexpr (sizeof(C) == 4) T = p * __builtin_fmaf(Z, Z, __builtin_fmaf(X, X, Y * Y));
    else T = p * (X * X + Y * Y + Z * Z);
    C F[TOP + 1];
    C eT;
    if constexpr (sizeof(C) == 8)
        // beyond T = 60, e^-T (< 9e-27) is below half an ulp of every term it enters (F_4(60) ~ 6e-8), so
        // dropping it leaves each F_m bitwise unchanged and saves the exponential for most (point, group) pairs
        eT = T > 60.0 ? 0.0 : exp(-T);
    else  // FP32: the hardware exponential of -T log2(e) (relative error < 1e-6 at T = 16, where e^-T adds 1e-13)
        eT = __expf(-T);
    boys<TOP, C>(T, eT, tab, F);
    C pw[L + 1];
    pw[0] = C(1.0);
#pragma unroll
    for (int n = 1; n <= L; ++n) pw[n] = pw[n - 1] * (C(-2.0) * p);
    R[0] = pw[L] * F[L];
    rlevels<L, L - 1, C>(R, X, Y, Z, F, pw);
}

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
// Loads and stores through a pointer typed as global memory.  The batch kernels read their arrays' addresses from a
// job table in device memory, and to the compiler such an address is generic: accesses through it become flat
// instructions, which also count against the LDS counter, so a wait for LDS would drain the wave's global loads in
// flight as well.  The Coulomb tiles load and store through these (with scalar or ext_vector
// types: a class type such as double4 would be copied through its generic-address copy constructor).
template <typename T>
__device__ __forceinline__ T gload(const T *p) {
    return *(const __attribute__((address_space(1))) T *)p;
}
template <typename T>
__device__ __forceinline__ void gstore(T *p, T v) {
    *(__attribute__((address_space(1))) T *)p = v;
}
// Load of read-only data at a wave-uniform address through the constant address space: a scalar load (lgkm
// counter), which leaves the wave's vector loads in flight.  A vector load there would need a vmcnt wait before
// its value could be made uniform, draining the H loads in flight with it.
template <typename T>
__device__ __forceinline__ T cload(const T *p) {
    return *(const __attribute__((address_space(4))) T *)p;
}

// chunk record c with every field read into scalar registers.  The tile code loops and branches on these fields; read
// through a pointer that the compiler cannot prove unwritten during the kernel (the batch kernels take it from a job
// record in device memory) they would otherwise be per-lane values, and those loops divergent ones.
__device__ __forceinline__ ChunkDev chunk_at(const ChunkDev *__restrict__ chunks, int c) {
    static_assert(sizeof(ChunkDev) % 4 == 0, "chunk record in 32-bit words");
    constexpr int NW = sizeof(ChunkDev) / 4;
    const unsigned *src = reinterpret_cast<const unsigned *>(chunks + c);
    unsigned w[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) w[i] = __builtin_amdgcn_readfirstlane(cload(src + i));
    ChunkDev ch;
    __builtin_memcpy(&ch, w, sizeof(ch));
    return ch;
}
// s_waitcnt lgkmcnt(0) alone (vmcnt 63, expcnt 7)
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xF | (7 << 4) | (0 << 8) | (3 << 14)); }
__device__ __forceinline__ void wave_lds_sync() {  // this wave's LDS stores before its later loads (no instruction)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
template <int CW>
__device__ __forceinline__ void tile_sync() {  // the waves that share R
    if constexpr (CW == 1) wave_lds_sync();
    else __syncthreads();
}

// the type in which R is generated: FP64 for the FP64 form, FP32 for the FP32 and split-BF16 operands
template <typename T>
using RType = typename std::conditional<sizeof(T) == 8, double, float>::type;

template <typename T> struct MfmaTraits;
// Operands of both 16x16x4 forms: lane l holds A[l%16][l/16] and B[l/16][l%16].  The accumulators differ:
// FP32 register r of lane l holds D[4*(l/16) + r][l%16], FP64 register r holds D[l/16 + 4*r][l%16].
template <> struct MfmaTraits<double> {
    using acc = v4d;
    static __device__ __forceinline__ acc mma(double a, double b, acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lr, int r) { return lr + 4 * r; }
};
template <> struct MfmaTraits<float> {
    using acc = v4f;
    static __device__ __forceinline__ acc mma(float a, float b, acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lr, int r) { return 4 * lr + r; }
};

// ---------------------------------------------------------------------------------------------------
// Batched Coulomb: one launch over the (system, point tile, column block) items of every system of one form.
// Block b runs item b with the single-system tile code; the host orders the systems (heaviest items first) so
// that the dispatcher, which hands blocks to CUs in index order as CUs free up, balances them like a work queue.
// The grid is the queue, two blocks of four waves (split-BF16: one of eight) per CU at a time, and no block loops.
// ---------------------------------------------------------------------------------------------------
// Every job of a batch form in one launch.  The job records sit in device memory (a batch of 48 systems does not fit
// the kernel argument space); each block copies its job through readfirstlane word by word, so every field is a
// scalar (uniform) value in the tile code, as when it comes from the kernel arguments, and the tile's loop bounds
// stay scalar branches.  Jobs of different splits share the launch: the block switches on the column waves
// that its job's column tiles ask for, and all splits share the LDS of the largest.
template <typename T>
__device__ __forceinline__ CoulJob<T> uniform_job(const CoulJob<T> *__restrict__ jobs, int j) {
    static_assert(sizeof(CoulJob<T>) % 4 == 0, "job record in 32-bit words");
    constexpr int NW = sizeof(CoulJob<T>) / 4;
    const unsigned *src = reinterpret_cast<const unsigned *>(jobs + j);
    unsigned w[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) w[i] = __builtin_amdgcn_readfirstlane(cload(src + i));
    CoulJob<T> J;
    __builtin_memcpy(&J, w, sizeof(J));
    return J;
}
__device__ __forceinline__ int64_t uniform_i64(int64_t v) {
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)(uint64_t)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)((uint64_t)v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}
// Column tiles that a launch shares out: block cb of ncb takes tiles nct cb / ncb to nct (cb + 1) / ncb - 1, column wave cw of
// its CW likewise.  A wave whose count has no compiled instance would return with its columns unwritten, so every kernel
// asserts that its instances, those of NTLO to NTHI tiles, cover every share-out (cws(nct, ncb) the column waves of a block;
// blocks of the legal widths up to `widest` columns; 128 tiles are 2048 FLOs, and the counts per wave recur long before).
// single: the instances of the launch for one system, built for its largest wave's tiles and one less.
template <typename F>
constexpr bool split_covered(F cws, int widest, int CW, int NTLO, int NTHI, bool single) {
    for (int nfb = 64; nfb <= widest; nfb += 64)
        for (int nct = 1; nct <= 128; ++nct) {
            const int ncb = coulomb_col_blocks(16 * nct, nfb);
            if (cws(nct, ncb) != CW) continue;
            const int ntm = ((nct + ncb - 1) / ncb + CW - 1) / CW;
            if (single && ntm != NTHI) continue;
            for (int cb = 0; cb < ncb; ++cb) {
                const int tb = nct * (cb + 1) / ncb - nct * cb / ncb;
                for (int cw = 0; cw < CW; ++cw) {
                    const int nt = tb * (cw + 1) / CW - tb * cw / CW;
                    if (nt < NTLO || nt > NTHI) return false;
                }
            }
        }
    return true;
}
// block -> (job, local item): off[] ascending, off[0] = 0
__device__ __forceinline__ int job_of_block(const int64_t *__restrict__ off, int njobs, int64_t it, int64_t &local) {
    int lo = 0, hi = njobs - 1;  // largest j with off[j] <= it
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (uniform_i64(cload(off + mid)) <= it) lo = mid;
        else hi = mid - 1;
    }
    const int j = __builtin_amdgcn_readfirstlane(lo);
    local = it - uniform_i64(cload(off + j));
    return j;
}

}  // namespace flosic
