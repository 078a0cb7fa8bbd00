// Split-BF16 Coulomb kernels (k_coulomb_bf16 and its batched form) and the far-chunk bits.
#include "flosic_device.h"

namespace flosic {

// ---------------------------------------------------------------------------------------------------
// Split-BF16 Coulomb.  x = x1 + x2 (+ x3) in bf16 pieces, so the product x*y is carried by x1y1 + x1y2 + x2y1
// (+ x1y3 + x2y2 + x3y1) at ~2^-16 (2^-24) relative error, every term on the 16x16x32 bf16 MFMA (lane l holds
// A[l%16][8*(l/16) .. +7], B[8*(l/16) .. +7][l%16]; FP32 register r holds D[4*(l/16) + r][l%16]).
//
// Bound.  Per 32 Hermite rows and 64 points: 4 * 6 MFMAs of 16 cycles for every 16 columns against, once, R of the rows'
// groups (60-110 FP32 VALU instructions per group) and its split into pieces (176 VALU instructions).  Beside bf16 MFMAs
// FP32 VALU work overlaps only in part (measured: about a quarter of the shorter of the two), so R and the split are made
// once per 64 points and never again per column: a wave holds 64 points x NT <= 3 tiles of 16 columns (48 FP32
// accumulators and 48 FP64 sums), and its H operands come from L1/L2 straight into registers.
//
// Split.  Block = 8 wavefronts, one block per CU (256 registers per lane).
//   up to  48 FLOs  CW = 1: two tiles of 64 points (small meshes: one); the four (eight) waves of a tile hold all its columns,
//                   make R and the split by themselves for as many runs of chunks, and meet in the final sum.  No barrier.
//   up to  96 FLOs  CW = 2: two tiles of 64 points; up to 192 FLOs CW = 4: one tile.  More FLOs: further blocks.
// With CW > 1 the waves have roles, because the sums leave no room for both R and H operands loaded ahead (waves that did
// everything in turn ran 192 FLOs, 5.2e5 rows, 2.0e5 points at 272 ms, the registers spilling, against 192 ms with roles):
// waves 0-3 are consumers, CW on each tile, whose H operands are loaded one K step ahead; waves 4-7 producers, CW on each
// tile.  While the consumers run the MFMAs of chunk c, the producers work ahead, one barrier per chunk of 64 Hermite rows.
// CW = 2: they split R of chunk c + 1 into A operands and make R of chunk c + 2 (FP32, lane = point), both in two LDS
// buffers.  CW = 4: they make R of a pair of chunks in one phase (two, three or six groups of L = 4, 3, 2 do not share out over
// four waves, twice as many do) and split the pair in the next, A operands in three buffers.  The producers have the
// higher wave priority: their VALU instructions fit beside the consumer's MFMAs, and a late producer holds up all.
// The FP32 accumulators go into the FP64 sums at the chunks marked flush (every 256 or more rows), so the sums do not
// depend on the split.
// Measured, three pieces, against 16-wave blocks in which two waves of every block staged H through LDS: 10 FLOs (289 groups,
// 3.4e4 points) 0.279 -> 0.097 ms; 30 FLOs (1686, 1.2e5) 2.98 -> 1.18; 48 FLOs (4163, 1.9e5) 12.6 -> 5.1; 64 FLOs (7371,
// 2.4e5) 25.8 -> 17.5; 96 FLOs (15750, 3.7e5) 96.0 -> 68.2; 120 FLOs (24241, 3.1e5) 104 -> 85.5; 192 FLOs (60795, 2.0e5)
// 242 -> 192.  With CW = 1 making R bounds the loop (32 and 48 FLOs take nearly the same time per row and point).  With
// CW = 4 the MFMAs are 57% busy there (52% by counters at 7.4e5 points, 5.7e5 rows): of the 192 ms the MFMAs alone need 111,
// with A from LDS 118, with the FP64 sums 130, with H from L2 (three quarters of a gigabyte per tile, 96% hits) 168; the rest
// is what the producers take from the consumers.  In far chunks the product with the third piece of H runs on zeros.
// ---------------------------------------------------------------------------------------------------
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef unsigned v4w __attribute__((ext_vector_type(4)));

template <int NP>
__device__ __forceinline__ void split_bf16(double x, __bf16 *out, int64_t stride) {
    double r = x;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const __bf16 b = (__bf16)(float)r;
        out[p * stride] = b;
        r -= (double)(float)b;
    }
}

// Hs[p][g][ct][lane][e]: piece p of H row 32g + 8*(lane/16) + e, column 16ct + lane%16 (zero-extended rows and
// columns); one block per chunk of the bf16 chunk list
template <int NP>
__global__ void k_split_h(const ChunkDev *__restrict__ chunks, const double *__restrict__ H, int ldh, int nF,
                          int64_t nsteps, __bf16 *__restrict__ Hs) {
    const ChunkDev ch = chunks[blockIdx.x];
    const int rpg = chunk_rpg(ch.L), nt = ntuv(chunk_herm(ch.L)), roff = chunk_roff(ch.L);
    const int nreal = (ch.pe - ch.pb) * rpg;
    const int nct = ldh / 16;
    for (int e = threadIdx.x; e < ldh * ch.kr; e += blockDim.x) {
        const int f = e / ch.kr, r = e - f * ch.kr;
        // chunk row r: row roff + r % rpg of group r / rpg, whose Hermite block starts nt rows after the previous one
        const int64_t hr = ch.hrow0 + (int64_t)(r / rpg) * nt + roff + r % rpg;
        const double v = (r < nreal && f < nF) ? H[hr * ldh + f] : 0.0;
        const int64_t R = ch.prow0 + r;
        const int64_t idx = ((R / 32) * nct + f / 16) * 512 + (16 * ((R % 32) / 8) + f % 16) * 8 + R % 8;
        split_bf16<NP>(v, Hs + idx, nsteps * nct * 512);
    }
}

// Far-chunk bits, one block of 256 threads per 64-point tile.  The tile's centroid o and radius rho (largest distance
// of its points from o) bound every point's distance to a group centre P from below by |P - o| - rho, so
// p (|P - o| - rho)^2 bounds T = p|r - P|^2 of every (point, group) pair; a chunk is far when the bound of each of its
// groups exceeds tfar.  Each wave assembles 64 chunk bits with one ballot.
__global__ void __launch_bounds__(256) k_far_bits(const double *__restrict__ X, const double *__restrict__ Y,
                                                  const double *__restrict__ Z, int64_t M,
                                                  const ChunkDev *__restrict__ chunks, int nchunks,
                                                  const double4 *__restrict__ pP, double tfar, int farw,
                                                  unsigned *__restrict__ far, double *__restrict__ farrows) {
    __shared__ double geo[4];
    const int64_t t = blockIdx.x, k0 = t * 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (wave == 0) {
        const int64_t k = k0 + lane;
        const bool valid = k < M;
        const double x = valid ? X[k] : 0.0, y = valid ? Y[k] : 0.0, z = valid ? Z[k] : 0.0;
        double sx = x, sy = y, sz = z, n = valid ? 1.0 : 0.0;
        for (int o = 32; o > 0; o >>= 1) {
            sx += __shfl_xor(sx, o);
            sy += __shfl_xor(sy, o);
            sz += __shfl_xor(sz, o);
            n += __shfl_xor(n, o);
        }
        const double cx = sx / n, cy = sy / n, cz = sz / n;
        double d = valid ? sqrt((x - cx) * (x - cx) + (y - cy) * (y - cy) + (z - cz) * (z - cz)) : 0.0;
        for (int o = 32; o > 0; o >>= 1) d = fmax(d, __shfl_xor(d, o));
        if (lane == 0) {
            geo[0] = cx;
            geo[1] = cy;
            geo[2] = cz;
            geo[3] = d;
        }
    }
    __syncthreads();
    const double cx = geo[0], cy = geo[1], cz = geo[2], rho = geo[3];
    double rows = 0.0;
    for (int base = wave * 64; base < farw * 32; base += 256) {
        const int c = base + lane;
        bool is_far = false;
        if (c < nchunks) {
            const ChunkDev ch = chunks[c];
            double tmin = INFINITY;
            for (int g = ch.pb; g < ch.pe; ++g) {
                const double4 q = pP[g];
                const double dx = q.x - cx, dy = q.y - cy, dz = q.z - cz;
                const double d = fmax(sqrt(dx * dx + dy * dy + dz * dz) - rho, 0.0);
                tmin = fmin(tmin, q.w * d * d);
            }
            is_far = tmin > tfar;
            if (is_far) rows += ch.kr;
        }
        const unsigned long long m = __ballot(is_far);
        const int w = base / 32;
        if (lane == 0) far[t * farw + w] = (unsigned)m;
        if (lane == 1 && w + 1 < farw) far[t * farw + w + 1] = (unsigned)(m >> 32);
    }
    for (int o = 32; o > 0; o >>= 1) rows += __shfl_xor(rows, o);
    if (lane == 0 && rows > 0.0) atomicAdd(farrows, rows);
}

void launch_far_bits(const double *x, const double *y, const double *z, int64_t M, const ChunkDev *chunks,
                     int nchunks, const double4 *pairP, double tfar, int farw, unsigned *far, double *farrows,
                     hipStream_t s) {
    launch_fill_zero(farrows, 1, s);
    if (M <= 0 || farw <= 0) return;
    hipLaunchKernelGGL(k_far_bits, dim3((unsigned)((M + 63) / 64)), dim3(256), 0, s, x, y, z, M, chunks, nchunks,
                       pairP, tfar, farw, far, farrows);
}

// A operand of one K step: the 8 FP32 rows of this lane's point split into NP bf16 pieces, each the rounded
// remainder of the previous ones, so that the pieces shrink by 2^-8 each and the last remainder is below 2^-8 of
// the last piece.  (An exact split by truncation, keeping the upper 16 bits of each remainder, is 1% faster here
// but its pieces shrink only by 2^-7, which triples the worst dropped cross product.)
// Rows go two at a time through one packed conversion (v_cvt_pk_bf16_f32, round to nearest even like the scalar cast);
// v_dot2_f32_bf16 with (-1, 0) or (0, -1) subtracts one half of the packed word from its row (an exact difference: checked
// bit for bit against the FP32 subtraction over 2^-149 .. 2^40), so a piece of two rows costs 3 VALU operations, where
// shift, mask and two subtractions would make it 5.  The constants go through registers: as an inline constant -1.0 they
// would be read as one 32-bit value.
template <int NP>
__device__ __forceinline__ void split_a(v4f x0, v4f x1, v8bf (&a)[NP]) {
    float r[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
    unsigned lo = 0x0000bf80u, hi = 0xbf800000u;
    asm("" : "+s"(lo), "+s"(hi));
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        v4w w;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const v2bf u = __builtin_convertvector((v2f){r[2 * e], r[2 * e + 1]}, v2bf);
            w[e] = __builtin_bit_cast(unsigned, u);
            if (p + 1 < NP) {
                r[2 * e] = __builtin_amdgcn_fdot2_f32_bf16(u, __builtin_bit_cast(v2bf, lo), r[2 * e], false);
                r[2 * e + 1] = __builtin_amdgcn_fdot2_f32_bf16(u, __builtin_bit_cast(v2bf, hi), r[2 * e + 1], false);
            }
        }
        a[p] = __builtin_bit_cast(v8bf, w);
    }
}

// R of a chunk in LDS: 64 rows of 64 points in FP32.  PAD: 68 floats per point (16-byte accesses free of conflicts, offsets
// inside a group immediate); else 64 floats per point whose 16-byte slots are permuted by the point (CW = 2, where the
// padding does not fit).
template <bool PAD>
constexpr int bf_rsize = 64 * (PAD ? 68 : 64);
template <bool PAD>
__device__ __forceinline__ int r_at(int point, int row) {
    return PAD ? point * 68 + row : point * 64 + (((row >> 2) ^ (point & 15)) << 2) + (row & 3);
}

template <int NP, int CW>
struct BfTile {                         // LDS of one 64-point tile with CW > 1
    float R[2][bf_rsize<CW == 4>];
    v8bf A[CW == 4 ? 3 : 2][2][4][NP][64];  // A operands [buffer][K step][point tile][piece][lane]
};
constexpr int kBfTab = kBoysRows * kBoysCols * 4;  // the FP32 Boys table, in LDS with CW = 4
template <int NP, int CW>
constexpr int bf_lds = CW == 1 ? 8 * bf_rsize<true> * 4 : (4 / CW) * (int)sizeof(BfTile<NP, CW>) + (CW == 4 ? kBfTab : 0);
template <int NP>
constexpr int bf_lds_all = bf_lds<NP, 1> > bf_lds<NP, 2> && bf_lds<NP, 1> > bf_lds<NP, 4> ? bf_lds<NP, 1>
                           : bf_lds<NP, 2> > bf_lds<NP, 4>                                ? bf_lds<NP, 2>
                                                                                          : bf_lds<NP, 4>;
constexpr int kBfOut = 16 * 66;  // one column tile of FP64 sums in the epilogue, per wave

// hermite_R<L, float> of NG groups at once: the same operations, ordered so that two groups' chains overlap.  The far branch
// of the Boys functions (12 VALU instructions) is taken by every lane, the near one (table) if a lane of the wave needs it.
// TAIL: only the last three rows of L = 4, R_022, R_013 and R_004 (chunk type 6), which need 15 of the 65 steps.
template <int L, int NG, bool TAIL>
__device__ __forceinline__ void hermite_Rn(const float *p, const float (*X)[3], const float *__restrict__ tab,
                                           float (*R)[ntuv(L)]) {
    constexpr int TOP = L < 2 ? 2 : L;
    float T[NG], eT[NG], F[NG][TOP + 1];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        T[g] = p[g] * __builtin_fmaf(X[g][2], X[g][2], __builtin_fmaf(X[g][0], X[g][0], X[g][1] * X[g][1]));
        eT[g] = __expf(-T[g]);
        boys32_far<TOP>(T[g], eT[g], F[g]);
    }
    if (__any(!(T[0] > 16.0f) || !(T[NG - 1] > 16.0f))) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const bool far = T[g] > 16.0f;
            float N[TOP + 1];
            boys32_near<TOP>(far ? 0.0f : T[g], eT[g], tab, N);
#pragma unroll
            for (int m = 0; m <= TOP; ++m) F[g][m] = far ? F[g][m] : N[m];
        }
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        float pw[L + 1];
        pw[0] = 1.0f;
#pragma unroll
        for (int n = 1; n <= L; ++n) pw[n] = pw[n - 1] * (-2.0f * p[g]);
        if constexpr (TAIL) {
            const float Y = X[g][1], Z = X[g][2];
            const float a = pw[3] * F[g][3], b = a * Z;                          // R_000 of level 3, R_001 of level 2
            const float d = __builtin_fmaf(pw[4] * F[g][4] * Z, Z, a);           // R_002 of level 2
            const float e = __builtin_fmaf(2.0f, b, d * Z);                      // R_003 of level 1
            const float f = __builtin_fmaf(pw[2], F[g][2], b * Z);               // R_002 of level 1
            R[g][32] = __builtin_fmaf(d * Y, Y, f);
            R[g][33] = e * Y;
            R[g][34] = __builtin_fmaf(3.0f, f, e * Z);
        } else {
            R[g][0] = pw[L] * F[g][L];
            rlevels<L, L - 1, float>(R[g], X[g][0], X[g][1], X[g][2], F[g], pw);
        }
    }
}

// Consecutive groups of one chunk type, [pb, pb + np): those from np0 on belong to the next chunk, whose R lies bf_rsize
// further.  P: the records of the first two this wave makes (bf_records).
struct BfGroups {
    int type, pb, np, np0;
};
__device__ __forceinline__ v4d bf_record(const double4 *__restrict__ pP, const BfGroups &G, int g) {
    return cload(reinterpret_cast<const v4d *>(pP + G.pb + min(g, G.np - 1)));
}
// R of NG groups, g0 and g0 + step (rows RPG g .. of the chunk hold rows ROFF .. of its group g), for this lane's point; P
// their centres and exponents
template <bool PAD, int L, int RPG, int ROFF, int NG>
__device__ __forceinline__ void bf_groups(const v4d *P, const BfGroups &G, int g0, int step, int lane, double px, double py, double pz,
                                          const float *__restrict__ tab, float *__restrict__ R0) {
    float p[NG], X[NG][3], r[NG][ntuv(L)];
#pragma unroll
    for (int e = 0; e < NG; ++e) {
        p[e] = (float)P[e].w;
        X[e][0] = (float)(P[e].x - px);
        X[e][1] = (float)(P[e].y - py);
        X[e][2] = (float)(P[e].z - pz);
    }
    hermite_Rn<L, NG, ROFF == 32>(p, X, tab, r);
#pragma unroll
    for (int e = 0; e < NG; ++e) {
        const int ge = g0 + e * step, row0 = (ge < G.np0 ? ge : ge - G.np0) * RPG;
        float *__restrict__ R = R0 + (ge < G.np0 ? 0 : bf_rsize<PAD>);
        if constexpr (RPG % 4 == 0) {
#pragma unroll
            for (int t = 0; t < RPG; t += 4)
                *(v4f *)(R + r_at<PAD>(lane, row0 + t)) =
                    v4f{r[e][ROFF + t], r[e][ROFF + t + 1], r[e][ROFF + t + 2], r[e][ROFF + t + 3]};
        } else if constexpr (RPG % 2 == 0) {
#pragma unroll
            for (int t = 0; t < RPG; t += 2) *(v2f *)(R + r_at<PAD>(lane, row0 + t)) = v2f{r[e][ROFF + t], r[e][ROFF + t + 1]};
        } else {
#pragma unroll
            for (int t = 0; t < RPG; ++t) R[r_at<PAD>(lane, row0 + t)] = r[e][ROFF + t];
        }
    }
}
// groups first, first + step, ..., two at a time, the next two's records on their way meanwhile
template <bool PAD, int L, int RPG = ntuv(L), int ROFF = 0>
__device__ __forceinline__ void bf_chunk_R(const BfGroups &G, int first, int step, const double4 *__restrict__ pP,
                                           v4d (&P)[2], int lane, double px, double py, double pz,
                                           const float *__restrict__ tab, float *__restrict__ R) {
    int g = first;
    for (; g + step < G.np; g += 2 * step) {
        const v4d Q[2] = {bf_record(pP, G, g + 2 * step), bf_record(pP, G, g + 3 * step)};
        __builtin_amdgcn_sched_barrier(0);
        bf_groups<PAD, L, RPG, ROFF, 2>(P, G, g, step, lane, px, py, pz, tab, R);
        P[0] = Q[0];
        P[1] = Q[1];
    }
    if (g < G.np) bf_groups<PAD, L, RPG, ROFF, 1>(P, G, g, step, lane, px, py, pz, tab, R);
}

template <bool PAD>
__device__ __forceinline__ void bf_make_R(const BfGroups &G, int first, int step, const double4 *__restrict__ pP,
                                          v4d (&P)[2], int lane, double px, double py, double pz,
                                          const float *__restrict__ tab, float *__restrict__ R) {
    switch (G.type) {
        case 0: bf_chunk_R<PAD, 0>(G, first, step, pP, P, lane, px, py, pz, tab, R); break;
        case 1: bf_chunk_R<PAD, 1>(G, first, step, pP, P, lane, px, py, pz, tab, R); break;
        case 2: bf_chunk_R<PAD, 2>(G, first, step, pP, P, lane, px, py, pz, tab, R); break;
        case 3: bf_chunk_R<PAD, 3>(G, first, step, pP, P, lane, px, py, pz, tab, R); break;
        case 5: bf_chunk_R<PAD, 4, chunk_rpg(5), chunk_roff(5)>(G, first, step, pP, P, lane, px, py, pz, tab, R); break;
        default: bf_chunk_R<PAD, 4, chunk_rpg(6), chunk_roff(6)>(G, first, step, pP, P, lane, px, py, pz, tab, R); break;
    }
}
__device__ __forceinline__ BfGroups bf_chunk_groups(const ChunkDev &c) { return BfGroups{c.L, c.pb, c.pe - c.pb, c.pe - c.pb}; }
// rows 32 q + 8 lr .. + 7 of point 16 i + lc, split
template <int NP, bool PAD>
__device__ __forceinline__ void bf_rows8(const float *R, int i, int q, int lr, int lc, v8bf (&a)[NP]) {
    const int pt = 16 * i + lc, row = 32 * q + 8 * lr;
    split_a<NP>(*(const v4f *)(R + r_at<PAD>(pt, row)), *(const v4f *)(R + r_at<PAD>(pt, row + 4)), a);
}

template <int NP, int NT>
struct BfAcc {
    v4f acc[4][NT];
    double sum[4][NT][4];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    acc[i][j][r] = 0.0f;
                    sum[i][j][r] = 0.0;
                }
    }
    __device__ __forceinline__ void flush() {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    sum[i][j][r] += (double)acc[i][j][r];
                    acc[i][j][r] = 0.0f;
                }
    }
    // one K step: products of the pieces in the order a0b0, a0b1, a1b0 (a0b2, a1b1, a2b0) for every accumulator, one point
    // tile after the other.  next_a(i, a) gives the A operand of tile i, i = 4: of the next K step's tile 0 (or nothing);
    // it is issued before the MFMAs of tile i - 1 and, with HOLD, the scheduler is kept from moving it down to its use.
    // a[0]: the operand of tile 0.
    template <bool HOLD, typename F>
    __device__ __forceinline__ void step(v8bf (&a)[2][NP], F next_a, const v8bf (&b)[NT][NP]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            next_a(i + 1, a[(i + 1) & 1]);
            if constexpr (HOLD) __builtin_amdgcn_sched_barrier(0);
#define FLOSIC_BF(pa, pb)                          \
    _Pragma("unroll") for (int j = 0; j < NT; ++j) \
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i & 1][pa], b[j][pb], acc[i][j], 0, 0, 0)
            FLOSIC_BF(0, 0);
            FLOSIC_BF(0, 1);
            FLOSIC_BF(1, 0);
            if constexpr (NP == 3) {
                FLOSIC_BF(0, 2);
                FLOSIC_BF(1, 1);
                FLOSIC_BF(2, 0);
            }
#undef FLOSIC_BF
            if constexpr (HOLD) __builtin_amdgcn_sched_barrier(0);
        }
    }
};
// B operands of the K step at h (piece 0 of this wave's first column tile).  In a far chunk the third piece counts as zero:
// it is loaded from `zero` (this lane's place in a run of zeros), so that every K step issues the same loads and the waits
// for them can be counted.
template <int NP, int NT>
__device__ __forceinline__ void bf_load(v8bf (&b)[NT][NP], const char *h, int64_t pstride, bool far, const char *zero) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const char *src = p == 2 && far ? zero : h + p * pstride;
#pragma unroll
        for (int j = 0; j < NT; ++j) b[j][p] = gload((const v8bf *)(src + j * 1024));
    }
}
template <int NP>
__device__ __forceinline__ bool bf_far(const unsigned *far, int c) {  // far: this tile's chunk bits, or null
    if (NP != 3 || !far) return false;
    return (__builtin_amdgcn_readfirstlane(cload(far + (c >> 5))) >> (c & 31)) & 1u;
}

// Barrier between producers and consumers: this wave's LDS accesses are done, its global loads stay in flight (the fence
// of __syncthreads would wait for them)
__device__ __forceinline__ void role_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// Epilogue: one column tile of sums at a time through LDS, [column][66 points]: 512 contiguous bytes per store.  The sums of
// the RW runs of a tile (CW = 1) are added there and each stores 16 / RW columns.
template <int NP, int RW, int NT>
__device__ __forceinline__ void bf_store(unsigned char *__restrict__ lds, const CoulJob<__bf16> &J, const BfAcc<NP, NT> &A,
                                         int64_t kl, bool valid, int wave, int ct0, int ntmax) {
    const int lane = threadIdx.x & 63, lr = lane >> 4, lc = lane & 15, rg = wave % RW, w0 = wave - rg;
    double *o = reinterpret_cast<double *>(lds);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        if (j >= ntmax) break;
        __syncthreads();
        if (j < NT) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    o[wave * kBfOut + lc * 66 + i * 16 + 4 * lr + r] = A.sum[i][j < NT ? j : 0][r];
        }
        __syncthreads();
        if (j < NT) {
#pragma unroll
            for (int q = 0; q < 16 / RW; ++q) {
                const int col = rg * (16 / RW) + q, f = (ct0 + j) * 16 + col;
                double v = o[w0 * kBfOut + col * 66 + lane];
#pragma unroll
                for (int g = 1; g < RW; ++g) v += o[(w0 + g) * kBfOut + col * 66 + lane];
                if (f < J.nF && valid) gstore(J.V + (int64_t)f * J.ldv + kl, v);
            }
        }
    }
}

// this lane's point of a tile
struct BfPoint {
    int64_t k;
    bool valid;
    double x, y, z;
};
__device__ __forceinline__ BfPoint bf_point(const CoulJob<__bf16> &J, int64_t tile) {
    BfPoint p;
    p.k = tile * 64 + (threadIdx.x & 63);
    p.valid = p.k < J.M;
    p.x = p.valid ? gload(J.X + p.k) : 0.0;
    p.y = p.valid ? gload(J.Y + p.k) : 0.0;
    p.z = p.valid ? gload(J.Z + p.k) : 0.0;
    return p;
}
__device__ __forceinline__ const unsigned *bf_far_row(const CoulJob<__bf16> &J, int64_t tile) {
    return J.far && tile * 64 < J.M ? J.far + tile * J.farw : nullptr;
}

// CW = 1: a wave on its own run of chunks (of RW), all columns
template <int NP, int NT, int RW>
__device__ __forceinline__ void bf_alone(unsigned char *__restrict__ lds, const CoulJob<__bf16> &J,
                                         const double *__restrict__ tab, int64_t tile, int wave, int ct0) {
    const int lane = threadIdx.x & 63, lr = lane >> 4, lc = lane & 15, rg = wave % RW;
    const BfPoint P = bf_point(J, tile);
    const float *ctab = (const float *)(tab + kBoysRows * kBoysCols);
    const char *zero = (const char *)(tab + kBoysTableDoubles) + lane * 16;
    float *R = reinterpret_cast<float *>(lds) + wave * bf_rsize<true>;
    const int c0 = J.rgc[rg * (kRunsBf16 / RW)], c1 = J.rgc[(rg + 1) * (kRunsBf16 / RW)];
    const unsigned *far = bf_far_row(J, tile);
    // rows of a chunk beyond its groups are never written and meet zero rows of H: they only have to be finite
    for (int i = lane; i < bf_rsize<true> / 4; i += 64) ((v4f *)R)[i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    wave_lds_sync();
    BfAcc<NP, NT> A;
    A.clear();
    const int64_t pstride = J.nsteps * J.nct * 1024, hstep = (int64_t)J.nct * 1024;
    const char *h = (const char *)J.H + ((int64_t)ct0 * 64 + lane) * 16;  // piece 0 of the next K step to be loaded
    v8bf b[NT][NP];
    if (c0 < c1) {
        h += (int64_t)(chunk_at(J.chunks, c0).prow0 / 32) * hstep;
        bf_load<NP, NT>(b, h, pstride, bf_far<NP>(far, c0), zero);
    }
    for (int c = c0; c < c1;) {
        int flush;
        do {
        const ChunkDev ch = chunk_at(J.chunks, c);
        __builtin_amdgcn_s_setprio(0);
        v4d rec[2] = {bf_record(J.pP, bf_chunk_groups(ch), 0), bf_record(J.pP, bf_chunk_groups(ch), 1)};
        bf_make_R<true>(bf_chunk_groups(ch), 0, 1, J.pP, rec, lane, P.x, P.y, P.z, ctab, R);
        __builtin_amdgcn_s_setprio(2);  // the MFMA half goes first (30 FLOs 1.26 -> 1.18 ms, 48 FLOs 5.26 -> 5.07)
        wave_lds_sync();
        const bool f = bf_far<NP>(far, c);
#pragma unroll 1
        for (int q = 0; q < 2; ++q) {
            auto next_a = [&](int i, v8bf(&x)[NP]) {
                if (i < 4) bf_rows8<NP, true>(R, i, q, lr, lc, x);
            };
            v8bf a[2][NP];
            next_a(0, a[0]);
            A.template step<true>(a, next_a, b);
            h += hstep;
            if (q == 0) bf_load<NP, NT>(b, h, pstride, f, zero);
            else if (c + 1 < c1) bf_load<NP, NT>(b, h, pstride, bf_far<NP>(far, c + 1), zero);
        }
        flush = ch.flush;
        ++c;
        wave_lds_sync();
        } while (!flush);
        A.flush();
    }
    bf_store<NP, RW, NT>(lds, J, A, P.k, P.valid, wave, ct0, NT);
}

template <int NP, int CW>
__device__ __forceinline__ void bf_producer(BfTile<NP, CW> &T, const CoulJob<__bf16> &J, const float *__restrict__ ctab,
                                            int64_t tile, int pi, int ntmax) {
    constexpr bool PAD = CW == 4;
    const int lane = threadIdx.x & 63, lr = lane >> 4, lc = lane & 15;
    const BfPoint P = bf_point(J, tile);
    const int n = J.nchunks;
    __builtin_amdgcn_s_setprio(2);  // a producer's VALU instructions go into the cycles in which the consumer's MFMA runs
    // rows of a chunk beyond its groups are never written and meet zero rows of H: they only have to be finite
    for (int i = pi * 64 + lane; i < bf_rsize<PAD> / 2; i += 64 * CW) ((v4f *)T.R[0])[i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    role_barrier();
    auto split = [&](int c, int slot) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int e = 0; e < 4 / CW; ++e) {
                const int i = pi * (4 / CW) + e;
                v8bf a[NP];
                bf_rows8<NP, PAD>(T.R[c & 1], i, q, lr, lc, a);
#pragma unroll
                for (int p = 0; p < NP; ++p) T.A[slot][q][i][p][lane] = a[p];
            }
    };
    if constexpr (CW == 4) {  // chunks in pairs (even, odd): R of a pair in one phase, its split in the next
        BfGroups G[2];
        v4d rec[2];
        int parts;
        auto plan = [&](int c) {  // the groups of chunks c and c + 1, in one list where they follow one another
            const ChunkDev x = chunk_at(J.chunks, c);
            G[0] = G[1] = bf_chunk_groups(x);
            parts = 1;
            if (c + 1 < n) {
                const ChunkDev y = chunk_at(J.chunks, c + 1);
                if (y.L == x.L && y.pb == x.pe) {
                    G[0].np += y.pe - y.pb;
                } else {
                    G[1] = bf_chunk_groups(y);
                    parts = 2;
                }
            }
#pragma unroll
            for (int e = 0; e < 2; ++e) rec[e] = bf_record(J.pP, G[0], pi + 4 * e);
        };
        auto make = [&]() {
            bf_make_R<PAD>(G[0], pi, 4, J.pP, rec, lane, P.x, P.y, P.z, ctab, T.R[0]);
            if (parts == 2) {
#pragma unroll
                for (int e = 0; e < 2; ++e) rec[e] = bf_record(J.pP, G[1], 3 - pi + 4 * e);
                bf_make_R<PAD>(G[1], 3 - pi, 4, J.pP, rec, lane, P.x, P.y, P.z, ctab, T.R[1]);
            }
        };
        plan(0);
        make();
        role_barrier();
        split(0, 0);
        if (n > 1) split(1, 1);
        if (n > 2) plan(2);
        role_barrier();
        for (int c = 0, slot = 0; c < n; ++c) {  // slot = c % 3
            slot = slot == 2 ? 0 : slot + 1;
            if (c & 1) {
                if (c + 1 < n) split(c + 1, slot);
                if (c + 2 < n) split(c + 2, slot == 2 ? 0 : slot + 1);
                if (c + 3 < n) plan(c + 3);
            } else if (c + 2 < n) {
                make();
            }
            role_barrier();
        }
    } else {
        auto make = [&](int c) {  // which producer begins changes from chunk to chunk
            const BfGroups G = bf_chunk_groups(chunk_at(J.chunks, c));
            const int first = (pi + c) % CW;
            v4d rec[2] = {bf_record(J.pP, G, first), bf_record(J.pP, G, first + CW)};
            bf_make_R<PAD>(G, first, CW, J.pP, rec, lane, P.x, P.y, P.z, ctab, T.R[c & 1]);
        };
        make(0);
        role_barrier();
        split(0, 0);
        if (n > 1) make(1);
        role_barrier();
        for (int c = 0; c < n; ++c) {
            if (c + 1 < n) split(c + 1, (c + 1) & 1);
            if (c + 2 < n) make(c + 2);
            role_barrier();
        }
    }
    for (int j = 0; j < ntmax; ++j) {  // the consumers' epilogue
        __syncthreads();
        __syncthreads();
    }
}

template <int NP, int CW, int NT>
__device__ __forceinline__ void bf_consumer(unsigned char *__restrict__ lds, BfTile<NP, CW> &T, const CoulJob<__bf16> &J,
                                            const char *zero, int64_t tile, int wave, int ct0, int ntmax) {
    const int lane = threadIdx.x & 63;
    const int64_t kl = tile * 64 + lane;
    const int n = J.nchunks;
    const unsigned *far = bf_far_row(J, tile);
    BfAcc<NP, NT> A;
    A.clear();
    const int64_t pstride = J.nsteps * J.nct * 1024, hstep = (int64_t)J.nct * 1024;
    const char *h = (const char *)J.H + ((int64_t)ct0 * 64 + lane) * 16;  // piece 0 of this chunk's first K step
    v8bf b0[NT][NP], b1[NT][NP];
    bool f = bf_far<NP>(far, 0);
    bf_load<NP, NT>(b0, h, pstride, f, zero);
    bf_load<NP, NT>(b1, h + hstep, pstride, f, zero);
    role_barrier();
    role_barrier();
    role_barrier();
    for (int c = 0, slot = 0; c < n;) {  // slot = c % 2 or 3
        int flush;
        do {  // up to the next flush, which the last chunk has: the sums are not live across a branch
        const bool more = c + 1 < n, fn = more && bf_far<NP>(far, c + 1);
        flush = __builtin_amdgcn_readfirstlane(cload(&J.chunks[c].flush));
        if (more) h += 2 * hstep;  // the last chunk's are loaded again
        const auto &As = T.A[slot];
        auto a0 = [&](int i, v8bf(&x)[NP]) {
#pragma unroll
            for (int p = 0; p < NP; ++p) x[p] = As[i >> 2][i & 3][p][lane];
        };
        auto a1 = [&](int i, v8bf(&x)[NP]) {
#pragma unroll
            for (int p = 0; p < NP; ++p)
                if (i < 4) x[p] = As[1][i & 3][p][lane];
        };
        v8bf a[2][NP];
        a0(0, a[0]);
        A.template step<CW == 4>(a, a0, b0);
        bf_load<NP, NT>(b0, h, pstride, fn, zero);
        A.template step<CW == 4>(a, a1, b1);
        bf_load<NP, NT>(b1, h + hstep, pstride, fn, zero);
        slot = slot == (CW == 4 ? 2 : 1) ? 0 : slot + 1;
        f = fn;
        ++c;
        role_barrier();
        } while (!flush);
        A.flush();
    }
    bf_store<NP, 1, NT>(lds, J, A, kl, kl < J.M, wave, ct0, ntmax);
}

// Waves per tile with CW = 1.  Two tiles of four waves share the H that they read at the same time, one tile of eight leaves
// less of the chip idle in the last round of 256 blocks: 48 FLOs, 2903 tiles 5.07 and 5.64 ms; 30 FLOs, 1816 tiles 1.18 and
// 1.24; 10 FLOs, 530 tiles 0.125 and 0.097.  So eight where that saves more than a tenth of the rounds (a round of two tiles
// counts twice).  In a batch the systems share a launch and only the last of them has such a round, yet the split is
// each system's own, so that it has the bits of its single launch.
__host__ __device__ inline int bf_runs(int64_t M) {
    const int64_t tiles = (M + 63) / 64;
    return 11 * ((tiles + 255) / 256) < 20 * ((tiles + 511) / 512) ? 8 : 4;
}
// Work item `item` of a system: 64-point tiles 2 item and 2 item + 1 (CW = 4: tile item), column block cb of ncb; the
// column tiles are shared out evenly over the blocks and over a block's column waves
template <int NP, int CW, int NTLO, int NTHI>
__device__ __forceinline__ void coulomb_tile_bf16(unsigned char *__restrict__ lds, const CoulJob<__bf16> &J,
                                                  const double *__restrict__ tab, int64_t item, int cb) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tb0 = J.nct * cb / J.ncb, tb = J.nct * (cb + 1) / J.ncb - tb0;
    if constexpr (CW == 1) {
        const bool one = bf_runs(J.M) == 8;  // one tile per block
        const int64_t tile = one ? item : 2 * item + wave / 4;
        if constexpr (NTHI >= 3) {
            if (tb == 3)
                return one ? bf_alone<NP, 3, 8>(lds, J, tab, tile, wave, tb0) : bf_alone<NP, 3, 4>(lds, J, tab, tile, wave, tb0);
        }
        if constexpr (NTLO <= 2 && NTHI >= 2) {
            if (tb == 2)
                return one ? bf_alone<NP, 2, 8>(lds, J, tab, tile, wave, tb0) : bf_alone<NP, 2, 4>(lds, J, tab, tile, wave, tb0);
        }
        if constexpr (NTLO <= 1) {
            if (tb == 1)
                return one ? bf_alone<NP, 1, 8>(lds, J, tab, tile, wave, tb0) : bf_alone<NP, 1, 4>(lds, J, tab, tile, wave, tb0);
        }
    } else {
        const int w = wave & 3, cw = w % CW, ntmax = (tb + CW - 1) / CW;
        const int64_t tile = CW == 2 ? 2 * item + w / 2 : item;
        BfTile<NP, CW> &T = reinterpret_cast<BfTile<NP, CW> *>(lds)[CW == 2 ? w / 2 : 0];
        const float *ctab = (const float *)(tab + kBoysRows * kBoysCols);
        if constexpr (CW == 4) {  // the table in LDS: R's lookups are the longest wait of a producer
            float *lt = reinterpret_cast<float *>(lds + sizeof(BfTile<NP, CW>));
            for (int i = threadIdx.x; i < kBfTab / 16; i += 512) ((v4f *)lt)[i] = ((const v4f *)ctab)[i];
            __syncthreads();
            if (wave >= 4) return bf_producer<NP, CW>(T, J, lt, tile, cw, ntmax);
        } else {
            if (wave >= 4) return bf_producer<NP, CW>(T, J, ctab, tile, cw, ntmax);
        }
        const int c0 = tb * cw / CW, nt = tb * (cw + 1) / CW - c0;
        const char *zero = (const char *)(tab + kBoysTableDoubles) + (threadIdx.x & 63) * 16;
        if constexpr (NTHI >= 3) {
            if (nt == 3) return bf_consumer<NP, CW, 3>(lds, T, J, zero, tile, wave, tb0 + c0, ntmax);
        }
        if constexpr (NTLO <= 2 && NTHI >= 2) {
            if (nt == 2) return bf_consumer<NP, CW, 2>(lds, T, J, zero, tile, wave, tb0 + c0, ntmax);
        }
        if constexpr (NTLO <= 1) {
            if (nt == 1) return bf_consumer<NP, CW, 1>(lds, T, J, zero, tile, wave, tb0 + c0, ntmax);
        }
    }
}

__host__ __device__ constexpr int bf_col_waves(int nct, int ncb) {
    const int tb = (nct + ncb - 1) / ncb;
    return tb <= 3 ? 1 : tb <= 6 ? 2 : 4;
}
int64_t bf16_items(int64_t M, int nct, int ncb) {
    const int64_t tiles = (M + 63) / 64;
    const int cw = bf_col_waves(nct, ncb);
    return cw == 2 || (cw == 1 && bf_runs(M) == 4) ? (tiles + 1) / 2 : tiles;
}

template <int NP, int CW, int NTM>
__global__ void __launch_bounds__(512, 2) k_coulomb_bf16(CoulJob<__bf16> J, const double *__restrict__ tab) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[bf_lds<NP, CW>];
    static_assert(split_covered(bf_col_waves, 192, CW, (NTM > 1 ? NTM - 1 : 1), NTM, true), "a wave's tiles have no instance");
    coulomb_tile_bf16<NP, CW, (NTM > 1 ? NTM - 1 : 1), NTM>(lds, J, tab, blockIdx.x, blockIdx.y);
}

template <int NP>
__global__ void __launch_bounds__(512, 2) k_coulomb_bf16_batch_all(const CoulJob<__bf16> *__restrict__ jobs,
                                                                   const int64_t *__restrict__ off, int njobs,
                                                                   const double *__restrict__ tab) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[bf_lds_all<NP>];
    int64_t local = 0;
    const int j = job_of_block(off, njobs, (int64_t)blockIdx.x, local);
    const CoulJob<__bf16> J = uniform_job(jobs, j);
    const int64_t item = local / J.ncb;
    const int cb = (int)(local - item * J.ncb);
    static_assert(split_covered(bf_col_waves, 192, 1, 1, 3, false) && split_covered(bf_col_waves, 192, 2, 1, 3, false) &&
                      split_covered(bf_col_waves, 192, 4, 1, 3, false), "a wave's tiles have no instance");
    switch (bf_col_waves(J.nct, J.ncb)) {
        case 1: coulomb_tile_bf16<NP, 1, 1, 3>(lds, J, tab, item, cb); break;
        // blocks of 64 columns share 7, 10, 11 .. tiles out as three and four: the waves of three hold one and two
        case 2: coulomb_tile_bf16<NP, 2, 1, 3>(lds, J, tab, item, cb); break;
        default: coulomb_tile_bf16<NP, 4, 1, 3>(lds, J, tab, item, cb); break;
    }
}

void launch_split_h(int npieces, const ChunkDev *chunks, int nchunks, const double *H, int ldh, int nF,
                    int64_t nsteps, __bf16 *Hs, hipStream_t s) {
    if (nchunks <= 0) return;
    if (npieces == 2)
        hipLaunchKernelGGL((k_split_h<2>), dim3(nchunks), dim3(256), 0, s, chunks, H, ldh, nF, nsteps, Hs);
    else
        hipLaunchKernelGGL((k_split_h<3>), dim3(nchunks), dim3(256), 0, s, chunks, H, ldh, nF, nsteps, Hs);
}

void launch_coulomb_bf16(int npieces, const CoulJob<__bf16> &J, const double *btab, hipStream_t s) {
    if (J.nchunks <= 0 || J.M <= 0) return;
    const int cw = bf_col_waves(J.nct, J.ncb), tb = (J.nct + J.ncb - 1) / J.ncb, ntm = (tb + cw - 1) / cw;
    const dim3 grid((unsigned)bf16_items(J.M, J.nct, J.ncb), (unsigned)J.ncb), blk(512);
#define FLOSIC_BFL(NP, CW, NTM) hipLaunchKernelGGL((k_coulomb_bf16<NP, CW, NTM>), grid, blk, 0, s, J, btab)
#define FLOSIC_BFN(NP)                           \
    switch (10 * cw + ntm) {                     \
        case 11: FLOSIC_BFL(NP, 1, 1); break;    \
        case 12: FLOSIC_BFL(NP, 1, 2); break;    \
        case 13: FLOSIC_BFL(NP, 1, 3); break;    \
        case 22: FLOSIC_BFL(NP, 2, 2); break;    \
        case 23: FLOSIC_BFL(NP, 2, 3); break;    \
        case 42: FLOSIC_BFL(NP, 4, 2); break;    \
        default: FLOSIC_BFL(NP, 4, 3); break;    \
    }
    if (npieces == 2) {
        FLOSIC_BFN(2)
    } else {
        FLOSIC_BFN(3)
    }
#undef FLOSIC_BFN
#undef FLOSIC_BFL
}

void launch_coulomb_bf16_batch_all(int npieces, const CoulJob<__bf16> *jobs, const int64_t *off, int njobs,
                                   int64_t items, const double *btab, hipStream_t s) {
    if (njobs <= 0 || items <= 0) return;
    if (npieces == 2)
        hipLaunchKernelGGL((k_coulomb_bf16_batch_all<2>), dim3((unsigned)items), dim3(512), 0, s, jobs, off, njobs, btab);
    else
        hipLaunchKernelGGL((k_coulomb_bf16_batch_all<3>), dim3((unsigned)items), dim3(512), 0, s, jobs, off, njobs, btab);
}

}  // namespace flosic
