// Split-BF16 Coulomb kernels (k_coulomb_ws_bf16 and its batched form) and the far-chunk bits.
#include "flosic_device.h"

namespace flosic {

constexpr int kCoulThreads = 1024;  // 16 wavefronts: R waves, copy waves, then 8 consumer waves
constexpr int kConsumerWave0 = 8;
// split-BF16: the consumers' FP32 accumulators go into their FP64 sums once at least this many Hermite rows have
// been accumulated (at chunk ends, and after the last chunk).  On the K=64 workload (same box): every 64 rows
// 1109 ms, 128 rows 1083 ms, 256 rows 1060-1070 ms, 512 rows 1053 ms, with |dE| against FP64 of 4.9e-7, 5.3e-7,
// 4.4e-7 and 6.2e-7 Ha; the flush (24 FP64 conversions and adds per consumer lane) is VALU work that the kernel's
// sub-steps wait for.  (The FP32 MFMA form keeps its flush per chunk: every 256 rows saved it under 1% there.)
constexpr int kFlushRowsBf16 = 256;
constexpr int kSlotsReg = 2;  // split-BF16: H staged through the copy waves' registers, the sub-step in use and the next

// position in the chunk / sub-step sequence
struct SubStep {
    int c, q;
};
__device__ __forceinline__ void advance(SubStep &p, const ChunkDev *chunks, int sr) {
    if (++p.q * sr >= chunk_at(chunks, p.c).kr) {
        p.q = 0;
        ++p.c;
    }
}

// R of the groups [np*q/nq, np*(q+1)/nq) of chunk `ch` (share q of nq) for the block's 64 points: R wave rw of
// nrw takes every nrw-th group (wave-uniform, so the group's centre and exponent are scalar loads) and lane l
// the point k0 + l, whose coordinates (px, py, pz) stay in registers.  LAYOUT 0: Rl[row * LD + point] in T;
// LAYOUT 2: Rl[point * LD + row] in T.  Share 0 also zeroes the rows beyond the groups.
// R is computed in FP64 for the FP64 form and in FP32 for the FP32 and split-BF16 operands, with the Boys table of
// that precision (the FP32 copy follows the FP64 table in device memory; the split-BF16 kernel reads it from LDS)
// RPG rows per group from Hermite row ROFF on (the whole group by default; the split-BF16 list's L = 4 head / tail
// chunks take rows [0, 32) / [32, 35) of each group, see chunk_rpg)
template <int L, typename T, int LD, int LAYOUT, int NP, int RPG = ntuv(L), int ROFF = 0>
__device__ __forceinline__ void chunk_R(int rw, int nrw, int lane, double px, double py, double pz, bool valid, int q,
                                        int nq, const ChunkDev &ch, const double4 *__restrict__ pP,
                                        const RType<T> *__restrict__ ctab, T *Rl) {
    constexpr int nt = ntuv(L);
    static_assert(ROFF + RPG <= nt, "chunk rows beyond the group's Hermite block");
    using C = RType<T>;
    const int np = ch.pe - ch.pb;
    const int glo = np * q / nq, ghi = np * (q + 1) / nq;
    for (int g = glo + rw; g < ghi; g += nrw) {
        const v4d P = gload(reinterpret_cast<const v4d *>(pP + ch.pb + g));  // x, y, z, p
        // lanes past the mesh end (valid false, coordinates 0) compute finite values too: an A row feeds only its own
        // point's output row, which is never stored, so no lane needs its R zeroed (that took nt moves per group)
        C R[nt];
        hermite_R<L, C>((C)P.w, (C)(P.x - px), (C)(P.y - py), (C)(P.z - pz), ctab, R);
#pragma unroll
        for (int t = 0; t < RPG; ++t) {
            if constexpr (LAYOUT == 0)
                Rl[(g * RPG + t) * LD + lane] = (T)R[ROFF + t];
            else
                Rl[lane * LD + g * RPG + t] = (T)R[ROFF + t];
        }
    }
    if (q == 0)
        for (int r = np * RPG + rw; r < ch.kr; r += nrw) {
            if constexpr (LAYOUT == 0)
                Rl[r * LD + lane] = (T)0;
            else
                Rl[lane * LD + r] = (T)0;
        }
}

template <typename T, int LD, int LAYOUT, int NP>
__device__ __forceinline__ void produce_R(int rw, int nrw, int lane, double px, double py, double pz, bool valid,
                                          int q, int nq, const ChunkDev &ch, const double4 *__restrict__ pP,
                                          const RType<T> *__restrict__ tab, T *Rl) {
    switch (ch.L) {
        case 0: chunk_R<0, T, LD, LAYOUT, NP>(rw, nrw, lane, px, py, pz, valid, q, nq, ch, pP, tab, Rl); break;
        case 1: chunk_R<1, T, LD, LAYOUT, NP>(rw, nrw, lane, px, py, pz, valid, q, nq, ch, pP, tab, Rl); break;
        case 2: chunk_R<2, T, LD, LAYOUT, NP>(rw, nrw, lane, px, py, pz, valid, q, nq, ch, pP, tab, Rl); break;
        case 3: chunk_R<3, T, LD, LAYOUT, NP>(rw, nrw, lane, px, py, pz, valid, q, nq, ch, pP, tab, Rl); break;
        case 4: chunk_R<4, T, LD, LAYOUT, NP>(rw, nrw, lane, px, py, pz, valid, q, nq, ch, pP, tab, Rl); break;
        case 5:
            chunk_R<4, T, LD, LAYOUT, NP, chunk_rpg(5), chunk_roff(5)>(rw, nrw, lane, px, py, pz, valid, q, nq, ch, pP,
                                                                      tab, Rl);
            break;
        default:
            chunk_R<4, T, LD, LAYOUT, NP, chunk_rpg(6), chunk_roff(6)>(rw, nrw, lane, px, py, pz, valid, q, nq, ch, pP,
                                                                      tab, Rl);
            break;
    }
}

// s_waitcnt lgkmcnt(0) alone (vmcnt 63, expcnt 7)
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xF | (7 << 4) | (0 << 8) | (3 << 14)); }

// ---------------------------------------------------------------------------------------------------
// Split-BF16 Coulomb.  x = x1 + x2 (+ x3) in bf16 pieces, so the product x*y is carried by x1y1 + x1y2 + x2y1
// (+ x1y3 + x2y2 + x3y1) at ~2^-16 (2^-24) relative error, every term on the 16x16x32 bf16 MFMA (lane l holds
// A[l%16][8*(l/16) .. +7], B[8*(l/16) .. +7][l%16]; FP32 register r holds D[4*(l/16) + r][l%16]).  Same block
// organisation as k_coulomb_ws with one 32-row K step per sub-step and consumer waves of 16 points x half the
// columns.  R is kept in LDS as FP32 [point][row]; each consumer splits its 8-row A operand when it loads it; H
// pieces come from k_split_h in operand order.  The copy waves stage H through their registers (ordinary 16-byte
// loads one sub-step ahead, 16-byte LDS stores into two slots): on the 36 KiB split-BF16 sub-steps this moves H
// faster than the asynchronous global->LDS loads of the FP kernels, which remain faster for their 24 KiB steps.
// ---------------------------------------------------------------------------------------------------
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

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
// Rows go two at a time through one packed conversion (v_cvt_pk_bf16_f32, round to nearest even like the scalar
// cast); a piece's bf16 value is back in FP32 by a shift (low half) or a mask (high half) of the packed word, so a
// piece of two rows costs 5 VALU operations and the split needs no repacking into the operand vector.
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef unsigned v4w __attribute__((ext_vector_type(4)));
template <int NP>
__device__ __forceinline__ void split_a(const float *src, v8bf (&a)[NP]) {
    const v4f x0 = *(const v4f *)src, x1 = *(const v4f *)(src + 4);
    float r[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        v4w w;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const unsigned u = __builtin_bit_cast(unsigned, __builtin_convertvector((v2f){r[2 * e], r[2 * e + 1]}, v2bf));
            w[e] = u;
            if (p + 1 < NP) {
                r[2 * e] -= __builtin_bit_cast(float, u << 16);
                r[2 * e + 1] -= __builtin_bit_cast(float, u & 0xffff0000u);
            }
        }
        a[p] = __builtin_bit_cast(v8bf, w);
    }
}

// The 1 KiB units (64 lanes x 16 bytes) of one staged K step that copy wave cw of NCPW moves, through registers:
// unit u = pc * NFB/16 + v is KiB v of piece pc's run for the block's columns, at LDS slot offset u KiB.
template <int NP, int NFB, int NCPW>
struct HUnits {
    static constexpr int UPP = NFB / 16, NU = NP * UPP, UPW = (NU + NCPW - 1) / NCPW;
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    v4u r[UPW];
    // the units of the sub-step whose piece-0 run for the block's columns starts at sub_base, the pieces pstride bytes
    // apart; npe: pieces read from H (NP, or 2 for a far chunk, whose third piece is staged as zeros)
    __device__ __forceinline__ void load_at(const char *sub_base, int64_t pstride, int cw, int lane, int npe) {
#pragma unroll
        for (int k = 0; k < UPW; ++k) {
            const int u = cw + k * NCPW;
            if (u < npe * UPP) {
                const int pc = u / UPP, v = u - pc * UPP;
                r[k] = gload((const v4u *)(sub_base + pc * pstride + v * 1024 + lane * 16));
            } else if (u < NU) {
                r[k] = v4u{0u, 0u, 0u, 0u};
            }
        }
    }
    __device__ __forceinline__ void store(__bf16 *slot, int cw, int lane) const {
#pragma unroll
        for (int k = 0; k < UPW; ++k) {
            const int u = cw + k * NCPW;
            if (u < NU) *(v4u *)((char *)slot + u * 1024 + lane * 16) = r[k];
        }
    }
};

// LDS of one split-BF16 Coulomb tile: the two FP32 R tiles, the ring of staged H sub-steps, the FP32 Boys table
template <int NP, int NFB>
struct Bf16TileLds {
    static constexpr int LDK = kChunkRowsBf16 + 4;  // FP32 point rows of 272 bytes: conflict-free 16-byte reads
    static constexpr int SLOT = NP * NFB * 32;      // bf16 elements of one staged K step
    __attribute__((aligned(16))) float Rf[2][64 * LDK];
    __attribute__((aligned(16))) __bf16 Hl[kSlotsReg][SLOT];
    __attribute__((aligned(16))) float Tb[kBoysRows * kBoysCols];
    unsigned Fl[NP == 3 ? kFarWords : 1];  // far-chunk bits of this tile (three-piece form)
};

// One 32-row K step of a consumer wave (16 points x NFB/2 columns): the A operand split into NPE pieces and the
// products of the pieces down to order 2^-8(NPE-1): 3 (a0b0, a0b1, a1b0) for NPE = 2, plus a0b2, a1b1, a2b0 for
// NPE = 3 (zero for a0b2 in a far chunk, whose staged third H piece is zero)
template <int NPE, int NFB>
__device__ __forceinline__ void bf16_substep(const float *Rrow, const __bf16 *Hs_, int cl0, int lane,
                                             v4f (&acc)[NFB / 32]) {
    v8bf a[NPE];
    split_a<NPE>(Rrow, a);
#pragma unroll
    for (int j = 0; j < NFB / 32; ++j) {
        v8bf b[NPE];
#pragma unroll
        for (int p = 0; p < NPE; ++p) b[p] = *(const v8bf *)(Hs_ + ((p * (NFB / 16) + cl0 + j) * 64 + lane) * 8);
        v4f cc = acc[j];
        cc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[0], cc, 0, 0, 0);
        cc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[1], cc, 0, 0, 0);
        cc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[0], cc, 0, 0, 0);
        if constexpr (NPE == 3) {
            cc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[2], cc, 0, 0, 0);
            cc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[1], cc, 0, 0, 0);
            cc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[2], b[0], cc, 0, 0, 0);
        }
        acc[j] = cc;
    }
}

// far: null, or the far-chunk bits of every tile (farw 32-bit words per tile, bit c of a tile's row set where every
// (point, group) pair of tile and chunk c has T = p|r - P|^2 above the far threshold): the three-piece form reads
// two H pieces of those chunks from memory and stages the third as zeros (H to ~2^-17 there, R still in three)
template <int NP, int NFB>
__device__ __forceinline__ void coulomb_tile_bf16(Bf16TileLds<NP, NFB> &L, const ChunkDev *__restrict__ chunks,
                                                  int nchunks, int64_t nsteps,
                                                  const double4 *__restrict__ pP, const __bf16 *__restrict__ Hs,
                                                  int nct, const double *__restrict__ X, const double *__restrict__ Y,
                                                  const double *__restrict__ Z, int64_t M, int nF,
                                                  double *__restrict__ V, int64_t ldv,
                                                  const double *__restrict__ tab, int64_t tile, int cb,
                                                  const unsigned *__restrict__ far, int farw) {
    constexpr int TP = 64, NCW = NFB / 32, SR = 32;  // consumer wave: 16 points x NFB/2 columns
    constexpr int NCPW = NP == 3 ? 2 : 1, NRW = kConsumerWave0 - NCPW;
    constexpr int LDK = Bf16TileLds<NP, NFB>::LDK;
    constexpr int SLOT = Bf16TileLds<NP, NFB>::SLOT;
    float(&Rf)[2][TP * LDK] = L.Rf;
    __bf16(&Hl)[kSlotsReg][SLOT] = L.Hl;
    float(&Tb)[kBoysRows * kBoysCols] = L.Tb;  // FP32 Boys table for the R waves
    const int64_t k0 = tile * TP;
    const int fb = cb * NFB;
    // the wave index through readfirstlane: the compiler then knows it (and every role, group, unit and tile index
    // derived from it) to be wave-uniform and keeps that arithmetic and the load addresses built on it scalar
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const bool use_far = NP == 3 && far != nullptr;
    {  // the table in LDS keeps the R waves' per-lane table lookups off the load path of the H copies
        const v4f *src = (const v4f *)(tab + kBoysRows * kBoysCols);
        for (int i = threadIdx.x; i < kBoysRows * kBoysCols / 4; i += kCoulThreads) ((v4f *)Tb)[i] = src[i];
        if (use_far)
            for (int i = threadIdx.x; i < farw; i += kCoulThreads) L.Fl[i] = gload(far + tile * farw + i);
        __syncthreads();
    }
    // H pieces read from memory for chunk c (uniform)
    auto pieces = [&](int c) -> int {
        if (!use_far) return NP;
        const unsigned w = __builtin_amdgcn_readfirstlane(L.Fl[c >> 5]);
        return (w >> (c & 31)) & 1u ? 2 : NP;
    };
    if (wave < NRW) {  // R waves: lane l works on point k0 + l throughout
        const int64_t k = k0 + lane;
        const bool valid = k < M;
        const double px = valid ? gload(X + k) : 0.0, py = valid ? gload(Y + k) : 0.0, pz = valid ? gload(Z + k) : 0.0;
        produce_R<float, LDK, 2, 1>(wave, NRW, lane, px, py, pz, valid, 0, 1, chunk_at(chunks, 0), pP, Tb, Rf[0]);
        __syncthreads();
        for (int c = 0; c < nchunks; ++c) {
            const int nsub = chunk_at(chunks, c).kr / SR;
            for (int q = 0; q < nsub; ++q) {
                if (c + 1 < nchunks)
                    produce_R<float, LDK, 2, 1>(wave, NRW, lane, px, py, pz, valid, q, nsub, chunk_at(chunks, c + 1),
                                                pP, Tb, Rf[(c + 1) & 1]);
                __syncthreads();
            }
        }
    } else if (wave < kConsumerWave0) {  // copy waves: H of sub-step gs + 2 is loaded in iteration gs, stored in gs + 1
        const int cw = wave - NRW;
        HUnits<NP, NFB, NCPW> h;
        SubStep nxt{0, 0};
        // H of sub-step g (chunk c, step q: g = prow0(c) / 32 + q, the sub-steps consecutive in the padded row space)
        // for the block's columns starts g * nct KiB after hb; the pieces' runs are pstride bytes apart
        const int64_t pstride = nsteps * nct * 1024;
        const char *hb = (const char *)(Hs + (fb / 16) * 512);
        int64_t gnext = 0;  // sub-step index of nxt
        h.load_at(hb, pstride, cw, lane, pieces(0));
        h.store(Hl[0], cw, lane);
        advance(nxt, chunks, SR);
        ++gnext;
        bool held = nxt.c < nchunks;  // h holds the next sub-step
        if (held) {
            h.load_at(hb + gnext * nct * 1024, pstride, cw, lane, pieces(nxt.c));
            advance(nxt, chunks, SR);
            ++gnext;
        }
        wait_lgkm0();
        __builtin_amdgcn_s_barrier();
        int gs = 0;
        for (int c = 0; c < nchunks; ++c) {
            const int nsub = chunk_at(chunks, c).kr / SR;
            for (int q = 0; q < nsub; ++q, ++gs) {
                if (held) h.store(Hl[(gs + 1) % kSlotsReg], cw, lane);
                held = nxt.c < nchunks;
                if (held) {
                    h.load_at(hb + gnext * nct * 1024, pstride, cw, lane, pieces(nxt.c));
                    advance(nxt, chunks, SR);
                    ++gnext;
                }
                // the stores must have landed; the loads just issued stay in flight across the barrier
                wait_lgkm0();
                __builtin_amdgcn_s_barrier();
            }
        }
    } else {
    const int cwv = wave - kConsumerWave0;
    const int lr = lane >> 4, lc = lane & 15;
    const int pw = (cwv >> 1) * 16;   // point tile of this wave
    const int cl0 = (cwv & 1) * NCW;  // first column tile of this wave inside the block
    v4f acc[NCW];
    double sum[NCW][4];
#pragma unroll
    for (int j = 0; j < NCW; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            acc[j][r] = 0.0f;
            sum[j][r] = 0.0;
        }
    __syncthreads();
    int gs = 0, since = 0;  // since: rows accumulated in FP32 since the last flush into the FP64 sums
    for (int c = 0; c < nchunks; ++c) {
        const int kr = chunk_at(chunks, c).kr, nsub = kr / SR;
        const float *R = Rf[c & 1];
        since += kr;
        const bool flush = since >= kFlushRowsBf16 || c + 1 == nchunks;
        if (flush) since = 0;
        for (int q = 0; q < nsub; ++q, ++gs) {
            bf16_substep<NP, NFB>(R + (pw + lc) * LDK + SR * q + 8 * lr, Hl[gs % kSlotsReg], cl0, lane, acc);
            if (flush && q + 1 == nsub) {
#pragma unroll
                for (int j = 0; j < NCW; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        sum[j][r] += (double)acc[j][r];
                        acc[j][r] = 0.0f;
                    }
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int j = 0; j < NCW; ++j) {
        const int f = fb + (cl0 + j) * 16 + lc;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t k = k0 + pw + 4 * lr + r;
            if (f < nF && k < M) gstore(V + (int64_t)f * ldv + k, sum[j][r]);
        }
    }
    }
}

template <int NP, int NFB>
__global__ void __launch_bounds__(kCoulThreads) k_coulomb_ws_bf16(CoulJob<__bf16> J, const double *__restrict__ tab) {
    __shared__ Bf16TileLds<NP, NFB> lds;
    coulomb_tile_bf16<NP, NFB>(lds, J.chunks, J.nchunks, J.nsteps, J.pP, (const __bf16 *)J.H, J.nct, J.X, J.Y, J.Z, J.M,
                               J.nF, J.V, J.ldv, tab, blockIdx.x, blockIdx.y, J.far, J.farw);
}

template <int NP>
constexpr size_t bf16_lds_bytes() {
    size_t b = sizeof(Bf16TileLds<NP, 64>);
    b = b > sizeof(Bf16TileLds<NP, 128>) ? b : sizeof(Bf16TileLds<NP, 128>);
    b = b > sizeof(Bf16TileLds<NP, 192>) ? b : sizeof(Bf16TileLds<NP, 192>);
    return b;
}
template <int NP>
__global__ void __launch_bounds__(kCoulThreads) k_coulomb_ws_bf16_batch_all(const CoulJob<__bf16> *__restrict__ jobs,
                                                                            const int64_t *__restrict__ off,
                                                                            int njobs, const double *__restrict__ tab) {
    __shared__ __attribute__((aligned(16))) unsigned char raw[bf16_lds_bytes<NP>()];
    int64_t local = 0;
    const int j = job_of_block(off, njobs, (int64_t)blockIdx.x, local);
    const CoulJob<__bf16> J = uniform_job(jobs, j);
    const int64_t tile = local / J.ncb;
    const int cb = (int)(local - tile * J.ncb);
#define FLOSIC_TILE_BF(NFB)                                                                                         \
    coulomb_tile_bf16<NP, NFB>(*reinterpret_cast<Bf16TileLds<NP, NFB> *>(raw), J.chunks, J.nchunks, J.nsteps, J.pP, \
                               (const __bf16 *)J.H, J.nct, J.X, J.Y, J.Z, J.M, J.nF, J.V, J.ldv, tab, tile, cb,  \
                               J.far, J.farw)
    switch (J.nfb) {
        case 64: FLOSIC_TILE_BF(64); break;
        case 128: FLOSIC_TILE_BF(128); break;
        default: FLOSIC_TILE_BF(192); break;
    }
#undef FLOSIC_TILE_BF
}

void launch_split_h(int npieces, const ChunkDev *chunks, int nchunks, const double *H, int ldh, int nF,
                    int64_t nsteps, __bf16 *Hs, hipStream_t s) {
    if (nchunks <= 0) return;
    if (npieces == 2)
        hipLaunchKernelGGL((k_split_h<2>), dim3(nchunks), dim3(256), 0, s, chunks, H, ldh, nF, nsteps, Hs);
    else
        hipLaunchKernelGGL((k_split_h<3>), dim3(nchunks), dim3(256), 0, s, chunks, H, ldh, nF, nsteps, Hs);
}

void launch_coulomb_bf16(int npieces, const ChunkDev *chunks, int nchunks, int64_t nsteps, const double4 *pairP,
                         const __bf16 *Hs, int ldh, const double *x, const double *y, const double *z, int64_t M,
                         const double *btab, int nF, double *V, int64_t ldv, hipStream_t s, int nfb,
                         const unsigned *far, int farw) {
    if (nchunks <= 0 || M <= 0) return;
    if (nfb <= 0) nfb = coulomb_cols_split(nF);
    const CoulJob<__bf16> J{chunks, nchunks, pairP, Hs, ldh / 16, x, y, z, M, nF, V, ldv, nsteps, ldh / nfb, nfb,
                            npieces == 3 ? far : nullptr, npieces == 3 ? farw : 0, FpSegs{}};
    const dim3 grid((unsigned)((M + 63) / 64), (unsigned)(ldh / nfb)), blk(kCoulThreads);
#define FLOSIC_WSB(NP, NFB) hipLaunchKernelGGL((k_coulomb_ws_bf16<NP, NFB>), grid, blk, 0, s, J, btab)
#define FLOSIC_WSB_NFB(NP)                        \
    switch (nfb) {                                \
        case 64: FLOSIC_WSB(NP, 64); break;       \
        case 128: FLOSIC_WSB(NP, 128); break;     \
        default: FLOSIC_WSB(NP, 192); break;      \
    }
    if (npieces == 2) {
        FLOSIC_WSB_NFB(2)
    } else {
        FLOSIC_WSB_NFB(3)
    }
#undef FLOSIC_WSB_NFB
#undef FLOSIC_WSB
}

void launch_coulomb_bf16_batch_all(int npieces, const CoulJob<__bf16> *jobs, const int64_t *off, int njobs,
                                   int64_t items, const double *btab, hipStream_t s) {
    if (njobs <= 0 || items <= 0) return;
    if (npieces == 2)
        hipLaunchKernelGGL((k_coulomb_ws_bf16_batch_all<2>), dim3((unsigned)items), dim3(kCoulThreads), 0, s, jobs, off,
                           njobs, btab);
    else
        hipLaunchKernelGGL((k_coulomb_ws_bf16_batch_all<3>), dim3((unsigned)items), dim3(kCoulThreads), 0, s, jobs, off,
                           njobs, btab);
}

}  // namespace flosic
