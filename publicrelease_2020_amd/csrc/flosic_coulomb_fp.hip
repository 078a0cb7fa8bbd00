// FP64 and FP32 MFMA Coulomb kernels (k_coulomb_ws and its batched form).
#include "flosic_device.h"

namespace flosic {

// ---------------------------------------------------------------------------------------------------
// MFMA Coulomb.  V[f][k] = sum_rows R[k][row] H[row][f]: R_tuv(p, P - r_k) is generated on the fly (FP64 Boys
// and Hermite recursion), H is the Hermite-coefficient matrix of every exponent-pair group for every FLO, stored
// in MFMA operand order.  Block = 16 wavefronts on a tile of TP = 64 points x NFB FLO columns (NFB covers all
// FLOs up to 256, so R is computed once per (point, group)).  A chunk of Hermite rows is consumed in sub-steps
// of SR rows; per sub-step, separated by one barrier:
//   * R waves generate their share of R of the next chunk into the other of two LDS tiles,
//   * copy waves move the H rows of the sub-step two ahead into a 3-slot LDS ring with asynchronous
//     global->LDS loads (global_load_lds_dwordx4: lane l of a wave lands at base + 16 l bytes), then wait until
//     the rows of the next sub-step have landed (vmcnt counts only their own copies),
//   * 8 consumer waves (2 point halves x 4 column quarters) run the MFMAs of the current sub-step from LDS.
// FP32 and split-BF16 accumulators are added into FP64 sums after every chunk.
// ---------------------------------------------------------------------------------------------------
constexpr int kCoulThreads = 1024;  // 16 wavefronts: R waves, copy waves, then 8 consumer waves
constexpr int kConsumerWave0 = 8;
constexpr int kSlots = 3;     // FP operand stream: ring of LDS slots filled by asynchronous global->LDS loads
typedef __attribute__((address_space(3))) void lds_void;

// s_waitcnt with vmcnt <= n and no wait on the other counters (gfx9 encoding: vmcnt bits 3:0 and 15:14)
template <int N>
__device__ __forceinline__ void wait_vm_le() {
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
__device__ __forceinline__ void wait_vm(int n) {
    switch (n) {
#define FLOSIC_W(k) \
    case k: wait_vm_le<k>(); break;
        FLOSIC_W(0) FLOSIC_W(1) FLOSIC_W(2) FLOSIC_W(3) FLOSIC_W(4) FLOSIC_W(5) FLOSIC_W(6) FLOSIC_W(7)
        FLOSIC_W(8) FLOSIC_W(9) FLOSIC_W(10) FLOSIC_W(11) FLOSIC_W(12) FLOSIC_W(13) FLOSIC_W(14) FLOSIC_W(15)
        FLOSIC_W(16) FLOSIC_W(17) FLOSIC_W(18) FLOSIC_W(19) FLOSIC_W(20) FLOSIC_W(21) FLOSIC_W(22) FLOSIC_W(23)
        FLOSIC_W(24) FLOSIC_W(25) FLOSIC_W(26) FLOSIC_W(27) FLOSIC_W(28) FLOSIC_W(29) FLOSIC_W(30) FLOSIC_W(31)
#undef FLOSIC_W
        default: wait_vm_le<0>(); break;
    }
}

// KiB units [0, units) of a contiguous 16-byte aligned global run into LDS; unit u goes to copy wave
// u % ncw; returns the number of loads this wave issued
__device__ __forceinline__ int lds_copy_async(const char *src, char *dst, int units, int cw, int ncw, int lane,
                                              int first) {
    int n = 0;
    for (int u = (cw - first % ncw + ncw) % ncw; u < units; u += ncw, ++n)
        __builtin_amdgcn_global_load_lds((const void *)(src + (size_t)u * 1024 + lane * 16),
                                         (lds_void *)(dst + (size_t)u * 1024), 16, 0, 0);
    return n;
}

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

// one wave64 fragment of H in operand order: lane l holds row 4s + l/16 and column 16*ct + l%16 (FP64/FP32)
template <typename T>
__global__ void k_frag_h(const ChunkDev *__restrict__ chunks, const double *__restrict__ H, int ldh, int nF,
                         T *__restrict__ Hf) {
    const ChunkDev ch = chunks[blockIdx.x];
    const int nreal = (ch.pe - ch.pb) * ntuv(ch.L);
    const int nct = ldh / 16;
    for (int e = threadIdx.x; e < ch.kr * ldh; e += blockDim.x) {
        const int r = e / ldh, f = e - r * ldh;
        const double v = (r < nreal && f < nF) ? H[(int64_t)(ch.hrow0 + r) * ldh + f] : 0.0;
        const int64_t s = (ch.prow0 + r) / 4;
        Hf[(s * nct + f / 16) * 64 + (r % 4) * 16 + f % 16] = (T)v;
    }
}

// R of the groups [np*q/nq, np*(q+1)/nq) of chunk `ch` (share q of nq) for the block's 64 points: R wave rw of
// nrw takes every nrw-th group (wave-uniform, so the group's centre and exponent are scalar loads) and lane l
// the point k0 + l, whose coordinates (px, py, pz) stay in registers.  LAYOUT 0: Rl[row * LD + point] in T;
// LAYOUT 2: Rl[point * LD + row] in T.  Share 0 also zeroes the rows beyond the groups.
// R is computed in FP64 for the FP64 form and in FP32 for the FP32 and split-BF16 operands, with the Boys table of
// that precision (the FP32 copy follows the FP64 table in device memory; the split-BF16 kernel reads it from LDS)
template <typename T>
using RType = typename std::conditional<sizeof(T) == 8, double, float>::type;

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

// H rows of sub-step p (FP operand stream, rows multiple of 4) for block columns [fb, fb + NFB) into an LDS slot
// laid out [step][NFB/16 column tiles][64 lanes]; returns this copy wave's load count
template <typename T, int NFB, int SR>
__device__ __forceinline__ int stage_h_fp(const ChunkDev *__restrict__ chunks, SubStep p, const T *__restrict__ Hf,
                                          int nct, int fb, T *slot, int cw, int ncw, int lane) {
    constexpr int UPS = NFB * 4 * (int)sizeof(T) / 1024;  // KiB per K step
    const ChunkDev ch = chunk_at(chunks, p.c);
    const int64_t r0 = ch.prow0 + (int64_t)p.q * SR;
    const int nstep = min(SR, ch.kr - p.q * SR) / 4;
    int n = 0;
    for (int s = 0; s < nstep; ++s) {
        const char *src = (const char *)(Hf + ((r0 / 4 + s) * (int64_t)nct + fb / 16) * 64);
        n += lds_copy_async(src, (char *)(slot + (size_t)s * NFB * 4), UPS, cw, ncw, lane, s * UPS);
    }
    return n;
}

// One (point tile, column block) of one system's Coulomb contraction, executed by a whole block.  All waves
// return from here together; the persistent batch kernel calls it once per work item.
// LDS of one FP Coulomb tile: the two R tiles and the ring of staged H sub-steps
template <typename T, int NFB>
struct FpTileLds {
    static constexpr int SR = sizeof(T) == 4 ? 32 : (NFB <= 192 ? 16 : 8);  // Hermite rows per sub-step
    static constexpr int LDR = 64 + (sizeof(T) == 8 ? 8 : 16);
    T Rl[2][kChunkRows * LDR];
    __attribute__((aligned(16))) T Hl[kSlots][SR * NFB];
};

template <typename T, int NFB>
__device__ __forceinline__ void coulomb_tile_fp(FpTileLds<T, NFB> &L, const ChunkDev *__restrict__ chunks, int nchunks,
                                                const double4 *__restrict__ pP, const T *__restrict__ Hf, int nct,
                                                const double *__restrict__ X, const double *__restrict__ Y,
                                                const double *__restrict__ Z, int64_t M, int nF,
                                                double *__restrict__ V, int64_t ldv, const double *__restrict__ tab,
                                                int64_t tile, int cb) {
    constexpr int TP = 64, NRT = 2, NCW = NFB / 64;  // consumer wave: 32 points x NFB/4 columns (TP = wave size)
    constexpr int SR = FpTileLds<T, NFB>::SR;        // Hermite rows per sub-step
    constexpr int NRW = 7, NCPW = 1;                 // R waves, copy waves
    constexpr int LDR = FpTileLds<T, NFB>::LDR;
    T(&Rl)[2][kChunkRows * LDR] = L.Rl;
    T(&Hl)[kSlots][SR * NFB] = L.Hl;
    using Tr = MfmaTraits<T>;
    using acc_t = typename Tr::acc;
    const int64_t k0 = tile * TP;
    const int fb = cb * NFB;
    // the wave index through readfirstlane: the compiler then knows it (and every role, group, unit and tile index
    // derived from it) to be wave-uniform and keeps that arithmetic and the load addresses built on it scalar
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (wave < NRW) {  // R waves: lane l works on point k0 + l throughout
        const int64_t k = k0 + lane;
        const bool valid = k < M;
        const double px = valid ? gload(X + k) : 0.0, py = valid ? gload(Y + k) : 0.0, pz = valid ? gload(Z + k) : 0.0;
        const RType<T> *ctab = sizeof(T) == 8 ? (const RType<T> *)tab : (const RType<T> *)(tab + kBoysRows * kBoysCols);
        produce_R<T, LDR, 0, 1>(wave, NRW, lane, px, py, pz, valid, 0, 1, chunk_at(chunks, 0), pP, ctab, Rl[0]);
        __syncthreads();
        for (int c = 0; c < nchunks; ++c) {
            const int nsub = (chunk_at(chunks, c).kr + SR - 1) / SR;
            for (int q = 0; q < nsub; ++q) {
                if (c + 1 < nchunks)
                    produce_R<T, LDR, 0, 1>(wave, NRW, lane, px, py, pz, valid, q, nsub, chunk_at(chunks, c + 1), pP,
                                            ctab, Rl[(c + 1) & 1]);
                __syncthreads();
            }
        }
    } else if (wave < kConsumerWave0) {  // copy waves: keep the sub-step two ahead in flight
        const int cw = wave - NRW;
        SubStep nxt{0, 0};
        int gs_ahead = 0, pend = 0;
        pend = stage_h_fp<T, NFB, SR>(chunks, nxt, Hf, nct, fb, Hl[0], cw, NCPW, lane);
        advance(nxt, chunks, SR);
        ++gs_ahead;
        if (nxt.c < nchunks) {
            pend = stage_h_fp<T, NFB, SR>(chunks, nxt, Hf, nct, fb, Hl[1], cw, NCPW, lane);
            advance(nxt, chunks, SR);
            ++gs_ahead;
        } else {
            pend = 0;
        }
        wait_vm(pend);  // sub-step 0 has landed
        // raw barrier: a __syncthreads() fence would also wait for the copies still in flight
        __builtin_amdgcn_s_barrier();
        for (int c = 0; c < nchunks; ++c) {
            const int nsub = (chunk_at(chunks, c).kr + SR - 1) / SR;
            for (int q = 0; q < nsub; ++q) {
                int issued = 0;
                if (nxt.c < nchunks) {
                    issued = stage_h_fp<T, NFB, SR>(chunks, nxt, Hf, nct, fb, Hl[gs_ahead % kSlots], cw, NCPW, lane);
                    advance(nxt, chunks, SR);
                    ++gs_ahead;
                }
                wait_vm(issued);  // everything but the newest sub-step has landed
                __builtin_amdgcn_s_barrier();
            }
        }
    } else {
    const int cwv = wave - kConsumerWave0;
    const int lr = lane >> 4, lc = lane & 15;
    const int pw = (cwv >> 2) * NRT * 16;  // first point of this wave
    const int cl0 = (cwv & 3) * NCW;        // first column tile of this wave inside the block
    acc_t acc[NRT][NCW];
    double sum[NRT][NCW][4];
#pragma unroll
    for (int i = 0; i < NRT; ++i)
#pragma unroll
        for (int j = 0; j < NCW; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                acc[i][j][r] = (T)0;
                sum[i][j][r] = 0.0;
            }
    __syncthreads();
    int gs = 0;
    for (int c = 0; c < nchunks; ++c) {
        const int kr = chunk_at(chunks, c).kr;
        const int nsub = (kr + SR - 1) / SR;
        const T *R = Rl[c & 1];
        for (int q = 0; q < nsub; ++q, ++gs) {
            const T *Hs = Hl[gs % kSlots];
            const int ns = min(SR, kr - q * SR) / 4;
            for (int s = 0; s < ns; ++s) {
                T a[NRT], b[NCW];
#pragma unroll
                for (int j = 0; j < NCW; ++j) b[j] = Hs[(s * (NFB / 16) + cl0 + j) * 64 + lane];
#pragma unroll
                for (int i = 0; i < NRT; ++i) a[i] = R[(q * SR + 4 * s + lr) * LDR + pw + i * 16 + lc];
#pragma unroll
                for (int i = 0; i < NRT; ++i)
#pragma unroll
                    for (int j = 0; j < NCW; ++j) acc[i][j] = Tr::mma(a[i], b[j], acc[i][j]);
            }
            if (q + 1 == nsub) {
                if constexpr (sizeof(T) == 4) {
#pragma unroll
                    for (int i = 0; i < NRT; ++i)
#pragma unroll
                        for (int j = 0; j < NCW; ++j)
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                sum[i][j][r] += (double)acc[i][j][r];
                                acc[i][j][r] = 0.0f;
                            }
                }
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int i = 0; i < NRT; ++i)
#pragma unroll
        for (int j = 0; j < NCW; ++j) {
            const int f = fb + (cl0 + j) * 16 + lc;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t k = k0 + pw + i * 16 + Tr::row(lr, r);
                const double v = sizeof(T) == 4 ? sum[i][j][r] : (double)acc[i][j][r];
                if (f < nF && k < M) gstore(V + (int64_t)f * ldv + k, v);
            }
        }
    }
}

template <typename T, int NFB>
__global__ void __launch_bounds__(kCoulThreads) k_coulomb_ws(CoulJob<T> J, const double *__restrict__ tab) {
    __shared__ FpTileLds<T, NFB> lds;
    coulomb_tile_fp<T, NFB>(lds, J.chunks, J.nchunks, J.pP, (const T *)J.H, J.nct, J.X, J.Y, J.Z, J.M, J.nF, J.V, J.ldv, tab,
                            blockIdx.x, blockIdx.y);
}

template <typename T>
constexpr size_t fp_lds_bytes() {
    size_t b = sizeof(FpTileLds<T, 64>);
    b = b > sizeof(FpTileLds<T, 128>) ? b : sizeof(FpTileLds<T, 128>);
    b = b > sizeof(FpTileLds<T, 192>) ? b : sizeof(FpTileLds<T, 192>);
    b = b > sizeof(FpTileLds<T, 256>) ? b : sizeof(FpTileLds<T, 256>);
    return b;
}
template <typename T>
__global__ void __launch_bounds__(kCoulThreads) k_coulomb_ws_batch_all(const CoulJob<T> *__restrict__ jobs,
                                                                       const int64_t *__restrict__ off, int njobs,
                                                                       const double *__restrict__ tab) {
    __shared__ __attribute__((aligned(16))) unsigned char raw[fp_lds_bytes<T>()];
    int64_t local = 0;
    const int j = job_of_block(off, njobs, (int64_t)blockIdx.x, local);
    const CoulJob<T> J = uniform_job(jobs, j);
    const int64_t tile = local / J.ncb;
    const int cb = (int)(local - tile * J.ncb);
#define FLOSIC_TILE_FP(NFB)                                                                                          \
    coulomb_tile_fp<T, NFB>(*reinterpret_cast<FpTileLds<T, NFB> *>(raw), J.chunks, J.nchunks, J.pP, (const T *)J.H,   \
                            J.nct, J.X, J.Y, J.Z, J.M, J.nF, J.V, J.ldv, tab, tile, cb)
    switch (J.nfb) {
        case 64: FLOSIC_TILE_FP(64); break;
        case 128: FLOSIC_TILE_FP(128); break;
        case 192: FLOSIC_TILE_FP(192); break;
        default: FLOSIC_TILE_FP(256); break;
    }
#undef FLOSIC_TILE_FP
}

template <typename T>
void launch_frag_h(const ChunkDev *chunks, int nchunks, const double *H, int ldh, int nF, T *Hf, hipStream_t s) {
    if (nchunks <= 0) return;
    hipLaunchKernelGGL((k_frag_h<T>), dim3(nchunks), dim3(256), 0, s, chunks, H, ldh, nF, Hf);
}
template void launch_frag_h<double>(const ChunkDev *, int, const double *, int, int, double *, hipStream_t);
template void launch_frag_h<float>(const ChunkDev *, int, const double *, int, int, float *, hipStream_t);

template <typename T>
void launch_coulomb_mfma(const ChunkDev *chunks, int nchunks, int64_t nsteps, const double4 *pairP, const T *Hf,
                         int ldh, const double *x, const double *y, const double *z, int64_t M, const double *btab,
                         int nF, double *V, int64_t ldv, hipStream_t s, int nfb) {
    if (nchunks <= 0 || M <= 0) return;
    if (nfb <= 0) nfb = coulomb_cols(nF);
    const CoulJob<T> J{chunks, nchunks, pairP, Hf, ldh / 16, x, y, z, M, nF, V, ldv, nsteps, ldh / nfb};
    const dim3 grid((unsigned)((M + 63) / 64), (unsigned)(ldh / nfb)), blk(kCoulThreads);
    switch (nfb) {
        case 64: hipLaunchKernelGGL((k_coulomb_ws<T, 64>), grid, blk, 0, s, J, btab); break;
        case 128: hipLaunchKernelGGL((k_coulomb_ws<T, 128>), grid, blk, 0, s, J, btab); break;
        case 192: hipLaunchKernelGGL((k_coulomb_ws<T, 192>), grid, blk, 0, s, J, btab); break;
        default: hipLaunchKernelGGL((k_coulomb_ws<T, 256>), grid, blk, 0, s, J, btab); break;
    }
}
template void launch_coulomb_mfma<double>(const ChunkDev *, int, int64_t, const double4 *, const double *, int,
                                          const double *, const double *, const double *, int64_t, const double *, int,
                                          double *, int64_t, hipStream_t, int);
template void launch_coulomb_mfma<float>(const ChunkDev *, int, int64_t, const double4 *, const float *, int,
                                         const double *, const double *, const double *, int64_t, const double *, int,
                                         double *, int64_t, hipStream_t, int);

template <typename T>
void launch_coulomb_batch_all(const CoulJob<T> *jobs, const int64_t *off, int njobs, int64_t items,
                              const double *btab, hipStream_t s) {
    if (njobs <= 0 || items <= 0) return;
    hipLaunchKernelGGL((k_coulomb_ws_batch_all<T>), dim3((unsigned)items), dim3(kCoulThreads), 0, s, jobs, off, njobs,
                       btab);
}
template void launch_coulomb_batch_all<double>(const CoulJob<double> *, const int64_t *, int, int64_t,
                                               const double *, hipStream_t);
template void launch_coulomb_batch_all<float>(const CoulJob<float> *, const int64_t *, int, int64_t, const double *,
                                              hipStream_t);
}  // namespace flosic
