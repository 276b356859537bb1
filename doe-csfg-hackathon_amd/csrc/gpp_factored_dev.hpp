// gpp_factored_dev.hpp -- device building blocks of the factored form, shared
// by the single-instance kernels (gpp_factored.hip, one grid per stage) and
// the batched kernels (gpp_batch.hip, one work list per stage).
//
// Factorisation (wx_array is band-independent, gppComplex.cpp:323-329):
//   Mu[j,ig] = sum_{n1 >= nv} conj(aqsm[n1,igp(j)]) * aqsn[n1,ig]
//   Mo[j,ig] = sum_{n1 <  nv} conj(aqsm[n1,igp(j)]) * aqsn[n1,ig]
//   achtemp[iw] = sum_j 0.5 vcoul[igp(j)] sum_ig (P*Mu + sch*Mo)
//   asxtemp[iw] = sum_j occ vcoul[igp(j)] sum_ig ssx*Mo
// with P = delw*I_eps (noflagOCC_solver, :139-146) and sch, ssx from
// ssxt_scht_solver (:16-63); sch = P in branch 1 and 0 otherwise.
#pragma once

#include <type_traits>

#include "gpp_internal.hpp"

namespace gpp {
namespace fact {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int kWJ = 64, kWI = 32;  // wave tile of the fused Gram: 64 columns x 32 G-vectors
constexpr int kRedThreads = 256;   // pole-reduce and final-reduce blocks

// s_waitcnt vmcnt(N) lgkmcnt(0) (N < 64): at most N of the wave's loads from
// memory are in flight, and none of its LDS reads.
template <int N> __device__ __forceinline__ void wait_vm_lds()
{
    static_assert(N >= 0 && N < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
}

// Barrier of waves that order their memory with wait_vm_lds (no fence, which
// would wait for the loads of the stages ahead); the empty asm keeps the
// compiler from moving memory accesses across it.
__device__ __forceinline__ void ring_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// 16 bytes per lane from memory straight into LDS, in lane order from `dst`.
__device__ __forceinline__ void ring_load(const cplx *src, cplx *dst)
{
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
}

// Stage 2: Mu = conj(Bg)^T * aqsn over bands [k_begin, k_end) on
// v_mfma_f64_16x16x4f64.  Lane layout (measured on gfx950): A[l%16][l/16],
// B[l/16][l%16], result r of lane l = C[4r + l/16][l%16]; MFMA rows are G'
// columns j and MFMA columns are G-vectors ig, so each result row is
// contiguous in ig.  Three real products per complex product (3M): with
// b = Bg, a = aqsn,
//   P1 = sum br ar,  P2 = sum bi ai,  P3 = sum (br - bi)(ar + ai),
//   Re Mu = P1 + P2,  Im Mu = (P3 - P1) + P2  (= sum br ai - bi ar),
// three accumulators fed by one MFMA each per k-step instead of two fed by
// two.  Rounding: |P3| <= 2 sum |b||a|, so the error stays of order
// 1e-16 sum |b||a| (normwise), as with four products.  Every element is the
// same sum of the same products in the same order in every tile below.
//
// A tile of WJN x WIN waves, each owning SJ x SI sub-tiles of 16 G' columns x
// 16 G-vectors (TJ x TI in all).  Stages of KS bands go straight from memory
// into a ring of NB LDS buffers, NB - 1 stages ahead, with one barrier per
// stage.  Columns past the edge load the last column (their results are
// dropped); bands past the end load the last band and count as zero.
//
// What bounds them: the FP64 MFMA pipe (64 cycles per MFMA and SIMD), kept
// busy by the waves that do not wait for a stage's barrier and fragments.
// The tiles take at most 80 KB of LDS, so two blocks share a CU and one's
// stage turnover runs under the other's MFMAs; staging without registers
// leaves the 64 x 128 tile four waves per SIMD.  Measured (one launch, the
// 128 x 128 tile of eight waves staged through registers, one block per CU,
// against 64 x 128 here): 512/2/32768/1638 2587 -> 2530 us (65 TFLOP/s on the
// three products; a large FP64 library product reaches 70 on this chip),
// 1536/8/32768/1638 7564 -> 7451 us, 512/2/16384/819 794 -> 669 us (64 x 64).
template <int WJN_, int WIN_, int SJ_, int SI_, int KS_, int NB_, int OCC_> struct GramRing {
    static constexpr int WJN = WJN_, WIN = WIN_, SJ = SJ_, SI = SI_, KS = KS_, NB = NB_;
    static constexpr int OCC = OCC_;  // waves per SIMD
    static constexpr int NW = WJN * WIN, TJ = 16 * SJ * WJN, TI = 16 * SI * WIN, NT = 64 * NW;
    static constexpr int STAGE = KS * (TJ + TI);  // entries
    static constexpr int LDS = NB * STAGE;
};
typedef GramRing<2, 4, 2, 2, 8, 3, 4> GramL;   // 64 x 128
typedef GramRing<4, 2, 2, 2, 8, 3, 4> GramLt;  // 128 x 64
typedef GramRing<2, 2, 2, 2, 8, 4, 2> GramM;   // 64 x 64
typedef GramRing<2, 4, 1, 1, 16, 3, 4> GramS;  // 32 x 64

// One tile with SJC <= SJ sub-tile rows per wave: the first 16 SJC WJN columns
// from j0, for a last tile whose columns need no more.  NTS: non-temporal
// stores of Mu (a template parameter: under a run-time flag the compiler merged
// both kinds into plain stores, and the C1 reduce took 510 us instead of 424).
// The block's waves must be done with lds before the call.
template <class C, int SJC, bool NTS>
__device__ __forceinline__ void gram_ring_tile(const cplx *__restrict__ bg, const cplx *__restrict__ aqsn, int ngpown,
                                               int ncouls, int k_begin, int k_end, int j0, int i0, cplx *lds,
                                               cplx *__restrict__ mout)
{
    constexpr int KS = C::KS, NB = C::NB, TJ = C::TJ, TI = C::TI, SI = C::SI, NW = C::NW;
    constexpr int QB = KS * TJ / 64 / NW, QA = KS * TI / 64 / NW, LD = QB + QA;  // loads per wave and stage
    static_assert(QB * 64 * NW == KS * TJ && QA * 64 * NW == KS * TI && NB >= 3, "loads split evenly over the waves");
    static_assert(SJC >= 1 && SJC <= C::SJ && KS % 4 == 0, "sub-tiles of the tile, whole k-steps");
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int wj = (wave / C::WIN) * (16 * SJC), wi = (wave % C::WIN) * (16 * SI);
    const int nst = (k_end - k_begin + KS - 1) / KS;

    // Load q of a side fills elements [64 (q NW + wave), +64) of its rows of a
    // stage: this lane's source element of each, advanced from stage to stage.
    const cplx *pb[QB], *pa[QA];
#pragma unroll
    for (int q = 0; q < QB; ++q) {
        const int e = 64 * (q * NW + wave) + lane;
        pb[q] = bg + (size_t)(k_begin + e / TJ) * ngpown + min(j0 + e % TJ, ngpown - 1);
    }
#pragma unroll
    for (int q = 0; q < QA; ++q) {
        const int e = 64 * (q * NW + wave) + lane;
        pa[q] = aqsn + (size_t)(k_begin + e / TI) * ncouls + min(i0 + e % TI, ncouls - 1);
    }
    const size_t stepb = (size_t)KS * ngpown, stepa = (size_t)KS * ncouls;
    int ibuf = 0, rbuf = 0;  // next buffer to fill, to read
    auto issue = [&]() {
        cplx *buf = lds + ibuf * C::STAGE + 64 * wave;
        ibuf = ibuf + 1 == NB ? 0 : ibuf + 1;
#pragma unroll
        for (int q = 0; q < QB; ++q) {
            ring_load(pb[q], buf + 64 * NW * q);
            pb[q] += stepb;
        }
#pragma unroll
        for (int q = 0; q < QA; ++q) {
            ring_load(pa[q], buf + KS * TJ + 64 * NW * q);
            pa[q] += stepa;
        }
    };
    auto issue_last = [&]() {  // stage nst - 1: rows past the end load the last band
        cplx *buf = lds + ibuf * C::STAGE + 64 * wave;
        const int over0 = k_begin + (nst - 1) * KS - (k_end - 1);
#pragma unroll
        for (int q = 0; q < QB; ++q) {
            const int over = max(0, over0 + (64 * (q * NW + wave) + lane) / TJ);
            ring_load(pb[q] - (size_t)over * ngpown, buf + 64 * NW * q);
        }
#pragma unroll
        for (int q = 0; q < QA; ++q) {
            const int over = max(0, over0 + (64 * (q * NW + wave) + lane) / TI);
            ring_load(pa[q] - (size_t)over * ncouls, buf + KS * TJ + 64 * NW * q);
        }
    };

    v4d acc1[SJC][SI], acc2[SJC][SI], acc3[SJC][SI];  // P1, P2, P3
#pragma unroll
    for (int s = 0; s < SJC; ++s)
#pragma unroll
        for (int t = 0; t < SI; ++t) acc1[s][t] = acc2[s][t] = acc3[s][t] = v4d{0, 0, 0, 0};
    auto multiply = [&](auto last) {
        const cplx *sB = lds + rbuf * C::STAGE, *sA = sB + KS * TJ;
        rbuf = rbuf + 1 == NB ? 0 : rbuf + 1;
        __builtin_amdgcn_s_setprio(1);  // the wave with ready operands issues its MFMAs first
#pragma unroll
        for (int kk = 0; kk < KS; kk += 4) {
            const int kr = kk + lane / 16;
            const bool out = last && k_begin + (nst - 1) * KS + kr >= k_end;
            double are[SI], aim[SI], asum[SI];
#pragma unroll
            for (int t = 0; t < SI; ++t) {
                cplx a = sA[kr * TI + wi + 16 * t + lane % 16];
                if (out) a = czero();
                are[t] = a.re;
                aim[t] = a.im;
                asum[t] = a.re + a.im;
            }
#pragma unroll
            for (int s = 0; s < SJC; ++s) {
                cplx b = sB[kr * TJ + wj + 16 * s + lane % 16];
                if (out) b = czero();
                const double bdiff = b.re - b.im;
#pragma unroll
                for (int t = 0; t < SI; ++t) {
                    acc1[s][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(b.re, are[t], acc1[s][t], 0, 0, 0);
                    acc2[s][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(b.im, aim[t], acc2[s][t], 0, 0, 0);
                    acc3[s][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(bdiff, asum[t], acc3[s][t], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
    };

    // At the top of stage st, stages st .. st + NB - 2 have been issued: wait
    // for this wave's loads of stage st and its fragment reads of stage
    // st - 1, then (barrier) for every wave's; stage st + NB - 1 then takes the
    // buffer of stage st - 1.
    for (int st = 0; st < NB - 1 && st < nst; ++st) {
        if (st < nst - 1)
            issue();
        else
            issue_last();
    }
    int st = 0;
    for (; st < nst - NB; ++st) {  // the stages that issue a whole stage
        wait_vm_lds<(NB - 2) * LD>();
        ring_barrier();
        issue();
        multiply(std::integral_constant<bool, false>());
    }
    if (nst >= NB) {  // st = nst - NB: issues the last stage
        wait_vm_lds<(NB - 2) * LD>();
        ring_barrier();
        issue_last();
        multiply(std::integral_constant<bool, false>());
        ++st;
    }
    for (; st < nst - 1; ++st) {
        wait_vm_lds<0>();
        ring_barrier();
        multiply(std::integral_constant<bool, false>());
    }
    if (nst > 0) {
        wait_vm_lds<0>();
        ring_barrier();
        multiply(std::integral_constant<bool, true>());
    }
#pragma unroll
    for (int s = 0; s < SJC; ++s)
#pragma unroll
        for (int t = 0; t < SI; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = j0 + wj + 16 * s + 4 * r + lane / 16;
                const int ig = i0 + wi + 16 * t + lane % 16;
                if (j < ngpown && ig < ncouls) {
                    const cplx v = {acc1[s][t][r] + acc2[s][t][r], (acc3[s][t][r] - acc1[s][t][r]) + acc2[s][t][r]};
                    cplx *o = &mout[(size_t)j * ncouls + ig];
                    if constexpr (NTS) {
                        __builtin_nontemporal_store(v.re, &o->re);
                        __builtin_nontemporal_store(v.im, &o->im);
                    } else {
                        *o = v;
                    }
                }
            }
}

// One 16 x 16 tile of Mu by three waves, one per real product of the 3M form
// (P1, P2, P3 of gram_f64_acc, combined as there), for products with fewer
// tiles than the chip has SIMDs: the chain of dependent MFMAs over the bands
// bounds those, and a wave with one product per tile has a third of the chain
// of a wave with all three.  Stages of kSmK bands go straight from memory into
// a ring of kSmBuf LDS buffers, kSmBuf - 1 stages ahead (about 0.8 us of MFMA
// time); the fragments of stage st + 1 are read while stage st is multiplied.
// Columns past the edge load the last column (their results are dropped);
// bands past the end load the last band and count as zero.
constexpr int kSmK = 24, kSmBuf = 6, kSmThreads = 192;
constexpr int kSmStage = 2 * kSmK * 16;  // entries of a stage: Bg rows, then aqsn rows
template <int P>
__device__ __forceinline__ v4d gram_small_product(const cplx *__restrict__ bg, const cplx *__restrict__ aqsn,
                                                  int ngpown, int ncouls, int k_begin, int k_end, int j0, int i0,
                                                  cplx *lds)
{
    constexpr int STEPS = kSmK / 4;
    constexpr int ROWS = kSmK / 3;  // rows of a stage each wave loads, four per instruction
    static_assert(ROWS % 4 == 0, "a wave loads whole groups of four rows");
    constexpr int Q = ROWS / 4, LD = 2 * Q;  // loads per wave and stage: Q of each operand
    const int lane = threadIdx.x % kWave;
    const int nst = (k_end - k_begin + kSmK - 1) / kSmK;
    // This lane's element of the wave's rows (the wave of product P loads rows
    // [P ROWS, (P + 1) ROWS) of a stage), advanced from stage to stage.
    const int r0 = P * ROWS + lane / 16;
    const cplx *pb = bg + (size_t)(k_begin + r0) * ngpown + min(j0 + lane % 16, ngpown - 1);
    const cplx *pa = aqsn + (size_t)(k_begin + r0) * ncouls + min(i0 + lane % 16, ncouls - 1);
    const size_t rb = 4 * (size_t)ngpown, ra = 4 * (size_t)ncouls;
    int issued = 0, ibuf = 0;  // next stage to load and its buffer
    auto issue = [&]() {
        cplx *buf = lds + ibuf * kSmStage + P * ROWS * 16;
        if (issued < nst - 1) {
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                __builtin_amdgcn_global_load_lds(pb + q * rb, (__attribute__((address_space(3))) void *)(buf + q * 64),
                                                 16, 0, 0);
                __builtin_amdgcn_global_load_lds(
                    pa + q * ra, (__attribute__((address_space(3))) void *)(buf + kSmK * 16 + q * 64), 16, 0, 0);
            }
            pb += (kSmK / 4) * rb;
            pa += (kSmK / 4) * ra;
        } else {  // the last stage: rows past the end load the last band
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const long long over = max(0, k_begin + issued * kSmK + r0 + 4 * q - (k_end - 1));
                __builtin_amdgcn_global_load_lds(pb + q * rb - over * ngpown,
                                                 (__attribute__((address_space(3))) void *)(buf + q * 64), 16, 0, 0);
                __builtin_amdgcn_global_load_lds(
                    pa + q * ra - over * ncouls,
                    (__attribute__((address_space(3))) void *)(buf + kSmK * 16 + q * 64), 16, 0, 0);
            }
        }
        ++issued;
        ibuf = ibuf + 1 == kSmBuf ? 0 : ibuf + 1;
    };
    // Operands of a stage: the wave's part of the fragments (P1 real, P2
    // imaginary parts; P3 both, summed after they have arrived).
    struct Frag {
        double b[STEPS], a[STEPS], bi[P == 2 ? STEPS : 1], ai[P == 2 ? STEPS : 1];
    };
    Frag f0, f1;
    int rbuf = 0;  // buffer of the next stage to read
    auto read = [&](Frag &f, const cplx *buf, int s) {
        const cplx &b = buf[s * 64 + lane], &a = buf[kSmK * 16 + s * 64 + lane];
        f.b[s] = P == 1 ? b.im : b.re;
        f.a[s] = P == 1 ? a.im : a.re;
        if constexpr (P == 2) {
            f.bi[s] = b.im;
            f.ai[s] = a.im;
        }
    };
    auto finish = [&](Frag &f) {
        if constexpr (P == 2) {
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                f.b[s] -= f.bi[s];
                f.a[s] += f.ai[s];
            }
        }
    };
    v4d acc = {0, 0, 0, 0};
    // All of a wave's loads of stage st have landed (of the kSmBuf - 2 stages
    // st .. st + kSmBuf - 3 issued by now, those after it may be in flight)
    // and its fragment reads are done, then every wave's.  The empty asm keeps
    // the LDS reads below the barrier.
    auto arrive = [&](int st) {
        if (st + kSmBuf - 3 < nst)
            wait_vm_lds<(kSmBuf - 3) * LD>();
        else
            wait_vm_lds<0>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // Round st of all but the last: stage st + 1 lands; the buffer that stage
    // st + kSmBuf - 1 takes is that of stage st - 1, whose fragments every wave
    // has read.  The fragment reads of stage st + 1 go between the products of
    // stage st.
    auto round = [&](int st, Frag &cur, Frag &nxt) {
        finish(cur);
        arrive(st + 1);
        if (issued < nst) issue();
        const cplx *buf = lds + rbuf * kSmStage;
        rbuf = rbuf + 1 == kSmBuf ? 0 : rbuf + 1;
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(cur.b[s], cur.a[s], acc, 0, 0, 0);
            read(nxt, buf, s);
            __builtin_amdgcn_sched_group_barrier(8, 1, 0);      // one MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // two LDS reads
        }
    };
    auto last_round = [&](Frag &f) {
        finish(f);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const bool out = k_begin + (nst - 1) * kSmK + 4 * s + lane / 16 >= k_end;
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(out ? 0.0 : f.b[s], out ? 0.0 : f.a[s], acc, 0, 0, 0);
        }
    };
    if (nst == 0) return acc;
    for (int st = 0; st < kSmBuf - 1 && st < nst; ++st) issue();
    arrive(0);
#pragma unroll
    for (int s = 0; s < STEPS; ++s) read(f0, lds, s);
    rbuf = 1;
    int st = 0;
    for (; st + 2 < nst; st += 2) {
        round(st, f0, f1);
        round(st + 1, f1, f0);
    }
    if (st + 1 < nst) {
        round(st, f0, f1);
        last_round(f1);
    } else {
        last_round(f0);
    }
    return acc;
}

// The Gram tile of the fused Gram + pole reduce: 128 x 128 by 2 x 4 waves of
// 64 x 32, 16 bands per LDS stage staged through registers in two pieces of 8,
// each stored to the other buffer after its k-steps, so that its staging
// registers fit two waves per SIMD.
struct FuseCfg {
    static constexpr int WIN = 4, TJ = 2 * kWJ, TI = 4 * kWI, NT = 512;
    static constexpr int KS = 16, NH = 2;
};

// The sums of gram_ring_tile with the MFMA operands swapped: rows are
// G-vectors and columns G' columns, result r of lane l of sub-tile (s, t) is
// element (ig = wi + 16t + 4r + l/16, j = wj + 16s + l%16) -- each lane holds
// four G' columns and eight G-vectors of each, the layout the fused pole
// epilogue sums over G-vectors in.
__device__ __forceinline__ void gram_f64_acc(const cplx *__restrict__ bg, const cplx *__restrict__ aqsn, int ngpown,
                                             int ncouls, int k_begin, int k_end, int j0, int i0,
                                             cplx (*sB)[FuseCfg::KS][FuseCfg::TJ],
                                             cplx (*sA)[FuseCfg::KS][FuseCfg::TI], v4d (&acc1)[4][2],
                                             v4d (&acc2)[4][2], v4d (&acc3)[4][2])
{
    typedef FuseCfg C;
    constexpr int TJ = C::TJ, TI = C::TI, NT = C::NT, KS = C::KS, NH = C::NH;
    constexpr int PB = KS * TJ / NT / NH, PA = KS * TI / NT / NH;  // staged elements per thread and piece
    static_assert(PB * NT * NH == KS * TJ && PA * NT * NH == KS * TI, "stage must split evenly");
    static_assert((PB * NT) % TJ == 0 && (PA * NT) % TI == 0 && (KS / NH) % 4 == 0,
                  "a piece is whole band rows and whole k-steps");
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int wj = (wave / C::WIN) * kWJ;
    const int wi = (wave % C::WIN) * kWI;

#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc1[s][t] = acc2[s][t] = acc3[s][t] = v4d{0, 0, 0, 0};

    // piece h of a stage: band rows [h KS / NH, (h + 1) KS / NH)
    cplx stB[PB], stA[PA];
    auto load_piece = [&](int k0, int h) {
#pragma unroll
        for (int q = 0; q < PB; ++q) {
            const int e = threadIdx.x + (h * PB + q) * NT;
            const int kr = e / TJ, c = e % TJ, k = k0 + kr, j = j0 + c;
            stB[q] = (k < k_end && j < ngpown) ? bg[(size_t)k * ngpown + j] : czero();
        }
#pragma unroll
        for (int q = 0; q < PA; ++q) {
            const int e = threadIdx.x + (h * PA + q) * NT;
            const int kr = e / TI, c = e % TI, k = k0 + kr, ig = i0 + c;
            stA[q] = (k < k_end && ig < ncouls) ? aqsn[(size_t)k * ncouls + ig] : czero();
        }
    };
    auto store_piece = [&](int buf, int h) {
#pragma unroll
        for (int q = 0; q < PB; ++q) {
            const int e = threadIdx.x + (h * PB + q) * NT;
            sB[buf][e / TJ][e % TJ] = stB[q];
        }
#pragma unroll
        for (int q = 0; q < PA; ++q) {
            const int e = threadIdx.x + (h * PA + q) * NT;
            sA[buf][e / TI][e % TI] = stA[q];
        }
    };

    const int nst = (k_end - k_begin + KS - 1) / KS;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        load_piece(k_begin, h);
        store_piece(0, h);
    }
    __syncthreads();
    for (int st = 0; st < nst; ++st) {
        const int buf = st & 1;
#pragma unroll
        for (int h = 0; h < NH; ++h) {
        if (st + 1 < nst) load_piece(k_begin + (st + 1) * KS, h);
        __builtin_amdgcn_s_setprio(1);  // the MFMA section: the wave with ready operands issues first
        // scheduling hint: interleave the fragment reads from LDS with the MFMAs
        // (strategy 1; measured ~1 % faster than the default schedule and than strategy 0)
        __builtin_amdgcn_iglp_opt(1);
#pragma unroll
        for (int kk = h * (KS / NH); kk < (h + 1) * (KS / NH); kk += 4) {
            const int kr = kk + lane / 16;
            double are[2], aim[2], asum[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const cplx a = sA[buf][kr][wi + 16 * t + lane % 16];
                are[t] = a.re;
                aim[t] = a.im;
                asum[t] = a.re + a.im;
            }
            // one B sub-tile at a time keeps the fragments within the
            // register budget of two waves per SIMD
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const cplx b = sB[buf][kr][wj + 16 * s + lane % 16];
                const double bdiff = b.re - b.im;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    acc1[s][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(are[t], b.re, acc1[s][t], 0, 0, 0);
                    acc2[s][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(aim[t], b.im, acc2[s][t], 0, 0, 0);
                    acc3[s][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(asum[t], bdiff, acc3[s][t], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        if (st + 1 < nst) store_piece(buf ^ 1, h);
        }
        __syncthreads();
    }
}

// 2^-40 band around a threshold inside which a decision made on an estimate
// is remade in the reference's arithmetic.
constexpr double kBand = 1.0 / 1099511627776.0;

// The occupied solver's branch tests (gppComplex.cpp:35, :43) on |delw|^2 for
// one element and frequency: branch1 = |wdiff|^2 > 0.25 and |delw|^2 <
// limitone, above2 = |delw|^2 > to1.  wdiffr = |wdiff|^2 rounded as the
// reference rounds it, rden its reciprocal (rcp_1nr), wt2 = |wt|^2.
// est = wt2 * rden is within 1e-14 of the reference's rounded |delw|^2,
// relative to it (each rounding of delw is bounded by |delw|, with or
// without cancellation), so outside a 2^-40 band around the two thresholds
// it decides as the reference does; inside it, below the lower one and for a
// NaN est (|wdiff|^2 = 0 or beyond the double range: rcp_1nr returns NaN),
// the reference's delw and |delw|^2 are recomputed in its operation order
// with the correctly rounded reciprocal (:30-32).  An est of +inf (the
// product overflowed) means a |delw|^2 of at least about 1.8e308, far above
// both thresholds, where the reference decides alike (branch 2).
// The decisions from est alone; false where they are not sure.
__device__ __forceinline__ bool occ_branch_estimate(double wdiffr, double rden, double wt2, bool &branch1, bool &above2)
{
#pragma clang fp contract(off)
    constexpr double limitone = 1.0 / (kTo1 * 4.0);
    constexpr double kEstLo1 = limitone * (1 - kBand), kEstHi1 = limitone * (1 + kBand);
    constexpr double kEstHi2 = kTo1 * (1 + kBand);
    const double est = wt2 * rden;
    // below the to1 band (|delw|^2 < 1e-6, where |wdiff| exceeds |wt| a
    // thousandfold) is rare enough to take the exact path with the bands
    const bool below1 = est < kEstLo1;
    above2 = est > kEstHi2;
    branch1 = (wdiffr > 0.25) && below1;
    return (above2 & below1) | (est > kEstHi1);
}
__device__ __forceinline__ void occ_branch_tests(double wxf, cplx wt, double wdiffr, double rden, double wt2,
                                                 bool &branch1, bool &above2)
{
#pragma clang fp contract(off)
    if (!occ_branch_estimate(wdiffr, rden, wt2, branch1, above2)) {
        constexpr double limitone = 1.0 / (kTo1 * 4.0);
        const cplx wdiff = cdminus(wxf, wt);
        const cplx delw = cscale(cmul(wt, cconj(wdiff)), rcp_refined(wdiffr));
        const double delwr = cmul(delw, cconj(delw)).re;
        branch1 = (wdiffr > 0.25) && delwr < limitone;
        above2 = delwr > kTo1;
    }
}

// One instance's inputs and workspace as seen by the reduce stages.
struct ReduceArgs {
    const cplx *mu;  // [ngpown][ncouls]
    const cplx *ieps, *wtilde, *aqsn;
    const cplx *bg;  // [nb][ngpown]
    const int32_t *idx;
    const double *vcoul, *wx;
    int nv, ncouls, ngpown, nfreq, nsplit, chunk;
    int fpb;  // frequencies per block (single-instance grid: z = ceil(nfreq / fpb))
    double occ;
    cplx *col_ach, *col_asx;  // [ngpown][nsplit][nfreq]
    // Optional (acht_n1_loc): the pole factor of frequency acht_iw, p2 =
    // delw*I_eps [ngpown][ncouls], and br1 [ngpown][ncouls] = 1 where the
    // occupied solver takes branch 1 at that frequency (sch = p2 there, 0
    // elsewhere); p2 null when not requested, br1 null when nv == 0.
    cplx *p2;
    uint8_t *br1;
    int acht_iw;
    int neg;  // some frequency is negative: launch the NEG variant (host-side dispatch only)
    // With p2 and reduce_sums_acht_occ: the occupied bands' acht_n1_loc
    // partials, [ngpown][nsplit][nv], summed in the pass (br1 not written).
    cplx *part_occ;
    Stamp stamp;
};

// Whether the p2-storing reduce sums the occupied bands' acht_n1_loc terms
// itself or leaves them to acht_occ_item (br1): two occupied bands, whose
// aqsn values and sums fit beside the pass (with 4 or 8 the kernels spill,
// at 8 and 16 frequencies by 45-297 registers).
__host__ __device__ inline bool reduce_sums_acht_occ(int nv, int neg) { return !neg && nv == 2; }

// LDS of pole_reduce_item: block_sum's scratch, then (pole_stages) one aqsn
// value per occupied band and thread.
template <int FC, int NV> constexpr bool pole_stages() { return FC > 3 && NV > 0; }
template <int FC, int NV> constexpr int pole_lds_entries()
{
    return kRedThreads / kWave + (pole_stages<FC, NV>() ? NV * kRedThreads : 0);
}

// Stage 3: pole terms of column j over G-vectors [split*chunk, +chunk), for
// frequencies [iw0, iw0+FC).  Per element and frequency: wdiff, |wdiff|^2,
// delw = wt*conj(wdiff)*rden and |delw|^2 in the reference's order
// (gppComplex.cpp:139-144, no contraction; rden is the refined reciprocal,
// equal to the IEEE quotient), so the occupied branch tests (:35, :43) see
// the reference's values.  P = delw*ie, the branch-2 ssx in its reduced form
// -(I_eps wt / 2) / (wx + wt) and the accumulations use FMA.  sch = P in branch 1 (:37) shares the
// unoccupied product.  Block-wide fixed-order sums; writes the column
// partials (0.5*sum)*vcoul and sum*(occ*vcoul).  scratch: 4 entries.
// NV > 0: the occupied band count is NV (== a.nv), known at compile time, so
// the occupied loads are unrolled and issued together and conj(bg) of the
// column is loaded once; NV == 0: any a.nv.  NEG: some frequency may be
// negative, where the ssx cutoff of :58-59 is live; without it every
// frequency must be >= 0 (the launcher checks on the host) and the kernel
// carries no cutoff code.  P2 with NV == 2 (and no NEG): the pass holding
// frequency acht_iw also sums sum_ig aqsn[n1,ig] p2[j,ig] [branch 1] per
// occupied band n1 (the same products in the same order as acht_occ_item,
// whose partials it writes to part_occ).
template <int FC, int NV = 0, bool P2 = false, int FCT = FC, bool NEG = false>
__device__ __forceinline__ void pole_reduce_item(const ReduceArgs &a, int j, int split, int iw_begin, int iw_end,
                                                 cplx *lds)
{
#pragma clang fp contract(off)
    const int ncouls = a.ncouls;
    const int nv = NV > 0 ? NV : a.nv;
    constexpr bool kOccSum = P2 && NV == 2 && !NEG;  // reduce_sums_acht_occ
    // The occupied aqsn values of a thread's next G-vector load straight into
    // LDS (its own entries, so no barrier) while the current one is evaluated.
    // Loaded where they are used, the waves of these kernels (two or three a
    // SIMD, no registers to load ahead into) stood 42% of their time waiting:
    // reduce us 300/8/32768/1638/16 1574 -> 1488, 300/2/16384/819/8 220 -> 194,
    // 300/4/16384/819/24 663 -> 613.  Not for the general kernel (without
    // occupied bands 302 -> 330 us at 200/0/16384/819/16) nor for the kernels of at most
    // three frequencies, which the streams bound (four waves a SIMD; the
    // p2-storing one took 203 against 192 us at 300/2/16384/819).
    constexpr bool kStages = pole_stages<FC, NV>();
    cplx *const scratch = lds, *const occ_wave = lds + kRedThreads / kWave + (threadIdx.x & ~(kWave - 1));
    cplx *const occ_av = lds + kRedThreads / kWave + threadIdx.x;

    const int ig_begin = split * a.chunk;
    const int ig_end = ig_begin + a.chunk < ncouls ? ig_begin + a.chunk : ncouls;
    // conj(Bg[n1][j]) of the occupied bands, loaded once for the column (the
    // optional p2/br1 stores in the loop would otherwise keep the compiler
    // from hoisting these loads out of it).
    // Wave-uniform (the column's), so kept in scalar registers.
    cplx bgc[NV > 0 ? NV : 1];
    if constexpr (NV > 0) {
#pragma unroll
        for (int n1 = 0; n1 < NV; ++n1) bgc[n1] = uniform(cconj(a.bg[(size_t)n1 * a.ngpown + j]));
    }
    // Frequencies in passes of FC, the last one FCT wide when at most FCT
    // remain; the passes after the first re-read this block's G-vector range,
    // recently fetched, from the caches.
    auto pass = [&](auto width, auto fold, int iw0) {
        constexpr int F = decltype(width)::value;
        constexpr bool FOLD = decltype(fold)::value;
        double wxv[F], c1[F];  // branch-1 ssx = Omega2 * wx^2 / wx^4 (:38-41) = Omega2 * c1
#pragma unroll
        for (int f = 0; f < F; ++f) {
            // wave-uniform, so kept in scalar registers
            wxv[f] = uniform((iw0 + f < iw_end) ? a.wx[iw0 + f] : 1.0);
            const double wx2 = wxv[f] * wxv[f];
            c1[f] = uniform(wx2 * (1.00 / (wx2 * wx2)));
        }
        cplx sach[F], sasx[F];
#pragma unroll
        for (int f = 0; f < F; ++f) sach[f] = sasx[f] = czero();
        cplx oacc[kOccSum ? NV : 1];  // occupied acht_n1_loc sums (kOccSum)
#pragma unroll
        for (int n1 = 0; n1 < (kOccSum ? NV : 1); ++n1) oacc[n1] = czero();

        bool any_neg = false;  // the ssx cutoff of :58-59 applies only at negative frequencies
        if constexpr (NEG) {
#pragma unroll
            for (int f = 0; f < F; ++f) any_neg = any_neg || wxv[f] < 0.00;
        }

        const size_t row = (size_t)j * ncouls;
        // The next element's wtilde, I_eps and Mu load while this one is
        // evaluated (two elements in flight per thread; a third did not
        // help).
        // Kernels of at most three frequencies make one pass: their three
        // streams are read once, without keeping them in the caches.
        auto ld = [](const cplx *p) -> cplx {
            if constexpr (FC <= 3)
                return cplx{__builtin_nontemporal_load(&p->re), __builtin_nontemporal_load(&p->im)};
            else
                return *p;
        };
        // With kStages every lane loads: those past the end repeat the last
        // G-vector and skip the evaluation.
        cplx wt_n = czero(), ie_n = czero(), mu_n = czero();
        const int lane0 = kStages ? 0 : (int)threadIdx.x;  // the loop index: the block's, or the lane's
        auto load_next = [&](int i) {
            const int ig = kStages ? min(i + (int)threadIdx.x, ig_end - 1) : i;
            if constexpr (kStages) {
#pragma unroll
                for (int n1 = 0; n1 < NV; ++n1) ring_load(a.aqsn + (size_t)n1 * ncouls + ig, occ_wave + n1 * kRedThreads);
            }
            wt_n = ld(a.wtilde + row + ig);
            ie_n = ld(a.ieps + row + ig);
            mu_n = ld(a.mu + row + ig);
        };
        if (ig_begin + lane0 < ig_end) load_next(ig_begin + lane0);
        for (int i = ig_begin + lane0; i < ig_end; i += kStages ? kRedThreads : blockDim.x) {
            const int ig = kStages ? i + (int)threadIdx.x : i;
            if constexpr (kStages) {
                // the loads of this element, all older than the rest
                __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));  // vmcnt(0)
                asm volatile("" ::: "memory");
            }
            const cplx wt = wt_n, ie = ie_n, mu = mu_n;
            // Mo over the occupied bands, in band order: folded passes
            // take four FMAs per band (C3 reduce 7.54 -> 7.33 ms, C4 14.39
            // -> 14.14 ms), the three-frequency kernel a product and a sum
            // (0.487 against 0.501 ms at 512/2/32768/1638)
            cplx mo = czero();
            cplx av[NV > 0 ? NV : 1];  // the occupied aqsn of this G-vector, loads issued together
            auto form_mo = [&]() {
                if constexpr (NV > 0 && kStages) {
#pragma unroll
                    for (int h = 0; h < NV; h += 4) {  // four at a time in registers
#pragma unroll
                        for (int n1 = h; n1 < NV && n1 < h + 4; ++n1) av[n1] = occ_av[n1 * kRedThreads];
#pragma unroll
                        for (int n1 = h; n1 < NV && n1 < h + 4; ++n1)
                            mo = !FOLD ? cadd(mo, cmul_fast(bgc[n1], av[n1]))
                                       : n1 == 0 ? cmul_fast(bgc[0], av[0]) : cfma(bgc[n1], av[n1], mo);
                        asm volatile("" : "+v"(mo.re), "+v"(mo.im));
                    }
                } else if constexpr (NV > 0) {
#pragma unroll
                    for (int n1 = 0; n1 < NV; ++n1) av[n1] = a.aqsn[(size_t)n1 * ncouls + ig];
#pragma unroll
                    for (int n1 = 0; n1 < NV; ++n1) mo = cadd(mo, cmul_fast(bgc[n1], av[n1]));
                } else {
                    for (int n1 = 0; n1 < nv; ++n1) {
                        const cplx b = cconj(a.bg[(size_t)n1 * a.ngpown + j]);
                        const cplx v = a.aqsn[(size_t)n1 * ncouls + ig];
                        mo = FOLD ? cfma(b, v, mo) : cadd(mo, cmul_fast(b, v));
                    }
                }
            };
            if constexpr (kStages) {
                form_mo();
                asm volatile("" ::: "memory");  // the reads before the next loads
            }
            if (i + (int)(kStages ? kRedThreads : blockDim.x) < ig_end) load_next(i + (kStages ? kRedThreads : blockDim.x));
            if (kStages && ig >= ig_end) break;
            // P = delw I_eps = q conj(wdiff) / |wdiff|^2 with q = wt I_eps and
            // conj(wdiff) = (wx - wt.re, wt.im) =: (wdr, wt.im).  FOLD (problems
            // with 4 or more frequencies) folds Mu and Mo into the products
            // once per element -- u = q Mu (every element), uo = q Mo (branch
            // 1: sch = P for the occupied bands) and Omega2 Mo (branch 1's ssx
            // Mo = c1 Omega2 Mo) -- so each frequency adds u conj(wdiff) /
            // |wdiff|^2 with four FMAs (C4 reduce 18.2 -> 14.9 ms); with fewer
            // frequencies P is formed and Mu or Mu + Mo selected per
            // frequency, which is faster there (C1: 0.50 against 0.55 ms
            // folded).
            const cplx q = cmul_fast(wt, ie);
            // wdiff.im^2 rounded as the reference's |wdiff|^2 (:27, :33) rounds it
            const double wti2 = wt.im * wt.im;
            // q.im wt.im and q.re wt.im: kept per element when P is formed every
            // frequency, recomputed on the rare paths otherwise
            const double q_im_wti_e = FOLD ? 0.0 : q.im * wt.im, q_re_wti_e = FOLD ? 0.0 : q.re * wt.im;
            cplx om2 = czero(), mum = mu, u0 = czero(), uo = czero(), w1 = czero();
            double u0_im_wti = 0.0, u0_re_wti = 0.0, uo_im_wti = 0.0, uo_re_wti = 0.0, ie_cut = 0.0, wt2 = 0.0;
            if constexpr (FOLD) {
                u0 = cmul_fast(q, mu);
                u0_im_wti = u0.im * wt.im;
                u0_re_wti = u0.re * wt.im;
            }
            if (nv > 0) {
                if constexpr (!kStages) form_mo();
                om2 = cmul(csquare(wt), ie);  // Omega2 = wtilde^2 * I_eps, flagOCC_solver :117-118
                if constexpr (FOLD) {
                    uo = cmul_fast(q, mo);
                    uo_im_wti = uo.im * wt.im;
                    uo_re_wti = uo.re * wt.im;
                    w1 = cmul_fast(om2, mo);
                } else {
                    mum = cadd(mu, mo);
                }
                wt2 = __builtin_fma(wt.re, wt.re, wti2);
                if (NEG && any_neg) {
                    // A real (uniform) branch: the empty asm keeps the compiler
                    // from evaluating the square root for every element.
                    asm volatile("" ::: "memory");
                    ie_cut = cabs_(ie) * kSexcut;
                }
            }
            // Frequencies in groups: their reciprocals, u terms and branch
            // estimates are formed together, before any branch on them, and
            // overlap (with two or three waves a SIMD nothing else hides a
            // reciprocal's latency).  Two: 300/8/32768/1638/16 1488 -> 1430 us,
            // 300/4/16384/819/24 613 -> 583; groups of four need more registers
            // than three waves have.
            // Masking the occupied terms too instead of branching on them took
            // 13% longer: it adds more instructions than it overlaps.
            constexpr int kGrp = FOLD && !NEG && NV > 0 ? 2 : 1;
            double wdrs[kGrp], rdens[kGrp];
            bool b1s[kGrp], a2s[kGrp];
#pragma unroll
            for (int f = 0; f < F; ++f) {
                if (f % kGrp == 0) {
                    double wdiffrs[kGrp];
                    bool unsure = false;
#pragma unroll
                    for (int k = 0; k < kGrp && f + k < F; ++k) {
                        wdrs[k] = wxv[f + k] - wt.re;                // wdiff = (wdr, -wt.im), :27
                        wdiffrs[k] = wdrs[k] * wdrs[k] + wti2;       // |wdiff|^2 exactly as the reference rounds it
                        rdens[k] = rcp_1nr(wdiffrs[k]);
                        if constexpr (FOLD) {  // P Mu
                            cplx &t = sach[f + k];
                            t.re = __builtin_fma(__builtin_fma(u0.re, wdrs[k], -u0_im_wti), rdens[k], t.re);
                            t.im = __builtin_fma(__builtin_fma(u0.im, wdrs[k], u0_re_wti), rdens[k], t.im);
                        }
                        b1s[k] = a2s[k] = false;
                        if constexpr (kGrp == 1) {
                            if (nv > 0) occ_branch_tests(wxv[f], wt, wdiffrs[k], rdens[k], wt2, b1s[k], a2s[k]);
                        } else if (nv > 0) {
                            unsure |= !occ_branch_estimate(wdiffrs[k], rdens[k], wt2, b1s[k], a2s[k]);
                        }
                    }
                    if (unsure) {
#pragma unroll
                        for (int k = 0; k < kGrp && f + k < F; ++k)
                            occ_branch_tests(wxv[f + k], wt, wdiffrs[k], rdens[k], wt2, b1s[k], a2s[k]);
                    }
                }
                const double wdr = wdrs[f % kGrp], rden = rdens[f % kGrp];
                const bool branch1 = b1s[f % kGrp], above2 = a2s[f % kGrp];
                // Branch 2 (:46-50) with cden = 4 wt^2 (0.5 + delw), Omega2 =
                // wt^2 I_eps and delw = wt / (wx - wt):
                //   -Omega2 conj(cden) delw / |cden|^2 = -I_eps delw / (2 + 4 delw)
                //                                     = -(q / 2) / (wx + wt),
                // a pole at -wt, far from cancellation for wx > 0, with
                // wx + wt = (s, wt.im).
                const bool neg_f = NEG && wxv[f] < 0.00;
                if (!FOLD || neg_f) {
                    const double q_im_wti = FOLD ? q.im * wt.im : q_im_wti_e;
                    const double q_re_wti = FOLD ? q.re * wt.im : q_re_wti_e;
                    const cplx p = {__builtin_fma(q.re, wdr, -q_im_wti) * rden,
                                    __builtin_fma(q.im, wdr, q_re_wti) * rden};
                    if (nv > 0) {
                        cplx ssx = czero();
                        if (branch1) {
                            ssx = cscale(om2, c1[f]);
                        } else if (above2) {
                            const double s = wxv[f] + wt.re;
                            const double rr = 0.5 * rcp_1nr(__builtin_fma(s, s, wti2));
                            ssx = cplx{-__builtin_fma(q.re, s, q_im_wti) * rr, -__builtin_fma(q.im, s, -q_re_wti) * rr};
                        }
                        // The ssx cutoff of :58-59 (only at negative
                        // frequencies), decided on the reference's |ssx|.
                        // Branch 1: the reference's ssx is ((Omega2 wx^2)
                        // (1/wx^4)) (:38-41) with Omega2 already in its
                        // operation order.  Branch 2: this ssx is within about
                        // 2^-45 of the reference's, relative (rcp_1nr, the
                        // reduced form), so outside a 2^-40 band around the
                        // cutoff it decides as the reference does; inside it
                        // the reference's ssx is recomputed and decides.
                        if (neg_f) {
                            bool cut;
                            if (branch1) {
                                const double wx2 = wxv[f] * wxv[f];
                                cut = cabs_(cscale2(om2, wx2, 1.00 / (wx2 * wx2))) > ie_cut;
                            } else {
                                const double ax = cabs_(ssx);
                                cut = ax > ie_cut;
                                if (__builtin_fabs(ax - ie_cut) <= kBand * ie_cut)
                                    cut = occ_branch2_abs_ssx(wxv[f], wt, ie) > ie_cut;
                            }
                            if (cut) ssx = czero();
                        }
                        sasx[f] = cfma(ssx, mo, sasx[f]);
                    }
                    if constexpr (FOLD) {
                        if (branch1) sach[f] = cfma(p, mo, sach[f]);  // P Mu is in already
                    } else {
                        sach[f] = cfma(p, branch1 ? mum : mu, sach[f]);
                    }
                } else if (branch1) {  // P Mo and c1 Omega2 Mo
                    sach[f].re = __builtin_fma(__builtin_fma(uo.re, wdr, -uo_im_wti), rden, sach[f].re);
                    sach[f].im = __builtin_fma(__builtin_fma(uo.im, wdr, uo_re_wti), rden, sach[f].im);
                    sasx[f].re = __builtin_fma(c1[f], w1.re, sasx[f].re);
                    sasx[f].im = __builtin_fma(c1[f], w1.im, sasx[f].im);
                } else if (above2) {  // -(uo / 2) conj(wx + wt) / |wx + wt|^2
                    const double s = wxv[f] + wt.re;
                    const double rr = -0.5 * rcp_1nr(__builtin_fma(s, s, wti2));
                    sasx[f].re = __builtin_fma(rr, __builtin_fma(uo.re, s, uo_im_wti), sasx[f].re);
                    sasx[f].im = __builtin_fma(rr, __builtin_fma(uo.im, s, -uo_re_wti), sasx[f].im);
                }
                if (P2 && iw0 + f == a.acht_iw && iw0 + f < iw_end) {
                    const cplx pv = {__builtin_fma(q.re, wdr, -(FOLD ? q.im * wt.im : q_im_wti_e)) * rden,
                                     __builtin_fma(q.im, wdr, FOLD ? q.re * wt.im : q_re_wti_e) * rden};
                    __builtin_nontemporal_store(pv.re, &a.p2[row + ig].re);  // streamed, read once by the acht product
                    __builtin_nontemporal_store(pv.im, &a.p2[row + ig].im);
                    if constexpr (kOccSum) {
                        if (branch1) {  // sch = P (:37)
#pragma unroll
                            for (int n1 = 0; n1 < (kOccSum ? NV : 1); ++n1) oacc[n1] = cfma(av[n1], pv, oacc[n1]);
                        }
                    } else if (a.br1) {
                        a.br1[row + ig] = branch1 ? 1 : 0;
                    }
                }
            }
        }
        const double vc = a.vcoul[igp_of(a.idx, j, ncouls)];
#pragma unroll
        for (int f = 0; f < F; ++f) {
            const cplx s = block_sum(sach[f], scratch);
            const cplx x = block_sum(sasx[f], scratch);
            if (threadIdx.x == 0 && iw0 + f < iw_end) {
                // (0.5 * sum) * vcoul and sum * (occ * vcoul), gppComplex.cpp:361-363, :379
                const size_t o = ((size_t)j * a.nsplit + split) * a.nfreq + iw0 + f;
                a.col_ach[o] = cscale(cscale(s, 0.5), vc);
                a.col_asx[o] = cscale(x, a.occ * vc);
            }
        }
        if constexpr (kOccSum) {
            if (a.acht_iw >= iw0 && a.acht_iw < iw0 + F && a.acht_iw < iw_end) {  // uniform
                // 0.5 vcoul[igp(j)] conj(aqsm[n1,igp(j)]) sum, gppComplex.cpp:381
                const double w = 0.5 * vc;
#pragma unroll
                for (int n1 = 0; n1 < (kOccSum ? NV : 1); ++n1) {
                    const cplx s = block_sum(oacc[n1], scratch);
                    if (threadIdx.x == 0)
                        a.part_occ[((size_t)j * a.nsplit + split) * NV + n1] = cscale(cmul_fast(bgc[n1], s), w);
                }
            }
        }
    };
    // The choice depends on the problem's frequency count only, so every
    // grouping of its frequencies into passes (and blocks) sums alike.
    using fold_off = std::integral_constant<bool, false>;
    using fold_on = std::integral_constant<bool, true>;
    int iw0 = iw_begin;
    if constexpr (FC <= 3) {
        for (; iw_end - iw0 > FCT; iw0 += FC) pass(std::integral_constant<int, FC>(), fold_off(), iw0);
        if (iw0 < iw_end) pass(std::integral_constant<int, FCT>(), fold_off(), iw0);
    } else if (a.nfreq < 4) {  // at most 3 frequencies: one pass FCT (>= 4) wide
        if (iw0 < iw_end) pass(std::integral_constant<int, FCT>(), fold_off(), iw0);
    } else if constexpr (FC >= 16) {
        // passes of 16 while more than 12 remain, then at most one of 8 and
        // one of 4, so no pass runs more than 3 idle frequencies beyond the
        // first (24: 16 + 8 instead of 16 + 16)
        for (; iw_end - iw0 > 12; iw0 += 16) pass(std::integral_constant<int, 16>(), fold_on(), iw0);
        if (iw_end - iw0 > 4) {
            pass(std::integral_constant<int, 8>(), fold_on(), iw0);
            iw0 += 8;
        }
        if (iw0 < iw_end) pass(std::integral_constant<int, 4>(), fold_on(), iw0);
    } else if constexpr (FC == 8) {
        // passes of 8 while more than 8 remain, then one of 8, 6, 4 or 2: at
        // most one idle frequency (13: 8 + 6; C4 reduce 11.5 -> 11.1 ms
        // against a last pass of 4 or 8)
        for (; iw_end - iw0 > 8; iw0 += 8) pass(std::integral_constant<int, 8>(), fold_on(), iw0);
        const int rem = iw_end - iw0;
        if (rem > 6)
            pass(std::integral_constant<int, 8>(), fold_on(), iw0);
        else if (rem > 4)
            pass(std::integral_constant<int, 6>(), fold_on(), iw0);
        else if (rem > 2)
            pass(std::integral_constant<int, 4>(), fold_on(), iw0);
        else if (rem > 0)
            pass(std::integral_constant<int, 2>(), fold_on(), iw0);
    } else {
        for (; iw_end - iw0 > FCT; iw0 += FC) pass(std::integral_constant<int, FC>(), fold_on(), iw0);
        if (iw0 < iw_end) pass(std::integral_constant<int, FCT>(), fold_on(), iw0);
    }
}

// One element's pole terms at F frequencies, evaluated as pole_reduce_item
// does with fewer than four frequencies and none negative: P = delw I_eps
// formed per frequency, sch = P Mu, or P (Mu + Mo) in branch 1; ssx from the
// branch (branch 1: c1 Omega2; branch 2: the reduced form -(q / 2) /
// (wx + wt)) times Mo.  occ: the problem has occupied bands.
template <int F>
__device__ __forceinline__ void pole_element_plain(const double (&wxv)[F], const double (&c1)[F], bool occ, cplx wt,
                                                   cplx ie, cplx mu, cplx mo, cplx (&sach)[F], cplx (&sasx)[F])
{
#pragma clang fp contract(off)
    const cplx q = cmul_fast(wt, ie);
    const double wti2 = wt.im * wt.im;  // rounded as the reference's |wdiff|^2 rounds it
    const double q_im_wti = q.im * wt.im, q_re_wti = q.re * wt.im;
    cplx om2 = czero(), mum = mu;
    double wt2 = 0.0;
    if (occ) {
        om2 = cmul(csquare(wt), ie);  // Omega2 = wtilde^2 * I_eps, flagOCC_solver :117-118
        mum = cadd(mu, mo);
        wt2 = __builtin_fma(wt.re, wt.re, wti2);
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const double wdr = wxv[f] - wt.re;       // wdiff = (wdr, -wt.im), :27
        const double wdiffr = wdr * wdr + wti2;  // |wdiff|^2 exactly as the reference rounds it
        const double rden = rcp_1nr(wdiffr);
        bool branch1 = false, above2 = false;
        if (occ) occ_branch_tests(wxv[f], wt, wdiffr, rden, wt2, branch1, above2);
        const cplx p = {__builtin_fma(q.re, wdr, -q_im_wti) * rden, __builtin_fma(q.im, wdr, q_re_wti) * rden};
        if (occ) {
            cplx ssx = czero();
            if (branch1) {
                ssx = cscale(om2, c1[f]);
            } else if (above2) {
                const double sr = wxv[f] + wt.re;
                const double rr = 0.5 * rcp_1nr(__builtin_fma(sr, sr, wti2));
                ssx = cplx{-__builtin_fma(q.re, sr, q_im_wti) * rr, -__builtin_fma(q.im, sr, -q_re_wti) * rr};
            }
            sasx[f] = cfma(ssx, mo, sasx[f]);
        }
        sach[f] = cfma(p, branch1 ? mum : mu, sach[f]);
    }
}

// Inputs and outputs of the Gram product with the pole reduce fused into its
// epilogue (at most 3 frequencies, none negative, acht_n1_loc not requested).
struct PoleTileArgs {
    const cplx *aqsn, *ieps, *wtilde;
    const cplx *bg;  // [nb][ngpown]
    const double *wx;
    int nb, nv, ncouls, ngpown, nsplit;  // nsplit = G-vector tiles
    cplx *col_ach, *col_asx;             // [ngpown][nsplit][F], unscaled tile sums
    Stamp stamp;
};

// LDS of the fused Gram + pole reduce block (128 x 128 tile, 8 waves), in
// complex entries: the Gram's double-buffered band stages (sB, sA: 4096
// entries) during the product; afterwards, for the epilogue rounds, wtilde,
// I_eps and Mu of 32 columns x 64 G-vectors (rows padded to 65 entries, so
// the transposed reads of 8 lanes fall in 8 different 16-byte bank groups),
// conj(Bg) and aqsn of the tile's occupied bands (at most kFuseNv), and the
// per-wave column sums of one column round.
constexpr int kFuseNv = 4;
template <int F> struct FuseLds {
    typedef FuseCfg C;
    static constexpr int kCols = 32, kRows = 64;   // columns x G-vectors per round
    static constexpr int kPitch = kRows + 1;       // entries per staged row
    static constexpr int kWt = 0, kIe = kCols * kPitch, kMu = 2 * kCols * kPitch;
    static constexpr int kBg = 3 * kCols * kPitch;     // [kFuseNv][TJ]
    static constexpr int kAq = kBg + kFuseNv * C::TJ;  // [kFuseNv][TI]
    static constexpr int kRed = kAq + kFuseNv * C::TI;  // [WIN = 4][kCols][2F]
    static constexpr int kTotal = kRed + 4 * kCols * 2 * F;
    static constexpr int kGram = 2 * C::KS * (C::TJ + C::TI);  // the Gram's stage buffers
    static constexpr int kLds = kTotal > kGram ? kTotal : kGram;
};

// Epilogue of one 128 x 128 tile (G-vector tile `itile`) after
// gram_f64_acc: the accumulators are folded into Mu at once (128
// registers instead of 192), and the elements are evaluated in eight rounds
// (s, t): 32 columns (sub-tile s of both 64-column halves) x 64 G-vectors
// (sub-tile t of the four 32-G-vector quarters).  In a round all 512 threads
// stage its wtilde and I_eps rows into LDS with coalesced loads (the tile's
// occupied conj(Bg) and aqsn with the first), each wave writes its Mu of the
// round beside them, and each lane evaluates its four elements of the round
// in a loop -- Mo over the occupied bands (four FMAs per band), the pole
// terms at the F frequencies (pole_element_plain) -- summing per column over
// both rounds of a column sub-tile; then the four lane groups are summed by
// xor butterfly (every lane of a column ends with the same bits) and the
// four waves of a column range in wave order: one sum per (column, tile,
// frequency), written unscaled.
template <int F>
__device__ __forceinline__ void gram_pole_epilogue(const PoleTileArgs &a, int j0, int i0, int itile,
                                                   const v4d (&acc1)[4][2], const v4d (&acc2)[4][2],
                                                   const v4d (&acc3)[4][2], cplx *lds)
{
#pragma clang fp contract(off)
    typedef FuseLds<F> L;
    typedef FuseCfg C;
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int wjn = wave / 4, wv = wave % 4;  // 64-column half, 32-G-vector quarter
    const int ncouls = a.ncouls, ngpown = a.ngpown, nv = a.nv;

    cplx mu[4][2][4];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                mu[s][t][r] = cplx{acc1[s][t][r] + acc2[s][t][r], (acc3[s][t][r] - acc1[s][t][r]) + acc2[s][t][r]};

    double wxv[F], c1[F];  // branch-1 ssx = Omega2 * wx^2 / wx^4 (:38-41) = Omega2 * c1
#pragma unroll
    for (int f = 0; f < F; ++f) {
        wxv[f] = a.wx[f];
        const double wx2 = wxv[f] * wxv[f];
        c1[f] = wx2 * (1.00 / (wx2 * wx2));
    }
    // tile-local column of staged row c and G-vector of staged entry q in round (s, t)
    auto col_of = [](int c, int s) { return (c >> 4) * kWJ + 16 * s + (c & 15); };
    auto gv_of = [](int q, int t) { return (q >> 4) * kWI + 16 * t + (q & 15); };
    constexpr int PER = L::kCols * L::kRows / C::NT;  // staged entries per thread and array (4)
    const int jc = wjn * 16 + lane % 16;              // this lane's staged row

#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int jl = col_of(jc, s);
        cplx sach[F], sasx[F];
#pragma unroll
        for (int f = 0; f < F; ++f) sach[f] = sasx[f] = czero();
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int arr = 0; arr < 2; ++arr) {
                const cplx *src = arr ? a.ieps : a.wtilde;
                cplx v[PER];
#pragma unroll
                for (int k = 0; k < PER; ++k) {
                    const int e = threadIdx.x + k * C::NT;
                    const int j = j0 + col_of(e / L::kRows, s), ig = i0 + gv_of(e % L::kRows, t);
                    v[k] = (j < ngpown && ig < ncouls) ? src[(size_t)j * ncouls + ig] : czero();
                }
#pragma unroll
                for (int k = 0; k < PER; ++k) {
                    const int e = threadIdx.x + k * C::NT;
                    lds[(arr ? L::kIe : L::kWt) + (e / L::kRows) * L::kPitch + e % L::kRows] = v[k];
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) lds[L::kMu + jc * L::kPitch + wv * 16 + 4 * r + lane / 16] = mu[s][t][r];
            if (s == 0 && t == 0) {
                for (int e = threadIdx.x; e < nv * C::TJ; e += C::NT) {
                    const int n = e / C::TJ, c = e % C::TJ;
                    lds[L::kBg + e] = j0 + c < ngpown ? cconj(a.bg[(size_t)n * ngpown + j0 + c]) : czero();
                    lds[L::kAq + e] = i0 + c < ncouls ? a.aqsn[(size_t)n * ncouls + i0 + c] : czero();
                }
            }
            __syncthreads();
            if (j0 + jl < ngpown) {
#pragma unroll 1
                for (int r = 0; r < 4; ++r) {
                    const int q = wv * 16 + 4 * r + lane / 16;  // staged entry
                    const int igl = gv_of(q, t);
                    if (i0 + igl < ncouls) {
                        cplx mo = czero();  // occupied bands in band order
                        for (int n1 = 0; n1 < nv; ++n1)
                            mo = cfma(lds[L::kBg + n1 * C::TJ + jl], lds[L::kAq + n1 * C::TI + igl], mo);
                        const int o = jc * L::kPitch + q;
                        pole_element_plain<F>(wxv, c1, nv > 0, lds[L::kWt + o], lds[L::kIe + o], lds[L::kMu + o], mo,
                                              sach, sasx);
                    }
                }
            }
            // every wave's reads of the round's rows are done before the next
            // round stages over them
            __syncthreads();
        }
#pragma unroll
        for (int f = 0; f < F; ++f) {
#pragma unroll
            for (int m = 16; m < kWave; m <<= 1) {
                sach[f].re += __shfl_xor(sach[f].re, m, kWave);
                sach[f].im += __shfl_xor(sach[f].im, m, kWave);
                sasx[f].re += __shfl_xor(sasx[f].re, m, kWave);
                sasx[f].im += __shfl_xor(sasx[f].im, m, kWave);
            }
        }
        if (lane < 16) {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                lds[L::kRed + (wv * L::kCols + jc) * 2 * F + f] = sach[f];
                lds[L::kRed + (wv * L::kCols + jc) * 2 * F + F + f] = sasx[f];
            }
        }
        // the next column round writes its sums only after two more barriers
        __syncthreads();
        for (int e = threadIdx.x; e < L::kCols * 2 * F; e += C::NT) {
            const int c = e / (2 * F), k = e % (2 * F);
            const int j = j0 + col_of(c, s);
            if (j >= ngpown) continue;
            cplx v = lds[L::kRed + c * 2 * F + k];
#pragma unroll
            for (int w = 1; w < 4; ++w) v = cadd(v, lds[L::kRed + (w * L::kCols + c) * 2 * F + k]);
            const size_t o = ((size_t)j * a.nsplit + itile) * F + (k % F);
            if (k < F)
                a.col_ach[o] = v;
            else
                a.col_asx[o] = v;
        }
    }
}

// Column sums of the fused epilogue's tile sums: one wave per column j, the
// tiles summed in a fixed order (strided per lane, then xor butterfly), then
// scaled as the reduce scales them, (0.5 * sum) * vcoul and sum * (occ *
// vcoul) (gppComplex.cpp:361-363, :379); out [ngpown][nfreq].
__device__ __forceinline__ void pole_cols_wave(const cplx *col_ach, const cplx *col_asx, int nsplit, int nfreq,
                                               const int32_t *idx, const double *vcoul, int ncouls, double occ,
                                               int j, cplx *out_ach, cplx *out_asx)
{
    const int lane = threadIdx.x % kWave;
    const double vc = vcoul[igp_of(idx, j, ncouls)];
    for (int f = 0; f < nfreq; ++f) {
        cplx s = czero(), x = czero();
        for (int it = lane; it < nsplit; it += kWave) {
            s = cadd(s, col_ach[((size_t)j * nsplit + it) * nfreq + f]);
            x = cadd(x, col_asx[((size_t)j * nsplit + it) * nfreq + f]);
        }
        s = wave_sum(s);
        x = wave_sum(x);
        if (lane == 0) {
            out_ach[(size_t)j * nfreq + f] = cscale(cscale(s, 0.5), vc);
            out_asx[(size_t)j * nfreq + f] = cscale(x, occ * vc);
        }
    }
}

// acht_n1_loc (gppComplex.cpp:381, sch_array[2] of each band and column):
//   acht[n1] = sum_j 0.5 vcoul[igp(j)] conj(aqsm[n1,igp(j)]) sum_ig aqsn[n1,ig] R[j,ig]
// with R = p2 (P = delw*I_eps at that frequency) for the unoccupied bands and
// R = p2 masked by br1 (sch of ssxt_scht_solver, :37) for the occupied ones
// (acht_occ_item below: few bands, a streaming pass).  For the unoccupied
// bands Y = R * aqsn^T is a second Gram-type product (rows j, columns n1, K = G);
// one block computes a TJ x TN tile of Y over G-vectors [k_begin, k_end) on
// v_mfma_f64_16x16x4f64 with three real products per complex product (3M:
// P1 = sum rr ar, P2 = sum ri ai, P3 = sum (rr + ri)(ar + ai), Re Y = P1 - P2,
// Im Y = (P3 - P1) - P2) and reduces it at once to the column sums
// sum_j w_j conj(bg[n1][j]) Y[j][n1], written to part[n1] (one entry per
// column of the tile).  The tile runs through the same ring of LDS stages as
// gram_ring_tile (C::KS = 8 G-vectors a stage), both operands K-fastest: rows
// of 8 complex (128 bytes), element (row, k) at slot k ^ (row & 7), which makes
// the MFMA reads (16 rows per 16 lanes) free of LDS bank conflicts on gfx950
// (a padded pitch of 9 complex is not); each lane of a stage's loads takes the
// element its slot holds.  Bounded by the FP64 MFMA pipe, as the Gram product.
// Rows and bands past the edge load the last one (their results are dropped),
// G-vectors past the end the last one, counted as zero.  SJ <= C::SJ: sub-tile
// rows per wave, fewer for a last tile with fewer rows.
template <class C, int SJ>
__device__ __forceinline__ void acht_ring_tile(const cplx *__restrict__ p2, const cplx *__restrict__ aqsn,
                                               const cplx *__restrict__ bg, const int32_t *__restrict__ idx,
                                               const double *__restrict__ vcoul, int ngpown, int ncouls, int n1_end,
                                               int k_begin, int k_end, int j0, int c0, cplx *lds,
                                               cplx *__restrict__ part)
{
    constexpr int KS = C::KS, NB = C::NB, TJ = C::TJ, TN = C::TI, SI = C::SI, NW = C::NW;
    constexpr int QR = KS * TJ / 64 / NW, QA = KS * TN / 64 / NW, LD = QR + QA;  // loads per wave and stage
    static_assert(KS == 8 && QR * 64 * NW == KS * TJ && QA * 64 * NW == KS * TN && NB >= 3,
                  "rows of 8, loads split evenly over the waves");
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int wjn = wave / C::WIN;
    const int wj = wjn * (16 * SJ), wi = (wave % C::WIN) * (16 * SI);
    const int nst = (k_end - k_begin + KS - 1) / KS;  // >= 1: a split is never empty

    // Load q of a side fills rows [8 (q NW + wave), +8): lane l row l / 8,
    // slot l % 8, so G-vector (l % 8) ^ (l / 8) of the stage.
    const int lk = (lane % 8) ^ (lane / 8);
    const cplx *pr[QR], *pa[QA];
#pragma unroll
    for (int q = 0; q < QR; ++q)
        pr[q] = p2 + (size_t)min(j0 + 8 * (q * NW + wave) + lane / 8, ngpown - 1) * ncouls + k_begin + lk;
#pragma unroll
    for (int q = 0; q < QA; ++q)
        pa[q] = aqsn + (size_t)min(c0 + 8 * (q * NW + wave) + lane / 8, n1_end - 1) * ncouls + k_begin + lk;
    int ibuf = 0, rbuf = 0;  // next buffer to fill, to read
    // over: how far this lane's G-vector lies past the end (last stage only)
    auto issue = [&](int over) {
        cplx *buf = lds + ibuf * C::STAGE + 64 * wave;
        ibuf = ibuf + 1 == NB ? 0 : ibuf + 1;
#pragma unroll
        for (int q = 0; q < QR; ++q) {
            ring_load(pr[q] - over, buf + 64 * NW * q);
            pr[q] += KS;
        }
#pragma unroll
        for (int q = 0; q < QA; ++q) {
            ring_load(pa[q] - over, buf + KS * TJ + 64 * NW * q);
            pa[q] += KS;
        }
    };
    const int over_last = max(0, k_begin + (nst - 1) * KS + lk - (k_end - 1));

    v4d acc1[SJ][SI], acc2[SJ][SI], acc3[SJ][SI];  // P1, P2, P3
#pragma unroll
    for (int s = 0; s < SJ; ++s)
#pragma unroll
        for (int t = 0; t < SI; ++t) acc1[s][t] = acc2[s][t] = acc3[s][t] = v4d{0, 0, 0, 0};
    auto multiply = [&](auto last) {
        const cplx *sR = lds + rbuf * C::STAGE, *sA = sR + KS * TJ;
        rbuf = rbuf + 1 == NB ? 0 : rbuf + 1;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < KS; kk += 4) {
            const int kr = (kk + lane / 16) ^ (lane & 7);  // every row read below is = lane (mod 8)
            const bool out = last && k_begin + (nst - 1) * KS + kk + lane / 16 >= k_end;
            double are[SI], aim[SI], asum[SI];
#pragma unroll
            for (int t = 0; t < SI; ++t) {
                cplx a = sA[(wi + 16 * t + lane % 16) * KS + kr];
                if (out) a = czero();
                are[t] = a.re;
                aim[t] = a.im;
                asum[t] = a.re + a.im;
            }
#pragma unroll
            for (int s = 0; s < SJ; ++s) {
                cplx r = sR[(wj + 16 * s + lane % 16) * KS + kr];
                if (out) r = czero();
                const double rsum = r.re + r.im;
#pragma unroll
                for (int t = 0; t < SI; ++t) {
                    acc1[s][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(r.re, are[t], acc1[s][t], 0, 0, 0);
                    acc2[s][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(r.im, aim[t], acc2[s][t], 0, 0, 0);
                    acc3[s][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(rsum, asum[t], acc3[s][t], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
    };
    // the schedule of gram_ring_tile
    for (int st = 0; st < NB - 1 && st < nst; ++st) issue(st < nst - 1 ? 0 : over_last);
    int st = 0;
    for (; st < nst - NB; ++st) {
        wait_vm_lds<(NB - 2) * LD>();
        ring_barrier();
        issue(0);
        multiply(std::integral_constant<bool, false>());
    }
    if (nst >= NB) {
        wait_vm_lds<(NB - 2) * LD>();
        ring_barrier();
        issue(over_last);
        multiply(std::integral_constant<bool, false>());
        ++st;
    }
    for (; st < nst - 1; ++st) {
        wait_vm_lds<0>();
        ring_barrier();
        multiply(std::integral_constant<bool, false>());
    }
    wait_vm_lds<0>();
    ring_barrier();
    multiply(std::integral_constant<bool, true>());

    // Epilogue: result r of lane l is Y[j][n1] with j = 4r + l/16 + 16s + wj,
    // n1 = l%16 + 16t + wi.  Weight by 0.5 vcoul[igp(j)] conj(bg[n1][j]), sum
    // the wave's 16 SJ rows (fixed order: s, r, then the xor butterfly over
    // l/16), then the WJN waves of one column range in wave order.
    __syncthreads();  // every wave is done with the stages
    auto *red = reinterpret_cast<cplx(*)[TN]>(lds);
    cplx sum[SI];
#pragma unroll
    for (int t = 0; t < SI; ++t) sum[t] = czero();
#pragma unroll
    for (int s = 0; s < SJ; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = j0 + wj + 16 * s + 4 * r + lane / 16;
            if (j < ngpown) {
                const double w = 0.5 * vcoul[igp_of(idx, j, ncouls)];
#pragma unroll
                for (int t = 0; t < SI; ++t) {
                    const int n1 = min(c0 + wi + 16 * t + lane % 16, n1_end - 1);
                    const cplx b = bg[(size_t)n1 * ngpown + j];
                    const cplx y = cplx{acc1[s][t][r] - acc2[s][t][r], (acc3[s][t][r] - acc1[s][t][r]) - acc2[s][t][r]};
                    sum[t] = cadd(sum[t], cscale(cmul_fast(cconj(b), y), w));
                }
            }
        }
#pragma unroll
    for (int t = 0; t < SI; ++t) {
        sum[t].re += __shfl_xor(sum[t].re, 16);
        sum[t].im += __shfl_xor(sum[t].im, 16);
        sum[t].re += __shfl_xor(sum[t].re, 32);
        sum[t].im += __shfl_xor(sum[t].im, 32);
        if (lane < 16) red[wjn][wi + 16 * t + lane] = sum[t];
    }
    __syncthreads();
    for (int col = threadIdx.x; col < TN; col += C::NT) {
        cplx s = czero();
#pragma unroll
        for (int w2 = 0; w2 < C::WJN; ++w2) s = cadd(s, red[w2][col]);
        if (c0 + col < n1_end) part[c0 + col] = s;
    }
}

// acht_n1_loc of the occupied bands n1 < nv for column j over G-vectors
// [split*chunk, +chunk): sum_ig aqsn[n1,ig] p2[j,ig] where the occupied solver
// took branch 1 (sch = P, else 0), bands in groups of 8 held in registers,
// block-wide fixed-order sums, weighted by 0.5 vcoul[igp(j)]
// conj(aqsm[n1,igp(j)]) and written to part[n1] (nv entries).
__device__ __forceinline__ void acht_occ_item(const cplx *__restrict__ p2, const uint8_t *__restrict__ br1,
                                              const cplx *__restrict__ aqsn, const cplx *__restrict__ bg,
                                              const int32_t *__restrict__ idx, const double *__restrict__ vcoul,
                                              int ngpown, int ncouls, int nv, int chunk, int j, int split,
                                              cplx *__restrict__ part, cplx *scratch)
{
    constexpr int G = 8;
    const int ig_begin = split * chunk;
    const int ig_end = ig_begin + chunk < ncouls ? ig_begin + chunk : ncouls;
    const size_t row = (size_t)j * ncouls;
    const double w = 0.5 * vcoul[igp_of(idx, j, ncouls)];
    for (int n0 = 0; n0 < nv; n0 += G) {
        cplx acc[G];
#pragma unroll
        for (int u = 0; u < G; ++u) acc[u] = czero();
        for (int ig = ig_begin + threadIdx.x; ig < ig_end; ig += blockDim.x) {
            if (!br1[row + ig]) continue;
            const cplx q = p2[row + ig];
#pragma unroll
            for (int u = 0; u < G; ++u)
                if (n0 + u < nv) acc[u] = cfma(aqsn[(size_t)(n0 + u) * ncouls + ig], q, acc[u]);
        }
#pragma unroll
        for (int u = 0; u < G; ++u) {
            if (n0 + u >= nv) break;  // uniform
            const cplx s = block_sum(acc[u], scratch);
            if (threadIdx.x == 0)
                part[n0 + u] = cscale(cmul_fast(cconj(bg[(size_t)(n0 + u) * ngpown + j]), s), w);
        }
    }
}

// Stage 3 of buckets without occupied bands (band-dependent frequencies): one
// pass over the elements of column j and G-vectors [split*chunk, +chunk)
// evaluates every bucket's pole terms and adds them to the same sums, so
// wtilde and I_eps are read once for all buckets instead of once for each and
// a block has only its F sums to reduce.  A thread holds kBareE elements; each
// bucket's Mu loads while the one before is evaluated.  What bounds it is the
// memory below about four frequencies, the FP64 units above.  F frequencies
// from blockIdx.z * F.
constexpr int kBareE = 4, kBareStep = kBareE * kRedThreads;
struct BareArgs {
    const cplx *mu;        // [nslots][ngpown][ncouls]
    const int32_t *slots;  // [nslots][3]: the third entry is the slot's row of wx
    int nslots;
    const cplx *ieps, *wtilde;
    const int32_t *idx;
    const double *vcoul, *wx;
    int ncouls, ngpown, nfreq, nsplit, chunk;
    cplx *col_ach, *col_asx;  // [ngpown][nsplit][nfreq]
};
template <int F> __device__ __forceinline__ void pole_reduce_bare(const BareArgs &a, cplx *scratch)
{
    const int j = blockIdx.x, split = blockIdx.y, iw0 = blockIdx.z * F;
    const int ig_begin = split * a.chunk;
    const int ig_end = ig_begin + a.chunk < a.ncouls ? ig_begin + a.chunk : a.ncouls;
    const size_t row = (size_t)j * a.ncouls, mu_step = (size_t)a.ngpown * a.ncouls;
    cplx sach[F];
#pragma unroll
    for (int f = 0; f < F; ++f) sach[f] = czero();
    auto ld = [](const cplx *p) {  // read once
        return cplx{__builtin_nontemporal_load(&p->re), __builtin_nontemporal_load(&p->im)};
    };
    for (int ig0 = ig_begin + threadIdx.x; ig0 < ig_end; ig0 += kBareStep) {
        cplx wt[kBareE], q[kBareE], mu[kBareE];
        double wti2[kBareE];
        size_t at[kBareE];
#pragma unroll
        for (int e = 0; e < kBareE; ++e) {  // elements past the end load the last one again and add nothing
            at[e] = row + min(ig0 + e * kRedThreads, ig_end - 1);
            wt[e] = a.wtilde[at[e]];
            q[e] = a.ieps[at[e]];
            mu[e] = ld(a.mu + at[e]);
        }
#pragma unroll
        for (int e = 0; e < kBareE; ++e) {
            q[e] = cmul_fast(wt[e], q[e]);
            wti2[e] = wt[e].im * wt[e].im;
        }
        const cplx *mub = a.mu;
        for (int b = 0; b < a.nslots; ++b) {
            const double *const wx = a.wx + (size_t)a.slots[3 * b + 2] * a.nfreq;
            double wxv[F];
#pragma unroll
            for (int f = 0; f < F; ++f) wxv[f] = wx[min(iw0 + f, a.nfreq - 1)];
            if (b + 1 < a.nslots) mub += mu_step;
            cplx mu_n[kBareE];
#pragma unroll
            for (int e = 0; e < kBareE; ++e) mu_n[e] = ld(mub + at[e]);
#pragma unroll
            for (int e = 0; e < kBareE; ++e) {
                if (ig0 + e * kRedThreads >= ig_end) break;
                // u conj(wdiff) / |wdiff|^2 with u = q Mu (pole_reduce_item)
                const cplx u = cmul_fast(q[e], mu[e]);
                const double uiw = u.im * wt[e].im, urw = u.re * wt[e].im;
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    const double wdr = wxv[f] - wt[e].re;
                    const double rden = rcp_1nr(__builtin_fma(wdr, wdr, wti2[e]));
                    sach[f].re = __builtin_fma(__builtin_fma(u.re, wdr, -uiw), rden, sach[f].re);
                    sach[f].im = __builtin_fma(__builtin_fma(u.im, wdr, urw), rden, sach[f].im);
                }
            }
#pragma unroll
            for (int e = 0; e < kBareE; ++e) mu[e] = mu_n[e];
        }
    }
    const double vc = a.vcoul[igp_of(a.idx, j, a.ncouls)];
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const cplx s = block_sum(sach[f], scratch);
        if (threadIdx.x == 0 && iw0 + f < a.nfreq) {
            const size_t o = ((size_t)j * a.nsplit + split) * a.nfreq + iw0 + f;
            a.col_ach[o] = cscale(cscale(s, 0.5), vc);
            a.col_asx[o] = czero();
        }
    }
}

// Stage 4: block `part` < nfreq forms achtemp[part] / asxtemp[part] as
// fixed-order sums over the (column, split) partials; block part == nfreq
// sets acht_n1_loc to NaN (nan_acht; the factored forms write it in a stage of
// its own when it is requested) and sums the per-(band, column group) achstemp
// partials.
__device__ __forceinline__ void final_block(const cplx *col_ach, const cplx *col_asx, const cplx *part_achs,
                                            long long ncols, int nfreq, int nb, int nv, cplx *out, cplx *scratch, int part,
                                            bool nan_acht = true)
{
    if (part < nfreq) {
        const int iw = part;
        cplx s = czero(), x = czero();
        for (long long c = threadIdx.x; c < ncols; c += blockDim.x) {
            s = cadd(s, col_ach[(size_t)c * nfreq + iw]);
            x = cadd(x, col_asx[(size_t)c * nfreq + iw]);
        }
        s = block_sum(s, scratch);
        x = block_sum(x, scratch);
        if (threadIdx.x == 0) {
            out[iw] = s;
            out[nfreq + iw] = nv > 0 ? x : czero();
        }
        return;
    }
    const double nan = __builtin_nan("");
    for (int n1 = threadIdx.x; nan_acht && n1 < nb; n1 += blockDim.x) out[2 * nfreq + n1] = cplx{nan, nan};
    cplx h = czero();
    for (int t = threadIdx.x; t < nb * kAchSplit; t += blockDim.x) h = cadd(h, part_achs[t]);
    h = block_sum(h, scratch);
    if (threadIdx.x == 0) out[2 * nfreq + nb] = h;
}

}  // namespace fact
}  // namespace gpp
