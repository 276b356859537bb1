// gpp_factored.hip -- factored form of the GPP sigma band loop on gfx950,
// one problem per call (the batched persistent form is gpp_batch.hip).
//
// Stages (device bodies in gpp_factored_dev.hpp):
//   1. k_achstemp      Bg[n1][j] = aqsm[n1][igp(j)] (13 MB at 512x1638) and the
//                      achstemp band sums (reduce_achstemp, gppComplex.cpp:66-101)
//   2. Gram product    Mu = conj(Bg)^T * aqsn over bands [nv, nb):
//        FP64 MFMA (k_gram_f64 or k_gram_small, tile by gram_tile_for), or the Ozaki
//        split of gpp_ozaki.hip; written to HBM as [ngpown][ncouls]
//   3. k_pole_reduce   streams wtilde, I_eps, Mu (and the nv occupied aqsn rows),
//                      evaluates the pole factors in FP64, reduces per column
//   4. k_fact_final    fixed-order column reduction; achstemp (reduce_achstemp,
//                      gppComplex.cpp:66-101) from k_achstemp.
// When acht_n1_loc is requested (GramKind::acht), stage 3 also writes the
// pole factor p2 of frequency 2 and, with two occupied bands (and no negative
// frequency), sums the occupied bands' terms (the masked p2 against their
// aqsn rows, already loaded for Mo); and
//   5. k_acht_f64      second FP64 MFMA product Y = P2 * aqsn^T for the
//                      unoccupied bands, split over G-vectors, reduced per
//                      band in its epilogue; for the other occupied band
//                      counts k_acht_occ streams the masked P2 (stage 3
//                      writes the branch mask) against the occupied aqsn rows
//   6. k_acht_final    fixed-order sum of the per-band partials.
#include <math.h>
#include <string.h>

#include <algorithm>

#include "gpp_factored_dev.hpp"

namespace gpp {
namespace {

using namespace fact;

__host__ inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

constexpr double kGramCus = 256;  // compute units of an MI355X

// Rounds of blocks over the CUs for `whole` tiles and then `halves` tiles of
// half their work, which fill the last round as far as they fit.
double tile_rounds(double whole, double halves)
{
    const double rounds = ceil(whole / kGramCus), over = halves / 2 - (rounds * kGramCus - whole);
    return over > 0 ? rounds + ceil(2 * over / kGramCus) / 2 : rounds;
}

// acht product tiles (rows j x bands): 64 x 128, or 64 x 64 (narrow).
struct AchtSplit {
    int jtiles, ntiles, nks, chunk;
    bool narrow;
    bool cut;  // the last j tile has at most 32 rows: one sub-tile row per wave
};

// Tile and split of the G-vector sum of the acht product: the least estimated
// time over splits that give each CU a whole number of blocks.  A block's
// k-steps run at the Gram product's rates (gram_tile_for); kBlock covers its
// first loads and its epilogue, kPart the fixed-order sum of the partials.
// acht stage, us, against one 128 x 128 tile staged through registers and at
// least 512 G-vectors a block: 24/2/1000/50 389 -> 14, 512/2/4096/409
// 227 -> 110, 512/2/32768/1638 2805 -> 2550.
AchtSplit acht_split(const DevProblem &p)
{
    AchtSplit a;
    const int nu = p.nb - p.nv, rem = p.ngpown % GramL::TJ;
    a.jtiles = (p.ngpown + GramL::TJ - 1) / GramL::TJ;
    a.cut = rem > 0 && rem <= GramL::TJ / 2;
    const double kBlock = 3.0, kPart = 0.01;  // us
    double best = 1e300;
    for (int narrow = 0; narrow < 2; ++narrow) {
        const int tn = narrow ? GramM::TI : GramL::TI;
        const int ntiles = std::max(1, (nu + tn - 1) / tn);
        const double tiles = (a.jtiles - (a.cut ? 0.5 : 0.0)) * ntiles, sub = GramL::TJ / 16 * (tn / 16);
        const double whole = (a.jtiles - (a.cut ? 1 : 0)) * ntiles, halves = a.cut ? ntiles : 0;
        for (int r = 1; r <= 32; ++r) {
            int nks = (int)(r * kGramCus / tiles);
            nks = std::max(1, std::min(nks, (p.ncouls + 31) / 32));
            const int chunk = ((p.ncouls + nks - 1) / nks + GramL::KS - 1) / GramL::KS * GramL::KS;
            nks = (p.ncouls + chunk - 1) / chunk;
            const double rounds = tile_rounds(whole * nks, halves * nks);
            const double rate = rounds <= 1 ? (narrow ? 0.0287 : 0.0258) : narrow ? 0.0247 : 0.0237;
            const double us = rounds * (sub * (chunk / 4) * rate + kBlock) + kPart * a.jtiles * nks;
            if (us < best) best = us, a.nks = nks, a.chunk = chunk, a.ntiles = ntiles, a.narrow = narrow != 0;
        }
    }
    return a;
}

// The fused Gram + pole reduce (k_gram_pole) serves at most three
// frequencies, none negative, at most kFuseNv occupied bands, without
// acht_n1_loc, on its own 128 x 128 FP64 tile.
bool fused_reduce(const DevProblem &p, const GramKind &k)
{
    return k.fuse && k.ozaki_slices == 0 && k.tile == 0 && !k.acht && p.nfreq <= 3 && !p.wx_neg &&
           p.nv <= kFuseNv;
}

// Mu is stored past the caches when it is larger than the L2s (32 MB): it is
// written once and read back once, by the pole reduce.  us, plain against
// non-temporal stores: 512/2/32768/1638 (859 MB) reduce 510 -> 422, Gram alike;
// 512/2/32768/205 (107 MB) reduce 80 -> 72, Gram 357 -> 363.
// n products of one launch count together.
bool mu_streams(const DevProblem &p, int n) { return sizeof(cplx) * (size_t)p.ngpown * p.ncouls * n > ((size_t)32 << 20); }

// The products of one Gram launch: one over bands [nv, nb), or n of them over
// the rows in dev (gram_slot), `bands` in all.
struct GramSlots {
    const int32_t *dev = nullptr;
    int n = 1;
    long long bands = 0;
};

// G-vectors per block of k_acht_occ: the reduce's range, halved while the
// launch has fewer than 2048 blocks (each thread waits on its own loads:
// 100/8/3000/200/5 33 -> 21 us).
int acht_occ_chunk(const DevProblem &p, int red_chunk)
{
    int chunk = red_chunk;
    while (chunk > 512 && (long long)p.ngpown * ((p.ncouls + chunk - 1) / chunk) < 2048) chunk /= 2;
    return chunk;
}

// The frequency of acht_n1_loc: sch_array[2], gppComplex.cpp:381.
int acht_frequency(const DevProblem &p) { return p.nfreq > 2 ? 2 : p.nfreq - 1; }

struct FactLayout {
    size_t bg, m, col_ach, col_asx, col2_ach, col2_asx, part_achs, p2, br1, acht_part, acht_occ, total;
    int nsplit;  // G-vector ranges of the pole-reduce partials (the fused form: G-vector tiles)
    int occ_chunk = 0, occ_nsplit = 0;  // G-vector ranges of the occupied bands' acht_n1_loc partials
    bool fused;
    AchtSplit as;
};

FactLayout fact_layout(const DevProblem &p, const GramKind &k)
{
    FactLayout L;
    L.fused = fused_reduce(p, k);
    L.nsplit = L.fused ? (p.ncouls + FuseCfg::TI - 1) / FuseCfg::TI : (p.ncouls + k.red_chunk - 1) / k.red_chunk;
    size_t off = 0;
    L.bg = off;        off += align256(sizeof(cplx) * (size_t)p.nb * p.ngpown);
    L.m = off;         off += L.fused ? 0 : align256(sizeof(cplx) * (size_t)p.ngpown * p.ncouls);
    L.col_ach = off;   off += align256(sizeof(cplx) * (size_t)p.ngpown * L.nsplit * p.nfreq);
    L.col_asx = off;   off += align256(sizeof(cplx) * (size_t)p.ngpown * L.nsplit * p.nfreq);
    L.col2_ach = L.col2_asx = off;
    if (L.fused) {
        L.col2_ach = off; off += align256(sizeof(cplx) * (size_t)p.ngpown * p.nfreq);
        L.col2_asx = off; off += align256(sizeof(cplx) * (size_t)p.ngpown * p.nfreq);
    }
    L.part_achs = off; off += align256(sizeof(cplx) * ach_region_entries(p.nb, p.ngpown));
    L.p2 = L.br1 = L.acht_part = L.acht_occ = off;
    L.as = AchtSplit{};
    if (k.acht) {
        L.as = acht_split(p);
        L.p2 = off;        off += align256(sizeof(cplx) * (size_t)p.ngpown * p.ncouls);
        // branch-1 mask for k_acht_occ, where the reduce does not sum the
        // occupied bands itself
        L.br1 = off;       off += p.nv > 0 && !reduce_sums_acht_occ(p.nv, p.wx_neg) ? align256((size_t)p.ngpown * p.ncouls) : 0;
        L.acht_part = off; off += align256(sizeof(cplx) * (size_t)L.as.jtiles * L.as.nks * p.nb);
        L.occ_chunk = acht_occ_chunk(p, k.red_chunk);
        L.occ_nsplit = reduce_sums_acht_occ(p.nv, p.wx_neg) ? L.nsplit : (p.ncouls + L.occ_chunk - 1) / L.occ_chunk;
        L.acht_occ = off;  off += align256(sizeof(cplx) * (size_t)p.ngpown * L.occ_nsplit * (p.nv > 0 ? p.nv : 1));
    }
    L.total = off;
    return L;
}

// Product blockIdx.y of a launch over several (band-dependent frequencies):
// its bands are rows [slots[3y], slots[3y+1]), its Mu is the y-th.
__device__ __forceinline__ void gram_slot(const int32_t *slots, int ngpown, int ncouls, int &k_begin, int &k_end,
                                          cplx *__restrict__ &mout)
{
    if (!slots) return;
    k_begin = slots[3 * blockIdx.y];
    k_end = slots[3 * blockIdx.y + 1];
    mout += (size_t)blockIdx.y * ngpown * ncouls;
}

// Grid x over the ceil(ngpown/TJ) x ceil(ncouls/TI) tiles, G' tiles
// fastest in tile order and tiles spread over the XCDs by xcd_tile, so the
// blocks sharing one aqsn tile run on one XCD.  The last G' tile runs SJR <= SJ
// sub-tiles per wave, as many as its columns need (the launcher picks SJR).
template <class C, int SJR, bool NTS>
__global__ __launch_bounds__(C::NT) __attribute__((amdgpu_waves_per_eu(C::OCC))) void k_gram_f64(
    const cplx *__restrict__ bg, const cplx *__restrict__ aqsn, int ngpown, int ncouls, int k_begin, int k_end,
    const int32_t *__restrict__ slots, cplx *__restrict__ mout, Stamp stamp)
{
    stamp_start(stamp);
    __shared__ cplx lds[C::LDS];
    gram_slot(slots, ngpown, ncouls, k_begin, k_end, mout);
    const int nj = (ngpown + C::TJ - 1) / C::TJ, ni = (ncouls + C::TI - 1) / C::TI;
    if constexpr (SJR == C::SJ) {
        const int t = xcd_tile(blockIdx.x, nj * ni);
        gram_ring_tile<C, C::SJ, NTS>(bg, aqsn, ngpown, ncouls, k_begin, k_end, (t % nj) * C::TJ, (t / nj) * C::TI,
                                      lds, mout);
    } else {
        // the shorter tiles come last, so that they fill the last round
        const int full = (nj - 1) * ni, b = blockIdx.x;
        if (b < full) {
            const int t = xcd_tile(b, full);
            gram_ring_tile<C, C::SJ, NTS>(bg, aqsn, ngpown, ncouls, k_begin, k_end, (t % (nj - 1)) * C::TJ,
                                          (t / (nj - 1)) * C::TI, lds, mout);
        } else {
            const int t = xcd_tile(b - full, ni);
            gram_ring_tile<C, SJR, NTS>(bg, aqsn, ngpown, ncouls, k_begin, k_end, (nj - 1) * C::TJ, t * C::TI, lds,
                                        mout);
        }
    }
}

// 16 x 16 tiles, three waves each (gram_small_product); same tile order.
__global__ __launch_bounds__(kSmThreads) void k_gram_small(const cplx *__restrict__ bg, const cplx *__restrict__ aqsn,
                                                           int ngpown, int ncouls, int k_begin, int k_end,
                                                           const int32_t *__restrict__ slots,
                                                           cplx *__restrict__ mout, Stamp stamp)
{
    stamp_start(stamp);
    gram_slot(slots, ngpown, ncouls, k_begin, k_end, mout);
    // one array (with a second one the compiler waits for every outstanding
    // load before each fragment read): the stages, then P2 and P3
    __shared__ cplx lds[kSmBuf * kSmStage];
    auto *prod = reinterpret_cast<double(*)[4][kWave]>(lds);
    const int nj = (ngpown + 15) / 16, ni = (ncouls + 15) / 16;
    const int t = xcd_tile(blockIdx.x, nj * ni);
    const int j0 = (t % nj) * 16, i0 = (t / nj) * 16;
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    v4d p;
    if (wave == 0)
        p = gram_small_product<0>(bg, aqsn, ngpown, ncouls, k_begin, k_end, j0, i0, lds);
    else if (wave == 1)
        p = gram_small_product<1>(bg, aqsn, ngpown, ncouls, k_begin, k_end, j0, i0, lds);
    else
        p = gram_small_product<2>(bg, aqsn, ngpown, ncouls, k_begin, k_end, j0, i0, lds);
    __syncthreads();  // every wave is done with the stages
    if (wave > 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) prod[wave - 1][r][lane] = p[r];
    }
    __syncthreads();
    if (wave == 0) {
        const int ig = i0 + lane % 16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = j0 + 4 * r + lane / 16;
            const double p2 = prod[0][r][lane], p3 = prod[1][r][lane];
            if (j < ngpown && ig < ncouls) mout[(size_t)j * ncouls + ig] = cplx{p[r] + p2, (p3 - p[r]) + p2};
        }
    }
}

// Stages 2 and 3 fused (at most three frequencies, none negative,
// acht_n1_loc not requested): the Gram tile of k_gram_f64 in the transposed
// orientation, then the pole terms of its elements summed per column in the
// epilogue (gram_pole_epilogue), so Mu never reaches HBM.  Same tile order as
// k_gram_f64; col_ach/col_asx get one sum per (column, G-vector
// tile, frequency).
template <int F>
__global__ __launch_bounds__(512, 1) void k_gram_pole(PoleTileArgs a)
{
    stamp_start(a.stamp);
    typedef FuseCfg C;
    __shared__ cplx lds[FuseLds<F>::kLds];
    auto *sB = reinterpret_cast<cplx(*)[C::KS][C::TJ]>(lds);
    auto *sA = reinterpret_cast<cplx(*)[C::KS][C::TI]>(lds + 2 * C::KS * C::TJ);
    const int nj = (a.ngpown + C::TJ - 1) / C::TJ;
    const int ni = (a.ncouls + C::TI - 1) / C::TI;
    const int t = xcd_tile(blockIdx.x, nj * ni);
    const int j0 = (t % nj) * C::TJ, itile = t / nj, i0 = itile * C::TI;
    v4d acc1[4][2], acc2[4][2], acc3[4][2];
    gram_f64_acc(a.bg, a.aqsn, a.ngpown, a.ncouls, a.nv, a.nb, j0, i0, sB, sA, acc1, acc2, acc3);
    gram_pole_epilogue<F>(a, j0, i0, itile, acc1, acc2, acc3, lds);
}

// One wave per column: the fused epilogue's tile sums, summed and scaled.
__global__ __launch_bounds__(256) void k_pole_cols(const cplx *col_ach, const cplx *col_asx, int nsplit, int nfreq,
                                                   const int32_t *idx, const double *vcoul, int ncouls, int ngpown,
                                                   double occ, cplx *out_ach, cplx *out_asx, Stamp stamp)
{
    stamp_start(stamp);
    const int j = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (j < ngpown) pole_cols_wave(col_ach, col_asx, nsplit, nfreq, idx, vcoul, ncouls, occ, j, out_ach, out_asx);
}

// Grid (ngpown, nsplit, ceil(nfreq/FC)).  NV: occupied band count fixed at
// compile time (0: any).  Three waves per SIMD: with the wave-uniform pole
// inputs held in scalar registers the FC = 8 kernels fit 168 VGPRs (142-165;
// the p2-storing ones 154-168, of which at most 8 spill).  Two waves are slower
// or no faster (reduce, us, three / two, 40/nv/16384/819 and 8 frequencies: 2
// bands 198 / 204, 8 bands 234 / 237, with p2 6 bands 249 / 284).  Two for FC =
// 16 (its 64 accumulators; 207-239 VGPRs).  Four for the plain kernels of at
// most three frequencies: their waves wait on memory half of the time, and a
// fourth hides more of it despite 8-21 spilled registers at three frequencies
// (40/nv/16384/819, four / three: 1 band 121 / 130, 2 bands 126 / 138, from 3
// bands up within 2%); the p2-storing and negative-frequency ones take up to
// 159 and keep three (the p2 one at four: 0.70 -> 1.28 ms at 512/2/32768/1638).
// The negative-frequency kernels of 8 frequencies per pass run two (their
// cutoff code spilled 84-186 registers at three).
template <int FC, int NV, bool P2, bool NEG = false>
__global__ __launch_bounds__(kRedThreads, (FC <= 3 && !P2 && !NEG) ? 4 : FC > 8 || (NEG && FC > 4) ? 2 : 3) void k_pole_reduce(ReduceArgs a)
{
    int fpb = a.fpb;
    const StampStart stamp(a.stamp, fpb);
    __shared__ __attribute__((aligned(16))) cplx lds[pole_lds_entries<FC, NV>()];
    const int iw_begin = blockIdx.z * fpb;
    const int iw_end = iw_begin + fpb < a.nfreq ? iw_begin + fpb : a.nfreq;
    pole_reduce_item<FC, NV, P2, (FC > 4 ? 4 : FC), NEG>(a, blockIdx.x, blockIdx.y, iw_begin, iw_end, lds);
    stamp.store();
}

__global__ __launch_bounds__(kRedThreads) void k_fact_final(const cplx *col_ach, const cplx *col_asx,
                                                            const cplx *part_achs, long long ncols, int nfreq, int nb,
                                                            int nv, cplx *out, bool nan_acht, Stamp stamp,
                                                            StampEnd end)
{
    stamp_start(stamp);
    __shared__ cplx scratch[kRedThreads / kWave];
    final_block(col_ach, col_asx, part_achs, ncols, nfreq, nb, nv, out, scratch, blockIdx.x, nan_acht);
    stamp_end(end);
}

// 1-D grid over (band tiles, j tiles, G-vector splits), band tiles fastest in
// tile order and spread over the XCDs by xcd_tile, so the blocks that share one
// R tile run on one XCD.  part: [jtiles * nks][nb].  CUT: the last j tile runs
// one sub-tile row per wave.
template <class C, bool CUT>
__global__ __launch_bounds__(C::NT) __attribute__((amdgpu_waves_per_eu(C::OCC))) void k_acht_f64(
    const cplx *__restrict__ p2, const cplx *__restrict__ aqsn, const cplx *__restrict__ bg,
    const int32_t *__restrict__ idx, const double *__restrict__ vcoul, int ngpown, int ncouls, int nb, int n1_begin,
    int n1_end, int chunk, int nks, int jtiles, cplx *__restrict__ part, Stamp stamp)
{
    stamp_start(stamp);
    __shared__ cplx lds[C::LDS];
    const int nn = (n1_end - n1_begin + C::TI - 1) / C::TI;
    // CUT: the last j tile's blocks come after the others, filling the last round
    const int nj = CUT ? jtiles - 1 : jtiles, full = nn * nj * nks, b = blockIdx.x;
    const bool last = CUT && b >= full;
    const int t = last ? xcd_tile(b - full, nn * nks) : xcd_tile(b, full);
    const int ct = t % nn, jt = last ? nj : (t / nn) % nj, ks = last ? t / nn : t / (nn * nj);
    const int k_begin = ks * chunk;
    const int k_end = k_begin + chunk < ncouls ? k_begin + chunk : ncouls;
    cplx *const out = part + ((size_t)jt * nks + ks) * nb;
    if (last)
        acht_ring_tile<C, 1>(p2, aqsn, bg, idx, vcoul, ngpown, ncouls, n1_end, k_begin, k_end, jt * C::TJ,
                             n1_begin + ct * C::TI, lds, out);
    else
        acht_ring_tile<C, C::SJ>(p2, aqsn, bg, idx, vcoul, ngpown, ncouls, n1_end, k_begin, k_end, jt * C::TJ,
                                 n1_begin + ct * C::TI, lds, out);
}

// Grid (ngpown, nsplit): the occupied bands' acht_n1_loc partials (where the
// reduce does not sum them: reduce_sums_acht_occ).
__global__ __launch_bounds__(kRedThreads) void k_acht_occ(const cplx *__restrict__ p2,
                                                          const uint8_t *__restrict__ br1,
                                                          const cplx *__restrict__ aqsn, const cplx *__restrict__ bg,
                                                          const int32_t *__restrict__ idx,
                                                          const double *__restrict__ vcoul, int ngpown, int ncouls,
                                                          int nv, int chunk, int nsplit, cplx *__restrict__ part_occ,
                                                          Stamp stamp)
{
    stamp_start(stamp);
    __shared__ cplx scratch[kRedThreads / kWave];
    acht_occ_item(p2, br1, aqsn, bg, idx, vcoul, ngpown, ncouls, nv, chunk, blockIdx.x, blockIdx.y,
                  part_occ + ((size_t)blockIdx.x * nsplit + blockIdx.y) * nv, scratch);
}

// acht_n1_loc[n1] as the fixed-order sum of its partials.  Blocks
// [0, ceil(nb/16)): 16 bands x 16 contiguous groups of the (j tile, split)
// partials of the product (bands n1 >= nv), groups combined in order.
// Blocks after them: one per occupied band n1 < nv, its (column, split)
// partials of k_acht_occ strided over the 256 threads, then block_sum.
// perm: row n1 is band perm[n1] of out (null: n1).
constexpr int kAchtFinalBands = 16;
__global__ __launch_bounds__(256) void k_acht_final(const cplx *__restrict__ part, int nparts,
                                                    const cplx *__restrict__ part_occ, int nparts_occ, int nb,
                                                    int nv, const int32_t *__restrict__ perm,
                                                    cplx *__restrict__ out, Stamp stamp, StampEnd end)
{
    stamp_start(stamp);  // where no launch of the stage came before
    __shared__ cplx grp[256 / kAchtFinalBands][kAchtFinalBands];
    const int nblk = (nb + kAchtFinalBands - 1) / kAchtFinalBands;
    if ((int)blockIdx.x < nblk) {
        const int n1 = blockIdx.x * kAchtFinalBands + threadIdx.x % kAchtFinalBands;
        const int g = threadIdx.x / kAchtFinalBands;
        constexpr int NG = 256 / kAchtFinalBands;
        cplx s = czero();
        if (n1 >= nv && n1 < nb) {
            const int q0 = (int)((long long)nparts * g / NG), q1 = (int)((long long)nparts * (g + 1) / NG);
            for (int q = q0; q < q1; ++q) s = cadd(s, part[(size_t)q * nb + n1]);
        }
        grp[g][threadIdx.x % kAchtFinalBands] = s;
        __syncthreads();
        if (g == 0 && n1 >= nv && n1 < nb) {
            cplx t = grp[0][threadIdx.x];
            for (int k = 1; k < NG; ++k) t = cadd(t, grp[k][threadIdx.x]);
            out[perm ? perm[n1] : n1] = t;
        }
    } else {
        const int n1 = (int)blockIdx.x - nblk;  // < nv
        cplx s = czero();
        for (int q = threadIdx.x; q < nparts_occ; q += blockDim.x) s = cadd(s, part_occ[(size_t)q * nv + n1]);
        s = block_sum(s, &grp[0][0]);
        if (threadIdx.x == 0) out[perm ? perm[n1] : n1] = s;
    }
    stamp_end(end);
}

template <class C, bool NTS>
void launch_gram_nts(const DevProblem &p, const GramSlots &g, const cplx *bg, cplx *mu, Stamp stamp, hipStream_t s)
{
    const unsigned tiles = (unsigned)((p.ngpown + C::TJ - 1) / C::TJ) * (unsigned)((p.ncouls + C::TI - 1) / C::TI);
    const int rem = p.ngpown % C::TJ;
    if (C::SJ == 2 && rem > 0 && rem <= 16 * C::WJN)
        hipLaunchKernelGGL((k_gram_f64<C, 1, NTS>), dim3(tiles, g.n), dim3(C::NT), 0, s, bg, p.aqsn, p.ngpown,
                           p.ncouls, p.nv, p.nb, g.dev, mu, stamp);
    else
        hipLaunchKernelGGL((k_gram_f64<C, C::SJ, NTS>), dim3(tiles, g.n), dim3(C::NT), 0, s, bg, p.aqsn, p.ngpown,
                           p.ncouls, p.nv, p.nb, g.dev, mu, stamp);
}

template <class C>
void launch_gram_ring(const DevProblem &p, const GramSlots &g, const cplx *bg, cplx *mu, Stamp stamp, hipStream_t s)
{
    if (mu_streams(p, g.n))
        launch_gram_nts<C, true>(p, g, bg, mu, stamp, s);
    else
        launch_gram_nts<C, false>(p, g, bg, mu, stamp, s);
}

template <class C, bool CUT>
void launch_acht(const DevProblem &p, const AchtSplit &as, const cplx *p2, const cplx *bg, cplx *part, Stamp stamp,
                 hipStream_t s)
{
    hipLaunchKernelGGL((k_acht_f64<C, CUT>), dim3((unsigned)as.ntiles * as.jtiles * as.nks), dim3(C::NT), 0, s, p2,
                       p.aqsn, bg, p.idx, p.vcoul, p.ngpown, p.ncouls, p.nb, p.nv, p.nb, as.chunk, as.nks, as.jtiles,
                       part, stamp);
}

// P2: also store the pole factor of frequency acht_iw and either sum the
// occupied bands' acht_n1_loc terms (reduce_sums_acht_occ) or store the
// occupied branch mask.  Problems with a negative frequency run the generic
// NEG kernel.
template <int FC, bool P2>
void launch_reduce_p2(const ReduceArgs &a, dim3 grid, hipStream_t s)
{
    if (a.neg) {  // at most 8 per pass (the 16-wide variant spills)
        hipLaunchKernelGGL((k_pole_reduce<(FC > 8 ? 8 : FC), 0, P2, true>), grid, dim3(kRedThreads), 0, s, a);
        return;
    }
    // Up to eight occupied bands a kernel for each count (their loads issued
    // together, conj(bg) in scalar registers), beyond it the general one.
    // Reduce, us, general / own: 300/nv/16384/819, nv = 3 and 3 frequencies 184
    // / 137, 7 and 3 233 / 177, 1 and 8 229 / 187, 5 and 13 562 / 376, 6 and 24
    // 917 / 604; with p2 40/nv/16384/819, 1 and 8 267 / 220, 3 and 4 256 / 200,
    // 5 and 16 666 / 489, 7 and 8 458 / 254; the p2-storing one of one band and
    // at most 3 frequencies the other way, 186 / 194.
    switch (a.nv) {
    case 1: hipLaunchKernelGGL((k_pole_reduce<FC, (P2 && FC <= 3) ? 0 : 1, P2>), grid, dim3(kRedThreads), 0, s, a); break;
    case 2: hipLaunchKernelGGL((k_pole_reduce<FC, 2, P2>), grid, dim3(kRedThreads), 0, s, a); break;
    case 3: hipLaunchKernelGGL((k_pole_reduce<FC, 3, P2>), grid, dim3(kRedThreads), 0, s, a); break;
    case 4: hipLaunchKernelGGL((k_pole_reduce<FC, 4, P2>), grid, dim3(kRedThreads), 0, s, a); break;
    case 5: hipLaunchKernelGGL((k_pole_reduce<FC, 5, P2>), grid, dim3(kRedThreads), 0, s, a); break;
    case 6: hipLaunchKernelGGL((k_pole_reduce<FC, 6, P2>), grid, dim3(kRedThreads), 0, s, a); break;
    case 7: hipLaunchKernelGGL((k_pole_reduce<FC, 7, P2>), grid, dim3(kRedThreads), 0, s, a); break;
    case 8: hipLaunchKernelGGL((k_pole_reduce<FC, 8, P2>), grid, dim3(kRedThreads), 0, s, a); break;
    default: hipLaunchKernelGGL((k_pole_reduce<FC, 0, P2>), grid, dim3(kRedThreads), 0, s, a); break;
    }
}

template <int FC>
void launch_reduce_fc(ReduceArgs a, hipStream_t s)
{
    if (a.fpb < FC) a.fpb = FC;
    dim3 grid(a.ngpown, a.nsplit, (a.nfreq + a.fpb - 1) / a.fpb);
    if (a.p2)
        launch_reduce_p2<FC, true>(a, grid, s);
    else
        launch_reduce_p2<FC, false>(a, grid, s);
}

template <int F>
void launch_gram_pole_f(const DevProblem &p, const PoleTileArgs &a, hipStream_t s)
{
    const unsigned tiles =
        (unsigned)((p.ngpown + FuseCfg::TJ - 1) / FuseCfg::TJ) * (unsigned)((p.ncouls + FuseCfg::TI - 1) / FuseCfg::TI);
    hipLaunchKernelGGL((k_gram_pole<F>), dim3(tiles), dim3(FuseCfg::NT), 0, s, a);
}

#define GPP_TRY(x)                       \
    do {                                 \
        hipError_t e_ = (x);             \
        if (e_ != hipSuccess) return e_; \
    } while (0)

}  // namespace

size_t factored_workspace_bytes(const DevProblem &p, GramKind kind)
{
    size_t n = fact_layout(p, kind).total;
    if (kind.ozaki_slices) n += ozaki_workspace_bytes(p, kind.ozaki_slices, kind.int8);
    return n;
}

// The Gram tile of a problem by size (GPP_OPT_GRAM_TILE 0): the least
// estimated time, the sub-tiles a CU works through (its rounds of whole tiles;
// the shorter last-row tiles fill the last round as far as they fit) times the
// time per 16 x 16 sub-tile and k-step of 4 bands.  A CU with one block runs
// its MFMAs with fewer waves beside them than one with two.  The times are
// fitted to 17 shapes from 24/2/1000/50 to 1536/8/32768/1638 (us measured /
// estimated: 512/2/4096/409 64 x 64 102 / 101, 128 x 64 111 / 106, 32 x 64
// 114 / 115, 16 x 16 154 / 170; 512/2/32768/205 64 x 128 347 / 340, 64 x 64
// 358 / 354; 512/2/800/40 16 x 16 9.6 / 9.7, 32 x 64 35 / 38).  Larger tiles
// re-read less and turn stages over less often; smaller ones leave fewer CUs
// idle, and the 16 x 16 tile has the shortest chain of MFMAs per wave.
// Several products in one launch count with their mean number of bands.
namespace {
enum GramTile { kTileL = 0, kTileLt, kTileM, kTileS, kTileX };
int gram_tile_for(const DevProblem &p, const GramSlots &g)
{
    struct Kind {
        int tile, tj, ti, short_j;  // short_j: rows of a short last tile (0: none)
        double one, many;           // us per sub-tile and k-step: one block per CU, more
    };
    static const Kind kinds[] = {{kTileLt, GramLt::TJ, GramLt::TI, GramLt::TJ / 2, 0.0258, 0.0235},
                                 {kTileL, GramL::TJ, GramL::TI, GramL::TJ / 2, 0.0258, 0.0237},
                                 {kTileM, GramM::TJ, GramM::TI, GramM::TJ / 2, 0.0287, 0.0247},
                                 {kTileS, GramS::TJ, GramS::TI, 0, 0.0344, 0.0273},
                                 {kTileX, 16, 16, 0, 0.0547, 0.0469}};
    const double ksteps = g.dev ? std::max(1.0, (double)g.bands / (4 * g.n)) : (p.nb - p.nv + 3) / 4;
    double best = 1e300;
    int tile = kTileL;
    for (const Kind &k : kinds) {
        const int rem = p.ngpown % k.tj;
        const bool cut = rem > 0 && rem <= k.short_j;
        const double ni = (p.ncouls + k.ti - 1) / k.ti, sub = k.tj / 16 * (k.ti / 16);
        const double whole = g.n * ni * ((p.ngpown + k.tj - 1) / k.tj - (cut ? 1 : 0));
        const double rounds = tile_rounds(whole, cut ? g.n * ni : 0);
        double us = rounds * sub * ksteps * (rounds <= 1 ? k.one : k.many);
        if (k.tile == kTileX) us += 1.2 * ceil(rounds / 2);  // the first loads of its ring, two blocks at a time
        if (us < best) best = us, tile = k.tile;
    }
    return tile;
}

hipError_t launch_gram_f64(const DevProblem &p, const GramSlots &g, int tile, const cplx *bg, cplx *mu, Stamp stamp,
                           hipStream_t s)
{
    // GPP_OPT_GRAM_TILE: 0 by size, then the ring tiles
    static const int kinds[kGramTiles] = {-1, kTileL, kTileLt, kTileM};
    if (tile < 0 || tile >= kGramTiles) return hipErrorInvalidValue;
    switch (tile == 0 ? gram_tile_for(p, g) : kinds[tile]) {
    case kTileL: launch_gram_ring<GramL>(p, g, bg, mu, stamp, s); break;
    case kTileLt: launch_gram_ring<GramLt>(p, g, bg, mu, stamp, s); break;
    case kTileM: launch_gram_ring<GramM>(p, g, bg, mu, stamp, s); break;
    case kTileS: launch_gram_ring<GramS>(p, g, bg, mu, stamp, s); break;
    default: {
        const unsigned tiles = (unsigned)((p.ngpown + 15) / 16) * (unsigned)((p.ncouls + 15) / 16);
        hipLaunchKernelGGL(k_gram_small, dim3(tiles, g.n), dim3(kSmThreads), 0, s, bg, p.aqsn, p.ngpown, p.ncouls,
                           p.nv, p.nb, g.dev, mu, stamp);
        break;
    }
    }
    return hipGetLastError();
}

// red_fc 0: passes of 16 from 16 frequencies up, none negative (C3, 16
// frequencies: one pass, 7.19 -> 6.74 ms against two of 8), else 8.  With a
// negative frequency at most 8 (that kernel spills at 16).
hipError_t launch_pole_reduce(const ReduceArgs &ra, int red_fc, hipStream_t s)
{
    int fc = red_fc == 4 || red_fc == 8 || red_fc == 16 ? red_fc : ra.nfreq >= 16 && !ra.neg ? 16 : 8;
    if (ra.neg && fc > 8) fc = 8;
    switch (ra.nfreq < 4 ? ra.nfreq : fc) {
    case 1: launch_reduce_fc<1>(ra, s); break;
    case 2: launch_reduce_fc<2>(ra, s); break;
    case 3: launch_reduce_fc<3>(ra, s); break;
    case 4: launch_reduce_fc<4>(ra, s); break;
    case 16: launch_reduce_fc<16>(ra, s); break;
    default: launch_reduce_fc<8>(ra, s); break;
    }
    return hipGetLastError();
}

// Where stage 3 puts what acht_n1_loc needs, and the later stages' partials.
struct AchtBufs {
    cplx *p2 = nullptr;  // null: acht_n1_loc is not requested
    uint8_t *br1 = nullptr;
    cplx *part = nullptr, *part_occ = nullptr;
};

// Stage 3 of one problem; its partials to col_ach/col_asx [ngpown][nsplit][nfreq].
hipError_t run_pole_reduce(const DevProblem &p, const GramKind &kind, const cplx *mu, const cplx *bg, cplx *col_ach,
                           cplx *col_asx, int nsplit, const AchtBufs &ab, Stamp stamp, hipStream_t s)
{
    ReduceArgs ra;
    ra.mu = mu; ra.ieps = p.ieps; ra.wtilde = p.wtilde; ra.aqsn = p.aqsn; ra.bg = bg; ra.idx = p.idx;
    ra.vcoul = p.vcoul; ra.wx = p.wx; ra.nv = p.nv; ra.ncouls = p.ncouls; ra.ngpown = p.ngpown;
    ra.nfreq = p.nfreq; ra.occ = p.occ; ra.col_ach = col_ach; ra.col_asx = col_asx;
    ra.nsplit = nsplit; ra.chunk = kind.red_chunk;
    ra.fpb = kind.red_fpb > 0 ? kind.red_fpb : p.nfreq;
    ra.p2 = ab.p2;
    const bool occ_in_reduce = ab.p2 && p.nv > 0 && reduce_sums_acht_occ(p.nv, p.wx_neg);
    ra.br1 = ab.p2 && p.nv > 0 && !occ_in_reduce ? ab.br1 : nullptr;
    ra.part_occ = occ_in_reduce ? ab.part_occ : nullptr;
    ra.acht_iw = acht_frequency(p);
    ra.neg = p.wx_neg;
    ra.stamp = stamp;
    return launch_pole_reduce(ra, kind.red_fc, s);
}

// Stages 2 and 3 fused; column sums to col_ach/col_asx [ngpown][nfreq].
// tile_ach/tile_asx: [ngpown][nsplit][nfreq].
hipError_t run_gram_pole(const DevProblem &p, const cplx *bg, cplx *tile_ach, cplx *tile_asx, int nsplit,
                         cplx *col_ach, cplx *col_asx, Stamp stamp, StageTimer *timer, hipStream_t s)
{
    PoleTileArgs pa;
    pa.aqsn = p.aqsn; pa.ieps = p.ieps; pa.wtilde = p.wtilde; pa.bg = bg; pa.wx = p.wx;
    pa.nb = p.nb; pa.nv = p.nv; pa.ncouls = p.ncouls; pa.ngpown = p.ngpown; pa.nsplit = nsplit;
    pa.col_ach = tile_ach; pa.col_asx = tile_asx;
    pa.stamp = stamp;
    switch (p.nfreq) {
    case 1: launch_gram_pole_f<1>(p, pa, s); break;
    case 2: launch_gram_pole_f<2>(p, pa, s); break;
    default: launch_gram_pole_f<3>(p, pa, s); break;
    }
    GPP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_pole_cols, dim3((p.ngpown + 3) / 4), dim3(256), 0, s, tile_ach, tile_asx, nsplit, p.nfreq,
                       p.idx, p.vcoul, p.ncouls, p.ngpown, p.occ, col_ach, col_asx,
                       timer ? timer->stage("factored_pole_cols") : Stamp{});
    return hipGetLastError();
}

unsigned acht_final_blocks(const DevProblem &p)
{
    return (p.nb + kAchtFinalBands - 1) / kAchtFinalBands + p.nv;
}

// Stages 5 and 6: acht_n1_loc of the problem's bands, row n1 to
// out[perm ? perm[n1] : n1].  st: for the first launch.
hipError_t run_acht(const DevProblem &p, const AchtSplit &as, int occ_chunk, int occ_nsplit, const AchtBufs &ab,
                    const cplx *bg, const int32_t *perm, cplx *out, Stamp st, StampEnd end, hipStream_t s)
{
    if (p.nb > p.nv) {
        if (as.narrow)
            as.cut ? launch_acht<GramM, true>(p, as, ab.p2, bg, ab.part, st, s)
                   : launch_acht<GramM, false>(p, as, ab.p2, bg, ab.part, st, s);
        else
            as.cut ? launch_acht<GramL, true>(p, as, ab.p2, bg, ab.part, st, s)
                   : launch_acht<GramL, false>(p, as, ab.p2, bg, ab.part, st, s);
        GPP_TRY(hipGetLastError());
        st = Stamp{};
    }
    if (p.nv > 0 && !reduce_sums_acht_occ(p.nv, p.wx_neg)) {  // else summed by the reduce
        hipLaunchKernelGGL(k_acht_occ, dim3(p.ngpown, occ_nsplit), dim3(kRedThreads), 0, s, ab.p2, ab.br1, p.aqsn,
                           bg, p.idx, p.vcoul, p.ngpown, p.ncouls, p.nv, occ_chunk, occ_nsplit, ab.part_occ, st);
        GPP_TRY(hipGetLastError());
        st = Stamp{};
    }
    hipLaunchKernelGGL(k_acht_final, dim3(acht_final_blocks(p)), dim3(256), 0, s,
                       ab.part, as.jtiles * as.nks, ab.part_occ, p.ngpown * occ_nsplit, p.nb, p.nv, perm, out, st, end);
    return hipGetLastError();
}

}  // namespace

hipError_t run_factored(const DevProblem &p, GramKind kind, void *work, const DevResults &res, hipStream_t s,
                        StageTimer *timer)
{
    if (p.wx_stride != 0) return hipErrorInvalidValue;  // the band sum factors only for a shared wx row
    const FactLayout L = fact_layout(p, kind);
    char *w = static_cast<char *>(work);
    cplx *bg = reinterpret_cast<cplx *>(w + L.bg);
    cplx *mu = reinterpret_cast<cplx *>(w + L.m);
    cplx *col_ach = reinterpret_cast<cplx *>(w + L.col_ach);
    cplx *col_asx = reinterpret_cast<cplx *>(w + L.col_asx);
    cplx *part_achs = reinterpret_cast<cplx *>(w + L.part_achs);

    const auto stage = [&](const char *nm) { return timer ? timer->stage(nm) : Stamp{}; };
    const auto end = [&](unsigned blocks) { return timer ? timer->end(blocks) : StampEnd{}; };
    if (timer) timer->begin();
    // also gathers Bg
    GPP_TRY(launch_achstemp(p, part_achs, bg, stage("factored_gather_achstemp"), s));
    if (L.fused) {
        cplx *c2a = reinterpret_cast<cplx *>(w + L.col2_ach);
        cplx *c2x = reinterpret_cast<cplx *>(w + L.col2_asx);
        GPP_TRY(run_gram_pole(p, bg, col_ach, col_asx, L.nsplit, c2a, c2x, stage("factored_gram_pole"), timer, s));
        const Stamp st = stage("factored_final");
        hipLaunchKernelGGL(k_fact_final, dim3(p.nfreq + 1), dim3(kRedThreads), 0, s, c2a, c2x, part_achs, p.ngpown,
                           p.nfreq, p.nb, p.nv, res.base, true, st, end(p.nfreq + 1));
        return hipGetLastError();
    }
    if (kind.ozaki_slices) {
        GPP_TRY(launch_gram_ozaki(p, kind.ozaki_slices, kind.int8, kind.layout, kind.group, bg, w + L.total, mu,
                                  stage(kind.int8 ? "factored_gram_ozaki_i8" : "factored_gram_ozaki"), s));
    } else {
        GPP_TRY(launch_gram_f64(p, GramSlots{}, kind.tile, bg, mu, stage("factored_gram_f64"), s));
    }
    AchtBufs ab;
    if (kind.acht) {
        ab.p2 = reinterpret_cast<cplx *>(w + L.p2);
        ab.br1 = reinterpret_cast<uint8_t *>(w + L.br1);
        ab.part = reinterpret_cast<cplx *>(w + L.acht_part);
        ab.part_occ = reinterpret_cast<cplx *>(w + L.acht_occ);
    }
    GPP_TRY(run_pole_reduce(p, kind, mu, bg, col_ach, col_asx, L.nsplit, ab, stage("factored_pole_reduce"), s));
    const Stamp st_final = stage("factored_final");
    hipLaunchKernelGGL(k_fact_final, dim3(p.nfreq + 1), dim3(kRedThreads), 0, s, col_ach, col_asx, part_achs,
                       p.ngpown * L.nsplit, p.nfreq, p.nb, p.nv, res.base, true, st_final,
                       kind.acht ? StampEnd{} : end(p.nfreq + 1));
    GPP_TRY(hipGetLastError());
    if (!kind.acht) return hipSuccess;
    const Stamp st = stage("factored_acht");
    return run_acht(p, L.as, L.occ_chunk, L.occ_nsplit, ab, bg, nullptr, res.acht_n1_loc(), st,
                    end(acht_final_blocks(p)), s);
}

// ---------------------------------------------------------------------------
// Band-dependent frequencies.  The band sum factors over any set of bands
// that share one wx row, so bands are grouped by identical rows ("buckets"),
// each a factored sub-problem of its own Mu and row.  Bg and aqsn are laid out
// with each bucket's bands contiguous, occupied ones first (as they are where
// the bands already lie so).  One launch forms every bucket's Mu, one more
// pass adds up the pole terms of all buckets without occupied bands
// (pole_reduce_bare); a bucket with occupied bands runs the reduce of the
// plain form.  The Mu of GramKind::bucket_mu bytes of buckets are held at a time.
// 512/8/8192/409/3 in 8 buckets: 704 us with a factored evaluation per
// bucket and both arrays permuted, 368 so (Gram 215 of them, with 429 MB of Mu
// to store; the reduces 56 and 84, the latter at 5.7 TB/s).

namespace {

__global__ void k_permute_rows(const cplx *__restrict__ src, const int32_t *__restrict__ perm, int nrows,
                               int ncols, cplx *__restrict__ dst)
{
    const size_t n = (size_t)nrows * ncols;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
        const size_t r = t / ncols, c = t % ncols;
        dst[t] = src[(size_t)perm[r] * ncols + c];
    }
}

template <int F> __global__ __launch_bounds__(kRedThreads, 4) void k_reduce_bare(BareArgs a)
{
    __shared__ cplx scratch[kRedThreads / kWave];
    pole_reduce_bare<F>(a, scratch);
}

// P = delw I_eps of one frequency (the p2 of the reduce), for the buckets
// whose reduce does not write it.
__global__ __launch_bounds__(256) void k_pole_p2(const cplx *__restrict__ wtilde, const cplx *__restrict__ ieps,
                                                 const double *__restrict__ wx, size_t n, cplx *__restrict__ p2)
{
    const double w = *wx;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
        const cplx wt = wtilde[t], q = cmul_fast(wt, ieps[t]);
        const double wdr = w - wt.re, rden = rcp_1nr(__builtin_fma(wdr, wdr, wt.im * wt.im));
        __builtin_nontemporal_store(__builtin_fma(q.re, wdr, -(q.im * wt.im)) * rden, &p2[t].re);
        __builtin_nontemporal_store(__builtin_fma(q.im, wdr, q.re * wt.im) * rden, &p2[t].im);
    }
}

// Frequencies per block of k_reduce_bare: equal passes of at most 8.
int bare_width(int nfreq)
{
    const int passes = (nfreq + 7) / 8, f = (nfreq + passes - 1) / passes;
    return f <= 4 ? f : f <= 6 ? 6 : 8;
}

void launch_reduce_bare(const BareArgs &a, hipStream_t s)
{
    const int f = bare_width(a.nfreq);
    const dim3 grid(a.ngpown, a.nsplit, (a.nfreq + f - 1) / f);
    switch (f) {
    case 1: hipLaunchKernelGGL(k_reduce_bare<1>, grid, dim3(kRedThreads), 0, s, a); break;
    case 2: hipLaunchKernelGGL(k_reduce_bare<2>, grid, dim3(kRedThreads), 0, s, a); break;
    case 3: hipLaunchKernelGGL(k_reduce_bare<3>, grid, dim3(kRedThreads), 0, s, a); break;
    case 4: hipLaunchKernelGGL(k_reduce_bare<4>, grid, dim3(kRedThreads), 0, s, a); break;
    case 6: hipLaunchKernelGGL(k_reduce_bare<6>, grid, dim3(kRedThreads), 0, s, a); break;
    default: hipLaunchKernelGGL(k_reduce_bare<8>, grid, dim3(kRedThreads), 0, s, a); break;
    }
}

// How a slot's stage 3 runs: fused with its Gram product, with the plain
// form's reduce, or together with the other buckets without occupied bands.
// With GPP_OPT_FUSED_REDUCE no bucket runs together with others.
enum SlotKind { kSlotFused, kSlotPlain, kSlotBare };

struct BucketLayout {
    size_t aqsn, bg, mu, part_achs, col_ach, col_asx, tile_ach, tile_asx, p2, br1, acht_part, acht_occ, sub, total;
    int group;   // buckets whose Mu are held at a time
    int nsplit;  // G-vector ranges of a plain reduce
    int bare_chunk, bare_nsplit;
    long long ncols;  // column partials of all buckets
};

// Bucket b over its rows of the permuted aqsn.
DevProblem bucket_problem(const DevProblem &p, const BucketPlan &bp, int b, const cplx *aqsn_p)
{
    DevProblem q = p;
    q.nb = bp.size[b];
    q.nv = bp.nocc[b];
    q.aqsm = nullptr;  // Bg is gathered for all buckets
    q.aqsn = aqsn_p + (size_t)bp.start[b] * p.ncouls;
    q.wx = p.wx + (size_t)bp.row[b] * p.nfreq;
    q.wx_stride = 0;
    q.wx_neg = bp.neg[b];
    return q;
}

SlotKind slot_kind(const DevProblem &q, const GramKind &k)
{
    if (fused_reduce(q, k)) return kSlotFused;
    return q.nv > 0 || k.fuse ? kSlotPlain : kSlotBare;
}

BucketLayout bucket_layout(const DevProblem &p, const GramKind &k, const BucketPlan &bp)
{
    BucketLayout L;
    const int nbk = (int)bp.slot.size();
    const size_t mu_bytes = sizeof(cplx) * (size_t)p.ngpown * p.ncouls;
    // with the fused reduce the buckets run one after the other
    L.group = k.fuse ? 1 : (int)std::max<size_t>(1, std::min<size_t>(std::min(nbk, 4096), k.bucket_mu / mu_bytes));
    L.nsplit = (p.ncouls + k.red_chunk - 1) / k.red_chunk;
    // G ranges of the reduce over the bare buckets: whole steps of a block,
    // about 2048 blocks
    const int steps = (p.ncouls + kBareStep - 1) / kBareStep;
    const int want = std::max(1, std::min(steps, 2048 / p.ngpown));
    L.bare_chunk = (steps + want - 1) / want * kBareStep;
    L.bare_nsplit = (p.ncouls + L.bare_chunk - 1) / L.bare_chunk;
    bool mu = false, fused = false;
    L.ncols = 0;
    size_t br1 = 0, part = 0, occ = 0, sub = 0;
    for (int s0 = 0; s0 < nbk; s0 += L.group) {
        bool bare = false;
        for (int sl = s0; sl < std::min(nbk, s0 + L.group); ++sl) {
            const DevProblem q = bucket_problem(p, bp, bp.slot[sl], nullptr);
            const SlotKind kind = slot_kind(q, k);
            (kind == kSlotFused ? fused : mu) = true;
            if (kind == kSlotBare) bare = true;
            else L.ncols += (long long)p.ngpown * (kind == kSlotFused ? 1 : L.nsplit);
            if (k.ozaki_slices) sub = std::max(sub, ozaki_workspace_bytes(q, k.ozaki_slices, k.int8));
            if (!k.acht) continue;
            const AchtSplit as = acht_split(q);
            part = std::max(part, sizeof(cplx) * (size_t)as.jtiles * as.nks * q.nb);
            if (q.nv == 0) continue;
            const bool in_reduce = reduce_sums_acht_occ(q.nv, q.wx_neg);
            const int chunk = acht_occ_chunk(q, k.red_chunk);
            const int nsplit = in_reduce ? L.nsplit : (p.ncouls + chunk - 1) / chunk;
            if (!in_reduce) br1 = (size_t)p.ngpown * p.ncouls;
            occ = std::max(occ, sizeof(cplx) * (size_t)p.ngpown * nsplit * q.nv);
        }
        if (bare) L.ncols += (long long)p.ngpown * L.bare_nsplit;
    }
    size_t off = 0;
    const auto take = [&off](size_t bytes) {
        const size_t at = off;
        off += align256(bytes);
        return at;
    };
    const size_t tiles = fused ? sizeof(cplx) * (size_t)p.ngpown * ((p.ncouls + FuseCfg::TI - 1) / FuseCfg::TI) * p.nfreq : 0;
    L.aqsn = take(bp.identity ? 0 : sizeof(cplx) * (size_t)p.nb * p.ncouls);
    L.bg = take(sizeof(cplx) * (size_t)p.nb * p.ngpown);
    L.mu = take(mu ? mu_bytes * L.group : 0);
    L.part_achs = take(sizeof(cplx) * ach_region_entries(p.nb, p.ngpown));
    L.col_ach = take(sizeof(cplx) * (size_t)L.ncols * p.nfreq);
    L.col_asx = take(sizeof(cplx) * (size_t)L.ncols * p.nfreq);
    L.tile_ach = take(tiles);
    L.tile_asx = take(tiles);
    L.p2 = take(k.acht ? mu_bytes : 0);
    L.br1 = take(br1);
    L.acht_part = take(part);
    L.acht_occ = take(occ);
    L.sub = off;
    L.total = off + sub;
    return L;
}

}  // namespace

BucketPlan plan_buckets(const double *wx_rows, int nb, int nv, int nfreq)
{
    BucketPlan bp;
    std::vector<int> bucket(nb, -1);
    for (int n1 = 0; n1 < nb; ++n1) {
        const double *r = wx_rows + (size_t)n1 * nfreq;
        for (int b = 0; b < (int)bp.row.size(); ++b)
            if (memcmp(r, wx_rows + (size_t)bp.row[b] * nfreq, sizeof(double) * nfreq) == 0) {
                bucket[n1] = b;
                break;
            }
        if (bucket[n1] < 0) {
            bucket[n1] = (int)bp.row.size();
            bp.row.push_back(n1);
            bp.neg.push_back(wx_has_negative(r, nfreq));
        }
    }
    const int nbk = (int)bp.row.size();
    bp.start.assign(nbk, 0);
    bp.size.assign(nbk, 0);
    bp.nocc.assign(nbk, 0);
    for (int b = 0; b < nbk; ++b) {
        bp.start[b] = (int)bp.perm.size();
        for (int pass = 0; pass < 2; ++pass)  // occupied bands first, each in band order
            for (int n1 = 0; n1 < nb; ++n1)
                if (bucket[n1] == b && (n1 < nv) == (pass == 0)) {
                    bp.perm.push_back(n1);
                    ++bp.size[b];
                    if (pass == 0) ++bp.nocc[b];
                }
        bp.slot.push_back(b);
    }
    std::stable_sort(bp.slot.begin(), bp.slot.end(), [&](int x, int y) {
        if ((bp.nocc[x] > 0) != (bp.nocc[y] > 0)) return bp.nocc[x] > 0;
        return bp.size[x] - bp.nocc[x] > bp.size[y] - bp.nocc[y];
    });
    bp.identity = true;
    for (int n1 = 0; n1 < nb; ++n1) bp.identity = bp.identity && bp.perm[n1] == n1;
    return bp;
}

std::vector<int32_t> BucketPlan::tables() const
{
    std::vector<int32_t> t = perm;
    for (int b : slot) {
        t.push_back(start[b] + nocc[b]);
        t.push_back(start[b] + size[b]);
        t.push_back(row[b]);
    }
    return t;
}

size_t bucketed_workspace_bytes(const DevProblem &p, GramKind kind, const BucketPlan &bp)
{
    return bucket_layout(p, kind, bp).total;
}

hipError_t run_factored_bucketed(const DevProblem &p, GramKind kind, const BucketPlan &bp, void *work,
                                 const DevResults &res, hipStream_t s, StageTimer *timer)
{
    if (p.wx_stride != p.nfreq || (int)bp.perm.size() != p.nb || !bp.dev) return hipErrorInvalidValue;
    const BucketLayout L = bucket_layout(p, kind, bp);
    char *w = static_cast<char *>(work);
    const auto at = [w](size_t off) { return reinterpret_cast<cplx *>(w + off); };
    cplx *const bg = at(L.bg), *const mu = at(L.mu), *const part_achs = at(L.part_achs);
    AchtBufs ab;
    if (kind.acht) {
        ab.p2 = at(L.p2);
        ab.br1 = reinterpret_cast<uint8_t *>(w + L.br1);
        ab.part = at(L.acht_part);
        ab.part_occ = at(L.acht_occ);
    }
    const int nbk = (int)bp.slot.size();
    const int32_t *const perm = bp.identity ? nullptr : bp.dev_perm();
    const auto stage = [&](const char *nm) { return timer ? timer->stage(nm) : Stamp{}; };
    if (timer) timer->begin();
    GPP_TRY(launch_achstemp(p, part_achs, bg, stage("bucket_permute"), s, perm));  // also gathers Bg
    const cplx *aqsn_p = p.aqsn;
    if (!bp.identity) {
        const size_t blocks = std::min<size_t>(8192, ((size_t)p.nb * p.ncouls + 255) / 256);
        hipLaunchKernelGGL(k_permute_rows, dim3((unsigned)blocks), dim3(256), 0, s, p.aqsn, perm, p.nb, p.ncouls,
                           at(L.aqsn));
        GPP_TRY(hipGetLastError());
        aqsn_p = at(L.aqsn);
    }
    DevProblem all = p;
    all.aqsn = aqsn_p;
    Stamp st = stage("bucket_factored");  // for the first launch of the stage
    const auto first = [&st]() {
        const Stamp f = st;
        st = Stamp{};
        return f;
    };
    size_t col = 0;  // next free column partial
    for (int s0 = 0; s0 < nbk; s0 += L.group) {
        const int s1 = std::min(nbk, s0 + L.group);
        GramSlots g;
        g.dev = bp.dev_slots() + 3 * s0;
        g.n = s1 - s0;
        int bare0 = s1;  // first slot of the group's bare buckets (they come last)
        for (int sl = s1; sl-- > s0;) {
            const DevProblem q = bucket_problem(p, bp, bp.slot[sl], aqsn_p);
            if (slot_kind(q, kind) == kSlotBare) bare0 = sl;
            g.bands += q.nb - q.nv;
        }
        const bool together = !kind.ozaki_slices && !kind.fuse;
        if (together) GPP_TRY(launch_gram_f64(all, g, kind.tile, bg, mu, first(), s));
        for (int sl = s0; sl < s1; ++sl) {
            const int b = bp.slot[sl];
            const DevProblem q = bucket_problem(p, bp, b, aqsn_p);
            const cplx *const bgq = bg + (size_t)bp.start[b] * p.ngpown;
            cplx *const muq = mu + (size_t)(sl - s0) * p.ngpown * p.ncouls;
            cplx *const ca = at(L.col_ach) + col * p.nfreq, *const cx = at(L.col_asx) + col * p.nfreq;
            const SlotKind k = slot_kind(q, kind);
            if (k == kSlotFused) {
                GPP_TRY(run_gram_pole(q, bgq, at(L.tile_ach), at(L.tile_asx), (p.ncouls + FuseCfg::TI - 1) / FuseCfg::TI,
                                      ca, cx, first(), nullptr, s));
                col += p.ngpown;
                continue;
            }
            if (kind.ozaki_slices)
                GPP_TRY(launch_gram_ozaki(q, kind.ozaki_slices, kind.int8, kind.layout, kind.group, bgq, w + L.sub, muq,
                                          first(), s));
            else if (!together)
                GPP_TRY(launch_gram_f64(all, GramSlots{bp.dev_slots() + 3 * sl, 1, q.nb - q.nv}, kind.tile, bg, muq,
                                        first(), s));
            if (k == kSlotPlain) {
                GPP_TRY(run_pole_reduce(q, kind, muq, bgq, ca, cx, L.nsplit, ab, Stamp{}, s));
                col += (size_t)p.ngpown * L.nsplit;
            } else if (kind.acht) {
                hipLaunchKernelGGL(k_pole_p2, dim3(2048), dim3(256), 0, s, q.wtilde, q.ieps, q.wx + acht_frequency(q),
                                   (size_t)p.ngpown * p.ncouls, ab.p2);
                GPP_TRY(hipGetLastError());
            }
            if (kind.acht) {
                const int chunk = acht_occ_chunk(q, kind.red_chunk);
                const int nsplit = reduce_sums_acht_occ(q.nv, q.wx_neg) ? L.nsplit : (p.ncouls + chunk - 1) / chunk;
                GPP_TRY(run_acht(q, acht_split(q), chunk, nsplit, ab, bgq, bp.dev_perm() + bp.start[b],
                                 res.acht_n1_loc(), Stamp{}, StampEnd{}, s));
            }
        }
        if (bare0 < s1) {
            BareArgs a;
            a.mu = mu + (size_t)(bare0 - s0) * p.ngpown * p.ncouls;
            a.slots = bp.dev_slots() + 3 * bare0;
            a.nslots = s1 - bare0;
            a.ieps = p.ieps; a.wtilde = p.wtilde; a.idx = p.idx; a.vcoul = p.vcoul; a.wx = p.wx;
            a.ncouls = p.ncouls; a.ngpown = p.ngpown; a.nfreq = p.nfreq;
            a.nsplit = L.bare_nsplit; a.chunk = L.bare_chunk;
            a.col_ach = at(L.col_ach) + col * p.nfreq;
            a.col_asx = at(L.col_asx) + col * p.nfreq;
            launch_reduce_bare(a, s);
            GPP_TRY(hipGetLastError());
            col += (size_t)p.ngpown * L.bare_nsplit;
        }
    }
    st = stage("bucket_combine");
    hipLaunchKernelGGL(k_fact_final, dim3(p.nfreq + 1), dim3(kRedThreads), 0, s, at(L.col_ach), at(L.col_asx),
                       part_achs, L.ncols, p.nfreq, p.nb, p.nv, res.base, !kind.acht, st,
                       timer ? timer->end(p.nfreq + 1) : StampEnd{});
    return hipGetLastError();
}

}  // namespace gpp

// Not part of the interface: which kernels the size rules pick, for the tests
// that run those kernels at their edges.
extern "C" {

static gpp::DevProblem sizes_only(int nb, int nv, int ncouls, int ngpown)
{
    gpp::DevProblem p;
    p.nb = nb; p.nv = nv; p.ncouls = ncouls; p.ngpown = ngpown; p.nfreq = 3;
    return p;
}

// The FP64 Gram tile of GPP_OPT_GRAM_TILE 0 for one product, or for `groups` of
// them over `bands` unoccupied bands in all: 1000 x G' columns + G-vectors.
int gpp_test_gram_tile(int nb, int nv, int ncouls, int ngpown, int groups, int bands)
{
    static const int tiles[] = {64128, 128064, 64064, 32064, 16016};  // of GramTile
    static const int32_t some = 0;
    gpp::GramSlots g;
    if (groups > 0) g = gpp::GramSlots{&some, groups, bands};
    return tiles[gpp::gram_tile_for(sizes_only(nb, nv, ncouls, ngpown), g)];
}

// The acht_n1_loc product: its tile likewise, 1000000 more with a short last one.
int gpp_test_acht_tile(int nb, int nv, int ncouls, int ngpown)
{
    const gpp::AchtSplit as = gpp::acht_split(sizes_only(nb, nv, ncouls, ngpown));
    return (as.cut ? 1000000 : 0) + (as.narrow ? 64064 : 64128);
}

}
