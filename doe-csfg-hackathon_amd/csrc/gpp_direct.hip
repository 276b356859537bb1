// gpp_direct.hip -- direct FP64 form of the GPP sigma band loop on gfx950.
//
// Reference: gppComplex.cpp:335-383 (band loop), :131-150 (noflagOCC_solver,
// unoccupied bands), :107-128 + :16-63 (flagOCC_solver + ssxt_scht_solver,
// occupied bands), :66-101 (reduce_achstemp).
//
// Every update (n1, j, ig, iw) evaluates its own pole factor, the complex
// division included; only the frequency-independent matrix element
// a = conj(aqsm[n1,igp]) * aqsn[n1,ig] is shared across the frequencies of
// one (n1, j, ig), which the reference also computes identically per iw.
//
// One launch holds three kinds of blocks, the long chains first:
//   occupied bands   block = 4 G'-columns of one band, two waves per column
//                    (each half of the block's G range), lane = one G-vector;
//   achstemp         one wave per (band, column group), gpp_device.hpp;
//   unoccupied bands (the hot loop)
//     block  = NW waves = NW bands (one per wave) x BJ G'-columns;
//     lane   = one G-vector ig of a 64-wide chunk; the chunk loop streams the
//              block's G range;
//     LDS    = the chunk's wtilde / I_eps rows of the BJ columns, loaded once
//              per block and read by all NW waves (double-buffered, one barrier
//              per chunk);
//     VGPRs  = the BJ x F per-frequency complex accumulators of each lane.
// The G range is split (DirectArgs::gs) where whole ranges would leave the last
// round of blocks nearly empty.  After its range each wave reduces its
// accumulators by xor butterfly, scales by 0.5*vcoul[igp] and sums its BJ
// columns in column order, writing one partial per (band, column tile, range,
// frequency).  Two fixed-order passes then reduce the partials, so results are
// bitwise reproducible.
//
// The unoccupied bands' loop is bound by the FP64 VALU (about 18 issue slots
// per update, the reciprocal four of them); the occupied ones' by the latency
// of their division chain, so they run beside it: us per call, occupied and
// unoccupied as two launches against one, 512/2/1600/80 33 + 152 -> 161.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "gpp_internal.hpp"

namespace gpp {
namespace {

constexpr int kBJ = 4;   // G' columns per block
constexpr int kNW = 8;   // waves per block (bands, unoccupied; half-columns, occupied)
constexpr int kReduceThreads = 256;
constexpr int kDirectSlots = 512;  // blocks in flight: two per CU

struct DirectArgs {
    const cplx *aqsm, *aqsn, *ieps, *wtilde;
    const int32_t *idx;
    const double *vcoul, *wx;
    int nb, nv, ncouls, ngpown, nfreq;
    int njt, gs, nt;  // column tiles, G ranges, partials per (band, frequency): njt * gs
    int nz;           // frequency passes
    int wx_stride;    // 0: shared wx row; nfreq: band n1 reads wx[n1 * nfreq + iw]
    unsigned occ_blocks, ach_blocks, blocks;  // of the launch: before the unoccupied bands', and all
    double occ;
    cplx *part_ach;   // [nb][nt][nfreq]
    cplx *part_asx;   // [max(nv,1)][nt][nfreq]
    cplx *part_achs;  // [nb][kAchSplit], then the AchCol entries (ach_cols_entry)
    cplx *band_ach;   // [nb][nfreq]
    cplx *band_asx;   // [max(nv,1)][nfreq]
    cplx *bg;         // optional gathered rows of aqsm (factored forms), else null
    const int32_t *perm;  // achstemp launch: row r of bg and part_achs is band perm[r] (null: r)
    Stamp stamp;      // the launch's stage start
    StampEnd end;     // the evaluation's end (last launch)
};

struct WorkLayout {
    size_t part_ach, part_asx, part_achs, band_ach, band_asx, total;
};

__host__ inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

constexpr int kPassWidth = 4;  // frequencies per pass, the last one what remains

// The workspace with gs G ranges.
WorkLayout layout_for(const DevProblem &p, int gs)
{
    const size_t nt = (size_t)((p.ngpown + kBJ - 1) / kBJ) * gs;
    const size_t nvx = p.nv > 0 ? (size_t)p.nv : 1;
    WorkLayout L;
    size_t off = 0;
    L.part_ach = off;  off += align256(sizeof(cplx) * (size_t)p.nb * nt * p.nfreq + sizeof(cplx));
    L.part_asx = off;  off += align256(sizeof(cplx) * nvx * nt * p.nfreq);
    L.part_achs = off; off += align256(sizeof(cplx) * ach_region_entries(p.nb, p.ngpown));
    L.band_ach = off;  off += align256(sizeof(cplx) * ((size_t)p.nb * p.nfreq + 1));
    L.band_asx = off;  off += align256(sizeof(cplx) * nvx * p.nfreq);
    L.total = off;
    return L;
}

// G ranges per (band, column tile): the split that leaves the blocks in flight
// least idle in the last round, with at least six chunks of 64 G-vectors per
// range (a range costs its staging's start and a reduction of its
// accumulators, about 1 % of a block per extra range).  Launches of more than
// 4096 blocks stay whole, and a split's partial sums stay within the scratch of
// the launcher that allocates nothing (they grow with every band, the blocks
// only with the unoccupied ones).
int direct_split(const DevProblem &p)
{
    const int njt = (p.ngpown + kBJ - 1) / kBJ, nun = p.nb - p.nv;
    const double blocks = (double)(nun > 0 ? (nun + kNW - 1) / kNW : p.nv) * njt * ((p.nfreq + 3) / 4);
    if (blocks > 4096) return 1;
    const int chunks = (p.ncouls + kWave - 1) / kWave;
    int best_gs = 1;
    double best = 1e300;
    for (int gs = 1; gs <= 16 && gs * 6 <= std::max(6, chunks) && (gs == 1 || blocks * gs <= 8192); ++gs) {
        if (gs > 1 && kNoAllocHeadBytes + layout_for(p, gs).total > kNoAllocScratchBytes) break;
        const double t = std::ceil(blocks * gs / kDirectSlots) / gs * (1.0 + 0.01 * gs);
        if (t < best) best = t, best_gs = gs;
    }
    return best_gs;
}

DirectArgs make_args(const DevProblem &p, void *work)
{
    const int gs = direct_split(p);
    const WorkLayout L = layout_for(p, gs);
    char *w = static_cast<char *>(work);
    DirectArgs a;
    a.aqsm = p.aqsm; a.aqsn = p.aqsn; a.ieps = p.ieps; a.wtilde = p.wtilde;
    a.idx = p.idx; a.vcoul = p.vcoul; a.wx = p.wx; a.wx_stride = p.wx_stride;
    a.nb = p.nb; a.nv = p.nv; a.ncouls = p.ncouls; a.ngpown = p.ngpown; a.nfreq = p.nfreq;
    a.njt = (p.ngpown + kBJ - 1) / kBJ;
    a.gs = gs;
    a.nt = a.njt * a.gs;
    a.nz = 1;
    a.occ_blocks = a.ach_blocks = a.blocks = 0;
    a.occ = p.occ;
    a.part_ach = reinterpret_cast<cplx *>(w + L.part_ach);
    a.part_asx = reinterpret_cast<cplx *>(w + L.part_asx);
    a.part_achs = reinterpret_cast<cplx *>(w + L.part_achs);
    a.band_ach = reinterpret_cast<cplx *>(w + L.band_ach);
    a.band_asx = reinterpret_cast<cplx *>(w + L.band_asx);
    a.bg = nullptr;
    a.perm = nullptr;
    a.end = StampEnd{};
    return a;
}

// ---------------------------------------------------------------------------
// Per-update arithmetic of the unoccupied bands.
//
// Fast form: with a = conj(aqsm)*aqsn, the reference's term
//   a * ((wtilde * conj(wdiff) * rden) * I_eps),  rden = 1/|wdiff|^2
// is evaluated as ((a * (wtilde * I_eps)) * conj(wdiff)) * rden, the same
// product re-associated; wdiff = wx - wtilde and the reciprocal are formed
// per update as in gppComplex.cpp:139-143, the reciprocal refined to third
// order (rcp_2o: about one rounding, unbiased, as the reference's quotient).
// wtie = wtilde * I_eps, formed once per (column, G-vector) when staged.
template <int FC>
__device__ __forceinline__ void unocc_update_fast(cplx (&acc)[FC], cplx cm, cplx an, cplx wt,
                                                  cplx wtie, const double (&wxv)[FC])
{
    const cplx a = cmul_fast(cm, an);
    const cplx q = cmul_fast(a, wtie);
#pragma unroll
    for (int f = 0; f < FC; ++f) {
        const double wdr = wxv[f] - wt.re;   // wdiff = (wx - wt.re, -wt.im)
        const double d = wdr * wdr + wt.im * wt.im;
        const double r = rcp_2o(d);
        // q * conj(wdiff) = q * (wdr, wt.im)
        const double tr = q.re * wdr - q.im * wt.im;
        const double ti = q.im * wdr + q.re * wt.im;
        acc[f].re += tr * r;
        acc[f].im += ti * r;
    }
}

// Strict form: the reference's operation order for one term,
// gppComplex.cpp:139-146, IEEE division, no FMA contraction.
template <int FC>
__device__ __forceinline__ void unocc_update_strict(cplx (&acc)[FC], cplx cm, cplx an, cplx wt,
                                                    cplx ie, const double (&wxv)[FC])
{
#pragma clang fp contract(off)
    const cplx a = cmul(cm, an);  // product(mygpvar1, aqsn), :146
#pragma unroll
    for (int f = 0; f < FC; ++f) {
        const cplx wdiff = cdminus(wxv[f], wt);                 // :139
        const double wdiffr = cmul(wdiff, cconj(wdiff)).re;     // :140
        const double rden = 1 / wdiffr;                         // :141
        const cplx delw = cscale(cmul(wt, cconj(wdiff)), rden); // :143
        cacc(acc[f], cmul(a, cmul(delw, ie)));                  // :146
    }
}

// ---------------------------------------------------------------------------
// Chunks [c0, c1) of 64 G-vectors of range g.
__device__ __forceinline__ void range_chunks(const DirectArgs &a, int ncouls, int g, int &c0, int &c1)
{
    const int nchunks = (ncouls + kWave - 1) / kWave;
    c0 = (int)((long long)nchunks * g / a.gs);
    c1 = (int)((long long)nchunks * (g + 1) / a.gs);
}

// Unoccupied bands: block b of their share of the launch, frequencies
// [iw0, iw0 + F).  lds: 4 kBJ kWave entries.
template <int F, bool STRICT>
__device__ __forceinline__ void unocc_block(const DirectArgs &a, int ncouls, unsigned b, int iw0, cplx *lds)
{
    constexpr int TILE = kBJ * kWave;  // (column, G-vector) positions per chunk
    static_assert(TILE <= kNW * kWave, "one position per staging thread");
    auto *s_wt = reinterpret_cast<cplx(*)[kBJ][kWave]>(lds);
    auto *s_ie = s_wt + 2;  // I_eps (strict) or wtilde * I_eps (fast)

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const unsigned ngroups = (a.nb - a.nv + kNW - 1) / kNW;
    const int n1 = a.nv + (int)(b % ngroups) * kNW + wave;
    const bool band_ok = n1 < a.nb;
    const int jt = (int)(b / ngroups % (unsigned)a.njt), g = (int)(b / ngroups / (unsigned)a.njt);
    const int j0 = jt * kBJ;

    // conj(aqsm[n1, igp(j)]) per column (mygpvar1, gppComplex.cpp:134).
    cplx cm[kBJ];
#pragma unroll
    for (int jj = 0; jj < kBJ; ++jj) {
        const int j = j0 + jj;
        cm[jj] = czero();
        if (band_ok && j < a.ngpown) cm[jj] = cconj(a.aqsm[(size_t)n1 * ncouls + igp_of(a.idx, j, ncouls)]);
    }
    double wxv[F];
#pragma unroll
    for (int f = 0; f < F; ++f) wxv[f] = band_ok ? a.wx[(size_t)n1 * a.wx_stride + iw0 + f] : 0.0;

    cplx acc[kBJ][F];
#pragma unroll
    for (int jj = 0; jj < kBJ; ++jj)
#pragma unroll
        for (int f = 0; f < F; ++f) acc[jj][f] = czero();

    // Staging of one chunk's wtilde/I_eps tile: thread t < TILE loads both at
    // position t; the fast form stores wtilde * I_eps, formed here once
    // instead of once per band.  Out-of-range entries get wtilde = i (so
    // |wdiff|^2 >= 1) and I_eps = 0: their terms are exact zeros.
    const bool stager = threadIdx.x < TILE;
    const int s_jj = (threadIdx.x % TILE) / kWave, s_l = threadIdx.x % kWave;
    cplx st_wt = czero(), st_ie = czero();
    auto load_chunk = [&](int c) {
        if (!stager) return;
        const int j = j0 + s_jj, ig = c * kWave + s_l;
        const bool ok = j < a.ngpown && ig < ncouls;
        st_wt = ok ? a.wtilde[(size_t)j * ncouls + ig] : mk(0.0, 1.0);
        st_ie = ok ? a.ieps[(size_t)j * ncouls + ig] : czero();
    };
    auto store_chunk = [&](int buf) {
        if (!stager) return;
        s_wt[buf][s_jj][s_l] = st_wt;
        s_ie[buf][s_jj][s_l] = STRICT ? st_ie : cmul_fast(st_wt, st_ie);
    };

    auto load_an = [&](int c) {
        const int ig = c * kWave + lane;
        return band_ok && ig < ncouls ? a.aqsn[(size_t)n1 * ncouls + ig] : czero();
    };
    int c0, c1;
    range_chunks(a, ncouls, g, c0, c1);
    // the fast form loads aqsn of the next chunk while this one is evaluated
    // (the strict form has no registers for it)
    cplx an_next = czero();
    if (!STRICT) an_next = load_an(c0);
    load_chunk(c0);
    store_chunk(0);
    __syncthreads();
    for (int c = c0; c < c1; ++c) {
        const int buf = (c - c0) & 1;
        cplx an = an_next;
        // taken before the next loads are issued: the compiler else put the wait
        // for it after them, which waited for them too (us, with / without:
        // 512/2/16384/819/3 12940 / 12090, 1536/8/65536/1638/4 405500 / 381700)
        if (!STRICT) asm volatile("" : "+v"(an.re), "+v"(an.im));
        if (c + 1 < c1) {
            load_chunk(c + 1);
            if (!STRICT) an_next = load_an(c + 1);
        }
        if (STRICT) an = load_an(c);
        if (band_ok) {
#pragma unroll
            for (int jj = 0; jj < kBJ; ++jj) {
                const cplx wt = s_wt[buf][jj][lane];
                const cplx ie = s_ie[buf][jj][lane];
                if (STRICT) unocc_update_strict<F>(acc[jj], cm[jj], an, wt, ie, wxv);
                else unocc_update_fast<F>(acc[jj], cm[jj], an, wt, ie, wxv);
            }
        }
        if (c + 1 < c1) store_chunk(buf ^ 1);
        __syncthreads();
    }

    if (!band_ok) return;
    // scht per (column, frequency); then sum_j (0.5*scht)*vcoul[igp] in
    // column order (gppComplex.cpp:374, :379).  The wave's sums by the xor
    // butterfly of wave_sum (the same additions), each step on the half of the
    // values this lane goes on with: after three steps lane l holds F of its
    // column's 2 F parts (10 F exchanges of doubles instead of 48 F).  The
    // halves are constants of each step's code: with a loop over them the
    // compiler left the passes of two to index v at run time (890 selects).
    static_assert(kBJ == 4, "two steps split the columns, one the parts");
    double v[kBJ * 2 * F];
#pragma unroll
    for (int jj = 0; jj < kBJ; ++jj)
#pragma unroll
        for (int f = 0; f < F; ++f) {
            v[(jj * F + f) * 2] = acc[jj][f].re;
            v[(jj * F + f) * 2 + 1] = acc[jj][f].im;
        }
    const auto halve = [&](auto half, int m) {
        constexpr int N = decltype(half)::value;
        const bool up = lane & m;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const double keep = up ? v[N + i] : v[i], give = up ? v[i] : v[N + i];
            v[i] = keep + __shfl_xor(give, m, kWave);
        }
    };
    halve(std::integral_constant<int, kBJ * F>(), 1);
    halve(std::integral_constant<int, kBJ * F / 2>(), 2);
    halve(std::integral_constant<int, kBJ * F / 4>(), 4);
    const int col = 2 * (lane & 1) + ((lane >> 1) & 1);  // this lane's column
    const double vc = a.vcoul[igp_of(a.idx, min(j0 + col, a.ngpown - 1), ncouls)];
    double s[F];
#pragma unroll
    for (int i = 0; i < F; ++i) {
        for (int m = 8; m < kWave; m <<= 1) v[i] += __shfl_xor(v[i], m, kWave);
        v[i] = v[i] * 0.5 * vc;
        s[i] = 0.0;
#pragma unroll
        for (int jj = 0; jj < kBJ; ++jj) {
            const double t = __shfl(v[i], (lane & ~3) | (jj >> 1) | ((jj & 1) << 1), kWave);
            if (j0 + jj < a.ngpown) s[i] = t + s[i];
        }
    }
    if ((lane & ~4) == 0) {  // lane 0: the first F parts, lane 4: the others
        double *o = &a.part_ach[((size_t)n1 * a.nt + jt * a.gs + g) * a.nfreq + iw0].re + (lane ? F : 0);
#pragma unroll
        for (int i = 0; i < F; ++i) o[i] = s[i];
    }
}

// Occupied bands n1 < nv: block b of their share, 4 columns of one band over
// one G range; waves jj and jj + 4 take column jj over the range's halves.  The
// sums are combined half by half, then in column order, through LDS.
template <int F>
__device__ __forceinline__ void occ_block(const DirectArgs &a, int ncouls, unsigned b, int iw0, cplx *lds)
{
    auto *s_sum = reinterpret_cast<cplx(*)[2][kBJ][F]>(lds);  // [ach, asx][half][column]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const int jj = wave % kBJ, half = wave / kBJ;
    const unsigned njt = a.njt, nv = a.nv;
    const int jt = (int)(b % njt), n1 = (int)(b / njt % nv), g = (int)(b / njt / nv);
    const int j = jt * kBJ + jj;
    const bool ok = j < a.ngpown;

    double wxv[F], wx2[F], rwx4[F];
#pragma unroll
    for (int f = 0; f < F; ++f) {
        wxv[f] = a.wx[(size_t)n1 * a.wx_stride + iw0 + f];
        // std::pow(wxt,2) and std::pow(cden,2), gppComplex.cpp:38-40
        wx2[f] = wxv[f] * wxv[f];
        rwx4[f] = 1.00 / (wx2[f] * wx2[f]);
    }
    cplx ssxt[F], scht[F];
#pragma unroll
    for (int f = 0; f < F; ++f) ssxt[f] = scht[f] = czero();
    if (ok) {
        const cplx mv1 = cconj(a.aqsm[(size_t)n1 * ncouls + igp_of(a.idx, j, ncouls)]);
        int c0, c1;
        range_chunks(a, ncouls, g, c0, c1);
        const int mid = (c0 + c1 + 1) / 2;
        const int end = (half ? c1 : mid) * kWave < ncouls ? (half ? c1 : mid) * kWave : ncouls;
        for (int ig = (half ? mid : c0) * kWave + lane; ig < end; ig += kWave) {
            const cplx an = a.aqsn[(size_t)n1 * ncouls + ig];
            const cplx wt = a.wtilde[(size_t)j * ncouls + ig];
            const cplx ie = a.ieps[(size_t)j * ncouls + ig];
            const cplx m = cmul(an, mv1);  // matngmatmgp, gppComplex.cpp:121
#pragma unroll
            for (int f = 0; f < F; ++f) {
                cplx sch, ssx;
                occ_pole_terms(wxv[f], wx2[f], rwx4[f], wt, ie, sch, ssx);
                cacc(ssxt[f], cmul(m, ssx));  // :61, :125
                cacc(scht[f], cmul(m, sch));  // :62, :126
            }
        }
    }
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const cplx sx = wave_sum(ssxt[f]);
        const cplx sc = wave_sum(scht[f]);
        if (lane == 0) {
            s_sum[0][half][jj][f] = sc;
            s_sum[1][half][jj][f] = sx;
        }
    }
    __syncthreads();
    if (threadIdx.x < F) {
        const int f = threadIdx.x;
        cplx sa = czero(), sx = czero();
        for (int q = 0; q < kBJ && jt * kBJ + q < a.ngpown; ++q) {
            // achtemp: (0.5*scht)*vcoul (:361, :379); asxtemp: ssxt*(occ*vcoul) (:363)
            const double vc = a.vcoul[igp_of(a.idx, jt * kBJ + q, ncouls)];
            cacc(sa, cscale(cscale(cadd(s_sum[0][0][q][f], s_sum[0][1][q][f]), 0.5), vc));
            cacc(sx, cscale(cadd(s_sum[1][0][q][f], s_sum[1][1][q][f]), a.occ * vc));
        }
        const size_t o = ((size_t)n1 * a.nt + jt * a.gs + g) * a.nfreq + iw0 + f;
        a.part_ach[o] = sa;
        a.part_asx[o] = sx;
    }
}

// One band kind's block `b` of frequency pass z: W frequencies, with R > 0 the
// last pass R.
template <int W, int R, bool STRICT, bool OCC>
__device__ __forceinline__ void direct_pass(const DirectArgs &a, int ncouls, unsigned b, int z, cplx *lds)
{
    const int iw0 = W * z;
    const auto run = [&](auto f) {
        if constexpr (OCC)
            occ_block<decltype(f)::value>(a, ncouls, b, iw0, lds);
        else
            unocc_block<decltype(f)::value, STRICT>(a, ncouls, b, iw0, lds);
    };
    if constexpr (R > 0) {
        if (z == a.nz - 1) {
            run(std::integral_constant<int, R>());
            return;
        }
    }
    run(std::integral_constant<int, W>());
}

// Grids of this many blocks a row: HIP takes at most 2^32 threads along one
// dimension, and many bands and columns over few G-vectors make more.
constexpr unsigned kGridRow = 1u << 20;
__host__ inline dim3 grid_rows(unsigned blocks)
{
    return blocks <= kGridRow ? dim3(blocks) : dim3(kGridRow, (blocks + kGridRow - 1) / kGridRow);
}
__device__ __forceinline__ unsigned block_of_rows() { return blockIdx.y * gridDim.x + blockIdx.x; }

// Blocks in row order (grid_rows): occ_blocks, ach_blocks, then the unoccupied
// bands'.  Each kind's frequency passes one after the other, not by turns: the
// dispatcher deals blocks round robin to eight XCDs, and two passes of unequal
// width by turns gave four of them all the wide ones (us, 200/3/3000/150: five
// frequencies 511 by turns, 409 so).  Passes of equal width take turns by column
// tile, where all bands' blocks run one pass after the other and the tile's rows
// and aqsn are still in the caches (ms, one after the other / by tile:
// 512/2/8192/819/32 58.1 / 57.1, 1536/8/65536/3276/16 3065 / 3049).
// A kernel for each pair of widths (W, the last pass R; 0: W): one with every
// width took 4 registers more than it has, the strict one 29, and ran the
// strict form in passes of three (us, 512/2/16384/819 strict 4 frequencies
// 37600, with a kernel of its own 32200; 200/3/3000/150 direct 2 242, 216).
template <int W, int R, bool STRICT>
__global__ __launch_bounds__(kNW *kWave) __attribute__((amdgpu_waves_per_eu(4))) void k_direct(DirectArgs a)
{
    int ncouls = a.ncouls;
    const StampStart stamp(a.stamp, ncouls);
    __shared__ cplx lds[4 * kBJ * kWave];
    const unsigned b = block_of_rows();
    if (b >= a.blocks) return;
    if (b < a.occ_blocks) {
        const unsigned pass = a.occ_blocks / (unsigned)a.nz;
        direct_pass<W, R, STRICT, true>(a, ncouls, b % pass, b / pass, lds);
    } else if (b < a.occ_blocks + a.ach_blocks) {
        const int item = (int)(b - a.occ_blocks) * kNW + threadIdx.x / kWave;  // band * kAchSplit + column group
        if (item < a.nb * kAchSplit) {
            const auto col = [&](int j) { return ach_col(a.ieps, a.idx, a.vcoul, ncouls, j); };
            const cplx s = achstemp_band(a.aqsm, a.aqsn, col, ncouls, a.ngpown, item / kAchSplit, item % kAchSplit,
                                         nullptr);
            if (threadIdx.x % kWave == 0) a.part_achs[item] = s;
        }
    } else {
        const unsigned before = a.occ_blocks + a.ach_blocks, u = b - before, nz = a.nz;
        if constexpr (R == 0) {
            const unsigned ngroups = (a.nb - a.nv + kNW - 1) / kNW, q = u / ngroups;
            direct_pass<W, R, STRICT, false>(a, ncouls, q / nz * ngroups + u % ngroups, q % nz, lds);
        } else {
            const unsigned pass = (a.blocks - before) / nz;
            direct_pass<W, R, STRICT, false>(a, ncouls, u % pass, u / pass, lds);
        }
    }
    stamp.store();
}

// ---------------------------------------------------------------------------
// achstemp per band, reduce_achstemp (gppComplex.cpp:66-101): one wave per
// band and block, so that the few hundred bands spread over every CU.
// With COLS the columns' entries come from the table k_ach_cols wrote, without
// it each wave forms them itself (one launch instead of two).
constexpr int kAchWaves = 1;
template <bool COLS>
__global__ __launch_bounds__(kAchWaves * kWave) void k_achstemp(DirectArgs a)
{
    if (!COLS) stamp_start(a.stamp);
    const int item = blockIdx.x * kAchWaves + threadIdx.x / kWave;  // band * kAchSplit + column group
    if (item >= a.nb * kAchSplit) return;
    const AchCol *cols = reinterpret_cast<const AchCol *>(a.part_achs + ach_cols_entry(a.nb));
    const auto col = [&](int j) { return COLS ? cols[j] : ach_col(a.ieps, a.idx, a.vcoul, a.ncouls, j); };
    const int r = item / kAchSplit, n1 = a.perm ? a.perm[r] : r;
    const cplx s = achstemp_band(a.aqsm, a.aqsn, col, a.ncouls, a.ngpown, n1, item % kAchSplit,
                                 a.bg ? a.bg + (size_t)r * a.ngpown : nullptr);
    if (threadIdx.x % kWave == 0) a.part_achs[item] = s;
}

__global__ __launch_bounds__(256) void k_ach_cols(DirectArgs a)
{
    stamp_start(a.stamp);
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < a.ngpown)
        reinterpret_cast<AchCol *>(a.part_achs + ach_cols_entry(a.nb))[j] =
            ach_col(a.ieps, a.idx, a.vcoul, a.ncouls, j);
}

// The (band, column group) partials (and the Bg gather when a.bg is set), after
// the columns' entries where forming them once saves more than their launch
// costs.  Without it each of a band's 256 lanes forms every 256th entry, one
// after the other, so the number of columns decides, however many bands there
// are.  Gather stage, us, one launch / two: 512 bands x 40 columns 3.9 / 6.3,
// 512 x 409 9.0 / 12.0, 512 x 1638 33.0 / 33.9, 1536 x 800 40.6 / 43.6, 100 x
// 2600 13.6 / 15.0, 1536 x 3276 162.8 / 158.4, 100 x 5000 27.1 / 25.8, 24 x
// 8000 30.9 / 29.1.
hipError_t launch_ach(const DirectArgs &a, hipStream_t s)
{
    const dim3 grid((a.nb * kAchSplit + kAchWaves - 1) / kAchWaves), block(kAchWaves * kWave);
    if (a.ngpown >= 3072) {
        hipLaunchKernelGGL(k_ach_cols, dim3((a.ngpown + 255) / 256), dim3(256), 0, s, a);
        hipLaunchKernelGGL((k_achstemp<true>), grid, block, 0, s, a);
    } else {
        hipLaunchKernelGGL((k_achstemp<false>), grid, block, 0, s, a);
    }
    return hipGetLastError();
}

// Per (band, frequency), one wave: the partials over column tiles and G ranges
// -> band_ach[n1][iw] (and band_asx for occupied bands).
__global__ __launch_bounds__(kReduceThreads) void k_reduce_bands(DirectArgs a, int n1_begin, int n1_end)
{
    stamp_start(a.stamp);
    const long long pair = (long long)block_of_rows() * (kReduceThreads / kWave) + threadIdx.x / kWave;
    if (pair >= (long long)(n1_end - n1_begin) * a.nfreq) return;
    const int n1 = n1_begin + (int)(pair / a.nfreq), iw = (int)(pair % a.nfreq), lane = threadIdx.x % kWave;
    cplx s = czero(), x = czero();
    for (int t = lane; t < a.nt; t += kWave) {
        const size_t o = ((size_t)n1 * a.nt + t) * a.nfreq + iw;
        s = cadd(s, a.part_ach[o]);
        if (n1 < a.nv) x = cadd(x, a.part_asx[o]);
    }
    s = wave_sum(s);
    x = wave_sum(x);
    if (lane == 0) {
        a.band_ach[(size_t)n1 * a.nfreq + iw] = s;
        if (n1 < a.nv) a.band_asx[(size_t)n1 * a.nfreq + iw] = x;
    }
}

// Final pass over bands [n1_begin, n1_end): block iw < nfreq forms achtemp[iw]
// and asxtemp[iw], block nfreq acht_n1_loc and (with_achs) achstemp -- written
// to out (DevResults), or, with out null, added to the reference launchers'
// split outputs unless the index check found negative entries.
__global__ __launch_bounds__(kReduceThreads) void k_reduce_final(DirectArgs a, cplx *out, CompatOut co, int n1_begin,
                                                                 int n1_end, int with_achs)
{
    __shared__ cplx scratch[kReduceThreads / kWave];
    const int nf = a.nfreq, iw = blockIdx.x;
    const bool add = !out && !(co.bad && *co.bad);
    if (iw < nf) {
        cplx s = czero(), x = czero();
        for (int n1 = n1_begin + threadIdx.x; n1 < n1_end; n1 += blockDim.x) {
            s = cadd(s, a.band_ach[(size_t)n1 * nf + iw]);
            if (n1 < a.nv) x = cadd(x, a.band_asx[(size_t)n1 * nf + iw]);
        }
        s = block_sum(s, scratch);
        x = block_sum(x, scratch);
        if (threadIdx.x == 0) {
            if (out) {
                out[iw] = s;
                out[nf + iw] = x;
            } else if (add) {
                if (co.achtemp_re) co.achtemp_re[iw] += s.re;
                if (co.achtemp_im) co.achtemp_im[iw] += s.im;
                if (co.asxtemp) cacc(co.asxtemp[iw], x);
            }
        }
    } else {
        const int acht_iw = nf > 2 ? 2 : nf - 1;  // gppComplex.cpp:381
        if (out) {
            for (int n1 = threadIdx.x; n1 < a.nb; n1 += blockDim.x)
                out[2 * nf + n1] = (n1 >= n1_begin && n1 < n1_end) ? a.band_ach[(size_t)n1 * nf + acht_iw] : czero();
        } else if (add && co.acht_n1) {
            for (int n1 = n1_begin + threadIdx.x; n1 < n1_end; n1 += blockDim.x)
                cacc(co.acht_n1[n1], a.band_ach[(size_t)n1 * nf + acht_iw]);
        }
        cplx h = czero();
        if (with_achs)
            for (int t = threadIdx.x; t < a.nb * kAchSplit; t += blockDim.x) h = cadd(h, a.part_achs[t]);
        h = block_sum(h, scratch);
        if (threadIdx.x == 0) {
            if (out) {
                out[2 * nf + a.nb] = h;
            } else if (add && with_achs) {
                co.achstemp_re[0] += h.re;
                co.achstemp_im[0] += h.im;
            }
        }
    }
    stamp_end(a.end);
}

__global__ void k_zero_ints(int *p, int n)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}

__global__ void k_check_index(const int32_t *idx, int n, int *count)
{
    int bad = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) bad += idx[i] < 0;
    if (bad) atomicAdd(count, bad);
}

// One block: the negative entries counted into *count and, for a host that
// polls it, *host (pinned memory).
__global__ __launch_bounds__(1024) void k_check_index_once(const int32_t *idx, int n, int *count, int *host)
{
    __shared__ int total;
    if (threadIdx.x == 0) total = 0;
    __syncthreads();
    int bad = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) bad += idx[i] < 0;
    if (bad) atomicAdd(&total, bad);
    __syncthreads();
    if (threadIdx.x == 0) {
        *count = total;
        __hip_atomic_store(host, total, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// The kernel of the problem's pass widths: one pass of up to three frequencies,
// or passes of four and what remains.
template <bool STRICT>
void launch_direct_widths(const DirectArgs &a, dim3 grid, dim3 block, hipStream_t s)
{
    switch (a.nfreq < 4 ? a.nfreq : 4 + a.nfreq % 4) {
    case 1: hipLaunchKernelGGL((k_direct<1, 0, STRICT>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((k_direct<2, 0, STRICT>), grid, block, 0, s, a); break;
    case 3: hipLaunchKernelGGL((k_direct<3, 0, STRICT>), grid, block, 0, s, a); break;
    case 4: hipLaunchKernelGGL((k_direct<4, 0, STRICT>), grid, block, 0, s, a); break;
    case 5: hipLaunchKernelGGL((k_direct<4, 1, STRICT>), grid, block, 0, s, a); break;
    case 6: hipLaunchKernelGGL((k_direct<4, 2, STRICT>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((k_direct<4, 3, STRICT>), grid, block, 0, s, a); break;
    }
}

// The bands' blocks (occ, unocc) and the achstemp partials (achs) in one launch.
hipError_t launch_direct(DirectArgs &a, bool strict, bool occ, bool achs, bool unocc, hipStream_t s)
{
    a.nz = (a.nfreq + kPassWidth - 1) / kPassWidth;
    const int nun = unocc ? a.nb - a.nv : 0;
    const unsigned long long nocc = occ ? (unsigned long long)a.nt * a.nv * a.nz : 0;
    const unsigned long long nach = achs ? ((unsigned long long)a.nb * kAchSplit + kNW - 1) / kNW : 0;
    const unsigned long long all = nocc + nach + (unsigned long long)((nun + kNW - 1) / kNW) * a.nt * a.nz;
    if (all == 0) return hipSuccess;
    if (all > 0x7fffffffull) return hipErrorInvalidConfiguration;
    a.occ_blocks = (unsigned)nocc;
    a.ach_blocks = (unsigned)nach;
    a.blocks = (unsigned)all;
    const dim3 grid = grid_rows(a.blocks), block(kNW * kWave);
    if (strict)
        launch_direct_widths<true>(a, grid, block, s);
    else
        launch_direct_widths<false>(a, grid, block, s);
    return hipGetLastError();
}

// Bands [n1_begin, n1_end) of the partials to the results.
hipError_t launch_reduce(const DirectArgs &a, cplx *out, const CompatOut &co, int n1_begin, int n1_end, int with_achs,
                         hipStream_t s)
{
    const long long pairs = (long long)(n1_end - n1_begin) * a.nfreq;
    DirectArgs f = a;
    f.stamp = Stamp{};
    if (pairs > 0) {
        DirectArgs b = a;
        b.end = StampEnd{};
        hipLaunchKernelGGL(k_reduce_bands, grid_rows((unsigned)((pairs + 3) / 4)), dim3(kReduceThreads), 0, s, b,
                           n1_begin, n1_end);
    }
    hipLaunchKernelGGL(k_reduce_final, dim3(a.nfreq + 1), dim3(kReduceThreads), 0, s, f, out, co, n1_begin, n1_end,
                       with_achs);
    return hipGetLastError();
}

#define GPP_TRY(x)                         \
    do {                                   \
        hipError_t e_ = (x);               \
        if (e_ != hipSuccess) return e_;   \
    } while (0)

}  // namespace

size_t direct_workspace_bytes(const DevProblem &p) { return layout_for(p, direct_split(p)).total; }

hipError_t run_direct(const DevProblem &p, bool strict, void *work, const DevResults &res,
                      hipStream_t s, StageTimer *timer)
{
    DirectArgs a = make_args(p, work);
    const auto stage = [&](const char *nm) { a.stamp = timer ? timer->stage(nm) : Stamp{}; };
    if (timer) timer->begin();
    stage(p.nb == p.nv ? "direct_occupied" : strict ? "direct_unoccupied_strict" : "direct_unoccupied");
    GPP_TRY(launch_direct(a, strict, true, true, true, s));
    stage("direct_reduce");
    if (timer) a.end = timer->end(p.nfreq + 1);
    return launch_reduce(a, res.base, CompatOut{}, 0, p.nb, 1, s);
}

hipError_t run_direct_part(const DevProblem &p, int which, void *work, const CompatOut &co, hipStream_t s)
{
    DirectArgs a = make_args(p, work);
    a.stamp = Stamp{};
    // achstemp alone, with no bands' work to hide it: as the factored forms do it
    // where the columns are many (blocks of one wave, the entries first from 3072
    // columns up).  d_reduce_achstemp, us, k_direct / so: 24 bands x 20000
    // columns 136 / 79, 100 x 2600 32 / 26, 1536 x 3276 126 / 99, 512 x 1638 40 /
    // 37, 512 x 1024 35 / 33, 1536 x 200 34 / 34, 4000 x 100 48 / 58.
    const bool achs = which == 2, alone = achs && p.ngpown >= 1024;
    GPP_TRY(alone ? launch_ach(a, s) : launch_direct(a, false, which == 0, achs, which == 1, s));
    if (which == 0) return launch_reduce(a, nullptr, co, 0, p.nv, 0, s);
    if (which == 1) return launch_reduce(a, nullptr, co, p.nv, p.nb, 0, s);
    return launch_reduce(a, nullptr, co, 0, 0, 1, s);
}

hipError_t launch_achstemp(const DevProblem &p, cplx *part_achs, cplx *bg, Stamp stamp, hipStream_t s,
                           const int32_t *perm)
{
    DirectArgs a = make_args(p, nullptr);
    a.part_achs = part_achs;
    a.bg = bg;
    a.perm = perm;
    a.stamp = stamp;
    return launch_ach(a, s);
}

hipError_t launch_check_index(const int32_t *d_idx, int ngpown, int *d_count, hipStream_t s)
{
    if (ngpown <= 0) return hipSuccess;
    const int blocks = (ngpown + 255) / 256 < 1024 ? (ngpown + 255) / 256 : 1024;
    hipLaunchKernelGGL(k_check_index, dim3(blocks), dim3(256), 0, s, d_idx, ngpown, d_count);
    return hipGetLastError();
}

hipError_t launch_zero_ints(int *d_p, int n, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_zero_ints, dim3((n + 255) / 256 < 64 ? (n + 255) / 256 : 64), dim3(256), 0, s, d_p, n);
    return hipGetLastError();
}

hipError_t launch_check_index_once(const int32_t *d_idx, int ngpown, int *d_count, int *host, hipStream_t s)
{
    hipLaunchKernelGGL(k_check_index_once, dim3(1), dim3(1024), 0, s, d_idx, ngpown, d_count, host);
    return hipGetLastError();
}

}  // namespace gpp
