// Verlet list build (Cabana VerletList<HalfNeighborTag, VerletLayout2D> semantics) in a
// tiled, LDS-staged form.
//
// All records (local and ghost) are binned on Cabana's grid and sorted by cell.  A tile
// is a run of K cells along z in a x a neighbouring (i, j) columns; its rows are one
// contiguous range of sorted slots per column, and every cell of its stencils lies in the
// (a + 2R)^2 columns around it, each again a contiguous slot range.  One workgroup per tile
// copies those ranges into LDS once and every row scans its stencil cells (Cabana's i, j, k
// order and min-distance prune) from LDS.  An entry's low 15 bits are the LDS slot of the
// neighbour times eight (the slot itself where the tile stages in global memory, see entryShift),
// the highest flags the pairs that Cabana's position-lexicographic half discriminator keeps, so
// the exact half list is a sub-list and the force kernels stage the same tile and never gather
// from global memory in their inner loop (dense tiles aside).  Global-index rows (for the API, the
// adjoint and the half-list kernels) are converted from this form on demand.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>

#include <type_traits>

#include "nlist.hpp"

using namespace mrmd_hip;

namespace
{
struct TileGeom
{
    int n0, n1, n2, K, tilesPerCol, R, cols, nbj;
    int o0, o1, o2;  ///< first cell of the region that holds rows, per axis
    int e0, e1, e2;  ///< its extent in cells
};

// first column (i0, j0) and z-run [k0, k1) of tile t; tiles cover only the cells that hold
// list rows (a ghost layer of the grid holds none), so no lane of a tile sits on a cell
// of ghost records
__device__ inline void tileCoords(const TileGeom& tg, int64_t t, int& i0, int& j0, int& k0, int& k1)
{
    const int col = int(t / tg.tilesPerCol);
    const int kb = int(t % tg.tilesPerCol);
    i0 = tg.o0 + (col / tg.nbj) * tg.cols;
    j0 = tg.o1 + (col % tg.nbj) * tg.cols;
    k0 = tg.o2 + kb * tg.K;
    k1 = min(k0 + tg.K, tg.o2 + tg.e2);
}

// tile of a cell inside the row region
__device__ inline int64_t tileOfCell(const TileGeom& tg, int cell)
{
    const int k = cell % tg.n2, ij = cell / tg.n2, i = ij / tg.n1, j = ij % tg.n1;
    return (int64_t((i - tg.o0) / tg.cols) * tg.nbj + (j - tg.o1) / tg.cols) * tg.tilesPerCol + (k - tg.o2) / tg.K;
}

// the maxima of a build (words of the slots in the context's scratch, see raiseTo): the largest staged
// neighbourhood, the widest row, whether there is a record of more than one atom; the rows' cell box
// from BOX_WORD
constexpr int STAGED_WORD = 0, WIDTH_WORD = 1, MULTI_WORD = 2;

// half a wave per tile, a lane per range: row ranges, neighbourhood column ranges and their LDS
// bases.  The ranges' places are prefix sums
// over the lanes and the description goes out in neighbouring words.  (One lane per tile, 150
// scattered loads and 100 scattered stores each, took 12 us at any size up to 20,000 tiles.)
constexpr int SETUP_LANES = 32;
static_assert(MAX_RANGES <= SETUP_LANES);
__global__ __launch_bounds__(BLOCK) void k_tileSetup(TileGeom tg, int64_t ntiles, const int32_t* offsets,
                                                     const int32_t* counts, TileInfo* tiles, int32_t* slots)
{
    const int64_t t = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) / SETUP_LANES;
    if (t >= ntiles) return;  // (whole groups leave together)
    const int q = int(threadIdx.x) % SETUP_LANES;
    int i0, j0, k0, k1;
    tileCoords(tg, t, i0, j0, k0, k1);
    const int span = tg.cols + 2 * tg.R, nr = span * span;
    const int kl = max(k0 - tg.R, 0), kh = min(k1 + tg.R, tg.n2);
    const int iEnd = min(i0 + tg.cols, tg.o0 + tg.e0), jEnd = min(j0 + tg.cols, tg.o1 + tg.e1);
    const int ii = i0 - tg.R + q / span, jj = j0 - tg.R + q % span;
    const bool in = q < nr && ii >= 0 && ii < tg.n0 && jj >= 0 && jj < tg.n1;
    const bool self = in && ii >= i0 && ii < iEnd && jj >= j0 && jj < jEnd;
    const int col = (ii * tg.n1 + jj) * tg.n2;
    int begin = 0, len = 0, selfBegin = 0, rows = 0;
    if (in)
    {
        begin = offsets[col + kl];
        len = offsets[col + kh - 1] + counts[col + kh - 1] - begin;
    }
    if (self)
    {
        selfBegin = offsets[col + k0];
        rows = offsets[col + k1 - 1] + counts[col + k1 - 1] - selfBegin;
    }
    // inclusive sums over the group's lanes
    int lenTo = len, rowsTo = rows, selfTo = self ? 1 : 0;
    for (int off = 1; off < SETUP_LANES; off <<= 1)
    {
        const int a = __shfl_up(lenTo, off, SETUP_LANES), b = __shfl_up(rowsTo, off, SETUP_LANES),
                  c = __shfl_up(selfTo, off, SETUP_LANES);
        if (q >= off)
        {
            lenTo += a;
            rowsTo += b;
            selfTo += c;
        }
    }
    TileInfo& ti = tiles[t];
    if (q < nr)
    {
        ti.base[q] = lenTo - len;
        ti.begin[q] = begin;
    }
    if (self)
    {
        ti.selfRange[selfTo - 1] = q;
        ti.selfBegin[selfTo - 1] = selfBegin;
        ti.selfPrefix[selfTo - 1] = rowsTo - rows;
    }
    if (q == SETUP_LANES - 1)
    {
        ti.selfPrefix[selfTo] = rowsTo;
        ti.nr = nr;
        ti.staged = lenTo;
        ti.nself = selfTo;
        ti.nrows = rowsTo;
        raiseTo(slots, STAGED_WORD, lenTo);
    }
}

__global__ void k_listClear(int32_t* cnt, int64_t n)
{
    const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < n) cnt[k] = 0;
}

constexpr int MAX_SPAN = 64;  // cells of a tile's column range along z (K + 2R)
// records of LDS past the staged neighbourhood that a candidate pass may read (its group of
// four runs up to three records beyond the column run; their bits are cleared)
constexpr int STAGE_PAD = 4;
constexpr size_t LDS_LIMIT = 64000;  // dynamic LDS of a list build workgroup (64 KB less its static part)
// entries of a row that the list build collects in LDS (the least list width, and the least number
// of entries: bufCap); a row's further entries are stored one by one.  A liquid's rows of some 80 fit.
// With buffers of the list's width, at 260,000 atoms a caller's hint of 0, 60, 150 or 300
// neighbours made it 114, 121, 191 or 323 us, and wider rows did not fit at all; now 110 for any
// hint, and rows of 240 take 303 instead of 385.
constexpr int ROW_BUF = 96;
// Where the widest row met so far is a little wider the buffers hold it: rows of up to 109 and 129
// entries, 129 and 154 us, with 96 entries 139 and 174; rows of up to 200 take 288 us with 96 and 313
// with 128 or 144.
constexpr int ROW_BUF_MOST = 144;
// Up to here every workgroup has its LDS to itself (two a CU), and buffers of the list's width are
// taken if four waves have room for them (4,000 atoms, rows of 140 and 240: 31 and 47 us, with 96
// entries 37 and 62)
constexpr int64_t WIDE_BUF_TILES = 2 * 256;
static_assert(ROW_BUF % CHUNK == 0 && ROW_BUF_MOST % CHUNK == 0);

// The list build.  S = 2R + 1 lanes share a row, one per j offset of the stencil, and walk the
// S i offsets together, so a row's columns come in Cabana's i, j, k order: in each step a lane
// takes one column, the S lanes' counts are summed in order, and every lane appends its
// hits behind those of the lanes before it.
//
// What bounds it is vector instruction issue (one lane per row in FP64 took 180 instructions a
// row: 10 per candidate, some 250 candidates, and 20 per entry in a loop that a wave ran 2.4
// times as often as its mean lane).  Candidates are therefore tested on 16-bit coordinates,
// relative to the tile's neighbourhood, 8 bytes a record: two packed subtractions and two
// 16-bit dot products give the squared distance less a threshold in 4 instructions, one more
// shifts its sign into the hit bits and two the sign against a wider threshold.  A coordinate is
// rounded by at most half a unit, so a distance is off by at most sqrt(3) units; pairs
// within 1.75 units of r_n (about 1 in 2,000 candidates) are decided by the FP64 test on the
// records in memory, the unfused expression of the reference, and so is the half-list bit
// of partners whose x differs by less than two units: the list is the exact one.  A record
// outside its tile's range (positions beyond the grid) makes every pair of the tile go that
// way.  The window search runs on the 16-bit z, widened by two units.  A row's first bufCap
// entries are collected in LDS and stored as whole 16-byte chunks of neighbouring rows.
// WIDE: list offsets in 64-bit arithmetic (lists of 2^31 entries or more); 32-bit otherwise
// GS (dense inputs): the 16-bit records in the tile's slice of global memory, entries stored
// one by one
// BUF: the row buffers' entries where the compiler knows them (ROW_BUF, the usual case: 1 % faster)
// or 0 (bufEntries)
constexpr int BUILD_BLOCK = 12 * WAVE;

// (5 waves per SIMD: 96 registers; with 98 it measured 1.14 instead of 1.06 ms at 4M atoms)
template <int R, bool WIDE, bool GS, int BUF>
__global__ __launch_bounds__(BUILD_BLOCK, R == 1 && !GS ? 5 : 4) void k_verletTiled(const double4* __restrict__ sortedPos,
                                                       const int32_t* __restrict__ sorted,
                                                       const int32_t* __restrict__ offsets,
                                                       const TileInfo* __restrict__ tiles, TileGeom tg, GridD g,
                                                       int64_t rowLo, int64_t rowHi, double rsq, double rn,
                                                       uint16_t* nbr, int64_t strideS, int cap, int bufEntries,
                                                       int32_t* cnt, int32_t* slots, int stagedCap, double4* gstage,
                                                       int64_t gstageRecs, double bandLo, double bandHi,
                                                       int8_t* tileSkip)
{
    constexpr int S = 2 * R + 1;
    constexpr int RW = WAVE / S;  // rows of a wave
    constexpr int SH = entryShift(GS);
    const int bufCap = BUF > 0 ? BUF : bufEntries;
    extern __shared__ double4 stRaw[];
    __shared__ TileInfo ti;
    __shared__ int wild;
    const int64_t t = blockIdx.x;
    const int lane = int(threadIdx.x) % WAVE, waves = int(blockDim.x) / WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    // LDS: the waves' row buffers (RW rows of bufCap entries), the 16-bit records, then the LDS slot
    // of the first record of cell kl + z of range r, cstart[r * cz + z] with cz = K + 2R + 1;
    // entry z = nk closes the range (ranges outside the grid are empty)
    uint16_t* const rowBuf = reinterpret_cast<uint16_t*>(stRaw) + (GS ? 0 : wave * RW * bufCap);
    uint2* const ldsRec = reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(stRaw) + (GS ? 0 : waves * RW * bufCap));
    uint2* const rec = GS ? reinterpret_cast<uint2*>(gstage + t * gstageRecs) : ldsRec;
    int* const cstart = reinterpret_cast<int*>(ldsRec + (GS ? 0 : stagedCap + STAGE_PAD));
    const int cz = tg.K + 2 * R + 1;
    loadTile(ti, tiles, t);
    if (threadIdx.x == 0) wild = 0;
    __syncthreads();
    if (ti.nrows == 0) return;
    int i0, j0, k0, k1;
    tileCoords(tg, t, i0, j0, k0, k1);
    if (bandLo <= bandHi)
    {
        // x range of the neighbourhood's cells (the edge cells take every record beyond
        // the grid; widened by 1e-9 of a cell for records binned across a face by rounding)
        const int ia = max(i0 - R, 0), ib = min(i0 + tg.cols - 1 + R, tg.n0 - 1);
        const double xlo = ia == 0 ? -HUGE_VAL : g.min[0] + double(ia) * g.dx[0] - 1e-9 * g.dx[0];
        const double xhi = ib == tg.n0 - 1 ? HUGE_VAL : g.min[0] + double(ib + 1) * g.dx[0] + 1e-9 * g.dx[0];
        const bool skip = xhi < bandLo || xlo > bandHi;
        if (threadIdx.x == 0) tileSkip[t] = skip ? 1 : 0;
        if (skip)
        {
            for (int row = threadIdx.x; row < ti.nrows; row += blockDim.x)
            {
                int self;
                cnt[tileRow(ti, row, self)] = 0;
            }
            return;
        }
    }
    const int span = tg.cols + 2 * R;
    const int kl = max(k0 - R, 0), nk = min(k1 + R, tg.n2) - kl;
    // units of the 16-bit coordinates: the neighbourhood's longest edge is QUANT_RANGE of them, so
    // the differences of a row and a candidate (at most R + 1 of 2R + 1 cells) keep the dot
    // products inside 32 bits
    const double scale =
        QUANT_RANGE / fmax(fmax(double(span) * g.dx[0], double(span) * g.dx[1]), double(tg.K + 2 * R) * g.dx[2]);
    const double ox = g.min[0] + double(i0 - R) * g.dx[0], oy = g.min[1] + double(j0 - R) * g.dx[1],
                 oz = g.min[2] + double(k0 - R) * g.dx[2];
    const Grid16 grid16{ox, oy, oz, scale};
    int sure, doubt;
    grid16.thresholds(rn, sure, doubt);
    bool outside = false;
    stageRecords(ti, sortedPos, [&](int q, const double4& v, int) {
        rec[q] = grid16(v, outside);
    });
    if (outside) wild = 1;
    for (int x = threadIdx.x; x < ti.nr * (nk + 1); x += blockDim.x)
    {
        const int r = x / (nk + 1), z = x % (nk + 1);
        const int ii = i0 - R + r / span, jj = j0 - R + r % span;
        int v = ti.base[r];
        if (ii >= 0 && ii < tg.n0 && jj >= 0 && jj < tg.n1)
        {
            if (z < nk)
                v = ti.base[r] + (offsets[(ii * tg.n1 + jj) * tg.n2 + kl + z] - ti.begin[r]);
            else
                v = r + 1 < ti.nr ? ti.base[r + 1] : ti.staged;
        }
        cstart[r * cz + z] = v;
    }
    __syncthreads();
    const bool exactAll = wild != 0;
    using Off = std::conditional_t<WIDE, int64_t, uint32_t>;
    const int sub = lane % S, group = lane / S, first = group * S;
    int localMax = 0;
    for (int row0 = wave * RW; row0 < ti.nrows; row0 += waves * RW)
    {
        const int row = row0 + group;
        const bool live = group < RW && row < ti.nrows;
        int self = 0;
        const int s = tileRow(ti, live ? row : 0, self);
        const int32_t p = sorted[s];
        const double4 xp = sortedPos[s];
        const bool isRow = live && p >= rowLo && p < rowHi;
        const int selfRange = ti.selfRange[self];
        const int qSelf = ldsSlot(ti, selfRange, s);
        const uint2 own = rec[qSelf];
        const Short2 ownXY = asShort2(own.x), ownZ = asShort2(own.y);
        const int zq = int(int16_t(own.y));
        const int i = i0 - R + selfRange / span, jj = j0 - R + selfRange % span + sub - R;
        const int ck = g.locate1(xp.z, 2);
        // per-axis terms of Cabana's minDistanceToPoint (r per axis of the cell box, summed
        // as r2 = ((0 + rx^2) + ry^2) + rz^2, so lateral part + rz^2 rounds exactly as the
        // full sum) and of the z window (the lateral distances shrunk by 1e-9 of a cell,
        // far more than a record binned across a face by rounding can stray)
        auto boxDistSqr = [&](double x, int cell, int d, double shrink) {
            const double c = g.min[d] + (double(cell) + 0.5) * g.dx[d];
            double r = fabs(x - c) - 0.5 * g.dx[d] - shrink;
            r = r > 0.0 ? r : 0.0;
            return r * r;
        };
        const double ry2 = boxDistSqr(xp.y, jj, 1, 0.0), wy2 = boxDistSqr(xp.y, jj, 1, 1e-9 * g.dx[1]);
        double rz2[S];
#pragma unroll
        for (int dc = 0; dc < S; ++dc) rz2[dc] = boxDistSqr(xp.z, ck - R + dc, 2, 0.0);
        int n = 0;  // entries of the row so far (the same in its S lanes)
        auto step = [&](auto daC) {
            constexpr int da = decltype(daC)::value;
            const int ii = i + da;
            int lo = 0, hi = 0, range = 0;
            if (isRow && ii >= 0 && ii < tg.n0 && jj >= 0 && jj < tg.n1)
            {
                range = (ii - (i0 - R)) * span + (jj - (j0 - R));
                const int* cs0 = cstart + range * cz - kl;
                // Cabana's prune per cell of the column: the distance is unimodal in k, so
                // the surviving cells are one run [kLo, kHi]
                const double lat = boxDistSqr(xp.x, ii, 0, 0.0) + ry2;
                int kLo = INT_MAX, kHi = -1;
#pragma unroll
                for (int dc = 0; dc < S; ++dc)
                {
                    const int kk = ck - R + dc;
                    if (kk >= 0 && kk < tg.n2 && lat + rz2[dc] <= rsq)
                    {
                        kLo = min(kLo, kk);
                        kHi = kk;
                    }
                }
                if (kLo <= kHi)
                {
                    // records inside a column run are z-sorted: the candidates that can pass are
                    // those whose |dz| stays within sqrt(rsq less the squared lateral distance
                    // from the row to the column), widened by 1e-12 rsq, the float root's
                    // rounding and two units; the window's lower edge lies in cell kLo and its
                    // upper edge in cell kHi, so each binary search runs over one cell
                    const double zsq = rsq - (boxDistSqr(xp.x, ii, 0, 1e-9 * g.dx[0]) + wy2) + 1e-12 * rsq;
                    const int reach = zsq >= 0.0 ? int(sqrtf(float(zsq)) * float(scale) * 1.00001f) + 2 : -1;
                    if (reach >= 0)
                    {
                        int a = cs0[kLo], b = cs0[kLo + 1];
                        while (a < b)
                        {
                            const int m = (a + b) >> 1;
                            if (int(int16_t(rec[m].y)) < zq - reach) a = m + 1;
                            else b = m;
                        }
                        lo = a;
                        a = max(lo, cs0[kHi]);
                        b = cs0[kHi + 1];
                        while (a < b)
                        {
                            const int m = (a + b) >> 1;
                            if (int(int16_t(rec[m].y)) > zq + reach) b = m;
                            else a = m + 1;
                        }
                        hi = a;
                    }
                }
            }
            // the hits among up to 32 candidates from qb, candidate u at bit 31 - u, and, for the
            // columns of the row's own x index, their half bits
            auto test = [&](int qb, uint32_t& half) -> uint32_t {
                half = 0;
                const int nq = min(32, hi - qb);
                if (nq <= 0) return 0u;
                uint32_t near = 0, maybe = 0, tie = 0;
                const uint2* q = rec + qb;
                int m = 0;
                // groups of four, whose reads may run up to three records past the run (inside the
                // LDS pad; their bits are cleared below); the bits are shifted in from the
                // sign of the squared distance less either threshold
                for (; m < nq; m += 4)
                {
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                    {
                        const uint2 w = q[m + u];
                        const Short2 dxy = ownXY - asShort2(w.x);
                        const int over = dotSelf(ownZ - asShort2(w.y), dotSelf(dxy, -sure - 1));
                        near = __builtin_amdgcn_alignbit(near, uint32_t(over), 31u);
                        maybe = __builtin_amdgcn_alignbit(maybe, uint32_t(over - doubt), 31u);
                        if constexpr (da == 0)
                        {
                            // the sign of dx (the upper half), and whether it is within two units
                            const uint32_t d = __builtin_bit_cast(uint32_t, dxy);
                            half = __builtin_amdgcn_alignbit(half, d, 31u);
                            unsigned carry;
                            tie = __builtin_addc(tie, tie, unsigned(d + 0x20000u < 0x50000u), &carry);
                        }
                    }
                }
                // align; drop the candidates past the run and the row itself
                const int sh = 32 - m;  // m is 4..32
                uint32_t valid = ~((1u << (32 - nq)) - 1u);
                if (qSelf >= qb && qSelf < qb + nq) valid &= ~(0x80000000u >> (qSelf - qb));
                uint32_t hits = (near << sh) & valid;
                uint32_t unsure = ((maybe & (~near | tie)) << sh) & valid;
                if constexpr (da == 0) half <<= sh;
                if (exactAll)
                {
                    hits = 0;
                    unsure = valid;
                }
                while (unsure)
                {
                    // in FP64: the reference's test, and the half bit, Cabana's lexicographic
                    // discriminator
                    const int u = __builtin_clz(unsure);
                    const uint32_t bit = 0x80000000u >> u;
                    unsure ^= bit;
                    const double4 xn = sortedPos[ti.begin[range] + (qb + u - ti.base[range])];
                    const double dx = xp.x - xn.x, dy = xp.y - xn.y, dz = xp.z - xn.z;
                    hits = dx * dx + dy * dy + dz * dz <= rsq ? hits | bit : hits & ~bit;
                    if constexpr (da == 0)
                    {
                        const bool h = xn.x > xp.x ||
                                       (xn.x == xp.x && (xn.y > xp.y || (xn.y == xp.y && xn.z > xp.z)));
                        half = h ? half | bit : half & ~bit;
                    }
                }
                return hits;
            };
            uint32_t half0, half1, halfT;
            const uint32_t hits0 = test(lo, half0), hits1 = test(lo + 32, half1);
            int mine = __builtin_popcount(hits0) + __builtin_popcount(hits1);
            const bool longRun = __any(hi - lo > 64);  // (dense inputs: the rest is tested twice)
            if (longRun)
                for (int qb = lo + 64; qb < hi; qb += 32) mine += __builtin_popcount(test(qb, halfT));
            // places: behind the row's entries so far and those of the lanes before this one
            int at = n, total = 0;
#pragma unroll
            for (int k = 0; k < S; ++k)
            {
                const int c = __shfl(mine, first + k, WAVE);
                at += k < sub ? c : 0;
                total += c;
            }
            uint16_t* out = rowBuf + group * bufCap + at;
            // the half bit: columns of a larger x index hold larger x (binning is monotone in x),
            // smaller index smaller x; in the row's own x index the sign of dx decides
            auto append = [&](auto checked, int qb, uint32_t hits, uint32_t half) {
                while (hits)
                {
                    const int u = __builtin_clz(hits);
                    hits ^= 0x80000000u >> u;
                    uint32_t v = uint32_t(qb + u) << SH;
                    if (da > 0) v |= 0x8000u;
                    if (da == 0) v |= ((half << u) >> 16) & 0x8000u;
                    if (!GS && (!decltype(checked)::value || at < bufCap))
                        *out = uint16_t(v);
                    else if (!decltype(checked)::value || at < cap)
                        nbr[(Off(at >> 3) * Off(strideS) + Off(s)) * CHUNK + (at & 7)] = uint16_t(v);
                    if (GS || decltype(checked)::value) ++at;
                    ++out;
                }
            };
            // a row that overflows the capacity counts its further hits without storing
            auto appendAll = [&](auto checked) {
                append(checked, lo, hits0, half0);
                append(checked, lo + 32, hits1, half1);
                if (longRun)
                    for (int qb = lo + 64; qb < hi; qb += 32)
                    {
                        const uint32_t h = test(qb, halfT);
                        append(checked, qb, h, halfT);
                    }
            };
            n += total;
            if (__any(n > (GS ? cap : bufCap)))
                appendAll(std::true_type{});
            else
                appendAll(std::false_type{});
        };
        [&]<int... A>(std::integer_sequence<int, A...>) {
            (step(std::integral_constant<int, A - R>{}), ...);
        }(std::make_integer_sequence<int, S>{});
        // pad the last chunk with the sentinel slot (a record beyond every cutoff), so the
        // force kernels' chunk loop needs no bounds test
        const uint32_t pad = uint32_t(sentinelSlot(stagedCap)) << SH;
        const int kept = min(n, cap), nch = (kept + CHUNK - 1) / CHUNK;
        auto padRow = [&](auto checked) {
            for (int k = kept + sub; k < nch * CHUNK; k += S)
            {
                if (!GS && (!decltype(checked)::value || k < bufCap))
                    rowBuf[group * bufCap + k] = uint16_t(pad);
                else
                    nbr[(Off(k >> 3) * Off(strideS) + Off(s)) * CHUNK + (k & 7)] = uint16_t(pad);
            }
        };
        const bool beyond = !GS && __any(n > bufCap);
        if (isRow) beyond ? padRow(std::true_type{}) : padRow(std::false_type{});
        if (live && sub == 0) cnt[s] = isRow ? kept : 0;  // the true width goes to WIDTH_WORD
        localMax = max(localMax, isRow ? n : 0);
        if constexpr (!GS)
        {
            // the wave's rows go out chunk by chunk, neighbouring rows (mostly neighbouring slots)
            // from neighbouring lanes
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            const int bufCh = !isRow ? 0 : beyond ? min(nch, bufCap / CHUNK) : nch;
            const int chunks = RW * waveMaxInt(bufCh);
            for (int x = lane; x - lane < chunks; x += WAVE)
            {
                const int r = x % RW, ch = x / RW;
                const int sr = __shfl(s, r * S, WAVE), nr = __shfl(bufCh, r * S, WAVE);
                if (ch < nr)
                    reinterpret_cast<uint4*>(nbr)[Off(ch) * Off(strideS) + Off(sr)] =
                        reinterpret_cast<const uint4*>(rowBuf + r * bufCap)[ch];
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    }
    // one atomic per wave (every lane of the workgroup reaches this point)
    localMax = waveMaxInt(localMax);
    if (lane == 0 && localMax > 0) raiseTo(slots, WIDTH_WORD, localMax);
}

// tiled rows (per sorted slot, LDS slots) -> global rows (per record begin+r, record indices)
__global__ void k_toGlobal(const uint16_t* nbr16, const int32_t* cnt16, int64_t strideS, const TileInfo* tiles,
                           TileGeom tg, const int32_t* sorted, const int32_t* cellOf, int64_t nslots, int64_t rowLo,
                           int64_t rowHi, uint32_t* nbr, int32_t* cnt, int64_t stride, int shift)
{
    const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s >= nslots) return;
    const int32_t p = sorted[s];
    if (p < rowLo || p >= rowHi) return;
    const int64_t r = p - rowLo;
    const TileInfo& ti = tiles[tileOfCell(tg, cellOf[p])];
    const int c = cnt16[s];
    for (int k = 0; k < c; ++k)
    {
        const uint16_t e = nbr16[entryIndex(k, s, strideS)];
        const int q = (e & 0x7fff) >> shift;
        int rr = 0;
        while (rr + 1 < ti.nr && ti.base[rr + 1] <= q) ++rr;
        const int32_t jrec = sorted[ti.begin[rr] + (q - ti.base[rr])];
        nbr[int64_t(k) * stride + r] = uint32_t(jrec) | ((e & 0x8000) ? 0x80000000u : 0u);
    }
    cnt[r] = c;
}

__global__ void k_gatherSorted(const double4* pos, const int32_t* sorted, int64_t n, double4* out)
{
    const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s < n) out[s] = pos[sorted[s]];
}

__global__ void k_scatterSorted(const double4* sortedPos, const int32_t* sorted, int64_t n, double4* pos)
{
    const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < n) pos[sorted[k]] = sortedPos[k];
}

__global__ void k_invertSorted(const int32_t* sorted, int64_t n, int32_t* slotOf)
{
    const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s < n) slotOf[sorted[s]] = int32_t(s);
}

__global__ void k_zeroI32v(int32_t* p, int64_t n)
{
    const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < n) p[k] = 0;
}

__global__ void k_halfExtract(const uint32_t* nbr, const int32_t* cnt, int64_t nrows, int64_t stride, int32_t* hnbr,
                              int32_t* hcnt)
{
    const int64_t r = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r >= nrows) return;
    const int c = cnt[r];
    int h = 0;
    for (int k = 0; k < c; ++k)
    {
        const uint32_t e = nbr[int64_t(k) * stride + r];
        if (e & 0x80000000u) hnbr[int64_t(h++) * stride + r] = int32_t(e & 0x7fffffffu);
    }
    hcnt[r] = h;
}

__global__ void k_countWithin(const double4* pos, const uint32_t* nbr, const int32_t* cnt, int64_t begin, int64_t rows,
                              int64_t stride, double r2, unsigned long long* out)
{
    const int64_t r = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    unsigned long long h = 0, f = 0;
    if (r < rows)
    {
        const double4 pi = pos[begin + r];
        for (int k = 0; k < cnt[r]; ++k)
        {
            const uint32_t e = nbr[int64_t(k) * stride + r];
            const double4 pj = pos[e & 0x7fffffffu];
            const double dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            if (dx * dx + dy * dy + dz * dz <= r2)
            {
                ++f;
                if (e & 0x80000000u) ++h;
            }
        }
    }
    for (int off = WAVE / 2; off > 0; off >>= 1)
    {
        h += __shfl_xor(h, off, WAVE);
        f += __shfl_xor(f, off, WAVE);
    }
    if (threadIdx.x % WAVE == 0)
    {
        atomicAdd(&out[0], h);
        atomicAdd(&out[1], f);
    }
}

__global__ void k_rowsToHost(const uint32_t* nbr, const int32_t* cnt, int64_t nrows, int64_t stride, int32_t* out,
                             int64_t rowStride, int mask)
{
    const int64_t r = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r >= nrows) return;
    const int c = cnt[r];
    for (int k = 0; k < c && k < rowStride; ++k)
    {
        uint32_t e = nbr[int64_t(k) * stride + r];
        if (mask) e &= 0x7fffffffu;
        out[r * rowStride + k] = int32_t(e);
    }
}

TileGeom geom(const mrmd_verlet_list* vl)
{
    const GridD& g = vl->bin.grid;
    const int a = vl->tileCols;
    return TileGeom{g.n[0], g.n[1], g.n[2], vl->tileK, vl->tilesPerCol, vl->range, a,
                    (vl->rowExtent[1] + a - 1) / a,
                    vl->rowOrigin[0], vl->rowOrigin[1], vl->rowOrigin[2],
                    vl->rowExtent[0], vl->rowExtent[1], vl->rowExtent[2]};
}

int32_t* buildSlots(mrmd_ctx* ctx)
{
    return static_cast<int32_t*>(ctxScratch(ctx, 2, sizeof(int32_t) * MAX_SLOTS * MAX_WORDS));
}

// cell box of the list rows, posted by the binning
void rowRegion(mrmd_verlet_list* vl, const RowBox& rowBox)
{
    const int64_t rows = vl->end - vl->begin;
    int32_t h[6];
    takeI32(vl->ctx, rowBox.tag, 6, h);
    for (int d = 0; d < 3; ++d)
    {
        vl->rowOrigin[d] = 0;
        vl->rowExtent[d] = 0;
        if (rows <= 0) continue;
        // rows exist, so every axis holds at least one cell of them
        if (-h[d] < 0 || h[3 + d] < -h[d] || h[3 + d] >= vl->bin.grid.n[d])
            fail(MRMD_ERR_STATE, "cell box of the list rows out of the grid: axis %d cells [%d, %d] of %d (%lld rows)",
                 d, -h[d], h[3 + d], vl->bin.grid.n[d], (long long)rows);
        vl->rowOrigin[d] = -h[d];
        vl->rowExtent[d] = h[3 + d] + h[d] + 1;
    }
}

// (the slots' STAGED_WORD is zero before the call)
void setupTiles(mrmd_verlet_list* vl, int K)
{
    mrmd_ctx* ctx = vl->ctx;
    vl->tileK = K;
    vl->tilesPerCol = (vl->rowExtent[2] + K - 1) / K;
    const int a = vl->tileCols;
    vl->ntiles = int64_t((vl->rowExtent[0] + a - 1) / a) * ((vl->rowExtent[1] + a - 1) / a) * vl->tilesPerCol;
    vl->tiles.ensure(ctx, std::max<int64_t>(vl->ntiles, 1));
    if (vl->ntiles > 0)
        hipLaunchKernelGGL(k_tileSetup, dim3(gridFor(vl->ntiles * SETUP_LANES)), dim3(BLOCK), 0, ctx->stream, geom(vl),
                           vl->ntiles, vl->bin.offsets.p, vl->bin.counts.p, vl->tiles.p, buildSlots(ctx));
    checkLaunch();
}

// whether there are records whose atom count is not 1 (molecule lists only)
__global__ void k_anyNotOne(const int64_t* numAtoms, int64_t n, int32_t* slots)
{
    const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < n && numAtoms[k] != 1) raiseTo(slots, MULTI_WORD, 1);
}

__global__ void k_clearWord(int32_t* slots, int word) { slots[int(threadIdx.x) * MAX_WORDS + word] = 0; }

// numAtoms (molecule lists) is checked for records of one atom; returns whether all are
bool verletBuild(mrmd_verlet_list* vl, const double4* pos, int64_t nall, int64_t begin, int64_t end, double rn,
                 double ratio, const double* gmin, const double* gmax, int64_t maxNeigh,
                 const int64_t* numAtoms = nullptr)
{
    mrmd_ctx* ctx = vl->ctx;
    REQUIRE(begin >= 0 && begin <= end && end <= nall, "invalid row range [%lld, %lld) of %lld", (long long)begin,
            (long long)end, (long long)nall);
    REQUIRE(rn > 0.0 && ratio > 0.0, "invalid radius / cell ratio");
    REQUIRE(nall < (int64_t(1) << 31) - 1, "more than 2^31 records");
    KTimer t(ctx, "verlet_build");
    vl->nrows = nall;
    vl->begin = begin;
    vl->end = end;
    vl->rn = rn;
    vl->ratio = ratio;
    vl->range = int(std::ceil(1.0 / ratio));
    if (vl->range > 2) fail(MRMD_ERR_UNSUP, "cell ratio %g needs a stencil wider than 5 cells", ratio);
    const double gs = ratio * rn;
    const double delta[3] = {gs, gs, gs};
    const GridD g = makeGrid(gmin, gmax, delta);
    vl->sentinel = std::max({gmax[0], gmax[1], gmax[2]}) + SENTINEL_GAP + 4.0 * rn;
    // the binning's z sort also writes each record's slot (slotOf)
    vl->slotOf.ensure(ctx, std::max<int64_t>(nall, 1));
    int32_t* const slots = buildSlots(ctx);
    RowBox rowBox{begin, end, slots, 0};
    vl->bin.build(ctx, pos, 0, nall, g, true, true, nullptr, nullptr, vl->slotOf.p, &rowBox);
    vl->strideS = std::max<int64_t>(64, (nall + 63) / 64 * 64);
    vl->cnt16.ensure(ctx, vl->strideS);
    if (nall > 0)
        hipLaunchKernelGGL(k_listClear, dim3(gridFor(nall)), dim3(BLOCK), 0, ctx->stream, vl->cnt16.p, nall);
    if (numAtoms && nall > 0)
        hipLaunchKernelGGL(k_anyNotOne, dim3(gridFor(nall)), dim3(BLOCK), 0, ctx->stream, numAtoms, nall, slots);
    rowRegion(vl, rowBox);
    vl->globalValid = false;
    vl->halfValid = false;
    vl->banded = vl->bandLo <= vl->bandHi;
    vl->slotOfValid = true;
    vl->sortedFresh = false;
    // tile shape: a x a columns (a <= 3; 1 when the stencil reaches two cells), height K
    // chosen to stage ~1650 records; shrink until every tile fits in LDS
    const int R = vl->range;
    const int64_t rows = end - begin;
    const double regionCells =
        double(std::max(vl->rowExtent[0], 1)) * std::max(vl->rowExtent[1], 1) * std::max(vl->rowExtent[2], 1);
    const double perCell = std::max(double(std::max<int64_t>(rows, 1)) / regionCells, 1e-3);
    vl->splitRows = rows;
    if (vl->banded)
    {
        // (the neighbourhoods that reach into the band)
        const double width = gmax[0] - gmin[0];
        const double part = std::min(gmax[0], vl->bandHi + rn) - std::max(gmin[0], vl->bandLo - rn);
        vl->splitRows = int64_t(double(rows) * std::min(1.0, std::max(0.0, part / width)));
    }
    // A shape nobody asked for follows the rows: where they are too few to fill the chip, tiles of
    // as many rows as a workgroup of the force kernel holds with its lanes per row, one cell
    // column wide from four lanes on, so that there are more of them.
    const int lg = rowSplit(vl->splitRows);
    // (in sparse cells even the tallest tile of one column has fewer rows than that: two columns)
    const double cells = double(vl->block >> lg) / perCell;
    const bool narrow = lg >= 2 && cells <= double(std::min(g.n[2], MAX_SPAN - 2 * R));
    const int wantCols = vl->givenCols > 0 ? vl->givenCols : narrow ? 1 : mrmd_verlet_list::DEFAULT_COLS;
    int a = std::min(wantCols, R == 1 ? 3 : 1);
    int K = vl->givenCells;
    if (K <= 0 && vl->givenCols <= 0 && lg > 0) K = std::max(1, int(std::min(cells / (a * a), double(MAX_SPAN))));
    if (K <= 0)
    {
        const int W = a + 2 * R;
        K = std::max(1, int(1650.0 / (W * W * perCell) - 2 * R));
    }
    K = std::min({K, g.n[2], MAX_SPAN - 2 * R});
    // The shape is kept for as long as the system is the same: its rows, its grid, and the cells that
    // hold rows within a factor of four (atoms that just reach into further cells do not make it
    // another one).  A shape that had to shrink is where its next build starts (a shape that does not
    // fit costs a launch and a wait), unless the chosen one would now fit at the density of its
    // fullest neighbourhood, which larger neighbourhoods do not exceed.
    mrmd_verlet_list::TileChoice choice{rows, vl->splitRows, {g.n[0], g.n[1], g.n[2]}, R, vl->stageLimit,
                                        regionCells, a, K};
    const bool sameSystem = choice.sameSystem(vl->tileChoice);
    if (sameSystem)
    {
        choice = vl->tileChoice;
        a = choice.cols;
        K = choice.cells;
    }
    auto cellsAround = [&](int cols, int height) {
        return double(std::min(cols + 2 * R, g.n[0])) * std::min(cols + 2 * R, g.n[1]) *
               std::min(height + 2 * R, g.n[2]);
    };
    if (sameSystem && vl->tileK > 0 &&
        vl->maxStaged * cellsAround(a, K) > vl->stageLimit * cellsAround(vl->tileCols, vl->tileK))
    {
        a = vl->tileCols;
        K = vl->tileK;
    }
    vl->tileChoice = choice;
    vl->globalStage = false;
    for (bool again = false;; again = true)
    {
        vl->tileCols = a;
        if (again) hipLaunchKernelGGL(k_clearWord, dim3(1), dim3(MAX_SLOTS), 0, ctx->stream, slots, STAGED_WORD);
        setupTiles(vl, K);
        takeI32(ctx, postMax(ctx, slots, STAGED_WORD, 1), 1, &vl->maxStaged);
        if (vl->maxStaged <= vl->stageLimit) break;
        if (K > 1)
            K = std::max(1, K / 2);
        else if (a > 1)
            --a;
        else
        {
            // dense input: even one cell column by one cell exceeds the LDS limit, so each
            // tile stages its neighbourhood in its own slice of global memory
            vl->globalStage = true;
            break;
        }
    }
    if (vl->globalStage)
    {
        REQUIRE(vl->maxStaged < 32767, "a tile neighbourhood of %d records exceeds the 15-bit entry slots",
                vl->maxStaged);
        vl->gstageRecs = (int64_t(vl->maxStaged) + STAGE_PAD + 1 + 3) / 4 * 4;
        vl->gstage.ensure(ctx, std::max<int64_t>(vl->ntiles, 1) * vl->gstageRecs);
    }
    if (vl->banded) vl->tileSkip.ensure(ctx, std::max<int64_t>(vl->ntiles, 1));
    if (vl->capFull <= 0) vl->capFull = int32_t(std::max<int64_t>(2 * maxNeigh + 16, ROW_BUF));
    vl->capFull = (vl->capFull + CHUNK - 1) / CHUNK * CHUNK;
    bool mono = false;
    const int stagedCap = std::max(vl->maxStaged, 1);
    for (int attempt = 0; attempt < 2; ++attempt)
    {
        vl->nbr16.ensure(ctx, int64_t(vl->capFull) * vl->strideS);
        if (attempt > 0) hipLaunchKernelGGL(k_clearWord, dim3(1), dim3(MAX_SLOTS), 0, ctx->stream, slots, WIDTH_WORD);
        if (vl->ntiles > 0 && end > begin)
        {
            KTimer tk(ctx, "verlet_tiled");
            // LDS: the row buffers, the 16-bit records and the per-cell start table of (a + 2R)^2 ranges
            // x (K + 2R + 1); at most 23,000 bytes without the row buffers, so that six waves fit
            const int W = vl->tileCols + 2 * R, rowsPerWave = WAVE / (2 * R + 1);
            const size_t fixed = (vl->globalStage ? 0 : size_t(stagedCap + STAGE_PAD) * sizeof(uint2)) +
                                 size_t(W * W * (vl->tileK + 2 * R + 1)) * sizeof(int);
            auto perWave = [&](int entries) {
                return vl->globalStage ? 0 : size_t(rowsPerWave) * entries * sizeof(uint16_t);
            };
            const bool wideBuf = vl->ntiles <= WIDE_BUF_TILES && fixed + 4 * perWave(vl->capFull) <= LDS_LIMIT;
            const int widest = (vl->maxFull + CHUNK - 1) / CHUNK * CHUNK;  // (of the last build)
            const int bufCap = wideBuf ? vl->capFull : widest > ROW_BUF && widest <= ROW_BUF_MOST ? widest : ROW_BUF;
            // four waves a workgroup fill the chip from 1,280 tiles on (five waves a SIMD); with
            // fewer tiles their rows go to up to twelve waves
            int waves = int(std::max<int64_t>(vl->block / WAVE, std::min<int64_t>(12, 5120 / vl->ntiles)));
            while (waves > 1 && fixed + waves * perWave(bufCap) > LDS_LIMIT) --waves;
            const size_t lds = fixed + waves * perWave(bufCap);
            auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(unsigned(vl->ntiles)), dim3(waves * WAVE), lds, ctx->stream,
                                   vl->bin.sortedPos.p, vl->bin.sorted.p, vl->bin.offsets.p, vl->tiles.p, geom(vl), g,
                                   begin, end, rn * rn, rn, vl->nbr16.p, vl->strideS, vl->capFull, bufCap,
                                   vl->cnt16.p, slots, stagedCap, vl->gstage.p, vl->gstageRecs, vl->bandLo, vl->bandHi, vl->tileSkip.p);
            };
            const bool wide = vl->forceWide || int64_t(vl->capFull) * vl->strideS >= (int64_t(1) << 31);
            // plain block order: measured faster here than the XCD-contiguous order (1.54 against
            // 1.59 ms at 4M atoms), each XCD's L2 then serves a spread of the grid's columns
            if (vl->globalStage)
            {
                if (R == 1)
                    wide ? launch(k_verletTiled<1, true, true, 0>) : launch(k_verletTiled<1, false, true, 0>);
                else
                    wide ? launch(k_verletTiled<2, true, true, 0>) : launch(k_verletTiled<2, false, true, 0>);
            }
            else if (wide)
                R == 1 ? launch(k_verletTiled<1, true, false, 0>) : launch(k_verletTiled<2, true, false, 0>);
            else if (bufCap == ROW_BUF)
                R == 1 ? launch(k_verletTiled<1, false, false, ROW_BUF>)
                       : launch(k_verletTiled<2, false, false, ROW_BUF>);
            else
                R == 1 ? launch(k_verletTiled<1, false, false, 0>) : launch(k_verletTiled<2, false, false, 0>);
        }
        checkLaunch();
        int32_t hp[2];
        takeI32(ctx, postMax(ctx, slots, WIDTH_WORD, 2), 2, hp);
        const int32_t hmax = hp[0];
        mono = hp[1] == 0;
        vl->maxFull = hmax;
        if (hmax <= vl->capFull) break;
        // Cabana VerletLayout2D: re-count and refill with the larger width
        vl->capFull = (hmax + hmax / 8 + 8 + CHUNK - 1) / CHUNK * CHUNK;
    }
    if (vl->maxFull > vl->capFull) fail(MRMD_ERR_STATE, "neighbour rows did not fit after a re-count");
    return mono;
}
}  // namespace

void mrmd_verlet_list::refreshSorted(const double4* pos)
{
    if (nrows > 0)
        hipLaunchKernelGGL(k_gatherSorted, dim3(gridFor(nrows)), dim3(BLOCK), 0, ctx->stream, pos, bin.sorted.p, nrows,
                           bin.sortedPos.p);
    checkLaunch();
}

void mrmd_verlet_list::positionsFromSlots(double4* pos)
{
    if (nrows > 0)
        hipLaunchKernelGGL(k_scatterSorted, dim3(gridFor(nrows)), dim3(BLOCK), 0, ctx->stream, bin.sortedPos.p,
                           bin.sorted.p, nrows, pos);
    checkLaunch();
}

// (the error paths of the time loop: a launch error is left for the caller's next call)
void mrmd_verlet_list::positionsFromSlotsNoThrow(double4* pos) noexcept
{
    if (nrows > 0)
        hipLaunchKernelGGL(k_scatterSorted, dim3(gridFor(nrows)), dim3(BLOCK), 0, ctx->stream, bin.sortedPos.p,
                           bin.sorted.p, nrows, pos);
}

const int32_t* mrmd_verlet_list::ensureSlotOf()
{
    if (!slotOfValid)
    {
        slotOf.ensure(ctx, std::max<int64_t>(nrows, 1));
        if (nrows > 0)
            hipLaunchKernelGGL(k_invertSorted, dim3(gridFor(nrows)), dim3(BLOCK), 0, ctx->stream, bin.sorted.p, nrows,
                               slotOf.p);
        checkLaunch();
        slotOfValid = true;
    }
    return slotOf.p;
}

void mrmd_verlet_list::ensureGlobal()
{
    if (banded)
        fail(MRMD_ERR_STATE, "the list holds only the rows within reach of the slab's weighted region (built "
                             "inside the AdResS time loop); rebuild it for this use");
    if (globalValid) return;
    const int64_t rows = end - begin;
    stride = std::max<int64_t>(64, (rows + 63) / 64 * 64);
    cnt.ensure(ctx, stride);
    nbr.ensure(ctx, int64_t(std::max(maxFull, 1)) * stride);
    if (rows > 0)
    {
        hipLaunchKernelGGL(k_zeroI32v, dim3(gridFor(rows)), dim3(BLOCK), 0, ctx->stream, cnt.p, rows);
        hipLaunchKernelGGL(k_toGlobal, dim3(gridFor(nrows)), dim3(BLOCK), 0, ctx->stream, nbr16.p, cnt16.p, strideS,
                           tiles.p, geom(this), bin.sorted.p, bin.cellOf.p, nrows, begin, end, nbr.p, cnt.p, stride,
                           entryShift(globalStage));
    }
    checkLaunch();
    globalValid = true;
}

void mrmd_verlet_list::ensureHalf()
{
    if (halfValid) return;
    ensureGlobal();
    const int64_t rows = end - begin;
    capHalf = std::max(maxFull, 1);
    hnbr.ensure(ctx, int64_t(capHalf) * stride);
    hcnt.ensure(ctx, stride);
    if (rows > 0)
        hipLaunchKernelGGL(k_halfExtract, dim3(gridFor(rows)), dim3(BLOCK), 0, ctx->stream, nbr.p, cnt.p, rows, stride,
                           hnbr.p, hcnt.p);
    checkLaunch();
    halfValid = true;
}

extern "C" {

int mrmd_verlet_create(mrmd_ctx* c, mrmd_verlet_list** out)
{
    MRMD_API_BEGIN(c)
    REQUIRE(out, "null output");
    auto* v = new mrmd_verlet_list();
    v->ctx = c;
    *out = v;
    MRMD_API_END
}

int mrmd_verlet_destroy(mrmd_verlet_list* v)
{
    if (!v) return MRMD_OK;
    (void)hipStreamSynchronize(v->ctx->stream);
    delete v;
    return MRMD_OK;
}

int mrmd_verlet_set_tiling(mrmd_verlet_list* vl, int tile_cells, int tile_columns, int block)
{
    MRMD_API_BEGIN(vl ? vl->ctx : nullptr)
    REQUIRE(vl && tile_cells >= 0 && tile_columns >= 1 && tile_columns <= 3, "invalid tiling");
    REQUIRE(block == 64 || block == 128 || block == 192 || block == 256, "workgroup size must be 64, 128, 192 or 256");
    vl->givenCells = tile_cells;
    vl->givenCols = tile_cells > 0 || tile_columns != mrmd_verlet_list::DEFAULT_COLS ? tile_columns : 0;
    vl->tileK = tile_cells;
    vl->tileCols = tile_columns;
    vl->tileChoice = {};
    vl->block = block;
    MRMD_API_END
}

int mrmd_verlet_set_stage_limit(mrmd_verlet_list* vl, int limit)
{
    MRMD_API_BEGIN(vl ? vl->ctx : nullptr)
    REQUIRE(vl && limit >= 0 && limit <= STAGE_MAX, "the stage limit must lie in [0, %d]", STAGE_MAX);
    vl->stageLimit = limit > 0 ? limit : STAGE_MAX;
    MRMD_API_END
}

int mrmd_verlet_set_wide_offsets(mrmd_verlet_list* vl, int on)
{
    MRMD_API_BEGIN(vl ? vl->ctx : nullptr)
    REQUIRE(vl, "null list");
    vl->forceWide = on != 0;
    MRMD_API_END
}

int mrmd_verlet_get_tiling(const mrmd_verlet_list* vl, int* tile_cells, int* tile_columns, int* block,
                           int* max_staged)
{
    if (!vl) return MRMD_ERR_ARG;
    if (tile_cells) *tile_cells = vl->tileK;
    if (tile_columns) *tile_columns = vl->tileCols;
    if (block) *block = vl->block;
    if (max_staged) *max_staged = vl->maxStaged;
    return MRMD_OK;
}

int mrmd_verlet_build(mrmd_verlet_list* vl, const mrmd_atoms* a, int64_t begin, int64_t end, double rn, double ratio,
                      const double* gmin, const double* gmax, int64_t maxNeigh)
{
    MRMD_API_BEGIN(vl ? vl->ctx : nullptr)
    REQUIRE(vl && a && gmin && gmax, "invalid arguments");
    vl->monoOf = nullptr;
    verletBuild(vl, a->pos.p, a->nlocal + a->nghost, begin, end, rn, ratio, gmin, gmax, maxNeigh);
    MRMD_API_END
}

int mrmd_verlet_build_molecules(mrmd_verlet_list* vl, const mrmd_molecules* m, int64_t begin, int64_t end, double rn,
                                double ratio, const double* gmin, const double* gmax, int64_t maxNeigh)
{
    MRMD_API_BEGIN(vl ? vl->ctx : nullptr)
    REQUIRE(vl && m && gmin && gmax, "invalid arguments");
    vl->monoOf = nullptr;
    if (verletBuild(vl, m->pos.p, m->nlocal + m->nghost, begin, end, rn, ratio, gmin, gmax, maxNeigh, m->numAtoms.p))
    {
        vl->monoOf = m;
        vl->monoVersion = m->layoutVersion;
    }
    MRMD_API_END
}

int mrmd_verlet_half_counts(mrmd_verlet_list* vl, int32_t* counts, int64_t n, int64_t* total)
{
    MRMD_API_BEGIN(vl ? vl->ctx : nullptr)
    REQUIRE(vl, "null list");
    vl->ensureHalf();
    const int64_t rows = vl->end - vl->begin;
    std::vector<int32_t> h(static_cast<size_t>(rows));
    if (rows) HIPCHECK(hipMemcpyAsync(h.data(), vl->hcnt.p, size_t(rows) * 4, hipMemcpyDeviceToHost, vl->ctx->stream));
    sync(vl->ctx);
    int64_t tot = 0;
    for (auto v : h) tot += v;
    if (total) *total = tot;
    if (counts)
        for (int64_t i = 0; i < n; ++i)
            counts[i] = (i >= vl->begin && i < vl->end) ? h[size_t(i - vl->begin)] : 0;
    MRMD_API_END
}

int mrmd_verlet_half_neighbors(mrmd_verlet_list* vl, int32_t* host, int64_t n, int64_t rowStride)
{
    MRMD_API_BEGIN(vl ? vl->ctx : nullptr)
    REQUIRE(vl && host && rowStride > 0, "invalid arguments");
    vl->ensureHalf();
    mrmd_ctx* ctx = vl->ctx;
    const int64_t rows = std::min<int64_t>(n, vl->end - vl->begin);
    if (rows <= 0) return MRMD_OK;
    DBuf<int32_t> dev;
    dev.reserve(ctx, rows * rowStride);
    hipLaunchKernelGGL(k_rowsToHost, dim3(gridFor(rows)), dim3(BLOCK), 0, ctx->stream,
                       reinterpret_cast<const uint32_t*>(vl->hnbr.p), vl->hcnt.p, rows, vl->stride, dev.p, rowStride, 0);
    HIPCHECK(hipMemcpyAsync(host, dev.p, size_t(rows * rowStride) * 4, hipMemcpyDeviceToHost, ctx->stream));
    sync(ctx);
    MRMD_API_END
}

int mrmd_verlet_full_neighbors(mrmd_verlet_list* vl, int32_t* host, int32_t* counts, int64_t n, int64_t rowStride)
{
    MRMD_API_BEGIN(vl ? vl->ctx : nullptr)
    REQUIRE(vl && rowStride > 0, "invalid arguments");
    vl->ensureGlobal();
    mrmd_ctx* ctx = vl->ctx;
    const int64_t rows = std::min<int64_t>(n, vl->end - vl->begin);
    if (rows <= 0) return MRMD_OK;
    if (counts) HIPCHECK(hipMemcpyAsync(counts, vl->cnt.p, size_t(rows) * 4, hipMemcpyDeviceToHost, ctx->stream));
    if (host)
    {
        DBuf<int32_t> dev;
        dev.reserve(ctx, rows * rowStride);
        hipLaunchKernelGGL(k_rowsToHost, dim3(gridFor(rows)), dim3(BLOCK), 0, ctx->stream, vl->nbr.p, vl->cnt.p, rows,
                           vl->stride, dev.p, rowStride, 1);
        HIPCHECK(hipMemcpyAsync(host, dev.p, size_t(rows * rowStride) * 4, hipMemcpyDeviceToHost, ctx->stream));
        sync(ctx);
    }
    sync(ctx);
    MRMD_API_END
}

int mrmd_verlet_count_within(mrmd_verlet_list* vl, const mrmd_atoms* a, double r, int64_t* half, int64_t* full)
{
    MRMD_API_BEGIN(vl ? vl->ctx : nullptr)
    REQUIRE(vl && a && vl->nrows <= a->size, "invalid arguments");
    vl->ensureGlobal();
    mrmd_ctx* ctx = vl->ctx;
    const int64_t rows = vl->end - vl->begin;
    unsigned long long* d = static_cast<unsigned long long*>(ctxScratch(ctx, 2, 64));
    HIPCHECK(hipMemsetAsync(d, 0, 16, ctx->stream));
    if (rows > 0)
        hipLaunchKernelGGL(k_countWithin, dim3(gridFor(rows)), dim3(BLOCK), 0, ctx->stream, a->pos.p, vl->nbr.p,
                           vl->cnt.p, vl->begin, rows, vl->stride, r * r, d);
    checkLaunch();
    unsigned long long h[2];
    HIPCHECK(hipMemcpyAsync(h, d, 16, hipMemcpyDeviceToHost, ctx->stream));
    sync(ctx);
    if (half) *half = int64_t(h[0]);
    if (full) *full = int64_t(h[1]);
    MRMD_API_END
}

int mrmd_verlet_info(const mrmd_verlet_list* vl, int64_t* rows, int32_t* maxFull, int64_t* totalFull, int32_t* dims)
{
    if (!vl) return MRMD_ERR_ARG;
    MRMD_API_BEGIN(vl->ctx)
    if (rows) *rows = vl->end - vl->begin;
    if (maxFull) *maxFull = vl->maxFull;
    if (totalFull)
    {
        auto* v = const_cast<mrmd_verlet_list*>(vl);
        const int64_t r = v->end - v->begin;
        std::vector<int32_t> h(static_cast<size_t>(r));
        if (r)
        {
            v->ensureGlobal();
            HIPCHECK(hipMemcpyAsync(h.data(), v->cnt.p, size_t(r) * 4, hipMemcpyDeviceToHost, v->ctx->stream));
            sync(v->ctx);
        }
        int64_t t = 0;
        for (auto c : h) t += c;
        *totalFull = t;
    }
    if (dims)
        for (int d = 0; d < 3; ++d) dims[d] = vl->bin.grid.n[d];
    MRMD_API_END
}

}  // extern "C"
