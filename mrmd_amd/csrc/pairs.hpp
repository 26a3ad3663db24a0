// Pair terms of the tiled force kernels: four list entries at a time.
#pragma once

#include "nlist.hpp"
#include "physics.hpp"

namespace mrmd_hip
{
// 1/d^2 outside the cutoff made negligible with one select: the high word cleared leaves a
// value below 2^-1022 whose square underflows to zero, so every term of the pair (f2^3, its
// products and the force) comes out zero as from a zeroed reciprocal, with the same signs
__device__ inline double maskReciprocal(double f2, bool in)
{
    const long long b = __double_as_longlong(f2);
    return __hiloint2double(in ? int(b >> 32) : 0, int(b));
}

// the staged records of four consecutive list entries
struct Quad
{
    double x[4], y[4], z[4], w[4];
};
template <bool GS, class St>
__device__ inline Quad loadQuad(const St& st, uint32_t lo, uint32_t hi)
{
    Quad q;
    const uint32_t e[4] = {lo & 0x7fffu, (lo >> 16) & 0x7fffu, hi & 0x7fffu, (hi >> 16) & 0x7fffu};
#pragma unroll
    for (int u = 0; u < 4; ++u)
    {
        const double4 v = st.at(e[u] << (3 - entryShift(GS)));
        q.x[u] = v.x;
        q.y[u] = v.y;
        q.z[u] = v.z;
        q.w[u] = v.w;
    }
    return q;
}

// The entries of one row (c of them, chunks of eight at `chunk`, the first already in `cur`),
// four at a time in order; an index chunk is requested a chunk ahead.  BOTH: the two fours of a
// chunk are laid out in a row (for bodies that leave registers for it), not in a loop.  From global
// memory (GS) both fours and then the next index chunk are loaded before either is computed: few
// tiles are in flight there, and a four's loads are a wait for memory.  (Two fours in flight from
// LDS, the next loaded while one is computed, measured no faster: 419 against 415 us at 4M atoms.)
template <bool BOTH, bool GS, class St, class Body>
__device__ inline void walkRow(const St& st, const uint4* __restrict__ chunk, int64_t stride, int c, uint4 cur,
                               Body body)
{
    const int nch = (c + CHUNK - 1) / CHUNK;
    if (nch == 0) return;
    uint4 nxt = cur;
    if (nch > 1) nxt = chunk[stride];
    for (int ch = 0; ch < nch; ++ch)
    {
        const uint4 now = cur;
        cur = nxt;
        if constexpr (GS)
        {
            const Quad a = loadQuad<GS>(st, now.x, now.y), b = loadQuad<GS>(st, now.z, now.w);
            if (ch + 2 < nch) nxt = chunk[int64_t(ch + 2) * stride];
            body(a);
            body(b);
            continue;
        }
        if (ch + 2 < nch) nxt = chunk[int64_t(ch + 2) * stride];
        if constexpr (BOTH)
        {
            body(loadQuad<GS>(st, now.x, now.y));
            body(loadQuad<GS>(st, now.z, now.w));
        }
        else
        {
#pragma unroll 1
            for (int h = 0; h < 2; ++h) body(loadQuad<GS>(st, h ? now.z : now.x, h ? now.w : now.y));
        }
    }
}

// The same for one of the 2^lg lanes that share the row: fours sub, sub + 2^lg, ...  PAIR: two of them
// loaded before either is computed
template <bool PAIR, bool GS, class St, class Body>
__device__ inline void walkRowSplit(const St& st, const uint4* __restrict__ chunk, int64_t stride, int c,
                                    int sub, int lg, Body body)
{
    const int nq = (c + 3) / 4, step = 1 << lg;
    auto four = [&](int q) { return reinterpret_cast<const uint2*>(chunk + int64_t(q >> 1) * stride)[q & 1]; };
    uint2 nxt = {0, 0};
    if (sub < nq) nxt = four(sub);
    if constexpr (PAIR)
    {
        // (a lane without a second four loads some record for it; every four is computed inside the
        // loop, so that the lane with the most of them takes part wherever another does: PairSums
        // counts on it)
        uint2 nxt2 = {0, 0};
        if (sub + step < nq) nxt2 = four(sub + step);
        for (int q = sub; q < nq; q += 2 * step)
        {
            const Quad a = loadQuad<GS>(st, nxt.x, nxt.y), b = loadQuad<GS>(st, nxt2.x, nxt2.y);
            if (q + 2 * step < nq) nxt = four(q + 2 * step);
            if (q + 3 * step < nq) nxt2 = four(q + 3 * step);
            body(a);
            if (q + step < nq) body(b);
        }
        return;
    }
    for (int q = sub; q < nq; q += step)
    {
        const uint2 now = nxt;
        if (q + step < nq) nxt = four(q + step);
        body(loadQuad<GS>(st, now.x, now.y));
    }
}

__device__ inline void quadDistances(const double4& pi, const Quad& q, double dx[4], double dy[4], double dz[4],
                                     double d2[4])
{
#pragma clang fp contract(fast)
#pragma unroll
    for (int u = 0; u < 4; ++u)
    {
        dx[u] = pi.x - q.x[u];
        dy[u] = pi.y - q.y[u];
        dz[u] = pi.z - q.z[u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) d2[u] = dx[u] * dx[u] + dy[u] * dy[u] + dz[u] * dz[u];
}

// What a lane sums up.  Multi-type tables: e = energies, w = sum of ff d^2.  Single-type tables
// (ljQuadOne): e = sum of f6 = d^-6 and w = sum of g = f6 (ff1 f6 - ff2) = ff d^2 over the
// uncapped pairs, eCap and wCap the energies (without the shift) and ff d^2 of the capped ones,
// and the number of pairs inside rc, which the shift needs: popcounts of the wave's active
// lanes on the scalar unit and one vector add per four entries, so the lane with the longest
// row has seen every pair of the wave in a round (pairs), and endRound takes the largest.
struct PairSums
{
    double fx = 0.0, fy = 0.0, fz = 0.0, e = 0.0, w = 0.0, eCap = 0.0, wCap = 0.0;
    int pairs = 0, total = 0;
    __device__ void startRow()
    {
        fx = fy = fz = 0.0;
        pairs = 0;
    }
    /// the row's force, summed over its 2^lg lanes (all of them, in a fixed order)
    __device__ void joinRow(int lg)
    {
        for (int off = 1; off < 1 << lg; off <<= 1)
        {
            fx += __shfl_xor(fx, off, WAVE);
            fy += __shfl_xor(fy, off, WAVE);
            fz += __shfl_xor(fz, off, WAVE);
        }
    }
    /// every lane of the wave, after its row of this round (if any)
    __device__ void endRound()
    {
        total += waveMaxInt(pairs);
        pairs = 0;
    }
    /// this lane's energy and virial sums (the wave's shift on lane 0): energy ef1 sum f6^2 -
    /// ef2 sum f6 - shift n with sum f6^2 = (sum g + ff2 sum f6) / ff1
    template <bool CAP>
    __device__ void finish(const Pre& p, double& energy, double& virial) const
    {
#pragma clang fp contract(fast)
        const double s12 = p.ff1 != 0.0 ? (w + p.ff2 * e) / p.ff1 : 0.0;
        // (where sum f6 overflows so does sum f6^2, and the energy is the latter's infinity)
        energy = p.ef1 * s12 - (isinf(e) ? 0.0 : p.ef2 * e);
        virial = w;
        if (CAP)
        {
            energy += eCap;
            virial += wCap;
        }
        if (threadIdx.x % WAVE == 0) energy -= p.shift * double(total);
    }
};

// Branch-free pair terms of four entries of a single-type table, written stage by stage so that
// the four dependency chains interleave.  Padding entries (the sentinel record) and pairs
// beyond rc have their reciprocal masked, so every term of theirs is zero.  CAP: the table has a
// capping distance; the capped form (LennardJones.hpp:68-75) runs, one entry after the other
// (its square root and quotient need many registers), only where some lane of the wave has a
// capped pair, and such a pair is masked out of the other sums.  allowed(u, d2): whether the pair
// of entry u counts at all.  Products and sums may contract to FMAs here (the neighbour decision of
// the list is unaffected: it is made, unfused, at build time); the forces then differ from the
// unfused CPU arithmetic by a few ulps per term.
template <bool CAP, class Allowed>
__device__ inline void ljQuadOne(const Pre& p, double rcSqr, const double4& pi, const Quad& q, PairSums& s,
                                 Allowed allowed)
{
#pragma clang fp contract(fast)
    double dx[4], dy[4], dz[4], d2[4], frac2[4];
    bool in[4], capped = false;
    quadDistances(pi, q, dx, dy, dz, d2);
#pragma unroll
    for (int u = 0; u < 4; ++u)
    {
        // padding entries point at the sentinel record beyond every cutoff, so the cutoff test
        // alone decides
        in[u] = d2[u] <= rcSqr && allowed(u, d2[u]);
        if (CAP) capped = capped || (in[u] && d2[u] < p.capDistSqr);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) frac2[u] = recipNewton(d2[u]);
    int pairs = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) pairs += __popcll(__ballot(in[u]));
    s.pairs += pairs;
    if (CAP && __any(capped))
    {
#pragma unroll
        for (int u = 0; u < 4; ++u)
        {
            const bool c = in[u] && d2[u] < p.capDistSqr;
            if (__any(c))
            {
                // keeps the block a branch: the compiler would otherwise evaluate it every time
                asm volatile("" ::: "memory");
                const double dist = sqrt(d2[u]);
                const double ff = c ? p.capCoeff / dist : 0.0;
                s.fx += dx[u] * ff;
                s.fy += dy[u] * ff;
                s.fz += dz[u] * ff;
                s.eCap += c ? p.eCap - (dist - p.capDist) * p.capCoeff : 0.0;
                s.wCap += ff * d2[u];
                in[u] = in[u] && !c;
            }
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
    {
        const double f2 = maskReciprocal(frac2[u], in[u]);
        const double f4 = f2 * f2, f6 = f4 * f2;
        const double t = p.ff1 * f6 - p.ff2, g = f6 * t;
        const double ff = g * f2;
        s.fx += dx[u] * ff;
        s.fy += dy[u] * ff;
        s.fz += dz[u] * ff;
        // (spelt out: contracted or not according to the block that the compiler leaves them in,
        // the kernels of one table would differ in the last bit of their energies)
        s.e = __builtin_fma(f4, f2, s.e);
        s.w = __builtin_fma(f6, t, s.w);
    }
}
}  // namespace mrmd_hip
