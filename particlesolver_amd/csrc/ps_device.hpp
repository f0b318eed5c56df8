// ps_device.hpp — device helpers shared by the forward kernels
// (ps_kernels.hip) and the adjoint kernels (ps_adjoint.hip): launch mapping,
// neighbour-table access, the pair arithmetic shared with the CPU oracle,
// the wall-jitter RNG and the world-box projection.
#pragma once

#include "ps_internal.hpp"

namespace ps {

__device__ __forceinline__ uint32_t xcd_block(uint32_t b = blockIdx.x, uint32_t nb = gridDim.x)
{
    const uint32_t x = b & 7u, q = nb >> 3, r = nb & 7u;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// A status word as this kernel has updated it so far, read before an atomic
// that may change nothing.  The words only grow (bits set, maxima raised)
// within a kernel, so a stale value can only cost a redundant atomic.
__device__ __forceinline__ uint32_t status_peek(const uint32_t *w)
{
    return __atomic_load_n(w, __ATOMIC_RELAXED);
}

// Cell coordinate of p on one axis (calcGridPos, integration_kernel.cuh:
// 187-194): floor((p - o) / cell) by IEEE division, clamped into [0, g - 1]
// of the dense grid (positions outside raise PS_STATUS_OUTSIDE_GRID in
// flags, non-finite ones PS_STATUS_NONFINITE and land in cell 0).
__device__ __forceinline__ uint32_t cell_axis(float p, float o, float cell, uint32_t g,
                                              uint32_t &flags)
{
    float f = floorf((p - o) / cell);
    if (!(f >= 0.0f)) {
        flags |= (f != f) ? PS_STATUS_NONFINITE : PS_STATUS_OUTSIDE_GRID;
        return 0u;
    }
    if (f >= (float)g) {
        flags |= PS_STATUS_OUTSIDE_GRID;
        return g - 1u;
    }
    return (uint32_t)f;
}

// chunk m (entries 4m..4m+3) of particle i is nbr_lane(b, i)[m * 64]
__device__ __forceinline__ const uint4 *nbr_lane(const DevBuffers &b, uint32_t i)
{
    return reinterpret_cast<const uint4 *>(b.nbr) + (size_t)(i >> 6) * b.kq * 64 + (i & 63);
}

// A staged unit's table holds 16-bit LDS indices: eight entries (two chunks
// of four) per uint4, in the first half of its particles' share of nbr.
// Chunk m (entries 4m..4m+3) is the uint2 nbr16_chunk(b, i, m); the two
// chunks of a pair and consecutive lanes are contiguous.
__device__ __forceinline__ const uint2 *nbr16_chunk(const DevBuffers &b, uint32_t i, uint32_t m)
{
    return reinterpret_cast<const uint2 *>(b.nbr) +
           (((size_t)(i >> 6) * b.kq + (m >> 1)) * 64 + (i & 63)) * 2 + (m & 1u);
}

// One lane's share of a staged particle's table, its chunks first, first +
// STRIDE, ...; the first PRE of them are loaded by load(), which a kernel
// calls before it stages its unit, so these loads and the staging loads wait
// together.  (The loads do not depend on the entry count: they are clamped
// to the particle's share of the table, and chunks past the count hold
// whatever is there and are never visited.)  The chunks a particle uses are
// visited whole: the builder pads the last one with the sentinel record,
// which fails every pair test.  32 entries a particle (PRE chunks of two
// halves, or of four quarters) cover the mean of about 28.
// With 32-bit entries fetched as they are visited, at 4,194,304 particles
// (a table of 470 MB, past the 256 MB of the last-level cache) lambda took
// 200 us, the solve 221 and finalize 286; with 16-bit entries loaded ahead
// 159, 200 and 241.  At 1,048,576: 38.0, 43.9 and 56.1 us, now 35.6, 43.5
// (bound by VALU issue) and 52.1.
// PIPE: the LDS records of the next chunk go in flight before a chunk is
// visited; without it a chunk's four records are all that is held (for
// records of tens of bytes).
template <uint32_t STRIDE, uint32_t PRE, bool PIPE = true>
struct StagedTable {
    static constexpr uint32_t kRows = STRIDE / 2;  // chunk pairs per step
    const uint2 *base;
    uint2 q[PRE];

    __device__ __forceinline__ void load(const DevBuffers &b, uint32_t i, uint32_t first)
    {
        base = nbr16_chunk(b, i, first);
        const uint32_t room = b.kq - 1u, r0 = first >> 1;  // pairs of this share: 0 .. room
#pragma unroll
        for (uint32_t t = 0; t < PRE; t++)
            q[t] = *nbr16_chunk(b, i, 2u * min(r0 + kRows * t, room) + (first & 1u));
    }

    // fn(entry, gather(entry)) for this lane's entries of the first c, in
    // table order
    template <typename G, typename Fn>
    __device__ __forceinline__ void visit(uint32_t first, uint32_t c, G gather, Fn fn) const
    {
        const uint32_t nch = (c + 3u) >> 2;  // chunks in use
        const uint32_t mine = nch > first ? (nch - first + STRIDE - 1u) / STRIDE : 0u;
        constexpr uint32_t kSent = kStageSentinel | (kStageSentinel << 16);
        auto take = [&](uint32_t t) {
            return t < mine ? q[t] : make_uint2(kSent, kSent);
        };
        struct Four {
            decltype(gather(0u)) a, b, c, d;
        };
        auto gather4 = [&](const uint2 &e) {
            return Four{gather(e.x & 0xffffu), gather(e.x >> 16), gather(e.y & 0xffffu), gather(e.y >> 16)};
        };
        auto visit4 = [&](const uint2 &e, const Four &r) {
            fn(e.x & 0xffffu, r.a);
            fn(e.x >> 16, r.b);
            fn(e.y & 0xffffu, r.c);
            fn(e.y >> 16, r.d);
        };
        if constexpr (PIPE) {
            uint2 e = take(0);
            Four r = gather4(e);
#pragma unroll
            for (uint32_t t = 0; t < PRE; t++) {
                const uint2 en = t + 1 < PRE ? take(t + 1) : e;
                Four rn = r;
                if (t + 1 < PRE) rn = gather4(en);
                if (t < mine) visit4(e, r);
                e = en;
                r = rn;
            }
        } else {
#pragma unroll
            for (uint32_t t = 0; t < PRE; t++)
                if (t < mine) visit4(q[t], gather4(q[t]));
        }
        if (mine > PRE) {
            uint2 e = base[(size_t)PRE * kRows * 128];
            for (uint32_t t = PRE; t < mine; t++) {
                const uint2 en = base[(size_t)min(t + 1u, mine - 1u) * kRows * 128];
                visit4(e, gather4(e));
                e = en;
            }
        }
    }
};

// The entries of half h of a staged particle's first c neighbours in table
// order, one at a time: for the rarely taken recomputation of one half.
template <typename Fn>
__device__ __forceinline__ void for_staged_half_plain(const DevBuffers &b, uint32_t i, uint32_t c, uint32_t h,
                                                      Fn fn)
{
    for (uint32_t q0 = 4u * h; q0 < c; q0 += 8u)
        for (uint32_t q = q0; q < q0 + 4u && q < c; q++)
            fn((uint32_t)reinterpret_cast<const uint16_t *>(nbr16_chunk(b, i, q >> 2))[q & 3u]);
}

// The fluid sums (density, λ's gradient sums, the Δp sum) are formed in two
// halves, h = 0 over the table's chunks 0, 2, 4, ... and h = 1 over chunks
// 1, 3, 5, ..., each in table order, and then added as half 0 + half 1.  The
// staged kernels give each half its own lane (two lanes per particle, twice
// the wavefronts for the same LDS); the others visit both halves in turn.
// Visits the entries of half h of particle i's first c neighbours (global
// slots) in table order, calling fn(j, gather(j)) for each.
// Software-pipelined: while chunk m of the half is processed, the four gathers
// of chunk m + 1 and the index load of chunk m + 2 are already in flight.  The
// loop is unrolled over two chunks whose record sets swap roles, so no records
// are copied between registers.  Every entry of a chunk at or below the last
// one is a valid slot (the builder pads the last chunk with the particle's
// own), so all loads are unconditional; only fn is guarded.
template <typename G, typename Fn>
__device__ __forceinline__ void for_neighbors_half(const DevBuffers &b, uint32_t i, uint32_t c, uint32_t h,
                                                   G gather, Fn fn)
{
    const uint32_t nch = (c + 3u) >> 2;  // chunks in use
    if (h >= nch) return;
    const uint4 *nb = nbr_lane(b, i);
    const uint32_t last = ((nch - h + 1u) >> 1) - 1u;  // this half's chunks: 2m + h, m <= last
    auto chunk = [&](uint32_t m) { return nb[(size_t)(2u * min(m, last) + h) * 64]; };
    auto visit = [&](const uint4 &jj, uint32_t m, const auto &d0, const auto &d1, const auto &d2,
                     const auto &d3) {
        const uint32_t q = (2u * m + h) << 2;  // table position of jj.x
        fn(jj.x, d0);
        if (q + 1 < c) fn(jj.y, d1);
        if (q + 2 < c) fn(jj.z, d2);
        if (q + 3 < c) fn(jj.w, d3);
    };
    uint4 ja = chunk(0);
    uint4 jb = chunk(1);
    auto a0 = gather(ja.x);
    auto a1 = gather(ja.y);
    auto a2 = gather(ja.z);
    auto a3 = gather(ja.w);
    for (uint32_t m = 0;; m += 2) {
        const uint4 jc = chunk(m + 2);
        auto b0 = gather(jb.x);
        auto b1 = gather(jb.y);
        auto b2 = gather(jb.z);
        auto b3 = gather(jb.w);
        visit(ja, m, a0, a1, a2, a3);
        if (m + 1 > last) break;
        const uint4 jd = chunk(m + 3);
        a0 = gather(jc.x);
        a1 = gather(jc.y);
        a2 = gather(jc.z);
        a3 = gather(jc.w);
        visit(jb, m + 1, b0, b1, b2, b3);
        if (m + 2 > last) break;
        ja = jc;
        jb = jd;
    }
}

// The chunks first, first + stride, first + 2 stride, ... of particle i's
// first c neighbours, one chunk at a time (four records in flight), each in
// table order: quarter q of the table is first = q, stride = 4.
template <typename G, typename Fn>
__device__ __forceinline__ void for_neighbors_strided_chunked(const DevBuffers &b, uint32_t i, uint32_t c,
                                                              uint32_t first, uint32_t stride, G gather,
                                                              Fn fn)
{
    const uint32_t nch = (c + 3u) >> 2;  // chunks in use
    if (first >= nch) return;
    const uint4 *nb = nbr_lane(b, i);
    uint4 jj = nb[(size_t)first * 64];
    for (uint32_t m = first; m < nch; m += stride) {
        const uint4 jn = nb[(size_t)(m + stride < nch ? m + stride : m) * 64];
        auto d0 = gather(jj.x);
        auto d1 = gather(jj.y);
        auto d2 = gather(jj.z);
        auto d3 = gather(jj.w);
        const uint32_t q = m << 2;
        fn(jj.x, d0);
        if (q + 1 < c) fn(jj.y, d1);
        if (q + 2 < c) fn(jj.z, d2);
        if (q + 3 < c) fn(jj.w, d3);
        jj = jn;
    }
}

// The value of lane S of each four, and of lane L of each sixteen.  (Every
// lane read from must be active.)
template <int S>
__device__ __forceinline__ uint32_t quad_value(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, S * 0x55, 0xf, 0xf, true);
}
template <int S>
__device__ __forceinline__ float quad_value(float v)
{
    return __uint_as_float(quad_value<S>(__float_as_uint(v)));
}

// The value of lane S of each U lanes (U = 1, 4 or 16).
template <uint32_t U, int S>
__device__ __forceinline__ float group_value(float v)
{
    if constexpr (U == 1)
        return v;
    else if constexpr (U == 4)
        return quad_value<S>(v);
    else
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + S, 0xf, 0xf, true));
}

// Quarter h of particle i's first c neighbours (its chunks h, h + 4, ...) by
// U lanes (1 or 4): fn(record, in use) for entry U s + u of a chunk in
// lane u, s = 0, 1, ..., with D records in flight and the entries after them.
// An entry past the table's end reads particle i's record and is not in use.
// The U lanes make the same calls.  (One lane loading a chunk's four entries
// with one 16-byte load was slower: the reverse kernels took 52, 62 and 70 us
// instead of 48, 54 and 66 at 328k particles.)
template <uint32_t U, uint32_t D, typename G, typename Fn>
__device__ __forceinline__ void for_neighbors_quarter(const DevBuffers &b, uint32_t i, uint32_t c, uint32_t h,
                                                      uint32_t u, G gather, Fn fn)
{
    if (4u * h >= c) return;
    const uint32_t *nb = reinterpret_cast<const uint32_t *>(nbr_lane(b, i));
    constexpr uint32_t kS = 4u / U;  // steps a chunk
    // where step t begins in the table
    auto begin = [&](uint32_t t) { return 4u * (h + 4u * (t / kS)) + U * (t % kS); };
    auto entry = [&](uint32_t t) {
        const uint32_t q = begin(t) + u;
        return q < c ? nb[(size_t)(q >> 2) * 256 + (q & 3u)] : i;
    };
    uint32_t j[D];
#pragma unroll
    for (uint32_t e = 0; e < D; e++) j[e] = entry(e);
    for (uint32_t t = 0; begin(t) < c; t += D) {
        decltype(gather(0u)) d[D];
#pragma unroll
        for (uint32_t e = 0; e < D; e++) d[e] = gather(j[e]);
#pragma unroll
        for (uint32_t e = 0; e < D; e++) j[e] = entry(t + D + e);
#pragma unroll
        for (uint32_t e = 0; e < D; e++)
            if (begin(t + e) < c) fn(d[e], begin(t + e) + u < c);
    }
}

// The entries of half h of particle i's first c neighbours in table order,
// one at a time: for the rarely taken recomputation of one half.
template <typename G, typename Fn>
__device__ __forceinline__ void for_neighbors_half_plain(const DevBuffers &b, uint32_t i, uint32_t c,
                                                         uint32_t h, G gather, Fn fn)
{
    for (uint32_t q0 = 4u * h; q0 < c; q0 += 8u)
        for (uint32_t q = q0; q < q0 + 4u && q < c; q++) {
            const uint32_t j = reinterpret_cast<const uint32_t *>(nbr_lane(b, i) + (size_t)(q >> 2) * 64)[q & 3u];
            fn(j, gather(j));
        }
}

// Both halves in one pass, pipelined as for_neighbors_half: fn0 gets the entries of the
// even chunks (half 0), fn1 those of the odd chunks (half 1), each half in
// table order.  The pipelined loop's two record sets hold an even and an
// odd chunk, so the half of every call is fixed where it is made.
template <typename G, typename Fn0, typename Fn1>
__device__ __forceinline__ void for_neighbors_split(const DevBuffers &b, uint32_t i, uint32_t c, G gather,
                                                    Fn0 fn0, Fn1 fn1)
{
    if (c == 0) return;
    const uint4 *nb = nbr_lane(b, i);
    const uint32_t last = (c - 1) >> 2;
    auto chunk = [&](uint32_t m) { return nb[(size_t)min(m, last) * 64]; };
    auto visit = [&](auto &fn, const uint4 &jj, uint32_t q, const auto &d0, const auto &d1,
                     const auto &d2, const auto &d3) {
        fn(jj.x, d0);
        if (q + 1 < c) fn(jj.y, d1);
        if (q + 2 < c) fn(jj.z, d2);
        if (q + 3 < c) fn(jj.w, d3);
    };
    uint4 ja = nb[0];
    uint4 jb = chunk(1);
    auto a0 = gather(ja.x);
    auto a1 = gather(ja.y);
    auto a2 = gather(ja.z);
    auto a3 = gather(ja.w);
    for (uint32_t m = 0;; m += 2) {
        // a*: chunk m (even), b*: chunk m+1 (odd)
        const uint4 jc = chunk(m + 2);
        auto b0 = gather(jb.x);
        auto b1 = gather(jb.y);
        auto b2 = gather(jb.z);
        auto b3 = gather(jb.w);
        visit(fn0, ja, m << 2, a0, a1, a2, a3);
        if (m + 1 > last) break;
        const uint4 jd = chunk(m + 3);
        a0 = gather(jc.x);
        a1 = gather(jc.y);
        a2 = gather(jc.z);
        a3 = gather(jc.w);
        visit(fn1, jb, (m + 1) << 2, b0, b1, b2, b3);
        if (m + 2 > last) break;
        ja = jc;
        jb = jd;
    }
}

struct PX {
    float4 p, x;
};

// position and neighbour density mass (DevBuffers::mj)
struct PM {
    float4 p;
    float m;
};

// ---------------------------------------------------------------------------
// Pair arithmetic shared with the CPU oracle: squared distances and sums use
// fused multiply-add, and 1/r comes from rsq() instead of sqrt + division
// (an IEEE square root and division cost ~30 VALU per pair, rsq 9).

// |d|^2 = fma(dz, dz, fma(dy, dy, dx dx))
__device__ __forceinline__ float dist2(float dx, float dy, float dz)
{
    return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
}

// 1/sqrt(x), x > 0 normal: integer seed y0 = 0x5f375a86 - (bits(x) >> 1)
// (the "fast inverse square root" constant of C. Lomont, 2003; relative
// error up to 3.4e-2), then one fourth-order correction.  With
// e = 1 - x y0^2, 1/sqrt(x) = y0 (1 - e)^(-1/2) = y0 (1 + e p(e)), p the
// binomial series 1/2 + 3/8 e + 5/16 e^2 + 35/128 e^3 + ..., truncated
// after e^3 and its four coefficients re-fitted minimax over the seed's
// range of e (|e| < 0.07): y = fma(y0 e, p(e), y0), p by Horner in FMA.
// 9 operations; relative error below 1e-7 over [1e-8, 16] (the three
// Newton steps it replaces took 12 for 1.3e-7).
__device__ __forceinline__ float rsq(float x)
{
    const float y0 = __uint_as_float(0x5f375a86u - (__float_as_uint(x) >> 1));
    const float xy = x * y0;
    const float e = __builtin_fmaf(-xy, y0, 1.0f);
    float p = __builtin_fmaf(__uint_as_float(0x3e8c5420u), e, __uint_as_float(0x3ea0bc22u));
    p = __builtin_fmaf(p, e, __uint_as_float(0x3ec0000cu));
    p = __builtin_fmaf(p, e, __uint_as_float(0x3effffc8u));
    return __builtin_fmaf(y0 * e, p, y0);
}

// below this squared distance a pair has no direction
constexpr float kDegenerateR2 = 1e-8f;

// ---------------------------------------------------------------------------
// helpers of the solve kernel

__device__ __forceinline__ uint64_t mix64(uint64_t z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// Wall-jitter uniform in [0,1): SplitMix64 finaliser of seed + golden*counter,
// counter = (iteration, insertion index, wall), top 24 bits.
__device__ __forceinline__ float wall_uniform(uint64_t seed, uint64_t iter, uint32_t orig,
                                              uint32_t wall)
{
    uint64_t ctr = (iter << 35) | ((uint64_t)orig << 3) | (uint64_t)wall;
    uint64_t z = mix64(seed + ctr * 0x9E3779B97F4A7C15ull);
    return (float)(uint32_t)(z >> 40) * (1.0f / 16777216.0f);
}

// e^x: Cody-Waite reduction x = k ln2 + r, degree-7 Taylor polynomial of
// e^r (Horner), exact scaling by 2^k.
__device__ __forceinline__ float ps_exp(float x)
{
    if (x > 80.0f) x = 80.0f;
    if (x < -80.0f) x = -80.0f;
    float kk = floorf((x * 1.44269504088896341f) + 0.5f);
    float r = (x - (kk * 0.693145751953125f)) - (kk * 1.42860682030941723e-6f);
    float p = 1.98412698412698413e-4f;
    p = (p * r) + 1.38888888888888889e-3f;
    p = (p * r) + 8.33333333333333333e-3f;
    p = (p * r) + 4.16666666666666667e-2f;
    p = (p * r) + 1.66666666666666667e-1f;
    p = (p * r) + 0.5f;
    p = (p * r) + 1.0f;
    p = (p * r) + 1.0f;
    return ldexpf(p, (int)kk);
}

__device__ __forceinline__ float ipow(float x, uint32_t n)
{
    float r = 1.0f, bb = x;
    bool first = true;
    while (n) {
        if (n & 1u) {
            r = first ? bb : (r * bb);
            first = false;
        }
        n >>= 1;
        if (n) bb = bb * bb;
    }
    return r;
}

// a8: world box (collide_world_functor, integration_kernel.cuh:57-157).
struct WallBox {
    float lo[3], hi[3];
    uint64_t seed;
    uint32_t o;  // index of the particle inside its scene
};

__device__ __forceinline__ WallBox wall_box(const KConst &k, const DevBuffers &b, uint32_t i,
                                            uint32_t orig)
{
    WallBox w;
    if (k.nscenes > 1u) {
        const SceneDev &sc = b.scenes[b.sid[i]];
        for (int a = 0; a < 3; a++) {
            w.lo[a] = sc.box_min[a];
            w.hi[a] = sc.box_max[a];
        }
        w.seed = sc.seed;
        w.o = orig - sc.first;
    } else {
        for (int a = 0; a < 3; a++) {
            w.lo[a] = k.box_min[a];
            w.hi[a] = k.box_max[a];
        }
        w.seed = k.seed;
        w.o = orig;
    }
    return w;
}

// Returns what it did, for the adjoint: bits 0-2 the coordinates a wall
// set, bit 3 wall friction acted, bit 4 the kinetic branch with f < 1 (the
// solve kernel adds bit 5 for a pin, with bits 0-2).  When friction acts,
// rec = (position before friction, (n_x+1)*9 + (n_y+1)*3 + (n_z+1)).
constexpr uint32_t kWallFriction = 8u, kWallKinetic = 16u, kPinned = 32u;

__device__ __forceinline__ uint32_t walls(const KConst &k, const WallBox &wb, int32_t ph, float4 xs,
                                          float &px, float &py, float &pz, uint64_t iter, float4 &rec)
{
    uint32_t set = 0u;
    const float r = k.radius;
    const uint32_t o = wb.o;
    float nx = 0.0f, ny = 0.0f, nz = 0.0f;
    const float efl = ph < PS_PHASE_SOLID ? k.jitter : 0.0f;
    if (py < wb.lo[1] + r) {
        py = (wb.lo[1] + r) + (wall_uniform(wb.seed, iter, o, 5) * efl);
        set |= 2u;
        ny = ny + 1.0f;
    }
    if (px > wb.hi[0] - r) {
        px = wb.hi[0] - (r + (wall_uniform(wb.seed, iter, o, 0) * k.jitter));
        set |= 1u;
        nx = nx - 1.0f;
    }
    if (px < wb.lo[0] + r) {
        px = wb.lo[0] + (r + (wall_uniform(wb.seed, iter, o, 1) * k.jitter));
        set |= 1u;
        nx = nx + 1.0f;
    }
    if (py > wb.hi[1] - r) {
        py = wb.hi[1] - (r + (wall_uniform(wb.seed, iter, o, 2) * k.jitter));
        set |= 2u;
        ny = ny - 1.0f;
    }
    if (k.dims != 2u) {
        if (pz > wb.hi[2] - r) {
            pz = wb.hi[2] - (r + (wall_uniform(wb.seed, iter, o, 3) * k.jitter));
            set |= 4u;
            nz = nz - 1.0f;
        }
        if (pz < wb.lo[2] + r) {
            pz = wb.lo[2] + (r + (wall_uniform(wb.seed, iter, o, 4) * k.jitter));
            set |= 4u;
            nz = nz + 1.0f;
        }
    }
    if (ph < PS_PHASE_CLOTH) return set;
    if (nx == 0.0f && ny == 0.0f && nz == 0.0f) return set;
    float ex = px - xs.x, ey = py - xs.y, ez = pz - xs.z;
    float dn = ((ex * nx) + (ey * ny)) + (ez * nz);
    float tx = ex - (dn * nx), ty = ey - (dn * ny), tz = ez - (dn * nz);
    float l = sqrtf(((tx * tx) + (ty * ty)) + (tz * tz));
    if (l < 0.001f) return set;
    set |= kWallFriction;
    rec = make_float4(px, py, pz,
                      (float)((((int)nx + 1) * 9 + ((int)ny + 1) * 3) + ((int)nz + 1)));
    if (l < k.wall_s) {
        px = px - tx;
        py = py - ty;
        pz = pz - tz;
    } else {
        float f = k.wall_k / l;
        if (f > 1.0f)
            f = 1.0f;
        else
            set |= kWallKinetic;
        px = px - (tx * f);
        py = py - (ty * f);
        pz = pz - (tz * f);
    }
    return set;
}

}  // namespace ps
