// ps_kernels.hip — gfx950 kernels of the particle-solver substep.
//
// Layout: every per-particle array is in cell-sorted storage order; a
// particle's insertion index travels in Attr::orig.  Positions and the PBF
// multiplier share one float4 (x, y, z, lambda), so each neighbour visit in
// the lambda and delta-p kernels is a single 16-byte gather.  The neighbour
// table is a sliced ELL in chunks of four: for each group of 64 consecutive
// particles, entries 4m..4m+3 of every lane form one uint4, and the 64 lanes'
// uint4s are contiguous, so a wavefront reads four neighbour indices per lane
// with one coalesced 1-KiB load.  A unit staged in LDS holds 16-bit LDS
// indices instead, eight to a uint4 (nbr16_chunk): the table is read nine
// times a substep, and with 32-bit entries it was most of the traffic of the
// kernels that read it.
//
// Arithmetic: built with -ffp-contract=off and IEEE division/sqrt, and every
// expression is parenthesised as in the CPU oracle, so FP32 results are
// reproducible operation by operation.  Accumulations run over the neighbour
// table in ascending slot order; no floating-point atomics anywhere.
//
// Launch mapping: blocks of the neighbour-gathering kernels are remapped so
// that each of the 8 XCDs (which receive workgroups round-robin) owns one
// contiguous range of sorted particles, keeping a spatial region's
// neighbour data inside one XCD's L2.

#include "ps_blocks.hpp"
#include "ps_device.hpp"

namespace ps {

static constexpr uint32_t kBlock = 256;     // fixed-shape kernels (scan, scatter, shape)
static constexpr uint32_t kMaxBlock = 512;  // tunable kernels run with 64..512 threads
static constexpr uint32_t kScanPerThread = 16;
static constexpr uint32_t kScanTile = kBlock * kScanPerThread;
static_assert(kScanTile == kScanTileCells, "scan tile size");


__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t t = __shfl_up(v, d, 64);
        if (lane >= d) v += t;
    }
    return v;
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v)
{
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v)
{
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        uint32_t t = __shfl_xor(v, d, 64);
        v = t > v ? t : v;
    }
    return v;
}


// ---------------------------------------------------------------------------
// a1 + a2: predict (integrate_functor, integration_kernel.cuh:159-184) and
// cell hash (calcGridPos/calcGridHash/calcHashD :187-225) with a dense,
// clamped grid.  The atomic's return value is the particle's arrival rank in
// its cell, used only to place it provisionally; the final in-cell order is
// fixed by insertion index in reorder_k.

template <bool PRED, bool HASH>
__global__ __launch_bounds__(kMaxBlock) void predict_hash_k(DevBuffers b, KConst k, uint32_t n,
                                                         float dt)
{
    const uint32_t s = xcd_block() * blockDim.x + threadIdx.x;
    const bool valid = s < n;
    const bool multi = k.nscenes > 1u;
    const SceneDev *sc = (multi && valid) ? &b.scenes[b.sid[s]] : nullptr;
    float px = 0.0f, py = 0.0f, pz = 0.0f;
    if (valid) {
        if (PRED) {
            // the three loads go out together (a static particle's velocity
            // is read and not used)
            const float4 x = b.X[s];
            const Attr a = b.A[s];
            const float4 v = b.V[s];
            px = x.x;
            py = x.y;
            pz = x.z;
            if (a.w != 0.0f) {
                const float gx = multi ? sc->gravity[0] : k.gravity[0];
                const float gy = multi ? sc->gravity[1] : k.gravity[1];
                const float gz = multi ? sc->gravity[2] : k.gravity[2];
                float vx = v.x + (gx * dt);
                float vy = v.y + (gy * dt);
                float vz = v.z + (gz * dt);
                px = x.x + (vx * dt);
                py = x.y + (vy * dt);
                pz = k.dims == 2u ? x.z : (x.z + (vz * dt));
            }
            b.P[s] = make_float4(px, py, pz, 0.0f);
        } else {
            const float4 p = b.P[s];
            px = p.x;
            py = p.y;
            pz = p.z;
        }
    }
    if (HASH) {
        uint32_t flags = 0, key = 0xffffffffu;
        if (valid) {
            if (multi) {
                uint32_t cx = cell_axis(px, sc->origin[0], k.cell, sc->grid[0], flags);
                uint32_t cy = cell_axis(py, sc->origin[1], k.cell, sc->grid[1], flags);
                uint32_t cz = cell_axis(pz, sc->origin[2], k.cell, sc->grid[2], flags);
                key = sc->cell_base + (cz * sc->grid[1] + cy) * sc->grid[0] + cx;
            } else {
                uint32_t cx = cell_axis(px, k.origin[0], k.cell, k.grid[0], flags);
                uint32_t cy = cell_axis(py, k.origin[1], k.cell, k.grid[1], flags);
                uint32_t cz = cell_axis(pz, k.origin[2], k.cell, k.grid[2], flags);
                key = (cz * k.grid[1] + cy) * k.grid[0] + cx;
            }
        }
        // Storage is in last substep's cell order, so equal keys sit in runs
        // of adjacent lanes: one atomic per run hands out the run's ranks.
        const uint32_t lane = threadIdx.x & 63u;
        const uint32_t prev = __shfl_up(key, 1, 64);
        const bool head = valid && (lane == 0 || key != prev);
        const uint64_t heads = __ballot(head);
        const uint64_t upto = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);
        const uint64_t mine = heads & upto;
        const uint32_t seg = mine ? 63u - (uint32_t)__clzll((unsigned long long)mine) : lane;
        const uint64_t later = heads & ~upto;
        const uint64_t vmask = __ballot(valid);
        const uint32_t vend = vmask == ~0ull ? 64u : (uint32_t)__ffsll((unsigned long long)~vmask) - 1u;
        const uint32_t next = later ? (uint32_t)__ffsll((unsigned long long)later) - 1u : vend;
        uint32_t base = 0;
        if (head) base = atomicAdd(&b.cell_count[key], next - seg);
        base = __shfl(base, seg, 64);
        if (valid) {
            b.key[s] = key;
            b.rank[s] = base + (lane - seg);
        }
        // status bits: one atomic per wavefront, not per particle (a splash
        // can put thousands of predictions outside the grid at once), and
        // none once the bits are set (atomics on one address serialise)
        const uint64_t nf = __ballot((flags & PS_STATUS_NONFINITE) != 0u);
        const uint64_t og = __ballot((flags & PS_STATUS_OUTSIDE_GRID) != 0u);
        if (lane == 0 && (nf | og)) {
            const uint32_t want = (nf ? PS_STATUS_NONFINITE : 0u) | (og ? PS_STATUS_OUTSIDE_GRID : 0u);
            if ((status_peek(&b.status->flags) & want) != want) atomicOr(&b.status->flags, want);
        }
    }
}

// ---------------------------------------------------------------------------
// a4 part 1: exclusive scan of the per-cell counts into cell offsets
// (cell c = sorted slots [off[c], off[c+1]); the reference's cellStart/End,
// reorderDataAndFindCellStartD integration_kernel.cuh:229-299), over tiles of
// 4096 cells, a block of 1024 threads each.  A block needs the sum of the
// tiles before its own: of few tiles it adds up the counts themselves, of
// more it reads their sums, which scan_partials_k forms before.  The counts
// stay (a block may still read them): the scatter clears those it finds.

__global__ __launch_bounds__(kBlock) void scan_partials_k(const uint32_t *cnt, uint32_t *part,
                                                          uint32_t C)
{
    __shared__ uint32_t lds4[4];
    const uint32_t base = blockIdx.x * kScanTile;
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t q = 0; q < kScanPerThread; q++) {
        uint32_t c = base + q * kBlock + threadIdx.x;
        if (c < C) sum += cnt[c];
    }
    sum = wave_sum(sum);
    if ((threadIdx.x & 63u) == 0) lds4[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = lds4[0] + lds4[1] + lds4[2] + lds4[3];
}

// The tiles up to which the sums are formed from the counts: the last of 32
// blocks reads 32 tiles of 16 KB from the L2, eight loads in flight, which
// costs less than a launch: one tile 1.7 us (two launches of 256 threads: 6.7),
// 8 tiles 5.3 (10.7), 25 tiles 7.4 (9.6).  With 256 tiles the second launch
// is 5.0 us (6.1 with 256 threads, 16 cells each, through LDS).
static constexpr uint32_t kScanDirect = 32;

template <bool DIRECT>
__global__ __launch_bounds__(kScanTile / 4) void scan_k(const uint32_t *cnt, const uint32_t *part, uint32_t *off,
                                                        uint32_t C)
{
    constexpr uint32_t kThreads = kScanTile / 4, kWaves = kThreads / 64;
    __shared__ uint32_t wtot[kWaves], ptot[kWaves];
    const uint32_t tid = threadIdx.x, w = tid >> 6;
    const uint32_t c = blockIdx.x * kScanTile + 4u * tid;
    const bool whole = c < C && C - c >= 4u;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (whole) {
        v = *reinterpret_cast<const uint4 *>(cnt + c);
    } else if (c < C) {
        v.x = cnt[c];
        if (C - c > 1u) v.y = cnt[c + 1];
        if (C - c > 2u) v.z = cnt[c + 2];
    }
    uint32_t pre = 0;
    if (DIRECT) {
#pragma unroll 8
        for (uint32_t t = 0; t < blockIdx.x; t++) {
            const uint4 u = *reinterpret_cast<const uint4 *>(cnt + t * kScanTile + 4u * tid);
            pre += (u.x + u.y) + (u.z + u.w);
        }
    } else {
        for (uint32_t t = tid; t < blockIdx.x; t += kThreads) pre += part[t];
    }
    const uint32_t local = (v.x + v.y) + (v.z + v.w);
    const uint32_t incl = wave_incl_scan(local);
    pre = wave_sum(pre);
    if ((tid & 63u) == 63u) {
        wtot[w] = incl;
        ptot[w] = pre;
    }
    __syncthreads();
    uint32_t run = incl - local;
#pragma unroll
    for (uint32_t q = 0; q < kWaves; q++) run += ptot[q] + (q < w ? wtot[q] : 0u);
    const uint4 o = make_uint4(run, run + v.x, run + v.x + v.y, run + v.x + v.y + v.z);
    if (whole) {
        *reinterpret_cast<uint4 *>(off + c) = o;
    } else if (c < C) {
        off[c] = o.x;
        if (C - c > 1u) off[c + 1] = o.y;
        if (C - c > 2u) off[c + 2] = o.z;
    }
    if (blockIdx.x == gridDim.x - 1 && tid == kThreads - 1) off[C] = run + local;
}

// a4 part 2: provisional placement by arrival rank (insertion indices only).
// The counts are cleared for the next build here, where nothing reads them:
// by the first particle of each run of equal keys in a wavefront.
__global__ __launch_bounds__(kBlock) void scatter_k(DevBuffers b, uint32_t n)
{
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= n) return;
    const uint32_t key = b.key[s];
    const uint32_t prev = __shfl_up(key, 1, 64);
    if ((threadIdx.x & 63u) == 0u || key != prev) b.cell_count[key] = 0;
    const uint32_t t = b.cell_off[key] + b.rank[s];
    if (t < n)
        b.tmp_orig[t] = b.A[s].orig;
    else
        atomicOr(&b.status->flags, PS_STATUS_INTERNAL);
}

// a3 + a4 part 3: final slot = cell start + number of particles in the same
// cell with a smaller insertion index, i.e. a sort by (cell, insertion
// index): a stable sort of insertion-ordered input, as thrust::sort_by_key
// of (hash, index) in sortParticles (integration.cu:270-275) is meant to
// give.  Every per-particle array moves with the particle.
// mj_solid >= 0: also write mj (the neighbour density mass) with s_solid =
// mj_solid, and the particle's marks.
__global__ __launch_bounds__(kMaxBlock) void reorder_k(DevBuffers b, uint32_t n, float mj_solid)
{
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t c = b.key[s];
    const Attr a = b.A[s];
    // the particle's own records go in flight before the count
    const float4 p = b.P[s], xs = b.X[s], vs = b.V[s];
    const uint32_t b0 = b.cell_off[c], b1 = b.cell_off[c + 1];
    if (b1 > n || b0 >= b1 || a.orig >= n) {
        atomicOr(&b.status->flags, PS_STATUS_INTERNAL);
        return;
    }
    // the count in groups of four independent loads (one wait per group
    // instead of one per member)
    uint32_t r = 0;
    for (uint32_t u = b0; u < b1; u += 4) {
        uint32_t t[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) t[k] = b.tmp_orig[min(u + k, b1 - 1u)];
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) r += (u + k < b1 && t[k] < a.orig) ? 1u : 0u;
    }
    const uint32_t d = b0 + r;
    // scenes that are not a uniform fluid: x*.w carries the particle's XSPH
    // mass as a neighbour, 1/w for a fluid particle, -1 for any other
    b.X2[d] = mj_solid >= 0.0f
                  ? make_float4(xs.x, xs.y, xs.z, a.phase == PS_PHASE_FLUID ? 1.0f / a.w : -1.0f)
                  : xs;
    b.Q[d] = make_float4(p.x, p.y, p.z, 0.0f);
    b.V2[d] = vs;
    b.A2[d] = a;
    b.key2[d] = c;
    if (mj_solid >= 0.0f) {
        // the neighbour mass of the fluid sums, as they form it per pair
        float m = -1.0f;
        if (a.w != 0.0f) {
            m = 1.0f / a.w;
            if (a.phase != PS_PHASE_FLUID) m = m * mj_solid;
        }
        b.mj[d] = m;
        // the phase as the contact walk reads it
        b.phs[d] = a.w != 0.0f ? a.phase : (int32_t)((uint32_t)a.phase | 0x80000000u);
        // where the constraint blocks find it
        const uint8_t mark = b.omark[a.orig];
        b.smark[d] = mark;
        if (a.phase >= PS_PHASE_CLOTH && a.w != 0.0f) b.walk_slot[b.walk_rank[a.orig]] = d;
        if (mark & kMarkDist) b.link_slot[b.link_rank[a.orig]] = d;
    }
    if (b.sid) b.sid2[d] = b.sid[s];
    // a scatter by insertion index: skipped when no kernel reads it
    if (b.track_slots) b.slot_of[a.orig] = d;
    // recording for the reverse pass: the same records into the tape slot
    if (b.tape_x) {
        b.tape_x[d] = xs;
        b.tape_a[d] = a;
        if (b.track_slots) b.tape_s[a.orig] = d;
    }
}


// ---------------------------------------------------------------------------
// Neighbour table (collideCell/collideCellRadius, integration_kernel.cuh:
// 303-356,481-518): every j != i with r^2 < search_r2, scanning the 3x3 rows
// of x-adjacent cells; a row's three cells are one contiguous slot range.

// Scan the nine stencil rows of particle i in order (t = (dz+1)*3 + dy+1)
// and write its table of global slots: every slot j != i of range(t) =
// [j0, j1) with |p - P[j]|^2 < search_r2, in ascending j; i's own slot fills
// the last chunk.  Returns the number found (the table keeps the first kmax).
// A row is tested in windows of 32 candidates without branches: each test
// sets one bit of a mask (i's own bit is cleared), and the set bits are then
// emitted lowest first, so the entries come out in ascending j as from a
// plain loop over the row, and only accepted candidates pay for the table.
// p is taken by value: a reference into b.P would be re-read after every
// table store (the compiler cannot rule out aliasing).
template <typename Range>
__device__ __forceinline__ uint32_t scan_stencil(const DevBuffers &b, const KConst &k, uint32_t i, const float4 p,
                                                 uint32_t kmax, Range range)
{
    uint4 *out = const_cast<uint4 *>(nbr_lane(b, i));
    uint4 buf = make_uint4(i, i, i, i);
    uint32_t cnt = 0;
    const float r2max = k.search_r2;
    // an accepted candidate: shifted into buf, which after the 4th entry of
    // a chunk holds it in order (x first); chunks past kmax are not stored
    auto accept = [&](uint32_t j) {
        buf.x = buf.y;
        buf.y = buf.z;
        buf.z = buf.w;
        buf.w = j;
        if ((cnt & 3u) == 3u && cnt < kmax) out[(size_t)(cnt >> 2) * 64] = buf;
        cnt++;
    };
    for (uint32_t t = 0; t < 9; t++) {
        uint32_t j0 = 0, j1 = 0;
        if (!range(t, j0, j1)) continue;
        const float4 *q0 = b.P + j0;
        for (uint32_t w0 = j0; w0 < j1; w0 += 32u) {
            const uint32_t we = min(w0 + 32u, j1);
            uint32_t m = 0;
            uint32_t jb = w0;
            // whole groups of four: no bound test; the loads go ahead of
            // the tests
            for (; jb + 4u <= we; jb += 4u) {
                // one address per group, immediate offsets for the four
                float4 qv[4];
#pragma unroll
                for (uint32_t u = 0; u < 4; u++) qv[u] = q0[jb - j0 + u];
                uint32_t g = 0;
#pragma unroll
                for (uint32_t u = 0; u < 4; u++)
                    g |= (dist2(p.x - qv[u].x, p.y - qv[u].y, p.z - qv[u].z) < r2max ? 1u : 0u) << u;
                m |= g << (jb - w0);
            }
            // the last one to three
            if (jb < we) {
                float4 qv[3];
#pragma unroll
                for (uint32_t u = 0; u < 3; u++) qv[u] = q0[min(jb + u, we - 1u) - j0];
                uint32_t g = 0;
#pragma unroll
                for (uint32_t u = 0; u < 3; u++)
                    g |= (jb + u < we && dist2(p.x - qv[u].x, p.y - qv[u].y, p.z - qv[u].z) < r2max
                              ? 1u : 0u) << u;
                m |= g << (jb - w0);
            }
            // i itself (in its own row only)
            if (i - w0 < 32u) m &= ~(1u << (i - w0));
            while (m != 0u) {
                const uint32_t u = (uint32_t)__builtin_ctz(m);
                m &= m - 1u;
                accept(w0 + u);
            }
        }
    }
    const uint32_t kept = cnt < kmax ? cnt : kmax;
    // a partial last chunk: its r entries sit at the right end of buf
    const uint32_t r = kept & 3u;
    if (r == 1u) out[(size_t)(kept >> 2) * 64] = make_uint4(buf.w, i, i, i);
    else if (r == 2u) out[(size_t)(kept >> 2) * 64] = make_uint4(buf.z, buf.w, i, i);
    else if (r == 3u) out[(size_t)(kept >> 2) * 64] = make_uint4(buf.y, buf.z, buf.w, i);
    b.ncnt[i] = kept;
    return cnt;
}

// one status update per block: max count and overflow
__device__ __forceinline__ void neighbor_status(const DevBuffers &b, uint32_t cnt, uint32_t kmax,
                                                uint32_t *ldsw)
{
    uint32_t m = wave_max(cnt);
    const uint32_t w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) ldsw[w] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t mm = ldsw[0];
        for (uint32_t q = 1; q < (blockDim.x >> 6); q++) mm = ldsw[q] > mm ? ldsw[q] : mm;
        // one address for every block: skip the atomics that change nothing
        if (mm > 0 && mm > status_peek(&b.status->max_neighbors)) atomicMax(&b.status->max_neighbors, mm);
        if (mm > kmax && !(status_peek(&b.status->flags) & PS_STATUS_NEIGHBOR_OVERFLOW))
            atomicOr(&b.status->flags, (uint32_t)PS_STATUS_NEIGHBOR_OVERFLOW);
    }
}

__global__ __launch_bounds__(kMaxBlock) void neighbors_k(DevBuffers b, KConst k, uint32_t n,
                                                      uint32_t kmax)
{
    __shared__ uint32_t ldsw[kMaxBlock / 64];
    const uint32_t i = xcd_block() * blockDim.x + threadIdx.x;
    uint32_t cnt = 0;
    if (i < n) {
        uint32_t gx = k.grid[0], gy = k.grid[1], gz = k.grid[2], base = 0;
        if (k.nscenes > 1u) {
            const SceneDev &sc = b.scenes[b.sid[i]];
            gx = sc.grid[0];
            gy = sc.grid[1];
            gz = sc.grid[2];
            base = sc.cell_base;
        }
        const uint32_t key = b.key[i] - base;
        const uint32_t cx = key % gx, cy = (key / gx) % gy, cz = key / (gx * gy);
        const uint32_t x0 = cx > 0 ? cx - 1 : 0, x1 = cx + 1 < gx ? cx + 1 : gx - 1;
        auto range = [&](uint32_t t, uint32_t &j0, uint32_t &j1) {
            const int z = (int)cz + (int)(t / 3) - 1, y = (int)cy + (int)(t % 3) - 1;
            if (z < 0 || z >= (int)gz || y < 0 || y >= (int)gy) return false;
            const uint32_t row = base + ((uint32_t)z * gy + (uint32_t)y) * gx;
            j0 = b.cell_off[row + x0];
            j1 = min(b.cell_off[row + x1 + 1], n);
            return j0 < j1;
        };
        cnt = scan_stencil(b, k, i, b.P[i], kmax, range);
    }
    neighbor_status(b, cnt, kmax, ldsw);
}

// A staged unit's chunk sources for one thread: with THREADS threads, thread
// t handles element t % 16 of chunks c = (THREADS/16) k + t / 16.  load() is
// called before the descriptor's header is known (an unused chunk's source
// is whatever is there, and is not used), so that the sources, the header
// and the particle's own records wait together.
template <uint32_t THREADS>
struct StageSrc {
    static_assert(THREADS % kStageChunk == 0 && kStageChunks % (THREADS / kStageChunk) == 0,
                  "whole chunks per step");
    static constexpr uint32_t kPerStep = THREADS / kStageChunk;  // chunks per step
    static constexpr uint32_t kSteps = kStageChunks / kPerStep;
    uint32_t src[kSteps];

    __device__ __forceinline__ void load(const StageDesc *d)
    {
        const uint32_t c0 = threadIdx.x / kStageChunk;
#pragma unroll
        for (uint32_t k = 0; k < kSteps; k++) src[k] = d->src[k * kPerStep + c0];
    }
};

// Copy a staged unit's chunks of the current data into LDS, BATCH chunks'
// loads in flight at a time; a chunk's elements past its interval read a
// clamped slot and fill padding that no table entry refers to.  load(j)
// reads slot j, store(l, v) writes LDS index l.  Every thread of the block
// calls it.
template <uint32_t BATCH, uint32_t THREADS, typename Load, typename Store>
__device__ __forceinline__ void stage_copy(const StageSrc<THREADS> &ss, uint32_t nch, uint32_t n, Load load,
                                           Store store)
{
    constexpr uint32_t kPerStep = StageSrc<THREADS>::kPerStep, kSteps = StageSrc<THREADS>::kSteps;
    static_assert(kSteps % BATCH == 0, "whole batches");
    const uint32_t sub = threadIdx.x % kStageChunk, c0 = threadIdx.x / kStageChunk;
#pragma unroll
    for (uint32_t k0 = 0; k0 < kSteps; k0 += BATCH) {
        if (k0 * kPerStep >= nch) break;
        decltype(load(0u)) v[BATCH];
#pragma unroll
        for (uint32_t k = 0; k < BATCH; k++) {
            const uint32_t c = (k0 + k) * kPerStep + c0;
            v[k] = load(c < nch ? min(ss.src[k0 + k] + sub, n - 1u) : 0u);
        }
#pragma unroll
        for (uint32_t k = 0; k < BATCH; k++) {
            const uint32_t c = (k0 + k) * kPerStep + c0;
            if (c < nch) store(c * kStageChunk + sub, v[k]);
        }
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// The staged build.  A unit's plan: its intervals (kStageRows), their union as
// slot segments laid out in LDS, and the chunk table from which the kernels
// that stage the unit copy it; a unit spanning more rows or slots than they
// allow, or two scenes of a batch, keeps global slots (staged = 0).  Then the
// search, in one of two forms.
// The union is what a unit of several rows needs: the stencils of adjacent
// rows share two of three target rows.  With three rows a unit and every
// interval laid out apart, 79 % of the units of a 128-scene ensemble (2.55 M
// particles) staged, with seven merged rows 94 %: lambda 147 -> 118 us, the
// solve 202 -> 187, finalize 185 -> 140 a launch.  The plan is the first
// wavefront's work (on all four it cost the build 10 us at 1,048,576
// particles).

struct UnitPlan {  // in LDS
    uint32_t wfirst[4], wlast[4], wheads[4], total;
    uint32_t rrow[kStageRows], xa[kStageRows], xb[kStageRows];
    uint32_t st[kStageIv], en[kStageIv], delta[kStageIv];  // per interval
    uint32_t src[kStageChunks];
    uint8_t q[kStageUnit];  // unit row of each particle
};
static_assert(kStageIv <= 64, "one lane of a wavefront plans each interval");

// the grid a particle's key refers to: its scene's in a batch
struct GridOf {
    uint32_t gx, gy, gz, base;
};
__device__ __forceinline__ GridOf grid_of(const DevBuffers &b, const KConst &k, uint32_t sid)
{
    if (k.nscenes > 1u) {
        const SceneDev &sc = b.scenes[sid];
        return GridOf{sc.grid[0], sc.grid[1], sc.grid[2], sc.cell_base};
    }
    return GridOf{k.grid[0], k.grid[1], k.grid[2], 0u};
}

// inclusive scan over the wavefront
template <typename Op>
__device__ __forceinline__ uint32_t wave_scan(uint32_t v, Op op)
{
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(v, d, 64);
        if (lane >= (uint32_t)d) v = op(v, t);
    }
    return v;
}

__device__ __forceinline__ uint32_t lane_u(uint32_t v, uint32_t l)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}

struct Planned {
    bool staged;
    uint32_t nch;
    GridOf gr;          // of the thread's particle (tid of the unit)
    uint32_t row, x;    // its cell: row = z gy + y
};

// kStageUnit threads, thread tid planning particle first + tid (nu of them)
__device__ __forceinline__ Planned plan_unit(const DevBuffers &b, const KConst &k, uint32_t n, uint32_t first,
                                             uint32_t nu, UnitPlan &L)
{
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const bool pv = tid < nu;
    const uint32_t ui = first + tid;
    const bool multi = k.nscenes > 1u;
    uint32_t sid = 0;
    bool one_scene = true;
    if (multi) {
        const uint32_t su = b.sid[first];
        one_scene = b.sid[first + nu - 1u] == su;
        sid = pv ? b.sid[ui] : su;
    }
    Planned r;
    r.gr = grid_of(b, k, sid);
    const GridOf gr = r.gr;
    const uint32_t key = pv ? b.key[ui] - gr.base : 0u;
    const uint32_t row = key / gr.gx, x = key % gr.gx;
    r.row = row;
    r.x = x;
    if (lane == 0u) L.wfirst[w] = row;
    if (lane == 63u) L.wlast[w] = row;
    __syncthreads();
    uint32_t prev = __shfl_up(row, 1, 64), next = __shfl_down(row, 1, 64);
    if (lane == 0u && w > 0u) prev = L.wlast[w - 1u];
    if (lane == 63u && w < 3u) next = L.wfirst[w + 1u];
    const bool head = pv && (tid == 0u || row != prev);
    const bool tail = pv && (tid + 1u == nu || row != next);
    const uint64_t hm = __ballot(head);
    if (lane == 0u) L.wheads[w] = (uint32_t)__popcll(hm);
    __syncthreads();
    uint32_t before = 0, nrows = 0;
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) {
        before += q < w ? L.wheads[q] : 0u;
        nrows += L.wheads[q];
    }
    const bool planned = one_scene && nrows <= kStageRows;
    if (planned && pv) {
        const uint64_t upto = lane == 63u ? ~0ull : ((2ull << lane) - 1ull);
        const uint32_t q = before + (uint32_t)__popcll(hm & upto) - 1u;  // this particle's row
        L.q[tid] = (uint8_t)q;
        if (head) {
            L.rrow[q] = row;
            L.xa[q] = x;  // keys ascend: the row's first particle has its lowest x
        }
        if (tail) L.xb[q] = x;
    }
    __syncthreads();
    // The rest is the first wavefront's (the others wait): lane 9q + t takes
    // the interval of target row t of unit row q.
    if (w == 0u) {
        const uint32_t niv = planned ? 9u * nrows : 0u;
        uint32_t st = 0, en = 0;
        if (lane < niv) {
            const uint32_t qq = lane / 9u, t = lane % 9u;
            const uint32_t rr = L.rrow[qq], ry = rr % gr.gy, rz = rr / gr.gy;
            const int z = (int)rz + (int)(t / 3u) - 1, y = (int)ry + (int)(t % 3u) - 1;
            if (z >= 0 && z < (int)gr.gz && y >= 0 && y < (int)gr.gy) {
                const uint32_t r2 = gr.base + ((uint32_t)z * gr.gy + (uint32_t)y) * gr.gx;
                const uint32_t xa = L.xa[qq], xb = L.xb[qq];
                st = b.cell_off[r2 + (xa > 0u ? xa - 1u : 0u)];
                en = min(b.cell_off[r2 + (xb + 1u < gr.gx ? xb + 1u : gr.gx - 1u) + 1u], n);
            }
            if (en <= st) st = en = 0xffffffffu;  // empty: behind all others
            L.st[lane] = st;
            L.en[lane] = en;
        } else {
            st = en = 0xffffffffu;
        }
        // in order of their start: lane l of ost, oen is the l-th interval
        uint32_t rank = 0;
        for (uint32_t q = 0; q < niv; q++) {
            const uint32_t a = lane_u(st, q);
            rank += (a < st || (a == st && q < lane)) ? 1u : 0u;
        }
        if (lane >= niv) rank = lane;
        const uint32_t ost = (uint32_t)__builtin_amdgcn_ds_permute((int)(rank << 2), (int)st);
        const uint32_t oen = (uint32_t)__builtin_amdgcn_ds_permute((int)(rank << 2), (int)en);
        const bool have = ost != 0xffffffffu;
        const uint32_t m = (uint32_t)__popcll(__ballot(have));  // a prefix of the lanes
        // Their union: an interval that starts past the end of all before it
        // starts a segment.  A segment's LDS base is the sum of the padded
        // lengths of those before, each taken by the next one's head.
        auto mx = [](uint32_t a, uint32_t c) { return a > c ? a : c; };
        auto add = [](uint32_t a, uint32_t c) { return a + c; };
        auto pad = [](uint32_t len) { return (len + kStageChunk - 1u) / kStageChunk * kStageChunk; };
        const uint32_t emax = wave_scan(have ? oen : 0u, mx);
        const uint32_t ebefore = __shfl_up(emax, 1, 64);  // end of all before
        const bool shead = have && (lane == 0u || ost > ebefore);
        const uint32_t shst = wave_scan(shead ? ost : 0u, mx);  // start of the interval's segment
        const uint32_t sbefore = __shfl_up(shst, 1, 64);
        const uint32_t plen = shead && lane > 0u ? pad(ebefore - sbefore) : 0u;
        const uint32_t base = wave_scan(plen, add);
        const uint32_t mylast = pad(emax - shst);
        // LDS index = slot + delta, back in interval order
        const uint32_t dl = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(rank << 2), (int)(base - shst));
        if (lane < niv) L.delta[lane] = dl;
        const uint32_t total = m ? lane_u(base + mylast, m - 1u) : 0xffffffffu;
        if (lane == 0u) L.total = total;
        if (total <= kStageSlots) {
            // chunk table: a segment's chunks by the next one's head, the
            // last's by the last interval
            for (uint32_t c = 0; c < plen; c += kStageChunk) L.src[(base - plen + c) / kStageChunk] = sbefore + c;
            if (lane == m - 1u)
                for (uint32_t c = 0; c < mylast; c += kStageChunk) L.src[(base + c) / kStageChunk] = shst + c;
        }
    }
    __syncthreads();
    r.staged = planned && L.total <= kStageSlots;
    r.nch = r.staged ? L.total / kStageChunk : 0u;
    return r;
}

// the descriptor the other staged kernels of this substep read
__device__ __forceinline__ void put_desc(StageDesc *desc, const Planned &pl, const UnitPlan &L)
{
    const uint32_t tid = threadIdx.x;
    if (tid == 0u) {
        desc->staged = pl.staged ? 1u : 0u;
        desc->nchunks = pl.nch;
    }
    if (tid < pl.nch) desc->src[tid] = L.src[tid];
}

// (m << 1) | (a < b): the compare's carry shifted in, false for a NaN
__device__ __forceinline__ uint32_t push_less(uint32_t m, float a, float b)
{
    asm("v_cmp_lt_f32 vcc, %1, %2\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(m) : "v"(a), "v"(b) : "vcc");
    return m;
}

// The search of a chip full of units: one particle a lane, a unit a block.
// Per stencil row the wavefront's lanes, consecutive sorted particles, mostly
// share one grid row, so their ranges lie in [lo, hi), lo the range start of
// lane 0 and hi the range end of the last valid lane (lastv), about 80 slots.
// When that span fits kWaveRowSlots the wavefront copies it into its own LDS
// (wl) with coalesced loads, and a lane whose range lies inside it reads its
// candidates there; any other lane or row reads global memory.  A candidate
// costs 8 VALU: the squared distance (6), its comparison and the carry that
// shifts the result into the row's mask (10 with the result as a number ored
// in); the set bits are then emitted from the top, in ascending slot.  Bound
// by VALU issue at 1,048,576 particles: 111.6 -> 108.6 us.  Reading the rows'
// ranges and first slots ahead took it from 60 to 76 VGPRs (64 with spills)
// and was slower: 117 (131) us, and at 131,072 particles, two wavefronts a
// SIMD, 49 against 44 us.
template <bool GLOB, bool S16>
__device__ __forceinline__ uint32_t scan_unit_rows(const DevBuffers &b, const KConst &k, uint32_t n, uint32_t kmax,
                                                   uint32_t i, bool valid, uint32_t lastv, const Planned &pl,
                                                   const UnitPlan &L, float *wl)
{
    const uint32_t lane = threadIdx.x & 63u;
    const GridOf gr = pl.gr;
    const float4 p = valid ? b.P[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float r2max = k.search_r2;
    const uint32_t q9 = S16 ? 9u * L.q[threadIdx.x] : 0u;
    const uint32_t ry = pl.row % gr.gy, rz = pl.row / gr.gy;
    const uint32_t x0 = pl.x > 0u ? pl.x - 1u : 0u, x1 = pl.x + 1u < gr.gx ? pl.x + 1u : gr.gx - 1u;
    uint4 *out = const_cast<uint4 *>(nbr_lane(b, i));
    uint2 *out16 = const_cast<uint2 *>(nbr16_chunk(b, i, 0));
    uint4 *out2 = GLOB ? reinterpret_cast<uint4 *>(b.nbr_glob) + (size_t)(i >> 6) * b.kq * 64 + (i & 63) : nullptr;
    uint4 buf = make_uint4(i, i, i, i), buf2 = make_uint4(i, i, i, i);
    uint32_t cnt = 0;
    // an accepted candidate: shifted into buf, which after the 4th entry of
    // a chunk holds it in order (x first); chunks past kmax are not stored
    auto accept = [&](uint32_t e, uint32_t j) {
        if (S16) {
            buf.x = __builtin_amdgcn_alignbit(buf.y, buf.x, 16);
            buf.y = __builtin_amdgcn_alignbit(e, buf.y, 16);
        } else {
            buf.x = buf.y;
            buf.y = buf.z;
            buf.z = buf.w;
            buf.w = e;
        }
        if (GLOB) {
            buf2.x = buf2.y;
            buf2.y = buf2.z;
            buf2.z = buf2.w;
            buf2.w = j;
        }
        if ((cnt & 3u) == 3u && cnt < kmax) {
            if (S16)
                out16[(size_t)(cnt >> 3) * 128 + ((cnt >> 2) & 1u)] = make_uint2(buf.x, buf.y);
            else
                out[(size_t)(cnt >> 2) * 64] = buf;
            if (GLOB) out2[(size_t)(cnt >> 2) * 64] = buf2;
        }
        cnt++;
    };
    // the candidates [j0, j1) of one stencil row; at(j - j0) reads slot j
    auto scan_row = [&](uint32_t j0, uint32_t j1, uint32_t eoff, auto at) {
        for (uint32_t w0 = j0; w0 < j1; w0 += 32u) {
            const uint32_t we = min(w0 + 32u, j1);
            uint32_t m = 0;
            uint32_t jb = w0;
            // whole groups of four: no bound test, one address, immediate
            // offsets; the loads go ahead of the tests
            for (; jb + 4u <= we; jb += 4u) {
                float4 qv[4];
#pragma unroll
                for (uint32_t u = 0; u < 4; u++) qv[u] = at(jb - j0 + u);
#pragma unroll
                for (uint32_t u = 0; u < 4; u++)
                    m = push_less(m, dist2(p.x - qv[u].x, p.y - qv[u].y, p.z - qv[u].z), r2max);
            }
            // the last one to three
            if (jb < we) {
                float4 qv[3];
#pragma unroll
                for (uint32_t u = 0; u < 3; u++) qv[u] = at(min(jb + u, we - 1u) - j0);
#pragma unroll
                for (uint32_t u = 0; u < 3; u++)
                    m = push_less(m, dist2(p.x - qv[u].x, p.y - qv[u].y, p.z - qv[u].z), r2max);
                m >>= 3u - (we - jb);
            }
            m <<= 32u - (we - w0);  // candidate w0 + u at bit 31 - u
            // i itself (in its own row only)
            if (i - w0 < 32u) m &= ~(0x80000000u >> (i - w0));
            while (m != 0u) {
                const uint32_t u = (uint32_t)__builtin_clz(m);
                m ^= 0x80000000u >> u;
                accept(w0 + u + eoff, w0 + u);
            }
        }
    };
    for (uint32_t t = 0; t < 9u; t++) {
        uint32_t j0 = 0, j1 = 0, eoff = 0;
        const int z = (int)rz + (int)(t / 3u) - 1, y = (int)ry + (int)(t % 3u) - 1;
        if (valid && z >= 0 && z < (int)gr.gz && y >= 0 && y < (int)gr.gy) {
            const uint32_t r2 = gr.base + ((uint32_t)z * gr.gy + (uint32_t)y) * gr.gx;
            j0 = b.cell_off[r2 + x0];
            j1 = min(b.cell_off[r2 + x1 + 1u], n);
        }
        // every lane is here: the span and the copy are the wavefront's
        const uint32_t lo = __shfl(j0, 0, 64), hi = __shfl(j1, (int)lastv, 64);
        const bool rowl = lo < hi && hi - lo <= kWaveRowSlots;
        if (rowl) {
            // the previous row's LDS reads were issued before these writes,
            // and a wavefront's LDS operations run in order
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            for (uint32_t s = lane; s < hi - lo; s += 64u) {
                const float4 v = b.P[lo + s];
                wl[3u * s] = v.x;
                wl[3u * s + 1u] = v.y;
                wl[3u * s + 2u] = v.z;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        if (j0 >= j1) continue;
        if (S16) {
            // the row range lies inside its interval (by construction)
            const uint32_t iv = q9 + t;
            eoff = L.delta[iv];
            if (j0 < L.st[iv] || j1 > L.en[iv]) {
                atomicOr(&b.status->flags, PS_STATUS_INTERNAL);
                continue;
            }
        }
        if (rowl && j0 >= lo && j1 <= hi) {
            const float *w3 = wl + 3u * (j0 - lo);
            scan_row(j0, j1, eoff, [&](uint32_t d) {
                return make_float4(w3[3u * d], w3[3u * d + 1u], w3[3u * d + 2u], 0.0f);
            });
        } else {
            const float4 *q0 = b.P + j0;
            scan_row(j0, j1, eoff, [&](uint32_t d) { return q0[d]; });
        }
    }
    const uint32_t kept = cnt < kmax ? cnt : kmax;
    // a partial last chunk: its c entries sit at the right end of buf; a
    // staged unit pads with its sentinel record, a global one with i
    const uint32_t c = kept & 3u;
    if (c != 0u) {
        if (S16) {
            for (uint32_t u = c; u < 4u; u++) {
                buf.x = __builtin_amdgcn_alignbit(buf.y, buf.x, 16);
                buf.y = __builtin_amdgcn_alignbit(kStageSentinel, buf.y, 16);
            }
            out16[(size_t)(kept >> 3) * 128 + ((kept >> 2) & 1u)] = make_uint2(buf.x, buf.y);
        } else {
            out[(size_t)(kept >> 2) * 64] = c == 1u   ? make_uint4(buf.w, i, i, i)
                                            : c == 2u ? make_uint4(buf.z, buf.w, i, i)
                                                      : make_uint4(buf.y, buf.z, buf.w, i);
        }
        if (GLOB)
            out2[(size_t)(kept >> 2) * 64] = c == 1u   ? make_uint4(buf2.w, i, i, i)
                                             : c == 2u ? make_uint4(buf2.z, buf2.w, i, i)
                                                       : make_uint4(buf2.y, buf2.z, buf2.w, i);
    }
    if (valid) b.ncnt[i] = kept;
    return cnt;
}

template <bool GLOB>
__global__ __launch_bounds__(kStageUnit) void neighbors_staged_k(DevBuffers b, KConst k, uint32_t n, uint32_t kmax)
{
    __shared__ UnitPlan L;
    __shared__ uint32_t ldsw[kStageUnit / 64];
    __shared__ float s_wrow[kStageUnit / 64][3 * kWaveRowSlots];  // each wavefront's stencil row (x, y, z)
    const uint32_t unit = xcd_block(), first = unit * kStageUnit, nu = min(kStageUnit, n - first);
    const uint32_t tid = threadIdx.x, w = tid >> 6;
    const Planned pl = plan_unit(b, k, n, first, nu, L);
    put_desc(b.stage + unit, pl, L);
    uint32_t cnt = 0;
    if ((tid & ~63u) < nu) {
        const uint32_t lastv = min(63u, nu - 1u - (tid & ~63u));
        if (pl.staged)
            cnt = scan_unit_rows<GLOB, true>(b, k, n, kmax, first + tid, tid < nu, lastv, pl, L, s_wrow[w]);
        else
            cnt = scan_unit_rows<GLOB, false>(b, k, n, kmax, first + tid, tid < nu, lastv, pl, L, s_wrow[w]);
    }
    neighbor_status(b, cnt, kmax, ldsw);
}

// The search of a few units, bound by its chain of dependent loads: each
// unit's particles go to four blocks (each plans the unit for itself), four
// lanes a particle, lane g over the stencil rows from row_of(g) to
// row_of(g + 1).  A lane reads its rows' ranges and the first eight
// candidates before the plan, which only the entries need, and from then on
// the next eight while it tests eight.  A lane's accepted entries go to its
// list in LDS; the lists of a particle, in lane order, are its table, written
// as whole uint4s.  A particle with a list past kLaneOut has its rows
// searched again, with the positions known, into memory.
// With one lane a particle the nine rows follow one another, each waiting
// for its range and its slots: 20.8 us at 2,048 particles (8 units), now 14.1;
// 26.3 -> 17.7 at 7,096 of a mixed scene (28 units).  Every lane's loads are
// its own, so the gain ends where the chip begins to fill.  Split against one
// lane after 60 to 80 substeps, in us: 32 units 34.9 / 35.7, 48 35.5 / 35.5, 49
// 34.1 / 35.0, 55 (mixed) 37.2 / 34.8, 61 (cloth over a pool) 33.6 / 33.8, 64
// 35.1 / 34.8, 66 (a filled tank) 39.4 / 37.6, 68 38.2 / 36.3, 71 (mixed) 39.4 /
// 36.6, 96 37.3 / 34.8, 128 37.4 / 34.9, and at 512 111 / 44.  From 32 to 64
// units it depends on the scene; the line is the last count measured where no
// scene lost by it.

constexpr uint32_t kNbrParts = 4;                  // blocks per unit
constexpr uint32_t kNbrOwn = kStageUnit / kNbrParts;
constexpr uint32_t kLaneOut = 28;                  // entries of a lane's list
constexpr uint32_t kLaneStride = kLaneOut + 1;     // odd: lanes on distinct banks
constexpr uint32_t kNbrSplitUnits = 32;            // up to here a unit's search is split over four blocks

__device__ __forceinline__ uint32_t row_of(uint32_t g) { return g == 0u ? 0u : 2u * g + 1u; }  // 0, 3, 5, 7, 9

template <bool GLOB>
__global__ __launch_bounds__(kStageUnit) void neighbors_split_k(DevBuffers b, KConst k, uint32_t n, uint32_t kmax)
{
    __shared__ UnitPlan L;
    __shared__ uint32_t ldsw[kStageUnit / 64];
    __shared__ uint32_t s_list[kStageUnit * kLaneStride];
    const uint32_t bid = xcd_block(), unit = bid / kNbrParts, part = bid % kNbrParts;
    const uint32_t first = unit * kStageUnit, nu = min(kStageUnit, n - first);
    const uint32_t g = threadIdx.x & 3u, li = part * kNbrOwn + (threadIdx.x >> 2);
    const bool valid = li < nu;
    const uint32_t i = first + li, ic = valid ? i : first;
    const float r2max = k.search_r2;
    const GridOf gr = grid_of(b, k, k.nscenes > 1u ? b.sid[ic] : 0u);
    const uint32_t key = b.key[ic] - gr.base;
    const float4 p = b.P[ic];
    const uint32_t x = key % gr.gx, row = key / gr.gx, ry = row % gr.gy, rz = row / gr.gy;
    const uint32_t x0 = x > 0u ? x - 1u : 0u, x1 = x + 1u < gr.gx ? x + 1u : gr.gx - 1u;
    // the ranges of the lane's rows (three for lane 0, two for the others)
    const uint32_t t0 = row_of(g), nt = row_of(g + 1u) - t0;
    uint32_t ja[3], je[3];
#pragma unroll
    for (uint32_t u = 0; u < 3; u++) {
        const uint32_t t = t0 + u;
        const int z = (int)rz + (int)(t / 3u) - 1, y = (int)ry + (int)(t % 3u) - 1;
        ja[u] = je[u] = 0u;
        if (valid && u < nt && z >= 0 && z < (int)gr.gz && y >= 0 && y < (int)gr.gy) {
            const uint32_t r2 = gr.base + ((uint32_t)z * gr.gy + (uint32_t)y) * gr.gx;
            ja[u] = b.cell_off[r2 + x0];
            je[u] = min(b.cell_off[r2 + x1 + 1u], n);
            if (je[u] < ja[u]) je[u] = ja[u];
        }
    }
    // eight candidates from j of row u (u = 3: none left)
    struct At {
        uint32_t u, j, e;
    };
    auto from = [&](uint32_t u) {  // the first non-empty row from u on
        At a = {3u, 0u, 0u};
        if (u <= 2u && ja[2] < je[2]) a = At{2u, ja[2], je[2]};
        if (u <= 1u && ja[1] < je[1]) a = At{1u, ja[1], je[1]};
        if (u == 0u && ja[0] < je[0]) a = At{0u, ja[0], je[0]};
        return a;
    };
    auto after = [&](const At &a) { return a.j + 8u < a.e ? At{a.u, a.j + 8u, a.e} : from(a.u + 1u); };
    struct Eight {
        float4 c[8];
    };
    auto fetch = [&](const At &a) {
        Eight v;
        if (a.u < 3u) {
#pragma unroll
            for (uint32_t q = 0; q < 8; q++) v.c[q] = b.P[min(a.j + q, a.e - 1u)];
        }
        return v;
    };
    At at = from(0u);
    Eight v = fetch(at);
    const Planned pl = plan_unit(b, k, n, first, nu, L);
    const bool staged = pl.staged;
    if (part == 0u) put_desc(b.stage + unit, pl, L);
    // LDS index = slot + dl of the row
    uint32_t dl[3] = {0u, 0u, 0u};
    if (staged && valid) {
#pragma unroll
        for (uint32_t u = 0; u < 3; u++)
            if (ja[u] < je[u]) {
                // the range lies inside its interval (by construction)
                const uint32_t iv = 9u * L.q[li] + t0 + u;
                dl[u] = L.delta[iv];
                if (ja[u] < L.st[iv] || je[u] > L.en[iv]) {
                    atomicOr(&b.status->flags, PS_STATUS_INTERNAL);
                    at.u = 3u;
                }
            }
    }
    // every accepted candidate of the lane in order: put(m, j, dl), m of them
    // before; returns how many
    auto search = [&](At a, Eight w, auto put) {
        uint32_t m = 0;
        while (a.u < 3u) {
            const At na = after(a);
            const Eight nw = fetch(na);
            uint32_t bits = 0;
#pragma unroll
            for (uint32_t q = 0; q < 8; q++)
                bits = push_less(bits, dist2(p.x - w.c[q].x, p.y - w.c[q].y, p.z - w.c[q].z), r2max);
            bits <<= 24;  // candidate j + q at bit 31 - q
            if (a.e - a.j < 8u) bits &= 0xffffffffu << (32u - (a.e - a.j));
            if (i - a.j < 8u) bits &= ~(0x80000000u >> (i - a.j));
            const uint32_t d = a.u == 0u ? dl[0] : a.u == 1u ? dl[1] : dl[2];
            while (bits) {
                const uint32_t q = (uint32_t)__builtin_clz(bits);
                bits ^= 0x80000000u >> q;
                put(m++, a.j + q, d);
            }
            a = na;
            w = nw;
        }
        return m;
    };
    uint32_t *list = s_list + threadIdx.x * kLaneStride;
    const uint32_t own = search(at, v, [&](uint32_t m, uint32_t j, uint32_t d) {
        if (m < kLaneOut) list[m] = j + d;
    });
    // the particle's lanes: entries before this one's, and in all
    const uint32_t c1 = __shfl_xor(own, 1, 64), p2 = own + c1, p2o = __shfl_xor(p2, 2, 64);
    const uint32_t pre = ((g & 1u) ? c1 : 0u) + (g >= 2u ? p2o : 0u);
    const uint32_t cnt = p2 + p2o, kept = min(cnt, kmax);
    uint32_t over = own > kLaneOut ? 1u : 0u;
    over |= __shfl_xor(over, 1, 64);
    over |= __shfl_xor(over, 2, 64);
    uint16_t *g16 = reinterpret_cast<uint16_t *>(const_cast<uint2 *>(nbr16_chunk(b, ic, 0)));
    uint32_t *g32 = reinterpret_cast<uint32_t *>(const_cast<uint4 *>(nbr_lane(b, ic)));
    uint32_t *gl = GLOB ? b.nbr_glob + ((size_t)(ic >> 6) * b.kq * 64 + (ic & 63u)) * 4 : nullptr;
    if (valid && over) {
        search(from(0u), fetch(from(0u)), [&](uint32_t m, uint32_t j, uint32_t d) {
            const uint32_t pos = pre + m;
            if (pos >= kmax) return;
            if (staged)
                g16[(size_t)(pos >> 3) * 512 + (pos & 7u)] = (uint16_t)(j + d);
            else
                g32[(size_t)(pos >> 2) * 256 + (pos & 3u)] = j;
            if (GLOB) gl[(size_t)(pos >> 2) * 256 + (pos & 3u)] = j;
        });
        // padding of the last chunk: the sentinel record, in a global table i
        const uint32_t pos = kept + g;
        if (pos < ((kept + 3u) & ~3u)) {
            if (staged)
                g16[(size_t)(pos >> 3) * 512 + (pos & 7u)] = (uint16_t)kStageSentinel;
            else
                g32[(size_t)(pos >> 2) * 256 + (pos & 3u)] = i;
            if (GLOB) gl[(size_t)(pos >> 2) * 256 + (pos & 3u)] = i;
        }
    }
    if (valid && g == 0u) b.ncnt[i] = kept;
    // the lists meet in a wavefront's LDS (its operations run in order)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // where the lists of lanes 1, 2 and 3 begin
    const uint32_t lane0 = (threadIdx.x & 63u) & ~3u;
    const uint32_t b1 = __shfl(pre, (int)lane0 + 1, 64), b2 = __shfl(pre, (int)lane0 + 2, 64),
                   b3 = __shfl(pre, (int)lane0 + 3, 64);
    if (valid && !over) {
        const uint32_t *l0 = s_list + (threadIdx.x & ~3u) * kLaneStride;
        const uint32_t fill = staged ? kStageSentinel : i;
        auto entry = [&](uint32_t pos) {
            const uint32_t o = pos < b1   ? pos
                               : pos < b2 ? kLaneStride + pos - b1
                               : pos < b3 ? 2u * kLaneStride + pos - b2
                                          : 3u * kLaneStride + pos - b3;
            return pos < kept ? l0[o] : fill;
        };
        auto slot = [&](uint32_t e) {
            return !staged ? e : e >= kStageSlots ? i : L.src[e / kStageChunk] + e % kStageChunk;
        };
        // four entries (a chunk) at a time, the lanes in turn
        for (uint32_t c = g; c * 4u < kept; c += 4u) {
            const uint4 e = make_uint4(entry(4u * c), entry(4u * c + 1u), entry(4u * c + 2u), entry(4u * c + 3u));
            if (staged)
                *const_cast<uint2 *>(nbr16_chunk(b, i, c)) = make_uint2(e.x | (e.y << 16), e.z | (e.w << 16));
            else
                const_cast<uint4 *>(nbr_lane(b, i))[(size_t)c * 64] = e;
            if (GLOB)
                reinterpret_cast<uint4 *>(gl)[(size_t)c * 64] = make_uint4(slot(e.x), slot(e.y), slot(e.z), slot(e.w));
        }
    }
    neighbor_status(b, valid ? cnt : 0u, kmax, ldsw);
}

// ---------------------------------------------------------------------------
// a12: shape matching per body (one wavefront per body): centre of mass, A_pq,
// rotation by the fixed-point quaternion iteration (Mueller, Bender,
// Chentanez, Macklin, MIG 2016) with a first-order quaternion step, goals.

__device__ __forceinline__ void quat_to_mat(float w, float x, float y, float z, float *m)
{
    m[0] = 1.0f - (2.0f * ((y * y) + (z * z)));
    m[1] = 2.0f * ((x * y) - (w * z));
    m[2] = 2.0f * ((x * z) + (w * y));
    m[3] = 2.0f * ((x * y) + (w * z));
    m[4] = 1.0f - (2.0f * ((x * x) + (z * z)));
    m[5] = 2.0f * ((y * z) - (w * x));
    m[6] = 2.0f * ((x * z) - (w * y));
    m[7] = 2.0f * ((y * z) + (w * x));
    m[8] = 1.0f - (2.0f * ((x * x) + (y * y)));
}

// The sum of v over the 64 lanes in pairwise order, v[l] + v[l + s] for
// s = 32, 16, ..., 1 (the oracle's lane_tree_sum), returned to every lane.
__device__ __forceinline__ float wave_tree_sum(float v)
{
#pragma unroll
    for (uint32_t s = 32; s > 0; s >>= 1) v = v + __shfl_down(v, s, 64);
    return __shfl(v, 0, 64);
}

// One wavefront per body: member q (of a0..a1) belongs to lane (q - a0) %
// 64, each lane sums its members in order and the lanes are added pairwise;
// every lane then runs the same rotation iteration on the same sums, and
// the members' goals are written lane-parallel.
__device__ __forceinline__ void shape_body(const DevBuffers &b, uint32_t bd)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t a0 = b.body_off[bd], a1 = b.body_off[bd + 1];
    const float M = b.body_mass[bd];
    float cx = 0.0f, cy = 0.0f, cz = 0.0f;
    for (uint32_t q = a0 + lane; q < a1; q += 64u) {
        const uint32_t t = b.slot_of[b.body_idx[q]];
        const float m = 1.0f / b.A[t].w;
        const float4 p = b.P[t];
        cx = cx + (m * p.x);
        cy = cy + (m * p.y);
        cz = cz + (m * p.z);
    }
    cx = wave_tree_sum(cx) / M;
    cy = wave_tree_sum(cy) / M;
    cz = wave_tree_sum(cz) / M;
    float A[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (uint32_t q = a0 + lane; q < a1; q += 64u) {
        const uint32_t t = b.slot_of[b.body_idx[q]];
        const float m = 1.0f / b.A[t].w;
        const float4 p = b.P[t];
        const float ux = m * (p.x - cx), uy = m * (p.y - cy), uz = m * (p.z - cz);
        const float4 r = b.body_rest[q];
        A[0] = A[0] + (ux * r.x); A[1] = A[1] + (ux * r.y); A[2] = A[2] + (ux * r.z);
        A[3] = A[3] + (uy * r.x); A[4] = A[4] + (uy * r.y); A[5] = A[5] + (uy * r.z);
        A[6] = A[6] + (uz * r.x); A[7] = A[7] + (uz * r.y); A[8] = A[8] + (uz * r.z);
    }
#pragma unroll
    for (int e = 0; e < 9; e++) A[e] = wave_tree_sum(A[e]);
    float4 qt = b.body_q[bd];
    float qw = qt.x, qx = qt.y, qy = qt.z, qz = qt.w;
    for (int it = 0; it < 10; it++) {
        float m[9];
        quat_to_mat(qw, qx, qy, qz, m);
        float ox = 0.0f, oy = 0.0f, oz = 0.0f, dot = 0.0f;
        for (int col = 0; col < 3; col++) {
            float rx = m[col], ry = m[3 + col], rz = m[6 + col];
            float ax_ = A[col], ay_ = A[3 + col], az_ = A[6 + col];
            ox = ox + ((ry * az_) - (rz * ay_));
            oy = oy + ((rz * ax_) - (rx * az_));
            oz = oz + ((rx * ay_) - (ry * ax_));
            dot = dot + (((rx * ax_) + (ry * ay_)) + (rz * az_));
        }
        float den = (dot < 0.0f ? -dot : dot) + 1e-9f;
        ox = ox / den;
        oy = oy / den;
        oz = oz / den;
        float wl2 = ((ox * ox) + (oy * oy)) + (oz * oz);
        if (wl2 < 1e-18f) break;  // the same on every lane
        float dw = 1.0f, dx = ox * 0.5f, dy = oy * 0.5f, dz = oz * 0.5f;
        float nw = (((dw * qw) - (dx * qx)) - (dy * qy)) - (dz * qz);
        float nx = (((dw * qx) + (dx * qw)) + (dy * qz)) - (dz * qy);
        float ny = (((dw * qy) - (dx * qz)) + (dy * qw)) + (dz * qx);
        float nz = (((dw * qz) + (dx * qy)) - (dy * qx)) + (dz * qw);
        float nl = sqrtf((((nw * nw) + (nx * nx)) + (ny * ny)) + (nz * nz));
        qw = nw / nl;
        qx = nx / nl;
        qy = ny / nl;
        qz = nz / nl;
    }
    if (lane == 0) b.body_q[bd] = make_float4(qw, qx, qy, qz);
    float m[9];
    quat_to_mat(qw, qx, qy, qz, m);
    for (uint32_t q = a0 + lane; q < a1; q += 64u) {
        const float4 r = b.body_rest[q];
        b.body_goal[q] = make_float4((((m[0] * r.x) + (m[1] * r.y)) + (m[2] * r.z)) + cx,
                                     (((m[3] * r.x) + (m[4] * r.y)) + (m[5] * r.z)) + cy,
                                     (((m[6] * r.x) + (m[7] * r.y)) + (m[8] * r.z)) + cz, 0.0f);
    }
}

// ---------------------------------------------------------------------------
// a7 and a9 of one iteration, for the particles that have them: contact
// corrections of those that walk their table for contacts (walk_slot: phase
// from cloth up, w != 0) to con_c (xyz, and the contact count in w), distance
// corrections of those with distance constraints (link_slot) to con_d.  Neither
// reads lambda, so they and shape matching are the first blocks of the lambda
// launch (constraint_block), beside the fluid's, and the solve adds their
// results in its order.
//
// Inside the solve, a walker's chain of waits (its table, the partners'
// records, its constraints' indices, pairs, slots and records) held up the 31
// others of its wavefront, and the contact lists and staged phases took its
// block from 49 to 78 KB of LDS, two blocks a CU instead of three.  Lambda,
// shape matching and solve, before and with these blocks, in us a launch:
// 766k particles (cloth 65k, 3,125 bodies) 42 + 20 + 143, 119 + 49; an
// ensemble of 2.6M with 128 ropes 118 + 187 (solve), 121 + 142; 7k mixed
// 5.2 + 9.1 + 12.5, 11.3 + 6.9; cloth over a pool, 82k, 10 + 24, 12 + 11.

// a7: particle contacts + friction (collideD, integration_kernel.cuh:358-462).
// The corrections are summed in the two halves of the table, each in table
// order, then added half 0 + half 1 (the oracle's order).  Eight lanes a
// particle, four a half: in the counting walk lane s of the four takes every
// fourth chunk of its half (with up to 32 neighbours one chunk each, so the
// chain of table, slots and records is waited for once), and the contacts are
// listed in the half's LDS in table order; then each of the four forms the
// terms of every fourth contact (about 300 VALU between solids) and all add
// them in order.  With one lane a half the lambda launch was 23.6 us at the
// 82k cloth scene and 15.0 at its 5k one (12.3 and 7.6 with four: a chain of
// up to eight chunks, one after the other, is what it waited for), and 115 at
// the 766k scene (119), which has walkers enough to hide it.
__device__ __forceinline__ void constrain_contacts(const DevBuffers &b, const KConst &k, uint32_t q, uint32_t lane8,
                                                   uint32_t *list, uint32_t cap)
{
    const uint32_t hh = lane8 >> 2, s = lane8 & 3u;
    const uint32_t i = b.walk_slot[q];
    const Attr a = b.A[i];
    const float4 p = b.P[i], xi = b.X[i];
    const uint32_t c = b.ncnt[i];
    const StageDesc *d = b.stage + i / kStageUnit;
    const bool staged = b.staging && d->staged;
    const float px = p.x, py = p.y, pz = p.z;
    const int32_t ph = a.phase;
    const float wi = a.w;
    const uint32_t nch = (c + 3u) >> 2, half = nch > hh ? (nch - hh + 1u) >> 1 : 0u;  // chunks hh + 2t
    auto chunk = [&](uint32_t t) {
        if (!staged) return nbr_lane(b, i)[(size_t)(hh + 2u * t) * 64];
        const uint2 e = *nbr16_chunk(b, i, hh + 2u * t);
        return make_uint4(e.x & 0xffffu, e.x >> 16, e.y & 0xffffu, e.y >> 16);
    };
    // the slot of an entry (a staged unit's sentinel padding maps to i)
    auto slot = [&](uint32_t e) {
        return !staged ? e : e >= kStageSlots ? i : d->src[e / kStageChunk] + e % kStageChunk;
    };
    auto is_contact = [&](const float4 &qj, int32_t pj) {
        if (ph > PS_PHASE_SOLID && ph == pj) return false;
        const float dx = px - qj.x, dy = py - qj.y, dz = pz - qj.z;
        const float r2 = ((dx * dx) + (dy * dy)) + (dz * dz);
        return r2 < k.collide_r2;
    };
    uint32_t found = 0;  // contacts of the half (listed up to cap), the same in its four lanes
    for (uint32_t t0 = 0; t0 < half; t0 += 4u) {
        const uint32_t t = t0 + s;
        uint32_t mine = 0, j[4] = {i, i, i, i};  // a bit per contact of the chunk
        if (t < half) {
            const uint4 e = chunk(t);
            j[0] = slot(e.x);
            j[1] = slot(e.y);
            j[2] = slot(e.z);
            j[3] = slot(e.w);
            float4 r[4];
            int32_t pj[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; u++) {
                r[u] = b.P[j[u]];
                pj[u] = b.phs[j[u]] & 0x7fffffff;
            }
            const uint32_t at = (hh + 2u * t) << 2;
#pragma unroll
            for (uint32_t u = 0; u < 4; u++)
                if (at + u < c && is_contact(r[u], pj[u])) mine |= 1u << u;
        }
        const uint32_t n = (uint32_t)__popc(mine);
        const uint32_t n0 = quad_value<0>(n), n1 = quad_value<1>(n), n2 = quad_value<2>(n), n3 = quad_value<3>(n);
        uint32_t m = found + (s > 0u ? n0 : 0u) + (s > 1u ? n1 : 0u) + (s > 2u ? n2 : 0u);
#pragma unroll
        for (uint32_t u = 0; u < 4; u++)
            if (mine & (1u << u)) {
                if (m < cap) list[m] = j[u];
                m++;
            }
        found += n0 + n1 + n2 + n3;
    }
    const uint32_t nc = found + __shfl_xor(found, 4, 64);
    float cx = 0.0f, cy = 0.0f, cz = 0.0f;  // the half's sum
    if (nc > 0) {
        const float fnc = (float)nc;
        const float ewi = wi * ps_exp(py);
        // a contact's terms: e is added, then f subtracted (0 if left out:
        // the sums start at +0 and never are -0)
        struct Terms {
            float ex, ey, ez, fx, fy, fz;
        };
        auto terms = [&](uint32_t j) {
            Terms r = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            const float4 qj = b.P[j];
            const Attr aj = b.A[j];
            const int32_t pj = aj.phase;
            float dx = px - qj.x, dy = py - qj.y, dz = pz - qj.z;
            float r2 = ((dx * dx) + (dy * dy)) + (dz * dz);
            float dist = sqrtf(r2);
            if (dist < 1e-6f) return r;
            const float wj = aj.w;
            float cw = wi, cw2 = wj;
            const bool solid = ph >= PS_PHASE_SOLID && pj >= PS_PHASE_SOLID;
            if (solid) {
                cw = ewi;
                cw2 = wj * ps_exp(qj.y);
            }
            float wsum = cw + cw2;
            if (wsum == 0.0f) return r;
            float mag = dist - k.collide_dist;
            float sc = (((mag / wsum) / dist) * cw) / fnc;
            r.ex = -(sc * dx);
            r.ey = -(sc * dy);
            r.ez = -(sc * dz);
            if (!solid) return r;
            const float4 xj = b.X[j];
            float sc2 = (((mag / wsum) / dist) * cw2) / fnc;
            float gx = sc2 * dx, gy = sc2 * dy, gz = sc2 * dz;
            float rx = ((px + r.ex) - xi.x) - ((qj.x + gx) - xj.x);
            float ry = ((py + r.ey) - xi.y) - ((qj.y + gy) - xj.y);
            float rz = ((pz + r.ez) - xi.z) - ((qj.z + gz) - xj.z);
            float nx = dx / dist, ny = dy / dist, nz = dz / dist;
            float dn = ((rx * nx) + (ry * ny)) + (rz * nz);
            float tx = rx - (dn * nx), ty = ry - (dn * ny), tz = rz - (dn * nz);
            float lt = sqrtf(((tx * tx) + (ty * ty)) + (tz * tz));
            if (lt < 0.001f) return r;
            float share = cw / wsum;
            if (lt < (k.mu_s * dist)) {
                r.fx = tx * share;
                r.fy = ty * share;
                r.fz = tz * share;
            } else {
                float f = (k.mu_k * dist) / lt;
                if (f > 1.0f) f = 1.0f;
                r.fx = (tx * f) * share;
                r.fy = (ty * f) * share;
                r.fz = (tz * f) * share;
            }
            return r;
        };
        if (found <= cap) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the list is the wavefront's
            for (uint32_t m = 0; m < found; m += 4u) {
                Terms r = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
                if (m + s < found) r = terms(list[m + s]);
                cx = (cx + quad_value<0>(r.ex)) - quad_value<0>(r.fx);
                cy = (cy + quad_value<0>(r.ey)) - quad_value<0>(r.fy);
                cz = (cz + quad_value<0>(r.ez)) - quad_value<0>(r.fz);
                cx = (cx + quad_value<1>(r.ex)) - quad_value<1>(r.fx);
                cy = (cy + quad_value<1>(r.ey)) - quad_value<1>(r.fy);
                cz = (cz + quad_value<1>(r.ez)) - quad_value<1>(r.fz);
                cx = (cx + quad_value<2>(r.ex)) - quad_value<2>(r.fx);
                cy = (cy + quad_value<2>(r.ey)) - quad_value<2>(r.fy);
                cz = (cz + quad_value<2>(r.ez)) - quad_value<2>(r.fz);
                cx = (cx + quad_value<3>(r.ex)) - quad_value<3>(r.fx);
                cy = (cy + quad_value<3>(r.ey)) - quad_value<3>(r.fy);
                cz = (cz + quad_value<3>(r.ez)) - quad_value<3>(r.fz);
            }
        } else {
            // more contacts than the list holds (rare): each of the four
            // lanes walks the half again
            for (uint32_t t = 0; t < half; t++) {
                const uint4 e = chunk(t);
                const uint32_t at = (hh + 2u * t) << 2;
                for (uint32_t u = 0; u < 4u && at + u < c; u++) {
                    const uint32_t j = slot(u == 0u ? e.x : u == 1u ? e.y : u == 2u ? e.z : e.w);
                    if (!is_contact(b.P[j], b.phs[j] & 0x7fffffff)) continue;
                    const Terms r = terms(j);
                    cx = (cx + r.ex) - r.fx;
                    cy = (cy + r.ey) - r.fy;
                    cz = (cz + r.ez) - r.fz;
                }
            }
        }
    }
    const float hx = __shfl_xor(cx, 4, 64), hy = __shfl_xor(cy, 4, 64), hz = __shfl_xor(cz, 4, 64);
    if (!lane8) b.con_c[i] = make_float4(cx + hx, cy + hy, cz + hz, __uint_as_float(nc));
}

// a9: distance constraints, gathered over a particle's incident list in order
// (links: the partner's insertion index, rest length, stiffness and the
// partner's inverse mass).  The partner's position is two loads away; four
// lanes take a particle's links in turn, three of each at once, so a cloth
// particle's twelve wait together, and every lane subtracts all terms in
// order.
__device__ __forceinline__ void constrain_links(const DevBuffers &b, uint32_t q, uint32_t g)
{
    const uint32_t i = b.link_slot[q];
    const uint2 ends = b.link_ends[q];
    const uint32_t a0 = ends.x, a1 = ends.y;
    const float2 own = b.link_own[q];  // its inverse mass and incidence count
    const float wi = own.x;
    const float4 p = b.P[i];
    float cx = 0.0f, cy = 0.0f, cz = 0.0f;
    constexpr uint32_t kR = 3;
    for (uint32_t q0 = a0; q0 < a1; q0 += 4u * kR) {  // the same trip count in the four lanes
        float4 ln[kR], pj[kR];
#pragma unroll
        for (uint32_t r = 0; r < kR; r++) ln[r] = b.links[min(q0 + 4u * r + g, a1 - 1u)];
#pragma unroll
        for (uint32_t r = 0; r < kR; r++) pj[r] = b.P[b.slot_of[__float_as_uint(ln[r].x)]];
#pragma unroll
        for (uint32_t r = 0; r < kR; r++) {
            float tx = 0.0f, ty = 0.0f, tz = 0.0f;  // a term that is left out subtracts 0
            const float dx = p.x - pj[r].x, dy = p.y - pj[r].y, dz = p.z - pj[r].z;
            const float dist = sqrtf(((dx * dx) + (dy * dy)) + (dz * dz));
            const float wsum = wi + ln[r].w;
            if (q0 + 4u * r + g < a1 && !(dist < 1e-6f || wsum == 0.0f)) {
                const float sc = ((((dist - ln[r].y) / wsum) / dist) * wi) * ln[r].z;
                tx = sc * dx;
                ty = sc * dy;
                tz = sc * dz;
            }
            cx = (((cx - quad_value<0>(tx)) - quad_value<1>(tx)) - quad_value<2>(tx)) - quad_value<3>(tx);
            cy = (((cy - quad_value<0>(ty)) - quad_value<1>(ty)) - quad_value<2>(ty)) - quad_value<3>(ty);
            cz = (((cz - quad_value<0>(tz)) - quad_value<1>(tz)) - quad_value<2>(tz)) - quad_value<3>(tz);
        }
    }
    if (!g) b.con_d[i] = make_float4(cx / own.y, cy / own.y, cz / own.y, 0.0f);
}

// Block bid of the constraint blocks (con_parts): contacts (lds holds their
// lists, cap entries a lane), links, bodies, the longest chains first.
__device__ __forceinline__ void constraint_block(const DevBuffers &b, const KConst &k, const ConBlocks &con,
                                                 uint32_t *lds, uint32_t cap)
{
    const uint32_t bid = con.first + blockIdx.x;
    // the first item of the block, counted in items: bid times the threads
    // may be past 32 bits
    if (bid < con.walks) {
        // a half's list is its four lanes' share
        const uint32_t q = bid * (blockDim.x >> 3) + (threadIdx.x >> 3);
        if (q < b.nwalk)
            constrain_contacts(b, k, q, threadIdx.x & 7u, lds + (threadIdx.x & ~3u) * cap, 4u * cap);
    } else if (bid - con.walks < con.links) {
        const uint32_t q = (bid - con.walks) * (blockDim.x >> 2) + (threadIdx.x >> 2);
        if (q < b.nlink) constrain_links(b, q, threadIdx.x & 3u);
    } else {
        const uint32_t bd = (bid - con.walks - con.links) * (blockDim.x >> 6) + (threadIdx.x >> 6);
        if (bd < b.nbody) shape_body(b, bd);
    }
}

// ---------------------------------------------------------------------------
// a5: PBF multiplier (findLambdasD, integration_kernel.cuh:521-593)
//   rho_i = W(0)/w_i + sum_j s_j W(r)/w_j,  grad_j = a d,
//   a = (spiky/rho0_i) (h-r)^2 / r,
//   lambda_i = -(rho_i/rho0_i - 1) / (sum |grad_j|^2 + |sum grad_j|^2 + eps)
// Per pair, with t = h^2 - r^2, 1/r = rsq(r^2) and q = h - r =
// fma(-r^2, 1/r, h): the density term t^3 m_j, the gradient term q^2 (1/r) d
// and |grad_j|^2 as q^4; the constants poly6 and sk = spiky/rho0_i multiply
// the finished sums (rho = fma(poly6, sum, W(0)/w_i), grad sum sk S,
// sum |grad_j|^2 = sk^2 sum q^4).  Degenerate pairs (r^2 < 1e-8) add density
// only.
// UNIFORM: every particle is fluid with inverse mass wu (no Attr gathers).

// TAPE (reverse-pass recording): also store S, D and rho per particle.
// A scene that is not a uniform fluid: the first con.blocks blocks (a multiple
// of the XCDs) are its constraints' from con.first on (constraint_block).  Six wavefronts a
// SIMD (80 VGPRs) are what three staged blocks a CU take.
template <bool UNIFORM, bool STAGED, bool TAPE = false>
__global__ __launch_bounds__(kMaxBlock, UNIFORM ? 1 : 6) void lambda_k(DevBuffers b, KConst k, uint32_t n, float mu,
                                                                       ConBlocks con)
{
    // staged: a uniform fluid stages neighbour positions only, 12 bytes
    // per slot (36 KB, so four blocks fit in a CU's LDS where 16-byte slots
    // allow three); other scenes stage (x, y, z, mj), a particle with w = 0
    // as a position at infinity, which every pair test rejects as the
    // global path leaves it out.  Then the sentinel record; two lanes per
    // particle (2 kStageUnit threads), lane hh summing half hh
    __shared__ float lds3[STAGED && UNIFORM ? 3 * (kStageSlots + 1) : 1];
    __shared__ float4 lds4[STAGED && !UNIFORM ? kStageSlots + 1 : 1];
    extern __shared__ uint32_t contact_lds[];
    uint32_t unit;
    if constexpr (UNIFORM) {
        unit = xcd_block();
    } else {
        if (blockIdx.x < con.blocks) {
            if (STAGED)
                constraint_block(b, k, con, reinterpret_cast<uint32_t *>(lds4), 4u * kStageSlots / (2u * kStageUnit));
            else
                constraint_block(b, k, con, contact_lds, kContactList);
            return;
        }
        unit = xcd_block(blockIdx.x - con.blocks, gridDim.x - con.blocks);
    }
    const uint32_t hh = STAGED ? (threadIdx.x & 1u) : 0u;
    const uint32_t i = STAGED ? unit * kStageUnit + (threadIdx.x >> 1) : unit * blockDim.x + threadIdx.x;
    bool staged = false;
    // staged: the particle's own records and the first chunks of its table
    // go in flight with the staging loads (a thread past the end reads the
    // last particle's)
    StagedTable<2, 4> tab;
    Attr a;
    float4 p;
    uint32_t c = 0;
    if (STAGED) {
        const StageDesc *d = b.stage + unit;
        StageSrc<2 * kStageUnit> ss;
        const uint32_t ic = min(i, n - 1u);
        ss.load(d);
        tab.load(b, ic, hh);
        a = b.A[ic];
        p = b.P[ic];
        c = b.ncnt[ic];
        staged = d->staged != 0u;
        const uint32_t nch = d->nchunks;
        if (UNIFORM) {
            if (staged && threadIdx.x < 3) lds3[3 * kStageSentinel + threadIdx.x] = __builtin_inff();
            if (staged)
                stage_copy<6>(ss, nch, n, [&](uint32_t j) { return b.P[j]; },
                              [&](uint32_t l, const float4 &v) {
                                  lds3[3 * l] = v.x;
                                  lds3[3 * l + 1] = v.y;
                                  lds3[3 * l + 2] = v.z;
                              });
        } else {
            const float inf = __builtin_inff();
            if (staged && threadIdx.x == 0) lds4[kStageSentinel] = make_float4(inf, inf, inf, 0.0f);
            if (staged)
                stage_copy<6>(ss, nch, n, [&](uint32_t j) { return PM{b.P[j], b.mj[j]}; },
                              [&](uint32_t l, const PM &v) {
                                  lds4[l] = v.m < 0.0f ? make_float4(inf, inf, inf, 0.0f)
                                                       : make_float4(v.p.x, v.p.y, v.p.z, v.m);
                              });
        }
    }
    if (i >= n) return;
    float *Pw = reinterpret_cast<float *>(b.P);
    if (!STAGED) a = b.A[i];
    if (!UNIFORM && a.phase != PS_PHASE_FLUID) {
        Pw[4 * (size_t)i + 3] = 0.0f;
        if (TAPE) {
            const float4 pn = STAGED ? p : b.P[i];
            b.tape_lq[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            b.tape_rho[i] = 0.0f;
            b.tape_pit[i] = make_float4(pn.x, pn.y, pn.z, 0.0f);
        }
        return;
    }
    if (!STAGED) {
        p = b.P[i];
        c = b.ncnt[i];
    }
    const float r0 = a.rho0;
    const float sk = k.spiky * (1.0f / r0);
    // the sums of one half of the table
    struct Sums {
        float rho, gix, giy, giz, den;
    };
    const float self = k.w_zero * (UNIFORM ? mu : (1.0f / a.w));
    // mj: 1/w_j, times s_solid for a non-fluid neighbour
    auto body = [&](Sums &s, const float4 &pj, float mj) {
        float dx = p.x - pj.x, dy = p.y - pj.y, dz = p.z - pj.z;
        float r2 = dist2(dx, dy, dz);
        if (!(r2 < k.h2)) return;
        float t = k.h2 - r2;
        s.rho = __builtin_fmaf((t * t) * t, mj, s.rho);
        if (r2 < kDegenerateR2) return;  // density only
        const float ri = rsq(r2);
        const float qq = __builtin_fmaf(-r2, ri, k.h);
        const float q2 = qq * qq;
        const float aa = q2 * ri;
        s.den = __builtin_fmaf(q2, q2, s.den);
        s.gix = __builtin_fmaf(aa, dx, s.gix);
        s.giy = __builtin_fmaf(aa, dy, s.giy);
        s.giz = __builtin_fmaf(aa, dz, s.giz);
    };
    Sums s0 = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f}, s1 = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (STAGED) {
        // this lane's half (from LDS, or from global memory for a unit that
        // was not staged); the partner lane (lane ^ 1) holds the other.
        // Both lanes form half 0 + half 1 (addition commutes)
        Sums mine = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        if (UNIFORM && staged)
            tab.visit(
                hh, c,
                [&](uint32_t l) {
                    // byte offset 12 l by the full-rate 24-bit multiply (l <= kStageSentinel)
                    const float *q = reinterpret_cast<const float *>(reinterpret_cast<const char *>(lds3) +
                                                                     __umul24(l, 12u));
                    return make_float4(q[0], q[1], q[2], 0.0f);
                },
                [&](uint32_t, const float4 &pj) { body(mine, pj, mu); });
        else if (UNIFORM)
            for_neighbors_half(
                b, i, c, hh, [&](uint32_t j) { return b.P[j]; },
                [&](uint32_t, const float4 &pj) { body(mine, pj, mu); });
        else if (staged)
            tab.visit(hh, c, [&](uint32_t l) { return lds4[l]; },
                      [&](uint32_t, const float4 &pj) { body(mine, pj, pj.w); });
        else
            for_neighbors_half(
                b, i, c, hh, [&](uint32_t j) { return PM{b.P[j], b.mj[j]}; },
                [&](uint32_t, const PM &d) {
                    if (d.m >= 0.0f) body(mine, d.p, d.m);
                });
        const Sums other = {__shfl_xor(mine.rho, 1, 64), __shfl_xor(mine.gix, 1, 64),
                            __shfl_xor(mine.giy, 1, 64), __shfl_xor(mine.giz, 1, 64),
                            __shfl_xor(mine.den, 1, 64)};
        s0 = hh ? other : mine;
        s1 = hh ? mine : other;
    } else if (UNIFORM) {
        for_neighbors_split(
            b, i, c, [&](uint32_t j) { return b.P[j]; },
            [&](uint32_t, const float4 &pj) { body(s0, pj, mu); },
            [&](uint32_t, const float4 &pj) { body(s1, pj, mu); });
    } else {
        // the neighbour's mass from the sort's mj (-1: w = 0, left out)
        auto gen = [&](Sums &s, const PM &d) {
            if (d.m < 0.0f) return;
            body(s, d.p, d.m);
        };
        for_neighbors_split(
            b, i, c, [&](uint32_t j) { return PM{b.P[j], b.mj[j]}; },
            [&](uint32_t, const PM &d) { gen(s0, d); }, [&](uint32_t, const PM &d) { gen(s1, d); });
    }
    const float rho = __builtin_fmaf(k.poly6, s0.rho + s1.rho, self);
    const float gix = sk * (s0.gix + s1.gix), giy = sk * (s0.giy + s1.giy), giz = sk * (s0.giz + s1.giz);
    const float den = __builtin_fmaf(sk * sk, s0.den + s1.den, dist2(gix, giy, giz));
    float C = (rho / r0) - 1.0f;
    if (STAGED && hh) return;  // the pair's lane 0 writes
    const float lam = -C / (den + k.relax);
    Pw[4 * (size_t)i + 3] = lam;
    if (TAPE) {
        b.tape_pit[i] = make_float4(p.x, p.y, p.z, lam);
        b.tape_lq[i] = make_float4(gix, giy, giz, den);
        b.tape_rho[i] = rho;
    }
}


// ---------------------------------------------------------------------------
// One Jacobi iteration for every particle: contacts (a7), fluid delta-p
// (a6), distance (a9), shape goal (a12) summed in that order from the same
// snapshot P, then walls (a8) and pins (a10); result to Q.  The contact and
// distance corrections come from the constraint blocks (con_c, con_d).

// GEN: the scene has contact phases, constraints, bodies or pins; smark says
// per slot which of them a particle has.  TAPE (reverse-pass recording): also
// store the fluid sum f (before the division by rho0) and the contact count
// per particle.
template <bool GEN, bool UNIFORM, uint32_t NC, bool STAGED, bool TAPE = false>
__global__ __launch_bounds__(kMaxBlock) void solve_k(DevBuffers b, KConst k, uint32_t n, float wu,
                                                  uint32_t it)
{
    // staged: two lanes per particle (2 kStageUnit threads), lane hh summing
    // half hh of the fluid sum; lane 0 finishes the particle.  The LDS holds
    // the unit's slots and the sentinel record.  In a scene that is not a
    // uniform fluid a particle with w = 0 is staged as a position at infinity
    // (the fluid sum leaves it out, as the global path does).
    __shared__ float4 lds[STAGED ? kStageSlots + 1 : 1];
    const uint32_t unit = xcd_block();
    const uint32_t hh = STAGED ? (threadIdx.x & 1u) : 0u;
    const uint32_t i = STAGED ? unit * kStageUnit + (threadIdx.x >> 1) : unit * blockDim.x + threadIdx.x;
    bool staged = false;
    // staged: the particle's own records and the first chunks of its table
    // go in flight with the staging loads, as in lambda_k
    StagedTable<2, 4> tab;
    Attr a;
    float4 p;
    uint32_t c = 0;
    if (STAGED) {
        const StageDesc *d = b.stage + unit;
        StageSrc<2 * kStageUnit> ss;
        const uint32_t ic = min(i, n - 1u);
        ss.load(d);
        tab.load(b, ic, hh);
        a = b.A[ic];
        p = b.P[ic];
        c = b.ncnt[ic];
        staged = d->staged != 0u;
        const uint32_t nch = d->nchunks;
        const float inf = __builtin_inff();
        if (staged && threadIdx.x == 0) lds[kStageSentinel] = make_float4(inf, inf, inf, 0.0f);
        if (UNIFORM && staged)
            stage_copy<6>(ss, nch, n, [&](uint32_t j) { return b.P[j]; },
                          [&](uint32_t l, const float4 &v) { lds[l] = v; });
        else if (staged)
            stage_copy<6>(ss, nch, n, [&](uint32_t j) { return PM{b.P[j], b.mj[j]}; },
                          [&](uint32_t l, const PM &v) {
                              lds[l] = v.m < 0.0f ? make_float4(inf, inf, inf, 0.0f) : v.p;
                          });
    }
    if (i >= n) return;
    if (!STAGED) {
        p = b.P[i];
        a = b.A[i];
        c = b.ncnt[i];
    }
    const float px = p.x, py = p.y, pz = p.z;
    const int32_t ph = UNIFORM ? PS_PHASE_FLUID : a.phase;
    const float wi = UNIFORM ? wu : a.w;
    float ax = 0.0f, ay = 0.0f, az = 0.0f;
    float4 tape = make_float4(0.0f, 0.0f, 0.0f, 0.0f);  // (f, contact count) when TAPE

    const uint32_t mark = GEN ? b.smark[i] : 0u;
    // a7: particle contacts + friction
    if (GEN && ph >= PS_PHASE_CLOTH && wi != 0.0f && (!STAGED || !hh)) {
        const float4 cc = b.con_c[i];
        ax = ax + cc.x;
        ay = ay + cc.y;
        az = az + cc.z;
        if (TAPE) tape.w = cc.w;
    }

    // a6: PBF delta-p with tensile correction s_corr = -k h^2 (W/W(dq h))^n
    // (solveFluidsD :596-642); k.k_corr already holds k h^2 (or k).  Per
    // pair, with t = h^2 - r^2, 1/r = rsq(r^2) and q = h - r =
    // fma(-r^2, 1/r, h): W/W(dq h) = s^3 with s = (h^2 - r^2)/(h^2 - (dq h)^2)
    // = fma(-w_scale, r^2, w_scale_h2), coef = fma(-k, (W/W(dq h))^n,
    // l_i + l_j), and the term -coef q^2 (1/r) d; spiky multiplies the
    // finished sum
    {
        if (ph == PS_PHASE_FLUID) {
            const float li = p.w, ir0 = 1.0f / a.rho0;
            // r^2 < 1e-8: gradient (0, -0.001 spiky h^2, 0) (integration_kernel.cuh:625-626)
            const float gdeg = (k.h * k.h) * 0.001f;
            // the sum of one half of the table; deg: a degenerate pair was
            // left out, and the half must be formed again by exact()
            struct Sums {
                float fx, fy, fz;
                bool deg;
            };
            // w_scale_h2 held in a vector register for the loop: an FMA may
            // read one scalar operand only, and w_scale is the other
            float wsh2 = k.w_scale_h2;
            asm volatile("" : "+v"(wsh2));
            auto coef_of = [&](float r2, float lj) {
                const float sw = __builtin_fmaf(-k.w_scale, r2, wsh2);
                const float x = (sw * sw) * sw;
                return __builtin_fmaf(-k.k_corr, ipow(x, NC ? NC : k.n_corr), li + lj);
            };
            auto term = [&](Sums &s, float coef, float r2, float dx, float dy, float dz) {
                const float ri = rsq(r2);
                const float qq = __builtin_fmaf(-r2, ri, k.h);
                const float g = coef * ((qq * qq) * ri);
                s.fx = __builtin_fmaf(-g, dx, s.fx);
                s.fy = __builtin_fmaf(-g, dy, s.fy);
                s.fz = __builtin_fmaf(-g, dz, s.fz);
            };
            // every pair but a degenerate one (essentially never present)
            auto fast = [&](Sums &s, const float4 &pj) {
                float dx = px - pj.x, dy = py - pj.y, dz = pz - pj.z;
                float r2 = dist2(dx, dy, dz);
                if (!(r2 < k.h2)) return;
                const bool dg = r2 < kDegenerateR2;
                s.deg = s.deg || dg;
                if (dg) return;
                term(s, coef_of(r2, pj.w), r2, dx, dy, dz);
            };
            // the reference's sum, degenerate pairs in their place
            auto exact = [&](Sums &s, const float4 &pj) {
                float dx = px - pj.x, dy = py - pj.y, dz = pz - pj.z;
                float r2 = dist2(dx, dy, dz);
                if (!(r2 < k.h2)) return;
                const float coef = coef_of(r2, pj.w);
                if (r2 < kDegenerateR2)
                    s.fy = s.fy - (coef * gdeg);
                else
                    term(s, coef, r2, dx, dy, dz);
            };
            Sums s0 = {0.0f, 0.0f, 0.0f, false}, s1 = {0.0f, 0.0f, 0.0f, false};
            if constexpr (STAGED) {
                // this lane's half; the partner lane (lane ^ 1) holds the other
                Sums mine = {0.0f, 0.0f, 0.0f, false};
                auto from_lds = [&](uint32_t l) { return lds[l]; };
                auto from_glob = [&](uint32_t j) { return b.P[j]; };
                // a unit that was not staged, in a scene that is not a uniform fluid
                auto from_glob_m = [&](uint32_t j) { return PM{b.P[j], b.mj[j]}; };
                if (staged)
                    tab.visit(hh, c, from_lds, [&](uint32_t, const float4 &pj) { fast(mine, pj); });
                else if (UNIFORM)
                    for_neighbors_half(b, i, c, hh, from_glob,
                                       [&](uint32_t, const float4 &pj) { fast(mine, pj); });
                else
                    for_neighbors_half(b, i, c, hh, from_glob_m, [&](uint32_t, const PM &d) {
                        if (d.m >= 0.0f) fast(mine, d.p);
                    });
                if (mine.deg) {
                    mine = {0.0f, 0.0f, 0.0f, false};
                    auto ex = [&](uint32_t, const float4 &pj) { exact(mine, pj); };
                    if (staged)
                        for_staged_half_plain(b, i, c, hh, [&](uint32_t e) { exact(mine, lds[e]); });
                    else if (UNIFORM)
                        for_neighbors_half_plain(b, i, c, hh, from_glob, ex);
                    else
                        for_neighbors_half_plain(b, i, c, hh, from_glob_m, [&](uint32_t, const PM &d) {
                            if (d.m >= 0.0f) exact(mine, d.p);
                        });
                }
                const Sums other = {__shfl_xor(mine.fx, 1, 64), __shfl_xor(mine.fy, 1, 64),
                                    __shfl_xor(mine.fz, 1, 64), false};
                s0 = hh ? other : mine;
                s1 = hh ? mine : other;
            } else if (UNIFORM) {
                auto gather = [&](uint32_t j) { return b.P[j]; };
                for_neighbors_split(
                    b, i, c, gather, [&](uint32_t, const float4 &pj) { fast(s0, pj); },
                    [&](uint32_t, const float4 &pj) { fast(s1, pj); });
                if (s0.deg || s1.deg) {
                    s0 = {0.0f, 0.0f, 0.0f, false};
                    s1 = {0.0f, 0.0f, 0.0f, false};
                    for_neighbors_half_plain(b, i, c, 0u, gather,
                                             [&](uint32_t, const float4 &pj) { exact(s0, pj); });
                    for_neighbors_half_plain(b, i, c, 1u, gather,
                                             [&](uint32_t, const float4 &pj) { exact(s1, pj); });
                }
            } else {
                // neighbours with w = 0 are left out (mj < 0)
                auto gather = [&](uint32_t j) { return PM{b.P[j], b.mj[j]}; };
                for_neighbors_split(
                    b, i, c, gather,
                    [&](uint32_t, const PM &d) {
                        if (d.m >= 0.0f) fast(s0, d.p);
                    },
                    [&](uint32_t, const PM &d) {
                        if (d.m >= 0.0f) fast(s1, d.p);
                    });
                if (s0.deg || s1.deg) {
                    s0 = {0.0f, 0.0f, 0.0f, false};
                    s1 = {0.0f, 0.0f, 0.0f, false};
                    for_neighbors_half_plain(b, i, c, 0u, gather, [&](uint32_t, const PM &d) {
                        if (d.m >= 0.0f) exact(s0, d.p);
                    });
                    for_neighbors_half_plain(b, i, c, 1u, gather, [&](uint32_t, const PM &d) {
                        if (d.m >= 0.0f) exact(s1, d.p);
                    });
                }
            }
            const float fx = k.spiky * (s0.fx + s1.fx), fy = k.spiky * (s0.fy + s1.fy),
                        fz = k.spiky * (s0.fz + s1.fz);
            ax = ax + (fx * ir0);
            ay = ay + (fy * ir0);
            az = az + (fz * ir0);
            if (TAPE) {
                tape.x = fx;
                tape.y = fy;
                tape.z = fz;
            }
        }
    }

    // staged: the pair's lane 0 finishes the particle
    if (STAGED && hh) return;

    // a9: distance constraints
    if (GEN && (mark & kMarkDist)) {
        const float4 cd = b.con_d[i];
        ax = ax + cd.x;
        ay = ay + cd.y;
        az = az + cd.z;
    }

    // a12: shape-matching goal pull
    if (GEN && (mark & kMarkBody)) {
        const uint32_t o = a.orig;
        const float4 g = b.body_goal[b.member_of[o]];
        const float st = b.body_stiff[b.body_of[o] - 1];
        ax = ax + ((g.x - px) * st);
        ay = ay + ((g.y - py) * st);
        az = az + ((g.z - pz) * st);
    }

    float nxp = px + ax, nyp = py + ay, nzp = pz + az;
    if (k.dims == 2u) nzp = pz;
    const float4 xs = (ph >= PS_PHASE_CLOTH) ? b.X[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const uint64_t iter = b.status->iter + it;
    float4 wrec;
    uint32_t set = walls(k, wall_box(k, b, i, a.orig), ph, xs, nxp, nyp, nzp, iter, wrec);
    if (GEN && (mark & kMarkPin)) {
        const float4 t = b.pin_xyz[b.pin_of[a.orig] - 1];
        nxp = t.x;
        nyp = t.y;
        nzp = t.z;
        set |= 7u | kPinned;
    }
    if (TAPE) {
        b.clamp_rec[i] = (uint8_t)set;
        if (set & kWallFriction) b.wall_rec[i] = wrec;
        b.tape_f[i] = tape;
    }
    b.Q[i] = make_float4(nxp, nyp, nzp, 0.0f);
    if (TAPE && b.tape_q) b.tape_q[i] = make_float4(nxp, nyp, nzp, 0.0f);
}

// ---------------------------------------------------------------------------
// a11: v = (x - x*)/dt (subtract_functor, integration_kernel.cuh:465-475)
// plus XSPH over fluid neighbours from displacements u = x - x*:
//   v_i = u_i/dt + ((c/rho0_i) sum_j (u_j - u_i) m_j W_ij)/dt
// with the pair term (u_j - u_i) m_j t^3, t = h^2 - r^2, and poly6
// multiplying the finished sum.  Four lanes per particle: lane hh sums
// quarter hh of the table (its chunks hh, hh + 4, ..., in table order), and
// two shuffles add the quarters as (q0 + q2) + (q1 + q3).  Its one sum is
// short (about 17 VALU per pair), so the kernel is bound by latency more
// than by issue: four lanes give the 256 particles of a staged unit (24
// bytes of LDS per slot, two units per CU) eight wavefronts per SIMD.

static constexpr uint32_t kFinalizeStagedBlock = 4u * kStageUnit;

template <bool UNIFORM, bool STAGED, bool MASS = false>
__global__ __launch_bounds__(STAGED ? kFinalizeStagedBlock : kMaxBlock) void finalize_k(
    DevBuffers b, KConst k, uint32_t n, float mu, float dt, uint32_t its)
{
    // staged: neighbour position and displacement u = p - x* (x, y, z, u.x)
    // and (u.y, u.z), formed with the same subtractions as the global path
    // (and the sentinel record).  In a scene that is not a uniform fluid a
    // particle that is not fluid is staged at infinity: the XSPH sum leaves
    // it out, as the global path does by its x*.w < 0.  With every fluid
    // particle of one mass (mu >= 0) the mass is mu; with fluid masses that
    // differ (MASS) each slot's mass (x*.w) is staged as well, 12 KB more
    // LDS (one block per CU instead of two).  A unit that was not staged
    // gathers from global memory.
    __shared__ float4 lds_pu[STAGED ? kStageSlots + 1 : 1];
    __shared__ float2 lds_u[STAGED ? kStageSlots + 1 : 1];
    __shared__ float lds_m[STAGED && MASS ? kStageSlots + 1 : 1];
    const uint32_t unit = xcd_block();
    const uint32_t hh = threadIdx.x & 3u;
    const uint32_t i = STAGED ? unit * kStageUnit + (threadIdx.x >> 2) : (unit * blockDim.x + threadIdx.x) >> 2;
    bool staged = false;
    // staged: the particle's own records and the first chunks of its table
    // go in flight with the staging loads, as in lambda_k
    StagedTable<4, 2, false> tab;
    float4 p, x;
    Attr a;
    uint32_t c = 0;
    if (STAGED) {
        const StageDesc *d = b.stage + unit;
        StageSrc<kFinalizeStagedBlock> ss;
        const uint32_t ic = min(i, n - 1u);
        ss.load(d);
        tab.load(b, ic, hh);
        p = b.P[ic];
        x = b.X[ic];
        a = b.A[ic];
        c = b.ncnt[ic];
        staged = d->staged != 0u;
        const uint32_t nch = d->nchunks;
        const float inf = __builtin_inff();
        if (staged && threadIdx.x == 0) {
            lds_pu[kStageSentinel] = make_float4(inf, inf, inf, 0.0f);
            lds_u[kStageSentinel] = make_float2(0.0f, 0.0f);
            if (MASS) lds_m[kStageSentinel] = 0.0f;
        }
        if (MASS && staged)
            stage_copy<3>(ss, nch, n, [&](uint32_t j) { return PX{b.P[j], b.X[j]}; },
                          [&](uint32_t l, const PX &v) {
                              lds_pu[l] = v.x.w < 0.0f ? make_float4(inf, inf, inf, 0.0f)
                                                       : make_float4(v.p.x, v.p.y, v.p.z, v.p.x - v.x.x);
                              lds_u[l] = make_float2(v.p.y - v.x.y, v.p.z - v.x.z);
                              lds_m[l] = v.x.w;
                          });
        else if (staged)
            stage_copy<3>(ss, nch, n, [&](uint32_t j) { return PX{b.P[j], b.X[j]}; },
                          [&](uint32_t l, const PX &v) {
                              lds_pu[l] = !UNIFORM && v.x.w < 0.0f ? make_float4(inf, inf, inf, 0.0f)
                                                                   : make_float4(v.p.x, v.p.y, v.p.z, v.p.x - v.x.x);
                              lds_u[l] = make_float2(v.p.y - v.x.y, v.p.z - v.x.z);
                          });
    }
    // every solve of this substep has completed
    if (i == 0 && hh == 0) b.status->iter += its;
    if (i >= n) return;  // the four lanes of a particle leave together
    if (!STAGED) {
        p = b.P[i];
        x = b.X[i];
        a = b.A[i];
        c = b.ncnt[i];
    }
    const float ux = p.x - x.x, uy = p.y - x.y, uz = p.z - x.z;
    float vx = ux / dt, vy = uy / dt, vz = uz / dt;
    if ((UNIFORM || a.phase == PS_PHASE_FLUID) && k.xsph_c != 0.0f) {
        // the XSPH sum of this lane's quarter of the table
        struct Sums {
            float sx, sy, sz;
        };
        Sums s = {0.0f, 0.0f, 0.0f};
        // qj: neighbour position, e: its displacement over the substep
        auto body = [&](const float4 &qj, float ex, float ey, float ez, float mj) {
            float dx = p.x - qj.x, dy = p.y - qj.y, dz = p.z - qj.z;
            float r2 = dist2(dx, dy, dz);
            if (!(r2 < k.h2)) return;
            float t = k.h2 - r2;
            float m = ((t * t) * t) * mj;
            s.sx = __builtin_fmaf(ex - ux, m, s.sx);
            s.sy = __builtin_fmaf(ey - uy, m, s.sy);
            s.sz = __builtin_fmaf(ez - uz, m, s.sz);
        };
        struct PU {
            float4 pu;
            float2 u;
        };
        auto glob = [&](const PX &d) { body(d.p, d.p.x - d.x.x, d.p.y - d.x.y, d.p.z - d.x.z, mu); };
        // the neighbour's mass from x*.w (the sort's 1/w for a fluid
        // particle, -1 for any other: left out)
        auto gen = [&](const PX &d) {
            if (d.x.w < 0.0f) return;
            body(d.p, d.p.x - d.x.x, d.p.y - d.x.y, d.p.z - d.x.z, d.x.w);
        };
        struct PUM {
            float4 pu;
            float2 u;
            float m;
        };
        if (STAGED && MASS && staged)
            tab.visit(
                hh, c, [&](uint32_t l) { return PUM{lds_pu[l], lds_u[l], lds_m[l]}; },
                [&](uint32_t, const PUM &d) { body(d.pu, d.pu.w, d.u.x, d.u.y, d.m); });
        else if (STAGED && staged)
            tab.visit(
                hh, c, [&](uint32_t l) { return PU{lds_pu[l], lds_u[l]}; },
                [&](uint32_t, const PU &d) { body(d.pu, d.pu.w, d.u.x, d.u.y, mu); });
        else
            for_neighbors_strided_chunked(
                b, i, c, hh, 4u, [&](uint32_t j) { return PX{b.P[j], b.X[j]}; },
                [&](uint32_t, const PX &d) {
                    if (UNIFORM)
                        glob(d);
                    else
                        gen(d);
                });
        // lanes 0 and 1 form q0 + q2 and q1 + q3, lane 0 their sum
        s.sx = s.sx + __shfl_xor(s.sx, 2, 64);
        s.sy = s.sy + __shfl_xor(s.sy, 2, 64);
        s.sz = s.sz + __shfl_xor(s.sz, 2, 64);
        const Sums o = {__shfl_xor(s.sx, 1, 64), __shfl_xor(s.sy, 1, 64), __shfl_xor(s.sz, 1, 64)};
        const float sx = k.poly6 * (s.sx + o.sx), sy = k.poly6 * (s.sy + o.sy), sz = k.poly6 * (s.sz + o.sz);
        const float cr = k.xsph_c / a.rho0;
        vx = vx + ((cr * sx) / dt);
        vy = vy + ((cr * sy) / dt);
        vz = vz + ((cr * sz) / dt);
    }
    if (hh) return;  // the particle's lane 0 writes
    b.V[i] = make_float4(vx, vy, vz, 0.0f);
}

// Sleeping (Particle::confirmGuess, cpu/src/particle.h:60-65): a particle
// that moved less than 1e-4 keeps its start position and gets v = 0.
__global__ __launch_bounds__(kBlock) void sleep_k(DevBuffers b, uint32_t n)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float4 p = b.P[i];
    const float4 x = b.X[i];
    float ex = p.x - x.x, ey = p.y - x.y, ez = p.z - x.z;
    float l = sqrtf(((ex * ex) + (ey * ey)) + (ez * ez));
    if (l < 1e-4f) {
        b.V[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        b.P[i] = make_float4(x.x, x.y, x.z, 0.0f);
    }
}

// ---------------------------------------------------------------------------
// launchers

thread_local LaunchEvents g_launch_events;

static inline uint32_t blocks_for(uint32_t n, uint32_t bs = kBlock) { return (n + bs - 1) / bs; }

uint32_t scan_tiles(uint32_t num_cells) { return (num_cells + kScanTile - 1) / kScanTile; }

hipError_t launch_predict_hash(hipStream_t st, const DevBuffers &b, const KConst &k, uint32_t n,
                               float dt, bool predict, bool hash, uint32_t bs)
{
    if (n == 0) return hipSuccess;
    const dim3 g(blocks_for(n, bs)), t(bs);
    if (predict && hash)
        PS_LAUNCH((predict_hash_k<true, true>), g, t, 0, st, b, k, n, dt);
    else if (predict)
        PS_LAUNCH((predict_hash_k<true, false>), g, t, 0, st, b, k, n, dt);
    else if (hash)
        PS_LAUNCH((predict_hash_k<false, true>), g, t, 0, st, b, k, n, dt);
    return hipGetLastError();
}

hipError_t launch_scan(hipStream_t st, const DevBuffers &b, uint32_t num_cells)
{
    const uint32_t tiles = scan_tiles(num_cells);
    const dim3 t(kScanTile / 4);
    if (tiles <= kScanDirect) {
        hipLaunchKernelGGL(scan_k<true>, dim3(tiles), t, 0, st, b.cell_count, b.scan_part, b.cell_off, num_cells);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(scan_partials_k, dim3(tiles), dim3(kBlock), 0, st, b.cell_count, b.scan_part, num_cells);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(scan_k<false>, dim3(tiles), t, 0, st, b.cell_count, b.scan_part, b.cell_off, num_cells);
    return hipGetLastError();
}

hipError_t launch_scatter(hipStream_t st, const DevBuffers &b, uint32_t n)
{
    if (n == 0) return hipSuccess;
    PS_LAUNCH(scatter_k, dim3(blocks_for(n)), dim3(kBlock), 0, st, b, n);
    return hipGetLastError();
}

hipError_t launch_reorder(hipStream_t st, const DevBuffers &b, uint32_t n, uint32_t bs, float mj_solid)
{
    if (n == 0) return hipSuccess;
    PS_LAUNCH(reorder_k, dim3(blocks_for(n, bs)), dim3(bs), 0, st, b, n, mj_solid);
    return hipGetLastError();
}

hipError_t launch_neighbors(hipStream_t st, const DevBuffers &b, const KConst &k, uint32_t n,
                            uint32_t kmax, uint32_t bs)
{
    if (n == 0) return hipSuccess;
    if (b.staging) {
        // few units: their search split over four blocks each
        const uint32_t units = blocks_for(n, kStageUnit);
        const dim3 t(kStageUnit);
        if (units <= kNbrSplitUnits && b.nbr_glob)  // recording: the global-slot copy as well
            PS_LAUNCH(neighbors_split_k<true>, dim3(kNbrParts * units), t, 0, st, b, k, n, kmax);
        else if (units <= kNbrSplitUnits)
            PS_LAUNCH(neighbors_split_k<false>, dim3(kNbrParts * units), t, 0, st, b, k, n, kmax);
        else if (b.nbr_glob)
            PS_LAUNCH(neighbors_staged_k<true>, dim3(units), t, 0, st, b, k, n, kmax);
        else
            PS_LAUNCH(neighbors_staged_k<false>, dim3(units), t, 0, st, b, k, n, kmax);
    }
    else
        PS_LAUNCH(neighbors_k, dim3(blocks_for(n, bs)), dim3(bs), 0, st, b, k, n, kmax);
    return hipGetLastError();
}

hipError_t launch_lambda(hipStream_t st, const DevBuffers &b, const KConst &k, uint32_t n,
                         bool uniform, float wu, uint32_t bs)
{
    if (n == 0) return hipSuccess;
    const float mu = 1.0f / wu;
    // staged: two lanes per particle
    const uint32_t threads = b.staging ? 2u * kStageUnit : bs;
    const uint32_t blocks = blocks_for(n, b.staging ? kStageUnit : bs);
    const dim3 t(threads);
    ConBlocks con{};
    if (uniform) {
        const dim3 g(blocks);
        if (b.tape_lq && b.staging)  // recording for the reverse pass
            PS_LAUNCH((lambda_k<true, true, true>), g, t, 0, st, b, k, n, mu, con);
        else if (b.tape_lq)
            PS_LAUNCH((lambda_k<true, false, true>), g, t, 0, st, b, k, n, mu, con);
        else if (b.staging)
            PS_LAUNCH((lambda_k<true, true>), g, t, 0, st, b, k, n, mu, con);
        else
            PS_LAUNCH((lambda_k<true, false>), g, t, 0, st, b, k, n, mu, con);
        return hipGetLastError();
    }
    // the constraint blocks first, as many launches of them alone as it takes
    // until the rest fits in one with the fluid's
    const ConParts parts = con_parts(b.nwalk, b.nlink, b.nbody, threads);
    con.walks = parts.walks;
    con.links = parts.links;
    // contact lists of the global-slot variants (the staged ones' share the
    // staged cells' LDS)
    const size_t cl = b.nwalk ? sizeof(uint32_t) * kContactList * bs : 0;
    for (;;) {
        const ConLaunch part = con_launch(parts.all, con.first, blocks, threads);
        con.blocks = part.blocks;
        const dim3 g(part.blocks + (part.last ? blocks : 0u));
        if (b.tape_lq && b.staging)
            PS_LAUNCH((lambda_k<false, true, true>), g, t, 0, st, b, k, n, mu, con);
        else if (b.tape_lq)
            PS_LAUNCH((lambda_k<false, false, true>), g, t, cl, st, b, k, n, mu, con);
        else if (b.staging)
            PS_LAUNCH((lambda_k<false, true>), g, t, 0, st, b, k, n, mu, con);
        else
            PS_LAUNCH((lambda_k<false, false>), g, t, cl, st, b, k, n, mu, con);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess || part.last) return e;
        con.first += part.blocks;
    }
}

// NC: tensile exponent known at compile time (4, as in the reference's
// E_P, integration_kernel.cuh:34) or 0 = read from the parameters
template <bool GEN, bool UNIFORM, uint32_t NC>
static void solve_variant(hipStream_t st, const DevBuffers &b, const KConst &k, uint32_t n, float wu, uint32_t iter,
                          uint32_t bs)
{
    const dim3 g(blocks_for(n, bs)), t(bs);
    const dim3 gs(blocks_for(n, kStageUnit)), ts(2 * kStageUnit);  // two lanes per particle
    if (b.tape_f && b.staging)  // recording for the reverse pass
        PS_LAUNCH((solve_k<GEN, UNIFORM, NC, true, true>), gs, ts, 0, st, b, k, n, wu, iter);
    else if (b.tape_f)
        PS_LAUNCH((solve_k<GEN, UNIFORM, NC, false, true>), g, t, 0, st, b, k, n, wu, iter);
    else if (b.staging)
        PS_LAUNCH((solve_k<GEN, UNIFORM, NC, true>), gs, ts, 0, st, b, k, n, wu, iter);
    else
        PS_LAUNCH((solve_k<GEN, UNIFORM, NC, false>), g, t, 0, st, b, k, n, wu, iter);
}

template <uint32_t NC>
static void solve_composition(hipStream_t st, const DevBuffers &b, const KConst &k, uint32_t n, uint32_t features,
                              bool uniform, float wu, uint32_t iter, uint32_t bs)
{
    if (features != F_FLUID)
        solve_variant<true, false, NC>(st, b, k, n, wu, iter, bs);
    else if (uniform)
        solve_variant<false, true, NC>(st, b, k, n, wu, iter, bs);
    else
        solve_variant<false, false, NC>(st, b, k, n, wu, iter, bs);
}

hipError_t launch_solve(hipStream_t st, const DevBuffers &b, const KConst &k, uint32_t n,
                        uint32_t features, bool uniform, float wu, uint32_t iter, uint32_t bs)
{
    if (n == 0) return hipSuccess;
    if (k.n_corr == 4u)
        solve_composition<4>(st, b, k, n, features, uniform, wu, iter, bs);
    else
        solve_composition<0>(st, b, k, n, features, uniform, wu, iter, bs);
    return hipGetLastError();
}

hipError_t launch_finalize(hipStream_t st, const DevBuffers &b, const KConst &k, uint32_t n,
                           float dt, bool sleeping, bool uniform, float wu, float wf, uint32_t its,
                           uint32_t bs)
{
    if (n == 0) return hipSuccess;
    // four lanes per particle (bs is a multiple of 64)
    const dim3 g(blocks_for(n, bs / 4u)), t(bs);
    const float mu = 1.0f / wu;
    if (uniform && b.staging)
        PS_LAUNCH((finalize_k<true, true>), dim3(blocks_for(n, kStageUnit)),
                           dim3(kFinalizeStagedBlock), 0, st, b, k, n, mu, dt, its);
    else if (b.staging && wf >= 0.0f)  // every fluid particle of inverse mass wf
        PS_LAUNCH((finalize_k<false, true>), dim3(blocks_for(n, kStageUnit)),
                           dim3(kFinalizeStagedBlock), 0, st, b, k, n, 1.0f / wf, dt, its);
    else if (b.staging)  // fluid masses that differ: staged with each slot's mass
        PS_LAUNCH((finalize_k<false, true, true>), dim3(blocks_for(n, kStageUnit)),
                           dim3(kFinalizeStagedBlock), 0, st, b, k, n, -1.0f, dt, its);
    else if (uniform)
        PS_LAUNCH((finalize_k<true, false>), g, t, 0, st, b, k, n, mu, dt, its);
    else
        PS_LAUNCH((finalize_k<false, false>), g, t, 0, st, b, k, n, mu, dt, its);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !sleeping) return e;
    hipLaunchKernelGGL(sleep_k, dim3(blocks_for(n)), dim3(kBlock), 0, st, b, n);
    return hipGetLastError();
}

}  // namespace ps
