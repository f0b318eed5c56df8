// ps_adjoint.hip — reverse-mode adjoint of one substep (ps_step_backward).
//
// The forward map of a substep is predict -> I Jacobi iterations -> velocity
// + XSPH.  With the neighbour table, the contact sets and counts, the
// coordinates walls and pins set and the wall-friction branches frozen (as
// the recomputed forward pass recorded them), each piece is smooth and its
// vector-Jacobian product is written out by hand below.  Every transposed
// sum is a gather over the particle's own neighbour table, which holds the
// same pairs as its neighbours' tables (r^2 < R^2 is symmetric and no table
// overflowed), so there are no scatters and no atomics: four or sixteen lanes
// per particle, sums in table order.  The
// arithmetic is the CPU oracle's, operation by operation (built with
// -ffp-contract=off), so FP32 gradients match it bit for bit.
//
// Per iteration, with y = p + Delta before walls and pins:
//   Delta_i = f_i / rho0_i (fluid) + contacts + distance terms,
//   f_i = sum_j (l_i + l_j + s_ij) G_ij, G_ij = -b(r) d_ij,
//   b = spiky (h - r)^2 / r (G = (0, -gdeg, 0) for a degenerate pair),
//   l_i = -C_i / (D_i + eps), C_i = rho_i / rho0_i - 1,
//   D_i = sum_j a_ij^2 r^2 + |S_i|^2, S_i = sum_j a_ij d_ij, a = b / rho0_i.
// Kernels per reversed iteration: adj_lambda_k (dL/dl -> dL/dC, dL/dD),
// adj_position_k (dL/dp: pair, density, D, contact and distance terms, and
// dL/dstiffness per constraint), which ends with the next iteration's
// pre-step (adj_pre_one: walls, pins and wall friction backwards, the rho0
// term of f).  Per substep: adj_xsph_k and adj_finalize_k (velocity + XSPH
// backwards, then the last iteration's pre-step) before the iterations,
// adj_predict_k after them.

#include "ps_device.hpp"

namespace ps {

// The kernels that gather over the neighbour table map blocks with
// xcd_block(), so each XCD reverses one contiguous range of sorted particles
// and its L2 holds that region's records.
static constexpr uint32_t kAdjBlock = 256;

__device__ __forceinline__ float dot3(const float *a, const float *b)
{
    return ((a[0] * b[0]) + (a[1] * b[1])) + (a[2] * b[2]);
}

// G_ij for d = p_i - p_j (r2 = |d|^2 < h2)
__device__ __forceinline__ void adj_gamma(const KConst &k, const float *dv, float r2, float *g)
{
    if (r2 < kDegenerateR2) {
        g[0] = 0.0f;
        g[1] = -((k.spiky * (k.h * k.h)) * 0.001f);
        g[2] = 0.0f;
        return;
    }
    const float ri = rsq(r2);
    const float q = k.h - (r2 * ri);
    const float bb = (k.spiky * (q * q)) * ri;
    for (int a = 0; a < 3; a++) g[a] = -(bb * dv[a]);
}

// gradient of W_poly6(|d|) in d: -6 poly6 (h^2 - r^2)^2 d
__device__ __forceinline__ void adj_grad_w6(const KConst &k, const float *dv, float r2, float *g)
{
    const float t = k.h2 - r2;
    const float c = -((6.0f * k.poly6) * (t * t));
    for (int a = 0; a < 3; a++) g[a] = c * dv[a];
}

// Cloth contact of owner i with j (collideD without friction: a distance
// constraint of rest collide_dist, stiffness 1, count nc): M^T y for
// M = -(w_i / (wsum nc)) [(1 - cd/r) I + (cd/r^3) d d^T]; false when the
// pair is not in i's contact set.
__device__ __forceinline__ bool adj_contact(const KConst &k, float wi, int32_t ph, float wj, int32_t phj,
                                            uint32_t nci, const float *dv, const float *y, float *out)
{
    if (ph < PS_PHASE_CLOTH || wi == 0.0f || nci == 0u) return false;
    if (ph > PS_PHASE_SOLID && ph == phj) return false;
    const float r2 = ((dv[0] * dv[0]) + (dv[1] * dv[1])) + (dv[2] * dv[2]);
    if (!(r2 < k.collide_r2)) return false;
    const float dist = sqrtf(r2);
    if (dist < 1e-6f) return false;
    const float wsum = wi + wj;
    if (wsum == 0.0f) return false;
    const float cf = -((wi / wsum) / (float)nci);
    const float k1 = 1.0f - (k.collide_dist / dist), k2 = k.collide_dist / ((dist * dist) * dist);
    const float dy = dot3(dv, y);
    for (int a = 0; a < 3; a++) out[a] = cf * ((k1 * y[a]) + ((k2 * dy) * dv[a]));
    return true;
}

// masked dL/dy of particle i as the Jacobian uses it (z dropped in 2D)
__device__ __forceinline__ void yd_of(const KConst &k, const float4 &Y, float *yd)
{
    yd[0] = Y.x;
    yd[1] = Y.y;
    yd[2] = k.dims == 2u ? 0.0f : Y.z;
}

// Both owners' fluid terms of the pair (p, j) in dL/dp_p, d = p_p - p_j:
// E_p - E_j, with E_i = d/dd [mu_i . (l_i + l_j + s(d)) G(d)] for owner i
// (J_G = -(b I + (b'/r) d d^T), b' = -spiky (h - r)(h + r) / r^2), plus
// cm_p g6(d) - cm_j g6(-d) (the density term, g6 = dW/dd) and
// Db_p dD_p(d) - Db_j dD_j(-d) (dD_i/dd of the denominator D_i).  Folded
// into one expression,
//   (alpha - K mD + cms c6) d + 2A dV - cb dmu,
//   dmu = mu_p - mu_j, mD = d.dmu, K = b cc + coef b'/r, cb = coef b,
//   dV = V_p - V_j, alpha = C us - 2 Bq (d.dV), us = u_p + u_j,
//   A = (h - r)^2 / r, Bq = (h - r)(h + r) / r^3, C = -4 (h - r)^3 / r,
//   cms = Cr_p m_j + Cr_j m_p,
// with the per-particle factors of adj_lambda_k (MC: mu, Cr; KV: V, u).  An
// owner that does not take part (op, oj false) enters with zeros.  cc and
// c6 are the tensile term's and W's gradient factors (dW/dd = c6 d).  A
// degenerate pair (G the constant (0, g0y, 0) for both owners) adds
// (cc g0y (mu_p.y + mu_j.y) + cms c6) d.  The sum goes to out.
__device__ __forceinline__ void adj_pair_sum(const KConst &k, const float *dv, float r2, float lsum, bool op,
                                             bool oj, const float4 &mcp, const float4 &mcj, const float4 &kvp,
                                             const float4 &kvj, float massp, float massj, float *out)
{
    const float t = k.h2 - r2;
    const float tt = t * t;
    const float W = k.poly6 * (tt * t);
    const float x = W * k.inv_w_dq;
    const uint32_t n = k.n_corr;
    const float s = -(k.k_corr * ipow(x, n));
    const float xn1 = n > 1u ? ipow(x, n - 1u) : 1.0f;
    const float cc = (((k.k_corr * (float)n) * xn1) * k.inv_w_dq) * ((6.0f * k.poly6) * tt);
    const float c6 = -((6.0f * k.poly6) * tt);
    const float coef = lsum + s;
    const float mup[3] = {op ? mcp.x : 0.0f, op ? mcp.y : 0.0f, op ? mcp.z : 0.0f};
    const float muj[3] = {oj ? mcj.x : 0.0f, oj ? mcj.y : 0.0f, oj ? mcj.z : 0.0f};
    const float cms = (op ? mcp.w * massj : 0.0f) + (oj ? mcj.w * massp : 0.0f);
    if (r2 < kDegenerateR2) {
        const float g0y = -((k.spiky * (k.h * k.h)) * 0.001f);
        const float be = (cc * (g0y * (mup[1] + muj[1]))) + (cms * c6);
        for (int a = 0; a < 3; a++) out[a] = be * dv[a];
        return;
    }
    const float ri = rsq(r2);
    const float r = r2 * ri;
    const float q = k.h - r;
    const float qq = q * q;
    const float bb = (k.spiky * qq) * ri;
    const float bp = -(((k.spiky * q) * (k.h + r)) * (ri * ri));
    const float dmu[3] = {mup[0] - muj[0], mup[1] - muj[1], mup[2] - muj[2]};
    const float mD = dot3(dv, dmu);
    const float K = (bb * cc) + (coef * (bp * ri));
    const float cb = coef * bb;
    const float A2 = 2.0f * (qq * ri);
    const float Bq = ((q * (k.h + r)) * (ri * ri)) * ri;
    const float C = -((4.0f * (qq * q)) * ri);
    const float us = (op ? kvp.w : 0.0f) + (oj ? kvj.w : 0.0f);
    const float dV[3] = {(op ? kvp.x : 0.0f) - (oj ? kvj.x : 0.0f), (op ? kvp.y : 0.0f) - (oj ? kvj.y : 0.0f),
                         (op ? kvp.z : 0.0f) - (oj ? kvj.z : 0.0f)};
    const float vD = dot3(dv, dV);
    const float al = (C * us) - ((2.0f * Bq) * vD);
    const float be = (al - (K * mD)) + (cms * c6);
    for (int a = 0; a < 3; a++) out[a] = (be * dv[a]) + ((A2 * dV[a]) - (cb * dmu[a]));
}

// density multiplier of a neighbour in rho_i
__device__ __forceinline__ float adj_mass(const KConst &k, float wj, int32_t phj)
{
    float m = 1.0f / wj;
    if (phj != PS_PHASE_FLUID) m = m * k.s_solid;
    return m;
}

// Neighbour records of the gathers.  UNIFORM (every particle fluid, one
// inverse mass) variants leave out the attribute loads.
struct GLam {
    float4 p, m;
};
struct GLamAttr {
    float4 p, m;
    AdjAttr a;
};
struct GPos {
    float4 p, mc, kv;
};
struct GPosAttr {
    float4 p, mc, kv;
    AdjAttr a;
};
struct GXA {
    float4 p, x;
    Attr a;
};
struct GXY {
    float4 p, x, y;
};
struct GXYA {
    float4 p, x, y;
    Attr a;
};

// ---------------------------------------------------------------------------
// The gathers take 4 U lanes a particle: quarter h of its table is lanes U h
// .. U h + U - 1, each forming the terms of one entry of a chunk at a time,
// and all U add them in table order, so each holds the quarter's sum; then
// (q0 + q2) + (q1 + q3) in every lane.  A term left out is -0, which changes
// no sum it is added to.

// s and the U lanes' terms v (then w), lane by lane
template <uint32_t U, int S = 0>
__device__ __forceinline__ float group_add(float s, float v)
{
    s = s + group_value<U, S>(v);
    if constexpr (S + 1 < (int)U) s = group_add<U, S + 1>(s, v);
    return s;
}
template <uint32_t U, int S = 0>
__device__ __forceinline__ float group_add(float s, float v, float w)
{
    s = (s + group_value<U, S>(v)) + group_value<U, S>(w);
    if constexpr (S + 1 < (int)U) s = group_add<U, S + 1>(s, v, w);
    return s;
}
template <uint32_t U, int S = 0>
__device__ __forceinline__ float group_add(float s, float v, float w, float x)
{
    s = ((s + group_value<U, S>(v)) + group_value<U, S>(w)) + group_value<U, S>(x);
    if constexpr (S + 1 < (int)U) s = group_add<U, S + 1>(s, v, w, x);
    return s;
}
template <uint32_t U, int S = 0>
__device__ __forceinline__ float group_fma(float s, float v, float w)
{
    s = __builtin_fmaf(group_value<U, S>(v), group_value<U, S>(w), s);
    if constexpr (S + 1 < (int)U) s = group_fma<U, S + 1>(s, v, w);
    return s;
}

// The same over sixteen lanes, lane l adding its terms to the sum of those
// before it (every lane's values fetched at once would take 96 registers).
__device__ __forceinline__ float row_add(float s, float v, float w)
{
    s = (s + v) + w;
#pragma unroll
    for (int l = 1; l < 16; l++)
        s = (__int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(s), 0x111, 0xf, 0xf, true)) + v) + w;
    return group_value<16, 15>(s);
}

// the quarters' sums q0..q3 as (q0 + q2) + (q1 + q3)
template <uint32_t U>
__device__ __forceinline__ float quarters_sum(float s)
{
    s = s + __shfl_xor(s, 2 * U, 64);
    return s + __shfl_xor(s, U, 64);
}

// ---------------------------------------------------------------------------
// Pins, walls and wall friction backwards, and the fluid sum's rho0 term,
// of one particle (the pre-step of a reversed iteration, from the recorded
// forward quantities: f and the contact count of the solve, the clamp bits
// and wall-friction records of walls()), for g = dL/dp after the iteration.
// Wall friction (walls(): p'' = p' - t f, t = e - (e.n) n, e = p' - x*):
// static, or kinetic clamped to f = 1: dp''/dp' = n n^T,
// dp''/dx* = I - n n^T; kinetic with f = wall_k / l < 1:
// dp''/dp' = I - wall_k K (I - n n^T), K = (I - t^ t^T) / l, the x* part its
// negative second term, and dp''/dwall_k = -t / l.  Writes the iteration's
// Yn (masked dL/dy), M = (mu = yd / rho0 for fluid, yd otherwise; 1 / rho0)
// and the attribute record ABn the later kernels gather; updates xsb, wkb
// and r0b.  Run at the end of the kernel that forms g (adj_finalize_k,
// adj_position_k), by the particle's lane 0.
// The caller loads the records (AdjPreIn), early where registers allow, so
// that this tail waits on no load unless the particle has wall friction.
struct AdjPreIn {
    uint32_t cl;  // clamp bits
    float4 tf;    // recorded fluid sum and contact count
    float r0b;    // dL/drho0 so far
};

__device__ __forceinline__ AdjPreIn adj_pre_load(const AdjBuffers &a, uint32_t i)
{
    AdjPreIn q;
    q.cl = a.clampn[i];
    q.tf = a.tfn[i];
    q.r0b = a.r0b[i];
    return q;
}

template <bool UNIFORM>
__device__ __forceinline__ void adj_pre_one(const DevBuffers &b, const KConst &k, const AdjBuffers &a,
                                            uint32_t i, const Attr &ai, const AdjPreIn &in, float *g)
{
    const uint32_t cl = in.cl;
    const float4 tf = in.tf;
    if (cl & kPinned) {
        g[0] = g[1] = g[2] = 0.0f;
    } else if (cl & kWallFriction) {
        const float4 rec = a.wrecn[i];
        const float4 xs = b.X[i];
        const int code = (int)rec.w;
        const float nn[3] = {(float)(code / 9 - 1), (float)((code / 3) % 3 - 1), (float)(code % 3 - 1)};
        const float e[3] = {rec.x - xs.x, rec.y - xs.y, rec.z - xs.z};
        const float dn = dot3(e, nn);
        const float t[3] = {e[0] - (dn * nn[0]), e[1] - (dn * nn[1]), e[2] - (dn * nn[2])};
        float4 xb = a.xsb[i];
        float xv[3] = {xb.x, xb.y, xb.z};
        if (!(cl & kWallKinetic)) {
            const float ng = dot3(nn, g);
            for (int q = 0; q < 3; q++) {
                const float pa = ng * nn[q];
                xv[q] = xv[q] + (g[q] - pa);
                g[q] = pa;
            }
        } else {
            const float l = sqrtf(dot3(t, t));
            const float tg = dot3(t, g);
            float kg[3];
            for (int q = 0; q < 3; q++) kg[q] = (g[q] - ((t[q] * tg) / (l * l))) / l;
            const float nk = dot3(nn, kg);
            for (int q = 0; q < 3; q++) {
                const float qq = k.wall_k * (kg[q] - (nk * nn[q]));
                xv[q] = xv[q] + qq;
                g[q] = g[q] - qq;
            }
            a.wkb[i] = a.wkb[i] - (tg / l);
        }
        a.xsb[i] = make_float4(xv[0], xv[1], xv[2], 0.0f);
    }
    for (int q = 0; q < 3; q++)
        if (cl & (1u << q)) g[q] = 0.0f;
    const float yd[3] = {g[0], g[1], k.dims == 2u ? 0.0f : g[2]};
    const bool fl = UNIFORM || ai.phase == PS_PHASE_FLUID;
    const float ir0 = 1.0f / ai.rho0;
    if (fl) {
        const float f[3] = {tf.x, tf.y, tf.z};
        a.r0b[i] = in.r0b - (dot3(yd, f) * (ir0 * ir0));
    }
    a.Yn[i] = make_float4(g[0], g[1], g[2], 0.0f);
    a.M[i] = fl ? make_float4(yd[0] * ir0, yd[1] * ir0, yd[2] * ir0, ir0) : make_float4(yd[0], yd[1], yd[2], ir0);
    if (!UNIFORM) {
        const uint32_t nc = __float_as_uint(tf.w);
        a.nc[i] = nc;
        a.ABn[i] = AdjAttr{ai.w, ai.phase, nc, adj_mass(k, ai.w, ai.phase)};
    }
}

// dL/dl -> dL/dC = -lb / (D + eps), dL/dD = -lb l / (D + eps); rho0 terms.
// Lane 0 of a particle finishes.
template <bool UNIFORM, uint32_t U>
__global__ __launch_bounds__(kAdjBlock) void adj_lambda_k(DevBuffers b, KConst k, AdjBuffers a, uint32_t n)
{
    const uint32_t i = xcd_block() * (kAdjBlock / (4u * U)) + threadIdx.x / (4u * U);
    const uint32_t lane = threadIdx.x % (4u * U);
    if (i >= n) return;  // the lanes of a particle leave together
    // every per-particle load goes out before the first wait (lane 0's
    // finish would otherwise wait on three more after the sum)
    const float4 mi = a.M[i];
    const int32_t phi = UNIFORM ? (int32_t)PS_PHASE_FLUID : b.A[i].phase;
    const float4 pi = a.Pit[i];
    const uint32_t c = b.ncnt[i];
    const float4 sd = a.SD[i];
    const float rhoi = a.rho[i];
    float r = a.r0b[i];
    if (!UNIFORM && phi != PS_PHASE_FLUID) {
        if (!lane) {
            a.MC[i] = make_float4(mi.x, mi.y, mi.z, 0.0f);
            a.KV[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        return;
    }
    const float mu[3] = {mi.x, mi.y, mi.z};
    const float ir0 = mi.w;
    float lb = 0.0f;
    auto body = [&](const float4 &pj, const float4 &mj, float wj, int32_t phj, bool used) {
        float own = -0.0f, other = -0.0f;
        const float dv[3] = {pi.x - pj.x, pi.y - pj.y, pi.z - pj.z};
        const float r2 = dist2(dv[0], dv[1], dv[2]);
        if (used && wj != 0.0f && r2 < k.h2) {
            float g[3];
            adj_gamma(k, dv, r2, g);
            own = dot3(mu, g);
            if (phj == PS_PHASE_FLUID) {
                // G(-d) = -G(d) exactly (rounding is symmetric); the
                // degenerate direction is the same for both
                const bool deg = r2 < kDegenerateR2;
                const float gj[3] = {deg ? g[0] : -g[0], deg ? g[1] : -g[1], deg ? g[2] : -g[2]};
                const float muj[3] = {mj.x, mj.y, mj.z};
                other = dot3(muj, gj);
            }
        }
        lb = group_add<U>(lb, own, other);
    };
    constexpr uint32_t kFlight = U == 4 ? 2 : 4;
    if (UNIFORM) {
        for_neighbors_quarter<U, kFlight>(
            b, i, c, lane / U, lane % U, [&](uint32_t j) { return GLam{a.Pit[j], a.M[j]}; },
            [&](const GLam &d, bool used) { body(d.p, d.m, 1.0f, PS_PHASE_FLUID, used); });
    } else {
        for_neighbors_quarter<U, kFlight>(
            b, i, c, lane / U, lane % U, [&](uint32_t j) { return GLamAttr{a.Pit[j], a.M[j], a.AB[j]}; },
            [&](const GLamAttr &d, bool used) { body(d.p, d.m, d.a.w, d.a.phase, used); });
    }
    lb = quarters_sum<U>(lb);
    if (lane) return;
    const float den = sd.w + k.relax;
    const float lam = pi.w;
    const float Cb = -(lb / den);
    const float Db = -((lb * lam) / den);
    r = r - (Cb * (rhoi * (ir0 * ir0)));
    r = r - (Db * ((2.0f * sd.w) * ir0));
    a.r0b[i] = r;
    // the factors adj_position_k combines per pair
    const float sk = k.spiky * ir0;
    const float dk = Db * sk;
    a.MC[i] = make_float4(mu[0], mu[1], mu[2], Cb * ir0);
    a.KV[i] = make_float4(dk * sd.x, dk * sd.y, dk * sd.z, Db * (sk * sk));
}

// dL/dp before the iteration: pair and contact terms (quarter 0 starts from
// dL/dy), then the distance constraints, a lane each, 4 U at a time.
template <bool UNIFORM, uint32_t U>
__global__ __launch_bounds__(kAdjBlock, U == 4 ? 4 : 5) void adj_position_k(DevBuffers b, KConst k, AdjBuffers a, uint32_t n)
{
    const uint32_t p = xcd_block() * (kAdjBlock / (4u * U)) + threadIdx.x / (4u * U);
    const uint32_t lane = threadIdx.x % (4u * U);
    if (p >= n) return;  // the lanes of a particle leave together
    const float4 pp = a.Pit[p];
    const Attr ap = b.A[p];
    const float4 Yp = a.Y[p];
    // a constraint is a chain of loads (list, partner's slot, records); the
    // lane's first kR go out together, ahead of the neighbours' where
    // registers are not short (U = 4)
    struct Link {
        float4 l;
        float3 p, y;
        uint32_t occ;
    };
    uint32_t e0 = 0, e1 = 0;
    constexpr uint32_t kLanes = 4u * U, kR = U == 1 ? 2 : 1;
    Link ln[kR] = {};
    if (a.dist) {
        e0 = b.dist_off[ap.orig];
        e1 = b.dist_off[ap.orig + 1];
    }
    auto links = [&](uint32_t base) {
#pragma unroll
        for (uint32_t r = 0; r < kR; r++) ln[r].l = b.links[min(base + kLanes * r + lane, e1 - 1u)];
        uint32_t j[kR];
#pragma unroll
        for (uint32_t r = 0; r < kR; r++) {
            j[r] = b.slot_of[__float_as_uint(ln[r].l.x)];
            ln[r].occ = b.occ[__float_as_uint(ln[r].l.x)];
        }
#pragma unroll
        for (uint32_t r = 0; r < kR; r++) {
            ln[r].p = reinterpret_cast<const float3 &>(a.Pit[j[r]]);
            ln[r].y = reinterpret_cast<const float3 &>(a.Y[j[r]]);
        }
    };
    if (U == 4 && e0 < e1) links(e0);
    const bool q0 = lane < U;
    float acc[3] = {q0 ? Yp.x : 0.0f, q0 ? Yp.y : 0.0f, q0 ? Yp.z : 0.0f};
    float ydp[3];
    yd_of(k, Yp, ydp);
    const bool pf = UNIFORM || ap.phase == PS_PHASE_FLUID;
    const float4 mcp = a.MC[p];  // mu_p, Cr_p
    const float4 kvp = a.KV[p];  // V_p, u_p
    const uint32_t ncp = UNIFORM ? 0u : a.nc[p];
    const bool contacts = !UNIFORM && a.contacts;
    const float massp = adj_mass(k, ap.w, ap.phase);  // p as a neighbour of j
    auto body = [&](const float4 &pj, const float4 &mcj, const float4 &kvj, float wj, int32_t phj, uint32_t ncj,
                    float massj, bool used) {
        const float dv[3] = {pp.x - pj.x, pp.y - pj.y, pp.z - pj.z};
        const float r2 = dist2(dv[0], dv[1], dv[2]);
        float m[3] = {-0.0f, -0.0f, -0.0f};
        // p owns the pair when fluid and j moves, j when fluid and p moves
        const bool op = pf && wj != 0.0f;
        const bool oj = (UNIFORM || phj == PS_PHASE_FLUID) && ap.w != 0.0f;
        if (used && r2 < k.h2 && (op || oj))
            adj_pair_sum(k, dv, r2, pp.w + pj.w, op, oj, mcp, mcj, kvp, kvj, massp, massj, m);
        // cloth contacts: p's own, then p as the partner of j's (for a
        // non-fluid j, MC holds its masked dL/dy)
        const float dj[3] = {-dv[0], -dv[1], -dv[2]};
        const float ydj[3] = {mcj.x, mcj.y, mcj.z};
        if constexpr (U == 1) {
            for (int q2 = 0; q2 < 3; q2++) acc[q2] = acc[q2] + m[q2];
            if (contacts) {
                if (adj_contact(k, ap.w, ap.phase, wj, phj, ncp, dv, ydp, m))
                    for (int q2 = 0; q2 < 3; q2++) acc[q2] = acc[q2] + m[q2];
                if (adj_contact(k, wj, phj, ap.w, ap.phase, ncj, dj, ydj, m))
                    for (int q2 = 0; q2 < 3; q2++) acc[q2] = acc[q2] - m[q2];
            }
        } else {
            float mo[3] = {-0.0f, -0.0f, -0.0f}, mj[3] = {0.0f, 0.0f, 0.0f};
            bool touch = false;
            if (contacts && used) {
                touch = adj_contact(k, ap.w, ap.phase, wj, phj, ncp, dv, ydp, mo);
                touch = adj_contact(k, wj, phj, ap.w, ap.phase, ncj, dj, ydj, mj) || touch;
            }
            if (contacts && __any(touch))
                for (int q2 = 0; q2 < 3; q2++) acc[q2] = group_add<U>(acc[q2], m[q2], mo[q2], -mj[q2]);
            else
                for (int q2 = 0; q2 < 3; q2++) acc[q2] = group_add<U>(acc[q2], m[q2]);
        }
    };
    const uint32_t c = b.ncnt[p];
    // two records (48 or 64 bytes each) in flight per lane: four would cost
    // registers the waves need
    constexpr uint32_t kFlight = 2;
    if (UNIFORM) {
        for_neighbors_quarter<U, kFlight>(
            b, p, c, lane / U, lane % U, [&](uint32_t j) { return GPos{a.Pit[j], a.MC[j], a.KV[j]}; },
            [&](const GPos &d, bool used) { body(d.p, d.mc, d.kv, ap.w, PS_PHASE_FLUID, 0u, massp, used); });
    } else {
        for_neighbors_quarter<U, kFlight>(
            b, p, c, lane / U, lane % U, [&](uint32_t j) { return GPosAttr{a.Pit[j], a.MC[j], a.KV[j], a.AB[j]}; },
            [&](const GPosAttr &d, bool used) {
                body(d.p, d.mc, d.kv, d.a.w, d.a.phase, d.a.nc, d.a.mass, used);
            });
    }
    for (int q2 = 0; q2 < 3; q2++) acc[q2] = quarters_sum<U>(acc[q2]);
    // distance constraints incident to p, in their order; for a constraint
    // whose first particle p is, also its dL/dstiffness (one writer per
    // constraint): T_a / st = -(w_a / (wsum occ_a)) (1 - L/r) d_ab, and T_b
    // its mirror.  Each lane forms one constraint's p term X and the negative
    // of its j term, Z; all lanes add them in constraint order.
    if (e0 < e1) {
        if (U != 4) links(e0);
        const float occo = (float)b.occ[ap.orig];
        for (uint32_t base = e0;;) {  // the same trip count in the particle's lanes
#pragma unroll
            for (uint32_t r = 0; r < kR; r++) {
                float X[3] = {-0.0f, -0.0f, -0.0f}, Z[3] = {-0.0f, -0.0f, -0.0f};
                const uint32_t e = base + kLanes * r + lane;
                const float wj = ln[r].l.w;
                const float dv[3] = {pp.x - ln[r].p.x, pp.y - ln[r].p.y, pp.z - ln[r].p.z};
                const float dist = sqrtf(((dv[0] * dv[0]) + (dv[1] * dv[1])) + (dv[2] * dv[2]));
                const float wsum = ap.w + wj;
                if (e < e1 && !(dist < 1e-6f || wsum == 0.0f)) {
                    const float L = ln[r].l.y, st = ln[r].l.z;
                    const float k1 = 1.0f - (L / dist), k2 = L / ((dist * dist) * dist);
                    float gs = 0.0f;
                    // M(d) = -(w st / (wsum occ)) [(1 - L/r) I + (L/r^3) d d^T]
                    if (ap.w != 0.0f) {
                        const float cf = -(((ap.w * st) / wsum) / occo);
                        const float dy = dot3(dv, ydp);
                        for (int q2 = 0; q2 < 3; q2++) X[q2] = cf * ((k1 * ydp[q2]) + ((k2 * dy) * dv[q2]));
                        gs = gs - (((ap.w / wsum) / occo) * (k1 * dy));
                    }
                    if (wj != 0.0f) {
                        const float ydj[3] = {ln[r].y.x, ln[r].y.y, k.dims == 2u ? 0.0f : ln[r].y.z};
                        const float cf = -(((wj * st) / wsum) / (float)ln[r].occ);
                        const float dy = dot3(dv, ydj);
                        for (int q2 = 0; q2 < 3; q2++) Z[q2] = -(cf * ((k1 * ydj[q2]) + ((k2 * dy) * dv[q2])));
                        gs = gs + (((wj / wsum) / (float)ln[r].occ) * (k1 * dy));
                    }
                    // the first particle of the constraint (d = p_a - p_b)
                    const uint32_t id = b.link_id[e];
                    if (!(id & 1u)) a.sb[id >> 1] = a.sb[id >> 1] + gs;
                }
                for (int q2 = 0; q2 < 3; q2++)
                    acc[q2] = U == 4 ? row_add(acc[q2], X[q2], Z[q2]) : group_add<kLanes>(acc[q2], X[q2], Z[q2]);
            }
            base += kLanes * kR;
            if (base >= e1) break;
            links(base);
        }
    }
    if (lane) return;
    // the next iteration's pre-step (its records loaded here: held from the
    // start they would cost this kernel a wavefront per SIMD)
    if (a.clampn)
        adj_pre_one<UNIFORM>(b, k, a, p, ap, adj_pre_load(a, p), acc);
    else
        a.pb[p] = make_float4(acc[0], acc[1], acc[2], 0.0f);
}

// ---------------------------------------------------------------------------
// velocity + XSPH backwards: v_i = u_i/dt + ((c/rho0_i) S_i)/dt,
// S_i = sum_fluid j (u_j - u_i) m_j W_ij, u = p - x*.  adj_xsph_k forms
// dL/dS_i = (c/rho0_i) vbar_i / dt (in Y) and the rho0 term; adj_finalize_k
// gathers dL/dp (the final iterate) and dL/dx*.

template <bool UNIFORM, uint32_t U>
__global__ __launch_bounds__(kAdjBlock) void adj_xsph_k(DevBuffers b, KConst k, AdjBuffers a, uint32_t n,
                                                     float dt)
{
    const uint32_t i = xcd_block() * (kAdjBlock / (4u * U)) + threadIdx.x / (4u * U);
    const uint32_t lane = threadIdx.x % (4u * U);  // lane 0 finishes
    if (i >= n) return;  // the lanes of a particle leave together
    // the particle's own loads go out together
    const Attr ai = b.A[i];
    const float4 pi = b.P[i], xi = b.X[i];
    const uint32_t c = b.ncnt[i];
    float r0 = 0.0f;
    float Sh[3] = {0.0f, 0.0f, 0.0f};
    if (k.xsph_c != 0.0f && (UNIFORM || ai.phase == PS_PHASE_FLUID)) {
        const float ui[3] = {pi.x - xi.x, pi.y - xi.y, pi.z - xi.z};
        const float4 vb = a.gv[ai.orig];
        const float vbn[3] = {vb.x, vb.y, vb.z};
        const float cr = k.xsph_c / ai.rho0;
        // S exactly as finalize_k forms it: four quarters of the table
        float Sm[3] = {0.0f, 0.0f, 0.0f};
        auto body = [&](const float4 &pj, const float4 &xj, float wj, bool used) {
            const float r2 = dist2(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z);
            float d[3] = {0.0f, 0.0f, 0.0f}, m = 0.0f;  // a sum that starts at +0 never is -0
            if (used && r2 < k.h2) {
                const float t = k.h2 - r2;
                m = ((t * t) * t) * (1.0f / wj);
                d[0] = (pj.x - xj.x) - ui[0];
                d[1] = (pj.y - xj.y) - ui[1];
                d[2] = (pj.z - xj.z) - ui[2];
            }
            for (int q = 0; q < 3; q++) Sm[q] = group_fma<U>(Sm[q], d[q], m);
        };
        constexpr uint32_t kFlight = U == 4 ? 2 : 4;
        if (UNIFORM) {
            for_neighbors_quarter<U, kFlight>(
                b, i, c, lane / U, lane % U, [&](uint32_t j) { return PX{b.P[j], b.X[j]}; },
                [&](const PX &d, bool used) { body(d.p, d.x, ai.w, used); });
        } else {
            for_neighbors_quarter<U, kFlight>(
                b, i, c, lane / U, lane % U, [&](uint32_t j) { return GXA{b.P[j], b.X[j], b.A[j]}; },
                [&](const GXA &d, bool used) {
                    body(d.p, d.x, d.a.w, used && d.a.phase == PS_PHASE_FLUID);
                });
        }
        for (int q = 0; q < 3; q++) Sm[q] = quarters_sum<U>(Sm[q]);
        if (lane) return;
        const float S[3] = {k.poly6 * Sm[0], k.poly6 * Sm[1], k.poly6 * Sm[2]};
        const float vS = dot3(vbn, S);
        r0 = r0 - (((k.xsph_c / (ai.rho0 * ai.rho0)) * vS) / dt);
        for (int q = 0; q < 3; q++) Sh[q] = (vbn[q] * cr) / dt;
    }
    if (lane) return;
    a.r0b[i] = r0;
    a.wkb[i] = 0.0f;
    a.Y[i] = make_float4(Sh[0], Sh[1], Sh[2], 0.0f);
}

// Quarter 0 starts from dL/dx and dL/dv / dt.
template <bool UNIFORM, uint32_t U>
__global__ __launch_bounds__(kAdjBlock) void adj_finalize_k(DevBuffers b, KConst k, AdjBuffers a, uint32_t n,
                                                         float dt)
{
    const uint32_t p = xcd_block() * (kAdjBlock / (4u * U)) + threadIdx.x / (4u * U);
    const uint32_t lane = threadIdx.x % (4u * U);
    if (p >= n) return;  // the lanes of a particle leave together
    // the particle's own loads go out together (and the last iteration's
    // pre-step records)
    const Attr ap = b.A[p];
    const float4 pp = b.P[p], xp = b.X[p];
    const float4 shp4 = a.Y[p];
    const uint32_t c = b.ncnt[p];
    AdjPreIn pre{};
    if (a.clampn && lane == 0) pre = adj_pre_load(a, p);
    const float4 vb = a.gv[ap.orig], xb = a.gx[ap.orig];
    float ub[3] = {vb.x / dt, vb.y / dt, vb.z / dt};
    float acc[3] = {xb.x, xb.y, xb.z};
    if (lane >= U)
        for (int q = 0; q < 3; q++) ub[q] = acc[q] = 0.0f;
    if (k.xsph_c != 0.0f && (UNIFORM || ap.phase == PS_PHASE_FLUID)) {
        const float up[3] = {pp.x - xp.x, pp.y - xp.y, pp.z - xp.z};
        const float Shp[3] = {shp4.x, shp4.y, shp4.z};
        const float mp = 1.0f / ap.w;
        auto body = [&](const float4 &pj, const float4 &xj, const float4 &shj4, float wj, bool used) {
            const float dv[3] = {pp.x - pj.x, pp.y - pj.y, pp.z - pj.z};
            const float r2 = dist2(dv[0], dv[1], dv[2]);
            // u gains us, then ua, the gradient g1, then g2
            float us[3] = {-0.0f, -0.0f, -0.0f}, ua[3] = {-0.0f, -0.0f, -0.0f};
            float g1[3] = {-0.0f, -0.0f, -0.0f}, g2[3] = {-0.0f, -0.0f, -0.0f};
            if (used && r2 < k.h2) {
                const float t = k.h2 - r2;
                const float W = k.poly6 * ((t * t) * t);
                float g6[3];
                adj_grad_w6(k, dv, r2, g6);
                const float uj[3] = {pj.x - xj.x, pj.y - xj.y, pj.z - xj.z};
                const float Shj[3] = {shj4.x, shj4.y, shj4.z};
                // p as owner: S_p += (u_j - u_p) m_j W; p as neighbour of j
                const float mj = 1.0f / wj;
                const float wb = mj * ((((uj[0] - up[0]) * Shp[0]) + ((uj[1] - up[1]) * Shp[1])) +
                                       ((uj[2] - up[2]) * Shp[2]));
                const float wb2 = mp * ((((up[0] - uj[0]) * Shj[0]) + ((up[1] - uj[1]) * Shj[1])) +
                                        ((up[2] - uj[2]) * Shj[2]));
                for (int q2 = 0; q2 < 3; q2++) {
                    us[q2] = -((mj * W) * Shp[q2]);
                    ua[q2] = (mp * W) * Shj[q2];
                    g1[q2] = wb * g6[q2];
                    g2[q2] = wb2 * g6[q2];
                }
            }
            for (int q2 = 0; q2 < 3; q2++) {
                ub[q2] = group_add<U>(ub[q2], us[q2], ua[q2]);
                acc[q2] = group_add<U>(acc[q2], g1[q2], g2[q2]);
            }
        };
        constexpr uint32_t kFlight = U == 4 ? 2 : 4;
        if (UNIFORM) {
            for_neighbors_quarter<U, kFlight>(
                b, p, c, lane / U, lane % U, [&](uint32_t j) { return GXY{b.P[j], b.X[j], a.Y[j]}; },
                [&](const GXY &d, bool used) { body(d.p, d.x, d.y, ap.w, used); });
        } else {
            for_neighbors_quarter<U, kFlight>(
                b, p, c, lane / U, lane % U, [&](uint32_t j) { return GXYA{b.P[j], b.X[j], a.Y[j], b.A[j]}; },
                [&](const GXYA &d, bool used) {
                    body(d.p, d.x, d.y, d.a.w, used && d.a.phase == PS_PHASE_FLUID);
                });
        }
    }
    for (int q = 0; q < 3; q++) {
        ub[q] = quarters_sum<U>(ub[q]);
        acc[q] = quarters_sum<U>(acc[q]);
    }
    if (lane) return;
    a.xsb[p] = make_float4(-ub[0], -ub[1], -ub[2], 0.0f);
    float g[3] = {acc[0] + ub[0], acc[1] + ub[1], acc[2] + ub[2]};
    if (a.clampn)
        adj_pre_one<UNIFORM>(b, k, a, p, ap, pre, g);  // the last iteration's pre-step
    else
        a.pb[p] = make_float4(g[0], g[1], g[2], 0.0f);
}

// predict backwards: p0 = x* + dt (v + dt g) for w != 0 (z held in 2D);
// results to insertion order, rho0 and wall_k terms accumulated there
__global__ __launch_bounds__(kAdjBlock) void adj_predict_k(DevBuffers b, KConst k, AdjBuffers a, uint32_t n,
                                                        float dt)
{
    const uint32_t t = blockIdx.x * kAdjBlock + threadIdx.x;
    if (t >= n) return;
    const Attr at = b.A[t];
    const uint32_t o = at.orig;
    const float4 xs = a.xsb[t], pb = a.pb[t];
    const bool mv = at.w != 0.0f;
    const bool twod = k.dims == 2u;
    a.gx[o] = make_float4(xs.x + pb.x, xs.y + pb.y, xs.z + pb.z, 0.0f);
    a.gv[o] = make_float4(mv ? dt * pb.x : 0.0f, mv ? dt * pb.y : 0.0f, (mv && !twod) ? dt * pb.z : 0.0f,
                          0.0f);
    a.drho[o] = a.drho[o] + a.r0b[t];
    a.dwk[o] = a.dwk[o] + a.wkb[t];
}

// ---------------------------------------------------------------------------

static inline uint32_t adj_blocks(uint32_t n) { return (n + kAdjBlock - 1) / kAdjBlock; }

// Lanes a quarter: four while the particles are too few to fill the chip with
// one (65,536 of them make four wavefronts a SIMD), one from there on, where
// the four lanes' repeated sums and the 4 times as many wavefronts' own
// records cost more than the shorter chains give.  adj_position_k, then
// adj_lambda_k, with one lane and with four, in us: 5k particles 20.8 / 10.9,
// 6.8 / 4.4; 12k 16.3 / 9.2, 6.6 / 5.0; 32k 18.4 / 15.3, 8.5 / 7.6; 50k 23.3 /
// 21.7, 12.3 / 10.3; 82k 39.6 / 44.1, 15.5 / 15.6; 328k 81 / 126, 48 / 51.
static constexpr uint32_t kAdjSpread = 65536;

hipError_t launch_adj(hipStream_t st, AdjKernel which, const DevBuffers &b, const KConst &k,
                      const AdjBuffers &a, uint32_t count, float dt, bool uniform)
{
    if (count == 0) return hipSuccess;
    const dim3 grid(adj_blocks(count)), block(kAdjBlock);
    // 4 U lanes per particle
#define PS_ADJ_LAUNCH_U(kern, U, ...)                                                              \
    do {                                                                                           \
        const dim3 g((count + kAdjBlock / (4 * U) - 1) / (kAdjBlock / (4 * U)));                   \
        if (uniform)                                                                               \
            PS_LAUNCH((kern<true, U>), g, block, 0, st, __VA_ARGS__);                              \
        else                                                                                       \
            PS_LAUNCH((kern<false, U>), g, block, 0, st, __VA_ARGS__);                             \
    } while (0)
#define PS_ADJ_LAUNCH(kern, ...)                                                                   \
    do {                                                                                           \
        if (count <= kAdjSpread)                                                                   \
            PS_ADJ_LAUNCH_U(kern, 4, __VA_ARGS__);                                                 \
        else                                                                                       \
            PS_ADJ_LAUNCH_U(kern, 1, __VA_ARGS__);                                                 \
    } while (0)
    switch (which) {
    case ADJ_XSPH: PS_ADJ_LAUNCH(adj_xsph_k, b, k, a, count, dt); break;
    case ADJ_FINALIZE: PS_ADJ_LAUNCH(adj_finalize_k, b, k, a, count, dt); break;
    case ADJ_LAMBDA: PS_ADJ_LAUNCH(adj_lambda_k, b, k, a, count); break;
    case ADJ_POSITION: PS_ADJ_LAUNCH(adj_position_k, b, k, a, count); break;
    case ADJ_PREDICT: PS_LAUNCH(adj_predict_k, grid, block, 0, st, b, k, a, count, dt); break;
    default: return hipErrorInvalidValue;
    }
#undef PS_ADJ_LAUNCH
#undef PS_ADJ_LAUNCH_U
    return hipGetLastError();
}

}  // namespace ps
