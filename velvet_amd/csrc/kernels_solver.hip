// XPBD solver passes for gfx950.
//
// One workgroup = one particle tile of one segment (VTX_TILE threads, one particle each).
// Every constraint pass is an atomic-free gather: a particle walks its own incident
// constraints (sliced ELL), evaluates each one in full from the pass's input positions and
// keeps only its own correction, so the reference's Jacobi scatter-with-atomics
// (Velvet/VtClothSolverGPU.cu:13-21, 65-251) becomes a fixed-order, deterministic sum and a
// pass reads P[in] and writes P[out]. The reference's ApplyDeltas (cu:253-270) is fused
// into the end of each pass; Finalize (cu:388-417) and the next substep's PredictPositions
// (cu:42-63) are fused into the last pass of a substep.
#include <hip/hip_runtime.h>

#include "launch.hpp"
#include "vec.hpp"
#include "vtx_device.hpp"

namespace vtx {

// Hardware reciprocal / reciprocal square root / square root (1 ulp) for the solver passes.
// (The library is built with correctly rounded division and square root, which the hash needs
// for bit-exact cell coordinates; the solver passes are held to the FP64 oracle's tolerance.)
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float frsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float flen(V3 a) { return fsqrt(dot(a, a)); }

// arccos on [-1, 1]: the minimax form sqrt(1 - x) * (a0 + a1 x + ... + a7 x^7) of Abramowitz &
// Stegun, Handbook of Mathematical Functions, 4.4.46 (|error| <= 2e-8 on [0, 1]), with
// acos(x) = pi - acos(-x) below 0. In binary32 it stays within 4.3e-7 of the exact value
// (checked against double-precision arccos over [-1, 1]), 2.3e-8 near 1 where bending angles
// are small.
__device__ __forceinline__ float facos(float x) {
    const float ax = fabsf(x);
    float p = -0.0012624911f;
    p = fmaf(p, ax, 0.0066700901f);
    p = fmaf(p, ax, -0.0170881256f);
    p = fmaf(p, ax, 0.0308918810f);
    p = fmaf(p, ax, -0.0501743046f);
    p = fmaf(p, ax, 0.0889789874f);
    p = fmaf(p, ax, -0.2145988016f);
    p = fmaf(p, ax, 1.5707963050f);
    const float q = fsqrt(1.0f - ax);
    return x < 0.f ? fmaf(-q, p, 3.14159265358979f) : q * p;
}

// ComputeFriction (Velvet/VtClothSolverGPU.cu:272-287). tl == 0 gives mt * inf = inf, clamped
// to 1 as the reference's mt / 0 is.
__device__ __forceinline__ V3 friction_of(V3 correction, V3 rel, float friction) {
    V3 f = v3(0.f, 0.f, 0.f);
    float cl = flen(correction);
    if (friction > 0.f && cl > 0.f) {
        V3 nrm = correction * frcp(cl);
        V3 tan = rel - nrm * dot(rel, nrm);
        float tl = flen(tan);
        float mt = cl * friction;
        f = -tan * fminf(mt * frcp(tl), 1.0f);
    }
    return f;
}

__device__ __forceinline__ float sgnf(float v) { return (v > 0.f) ? 1.0f : (v < 0.f ? -1.0f : 0.0f); }

// SDFCollider::ComputeSDF (Velvet/VtClothSolverGPU.cuh:22-89).
__device__ V3 compute_sdf(const ColliderDev& c, V3 p, float margin) {
    if (c.type == 1) {
        float offset = p.y - (c.pos[1] + margin);
        if (offset < 0.f) return v3(0.f, -offset, 0.f);
    } else if (c.type == 0) {
        float radius = c.scale[0] + margin;
        V3 diff = p - v3(c.pos[0], c.pos[1], c.pos[2]);
        float distance = flen(diff);
        float offset = distance - radius;
        if (offset < 0.f) {
            V3 direction = diff * frcp(distance);
            return -offset * direction;
        }
    } else if (c.type == 2) {
        V3 correction = v3(0.f, 0.f, 0.f);
        V3 local = xform_point(c.inv, p);
        V3 size = v3(0.5f + margin * frcp(c.scale[0]), 0.5f + margin * frcp(c.scale[1]),
                     0.5f + margin * frcp(c.scale[2]));
        V3 offset = vabs(local) - size;
        float maxv = fmaxf(offset.x, fmaxf(offset.y, offset.z));
        float minv = fminf(offset.x, fminf(offset.y, offset.z));
        float midv = offset.x + offset.y + offset.z - maxv - minv;
        float scalar = 1.0f;
        if (maxv < 0.f) {
            const float m = 0.03f;
            if (midv > -m) scalar = 0.2f;
            if (minv > -m) {
                V3 mask = v3(offset.x < 0.f ? sgnf(local.x) : 0.f, offset.y < 0.f ? sgnf(local.y) : 0.f,
                             offset.z < 0.f ? sgnf(local.z) : 0.f);
                V3 vec = offset + v3(m, m, m);
                float l = flen(vec);
                if (l < m) {
                    V3 nv = vec * frsq(dot(vec, vec));   // glm::normalize
                    correction = v3(mask.x * nv.x * (m - l), mask.y * nv.y * (m - l), mask.z * nv.z * (m - l));
                }
            } else if (offset.x == maxv) {
                correction = v3(copysignf(-offset.x, local.x), 0.f, 0.f);
            } else if (offset.y == maxv) {
                correction = v3(0.f, copysignf(-offset.y, local.y), 0.f);
            } else if (offset.z == maxv) {
                correction = v3(0.f, 0.f, copysignf(-offset.z, local.z));
            }
        }
        return xform_vec(c.cur3, correction * scalar);
    }
    return v3(0.f, 0.f, 0.f);
}

// CollideSDF_Kernel body (Velvet/VtClothSolverGPU.cu:289-314) for one particle: colliders in
// order, friction only for a nonzero correction, collider velocity from VelocityAt
// (Velvet/VtClothSolverGPU.cuh:91-96).
__device__ V3 collide_sdf(V3 pred, V3 pos, const ColliderDev* cols, uint32_t cb, uint32_t cc,
                          float margin, float friction, float dt) {
    for (uint32_t c = cb; c < cb + cc; c++) {
        const ColliderDev& col = cols[c];
        V3 corr = compute_sdf(col, pred, margin);
        pred += corr;
        if (dot(corr, corr) > 0.f) {
            V3 lastp = xform_point(col.rel, pred);
            V3 vel = (pred - lastp) * frcp(col.dt);
            V3 relv = pred - pos - vel * dt;
            pred += friction_of(corr, relv, friction);
        }
    }
    return pred;
}

// Pre-stabilisation SDF on positions with the frame time (Velvet/VtClothSolverGPU.hpp:73) and
// the first substep's PredictPositions (cu:42-53). The predicted velocity is not stored: every
// substep ends in Finalize, which derives the velocity from the positions alone and stores it, so
// between frames (where the host and the failure check read it) V holds Finalize's value, as in
// the reference, and nothing reads V inside a frame.
__global__ __launch_bounds__(VTX_TILE) void k_frame_begin(DevState d, float frame_dt, float h) {
    const TileDev t = d.tiles[tile_of(d.remap)];
    if (threadIdx.x >= t.count) return;
    const SegDev sg = d.segs[t.seg];
    const uint32_t g = t.begin + threadIdx.x;
    float4 x4 = d.X[g];
    V3 x = xyz(x4);
    if (sg.ccount) {
        x = collide_sdf(x, x, d.cols, sg.cbase, sg.ccount, sg.margin, sg.friction, frame_dt);
        d.X[g] = f4(x, x4.w);
    }
    const V3 v = xyz(d.V[g]) + v3(sg.gx, sg.gy, sg.gz) * h;
    d.P[0][g] = f4(x + v * h, x4.w);
}

// CollideParticles_Kernel + ApplyDeltas (Velvet/VtClothSolverGPU.cu:329-386) followed by the
// substep's CollideSDF (cu:289-314, hpp:87).
template <int BS, int U>
__global__ __launch_bounds__(BS) void k_collide(DevState d, int in, float h) {
    constexpr bool AHEAD = U > 4;
    uint32_t tix, lane;
    tile_lane<VTX_TILE, BS>(d.remap, tix, lane);
    const TileDev t = d.tiles[tix];
    if (lane >= t.count) return;
    const SegDev sg = d.segs[t.seg];
    const uint32_t g = t.begin + lane;
    const float4* __restrict__ P = d.P[in];
    const float4 p4 = P[g];
    V3 p = xyz(p4);
    const float w = p4.w;
    const V3 x = xyz(d.X[g]);
    if (sg.flags & VTX_SEG_SELFCOL) {
        const uint32_t n = sg.n;
        // the list in chunks of four entries: chunk c at nb4[c * n] (32-bit entries) or nb2[c * n]
        // (16-bit entries, 0xffff >= n the sentinel)
        const uint32_t* __restrict__ table = d.nbr + ((uint64_t)sg.nbase_hi << 32 | sg.nbase_lo);
        const uint4* __restrict__ nb4 = reinterpret_cast<const uint4*>(table) + (g - sg.pbase);
        const uint2* __restrict__ nb2 = reinterpret_cast<const uint2*>(table) + (g - sg.pbase);
        const bool n16 = sg.flags & VTX_SEG_NBR16;
        V3 delta = v3(0.f, 0.f, 0.f);
        int cnt = 0;
        const V3 vel_i = p - x;
        // neighbours U at a time (chunks of four): while a group's positions load, the next chunks
        // load too; the terms are then added in list order. An entry counts only if every
        // entry before it is a particle index (the list ends at the first sentinel, later rows are
        // stale). A neighbour's start-of-substep position enters only the friction of a contact,
        // so it is loaded for contacts alone unless AHEAD: most listed neighbours of a resting cloth lie
        // beyond the diameter, and a large pass is bound by the cache lines its gathers touch.
        bool live = true;
        const uint32_t K = sg.max_nbr;
        uint32_t jn[U];
        auto load = [&](uint32_t k0, uint32_t* jn) {   // entries k0..k0+3, those at K or beyond as sentinels
            uint4 c;
            if (n16) {
                const uint2 h = nb2[(size_t)(k0 >> 2) * n];
                c = make_uint4(h.x & 0xFFFFu, h.x >> 16, h.y & 0xFFFFu, h.y >> 16);
            } else {
                c = nb4[(size_t)(k0 >> 2) * n];
            }
            jn[0] = c.x;
            jn[1] = k0 + 1 < K ? c.y : VTX_INVALID;
            jn[2] = k0 + 2 < K ? c.z : VTX_INVALID;
            jn[3] = k0 + 3 < K ? c.w : VTX_INVALID;
        };
        auto chunk = [&](uint32_t k0) {
            load(k0, jn);
#pragma unroll
            for (int u = 4; u < U; u += 4) {
                jn[u] = jn[u + 1] = jn[u + 2] = jn[u + 3] = VTX_INVALID;
                if (k0 + u < K) load(k0 + u, jn + u);
            }
        };
        chunk(0);
        for (uint32_t k0 = 0; k0 < K && live; k0 += U) {
            bool ok[U];
            uint32_t jg[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                live = live && jn[u] < n;
                ok[u] = live;
                jg[u] = sg.pbase + (ok[u] ? jn[u] : 0u);
            }
            float4 pj4[U], xj4[U];
#pragma unroll
            for (int u = 0; u < U; u++) pj4[u] = P[jg[u]];
            if (AHEAD) {
#pragma unroll
                for (int u = 0; u < U; u++) xj4[u] = d.X[jg[u]];
            }
            if (live && k0 + U < K) chunk(k0 + U);
            bool hit[U];
            float dist[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                dist[u] = flen(p - xyz(pj4[u]));
                hit[u] = ok[u] && !(w + pj4[u].w <= 0.f) && !(dist[u] >= sg.diameter);
                if (!AHEAD && hit[u]) xj4[u] = d.X[jg[u]];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (!hit[u]) continue;
                const float denom = w + pj4[u].w;
                const V3 pj = xyz(pj4[u]);
                const V3 diff = p - pj;
                const V3 grad = diff * frcp(dist[u] + VTX_EPSILON);
                const float lambda = (dist[u] - sg.diameter) * frcp(denom);
                const V3 common = lambda * grad;
                cnt++;
                delta -= w * common;
                const V3 relv = vel_i - (pj - xyz(xj4[u]));
                delta += w * friction_of(common, relv, sg.friction);
            }
        }
        if (cnt > 0) p += delta * (frcp((float)cnt) * sg.omega);
    }
    if (sg.ccount) p = collide_sdf(p, x, d.cols, sg.cbase, sg.ccount, sg.margin, sg.friction, h);
    d.P[in ^ 1][g] = f4(p, w);
}

// Epilogue modes of the Jacobi pass.
enum { EPI_NONE = 0, EPI_FINALIZE = 1, EPI_FINALIZE_PREDICT = 2 };

// One stretch constraint seen from one endpoint (Velvet/VtClothSolverGPU.cu:80-98): bilateral,
// compliance 0, eps in the gradient denominator. q = other endpoint (xyz, inverse mass);
// nws = -w * stiffness, the endpoint's factor of every one of its terms.
__device__ __forceinline__ void stretch_term(V3 p, float w, float nws, float4 q, float rest, V3& delta, int& cnt) {
    const V3 diff = p - xyz(q);
    const float dist = fsqrt(dot_fma(diff, diff));
    const float wsum = w + q.w;
    if (dist != rest && wsum > 0.f) {
        delta = madd(delta, diff, (dist - rest) * nws * frcp(wsum * (dist + VTX_EPSILON)));
        cnt++;
    }
}

// One long-range attachment (Velvet/VtClothSolverGPU.cu:218-234): with t the target distance,
// a particle farther than t from its slot moves by -diff + diff / |diff| * t, which is
// diff * (t / |diff| - 1); "|diff| > t" is the same test as "t / |diff| - 1 < 0", so one
// reciprocal square root serves both. Branch-free (selects): the slot position is used on every
// path, so its loads can be issued ahead of the term instead of inside a conditional block.
__device__ __forceinline__ void attach_to(V3 p, float w, float4 slot, float target, V3& delta, int& cnt) {
    const V3 diff = p - xyz(slot);
    const float f = __builtin_fmaf(target, frsq(dot_fma(diff, diff)), -1.0f);
    // the reference returns early for a pinned particle with a positive target
    const bool act = !(w == 0.f && target > 0.f) && f < 0.f;
    const float k = act ? f : 0.f;
    delta.x = __builtin_fmaf(diff.x, k, delta.x);
    delta.y = __builtin_fmaf(diff.y, k, delta.y);
    delta.z = __builtin_fmaf(diff.z, k, delta.z);
    cnt += act ? 1 : 0;
}

__device__ __forceinline__ void attach_term(V3 p, float w, float4 slot, float dist0, float lrs, V3& delta,
                                            int& cnt) {
    attach_to(p, w, slot, dist0 * lrs, delta, cnt);
}

// Slot range [s0, s1) of part q of a segment's attachments (see VTX_LRA_PARTS).
__device__ __forceinline__ void lra_part_range(const SegDev& sg, uint32_t q, uint32_t& s0, uint32_t& s1) {
    const uint32_t qs = (sg.scount + VTX_LRA_PARTS - 1) / VTX_LRA_PARTS;
    s0 = min(q * qs, sg.scount);
    s1 = min(s0 + qs, sg.scount);
}

// Dense attachments of one particle to slots [s0, s1), summed from zero in slot order.
// Distances are fetched four slots at a time so that several loads are in flight per lane.
__device__ __forceinline__ void attach_dense(const DevState& d, const SegDev& sg, uint32_t local, uint32_t s0,
                                             uint32_t s1, V3 p, float w, V3& part, int& cnt) {
    const float* __restrict__ lra = d.lra + 4 * (size_t)sg.lbase + local;
    const float4* __restrict__ slot = d.slots + sg.sbase;
    const size_t n = sg.n;
    uint32_t s = s0;
    for (; s + 4 <= s1; s += 4) {
        float r[4];
        float4 q[4];                                        // wave-uniform
#pragma unroll
        for (int u = 0; u < 4; u++) r[u] = lra[(size_t)(s + u) * n];
#pragma unroll
        for (int u = 0; u < 4; u++) q[u] = slot[s + u];
#pragma unroll
        for (int u = 0; u < 4; u++) attach_term(p, w, q[u], r[u], sg.lrs, part, cnt);
    }
    for (; s < s1; s++) attach_term(p, w, slot[s], lra[(size_t)s * n], sg.lrs, part, cnt);
}

// The same from a tile's target distances (VTX_SEG_LRA_TILED): dist = the part's first group of this
// lane, one float4 per group of four slots, VTX_TILE apart. B groups are in flight while the B before
// them are summed, and a group's slot positions (wave-uniform) while the group before it is; `first`
// holds the first B groups, loaded by the caller as early as it can.
template <int B>
struct TiledBatch {
    float4 r[B];
    __device__ __forceinline__ void load(const float4* __restrict__ dist, uint32_t g, uint32_t groups) {
#pragma unroll
        for (int u = 0; u < B; u++) r[u] = dist[(size_t)min(g + u, groups - 1u) * VTX_TILE];
    }
};

struct SlotGroup {
    float4 q[4];
    __device__ __forceinline__ void load(const float4* __restrict__ slot) {
#pragma unroll
        for (int k = 0; k < 4; k++) q[k] = slot[k];
    }
};

template <int B>
__device__ __forceinline__ void attach_tiled(const DevState& d, const SegDev& sg, const float4* __restrict__ dist,
                                             TiledBatch<B> cur, uint32_t s0, uint32_t s1, V3 p, float w, V3& part,
                                             int& cnt) {
    const float4* __restrict__ slot = d.slots + sg.sbase + s0;
    const uint32_t groups = (s1 - s0 + 3) / 4, full = (s1 - s0) / 4;
    if (full) {
        SlotGroup now;
        now.load(slot);
        for (uint32_t g = 0; g < full; g += B) {
            TiledBatch<B> next;
            next.load(dist, g + B, groups);
#pragma unroll
            for (int u = 0; u < B; u++) {
                if (g + u >= full) break;
                SlotGroup then;
                then.load(slot + 4 * min(g + u + 1, full - 1u));
                attach_to(p, w, now.q[0], cur.r[u].x, part, cnt);
                attach_to(p, w, now.q[1], cur.r[u].y, part, cnt);
                attach_to(p, w, now.q[2], cur.r[u].z, part, cnt);
                attach_to(p, w, now.q[3], cur.r[u].w, part, cnt);
                now = then;
            }
            cur = next;
        }
    }
    if (full < groups) {                                    // one to three slots left
        const float4 r = dist[(size_t)full * VTX_TILE];
        attach_to(p, w, slot[4 * full], r.x, part, cnt);
        if (s0 + 4 * full + 1 < s1) attach_to(p, w, slot[4 * full + 1], r.y, part, cnt);
        if (s0 + 4 * full + 2 < s1) attach_to(p, w, slot[4 * full + 2], r.z, part, cnt);
    }
}

// First group of part q of a tile's lane.
__device__ __forceinline__ const float4* tiled_part(const DevState& d, const SegDev& sg, uint32_t at_off, uint32_t q,
                                                    uint32_t lane) {
    const uint32_t qs = (sg.scount + VTX_LRA_PARTS - 1) / VTX_LRA_PARTS;
    return reinterpret_cast<const float4*>(d.lra) + at_off + (size_t)q * ((qs + 3) / 4) * VTX_TILE + lane;
}

// All attachments of one particle, added to delta part by part (VTX_LRA_PARTS): dense
// (slot-major distances, the slot position is the same for every lane) or from the tile's attach
// ELL in registration order, where a part ends wherever the slot's part changes -- so attachments
// registered particle-major in slot order sum exactly as the dense form does. NA listed attachments are in
// flight: one after another each waits for its entry and then for its slot (general path, frames of 32 passes,
// 131,769 particles with 35: 1,979 -> 1,339 us, 360,000 with 16: 2,296 -> 1,720); the stencil tiles have no
// registers left for more than one.
template <uint32_t NA>
__device__ __forceinline__ void attach_terms(const DevState& d, const SegDev& sg, uint32_t at_off, uint32_t at_k,
                                             uint32_t lane, uint32_t local, V3 p, float w, V3& delta, int& cnt) {
    if (sg.flags & VTX_SEG_LRA_DENSE) {
        if (sg.scount <= VTX_LRA_PARTS) {   // every slot is a part of its own
            const float* __restrict__ lra = d.lra + 4 * (size_t)sg.lbase + local;
            const float4* __restrict__ slot = d.slots + sg.sbase;
            for (uint32_t s = 0; s < sg.scount; s++) {
                V3 part = v3(0.f, 0.f, 0.f);
                attach_term(p, w, slot[s], lra[(size_t)s * sg.n], sg.lrs, part, cnt);
                delta += part;
            }
            return;
        }
#pragma unroll 1
        for (uint32_t q = 0; q < VTX_LRA_PARTS; q++) {
            uint32_t s0, s1;
            lra_part_range(sg, q, s0, s1);
            V3 part = v3(0.f, 0.f, 0.f);
            attach_dense(d, sg, local, s0, s1, p, w, part, cnt);
            delta += part;
        }
        return;
    }
    const uint32_t qs = (sg.scount + VTX_LRA_PARTS - 1) / VTX_LRA_PARTS;
    const uint2* __restrict__ at = d.at + at_off + lane;
    static_assert(VTX_LRA_PARTS == 4, "the part of a listed slot is found with three compares");
    V3 part = v3(0.f, 0.f, 0.f);
    uint32_t cur = 0;
    for (uint32_t k0 = 0; k0 < at_k; k0 += NA) {
        uint2 e[NA];
        float4 slot[NA];
#pragma unroll
        for (uint32_t k = 0; k < NA; k++) e[k] = at[(size_t)min(k0 + k, at_k - 1u) * VTX_TILE];
#pragma unroll
        for (uint32_t k = 0; k < NA; k++) slot[k] = d.slots[sg.sbase + (e[k].x == VTX_INVALID ? 0u : e[k].x)];
#pragma unroll
        for (uint32_t k = 0; k < NA; k++) {
            if (k0 + k >= at_k || e[k].x == VTX_INVALID) continue;
            const uint32_t q = (e[k].x >= qs ? 1u : 0u) + (e[k].x >= 2 * qs ? 1u : 0u) + (e[k].x >= 3 * qs ? 1u : 0u);
            if (q != cur) {
                delta += part;
                part = v3(0.f, 0.f, 0.f);
                cur = q;
            }
            attach_term(p, w, slot[k], __uint_as_float(e[k].y), sg.lrs, part, cnt);
        }
    }
    delta += part;
}

// The dihedral bending constraint (Velvet/VtClothSolverGPU.cu:128-177), evaluated through the
// edge vector e = p3 - p2, a = p2 - p0 and b = p3 - p1:
//   c1 = (p2-p0) x (p3-p0) = a x e,   c2 = (p3-p1) x (p2-p1) = e x b,
//   (p0-p3).e = -(a.e) - |e|^2,        (p1-p3).e = -(b.e),
//   (c1 x c2).e = |e|^2 (a.c2)         (since e.c2 = 0), so the sign rule needs one dot product.
// With r1 = 1/|c1| and r2 = 1/|c2| (one reciprocal square root each), the reference's
// n1 = c1 r1^2, n2 = c2 r2^2 and normalize(n1).normalize(n2) = (c1.c2) r1 r2, so every gradient is
// a combination of c1 and c2: d0 = k0 c1, d1 = k1 c2 (k0 = |e| r1^2, k1 = |e| r2^2) and
// d2 = s1 c1 + s2 c2, d3 = -(d0 + d1 + d2) = t1 c1 + t2 c2 (the four gradients of a dihedral
// angle sum to zero; the reference's d3 = (p2-p0).e/|e| n1 + (p2-p1).e/|e| n2 is the same).
// Returns false on the reference's early-outs; else lam carries the sign rule and the correction
// of vertex k is -w_k * lam * d_k.
struct BendGrad {
    V3 c1, c2, d2;   // d0 = k0 c1, d1 = k1 c2, d3 = -(d0 + d1 + d2)
    float k0, k1;
};

//
// The multiply-adds are spelled out, so that every kernel that evaluates a constraint rounds it alike
// (the sign test at the end decides the whole correction of a flat pair, so a last bit can show). The
// stencil path (GRID) and the general path differ in the order of some sums.
template <bool GRID>
__device__ __forceinline__ bool bend_eval(float4 q0, float4 q1, float4 q2, float4 q3, float rest, float xpbd,
                                          float& lam, BendGrad& g) {
#pragma clang fp contract(off)
    const auto dot_ge = [](V3 u, V3 v) {
        return GRID ? dot_fma(u, v) : __builtin_fmaf(u.z, v.z, __builtin_fmaf(u.y, v.y, u.x * v.x));
    };
    const V3 p0 = xyz(q0), p1 = xyz(q1), p2 = xyz(q2), p3 = xyz(q3);
    const V3 e = p3 - p2;
    const float ee = dot_fma(e, e);
    if (ee < VTX_EPSILON * VTX_EPSILON) return false;   // |e| < eps
    const float inv_elen = frsq(ee);                      // |e| and 1/|e| from one rsq
    const float elen = ee * inv_elen;
    const V3 a = p2 - p0, b = p3 - p1;
    g.c1 = cross_fma(a, e);
    g.c2 = cross_fma(e, b);
    const float g11 = dot_fma(g.c1, g.c1), g22 = dot_fma(g.c2, g.c2), g12 = dot_fma(g.c1, g.c2);
    const float r1 = frsq(g11), r2 = frsq(g22);
    const float r1s = r1 * r1, r2s = r2 * r2;
    g.k0 = elen * r1s;
    g.k1 = elen * r2s;
    const float s1 = ((-dot_ge(a, e) - ee) * inv_elen) * r1s, s2 = (-dot_ge(b, e) * inv_elen) * r2s;
    g.d2 = GRID ? madd(s2 * g.c2, g.c1, s1) : madd(s1 * g.c1, g.c2, s2);
    const float cd = fminf(fmaxf(g12 * (r1 * r2), -1.0f), 1.0f);
    const float phi = facos(cd);
    // |d0|^2 = |e|^2 r1^2, |d1|^2 = |e|^2 r2^2, and d3 = t1 c1 + t2 c2 from the Gram entries:
    // |d3|^2 = t1 (t1 g11 + 2 t2 g12) + t2^2 g22
    const float t1 = -__builtin_fmaf(elen, r1s, s1), t2 = -__builtin_fmaf(elen, r2s, s2), t2g = t2 * g12;
    const float d3s = __builtin_fmaf(t1, __builtin_fmaf(t1, g11, t2g + t2g), t2 * (t2 * g22));
    const float w01 = GRID ? __builtin_fmaf(q0.w, r1s, q1.w * r2s) : __builtin_fmaf(q1.w, r2s, q0.w * r1s);
    float l = __builtin_fmaf(q3.w, d3s, __builtin_fmaf(ee, w01, q2.w * dot_fma(g.d2, g.d2)));
    if (l < VTX_EPSILON) return false;
    l = (phi - rest) * frcp(l + xpbd);
    if (dot_ge(a, g.c2) > 0.0f) l = -l;      // (n1 x n2).e > 0
    lam = l;
    return true;
}

// Finalize (Velvet/VtClothSolverGPU.cu:396-406) and optionally the next substep's Predict, whose
// velocity is not stored (the next Finalize overwrites it; see k_frame_begin).
template <int EPI>
__device__ __forceinline__ void epilogue(const DevState& d, const SegDev& sg, uint32_t g, int in, V3 p, float w,
                                         float h) {
    if (EPI == EPI_NONE) {
        d.P[in ^ 1][g] = f4(p, w);
    } else {
        const float4 x4 = d.X[g];
        const V3 x = xyz(x4);
        V3 raw = (p - x) * frcp(h);
        const float rl = fsqrt(dot_fma(raw, raw));
        if (rl > sg.max_speed) {
            raw = raw * (frcp(rl) * sg.max_speed);
            p = madd(x, raw, h);
        }
        V3 v = raw * __builtin_fmaf(-sg.damping, h, 1.0f);
        d.X[g] = f4(p, x4.w);
        if (EPI == EPI_FINALIZE_PREDICT) {
            v = madd(v, v3(sg.gx, sg.gy, sg.gz), h);
            d.P[in ^ 1][g] = f4(madd(p, v, h), x4.w);
        } else {
            d.V[g] = f4(v, 0.f);
        }
    }
}

// A pass without constraints (no iterations): only the epilogue, over every particle.
template <int EPI>
__global__ __launch_bounds__(VTX_TILE) void k_epilogue(DevState d, int in, float h) {
    const TileDev t = d.tiles[tile_of(d.remap)];
    if (threadIdx.x >= t.count) return;
    const SegDev sg = d.segs[t.seg];
    const uint32_t g = t.begin + threadIdx.x;
    const float4 p4 = d.P[in][g];
    epilogue<EPI>(d, sg, g, in, xyz(p4), p4.w, h);
}

// The stretch terms of a particle on the general path (lane of its tile, local index), eight neighbours in flight.
__device__ __forceinline__ void stretch_terms(const DevState& d, const SegDev& sg, const TileDev& t,
                                              const float4* __restrict__ P, uint32_t lane, uint32_t local, V3 p, float w,
                                              V3& delta, int& cnt) {
    constexpr uint32_t NS = 8;
    const float nws = -w * sg.stiffness;
    for (uint32_t k0 = 0; k0 < t.st_k; k0 += NS) {
        uint2 c[NS];
        float4 q[NS];
#pragma unroll
        for (uint32_t k = 0; k < NS; k++) c[k] = (d.st + t.st_off + min(k0 + k, t.st_k - 1u) * VTX_TILE)[lane];
#pragma unroll
        for (uint32_t k = 0; k < NS; k++) q[k] = P[c[k].x == VTX_INVALID ? local : c[k].x];
#pragma unroll
        for (uint32_t k = 0; k < NS; k++)
            if (k0 + k < t.st_k && c[k].x != VTX_INVALID)
                stretch_term(p, w, nws, q[k], __uint_as_float(c[k].y), delta, cnt);
    }
}

// One pass of a particle (lane of its tile) that has no bending constraints.
template <int EPI>
__device__ __forceinline__ void plain_particle(const DevState& d, const TileDev& t, uint32_t lane, int in, float h) {
    if (lane >= t.count) return;
    const SegDev sg = d.segs[t.seg];
    const uint32_t g = t.begin + lane;
    const float4* __restrict__ P = d.P[in] + sg.pbase;
    const float4 p4 = P[g - sg.pbase];
    V3 p = xyz(p4), delta = v3(0.f, 0.f, 0.f);
    const float w = p4.w;
    int cnt = 0;
    stretch_terms(d, sg, t, P, lane, g - sg.pbase, p, w, delta, cnt);
    attach_terms<4>(d, sg, t.at_off, t.at_k, lane, g - sg.pbase, p, w, delta, cnt);
    if (cnt > 0) p = madd(p, delta, frcp((float)cnt) * sg.omega);
    epilogue<EPI>(d, sg, g, in, p, w, h);
}

// One Jacobi pass on the general path: SolveStretch (cu:65-102) + SolveAttachment
// (cu:205-235) + SolveBending (cu:117-189) gathered per particle over its incident
// constraints (sliced ELL), then ApplyDeltas (cu:253-264) and the epilogue.
//
// A workgroup of 768 threads takes a tile of 256 particles. All threads evaluate the tile's bend
// records (every bending constraint that touches the tile, once), RPT per thread and round, into LDS: per role
// the gradient d_r with lam in w. Meanwhile the first 256 threads, one per particle, add the stretch and
// attachment terms; then they add their bending terms from LDS in registration order. One particle per
// thread with its bends one after the other, each evaluated by all its four particles, was a chain of a
// dozen dependent gathers and evaluations: 20.7 us a pass for 22,801 particles in 90 tiles, now 8.5 us;
// 4,608 particles 15.4 -> 7.1, 90,000 19.0 -> 15.4, 490,000 63.5 -> 57.8 us, where the halves even out:
// a tile of consecutive particles of a mesh meets 1.7 times the bends it owns.
//
// ANY: sets whose last nptiles tiles have no bends, of which a workgroup takes MT / 256, a thread per particle (one
// each kept two thirds of the threads idle: 490,000 particles without bends beside 90,000 with them 2,067 -> 1,017
// us a frame of 32 passes), or that have particles of more than VTX_MANY_BENDS bends. Its branches cost a pass 2
// to 4%, so other sets do without them.
#define VTX_MT 768             // threads of the workgroup
template <int EPI, int RPT, bool ANY, int MT>
__global__ __launch_bounds__(MT, RPT == 1 ? 6 : 3) void k_iterate(DevState d, const TileDev* __restrict__ tiles, int in, float h) {
    constexpr uint32_t UB = RPT * MT;               // records of a round
    __shared__ float4 grad[4][UB];
    __shared__ uint32_t act[UB];
    constexpr uint32_t NE = 12;                         // bend entries of a particle staged in LDS
    __shared__ uint32_t ent[NE * VTX_TILE];
    const uint32_t tid = threadIdx.x, wg = tile_of(d.remap);
    const uint32_t nbent = d.nitiles - d.nptiles;
    if (ANY && RPT == 1 && wg >= nbent) {
        constexpr uint32_t PT = MT / VTX_TILE;
        const uint32_t i = nbent + PT * (wg - nbent) + __builtin_amdgcn_readfirstlane(tid / VTX_TILE);
        if (i < d.nitiles) plain_particle<EPI>(d, tiles[i], tid % VTX_TILE, in, h);
        return;
    }
    const TileDev t = tiles[wg];
    const SegDev sg = d.segs[t.seg];
    const bool vertex = tid < t.count;
    const uint32_t g = t.begin + tid;
    const float4* __restrict__ P = d.P[in] + sg.pbase;
    const float xpbd_bend = sg.bend_compliance * frcp(h) * frcp(h);   // compliance / h^2 (cu:173)
    V3 p = v3(0.f, 0.f, 0.f), delta = p;
    float w = 0.f;
    int cnt = 0;
    // records [u0, u0 + UB) of the tile, the last waves first: the first ones hold the particles
    const auto evaluate = [&](uint32_t u0) {
        const uint32_t u = MT - 1u - tid;
        if (u0 + u >= t.ub_n) return;
        const uint4* __restrict__ rec = d.brec + t.ub_off + u0;
        uint4 ix[RPT];
        float rest[RPT];
        float4 q[RPT][4];
#pragma unroll
        for (int r = 0; r < RPT; r++) {                 // a record past the last repeats it, unused
            const uint32_t v = min(u + r * MT, t.ub_n - 1u - u0);
            ix[r] = rec[v];
            rest[r] = (d.brest + t.ub_off + u0)[v];
        }
#pragma unroll
        for (int r = 0; r < RPT; r++) {
            q[r][0] = P[ix[r].x];
            q[r][1] = P[ix[r].y];
            q[r][2] = P[ix[r].z];
            q[r][3] = P[ix[r].w];
        }
#pragma unroll
        for (int r = 0; r < RPT; r++) {
            const uint32_t v = u + r * MT;
            if (r && u0 + v >= t.ub_n) break;
            float lam;
            BendGrad bg;
            const bool on = bend_eval<false>(q[r][0], q[r][1], q[r][2], q[r][3], rest[r], xpbd_bend, lam, bg);
            act[v] = on ? 1u : 0u;
            if (on) {
                grad[0][v] = f4(bg.k0 * bg.c1, lam);
                grad[1][v] = f4(bg.k1 * bg.c2, lam);
                grad[2][v] = f4(bg.d2, lam);
                grad[3][v] = f4(-(madd(bg.k0 * bg.c1, bg.c2, bg.k1) + bg.d2), lam);
            }
        }
    };
    // four entries from k0 on, those of records [u0, u0 + nu); returns the last one's record from u0 on
    const auto add4 = [&](uint32_t u0, uint32_t nu, uint32_t k0) {
        float4 v[4];
        bool on[4];
        uint32_t last = 0;
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) {
            const uint32_t r = min(k0 + k, t.bd_k - 1u) * VTX_TILE + tid;
            const uint32_t e = k0 < NE ? ent[r] : (d.bd + t.bd_off)[r];
            const uint32_t j = (e & 0x3FFFFFFFu) - u0;
            const bool mine = k0 + k < t.bd_k && e != VTX_INVALID && j < nu;
            v[k] = grad[e >> 30][mine ? j : 0u];
            on[k] = mine && act[mine ? j : 0u];
            last = j;
        }
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) {
            const V3 sum = madd(delta, xyz(v[k]), -w * v[k].w);
            delta = v3(on[k] ? sum.x : delta.x, on[k] ? sum.y : delta.y, on[k] ? sum.z : delta.z);
            cnt += on[k] ? 1 : 0;
        }
        return last;
    };
    // the particle's terms among the round's records. Its entries ascend, so the rounds keep the order, and where
    // there are many a later round goes on at the first group of four (next) that was not used up: with every
    // round over all entries, a mesh with a vertex of 20,000 bends took 707 ms a frame of 8 passes (now 87). Few
    // entries are gone over again in each round, as the lanes' own places cost more (251,001 particles of an
    // irregular mesh 1,271 us a frame of 32 passes, with them 1,490)
    uint32_t next = 0;
    const auto add = [&](uint32_t u0) {
        const uint32_t nu = min(t.ub_n - u0, (uint32_t)UB);
        if (!ANY || t.ub_n <= UB || t.bd_k <= VTX_MANY_BENDS) {
            for (uint32_t k0 = 0; k0 < t.bd_k; k0 += 4) add4(u0, nu, k0);
            return;
        }
        for (; next < t.bd_k; next += 4)
            if (add4(u0, nu, next) >= nu) break;
    };

    // the first entry rows (contiguous: row k at k * VTX_TILE), loaded while the records are evaluated
    constexpr uint32_t ER = NE * VTX_TILE / MT;
    uint32_t er[ER];
    const uint32_t nent = min(t.bd_k, NE) * VTX_TILE;
#pragma unroll
    for (uint32_t k = 0; k < ER; k++) er[k] = k * MT + tid < nent ? (d.bd + t.bd_off)[k * MT + tid] : VTX_INVALID;
    evaluate(0);
    if (vertex) {
        const float4 p4 = P[g - sg.pbase];
        p = xyz(p4);
        w = p4.w;
        stretch_terms(d, sg, t, P, tid, g - sg.pbase, p, w, delta, cnt);
        attach_terms<4>(d, sg, t.at_off, t.at_k, tid, g - sg.pbase, p, w, delta, cnt);
    }
#pragma unroll
    for (uint32_t k = 0; k < ER; k++) ent[k * MT + tid] = er[k];
    __syncthreads();
    if (vertex) add(0);
    for (uint32_t u0 = UB; u0 < t.ub_n; u0 += UB) {
        __syncthreads();                                // the records of the round before are read
        evaluate(u0);
        __syncthreads();
        if (vertex) add(u0);
    }
    if (!vertex) return;
    if (cnt > 0) p = madd(p, delta, frcp((float)cnt) * sg.omega);
    epilogue<EPI>(d, sg, g, in, p, w, h);
}

// Tiles without bending constraints in a set that has no others: one thread per particle and no LDS, of which
// k_iterate holds 64 KB (490,000 particles 605 -> 419 us a frame of 32 passes, 576 particles 133 -> 127).
template <int EPI>
__global__ __launch_bounds__(VTX_TILE) void k_iterate_plain(DevState d, const TileDev* __restrict__ tiles, int in, float h) {
    plain_particle<EPI>(d, tiles[tile_of(d.remap)], threadIdx.x, in, h);
}

// ---------------------------------------------------------------- grid stencil path
// A segment whose cloth is an R x C vertex grid with the reference's topology (structural +
// shear stretch, bending on the X/R/D slots of the cells) runs its Jacobi pass on 16 x 16
// tiles. The tile's positions plus a halo of 2 are staged in LDS; every bending slot touching
// the tile is evaluated once (not once per member vertex), its four corrections are kept in
// LDS, and each vertex gathers its 8 stretch terms, its attachments and its 12 bending terms in
// a fixed order. The three slot types are evaluated one after another through the same LDS
// area (X, then R, then D), which keeps the workgroup at ~18 KB of LDS (8 workgroups per CU). A large live
// set is bound by VALU issue (1024 x 1024: 99% of the 24 us in which the CUs are busy, of 28.2 us a pass):
// of 869 instructions a wave, 430 are the slots' arithmetic, 180 the stretch terms. Cell indices by 24-bit products with the division shared between types, and staging
// without divisions took it from 28.7 to 28.2 us (512 cloths of 963,130 particles 3174 -> 3129 us a frame
// pair). Vectors of four per role instead of the planes take 21 KB, one workgroup less per CU: 31.5 us.
// Slot owner ranges relative to the tile origin (a0, b0): X rows/cols [-1, 15] (17 x 17),
// R rows [-1, 16] cols [-1, 15] (18 x 17), D rows [-1, 15] cols [-1, 16] (17 x 18).
#define VTX_NSX (17 * 17)
#define VTX_NSR (18 * 17)
#define VTX_NSD (17 * 18)
#define VTX_NSMAX VTX_NSR
#define VTX_NSP 320   // plane pitch: whole banks, so two planes go in one LDS instruction

// Owner cells of one slot type that can hold a slot in a tile, tile-relative: rows
// [ra0, ra0 + h), columns [rb0, rb0 + w). The type's owner range of the tile (X: rows and columns
// -1..15, R: rows -1..16, D: columns -1..16) clipped to the cells where the slot is geometrically
// possible (X: a <= R-2, b <= C-2; R: also a >= 1; D: also b >= 1). h or w <= 0: none.
template <int TYPE>
__device__ __forceinline__ void slot_rect(int a0, int b0, int rows, int cols, int& ra0, int& rb0, int& h, int& w) {
    constexpr int RA1 = TYPE == 1 ? 16 : 15, RB1 = TYPE == 2 ? 16 : 15;
    ra0 = max(-1, (TYPE == 1 ? 1 : 0) - a0);
    rb0 = max(-1, (TYPE == 2 ? 1 : 0) - b0);
    h = min(RA1, rows - 2 - a0) - ra0 + 1;
    w = min(RB1, cols - 2 - b0) - rb0 + 1;
}

// Offsets of a slot's vertices from its owner cell in a staged tile of row pitch PITCH: the canonical
// vertex order per type (vtx_device.hpp).
template <int TYPE, int PITCH>
struct SlotAt {
    static constexpr int i0 = TYPE == 0 ? 0 : TYPE == 1 ? -PITCH + 1 : PITCH - 1;
    static constexpr int i1 = TYPE == 0 ? PITCH + 1 : TYPE == 1 ? PITCH : 1;
    static constexpr int i2 = TYPE == 0 ? 1 : TYPE == 1 ? 0 : PITCH;
    static constexpr int i3 = TYPE == 0 ? PITCH : TYPE == 1 ? 1 : 0;
};

// The cells of a type's rectangle are dealt to the threads densely (thread t: row t / w, column t % w), so
// a tile cut by the cloth's edge runs no lanes on cells that cannot hold a slot. X and R have the same
// columns, so one division serves both. recip: GridTileDev::recip (t < 324, w <= 18).
struct SlotCell {
    uint32_t t, q, c;
    __device__ __forceinline__ SlotCell(uint32_t t_, uint32_t w, uint32_t recip) : t(t_) {
        q = __umul24(t, recip) >> 15;
        c = t - __umul24(q, w);
    }
};

// Evaluate one cell's bending slot of a type into LDS at its row-major index in the type's range, in
// planes 3k..3k+2 of corr: g_k = -lam d_k for roles 0..2, the type's mark in act. Role 3's is
// -(g_0 + g_1 + g_2), as the four gradients of a dihedral angle sum to zero, and each vertex scales the
// sum of its terms by its own inverse mass. A slot that contributes nothing keeps an older mark.
// ra0, rb0: slot_rect's; base: the rectangle's first cell.
template <int TYPE>
__device__ __forceinline__ void eval_slot(const DevState& d, const SegDev& sg, const float4* sp,
                                          float (*corr)[VTX_NSP], uint8_t* act, uint32_t base, int cols, int ra0, int rb0,
                                          SlotCell s, float xpbd) {
    constexpr uint32_t W = TYPE == 2 ? 18 : 17;                             // owner columns of the range
    // in the rectangle every slot of a FULL type is present; otherwise the cell's flags tell
    const uint32_t cell = __umul24(s.q, (uint32_t)cols) + s.c;              // from the rectangle's first
    if (!((sg.flags >> (3 + TYPE)) & 1u) && !(((d.gflags + base)[cell] >> TYPE) & 1u)) return;
    const uint32_t o = __umul24(s.q, VTX_GP) + s.c + (uint32_t)((ra0 + VTX_GH) * VTX_GP + rb0 + VTX_GH);   // staged owner
    using A = SlotAt<TYPE, VTX_GP>;
    const float4 q0 = sp[o + A::i0], q1 = sp[o + A::i1], q2 = sp[o + A::i2], q3 = sp[o + A::i3];
    float rest = 0.f;
    if (!(sg.flags & VTX_SEG_BEND_REST0)) rest = reinterpret_cast<const float*>(d.brest4 + base + cell)[TYPE];
    float lam;
    BendGrad bg;
    if (!bend_eval<true>(q0, q1, q2, q3, rest, xpbd, lam, bg)) return;
    const uint32_t j = __umul24(s.q, W) + s.c + (uint32_t)((ra0 + 1) * (int)W + rb0 + 1);
    const V3 g0 = (-lam * bg.k0) * bg.c1, g1 = (-lam * bg.k1) * bg.c2, g2 = -lam * bg.d2;
    corr[0][j] = g0.x; corr[1][j] = g0.y; corr[2][j] = g0.z;
    corr[3][j] = g1.x; corr[4][j] = g1.y; corr[5][j] = g1.z;
    corr[6][j] = g2.x; corr[7][j] = g2.y; corr[8][j] = g2.z;
    act[j] = TYPE + 1;
}

// One slot type of a tile: the evaluations, then every tile vertex adds its four memberships of this type
// in role order to bend (gradients times -lam; the vertex's inverse mass is applied to the sum).
template <int TYPE>
__device__ __forceinline__ void bend_type_pass(const DevState& d, const SegDev& sg, const float4* sp,
                                               float (*corr)[VTX_NSP], uint8_t* act, int a0, int b0, int rows, int cols,
                                               SlotCell s0, SlotCell s1, float xpbd, bool inside, int ty, int tx,
                                               V3& bend, int& cnt) {
    if (!((sg.flags >> (6 + TYPE)) & 1u)) {   // the type is present at all
        int ra0, rb0, h, w;
        slot_rect<TYPE>(a0, b0, rows, cols, ra0, rb0, h, w);
        const uint32_t n = h > 0 && w > 0 ? (uint32_t)(h * w) : 0u;
        const uint32_t base = sg.pbase + (uint32_t)((a0 + ra0) * cols + b0 + rb0);
        static_assert(2 * VTX_TILE >= VTX_NSMAX, "a slot type fits two rounds of the workgroup");
        if (s0.t < n) eval_slot<TYPE>(d, sg, sp, corr, act, base, cols, ra0, rb0, s0, xpbd);
        if (s1.t < n) eval_slot<TYPE>(d, sg, sp, corr, act, base, cols, ra0, rb0, s1, xpbd);
    }
    __syncthreads();
    if (inside) {
        // role r of the slot owned at (ty + dy_r, tx + dx_r), per type:
        //   X: (0,0) (-1,-1) (0,-1) (-1,0);  R: (1,-1) (-1,0) (0,0) (0,-1);  D: (-1,1) (0,-1) (-1,0) (0,0)
        constexpr int W = TYPE == 2 ? 18 : 17;
        constexpr int DY[4] = {TYPE == 0 ? 0 : TYPE == 1 ? 1 : -1, TYPE == 2 ? 0 : -1, TYPE == 2 ? -1 : 0, TYPE == 0 ? -1 : 0};
        constexpr int DX[4] = {TYPE == 0 ? 0 : TYPE == 1 ? -1 : 1, TYPE == 1 ? 0 : -1, TYPE == 0 ? -1 : 0, TYPE == 1 ? -1 : 0};
        const int j0 = (ty + 1) * W + tx + 1;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = j0 + DY[r] * W + DX[r];
            if (act[j] != TYPE + 1) continue;
            if (r < 3)
                bend += v3(corr[3 * r][j], corr[3 * r + 1][j], corr[3 * r + 2][j]);
            else
                bend -= v3(corr[0][j], corr[1][j], corr[2][j]) + v3(corr[3][j], corr[4][j], corr[5][j]) +
                        v3(corr[6][j], corr[7][j], corr[8][j]);
            cnt++;
        }
    }
    __syncthreads();   // the next type reuses corr
}

__device__ __forceinline__ float4 nan4() {
    const float q = __int_as_float(0x7FC00000);
    return make_float4(q, q, q, q);
}

template <int EPI>
__global__ __launch_bounds__(VTX_TILE) void k_iterate_grid(DevState d, const GridTileDev* __restrict__ tiles,
                                                                   int in, float h) {
    __shared__ float4 sp[VTX_GP * VTX_GP];
    __shared__ float corr[9][VTX_NSP];           // plane r*3+c: component c of role r's g_r
    __shared__ uint32_t actw[(VTX_NSMAX + 3) / 4];   // the type whose slot last contributed there
    uint8_t* const act = reinterpret_cast<uint8_t*>(actw);
    const GridTileDev t = tiles[tile_of(d.remap)];
    const SegDev sg = d.segs[t.seg];
    const int rows = (int)sg.rows, cols = (int)sg.cols;
    const int a0 = (int)t.a0, b0 = (int)t.b0;
    const uint32_t tid = threadIdx.x;
    const float4* __restrict__ P = d.P[in];
    const int ty = (int)(tid / VTX_GT), tx = (int)(tid % VTX_GT);
    const int a = a0 + ty, b = b0 + tx;
    const bool inside = a < rows && b < cols;
    // offsets from the tile's first vertex stay in 32 bits (cols < 2^22)
    const uint32_t first = sg.pbase + (uint32_t)(a0 * cols + b0);
    const uint32_t own = inside ? __umul24((uint32_t)ty, (uint32_t)cols) + (uint32_t)tx : 0u;
    const uint32_t g = first + own;
    // stretch rest lengths: R own/left, D own/up, X-diagonal own/up-left, anti-diagonal of left/up,
    // issued before the staging loads and always (from the vertex itself where a neighbour is
    // missing): a load that a lane may skip leaves the outstanding count unknown to the compiler,
    // which then waits for every load before the first use
    const float4 r_own = d.rest4[g];
    float4 r_left = d.rest4[inside && b > 0 ? g - 1 : g];
    float4 r_up = d.rest4[inside && a > 0 ? g - cols : g];
    float4 r_ul = d.rest4[inside && a > 0 && b > 0 ? g - cols - 1 : g];
    if (!(b > 0)) r_left = nan4();
    if (!(a > 0)) r_up = nan4();
    if (!(a > 0 && b > 0)) r_ul = nan4();

    // clear the slot marks; stage positions of rows [a0-2, a0+18) x cols [b0-2, b0+18)
    if (tid < (VTX_NSMAX + 3) / 4) actw[tid] = 0u;
    uint32_t sr = (tid * 3277u) >> 16, scol = tid - sr * VTX_GP;               // tid / 20 for tid < 256
#pragma unroll
    for (uint32_t e = tid; e < VTX_GP * VTX_GP; e += VTX_TILE) {
        const int sa = a0 - VTX_GH + (int)sr, sb = b0 - VTX_GH + (int)scol;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if ((uint32_t)sa < (uint32_t)rows && (uint32_t)sb < (uint32_t)cols)
            v = P[sg.pbase + (__umul24((uint32_t)sa, (uint32_t)cols) + (uint32_t)sb)];
        sp[e] = v;
        sr += VTX_TILE / VTX_GP;                                                // 256 = 12 rows and 16 columns on
        scol += VTX_TILE % VTX_GP;
        if (scol >= VTX_GP) {
            scol -= VTX_GP;
            sr++;
        }
    }

    __syncthreads();

    const int sc = (ty + VTX_GH) * VTX_GP + (tx + VTX_GH);    // staged index of this vertex
    const float4 p4 = sp[sc];
    V3 p = xyz(p4);
    const float w = p4.w;
    V3 delta = v3(0.f, 0.f, 0.f);
    int cnt = 0;

    if (inside) {
        const float k = -w * sg.stiffness;
        if (r_own.x == r_own.x) stretch_term(p, w, k, sp[sc + 1], r_own.x, delta, cnt);
        if (r_left.x == r_left.x) stretch_term(p, w, k, sp[sc - 1], r_left.x, delta, cnt);
        if (r_own.y == r_own.y) stretch_term(p, w, k, sp[sc + VTX_GP], r_own.y, delta, cnt);
        if (r_up.y == r_up.y) stretch_term(p, w, k, sp[sc - VTX_GP], r_up.y, delta, cnt);
        if (r_own.z == r_own.z) stretch_term(p, w, k, sp[sc + VTX_GP + 1], r_own.z, delta, cnt);
        if (r_ul.z == r_ul.z) stretch_term(p, w, k, sp[sc - VTX_GP - 1], r_ul.z, delta, cnt);
        if (r_left.w == r_left.w) stretch_term(p, w, k, sp[sc + VTX_GP - 1], r_left.w, delta, cnt);
        if (r_up.w == r_up.w) stretch_term(p, w, k, sp[sc - VTX_GP + 1], r_up.w, delta, cnt);
        attach_terms<1>(d, sg, t.at_off, t.at_k, tid, (uint32_t)(a * cols + b), p, w, delta, cnt);
    }
    // bending: X roles 0..3, R roles 0..3, D roles 0..3
    const float xpbd_bend = sg.bend_compliance * frcp(h) * frcp(h);   // compliance / h^2 (cu:173)
    V3 bend = v3(0.f, 0.f, 0.f);
    // the rectangles' columns: X and R from b0 (or 0) - 1, D from b0 (or 1) - 1 to one more (slot_rect)
    const uint32_t wx = (uint32_t)max(min(15, cols - 2 - b0) - max(-1, -b0) + 1, 0);
    const uint32_t wd = (uint32_t)max(min(16, cols - 2 - b0) - max(-1, 1 - b0) + 1, 0);
    const SlotCell x0(tid, wx, t.recip & 0xFFFFu), x1(tid + VTX_TILE, wx, t.recip & 0xFFFFu);
    bend_type_pass<0>(d, sg, sp, corr, act, a0, b0, rows, cols, x0, x1, xpbd_bend, inside, ty, tx, bend, cnt);
    bend_type_pass<1>(d, sg, sp, corr, act, a0, b0, rows, cols, x0, x1, xpbd_bend, inside, ty, tx, bend, cnt);
    const SlotCell d0(tid, wd, t.recip >> 16), d1(tid + VTX_TILE, wd, t.recip >> 16);
    bend_type_pass<2>(d, sg, sp, corr, act, a0, b0, rows, cols, d0, d1, xpbd_bend, inside, ty, tx, bend, cnt);
    if (!inside) return;
    delta = madd(delta, bend, w);
    if (cnt > 0) p = madd(p, delta, frcp((float)cnt) * sg.omega);
    epilogue<EPI>(d, sg, g, in, p, w, h);
}

// Several Jacobi passes of a T x T tile in one launch. A small or medium cloth gives a pass too little
// work for the chip: a pass is then its launch, the staging load and three barrier-separated slot
// phases, about 8 us whatever the size up to 200 x 200 vertices. Here a workgroup stages its tile with
// a halo of 2 vertices per pass and runs the passes on it in LDS, each on the region that the passes
// after it still need (2 vertices less on every side), so the halo's vertices are worked out again by
// the tiles that own them. Every vertex adds the terms of k_iterate_grid in the same order: the same
// result, bit for bit. The staged side is VTX_FS = 24 for every T: at most 4 passes for T = 8, 3 for
// T = 12, 2 for T = 16. A pass is bound by its chain of LDS reads and dependent arithmetic, so the
// three slot types are evaluated side by side (two barriers a pass), a slot leaves one 16-B word per
// role, and the sums run without branches. Per launch (40 x 40, T = 8): 4.4, 6.3, 9.0, 11.1 us for
// 1 to 4 passes, against 8.0 us for one pass of k_iterate_grid; of the 11.1 us, 6.1 us are VALU issue.
// Attachments: none, or dense ones of at most VTX_LRA_PARTS slots.
template <int T, int R = VTX_FS - 4>
struct FuseTile {
    static constexpr int HS = (VTX_FS - T) / 2;                          // staged halo
    static constexpr int LO = HS + (T - R) / 2;                          // staged row / column of region (0, 0)
    // slots around the region by type (X, R, D): owner rows and columns from -1
    static constexpr int NX = (R + 1) * (R + 1), NR = (R + 2) * (R + 1);
    static constexpr int NS = NX + 2 * NR;
    static constexpr int UX = (NX + 63) / 64, UR = (NR + 63) / 64, UNITS = UX + 2 * UR;   // waves' shares
};

// One slot of type TYPE (index e of the type's range around the region) into corr[role][slot], NR roles:
// g_r and the pass's mark in w. A slot that contributes nothing keeps an older mark.
template <int T, int R, int TYPE, int NR, int NS>
__device__ __forceinline__ void fuse_slot(const DevState& d, const SegDev& sg, const float4* sp, float4 (&corr)[NR][NS],
                                          uint32_t mark, int a0, int b0, int e,
                                          float xpbd) {
#pragma clang fp contract(off)   // role 3: the products round before they are added, as in k_iterate_grid's gather
    using F = FuseTile<T, R>;
    constexpr int W = R + (TYPE == 2 ? 2 : 1);
    const int ra = e / W, rb = e % W;                      // owner cell + (1, 1), relative to the region
    const int a = a0 + F::LO - F::HS + ra - 1, b = b0 + F::LO - F::HS + rb - 1;
    const int rows = (int)sg.rows, cols = (int)sg.cols;
    if (e >= (TYPE == 0 ? F::NX : F::NR) || a < (TYPE == 1 ? 1 : 0) || a > rows - 2 || b < (TYPE == 2 ? 1 : 0) ||
        b > cols - 2)
        return;
    const uint32_t cell = sg.pbase + (uint32_t)(a * cols + b);
    if (!((sg.flags >> (3 + TYPE)) & 1u) && !((d.gflags[cell] >> TYPE) & 1u)) return;
    const int o = (ra + F::LO - 1) * VTX_FS + rb + F::LO - 1;
    using A = SlotAt<TYPE, VTX_FS>;
    const float4 q0 = sp[o + A::i0], q1 = sp[o + A::i1], q2 = sp[o + A::i2], q3 = sp[o + A::i3];
    float rest = 0.f;
    if (!(sg.flags & VTX_SEG_BEND_REST0)) rest = reinterpret_cast<const float*>(d.brest4 + cell)[TYPE];
    float lam;
    BendGrad bg;
    if (!bend_eval<true>(q0, q1, q2, q3, rest, xpbd, lam, bg)) return;
    const V3 g0 = (-lam * bg.k0) * bg.c1, g1 = (-lam * bg.k1) * bg.c2, g2 = -lam * bg.d2;
    const int j = (TYPE == 0 ? 0 : TYPE == 1 ? F::NX : F::NX + F::NR) + e;
    corr[0][j] = f4(g0, __uint_as_float(mark));
    corr[1][j] = f4(g1, __uint_as_float(mark));
    corr[2][j] = f4(g2, __uint_as_float(mark));
    if constexpr (NR > 3)
        corr[3][j] = make_float4(-((g0.x + g1.x) + g2.x), -((g0.y + g1.y) + g2.y), -((g0.z + g1.z) + g2.z),
                                 __uint_as_float(mark));
}

// The four memberships of region vertex (y, x) in one slot type, added in role order. All LDS reads are
// issued before the first use; a slot that contributes nothing adds +0, which changes no sum.
template <int T, int R, int TYPE, int NR, int NS>
__device__ __forceinline__ void fuse_gather(const float4 (&corr)[NR][NS], uint32_t mark, int y, int x, V3& bend, int& cnt) {
    using F = FuseTile<T, R>;
    // role r of the slot owned at (y + dy_r, x + dx_r), per type (bend_type_pass)
    constexpr int dy[3][4] = {{0, -1, 0, -1}, {1, -1, 0, 0}, {-1, 0, -1, 0}};
    constexpr int dx[3][4] = {{0, -1, -1, 0}, {-1, 0, 0, -1}, {1, -1, 0, 0}};
    constexpr int W = R + (TYPE == 2 ? 2 : 1);
    const int o = (TYPE == 0 ? 0 : TYPE == 1 ? F::NX : F::NX + F::NR) + (y + 1) * W + x + 1;
    float4 g[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int j = o + dy[TYPE][r] * W + dx[TYPE][r];
        if (r < NR) {
            g[r] = corr[r][j];
        } else {
            const float4 u = corr[0][j], v = corr[1][j], q = corr[2][j];
            g[r] = make_float4(-((u.x + v.x) + q.x), -((u.y + v.y) + q.y), -((u.z + v.z) + q.z), u.w);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const bool on = __float_as_uint(g[r].w) == mark;
        bend += v3(on ? g[r].x : 0.f, on ? g[r].y : 0.f, on ? g[r].z : 0.f);
        cnt += on ? 1 : 0;
    }
}

// The eight stretch terms of the vertex at staged index sc, in the order of k_iterate_grid, with selects
// (an absent constraint has a NaN rest length); STEP neighbours are read at a time.
template <int STEP>
__device__ __forceinline__ void fuse_stretch(const SegDev& sg, const float4* sp, const float4* sr, int sc, V3 p, float w,
                                             V3& delta, int& cnt) {
    const float k = -w * sg.stiffness;
    const float4 r_own = sr[sc], r_left = sr[sc - 1], r_up = sr[sc - VTX_FS];
    const float rest[8] = {r_own.x, r_left.x, r_own.y, r_up.y, r_own.z, sr[sc - VTX_FS - 1].z, r_left.w, r_up.w};
    constexpr int at[8] = {1, -1, VTX_FS, -VTX_FS, VTX_FS + 1, -VTX_FS - 1, VTX_FS - 1, -VTX_FS + 1};
#pragma unroll
    for (int e0 = 0; e0 < 8; e0 += STEP) {
        float4 q[STEP];
#pragma unroll
        for (int e = 0; e < STEP; e++) q[e] = sp[sc + at[e0 + e]];
#pragma unroll
        for (int e = 0; e < STEP; e++) {   // stretch_term
            const float r = rest[e0 + e];
            const V3 diff = p - xyz(q[e]);
            const float dist = fsqrt(dot_fma(diff, diff)), wsum = w + q[e].w;
            const bool on = r == r && dist != r && wsum > 0.f;
            const V3 sum = madd(delta, diff, (dist - r) * k * frcp(wsum * (dist + VTX_EPSILON)));
            delta = v3(on ? sum.x : delta.x, on ? sum.y : delta.y, on ? sum.z : delta.z);
            cnt += on ? 1 : 0;
        }
        if (STEP < 8) __builtin_amdgcn_sched_barrier(0);
    }
}

// One pass on the region of side R centred on the tile; EPI applies to the last one (R == T). keep 1 or 2: the
// tile's positions before the last or the next to last pass go to P[in ^ 1] (launch_iterate_fused).
template <int EPI, int T, int R>
__device__ __forceinline__ void fuse_pass(const DevState& d, const SegDev& sg, float4* sp, const float4* sr,
                                          const float (*sl)[VTX_FS * VTX_FS], float4 (&corr)[4][FuseTile<T>::NS],
                                          uint32_t nslots, int a0, int b0, int in, int keep, float h, float xpbd) {
    using F = FuseTile<T, R>;
    constexpr uint32_t mark = (VTX_FS - R) / 4;            // one per region size
    const int tid = (int)threadIdx.x, lane = tid & 63;
    // bending slots, 64 of one type per wave and round; the last waves first, as the first ones hold
    // the vertices
    const int wave = (int)__builtin_amdgcn_readfirstlane((uint32_t)tid >> 6);
#pragma unroll
    for (int u0 = 0; u0 < F::UNITS; u0 += 16) {
        const int u = u0 + 15 - wave;
        if (u < F::UX) {
            if (!(sg.flags & VTX_SEG_NONE_X)) fuse_slot<T, R, 0>(d, sg, sp, corr, mark, a0, b0, u * 64 + lane, xpbd);
        } else if (u < F::UX + F::UR) {
            if (!(sg.flags & VTX_SEG_NONE_R))
                fuse_slot<T, R, 1>(d, sg, sp, corr, mark, a0, b0, (u - F::UX) * 64 + lane, xpbd);
        } else if (u < F::UNITS) {
            if (!(sg.flags & VTX_SEG_NONE_D))
                fuse_slot<T, R, 2>(d, sg, sp, corr, mark, a0, b0, (u - F::UX - F::UR) * 64 + lane, xpbd);
        }
    }
    const int y = tid / R, x = tid % R;
    const int a = a0 + F::LO - F::HS + y, b = b0 + F::LO - F::HS + x;
    const bool inside = tid < R * R && a >= 0 && a < (int)sg.rows && b >= 0 && b < (int)sg.cols;
    const int sc = (y + F::LO) * VTX_FS + x + F::LO;
    V3 p = v3(0.f, 0.f, 0.f), delta = p;
    float w = 0.f;
    int cnt = 0;
    if (inside) {
        const float4 p4 = sp[sc];
        p = xyz(p4);
        w = p4.w;
        if (EPI == EPI_FINALIZE && R <= T + 4 && keep == (R - T) / 4 + 1) {
            constexpr int O = (R - T) / 2;                  // the tile within the region
            if (y >= O && y < O + T && x >= O && x < O + T) d.P[in ^ 1][sg.pbase + (uint32_t)(a * (int)sg.cols + b)] = p4;
        }
        fuse_stretch<8>(sg, sp, sr, sc, p, w, delta, cnt);
        for (uint32_t s = 0; s < nslots; s++) {                 // every slot is a part of its own
            V3 part = v3(0.f, 0.f, 0.f);
            attach_term(p, w, d.slots[sg.sbase + s], sl[s][sc], sg.lrs, part, cnt);
            delta += part;
        }
    }
    __syncthreads();
    if (inside) {
        V3 bend = v3(0.f, 0.f, 0.f);
        fuse_gather<T, R, 0>(corr, mark, y, x, bend, cnt);
        fuse_gather<T, R, 1>(corr, mark, y, x, bend, cnt);
        fuse_gather<T, R, 2>(corr, mark, y, x, bend, cnt);
        delta = madd(delta, bend, w);
        if (cnt > 0) p = madd(p, delta, frcp((float)cnt) * sg.omega);
        if (R > T) sp[sc] = f4(p, w);
        else epilogue<EPI>(d, sg, sg.pbase + (uint32_t)(a * (int)sg.cols + b), in, p, w, h);
    }
    if (R > T) __syncthreads();
}

template <int EPI, int T>
__global__ __launch_bounds__(1024) void k_iterate_fused(DevState d, const GridTileDev* __restrict__ tiles, int in,
                                                        int passes, int keep, float h) {
    using F = FuseTile<T>;
    __shared__ float4 sp[VTX_FS * VTX_FS];                    // positions
    __shared__ float4 sr[VTX_FS * VTX_FS];                    // owned stretch rest lengths, NaN off the cloth
    __shared__ float sl[VTX_LRA_PARTS][VTX_FS * VTX_FS];      // attachment distances
    __shared__ float4 corr[4][F::NS];                         // per role: g, mark of the pass that wrote it
    const GridTileDev t = tiles[tile_of(d.remap)];
    const SegDev sg = d.segs[t.seg];
    const int rows = (int)sg.rows, cols = (int)sg.cols, a0 = (int)t.a0, b0 = (int)t.b0;
    const int tid = (int)threadIdx.x;
    const uint32_t nslots = sg.flags & VTX_SEG_LRA_DENSE ? sg.scount : 0u;
    {
        const int ra = tid / VTX_FS - F::HS, rb = tid % VTX_FS - F::HS, a = a0 + ra, b = b0 + rb, H = 2 * passes;
        float4 p = make_float4(0.f, 0.f, 0.f, 0.f), r = nan4();
        const bool in_cloth = tid < VTX_FS * VTX_FS && ra >= -H && ra < T + H && rb >= -H && rb < T + H && a >= 0 &&
                              a < rows && b >= 0 && b < cols;
        const uint32_t v = in_cloth ? (uint32_t)(a * cols + b) : 0u;
        if (in_cloth) {
            p = d.P[in][sg.pbase + v];
            r = d.rest4[sg.pbase + v];
        }
        for (int e = tid; e < F::NS; e += 1024)                           // while the loads are in flight
#pragma unroll
            for (int r = 0; r < 4; r++) corr[r][e].w = 0.f;
        if (in_cloth)
            for (uint32_t s = 0; s < nslots; s++) sl[s][tid] = d.lra[4 * (size_t)sg.lbase + (size_t)s * sg.n + v];
        if (tid < VTX_FS * VTX_FS) {
            sp[tid] = p;
            sr[tid] = r;
        }
    }
    __syncthreads();
    const float xpbd = sg.bend_compliance * frcp(h) * frcp(h);   // compliance / h^2 (cu:173)
    if constexpr (T <= 8)
        if (passes > 3) fuse_pass<EPI, T, T + 12>(d, sg, sp, sr, sl, corr, nslots, a0, b0, in, keep, h, xpbd);
    if constexpr (T <= 12)
        if (passes > 2) fuse_pass<EPI, T, T + 8>(d, sg, sp, sr, sl, corr, nslots, a0, b0, in, keep, h, xpbd);
    if (passes > 1) fuse_pass<EPI, T, T + 4>(d, sg, sp, sr, sl, corr, nslots, a0, b0, in, keep, h, xpbd);
    fuse_pass<EPI, T, T>(d, sg, sp, sr, sl, corr, nslots, a0, b0, in, keep, h, xpbd);
}

// One pass of a 16 x 16 tile of a cloth with many dense attachments (VTX_SEG_LRA_TILED, at least
// VTX_LRA_SPLIT_MIN slots), four threads per vertex: thread q of a vertex sums attachment part q, the
// first adds the parts in order after its stretch terms, and the other waves evaluate the bending slots.
// A 256 x 256 cloth gives one tile per CU: the distances come as one 16-B load per four slots,
// contiguous over the tile (the slot-major order gives 64-B runs), started before the positions are
// staged, and there is one barrier between the terms and the sums. At 256 slots the pass is bound by the
// 67 MB of distances, which no L2 keeps from one launch to the next: 19.6 -> 17.9 us alone (67 MB at the
// 5.2 TB/s that overlapping passes reach are 12.9 us), 862 -> 652 us a frame with three solvers' passes
// overlapping, for which the registers and LDS leave room for two workgroups per CU (with all four roles
// in LDS and one workgroup per CU 16.7 us alone, but 743 us a frame overlapping).
template <int EPI, int B>
__global__ __launch_bounds__(1024, 8) void k_iterate_split(DevState d, const GridTileDev* __restrict__ tiles, int in, float h) {
    constexpr int T = VTX_GT;
    using F = FuseTile<T, T>;
    __shared__ float4 sp[VTX_FS * VTX_FS];
    __shared__ float4 sr[VTX_FS * VTX_FS];
    __shared__ float4 corr[3][F::NS];                         // role 3 from the others: two workgroups per CU
    __shared__ float4 lpart[VTX_LRA_PARTS - 1][VTX_TILE];
    static_assert(VTX_LRA_PARTS * VTX_TILE == 1024, "a thread per vertex and part");
    const GridTileDev t = tiles[tile_of(d.remap)];
    const SegDev sg = d.segs[t.seg];
    const int rows = (int)sg.rows, cols = (int)sg.cols, a0 = (int)t.a0, b0 = (int)t.b0;
    const int tid = (int)threadIdx.x, lane = tid % VTX_TILE;
    const uint32_t qpart = __builtin_amdgcn_readfirstlane((uint32_t)tid / VTX_TILE);   // wave-uniform
    uint32_t s0, s1;
    lra_part_range(sg, qpart, s0, s1);
    const float4* __restrict__ dist = tiled_part(d, sg, t.at_off, qpart, (uint32_t)lane);
    TiledBatch<B> first = {};
    if (s0 < s1) first.load(dist, 0, (s1 - s0 + 3) / 4);
    {   // positions and rest lengths of the tile and two vertices around it
        const int ra = tid / VTX_FS - F::HS, rb = tid % VTX_FS - F::HS, a = a0 + ra, b = b0 + rb;
        const bool in_cloth = tid < VTX_FS * VTX_FS && ra >= -2 && ra < T + 2 && rb >= -2 && rb < T + 2 && a >= 0 &&
                              a < rows && b >= 0 && b < cols;
        float4 p = make_float4(0.f, 0.f, 0.f, 0.f), r = nan4();
        if (in_cloth) {
            const uint32_t v = sg.pbase + (uint32_t)(a * cols + b);
            p = d.P[in][v];
            r = d.rest4[v];
        }
        for (int e = tid; e < F::NS; e += 1024)                           // no slot marked
#pragma unroll
            for (int r = 0; r < 3; r++) corr[r][e].w = 0.f;
        if (tid < VTX_FS * VTX_FS) {
            sp[tid] = p;
            sr[tid] = r;
        }
    }
    __syncthreads();
    const float xpbd = sg.bend_compliance * frcp(h) * frcp(h);   // compliance / h^2 (cu:173)
    constexpr uint32_t mark = 1;
    const int y = lane / T, x = lane % T, a = a0 + y, b = b0 + x;
    const int sc = (y + F::LO) * VTX_FS + x + F::LO;
    const bool in_cloth = a < rows && b < cols, inside = in_cloth && qpart == 0;
    const float4 p4 = sp[sc];
    V3 p = xyz(p4), delta = v3(0.f, 0.f, 0.f), part = delta;
    const float w = p4.w;
    int cnt = 0, pc = 0;
    if (inside) fuse_stretch<2>(sg, sp, sr, sc, p, w, delta, cnt);
    if (in_cloth) {
        if (s0 < s1) attach_tiled<B>(d, sg, dist, first, s0, s1, p, w, part, pc);
        if (qpart > 0) lpart[qpart - 1][lane] = f4(part, __int_as_float(pc));
    }
    // bending slots, 64 of one type per wave and round, on the waves of parts 1..3
    const int wave = (int)__builtin_amdgcn_readfirstlane((uint32_t)tid >> 6), nw = 12;
    if (qpart > 0)
#pragma unroll
        for (int u0 = 0; u0 < F::UNITS; u0 += nw) {
            const int u = u0 + 15 - wave;
            if (u < F::UX) {
                if (!(sg.flags & VTX_SEG_NONE_X)) fuse_slot<T, T, 0>(d, sg, sp, corr, mark, a0, b0, u * 64 + tid % 64, xpbd);
            } else if (u < F::UX + F::UR) {
                if (!(sg.flags & VTX_SEG_NONE_R))
                    fuse_slot<T, T, 1>(d, sg, sp, corr, mark, a0, b0, (u - F::UX) * 64 + tid % 64, xpbd);
            } else if (u < F::UNITS) {
                if (!(sg.flags & VTX_SEG_NONE_D))
                    fuse_slot<T, T, 2>(d, sg, sp, corr, mark, a0, b0, (u - F::UX - F::UR) * 64 + tid % 64, xpbd);
            }
        }
    __syncthreads();
    if (!inside) return;
    delta += part;
    cnt += pc;
#pragma unroll
    for (int q = 0; q < VTX_LRA_PARTS - 1; q++) {
        const float4 e = lpart[q][lane];
        delta += xyz(e);
        cnt += __float_as_int(e.w);
    }
    __builtin_amdgcn_sched_barrier(0);                      // few words live at a time: 64 registers a thread
    V3 bend = v3(0.f, 0.f, 0.f);
    fuse_gather<T, T, 0>(corr, mark, y, x, bend, cnt);
    __builtin_amdgcn_sched_barrier(0);
    fuse_gather<T, T, 1>(corr, mark, y, x, bend, cnt);
    __builtin_amdgcn_sched_barrier(0);
    fuse_gather<T, T, 2>(corr, mark, y, x, bend, cnt);
    delta = madd(delta, bend, w);
    if (cnt > 0) p = madd(p, delta, frcp((float)cnt) * sg.omega);
    epilogue<EPI>(d, sg, sg.pbase + (uint32_t)(a * cols + b), in, p, w, h);
}

// ComputeTriangleNormals + ComputeVertexNormals (Velvet/VtClothSolverGPU.cu:419-450) as a
// per-vertex gather over incident triangles (segments off the grid path).
__global__ __launch_bounds__(VTX_TILE) void k_normals(DevState d, const TileDev* __restrict__ tiles) {
    const TileDev t = tiles[tile_of(d.remap)];
    const uint32_t lane = threadIdx.x;
    if (lane >= t.count) return;
    const SegDev sg = d.segs[t.seg];
    const uint32_t g = t.begin + lane;
    V3 s = v3(0.f, 0.f, 0.f);
    const uint32_t* __restrict__ tr = d.tr + t.tr_off + lane;
    for (uint32_t k = 0; k < t.tr_k; k++) {
        const uint32_t e = tr[(size_t)k * VTX_TILE];
        if (e == VTX_INVALID) continue;
        const uint4 ix = d.trec[sg.trbase + e];
        const uint32_t pb = sg.pbase;
        const V3 a = xyz(d.X[pb + ix.x]), b = xyz(d.X[pb + ix.y]), c = xyz(d.X[pb + ix.z]);
        s += cross(b - a, c - a);
    }
    d.Nrm[g] = f4(normalize(s), 0.f);
}

// The same for a grid segment's 16 x 16 tile: positions of the tile and a one-vertex halo staged
// in LDS, one read per vertex instead of the incidence gather. Quad (a, b) holds triangles
// (A, B, C) and (C, B, D) with A = (a, b), B = (a+1, b), C = (a, b+1), D = (a+1, b+1) (the grid
// the stencil path accepts), so a vertex's incident triangles in triangle-index order are T1 of
// quad (r-1, c-1), T0 and T1 of (r-1, c), T0 and T1 of (r, c-1), T0 of (r, c), each crossed as
// cross(b - a, c - a) in its stored vertex order: the terms and the order of the general gather.
__global__ __launch_bounds__(VTX_TILE) void k_normals_grid(DevState d, const GridTileDev* __restrict__ tiles) {
    constexpr int GS = VTX_GT + 2;                 // staged side: tile + one-vertex halo
    __shared__ float4 sx[GS * GS];
    const GridTileDev t = tiles[tile_of(d.remap)];
    const SegDev sg = d.segs[t.seg];
    const int rows = (int)sg.rows, cols = (int)sg.cols, a0 = (int)t.a0, b0 = (int)t.b0;
    for (uint32_t e = threadIdx.x; e < GS * GS; e += VTX_TILE) {
        const int a = a0 - 1 + (int)(e / GS), b = b0 - 1 + (int)(e % GS);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (a >= 0 && a < rows && b >= 0 && b < cols) v = d.X[sg.pbase + (uint32_t)(a * cols + b)];
        sx[e] = v;
    }
    __syncthreads();
    const int ty = (int)(threadIdx.x / VTX_GT), tx = (int)(threadIdx.x % VTX_GT);
    const int r = a0 + ty, c = b0 + tx;
    if (r >= rows || c >= cols) return;
    auto at = [&](int dr, int dc) { return xyz(sx[(ty + 1 + dr) * GS + (tx + 1 + dc)]); };
    const V3 v = at(0, 0);
    V3 s = v3(0.f, 0.f, 0.f);
    if (r >= 1 && c >= 1) {                        // quad (r-1, c-1): v = D
        const V3 B = at(0, -1), C = at(-1, 0);
        s += cross(B - C, v - C);
    }
    if (r >= 1 && c + 1 < cols) {                  // quad (r-1, c): v = B
        const V3 A = at(-1, 0), C = at(-1, 1), D = at(0, 1);
        s += cross(v - A, C - A);
        s += cross(v - C, D - C);
    }
    if (r + 1 < rows && c >= 1) {                  // quad (r, c-1): v = C
        const V3 A = at(0, -1), B = at(1, -1), D = at(1, 0);
        s += cross(B - A, v - A);
        s += cross(B - v, D - v);
    }
    if (r + 1 < rows && c + 1 < cols) {            // quad (r, c): v = A
        const V3 B = at(1, 0), C = at(0, 1);
        s += cross(B - v, C - v);
    }
    d.Nrm[sg.pbase + (uint32_t)(r * cols + c)] = f4(normalize(s), 0.f);
}

// Failure detection: flags[t.seg] = 1 when a particle of the segment has a non-finite position
// or velocity (the reference has no such check; its only net is the speed clamp, cu:399-404).
__global__ void k_clear_flags(uint32_t* flags, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flags[i] = 0;
}

__global__ __launch_bounds__(VTX_TILE) void k_check_finite(DevState d, uint32_t* flags) {
    const TileDev t = d.tiles[tile_of(d.remap)];
    bool bad = false;
    if (threadIdx.x < t.count) {
        const uint32_t g = t.begin + threadIdx.x;
        const float4 x = d.X[g], v = d.V[g];
        bad = !(isfinite(x.x) && isfinite(x.y) && isfinite(x.z) && isfinite(v.x) && isfinite(v.y) && isfinite(v.z));
    }
    if (__any(bad) && (threadIdx.x & 63u) == 0) flags[t.seg] = 1u;   // same value from any wave: no race on the result
}

// ---------------------------------------------------------------- host launchers
static inline hipError_t last_launch() { return hipGetLastError(); }

// Collider and slot updates between two frames: the values are the launch's arguments, so nothing waits
// for the frame in flight and no host buffer has to outlive the call (a copy from host memory did both).
struct ColliderArgs {
    ColliderDev c[8];
};

__global__ __launch_bounds__(64) void k_set_colliders(ColliderDev* __restrict__ dst, ColliderArgs a, uint32_t n) {
    const uint32_t words = n * (uint32_t)(sizeof(ColliderDev) / 4);
    for (uint32_t i = threadIdx.x; i < words; i += 64)
        reinterpret_cast<uint32_t*>(dst)[i] = reinterpret_cast<const uint32_t*>(a.c)[i];
}

__global__ __launch_bounds__(64) void k_set_slot(float4* __restrict__ dst, float4 v) {
    if (threadIdx.x == 0) *dst = v;
}

hipError_t launch_set_colliders(ColliderDev* dst, const ColliderDev* src, uint32_t n, hipStream_t s) {
    for (uint32_t c0 = 0; c0 < n; c0 += 8) {
        ColliderArgs a{};
        const uint32_t k = n - c0 < 8 ? n - c0 : 8u;
        for (uint32_t c = 0; c < k; c++) a.c[c] = src[c0 + c];
        hipLaunchKernelGGL(k_set_colliders, dim3(1), dim3(64), 0, s, dst + c0, a, k);
    }
    return hipGetLastError();
}

hipError_t launch_set_slot(float4* dst, float4 v, hipStream_t s) {
    hipLaunchKernelGGL(k_set_slot, dim3(1), dim3(64), 0, s, dst, v);
    return hipGetLastError();
}

hipError_t launch_frame_begin(const DevState& d, float frame_dt, float h, hipStream_t s) {
    if (!d.ntiles) return hipSuccess;
    hipLaunchKernelGGL(k_frame_begin, dim3(d.ntiles), dim3(VTX_TILE), 0, s, d, frame_dt, h);
    return last_launch();
}

hipError_t launch_collide(const DevState& d, int in, float h, int block, hipStream_t s) {
    if (!d.ntiles) return hipSuccess;
    const auto launch = [&](auto kernel, uint32_t bs) {
        hipLaunchKernelGGL(kernel, dim3(d.ntiles * (VTX_TILE / bs)), dim3(bs), 0, s, d, in, h);
    };
    // few particles with neighbours: the pass is the chain of its loads, so eight neighbours and their start positions at a
    // time, on many CUs; many: the lines it touches and the registers (102 for 72) count, so four, and start
    // positions of contacts only. Folded cloths, us a frame of ten contact passes, 4 / 8: 4,096 particles
    // 158 / 137, 40,000 190 / 175, 65,536 242 / 232, 131,044 302 / 313, 1,048,576 1109 / 1280. With segments on
    // several streams the launch's own particles count, for the search too (search_small): three folded cloths
    // of 230 x 230 on two / three streams 354 / 366 us a frame, with the live set's count 377 / 393; of
    // 350 x 350 579 / 591 and 580 / 600.
    if (collide_ahead(d)) launch(k_collide<64, 8>, 64);
    else if (block == 64) launch(k_collide<64, 4>, 64);
    else if (block == 128) launch(k_collide<128, 4>, 128);
    else launch(k_collide<256, 4>, 256);
    return last_launch();
}

static void launch_iterate_grid(const DevState& d, int in, float h, int epilogue, hipStream_t s) {
    if (!d.ngtiles) return;
    const dim3 gr(d.ngtiles), bl(VTX_TILE);
    if (epilogue == EPI_NONE) hipLaunchKernelGGL(k_iterate_grid<EPI_NONE>, gr, bl, 0, s, d, d.gtiles, in, h);
    else if (epilogue == EPI_FINALIZE) hipLaunchKernelGGL(k_iterate_grid<EPI_FINALIZE>, gr, bl, 0, s, d, d.gtiles, in, h);
    else hipLaunchKernelGGL(k_iterate_grid<EPI_FINALIZE_PREDICT>, gr, bl, 0, s, d, d.gtiles, in, h);
}

// B: groups of four distances in flight per thread
template <int B>
static void launch_iterate_split(const DevState& d, int in, float h, int epilogue, hipStream_t s) {
    if (!d.nltiles) return;
    const dim3 gr(d.nltiles), bl(VTX_TILE * VTX_LRA_PARTS);
    if (epilogue == EPI_NONE) hipLaunchKernelGGL((k_iterate_split<EPI_NONE, B>), gr, bl, 0, s, d, d.ltiles, in, h);
    else if (epilogue == EPI_FINALIZE) hipLaunchKernelGGL((k_iterate_split<EPI_FINALIZE, B>), gr, bl, 0, s, d, d.ltiles, in, h);
    else hipLaunchKernelGGL((k_iterate_split<EPI_FINALIZE_PREDICT, B>), gr, bl, 0, s, d, d.ltiles, in, h);
}

template <int RPT, bool ANY, int MT>
static void launch_iterate_mesh(const DevState& d, int in, float h, int epilogue, hipStream_t s) {
    constexpr uint32_t PT = MT / VTX_TILE;
    const uint32_t plain = ANY && RPT == 1 ? d.nptiles : 0u;
    const dim3 gr(d.nitiles - plain + (plain + PT - 1) / PT), bl(MT);
    const auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, gr, bl, 0, s, d, d.itiles, in, h); };
    if (epilogue == EPI_NONE) launch(k_iterate<EPI_NONE, RPT, ANY, MT>);
    else if (epilogue == EPI_FINALIZE) launch(k_iterate<EPI_FINALIZE, RPT, ANY, MT>);
    else launch(k_iterate<EPI_FINALIZE_PREDICT, RPT, ANY, MT>);
}

static void launch_iterate_plain(const DevState& d, int in, float h, int epilogue, hipStream_t s) {
    const dim3 gr(d.nptiles), bl(VTX_TILE);
    const auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, gr, bl, 0, s, d, d.itiles, in, h); };
    if (epilogue == EPI_NONE) launch(k_iterate_plain<EPI_NONE>);
    else if (epilogue == EPI_FINALIZE) launch(k_iterate_plain<EPI_FINALIZE>);
    else launch(k_iterate_plain<EPI_FINALIZE_PREDICT>);
}

hipError_t launch_iterate(const DevState& d, int in, float h, int epilogue, bool constraints, int lra_batch,
                          hipStream_t s) {
    if (!constraints) {   // no Jacobi pass: only the epilogue, over every particle
        if (!d.ntiles) return hipSuccess;
        dim3 gr(d.ntiles), bl(VTX_TILE);
        if (epilogue == EPI_NONE) hipLaunchKernelGGL(k_epilogue<EPI_NONE>, gr, bl, 0, s, d, in, h);
        else if (epilogue == EPI_FINALIZE) hipLaunchKernelGGL(k_epilogue<EPI_FINALIZE>, gr, bl, 0, s, d, in, h);
        else hipLaunchKernelGGL(k_epilogue<EPI_FINALIZE_PREDICT>, gr, bl, 0, s, d, in, h);
        return last_launch();
    }
    launch_iterate_grid(d, in, h, epilogue, s);
    // four threads per vertex leave 128 registers a thread: a batch of 64 distances runs as 16
    if (lra_batch >= 16) launch_iterate_split<4>(d, in, h, epilogue, s);
    else launch_iterate_split<1>(d, in, h, epilogue, s);
    if (!d.nitiles) return last_launch();
    if (d.nptiles == d.nitiles) {
        launch_iterate_plain(d, in, h, epilogue, s);
        return last_launch();
    }
    // a tile's records in one round while every tile has a CU of its own (8.5 against 11.5 us for 90
    // tiles of 1,334 records), else in rounds of half the LDS and twice the workgroups per CU (625 tiles
    // 28.5 against 33.4 us). Then 512 tiles are in flight at a time with 768 threads a tile, 768 with 512
    // threads, which take 1.3 times as long each: the fewer turns count. Frames of 32 passes, 768 / 512
    // threads: 352 tiles 459 / 503 us, 515 787 / 622 (one thread per particle 676), 791 925 / 1,013, 1,407
    // 1,361 / 1,207, 2,823 2,526 / 2,206, 981 of an irregular mesh 1,268 / 1,432 (three plain tiles as one)
    const bool many = d.live & VTX_LIVE_MANY_BENDS, any = many || d.nptiles;
    const uint32_t wg = d.nitiles - d.nptiles + d.nptiles / 3;
    const bool narrow = 13 * ((wg + 767) / 768) < 10 * ((wg + 511) / 512);
    if (d.nitiles <= 256) {
        if (many) launch_iterate_mesh<2, true, VTX_MT>(d, in, h, epilogue, s);
        else launch_iterate_mesh<2, false, VTX_MT>(d, in, h, epilogue, s);
    } else if (narrow) {
        if (any) launch_iterate_mesh<1, true, 512>(d, in, h, epilogue, s);
        else launch_iterate_mesh<1, false, 512>(d, in, h, epilogue, s);
    } else {
        if (any) launch_iterate_mesh<1, true, VTX_MT>(d, in, h, epilogue, s);
        else launch_iterate_mesh<1, false, VTX_MT>(d, in, h, epilogue, s);
    }
    return last_launch();
}

template <int T>
static void launch_fused(const DevState& d, int in, int passes, int keep, float h, int epilogue, hipStream_t s) {
    const dim3 gr(d.nftiles), bl(1024);
    if (epilogue == EPI_NONE) hipLaunchKernelGGL((k_iterate_fused<EPI_NONE, T>), gr, bl, 0, s, d, d.ftiles, in, passes, keep, h);
    else if (epilogue == EPI_FINALIZE) hipLaunchKernelGGL((k_iterate_fused<EPI_FINALIZE, T>), gr, bl, 0, s, d, d.ftiles, in, passes, keep, h);
    else hipLaunchKernelGGL((k_iterate_fused<EPI_FINALIZE_PREDICT, T>), gr, bl, 0, s, d, d.ftiles, in, passes, keep, h);
}

hipError_t launch_iterate_fused(const DevState& d, int in, int passes, int keep, float h, int epilogue, hipStream_t s) {
    if (!d.nftiles) return hipSuccess;
    if (passes < 1 || passes > fuse_passes(d.fside)) return hipErrorInvalidValue;   // the staged halo
    if (keep && (epilogue != EPI_FINALIZE || keep > passes)) return hipErrorInvalidValue;
    if (d.fside == 8) launch_fused<8>(d, in, passes, keep, h, epilogue, s);
    else if (d.fside == 12) launch_fused<12>(d, in, passes, keep, h, epilogue, s);
    else launch_fused<16>(d, in, passes, keep, h, epilogue, s);
    return last_launch();
}

hipError_t launch_check_finite(const DevState& d, uint32_t* flags, uint32_t nseg, hipStream_t s) {
    hipLaunchKernelGGL(k_clear_flags, dim3((nseg + 255) / 256), dim3(256), 0, s, flags, nseg);
    if (d.ntiles) hipLaunchKernelGGL(k_check_finite, dim3(d.ntiles), dim3(VTX_TILE), 0, s, d, flags);
    return last_launch();
}

hipError_t launch_normals(const DevState& d, hipStream_t s) {
    if (d.nitiles) hipLaunchKernelGGL(k_normals, dim3(d.nitiles), dim3(VTX_TILE), 0, s, d, d.itiles);
    if (d.ngtiles) hipLaunchKernelGGL(k_normals_grid, dim3(d.ngtiles), dim3(VTX_TILE), 0, s, d, d.gtiles);
    if (d.nltiles) hipLaunchKernelGGL(k_normals_grid, dim3(d.nltiles), dim3(VTX_TILE), 0, s, d, d.ltiles);
    if (d.nmtiles) hipLaunchKernelGGL(k_normals_grid, dim3(d.nmtiles), dim3(VTX_TILE), 0, s, d, d.mtiles);
    return last_launch();
}

}  // namespace vtx
