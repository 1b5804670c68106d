// pga_adjoint.hip - reverse mode over a derivation tape (gfx950).
//
// A tape-mode derivation keeps every level's parent records and child
// descriptors, materialises every fan-out (no in-place leaf expansion), and
// records one outcome per child: the terminal instance it emitted, or the
// parent record and descriptor range of the fan-out it became, or nothing.
// The tape freezes the topology (branches, repetition counts, rule choices).
//
// The backward pass runs one launch per level, last level first, one thread
// per child. Each thread recomputes its child from the tape (the parent
// record and the descriptor: the checkpoint of that depth), replays the
// child's chain of single-child operators, and propagates adjoints back:
//   instance = model4 * scale(size)  <- dL/dinstance of its terminal, or
//   the fan-out it became            <- the adjoints its children left in
//                                       their slots (parent state, offset and
//                                       size along the split axis), through
//                                       the running offsets of the split;
//   chain of single-child operators  (recomputed forward from its start);
//   child construction               -> this child's slot, read by its
//                                       parent's thread in the next launch.
// Parameter adjoints of PGA_PT_AXIOM_PARAM slots are summed with FP64
// atomic adds (many terms of both signs per parameter) and rounded to FP32
// once; every other parameter is a constant. Each slot is written
// by one thread and read by one, so the state adjoints are deterministic.
#include "pga_kernels.h"

namespace pga {

struct Adj {
    float m[12];
    float s[3];
};

__device__ __forceinline__ void adj_zero(Adj& d) {
#pragma unroll
    for (int i = 0; i < 12; ++i) d.m[i] = 0.0f;
    d.s[0] = d.s[1] = d.s[2] = 0.0f;
}

// dL/dparams of one thread. A thread replays one child, so every
// contribution is to the same axiom: up to kGradSlots per-axiom parameters
// accumulate in FP64 and leave once, at the end (flush_grads). The sums are in
// LDS, parameter q of the wave's lane l at word q * 64 + l of the wave's 4 KB:
// one LDS addition a contribution, where sums in registers, whose index must
// be a constant, took eight selected FP64 additions and 16 registers.
constexpr uint32_t kGradSlots = 8;
typedef __attribute__((address_space(3))) double lds_f64;
struct GradAcc {
    lds_f64* v;       // the lane's: parameter q at v[q * 64]
    uint32_t axiom;   // ~0u: no contribution yet
};

__device__ __forceinline__ void grad_zero(GradAcc& ga, lds_f64* wave) {
    ga.v = wave + (threadIdx.x & 63u);
#pragma unroll
    for (uint32_t q = 0; q < kGradSlots; ++q) ga.v[q * 64u] = 0.0;
    ga.axiom = ~0u;
}

// dL/dparam k of entry e for the shape of `axiom`: only per-axiom parameters
// are differentiable.
__device__ __forceinline__ void grad_param(const Ctx& c, const AdjArgs& g, GradAcc& ga, const EntryV& e, uint32_t k,
                                           uint32_t axiom, float v) {
    if (v == 0.0f || k >= e.nparams()) return;
    if (k < 3u && ((e.inl() >> k) & 1u)) return;
    const DevParam p = e.param(c, k);
    if (p.type != PGA_PT_AXIOM_PARAM || c.aparams_per == 0u) return;
    const uint32_t slot = (uint32_t)p.a;
    if (c.aparams_per <= kGradSlots && slot < kGradSlots && (ga.axiom == ~0u || ga.axiom == axiom)) {
        ga.axiom = axiom;
        // the lane's own word: an atomic for its form, one instruction and no wait
        __hip_atomic_fetch_add(ga.v + slot * 64u, (double)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    } else {
        atomicAdd(g.grad + (size_t)axiom * c.aparams_per + slot, (double)v);
    }
}

// The wave's contributions to the FP64 gradient, axiom by axiom: the lanes of
// one axiom are summed first, and every parameter of it is one global atomic.
// Eight lanes take a parameter each, so that all are summed at once: eight
// LDS reads (no two of the eight groups on the same chunk of lanes, against
// bank conflicts) and three shuffles, where a parameter after the other went
// through six shuffles of the whole wave. Fewer than eight lanes of an axiom
// add for themselves, which measures what reducing from two lanes on does; the
// atomics of many lanes on one line are what costs (reducing from 24 lanes on:
// 609 us instead of 434 for the second level from the end of 4,096 lots, 94
// instead of 32 for 256 lots). Every lane of the wave calls it.
__device__ __forceinline__ void flush_grads(const Ctx& c, const AdjArgs& g, const GradAcc& ga) {
    const uint32_t per = c.aparams_per;
    if (per == 0u || per > kGradSlots) return;
    unsigned long long left = __ballot(ga.axiom != ~0u);
    if (left == 0ull) return;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t lane = threadIdx.x & 63u, q = lane >> 3;
    const lds_f64* wave = ga.v - lane;
#pragma unroll 1
    while (left != 0ull) {
        const uint32_t ax = (uint32_t)__builtin_amdgcn_readlane((int)ga.axiom, __ffsll((long long)left) - 1);
        const unsigned long long of = __ballot(ga.axiom == ax);
        left &= ~of;
        if (__popcll(of) >= 8) {
            double x = 0.0;
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) {
                const uint32_t l = (lane & 7u) + 8u * ((k + q) & 7u);
                const double w = wave[q * 64u + l];
                x += (of >> l) & 1ull ? w : 0.0;
            }
#pragma unroll
            for (int d = 4; d >= 1; d >>= 1) x += __shfl_xor(x, d);
            if ((lane & 7u) == 0u && q < per && x != 0.0) atomicAdd(g.grad + (size_t)ax * per + q, x);
        } else if (ga.axiom == ax) {
            for (uint32_t k = 0; k < per; ++k) {
                const double w = ga.v[k * 64u];
                if (w != 0.0) atomicAdd(g.grad + (size_t)ax * per + k, w);
            }
        }
    }
}

// c = a * translate(t): da, dt from dc.
__device__ __forceinline__ void translate_adj(const float a[12], const float t[3], const float dc[12], float da[12],
                                              float dt[3]) {
    dt[0] = dt[1] = dt[2] = 0.0f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float d3 = dc[i * 4 + 3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            da[i * 4 + k] = dc[i * 4 + k] + d3 * t[k];
            dt[k] += a[i * 4 + k] * d3;
        }
        da[i * 4 + 3] = d3;
    }
}

// c = a * b (a 3x4 with the implicit row 0 0 0 1, b 4x4): da = dc * b^T.
__device__ __forceinline__ void mul_adj_a(const float b[16], const float dc[12], float da[12]) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            float s = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) s += dc[i * 4 + j] * b[k * 4 + j];
            da[i * 4 + k] = s;
        }
}

// Instance = model4 * scale(size) (GenerationFunctions.cuh:155-189).
__device__ __forceinline__ void emit_adj(const Rec& r, const float* dl, Adj& d) {
    float di[12];   // rows 0..2 of dL/dinstance, three 16-byte global loads
    // (the pointer comes from a table, so without the address space the
    // loads would be flat loads, which also hold up the next LDS wait)
    typedef float vf4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(1))) const vf4 gcf4;
    const gcf4* d4 = (const gcf4*)dl;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const vf4 v = d4[i];
        di[i * 4] = v.x; di[i * 4 + 1] = v.y; di[i * 4 + 2] = v.z; di[i * 4 + 3] = v.w;
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            d.m[i * 4 + j] += di[i * 4 + j] * r.s[j];
            d.s[j] += di[i * 4 + j] * r.m[i * 4 + j];
        }
        d.m[i * 4 + 3] += di[i * 4 + 3];
    }
}

// Reverse of one single-child operator applied to the state `r` (before
// the operator): d holds the adjoint after it and is turned into the
// adjoint before it.
__device__ __forceinline__ void single_adj(const Ctx& c, const AdjArgs& g, GradAcc& ga, const EntryV& e, const Rec& r,
                                           Adj& d) {
    const uint32_t k = e.kind();
    if (k == K_IFSIZELESS || k == K_IF || k == K_RANDOM) return;
    float v0, v1, v2;
    eval3(c, e, r, v0, v1, v2);
    if (k == K_TRANSLATE) {
        const float t[3] = {v0, v1, v2};
        float dm[12], dt[3];
        translate_adj(r.m, t, d.m, dm, dt);
#pragma unroll
        for (int i = 0; i < 12; ++i) d.m[i] = dm[i];
        grad_param(c, g, ga, e, 0, r.axiom, dt[0]);
        grad_param(c, g, ga, e, 1, r.axiom, dt[1]);
        grad_param(c, g, ga, e, 2, r.axiom, dt[2]);
        return;
    }
    if (k == K_ROTATE) {                       // m' = m * R(alpha, beta, gamma)
        const float kd = 3.1415926535897932384626434f / 180.0f;
        float sa, sb, sg, ca, cb, cg;
        sincos_f32(v0 * kd, &sa, &ca);
        sincos_f32(v1 * kd, &sb, &cb);
        sincos_f32(v2 * kd, &sg, &cg);
        const float R[16] = {cb * cg, cg * sa * sb - ca * sg, ca * cg * sb + sa * sg, 0.0f,
                             cb * sg, ca * cg + sa * sb * sg, -cg * sa + ca * sb * sg, 0.0f,
                             -sb, cb * sa, ca * cb, 0.0f,
                             0.0f, 0.0f, 0.0f, 1.0f};
        // dR[k][j] = sum_i m[i][k] dm'[i][j] (3x3 part)
        float dR[9];
#pragma unroll
        for (int kk = 0; kk < 3; ++kk)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                float s = 0.0f;
#pragma unroll
                for (int i = 0; i < 3; ++i) s += r.m[i * 4 + kk] * d.m[i * 4 + j];
                dR[kk * 3 + j] = s;
            }
        const float Ra[9] = {0.0f, cg * ca * sb + sa * sg, -sa * cg * sb + ca * sg,
                             0.0f, -sa * cg + ca * sb * sg, -cg * ca - sa * sb * sg,
                             0.0f, cb * ca, -sa * cb};
        const float Rb[9] = {-sb * cg, cg * sa * cb, ca * cg * cb,
                             -sb * sg, sa * cb * sg, ca * cb * sg,
                             -cb, -sb * sa, -ca * sb};
        const float Rg[9] = {-cb * sg, -sg * sa * sb - ca * cg, -ca * sg * sb + sa * cg,
                             cb * cg, -ca * sg + sa * sb * cg, sg * sa + ca * sb * cg,
                             0.0f, 0.0f, 0.0f};
        float dal = 0.0f, dbe = 0.0f, dgm = 0.0f;   // dL/d(alpha, beta, gamma) in radians
#pragma unroll
        for (int q = 0; q < 9; ++q) { dal += dR[q] * Ra[q]; dbe += dR[q] * Rb[q]; dgm += dR[q] * Rg[q]; }
        float dm[12];
        mul_adj_a(R, d.m, dm);
#pragma unroll
        for (int i = 0; i < 12; ++i) d.m[i] = dm[i];
        grad_param(c, g, ga, e, 0, r.axiom, dal * kd);
        grad_param(c, g, ga, e, 1, r.axiom, dbe * kd);
        grad_param(c, g, ga, e, 2, r.axiom, dgm * kd);
        return;
    }
    if (k == K_SCALE) {                        // s'_i = v_i > 0 ? v_i : (v_i < 0 ? -s_i v_i : 0)
        const float v[3] = {v0, v1, v2};
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const float ds = d.s[i];
            if (v[i] < 0.0f) {
                d.s[i] = ds * -v[i];
                grad_param(c, g, ga, e, (uint32_t)i, r.axiom, ds * -r.s[i]);
            } else {
                d.s[i] = 0.0f;
                if (v[i] > 0.0f) grad_param(c, g, ga, e, (uint32_t)i, r.axiom, ds);
            }
        }
        return;
    }
    if (k == K_SWAPSIZE) {                     // s'_k = s[a_k]
        const uint32_t a0 = min(f2u_rd(v0), 2u), a1 = min(f2u_rd(v1), 2u), a2 = min(f2u_rd(v2), 2u);
        const float d0 = d.s[0], d1 = d.s[1], d2 = d.s[2];
        // d.s[a_k] += d_k in k order, written with selects (no indexed local)
#pragma unroll
        for (uint32_t q = 0; q < 3; ++q) {
            float x = 0.0f;
            x = a0 == q ? x + d0 : x;
            x = a1 == q ? x + d1 : x;
            x = a2 == q ? x + d2 : x;
            d.s[q] = x;
        }
        return;
    }
    // K_EXTRUDE: m' = m * B, s' = (s0, v1, s1)
    const float B[16] = {1.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, -1.0f, 0.0f,
                         0.0f, 1.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 1.0f};
    float dm[12];
    mul_adj_a(B, d.m, dm);
#pragma unroll
    for (int i = 0; i < 12; ++i) d.m[i] = dm[i];
    const float ds0 = d.s[0], ds1 = d.s[1], ds2 = d.s[2];
    d.s[0] = ds0;
    d.s[1] = ds2;
    d.s[2] = 0.0f;
    grad_param(c, g, ga, e, 1, r.axiom, ds1);
}

// Reverse of build_child: the child state adjoint dc becomes the parent
// state adjoint dp and the adjoints of the child's offset and size.
__device__ __forceinline__ void build_adj(const Rec& p, const EntryV& pe, uint32_t j, uint32_t axis, float o,
                                          const Adj& dc, Adj& dp, float& d_o, float& d_ns) {
    adj_zero(dp);
    d_o = 0.0f;
    d_ns = 0.0f;
    const uint32_t kind = pe.kind();
    if (kind == K_SUBDIV || kind == K_REPEAT) {
        float t[3];
        axis_vec(axis, o, t[0], t[1], t[2]);
        float dt[3];
        translate_adj(p.m, t, dc.m, dp.m, dt);
        // selects, not indexing by `axis`: an indexed local lives in scratch
        d_o = axis == 0u ? dt[0] : (axis == 1u ? dt[1] : dt[2]);
#pragma unroll
        for (uint32_t q = 0; q < 3; ++q) dp.s[q] = q == axis ? 0.0f : dc.s[q];
        d_ns = axis == 0u ? dc.s[0] : (axis == 1u ? dc.s[1] : dc.s[2]);
        return;
    }
    if (kind == K_COMPSPLIT) {                 // m_c = (m * translate(t_j)) * B_j
        const float hx = p.s[0] * 0.5f, hy = p.s[1] * 0.5f, hz = p.s[2] * 0.5f;
        float t[3] = {0.0f, 0.0f, 0.0f};
        float b00 = 1.0f, b02 = 0.0f, b06 = 0.0f, b09 = 0.0f, b08 = 0.0f, b10 = 1.0f, b05 = 1.0f;
        bool rotate = true;
        if (j == 0) { t[2] = -hz; b00 = -1.0f; b10 = -1.0f; }
        else if (j == 1) { t[2] = hz; rotate = false; }
        else if (j == 2) { t[0] = -hx; b00 = 0.0f; b02 = -1.0f; b08 = 1.0f; b10 = 0.0f; }
        else if (j == 3) { t[0] = hx; b00 = 0.0f; b02 = 1.0f; b08 = -1.0f; b10 = 0.0f; }
        else if (j == 4) { t[1] = -hy; b05 = 0.0f; b06 = -1.0f; b09 = 1.0f; b10 = 0.0f; }
        else { t[1] = hy; b05 = 0.0f; b06 = 1.0f; b09 = -1.0f; b10 = 0.0f; }
        float dtmp[12];
        if (rotate) {
            const float B[16] = {b00, 0.0f, b02, 0.0f, 0.0f, b05, b06, 0.0f,
                                 b08, b09, b10, 0.0f, 0.0f, 0.0f, 0.0f, 1.0f};
            mul_adj_a(B, dc.m, dtmp);
        } else {
#pragma unroll
            for (int i = 0; i < 12; ++i) dtmp[i] = dc.m[i];
        }
        float dt[3];
        translate_adj(p.m, t, dtmp, dp.m, dt);
        const float sgn = (j == 0 || j == 2 || j == 4) ? -0.5f : 0.5f;
        // (selects: an array indexed at run time lives in scratch)
        const float dta = sgn * (j < 2 ? dt[2] : (j < 4 ? dt[0] : dt[1]));
        dp.s[0] += j >= 2 && j < 4 ? dta : 0.0f;
        dp.s[1] += j >= 4 ? dta : 0.0f;
        dp.s[2] += j < 2 ? dta : 0.0f;
        // sizes: s_c = ((j == 2 || j == 3) ? sz : sx, j < 4 ? sy : sz, 1)
        dp.s[2] += j == 2 || j == 3 ? dc.s[0] : 0.0f;
        dp.s[0] += j == 2 || j == 3 ? 0.0f : dc.s[0];
        dp.s[1] += j < 4 ? dc.s[1] : 0.0f;
        dp.s[2] += j < 4 ? 0.0f : dc.s[1];
        return;
    }
    // K_REPLICATE: a copy
    dp = dc;
}

__device__ __forceinline__ const float4* slot_at(const AdjArgs& g, uint32_t child) {
    return g.slots + (size_t)child * (kSlotFloats / 4u);
}

// Reverse of a fan-out at state `r` (entry e), whose children's slots start
// at child index `first` of the next level.
__device__ __forceinline__ void fan_adj(const Ctx& c, const AdjArgs& g, GradAcc& ga, const EntryV& e, const Rec& r, uint32_t first,
                                        uint32_t nd, bool self, Adj& d) {
    const uint32_t kind = e.kind();
    const bool split = !self && (kind == K_SUBDIV || kind == K_REPEAT);
    Fan f;
    f.n = 0;
    f.axis = 3u;
    if (split) fan_init(c, r, e, f);
    // parent-state adjoints the children left (four 16-byte loads per slot),
    // and the sum of their offset adjoints in child order
    float total_o = 0.0f;
#pragma unroll 2                       // two children's loads in flight: 434 -> 417 us (see k_adjoint)
    for (uint32_t q = 0; q < nd; ++q) {
        const float4* sl = slot_at(g, first + q);
        float4 a = sl[0], b = sl[1], cc = sl[2], dd = sl[3];
        dd.x = f.axis == 0u ? 0.0f : dd.x;       // the child's size adjoint, below
        dd.y = f.axis == 1u ? 0.0f : dd.y;
        dd.z = f.axis == 2u ? 0.0f : dd.z;
        d.m[0] += a.x; d.m[1] += a.y; d.m[2] += a.z; d.m[3] += a.w;
        d.m[4] += b.x; d.m[5] += b.y; d.m[6] += b.z; d.m[7] += b.w;
        d.m[8] += cc.x; d.m[9] += cc.y; d.m[10] += cc.z; d.m[11] += cc.w;
        d.s[0] += dd.x; d.s[1] += dd.y; d.s[2] += dd.z;
        total_o += dd.w;
    }
    if (!split || f.n == 0u) return;
    uint32_t skipm = c.prog.entries[e.idx].aux[0];
    if (kind == K_REPEAT) skipm = (skipm & 1u) ? 0xFFFFFFFFu : 0u;
    // o_j = off_j + ns_j / 2, off_{j+1} = off_j + ns_j, off_0 = -total / 2:
    //   dL/doff_0 = sum_j do_j, dL/dns_j = dns_j + do_j / 2 + sum_{k > j} do_k
    float prefix = 0.0f, d_r2a = 0.0f, d_e1 = 0.0f, d_e2 = 0.0f, d_e3 = 0.0f;
    uint32_t q = 0;
    Fan ff = f;
    for (uint32_t j = 0; j < f.n; ++j) {
        float o, ns, fac = 0.0f;
        const bool keep = fan_geom(c, r, e, ff, j, o, ns, &fac);
        const bool skip = j < 32u ? ((skipm >> j) & 1u) != 0u : skipm == 0xFFFFFFFFu;
        float d_oj = 0.0f, d_nsj = 0.0f;
        if (!skip) {
            if (q < nd) {
                const float4 dd = slot_at(g, first + q)[3];
                d_oj = dd.w;
                d_nsj = f.axis == 0u ? dd.x : (f.axis == 1u ? dd.y : dd.z);
            }
            ++q;
        }
        if (!keep) continue;
        prefix += d_oj;
        const float dn = d_nsj + 0.5f * d_oj + (total_o - prefix);
        if (kind == K_SUBDIV) {
            if (fac > 0.0f) {
                grad_param(c, g, ga, e, j + 1u, r.axiom, dn);
            } else if (fac < 0.0f) {
                d_r2a += dn * -fac;
                grad_param(c, g, ga, e, j + 1u, r.axiom, dn * -f.r2a);
            }
        } else {
            if (j == 0u) d_e1 += dn;
            else if (j + 1u < f.reps) d_e2 += dn;
            else d_e3 += dn;
        }
    }
    float d_total = -0.5f * total_o;
    if (kind == K_SUBDIV) {
        // r2a = (total - sum of absolute factors) / (sum of |relative factors|)
        float abs_sum = 0.0f, rel_sum = 0.0f;
        const uint32_t ax = r.axiom, pa = r.path, de = rec_depth(c, r);
        for (uint32_t i = 1; i < e.nparams(); ++i) {
            const float fac = P(c, e, i, r, ax, pa, de);
            abs_sum += (float)(fac > 0.0f) * fac;
            rel_sum += (float)(fac < 0.0f) * (fac * -1.0f);
        }
        if (rel_sum != 0.0f && d_r2a != 0.0f) {
            d_total += d_r2a / rel_sum;
            const float d_abs = -d_r2a / rel_sum, d_rel = -d_r2a * f.r2a / rel_sum;
            for (uint32_t i = 1; i < e.nparams(); ++i) {
                const float fac = P(c, e, i, r, ax, pa, de);
                if (fac > 0.0f) grad_param(c, g, ga, e, i, r.axiom, d_abs);
                else if (fac < 0.0f) grad_param(c, g, ga, e, i, r.axiom, -d_rel);
            }
        }
    } else {
        // Repeat pieces from (size, extent), the repetition count frozen
        float v0, ex, v2;
        eval3(c, e, r, v0, ex, v2);
        const uint32_t mode = f2u_rd(v2);
        const float sz = f.total;
        const float extent = (((float)(ex < 0.0f) * sz) * fabsf(ex)) + ((float)(ex > 0.0f) * ex);
        float d_sz = 0.0f, d_ext = 0.0f;
        if (mode == PGA_ADJUST_TO_FILL) {
            if (f.reps > 0u) d_sz += (d_e1 + d_e2 + d_e3) / (float)f.reps;
        } else {
            // the remainder piece rest = fmod(sz, extent) (extent when exact)
            // is the first piece (ANCHOR_TO_START) or the last (ANCHOR_TO_END)
            const bool start = mode == PGA_ANCHOR_TO_START;
            const float d_rest = start ? d_e1 : d_e3;
            d_ext += start ? (d_e2 + d_e3) : (d_e1 + d_e2);
            const float rest = fmodf(sz, extent);
            if (rest == 0.0f) {
                d_ext += d_rest;
            } else {
                d_sz += d_rest;
                d_ext += d_rest * -truncf(sz / extent);
            }
        }
        if (ex > 0.0f) {
            grad_param(c, g, ga, e, 1, r.axiom, d_ext);
        } else if (ex < 0.0f) {
            d_sz += d_ext * -ex;
            grad_param(c, g, ga, e, 1, r.axiom, d_ext * -sz);
        }
        d_total += d_sz;
    }
#pragma unroll
    for (uint32_t q = 0; q < 3; ++q) d.s[q] = q == f.axis ? d.s[q] + d_total : d.s[q];
}

// The program image and the tables a child looks up by terminal, in LDS: read
// from global memory, every operator of every chain waited for its entry.
struct AdjLDS {
    unsigned long long cap[PGA_MAX_TERMINALS];
    const float* dl[PGA_MAX_TERMINALS];
};
extern __shared__ __align__(16) unsigned char adj_smem[];

__device__ __forceinline__ void adj_stage(const KArgs& a, const AdjArgs& g, AdjLDS& T) {
    uint4* dst = reinterpret_cast<uint4*>(adj_smem);
    for (uint32_t i = threadIdx.x; i < a.image_bytes / 16u; i += blockDim.x) dst[i] = a.image[i];
    for (uint32_t i = threadIdx.x; i < PGA_MAX_TERMINALS; i += blockDim.x) {
        T.cap[i] = a.inst_cap[i];
        T.dl[i] = g.dl[i];
    }
    __syncthreads();
}

__device__ __forceinline__ Ctx adj_ctx(const KArgs& a, const AdjLDS& T) {
    Ctx c;
    c.prog.entries = reinterpret_cast<const DevEntry*>(adj_smem);
    c.prog.params = reinterpret_cast<const DevParam*>(adj_smem + a.off_params);
    c.prog.succ = reinterpret_cast<const int32_t*>(adj_smem + a.off_succ);
    c.prog.exp = reinterpret_cast<const uint32_t*>(adj_smem + a.off_exp);
    c.prog.term_slot = adj_smem + a.off_slots;
    c.prog.slot_term = adj_smem + a.off_slots + PGA_MAX_TERMINALS;
    c.prog.nentries = a.prog.nentries;
    c.prog.nslots = a.prog.nslots;
    c.inst = nullptr;
    c.inst_cap = T.cap;
    c.aparams = a.aparams;
    c.aparams_per = a.aparams_per;
    c.naxioms_total = a.naxioms_total;
    c.key0 = a.key0;
    c.key1 = a.key1;
    c.term_counts = a.term_counts;
    c.par_out = nullptr;
    c.desc_out = nullptr;
    c.par_count = nullptr;
    c.desc_count = nullptr;
    c.par_cap = a.cap_par;
    c.desc_cap = a.cap_desc;
    c.err = a.err;
    c.max_chain = a.max_chain;
    c.geom = 1u;
    c.seed = a.use_seed;
    c.poly = 0u;             // the tape refuses dynamic polygons
    c.tape = 1u;
    c.ctxs = 0u;             // one-phase programs without Collider / IfCollides only
    c.dmask = 0xFFFFu;
    c.phase = 0u;
    c.wr = 0u;
    c.coll = nullptr;
    c.coll_count = nullptr;
    c.coll_visible = nullptr;
    c.coll_cap = 0u;
    c.bvh_wide = nullptr;
    c.bvh_keys = nullptr;
    c.coll_bits = nullptr;
    c.coll_bits_cap = 0u;
    return c;
}

__device__ __forceinline__ void load_rec(const Rec* src, Rec& r) {
    const float4* s = reinterpret_cast<const float4*>(src);
    const float4 a = s[0], b = s[1], c = s[2], d = s[3], e = s[4];
    r.m[0] = a.x; r.m[1] = a.y; r.m[2] = a.z; r.m[3] = a.w;
    r.m[4] = b.x; r.m[5] = b.y; r.m[6] = b.z; r.m[7] = b.w;
    r.m[8] = c.x; r.m[9] = c.y; r.m[10] = c.z; r.m[11] = c.w;
    r.s[0] = d.x; r.s[1] = d.y; r.s[2] = d.z; r.seed = d.w;
    r.custom = e.x; r.ed = __float_as_uint(e.y); r.axiom = __float_as_uint(e.z); r.path = __float_as_uint(e.w);
}

// A child's starting state: the axiom's record, or what its descriptor names.
struct ChildRef {
    uint4 dv;                           // descriptor (levels > 0)
    uint32_t i;                         // child of the level
};
__device__ __forceinline__ void child_parent(const KArgs& a, const AdjArgs& g, const ChildRef& ch, Rec& par) {
    load_rec(a.tape_par + g.par_in_base + ch.dv.x, par);
}
__device__ __forceinline__ void child_start(const KArgs& a, const AdjArgs& g, const Ctx& c, const ChildRef& ch,
                                            Rec& r) {
    if (g.level == 0u) {
        const pga_axiom& ax = a.axioms[a.first_axiom + ch.i];
#pragma unroll
        for (int k = 0; k < 12; ++k) r.m[k] = ax.model[k];
        r.s[0] = ax.size[0]; r.s[1] = ax.size[1]; r.s[2] = ax.size[2];
        r.seed = ax.seed;
        r.custom = ax.custom;
        r.axiom = a.first_axiom + ch.i;
        r.path = 0u;
        r.ed = (uint32_t)max(ax.entry_index, 0);
        return;
    }
    Rec par;
    child_parent(a, g, ch, par);
    const uint32_t j = ch.dv.y & 0x3FFFFFFFu;
    if (j == kDescSelf) { r = par; return; }
    build_child(c, par, load_entry(c, rec_entry(par)), j, ch.dv.y >> 30, __uint_as_float(ch.dv.z),
                __uint_as_float(ch.dv.w), r);
}

// One thread per child of the level. What bounds it is the latency of a chain
// of loads (outcome and descriptor, parent, its children's slots or its
// instance's gradient) at few waves per SIMD, so registers: a thread holds
// one record at a time and derives it again from the tape where it needs it
// later (the parent is in L2), instead of the parent, the starting state and
// the end of the chain side by side. Slots are 64 bytes and leave through LDS:
// stored lane by lane, the 312 MB of the last level's became 716 MB of writes
// (502 MB now, scratch included). The levels of
// 4,096 parameterised lots, last first: 372 / 661 / 295 / 67 us with 80-byte
// slots, the program read from memory and 48 bytes of scratch a lane; 299 /
// 559 / 227 / 52 us with that; 297 / 434 / 190 / 60 with the gradient sums in
// LDS too, and 285 / 389 / 187 / 62 with four waves per SIMD instead of three,
// which the registers that these sums took now allow (64 bytes of scratch a
// lane instead of 32: 256 lots, a third of a round of the grid, lose 3 of 125
// us by it), and the loads of two children's slots in flight.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_adjoint(KArgs a, AdjArgs g) {
    __shared__ AdjLDS T;
    __shared__ float4 stage[4][256];     // per wave: the gradient sums, then 64 slots on their way out
    adj_stage(a, g, T);
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const Ctx c = adj_ctx(a, T);
    const uint32_t gi = g.child_base + i;
    const bool here = i < g.n_children && gi < a.tape_out_cap && gi < g.slots_cap;
    uint4 out = make_uint4(T_DROP, 0u, 0u, 0u);
    ChildRef ch;
    ch.i = i;
    ch.dv = make_uint4(0u, kDescNone, 0u, 0u);
    if (here) {
        out = a.tape_out[gi];
        if (g.level != 0u) ch.dv = *reinterpret_cast<const uint4*>(a.tape_desc + g.desc_in_base + i);
    }
    const uint32_t jj = ch.dv.y & 0x3FFFFFFFu;
    const bool none = g.level != 0u && (out.x == T_DROP || ch.dv.x >= a.cap_par || jj == kDescNone);
    const uint32_t kind = none || !here ? (uint32_t)T_DROP : out.x & 0xFFu;
    const bool self_copy = g.level != 0u && jj == kDescSelf;
    Adj d;
    adj_zero(d);
    GradAcc ga;
    grad_zero(ga, (lds_f64*)stage[threadIdx.x >> 6]);
    if (kind != T_DROP) {
        // replay the chain of single-child operators to its end
        uint32_t steps = 0;
        {
            Rec r;
            child_start(a, g, c, ch, r);
            for (; steps < c.max_chain; ++steps) {
                const EntryV e = load_entry(c, rec_entry(r));
                if (!(e.kind() != K_GENERATE && e.kind() != K_DISCARD && !is_fanout(e.kind()))) break;
                uint32_t ord;
                const int32_t next = apply_single(c, e, r, &ord);
                if (!advance(c, r, next, ord)) break;
            }
            // the adjoint of the chain's end
            if (kind == T_TERM) {
                const uint32_t slot = (out.x >> 8) & 0xFFu;
                const uint32_t t = slot < c.prog.nslots ? c.prog.slot_term[slot] : PGA_MAX_TERMINALS;
                if (t < PGA_MAX_TERMINALS && T.dl[t] != nullptr && (unsigned long long)out.y < T.cap[t])
                    emit_adj(r, T.dl[t] + (size_t)out.y * 16u, d);
            } else {   // T_FAN / T_SELF: the children of the fan-out are in the next level
                const uint32_t first = g.next_child_base + out.z;
                const uint32_t nd = first <= g.slots_cap && out.w <= g.slots_cap - first ? out.w : 0u;
                fan_adj(c, g, ga, load_entry(c, rec_entry(r)), r, first, nd, kind == T_SELF, d);
            }
        }
        // back through the chain, recomputing each operator's input state
        for (uint32_t t = steps; t-- > 0;) {
            Rec q;
            child_start(a, g, c, ch, q);
            for (uint32_t u = 0; u < t; ++u) {
                const EntryV e = load_entry(c, rec_entry(q));
                uint32_t ord;
                const int32_t next = apply_single(c, e, q, &ord);
                advance(c, q, next, ord);
            }
            single_adj(c, g, ga, load_entry(c, rec_entry(q)), q, d);
        }
    }
    flush_grads(c, g, ga);
    if (g.level == 0u) return;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");      // the sums are read: the words are the slots'
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    Adj dp;
    float d_o = 0.0f, d_ns = 0.0f;
    const uint32_t axis = ch.dv.y >> 30;
    uint32_t pk = 0xFFu;
    if (kind == T_DROP) {
        adj_zero(dp);
    } else if (self_copy) {
        dp = d;
    } else {
        Rec par;
        child_parent(a, g, ch, par);
        const EntryV pe = load_entry(c, rec_entry(par));
        pk = pe.kind();
        build_adj(par, pe, ch.dv.y & 0x3FFFFFFFu, axis, __uint_as_float(ch.dv.z), d, dp, d_o, d_ns);
    }
    if (pk == K_SUBDIV || pk == K_REPEAT) {       // build_adj left 0 there
        dp.s[0] = axis == 0u ? d_ns : dp.s[0];
        dp.s[1] = axis == 1u ? d_ns : dp.s[1];
        dp.s[2] = axis == 2u ? d_ns : dp.s[2];
    }
    // the wave's slots are consecutive: through LDS (record r's words rotated
    // by r / 4 against bank conflicts) into whole lines
    float4* S = stage[threadIdx.x >> 6];
    const uint32_t lane = threadIdx.x & 63u;
    auto at = [](uint32_t r, uint32_t k) { return r * 4u + ((k + (r >> 2)) & 3u); };
    S[at(lane, 0u)] = make_float4(dp.m[0], dp.m[1], dp.m[2], dp.m[3]);
    S[at(lane, 1u)] = make_float4(dp.m[4], dp.m[5], dp.m[6], dp.m[7]);
    S[at(lane, 2u)] = make_float4(dp.m[8], dp.m[9], dp.m[10], dp.m[11]);
    S[at(lane, 3u)] = make_float4(dp.s[0], dp.s[1], dp.s[2], d_o);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t n = (uint32_t)__popcll(__ballot(here));    // the lanes of `here` come first
    float4* dst = g.slots + (size_t)(gi - lane) * (kSlotFloats / 4u);
#pragma unroll
    for (uint32_t u = 0; u < 4u; ++u) {
        const uint32_t q = lane + 64u * u;
        if (q < n * 4u) dst[q] = S[at(q >> 2, q & 3u)];
    }
}

} // namespace pga

namespace pga {
__global__ void __launch_bounds__(256) k_grad_out(const double* acc, float* out, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (float)acc[i];
}
} // namespace pga

hipError_t pga_launch_grad_out(const double* acc, float* out, uint32_t n, hipStream_t s) {
    if (n == 0u) return hipSuccess;
    hipLaunchKernelGGL(pga::k_grad_out, dim3((n + 255u) / 256u), dim3(256), 0, s, acc, out, n);
    return hipGetLastError();
}

hipError_t pga_launch_adjoint(const pga::KArgs& a, const pga::AdjArgs& g, hipStream_t s) {
    if (g.n_children == 0u) return hipSuccess;
    hipLaunchKernelGGL(pga::k_adjoint, dim3((g.n_children + 255u) / 256u), dim3(256), a.image_bytes, s, a, g);
    return hipGetLastError();
}
