/*
 * tracer_dev.h -- device code shared by the Whitted kernels (gfx950).
 *
 * QuadRay's per-ray path restated for one work-item per ray: the surface
 * list walk with transform caching, quadric / plane / two-plane roots,
 * axis and custom clippers, normals, texturing, lighting with hard shadows,
 * and the refraction / reflection set-up with Fresnel.  Arithmetic is fp32
 * in QuadRay's operation order: compiled with -ffp-contract=off and correctly
 * rounded division and square root, 1/sqrt(x) as an IEEE sqrt followed by an
 * IEEE divide, as in QuadRay's full-precision builds
 * (core/config/rtconf.h:166-211).
 *
 * Scene tables are read through the constant address space, so a read at a
 * wave-uniform index (the list walk, clip lists, lights) is a scalar load
 * into SGPRs and never occupies VGPRs or LDS.
 */
#ifndef QR_TRACER_DEV_H
#define QR_TRACER_DEV_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qr_soa.h"
#include "tracer_kernels.h"

namespace {

constexpr uint32_t SIGN = 0x80000000u;
constexpr int FLAG_PASS = 2;
constexpr int FLAG_SHAD = 4;
constexpr int MAX_STACK = 16;

struct V3 { float x, y, z; };

__device__ __forceinline__ float bitsf(uint32_t u) { return __uint_as_float(u); }
__device__ __forceinline__ uint32_t fbits(float f) { return __float_as_uint(f); }
__device__ __forceinline__ float fxor(float v, uint32_t m) { return bitsf(fbits(v) ^ m); }
__device__ __forceinline__ float negif(float v, int n) { return n ? -v : v; }

/* wave masks: one bit per active lane where b holds, and back */
__device__ __forceinline__ uint64_t lanes(bool b)
{
    return __builtin_amdgcn_ballot_w64(b);
}
__device__ __forceinline__ bool in_lane(uint64_t m)
{
    return __builtin_amdgcn_inverse_ballot_w64(m);
}

/* the correctly rounded square root of x in [2^-96, inf], and of 0 (sqrtf's own
 * steps without those for smaller values): the hardware root, corrected by
 * the signs of the residuals of its neighbours */
__device__ __forceinline__ float sqrt_mid(float x)
{
    const float s = __builtin_amdgcn_sqrtf(x);
    const float lo = bitsf(fbits(s) - 1u), hi = bitsf(fbits(s) + 1u);
    float q = __builtin_fmaf(-lo, s, x) <= 0.0f ? lo : s;
    q = __builtin_fmaf(-hi, s, x) > 0.0f ? hi : q;
    return q;
}
constexpr float SQRT_MID_MIN = 1.2621774483536189e-29f;     /* 2^-96 */

/* does every active lane hold a value in [2^-96, FLT_MAX] */
__device__ __forceinline__ bool all_mid(float x)
{
    return lanes(fbits(x) - fbits(SQRT_MID_MIN) > 0x7f7fffffu - fbits(SQRT_MID_MIN)) == 0;
}

/* sqrtf(x) and 1.0f / sqrtf(x), both roundings as they are: the short forms
 * where the whole wave's values are in sqrt_mid's range (nearly always).
 * There the root is in [2^-48, 2^64), and the hardware reciprocal with one
 * Newton step is the correctly rounded reciprocal (tests/test_gpu_math.py
 * compares every float).  12 VALU instructions and the test
 * instead of 27. */
__device__ __forceinline__ float root(float x)
{
    return all_mid(x) ? sqrt_mid(x) : sqrtf(x);
}
__device__ __forceinline__ float rsq(float x)
{
    if (all_mid(x))
    {
        const float s = sqrt_mid(x);
        const float y = __builtin_amdgcn_rcpf(s);
        return __builtin_fmaf(__builtin_fmaf(-s, y, 1.0f), y, y);
    }
    return 1.0f / sqrtf(x);
}
/* c / 255.0f for whole c in 0..255, correctly rounded: the quotient by the
 * reciprocal, corrected by its residual (equal for all 256) */
__device__ __forceinline__ float unorm8(uint32_t c)
{
    const float v = (float)c, y = 1.0f / 255.0f;
    const float q = v * y;
    return __builtin_fmaf(__builtin_fmaf(-255.0f, q, v), y, q);
}

/* Component access at a run-time index.  pick() selects values, not
 * references: a branch between two fields is merged by the optimiser into
 * one access at a computed address, which gives the walk registers an
 * address and moves them to scratch memory. */
__device__ __forceinline__ float sel(const V3 &v, int i)
{
    return i == 0 ? v.x : (i == 1 ? v.y : v.z);
}
__device__ __forceinline__ V3 pick(bool c, V3 a, V3 b)
{
    return V3{c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z};
}
__device__ __forceinline__ void put(V3 &v, int i, float f)
{
    if (i == 0) v.x = f; else if (i == 1) v.y = f; else v.z = f;
}
/* x86 float->int conversion semantics: out of range and NaN give INT_MIN */
__device__ __forceinline__ int32_t cvt_floor(float x)
{
    float f = floorf(x);
    return (f >= -2147483648.0f && f < 2147483648.0f) ? (int32_t)f : (int32_t)SIGN;
}
__device__ __forceinline__ int32_t cvt_rne(float x)
{
    float f = rintf(x);
    return (f >= -2147483648.0f && f < 2147483648.0f) ? (int32_t)f : (int32_t)SIGN;
}

/* Scene tables are read through the constant address space: a read at a
 * wave-uniform index (list walk, clip lists, lights) becomes a scalar load
 * into SGPRs, a read at a per-lane index a vector load. */
#define QC __attribute__((address_space(4)))

struct Scene
{
    const QC qr_surface  *srf;
    const QC qr_dev_surf *hot;          /* the surfaces as the walks read them */
    const QC qr_material *mat;
    const QC qr_light    *lgt;
    const QC qr_clip     *clp;
    const QC qr_elem     *elem;
    const QC uint32_t    *texel;
    const QC qr_dev_step *step;         /* nearest-hit program (ends in an end step) */
    const QC qr_dev_step *step_any;     /* any-hit program (ends in an end step) */
    int n_elem, n_lgt;
    float ref_x, ref_y, ref_z;          /* reference point of the world boxes */
};

/* kernel view of the device tables */
inline Scene scene_of(const qr_device_tables *t)
{
    Scene sc;
    sc.srf = (const QC qr_surface *)t->surfaces;
    sc.hot = (const QC qr_dev_surf *)t->hot;
    sc.mat = (const QC qr_material *)t->materials;
    sc.lgt = (const QC qr_light *)t->lights;
    sc.clp = (const QC qr_clip *)t->clips;
    sc.elem = (const QC qr_elem *)t->elems;
    sc.texel = (const QC uint32_t *)t->texels;
    sc.step = (const QC qr_dev_step *)t->steps;
    sc.step_any = (const QC qr_dev_step *)t->steps_any;
    sc.n_elem = t->n_elem;
    sc.n_lgt = t->n_lgt;
    sc.ref_x = t->cull_ref[0];
    sc.ref_y = t->cull_ref[1];
    sc.ref_z = t->cull_ref[2];
    return sc;
}

struct Ray
{
    V3    org, dir;
    float t_min, t_max;
    int   flags;        /* side | pass (| shadow) of the originating hit */
    int   origin;       /* originating surface record or -1 */
    V3    oloc;         /* origin's local hit */
    int   depth;
};

struct Hit
{
    int   srf, side;
    float t;
    V3    hit, loc;
    float u, v;
};

template <class P>
__device__ __forceinline__ V3 sub3(const V3 &a, P p)
{
    return V3{a.x - p[0], a.y - p[1], a.z - p[2]};
}

/* inverse-matrix product, diagonal first (tracer.cpp:2536-2568); td its
 * diagonal, to the rest */
__device__ __forceinline__ V3 xform_full(const float td[3], const float to[6], const V3 &d)
{
    V3 o;
    o.x = td[0] * d.x;
    o.y = td[1] * d.y;
    o.z = td[2] * d.z;
    o.x = o.x + to[0] * d.y;
    o.x = o.x + to[1] * d.z;
    o.y = o.y + to[2] * d.x;
    o.y = o.y + to[3] * d.z;
    o.z = o.z + to[4] * d.x;
    o.z = o.z + to[5] * d.y;
    return o;
}

__device__ __forceinline__ V3 xform_diag(const float td[3], const V3 &d)
{
    return V3{td[0] * d.x, td[1] * d.y, td[2] * d.z};
}

/* the first 64 bytes of a qr_dev_surf, and the rest of its transform */
struct SurfHead
{
    float    pos[3];
    uint32_t flags;
    float    sci[4];
    float    scj[3];
    float    d_eps, t_eps;
    float    td[3];
};
static_assert(sizeof(SurfHead) == 64, "one scalar load");
struct SurfOff
{
    float to[6];
};
struct SurfClip
{
    float cmin[3], cmax[3];
};

template <class T, class S>
__device__ __forceinline__ T ldk(const QC S *p)
{
    T v;
    __builtin_memcpy(&v, p, sizeof(T));
    return v;
}

/* the record at byte offset "off" of the table (wave-uniform: one scalar
 * load of 64 bytes) */
__device__ __forceinline__ const QC qr_dev_surf *surf_at(const Scene &sc, uint32_t off)
{
    return (const QC qr_dev_surf *)((const QC char *)sc.hot + off);
}

__device__ __forceinline__ V3 xform(const SurfHead &s, const QC qr_dev_surf *p, const V3 &d)
{
    if ((s.flags & QR_DS_TRM) == QR_DS_TRM_DIAG) return xform_diag(s.td, d);
    if ((s.flags & QR_DS_TRM) == 0 && p->info == QR_DI_TRM_DIAG) return xform_diag(s.td, d);
    return xform_full(s.td, ldk<SurfOff>(p->to).to, d);
}

__device__ __forceinline__ int amap(uint32_t flags, int a)
{
    return (int)((flags >> (QR_DS_AMAP_BIT + 2 * a)) & 3u);
}
__device__ __forceinline__ int asgn(uint32_t flags, int a)
{
    return (int)((flags >> (QR_DS_ASGN_BIT + a)) & 1u);
}
/* scaler of world-aligned axis m */
__device__ __forceinline__ float sci_at(const float sci[4], int m)
{
    return m == 0 ? sci[0] : (m == 1 ? sci[1] : sci[2]);
}

/* clipper evaluation (PL_clp 5696, QD_clp 6292, TP_clp 6466) */
__device__ __forceinline__ bool clip_keep(const SurfHead &c, const V3 &nx, const V3 &ni, int rel)
{
    const uint32_t kind = (c.flags >> QR_DS_CLP_BIT) & 3u;
    const V3 p = pick((c.flags & QR_DS_SHIFT) != 0, ni, nx);
    float f;
    if (kind == 1)
    {
        f = negif(sel(p, amap(c.flags, 2)), asgn(c.flags, 2));
    }
    else
    {
        float d0 = (p.x * p.x) * c.sci[0];
        float d1 = (p.y * p.y) * c.sci[1];
        float d2 = (p.z * p.z) * c.sci[2];
        if (kind == 2)
        {
            d0 = d0 - (c.scj[0] + c.scj[0]) * p.x;
            d1 = d1 - (c.scj[1] + c.scj[1]) * p.y;
            d2 = d2 - (c.scj[2] + c.scj[2]) * p.z;
        }
        f = d0 - c.sci[3];
        f = f + d1;
        f = f + d2;
    }
    return rel < 0 ? (f >= 0.0f) : (f <= 0.0f);
}

/* apex snap of a local hit near a cone's or two planes' apex (tracer.cpp
 * 2773-2944), for a root with a near-zero discriminant; dd: the ray's
 * origin in the surface's tracing frame */
__device__ __forceinline__ void apex_snap(uint32_t flags, const float sci[4], float t_eps,
                                          const V3 &dd, int side, uint32_t amask, V3 &loc)
{
    const int ai = amap(flags, 0), aj = amap(flags, 1), ak = amap(flags, 2);
    const bool two = (flags & QR_DS_APEX_TWO) != 0;
    float li = sel(loc, ai);
    float rr = li * li;
    if (!two)
    {
        float lj = sel(loc, aj);
        rr = rr + lj * lj;
    }
    float lk = sel(loc, ak);
    rr = rr + lk * lk;
    if (rr < t_eps)
    {
        float ci = bitsf((fbits(sel(dd, ai)) & SIGN) ^ fbits(1.0f));
        float cj = 0.0f;
        float sk = sci_at(sci, ai);
        float lr = 1.0f;
        if (!two)
        {
            cj = bitsf((fbits(sel(dd, aj)) & SIGN) ^ fbits(1.0f));
            sk = sk + sci_at(sci, aj);
            lr = lr + 1.0f;
        }
        sk = sk / sci_at(sci, ak);
        sk = fxor(sk, SIGN);
        float ck = sqrtf(sk);
        float lc2 = sk + lr;
        float inv = rsq(lc2);
        inv = inv * t_eps;
        ci = ci * inv;
        cj = cj * inv;
        ck = ck * inv;
        uint32_t ts = side ? SIGN : 0u;
        ck = fxor(ck, fbits(sel(dd, ak)) & SIGN);
        ck = fxor(ck, (ts & amask) ^ amask);
        uint32_t tsg = (ts | amask) ^ amask;
        ci = fxor(ci, tsg);
        cj = fxor(cj, tsg);
        put(loc, ai, ci);
        if (!two) put(loc, aj, cj);
        put(loc, ak, ck);
    }
}

__device__ __forceinline__ V3 ray_at(const V3 &dir, const V3 &org, float t)
{
    return V3{dir.x * t + org.x, dir.y * t + org.y, dir.z * t + org.z};
}

/* axis and custom clipping of one root at distance t (CC_clp, tracer.cpp
 * 2686-3236) of the surface with record s at p, whose tracing frame has the
 * ray rr from dd; the lanes that keep it.
 *
 * QuadRay keeps two local-hit registers, NEW_X (world-aligned, from HIT) and
 * NEW_I (transformed, from RAY_I and DFF_I): a surface with a transform
 * (trm) refreshes NEW_I, one without refreshes NEW_X, and clipping reads
 * NEW_I when the surface is traced in its transform node's frame (shift),
 * NEW_X otherwise.  The engine only emits surfaces whose trm and shift
 * agree (a transformed surface always has a transform node, and a surface
 * under one always inherits its rotation), so the register read is always
 * the one refreshed for that root: one local hit. */
__device__ __forceinline__ uint64_t clip_root(const Scene &sc, const Ray &r, const SurfHead &s,
                                              uint32_t flags, const QC qr_dev_surf *p,
                                              const V3 &rr, const V3 &dd, float t, uint64_t side,
                                              uint64_t dmask, float a_val)
{
    V3 hit = V3{0.0f, 0.0f, 0.0f};
    if (!(flags & QR_DS_SHIFT) || (flags & QR_DS_CLIPS)) hit = ray_at(r.dir, r.org, t);
    V3 loc;
    if (flags & QR_DS_SHIFT) loc = ray_at(rr, dd, t);
    else loc = sub3(hit, s.pos);
    if ((flags & QR_DS_APEX) && dmask != 0)
    {
        if (in_lane(dmask))
        {
            apex_snap(flags, s.sci, s.t_eps, dd, in_lane(side) ? 1 : 0, fbits(a_val) & SIGN, loc);
        }
    }

    uint64_t ok = ~0ull;
    if (flags & QR_DS_AXIS_CLIP)
    {
        const SurfClip c = ldk<SurfClip>(p->cmin);
        if (flags & (1u << QR_DS_CMIN_BIT)) ok &= lanes(c.cmin[0] <= loc.x);
        if (flags & (2u << QR_DS_CMIN_BIT)) ok &= lanes(c.cmin[1] <= loc.y);
        if (flags & (4u << QR_DS_CMIN_BIT)) ok &= lanes(c.cmin[2] <= loc.z);
        if (flags & (1u << QR_DS_CMAX_BIT)) ok &= lanes(c.cmax[0] >= loc.x);
        if (flags & (2u << QR_DS_CMAX_BIT)) ok &= lanes(c.cmax[1] >= loc.y);
        if (flags & (4u << QR_DS_CMAX_BIT)) ok &= lanes(c.cmax[2] >= loc.z);
    }
    if (flags & QR_DS_CLIPS)
    {
        const int beg = p->clip_beg, cnt = p->clip_cnt;
        uint64_t saved = 0;
        int cache = -1;
        V3 nx = {0, 0, 0}, ni = {0, 0, 0};
        for (int k = 0; k < cnt; k++)
        {
            const qr_clip e = ldk<qr_clip>(&sc.clp[beg + k]);
            if (e.kind == QR_CLIP_ENTER) { saved = ok; ok = ~0ull; continue; }
            if (e.kind == QR_CLIP_LEAVE) { ok = ~ok & saved; continue; }
            const QC qr_dev_surf *cp = &sc.hot[e.surf];
            const SurfHead c = ldk<SurfHead>(cp);
            if (e.kind == QR_CLIP_TRNODE)
            {
                if (e.surf == p->trnode)
                {
                    nx.x = loc.x + s.pos[0];
                    nx.y = loc.y + s.pos[1];
                    nx.z = loc.z + s.pos[2];
                }
                else
                {
                    nx = xform(c, cp, sub3(hit, c.pos));
                }
                cache = e.rel;
                continue;
            }
            if (cache >= 0)
            {
                ni = sub3(nx, c.pos);
                if (k == cache) cache = -1;
            }
            else
            {
                nx = sub3(hit, c.pos);
                if (c.flags & QR_DS_TRM) ni = xform(c, cp, nx);
            }
            ok &= lanes(clip_keep(c, nx, ni, e.rel));
        }
    }
    return ok;
}

/* roots of a quadric or two-plane surface in the order they are tested:
 * n1 / d1, then n2 / d2, undefined where the denominator is 0 */
struct Roots
{
    float n1, d1, n2, d2;
};

/* coefficients of the root equation (QD_rt1 5722-5900, TP_rt1 6337-6390) of
 * the surface with flags, scalers sci and scj: rr, dd the ray's direction
 * and origin in its tracing frame; returns the discriminant */
__device__ __forceinline__ float quadric_abc(uint32_t flags, const float sci[4],
                                             const float scj[3], const V3 &rr, const V3 &dd,
                                             float &a_val, float &b_val, float &c_val)
{
    const uint32_t cls = flags & QR_DS_CLASS;
    if (cls != QR_DC_TWOPLANE)
    {
        V3 sr, sd, sc;
        if (cls == QR_DC_SPHERE)
        {
            sr = rr;
            sd = sc = dd;
        }
        else
        {
            sr = V3{sci[0] * rr.x, sci[1] * rr.y, sci[2] * rr.z};
            sd = sc = V3{sci[0] * dd.x, sci[1] * dd.y, sci[2] * dd.z};
            if (cls == QR_DC_QUADRIC)
            {
                sd = sub3(sd, scj);
                sc = sub3(sd, scj);
            }
        }
        a_val = rr.x * sr.x + rr.y * sr.y;
        b_val = rr.x * sd.x + rr.y * sd.y;
        c_val = dd.x * sc.x + dd.y * sc.y;
        a_val = a_val + rr.z * sr.z;
        b_val = b_val + rr.z * sd.z;
        c_val = c_val + dd.z * sc.z;
        c_val = c_val - sci[3];
        return b_val * b_val - c_val * a_val;
    }
    const int mi = amap(flags, 0), mk = amap(flags, 2);
    float ri = sel(rr, mi), di = sel(dd, mi);
    float rk = sel(rr, mk), dk = sel(dd, mk);
    float si_ = sci_at(sci, mi), sk_ = sci_at(sci, mk);
    float dx = di * rk - dk * ri;
    dx = dx * dx;
    dx = dx * si_;
    dx = dx * sk_;
    float bi = si_ * di, bk = sk_ * dk;
    bi = bi * ri;
    bk = bk * rk;
    b_val = bi + bk;
    float ci = di * di, ck = dk * dk;
    ci = ci * si_;
    ck = ck * sk_;
    c_val = ci + ck;
    float ai = ri * ri, ak = rk * rk;
    ai = ai * si_;
    ak = ak * sk_;
    a_val = ai + ak;
    return fabsf(dx);
}

/* roots from the coefficients and a discriminant >= 0, any of them
 * (QD_rt1 5900-6206, TP_rt1 6390-6413); side 1 (root 2) is tested first
 * where a < 0.  A near-zero discriminant's roots are formed here, as a
 * quotient by 1 (exact) or, where undefined, by 0. */
__device__ void roots_any(float a_val, float b_val, float c_val, float d_val, float d_eps,
                          float t_eps, Roots &q)
{
    float nb = -b_val;
    float sd = sqrtf(d_val);
    sd = fxor(sd, fbits(nb) & SIGN);
    float qq = nb + sd;
    const bool m_pos = 0.0f <= sd;
    const bool m_neg = 0.0f > sd;
    float n1 = m_neg ? qq : (m_pos ? c_val : 0.0f);
    float d1 = m_neg ? a_val : (m_pos ? qq : 0.0f);
    float n2 = m_neg ? c_val : (m_pos ? qq : 0.0f);
    float d2 = m_neg ? qq : (m_pos ? a_val : 0.0f);
    const uint32_t amask = fbits(a_val) & SIGN;
    if (d_val < d_eps)
    {
        if (n1 == 0.0f) d1 = 1.0f;
        if (n2 == 0.0f) d2 = 1.0f;
        float t1 = n1 / d1;
        float t2 = n2 / d2;
        const bool t1m = d1 != 0.0f, t2m = d2 != 0.0f;
        float tdf = t1 - t2;
        tdf = fxor(tdf, amask);
        bool fm = 0.0f <= tdf;
        if (!fm) tdf = 0.0f;
        float te = fm ? t_eps : 0.0f;
        te = te * t1;
        te = fabsf(te);
        tdf = tdf * -0.5f;
        tdf = tdf - te;
        tdf = fxor(tdf, amask);
        if (!(t1m && t2m)) tdf = 0.0f;
        n1 = t1 + tdf;
        n2 = t2 - tdf;
        d1 = t1m ? 1.0f : 0.0f;
        d2 = t2m ? 1.0f : 0.0f;
    }
    const bool second = 0.0f > a_val;
    q.n1 = second ? n2 : n1;
    q.d1 = second ? d2 : d1;
    q.n2 = second ? n1 : n2;
    q.d2 = second ? d1 : d2;
}

/* the same for a discriminant >= d_eps and in sqrt_mid's range: the signed
 * root of it is not 0, so root 1 is qq / a and root 2 c / qq where b > 0
 * (or +0), the other way round elsewhere */
__device__ __forceinline__ void roots_mid(float a_val, float b_val, float c_val, float d_val,
                                          uint64_t second, Roots &q)
{
    const float nb = -b_val;
    const float qq = nb + __builtin_copysignf(sqrt_mid(d_val), nb);
    const bool x = in_lane(lanes((int32_t)fbits(nb) < 0) ^ second);
    q.n1 = x ? qq : c_val;
    q.d1 = x ? a_val : qq;
    q.n2 = x ? c_val : qq;
    q.d2 = x ? qq : a_val;
}

/* the next float above t_lim; 0 for one below zero (a kept distance of a ray
 * whose t_min is), which turns away no root the limit allows */
template <bool T0>
__device__ __forceinline__ float above(float t_lim)
{
    const int32_t next = (int32_t)(fbits(t_lim) + 1u);
    return bitsf((uint32_t)(T0 || next > 0 ? next : 0));
}

/* the lanes whose n / d, rounded, may lie above t_min and at or below
 * t_lim, given the next float above t_lim; never without one that does.  With n'
 * = n times the sign of d and d' = |d|: rounding is monotonic and t_min a
 * float, so round(n/d) > t_min means n'/d' > t_min, n' > t_min * d' and, n'
 * being a float, n' >= round(t_min * d'); likewise above.  A zero or NaN
 * denominator's root is undefined, or rejected by the exact comparisons
 * that follow. */
template <bool T0>
__device__ __forceinline__ uint64_t roots_near(float n, float d, float t_min, float t_next)
{
    const float nn = fxor(n, fbits(d) & SIGN);
    const float lo = T0 ? 0.0f : t_min * fabsf(d);
    return lanes(nn >= lo) & lanes(nn <= t_next * fabsf(d));
}

/* reciprocal of a direction component for the slab tests: approximate, and
 * clamped to +-1e30 so that a zero component gives finite slab distances
 * (never 0 * inf) */
__device__ __forceinline__ float slab_rcp(float d)
{
    return fminf(fmaxf(__builtin_amdgcn_rcpf(d), -1e30f), 1e30f);
}

/* the step at byte offset "off" of a culling program (wave-uniform: one
 * 32-byte scalar load) */
__device__ __forceinline__ qr_dev_step step_at(const QC qr_dev_step *prog, uint32_t off)
{
    qr_dev_step v;
    __builtin_memcpy(&v, (const QC qr_dev_step *)((const QC char *)prog + off), sizeof(v));
    return v;
}

/* a ray's side of the box tests: its clamped reciprocal direction and, per
 * axis, the offsets that place a box's bounds on the ray, with the ray's
 * share of the allowance (QR_CULL_FUZZ times the L1 distance of its origin
 * o from the boxes' reference point) moving each bound outwards */
struct BoxRay
{
    float ix, iy, iz;
    float lx, ly, lz;       /* -(o + m) * i, for the lower bounds */
    float hx, hy, hz;       /* -(o - m) * i, for the upper bounds */
};

__device__ __forceinline__ BoxRay box_ray(const V3 &o, const V3 &dir, float rx, float ry,
                                          float rz)
{
    BoxRay b;
    b.ix = slab_rcp(dir.x);
    b.iy = slab_rcp(dir.y);
    b.iz = slab_rcp(dir.z);
    const float m = QR_CULL_FUZZ * (fabsf(o.x - rx) + fabsf(o.y - ry) + fabsf(o.z - rz));
    b.lx = -((o.x + m) * b.ix);
    b.ly = -((o.y + m) * b.iy);
    b.lz = -((o.z + m) * b.iz);
    b.hx = -((o.x - m) * b.ix);
    b.hy = -((o.y - m) * b.iy);
    b.hz = -((o.z - m) * b.iz);
    return b;
}

/* can the segment (t_min, t_buf) of the ray meet the box?  Slab test: the
 * ray's entry into the box must come no later than its exit and overlap
 * the segment.  The slab distances are formed with fused multiply-adds: the
 * test only decides what may be skipped, and the allowance is far above
 * their rounding. */
__device__ __forceinline__ bool box_pass(const qr_dev_step &st, const BoxRay &b,
                                         float t_min, float t_buf)
{
    const float x0 = __builtin_fmaf(st.lo[0], b.ix, b.lx);
    const float x1 = __builtin_fmaf(st.hi[0], b.ix, b.hx);
    const float y0 = __builtin_fmaf(st.lo[1], b.iy, b.ly);
    const float y1 = __builtin_fmaf(st.hi[1], b.iy, b.hy);
    const float z0 = __builtin_fmaf(st.lo[2], b.iz, b.lz);
    const float z1 = __builtin_fmaf(st.hi[2], b.iz, b.hz);
    const float tn = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fminf(z0, z1));
    const float tf = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fmaxf(z0, z1));
    return fmaxf(tn, t_min) <= fminf(tf, t_buf);
}

/* whether QuadRay gives a surface a nearest-hit list of its own for the
 * rays leaving it (reflecting or not opaque on either side,
 * core/engine/engine.cpp:2180-2201), built in the reverse of the global
 * list's order; other surfaces' rays walk the global list itself */
__device__ __forceinline__ bool own_list(const Scene &sc, int surf)
{
    return (sc.hot[surf].flags & QR_DS_OWN_LIST) != 0;
}

/* most work-items in a workgroup of a kernel that walks the surface list */
#define QR_WALK_MAX_WG 256

/* walk the surface list through the culling program: nearest accepted root
 * (h.srf, h.side, h.t), or any shadowing root (SHADOW).  Accepted roots follow
 * QuadRay's overwrite rules: the second root of a surface is skipped once the
 * first is accepted, and of roots at the same distance the first in list
 * order wins, or with "rev" the last: camera rays, and the rays leaving a
 * surface that has its own list (own_list: every secondary ray of the
 * Whitted tracer), walk lists that QuadRay builds in the reverse of this
 * one's order.  T0: the ray's t_min is 0.
 *
 * The loop has one exit, taken by the whole wave: a lane whose shadow test
 * is decided stops keeping boxes open, and the wave leaves once every lane
 * is decided (a lane leaving on its own would split the loop's exit and cost
 * every iteration a per-lane state dispatch).
 *
 * An element's registers (DFF_X / DFF_I / RAY_I of QuadRay's list walk,
 * OO_loc, tracer.cpp:2466-2684) are the ray's origin and direction in the
 * frame of the surface (dd, rr) and of the open transform node (node_o,
 * node_d).  What decides between them is the same for the whole wave, so
 * the branches are scalar; only a ray leaving the surface itself differs,
 * which takes its origin's local hit.  Which lanes keep a root is held in
 * wave masks: no branch of the element work changes the active lanes, but
 * for the rare near-zero discriminants and apexes.
 *
 * What bounds it is VALU issue (the path tracer's bounces are busy with it 85 %
 * of their time), so a quadric takes only what its class needs,
 * its quotients are formed only for roots that can lie in the ray's range,
 * and a hit point only where the surface clips: 1.77e10 wave-level VALU
 * instructions and 6.5e8 scalar loads in the bounces of a 1280x720 64-spp
 * frame, 2.09e10 and 2.2e9 with a division and a clipping stage per root read
 * from the 208-byte record (37.5 -> 31.4 ms). */
template <bool SHADOW, bool T0 = SHADOW>
__device__ bool walk(const Scene &sc, const Ray &r, Hit &best, bool rev = true)
{
    V3 node_o = V3{0, 0, 0};
    V3 node_d = V3{0, 0, 0};
    int cache_last = -1;    /* trnode: last element of the group, -1 off */
    int cache_first = 0;    /* the group's transform-node element */
    /* The largest distance wanted.  The depth test is strict, but a
     * nearest-hit walk takes a root equal to the kept one (a tie, "rev"), so
     * the limit is the kept distance itself or the float below it; with no
     * hit yet no root ties with t_max. */
    const uint32_t below = rev ? 0u : 1u;
    float t_lim = bitsf(fbits(r.t_max) - 1u);
    int kept = -1;          /* record's byte offset | side */
    /* lanes that still keep boxes open (any-hit walks: not yet shadowed),
     * as a wave mask that the box tests' ballots are masked with */
    uint64_t live = lanes(true);

    /* the ray's side of the world boxes (the reciprocal direction is
     * approximate: the boxes carry an allowance far above its error) */
    const BoxRay br = box_ray(r.org, r.dir, sc.ref_x, sc.ref_y, sc.ref_z);

    const QC qr_dev_step *prog = SHADOW ? sc.step_any : sc.step;
    /* the ray's side of the open transform-node group's member boxes, in the
     * node's frame: kept in LDS, a slot per work-item, not in registers the
     * whole loop would hold.  A member's step is reached only through its
     * node's step: the upload gives a member step that kind only in a
     * program where that holds. */
    __shared__ float s_gb[9][QR_WALK_MAX_WG];
    const unsigned tid = threadIdx.x;
    /* the byte offset of the ray's origin surface record (none: matches no
     * record) */
    const uint32_t org_off = r.origin >= 0 ? (uint32_t)r.origin * (uint32_t)sizeof(qr_dev_surf)
                                           : 0xffffffffu;
    /* two loops: the inner one runs the box steps up to the next element
     * step and touches no walk register, so the element work is the only
     * path back to the outer loop's head (the walk registers then need no
     * copies where paths merge).  The step is addressed by its byte offset
     * and a box step's skip is one, and the program's end step stops the
     * walk, so a box step costs its test, one select and one load. */
    for (uint32_t off = 0;; off += QR_DEV_STEP_BYTES)
    {
        /* a step is one 32-byte scalar load (box, element and skip
         * together), so a box step waits for one load, not three in a row */
        qr_dev_step st = step_at(prog, off);
        while (st.elem < 0)
        {
            const uint64_t near = lanes(box_pass(st, br, r.t_min, t_lim));
            off = (near & live) != 0 ? off + QR_DEV_STEP_BYTES : (uint32_t)st.skip;
            st = step_at(prog, off);
        }
        if (st.elem == QR_DEV_STEP_END) break;
        const int e = st.elem;
        const int kind = qr_dev_step_local(&st);
        /* a member of the open group: its box in the group's frame, before
         * anything of the surface is loaded (a member's skipped set-up
         * changes nothing for the elements after it) */
        /* the loop body has one path back to its head (no continue): the
         * element is tested only while some live lane keeps it */
        uint64_t keep = live;
        if (kind == QR_LOCAL_GROUP)
        {
            BoxRay gb;
            gb.ix = s_gb[0][tid];
            gb.iy = s_gb[1][tid];
            gb.iz = s_gb[2][tid];
            gb.lx = s_gb[3][tid];
            gb.ly = s_gb[4][tid];
            gb.lz = s_gb[5][tid];
            gb.hx = s_gb[6][tid];
            gb.hy = s_gb[7][tid];
            gb.hz = s_gb[8][tid];
            keep &= lanes(box_pass(st, gb, r.t_min, t_lim));
        }
        if (keep != 0)
        {
            /* the record's byte offset (the index only for a kept hit), and
             * its head: one load */
            const uint32_t soff = (uint32_t)st.skip & ~3u;
            const QC qr_dev_surf *const sp = surf_at(sc, soff);
            const SurfHead s = ldk<SurfHead>(sp);
            /* the cache holds only inside its group, whose last element may
             * have been skipped (the any-hit program also visits groups out
             * of list order) */
            if (e > cache_last || e < cache_first) cache_last = -1;
            V3 rr, dd;
            if (cache_last >= 0 && (s.flags & QR_DS_SOLO) == 0)
            {
                dd = sub3(node_o, s.pos);
                rr = node_d;
                if (e == cache_last) cache_last = -1;
            }
            else
            {
                dd = sub3(r.org, s.pos);
                rr = r.dir;
                if (s.flags & QR_DS_TRM)
                {
                    if ((s.flags & QR_DS_TRM) != QR_DS_TRM_DIAG)
                    {
                        const SurfOff o = ldk<SurfOff>(sp->to);
                        dd = xform_full(s.td, o.to, dd);
                        rr = xform_full(s.td, o.to, rr);
                    }
                    else
                    {
                        dd = xform_diag(s.td, dd);
                        rr = xform_diag(s.td, rr);
                    }
                    if (s.flags & QR_DS_SOLO)
                    {
                        /* a transform node (never a ray's origin) opens its
                         * group, whose end its step holds: the ray in the
                         * node's frame, about the node's origin */
                        node_o = dd;
                        node_d = rr;
                        cache_last = __float_as_int(st.lo[0]);
                        cache_first = e;
                        const BoxRay gb = box_ray(dd, rr, 0.0f, 0.0f, 0.0f);
                        s_gb[0][tid] = gb.ix;
                        s_gb[1][tid] = gb.iy;
                        s_gb[2][tid] = gb.iz;
                        s_gb[3][tid] = gb.lx;
                        s_gb[4][tid] = gb.ly;
                        s_gb[5][tid] = gb.lz;
                        s_gb[6][tid] = gb.hx;
                        s_gb[7][tid] = gb.hy;
                        s_gb[8][tid] = gb.hz;
                        /* (were the node a surface in world coordinates) */
                        if (!(s.flags & QR_DS_SHIFT)) rr = r.dir;
                    }
                }
                else if (cache_last >= 0)
                {
                    /* inside a group, but in world coordinates (caller
                     * tables alone): the origin register holds what the node
                     * left, or the ray's own surface's local hit; a node
                     * without a transform leaves it its own */
                    if ((sp->info & QR_DI_NODE) == 0)
                    {
                        dd = pick(soff == org_off, r.oloc, node_o);
                        if (e == cache_last) cache_last = -1;
                    }
                    node_o = dd;
                }
            }
            const uint64_t same = lanes(soff == org_off);
            if (same != 0)
            {
                const bool m = in_lane(same);
                dd = pick(m, r.oloc, dd);
            }
            const uint32_t cls = s.flags & QR_DS_CLASS;
            if (cls != QR_SOLVE_NONE)
            {
                if (kind == QR_LOCAL_OWN)
                {
                    /* the surface's own box, in its tracing frame (the
                     * registers the roots are computed from), whose
                     * reference point is the surface's origin */
                    const BoxRay bl = box_ray(dd, rr, 0.0f, 0.0f, 0.0f);
                    keep &= lanes(box_pass(st, bl, r.t_min, t_lim));
                }
                if (keep != 0)
                {
                    const float t_next = above<T0>(t_lim);
                    /* the lanes with a first and a second root, and those
                     * whose first is of side 1 */
                    uint64_t m1, m2 = 0, side, dmask = 0;
                    float n, d, a_val = 0.0f, n2 = 0.0f, d2 = 0.0f;
                    if (cls == QR_DC_PLANE)
                    {
                        const int k = amap(s.flags, 2);
                        if (k == 0)
                        {
                            n = -dd.x;
                            d = rr.x;
                        }
                        else if (k == 1)
                        {
                            n = -dd.y;
                            d = rr.y;
                        }
                        else
                        {
                            n = -dd.z;
                            d = rr.z;
                        }
                        /* (-dff) / ray, both negated where the plane's axis
                         * is: the quotient is the same */
                        side = lanes(!(d < 0.0f));
                        if (asgn(s.flags, 2)) side = lanes(!(d > 0.0f));
                        m1 = roots_near<T0>(n, d, r.t_min, t_next) & ~same;
                    }
                    else
                    {
                        float b_val, c_val;
                        const float d_val = quadric_abc(s.flags, s.sci, s.scj, rr, dd, a_val,
                                                        b_val, c_val);
                        m1 = lanes(0.0f <= d_val);
                        side = 0;
                        n = d = 0.0f;
                        if (m1 != 0)
                        {
                            side = lanes(0.0f > a_val);
                            Roots q;
                            dmask = lanes(d_val < s.d_eps) & m1;
                            if (dmask != 0 || !(s.d_eps >= SQRT_MID_MIN))
                            {
                                roots_any(a_val, b_val, c_val, d_val, s.d_eps, s.t_eps, q);
                            }
                            else
                            {
                                roots_mid(a_val, b_val, c_val, d_val, side, q);
                            }
                            n = q.n1;
                            d = q.d1;
                            n2 = q.n2;
                            d2 = q.d2;
                            m2 = roots_near<T0>(n2, d2, r.t_min, t_next) & m1;
                            m1 &= roots_near<T0>(n, d, r.t_min, t_next);
                            if (same != 0)
                            {
                                /* a ray leaving this surface skips the root
                                 * it starts from: the other side's, or its
                                 * own when it passes through */
                                const uint64_t own = lanes((r.flags & 1) != 0) ^
                                                     lanes((r.flags & 2) == 0);
                                m1 &= ~(same & ~(own ^ side));
                                m2 &= ~(same & (own ^ side));
                            }
                        }
                    }
                    /* the roots in their order: the second only where the
                     * first is not accepted */
                    uint64_t take = m1 | m2;
                    while (take != 0)
                    {
                        /* (the flags' tests stay inside the loop: hoisted,
                         * their lane masks do not fit the scalar registers) */
                        uint32_t flags = s.flags;
                        asm volatile("" : "+s"(flags));
                        const uint64_t use2 = take & ~m1;
                        if (use2 != 0)
                        {
                            const bool u = in_lane(use2);
                            n = u ? n2 : n;
                            d = u ? d2 : d;
                            side ^= use2;
                        }
                        const float t = n / d;
                        uint64_t acc = take & lanes(t <= t_lim) & lanes(r.t_min < t);
                        if ((flags & (QR_DS_AXIS_CLIP | QR_DS_CLIPS)) && acc != 0)
                        {
                            acc &= clip_root(sc, r, s, flags, sp, rr, dd, t, side, dmask, a_val);
                        }
                        take = m1 & m2 & ~acc;
                        m1 = 0;
                        if (SHADOW)
                        {
                            uint64_t cast = 0;
                            if (flags & (1u << QR_DS_SHADOW_BIT)) cast |= ~side;
                            if (flags & (2u << QR_DS_SHADOW_BIT)) cast |= side;
                            live &= ~(acc & cast);
                        }
                        else
                        {
                            const bool u = in_lane(acc);
                            t_lim = u ? bitsf(fbits(t) - below) : t_lim;
                            const int code = (int)soff | (in_lane(side) ? 1 : 0);
                            kept = u ? code : kept;
                        }
                    }
                    if (SHADOW && live == 0) break;
                }
            }
        }
    }
    if (SHADOW) return !in_lane(live);
    best.srf = kept < 0 ? -1 : kept / (int)sizeof(qr_dev_surf);
    best.side = kept & 1;
    best.t = bitsf(fbits(t_lim) + below);
    return kept >= 0;
}

/* hit point, local hit and plane texture coordinates of an accepted root,
 * recomputed with the operations the walk applied to it: the element set-up
 * (after its transform node's, for a grouped surface), the roots' apex snap
 * and the local hit of that surface */
__device__ void hit_info(const Scene &sc, const Ray &r, Hit &h)
{
    const QC qr_dev_surf &s = sc.hot[h.srf];
    const uint32_t flags = s.flags;
    const bool same = h.srf == r.origin;
    const float td[3] = {s.td[0], s.td[1], s.td[2]};
    const V3 pos = V3{s.pos[0], s.pos[1], s.pos[2]};
    V3 dd, rr;
    bool cached = false;
    const int node = s.trnode;
    if ((s.info & QR_DI_NODE) == 0 && node >= 0 && node != h.srf)
    {
        const QC qr_dev_surf &n = sc.hot[node];
        const uint32_t nf = n.flags;
        if ((nf & QR_DS_SOLO) != 0 && (nf & QR_DS_TRM) != 0)
        {
            const float nd[3] = {n.td[0], n.td[1], n.td[2]};
            const V3 d = sub3(r.org, n.pos);
            if ((nf & QR_DS_TRM) != QR_DS_TRM_DIAG)
            {
                const float to[6] = {n.to[0], n.to[1], n.to[2], n.to[3], n.to[4], n.to[5]};
                dd = xform_full(nd, to, d);
                rr = xform_full(nd, to, r.dir);
            }
            else
            {
                dd = xform_diag(nd, d);
                rr = xform_diag(nd, r.dir);
            }
            cached = true;
        }
    }
    if (cached)
    {
        if (flags & QR_DS_SHIFT)
        {
            dd = V3{dd.x - pos.x, dd.y - pos.y, dd.z - pos.z};
        }
        else
        {
            rr = r.dir;     /* dff_x: the node's */
        }
    }
    else
    {
        dd = V3{r.org.x - pos.x, r.org.y - pos.y, r.org.z - pos.z};
        rr = r.dir;
        if (flags & QR_DS_SHIFT)
        {
            if ((flags & QR_DS_TRM) != QR_DS_TRM_DIAG)
            {
                const float to[6] = {s.to[0], s.to[1], s.to[2], s.to[3], s.to[4], s.to[5]};
                dd = xform_full(td, to, dd);
                rr = xform_full(td, to, rr);
            }
            else
            {
                dd = xform_diag(td, dd);
                rr = xform_diag(td, rr);
            }
        }
    }
    if (same) dd = r.oloc;
    h.hit = ray_at(r.dir, r.org, h.t);
    if (flags & QR_DS_SHIFT) h.loc = ray_at(rr, dd, h.t);
    else h.loc = V3{h.hit.x - pos.x, h.hit.y - pos.y, h.hit.z - pos.z};
    if (flags & QR_DS_APEX)
    {
        const float sci[4] = {s.sci[0], s.sci[1], s.sci[2], s.sci[3]};
        const float scj[3] = {s.scj[0], s.scj[1], s.scj[2]};
        float a_val, b_val, c_val;
        const float d_val = quadric_abc(flags, sci, scj, rr, dd, a_val, b_val, c_val);
        if (0.0f <= d_val && d_val < s.d_eps)
        {
            apex_snap(flags, sci, s.t_eps, dd, h.side, fbits(a_val) & SIGN, h.loc);
        }
    }
    if ((flags & QR_DS_CLASS) == QR_DC_PLANE)
    {
        h.u = negif(sel(h.loc, amap(flags, 0)), asgn(flags, 0));
        h.v = negif(sel(h.loc, amap(flags, 1)), asgn(flags, 1));
    }
    else
    {
        h.u = 0.0f;
        h.v = 0.0f;
    }
}

/* surface normal in world space (PL 5669-5685, QD 6237-6281, TP 6415-6455,
 * transform 3273-3348) */
__device__ V3 normal_at(const Scene &sc, const Hit &h)
{
    const QC qr_dev_surf &s = sc.hot[h.srf];
    const uint32_t flags = s.flags;
    const uint32_t kind = (flags >> QR_DS_NRM_BIT) & 3u;
    V3 n;
    const uint32_t ts = h.side ? SIGN : 0u;
    if (kind == 1)
    {
        V3 z = {0.0f, 0.0f, 0.0f};
        put(z, amap(flags, 2), negif(fxor(1.0f, ts), asgn(flags, 2)));
        n = z;
    }
    else
    {
        V3 l;
        l.x = h.loc.x * s.sci[0];
        l.y = h.loc.y * s.sci[1];
        l.z = h.loc.z * s.sci[2];
        if (kind == 2)
        {
            l.x = l.x - s.scj[0];
            l.y = l.y - s.scj[1];
            l.z = l.z - s.scj[2];
        }
        float rr = l.x * l.x + l.y * l.y;
        rr = rr + l.z * l.z;
        float inv = fxor(rsq(rr), ts);
        n = V3{l.x * inv, l.y * inv, l.z * inv};
    }
    if ((s.info & QR_DI_TRM) == 0) return n;

    const QC qr_dev_surf &t = sc.hot[s.trnode];
    const uint32_t trm = t.info & QR_DI_TRM;
    float x = t.td[0] * n.x;
    float y = t.td[1] * n.y;
    float z = t.td[2] * n.z;
    bool renorm = true;
    if (trm != QR_DI_TRM_DIAG)
    {
        /* the transposed matrix: to holds 01 02 10 12 20 21 */
        x = x + t.to[2] * n.y;
        x = x + t.to[4] * n.z;
        y = y + t.to[0] * n.x;
        y = y + t.to[5] * n.z;
        z = z + t.to[1] * n.x;
        z = z + t.to[3] * n.y;
        renorm = trm != QR_DI_TRM_ROT;
    }
    if (renorm)
    {
        float rr = x * x + y * y;
        rr = rr + z * z;
        float inv = rsq(rr);
        x = x * inv; y = y * inv; z = z * inv;
    }
    return V3{x, y, z};
}

/* vector to a light and its dot product with the normal (LT, 4015-4035) */
__device__ __forceinline__ float light_vec(const QC qr_light &l, const V3 &hit,
                                           const V3 &nrm, V3 &L)
{
    L = V3{l.pos[0] - hit.x, l.pos[1] - hit.y, l.pos[2] - hit.z};
    float dot = L.x * nrm.x + L.y * nrm.y;
    dot = dot + L.z * nrm.z;
    return dot;
}

/* fixed point 28.4 specular power (tracer.cpp:4225-4283) */
__device__ float spec_pow(float s, uint32_t pw)
{
    uint32_t fr = pw & 0xF;
    float x2 = s, x4 = s, r = 1.0f;
    while (fr != 0)
    {
        x4 = sqrtf(x4);
        uint32_t bit = 0x8 & fr;
        fr = (fr << 1) & 0xF;
        if (bit) r = r * x4;
    }
    uint32_t ip = pw >> 4;
    if (ip != 0)
    {
        float fp = r;
        r = 1.0f;
        while (ip != 0)
        {
            if (ip & 1) r = r * x2;
            ip >>= 1;
            x2 = x2 * x2;
        }
        r = r * fp;
    }
    return r;
}

/* surface colour at a hit: texel lookup and gamma to linear (MT_tex
 * 3382-3416, PAINT_SIMD 985) */
__device__ __forceinline__ V3 texel_color(const Scene &sc, const QC qr_material &m,
                                          uint32_t props, const Hit &h)
{
    uint32_t idx = 0;
    if (props & QR_PROP_TEXTURE)
    {
        float tx = m.tmap[0] ? h.v : h.u;
        float ty = m.tmap[1] ? h.v : h.u;
        tx = tx - m.xoffs;
        ty = ty - m.yoffs;
        tx = tx * m.xscal;
        ty = ty * m.yscal;
        uint32_t ix = (uint32_t)cvt_floor(tx) & m.xmask;
        uint32_t iy = (uint32_t)cvt_floor(ty) & m.ymask;
        idx = ix + (iy << m.yshft);
    }
    const uint32_t tv = sc.texel[m.tex_off + idx];
    V3 tex;
    tex.x = unorm8((tv >> 16) & 0xFFu);
    tex.y = unorm8((tv >> 8) & 0xFFu);
    tex.z = unorm8(tv & 0xFFu);
    if (props & QR_PROP_GAMMA)
    {
        tex.x = tex.x * tex.x;
        tex.y = tex.y * tex.y;
        tex.z = tex.z * tex.z;
    }

    return tex;
}

/* refraction and reflection set-up of a hit: which children it spawns,
 * their directions, and the transmitted / reflected fractions with Fresnel
 * and total inner reflection (TR 4442-4936, RF 4944-5357).  The transparent,
 * the opaque and the metal Fresnel terms are two quotients each, formed by
 * one pair of divisions for all of a wave's lanes, and the ray's direction
 * is normalised once for both children (with the short roots above and the
 * path tracer's one append per workgroup: 1.64e10 -> 1.57e10 wave-level VALU
 * instructions in the bounces of a 1280x720 64-spp frame, 30.3 -> 29.7 ms). */
struct TrRf
{
    bool  tr, rf;
    bool  fresnel_tr;       /* Fresnel computed in the transparency block */
    float c_trn, c_rfl;
    V3    tdir, rdir;
};

__device__ __forceinline__ TrRf trrf_setup(const QC qr_material &m, uint32_t props,
                                           const V3 &rd, const V3 &nrm)
{
    TrRf t;
    const bool transp = !(props & QR_PROP_OPAQUE);
    const bool fresnel = (props & QR_PROP_FRESNEL) != 0;
    const bool bend = transp && ((props & QR_PROP_REFRACT) || fresnel);
    t.tr = transp;
    t.rf = (props & QR_PROP_REFLECT) || (transp && fresnel);
    t.fresnel_tr = transp && fresnel;
    t.tdir = rd;
    t.c_trn = m.c_trn;
    t.c_rfl = m.c_rfl;
    if (!bend && !t.rf) return t;

    float r2 = rd.x * rd.x;
    r2 = r2 + rd.y * rd.y;
    r2 = r2 + rd.z * rd.z;
    const float inv = rsq(r2);
    const V3 rn = {rd.x * inv, rd.y * inv, rd.z * inv};
    float dot = rn.x * nrm.x;
    dot = dot + rn.y * nrm.y;
    dot = dot + rn.z * nrm.z;

    /* Fresnel's quotients n0 / d0 and n1 / d1 */
    bool quot = fresnel;
    const bool metal = fresnel && !transp && (props & QR_PROP_METAL);
    float n0 = 0.0f, d0 = 1.0f, n1 = 0.0f, d1 = 1.0f;
    if (metal)
    {
        float x6 = m.c_rcp;
        float x4 = dot * x6;
        x4 = x4 + x4;
        float x0 = dot * dot;
        x6 = x6 * x6;
        x6 = x6 + m.ext_2;
        float x1 = x0 * x6;
        x0 = x0 + x6;
        x1 = x1 + 1.0f;
        n0 = x0 + x4;
        n1 = x1 + x4;
        d0 = x0 - x4;
        d1 = x1 - x4;
    }
    else if (bend || fresnel)
    {
        const float n = m.c_rfr;
        float x0 = dot * n;
        float k = x0 * x0;
        k = k + 1.0f;
        k = k - m.rfr_2;
        if (transp && fresnel && !(0.0f <= k))
        {
            /* total inner reflection */
            t.tr = false;
            t.c_trn = 0.0f;
            t.c_rfl = m.c_rfl + m.c_trn;
            quot = false;
        }
        else
        {
            const float sk = root(k);
            x0 = x0 + sk;
            if (transp && (props & QR_PROP_REFRACT))
            {
                float v;
                v = nrm.x * x0; t.tdir.x = rn.x * n; t.tdir.x = t.tdir.x - v;
                v = nrm.y * x0; t.tdir.y = rn.y * n; t.tdir.y = t.tdir.y - v;
                v = nrm.z * x0; t.tdir.z = rn.z * n; t.tdir.z = t.tdir.z - v;
            }
            n0 = x0;
            d0 = dot * n;
            d0 = d0 - sk;
            const float skn = sk * n;
            n1 = dot + skn;
            d1 = dot - skn;
        }
    }
    if (quot)
    {
        float q0 = n0 / d0;
        float q1 = n1 / d1;
        if (!metal)
        {
            q0 = q0 * q0;
            q1 = q1 * q1;
        }
        q0 = q0 + q1;
        q0 = q0 * -0.5f;
        float f0 = fabsf(q0);
        if (transp)
        {
            f0 = f0 * m.c_trn;
            t.c_trn = m.c_trn - f0;
        }
        else
        {
            f0 = f0 - 1.0f;
            f0 = f0 * m.c_rfl;
        }
        t.c_rfl = m.c_rfl + f0;
    }
    float v;
    v = nrm.x * dot; t.rdir.x = rn.x - v; t.rdir.x = t.rdir.x - v;
    v = nrm.y * dot; t.rdir.y = rn.y - v; t.rdir.y = t.rdir.y - v;
    v = nrm.z * dot; t.rdir.z = rn.z - v; t.rdir.z = t.rdir.z - v;
    return t;
}

/* ARGB8 packing of a resolved colour with optional gamma (1922-1945) */
__device__ __forceinline__ uint32_t pack_argb(const qr_frame_desc &fd, const V3 &c)
{
    const float v[3] = {c.x, c.y, c.z};
    uint32_t px = 0;
    #pragma unroll
    for (int ch = 0; ch < 3; ch++)
    {
        float f = v[ch];
        if (fd.gamma & QR_PROP_GAMMA) f = sqrtf(f);
        f = f * 255.0f;
        px |= ((uint32_t)cvt_rne(f) & 0xFFu) << (16 - 8 * ch);
    }
    return px;
}

/* anti-aliasing resolve of a pixel's clamped samples, halve then pairwise
 * add per pass (7047-7133), and ARGB8 packing */
__device__ __forceinline__ uint32_t resolve_pack(const qr_frame_desc &fd, int ns,
                                                 const V3 &a0, const V3 &a1,
                                                 const V3 &a2, const V3 &a3)
{
    V3 c;
    if (ns == 1)
    {
        c = a0;
    }
    else if (ns == 2)
    {
        c.x = a0.x * 0.5f + a1.x * 0.5f;
        c.y = a0.y * 0.5f + a1.y * 0.5f;
        c.z = a0.z * 0.5f + a1.z * 0.5f;
    }
    else
    {
        float p0, p1;
        p0 = a0.x * 0.5f + a1.x * 0.5f; p1 = a2.x * 0.5f + a3.x * 0.5f;
        c.x = p0 * 0.5f + p1 * 0.5f;
        p0 = a0.y * 0.5f + a1.y * 0.5f; p1 = a2.y * 0.5f + a3.y * 0.5f;
        c.y = p0 * 0.5f + p1 * 0.5f;
        p0 = a0.z * 0.5f + a1.z * 0.5f; p1 = a2.z * 0.5f + a3.z * 0.5f;
        c.z = p0 * 0.5f + p1 * 0.5f;
    }
    return pack_argb(fd, c);
}

/* the same resolve of a pixel's samples held by ns neighbouring groups of
 * "span" lanes (sample k in group k of an aligned run of groups): halve,
 * then add the partner's value per pass; every lane of the wave calls it with
 * the same ns, and each lane of the groups gets the pixel */
template <int span = 1>
__device__ __forceinline__ uint32_t resolve_lanes(const qr_frame_desc &fd, int ns, V3 c)
{
    for (int d = span; d < ns * span; d <<= 1)
    {
        const V3 h = V3{c.x * 0.5f, c.y * 0.5f, c.z * 0.5f};
        c.x = h.x + __shfl_xor(h.x, d);
        c.y = h.y + __shfl_xor(h.y, d);
        c.z = h.z + __shfl_xor(h.z, d);
    }
    return pack_argb(fd, c);
}

/* a pending node of the Whitted tree */
struct Node
{
    V3    col;          /* colour accumulated so far */
    float c_trn, c_rfl;
    V3    org;          /* hit point: origin of the children */
    V3    tdir, rdir;   /* refraction and reflection directions */
    V3    loc;          /* local hit for the children's self-tests */
    int   srf, side;
    int   depth;
    int   todo;         /* bit 0: refraction pending, bit 1: reflection */
};

/* colour of a hit without its lights (MT): a LIGHT material's own colour
 * ("lit" false), or the ambient part, with the texel the lights use */
__device__ __forceinline__ V3 shade_base(const Scene &sc, const qr_frame_desc &fd, const Hit &h,
                                         V3 &tex, bool &lit)
{
    const QC qr_surface &s = sc.srf[h.srf];
    const uint32_t props = s.props[h.side];
    const QC qr_material &m = sc.mat[s.mat[h.side]];
    tex = texel_color(sc, m, props, h);
    lit = !(props & QR_PROP_LIGHT);
    if (!lit) return tex;
    V3 col;
    col.x = tex.x * fd.amb[0];
    col.y = tex.y * fd.amb[1];
    col.z = tex.z * fd.amb[2];
    float f = 1.0f - m.c_trn;
    f = f - m.c_rfl;
    if (!(0.0f <= f)) f = 0.0f;
    col.x = col.x * f;
    col.y = col.y * f;
    col.z = col.z * f;
    return col;
}

/* a visible light's part of a hit's colour added to it (LT): L the vector to
 * the light, dot its product with the normal, rdir the ray's direction */
__device__ __forceinline__ void shade_light(const Scene &sc, const QC qr_light &l, const V3 &rdir,
                                            const Hit &h, const V3 &nrm, const V3 &tex, const V3 &L,
                                            float dot, V3 &col)
{
    const QC qr_surface &s = sc.srf[h.srf];
    const uint32_t props = s.props[h.side];
    const QC qr_material &m = sc.mat[s.mat[h.side]];
    float r2 = L.x * L.x + L.y * L.y;
    r2 = r2 + L.z * L.z;

    float dff = 0.0f;
    if (props & QR_PROP_DIFFUSE)
    {
        float ir = rsq(r2);
        float r1 = ir * r2;
        float at = r2 * l.a_qdr;
        float lr = r1 * l.a_lnr;
        at = at + l.a_cnt;
        at = at + lr;
        float ia = rsq(at);
        dff = dot * ia;
        dff = dff * ir;
        dff = dff * m.l_dff;
    }

    bool plain_spc = false;
    float spc = 0.0f;
    if (props & QR_PROP_SPECULAR)
    {
        V3 R;
        float v = dot * nrm.x;
        R.x = L.x - v; R.x = R.x - v;
        v = dot * nrm.y;
        R.y = L.y - v; R.y = R.y - v;
        v = dot * nrm.z;
        R.z = L.z - v; R.z = R.z - v;
        float rr2 = rdir.z * rdir.z;
        rr2 = rr2 + rdir.x * rdir.x;
        rr2 = rr2 + rdir.y * rdir.y;
        float sn = R.x * rdir.x + R.y * rdir.y;
        sn = sn + R.z * rdir.z;
        if (0.0f < sn)
        {
            sn = sn * rsq(rr2);
            sn = sn * rsq(r2);
            spc = spec_pow(sn, m.l_pow);
            spc = spc * m.l_spc;
            if (props & QR_PROP_METAL) dff = dff + spc;
            else plain_spc = true;
        }
    }

    V3 lc;
    if (plain_spc)
    {
        float v;
        v = tex.x * dff; v = v * l.col[0]; lc.x = v + l.col[0] * spc;
        v = tex.y * dff; v = v * l.col[1]; lc.y = v + l.col[1] * spc;
        v = tex.z * dff; v = v * l.col[2]; lc.z = v + l.col[2] * spc;
    }
    else
    {
        lc.x = (tex.x * l.col[0]) * dff;
        lc.y = (tex.y * l.col[1]) * dff;
        lc.z = (tex.z * l.col[2]) * dff;
    }
    col.x = lc.x + col.x;
    col.y = lc.y + col.y;
    col.z = lc.z + col.z;
}

/* local shading of a hit (MT, LT): its colour; visible(light) answers the
 * hard-shadow test of one light facing it */
template <class Visible>
__device__ V3 shade_color(const Scene &sc, const qr_frame_desc &fd, const V3 &rdir, const Hit &h,
                          const V3 &nrm, Visible visible)
{
    V3 tex;
    bool lit;
    V3 col = shade_base(sc, fd, h, tex, lit);
    if (lit)
    {
        for (int li = 0; li < sc.n_lgt; li++)
        {
            const QC qr_light &l = sc.lgt[li];
            V3 L;
            const float dot = light_vec(l, h.hit, nrm, L);
            if (!(0.0f < dot) || !visible(li)) continue;
            shade_light(sc, l, rdir, h, nrm, tex, L, dot, col);
        }
    }
    return col;
}

/* set-up of a hit's children (TR, RF), which does not depend on its
 * lighting: origin, directions, coefficients and which are pending */
__device__ __forceinline__ void node_children(const Scene &sc, const Ray &r, const Hit &h,
                                              const V3 &nrm, Node &nd)
{
    const QC qr_surface &s = sc.srf[h.srf];
    const uint32_t props = s.props[h.side];
    const QC qr_material &m = sc.mat[s.mat[h.side]];
    nd.org = h.hit;
    nd.loc = h.loc;
    nd.srf = h.srf;
    nd.side = h.side;
    nd.depth = r.depth;
    nd.todo = 0;

    const TrRf t = trrf_setup(m, props, r.dir, nrm);
    nd.todo |= (t.tr ? 1 : 0) | (t.rf ? 2 : 0);
    nd.tdir = t.tdir;
    nd.rdir = t.rdir;
    nd.c_trn = t.c_trn;
    nd.c_rfl = t.c_rfl;
    if (r.depth == 0) nd.todo = 0;
}

} /* namespace */

#endif /* QR_TRACER_DEV_H */
