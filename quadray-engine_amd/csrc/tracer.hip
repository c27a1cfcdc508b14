/*
 * tracer.hip -- one-kernel Whitted tracer for MI355X (gfx950).
 *
 * 1 to 16 work-items per camera sample (the fewer samples, the more); the
 * whole reflection / refraction tree of a sample is traced inside the kernel.
 * QuadRay's recursive context stack (shadow, refraction and reflection rays
 * re-entering the list walk, core/tracer/tracer.cpp 4046-4077, 4770-4862,
 * 5160-5277) becomes an explicit per-lane stack of pending tree nodes;
 * colours are accumulated bottom-up in QuadRay's order.
 * The level-by-level pipeline (tracer_wf.hip) is the default path; this
 * kernel serves frames without secondary rays, scenes beyond that pipeline's
 * light-mask limit, and callers that cannot allocate.
 *
 * Its time is that of its longest waves, whose lanes' trees are walked node
 * by node while the rest of the chip has run dry (vector issue was 4% busy
 * over a 640x360 frame of glass and mirrors at 2 samples).  So a lane takes
 * one sample, not a pixel's one after another, and where the frame leaves the
 * chip idle a wave holds fewer samples (its walks test only surfaces that
 * some lane of it needs, and the union of 4 samples' trees is shorter than
 * that of 64), SPLIT lanes each, which follow the same rays and test that
 * many lights' shadow rays at once: a node in a scene of four lights costs
 * two walks instead of five.
 *
 * Times, one pixel per lane before -> now: 640x360 at 2 samples, depth 4:
 * 2.55 -> 0.61 ms; 641x359 at 4, depth 8: 102 -> 11.0; 1281x719 at 2:
 * 9.4 -> 3.3; 64x64: 1.12 -> 0.29; 1920x1080 at 4: 5.2 -> 1.8.
 *
 * A frame without secondary rays needs no stack (1360 bytes of scratch and
 * 20 registers): 800x480 with one light 20 -> 14 us, 1920x1080 at 4 samples
 * 247 -> 162, with four lights 741 -> 561.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qr_soa.h"
#include "tracer_dev.h"
#include "tracer_kernels.h"

namespace {

__device__ __forceinline__ Ray child(const Node &nd, int which)
{
    Ray c;
    c.org = nd.org;
    c.dir = which == 1 ? nd.tdir : nd.rdir;
    c.t_min = 0.0f;
    c.t_max = 3.402823466e+38f;
    c.flags = nd.side | (which == 1 ? FLAG_PASS : 0);
    c.origin = nd.srf;
    c.oloc = nd.loc;
    c.depth = nd.depth - 1;
    return c;
}

/* the colour of a hit, its lights' shadow rays tested by the SPLIT lanes that
 * hold the sample, one each at a time */
template <int SPLIT>
__device__ __forceinline__ V3 hit_colour(const Scene &sc, const qr_frame_desc &fd, const Ray &ray,
                                         const Hit &h, const V3 &nrm)
{
    const int sub = (int)(threadIdx.x & (SPLIT - 1));
    const int group = __lane_id() & ~(SPLIT - 1);
    V3 tex;
    bool lit;
    V3 col = shade_base(sc, fd, h, tex, lit);
    for (int l0 = 0; lit && l0 < sc.n_lgt; l0 += SPLIT)
    {
        /* this lane's light of the next SPLIT, then all of them added in
         * their order */
        const int li = l0 + sub;
        Ray sr;
        bool vis = li < sc.n_lgt && 0.0f < light_vec(sc.lgt[li], h.hit, nrm, sr.dir);
        if (vis)
        {
            sr.org = h.hit;
            sr.t_min = 0.0f;
            sr.t_max = sc.lgt[li].t_max;
            sr.flags = h.side | FLAG_SHAD;
            sr.origin = h.srf;
            sr.oloc = h.loc;
            sr.depth = 0;
            Hit sh;
            vis = !walk<true>(sc, sr, sh);
        }
        const uint32_t seen = (uint32_t)(lanes(vis) >> group);
        for (int k = 0; k < SPLIT && l0 + k < sc.n_lgt; k++)
        {
            if (!((seen >> k) & 1u)) continue;
            const QC qr_light &l = sc.lgt[l0 + k];
            V3 L;
            const float dot = light_vec(l, h.hit, nrm, L);
            shade_light(sc, l, ray.dir, h, nrm, tex, L, dot, col);
        }
    }
    return col;
}

/* one camera sample of a frame without secondary rays */
template <int SPLIT>
__device__ V3 trace_camera(const Scene &sc, const qr_frame_desc &fd, const Ray &ray,
                           int32_t *hit_id)
{
    Hit h;
    if (!walk<false>(sc, ray, h))
    {
        *hit_id = -1;
        return V3{0.0f, 0.0f, 0.0f};
    }
    *hit_id = (sc.srf[h.srf].id << 1) | h.side;
    hit_info(sc, ray, h);
    return hit_colour<SPLIT>(sc, fd, ray, h, normal_at(sc, h));
}

/* one camera sample through the whole Whitted tree: a node waits on the
 * stack for its refraction child, then its reflection child, and folds each
 * result into its colour as QuadRay's TR_mix / RF_mix do */
template <int SPLIT>
__device__ V3 trace_sample(const Scene &sc, const qr_frame_desc &fd, Ray ray,
                           int32_t *hit_id)
{
    Node stk[MAX_STACK];
    int sp = 0;
    V3 ret = {0.0f, 0.0f, 0.0f};

    for (;;)
    {
        /* trace "ray" into node sp */
        Hit h;
        bool descend = false;
        if (!walk<false>(sc, ray, h))
        {
            ret = V3{0.0f, 0.0f, 0.0f};
            if (ray.origin < 0) *hit_id = -1;       /* (the camera's ray) */
        }
        else
        {
            if (ray.origin < 0) *hit_id = (sc.srf[h.srf].id << 1) | h.side;
            hit_info(sc, ray, h);
            const V3 nrm = normal_at(sc, h);
            Node &nd = stk[sp];
            nd.col = hit_colour<SPLIT>(sc, fd, ray, h, nrm);
            node_children(sc, ray, h, nrm, nd);
            if (nd.todo & 1)
            {
                nd.todo |= 4;
                ray = child(nd, 1);
                descend = true;
            }
            else if (nd.todo & 2)
            {
                nd.todo |= 8;
                ray = child(nd, 2);
                descend = true;
            }
            else
            {
                ret = nd.col;
            }
        }
        if (descend)
        {
            sp++;
            continue;
        }

        /* fold completed results into their parents */
        for (;;)
        {
            if (sp == 0) return ret;
            sp--;
            Node &nd = stk[sp];
            if (nd.todo & 4)
            {
                nd.col.x = ret.x * nd.c_trn + nd.col.x;
                nd.col.y = ret.y * nd.c_trn + nd.col.y;
                nd.col.z = ret.z * nd.c_trn + nd.col.z;
                nd.todo &= ~4;
                if (nd.todo & 2)
                {
                    nd.todo |= 8;
                    ray = child(nd, 2);
                    descend = true;
                    break;
                }
                ret = nd.col;
                continue;
            }
            nd.col.x = ret.x * nd.c_rfl + nd.col.x;
            nd.col.y = ret.y * nd.c_rfl + nd.col.y;
            nd.col.z = ret.z * nd.c_rfl + nd.col.z;
            ret = nd.col;
        }
        sp++;
    }
}

constexpr int log2i(int n) { return n < 2 ? 0 : 1 + log2i(n / 2); }

/* a wave's tile of pixels: its 64 / SPLIT samples, ns to a pixel, as near to
 * square as powers of two allow (wider before higher) */
template <int SPLIT>
__host__ __device__ constexpr int tile_w(int ns)
{
    return 1 << ((log2i(64 / SPLIT / ns) + 1) / 2);
}
template <int SPLIT>
__host__ __device__ constexpr int tile_h(int ns)
{
    return 1 << (log2i(64 / SPLIT / ns) / 2);
}

/* without a tree: 6 waves per SIMD spare a full chip more than their 36 bytes
 * of spills cost (397 surfaces at 1920x1080 and 4 samples, 5 -> 6 waves:
 * 2784 -> 2578 us); a frame that leaves it idle gains nothing by them (64x64
 * 47 -> 49).  Four waves per workgroup, their tiles side by side; a pixel's samples in neighbouring
 * groups of SPLIT lanes */
template <int SPLIT, bool TREE>
__global__ void __launch_bounds__(256, !TREE && SPLIT == 1 ? 6 : 4)
whitted_kernel(Scene sc, qr_frame_desc fd, int ns, uint32_t *__restrict__ frame,
               int32_t *__restrict__ ids)
{
    const int tw = ns == 1 ? tile_w<SPLIT>(1) : ns == 2 ? tile_w<SPLIT>(2) : tile_w<SPLIT>(4);
    const int th = ns == 1 ? tile_h<SPLIT>(1) : ns == 2 ? tile_h<SPLIT>(2) : tile_h<SPLIT>(4);
    const int wv = threadIdx.x / 64;
    const int s = (threadIdx.x & 63) / SPLIT;
    const int p = s / ns, k = s - p * ns;
    const int x = (blockIdx.x * 4 + wv) * tw + p % tw;
    const int y = (blockIdx.z * gridDim.y + blockIdx.y) * th + p / tw;
    const bool in = x < fd.x_res && y < fd.y_res;
    const bool first = (threadIdx.x & (SPLIT - 1)) == 0;

    V3 c = V3{0.0f, 0.0f, 0.0f};
    if (in)
    {
        int sk = k;
        if (fd.fsaa == 1 && (x & 1)) sk = k + 2;
        float hs = (float)x;
        float vs = (float)y;
        if (fd.fsaa != 0)
        {
            hs = hs + fd.aa_h[sk];
            vs = vs + fd.aa_v[sk];
        }
        Ray r;
        float hx, vx;
        hx = fd.hor[0] * hs; vx = fd.ver[0] * vs; hx = hx + vx; r.dir.x = hx + fd.dir[0];
        hx = fd.hor[1] * hs; vx = fd.ver[1] * vs; hx = hx + vx; r.dir.y = hx + fd.dir[1];
        hx = fd.hor[2] * hs; vx = fd.ver[2] * vs; hx = hx + vx; r.dir.z = hx + fd.dir[2];
        r.org = V3{fd.org[0], fd.org[1], fd.org[2]};
        r.t_min = fd.t_min;
        r.t_max = 3.402823466e+38f;
        r.flags = 0;
        r.origin = -1;
        r.oloc = V3{0.0f, 0.0f, 0.0f};
        r.depth = fd.depth;
        int32_t id;
        c = TREE ? trace_sample<SPLIT>(sc, fd, r, &id) : trace_camera<SPLIT>(sc, fd, r, &id);
        c.x = c.x < 1.0f ? c.x : 1.0f;
        c.y = c.y < 1.0f ? c.y : 1.0f;
        c.z = c.z < 1.0f ? c.z : 1.0f;
        if (ids != nullptr && first)
        {
            ids[((size_t)y * fd.x_res + x) * ns + k] = id;
        }
    }
    const uint32_t px = resolve_lanes<SPLIT>(fd, ns, c);
    if (in && first && k == 0) frame[(ptrdiff_t)y * fd.x_row + x] = px;
}

template <int SPLIT, bool TREE>
void launch(const Scene &sc, const qr_frame_desc &fd, int ns, uint32_t *frame, int32_t *ids,
            hipStream_t stream)
{
    const int tw = 4 * tile_w<SPLIT>(ns), th = tile_h<SPLIT>(ns);
    const unsigned nx = (unsigned)((fd.x_res - 1) / tw + 1), ny = (unsigned)((fd.y_res - 1) / th + 1);
    const unsigned gy = ny < 65535u ? ny : 65535u;
    hipLaunchKernelGGL((whitted_kernel<SPLIT, TREE>), dim3(nx, gy, (ny + gy - 1) / gy), dim3(256), 0, stream,
                       sc, fd, ns, frame, ids);
}

} /* namespace */

hipError_t qr_launch_whitted(const qr_device_tables *t, const qr_frame_desc *fd,
                             uint32_t *frame, int32_t *ids, hipStream_t stream)
{
    const Scene sc = scene_of(t);
    if (fd->depth < 0 || fd->depth > MAX_STACK - 2)
    {
        return hipErrorInvalidValue;
    }
    const int ns = fd->fsaa == 2 ? 4 : fd->fsaa == 1 ? 2 : 1;
    /* lanes per sample, by how many samples there are to fill the chip (a
     * frame without secondary rays, whose waves all take about as long, fills
     * it with a sixteenth).  ms at 1, 2, 4 and 16 lanes: 320x180 1.43 0.89
     * 0.55 0.37; 640x360 at 2 samples 1.22 0.83 0.61 0.89; 1920x1080 1.32 1.09
     * 0.96 2.68; at 2 samples 1.49 1.30 1.51 5.41; at 4 1.80 1.88 2.99 9.75;
     * without secondary rays, 64x64 0.148 0.092 0.060 0.048; 640x360 at 2
     * 0.089 0.089 0.125 0.431 (8 lanes lie between 4 and 16) */
    const uint64_t n = (uint64_t)fd->x_res * (uint64_t)fd->y_res * (uint64_t)ns;
    if (!qr_frame_has_tree(t, fd))
    {
        if (n <= (1u << 14)) launch<16, false>(sc, *fd, ns, frame, ids, stream);
        else if (n <= (1u << 17)) launch<4, false>(sc, *fd, ns, frame, ids, stream);
        else launch<1, false>(sc, *fd, ns, frame, ids, stream);
    }
    else if (n <= (1u << 18)) launch<16, true>(sc, *fd, ns, frame, ids, stream);
    else if (n <= (1u << 21)) launch<4, true>(sc, *fd, ns, frame, ids, stream);
    else if (n <= (1u << 22)) launch<2, true>(sc, *fd, ns, frame, ids, stream);
    else launch<1, true>(sc, *fd, ns, frame, ids, stream);
    return hipGetLastError();
}
