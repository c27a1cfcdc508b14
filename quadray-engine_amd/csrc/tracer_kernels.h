/*
 * tracer_kernels.h -- launch interface of the HIP kernels (internal to
 * libqrhip; the public boundary is include/qrhip.h).
 */
#ifndef QR_TRACER_KERNELS_H
#define QR_TRACER_KERNELS_H

#include <hip/hip_runtime.h>

#include "qr_soa.h"
#include "refit.h"

/* a culling step as the kernels read it: the box of a qr_cull_step as
 * bounds grown by the box's share of the allowance, QR_CULL_FUZZ times the
 * L1 distance of its centre from the reference point (world boxes:
 * cull_ref; local boxes: the origin of the frame they are in).  A ray adds its own
 * share, QR_CULL_FUZZ times the L1 distance of its origin from the same
 * point; the sum bounds QR_CULL_FUZZ times the distance from the origin to
 * the centre, so every box is at least the one the allowance defines. */
typedef struct qr_dev_step
{
    float    lo[3], hi[3];
    int32_t  elem;
    int32_t  skip;
} qr_dev_step;

/* A box step has elem -1 and skip = the byte offset of the step after its
 * range (QR_DEV_STEP_BYTES times its index), which the walk adds to the
 * program's address as it is.  An element step carries what the walk needs
 * before it can load the surface record, so one scalar load of the step
 * starts it: skip is the byte offset of its qr_dev_surf record with the
 * kind of its local box in the low two bits (records are 4-byte multiples),
 * and an element without a local box keeps its "last" (a transform node's
 * group end, else -1) in lo[0]'s bits.  Local boxes:
 *
 *   QR_LOCAL_GROUP  a surface in a transform node's frame (a member of the
 *                   node's group): the box in that frame, about the node's
 *                   origin, tested against the ray as the node's step left
 *                   it in that frame, before the surface's own set-up;
 *   QR_LOCAL_OWN    a surface that is its own transform node: the box in its
 *                   frame about its origin, tested after its set-up.
 *
 * A device program of n steps is followed by an end step (elem
 * QR_DEV_STEP_END), where every walk stops, so a walk never compares a
 * step's index with the program's length. */
#define QR_DEV_STEP_BYTES 32
#define QR_DEV_STEP_END   0x7fffffff
/* most steps a device program holds (its byte offsets fit an int32) */
#define QR_DEV_STEP_MAX   ((1 << 26) - 1)
#define QR_LOCAL_NONE  0
#define QR_LOCAL_GROUP 1
#define QR_LOCAL_OWN   2
/* most records a surface table of the kernels holds (byte offsets fit an
 * int32) */
#define QR_DEV_SURF_MAX ((int)(0x7fffffff / sizeof(qr_surface)))

/* A surface as the walks read it: what one list element needs of its
 * qr_surface record, in the order of use, with the small integers packed in
 * one flag word.  The first 64 bytes (up to td) are one scalar load, which
 * every element step issues at once; the rest is read by the surfaces that
 * have clips or a full rotation.  Read from the 208-byte record, an element
 * step was about fifteen scalar loads one after another, each for a control
 * word that decided which came next, and a wave waited for each of them. */
typedef struct qr_dev_surf
{
    float    pos[3];
    uint32_t flags;             /* QR_DS_* */
    float    sci[4];
    float    scj[3];
    float    d_eps, t_eps;
    float    td[3];             /* diagonal of the inverse transform tc */
    float    cmin[3], cmax[3];
    float    to[6];             /* off its diagonal: 01 02 10 12 20 21 */
    int32_t  clip_beg, clip_cnt;
    int32_t  trnode;            /* record of the transform node, -1: none */
    uint32_t info;              /* QR_DI_* */
} qr_dev_surf;
#define QR_DS_CLASS     0x7u            /* QR_DC_* */
#define QR_DS_SHIFT     0x8u            /* traced in its node's or its own frame */
#define QR_DS_TRM       0x30u           /* the transform into that frame (a node's: */
#define QR_DS_TRM_DIAG  0x10u           /* its group's); bits: none, diagonal,
                                           rotation, rotation and scale */
#define QR_DS_SOLO      0x40u           /* not in an open group's frame: a transform
                                           node, or a surface without "shift",
                                           which is traced in world coordinates
                                           (and has no QR_DS_TRM, whatever
                                           transform its record holds) */
#define QR_DS_APEX      0x80u
#define QR_DS_APEX_TWO  0x100u          /* apex kind 2 (two planes) */
#define QR_DS_CMIN_BIT  9               /* bit 9 + a: axis a has a min clip */
#define QR_DS_CMAX_BIT  12
#define QR_DS_AXIS_CLIP 0x7e00u
#define QR_DS_CLIPS     0x8000u         /* has custom clippers */
#define QR_DS_CLP_BIT   16              /* two bits: clp_kind 1, 2 or 3 */
#define QR_DS_AMAP_BIT  18              /* two bits per local axis */
#define QR_DS_ASGN_BIT  24              /* a bit per local axis */
#define QR_DS_SHADOW_BIT 27             /* bit 27 + side: it casts shadows */
#define QR_DS_NRM_BIT   29              /* two bits: nrm_kind 1, 2 or 3 */
#define QR_DS_OWN_LIST  0x80000000u     /* rays leaving it walk a list of its own */
/* what the walk's loop does not read: the record's transform as it stands
 * (normals turn by their node's), and whether it is a transform node (an
 * array) */
#define QR_DI_TRM       0x3u
#define QR_DI_TRM_DIAG  0x1u
#define QR_DI_TRM_ROT   0x2u
#define QR_DI_NODE      0x4u
/* classes: QR_SOLVE_* with the quadrics that need fewer operations apart.
 * x - (+0) and x * 1 are x for every x, so those are the same roots. */
#define QR_DC_PLANE     1
#define QR_DC_QUADRIC   2
#define QR_DC_TWOPLANE  3
#define QR_DC_PURE      4               /* quadric, scj all +0 */
#define QR_DC_SPHERE    5               /* pure, and sci[0..2] all 1 */

/* does a surface side with these properties cast a shadow */
static inline QR_HD int qr_casts_shadow(uint32_t p)
{
    if (p & QR_PROP_LIGHT) return 0;
    if ((p & QR_PROP_TRANSP) && !(p & QR_PROP_REFRACT)) return 0;
    return 1;
}
static inline QR_HD void qr_dev_surf_of(const qr_surface *r, int n_surf, qr_dev_surf *d)
{
    uint32_t f = r->solver >= QR_SOLVE_NONE && r->solver <= QR_SOLVE_QUADRIC
                     ? (uint32_t)r->solver : (uint32_t)QR_DC_TWOPLANE;
    if (f == QR_DC_QUADRIC)
    {
        int pure = 1, unit = 1;
        for (int a = 0; a < 3; a++)
        {
            /* (+0 alone: x - (-0) is not x for x = -0) */
            if (!(r->scj[a] == 0.0f && !__builtin_signbit(r->scj[a]))) pure = 0;
            if (!(r->sci[a] == 1.0f)) unit = 0;
        }
        if (pure) f = unit ? QR_DC_SPHERE : QR_DC_PURE;
    }
    const uint32_t cls = f;
    if (r->shift != 0) f |= QR_DS_SHIFT;
    const uint32_t trm = r->trm == 0 ? 0u : r->trm == 1 ? QR_DI_TRM_DIAG
                                          : r->trm == 2 ? QR_DI_TRM_ROT : QR_DI_TRM;
    if (r->shift != 0 || r->tag < 0) f |= trm * QR_DS_TRM_DIAG;
    if (r->shift == 0 || r->tag < 0) f |= QR_DS_SOLO;
    /* (a plane has no apex, whatever its record says) */
    if (r->apex != 0 && cls != QR_DC_PLANE) f |= QR_DS_APEX;
    if (r->apex == 2) f |= QR_DS_APEX_TWO;
    f |= ((uint32_t)r->cmin_on & 7u) << QR_DS_CMIN_BIT;
    f |= ((uint32_t)r->cmax_on & 7u) << QR_DS_CMAX_BIT;
    if (r->clip_cnt > 0) f |= QR_DS_CLIPS;
    f |= (r->clp_kind == 1 || r->clp_kind == 2 ? (uint32_t)r->clp_kind : 3u) << QR_DS_CLP_BIT;
    f |= (r->nrm_kind == 1 || r->nrm_kind == 2 ? (uint32_t)r->nrm_kind : 3u) << QR_DS_NRM_BIT;
    for (int a = 0; a < 3; a++)
    {
        const uint32_t m = r->amap[a] == 0 ? 0u : r->amap[a] == 1 ? 1u : 2u;
        f |= m << (QR_DS_AMAP_BIT + 2 * a);
        if (r->asgn[a] != 0) f |= 1u << (QR_DS_ASGN_BIT + a);
    }
    for (int k = 0; k < 2; k++)
    {
        if (qr_casts_shadow(r->props[k])) f |= 1u << (QR_DS_SHADOW_BIT + k);
    }
    /* QuadRay gives a surface a nearest-hit list of its own for the rays
     * leaving it when a side reflects or is not opaque
     * (core/engine/engine.cpp:2180-2201) */
    if (((r->props[0] | r->props[1]) & QR_PROP_REFLECT) != 0 ||
        (r->props[0] & r->props[1] & QR_PROP_OPAQUE) == 0)
    {
        f |= QR_DS_OWN_LIST;
    }
    d->flags = f;
    for (int a = 0; a < 3; a++)
    {
        d->pos[a] = r->pos[a];
        d->sci[a] = r->sci[a];
        d->scj[a] = r->scj[a];
        d->td[a] = r->tc[a][a];
        d->cmin[a] = r->cmin[a];
        d->cmax[a] = r->cmax[a];
    }
    d->sci[3] = r->sci[3];
    d->d_eps = r->d_eps;
    d->t_eps = r->t_eps;
    d->to[0] = r->tc[0][1];
    d->to[1] = r->tc[0][2];
    d->to[2] = r->tc[1][0];
    d->to[3] = r->tc[1][2];
    d->to[4] = r->tc[2][0];
    d->to[5] = r->tc[2][1];
    d->clip_beg = r->clip_beg;
    d->clip_cnt = r->clip_cnt;
    d->trnode = r->trnode >= 0 && r->trnode < n_surf ? r->trnode : -1;
    d->info = trm | (r->tag < 0 ? QR_DI_NODE : 0u);
}
static inline QR_HD void qr_dev_box_step(qr_dev_step *d, int skip_index)
{
    d->elem = -1;
    d->skip = QR_DEV_STEP_BYTES * skip_index;
}
static inline QR_HD int qr_dev_box_end(const qr_dev_step *d)
{
    return d->skip / QR_DEV_STEP_BYTES;
}
static inline QR_HD void qr_dev_end_step(qr_dev_step *d)
{
    for (int a = 0; a < 3; a++) d->lo[a] = d->hi[a] = 0.0f;
    d->elem = QR_DEV_STEP_END;
    d->skip = -1;
}
static inline QR_HD void qr_dev_elem_step(qr_dev_step *d, int elem, int surf, int last,
                                          int local)
{
    d->elem = elem;
    d->skip = (int32_t)(surf * (int)sizeof(qr_dev_surf)) | local;
    if (local == QR_LOCAL_NONE)
    {
        for (int a = 0; a < 3; a++) d->lo[a] = d->hi[a] = 0.0f;
        union { int32_t i; float f; } u;
        u.i = last;
        d->lo[0] = u.f;
    }
}
/* the kind of an element step's local box (QR_LOCAL_*) */
static inline QR_HD int qr_dev_step_local(const qr_dev_step *d)
{
    return d->skip & 3;
}
static inline QR_HD int qr_dev_step_surf(const qr_dev_step *d)
{
    return (d->skip & ~3) / (int)sizeof(qr_dev_surf);
}
/* the kind of local box the kernels give a list element whose program step
 * has one (a qr_cull_step with skip -2); groups 0: a program whose group
 * members are not always reached through their node's step (qr_groups_sound)
 * tests no member box */
static inline QR_HD int qr_local_kind(const qr_surface *srf, int surf, int groups)
{
    return srf[surf].trnode == surf ? QR_LOCAL_OWN : groups ? QR_LOCAL_GROUP : QR_LOCAL_NONE;
}
/* the kernels' bounds of an element's local box (centre c, half extents
 * h, about the surface's origin in its tracing frame) */
static inline QR_HD void qr_local_bounds(const qr_surface *srf, int surf, const float *c,
                                         const float *h, float *lo, float *hi)
{
    if (srf[surf].trnode == surf)
    {
        const float zero[3] = {0.0f, 0.0f, 0.0f};
        refit_bounds(c, h, 0, zero, lo, hi);
    }
    else
    {
        refit_bounds_about(c, h, srf[surf].pos, lo, hi);
    }
}

/* device copies of the scene tables (device pointers) */
typedef struct qr_device_tables
{
    qr_surface  *surfaces;
    qr_dev_surf *hot;           /* the surfaces as the walks read them */
    qr_material *materials;
    qr_light    *lights;
    qr_clip     *clips;
    qr_elem     *elems;
    uint32_t    *texels;
    qr_dev_step *steps;         /* nearest-hit culling program (n_step + 1 steps:
                                   the last is the end step) */
    qr_dev_step *steps_any;     /* any-hit culling program (n_step_any + 1) */
    int32_t      n_surf, n_mat, n_lgt, n_clip, n_elem, n_texel, n_step, n_step_any;
    float        cull_ref[4];   /* reference point of the world boxes */
    int32_t      spawns;        /* some surface reflects or transmits: a frame of
                                   a scene where none does has no secondary
                                   rays at any depth */
} qr_device_tables;
/* does a hit on a side with these properties have children (trrf_setup) */
static inline int qr_side_spawns(uint32_t props)
{
    return (props & QR_PROP_REFLECT) != 0 || (props & QR_PROP_OPAQUE) == 0;
}

/* can a ray of the frame have children? */
static inline bool qr_frame_has_tree(const qr_device_tables *t, const qr_frame_desc *fd)
{
    return t->spawns != 0 && fd->depth > 0;
}

/* hot[i] from srf[i] for every record, on the device */
hipError_t qr_dev_surfaces(const qr_surface *srf, int n, qr_dev_surf *hot, hipStream_t stream);

/* the device update stage's records (update.hip): every record of the
 * surface table with its form for the walks (hot), the planes' texture transforms in mat, and the surface
 * list's element inputs of the culling programs, from the records' inputs
 * (fields.h); clips is the table's clip list; expect holds per element the
 * world and local flags the programs were built for, and an element that
 * differs sets *mismatch */
struct qr_geom;
hipError_t qr_update_records(const struct qr_geom *geoms, int n_rec, const qr_clip *clips,
                             qr_surface *srf, qr_dev_surf *hot, qr_material *mat,
                             struct qr_refit_elem *refit_in, const int32_t *expect, uint32_t *mismatch, hipStream_t stream);

/* the device update stage's refit (update.hip): both programs' boxes (lo/hi
 * of every box step and of every element step with a local box) from the
 * element inputs and the surface records (srf: a member's position in its
 * group's frame), ranges and elements unchanged (n_step and n_step_any do
 * not count the end steps, which stay as they are); scratch holds 8 floats
 * per element; steps_any may be null when n_step_any is 0 */
hipError_t qr_refit_programs(qr_dev_step *steps, int n_step, qr_dev_step *steps_any,
                             int n_step_any, const qr_refit_elem *elems, int n_elem,
                             const qr_surface *srf, const float ref[4], float *scratch,
                             hipStream_t stream);

/* Whitted frame: ARGB8 into frame (row y at frame + y * fd->x_row), and the
 * first-hit id of every sample into ids when ids is not null */
hipError_t qr_launch_whitted(const qr_device_tables *t, const qr_frame_desc *fd,
                             uint32_t *frame, int32_t *ids, hipStream_t stream);

/* the path tracer (tracer_pt.hip), traced as a wavefront: queues of one
 * user (a scene, a server step, a device), reused by every launch */
typedef struct qr_pt_state qr_pt_state;
hipError_t qr_pt_create(qr_pt_state **out);
void       qr_pt_destroy(qr_pt_state *s);
/* a path-traced frame's start: cleared planes (3 x slots floats) and the
 * initial seed plane of a frame of x_res x y_res with rows of |x_row| pixels,
 * in the slot order below (at most 2^32 - 1 slots) */
hipError_t qr_pt_start(float *planes, uint32_t *seeds, int x_res, int y_res, int x_row,
                       int fsaa, hipStream_t stream);
/* "passes" passes over the chunk of 8x8-pixel tiles tile0 .. tile0 +
 * ntiles - 1 (ntiles 0: all), fd->pts_c counting the first: planes (red,
 * green, blue running means, 3 x slots floats) and seeds (one per slot),
 * slot = (y * x_res + x) * samples + k, are updated, and the chunk's pixels
 * resolved into frame (pitch fd->x_res) */
hipError_t qr_pt_launch(qr_pt_state *s, const qr_device_tables *t, const qr_frame_desc *fd,
                        float *planes, uint32_t *seeds, uint32_t *frame, uint32_t tile0,
                        uint32_t ntiles, int passes, hipStream_t stream);
/* after the stream finished a launch: 0 if it is complete, 1 if its last
 * run of passes overflowed a queue (it wrote nothing; the queues are grown:
 * call qr_pt_retry, then check again) */
int        qr_pt_check(qr_pt_state *s);
hipError_t qr_pt_retry(qr_pt_state *s, hipStream_t stream);
uint32_t   qr_pt_tiles(int x_res, int y_res);
/* device memory of a state's queues for runs of up to "samples" samples
 * (slots times passes; an overflowed queue grows beyond it) */
uint64_t   qr_pt_run_bytes(uint64_t samples);

/* level-by-level pipeline (tracer_wf.hip): queues and counters of one
 * device, reused by every frame traced with it */
typedef struct qr_wf_state qr_wf_state;

typedef struct qr_wf_stats
{
    uint32_t level_rays[16];    /* rays queued per tree level (level 0: 0) */
} qr_wf_stats;

/* most lights the pipeline handles (visibility mask bits) */
int        qr_wf_max_lights(void);
hipError_t qr_wf_create(qr_wf_state **out);
void       qr_wf_destroy(qr_wf_state *s);
/* enqueue one Whitted frame on "stream" (frame pitch fd->x_res) */
hipError_t qr_wf_launch(qr_wf_state *s, const qr_device_tables *t,
                        const qr_frame_desc *fd, uint32_t *frame, int32_t *ids,
                        hipStream_t stream);
/* after the stream finished the frame: 0 if it is complete, 1 if a queue
 * overflowed (queues are grown; trace the frame again) */
int        qr_wf_check(qr_wf_state *s, qr_wf_stats *stats);
/* the frame launched last went another way: there is nothing to check */
void       qr_wf_skip(qr_wf_state *s);

/* Batches: many frames, each with its own queues (state), tables, camera,
 * resolution, anti-aliasing and depth, traced by one launch per stage.  The
 * launches depend only on the number of frames and the deepest depth, so a
 * batch's launch sequence can be captured in a HIP graph once its frame
 * arguments are on the device (they are uploaded when they change). */
#define QR_WF_MAX_BATCH 65536
typedef struct qr_wf_batch qr_wf_batch;
typedef struct qr_wf_item
{
    qr_wf_state              *s;        /* the frame's queues */
    const qr_device_tables   *t;
    const qr_frame_desc      *fd;
    uint32_t                 *frame;    /* device, pitch fd->x_res */
    int32_t                  *ids;      /* device first-hit ids or null */
    uint32_t                  tile0;    /* a chunk of the frame: level-0 tiles */
    uint32_t                  ntiles;   /* tile0 .. tile0 + ntiles - 1; 0: all */
} qr_wf_item;

hipError_t qr_wf_batch_create(qr_wf_batch **out);
/* second streams made so far (one per device at most, shared by batches) */
int        qr_wf_side_streams(void);
void       qr_wf_batch_destroy(qr_wf_batch *b);
/* launch shape: persistent workgroups per compute unit (1..64), level-0
 * tile width in pixels (4, 8, 16 or 32; tiles hold 64 pixels), rays per
 * thread (1..QR_WF_MAX_RPT: blocks of 256 queue entries a virtual workgroup
 * takes) and compaction cadence (1..QR_WF_MAX_CADENCE: children are
 * compacted into the queue of level L only when L is a multiple of it) */
#define QR_WF_MAX_RPT 8
#define QR_WF_MAX_CADENCE 4
hipError_t qr_wf_batch_config(qr_wf_batch *b, int grid_per_cu, int tile_w, int rpt,
                              int cadence);
/* level-0 tiles of an x_res x y_res frame under the batch's tile shape */
uint32_t   qr_wf_batch_tiles(const qr_wf_batch *b, int x_res, int y_res);
hipError_t qr_wf_batch_launch(qr_wf_batch *b, const qr_wf_item *items, int n,
                              hipStream_t stream);
/* after the stream finished the batch: 1 if a frame's queue overflowed (its
 * queues are grown; trace the batch again), else 0 */
int        qr_wf_batch_check(qr_wf_batch *b, const qr_wf_item *items, int n);
void       qr_wf_batch_stats(const qr_wf_batch *b, int k, qr_wf_stats *stats);

#endif /* QR_TRACER_KERNELS_H */
