/*
 * kernels_host.h -- stand-ins for the library's kernels (tracer_kernels.h) on
 * host memory, for tests of the host code around them: a traced pixel is a
 * hash of the surface table its launch was given and of its place.
 */
#ifndef KERNELS_HOST_H
#define KERNELS_HOST_H

#include "hip_host.h"
#include "capi_internal.h"

static uint32_t table_hash(const qr_device_tables *t)
{
    uint32_t h = 2166136261u;
    const uint8_t *p = (const uint8_t *)t->surfaces;
    for (size_t i = 0; i < sizeof(qr_surface) * (size_t)t->n_surf; i++) h = (h ^ p[i]) * 16777619u;
    return h;
}
static uint32_t pixel(uint32_t hash, int x, int y)
{
    return (hash ^ ((uint32_t)y * 40503u + (uint32_t)x)) * 2654435761u;
}
static hipError_t trace(const qr_device_tables *t, const qr_frame_desc *fd, uint32_t *frame)
{
    if (hip_step() != hipSuccess) return hipErrorUnknown;
    const uint32_t h = table_hash(t);
    for (int y = 0; y < fd->y_res; y++)
    {
        for (int x = 0; x < fd->x_res; x++) frame[(size_t)y * fd->x_res + x] = pixel(h, x, y);
    }
    return hipSuccess;
}

hipError_t qr_dev_surfaces(const qr_surface *srf, int n, qr_dev_surf *hot, hipStream_t)
{
    if (hip_step() != hipSuccess) return hipErrorUnknown;
    for (int i = 0; i < n; i++) qr_dev_surf_of(&srf[i], n, &hot[i]);
    return hipSuccess;
}
hipError_t qr_update_records(const qr_geom *, int, const qr_clip *, qr_surface *, qr_dev_surf *,
                             qr_material *, qr_refit_elem *, const int32_t *, uint32_t *mismatch,
                             hipStream_t)
{
    *mismatch = 1u;                 /* to the host */
    return hip_step();
}
hipError_t qr_refit_programs(qr_dev_step *, int, qr_dev_step *, int, const qr_refit_elem *, int,
                             const qr_surface *, const float *, float *, hipStream_t)
{
    return hip_step();
}
hipError_t qr_launch_whitted(const qr_device_tables *t, const qr_frame_desc *fd, uint32_t *frame,
                             int32_t *, hipStream_t)
{
    return trace(t, fd, frame);
}

struct qr_wf_state { int unused; };
struct qr_wf_batch { int unused; };
struct qr_pt_state { int unused; };
int qr_wf_max_lights(void) { return 32; }
int qr_wf_side_streams(void) { return 0; }
hipError_t qr_wf_create(qr_wf_state **s) { *s = new qr_wf_state(); return hip_step(); }
void qr_wf_destroy(qr_wf_state *s) { delete s; }
hipError_t qr_wf_launch(qr_wf_state *, const qr_device_tables *t, const qr_frame_desc *fd,
                        uint32_t *frame, int32_t *, hipStream_t)
{
    return trace(t, fd, frame);
}
int qr_wf_check(qr_wf_state *, qr_wf_stats *) { return 0; }
void qr_wf_skip(qr_wf_state *) {}
hipError_t qr_wf_batch_create(qr_wf_batch **b) { *b = new qr_wf_batch(); return hip_step(); }
void qr_wf_batch_destroy(qr_wf_batch *b) { delete b; }
hipError_t qr_wf_batch_config(qr_wf_batch *, int, int, int, int) { return hipSuccess; }
uint32_t qr_wf_batch_tiles(const qr_wf_batch *, int x_res, int y_res)
{
    return (uint32_t)((x_res + 7) / 8) * (uint32_t)((y_res + 7) / 8);
}
hipError_t qr_wf_batch_launch(qr_wf_batch *, const qr_wf_item *items, int n, hipStream_t)
{
    for (int k = 0; k < n; k++)
    {
        const hipError_t e = trace(items[k].t, items[k].fd, items[k].frame);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
int qr_wf_batch_check(qr_wf_batch *, const qr_wf_item *, int) { return 0; }
hipError_t qr_pt_create(qr_pt_state **s) { *s = new qr_pt_state(); return hip_step(); }
void qr_pt_destroy(qr_pt_state *s) { delete s; }
hipError_t qr_pt_start(float *, uint32_t *, int, int, int, int, hipStream_t) { return hip_step(); }
hipError_t qr_pt_launch(qr_pt_state *, const qr_device_tables *t, const qr_frame_desc *fd, float *,
                        uint32_t *, uint32_t *frame, uint32_t, uint32_t, int, hipStream_t)
{
    return trace(t, fd, frame);
}
int qr_pt_check(qr_pt_state *) { return 0; }
hipError_t qr_pt_retry(qr_pt_state *, hipStream_t) { return hipSuccess; }
uint32_t qr_pt_tiles(int x_res, int y_res) { return qr_wf_batch_tiles(nullptr, x_res, y_res); }
uint64_t qr_pt_run_bytes(uint64_t samples) { return samples; }

namespace qrhip_impl {
hipError_t noalloc_setup(int) { return hipSuccess; }
}

#endif /* KERNELS_HOST_H */
