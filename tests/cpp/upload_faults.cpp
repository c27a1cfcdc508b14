/*
 * upload_faults.cpp -- DevTables (capi_internal.h) when a runtime call of an
 * upload fails: whatever call it was, the next upload of the same tables, of
 * other ones, or after a device update leaves every device table as a fresh
 * upload would, the walks' form of the surfaces and the programs included.
 * Host memory stands for the device's.
 */
#include <cstdio>

#include "hip_host.h"
#include "capi_internal.h"
#include "scenegen.hpp"

using namespace qrhip_impl;

hipError_t qr_dev_surfaces(const qr_surface *srf, int n, qr_dev_surf *hot, hipStream_t)
{
    if (hip_step() != hipSuccess) return hipErrorUnknown;
    for (int i = 0; i < n; i++) qr_dev_surf_of(&srf[i], n, &hot[i]);
    return hipSuccess;
}
/* the device update stage: records and boxes the host has no copy of */
hipError_t qr_update_records(const qr_geom *, int n_rec, const qr_clip *, qr_surface *srf,
                             qr_dev_surf *hot, qr_material *, qr_refit_elem *, const int32_t *,
                             uint32_t *, hipStream_t)
{
    if (hip_step() != hipSuccess) return hipErrorUnknown;
    memset((void *)srf, 0x5A, sizeof(qr_surface) * (size_t)n_rec);
    memset((void *)hot, 0x5A, sizeof(qr_dev_surf) * (size_t)n_rec);
    return hipSuccess;
}
hipError_t qr_refit_programs(qr_dev_step *prog0, int n0, qr_dev_step *prog1, int n1,
                             const qr_refit_elem *, int, const qr_surface *, const float *,
                             float *, hipStream_t)
{
    if (hip_step() != hipSuccess) return hipErrorUnknown;
    for (int k = 0; k < n0; k++) prog0[k].lo[0] = 1.0f;
    for (int k = 0; k < n1; k++) prog1[k].lo[0] = 1.0f;
    return hipSuccess;
}

static int bad = 0;

template <class T>
static void same(const char *what, const void *got, const T *want, int n, long call)
{
    if (n == 0 || (got != nullptr && memcmp(got, want, sizeof(T) * (size_t)n) == 0)) return;
    printf("%s: stale after call %ld failed\n", what, call);
    bad++;
}

/* the device's tables against the host's ("refitted": the device has put
 * boxes of its own into the programs) */
static void check(const DevTables &dt, const qr_scene_tables &h, const float *ref, bool refitted,
                  long call)
{
    std::vector<qr_dev_surf> hot((size_t)h.n_surf);
    for (int i = 0; i < h.n_surf; i++) qr_dev_surf_of(&h.surfaces[i], h.n_surf, &hot[(size_t)i]);
    same("surfaces", dt.t.surfaces, h.surfaces, h.n_surf, call);
    same("walk surfaces", dt.t.hot, hot.data(), h.n_surf, call);
    same("materials", dt.t.materials, h.materials, h.n_mat, call);
    same("lights", dt.t.lights, h.lights, h.n_lgt, call);
    same("clips", dt.t.clips, h.clips, h.n_clip, call);
    same("elements", dt.t.elems, h.elems, h.n_elem, call);
    same("texels", dt.t.texels, h.texels, h.n_texel, call);
    if (dt.t.n_surf != h.n_surf || dt.t.n_step != h.n_step || dt.t.n_step_any != h.n_step_any)
    {
        printf("counts after call %ld failed\n", call);
        bad++;
    }
    for (int k = 0; k < 2; k++)
    {
        const int n = k == 0 ? h.n_step : h.n_step_any;
        std::vector<qr_dev_step> want;
        dev_steps(k == 0 ? h.steps : h.steps_any, n, ref, h.elems, h.surfaces, want);
        const qr_dev_step *got = k == 0 ? dt.t.steps : dt.t.steps_any;
        if (!refitted)
        {
            same(k == 0 ? "program" : "any-hit program", got, want.data(), n + 1, call);
            continue;
        }
        /* (the boxes are the device's own) */
        for (int p = 0; p <= n; p++)
        {
            const qr_dev_step &w = want[(size_t)p];
            if (got[p].elem == w.elem && got[p].skip == w.skip) continue;
            printf("program %d: stale after call %ld failed\n", k, call);
            bad++;
            break;
        }
    }
}

static hipError_t upload(DevTables &dt, const qr::Engine &eng)
{
    const ProgramInputs in = program_inputs(eng);
    return dt.upload(eng.tables(), nullptr, &in);
}

int main()
{
    qrgen::Scene *sa = qrgen::build(8, 41), *sb = qrgen::build(7, 42);
    qrgen::animate(*sa);
    long calls = 0;
    int tries = 0;
    /* what the device holds before the call that fails, which is an upload
     * of the scene or a device update of it, and whether the scene has moved
     * on (a refit) by the next upload */
    enum { NOTHING, SCENE, OTHER };
    const struct { int first, update, moved; } modes[] = {
        {NOTHING, 0, 0}, {NOTHING, 0, 1}, {SCENE, 0, 0}, {SCENE, 0, 1},
        {SCENE, 1, 0}, {SCENE, 1, 1}, {OTHER, 0, 0}, {OTHER, 0, 1}};
    for (const auto &m : modes)
    {
        for (long call = 0;; call++)
        {
            qr::Engine a(&sa->root, 64, 64, 64), b(&sb->root, 64, 64, 64);
            a.update(0);
            b.update(0);
            DevTables dt;
            memset((void *)&dt.t, 0, sizeof(dt.t));
            hip_fail_at(-1);
            if (m.first != NOTHING && upload(dt, m.first == SCENE ? a : b) != hipSuccess) return 2;
            if (m.first == OTHER) dt.build_on_dev = 0;
            if (m.first == SCENE) a.update(40);       /* records move: a refit */
            hip_fail_at(call);
            hipError_t e;
            if (m.update)
            {
                bool ok = false;
                if (!dt.holds_build(a) || !a.update_transforms(80)) return 3;
                e = dt.update_device(a, nullptr, &ok);
            }
            else
            {
                e = upload(dt, a);
            }
            const bool failed = e != hipSuccess;
            calls += hip_calls;
            hip_fail_at(-1);
            if (failed)
            {
                tries++;
                /* the same tables again, then the other scene's */
                a.materialize();
                if (m.moved) a.update(120);
                const int was = dt.refits;
                if (upload(dt, a) != hipSuccess) return 4;
                check(dt, a.tables(), dt.t.cull_ref, dt.refits > was, call);
                const int was_b = dt.refits;
                dt.build_on_dev = 0;
                if (upload(dt, b) != hipSuccess) return 5;
                check(dt, b.tables(), dt.t.cull_ref, dt.refits > was_b, call);
            }
            dt.release();
            if (!failed) break;
        }
    }
    printf("%d failing calls, %ld calls, %d stale tables\n", tries, calls, bad);
    return bad != 0 || tries < 20 ? 1 : 0;
}
