/*
 * serve_faults.cpp -- the serving loop on host memory: whichever runtime call
 * of a request fails, later requests of any scene return their own frames
 * (a slot whose upload failed holds no scene's tables).
 */
#include <cstdio>
#include <vector>

#include "kernels_host.h"
#include "scenegen.hpp"

constexpr int X = 40, Y = 24;

/* a request's status, its frame compared with the scene's own */
static int ask(qrhip_server *srv, int scene, qrhip_scene *s, bool *right)
{
    std::vector<uint32_t> frame((size_t)X * Y, 0u);
    qrhip_request r;
    memset(&r, 0, sizeof(r));
    r.tag = 1;
    r.scene = scene;
    r.x_res = X;
    r.y_res = Y;
    r.depth = 2;
    r.frame = frame.data();
    if (qrhip_server_submit(srv, &r) != 0) exit(2);
    qrhip_result res;
    while (qrhip_server_poll(srv, &res, 1, 1000) == 0) {}
    *right = true;
    const uint32_t h = table_hash(&s->dt.t);
    for (int y = 0; y < Y; y++)
    {
        for (int x = 0; x < X; x++) *right &= frame[(size_t)y * X + x] == pixel(h, x, y);
    }
    return res.status;
}

int main()
{
    int failed = 0, bad = 0;
    for (long n = 0;; n++)
    {
        hip_fail_at(-1);
        qrhip_dev *dev = nullptr;
        if (qrhip_device_open(0, &dev) != 0) return 3;
        qrgen::Scene *sc[2];
        qrhip_scene *scene[2];
        for (int k = 0; k < 2; k++)
        {
            sc[k] = qrgen::build(k == 0 ? 2 : 8, 90 + k);
            if (qrhip_scene_create(dev, &sc[k]->root, X, Y, X, nullptr, &scene[k]) != 0 ||
                qrhip_scene_update(scene[k], 0) != 0)
            {
                return 4;
            }
        }
        qrhip_server *srv = nullptr;
        if (qrhip_server_create(dev, scene, 2, 1ull << 32, 1, 0, &srv) != 0) return 5;
        bool right;
        if (ask(srv, 0, scene[0], &right) != 0 || !right) return 6;
        hip_fail_at(n);
        const int rc = ask(srv, 1, scene[1], &right);
        const bool reached = hip_calls > n;
        hip_fail_at(-1);
        if (rc == 0 && !right) return 7;
        failed += rc != 0;
        for (int k : {0, 1, 0})
        {
            if (ask(srv, k, scene[k], &right) == 0 && right) continue;
            printf("after call %ld failed: scene %d has another frame\n", n, k);
            bad++;
        }
        (void)qrhip_server_destroy(srv);
        for (int k = 0; k < 2; k++)
        {
            qrhip_scene_destroy(scene[k]);
            delete sc[k];
        }
        qrhip_device_close(dev);
        if (!reached) break;
    }
    printf("%d failing requests, %d wrong frames\n", failed, bad);
    return bad != 0 || failed < 10;
}
