/*
 * batch_download.cpp -- qrhip_batch_download on host memory: frames that
 * share a buffer, wholly or in part, leave what downloads one after another
 * in request order would ("shared"); and whichever allocation or runtime call
 * of a download fails, it returns an error or the frames, and the next one
 * returns the frames ("faults").
 */
#include <cstdio>
#include <new>
#include <string>
#include <vector>

#include "kernels_host.h"
#include "scenegen.hpp"

static std::atomic<long> news{0}, new_fail_on{-1};

void *operator new(size_t n)
{
    if (new_fail_on >= 0 && news++ == new_fail_on) throw std::bad_alloc();
    void *p = malloc(n != 0 ? n : 1);
    if (p == nullptr) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

struct Size
{
    int    x, y;
    size_t at;                      /* its frame's place in the callers' memory */
};

struct Batch
{
    qrgen::Scene                *sc[2];
    qrhip_dev                   *dev = nullptr;
    qrhip_scene                 *scene[2] = {};
    qrhip_batch                 *b = nullptr;
    std::vector<uint32_t>        mem, want;
    std::vector<qrhip_frame_req> req;

    Batch(const std::vector<Size> &sizes, size_t words) : mem(words), want(words)
    {
        if (qrhip_device_open(0, &dev) != 0 || qrhip_batch_create(dev, &b) != 0) exit(2);
        for (int k = 0; k < 2; k++)
        {
            sc[k] = qrgen::build(1, 70 + k);
            if (qrhip_scene_create(dev, &sc[k]->root, 64, 64, 64, nullptr, &scene[k]) != 0 ||
                qrhip_scene_update(scene[k], 0) != 0)
            {
                exit(3);
            }
        }
        for (size_t k = 0; k < sizes.size(); k++)
        {
            const Size &z = sizes[k];
            req.push_back(qrhip_frame_req{scene[k & 1], z.x, z.y, 0, 1, mem.data() + z.at});
        }
        if (qrhip_batch_set(b, req.data(), (int)req.size()) != 0 ||
            qrhip_batch_launch(b, QRHIP_BATCH_DIRECT) != 0 || qrhip_batch_sync(b) != 0)
        {
            exit(4);
        }
        for (size_t k = 0; k < sizes.size(); k++)
        {
            const uint32_t h = table_hash(&scene[k & 1]->dt.t);
            for (int y = 0; y < sizes[k].y; y++)
            {
                for (int x = 0; x < sizes[k].x; x++)
                {
                    want[sizes[k].at + (size_t)y * sizes[k].x + x] = pixel(h, x, y);
                }
            }
        }
    }
    ~Batch()
    {
        qrhip_batch_destroy(b);
        for (int k = 0; k < 2; k++)
        {
            qrhip_scene_destroy(scene[k]);
            delete sc[k];
        }
        qrhip_device_close(dev);
    }
    int download()
    {
        std::fill(mem.begin(), mem.end(), 0u);
        return qrhip_batch_download(b, -1);
    }
};

int main(int argc, char **argv)
{
    const std::string mode = argc > 1 ? argv[1] : "";
    if (mode == "shared")
    {
        /* one buffer for all, of frames many of which are copied side by
         * side; frames that overlap in part, in and out of order; and frames
         * that only touch */
        std::vector<std::vector<Size>> cases(4);
        for (int k = 0; k < 60; k++)
        {
            cases[0].push_back({256, 256, 0});
            cases[1].push_back({200 + k, 300 - k, (size_t)k * 3000});
            cases[2].push_back({256, 256, (size_t)(59 - k) * 20000});
            cases[3].push_back({256, 256, (size_t)(k * 7 % 60) * 65536});
        }
        int bad = 0;
        for (size_t c = 0; c < cases.size(); c++)
        {
            Batch b(cases[c], 4u << 20);
            for (int rep = 0; rep < 20; rep++)
            {
                if (b.download() != 0) return 5;
                if (b.mem != b.want)
                {
                    printf("case %d run %d differs\n", (int)c, rep);
                    bad++;
                    break;
                }
            }
        }
        return bad != 0;
    }
    /* faults */
    const std::vector<Size> sizes = {{1024, 1024, 0}, {1500, 1000, 1u << 20}, {33, 17, 3u << 20}};
    int failed = 0;
    for (int what = 0; what < 2; what++)
    {
        for (long n = 0;; n++)
        {
            Batch b(sizes, 4u << 20);
            news = 0;
            if (what == 0) hip_fail_at(n);
            else new_fail_on = n;
            const int rc = b.download();
            hip_fail_at(-1);
            new_fail_on = -1;
            if (rc == 0 && b.mem != b.want)
            {
                printf("%s %ld: wrong frames\n", what == 0 ? "call" : "allocation", n);
                return 6;
            }
            if (b.download() != 0 || b.mem != b.want)
            {
                printf("%s %ld: wrong frames afterwards\n", what == 0 ? "call" : "allocation", n);
                return 7;
            }
            failed += rc != 0;
            const long reached = what == 0 ? (long)hip_calls : (long)news;
            if (rc == 0 && (what == 0 || reached <= n)) break;
        }
    }
    printf("%d failing downloads\n", failed);
    return failed < 10;
}
