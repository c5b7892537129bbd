// Drives the library's host code over the CPU stand-in of host_hip.cpp.
//   host_calls_check NAME [FILE]     runs one check; prints "ok"
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

#include "../../include/sister.h"
#include "host_hip.h"

#define CHECK(c)                                                   \
    do {                                                           \
        if (!(c)) {                                                \
            std::printf("FAIL %s line %d\n", #c, __LINE__);        \
            std::fflush(stdout);                                   \
            std::_Exit(1);                                         \
        }                                                          \
    } while (0)

namespace {

// a rig in host memory with views of `seed`, and its outputs
struct Rig {
    int W, H, D;
    std::vector<uint8_t> view[5];
    std::vector<uint16_t> out[3], disp;
    std::vector<float> sub;
    std::vector<uint16_t> want[4];   // the stand-in's maps, and its integer map
    std::vector<float> want_sub;
    sister_rig r;
    Rig(int w, int h, int d, unsigned seed) : W(w), H(h), D(d)
    {
        std::memset(&r, 0, sizeof r);
        r.width = W; r.height = H; r.stride = W; r.disp_count = D;
        for (int i = 0; i < 5; i++) {
            view[i].resize((size_t)W * H);
            for (auto& b : view[i]) b = (uint8_t)((seed = seed * 1664525u + 1013904223u) >> 24);
            r.view[i] = view[i].data();
        }
        for (int p = 0; p < W * H; p++) {
            int v = 0;
            for (int i = 0; i < 5; i++) v += (i + 1) * view[i][p];
            for (int m = 0; m < 3; m++) want[m].push_back((uint16_t)host_hip::map_value(v, m));
            want[3].push_back((uint16_t)v);
            want_sub.push_back((float)v);
        }
        for (auto& o : out) o.resize((size_t)W * H);
        disp.resize((size_t)W * H);
        sub.resize((size_t)W * H);
        r.out_multiview = out[0].data();
        r.out_horizontal = out[1].data();
        r.out_vertical = out[2].data();
        r.out_disp = disp.data();
        r.out_subpix = sub.data();
    }
    void clear()
    {
        for (auto& o : out) std::fill(o.begin(), o.end(), 0xFFFF);
        std::fill(disp.begin(), disp.end(), 0xFFFF);
        std::fill(sub.begin(), sub.end(), -1.f);
    }
    bool right(int modes) const
    {
        for (int m = 0; m < 3; m++)
            if ((modes >> m & 1) && out[m] != want[m]) return false;
        return !(modes & 1) || (disp == want[3] && sub == want_sub);
    }
};

sister_ctx* create(size_t budget = 0)
{
    sister_config cfg{0, 0, budget};
    sister_ctx* c = nullptr;
    CHECK(sister_create(&cfg, &c) == SISTER_OK);
    return c;
}

// Threads that compute rigs of different sizes (one copy for all views, a copy
// per view, a staging that has to grow) on one context, as callers of the class
// with its shared context do: each gets its own maps.
void host_form_threads()
{
    host_hip::step_us = 100;
    sister_ctx* c = create();
    const int dims[3][3] = {{64, 48, 16}, {640, 480, 64}, {320, 240, 32}};
    std::vector<std::thread> th;
    for (int k = 0; k < 3; k++)
        th.emplace_back([=] {
            Rig r(dims[k][0], dims[k][1], dims[k][2], 10u + k);
            const int modes = k == 2 ? 1 : 7;
            for (int i = 0; i < 12; i++) {
                r.clear();
                CHECK(sister_compute_rig(c, &r.r, modes) == SISTER_OK);
                CHECK(r.right(modes));
            }
        });
    for (auto& t : th) t.join();
    sister_destroy(c);
    CHECK(host_hip::pinned_bytes == 0);
}

// A thread that computes rigs from host memory beside one that runs batches on
// the same context: neither call may take the plan of the other's work while
// that work runs.  Equal sizes: a plan built too early has its launch tables
// in the other's place.
void host_form_beside_batches()
{
    host_hip::step_us = 30;
    sister_ctx* c = create();
    std::thread host([=] {
        Rig r(1024, 512, 8, 3);
        for (int i = 0; i < 600; i++) {
            r.clear();
            CHECK(sister_compute_rig(c, &r.r, 1) == SISTER_OK);
            CHECK(r.right(1));
        }
    });
    Rig r(1024, 512, 8, 4);
    for (int i = 0; i < 600; i++) {
        r.clear();
        CHECK(sister_run_device(c, &r.r, 1, 1) == SISTER_OK);
        CHECK(sister_sync(c) == SISTER_OK);
        CHECK(r.right(1));
    }
    host.join();
    sister_destroy(c);
}

// A rig whose staging is too large to keep and whose device block cannot be
// had: refused, and nothing pinned stays behind.
void host_form_refused()
{
    sister_ctx* c = create((size_t)64 << 20);
    Rig r(4096, 4096, 8, 5);
    CHECK(sister_compute_rig(c, &r.r, 1) == SISTER_ENOMEM);
    CHECK(host_hip::pinned_bytes == 0);
    Rig s(64, 48, 16, 6);
    CHECK(sister_compute_rig(c, &s.r, 7) == SISTER_OK && s.right(7));
    sister_destroy(c);
    CHECK(host_hip::pinned_bytes == 0);
}

int octave(double v) { return (int)std::floor(std::log2(v) * 2.0); }   // the forms file's half octaves
double cells(const sister_rig& r)
{
    return (double)(r.width + 2 * r.disp_count) * (r.height + 2 * r.disp_count) * r.disp_count;
}

// sister_autotune captures a batch once, in the forms of a file; a batch with a
// shape that no file names is refused before anything is captured.
void forms_capture_once(const char* path)
{
    sister_ctx* c = create();
    std::vector<Rig> rigs;
    for (int k = 0; k < 4; k++) rigs.emplace_back(64 + 16 * k, 48, 8 * (k + 1), 30u + k);
    std::vector<sister_rig> batch;
    double total = 0;
    for (Rig& r : rigs) {
        batch.push_back(r.r);
        total += cells(r.r);
    }
    CHECK(sister_graph_capture(c, batch.data(), 4, 1) == SISTER_OK);
    CHECK(sister_autotune(c, batch.data(), 4, 1, nullptr) == SISTER_EINVAL);
    CHECK(sister_autotune(c, batch.data(), 4, 1, path) == SISTER_EINVAL);
    FILE* fp = std::fopen(path, "r");
    CHECK(!fp);   // refused: no file is written
    fp = std::fopen(path, "w");
    std::fprintf(fp, "batch 4 4 %d 1 parts 2 by_d 0 stagger 0\n", octave(total));
    for (Rig& r : rigs)
        std::fprintf(fp, "group %d %d %d fused 0 kl 0 0 0 0 msum_split 0\n", r.D, octave(r.W + 2 * r.D), octave(r.H + 2 * r.D));
    std::fclose(fp);
    CHECK(host_hip::captures == 1);
    // the first capture is still there
    for (Rig& r : rigs) r.clear();
    CHECK(sister_graph_launch(c) == SISTER_OK && sister_sync(c) == SISTER_OK);
    for (Rig& r : rigs) CHECK(r.right(1));
    CHECK(sister_autotune(c, batch.data(), 4, 1, path) == SISTER_OK);
    CHECK(host_hip::captures == 2);
    for (int i = 0; i < 3; i++) {
        for (Rig& r : rigs) r.clear();
        CHECK(sister_graph_launch(c) == SISTER_OK && sister_sync(c) == SISTER_OK);
        for (Rig& r : rigs) CHECK(r.right(1));
    }
    // one more disparity count: not in the table
    rigs.emplace_back(64, 48, 64, 40u);
    batch.push_back(rigs.back().r);
    CHECK(sister_autotune(c, batch.data(), 5, 1, path) == SISTER_EINVAL);
    CHECK(host_hip::captures == 2);
    sister_destroy(c);
}

// Graph branches: as many as a form asks for, at most four.
void graph_branches(const char* path)
{
    std::vector<Rig> rigs;
    for (int k = 0; k < 9; k++) rigs.emplace_back(64, 48, 8 * (k % 6 + 1), 50u + k);
    std::vector<sister_rig> batch;
    double total = 0;
    for (Rig& r : rigs) {
        batch.push_back(r.r);
        total += cells(r.r);
    }
    const struct { int n, parts, by_d, want; } cases[] = {{9, 1, 0, 1}, {9, 3, 0, 3}, {9, 4, 0, 4}, {9, 5, 0, 4}, {9, 8, 0, 4}, {9, 0, 1, 4}};
    for (const auto& q : cases) {
        sister_ctx* c = create();
        FILE* fp = std::fopen(path, "w");
        std::fprintf(fp, "batch %d 6 %d 1 parts %d by_d %d stagger 0\n", q.n, octave(total), q.parts, q.by_d);
        // every split of the nine rigs: one or two of a disparity count in a part
        for (int d = 8; d <= 48; d += 8)
            for (int m = 1; m <= 2; m++)
                std::fprintf(fp, "group %d %d %d fused 0 kl 0 0 0 0 msum_split 0\n", d, octave(m * (64 + 2 * d)), octave(48 + 2 * d));
        std::fclose(fp);
        host_hip::branches = 0;
        CHECK(sister_autotune(c, batch.data(), q.n, 1, path) == SISTER_OK);
        CHECK(host_hip::branches == q.want);
        for (Rig& r : rigs) r.clear();
        CHECK(sister_graph_launch(c) == SISTER_OK && sister_sync(c) == SISTER_OK);
        for (Rig& r : rigs) CHECK(r.right(1));
        sister_destroy(c);
    }
}

}  // namespace

int main(int argc, char** argv)
{
    const std::string name = argc > 1 ? argv[1] : "";
    if (name == "host_form_threads") host_form_threads();
    else if (name == "host_form_beside_batches") host_form_beside_batches();
    else if (name == "host_form_refused") host_form_refused();
    else if (name == "forms_capture_once") forms_capture_once(argv[2]);
    else if (name == "graph_branches") graph_branches(argv[2]);
    else return 2;
    std::printf("ok\n");
    return 0;
}
