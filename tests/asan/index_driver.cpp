// Host UndefinedBehaviorSanitizer run of the delay-and-sum kernels' own index arithmetic
// (ffdas_amd/csrc/das_index.h).  Exit status 0 and no sanitizer report is the pass condition.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "das_index.h"

using namespace ffdas::dev;

#define CHECK(c)                                                       \
    do {                                                               \
        if (!(c)) {                                                    \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);        \
            std::exit(1);                                              \
        }                                                              \
    } while (0)

// Every scalar offset of a round of slots stays inside the channel's block of K transmits.
static long slots() {
    long n = 0;
    for (int KC : {8, 16})
        for (int TB : {1, 2, 4})
            for (int K = 1; K <= 40; K++)
                for (int kc = 0; kc < K; kc += KC)
                    for (int j0 = 0; j0 < KC && kc + j0 < K; j0 += TB)
                        for (int u = 0; u < TB; u++) {
                            const int step = 1 << 20, j = kc + j0 + u;
                            const int at = slot_offset(j, K, step);
                            CHECK(at >= 0 && at <= (K - 1) * step);
                            CHECK(j >= K || at == j * step);
                            n++;
                        }
    return n;
}

// Every voxel is in exactly one tile of the shape the kernels choose, within the tiles launched.
static long tiles() {
    long n = 0;
    const int grids[][3] = {{2, 2, 2}, {9, 5, 7}, {3, 17, 2}, {2, 3, 33}, {33, 3, 2}, {5, 16, 33},
                            {33, 30, 29}, {64, 20, 17}, {17, 1, 5}};
    const float steps[] = {0.0f, 0.4f, 3.0f, 40.0f, NAN};
    for (const auto &s : grids)
        for (float flat : {32.0f, 70.0f, 300.0f})
            for (float da : steps)
                for (float dh : steps)
                    for (float dw : steps) {
                        Tiling t{};
                        t.A = s[0]; t.H = s[1]; t.W = s[2];
                        t.flat = flat;
                        t = shaped(t, da, dh, dw);
                        const int count = t.nta * t.nth * t.ntw;
                        CHECK(t.ta * t.th * t.tw == 64);
                        CHECK(count <= flat_most(t.A, t.H, t.W));
                        std::vector<int> seen((size_t)t.A * t.H * t.W, 0);
                        for (int b = 0; b < count + 3; b++)
                            for (int lane = 0; lane < 64; lane++) {
                                bool valid;
                                const int v = voxel_of(t, b, lane, valid);
                                if (!valid) continue;
                                CHECK(v >= 0 && v < (int)seen.size());
                                seen[v]++;
                            }
                        for (int v : seen) CHECK(v == 1);
                        n++;
                    }
    return n;
}

// Which volumes are shaped: dense ones from 4 voxels on along every axis, or with cubes for every CU;
// with few frames all, sparse ones with 256 cubes.
static long volumes() {
    for (bool swap : {false, true})
        for (int thin : {2, 3, 4, 5}) {
            CHECK(flat_volume(17, swap ? thin : 65, swap ? 65 : thin, false, true) == (thin >= 4));
            CHECK(flat_volume(thin, 16, 16, false, false));
            CHECK(flat_volume(256, swap ? thin : 256, swap ? 256 : thin, false, true));
            CHECK(!flat_volume(24, 24, swap ? 24 : thin, true, true));
        }
    CHECK(flat_volume(8, 8, 8, false, true) && flat_volume(30, 30, 30, true, true));
    // few taps are not worth the look
    for (bool sparse : {false, true})
        for (bool frame_inner : {false, true}) {
            CHECK(!flat_volume(64, 64, 64, sparse, frame_inner, 63));
            CHECK(flat_volume(64, 64, 64, sparse, frame_inner, 1024) == (sparse || frame_inner));
            CHECK(flat_volume(64, 64, 64, sparse, frame_inner, 1024 * 8));
        }
    return 4;
}

// The orders of the blocks over the XCDs are bijections, partial last rounds included.
static long orders() {
    long n = 0;
    for (int nb = 1; nb < 1200; nb += 1 + nb / 40)
        for (int xcd : {0, 1, 8, 64}) {
            std::vector<int> seen(nb, 0);
            for (int b = 0; b < nb; b++) {
                const int to = xcd_order(xcd, b, nb);
                CHECK(to >= 0 && to < nb);
                seen[to]++;
            }
            for (int v : seen) CHECK(v == 1);
            n++;
        }
    return n;
}

// Sparse images go in chunks only where their samples outgrow the shared caches, in the parameter
// adjoint only where a tap is long besides; few tiles never, shaped volumes always.
static long shares() {
    const int64_t few = 128 * 9 * 2000, many = 128 * 64 * 2000;
    for (bool params : {false, true}) {
        for (int64_t record : {16, 32, 64}) {
            CHECK(!sparse_chunks(false, 1024, record, few / 2, 4, params));
            CHECK(!sparse_chunks(false, 511, record, many, 4, params));
            CHECK(sparse_chunks(true, 8, record, few, 4, params));
        }
        CHECK(sparse_chunks(false, 1024, 64, many, 16, params));
        CHECK(sparse_chunks(false, 1024, 32, many, 8, params));
        CHECK(sparse_chunks(false, 1024, 32, many, 9, params) == !params);
        CHECK(sparse_chunks(false, 1024, 16, many, 8, params) == !params);
        CHECK(sparse_chunks(false, 512, 0, few, 8, params));
    }
    return 2;
}

// One to three frames stay with das_fwd_few_kernel where the tiles are few or the slots many.
static long routes() {
    for (bool volume : {false, true})
        for (int B : {1, 2, 3})
            for (bool cplx : {false, true})
                for (bool narrow : {false, true})
                    for (bool sparse : {false, true}) {
                        const bool words = narrow && !cplx;
                        const bool wide = words && B >= 2 && volume;
                        CHECK(few_pays(999, volume, 16, 1, B, cplx, narrow, sparse));
                        CHECK(few_pays(1499, volume, 64, 1, B, cplx, narrow, sparse));
                        CHECK(few_pays(2999, volume, 64, 1, B, cplx, narrow, sparse) == !(sparse && words));
                        CHECK(!few_pays(1000, volume, 32, 1, B, cplx, narrow, sparse));
                        CHECK(!few_pays(3000, volume, 64, 1, B, cplx, narrow, sparse));
                        CHECK(few_pays(100000, volume, 64, 4, B, cplx, narrow, sparse) ==
                              !(wide || (sparse && (words || (!volume && B >= 2)))));
                    }
    return 2;
}

// Terms of every size and sign, h just below an integer among them, convert without leaving 32 bits
// and hold h + l to 2^-31; between -1 and 0, where h has more places than its fraction, to 2^-24.
static long terms() {
    long n = 0;
    std::vector<float> hs = {0.0f, -0.0f, 4194303.75f, -4194303.75f, -1e-38f, -1e-45f, 1e-45f};
    for (int e = -40; e < 22; e++)
        for (float m : {1.0f, 1.25f, 1.9999999f}) {
            const float v = std::ldexp(m, e);
            hs.push_back(v);
            hs.push_back(-v);
            hs.push_back(std::nextafter(std::floor(v), -INFINITY));
            hs.push_back(-std::nextafter(std::floor(v), INFINITY));
        }
    for (float h : hs)
        for (float part : {0.0f, 0.5f, -0.5f, 0.37f}) {
            const float ulp = std::nextafter(std::fabs(h), INFINITY) - std::fabs(h);
            const float l = part * ulp;
            const int64_t v = to_fixed(h, l);
            const double want = std::ldexp((double)h + (double)l, 32);
            CHECK(std::fabs((double)v - want) <= (h < 0.0f && h > -1.0f ? 256.0 : 2.0));
            n++;
        }
    return n;
}

// An offset that is passed over selects no sample with any radius, in exact arithmetic; one within
// the limit or not finite is not passed over.
static long beyond() {
    long n = 0;
    for (int S : {2, 83, 4096, 4194303, 4194304, 4194305, 1 << 29})
        for (float h : {-INFINITY, -3e38f, -6e6f, -4194304.5f, -4194304.0f, -4194303.75f, -1.0f, 0.0f, 5e3f,
                        4194303.75f, 4194304.0f, 5e6f, 1e9f, 3e38f, INFINITY, NAN}) {
            const bool far = beyond_samples(h, S);
            if (!std::isfinite(h) || std::fabs(h) < kFixedLimit) CHECK(!far);
            else if (S <= 4194304 && std::fabs(h) < 3e38f) CHECK(far);
            for (double r : {0.0, 0.25, 700.0, 4194303.0, 4194303.9999}) {
                const double k = std::floor((double)h + r);
                if (far) CHECK(!(k >= 0.0 && k < (double)(S - 1)));
                n++;
            }
        }
    return n;
}

int main() {
    std::printf("slots %ld, tiles %ld, volumes %ld, orders %ld, shares %ld, routes %ld, terms %ld, offsets %ld: "
                "index arithmetic clean\n", slots(), tiles(), volumes(), orders(), shares(), routes(),
                terms(), beyond());
    return 0;
}
