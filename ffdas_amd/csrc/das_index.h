// Index and fixed-point arithmetic of the delay-and-sum kernels: no device intrinsics, so that it is
// also run on the CPU (tests/asan/index_driver.cpp).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ffdas {
namespace dev {

// ---------------------------------------------------------------------------------------
// delays in 32.32 fixed point
// ---------------------------------------------------------------------------------------
// tau = scale * ofs + scale * r is a sum of one term per (voxel, slot) and one per (voxel,
// channel).  With both terms in 32.32 fixed point the sum of a tap is one 64-bit integer
// addition whose high word is floor(tau) and whose low word is the fraction, where the
// floating-point form needs about fifteen operations (TwoSum, scale, two floors) for each
// tap.  The terms carry the compensated pairs to within 2^-31 of a sample, below the FP32
// rounding of the fraction that follows either way (a term between -1 and 0, whose fraction has
// the places of a number near 1, to within 2^-24).
constexpr float kFixedLimit = 4194304.0f;      // |term| < 2^22: its low part fits 31 bits
constexpr int kFixedNone = 0x40000000;         // high word of a term that selects no sample

// The fraction of h, which for h just below an integer is at most the largest float below 1 (h less
// its floor rounds to 1 there, and 2^32 does not convert to 32 bits).
__host__ __device__ __forceinline__ float fraction(float h) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_fractf(h);
#else
    return __builtin_fminf(h - __builtin_floorf(h), 0x1.fffffep-1f);
#endif
}

// h + l (|h| < 2^22, |l| <= ulp(h)) as 32.32 fixed point.
__host__ __device__ __forceinline__ int64_t to_fixed(float h, float l) {
#pragma clang fp contract(off)
    const float f = __builtin_floorf(h);
    const uint32_t lo = (uint32_t)(fraction(h) * 4294967296.0f);
    const int li = (int)__builtin_rintf(l * 4294967296.0f);
    return (int64_t)((uint64_t)(uint32_t)(int)f << 32 | lo) + (int64_t)li;
}

// Whether a finite delay h of a slot, beyond the limit, selects no sample of S whatever radius
// within the limit (0 <= r < 2^22) is added: the slot is passed over, as one without a transmit
// is, and its wave keeps the fixed-point taps.  (An infinite delay makes its voxel NaN.)
__host__ __device__ __forceinline__ bool beyond_samples(float h, int S) {
    return __builtin_fabsf(h) < 3e38f && (h <= -kFixedLimit || (h >= kFixedLimit && S <= (int)kFixedLimit));
}

// scale * (h + l) as a float pair; exact for scale == 1.
__host__ __device__ __forceinline__ void scale_pair(float scale, float &h, float &l) {
#pragma clang fp contract(off)
    const float sh = scale * h;
    const float sl = __builtin_fmaf(scale, h, -sh);
    l = __builtin_fmaf(scale, l, sl);
    h = sh;
}

// Scalar byte offset of the rows of slot j (dense compounding: its transmit) from the start of a
// channel's block of K transmits, `step` bytes each.  A group of taps may reach past the last slot;
// the vector offsets of those taps are past the block and read zeros, but the range check of a raw
// buffer is against what the scalar offset leaves of it, which must not be less than nothing.
__host__ __device__ __forceinline__ int slot_offset(int j, int K, int step) {
    return (j < K ? j : K - 1) * step;
}

// ---------------------------------------------------------------------------------------
// voxel tiling: a wave covers a compact (ta x th x tw) tile of the (A, H, W) voxel grid
// ---------------------------------------------------------------------------------------
struct Tiling {
    int A, H, W;        // spatial view (outer dims folded into A)
    int ta, th, tw;     // wave tile, ta*th*tw == 64
    int nta, nth, ntw;  // tile counts
    int tiles;          // tiles a launch covers (flat: of the shape with most)
    int xcd;            // order of the blocks over the XCDs (xcd_order)
    float flat;         // a volume whose tiles the kernel shapes (oriented): the cost of a tap
                        // beside its window, in samples of window; 0: fixed tiles
    int steep;          // oriented: the axis the tiles are thin along (0 A, 1 H, 2 W)
};

// Tiles of a volume whose steep axis has n voxels and the other two u and v, as log2 of the edges
// ln | lu << 4 | lv << 8, and their count.
constexpr int kFlatTiles = 6;
__host__ __device__ __forceinline__ int flat_shape(int c) {
    constexpr int shape[kFlatTiles] = {0x330, 0x420, 0x240, 0x231, 0x321, 0x222};
    return shape[c];
}
__host__ __device__ __forceinline__ int64_t flat_count(int shape, int n, int u, int v) {
    const int ln = shape & 15, lu = (shape >> 4) & 15, lv = shape >> 8;
    return (int64_t)((n + (1 << ln) - 1) >> ln) * ((u + (1 << lu) - 1) >> lu) *
           ((v + (1 << lv) - 1) >> lv);
}
// Shapes with more tiles than a sixteenth above the fewest compute too many voxels beyond the grid.
__host__ __device__ __forceinline__ int64_t flat_limit(int n, int u, int v) {
    int64_t least = flat_count(flat_shape(0), n, u, v);
    for (int c = 1; c < kFlatTiles; c++) {
        const int64_t k = flat_count(flat_shape(c), n, u, v);
        least = k < least ? k : least;
    }
    return least + least / 16;
}

// The most tiles that any shape the kernels may choose (shaped) has on an A x H x W volume.
__host__ __device__ __forceinline__ int64_t flat_most(int A, int H, int W) {
    const int size[3][3] = {{A, H, W}, {H, A, W}, {W, A, H}};
    int64_t most = 0;
    for (const auto &n : size) {
        const int64_t limit = flat_limit(n[0], n[1], n[2]);
        for (int c = 0; c < kFlatTiles; c++) {
            const int64_t k = flat_count(flat_shape(c), n[0], n[1], n[2]);
            if (k <= limit && k > most) most = k;
        }
    }
    return most;
}

// Whether the kernels shape a volume's tiles, or keep cubes of 4 x 4 x 4 voxels: a launch that leaves
// CUs idle takes as long as one of its tiles does, and the cubes of a grid thinner than they are hold
// fewer voxels.  Frame-inner rows, 17 x 3 x 65 voxels with depth last, 256 channels, 4 transmits:
// forward 77 us in cubes, 132 shaped, parameter adjoint 90 and 134; turned round, from 0.71 to 1.7 of
// the cubes' time.  Few frames, whose taps are bound by the VALU, are shaped whatever the grid.  Sparse volumes need
// 256 cubes (24^3 voxels 158 us, shaped 164; 30^3 voxels 312 and 265).
// taps, channels times slots, have to be worth the look at the delays that shaping takes (4 us, and
// 6 with more tiles than cubes fill): 40^3 voxels, 64 channels, one slot, 4 frames 37 us shaped and
// 31 in cubes, one frame 37 and 26; at 512 taps from 0.81 to 1.03 of the cubes' time, at 1024 channels
// and 8 slots 0.59 to 0.88.  Few frames gain later, 24^3 voxels 0.87 there and 1.09 at 256 x 4;
// sparse volumes sooner: 64^3 voxels, 64 channels, 2 slots, 2 complex frames 123 us and 188.
__host__ __device__ __forceinline__ bool flat_volume(int A, int H, int W, bool sparse, bool frame_inner,
                                                     int64_t taps = INT64_MAX) {
    const int64_t cubes = (int64_t)((A + 3) / 4) * ((H + 3) / 4) * ((W + 3) / 4);
    if (taps < (sparse ? 64 : frame_inner ? 512 : 8192)) return false;
    if (sparse) return cubes >= 256;
    return !frame_inner || cubes >= 512 || (A >= 4 && H >= 4 && W >= 4);
}

// The tiles of a volume whose delay changes by da, dh and dw a step along its axes: the shape whose
// taps cost least, a tap costing tl.flat and the window of samples that the lanes of a wave read of
// a row, which is what those steps span over a tile (da, dh, dw are sums over 16 pairs).  The axis
// of the largest step (depth, first in the (z, y, x) grids of the examples, last in column-major
// callers') is walked last.
__host__ __device__ __forceinline__ Tiling shaped(Tiling tl, float da, float dh, float dw) {
    tl.steep = dw > da && dw >= dh ? 2 : dh > da ? 1 : 0;
    const int size = tl.steep == 0 ? tl.A : tl.steep == 1 ? tl.H : tl.W;
    const int u = tl.steep == 0 ? tl.H : tl.A, v = tl.steep == 2 ? tl.H : tl.W;
    const float ds = tl.steep == 0 ? da : tl.steep == 1 ? dh : dw;
    const float du = tl.steep == 0 ? dh : da, dv = tl.steep == 2 ? dh : dw;
    const int64_t limit = flat_limit(size, u, v);
    int best = -1;
    float cost = 0.0f;
    for (int c = 0; c < kFlatTiles; c++) {
        const int shape = flat_shape(c);
        const int64_t count = flat_count(shape, size, u, v);
        if (count > limit) continue;
        const float window = (float)((1 << (shape & 15)) - 1) * ds +
                             (float)((1 << ((shape >> 4) & 15)) - 1) * du +
                             (float)((1 << (shape >> 8)) - 1) * dv;
        const float k = (float)count * (16.0f * tl.flat + window);
        if (best < 0 || k < cost) {
            best = shape;
            cost = k;
        }
    }
    const int e0 = 1 << (best & 15), e1 = 1 << ((best >> 4) & 15), e2 = 1 << (best >> 8);
    tl.ta = tl.steep == 0 ? e0 : e1;
    tl.th = tl.steep == 1 ? e0 : tl.steep == 0 ? e1 : e2;
    tl.tw = tl.steep == 2 ? e0 : e2;
    tl.nta = (tl.A + tl.ta - 1) / tl.ta;
    tl.nth = (tl.H + tl.th - 1) / tl.th;
    tl.ntw = (tl.W + tl.tw - 1) / tl.tw;
    return tl;
}

// Workgroups are dispatched to the eight XCDs in turn (linear block id mod 8).  With xcd
// set, linear id b is read as block (b mod 8) * (nb / 8) + b / 8 of the grid's order, so the
// blocks of one XCD form a contiguous range of tiles and share that XCD's L2.  A bijection
// on the complete rounds of 8; the last nb mod 8 blocks keep their ids.
__host__ __device__ __forceinline__ int xcd_block(int b, int nb) {
    const int full = nb & ~7;
    if (b >= full) return b;
    return (b & 7) * (full >> 3) + (b >> 3);
}

// The same in chunks of q tiles: each XCD still works on neighbouring tiles, but regions whose
// tiles cost less (channels outside their cones are passed over) are shared out over all of
// them.  The chunk an XCD takes moves on by one each round of 8, so that a period in the grid
// does not give one XCD the cheap tiles every time.  A bijection on the complete rounds.
__host__ __device__ __forceinline__ int xcd_chunk(int b, int nb, int q) {
    const int round = b / (8 * q), i = b - round * 8 * q;
    if ((round + 1) * 8 * q > nb) return b;
    return round * 8 * q + ((i + round) & 7) * q + (i >> 3);
}

// Whether the forward of one to three frames goes to das_fwd_few_kernel: it shares a tile's channels
// out over waves and its taps cost less, and pays for that a setup a tile and a term a channel.  tiles
// are those of das_fwd_kernel, which has one wave a tile: below a thousand it cannot fill the chip.
// Few against that kernel, from 1 slot up where it starts to pay:
//   512 x 512, FP32, 1 frame, 64 channels          1 slot 1.23, 2: 1.08, 3: 0.98, 4: 0.78, 8: 0.45
//   96^3, FP32, 2 frames, 64 channels              1.33, 1.08, 1.06, 0.95, 0.93
//   1024 x 512, complex FP32, 1 frame, 256         1.27, 1.01, 0.96, 0.86, 0.78
//   400 x 256, FP32, 1 frame, 16 channels          1.47, 1.29, 1.07, 1.01, 0.78; 256 channels below 1
//   96^3, FP16, 2 frames, 64 channels              1.26, 1.11, 1.16, 1.14, 1.22 (16 slots 1.21)
//   64^3, FP16, 2 frames, sparse, 64 channels      1.84, 2.00 and (4) 2.03, (8) 2.05; 1000 tiles 0.93 to 1.07
//   64^3, FP32, 1 frame, sparse, 64 channels       1.61, 1.20 and (4) 0.90
//   512 x 512, FP32, 2 frames, sparse, 64 channels 1.28, 1.21 and (4) 1.14, (8) 1.07
inline bool few_pays(int64_t tiles, bool volume, int C, int K, int B, bool cplx, bool narrow,
                     bool sparse) {
    const bool words = !cplx && narrow;        // 16-bit samples, two loads a tap
    const bool wide = tiles >= 3000;
    if (tiles < 1000) return true;
    if (words && B >= 2 && volume && (wide || C <= 32)) return false;
    if (C <= 32) {                             // few channels to share out
        if (sparse && (words || (volume ? !wide : tiles >= 1500))) return false;
        return K >= (volume || tiles >= 1500 ? 4 : 2);
    }
    if (sparse && words) return tiles < 1500;
    if (!wide) return true;
    if (sparse && !volume && B >= 2) return false;
    if (cplx) return K >= 2;
    if (sparse) return K >= (B == 1 ? 3 : 2);
    if (words && B >= 2) return K >= 4;
    return K >= (B >= 2 && tiles >= 8000 ? 4 : 3);
}

// Whether sparse compounding takes chunks rather than contiguous ranges.  Shaped volumes do.  Images
// do where their samples outgrow the caches that the XCDs share and a tap is long enough to wait for
// them: chunks then keep the XCDs at one part of the samples, and ranges are the better while it is
// the tiles' own rows that each L2 must hold.  record: bytes of all frames of a sample in a record
// (0: rows in their natural order, or several problems in a launch, which go by the tiles alone);
// samples: C * T * S; params: the parameter adjoint, which writes each slot besides, and passes over
// the samples once in eight slots.  Chunks against ranges, 128 channels of 2000 samples:
//   forward    256 x 256, FP32, 8 frames, 64 transmits (500 MiB), 8 slots     823 and 891 us
//              500 x 260, FP16, 8 frames, 64 transmits (250 MiB), 8 slots     838 and 882
//              256 x 256, FP32, 8 frames, 16 transmits (125 MiB), 8 slots     421 and 432
//              256 x 256, FP32, 4 frames, 16 transmits (62 MiB), 8 slots      210 and 199
//              256 x 256, BF16, 16 frames, 9 transmits (70 MiB), 2 slots      147 and 138
//   adjoint    500 x 260, FP32, 16 frames, 64 transmits (1000 MiB), 8 slots   2.32 and 2.84 ms
//              500 x 260, complex, 4 frames, 64 transmits (500 MiB), 8 slots  1.72 and 1.94
//              256 x 256, FP32, 8 frames, 64 transmits (500 MiB), 16 slots    1.68 and 1.56
//              256 x 256, FP16, 8 frames, 64 transmits (250 MiB), 8 slots     522 and 482 us
//              256 x 256, FP16, 8 frames, 9 transmits (35 MiB), 1 slot        52 and 49
inline bool sparse_chunks(bool shaped, int64_t tiles, int64_t record, int64_t samples, int K,
                          bool params) {
    if (shaped || tiles < 512) return shaped;
    if (record == 0) return true;
    const int64_t mib = (record * samples) >> 20;
    return params ? mib >= 240 && (record >= 64 || (record >= 32 && K <= 8)) : mib >= 120;
}

// The order of Tiling::xcd: 0 the hardware's, 1 contiguous ranges, more: chunks of so many blocks.
__host__ __device__ __forceinline__ int xcd_order(int xcd, int b, int nb) {
    return xcd == 0 ? b : xcd == 1 ? xcd_block(b, nb) : xcd_chunk(b, nb, xcd);
}

__host__ __device__ __forceinline__ int voxel_of(const Tiling &tl, int tile, int lane, bool &valid) {
    const int ntiles = tl.nta * tl.nth * tl.ntw;
    valid = tile < ntiles;
    // tiles in the order (w, h, a); where w or h is the steep axis, it comes last
    int ia, ih, iw;
    if (tl.steep == 2) {
        ih = tile % tl.nth;
        const int rest = tile / tl.nth;
        ia = rest % tl.nta;
        iw = rest / tl.nta;
    } else {
        iw = tile % tl.ntw;
        const int rest = tile / tl.ntw;
        const int nin = tl.steep == 1 ? tl.nta : tl.nth;
        const int in = rest % nin, out = rest / nin;
        ih = tl.steep == 1 ? out : in;
        ia = tl.steep == 1 ? in : out;
    }
    const int lw = lane % tl.tw;
    const int lh = (lane / tl.tw) % tl.th;
    const int la = lane / (tl.tw * tl.th);
    const int w = iw * tl.tw + lw, h = ih * tl.th + lh, a = ia * tl.ta + la;
    valid = valid && w < tl.W && h < tl.H && a < tl.A;
    return (a * tl.H + h) * tl.W + w;
}

}  // namespace dev
}  // namespace ffdas
