// The delay-and-sum forward for few frames (natural layout, one or two frames a chunk).
#include "das_device.h"

namespace ffdas {
namespace dev {

// Few frames (natural layout, one or two frames a chunk): nothing amortises the delay of a
// (voxel, channel, slot) over frames, so the kernel is bound by the VALU work of a tap.  Its
// delay is one 64-bit fixed-point addition (das_device.h), a slot that reads nothing and a
// channel outside its cone are terms past every row, and the loads go through a buffer
// resource over the channel's rows, where a tap out of range takes an offset past the block
// and reads zeros: per tap an add with carry, a compare, a select, a shift, a conversion and
// four FMA-class operations.  A wave issues the loads of TB taps before it uses the first,
// and G waves share a voxel tile by channels, so that small images fill the chip too.
//
// A finite offset beyond every sample is a slot that reads nothing.  Other terms that fixed point
// does not hold (not finite, a radius beyond 2^22 samples, or a real weight whose product with 2^-32
// is not exact) take the floating-point tap of the plain kernel; a wave meets them together.
//
// 128^3 voxels, 1024 channels, 16 transmits, FP32, cone of 30 degrees: 27.8 ms with the
// floating-point tap at one wave per tile, 11.2 ms (3.1e12 units/s) with the fixed-point tap, 16
// slots a round, flat tiles and the XCDs sharing the grid in chunks.
constexpr int kXcdTiles = 64;

template <Storage ST, int CW> struct FewRows {
    using raw = typename Elem<ST>::raw;
    static constexpr int ES = (int)sizeof(raw) * CW;      // bytes of a sample
    // x[k], x[k+1] of one frame as loaded
    struct Pair { uint32_t w[ES >= 4 ? ES / 2 : 2]; };
    static __device__ __forceinline__ Pair load(__amdgpu_buffer_rsrc_t rows, uint32_t off, int row) {
        Pair q;
        if constexpr (ES == 2) {
            q.w[0] = __builtin_amdgcn_raw_buffer_load_b16(rows, (int)off, row, 0);
            q.w[1] = __builtin_amdgcn_raw_buffer_load_b16(rows, (int)off + 2, row, 0);
        } else if constexpr (ES == 4) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(rows, (int)off, row, 0);
            q.w[0] = v[0]; q.w[1] = v[1];
        } else {
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(rows, (int)off, row, 0);
            q.w[0] = v[0]; q.w[1] = v[1]; q.w[2] = v[2]; q.w[3] = v[3];
        }
        return q;
    }
    // part c of x[k + h]
    static __device__ __forceinline__ float part(const Pair &q, int h, int c) {
        if constexpr (sizeof(raw) == 4) {
            return __uint_as_float(q.w[h * CW + c]);
        } else {
            const uint16_t b = (uint16_t)(CW == 2 ? q.w[h] >> (16 * c) : q.w[h]);
            raw r;
            __builtin_memcpy(&r, &b, 2);
            return Elem<ST>::real(r);
        }
    }
};

template <Storage ST, bool CPLX, int FT, int KC, int TB, bool SPARSE>
__global__ __launch_bounds__(1024) void das_fwd_few_kernel(Geo g, Tiling tl,
                                                           const void *__restrict__ xv,
                                                           int64_t xs_b, int64_t xs_c, int64_t xs_t,
                                                           void *__restrict__ outv, int64_t os_b,
                                                           double beta_re, double beta_im) {
    static_assert(KC % (2 * TB) == 0, "taps per group must divide taps per round");
    constexpr int CW = CPLX ? 2 : 1;
    using Rows = FewRows<ST, CW>;
    using raw = typename Rows::raw;
    extern __shared__ unsigned char few_lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = blockDim.x >> 6;
    int tile = blockIdx.x, chunk = blockIdx.y;
    if (tl.xcd) {
        const int b = xcd_chunk(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y,
                                kXcdTiles);
        chunk = b / gridDim.x;
        tile = b - chunk * gridDim.x;
    }
    bool valid;
    const Tiling ot = oriented(tl, g);
    if (tile >= ot.nta * ot.nth * ot.ntw) return;            // the whole workgroup
    int n = voxel_of(ot, tile, lane, valid);
    if (!valid) n = 0;          // computed, never stored: keeps every lane at the barrier
    const SplitPt yp = split_point(g.dstpos[3 * n], g.dstpos[3 * n + 1], g.dstpos[3 * n + 2]);
    const uint32_t last = (uint32_t)(g.S - 1);
    const int span = (int)(((int64_t)(g.T - 1) * xs_t + g.S) * Rows::ES);   // bytes, host-checked
    const raw *frame[FT];
#pragma unroll
    for (int f = 0; f < FT; f++)
        frame[f] = static_cast<const raw *>(xv) + (int64_t)min(chunk * FT + f, g.B - 1) * xs_b * CW;
    float acc[FT][CW];
#pragma unroll
    for (int f = 0; f < FT; f++)
#pragma unroll
        for (int c = 0; c < CW; c++) acc[f][c] = 0.0f;

    auto add = [&](int f, const typename Rows::Pair &q, float wt, float tk, float t, float sn, float cs) {
        if constexpr (!CPLX) {
            const float c = wt * tk;                 // weight of x[k+1]
            const float a = __builtin_fmaf(wt, t, -c);   // the whole weight less c
            acc[f][0] = fmaA(c, Rows::part(q, 1, 0), fmaA(a, Rows::part(q, 0, 0), acc[f][0]));
        } else {
            const float x0r = Rows::part(q, 0, 0), x0i = Rows::part(q, 0, 1);
            const float lr = x0r + t * (Rows::part(q, 1, 0) - x0r);
            const float li = x0i + t * (Rows::part(q, 1, 1) - x0i);
            acc[f][0] += cs * lr - sn * li;          // (cs, sn): the rotated weight
            acc[f][1] += cs * li + sn * lr;
        }
    };

    for (int kc = 0; kc < g.K && g.S >= 2; kc += KC) {
        int64_t ofs[KC];            // scale * offset, 32.32
        float wt[KC], wi[CPLX ? KC : 1];   // complex: the weight times e^{i wavenum scale offset}
        uint32_t rowoff[SPARSE ? KC : 1];
        bool plainly = true;
#pragma unroll
        for (int j = 0; j < KC; j++) {
            const int jj = kc + j;
            ofs[j] = (int64_t)kFixedNone << 32;
            wt[j] = 0.0f;
            if constexpr (CPLX) wi[j] = 0.0f;
            if constexpr (SPARSE) rowoff[j] = 0;
            if (jj < g.K) {
                const int64_t o = (int64_t)jj * g.N + n;
                float h = g.offsets[o], l = 0.0f;
                wt[j] = g.weights[o];
                bool any = true;
                if constexpr (SPARSE) {
                    const int sq = g.sparse[o];
                    any = (uint32_t)sq < (uint32_t)g.T;
                    if (any) rowoff[j] = (uint32_t)sq * (uint32_t)xs_t * (uint32_t)Rows::ES;
                }
                scale_pair(g.scale, h, l);
                any = any && !beyond_samples(h, g.S);
                const float aw = __builtin_fabsf(wt[j]);
                const bool good = __builtin_fabsf(h) < kFixedLimit && aw < 3e38f &&
                                  (CPLX || aw == 0.0f || aw > 1e-27f);
                if (any && good) ofs[j] = to_fixed(h, l);
                else wt[j] = 0.0f;                       // it meets zeros: no NaN from it
                if (any && !good) plainly = false;
                if constexpr (!CPLX) {
                    wt[j] *= 2.3283064365386963e-10f;    // 2^-32
                } else {
                    float sn, cs;
                    phase_term(g.rev_h, g.rev_l, any && good ? h : 0.0f, l, sn, cs);
                    wi[j] = wt[j] * sn;
                    wt[j] *= cs;
                }
            }
        }
        const bool fixed_slots = __builtin_amdgcn_ballot_w64(!plainly) == 0;
        for (int m = wave; m < g.C; m += G) {
            const SplitPt pp = split_point(g.srcpos[3 * m], g.srcpos[3 * m + 1], g.srcpos[3 * m + 2]);
            const Radius R = radius_precise(yp, pp);
            bool dok = true;
            if (g.srcdir) {
                const float *sd = g.srcdir + 4 * m;
                dok = (R.dx * sd[0] + R.dy * sd[1] + R.dz * sd[2]) * R.rinv > sd[3];
                if (__builtin_amdgcn_ballot_w64(dok) == 0) continue;
            }
            float rh = R.rh, rl = R.rl;
            if (g.scale != 1.0f) scale_pair(g.scale, rh, rl);
            // the sum is NaN where either part is (a NaN position leaves rh finite)
            const bool fixed = fixed_slots && __builtin_amdgcn_ballot_w64(!(rh + rl < kFixedLimit)) == 0;
            if (__builtin_expect(!fixed, 0)) {
#pragma unroll 1
                for (int jj = kc; jj < min(kc + KC, g.K); jj++) {
                    const int64_t o = (int64_t)jj * g.N + n;
                    const int sq = SPARSE ? g.sparse[o] : jj;
                    const float w = g.weights[o];
                    const Tap tp = make_tap<true>(g.offsets[o], R, g.scale);
                    if (!(dok && (uint32_t)tp.k < last && (uint32_t)sq < (uint32_t)g.T)) continue;
                    float sn = 0.0f, cs = w;
                    if constexpr (CPLX) {
                        phase<true>(g.rev_h, g.rev_l, tp, sn, cs);
                        sn *= w;
                        cs *= w;
                    }
                    const int64_t e = (int64_t)m * xs_c + (int64_t)sq * xs_t + tp.k;
#pragma unroll
                    for (int f = 0; f < FT; f++) {
                        typename Rows::Pair q;
                        const raw *s = frame[f] + e * CW;
                        if constexpr (Rows::ES == 2) {
                            uint16_t b[2];
                            __builtin_memcpy(b, s, 4);
                            q.w[0] = b[0];
                            q.w[1] = b[1];
                        } else {
                            __builtin_memcpy(&q, s, 2 * Rows::ES);
                        }
                        add(f, q, w, tp.t, CPLX ? tp.t : 1.0f, sn, cs);
                    }
                }
                continue;
            }
            int64_t rf = to_fixed(rh, rl);
            if (!dok) rf = (int64_t)kFixedNone << 32;
            float sr = 0.0f, cr = 1.0f;
            if constexpr (CPLX) phase_term(g.rev_h, g.rev_l, rh, rl, sr, cr);
            __amdgpu_buffer_rsrc_t rows[FT];
#pragma unroll
            for (int f = 0; f < FT; f++)
                rows[f] = __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<raw *>(frame[f] + (int64_t)m * xs_c * CW), (short)0, span, kBufWord3);
            // the taps of group j0: delays and loads, then (use) their sums
            auto issue = [&](int j0, auto full, auto &q, auto &tau) {
#pragma unroll
                for (int u = 0; u < (int)std::extent_v<std::remove_reference_t<decltype(tau)>>; u++) {
                    const int j = j0 + u;
                    if (!decltype(full)::value && kc + j >= g.K) break;
                    tau[u] = (uint64_t)ofs[j] + (uint64_t)rf;
                    const uint32_t k = (uint32_t)(tau[u] >> 32);
                    uint32_t off = k * (uint32_t)Rows::ES;
                    if constexpr (SPARSE) off += rowoff[j];
                    off = k < last ? off : kNoRows;
                    const int row = SPARSE ? 0 : (kc + j) * (int)xs_t * Rows::ES;
#pragma unroll
                    for (int f = 0; f < FT; f++) q[u][f] = Rows::load(rows[f], off, row);
                }
            };
            auto use = [&](int j0, auto full, const auto &q, const auto &tau) {
#pragma unroll
                for (int u = 0; u < (int)std::extent_v<std::remove_reference_t<decltype(tau)>>; u++) {
                    const int j = j0 + u;
                    if (!decltype(full)::value && kc + j >= g.K) break;
                    const float tf = (float)(uint32_t)tau[u];         // fraction * 2^32
                    if constexpr (!CPLX) {
                        // a tap out of range read zeros, and its weights are finite
#pragma unroll
                        for (int f = 0; f < FT; f++)
                            add(f, q[u][f], wt[j], tf, 4294967296.0f, 0.0f, 0.0f);
                    } else {
                        // the slot's rotation times the channel's: no sine or cosine a tap
                        const float sn = wt[j] * sr + wi[j] * cr, cs = wt[j] * cr - wi[j] * sr;
#pragma unroll
                        for (int f = 0; f < FT; f++)
                            add(f, q[u][f], 0.0f, 0.0f, tf * 2.3283064365386963e-10f, sn, cs);
                    }
                }
            };
            if (!CPLX && kc + KC <= g.K) {
                // a whole round: the loads of a group are issued before the sums of the one
                // before it (complex data, whose phase keeps many values live, spills then)
                typename Rows::Pair q[2][TB][FT];
                uint64_t tau[2][TB];
                issue(0, std::true_type{}, q[0], tau[0]);
#pragma unroll
                for (int j0 = 0; j0 < KC; j0 += TB) {
                    const int i = (j0 / TB) & 1;
                    if (j0 + TB < KC) issue(j0 + TB, std::true_type{}, q[1 - i], tau[1 - i]);
                    __builtin_amdgcn_sched_barrier(0);
                    use(j0, std::true_type{}, q[i], tau[i]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int j0 = 0; j0 < KC; j0 += TB) {
                    if (kc + j0 >= g.K) break;
                    typename Rows::Pair q[TB][FT];
                    uint64_t tau[TB];
                    issue(j0, std::false_type{}, q, tau);
                    __builtin_amdgcn_sched_barrier(0);
                    use(j0, std::false_type{}, q, tau);
                }
            }
        }
    }
    if (G == 1) {
        if (valid) store_out<false, CPLX, FT>(acc, outv, os_b, n, chunk * FT, g.B, beta_re, beta_im);
        return;
    }
    float *red = reinterpret_cast<float *>(few_lds);      // red[w][f * CW + c][lane]
#pragma unroll
    for (int f = 0; f < FT; f++)
#pragma unroll
        for (int c = 0; c < CW; c++) red[(wave * FT * CW + f * CW + c) * 64 + lane] = acc[f][c];
    __syncthreads();
    if (wave > 0 || !valid) return;
#pragma unroll
    for (int f = 0; f < FT; f++)
#pragma unroll
        for (int c = 0; c < CW; c++) {
            float sum = 0.0f;
            for (int w = 0; w < G; w++) sum += red[(w * FT * CW + f * CW + c) * 64 + lane];
            acc[f][c] = sum;
        }
    store_out<false, CPLX, FT>(acc, outv, os_b, n, chunk * FT, g.B, beta_re, beta_im);
}

}  // namespace dev

namespace {

// Taps of a group; a wave has two groups in flight.  Complex data and two frames at 4 spill.
template <bool CPLX, int FT> constexpr int tap_group() { return CPLX || FT > 1 ? 2 : 4; }

// Waves per voxel tile of das_fwd_few_kernel: enough to put eight on each SIMD, at most 16 and
// at most one per channel (128-element, 3-transmit image of 256 x 128: 147 us with one wave
// per tile and the old tap, 21 us with 16).  Slots a lane holds at a time: 8, and 16, which forms the
// radius half as often, where they leave no remainder or one below 4; a longer one costs more, since it
// is not pipelined, than whole rounds of 8.  By 16 and by 8, 64^3 voxels and 256 channels, one frame:
// 16 slots 554 and 587 us, 17 709 and 707, 20 794 and 760, 24 976 and 816, 31 1312 and 1122, 32 1049 and
// 1084, 40 1494 and 1356, 48 1596 and 1632; 96^3 voxels and 1024 channels, 17 slots 7.98 and 8.21 ms, 24
// 10.99 and 9.85; below 16 there are only rounds of 8 to fill (192 channels to 400 x 300, 11 slots: 213
// and 198 us).
template <Storage ST, bool CPLX, int FT>
hipError_t launch_few_ft(hipStream_t st, const dev::Geo &g, const dev::Tiling &tl, const XView &xv,
                         void *out, int64_t os_b, double br, double bi) {
    constexpr int TB = tap_group<CPLX, FT>();
    const int ntiles = tl.tiles;
    dim3 grid(ntiles, (g.B + FT - 1) / FT);
    int G = 1;
    while (G < 16 && (int64_t)ntiles * grid.y * G < 8192 && 2 * G <= g.C) G *= 2;
    const size_t lds = G > 1 ? (size_t)G * FT * (CPLX ? 2 : 1) * 64 * sizeof(float) : 0;
    ProfScope ps(st, "das_fwd_few");
    auto go = [&](auto kern) {
        kern<<<grid, 64 * G, lds, st>>>(g, tl, xv.ptr, xv.sb, xv.sc, xv.st, out, os_b, br, bi);
        return hipGetLastError();
    };
    if (g.sparse) return go(dev::das_fwd_few_kernel<ST, CPLX, FT, 8, TB, true>);
    if constexpr (!CPLX && FT == 1)
        if (g.K >= 16 && g.K % 16 < 4) return go(dev::das_fwd_few_kernel<ST, CPLX, FT, 16, TB, false>);
    return go(dev::das_fwd_few_kernel<ST, CPLX, FT, 8, TB, false>);
}

template <Storage ST, bool CPLX>
hipError_t launch_few_t(hipStream_t st, const dev::Geo &g, const dev::Tiling &tl, const XView &xv,
                        void *out, int64_t os_b, double br, double bi) {
    return g.B >= 2 ? launch_few_ft<ST, CPLX, 2>(st, g, tl, xv, out, os_b, br, bi)
                    : launch_few_ft<ST, CPLX, 1>(st, g, tl, xv, out, os_b, br, bi);
}

}  // namespace

// Whether das_fwd_few_kernel takes a natural-layout forward: up to two frames a chunk, float
// data, the rows of a channel within 32-bit byte offsets of its first sample, and complex
// samples on whole words (they are loaded as such).
bool few_frames_ok(const DasProblem &p, const XView &xv) {
    const int es = (int)storage_bytes(p.k_storage) * (p.cplx ? 2 : 1);
    if (p.plain || p.acc64 || p.k_storage == Storage::F64 || p.B >= 4) return false;
    const double span = ((double)(p.T - 1) * (double)xv.st + p.S) * es;
    return span < 2147483648.0 - 64.0 && (!p.cplx || reinterpret_cast<uintptr_t>(xv.ptr) % 4 == 0);
}

hipError_t launch_forward_few(hipStream_t st, const dev::Geo &g, const dev::Tiling &tl,
                              const DasProblem &p, const XView &xv, void *out, double beta_re,
                              double beta_im) {
    const int64_t os_b = p.os_b;
    switch (p.k_storage) {
        case Storage::F16:
            return p.cplx ? launch_few_t<Storage::F16, true>(st, g, tl, xv, out, os_b, beta_re, beta_im)
                          : launch_few_t<Storage::F16, false>(st, g, tl, xv, out, os_b, beta_re, beta_im);
        case Storage::BF16:
            return p.cplx ? launch_few_t<Storage::BF16, true>(st, g, tl, xv, out, os_b, beta_re, beta_im)
                          : launch_few_t<Storage::BF16, false>(st, g, tl, xv, out, os_b, beta_re, beta_im);
        default:
            return p.cplx ? launch_few_t<Storage::F32, true>(st, g, tl, xv, out, os_b, beta_re, beta_im)
                          : launch_few_t<Storage::F32, false>(st, g, tl, xv, out, os_b, beta_re, beta_im);
    }
}

}  // namespace ffdas
