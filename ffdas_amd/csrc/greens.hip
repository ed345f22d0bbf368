// Frequency-domain Green's function summation (ffdas_greens):
//   out[b, t, f] = sum_s x[b, s, f] e^{i k_f r_ts} / r_ts,   r_ts = |dst_t - src_s|.
// One event, and up to four at few frequencies and many targets (greens_kernel): one lane per
// target, its position and per-source distance in registers; the source position and the x values
// of a (source, frequency chunk, event) are the same for the whole wave, so they come through the
// scalar unit; each thread keeps FPT frequencies x BT events of complex sums on the VALU.  More
// events and frequencies (greens_mfma_kernel): the sums on the MFMA, see there.  FP32 throughout (the
// input may be stored as FP16).
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <climits>

#include "internal.h"

namespace ffdas {
namespace {

constexpr int kGreensFPT = 8;     // frequencies per thread

template <typename XT>
__device__ __forceinline__ float2 load_x(const XT *p);
template <>
__device__ __forceinline__ float2 load_x<float2>(const float2 *p) { return *p; }
template <>
__device__ __forceinline__ float2 load_x<__half2>(const __half2 *p) { return __half22float2(*p); }

template <typename XT, int BT>
__global__ __launch_bounds__(256) void greens_kernel(const float *__restrict__ src,
                                                     const float *__restrict__ wav,
                                                     const XT *__restrict__ x,
                                                     const float *__restrict__ dst,
                                                     float2 *__restrict__ out, int nsrc, int nfreq,
                                                     int ndst, int B) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int f0 = blockIdx.y * kGreensFPT;
    const int b0 = blockIdx.z * BT;
    const int nf = min(kGreensFPT, nfreq - f0), nb = min(BT, B - b0);
    const bool valid = t < ndst;
    float px = 0, py = 0, pz = 0;
    if (valid) {
        px = dst[3 * (int64_t)t];
        py = dst[3 * (int64_t)t + 1];
        pz = dst[3 * (int64_t)t + 2];
    }
    float k[kGreensFPT];
#pragma unroll
    for (int f = 0; f < kGreensFPT; f++) k[f] = f < nf ? wav[f0 + f] : 0.0f;
    float ar[kGreensFPT][BT], ai[kGreensFPT][BT];
#pragma unroll
    for (int f = 0; f < kGreensFPT; f++)
#pragma unroll
        for (int b = 0; b < BT; b++) ar[f][b] = ai[f][b] = 0.0f;

    for (int s = 0; s < nsrc; s++) {
        // r = rsq * rsqrt(rsq), as the reference (greens_kernels.cuh:59-61)
        const float dx = px - src[3 * s], dy = py - src[3 * s + 1], dz = pz - src[3 * s + 2];
        const float rsq = dx * dx + dy * dy + dz * dz;
        const float rinv = rsqrtf(rsq);
        const float r = rsq * rinv;
        const XT *xs = x + ((int64_t)b0 * nsrc + s) * nfreq + f0;
#pragma unroll
        for (int f = 0; f < kGreensFPT; f++) {
            if (f < nf) {
                float sn, cs;
                __sincosf(k[f] * r, &sn, &cs);
                const float gr = cs * rinv, gi = sn * rinv;
#pragma unroll
                for (int b = 0; b < BT; b++) {
                    if (b < nb) {
                        const float2 v = load_x<XT>(xs + (int64_t)b * nsrc * nfreq + f);
                        ar[f][b] += gr * v.x - gi * v.y;
                        ai[f][b] += gr * v.y + gi * v.x;
                    }
                }
            }
        }
    }
    if (!valid) return;
#pragma unroll
    for (int b = 0; b < BT; b++) {
        if (b >= nb) break;
        float2 *o = out + ((int64_t)(b0 + b) * ndst + t) * nfreq + f0;
#pragma unroll
        for (int f = 0; f < kGreensFPT; f++)
            if (f < nf) o[f] = float2{ar[f][b], ai[f][b]};
    }
}

// More events: the multiply-adds on the MFMA, as a real product.  A wave has a tile of 16
// targets x 8 events x 8 frequencies (NT = 2: two such tiles, 16 events); the 16 columns of a
// tile are the real parts of its events, then the imaginary parts.  Per step of 4 sources, lane
// (jl, g) = (lane % 16, lane / 16) generates the Green's function of target t0 + jl and source
// s0 + g (the A operand of v_mfma_f32_16x16x4f32); column (b, re) sums gr xr - gi xi and column
// (b, im) gr xi + gi xr, so a tile takes two MFMAs a step into one accumulator.  Output register
// v of lane (jl, g) holds target t0 + 4 g + v.
//
// The workgroup's four waves (64 targets) read the same x, which is staged in LDS for 8 sources
// at a time, two buffers in turn, as the B operands themselves: X1 = (xr | xi) for the real
// part of the Green's function and X2 = (-xi | xr) for its imaginary part, four frequencies of a
// column contiguous (one 16-byte read, consecutive lanes on consecutive banks).
//
// Bound by the MFMA pipe (64 cycles a step and frequency) and by one sincos per (target,
// source, frequency) on the VALU beside it (about 56 cycles).  128 sources to 256 x 128 targets,
// 512 frequencies, 8 events: 3.24 ms with 16 complex columns a tile (half of them idle, four
// MFMAs a step), 2.02 ms with the real columns and x read from memory by every wave (the vector
// L1 at its access rate), 1.81 ms with x staged, 1.60 ms with the MFMAs of a step in one run,
// 1.51 ms at five waves per SIMD (91 TFLOP/s of the sums' multiply-adds).
constexpr int kGreensFPW = 8;
constexpr int kGreensSrc = 8;                                         // sources staged at a time
typedef float GV4 __attribute__((ext_vector_type(4)));
typedef float GV4p __attribute__((ext_vector_type(4), aligned(8)));   // two packed float2

// the two values of x from p; complex values lie on 8-byte (FP16: 4-byte) boundaries
__device__ __forceinline__ void load_two(const float2 *p, float2 (&v)[2]) {
    const GV4p q = *reinterpret_cast<const GV4p *>(p);
    v[0] = float2{q[0], q[1]};
    v[1] = float2{q[2], q[3]};
}
__device__ __forceinline__ void load_two(const __half2 *p, float2 (&v)[2]) {
    v[0] = __half22float2(p[0]);
    v[1] = __half22float2(p[1]);
}

template <typename XT, int NT>
__global__ __launch_bounds__(256, NT == 1 ? 5 : 3) void greens_mfma_kernel(const float *__restrict__ src,
                                                          const float *__restrict__ wav,
                                                          const XT *__restrict__ x,
                                                          const float *__restrict__ dst,
                                                          float2 *__restrict__ out, int nsrc,
                                                          int nfreq, int ndst, int B) {
    constexpr int FPW = kGreensFPW, SC = kGreensSrc;
    // [buffer][operand][source][half of the frequencies][tile, column]
    __shared__ GV4 xs[2][2][SC][2][16 * NT];
    __shared__ GV4 sp[2][SC];                // source positions
    const int lane = threadIdx.x & 63, jl = lane & 15, g = lane >> 4;
    const int t0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16;
    const int f0 = blockIdx.y * FPW;
    const int b0 = blockIdx.z * (8 * NT);
    const int nf = min(FPW, nfreq - f0);
    const bool whole = nf == FPW;            // uniform
    const bool im = jl >= 8;                 // this lane's column is an imaginary part
    const int ta = t0 + jl;                  // this lane's target in the A operand
    const bool tok = ta < ndst;
    float px = 0, py = 0, pz = 0;
    if (tok) {
        px = dst[3 * (int64_t)ta];
        py = dst[3 * (int64_t)ta + 1];
        pz = dst[3 * (int64_t)ta + 2];
    }
    int be[NT];                              // this lane's event in each tile
#pragma unroll
    for (int n = 0; n < NT; n++) be[n] = b0 + 8 * n + (jl & 7);
    float k[FPW];
#pragma unroll
    for (int f = 0; f < FPW; f++) k[f] = f < nf ? wav[f0 + f] : 0.0f;
    GV4 c[NT][FPW];
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int f = 0; f < FPW; f++) c[n][f] = GV4{0.0f, 0.0f, 0.0f, 0.0f};

    // staging: a thread takes frequencies 2 p, 2 p + 1 of event e, source sl (NT of them)
    const int p = threadIdx.x & 3, e = (threadIdx.x >> 2) & 7, sl = threadIdx.x >> 5;
    float2 v[NT][2];
    GV4 pos{0.0f, 0.0f, 0.0f, 0.0f};
    auto fetch = [&](int s0) {
        const int s = s0 + sl;
#pragma unroll
        for (int n = 0; n < NT; n++) {
            const int b = b0 + 8 * n + e;
            const XT *xp = x + ((int64_t)b * nsrc + s) * nfreq + f0 + 2 * p;
            if (whole && b < B && s < nsrc) {
                load_two(xp, v[n]);
            } else {
#pragma unroll
                for (int f = 0; f < 2; f++)
                    v[n][f] = b < B && s < nsrc && 2 * p + f < nf ? load_x<XT>(xp + f)
                                                                  : float2{0.0f, 0.0f};
            }
        }
        if (threadIdx.x < SC && nsrc > 0) {
            const int q = min(s0 + (int)threadIdx.x, nsrc - 1);
            pos = GV4{src[3 * q], src[3 * q + 1], src[3 * q + 2], 0.0f};
        }
    };
    auto put = [&](GV4 &at, float a, float b) {
        reinterpret_cast<float2 *>(&at)[p & 1] = float2{a, b};
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int n = 0; n < NT; n++) {
            GV4 *o1 = xs[buf][0][sl][p >> 1] + 16 * n + e, *o2 = xs[buf][1][sl][p >> 1] + 16 * n + e;
            put(o1[0], v[n][0].x, v[n][1].x);
            put(o1[8], v[n][0].y, v[n][1].y);
            put(o2[0], -v[n][0].y, -v[n][1].y);
            put(o2[8], v[n][0].x, v[n][1].x);
        }
        if (threadIdx.x < SC) sp[buf][threadIdx.x] = pos;
    };
    fetch(0);
    stage(0);
    __syncthreads();
    for (int s0 = 0, buf = 0; s0 < nsrc; s0 += SC, buf ^= 1) {
        const bool more = s0 + SC < nsrc;     // uniform
        if (more) fetch(s0 + SC);
#pragma unroll
        for (int q = 0; q < SC; q += 4) {     // sources past the last: zero x and zero g
            const GV4 ps = sp[buf][q + g];
            const float dx = px - ps[0], dy = py - ps[1], dz = pz - ps[2];
            const float rsq = dx * dx + dy * dy + dz * dz;
            const bool ok = tok && s0 + q + g < nsrc;
            const float ri = rsqrtf(rsq);
            const float rinv = ok ? ri : 0.0f, r = ok ? rsq * ri : 0.0f;
            GV4 x1[NT][2], x2[NT][2];
#pragma unroll
            for (int n = 0; n < NT; n++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    x1[n][h] = xs[buf][0][q + g][h][16 * n + jl];
                    x2[n][h] = xs[buf][1][q + g][h][16 * n + jl];
                }
            // all sincos of the step, then all its MFMAs: one wave's run of MFMAs leaves the
            // VALU to the others (term by term both pipes wait: 1.81 ms against 1.60)
            float ar[FPW], ai[FPW];
#pragma unroll
            for (int f = 0; f < FPW; f++) {
                float sn, cs;
                __sincosf(k[f] * r, &sn, &cs);
                ar[f] = cs * rinv;
                ai[f] = sn * rinv;
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < NT; n++)
#pragma unroll
                for (int f = 0; f < FPW; f++)
                    c[n][f] = __builtin_amdgcn_mfma_f32_16x16x4f32(ar[f], x1[n][f / 4][f & 3],
                                                                   c[n][f], 0, 0, 0);
#pragma unroll
            for (int n = 0; n < NT; n++)
#pragma unroll
                for (int f = 0; f < FPW; f++)
                    c[n][f] = __builtin_amdgcn_mfma_f32_16x16x4f32(ai[f], x2[n][f / 4][f & 3],
                                                                   c[n][f], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        // the other buffer was last read before the previous barrier
        if (more) stage(buf ^ 1);
        __syncthreads();
    }

    // Lanes jl and jl ^ 8 hold the real and imaginary parts of an event: the first takes the
    // lower half of the frequencies, the second the upper half, and each gets the other's part
    // of its half (a rotation by 8 within the row of 16 lanes), so that each lane writes one
    // contiguous run of complex values.
    constexpr int H = FPW / 2;
#pragma unroll
    for (int n = 0; n < NT; n++) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            float2 o[H];
#pragma unroll
            for (int f = 0; f < H; f++) {
                const float give = im ? c[n][f][v] : c[n][f + H][v];
                const float got = __int_as_float(__builtin_amdgcn_update_dpp(
                    0, __float_as_int(give), 0x128, 0xf, 0xf, false));      // row_ror:8
                o[f] = im ? float2{got, c[n][f + H][v]} : float2{c[n][f][v], got};
            }
            const int t = t0 + 4 * g + v;
            if (t >= ndst || be[n] >= B) continue;
            const int fo = im ? H : 0;
            float2 *po = out + ((int64_t)be[n] * ndst + t) * nfreq + f0 + fo;
            if (whole) {
#pragma unroll
                for (int f = 0; f < H; f += 2)
                    *reinterpret_cast<GV4p *>(po + f) = GV4p{o[f].x, o[f].y, o[f + 1].x, o[f + 1].y};
            } else {
#pragma unroll
                for (int f = 0; f < H; f++)
                    if (fo + f < nf) po[f] = o[f];
            }
        }
    }
}

// Whether the sums stay on the VALU.  One event always (one column pair of the 8-event tile would be
// in use: 128 sources to 256 x 128 targets, 512 frequencies 0.84 ms, on the MFMA 1.5).  Two to four where the
// last chunk of frequencies leaves the MFMA tile, which forms all eight, mostly empty and there are
// targets enough to fill the chip with one wave per 64 (the MFMA kernel has four times the waves).
// 128 sources to 2^20 targets, VALU and MFMA: one frequency, 2 events 162 and 741 us, 4 events 201 and
// 745; four frequencies, 4 events 470 and 760; eight, 2 events 591 and 754, 4 events 960 and 756.  To 2^15
// targets the MFMA is the faster from one frequency on (2 events 45 and 30 us; 512 frequencies 1.79 and 1.5 ms).
// With few sources the writes weigh more, and so does a second chunk of frequencies: 16 sources to 2^19
// targets, 3 events, 12 frequencies 144 and 118 us.
// Two events besides where the VALU kernel's workgroups, three a CU, fill the rounds they take: for a
// quarter of the columns the MFMA tile then costs more.  11808 targets, 159 sources, 512 frequencies
// (1504 workgroups, 0.98 of two rounds) 626 and 712 us, 32768 targets, 384 frequencies (four rounds) 1.16
// and 1.42 ms; at 0.65 of the rounds (16000 targets, 256 frequencies) 510 and 481.
bool on_valu(int B, int nsrc, int nfreq, int ndst) {
    if (B == 1) return true;
    if (B > 4) return false;
    const int chunks = (nfreq + kGreensFPT - 1) / kGreensFPT;
    const double waves = (double)((ndst + 255) / 256) * 4.0 * chunks;
    // frequencies a chunk up to which the VALU is the faster where it fills the chip, and fewer
    // waves in proportion
    const bool many = nsrc >= 64;
    const double full = B == 4 ? 4.0 : B == 3 ? 5.0 : many ? 7.0 : 6.0;
    double most = full * std::min(waves / 4096.0, 1.0);
    if (many && waves >= 2048.0) most = std::min(full, most + 0.5);
    if (many && waves >= 8192.0 && B > 2) most += 1.0;
    if (many && waves >= 16384.0 && (B == 3 || (B == 2 && nfreq <= 64))) most += 1.0;
    if (B == 3 && chunks > 1) most -= 1.0;
    if ((double)nfreq / chunks <= most) return true;
    const int64_t groups = (int64_t)((ndst + 255) / 256) * chunks, round = 768;
    const int64_t rounds = (groups + round - 1) / round;
    return B == 2 && many && (double)groups >= 0.87 * (double)(rounds * round);
}

template <typename XT>
ffdas_error_t launch(hipStream_t st, const float *src, const float *wav, const void *x,
                     const float *dst, void *out, int nsrc, int nfreq, int ndst, int B) {
    if (on_valu(B, nsrc, nfreq, ndst)) {
        const dim3 grid((unsigned)((ndst + 255) / 256),
                        (unsigned)((nfreq + kGreensFPT - 1) / kGreensFPT), 1);
        ProfScope ps(st, "greens");
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, src, wav, static_cast<const XT *>(x), dst,
                               static_cast<float2 *>(out), nsrc, nfreq, ndst, B);
            return hip_status(hipGetLastError(), FFDAS_ERROR_CUDA_LAUNCH_FAILED);
        };
        return B == 1 ? go(greens_kernel<XT, 1>) : go(greens_kernel<XT, 4>);
    }
    const int events = B <= 8 ? 8 : 16;
    const dim3 g((unsigned)((ndst + 63) / 64), (unsigned)((nfreq + kGreensFPW - 1) / kGreensFPW),
                 (unsigned)((B + events - 1) / events));
    ProfScope ps(st, "greens");
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, g, dim3(256), 0, st, src, wav, static_cast<const XT *>(x), dst,
                           static_cast<float2 *>(out), nsrc, nfreq, ndst, B);
        return hip_status(hipGetLastError(), FFDAS_ERROR_CUDA_LAUNCH_FAILED);
    };
    return events == 8 ? go(greens_mfma_kernel<XT, 1>) : go(greens_mfma_kernel<XT, 2>);
}

bool packed(const ffdas_tensor_desc &d) {
    int64_t expect = 1;
    for (size_t k = d.dims.size(); k-- > 0;) {
        if (d.dims[k] > 1 && d.strides[k] != expect) return false;
        expect *= d.dims[k];
    }
    return true;
}

}  // namespace
}  // namespace ffdas

using namespace ffdas;

static ffdas_error_t greens_call(ffdas_handle_t handle, const float *srcpos,
                                      const float *wavenums, ffdas_tensor_desc_t x_desc,
                                      const void *x, const float *dstpos,
                                      ffdas_tensor_desc_t out_desc, void *out) {
    if (!handle) return FFDAS_ERROR_INVALID_HANDLE;
    if (!x_desc || !out_desc) return FFDAS_ERROR_NULL_POINTER;
    FFDAS_TRY(handle->check_device());
    const ffdas_tensor_desc &xd = *x_desc, &od = *out_desc;
    const bool half_in = xd.dtype == FFDAS_C_16F;
    if ((xd.dtype != FFDAS_C_32F && !half_in) || od.dtype != FFDAS_C_32F)
        return FFDAS_ERROR_UNSUPPORTED_TYPE;
    if (xd.dims.size() != 3) return FFDAS_ERROR_INVALID_DIMS;
    const int64_t B = xd.dims[0], nsrc = xd.dims[1], nfreq = xd.dims[2];
    if (od.dims.size() != 3 || od.dims[0] != B || od.dims[2] != nfreq)
        return FFDAS_ERROR_INVALID_DIMS;
    const int64_t ndst = od.dims[1];
    if (B > INT_MAX || nsrc > INT_MAX || nfreq > INT_MAX || ndst > INT_MAX)
        return FFDAS_ERROR_DIMS_TOO_LARGE;
    if (!packed(xd) || !packed(od)) return FFDAS_ERROR_NON_CONTIGUOUS;
    if (B * ndst * nfreq == 0) return FFDAS_SUCCESS;
    if (!srcpos || !wavenums || !x || !dstpos || !out) return FFDAS_ERROR_NULL_POINTER;
    if ((B + 3) / 4 > 65535 || (nfreq + kGreensFPT - 1) / kGreensFPT > 65535)
        return FFDAS_ERROR_DIMS_TOO_LARGE;
    return half_in ? launch<__half2>(handle->stream, srcpos, wavenums, x, dstpos, out, (int)nsrc,
                                     (int)nfreq, (int)ndst, (int)B)
                   : launch<float2>(handle->stream, srcpos, wavenums, x, dstpos, out, (int)nsrc,
                                    (int)nfreq, (int)ndst, (int)B);
}

extern "C" ffdas_error_t ffdas_greens(ffdas_handle_t handle, const float *srcpos,
                                      const float *wavenums, ffdas_tensor_desc_t x_desc,
                                      const void *x, const float *dstpos,
                                      ffdas_tensor_desc_t out_desc, void *out) {
    ffdas::CallScope cs(handle, "ffdas_greens");
    return cs.done(greens_call(handle, srcpos, wavenums, x_desc, x, dstpos, out_desc, out));
}
