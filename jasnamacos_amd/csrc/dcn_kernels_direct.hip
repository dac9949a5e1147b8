// Direct DCNv2 kernels: one thread per output element, summation in the CPU oracle's
// order (DeformConv.swift:98-135), no contraction. They are the FP32 entry point
// (deform_conv2d_fp32, MetalShader.swift:76-124) and the FP16 reference semantics
// (deform_conv2d_fp16, MetalShader.swift:126-174), for any valid shape.
//
// Bit-exactness rests on three facts: the file is compiled with -ffp-contract=off
// (and the pragma below), every FP16 operand widens exactly to FP32, and the
// bilinear expression keeps the reference's association
// ((v00*(1-ly))*(1-lx)) + ((v01*(1-ly))*lx) + ((v10*ly)*(1-lx)) + ((v11*ly)*lx).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "dcn_device.hpp"
#include "dcn_internal.hpp"

#pragma clang fp contract(off)

namespace dcn {
namespace {

template <typename T>
__device__ __forceinline__ float widen(T v);
template <>
__device__ __forceinline__ float widen<float>(float v) {
    return v;
}
template <>
__device__ __forceinline__ float widen<uint16_t>(uint16_t v) {
    return (float)__builtin_bit_cast(_Float16, v);
}

// DeformConvCPU.bilinear (DeformConv.swift:146-165); a corner outside the input is 0.
template <typename T>
__device__ __forceinline__ float bilinear(const T* __restrict__ input, long base, int height,
                                          int width, float y, float x) {
    // floor() of a finite float below 2^31 converts exactly; larger magnitudes are
    // clamped first so the conversion is defined (they are out of bounds either way).
    const float fy = fminf(fmaxf(floorf(y), -4.0f), (float)height + 4.0f);
    const float fx = fminf(fmaxf(floorf(x), -4.0f), (float)width + 4.0f);
    const int y0 = (int)fy;
    const int x0 = (int)fx;
    const int y1 = y0 + 1;
    const int x1 = x0 + 1;
    const float ly = y - floorf(y);
    const float lx = x - floorf(x);
    const bool ry0 = y0 >= 0 && y0 < height, ry1 = y1 >= 0 && y1 < height;
    const bool rx0 = x0 >= 0 && x0 < width, rx1 = x1 >= 0 && x1 < width;
    const float v00 = (ry0 && rx0) ? widen(input[base + (long)y0 * width + x0]) : 0.0f;
    const float v01 = (ry0 && rx1) ? widen(input[base + (long)y0 * width + x1]) : 0.0f;
    const float v10 = (ry1 && rx0) ? widen(input[base + (long)y1 * width + x0]) : 0.0f;
    const float v11 = (ry1 && rx1) ? widen(input[base + (long)y1 * width + x1]) : 0.0f;
    return v00 * (1.0f - ly) * (1.0f - lx) + v01 * (1.0f - ly) * lx +
           v10 * ly * (1.0f - lx) + v11 * ly * lx;
}

template <typename T>
__device__ __forceinline__ void store_out(T* out, long i, float v);
template <>
__device__ __forceinline__ void store_out<float>(float* out, long i, float v) {
    out[i] = v;
}
template <>
__device__ __forceinline__ void store_out<uint16_t>(uint16_t* out, long i, float v) {
    out[i] = __builtin_bit_cast(uint16_t, round_f16(v));  // half(sum), round to nearest even
}

template <typename T>
__global__ __launch_bounds__(256) void direct_kernel(const T* __restrict__ input,
                                                     const T* __restrict__ offset,
                                                     const T* __restrict__ mask,
                                                     const T* __restrict__ weight,
                                                     const T* __restrict__ bias,
                                                     T* __restrict__ output, KShape s,
                                                     long total) {
    const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= total) return;
    const long ox = gid % s.Wo;
    long q = gid / s.Wo;
    const long oy = q % s.Ho;
    q /= s.Ho;
    const long oc = q % s.Cout;
    const long n = q / s.Cout;
    const long cpg = s.Cin / s.groups;
    const long opg = s.Cout / s.groups;
    const long cpog = s.Cin / s.og;
    const long group = oc / opg;
    const long input_plane = (long)s.H * s.W;
    const long output_plane = (long)s.Ho * s.Wo;
    const long kernel_area = (long)s.KH * s.KW;
    const long spatial = oy * s.Wo + ox;
    const long offset_base = n * 2 * s.og * kernel_area * output_plane;
    const long mask_base = n * s.og * kernel_area * output_plane;
    float sum = widen(bias[oc]);
    for (long local_ic = 0; local_ic < cpg; ++local_ic) {
        const long ic = group * cpg + local_ic;
        const long og = ic / cpog;
        const long input_base = (n * s.Cin + ic) * input_plane;
        for (long ky = 0; ky < s.KH; ++ky) {
            for (long kx = 0; kx < s.KW; ++kx) {
                const long k = ky * s.KW + kx;
                const long offset_channel = 2 * (og * kernel_area + k);
                const float off_y = widen(offset[offset_base + offset_channel * output_plane + spatial]);
                const float off_x =
                    widen(offset[offset_base + (offset_channel + 1) * output_plane + spatial]);
                const float y = (float)(oy * s.sh - s.ph + ky * s.dh) + off_y;
                const float x = (float)(ox * s.sw - s.pw + kx * s.dw) + off_x;
                const float sampled = bilinear(input, input_base, s.H, s.W, y, x);
                const float m = widen(mask[mask_base + (og * kernel_area + k) * output_plane + spatial]);
                const float w = widen(weight[((oc * cpg + local_ic) * s.KH + ky) * s.KW + kx]);
                sum += sampled * m * w;
            }
        }
    }
    store_out(output, gid, sum);
}

template <typename T>
hipError_t launch_direct(const KShape& s, const T* in, const T* off, const T* mask, const T* w,
                         const T* b, T* out, hipStream_t stream) {
    const long total = (long)s.B * s.Cout * s.Ho * s.Wo;
    const int block = 256;
    const long grid = (total + block - 1) / block;
    if (grid <= 0) return hipSuccess;
    hipLaunchKernelGGL(direct_kernel<T>, dim3((unsigned)grid), dim3(block), 0, stream, in, off,
                       mask, w, b, out, s, total);
    return hipGetLastError();
}

// ---- shared samples --------------------------------------------------------------------
// direct_kernel evaluates every bilinear sample once per output channel. Here a workgroup
// owns 16 output pixels x OC output channels of one group: each (pixel, ic, tap) sample is
// evaluated once, as sampled * mask, into LDS, and every output channel of the workgroup
// reads it there. Each output still sums bias, then ic, ky, kx in order, as
// sum + ((sampled * mask) * weight) with one rounding per operation (no contraction), so
// the result is direct_kernel's, and the oracle's, bit for bit.
//
// Bound: one FP32 multiply and one add per (output, ic, tap), 604 M lane operations at
// 1x128x64x64 -> 64, 15.4 us at 64 per CU and clock. With both operands read from LDS a wave's
// two 16-byte reads per 4 taps cost 64 of a CU's LDS clocks for 32 of its VALU's (34.9 us),
// so only the samples come from LDS: lane l holds pixel l % 16 of output channels
// OCL * (l / 16) + e, the 16 lanes of a row share their channels, and each keeps one weight of
// every 16 consecutive (ic, tap) in a register that the multiply reads through a DPP row
// broadcast (4.2 clocks against 3.1 for a plain multiply, measured). Weights go from memory
// to registers, one whole stage ahead; the stage is in the load's scalar offset, which the
// buffer's range check may leave out, so these loads stay inside a channel's run by
// themselves (shared_stage_start), and the partial stage's have their address in the vector
// offset. 34.9 -> 28.0 us FP32; FP16 2x128x45x61 -> 64, which ran
// direct_kernel, 1584 -> 48.7 us (343 workgroups on 256 CUs; 45x61 alone 25.5 us). The corner
// gathers come next: a pixel's samples are a cache line per channel and corner row, so the
// two columns of a row are one load (four single loads: 38.6 us against 28.0).
//
// NW waves run the chains and SW more sample: the input channels go by in stages of 16
// (J = 16 * KA samples per pixel, KA chunks of 16); while the chains consume stage st from
// one LDS buffer, the sampling waves fill the other with stage st + 1 and request the
// offsets of stage st + 2. In the chains' own waves each wait for a weight would
// also wait for the gathers. A sampling item is one (pixel, tap) of CPI channels that
// share an offset group: position and corner weights once, CPI x 4 corner loads.
constexpr int kSharedPix = 16;

template <typename T>
struct SharedArgs {
    const T *input, *offset, *mask, *weight, *bias;
    T* output;
    KShape s;
    long pixels;
    int cpg, opg, cpog;   // channels per group, output channels per group, channels per offset group
    int oc_tiles;         // workgroups along one group's output channels
    uint32_t off_bytes, mask_bytes, weight_bytes;
};

constexpr int shared_sampling_waves(int ka, int cpi) {
    const int items = kSharedPix * ka * (kSharedCh / cpi);
    return items >= 512 ? 8 : (items + 63) / 64;
}
template <int KA, int CPI>
struct SharedLayout {
    static constexpr int J = kSharedCh * KA;
    static constexpr int JP = J + 4;  // padded row (floats): 16-byte aligned rows, odd in 16-byte units
    static constexpr int ITEMS = kSharedPix * KA * (kSharedCh / CPI);
    static constexpr int SW = shared_sampling_waves(KA, CPI);
    static constexpr int PER = (ITEMS + 64 * SW - 1) / (64 * SW);    // items per sampling lane
};

template <typename T>
__device__ __forceinline__ float load_widened(__amdgpu_buffer_rsrc_t r, uint32_t element, uint32_t soff = 0) {
    if constexpr (sizeof(T) == 4)
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)(element * 4u), (int)soff, 0));
    return dev::load_half(r, element * 2u, soff);
}

// Two neighbouring elements of a row, one load (any element alignment).
template <typename T>
struct Pair;
template <>
struct Pair<float> {
    float2 v;
};
template <>
struct Pair<uint16_t> {
    uint32_t v;
};
template <typename T>
__device__ __forceinline__ Pair<T> load_pair(const T* p) {
    Pair<T> r;
    __builtin_memcpy(&r.v, p, 2 * sizeof(T));
    return r;
}
__device__ __forceinline__ float first(const Pair<float>& p) { return p.v.x; }
__device__ __forceinline__ float second(const Pair<float>& p) { return p.v.y; }
__device__ __forceinline__ float first(const Pair<uint16_t>& p) { return widen((uint16_t)p.v); }
__device__ __forceinline__ float second(const Pair<uint16_t>& p) { return widen((uint16_t)(p.v >> 16)); }

// t[i] = s[i] * w of lane 4 Q + i of the caller's row of 16 lanes. In assembly because the
// compiler makes the broadcasts of a whole stage first, as moves, and spills them. A DPP
// operand may not have been written by the two vector instructions before: s_nop at the
// chunk's first use of w, which the volatile order keeps first.
template <int Q>
__device__ __forceinline__ void row_products(const float4& s, float w, float (&t)[4]) {
    if constexpr (Q == 0)
        __asm__ volatile(
            "s_nop 1\n\t"
            "v_mul_f32_dpp %0, %4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
            "v_mul_f32_dpp %1, %4, %6 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
            "v_mul_f32_dpp %2, %4, %7 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
            "v_mul_f32_dpp %3, %4, %8 row_newbcast:%12 row_mask:0xf bank_mask:0xf"
            : "=&v"(t[0]), "=&v"(t[1]), "=&v"(t[2]), "=&v"(t[3])
            : "v"(w), "v"(s.x), "v"(s.y), "v"(s.z), "v"(s.w), "n"(4 * Q), "n"(4 * Q + 1), "n"(4 * Q + 2), "n"(4 * Q + 3));
    else
        __asm__ volatile(
            "v_mul_f32_dpp %0, %4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
            "v_mul_f32_dpp %1, %4, %6 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
            "v_mul_f32_dpp %2, %4, %7 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
            "v_mul_f32_dpp %3, %4, %8 row_newbcast:%12 row_mask:0xf bank_mask:0xf"
            : "=&v"(t[0]), "=&v"(t[1]), "=&v"(t[2]), "=&v"(t[3])
            : "v"(w), "v"(s.x), "v"(s.y), "v"(s.z), "v"(s.w), "n"(4 * Q), "n"(4 * Q + 1), "n"(4 * Q + 2), "n"(4 * Q + 3));
}

// The first `count` of samples 4 Q .. 4 Q + 3 of a chunk: sum + (sample * weight), in order.
template <int Q, int OCL, bool ALL>
__device__ __forceinline__ void chain4(float (&acc)[OCL], const float4& s, const float (&w)[OCL], int count) {
    float t[OCL][4];
#pragma unroll
    for (int e = 0; e < OCL; ++e) row_products<Q>(s, w[e], t[e]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < OCL; ++e)
            if (ALL || i < count) acc[e] = acc[e] + t[e][i];
}

template <typename T, int KA, int NW, int OCL, int CPI>
__global__ __launch_bounds__(64 * (NW + SharedLayout<KA, CPI>::SW)) void shared_kernel(SharedArgs<T> a) {
    using L = SharedLayout<KA, CPI>;
    constexpr int JP = L::JP;
    __shared__ __attribute__((aligned(16))) float sm[2][kSharedPix][JP];  // sampled * mask
    const KShape& s = a.s;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p = threadIdx.x & 15;
    const int group = blockIdx.y / a.oc_tiles;
    const long pix0 = (long)blockIdx.x * kSharedPix;
    const long plane = (long)s.Ho * s.Wo;
    const long pix = min(pix0 + p, a.pixels - 1);
    const int n = (int)(pix / plane);
    const int spatial = (int)(pix - n * plane);
    const int stages = (a.cpg + kSharedCh - 1) / kSharedCh;

    if (wave >= NW) {
        // Sampling waves: item t = (tap, channel block) * 16 + pixel. Lanes past the last
        // item repeat it (the same value to the same place).
        const int oy = spatial / s.Wo;
        const int ox = spatial - oy * s.Wo;
        const uint32_t in_plane = (uint32_t)s.H * s.W;
        const __amdgpu_buffer_rsrc_t offr = dev::make_rsrc(a.offset, a.off_bytes);
        const __amdgpu_buffer_rsrc_t maskr = dev::make_rsrc(a.mask, a.mask_bytes);
        int k[L::PER], ch[L::PER];
        float y0f[L::PER], x0f[L::PER];
#pragma unroll
        for (int i = 0; i < L::PER; ++i) {
            const int rest = min((int)(threadIdx.x - 64 * NW + 64 * L::SW * i) >> 4, L::ITEMS / 16 - 1);
            k[i] = rest % KA;
            ch[i] = rest / KA * CPI;
            const int ky = k[i] / s.KW;
            y0f[i] = (float)(oy * s.sh - s.ph + ky * s.dh);
            x0f[i] = (float)(ox * s.sw - s.pw + (k[i] - ky * s.KW) * s.dw);
        }
        float ofy[L::PER], ofx[L::PER], mk[L::PER];
        // Offsets and masks of stage st; channels past the group's repeat its last block.
        auto channel = [&](int st, int i) { return min(st * kSharedCh + ch[i], a.cpg - CPI); };
        auto load_stage = [&](int st) {
#pragma unroll
            for (int i = 0; i < L::PER; ++i) {
                const int og = (group * a.cpg + channel(st, i)) / a.cpog;
                const uint32_t m = (uint32_t)((n * s.og + og) * KA + k[i]) * (uint32_t)plane + spatial;
                const uint32_t o = m * 2 - spatial;
                ofy[i] = load_widened<T>(offr, o);
                ofx[i] = load_widened<T>(offr, o + (uint32_t)plane);
                mk[i] = load_widened<T>(maskr, m);
            }
        };
        // Stage st's samples (DeformConvCPU.bilinear's association; a corner outside the
        // input reads 0) times the mask into buffer st % 2; the next stage's offsets are
        // requested behind the corners.
        auto sample_stage = [&](int st, bool more) {
            Pair<T> top[L::PER][CPI], low[L::PER][CPI];
            float ly[L::PER], lx[L::PER], m[L::PER];
            bool ry0[L::PER], ry1[L::PER], rx0[L::PER], rx1[L::PER], shift[L::PER];
#pragma unroll
            for (int i = 0; i < L::PER; ++i) {
                const float y = y0f[i] + ofy[i];
                const float x = x0f[i] + ofx[i];
                m[i] = mk[i];
                const float fy = floorf(y), fx = floorf(x);
                ly[i] = y - fy;
                lx[i] = x - fx;
                // floor() of a finite float converts exactly once clamped (clamped values are
                // out of bounds either way; NaN clamps to the lower bound).
                const int y0 = (int)fminf(fmaxf(fy, -4.0f), (float)s.H + 4.0f);
                const int x0 = (int)fminf(fmaxf(fx, -4.0f), (float)s.W + 4.0f);
                ry0[i] = y0 >= 0 && y0 < s.H;
                ry1[i] = y0 + 1 >= 0 && y0 + 1 < s.H;
                rx0[i] = x0 >= 0 && x0 < s.W;
                rx1[i] = x0 + 1 >= 0 && x0 + 1 < s.W;
                // The pair of columns loaded: x0 and x0 + 1, moved into the row at its ends.
                const int xb = min(max(x0, 0), s.W - 2);
                shift[i] = xb != x0;
                const uint32_t plane0 = (uint32_t)(n * s.Cin + group * a.cpg + channel(st, i)) * in_plane + xb;
                const T* r0 = a.input + (plane0 + (uint32_t)(min(max(y0, 0), s.H - 1) * s.W));
                const T* r1 = a.input + (plane0 + (uint32_t)(min(max(y0 + 1, 0), s.H - 1) * s.W));
#pragma unroll
                for (int c = 0; c < CPI; ++c) {
                    top[i][c] = load_pair<T>(r0 + (size_t)c * in_plane);
                    low[i][c] = load_pair<T>(r1 + (size_t)c * in_plane);
                }
            }
            if (more) load_stage(st + 1);
#pragma unroll
            for (int i = 0; i < L::PER; ++i) {
                const float cy = 1.0f - ly[i], cx = 1.0f - lx[i];
                // A moved pair holds column x0 second (x0 the last column) or x0 + 1 first.
                const bool a0 = ry0[i] && rx0[i], a1 = ry0[i] && rx1[i], b0 = ry1[i] && rx0[i], b1 = ry1[i] && rx1[i];
#pragma unroll
                for (int c = 0; c < CPI; ++c) {
                    const float t0 = first(top[i][c]), t1 = second(top[i][c]);
                    const float u0 = first(low[i][c]), u1 = second(low[i][c]);
                    const float v00 = a0 ? (shift[i] ? t1 : t0) : 0.0f;
                    const float v01 = a1 ? (shift[i] ? t0 : t1) : 0.0f;
                    const float v10 = b0 ? (shift[i] ? u1 : u0) : 0.0f;
                    const float v11 = b1 ? (shift[i] ? u0 : u1) : 0.0f;
                    const float sampled = v00 * cy * cx + v01 * cy * lx[i] + v10 * ly[i] * cx + v11 * ly[i] * lx[i];
                    sm[st & 1][p][(ch[i] + c) * KA + k[i]] = sampled * m[i];
                }
            }
        };
        load_stage(0);
        for (int st = 0; st < stages; ++st) {
            sample_stage(st, st + 1 < stages);
            __syncthreads();  // stage st is ready; stage st - 1's buffer is free
        }
        if (a.cpg % kSharedCh == 0) __syncthreads();  // the chains' barrier after their last whole stage
        return;
    }

    // Chain waves. This row's weights: chunk c of a stage is lane p's element 16 c + p of the
    // stage's (ic, tap) run. Channels past the group's load its last one. Elements past a
    // channel's run (in a partial stage) are the next one's or, past the tensor, zero (the
    // buffer's range check): nothing uses them.
    const int oc0 = (blockIdx.y - group * a.oc_tiles) * (4 * NW * OCL) + (threadIdx.x >> 4) * OCL;  // in the group
    const __amdgpu_buffer_rsrc_t wr = dev::make_rsrc(a.weight, a.weight_bytes);
    uint32_t wbase[OCL];
    float acc[OCL], w[KA][OCL];
#pragma unroll
    for (int e = 0; e < OCL; ++e) {
        const int oc = group * a.opg + min(oc0 + e, a.opg - 1);
        wbase[e] = (uint32_t)oc * (uint32_t)(a.cpg * KA) + p;
        acc[e] = widen(a.bias[oc]);
    }
    const int full = a.cpg / kSharedCh;  // whole stages
    auto load_weights = [&](int st, int c) {
        const uint32_t soff = (uint32_t)(shared_stage_start(st, full, KA) + 16 * c) * (uint32_t)sizeof(T);
#pragma unroll
        for (int e = 0; e < OCL; ++e) w[c][e] = load_widened<T>(wr, wbase[e], soff);
    };
    auto load_run = [&](int j0, float (&v)[OCL]) {
#pragma unroll
        for (int e = 0; e < OCL; ++e) v[e] = load_widened<T>(wr, wbase[e] + (uint32_t)j0);
    };
    auto row4 = [&](int nb, int j) { return *reinterpret_cast<const float4*>(&sm[nb][p][j]); };
    // The first stage unconditionally: under a branch the compiler converts FP16 weights as they
    // are loaded, stage by stage (2x128x45x61 56.6 us against 47.9).
#pragma unroll
    for (int c = 0; c < KA; ++c) load_run(16 * c, w[c]);
    __syncthreads();
#pragma unroll 1
    for (int st = 0; st < full; ++st) {
        const int nb = st & 1;
#pragma unroll
        for (int c = 0; c < KA; ++c) {
            const float4 s0 = row4(nb, 16 * c), s1 = row4(nb, 16 * c + 4);
            const float4 s2 = row4(nb, 16 * c + 8), s3 = row4(nb, 16 * c + 12);
            chain4<0, OCL, true>(acc, s0, w[c], 4);
            chain4<1, OCL, true>(acc, s1, w[c], 4);
            chain4<2, OCL, true>(acc, s2, w[c], 4);
            chain4<3, OCL, true>(acc, s3, w[c], 4);
            load_weights(st + 1, c);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
    }
    if (full < stages) {
        // The last, partial stage: its weights again, a chunk ahead.
        const int nb = full & 1;
        const int count = (a.cpg - full * kSharedCh) * KA;
        load_run(full * L::J, w[0]);
#pragma unroll 1
        for (int c = 0; 16 * c < count; ++c) {
            float wt[OCL];
#pragma unroll
            for (int e = 0; e < OCL; ++e) wt[e] = w[0][e];
            load_run(full * L::J + 16 * (c + 1), w[0]);
            const int left = count - 16 * c;
            const float4 s0 = row4(nb, 16 * c), s1 = row4(nb, 16 * c + 4);
            const float4 s2 = row4(nb, 16 * c + 8), s3 = row4(nb, 16 * c + 12);
            if (left >= 16) {
                chain4<0, OCL, true>(acc, s0, wt, 4);
                chain4<1, OCL, true>(acc, s1, wt, 4);
                chain4<2, OCL, true>(acc, s2, wt, 4);
                chain4<3, OCL, true>(acc, s3, wt, 4);
            } else {
                chain4<0, OCL, false>(acc, s0, wt, left);
                chain4<1, OCL, false>(acc, s1, wt, left - 4);
                chain4<2, OCL, false>(acc, s2, wt, left - 8);
                chain4<3, OCL, false>(acc, s3, wt, left - 12);
            }
        }
    }

    if (pix0 + p >= a.pixels) return;
#pragma unroll
    for (int e = 0; e < OCL; ++e)
        if (oc0 + e < a.opg)
            store_out(a.output, ((long)n * s.Cout + group * a.opg + oc0 + e) * plane + spatial, acc[e]);
}

template <typename T, int KA, int NW, int OCL, int CPI>
hipError_t launch_shared_as(SharedArgs<T> a, hipStream_t stream) {
    constexpr int OC = 4 * NW * OCL;
    a.oc_tiles = (a.opg + OC - 1) / OC;
    const dim3 grid((unsigned)((a.pixels + kSharedPix - 1) / kSharedPix), (unsigned)(a.s.groups * a.oc_tiles));
    hipLaunchKernelGGL((shared_kernel<T, KA, NW, OCL, CPI>), grid, dim3(64 * (NW + SharedLayout<KA, CPI>::SW)), 0,
                       stream, a);
    return hipGetLastError();
}

// Output channels per workgroup: the fewest whose workgroups still fit the 256 CUs at once
// (more CUs busy beat the samples evaluated again per channel tile), else as many as the
// group has, up to 64. Measured for 128 -> 64 channels FP32, us at 16 / 32 / 64 channels:
// 32x32 pixels (64 pixel tiles) 17.0 / 18.4 / 22.6, 45x61 (172) 41.9 / 34.9 / 25.5, 64x64 (256)
// 69.5 / 34.3 / 28.0. Up to 16 channels on more than 256 workgroups take two chain waves of
// two channels per lane: 2x60x60, 4 groups of 24 -> 10, 30.3 -> 26.5 us.
struct SharedSplit {
    int nw, ocl;  // chain waves, output channels per lane
};
SharedSplit shared_split(long tiles, int opg) {
    const auto fits = [&](int oc) { return tiles * ((opg + oc - 1) / oc) <= 256; };
    if (fits(16)) return {4, 1};
    if (opg <= 16) return {2, 2};
    if (opg <= 32 || fits(32)) return {4, 2};
    return {8, 2};
}
// Pixel tiles over all groups.
long shared_tiles(const KShape& s) {
    return ((long)s.B * s.Ho * s.Wo + kSharedPix - 1) / kSharedPix * s.groups;
}
// Input channels of a sampling item.
int shared_item_channels(const KShape& s) {
    if (s.KH * s.KW != 9) return 1;
    const int both = (s.Cin / s.groups) | (s.Cin / s.og);
    return both % 8 == 0 ? 8 : both % 4 == 0 ? 4 : 1;
}

template <typename T, int KA, int CPI>
hipError_t launch_shared_ka(const SharedArgs<T>& a, hipStream_t stream) {
    const SharedSplit p = shared_split(shared_tiles(a.s), a.opg);
    if (p.nw == 2) return launch_shared_as<T, KA, 2, 2, CPI>(a, stream);
    if (p.nw == 8) return launch_shared_as<T, KA, 8, 2, CPI>(a, stream);
    return p.ocl == 1 ? launch_shared_as<T, KA, 4, 1, CPI>(a, stream) : launch_shared_as<T, KA, 4, 2, CPI>(a, stream);
}

template <typename T>
hipError_t launch_forward(const KShape& s, const T* in, const T* off, const T* mask, const T* w, const T* b, T* out,
                          hipStream_t stream) {
    if (!shared_forward_chosen(s, sizeof(T))) return launch_direct<T>(s, in, off, mask, w, b, out, stream);
    SharedArgs<T> a{in, off, mask, w, b, out, s, (long)s.B * s.Ho * s.Wo, s.Cin / s.groups, s.Cout / s.groups,
                    s.Cin / s.og, 0, 0, 0, 0};
    const int ka = s.KH * s.KW;
    a.mask_bytes = (uint32_t)((size_t)a.pixels * s.og * ka * sizeof(T));
    a.off_bytes = 2 * a.mask_bytes;
    a.weight_bytes = (uint32_t)((size_t)s.Cout * a.cpg * ka * sizeof(T));
    switch (ka) {
        case 1: return launch_shared_ka<T, 1, 1>(a, stream);
        case 2: return launch_shared_ka<T, 2, 1>(a, stream);
        case 3: return launch_shared_ka<T, 3, 1>(a, stream);
        case 4: return launch_shared_ka<T, 4, 1>(a, stream);
        case 6: return launch_shared_ka<T, 6, 1>(a, stream);
        default: break;
    }
    switch (shared_item_channels(s)) {
        case 8: return launch_shared_ka<T, 9, 8>(a, stream);
        case 4: return launch_shared_ka<T, 9, 4>(a, stream);
        default: return launch_shared_ka<T, 9, 1>(a, stream);
    }
}

}  // namespace

bool shared_forward_chosen(const KShape& s, size_t element) {
    const int ka = s.KH * s.KW, opg = s.Cout / s.groups;
    if (!(ka == 1 || ka == 2 || ka == 3 || ka == 4 || ka == 6 || ka == 9) || s.W < 2) return false;
    // The kernel addresses each tensor with 32-bit byte offsets below 2^31 and its sampling
    // positions with 32-bit integers; grid y is one workgroup column per group and channel
    // tile, and a launch has fewer than 2^32 threads along x.
    const double limit = 2147483648.0;
    const double in_bytes = (double)s.B * s.Cin * s.H * s.W * element;
    const double off_bytes = 2.0 * s.B * s.Ho * s.Wo * s.og * ka * element;
    const double weight_bytes = (double)s.Cout * (s.Cin / s.groups) * ka * element;
    // Strides, dilations and pads may have either sign.
    const auto reach = [](double out, double stride, double pad, double taps, double dilation) {
        return out * std::fabs(stride) + std::fabs(pad) + taps * std::fabs(dilation);
    };
    if (in_bytes >= limit || off_bytes >= limit || weight_bytes >= limit ||
        reach(s.Ho, s.sh, s.ph, s.KH, s.dh) >= 1e9 || reach(s.Wo, s.sw, s.pw, s.KW, s.dw) >= 1e9 ||
        (double)s.groups * ((opg + 15) / 16) >= 65536.0)
        return false;
    const long tiles = shared_tiles(s);
    const SharedSplit split = shared_split(tiles, opg);
    const int items = shared_item_channels(s);
    if ((double)(tiles / s.groups) * (split.nw + shared_sampling_waves(ka, items)) * 64 >= 4294967296.0) return false;
    // Groups of few channels: a workgroup samples 16 input channels and sums 16 output channels
    // or more however few the group has, so depthwise layers and their like run one thread per
    // output, where there are enough of them. Fitted to both kernels' times over 946 layers
    // (FP32 and FP16; 1, 4, 9 taps; 256 to 262,144 pixels; 1 to 128 channels a group): the
    // shared-sample kernel 1.3 ns per workgroup, stage and tap (0.6 with items of eight
    // channels), the other 5 ps per sample and output (FP16 4.5) or, with few outputs, 0.6 us
    // per sample of one. us per call, shared / one thread per output, FP16: 64 groups of 1 -> 1
    // on 64x64 221 / 12.6 and on 180x320 3182 / 207, 3 groups of 2 -> 2 there 158 / 44, 16
    // of 4 -> 4 on 64x64 47.7 / 41.6, 3 -> 3 on 64x64 5.9 / 20.9, 8 groups of 4 -> 8 there
    // 25.7 / 40.6. From two whole stages on the samples' sharing wins in nearly all.
    const int cpg = s.Cin / s.groups, oc = 4 * split.nw * split.ocl;
    if (cpg >= 2 * kSharedCh) return true;
    const double samples = (double)s.B * s.Ho * s.Wo * s.Cout * cpg * ka;
    const double direct_us = std::max(0.6 * cpg * ka, samples * (element == 2 ? 4.5e-6 : 5e-6));
    const double shared_us = (double)tiles * ((opg + oc - 1) / oc) * ((cpg + kSharedCh - 1) / kSharedCh) * ka *
                             (items == 8 ? 0.6e-3 : 1.3e-3);
    return shared_us <= direct_us;
}

hipError_t launch_direct_f32(const KShape& s, const float* in, const float* off,
                             const float* mask, const float* w, const float* b, float* out,
                             hipStream_t stream) {
    return launch_forward<float>(s, in, off, mask, w, b, out, stream);
}

hipError_t launch_direct_f16(const KShape& s, const uint16_t* in, const uint16_t* off,
                             const uint16_t* mask, const uint16_t* w, const uint16_t* b,
                             uint16_t* out, hipStream_t stream) {
    return launch_forward<uint16_t>(s, in, off, mask, w, b, out, stream);
}

}  // namespace dcn
