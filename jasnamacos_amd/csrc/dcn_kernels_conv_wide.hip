// The body's 3x3 convolutions over many pixels (large maps, batches of tiles): 16-wide
// output tiles whose input stays in LDS, so that a weight fragment serves a hundred pixels
// or more instead of sixteen.
//
// Same arithmetic, bit for bit, as dcn_kernels_conv.hip: K-step s multiplies K-blocks 4 s ..
// 4 s + 3 (K-block tap * CB + cb) on v_mfma_f32_16x16x32_f16, the K-steps of each eighth of
// the range [r * ksteps / 8, (r + 1) * ksteps / 8) form one accumulator chain from zero, and
// the eight partial sums are added in order. There eight waves own an eighth each and add
// through LDS; here one wave runs all eighths of its pixels and adds in registers. The
// operands swap places (weights in A, pixels in B): the products and their order are the
// same, and a lane then holds four consecutive channels of one pixel, an 8-byte store.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "dcn_device.hpp"
#include "dcn_internal.hpp"

#pragma clang fp contract(off)

namespace dcn {
namespace {

using namespace dev;

constexpr int kWideTW = 16;  // output tile width
constexpr int kSteps64 = 18;  // K-steps of 64 input channels

struct WidePairArgs {
    const void* xin;
    const void* wpk1;
    const void* wpk2;
    const float* bias1;
    const float* bias2;
    const uint16_t* res1;
    const uint16_t* res2;
    uint16_t* out;
    uint16_t* out2;
    uint32_t xin_bytes, wpk_bytes;
    int act1, act2;
    float slope;
    int res1_layout, res2_layout, out_layout, res2_coff;
    int H, W, Hp, Wp, tiles_x, tiles_image, tiles;
    long xin_ts, res1_ts, res2_ts, out_ts, out2_ts;
};

// Four consecutive channels c .. c + 3 (c % 4 == 0) of pixel (y, x).
struct Half4 {
    uint32_t v[2];
};
__device__ __forceinline__ float half_at(const Half4& h, int i) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(h.v[i >> 1] >> (16 * (i & 1))));
}
struct Place {
    int H, W, pad;  // image, and border of a CB8 tensor
};
// The first `live` of them of an NCHW tensor (a CB8 one holds all four).
__device__ __forceinline__ Half4 load4(const uint16_t* t, int layout, int c, int y, int x, const Place& a, int live = 4) {
    Half4 r;
    if (layout == kLayoutCB8) {
        const size_t unit = ((size_t)(c >> 3) * (a.H + 2 * a.pad) + y + a.pad) * (a.W + 2 * a.pad) + x + a.pad;
        const uint2 u = *reinterpret_cast<const uint2*>(t + unit * 8 + (c & 7));
        r.v[0] = u.x;
        r.v[1] = u.y;
    } else {
        const size_t plane = (size_t)a.H * a.W;
        const uint16_t* p = t + (size_t)c * plane + (size_t)y * a.W + x;
        const uint32_t h0 = p[0], h1 = live > 1 ? p[plane] : 0u;
        const uint32_t h2 = live > 2 ? p[2 * plane] : 0u, h3 = live > 3 ? p[3 * plane] : 0u;
        r.v[0] = h0 | (h1 << 16);
        r.v[1] = h2 | (h3 << 16);
    }
    return r;
}
__device__ __forceinline__ void store4(uint16_t* t, int layout, int c, int y, int x, const Place& a, const Half4& h,
                                       int live = 4) {
    if (layout == kLayoutCB8) {
        const size_t unit = ((size_t)(c >> 3) * (a.H + 2 * a.pad) + y + a.pad) * (a.W + 2 * a.pad) + x + a.pad;
        *reinterpret_cast<uint2*>(t + unit * 8 + (c & 7)) = make_uint2(h.v[0], h.v[1]);
    } else {
        const size_t plane = (size_t)a.H * a.W;
        uint16_t* p = t + (size_t)c * plane + (size_t)y * a.W + x;
        p[0] = (uint16_t)h.v[0];
        if (live > 1) p[plane] = (uint16_t)(h.v[0] >> 16);
        if (live > 2) p[2 * plane] = (uint16_t)h.v[1];
        if (live > 3) p[3 * plane] = (uint16_t)(h.v[1] >> 16);
    }
}
__device__ __forceinline__ Half4 pack4(const float (&f)[4]) {
    Half4 h;
#pragma unroll
    for (int i = 0; i < 2; ++i)
        h.v[i] = (uint32_t)__builtin_bit_cast(uint16_t, round_f16(f[2 * i])) |
                 ((uint32_t)__builtin_bit_cast(uint16_t, round_f16(f[2 * i + 1])) << 16);
    return h;
}
__device__ __forceinline__ float activate(float v, int act, float slope) {
    if (act == 1 && v < 0.0f) v = v * slope;
    if (act == 2 && v < 0.0f) v = 0.0f;
    return v;
}

// 64 input channels over P 16-pixel groups and two 16-channel blocks: the sums of a tile
// whose pixel units are in LDS as [8 blocks][PLANE], rows ROW apart, `base` the byte address
// of each group's lane unit (block lane / 16, tap (0, 0)).
template <int P, int PLANE, int ROW>
__device__ __forceinline__ void gemm64(const uint8_t* lds, const uint32_t (&base)[P], __amdgpu_buffer_rsrc_t wr,
                                       uint32_t wlane, f32x4 (&sum)[P][2]) {
    // Everything is requested in the order it is used: the weights of the next eighth at the
    // start of this one, the pixels of the next K-step before this one's products. Left to
    // itself the compiler requests far more at once than the registers hold.
    h8 B[2][3][2];
    h8 X[2][P];
    auto load_weights = [&](int r) {
        __asm__ volatile("" : "+v"(wlane));
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int s = r * kSteps64 / 8 + i;
            if (s >= (r + 1) * kSteps64 / 8) continue;
#pragma unroll
            for (int n = 0; n < 2; ++n)
                B[r & 1][i][n] = __builtin_bit_cast(h8, load16(wr, wlane, (uint32_t)(s * 4 + n) * 1024u));
        }
    };
    auto load_pixels = [&](int s) {
        const int tap = s >> 1;
        const uint32_t off = (uint32_t)((s & 1) * 4 * PLANE + tap / 3 * ROW + tap % 3) * 16u;
#pragma unroll
        for (int p = 0; p < P; ++p) X[s & 1][p] = *reinterpret_cast<const h8*>(lds + base[p] + off);
    };
    f32x4 acc[P][2];
    load_weights(0);
    load_pixels(0);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        if (r < 7) load_weights(r + 1);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int s = r * kSteps64 / 8 + i;
            if (s >= (r + 1) * kSteps64 / 8) continue;
            if (s + 1 < kSteps64) load_pixels(s + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int p = 0; p < P; ++p)
#pragma unroll
                for (int n = 0; n < 2; ++n)
                    acc[p][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(B[r & 1][i][n], X[s & 1][p],
                                                                       i == 0 ? f32x4{} : acc[p][n], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                // A chain from +0 never ends in -0, so the first partial sum is the sum from 0.
                if (r == 0)
                    sum[p][n] = acc[p][n];
                else
#pragma unroll
                    for (int v = 0; v < 4; ++v) sum[p][n][v] = sum[p][n][v] + acc[p][n][v];
                __asm__ volatile("" : "+v"(sum[p][n]));  // added now: eight sets of partial sums do not fit
            }
    }
}

template <int TH, int PG>
struct WidePair {
    static constexpr int NW = 2 * PG;  // waves: PG pixel groups x 2 halves of 64 output channels
    static constexpr int IW = kWideTW + 4, IPX = (TH + 4) * IW;     // input tile
    static constexpr int HW = kWideTW + 2, HPX = (TH + 2) * HW;     // halo of the tile: t
    static constexpr int P1 = ((HPX + 15) / 16 + PG - 1) / PG;  // 16-pixel groups per wave, conv1
    static constexpr int P2 = (TH + PG - 1) / PG;          // conv2: one row each
    static constexpr size_t lds = (size_t)8 * (IPX + HPX) * 16;
};

// Two chained 64 -> 64 convs (conv_pair_kernel's contract) on a TH x 16 output tile. The
// input tile (two pixels more on each side) is copied into LDS once; conv1 runs over the
// tile's halo into LDS, conv2 from there. Each wave multiplies PG-th rows of pixels by one
// half of the output channels: a pixel fragment (LDS) serves two products and a weight
// fragment (L1) up to P1. At 180 x 320 (240 tiles of 16 x 16, one per CU) 78 -> 17.3 us, 490
// TFLOP/s, against conv_pair_kernel, whose 3,600 workgroups fetch all 148 KB of weights for 16
// pixels each; 16 maps of 64 x 64 53 -> 18 us. No pipe is full (counters, per CU of 35.7 K cycles
// at 180 x 320: matrix cores 32 %, other VALU 36 %, LDS 33 % with 45 % of that in bank conflicts,
// addresser 48 %): with two waves per SIMD and one round of workgroups the time is the latency
// of the copy and of two dependent convs.
template <int TH, int PG>
__global__ __launch_bounds__((64 * WidePair<TH, PG>::NW)) void conv_pair_wide_kernel(WidePairArgs a) {
    using L = WidePair<TH, PG>;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    u32x4* xt = reinterpret_cast<u32x4*>(lds);                   // [8][IPX]
    uint8_t* tt = lds + (size_t)8 * L::IPX * 16;                 // [8][HPX] units
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = wave >> 1;
    const int half = wave & 1;
    const int quarter = lane >> 4;

    const int per_xcd = (a.tiles + 7) / 8;
    const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tile >= a.tiles) return;  // whole workgroup, before any barrier
    const int z = tile / a.tiles_image;
    const int ti = tile - z * a.tiles_image;
    const int ty = ti / a.tiles_x;
    const int oy0 = ty * TH;
    const int ox0 = (ti - ty * a.tiles_x) * kWideTW;

    // Input unit (block, row, column) of the tile; past the padded plane a clamped one, which
    // only reaches outputs outside the image.
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(static_cast<const uint16_t*>(a.xin) + z * a.xin_ts, a.xin_bytes);
    constexpr int kUnits = 8 * L::IPX;
    constexpr int kIter = (kUnits + 64 * L::NW - 1) / (64 * L::NW);
    u32x4 q[kIter];
#pragma unroll
    for (int j = 0; j < kIter; ++j) {
        const int u = min(tid + j * 64 * L::NW, kUnits - 1);
        const int cb = u / L::IPX;
        const int r = u - cb * L::IPX;
        const int row = r / L::IW;
        const int py = min(oy0 + row, a.Hp - 1);
        const int px = min(ox0 + r - row * L::IW, a.Wp - 1);
        q[j] = load16(xr, (uint32_t)((cb * a.Hp + py) * a.Wp + px) * 16u);
    }
    const __amdgpu_buffer_rsrc_t w1 = make_rsrc(a.wpk1, a.wpk_bytes);
    const __amdgpu_buffer_rsrc_t w2 = make_rsrc(a.wpk2, a.wpk_bytes);
    const uint32_t wlane = (uint32_t)(half * 2 * 64 + lane) * 16u;
    // This lane's channels: oc(n) .. oc(n) + 3.
    auto oc = [&](int n) { return (half * 2 + n) * 16 + quarter * 4; };
    float b1[2][4], b2[2][4];
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            b1[n][v] = a.bias1[oc(n) + v];
            b2[n][v] = a.bias2[oc(n) + v];
        }
#pragma unroll
    for (int j = 0; j < kIter; ++j) xt[min(tid + j * 64 * L::NW, kUnits - 1)] = q[j];
    __syncthreads();

    {
        uint32_t base[L::P1];
#pragma unroll
        for (int p = 0; p < L::P1; ++p) {
            const int hp = min((group + PG * p) * 16 + (lane & 15), L::HPX - 1);
            const int hy = hp / L::HW;
            base[p] = (uint32_t)(quarter * L::IPX + hy * L::IW + hp - hy * L::HW) * 16u;
        }
        f32x4 sum[L::P1][2];
        gemm64<L::P1, L::IPX, L::IW>(lds, base, w1, wlane, sum);
        // t, zero outside the image (conv2's padding).
#pragma unroll
        for (int p = 0; p < L::P1; ++p) {
            const int hp = (group + PG * p) * 16 + (lane & 15);
            const int hy = min(hp, L::HPX - 1) / L::HW;
            const int iy = oy0 - 1 + hy;
            const int ix = ox0 - 1 + hp - hy * L::HW;
            const bool inside = iy >= 0 && iy < a.H && ix >= 0 && ix < a.W;
            if (hp >= L::HPX) continue;
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                float f[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) f[v] = activate(sum[p][n][v] + b1[n][v], a.act1, a.slope);
                const Half4 h = pack4(f);
                *reinterpret_cast<uint2*>(tt + ((oc(n) >> 3) * L::HPX + hp) * 16 + (quarter & 1) * 8) =
                    inside ? make_uint2(h.v[0], h.v[1]) : make_uint2(0u, 0u);
            }
        }
    }
    __syncthreads();

    uint32_t base[L::P2];
#pragma unroll
    for (int p = 0; p < L::P2; ++p)
        base[p] = (uint32_t)(quarter * L::HPX + (group + PG * p) * L::HW + (lane & 15)) * 16u;
    f32x4 sum[L::P2][2];
    gemm64<L::P2, L::HPX, L::HW>(tt, base, w2, wlane, sum);
    const uint16_t* res1 = a.res1 ? a.res1 + z * a.res1_ts : nullptr;
    const uint16_t* res2 = a.res2 ? a.res2 + z * a.res2_ts : nullptr;
    uint16_t* out = a.out + z * a.out_ts;
    uint16_t* out2 = a.out2 ? a.out2 + z * a.out2_ts : nullptr;
    const int x = ox0 + (lane & 15);
    const Place place{a.H, a.W, kPad};
#pragma unroll
    for (int p = 0; p < L::P2; ++p) {
        const int y = oy0 + group + PG * p;
        if (y >= a.H || x >= a.W) continue;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const int c = oc(n);
            float f[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) f[v] = activate(sum[p][n][v] + b2[n][v], a.act2, a.slope);
            if (res1 != nullptr) {
                const Half4 h = load4(res1, a.res1_layout, c, y, x, place);
#pragma unroll
                for (int v = 0; v < 4; ++v) f[v] = half_at(h, v) + f[v];
            }
            if (res2 != nullptr) {
                const Half4 h = load4(res2, a.res2_layout, a.res2_coff + c, y, x, place);
#pragma unroll
                for (int v = 0; v < 4; ++v) f[v] = half_at(h, v) + (float)round_f16(f[v]);
            }
            const Half4 h = pack4(f);
            store4(out, a.out_layout, c, y, x, place, h);
            if (out2 != nullptr) store4(out2, kLayoutCB8, c, y, x, place, h);
        }
    }
}

template <int TH, int PG>
hipError_t launch_pair_wide(WidePairArgs a, int images, hipStream_t stream) {
    using L = WidePair<TH, PG>;
    a.tiles_x = (a.W + kWideTW - 1) / kWideTW;
    a.tiles_image = (a.H + TH - 1) / TH * a.tiles_x;
    a.tiles = images * a.tiles_image;
    auto kernel = &conv_pair_wide_kernel<TH, PG>;
    const hipError_t attr = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), WidePair<TH, PG>::lds);
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((a.tiles + 7) / 8 * 8)), dim3(64 * L::NW), L::lds, stream, a);
    return hipGetLastError();
}

// One KS x KS conv of 8 * CB input channels (conv3x3_kernel's contract, and convk_kernel's) on a
// TH x 16 output tile: the tile's input (KS / 2 pixels more on each side, all channels: K runs
// over taps outside and channels inside) comes into LDS by DMA. NH * PG waves: each multiplies
// every PG-th row by N of the NH * N 16-channel blocks.
//
// 3x3 over 16 maps of 64x64: 320 -> 64 channels 80.5 -> 31.8 us (760 TFLOP/s), 196 -> 64
// 37.2 -> 19.1 us; 180x320 64 -> 432 130 -> 39.9 us. What bounds it: the weight fragments through
// the vector L1, 2 KB per wave and K-step for 4 or 8 products. The addresser is busy 88 % of the
// time at 320 -> 64 (4 products) and 73 % at 196 -> 64 (8), the matrix cores 35 and
// 41 %, the LDS 35 and 40 % (half of it bank conflicts).
struct WideConvArgs {
    const void* xin;
    const void* wpk;
    const float* bias;
    const uint16_t* res1;
    const uint16_t* res2;
    uint16_t* out;
    uint32_t xin_bytes, wpk_bytes;
    int act;
    float slope;
    int res1_layout, res2_layout, out_layout, res2_coff;
    int H, W, pad, Cout, NBT, tiles_x, tiles_image, tiles;  // pad: border of every CB8 tensor
    long xin_ts, res1_ts, res2_ts, out_ts;
};

template <int KS, int CB, int NH, int N, int TH, int PG>
struct WideConv {
    static constexpr int NW = NH * PG;
    static constexpr int IW = kWideTW + KS - 1, IPX = (TH + KS - 1) * IW;
    static constexpr int P = TH / PG;
    static constexpr int KB = KS * KS * CB, KSTEPS = (KB + 3) / 4;
    static constexpr int UNITS = (CB * IPX + 63) / 64 * 64;  // whole waves of DMA
    static constexpr size_t lds = (size_t)UNITS * 16;
    // LDS unit of K-block kb of the pixel whose tap (0, 0) is unit 0 (a padding K-block: the
    // last one's), and lane quarter q's at K-block 0.
    static constexpr int unit(int kb) {
        const int k = kb < KB ? kb : KB - 1;
        return k % CB * IPX + k / CB / KS * IW + k / CB % KS;
    }
    static constexpr int first(int q) { return CB >= 4 ? q * IPX : q % CB * IPX + q / CB; }
};

template <int KS, int CB, int NH, int N, int TH, int PG>
__global__ __launch_bounds__((64 * NH * PG)) void conv_wide_kernel(WideConvArgs a) {
    using L = WideConv<KS, CB, NH, N, TH, PG>;
    constexpr int P = L::P;
    constexpr int D = P == 4 ? 4 : P == 2 ? 6 : 8;  // K-steps of weights in flight
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = wave / NH;
    const int half = wave % NH;
    const int quarter = lane >> 4;
    const int Hp = a.H + 2 * a.pad, Wp = a.W + 2 * a.pad;

    const int per_xcd = (a.tiles + 7) / 8;
    const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tile >= a.tiles) return;  // whole workgroup, before any barrier
    const int z = tile / a.tiles_image;
    const int ti = tile - z * a.tiles_image;
    const int ty = ti / a.tiles_x;
    const int oy0 = ty * TH;
    const int ox0 = (ti - ty * a.tiles_x) * kWideTW;
    const int chunk = blockIdx.y;

    // Input unit u = (block, row, column) of the tile, from KS / 2 pixels up and left of it;
    // past the padded plane a clamped one, which only reaches outputs outside the image.
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(static_cast<const uint16_t*>(a.xin) + z * a.xin_ts, a.xin_bytes);
    for (int u0 = wave * 64; u0 < L::UNITS; u0 += 64 * L::NW) {
        const int u = min(u0 + lane, CB * L::IPX - 1);
        const int cb = u / L::IPX;
        const int r = u - cb * L::IPX;
        const int row = r / L::IW;
        const int py = min(oy0 + row + a.pad - KS / 2, Hp - 1);
        const int px = min(ox0 + r - row * L::IW + a.pad - KS / 2, Wp - 1);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)(lds + u0 * 16), 16,
                                                 (int)((uint32_t)((cb * Hp + py) * Wp + px) * 16u), 0, 0, 0);
    }
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(a.wpk, a.wpk_bytes);
    uint32_t wlane = (uint32_t)(((chunk * NH + half) * N) * 64 + lane) * 16u;
    auto oc = [&](int n) { return ((chunk * NH + half) * N + n) * 16 + quarter * 4; };
    h8 B[D][N];
    auto load_weights = [&](int s) {
        __asm__ volatile("" : "+v"(wlane));  // requested here and not earlier
#pragma unroll
        for (int n = 0; n < N; ++n)
            B[s % D][n] = __builtin_bit_cast(h8, load16(wr, wlane, (uint32_t)(s * a.NBT + n) * 1024u));
    };
    float bias[N][4];
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int v = 0; v < 4; ++v) bias[n][v] = a.bias[min(oc(n) + v, a.Cout - 1)];
    __builtin_amdgcn_s_waitcnt(0);  // this wave's copies (the compiler does not track them)
    __syncthreads();
#pragma unroll
    for (int s = 0; s < D - 1 && s < L::KSTEPS; ++s) load_weights(s);

    // Byte address of this lane's unit of each row at K-block quarter; later steps add the
    // same offset in every lane, except where a step's K-blocks cross a tap or a tap row.
    uint32_t base[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int q0 = CB >= 4 ? quarter * L::IPX : quarter % CB * L::IPX + quarter / CB;
        base[p] = (uint32_t)(q0 + (group + PG * p) * L::IW + (lane & 15)) * 16u;
    }
    h8 X[2][P];
    auto load_pixels = [&](int s) {
        const int kb = 4 * s;
        const uint32_t off = (uint32_t)L::unit(kb) * 16u;
        uint32_t more = 0;
#pragma unroll
        for (int q = 1; q < 4; ++q) {
            const int d = L::unit(kb + q) - L::unit(kb) - L::first(q);
            const int before = q == 1 ? 0 : L::unit(kb + q - 1) - L::unit(kb) - L::first(q - 1);
            if (d != before) more = quarter >= q ? (uint32_t)(d * 16) : more;
        }
#pragma unroll
        for (int p = 0; p < P; ++p) X[s & 1][p] = *reinterpret_cast<const h8*>(lds + (base[p] + off + more));
        if (kb + 4 > L::KB) {
            // Padding K-blocks multiply zero weights; zero pixels keep a non-finite input from
            // turning 0 * inf into NaN there.
            const h8 zero = __builtin_bit_cast(h8, u32x4{0u, 0u, 0u, 0u});
#pragma unroll
            for (int p = 0; p < P; ++p) X[s & 1][p] = kb + quarter < L::KB ? X[s & 1][p] : zero;
        }
    };
    f32x4 acc[P][N], sum[P][N];
    load_pixels(0);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        constexpr int K = L::KSTEPS;
        const int s0 = r * K / 8, s1 = (r + 1) * K / 8;
#pragma unroll
        for (int s = s0; s < s1; ++s) {
            if (s + D - 1 < K) load_weights(s + D - 1);
            if (s + 1 < K) load_pixels(s + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int p = 0; p < P; ++p)
#pragma unroll
                for (int n = 0; n < N; ++n)
                    acc[p][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(B[s % D][n], X[s & 1][p],
                                                                       s == s0 ? f32x4{} : acc[p][n], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int n = 0; n < N; ++n) {
                if (r == 0)
                    sum[p][n] = acc[p][n];
                else
#pragma unroll
                    for (int v = 0; v < 4; ++v) sum[p][n][v] = sum[p][n][v] + acc[p][n][v];
                __asm__ volatile("" : "+v"(sum[p][n]));
            }
    }

    const uint16_t* res1 = a.res1 ? a.res1 + z * a.res1_ts : nullptr;
    const uint16_t* res2 = a.res2 ? a.res2 + z * a.res2_ts : nullptr;
    uint16_t* out = a.out + z * a.out_ts;
    const int x = ox0 + (lane & 15);
    const Place place{a.H, a.W, a.pad};
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int y = oy0 + group + PG * p;
        if (y >= a.H || x >= a.W) continue;
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const int c = oc(n);
            if (c >= a.Cout) continue;
            const int live = min(4, a.Cout - c);
            float f[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) f[v] = activate(sum[p][n][v] + bias[n][v], a.act, a.slope);
            if (res1 != nullptr) {
                const Half4 h = load4(res1, a.res1_layout, c, y, x, place, live);
#pragma unroll
                for (int v = 0; v < 4; ++v) f[v] = half_at(h, v) + f[v];
            }
            if (res2 != nullptr) {
                const Half4 h = load4(res2, a.res2_layout, a.res2_coff + c, y, x, place, live);
#pragma unroll
                for (int v = 0; v < 4; ++v) f[v] = half_at(h, v) + (float)round_f16(f[v]);
            }
            store4(out, a.out_layout, c, y, x, place, pack4(f), live);
        }
    }
}

template <int KS, int CB, int NH, int N, int TH, int PG>
hipError_t launch_wide_as(WideConvArgs a, int images, int chunks, hipStream_t stream) {
    using L = WideConv<KS, CB, NH, N, TH, PG>;
    a.tiles_x = (a.W + kWideTW - 1) / kWideTW;
    a.tiles_image = (a.H + TH - 1) / TH * a.tiles_x;
    a.tiles = images * a.tiles_image;
    auto kernel = &conv_wide_kernel<KS, CB, NH, N, TH, PG>;
    const hipError_t attr = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), L::lds);
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((a.tiles + 7) / 8 * 8), (unsigned)chunks), dim3(64 * L::NW), L::lds, stream, a);
    return hipGetLastError();
}

}  // namespace

static long wide_tiles(int height, int width, int images, int th) {
    return (long)images * ((height + th - 1) / th) * ((width + kWideTW - 1) / kWideTW);
}

// The wide kernels read and write four channels of a CB8 unit at once: those tensors must be
// 8-byte aligned.
static bool ends_aligned(const ConvEnds& t) {
    const auto ok = [](const void* p, int layout) { return layout != kLayoutCB8 || (uintptr_t)p % 8 == 0; };
    return ok(t.res1, t.res1_layout) && ok(t.res2, t.res2_layout) && ok(t.out, t.out_layout) && ok(t.out2, kLayoutCB8);
}
static long tiles_2x8(int height, int width, int images) { return (long)images * ((height + 1) / 2) * ((width + 7) / 8); }

// Up to 256 tiles of 2 x 8 pixels the 16-pixel kernels of dcn_kernels_conv.hip run as one
// workgroup per CU and are faster (a pair at 64x64, 256 of them: 6.7 against 7.1 us; at
// 64x72, 288: 11.5 against 7.5).
bool conv_wide_chosen(int height, int width, int images, const ConvEnds& t) {
    return tiles_2x8(height, width, images) > 256 && ends_aligned(t);
}

// One conv over one image: both kernels' times by their workgroups, `flat` of 16 pixels and `wide` of
// 4 x 16, timed for 11 channel counts at 294 sizes. Up to 512 flat ones (two per CU) stay one round;
// the wide kernel beats that only with more than 64 channels to read, and one workgroup per CU
// itself (us flat / wide: 64x72 320 -> 64 10.1 / 9.9, 128 -> 64 7.4 / 6.1, 64 -> 64 4.6 / 5.0). Beyond,
// by the time of a workgroup of each: a map narrower than 4 to 8 columns leaves most of a
// 16-wide tile empty (1030x3 320 -> 64 7.1 / 15.0; 2600x4 64 -> 64 6.6 / 8.6; 1696x5 256 -> 64
// 12.1 / 12.6, 128 -> 64 10.6 / 8.2). Over several images: as the pair, whose workgroups it shares.
// The input comes by 16-byte LDS DMA and must be 16-byte aligned.
bool conv3x3_wide_chosen(const ConvGeometry& g, const void* x_cb8, int images, const ConvEnds& t) {
    const int cb = g.cb;
    const bool supported = (cb == 8 || cb == 16 || cb == 24 || cb == 25 || cb == 32 || cb == 40) && g.cout % 4 == 0;
    if (!supported || images < 1 || (uintptr_t)x_cb8 % 16 != 0 || !ends_aligned(t)) return false;
    if (images > 1) return tiles_2x8(g.h, g.w, images) * g.chunks > 256;
    const long flat = ((long)g.h * g.w + 15) / 16 * g.chunks, wide = wide_tiles(g.h, g.w, 1, 4) * g.chunks;
    if (flat <= 512) return flat > 256 && cb > 8 && wide <= 256;
    return wide * (cb == 8 ? 1.4 : cb <= 25 ? 1.0 : 1.8) <= (double)flat;
}

hipError_t launch_conv3x3_pair_wide(const ConvGeometry& g, const void* x_cb8, const void* wpk1, const float* bias1,
                                    int act1, const void* wpk2, const float* bias2, int act2, float slope,
                                    const uint16_t* res1, int res1_layout, const uint16_t* res2, int res2_layout,
                                    uint16_t* out, int out_layout, hipStream_t stream, int res2_coff,
                                    const ConvBatch& batch, uint16_t* out2_cb8) {
    WidePairArgs a{};
    a.xin = x_cb8;
    a.wpk1 = wpk1;
    a.wpk2 = wpk2;
    a.bias1 = bias1;
    a.bias2 = bias2;
    a.res1 = res1;
    a.res2 = res2;
    a.out = out;
    a.out2 = out2_cb8;
    a.act1 = act1;
    a.act2 = act2;
    a.slope = slope;
    a.res1_layout = res1_layout;
    a.res2_layout = res2_layout;
    a.out_layout = out_layout;
    a.res2_coff = res2_coff;
    a.xin_ts = batch.x;
    a.res1_ts = batch.res1;
    a.res2_ts = batch.res2;
    a.out_ts = batch.out;
    a.out2_ts = batch.out2;
    a.H = g.h;
    a.W = g.w;
    a.Hp = g.h + 2 * kPad;
    a.Wp = g.w + 2 * kPad;
    a.xin_bytes = (uint32_t)((size_t)g.cb * a.Hp * a.Wp * 16);
    a.wpk_bytes = (uint32_t)conv_packed_bytes(g);
    // The smallest tile whose workgroups fit the 256 CUs at once, else the largest: a round of
    // workgroups costs mostly its latency, and beyond one round the halo counts. Measured
    // us at TH 2 / 4 / 8 / 16: 90x91 (270 tiles of 2 rows, 138 of 4) 9.2 / 8.7 / 10.0 / 15.0,
    // 180x320 (240 of 16) 29.1 / 28.4 / 21.0 / 17.3.
    const auto fits = [&](int th) { return wide_tiles(g.h, g.w, batch.images, th) <= 256; };
    if (fits(2)) return launch_pair_wide<2, 2>(a, batch.images, stream);
    if (fits(4)) return launch_pair_wide<4, 4>(a, batch.images, stream);
    if (fits(8)) return launch_pair_wide<8, 4>(a, batch.images, stream);
    return launch_pair_wide<16, 4>(a, batch.images, stream);
}

namespace {

// Tiles of 4 rows, two or more workgroups per CU; of 8 rows (half the weight traffic per pixel)
// where there are more than 256 of those and the channels leave room for two in a CU's LDS.
// us at TH 4 / 8: 256x256 128 -> 64 15.7 / 13.7, 196 -> 64 21.3 / 19.1, 320 -> 64 31.8 / 33.2;
// 128x128 (128 tiles of 8 rows) 128 -> 64 6.3 / 8.8, 64 -> 432 14.8 / 17.3.
template <int CB>
hipError_t launch_wide_cb(const WideConvArgs& a, int images, int chunks, hipStream_t stream) {
    if constexpr (CB <= 25)
        if (wide_tiles(a.H, a.W, images, 8) > 256) return launch_wide_as<3, CB, 2, 2, 8, 2>(a, images, chunks, stream);
    return launch_wide_as<3, CB, 2, 2, 4, 2>(a, images, chunks, stream);
}

}  // namespace

hipError_t launch_conv3x3_wide(const ConvGeometry& g, const void* x_cb8, const void* wpk, const float* bias, int act,
                               float slope, const uint16_t* res1, int res1_layout, const uint16_t* res2,
                               int res2_layout, uint16_t* out, int out_layout, hipStream_t stream, int res2_coff,
                               const ConvBatch& batch) {
    WideConvArgs a{};
    a.xin = x_cb8;
    a.wpk = wpk;
    a.bias = bias;
    a.res1 = res1;
    a.res2 = res2;
    a.out = out;
    a.act = act;
    a.slope = slope;
    a.res1_layout = res1_layout;
    a.res2_layout = res2_layout;
    a.out_layout = out_layout;
    a.res2_coff = res2_coff;
    a.xin_ts = batch.x;
    a.res1_ts = batch.res1;
    a.res2_ts = batch.res2;
    a.out_ts = batch.out;
    a.H = g.h;
    a.W = g.w;
    a.pad = kPad;
    a.Cout = g.cout;
    a.NBT = g.nbt;
    a.xin_bytes = (uint32_t)((size_t)g.cb * (g.h + 2 * kPad) * (g.w + 2 * kPad) * 16);
    a.wpk_bytes = (uint32_t)conv_packed_bytes(g);
    switch (g.cb) {
        case 8: return launch_wide_cb<8>(a, batch.images, g.chunks, stream);
        case 16: return launch_wide_cb<16>(a, batch.images, g.chunks, stream);
        case 24: return launch_wide_cb<24>(a, batch.images, g.chunks, stream);
        case 25: return launch_wide_cb<25>(a, batch.images, g.chunks, stream);
        case 32: return launch_wide_cb<32>(a, batch.images, g.chunks, stream);
        case 40: return launch_wide_cb<40>(a, batch.images, g.chunks, stream);
    }
    return hipErrorInvalidValue;
}

namespace {

// The smallest tile whose workgroups fit the 256 CUs at once, else 16 rows, or 8 for the layers
// with little work per pixel. us per layer (8 -> 32 / 32 -> 64 / 64 -> 32 / 32 -> 16 / 16 -> 2) over 58
// images, 16x16 at 4 rows 4.8 / 9.7 / 9.9 / 5.3 / 4.6, at 8 rows 5.4 / 10.5 / 11.0 / 6.1 / 5.9; 32x32 at 8
// rows 6.4 / 19.1 / 18.5 / 8.7 / 6.0, at 16 rows (232 tiles) 7.5 / 15.3 / 16.7 / 9.7 / 7.9; 64x64 at 8 rows
// 15.8 / 62.1 / 60.9 / 22.0 / 12.1, at 16 rows 16.2 / 48.7 / 45.7 / 21.0 / 13.0 (980 TFLOP/s at 32 -> 64).
template <int CB, int NH, int N>
hipError_t launch_convk_as(const WideConvArgs& a, int images, hipStream_t stream) {
    const auto fits = [&](int th) { return wide_tiles(a.H, a.W, images, th) <= 256; };
    if (fits(4)) return launch_wide_as<7, CB, NH, N, 4, 2>(a, images, 1, stream);
    if (N == 1 || CB == 1 || fits(8)) return launch_wide_as<7, CB, NH, N, 8, 4>(a, images, 1, stream);
    return launch_wide_as<7, CB, NH, N, 16, 4>(a, images, 1, stream);
}

}  // namespace

// Above two 16-pixel workgroups of convk_kernel per CU, on maps at least a tile wide: SPyNet
// on one pair (512 of them at 64x64) 151.6 us with convk_kernel, 168.7 with this; on 4 pairs
// 212.7 against 188.4, on 29 744 against 333.
bool convk_wide_chosen(const ConvKGeometry& g, int batch, const uint16_t* out, int out_cb8) {
    const bool layer = (g.cb == 1 && g.nbt == 2) || (g.cb == 4 && g.nbt == 4) || (g.cb == 8 && g.nbt == 2) ||
                       (g.cb == 4 && g.nbt == 1) || (g.cb == 2 && g.nbt == 1);
    return g.ks == 7 && g.chunks == 1 && layer && g.w >= kWideTW && (long)batch * g.h * g.w > 512 * 16 &&
           (!out_cb8 || (g.cout % 4 == 0 && (uintptr_t)out % 8 == 0));
}

hipError_t launch_convk_wide(const ConvKGeometry& g, int batch, int pad, const void* x_cb8, const void* wpk,
                             const float* bias, int act, const uint16_t* base, uint16_t* out, int out_cb8,
                             hipStream_t stream) {
    WideConvArgs a{};
    const long padded = (long)(g.h + 2 * pad) * (g.w + 2 * pad) * 8, plane = (long)g.h * g.w;
    a.xin = x_cb8;
    a.wpk = wpk;
    a.bias = bias;
    a.res2 = base;
    a.out = out;
    a.act = act;
    a.res2_layout = kLayoutNCHW;
    a.out_layout = out_cb8 ? kLayoutCB8 : kLayoutNCHW;
    a.H = g.h;
    a.W = g.w;
    a.pad = pad;
    a.Cout = g.cout;
    a.NBT = g.nbt;
    a.xin_ts = g.cb * padded;
    a.res2_ts = g.cout * plane;
    a.out_ts = out_cb8 ? (g.cout + 7) / 8 * padded : g.cout * plane;
    a.xin_bytes = (uint32_t)(a.xin_ts * 2);
    a.wpk_bytes = (uint32_t)convk_packed_bytes(g);
    if (g.cb == 1 && g.nbt == 2) return launch_convk_as<1, 1, 2>(a, batch, stream);
    if (g.cb == 4 && g.nbt == 4) return launch_convk_as<4, 2, 2>(a, batch, stream);
    if (g.cb == 8 && g.nbt == 2) return launch_convk_as<8, 1, 2>(a, batch, stream);
    if (g.cb == 4 && g.nbt == 1) return launch_convk_as<4, 1, 1>(a, batch, stream);
    if (g.cb == 2 && g.nbt == 1) return launch_convk_as<2, 1, 1>(a, batch, stream);
    return hipErrorInvalidValue;
}

}  // namespace dcn
