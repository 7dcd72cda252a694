// The fp32 backward's GEMM kernels.
//
// Column gradient (dcn2_colgrad_f32_kernel), with its consumers: for a tile of
// output pixels and CT channels of one tap and group
//     cg[c][n] = sum_m W[m][c, tap] gO[m][n]                (com.cu:789-793)
// on 32x32x2 fp32 MFMAs, kept on chip; then per pixel the corner sums
// S_q = sum_c cg_c x_c(corner q), from which grad_offset / grad_mask follow
// (com.cu:388-501), and the masked row for grad_input (com.cu:526-609).
//
// Bound: the fp32 matrix rate for wide layers, the hand-off rows and grad_output
// for narrow ones.  What cost the time before (one 8-wave workgroup per 128
// pixels of an image that walked every chunk of K, one to a CU) was idle CUs: 64
// workgroups at 32 x 14 x 14, 32 at 32 x 7 x 7, each reloading all of grad_output
// per chunk there.  Here every (pixel tile, channel tile) is its own 4-wave
// workgroup, several to a CU, and pixels are numbered through the batch.  Measured
// (us, old -> new; 3.3-3.7 GFLOP each, 21-24 us at the 154 TFLOP/s of a large
// product): 203 -> 62 at Cout 256, K 64, 32 x 56 x 56; 392 -> 60 at 256, 1024, 32 x
// 14 x 14; 1558 -> 62 at 2048, 512, 32 x 7 x 7; 142 -> 62 at 128, 1152, 4 x 56 x 56.
#include <algorithm>
#include <cstddef>

#include "dcn2_backward.h"
#include "../../include/dcnv2_amd.h"

namespace dcn2 {

// Value of lane i ^ 1, i ^ 2, and of the mirrored lane of 8 / 16 (DPP); summing
// with each in turn sums groups of 2, 4, 8, 16 lanes.
template <int CTRL> __device__ __forceinline__ float dpp_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int LANES> __device__ __forceinline__ float lane_sum(float v) {
    v = dpp_add<0xB1>(v);   // quad_perm 1,0,3,2
    v = dpp_add<0x4E>(v);   // quad_perm 2,3,0,1
    if constexpr (LANES >= 8) v = dpp_add<0x141>(v);   // row_half_mirror
    if constexpr (LANES >= 16) v = dpp_add<0x140>(v);  // row_mirror
    return v;
}

struct CgF32Params {
    BwdParams p;
    int b0, total;      // first image and pixels (images * N) of this launch
    uint32_t x_bytes;   // bytes of its images of xt
    int ptiles, ctiles; // pixel tiles, channel tiles (taps * groups * Cgp / CT)
    int cpg, cpw, cog;  // channel tiles per group; per weight group, and its rows (0: no split)
};

constexpr int kCgM = 32;  // rows of grad_output per step

// JB x (CB == 2 ? 2 : 4) blocks of 32 pixels, CB blocks of 32 channels.  GN:
// grad_output is channels-last.
template <int JB, int CB, bool GN>
__global__ __launch_bounds__(256) void dcn2_colgrad_f32_kernel(const CgF32Params c) {
    constexpr int NW = 4 / CB, NT = 32 * JB * NW, CT = 32 * CB;
    constexpr int LDG = NT + 8;  // floats per staged row: the two lane halves read rows 4 apart, on other banks
    constexpr int LDC = CT + 4;
    constexpr int NG = NT * kCgM / 256;
    struct Px {
        uint32_t off[4];
        float m, ly, lx;
        int valid, row, cs, pad0, pad1;
    };
    constexpr size_t kG = sizeof(float) * 2 * kCgM * LDG, kC = sizeof(float) * NT * LDC;
    __shared__ __attribute__((aligned(16))) char smem[kG > kC ? kG : kC];
    __shared__ __attribute__((aligned(16))) Px sP[NT];
    __shared__ f32x4 sS[NT];
    float(*const sG)[kCgM][LDG] = reinterpret_cast<float(*)[kCgM][LDG]>(smem);
    float(*const sC)[LDC] = reinterpret_cast<float(*)[LDC]>(smem);

    const BwdParams &p = c.p;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cb = wave % CB, nb = wave / CB * JB;
    // the channel tiles of one pixel tile are neighbours, on one XCD: they read the same grad_output
    const int t = xcd_remap(blockIdx.x, c.ptiles * c.ctiles);
    const int ct = t % c.ctiles, n0 = t / c.ctiles * NT;
    const int live_px = min(NT, c.total - n0);
    const int N = p.Ho * p.Wo, KK = p.kh * p.kw;
    const int cc = ct % c.cpg, tg = ct / c.cpg, tap = tg / p.G, g = tg - tap * p.G;
    const int plane = g * KK + tap;
    // rows of grad_output this tile depends on: all, or its weight group's
    int mbeg = 0, mend = p.Cout;
    if (c.cog) {
        const int wg = (g * c.cpg + cc) / c.cpw;
        mbeg = wg * c.cog;
        mend = mbeg + c.cog;
    }

    // grad_output, kCgM rows x NT pixels per step: thread's pixel and first row
    // (channels-last: row and first pixel)
    const int gcol = GN ? tid / kCgM : tid % NT, grow = GN ? tid % kCgM : tid / NT;
    const float *gsrc;
    if constexpr (GN) {
        gsrc = (const float *)p.gout + ((size_t)c.b0 * N + n0) * p.Cout;
    } else {
        const unsigned n = n0 + min(gcol, live_px - 1), b = n / (unsigned)N;
        gsrc = (const float *)p.gout + (size_t)(c.b0 + b) * p.Cout * N + (n - b * (unsigned)N);
    }
    float gr[NG];
    auto load_g = [&](int m0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            if constexpr (GN) {
                const int px = min(gcol + i * (256 / kCgM), live_px - 1), m = m0 + grow;
                gr[i] = m < mend ? gsrc[(size_t)px * p.Cout + m] : 0.0f;
            } else {
                const int m = m0 + grow + i * (256 / NT);
                gr[i] = m < mend ? gsrc[(size_t)m * N] : 0.0f;
            }
        }
    };
    auto store_g = [&](int st) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            if constexpr (GN) sG[st][grow][gcol + i * (256 / kCgM)] = gr[i];
            else sG[st][grow + i * (256 / NT)][gcol] = gr[i];
        }
    };
    // W'^T fragments: channel block, 8-row group -> 64 lanes x 4 rows
    const float *wsrc = (const float *)p.wt + (size_t)(ct * CB + cb) * (p.Mp / 8) * 256 + lane * 4;
    f32x4 a[2][kCgM / 8];
    auto load_a = [&](int set, int m0) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kCgM / 8; ++k)
            a[set][k] = *reinterpret_cast<const f32x4 *>(wsrc + (size_t)(m0 / 8 + k) * 256);
    };
    load_a(0, mbeg);
    load_g(mbeg);

    // thread's pixel of the consumers' descriptors
    float f_m = 0.0f, f_ly = 0.0f, f_lx = 0.0f;
    int f_b = 0, f_nn = 0;
    if (tid < NT) {
        const bool live = tid < live_px;
        const unsigned n = n0 + (live ? tid : 0), b = n / (unsigned)N;
        f_b = c.b0 + b;
        f_nn = n - b * (unsigned)N;
        const int oy = f_nn / p.Wo, ox = f_nn - oy * p.Wo;
        const float *off = (const float *)p.offset + f_b * p.off_bs + (size_t)plane * 2 * N + f_nn;
        const float y = (float)(oy * p.sh - p.ph + tap / p.kw * p.dh) + off[0];
        const float x = (float)(ox * p.sw - p.pw + tap % p.kw * p.dw) + off[N];
        f_m = p.mask ? mask_value(((const float *)p.mask)[f_b * p.msk_bs + (size_t)plane * N + f_nn], p.msk_logit)
                     : 1.0f;
        const int smp = (f_b * p.G * KK + plane) * N + f_nn;
        const SamplePos sp = sample_pos(y, x, p.H, p.W);
        f_ly = sp.ly;
        f_lx = sp.lx;
        const uint32_t cs = p.G * p.Cgp * 4u, row = cs * (uint32_t)p.W;
        const uint32_t base = (b * (uint32_t)(p.H * p.W) + (uint32_t)(sp.y0 * p.W + sp.x0)) * cs;
        Px d;
        d.off[0] = sp.vy0 && sp.vx0 ? base : c.x_bytes;
        d.off[1] = sp.vy0 && sp.vx1 ? base + cs : c.x_bytes;
        d.off[2] = sp.vy1 && sp.vx0 ? base + row : c.x_bytes;
        d.off[3] = sp.vy1 && sp.vx1 ? base + row + cs : c.x_bytes;
        d.m = f_m;
        d.row = live ? p.sidx[smp] : -1;
        d.cs = live ? smp : -1;
        d.ly = d.lx = 0.0f;
        d.valid = d.pad0 = d.pad1 = 0;
        sP[tid] = d;
    }

    // Even and odd steps sum apart: half as long a chain of fp32 additions (the
    // error of a 2048-row sum against 64 bits: 8.2e-7 in one chain, 5.8e-7 in two).
    f32x16 acc[2][JB];
#pragma unroll
    for (int j = 0; j < JB; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][j][r] = acc[1][j][r] = 0.0f;
    store_g(0);
    __syncthreads();
    auto step = [&](auto set_c, int m0) __attribute__((always_inline)) {
        constexpr int S = decltype(set_c)::value;
        const bool more = m0 + kCgM < mend;  // (uniform)
        if (more) {
            load_a(S ^ 1, m0 + kCgM);
            load_g(m0 + kCgM);
        }
#pragma unroll
        for (int k = 0; k < kCgM / 8; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < JB; ++j)
                    acc[S][j] = Mma<float>::mma(
                        a[S][k][e], sG[S][8 * k + 4 * (lane >> 5) + e][(nb + j) * 32 + (lane & 31)], acc[S][j]);
        if (more) store_g(S ^ 1);
        __syncthreads();
    };
    int m0 = mbeg;
    for (; m0 + kCgM < mend; m0 += 2 * kCgM) {
        step(std::integral_constant<int, 0>{}, m0);
        step(std::integral_constant<int, 1>{}, m0 + kCgM);
    }
    if (m0 < mend) step(std::integral_constant<int, 0>{}, m0);

    // acc[4*rq + e] of lane l: channel 8*rq + 4*(l/32) + e of pixel l%32
#pragma unroll
    for (int j = 0; j < JB; ++j) {
        const f32x16 v = acc[0][j] + acc[1][j];
#pragma unroll
        for (int rq = 0; rq < 4; ++rq)
            *reinterpret_cast<f32x4 *>(&sC[(nb + j) * 32 + (lane & 31)][cb * 32 + 8 * rq + 4 * (lane >> 5)]) =
                f32x4{v[4 * rq], v[4 * rq + 1], v[4 * rq + 2], v[4 * rq + 3]};
    }
    __syncthreads();

    // Consumers: LP lanes x 4 channels per pixel.
    constexpr int LP = CT / 4, PPP = 256 / LP;
    const int l4 = tid % LP * 4;
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>((const float *)p.xt + (size_t)c.b0 * p.H * p.W * p.G * p.Cgp), (short)0,
        (int)c.x_bytes, 0x00020000);
    const int soff = (g * p.Cgp + cc * CT) * 4;
    float *const rows = (float *)p.cgm + cc * CT + l4;
#pragma unroll 2
    for (int px = tid / LP; px < NT; px += PPP) {
        const Px d = sP[px];
        f32x4 x[4];
        // (a corner outside the image has an offset past the buffer and reads 0)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            x[q] = __builtin_bit_cast(
                f32x4, __builtin_amdgcn_raw_buffer_load_b128(xrs, (int)(d.off[q] + l4 * 4u), soff, 0));
        const f32x4 v = *reinterpret_cast<const f32x4 *>(&sC[px][l4]);
        if (d.row >= 0) *reinterpret_cast<f32x4 *>(rows + (size_t)d.row * p.Cgp) = v * d.m;
        f32x4 S;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            S[q] = lane_sum<LP>(fmaf(v[0], x[q][0], fmaf(v[1], x[q][1], fmaf(v[2], x[q][2], v[3] * x[q][3]))));
        if (l4 == 0) sS[px] = S;
    }
    __syncthreads();
    if (c.cpg > 1) {
        // the group's channel tiles add their corner sums up
        for (int i = tid; i < NT * 4; i += 256)
            if (const int smp = sP[i >> 2].cs; smp >= 0)
                unsafeAtomicAdd(p.csum + (size_t)smp * 4 + (i & 3), sS[i >> 2][i & 3]);
        return;
    }
    if (tid < live_px) {
        const f32x4 S = sS[tid];
        const float hy = 1.0f - f_ly, hx = 1.0f - f_lx;
        const float gm = hy * hx * S[0] + hy * f_lx * S[1] + f_ly * hx * S[2] + f_ly * f_lx * S[3];
        float *goff = (float *)p.goff + f_b * p.off_bs + (size_t)plane * 2 * N + f_nn;
        goff[0] = f_m * (hx * (S[2] - S[0]) + f_lx * (S[3] - S[1]));
        goff[N] = f_m * (hy * (S[1] - S[0]) + f_ly * (S[3] - S[2]));
        // d/d(logit) of sigmoid = s (1 - s), s = the mask value used
        if (p.gmask)
            ((float *)p.gmask)[f_b * p.msk_bs + (size_t)plane * N + f_nn] =
                p.msk_logit ? gm * f_m * (1.0f - f_m) : gm;
    }
}

// Images of one launch over g's images (g.B of them): the bytes of their xt and
// their pixels stay in 32 bits (one image always fits, see make_geo).
static int f32_images(const Geo &g) {
    const long long img = std::max((long long)g.H * g.W * g.cs * 4, 2LL * g.N);
    return (int)std::max(1LL, std::min((long long)g.B, 0xffff0000LL / img));
}

template <int JB, int CB>
static void colgrad_f32_launch(CgF32Params &c, hipStream_t s) {
    c.ptiles = ceil_div(c.total, 32 * JB * (4 / CB));
    if (c.p.go_nhwc) dcn2_colgrad_f32_kernel<JB, CB, true><<<c.ptiles * c.ctiles, 256, 0, s>>>(c);
    else dcn2_colgrad_f32_kernel<JB, CB, false><<<c.ptiles * c.ctiles, 256, 0, s>>>(c);
}

hipError_t launch_colgrad_f32(const Geo &g, const BwdParams &p, hipStream_t s) {
    CgF32Params c;
    c.p = p;
    const int CT = f32_chan_tile(g), nimg = f32_images(g);
    c.ctiles = g.Kp / CT;
    c.cpg = g.Cgp / CT;
    c.cpw = g.cpw * 32 / CT;
    c.cog = g.gsplit ? g.Cout / g.WG : 0;
    for (int b = 0; b < g.B; b += nimg) {
        const int nb = std::min(nimg, g.B - b);
        c.b0 = b;
        c.total = nb * g.N;
        c.x_bytes = (uint32_t)((long long)nb * g.H * g.W * g.cs * 4);
        // 128-pixel tiles (the weight read once for twice the pixels) where three
        // to a CU remain, else 64: at 2048, 512, 32 x 7 x 7 the 128-pixel tiles
        // would be 104 workgroups, the 64-pixel ones are 200.
        if (CT == 32) colgrad_f32_launch<1, 1>(c, s);
        else if ((long long)ceil_div(c.total, 128) * c.ctiles >= 768) colgrad_f32_launch<2, 2>(c, s);
        else colgrad_f32_launch<1, 2>(c, s);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace dcn2
