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
// product): 203 -> 53 at Cout 256, K 64, 32 x 56 x 56; 392 -> 52 at 256, 1024, 32 x
// 14 x 14; 1558 -> 60 at 2048, 512, 32 x 7 x 7; 142 -> 57 at 128, 1152, 4 x 56 x 56.
#include <algorithm>
#include <cstddef>
#include <type_traits>

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
    if constexpr (LANES >= 32) v += __shfl_xor(v, 16, 64);
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

// 4 / CB blocks of 32 pixels x CB blocks of 32 channels, one per wave.  GN:
// grad_output is channels-last.
template <int CB, bool GN>
__global__ __launch_bounds__(256) void dcn2_colgrad_f32_kernel(const CgF32Params c) {
    constexpr int NT = 32 * (4 / CB), CT = 32 * CB;
    constexpr int LDG = NT + 8;  // floats per staged row: the two lane halves read rows 4 apart, on other banks
    constexpr int LDC = CT + 4;
    constexpr int NG = NT * kCgM / 256;
    struct Px {
        uint32_t off[4];
        float m;
        int row, pad[2];
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
    const int cb = wave % CB, nb = wave / CB;
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
    int f_b = 0, f_nn = 0, f_smp = 0;
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
        f_smp = (f_b * p.G * KK + plane) * N + f_nn;
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
        d.row = live ? p.sidx[f_smp] : -1;
        d.pad[0] = d.pad[1] = 0;
        sP[tid] = d;
    }

    // Even and odd steps sum apart: half as long a chain of fp32 additions (the
    // error of a 2048-row sum against 64 bits: 8.2e-7 in one chain, 5.8e-7 in two).
    f32x16 acc[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.0f;
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
                acc[S] = Mma<float>::mma(a[S][k][e], sG[S][8 * k + 4 * (lane >> 5) + e][nb * 32 + (lane & 31)],
                                         acc[S]);
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
    const f32x16 cg = acc[0] + acc[1];
#pragma unroll
    for (int rq = 0; rq < 4; ++rq)
        *reinterpret_cast<f32x4 *>(&sC[nb * 32 + (lane & 31)][cb * 32 + 8 * rq + 4 * (lane >> 5)]) =
            f32x4{cg[4 * rq], cg[4 * rq + 1], cg[4 * rq + 2], cg[4 * rq + 3]};
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
        // (nothing from a corner outside, also where the column gradient is not finite)
#pragma unroll
        for (int q = 0; q < 4; ++q) S[q] = d.off[q] != c.x_bytes ? S[q] : 0.0f;
        if (l4 == 0) sS[px] = S;
    }
    __syncthreads();
    if (c.cpg > 1) {
        // each of the group's channel tiles stores its part in a plane of its own:
        // added up with atomics, whose order varies, grad_offset and grad_mask of
        // fp32 would differ in their last bits from run to run
        if (tid < live_px)
            *reinterpret_cast<f32x4 *>(p.csum + cc * p.csum_ps + (size_t)f_smp * 4) = sS[tid];
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

// ---------------------------------------------------------------------------
// grad_weight / grad_bias (com.cu:637-706, 829-835):
//     gW[m][c, tap] += sum_n gO[m][n] col[c, tap][n]
// over a range of the batch's pixels, for BM rows and CT channels of one tap and
// group.  Steps of PS pixels: grad_output rows and resampled columns of step t+1
// are loaded while step t is multiplied, both through LDS (two stages).  A lane
// of an MFMA covers pixels {e, e + 4} of a group of 8 (e = 0..3): the row operand
// is one 16-byte LDS read per four MFMAs, the column operand four 4-byte reads.
//
// Bound: the fp32 matrix rate; then the fp32 atomics that add the ranges' partial
// blocks (one set per workgroup).  128 x 64 blocks on 4 waves: 256 x 64 on 8 waves
// measured the same at 256 rows and more (57.6-61.8 us) and 85-97 against 58 at 128.
// Against the 8-wave kernel this replaces, whose rows came by one 4-byte load per
// MFMA in the MFMA loop (us): 125 -> 62, 122 -> 56, 195 -> 56, 170 -> 57 at the
// column gradient's four shapes.
// n / d for n < 2^31 as (umulhi(n, mul) + n) >> shift: division by an invariant
// integer after Granlund and Montgomery ("Division by Invariant Integers using
// Multiplication", PLDI 1994), whose 33-bit multiplier 2^32 + mul is applied in two parts.
struct FastDiv {
    uint32_t mul, d;
    int shift;
};
static FastDiv fast_div(uint32_t d) {
    FastDiv f;
    f.d = d;
    f.shift = 0;
    while ((1ull << f.shift) < d) ++f.shift;
    f.mul = (uint32_t)(((1ull << 32) * ((1ull << f.shift) - d)) / d + 1);
    return f;
}
__device__ __forceinline__ uint32_t operator/(uint32_t n, const FastDiv &f) {
    return (__umulhi(n, f.mul) + n) >> f.shift;
}

struct GwF32Params {
    BwdParams p;
    int b0, total;     // first image and pixels (images * N) of this launch
    uint32_t x_bytes;  // bytes of its images of xt
    FastDiv dN, dWo;
    int mtiles, ktiles, splits;  // M tiles, channel tiles walked per M tile, pixel ranges
    int cpg;                     // channel tiles per group
    int cpt, cpw, cog;  // channel tiles per tap; per weight group, and its rows (0: no split)
};

// GM: grad_output by 0 16-byte loads of 4 pixels (NCHW, N % 4 == 0, aligned),
// 1 4-byte loads (NCHW), 2 4-byte loads along channels (channels-last).
template <int IB, int WM, int CB, int GM, bool MASK>
__global__ __launch_bounds__(64 * WM * CB) void dcn2_gradw_f32_kernel(const GwF32Params c) {
    constexpr int NT = 64 * WM * CB, BM = 32 * IB * WM, CT = 32 * CB, LP = CT / 4;
    constexpr int PS = NT / LP;  // pixels per step: one sampling slot per thread
    constexpr int LDG = PS + 4, LDC = CT == 64 ? 72 : 40;
    constexpr int GE = GM == 0 ? 4 : 1;            // pixels per grad_output load
    constexpr int NG = BM * PS / GE / NT;          // its loads per thread and step
    static_assert(NT * NG * GE == BM * PS && (GM != 2 || NT % BM == 0), "thread maps");
    __shared__ __attribute__((aligned(16))) float sG[2][BM][LDG];
    __shared__ __attribute__((aligned(16))) float sC[2][PS][LDC];

    const BwdParams &p = c.p;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cb = wave % CB, wm = wave / CB;
    // ranges slowest: an XCD works on neighbouring pixels for all rows and channels
    const int wi = xcd_remap(blockIdx.x, c.splits * c.ktiles * c.mtiles);
    const int mt = wi % c.mtiles, j = wi / c.mtiles % c.ktiles, sp = wi / (c.mtiles * c.ktiles);
    const int m0 = mt * BM;
    int ct = j;  // channel tile (tap, group, channels)
    if (c.cog) ct = j / c.cpw * c.cpt + m0 / c.cog * c.cpw + j % c.cpw;
    const int N = p.Ho * p.Wo, KK = p.kh * p.kw;
    const int cc = ct % c.cpg, tg = ct / c.cpg, tap = tg / p.G, g = tg - tap * p.G;
    const int plane = g * KK + tap, ty = tap / p.kw * p.dh - p.ph, tx = tap % p.kw * p.dw - p.pw;
    const int nt = ceil_div(c.total, PS);
    const int t0 = (int)((long long)nt * sp / c.splits), t1 = (int)((long long)nt * (sp + 1) / c.splits);
    if (t0 >= t1) return;

    // grad_output
    const int grow = GM == 2 ? tid % BM : tid / (PS / GE), gpx = GM == 2 ? tid / BM : tid % (PS / GE) * GE;
    constexpr int GRS = GM == 2 ? 0 : NT * GE / PS, GPS = GM == 2 ? NT / BM : 0;  // row / pixel step of a load
    const float *const go = (const float *)p.gout + (size_t)c.b0 * p.Cout * N;
    f32x4 gr[NG];  // (only [0] used by 4-byte loads)
    auto load_g = [&](int t) __attribute__((always_inline)) {
        if constexpr (GM == 2) {
#pragma unroll
            for (int i = 0; i < NG; ++i) {
                const int n = t * PS + gpx + i * GPS, m = m0 + grow;
                gr[i][0] = m < p.Cout && n < c.total ? go[(size_t)n * p.Cout + m] : 0.0f;
            }
        } else {
            const uint32_t n = t * PS + gpx, b = n / c.dN, nn = n - b * (uint32_t)N;
            const float *src = go + (size_t)b * ((size_t)p.Cout * N) + nn;
            const bool in = (int)n < c.total;  // (GE pixels together: the total is a multiple of 4 there)
#pragma unroll
            for (int i = 0; i < NG; ++i) {
                const int m = m0 + grow + i * GRS;
                gr[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                if (in && m < p.Cout) {
                    if constexpr (GM == 0) gr[i] = *reinterpret_cast<const f32x4 *>(src + (size_t)m * N);
                    else gr[i][0] = src[(size_t)m * N];
                }
            }
        }
    };
    const bool do_bias = p.gb_acc != nullptr && j == 0;
    float bsum[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) bsum[i] = 0.0f;
    auto store_g = [&](int st) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            float *dst = &sG[st][grow + i * GRS][gpx + i * GPS];
            if constexpr (GM == 0) *reinterpret_cast<f32x4 *>(dst) = gr[i];
            else *dst = gr[i][0];
            bsum[i] += GM == 0 ? (gr[i][0] + gr[i][1]) + (gr[i][2] + gr[i][3]) : gr[i][0];
        }
    };

    // columns: LP lanes x 4 channels per pixel
    const int spx = tid / LP, l4 = tid % LP * 4;
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>((const float *)p.xt + (size_t)c.b0 * p.H * p.W * p.G * p.Cgp), (short)0,
        (int)c.x_bytes, 0x00020000);
    const int soff = (g * p.Cgp + cc * CT) * 4;
    const float *const offp = (const float *)p.offset + c.b0 * p.off_bs + (size_t)plane * 2 * N;
    const float *const mskp = MASK ? (const float *)p.mask + c.b0 * p.msk_bs + (size_t)plane * N : nullptr;
    float dy, dx, mv = 1.0f;
    auto load_om = [&](int t) __attribute__((always_inline)) {
        const uint32_t n = min(t * PS + spx, c.total - 1), b = n / c.dN, nn = n - b * (uint32_t)N;
        const float *o = offp + b * p.off_bs + nn;
        dy = o[0];
        dx = o[N];
        if (MASK) mv = mskp[b * p.msk_bs + nn];
    };
    f32x4 x[4];
    float w[4];
    auto gather = [&](int t) __attribute__((always_inline)) {
        const uint32_t n0 = t * PS + spx, n = min(n0, (uint32_t)c.total - 1), b = n / c.dN, nn = n - b * (uint32_t)N;
        const bool live = n0 < (uint32_t)c.total;
        const int oy = nn / c.dWo, ox = nn - oy * p.Wo;
        const SamplePos s = sample_pos((float)(oy * p.sh + ty) + dy, (float)(ox * p.sw + tx) + dx, p.H, p.W);
        const float m = MASK ? mask_value(mv, p.msk_logit) : 1.0f;
        const float hy = (1.0f - s.ly) * m, ly = s.ly * m, hx = 1.0f - s.lx, lx = s.lx;
        const uint32_t cs = p.G * p.Cgp * 4u, row = cs * (uint32_t)p.W;
        const uint32_t base = (b * (uint32_t)(p.H * p.W) + (uint32_t)(s.y0 * p.W + s.x0)) * cs + l4 * 4u;
        // A corner outside the image, or of a pixel past the end, reads 0 and has
        // weight 0 (0 times a mask that is not finite is not 0).
        const bool v[4] = {live && s.vy0 && s.vx0, live && s.vy0 && s.vx1, live && s.vy1 && s.vx0,
                           live && s.vy1 && s.vx1};
        const uint32_t o[4] = {base, base + cs, base + row, base + row + cs};
        const float wq[4] = {hy * hx, hy * lx, ly * hx, ly * lx};
        uint32_t off[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            off[q] = v[q] ? o[q] : c.x_bytes;
            w[q] = v[q] ? wq[q] : 0.0f;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            x[q] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xrs, (int)off[q], soff, 0));
    };
    auto blend = [&](int st) __attribute__((always_inline)) {
        f32x4 v = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = fmaf(w[q], x[q][e], v[e]);
        *reinterpret_cast<f32x4 *>(&sC[st][spx][l4]) = v;
    };

    f32x16 acc[IB];
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
    auto mma = [&](int st) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < PS / 8; ++k) {
            f32x4 af[IB];
#pragma unroll
            for (int i = 0; i < IB; ++i)
                af[i] = *reinterpret_cast<const f32x4 *>(
                    &sG[st][(wm * IB + i) * 32 + (lane & 31)][8 * k + 4 * (lane >> 5)]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float bf = sC[st][8 * k + 4 * (lane >> 5) + e][cb * 32 + (lane & 31)];
#pragma unroll
                for (int i = 0; i < IB; ++i) acc[i] = Mma<float>::mma(af[i][e], bf, acc[i]);
            }
        }
    };

    load_g(t0);
    load_om(t0);
    gather(t0);
    load_om(t0 + 1);
    blend(0);
    store_g(0);
    __syncthreads();
    auto step = [&](auto set_c, int t) __attribute__((always_inline)) {
        constexpr int S = decltype(set_c)::value;
        const bool more = t + 1 < t1;  // (uniform)
        if (more) {
            load_g(t + 1);
            gather(t + 1);
            load_om(t + 2);
        }
        mma(S);
        if (more) {
            store_g(S ^ 1);
            blend(S ^ 1);
        }
        __syncthreads();
    };
    int t = t0;
    for (; t + 1 < t1; t += 2) {
        step(std::integral_constant<int, 0>{}, t);
        step(std::integral_constant<int, 1>{}, t + 1);
    }
    if (t < t1) step(std::integral_constant<int, 0>{}, t);

    const int k = ct * CT + cb * 32 + (lane & 31);
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = m0 + (wm * IB + i) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            if (m < p.Cout) unsafeAtomicAdd(p.gw_acc + (size_t)m * p.Kp + k, acc[i][r]);
        }
    if (do_bias) {
        // One atomic per row and workgroup, 64 rows to an instruction: the atomics of all
        // workgroups meet on a few cache lines.  From the threads that hold the sums (two
        // rows to an instruction, or one per load where a thread's loads are of one row)
        // they took longer than the rest: grad_weight 34 against 15 us at 1x1, C 11 -> 20, 2
        // x 151 x 105, and 118 against 13 at C 28 -> 91, 5 x 42 x 86, channels-last.
        float *const red = &sG[0][0][0];  // (the stages are free after the last barrier)
        constexpr int RN = GM == 2 ? NT / BM : 1;  // parts of a row's sum
        if constexpr (GM == 2) {
            float v = 0.0f;
#pragma unroll
            for (int i = 0; i < NG; ++i) v += bsum[i];
            red[gpx * BM + grow] = v;
        } else {
#pragma unroll
            for (int i = 0; i < NG; ++i) {
                const float v = lane_sum<PS / GE>(bsum[i]);
                if (gpx == 0) red[grow + i * GRS] = v;
            }
        }
        __syncthreads();
        if (tid < BM && m0 + tid < p.Cout) {
            float v = 0.0f;
#pragma unroll
            for (int k = 0; k < RN; ++k) v += red[k * BM + tid];
            unsafeAtomicAdd(p.gb_acc + m0 + tid, v);
        }
    }
}

// Images of one launch over g's images (g.B of them): the bytes of their xt and
// their pixels stay in 32 bits (one image always fits, see make_geo).
static int f32_images(const Geo &g) {
    const long long img = std::max((long long)g.H * g.W * g.cs * 4, 2LL * g.N);
    return (int)std::max(1LL, std::min((long long)g.B, 0xffff0000LL / img));
}

template <int CB>
static void colgrad_f32_launch(CgF32Params &c, hipStream_t s) {
    c.ptiles = ceil_div(c.total, 32 * (4 / CB));
    if (c.p.go_nhwc) dcn2_colgrad_f32_kernel<CB, true><<<c.ptiles * c.ctiles, 256, 0, s>>>(c);
    else dcn2_colgrad_f32_kernel<CB, false><<<c.ptiles * c.ctiles, 256, 0, s>>>(c);
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
        // 64 pixels x 64 channels (or 128 x 32): 128 x 64 reads the weight once for
        // twice the pixels but leaves three workgroups to a CU, 62 against 54 us at
        // Cout 256, K 64, 32 x 56 x 56 and 58 against 50 at 256, 1024, 32 x 14 x 14.
        if (CT == 32) colgrad_f32_launch<1>(c, s);
        else colgrad_f32_launch<2>(c, s);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int IB, int WM, int CB>
static void gradw_f32_launch(GwF32Params &c, const Geo &g, int ncu, hipStream_t s) {
    constexpr int NT = 64 * WM * CB, PS = NT / (8 * CB);
    c.mtiles = ceil_div(g.Cout, 32 * IB * WM);
    const long long tiles = (long long)c.mtiles * c.ktiles;
    // Three workgroups to a CU (of the 128-row ones), each with at least four
    // steps.  Kernel us at 1 / 2 / 3 / 4 to a CU: 77 / 63 / 66 / 74 at Cout 256, K
    // 64, 32 x 56 x 56; 75 / 59 / 57 / 62 at 256, 1024, 32 x 14 x 14; 80 / 59 / 58 /
    // 63 at 2048, 512, 32 x 7 x 7; 74 / 60 / 58 / 64 at 128, 1152, 4 x 56 x 56: more
    // ranges add more partial blocks with atomics, fewer leave gathers exposed.
    c.splits = (int)std::max(1LL, std::min(ncu * 3LL / tiles, (long long)ceil_div(c.total, PS) / 4));
    const unsigned grid = (unsigned)(c.splits * tiles);
    const int gm = c.p.go_nhwc ? 2 : (g.N % 4 == 0 && ((uintptr_t)c.p.gout & 15) == 0 ? 0 : 1);
    auto launch = [&](auto mask) {
        constexpr bool M = decltype(mask)::value;
        if (gm == 0) dcn2_gradw_f32_kernel<IB, WM, CB, 0, M><<<grid, NT, 0, s>>>(c);
        else if (gm == 1) dcn2_gradw_f32_kernel<IB, WM, CB, 1, M><<<grid, NT, 0, s>>>(c);
        else dcn2_gradw_f32_kernel<IB, WM, CB, 2, M><<<grid, NT, 0, s>>>(c);
    };
    if (c.p.mask) launch(std::true_type{});
    else launch(std::false_type{});
}

hipError_t launch_gradw_f32(const Geo &g, const BwdParams &p, int ncu, hipStream_t s) {
    GwF32Params c;
    c.p = p;
    const int CT = f32_chan_tile(g), nimg = f32_images(g);
    c.dN = fast_div(g.N);
    c.dWo = fast_div(g.Wo);
    c.cpg = g.Cgp / CT;
    c.cpt = g.cpt * 32 / CT;
    c.cpw = g.cpw * 32 / CT;
    c.cog = g.gsplit ? g.Cout / g.WG : 0;
    c.ktiles = g.KK * c.cpw;
    for (int b = 0; b < g.B; b += nimg) {
        const int nb = std::min(nimg, g.B - b);
        c.b0 = b;
        c.total = nb * g.N;
        c.x_bytes = (uint32_t)((long long)nb * g.H * g.W * g.cs * 4);
        if (CT == 32) gradw_f32_launch<1, 4, 1>(c, g, ncu, s);
        else gradw_f32_launch<2, 2, 2>(c, g, ncu, s);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace dcn2
