// Fused DCNv2 forward for fp32: bilinear, mask-modulated sampling into LDS
// feeding 32x32x2 fp32 MFMAs (the reference's im2colcuda + gemm_cuda,
// com.cu:46-195, without the column matrix in HBM).
//
// Bound: the fp32 matrix rate.  One 32x32x2 MFMA holds the matrix core for 64
// cycles, so a wave needs few operand reads per cycle, and small workgroups of
// 4 waves, several to a CU, hide the sampling behind each other's MFMAs
// without role-specialised waves.  What cost the time before (8-wave workgroups
// of 128 pixels of one image, one to a CU) was idle CUs and padding: a 14 x 14
// map filled 196 of 256 tile pixels and ran two workgroups per image.  So:
//   * output pixels are numbered through the whole batch (pixel i of the launch
//     is pixel i % N of image i / N), and a tile may span images;
//   * the tile is chosen by how many workgroups it gives (launch_forward_f32),
//     and where they are few K is split over the waves of a workgroup (WK).
// Measured against the 8-wave kernel this replaces (us): 79.0 -> 64.7 at Cout 256,
// K 64, 32 x 56 x 56; 174.9 -> 49.9 at 256, 1024, 32 x 14 x 14; 100.2 -> 48.7 at
// 2048, 512, 32 x 7 x 7; 111.2 -> 59.9 at 128, 1152, 4 x 56 x 56 (3x3); 31.3 ->
// 9.6 at 32, 144, 32 x 32 (3x3).  The 3.29 GFLOP of the first three take 21 us at
// the 154 TFLOP/s a large fp32 matrix product reaches here.
//
// A workgroup owns 32*IB*WM output rows x 32*JB*WN pixels and walks K in steps
// of WK chunks (32 channels of one tap and group each).  Step s:
//   weight fragments and corner gathers of step s+1, offsets of step s+2 issued
//   MFMAs of step s over its LDS stage
//   blend of step s+1 into the other stage; barrier
// An MFMA multiplies K pairs {e, e + 4} of an 8-channel group (e = 0..3): both
// operands of four MFMAs are then one 16-byte read per lane, four consecutive
// channels of the lane's row (weight, straight from the fragment-ordered pack)
// or pixel (LDS, pitch 36 floats: the 16-byte reads of 16 lanes cover all banks
// once).
#include <algorithm>
#include <type_traits>

#include "dcn2_common.h"
#include "dcn2_sampler.h"
#include "dcn2_kernels.h"
#include "../../include/dcnv2_amd.h"

namespace dcn2 {

struct F32FwdParams {
    const float *xt, *wp, *offset, *mask, *bias;
    const int4 *tab;
    float *out;
    int H, W, Cout, N, Wo, sh, sw, ph, pw, cs;
    int nch_all;  // chunks of the packed weight rows
    // chunk walk of this launch (see FwdParams of dcn2_forward.hip): the
    // nch = KK*cpw chunks tap*cpt + cb + i, i < cpw
    int nch, cpt, cpw, cb;
    int m_base, m_end, mtiles, tiles;  // output rows [m_base, m_end) of this launch
    int total;                         // pixels of this launch (images * N)
    uint32_t x_bytes;                  // bytes of its images of xt
    long long off_bs, msk_bs;
    int msk_logit;
};

constexpr int kF32Pitch = 36;  // floats per pixel of an LDS stage (32 channels)

template <int IB, int JB, int WM, int WN, int WK, bool MASK, bool ONHWC>
__global__ __launch_bounds__(64 * WM * WN * WK) void dcn2_fwd_f32_kernel(const F32FwdParams p) {
    constexpr int NT = 64 * WM * WN * WK;
    constexpr int BM = 32 * IB * WM, BN = 32 * JB * WN;
    constexpr int PPP = NT / 8;            // (pixel, chunk) pairs sampled per pass
    constexpr int SPT = BN * WK / PPP;  // sampling slots (pixel, chunk, 4 channels) per thread
    static_assert(BN * WK % PPP == 0 && (BN % PPP == 0 || PPP % BN == 0), "whole passes");
    static_assert(WK == 1 || IB * JB * 4 % WK == 0, "the K split's reduction shares row quads out evenly");
    // the two sampled stages; after the last one the K split's partial blocks
    constexpr int kStage = 2 * WK * BN * kF32Pitch, kRed = WK > 1 ? WK * WM * WN * 4 * 64 * 4 : 0;
    __shared__ __attribute__((aligned(16))) float smem[kStage > kRed ? kStage : kRed];
    float(&sB)[2][WK][BN][kF32Pitch] = *reinterpret_cast<float(*)[2][WK][BN][kF32Pitch]>(smem);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave / (WM * WN), wm = (wave / WN) % WM, wn = wave % WN;
    // M tiles of one pixel tile are neighbours, on one XCD: they sample the same corners
    const int t = xcd_remap(blockIdx.x, p.tiles);
    const int mt = t % p.mtiles, n0 = t / p.mtiles * BN;
    const int m0 = p.m_base + mt * BM + wm * 32 * IB;  // this wave's first row
    const int live_px = min(BN, p.total - n0);
    const int last = p.nch - 1, nsteps = (p.nch + WK - 1) / WK;

    // The chunk table is read through the constant address space (scalar loads).
    typedef const __attribute__((address_space(4))) int *ConstTab;
    const ConstTab tab = (ConstTab)(uintptr_t)p.tab;
    // Cursor over the chunk walk: j-th chunk = (tap, i), packed chunk ch,
    // advanced with compares; it stops at the last chunk.
    struct Cursor { int j, i, ch; };
    auto advance = [&](Cursor &c, int by) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < by; ++k) {
            if (c.j >= last) return;
            const bool wrap = c.i + 1 == p.cpw;
            ++c.j;
            c.ch += wrap ? 1 + p.cpt - p.cpw : 1;
            c.i = wrap ? 0 : c.i + 1;
        }
    };
    auto cursor = [&](int j) __attribute__((always_inline)) {
        Cursor c = {0, 0, p.cb};
        advance(c, j);
        return c;
    };

    // Slot i of a thread: chunk slot_k(i) of the step, pixel slot_px(i), channels 4*(tid % 8) ..; 8 lanes read one 128-byte corner line.
    const int cq = tid & 7;
    auto slot_px = [&](int i) __attribute__((always_inline)) { return (PPP * i + (tid >> 3)) % BN; };
    // (uniform over the wave)
    auto slot_k = [&](int i) __attribute__((always_inline)) {
        return WK == 1 ? 0 : (PPP <= BN ? PPP * i / BN : i * (PPP / BN) + wave * 8 / BN);
    };
    uint32_t ooff[SPT], moff[SPT], ximg[SPT];  // byte offsets of the pixel's offset, mask, image
    int by[SPT], bx[SPT];
    bool live[SPT];
#pragma unroll
    for (int i = 0; i < SPT; ++i) {
        const int pl = slot_px(i);
        live[i] = pl < live_px;
        const unsigned n = n0 + (live[i] ? pl : 0), b = n / (unsigned)p.N, nn = n - b * (unsigned)p.N;
        const int oy = nn / (unsigned)p.Wo, ox = nn - oy * p.Wo;
        by[i] = oy * p.sh - p.ph;
        bx[i] = ox * p.sw - p.pw;
        ooff[i] = (b * (uint32_t)p.off_bs + nn) * 4u;
        moff[i] = MASK ? (b * (uint32_t)p.msk_bs + nn) * 4u : 0u;
        ximg[i] = b * (uint32_t)(p.H * p.W);
    }
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(p.xt), (short)0, (int)p.x_bytes, 0x00020000);
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

    // Sampling state of a slot: the plane its descriptor (corner byte offsets
    // and mask-folded weights) is of, and the offsets loaded for the next one.
    // Chunks of one plane (the channel chunks of a group) share a descriptor.
    float dy[SPT], dx[SPT], mv[SPT], w[SPT][4];
    uint32_t co[SPT][4];
    int plane_d[SPT], plane_o[SPT];
    auto load_om = [&](int i, const Cursor &c) __attribute__((always_inline)) {
        const int plane = tab[4 * c.ch];
        if (plane == plane_d[i] || plane == plane_o[i]) return;
        plane_o[i] = plane;
        const char *ob = (const char *)(p.offset + (size_t)plane * 2 * p.N);
        dy[i] = *(const float *)(ob + ooff[i]);
        dx[i] = *(const float *)(ob + (size_t)p.N * 4 + ooff[i]);
        if (MASK) mv[i] = *(const float *)((const char *)(p.mask + (size_t)plane * p.N) + moff[i]);
    };
    f32x4 raw[SPT][4];
    auto gather = [&](int i, const Cursor &c) __attribute__((always_inline)) {
        const ConstTab e = tab + 4 * c.ch;
        if (e[0] != plane_d[i]) {
            plane_d[i] = e[0];
            const float y = (float)(by[i] + e[1]) + dy[i];
            const float x = (float)(bx[i] + e[2]) + dx[i];
            float m = MASK ? mask_value(mv[i], p.msk_logit) : 1.0f;
            m = live[i] ? m : 0.0f;
            const SamplePos sp = sample_pos(y, x, p.H, p.W);
            const float hy = (1.0f - sp.ly) * m, ly = sp.ly * m, hx = 1.0f - sp.lx, lx = sp.lx;
            const uint32_t base = (ximg[i] + (uint32_t)(sp.y0 * p.W + sp.x0)) * (uint32_t)(p.cs * 4) + cq * 16u;
            const uint32_t px = (uint32_t)p.cs * 4u, row = px * (uint32_t)p.W, out = p.x_bytes;
            co[i][0] = sp.vy0 && sp.vx0 ? base : out;
            co[i][1] = sp.vy0 && sp.vx1 ? base + px : out;
            co[i][2] = sp.vy1 && sp.vx0 ? base + row : out;
            co[i][3] = sp.vy1 && sp.vx1 ? base + row + px : out;
            w[i][0] = hy * hx;
            w[i][1] = hy * lx;
            w[i][2] = ly * hx;
            w[i][3] = ly * lx;
        }
        // (a corner outside the image has an offset past the buffer and reads 0)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            raw[i][q] = __builtin_bit_cast(
                f32x4, __builtin_amdgcn_raw_buffer_load_b128(xrs, (int)co[i][q], e[3] * 4, 0));
    };
    auto blend = [&](int st) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < SPT; ++i) {
            f32x4 v = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = fmaf(w[i][q], raw[i][q][e], v[e]);
            *reinterpret_cast<f32x4 *>(&sB[st][slot_k(i)][slot_px(i)][cq * 4]) = v;
        }
    };
    // weight fragments: row block rb, chunk ch, 8-channel group k8 -> 64 lanes x 4 floats
    f32x4 a[2][IB][4];
    const float *wrow = p.wp + (size_t)(m0 / 32) * p.nch_all * 1024 + lane * 4;
    auto load_a = [&](int set, const Cursor &cur) __attribute__((always_inline)) {
        const size_t c = (size_t)cur.ch * 1024;
#pragma unroll
        for (int i = 0; i < IB; ++i)
#pragma unroll
            for (int k8 = 0; k8 < 4; ++k8)
                a[set][i][k8] = *reinterpret_cast<const f32x4 *>(
                    wrow + (size_t)i * p.nch_all * 1024 + c + k8 * 256);
    };
    f32x16 acc[IB][JB];
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < JB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    // Channels-last output: the operands swap, so that a lane holds one row
    // (m = lane % 32) of 16 pixels and stores run along the channels.
    auto mma = [&](int set) __attribute__((always_inline)) {
#pragma unroll
        for (int k8 = 0; k8 < 4; ++k8) {
            f32x4 bf[JB];
#pragma unroll
            for (int j = 0; j < JB; ++j)
                bf[j] = *reinterpret_cast<const f32x4 *>(
                    &sB[set][wk][(wn * JB + j) * 32 + (lane & 31)][k8 * 8 + 4 * (lane >> 5)]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < IB; ++i)
#pragma unroll
                    for (int j = 0; j < JB; ++j)
                        acc[i][j] = ONHWC ? Mma<float>::mma(bf[j][e], a[set][i][k8][e], acc[i][j])
                                         : Mma<float>::mma(a[set][i][k8][e], bf[j][e], acc[i][j]);
        }
    };

    // The packed rows are padded to 128, so a wave past them holds nothing.
    const bool rows = m0 < p.m_end;
    // cursors: each slot's first chunk and the one sampled next, this wave's weight chunk
    Cursor cg[SPT], cn[SPT], ca = cursor(wk);
#pragma unroll
    for (int i = 0; i < SPT; ++i) {
        cg[i] = cursor(slot_k(i));
        cn[i] = cg[i];
        advance(cn[i], WK);
    }
    if (rows) load_a(0, ca);
#pragma unroll
    for (int i = 0; i < SPT; ++i) {
        plane_d[i] = plane_o[i] = -1;
        load_om(i, cg[i]);
    }
#pragma unroll
    for (int i = 0; i < SPT; ++i) gather(i, cg[i]);
#pragma unroll
    for (int i = 0; i < SPT; ++i) load_om(i, cn[i]);
    blend(0);
    __syncthreads();
    auto step = [&](auto set_c, int s) __attribute__((always_inline)) {
        constexpr int S = decltype(set_c)::value;
        const bool more = s + 1 < nsteps;  // (uniform)
        if (more) {
            advance(ca, WK);
            if (rows) load_a(S ^ 1, ca);
#pragma unroll
            for (int i = 0; i < SPT; ++i) gather(i, cn[i]);
#pragma unroll
            for (int i = 0; i < SPT; ++i) {
                advance(cn[i], WK);
                load_om(i, cn[i]);
            }
        }
        if (rows && (WK == 1 || s * WK + wk <= last)) mma(S);
        if (more) blend(S ^ 1);
        __syncthreads();
    };
    int s = 0;
    for (; s + 1 < nsteps; s += 2) {
        step(std::integral_constant<int, 0>{}, s);
        step(std::integral_constant<int, 1>{}, s + 1);
    }
    if (s < nsteps) step(std::integral_constant<int, 0>{}, s);

    // acc[i][j][4*rq + e] of lane l: row 8*rq + 4*(l/32) + e, pixel l%32 of
    // the 32x32 block (channels-last: the two swapped).
    const int lr = 4 * (lane >> 5), lc = lane & 31;
    auto store4 = [&](int i, int j, int rq, f32x4 v) __attribute__((always_inline)) {
        const int mb = m0 + i * 32, pb = (wn * JB + j) * 32;
        if constexpr (ONHWC) {
            const int m = mb + lc;
            if (m >= p.m_end) return;
            const float bv = p.bias ? p.bias[m] : 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int pl = pb + 8 * rq + lr + e;
                if (pl < live_px) p.out[(size_t)(n0 + pl) * p.Cout + m] = v[e] + bv;
            }
        } else {
            const int pl = pb + lc;
            if (pl >= live_px) return;
            const unsigned n = n0 + pl, b = n / (unsigned)p.N;
            float *o = p.out + (size_t)b * p.Cout * p.N + (n - b * (unsigned)p.N);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = mb + 8 * rq + lr + e;
                if (m < p.m_end) o[(size_t)m * p.N] = v[e] + (p.bias ? p.bias[m] : 0.0f);
            }
        }
    };
    if constexpr (WK == 1) {
        if (!rows) return;
#pragma unroll
        for (int i = 0; i < IB; ++i)
#pragma unroll
            for (int j = 0; j < JB; ++j)
#pragma unroll
                for (int rq = 0; rq < 4; ++rq)
                    store4(i, j, rq, f32x4{acc[i][j][4 * rq], acc[i][j][4 * rq + 1], acc[i][j][4 * rq + 2],
                                           acc[i][j][4 * rq + 3]});
    } else {
        // K split: the waves' partial blocks through LDS (the stages are free
        // after the last barrier), one (i, j) block at a time; K group wk sums
        // and stores the row quads rq of its share.
        constexpr int RQ = 4 / WK;
        f32x4(*red)[WM * WN][4][64] = reinterpret_cast<f32x4(*)[WM * WN][4][64]>(smem);
        const int wmn = wave % (WM * WN);
#pragma unroll
        for (int ij = 0; ij < IB * JB; ++ij) {
            const f32x16 v = acc[ij / JB][ij % JB];
            if (ij) __syncthreads();
#pragma unroll
            for (int rq = 0; rq < 4; ++rq)
                red[wk][wmn][rq][lane] = f32x4{v[4 * rq], v[4 * rq + 1], v[4 * rq + 2], v[4 * rq + 3]};
            __syncthreads();
#pragma unroll
            for (int k = 0; k < RQ; ++k) {
                const int rq = wk * RQ + k;
                f32x4 sum = red[0][wmn][rq][lane];
#pragma unroll
                for (int o = 1; o < WK; ++o) sum += red[o][wmn][rq][lane];
                if (rows) store4(ij / JB, ij % JB, rq, sum);
            }
        }
    }
}

template <int IB, int JB, int WM, int WN, int WK>
static hipError_t launch_fwd_f32_t(F32FwdParams p, int rows, bool nhwc, hipStream_t s) {
    constexpr int NT = 64 * WM * WN * WK;
    p.mtiles = ceil_div(rows, 32 * IB * WM);
    p.tiles = ceil_div(p.total, 32 * JB * WN) * p.mtiles;
    if (p.mask && nhwc) dcn2_fwd_f32_kernel<IB, JB, WM, WN, WK, true, true><<<p.tiles, NT, 0, s>>>(p);
    else if (p.mask) dcn2_fwd_f32_kernel<IB, JB, WM, WN, WK, true, false><<<p.tiles, NT, 0, s>>>(p);
    else if (nhwc) dcn2_fwd_f32_kernel<IB, JB, WM, WN, WK, false, true><<<p.tiles, NT, 0, s>>>(p);
    else dcn2_fwd_f32_kernel<IB, JB, WM, WN, WK, false, false><<<p.tiles, NT, 0, s>>>(p);
    return hipGetLastError();
}

hipError_t launch_forward_f32(const Geo &g, const void *xt, const void *wp, const void *tab,
                              const void *offset, const void *mask, const void *bias, void *out,
                              hipStream_t s) {
    if (g.B == 0) return hipSuccess;
    F32FwdParams p;
    p.wp = (const float *)wp;
    p.tab = (const int4 *)tab;
    p.bias = (const float *)bias;
    p.H = g.H;
    p.W = g.W;
    p.Cout = g.Cout;
    p.N = g.N;
    p.Wo = g.Wo;
    p.sh = g.sh;
    p.sw = g.sw;
    p.ph = g.ph;
    p.pw = g.pw;
    p.cs = g.cs;
    p.nch_all = g.Kp / g.KC;
    p.cpt = g.cpt;
    p.off_bs = g.off_bs;
    p.msk_bs = g.msk_bs;
    p.msk_logit = mask ? g.msk_logit : 0;
    // Images per launch: the input, offset and mask bytes and the pixel count of
    // a launch stay in 32 bits (one image always fits, see make_geo).
    const long long img = std::max({(long long)g.H * g.W * g.cs * 4, g.off_bs * 4, g.msk_bs * 4, 2LL * g.N});
    const int nimg = (int)std::max(1LL, std::min((long long)g.B, 0xffff0000LL / img));
    // One launch over all rows and chunks, or one per weight group over the
    // group's rows (a multiple of 128) and chunks.
    const int groups = g.gsplit ? g.WG : 1, rows = g.Cout / groups;
    p.cpw = g.gsplit ? g.cpw : g.cpt;
    p.nch = g.KK * p.cpw;
    for (int b = 0; b < g.B; b += nimg) {
        const int nb = std::min(nimg, g.B - b);
        p.total = nb * g.N;
        p.x_bytes = (uint32_t)((long long)nb * g.H * g.W * g.cs * 4);
        p.xt = (const float *)xt + (size_t)b * g.H * g.W * g.cs;
        p.offset = (const float *)offset + (size_t)b * g.off_bs;
        p.mask = mask ? (const float *)mask + (size_t)b * g.msk_bs : nullptr;
        p.out = (float *)out + (size_t)b * g.Cout * g.N;
        for (int w = 0; w < groups; ++w) {
            p.cb = w * p.cpw;
            p.m_base = w * rows;
            p.m_end = p.m_base + rows;
            // Tile rule: the largest tile that keeps the CUs busy.  Measured (us at
            // Cout, K, pixels; tiles in brackets):
            //   256x64, 8 waves: a pixel is sampled once for 256 rows.  64.7 against
            //     71.1 for 128x64 at 256, 64, 100352 [1568]; 48.7 against 51.7 at
            //     2048, 512, 1568 [200]; 79.9 against 57.7 at 256, 1024, 6272 [98].
            //   128x64: with K split over 8 waves when tiles are few and K long:
            //     49.9 against 57.7 at 256, 1024, 6272 [196] and 59.9 against 66.3
            //     at 128, 1152, 12544 [196]; 98.8 against 71.1 at K = 64 [3136].
            //   32 pixels, K split: 9.6 (64x32) against 11.6 (128x32) and 18.7
            //     (128x64) at 32, 288, 1024.
            auto tiles = [&](int bm, int bn) { return (long long)ceil_div(rows, bm) * ceil_div(p.total, bn); };
            hipError_t e;
            if (rows > 128 && tiles(256, 64) >= 192)
                e = launch_fwd_f32_t<1, 2, 8, 1, 1>(p, rows, g.out_nhwc, s);
            else if (rows > 64 && (tiles(128, 64) >= 512 || (tiles(128, 64) >= 160 && p.nch < 8)))
                e = launch_fwd_f32_t<1, 2, 4, 1, 1>(p, rows, g.out_nhwc, s);
            else if (rows > 64 && tiles(128, 64) >= 160)
                e = launch_fwd_f32_t<1, 2, 4, 1, 2>(p, rows, g.out_nhwc, s);
            else if (rows > 64 && tiles(128, 32) >= 128)
                e = launch_fwd_f32_t<1, 1, 4, 1, 2>(p, rows, g.out_nhwc, s);
            else if (rows <= 64 && tiles(64, 64) >= 256)
                e = launch_fwd_f32_t<1, 1, 2, 2, 1>(p, rows, g.out_nhwc, s);
            else if (rows > 32)
                e = launch_fwd_f32_t<1, 1, 2, 1, 4>(p, rows, g.out_nhwc, s);
            else
                e = launch_fwd_f32_t<1, 1, 1, 1, 4>(p, rows, g.out_nhwc, s);
            if (e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

}  // namespace dcn2
