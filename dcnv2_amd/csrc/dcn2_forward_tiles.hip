// Fused DCNv2 forward in small tiles: bilinear, mask-modulated sampling into LDS
// feeding 32x32 MFMAs (the reference's im2colcuda + gemm_cuda, com.cu:46-195,
// without the column matrix in HBM).  Serves every fp32 shape, and the 2-byte
// shapes that have too few 128-pixel tiles for the persistent kernels of
// dcn2_forward.hip / dcn2_forward_rw.hip or more rows than those hold.
//
// Bound: for fp32 the matrix rate (a 32x32x2 MFMA holds the matrix core for 64
// cycles, so workgroups of 4 or 8 waves hide their sampling behind each other's
// MFMAs without role-specialised waves); for the small problems the chain of
// gathers, blend and barrier of a step (about 1.2 us at one workgroup to a CU;
// issuing the gathers two steps ahead and fetching table entries a step early
// both measured the same).  What cost the time before was idle CUs and padding: a
// 14 x 14 map filled 196 of 256 tile pixels and ran two workgroups per image.  So:
//   * output pixels are numbered through the whole batch (pixel i of the launch
//     is pixel i % N of image i / N), and a tile may span images;
//   * the tile is chosen by how many workgroups it gives (forward_tiles), and where
//     they are few K is split over the waves of a workgroup (WK).
// Measured against the kernels this replaces (us): fp32 79.0 -> 64.9 at Cout 256,
// K 64, 32 x 56 x 56; 174.9 -> 51.9 at 256, 1024, 32 x 14 x 14; 100.2 -> 48.1 at
// 2048, 512, 32 x 7 x 7; 111.2 -> 58.2 at 128, 1152, 4 x 56 x 56 (3x3); 31.3 -> 9.6
// at 32, 144, 32 x 32 (3x3).  The 3.29 GFLOP of the first three take 21 us at the
// 154 TFLOP/s a large fp32 matrix product reaches here.  16 bits, 3x3: 50.5 -> 31.0
// at 256, 2304, 50 x 84 (channels-last 51.1 -> 28.9); 65.3 -> 21.4 at 256, 2304, 2 x 25 x
// 42; 92.3 -> 31.8 at 512, 4608, 32 x 32; 25.7 -> 13.0 at 128, 1152, 64 x 64.
//
// A workgroup owns 32*IB*WM output rows x 32*JB*WN pixels and walks K in steps
// of WK chunks (128 bytes of channels of one tap and group each).  Step s:
//   weight fragments and corner gathers of step s+1, offsets of step s+2 issued
//   MFMAs of step s over its LDS stage
//   blend of step s+1 into the other stage; barrier
// Operands are one 16-byte read per lane: a row's piece from the fragment-ordered
// weight, a pixel's from LDS (pitch 144 bytes: the reads of 16 lanes cover all
// banks once).  For 2-byte types that is one 32x32x16 MFMA; for fp32 four 32x32x2
// ones, the e-th multiplying channels e and e + 4 of a group of 8.
#include <algorithm>
#include <type_traits>

#include "dcn2_common.h"
#include "dcn2_sampler.h"
#include "dcn2_kernels.h"
#include "../../include/dcnv2_amd.h"

namespace dcn2 {

struct TileParams {
    const void *xt, *wp, *offset, *mask, *bias;
    const int4 *tab;
    void *out;
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

constexpr int kTilePitch = 144;  // bytes per pixel of an LDS stage (one chunk: 128 bytes)

template <typename T, int IB, int JB, int WM, int WN, int WK, bool MASK, bool ONHWC>
__global__ __launch_bounds__(64 * WM * WN * WK) void dcn2_fwd_tile_kernel(const TileParams p) {
    constexpr int NT = 64 * WM * WN * WK;
    constexpr int BM = 32 * IB * WM, BN = 32 * JB * WN;
    constexpr int PPP = NT / 8;            // (pixel, chunk) pairs sampled per pass
    constexpr int SPT = BN * WK / PPP;  // sampling slots (pixel, chunk, 4 channels) per thread
    static_assert(BN * WK % PPP == 0 && (BN % PPP == 0 || PPP % BN == 0), "whole passes");
    static_assert(WK == 1 || IB * JB * 4 % WK == 0, "the K split's reduction shares row quads out evenly");
    // the two sampled stages; after the last one the K split's partial blocks
    constexpr int kStage = 2 * WK * BN * kTilePitch, kRed = WK > 1 ? WK * WM * WN * 4 * 64 * 16 : 0;
    __shared__ __attribute__((aligned(16))) char smem[kStage > kRed ? kStage : kRed];
    char(&sB)[2][WK][BN][kTilePitch] = *reinterpret_cast<char(*)[2][WK][BN][kTilePitch]>(smem);

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

    // Slot i of a thread: chunk slot_k(i) of the step, pixel slot_px(i), 16-byte piece tid % 8 of the chunk; 8 lanes read one 128-byte corner line.
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
        ooff[i] = (b * (uint32_t)p.off_bs + nn) * (uint32_t)sizeof(T);
        moff[i] = MASK ? (b * (uint32_t)p.msk_bs + nn) * (uint32_t)sizeof(T) : 0u;
        ximg[i] = b * (uint32_t)(p.H * p.W);
    }
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void *>(p.xt), (short)0, (int)p.x_bytes, 0x00020000);
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

    // Sampling state of a slot: the plane its descriptor (corner byte offsets
    // and mask-folded weights) is of, and the offsets loaded for the next one.
    // Chunks of one plane (the channel chunks of a group) share a descriptor.
    T dy[SPT], dx[SPT], mv[SPT];
    float w[SPT][4];
    uint32_t co[SPT][4];
    int plane_d[SPT], plane_o[SPT];
    auto load_om = [&](int i, const Cursor &c) __attribute__((always_inline)) {
        const int plane = tab[4 * c.ch];
        if (plane == plane_d[i] || plane == plane_o[i]) return;
        plane_o[i] = plane;
        const char *ob = (const char *)((const T *)p.offset + (size_t)plane * 2 * p.N);
        dy[i] = *(const T *)(ob + ooff[i]);
        dx[i] = *(const T *)(ob + (size_t)p.N * sizeof(T) + ooff[i]);
        if (MASK) mv[i] = *(const T *)((const char *)((const T *)p.mask + (size_t)plane * p.N) + moff[i]);
    };
    u32x4 raw[SPT][4];
    auto gather = [&](int i, const Cursor &c) __attribute__((always_inline)) {
        const ConstTab e = tab + 4 * c.ch;
        if (e[0] != plane_d[i]) {
            plane_d[i] = e[0];
            const float y = (float)(by[i] + e[1]) + to_f32(dy[i]);
            const float x = (float)(bx[i] + e[2]) + to_f32(dx[i]);
            float m = MASK ? mask_value(to_f32(mv[i]), p.msk_logit) : 1.0f;
            m = live[i] ? m : 0.0f;
            const SamplePos sp = sample_pos(y, x, p.H, p.W);
            const float hy = (1.0f - sp.ly) * m, ly = sp.ly * m, hx = 1.0f - sp.lx, lx = sp.lx;
            const uint32_t base = (ximg[i] + (uint32_t)(sp.y0 * p.W + sp.x0)) * (uint32_t)(p.cs * sizeof(T)) + cq * 16u;
            const uint32_t px = (uint32_t)p.cs * (uint32_t)sizeof(T), row = px * (uint32_t)p.W, out = p.x_bytes;
            // (weight 0 as well outside: 0 times a mask that is not finite is not 0)
            const bool v[4] = {sp.vy0 && sp.vx0, sp.vy0 && sp.vx1, sp.vy1 && sp.vx0, sp.vy1 && sp.vx1};
            const uint32_t o[4] = {base, base + px, base + row, base + row + px};
            const float wq[4] = {hy * hx, hy * lx, ly * hx, ly * lx};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                co[i][q] = v[q] ? o[q] : out;
                w[i][q] = v[q] ? wq[q] : 0.0f;
            }
        }
        // (a corner outside the image has an offset past the buffer and reads 0)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            raw[i][q] = __builtin_amdgcn_raw_buffer_load_b128(xrs, (int)co[i][q], e[3] * (int)sizeof(T), 0);
    };
    auto blend = [&](int st) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < SPT; ++i) {
            constexpr int E = 16 / sizeof(T);
            float v[E];
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float x[E];
                Unpack<T>::run(make_uint4(raw[i][q].x, raw[i][q].y, raw[i][q].z, raw[i][q].w), x);
#pragma unroll
                for (int e = 0; e < E; ++e) v[e] = fmaf(w[i][q], x[e], v[e]);
            }
            *reinterpret_cast<uint4 *>(&sB[st][slot_k(i)][slot_px(i)][cq * 16]) = pack16<T>(v);
        }
    };
    // weight fragments: row block rb, chunk ch, quarter ks of it -> 64 lanes x 16 bytes
    u32x4 a[2][IB][4];
    const u32x4 *wrow = (const u32x4 *)p.wp + (size_t)(m0 / 32) * p.nch_all * 256 + lane;
    auto load_a = [&](int set, const Cursor &cur) __attribute__((always_inline)) {
        const u32x4 *src = wrow + (size_t)cur.ch * 256;
#pragma unroll
        for (int i = 0; i < IB; ++i)
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) a[set][i][ks] = src[(size_t)i * p.nch_all * 256 + ks * 64];
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
        typedef typename Mma<T>::frag frag;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            u32x4 bf[JB];
#pragma unroll
            for (int j = 0; j < JB; ++j)
                bf[j] = *reinterpret_cast<const u32x4 *>(
                    &sB[set][wk][(wn * JB + j) * 32 + (lane & 31)][ks * 32 + 16 * (lane >> 5)]);
            auto mul = [&](auto af, auto bv, int i, int j) __attribute__((always_inline)) {
                acc[i][j] = ONHWC ? Mma<T>::mma(bv, af, acc[i][j]) : Mma<T>::mma(af, bv, acc[i][j]);
            };
            if constexpr (sizeof(T) == 4) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < IB; ++i)
#pragma unroll
                        for (int j = 0; j < JB; ++j)
                            mul(__uint_as_float(a[set][i][ks][e]), __uint_as_float(bf[j][e]), i, j);
            } else {
#pragma unroll
                for (int i = 0; i < IB; ++i)
#pragma unroll
                    for (int j = 0; j < JB; ++j)
                        mul(__builtin_bit_cast(frag, a[set][i][ks]), __builtin_bit_cast(frag, bf[j]), i, j);
            }
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
            const float bv = p.bias ? to_f32(((const T *)p.bias)[m]) : 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int pl = pb + 8 * rq + lr + e;
                if (pl < live_px) ((T *)p.out)[(size_t)(n0 + pl) * p.Cout + m] = from_f32<T>(v[e] + bv);
            }
        } else {
            const int pl = pb + lc;
            if (pl >= live_px) return;
            const unsigned n = n0 + pl, b = n / (unsigned)p.N;
            T *o = (T *)p.out + (size_t)b * p.Cout * p.N + (n - b * (unsigned)p.N);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = mb + 8 * rq + lr + e;
                if (m < p.m_end) o[(size_t)m * p.N] = from_f32<T>(v[e] + (p.bias ? to_f32(((const T *)p.bias)[m]) : 0.0f));
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

template <typename T, int IB, int JB, int WM, int WN, int WK>
static hipError_t launch_tile(TileParams p, int rows, bool nhwc, hipStream_t s) {
    constexpr int NT = 64 * WM * WN * WK;
    p.mtiles = ceil_div(rows, 32 * IB * WM);
    p.tiles = ceil_div(p.total, 32 * JB * WN) * p.mtiles;
    if (p.mask && nhwc) dcn2_fwd_tile_kernel<T, IB, JB, WM, WN, WK, true, true><<<p.tiles, NT, 0, s>>>(p);
    else if (p.mask) dcn2_fwd_tile_kernel<T, IB, JB, WM, WN, WK, true, false><<<p.tiles, NT, 0, s>>>(p);
    else if (nhwc) dcn2_fwd_tile_kernel<T, IB, JB, WM, WN, WK, false, true><<<p.tiles, NT, 0, s>>>(p);
    else dcn2_fwd_tile_kernel<T, IB, JB, WM, WN, WK, false, false><<<p.tiles, NT, 0, s>>>(p);
    return hipGetLastError();
}

template <typename T>
static hipError_t forward_tiles(const Geo &g, const void *xt, const void *wp, const void *tab,
                              const void *offset, const void *mask, const void *bias, void *out,
                              hipStream_t s) {
    TileParams p;
    p.wp = wp;
    p.tab = (const int4 *)tab;
    p.bias = bias;
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
    const long long img = std::max({(long long)g.H * g.W * g.cs * g.esz, g.off_bs * g.esz, g.msk_bs * g.esz, 2LL * g.N});
    const int nimg = (int)std::max(1LL, std::min((long long)g.B, 0xffff0000LL / img));
    // One launch over all rows and chunks, or one per weight group over the
    // group's rows (a multiple of 128) and chunks.
    const int groups = g.gsplit ? g.WG : 1, rows = g.Cout / groups;
    p.cpw = g.gsplit ? g.cpw : g.cpt;
    p.nch = g.KK * p.cpw;
    for (int b = 0; b < g.B; b += nimg) {
        const int nb = std::min(nimg, g.B - b);
        p.total = nb * g.N;
        p.x_bytes = (uint32_t)((long long)nb * g.H * g.W * g.cs * g.esz);
        p.xt = (const T *)xt + (size_t)b * g.H * g.W * g.cs;
        p.offset = (const T *)offset + (size_t)b * g.off_bs;
        p.mask = mask ? (const T *)mask + (size_t)b * g.msk_bs : nullptr;
        p.out = (T *)out + (size_t)b * g.Cout * g.N;
        for (int w = 0; w < groups; ++w) {
            p.cb = w * p.cpw;
            p.m_base = w * rows;
            p.m_end = p.m_base + rows;
            // Tile rule for this card's 256 CUs, measured in us (rows, K, pixels; tile: rows x pixels, all with
            // 8 waves and one or two workgroups to a CU unless noted):
            //   64x32, K over 4 groups of waves, while one workgroup to a CU does: fp16
            //     13.5 against 16.2 (128x32) at 128, 1152, 4096; 32 against 39 at 512,
            //     4608, 1024; fp32 9.6 against 11.6 at 32, 288, 1024.  Past that 38
            //     against 24 at 256, 2304, 2100.
            //   128x32, K over 2, while two and a half do: fp32 50.7 against 79.9 (256x64)
            //     at 256, 1024, 6272; 16 bits, more than 128 rows and 8 chunks: two, fp16
            //     38.2 at 256, 2304, 8192 but past that 52.3 against 48.9 at 8704, 77.8 /
            //     72.5 at 512, 3136, 4352 and 115.7 / 97.8 at 1000, 4800, 2176.
            //   256x64 (a pixel is sampled once for 256 rows): fp32 64.7 against 71.1
            //     for 128x64 at 256, 64, 100352; 48.7 against 51.7 at 2048, 512, 1568.
            //   128x64 (fp32: 16-bit layers of 65 to 128 rows that come here stay below the
            //     line above) and 64x64 (4 waves): the rest, whose rows 256x64 would pad.
            auto tiles = [&](int bm, int bn) { return (long long)ceil_div(rows, bm) * ceil_div(p.total, bn); };
            const int most = sizeof(T) == 2 && rows > 128 && p.nch > 8 ? 512 : 640;
            hipError_t e;
            if (tiles(64, 32) <= 256)
                e = launch_tile<T, 1, 1, 2, 1, 4>(p, rows, g.out_nhwc, s);
            else if (rows > 64 && tiles(128, 32) <= most)
                e = launch_tile<T, 1, 1, 4, 1, 2>(p, rows, g.out_nhwc, s);
            else if (rows > 128)
                e = launch_tile<T, 1, 2, 8, 1, 1>(p, rows, g.out_nhwc, s);
            else if constexpr (sizeof(T) == 4)
                e = rows > 64 ? launch_tile<T, 1, 2, 4, 1, 1>(p, rows, g.out_nhwc, s)
                              : launch_tile<T, 1, 1, 2, 2, 1>(p, rows, g.out_nhwc, s);
            else
                e = launch_tile<T, 1, 1, 2, 2, 1>(p, rows, g.out_nhwc, s);
            if (e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

hipError_t launch_forward_tiles(const Geo &g, const void *xt, const void *wp, const void *tab,
                                const void *offset, const void *mask, const void *bias, void *out,
                                hipStream_t s) {
    switch (g.dtype) {
    case DCN2_F16: return forward_tiles<f16>(g, xt, wp, tab, offset, mask, bias, out, s);
    case DCN2_BF16: return forward_tiles<bf16>(g, xt, wp, tab, offset, mask, bias, out, s);
    default: return forward_tiles<float>(g, xt, wp, tab, offset, mask, bias, out, s);
    }
}

}  // namespace dcn2
