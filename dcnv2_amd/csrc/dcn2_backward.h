// Parameters shared by the backward's kernels (dcn2_backward.hip and
// dcn2_backward_f32.hip).
#pragma once

#include "dcn2_common.h"
#include "dcn2_kernels.h"

namespace dcn2 {

// Record of a placed sample: its floor corner (y0 in the low, x0 in the high
// 16 bits, both >= -2) and the bilinear fractions (12 bytes: the consumers
// find the sample's hand-off row from the record's own position).
struct BucketRec {
    int yx;
    float ly, lx;
};

struct BwdParams {
    const void *xt, *wt, *tab, *offset, *mask, *gout;
    void *goff, *gmask;
    float *gi_acc, *gw_acc, *gb_acc;
    int B, H, W, Cout, kh, kw, sh, sw, ph, pw, dh, dw, G, Cg, Cgp, Ho, Wo, Kp, Mp;
    int tiles_per_img, splits;
    int go_nhwc;  // grad_output is channels-last [B][Ho][Wo][Cout]
    // grad_output can be read with 16-byte loads: 8 consecutive pixels of a row
    // (NCHW, N % 8 == 0) or channels of a pixel (channels-last, Cout % 8 == 0),
    // from a 16-byte aligned base
    int go_vec;
    int go_n;  // elements between rows of NCHW grad_output: N, or more in a padded copy (zeros past N)
    // grad_input gather: cell-tile buckets (see dcn2_gi_gather_kernel).  The
    // rows of all buckets are packed back to back, bucket k owning rows
    // [bstart[k], bstart[k+1]); there are at most B*G*KK*N of them (one per
    // sample), so the storage is sized exactly and no bucket can overflow.
    void *cgm;          // [rows][Cgp] masked column gradient rows (RowOf)
    unsigned char *rsc; // [rows][Cgp/32] scale codes of bf16 rows (row_block_scale)
    float *csum;        // corner sums of groups that workgroups share (csum_planes)
    int csum_n;         // its planes [B][G*KK][N][4]
    size_t csum_ps;     // floats between them (0: one plane, added to with atomics)
    struct BucketRec *rec;  // [rows] sample records, in bucket order
    int *bcnt;          // [nbuckets] samples per bucket (count pass)
    int *bstart;        // [nbuckets + 1] first row of each bucket (exclusive scan of bcnt)
    int *bcur;          // [nbuckets] next free row of each bucket (place pass)
    int *sidx;          // [B][G*KK][N] bucket row of each sample; -1 no corner inside
    int ntx, nty;       // cell tiles per row / column
    float *ring;        // [nbuckets][kRing][Cgp] grad_input sums of each window's border ring
    // grad_input written directly by the per-cell kernel and ring_final_kernel
    // (no fp32 accumulator): the caller's buffer, whether it is channels-last
    // [B][H][W][C] (else [B][C][H][W]), and whether 8-element runs take vector
    // stores there (NCHW: W % 8 == 0; channels-last: C and C/G multiples of
    // 8; both with a 16-byte aligned base)
    void *gi_out;
    int gi_nhwc, gi_vec;
    // parts a bucket's grad_input work is split into, one workgroup each: ranges
    // of channel chunks and (per-pixel kernel) interleaved passes of 8 pixels
    int gi_cs, gi_rs;
    // offset / mask (and grad_offset / grad_mask) elements between images, and
    // whether the mask buffer holds logits (see mask_value; grad_mask is then
    // the gradient of the logits)
    long long off_bs, msk_bs;
    int msk_logit;
    // grad_weight work items: gw_nch chunks per M chunk.  Ungrouped (gw_cog
    // 0): every chunk.  Weight groups whose chunks never mix: an M chunk of
    // group w = m0 / gw_cog walks only that group's chunks tap*gw_cpt +
    // w*gw_cpw + i, i < gw_cpw (the other blocks of the block-diagonal packed
    // weight are zero and their grad_weight is not kept).
    int gw_nch, gw_cpt, gw_cpw, gw_cog;
};

// dcn2_backward_f32.hip: the fp32 column gradient with its consumers
// (grad_offset / grad_mask or the corner sums in csum, and the hand-off rows).
hipError_t launch_colgrad_f32(const Geo &g, const BwdParams &p, hipStream_t s);
// The fp32 grad_weight / grad_bias, added to gw_acc / gb_acc.
hipError_t launch_gradw_f32(const Geo &g, const BwdParams &p, int ncu, hipStream_t s);

}  // namespace dcn2
