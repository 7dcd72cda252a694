// Prints what the library's host code plans, without a GPU: linked before the
// library's objects, the launchers defined here take the place of its own.
//
// Each input line: slice budget, option gi_push, the 18 fields of a dcn2_desc.
// First one line: whether the forward keeps the weight in registers, whether it is one of
// few tiles, and whether the backward reads a padded copy of grad_output.  Then per backward slice one line: images, whether grad_input goes by cells, and for
// gi_acc, the hand-off rows, the corner sums and the records the bytes that the slice
// uses and those that the workspace holds for it.
#include <cstdio>

#include "../dcnv2_amd/csrc/dcn2_kernels.h"
#include "../include/dcnv2_amd.h"

namespace dcn2 {

hipError_t launch_pack(const Geo &, const void *, void *, const void *, void *, void *, bool, hipStream_t,
                       const ClearList *, const void *, void *) {
    return hipSuccess;
}

hipError_t launch_backward(const Geo &g, const void *, const void *, const void *, const void *, const void *,
                           const void *, void *, void *, void *, void *, void *, float *gi_acc, float *gw_acc,
                           float *, void *cgm, void *rsc, float *csum, void *rec, int *bcnt, int *, int *, int *,
                           float *, const void *, bool, hipStream_t) {
    const GatherGeo gg = gather_geometry(g);
    auto room = [](const void *a, const void *b) { return (long)((const char *)b - (const char *)a); };
    const long sums = (long)csum_planes(g) * g.B * g.G * g.KK * g.N * 16;
    printf("%d %d  %ld %ld  %ld %ld  %ld %ld  %ld %ld\n", g.B, g.by_cells, gg.acc_bytes, room(gi_acc, gw_acc),
           gg.rows * g.Cgp * gg.row_esz, room(cgm, rsc), sums, room(csum, rec), gg.rows * 12, room(rec, bcnt));
    return hipSuccess;
}

}  // namespace dcn2

int main() {
    long long budget, push;
    while (scanf("%lld %lld", &budget, &push) == 2) {
        dcn2_desc d;
        static_assert(sizeof(d) == 18 * sizeof(int32_t), "plain int32 fields");
        for (int i = 0; i < 18; ++i)
            if (scanf("%d", (int32_t *)&d + i) != 1) return 2;
        dcn2_set_option(DCN2_OPT_BWD_SLICE_BYTES, budget);
        dcn2_set_option(DCN2_OPT_GI_PUSH, push);
        dcn2::Geo g;
        if (dcn2::make_geo(&d, g)) return 3;
        printf("%d %d %d\n", g.rw, (int)dcn2::forward_few_tiles(g), g.go_pad);
        char *const p = (char *)0x10000;  // (never read: nothing is launched)
        const int rc = dcn2_backward(&d, p, p, p, p, p, p, p, p, p, p, p, dcn2_backward_workspace_bytes(&d), nullptr);
        if (rc) return fprintf(stderr, "%s\n", dcn2_last_error()), 3;
        printf("\n");
    }
    return 0;
}
