// Instances and launcher of the block-sparse prefill kernel for one 16-bit element type (the templates live in
// br_prefill_mfma_impl.h).  The including file defines BR_LAUNCH_PREFILL, the launcher's name, and, for fp16,
// BR_E16 / BR_E16_IS_F16.
#include "br_prefill_mfma_impl.h"

namespace {

// The instance is picked by what the call uses: score partials / log-sum-exp, Q rotation, or neither.
template <int D, int NW>
void launch(const BrPrefillParams& p, int grid, hipStream_t stream) {
    const bool sc = p.score_part != nullptr || p.lse != nullptr, rope = p.rope_cos != nullptr;
    if (sc && rope) hipLaunchKernelGGL((br_prefill_mfma_kernel<D, NW, false, true, true>), dim3(grid), dim3(NW * 64), 0, stream, p);
    else if (sc) hipLaunchKernelGGL((br_prefill_mfma_kernel<D, NW, false, true, false>), dim3(grid), dim3(NW * 64), 0, stream, p);
    else if (rope) hipLaunchKernelGGL((br_prefill_mfma_kernel<D, NW, false, false, true>), dim3(grid), dim3(NW * 64), 0, stream, p);
    else hipLaunchKernelGGL((br_prefill_mfma_kernel<D, NW, false, false, false>), dim3(grid), dim3(NW * 64), 0, stream, p);
}

}  // namespace

// Returns 0 on success, -1 if (D, NW) has no instantiation (nothing is launched then).
int BR_LAUNCH_PREFILL(const BrPrefillParams& p, int D, int NW, int n_cu, int combine_grid, hipStream_t stream,
                           hipEvent_t ev_start, hipEvent_t ev_stop, const BrTileScoreParams* rank) {
    // Workgroups per compute unit: two of four waves, one of more.  At head dim 64 the registers (and LDS) of a third fit; it
    // pays where there are items enough for all of them and only lengthens the start where there are not.  32/8 heads, us with
    // two and three: 8 x 30 documents of 384 to 512 tokens 578 and 520, 8 x 20 of 96 to 224 123 and 113, 4 x 20 of 160 (3520
    // items) 59.5 and 58.3; 8/2 heads, 8 x 20 of 96 to 224 (2464) 44.6 and 45.9.
    // The host knows the sizes only, so the items are counted as if every block were full: several times too many for the most
    // ragged batches.  Packed, 32/8 heads, true items of counted ones: 1 x 100 documents of 64 to 384 tokens, 5736 of 9792, 106
    // and 95 us; 2 x 50, lognormal about 160, 5360 of 13312, 97 and 90; about 90, 3328 of 11648, 62 and 64; 20 of 16 to 64 with one
    // of 512, 8 requests (3200 of 23552) 59 and 62, 4 (1600 of 11776) 39.0 and 37.7.  Where documents are short it is 5 % either
    // way, of full batches too (4 x 20 of 96 to 224: 62 and 65); a count of the real work in the plan, by which the third workgroups
    // left again, told these no better apart.
    const long long items = (long long)p.B * p.M * ((p.H + br_tokens_per_tile(p.geom) - 1) / br_tokens_per_tile(p.geom)) * p.geom.NHG;
    const int per_cu = NW > 4 ? 1 : D == 64 && items >= 10LL * n_cu ? 3 : 2;
    const int grid = n_cu * per_cu;
    if (ev_start) (void)hipEventRecord(ev_start, stream);
#define BR_CASE(DD, WW)                                   \
    if (D == DD && NW == WW) {                            \
        launch<DD, WW>(p, grid, stream);                  \
        goto launched;                                    \
    }
    BR_CASE(128, 4) BR_CASE(128, 5) BR_CASE(128, 6) BR_CASE(128, 7) BR_CASE(128, 8)
    BR_CASE(64, 4) BR_CASE(64, 5) BR_CASE(64, 6) BR_CASE(64, 7) BR_CASE(64, 8)
#undef BR_CASE
    return -1;
launched:
    if (ev_stop) (void)hipEventRecord(ev_stop, stream);
    if (D == 128) br_launch_finish_scores<BR_E16, 128>(p, NW, combine_grid, rank, stream);
    else br_launch_finish_scores<BR_E16, 64>(p, NW, combine_grid, rank, stream);
    return 0;
}
