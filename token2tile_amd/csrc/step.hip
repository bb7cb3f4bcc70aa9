// One attention call's launches in one entry point.  The stages are the
// library's own entry points, called in the order of MaskedStepDeploy.step
// (operator/deploy_step.py:286-477): a small call's kernels take 2-40 us each,
// and reaching each of them through its own foreign call with its own checks
// and workspace queries took the host longer than the GPU took to run them
// (2 x 4096 tokens: 375 us of host time for 225 us of kernels; now 175).
#include "t2t_common.h"

#define ST_CHECK(x)      \
  do {                   \
    int _rc = (x);       \
    if (_rc) return _rc; \
  } while (0)

extern "C" int t2t_step(const t2t_step_args* a, unsigned stages, void* stream) {
  T2T_REQUIRE(a && a->struct_bytes == sizeof(t2t_step_args), "step: argument struct of %zu bytes, need %zu",
              a ? a->struct_bytes : (size_t)0, sizeof(t2t_step_args));
  const int H = a->H, N = a->N, CQ = a->CQ, CK = a->CK, dt = a->dtype;
  const long long hs = (long long)N * 128;
  // Stages asked for together share kernels where their results allow: both
  // projections one launch; the finalised centroids come from the key sums
  // and the tile image from the value statistics (2 x 4096 tokens: three
  // launches of 3-5 us less), unless a FINALIZE after them is still to write the
  // centroids that the image holds
  const unsigned pair = T2T_STEP_PROJECT_Q | T2T_STEP_PROJECT_K;
  const bool fin = (stages & T2T_STEP_KMEANS) && (stages & T2T_STEP_FINALIZE) && a->ck16 && a->cks;
  const bool tiles = (stages & T2T_STEP_TILES) && CK == 2048 && a->cks && a->tiles &&
                     (fin || ((stages & T2T_STEP_VSTATS) && !(stages & T2T_STEP_FINALIZE)));
  if ((stages & pair) == pair)
    ST_CHECK(t2t_project_pair(a->q, a->q_head_stride, a->q_row_stride, a->Uq, a->QU, a->k,
                              a->k_head_stride, a->k_row_stride, a->Uk, a->KU, dt, H, N, stream));
  else if (stages & T2T_STEP_PROJECT_Q)
    ST_CHECK(t2t_project_strided(a->q, dt, a->Uq, a->QU, H, N, 128, 32, a->q_head_stride,
                                 a->q_row_stride, stream));
  else if (stages & T2T_STEP_PROJECT_K)
    ST_CHECK(t2t_project_strided(a->k, dt, a->Uk, a->KU, H, N, 128, 32, a->k_head_stride,
                                 a->k_row_stride, stream));
  const T2tCentroidOut co{fin ? a->ck16 : nullptr, fin || tiles ? a->cks : nullptr, a->scale,
                          tiles ? a->tiles : nullptr};
  if (stages & T2T_STEP_KMEANS)
    ST_CHECK(t2t_kmm_run_out(a->QU, a->KU, a->v, dt, a->v_head_stride, a->v_row_stride, a->cq0, a->ck0,
                             a->qlab, a->cq2, a->klab, a->ck2, a->qcounts, a->qperm, a->kcounts,
                             a->kperm, a->vp, a->sumv, a->lam, H, N, CQ, CK, a->pin_tail, a->ws_kmm,
                             a->ws_kmm_bytes, co, stream));
  if (stages & T2T_STEP_VSTATS)
    ST_CHECK(t2t_vstats_gather_out(a->v, dt, a->v_head_stride, a->v_row_stride, a->kperm, a->kcounts,
                                   a->vp, a->sumv, a->lam, H, N, CK, a->ws_vst, a->ws_vst_bytes, co,
                                   stream));
  if ((stages & T2T_STEP_FINALIZE) && !fin)
    ST_CHECK(t2t_centroid_finalize(a->ck2, a->ck16, a->cks, a->scale, H, CK, 32, stream));
  if (stages & T2T_STEP_SELECT) {
    ST_CHECK(t2t_score_select_packed(a->QU, a->cks, a->kcounts, a->qperm, a->qcounts, a->ns, a->unip,
                                     a->rowcnt, H, N, CQ, a->ws_sel, a->ws_sel_bytes, stream));
    if (a->pin_tail) ST_CHECK(t2t_union_or_last(a->unip, H, CQ, CK, stream));
  }
  if ((stages & T2T_STEP_GATHER_K) && a->kp) {
    T2T_REQUIRE(a->k_head_stride == hs && a->k_row_stride == 128, "step: the separate K gather needs "
                "contiguous k");
    ST_CHECK(t2t_fast_gather(a->k, dt, a->kperm, a->kp, H, N, 128, stream));
  }
  if (stages & T2T_STEP_PLAN)
    ST_CHECK(t2t_tile_plan(a->qcounts, a->kcounts, a->unip, a->plan, H, N, CQ, stream));
  if (stages & T2T_STEP_EXACT)
    ST_CHECK(t2t_exact_split_parts(
        a->q, a->q_head_stride, a->q_row_stride, a->kp ? a->kp : a->k, a->kp ? hs : a->k_head_stride,
        a->kp ? 128 : a->k_row_stride, a->vp ? a->vp : a->v, a->vp ? hs : a->v_head_stride,
        a->vp ? 128 : a->v_row_stride, a->kperm, a->kp ? 0 : (a->vp ? 1 : 2), dt, a->kcounts, a->unip,
        a->qlab, a->qperm, a->plan, a->out, a->out_head_stride, a->out_row_stride, a->lse, H, N, CQ,
        a->ws_split, a->ws_split_bytes, stream));
  if ((stages & T2T_STEP_TILES) && !tiles) ST_CHECK(t2t_centroid_tiles(a->cks, a->sumv, a->tiles, H, stream));
  if (stages & T2T_STEP_RESIDUAL)
    ST_CHECK(t2t_resid_merge_parts(a->out, a->out_head_stride, a->out_row_stride, a->lse, a->QU,
                                   a->tiles, a->kcounts, a->unip, a->qlab, a->qperm, a->plan, a->lam,
                                   a->tailw, dt, H, N, CQ, a->ws_split, a->ws_split_bytes, stream));
  return T2T_OK;
}
