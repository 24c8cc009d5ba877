// ti_bonsai_batch.h — launchers of the Bonsai decoder's T-token kernels (k_bonsai_batch.hip).
#pragma once
#include "ti_internal.h"

#define TI_BB_TOKENS 256      // tokens of one batch, at most; longer prompts run in batches
#define TI_BB_SPLITS 16       // key ranges of one attention launch, at most
#define TI_BB_ROWSPLITS 65536 // (token, head, key range) partials of one launch, at most

// the quantized rows that a projection reads: act [T][n], xsum [T][n / 64]
struct ti_bb_rows {
    uint32_t* act;
    int32_t* xsum;
    int T;
};
// x rows (embedded from hist when emb is given, else x + add / add_scale) -> RMSNorm -> rows, scale [T]
int ti_bb_norm(ti_ctx* c, const ti_bb_rows& R, float* x, const float* add, const float* add_scale, const float* w, float eps,
               int H, const uint32_t* hist, const uint16_t* emb, int vocab, float* scale);
int ti_bb_swiglu(ti_ctx* c, const ti_bb_rows& R, const float* g, const float* u, const float* gu_scale, int I, float* scale);
// rope, kc and vc stand at the first token's position
int ti_bb_rope(ti_ctx* c, const float* q, const float* k, const float* v, const float* act_scale, const float* qn,
               const float* kn, const float* rope, float eps, float* qrot, float* kc, float* vc, int T, int nHq, int nKv);
// kc and vc stand at position 0
int ti_bb_attn(ti_ctx* c, const ti_bb_rows& R, const float* qrot, const float* kc, const float* vc, int pos, int nHq, int nKv,
               float* po, float* pml, long rowsplits, float* scale);
