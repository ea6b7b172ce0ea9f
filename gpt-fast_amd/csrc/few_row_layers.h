// What one native call needs to launch the few-row step of a run of plain decoder layers: pre-norm
// attention with interleaved rotation and a gated feed-forward (gemm_bf16.hip: gfa_few_row_layers_bf16,
// core.hip: gfa_few_row_layers_f32).
#pragma once
#include "common.h"

// One layer's tensors.
struct FewRowLayer {
    const void *wqkv, *wo, *w13, *w2;
    const float *norm_mixer, *norm_ffn;   // weights of the norms before the attention and before the feed-forward
    void *k_pages, *v_pages;
    const int* table;
};

// What all layers share.
struct FewRowStep {
    // bfloat16: the rows of the first layer's norm: plain [M, D], or with ssq0 [t0, gfa_share_rows(M)] in the two
    // halves of gfa_skinny_into_chain_bf16
    const void* x0;
    const float* ssq0;
    float* residual;                      // [M, D], updated in place
    const float* freqs;
    const int *tok_seq, *tok_pos, *q_start, *start_pos;
    void* work;                           // of the entry's own size
    // bfloat16: gfa_attention_bf16 and gfa_attention_tiled_bf16, which another library holds
    int (*attend)(const void*, const void*, const void*, const int*, const int*, const int*, int, void*, float*, float*,
                  int, int, int, int, int, float, int, int, int, int, int, int, int, hipStream_t);
    int (*attend_tiled)(const void*, const void*, const void*, const int*, const int*, const int*, int, void*, int, int,
                        int, int, int, float, int, int, int, hipStream_t);
    int t0, M, D, I, H, Hkv, hd, rot, table_stride, n_seqs, window;
    int gate_mode;                        // bfloat16: 3 silu, 6 gelu (tanh form); float32: 0, 1
    int rows_tiled;                       // (token, head) rows per kv head for attend_tiled, 0: attend
    int row_tiles, n_waves, max_tiles, n_splits, one_token_each;
    float eps_mixer, eps_ffn, scale;
};
