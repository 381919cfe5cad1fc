// The order in which a wave of the plain grouped product (pf_moe_prefill.hip) requests and multiplies the weight batches of
// its rows, in one place for the kernel and for the host-side check (tests/check_plain_walk.cpp).
//
// A row's columns pass in rounds of PF_PLAIN_CHUNK staged activation columns; a batch is `batch_cols` columns of weights
// (PF_PLAIN_CHUNK is whole batches of every format).  A wave takes every `parts`-th batch of the whole row, from batch `part`
// on, and requests a batch's successor before it multiplies it.  Batches are counted over the whole row and not within a
// round: a round of the 256-column format holds two batches, fewer than the four waves of a split workgroup, so a wave's next
// batch lies a round or two further on.
#pragma once

#define PF_PLAIN_CHUNK 512

#ifdef __HIPCC__
#define PF_WALK_FN __device__ __forceinline__
#else
#define PF_WALK_FN inline
#endif

// stage(c0, cols): the round's columns c0 .. c0 + cols - 1, by every wave of the workgroup (barriers inside).
// request(batch): the batch's weights are on their way.  take(): what was requested last is the present batch.
// multiply(k0, cols): the present batch against the staged columns from k0 on.
template <class Stage, class Request, class Take, class Multiply>
PF_WALK_FN void pf_plain_walk(int a_cols, int batch_cols, int part, int parts, bool active, Stage stage, Request request, Take take,
                              Multiply multiply) {
    const int batches = (a_cols + batch_cols - 1) / batch_cols;
    int batch = part;
    if (active && batch < batches) request(batch);   // on its way while the first columns are staged
    for (int c0 = 0; c0 < a_cols; c0 += PF_PLAIN_CHUNK) {
        const int cols = a_cols - c0 < PF_PLAIN_CHUNK ? a_cols - c0 : PF_PLAIN_CHUNK;
        stage(c0, cols);
        if (!active) continue;
        for (; batch * batch_cols < c0 + cols; batch += parts) {
            take();
            if (batch + parts < batches) request(batch + parts);
            multiply(batch * batch_cols - c0, cols);
        }
    }
}
