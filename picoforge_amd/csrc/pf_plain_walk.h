// The order in which a wave of the plain grouped product (pf_moe_prefill.hip) requests and multiplies the weight batches of
// its rows, in one place for the kernel and for the host-side check (tests/check_plain_walk.cpp).
//
// A row's columns pass in rounds of PF_PLAIN_CHUNK staged activation columns; a batch is `batch_cols` columns of weights
// (PF_PLAIN_CHUNK is whole batches of every format).  The waves that share a row take its batches in turn, and each requests
// its next batch before it multiplies the present one.  No more waves take part than a round holds batches, so that a wave's
// batches lie equally in every round: two of the four waves of a split workgroup for the 256-column format, whose batches a
// wave would otherwise meet in every other round only.  (Counting the batches over the whole row, so that all four take part,
// costs the other formats 2 % of the launch: the compiler then forms every batch's address anew.)
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
    const int batches = (a_cols + batch_cols - 1) / batch_cols, held = PF_PLAIN_CHUNK / batch_cols;
    const int stride = held >= 4 || parts < held ? parts : held;   // (at most four waves share a row)
    const bool takes = active && part < stride;
    if (takes && part < batches) request(part);   // on its way while the first columns are staged
    for (int c0 = 0; c0 < a_cols; c0 += PF_PLAIN_CHUNK) {
        const int cols = a_cols - c0 < PF_PLAIN_CHUNK ? a_cols - c0 : PF_PLAIN_CHUNK;
        stage(c0, cols);
        if (!takes) continue;
        for (int k0 = batch_cols * part; k0 < cols; k0 += batch_cols * stride) {
            take();
            const int after = (c0 + k0) / batch_cols + stride;
            if (after < batches) request(after);
            multiply(k0, cols);
        }
    }
}
