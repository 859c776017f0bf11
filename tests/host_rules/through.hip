// Which batches are stored through the L2 (store_granule, mrb_rows.h), on the host: fields' row sizes, bytes of the batch, workgroups to a row, and
// an offset of the caller's matrices. Prints a digit for each: a sample and a gather by workgroups or waves, and a gather and a sample whose granules are
// numbered over all rows.
#include <stdio.h>
#include <stdlib.h>

#include "mrb_rows.h"

using namespace mrb;

int main(int argc, char** argv) {
    const uint64_t bytes = strtoull(argv[1], nullptr, 0), offset = strtoull(argv[3], nullptr, 0);
    const uint32_t split = (uint32_t)atoi(argv[2]);
    IoTable t{};
    WidePlan plan{};
    bool whole = true;
    for (int i = 4; i < argc; ++i) {
        const uint32_t rb = (uint32_t)atoi(argv[i]), units = (rb + 15) / 16;
        const int f = t.nfields++;
        t.io[f] = (uint8_t*)((uint64_t)(f + 1) << 32 | offset);
        t.row_bytes[f] = rb;
        t.vec_log2[f] = 4;
        t.units[f] = units;
        plan.f[f].dst = t.io[f];
        plan.f[f].rb = rb;
        plan.wide_items += units;
        plan.nwide += 1;
        whole = whole && whole_pieces(t, f);
    }
    plan.split = (int)split;
    plan.share = (plan.wide_items + split - 1) / split;
    const bool pieces = whole_pieces(plan);
    printf("%d%d%d%d\n", stores_through(bytes, kThroughSample, pieces), stores_through(bytes, kThroughGather, pieces),
           stores_through(bytes, kThroughGather, whole), stores_through(bytes, kThroughSample, whole));
    return 0;
}
