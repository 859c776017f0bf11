// Which fields a sample of many rows copies by themselves (large_field, mrb_lds_sample.h), on the host: bytes of a row of the field, strata to a
// workgroup, batches, bytes of the batches and of the rows held. Prints a digit.
#include <stdio.h>
#include <stdlib.h>

#include "mrb_lds_sample.h"

int main(int, char** argv) {
    mrb::IoTable t{};
    t.nfields = 1;
    t.row_bytes[0] = (uint32_t)atoi(argv[1]);
    t.units[0] = (t.row_bytes[0] + 15) / 16;
    t.vec_log2[0] = t.row_bytes[0] >= 16 ? 4 : 0;
    printf("%d\n", mrb::large_field(t, 0, atoi(argv[2]), atoi(argv[3]), strtoull(argv[4], nullptr, 0), strtoull(argv[5], nullptr, 0)));
    return 0;
}
