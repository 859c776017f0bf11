// Which batches are stored through the L2 (store_granule, mrb_rows.h), on the host: by their bytes. Prints a digit for a sample and one for a gather.
#include <stdio.h>
#include <stdlib.h>

#include "mrb_rows.h"

int main(int, char** argv) {
    const uint64_t bytes = strtoull(argv[1], nullptr, 0);
    printf("%d%d\n", mrb::stores_through(bytes, mrb::kThroughSample), mrb::stores_through(bytes, mrb::kThroughGather));
    return 0;
}
