#include "qmm_resident.h"

dflash::resident::Kernel dflash::resident::bf16_rows_kernel(int row_tiles, int group_size, int chunks, bool silu) {
  return rows_kernel<false>(row_tiles, group_size, chunks, silu);
}
