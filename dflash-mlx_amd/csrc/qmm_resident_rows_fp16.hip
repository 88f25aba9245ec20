#include "qmm_resident.h"

dflash::resident::Kernel dflash::resident::fp16_rows_kernel(int row_tiles, int group_size, int chunks, bool silu) {
  return rows_kernel<true>(row_tiles, group_size, chunks, silu);
}
