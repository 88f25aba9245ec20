#include "qmm_resident.h"

dflash::resident::Kernel dflash::resident::bf16_kernel(int group_size, int chunks, bool silu, bool packed) {
  return few_kernel<false>(group_size, chunks, silu, packed);
}
