#include "qmm_resident.h"

dflash::resident::Kernel dflash::resident::fp16_kernel(int group_size, int chunks, bool silu, bool packed) {
  return few_kernel<true>(group_size, chunks, silu, packed);
}
