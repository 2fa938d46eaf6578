// Tiles of pgemm4.hip's kernel (pgemm4_kernel.h), in a unit of their own for the build's sake.
#include "pgemm4_kernel.h"

namespace k8sllm {

int p4_tiles(const P4Args& a, int cfg, int epi, int norm, hipStream_t s) {
  return p4_cfg<P4_TILES, P4_WIDE>(a, cfg, epi, norm, s);
}
int p4_tiles_act(const P4Args& a, int cfg, int kind, bool grouped, hipStream_t s) {
  return grouped ? p4_act_cfg<true, P4_TILES, P4_WIDE>(a, cfg, kind, s) : p4_act_cfg<false, P4_TILES, P4_WIDE>(a, cfg, kind, s);
}

}  // namespace k8sllm
