// pkv_attention_grouped.hip -- the decode kernels that run one wave per run by
// default, in their grouped form: kGroup waves share a run's tiles and combine
// in LDS (attn_kernel, pkv_attn_kernel.h).
#include "pkv_attn_kernel.h"

namespace pkv {

AttnKernel select_grouped(const Geo &g, int rows, bool append) {
  if (append) {
    if (rows <= 4) return select_shape<1, 4, true, true>(g);
    if (rows <= 8) return select_shape<1, 2, true, true>(g);
    return nullptr;
  }
  if (rows <= 4) return select_shape<1, 4, false, true>(g);
  if (rows <= 8) return select_shape<1, 2, false, true>(g);
  if (rows <= 16) return select_shape<1, 1, false, true>(g);
  return nullptr;
}

}  // namespace pkv
