// fp16 instantiation of the backward in one launch.
#include "attn_bwd_both_impl.h"

namespace slapo {
int attn_bwd_both_mfma_f16(const AttnArgs& a, hipStream_t st) {
    return bwd_both::dispatch<f16_t>(a, st);
}
}  // namespace slapo
