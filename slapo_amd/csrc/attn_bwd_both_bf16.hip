// bf16 instantiation of the backward in one launch.
#include "attn_bwd_both_impl.h"

namespace slapo {
int attn_bwd_both_mfma_bf16(const AttnArgs& a, hipStream_t st) {
    return bwd_both::dispatch<bf16_t>(a, st);
}
}  // namespace slapo
