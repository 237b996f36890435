// The closed loop (recon.h) in 512-thread workgroups, one per compute unit: the persistent schedule of single images and
// small batches.
#define AV1M_RC_THREADS 512
#define AV1M_RC_SPACE rc_wide
#include "recon.h"

namespace av1m {

size_t recon_wide_smem() { return sizeof(rc_wide::RcShared); }
const void *recon_wide_kernel(int bd) {
    return bd == 10 ? (const void *)rc_wide::k_recon_queue<uint16_t> : (const void *)rc_wide::k_recon_queue<uint8_t>;
}

}  // namespace av1m
