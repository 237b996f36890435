// The closed loop (recon.h) in 256-thread workgroups, two per compute unit: the persistent schedule of batches, and the
// schedule of one launch per wavefront step; and the launches of both instances.
#define AV1M_RC_THREADS 256
#define AV1M_RC_SPACE rc_narrow
#include <algorithm>
#include "recon.h"

namespace av1m {
using namespace rc_narrow;

struct RcStepArgs {
    Batch B;
    SearchParams P;
    const uint32_t *sbList;
};
// one launch per wavefront step: workgroup b takes superblock sbList[b]
template <typename Px>
AV1M_RC_KERNEL k_recon(RcStepArgs) {
    extern __shared__ __align__(16) char smraw[];
    lds<RcShared> &S = *(lds<RcShared> *)(lds<char> *)smraw;
    const RcStepArgs &A = kernel_args<RcStepArgs>();
    const Batch &B = A.B;
    const uint32_t sb = A.sbList[blockIdx.x];
    stage_tables(S, *B.T, A.P, B.img[B.sbImg[sb]].qctx, true);
    __syncthreads();
    recon_part<Px, 0>(S, B, sb, nullptr);
    __syncthreads();
    if (!S.img.mono) recon_part<Px, 1>(S, B, sb, nullptr);
}

// the 512-thread instance (k_recon_wide.hip)
size_t recon_wide_smem();
const void *recon_wide_kernel(int bd);

static const void *queue_kernel(int bd, int wpe) {
    return wpe == 1 ? recon_wide_kernel(bd) : bd == 10 ? (const void *)k_recon_queue<uint16_t> : (const void *)k_recon_queue<uint8_t>;
}
static size_t queue_smem(int wpe) { return wpe == 1 ? recon_wide_smem() : sizeof(RcShared); }
static int queue_threads(int wpe) { return wpe == 1 ? 512 : RC_NT; }
size_t recon_smem_bytes() { return std::max(recon_wide_smem(), sizeof(RcShared)); }

int recon_prepare(int bd) {
    const void *step = bd == 10 ? (const void *)k_recon<uint16_t> : (const void *)k_recon<uint8_t>;
    if (hipFuncSetAttribute(step, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(RcShared)) != hipSuccess) return -1;
    for (int wpe = 1; wpe <= 2; wpe++)
        if (hipFuncSetAttribute(queue_kernel(bd, wpe), hipFuncAttributeMaxDynamicSharedMemorySize, (int)queue_smem(wpe)) != hipSuccess) return -1;
    return 0;
}

void launch_recon(const Batch &B, const SearchParams &P, const uint32_t *dSbList, uint32_t n, int bd, hipStream_t st) {
    if (!n) return;
    const RcStepArgs a{B, P, dSbList};
    if (bd == 10) hipLaunchKernelGGL(k_recon<uint16_t>, dim3(n), dim3(RC_NT), sizeof(RcShared), st, a);
    else hipLaunchKernelGGL(k_recon<uint8_t>, dim3(n), dim3(RC_NT), sizeof(RcShared), st, a);
}

// resident workgroups of the persistent kernel per compute unit
int recon_queue_slots(int bd, int wpe) {
    int n = 0;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, queue_kernel(bd, wpe), queue_threads(wpe), queue_smem(wpe)) == hipSuccess ? n : 0;
}

void launch_recon_queue(const Batch &B, const SearchParams &P, const RcQueue &Q, uint32_t blocks, int bd, int wpe, hipStream_t st) {
    if (!Q.n || !blocks) return;
    RcQueueArgs a{B, P, Q};
    void *args[] = {&a};
    (void)hipLaunchKernel(queue_kernel(bd, wpe), dim3(blocks), dim3(queue_threads(wpe)), args, queue_smem(wpe), st);
}

}  // namespace av1m
