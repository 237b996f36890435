// Host check of pred_4x4 (av1gpu_amd/csrc/av1m_common.h) against pred_px, sample by sample: every mode and angle delta, every
// block size of 4..64 on each side, every 4x4 of the block, random 8- and 10-bit edges without upsampling.  Prints
// "ok <cases>" or the first mismatch and exits 1.
#include <cstdio>
#include <cstdint>
#include "../../av1gpu_amd/csrc/av1m_common.h"

using namespace av1m;

static uint32_t rng = 777;
static int rnd(int n) { rng = rng * 1664525u + 1013904223u; return (int)((rng >> 8) % (uint32_t)n); }

int main() {
    static uint16_t abuf[512], lbuf[512];
    long cases = 0;
    for (int bd = 8; bd <= 10; bd += 2)
        for (int lw = 2; lw <= 6; lw++)
            for (int lh = 2; lh <= 6; lh++) {
                for (int k = 0; k < 512; k++) { abuf[k] = (uint16_t)rnd(1 << bd); lbuf[k] = (uint16_t)rnd(1 << bd); }
                const uint16_t *A = abuf + 64, *L = lbuf + 64;
                const int dcv = rnd(1 << bd);
                for (int mode = 0; mode <= PAETH_PRED; mode++)
                    for (int d = -3; d <= 3; d++) {
                        if (!is_dir(mode) && d) continue;
                        const int pa = pangle(mode, d);
                        for (int y = 0; y < 1 << lh; y += 4)
                            for (int x = 0; x < 1 << lw; x += 4) {
                                int o[16];
                                pred_4x4(mode, pa, dcv, y, x, lw, lh, A, L, o);
                                for (int k = 0; k < 16; k++) {
                                    const int i = y + k / 4, j = x + k % 4;
                                    const int want = mode == DC_PRED ? dcv : pred_px(mode, pa, i, j, lw, lh, A, L, 0, 0);
                                    cases++;
                                    if (o[k] != want) {
                                        printf("mismatch mode %d pa %d %dx%d row %d col %d: %d != %d\n", mode, pa, 1 << lw, 1 << lh, i, j, o[k], want);
                                        return 1;
                                    }
                                }
                            }
                    }
            }
    printf("ok %ld\n", cases);
    return 0;
}
