// Host check of the quantizer's division by a step with the step's reciprocal at hand (quot_step, av1m_common.h) against
// the IEEE division: every quantizer step of both bit depths, magnitudes over 2^-10 .. 2^24, and products of a step with
// the dead zone's and the rounding's thresholds moved by up to 4 units in the last place.
#include <cstdio>
#include <cstring>
#include "../../av1gpu_amd/csrc/av1m_common.h"

static uint64_t s = 88172645463325252ull;
static uint64_t rnd() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s; }

int main() {
    long n = 0;
    for (int b = 0; b < 2; b++)
        for (int dc = 0; dc < 2; dc++)
            for (int q = 0; q < 256; q++) {
                const float d = dc ? av1t::Dc_Qlookup[b][q] : av1t::Ac_Qlookup[b][q], y = 1.f / d;
                for (int k = 0; k < 20000; k++) {
                    const int m = k & 3;
                    float v;
                    if (m == 0) v = (float)((double)(rnd() >> 11) / 9007199254740992.0 * pow(2.0, (int)(rnd() % 34) - 10));
                    else {
                        v = (float)((double)(rnd() % 400000) / 8.0 + (m == 1 ? 0.656 : m == 2 ? 0.625 : 0.0)) * d;
                        uint32_t u;
                        memcpy(&u, &v, 4);
                        u += (uint32_t)(rnd() % 9) - 4;
                        memcpy(&v, &u, 4);
                        if (!(v >= 0)) v = 0;
                    }
                    const float e = v / d, g = av1m::quot_step(v, d, y);
                    n++;
                    if (memcmp(&e, &g, 4)) { printf("%a / %a: %a, quot_step %a\n", v, d, e, g); return 1; }
                }
            }
    printf("ok %ld\n", n);
    return 0;
}
