// The lane words that kf_graph makes (pixel.hpp: luma_sum, luma_quotient,
// luma_whole, lane_fields), on the host, for every colour and several fourth
// bytes: the fields of the oracle's packed word.  The rows that take luma() for
// one pixel take it for all, so luma() equals the quotient wherever the colour
// is not one of the multiples.  (Their comparison, lane_similar, is in
// colour_check.cpp.)
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include "depixel_oracle.h"
#include "pixel.hpp"

using namespace dpx;

int main()
{
    long long bad = 0, whole = 0;
    const uint32_t fourth[] = { 0x00, 0xFF, 0x5A, 0x81 };
    for (uint32_t c = 0; c < (1u << 24); c++) {
        const uint32_t want = yuv_lanes(orc_rgb_to_yuv(c));
        for (uint32_t b3 : fourth) {
            const uint32_t w = c | b3 << 24, n = luma_sum(w);
            const uint32_t exact = (uint32_t)luma((int)(c & 0xFFu), (int)((c >> 8) & 0xFFu), (int)(c >> 16));
            const bool is_whole = luma_whole(n);
            const uint32_t y = is_whole ? exact : luma_quotient(n);
            whole += is_whole;
            if (lane_fields(w, y) != want || (!is_whole && y != exact)) {
                if (bad++ < 5) printf("colour %06x: lanes %08x, oracle's %08x\n", c, lane_fields(w, y), want);
            }
        }
    }
    printf("%lld multiples, mismatches %lld\n", whole / 4, bad);
    return bad != 0;
}
