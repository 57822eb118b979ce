// graph_strips_bound (strips.hpp) against batches of random and extreme item
// shapes: never fewer than the batch's strips.  Prints the batches looked at
// and the largest share of the bound that one took, in thousandths.
#include <stdio.h>

#include <random>
#include <vector>

#include "strips.hpp"
using namespace dpx;

int main()
{
    std::mt19937_64 rng(11);
    auto uni = [&](int64_t a, int64_t b) { return a + (int64_t)(rng() % (uint64_t)(b - a + 1)); };
    auto log_uni = [&](int64_t a, int64_t b) {
        double l = 1.0;
        for (; (double)a * l < (double)b && uni(0, 9); ) l *= 1.9;
        const int64_t top = (int64_t)((double)a * l);
        return uni(a, top > b ? b : top < a ? a : top);
    };
    long batches = 0, most = 0;
    for (int it = 0; it < 60000; it++) {
        const int64_t pixels = log_uni(1, 4 << 20);
        const size_t n = (size_t)log_uni(1, 600);
        const int kind = (int)uni(0, 4);  // shapes at random, tall, wide, two rows of a block over its height, alike
        const int64_t w_all = uni(1, std::min<int64_t>(32768, pixels));
        uint64_t total = 0;
        std::vector<int> W(n), H(n);
        for (size_t k = 0; k < n; k++) {
            const int64_t px = uni(0, 3) ? pixels : uni(1, pixels);
            int64_t w = kind == 0 ? uni(1, std::min<int64_t>(32768, px)) : kind == 1 ? uni(1, std::min<int64_t>(3, px))
                      : kind == 2 ? std::min<int64_t>(32768, px) - (px > 1 ? uni(0, 1) : 0)
                      : kind == 3 ? std::max<int64_t>(1, std::min<int64_t>(32768, px / uni(1, 70))) : std::min(w_all, px);
            const int64_t h = std::min<int64_t>(32768, std::max<int64_t>(1, px / w));
            W[k] = (int)w;
            H[k] = (int)h;
            total += (uint64_t)w * h;
        }
        const int rows = graph_rows(total);
        uint64_t strips = 0;
        for (size_t k = 0; k < n; k++) strips += graph_split(W[k], H[k], rows).strips;
        const size_t bound = graph_strips_bound(n, (size_t)pixels);
        batches++;
        if (strips > bound) {
            printf("%zu items of %lld pixels: %llu strips, bound %zu\n", n, (long long)pixels, (unsigned long long)strips, bound);
            return 1;
        }
        most = std::max(most, (long)(1000 * strips / bound));
    }
    printf("%ld %ld\n", batches, most);
    return 0;
}
