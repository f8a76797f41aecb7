// prefill_attn.hip's host side, for test_launch_rules.py: for every "rows keys heads head_size window" of the input the most key tiles of a range and the ranges
// of the longest query block (0 0: not split), having checked that the ranges of every block are what the kernels take them for. A wrong one
// ends the program, as undefined behaviour does (-fsanitize-trap).
#include "../ferric_amd/csrc/prefill_attn.hip"
#include "launch_rules.hpp"

int main() {
    long long t, s, heads, hd, window;
    while (scanf("%lld %lld %lld %lld %lld", &t, &s, &heads, &hd, &window) == 5) {
        const int win = fhip::causal_window((size_t)window, (size_t)s);
        const fhip::CausalSplit sp = fhip::causal_split((size_t)t, (size_t)s, (size_t)heads, (size_t)hd, win);
        for (int first = 0; first < t; first += 16 * CUT_WAVES) {
            const int last = (int)(first + 16 * CUT_WAVES < t ? first + 16 * CUT_WAVES : t) - 1, off = (int)(s - t);
            const KeyTiles k = key_tiles(off, first, last, win);
            if (k.lo < 0 || k.hi < k.lo || k.hi != (off + last) / 32 || (win > 0 && 32 * k.lo > (off + first - win + 1 > 0 ? off + first - win + 1 : 0))) return 2;
            for (int most = sp.most ? sp.most : 1; most <= (sp.most ? sp.most : k.count() + 1); most += 1 + most / 8) {
                const KeyRanges r = key_ranges(k.count(), most);
                if (r.n < 1 || r.per < 1 || r.per > most || (r.n - 1) * r.per >= k.count() || r.n * r.per < k.count() || (sp.most && r.n > sp.slots)) return 3;
            }
        }
        printf("%d %d\n", sp.most, sp.slots);
    }
}
