// Host-only: the passes' shortest contiguous run (low consecutive tile bits) of a plan and the vectors that
// it streams non-temporally.  Input file: int32 {n, ibond, colbits, tile_bits, dtype}, ipair[2*ibond],
// ibond_type[ibond], xlocal_Ham (9*16 complex128), llocal_Ham (9*16 int32).  Prints "run nt".
#include <algorithm>
#include <cstdio>
#include <vector>

#include "../../pned_amd/csrc/internal.h"

int main(int argc, char **argv)
{
    FILE *f = argc == 2 ? fopen(argv[1], "rb") : nullptr;
    int h[5];
    if (!f || fread(h, 4, 5, f) != 5) return 2;
    std::vector<int32_t> ip(2 * h[1]), bt(h[1]), ll(144);
    std::vector<double> xl(288);
    if (fread(ip.data(), 4, ip.size(), f) != ip.size() || fread(bt.data(), 4, bt.size(), f) != bt.size() ||
        fread(xl.data(), 8, 288, f) != 288 || fread(ll.data(), 4, 144, f) != 144)
        return 2;
    fclose(f);
    pned::S12Plan pl;
    if (pned::s12_decompose(h[0], h[1], ip.data(), bt.data(), xl.data(), ll.data(), pl)) return 1;
    if (pned::s12_make_passes(pl, h[2], h[3], 3)) return 1;
    int run = 31;
    for (const auto &p : pl.passes) {
        int k = 0;
        while (k < (int)p.tb.size() && p.tb[k] == k) ++k;
        run = std::min(run, k);
    }
    printf("%d %d\n", run, pned::s12_nt_streams(pl, h[4], (size_t)(h[4] ? 8 : 16) << (h[0] + h[2])));
    return 0;
}
