// The tiles chosen over a batch, for tests/test_tile_rules.py (host code only).
//
//   tile_rules <nr> <nphi> <adiabatic> [<nr> <nphi> <adiabatic> ...]
// Prints the kick walk's tile of the members in the order given and in the reverse
// order, each member's on its place in the first.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../fargocpt_amd/csrc/fcpt_device.hpp"
#include "../../fargocpt_amd/csrc/fcpt_kernels.hpp"

int main(int argc, char **argv)
{
    std::vector<fcpt::KParams> a;
    for (int k = 1; k + 2 < argc; k += 3) {
        fcpt::KParams P{};
        P.nr = std::atoi(argv[k]);
        P.ns = std::atoi(argv[k + 1]);
        P.adiabatic = std::atoi(argv[k + 2]);
        P.artvisc = FCPT_ARTVISC_SN;
        a.push_back(P);
    }
    std::vector<fcpt::KParams> b(a.rbegin(), a.rend());
    fcpt::resolve_kv_tiles(a);
    fcpt::resolve_kv_tiles(b);
    for (size_t k = 0; k < a.size(); ++k) std::printf("%d %d\n", a[k].kv_tile, b[a.size() - 1 - k].kv_tile);
    return 0;
}
