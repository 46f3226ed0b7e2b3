// Which shapes the specialised kernels take, asked of the library's own rules:
//   shapes plane <norder> <npw> <lds limit>    2-D kernels
//   shapes lowp  <norder> <npw> <lds limit>    3-D reduced precision
// prints 1 or 0.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "kernels.h"

int main(int argc, char** argv) {
    if (argc != 5) return 2;
    const bool plane = !std::strcmp(argv[1], "plane");
    fgt::Geom g{};
    fgt::DevTables t{};
    t.n = std::atoi(argv[2]);
    t.npw = g.npw = std::atoi(argv[3]);
    t.lds_limit = std::strtoull(argv[4], nullptr, 10);
    g.ndim = plane ? 2 : 3;
    g.nd = 1;
    g.px = t.npw;
    g.py = plane ? 1 : t.npw;
    g.pz = (t.npw + 1) / 2;
    std::printf("%d\n", plane ? fgt::plane_supported(g, t, 0) : fgt::pw2pot_3d_supported(g, t));
    return 0;
}
