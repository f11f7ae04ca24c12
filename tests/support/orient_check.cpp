// orient3d_exact_sign of mcut_amd/csrc/geom.hpp on the host.
// Usage: orient_check FILE (12 doubles a test: a, b, c, d); prints a sign a line.
#include <cstdio>

#include "geom.hpp"

int main(int argc, char** argv)
{
    FILE* f = argc > 1 ? fopen(argv[1], "rb") : nullptr;
    if (!f) return 2;
    for (double p[12]; fread(p, sizeof p, 1, f) == 1;) printf("%d\n", mcgpu::orient3d_exact_sign(p, p + 3, p + 6, p + 9));
    fclose(f);
    return 0;
}
