// Every slot of a line's LDS buffers that the sweep kernels touch lies in the
// line's own part of the workgroup's array (host program; Skew and the explicit
// rows' numbering of nuc_lines.h, the accesses of sweep_body and line_half).
#include "nuc_lines.h"

#include <cstdio>

using namespace nucdev;

static int bad = 0;

template <int R, int NL> static void line(const char *what, int slot)
{
    if (slot >= 0 && slot < Skew<R, NL>::pitch(NL * R)) return;
    if (bad++ < 40) std::printf("R %d, %d lanes: %s at slot %d of %d\n", R, NL, what, slot, Skew<R, NL>::pitch(NL * R));
}

template <int R, int NL> static void form()
{
    using Sk = Skew<R, NL>;
    const int cap = NL * R;
    // the write-only dummies of the halo copies (f^+, mirrored f^-, viscous flux)
    line<R, NL>("f+ dummy", Sk::at(cap + HALO));
    line<R, NL>("f- dummy", Sk::mir(cap + HALO));
    if (cap + HALO + HALO >= plain_pitch(cap)) { std::printf("R %d: viscous dummy past the line\n", R); bad++; }
    for (int n = cap; n > cap - NL && n >= 4; n--) {
        // cells and their halo (a segment has n + 1 <= cap interfaces)
        for (int c = -HALO; c < n + HALO; c++) {
            line<R, NL>("f+ cell", Sk::at(c));
            line<R, NL>("f- cell", Sk::mir(c));
        }
        // the cells that the rows past the last interface read, set to zero
        for (int c = n + HALO; c <= cap + 2; c++) {
            line<R, NL>("f+ tail", Sk::at(c));
            line<R, NL>("f- tail", Sk::mir(c));
        }
        for (int m = 0; m <= n && m < cap + 1; m++) {
            line<R, NL>("f+ interface", Sk::at(m));
            line<R, NL>("f- interface", Sk::mir(m));
        }
    }
    // the lanes' windows: up to three points upwind and one more downwind
    for (int h = 0; h < NL; h++)
        for (int rad = 1; rad <= 3; rad++)
            for (int t = 0; t < R + 2 * rad + 1; t++) line<R, NL>("window", h * (R + 1) + Sk::at(t - rad - 1));
    // slots are distinct per position, so no pad slot is a position's
    for (int y = -HALO - 2; y <= cap + HALO; y++)
        if (Sk::at(y) % (R + 1) == R) { std::printf("R %d: position %d on a pad slot\n", R, y); bad++; }
    if constexpr (R > 2)
        for (int k = 0; k < 18; k++) line<R, NL>("explicit row", edge_slot<R, NL>(k));
}

int main()
{
    form<2, 32>(); form<3, 32>(); form<4, 32>(); form<5, 32>();
    form<6, 32>(); form<8, 32>(); form<12, 32>(); form<16, 32>();
    form<5, 64>(); form<6, 64>(); form<8, 64>();
    std::printf("%d slots out of range\n", bad);
    return bad != 0;
}
