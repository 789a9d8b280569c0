// Walks every row of cells of every tile of the one-launch time loop, as the
// plan of a grid lays them out, and looks where the material loads go (no GPU).
// Prints the number of plans, of loads outside the padded grid, and of rows
// whose own cell would have been outside it.
#include <cstdio>

#include "ifos_resident.h"

using namespace ifos;

int main()
{
    long plans = 0, outside = 0, unguarded = 0;
    for (int N : {1, 2, 4, 6})
        for (int L : {0, 1, 2, 3})
            for (int NX : {64, 65, 200, 511, 960, 1024, 1700})
                for (int NY : {17, 40, 101, 350, 513, 600, 767, 1025, 1224, 1537})
                    for (int prec : {0, 1}) {
                        StepGeom g{};
                        g.NX = NX; g.NY = NY; g.N = N; g.FREE_SURF = 1;
                        // the engine's padding: interior column 1 at float 16, N + 1 columns and rows around
                        const int H = N + 1, rows = NY + 2 * H + 1;
                        g.pitch = (16 + NX + H + 63) / 64 * 64;
                        const long off = (long)H * g.pitch + 15, field = (long)g.pitch * rows;
                        const ResidentPlan p = resident_plan(g, L, 1, prec, 256, 163840);
                        if (!p.rows) continue;
                        plans++;
                        for (int by = 0; by < p.tiles_y; by++)
                            for (int ty = 0; ty < p.ty; ty++)
                                for (int bx = 0; bx <= (NX - 1) / kTileX; bx++)
                                    for (int tx : {0, kTileX - 1})
                                        for (int r = 0; r < p.rows; r++) {
                                            const int i = bx * kTileX + tx + 1, j = by * p.th + ty * p.rows + 1;
                                            const unsigned c = (unsigned)(j * g.pitch + i);
                                            const bool live = i <= NX && j + r <= NY;
                                            outside += off + (long)material_cell(c, r, g.pitch, live) >= field;
                                            unguarded += off + (long)c + (long)r * g.pitch >= field;
                                        }
                    }
    printf("%ld %ld %ld\n", plans, outside, unguarded);
    return 0;
}
