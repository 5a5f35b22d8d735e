// Geometry of the on-chip solver's blocks (csrc/chip_geom.h) against the cells themselves: every
// tile has one slot, every neighbour of a cell is found where the kernel looks for it, every
// index stays inside its buffer.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../reef3d_amd/csrc/chip_geom.h"

using namespace reef;

#define CHECK(c)                                                                                        \
    do                                                                                                  \
    {                                                                                                   \
        if(!(c))                                                                                        \
        {                                                                                               \
            printf("FAIL %s: n %d %d %d ty %d tz %d cpt %d nb %d b %d\n", #c, nx, ny, nz, ty, tz, cpt, nb, b); \
            return 1;                                                                                   \
        }                                                                                               \
    } while(0)

static int check(int nx, int ny, int nz, int ty, int tz, int cpt)
{
    const TileShape s = make_shape(nx, ny, nz, ty, tz, cpt);
    const int NTH = 256, most = 2 * (CHIP_SLOTS / cpt);
    int used = 0;
    for(int nb = 1; nb <= 256 && nb <= s.nitems; nb *= 2)
    {
        int b = 0;
        if((s.nitems + nb - 1) / nb > most) continue;
        const int hm = chip_halo(s, nb);
        if(hm > CHIP_HALO_MAX) continue;
        ++used;
        std::vector<int> seen(s.ntiles, 0);
        for(b = 0; b < nb; ++b)
        {
            int off[2 * CHIP_SLOTS][6], o = 0;
            CHECK(chip_items(s, nb, b) >= 1 && chip_items(s, nb, b) <= most);
            for(int sl = 0; sl < 2 * CHIP_SLOTS; ++sl)
            {
                const int t = chip_slot_tile(s, nb, b, sl);
                if(t >= 0)
                {
                    ++seen[t];
                    CHECK(t < s.ntiles && chip_tile_slot(s, nb, b, t) == sl);
                }
                for(int f = 0; f < 6; ++f)
                {
                    off[sl][f] = o;
                    const int nt = t >= 0 ? chip_face_tile(s, t, f) : -1;
                    if(nt >= 0 && chip_tile_slot(s, nb, b, nt) < 0) o += chip_face_size(s, f);
                }
            }
            CHECK(o <= hm);
            // where each cell of the halo comes from
            std::vector<int> src(o > 0 ? o : 1, -1);
            for(int sl = 0; sl < 2 * CHIP_SLOTS; ++sl)
                for(int f = 0; f < 6; ++f)
                {
                    const int t = chip_slot_tile(s, nb, b, sl), nt = t >= 0 ? chip_face_tile(s, t, f) : -1;
                    if(nt < 0 || chip_tile_slot(s, nb, b, nt) >= 0) continue;
                    for(int q = 0; q < chip_face_size(s, f); ++q)
                    {
                        const int far = chip_face_far(s, f, q);
                        CHECK(far >= 0 && far < NTH && off[sl][f] + q < o && src[off[sl][f] + q] == -1);
                        src[off[sl][f] + q] = nt * NTH + far;
                    }
                }
            for(int sl = 0; sl < 2 * CHIP_SLOTS; ++sl)
                for(int th = 0; th < NTH; ++th)
                {
                    const int t = chip_slot_tile(s, nb, b, sl);
                    int i, j, k;
                    if(t < 0 || !tile_cell_of(s, nx, ny, nz, t, th, i, j, k)) continue;
                    const int want[6][3] = {{i + 1, j, k}, {i - 1, j, k}, {i, j + 1, k}, {i, j - 1, k}, {i, j, k + 1}, {i, j, k - 1}};
                    for(int f = 0; f < 6; ++f)
                    {
                        const int* w = want[f];
                        if(w[0] < 0 || w[0] >= nx || w[1] < 0 || w[1] >= ny || w[2] < 0 || w[2] >= nz) continue;
                        int nt = t, nth;
                        if(!chip_on_face(s, f, th >> 6, th & 63))
                            nth = th + chip_face_step(s, f);
                        else
                        {
                            const int fp = chip_face_pos(s, f, th >> 6, th & 63);
                            nt = chip_face_tile(s, t, f);
                            CHECK(nt >= 0 && fp >= 0 && fp < chip_face_size(s, f));
                            nth = chip_face_far(s, f, fp);
                            const int ns = chip_tile_slot(s, nb, b, nt);
                            CHECK(ns < 2 * CHIP_SLOTS);
                            if(ns < 0) CHECK(src[off[sl][f] + fp] == nt * NTH + nth);
                        }
                        int a, c, d;
                        CHECK(nth >= 0 && nth < NTH && tile_cell_of(s, nx, ny, nz, nt, nth, a, c, d));
                        CHECK(a == w[0] && c == w[1] && d == w[2]);
                    }
                }
        }
        b = -1;
        for(int t = 0; t < s.ntiles; ++t) CHECK(seen[t] == 1);
    }
    printf("%d %d %d ty %d tz %d cpt %d: %d block counts\n", nx, ny, nz, ty, tz, cpt, used);
    return 0;
}

int main()
{
    const int sizes[][3] = {{1, 1, 1}, {63, 1, 5}, {64, 1, 4}, {65, 1, 9}, {256, 1, 64}, {1150, 1, 157}, {2048, 1, 256},
                            {16, 6, 12}, {40, 8, 24}, {96, 24, 48}, {130, 33, 37}, {64, 5, 33}, {200, 17, 40}};
    for(const auto& n : sizes)
    {
        if(n[1] == 1 && check(n[0], 1, n[2], 1, 4, 1)) return 1;
        if(n[1] == 1) continue;
        for(int cpt = 1; cpt <= 4; ++cpt)
            if(check(n[0], n[1], n[2], 4, 1, cpt) || check(n[0], n[1], n[2], 2, 2, cpt) || check(n[0], n[1], n[2], 1, 4, cpt))
                return 1;
    }
    printf("ok\n");
    return 0;
}
