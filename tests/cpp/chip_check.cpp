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
            printf("FAIL %s: n %d %d %d ty %d tz %d cpt %d ct %d nb %d b %d\n", #c, nx, ny, nz, ty, tz, cpt, ct, nb, b); \
            return 1;                                                                                   \
        }                                                                                               \
    } while(0)

static int check(int nx, int ny, int nz, int ty, int tz, int cpt, int ct)
{
    if(cpt > ct) return 0;
    const TileShape s = make_shape(nx, ny, nz, ty, tz, cpt);
    const int NTH = 256, most = 2 * (ct / cpt);
    int used = 0;
    {
        // item_spread deals every item once
        int nb = 0, b = 0;
        std::vector<int> dealt(s.nitems, 0);
        for(int l = 0; l < s.nitems; ++l)
        {
            const int it = item_spread(s, l);
            CHECK(it >= 0 && it < s.nitems && !dealt[it]++);
        }
    }
    for(int nb = 1; nb <= 256 && nb <= s.nitems; nb *= 2)
    {
        int b = 0;
        if((s.nitems + nb - 1) / nb > most) continue;
        const int hm = chip_halo(s, nb);
        if(hm > chip_halo_max(ny > 1, ct, 4)) continue;
        ++used;
        std::vector<int> seen(s.ntiles, 0);
        for(b = 0; b < nb; ++b)
        {
            int off[2 * ct][6], o = 0;
            CHECK(chip_items(s, nb, b) >= 1 && chip_items(s, nb, b) <= most);
            for(int sl = 0; sl < 2 * ct; ++sl)
            {
                const int t = chip_slot_tile(s, ct, nb, b, sl);
                if(t >= 0)
                {
                    ++seen[t];
                    CHECK(t < s.ntiles && chip_tile_slot(s, ct, nb, b, t) == sl);
                }
                for(int f = 0; f < 6; ++f)
                {
                    off[sl][f] = o;
                    const int nt = t >= 0 ? chip_face_tile(s, t, f) : -1;
                    if(nt >= 0 && chip_tile_slot(s, ct, nb, b, nt) < 0) o += chip_face_size(s, f);
                }
            }
            CHECK(o <= hm);
            // where each cell of the halo comes from
            std::vector<int> src(o > 0 ? o : 1, -1);
            for(int sl = 0; sl < 2 * ct; ++sl)
                for(int f = 0; f < 6; ++f)
                {
                    const int t = chip_slot_tile(s, ct, nb, b, sl), nt = t >= 0 ? chip_face_tile(s, t, f) : -1;
                    if(nt < 0 || chip_tile_slot(s, ct, nb, b, nt) >= 0) continue;
                    for(int q = 0; q < chip_face_size(s, f); ++q)
                    {
                        const int far = chip_face_far(s, f, q);
                        CHECK(far >= 0 && far < NTH && off[sl][f] + q < o && src[off[sl][f] + q] == -1);
                        src[off[sl][f] + q] = nt * NTH + far;
                    }
                }
            for(int sl = 0; sl < 2 * ct; ++sl)
                for(int th = 0; th < NTH; ++th)
                {
                    const int t = chip_slot_tile(s, ct, nb, b, sl);
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
                            const int ns = chip_tile_slot(s, ct, nb, b, nt);
                            CHECK(ns < 2 * ct);
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
    printf("%d %d %d ty %d tz %d cpt %d ct %d: %d block counts\n", nx, ny, nz, ty, tz, cpt, ct, used);
    return 0;
}

int main()
{
    const int sizes[][3] = {{1, 1, 1}, {63, 1, 5}, {64, 1, 4}, {65, 1, 9}, {256, 1, 64}, {1150, 1, 157}, {2048, 1, 256},
                            {16, 6, 12}, {40, 8, 24}, {96, 24, 48}, {130, 33, 37}, {64, 5, 33}, {200, 17, 40}, {224, 40, 96}};
    for(const auto& n : sizes)
        for(int ct = 2; ct <= CHIP_CT_MAX; ct *= 2)
        {
            if(n[1] == 1 && check(n[0], 1, n[2], 1, 4, 1, ct)) return 1;
            if(n[1] == 1) continue;
            for(int cpt = 1; cpt <= 4; ++cpt)
                if(check(n[0], n[1], n[2], 4, 1, cpt, ct) || check(n[0], n[1], n[2], 2, 2, cpt, ct) ||
                   check(n[0], n[1], n[2], 1, 4, cpt, ct))
                    return 1;
        }
    // no tank gets more blocks than the card has CUs; a whole card takes 2048 tiles
    for(const auto& n : sizes)
        for(int per = 2; per <= 2 * CHIP_CT_MAX; per *= 2)
            for(int cus : {0, 1, 32, 38, 64, 128, 256, 304})
            {
                const int d3 = n[1] > 1;
                const TileShape s = d3 ? make_shape(n[0], n[1], n[2], 4, 1, 1) : make_shape(n[0], 1, n[2], 1, 4, 1);
                int halo[9];
                std::fill(halo, halo + 9, -1);
                const int nb = chip_blocks(s, d3, 4, per, cus, halo);
                if(nb > cus || nb > CHIP_BLOCKS || (nb & (nb - 1)) || (nb && s.nitems > nb * per) ||
                   (!nb && cus >= 256 && !d3 && s.ntiles <= CHIP_BLOCKS * per))
                    return printf("%d %d %d: %d blocks of %d tiles on %d CUs\n", n[0], n[1], n[2], nb, per, cus), 1;
            }
    for(int vsize = 4; vsize <= 8; vsize += 4)
        for(int d3 = 0; d3 < 2; ++d3)
            for(int ct = 2; ct <= CHIP_CT_MAX; ct *= 2)
            {
                const int h = chip_halo_max(d3, ct, vsize);
                if(h > chip_sl(d3, ct) * CHIP_NT || chip_lds_bytes(ct, vsize, h) > (size_t)CHIP_LDS_MAX) return 1;
                if(!d3 && h < 2 * ct * 136) return printf("2-D halo of %d slots does not fit\n", ct), 1;
                if(2 * ct * 256 + 1 + h >= 65536) return 1;   // operand indices are 16 bits
            }
    printf("ok\n");
    return 0;
}
