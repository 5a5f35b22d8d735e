// Limits of the on-chip solver (kernels_chip.hip) and the geometry of its blocks, host and
// device: which tiles a block keeps, and where the neighbours of a tile's cells are.
#pragma once

#include "tiling.h"

#include <algorithm>
#include <cstddef>
#include <vector>

namespace reef {

constexpr int CHIP_NT = 512;                 // threads per block: two 256-thread groups
constexpr int CHIP_BLOCKS = 256;             // blocks of a tank, at most
constexpr int CHIP_TANKS = 64;               // tanks per launch
constexpr int CHIP_TILES = 8192;             // tile slots of all blocks of a launch, at most
constexpr int CHIP_DIRECT = 64;              // blocks up to which 64 accumulators are added in one hop
constexpr int CHIP_COPIES = 16;              // places the wave sums of a total are published in
constexpr int CHIP_COPY_WORDS = 32;          // 4 waves x 3 sums x 2 words, own cache lines
// per tank two buffers of 256 accumulators x 3 sums x 2 words and the copies
constexpr int CHIP_ACC_HALF = 3 * 256 * 2 + CHIP_COPIES * CHIP_COPY_WORDS;
constexpr int CHIP_ACC_WORDS = 2 * CHIP_ACC_HALF;
constexpr int CHIP_LDS_MAX = 152 * 1024;     // dynamic LDS of a block (160 KB less the static arrays)
constexpr int CHIP_CTL = 4096;               // commit words, used in turn
// exchanges of a launch are numbered from its epoch; an iteration makes at most five
constexpr int CHIP_CAP = 1024;               // iterations per launch
constexpr unsigned CHIP_EPOCHS = 5 * CHIP_CAP + 8;

// Tile slots per group (ct: 2 or 4; with 8 the FP32 kernel spills and takes 1.2 to 1.9 times
// as long per iteration, more than it gains in tiles) and the halo cells a thread may keep
// (sl): both set the registers of a thread, see the kernel's variants.  A 2-D tile has a halo
// of 136 cells, a 3-D tile of up to 648.
constexpr int CHIP_CT_MAX = 4;
constexpr int chip_sl(int d3, int ct) { return d3 ? (ct == 2 ? 6 : 8) : (ct == 2 ? 2 : 3); }
// dynamic LDS: operand of the own cells, a zero and the halo (8 bytes each, the FP64 residual
// of the mixed solve uses it too), r, p, v of the halo (vsize bytes each) and its exchange index
constexpr size_t chip_lds_bytes(int ct, int vsize, int hmax)
{
    return (size_t)(2 * ct * 256 + 1 + hmax) * 8 + (size_t)hmax * (3 * vsize + 4);
}
// halo cells of a block, at most
constexpr int chip_halo_max(int d3, int ct, int vsize)
{
    const int lds = (int)((CHIP_LDS_MAX - chip_lds_bytes(ct, vsize, 0)) / (8 + 3 * vsize + 4));
    return lds < chip_sl(d3, ct) * CHIP_NT ? lds : chip_sl(d3, ct) * CHIP_NT;
}

// ---- geometry of a block, host and device.  Block b of nb keeps the items b, b + nb, ...; its
// tile slot sl = group * ct + c holds tile c % cpt of its local item (c / cpt) * 2 + group.
// Faces of a tile: 0 +x, 1 -x, 2 +y, 3 -y, 4 +z, 5 -z; a cell of a tile is its thread number.
REEF_HD int chip_items(const TileShape& s, int nb, int b) { return (s.nitems - b + nb - 1) / nb; }

// the tile in a slot, -1 empty
REEF_HD int chip_slot_tile(const TileShape& s, int ct, int nb, int b, int sl)
{
    const int c = sl % ct, gr = sl / ct, kk = c / s.cpt, li = kk * 2 + gr;
    if(kk >= ct / s.cpt || li >= chip_items(s, nb, b)) return -1;
    const int t = (b + li * nb) * s.cpt + (c - kk * s.cpt);
    return t < s.ntiles ? t : -1;
}

// the slot of a tile in block b, -1 when another block has it
REEF_HD int chip_tile_slot(const TileShape& s, int ct, int nb, int b, int t)
{
    const int it = t / s.cpt;
    if(it % nb != b) return -1;
    const int li = it / nb;
    return (li % 2) * ct + (li / 2) * s.cpt + (t - it * s.cpt);
}

// the tile across face f of tile t, -1 at the tank's boundary
REEF_HD int chip_face_tile(const TileShape& s, int t, int f)
{
    const int col = t / s.nbz, bz = t - col * s.nbz, by = col / s.nbx, bx = col - by * s.nbx;
    switch(f)
    {
        case 0: return bx + 1 < s.nbx ? t + s.nbz : -1;
        case 1: return bx > 0 ? t - s.nbz : -1;
        case 2: return by + 1 < s.nby ? t + s.nbx * s.nbz : -1;
        case 3: return by > 0 ? t - s.nbx * s.nbz : -1;
        case 4: return bz + 1 < s.nbz ? t + 1 : -1;
        default: return bz > 0 ? t - 1 : -1;
    }
}

// cells of a face, the number of a cell (tile row `row`, lane) among them, and the cell of the
// neighbour tile across it
REEF_HD int chip_face_size(const TileShape& s, int f) { return f < 2 ? 4 : 64 * (f < 4 ? s.tz : s.ty); }
REEF_HD bool chip_on_face(const TileShape& s, int f, int row, int lane)
{
    const int ry = row >> s.tzl, rz = row & (s.tz - 1);
    switch(f)
    {
        case 0: return lane == 63;
        case 1: return lane == 0;
        case 2: return ry == s.ty - 1;
        case 3: return ry == 0;
        case 4: return rz == s.tz - 1;
        default: return rz == 0;
    }
}
REEF_HD int chip_face_pos(const TileShape& s, int f, int row, int lane)
{
    return f < 2 ? row : (f < 4 ? (row & (s.tz - 1)) : (row >> s.tzl)) * 64 + lane;
}
REEF_HD int chip_face_far(const TileShape& s, int f, int q)
{
    const int ql = q & 63, qr = q >> 6;
    switch(f)
    {
        case 0: return q * 64;
        case 1: return q * 64 + 63;
        case 2: return qr * 64 + ql;
        case 3: return ((s.ty - 1) * s.tz + qr) * 64 + ql;
        case 4: return qr * s.tz * 64 + ql;
        default: return (qr * s.tz + s.tz - 1) * 64 + ql;
    }
}
// thread distance of the neighbour inside the tile
REEF_HD int chip_face_step(const TileShape& s, int f)
{
    return f == 0 ? 1 : f == 1 ? -1 : f == 2 ? s.tz * 64 : f == 3 ? -s.tz * 64 : f == 4 ? 64 : -64;
}

// the most halo cells any of nb blocks keeps (nb a power of two)
inline int chip_halo(const TileShape& s, int nb)
{
    std::vector<int> h(nb, 0);
    for(int t = 0; t < s.ntiles; ++t)
    {
        const int b = (t / s.cpt) % nb;
        for(int f = 0; f < 6; ++f)
        {
            const int nt = chip_face_tile(s, t, f);
            if(nt >= 0 && (nt / s.cpt) % nb != b) h[b] += chip_face_size(s, f);
        }
    }
    return *std::max_element(h.begin(), h.end());
}

// Tile slots per group of the kernel variant for at most per_block tiles per block.
inline int chip_ct(int per_block) { return std::max(2, per_block / 2); }

// Blocks of a tank with at most per_block tiles each: the smallest power of two, at most 256,
// the CUs of the card (the blocks of a tank wait for each other and need one each) and the
// tank's items; 0 when the tank does not fit or its sums are taken in another order (a 2-D tank
// with cpt > 1 walks its rows in the streaming v and t phases).  halo[q]: chip_halo of 2^q
// blocks where it is known, else -1.
inline int chip_blocks(const TileShape& s, int d3, int vsize, int per_block, int cus, int* halo)
{
    const int ct = chip_ct(per_block), limit = std::min(std::min(CHIP_BLOCKS, cus), s.nitems);
    if(s.cpt > ct || (d3 == 0 && s.cpt > 1) || s.ntiles > CHIP_BLOCKS * per_block) return 0;
    const int most = std::max(1, std::min(2 * (ct / s.cpt), per_block / s.cpt));   // items per block
    const int hmax = chip_halo_max(d3, ct, vsize);
    for(int q = 0, nb = 1; nb <= limit; ++q, nb *= 2)
    {
        if((s.nitems + nb - 1) / nb > most) continue;
        if(halo[q] < 0) halo[q] = chip_halo(s, nb);
        if(halo[q] <= hmax) return nb;
    }
    return 0;
}

}  // namespace reef
