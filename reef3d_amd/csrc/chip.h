// Host view of the on-chip solver (kernels_chip.hip): the tanks one launch covers.
#pragma once

#include "batch.h"
#include "chip_geom.h"

namespace reef {

enum ChipKind { CHIP_FP64 = 0, CHIP_MIXED = 1, CHIP_MAT = 2 };

struct ChipSet
{
    const TankDev* tanks;
    unsigned long long* halo;      // three buffers of halo_words: 256 cells x 2 words per tile slot
    size_t halo_words;
    unsigned long long* acc;       // CHIP_ACC_WORDS per tank of the launch
    unsigned* ctl;                 // commit word per tank of the launch, 0 before it
    unsigned epoch;                // tag of the launch's first exchange
    int cap;                       // iterations at most
    int hmax;                      // largest halo of a block
    int d3, ct;                    // 3-D tanks; tile slots per group
    int n;
    int slot[CHIP_TANKS];
    int blk0[CHIP_TANKS + 1];      // first block of each tank
    int tile0[CHIP_TANKS];         // first exchange tile of each tank
};

// dynamic LDS limit of the kernels; 0 or a REEF_E status
int chip_prepare();
void bl_chip_solve(const ChipSet& S, int kind, int x, int rhs, hipStream_t s);

}  // namespace reef
