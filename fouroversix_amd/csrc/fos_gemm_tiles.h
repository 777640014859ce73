// Which output tile a workgroup of the GEMM kernels gets, and what a number of tiles costs.
#pragma once

#include <stdint.h>

#include "fos_device.h"

namespace fos {

// Output tile of workgroup `bid`: workgroups with equal bid % 8 share an XCD; give each
// XCD a contiguous run of tiles, ordered in column bands of 8 tile rows.
FOS_DEVICE void tile_of(int bid, int tiles_m, int tiles_n, int &tm, int &tn) {
    const int per_xcd = tiles_m * tiles_n / 8;
    const int t = bid < 8 * per_xcd ? (bid & 7) * per_xcd + (bid >> 3) : bid;  // (the remainder in plain order)
    constexpr int kBand = 8;
    const int band = t / (kBand * tiles_n), in_band = t - band * kBand * tiles_n;
    const int rows = (tiles_m - band * kBand) < kBand ? (tiles_m - band * kBand) : kBand;
    tm = band * kBand + in_band % rows;
    tn = in_band / rows;
}

// Time of `tiles` output tiles: whole generations (as many tiles as run at a time) at `generation` each, then the
// last, partial one, whose time depends on how full the chip is (fewer compute units clock higher): `tail`, by
// eighths of a generation.
inline float tiles_cost(int64_t tiles, int64_t per_generation, float generation, const float (&tail)[8]) {
    const int64_t whole = tiles / per_generation, rest = tiles % per_generation;
    if (rest == 0) return whole == 1 ? tail[7] : (float)whole * generation;
    return (float)whole * generation + tail[(rest * 8 - 1) / per_generation];
}

}  // namespace fos
