// Which output tile, K slice and batch entry a workgroup of the matrix-core kernels takes.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mb {

// Grid (tiles, K slices, batch entries).  The hardware hands consecutive workgroups to the 8 XCDs
// in turn and each XCD has its own L2, so the workgroup index is remapped to give every XCD a
// contiguous run: of (batch entry, tile) indices where `batched` asks for it, so that the tiles of a
// batch entry, which read the same operands, share an L2, else of the tiles of each entry and slice.
// Remapping each batch entry's tiles by themselves spread every entry over all 8 XCDs, which
// read its operands 8 times from the Infinity Cache (MI355X, bf16 bmm, us: 32 x 1024 x 128 x 1024
// 25.1 -> 18.8, 32 x 512^3 21.3 -> 15.1, 16 x 1024^3 38.9 -> 34.5, 32 x 1024 x 1024 x 128 30.0 ->
// 26.0), from 16 MiB of operands on (GemmArgs::xcd_batch); smaller ones, whose every entry is in
// every L2 soon, start faster spread out (8 x 512 x 512 x 256 6.5 -> 7.2, 16 x 320 x 320 x 64 5.3 ->
// 5.9), and runs over whole K slices lost (1024 x 1024 x 4096 over 4 slices 23.5 -> 25.2).  Within an
// entry, groups of 2^swz tile rows are walked column by column.  `bz` is the first batch entry
// of the workgroup's batch loop.
__device__ __forceinline__ void work_coords(int tiles_m, int tiles_n, int swz, bool batched, int &tm, int &tn, int &ks,
                                            int &bz) {
    const uint32_t tiles = gridDim.x;
    uint32_t tile = blockIdx.x;
    ks = blockIdx.y;
    bz = blockIdx.z;
    const uint64_t n = batched ? (uint64_t)tiles * gridDim.z : tiles;
    if (n >= 16 && n < (1u << 31)) {
        const uint32_t lin = batched ? tile + tiles * blockIdx.z : tile, base = (uint32_t)n >> 3, rem = (uint32_t)n & 7;
        const uint32_t xcd = lin & 7, w = xcd * base + (xcd < rem ? xcd : rem) + (lin >> 3);
        if (batched && gridDim.z > 1) bz = (int)(tiles == 1 ? w : w / tiles);
        tile = batched ? w - (uint32_t)bz * tiles : w;
    }
    const int G = 1 << swz;
    const int width = G * tiles_n;
    const int grp = (int)tile / width;
    const int first_m = grp * G;
    const int gsz = min(tiles_m - first_m, G);
    const int in = (int)tile - grp * width;
    tm = first_m + in % gsz;
    tn = in / gsz;
}

}  // namespace mb
