// Where the loads of the products that go from global memory straight into LDS lie, as plain constexpr functions: the kernels
// address with them, and a host test walks them over whole operands and finds no load outside.
//
// A raw buffer load reads base + lane offset + scalar offset, and its range check compares the LANE offset alone with the
// size in the descriptor.  What decides whether something exists therefore goes into the descriptor or the lane offset, and
// a scalar offset only moves a load inside what the check has let pass.
#pragma once

#include <stdint.h>

namespace fos {

// 1 KiB fragments of 16 rows x 32 k: eight make a step of a band of 128 rows, four steps a chunk of 128 k.
constexpr int kFragmentStep = 8192, kBandChunkBytes = 32768;

// The tiles of gemm_half_kernel, and a wavefront's loads: of A (and, IF4, of B) fragments per step; of B's codes (16 rows
// each) and scales (256 bytes each) per chunk.
template <int WAVES_M, int WAVES_N, int WM, bool IF4>
struct HalfTile {
    static constexpr int NW = WAVES_M * WAVES_N, BM = 16 * WM * WAVES_M, BN = 64 * WAVES_N;
    static constexpr int LA = BM / 16 / NW, LB = BN / 16 / NW, LS = IF4 ? 0 : BN / 32 / NW;
    // every wavefront has descriptors of its own, of the 128 rows its share lies in (codes: of its own rows)
    static_assert(LA * NW * 16 == BM && LB * NW * 16 == BN && 8 % LA == 0 && 8 % LB == 0 && (IF4 || 4 % LS == 0), "no share crosses a multiple of 128 rows");
};

// Size in the descriptor of a share that begins at row `first` of a tile of which `inside` rows exist (a multiple of 128): nothing
// where the share lies beyond (its loads give zeros without touching memory).
constexpr uint32_t share_bytes(int first, int inside, uint32_t bytes) { return first < inside ? bytes : 0u; }

// Fragment f (of 16 rows) of the tile at row0; `band`: bytes of 128 rows.
constexpr int64_t fragment_base(int64_t row0, int f, uint32_t band) { return ((row0 >> 7) + (f >> 3)) * (int64_t)band; }
constexpr uint32_t fragment_lane(int lane) { return (uint32_t)lane * 16; }
constexpr uint32_t fragment_scalar(int f, int step) { return (uint32_t)step * kFragmentStep + (uint32_t)(f & 7) * 1024; }

// K % 128 = 64: of the last chunk only the first half exists.  A lane of the upper half of a wavefront, which holds the k of the other
// half, then gets an offset beyond every descriptor; nobody uses what it receives (its scales are masked).
constexpr uint32_t kNoRead = 0x80000000u;
constexpr bool is_half(int chunk, uint32_t kbytes) { return (uint32_t)chunk * 64 + 64 > kbytes; }
constexpr uint32_t whole_or(bool half, int lane, uint32_t offset) { return half && lane >= 32 ? kNoRead : offset; }

// B's codes, `kbytes` a row: load t of a wavefront's share takes 64 bytes of 16 rows.
constexpr uint32_t codes_lane(int lane, uint32_t kbytes) { return (uint32_t)(lane & 15) * kbytes + (uint32_t)(lane >> 4) * 16; }
constexpr uint32_t codes_scalar(int t, int chunk, uint32_t kbytes) { return (uint32_t)t * 16 * kbytes + (uint32_t)chunk * 64; }

// B's scales, of 128 rows in tiles of 512 bytes per 64 k (`band` bytes): run g of the tile at row0 takes 256 bytes, the first two of
// four those of the first 64 k of a chunk.  (Of half a chunk all four take those.)
constexpr int64_t scales_base(int64_t row0, int g, uint32_t band) { return ((row0 >> 7) + (g >> 2)) * (int64_t)band; }
constexpr uint32_t scales_lane(int lane) { return (uint32_t)lane * 4; }
constexpr uint32_t scales_scalar(int g, int chunk, bool half) { return (uint32_t)chunk * 1024 + (uint32_t)(g & (half ? 1 : 3)) * 256; }

// gemm_half_stream_kernel: a workgroup's 64 rows from n0, loads j of 16 rows each (scalar offsets: 64 bytes of codes and 1024 of scales
// a chunk).  A lane's two scales lie in the word of its row, rows n0 % 128 + 16 j + (lane & 15): two adjacent words of 32-row groups, 256
// bytes apart for the odd j.
constexpr uint32_t stream_codes_lane(int lane, int j, uint32_t kbytes, bool half) {
    return whole_or(half, lane, codes_lane(lane, kbytes)) + (uint32_t)j * 16 * kbytes;
}
constexpr uint32_t stream_scales_lane(int lane, int j, int64_t n0, bool half) {
    return whole_or(half, lane, (uint32_t)(lane >> 5) * 512 + (uint32_t)(lane & 15) * 16 + ((uint32_t)(n0 & 127) >> 5) * 4 + (uint32_t)(lane >> 4 & 1) * 2) +
           (uint32_t)(j & 1) * 256 + (uint32_t)(j >> 1) * 4;
}

// gemm_mxfp4_dma_kernel: steps of 256 codes (128 bytes a row), 8 rows a load.  The lane that fills 16-byte unit c of row rho fetches unit
// c ^ ((rho >> 1) & 7), so every other load (rows 8 ... 15 of 16: `odd`) has the units' upper halves exchanged.  Of a last
// step that K fills by half (K % 256 = 128) the units from 64 bytes on and the second of the two scale tiles don't exist.
constexpr uint32_t mx_unit(int lane, bool odd) { return (uint32_t)(((lane & 7) ^ (lane >> 4)) * 16) ^ (odd ? 64u : 0u); }
constexpr bool mx_is_half(int step, uint32_t kbytes) { return (uint32_t)step * 128 + 128 > kbytes; }
constexpr uint32_t mx_codes_lane(int first_row, int lane, bool odd, uint32_t kbytes) {
    return (uint32_t)(first_row + (lane >> 3)) * kbytes + mx_unit(lane, odd);
}
constexpr uint32_t mx_whole_or(bool half, int lane, bool odd, uint32_t offset) { return half && mx_unit(lane, odd) >= 64 ? kNoRead : offset; }
constexpr int mx_codes_scalar(int t, int step, int kbytes) { return step * 128 + t * 8 * kbytes; }
constexpr uint32_t mx_scales_lane(int lane) { return (uint32_t)lane * 16; }
constexpr int mx_scales_scalar(int step) { return step * 1024; }

}  // namespace fos
