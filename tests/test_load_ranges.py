"""Global loads of the product kernels stay inside their operands.

The kernels that load straight into LDS compute their addresses with the functions of fos_load_ranges.h.  A host program
built from that header walks every load of every lane over whole operands, by the rule of raw buffer loads: what the
descriptor's size is compared with is the lane offset alone.
"""

import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fouroversix_amd", "csrc")

COMMON = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include "fos_load_ranges.h"
using namespace fos;
using i64 = int64_t;

// One load of a lane: nothing where the check rejects it, otherwise bytes [at, at + size) of an operand.
static void touch(const char *what, i64 base, uint32_t records, uint32_t lane, uint32_t scalar, int size, i64 operand, i64 expect) {
    if (lane >= records) {
        if (expect >= 0) { printf("%s: byte %lld is not loaded\n", what, (long long)expect); exit(1); }
        return;
    }
    const i64 at = base + (i64)lane + (i64)scalar;
    if (at < 0 || at + size > operand) { printf("%s: bytes %lld .. %lld of %lld\n", what, (long long)at, (long long)at + size, (long long)operand); exit(1); }
    if (expect >= 0 && at != expect) { printf("%s: byte %lld in the place of %lld\n", what, (long long)at, (long long)expect); exit(1); }
}
"""

# what each lane has to receive (`expect`) where the row or column exists, and the operand's size
HALF = r"""
template <class T, bool IF4>
static void walk(int M, int N, int K) {
    const int chunks = (K + 127) / 128;
    const uint32_t band = (uint32_t)chunks * kBandChunkBytes, kbytes = K / 2, scale_band = (uint32_t)K * 8;
    const i64 frags_a = (i64)(M / 128) * band, frags_b = (i64)(N / 128) * band, codes = (i64)N * kbytes, scales = (i64)(N / 128) * scale_band;
    for (int m0 = 0; m0 < M; m0 += T::BM)
        for (int n0 = 0; n0 < N; n0 += T::BN) {
            const int rows_a = M - m0 < T::BM ? M - m0 : T::BM, rows_b = N - n0 < T::BN ? N - n0 : T::BN;
            for (int wave = 0; wave < T::NW; ++wave)
                for (int lane = 0; lane < 64; ++lane) {
                    auto fragments = [&](const char *what, int row0, int inside, int f0, int loads, i64 operand) {
                        for (int t = 0; t < loads; ++t)
                            for (int step = 0; step < 4 * chunks; ++step) {
                                const int f = f0 + t, row = row0 + f * 16;
                                const bool real = f * 16 < inside;
                                touch(what, fragment_base(row0, f0, band), share_bytes(f0 * 16, inside, band), fragment_lane(lane), fragment_scalar(f, step), 16,
                                      operand, real ? (i64)(row / 128) * band + (i64)step * kFragmentStep + row % 128 / 16 * 1024 + lane * 16 : -1);
                            }
                    };
                    fragments("fragments of A", m0, rows_a, wave * T::LA, T::LA, frags_a);
                    if (IF4) {
                        fragments("fragments of B", n0, rows_b, wave * T::LB, T::LB, frags_b);
                        continue;
                    }
                    for (int chunk = 0; chunk < chunks; ++chunk) {
                        const int f0 = wave * T::LB, g0 = wave * T::LS;
                        for (int t = 0; t < T::LB; ++t) {
                            const int row = n0 + (f0 + t) * 16 + (lane & 15), byte = chunk * 64 + (lane >> 4) * 16;
                            touch("codes", (i64)(n0 + f0 * 16) * kbytes, share_bytes(f0 * 16, rows_b, T::LB * 16 * kbytes),
                                  whole_or(is_half(chunk, kbytes), lane, codes_lane(lane, kbytes)),
                                  codes_scalar(t, chunk, kbytes), 16, codes, (f0 + t) * 16 < rows_b && byte < (int)kbytes ? (i64)row * kbytes + byte : -1);
                        }
                        for (int t = 0; t < T::LS; ++t) {
                            const int g = g0 + t, tile = 2 * chunk + (g & 3) / 2;  // (64 k each)
                            touch("scales", scales_base(n0, g0, scale_band), share_bytes(g0 * 32, rows_b, scale_band), scales_lane(lane),
                                  scales_scalar(g, chunk, is_half(chunk, kbytes)), 4, scales,
                                  g * 32 < rows_b && tile * 64 < K ? (i64)((n0 + g * 32) / 128) * scale_band + tile * 512 + (g & 1) * 256 + lane * 4 : -1);
                        }
                    }
                }
        }
}
template <int WAVES_M, int WAVES_N, int WM>
static void tiles() {
    for (int M : {128, 256, 384, 640})
        for (int N : {128, 256, 384, 640})
            for (int K : {64, 128, 192, 384, 1024, 1088}) {
                walk<HalfTile<WAVES_M, WAVES_N, WM, false>, false>(M, N, K);
                walk<HalfTile<WAVES_M, WAVES_N, WM, true>, true>(M, N, K);
            }
}
int main() {
    tiles<2, 4, 8>();
    tiles<1, 4, 8>();
    tiles<2, 2, 4>();
    puts("inside");
}
"""

STREAM = r"""
int main() {
    for (int N : {128, 384})
        for (int K : {8192, 8256, 8320})
            for (int n0 = 0; n0 < N; n0 += 64) {
                const uint32_t kbytes = K / 2, scale_band = (uint32_t)K * 8;
                const i64 codes = (i64)N * kbytes, scales = (i64)(N / 128) * scale_band;
                for (int chunk = 0; chunk * 128 < K; ++chunk)
                    for (int lane = 0; lane < 64; ++lane)
                        for (int j = 0; j < 4; ++j) {
                            const bool half = is_half(chunk, kbytes);
                            const int row = n0 + 16 * j + (lane & 15), k = chunk * 128 + (lane >> 4) * 32, in_band = row & 127;
                            touch("codes", (i64)n0 * kbytes, 64 * kbytes, stream_codes_lane(lane, j, kbytes, half), chunk * 64, 16, codes,
                                  k < K ? (i64)row * kbytes + k / 2 : -1);
                            touch("scales", (i64)(n0 / 128) * scale_band, scale_band, stream_scales_lane(lane, j, n0, half), chunk * 1024, 2, scales,
                                  k < K ? (i64)(row / 128) * scale_band + k / 64 * 512 + (in_band & 31) * 16 + in_band / 32 * 4 + (k & 32) / 16 : -1);
                        }
            }
    puts("inside");
}
"""

MXFP4 = r"""
// rows of one operand in a tile of BROWS rows: lane i of a load fills unit i & 7 of row i >> 3
static void walk(int tile_rows, int rows, int K) {
    const uint32_t kbytes = K / 2, chunks = K / 128;
    const int steps = (K + 255) / 256;
    for (int row0 = 0; row0 < rows; row0 += tile_rows) {
        const int inside = rows - row0 < tile_rows ? rows - row0 : tile_rows;
        for (int step = 0; step < steps; ++step)
            for (int lane = 0; lane < 64; ++lane) {
                const bool half = mx_is_half(step, kbytes);
                for (int wave = 0; wave < 8; ++wave)
                    for (int t = 0; t < tile_rows / 64; ++t) {
                        const int row = wave * (tile_rows / 8) + t * 8 + lane / 8, byte = step * 128 + (((lane & 7) ^ (row / 2 % 8)) * 16);
                        touch("codes", (i64)row0 * kbytes, (uint32_t)inside * kbytes,
                              mx_whole_or(half, lane, t & 1, mx_codes_lane(wave * (tile_rows / 8), lane, t & 1, kbytes)), mx_codes_scalar(t, step, kbytes), 16,
                              (i64)rows * kbytes, row < inside && byte < (int)kbytes ? (i64)(row0 + row) * kbytes + byte : -1);
                    }
                for (int band = 0; band < inside / 128; ++band) {
                    const i64 at = (i64)(row0 / 128 + band) * chunks * 512, of_step = step * 1024 + lane * 16;
                    touch("scales", at, chunks * 512, whole_or(half, lane, mx_scales_lane(lane)), mx_scales_scalar(step), 16, (i64)(rows / 128) * chunks * 512,
                          of_step < (i64)chunks * 512 ? at + of_step : -1);
                }
            }
    }
}
int main() {
    for (int rows : {128, 256, 384, 640})
        for (int K : {128, 256, 384, 1024, 1152}) {
            walk(128, rows, K);
            walk(256, rows, K);
        }
    puts("inside");
}
"""


@pytest.mark.parametrize("source", [HALF, STREAM, MXFP4], ids=["converted_ahead", "weight_streamed", "mxfp4"])
def test_loads_stay_inside_their_operands(tmp_path, source):
    compiler = os.environ.get("CXX") or shutil.which("g++")
    (tmp_path / "walk.cpp").write_text(COMMON + source)
    subprocess.run([compiler, "-std=c++17", "-O1", f"-I{CSRC}", str(tmp_path / "walk.cpp"), "-o", str(tmp_path / "walk")], check=True)
    run = subprocess.run([str(tmp_path / "walk")], capture_output=True, text=True)
    assert run.stdout == "inside\n", run.stdout
