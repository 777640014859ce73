// gfx950 NVFP4 / IF4 products with one operand converted ahead: A as fp16(value * scale) in the order the matrix
// instructions read it, B packed.
//
// What bounds the products of more than a few hundred rows is power: the matrix cores run at the clock the board allows,
// so everything else a K step does costs clock.  Against the kernel that reads both operands packed (gemm_nvfp4_kernel,
// every code of A converted again by every column of tiles and staged through registers), A arrives in LDS without passing
// through registers, its fragments are read with one instruction each, conflict-free and without address arithmetic,
// and only B's conversions are left, 32 VALU instructions per wavefront and 32 matrix instructions.  16 x 16 x 32 matrix
// instructions draw less than 32 x 32 x 16 (the accumulators are read and written half as often per product).
// Measured on one box, products alone (us): 16384 x 4096 -> 14336 1392 -> 1189, 8192 x 4096 -> 4096 202 -> 172,
// 1024 x 4096 -> 14336 95 -> 78, 2048 x 4096 -> 4096 60 -> 51; with B converted ahead as well (and read through LDS):
// 1195, 166, 78, 48, before the passes that convert it, 24 us for 14336 x 4096.
//
// Layout of A ("fragments"): bands of 128 rows; inside a band chunks of 128 k; inside a chunk four steps w of 32 k; inside
// a step eight fragments of 16 rows, 1 KiB each: 16 bytes per lane, lane (m = l & 15, q = l >> 4) holding the eight
// k = 32 q + 8 w ... 32 q + 8 w + 7 of the chunk of row m.  The contraction index is permuted that way so that the codes a lane
// multiplies over the four steps of a chunk are 16 consecutive bytes of its row of B; A and B use the same permutation.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fos_buffer.h"
#include "fos_gemm_common.h"
#include "fos_gemm_half.h"
#include "fos_gemm_tiles.h"

namespace fos {

namespace {

typedef float float4v __attribute__((ext_vector_type(4)));
typedef int int4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void *LdsPtr;

// Buffer descriptor as four plain words (for inline assembly): base, stride 0, size in bytes, raw 32-bit offsets with
// range checking.
FOS_DEVICE int4v raw_rsrc(const void *base, uint32_t bytes) {
    const uint64_t a = (uint64_t)(uintptr_t)base;
    int4v v = {(int)(uint32_t)a, (int)(uint32_t)((a >> 32) & 0xffffu), (int)bytes, 0x00020000};
    return v;
}

// The two block scales a lane multiplies over a chunk, of which `left` blocks of the lane's pair exist (padding of the
// inner dimension may hold anything: its scales are taken for zeros).
FOS_DEVICE uint32_t tail_mask(int left) { return left <= 0 ? 0u : left == 1 ? 0xffu : 0xffffu; }

}  // namespace

// ---------------------------------------------------------------------------------------
// Codes and scales -> fragments.  Memory-bound: 0.5625 bytes read and 2 written per element; 16384 x 4096 27 us = 6.4 TB/s.
// A workgroup takes 16 rows and four chunks, a wavefront a chunk: 64 contiguous bytes of each of 16 rows in, four whole
// KiB out.  Rows from `rows` on (a band is written whole) and blocks from `depth` on are zeros.  A second operand follows
// in the same launch (blocks of rows from p.groups on).
constexpr int kExpandGroupsY = 32768;  // (a grid has at most 65535 workgroups along y and z: more blocks of rows go on along z)
template <bool IF4>
__global__ __launch_bounds__(256) void expand_fragments_kernel(const ExpandParams p) {
    const int64_t chunks = (p.K + 127) >> 7, chunk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (chunk >= chunks) return;
    const int group = (int)(blockIdx.z * kExpandGroupsY + blockIdx.y);
    if (group >= p.groups_all) return;
    const int second = group >= p.groups;  // (uniform)
    const ExpandOperand &o = p.operand[second];
    const int lane = threadIdx.x & 63, q = lane >> 4;
    const int64_t row = (int64_t)(group - (second ? p.groups : 0)) * 16 + (lane & 15), k0 = chunk * 128 + q * 32;
    uint4 w = make_uint4(0u, 0u, 0u, 0u);
    uint32_t s = 0u;
    if (row < o.rows && k0 < p.K) {
        w = *reinterpret_cast<const uint4 *>(o.codes + row * (p.K >> 1) + (k0 >> 1));
        const int64_t at = IF4 ? row * (p.K >> 4) + (k0 >> 4)
                               : ((row >> 7) * (p.K >> 6) + (k0 >> 6)) * 512 + (row & 31) * 16 + ((row & 127) >> 5) * 4 + ((k0 >> 4) & 3);
        s = *reinterpret_cast<const uint16_t *>(o.sf + at) & tail_mask((int)((p.depth - k0 + 15) >> 4));
    }
    uint8_t *out = o.out + ((row >> 7) * chunks + chunk) * kBandChunkBytes + ((row & 127) >> 4) * 1024 + lane * 16;
    *reinterpret_cast<half8_t *>(out) = dequant_word<IF4>(w.x, s, 0);
    *reinterpret_cast<half8_t *>(out + kFragmentStep) = dequant_word<IF4>(w.y, s, 0);
    *reinterpret_cast<half8_t *>(out + 2 * kFragmentStep) = dequant_word<IF4>(w.z, s, 1);
    *reinterpret_cast<half8_t *>(out + 3 * kFragmentStep) = dequant_word<IF4>(w.w, s, 1);
}

int launch_expand_fragments(ExpandParams p, bool if4, hipStream_t s) {
    p.groups = (int)((p.operand[0].rows + 127) / 128 * 8);
    p.groups_all = p.groups + (int)((p.operand[1].rows + 127) / 128 * 8);
    const int along_y = p.groups_all < kExpandGroupsY ? p.groups_all : kExpandGroupsY;
    const dim3 grid((unsigned)((p.K + 511) / 512), (unsigned)along_y, (unsigned)((p.groups_all + along_y - 1) / along_y));
    if (if4) hipLaunchKernelGGL(expand_fragments_kernel<true>, grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL(expand_fragments_kernel<false>, grid, dim3(256), 0, s, p);
    return hipGetLastError() == hipSuccess ? FOS_OK : FOS_E_LAUNCH;
}

// ---------------------------------------------------------------------------------------
// The product.  WAVES_M x WAVES_N wavefronts, each 16 WM rows x 64 columns.  As in the other kernels the matrix
// instruction's first operand is B (rows n), so that a lane's four accumulators are four consecutive n of row m = lane & 15.
//
// K runs in steps of 32.  A's share of a step (BM / 16 KiB) and B's of a chunk of four steps (BN rows x 64 bytes of codes and
// 8 of scales) go from global memory straight into LDS: kSlotsA steps and two chunks are in flight or in use.  The one
// wait and barrier of a step stands BAR matrix instructions into it: every wavefront has then read what it needs of step
// k (into registers, during step k - 1), so its slot takes the loads of step k + kSlotsA, and step k + 1 has arrived, whose
// fragments are read one at a time between the matrix instructions that follow.  B's codes go from LDS to registers once a
// chunk; the fragment of the next 16 columns is converted between the matrix instructions of the current ones.  Everything
// is issued in the order it is written in (sched_barrier): left to itself the scheduler bunches the reads.
// The loads are inline assembly without outputs: the compiler would order a wait for all loads in flight before every LDS
// read behind a load into LDS that it knows about.  No other vector-memory load is in the loop, so the waits by hand are all there are.
constexpr int kSlotsA = 4, kSlotsB = 2;

constexpr int half_lds_bytes(int BM, int BN, bool if4) {
    const int loop = kSlotsA * BM * 64 + (if4 ? kSlotsA * BN * 64 : kSlotsB * BN * 72), epilogue = BM * BN / 8192 * 32 * 144;
    return loop > epilogue ? loop : epilogue;
}

template <int I>
FOS_DEVICE void convert_pair(half8_t &f, uint32_t word, half2_t s) {
    const half2_t v = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, I) * s;
    f[2 * I] = v.x;
    f[2 * I + 1] = v.y;
}

// IF4: B as fragments too, loaded and read as A is.  Its conversion takes 34 instructions a word and in the loop bounded the
// product (2048 x 4096 x 4096 123 us on 128 x 128 tiles, the others spilled; 95 in gemm_nvfp4_kernel); ahead of it, it
// is bound by memory.
template <int WAVES_M, int WAVES_N, int WM, int BAR, int OCC, int OUT, bool IF4>
__global__ __launch_bounds__(64 * WAVES_M *WAVES_N, OCC) void gemm_half_kernel(const GemmParams p) {
    constexpr bool OUT_BF16 = OUT == kOutBF16;
    typedef HalfTile<WAVES_M, WAVES_N, WM, IF4> Tile;
    constexpr int WN = 4, NW = Tile::NW, BM = Tile::BM, BN = Tile::BN, MFMAS = WM * WN;
    constexpr int kSlotA = BM * 64, kCodesB = BN * 64, kSlotB = IF4 ? BN * 64 : BN * 72, kBaseB = kSlotsA * kSlotA;
    constexpr int LA = Tile::LA, LB = Tile::LB, LS = Tile::LS, LSTEP = IF4 ? LA + LB : LA, LCHUNK = IF4 ? 0 : LB + LS;
    static_assert(LA == 2 && LB >= 1 && (WM == 4 || WM == 8), "shares of the loads");
    extern __shared__ __attribute__((aligned(16))) uint8_t half_lds[];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), q = lane >> 4;
    int tile_m, tile_n;
    tile_of(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n);
    const int64_t m0 = (int64_t)tile_m * BM, n0 = (int64_t)tile_n * BN;
    // (M and N are multiples of 128: a 256-wide tile may hang over the last 128 rows or columns)
    const int rows_a = (int)(p.M - m0 < BM ? p.M - m0 : BM), rows_b = (int)(p.N - n0 < BN ? p.N - n0 : BN);
    const int chunks_all = (int)((p.K + 127) >> 7);
    const int c0 = OUT == kOutPartial ? (int)blockIdx.y * p.ksteps_per_split : 0;
    const int chunks = OUT == kOutPartial ? (chunks_all - c0 < p.ksteps_per_split ? chunks_all - c0 : p.ksteps_per_split) : chunks_all;
    const int steps = 4 * chunks;
    const uint32_t band = (uint32_t)chunks_all * kBandChunkBytes, kbytes = (uint32_t)(p.K >> 1);
    const uint32_t scale_band = (uint32_t)p.K * 8u;
    // a wavefront's descriptors end with its own share of a tile, or are empty where that lies past the edge
    const int fa0 = wave * LA, fb0 = wave * LB, gs0 = wave * LS;
    const int4v ra = raw_rsrc(p.frags + fragment_base(m0, fa0, band), share_bytes(fa0 * 16, rows_a, band));
    const int4v rb = IF4 ? raw_rsrc(p.frags_b + fragment_base(n0, fb0, band), share_bytes(fb0 * 16, rows_b, band))
                         : raw_rsrc(p.B + (n0 + fb0 * 16) * kbytes, share_bytes(fb0 * 16, rows_b, LB * 16 * kbytes));
    const int4v rs = raw_rsrc(p.sfB + scales_base(n0, gs0, scale_band), share_bytes(gs0 * 32, rows_b, scale_band));  // (NVFP4)
    const uint32_t lds_base = (uint32_t)(uintptr_t)(LdsPtr)half_lds;
    const uint32_t va = fragment_lane(lane), vb = codes_lane(lane, kbytes), vs = scales_lane(lane);

    // m0 = LDS address of the run a wavefront fills (lane i: unit i); one wait state between a write of m0 and its use
    auto load16 = [&](uint32_t to, uint32_t offset, const int4v &r, uint32_t base) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(to), "v"(offset), "s"(r), "s"(base) : "memory");
    };
    auto load_step = [&](int step, int slot, int t) {
        if (t >= LA) {  // (IF4)
            const int f = fb0 + t - LA;
            load16(lds_base + kBaseB + slot * kSlotB + f * 1024, va, rb, fragment_scalar(f, c0 * 4 + step));
            return;
        }
        const int f = fa0 + t;
        load16(lds_base + slot * kSlotA + f * 1024, va, ra, fragment_scalar(f, c0 * 4 + step));
    };
    auto load_b = [&](int chunk, int slot, int t) {
        const uint32_t base = lds_base + kBaseB + slot * kSlotB;
        const bool half = is_half(c0 + chunk, kbytes);
        if (t < LB) {
            load16(base + (fb0 + t) * 1024, whole_or(half, lane, vb), rb, codes_scalar(t, c0 + chunk, kbytes));
        } else {
            const int g = gs0 + t - LB;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                         ::"s"(base + kCodesB + g * 256), "v"(vs), "s"(rs), "s"(scales_scalar(g, c0 + chunk, half)) : "memory");
        }
    };

    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const uint8_t *lds_a = half_lds + wm * WM * 1024 + lane * 16;
    const uint8_t *lds_b = half_lds + kBaseB + wn * 4096 + lane * 16;
    // scale bytes of column 64 wn + 16 j + (lane & 15), blocks 2 q and 2 q + 1 of the chunk
    const uint8_t *lds_s = half_lds + kBaseB + kCodesB + (wn >> 1) * 1024 + (q >> 1) * 512 + (lane & 15) * 16 + (wn & 1) * 8 + (q & 1) * 2;
    half8_t fa[2][WM], fb[2][IF4 ? WN : 1];  // (NVFP4: the current and the next 16 columns; IF4: the current and the next step)
    uint4 codes[2][WN];
    uint32_t scales[2][WN];
    half2_t s2[WN];
    auto read_step = [&](int slot, int set, int t) {
        if (t < WM) fa[set][t] = *reinterpret_cast<const half8_t *>(lds_a + slot * kSlotA + t * 1024);
        else if constexpr (IF4) fb[set][t - WM] = *reinterpret_cast<const half8_t *>(lds_b + slot * kSlotB + (t - WM) * 1024);
    };
    auto read_chunk = [&](int slot, int set, int t) {
        if (t < WN) codes[set][t] = *reinterpret_cast<const uint4 *>(lds_b + slot * kSlotB + t * 1024);
        else scales[set][t - WN] = *reinterpret_cast<const uint16_t *>(lds_s + slot * kSlotB + ((t - WN) & 1) * 256 + ((t - WN) >> 1) * 4);
    };
    const uint32_t last_mask = tail_mask((int)((p.depth - (int64_t)(chunks_all - 1) * 128 + 15) >> 4) - 2 * q);
    auto widen_scales = [&](int chunk, int set) {
        const uint32_t mask = c0 + chunk + 1 >= chunks_all ? last_mask : 0xffffu;
#pragma unroll
        for (int t = 0; t < WN; ++t) s2[t] = e4m3x2_to_half2(scales[set][t] & mask);
    };
    // pair i (0 .. 3) of word w of the next fragment: columns j of the chunk in register set `set`
    auto convert = [&](auto ic, half8_t &f, int set, int j, int w) {
        const uint4 &c = codes[set][j];
        const uint32_t word = w == 0 ? c.x : w == 1 ? c.y : w == 2 ? c.z : c.w;
        const half2_t s = w >= 2 ? __builtin_shufflevector(s2[j], s2[j], 1, 1) : __builtin_shufflevector(s2[j], s2[j], 0, 0);
        convert_pair<decltype(ic)::value>(f, word, s);
    };

    float4v acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.0f;

    // chunks 0, 1 of B and steps 0 .. 3 of A in flight (past the end: the last ones once more, into slots nobody reads)
    if constexpr (!IF4) {
#pragma unroll
        for (int c = 0; c < kSlotsB; ++c)
#pragma unroll
            for (int t = 0; t < LCHUNK; ++t) load_b(c < chunks ? c : chunks - 1, c, t);
    }
#pragma unroll
    for (int k = 0; k < kSlotsA; ++k)
#pragma unroll
        for (int t = 0; t < LSTEP; ++t) load_step(k, k, t);
#define FOS_HALF_WAIT(n) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(n) : "memory")
    FOS_HALF_WAIT((kSlotsA - 1) * LSTEP);
    constexpr int READS = WM + (IF4 ? WN : 0);  // fragments a wavefront reads per step
    if constexpr (!IF4) {
#pragma unroll
        for (int t = 0; t < 2 * WN; ++t) read_chunk(0, 0, t);
    }
#pragma unroll
    for (int t = 0; t < READS; ++t) read_step(0, 0, t);
    if constexpr (!IF4) {
        widen_scales(0, 0);
        static_for<0, 4>([&](auto ic) { convert(ic, fb[0][0], 0, 0, 0); });
    }

    int slot_b = 0;
    // (a chunk's four steps use the four slots of A in order; its codes are in register set CUR)
    auto chunk_steps = [&](int c, auto cur_c) {
        constexpr int CUR = decltype(cur_c)::value;
        const int c_next = c + kSlotsB < chunks ? c + kSlotsB : chunks - 1;
        static_for<0, 4>([&](auto wc) {
            constexpr int w = decltype(wc)::value, set = w & 1;
            const int k_next = 4 * c + w + kSlotsA < steps ? 4 * c + w + kSlotsA : steps - 1;
            static_for<0, MFMAS>([&](auto mc) {
                constexpr int m = decltype(mc)::value, j = m / WM, i = m % WM;
                if constexpr (m == BAR) {
                    // newer than the loads of step k + 1: two steps of A, and from the second step of a chunk on its B
                    // (issued behind A in the first step; a chunk is asked for seven steps ahead of its use)
                    FOS_HALF_WAIT(LSTEP * (kSlotsA - 2) + (w >= 1 ? LCHUNK : 0));
                    __builtin_amdgcn_sched_barrier(0);
                }
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(IF4 ? fb[set][IF4 ? j : 0] : fb[j & 1][0], fa[set][i], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                // conversion of the next fragment of B: the next columns of this step, or the first ones of the next step
                if constexpr (!IF4 && i % (WM / 4) == 0) {
                    constexpr int jn = (j + 1) % WN, wn_next = j + 1 == WN ? (w + 1) & 3 : w, from = j + 1 == WN && w == 3 ? CUR ^ 1 : CUR;
                    if constexpr (from != CUR && i == 0) widen_scales(c + 1, from);
                    convert(std::integral_constant<int, i / (WM / 4)>{}, fb[(j & 1) ^ 1][0], from, jn, wn_next);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (m >= BAR) {
                    // the reads of step k + 1, spread; ahead of the last step's the next chunk's codes and scales, which
                    // are converted from the last columns on
                    constexpr int x = m - BAR, nb = !IF4 && w == 3 ? 2 * WN : 0, reads = READS + nb, span = (nb ? 3 * WM - 2 : MFMAS) - BAR;
                    constexpr int first = x * reads / span < reads ? x * reads / span : reads,
                                  end = (x + 1) * reads / span < reads ? (x + 1) * reads / span : reads;
                    static_for<first, end>([&](auto tc) {
                        constexpr int t = decltype(tc)::value;
                        if constexpr (t < nb) read_chunk(slot_b ^ 1, CUR ^ 1, t);
                        else read_step((w + 1) & 3, set ^ 1, IF4 ? (t + WM) % READS : t - nb);  // (IF4: B's first)
                        __builtin_amdgcn_sched_barrier(0);
                    });
                    constexpr int gap = IF4 ? 2 : WM == 8 ? 4 : 2;
                    if constexpr (x >= 1 && (x - 1) % gap == 0 && (x - 1) / gap < LSTEP) {
                        load_step(k_next, w, (x - 1) / gap);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    constexpr int behind = 2 + gap * (LSTEP - 1);
                    if constexpr (w == 0 && x >= behind && x < behind + LCHUNK) {
                        load_b(c_next, slot_b, x - behind);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    static_assert(BAR + behind + LCHUNK <= MFMAS && span > 0, "room for the loads and reads behind the barrier");
                }
            });
        });
        slot_b ^= 1;
    };
    int c = 0;
    for (; c + 2 <= chunks; c += 2) {
        chunk_steps(c, std::integral_constant<int, 0>{});
        chunk_steps(c + 1, std::integral_constant<int, 1>{});
    }
    if (c < chunks) chunk_steps(c, std::integral_constant<int, 0>{});
    // loads still in flight write LDS: drain them, in every wavefront, before the slots are used again
    FOS_HALF_WAIT(0);

    // acc[i][j][e] is D[m][n] with m = 16 (wm WM + i) + (lane & 15), n = 64 wn + 16 j + 4 q + e
    // (a wavefront's 64 columns and every 32 rows lie wholly inside or outside the output)
    const bool columns_inside = wn * 64 < rows_b;
    if (OUT == kOutPartial) {
        if (!columns_inside) return;
        float *P = p.partials + (int64_t)blockIdx.y * p.M * p.N;
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            if ((wm * WM + i) * 16 >= rows_a) break;
            const int64_t m = m0 + (wm * WM + i) * 16 + (lane & 15);
#pragma unroll
            for (int j = 0; j < WN; ++j) *reinterpret_cast<float4v *>(P + m * p.N + n0 + wn * 64 + j * 16 + q * 4) = acc[i][j];
        }
        return;
    }
    float post;
    const float alpha = load_alpha(p, post);
    uint16_t *D = reinterpret_cast<uint16_t *>(p.D);
    // each wavefront turns 32 rows at a time round in LDS and stores whole rows of its 64 columns, 16 bytes a lane
    constexpr int kPitchOut = 144;
    uint8_t *epi = half_lds + wave * 32 * kPitchOut;
    const int real_cols = (int)(p.cols - n0 < BN ? p.cols - n0 : BN);
    const int real_rows = (int)(p.rows - m0 < BM ? p.rows - m0 : BM);  // (negative for a tile of padding)
    uint32_t umax = 0u;
#pragma unroll
    for (int i = 0; i < WM; i += 2) {
        const int row0 = (wm * WM + i) * 16;
        if (!columns_inside || row0 >= rows_a) break;  // (uniform over the wavefront)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            uint32_t um = 0u;
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = IF4 ? (alpha * acc[i + u][j][e]) * post : alpha * acc[i + u][j][e];
                *reinterpret_cast<uint2 *>(epi + (u * 16 + (lane & 15)) * kPitchOut + (j * 16 + q * 4) * 2) =
                    pack_outputs<OUT_BF16>(v, p.bias, n0 + wn * 64 + j * 16 + q * 4, um);
            }
            um = row0 + u * 16 + (lane & 15) < real_rows ? um : 0u;
            umax = max_pairs(umax, um);
        }
        // (LDS operations of one wavefront complete in order: its own writes are visible to its reads)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int row = t * 8 + (lane >> 3), c16 = lane & 7;
            const uint4 v = *reinterpret_cast<const uint4 *>(epi + row * kPitchOut + c16 * 16);
            if (!IF4 || wn * 64 + c16 * 8 < real_cols)
                *reinterpret_cast<uint4 *>(D + (m0 + row0 + row) * p.ldd + n0 + wn * 64 + c16 * 8) = v;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    if (p.d_amax) {
        __syncthreads();  // every wavefront is done with its piece of the staging
        fold_amax<OUT_BF16, NW>(p.d_amax, umax, reinterpret_cast<uint32_t *>(half_lds));
    }
}

// ---------------------------------------------------------------------------------------
// M <= 128: the weight is streamed once, a workgroup owns 64 columns (and a share of K, blockIdx.y), its four wavefronts take
// the chunks of K in turn, each with all rows: 128 rows x 64 columns of accumulators a wavefront, one wavefront per SIMD.  Nothing
// is shared in the loop: fragments of A are whole KiB out of L2 into registers, B's codes 64 contiguous bytes of 16
// rows, both a chunk ahead, no barrier.  A kernel that reads A packed is bound by its conversion, which every 64 columns
// repeat (gemm_nvfp4_skinny_kernel); this one by what a compute unit reads of A out of L2, about 30 bytes a cycle.
// (Eight wavefronts with A a step ahead: 24.5 us at 128 x 4096 x 14336 in four splits, 23.5 here.)
// The accumulators are summed over the wavefronts in two halves through LDS, in fixed order.
// HALF_CHUNK: K % 128 = 64, whose last chunk exists by half (the choice of lane offsets in the loop cost 1 % of the layer of 128 x 14336 -> 4096).
template <int OUT, bool HALF_CHUNK>
__global__ __launch_bounds__(256, 1) void gemm_half_stream_kernel(const GemmParams p) {
    constexpr bool OUT_BF16 = OUT == kOutBF16;
    constexpr int WM = 8, WN = 4, kWaves = 4, HALF = WM * WN / 2;  // HALF: groups of four accumulators a lane hands over at a time
    extern __shared__ __attribute__((aligned(16))) uint8_t half_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), q = lane >> 4;
    const int64_t n0 = (int64_t)blockIdx.x * 64;
    const int chunks_all = (int)((p.K + 127) >> 7);
    const int c0 = OUT == kOutPartial ? (int)blockIdx.y * p.ksteps_per_split : 0;
    const int c1 = OUT == kOutPartial ? (c0 + p.ksteps_per_split < chunks_all ? c0 + p.ksteps_per_split : chunks_all) : chunks_all;
    const uint32_t kbytes = (uint32_t)(p.K >> 1), scale_band = (uint32_t)p.K * 8u;
    const BufferRsrc ra = make_rsrc(p.frags, (uint32_t)chunks_all * kBandChunkBytes);
    const BufferRsrc rb = make_rsrc(p.B + n0 * kbytes, 64u * kbytes);
    const BufferRsrc rs = make_rsrc(p.sfB + (n0 >> 7) * (int64_t)scale_band, scale_band);
    const uint32_t va = fragment_lane(lane);

    half8_t fa[4][WM];  // a chunk; refilled one at a time with the next chunk's, behind the matrix instructions that read it last
    u32x4 codes[2][WN];
    uint32_t scales[2][WN];
    auto load_a = [&](int chunk, int w, int i) {
        const uint32_t at = (uint32_t)chunk * kBandChunkBytes + (uint32_t)w * kFragmentStep;
        fa[w][i] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(ra, (int)(va + i * 1024), (int)at, 0));
    };
    auto load_b = [&](int chunk, int set) {
        const bool half = HALF_CHUNK && is_half(chunk, kbytes);
#pragma unroll
        for (int j = 0; j < WN; ++j)
            codes[set][j] = __builtin_amdgcn_raw_buffer_load_b128(rb, (int)stream_codes_lane(lane, j, kbytes, half), chunk * 64, 0);
#pragma unroll
        for (int j = 0; j < WN; ++j)
            scales[set][j] = __builtin_amdgcn_raw_buffer_load_b16(rs, (int)stream_scales_lane(lane, j, n0, half), chunk * 1024, 0);
    };
    const uint32_t last_mask = tail_mask((int)((p.depth - (int64_t)(chunks_all - 1) * 128 + 15) >> 4) - 2 * q);

    float4v acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

    // (past the end: the last chunk once more, which nobody multiplies)
    auto clamp = [&](int c) { return c < c1 ? c : c1 - 1; };
    load_b(clamp(c0 + wave), 0);
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int i = 0; i < WM; ++i) load_a(clamp(c0 + wave), w, i);
    auto chunk_steps = [&](int c, auto cur_c) {
        constexpr int CUR = decltype(cur_c)::value;
        load_b(clamp(c + kWaves), CUR ^ 1);
        half2_t s2[WN];
        const uint32_t mask = c + 1 == chunks_all ? last_mask : 0xffffu;
#pragma unroll
        for (int j = 0; j < WN; ++j) s2[j] = e4m3x2_to_half2(scales[CUR][j] & mask);
        static_for<0, 4>([&](auto wc) {
            constexpr int w = decltype(wc)::value;
            half8_t fb[WN];
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                const uint32_t word = w == 0 ? codes[CUR][j].x : w == 1 ? codes[CUR][j].y : w == 2 ? codes[CUR][j].z : codes[CUR][j].w;
                fb[j] = dequant8(word, w >= 2 ? __builtin_shufflevector(s2[j], s2[j], 1, 1) : __builtin_shufflevector(s2[j], s2[j], 0, 0));
            }
#pragma unroll
            for (int i = 0; i < WM; ++i) {
#pragma unroll
                for (int j = 0; j < WN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[j], fa[w][i], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                load_a(clamp(c + kWaves), w, i);
                __builtin_amdgcn_sched_barrier(0);
            }
        });
    };
    int c = c0 + wave;
    for (; c + kWaves < c1; c += 2 * kWaves) {
        chunk_steps(c, std::integral_constant<int, 0>{});
        chunk_steps(c + kWaves, std::integral_constant<int, 1>{});
    }
    if (c < c1) chunk_steps(c, std::integral_constant<int, 0>{});

    // Sum over the wavefronts: of either half of the rows' fragments every wavefront leaves its HALF groups in LDS, then sums
    // its share of them over all wavefronts in order and stores those.
    float post;
    const float alpha = OUT == kOutPartial ? 0.0f : load_alpha(p, post);
    constexpr int kMine = HALF / kWaves;
    uint32_t umax = 0u;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        __syncthreads();
#pragma unroll
        for (int f = 0; f < HALF; ++f)
            *reinterpret_cast<float4v *>(half_lds + ((wave * HALF + f) * 64 + lane) * 16) = acc[h * (WM / 2) + f / WN][f % WN];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kMine; ++u) {
            const int f = wave * kMine + u, i = h * (WM / 2) + f / WN, j = f % WN;
            float4v sum = *reinterpret_cast<const float4v *>(half_lds + (f * 64 + lane) * 16);
#pragma unroll
            for (int w = 1; w < kWaves; ++w) sum += *reinterpret_cast<const float4v *>(half_lds + ((w * HALF + f) * 64 + lane) * 16);
            const int64_t m = 16 * i + (lane & 15), n = n0 + 16 * j + 4 * q;
            if (m >= p.M) continue;
            if (OUT == kOutPartial) {
                *reinterpret_cast<float4v *>(p.partials + ((int64_t)blockIdx.y * p.M + m) * p.N + n) = sum;
            } else {
                const float v[4] = {alpha * sum[0], alpha * sum[1], alpha * sum[2], alpha * sum[3]};
                uint32_t um = 0u;
                *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(p.D) + m * p.ldd + n) = pack_outputs<OUT_BF16>(v, p.bias, n, um);
                if (m < p.rows) umax = max_pairs(umax, um);
            }
        }
    }
    if (OUT != kOutPartial && p.d_amax) {
        __syncthreads();
        fold_amax<OUT_BF16, kWaves>(p.d_amax, umax, reinterpret_cast<uint32_t *>(half_lds));
    }
}

template <bool HALF_CHUNK>
static int launch_stream(GemmParams &p, int out_type, hipStream_t s) {
    constexpr int lds_bytes = 64 * 1024;  // half the accumulators of four wavefronts
    auto kernel = p.splits > 1 ? gemm_half_stream_kernel<kOutPartial, HALF_CHUNK>
                  : out_type == FOS_T_BF16 ? gemm_half_stream_kernel<kOutBF16, HALF_CHUNK> : gemm_half_stream_kernel<kOutF16, HALF_CHUNK>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(p.N / 64), (unsigned)p.splits), dim3(256), lds_bytes, s, p);
    return hipGetLastError() == hipSuccess ? FOS_OK : FOS_E_LAUNCH;
}

template <int WAVES_M, int WAVES_N, int WM, int BAR, int OCC, bool IF4>
static int launch_tiles(GemmParams &p, int out_type, hipStream_t s) {
    constexpr int BM = 16 * WM * WAVES_M, BN = 64 * WAVES_N, lds_bytes = half_lds_bytes(BM, BN, IF4);
    p.tiles_m = (int)((p.M + BM - 1) / BM);
    p.tiles_n = (int)((p.N + BN - 1) / BN);
    auto kernel = p.splits > 1             ? gemm_half_kernel<WAVES_M, WAVES_N, WM, BAR, OCC, kOutPartial, IF4>
                  : out_type == FOS_T_BF16 ? gemm_half_kernel<WAVES_M, WAVES_N, WM, BAR, OCC, kOutBF16, IF4>
                                           : gemm_half_kernel<WAVES_M, WAVES_N, WM, BAR, OCC, kOutF16, IF4>;
    if (lds_bytes > 64 * 1024 && hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess)
        return FOS_E_LAUNCH;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(p.tiles_m * p.tiles_n), (unsigned)p.splits), dim3(64 * WAVES_M * WAVES_N), lds_bytes, s, p);
    return hipGetLastError() == hipSuccess ? FOS_OK : FOS_E_LAUNCH;
}

int launch_gemm_half(GemmParams &p, int tile, bool if4, int out_type, hipStream_t s) {
    if (if4) {
        if (tile == kHalf256) return launch_tiles<2, 4, 8, 12, 2, true>(p, out_type, s);
        if (tile == kHalfWide) return launch_tiles<1, 4, 8, 12, 2, true>(p, out_type, s);
        return launch_tiles<2, 2, 4, 4, 2, true>(p, out_type, s);
    }
    if (tile == kHalfStream) return p.K % 128 ? launch_stream<true>(p, out_type, s) : launch_stream<false>(p, out_type, s);
    if (tile == kHalf256) return launch_tiles<2, 4, 8, 12, 2, false>(p, out_type, s);
    if (tile == kHalfWide) return launch_tiles<1, 4, 8, 12, 2, false>(p, out_type, s);
    return launch_tiles<2, 2, 4, 4, 2, false>(p, out_type, s);
}

}  // namespace fos
