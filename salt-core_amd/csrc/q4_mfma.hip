// Prefill-sized affine-Q4 matmul on the MFMA units (tolerance class).
//
// When many tokens meet one weight matrix the work is a dense contraction and
// the 32-chain order of the decode kernels cannot be kept at matrix-core speed.
// This kernel computes Y[token][row] = sum_c (q*s + b)[row][c] * x[token][c]
// with fp32-level accuracy but in a different summation order; callers opt in
// and are told so (the engine's bit-exact path remains the tiled kernels).
//
// How the affine weights reach the matrix cores without losing bits:
//  * q s + b = s (q - 8) + (b + 8 s).  q - 8 lies in -8..7: three significant
//    bits, or a power of two.  Times the eight of a bf16 scale that is at most
//    eleven, an fp16 significand, so s (q - 8) is an exact fp16 operand and the
//    whole row accumulates in the matrix cores with no work per scale group.
//  * fp16's exponents are the limit: a row's scales are brought to the top of
//    its range by a power of two 2^(11 - E) (E from the row's largest |s| and
//    |b| / 8), below which 28 binades are exact.  A tile with scales further
//    apart walks its columns once per 28 binades ("window"), each time with the
//    other scales taken as zero, and adds the results in the output.  Weights in
//    earnest span a few binades: one window.
//  * a nibble becomes the fp16 value 16 + q with two bit operations per pair,
//    and fma(16 + q, s, -24 s) is s (q - 8), exact at every step.
//  * the activation row is scaled by a power of two that puts its largest
//    magnitude in [2^13, 2^14) and split into two fp16 planes, x * 2^k = hi + lo
//    (each rounded to nearest: 23 significant bits, |x 2^k - hi - lo| <= 2^-22
//    of the element's own magnitude, or 2^-25 of the scaled row for elements so
//    small that lo is subnormal); each plane is an exact MFMA operand,
//    accumulation is fp32, and the powers of two leave with the store.
//  * the bias term sum_g (b_g + 8 s_g) * X_g (X_g = the group sums of x) is
//    itself a small contraction over the groups; b and s are bf16, so it runs
//    on the matrix cores once per tile before the main loop, with X_g split
//    into three bf16 planes (v = hi + mid + lo to 2^-24).
//
// Tiling.  A wave computes 64 tokens x 64 weight rows as 2 x 2 blocks of
// v_mfma_f32_32x32x16_f16 (tokens are the M rows, weight rows the N columns).
// The codes of its rows go from memory to its registers and are converted
// there, once per 64 tokens; the token planes are staged in LDS for the
// workgroup, two stages, the next one's loads in flight during the matrix work,
// one barrier per stage.  Per 16 columns a wave reads 4 KB of LDS for eight
// matrix instructions, 64 bytes per clock of the 128 a compute unit has, and
// issues 24 other vector instructions in their shadow.  The four waves of a
// workgroup are four row blocks: the tile is 64 tokens x 256 rows, or 32 tokens
// where a launch is small.
//
// Order of the sums.  A wave walks all columns of its block from the first to
// the last, so an output depends on its token and its row alone: not on the
// number of tokens or rows in the call nor on the tile that holds it, and a
// prompt cut into pieces gives the same bits.  Launches with fewer tiles than
// compute units pay for that.  Two or four parts of the columns side by side in
// a workgroup, added at the end, are faster there (33 tokens against 8192 x 2816
// 25.6 us in four parts, 39.5 in one; against 8192 x 8192 51 and 97) and slower
// in larger launches (333 tokens against 16384 x 2816: 175 us in four parts, 114
// in two, 84 in one), so that the order would follow the number of tokens.
// Fixed parts, one after the other in one workgroup where the launch is large,
// cost that one 129 us (the sums meet in the output), and two fixed parts on
// eight waves 102.
//
// Bound: the matrix cores, which execute twice the useful operations, at the
// clock that their power leaves them: in the grouped prefill (2048 tokens, 128
// experts, top-8, 2816/704: 946 -> 592 us a layer) 51 % busy in gate and up, 37 % in
// down, at 1.6 to 2.1 GHz;
// one 16384 x 2816 matrix, 333 tokens: 101 -> 76 us (256 tokens, one tile of 64
// for each compute unit, 55 us: 1.1 PFLOP/s of both planes).  Before, every scale
// group cost 16 multiply-adds per block and a conversion in each of two waves,
// and each 32 bytes of codes and each scale fetched a cache line of its own.
// Calls of few tiles are bound by one wave per SIMD, whose dependent vector
// instructions issue eight clocks apart: 33 tokens, 8192 x 2816 39.5 -> 34.1 us
// and 8192 x 8192 98.7 -> 84.9, 64 tokens, 4096 x 4096 54.3 -> 46.2 once nothing
// in the walk waits but what has to (lds_load.h).
//
// Inside every aligned run of eight columns the planes are stored in the order
// 0,4,1,5,2,6,3,7, which is the order the pair extraction yields the codes in;
// the two lane halves of an instruction take columns 32 h + 8 k .. + 7 of a
// scale group, so that a lane's codes of a group are 16 consecutive bytes.
#include "device_math.h"
#include "lds_load.h"
#include "mi355_internal.h"

#include <stddef.h>

#include <type_traits>

namespace mi355 {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 __attribute__((aligned(2))) u32x4_any;                 // rows of scales start on any even address
typedef const uint64_t __attribute__((address_space(4))) *uniform_u64_ptr;
typedef const u32x4 __attribute__((address_space(1))) *global_u128_ptr;
typedef const u32x4_any __attribute__((address_space(1))) *global_u128_any_ptr;
typedef const uint16_t __attribute__((address_space(1))) *global_u16_ptr;
typedef const uint8_t __attribute__((address_space(1))) *global_u8_ptr;
typedef const int __attribute__((address_space(1))) *global_i32_ptr;
typedef float __attribute__((address_space(1))) *global_f32_out;

constexpr int TM = MFMA_TM;                 // tokens per workgroup, or half of it
constexpr int CUS = 256;
constexpr int X_PLANES = 2;                 // fp16 planes of the scaled activation
constexpr int WINDOW = 28;                  // binades of scale that are exact fp16 operands at a time
constexpr int MAX_WINDOWS = 10;             // all of a bf16's binades
constexpr int WEIGHT_TOP = 11;              // scales are brought below 2^WEIGHT_TOP: 24 * 2^11 is inside fp16

// A row of the third plane holds what the split has to say about its row of x: at byte 0 the exponent k of the power
// of two 2^-k that undoes its scaling, from byte 16 on the group sums in blocks of sixteen groups, a block as three bf16
// planes of sixteen entries (96 bytes).
// The bias pass reads scales, biases and sums eight groups at a time, the last eight of a row from its end backwards,
// so that it never reads past the row: entry j of eight c stands for group eight_start(c) + j, and is zero where an
// earlier eight already holds that group.  16 + 6 * padded_groups(C / 64) bytes fit the 2 * C of the row for every C.
__host__ __device__ constexpr int padded_groups(int ngrp) { return (ngrp + 15) & ~15; }
__device__ __forceinline__ int sum_entry(int at, int plane) { return 8 + (at >> 4) * 48 + plane * 16 + (at & 15); }   // in halves
__device__ __forceinline__ int eight_start(int c, int ngrp) {
    const int last = ngrp > 8 ? ngrp - 8 : 0;
    return 8 * c < last ? 8 * c : last;
}

// LDS holds two stages of the token planes, one scale group each, and for every wave one chunk, CH groups, of the codes
// and the scale bits of its own 64 rows: 128 bytes of a row at a time, because a cache line that is fetched again for
// each of its quarters costs as much as four lines.
constexpr int ROW_WAVES = 4;
constexpr int CH = 4;
constexpr int STAGE_BYTES = X_PLANES * TM * 128;
constexpr int W_OFF = 2 * STAGE_BYTES, W_BYTES = 64 * 32 * CH;           // of one wave
constexpr int S_OFF = W_OFF + ROW_WAVES * W_BYTES, S_BYTES = 64 * 4 * CH;
// Blocks of group sums of all tokens for the bias pass: three at a time, two of them where the second stage of planes comes
// later and one of its own.
constexpr int SUM_BYTES = TM * 96, SUM_OFF = S_OFF + ROW_WAVES * S_BYTES, SUM_BLOCKS = 3;
constexpr int LDS_BYTES = SUM_OFF + SUM_BYTES;
static_assert(2 * SUM_BYTES <= STAGE_BYTES && 2 * (LDS_BYTES + 2048) <= 160 * 1024, "two workgroups per compute unit");
__device__ __forceinline__ int sum_place(int block) { return block < 2 ? STAGE_BYTES + block * SUM_BYTES : SUM_OFF; }
constexpr int XT = TM / (8 * ROW_WAVES);         // loads per wave and plane: eight token rows each
constexpr int PIECES = 2 * CH;                   // 16-byte pieces of a row's chunk
constexpr int WT = PIECES;                       // loads per wave and chunk: 64 / PIECES rows each
static_assert(MFMA_TN == 64 * ROW_WAVES, "a wave has 64 of the tile's rows");

// Planes arrive in LDS by loads that write 64 consecutive 16-byte pieces, so rows cannot be padded: piece p of token
// row r lies at place p ^ place_mask(r), which spreads the sixteen rows of an LDS read phase over all banks.  The
// same for the codes.
static_assert(PIECES == 8, "place_mask covers rows of eight pieces");
__device__ __forceinline__ int place_mask(int row) { return (row >> 1) & 7; }

template <int N> __device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The workgroup meets; a wave's LDS reads are done, its loads on their way stay there (__syncthreads waits for them).
__device__ __forceinline__ void meet() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

static_assert(sizeof(MfmaJob) == 56, "find_job reads a job record as seven 64-bit words");

// In a table every job has L.row_tiles tiles of rows: the job follows from the tile's number by one load.
__device__ __forceinline__ MfmaJob find_job(const MfmaLaunch &L, int tile) {
    if (L.table == nullptr) return L.one;
    const int at = ((const int __attribute__((address_space(4))) *)(uintptr_t)L.tile_jobs)[tile / L.row_tiles];
    const uniform_u64_ptr rec = (uniform_u64_ptr)(uintptr_t)L.table + 7 * at;
    MfmaJob job;
    job.vals = (const uint8_t *)rec[0];
    job.scales = (const uint8_t *)rec[1];
    job.biases = (const uint8_t *)rec[2];
    job.planes = (const uint16_t *)rec[3];
    job.y = (float *)rec[4];
    job.tokens = (int)(uint32_t)rec[5];
    job.rows = (int)(rec[5] >> 32);
    job.tile0 = (int)(uint32_t)rec[6];
    job.row_base = (int)(rec[6] >> 32);
    return job;
}

__device__ __forceinline__ float bf16_to_f32(uint32_t half) { return __uint_as_float(half << 16); }

// Eight nibbles -> eight fp16 values s (q - 8), in the column order 0,4,1,5,2,6,3,7.  A code's four bits land on
// mantissa bits 6..9 of 16.0, which makes 16 + q; `less` is -24 s.
__device__ __forceinline__ f16x8 weights_to_f16(uint32_t w, uint32_t mask, uint32_t sixteen, f16x2 s, f16x2 less) {
    auto pair = [&](uint32_t shifted) {
        return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, (shifted & mask) | sixteen), s, less));
    };
    const u32x4 r = {pair(w << 6), pair(w << 2), pair(w >> 2), pair(w >> 6)};
    return __builtin_bit_cast(f16x8, r);
}

__device__ __forceinline__ uint32_t f32_to_bf16_rne(float v) {
    const uint32_t bits = __float_as_uint(v);
    return (bits + 0x7FFFu + ((bits >> 16) & 1u)) >> 16;
}

// v = hi + mid + lo, each a bf16 (bit patterns in the low halves)
__device__ __forceinline__ void split3(float v, uint32_t &h, uint32_t &m, uint32_t &l) {
    h = f32_to_bf16_rne(v);
    const float r1 = v - bf16_to_f32(h);
    m = f32_to_bf16_rne(r1);
    const float r2 = r1 - bf16_to_f32(m);
    l = f32_to_bf16_rne(r2);
}

// The first eight bf16 of a row of fewer than eight, zeros past its end.
__device__ __forceinline__ u32x4 load_short(global_u16_ptr row, int ngrp) {
    u32x4 v = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 8; ++j)
        if (j < ngrp) v[j >> 1] |= (uint32_t)row[j] << (16 * (j & 1));
    return v;
}

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_max(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t pk_min(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t pk_less_one(uint32_t a) {            // zeros wrap to 0xffff
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) - (u16x2){1, 1}));
}

// The codes and the scale bits of a lane's two rows for one chunk of scale groups.
struct Weights { u32x4 w[CH][2]; uint32_t s[CH][2]; };

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2), amdgpu_num_vgpr(256)))
void q4_mfma_kernel(const MfmaLaunch L) {
    __shared__ __attribute__((aligned(16))) uint8_t stage[LDS_BYTES];
    __shared__ int s_down[TM];                     // per token: exponent of the power of two that undoes the split's scaling
    __shared__ int s_windows[4];
    __shared__ uint32_t s_row[TM];                 // per token: its row of the planes

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;

    // Workgroups go round the eight partitions of the device in turn; a partition takes one run of consecutive tiles of 64
    // tokens, so that the tiles of one weight matrix, or of one expert, meet in one partition's cache, and then one of the
    // tiles of 32: no partition is left with the longer tiles, and the shorter ones fill the end
    // (all tiles in one run each: grouped prefill of 256 tokens over 128 experts 225 -> 234 us, 512 over 32 79 -> 82; one
    // matrix of 65500 x 2816, 96 tokens, 80 -> 86).
    int wide_tiles = L.wide_tiles, narrow_tiles = L.narrow_tiles;
    if (L.table) {
        const int __attribute__((address_space(4))) *counts = (const int __attribute__((address_space(4))) *)(uintptr_t)L.tiles_dev;
        wide_tiles = counts[0];
        narrow_tiles = counts[1];
    }
    const int wide_run = (wide_tiles + 7) >> 3, narrow_run = (narrow_tiles + 7) >> 3;
    const int part = (int)(blockIdx.x & 7), turn = (int)(blockIdx.x >> 3);
    const bool first = turn < wide_run;
    const int nth = first ? part * wide_run + turn : part * narrow_run + turn - wide_run;
    if (nth >= (first ? wide_tiles : narrow_tiles) || turn >= wide_run + narrow_run) return;  // uniform: the whole workgroup leaves
    const MfmaJob job = find_job(L, first ? nth : wide_tiles + nth);
    const int C = L.cols, ngrp = C >> 6;
    // Blocks of tokens: in a table as many of 64 as hold more than 32, and one of 32 for the rest.
    const int wide_blocks = L.table ? (job.tokens + 31) >> 6 : L.wide_blocks;
    int tok0, row_tile;
    if (first) {
        const int t = nth - job.tile0;
        row_tile = t / wide_blocks;
        tok0 = (t - row_tile * wide_blocks) * TM;
    } else if (L.table) {
        row_tile = nth % L.row_tiles;
        tok0 = wide_blocks * TM;
    } else {
        row_tile = nth / L.narrow_blocks;
        tok0 = wide_blocks * TM + (nth - row_tile * L.narrow_blocks) * (TM / 2);
    }
    const int row0 = row_tile * MFMA_TN + wave * 64;
    const int tm = first ? TM : TM / 2;
    const int toks_here = job.tokens - tok0 < tm ? job.tokens - tok0 : tm;
    const bool wide = toks_here > 32;               // both token blocks hold tokens
    const bool live = row0 < job.rows;              // this wave has rows; the others only help to stage

    // Token t of the job is row (tok0 + t) of the planes, or, with a map, row
    // row_map[row_base + tok0 + t] / map_divisor (the grouped MoE gather); tokens past the end repeat the last one.
    if (tid < TM) {
        const int tc = tid < toks_here ? tid : toks_here - 1;
        s_row[tid] = L.row_map ? (uint32_t)(L.row_map[job.row_base + tok0 + tc] / L.map_divisor) : (uint32_t)(tok0 + tc);
    }
    __syncthreads();
    const global_u8_ptr plane0 = uniform_address((global_u8_ptr)(uintptr_t)job.planes);
    const global_u8_ptr plane1 = plane0 + 2 * L.plane_stride, notes = plane0 + 4 * L.plane_stride;

    // Staging geometry of this lane: load i of a wave brings the eight token rows from (i * ROW_WAVES + wave) * 8 on;
    // which piece of its row a lane fetches follows from the place that the load will put it in.
    uint32_t x_src[XT];                          // byte offsets below 2^32
#pragma unroll
    for (int i = 0; i < XT; ++i) {
        const int r = (i * ROW_WAVES + wave) * 8 + (lane >> 3);
        const int piece = (lane & 7) ^ place_mask(r);
        x_src[i] = s_row[r] * (uint32_t)(2 * C) + (uint32_t)piece * 16u;
    }

    // rows of this lane, clamped to the matrix
    uint32_t row[2];
    global_u16_ptr scales[2];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
        const int r = row0 + nb * 32 + l32;
        row[nb] = (uint32_t)(r < job.rows ? r : job.rows - 1);
        scales[nb] = (global_u16_ptr)(uintptr_t)job.scales + (size_t)row[nb] * (size_t)ngrp;
    }
    // codes of the wave's rows: load j of a chunk brings rows j * 64 / PIECES .., clamped to the matrix
    const int rows_left = live ? job.rows - row0 : 1;
    const int row_base = live ? row0 : 0;           // waves without rows fetch the first row and use nothing
    const global_u8_ptr codes = uniform_address((global_u8_ptr)(uintptr_t)job.vals + (size_t)row_base * (size_t)(C >> 1));
    const global_u8_ptr scale_rows = uniform_address((global_u8_ptr)(uintptr_t)job.scales + (size_t)row_base * (size_t)(2 * ngrp));

    // Everything staged goes from memory into LDS without passing through registers, so that a wave's loads complete
    // in the order they were sent in and a wait can leave the younger ones in flight (meet(), not __syncthreads, which
    // waits for all of them: 33 tokens against 8192 x 2816 44.7 -> 39.5 us, grouped prefill of 2048 tokens 611 -> 602).
    auto issue_x = [&](int it) {
        uint8_t *const x = stage + (it & 1) * STAGE_BYTES + wave * 1024;
        uint32_t at = (uint32_t)it * 128u;
        asm volatile("" : "+s"(at));                 // addresses are made here, not kept in registers through the loops
#pragma unroll
        for (int i = 0; i < XT; ++i) {
            if (i * ROW_WAVES * 8 >= 32 && !wide) break;
            uint8_t *const to = x + i * (ROW_WAVES * 1024);
            load_to_lds<16>(plane0, x_src[i] + at, to);
            load_to_lds<16>(plane1, x_src[i] + at, to + TM * 128);
        }
    };
    constexpr int CHUNK_LOADS = WT + CH;
    auto issue_weights = [&](int it) {               // the chunk that starts with group `it`
        const uint32_t at = (uint32_t)it * 32u, last = (uint32_t)ngrp * 32u - 16u;
        uint32_t lane_row = (uint32_t)lane / PIECES;
        uint32_t scale_at = (uint32_t)(lane < rows_left ? lane : rows_left - 1) * (uint32_t)(2 * ngrp);
        asm volatile("" : "+v"(lane_row), "+v"(scale_at));
#pragma unroll
        for (int j = 0; j < WT; ++j) {
            uint32_t r = j * (64 / PIECES) + lane_row;
            const uint32_t piece = ((uint32_t)lane & (PIECES - 1)) ^ (uint32_t)place_mask((int)r);
            uint32_t byte = at + piece * 16u;
            byte = byte < last ? byte : last;
            r = r < (uint32_t)rows_left ? r : (uint32_t)rows_left - 1u;
            load_to_lds<16>(codes, __umul24(r, (uint32_t)(C >> 1)) + byte, stage + W_OFF + wave * W_BYTES + j * 1024);
        }
#pragma unroll
        for (int gi = 0; gi < CH; ++gi) {
            const int g = it + gi;
            load_to_lds<2>(scale_rows, scale_at + 2u * (uint32_t)(g < ngrp ? g : ngrp - 1), stage + S_OFF + wave * S_BYTES + gi * 256);
        }
    };
    typedef const u32x4 __attribute__((address_space(3))) *lds_u128_ptr;
    typedef const uint32_t __attribute__((address_space(3))) *lds_u32_ptr;
    auto take_weights = [&](Weights &r) {     // and leave their place to the next chunk
        const lds_u128_ptr w = (lds_u128_ptr)(stage + W_OFF + wave * W_BYTES);
        const lds_u32_ptr sc = (lds_u32_ptr)(stage + S_OFF + wave * S_BYTES);
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            const int at = (nb * 32 + l32) * PIECES, turn = place_mask(nb * 32 + l32);
#pragma unroll
            for (int gi = 0; gi < CH; ++gi) {
                r.w[gi][nb] = w[at + ((gi * 2 + half) ^ turn)];
                r.s[gi][nb] = sc[gi * 64 + nb * 32 + l32];
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };

    // What the bias pass needs is sent for before the first planes and codes, whose arrival nobody has to wait for there.
    // The group sums go to LDS once for all waves, in 16-byte pieces of a token's contiguous 96: read by every wave for
    // itself, 32 tokens a load, they were more than half of the cache lines that a tile's start asks for.
    const int blocks = padded_groups(ngrp) >> 4;
    auto issue_sums = [&](int first) {              // blocks first .. first + SUM_BLOCKS - 1
        for (int i = wave; i < 6 * SUM_BLOCKS; i += ROW_WAVES) {
            const int block = i / 6;
            if (first + block >= blocks) break;     // uniform over the wave
            const int piece = (i - 6 * block) * 64 + lane, token = piece / 6;
            load_to_lds<16>(notes, s_row[token] * (uint32_t)(2 * C) + (uint32_t)(16 + (first + block) * 96 + (piece - 6 * token) * 16),
                            stage + sum_place(block) + (i - 6 * block) * 1024);
        }
    };
    global_u16_ptr biases[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
        biases[k] = (global_u16_ptr)(uintptr_t)(job.biases ? job.biases : job.scales) + (size_t)row[k] * (size_t)ngrp;
    struct Eights { u32x4 s[2], b[2]; };            // sixteen groups, eight per lane half
    auto fetch = [&](int block, Eights &e) {
        const int first = eight_start(2 * block + half, ngrp);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            e.s[k] = *(global_u128_any_ptr)(scales[k] + first);
            e.b[k] = *(global_u128_any_ptr)(biases[k] + first);
        }
    };
    constexpr int AHEAD = SUM_BLOCKS;
    issue_sums(0);
    int my_down = 0;
    if (tid < TM) my_down = *(global_i32_ptr)(notes + (size_t)s_row[tid] * (size_t)(2 * C));
    Eights e[AHEAD];
    if (ngrp >= 8) {
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) fetch(j < blocks ? j : blocks - 1, e[j]);
    } else {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            e[0].s[k] = load_short(scales[k], ngrp);
            e[0].b[k] = load_short(biases[k], ngrp);
        }
#pragma unroll
        for (int j = 1; j < AHEAD; ++j) e[j] = e[0];
    }
    wait_loads<0>();
    // the compiler's own wait for these stands here, where it is none
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
#pragma unroll
        for (int k = 0; k < 2; ++k) asm volatile("" : "+v"(e[j].s[k]), "+v"(e[j].b[k]));
    asm volatile("" : "+v"(my_down));
    meet();
    issue_weights(0);
    issue_x(0);

    // ---- bias term of the tile, acc[tok][row] = sum_g (b[row][g] + 8 s[row][g]) * X[tok][g], and the rows' exponents
    const f32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    f32x16 acc[2][2] = {{zero, zero}, {zero, zero}};
    int top[2] = {0, 0};                            // row block nb: the scales of this lane's row are below 2^top[nb]
    int windows = 1;
    auto more_sums = [&](int first) {               // the workgroup is done with the blocks in LDS: the next ones
        meet();
        issue_sums(first);
        wait_loads<0>();
        meet();
    };
    if (!live)                                      // the other waves meet here
        for (int first = SUM_BLOCKS; first < blocks; first += SUM_BLOCKS) more_sums(first);
    if (live) {
        const uint32_t keep = job.biases ? 0xffffffffu : 0u;        // without biases the scales stand in, masked
        f32x16 tb[2][2] = {{zero, zero}, {zero, zero}}, ts[2][2] = {{zero, zero}, {zero, zero}};
        uint32_t s_max[2] = {0, 0}, b_max[2] = {0, 0}, s_min[2] = {0xffffffffu, 0xffffffffu};
        typedef const u32x4 __attribute__((address_space(3))) *sums_ptr;
        auto add_block = [&](int slot, Eights &c) {
            u32x4 x[3][2];
            const sums_ptr at = (sums_ptr)(stage + sum_place(slot) + l32 * 96 + half * 16);
#pragma unroll
            for (int plane = 0; plane < 3; ++plane)
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) x[plane][mb] = at[mb * (32 * 6) + plane * 2];
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                for (int j = 0; j < 4; ++j) c.b[nb][j] &= keep;
#pragma unroll
            for (int plane = 0; plane < 3; ++plane)
#pragma unroll
                for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                    for (int nb = 0; nb < 2; ++nb) {
                        const bf16x8 a = __builtin_bit_cast(bf16x8, x[plane][mb]);
                        tb[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(bf16x8, c.b[nb]),
                                                                             tb[mb][nb], 0, 0, 0);
                        ts[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(bf16x8, c.s[nb]),
                                                                             ts[mb][nb], 0, 0, 0);
                    }
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t sa = c.s[nb][j] & 0x7fff7fffu;
                    s_max[nb] = pk_max(s_max[nb], sa);
                    s_min[nb] = pk_min(s_min[nb], pk_less_one(sa));
                    b_max[nb] = pk_max(b_max[nb], c.b[nb][j] & 0x7fff7fffu);
                }
        };
        for (int block = 0; block < blocks; block += AHEAD) {
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) {
                if (block + j >= blocks) break;
                if (j == 0 && block > 0) more_sums(block);
                add_block(j, e[j]);
                if (block + j + AHEAD < blocks) fetch(block + j + AHEAD, e[j]);
            }
        }
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            const uint32_t s2 = pk_max(s_max[nb], (uint32_t)__shfl_xor((int)s_max[nb], 32, 64));
            const uint32_t b2 = pk_max(b_max[nb], (uint32_t)__shfl_xor((int)b_max[nb], 32, 64));
            const uint32_t m2 = pk_min(s_min[nb], (uint32_t)__shfl_xor((int)s_min[nb], 32, 64));
            const uint32_t sm = (s2 & 0xffffu) > (s2 >> 16) ? (s2 & 0xffffu) : (s2 >> 16);
            const uint32_t bm = (b2 & 0xffffu) > (b2 >> 16) ? (b2 & 0xffffu) : (b2 >> 16);
            const uint32_t lowest = ((m2 & 0xffffu) < (m2 >> 16) ? (m2 & 0xffffu) : (m2 >> 16)) + 1u;
            const float big_s = bf16_to_f32(sm), big_b = bf16_to_f32(bm) * 0.125f;
            top[nb] = __builtin_amdgcn_frexp_expf(big_s > big_b ? big_s : big_b);      // 0 for 0, infinities and NaN
            if (lowest <= 0x7f7fu) {
                const int span = top[nb] - __builtin_amdgcn_frexp_expf(bf16_to_f32(lowest));
                const int need = span < 0 ? 1 : span / WINDOW + 1;
                windows = need > windows ? need : windows;
            }
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[mb][nb][i] = __builtin_fmaf(8.0f, ts[mb][nb][i], tb[mb][nb][i]);
        }
        windows = windows > MAX_WINDOWS ? MAX_WINDOWS : windows;
        if (__ballot(windows > 1)) {
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int other = __shfl_xor(windows, d, 64);
                windows = windows > other ? windows : other;
            }
        }
    }
    if (lane == 0) s_windows[wave] = windows;
    if (tid < TM) s_down[tid] = my_down;
    wait_loads<0>();
    __syncthreads();                                // the first stage and chunk are there as well
    windows = s_windows[0];
#pragma unroll
    for (int w = 1; w < 4; ++w) windows = windows > s_windows[w] ? windows : s_windows[w];
    windows = __builtin_amdgcn_readfirstlane(windows);
    // the main loop works on s 2^(11 - top) and x 2^-down: the bias term joins it at that scale
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int down = s_down[mb * 32 + (i >> 2) * 8 + half * 4 + (i & 3)];
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
                acc[mb][nb][i] = __builtin_amdgcn_ldexpf(acc[mb][nb][i], WEIGHT_TOP - top[nb] - down);
        }

    const int mix = place_mask(l32);             // rows 32 apart share it
    uint32_t code_mask, sixteen;                    // opaque, so that (w & mask) | 16.0 stays one instruction
    asm("s_mov_b32 %0, 0x03C003C0" : "=s"(code_mask));
    asm("v_mov_b32 %0, 0x4C004C00" : "=v"(sixteen));
    int raise[2];                                   // row block nb: the power of two that its scales are brought up by

    // The wave's walk over the columns for MB blocks of 32 tokens, in steps of 16 columns: while the matrix
    // cores work on a step, the operands of the next one are read and converted (left to itself the compiler reads
    // a whole group ahead and spills).  The workgroup meets before the last step of a group: its planes are then in
    // everybody's registers, so their place takes the group after the next one.
    auto walk = [&](auto blocks) {
        constexpr int MB = decltype(blocks)::value;
        constexpr int LAST = CH - 1;
        Weights now;
        f16x8 a[2][MB][X_PLANES], b[2][2];
        f16x2 s[2], less[2], s_next[2], less_next[2];
        auto read = [&](int it, int step, f16x8 (&to)[MB][X_PLANES]) {
            const lds_u128_ptr x = (lds_u128_ptr)(stage + (it & 1) * STAGE_BYTES + l32 * 128);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int plane = 0; plane < X_PLANES; ++plane)
                    to[mb][plane] = __builtin_bit_cast(
                        f16x8, x[plane * (TM * 8) + mb * (32 * 8) + ((half * 4 + step) ^ mix)]);
        };
        // Scales that the window does not bring into the WINDOW binades below 2^WEIGHT_TOP count as zero.
        auto scale = [&](const uint32_t (&bits)[2], f16x2 (&s)[2], f16x2 (&less)[2]) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
                const float value = bf16_to_f32(bits[nb]);
                const int place = __builtin_amdgcn_frexp_expf(value) + raise[nb];  // at most WEIGHT_TOP in this window
                float raised = __builtin_amdgcn_ldexpf(value, raise[nb]);
                const bool finite = __builtin_fabsf(value) < __builtin_inff();
                if (finite && (unsigned)(WEIGHT_TOP - place) >= (unsigned)WINDOW) raised = 0.0f;
                const _Float16 h = (_Float16)raised;
                const _Float16 l = (_Float16)-24.0f * h;
                s[nb] = f16x2{h, h};
                less[nb] = f16x2{l, l};
            }
        };
        auto convert = [&](const u32x4 (&w)[2], int step, f16x8 (&to)[2]) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) to[nb] = weights_to_f16(w[nb][step], code_mask, sixteen, s[nb], less[nb]);
        };
        auto multiply = [&](const f16x8 (&x)[MB][X_PLANES], const f16x8 (&w)[2]) {
#pragma unroll
            for (int plane = 0; plane < X_PLANES; ++plane)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int nb = 0; nb < 2; ++nb)
                        acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[mb][plane], w[nb], acc[mb][nb], 0, 0, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, MB * X_PLANES, 0);      // LDS reads first, then one matrix
#pragma unroll
            for (int k = 0; k < 4 * MB; ++k) {                                  // instruction and its share of the rest
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 24 / (4 * MB) + 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        // made here and not sunk to the use behind the workgroup's meeting, where nothing covers it
        auto pin = [](auto (&values)[2]) {
#pragma unroll
            for (int k = 0; k < 2; ++k) asm volatile("" : "+v"(values[k]));
        };
        take_weights(now);
        if (CH < ngrp) issue_weights(CH);
        read(0, 0, a[0]);
        scale(now.s[0], s, less);
        convert(now.w[0], 0, b[0]);
        __builtin_amdgcn_sched_barrier(0);
        for (int it0 = 0; it0 < ngrp; it0 += CH) {
#pragma unroll
            for (int gi = 0; gi < CH; ++gi) {
                const int it = it0 + gi;
#pragma unroll
                for (int step = 0; step < 3; ++step) {
                    read(it, step + 1, a[(step + 1) & 1]);
                    convert(now.w[gi], step + 1, b[(step + 1) & 1]);
                    if (step == 1 && gi < LAST) {
                        scale(now.s[gi < LAST ? gi + 1 : 0], s_next, less_next);
                        pin(s_next); pin(less_next);
                    }
                    multiply(a[step & 1], b[step & 1]);
                }
                pin(b[1]);
                // the next planes were sent for before the chunk that may still be on its way
                if (gi == 0 && it0 + CH < ngrp) wait_loads<CHUNK_LOADS>(); else wait_loads<0>();
                meet();
                if (it + 2 < ngrp) issue_x(it + 2);
                if (gi == CH - 1) {
                    take_weights(now);
                    if (it + 1 + CH < ngrp) issue_weights(it + 1 + CH);
                }
                // after the last group these are stale and unused
                if (gi == LAST) scale(now.s[0], s_next, less_next);
#pragma unroll
                for (int nb = 0; nb < 2; ++nb) { s[nb] = s_next[nb]; less[nb] = less_next[nb]; }
                read(it + 1, 0, a[0]);
                convert(now.w[gi == LAST ? 0 : gi + 1], 0, b[0]);
                multiply(a[1], b[1]);
                if (it + 1 >= ngrp) break;
            }
        }
    };
    // A wave without rows helps to stage.
    auto stage_only = [&]() {
        for (int it = 0; it < ngrp; ++it) {
            wait_loads<0>();
            meet();
            if (it + 2 < ngrp) issue_x(it + 2);
        }
    };
    for (int window = 0;;) {
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) raise[nb] = WEIGHT_TOP - top[nb] + WINDOW * window;
        // ---- main loop: acc += s (q - 8) x
        if (ngrp > 1) issue_x(1);
        if (!live) stage_only();
        else if (wide) walk(std::integral_constant<int, 2>{});
        else walk(std::integral_constant<int, 1>{});

        if (live) {
            // WHOLE: the wave's block of rows and tokens is inside the output and new, and nothing is asked about a value (with a
            // test for each the stores took 6700 to 8000 clocks of a tile's 50000 to 130000, without 4000 to 5000)
            auto store = [&](auto all, int mb) {
                constexpr bool WHOLE = decltype(all)::value;
                int tok_base = mb * 32 + half * 4;
                asm volatile("" : "+v"(tok_base));      // the output addresses are made here, not kept through the loop
                global_f32_out line = (global_f32_out)(uintptr_t)job.y + (size_t)(tok0 + tok_base) * job.rows + row0 + l32;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int tok = tok_base + (i >> 2) * 8 + (i & 3);
                    const int down = s_down[tok];
#pragma unroll
                    for (int nb = 0; nb < 2; ++nb) {
                        if (WHOLE || (tok < toks_here && row0 + nb * 32 + l32 < job.rows)) {
                            float v = __builtin_amdgcn_ldexpf(mb ? acc[1][nb][i] : acc[0][nb][i], down - raise[nb]);
                            if (!WHOLE && window != 0) v = line[nb * 32] + v;
                            line[nb * 32] = v;
                        }
                    }
                    line += (size_t)job.rows * ((i & 3) == 3 ? 5 : 1);
                }
            };
            const bool rows_inside = row0 + 64 <= job.rows && window == 0;
            if (rows_inside && toks_here >= 32) store(std::true_type{}, 0); else store(std::false_type{}, 0);
            if (rows_inside && toks_here == TM) store(std::true_type{}, 1);
            else if (wide) store(std::false_type{}, 1);
        }
        if (++window >= windows) break;             // uniform over the workgroup
        __syncthreads();                            // the last group has been read by every wave
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) acc[mb][nb] = zero;
        wait_loads<0>();
        issue_weights(0);
        issue_x(0);
        wait_loads<0>();
        __syncthreads();
    }
}

// fp32 rows -> two fp16 planes of the row scaled by a power of two (columns permuted inside every run of eight, see
// the top of the file) and the row's notes in a third plane: the exponent that undoes the scaling and the
// per-64-column sums of the unscaled values in three bf16 planes.  Row r of the output is row row_map[r] /
// map_divisor of the input when a map is given (the grouped MoE gather).  ROW_WAVES waves per row, because the scale
// needs the row's largest magnitude: a whole workgroup, or one wave where a row is short enough for that.
// With GATED the value split is gelu_tanh(gate) * x (the expert activation, reference gemma4_text.c:8749-9137
// "down input"), so the activations never make a round trip through memory in fp32.
constexpr int SPLIT_MAX_ITEMS = 4;          // eight columns per item and thread: rows of up to 2048 columns per wave

template <bool GATED, int ROW_WAVES>
__global__ __launch_bounds__(256) void x_split_kernel(const float *__restrict__ x, const float *__restrict__ gate,
                                                      const int *__restrict__ row_map, int map_divisor, int x_stride,
                                                      int rows, int cols, uint16_t *__restrict__ planes,
                                                      size_t plane_stride, uint32_t *__restrict__ clear, int clear_words) {
    __shared__ uint32_t wave_top[4];
    constexpr int THREADS = 64 * ROW_WAVES;
    const int tid = threadIdx.x & (THREADS - 1);
    const int row = ROW_WAVES == 4 ? (int)blockIdx.x : (int)(blockIdx.x * 4 + (threadIdx.x >> 6));
    for (int i = blockIdx.x * 256 + threadIdx.x; i < clear_words; i += gridDim.x * 256) clear[i] = 0u;
    if (row >= rows) return;                        // whole waves, and only where no barrier follows
    const int src_row = row_map ? row_map[row] / map_divisor : row;
    float v[SPLIT_MAX_ITEMS][8];
    uint32_t top = 0u;                              // largest magnitude as a bit pattern: a NaN or an infinity wins it
#pragma unroll
    for (int it = 0; it < SPLIT_MAX_ITEMS; ++it) {
        const int c0 = (it * THREADS + tid) * 8;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[it][j] = 0.0f;
        if (c0 < cols) {
            const float4 *src = reinterpret_cast<const float4 *>(x + (size_t)src_row * x_stride + c0);
            const float4 a = src[0], b = src[1];
            v[it][0] = a.x; v[it][1] = a.y; v[it][2] = a.z; v[it][3] = a.w;
            v[it][4] = b.x; v[it][5] = b.y; v[it][6] = b.z; v[it][7] = b.w;
            if (GATED) {
                const float4 *gsrc = reinterpret_cast<const float4 *>(gate + (size_t)src_row * x_stride + c0);
                const float4 ga = gsrc[0], gb = gsrc[1];
                const float gv[8] = {ga.x, ga.y, ga.z, ga.w, gb.x, gb.y, gb.z, gb.w};
#pragma unroll
                for (int j = 0; j < 8; ++j) v[it][j] = det_gelu_tanh(gv[j]) * v[it][j];
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t mag = __float_as_uint(v[it][j]) & 0x7fffffffu;
                top = top > mag ? top : mag;
            }
        }
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t other = (uint32_t)__shfl_xor((int)top, d, 64);
        top = top > other ? top : other;
    }
    if (ROW_WAVES == 4) {
        if ((threadIdx.x & 63) == 0) wave_top[threadIdx.x >> 6] = top;
        __syncthreads();
        top = wave_top[0];
#pragma unroll
        for (int w = 1; w < 4; ++w) top = top > wave_top[w] ? top : wave_top[w];
    }
    // top in [2^E, 2^(E+1)) -> x * 2^(13 - E) in [2^13, 2^14); rows of zeros or tiny values are pinned
    int eb = (int)(top >> 23);
    eb = eb < 14 ? 14 : (eb > 253 ? 253 : eb);
    const float up = __uint_as_float((uint32_t)(267 - eb) << 23);          // 2^(13 - E)
    uint16_t *const notes = planes + 2 * plane_stride + (size_t)row * cols;
    const int ngrp = cols >> 6, padded = padded_groups(ngrp);
    if (tid == 0) *reinterpret_cast<int *>(notes) = eb - 140;              // E - 13
    // the last eight groups sit at the end of theirs (eight_start): entries that stand for no group of their own are zero
    const int tail = ((ngrp + 7) >> 3) - 1, shift = ngrp > 8 ? 8 * tail - (ngrp - 8) : 0;
    for (int at = 8 * tail + tid; at < padded; at += THREADS)
        if (at < 8 * tail + shift || at >= ngrp + shift)
#pragma unroll
            for (int plane = 0; plane < 3; ++plane) notes[sum_entry(at, plane)] = 0;
#pragma unroll
    for (int it = 0; it < SPLIT_MAX_ITEMS; ++it) {
        const int c0 = (it * THREADS + tid) * 8;
        const bool inside = c0 < cols;
        uint32_t hi[4], lo[4];
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float scaled = v[it][j] * up;
            const _Float16 h = (_Float16)scaled;
            const _Float16 l = (_Float16)(scaled - (float)h);
            const uint32_t hb = __builtin_bit_cast(uint16_t, h), lb = __builtin_bit_cast(uint16_t, l);
            const int k = j & 3;                           // dword k holds columns k (low half) and k + 4 (high half)
            if (j & 4) { hi[k] |= hb << 16; lo[k] |= lb << 16; }
            else { hi[k] = hb; lo[k] = lb; }
            sum += v[it][j];
        }
        // eight lanes cover one 64-column group
        sum += __shfl_xor(sum, 1, 64);
        sum += __shfl_xor(sum, 2, 64);
        sum += __shfl_xor(sum, 4, 64);
        if (inside) {
            uint16_t *dst = planes + (size_t)row * cols + c0;
            *reinterpret_cast<uint4 *>(dst) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
            *reinterpret_cast<uint4 *>(dst + plane_stride) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
            if ((tid & 7) == 0) {
                uint32_t h, m, l;
                split3(sum, h, m, l);
                const int g = c0 >> 6;
                uint16_t *const at = notes + sum_entry(g < 8 * tail ? g : g + shift, 0);
                at[0] = (uint16_t)h; at[16] = (uint16_t)m; at[32] = (uint16_t)l;
            }
        }
    }
}

}  // namespace

int q4_mfma_launch(const MfmaLaunch &launch, hipStream_t stream) {
    MfmaLaunch L = launch;
    if (L.cols < 64 || (L.cols & 63)) return -1;
    int turns;                                  // of the eight partitions
    if (L.table == nullptr) {                   // one job: the tiling is chosen here
        const int halves = (L.one.tokens + TM / 2 - 1) / (TM / 2), row_tiles = (L.one.rows + MFMA_TN - 1) / MFMA_TN;
        // Tiles of half the tokens where each still finds a compute unit of its own: half the matrix work per step of a
        // walk that is bound by its waits (4096 x 4096, 64 tokens: 67 us in 64-token tiles, 54 in these).  Else tiles of 64
        // and, for what is left, one of 32; but between two and three halves per compute unit no unit gets two tiles of 64
        // while others have one: as many of those as there are units, then tiles of 32, as long as all of them are at work
        // at once (2816 columns, us with the cap and without: 16384 rows, 333 tokens 74.6 and 79.1; 2816, 1600 74.7 and
        // 83.3; 25600, 224 77.2 and 80.5; with four tiles left over for a third turn, 33000, 150, 88.3 and 79.1).
        const long long work = (long long)halves * row_tiles;
        L.wide_blocks = halves / 2;
        if (work <= CUS) L.wide_blocks = 0;
        else if (work > 2 * CUS && work <= 3 * CUS) {
            const int cap = CUS / row_tiles;
            if (cap < L.wide_blocks && work - (long long)cap * row_tiles <= 2 * CUS) L.wide_blocks = cap;
        }
        L.narrow_blocks = halves - 2 * L.wide_blocks;
        L.one.tile0 = 0;
        L.row_tiles = row_tiles;
        if (L.one.tokens < 1 || L.one.rows < 1 || work > (1 << 30)) return -1;
        L.wide_tiles = L.wide_blocks * row_tiles;
        L.narrow_tiles = L.narrow_blocks * row_tiles;
        turns = (L.wide_tiles + 7) / 8 + (L.narrow_tiles + 7) / 8;
        if (L.wide_blocks && L.narrow_blocks)
            note_kernel("q4_mfma_kernel, %d blocks of %d tokens and %d of %d", L.wide_blocks, TM, L.narrow_blocks, TM / 2);
        else
            note_kernel("q4_mfma_kernel, tiles of %d tokens", L.wide_blocks ? TM : TM / 2);
    } else {
        if (L.most_tiles < 1 || L.row_tiles < 1 || !L.tile_jobs || !L.tiles_dev) return -1;
        turns = (L.most_tiles + 14) / 8;        // both runs, each rounded up
        note_kernel("q4_mfma_kernel, blocks of %d and of %d tokens by table", TM, TM / 2);
    }
    if (3 * (unsigned long long)L.plane_stride >= (1ull << 32)) return -1;      // 32-bit byte offsets inside a plane
    if (L.row_map && L.map_divisor < 1) return -1;
    hipLaunchKernelGGL(q4_mfma_kernel, dim3(turns * 8), dim3(256), 0, stream, L);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int x_split_launch(const float *x, const float *gate, const int *row_map, int map_divisor, int x_stride, int rows,
                   int cols, uint16_t *planes, size_t plane_stride, uint32_t *clear, int clear_words, hipStream_t stream) {
    if (rows < 1 || cols < 64 || (cols & 63) || cols > SPLIT_MAX_ITEMS * 256 * 8) return -1;
    // A wave per row leaves no thread of a short row idle (gelu_tanh(gate) * up, 16384 rows of 704: 50 -> 41 us), a
    // workgroup per row shortens the chain of a call with few rows (900 rows of 704: 5.9 against 7.2 us).
    const bool one_wave = cols <= SPLIT_MAX_ITEMS * 64 * 8 && rows >= 4096;
    const dim3 grid(one_wave ? (rows + 3) / 4 : rows);
    auto kernel = gate ? (one_wave ? x_split_kernel<true, 1> : x_split_kernel<true, 4>)
                       : (one_wave ? x_split_kernel<false, 1> : x_split_kernel<false, 4>);
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, x, gate, row_map, map_divisor, x_stride, rows, cols, planes,
                       plane_stride, clear, clear_words);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace mi355
