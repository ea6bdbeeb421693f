// Prefill-sized NVFP4 matmul on the MFMA units (tolerance class).
//
// reference src/nvfp4.c:228-256 computes, per output row, sum_c w_c * x_c with
// w_c = e2m1(code) * (e4m3(scale) * weight_global) and x_c the quantised and
// dequantised activation e2m1(code) * (e4m3(scale) / input_global), in its
// 32-chain order.  With hundreds of tokens the work is a dense contraction.
// Both operands factor into a part that is exact in fp16,
//     e2m1(code) * e4m3(block scale)        (two times four significant bits,
//                                            between 2^-10 and 2688),
// and a per-tensor fp32 factor, so the matrix cores see exact operands, the
// products are exact in fp32 and only the order of the fp32 additions (and the
// two per-tensor factors, applied once at the end) differs from the reference.
//
// Tiling.  A wave computes 64 tokens x 64 weight rows as 2 x 2 blocks of
// v_mfma_f32_32x32x16_f16.  The codes of its rows go through its own piece of
// LDS, 128 bytes of a row at a time, to its registers and are decoded there:
// one conversion and one packed multiply per pair, in the shadow of the matrix
// instructions, and a quarter of the LDS reads that decoded weights would take
// (with both operands read as 16-bit values the reads, 128 bytes per clock and
// compute unit, took as long as the matrix work).  The token planes are staged
// in LDS, 64 columns per stage, two stages.  Eight waves per workgroup, two per
// SIMD: RW row blocks of 64 times 8 / RW parts of the columns, which meet in LDS
// in part order; so a launch of 256 workgroups needs no partial sums in memory
// and no second kernel.  Smaller ones are also split over workgroups, whose
// partials a second kernel adds in split order.
//
// 8192 x 8192, 256 tokens: 64.2 -> 45.7 us with the activation pass (48.1 with a wait for all loads at every stage, by
// __syncthreads and by the compiler, see lds_load.h).
// Bound: lines from the cache to the compute unit (64 KB per stage of two rounds of matrix work, of which the planes
// are half), then the matrix cores.
#include "lds_load.h"
#include "mi355_internal.h"

#include <stddef.h>

#include <type_traits>

namespace mi355 {
namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef const uint8_t __attribute__((address_space(1))) *global_u8_ptr;
typedef float __attribute__((address_space(1))) *global_f32_out;
typedef const u32x4 __attribute__((address_space(3))) *lds_u128_ptr;
typedef const uint32_t __attribute__((address_space(3))) *lds_u32_ptr;

constexpr int TM = 64, KC = 64, CH = 4;        // tokens per workgroup; columns per stage; stages per chunk of codes
constexpr int FAR_COLS = 1 << 25;              // from here on the offsets inside a tile of 64 rows take 64 bits

template <int WAVES, int RW> struct Shape {
    static constexpr int KP = WAVES / RW;                            // parts of the columns
    static constexpr int TN = 64 * RW;
    static constexpr int X_BYTES = TM * 2 * KC;                      // one part's planes of one stage
    static constexpr int STAGE_BYTES = KP * X_BYTES;
    static constexpr int W_OFF = 2 * STAGE_BYTES, W_BYTES = 64 * 32 * CH;        // of one wave
    static constexpr int S_OFF = W_OFF + WAVES * W_BYTES, S_BYTES = 64 * 4 * 2 * CH;
    static constexpr int LDS_BYTES = S_OFF + WAVES * S_BYTES;
    static constexpr int XT = TM / (8 * RW);                         // plane loads per wave and stage: eight tokens each
    static constexpr int CODE_LOADS = 8;                             // per wave and chunk
    static_assert((KP - 1) * RW * 64 * 64 * 4 <= S_OFF, "the parts' sums reuse the staging memory");
};

struct Geometry {
    int m_tiles, n_tiles, chunks, chunks_per_split;                  // chunks of KC columns
};

// Piece p of a row lies at place p ^ place_mask(row): loads into LDS write 64 consecutive pieces, so rows cannot be
// padded, and this spreads the sixteen rows of a read phase over all banks.
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

// Whether the activation pass rejected its input: the launch's status word, or the OR of the pass's per-workgroup
// flags (every thread of the workgroup calls this; workgroup 0 then also publishes the outcome).
__device__ __forceinline__ bool rejected(const Fp4MfmaLaunch &L) {
    if (!L.flags) return *(const int __attribute__((address_space(4))) *)(uintptr_t)L.status != 0;
    int bad = 0;
    for (int i = threadIdx.x; i < L.nflags; i += blockDim.x) bad |= L.flags[i];
    const int any_bad = __syncthreads_or(bad);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *L.outcome = any_bad ? -1 : 0;
        if (L.outcome_copy) *L.outcome_copy = any_bad ? -1 : 0;
    }
    return any_bad != 0;
}

// Eight E2M1 codes times their block's scale, in column order.
__device__ __forceinline__ f16x8 weights_to_f16(uint32_t w, f16x2 s) {
    u32x4 r;
    r.x = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0)) * s));
    r.y = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1)) * s));
    r.z = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2)) * s));
    r.w = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3)) * s));
    return __builtin_bit_cast(f16x8, r);
}

template <int WAVES, int RW, bool FAR>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(2))) void fp4_mfma_kernel(const Fp4MfmaLaunch L, const Geometry G) {
    using S = Shape<WAVES, RW>;
    using Offset = typename std::conditional<FAR, uint64_t, uint32_t>::type;
    __shared__ __attribute__((aligned(16))) uint8_t stage[S::LDS_BYTES];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int part = wave / RW, wn = wave % RW;
    const int l32 = lane & 31, half = lane >> 5;

    // Workgroups go round the eight partitions of the device in turn; a partition takes one run of consecutive tiles,
    // token tiles fastest, so that the tiles of the same weight rows meet in one partition's cache.
    const int total = G.m_tiles * G.n_tiles * L.ksplit;
    const int run = (total + 7) >> 3;
    const int tile = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
    const bool present = (int)(blockIdx.x >> 3) < run && tile < total;
    if (!present) return;                           // uniform; workgroup 0 always has a tile
    const int mt = tile % G.m_tiles, nt = (tile / G.m_tiles) % G.n_tiles, split = tile / (G.m_tiles * G.n_tiles);
    const int tok0 = mt * TM, row0 = nt * S::TN + wn * 64;
    const int toks_here = L.tokens - tok0 < TM ? L.tokens - tok0 : TM;
    const bool wide = toks_here > 32;               // both token blocks hold tokens
    const bool live = row0 < L.rows;                // this wave has rows; the others only help to stage
    const int C = L.cols;

    // the split's columns, and the part's: `iterations` stages from first on, those from end on staged and unused
    const int split0 = split * G.chunks_per_split;
    const int split1 = split0 + G.chunks_per_split < G.chunks ? split0 + G.chunks_per_split : G.chunks;
    const int even = (split1 - split0 + S::KP - 1) / S::KP;
    const int iterations = even >= 4 * CH ? (even + CH - 1) / CH * CH : even;       // whole cache lines where it matters little
    const int first = split0 + part * iterations;
    const int end = first + iterations < split1 ? first + iterations : split1;
    const int last_chunk = G.chunks - 1;

    // load i of a wave brings the eight token rows from (i * RW + wn) * 8 on; which piece of its row a lane fetches
    // follows from the place that the load will put it in
    const global_u8_ptr plane = (global_u8_ptr)(uintptr_t)L.plane + (size_t)tok0 * (2 * (size_t)C);
    Offset x_src[S::XT];
#pragma unroll
    for (int i = 0; i < S::XT; ++i) {
        const int r = (i * RW + wn) * 8 + (lane >> 3);
        x_src[i] = (Offset)(r < toks_here ? r : toks_here - 1) * (2 * (Offset)C) + (uint32_t)((lane & 7) ^ place_mask(r)) * 16u;
    }
    const int rows_left = live ? L.rows - row0 : 1;
    const int row_base = live ? row0 : 0;           // waves without rows fetch the first row and use nothing
    const global_u8_ptr codes = (global_u8_ptr)(uintptr_t)L.packed + (size_t)row_base * (size_t)(C >> 1);
    const global_u8_ptr scale_rows = (global_u8_ptr)(uintptr_t)L.scales + (size_t)row_base * (size_t)(C >> 4);

    // Everything staged goes from memory into LDS without passing through registers, so that a wave's loads complete
    // in the order they were sent in and a wait can leave the younger ones in flight.
    auto issue_x = [&](int it) {
        const int g = first + it < G.chunks ? first + it : last_chunk;
        Offset at = (Offset)g * (2 * KC);
        asm volatile("" : "+s"(at));
        uint8_t *const x = stage + (it & 1) * S::STAGE_BYTES + part * S::X_BYTES + wn * 1024;
#pragma unroll
        for (int i = 0; i < S::XT; ++i) {
            if (i * RW * 8 >= 32 && !wide) break;
            load_to_lds<16>(plane, x_src[i] + at, x + i * (RW * 1024));
        }
    };
    // A row's scales of a chunk are 16 bytes.  They come in one load where addresses allow it: 64 rows are 64 cache
    // lines to look up however little of them is wanted, and eight loads of two bytes took longer than the matrix work.
    const bool whole_scales = ((uintptr_t)L.scales & 3) == 0 && G.chunks >= CH;
    auto issue_weights = [&](int it) {               // the chunk that starts with stage `it` of the part
        const uint32_t at = (uint32_t)(first + it) * 32u, last = (uint32_t)G.chunks * 32u - 16u;
        uint32_t lane_row = (uint32_t)lane >> 3;
        Offset scale_at = (Offset)(lane < rows_left ? lane : rows_left - 1) * (uint32_t)(C >> 4);
        asm volatile("" : "+v"(lane_row), "+v"(scale_at));   // addresses are made here, not kept in registers
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            uint32_t r = j * 8 + lane_row;
            uint32_t byte = at + (((uint32_t)lane & 7u) ^ (uint32_t)place_mask((int)r)) * 16u;
            byte = byte < last ? byte : last;
            r = r < (uint32_t)rows_left ? r : (uint32_t)rows_left - 1u;
            const Offset line = FAR ? (Offset)r * (uint32_t)(C >> 1) : (Offset)__umul24(r, (uint32_t)(C >> 1));
            load_to_lds<16>(codes, line + byte, stage + S::W_OFF + wave * S::W_BYTES + j * 1024);
        }
        if (whole_scales) {                          // a chunk's scales of a row at once, from the row's end backwards
            const uint32_t s_at = (uint32_t)(first + it) * 4u, s_last = (uint32_t)G.chunks * 4u - 16u;
            load_to_lds<16>(scale_rows, scale_at + (s_at < s_last ? s_at : s_last), stage + S::S_OFF + wave * S::S_BYTES);
            return;
        }
#pragma unroll
        for (int k = 0; k < 2 * CH; ++k) {           // the two scales of each half of each stage
            const int g = first + it + (k >> 1) < G.chunks ? first + it + (k >> 1) : last_chunk;
            load_to_lds<2>(scale_rows, scale_at + (uint32_t)(g * 4 + (k & 1) * 2), stage + S::S_OFF + wave * S::S_BYTES + k * 256);
        }
    };
    struct Weights { u32x4 w[CH][2]; uint32_t s[CH][2]; };
    auto take_weights = [&](int it, Weights &r) {    // and leave their place to the next chunk
        const lds_u128_ptr w = (lds_u128_ptr)(stage + S::W_OFF + wave * S::W_BYTES);
        const lds_u32_ptr sc = (lds_u32_ptr)(stage + S::S_OFF + wave * S::S_BYTES);
        const int beyond = first + it - (G.chunks - CH), back = beyond > 0 ? beyond : 0;     // stages fetched from before the chunk
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            const int at = (nb * 32 + l32) * 8, turn = place_mask(nb * 32 + l32);
#pragma unroll
            for (int gi = 0; gi < CH; ++gi) {
                r.w[gi][nb] = w[at + ((gi * 2 + half) ^ turn)];
                const int g = gi + back < CH ? gi + back : CH - 1;
                if (whole_scales) r.s[gi][nb] = sc[(nb * 32 + l32) * 4 + g];
                else r.s[gi][nb] = sc[(gi * 2 + half) * 64 + nb * 32 + l32];
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (whole_scales) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                for (int gi = 0; gi < CH; ++gi) r.s[gi][nb] >>= half * 16;
        }
    };

    const f32x16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    f32x16 acc[2][2] = {{zero, zero}, {zero, zero}};

    issue_weights(0);
    issue_x(0);
    wait_loads<0>();
    __syncthreads();
    if (iterations > 1) issue_x(1);

    // The two lane halves of an instruction take columns 32 h + 8 k .. + 7 of a stage, so that a lane's codes of a
    // stage are 16 consecutive bytes and its scales two.  While the matrix cores work on a step of 16 columns the
    // operands of the next one are read and decoded; the workgroup meets before the last step of a stage, when its
    // planes are in everybody's registers and their place can take the stage after the next one.
    if (live) {
        const int mix = place_mask(l32);             // rows 32 apart share it
        Weights now;
        f16x8 a[2][2], b[2][2];
        auto read = [&](int it, int step, f16x8 (&to)[2]) {
            const lds_u128_ptr x = (lds_u128_ptr)(stage + (it & 1) * S::STAGE_BYTES + part * S::X_BYTES + l32 * (2 * KC));
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) to[mb] = __builtin_bit_cast(f16x8, x[mb * (32 * 8) + ((half * 4 + step) ^ mix)]);
        };
        auto decode = [&](const u32x4 (&w)[2], const uint32_t (&bits)[2], int step, bool inside, f16x8 (&to)[2]) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
                const uint32_t pair = inside ? bits[nb] : 0u;
                const float scale = step < 2 ? __builtin_amdgcn_cvt_f32_fp8((int)pair, 0) : __builtin_amdgcn_cvt_f32_fp8((int)pair, 1);
                const _Float16 h = (_Float16)scale;
                to[nb] = weights_to_f16(w[nb][step], f16x2{h, h});
            }
        };
        auto multiply = [&](const f16x8 (&x)[2], const f16x8 (&w)[2]) {
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int nb = 0; nb < 2; ++nb)
                    acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[mb], w[nb], acc[mb][nb], 0, 0, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        take_weights(0, now);
        if (CH < iterations) issue_weights(CH);
        asm volatile("" ::: "memory");
        read(0, 0, a[0]);
        decode(now.w[0], now.s[0], 0, first < end, b[0]);
        __builtin_amdgcn_sched_barrier(0);
        for (int it0 = 0; it0 < iterations; it0 += CH) {
#pragma unroll
            for (int gi = 0; gi < CH; ++gi) {
                const int it = it0 + gi;
                const bool inside = first + it < end;
#pragma unroll
                for (int step = 0; step < 3; ++step) {
                    read(it, step + 1, a[(step + 1) & 1]);
                    decode(now.w[gi], now.s[gi], step + 1, inside, b[(step + 1) & 1]);
                    multiply(a[step & 1], b[step & 1]);
                }
                // made here and not sunk to the use behind the workgroup's meeting, where nothing covers it
                asm volatile("" : "+v"(b[1][0]), "+v"(b[1][1]));
                // the next planes were sent for before the chunk that may still be on its way
                if (gi == 0 && it0 + CH < iterations) {
                    if (whole_scales) wait_loads<S::CODE_LOADS + 1>(); else wait_loads<S::CODE_LOADS + 2 * CH>();
                } else {
                    wait_loads<0>();
                }
                meet();
                if (it + 2 < iterations) issue_x(it + 2);
                if (gi == CH - 1) {
                    take_weights(it + 1, now);
                    if (it + 1 + CH < iterations) issue_weights(it + 1 + CH);
                }
                // after the last stage these are stale and unused
                read(it + 1, 0, a[0]);
                decode(now.w[gi == CH - 1 ? 0 : gi + 1], now.s[gi == CH - 1 ? 0 : gi + 1], 0, first + it + 1 < end, b[0]);
                multiply(a[1], b[1]);
                if (it + 1 >= iterations) break;
            }
        }
    } else {
        for (int it = 0; it < iterations; ++it) {    // a wave without rows helps to stage
            wait_loads<0>();
            meet();
            if (it + 2 < iterations) issue_x(it + 2);
        }
    }

    // ---- the parts meet in part order
    float *sums = reinterpret_cast<float *>(stage);
    if (S::KP > 1) __syncthreads();
    if (part > 0) {
        float *mine = sums + ((part - 1) * RW + wn) * 4096 + lane;
#pragma unroll
        for (int k = 0; k < 64; ++k) mine[k * 64] = acc[k >> 5][(k >> 4) & 1][k & 15];
    }
    if (S::KP > 1) __syncthreads();
    const bool direct = L.ksplit == 1;
    if (direct && rejected(L)) return;
    if (part != 0 || !live) return;
#pragma unroll
    for (int p = 1; p < S::KP; ++p) {
        const float *theirs = sums + ((p - 1) * RW + wn) * 4096 + lane;
#pragma unroll
        for (int k = 0; k < 64; ++k) acc[k >> 5][(k >> 4) & 1][k & 15] += theirs[k * 64];
    }
    const global_f32_out out = (global_f32_out)(uintptr_t)(direct ? L.ys : L.partials + (size_t)split * L.tokens * L.rows);
    const float factor = direct ? L.out_scale : 1.0f;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
        global_f32_out line = out + (size_t)(tok0 + mb * 32 + half * 4) * L.rows + row0 + l32;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int tok = mb * 32 + half * 4 + (i >> 2) * 8 + (i & 3);
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
                if (tok < toks_here && row0 + nb * 32 + l32 < L.rows) line[nb * 32] = acc[mb][nb][i] * factor;
            line += (size_t)L.rows * ((i & 3) == 3 ? 5 : 1);
        }
    }
}

// ys = out_scale * (partial 0 + partial 1 + ...), added in split order
__global__ __launch_bounds__(256) void fp4_split_sum_kernel(const Fp4MfmaLaunch L, size_t n) {
    if (rejected(L)) return;
    const float *__restrict__ partials = L.partials;
    float *__restrict__ ys = L.ys;
    const int ksplit = L.ksplit;
    const float out_scale = L.out_scale;
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;
    if ((n & 3) == 0) {
        float4 sum = *reinterpret_cast<const float4 *>(partials + i);
        for (int s = 1; s < ksplit; ++s) {
            const float4 p = *reinterpret_cast<const float4 *>(partials + (size_t)s * n + i);
            sum.x += p.x; sum.y += p.y; sum.z += p.z; sum.w += p.w;
        }
        ys[i] = sum.x * out_scale; ys[i + 1] = sum.y * out_scale; ys[i + 2] = sum.z * out_scale;
        ys[i + 3] = sum.w * out_scale;
    } else {
        for (size_t j = i; j < n && j < i + 4; ++j) {
            float sum = partials[j];
            for (int s = 1; s < ksplit; ++s) sum += partials[(size_t)s * n + j];
            ys[j] = sum * out_scale;
        }
    }
}

}  // namespace

namespace {
// Tiles of 64 x 256 by four waves, two workgroups on a compute unit, where there are enough of them; else tiles of
// 64 x 128 by eight waves, four column parts.  Rows of FAR_COLS columns and more have the one form.
bool wide_tiles(int rows, int cols, int tokens) {
    return cols < FAR_COLS && (long long)((tokens + TM - 1) / TM) * ((rows + 255) / 256) >= 320;
}
}  // namespace

int fp4_mfma_splits(int rows, int cols, int tokens) {
    const int tn = wide_tiles(rows, cols, tokens) ? 256 : 128;
    const int tiles = ((tokens + TM - 1) / TM) * ((rows + tn - 1) / tn);
    const int chunks = cols / KC;
    int splits = 256 / tiles;                          // while every workgroup still has a compute unit of its own
    if (splits > 8) splits = 8;
    if (splits > chunks / 8) splits = chunks / 8;      // at least eight chunks per split, two per part
    // with chunks shared out in equal runs the last split must still own one (30 chunks in 7 splits of 5 would not)
    while (splits > 1 && (splits - 1) * ((chunks + splits - 1) / splits) >= chunks) --splits;
    return splits < 1 ? 1 : splits;
}

int fp4_mfma_launch(const Fp4MfmaLaunch &L, hipStream_t stream) {
    if (L.rows < 1 || L.tokens < 1 || L.cols < KC || (L.cols % KC) || L.ksplit < 1) return -1;
    if (L.flags ? (L.nflags < 1 || !L.outcome) : !L.status) return -1;
    const bool wide = wide_tiles(L.rows, L.cols, L.tokens);
    const int tn = wide ? 256 : 128;
    Geometry G;
    G.m_tiles = (L.tokens + TM - 1) / TM;
    G.n_tiles = (L.rows + tn - 1) / tn;
    G.chunks = L.cols / KC;
    G.chunks_per_split = (G.chunks + L.ksplit - 1) / L.ksplit;
    if ((L.ksplit - 1) * G.chunks_per_split >= G.chunks) return -1;        // every split owns a chunk
    if (L.ksplit > 1 && !L.partials) return -1;
    const long long grid = ((long long)G.m_tiles * G.n_tiles * L.ksplit + 7) / 8 * 8;
    if (grid > 0x7FFFFFFFLL) return -1;
    note_kernel("fp4_mfma_kernel<%s> ksplit %d", wide ? "4,4,0" : L.cols < FAR_COLS ? "8,2,0" : "8,2,1", L.ksplit);
    if (wide) hipLaunchKernelGGL((fp4_mfma_kernel<4, 4, false>), dim3((unsigned)grid), dim3(256), 0, stream, L, G);
    else if (L.cols < FAR_COLS) hipLaunchKernelGGL((fp4_mfma_kernel<8, 2, false>), dim3((unsigned)grid), dim3(512), 0, stream, L, G);
    else hipLaunchKernelGGL((fp4_mfma_kernel<8, 2, true>), dim3((unsigned)grid), dim3(512), 0, stream, L, G);
    if (L.ksplit > 1) {
        const size_t n = (size_t)L.tokens * L.rows;
        hipLaunchKernelGGL(fp4_split_sum_kernel, dim3((unsigned)((n / 4 + 256) / 256)), dim3(256), 0, stream, L, n);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace mi355
