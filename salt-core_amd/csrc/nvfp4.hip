// NVFP4 matvec and activation quantise/dequantise for gfx950, bit-identical to
// the engine's CPU reference (reference src/nvfp4.c).
//
// Weight element (reference nvfp4.c:173-192):
//     scaled = fl(e4m3(scale[row][col/16]) * weight_global_scale)
//     w      = fl(e2m1(code) * scaled);  p = fl(w * x[col]);  acc[col%32] += p
// with the same 32 chains and the same fold as the affine-Q4 row.  The matvec
// kernel has the Q4 kernel's shape (lane = row, wave-uniform chain slice,
// scalar-loaded activations, LDS-staged codes, in-order fold); only decoding
// differs: v_cvt_scalef32_pk_f32_fp4 turns one byte into two E2M1 values
// without any masking, and the per-16-column `scaled` factors are produced
// once per tile step into LDS with the hardware E4M3 decoder.
//
// E2M1 code 8 ("-0") decodes to +0 in the reference and to -0 in hardware.
// The difference never reaches a result: it only flips the sign of a zero
// product, and a chain accumulator that starts at +0 can never become -0.
//
// The activation pre-pass (reference nvfp4.c:82-130) runs four threads per
// 16-element block with closed-form round-to-nearest-even encoders in place of
// the reference's argmin scans (equality is proven on the host by the tests).
#include "mi355_internal.h"
#include "nvfp4_device.h"

#include <stddef.h>

namespace mi355 {
namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef const float __attribute__((address_space(4))) *uniform_f32_ptr;
typedef const uint64_t __attribute__((address_space(4))) *uniform_u64_ptr;
typedef const uint8_t __attribute__((address_space(1))) *global_u8_ptr;
typedef const uint16_t __attribute__((address_space(1))) *global_u16_ptr;
typedef u32x4 __attribute__((aligned(4))) u32x4_dword_aligned;       // 128-bit global loads need dword alignment only
typedef const u32x4_dword_aligned __attribute__((address_space(1))) *global_u128_ptr;
typedef float __attribute__((address_space(1))) *global_f32_out_ptr;

constexpr int TILE_ROWS = 64;
constexpr int CHUNK_BLOCKS = 16;                       // 32-column blocks per staged step
constexpr int W_PITCH = 16 * CHUNK_BLOCKS + 4;         // bytes per staged row of codes
constexpr int M_PITCH = 2 * CHUNK_BLOCKS + 1;          // floats per staged row of `scaled` factors (odd)
constexpr int FOLD_PITCH = 33;

static_assert(sizeof(Fp4Job) == 48 && offsetof(Fp4Job, weight_global_scale) == 32 && offsetof(Fp4Job, rows) == 36 &&
              offsetof(Fp4Job, tile0) == 40 && offsetof(Fp4Job, x_stride) == 44,
              "find_job reads a job record as six 64-bit words");

__device__ __forceinline__ Fp4Job find_job(const Fp4Launch &L, int tile) {
    if (L.table == nullptr) return L.one;
    const uniform_u64_ptr words = (uniform_u64_ptr)(uintptr_t)L.table;     // 6 words per record
    int lo = 0, hi = L.njobs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if ((int)(uint32_t)words[6 * mid + 5] <= tile) lo = mid; else hi = mid - 1;
    }
    const uniform_u64_ptr rec = words + 6 * lo;
    Fp4Job job;
    job.packed = (const uint8_t *)rec[0];
    job.scales = (const uint8_t *)rec[1];
    job.x = (const float *)rec[2];
    job.y = (float *)rec[3];
    job.weight_global_scale = __uint_as_float((uint32_t)rec[4]);
    job.rows = (int)(rec[4] >> 32);
    job.tile0 = (int)(uint32_t)rec[5];
    job.x_stride = (int)(rec[5] >> 32);
    return job;
}

// What a 16-element block's largest magnitude decides (reference nvfp4.c:82-130).
struct BlockScale { uint32_t code; float scale, to_code, from_code; };
__device__ __forceinline__ BlockScale block_scale(float top, float g) {
    const float sixth = top * (1.0f / 6.0f);
    float raw = g * sixth;
    if (raw > 448.0f) raw = 448.0f;
    BlockScale b;
    b.code = e4m3_encode_positive(raw);
    b.scale = __builtin_amdgcn_cvt_f32_fp8((int)b.code, 0);
    b.to_code = b.scale == 0.0f ? 0.0f : g / b.scale;
    b.from_code = b.scale / g;
    return b;
}
__device__ __forceinline__ uint32_t element_code(float v, const BlockScale &b) {
    float s = v * b.to_code;
    if (s > 6.0f) s = 6.0f;
    if (s < -6.0f) s = -6.0f;
    return e2m1_encode(s);
}
// code value * block scale: at most six significant bits between 2^-10 and 2688, exact in fp16
__device__ __forceinline__ uint32_t operand_half(float value, const BlockScale &b) {
    return __builtin_bit_cast(uint16_t, (_Float16)(value * b.scale));
}

// Quantises and dequantises one 16-element block.  Returns false when an element is not finite (the reference rejects
// the call).
__device__ __forceinline__ bool qdq_block(const float (&v)[16], float g, float (&out)[16]) {
    float top = 0.0f;
    bool finite = true;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float m = __builtin_fabsf(v[i]);
        finite = finite && (m < __builtin_inff());           // false for inf and NaN
        if (m > top) top = m;
    }
    if (!finite) return false;
    const BlockScale b = block_scale(top, g);
#pragma unroll
    for (int i = 0; i < 16; ++i) out[i] = e2m1_decode(element_code(v[i], b)) * b.from_code;
    return true;
}

constexpr int x_batch_blocks(int S, int NB) {
    const int fit = (S == 8 ? 32 : 64) / (S * NB);
    return fit >= 16 ? 16 : fit >= 8 ? 8 : fit >= 4 ? 4 : fit >= 2 ? 2 : 1;
}

// QDQ: the launch's single token is quantised and dequantised by every
// workgroup in its prologue (the activation pass of the reference matvec,
// nvfp4.c:228-256) into LDS, and the rows read it from there into vector
// registers (every lane the same words); workgroup 0 reports a non-finite activation (-1 into a
// status word the caller cleared) and nothing is published then.
//
// SPLIT (with QDQ): the tile is cut into SPLIT workgroups of 64 / SPLIT rows, as in the affine-Q4 kernel, for launches
// that would leave compute units idle; lane l of a wave holds row l % ROWS of chain slice SPLIT * wave + l / ROWS.
// 8192 x 8192, one token (128 tiles): 27.0 -> 18.5 us.
template <int S, int NB, bool QDQ = false, int SPLIT = 1>
__global__ __launch_bounds__((32 / (S * SPLIT)) * 64) void fp4_tile_kernel(const Fp4Launch L) {
    constexpr int ROWS = TILE_ROWS / SPLIT;
    constexpr int W_STAGE = ROWS * W_PITCH, M_STAGE = ROWS * M_PITCH;
    constexpr int WAVES = 32 / (S * SPLIT);
    constexpr int THREADS = WAVES * 64;
    constexpr int PIECES = (ROWS * CHUNK_BLOCKS) / THREADS;          // 16-byte pieces == (row, block) items
    constexpr int FOLD_BYTES = NB * ROWS * FOLD_PITCH * 4;
    constexpr int W_BYTES = 2 * W_STAGE > FOLD_BYTES ? 2 * W_STAGE : FOLD_BYTES;
    constexpr int XB = QDQ ? 2 : x_batch_blocks(S, NB);      // LDS-fed activations sit in vector registers: short batches
    constexpr int XN = XB * S;
    constexpr int W_ROW_STEP = THREADS / 16;
    static_assert(THREADS >= NB * ROWS, "fold needs one thread per (token, row)");
    static_assert(SPLIT == 1 || QDQ, "split tiles take their activations from LDS");

    __shared__ __attribute__((aligned(16))) uint8_t w_lds[W_BYTES];
    __shared__ float m_lds[2 * M_STAGE];
    __shared__ __attribute__((aligned(16))) float x_lds[QDQ ? FP4_FUSED_MAX_COLS : 4];
    __shared__ int x_bad;
    static_assert(!QDQ || NB == 1, "the fused activation pass serves single-token launches");

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // lane's row of the tile and its slice of the chains
    const int lane_row = lane & (ROWS - 1);
    const int slice = SPLIT == 1 ? wave : wave * SPLIT + lane / ROWS;
    const int tile = SPLIT == 1 ? (int)blockIdx.x : (int)blockIdx.x / SPLIT;
    const Fp4Job job = find_job(L, tile);
    if (QDQ) {
        if (tid == 0) x_bad = 0;
        __syncthreads();
        for (int blk = tid; blk < (L.cols >> 4); blk += THREADS) {
            const float4 *src = reinterpret_cast<const float4 *>(job.x + (size_t)blk * 16);
            float v[16];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 f = src[q];
                v[4 * q] = f.x; v[4 * q + 1] = f.y; v[4 * q + 2] = f.z; v[4 * q + 3] = f.w;
            }
            float out[16];
            if (!qdq_block(v, L.input_global_scale, out)) { x_bad = 1; continue; }
            float4 *dst = reinterpret_cast<float4 *>(x_lds + blk * 16);
#pragma unroll
            for (int q = 0; q < 4; ++q) dst[q] = make_float4(out[4 * q], out[4 * q + 1], out[4 * q + 2], out[4 * q + 3]);
        }
        __syncthreads();
        const int bad = x_bad;
        if (bad && blockIdx.x == 0 && tid == 0) *L.status = -1;        // like fp4_qdq_kernel: the caller cleared it
        if (bad) return;                                   // uniform
    }
    const int row0 = (tile - job.tile0) * TILE_ROWS + (SPLIT == 1 ? 0 : ((int)blockIdx.x % SPLIT) * ROWS);
    if (SPLIT > 1 && row0 >= job.rows) return;             // uniform: the rest of the last tile
    const int rows_here = job.rows - row0 < ROWS ? job.rows - row0 : ROWS;
    const int nblk = L.cols >> 5;
    const int nchunk = (nblk + CHUNK_BLOCKS - 1) / CHUNK_BLOCKS;
    const uint32_t row_bytes = (uint32_t)(L.cols >> 1);
    const uint32_t row_pairs = (uint32_t)nblk;                       // scale byte pairs per row
    const global_u8_ptr codes = (global_u8_ptr)(uintptr_t)job.packed + (size_t)row0 * row_bytes;
    const global_u16_ptr scale_pairs = (global_u16_ptr)(uintptr_t)job.scales + (size_t)row0 * row_pairs;
    const global_f32_out_ptr y = (global_f32_out_ptr)(uintptr_t)job.y;
    const uniform_f32_ptr xbase = (uniform_f32_ptr)(uintptr_t)job.x + S * wave;
    const float wg = job.weight_global_scale;

    // Piece i of a thread: row (tid>>4) + i*W_ROW_STEP, block column tid&15.
    // The same (row, block) item also owns that block's two scale bytes.
    const uint32_t seg = tid & 15;
    const uint32_t w_dst0 = (tid >> 4) * W_PITCH + seg * 16;
    const uint32_t m_dst0 = (tid >> 4) * M_PITCH + seg * 2;
    uint32_t src_row[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int row = (tid >> 4) + i * W_ROW_STEP;
        src_row[i] = (uint32_t)(row < rows_here ? row : rows_here - 1);
    }

    u32x4 wreg[PIECES];
    uint32_t mreg[PIECES];

    auto issue = [&](int ck) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            int blk = ck * CHUNK_BLOCKS + (int)seg;
            blk = blk < nblk ? blk : nblk - 1;
            wreg[i] = __builtin_nontemporal_load((global_u128_ptr)(codes + (src_row[i] * row_bytes + (uint32_t)blk * 16u)));
            mreg[i] = scale_pairs[src_row[i] * row_pairs + (uint32_t)blk];
        }
    };
    auto commit = [&](int stage) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            uint32_t *dst = reinterpret_cast<uint32_t *>(w_lds + stage * W_STAGE + w_dst0 + i * W_ROW_STEP * W_PITCH);
            dst[0] = wreg[i].x; dst[1] = wreg[i].y; dst[2] = wreg[i].z; dst[3] = wreg[i].w;
            float *m = m_lds + stage * M_STAGE + m_dst0 + i * W_ROW_STEP * M_PITCH;
            m[0] = __builtin_amdgcn_cvt_f32_fp8((int)mreg[i], 0) * wg;      // columns 0..15 of the block
            m[1] = __builtin_amdgcn_cvt_f32_fp8((int)mreg[i], 1) * wg;      // columns 16..31
        }
    };

    float acc[NB][S];
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int c = 0; c < S; ++c) acc[t][c] = 0.0f;

    issue(0);

    auto load_x = [&](int blk0, float (&xq)[NB][XN], int blocks) {
        if (QDQ) {                        // every lane reads the same LDS words: the activations travel in vector registers
            const float *xl = x_lds + blk0 * 32 + S * slice;
#pragma unroll
            for (int k = 0; k < XN; ++k)
                if (k < blocks * S) xq[0][k] = xl[(k / S) * 32 + (k % S)];
            return;
        }
        const uniform_f32_ptr xg = xbase + (size_t)blk0 * 32;
#pragma unroll
        for (int t = 0; t < NB; ++t)
#pragma unroll
            for (int k = 0; k < XN; ++k)
                if (k < blocks * S) xq[t][k] = xg[(size_t)t * job.x_stride + (k / S) * 32 + (k % S)];
    };

    // One block of one lane: S codes against the wave's S chains.
    auto consume = [&](uint32_t w, float scaled, const float (&xq)[NB][XN], int xat) {
#pragma unroll
        for (int b = 0; b < S / 2; ++b) {
            f32x2 v;
            switch (b) {                       // the byte selector is an immediate
                case 0: v = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 0); break;
                case 1: v = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 1); break;
                case 2: v = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 2); break;
                default: v = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 3); break;
            }
            const float w0 = v.x * scaled, w1 = v.y * scaled;
#pragma unroll
            for (int t = 0; t < NB; ++t) {
                const float p0 = w0 * xq[t][xat + 2 * b];
                acc[t][2 * b] = acc[t][2 * b] + p0;
                const float p1 = w1 * xq[t][xat + 2 * b + 1];
                acc[t][2 * b + 1] = acc[t][2 * b + 1] + p1;
            }
        }
    };

    for (int ck = 0; ck < nchunk; ++ck) {
        const int stage = ck & 1;
        const int remaining = nblk - ck * CHUNK_BLOCKS;
        const bool full = remaining >= CHUNK_BLOCKS;
        const int bcount = full ? CHUNK_BLOCKS : remaining;

        float xq[NB][XN];
        if (full) load_x(ck * CHUNK_BLOCKS, xq, XB);

        commit(stage);
        __syncthreads();
        if (ck + 1 < nchunk) issue(ck + 1);

        const uint8_t *wrow = w_lds + stage * W_STAGE + lane_row * W_PITCH + slice * (S / 2);
        // the slice's chains lie in the first (columns 0..15) or second half of a block
        const float *mrow = m_lds + stage * M_STAGE + lane_row * M_PITCH + ((S * slice) >> 4);

        auto fetch = [&](int blk, uint32_t &w, float &scaled) {
            scaled = mrow[2 * blk];
            if (S == 8) w = *reinterpret_cast<const uint32_t *>(wrow + blk * 16);
            else if (S == 4) w = *reinterpret_cast<const uint16_t *>(wrow + blk * 16);
            else w = wrow[blk * 16];
        };

        if (full) {
#pragma unroll
            for (int batch = 0; batch < CHUNK_BLOCKS / XB; ++batch) {
                if (batch > 0) load_x(ck * CHUNK_BLOCKS + batch * XB, xq, XB);
#pragma unroll
                for (int bl = 0; bl < XB; ++bl) {
                    uint32_t w;
                    float scaled;
                    fetch(batch * XB + bl, w, scaled);
                    consume(w, scaled, xq, bl * S);
                }
            }
        } else {
            for (int blk = 0; blk < bcount; ++blk) {
                uint32_t w;
                float scaled;
                fetch(blk, w, scaled);
                load_x(ck * CHUNK_BLOCKS + blk, xq, 1);
                consume(w, scaled, xq, 0);
            }
        }
    }

    __syncthreads();
    float *fold = reinterpret_cast<float *>(w_lds);
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int c = 0; c < S; ++c) fold[(t * ROWS + lane_row) * FOLD_PITCH + S * slice + c] = acc[t][c];
    __syncthreads();
    if (tid < NB * ROWS) {
        const int t = tid / ROWS;
        const float *f = fold + (t * ROWS + lane_row) * FOLD_PITCH;
        float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int a = 0; a < 8; ++a)
#pragma unroll
            for (int j = 0; j < 4; ++j) part[j] = part[j] + f[4 * a + j];
        const float even = part[0] + part[2];
        const float odd = part[1] + part[3];
        if (lane_row < rows_here) y[(size_t)t * job.rows + row0 + lane_row] = even + odd;
    }
}

template <int S>
int launch_tiles(const Fp4Launch &L, hipStream_t stream) {
    const dim3 grid(L.total_tiles), block((32 / S) * 64);
    if (L.qdq) {
        if (L.tokens != 1 || L.table || L.cols > FP4_FUSED_MAX_COLS || !L.status || ((uintptr_t)L.one.x & 15)) return -1;
        // sixteen-row workgroups while they find room at once, thirty-two-row ones up to one per compute unit
        // (64 tiles of 8192 columns 26.2 -> 18.1 us, 128 27.0 -> 18.5)
        if (S == 2 && L.total_tiles <= 64) {
            hipLaunchKernelGGL((fp4_tile_kernel<2, 1, true, 4>), dim3(4 * L.total_tiles), dim3(256), 0, stream, L);
            return hipGetLastError() == hipSuccess ? 0 : -1;
        }
        if (S == 2 && L.total_tiles <= 128) {
            hipLaunchKernelGGL((fp4_tile_kernel<2, 1, true, 2>), dim3(2 * L.total_tiles), dim3(512), 0, stream, L);
            return hipGetLastError() == hipSuccess ? 0 : -1;
        }
        hipLaunchKernelGGL((fp4_tile_kernel<S, 1, true>), grid, block, 0, stream, L);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    switch (L.tokens) {
        case 1: hipLaunchKernelGGL((fp4_tile_kernel<S, 1>), grid, block, 0, stream, L); break;
        case 2: hipLaunchKernelGGL((fp4_tile_kernel<S, 2>), grid, block, 0, stream, L); break;
        case 3: hipLaunchKernelGGL((fp4_tile_kernel<S, 3>), grid, block, 0, stream, L); break;
        case 4: hipLaunchKernelGGL((fp4_tile_kernel<S, 4>), grid, block, 0, stream, L); break;
        default: return -1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---------------------------------------------------------------- activation Q/DQ

// Four neighbouring lanes per 16-element block of one token, four elements each, so that a wave reads and writes whole
// cache lines (a lane per block read 64 bytes apart: 256 tokens of 8192 columns 9.0 -> 7.2 us).  FLAGS: the workgroup
// reports in the flag of its own number (0 or -1, always written) instead of setting *status.
constexpr int QDQ_THREADS = 1024, QDQ_BLOCKS = QDQ_THREADS / 4;
constexpr unsigned QDQ_GRID_X = 1u << 20;      // a grid's dimension holds less than 2^32 threads: the rest goes into rows of this many

template <bool FLAGS>
__global__ __launch_bounds__(QDQ_THREADS) void fp4_qdq_kernel(const float *__restrict__ input, int cols, int tokens,
                                                      float g, uint8_t *__restrict__ packed,
                                                      uint8_t *__restrict__ scales, float *__restrict__ dequant,
                                                      uint16_t *__restrict__ plane, int *__restrict__ status) {
    const int blocks_per_token = cols >> 4;
    const long long group = (long long)blockIdx.y * gridDim.x + blockIdx.x, items = (long long)blocks_per_token * tokens;
    if (group * QDQ_BLOCKS >= items) return;                 // uniform: past the last workgroup of the last row
    const long long item = group * QDQ_BLOCKS + (threadIdx.x >> 2);
    const int quarter = threadIdx.x & 3;
    const bool present = item < items;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (present) {
        const float4 f = reinterpret_cast<const float4 *>(input)[item * 4 + quarter];
        v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
    }
    // the block's largest magnitude as a bit pattern: infinities and NaN are the largest of all
    uint32_t top_bits = 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t m = __float_as_uint(v[i]) & 0x7fffffffu;
        top_bits = m > top_bits ? m : top_bits;
    }
#pragma unroll
    for (int d = 1; d < 4; d <<= 1) {
        const uint32_t other = (uint32_t)__shfl_xor((int)top_bits, d, 64);
        top_bits = other > top_bits ? other : top_bits;
    }
    const bool good = top_bits < 0x7f800000u;                // the reference rejects the whole call
    if (FLAGS) {
        const int any_bad = __syncthreads_or(good ? 0 : 1);
        if (threadIdx.x == 0) status[group] = any_bad ? -1 : 0;
        if (!present || !good) return;
    } else {
        if (present && !good) *status = -1;
        if (!present || !good) return;
    }
    const BlockScale b = block_scale(__uint_as_float(top_bits), g);
    uint32_t codes = 0u;
    float out[4];
    uint32_t halves[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t code = element_code(v[i], b);
        codes |= code << (4 * i);
        const float value = e2m1_decode(code);
        out[i] = value * b.from_code;
        const uint32_t h = operand_half(value, b);
        if (i & 1) halves[i >> 1] |= h << 16; else halves[i >> 1] = h;
    }
    if (scales && quarter == 0) scales[item] = (uint8_t)b.code;
    if (packed) reinterpret_cast<uint16_t *>(packed)[item * 4 + quarter] = (uint16_t)codes;
    if (dequant) reinterpret_cast<float4 *>(dequant)[item * 4 + quarter] = make_float4(out[0], out[1], out[2], out[3]);
    if (plane) reinterpret_cast<uint2 *>(plane)[item * 4 + quarter] = make_uint2(halves[0], halves[1]);
}

}  // namespace

int fp4_launch(const Fp4Launch &L, int chains_per_lane, hipStream_t stream) {
    if (L.total_tiles < 1 || L.tokens < 1 || L.tokens > 4 || L.cols < 32 || (L.cols & 31)) return -1;
    int S = chains_per_lane;
    // as for the affine-Q4 kernel: sixteen waves per tile up to one tile per compute unit, eight beyond (8192 columns,
    // one token: 23.9 against 30.2 us at 256 tiles, 42.5 against 36.0 at 320, 48.5 against 43.8 at 512)
    if (S == 0) S = L.total_tiles > 256 ? 4 : 2;
    switch (S) {
        case 8: return launch_tiles<8>(L, stream);
        case 4: return launch_tiles<4>(L, stream);
        case 2: return launch_tiles<2>(L, stream);
        default: return -1;
    }
}

namespace {
dim3 qdq_grid(long long groups) {
    return groups <= QDQ_GRID_X ? dim3((unsigned)groups) : dim3(QDQ_GRID_X, (unsigned)((groups + QDQ_GRID_X - 1) / QDQ_GRID_X));
}
}  // namespace

int fp4_qdq_launch(const float *input, int cols, int tokens, float input_global_scale, uint8_t *packed,
                   uint8_t *scales, float *dequant, uint16_t *plane, int *status, hipStream_t stream) {
    const long long items = (long long)(cols >> 4) * tokens;
    if (items < 1 || items >= (1ll << 32) || (cols & 15)) return -1;
    hipLaunchKernelGGL(fp4_qdq_kernel<false>, qdq_grid((items + QDQ_BLOCKS - 1) / QDQ_BLOCKS), dim3(QDQ_THREADS), 0, stream, input, cols, tokens, input_global_scale,
                       packed, scales, dequant, plane, status);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int fp4_qdq_flag_count(int cols, int tokens) {
    const long long items = (long long)(cols >> 4) * tokens;
    return items < 1 || items > (1ll << 38) ? 0 : (int)((items + QDQ_BLOCKS - 1) / QDQ_BLOCKS);
}

int fp4_qdq_flags_launch(const float *input, int cols, int tokens, float input_global_scale, uint16_t *plane,
                         int *flags, hipStream_t stream) {
    const int grid = fp4_qdq_flag_count(cols, tokens);
    if (grid < 1 || (cols & 15) || !flags) return -1;
    hipLaunchKernelGGL(fp4_qdq_kernel<true>, qdq_grid(grid), dim3(QDQ_THREADS), 0, stream, input, cols, tokens,
                       input_global_scale, (uint8_t *)nullptr, (uint8_t *)nullptr, (float *)nullptr, plane, flags);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace mi355
