// The fp32 cells around the MoE step of a decoder layer: RMS norm, router input, residual post-norm, parallel
// feed-forward combine, softcap (reference models/gemma4-26b-a4b/src/gemma4.c:46-130, 188-286; the backend ABI's
// exact cells, include/salt/gpu.h:211-234, src/gpu_hip.cpp:2034-2063, 2389-2458, 2688-2745).
//
// Every norm needs ss = x0*x0 + x1*x1 + ... added left to right in fp32.  The squares are computed by the whole
// workgroup into LDS; one wave per vector then adds them (ordered_sum: the bits of the left-to-right chain, most of it
// not walked).  inv = pow(ss / n + eps, -0.5) is six double-precision Newton steps from the
// 0x5f3759df seed (src/bitmath.c:114-142).  A cell that meets a non-finite input or result publishes nothing and
// sets the sticky status word to -1; a cell that finds the status word set does nothing.
#include "device_math.h"
#include "mi355_internal.h"

namespace mi355 {
namespace {

constexpr int THREADS = 1024;         // one workgroup per cell: sixteen waves keep enough loads in flight
constexpr int SLOTS = 4;              // elements a thread handles per pass: i = base + tid + k * THREADS
constexpr int SQ_CHUNK = SLOTS * THREADS;   // squares staged per pass of the serial adder
constexpr int SQ_TAIL = 64;           // floats the adder may read (and drop) past the staged squares

__device__ __forceinline__ double inverse_root64(float x) {
    const float seed = __uint_as_float(0x5f3759dfu - (__float_as_uint(x) >> 1));
    double y = (double)seed;
    const double wide = (double)x;
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        const double square = y * y;
        const double half = 0.5 * wide;
        const double step = 1.5 - half * square;
        y = y * step;
    }
    return y;
}

__device__ float det_rsqrtf(float x) {
    if (x != x) return x;
    if (x < 0.0f) return __uint_as_float(0x7fc00000u);
    if (x == 0.0f) return __uint_as_float(0x7f800000u);
    if (x == 1.0f) return 1.0f;
    if (x < 0x1p-126f) {                               // rescaled once: x * 2^24 is a normal number
        const float up = x * 0x1p24f;
        const float root = up == 1.0f ? 1.0f : (float)inverse_root64(up);
        return root * 0x1p12f;
    }
    return (float)inverse_root64(x);
}

__device__ float det_sqrtf(float x) {
    if (x != x) return x;
    if (x < 0.0f) return __uint_as_float(0x7fc00000u);
    if (x == 0.0f || x == 1.0f) return x;
    if (x < 0x1p-126f) {
        const float up = x * 0x1p24f;
        const float root = up == 1.0f ? 1.0f : (float)((double)up * inverse_root64(up));
        return root * 0x1p-12f;
    }
    return (float)((double)x * inverse_root64(x));
}

// salt_powf(x, -0.5f)
__device__ __forceinline__ float pow_minus_half(float x) {
    if (x == 1.0f) return 1.0f;
    if (x > 0.0f) return det_rsqrtf(x);
    return x;
}

// 1 for an infinity or a NaN; an unsigned, so that flags combine with | and no load hides behind a short circuit
__device__ __forceinline__ unsigned nonfinite(float v) { return (__float_as_uint(v) & 0x7f800000u) == 0x7f800000u; }

// Visits the elements [0, n) SLOTS at a time per thread: f(i, k) for the live slots of a pass, all loads of a pass
// being independent of each other.
template <typename F>
__device__ __forceinline__ void each_element(int n, F f) {
    for (int base = 0; base < n; base += SQ_CHUNK) {
#pragma unroll
        for (int k = 0; k < SLOTS; ++k) {
            const int i = base + (int)threadIdx.x + k * THREADS;
            if (i < n) f(i);
        }
    }
}

// acc + mine[0] + mine[1] + ... + mine[count - 1], left to right; count is a multiple of 32.  32 values per batch; the next
// batch is read from LDS while the current one is added, unconditionally one batch ahead (what is read past the end is
// dropped, the staging buffers have a tail for it).
__device__ __forceinline__ float add_staged(const float *mine, int count, float acc) {
    const int pairs = count & ~63;
    float4 a[8], b[8];
    auto fetch = [&](float4 (&dst)[8], int at) {
#pragma unroll
        for (int k = 0; k < 8; ++k) dst[k] = *(const float4 *)&mine[at + 4 * k];
    };
    auto add = [&](const float4 (&src)[8]) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            acc = acc + src[k].x;
            acc = acc + src[k].y;
            acc = acc + src[k].z;
            acc = acc + src[k].w;
        }
    };
    fetch(a, 0);
    for (int i = 0; i < pairs; i += 64) {
        fetch(b, i + 32);
        add(a);
        fetch(a, i + 64);
        add(b);
    }
    if (count != pairs) add(a);
    return acc;
}

// ---- the same chain, not walked
//
// Between two powers of two every value of the accumulator is a multiple of one unit u, and adding x >= 0 moves it by
// rint(x / u) units; only when x / u ends in exactly one half does the step depend on the accumulator, and then on its
// last bit alone.  So while it stays in one binade the accumulator's bit pattern moves by an integer that is a function
// of its last bit, and such functions compose: {d0, d1} is the number of units that a run of addends adds to an even
// and to an odd accumulator.  A wave cuts the addends into 256 parts (lane l has parts 4 l .. 4 l + 3), guesses where
// the chain stands at each part from plain sums, finds each part's {d0, d1} by adding its values to an even and an odd
// number of that binade, and composes them over the wave.  Parts in which a guess leaves its binade are walked; where
// the chain turns out to be in another binade than the guess, everything is: the guesses decide what is walked, never
// the result.
// (Subnormals and the lowest normal binade share their unit; a zero accumulator is even; infinities and NaN are walked.)
//
// 2816 squares of a normal vector: 9 of 235 parts are walked, 3.0 us instead of 10.1 for the chain (a lone wave's dependent
// vector instructions issue eight clocks apart, 3.6 ns, independent ones four, which is what counts here).  The
// feed-forward block of 2816/2112/704 with 128 experts, three such sums deep: 90.1 -> 63.8 us (57.5 since its branches
// share their launches); its first cell 13.5 -> 6.2 us, its last 30.6 -> 11.2.
constexpr int ORDERED_MIN = 736;      // below, the chain is quicker (a norm of 512 / 704 / 736 / 768 values 5.2 / 5.85 / 5.86 / 6.0 us,
                                      // 5.8 to 5.9 with ordered_sum)
constexpr int PARTS = 4;              // of a lane
constexpr int ORDERED_FLOATS = 64 * (SQ_CHUNK / 64 + 4);     // LDS of SQ_CHUNK addends; a lane's block is 4 floats apart
                                                             // from the next, so that 16-byte reads hit all banks
struct OrderedScratch { int4 run[64 * PARTS + 1]; int walked[64 * PARTS + 1]; };

// 16-byte words of a part: 1 to 4, so that 256 parts hold count <= SQ_CHUNK addends
__device__ __forceinline__ int part_words(int count) { return (count + 1023) >> 10; }
// place of addend i in LDS
__device__ __forceinline__ int ordered_place(int i, int words) {
    const int third = words == 3 ? 171 : 512 >> (words >> 1);     // (i / 16) / words, exact below 256
    const int lane = ((i >> 4) * third) >> 9;
    return i + 4 * lane;
}

struct Units { int d0, d1; bool cut; };             // cut: a walked part lies inside, what came before it is forgotten
__device__ __forceinline__ Units then(const Units &a, const Units &b) {
    const int a0 = a.d0, a1 = a.d1, b0 = b.d0, b1 = b.d1;         // values: a choice between members is one of addresses
    const int r0 = a0 + ((a0 & 1) ? b1 : b0), r1 = a1 + ((a1 & 1) ? b0 : b1);
    return {b.cut ? b0 : r0, b.cut ? b1 : r1, a.cut || b.cut};
}

// The value of another lane as the data-parallel control says; lanes and rows it gives nothing to get `none`.
template <int CTRL, int ROWS> __device__ __forceinline__ int from_lane(int none, int v) {
    return __builtin_amdgcn_update_dpp(none, v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS> __device__ __forceinline__ void scan_step(float &v) {
    v = __int_as_float(from_lane<CTRL, ROWS>(0, __float_as_int(v))) + v;
}
template <int CTRL, int ROWS> __device__ __forceinline__ void scan_step(Units &v) {
    const Units before = {from_lane<CTRL, ROWS>(0, v.d0), from_lane<CTRL, ROWS>(0, v.d1),
                          from_lane<CTRL, ROWS>(0, (int)v.cut) != 0};
    v = then(before, v);
}
// inclusive scan over the wave: within rows of 16 lanes (row_shr 1, 2, 4, 8), then across them (row_bcast 15, 31)
template <typename T> __device__ __forceinline__ void wave_scan(T &v) {
    scan_step<0x111, 0xf>(v); scan_step<0x112, 0xf>(v); scan_step<0x114, 0xf>(v); scan_step<0x118, 0xf>(v);
    scan_step<0x142, 0xa>(v); scan_step<0x143, 0xc>(v);
}
constexpr int WAVE_SHR1 = 0x138;

// acc + addend 0 + addend 1 + ..., left to right, by one whole wave; up to 1024 * WORDS addends at their ordered_place,
// zeros behind the last; finite or not, never negative.
template <int WORDS>
__device__ __forceinline__ float ordered_sum(const float *addends, float acc, OrderedScratch &scratch) {
    constexpr int PITCH = 16 * WORDS + 4;
    typedef const float4 *words_ptr;
    const int lane = threadIdx.x & 63;
    const words_ptr mine = (words_ptr)(addends + lane * PITCH);
    float total = 0.0f, sum[PARTS];
#pragma unroll
    for (int p = 0; p < PARTS; ++p) {
        sum[p] = 0.0f;
#pragma unroll
        for (int w = 0; w < WORDS; ++w) {
            const float4 v = mine[p * WORDS + w];
            sum[p] += (v.x + v.y) + (v.z + v.w);
        }
        total += sum[p];
    }
    wave_scan(total);
    float guess = acc + __int_as_float(from_lane<WAVE_SHR1, 0xf>(0, __float_as_int(total)));
    Units run[PARTS];
    int binade[PARTS];                              // of a part that stays in one, else -1
#pragma unroll
    for (int p = 0; p < PARTS; ++p) {
        const int start = __float_as_int(guess) & ~1;
        float even = __int_as_float(start), odd = __int_as_float(start | 1);
#pragma unroll
        for (int w = 0; w < WORDS; ++w) {
            const float4 v = mine[p * WORDS + w];
            even = even + v.x; odd = odd + v.x;
            even = even + v.y; odd = odd + v.y;
            even = even + v.z; odd = odd + v.z;
            even = even + v.w; odd = odd + v.w;
        }
        const int b = start >> 23;
        const bool stays = (__float_as_int(even) >> 23) == b && (__float_as_int(odd) >> 23) == b && b != 255;
        binade[p] = stays ? b : -1;
        run[p] = {stays ? __float_as_int(even) - start : 0, stays ? __float_as_int(odd) - (start | 1) : 0, !stays};
        guess += sum[p];
    }
    int before = from_lane<WAVE_SHR1, 0xf>(-1, binade[PARTS - 1]);
    int position = 0, walks = 0;                    // among the walked parts: of this lane's first, and their number
#pragma unroll
    for (int p = 0; p < PARTS; ++p) {
        if (before >= 0 && binade[p] >= 0 && before != binade[p]) run[p] = {0, 0, true};      // the next binade starts here
        before = binade[p];
        const uint64_t walked = __ballot(run[p].cut);
        position += __builtin_amdgcn_mbcnt_hi((uint32_t)(walked >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)walked, 0));
        walks += __popcll(walked);
    }
    // Record r of `run` stands before part r: what the parts since the last walked one add, the bits that their binade
    // has above the significand, and which of those bits to hold against it (none where the part before is walked itself).
#pragma unroll
    for (int p = 0; p < PARTS; ++p)
        if (run[p].cut) scratch.walked[position++] = lane * PARTS + p;
    if (lane == 0) {
        scratch.walked[walks] = 64 * PARTS;
        scratch.run[0] = make_int4(0, 0, 0, 0);
    }
    bool cut[PARTS];
#pragma unroll
    for (int p = 0; p < PARTS; ++p) cut[p] = run[p].cut;
#pragma unroll
    for (int p = 1; p < PARTS; ++p) run[p] = then(run[p - 1], run[p]);
    Units lanes = run[PARTS - 1];
    wave_scan(lanes);
    lanes = {from_lane<WAVE_SHR1, 0xf>(0, lanes.d0), from_lane<WAVE_SHR1, 0xf>(0, lanes.d1),
             from_lane<WAVE_SHR1, 0xf>(0, (int)lanes.cut) != 0};
#pragma unroll
    for (int p = 0; p < PARTS; ++p) {
        const Units all = then(lanes, run[p]);
        scratch.run[lane * PARTS + p + 1] = make_int4(all.d0, all.d1, binade[p] << 23, cut[p] ? 0 : (int)0xff800000u);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();

    // From here on every lane does the same: the parts between two walked ones in one addition to the bit pattern, the
    // walked ones addend by addend.  Lane l holds where the l-th walked part of a round of 64 lies; its record and its
    // addends are read one walked part ahead.  Few instructions matter here: a lone wave issues one in four to eight clocks.
    auto words_of = [&](int part) { return (words_ptr)(addends + (part >> 2) * PITCH + (part & 3) * 4 * WORDS); };
    auto add = [&](const float4 &v) {
        acc = acc + v.x;
        acc = acc + v.y;
        acc = acc + v.z;
        acc = acc + v.w;
    };
    const float before_all = acc;
    int wrong = 0;                                  // bits of a binade that was not the chain's
    for (int k0 = 0; k0 <= walks; k0 += 64) {
        const int part = scratch.walked[k0 + lane <= walks ? k0 + lane : walks];
        const int here = walks + 1 - k0 < 64 ? walks + 1 - k0 : 64;
        struct Ahead { int4 leap; float4 v[WORDS]; } even, odd;
        auto read = [&](Ahead &to, int l) {
            const int next = __builtin_amdgcn_readlane(part, l);
            to.leap = scratch.run[next];
            const words_ptr from = words_of(next < 64 * PARTS ? next : 0);
#pragma unroll
            for (int w = 0; w < WORDS; ++w) to.v[w] = from[w];
        };
        auto leap = [&](const Ahead &of) {
            const int bits = __float_as_int(acc), d0 = of.leap.x, d1 = of.leap.y;
            const int moved = bits + ((bits & 1) ? d1 : d0);
            wrong |= ((bits ^ of.leap.z) | (moved ^ of.leap.z)) & of.leap.w;
            acc = __int_as_float(moved);
        };
        auto walk = [&](const Ahead &of) {
#pragma unroll
            for (int w = 0; w < WORDS; ++w) add(of.v[w]);
        };
        const bool last_round = k0 + 64 > walks;    // its last entry is the end: a leap, nothing to walk
        read(even, 0);
        for (int l = 0;;) {
            read(odd, l + 1 < 64 ? l + 1 : 63);
            leap(even);
            if (++l == here && last_round) break;
            walk(even);
            if (l == here) break;
            read(even, l + 1 < 64 ? l + 1 : 63);
            leap(odd);
            if (++l == here && last_round) break;
            walk(odd);
            if (l == here) break;
        }
    }
    if (__builtin_amdgcn_readfirstlane(wrong)) {    // a guess on the other side of a power of two: rare, so in full
        acc = before_all;
        for (int part = 0; part < 64 * PARTS; ++part)
#pragma unroll
            for (int w = 0; w < WORDS; ++w) add(words_of(part)[w]);
    }
    return acc;
}

// LDS of the sums of V vectors
template <int V> struct SumScratch {
    __attribute__((aligned(16))) float sq[V * ORDERED_FLOATS + SQ_TAIL];
    OrderedScratch ordered[V];
    float ss[V];
};
static_assert(ORDERED_FLOATS >= SQ_CHUNK && ORDERED_MIN <= SQ_CHUNK, "both layouts fit");

// Sums of at most SQ_CHUNK staged squares: place(i) is where the square of element i of a vector of ORDERED_FLOATS goes, and
// zeros follow up to end(), which add nothing to a sum that is never negative; add(v, acc) is called by the whole wave v.
// LONG: whether a vector of ORDERED_MIN elements and more can come.  A kernel for shorter ones does not carry the code of
// ordered_sum (one norm of 64 values 3.8 us with it, 3.5 without).
template <bool LONG> struct Staged {
    int count, words;
    bool chain;
    __device__ explicit Staged(int n) : count(n), words(part_words(n)), chain(!LONG || n < ORDERED_MIN) {}
    __device__ int end() const { return chain ? (count + 31) & ~31 : 1024 * words; }
    __device__ int place(int i) const { return chain ? i : ordered_place(i, words); }
    __device__ __forceinline__ float add(const float *sq, float acc, OrderedScratch &scratch) const {
        if (chain) return add_staged(sq, end(), acc);
        switch (words) {
        case 1: return ordered_sum<1>(sq, acc, scratch);
        case 2: return ordered_sum<2>(sq, acc, scratch);
        case 3: return ordered_sum<3>(sq, acc, scratch);
        default: return ordered_sum<4>(sq, acc, scratch);
        }
    }
};

// The sums of squares of `vectors` (at most V) vectors of at most SQ_CHUNK elements that the threads already hold: val[v][k]
// is element SLOTS * tid + k of vector v (any value past the end).  RAGGED: n need not be a multiple of SLOTS.
template <int V, bool RAGGED>
__device__ __forceinline__ void chains_from_registers(const float (&val)[V][SLOTS], int vectors, int n,
                                                      SumScratch<V> &scratch, float (&ss)[V]) {
    static_assert(SLOTS == 4, "a thread's elements are 16 bytes");
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = SLOTS * tid;
    const Staged<true> staged(n);
    if (i < staged.end())
#pragma unroll
        for (int v = 0; v < V; ++v) {
            float square[SLOTS];
#pragma unroll
            for (int k = 0; k < SLOTS; ++k) square[k] = (RAGGED ? i + k : i) < n ? val[v][k] * val[v][k] : 0.0f;
            *(float4 *)&scratch.sq[v * ORDERED_FLOATS + staged.place(i)] = make_float4(square[0], square[1], square[2], square[3]);
        }
    __syncthreads();
    if (wave < vectors) {
        const float sum = staged.add(scratch.sq + wave * ORDERED_FLOATS, 0.0f, scratch.ordered[wave]);
        if ((tid & 63) == 0) scratch.ss[wave] = sum;
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < V; ++v) ss[v] = scratch.ss[v];
}

// A thread's elements i .. i + SLOTS - 1 of n, on any four-byte boundary; past the end the last elements again (n a multiple
// of SLOTS) or the last one (RAGGED, where the threads at the end ask for one at a time)
typedef float any_float4 __attribute__((ext_vector_type(4), aligned(4)));
template <bool RAGGED> __device__ __forceinline__ void load_slots(const float *from, int i, int n, float (&to)[SLOTS]) {
    if (RAGGED && i + SLOTS > n) {
#pragma unroll
        for (int k = 0; k < SLOTS; ++k) to[k] = from[i + k < n ? i + k : n - 1];
    } else {
        const any_float4 v = *(const any_float4 *)(from + (RAGGED || i < n ? i : n - SLOTS));
        to[0] = v.x; to[1] = v.y; to[2] = v.z; to[3] = v.w;
    }
}
template <bool RAGGED> __device__ __forceinline__ void store_slots(float *to, int i, int n, const float (&from)[SLOTS]) {
    if (RAGGED && i + SLOTS > n) {
#pragma unroll
        for (int k = 0; k < SLOTS; ++k)
            if (i + k < n) to[i + k] = from[k];
    } else if (i < n) {
        *(any_float4 *)(to + i) = any_float4{from[0], from[1], from[2], from[3]};
    }
}

// Serial sums of squares of V vectors of n floats: wave v adds vector v's squares left to right.  Returns the sums in
// ss_out[] on every thread; `bad` collects non-finite elements.
template <int V, bool LONG>
__device__ __forceinline__ void serial_square_sums(const float *const (&x)[V], int n, SumScratch<V> &scratch, float (&ss_out)[V],
                                   unsigned &bad) {
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float acc = 0.0f;
    for (int base = 0; base < n; base += SQ_CHUNK) {
        const Staged<LONG> staged(n - base < SQ_CHUNK ? n - base : SQ_CHUNK);
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const float *src = x[v] + base;
#pragma unroll
            for (int k = 0; k < SLOTS; ++k) {
                const int i = tid + k * THREADS;
                const float value = i < staged.count ? src[i] : 0.0f;
                bad |= nonfinite(value);
                if (i < staged.end()) scratch.sq[v * ORDERED_FLOATS + staged.place(i)] = value * value;
            }
        }
        __syncthreads();
        if (wave < V) acc = staged.add(scratch.sq + wave * ORDERED_FLOATS, acc, scratch.ordered[wave]);
        __syncthreads();
    }
    if (wave < V && (tid & 63) == 0) scratch.ss[wave] = acc;
    __syncthreads();
#pragma unroll
    for (int v = 0; v < V; ++v) ss_out[v] = scratch.ss[v];
    __syncthreads();
}

__device__ __forceinline__ float inverse_from_sum(float ss, int n, float eps) {
    const float mean = ss / (float)n;
    return pow_minus_half(mean + eps);
}

// kind 0: out = (x * inv) [* weight]            weight may be null
// kind 1: out = ((x * inv) * weight) * root     router input
// kind 2: out = residual + (x * inv) * weight   residual post-norm
struct NormArgs {
    const float *x, *weight, *residual;
    float *out;
    int n, kind;
    float eps, root;
    int *status;
};

template <bool LONG> __global__ __launch_bounds__(THREADS) void norm_cell_kernel(NormArgs a) {
    __shared__ SumScratch<1> scratch;
    if (*a.status != 0) return;
    unsigned bad = !(a.eps >= 0.0f) || nonfinite(a.eps);
    const float *const vec[1] = {a.x};
    float ss[1];
    serial_square_sums<1, LONG>(vec, a.n, scratch, ss, bad);
    const float inv = inverse_from_sum(ss[0], a.n, a.eps);
    bad |= nonfinite(inv);
    float root = a.root;
    if (a.kind == 1 && !(root > 0.0f)) root = 1.0f / det_sqrtf((float)a.n);
    auto value = [&](int i, unsigned &flag) {
        float y = a.x[i] * inv;
        if (a.weight) { const float w = a.weight[i]; flag |= nonfinite(w); y = y * w; }
        if (a.kind == 1) y = y * root;
        flag |= nonfinite(y);
        if (a.kind == 2) {
            const float r = a.residual[i];
            y = r + y;
            flag |= nonfinite(r) | nonfinite(y);
        }
        return y;
    };
    each_element(a.n, [&](int i) { (void)value(i, bad); });
    if (__syncthreads_or((int)bad)) {
        if (threadIdx.x == 0) *a.status = -1;
        return;
    }
    unsigned ignored = 0;
    each_element(a.n, [&](int i) { a.out[i] = value(i, ignored); });
}

// One pass over the residual for the three vectors a feed-forward block derives from it:
// norm_a = (r * inv) * w1, router_in = ((r * inv) * scale) * root, norm_b = (r * inv) * w2.
struct PreArgs {
    const float *residual, *w1, *w2, *router_scale;
    float *norm_a, *norm_b, *router_in;
    int n;
    float eps;
    int *status;               // written, not only set: this kernel opens the block
};

// n <= SQ_CHUNK, a multiple of SLOTS: every input is requested once, up front, and lives in registers from then on; a
// thread has SLOTS consecutive elements
__global__ __launch_bounds__(THREADS) void ffn_pre_small_kernel(PreArgs a) {
    __shared__ SumScratch<1> scratch;
    unsigned bad = !(a.eps >= 0.0f) || nonfinite(a.eps);
    const int i = SLOTS * (int)threadIdx.x;
    float r[1][SLOTS], w1[SLOTS], w2[SLOTS], rs[SLOTS];
    load_slots<false>(a.residual, i, a.n, r[0]);
    load_slots<false>(a.w1, i, a.n, w1);
    load_slots<false>(a.w2, i, a.n, w2);
    load_slots<false>(a.router_scale, i, a.n, rs);
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) bad |= nonfinite(r[0][k]) | nonfinite(w1[k]) | nonfinite(w2[k]) | nonfinite(rs[k]);
    float ss[1];
    chains_from_registers<1, false>(r, 1, a.n, scratch, ss);
    const float inv = inverse_from_sum(ss[0], a.n, a.eps);
    bad |= nonfinite(inv);
    const float root = 1.0f / det_sqrtf((float)a.n);
    float na[SLOTS], nb[SLOTS], ri[SLOTS];
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) {
        const float y = r[0][k] * inv;
        na[k] = y * w1[k];
        nb[k] = y * w2[k];
        ri[k] = (y * rs[k]) * root;
        bad |= nonfinite(y) | nonfinite(na[k]) | nonfinite(nb[k]) | nonfinite(ri[k]);
    }
    const bool failed = __syncthreads_or((int)bad);
    if (threadIdx.x == 0) *a.status = failed ? -1 : 0;
    if (failed) return;
    store_slots<false>(a.norm_a, i, a.n, na);
    store_slots<false>(a.norm_b, i, a.n, nb);
    store_slots<false>(a.router_in, i, a.n, ri);
}

__global__ __launch_bounds__(THREADS) void ffn_pre_kernel(PreArgs a) {
    __shared__ SumScratch<1> scratch;
    unsigned bad = !(a.eps >= 0.0f) || nonfinite(a.eps);
    const float *const vec[1] = {a.residual};
    float ss[1];
    serial_square_sums<1, true>(vec, a.n, scratch, ss, bad);
    const float inv = inverse_from_sum(ss[0], a.n, a.eps);
    bad |= nonfinite(inv);
    const float root = 1.0f / det_sqrtf((float)a.n);
    each_element(a.n, [&](int i) {
        const float y = a.residual[i] * inv, w1 = a.w1[i], w2 = a.w2[i], rs = a.router_scale[i];
        bad |= nonfinite(w1) | nonfinite(w2) | nonfinite(rs) | nonfinite(y) | nonfinite(y * w1) | nonfinite(y * w2) |
               nonfinite((y * rs) * root);
    });
    const bool failed = __syncthreads_or((int)bad);
    if (threadIdx.x == 0) *a.status = failed ? -1 : 0;
    if (failed) return;
    each_element(a.n, [&](int i) {
        const float y = a.residual[i] * inv;
        a.norm_a[i] = y * a.w1[i];
        a.norm_b[i] = y * a.w2[i];
        a.router_in[i] = (y * a.router_scale[i]) * root;
    });
}

// out = (residual + norm(norm(dense) * wd + norm(routed) * wr) * wf) * scalar.  `other` is a second status word
// (that of the routed branch) or null; sum is n floats of global scratch.
struct CombineArgs {
    const float *residual, *dense, *routed, *wd, *wr, *wf;
    float *sum, *out;
    int n;
    float eps, scalar;
    int *status;
    const int *other;
    // when expert_out is given, routed (writable then) is first filled with sum_k expert_out[k] * weights[k], k ascending
    const float *expert_out, *weights;
    int topk;
};

// n <= SQ_CHUNK: one load phase, everything else in registers and LDS; a thread has SLOTS consecutive elements (RAGGED: n need not be
// a multiple of them).  Bound by what one compute unit can fetch (six vectors and topk expert outputs, 158 KB at 2816 and eight, in
// 2 us; a wait for each expert and four bytes per load took 7), then by the two rounds of sums, 3 us each.
template <bool RAGGED> __global__ __launch_bounds__(THREADS) void combine_small_kernel(CombineArgs a) {
    __shared__ SumScratch<2> scratch;
    unsigned bad = !(a.eps >= 0.0f) || nonfinite(a.eps) || nonfinite(a.scalar);
    // Every input is asked for before anything is waited for, the status words among them; the experts' outputs eight
    // at a time.
    const int status = *a.status, other = a.other ? *a.other : 0;
    const int i = SLOTS * (int)threadIdx.x;
    float dr[2][SLOTS], res[SLOTS], wd[SLOTS], wr[SLOTS], wf[SLOTS];
    load_slots<RAGGED>(a.dense, i, a.n, dr[0]);
    if (!a.expert_out) load_slots<RAGGED>(a.routed, i, a.n, dr[1]);
    else {
#pragma unroll
        for (int k = 0; k < SLOTS; ++k) dr[1][k] = 0.0f;
        for (int e0 = 0; e0 < a.topk; e0 += 8) {
            float term[8][SLOTS], w[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (e0 + e >= a.topk) break;
                w[e] = a.weights[e0 + e];
                load_slots<RAGGED>(a.expert_out + (size_t)(e0 + e) * a.n, i, a.n, term[e]);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (e0 + e >= a.topk) break;
#pragma unroll
                for (int k = 0; k < SLOTS; ++k) {
                    const float product = term[e][k] * w[e];
                    dr[1][k] = dr[1][k] + product;
                }
            }
        }
    }
    load_slots<RAGGED>(a.residual, i, a.n, res);
    load_slots<RAGGED>(a.wd, i, a.n, wd);
    load_slots<RAGGED>(a.wr, i, a.n, wr);
    load_slots<RAGGED>(a.wf, i, a.n, wf);
    if (status != 0) return;
    if (other != 0) {
        if (threadIdx.x == 0) *a.status = -1;
        return;
    }
#pragma unroll
    for (int k = 0; k < SLOTS; ++k)
        bad |= nonfinite(res[k]) | nonfinite(wd[k]) | nonfinite(wr[k]) | nonfinite(wf[k]) | nonfinite(dr[0][k]) |
               nonfinite(dr[1][k]);
    // Two rounds of sums through the same instructions (twice the code is twice the time to fetch it): the two branches,
    // then their sum in dr[0].
    float inv = 0.0f;
#pragma unroll 1
    for (int vectors = 2; vectors >= 1; --vectors) {
        float ss[2];
        chains_from_registers<2, RAGGED>(dr, vectors, a.n, scratch, ss);
        // odd lanes see to the routed branch
        const bool odd = (threadIdx.x & 1) != 0 && vectors == 2;
        inv = inverse_from_sum(odd ? ss[1] : ss[0], a.n, a.eps);
        bad |= nonfinite(inv);
        if (vectors == 1) break;
        const float inv_d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv), 0));
        const float inv_r = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv), 1));
#pragma unroll
        for (int k = 0; k < SLOTS; ++k) {
            const float d0 = dr[0][k] * inv_d, r0 = dr[1][k] * inv_r;
            const float d = d0 * wd[k], r = r0 * wr[k];
            dr[0][k] = d + r;
            bad |= nonfinite(d0) | nonfinite(r0) | nonfinite(d) | nonfinite(r) | nonfinite(dr[0][k]);
        }
    }
    float y[SLOTS];
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) {
        const float f0 = dr[0][k] * inv;
        const float f = f0 * wf[k];
        y[k] = (res[k] + f) * a.scalar;
        bad |= nonfinite(f0) | nonfinite(f) | nonfinite(y[k]);
    }
    if (__syncthreads_or((int)bad)) {
        if (threadIdx.x == 0) *a.status = -1;
        return;
    }
    store_slots<RAGGED>(a.out, i, a.n, y);
}

__global__ __launch_bounds__(THREADS) void combine_cell_kernel(CombineArgs a) {
    __shared__ SumScratch<2> scratch;
    __shared__ SumScratch<1> scratch_sum;
    if (*a.status != 0) return;
    if (a.other && *a.other != 0) {
        if (threadIdx.x == 0) *a.status = -1;
        return;
    }
    unsigned bad = !(a.eps >= 0.0f) || nonfinite(a.eps) || nonfinite(a.scalar);
    if (a.expert_out) {                                 // each thread later reads back only what it wrote here
        float *routed = const_cast<float *>(a.routed);
        for (int base = 0; base < a.n; base += SQ_CHUNK) {
            float sum[SLOTS];
#pragma unroll
            for (int k = 0; k < SLOTS; ++k) sum[k] = 0.0f;
            for (int e = 0; e < a.topk; ++e) {
                const float w = a.weights[e];
#pragma unroll
                for (int k = 0; k < SLOTS; ++k) {
                    const int i = base + (int)threadIdx.x + k * THREADS;
                    if (i < a.n) {
                        const float term = a.expert_out[(size_t)e * a.n + i] * w;
                        sum[k] = sum[k] + term;
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < SLOTS; ++k) {
                const int i = base + (int)threadIdx.x + k * THREADS;
                if (i < a.n) routed[i] = sum[k];
            }
        }
    }
    const float *const vec[2] = {a.dense, a.routed};
    float ss[2];
    serial_square_sums<2, true>(vec, a.n, scratch, ss, bad);
    const float inv_d = inverse_from_sum(ss[0], a.n, a.eps), inv_r = inverse_from_sum(ss[1], a.n, a.eps);
    bad |= nonfinite(inv_d) | nonfinite(inv_r);
    each_element(a.n, [&](int i) {
        const float wd = a.wd[i], wr = a.wr[i], res = a.residual[i], wf = a.wf[i];
        const float d0 = a.dense[i] * inv_d, r0 = a.routed[i] * inv_r;
        const float d = d0 * wd, r = r0 * wr;
        const float s = d + r;
        bad |= nonfinite(res) | nonfinite(wd) | nonfinite(wr) | nonfinite(wf) | nonfinite(d0) | nonfinite(r0) | nonfinite(d) | nonfinite(r) |
               nonfinite(s);
        a.sum[i] = s;
    });
    const float *const vec2[1] = {a.sum};               // a thread reads back the elements it wrote itself
    float ss_sum[1];
    serial_square_sums<1, true>(vec2, a.n, scratch_sum, ss_sum, bad);
    const float inv_f = inverse_from_sum(ss_sum[0], a.n, a.eps);
    bad |= nonfinite(inv_f);
    each_element(a.n, [&](int i) {
        const float f0 = a.sum[i] * inv_f;
        const float f = f0 * a.wf[i];
        const float y = (a.residual[i] + f) * a.scalar;
        bad |= nonfinite(f0) | nonfinite(f) | nonfinite(y);
    });
    if (__syncthreads_or((int)bad)) {
        if (threadIdx.x == 0) *a.status = -1;
        return;
    }
    each_element(a.n, [&](int i) {
        const float f = (a.sum[i] * inv_f) * a.wf[i];
        a.out[i] = (a.residual[i] + f) * a.scalar;
    });
}

constexpr int WIDE = 256;             // threads per workgroup of the grid-wide elementwise kernels

__global__ __launch_bounds__(WIDE) void finite_check_kernel(const float *x, size_t n, int *status) {
    unsigned bad = 0;
    for (size_t i = (size_t)blockIdx.x * WIDE + threadIdx.x; i < n; i += (size_t)gridDim.x * WIDE) bad |= nonfinite(x[i]);
    if (__syncthreads_or((int)bad) && threadIdx.x == 0) *status = -1;      // every writer stores the same value
}

__global__ __launch_bounds__(WIDE) void softcap_kernel(float *logits, size_t n, float cap, const int *status) {
    if (*status != 0) return;
    const size_t i = (size_t)blockIdx.x * WIDE + threadIdx.x;
    if (i < n) logits[i] = cap * det_tanhf(logits[i] / cap);
}

__global__ void merge_status_kernel(int *status, const int *other) {
    if (*other != 0) *status = -1;
}

bool launched() { return hipGetLastError() == hipSuccess; }

}  // namespace

int norm_cell_launch(int kind, const float *x, const float *weight, const float *residual, float *out, int n, float eps,
                     float root, int *status, hipStream_t stream) {
    if (!x || !out || !status || n < 1 || kind < 0 || kind > 2 || (kind != 0 && !weight) || (kind == 2 && !residual))
        return -1;
    NormArgs a = {x, weight, residual, out, n, kind, eps, root, status};
    if (n < ORDERED_MIN) norm_cell_kernel<false><<<dim3(1), dim3(THREADS), 0, stream>>>(a);
    else norm_cell_kernel<true><<<dim3(1), dim3(THREADS), 0, stream>>>(a);
    return launched() ? 0 : -1;
}

int ffn_pre_launch(const float *residual, const float *w1, const float *w2, const float *router_scale, float *norm_a,
                   float *norm_b, float *router_in, int n, float eps, int *status, hipStream_t stream) {
    if (!residual || !w1 || !w2 || !router_scale || !norm_a || !norm_b || !router_in || !status || n < 1) return -1;
    PreArgs a = {residual, w1, w2, router_scale, norm_a, norm_b, router_in, n, eps, status};
    if (n <= SQ_CHUNK && n % SLOTS == 0) ffn_pre_small_kernel<<<dim3(1), dim3(THREADS), 0, stream>>>(a);
    else ffn_pre_kernel<<<dim3(1), dim3(THREADS), 0, stream>>>(a);
    return launched() ? 0 : -1;
}

int combine_cell_launch(const float *residual, const float *dense, const float *routed, const float *wd, const float *wr,
                        const float *wf, float *sum_scratch, float *out, int n, float eps, float scalar, int *status,
                        const int *other_status, const float *expert_out, const float *weights, int topk,
                        hipStream_t stream) {
    if (!residual || !dense || !routed || !wd || !wr || !wf || !sum_scratch || !out || !status || n < 1 ||
        (expert_out && (!weights || topk < 1)))
        return -1;
    CombineArgs a = {residual, dense, routed, wd, wr, wf, sum_scratch, out, n, eps, scalar, status, other_status,
                     expert_out, weights, topk};
    if (n > SQ_CHUNK) combine_cell_kernel<<<dim3(1), dim3(THREADS), 0, stream>>>(a);
    else if (n % SLOTS == 0) combine_small_kernel<false><<<dim3(1), dim3(THREADS), 0, stream>>>(a);
    else combine_small_kernel<true><<<dim3(1), dim3(THREADS), 0, stream>>>(a);
    return launched() ? 0 : -1;
}

int softcap_cell_launch(float *logits, size_t n, float cap, int *status, hipStream_t stream) {
    if (!logits || !status || n < 1 || !(cap > 0.0f) || !(cap < __builtin_inff())) return -1;
    const size_t blocks = (n + WIDE - 1) / WIDE;
    finite_check_kernel<<<dim3((unsigned)(blocks < 1024 ? blocks : 1024)), dim3(WIDE), 0, stream>>>(logits, n, status);
    if (!launched()) return -1;
    softcap_kernel<<<dim3((unsigned)blocks), dim3(WIDE), 0, stream>>>(logits, n, cap, status);
    return launched() ? 0 : -1;
}

int merge_status_launch(int *status, const int *other, hipStream_t stream) {
    merge_status_kernel<<<dim3(1), dim3(1), 0, stream>>>(status, other);
    return launched() ? 0 : -1;
}

}  // namespace mi355
