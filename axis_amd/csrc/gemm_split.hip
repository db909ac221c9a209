// fp32 products through three bf16 planes per operand (gemm_split.hpp has the arithmetic).
//
// A block stages 32-deep steps of both operands in LDS as three planes of rows [t][32] bf16; the
// fp32 values are loaded as gemm.hip's loaders do and split in registers on their way to LDS, so
// nothing is staged in device memory and each element is split once per block that reads it.
//
// What bounds it: power.  On random data a register-only loop of the instruction reaches 2.10 PFLOP/s
// (zeros: 2.44; v_mfma_f32_32x32x16_bf16: 1.86 random, 2.46 zeros, hence the smaller instruction), and
// in this kernel the matrix pipe is busy 0.64 of the cycles at about 2.0 GHz, with LDS 0.28 busy.
//
// Sums: the six partial products of a 32-deep step form a chain that starts from zero, smallest
// first, and one fp32 add takes it into the accumulator.  Accumulating the six instructions directly
// is 4-5% faster at 4096^3 and leaves an error of 8.9e-7 against 64 bits, as the fp32 matrix
// instruction does; the chain leaves 2.3e-7.  The instruction's own roundings lean one way whatever
// the sign (a weight gradient over 262,144 pixels was 7.9e-7 off, growing with the pixels; fp32
// instruction: 3.3e-7), so every other step runs on the negated first operand and is subtracted: the
// lean cancels, and the negation is an operand modifier.
//
// Values the planes cannot hold (infinities, NaN, magnitudes that round to infinity in bf16, blocks
// whose operand lies wholly below 2^-63, where the low planes approach the end of the exponent
// range) are found at the end of a block -- any such value leaves its accumulators non-finite, and
// the staged exponents are or-ed as they pass -- and the block then computes its tile again with
// the fp32 matrix instruction.  In a block with ordinary magnitudes too, an element below 2^-110 (1e-33)
// may lose what its low planes would hold below 2^-126, the smallest normal number: at most 2^-126 times
// what it is multiplied with, which shows only where a whole row of sums is that small.
#include <algorithm>

#include "gemm_split.hpp"

namespace axis {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kDepth = 32;  // reduction depth of a step

__device__ __forceinline__ uint32_t round2(float a, float b) {
    const floatx2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float low_half(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float high_half(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

// a and b as packed bf16 planes (the subtractions are exact).
__device__ __forceinline__ void split2(float a, float b, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
    hi = round2(a, b);
    a -= low_half(hi);
    b -= high_half(hi);
    mid = round2(a, b);
    a -= low_half(mid);
    b -= high_half(mid);
    lo = round2(a, b);
}

// The sign a step's first operand is staged with and its chains are added with.
struct Plus {
    __device__ __forceinline__ float operator()(float x) const { return x; }
    __device__ __forceinline__ void add(floatx4 &acc, floatx4 t) const { acc += t; }
};
struct Minus {
    __device__ __forceinline__ float operator()(float x) const { return -x; }
    __device__ __forceinline__ void add(floatx4 &acc, floatx4 t) const { acc -= t; }
};
// chosen at run time, where a loop unrolled by two would not fit the registers
struct Flip {
    uint32_t bit;
    __device__ __forceinline__ float operator()(float x) const {
        return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) ^ bit);
    }
    __device__ __forceinline__ void add(floatx4 &acc, floatx4 t) const {
        const float s = __builtin_bit_cast(float, 0x3f800000u ^ bit);
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[v] = __builtin_fmaf(t[v], s, acc[v]);
    }
};

// Vectors and LDS placement of one operand's BT rows for NT threads.
//
// A plane holds row slot p (64 bytes) at 64 p, its 16-byte chunk c (eight reduction elements, one
// MFMA operand) at chunk position c ^ ((p / 2) % 4): an operand read (16 consecutive slots, one
// chunk) and the stores below meet no bank conflict.  Tile row t sits in slot
// 64 (t / 64) + 16 (t % 4) + (t % 64) / 4, so block a of a wave (slots 16 a + l of its 64) holds rows
// 4 l + a and a lane's four column blocks are four adjacent output columns.
//
// r-contiguous: vector idx is four reduction elements of slot idx / 8; eight lanes read 128
// contiguous bytes of a row and store 64 contiguous bytes of each plane.
// t-contiguous: a thread holds patches of kRows (4 or 2) reduction elements by four rows t, loaded
// along t and stored along the reduction, 2 kRows bytes per row and plane.  Consecutive lanes take
// eight row quads, then the patches that complete a 16-byte chunk, then the rest.
template <int BT, int NT, bool RCONTIG>
struct PlaneStaging {
    static constexpr int kElems = BT * kDepth / NT;
    static constexpr int kVecs = kElems / 4;
    static constexpr int kRows = RCONTIG ? 1 : (kVecs < 4 ? kVecs : 4);
    static constexpr int kPatches = kVecs / kRows;
    static constexpr int kPlane = BT * 64;      // bytes
    static constexpr int kUnits = RCONTIG ? kVecs : 4 * kPatches;  // store() steps, see below
    static constexpr int kQuads = BT / 4;       // row quads
    static_assert(RCONTIG || kRows == 4 || kRows == 2, "patches of four or two reduction elements");
    float reg[kElems];
    uint32_t seen = 0;  // or of the hi planes: exponents that passed

    static __device__ __forceinline__ int slot_row(int p) { return (p & ~63) | ((p & 15) << 2) | ((p >> 4) & 3); }
    static __device__ __forceinline__ int line_r(int idx) { return (idx & 7) * 4; }
    static __device__ __forceinline__ int line_t(int idx) { return slot_row(idx >> 3); }
    // patch idx -> row quad and first reduction element / kRows
    static constexpr int kIn = kRows == 4 ? 1 : 2;  // bits of patches per chunk
    static __device__ __forceinline__ int patch_u(int idx) {
        return (idx & 7) | (((idx >> (3 + kIn)) & (kQuads / 8 - 1)) << 3);
    }
    static __device__ __forceinline__ int patch_q(int idx) {
        return ((idx >> 3) & ((1 << kIn) - 1)) | ((idx / (kQuads << kIn)) << kIn);
    }
    static_assert(RCONTIG || NT % (kQuads << kIn) == 0, "a thread's patches share their rows");
    static __device__ __forceinline__ int vec_t(int tid) { return 4 * patch_u(tid); }
    static __device__ __forceinline__ int vec_r(int tid, int e) {
        return kRows * patch_q(tid + (e / kRows) * NT) + e % kRows;
    }

    // Byte offset of the thread's vector (patch) `i` in a plane; a patch's row j is 1024 j further.
    static __device__ __forceinline__ int place(int tid, int i) {
        if constexpr (RCONTIG) {
            const int p = tid >> 3, q = tid & 7;  // NT / 8 slots further per vector: the same swizzle
            return p * 64 + (((q >> 1) ^ ((p >> 1) & 3)) << 4) + (q & 1) * 8 + i * (NT / 8) * 64;
        } else {
            const int u = patch_u(tid), q = patch_q(tid + i * NT);
            const int p = 64 * (u >> 4) + (u & 15);
            const int chunk = kRows == 4 ? q >> 1 : q >> 2, in = kRows == 4 ? (q & 1) * 8 : (q & 3) * 4;
            return p * 64 + ((chunk ^ ((p >> 1) & 3)) << 4) + in;
        }
    }

    // Splits and stores unit `unit` of the thread's values times sign: one vector, or one row of a patch.
    template <class Sign>
    __device__ __forceinline__ void store(char *__restrict__ planes, int tid, int unit, Sign sign) {
        auto value = [&](int i) { return sign(reg[i]); };
        if constexpr (RCONTIG || kRows == 4) {
            float v[4];
            int at;
            if constexpr (RCONTIG) {
#pragma unroll
                for (int c = 0; c < 4; ++c) v[c] = value(unit * 4 + c);
                at = place(tid, unit);
            } else {
                const int patch = unit / 4, j = unit % 4;
#pragma unroll
                for (int c = 0; c < 4; ++c) v[c] = value((patch * 4 + c) * 4 + j);
                at = place(tid, patch) + j * 1024;
            }
            uint32_t h0, h1, m0, m1, l0, l1;
            split2(v[0], v[1], h0, m0, l0);
            split2(v[2], v[3], h1, m1, l1);
            seen |= h0 | h1;
            *reinterpret_cast<u32x2 *>(planes + at) = u32x2{h0, h1};
            *reinterpret_cast<u32x2 *>(planes + at + kPlane) = u32x2{m0, m1};
            *reinterpret_cast<u32x2 *>(planes + at + 2 * kPlane) = u32x2{l0, l1};
        } else {
            const int patch = unit / 4, j = unit % 4;
            uint32_t h, m, l;
            split2(value(patch * 8 + j), value(patch * 8 + 4 + j), h, m, l);
            seen |= h;
            const int at = place(tid, patch) + j * 1024;
            *reinterpret_cast<uint32_t *>(planes + at) = h;
            *reinterpret_cast<uint32_t *>(planes + at + kPlane) = m;
            *reinterpret_cast<uint32_t *>(planes + at + 2 * kPlane) = l;
        }
    }

    // The same values as fp32 rows [slot][kPitch] (the recomputation's layout).
    static constexpr int kPitch = kDepth + 4;
    __device__ __forceinline__ void store_fp32(float *__restrict__ rows, int tid) const {
#pragma unroll
        for (int e = 0; e < kVecs; ++e) {
            if constexpr (RCONTIG) {
                const int idx = tid + e * NT;
                *reinterpret_cast<floatx4 *>(rows + (idx >> 3) * kPitch + (idx & 7) * 4) =
                    floatx4{reg[e * 4], reg[e * 4 + 1], reg[e * 4 + 2], reg[e * 4 + 3]};
            } else {
                const int u = patch_u(tid);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    rows[(64 * (u >> 4) + 16 * j + (u & 15)) * kPitch + vec_r(tid, e)] = reg[e * 4 + j];
            }
        }
    }
};

// Dense operand: element (t, r) at base[t * s_t + r * s_r], one of the strides 1.  As gemm.hip's
// DenseLoader: a wave-uniform buffer resource per step and 32-bit lane offsets fixed at init (the
// host keeps them below 2^29 elements).  AL: bases, pitches and extents let every vector start on
// 16 bytes and end inside its row.  Otherwise vectors start on any element (buffer loads need
// 4-byte alignment only), and those that may cross the end of a row -- in the last, partial step of
// an r-contiguous operand, in the last tile of a t-contiguous one -- are read as four single
// elements, each with its own bound.
template <int BT, int NT, bool RCONTIG, bool AL, bool TAPS>
struct PlaneDense : PlaneStaging<BT, NT, RCONTIG> {
    using S = PlaneStaging<BT, NT, RCONTIG>;
    const float *tile_base;
    uint32_t voff[S::kVecs];
    int64_t s_r;
    int32_t rows_left;  // rows of the operand from the tile's first
    TapSteps taps{};

    __device__ __forceinline__ void init(const float *b, int64_t st, int64_t sr, int64_t t0, int64_t t_end, int tid) {
        s_r = sr;
        tile_base = uniform_ptr(b + t0 * st);
        rows_left = t_end - t0 < BT ? (int32_t)(t_end - t0) : BT;
#pragma unroll
        for (int e = 0; e < S::kVecs; ++e) {
            const int t = RCONTIG ? S::line_t(tid + e * NT) : S::vec_t(tid);
            const int r = RCONTIG ? S::line_r(tid + e * NT) : S::vec_r(tid, e);
            voff[e] = t < rows_left ? (uint32_t)(t * st + r * sr) * 4u : kOutside;
        }
    }
    // Whether every vector of every whole step lies inside its rows.
    __device__ __forceinline__ bool inside() const { return RCONTIG || AL || rows_left == BT; }
    // FAST: a whole step of an operand that is inside() (no bound is tested).
    template <bool FAST>
    __device__ __forceinline__ void load(int64_t r0, int32_t room, int tid) {
        const int64_t step = TAPS ? taps.step(r0) : r0 * s_r;
        if constexpr (RCONTIG) {
            const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(uniform_ptr(tile_base + step));
            if (AL || FAST || room >= kDepth) {
#pragma unroll
                for (int e = 0; e < S::kVecs; ++e)
                    buffer_into<4>(this->reg + e * 4, rsrc,
                                   FAST || S::line_r(tid + e * NT) < room ? voff[e] : kOutside);
            } else {
#pragma unroll
                for (int e = 0; e < S::kVecs; ++e)
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        buffer_into<1>(this->reg + e * 4 + c, rsrc,
                                       S::line_r(tid + e * NT) + c < room ? voff[e] + 4 * c : kOutside);
            }
        } else {
            // rows past the step's depth start at or after byte room * s_r * 4 of the step
            const int32_t bytes = FAST || room >= kDepth ? 0x7fffffff : (int32_t)(room * s_r * 4);
            const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(uniform_ptr(tile_base + step), bytes);
            if (AL || FAST || rows_left == BT) {
#pragma unroll
                for (int e = 0; e < S::kVecs; ++e) buffer_into<4>(this->reg + e * 4, rsrc, voff[e]);
            } else {
#pragma unroll
                for (int e = 0; e < S::kVecs; ++e)
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        buffer_into<1>(this->reg + e * 4 + c, rsrc,
                                       S::vec_t(tid) + c < rows_left ? voff[e] + 4 * c : kOutside);
            }
        }
    }
};

// XMODE: 0 dense X, 2 convolution cols mode, 3 cols mode over aligned pixel steps, 4 rows mode with tap
// steps in block-major order, 5 rows mode with per-lane taps.  STAGES LDS stages of both operands' planes.
template <int BM, int BN, int WM, int WN, int STAGES, int PF, bool XR, bool YR, bool AL, int XMODE>
__global__ void __launch_bounds__(WM *WN * 64, BM / WM == 32 ? 3 : 2) split_gemm_kernel(GemmParams p) {
    constexpr int NT = WM * WN * 64;
    constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 16, FN = TN / 16;
    static_assert((TM == 64 || TM == 32) && (TN == 64 || TN == 32), "waves of 64 or 32 rows and columns");
    using SX = PlaneStaging<BM, NT, XR>;
    using LX = std::conditional_t<
        XMODE == 0, PlaneDense<BM, NT, XR, AL, false>,
        std::conditional_t<XMODE == 2, ConvColsLoader<SX, BM, kDepth, NT, 4>,
                           std::conditional_t<XMODE == 3, ConvColsStepLoader<SX, BM, kDepth, NT, 4>,
                                              ConvRowsBufferLoader<SX, BM, kDepth, NT, 4, XMODE == 4>>>>;
    using LY = PlaneDense<BN, NT, YR, AL, XMODE == 4>;
    constexpr int PX = SX::kPlane, PY = LY::kPlane, kStage = 3 * (PX + PY);
    static_assert((BM + BN) * SX::kPitch * 4 <= STAGES * kStage, "the recomputation's rows fit the stages");
    __shared__ __attribute__((aligned(16))) char lds[STAGES * kStage];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave % WM, wn = wave / WM;
    const int quad = lane >> 4, l16 = lane & 15;

    // XCD-aware order as gemm_body's; inside a slice, groups of 8 row panels, column-major, so that
    // the blocks an XCD runs at once share panels of both operands.
    const uint32_t tiles = (uint32_t)p.tiles_m * (uint32_t)p.tiles_n;
    const uint32_t L = blockIdx.x;
    const uint32_t logical = L < 8u * p.xcd_span ? (L % 8u) * p.xcd_span + L / 8u : L;
    const uint32_t tile = logical % tiles;
    const uint32_t slice = logical / tiles;
    const uint32_t per_group = 8u * (uint32_t)p.tiles_n;
    const uint32_t group = tile / per_group, first = group * 8u;
    const uint32_t height = (uint32_t)p.tiles_m - first < 8u ? (uint32_t)p.tiles_m - first : 8u;
    const uint32_t inside = tile - group * per_group;
    const int64_t i0 = (int64_t)(first + inside % height) * BM;
    const int64_t j0 = (int64_t)(inside / height) * BN;
    const int split = (int)(slice % (uint32_t)p.splits);
    const int64_t batch = (int64_t)(slice / (uint32_t)p.splits);
    const int64_t r_begin = (int64_t)split * p.k_chunk;
    const int64_t r_end = r_begin + p.k_chunk < p.k ? r_begin + p.k_chunk : p.k;
    const int32_t steps = r_begin < r_end ? (int32_t)((r_end - r_begin + kDepth - 1) / kDepth) : 0;
    const int32_t tail = (int32_t)(r_end - r_begin - (int64_t)(steps - 1) * kDepth);
    auto room_of = [&](int32_t step) { return step == steps - 1 ? tail : kDepth; };

    // PF register sets: step j waits in set j % PF on its way to LDS
    LX lx[PF];
    LY ly[PF];
    if constexpr (XMODE == 0)
        lx[0].init(p.x + batch * p.x_batch, p.x_si, p.x_sr, i0, p.m, tid);
    else
        lx[0].init(p.conv, i0, p.m, tid);
    ly[0].init(p.y + batch * p.y_batch, p.y_sj, p.y_sr, j0, p.n, tid);
    ly[0].taps = p.ytaps;
#pragma unroll
    for (int f = 1; f < PF; ++f) lx[f] = lx[0], ly[f] = ly[0];
    auto load_x = [&](int32_t step, int set, auto fast) {
        const int64_t r0 = r_begin + (int64_t)step * kDepth;
        if constexpr (XMODE == 0)
            lx[set].template load<decltype(fast)::value>(r0, room_of(step), tid);
        else
            lx[set].load(p.conv, r0, room_of(step), tid);
    };
    auto load_y = [&](int32_t step, int set, auto fast) {
        ly[set].template load<decltype(fast)::value>(r_begin + (int64_t)step * kDepth, room_of(step), tid);
    };
    const std::false_type any{};

    floatx4 acc[FM][FN];
    auto clear = [&]() {
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int b = 0; b < FN; ++b) acc[a][b] = floatx4{0.f, 0.f, 0.f, 0.f};
    };
    clear();

    // operand reads: slot 16 a + l16 of the wave's rows, chunk `quad`
    const int x_at = (wm * TM + l16) * 64 + ((quad ^ ((l16 >> 1) & 3)) << 4);
    const int y_at = 3 * PX + (wn * TN + l16) * 64 + ((quad ^ ((l16 >> 1) & 3)) << 4);

    auto store_all = [&](char *stage, auto sign) {
#pragma unroll
        for (int u = 0; u < LX::kUnits; ++u) lx[0].store(stage, tid, u, sign);
#pragma unroll
        for (int u = 0; u < LY::kUnits; ++u) ly[0].store(stage + 3 * PX, tid, u, Plus{});
    };

    // One staged step; in an odd one the first operand is staged negated and the chains subtracted (the
    // instruction's roundings lean one way, see the top).  between(b): work placed with column block
    // b's MFMAs (the next stage's splits and stores, the loads after them).
    // G column blocks run their chains together: four or more independent MFMAs per link of the chain
    // cover the instruction's latency.
    constexpr int G = FM == 2 ? 2 : 1;
    auto compute = [&](const char *stage, auto sign, auto between) {
        bf16x8 xa[FM][3], yb[2][G][3];
        floatx4 t[2][G][FM];
        auto read_y = [&](int b) {
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    yb[b & 1][g][q] = *reinterpret_cast<const bf16x8 *>(stage + y_at + (b * G + g) * 1024 + q * PY);
        };
        auto add = [&](int b) {
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int a = 0; a < FM; ++a) sign.add(acc[a][b * G + g], t[b & 1][g][a]);
        };
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int q = 0; q < 3; ++q) xa[a][q] = *reinterpret_cast<const bf16x8 *>(stage + x_at + a * 1024 + q * PX);
        read_y(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < FN / G; ++b) {
            if (b + 1 < FN / G) read_y(b + 1);
            between(b);
            // the chain of six, smallest first; the columns before are added while these run
            constexpr int kx[6] = {0, 2, 1, 0, 1, 0}, ky[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
            for (int s = 0; s < 6; ++s) {
#pragma unroll
                for (int g = 0; g < G; ++g)
#pragma unroll
                    for (int a = 0; a < FM; ++a) {
                        const floatx4 c = s == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : t[b & 1][g][a];
                        t[b & 1][g][a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[a][kx[s]], yb[b & 1][g][ky[s]], c, 0, 0, 0);
                    }
                if (s == 0 && b > 0) add(b - 1);
            }
            if constexpr (STAGES == 2) {
                // two vector instructions and now and then an LDS one behind each MFMA
#pragma unroll
                for (int g = 0; g < 6 * FM * G; ++g) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
                    if (g % 4 == 3) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                    if (g % 8 == 1) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        add(FN / G - 1);
    };

    if constexpr (STAGES == 2) {
        // Step s: its stage is computed while step s + 1 goes from its registers to the other stage,
        // whose readers passed the last barrier; the registers then take step s + 1 + PF.  Past the
        // end the last step is loaded and stored again, where nothing reads it, so that the loop has
        // no branch for the scheduler to stop at.
        const int32_t last = steps - 1;
        if (steps > 0) {
#pragma unroll
            for (int f = 0; f < PF; ++f) load_x(f < last ? f : last, f, any), load_y(f < last ? f : last, f, any);
            store_all(lds, Plus{});
            load_x(PF < last ? PF : last, 0, any);
            load_y(PF < last ? PF : last, 0, any);
        }
        __syncthreads();
        auto step = [&](int32_t s, const char *cur, char *next, auto sign, auto fast) {
            using Next = std::conditional_t<std::is_same_v<decltype(sign), Plus>, Minus, Plus>;
            constexpr int set = std::is_same_v<Next, Plus> ? 0 : 1 % PF;  // of step s + 1
            constexpr int kHalf = (FN / G + 1) / 2;
            const int32_t ahead = s + 1 + PF < last ? s + 1 + PF : last;
            compute(cur, sign, [&](int b) {
#pragma unroll
                for (int u = 0; u < LX::kUnits; ++u)
                    if (u * kHalf / LX::kUnits == b) lx[set].store(next, tid, u, Next{});
#pragma unroll
                for (int u = 0; u < LY::kUnits; ++u)
                    if (FN / G - kHalf + u * kHalf / LY::kUnits == b) ly[set].store(next + 3 * PX, tid, u, Plus{});
                if (b == FN / G - kHalf) load_x(ahead, set, fast);
                if (b == FN / G - 1) load_y(ahead, set, fast);
            });
            __syncthreads();
        };
        static_assert(PF == 1 || PF == 2, "sets rotate with the stages");
        int32_t s = 0;
        // Operands without aligned rows: whole steps first, then the ones that load the last step.
        if constexpr (!AL) {
            if (lx[0].inside() && ly[0].inside())
                for (; s + 2 + PF < last; s += 2) {
                    step(s, lds, lds + kStage, Plus{}, std::true_type{});
                    step(s + 1, lds + kStage, lds, Minus{}, std::true_type{});
                }
        }
        for (; s < steps; s += 2) {
            step(s, lds, lds + kStage, Plus{}, any);
            if (s + 1 < steps) step(s + 1, lds + kStage, lds, Minus{}, any);
        }
    } else {
        static_assert(PF == 1 || STAGES == 2, "one register set with one stage");
        if (steps > 0) {
            load_x(0, 0, any);
            load_y(0, 0, any);
            store_all(lds, Plus{});
        }
        __syncthreads();
        Flip sign{0u};
        for (int32_t s = 0; s < steps; ++s) {
            if (s + 1 < steps) {
                load_x(s + 1, 0, any);
                load_y(s + 1, 0, any);
            }
            compute(lds, sign, [](int) {});
            sign.bit ^= 0x80000000u;
            __syncthreads();
            store_all(lds, sign);
            __syncthreads();
        }
    }

    // Values that the planes do not hold: a wave's findings meet in LDS.
    {
        float probe = 0.f;
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int b = 0; b < FN; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) probe = __builtin_fmaf(acc[a][b][v], 0.f, probe);
        uint32_t seen_x = 0, seen_y = 0;
#pragma unroll
        for (int f = 0; f < PF; ++f) seen_x |= lx[f].seen, seen_y |= ly[f].seen;
        constexpr uint32_t kOrdinary = 0x60006000u, kAny = 0x7fff7fffu;  // exponent >= 2^-63; not zero
        const uint32_t found = (__any(probe != probe) ? 1u : 0u) | (__any(seen_x & kOrdinary) ? 2u : 0u) |
                               (__any(seen_x & kAny) ? 4u : 0u) | (__any(seen_y & kOrdinary) ? 8u : 0u) |
                               (__any(seen_y & kAny) ? 16u : 0u);
        uint32_t *const word = reinterpret_cast<uint32_t *>(lds);
        if (lane == 0) word[wave] = found;
        __syncthreads();
        uint32_t all = 0;
#pragma unroll
        for (int w = 0; w < WM * WN; ++w) all |= word[w];
        all = __builtin_amdgcn_readfirstlane(all);
        if ((all & 1u) || (all & 6u) == 4u || (all & 24u) == 16u) {
            // the tile again, on the fp32 matrix instruction (one stage, nothing overlapped)
            constexpr int kPitch = SX::kPitch;
            float *const xf = reinterpret_cast<float *>(lds);
            float *const yf = xf + BM * kPitch;
            clear();
            for (int32_t s = 0; s < steps; ++s) {
                load_x(s, 0, any);
                load_y(s, 0, any);
                __syncthreads();
                lx[0].store_fp32(xf, tid);
                ly[0].store_fp32(yf, tid);
                __syncthreads();
#pragma unroll 1
                for (int kk = 0; kk < kDepth; kk += 4) {
                    float av[FM], bv[FN];
#pragma unroll
                    for (int a = 0; a < FM; ++a) av[a] = xf[(wm * TM + 16 * a + l16) * kPitch + kk + quad];
#pragma unroll
                    for (int b = 0; b < FN; ++b) bv[b] = yf[(wn * TN + 16 * b + l16) * kPitch + kk + quad];
#pragma unroll
                    for (int a = 0; a < FM; ++a)
#pragma unroll
                        for (int b = 0; b < FN; ++b)
                            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[a], bv[b], acc[a][b], 0, 0, 0);
                }
            }
        }
    }

    // slot s of a group of 64 is row 4 (s % 16) + s / 16: acc[a][b][v] is row 4 (4 quad + v) of the wave's
    // group plus its first block of 16 slots plus a; columns alike.
    const int64_t row0 = i0 + wm * TM / 64 * 64 + wm * TM % 64 / 16 + 16 * quad;
    const int64_t col = j0 + wn * TN / 64 * 64 + wn * TN % 64 / 16 + 4 * l16;
    store_tile<FM, FN, 4>(p, acc, batch, split, row0, col);
}

// The 256x128 tile needs every register of its budget: kept where it fits without spilling.
constexpr bool big_fits(bool yr, bool aligned, int xmode) { return aligned && !(xmode == 4 && !yr); }

template <bool XR, bool YR, bool AL, int XMODE>
void launch(const GemmParams &p, SplitTile tile, unsigned blocks, hipStream_t stream) {
    if (tile == SplitTile::Big) {
        if constexpr (big_fits(YR, AL, XMODE))
            split_gemm_kernel<256, 128, 4, 2, 2, 1, XR, YR, AL, XMODE><<<blocks, 512, 0, stream>>>(p);
    } else if (tile == SplitTile::Mid) {
        split_gemm_kernel<128, 128, 2, 2, 1, 1, XR, YR, AL, XMODE><<<blocks, 256, 0, stream>>>(p);
    } else if (tile == SplitTile::Small) {
        split_gemm_kernel<64, 64, 2, 2, 2, 2, XR, YR, AL, XMODE><<<blocks, 256, 0, stream>>>(p);
    } else {
        split_gemm_kernel<256, 64, 4, 1, 1, 1, XR, YR, AL, XMODE><<<blocks, 256, 0, stream>>>(p);
    }
}

}  // namespace

double launch_us(int64_t blocks, double steps, const TileRate &t, int64_t cus) {
    const int64_t per_cu = (blocks + cus - 1) / cus;
    const int64_t rounds = per_cu / t.resident, rest = per_cu % t.resident;
    auto step_us = [&](int64_t r) { return std::max(t.alone_us, (double)r * t.step_us); };
    return steps * ((double)rounds * step_us(t.resident) + (rest ? step_us(rest) : 0.0)) +
           t.round_us * (double)(rounds + (rest ? 1 : 0));
}

double slices_us(int64_t splits, int64_t out_len) {
    return splits > 1 ? (double)(2 * splits + 1) * (double)out_len * 4.0 / 5.0e6 + 4.0 : 0.0;
}

SplitPlan split_plan(int64_t m, int64_t n, int64_t k, int64_t batch, int64_t cus, bool yr, bool aligned, int xmode,
                     double limit_us) {
    struct Shape {
        SplitTile tile;
        int rows, cols;
        TileRate rate;
    };
    // Measured on 4096^3 (256x128: 235 TFLOP/s, 128x128: 212, 256x64: 194), 8192x784x1024, 1024^3
    // (64x64: 24.7 us) and products of one to four steps.
    static constexpr Shape shapes[] = {{SplitTile::Big, 256, 128, {1, 2.28, 2.28, 6.0}},
                                       {SplitTile::Mid, 128, 128, {2, 1.28, 1.75, 6.0}},
                                       {SplitTile::Tall, 256, 64, {2, 1.41, 1.9, 6.0}},
                                       {SplitTile::Small, 64, 64, {3, 0.52, 0.62, 4.3}}};
    const int64_t out_len = batch * m * n;
    SplitPlan plan;
    double best_us = limit_us;
    for (const Shape &sh : shapes) {
        if (sh.tile == SplitTile::Big && !big_fits(yr, aligned, xmode)) continue;
        // single-element loads at ragged ends
        const double ragged = aligned ? 1.0 : 1.2;
        const int64_t tiles = ((m + sh.rows - 1) / sh.rows) * ((n + sh.cols - 1) / sh.cols) * batch;
        const int64_t most = std::max<int64_t>(1, std::min<int64_t>(k / (2 * kDepth), 512));
        // the least slice count of each slice length (most of 2 sqrt(k / 32) of them): 17 -> 6 us of host
        // time at [2, 100000] x [100000, 2], together with the sums' bound below
        for (int64_t want = 1, chunk; want <= most; want = (k + chunk - kDepth - 1) / (chunk - kDepth)) {
            chunk = ((k + want - 1) / want + kDepth - 1) / kDepth * kDepth;
            // slices, and range sums of more than 32 of them, stay within 64 MiB
            if (want > 1 && (want + (want > 32 ? (want + 31) / 32 : 0)) * out_len > (int64_t(16) << 20)) break;
            const double us = ragged * launch_us(tiles * want, (double)(chunk / kDepth), sh.rate, cus) +
                              slices_us(want, out_len);
            if (us < best_us) {
                best_us = us;
                plan = {sh.tile, sh.rows, sh.cols, want};
            }
            // more slices only add to the sum
            if (tiles * want > 8 * cus || sh.rate.round_us + slices_us(want, out_len) >= best_us) break;
            if (chunk <= kDepth) break;
        }
    }
    return plan;
}

int split_gemm(axis_device device, const GemmParams &p, SplitTile tile, bool xr, bool yr, bool aligned, int xmode,
               unsigned blocks) {
    const hipStream_t st = device->stream;
    if (xmode == 0 && xr && !yr && aligned)
        launch<true, false, true, 0>(p, tile, blocks, st);
    else if (xmode == 0 && xr && !yr)
        launch<true, false, false, 0>(p, tile, blocks, st);
    else if (xmode == 0 && xr && aligned)
        launch<true, true, true, 0>(p, tile, blocks, st);
    else if (xmode == 0 && xr)
        launch<true, true, false, 0>(p, tile, blocks, st);
    else if (xmode == 0 && aligned)
        launch<false, false, true, 0>(p, tile, blocks, st);
    else if (xmode == 0)
        launch<false, false, false, 0>(p, tile, blocks, st);
    else if (xmode == 4 && !yr)
        launch<true, false, true, 4>(p, tile, blocks, st);
    else if (xmode == 4)
        launch<true, true, true, 4>(p, tile, blocks, st);
    else if (xmode == 5)
        launch<true, false, true, 5>(p, tile, blocks, st);
    else if (xmode == 3)
        launch<false, false, true, 3>(p, tile, blocks, st);
    else
        launch<false, false, true, 2>(p, tile, blocks, st);
    return launch_status("split_gemm_kernel");
}

}  // namespace axis
