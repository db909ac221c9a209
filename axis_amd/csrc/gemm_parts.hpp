// Operands of the GEMM family (gemm.hip on the fp32 matrix cores, gemm_split.hip on bf16 planes):
// launch parameters, the gathered convolution loaders and the output tiles' epilogues.
//
// A loader is built on a staging policy S that says which vectors of the tile a thread holds and
// keeps them in registers (S::reg, kVecs vectors of VEC floats).  r-contiguous operands: vector idx
// (= thread + e * NT) covers reduction elements S::line_r(idx) .. + VEC - 1 of tile row
// S::line_t(idx); t-contiguous ones: vector e of a thread covers tile rows S::vec_t(tid) .. + VEC - 1
// of reduction element S::vec_r(tid, e).
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>
#include <type_traits>

#include "common.hpp"
#include "fastdiv.hpp"
#include "pool_rule.hpp"

namespace axis {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// Geometry of a gathered convolution operand (tensor [batch, height, width, channels]).
struct ConvGeom {
    const float *src;
    int64_t ld_b;                     // element strides of batch, channel, row, column
    int32_t ld_c, ld_h, ld_w;
    int32_t height, width, channels;  // gathered tensor
    int32_t out_h, out_w;             // output pixel grid the reduction/rows enumerate
    int32_t kh, kw, sy, sx, py, px;
    FastDiv c_div, kw_div, ow_div, oh_div;
    bool tap_steps;                   // channels % 32 == 0: a 32-deep K step stays in one tap
    // With tap steps, the buffer rows loader walks the reduction in 32-channel blocks, every tap
    // of a block before the next block: r = (cb * taps + pos) * 32 + ci.  A tile then re-reads
    // the same 32 channels of its neighbourhood on consecutive steps, which stay in L2, instead
    // of the whole tensor slab between one tap and the next.
    bool block_major;
    FastDiv taps_div;                 // kh * kw
    // Rows mode, 2x2 pooling epilogue: tile row t holds position t % 4 (ky major) of the tile's
    // window t / 4, windows numbered row-major over the tile's window rows (pw per row).  A tile
    // starts on an even output row and holds whole window rows.
    bool window_major;
    FastDiv pw_div;
};

// Output pixel of tile row t for a tile starting at pixel t0.
__device__ __forceinline__ int64_t tile_pixel(const ConvGeom &g, int64_t t0, int t) {
    if (!g.window_major) return t0 + t;
    const uint32_t w = (uint32_t)t >> 2, pos = (uint32_t)t & 3u;
    const uint32_t wr = g.pw_div.div(w), wc = w - wr * g.pw_div.d;
    return t0 + (int64_t)(2 * wr + (pos >> 1)) * g.out_w + 2 * wc + (pos & 1u);
}

// Second operand read straight from a convolution weight in the reference's [(c, ky, kx), n]
// layout: a K step starting at r0 begins at element hi * a + lo * b + c with r0 >> shift = hi * div + lo.
// The reduction index is r = pos * R + q (pos = ky * kw + kx, R rows per tap, R a multiple of the K
// step): hi = pos, lo = q; or, in the rows loader's block-major order r = (cb * taps + pos) * 32 + ci,
// hi = cb and lo = pos.
struct TapSteps {
    bool on;
    uint32_t shift;
    FastDiv div;
    int64_t a, b, c;

    // row q of tap pos at element q * q_stride + pos * tap_stride + origin
    static TapSteps make(bool block_major, int64_t rows, int64_t taps, int64_t q_stride, int64_t tap_stride,
                         int64_t origin) {
        if (block_major) return {true, 5, FastDiv((uint32_t)taps), 32 * q_stride, tap_stride, origin};
        return {true, 0, FastDiv((uint32_t)rows), tap_stride, q_stride, origin};
    }
    // plain rows (below 2^31 of them) in the same form
    static TapSteps rows(int64_t stride) { return {true, 0, FastDiv(0x80000000u), 0, stride, 0}; }
    __device__ __forceinline__ int64_t step(int64_t r0) const {
        const uint32_t t = (uint32_t)r0 >> shift;
        const uint32_t hi = div.div(t);
        return (int64_t)hi * a + (int64_t)(t - hi * div.d) * b + c;
    }
};

struct GemmParams {
    const float *x;
    const float *y;
    float *c;
    const float *bias;         // added to every row of C (length n), or null
    const float *d;            // out = beta * d + alpha * (A.B) when non-null (d shaped like out)
    float alpha, beta;
    int64_t m, n, k;           // C is [m, n]; reduction length k
    int64_t x_si, x_sr;        // dense X(i, r) = x[i * x_si + r * x_sr]
    int64_t y_sr, y_sj;        // Y(r, j) = y[r * y_sr + j * y_sj]
    int64_t x_batch, y_batch;  // batch strides (elements)
    int64_t c_batch;           // batch stride of the output (or of one slice of partials)
    int64_t c_split;           // stride between reduction slices in the output (partials)
    int64_t k_chunk;           // reduction length per slice (multiple of the tile depth)
    int64_t k_work;            // algorithmic reduction length for timing (k without padding), or 0
    int32_t splits;
    int32_t tiles_m, tiles_n;
    uint32_t xcd_span;         // blocks / 8: the first 8 * xcd_span blocks are remapped, the rest keep their order
    ConvGeom conv;
    // Pooling epilogue: output rows are pixels of a [.., out_h, out_w] grid (out_w = pool_ow).
    float *pooled;
    uint8_t *argmax;
    int32_t pool_h, pool_w, pool_ow;
    FastDiv pool_cols;         // pooled columns per output row (pool_ow / pool_w)
    TapSteps ytaps;            // Y read as a tap-major convolution weight
    // Output rows ordered (pos, c) with perm_c channels and perm_taps taps are written as rows
    // c * perm_taps + pos (the reference's weight layout); 0 = rows as computed.
    int32_t perm_c, perm_taps;
    bool bf16;                 // operands rounded to bf16 as they are staged (Device::cuda_bf16)
};

template <int VEC>
__device__ __forceinline__ void load_into(float *reg, const float *src, bool valid) {
    if constexpr (VEC == 4) {
        floatx4 v = {0.f, 0.f, 0.f, 0.f};
        if (valid) v = *reinterpret_cast<const floatx4 *>(src);
        reg[0] = v[0];
        reg[1] = v[1];
        reg[2] = v[2];
        reg[3] = v[3];
    } else {
        reg[0] = valid ? src[0] : 0.f;
    }
}

// Buffer loads: an offset at or past the resource's record count (2^31 - 1 bytes) reads as zero,
// so padding taps and reduction tails need neither a branch nor zeroed registers.
constexpr uint32_t kOutside = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const float *base, int32_t bytes = 0x7fffffff) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, bytes, 0x00020000);
}
template <int VEC>
__device__ __forceinline__ void buffer_into(float *reg, __amdgpu_buffer_rsrc_t rsrc, uint32_t byte_offset) {
    if constexpr (VEC == 4) {
        const floatx4 v = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, byte_offset, 0, 0));
        reg[0] = v[0];
        reg[1] = v[1];
        reg[2] = v[2];
        reg[3] = v[3];
    } else {
        reg[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, byte_offset, 0, 0));
    }
}

// A wave-uniform pointer moved to scalar registers, so that buffer resources built from it need no
// per-lane loop (the compiler cannot always prove such values uniform).
__device__ __forceinline__ const float *uniform_ptr(const float *p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const float *>(((uint64_t)hi << 32) | lo);
}

// Convolution operand, rows mode: t = output pixel, r = (ky*kw + kx)*channels + channel.
// Per row: the offset of its window origin and the origin's coordinates (for the padding test);
// per K step: one decode of the thread's r into a 32-bit offset shared by every row.
template <class S, int BT, int BK, int NT, int VEC>
struct ConvRowsLoader : S {
    uint32_t origin[S::kVecs];   // b*ld_b + iy0*ld_h + ix0*ld_w (mod 2^32; exact when valid)
    int32_t iy0[S::kVecs], ix0[S::kVecs];
    int rr;

    __device__ __forceinline__ void init(const ConvGeom &geom, int64_t t0, int64_t t_end, int tid) {
        rr = S::line_r(tid);  // the same for every e
#pragma unroll
        for (int e = 0; e < S::kVecs; ++e) {
            const int64_t gt = tile_pixel(geom, t0, S::line_t(tid + e * NT));
            // Rows past the end get an origin far outside the image, so every tap is padding;
            // computed branch-free so the per-row arrays stay in registers.
            const bool live = gt < t_end;
            const uint32_t pix = live ? (uint32_t)gt : 0u;
            const uint32_t q = geom.ow_div.div(pix);
            const int32_t ox = (int32_t)(pix - q * (uint32_t)geom.out_w);
            const uint32_t b = geom.oh_div.div(q);
            const int32_t oy = (int32_t)(q - b * (uint32_t)geom.out_h);
            const int32_t y0 = oy * geom.sy - geom.py;
            ix0[e] = ox * geom.sx - geom.px;
            origin[e] = b * (uint32_t)geom.ld_b + (uint32_t)y0 * (uint32_t)geom.ld_h +
                        (uint32_t)ix0[e] * (uint32_t)geom.ld_w;
            iy0[e] = live ? y0 : -(1 << 30);
        }
    }
    __device__ __forceinline__ void load(const ConvGeom &geom, int64_t r0, int32_t room, int) {
        const bool r_ok = rr < room;
        const uint32_t g = r_ok ? (uint32_t)(r0 + rr) : 0u;
        const uint32_t pos = geom.c_div.div(g);
        const int32_t c = (int32_t)(g - pos * (uint32_t)geom.channels);
        const int32_t ky = (int32_t)geom.kw_div.div(pos);
        const int32_t kx = (int32_t)pos - ky * geom.kw;
        const uint32_t delta = (uint32_t)(ky * geom.ld_h + kx * geom.ld_w + c * geom.ld_c);
#pragma unroll
        for (int e = 0; e < S::kVecs; ++e) {
            const bool valid = r_ok && (uint32_t)(iy0[e] + ky) < (uint32_t)geom.height &&
                               (uint32_t)(ix0[e] + kx) < (uint32_t)geom.width;
            load_into<VEC>(this->reg + e * VEC, geom.src + (valid ? origin[e] + delta : 0u), valid);
        }
    }
};

// Rows mode through buffer loads, for gathered tensors whose offsets fit 31-bit byte offsets and
// kernels of at most 32 taps.  Each row keeps its window origin's offset and a mask of the taps
// that fall outside the image (bit ky*kw + kx), so a K step tests one bit per vector.  When the
// channel count is a multiple of BK (geom.tap_steps), a K step covers BK channels of one tap and
// the step's tap decode is wave-uniform.
// STEPS: 1 the geometry has tap steps in block-major order, 0 it has no tap steps, -1 as it says.
template <class S, int BT, int BK, int NT, int VEC, int STEPS = -1>
struct ConvRowsBufferLoader : S {
    uint32_t origin4[S::kVecs];  // 4 * (b*ld_b + iy0*ld_h + ix0*ld_w) (mod 2^32; exact when valid)
    uint32_t outside[S::kVecs];  // taps of the row's window outside the image (all, for rows past the end)
    int rr;
    uint32_t lane_c4;            // 4 * rr * ld_c: the thread's channel offset inside a tap step, bytes

    __device__ __forceinline__ void init(const ConvGeom &geom, int64_t t0, int64_t t_end, int tid) {
        rr = S::line_r(tid);
        lane_c4 = (uint32_t)(rr * geom.ld_c) * 4u;
#pragma unroll
        for (int e = 0; e < S::kVecs; ++e) {
            const int64_t gt = tile_pixel(geom, t0, S::line_t(tid + e * NT));
            const bool live = gt < t_end;
            const uint32_t pix = live ? (uint32_t)gt : 0u;
            const uint32_t q = geom.ow_div.div(pix);
            const int32_t ox = (int32_t)(pix - q * (uint32_t)geom.out_w);
            const uint32_t b = geom.oh_div.div(q);
            const int32_t oy = (int32_t)(q - b * (uint32_t)geom.out_h);
            const int32_t y0 = oy * geom.sy - geom.py;
            const int32_t x0 = ox * geom.sx - geom.px;
            origin4[e] = (b * (uint32_t)geom.ld_b + (uint32_t)y0 * (uint32_t)geom.ld_h + (uint32_t)x0 * (uint32_t)geom.ld_w) * 4u;
            uint32_t cols = 0, taps = 0;
            for (int32_t kx = 0; kx < geom.kw; ++kx)
                cols |= (uint32_t)((uint32_t)(x0 + kx) < (uint32_t)geom.width) << kx;
            for (int32_t ky = 0; ky < geom.kh; ++ky)
                taps |= ((uint32_t)(y0 + ky) < (uint32_t)geom.height ? cols : 0u) << (ky * geom.kw);
            outside[e] = live ? ~taps : ~0u;
        }
    }
    __device__ __forceinline__ void load(const ConvGeom &geom, int64_t r0, int32_t room, int) {
        const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(geom.src);
        if (STEPS == 1 || (STEPS < 0 && geom.tap_steps)) {
            // The reduction is a multiple of BK here, so every k of the step is inside it; the
            // step's tap and first channel are wave-uniform (scalar arithmetic).  Per vector: the
            // offset, and the window's outside bit for this tap moved to bit 31, which puts a
            // masked lane's offset past the record count (three vector instructions).
            uint32_t pos;
            int32_t c0;
            if (STEPS == 1 || geom.block_major) {
                const uint32_t st = (uint32_t)r0 >> 5;
                const uint32_t cb = geom.taps_div.div(st);
                pos = st - cb * geom.taps_div.d;
                c0 = (int32_t)cb * 32;
            } else {
                pos = geom.c_div.div((uint32_t)r0);
                c0 = (int32_t)((uint32_t)r0 - pos * (uint32_t)geom.channels);
            }
            const int32_t ky = (int32_t)geom.kw_div.div(pos);
            const int32_t kx = (int32_t)pos - ky * geom.kw;
            const uint32_t delta4 =
                __builtin_amdgcn_readfirstlane((uint32_t)(ky * geom.ld_h + kx * geom.ld_w + c0 * geom.ld_c) * 4u) +
                lane_c4;
            const uint32_t up = 31u - __builtin_amdgcn_readfirstlane(pos);
#pragma unroll
            for (int e = 0; e < S::kVecs; ++e)
                buffer_into<VEC>(this->reg + e * VEC, rsrc, (origin4[e] + delta4) | ((outside[e] << up) & kOutside));
        } else {
            const bool r_ok = rr < room;
            const uint32_t g = r_ok ? (uint32_t)(r0 + rr) : 0u;
            const uint32_t pos = geom.c_div.div(g);
            const int32_t c = (int32_t)(g - pos * (uint32_t)geom.channels);
            const int32_t ky = (int32_t)geom.kw_div.div(pos);
            const int32_t kx = (int32_t)pos - ky * geom.kw;
            const uint32_t delta4 = (uint32_t)(ky * geom.ld_h + kx * geom.ld_w + c * geom.ld_c) * 4u;
#pragma unroll
            for (int e = 0; e < S::kVecs; ++e) {
                const bool valid = r_ok && ((outside[e] >> pos) & 1u) == 0;
                buffer_into<VEC>(this->reg + e * VEC, rsrc, valid ? origin4[e] + delta4 : kOutside);
            }
        }
    }
};

// Convolution operand, cols mode: t = (ky*kw + kx)*channels + channel, r = output pixel.  The
// thread's t is fixed; each row keeps its pixel's coordinates and offset and walks forward BK
// pixels per K step.
template <class S, int BT, int BK, int NT, int VEC>
struct ConvColsLoader : S {
    uint32_t tap;                // (ky-py)*ld_h + (kx-px)*ld_w + c*ld_c of the thread's t (mod 2^32)
    int32_t ky, kx;
    bool t_ok;
    int32_t ox[S::kVecs], oy[S::kVecs];
    uint32_t off[S::kVecs];      // b*ld_b + oy*sy*ld_h + ox*sx*ld_w (mod 2^32)
    int64_t next_r;              // r0 the state describes

    __device__ __forceinline__ void init(const ConvGeom &geom, int64_t t0, int64_t t_end, int tid) {
        const int64_t gt = t0 + S::vec_t(tid);
        t_ok = gt < t_end;
        const uint32_t g = t_ok ? (uint32_t)gt : 0u;
        const uint32_t pos = geom.c_div.div(g);
        const int32_t c = (int32_t)(g - pos * (uint32_t)geom.channels);
        ky = (int32_t)geom.kw_div.div(pos);
        kx = (int32_t)pos - ky * geom.kw;
        tap = (uint32_t)(ky - geom.py) * (uint32_t)geom.ld_h + (uint32_t)(kx - geom.px) * (uint32_t)geom.ld_w +
              (uint32_t)c * (uint32_t)geom.ld_c;
        next_r = -1;
    }
    __device__ __forceinline__ void locate(const ConvGeom &geom, int64_t r0, int tid) {
#pragma unroll
        for (int e = 0; e < S::kVecs; ++e) {
            const uint32_t pix = (uint32_t)(r0 + S::vec_r(tid, e));
            const uint32_t q = geom.ow_div.div(pix);
            ox[e] = (int32_t)(pix - q * (uint32_t)geom.out_w);
            const uint32_t b = geom.oh_div.div(q);
            oy[e] = (int32_t)(q - b * (uint32_t)geom.out_h);
            off[e] = b * (uint32_t)geom.ld_b + (uint32_t)(oy[e] * geom.sy) * (uint32_t)geom.ld_h +
                     (uint32_t)(ox[e] * geom.sx) * (uint32_t)geom.ld_w;
        }
        next_r = r0;
    }
    __device__ __forceinline__ void advance(const ConvGeom &geom) {
        const uint32_t col_step = (uint32_t)(geom.sx * geom.ld_w), row_step = (uint32_t)(geom.sy * geom.ld_h);
#pragma unroll
        for (int e = 0; e < S::kVecs; ++e) {
            ox[e] += BK;
            off[e] += BK * col_step;
            while (ox[e] >= geom.out_w) {
                ox[e] -= geom.out_w;
                off[e] += row_step - (uint32_t)geom.out_w * col_step;
                if (++oy[e] == geom.out_h) {
                    oy[e] = 0;
                    off[e] += (uint32_t)geom.ld_b - (uint32_t)geom.out_h * row_step;
                }
            }
        }
        next_r += BK;
    }
    __device__ __forceinline__ void load(const ConvGeom &geom, int64_t r0, int32_t room, int tid) {
        if (r0 != next_r) locate(geom, r0, tid);
#pragma unroll
        for (int e = 0; e < S::kVecs; ++e) {
            const int32_t iy = oy[e] * geom.sy + ky - geom.py, ix = ox[e] * geom.sx + kx - geom.px;
            const bool valid = t_ok && S::vec_r(tid, e) < room && (uint32_t)iy < (uint32_t)geom.height &&
                               (uint32_t)ix < (uint32_t)geom.width;
            load_into<VEC>(this->reg + e * VEC, geom.src + (valid ? off[e] + tap : 0u), valid);
        }
        advance(geom);
    }
};

// Cols mode when every K step covers whole aligned pixel runs: BK divides the output width or is
// a multiple of it, and the image's pixel count is a multiple of BK.  Then a step starting at
// pixel p0 (a multiple of BK) never leaves one image and the in-step pixel s sits at
// (oy0 + s / out_w, ox0 + s % out_w) for every step, so each vector's window position relative
// to the step origin is fixed at init and a step decodes only its wave-uniform origin.
template <class S, int BT, int BK, int NT, int VEC>
struct ConvColsStepLoader : S {
    static_assert(BK == 32, "steps of 32 pixels");
    uint32_t rel4[S::kVecs];  // bytes: (iy_rel + py)*ld_h + (ix_rel + px)*ld_w + c*ld_c (mod 2^32)
    // Bit (first | last << 1 | top << 2 | bottom << 3) set when the lane's element is padding (or
    // its row past the end) in a step whose pixels start the image's first / last 32-column
    // segment, first / last row group.  A step elsewhere has every element inside (the host
    // keeps px <= 32 sx and py <= (rows per step) sy), so these four flags decide.
    uint32_t bad[S::kVecs];

    __device__ __forceinline__ void init(const ConvGeom &geom, int64_t t0, int64_t t_end, int tid) {
        const int64_t gt = t0 + S::vec_t(tid);
        const bool t_ok = gt < t_end;
        const uint32_t g = t_ok ? (uint32_t)gt : 0u;
        const uint32_t pos = geom.c_div.div(g);
        const int32_t c = (int32_t)(g - pos * (uint32_t)geom.channels);
        const int32_t ky = (int32_t)geom.kw_div.div(pos);
        const int32_t kx = (int32_t)pos - ky * geom.kw;
        const int32_t seg = geom.out_w < 32 ? geom.out_w : 32;       // columns a step spans
        const int32_t rows = geom.out_w < 32 ? 32 / geom.out_w : 1;  // rows a step spans
        const int32_t last_x = (geom.out_w - seg) * geom.sx, last_y = (geom.out_h - rows) * geom.sy;
#pragma unroll
        for (int e = 0; e < S::kVecs; ++e) {
            const uint32_t s = (uint32_t)S::vec_r(tid, e);
            const int32_t dy = (int32_t)geom.ow_div.div(s);
            const int32_t dx = (int32_t)s - dy * geom.out_w;
            const int32_t iy_rel = dy * geom.sy + ky - geom.py, ix_rel = dx * geom.sx + kx - geom.px;
            rel4[e] = ((uint32_t)(iy_rel + geom.py) * (uint32_t)geom.ld_h + (uint32_t)(ix_rel + geom.px) * (uint32_t)geom.ld_w +
                       (uint32_t)c * (uint32_t)geom.ld_c) * 4u;
            uint32_t b = 0;
            for (uint32_t f = 0; f < 16; ++f) {
                const bool first = f & 1u, last = f & 2u, top = f & 4u, bottom = f & 8u;
                const int32_t x = first ? ix_rel : last ? last_x + ix_rel : 0;
                const int32_t y = top ? iy_rel : bottom ? last_y + iy_rel : 0;
                const bool in = t_ok && (!(first || last) || (uint32_t)x < (uint32_t)geom.width) &&
                                (!(top || bottom) || (uint32_t)y < (uint32_t)geom.height);
                b |= (in ? 0u : 1u) << f;
            }
            bad[e] = b;
        }
    }
    // Every step is whole: the reduction (batch * image pixels) and the slices are multiples of 32.
    __device__ __forceinline__ void load(const ConvGeom &geom, int64_t r0, int32_t, int) {
        const uint32_t p0 = (uint32_t)r0;
        const uint32_t q = geom.ow_div.div(p0);
        const int32_t ox0 = (int32_t)(p0 - q * (uint32_t)geom.out_w);
        const uint32_t b = geom.oh_div.div(q);
        const int32_t oy0 = (int32_t)(q - b * (uint32_t)geom.out_h);
        const int32_t seg = geom.out_w < 32 ? geom.out_w : 32;
        const int32_t rows = geom.out_w < 32 ? 32 / geom.out_w : 1;
        // sign bits rather than comparisons: compared flags reach vector registers as lane masks
        const uint32_t flags = ((uint32_t)(ox0 - 1) >> 31) | ((uint32_t)(geom.out_w - ox0 - seg - 1) >> 31 << 1) |
                               ((uint32_t)(oy0 - 1) >> 31 << 2) | ((uint32_t)(geom.out_h - oy0 - rows - 1) >> 31 << 3);
        const int32_t oys = oy0 * geom.sy, oxs = ox0 * geom.sx;
        // Buffer base at the step origin moved back by the padding, so that every valid lane's
        // offset (at least -py rows and -px columns from the origin) is non-negative.
        const int64_t shift = (int64_t)geom.py * geom.ld_h + (int64_t)geom.px * geom.ld_w;
        const int64_t base = (int64_t)b * geom.ld_b + (int64_t)oys * geom.ld_h + (int64_t)oxs * geom.ld_w - shift;
        const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(geom.src + base);
        // the padding bit of this step's case moved to bit 31: past the record count (two vector
        // instructions per vector)
#pragma unroll
        for (int e = 0; e < S::kVecs; ++e)
            buffer_into<VEC>(this->reg + e * VEC, rsrc, (((bad[e] >> flags) & 1u) << 31) | rel4[e]);
    }
};

// One wave's part of an output tile: acc[a][b][v] is row row0 + RS * v + a, column col + b, so a lane's
// FN columns are adjacent (row0, col: the lane's first row and column).  The bias
// and the axpby are applied only when the reduction is not split; split sums finish them at the end.
template <int FM, int FN, int RS = FM>
__device__ __forceinline__ void store_tile(const GemmParams &p, const floatx4 (&acc)[FM][FN], int64_t batch, int split,
                                           int64_t row0, int64_t col) {
    float *c = p.c + batch * p.c_batch + (int64_t)split * p.c_split;
    // bias / axpby apply to whole sums only; split sums finish them at the end
    const bool whole = p.splits == 1;
    const float *bias = whole ? p.bias : nullptr;
    const float *d = whole ? p.d : nullptr;
    const int64_t out_base = batch * p.m * p.n;
    if (p.n % FN == 0 && (reinterpret_cast<uintptr_t>(c) & (4 * FN - 1)) == 0) {
        // one FN-wide vector store per row (col < n implies all FN columns are)
        if (col < p.n) {
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int64_t row = row0 + RS * v + a;
                    if (row >= p.m) continue;
                    const int64_t idx = row * p.n + col;
                    if constexpr (FN == 4) {
                        floatx4 o;
#pragma unroll
                        for (int b = 0; b < 4; ++b)
                            o[b] = finish_value(bias, d, p.alpha, p.beta, acc[a][b][v], out_base + idx + b, col + b);
                        *reinterpret_cast<floatx4 *>(c + idx) = o;
                    } else {
                        float2 o;
                        o.x = finish_value(bias, d, p.alpha, p.beta, acc[a][0][v], out_base + idx, col);
                        o.y = finish_value(bias, d, p.alpha, p.beta, acc[a][1][v], out_base + idx + 1, col + 1);
                        *reinterpret_cast<float2 *>(c + idx) = o;
                    }
                }
        }
    } else {
        // rows that start on any element: the same vector stores (global memory takes them on 4 bytes)
        // where all FN columns are there, else one by one
        typedef float vec __attribute__((ext_vector_type(FN), aligned(4)));
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int64_t row = row0 + RS * v + a;
                if (row >= p.m || col >= p.n) continue;
                const int64_t idx = row * p.n + col;
                vec o;
#pragma unroll
                for (int b = 0; b < FN; ++b)
                    o[b] = col + b < p.n ? finish_value(bias, d, p.alpha, p.beta, acc[a][b][v], out_base + idx + b, col + b) : 0.f;
                if (col + FN <= p.n) {
                    *reinterpret_cast<vec *>(c + idx) = o;
                } else {
#pragma unroll
                    for (int b = 0; b < FN; ++b)
                        if (col + b < p.n) c[idx + b] = o[b];
                }
            }
    }
}

// The fused 2x2 max pool of one wave's tile part (EPI 1, window-major rows): wm is the wave's row
// block of TM rows, col the lane's first column.
template <int TM, int FN>
__device__ __forceinline__ void pool_tile(const GemmParams &p, const floatx4 (&acc)[4][FN], int64_t i0, int wm, int quad,
                                          int64_t col) {
    const int ow = p.pool_ow;
    const int pw = ow / p.pool_w;
    const int64_t pooled_row0 = i0 / ow / p.pool_h;
    // 2x2 windows, tile rows window-major: acc[a][b][v] is position a of the wave's window
    // 4 * quad + v, so each lane pools whole windows from its own registers (no LDS, no
    // barrier) and writes its FN adjacent columns as one vector of values and one of
    // winner bytes.
    float addv[FN];
    bool okv[FN];
#pragma unroll
    for (int b = 0; b < FN; ++b) {
        const int64_t at = col + b;
        okv[b] = at < p.n;
        addv[b] = (p.bias != nullptr && okv[b]) ? p.bias[at] : 0.0f;
    }
    const bool vec = p.n % FN == 0 && (reinterpret_cast<uintptr_t>(p.pooled) & (4 * FN - 1)) == 0 &&
                     (reinterpret_cast<uintptr_t>(p.argmax) & (FN - 1)) == 0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int w = wm * (TM / 4) + 4 * quad + v;  // window inside the tile
        const int wr = (int)p.pool_cols.div((uint32_t)w), wc = w - wr * pw;
        if (i0 + (int64_t)wr * 2 * ow >= p.m) continue;
        float best[FN];
        int winner[FN];
#pragma unroll
        for (int b = 0; b < FN; ++b) {
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = acc[e][b][v] + addv[b];
            relu_pool_window4(y, best[b], winner[b]);
        }
        const int64_t out = ((pooled_row0 + wr) * pw + wc) * p.n + col;
        if (vec && okv[0]) {
            if constexpr (FN == 4) {
                *reinterpret_cast<floatx4 *>(p.pooled + out) = floatx4{best[0], best[1], best[2], best[3]};
                *reinterpret_cast<uint32_t *>(p.argmax + out) =
                    (uint32_t)winner[0] | ((uint32_t)winner[1] << 8) | ((uint32_t)winner[2] << 16) |
                    ((uint32_t)winner[3] << 24);
            } else {
                *reinterpret_cast<float2 *>(p.pooled + out) = make_float2(best[0], best[1]);
                *reinterpret_cast<uint16_t *>(p.argmax + out) = (uint16_t)(winner[0] | (winner[1] << 8));
            }
        } else {
#pragma unroll
            for (int b = 0; b < FN; ++b) {
                if (!okv[b]) continue;
                p.pooled[out + b] = best[b];
                p.argmax[out + b] = (uint8_t)winner[b];
            }
        }
    }
}

}  // namespace axis
