// The small fp32 ops between the matmuls (piece::run_rows,
// src/xdna-exec.cpp:253-346), as HBM-bound row kernels. RMS_NORM (+ the scale
// row MUL after it) and the GLUs can also write the next matmul's input (the
// bfp16 pack, stored expanded) directly, so a normalised or gated row goes
// HBM -> registers -> matmul operand without a round trip through an fp32
// tensor.
#include <algorithm>

#include "zest_common.h"
#include "zest_device.h"

namespace {

constexpr int NORM_ROWS = 4;  // rows per workgroup, one wave each

// Writes 4 values of row r at columns [c, c+4) (c % 4 == 0) of the next
// matmul's input, the bfp16 pack stored expanded: the 8-column block is this
// lane's 4 and its neighbour's (lane ^ 1), whose largest exponent field one
// lane exchange finds; the 4 values are encoded as encode8 does and stored as
// the bf16 they stand for (8 bytes). Both lanes of a pair must call it.
__device__ inline void pack4_expanded(uint8_t * packed, int64_t R_pad, int64_t r, int64_t c, const float v[4]) {
    uint32_t e = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) e = max(e, (__float_as_uint(v[q]) >> 23) & 0xffu);
    e = max(e, (uint32_t) __builtin_amdgcn_update_dpp(0, (int) e, 0xb1, 0xf, 0xf, true));  // lanes 1, 0, 3, 2
    const int sh = 133 - (int) e;
    const float sc = zest::block_scale(e);
    uint32_t b[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const float qf = __builtin_amdgcn_fmed3f(__builtin_rintf(__builtin_ldexpf(v[q], sh)), -128.0f, 127.0f);
        b[q] = __float_as_uint(__builtin_fmaf(qf, sc, 0.0f));  // exact: at most 8 significant bits; + 0 makes -0 0
    }
    *reinterpret_cast<uint2 *>(packed + zest_xoffset(r, c, R_pad)) = make_uint2(
        __builtin_amdgcn_perm(b[1], b[0], 0x07060302u), __builtin_amdgcn_perm(b[3], b[2], 0x07060302u));
}

// Zeroes row r of an expanded operand (d_pad columns): a padding row past the
// last real row, which the GEMM reads as zero.
__device__ inline void zero_row_expanded(uint8_t * packed, int64_t R_pad, int64_t r, int64_t d_pad, int lane) {
    for (int64_t c = lane * 4; c < d_pad; c += 256)
        *reinterpret_cast<uint2 *>(packed + zest_xoffset(r, c, R_pad)) = make_uint2(0, 0);
}

// Rows wider than rms_norm_row_kernel takes: one wave per row, sum of
// squares (fp32), sc = 1/sqrt(ss/d + eps),
// y = x * sc (* w). Lane l takes the 4 floats at columns 4l + 256i, so a
// wave's load covers 1 KB of the row; the sum is a wave reduction, no LDS.
// The second pass re-reads the row (from L2) and writes y and/or the packed
// row, including the zero blocks of the K padding when d % 64 != 0; waves
// past the last row zero the packed operand's padding rows.
__global__ __launch_bounds__(NORM_ROWS * 64) void rms_norm_kernel(const float * __restrict__ x, int64_t rows,
                                                                  int64_t d, float eps, const float * __restrict__ w,
                                                                  float * __restrict__ y, uint8_t * __restrict__ packed,
                                                                  int64_t R_pad) {
    const int lane = threadIdx.x & 63;
    const int64_t r = (int64_t) blockIdx.x * NORM_ROWS + (threadIdx.x >> 6);
    const int64_t d_pad = zest_k_padded(d);
    if (r >= rows) {
        if (packed && r < R_pad) zero_row_expanded(packed, R_pad, r, d_pad, lane);
        return;
    }
    const float * xr = x + r * d;
    const bool vec = (d & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    auto load4 = [&](const float * p, int64_t c, float v[4]) {
        if (vec && c + 4 <= d) {
            const float4 q = *reinterpret_cast<const float4 *>(p + c);
            v[0] = q.x;
            v[1] = q.y;
            v[2] = q.z;
            v[3] = q.w;
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = c + i < d ? p[c + i] : 0.0f;
        }
    };
    float ss = 0.0f;
    for (int64_t c = lane * 4; c < d; c += 256) {
        float v[4];
        load4(xr, c, v);
#pragma unroll
        for (int i = 0; i < 4; i++) ss += v[i] * v[i];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
    const float sc = 1.0f / sqrtf(ss / (float) d + eps);
    const bool wvec = w && vec && (reinterpret_cast<uintptr_t>(w) & 15) == 0;
    for (int64_t c = lane * 4; c < (packed ? d_pad : d); c += 256) {
        float o[4];
        load4(xr, c, o);
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] *= sc;
        if (w) {
            float wv[4];
            if (wvec && c + 4 <= d) {
                const float4 q = *reinterpret_cast<const float4 *>(w + c);
                wv[0] = q.x;
                wv[1] = q.y;
                wv[2] = q.z;
                wv[3] = q.w;
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) wv[i] = c + i < d ? w[c + i] : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < 4; i++) o[i] *= wv[i];
        }
        if (y && c < d) {
            float * yr = y + r * d;
            if (vec && c + 4 <= d) {
                *reinterpret_cast<float4 *>(yr + c) = make_float4(o[0], o[1], o[2], o[3]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (c + i < d) yr[c + i] = o[i];
            }
        }
        if (packed) pack4_expanded(packed, R_pad, r, c, o);
    }
}

// One workgroup (four waves) per row, for rows of at most 1024*NCH columns
// (padding included): thread t holds the 4 floats at columns 4t + 1024i,
// loaded at once; the sum of squares is a wave reduction and then a sum of
// the four waves' partials through LDS. Four times the waves of
// rms_norm_kernel for the same rows, so more loads are in flight.
//
// Row order: workgroups are dealt to the eight XCDs in turn (workgroup b to
// XCD b % 8), and a row writes only 32 bytes of each 128-byte line of the
// expanded operand (the other 96 are rows r^1..r^3 of its 4-row quartet).
// With a grid of 8k workgroups, workgroup b takes row (b % 8) * k + b / 8,
// so each XCD owns a contiguous run of k rows, every line is completed
// inside one XCD's L2, and no line leaves an L2 partly written
// (2048 x 2560 with the pack: 9.5 -> 7.3 us).
template <int NCH>
__global__ __launch_bounds__(256) void rms_norm_row_kernel(const float * __restrict__ x, int64_t rows, int64_t d,
                                                           float eps, const float * __restrict__ w,
                                                           float * __restrict__ y, uint8_t * __restrict__ packed,
                                                           int64_t R_pad) {
    __shared__ float part[4];
    const int t = threadIdx.x, lane = t & 63;
    const int64_t G = gridDim.x, b = blockIdx.x;
    const int64_t r = G % 8 == 0 ? (b % 8) * (G / 8) + b / 8 : b;
    const int64_t d_pad = zest_k_padded(d);
    if (r >= rows) {  // a padding row of the packed operand (the whole workgroup takes this branch)
        for (int64_t c = t * 4; c < d_pad; c += 1024)
            *reinterpret_cast<uint2 *>(packed + zest_xoffset(r, c, R_pad)) = make_uint2(0, 0);
        return;
    }
    const float * xr = x + r * d;
    const bool vec = (d & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    float v[NCH][4];
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        const int64_t c = t * 4 + 1024 * i;
        if (vec && c + 4 <= d) {
            const float4 q = *reinterpret_cast<const float4 *>(xr + c);
            v[i][0] = q.x;
            v[i][1] = q.y;
            v[i][2] = q.z;
            v[i][3] = q.w;
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++) v[i][q] = c + q < d ? xr[c + q] : 0.0f;
        }
    }
#pragma unroll
    for (int i = 0; i < NCH; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) ss += v[i][q] * v[i][q];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
    if (lane == 0) part[t >> 6] = ss;
    __syncthreads();
    ss = (part[0] + part[1]) + (part[2] + part[3]);
    const float sc = 1.0f / sqrtf(ss / (float) d + eps);
    const bool wvec = w && vec && (reinterpret_cast<uintptr_t>(w) & 15) == 0;
    const int64_t c_end = packed ? d_pad : d;
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        const int64_t c = t * 4 + 1024 * i;
        if (c >= c_end) continue;  // pair-uniform: c_end is a multiple of 8
        float o[4];
#pragma unroll
        for (int q = 0; q < 4; q++) o[q] = v[i][q] * sc;
        if (w) {
            if (wvec && c + 4 <= d) {
                const float4 q = *reinterpret_cast<const float4 *>(w + c);
                o[0] *= q.x;
                o[1] *= q.y;
                o[2] *= q.z;
                o[3] *= q.w;
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++) o[q] *= c + q < d ? w[c + q] : 0.0f;
            }
        }
        if (y && c < d) {
            float * yr = y + r * d;
            if (vec && c + 4 <= d) {
                *reinterpret_cast<float4 *>(yr + c) = make_float4(o[0], o[1], o[2], o[3]);
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (c + q < d) yr[c + q] = o[q];
            }
        }
        if (packed) pack4_expanded(packed, R_pad, r, c, o);
    }
}

// Narrow rows (d <= 256 floats, d % 4 == 0, 16-byte aligned, no packed
// output): the per-head norms of q and k. A row is L lanes of one float4 each
// (L the power of two that covers d), so a 256-thread workgroup holds 256/L
// rows at once and ROWS of them a thread, every load issued before the first
// sum. HBM bound: one workgroup per row, as the wider rows run, leaves 7 of 8
// lanes idle at d = 128 and is bound by dispatching 65536 workgroups
// (65536 x 128: 45.5 -> 11.6 us, 67 MB at 5.8 TB/s; 16384 x 128: 13.8 -> 5.9). The sums are
// rms_norm_row_kernel's own: its lanes past the row add zeros.
template <int L, int ROWS>
__global__ __launch_bounds__(256) void rms_norm_narrow_kernel(const float * __restrict__ x, int64_t rows, int64_t d,
                                                              float eps, const float * __restrict__ w,
                                                              float * __restrict__ y) {
    const int l = threadIdx.x % L, c = 4 * l;
    const int64_t r0 = (int64_t) blockIdx.x * (256 / L * ROWS) + threadIdx.x / L;
    const bool col = c < d;
    float4 v[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
        const int64_t r = r0 + i * (256 / L);
        v[i] = col && r < rows ? *reinterpret_cast<const float4 *>(x + r * d + c) : make_float4(0, 0, 0, 0);
    }
    const float4 wv = w && col ? *reinterpret_cast<const float4 *>(w + c) : make_float4(1, 1, 1, 1);
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
        const int64_t r = r0 + i * (256 / L);
        float ss = 0.0f;
        ss += v[i].x * v[i].x;
        ss += v[i].y * v[i].y;
        ss += v[i].z * v[i].z;
        ss += v[i].w * v[i].w;
#pragma unroll
        for (int off = L / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
        const float sc = 1.0f / sqrtf(ss / (float) d + eps);
        if (col && r < rows)
            *reinterpret_cast<float4 *>(y + r * d + c) =
                make_float4(v[i].x * sc * wv.x, v[i].y * sc * wv.y, v[i].z * sc * wv.z, v[i].w * sc * wv.w);
    }
}

// y = act(g) * u (REGLU as g > 0 ? g*u : 0). A piece is 16 rows by 64 columns,
// thread t row t/16 and the 4 floats at column 4(t%16), so the 16 threads of a
// row read 256 contiguous bytes and a wave's packed store fills whole 128-byte
// lines (4 rows by 16 columns each). A workgroup takes PIECES pieces that
// follow each other along the rows (a row's last piece is followed by the
// next rows' first, so narrow and ragged widths leave no thread idle), every
// load issued before the first activation. HBM bound; a thread of 16
// consecutive columns, whose 16-byte loads lie 64 bytes apart across the
// lanes, is bound by the vector cache instead (SWIGLU 2048 x 9728 packed 36.1
// -> 28.4 us, 7.0 TB/s, to fp32 45.5 -> 34.6). Two pieces where the tensors
// stay in the 256 MB last-level cache or the result is packed alone (GEGLU
// 2048 x 2560 packed 10.7 us, with four 11.9, with 256 columns of 16 rows a
// workgroup 12.3; SWIGLU 30000 x 320 packed 14.9, 15.9 and 18.5), four where
// an fp32 result takes them past it (2286 x 17408 84.5 us, with two 88.7).
// With a packed output the grid also covers its padding rows and columns,
// written as zeros.
template <int KIND, int PIECES>
__global__ __launch_bounds__(256) void glu_kernel(const float * __restrict__ g, int64_t sg, const float * __restrict__ u,
                                                  int64_t su, int64_t rows, int64_t f, float * __restrict__ y,
                                                  uint8_t * __restrict__ packed, int64_t R_pad, unsigned across,
                                                  unsigned pieces, bool vec, bool vec_y) {
    const int tr = threadIdx.x >> 4, tc = (threadIdx.x & 15) * 4;
    const unsigned first = blockIdx.x * PIECES;
    // piece i's first row and column (uniform)
    int64_t r0[PIECES], c0[PIECES];
    unsigned band = first / across, at = first % across;
#pragma unroll
    for (int i = 0; i < PIECES; i++) {
        r0[i] = (int64_t) band * 16;
        c0[i] = (int64_t) at * 64;
        if (++at == across) {
            at = 0;
            band++;
        }
    }
    const float * gt = g + tr * sg + tc;
    const float * ut = u + tr * su + tc;
    float4 gv[PIECES], uv[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; i++) {
        const int64_t c = c0[i] + tc;
        const bool row_ok = r0[i] + tr < rows;
        const float * gp = gt + (r0[i] * sg + c0[i]);
        const float * up = ut + (r0[i] * su + c0[i]);
        if (row_ok && vec && c + 4 <= f) {
            gv[i] = *reinterpret_cast<const float4 *>(gp);
            uv[i] = *reinterpret_cast<const float4 *>(up);
        } else {
            float a[4], b[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                a[q] = row_ok && c + q < f ? gp[q] : 0.0f;
                b[q] = row_ok && c + q < f ? up[q] : 0.0f;
            }
            gv[i] = make_float4(a[0], a[1], a[2], a[3]);
            uv[i] = make_float4(b[0], b[1], b[2], b[3]);
        }
    }
#pragma unroll
    for (int i = 0; i < PIECES; i++) {
        if (first + i >= pieces) break;
        const int64_t r = r0[i] + tr, c = c0[i] + tc;
        const bool row_ok = r < rows;
        const float a[4] = {gv[i].x, gv[i].y, gv[i].z, gv[i].w}, b[4] = {uv[i].x, uv[i].y, uv[i].z, uv[i].w};
        float o[4];
#pragma unroll
        for (int q = 0; q < 4; q++) o[q] = row_ok && c + q < f ? zest::glu(KIND, a[q], b[q]) : 0.0f;
        if (y && row_ok) {
            if (vec_y && c + 4 <= f) {
                *reinterpret_cast<float4 *>(y + r * f + c) = make_float4(o[0], o[1], o[2], o[3]);
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (c + q < f) y[r * f + c + q] = o[q];
            }
        }
        // a whole piece: a packed operand is whole 64-column tiles of whole 16-row groups
        if (packed) pack4_expanded(packed, R_pad, r, c, o);
    }
}

// Row-wise binary ops over rows x d (row-major, contiguous): y = a OP b,
// with b either the same shape or one row broadcast to every row (b_row).
// Thread t of column block x takes columns 4t + 1024x of rows y, y + Y, ...
// (a 2-D grid: no division per element), four at a time with 16-byte loads
// and stores when VEC (d % 4 == 0 and every pointer 16-byte aligned).
template <int OP, bool VEC>  // OP 0: add, 1: mul
__global__ __launch_bounds__(256) void binary_rows_kernel(const float * __restrict__ a, const float * __restrict__ b,
                                                          int64_t rows, int64_t d, int b_row, float * __restrict__ y) {
    const int64_t c = ((int64_t) blockIdx.x * 256 + threadIdx.x) * 4;
    if (c >= d) return;
    for (int64_t r = blockIdx.y; r < rows; r += gridDim.y) {
        const float * ar = a + r * d;
        const float * br = b_row ? b : b + r * d;
        float * yr = y + r * d;
        if (VEC) {
            const float4 u = *reinterpret_cast<const float4 *>(ar + c), v = *reinterpret_cast<const float4 *>(br + c);
            *reinterpret_cast<float4 *>(yr + c) = OP == 0 ? make_float4(u.x + v.x, u.y + v.y, u.z + v.z, u.w + v.w)
                                                          : make_float4(u.x * v.x, u.y * v.y, u.z * v.z, u.w * v.w);
        } else {
            for (int64_t i = c; i < c + 4 && i < d; i++) yr[i] = OP == 0 ? ar[i] + br[i] : ar[i] * br[i];
        }
    }
}

// y = x * s + b over n floats, four a thread (16-byte accesses when VEC).
template <bool VEC>
__global__ __launch_bounds__(256) void scale_kernel(const float * __restrict__ x, int64_t n, float s, float b,
                                                    float * __restrict__ y) {
    const int64_t i = ((int64_t) blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;
    if (VEC && i + 4 <= n) {
        const float4 u = *reinterpret_cast<const float4 *>(x + i);
        *reinterpret_cast<float4 *>(y + i) = make_float4(u.x * s + b, u.y * s + b, u.z * s + b, u.w * s + b);
    } else {
        for (int64_t k = i; k < i + 4 && k < n; k++) y[k] = x[k] * s + b;
    }
}

// NaN or infinity anywhere in rows x cols (row stride ld) sets *flag. The test
// is on the bits (exponent field all ones), so no fast-math can fold it away.
// 2-D grid as binary_rows_kernel, four columns a thread.
__global__ __launch_bounds__(256) void check_finite_kernel(const float * __restrict__ y, int64_t rows, int64_t cols,
                                                           int64_t ld, uint32_t * flag) {
    const int64_t c = ((int64_t) blockIdx.x * 256 + threadIdx.x) * 4;
    if (c >= cols) return;
    bool bad = false;
    for (int64_t r = blockIdx.y; r < rows; r += gridDim.y)
        for (int64_t i = c; i < c + 4 && i < cols; i++)
            bad |= (__float_as_uint(y[r * ld + i]) & 0x7f800000u) == 0x7f800000u;
    if (bad) atomicOr(flag, 1u);
}

// ROPE: one workgroup per token. Thread 0 walks θ through the pairs as the
// reference's table loop does (src/xdna-exec.cpp:225-233): θ_0 = pos, and
// θ_{p+1} = θ_p * theta_scale, one float multiplication a pair; each thread
// then forms the cos and sin of its pairs (rope_yarn), and the token's heads
// are rotated from that table (the rotation of :326-339); dimensions past
// n_dims are copied. Shared memory: n_dims/2 angles, then n_dims/2 (cos, sin).
struct rope_angles {
    const float * ff;  // per-frequency factors, or null
    float theta_scale, freq_scale, ext_factor, attn_factor, corr0, corr1;
};

__device__ inline float2 * rope_table(float * sh, int half, float pos, const rope_angles & g) {
    float * theta = sh;
    float2 * cs = reinterpret_cast<float2 *>(sh + ((half + 1) & ~1));
    if (threadIdx.x == 0) {
        float th = pos;
        for (int p = 0; p < half; p++) {
            theta[p] = th;
            th *= g.theta_scale;
        }
    }
    __syncthreads();
    for (int p = threadIdx.x; p < half; p += blockDim.x) {
        const float theta_extrap = g.ff ? theta[p] / g.ff[p] : theta[p];
        float th = g.freq_scale * theta_extrap, mscale = g.attn_factor;
        if (g.ext_factor != 0.0f) {
            // every operation rounded on its own, as the CPU's expression is:
            // a fused multiply-add moves the angle by an ulp, which at
            // positions in the tens of thousands shows in its sine and cosine
#pragma clang fp contract(off)
            const float yv = ((float) p - g.corr0) / fmaxf(0.001f, g.corr1 - g.corr0);
            const float ramp_mix = (1.0f - fminf(1.0f, fmaxf(0.0f, yv))) * g.ext_factor;
            th = th * (1.0f - ramp_mix) + theta_extrap * ramp_mix;
            mscale *= 1.0f + 0.1f * logf(1.0f / g.freq_scale);
        }
        cs[p] = make_float2(cosf(th) * mscale, sinf(th) * mscale);
    }
    __syncthreads();
    return cs;
}

// A pair rotated. Which product of each sum is rounded is written out, so
// every kernel gives the same bits (left to the compiler, each contracts its
// sums its own way).
__device__ inline float2 rotated(float x0, float x1, float2 r) {
    return make_float2(fmaf(x0, r.x, -(x1 * r.y)), fmaf(x0, r.y, x1 * r.x));
}

__global__ __launch_bounds__(256) void rope_kernel(const float * __restrict__ x, int64_t heads, int64_t d,
                                                   const int32_t * __restrict__ pos, int n_dims, int neox,
                                                   rope_angles g, float * __restrict__ y) {
    extern __shared__ float rope_sh[];
    const int half = n_dims / 2;
    const int64_t t = blockIdx.x;
    const float2 * cs = rope_table(rope_sh, half, (float) pos[t], g);
    const int64_t off = neox ? half : 1;
    for (int64_t k = threadIdx.x; k < heads * half; k += blockDim.x) {
        const int64_t h = k / half, p = k - h * half;
        const float * src = x + (t * heads + h) * d;
        float * dst = y + (t * heads + h) * d;
        const int64_t ic = neox ? p : 2 * p;
        const float2 r = cs[p];
        const float2 o = rotated(src[ic], src[ic + off], r);
        dst[ic] = o.x;
        dst[ic + off] = o.y;
    }
    const int64_t rest = d - n_dims;
    if (rest > 0)
        for (int64_t k = threadIdx.x; k < heads * rest; k += blockDim.x) {
            const int64_t h = k / rest, i = n_dims + (k - h * rest);
            y[(t * heads + h) * d + i] = x[(t * heads + h) * d + i];
        }
}

// The same with 16-byte accesses: a piece is four pairs of a head (NeoX: 4
// floats of each half; normal: 4 consecutive floats, two pairs), where heads
// start 16-byte aligned and a head's halves (NeoX) or rotated dimensions
// (normal) are whole pieces. Each thread requests its first ROPE_AHEAD pieces before
// the table is made, so their latency and the table's overlap; HBM bound
// (4096 x 48 x 128 with YaRN 47.2 -> 33.2 us, 201 MB; 2048 x 32 x 128 NeoX
// 13.5 -> 11.4 us; 4096 x 8 x 128 12.9 -> 10.6). A token of few pieces takes
// as many waves as hold them, so more tokens' tables are made at once (30000 x
// 1 x 64 with four waves a token 24.4 us, slower than the 22.6 of the kernel
// above; now 12.8).
constexpr int ROPE_AHEAD = 4;

template <bool NEOX>
__global__ __launch_bounds__(256) void rope_vec_kernel(const float * __restrict__ x, int heads, int d,
                                                       const int32_t * __restrict__ pos, int n_dims, rope_angles g,
                                                       float * __restrict__ y) {
    extern __shared__ float rope_sh[];
    constexpr int A = NEOX ? ROPE_AHEAD / 2 : ROPE_AHEAD;  // pieces in flight: 64 bytes a thread either way
    const int half = n_dims / 2, per = (NEOX ? half : n_dims) / 4, n = heads * per, nt = blockDim.x;
    const int64_t t = blockIdx.x;
    const float * xt = x + t * heads * d;
    float * yt = y + t * heads * d;
    float4 a[A], b[A];
    auto at = [&](int k) { return k / per * d + k % per * 4; };
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < A; i++) {
            const int k = k0 + nt * i;
            if (k < n) {
                a[i] = *reinterpret_cast<const float4 *>(xt + at(k));
                if (NEOX) b[i] = *reinterpret_cast<const float4 *>(xt + at(k) + half);
            }
        }
    };
    load(threadIdx.x);
    const float2 * cs = rope_table(rope_sh, half, (float) pos[t], g);
    for (int k0 = threadIdx.x; k0 < n; k0 += nt * A) {
        if (k0 != (int) threadIdx.x) load(k0);
#pragma unroll
        for (int i = 0; i < A; i++) {
            const int k = k0 + nt * i;
            if (k >= n) continue;
            float * dst = yt + at(k);
            const float2 * r = cs + k % per * (NEOX ? 4 : 2);
            if (NEOX) {
                const float2 o[4] = {rotated(a[i].x, b[i].x, r[0]), rotated(a[i].y, b[i].y, r[1]),
                                     rotated(a[i].z, b[i].z, r[2]), rotated(a[i].w, b[i].w, r[3])};
                *reinterpret_cast<float4 *>(dst) = make_float4(o[0].x, o[1].x, o[2].x, o[3].x);
                *reinterpret_cast<float4 *>(dst + half) = make_float4(o[0].y, o[1].y, o[2].y, o[3].y);
            } else {
                const float2 o[2] = {rotated(a[i].x, a[i].y, r[0]), rotated(a[i].z, a[i].w, r[1])};
                *reinterpret_cast<float4 *>(dst) = make_float4(o[0].x, o[0].y, o[1].x, o[1].y);
            }
        }
    }
    const int rest = (d - n_dims) / 4;
    for (int k = threadIdx.x; k < heads * rest; k += nt) {
        const int o = k / rest * d + n_dims + k % rest * 4;
        *reinterpret_cast<float4 *>(yt + o) = *reinterpret_cast<const float4 *>(xt + o);
    }
}

unsigned blocks_for(int64_t n, int per) { return (unsigned) ((n + per - 1) / per); }

// rows x d as (column blocks of 1024, up to 65535 row slots)
dim3 row_grid(int64_t rows, int64_t d) {
    return dim3(blocks_for(d, 1024), (unsigned) std::min<int64_t>(rows, 65535));
}

bool aligned16(const void * p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <int L>
void rms_norm_narrow(const float * x, int64_t rows, int64_t d, float eps, const float * w, float * y, hipStream_t s) {
    constexpr int ROWS = 4;
    hipLaunchKernelGGL((rms_norm_narrow_kernel<L, ROWS>), dim3((unsigned) ((rows + 256 / L * ROWS - 1) / (256 / L * ROWS))),
                       dim3(256), 0, s, x, rows, d, eps, w, y);
}

template <int OP>
void binary_rows(const float * a, const float * b, int64_t rows, int64_t d, int b_row, float * y,
                        hipStream_t s) {
    if (d % 4 == 0 && aligned16(a) && aligned16(b) && aligned16(y))
        hipLaunchKernelGGL((binary_rows_kernel<OP, true>), row_grid(rows, d), dim3(256), 0, s, a, b, rows, d, b_row, y);
    else
        hipLaunchKernelGGL((binary_rows_kernel<OP, false>), row_grid(rows, d), dim3(256), 0, s, a, b, rows, d, b_row, y);
}


} // namespace

extern "C" {

int zest_rms_norm(const float * x, int64_t rows, int64_t d, float eps, const float * w, float * y, void * packed,
                  void * stream) {
    ZEST_REQUIRE(x && (y || packed), "zest_rms_norm: null pointer");
    ZEST_REQUIRE(rows > 0 && d > 0, "zest_rms_norm: rows=%lld d=%lld", (long long) rows, (long long) d);
    ZEST_REQUIRE(!packed || d % 8 == 0, "zest_rms_norm: packing needs d %% 8 == 0");
    ZEST_REQUIRE(aligned16(packed), "zest_rms_norm: packed must be 16-byte aligned");
    // with a packed output, the grid also covers its padding rows (zeroed)
    const int64_t R_pad = zest_rows_padded(rows), grid_rows = packed ? R_pad : rows;
    const int64_t chunks = (zest_k_padded(d) + 255) / 256;  // the output pass covers the padded width
    hipStream_t s = zest::as_stream(stream);
    uint8_t * pk = (uint8_t *) packed;
    if (!packed && d <= 256 && d % 4 == 0 && aligned16(x) && aligned16(y) && aligned16(w)) {
        // several rows a workgroup
        if (d > 128) rms_norm_narrow<64>(x, rows, d, eps, w, y, s);
        else if (d > 64) rms_norm_narrow<32>(x, rows, d, eps, w, y, s);
        else rms_norm_narrow<16>(x, rows, d, eps, w, y, s);
    } else if (chunks <= 4)  // up to 1024 columns: one workgroup per row
        hipLaunchKernelGGL(rms_norm_row_kernel<1>, dim3((unsigned) grid_rows), dim3(256), 0, s, x, rows, d, eps, w, y,
                           pk, R_pad);
    else if (chunks <= 12)  // up to 3072
        hipLaunchKernelGGL(rms_norm_row_kernel<3>, dim3((unsigned) grid_rows), dim3(256), 0, s, x, rows, d, eps, w, y,
                           pk, R_pad);
    else if (chunks <= 24)  // up to 6144
        hipLaunchKernelGGL(rms_norm_row_kernel<6>, dim3((unsigned) grid_rows), dim3(256), 0, s, x, rows, d, eps, w, y,
                           pk, R_pad);
    else
        hipLaunchKernelGGL(rms_norm_kernel, dim3((unsigned) ((grid_rows + NORM_ROWS - 1) / NORM_ROWS)),
                           dim3(NORM_ROWS * 64), 0, s, x, rows, d, eps, w, y, pk, R_pad);
    return zest::check_launch("zest_rms_norm");
}

int zest_glu(int kind, const float * g, int64_t sg, const float * u, int64_t su, int64_t rows, int64_t f, float * y,
             void * packed, void * stream) {
    ZEST_REQUIRE(g && u && (y || packed), "zest_glu: null pointer");
    ZEST_REQUIRE(rows > 0 && f > 0 && sg >= f && su >= f, "zest_glu: bad shape");
    ZEST_REQUIRE(!packed || f % 8 == 0, "zest_glu: packing needs f %% 8 == 0");
    ZEST_REQUIRE(aligned16(packed), "zest_glu: packed must be 16-byte aligned");
    const int64_t R_pad = zest_rows_padded(rows), gr = packed ? R_pad : rows;
    const int64_t across = (f + 63) / 64, pieces = (gr + 15) / 16 * across;
    ZEST_REQUIRE(pieces < (1ll << 31), "zest_glu: %lld x %lld is too large", (long long) rows, (long long) f);
    const bool four = y && 3.0 * sizeof(float) * (double) rows * (double) f > (double) (256 << 20);
    const dim3 grid(blocks_for(pieces, four ? 4 : 2));
    const bool vec = sg % 4 == 0 && su % 4 == 0 && aligned16(g) && aligned16(u), vec_y = f % 4 == 0 && aligned16(y);
    hipStream_t s = zest::as_stream(stream);
    uint8_t * p = (uint8_t *) packed;
#define ZEST_GLU(KIND)                                                                                                  \
    case KIND:                                                                                                          \
        hipLaunchKernelGGL((four ? glu_kernel<KIND, 4> : glu_kernel<KIND, 2>), grid, dim3(256), 0, s, g, sg, u, su,     \
                           rows, f, y, p, R_pad, (unsigned) across, (unsigned) pieces, vec, vec_y);                     \
        break
    switch (kind) {
        ZEST_GLU(ZEST_GLU_SWIGLU);
        ZEST_GLU(ZEST_GLU_GEGLU);
        ZEST_GLU(ZEST_GLU_GEGLU_ERF);
        ZEST_GLU(ZEST_GLU_GEGLU_QUICK);
        ZEST_GLU(ZEST_GLU_REGLU);
        default: return zest::fail(ZEST_E_UNSUPPORTED, "zest_glu: GLU kind %d", kind);
    }
#undef ZEST_GLU
    return zest::check_launch("zest_glu");
}

int zest_add(const float * a, const float * b, int64_t rows, int64_t d, int b_is_row, float * y, void * stream) {
    ZEST_REQUIRE(a && b && y && rows > 0 && d > 0, "zest_add: bad arguments");
    binary_rows<0>(a, b, rows, d, b_is_row != 0, y, zest::as_stream(stream));
    return zest::check_launch("zest_add");
}

int zest_mul_row(const float * x, const float * w, int64_t rows, int64_t d, float * y, void * stream) {
    ZEST_REQUIRE(x && w && y && rows > 0 && d > 0, "zest_mul_row: bad arguments");
    binary_rows<1>(x, w, rows, d, 1, y, zest::as_stream(stream));
    return zest::check_launch("zest_mul_row");
}

int zest_scale(const float * x, int64_t n, float s, float b, float * y, void * stream) {
    ZEST_REQUIRE(x && y && n > 0, "zest_scale: bad arguments");
    const dim3 grid(blocks_for(n, 1024));
    if (aligned16(x) && aligned16(y))
        hipLaunchKernelGGL((scale_kernel<true>), grid, dim3(256), 0, zest::as_stream(stream), x, n, s, b, y);
    else
        hipLaunchKernelGGL((scale_kernel<false>), grid, dim3(256), 0, zest::as_stream(stream), x, n, s, b, y);
    return zest::check_launch("zest_scale");
}

int zest_rope(const float * x, int64_t T, int64_t heads, int64_t d, const int32_t * pos, const float * ff, int n_dims,
              int mode, float freq_base, float freq_scale, float ext_factor, float attn_factor, float corr0, float corr1,
              float * y, void * stream) {
    ZEST_REQUIRE(x && pos && y && T > 0 && heads > 0 && d > 0, "zest_rope: bad arguments");
    ZEST_REQUIRE(n_dims > 0 && n_dims % 2 == 0 && n_dims <= d, "zest_rope: n_dims=%d d=%lld", n_dims, (long long) d);
    ZEST_REQUIRE(mode == 0 || mode == 2, "zest_rope: mode %d (normal 0 or neox 2)", mode);
    ZEST_REQUIRE(T <= 0x7fffffff, "zest_rope: %lld tokens", (long long) T);
    const float theta_scale = powf(freq_base, -2.0f / (float) n_dims);
    const int half = n_dims / 2;
    const size_t lds = (size_t) (((half + 1) & ~1) + 2 * half) * sizeof(float);
    ZEST_REQUIRE(lds <= 65536, "zest_rope: n_dims=%d needs %zu bytes of shared memory (at most 65536)", n_dims, lds);
    const rope_angles g{ff, theta_scale, freq_scale, ext_factor, attn_factor, corr0, corr1};
    const hipStream_t s = zest::as_stream(stream);
    // whole 16-byte pieces of every head (a token's offsets then fit 32 bits)
    const bool vec = d % 4 == 0 && (mode == 2 ? half : n_dims) % 4 == 0 && aligned16(x) && aligned16(y) &&
                     heads <= (1 << 30) / d;
    const int64_t pieces = heads * std::max<int64_t>(mode == 2 ? half : n_dims, d - n_dims) / 4;
    const dim3 threads(pieces <= 64 ? 64 : pieces <= 128 ? 128 : 256);
    if (vec && mode == 2)
        hipLaunchKernelGGL(rope_vec_kernel<true>, dim3((unsigned) T), threads, lds, s, x, (int) heads, (int) d, pos,
                           n_dims, g, y);
    else if (vec)
        hipLaunchKernelGGL(rope_vec_kernel<false>, dim3((unsigned) T), threads, lds, s, x, (int) heads, (int) d, pos,
                           n_dims, g, y);
    else
        hipLaunchKernelGGL(rope_kernel, dim3((unsigned) T), dim3(256), lds, s, x, heads, d, pos, n_dims, mode == 2, g,
                           y);
    return zest::check_launch("zest_rope");
}

int zest_check_finite(const float * y, int64_t rows, int64_t cols, int64_t ld, uint32_t * flag, void * stream) {
    ZEST_REQUIRE(y && flag && rows > 0 && cols > 0 && ld >= cols, "zest_check_finite: bad arguments");
    ZEST_REQUIRE((reinterpret_cast<uintptr_t>(flag) & 3) == 0, "zest_check_finite: flag must be 4-byte aligned");
    hipLaunchKernelGGL(check_finite_kernel, row_grid(rows, cols), dim3(256), 0, zest::as_stream(stream), y, rows, cols,
                       ld, flag);
    return zest::check_launch("zest_check_finite");
}

} // extern "C"
