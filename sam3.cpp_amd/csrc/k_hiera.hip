// k_hiera.hip — data movement of the SAM 2.x Hiera encoder around the shared
// GEMM and attention kernels (sam2_build_hiera_graph, sam3.cpp:4462-4527;
// sam2_hiera_block_forward, sam3.cpp:4295-4457; the FPN top-down path,
// sam3.cpp:4567-4590).  All activations are NHWC: token (y, x) is a row of
// channels.
#include "s3e_internal.h"

namespace s3e {
namespace {

// 8 values as fp16 (h) and as the fp16 of what that rounding left (l), packed
__device__ __forceinline__ void split8(const float (&v)[8], uint32_t (&h)[4], uint32_t (&l)[4]) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const _Float16 a = to_half(v[2 * j]), b = to_half(v[2 * j + 1]);
        h[j] = (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
        const _Float16 c = (_Float16)(v[2 * j] - (float)a), d = (_Float16)(v[2 * j + 1] - (float)b);
        l[j] = (uint32_t)__builtin_bit_cast(uint16_t, c) | ((uint32_t)__builtin_bit_cast(uint16_t, d) << 16);
    }
}

// im2col of the patch embedding (Conv2d 3→E, k×k, stride, pad): CHW f32
// [3][S][S] → rows [OH·OW][ldk] in F32 or F16 (ggml's im2col in the kernel
// type), K ordered [c][ky][kx] as the kernel rows are; taps outside the image
// and columns K..ldk are zero.  A thread makes 8 columns of one row (one
// 16-byte store per fp16 plane) and steps c, ky, kx from the first, so the
// divisions are paid once per 8 values; lanes run along the row.  1024² fp16: 36.6 → 18.5 µs.
__global__ __launch_bounds__(256) void k_im2col_conv(const float *__restrict__ chw, int S, int k, int stride, int pad,
                                                     int OW, uint32_t n8, uint32_t ld8, int kind, void *out,
                                                     _Float16 *lo) {
    // 32-bit index arithmetic (the launcher keeps T·ldk below 2^31)
    const uint32_t idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= n8) return;
    const uint32_t t = idx / ld8;
    const int k0 = (int)(idx - t * ld8) * 8;
    const int oy = (int)(t / (uint32_t)OW), ox = (int)(t - (uint32_t)oy * OW);
    const int y0 = oy * stride - pad, x0 = ox * stride - pad;
    int c = k0 / (k * k), r = k0 - c * k * k, ky = r / k, kx = r - ky * k;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int iy = y0 + ky, ix = x0 + kx;
        v[j] = c < 3 && iy >= 0 && iy < S && ix >= 0 && ix < S ? chw[((int64_t)c * S + iy) * S + ix] : 0.f;
        if (++kx == k) {
            kx = 0;
            if (++ky == k) { ky = 0; c++; }
        }
    }
    if (kind == A_F16 || kind == A_F16X2) {
        uint32_t h[4], l[4];
        split8(v, h, l);
        ((uint4 *)out)[idx] = make_uint4(h[0], h[1], h[2], h[3]);
        if (kind == A_F16X2) ((uint4 *)lo)[idx] = make_uint4(l[0], l[1], l[2], l[3]);
    } else {
        ((float4 *)out)[2 * (int64_t)idx] = make_float4(v[0], v[1], v[2], v[3]);
        ((float4 *)out)[2 * (int64_t)idx + 1] = make_float4(v[4], v[5], v[6], v[7]);
    }
}

// Attention operands of one Hiera block that the QKV GEMM does not write.
// Windows of wh × ww tokens, row-major over nwx per row, cover the
// zero-padded grid; a padded position takes the QKV bias, as ggml_pad's zero
// rows do after the projection.  Q is max-pooled 2×2 inside each window under
// Q stride (sam2_maxpool_2d on the window's grid).  Heads are zero-padded from
// HD to HDp channels.  Q, K: [b·NH + h][pos][HDp]; Vᵀ: [b·NH + h][HDp][ldv]
// with keys in vt_slot order and zeros for keys Nkv .. ldv − 1.  With lo
// planes the values are split hi + lo.
struct Prep {
    const float *qkv, *bias;  // Q rows (f32, bias added); the QKV bias
    int64_t ld;  // row stride of qkv in floats
    int H, W, C, NH, HD, HDp;
    int wh, ww, nwx, qs;
    int Nq, Nkv, ldv, NW;
    _Float16 *q, *k, *vt, *q_lo, *k_lo, *vt_lo;
};

// Max-pooled Q of a Q-stride block from its f32 Q rows: one thread per (b, h,
// query, 8 channels), so the index arithmetic and the window lookup are paid
// once per 8 values and rows go by 16 and 32 bytes (HD % 8 = 0).  256² tokens of
// 192 in 8 × 8 windows: 22.6 µs a value per thread, 11 so.
__global__ __launch_bounds__(256) void k_hiera_qpool(Prep p, uint32_t n8) {
    // 32-bit index arithmetic (the launcher keeps totals below 2^31)
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    const uint32_t nch = (uint32_t)p.HDp / 8;
    const uint32_t r = i / nch;
    const int d0 = (int)(i - r * nch) * 8;
    const uint32_t bh = r / (uint32_t)p.Nq;
    const int pos = (int)(r - bh * p.Nq);
    const int b = (int)(bh / (uint32_t)p.NH), h = (int)(bh - (uint32_t)b * p.NH);
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (d0 < p.HD) {
        const int col = h * p.HD + d0, qw = p.ww / 2;
        const int wy = b / p.nwx, wx = b - wy * p.nwx, qy = pos / qw, qx = pos - qy * qw;
        const int y = wy * p.wh + 2 * qy, x = wx * p.ww + 2 * qx;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int yy = y + (k >> 1), xx = x + (k & 1);
            const float *src = yy < p.H && xx < p.W ? p.qkv + ((int64_t)yy * p.W + xx) * p.ld + col : p.bias + col;
            const float4 a = *(const float4 *)src, c = *(const float4 *)(src + 4);
            const float u[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = k == 0 ? u[j] : fmaxf(v[j], u[j]);
        }
    }
    uint32_t hw[4], lw[4];
    split8(v, hw, lw);
    ((uint4 *)p.q)[i] = make_uint4(hw[0], hw[1], hw[2], hw[3]);
    if (p.q_lo) ((uint4 *)p.q_lo)[i] = make_uint4(lw[0], lw[1], lw[2], lw[3]);
}

// Window positions outside the grid (ggml pads the normed input with zeros, so
// after the projection they hold the QKV bias; zeros past HD) for Q (without
// Q stride), K and Vᵀ, and the Vᵀ slots from Nkv to ldv (zeros).  Threads
// cover only those places: first (padded grid position, head, 8 channels) —
// the padded positions are the rows H..Hp−1 of the padded Hp × Wp grid, then
// columns W..Wp−1 of rows 0..H−1 — then (window·head, tail slot, 8 channels).
// 32-bit index arithmetic (the launcher keeps the counts below 2^31).
__global__ void k_hiera_pad(Prep p, int with_q, uint32_t n_pad, uint32_t n_tail) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t nch = p.HDp / 8;
    if (i < n_pad) {
        const uint32_t r = i / nch, q = r / (uint32_t)p.NH;
        const int d0 = (int)(i - r * nch) * 8, h = (int)(r - q * p.NH);
        const uint32_t Wp = (uint32_t)p.nwx * p.ww, Hp = (uint32_t)(p.NW / p.nwx) * p.wh;
        const uint32_t below = (Hp - p.H) * Wp;  // positions in the rows past the grid
        uint32_t y, x;
        if (q < below) {
            y = p.H + q / Wp;
            x = q - (y - p.H) * Wp;
        } else {
            const uint32_t q2 = q - below, wr = Wp - p.W;
            y = q2 / wr;
            x = p.W + (q2 - y * wr);
        }
        const uint32_t wy = y / p.wh, wx = x / p.ww;
        const int b = (int)(wy * p.nwx + wx);
        const int pos = (int)((y - wy * p.wh) * p.ww + (x - wx * p.ww));
        const int64_t bh = (int64_t)b * p.NH + h;
        const int64_t vrow = bh * p.HDp;
        const int64_t slot = vt_slot(pos);
        // (HD is a multiple of 8: the 8 channels are all real or all padding)
        const bool real = d0 < p.HD;
        const int col = h * p.HD + d0;
        uint32_t hw[4], lw[4];
        auto bias8 = [&](int sel) {
            float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (real) {
                const float4 a = *(const float4 *)(p.bias + sel * p.C + col), c = *(const float4 *)(p.bias + sel * p.C + col + 4);
                v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
                v[4] = c.x; v[5] = c.y; v[6] = c.z; v[7] = c.w;
            }
            split8(v, hw, lw);
        };
        const int64_t o = (bh * p.Nkv + pos) * p.HDp + d0;
        bias8(1);
        *(uint4 *)(p.k + o) = make_uint4(hw[0], hw[1], hw[2], hw[3]);
        if (p.k_lo) *(uint4 *)(p.k_lo + o) = make_uint4(lw[0], lw[1], lw[2], lw[3]);
        if (with_q) {
            bias8(0);
            *(uint4 *)(p.q + o) = make_uint4(hw[0], hw[1], hw[2], hw[3]);
            if (p.q_lo) *(uint4 *)(p.q_lo + o) = make_uint4(lw[0], lw[1], lw[2], lw[3]);
        }
        if (real) {
            bias8(2);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int64_t ov = (vrow + d0 + j) * p.ldv + slot;
                p.vt[ov] = __builtin_bit_cast(_Float16, (uint16_t)(hw[j / 2] >> (16 * (j & 1))));
                if (p.vt_lo) p.vt_lo[ov] = __builtin_bit_cast(_Float16, (uint16_t)(lw[j / 2] >> (16 * (j & 1))));
            }
        }
        return;
    }
    const uint32_t j = i - n_pad;
    if (j >= n_tail) return;
    const uint32_t tails = (uint32_t)(p.ldv - p.Nkv);
    const uint32_t r = j / nch, bh = r / tails;
    const int d0 = (int)(j - r * nch) * 8;
    const int64_t slot = vt_slot(p.Nkv + (int)(r - bh * tails));
    const int64_t vrow = (int64_t)bh * p.HDp;
    for (int d = d0; d < d0 + 8; d++) {
        p.vt[(vrow + d) * p.ldv + slot] = (_Float16)0.f;
        if (p.vt_lo) p.vt_lo[(vrow + d) * p.ldv + slot] = (_Float16)0.f;
    }
}

// dst [side²][D] += nearest ×2 upsampling of src [(side/2)²][D]
// (ggml_upscale NEAREST, then ggml_add; sam3.cpp:4575-4580)
__global__ void k_upsample_add(float *__restrict__ dst, const float *__restrict__ src, int side, int D,
                               int64_t n4) {
    // 32-bit index arithmetic (the launcher keeps n4 below 2^31)
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (uint32_t)n4) return;
    const uint32_t d4 = D / 4;
    const uint32_t pix32 = i / d4;
    const int64_t pix = pix32;
    const int c = (int)(i - pix32 * d4) * 4;
    const int y = (int)(pix32 / (uint32_t)side), x = (int)(pix32 - (uint32_t)y * side);
    const float4 u = *(const float4 *)(src + ((int64_t)(y / 2) * (side / 2) + x / 2) * D + c);
    float4 *o = (float4 *)(dst + pix * D + c);
    const float4 a = *o;
    *o = make_float4(__fadd_rn(a.x, u.x), __fadd_rn(a.y, u.y), __fadd_rn(a.z, u.z), __fadd_rn(a.w, u.w));
}

}  // namespace

hipError_t launch_im2col_conv(const float *chw, int S, int k, int stride, int pad, int64_t ldk, AKind kind,
                              void *out, hipStream_t st, void *lo) {
    const int O = (S + 2 * pad - k) / stride + 1;
    if ((kind != A_F16 && kind != A_F32 && kind != A_F16X2) || (kind == A_F16X2 && !lo) || ldk < 3LL * k * k)
        return hipErrorInvalidValue;
    const int64_t T = (int64_t)O * O, total = T * ldk;
    if (total >= INT32_MAX || ldk % 8 != 0 || (uintptr_t)out % 16 != 0 || (uintptr_t)lo % 16 != 0) return hipErrorInvalidValue;
    const uint32_t n8 = (uint32_t)(total / 8);
    hipLaunchKernelGGL(k_im2col_conv, dim3((n8 + 255) / 256), dim3(256), 0, st, chw, S, k, stride, pad, O, n8,
                       (uint32_t)(ldk / 8), (int)kind, out, (_Float16 *)lo);
    return hipGetLastError();
}

namespace {

Prep make_prep(const HieraPrepArgs &a) {
    Prep p;
    p.qkv = a.qkv;
    p.bias = a.bias;
    p.ld = a.qkv_ld;
    p.H = a.H; p.W = a.W; p.C = a.C; p.NH = a.NH; p.HD = a.HD; p.HDp = a.HDp;
    p.qs = a.q_stride;
    if (a.window > 0) {
        p.wh = p.ww = a.window;
        p.nwx = (a.W + a.window - 1) / a.window;
        p.NW = p.nwx * ((a.H + a.window - 1) / a.window);
    } else {
        p.wh = a.H;
        p.ww = a.W;
        p.nwx = 1;
        p.NW = 1;
    }
    p.Nkv = p.wh * p.ww;
    p.Nq = a.q_stride ? (p.wh / 2) * (p.ww / 2) : p.Nkv;
    p.ldv = (int)vt_ld_for(p.Nkv);
    p.q = a.q; p.k = a.k; p.vt = a.vt; p.q_lo = a.q_lo; p.k_lo = a.k_lo; p.vt_lo = a.vt_lo;
    return p;
}

}  // namespace

hipError_t launch_hiera_qpool(const HieraPrepArgs &a, hipStream_t st) {
    const Prep p = make_prep(a);
    if (!a.q_stride || p.HD <= 0 || p.HD > p.HDp || p.HD % 8 != 0 || p.HDp % 8 != 0 || p.ld < p.C || p.ld % 4 != 0 ||
        p.C % 8 != 0 || p.wh % 2 != 0 || p.ww % 2 != 0 || !p.q || !p.qkv || !p.bias)
        return hipErrorInvalidValue;
    const int64_t n8 = (int64_t)p.NW * p.NH * p.Nq * (p.HDp / 8);
    if (n8 >= INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_hiera_qpool, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, st, p, (uint32_t)n8);
    return hipGetLastError();
}

hipError_t launch_hiera_pad(const HieraPrepArgs &a, hipStream_t st) {
    const Prep p = make_prep(a);
    if (p.HD > p.HDp || p.HD % 8 != 0 || p.HDp % 8 != 0 || !p.k || !p.vt || !p.bias || (!a.q_stride && !p.q))
        return hipErrorInvalidValue;
    const int64_t Wp = (int64_t)p.nwx * p.ww, Hp = (int64_t)(p.NW / p.nwx) * p.wh;
    if (Wp < p.W || Hp < p.H || (int64_t)(p.NW / p.nwx) * p.nwx != p.NW || p.ldv < p.Nkv) return hipErrorInvalidValue;
    const int64_t n_pad = (Hp * Wp - (int64_t)p.H * p.W) * p.NH * (p.HDp / 8);
    const int64_t n_tail = (int64_t)p.NW * p.NH * (p.ldv - p.Nkv) * (p.HDp / 8);
    // nothing to fill when the windows tile the grid and hold whole 16-key groups
    if (n_pad + n_tail == 0) return hipSuccess;
    if (n_pad + n_tail >= INT32_MAX) return hipErrorInvalidValue;
    const int64_t total = n_pad + n_tail;
    hipLaunchKernelGGL(k_hiera_pad, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, p, a.q_stride ? 0 : 1,
                       (uint32_t)n_pad, (uint32_t)n_tail);
    return hipGetLastError();
}

hipError_t launch_upsample_add(float *dst, const float *src, int side, int D, hipStream_t st) {
    if (D % 4 != 0 || side % 2 != 0) return hipErrorInvalidValue;
    const int64_t n4 = (int64_t)side * side * (D / 4);
    if (n4 >= INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_upsample_add, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st, dst, src, side, D, n4);
    return hipGetLastError();
}

}  // namespace s3e
