// The vision front-end of the GWP-0.5 request: the three camera views
// composed into one canvas and patchified for the VAE encoder, and the VAE's
// BF16 convolutions.
//
//  * preprocess_views_kernel (the role of wam.cpp's preprocess_kernel,
//    src/models/gwp05/kernels/cuda_preprocess.cu:45-137, and of the CPU
//    compose_and_patchify, src/models/gwp05/engine/vae.cpp:1-133): canvas
//    out_w x out_h, top half the high camera, bottom-left / bottom-right the
//    two wrist cameras; each view is resized to cover its region (scale =
//    max of the two axis ratios, sizes rounded half away from zero) and
//    centre-cropped, with a triangle (bilinear, antialiased when shrinking:
//    support max(1, 1/scale)) filter whose taps are clamped to the image and
//    normalised to sum 1, applied along x, then along y.  The canvas is
//    written 2x2 pixel-unshuffled as f32 [12][out_h/2][out_w/2], channel
//    4c + 2dx + dy, mapped to [-1, 1] (v * 2 - 1); u8 pixels are v / 255.
//    One thread per output value.
//  * conv2d: ggml_conv_2d_direct on bf16 (the patch's cuDNN implicit GEMM,
//    native-bf16.patch:174-218) as a GEMM on MFMA over an im2col of the
//    input taken a row range at a time (so the column matrix never exceeds a
//    workspace half): y[b][oc][p] = sum_k col[p][k] w[oc][k], k = ic*KH*KW +
//    ky*KW + kx, f32 accumulation, one rounding to the output type.
#include <algorithm>
#include <type_traits>

#include "../internal.h"
#include "device.h"

namespace wamx {

struct ViewDev {
    const void * data;
    int32_t format, w, h;       // format 0: u8 RGB, 1: f32 RGB in [0, 1]
    int32_t dw, dh, x0, y0;     // destination region of the canvas
};
struct Views {
    ViewDev v[3];
};

__device__ __forceinline__ float pixel(const ViewDev & v, int x, int y, int c) {
    const size_t i = ((size_t) y * v.w + x) * 3 + c;
    return v.format == 0 ? (float) ((const uint8_t *) v.data)[i] * (1.0f / 255.0f) : ((const float *) v.data)[i];
}

// Taps of output position `o` along one axis: the source range [first,
// last], the filter centre and support.
struct Axis {
    int first, last;
    float center, support;
};
__device__ __forceinline__ Axis axis_of(int o, int src, int resized, int dst) {
    const int crop = (resized - dst) / 2;
    const float scale = (float) resized / (float) src;
    Axis a;
    a.support = fmaxf(1.0f, 1.0f / scale);
    a.center = ((float) (o + crop) + 0.5f) / scale - 0.5f;
    a.first = (int) ceilf(a.center - a.support);
    a.last = (int) floorf(a.center + a.support);
    return a;
}
__device__ __forceinline__ float tap(const Axis & a, int s) {
    return fmaxf(0.0f, 1.0f - fabsf((float) s - a.center) / a.support);
}

__global__ __launch_bounds__(256) void preprocess_views_kernel(Views views, int out_w, int out_h, float * out) {
    const int pw = out_w / 2, ph = out_h / 2;
    const int64_t n = (int64_t) 12 * pw * ph;
    const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int x = (int) (i % pw), y = (int) ((i / pw) % ph), ch = (int) (i / ((int64_t) pw * ph));
    const int c = ch / 4, dx = (ch % 4) / 2, dy = ch % 2;
    const int cx = 2 * x + dx, cy = 2 * y + dy;
    const int vi = cy < out_h / 2 ? 0 : (cx < out_w / 2 ? 1 : 2);
    const ViewDev & v = views.v[vi];
    const int lx = cx - v.x0, ly = cy - v.y0;
    const float s = fmaxf((float) v.dw / (float) v.w, (float) v.dh / (float) v.h);
    const int rw = (int) roundf((float) v.w * s), rh = (int) roundf((float) v.h * s);
    const Axis ax = axis_of(lx, v.w, rw, v.dw), ay = axis_of(ly, v.h, rh, v.dh);
    float tx = 0.0f, ty = 0.0f;
    for (int sx = ax.first; sx <= ax.last; ++sx) tx += tap(ax, sx);
    for (int sy = ay.first; sy <= ay.last; ++sy) ty += tap(ay, sy);
    float acc = 0.0f;
    for (int sy = ay.first; sy <= ay.last; ++sy) {
        const int yy = min(max(sy, 0), v.h - 1);
        float row = 0.0f;
        for (int sx = ax.first; sx <= ax.last; ++sx)
            row += pixel(v, min(max(sx, 0), v.w - 1), yy, c) * (tap(ax, sx) / tx);
        acc += row * (tap(ay, sy) / ty);
    }
    out[i] = acc * 2.0f - 1.0f;
}

// Rows [p0, p0 + rows) of the column matrix of batch image `b`: col[r][k],
// zero where the tap falls in the padding.  Source bf16 or f32, column bf16
// (or f32 for an f32 convolution).
struct ConvDev {
    const void * x;
    void * col;
    int32_t x_type, col_type;
    int64_t IW, IH, IC, KW, KH, OW, OH;
    int32_t s0, s1, p0, p1, d0, d1;
};
__global__ __launch_bounds__(256) void conv_col_kernel(ConvDev c, int64_t b, int64_t p_begin, int64_t rows) {
    const int64_t K = c.IC * c.KH * c.KW;
    const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
    if (i >= rows * K) return;
    const int64_t r = i / K, k = i % K, p = p_begin + r;
    const int64_t oy = p / c.OW, ox = p % c.OW;
    const int64_t ic = k / (c.KH * c.KW), ky = (k / c.KW) % c.KH, kx = k % c.KW;
    const int64_t iy = oy * c.s1 - c.p1 + ky * c.d1, ix = ox * c.s0 - c.p0 + kx * c.d0;
    const bool in = iy >= 0 && iy < c.IH && ix >= 0 && ix < c.IW;
    const int64_t si = ((b * c.IC + ic) * c.IH + (in ? iy : 0)) * c.IW + (in ? ix : 0);
    if (c.col_type == WAMX_TYPE_BF16) {
        uint16_t v = 0;
        if (in) v = c.x_type == WAMX_TYPE_BF16 ? ((const uint16_t *) c.x)[si] : f32_to_bf16(((const float *) c.x)[si]);
        ((uint16_t *) c.col)[i] = v;
    } else {
        ((float *) c.col)[i] = in ? ((const float *) c.x)[si] : 0.0f;
    }
}

// ---------------------------------------------------------------------------
// bf16 convolution as an implicit GEMM.  A first launch lays the image out
// channels-last with its padding ([IH + 2 p1][IW + 2 p0][ICp], channels padded
// with zeros to a multiple of 32) and the kernel as [OC][tap][ICp].  In that
// order the column matrix needs no memory of its own: the 32 channels of one
// tap that a K step multiplies are 64 consecutive bytes of an output pixel's
// image row, at the pixel's address plus an offset that depends on the tap
// alone.  conv_gemm_kernel copies them from the image straight into its LDS
// ring (global_load_lds) as a plain product would its operand rows.
//
// The column matrix this replaces was 9 times the image, written and read
// back in workspace-sized pieces: 160 -> 160 channels, 3 x 3, 192 x 160 pixels
// took 204 us of column kernels, 77 us of products in 3 pieces and 31 us for the
// bias; now 10 us of packing and 33 us of product that writes the convolution
// and, with the bias node after it, its sum (425 TFLOP/s; about 0.5 us per K
// step, of which MFMAs and LDS reads account for 0.2).
// ---------------------------------------------------------------------------
struct ConvGemm {
    const uint16_t * x;   // image b [IC][IH][IW]
    const uint16_t * k;   // [OC][IC][taps]
    uint16_t * xp;        // [rows][IWp][ICp], padded image rows from row iy0
    uint16_t * kp;        // [OC][taps][ICp]
    uint16_t * y;         // image b [OC][P], at the band's first pixel
    uint16_t * out;       // y + bias (laid out as y), or null
    const uint16_t * bias;
    float * part;         // [splits][OC][P of the band], or null
    int64_t IW, IH, IC, OC, P;       // P: pixels of a whole output plane (row stride of y)
    int IWp, ICp, OW, pix;           // pix: output pixels of the band
    int iy0, rows;                   // first padded image row and rows of the band
    int KW, taps, s0, s1, p0, p1, d0, d1;
    int ksteps;                      // K steps (of 32) per slice
};

constexpr int kPackPix = 64;  // pixels per workgroup of the packing kernel

// Workgroups [0, image) pack 64 pixels of one padded row by 32 channels each,
// through LDS: reads along x, writes 64 bytes of channels per pixel.  The rest
// pack the kernel, 8 channels of one (output channel, tap) per thread.
__global__ __launch_bounds__(256) void conv_pack_kernel(ConvGemm c, int image) {
    __shared__ uint32_t tile[kPackPix][17];  // [pixel][channel pairs]
    const int t = threadIdx.x;
    if ((int) blockIdx.x >= image) {
        const int64_t i = (int64_t) ((int) blockIdx.x - image) * 256 + t, cpr = c.ICp / 8;
        if (i >= c.OC * c.taps * cpr) return;
        const int64_t oc = i / (c.taps * cpr), tap = i / cpr % c.taps, ic = 8 * (i % cpr);
        const uint16_t * src = c.k + (oc * c.IC + ic) * c.taps + tap;
        uint32_t e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = ic + j < c.IC ? src[j * c.taps] : 0;
        *(uint4 *) (c.kp + 8 * i) = make_uint4(e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16);
        return;
    }
    const int nx = (c.IWp + kPackPix - 1) / kPackPix, nc = c.ICp / 32;
    const int bx = (int) blockIdx.x % nx, bc = (int) blockIdx.x / nx % nc, row = (int) blockIdx.x / (nx * nc);
    const int iy = c.iy0 + row - c.p1;
    const int px = bx * kPackPix + (t & 63), ix = px - c.p0;
    const bool in = iy >= 0 && iy < c.IH && ix >= 0 && ix < c.IW;
    const int64_t plane = c.IH * c.IW;
    const uint16_t * src = c.x + (in ? (int64_t) iy * c.IW + ix : 0);
    const int ch = 32 * bc + 8 * (t >> 6);  // the thread's 8 channels of pixel px
    uint32_t v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = src[min((int64_t) (ch + j), c.IC - 1) * plane];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t lo = in && ch + 2 * j < c.IC ? v[2 * j] : 0, hi = in && ch + 2 * j + 1 < c.IC ? v[2 * j + 1] : 0;
        tile[t & 63][4 * (t >> 6) + j] = lo | hi << 16;
    }
    __syncthreads();
    const int q = t >> 2, part = t & 3, opx = bx * kPackPix + q;
    if (opx < c.IWp)
        *(uint4 *) (c.xp + ((int64_t) row * c.IWp + opx) * c.ICp + 32 * bc + 8 * part) =
            make_uint4(tile[q][4 * part], tile[q][4 * part + 1], tile[q][4 * part + 2], tile[q][4 * part + 3]);
}

typedef __attribute__((address_space(3))) void conv_lds_t;
typedef __attribute__((address_space(1))) void conv_glb_t;

// FR fragments at LDS address a and two at b, of 16 rows each (1 KB apart in a
// stage), read and waited for in one block.  Written out because the
// compiler's own waits cannot tell the ring's stages apart: before an ordinary
// LDS read it drains the copies into the other stages too (4-wave form of the
// kernel below, 160 -> 160 channels at 192 x 160: 42.9 us that way, 32.4 so).
template <int FR>
__device__ __forceinline__ void conv_read(bf16x8_t (&fa)[FR], bf16x8_t (&fb)[2], uint32_t a, uint32_t b) {
#define WAMX_RD(D, A, O) "ds_read_b128 %" D ", %" A " offset:" O "\n\t"
#define WAMX_B2(D0, D1, B) WAMX_RD(D0, B, "0") WAMX_RD(D1, B, "1024")
    if constexpr (FR == 5)
        asm volatile(WAMX_B2("5", "6", "8") WAMX_B2("0", "1", "7") WAMX_RD("2", "7", "2048") WAMX_RD("3", "7", "3072")
                         WAMX_RD("4", "7", "4096") "s_waitcnt lgkmcnt(0)"
                     : "=&v"(fa[0]), "=&v"(fa[1]), "=&v"(fa[2]), "=&v"(fa[3]), "=&v"(fa[FR - 1]), "=&v"(fb[0]),
                       "=&v"(fb[1])
                     : "v"(a), "v"(b)
                     : "memory");
    else if constexpr (FR == 4)
        asm volatile(WAMX_B2("4", "5", "7") WAMX_B2("0", "1", "6") WAMX_RD("2", "6", "2048") WAMX_RD("3", "6", "3072")
                         "s_waitcnt lgkmcnt(0)"
                     : "=&v"(fa[0]), "=&v"(fa[1]), "=&v"(fa[2]), "=&v"(fa[FR - 1]), "=&v"(fb[0]), "=&v"(fb[1])
                     : "v"(a), "v"(b)
                     : "memory");
    else if constexpr (FR == 2)
        asm volatile(WAMX_B2("2", "3", "5") WAMX_B2("0", "1", "4") "s_waitcnt lgkmcnt(0)"
                     : "=&v"(fa[0]), "=&v"(fa[FR - 1]), "=&v"(fb[0]), "=&v"(fb[1])
                     : "v"(a), "v"(b)
                     : "memory");
    else
        asm volatile(WAMX_B2("1", "2", "4") WAMX_RD("0", "3", "0") "s_waitcnt lgkmcnt(0)"
                     : "=&v"(fa[0]), "=&v"(fb[0]), "=&v"(fb[1])
                     : "v"(a), "v"(b)
                     : "memory");
#undef WAMX_B2
#undef WAMX_RD
}

// 32 FR output channels by 128 pixels per workgroup of 2 x 4 waves (16 FR
// channels by 32 pixels each, MFMA 16x16x32; two waves per SIMD, so that one
// reads its fragments while the other multiplies), K steps of 32 channels of
// one tap, two between barriers, through a ring of six LDS stages.  Slot p
// of a stage row holds 16-byte chunk p ^ ((row >> 2) & 3), which keeps the
// fragment reads free of bank conflicts.  blockIdx.y: K slices, as f32
// partials.
template <int FR>
__global__ __launch_bounds__(512) void conv_gemm_kernel(ConvGemm c) {
    constexpr int BM = 32 * FR, BN = 128, ROWS = BM + BN, P = (ROWS + 127) / 128, E = ROWS * 32, S = 6;
    __shared__ __align__(16) uint16_t st[S * E];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, r16 = lane & 15, wr = wave >> 2, wc = wave & 3;
    const int nt_oc = ((int) c.OC + BM - 1) / BM;
    // Workgroups go to the 8 XCDs in turn; each takes a contiguous range of the
    // tiles (output channels first), so that the image rows that neighbouring
    // pixel tiles share are in its own L2.
    const int xcd = (int) blockIdx.x % 8, each = (int) gridDim.x / 8, more = (int) gridDim.x % 8;
    const int tile = (int) blockIdx.x / 8 + xcd * each + min(xcd, more);
    const int oc0 = tile % nt_oc * BM, p0 = tile / nt_oc * BN;
    const int cps = c.ICp / 32, ktot = c.taps * cps;
    const int kb = (int) blockIdx.y * c.ksteps, nk = min(ktot - kb, c.ksteps);

    // Copy sources: instruction i, wave and lane give a stage row; 16 rows of a
    // wave's instruction are all output channels or all pixels (BM % 16 == 0).
    // Waves whose rows of the last instruction are past the stage skip it.
    const bool skip_last = (P - 1) * 128 + wave * 16 >= ROWS;
    const char * src[P];
    bool isw[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int r = i * 128 + wave * 16 + (lane >> 2), ch = (lane & 3) ^ ((r >> 2) & 3);
        isw[i] = i * 128 + wave * 16 < BM;
        if (isw[i]) {
            src[i] = (const char *) (c.kp + ((int64_t) min(oc0 + r, (int) c.OC - 1) * ktot + kb) * 32 + 8 * ch);
        } else {
            const int p = min(p0 + r - BM, c.pix - 1), oy = p / c.OW, ox = p % c.OW;
            src[i] = (const char *) (c.xp + ((int64_t) oy * c.s1 * c.IWp + ox * c.s0) * c.ICp + 8 * ch);
        }
    }
    // The next step to copy: tap (kx, ky), channel chunk cc, weight offset, stage.
    int cc = kb % cps, kx = kb / cps % c.KW, ky = kb / cps / c.KW, issued = 0, into = 0;
    int64_t woff = 0;
    auto dma = [&]() {
        const int64_t poff = (((int64_t) ky * c.d1 * c.IWp + kx * c.d0) * c.ICp + cc * 32) * 2;
        uint16_t * stage = st + into * E;
        into = into + 1 == S ? 0 : into + 1;
#pragma unroll
        for (int i = 0; i < P; ++i)
            if (i < P - 1 || !skip_last)
                __builtin_amdgcn_global_load_lds((conv_glb_t *) (src[i] + (isw[i] ? woff : poff)),
                                                 (conv_lds_t *) (stage + (i * 128 + wave * 16) * 32), 16, 0, 0);
        if (++issued < nk) {  // past the last step it is copied again, unused
            woff += 64;
            if (++cc == cps) {
                cc = 0;
                if (++kx == c.KW) kx = 0, ++ky;
            }
        }
    };
    f32x4_t acc[FR][2];
#pragma unroll
    for (int i = 0; i < FR; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // Byte offsets of this lane's fragment chunks in a stage (rows differ from r16 by multiples of 16).
    const uint32_t slot = (r16 * 32 + (g ^ ((r16 >> 2) & 3)) * 8) * 2;
    const uint32_t base = (uint32_t) (uintptr_t) (const __attribute__((address_space(3))) void *) st + slot;
    const uint32_t aoff = 16 * FR * wr * 64, boff = (BM + 32 * wc) * 64;
    auto step = [&](uint32_t at) {
        bf16x8_t a[FR], b[2];
        conv_read<FR>(a, b, at + aoff, at + boff);
#pragma unroll
        for (int i = 0; i < FR; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < S - 2; ++i) dma();
    uint32_t cur = base;
    for (int kt = 0; kt < nk; kt += 2) {
        // Two steps per barrier.  Their copies have landed once at most the next
        // two steps' are outstanding; past the barrier the previous two stages
        // are free.
        if (skip_last) __builtin_amdgcn_s_waitcnt((2 * (P - 1) & 0xF) | (7 << 4) | (0xF << 8));
        else __builtin_amdgcn_s_waitcnt((2 * P & 0xF) | (7 << 4) | (0xF << 8));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        dma();
        dma();
        step(cur);
        if (kt + 1 < nk) step(cur + E * 2);
        cur = cur == base + (S - 2) * E * 2 ? base : cur + 2 * E * 2;
    }
    __builtin_amdgcn_s_waitcnt((7 << 4) | (0xF << 8));  // the trailing copies land before the workgroup's LDS is reused

    // Lane holds pixel r16 of a fragment, register v output channel 4 g + v.
    const bool whole = oc0 + BM <= c.OC && p0 + BN <= c.pix;
    const int pb = p0 + 32 * wc + r16, ob = oc0 + 16 * FR * wr + 4 * g;
    auto store = [&](auto all) {
#pragma unroll
        for (int i = 0; i < FR; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int64_t oc = ob + 16 * i + v, p = pb + 16 * j;
                    if (!decltype(all)::value && (oc >= c.OC || p >= c.pix)) continue;
                    if (c.part) c.part[((int64_t) blockIdx.y * c.OC + oc) * c.pix + p] = acc[i][j][v];
                    else {
                        c.y[oc * c.P + p] = f32_to_bf16(acc[i][j][v]);
                        if (c.out) c.out[oc * c.P + p] = f32_to_bf16(round_bf16(acc[i][j][v]) + bf16_to_f32(c.bias[oc]));
                    }
                }
    };
    if (whole) store(std::true_type{});
    else store(std::false_type{});
}

// Returns hipErrorNotSupported, launching nothing, when not even one output
// row's image rows fit the workspace beside the packed kernel.
static hipError_t conv_implicit(const ConvDev & d, const void * kernel, void * dst, const void * bias, void * out,
                                int64_t OC, int64_t B, void * ws, size_t ws_bytes, hipStream_t s) {
    ConvGemm c{};
    c.IW = d.IW, c.IH = d.IH, c.IC = d.IC, c.OC = OC, c.P = d.OW * d.OH;
    c.k = (const uint16_t *) kernel;
    const int64_t ICp = (d.IC + 31) / 32 * 32, IWp = d.IW + 2 * d.p0, taps = d.KW * d.KH;
    const size_t kbytes = ((size_t) (OC * taps * ICp) * 2 + 255) / 256 * 256;
    const size_t row = (size_t) (IWp * ICp) * 2, reserve = ws_bytes / 3;  // reserve: partials
    if (!ws || ((uintptr_t) ws & 15) || kbytes + reserve > ws_bytes) return hipErrorNotSupported;
    const int64_t cap = (int64_t) ((ws_bytes - reserve - kbytes) / row), reach = (d.KH - 1) * d.d1 + 1;
    if (cap < reach || d.OW * d.OH > INT32_MAX / 2 || IWp > INT32_MAX / 2 || OC * taps * ICp > INT32_MAX)
        return hipErrorNotSupported;
    const int64_t band = std::min<int64_t>(d.OH, (cap - reach) / d.s1 + 1);
    c.kp = (uint16_t *) ((char *) ws + ws_bytes / 256 * 256 - kbytes);
    c.IWp = (int) IWp, c.ICp = (int) ICp, c.OW = (int) d.OW, c.KW = (int) d.KW, c.taps = (int) taps;
    c.s0 = d.s0, c.s1 = d.s1, c.p0 = d.p0, c.p1 = d.p1, c.d0 = d.d0, c.d1 = d.d1;
    const int ktot = (int) (taps * ICp / 32);
    // Channels per workgroup: the widest of 160, 128, 64, 32 that pads least.
    int fr = 5;
    int64_t pad = (OC + 159) / 160 * 160;
    for (int f : {4, 2, 1})
        if ((OC + 32 * f - 1) / (32 * f) * (32 * f) < pad) fr = f, pad = (OC + 32 * f - 1) / (32 * f) * (32 * f);
    for (int64_t b = 0; b < B; ++b)
        for (int64_t oy = 0; oy < d.OH; oy += band) {
            const int64_t n = std::min(band, d.OH - oy);
            c.x = (const uint16_t *) d.x + b * d.IC * d.IH * d.IW;
            c.y = (uint16_t *) dst + b * OC * c.P + oy * d.OW;
            c.out = out ? (uint16_t *) out + b * OC * c.P + oy * d.OW : nullptr;
            c.bias = (const uint16_t *) bias;
            c.iy0 = (int) (oy * d.s1), c.rows = (int) ((n - 1) * d.s1 + reach), c.pix = (int) (n * d.OW);
            c.xp = (uint16_t *) ((char *) c.kp - (((size_t) c.rows * row + 255) / 256 * 256));
            const int image = (int) ((IWp + kPackPix - 1) / kPackPix * (ICp / 32) * c.rows);
            const int kblocks = b == 0 && oy == 0 ? (int) ((OC * taps * (ICp / 8) + 255) / 256) : 0;
            hipLaunchKernelGGL(conv_pack_kernel, dim3((unsigned) (image + kblocks)), dim3(256), 0, s, c, image);
            // K slices up to one workgroup per CU (the ring allows no second), of
            // 8 steps or more.  640 -> 640 channels, 3 x 3, 48 x 40 pixels in 4
            // slices 53.8 us with packing and bias, in 8 63.8.
            const int64_t tiles = (OC + 32 * fr - 1) / (32 * fr) * ((c.pix + 127) / 128);
            const size_t room = (size_t) ((char *) c.xp - (char *) ws);
            int64_t splits = std::max<int64_t>(1, std::min<int64_t>(256 / tiles, ktot / 8));
            splits = std::min<int64_t>(splits, (int64_t) (room / ((size_t) OC * c.pix * 4)));
            splits = std::max<int64_t>(splits, 1);
            c.ksteps = (int) ((ktot + splits - 1) / splits);
            splits = (ktot + c.ksteps - 1) / c.ksteps;
            c.part = splits > 1 ? (float *) ws : nullptr;
            const dim3 grid((unsigned) tiles, (unsigned) splits);
            switch (fr) {
                case 5: hipLaunchKernelGGL(conv_gemm_kernel<5>, grid, dim3(512), 0, s, c); break;
                case 4: hipLaunchKernelGGL(conv_gemm_kernel<4>, grid, dim3(512), 0, s, c); break;
                case 2: hipLaunchKernelGGL(conv_gemm_kernel<2>, grid, dim3(512), 0, s, c); break;
                default: hipLaunchKernelGGL(conv_gemm_kernel<1>, grid, dim3(512), 0, s, c); break;
            }
            if (splits > 1) {
                const hipError_t e = launch_partial_sum((const float *) ws, (int) splits, OC, c.pix, c.y,
                                                        WAMX_TYPE_BF16, c.P, s, c.bias, c.out);
                if (e != hipSuccess) return e;
            }
        }
    return hipGetLastError();
}

hipError_t launch_conv2d(const TensorRef & kernel, const TensorRef & input, const TensorRef & dst, const int32_t * pp,
                         void * ws, size_t ws_bytes, hipStream_t s, const void * bias, void * out) {
    const bool bf = kernel.type == WAMX_TYPE_BF16;
    if ((bf && (input.type != WAMX_TYPE_BF16 || dst.type != WAMX_TYPE_BF16)) ||
        (!bf && (kernel.type != WAMX_TYPE_F32 || input.type != WAMX_TYPE_F32 || dst.type != WAMX_TYPE_F32)))
        return hipErrorInvalidValue;
    ConvDev c{};
    c.x = input.data;
    c.x_type = input.type;
    c.col_type = bf ? WAMX_TYPE_BF16 : WAMX_TYPE_F32;
    c.IW = input.ne[0];
    c.IH = input.ne[1];
    c.IC = input.ne[2];
    c.KW = kernel.ne[0];
    c.KH = kernel.ne[1];
    c.OW = dst.ne[0];
    c.OH = dst.ne[1];
    c.s0 = pp[0];
    c.s1 = pp[1];
    c.p0 = pp[2];
    c.p1 = pp[3];
    c.d0 = pp[4];
    c.d1 = pp[5];
    const int64_t K = c.IC * c.KH * c.KW, P = c.OW * c.OH, OC = kernel.ne[3], B = input.ne[3];
    const size_t es = bf ? 2 : 4;
    if (OC <= 0 || B <= 0 || P <= 0) return hipSuccess;  // no output
    if (K <= 0) return hipErrorInvalidValue;
    if (bf) {
        const hipError_t e = conv_implicit(c, kernel.data, dst.data, bias, out, OC, B, ws, ws_bytes, s);
        if (e != hipErrorNotSupported) return e;
    }
    if (out) return hipErrorNotSupported;
    // f32, and images of which not one band fits the workspace: column matrix.
    // Upper workspace half: the column chunk; lower half: the GEMM's split-K partials.
    const size_t half = ws_bytes / 2 / 256 * 256;
    int64_t cap = (int64_t) (half / (K * es));
    if (cap >= 64) cap = cap / 64 * 64;
    const int64_t chunk = std::min<int64_t>(P, cap);
    if (!ws || chunk < 1) return hipErrorInvalidValue;
    c.col = (char *) ws + half;
    for (int64_t b = 0; b < B; ++b)
        for (int64_t p = 0; p < P; p += chunk) {
            const int64_t rows = std::min(chunk, P - p);
            hipLaunchKernelGGL(conv_col_kernel, dim3((unsigned) ((rows * K + 255) / 256)), dim3(256), 0, s, c, b, p,
                               rows);
            GemmArgs g;
            g.w = c.col;
            g.w_type = c.col_type;
            g.ldw = K;
            g.x = kernel.data;
            g.x_type = kernel.type;
            g.ldx = K;
            g.y = (char *) dst.data + (size_t) ((b * OC) * P + p) * es;
            g.y_type = dst.type;
            g.ldy = P;
            g.M = rows;
            g.N = OC;
            g.K = K;
            g.ws = ws;
            g.ws_bytes = half;
            const hipError_t e = launch_gemm(g, s);
            if (e != hipSuccess) return e;
        }
    return hipGetLastError();
}

}  // namespace wamx

using namespace wamx;

struct wamx_preprocessor {
    wamx_backend_t be = nullptr;
    void * buf[3] = {};
    size_t cap[3] = {};
};

extern "C" {

wamx_preprocessor_t wamx_preprocessor_create(wamx_backend_t be) {
    clear_error();
    if (!be) {
        set_error("wamx_preprocessor_create: null backend");
        return nullptr;
    }
    auto * p = new (std::nothrow) wamx_preprocessor();
    if (p) p->be = be;
    return p;
}

void wamx_preprocessor_free(wamx_preprocessor_t p) {
    if (!p) return;
    for (void * b : p->buf)
        if (b) (void) hipFree(b);
    delete p;
}

wamx_status wamx_preprocess_views(wamx_preprocessor_t p, const wamx_image_view * views, int32_t n_views, int32_t out_w,
                                  int32_t out_h, float * out_device) {
    WAMX_REQUIRE(p && views && out_device, "wamx_preprocess_views: null argument");
    WAMX_REQUIRE(n_views == 3, "wamx_preprocess_views: exactly three camera views are required (got %d)", n_views);
    WAMX_REQUIRE(out_w > 0 && out_h > 0, "wamx_preprocess_views: invalid canvas %dx%d", out_w, out_h);
    hipStream_t s = (hipStream_t) wamx_backend_stream(p->be);
    Views v{};
    for (int i = 0; i < 3; ++i) {
        const wamx_image_view & im = views[i];
        WAMX_REQUIRE(im.data && im.w > 0 && im.h > 0 && (im.format == 0 || im.format == 1),
                     "wamx_preprocess_views: invalid image %d", i);
    }
    for (int i = 0; i < 3; ++i) {
        const wamx_image_view & im = views[i];
        const size_t bytes = (size_t) im.w * im.h * 3 * (im.format == 0 ? 1 : 4);
        if (bytes > p->cap[i]) {
            if (p->buf[i]) WAMX_HIP_TRY(hipFree(p->buf[i]));
            p->buf[i] = nullptr;
            p->cap[i] = 0;
            WAMX_HIP_TRY(hipMalloc(&p->buf[i], bytes));
            p->cap[i] = bytes;
        }
        WAMX_HIP_TRY(hipMemcpyAsync(p->buf[i], im.data, bytes, hipMemcpyHostToDevice, s));
        v.v[i].data = p->buf[i];
        v.v[i].format = im.format;
        v.v[i].w = im.w;
        v.v[i].h = im.h;
    }
    const int top = out_h / 2, left = out_w / 2;
    v.v[0].dw = out_w, v.v[0].dh = top, v.v[0].x0 = 0, v.v[0].y0 = 0;
    v.v[1].dw = left, v.v[1].dh = out_h - top, v.v[1].x0 = 0, v.v[1].y0 = top;
    v.v[2].dw = out_w - left, v.v[2].dh = out_h - top, v.v[2].x0 = left, v.v[2].y0 = top;
    const int64_t n = (int64_t) 12 * (out_w / 2) * (out_h / 2);
    if (n > 0)
        hipLaunchKernelGGL(preprocess_views_kernel, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, s, v, out_w, out_h,
                       out_device);
    WAMX_HIP_TRY(hipGetLastError());
    WAMX_HIP_TRY(hipStreamSynchronize(s));
    return WAMX_STATUS_SUCCESS;
}

}  // extern "C"
