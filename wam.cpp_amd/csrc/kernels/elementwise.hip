// Strided glue kernels for the ggml ops the engine's graphs contain besides
// the fused hot path (CPY/CONT/DUP, ADD/MUL with broadcast, SCALE, unary
// GELU/GELU_ERF/SILU, CONCAT, GET_ROWS, SOFT_MAX, ROPE), the per-layer adaLN
// modulation sum, and the seeded synthetic-weight generator.
//
// Tensors are 4-D strided views (ne[], byte strides nb[]), walked in
// ne[0]-fastest order so consecutive threads touch consecutive destination
// elements.  The map kernel takes the usual forms (broadcast by whole dims, at
// most 2^31 chunks) in 8, 4 or 1 elements per thread; the one-element kernels
// with 64-bit index arithmetic take the rest.
#include "../internal.h"
#include "device.h"

#include <algorithm>

namespace wamx {

struct Ref4 {
    char * data;
    int32_t type;
    int64_t ne0, ne1, ne2, ne3;
    int64_t nb0, nb1, nb2, nb3;
};

static Ref4 to_ref4(const TensorRef & t) {
    return Ref4{(char *) t.data, t.type, t.ne[0], t.ne[1], t.ne[2], t.ne[3], t.nb[0], t.nb[1], t.nb[2], t.nb[3]};
}

__device__ __forceinline__ void unravel(int64_t i, const Ref4 & r, int64_t & i0, int64_t & i1, int64_t & i2,
                                        int64_t & i3) {
    i0 = i % r.ne0;
    i /= r.ne0;
    i1 = i % r.ne1;
    i /= r.ne1;
    i2 = i % r.ne2;
    i3 = i / r.ne2;
}

__device__ __forceinline__ char * at(const Ref4 & r, int64_t i0, int64_t i1, int64_t i2, int64_t i3) {
    return r.data + i0 * r.nb0 + i1 * r.nb1 + i2 * r.nb2 + i3 * r.nb3;
}

__device__ __forceinline__ float ld(const Ref4 & r, const char * p) {
    switch (r.type) {
        case WAMX_TYPE_F32: return *(const float *) p;
        case WAMX_TYPE_BF16: return bf16_to_f32(*(const uint16_t *) p);
        case WAMX_TYPE_I32: return (float) *(const int32_t *) p;
        default: return (float) *(const _Float16 *) p;
    }
}
__device__ __forceinline__ void st(const Ref4 & r, char * p, float v) {
    switch (r.type) {
        case WAMX_TYPE_F32: *(float *) p = v; break;
        case WAMX_TYPE_BF16: *(uint16_t *) p = f32_to_bf16(v); break;
        case WAMX_TYPE_I32: *(int32_t *) p = (int32_t) v; break;
        default: *(_Float16 *) p = (_Float16) v; break;
    }
}

// Element k of src (in its own ne0-fastest order) goes to element k of dst.
__global__ void copy_kernel(Ref4 src, Ref4 dst, int64_t n) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int64_t a0, a1, a2, a3, b0, b1, b2, b3;
    unravel(i, src, a0, a1, a2, a3);
    unravel(i, dst, b0, b1, b2, b3);
    const char * ps = at(src, a0, a1, a2, a3);
    char * pd = at(dst, b0, b1, b2, b3);
    if (src.type == dst.type) {
        if (src.type == WAMX_TYPE_F32 || src.type == WAMX_TYPE_I32) *(uint32_t *) pd = *(const uint32_t *) ps;
        else *(uint16_t *) pd = *(const uint16_t *) ps;
    } else {
        st(dst, pd, ld(src, ps));
    }
}

// ---------------------------------------------------------------------------
// Strided map: copies and casts, ADD / MUL / REPEAT, unary ops and CONCAT over
// dims merged where every operand allows it, V consecutive elements of dim 0
// per thread.  The one-element kernels spend their time on three 64-bit
// divisions per operand and element and on 2- or 4-byte accesses; here the
// index takes at most three multiplications for 8 elements.  Measured: ADD of
// a [192, 160, 160] bf16 image and a per-channel bias 31 -> 7.6 us, concatenation
// of 9.6 M bf16 along dim 1 42 -> 9.5 us (along dim 0 at odd offsets:
// concat0_kernel).
// ---------------------------------------------------------------------------
// n / d for n < 2^31 by a multiplication (Granlund and Montgomery, "Division by
// Invariant Integers using Multiplication", 1994, figure 4.1: m' = floor(2^32
// (2^l - d) / d) + 1 with l = ceil(log2 d), quotient (mulhi(m', n) + n) >> l;
// the sum stays below 2^32 for such n).
struct FastDiv {
    uint32_t d, mul, shift;
};
static FastDiv fast_div(uint32_t d) {
    uint32_t l = 0;
    while ((1ull << l) < d) ++l;
    return FastDiv{d, (uint32_t) ((((1ull << l) - d) << 32) / d + 1), l};
}
__device__ __forceinline__ uint32_t div(uint32_t n, const FastDiv & f) { return (__umulhi(f.mul, n) + n) >> f.shift; }

struct MapOperand {
    char * p;
    int64_t s0, s1, s2, s3;  // byte strides; 0: broadcast
    int32_t type;
};
struct MapArgs {
    MapOperand a, b, d;
    FastDiv n0, n1, n2;      // chunks of dim 0, elements of dims 1 and 2
    uint32_t total;          // chunks
    float scale, bias;
    int32_t uop, dim;        // unary op; concatenated dim
    uint32_t split;          // chunks (dim 0) or elements of it that come from a
};
enum { kMapCopy = 0, kMapAdd, kMapMul, kMapUnary, kMapConcat };

template <int V>
__device__ __forceinline__ void map_load(int32_t type, const char * p, int64_t s0, float (&o)[V]) {
    if (V == 1 || s0 == 0) {
        float v;
        switch (type) {
            case WAMX_TYPE_F32: v = *(const float *) p; break;
            case WAMX_TYPE_BF16: v = bf16_to_f32(*(const uint16_t *) p); break;
            case WAMX_TYPE_I32: v = (float) *(const int32_t *) p; break;
            default: v = (float) *(const _Float16 *) p; break;
        }
#pragma unroll
        for (int i = 0; i < V; ++i) o[i] = v;
        return;
    }
    if constexpr (V > 1) {
        uint32_t u[V];
        if (type == WAMX_TYPE_F32 || type == WAMX_TYPE_I32) {
#pragma unroll
            for (int i = 0; i < V / 4; ++i) *(uint4 *) &u[4 * i] = ((const uint4 *) p)[i];
#pragma unroll
            for (int i = 0; i < V; ++i) o[i] = type == WAMX_TYPE_F32 ? __uint_as_float(u[i]) : (float) (int32_t) u[i];
        } else {
            if constexpr (V == 8) *(uint4 *) u = *(const uint4 *) p;
            else *(uint2 *) u = *(const uint2 *) p;
#pragma unroll
            for (int i = 0; i < V; ++i) {
                const uint16_t h = (uint16_t) (u[i / 2] >> (16 * (i & 1)));
                o[i] = type == WAMX_TYPE_BF16 ? bf16_to_f32(h) : (float) __builtin_bit_cast(_Float16, h);
            }
        }
    }
}
template <int V>
__device__ __forceinline__ void map_store(int32_t type, char * p, const float (&o)[V]) {
    if constexpr (V == 1) {
        store_from_f32(p, type, 0, o[0]);
    } else {
        uint32_t u[V];
        if (type == WAMX_TYPE_F32 || type == WAMX_TYPE_I32) {
#pragma unroll
            for (int i = 0; i < V; ++i) u[i] = type == WAMX_TYPE_F32 ? __float_as_uint(o[i]) : (uint32_t) (int32_t) o[i];
#pragma unroll
            for (int i = 0; i < V / 4; ++i) ((uint4 *) p)[i] = *(uint4 *) &u[4 * i];
        } else {
#pragma unroll
            for (int i = 0; i < V / 2; ++i)
                u[i] = type == WAMX_TYPE_BF16
                           ? pack_bf16x2(o[2 * i], o[2 * i + 1])
                           : (uint32_t) __builtin_bit_cast(uint16_t, (_Float16) o[2 * i]) |
                                 (uint32_t) __builtin_bit_cast(uint16_t, (_Float16) o[2 * i + 1]) << 16;
            if constexpr (V == 8) *(uint4 *) p = *(uint4 *) u;
            else *(uint2 *) p = *(uint2 *) u;
        }
    }
}
// V elements of one type, bit for bit.
template <int V>
__device__ __forceinline__ void map_move(int32_t type, const char * src, char * dst) {
    const bool wide = type == WAMX_TYPE_F32 || type == WAMX_TYPE_I32;
    if constexpr (V == 1) {
        if (wide) *(uint32_t *) dst = *(const uint32_t *) src;
        else *(uint16_t *) dst = *(const uint16_t *) src;
    } else if (wide) {
#pragma unroll
        for (int i = 0; i < V / 4; ++i) ((uint4 *) dst)[i] = ((const uint4 *) src)[i];
    } else if constexpr (V == 8) {
        *(uint4 *) dst = *(const uint4 *) src;
    } else {
        *(uint2 *) dst = *(const uint2 *) src;
    }
}

template <int OP, int V>
__global__ __launch_bounds__(256) void map_kernel(MapArgs m) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= m.total) return;
    uint32_t c[4];
    const uint32_t q0 = div(i, m.n0), q1 = div(q0, m.n1), q2 = div(q1, m.n2);
    c[0] = i - q0 * m.n0.d, c[1] = q0 - q1 * m.n1.d, c[2] = q1 - q2 * m.n2.d, c[3] = q2;
    auto at = [&](const MapOperand & o) {
        return o.p + c[0] * (V * o.s0) + c[1] * o.s1 + c[2] * o.s2 + c[3] * o.s3;
    };
    char * d = at(m.d);
    if constexpr (OP == kMapConcat) {
        const uint32_t cd = m.dim == 0 ? c[0] : m.dim == 1 ? c[1] : m.dim == 2 ? c[2] : c[3];
        // b's pointer is set back by the split, so the coordinates serve both.
        map_move<V>(m.d.type, cd < m.split ? at(m.a) : at(m.b), d);
    } else if constexpr (OP == kMapCopy) {
        if (m.a.type == m.d.type && (V == 1 || m.a.s0 != 0)) {
            map_move<V>(m.d.type, at(m.a), d);
        } else {
            float x[V];
            map_load<V>(m.a.type, at(m.a), m.a.s0, x);
            map_store<V>(m.d.type, d, x);
        }
    } else {
        float x[V];
        map_load<V>(m.a.type, at(m.a), m.a.s0, x);
        if constexpr (OP == kMapUnary) {
#pragma unroll
            for (int e = 0; e < V; ++e) switch (m.uop) {
                case WAMX_UNARY_GELU: x[e] = gelu_tanh(x[e]); break;
                case WAMX_UNARY_GELU_ERF: x[e] = gelu_erf(x[e]); break;
                case WAMX_UNARY_SILU: x[e] = silu(x[e]); break;
                default: x[e] = x[e] * m.scale + m.bias; break;
            }
        } else {
            float y[V];
            map_load<V>(m.b.type, at(m.b), m.b.s0, y);
#pragma unroll
            for (int e = 0; e < V; ++e) x[e] = OP == kMapAdd ? x[e] + y[e] : x[e] * y[e];
        }
        map_store<V>(m.d.type, d, x);
    }
}

// Concatenation along dim 0 of 2-byte elements at any offset (a cache's V^T
// rows behind a state token's: odd row lengths), 8 per thread at the element's
// own alignment, which gfx950's global accesses take; the chunk that holds the
// seam or the row's end goes element by element.  One workgroup row per row.
struct __attribute__((packed, aligned(2))) loose16_t {
    uint32_t x, y, z, w;
};
__global__ __launch_bounds__(256) void concat0_kernel(Ref4 a, Ref4 b, Ref4 dst) {
    const int64_t row = blockIdx.y, i1 = row % dst.ne1, i2 = row / dst.ne1 % dst.ne2, i3 = row / (dst.ne1 * dst.ne2);
    const int64_t i0 = 8 * ((int64_t) blockIdx.x * 256 + threadIdx.x);
    if (i0 >= dst.ne0) return;
    const uint16_t * pa = (const uint16_t *) at(a, 0, i1, i2, i3);
    const uint16_t * pb = (const uint16_t *) at(b, 0, i1, i2, i3) - a.ne0;
    uint16_t * pd = (uint16_t *) at(dst, 0, i1, i2, i3);
    if (i0 + 8 <= a.ne0) {
        *(loose16_t *) (pd + i0) = *(const loose16_t *) (pa + i0);
    } else if (i0 >= a.ne0 && i0 + 8 <= dst.ne0) {
        *(loose16_t *) (pd + i0) = *(const loose16_t *) (pb + i0);
    } else {
        for (int64_t i = i0; i < min(i0 + 8, dst.ne0); ++i) pd[i] = i < a.ne0 ? pa[i] : pb[i];
    }
}

static int64_t type_bytes(int32_t type) { return type == WAMX_TYPE_F32 || type == WAMX_TYPE_I32 ? 4 : 2; }

// The operand's strides over dst's dims (0 where it has one element); false
// when a dim repeats by modulo.
static bool map_operand(const TensorRef & t, const TensorRef & dst, MapOperand & o, int64_t (&st)[4]) {
    o.p = (char *) t.data;
    o.type = t.type;
    for (int i = 0; i < 4; ++i) {
        if (t.ne[i] != dst.ne[i] && t.ne[i] != 1) return false;
        st[i] = t.ne[i] == 1 ? 0 : t.nb[i];
    }
    return true;
}

// Runs op over dst's shape; false (nothing launched) when a form is not
// covered.  concat_dim >= 0: a and b are the parts.
template <int OP>
static bool try_map(const TensorRef & a, const TensorRef * b, const TensorRef & dst, int uop, float scale, float bias,
                    int concat_dim, hipStream_t s) {
    MapArgs m{};
    int64_t st[3][4] = {}, ne[4];
    const int nop = b ? 3 : 2;
    MapOperand * op[3] = {&m.d, &m.a, &m.b};
    for (int i = 0; i < 4; ++i) ne[i] = dst.ne[i];
    m.d = MapOperand{(char *) dst.data, 0, 0, 0, 0, dst.type};
    for (int i = 0; i < 4; ++i) st[0][i] = dst.nb[i];
    int64_t split = 0;
    if (concat_dim >= 0) {
        for (int k = 1; k < 3; ++k) {
            const TensorRef & t = k == 1 ? a : *b;
            op[k]->p = (char *) t.data;
            op[k]->type = t.type;
            for (int i = 0; i < 4; ++i) st[k][i] = t.nb[i];
        }
        split = a.ne[concat_dim];
        m.b.p -= split * st[2][concat_dim];
    } else if (!map_operand(a, dst, m.a, st[1]) || (b && !map_operand(*b, dst, m.b, st[2]))) {
        return false;
    }
    // Merge dims that every operand walks as one; drop dims of one element.
    int n = 0, cd = -1;
    int64_t e[4], t[3][4];
    bool open = false;  // the last kept dim may take the next one in
    for (int i = 0; i < 4; ++i) {
        if (ne[i] == 1 && i != concat_dim) continue;
        bool join = open && i != concat_dim;
        for (int k = 0; k < nop && join; ++k) join = st[k][i] == t[k][n - 1] * e[n - 1];
        if (join) {
            e[n - 1] *= ne[i];
        } else {
            e[n] = ne[i];
            for (int k = 0; k < nop; ++k) t[k][n] = st[k][i];
            if (i == concat_dim) cd = n;
            ++n;
        }
        open = i != concat_dim;
    }
    if (n == 0) {
        e[0] = 1;
        for (int k = 0; k < nop; ++k) t[k][0] = type_bytes(op[k]->type);
        n = 1;
    }
    int64_t count = 1;
    for (int i = 0; i < n; ++i) {
        if (count > INT32_MAX / std::max<int64_t>(e[i], 1)) return false;
        count *= e[i];
    }
    // Elements per thread: whole chunks of dim 0 at aligned addresses in every
    // operand; 8 where that still gives two workgroups per CU.
    auto fits = [&](int v) {
        if (e[0] % v || (cd == 0 && split % v)) return false;
        for (int k = 0; k < nop; ++k) {
            const int64_t es = type_bytes(op[k]->type), al = std::min<int64_t>(16, v * es);
            if (t[k][0] == 0 && k > 0 && concat_dim < 0) continue;
            if (t[k][0] != es || (uintptr_t) op[k]->p % (uintptr_t) al) return false;
            for (int i = 1; i < n; ++i)
                if (t[k][i] % al) return false;
        }
        return true;
    };
    const int v = count >= 8 * 256 * 512 && fits(8) ? 8 : fits(4) ? 4 : 1;
    uint32_t d[4] = {1, 1, 1, 1};
    for (int i = 0; i < n; ++i) d[i] = (uint32_t) (i == 0 ? e[0] / v : e[i]);
    m.n0 = fast_div(d[0]), m.n1 = fast_div(d[1]), m.n2 = fast_div(d[2]);
    for (int k = 0; k < nop; ++k) {
        op[k]->s0 = t[k][0];
        op[k]->s1 = n > 1 ? t[k][1] : 0;
        op[k]->s2 = n > 2 ? t[k][2] : 0;
        op[k]->s3 = n > 3 ? t[k][3] : 0;
    }
    m.total = (uint32_t) (count / v);
    m.scale = scale, m.bias = bias, m.uop = uop, m.dim = cd;
    m.split = (uint32_t) (cd == 0 ? split / v : split);
    const dim3 grid((m.total + 255) / 256);
    if (v == 8) hipLaunchKernelGGL((map_kernel<OP, 8>), grid, dim3(256), 0, s, m);
    else if (v == 4) hipLaunchKernelGGL((map_kernel<OP, 4>), grid, dim3(256), 0, s, m);
    else hipLaunchKernelGGL((map_kernel<OP, 1>), grid, dim3(256), 0, s, m);
    return true;
}

// A copy between two same-shape views of 2-byte elements that transposes
// dims 0 and 1 in memory: dst's dim 0 and src's dim 1 are contiguous (the
// V^T store of the attention caches: token-major V -> [head][dim][token]).
// 64 x 64 tiles through LDS, so both the reads (along dim 1) and the writes
// (along dim 0) are consecutive addresses across consecutive threads.
// transpose01_kernel with 16-byte global accesses: src dim 1 and dst dim 0
// contiguous, ne1 % 8 == 0 and 16-byte aligned row strides.  The destination
// may start `mis` elements past a 16-byte boundary (a cache written from token
// 1): `dst` is then the aligned view `mis` elements earlier, and destination
// element j holds source row j - mis.  A 64 x 64 tile of the destination's
// 16-byte grid per workgroup: 512 source chunks of 8 elements are loaded (two
// per thread, both issued before the LDS stores), transposed through LDS and
// stored as 512 destination chunks; chunks that are not whole inside
// [mis, ne0 of dst) are written element by element.
__global__ __launch_bounds__(256) void transpose01_vec_kernel(Ref4 src, Ref4 dst, int mis) {
    __shared__ uint32_t tile[64][33];  // tile[r][j]: elements 2j, 2j+1 of source row b0 + r - mis
    const int64_t b0 = (int64_t) blockIdx.x * 64, b1 = (int64_t) blockIdx.y * 64;
    const int64_t i2 = blockIdx.z % src.ne2, i3 = blockIdx.z / src.ne2;
    const int t = threadIdx.x;
    uint4 v[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int q = k * 256 + t, r = q >> 3, c8 = q & 7;
        const int64_t sr = b0 + r - mis;
        const bool ok = sr >= 0 && sr < src.ne0 && b1 + 8 * c8 < src.ne1;
        v[k] = ok ? *(const uint4 *) at(src, sr, b1 + 8 * c8, i2, i3) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int q = k * 256 + t, r = q >> 3, c8 = q & 7;
        tile[r][4 * c8] = v[k].x;
        tile[r][4 * c8 + 1] = v[k].y;
        tile[r][4 * c8 + 2] = v[k].z;
        tile[r][4 * c8 + 3] = v[k].w;
    }
    __syncthreads();
    const uint16_t * tl = (const uint16_t *) &tile[0][0];  // element (r, c) at r * 66 + c
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int q = k * 256 + t, d = q >> 3, c8 = q & 7;  // destination row b1 + d, elements b0 + 8 c8 ..
        if (b1 + d >= dst.ne1) continue;
        uint16_t e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = tl[(8 * c8 + i) * 66 + d];
        const int64_t j0 = b0 + 8 * c8;
        if (j0 >= mis && j0 + 8 <= dst.ne0) {
            *(uint4 *) at(dst, j0, b1 + d, i2, i3) =
                make_uint4(e[0] | (uint32_t) e[1] << 16, e[2] | (uint32_t) e[3] << 16, e[4] | (uint32_t) e[5] << 16,
                           e[6] | (uint32_t) e[7] << 16);
        } else {
            for (int i = 0; i < 8; ++i)
                if (j0 + i >= mis && j0 + i < dst.ne0) *(uint16_t *) at(dst, j0 + i, b1 + d, i2, i3) = e[i];
        }
    }
}

__global__ __launch_bounds__(256) void transpose01_kernel(Ref4 src, Ref4 dst) {
    __shared__ uint16_t tile[64][66];
    const int64_t b0 = (int64_t) blockIdx.x * 64, b1 = (int64_t) blockIdx.y * 64;
    const int64_t i2 = blockIdx.z % src.ne2, i3 = blockIdx.z / src.ne2;
    const int t = threadIdx.x;
#pragma unroll 4
    for (int k = 0; k < 16; ++k) {
        const int idx = k * 256 + t, r = idx >> 6, c = idx & 63;  // r: dim 0, c: dim 1
        if (b0 + r < src.ne0 && b1 + c < src.ne1) tile[r][c] = *(const uint16_t *) at(src, b0 + r, b1 + c, i2, i3);
    }
    __syncthreads();
#pragma unroll 4
    for (int k = 0; k < 16; ++k) {
        const int idx = k * 256 + t, r = idx >> 6, c = idx & 63;  // r: dim 1, c: dim 0
        if (b0 + c < dst.ne0 && b1 + r < dst.ne1) *(uint16_t *) at(dst, b0 + c, b1 + r, i2, i3) = tile[c][r];
    }
}

__global__ void binary_kernel(int op, Ref4 a, Ref4 b, Ref4 dst, int64_t n) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int64_t i0, i1, i2, i3;
    unravel(i, dst, i0, i1, i2, i3);
    const float y = ld(b, at(b, i0 % b.ne0, i1 % b.ne1, i2 % b.ne2, i3 % b.ne3));
    if (op == 2) {  // REPEAT: dst = b broadcast
        st(dst, at(dst, i0, i1, i2, i3), y);
        return;
    }
    const float x = ld(a, at(a, i0, i1, i2, i3));
    st(dst, at(dst, i0, i1, i2, i3), op == 0 ? x + y : x * y);
}

__global__ void unary_kernel(int op, Ref4 a, Ref4 dst, float scale, float bias, int64_t n) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int64_t i0, i1, i2, i3;
    unravel(i, dst, i0, i1, i2, i3);
    const float x = ld(a, at(a, i0, i1, i2, i3));
    float y;
    switch (op) {
        case WAMX_UNARY_GELU: y = gelu_tanh(x); break;
        case WAMX_UNARY_GELU_ERF: y = gelu_erf(x); break;
        case WAMX_UNARY_SILU: y = silu(x); break;
        default: y = x * scale + bias; break;
    }
    st(dst, at(dst, i0, i1, i2, i3), y);
}

__global__ void concat_kernel(Ref4 a, Ref4 b, Ref4 dst, int dim, int64_t n) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int64_t c[4];
    unravel(i, dst, c[0], c[1], c[2], c[3]);
    const int64_t ane[4] = {a.ne0, a.ne1, a.ne2, a.ne3};
    const char * src;
    if (c[dim] < ane[dim]) {
        src = at(a, c[0], c[1], c[2], c[3]);
    } else {
        c[dim] -= ane[dim];
        src = at(b, c[0], c[1], c[2], c[3]);
        c[dim] += ane[dim];
    }
    char * d = at(dst, c[0], c[1], c[2], c[3]);
    if (dst.type == WAMX_TYPE_F32 || dst.type == WAMX_TYPE_I32) *(uint32_t *) d = *(const uint32_t *) src;
    else *(uint16_t *) d = *(const uint16_t *) src;
}

// dst[i0, i1, i2] = a[i0, rows[i1, i2], i2 % a.ne2]
__global__ void get_rows_kernel(Ref4 a, const int32_t * rows, int64_t rows_ld, Ref4 dst, int64_t n) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int64_t i0, i1, i2, i3;
    if (n <= INT32_MAX) {  // 32-bit divisions
        const uint32_t n0 = (uint32_t) dst.ne0, n1 = (uint32_t) dst.ne1, n2 = (uint32_t) dst.ne2;
        const uint32_t q0 = (uint32_t) i / n0, q1 = q0 / n1, q2 = q1 / n2;
        i0 = (uint32_t) i - q0 * n0, i1 = q0 - q1 * n1, i2 = q1 - q2 * n2, i3 = q2;
    } else {
        unravel(i, dst, i0, i1, i2, i3);
    }
    const int64_t r = rows[i1 + i2 * rows_ld];
    st(dst, at(dst, i0, i1, i2, i3), ld(a, at(a, i0, r, i2 % a.ne2, i3 % a.ne3)));
}

// SOFT_MAX_EXT: y = exp(w - max) / sum over ne0 with w = scale * x + mask
// (mask row i1 of plane (i2 % ne2, i3 % ne3); no mask when m.data is null).
// One workgroup of W waves per row.  PER > 0: the row's values stay in
// registers (PER per thread), so it is read and written once; 0: any length.
// W = 1 for rows of at most 64, where three of four waves would hold nothing.
template <int PER, int W>
__global__ __launch_bounds__(64 * W) void softmax_kernel(Ref4 x, Ref4 m, Ref4 y, float scale) {
    __shared__ float red[4];
    constexpr int T = 64 * W;
    const int64_t row = blockIdx.x;
    const int64_t r1 = row % x.ne1, r2 = (row / x.ne1) % x.ne2, r3 = row / (x.ne1 * x.ne2);
    const char * xr = at(x, 0, r1, r2, r3);
    const char * mr = m.data ? at(m, 0, r1, r2 % m.ne2, r3 % m.ne3) : nullptr;
    char * yr = at(y, 0, r1, r2, r3);
    auto w_at = [&](int64_t c) {
        const float v = *(const float *) (xr + c * x.nb0) * scale;
        return mr ? v + ld(m, mr + c * m.nb0) : v;
    };
    constexpr int R = PER > 0 ? PER : 1;
    float v[R];
    float mx = -INFINITY;
    if constexpr (PER > 0) {
#pragma unroll
        for (int i = 0; i < R; ++i) v[i] = w_at(min((int64_t) threadIdx.x + i * T, x.ne0 - 1));
#pragma unroll
        for (int i = 0; i < R; ++i)
            if ((int64_t) threadIdx.x + i * T < x.ne0) mx = fmaxf(mx, v[i]);
    } else {
        for (int64_t c = threadIdx.x; c < x.ne0; c += T) mx = fmaxf(mx, w_at(c));
    }
    mx = wave_max(mx);
    if constexpr (W > 1) {
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
        __syncthreads();
        mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    }
    float sum = 0.0f;
    if constexpr (PER > 0) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            v[i] = expf(v[i] - mx);
            if ((int64_t) threadIdx.x + i * T < x.ne0) sum += v[i];
        }
    } else {
        for (int64_t c = threadIdx.x; c < x.ne0; c += T) {
            const float e = expf(w_at(c) - mx);
            *(float *) (yr + c * y.nb0) = e;
            sum += e;
        }
    }
    sum = W > 1 ? block_sum(sum, red) : wave_sum(sum);
    const float inv = 1.0f / sum;
    if constexpr (PER > 0) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int64_t c = (int64_t) threadIdx.x + i * T;
            if (c < x.ne0) *(float *) (yr + c * y.nb0) = v[i] * inv;
        }
    } else {
        for (int64_t c = threadIdx.x; c < x.ne0; c += T) *(float *) (yr + c * y.nb0) *= inv;
    }
}

// ROPE mode NORMAL on [head_dim, heads, tokens(, ne3)]: pairs (2i, 2i+1) for
// 2i < n_dims rotate by pos[token] * theta_scale^i; the rest is copied.
__global__ void rope_kernel(Ref4 x, const int32_t * pos, Ref4 y, int n_dims, float theta_scale, int64_t npairs) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npairs) return;
    const int64_t half = (x.ne0 + 1) / 2;
    int64_t ip, i1, i2, i3;
    if (npairs <= INT32_MAX) {  // 32-bit divisions
        const uint32_t h = (uint32_t) half, n1 = (uint32_t) x.ne1, n2 = (uint32_t) x.ne2;
        const uint32_t q0 = (uint32_t) i / h, q1 = q0 / n1, q2 = q1 / n2;
        ip = (uint32_t) i - q0 * h, i1 = q0 - q1 * n1, i2 = q1 - q2 * n2, i3 = q2;
    } else {
        ip = i % half;
        int64_t rest = i / half;
        i1 = rest % x.ne1;
        rest /= x.ne1;
        i2 = rest % x.ne2, i3 = rest / x.ne2;
    }
    const int64_t e = 2 * ip;
    const char * px = at(x, e, i1, i2, i3);
    char * py = at(y, e, i1, i2, i3);
    const float a = *(const float *) px;
    if (e + 1 >= x.ne0) {
        *(float *) py = a;
        return;
    }
    const float b = *(const float *) (px + x.nb0);
    if (e < n_dims) {
        const float theta = (float) pos[i2] * powf(theta_scale, (float) ip);
        float sn, cs;
        sincosf(theta, &sn, &cs);
        *(float *) py = a * cs - b * sn;
        *(float *) (py + y.nb0) = a * sn + b * cs;
    } else {
        *(float *) py = a;
        *(float *) (py + y.nb0) = b;
    }
}

// ggml_im2col, 2-D: dst[n][oh][ow][ic*KH*KW + kh*KW + kw] =
// src[n][ic][oh*s1 + kh*d1 - p1][ow*s0 + kw*d0 - p0] (zero outside).
__global__ void im2col_kernel(Ref4 src, Ref4 dst, int KW, int KH, int s0, int s1, int p0, int p1, int d0, int d1,
                              int64_t n) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int64_t c, ow, oh, b;
    unravel(i, dst, c, ow, oh, b);
    const int64_t kw = c % KW, kh = (c / KW) % KH, ic = c / (KW * KH);
    const int64_t iw = ow * s0 + kw * d0 - p0, ih = oh * s1 + kh * d1 - p1;
    float v = 0.0f;
    if (iw >= 0 && iw < src.ne0 && ih >= 0 && ih < src.ne1) v = ld(src, at(src, iw, ih, ic, b));
    st(dst, at(dst, c, ow, oh, b), v);
}

// out[l][j] = f32(mod[j]) + f32(tables[l][j])  (modulation_add, mot.cpp:137-145).
// out[s][r] = f32(mod[s][r % per_layer]) + f32(tables[r]) for the S columns
// (timesteps) of mod, r over the per_step = per_layer * layers table values.
__global__ void modulation_kernel(const void * mod, int32_t mod_type, const void * tables, int32_t tab_type, float * out,
                                  int64_t per_layer, int64_t per_step, int64_t n) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t st = i / per_step, r = i - st * per_step, j = r % per_layer;
    out[i] = load_as_f32(mod, mod_type, st * per_layer + j) + load_as_f32(tables, tab_type, r);
}

// scheduler_step (weights.cpp:885-902): bf16(f32(a) + f32(v) * dt), the
// product and the sum rounded separately as the MUL and ADD nodes do.
#pragma clang fp contract(off)
__global__ void euler_step_kernel(const uint16_t * __restrict__ a, const uint16_t * __restrict__ v,
                                  const float * __restrict__ dt, uint16_t * __restrict__ out, int64_t n) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float t = bf16_to_f32(v[i]) * dt[0];
    out[i] = f32_to_bf16(bf16_to_f32(a[i]) + t);
}
#pragma clang fp contract(on)

// Two small linear layers (widths <= kMlpMax) for 16 tokens per workgroup:
// the tokens' inputs transposed into LDS as f32 [k][16], one layer's weight
// staged as bf16 [m][k] (rows padded by one element); thread t owns feature
// t % 128 for tokens 8 (t / 128) .. +8 and accumulates in k order in f32.
// Each layer: bf16(bf16(acc) + bias), then GELU_ERF rounded to bf16 where
// its flag is set; layer 1's output is layer 2's input in LDS.
constexpr int kMlpMax = 128, kMlpTok = 16;
__global__ __launch_bounds__(256) void mlp_small_kernel(const uint16_t * __restrict__ x, const uint16_t * __restrict__ w1,
                                                        const uint16_t * __restrict__ b1,
                                                        const uint16_t * __restrict__ w2,
                                                        const uint16_t * __restrict__ b2, uint16_t * __restrict__ y,
                                                        int64_t N, int K0, int M1, int M2, int flags) {
    __shared__ __align__(16) float xt[kMlpMax][kMlpTok];
    __shared__ __align__(16) float ht[kMlpMax][kMlpTok];
    __shared__ uint16_t ws[kMlpMax * (kMlpMax + 1)];
    const int tid = threadIdx.x;
    const int64_t n0 = (int64_t) blockIdx.x * kMlpTok;
    for (int e = tid; e < kMlpTok * K0; e += 256) {
        const int n = e / K0, k = e % K0;
        float v = n0 + n < N ? bf16_to_f32(x[(n0 + n) * K0 + k]) : 0.0f;
        if (flags & WAMX_MLP_GELU_IN) v = round_bf16(gelu_erf(v));
        xt[k][n] = v;
    }
    const int m = tid % kMlpMax, g = tid / kMlpMax;  // feature, token group of 8
    auto layer = [&](const uint16_t * __restrict__ w, const uint16_t * __restrict__ b, int K, int M, bool gelu,
                     float (*in)[kMlpTok], float (*out)[kMlpTok], bool last) {
        const int pitch = K + 1;
        __syncthreads();  // the previous layer is done with the weight tile and has written `in`
        for (int e = tid; e < M * K; e += 256) ws[(e / K) * pitch + e % K] = w[e];
        __syncthreads();
        if (m >= M) return;
        float acc[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
        for (int k = 0; k < K; ++k) {
            const float wv = bf16_to_f32(ws[m * pitch + k]);
            const float4 xa = *(const float4 *) &in[k][8 * g], xb = *(const float4 *) &in[k][8 * g + 4];
            acc[0] = fmaf(wv, xa.x, acc[0]);
            acc[1] = fmaf(wv, xa.y, acc[1]);
            acc[2] = fmaf(wv, xa.z, acc[2]);
            acc[3] = fmaf(wv, xa.w, acc[3]);
            acc[4] = fmaf(wv, xb.x, acc[4]);
            acc[5] = fmaf(wv, xb.y, acc[5]);
            acc[6] = fmaf(wv, xb.z, acc[6]);
            acc[7] = fmaf(wv, xb.w, acc[7]);
        }
        const float bias = bf16_to_f32(b[m]);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float v = round_bf16(round_bf16(acc[j]) + bias);
            if (gelu) v = round_bf16(gelu_erf(v));
            const int64_t n = n0 + 8 * g + j;
            if (last) {
                if (n < N) y[n * M + m] = f32_to_bf16(v);
            } else {
                out[m][8 * g + j] = v;
            }
        }
    };
    layer(w1, b1, K0, M1, flags & WAMX_MLP_GELU_MID, xt, ht, false);
    layer(w2, b2, M1, M2, flags & WAMX_MLP_GELU_OUT, ht, nullptr, true);
}

// mlp_small_kernel's arithmetic (each output an f32 FMA chain over k in
// ascending order, then the same roundings, so the same bits) spread over
// more CUs: kMlpRegTok tokens per workgroup, thread t owning feature t % 128
// for tokens 2 (t / 128) .. +2.  The FMAs are VALU work (16 tokens x 128 x
// 128 per layer is 8k cycles of one CU), so the 16-token workgroups of
// mlp_small_kernel ran 19-21 us on 3 CUs.  Each thread's weight rows of both
// layers are loaded into registers up front as 16-byte chunks and the k loop
// is unrolled over them, so the only LDS traffic is the broadcast activation
// reads.  K0, M1 and M2 multiples of 8, weights 16-byte aligned.
constexpr int kMlpChunks = kMlpMax / 8, kMlpRegTok = 4, kMlpTpt = kMlpRegTok / 2;
__device__ __forceinline__ void mlp_row_load(const uint16_t * __restrict__ w, int K, int m, int M, uint4 (&r)[kMlpChunks]) {
#pragma unroll
    for (int c = 0; c < kMlpChunks; ++c)
        r[c] = (m < M && 8 * c < K) ? *(const uint4 *) (w + (int64_t) m * K + 8 * c) : make_uint4(0, 0, 0, 0);
}
__device__ __forceinline__ void mlp_row_dot(const uint4 (&r)[kMlpChunks], int K, const float (*in)[kMlpRegTok], int g,
                                            float (&acc)[kMlpTpt]) {
#pragma unroll
    for (int c = 0; c < kMlpChunks; ++c) {
        if (8 * c >= K) break;
        const uint32_t wp[4] = {r[c].x, r[c].y, r[c].z, r[c].w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float wv = __uint_as_float(e & 1 ? wp[e >> 1] & 0xffff0000u : wp[e >> 1] << 16);
            const float2 xv = *(const float2 *) &in[8 * c + e][kMlpTpt * g];
            acc[0] = fmaf(wv, xv.x, acc[0]);
            acc[1] = fmaf(wv, xv.y, acc[1]);
        }
    }
}
__global__ __launch_bounds__(256) void mlp_small_reg_kernel(const uint16_t * __restrict__ x,
                                                            const uint16_t * __restrict__ w1,
                                                            const uint16_t * __restrict__ b1,
                                                            const uint16_t * __restrict__ w2,
                                                            const uint16_t * __restrict__ b2, uint16_t * __restrict__ y,
                                                            int64_t N, int K0, int M1, int M2, int flags) {
    static_assert(kMlpTpt == 2, "two tokens per thread");
    __shared__ __align__(16) float xt[kMlpMax][kMlpRegTok];
    __shared__ __align__(16) float ht[kMlpMax][kMlpRegTok];
    const int tid = threadIdx.x;
    const int m = tid % kMlpMax, g = tid / kMlpMax;  // feature, token pair
    const int64_t n0 = (int64_t) blockIdx.x * kMlpRegTok;
    uint4 r1[kMlpChunks], r2[kMlpChunks];
    mlp_row_load(w1, K0, m, M1, r1);
    mlp_row_load(w2, M1, m, M2, r2);
    const float bias1 = m < M1 ? bf16_to_f32(b1[m]) : 0.0f, bias2 = m < M2 ? bf16_to_f32(b2[m]) : 0.0f;
    for (int e = tid; e < kMlpRegTok * K0; e += 256) {
        const int n = e / K0, k = e % K0;
        float v = n0 + n < N ? bf16_to_f32(x[(n0 + n) * K0 + k]) : 0.0f;
        if (flags & WAMX_MLP_GELU_IN) v = round_bf16(gelu_erf(v));
        xt[k][n] = v;
    }
    __syncthreads();
    float acc[kMlpTpt];
    if (m < M1) {
        acc[0] = acc[1] = 0.0f;
        mlp_row_dot(r1, K0, xt, g, acc);
#pragma unroll
        for (int j = 0; j < kMlpTpt; ++j) {
            float v = round_bf16(round_bf16(acc[j]) + bias1);
            if (flags & WAMX_MLP_GELU_MID) v = round_bf16(gelu_erf(v));
            ht[m][kMlpTpt * g + j] = v;
        }
    }
    __syncthreads();
    if (m >= M2) return;
    acc[0] = acc[1] = 0.0f;
    mlp_row_dot(r2, M1, ht, g, acc);
#pragma unroll
    for (int j = 0; j < kMlpTpt; ++j) {
        float v = round_bf16(round_bf16(acc[j]) + bias2);
        if (flags & WAMX_MLP_GELU_OUT) v = round_bf16(gelu_erf(v));
        const int64_t n = n0 + kMlpTpt * g + j;
        if (n < N) y[n * M2 + m] = f32_to_bf16(v);
    }
}

// splitmix64 (Steele, Lea, Flood: "Fast splittable pseudorandom number
// generators", OOPSLA 2014) on seed + (i+1)*golden gamma, then Box-Muller
// with two 24-bit uniforms in (0, 1).
__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ void fill_normal_kernel(void * dst, int32_t type, int64_t n, uint64_t seed, float mean, float stdv) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t z = splitmix64(seed + (uint64_t) (i + 1) * 0x9E3779B97F4A7C15ull);
    const float u1 = ((float) (z >> 40) + 0.5f) * (1.0f / 16777216.0f);
    const float u2 = ((float) ((z >> 16) & 0xFFFFFFull) + 0.5f) * (1.0f / 16777216.0f);
    const float r = sqrtf(-2.0f * logf(u1));
    const float v = mean + stdv * r * cosf(6.283185307179586f * u2);
    if (type == WAMX_TYPE_F32) ((float *) dst)[i] = v;
    else ((uint16_t *) dst)[i] = f32_to_bf16(v);
}

__global__ void fill_f32_kernel(float * dst, int64_t n, float v) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = v;
}

// ---------------------------------------------------------------------------
static int64_t nel(const TensorRef & t) { return t.ne[0] * t.ne[1] * t.ne[2] * t.ne[3]; }
static dim3 grid1d(int64_t n) { return dim3((unsigned) ((n + 255) / 256)); }

static bool dense(const TensorRef & t) {
    int64_t b = type_bytes(t.type);
    for (int i = 0; i < 4; ++i) {
        if (t.ne[i] != 1 && t.nb[i] != b) return false;
        b *= t.ne[i];
    }
    return true;
}

hipError_t launch_copy(const TensorRef & src, const TensorRef & dst, hipStream_t s) {
    const int64_t n = nel(dst);
    if (n <= 0) return hipSuccess;
    if (nel(src) != n) return hipErrorInvalidValue;
    const bool two_byte = src.type == dst.type && (src.type == WAMX_TYPE_BF16 || src.type == WAMX_TYPE_F16);
    const bool same_shape =
        src.ne[0] == dst.ne[0] && src.ne[1] == dst.ne[1] && src.ne[2] == dst.ne[2] && src.ne[3] == dst.ne[3];
    if (two_byte && same_shape && dst.nb[0] == 2 && src.nb[1] == 2 && src.nb[0] != 2 && src.ne[0] >= 64 &&
        src.ne[1] >= 16) {
        const dim3 grid((unsigned) ((src.ne[0] + 63) / 64), (unsigned) ((src.ne[1] + 63) / 64),
                        (unsigned) (src.ne[2] * src.ne[3]));
        auto a16 = [](const void * p, int64_t a, int64_t b, int64_t c) {
            return (((uintptr_t) p | (uintptr_t) a | (uintptr_t) b | (uintptr_t) c) & 15) == 0;
        };
        const int mis = (int) (((uintptr_t) dst.data & 15) / 2);  // elements past the 16-byte boundary
        if (src.ne[1] % 8 == 0 && ((uintptr_t) dst.data & 1) == 0 && a16(src.data, src.nb[0], src.nb[2], src.nb[3]) &&
            a16(nullptr, dst.nb[1], dst.nb[2], dst.nb[3])) {
            Ref4 dv = to_ref4(dst);
            dv.data -= 2 * mis;
            dv.ne0 += mis;
            const dim3 vgrid((unsigned) ((dv.ne0 + 63) / 64), grid.y, grid.z);
            hipLaunchKernelGGL(transpose01_vec_kernel, vgrid, dim3(256), 0, s, to_ref4(src), dv, mis);
        } else
            hipLaunchKernelGGL(transpose01_kernel, grid, dim3(256), 0, s, to_ref4(src), to_ref4(dst));
        return hipGetLastError();
    }
    if (same_shape && try_map<kMapCopy>(src, nullptr, dst, 0, 0, 0, -1, s)) return hipGetLastError();
    if (!same_shape && dense(src) && dense(dst)) {  // a reshape: both in memory order
        TensorRef f = src, d = dst;
        for (TensorRef * t : {&f, &d}) {
            t->nb[0] = type_bytes(t->type);  // a first dim of one element may have any stride
            t->ne[0] = n;
            t->ne[1] = t->ne[2] = t->ne[3] = 1;
        }
        if (try_map<kMapCopy>(f, nullptr, d, 0, 0, 0, -1, s)) return hipGetLastError();
    }
    hipLaunchKernelGGL(copy_kernel, grid1d(n), dim3(256), 0, s, to_ref4(src), to_ref4(dst), n);
    return hipGetLastError();
}

hipError_t launch_binary(int op, const TensorRef & a, const TensorRef & b, const TensorRef & dst, hipStream_t s) {
    const int64_t n = nel(dst);
    if (n <= 0) return hipSuccess;
    if (op == 0 ? try_map<kMapAdd>(a, &b, dst, 0, 0, 0, -1, s)
        : op == 1 ? try_map<kMapMul>(a, &b, dst, 0, 0, 0, -1, s)
                  : try_map<kMapCopy>(b, nullptr, dst, 0, 0, 0, -1, s))
        return hipGetLastError();
    hipLaunchKernelGGL(binary_kernel, grid1d(n), dim3(256), 0, s, op, to_ref4(a), to_ref4(b), to_ref4(dst), n);
    return hipGetLastError();
}

hipError_t launch_unary(int op, const TensorRef & a, const TensorRef & dst, float scale, float bias, hipStream_t s) {
    const int64_t n = nel(dst);
    if (n <= 0) return hipSuccess;
    if (try_map<kMapUnary>(a, nullptr, dst, op, scale, bias, -1, s)) return hipGetLastError();
    hipLaunchKernelGGL(unary_kernel, grid1d(n), dim3(256), 0, s, op, to_ref4(a), to_ref4(dst), scale, bias, n);
    return hipGetLastError();
}

hipError_t launch_concat(const TensorRef & a, const TensorRef & b, const TensorRef & dst, int dim, hipStream_t s) {
    const int64_t n = nel(dst);
    if (n <= 0) return hipSuccess;
    const int64_t rows = dst.ne[1] * dst.ne[2] * dst.ne[3];
    if (dim == 0 && dst.type != WAMX_TYPE_F32 && dst.type != WAMX_TYPE_I32 && a.nb[0] == 2 && b.nb[0] == 2 &&
        dst.nb[0] == 2 && dst.ne[0] >= 512 && rows <= 65535 && (a.ne[0] % 8 || dst.ne[0] % 8)) {
        // 9.6 M elements in rows of 3121: 26 us one element per thread, 15.3 so.
        hipLaunchKernelGGL(concat0_kernel, dim3((unsigned) ((dst.ne[0] + 2047) / 2048), (unsigned) rows), dim3(256), 0,
                           s, to_ref4(a), to_ref4(b), to_ref4(dst));
        return hipGetLastError();
    }
    if (try_map<kMapConcat>(a, &b, dst, 0, 0, 0, dim, s)) return hipGetLastError();
    hipLaunchKernelGGL(concat_kernel, grid1d(n), dim3(256), 0, s, to_ref4(a), to_ref4(b), to_ref4(dst), dim, n);
    return hipGetLastError();
}

hipError_t launch_get_rows(const TensorRef & a, const int32_t * rows, const TensorRef & dst, hipStream_t s) {
    const int64_t n = nel(dst);
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(get_rows_kernel, grid1d(n), dim3(256), 0, s, to_ref4(a), rows, dst.ne[1], to_ref4(dst), n);
    return hipGetLastError();
}

hipError_t launch_softmax_f32(const TensorRef & x, const TensorRef & mask, const TensorRef & y, float scale,
                              hipStream_t s) {
    const int64_t rows = x.ne[1] * x.ne[2] * x.ne[3];
    if (rows <= 0 || x.ne[0] <= 0) return hipSuccess;  // the kernel loads a row's last element for lanes past it
#define WAMX_SOFTMAX(PER, W)                                                                                       \
    hipLaunchKernelGGL((softmax_kernel<PER, W>), dim3((unsigned) rows), dim3(64 * W), 0, s, to_ref4(x), to_ref4(mask), \
                       to_ref4(y), scale)
    if (x.ne[0] <= 64) WAMX_SOFTMAX(1, 1);
    else if (x.ne[0] <= 512) WAMX_SOFTMAX(2, 4);
    else if (x.ne[0] <= 2048) WAMX_SOFTMAX(8, 4);
    else if (x.ne[0] <= 4096) WAMX_SOFTMAX(16, 4);
    else WAMX_SOFTMAX(0, 4);
#undef WAMX_SOFTMAX
    return hipGetLastError();
}

hipError_t launch_rope_f32(const TensorRef & x, const int32_t * pos, const TensorRef & y, int n_dims, float freq_base,
                           hipStream_t s) {
    const int64_t npairs = (x.ne[0] + 1) / 2 * x.ne[1] * x.ne[2] * x.ne[3];
    if (npairs <= 0) return hipSuccess;
    const float theta_scale = powf(freq_base, -2.0f / (float) n_dims);
    hipLaunchKernelGGL(rope_kernel, grid1d(npairs), dim3(256), 0, s, to_ref4(x), pos, to_ref4(y), n_dims, theta_scale,
                       npairs);
    return hipGetLastError();
}

hipError_t launch_im2col(const TensorRef & src, const TensorRef & dst, int KW, int KH, int s0, int s1, int p0, int p1,
                         int d0, int d1, hipStream_t s) {
    const int64_t n = nel(dst);
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(im2col_kernel, grid1d(n), dim3(256), 0, s, to_ref4(src), to_ref4(dst), KW, KH, s0, s1, p0, p1,
                       d0, d1, n);
    return hipGetLastError();
}

hipError_t launch_modulation(const void * mod, int32_t mod_type, const void * tables, int32_t tab_type, float * out,
                             int64_t per_layer, int64_t layers, hipStream_t s, int64_t steps) {
    const int64_t per_step = per_layer * layers, n = per_step * steps;
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(modulation_kernel, grid1d(n), dim3(256), 0, s, mod, mod_type, tables, tab_type, out, per_layer,
                       per_step, n);
    return hipGetLastError();
}

// Smallest index of an Inf or NaN of p[0, n) into *first (left as is when
// there is none; the caller starts it at UINT32_MAX).
__global__ void nonfinite_scan_kernel(const float * __restrict__ p, int64_t n, uint32_t * first) {
    for (int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t) gridDim.x * blockDim.x) {
        uint32_t u;
        memcpy(&u, p + i, sizeof u);
        if ((u & 0x7f800000u) == 0x7f800000u) atomicMin(first, (uint32_t) i);
    }
}

hipError_t launch_nonfinite_scan(const float * p, int64_t n, uint32_t * first, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (n >= (int64_t) UINT32_MAX) return hipErrorInvalidValue;
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, 2048);
    hipLaunchKernelGGL(nonfinite_scan_kernel, dim3((unsigned) blocks), dim3(256), 0, s, p, n, first);
    return hipGetLastError();
}

hipError_t launch_euler_step(const void * a, const void * v, const float * dt, void * out, int64_t n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(euler_step_kernel, grid1d(n), dim3(256), 0, s, (const uint16_t *) a, (const uint16_t *) v, dt,
                       (uint16_t *) out, n);
    return hipGetLastError();
}

hipError_t launch_mlp_small(const void * x, const void * w1, const void * b1, const void * w2, const void * b2, void * y,
                            int64_t N, int64_t K0, int64_t M1, int64_t M2, int32_t flags, hipStream_t s) {
    if (N <= 0) return hipSuccess;
    if (K0 < 1 || M1 < 1 || M2 < 1 || K0 > kMlpMax || M1 > kMlpMax || M2 > kMlpMax) return hipErrorInvalidValue;
    const bool reg = K0 % 8 == 0 && M1 % 8 == 0 && M2 % 8 == 0 && (((uintptr_t) w1 | (uintptr_t) w2) & 15) == 0;
    const int tok = reg ? kMlpRegTok : kMlpTok;
    hipLaunchKernelGGL(reg ? mlp_small_reg_kernel : mlp_small_kernel, dim3((unsigned) ((N + tok - 1) / tok)), dim3(256), 0, s,
                       (const uint16_t *) x, (const uint16_t *) w1, (const uint16_t *) b1, (const uint16_t *) w2,
                       (const uint16_t *) b2, (uint16_t *) y, N, (int) K0, (int) M1, (int) M2, (int) flags);
    return hipGetLastError();
}

hipError_t launch_fill_normal(void * dst, int32_t type, int64_t n, uint64_t seed, float mean, float stdv, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (type != WAMX_TYPE_F32 && type != WAMX_TYPE_BF16) return hipErrorInvalidValue;
    hipLaunchKernelGGL(fill_normal_kernel, grid1d(n), dim3(256), 0, s, dst, type, n, seed, mean, stdv);
    return hipGetLastError();
}

hipError_t launch_fill_f32(float * dst, int64_t n, float v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(fill_f32_kernel, grid1d(n), dim3(256), 0, s, dst, n, v);
    return hipGetLastError();
}

TensorRef ref_of(const wamx_tensor * t) {
    TensorRef r;
    r.data = t->data;
    r.type = t->type;
    for (int i = 0; i < 4; ++i) {
        r.ne[i] = t->ne[i];
        r.nb[i] = (int64_t) t->nb[i];
    }
    return r;
}

}  // namespace wamx
