// Eager elementwise kernels for gfx950: broadcast binary ops, tensor-scalar
// ops, unary math, dtype casts / strided packs, where-select and fills.
//
// The host collapses the output shape first (adjacent dimensions merge
// when every operand's strides allow it; size-1 dimensions drop), so most
// broadcasts reach the kernels as 1-2 dimensions.  Floating operands of one
// 32- or 16-bit dtype in such layouts take the vector path (16-byte loads and
// stores); every other layout and dtype mix runs the generic path, which
// decodes the collapsed index and converts through the compute type.
//
// Op semantics follow the reference functors (cuda_op_functors.cuh:12-449):
// operands are converted to the output dtype (float for f16/bf16 outputs),
// integer division by zero yields 0, ** takes the integer-exponent path
// when the exponent is integral, maximum/minimum are (a > b) ? a : b and
// (a < b) ? a : b, comparisons produce 1/0 in the output dtype, unary math
// on integers computes in float and converts back.  Math uses the accurate
// device libm (no fast-math); no contraction (-ffp-contract=off).
#include "pt_common.h"

#include <math.h>
#include <string.h>

#include <initializer_list>
#include <utility>

namespace pt {

struct EwShape {
    int ndims;
    long long shape[PT_MAX_DIMS];
    long long sa[PT_MAX_DIMS];
    long long sb[PT_MAX_DIMS];
    long long sc[PT_MAX_DIMS];
    long long total;
};

// 32-bit form of an EwShape, used when the element count and every
// operand's largest offset stay below 2^31: index decoding then costs 32-bit
// divisions instead of emulated 64-bit ones.
struct EwShape32 {
    int ndims;
    unsigned shape[PT_MAX_DIMS];
    unsigned sa[PT_MAX_DIMS];
    unsigned sb[PT_MAX_DIMS];
    unsigned sc[PT_MAX_DIMS];
    unsigned total;
};

static bool to32(const EwShape &s, EwShape32 &o)
{
    const long long lim = 0x7fffffffLL;
    if (s.total > lim) return false;
    long long ma = 0, mb = 0, mc = 0;
    for (int d = 0; d < s.ndims; d++) {
        ma += (s.shape[d] - 1) * s.sa[d];
        mb += (s.shape[d] - 1) * s.sb[d];
        mc += (s.shape[d] - 1) * s.sc[d];
    }
    if (ma > lim || mb > lim || mc > lim) return false;
    o.ndims = s.ndims;
    o.total = (unsigned)s.total;
    for (int d = 0; d < s.ndims; d++) {
        o.shape[d] = (unsigned)s.shape[d];
        o.sa[d] = (unsigned)s.sa[d];
        o.sb[d] = (unsigned)s.sb[d];
        o.sc[d] = (unsigned)s.sc[d];
    }
    return true;
}

// Merge dims so that each operand's addressing stays affine; drop extent-1.
static void collapse(const int *shape, int ndims, const size_t *sa, const size_t *sb,
                     const size_t *sc, EwShape &o)
{
    o.ndims = 0;
    o.total = 1;
    for (int d = 0; d < ndims; d++) {
        long long e = shape[d];
        o.total *= e;
        if (e == 1) continue;
        long long a = sa ? (long long)sa[d] : 0, b = sb ? (long long)sb[d] : 0,
                  c = sc ? (long long)sc[d] : 0;
        if (o.ndims > 0) {
            int k = o.ndims - 1;
            if (o.sa[k] == a * e && o.sb[k] == b * e && o.sc[k] == c * e) {
                o.shape[k] *= e;
                o.sa[k] = a;
                o.sb[k] = b;
                o.sc[k] = c;
                continue;
            }
        }
        o.shape[o.ndims] = e;
        o.sa[o.ndims] = a;
        o.sb[o.ndims] = b;
        o.sc[o.ndims] = c;
        o.ndims++;
    }
}

// ------------------------------------------------------------ conversions
template <typename CT>
__device__ __forceinline__ CT ld(const void *p, int dt, long long i)
{
    switch (dt) {
    case PT_FLOAT32: return (CT)((const float *)p)[i];
    case PT_FLOAT64: return (CT)((const double *)p)[i];
    case PT_FLOAT16: return (CT)f16_to_float(((const uint16_t *)p)[i]);
    case PT_BFLOAT16: return (CT)bf16_to_float(((const uint16_t *)p)[i]);
    case PT_INT8: return (CT)((const int8_t *)p)[i];
    case PT_INT16: return (CT)((const int16_t *)p)[i];
    case PT_INT32: return (CT)((const int32_t *)p)[i];
    case PT_INT64: return (CT)((const int64_t *)p)[i];
    case PT_UINT8: return (CT)((const uint8_t *)p)[i];
    case PT_UINT16: return (CT)((const uint16_t *)p)[i];
    case PT_UINT32: return (CT)((const uint32_t *)p)[i];
    case PT_UINT64: return (CT)((const uint64_t *)p)[i];
    case PT_BOOL: return (CT)(((const uint8_t *)p)[i] != 0);
    default: return (CT)0;
    }
}

template <typename CT>
__device__ __forceinline__ void st(void *p, int dt, long long i, CT v)
{
    switch (dt) {
    case PT_FLOAT32: ((float *)p)[i] = (float)v; break;
    case PT_FLOAT64: ((double *)p)[i] = (double)v; break;
    case PT_FLOAT16: ((uint16_t *)p)[i] = float_to_f16((float)v); break;
    case PT_BFLOAT16: ((uint16_t *)p)[i] = float_to_bf16((float)v); break;
    case PT_INT8: ((int8_t *)p)[i] = (int8_t)v; break;
    case PT_INT16: ((int16_t *)p)[i] = (int16_t)v; break;
    case PT_INT32: ((int32_t *)p)[i] = (int32_t)v; break;
    case PT_INT64: ((int64_t *)p)[i] = (int64_t)v; break;
    case PT_UINT8: ((uint8_t *)p)[i] = (uint8_t)v; break;
    case PT_UINT16: ((uint16_t *)p)[i] = (uint16_t)v; break;
    case PT_UINT32: ((uint32_t *)p)[i] = (uint32_t)v; break;
    case PT_UINT64: ((uint64_t *)p)[i] = (uint64_t)v; break;
    case PT_BOOL: ((uint8_t *)p)[i] = v != (CT)0; break;
    default: break;
    }
}

// Compute type of an output dtype: float for f32/f16/bf16, double for f64,
// int64 for signed integers, uint64 for unsigned integers and bool.
enum { CT_F32 = 0, CT_F64, CT_I64, CT_U64 };
static int compute_class(int dt)
{
    switch (dt) {
    case PT_FLOAT32: case PT_FLOAT16: case PT_BFLOAT16: return CT_F32;
    case PT_FLOAT64: return CT_F64;
    case PT_INT8: case PT_INT16: case PT_INT32: case PT_INT64: return CT_I64;
    default: return CT_U64;
    }
}

// Arithmetic is evaluated at the width of the output dtype: narrow integer
// results wrap exactly as the reference's scalar_t arithmetic does once
// stored, and int64/uint64 use their own width.
template <typename CT> __device__ __forceinline__ CT int_pow(CT base, int e)
{
    CT r = (CT)1;
    while (e > 0) {
        if (e & 1) r = r * base;
        base = base * base;
        e >>= 1;
    }
    return r;
}

template <typename CT>
__device__ __forceinline__ CT pow_op(CT a, CT b)
{
    if constexpr (sizeof(CT) == 8 && (CT)0.5 == (CT)0) {
        // integer types: integral exponent path only
        int e = (int)b;
        if (e == 0) return (CT)1;
        if (e == 1) return a;
        if (e == 2) return a * a;
        if (e == 3) return a * a * a;
        if (e < 0) return (CT)0;
        return int_pow(a, e);
    } else {
        if (b == floor(b)) {
            int e = (int)b;
            if (e == 0) return (CT)1;
            if (e == 1) return a;
            if (e == 2) return a * a;
            if (e == 3) return a * a * a;
            if (e < 0) return (CT)1 / int_pow(a, -e);
            return int_pow(a, e);
        }
        if constexpr (sizeof(CT) == 4) return powf(a, b);
        else return pow(a, b);
    }
}

template <typename CT>
__device__ __forceinline__ CT bin_op(int op, CT a, CT b)
{
    switch (op) {
    case PT_OP_ADD: return a + b;
    case PT_OP_SUB: return a - b;
    case PT_OP_MUL: return a * b;
    case PT_OP_DIV:
        if constexpr ((CT)0.5 == (CT)0) return b == (CT)0 ? (CT)0 : a / b;
        else return a / b;
    case PT_OP_POW: return pow_op<CT>(a, b);
    case PT_OP_MAXIMUM: return a > b ? a : b;
    case PT_OP_MINIMUM: return a < b ? a : b;
    case PT_OP_GT: return a > b ? (CT)1 : (CT)0;
    case PT_OP_LT: return a < b ? (CT)1 : (CT)0;
    case PT_OP_EQ: return a == b ? (CT)1 : (CT)0;
    case PT_OP_NE: return a != b ? (CT)1 : (CT)0;
    case PT_OP_GE: return a >= b ? (CT)1 : (CT)0;
    case PT_OP_LE: return a <= b ? (CT)1 : (CT)0;
    default: return (CT)0;
    }
}

// 32-bit integer outputs narrower than 64 bits evaluate in int64/uint64 and
// truncate on store, which equals wrapping arithmetic in the narrow type for
// + - * (modular), and is exact for comparisons / max / min.

template <typename SH, typename IT>
__device__ __forceinline__ IT offset_of(const SH &s, const IT *st, IT i)
{
    IT off = 0;
    for (int d = s.ndims - 1; d >= 0; d--) {
        IT e = s.shape[d];
        IT q = i / e;
        off += (i - q * e) * st[d];
        i = q;
    }
    return off;
}

// SH: EwShape (64-bit indices) or EwShape32.
template <typename CT, typename SH>
__global__ __launch_bounds__(256) void k_binary(const void *__restrict__ a, int dta,
                                                const void *__restrict__ b, int dtb,
                                                void *__restrict__ out, int dto, int op,
                                                SH s, int b_scalar, CT scalar, int reverse)
{
    using IT = decltype(s.total);
    IT i = (IT)blockIdx.x * blockDim.x + threadIdx.x;
    const IT stride = (IT)gridDim.x * blockDim.x;
    for (; i < s.total; i += stride) {
        CT x = ld<CT>(a, dta, offset_of(s, s.sa, i));
        CT y = b_scalar ? scalar : ld<CT>(b, dtb, offset_of(s, s.sb, i));
        st<CT>(out, dto, i, reverse ? bin_op<CT>(op, y, x) : bin_op<CT>(op, x, y));
    }
}

// ---------------------------------------------------- 16-byte vector path
// Floating outputs of 32 and 16 bits: each thread makes 16 bytes of the
// (contiguous) output, 4 or 8 elements, from operands that are contiguous
// too, walk the rows of a collapsed [rows, cols] output (column stride 1, any
// row stride, 0 for a broadcast row), hold one value per row (column stride
// 0), or are one immediate.  The output is cut into chunks as one flat
// array, so that chunks of it and of contiguous operands stay aligned
// whatever cols is; a chunk that crosses a row's end takes the other kinds of
// operand element by element.  All of these kernels are bound by HBM: one
// element per thread with an index decode, a dtype switch and a 2-byte load
// took 91 us for x + b on [8000, 3001] bf16 (96 MB); the six calls of an
// eager activation on it went from 499 to 150 us.
enum { OPND_FLAT = 0, OPND_IMM, OPND_ROWS, OPND_COL, OPND_ANY = -1 };
struct Opnd {
    const void *p;
    int mode;
    unsigned rs;  // row stride (OPND_ROWS, OPND_COL)
    float imm;
};

// A thread's chunk: elements i .. i + V - 1 of the output, element i being
// (r, c) of [rows, cols] where an operand needs that; `valid` of them exist.
// `whole`: every chunk of the block is complete, `even`: and none crosses a
// row's end, each one scalar test a block.
template <int V>
struct ChunkPos {
    size_t i;
    int valid;
    bool whole, even;
    unsigned r = 0, c = 0;
    __device__ __forceinline__ ChunkPos(size_t total, unsigned cols, bool rowwise)
    {
        const size_t b = (size_t)blockIdx.x * (256 * V);
        i = b + threadIdx.x * V;
        whole = b + 256 * V <= total;
        valid = whole || i + V <= total ? V : i < total ? (int)(total - i) : 0;
        even = whole && cols % V == 0;
        if (rowwise) {  // (the host keeps such outputs below 2^31 elements)
            r = (unsigned)i / cols;
            c = (unsigned)i - r * cols;
        }
    }
};

// N bytes at any element boundary (16 at a time where N allows).
typedef unsigned int u32x4v __attribute__((ext_vector_type(4), aligned(1)));
typedef unsigned int u32x2v __attribute__((ext_vector_type(2), aligned(1)));
template <int N, bool NT>
__device__ __forceinline__ void ld_bytes(void *dst, const void *src)
{
    if constexpr (N >= 16) {
#pragma unroll
        for (int q = 0; q < N / 16; q++) {
            u32x4v t;
            if constexpr (NT) t = __builtin_nontemporal_load((const u32x4v *)src + q);
            else t = ((const u32x4v *)src)[q];
            memcpy((char *)dst + 16 * q, &t, 16);
        }
    } else if constexpr (N == 8) {
        const u32x2v t = *(const u32x2v *)src;
        memcpy(dst, &t, 8);
    } else {
        memcpy(dst, src, N);
    }
}

// Elements of an operand for the chunk at q, as they lie in memory (T: an
// unsigned type of the element's size).  MODE: the operand's layout where
// the kernel is built for it (no branch around its load), else OPND_ANY.
template <int MODE, typename T, int V, bool NT>
__device__ __forceinline__ void fetch(const Opnd &o, const ChunkPos<V> &q, unsigned cols, T (&v)[V])
{
    const T *p = (const T *)o.p;
    const int mode = MODE == OPND_ANY ? o.mode : MODE;
    unsigned r = q.r, c = q.c;
    if (mode == OPND_IMM) return;
    if (mode == OPND_FLAT) {
        if (q.whole) {
            ld_bytes<V * sizeof(T), NT>(v, p + q.i);
        } else {
#pragma unroll
            for (int k = 0; k < V; k++) v[k] = k < q.valid ? p[q.i + k] : (T)0;
        }
    } else if (q.even || (c + V <= cols && q.valid == V)) {
        if (mode == OPND_ROWS) {
            ld_bytes<V * sizeof(T), false>(v, p + (size_t)r * o.rs + c);
        } else {
            const T t = p[(size_t)r * o.rs];
#pragma unroll
            for (int k = 0; k < V; k++) v[k] = t;
        }
    } else {
        const unsigned cs = mode == OPND_ROWS ? 1u : 0u;
#pragma unroll
        for (int k = 0; k < V; k++) {
            v[k] = k < q.valid ? p[(size_t)r * o.rs + c * cs] : (T)0;
            if (++c == cols) {
                c = 0;
                r++;
            }
        }
    }
}

template <int DT> struct VecT;
template <> struct VecT<PT_FLOAT32> {
    using T = uint32_t;
    __device__ static float to(T t) { return __uint_as_float(t); }
    __device__ static T from(float f) { return __float_as_uint(f); }
};
template <> struct VecT<PT_BFLOAT16> {
    using T = uint16_t;
    __device__ static float to(T t) { return bf16_to_float(t); }
    __device__ static T from(float f) { return float_to_bf16(f); }
};
template <> struct VecT<PT_FLOAT16> {
    using T = uint16_t;
    __device__ static float to(T t) { return f16_to_float(t); }
    __device__ static T from(float f) { return float_to_f16(f); }
};

template <int DT, int MODE, int V>
__device__ __forceinline__ void to_float(const Opnd &o, const typename VecT<DT>::T (&t)[V], float (&v)[V])
{
    const bool imm = MODE == OPND_ANY ? o.mode == OPND_IMM : MODE == OPND_IMM;
#pragma unroll
    for (int k = 0; k < V; k++) v[k] = imm ? o.imm : VecT<DT>::to(t[k]);
}

template <typename T, int V, bool NT>
__device__ __forceinline__ void put(T *out, const ChunkPos<V> &q, const T (&v)[V])
{
    if (q.whole) {
        constexpr int N = V * sizeof(T) / 16;
#pragma unroll
        for (int j = 0; j < N; j++) {
            u32x4v t;
            memcpy(&t, (const char *)v + 16 * j, 16);
            if constexpr (NT) __builtin_nontemporal_store(t, (u32x4v *)(out + q.i) + j);
            else ((u32x4v *)(out + q.i))[j] = t;
        }
    } else {
#pragma unroll
        for (int k = 0; k < V; k++)
            if (k < q.valid) out[q.i + k] = v[k];
    }
}

// f(op as an integral constant): the op's dispatch is one scalar branch a
// thread instead of one an element.
template <typename F>
__device__ __forceinline__ void with_bin_op(int op, F f)
{
    switch (op) {
    case PT_OP_ADD: f(std::integral_constant<int, PT_OP_ADD>{}); break;
    case PT_OP_SUB: f(std::integral_constant<int, PT_OP_SUB>{}); break;
    case PT_OP_MUL: f(std::integral_constant<int, PT_OP_MUL>{}); break;
    case PT_OP_DIV: f(std::integral_constant<int, PT_OP_DIV>{}); break;
    case PT_OP_POW: f(std::integral_constant<int, PT_OP_POW>{}); break;
    case PT_OP_MAXIMUM: f(std::integral_constant<int, PT_OP_MAXIMUM>{}); break;
    case PT_OP_MINIMUM: f(std::integral_constant<int, PT_OP_MINIMUM>{}); break;
    case PT_OP_GT: f(std::integral_constant<int, PT_OP_GT>{}); break;
    case PT_OP_LT: f(std::integral_constant<int, PT_OP_LT>{}); break;
    case PT_OP_EQ: f(std::integral_constant<int, PT_OP_EQ>{}); break;
    case PT_OP_NE: f(std::integral_constant<int, PT_OP_NE>{}); break;
    case PT_OP_GE: f(std::integral_constant<int, PT_OP_GE>{}); break;
    case PT_OP_LE: f(std::integral_constant<int, PT_OP_LE>{}); break;
    }
}

// DT: the operands' type, DTO: the output's (float32 where 16-bit operands
// divide).
template <int DT, int DTO, bool NT, int MA, int MB>
__global__ __launch_bounds__(256) void k_binary_vec(Opnd a, Opnd b, void *__restrict__ out, int op, size_t total,
                                                    unsigned cols)
{
    using T = typename VecT<DT>::T;
    using TO = typename VecT<DTO>::T;
    constexpr int V = 16 / sizeof(T);
    const ChunkPos<V> q(total, cols, (MA == OPND_ANY ? a.mode : MA) >= OPND_ROWS ||
                                         (MB == OPND_ANY ? b.mode : MB) >= OPND_ROWS);
    if (!q.valid) return;
    T u[V], w[V];
    fetch<MA, T, V, NT>(a, q, cols, u);
    fetch<MB, T, V, NT>(b, q, cols, w);
    float x[V], y[V];
    TO z[V];
    to_float<DT, MA>(a, u, x);
    to_float<DT, MB>(b, w, y);
    with_bin_op(op, [&](auto O) {
#pragma unroll
        for (int k = 0; k < V; k++) z[k] = VecT<DTO>::from(bin_op<float>(decltype(O)::value, x[k], y[k]));
    });
    put<TO, V, NT>((TO *)out, q, z);
}

// where(c, x, y): elements of ESZ bytes moved as bits, a condition of CSZ
// bytes an element that holds where the bits under `mask` (a float's without
// its sign) are not all zero.
template <int N> struct BitsT;
template <> struct BitsT<1> { using T = uint8_t; };
template <> struct BitsT<2> { using T = uint16_t; };
template <> struct BitsT<4> { using T = uint32_t; };
template <> struct BitsT<8> { using T = uint64_t; };

template <int ESZ, int CSZ, bool NT>
__global__ __launch_bounds__(256) void k_where_vec(Opnd cond, Opnd x, Opnd y, void *__restrict__ out, uint32_t mask,
                                                   size_t total, unsigned cols)
{
    using T = typename BitsT<ESZ>::T;
    using CT = typename BitsT<CSZ>::T;
    constexpr int V = 16 / ESZ;
    const ChunkPos<V> q(total, cols, cond.mode >= OPND_ROWS || x.mode >= OPND_ROWS || y.mode >= OPND_ROWS);
    if (!q.valid) return;
    CT c[V];
    T u[V], w[V];
    fetch<OPND_ANY, CT, V, NT>(cond, q, cols, c);
    fetch<OPND_ANY, T, V, NT>(x, q, cols, u);
    fetch<OPND_ANY, T, V, NT>(y, q, cols, w);
#pragma unroll
    for (int k = 0; k < V; k++) u[k] = ((uint32_t)c[k] & mask) ? u[k] : w[k];
    put<T, V, NT>((T *)out, q, u);
}

// Casts between the 32- and 16-bit floating types; V elements are 16 bytes
// of the narrower type.
template <int DTI, int DTO>
__global__ __launch_bounds__(256) void k_cast_vec(Opnd x, void *__restrict__ out, size_t total, unsigned cols)
{
    using TI = typename VecT<DTI>::T;
    using TO = typename VecT<DTO>::T;
    constexpr int V = 8;
    const ChunkPos<V> q(total, cols, x.mode >= OPND_ROWS);
    if (!q.valid) return;
    TI t[V];
    TO z[V];
    fetch<OPND_ANY, TI, V, false>(x, q, cols, t);
#pragma unroll
    for (int k = 0; k < V; k++) z[k] = VecT<DTO>::from(VecT<DTI>::to(t[k]));
    put<TO, V, false>((TO *)out, q, z);
}

// ------------------------------------------------------------------ unary
template <typename CT>
__device__ __forceinline__ CT unary_f(int op, CT v)
{
    constexpr bool F = sizeof(CT) == 4;
    switch (op) {
    case PT_OP_EXP: return F ? expf(v) : exp(v);
    case PT_OP_EXPM1: return F ? expm1f(v) : expm1(v);
    case PT_OP_EXP2: return F ? exp2f(v) : exp2(v);
    case PT_OP_LOG: return F ? logf(v) : log(v);
    case PT_OP_LOG1P: return F ? log1pf(v) : log1p(v);
    case PT_OP_LOG2: return F ? log2f(v) : log2(v);
    case PT_OP_LOG10: return F ? log10f(v) : log10(v);
    case PT_OP_SQRT: return F ? sqrtf(v) : sqrt(v);
    case PT_OP_SIN: return F ? sinf(v) : sin(v);
    case PT_OP_COS: return F ? cosf(v) : cos(v);
    case PT_OP_TAN: return F ? tanf(v) : tan(v);
    case PT_OP_ASIN: return F ? asinf(v) : asin(v);
    case PT_OP_ACOS: return F ? acosf(v) : acos(v);
    case PT_OP_ATAN: return F ? atanf(v) : atan(v);
    case PT_OP_SINH: return F ? sinhf(v) : sinh(v);
    case PT_OP_COSH: return F ? coshf(v) : cosh(v);
    case PT_OP_TANH: return F ? tanhf(v) : tanh(v);
    case PT_OP_ABS: return v < (CT)0 ? -v : v;
    case PT_OP_NEG: return -v;
    case PT_OP_FLOOR: return F ? floorf(v) : floor(v);
    case PT_OP_CEIL: return F ? ceilf(v) : ceil(v);
    case PT_OP_ROUND: return F ? roundf(v) : round(v);
    default: return v;
    }
}

template <typename CT, typename SH>
__global__ __launch_bounds__(256) void k_unary(const void *__restrict__ x, int dt,
                                               void *__restrict__ out, int op, SH s)
{
    using IT = decltype(s.total);
    IT i = (IT)blockIdx.x * blockDim.x + threadIdx.x;
    const IT stride = (IT)gridDim.x * blockDim.x;
    for (; i < s.total; i += stride) {
        IT off = offset_of(s, s.sa, i);
        if constexpr (sizeof(CT) == 8 && (CT)0.5 == (CT)0) {
            // integers: abs/neg exact, floor/ceil/round identity, the rest
            // through float (cuda_op_functors.cuh:153-449)
            CT v = ld<CT>(x, dt, off);
            CT r;
            if (op == PT_OP_ABS) r = v < (CT)0 ? (CT)0 - v : v;
            else if (op == PT_OP_NEG) r = (CT)0 - v;
            else if (op == PT_OP_FLOOR || op == PT_OP_CEIL || op == PT_OP_ROUND) r = v;
            else r = (CT)unary_f<float>(op, (float)v);
            st<CT>(out, dt, i, r);
        } else {
            st<CT>(out, dt, i, unary_f<CT>(op, ld<CT>(x, dt, off)));
        }
    }
}

// OPC >= 0: the op fixed at compile time (the per-element dispatch folds
// away); OPC < 0: the op comes from `op`.
template <int DT, int OPC, bool NT, int MX>
__global__ __launch_bounds__(256) void k_unary_vec(Opnd x, void *__restrict__ out, int op_arg, size_t total,
                                                   unsigned cols)
{
    using T = typename VecT<DT>::T;
    constexpr int V = 16 / sizeof(T);
    const int op = OPC >= 0 ? OPC : op_arg;
    const ChunkPos<V> q(total, cols, (MX == OPND_ANY ? x.mode : MX) >= OPND_ROWS);
    if (!q.valid) return;
    T t[V];
    fetch<MX, T, V, NT>(x, q, cols, t);
    T z[V];
#pragma unroll
    for (int k = 0; k < V; k++) z[k] = VecT<DT>::from(unary_f<float>(op, VecT<DT>::to(t[k])));
    put<T, V, NT>((T *)out, q, z);
}

// --------------------------------------------------------- cast / where
// Casts follow the reference's converting kernels: to f16/bf16 through
// float with RNE, floats to integers by C conversion, anything to bool by
// != 0 (factory_kernels.cu:128-163).
__device__ __forceinline__ void cast_elem(const void *x, int dti, long long oi, void *out, int dto,
                                          long long i)
{
    if (dti == dto) {
        switch (dtype_size(dti)) {
        case 1: ((uint8_t *)out)[i] = ((const uint8_t *)x)[oi]; return;
        case 2: ((uint16_t *)out)[i] = ((const uint16_t *)x)[oi]; return;
        case 4: ((uint32_t *)out)[i] = ((const uint32_t *)x)[oi]; return;
        default: ((uint64_t *)out)[i] = ((const uint64_t *)x)[oi]; return;
        }
    }
    const bool src_int64 = dti == PT_INT64, src_u64 = dti == PT_UINT64;
    if (src_int64) { st<long long>(out, dto, i, ((const int64_t *)x)[oi]); return; }
    if (src_u64) { st<unsigned long long>(out, dto, i, ((const uint64_t *)x)[oi]); return; }
    if (dto == PT_INT64) { st<long long>(out, dto, i, (long long)ld<double>(x, dti, oi)); return; }
    if (dto == PT_UINT64) { st<unsigned long long>(out, dto, i, (unsigned long long)ld<double>(x, dti, oi)); return; }
    st<double>(out, dto, i, ld<double>(x, dti, oi));
}

template <typename SH>
__global__ __launch_bounds__(256) void k_cast(const void *__restrict__ x, int dti,
                                              void *__restrict__ out, int dto, SH s)
{
    using IT = decltype(s.total);
    IT i = (IT)blockIdx.x * blockDim.x + threadIdx.x;
    const IT stride = (IT)gridDim.x * blockDim.x;
    for (; i < s.total; i += stride) cast_elem(x, dti, (long long)offset_of(s, s.sa, i), out, dto, (long long)i);
}

template <typename SH>
__global__ __launch_bounds__(256) void k_where(const void *__restrict__ c, int dtc,
                                               const void *__restrict__ x, const void *__restrict__ y,
                                               int esz, void *__restrict__ out, SH s)
{
    using IT = decltype(s.total);
    IT i = (IT)blockIdx.x * blockDim.x + threadIdx.x;
    const IT stride = (IT)gridDim.x * blockDim.x;
    for (; i < s.total; i += stride) {
        const IT co = offset_of(s, s.sc, i);
        bool pick = ld<double>(c, dtc, co) != 0.0;
        if (dtc == PT_INT64 || dtc == PT_UINT64) pick = ((const uint64_t *)c)[co] != 0;
        const void *src = pick ? x : y;
        IT o = offset_of(s, pick ? s.sa : s.sb, i);
        switch (esz) {
        case 1: ((uint8_t *)out)[i] = ((const uint8_t *)src)[o]; break;
        case 2: ((uint16_t *)out)[i] = ((const uint16_t *)src)[o]; break;
        case 4: ((uint32_t *)out)[i] = ((const uint32_t *)src)[o]; break;
        default: ((uint64_t *)out)[i] = ((const uint64_t *)src)[o]; break;
        }
    }
}

__global__ __launch_bounds__(256) void k_fill(void *__restrict__ out, int esz, long long n, uint64_t bits)
{
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        switch (esz) {
        case 1: ((uint8_t *)out)[i] = (uint8_t)bits; break;
        case 2: ((uint16_t *)out)[i] = (uint16_t)bits; break;
        case 4: ((uint32_t *)out)[i] = (uint32_t)bits; break;
        default: ((uint64_t *)out)[i] = bits; break;
        }
    }
}

// ------------------------------------------------------------------ host
static unsigned grid_for(long long n, int per_thread = 1)
{
    // one thread per work item: a full grid streams HBM faster on gfx950
    // than a capped grid-stride loop; the loops cover grids above the limit
    long long blocks = (n + 256LL * per_thread - 1) / (256LL * per_thread);
    if (blocks > 0x7fffffffLL) blocks = 0x7fffffffLL;
    if (blocks < 1) blocks = 1;
    return (unsigned)blocks;
}

static bool valid_binary_op(int op)
{
    return (op >= PT_OP_ADD && op <= PT_OP_POW) || (op >= PT_OP_GT && op <= PT_OP_LE) ||
           op == PT_OP_MAXIMUM || op == PT_OP_MINIMUM;
}

static bool valid_unary_op(int op)
{
    return (op >= PT_OP_EXP && op <= PT_OP_NEG) || (op >= PT_OP_CEIL && op <= PT_OP_ROUND);
}

// scalar value converted to a compute class
static double scalar_as_double(const pt_scalar_t *s)
{
    switch (s->dtype) {
    case PT_FLOAT32: return s->v.f32;
    case PT_FLOAT64: return s->v.f64;
    case PT_FLOAT16: {
        uint16_t h = s->v.u16;
        _Float16 f;
        memcpy(&f, &h, 2);
        return (double)f;
    }
    case PT_BFLOAT16: {
        uint32_t b = (uint32_t)s->v.u16 << 16;
        float f;
        memcpy(&f, &b, 4);
        return f;
    }
    case PT_UINT8: case PT_UINT16: case PT_UINT32: case PT_UINT64: case PT_BOOL:
        return (double)s->v.u64;
    default: return (double)s->v.i64;
    }
}

static long long scalar_as_i64(const pt_scalar_t *s)
{
    if (dtype_is_floating(s->dtype)) return (long long)scalar_as_double(s);
    return s->v.i64;
}

// An operand of the vector kernels from its collapsed strides st; false when
// its layout is none of theirs (the generic kernels decode any layout).
static bool as_opnd(const EwShape &s, const long long *st, const void *p, Opnd &o)
{
    o = Opnd{p, OPND_FLAT, 0u, 0.0f};
    if (s.ndims == 0) return true;
    if (s.ndims > 2) return false;
    const long long cols = s.shape[s.ndims - 1], cs = st[s.ndims - 1], rs = s.ndims == 2 ? st[0] : 0;
    if (cs == 1 && (s.ndims == 1 || rs == cols)) return true;
    const long long rows = s.ndims == 2 ? s.shape[0] : 1;
    if ((cs != 0 && cs != 1) || s.total > 0x7fffffffLL || rs < 0 || rs > 0x7fffffffLL ||
        (rows - 1) * rs + cols > 0x7fffffffLL)
        return false;
    o.mode = cs == 1 ? OPND_ROWS : OPND_COL;
    o.rs = (unsigned)rs;
    return true;
}

static unsigned opnd_cols(const EwShape &s)
{
    const long long c = s.ndims ? s.shape[s.ndims - 1] : 1;
    return c > 0x7fffffffLL ? 1u : (unsigned)c;  // only read where an operand is rowwise (at most 2^31 elements)
}

// Streaming accesses bypass cache retention (nontemporal) in calls through
// aligned chunks whose tensors do not fit the 256 MB Infinity Cache together:
// there is nothing left in it for the next call, and what such a call evicts is
// the result of the call before.  The line lies at 272 MB of one full operand
// and the output, at 344 MB of more operands.  Eager calls on one of four
// inputs in turn, us cached against nontemporal, by size of a tensor:
//   fp32 x * 2       128 MB 40.4 / 42.9, 144 MB 51.6 / 47.7, 256 MB 89.7 / 84.0
//   fp32 tanh        128 MB 41.0 / 42.0, 144 MB 51.3 / 46.7, 512 MB 173 / 163
//   fp32 x + m       100 MB 42.8 / 44.7, 112 MB 49.9 / 50.1, 120 MB 56.0 / 53.2,
//                    192 MB 96.2 / 86.4, 512 MB 251 / 233
//   fp32 where       100 MB 44.8 / 47.5, 120 MB 58.1 / 56.2, 192 MB 97.9 / 90.4
//   bf16 x * 2       128 MB 41.5 / 43.5, 144 MB 51.8 / 48.7
//   bf16 x + m       112 MB 52.1 / 53.2, 120 MB 57.7 / 56.3, 192 MB 94.8 / 90.0
// and chains of them alike (bias, scale and tanh of fp32 128 MB 160 / 178, 192 MB
// 273 / 262).  Calls that are as fast or faster cached at every size are not
// asked: 16-bit unary calls (512 MB 171 / 179), 16-bit where (272 / 294), 16-bit
// operands with one row or one value per row (184 / 188), and calls whose
// chunks have 32 bytes on one side, two stores of a lane to every line (a cast
// from bf16 to fp32: 128 MB 71 / 99, 512 MB 272 / 402).
constexpr size_t kStreamOne = (size_t)272 << 20, kStreamMore = (size_t)344 << 20;
static bool streams(size_t bytes, int operands, std::initializer_list<const void *> ptrs)
{
    for (const void *p : ptrs)
        if ((uintptr_t)p & 15) return false;
    return bytes >= (operands > 1 ? kStreamMore : kStreamOne);
}

static bool vec_float(int dt) { return dt == PT_FLOAT32 || dt == PT_FLOAT16 || dt == PT_BFLOAT16; }

// f(integral constant of the dtype) for the vector kernels' types.
template <typename F>
static void with_vec_dtype(int dt, F f)
{
    if (dt == PT_FLOAT32) f(std::integral_constant<int, PT_FLOAT32>{});
    else if (dt == PT_FLOAT16) f(std::integral_constant<int, PT_FLOAT16>{});
    else f(std::integral_constant<int, PT_BFLOAT16>{});
}

static pt_status binary_impl(const void *a, int dta, const size_t *sa, size_t offa,
                             const void *b, int dtb, const size_t *sb, size_t offb,
                             const pt_scalar_t *scalar, int reverse, void *out, int dto, int op,
                             const int *shape, int ndims, pt_stream_t stream)
{
    PT_TRY(ensure_init());
    if (!dtype_valid(dta) || !dtype_valid(dto) || (!scalar && !dtype_valid(dtb)))
        return fail(PT_ERR_INVALID, "elementwise: unknown dtype");
    if (!valid_binary_op(op)) return fail(PT_ERR_INVALID, "elementwise: unsupported op %d", op);
    if (ndims < 0 || ndims > PT_MAX_DIMS) return fail(PT_ERR_INVALID, "elementwise: rank %d", ndims);
    size_t cstr[PT_MAX_DIMS];
    size_t acc = 1;
    for (int d = ndims - 1; d >= 0; d--) {
        if (shape[d] < 0) return fail(PT_ERR_INVALID, "elementwise: negative extent");
        cstr[d] = acc;
        acc *= (size_t)shape[d];
    }
    EwShape s;
    collapse(shape, ndims, sa, scalar ? nullptr : sb, cstr, s);
    if (s.total == 0) return PT_OK;
    hipStream_t st_ = stream_of(stream);
    const char *pa = (const char *)a + offa * dtype_size(dta);
    const char *pb = scalar ? nullptr : (const char *)b + offb * dtype_size(dtb);
    Opnd oa, ob;
    bool vec = vec_float(dta) && (dto == dta || dto == PT_FLOAT32) && (scalar || dtb == dta) &&
               as_opnd(s, s.sa, pa, oa);
    if (vec && scalar) ob = Opnd{nullptr, OPND_IMM, 0u, (float)scalar_as_double(scalar)};
    else vec = vec && as_opnd(s, s.sb, pb, ob);
    if (vec) {
        if (reverse) std::swap(oa, ob);
        const size_t total = (size_t)s.total;
        auto full = [](const Opnd &o) { return o.mode == OPND_FLAT || o.mode == OPND_IMM; };
        const int operands = (oa.mode == OPND_FLAT) + (ob.mode == OPND_FLAT);
        const bool nt = dto == dta && (dta == PT_FLOAT32 || (full(oa) && full(ob))) &&
                        streams(total * dtype_size(dta) * (size_t)(operands + 1), operands,
                                {oa.mode == OPND_FLAT ? oa.p : nullptr, ob.mode == OPND_FLAT ? ob.p : nullptr, out});
        with_vec_dtype(dta, [&](auto D) {
            constexpr int DT = decltype(D)::value;
            const unsigned grid = grid_for(s.total, 16 / (int)sizeof(typename VecT<DT>::T)), cols = opnd_cols(s);
            auto go = [&](auto O, auto MA, auto MB) {
                constexpr int DO = decltype(O)::value, A = decltype(MA)::value, B = decltype(MB)::value;
                if constexpr (DO == DT) {
                    if (nt) {
                        k_binary_vec<DT, DO, true, A, B><<<grid, 256, 0, st_>>>(oa, ob, out, op, total, cols);
                        return;
                    }
                }
                k_binary_vec<DT, DO, false, A, B><<<grid, 256, 0, st_>>>(oa, ob, out, op, total, cols);
            };
            // the layouts of most calls have kernels of their own: y * z of
            // a row and [16384, 8192] fp32 took 181 us with the layouts read
            // at run time (two branches before the loads) against 169.5
            // (177 with the contiguous operand loaded before the row), one
            // value per row (x * c) 184 against 166
            using FL = std::integral_constant<int, OPND_FLAT>;
            using IM = std::integral_constant<int, OPND_IMM>;
            using RW = std::integral_constant<int, OPND_ROWS>;
            using CL = std::integral_constant<int, OPND_COL>;
            using AN = std::integral_constant<int, OPND_ANY>;
            if (dto != dta) go(std::integral_constant<int, PT_FLOAT32>{}, AN{}, AN{});
            else if (oa.mode == OPND_FLAT && ob.mode == OPND_FLAT) go(D, FL{}, FL{});
            else if (oa.mode == OPND_FLAT && ob.mode == OPND_IMM) go(D, FL{}, IM{});
            else if (oa.mode == OPND_FLAT && ob.mode == OPND_ROWS) go(D, FL{}, RW{});
            else if (oa.mode == OPND_ROWS && ob.mode == OPND_FLAT) go(D, RW{}, FL{});
            else if (oa.mode == OPND_FLAT && ob.mode == OPND_COL) go(D, FL{}, CL{});
            else if (oa.mode == OPND_COL && ob.mode == OPND_FLAT) go(D, CL{}, FL{});
            else go(D, AN{}, AN{});
        });
    } else {
        EwShape32 s32;
        const bool i32 = to32(s, s32);
#define PT_BIN(CT, SV)                                                                                          \
    (i32 ? (k_binary<CT, EwShape32><<<grid_for(s.total), 256, 0, st_>>>(pa, dta, pb, dtb, out, dto, op, s32, \
                                                                          scalar != nullptr, SV, reverse), 0) \
         : (k_binary<CT, EwShape><<<grid_for(s.total), 256, 0, st_>>>(pa, dta, pb, dtb, out, dto, op, s,     \
                                                                        scalar != nullptr, SV, reverse), 0))
        switch (compute_class(dto)) {
        case CT_F32: PT_BIN(float, scalar ? (float)scalar_as_double(scalar) : 0.0f); break;
        case CT_F64: PT_BIN(double, scalar ? scalar_as_double(scalar) : 0.0); break;
        case CT_I64: PT_BIN(long long, scalar ? scalar_as_i64(scalar) : 0LL); break;
        default: PT_BIN(unsigned long long, scalar ? (unsigned long long)scalar_as_i64(scalar) : 0ULL); break;
        }
#undef PT_BIN
    }
    PT_LAUNCH_CHECK("elementwise binary");
    counters().elementwise_calls++;
    return PT_OK;
}

}  // namespace pt

using namespace pt;

extern "C" {

pt_status pt_broadcast(const void *a, int dtype_a, const size_t *strides_a, size_t offset_a,
                       const void *b, int dtype_b, const size_t *strides_b, size_t offset_b,
                       void *out, int dtype_out, int op,
                       const int *shape, int ndims, pt_stream_t stream)
{
    return binary_impl(a, dtype_a, strides_a, offset_a, b, dtype_b, strides_b, offset_b, nullptr,
                       0, out, dtype_out, op, shape, ndims, stream);
}

pt_status pt_scalar(const void *input, int dtype_in, const size_t *strides, size_t offset,
                    const pt_scalar_t *scalar, int reverse, void *out, int dtype_out,
                    int op, const int *shape, int ndims, pt_stream_t stream)
{
    if (!scalar) return fail(PT_ERR_INVALID, "pt_scalar: missing scalar");
    return binary_impl(input, dtype_in, strides, offset, nullptr, dtype_in, nullptr, 0, scalar,
                       reverse, out, dtype_out, op, shape, ndims, stream);
}

pt_status pt_unary(const void *input, int dtype, const size_t *strides, size_t offset,
                   void *out, int op, const int *shape, int ndims, pt_stream_t stream)
{
    PT_TRY(ensure_init());
    if (!dtype_valid(dtype)) return fail(PT_ERR_INVALID, "unary: unknown dtype");
    if (!valid_unary_op(op)) return fail(PT_ERR_INVALID, "unary: unsupported op %d", op);
    if (ndims < 0 || ndims > PT_MAX_DIMS) return fail(PT_ERR_INVALID, "unary: rank %d", ndims);
    size_t cstr[PT_MAX_DIMS], acc = 1;
    for (int d = ndims - 1; d >= 0; d--) { cstr[d] = acc; acc *= (size_t)shape[d]; }
    EwShape s;
    collapse(shape, ndims, strides, nullptr, cstr, s);
    if (s.total == 0) return PT_OK;
    hipStream_t st_ = stream_of(stream);
    const char *px = (const char *)input + offset * dtype_size(dtype);
    Opnd ox;
    if (vec_float(dtype) && as_opnd(s, s.sa, px, ox)) {
        const size_t total = (size_t)s.total;
        const bool nt = dtype == PT_FLOAT32 &&
                        streams(total * dtype_size(dtype) * 2, 1, {ox.mode == OPND_FLAT ? px : nullptr, out});
        with_vec_dtype(dtype, [&](auto D) {
            constexpr int DT = decltype(D)::value;
            const unsigned grid = grid_for(s.total, 16 / (int)sizeof(typename VecT<DT>::T)), cols = opnd_cols(s);
            auto go = [&](auto O, auto N) {
                constexpr int OP = decltype(O)::value;
                constexpr bool NT = decltype(N)::value;
                if (ox.mode == OPND_FLAT)
                    k_unary_vec<DT, OP, NT, OPND_FLAT><<<grid, 256, 0, st_>>>(ox, out, op, total, cols);
                else
                    k_unary_vec<DT, OP, NT, OPND_ANY><<<grid, 256, 0, st_>>>(ox, out, op, total, cols);
            };
            auto pick = [&](auto N) {
                if (op == PT_OP_TANH) go(std::integral_constant<int, PT_OP_TANH>{}, N);
                else if (op == PT_OP_EXP) go(std::integral_constant<int, PT_OP_EXP>{}, N);
                else go(std::integral_constant<int, -1>{}, N);
            };
            if constexpr (DT == PT_FLOAT32) {
                if (nt) return pick(std::true_type{});
            }
            pick(std::false_type{});
        });
    } else {
        EwShape32 s32;
        const bool i32 = to32(s, s32);
#define PT_UN(CT)                                                                                     \
    (i32 ? (k_unary<CT, EwShape32><<<grid_for(s.total), 256, 0, st_>>>(px, dtype, out, op, s32), 0) \
         : (k_unary<CT, EwShape><<<grid_for(s.total), 256, 0, st_>>>(px, dtype, out, op, s), 0))
        switch (compute_class(dtype)) {
        case CT_F32: PT_UN(float); break;
        case CT_F64: PT_UN(double); break;
        case CT_I64: PT_UN(long long); break;
        default: PT_UN(unsigned long long); break;
        }
#undef PT_UN
    }
    PT_LAUNCH_CHECK("unary");
    counters().elementwise_calls++;
    return PT_OK;
}

pt_status pt_cast(const void *input, int dtype_in, const size_t *strides, size_t offset,
                  void *out, int dtype_out, const int *shape, int ndims, pt_stream_t stream)
{
    PT_TRY(ensure_init());
    if (!dtype_valid(dtype_in) || !dtype_valid(dtype_out)) return fail(PT_ERR_INVALID, "cast: unknown dtype");
    if (ndims < 0 || ndims > PT_MAX_DIMS) return fail(PT_ERR_INVALID, "cast: rank %d", ndims);
    size_t cstr[PT_MAX_DIMS], acc = 1;
    for (int d = ndims - 1; d >= 0; d--) { cstr[d] = acc; acc *= (size_t)shape[d]; }
    EwShape s;
    collapse(shape, ndims, strides, nullptr, cstr, s);
    if (s.total == 0) return PT_OK;
    hipStream_t st_ = stream_of(stream);
    const char *px = (const char *)input + offset * dtype_size(dtype_in);
    bool contig = s.ndims <= 1 && (s.ndims == 0 || s.sa[0] == 1);
    if (contig && dtype_in == dtype_out) {
        PT_TRY(check_hip(hipMemcpyAsync(out, px, (size_t)s.total * dtype_size(dtype_in),
                                        hipMemcpyDeviceToDevice, st_), "cast copy"));
        return PT_OK;
    }
    Opnd ox;
    EwShape32 s32;
    if (vec_float(dtype_in) && vec_float(dtype_out) && dtype_in != dtype_out && as_opnd(s, s.sa, px, ox)) {
        const size_t total = (size_t)s.total;
        with_vec_dtype(dtype_in, [&](auto I) {
            with_vec_dtype(dtype_out, [&](auto O) {
                constexpr int DI = decltype(I)::value, DO = decltype(O)::value;
                if constexpr (DI != DO) {
                    const unsigned grid = grid_for(s.total, 8);
                    k_cast_vec<DI, DO><<<grid, 256, 0, st_>>>(ox, out, total, opnd_cols(s));
                }
            });
        });
    } else if (to32(s, s32)) k_cast<EwShape32><<<grid_for(s.total), 256, 0, st_>>>(px, dtype_in, out, dtype_out, s32);
    else k_cast<EwShape><<<grid_for(s.total), 256, 0, st_>>>(px, dtype_in, out, dtype_out, s);
    PT_LAUNCH_CHECK("cast");
    counters().elementwise_calls++;
    return PT_OK;
}

pt_status pt_where(const void *cond, int dtype_cond, const size_t *strides_cond,
                   const void *x, const size_t *strides_x,
                   const void *y, const size_t *strides_y, int dtype_xy,
                   void *out, const int *shape, int ndims, pt_stream_t stream)
{
    PT_TRY(ensure_init());
    if (!dtype_valid(dtype_cond) || !dtype_valid(dtype_xy)) return fail(PT_ERR_INVALID, "where: unknown dtype");
    if (ndims < 0 || ndims > PT_MAX_DIMS) return fail(PT_ERR_INVALID, "where: rank %d", ndims);
    EwShape s;
    collapse(shape, ndims, strides_x, strides_y, strides_cond, s);
    if (s.total == 0) return PT_OK;
    hipStream_t st_ = stream_of(stream);
    Opnd oc, ox, oy;
    EwShape32 s32;
    const int csz = (int)dtype_size(dtype_cond), esz = (int)dtype_size(dtype_xy);
    if (csz <= 4 && (esz == 2 || esz == 4) && as_opnd(s, s.sc, cond, oc) && as_opnd(s, s.sa, x, ox) &&
        as_opnd(s, s.sb, y, oy)) {
        const size_t total = (size_t)s.total;
        // a floating condition holds unless it is +0 or -0; integers and bool unless they are 0
        const uint32_t mask = dtype_is_floating(dtype_cond) ? (csz == 4 ? 0x7fffffffu : 0x7fffu) : 0xffffffffu;
        const bool fc = oc.mode == OPND_FLAT, fx = ox.mode == OPND_FLAT, fy = oy.mode == OPND_FLAT;
        const bool nt = esz == 4 && streams(total * (size_t)(csz * fc + esz * (fx + fy + 1)), fc + fx + fy,
                                            {fc ? cond : nullptr, fx ? x : nullptr, fy ? y : nullptr, out});
        auto go = [&](auto E, auto C, auto N) {
            constexpr int ES = decltype(E)::value, CS = decltype(C)::value;
            k_where_vec<ES, CS, decltype(N)::value><<<grid_for(s.total, 16 / ES), 256, 0, st_>>>(oc, ox, oy, out, mask,
                                                                                              total, opnd_cols(s));
        };
        auto pick = [&](auto E, auto C) {
            if constexpr (decltype(E)::value == 4) {
                if (nt) return go(E, C, std::true_type{});
            }
            go(E, C, std::false_type{});
        };
        auto by_cond = [&](auto E) {
            if (csz == 1) pick(E, std::integral_constant<int, 1>{});
            else if (csz == 2) pick(E, std::integral_constant<int, 2>{});
            else pick(E, std::integral_constant<int, 4>{});
        };
        if (esz == 2) by_cond(std::integral_constant<int, 2>{});
        else by_cond(std::integral_constant<int, 4>{});
    } else if (to32(s, s32))
        k_where<EwShape32><<<grid_for(s.total), 256, 0, st_>>>(cond, dtype_cond, x, y, (int)dtype_size(dtype_xy), out,
                                                               s32);
    else
        k_where<EwShape><<<grid_for(s.total), 256, 0, st_>>>(cond, dtype_cond, x, y, (int)dtype_size(dtype_xy), out, s);
    PT_LAUNCH_CHECK("where");
    counters().elementwise_calls++;
    return PT_OK;
}

pt_status pt_fill(void *out, int dtype, size_t n, const pt_scalar_t *value, pt_stream_t stream)
{
    PT_TRY(ensure_init());
    if (!dtype_valid(dtype) || !value) return fail(PT_ERR_INVALID, "fill: bad arguments");
    if (!n) return PT_OK;
    uint64_t bits = 0;
    double d = scalar_as_double(value);
    long long iv = scalar_as_i64(value);
    switch (dtype) {
    case PT_FLOAT32: { float f = (float)d; memcpy(&bits, &f, 4); break; }
    case PT_FLOAT64: memcpy(&bits, &d, 8); break;
    case PT_FLOAT16: { _Float16 h = (_Float16)(float)d; uint16_t u; memcpy(&u, &h, 2); bits = u; break; }
    case PT_BFLOAT16: {
        float f = (float)d;
        uint32_t u;
        memcpy(&u, &f, 4);
        bits = ((u & 0x7f800000u) == 0x7f800000u && (u & 0x7fffffu)) ? ((u >> 16) | 0x40u)
                                                                       : ((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
        break;
    }
    case PT_BOOL: bits = d != 0.0; break;
    default: bits = dtype_is_floating(value->dtype) ? (uint64_t)(long long)d : (uint64_t)iv; break;
    }
    k_fill<<<grid_for((long long)n), 256, 0, stream_of(stream)>>>(out, (int)dtype_size(dtype), (long long)n, bits);
    PT_LAUNCH_CHECK("fill");
    return PT_OK;
}

}  // extern "C"
