// One generic kernel per PTIR op family: the executor's "fusion off" path and the fallback for
// every instruction no fused kernel claims.  Semantics follow the reference interpreter
// (crates/gpt-rs-backend-ref-cpu/src/cpu.rs) and docs/backend.md; integer / index ops are
// bit-exact, float ops compute in f32 and round once to the output dtype.
#include <cstring>

#include <mutex>

#include <algorithm>

#include "kernels.hpp"
#include "device_utils.hpp"

namespace gptrs {
namespace k {

static inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
static inline unsigned grid_for(int64_t n, int block, int64_t cap = 1 << 20) {
    int64_t g = cdiv(n, block);
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (unsigned)g;
}

// ------------------------------------------------------------------------------ strided copy
template <typename T>
__device__ __forceinline__ void copy_strided_one(T* __restrict__ dst, const T* __restrict__ src, const CopyDesc& d,
                                                 const int32_t* __restrict__ starts) {
    int64_t dyn_off = 0;
    if (d.dyn) {
        for (int i = 0; i < d.dyn_rank; ++i) {
            int64_t s = starts[i];
            s = s < 0 ? 0 : s;
            s = s > d.dyn_max[i] ? d.dyn_max[i] : s;
            dyn_off += s * d.dyn_stride[i];
        }
    }
    const int64_t src_base = d.src_off + (d.dyn == 1 ? dyn_off : 0);
    const int64_t dst_base = d.dst_off + (d.dyn == 2 ? dyn_off : 0);
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < d.total;
         idx += (int64_t)gridDim.x * blockDim.x) {
        int64_t rem = idx, so = src_base, dof = dst_base;
#pragma unroll
        for (int i = kMaxRank - 1; i >= 0; --i) {
            if (i < d.rank) {
                const int64_t c = rem % d.dims[i];
                rem /= d.dims[i];
                so += c * d.src_stride[i];
                dof += c * d.dst_stride[i];
            }
        }
        dst[dof] = src[so];
    }
}
template <typename T>
__global__ void copy_strided_kernel(T* __restrict__ dst, const T* __restrict__ src, CopyDesc d, const int32_t* __restrict__ starts) {
    copy_strided_one(dst, src, d, starts);
}
// grid (pieces, pairs).  Caches that outgrow their capacity are copied tensor by tensor of one shape, 24 for GPT-2 small and 416 for 8 sequences of 26 layers: a launch
// each is 2 to 4 us for 50 KB, and a program each 15 us of the host.  A call of 6 tokens that outgrows its caches once, 8 sequences of GPT-2 small: 7.4 -> 4.2 ms, one
// sequence 3.1 -> 2.5.
template <typename T>
__global__ void copy_strided_pairs_kernel(CopyPairs pairs, CopyDesc d, const int32_t* __restrict__ starts) {
    copy_strided_one((T*)pairs.dst[blockIdx.y], (const T*)pairs.src[blockIdx.y], d, starts);
}
void copy_strided_pairs(hipStream_t s, const CopyPairs& pairs, int count, int elem_size, const CopyDesc& d, const int32_t* starts) {
    if (d.total <= 0 || count <= 0) return;
    const dim3 grid(grid_for(d.total, 256, 4096), (unsigned)count);
    switch (elem_size) {
        case 1: copy_strided_pairs_kernel<uint8_t><<<grid, 256, 0, s>>>(pairs, d, starts); break;
        case 2: copy_strided_pairs_kernel<uint16_t><<<grid, 256, 0, s>>>(pairs, d, starts); break;
        case 4: copy_strided_pairs_kernel<uint32_t><<<grid, 256, 0, s>>>(pairs, d, starts); break;
        case 8: copy_strided_pairs_kernel<uint64_t><<<grid, 256, 0, s>>>(pairs, d, starts); break;
        case 16: copy_strided_pairs_kernel<uint4><<<grid, 256, 0, s>>>(pairs, d, starts); break;
        default: break;
    }
}

void copy_strided(hipStream_t s, void* dst, const void* src, int elem_size, const CopyDesc& d, const int32_t* starts) {
    if (d.total <= 0) return;
    const int block = 256;
    const unsigned grid = grid_for(d.total, block, 65536);
    switch (elem_size) {
        case 1: copy_strided_kernel<uint8_t><<<grid, block, 0, s>>>((uint8_t*)dst, (const uint8_t*)src, d, starts); break;
        case 2: copy_strided_kernel<uint16_t><<<grid, block, 0, s>>>((uint16_t*)dst, (const uint16_t*)src, d, starts); break;
        case 4: copy_strided_kernel<uint32_t><<<grid, block, 0, s>>>((uint32_t*)dst, (const uint32_t*)src, d, starts); break;
        case 8: copy_strided_kernel<uint64_t><<<grid, block, 0, s>>>((uint64_t*)dst, (const uint64_t*)src, d, starts); break;
        case 16: copy_strided_kernel<uint4><<<grid, block, 0, s>>>((uint4*)dst, (const uint4*)src, d, starts); break;
        default: break;
    }
}

__global__ void store_small_kernel(SmallBatch b) {
    const int e = blockIdx.x, i = threadIdx.x;
    if (i < b.bytes[e]) b.dst[e][i] = ((const uint8_t*)b.payload[e].w)[i];
}
void store_small(hipStream_t s, const SmallBatch& b, int count) {
    if (count > 0) store_small_kernel<<<count, 256, 0, s>>>(b);
}

__device__ __forceinline__ void fill_zero_range(uint8_t* dst, size_t nbytes, int64_t first, int64_t step) {
    uint4* d16 = reinterpret_cast<uint4*>(dst);
    const int64_t n16 = (int64_t)(nbytes / 16);
    for (int64_t i = first; i < n16; i += step) d16[i] = make_uint4(0, 0, 0, 0);
    const int64_t tail = (int64_t)(nbytes % 16);
    if (first < tail) dst[n16 * 16 + first] = 0;
}
__global__ void fill_zero_kernel(uint8_t* dst, size_t nbytes) {
    fill_zero_range(dst, nbytes, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, (int64_t)gridDim.x * blockDim.x);
}
void fill_zero(hipStream_t s, void* dst, size_t nbytes) {
    if (!nbytes) return;
    fill_zero_kernel<<<grid_for(nbytes / 16 ? (int64_t)(nbytes / 16) : 1, 256, 8192), 256, 0, s>>>((uint8_t*)dst, nbytes);
}
// Many fresh tensors in one launch (grid.y = tensor): a prompt of 16 sequences through 12 layers starts from 384 zeroed caches,
// 2.2 us each as launches of their own and more than that for the host to queue them.
__global__ void fill_zero_many_kernel(ZeroBatch b) {
    fill_zero_range(b.dst[blockIdx.y], b.bytes[blockIdx.y], (int64_t)blockIdx.x * blockDim.x + threadIdx.x, (int64_t)gridDim.x * blockDim.x);
}
void fill_zero_many(hipStream_t s, const ZeroBatch& b, int count) {
    if (count <= 0) return;
    size_t most = 0;
    for (int i = 0; i < count; ++i) most = b.bytes[i] > most ? b.bytes[i] : most;
    const int64_t blocks = (int64_t)(most / 16 + 1023) / 1024;   // four stores a thread
    fill_zero_many_kernel<<<dim3((unsigned)(blocks < 1 ? 1 : blocks > 1024 ? 1024 : blocks), (unsigned)count), 256, 0, s>>>(b);
}

// ------------------------------------------------------------------------------ elementwise
template <typename T> __device__ __forceinline__ float ldf(const T* p, int64_t i);
template <> __device__ __forceinline__ float ldf<float>(const float* p, int64_t i) { return p[i]; }
template <> __device__ __forceinline__ float ldf<bf16_t>(const bf16_t* p, int64_t i) { return bf16_to_f32(p[i]); }
template <typename T> __device__ __forceinline__ void stf(T* p, int64_t i, float v);
template <> __device__ __forceinline__ void stf<float>(float* p, int64_t i, float v) { p[i] = v; }
template <> __device__ __forceinline__ void stf<bf16_t>(bf16_t* p, int64_t i, float v) { p[i] = f32_to_bf16(v); }

__device__ __forceinline__ float apply_unary(int op, float v) {
    switch (op) {  // cpu.rs:1704-1714
        case 0: return -v;
        case 1: return fabsf(v);
        case 2: return expf(v);
        case 3: return logf(v);
        case 4: return tanhf(v);
        case 5: return erff(v);
        case 6: return 1.0f / sqrtf(v);
        default: return 1.0f / v;
    }
}
__device__ __forceinline__ float apply_binary(int op, float a, float b) {
    switch (op) {  // cpu.rs:1669-1677; Rust max/min return the non-NaN operand == fmaxf/fminf
        case 0: return a + b;
        case 1: return a - b;
        case 2: return a * b;
        case 3: return a / b;
        case 4: return fmaxf(a, b);
        default: return fminf(a, b);
    }
}

template <typename T>
__global__ void unary_kernel(int op, const T* __restrict__ x, T* __restrict__ y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        stf(y, i, apply_unary(op, ldf(x, i)));
}
template <typename T>
__global__ void binary_kernel(int op, const T* __restrict__ a, const T* __restrict__ b, T* __restrict__ y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        stf(y, i, apply_binary(op, ldf(a, i), ldf(b, i)));
}
template <typename T>
__global__ void binary_scalar_kernel(int op, const T* __restrict__ a, float b, T* __restrict__ y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        stf(y, i, apply_binary(op, ldf(a, i), b));
}

void unary(hipStream_t s, int dtype, int op, const void* x, void* y, int64_t n) {
    if (n <= 0) return;
    if (dtype == 0) unary_kernel<float><<<grid_for(n, 256, 16384), 256, 0, s>>>(op, (const float*)x, (float*)y, n);
    else unary_kernel<bf16_t><<<grid_for(n, 256, 16384), 256, 0, s>>>(op, (const bf16_t*)x, (bf16_t*)y, n);
}
void binary(hipStream_t s, int dtype, int op, const void* a, const void* b, void* y, int64_t n) {
    if (n <= 0) return;
    if (dtype == 0) binary_kernel<float><<<grid_for(n, 256, 16384), 256, 0, s>>>(op, (const float*)a, (const float*)b, (float*)y, n);
    else binary_kernel<bf16_t><<<grid_for(n, 256, 16384), 256, 0, s>>>(op, (const bf16_t*)a, (const bf16_t*)b, (bf16_t*)y, n);
}
void binary_scalar(hipStream_t s, int dtype, int op, const void* a, float b, void* y, int64_t n) {
    if (n <= 0) return;
    if (dtype == 0) binary_scalar_kernel<float><<<grid_for(n, 256, 16384), 256, 0, s>>>(op, (const float*)a, b, (float*)y, n);
    else binary_scalar_kernel<bf16_t><<<grid_for(n, 256, 16384), 256, 0, s>>>(op, (const bf16_t*)a, b, (bf16_t*)y, n);
}

template <typename T>
__device__ __forceinline__ bool cmp_apply(int op, T x, T y) {
    switch (op) {  // cpu.rs:2254-2261; float NaN rules are IEEE (docs/backend.md:199-202)
        case 0: return x < y;
        case 1: return x <= y;
        case 2: return x == y;
        case 3: return x >= y;
        case 4: return x > y;
        default: return x != y;
    }
}
__global__ void compare_i32_kernel(int op, const int32_t* a, const int32_t* b, uint8_t* y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = cmp_apply<int32_t>(op, a[i], b[i]) ? 1 : 0;
}
template <typename T>
__global__ void compare_f_kernel(int op, const T* a, const T* b, uint8_t* y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = cmp_apply<float>(op, ldf(a, i), ldf(b, i)) ? 1 : 0;
}
void compare(hipStream_t s, int dtype, int op, const void* a, const void* b, uint8_t* y, int64_t n) {
    if (n <= 0) return;
    const unsigned g = grid_for(n, 256, 16384);
    if (dtype == 3) compare_i32_kernel<<<g, 256, 0, s>>>(op, (const int32_t*)a, (const int32_t*)b, y, n);
    else if (dtype == 0) compare_f_kernel<float><<<g, 256, 0, s>>>(op, (const float*)a, (const float*)b, y, n);
    else compare_f_kernel<bf16_t><<<g, 256, 0, s>>>(op, (const bf16_t*)a, (const bf16_t*)b, y, n);
}

template <typename T>
__global__ void select_kernel(const uint8_t* p, const T* t, const T* f, T* y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = p[i] != 0 ? t[i] : f[i];
}
void select(hipStream_t s, int elem_size, const uint8_t* p, const void* t, const void* f, void* y, int64_t n) {
    if (n <= 0) return;
    const unsigned g = grid_for(n, 256, 16384);
    if (elem_size == 4) select_kernel<uint32_t><<<g, 256, 0, s>>>(p, (const uint32_t*)t, (const uint32_t*)f, (uint32_t*)y, n);
    else if (elem_size == 2) select_kernel<uint16_t><<<g, 256, 0, s>>>(p, (const uint16_t*)t, (const uint16_t*)f, (uint16_t*)y, n);
    else select_kernel<uint8_t><<<g, 256, 0, s>>>(p, (const uint8_t*)t, (const uint8_t*)f, (uint8_t*)y, n);
}

// cast (docs/backend.md:96-102; cpu.rs:1472-1583).  Source value is first widened to
// (is_int ? int32 : float); destination rules: float->int trunc + saturate, NaN -> 0;
// ->i1 is (x != 0); int->float nearest; float->float RNE.
__device__ __forceinline__ int32_t f32_to_i32_sat(float v) {
    if (v != v) return 0;
    const float t = truncf(v);
    if (t >= 2147483648.0f) return 2147483647;
    if (t <= -2147483648.0f) return (int32_t)0x80000000;
    return (int32_t)t;
}
__global__ void cast_kernel(int sd, int dd, const void* x, void* y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        float fv = 0.f;
        int32_t iv = 0;
        bool is_int = false;
        switch (sd) {
            case 0: fv = ((const float*)x)[i]; break;
            case 2: fv = bf16_to_f32(((const bf16_t*)x)[i]); break;
            case 3: iv = ((const int32_t*)x)[i]; is_int = true; break;
            case 4: iv = ((const uint8_t*)x)[i] != 0 ? 1 : 0; is_int = true; break;
            case 5: iv = ((const int8_t*)x)[i]; is_int = true; break;
            default: iv = ((const uint8_t*)x)[i]; is_int = true; break;
        }
        switch (dd) {
            case 0: ((float*)y)[i] = is_int ? (float)iv : fv; break;
            case 2: ((bf16_t*)y)[i] = f32_to_bf16(is_int ? (float)iv : fv); break;
            case 3: ((int32_t*)y)[i] = is_int ? iv : f32_to_i32_sat(fv); break;
            case 4: ((uint8_t*)y)[i] = is_int ? (iv != 0) : (fv != 0.0f); break;
            case 5: {
                int32_t v = is_int ? iv : f32_to_i32_sat(fv);
                ((int8_t*)y)[i] = (int8_t)(v < -128 ? -128 : (v > 127 ? 127 : v));
                break;
            }
            default: {
                int32_t v = is_int ? iv : f32_to_i32_sat(fv);
                ((uint8_t*)y)[i] = (uint8_t)(v < 0 ? 0 : (v > 255 ? 255 : v));
                break;
            }
        }
    }
}
void cast(hipStream_t s, int sd, int dd, const void* x, void* y, int64_t n) {
    if (n <= 0) return;
    cast_kernel<<<grid_for(n, 256, 16384), 256, 0, s>>>(sd, dd, x, y, n);
}

__global__ void iota_kernel(int32_t* y, int64_t total, int64_t axis_len, int64_t inner) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = (int32_t)((i / inner) % axis_len);
}
void iota(hipStream_t s, int32_t* y, int64_t outer, int64_t axis_len, int64_t inner) {
    const int64_t total = outer * axis_len * inner;
    if (total <= 0) return;
    iota_kernel<<<grid_for(total, 256, 16384), 256, 0, s>>>(y, total, axis_len, inner);
}

// ------------------------------------------------------------------------------ reduce
__device__ __forceinline__ float red_id(int kind) { return kind == 0 ? 0.f : (kind == 1 ? -INFINITY : INFINITY); }
__device__ __forceinline__ float red_op(int kind, float a, float b) {
    return kind == 0 ? a + b : (kind == 1 ? fmaxf(a, b) : fminf(a, b));
}

// inner == 1: one 256-thread block per row, wave64 shuffle tree then LDS across waves.
template <typename T>
__global__ void reduce_rows_kernel(int kind, const T* __restrict__ x, T* __restrict__ y, int64_t n) {
    __shared__ float part[4];
    const T* row = x + (int64_t)blockIdx.x * n;
    float acc = red_id(kind);
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) acc = red_op(kind, acc, ldf(row, i));
    for (int off = 32; off > 0; off >>= 1) acc = red_op(kind, acc, __shfl_down(acc, off, 64));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        float r = part[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = red_op(kind, r, part[w]);
        stf(y, (int64_t)blockIdx.x, r);
    }
}
// inner > 1: one thread per (outer, inner) column, sequential over the axis (coalesced across inner).
template <typename T>
__global__ void reduce_cols_kernel(int kind, const T* __restrict__ x, T* __restrict__ y, int64_t outer,
                                   int64_t axis_len, int64_t inner) {
    const int64_t total = outer * inner;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t o = idx / inner, i = idx % inner;
        const T* base = x + o * axis_len * inner + i;
        float acc = red_id(kind);
        for (int64_t a = 0; a < axis_len; ++a) acc = red_op(kind, acc, ldf(base, a * inner));
        stf(y, idx, acc);
    }
}
void reduce(hipStream_t s, int dtype, int kind, const void* x, void* y, int64_t outer, int64_t axis_len, int64_t inner) {
    if (outer * inner <= 0) return;
    if (inner == 1) {
        if (dtype == 0) reduce_rows_kernel<float><<<(unsigned)outer, 256, 0, s>>>(kind, (const float*)x, (float*)y, axis_len);
        else reduce_rows_kernel<bf16_t><<<(unsigned)outer, 256, 0, s>>>(kind, (const bf16_t*)x, (bf16_t*)y, axis_len);
    } else {
        const unsigned g = grid_for(outer * inner, 256, 16384);
        if (dtype == 0) reduce_cols_kernel<float><<<g, 256, 0, s>>>(kind, (const float*)x, (float*)y, outer, axis_len, inner);
        else reduce_cols_kernel<bf16_t><<<g, 256, 0, s>>>(kind, (const bf16_t*)x, (bf16_t*)y, outer, axis_len, inner);
    }
}

// ------------------------------------------------------------------------------ take
template <typename T> struct TakeRows { const T* table; const int32_t* idx; int64_t rows; };
template <typename T>
__global__ void take_kernel(const T* __restrict__ table, const int32_t* __restrict__ idx, T* __restrict__ y,
                            int64_t vocab, int64_t inner, int* err_flag) {
    const int64_t r = blockIdx.x;
    const int32_t id = idx[r];
    const bool ok = id >= 0 && (int64_t)id < vocab;
    if (!ok && threadIdx.x == 0) atomicExch(err_flag, 1);
    const T* src = table + (int64_t)(ok ? id : 0) * inner;
    T* dst = y + r * inner;
    for (int64_t i = threadIdx.x; i < inner; i += blockDim.x) dst[i] = ok ? src[i] : T{};
}
void take(hipStream_t s, int elem_size, const void* table, const int32_t* idx, void* y, int64_t n_idx, int64_t vocab,
          int64_t inner, int* err_flag) {
    if (n_idx <= 0 || inner <= 0) return;
    // widen to 16/8/4-byte words when the row allows it
    const size_t row_bytes = (size_t)inner * elem_size;
    const bool a16 = row_bytes % 16 == 0 && ((uintptr_t)table % 16 == 0) && ((uintptr_t)y % 16 == 0);
    if (a16) {
        take_kernel<uint4><<<(unsigned)n_idx, 256, 0, s>>>((const uint4*)table, idx, (uint4*)y, vocab, (int64_t)(row_bytes / 16), err_flag);
    } else if (elem_size == 4) {
        take_kernel<uint32_t><<<(unsigned)n_idx, 256, 0, s>>>((const uint32_t*)table, idx, (uint32_t*)y, vocab, inner, err_flag);
    } else if (elem_size == 2) {
        take_kernel<uint16_t><<<(unsigned)n_idx, 256, 0, s>>>((const uint16_t*)table, idx, (uint16_t*)y, vocab, inner, err_flag);
    } else {
        take_kernel<uint8_t><<<(unsigned)n_idx, 256, 0, s>>>((const uint8_t*)table, idx, (uint8_t*)y, vocab, inner, err_flag);
    }
}

// The sum of two gathered rows (token and position embeddings) without the rows in between: one launch of 5 us before a decode step where two gathers and an
// addition took 14.  V: values at a time (16 bytes where rows and addresses allow it).  As take_kernel, an index outside its table counts as
// a row of zeros and raises the flag.
template <typename T, int V>
__global__ __launch_bounds__(256) void take_add_kernel(TakeRows<T> a, TakeRows<T> b, T* __restrict__ y, int64_t inner, int* err_flag) {
    typedef T vec __attribute__((ext_vector_type(V)));
    const int64_t r = blockIdx.x;
    const int32_t ia = a.idx[r], ib = b.idx[r];
    const bool oka = ia >= 0 && (int64_t)ia < a.rows, okb = ib >= 0 && (int64_t)ib < b.rows;
    if ((!oka || !okb) && threadIdx.x == 0) atomicExch(err_flag, 1);
    const T *ra = a.table + (int64_t)(oka ? ia : 0) * inner, *rb = b.table + (int64_t)(okb ? ib : 0) * inner;
    for (int64_t i = (int64_t)threadIdx.x * V; i < inner; i += 256 * V) {
        alignas(16) T u[V], v[V];
        *reinterpret_cast<vec*>(u) = *reinterpret_cast<const vec*>(ra + i);
        *reinterpret_cast<vec*>(v) = *reinterpret_cast<const vec*>(rb + i);
#pragma unroll
        for (int e = 0; e < V; ++e) stf(u, e, (oka ? ldf(u, e) : 0.f) + (okb ? ldf(v, e) : 0.f));
        *reinterpret_cast<vec*>(y + r * inner + i) = *reinterpret_cast<const vec*>(u);
    }
}
void take_add(hipStream_t s, int dtype, const void* ta, const int32_t* ia, int64_t rows_a, const void* tb, const int32_t* ib, int64_t rows_b, void* y, int64_t n_idx, int64_t inner,
              int* err_flag) {
    if (n_idx <= 0 || inner <= 0) return;
    auto go = [&](auto type) {
        typedef decltype(type) T;
        constexpr int V = 16 / sizeof(T);
        const TakeRows<T> a{(const T*)ta, ia, rows_a}, b{(const T*)tb, ib, rows_b};
        const bool wide = inner % V == 0 && (((uintptr_t)ta | (uintptr_t)tb | (uintptr_t)y) & 15) == 0;
        if (wide) take_add_kernel<T, V><<<(unsigned)n_idx, 256, 0, s>>>(a, b, (T*)y, inner, err_flag);
        else take_add_kernel<T, 1><<<(unsigned)n_idx, 256, 0, s>>>(a, b, (T*)y, inner, err_flag);
    };
    if (dtype == 0) go(float());
    else go(bf16_t());
}

// ------------------------------------------------------------------------------ generic dot
// 32x32 output tile per 256-thread block, K stepped by 32 through LDS; arbitrary operand strides.
// Correctness path for dots no tuned kernel claims (attention score / PV contractions in prefill,
// odd shapes).  Accumulates in f32 in k order within a tile.
template <typename T, typename TO>
__global__ void dot_generic_kernel(const T* __restrict__ a, const T* __restrict__ b, TO* __restrict__ c, DotDesc d) {
    __shared__ float As[32][33];
    __shared__ float Bs[32][33];
    const int64_t bi = blockIdx.z;
    const int64_t m0 = (int64_t)blockIdx.y * 32, n0 = (int64_t)blockIdx.x * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // ty in 0..7
    const T* ab = a + bi * d.a_sb;
    const T* bb = b + bi * d.b_sb;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int64_t k0 = 0; k0 < d.k; k0 += 32) {
        for (int r = ty; r < 32; r += 8) {
            const int64_t m = m0 + r, kk = k0 + tx;
            As[r][tx] = (m < d.m && kk < d.k) ? ldf(ab, m * d.a_sm + kk * d.a_sk) : 0.f;
            const int64_t kr = k0 + r, n = n0 + tx;
            Bs[r][tx] = (kr < d.k && n < d.n) ? ldf(bb, kr * d.b_sk + n * d.b_sn) : 0.f;
        }
        __syncthreads();
#pragma unroll 8
        for (int kk = 0; kk < 32; ++kk) {
            const float bv = Bs[kk][tx];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] += As[ty + 8 * j][kk] * bv;
        }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t m = m0 + ty + 8 * j, n = n0 + tx;
        if (m < d.m && n < d.n) stf(c, bi * d.c_sb + m * d.c_sm + n, acc[j]);
    }
}
void dot_generic(hipStream_t s, int dtype, const void* a, const void* b, void* c, const DotDesc& d, bool out_f32) {
    if (d.batch * d.m * d.n <= 0) return;
    dim3 grid((unsigned)cdiv(d.n, 32), (unsigned)cdiv(d.m, 32), (unsigned)d.batch);
    if (dtype == 0) dot_generic_kernel<float, float><<<grid, 256, 0, s>>>((const float*)a, (const float*)b, (float*)c, d);
    else if (out_f32) dot_generic_kernel<bf16_t, float><<<grid, 256, 0, s>>>((const bf16_t*)a, (const bf16_t*)b, (float*)c, d);
    else dot_generic_kernel<bf16_t, bf16_t><<<grid, 256, 0, s>>>((const bf16_t*)a, (const bf16_t*)b, (bf16_t*)c, d);
}

// ------------------------------------------------------------------------------ sampling
// Greedy token of every row of logits [gridDim.y, n], in one launch: a workgroup leaves the (value, smallest index) of its share, and the one
// that draws a row's last ticket combines them.  Ties -> smallest index (docs/backend.md:270).  The token goes where the next step reads it
// (out64, one row, or out32) and, with `host`, straight into the pinned slot that the caller waits for, with the device's error flags beside
// it: host[0] the token of a single row, host[1] the flags, from host + 2 on the tokens of several.  Between two decode steps
// that is one launch of 6 us where two stages and two copies took 19.  A ticket is zero before and after every launch.
template <typename T, int VEC>
__global__ __launch_bounds__(256) void argmax_kernel(const T* __restrict__ logits, int64_t n, float* pv, int32_t* pi, unsigned* tickets, int64_t* out64, int32_t* out32,
                                                     int64_t* host, const int64_t* err_flags) {
    constexpr int U = 4;
    __shared__ float sv[4];
    __shared__ int32_t si[4];
    __shared__ unsigned ticket;
    const T* row = logits + (int64_t)blockIdx.y * n;
    float best = -INFINITY;
    int32_t bidx = 0x7fffffff;
    auto better = [&](float v, int32_t i) { if (v > best || (v == best && i < bidx)) { best = v; bidx = i; } };
    auto over_wave = [&]() {
        for (int off = 32; off > 0; off >>= 1) {
            const float ov = __shfl_down(best, off, 64);
            const int32_t oi = __shfl_down(bidx, off, 64);
            better(ov, oi);
        }
    };
    typedef T vec_t __attribute__((ext_vector_type(VEC)));
    const int64_t stride = (int64_t)gridDim.x * 256, whole = n / VEC;
    for (int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x; i0 < whole; i0 += U * stride) {
        vec_t v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = reinterpret_cast<const vec_t*>(row)[i0 + u * stride < whole ? i0 + u * stride : i0];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const T x = v[u][e];
                better(ldf(&x, 0), (int32_t)((i0 + u * stride < whole ? i0 + u * stride : i0) * VEC + e));
            }
    }
    if (blockIdx.x == 0 && threadIdx.x < n - whole * VEC) better(ldf(row, whole * VEC + threadIdx.x), (int32_t)(whole * VEC + threadIdx.x));
    over_wave();
    if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = best; si[threadIdx.x >> 6] = bidx; }
    __syncthreads();
    const int part = blockIdx.y * gridDim.x;
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w) better(sv[w], si[w]);
        __hip_atomic_store(pv + part + blockIdx.x, best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // (other XCDs read them)
        __hip_atomic_store(pi + part + blockIdx.x, bidx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_waitcnt(0x0F70);                                                             // vmcnt(0)
        asm volatile("" ::: "memory");
        ticket = __hip_atomic_fetch_add(tickets + blockIdx.y, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (ticket != gridDim.x - 1 || threadIdx.x >= 64) return;
    best = -INFINITY;
    bidx = 0x7fffffff;
    for (int i = threadIdx.x; i < (int)gridDim.x; i += 64)
        better(__hip_atomic_load(pv + part + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), __hip_atomic_load(pi + part + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    over_wave();
    if (threadIdx.x != 0) return;
    const int32_t token = bidx == 0x7fffffff ? 0 : bidx;
    if (out64) *out64 = token;
    if (out32) out32[blockIdx.y] = token;
    if (host) {
        if (out64) __hip_atomic_store(host, (int64_t)token, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (out32) __hip_atomic_store(reinterpret_cast<int32_t*>(host + 2) + blockIdx.y, token, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (blockIdx.y == 0) __hip_atomic_store(host + 1, *err_flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __hip_atomic_store(tickets + blockIdx.y, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
void argmax_tokens(hipStream_t s, int dtype, const void* logits, int64_t rows, int64_t vocab, int64_t* out64, int32_t* out32, const ArgmaxScratch& w, int64_t* host) {
    if (rows <= 0) return;
    // Up to 256 workgroups of four loads of a value each; beyond, 16 bytes a load and 256 workgroups, since all of them meet at tickets that share a line (us: 8 rows
    // of 131072 by 1024 workgroups 16.9, so 9.0; one row of 50257 5.7, with 16 bytes a load in 50 workgroups 6.1, in 13 5.9)
    const int vec = dtype == 0 ? 4 : 8;
    int64_t nb = cdiv(vocab, 256 * 4);
    const bool wide = rows * nb > 256 && ((uintptr_t)logits & 15u) == 0 && (rows == 1 || vocab % vec == 0);
    if (wide) nb = std::min<int64_t>(cdiv(vocab, 256 * vec), std::max<int64_t>(256 / rows, 1));
    if (nb > w.parts / rows) nb = w.parts / rows;
    if (nb < 1) nb = 1;
    const dim3 grid((unsigned)nb, (unsigned)rows);
    auto go = [&](auto kernel, auto* x) { kernel<<<grid, 256, 0, s>>>(x, vocab, w.val, w.idx, w.tickets, out64, out32, host, w.err_flags); };
    if (dtype == 0) { if (wide) go(argmax_kernel<float, 4>, (const float*)logits); else go(argmax_kernel<float, 1>, (const float*)logits); }
    else if (wide) go(argmax_kernel<bf16_t, 8>, (const bf16_t*)logits);
    else go(argmax_kernel<bf16_t, 1>, (const bf16_t*)logits);
}

// The same in two stages without tickets, for callers that may overlap (argmax_rows_noalloc): per-block partials, then one block per row; out[r] as si32.
template <typename T>
__global__ void argmax_rows_stage1(const T* __restrict__ logits, int64_t n, float* pv, int32_t* pi) {
    __shared__ float sv[4];
    __shared__ int32_t si[4];
    const T* row = logits + (int64_t)blockIdx.y * n;
    float best = -INFINITY;
    int32_t bidx = 0x7fffffff;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float v = ldf(row, i);
        if (v > best || (v == best && (int32_t)i < bidx)) { best = v; bidx = (int32_t)i; }
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_down(best, off, 64);
        const int32_t oi = __shfl_down(bidx, off, 64);
        if (ov > best || (ov == best && oi < bidx)) { best = ov; bidx = oi; }
    }
    if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = best; si[threadIdx.x >> 6] = bidx; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w)
            if (sv[w] > best || (sv[w] == best && si[w] < bidx)) { best = sv[w]; bidx = si[w]; }
        pv[blockIdx.y * gridDim.x + blockIdx.x] = best;
        pi[blockIdx.y * gridDim.x + blockIdx.x] = bidx;
    }
}
__global__ void argmax_rows_stage2(const float* pv, const int32_t* pi, int nparts, int32_t* out) {
    float best = -INFINITY;
    int32_t bidx = 0x7fffffff;
    for (int i = threadIdx.x; i < nparts; i += 64) {
        const float v = pv[blockIdx.x * nparts + i];
        const int32_t id = pi[blockIdx.x * nparts + i];
        if (v > best || (v == best && id < bidx)) { best = v; bidx = id; }
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_down(best, off, 64);
        const int32_t oi = __shfl_down(bidx, off, 64);
        if (ov > best || (ov == best && oi < bidx)) { best = ov; bidx = oi; }
    }
    if (threadIdx.x == 0) out[blockIdx.x] = bidx == 0x7fffffff ? 0 : bidx;
}
void argmax_rows(hipStream_t s, int dtype, const void* logits, int64_t rows, int64_t vocab, int32_t* out, float* scratch_val,
                 int32_t* scratch_idx, int scratch_cap) {
    if (rows <= 0) return;
    int nb = (int)cdiv(vocab, 256 * 8);
    if (nb > scratch_cap / (int)rows) nb = scratch_cap / (int)rows;
    if (nb < 1) nb = 1;
    const dim3 grid((unsigned)nb, (unsigned)rows);
    if (dtype == 0) argmax_rows_stage1<float><<<grid, 256, 0, s>>>((const float*)logits, vocab, scratch_val, scratch_idx);
    else argmax_rows_stage1<bf16_t><<<grid, 256, 0, s>>>((const bf16_t*)logits, vocab, scratch_val, scratch_idx);
    argmax_rows_stage2<<<(unsigned)rows, 64, 0, s>>>(scratch_val, scratch_idx, nb, out);
}

// The same two stages for callers that must not allocate: the per-block partial maxima (value, index) live in a
// file-scope device array instead of a buffer the backend allocated.  Each GPU holds its own copy of the array at its
// own address until the process ends; argmax_noalloc_init() resolves that address once per device (with the device
// current), and the launcher hands it to the kernels as an ordinary pointer argument.  Stage 1 overwrites every
// partial that stage 2 reads, so nothing has to start at zero; two calls that overlap on one GPU (two streams) race
// on the array.
constexpr int kNoAllocPartials = 4096;   // rows * blocks per row
static __device__ __align__(256) unsigned char scratch[kNoAllocPartials * (sizeof(float) + sizeof(int32_t))];
constexpr int kNoAllocMaxDevices = 64;
static void* g_noalloc_ptr[kNoAllocMaxDevices] = {};
static std::mutex g_noalloc_mu;

hipError_t argmax_noalloc_init(int device) {
    if (device < 0 || device >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> g(g_noalloc_mu);
    if (g_noalloc_ptr[device]) return hipSuccess;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    // load the kernels' code now, so that the first call does not do it
    hipFuncAttributes fa{};
    (void)hipFuncGetAttributes(&fa, (const void*)argmax_rows_stage1<float>);
    (void)hipFuncGetAttributes(&fa, (const void*)argmax_rows_stage1<bf16_t>);
    (void)hipFuncGetAttributes(&fa, (const void*)argmax_rows_stage2);
    g_noalloc_ptr[device] = p;
    return hipSuccess;
}
int argmax_noalloc_max_rows() { return 64; }
bool argmax_rows_noalloc(hipStream_t s, int device, int dtype, const void* logits, int64_t rows, int64_t vocab, int32_t* out) {
    if (device < 0 || device >= kNoAllocMaxDevices || rows < 1 || rows > argmax_noalloc_max_rows()) return false;
    void* p = g_noalloc_ptr[device];   // the device address, never the array's name (a host-side stand-in)
    if (!p) return false;
    float* val = reinterpret_cast<float*>(p);
    int32_t* idx = reinterpret_cast<int32_t*>(reinterpret_cast<unsigned char*>(p) + kNoAllocPartials * sizeof(float));
    argmax_rows(s, dtype, logits, rows, vocab, out, val, idx, kNoAllocPartials);
    return true;
}

// Temperature sampling, single block: softmax(logits/T) then inverse CDF at u.  The running
// sum is taken in index order by one wave so the chosen token does not depend on launch shape.
// Temperature sampling as the reference's device path does it
// (crates/gpt-rs-backend-triton/src/kernels/sample_temperature_last_axis_f32.triton:24-72): Gumbel-max with a
// stateless per-index hash of (index ^ seed); the score of index i is logit_i / temperature - log(-log(u_i)), the
// token is the index of the largest score, the smallest index on ties.  seed = bits(random_u) * 747796405 +
// 2891336453 (runtime/sampling.rs:98-101).
__device__ __forceinline__ float gumbel_of(uint32_t idx, uint32_t seed) {
    uint32_t x = idx ^ seed;
    x ^= x >> 16;
    x *= 0x7FEB352Du;
    x ^= x >> 15;
    x *= 0x846CA68Bu;
    x ^= x >> 16;
    float u = ((float)x + 1.0f) * 2.3283064365386963e-10f;   // f32(1 / 4294967297) = 2^-32
    u = fmaxf(u, 1e-7f);
    u = fminf(u, 1.0f - 1e-7f);
    return -logf(-logf(u));
}
template <typename T>
__global__ void sample_temperature_kernel(const T* __restrict__ row, int64_t n, float inv_t, uint32_t seed, int64_t* out) {
    __shared__ float s_score[16];
    __shared__ int64_t s_idx[16];
    float best = -INFINITY;
    int64_t best_i = 0;
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
        const float sc = ldf(row, i) * inv_t + gumbel_of((uint32_t)i, seed);
        if (sc > best) { best = sc; best_i = i; }   // ascending i per thread: the first maximum stays
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float os = __shfl_down(best, off, 64);
        const int64_t oi = __shfl_down(best_i, off, 64);
        if (os > best || (os == best && oi < best_i)) { best = os; best_i = oi; }
    }
    if ((threadIdx.x & 63) == 0) { s_score[threadIdx.x >> 6] = best; s_idx[threadIdx.x >> 6] = best_i; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w)
            if (s_score[w] > best || (s_score[w] == best && s_idx[w] < best_i)) { best = s_score[w]; best_i = s_idx[w]; }
        *out = best_i;
    }
}
void sample_temperature_last_row(hipStream_t s, int dtype, const void* logits, int64_t rows, int64_t vocab,
                                 float temperature, float u, int64_t* out) {
    const size_t off = (size_t)(rows - 1) * vocab;
    const float inv_t = 1.0f / temperature;
    uint32_t bits;
    memcpy(&bits, &u, 4);
    const uint32_t seed = bits * 747796405u + 2891336453u;
    if (dtype == 0) sample_temperature_kernel<float><<<1, 1024, 0, s>>>((const float*)logits + off, vocab, inv_t, seed, out);
    else sample_temperature_kernel<bf16_t><<<1, 1024, 0, s>>>((const bf16_t*)logits + off, vocab, inv_t, seed, out);
}

}  // namespace k
}  // namespace gptrs
