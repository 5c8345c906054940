// Batched-decode linear layers (2 <= M <= 16 rows, bf16 or f32) on the matrix cores.
//
// With a handful of rows a linear layer is still one pass over the weights, i.e. bound by HBM, but the
// per-element work of a vector GEMV grows with M (M multiply-adds per weight element plus the activation reads)
// until the vector ALUs, not memory, set the pace.  One v_mfma_f32_16x16x32_bf16 multiplies 16 rows by a
// 32 x 16 block of W at a cost that does not depend on M, so the kernel below only has to stream W.
//
// Weights are read from a derived copy Ws[tile][K/8][16 columns][8 k] (tile = 16 output columns, or 12: skinny_cols): the 64 lanes of
// a wave fetch 32 consecutive k of the tile's columns as ONE contiguous KiB in exactly the B-operand layout
// (lane = 16 * k-group + column holds 8 consecutive k of its column).  A workgroup owns one tile; its 8 or 16 waves
// (skinny_plan) take the 32-k steps round-robin (so the workgroup reads consecutive KiB) and add their partial products
// through LDS.  The A operand (lane = 16 * k-group + row) comes straight from x, which is small and stays in L2.
// DUAL computes silu(x.W) * (x.W2) (ops/functional/activation.rs:141-162) from two weight copies.
// f32 takes the same route with 4 k per 16-byte lane word (Ws[tile][K/4][16 or 12][4], 16-k steps) on four
// v_mfma_f32_16x16x4_f32 per word.
//
// Weight-only quantised layers (skinny_gemm_quant_kernel<QF, DUAL>) stream the CODES: a lane's 16-byte word holds 16
// int8 codes (k = 64 S + 16 kg + 0..15 of its column: two MFMA steps) or 32 int4 codes (k = 128 Q + 32 kg + 0..31: four
// steps, exactly one scale group), stored biased (+128 / +8) so the unsigned-byte converts apply; the biased codes are
// exact in bf16 and go to the matrix cores as they are, and a second MFMA per step against a column of ones yields
// sum_k x[row, k], which takes the bias out again (x.(q + b) - b.sum x).  int8 scales (per column) are applied in the
// epilogue, int4 group scales when a group's sums are added to the running total.
//
// A layer with few tiles is split along K over gridDim.y workgroups per tile so that more of the chip streams: each writes its
// 16 x 16 partial sums to a workspace and takes a ticket; the workgroup that draws the last ticket of a tile adds the partials in split
// order (so the result does not depend on which one that is), applies the epilogue and resets the ticket for the next launch.
#include <algorithm>
#include <type_traits>

#include "kernels.hpp"
#include "device_utils.hpp"

namespace gptrs {
namespace k {

namespace {

typedef __bf16 bf16x8_s __attribute__((ext_vector_type(8)));
typedef float f32x4_s __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_s __attribute__((ext_vector_type(4)));

inline int64_t cdiv_s(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Element types: KPC = k per 16-byte lane word; a step of the K loop is 4 k-groups x KPC (32 k of bf16, 16 k of f32).
// f32 runs on v_mfma_f32_16x16x4_f32: element e of both words is k = 4 * k-group + e of the step.
template <typename T> struct SkinnyT;
template <> struct SkinnyT<bf16_t> {
    static constexpr int KPC = 8;
    static __device__ __forceinline__ f32x4_s mma(const u32x4_s& a, const u32x4_s& b, f32x4_s c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_s, a), __builtin_bit_cast(bf16x8_s, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ float ld(const bf16_t* p, int64_t i) { return bf16_to_f32(p[i]); }
    static __device__ __forceinline__ void st(bf16_t* p, int64_t i, float v) { p[i] = f32_to_bf16(v); }
};
template <> struct SkinnyT<float> {
    static constexpr int KPC = 4;
    static __device__ __forceinline__ f32x4_s mma(const u32x4_s& a, const u32x4_s& b, f32x4_s c) {
        const f32x4_s af = __builtin_bit_cast(f32x4_s, a), bf = __builtin_bit_cast(f32x4_s, b);
#pragma unroll
        for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(af[e], bf[e], c, 0, 0, 0);
        return c;
    }
    static __device__ __forceinline__ float ld(const float* p, int64_t i) { return p[i]; }
    static __device__ __forceinline__ void st(float* p, int64_t i, float v) { p[i] = v; }
};

// Ws[tile][kb][c][i] = W[KPC kb + i][cols tile + c], zero outside [K) x [N); one thread per 16-byte group
template <typename T>
__global__ __launch_bounds__(256) void skinny_pack_kernel(const T* __restrict__ w, T* __restrict__ out, int64_t K, int64_t N,
                                                          int64_t KB, int64_t ntiles, int cols) {
    constexpr int KPC = SkinnyT<T>::KPC;
    const int64_t total = ntiles * KB * cols;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(g % cols);
        const int64_t kb = g / cols % KB, tile = g / cols / KB;
        const int64_t col = tile * cols + c;
        alignas(16) T r[KPC];
#pragma unroll
        for (int i = 0; i < KPC; ++i) {
            const int64_t kx = kb * KPC + i;
            r[i] = (col < N && kx < K) ? w[kx * N + col] : T(0);
        }
        *reinterpret_cast<uint4*>(out + g * KPC) = *reinterpret_cast<const uint4*>(r);
    }
}

__device__ __forceinline__ float skinny_finish(float v, float v2, bool dual, int act, float bias, bool has_res, float res, const GluParams& glu = GluParams(), float colscale = 1.0f) {
    if (dual) v = glu_combine(v, v2, glu.kind, glu.limit, glu.alpha, glu.shift);   // activation.rs:141-162
    v += bias;                                                      // tensor_ops.rs:42-56
    if (act == 1) v = (v * 0.5f) * (erff(v / 1.41421354f) + 1.0f);  // activation.rs:96-113
    v *= colscale;
    if (has_res) v += res;
    return v;
}

// The way out, shared by both kernels: the workgroup's first 256 threads add an output each, thread 16 m + c row m of the tile's column
// c, so a wave's LDS reads meet no bank twice and a row's stores are neighbours.  What an output needs besides its sum is requested
// before the first weight (the constructor) and has long arrived.  One output's code instead of four per lane of one wave, and no
// round trip to memory at the end: 8 rows, us: K = 9216,
// N = 3072 13.4 -> 12.8, N = 6144 9.9 -> 9.4, f32 K = 768, N = 768 4.7 -> 4.3; int4 pair of 9216 14.8 -> 12.8.
template <typename T, bool DUAL, int NW, int COLS>
struct SkinnyOut {
    static constexpr int NP = DUAL ? 2 : 1;
    const int m, c, n;
    const bool in;
    int64_t at;
    float bias, res, colscale;
    __device__ __forceinline__ SkinnyOut(int tile, int M, int N, const T* pbias, const void* residual, int out_f32, const float* pscale)
        : m((int)threadIdx.x >> 4), c((int)threadIdx.x & 15), n(tile * COLS + c), in(m < M && c < COLS && n < N), at((int64_t)m * N + n), bias(0.f), res(0.f), colscale(1.0f) {
        if (!in) return;
        if (pbias) bias = SkinnyT<T>::ld(pbias, n);
        if (pscale) colscale = pscale[n];
        if (residual) res = out_f32 ? static_cast<const float*>(residual)[at] : SkinnyT<T>::ld(static_cast<const T*>(residual), at);
    }
    // Behind a barrier after the waves' sums.  False: another workgroup finishes the tile, or the thread has no output.
    __device__ __forceinline__ bool sum(const float (*red)[NP][64][4], int tile, float* part, unsigned* tickets, unsigned* ticket_lds, float (&v)[2]) {
        asm volatile("" : "+v"(bias), "+v"(res), "+v"(colscale));       // requested up there, not here
        if (threadIdx.x >= 256) return false;
        const int lane = 16 * (m >> 2) + c, i = m & 3;                   // D: lane holds rows 4 kg .. 4 kg + 3 of column c
        v[0] = v[1] = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            v[0] += red[w][0][lane][i];
            if (DUAL) v[1] += red[w][NP - 1][lane][i];
        }
        const int ksplit = gridDim.y;
        if (ksplit > 1) {
            // partials and tickets cross workgroups through device-scope accesses only (coherent across the L2s of the
            // XCDs without cache maintenance): stores acknowledged, then the ticket
            float* mine = part + ((int64_t)tile * ksplit + blockIdx.y) * NP * 256 + threadIdx.x;
            __hip_atomic_store(mine, v[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (DUAL) __hip_atomic_store(mine + 256, v[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __builtin_amdgcn_s_waitcnt(0x0F70);                         // vmcnt(0)
            __syncthreads();                                            // (the waves that are left: 256 threads)
            if (threadIdx.x == 0) *ticket_lds = __hip_atomic_fetch_add(&tickets[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();                                            // the partials are read after the ticket is known
            if (*ticket_lds != (unsigned)(ksplit - 1)) return false;
            // every ticket of this launch has been drawn: leave the counter at zero for the next one
            if (threadIdx.x == 0) __hip_atomic_store(&tickets[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            v[0] = v[1] = 0.f;
            for (int q = 0; q < ksplit; ++q) {                           // device-scope loads: the partials come from other CUs
                const float* src = part + ((int64_t)tile * ksplit + q) * NP * 256 + threadIdx.x;
                v[0] += __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (DUAL) v[1] += __hip_atomic_load(src + 256, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        return in;
    }
    // out_f32: the f32 accumulator (plus an f32 residual) is stored as it is
    __device__ __forceinline__ void store(T* y, int out_f32, float o) {
        if (out_f32) reinterpret_cast<float*>(y)[at] = o;
        else SkinnyT<T>::st(y, at, o);
    }
};

template <typename T, bool DUAL, int NW, int U, int COLS>
__global__ __launch_bounds__(64 * NW) void skinny_gemm_kernel(const T* __restrict__ x, const T* __restrict__ ws,
                                                          const T* __restrict__ ws2, const T* __restrict__ bias,
                                                          const T* __restrict__ residual, T* __restrict__ y, int M, int K,
                                                          int N, int act, float* __restrict__ part, unsigned* __restrict__ tickets,
                                                          int out_f32, EpiExtra extra) {
    static_assert(COLS == 12 || COLS == 16, "columns of a tile");
    constexpr int KPC = SkinnyT<T>::KPC, KSTEP = 4 * KPC;
    // f32 over tiles of 16 columns, which 8 or 16 waves take by the rows: a wave of 8 adds its odd steps apart from its even ones, so that the sums are those of 16
    // waves, in their order, as near to 64 bits.  R: with one request in flight the loop takes two steps at a time to tell them apart (16 rows, K = 2048, N = 8192
    // 15.1 -> 15.4 us; over tiles of 12 columns, which 8 waves take whatever the rows, it would be 19.2 -> 21.1 for 12 rows of K = 3072, N = 4200).
    constexpr int CH = std::is_same<T, float>::value && NW == 8 && COLS == 16 ? 2 : 1, R = CH > U ? CH : 1;
    __shared__ float red[NW * CH][DUAL ? 2 : 1][64][4];
    __shared__ unsigned ticket;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));   // uniform: a matrix instruction does not look at the lane mask, so the tests of a step must be branches
    const int c = lane & 15, kg = lane >> 4;     // B: column c, k-group kg; A: row c, k-group kg
    const int tile = blockIdx.x;
    SkinnyOut<T, DUAL, NW * CH, COLS> out(tile, M, N, bias, residual, out_f32, extra.colscale);
    const int ksplit = gridDim.y, ks = blockIdx.y;
    const int s_begin = (int)((int64_t)(K / KSTEP) * ks / ksplit), nsteps = (int)((int64_t)(K / KSTEP) * (ks + 1) / ksplit);
    const int bcol = c < COLS ? c : COLS - 1;    // columns beyond the tile re-read its last one; their sums are never stored
    const int64_t b0 = (int64_t)tile * (K / KPC) * COLS + kg * COLS + bcol;
    const u32x4_s* bsrc = reinterpret_cast<const u32x4_s*>(ws) + b0;
    const u32x4_s* bsrc2 = DUAL ? reinterpret_cast<const u32x4_s*>(ws2) + b0 : nullptr;
    const int arow = c < M ? c : M - 1;          // rows beyond M re-read the last one; their products are never stored
    const u32x4_s* asrc = reinterpret_cast<const u32x4_s*>(x + (int64_t)arow * K + KPC * kg);

    // A ring of U steps: a step's registers are asked to fetch the wave's next but U - 1 as soon as they have been multiplied, so
    // a wave has U - 1 or U requests on their way all the time.  (Rounds of U requests, all awaited before the next were made, left the memory
    // pipeline empty once a round: K = 9216, N = 3072, 8 rows 17.0 us; this 14.9, with tiles of 12 columns 11.8.)
    f32x4_s acc[CH], acc2[CH];
#pragma unroll
    for (int h = 0; h < CH; ++h) acc[h] = acc2[h] = f32x4_s{0.f, 0.f, 0.f, 0.f};
    u32x4_s b[U], b2[DUAL ? U : 1], a[U];
    auto fetch = [&](int u, int s) {
        b[u] = __builtin_nontemporal_load(bsrc + (int64_t)s * (4 * COLS));
        if (DUAL) b2[DUAL ? u : 0] = __builtin_nontemporal_load(bsrc2 + (int64_t)s * (4 * COLS));
        a[u] = asrc[s * 4];
    };
    if (s_begin + wave < nsteps) {
#pragma unroll
        for (int u = 0; u < U; ++u) fetch(u, s_begin + wave + NW * u < nsteps ? s_begin + wave + NW * u : s_begin + wave);   // (a step past the end is not multiplied)
        for (int s0 = s_begin + wave; s0 < nsteps; s0 += NW * U * R) {
#pragma unroll
            for (int i = 0; i < U * R; ++i) {
                const int s = s0 + NW * i, u = i % U, h = i % CH;
                if (s < nsteps) {
                    acc[h] = SkinnyT<T>::mma(a[u], b[u], acc[h]);
                    if (DUAL) acc2[h] = SkinnyT<T>::mma(a[u], b2[DUAL ? u : 0], acc2[h]);
                }
                if (s + NW * U < nsteps) fetch(u, s + NW * U);
            }
        }
    }
#pragma unroll
    for (int h = 0; h < CH; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            red[wave + NW * h][0][lane][i] = acc[h][i];
            if (DUAL) red[wave + NW * h][DUAL ? 1 : 0][lane][i] = acc2[h][i];
        }
    __syncthreads();
    float v[2];
    if (!out.sum(red, tile, part, tickets, &ticket, v)) return;
    float o = skinny_finish(v[0], v[1], DUAL, act, out.bias, residual != nullptr, out.res, extra.glu, out.colscale);
    if (extra.softcap != 0.f) o = softcap_f32(o, extra.softcap);
    out.store(y, out_f32, o);
}

// An f32 layer whose rows are normed first (LayerNorm), a tile for each CU at most.  Every workgroup norms all rows, wave r row r, while its weights, all of them asked
// for before, are on their way from memory; the normed rows are the A operand in LDS, a row 16 bytes longer than it is, so that 16 rows' reads meet no bank twice.
// Asked for ahead of the rows the weights held them up (loads return in order): 7 rows of 768, N = 2304 5.11 us, so 4.75, the norm's launch in front 6.43 and the layer
// alone 4.21; N = 3072 4.96, 6.55 and 4.32; 16 rows 5.74 and 6.95, 5.85 and 7.09.  A tile for each CU at most, since every workgroup norms all rows.
constexpr int kNormSteps = 4;                     // steps of 16 k of a wave: K <= 1008, where 16 rows are 64 KB
template <int COLS>
__global__ __launch_bounds__(1024) void skinny_norm_kernel(const float* __restrict__ x, const float* __restrict__ gamma, const float* __restrict__ beta, const float* __restrict__ ws,
                                                           const float* __restrict__ bias, const float* __restrict__ residual, float* __restrict__ y, int M, int K, int N, int act,
                                                           float inv_n, float eps, EpiExtra extra) {
    constexpr int NW = 16;
    extern __shared__ __align__(16) float rows[];   // [M][K + 4], then the waves' sums
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int c = lane & 15, kg = lane >> 4, nsteps = K / 16, tile = blockIdx.x;
    const int items = K / 4;                      // of 16 bytes
    f32x4_s v[4], g[4], o[4];
    if (wave < M) {                               // (loads return in order: what is nearer is asked for first)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = reinterpret_cast<const f32x4_s*>(x + (int64_t)wave * K)[min(64 * j + lane, items - 1)];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            g[j] = reinterpret_cast<const f32x4_s*>(gamma)[min(64 * j + lane, items - 1)];
            o[j] = reinterpret_cast<const f32x4_s*>(beta)[min(64 * j + lane, items - 1)];
        }
    }
    const u32x4_s* bsrc = reinterpret_cast<const u32x4_s*>(ws) + (int64_t)tile * (K / 4) * COLS + kg * COLS + (c < COLS ? c : COLS - 1);
    u32x4_s b[kNormSteps];
#pragma unroll
    for (int u = 0; u < kNormSteps; ++u)
        if (wave + NW * u < nsteps) b[u] = __builtin_nontemporal_load(bsrc + (int64_t)(wave + NW * u) * (4 * COLS));
    SkinnyOut<float, false, NW, COLS> out(tile, M, N, bias, residual, 0, extra.colscale);
    if (wave < M) {
        float s = 0.f, q = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) s += 64 * j + lane < items ? (v[j].x + v[j].y) + (v[j].z + v[j].w) : 0.f;
        const float mean = wave_sum(s) * inv_n;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] -= mean;
            q += 64 * j + lane < items ? (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w) : 0.f;
        }
        const float inv_std = 1.0f / sqrtf(wave_sum(q) * inv_n + eps);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (64 * j + lane < items) *reinterpret_cast<f32x4_s*>(&rows[wave * (K + 4) + 4 * (64 * j + lane)]) = (v[j] * inv_std) * g[j] + o[j];
    }
    __syncthreads();
    f32x4_s acc = {0.f, 0.f, 0.f, 0.f};
    const float* a = &rows[(c < M ? c : M - 1) * (K + 4) + 4 * kg];   // rows beyond M re-read the last one; their products are never stored
#pragma unroll
    for (int u = 0; u < kNormSteps; ++u) {
        const int s = wave + NW * u;
        if (s < nsteps) acc = SkinnyT<float>::mma(*reinterpret_cast<const u32x4_s*>(a + 16 * s), b[u], acc);
    }
    __syncthreads();
    float (*red)[1][64][4] = reinterpret_cast<float (*)[1][64][4]>(rows);
    *reinterpret_cast<f32x4_s*>(red[wave][0][lane]) = acc;
    __syncthreads();
    float sum[2];
    if (!out.sum(red, tile, nullptr, nullptr, nullptr, sum)) return;
    out.store(y, 0, skinny_finish(sum[0], 0.f, false, act, out.bias, residual != nullptr, out.res, extra.glu, out.colscale));
}

// Qs[tile][S][lane = 16 kg + c][16 bytes]: byte i = code row (RPW S + RPL kg + i) of column 16 tile + c, xor flip.  int8:
// code rows are k, RPL = 16 rows per lane, flip 0x80.  int4: a code row is a packed byte of two k, RPL = 16 rows (32 k)
// per lane, flip 0x88.  Rows and columns outside the matrix hold the biased zero.
__global__ __launch_bounds__(256) void skinny_pack_codes_kernel(const uint8_t* __restrict__ q, uint8_t* __restrict__ out, int64_t rows,
                                                                int64_t N, int64_t S, int64_t ntiles, uint32_t flip) {
    const int64_t total = ntiles * S * 64;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (int64_t)gridDim.x * blockDim.x) {
        const int lane = (int)(g & 63), c = lane & 15, kg = lane >> 4;
        const int64_t sidx = (g >> 6) % S, tile = (g >> 6) / S;
        const int64_t col = tile * 16 + c, r0 = sidx * 64 + kg * 16;
        uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int64_t r = r0 + i;
            const uint32_t b = (col < N && r < rows) ? ((uint32_t)q[r * N + col] ^ flip) : flip;
            w[i >> 2] |= b << (8 * (i & 3));
        }
        *reinterpret_cast<uint4*>(out + g * 16) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

__device__ __forceinline__ bf16x8_s codes_to_bf16(float f0, float f1, float f2, float f3, float f4, float f5, float f6, float f7) {
    typedef float f32x2_s __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2_s __attribute__((ext_vector_type(2)));
    bf16x8_s r;
    const float f[8] = {f0, f1, f2, f3, f4, f5, f6, f7};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f32x2_s p;
        p.x = f[2 * i]; p.y = f[2 * i + 1];
        const bf16x2_s h = __builtin_convertvector(p, bf16x2_s);   // exact: integers below 256
        r[2 * i] = h.x; r[2 * i + 1] = h.y;
    }
    return r;
}
// 8 consecutive int8 codes (two dwords, biased by 128) as the B operand
__device__ __forceinline__ bf16x8_s bytes_to_bf16(uint32_t a, uint32_t b) {
    return codes_to_bf16((float)(a & 0xFFu), (float)((a >> 8) & 0xFFu), (float)((a >> 16) & 0xFFu), (float)(a >> 24),
                         (float)(b & 0xFFu), (float)((b >> 8) & 0xFFu), (float)((b >> 16) & 0xFFu), (float)(b >> 24));
}
// 8 consecutive int4 codes (one dword of packed bytes: k = 2 j in the low nibble of byte j, biased by 8)
__device__ __forceinline__ bf16x8_s nibbles_to_bf16(uint32_t w) {
    const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
    return codes_to_bf16((float)(lo & 0xFFu), (float)(hi & 0xFFu), (float)((lo >> 8) & 0xFFu), (float)((hi >> 8) & 0xFFu),
                         (float)((lo >> 16) & 0xFFu), (float)((hi >> 16) & 0xFFu), (float)(lo >> 24), (float)(hi >> 24));
}

// QF 1: int8, per-column scales [N]; QF 2: int4 in groups of 128, scales [K/128, N].  A word covers KPW = 64 / 128 k.  Pairs in 8 waves, which wide layers take: three
// workgroups to a CU (the compiler by itself uses 97 registers of int4's, room for two: K = 4096, N = 11008, 2 rows 19.2 us, this 15.0, 12 rows 23.0 and 16.8).
template <int QF, bool DUAL, int NW, int U>
__global__ __launch_bounds__(64 * NW, DUAL && NW == 8 ? 6 : 4) void skinny_gemm_quant_kernel(const bf16_t* __restrict__ x, const uint8_t* __restrict__ qs,
                                                                const uint8_t* __restrict__ qs2, const bf16_t* __restrict__ sc,
                                                                const bf16_t* __restrict__ sc2, const bf16_t* __restrict__ bias,
                                                                const bf16_t* __restrict__ residual, bf16_t* __restrict__ y, int M, int K,
                                                                int N, int act, float* __restrict__ part, unsigned* __restrict__ tickets,
                                                                int out_f32) {
    constexpr int KPW = QF == 1 ? 64 : 128;      // k per word
    constexpr int SPW = KPW / 32;                // MFMA steps per word
    constexpr int NP = DUAL ? 2 : 1;
    constexpr float BIAS = QF == 1 ? 128.0f : 8.0f;
    __shared__ float red[NW][NP][64][4];
    __shared__ unsigned ticket;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));   // uniform: a matrix instruction does not look at the lane mask, so the tests of a step must be branches
    const int c = lane & 15, kg = lane >> 4;
    const int tile = blockIdx.x;
    SkinnyOut<bf16_t, DUAL, NW, 16> out(tile, M, N, bias, residual, out_f32, nullptr);
    const int ksplit = gridDim.y, ks = blockIdx.y;
    const int nwords = K / KPW;
    const int s_begin = (int)((int64_t)nwords * ks / ksplit), s_end = (int)((int64_t)nwords * (ks + 1) / ksplit);
    const u32x4_s* bsrc = reinterpret_cast<const u32x4_s*>(qs) + (int64_t)tile * nwords * 64 + lane;
    const u32x4_s* bsrc2 = DUAL ? reinterpret_cast<const u32x4_s*>(qs2) + (int64_t)tile * nwords * 64 + lane : nullptr;
    const int arow = c < M ? c : M - 1;
    const bf16_t* arowp = x + (int64_t)arow * K + (KPW / 4) * kg;   // the lane's KPW / 4 consecutive k of a word
    const int ncol = tile * 16 + c < N ? tile * 16 + c : N - 1;     // scale column of this lane's outputs (clamped: never stored)
    bf16x8_s ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = (__bf16)1.0f;

    f32x4_s tot = {0.f, 0.f, 0.f, 0.f}, tot2 = {0.f, 0.f, 0.f, 0.f}, xsum = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = s_begin + wave; s0 < s_end; s0 += NW * U) {
        u32x4_s b[U], b2[DUAL ? U : 1], a[U][SPW];
        float gs[U], gs2[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = s0 + NW * u < s_end ? s0 + NW * u : s0;   // a word past the end repeats the first and is skipped below
            b[u] = __builtin_nontemporal_load(bsrc + (int64_t)s * 64);
            if (DUAL) b2[u] = __builtin_nontemporal_load(bsrc2 + (int64_t)s * 64);
#pragma unroll
            for (int t = 0; t < SPW; ++t) a[u][t] = *reinterpret_cast<const u32x4_s*>(arowp + (int64_t)s * KPW + 8 * t);
            if (QF == 2) {
                gs[u] = bf16_to_f32(sc[(int64_t)s * N + ncol]);
                if (DUAL) gs2[u] = bf16_to_f32(sc2[(int64_t)s * N + ncol]);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s0 + NW * u < s_end) {
                f32x4_s acc = {0.f, 0.f, 0.f, 0.f}, acc2 = {0.f, 0.f, 0.f, 0.f}, xs = {0.f, 0.f, 0.f, 0.f};
                const uint32_t bw[4] = {b[u].x, b[u].y, b[u].z, b[u].w};
                const uint32_t bw2[4] = {DUAL ? b2[DUAL ? u : 0].x : 0u, DUAL ? b2[DUAL ? u : 0].y : 0u, DUAL ? b2[DUAL ? u : 0].z : 0u,
                                         DUAL ? b2[DUAL ? u : 0].w : 0u};
#pragma unroll
                for (int t = 0; t < SPW; ++t) {
                    const bf16x8_s av = __builtin_bit_cast(bf16x8_s, a[u][t]);
                    const bf16x8_s bv = QF == 1 ? bytes_to_bf16(bw[2 * t], bw[2 * t + 1]) : nibbles_to_bf16(bw[t]);
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc, 0, 0, 0);
                    if (DUAL) {
                        const bf16x8_s bv2 = QF == 1 ? bytes_to_bf16(bw2[2 * t], bw2[2 * t + 1]) : nibbles_to_bf16(bw2[t]);
                        acc2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv2, acc2, 0, 0, 0);
                    }
                    xs = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, ones, xs, 0, 0, 0);   // sum_k x[row, k] in every column
                }
                if (QF == 1) {
                    tot += acc; xsum += xs;
                    if (DUAL) tot2 += acc2;
                } else {   // one scale group: take the bias out, scale, add
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        tot[i] += gs[u] * (acc[i] - BIAS * xs[i]);
                        if (DUAL) tot2[i] += gs2[u] * (acc2[i] - BIAS * xs[i]);
                    }
                }
            }
        }
    }
    if (QF == 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            tot[i] -= BIAS * xsum[i];
            if (DUAL) tot2[i] -= BIAS * xsum[i];
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        red[wave][0][lane][i] = tot[i];
        if (DUAL) red[wave][DUAL ? 1 : 0][lane][i] = tot2[i];
    }
    __syncthreads();
    float v[2];
    if (!out.sum(red, tile, part, tickets, &ticket, v)) return;
    const float s1 = QF == 1 ? bf16_to_f32(sc[out.n]) : 1.0f, s2 = QF == 1 && DUAL ? bf16_to_f32(sc2[out.n]) : 1.0f;
    out.store(y, out_f32, skinny_finish(v[0] * s1, v[1] * s2, DUAL, act, out.bias, residual != nullptr, out.res));
}

}  // namespace

bool skinny_gemm_supported(int dtype, int64_t m, int64_t k, int64_t n) {
    if (dtype != 0 && dtype != 2) return false;
    const int64_t kstep = dtype == 0 ? 16 : 32;
    return m >= 2 && m <= 16 && k >= kstep && k % kstep == 0 && n >= 1 && k < (1ll << 31) && n < (1ll << 31) - 16;
}
// Columns of a tile of the copy.  A workgroup is one tile, and while there are few of them the CU with the most columns sets the
// time: tiles of 12 where they leave fewer columns on it (N = 3072: 256 tiles, one for every CU, instead of 192; N = 9216 three a CU instead
// of three on some and two on others).  The MFMA's other four columns are wasted, which costs nothing here; from 768 tiles of 16 on
// the CUs are evenly loaded either way and whole instructions are the better use of the memory pipeline.  us with 16 and with 12 columns, 8
// rows: K = 9216, N = 3072 14.9 and 11.8, K = 4096 7.8 and 6.7, K = 3072 N = 6144 10.0 and 8.6, pair of 9216 23.0 and 19.7; N = 32768 35.7
// and 38.6.
static int skinny_cols(int64_t n) {
    const int64_t t16 = cdiv_s(n, 16), t12 = cdiv_s(n, 12);
    return t16 < 768 && cdiv_s(t12, 256) * 12 < cdiv_s(t16, 256) * 16 ? 12 : 16;
}
size_t skinny_weight_bytes(int dtype, int64_t k, int64_t n) {
    const int64_t kpc = dtype == 0 ? 4 : 8, cols = skinny_cols(n);
    return (size_t)(cdiv_s(n, cols) * cdiv_s(k, kpc) * cols) * 16;
}
void skinny_pack_weights(hipStream_t s, int dtype, const void* w, void* out, int64_t k, int64_t n) {
    const int64_t cols = skinny_cols(n), ntiles = cdiv_s(n, cols), kb = cdiv_s(k, dtype == 0 ? 4 : 8), total = ntiles * kb * cols;
    if (total <= 0) return;
    const unsigned g = (unsigned)(cdiv_s(total, 256) > 65536 ? 65536 : cdiv_s(total, 256));
    if (dtype == 0) skinny_pack_kernel<float><<<g, 256, 0, s>>>((const float*)w, (float*)out, k, n, kb, ntiles, (int)cols);
    else skinny_pack_kernel<bf16_t><<<g, 256, 0, s>>>((const bf16_t*)w, (bf16_t*)out, k, n, kb, ntiles, (int)cols);
}
// How a launch shares out the steps (words of codes) of a tile: waves per workgroup, requests of a wave, workgroups per tile.  Every layer
// is one pass over its weights; what is left beside HBM's pace are a wave's waits for its answers (1 to 1.5 us each) and, with
// several workgroups to a tile, their meeting (3 us).  Fitted to 45 layers (K = 256 .. 14336, N = 512 .. 50257, f32 and bf16, plain and pairs, 2 to 16 rows, weights from
// memory): of 711 that take over 8 us the rule's choice is 3.1 % from the best of 14 in the mean.  us:
//   one tile per CU or less   plain layers 16 waves with two steps in flight, from 9 rows on one: a step's 16 rows take more of the memory pipeline than its
//                    weights (16 rows, K = 9216, N = 3072 14.6, 8 waves of three 16.5).  Pairs, whose step is two requests and the rows', 8 waves of two (bf16, 12
//                    rows, K = 4096, N = 1024 8.2, 16 of one 9.5); of f32 only over tiles of 16 columns, over those of 12 as plain ones
//   tiles of 12 columns beyond   8 waves of two, from 9 rows on of one (8 rows, N = 6144 9.4, with 4 waves of four 9.7, 16 of one 10.2; 16 rows, pair of 9216 8 waves of one
//                    22.1, of two 24.8, 16 of one 29.2)
//   tiles of 16 columns, under three a CU   16 waves of two, from 9 rows on 8 of one (12 rows, bf16 pair of 11008 over K = 4096 29.6, 16 of one 36.9; f32 K = 2048, N = 8192
//                    14.9 and 16.9); pairs of f32 16 of one (the same pair 67.3 and 62.3)
//   three and more a CU   8 waves of two (8 rows, bf16, K = 512, N = 32000 8.5, 8 of four 11.0; 12 rows, pair of 50257 over K = 768 26.2, 16 of one 32.2); plain f32 up to
//                    8 rows of four (2 rows, K = 3072, N = 14432 30.4 and 31.9); plain layers of 9 rows and more whose sums are long enough for 16 waves those, of one (12 rows,
//                    K = 3072, N = 32768 40.4 and 37.1, K = 768, N = 50257 16.8 and 21.1)
//   few tiles        split while the launch stays within one workgroup per CU and a wave keeps six steps, of a pair three (8 rows: f32 K = 3072, N = 768
//                    8.5 -> 7.1, K = 12288 27.2 -> 12.1; bf16 K = 3072, N = 576, six steps already, 5.3, in two 5.7; 12 rows, pair K = 4096, N = 1024 11.9 -> 8.2)
//   codes            16 waves to a tile up to one tile per CU, else 8, one word in flight (a wave also has to convert it)
// Weights are read past the caches (nontemporal): 4-5 % of a layer whose weights come from memory.  Models that the 256 MB last-level cache
// holds gain or lose: whole f32 decode steps of 2 to 16 rows, against plain loads, take 0-15 % less with 16 MB of weights (5 % more at 2
// rows), 2-9 % more with 100 to 180 MB (13 % at 16 rows of three layers of 1024), the same with 210, up to 5 % less with 240 to 270 and 1-7 %
// less from 300 MB on.  One rule for all.
SkinnyPlan skinny_plan(int dtype, int64_t m, int64_t steps, int64_t n, bool dual, bool codes) {
    const int64_t cols = codes ? 16 : skinny_cols(n), tiles = cdiv_s(n, cols);
    int ks = 1;
    if (codes) {
        while (tiles * ks < 96 && steps / (32 * ks) >= 3) ks *= 2;
        return {tiles <= 256 ? 16 : 8, 1, ks};
    }
    while (tiles * ks <= 128 && steps / (16 * ks) >= (dual ? 6 : 12)) ks *= 2;
    const int few = m > 8 ? 1 : 2;   // requests that the rows leave room for
    if (tiles <= 256) return dual && (dtype == 2 || cols == 16) ? SkinnyPlan{8, 2, ks} : SkinnyPlan{16, few, ks};
    if (cols == 12) return {8, few, 1};
    if (tiles < 768) return m > 8 && !(dual && dtype == 0) ? SkinnyPlan{8, 1, 1} : SkinnyPlan{16, few, 1};
    if (!dual && m > 8 && steps >= 64) return {16, 1, 1};
    return {8, dtype == 0 && !dual && m <= 8 ? 4 : 2, 1};
}
static size_t skinny_part_bytes(int64_t n, bool dual, int cols, int ks) { return ks > 1 ? (size_t)cdiv_s(n, cols) * ks * (dual ? 2 : 1) * 256 * sizeof(float) : 0; }
size_t skinny_workspace_bytes(int64_t k, int64_t n, bool dual) {
    // whichever of rows and codes splits more (f32 has the most steps), over the narrower tiles
    return skinny_part_bytes(n, dual, 12, std::max(skinny_plan(0, 1, k / 16, n, dual, false).ks, skinny_plan(2, 1, k / 64, n, dual, true).ks));
}
// Workgroups of 8 waves of a pair of codes that fit a CU.
int skinny_pair_workgroups(int quant) {
    int n = 0;
    const void* f = quant == 1 ? (const void*)skinny_gemm_quant_kernel<1, true, 8, 1> : (const void*)skinny_gemm_quant_kernel<2, true, 8, 1>;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, f, 512, 0) == hipSuccess ? n : -1;
}
bool skinny_quant_supported(int dtype, int64_t m, int64_t k, int64_t n, int qf) {
    if ((qf != 1 && qf != 2) || dtype != 2) return false;
    return skinny_gemm_supported(dtype, m, k, n) && k % (qf == 1 ? 64 : 128) == 0;
}
size_t skinny_codes_bytes(int64_t k, int64_t n, int qf) { return (size_t)(cdiv_s(n, 16) * (k / (qf == 1 ? 64 : 128)) * 64 * 16); }
void skinny_pack_codes(hipStream_t s, const void* codes, void* out, int64_t k, int64_t n, int qf) {
    const int64_t ntiles = cdiv_s(n, 16), words = k / (qf == 1 ? 64 : 128), total = ntiles * words * 64;
    if (total <= 0) return;
    const unsigned g = (unsigned)(cdiv_s(total, 256) > 65536 ? 65536 : cdiv_s(total, 256));
    // int8: one code row per k; int4: one packed byte per two k
    skinny_pack_codes_kernel<<<g, 256, 0, s>>>((const uint8_t*)codes, (uint8_t*)out, qf == 1 ? k : k / 2, n, words, ntiles,
                                               qf == 1 ? 0x80u : 0x88u);
}

bool skinny_norm_fits(const SkinnyLinearArgs& a, const void* gamma, const void* beta) {
    return a.dtype == 0 && !a.quant && !a.ws2 && a.extra.softcap == 0.f && a.k <= 1008 && cdiv_s(a.n, skinny_cols(a.n)) <= 256 &&
           (((uintptr_t)a.x | (uintptr_t)gamma | (uintptr_t)beta) & 15) == 0;
}

void skinny_gemm(hipStream_t s, const SkinnyLinearArgs& a) {
    const bool dual = a.ws2 != nullptr;
    if (a.gamma) {   // (the caller has asked skinny_norm_fits)
        const int cols = skinny_cols(a.n);
        const unsigned grid = (unsigned)cdiv_s(a.n, cols);
        const size_t lds = std::max<size_t>((size_t)a.m * (a.k + 4) * sizeof(float), 16 * 64 * 4 * sizeof(float));
        const auto fn = cols == 12 ? skinny_norm_kernel<12> : skinny_norm_kernel<16>;
        fn<<<grid, 1024, lds, s>>>((const float*)a.x, a.gamma, a.beta, (const float*)a.ws, (const float*)a.bias, (const float*)a.residual, (float*)a.y, (int)a.m, (int)a.k,
                                   (int)a.n, a.act, a.inv_n, a.eps, a.extra);
        return;
    }
    const int64_t steps = a.k / (a.quant == 1 ? 64 : a.quant == 2 ? 128 : a.dtype == 0 ? 16 : 32);
    const int cols = a.quant ? 16 : skinny_cols(a.n);
    SkinnyPlan p = skinny_plan(a.dtype, a.m, steps, a.n, dual, a.quant != 0);
    if (p.ks > 1 && (!a.part || !a.tickets || a.part_bytes < skinny_part_bytes(a.n, dual, cols, p.ks))) p.ks = 1;
    const dim3 grid((unsigned)cdiv_s(a.n, cols), (unsigned)p.ks);
    if (a.quant) {
#define GPTRS_LAUNCH(QF, DUAL, NW)                                                                                          \
        skinny_gemm_quant_kernel<QF, DUAL, NW, 1><<<grid, 64 * NW, 0, s>>>((const bf16_t*)a.x, (const uint8_t*)a.ws, (const uint8_t*)a.ws2,  \
            (const bf16_t*)a.scale, (const bf16_t*)a.scale2, (const bf16_t*)a.bias, (const bf16_t*)a.residual, (bf16_t*)a.y,   \
            (int)a.m, (int)a.k, (int)a.n, a.act, (float*)a.part, a.tickets, a.out_f32)
#define GPTRS_LAUNCH_W(QF, DUAL) do { if (p.nw == 16) GPTRS_LAUNCH(QF, DUAL, 16); else GPTRS_LAUNCH(QF, DUAL, 8); } while (0)
        if (a.quant == 1) { if (dual) GPTRS_LAUNCH_W(1, true); else GPTRS_LAUNCH_W(1, false); }
        else { if (dual) GPTRS_LAUNCH_W(2, true); else GPTRS_LAUNCH_W(2, false); }
#undef GPTRS_LAUNCH_W
#undef GPTRS_LAUNCH
        return;
    }
    auto go = [&](auto type, auto pair, auto nw, auto depth, auto columns) {
        typedef decltype(type) T;
        constexpr int NW = decltype(nw)::value;
        skinny_gemm_kernel<T, decltype(pair)::value, NW, decltype(depth)::value, decltype(columns)::value><<<grid, 64 * NW, 0, s>>>(
            (const T*)a.x, (const T*)a.ws, (const T*)a.ws2, (const T*)a.bias, (const T*)a.residual, (T*)a.y, (int)a.m, (int)a.k, (int)a.n, a.act,
            (float*)a.part, a.tickets, a.dtype == 2 ? a.out_f32 : 0, a.extra);
    };
    auto shape = [&](auto type, auto pair) {
        constexpr std::integral_constant<int, 1> I1{};
        constexpr std::integral_constant<int, 2> I2{};
        constexpr std::integral_constant<int, 4> I4{};
        constexpr std::integral_constant<int, 8> I8{};
        constexpr std::integral_constant<int, 12> I12{};
        constexpr std::integral_constant<int, 16> I16{};
        auto tile = [&](auto columns) {
            if (p.nw == 16) { if (p.depth == 1) go(type, pair, I16, I1, columns); else go(type, pair, I16, I2, columns); }
            else if (p.depth == 1) go(type, pair, I8, I1, columns);
            else go(type, pair, I8, I2, columns);
        };
        if (cols == 12) return tile(I12);
        if constexpr (std::is_same<decltype(type), float>::value && !decltype(pair)::value)
            if (p.depth == 4) return go(type, pair, I8, I4, I16);
        tile(I16);
    };
    auto types = [&](auto pair) { if (a.dtype == 0) shape(float(), pair); else shape(bf16_t(), pair); };
    if (dual) types(std::true_type{});
    else types(std::false_type{});
}

}  // namespace k
}  // namespace gptrs
