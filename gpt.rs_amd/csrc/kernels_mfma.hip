// MFMA tile GEMM for prefill-sized linear layers (M > 16): bf16 in / f32 accumulate / bf16 out on
// v_mfma_f32_32x32x16_bf16; f32 throughout on v_mfma_f32_32x32x2_f32, and from 129 rows on as six bf16 products (gemm_split_kernel).
//
// Per lane the matrix cores want consecutive k of ONE row (A) or ONE column (B).  Activations x[M,K] are row-major,
// so A fragments are plain 16-byte loads.  Weights are stored [in,out] row-major (nn/layers/linear.rs:50-71), the
// wrong way round for B, so the GEMM reads a derived copy Wk[K/KPC][Npad][KPC] in which the KPC consecutive k of a
// column that fill 16 bytes (8 bf16 or 4 f32) are adjacent (Npad = N rounded up to the 128-column block tile, zero
// filled); the backend builds it once per weight and keeps it beside the original.  With it a block's B tile is, per
// 16-byte k-group, one contiguous 2 KiB run, and every data movement below is in 16-byte chunks whatever the type.
#include <algorithm>
#include <type_traits>

#include "kernels.hpp"
#include "device_utils.hpp"

namespace gptrs {
namespace k {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// Element types of the GEMM: KPC = k per 16-byte chunk; mma() multiplies one 32 x (2 KPC) A fragment by one
// (2 KPC) x 32 B fragment (a lane holds the KPC values of its row / column in k-group lane / 32).
template <typename T> struct Mma;
template <> struct Mma<bf16_t> {
    static constexpr int KPC = 8;
    typedef bf16x8_t frag;
    static __device__ __forceinline__ f32x16_t mma(const frag& a, const frag& b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ float ld(const bf16_t* p, int64_t i) { return bf16_to_f32(p[i]); }
    static __device__ __forceinline__ void st(bf16_t* p, int64_t i, float v) { p[i] = f32_to_bf16(v); }
};
template <> struct Mma<float> {
    static constexpr int KPC = 4;
    typedef f32x4_t frag;
    // four K = 2 products: element e of both fragments is k = 4 * (lane / 32) + e of the 8-k step
    static __device__ __forceinline__ f32x16_t mma(const frag& a, const frag& b, f32x16_t c) {
#pragma unroll
        for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], c, 0, 0, 0);
        return c;
    }
    static __device__ __forceinline__ float ld(const float* p, int64_t i) { return p[i]; }
    static __device__ __forceinline__ void st(float* p, int64_t i, float v) { p[i] = v; }
};

static inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

constexpr int kBN = 128;   // column padding unit of the derived weights
constexpr int kKb = 8;     // 16-byte k-groups per k tile: 64 k of bf16, 32 k of f32

static inline int kpc_of(int dtype) { return dtype == 0 ? 4 : 8; }
int64_t mfma_padded_n(int64_t n) { return cdiv(n, kBN) * kBN; }
size_t mfma_weight_bytes(int dtype, int64_t k, int64_t n) {
    return (size_t)cdiv(k, kpc_of(dtype)) * (size_t)mfma_padded_n(n) * 16;
}

// Wk[kb][n][i] = W[kb*KPC+i][n]; one thread per (kb, n); reads coalesced along n, one 16-byte store.
template <typename T>
__global__ __launch_bounds__(256) void k8_weights_kernel(const T* __restrict__ w, T* __restrict__ out, int64_t K, int64_t N,
                                                         int64_t Npad) {
    constexpr int KPC = Mma<T>::KPC;
    const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t kb = blockIdx.y;
    if (n >= Npad) return;
    alignas(16) T r[KPC];
#pragma unroll
    for (int i = 0; i < KPC; ++i) {
        const int64_t kx = kb * KPC + i;
        r[i] = (n < N && kx < K) ? w[kx * N + n] : T(0);
    }
    *reinterpret_cast<uint4*>(out + (kb * Npad + n) * KPC) = *reinterpret_cast<const uint4*>(r);
}

void mfma_pack_weights(hipStream_t s, int dtype, const void* w, void* out, int64_t k, int64_t n) {
    const int64_t npad = mfma_padded_n(n);
    dim3 grid((unsigned)cdiv(npad, 256), (unsigned)cdiv(k, kpc_of(dtype)));
    if (dtype == 0) k8_weights_kernel<float><<<grid, 256, 0, s>>>((const float*)w, (float*)out, k, n, npad);
    else k8_weights_kernel<bf16_t><<<grid, 256, 0, s>>>((const bf16_t*)w, (bf16_t*)out, k, n, npad);
}

// Weight-only quantised weights (bf16 activations): the GEMM reads the CODES, in the same k-grouped order, and turns
// them into the bf16 values of the dequantised matrix, bf16(code * scale), on the way to the matrix pipes; no dequantised
// copy exists.  Ck[kb][n] holds the 8 codes of k-group kb of column n with the sign bias added (int8: 8 bytes of q + 128;
// int4: one dword, nibble i = q(k = 8 kb + i) + 8), so a code converts with one unsigned-byte / bit-field instruction
// and one fma (u * s - bias * s is exactly (u - bias) * s, rounded once like the product the dequantiser forms).
// Padding (n >= N, k >= K) holds the code of zero.
template <int QF>
__global__ __launch_bounds__(256) void k8_codes_kernel(const uint8_t* __restrict__ q, uint32_t* __restrict__ out, int64_t K, int64_t N,
                                                       int64_t Npad) {
    const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t kb = blockIdx.y;
    if (n >= Npad) return;
    if (QF == 1) {
        uint32_t w[2] = {0x80808080u, 0x80808080u};
        if (n < N) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int64_t kx = kb * 8 + i;
                const uint32_t u = kx < K ? (uint32_t)(uint8_t)(q[kx * N + n] + 128u) : 128u;   // si8 [K, N]
                w[i >> 2] = (w[i >> 2] & ~(0xFFu << (8 * (i & 3)))) | (u << (8 * (i & 3)));
            }
        }
        *reinterpret_cast<uint2*>(out + (kb * Npad + n) * 2) = make_uint2(w[0], w[1]);
    } else {
        uint32_t w = 0x88888888u;
        if (n < N) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t k2 = kb * 4 + j;   // ui8 [K / 2, N]: low nibble k = 2 k2, high nibble k = 2 k2 + 1
                const uint32_t b = 2 * k2 < K ? (uint32_t)(q[k2 * N + n] ^ 0x88u) : 0x88u;
                w = (w & ~(0xFFu << (8 * j))) | (b << (8 * j));
            }
        }
        out[kb * Npad + n] = w;
    }
}
size_t mfma_codes_bytes(int64_t k, int64_t n, int quant) {
    return (size_t)cdiv(k, 8) * (size_t)mfma_padded_n(n) * (quant == 1 ? 8 : 4);
}
void mfma_pack_codes(hipStream_t s, const void* q, void* out, int64_t k, int64_t n, int quant) {
    const int64_t npad = mfma_padded_n(n);
    dim3 grid((unsigned)cdiv(npad, 256), (unsigned)cdiv(k, 8));
    if (quant == 1) k8_codes_kernel<1><<<grid, 256, 0, s>>>((const uint8_t*)q, (uint32_t*)out, k, n, npad);
    else k8_codes_kernel<2><<<grid, 256, 0, s>>>((const uint8_t*)q, (uint32_t*)out, k, n, npad);
}
__device__ __forceinline__ uint32_t mfma_pack_bf16(float lo, float hi) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    f32x2_t f;
    f.x = lo; f.y = hi;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2_t));   // round to nearest even
}

// Pairs' outputs from their N gates and up sums, the function that the decode kernels form (activation.rs:141-162): 28 instructions each, 4 us of a
// 256 x 256 tile's 86 more than exp2 and a reciprocal alone would take (pair of 9216, M = 8188: 789 us against 756), but those are off by up
// to 65 ulp of f32 where the gate is far below zero, against 3, and lose the result altogether from -87.4 on, where the
// reciprocal is subnormal.  The kind is looked at once, not at every output (420 us against 423 at M = 4000).
template <int N, typename G, typename U>
__device__ __forceinline__ void gemm_glu(G&& g, const U& u, const GluParams& p) {
    if (p.kind == 1) {
#pragma unroll
        for (int e = 0; e < N; ++e) g[e] = glu_combine(g[e], u[e], 1, p.limit, p.alpha, p.shift);
    } else {
#pragma unroll
        for (int e = 0; e < N; ++e) g[e] = glu_combine(g[e], u[e], 0, p.limit, p.alpha, p.shift);
    }
}

__device__ __forceinline__ float mfma_finish(float v, int act, float bias, bool has_res, float res, float colscale) {
    v += bias;                                                // tensor_ops.rs:42-56
    if (act == 1) v = (v * 0.5f) * (erff(v / 1.41421354f) + 1.0f);  // activation.rs:96-113
    v *= colscale;
    if (has_res) v += res;
    return v;
}

// Block tile BM x BN (128x128 as launched), BK = 64, four waves in a 2x2 grid; each wave owns
// (BM/2) x (BN/2) outputs as TM x TN MFMA tiles of 32x32.  LDS holds two stages of fragments,
// k-group-major ([kb][row or column][8 k], one spare row per k-group as CK does on gfx950), so a
// fragment read is a contiguous 512 bytes per half-wave.  Per k tile: one barrier; the tile after
// next is fetched global -> registers while the current one is multiplied, and the registers are
// stored into the idle LDS stage in the middle of the multiply.  Fragment reads run one k-step
// (16 k) ahead of the MFMAs that consume them.
//
// The staging registers are native vectors and every load is unconditional (the index is clamped
// instead): with HIP's uint4 struct and a guarded load the compiler keeps the staging array in
// scratch memory and waits for every load at once, which cost a factor of four.
//
// Requires K % (8 KPC) == 0 (64 for bf16, 32 for f32); M and N are guarded (rows clamp on load, stores are masked; the derived
// weights are padded to whole 128-column tiles).
// DUAL: SwiGLU pair silu(x.W) * (x.W2).  The block covers BN/2 real columns; the B tile holds, per
// wave column, TN/2 fragments of W followed by the same columns of W2, so gate and up of one
// output meet in the same lane.
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// QF: 0 = wk / wk2 hold values; 1 / 2 = they hold int8 / int4 codes (see k8_codes_kernel) and `scale` / `scale2` the
// scale tensors of the two matrices ([N] per column, or [K / 128, N] per group of 128 k), T = bf16 only.
template <typename T, int BM, int BN, bool DUAL, int QF>
__global__ __launch_bounds__(256) void gemm_mfma_kernel(const T* __restrict__ x, const T* __restrict__ wk,
                                                        const T* __restrict__ wk2, const T* __restrict__ bias,
                                                        const T* __restrict__ residual, T* __restrict__ y,
                                                        int M, int K, int N, int Npad, int act, int NT, int MT,
                                                        const T* __restrict__ scale, const T* __restrict__ scale2,
                                                        int full_tiles, int splits, float* __restrict__ part,
                                                        unsigned* __restrict__ tickets, int out_f32, EpiExtra extra) {
    constexpr int KPC = Mma<T>::KPC;
    constexpr int kBK = kKb * KPC;                            // k per tile
    typedef typename Mma<T>::frag frag_t;
    constexpr int SA = (BM + 1) * 16, SB = (BN + 1) * 16;     // bytes between k-groups
    constexpr int STAGE = kKb * (SA + SB);
    constexpr int TM = BM / 64, TN = BN / 64;
    constexpr int NTH = 256;
    constexpr int KSTEPS = kKb / 2;                           // k-steps (2 k-groups each) per wave and tile
    constexpr int CA = BM * kKb / NTH, CB = BN * kKb / NTH;   // 16-byte chunks per thread per tile
    constexpr int WN = BN / 2;                                // B-tile columns per wave column
    constexpr int NREAL = DUAL ? BN / 2 : BN;                 // output columns per block
    static_assert(!DUAL || TN % 2 == 0, "dual tiles need an even number of column fragments");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave >> 1) & 1, wn = wave & 1;
    // Tile order.  Consecutive workgroup ids go to the 8 XCDs in turn and each XCD has its own L2, so XCD c takes
    // the contiguous range [c * per, (c + 1) * per) of a grouped order in which up to 8 row blocks of one column
    // tile follow each other: the ~32 workgroups an XCD runs at a time then cover 8 row blocks x 4 column tiles, a
    // weight tile is fetched from memory once for all its row blocks (with row-major ids the 1024 column tiles of an
    // lm_head were each fetched once per row block) and an activation tile once per 4 column tiles.
    //
    // Split over k: tiles [full_tiles, total) of that order are each taken by `splits` workgroups (ids behind the whole
    // tiles' ids, so the XCDs share them) that multiply a contiguous range of k tiles each and meet through `part` and a
    // ticket per tile, see the end of the kernel.
    int bx, by;
    int t_begin = 0, t_end = K / kBK, tail = -1, split = 0;
    {
        const int total = NT * MT, per = (full_tiles + 7) / 8;
        int v;
        if (blockIdx.x < (unsigned)per * 8) {
            v = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
            if (v >= full_tiles) return;
        } else {
            const int u = (int)blockIdx.x - per * 8;
            tail = u / splits;
            split = u % splits;
            v = full_tiles + tail;
            if (v >= total) return;
            t_begin = (int)((int64_t)split * t_end / splits);
            t_end = (int)((int64_t)(split + 1) * t_end / splits);
        }
        const int gsz = 8 * NT, g = v / gsz, first = g * 8;
        const int gm = MT - first < 8 ? MT - first : 8;
        by = first + (v % gsz) % gm;
        bx = (v % gsz) / gm;
    }
    const int m0 = by * BM, n0 = bx * NREAL;

    // global -> LDS chunk assignment (16 bytes each)
    // A: chunk c -> kb = c % 8, row = c / 8: eight lanes read 128 contiguous bytes of one row
    // B: chunk c -> tile column = c % BN, kb = c / BN: contiguous runs of the k-grouped weights
    const T* a_src[CA];
    const T* b_src[CB];
    int a_dst[CA], b_dst[CB];
#pragma unroll
    for (int j = 0; j < CA; ++j) {
        const int c = tid + NTH * j;
        const int kb = c % kKb, row = c / kKb;
        int m = m0 + row;
        if (m > M - 1) m = M - 1;
        a_src[j] = x + (int64_t)m * K + kb * KPC;
        a_dst[j] = kb * SA + row * 16;
    }
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        const int c = tid + NTH * j;
        const int bc = c % BN, bkb = c / BN;
        int col = n0 + bc;
        const T* src = wk;
        if (DUAL) {
            // tile column -> (wave column, gate|up, column inside the half)
            const int wcol = bc / WN, in_w = bc % WN, half = in_w / (WN / 2), cc = in_w % (WN / 2);
            col = n0 + wcol * (WN / 2) + cc;
            src = half ? wk2 : wk;
        }
        // codes: 8 (int8) or 4 (int4) bytes per k-group and column instead of 16
        constexpr int64_t CW = QF == 0 ? KPC * (int64_t)sizeof(T) : (QF == 1 ? 8 : 4);
        b_src[j] = reinterpret_cast<const T*>(reinterpret_cast<const unsigned char*>(src) + ((int64_t)bkb * Npad + col) * CW);
        b_dst[j] = kKb * SA + bkb * SB + bc * 16;
    }
    // quantised: every chunk of a thread belongs to ONE tile column (256 % BN == 0), so one scale per thread (int8) or
    // per thread and k tile (int4: a tile of 64 k lies inside one group of 128)
    const T* s_src = nullptr;
    float q_scale = 0.f, q_scale_next = 0.f;
    if (QF != 0) {
        static_assert(NTH % BN == 0, "one tile column per thread");
        const int bc = tid % BN;
        int col = n0 + bc;
        const T* sp = scale;
        if (DUAL) {
            const int wcol = bc / WN, in_w = bc % WN, half = in_w / (WN / 2), cc = in_w % (WN / 2);
            col = n0 + wcol * (WN / 2) + cc;
            sp = half ? scale2 : scale;
        }
        if (col > N - 1) col = N - 1;   // padding columns hold the code of zero
        s_src = sp + col;
        if (QF == 1) q_scale = Mma<T>::ld(s_src, 0);
    }

    f32x16_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    u32x4_t ra[CA], rb[QF == 0 ? CB : 1];
    u32x2_t rq8[QF == 1 ? CB : 1];
    uint32_t rq4[QF == 2 ? CB : 1];
    const int nt = t_end;
    // bytes between consecutive k tiles of Wk
    const int64_t b_tile_step = (int64_t)kKb * Npad * (QF == 0 ? KPC * (int64_t)sizeof(T) : (QF == 1 ? 8 : 4));
    auto gload = [&](int t, int part, int nparts) {
#pragma unroll
        for (int j = 0; j < CA; ++j)
            if (j % nparts == part) ra[j] = *reinterpret_cast<const u32x4_t*>(a_src[j] + (int64_t)t * kBK);
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            if (j % nparts != part) continue;
            const unsigned char* p = reinterpret_cast<const unsigned char*>(b_src[j]) + (int64_t)t * b_tile_step;
            if (QF == 0) rb[j] = *reinterpret_cast<const u32x4_t*>(p);
            else if (QF == 1) rq8[j] = *reinterpret_cast<const u32x2_t*>(p);
            else rq4[j] = *reinterpret_cast<const uint32_t*>(p);
        }
        if (QF == 2 && part == nparts - 1) q_scale_next = Mma<T>::ld(s_src, (int64_t)(t * kBK / 128) * N);
    };
    // part p of NP: chunks j with j % NP == p
    auto lwrite = [&](int buf, int part, int nparts) {
        unsigned char* base = lds + buf * STAGE;
#pragma unroll
        for (int j = 0; j < CA; ++j)
            if (j % nparts == part) *reinterpret_cast<u32x4_t*>(base + a_dst[j]) = ra[j];
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            if (j % nparts != part) continue;
            u32x4_t v;
            if (QF == 0) {
                v = rb[j];
            } else if (QF == 1) {
                const float nb = -128.0f * q_scale;
                const uint32_t a = rq8[j].x, b = rq8[j].y;
                v.x = mfma_pack_bf16(__builtin_fmaf((float)(a & 0xFFu), q_scale, nb), __builtin_fmaf((float)((a >> 8) & 0xFFu), q_scale, nb));
                v.y = mfma_pack_bf16(__builtin_fmaf((float)((a >> 16) & 0xFFu), q_scale, nb), __builtin_fmaf((float)(a >> 24), q_scale, nb));
                v.z = mfma_pack_bf16(__builtin_fmaf((float)(b & 0xFFu), q_scale, nb), __builtin_fmaf((float)((b >> 8) & 0xFFu), q_scale, nb));
                v.w = mfma_pack_bf16(__builtin_fmaf((float)((b >> 16) & 0xFFu), q_scale, nb), __builtin_fmaf((float)(b >> 24), q_scale, nb));
            } else {
                const float nb = -8.0f * q_scale;
                const uint32_t c = rq4[j];
                float f[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) f[i] = __builtin_fmaf((float)((c >> (4 * i)) & 0xFu), q_scale, nb);
                v.x = mfma_pack_bf16(f[0], f[1]);
                v.y = mfma_pack_bf16(f[2], f[3]);
                v.z = mfma_pack_bf16(f[4], f[5]);
                v.w = mfma_pack_bf16(f[6], f[7]);
            }
            *reinterpret_cast<u32x4_t*>(base + b_dst[j]) = v;
        }
    };
    const int a_rd = (wm * (BM / 2) + (lane & 31)) * 16 + (lane >> 5) * SA;
    const int b_rd = kKb * SA + (wn * WN + (lane & 31)) * 16 + (lane >> 5) * SB;
    frag_t af[2][TM], bfr[2][TN];
    auto fread = [&](int buf, int kk, int slot) {
        const unsigned char* base = lds + buf * STAGE;
#pragma unroll
        for (int i = 0; i < TM; ++i) af[slot][i] = *reinterpret_cast<const frag_t*>(base + a_rd + kk * 2 * SA + i * 32 * 16);
#pragma unroll
        for (int j = 0; j < TN; ++j) bfr[slot][j] = *reinterpret_cast<const frag_t*>(base + b_rd + kk * 2 * SB + j * 32 * 16);
    };

    gload(t_begin, 0, 1);
    if (QF == 2) q_scale = q_scale_next;
    lwrite(0, 0, 1);
    gload(t_begin + 1 < nt ? t_begin + 1 : t_begin, 0, 1);
    __syncthreads();
    fread(0, 0, 0);
    // The order of issue inside a k-step is fixed by hand (the scheduling barriers): the fragments of the NEXT k-step
    // are requested before the MFMAs of this one, so their LDS latency runs under the matrix work; left to itself the
    // compiler sinks the reads below the MFMAs into the same registers and the matrix pipe waits for every fragment.
    // The tile's barrier sits between the two halves of the last k-step's MFMAs, and the first fragments of the next
    // tile are requested right behind it.
    // Unquantised operands: the stage index is a compile-time constant and the tile loop advances two tiles at a time, so
    // LDS addresses in the step loop are a register plus an immediate (vector additions beside MFMAs are not free: f32
    // M = 512, K = 3072, N = 768 63.8 -> 60.5 us).  With codes to convert the doubled loop body costs more than that
    // saves (int4: +4-8 %), so those keep the index in a register.
    auto tile_step = [&](auto stage, int t) {
        const int cur = stage;
#pragma unroll
        for (int kk = 0; kk < KSTEPS; ++kk) {
            if (kk + 1 < KSTEPS) fread(cur, kk + 1, (kk + 1) & 1);
            // tile t+1 goes registers -> LDS (codes are converted on the way) and tile t+2 memory -> registers a quarter
            // of the chunks per k-step, between the MFMAs; past the last tile this stores a copy nobody reads
            if (QF == 2 && kk == 0) q_scale = q_scale_next;   // the scale that came with tile t+1
            lwrite(cur ^ 1, kk, KSTEPS);
            gload(t + 2 < nt ? t + 2 : nt - 1, kk, KSTEPS);
            __builtin_amdgcn_sched_barrier(0);
            if (kk + 1 < KSTEPS) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = Mma<T>::mma(af[kk & 1][i], bfr[kk & 1][j], acc[i][j]);
            } else {
                static_assert(((KSTEPS - 1) & 1) == 1, "the last k-step's fragments are in slot 1, the next tile's first in slot 0");
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN / 2; ++j)
                        acc[i][j] = Mma<T>::mma(af[kk & 1][i], bfr[kk & 1][j], acc[i][j]);
                __builtin_amdgcn_sched_barrier(0);
                __syncthreads();
                fread(cur ^ 1, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = TN / 2; j < TN; ++j)
                        acc[i][j] = Mma<T>::mma(af[kk & 1][i], bfr[kk & 1][j], acc[i][j]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if constexpr (QF == 0) {
        int t = t_begin;
        for (; t + 2 <= nt; t += 2) {
            tile_step(std::integral_constant<int, 0>{}, t);
            tile_step(std::integral_constant<int, 1>{}, t + 1);
        }
        if (t < nt) tile_step(std::integral_constant<int, 0>{}, t);
    } else {
        for (int t = t_begin; t < nt; ++t) tile_step((t - t_begin) & 1, t);
    }

    if (tail >= 0) {
        // Partial sums of a split tile go to the workspace, [item][value][thread], through device-scope stores (coherent
        // across the L2s of the XCDs without cache maintenance); once they are acknowledged the workgroup draws the
        // tile's ticket.  The one that draws the last ticket adds all partials in split order, its own included, so
        // the result does not depend on which workgroup that is, leaves the ticket at zero and runs the epilogue.
        constexpr int E = TM * TN * 16;
        float* mine = part + ((int64_t)(tail * splits + split) * E) * 256 + tid;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    __hip_atomic_store(mine + ((i * TN + j) * 16 + v) * 256, acc[i][j][v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_waitcnt(0x0F70);                         // vmcnt(0)
        asm volatile("" ::: "memory");
        unsigned* flag = reinterpret_cast<unsigned*>(lds);          // the tiles in LDS are dead (the loop ended on a barrier)
        __syncthreads();
        if (tid == 0) *flag = __hip_atomic_fetch_add(&tickets[tail], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*flag != (unsigned)(splits - 1)) return;
        asm volatile("" ::: "memory");                              // the partials are read after the ticket is known
        if (tid == 0) __hip_atomic_store(&tickets[tail], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
        for (int q = 0; q < splits; ++q) {
            const float* src = part + ((int64_t)(tail * splits + q) * E) * 256 + tid;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        acc[i][j][v] += __hip_atomic_load(src + ((i * TN + j) * 16 + v) * 256, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // epilogue: lane holds column (lane % 32), rows 8*(v/4) + 4*(lane/32) + v%4 of each 32x32 tile (passing the sums
    // through LDS to store rows of 8, as the LDS-direct kernel below does, changed nothing here: 19.0 against 19.1 us at
    // K = 192, M = 1024, N = 6144)
    constexpr int TNO = DUAL ? TN / 2 : TN;
    if constexpr (DUAL) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TNO; ++j) gemm_glu<16>(acc[i][j], acc[i][j + TNO], extra.glu);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TNO; ++j) {
            const int n = n0 + wn * (NREAL / 2) + j * 32 + (lane & 31);
            if (n >= N) continue;
            const float bv = bias ? Mma<T>::ld(bias, n) : 0.f;
            const float cs = extra.colscale ? extra.colscale[n] : 1.0f;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int m = m0 + wm * (BM / 2) + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                if (m >= M) continue;
                // out_f32: the f32 accumulator (plus an f32 residual) is stored as it is
                const float r = residual ? (out_f32 ? reinterpret_cast<const float*>(residual)[(int64_t)m * N + n]
                                                    : Mma<T>::ld(residual, (int64_t)m * N + n)) : 0.f;
                const float o = mfma_finish(acc[i][j][v], act, bv, residual != nullptr, r, cs);
                if (out_f32) reinterpret_cast<float*>(y)[(int64_t)m * N + n] = o;
                else Mma<T>::st(y, (int64_t)m * N + n, o);
            }
        }
}

// ---------------------------------------------------------------------------------------------------------------
// GEMM whose tiles go memory -> LDS without passing through registers (global_load_lds_dwordx4), for unquantised bf16 and f32
// operands: no staging registers, no LDS store instructions, loads run NST - 1 k tiles ahead through a ring.  Sizes below are
// those of bf16; f32 has 4 k where bf16 has 8 and moves the same bytes.
//
// Workgroup: WM x WN waves; a wave owns (32 TM) x (32 TN) outputs as TM x TN fragments of 32 x 32, the tile is
// BM x BN = (32 TM WM) x (32 TN WN).  KW = 2: two such groups of waves share the staged tiles, each multiplies half of every k tile, and
// their sums meet through LDS in front of the epilogue.  A bf16 launch takes one of eight tiles and a number of splits over k, see tile_plan().
//
// What bounds it (bf16).  256 x 256 tiles, all CUs busy: the matrix pipes at the clock that random operands allow.  A tile's 32 k
// take 0.54 us on a quarter of the CUs and 0.8 us on all of them; over all-zero operands the same launch runs at 1.35 times
// the rate (M = 8188, K = 3072, N = 6144: 1680 against 1240 TFLOP/s), so it is power and not data that paces it.  Why 256 x
// 256: a k tile moves 1 / (2 BM) + 1 / (2 BN) bytes per flop from the L2s into LDS and as many fragments from LDS into
// registers, 5/6 of what 128 x 192 needs twice over; 8 waves of 128 x 64 read 6 fragments for 8 MFMAs (64 x 96: 5 for 6,
// each k-group its own).  Against the 128 x 192 tiles (two k-groups of 2 x 2 waves) that ran here before, us in a traced
// 26-layer prompt: M = 8188 qkv 340 -> 263, gate/up pair 1010 -> 798, out and down 337 (mean) -> 208 and 414; M = 333 (few tiles,
// weights from memory) qkv 32 -> 28, out and down 51 (mean) -> 29 with the launch that adds the splits, pair 81 -> 51.  k tiles of 32 in a ring of four beat k tiles of 64 in
// a ring of two there (1035 -> 1239 TFLOP/s: loads have three k tiles of time, not one); 4 waves of 128 x 128 lose (1090).
// Smaller tiles are for launches whose 256 x 256 tiles would leave CUs without work; they stage 64 k, the memory's lines.
// 128 x 192 in two k-groups of 2 x 2 waves: 8 waves that still read 5 fragments for 6 MFMAs (8 waves of 32 x 96 read 4 for 3, more than LDS
// delivers), for launches that its tiles fill in whole rounds: M = 1000, weights from memory, us against the best of the other six: N = 6144
// 44.6 -> 40.5, pair of 9216 153 -> 129, K = 9216 68 -> 64; M = 2047, K = 9216 117 -> 105; M = 6000, K = 9216 359 -> 304.
//
// LDS, per stage: A as rows of 2 BK bytes, B k-group-major ([k-group][column][8 k]).  One load instruction moves
// 64 x 16 bytes to 1 KiB of consecutive LDS, lane l to byte 16 l, so the layout is fixed by WHICH 16 bytes of memory a
// lane asks for: in A, position p of row r holds k-group p ^ swz(r), with swz(r) such that 16 consecutive rows of a
// fragment read (32 rows x 2 k-groups) touch every bank once; BK / 8 lanes still read one row's 2 BK contiguous bytes.
// B fragments are contiguous as they are.
//
// Order of issue, fixed by hand with scheduling barriers: the fragments of the next k-step are requested before the
// MFMAs of this one; in a tile's last k-step half the MFMAs are issued, then the wave waits for its own loads of the
// next tile (vmcnt, which counts only LDS-direct loads here), passes the barrier that makes that tile complete and this
// one free, requests the next tile's first fragments, issues the other half and, behind it, requests the tile NST
// ahead into the freed stage.  Nothing is requested past the last tile; from there on the wave waits for everything.
// MFMAs run at raised wave priority, so that the two waves of a SIMD take turns instead of stalling on each other's LDS
// reads (k tiles of 64: 1035 -> 1167 TFLOP/s; of 32: within the noise).
// DUAL (SwiGLU pair): the tile's first BN / 2 columns are columns of W, the others the same columns of W2, and a wave
// multiplies the same 16 TN columns of both, so gate and up of an output meet in one lane; with an odd TN wave column 0 multiplies
// W and wave column 1 W2, and they meet in the epilogue's LDS.
// One load instruction: lane l asks for the 16 bytes at base + offset(l) (a scalar base and a 32-bit offset per lane, so
// stepping to the next k tile is scalar arithmetic; vector instructions in the step loop cost the matrix pipe issue
// slots: per-lane 64-bit addresses were 5-10 % slower) and they land at LDS byte lds_addr + 16 l.
__device__ __forceinline__ void gemm_lds_load16(unsigned voff, unsigned long long sbase, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(sbase), "s"(lds_addr) : "memory", "m0");
}
__device__ __forceinline__ unsigned long long gemm_uniform64(unsigned long long p) {
    return ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(p >> 32)) << 32) |
           (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)p);
}
template <int N> __device__ __forceinline__ void gemm_wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }

// What happens to a sum on its way out (a pair has been combined before).
template <typename T>
struct TileEpilogue {
    const T* bias; const void* residual; void* y;
    int64_t N;
    int act, out_f32;
    EpiExtra extra;
};
// Eight neighbours of row m, columns n .. n + 7, from LDS: bias, GELU, column factor and residual, then one 16-byte store (two
// for f32 results; element by element when N is not a multiple of 8).  Kept short: with every output's options unrolled the
// epilogue was 13 000 to 18 000 instructions, more than the instruction cache holds (M = 8188, see gemm_tile_kernel).
// PAIR: `at_lds` holds gates and `up_lds` the up sums, still to be combined.
template <typename T, bool PAIR>
__device__ __forceinline__ void gemm_finish8(const TileEpilogue<T>& p, int64_t m, int64_t n, const float* at_lds, const float* up_lds) {
    const int64_t at = m * p.N + n;
    const bool f32 = std::is_same<T, float>::value || p.out_f32;     // y and residual
    if ((p.N & 7) != 0) {
#pragma unroll 1
        for (int e = 0; e < 8; ++e) {
            if (n + e >= p.N) break;
            const float bv = p.bias ? Mma<T>::ld(p.bias, n + e) : 0.f;
            const float rv = p.residual ? (f32 ? static_cast<const float*>(p.residual)[at + e] : Mma<T>::ld(static_cast<const T*>(p.residual), at + e)) : 0.f;
            float sum[1] = {at_lds[e]};
            if constexpr (PAIR) gemm_glu<1>(sum, up_lds + e, p.extra.glu);
            const float f = mfma_finish(sum[0], p.act, bv, p.residual != nullptr, rv, p.extra.colscale ? p.extra.colscale[n + e] : 1.0f);
            if (f32) static_cast<float*>(p.y)[at + e] = f;
            else Mma<T>::st(static_cast<T*>(p.y), at + e, f);
        }
        return;
    }
    float o[8];
    *reinterpret_cast<f32x4_t*>(o) = *reinterpret_cast<const f32x4_t*>(at_lds);
    *reinterpret_cast<f32x4_t*>(o + 4) = *reinterpret_cast<const f32x4_t*>(at_lds + 4);
    if constexpr (PAIR) {
        float u[8];
        *reinterpret_cast<f32x4_t*>(u) = *reinterpret_cast<const f32x4_t*>(up_lds);
        *reinterpret_cast<f32x4_t*>(u + 4) = *reinterpret_cast<const f32x4_t*>(up_lds + 4);
        gemm_glu<8>(o, u, p.extra.glu);
    }
    auto add_f32 = [&](const float* v) {
        const f32x4_t r0 = *reinterpret_cast<const f32x4_t*>(v), r1 = *reinterpret_cast<const f32x4_t*>(v + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) { o[e] += r0[e]; o[4 + e] += r1[e]; }
    };
    auto add_bf16 = [&](const void* v) {
        const u32x4_t w = *static_cast<const u32x4_t*>(v);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o[2 * e] += __uint_as_float(w[e] << 16);
            o[2 * e + 1] += __uint_as_float(w[e] & 0xFFFF0000u);
        }
    };
    if (p.bias) {                                                    // tensor_ops.rs:42-56
        if constexpr (std::is_same<T, float>::value) add_f32(p.bias + n);
        else add_bf16(p.bias + n);
    }
    if (p.act == 1) {
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (o[e] * 0.5f) * (erff(o[e] / 1.41421354f) + 1.0f);   // activation.rs:96-113
    }
    if (p.extra.colscale) {
        const f32x4_t c0 = *reinterpret_cast<const f32x4_t*>(p.extra.colscale + n), c1 = *reinterpret_cast<const f32x4_t*>(p.extra.colscale + n + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) { o[e] *= c0[e]; o[4 + e] *= c1[e]; }
    }
    if (p.residual) {
        if (f32) add_f32(static_cast<const float*>(p.residual) + at);
        else add_bf16(static_cast<const bf16_t*>(p.residual) + at);
    }
    if (f32) {
        *reinterpret_cast<f32x4_t*>(static_cast<float*>(p.y) + at) = *reinterpret_cast<const f32x4_t*>(o);
        *reinterpret_cast<f32x4_t*>(static_cast<float*>(p.y) + at + 4) = *reinterpret_cast<const f32x4_t*>(o + 4);
    } else {
        u32x4_t w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = mfma_pack_bf16(o[2 * e], o[2 * e + 1]);
        *reinterpret_cast<u32x4_t*>(static_cast<bf16_t*>(p.y) + at) = w;
    }
}
template <typename T, int KG, int NST, int WM, int WN, int KW, int TM, int TN, bool DUAL, int QF>
__global__ __launch_bounds__(64 * WM * WN * KW) void gemm_tile_kernel(const T* __restrict__ x, const T* __restrict__ wk, const T* __restrict__ wk2,
                                                                 int M, int K, int Npad, int row0, int col0, int NT, int MT, int splits, float* __restrict__ part, const T* __restrict__ scale, const T* __restrict__ scale2,
                                                                 TileEpilogue<T> epi) {
    static_assert(KG == 4 || KG == 8, "k-groups of a k tile");
    typedef typename Mma<T>::frag frag_t;
    constexpr int BK = KG * Mma<T>::KPC, ROWB = KG * 16, KS = KG / 2;  // k of a tile, bytes of an A row, k-steps
    constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN, NW = WM * WN * KW;
    constexpr int NREAL = DUAL ? BN / 2 : BN;                          // output columns per tile
    constexpr bool ACROSS = DUAL && TN % 2 != 0;                       // a pair's matrices are the two wave columns, not halves of a wave's fragments
    constexpr int TNO = DUAL && !ACROSS ? TN / 2 : TN;                 // output fragments per wave and row
    constexpr int KSW = KS / KW, TMO = TM / KW;                        // k-steps of a k-group of waves; rows of fragments that a wave finishes
    constexpr int CB = QF == 0 ? 16 : QF == 1 ? 8 : 4;                 // bytes of a column's k-group
    constexpr int A_BYTES = BM * ROWB, B_BYTES = BN * KG * CB, STAGE = A_BYTES + B_BYTES;
    constexpr int LAI = A_BYTES / 1024, LBI = B_BYTES / 1024;          // load instructions per tile
    constexpr int LA = LAI / NW, LB = (LBI + NW - 1) / NW, LPT = LA + LB;   // per wave (with fewer instructions than waves, two waves bring the same)
    static_assert(LA * NW == LAI && LBI * 1024 == B_BYTES && (LB * NW == LBI || NW % LBI == 0), "whole load instructions per wave");
    static_assert(QF == 0 || (KG == 8 && std::is_same<T, bf16_t>::value), "codes: bf16 activations, k tiles of 64");
    static_assert(KSW % 2 == 0, "the last k-step's fragments sit in slot 1, the next tile's first in slot 0");
    static_assert(!DUAL || NREAL * KG * CB % 1024 == 0, "a load instruction belongs to one matrix of the pair");
    static_assert(KW == 1 || (KW == 2 && TM % 2 == 0 && QF == 0 && std::is_same<T, bf16_t>::value), "two k-groups halve the rows of their sums");
    static_assert(!DUAL || ACROSS || KW == 1, "a wave's own pairs are combined where they were summed");
    static_assert(!ACROSS || (WN == 2 && TMO == 1 && QF == 0), "wave column 0 multiplies W, wave column 1 the same columns of W2");
    static_assert((NST - 2) * LPT < 64, "vmcnt is a 6-bit counter");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wg = KW == 1 ? 0 : wave / (WM * WN), wq = KW == 1 ? wave : wave % (WM * WN);   // k-group; place in it
    const int wm = wq / WN, wn = wq % WN;
    int bx, by, sidx;
    {
        // XCD c takes a contiguous range of a grouped tile order (see gemm_mfma_kernel: 8 row blocks by 4 column tiles run on
        // an XCD at a time; groups of 4 or 32 row blocks are 3-10 % slower at M = 8188); `splits` neighbours of that order
        // share a tile and take a contiguous range of its k tiles each
        const int total = NT * MT * splits, per = (total + 7) / 8;
        const int u = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
        if (u >= total) return;
        const int v = u / splits;
        sidx = u % splits;
        const int gsz = 8 * NT, g = v / gsz, first = g * 8;
        const int gm = MT - first < 8 ? MT - first : 8;
        by = first + (v % gsz) % gm;
        bx = (v % gsz) / gm;
    }
    const int m0 = row0 + by * BM, n0 = col0 + bx * NREAL;   // the tiles cover NT columns and MT rows of them from (row0, col0) on
    auto swz = [](int row) { return KG == 8 ? (row >> 1) & 7 : (row >> 2) & 3; };
    // what each of this wave's load instructions fetches, per lane
    unsigned a_off[LA], b_off[LB];
    unsigned long long b_base[LB];
#pragma unroll
    for (int j = 0; j < LA; ++j) {
        const int sl = (wave * LA + j) * 64 + lane, row = sl / KG, pos = sl % KG;
        int m = m0 + row;
        if (m > M - 1) m = M - 1;
        a_off[j] = (unsigned)(m - m0) * (unsigned)(K * sizeof(T)) + (unsigned)((pos ^ swz(row)) * 16);   // under 256 rows: fits 32 bits (K <= 2^21)
    }
#pragma unroll
    for (int j = 0; j < LB; ++j) {
        const int q = (wave * LB + j) % LBI, half = q * 1024 / (NREAL * KG * CB), at = q * 1024 - half * (NREAL * KG * CB) + lane * 16;
        const int kg = at / (NREAL * CB);
        int col = n0 + at % (NREAL * CB) / CB;                           // first of the 16 / CB columns that 16 bytes hold
        if (col > Npad - 16 / CB) col = Npad - 16 / CB;
        b_base[j] = (unsigned long long)(DUAL && half ? wk2 : wk);
        b_off[j] = (unsigned)(((unsigned long long)kg * Npad + col) * CB);
    }
    const unsigned long long a_base = (unsigned long long)(x + (int64_t)m0 * K);
    const int64_t b_tile_step = (int64_t)KG * Npad * CB;
    const unsigned lds0 = (unsigned)(uintptr_t)lds;
    const int kt_all = K / BK, kt0 = (int)((int64_t)sidx * kt_all / splits);
    const int nt = (int)((int64_t)(sidx + 1) * kt_all / splits) - kt0;   // this workgroup's k tiles: [kt0, kt0 + nt)
    auto issue = [&](int t, int st) {
        if (t >= nt) return;
        const unsigned long long ab = gemm_uniform64(a_base + (unsigned long long)(t + kt0) * ROWB);
        const unsigned long long bt = (unsigned long long)((t + kt0) * b_tile_step);
        const unsigned sbase = lds0 + st * STAGE;
#pragma unroll
        for (int j = 0; j < LA; ++j) gemm_lds_load16(a_off[j], ab, (unsigned)__builtin_amdgcn_readfirstlane((int)(sbase + (wave * LA + j) * 1024)));
#pragma unroll
        for (int j = 0; j < LB; ++j) gemm_lds_load16(b_off[j], gemm_uniform64(b_base[j] + bt), (unsigned)__builtin_amdgcn_readfirstlane((int)(sbase + A_BYTES + (wave * LB + j) % LBI * 1024)));
    };
    // f32 adds the two halves of every k tile apart: half as many roundings in a row, and the registers are there (K = 3072:
    // 7.0e-7 of the result's norm away from 64 bits, in one chain 9.9e-7; K = 768 3.5e-7 and 5.0e-7)
    constexpr int CHAINS = std::is_same<T, float>::value ? 2 : 1;
    f32x16_t sums[CHAINS][TM][TN];
    f32x16_t (&acc)[TM][TN] = sums[0];
#pragma unroll
    for (int c = 0; c < CHAINS; ++c)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) sums[c][i][j][v] = 0.f;
    const int fsel = lane >> 5;
    const int b_rd = A_BYTES + (ACROSS ? wn * (NREAL * KG * CB) : wn * 32 * TNO * CB) + (lane & 31) * CB;
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    typedef typename std::conditional<QF == 0, frag_t, typename std::conditional<QF == 1, u32x2_t, uint32_t>::type>::type raw_t;
    frag_t af[2][TM], bq[QF == 0 ? 1 : TN];
    raw_t bfr[2][TN];
    // the codes' scales: one per column (int8), or one per column and 128 k (int4), the latter for all of this workgroup's k in LDS
    float sc[QF == 0 ? 1 : TN];
    bf16_t* sc_lds = reinterpret_cast<bf16_t*>(lds + NST * STAGE);
    if constexpr (QF == 1) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int col = n0 + (wn * TNO + j % TNO) * 32 + (lane & 31);
            sc[j] = Mma<T>::ld(DUAL && j >= TNO ? scale2 : scale, col < (int)epi.N ? col : (int)epi.N - 1);
            asm volatile("" : : "v"(sc[j]));                             // arrived before the ring's loads are counted
        }
    }
    if constexpr (QF == 2) {
        const int groups = (kt0 + nt - 1) / 2 - kt0 / 2 + 1;
#pragma unroll 4
        for (int e = tid; e < groups * BN; e += 64 * NW) {
            const int g = kt0 / 2 + e / BN, c = e % BN, col = n0 + (DUAL ? c % NREAL : c);
            sc_lds[e] = (DUAL && c >= NREAL ? scale2 : scale)[(int64_t)g * epi.N + (col < epi.N ? col : epi.N - 1)];
        }
    }
    auto fread = [&](int st, int kw, int slot) {   // kw: k-step of the k-group
        const int kk = wg * KSW + kw;
        const unsigned char* base = lds + st * STAGE;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int row = wm * 32 * TM + i * 32 + (lane & 31), kg = 2 * kk + fsel;
            af[slot][i] = *reinterpret_cast<const frag_t*>(base + row * ROWB + ((kg ^ swz(row)) * 16));
        }
#pragma unroll
        for (int j = 0; j < TN; ++j)
            bfr[slot][j] = *reinterpret_cast<const raw_t*>(base + b_rd + (2 * kk + fsel) * (NREAL * CB) + (j / TNO) * (NREAL * KG * CB) + (j % TNO) * 32 * CB);   // ACROSS: j < TNO
    };
    // codes -> the bf16 values of the dequantised matrix, bf16(code * scale): u * s - bias * s is exactly (u - bias) * s, rounded
    // once like the product the dequantiser forms
    auto dequantise = [&](int slot) {
        if constexpr (QF != 0) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                float f[8];
                const float nb = (QF == 1 ? -128.0f : -8.0f) * sc[j];
                uint32_t w[2];
                if constexpr (QF == 1) { w[0] = bfr[slot][j].x; w[1] = bfr[slot][j].y; }
                else { w[0] = bfr[slot][j] & 0x0F0F0F0Fu; w[1] = (bfr[slot][j] >> 4) & 0x0F0F0F0Fu; }   // codes 0, 2, 4, 6 and 1, 3, 5, 7
#pragma unroll
                for (int e = 0; e < 8; ++e) f[QF == 1 ? e : 2 * (e & 3) + (e >> 2)] = __builtin_fmaf((float)((w[e >> 2] >> (8 * (e & 3))) & 0xFFu), sc[j], nb);
                u32x4_t v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = mfma_pack_bf16(f[2 * e], f[2 * e + 1]);
                bq[j] = __builtin_bit_cast(frag_t, v);
            }
        }
    };
    for (int st = 0; st < NST - 1; ++st) issue(st, st);
    if (nt >= NST - 1) gemm_wait_loads<(NST - 2) * LPT>();
    else gemm_wait_loads<0>();
    __syncthreads();
    issue(NST - 1, NST - 1);
    fread(0, 0, 0);
    // One k tile; the ring position is a compile-time constant (the tile loop below is unrolled over the ring), so every
    // LDS address of the step loop is a register plus an immediate.
    auto tile_step = [&](auto ring_pos, int t) {
        constexpr int ST = decltype(ring_pos)::value, ST1 = ST + 1 == NST ? 0 : ST + 1;
        auto mul = [&](int slot, int i0, int i1, int chain) {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    if (i * TN + j >= i0 && i * TN + j < i1) {
                        f32x16_t& to = sums[chain & (CHAINS - 1)][i][j];
                        if constexpr (QF == 0) to = Mma<T>::mma(af[slot][i], bfr[slot][j], to);
                        else to = Mma<T>::mma(af[slot][i], bq[j], to);
                    }
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
        };
        if constexpr (QF == 2) {
            const int g = (t + kt0) / 2 - kt0 / 2;
#pragma unroll
            for (int j = 0; j < TN; ++j) sc[j] = bf16_to_f32(sc_lds[g * BN + (j / TNO) * NREAL + (wn * TNO + j % TNO) * 32 + (lane & 31)]);
        }
#pragma unroll
        for (int kk = 0; kk + 1 < KSW; ++kk) {
            fread(ST, kk + 1, (kk + 1) & 1);
            dequantise(kk & 1);
            mul(kk & 1, 0, TM * TN, 2 * kk / KSW);
        }
        dequantise(1);
        mul(1, 0, TM * TN / 2, 1);
        if (t + NST - 1 < nt) gemm_wait_loads<(NST - 2) * LPT>();   // the loads of tiles t + 2 .. t + NST - 1 may be on their way
        else gemm_wait_loads<0>();
        __syncthreads();
        fread(ST1, 0, 0);
        mul(1, TM * TN / 2, TM * TN, 1);
        issue(t + NST, ST);   // behind the MFMAs: the address arithmetic and the requests run under them (6 % faster than ahead of them)
        __builtin_amdgcn_sched_barrier(0);
    };
    static_assert(NST >= 2 && NST <= 4, "the tile loop is unrolled over the ring");
    {
        constexpr std::integral_constant<int, 0> R0{};
        constexpr std::integral_constant<int, 1> R1{};
        constexpr std::integral_constant<int, NST == 2 ? 0 : 2> R2{};
        constexpr std::integral_constant<int, NST - 1> R3{};
        int t = 0;
        for (; t + NST <= nt; t += NST) {
            tile_step(R0, t);
            tile_step(R1, t + 1);
            if constexpr (NST > 2) tile_step(R2, t + 2);
            if constexpr (NST > 3) tile_step(R3, t + 3);
        }
        if (t < nt) tile_step(R0, t);
        if constexpr (NST > 2)
            if (t + 1 < nt) tile_step(R1, t + 1);
        if constexpr (NST > 3)
            if (t + 2 < nt) tile_step(R2, t + 2);
    }
#pragma unroll
    for (int c = 1; c < CHAINS; ++c)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] += sums[c][i][j];
    // two k-groups: group g gives the sums of the other half of its rows of fragments away and keeps half g, through LDS (the staged tiles
    // are dead: nothing is in flight, and every wave has read its last fragments in front of the last step's barrier)
    f32x16_t kept[KW == 1 ? 1 : TMO][KW == 1 ? 1 : TN];
    if constexpr (KW == 2) {
        constexpr int XCH = TMO * TN * 16 * 64;
        float* give = reinterpret_cast<float*>(lds) + wave * XCH + lane;
        const float* take = reinterpret_cast<const float*>(lds) + (wg == 0 ? wave + WM * WN : wave - WM * WN) * XCH + lane;
        auto hand_over = [&](int from) {
#pragma unroll
            for (int i = 0; i < TMO; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) give[((i * TN + j) * 16 + v) * 64] = acc[from + i][j][v];
        };
        auto keep = [&](int from) {
#pragma unroll
            for (int i = 0; i < TMO; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) kept[i][j][v] = acc[from + i][j][v] + take[((i * TN + j) * 16 + v) * 64];
        };
        if (wg == 0) hand_over(TMO);
        else hand_over(0);
        __syncthreads();
        if (wg == 0) keep(0);
        else keep(TMO);
        __syncthreads();   // every wave has taken its half before the area is written again
    }
    auto sum = [&](int i, int j, int v) {
        if constexpr (KW == 1) return acc[i][j][v];
        else return kept[i][j][v];
    };
    const int mw = m0 + (wm * TM + wg * TMO) * 32, nw = n0 + (ACROSS ? 0 : wn * 32 * TNO);   // the wave's first output
    if (splits > 1) {
        // partial sums, [split][row][columns padded to 8] f32 (a pair: W's columns, then W2's); gemm_reduce_kernel adds them
        const int np = ((int)epi.N + 7) & ~7, width = DUAL ? 2 * np : np;
#pragma unroll
        for (int i = 0; i < TMO; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = nw + (j % TNO) * 32 + (lane & 31);
                if (n >= np) continue;
                float* to = part + (int64_t)sidx * M * width + (ACROSS ? wn * np : DUAL ? (j / TNO) * np : 0) + n;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int m = mw + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                    if (m < M) to[(int64_t)m * width] = sum(i, j, v);
                }
            }
        return;
    }
    // Rows of 8 outputs: 32 x (32 TNO) sums at a time go through an LDS area of the wave's own (a lane holds one column of
    // four-row groups, memory wants runs along a row).  ACROSS: the two waves of a pair meet here, each takes half of the chunks and reads both areas.
    constexpr int RSF = 32 * TNO + 4;    // floats per row of an area
    constexpr int CH = 4 * TNO;          // chunks of 8 per row
    constexpr int PASSES = ACROSS ? CH / 4 : CH / 2;
    static_assert(!ACROSS || CH % 4 == 0, "whole passes of either wave");
    float* area = reinterpret_cast<float*>(lds) + wave * (32 * RSF);
    const float* gates = ACROSS ? area - wn * (32 * RSF) : area;
#pragma unroll
    for (int i = 0; i < TMO; ++i) {
#pragma unroll
        for (int j = 0; j < TNO; ++j) {
            if constexpr (DUAL && !ACROSS) gemm_glu<16>(acc[i][j], acc[i][j + TNO], epi.extra.glu);
#pragma unroll
            for (int v = 0; v < 16; ++v)
                area[(8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)) * RSF + j * 32 + (lane & 31)] = sum(i, j, v);
            }
        if (ACROSS) __syncthreads();
#pragma unroll 1
        for (int it = 0; it < PASSES; ++it) {
            const int c = (ACROSS ? wn * PASSES + it : it) * 64 + lane, r = c / CH, cc = c % CH;
            const int m = mw + i * 32 + r, n = nw + cc * 8;
            if (m < M && n < epi.N) gemm_finish8<T, ACROSS>(epi, m, n, gates + r * RSF + cc * 8, gates + 32 * RSF + r * RSF + cc * 8);
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// f32 layers of more than 128 rows, on the bf16 matrix cores.  An f32 value is the sum of three bf16 values, a = a1 + a2 + a3 exactly (8 bits of
// its 24 each, rounded to nearest, so |a2| <= 2^-8 |a| and |a3| <= 2^-17 |a|), and a product is
//   a b = a1 b1 + (a1 b2 + a2 b1) + (a2 b2 + a1 b3 + a3 b1) + what is left out: a2 b3 + a3 b2 + a3 b3 < 2^-23.9 |a b|,
// six bf16 products, each exact in f32.  The bf16 cores are 16 times as fast as the f32 cores, so six cost 0.375 of one f32 product.
//
// Precision.  What is left out is 2^-27 of a product in the mean square, far below the roundings of the sum.  a1 b1 and the five small products are
// summed apart (the small sum's roundings are 2^-8 of the large one's), and a sum of K terms is rounded about K / 8 times, where the f32
// cores round it K / 2 times.  Distance from 64 bits over the result's norm, normal operands: K = 768 1.6e-7 (f32 cores, two chains of sums: 3.5e-7; all
// six products in one chain: 4.2e-7), K = 3072 3.4e-7 (7.0e-7; 9.0e-7).
// Range.  bf16 has f32's exponents, so the second and third values of a small f32 value run out of them (below 2^-103 bits go, at 2^-120 eleven of 24
// or more).  Both operands are therefore split times 2^24, where every bit of every f32 value, subnormals too, is a normal bf16 value's, and the sums are
// divided by 2^48: powers of two, no rounding but a subnormal result's.  The eight multiplications more for a fragment's 8 values take 16 prompts of 512 through
// GPT-2 small from 11.01 to 11.13 ms (the matrix cores would flush subnormal pieces: without the scale rows or weights of 2^-135 were multiplied as zeros).
// Infinities, NaN, values from 2^104 on and sums from 2^80 on leave a scaled sum that is not finite (an infinity's second value is a NaN); such a sum is formed
// again, on the f32 cores, before anything is made of it.
//
// The weights are split once, into Ws[K/8][plane][Npad][8] (6 bytes a weight); the rows are staged in f32 and every wave splits the fragments it
// multiplies, 52 vector instructions for 8 values, so a wave takes one row of fragments and all of a large tile's columns: 256 x 96 in 8 waves of 32 x 96
// (18 MFMAs per 52), two k-steps of 16 to a staged tile; 128 x 96 in 4, one k-step, two workgroups to a CU; and 64 x 64 in 4 waves of 32 x 32 for
// launches of few rows (two k-steps: one barrier for 12 MFMAs, not 6; K = 768 in one round 19 -> 14.5 us).
// What bounds it: with the chip full, the matrix pipes at the clock that random operands allow (256 x 96 at M = 8192, K = 3072, N = 768: 211
// TFLOP/s = 1270 of bf16, the rate of the bf16 tiles); with K = 768 the tile's first loads and its epilogue.  us, programs of one layer, M = 8192, weights from memory, f32
// cores and this: K = 768, N = 3072 291 -> 205, N = 2304 217 -> 154, N = 768 81 -> 52; K = 3072, N = 768 302 -> 183; M = 1000, K = 768, N = 3072 46 -> 41;
// M = 512, N = 2304 29 -> 24.  Inside 16 prompts of 512 through GPT-2 small (14.07 -> 10.53 ms) the same layers take 241 (with GELU), 169 and, the last two in the
// mean, 131.  Dropped: 64 x 64 per wave (88 vector
// instructions per 24 MFMAs: 177 TFLOP/s against 193), 32 x 128 (the small products' own sums no longer fit the registers), fragments split a k tile
// ahead of their use, a ring of six (no change).
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;
__global__ __launch_bounds__(256) void split_weights_kernel(const float* __restrict__ w, bf16_t* __restrict__ out, int64_t K, int64_t N, int64_t Npad) {
    const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t kb = blockIdx.y;
    if (n >= Npad) return;
    alignas(16) bf16_t r[3][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int64_t kx = kb * 8 + i;
        float v = n < N && kx < K ? w[kx * N + n] * kSplitScale : 0.f;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            r[q][i] = f32_to_bf16(v);
            v -= bf16_to_f32(r[q][i]);
        }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<uint4*>(out + ((kb * 3 + q) * Npad + n) * 8) = *reinterpret_cast<const uint4*>(r[q]);
}
size_t mfma_split_bytes(int64_t k, int64_t n) { return (size_t)cdiv(k, 8) * 3 * (size_t)mfma_padded_n(n) * 16; }
void mfma_split_weights(hipStream_t s, const void* w, void* out, int64_t k, int64_t n) {
    const int64_t npad = mfma_padded_n(n);
    split_weights_kernel<<<dim3((unsigned)cdiv(npad, 256), (unsigned)cdiv(k, 8)), 256, 0, s>>>((const float*)w, (bf16_t*)out, k, n, npad);
}
struct SplitOperands {
    const float* x; const bf16_t* wp; const bf16_t* wp2;
    int K, Npad;
    const float* w; const float* w2;   // the same weights row-major, [K, N]
};
__device__ __forceinline__ void split_rows8(const f32x4_t& r0, const f32x4_t& r1, bf16x8_t* out) {
    u32x4_t p[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float lo = (e < 2 ? r0[2 * e] : r1[2 * e - 4]) * kSplitScale, hi = (e < 2 ? r0[2 * e + 1] : r1[2 * e - 3]) * kSplitScale;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            p[q][e] = mfma_pack_bf16(lo, hi);
            if (q < 2) {
                lo -= __uint_as_float(p[q][e] << 16);
                hi -= __uint_as_float(p[q][e] & 0xFFFF0000u);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) out[q] = __builtin_bit_cast(bf16x8_t, p[q]);
}

// WM x WN waves of 32 x (32 TN) outputs; order of issue, tile order, partial sums and epilogue as in gemm_tile_kernel.  DUAL: half of a wave's
// fragments are columns of W, the others the same columns of W2.
template <int WM, int WN, int TN, int KS, int NST, bool DUAL>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_split_kernel(int M, int NT, int MT, int splits, float* __restrict__ part, SplitOperands of, TileEpilogue<float> epi) {
    constexpr int BK = 16 * KS, ROWB = BK * 4;
    constexpr int BM = 32 * WM, BN = 32 * TN * WN, NW = WM * WN;
    constexpr int NREAL = DUAL ? BN / 2 : BN, TNO = DUAL ? TN / 2 : TN;
    constexpr int PLANE = NREAL * 16, MAT = 6 * KS * PLANE;            // bytes of a plane's k-group of 8 in LDS; of a matrix, [k-group][plane][column]
    constexpr int A_BYTES = BM * ROWB, B_BYTES = BN * 96 * KS, STAGE = A_BYTES + B_BYTES;
    constexpr int LAI = A_BYTES / 1024, LBI = B_BYTES / 1024, LA = LAI / NW, LB = (LBI + NW - 1) / NW, LPT = LA + LB;   // load instructions of a tile; of a wave
    constexpr bool EVEN = LBI % NW == 0;                               // otherwise the first LBI % NW waves bring one more than the others
    static_assert(LA * NW == LAI && LBI * 1024 == B_BYTES, "whole load instructions");
    static_assert(!DUAL || (TN % 2 == 0 && MAT % 1024 == 0), "a load instruction belongs to one matrix of the pair");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN, K = of.K, Npad = of.Npad;
    int bx, by, sidx;
    {
        const int total = NT * MT * splits, per = (total + 7) / 8;
        const int u = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
        if (u >= total) return;
        const int v = u / splits;
        sidx = u % splits;
        const int gsz = 8 * NT, g = v / gsz, first = g * 8;
        const int gm = MT - first < 8 ? MT - first : 8;
        by = first + (v % gsz) % gm;
        bx = (v % gsz) / gm;
    }
    const int m0 = by * BM, n0 = bx * NREAL;
    auto swz = [](int row) { return KS == 2 ? (row >> 1) & 7 : (row >> 2) & 3; };   // position p of a row holds its 4 k of chunk p ^ swz(row)
    unsigned a_off[LA], b_off[LB];
    unsigned long long b_base[LB];
#pragma unroll
    for (int j = 0; j < LA; ++j) {
        const int sl = (wave * LA + j) * 64 + lane, row = sl / (4 * KS), pos = sl % (4 * KS);
        int m = m0 + row;
        if (m > M - 1) m = M - 1;
        a_off[j] = (unsigned)(m - m0) * (unsigned)(K * 4) + (unsigned)((pos ^ swz(row)) * 16);   // under 256 rows: fits 32 bits (K <= 2^21)
    }
#pragma unroll
    for (int j = 0; j < LB; ++j) {
        const int q = wave + j * NW < LBI ? wave + j * NW : wave, half = q * 1024 / MAT, at = q * 1024 + lane * 16 - half * MAT;
        int col = n0 + at % PLANE / 16;
        if (col > Npad - 1) col = Npad - 1;
        b_base[j] = (unsigned long long)(DUAL && half ? of.wp2 : of.wp);
        b_off[j] = (unsigned)(((unsigned long long)(at / PLANE) * Npad + col) * 16);
    }
    const unsigned long long a_base = (unsigned long long)(of.x + (int64_t)m0 * K);
    const int64_t b_tile_step = (int64_t)6 * KS * Npad * 16;
    const unsigned lds0 = (unsigned)(uintptr_t)lds;
    const int kt_all = K / BK, kt0 = (int)((int64_t)sidx * kt_all / splits);
    const int nt = (int)((int64_t)(sidx + 1) * kt_all / splits) - kt0;   // this workgroup's k tiles: [kt0, kt0 + nt)
    const bool all_loads = EVEN || wave < LBI % NW;
    auto issue = [&](int t, int st) {
        if (t >= nt) return;
        const unsigned long long ab = gemm_uniform64(a_base + (unsigned long long)(t + kt0) * ROWB);
        const unsigned long long bt = (unsigned long long)((t + kt0) * b_tile_step);
        const unsigned sbase = lds0 + st * STAGE;
#pragma unroll
        for (int j = 0; j < LA; ++j) gemm_lds_load16(a_off[j], ab, (unsigned)__builtin_amdgcn_readfirstlane((int)(sbase + (wave * LA + j) * 1024)));
#pragma unroll
        for (int j = 0; j < LB; ++j)
            if (j + 1 < LB || all_loads) gemm_lds_load16(b_off[j], gemm_uniform64(b_base[j] + bt), (unsigned)__builtin_amdgcn_readfirstlane((int)(sbase + A_BYTES + (wave + j * NW) * 1024)));
    };
    f32x16_t acc[TN], small[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[j][v] = small[j][v] = 0.f;
    const int fsel = lane >> 5, r32 = lane & 31;
    int a_rd[KS][2];
#pragma unroll
    for (int kk = 0; kk < KS; ++kk)
#pragma unroll
        for (int c = 0; c < 2; ++c) a_rd[kk][c] = (wm * 32 + r32) * ROWB + (((4 * kk + 2 * fsel + c) ^ swz(r32)) * 16);
    const int b_rd = A_BYTES + fsel * 3 * PLANE + (wn * 32 * TNO + r32) * 16;
    f32x4_t ar[2];
    bf16x8_t as[2][3], bs[2][TN][3];
    auto fread = [&](int st, int kk, int slot) {
        const unsigned char* base = lds + st * STAGE;
#pragma unroll
        for (int c = 0; c < 2; ++c) ar[c] = *reinterpret_cast<const f32x4_t*>(base + a_rd[kk][c]);
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int p = 0; p < 3; ++p) bs[slot][j][p] = *reinterpret_cast<const bf16x8_t*>(base + b_rd + (6 * kk + p) * PLANE + (j / TNO) * MAT + (j % TNO) * 32 * 16);
    };
    auto wait_for = [&](int t) {   // tile t has landed; those up to t + NST - 2 may be on their way
        if (t + NST - 2 < nt) {
            if (all_loads) gemm_wait_loads<(NST - 2) * LPT>();
            else gemm_wait_loads<(NST - 2) * (LPT - 1)>();
        } else {
            gemm_wait_loads<0>();
        }
    };
    for (int st = 0; st < NST - 1; ++st) issue(st, st);
    wait_for(0);
    __syncthreads();
    issue(NST - 1, NST - 1);
    fread(0, 0, 0);
    split_rows8(ar[0], ar[1], as[0]);
    auto tile_step = [&](auto ring_pos, int t) {
        constexpr int ST = decltype(ring_pos)::value, ST1 = (ST + 1) % NST;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
            const int slot = KS == 2 ? kk : ST & 1;
            auto mul = [&](int pa, int pb, f32x16_t* to) {
#pragma unroll
                for (int j = 0; j < TN; ++j) to[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as[slot][pa], bs[slot][j][pb], to[j], 0, 0, 0);
            };
            __builtin_amdgcn_sched_barrier(0);
            if (kk + 1 < KS) fread(ST, kk + 1, slot ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
            mul(2, 0, small);
            mul(1, 1, small);
            mul(0, 2, small);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
            if (kk + 1 == KS) {
                wait_for(t + 1);
                __syncthreads();
                fread(ST1, 0, slot ^ 1);
            }
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
            mul(1, 0, small);
            mul(0, 1, small);
            mul(0, 0, acc);
            split_rows8(ar[0], ar[1], as[slot ^ 1]);
            if (kk + 1 == KS) issue(t + NST, ST);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    static_assert(KS == 1 || KS == 2, "");
    static_assert((KS == 2 && NST == 3) || NST == 4, "a k-step's fragments alternate between two slots; the tile loop is unrolled over the ring");
    {
        constexpr std::integral_constant<int, 0> R0{};
        constexpr std::integral_constant<int, 1> R1{};
        constexpr std::integral_constant<int, 2> R2{};
        constexpr std::integral_constant<int, NST - 1> R3{};
        int t = 0;
        for (; t + NST <= nt; t += NST) {
            tile_step(R0, t);
            tile_step(R1, t + 1);
            tile_step(R2, t + 2);
            if constexpr (NST > 3) tile_step(R3, t + 3);
        }
        if (t < nt) tile_step(R0, t);
        if (t + 1 < nt) tile_step(R1, t + 1);
        if constexpr (NST > 3)
            if (t + 2 < nt) tile_step(R2, t + 2);
    }
    const int mw = m0 + wm * 32, nw = n0 + wn * 32 * TNO;              // the wave's first output
    float odd = 0.f;                                                   // a NaN once any scaled sum is not finite
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        acc[j] += small[j];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            odd += acc[j][v] * 0.f;
            acc[j][v] *= kSplitUnscale;
        }
    }
    if (__any(!(odd == 0.f))) {
        // Sums that are not finite are formed again over this workgroup's k, on the f32 cores: x and the row-major weights straight from memory, a lane's four k of
        // every 8 in two chains as in gemm_tile_kernel.  All of the wave's fragments at once, so that a round trip to memory brings 16 k of each; rows and columns
        // past the end repeat the last one.
        const float* xr = of.x + (int64_t)(mw + r32 < M ? mw + r32 : M - 1) * K + 4 * fsel;
        const float* wc[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = nw + (j % TNO) * 32 + r32;
            wc[j] = (j >= TNO ? of.w2 : of.w) + (n < (int)epi.N ? n : (int)epi.N - 1);
        }
        f32x16_t sums[2][TN];
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) sums[0][j][v] = sums[1][j][v] = 0.f;
#pragma unroll 1
        for (int k0 = kt0 * BK; k0 < (kt0 + nt) * BK; k0 += 16) {
            f32x4_t a[2];
            float b[2][TN][4];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                a[h] = *reinterpret_cast<const f32x4_t*>(xr + k0 + 8 * h);
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) b[h][j][e] = wc[j][(int64_t)(k0 + 8 * h + 4 * fsel + e) * epi.N];
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < TN; ++j) sums[e >> 1][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[h][e], b[h][j][e], sums[e >> 1][j], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            sums[0][j] += sums[1][j];
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[j][v] = __builtin_isfinite(acc[j][v]) ? acc[j][v] : sums[0][j][v];
        }
    }
    const int r0 = 4 * fsel;                                           // value v of a lane: row 8 (v / 4) + r0 + v % 4, column r32
    if (splits > 1) {
        const int np = ((int)epi.N + 7) & ~7, width = DUAL ? 2 * np : np;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = nw + (j % TNO) * 32 + r32;
            if (n >= np) continue;
            float* to = part + (int64_t)sidx * M * width + (j / TNO) * np + n;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int m = mw + 8 * (v >> 2) + r0 + (v & 3);
                if (m < M) to[(int64_t)m * width] = acc[j][v];
            }
        }
        return;
    }
    constexpr int RSF = 32 * TNO + 4, CH = 4 * TNO, PASSES = CH / 2;   // as in gemm_tile_kernel
    float* area = reinterpret_cast<float*>(lds) + wave * (32 * RSF);
#pragma unroll
    for (int j = 0; j < TNO; ++j) {
        if constexpr (DUAL) gemm_glu<16>(acc[j], acc[j + TNO], epi.extra.glu);
#pragma unroll
        for (int v = 0; v < 16; ++v) area[(8 * (v >> 2) + r0 + (v & 3)) * RSF + j * 32 + r32] = acc[j][v];
    }
#pragma unroll 1
    for (int it = 0; it < PASSES; ++it) {
        const int c = it * 64 + lane, r = c / CH, cc = c % CH;
        const int m = mw + r, n = nw + cc * 8;
        if (m < M && n < epi.N) gemm_finish8<float, false>(epi, m, n, area + r * RSF + cc * 8, nullptr);
    }
}

// Adds the partial sums of a launch whose tiles were split over k, in split order (the result does not depend on which
// workgroup ended first), and finishes the outputs.  One thread per 8 outputs.  A launch of its own over the whole chip:
// with the last workgroup of a tile adding them, 48 tiles of M = 333 kept 48 CUs busy reading while 208 waited.
template <typename T, bool DUAL>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const float* __restrict__ part, int M, int splits, TileEpilogue<T> epi) {
    const int np = ((int)epi.N + 7) & ~7, chunks = np / 8, width = DUAL ? 2 * np : np;
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= (int64_t)M * chunks) return;
    const int64_t m = id / chunks;
    const int n = (int)(id % chunks) * 8;
    auto sum8 = [&](const float* p, float* o) {
        f32x4_t a = {0.f, 0.f, 0.f, 0.f}, b = a;
        for (int s = 0; s < splits; ++s, p += (int64_t)M * width) {
            a += *reinterpret_cast<const f32x4_t*>(p);
            b += *reinterpret_cast<const f32x4_t*>(p + 4);
        }
        *reinterpret_cast<f32x4_t*>(o) = a;
        *reinterpret_cast<f32x4_t*>(o + 4) = b;
    };
    __shared__ __attribute__((aligned(16))) float rows[256][12];   // finish8 reads its eight from LDS; each thread its own
    float* o = rows[threadIdx.x];
    sum8(part + m * width + n, o);
    if (DUAL) {
        float u[8];
        sum8(part + m * width + np + n, u);
        gemm_glu<8>(o, u, epi.extra.glu);
    }
    gemm_finish8<T, false>(epi, m, n, o, nullptr);
}

// The same for a layer whose f32 rows (plus a residual) go into an RMS norm next: a workgroup adds and stores one row and normalises it while it
// holds it, a launch and a pass over the rows less (M = 333, N = 3072, three splits: 5.4 + 5.2 -> 6.6 us).  A thread has 8 neighbours; sums, square sums and
// rounding in the order of gemm_reduce_kernel and rms_norm_f32_to_bf16, so the results are theirs bit for bit.
template <int SP>
__global__ __launch_bounds__(1024) void gemm_reduce_norm_kernel(const float* __restrict__ part, int M, int N, const float* __restrict__ residual, float* __restrict__ y,
                                                                const float* __restrict__ gamma, bf16_t* __restrict__ normed, float inv_n, float eps) {
    __shared__ float red[16];
    const int64_t at = (int64_t)blockIdx.x * N + threadIdx.x * 8;
    const bool live = (int)threadIdx.x * 8 < N;
    f32x4_t a = {0.f, 0.f, 0.f, 0.f}, b = a, ga = a, gb = a;
    if (live) {
        f32x4_t p[SP][2], ra = a, rb = a;
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            p[s][0] = *reinterpret_cast<const f32x4_t*>(part + (int64_t)s * M * N + at);
            p[s][1] = *reinterpret_cast<const f32x4_t*>(part + (int64_t)s * M * N + at + 4);
        }
        if (residual) { ra = *reinterpret_cast<const f32x4_t*>(residual + at); rb = *reinterpret_cast<const f32x4_t*>(residual + at + 4); }
        ga = *reinterpret_cast<const f32x4_t*>(gamma + threadIdx.x * 8);
        gb = *reinterpret_cast<const f32x4_t*>(gamma + threadIdx.x * 8 + 4);
#pragma unroll
        for (int s = 0; s < SP; ++s) { a += p[s][0]; b += p[s][1]; }
        if (residual) { a += ra; b += rb; }
        *reinterpret_cast<f32x4_t*>(y + at) = a;
        *reinterpret_cast<f32x4_t*>(y + at + 4) = b;
    }
    float q = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) q += a[e] * a[e];
#pragma unroll
    for (int e = 0; e < 4; ++e) q += b[e] * b[e];
    const float inv_rms = 1.0f / sqrtf(block_sum(q, red) * inv_n + eps);
    if (!live) return;
    u32x4_t o;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        o[e] = pack_bf16x2((a[2 * e] * inv_rms) * ga[2 * e], (a[2 * e + 1] * inv_rms) * ga[2 * e + 1]);
        o[2 + e] = pack_bf16x2((b[2 * e] * inv_rms) * gb[2 * e], (b[2 * e + 1] * inv_rms) * gb[2 * e + 1]);
    }
    *reinterpret_cast<u32x4_t*>(normed + at) = o;
}
// What a row norm behind the layer needs to be taken along with the adding of its splits.
static bool norm_fits(const MfmaLinearArgs& a) {
    const uintptr_t p = (uintptr_t)a.residual | (uintptr_t)a.y | (uintptr_t)a.norm_gamma | (uintptr_t)a.norm_y;
    return a.norm_gamma && a.dtype == 2 && a.out_f32 && !a.bias && !a.act && !a.extra.colscale && !a.wk2 && a.n % 8 == 0 && a.n <= 8192 && (p & 15) == 0;
}
static void launch_reduce_norm(hipStream_t s, const MfmaLinearArgs& a, int splits) {
    const int64_t chunks = a.n / 8;
    const unsigned threads = chunks <= 64 ? 64 : chunks <= 256 ? 256 : chunks <= 512 ? 512 : 1024;   // rms_norm_f32_to_bf16's
    auto go = [&](auto sp) {
        gemm_reduce_norm_kernel<decltype(sp)::value><<<(unsigned)a.m, threads, 0, s>>>((const float*)a.part, (int)a.m, (int)a.n, (const float*)a.residual, (float*)a.y, (const float*)a.norm_gamma,
                                                                                     (bf16_t*)a.norm_y, a.norm_inv_n, a.norm_eps);
    };
    if (splits == 2) go(std::integral_constant<int, 2>{});
    else if (splits == 3) go(std::integral_constant<int, 3>{});
    else if (splits == 4) go(std::integral_constant<int, 4>{});
    else if (splits == 6) go(std::integral_constant<int, 6>{});
    else go(std::integral_constant<int, 8>{});
    *a.normed = true;
}

// The tiles, in the order of tile_cost's table.
enum TileId { kT256x256, kT256x192, kT192x192, kT128x256, kT128x192, kT128x128, kT64x256, kT64x128, kTiles };
// The part of a layer's outputs that a launch forms: whole tiles from (row0, col0) on; no rows or columns: to the end.  (A layer whose k
// is split is formed by one launch.)
struct TileRegion { int64_t row0 = 0, col0 = 0, rows = 0, cols = 0; };
// rest_tile >= 0 (bf16): the layer takes two launches, `tile` over `first` and `rest_tile` over `rest`.
struct TilePlan { int tile; int splits; int rest_tile = -1; TileRegion first = {}, rest = {}; };
constexpr int kTileLds = 160 * 1024;   // LDS of one CU

// LDS of an int4 tile: a ring of three and, behind it, the scales of the groups of 128 k that a workgroup's share of K touches.
static int64_t int4_lds_bytes(int64_t bm, int64_t bn, int64_t k, int64_t splits) { return 3 * (bm * 128 + bn * 32) + (cdiv(cdiv(k, 64), splits) / 2 + 2) * bn * 2; }

template <typename T, int KG, int NST, int WM, int WN, int TM, int TN, bool DUAL, int QF = 0, int KW = 1>
static void launch_tile(hipStream_t s, const MfmaLinearArgs& a, int splits, TileRegion at = {}) {
    constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN, NREAL = DUAL ? BN / 2 : BN;
    constexpr int ring = NST * (BM * KG * 16 + BN * KG * (QF == 0 ? 16 : QF == 1 ? 8 : 4)), area = WM * WN * KW * 32 * (32 * (DUAL && TN % 2 == 0 ? TN / 2 : TN) + 4) * 4;
    constexpr int rows = KW == 1 ? area : std::max(area, WM * WN * KW * (TM / KW) * TN * 16 * 64 * 4);   // what the epilogue puts where the ring was
    constexpr int lds_most = QF == 2 ? kTileLds : ring > rows ? ring : rows;
    static_assert(ring <= kTileLds && lds_most <= kTileLds, "LDS of one CU");
    static_assert(QF != 2 || (NST == 3 && KG == 8), "int4_lds_bytes()");
    const int lds_bytes = QF == 2 ? std::max(rows, (int)int4_lds_bytes(BM, BN, a.k, splits)) : lds_most;
    auto kern = gemm_tile_kernel<T, KG, NST, WM, WN, KW, TM, TN, DUAL, QF>;
    static bool configured = false;  // the attribute is per function, not per stream or device state
    if (!configured) {
        (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_most);
        configured = true;
    }
    const int64_t nt = cdiv((at.cols ? at.cols : a.n - at.col0), NREAL), mt = cdiv((at.rows ? at.rows : a.m - at.row0), BM);
    TileEpilogue<T> epi{(const T*)a.bias, a.residual, a.y, a.n, a.act, a.out_f32, a.extra};
    kern<<<(unsigned)(cdiv(nt * mt * splits, 8) * 8), 64 * WM * WN * KW, lds_bytes, s>>>((const T*)a.x, (const T*)a.wk, (const T*)a.wk2, (int)a.m, (int)a.k,
                                                                                   (int)mfma_padded_n(a.n), (int)at.row0, (int)at.col0, (int)nt, (int)mt, splits, (float*)a.part,
                                                                                   (const T*)a.scale, (const T*)a.scale2, epi);
    if constexpr (std::is_same<T, bf16_t>::value && !DUAL)
        if (splits > 1 && norm_fits(a)) return launch_reduce_norm(s, a, splits);
    if (splits > 1) gemm_reduce_kernel<T, DUAL><<<(unsigned)cdiv(a.m * cdiv(a.n, 8), 256), 256, 0, s>>>((const float*)a.part, (int)a.m, splits, epi);
}
static size_t tile_part_bytes(int64_t m, int64_t n, bool dual, int splits) {
    return splits > 1 ? (size_t)splits * m * cdiv(n, 8) * 8 * (dual ? 2 : 1) * sizeof(float) : 0;
}

constexpr size_t kMostPart = 64u << 20;   // bytes of partial sums that a plan may take
static bool splits_allowed() {
    static const bool on = [] { const char* e = getenv("GPTRS_HIP_GEMM_TAILSPLIT"); return !(e && e[0] == '0'); }();
    return on;
}

// Which tile a launch takes, and over how many workgroups a tile's k is split, with `room` bytes for their partial sums.  Estimated time in us of every choice, from a
// linear fit (within 6 % rms, 128 x 192 10 %) to measurements at M = 40 .. 1500 of the 3072-wide layers (K = 3072, 4096, 9216; N = 3072, 6144,
// a pair of 9216; weights from memory): rounds of workgroups x (fixed + per k tile of 64) + what a k tile costs more with the
// chip full, and for a split the second launch plus its bytes.  Over 158 shapes (M = 20 .. 8188 of those layers and of K = 768 .. 6144,
// N = 512 .. 14432) what it picks is 3.0 % slower than the best measured choice in the mean (4.8 % without the 128 x 192 tiles).
// 192 x 192 (4 waves of 96 x 96, plain layers) is for one round of long sums that the 256-wide tiles leave a quarter of the CUs out of: M = 3064,
// N = 3072 is 256 of them, 192 of 256 x 192.  us, against the best of the others: K = 9216 157 and 178 (M = 2900 155 and 161), K = 6144 107 and
// 117; below 80 k tiles its long start and way out cost what it gains (K = 4096 72 and 70), and in two rounds 128 x 192 is better
// (M = 5500, K = 9216 296 and 278).
struct TileCost { int bm, bn, slots; double fixed, per_kt, full_kt, split, split_mb; };
static const TileCost kTileCost[kTiles] = {
    {256, 256, 256, 5.45, 1.237, 0.379, 2.8, 0.30}, {256, 192, 256, 1.16, 1.206, 0.122, 4.7, 0.35}, {192, 192, 256, 12.0, 0.86, 0.14, 0.0, 0.0}, {128, 256, 256, 6.87, 0.661, 0.171, 3.1, 0.26}, {128, 192, 256, 7.9, 0.48, 0.266, 5.1, 0.10},
    {128, 128, 256, 4.48, 0.425, 0.055, 3.9, 0.31}, {64, 256, 256, 4.59, 0.572, 0.0, 5.4, 0.13}, {64, 128, 512, 2.58, 0.361, 0.143, 5.0, 0.34},
};
static TilePlan tile_plan(int64_t m, int64_t k, int64_t n, bool dual, size_t room = SIZE_MAX) {
    TilePlan best{kT256x256, 1};
    double least = 1e300;
    for (int t = 0; t < kTiles; ++t) {
        const TileCost& c = kTileCost[t];
        if (dual && (t == kT256x192 || t == kT192x192)) continue;   // a wave's three fragments do not divide between the matrices
        const int64_t tiles = cdiv(m, c.bm) * cdiv(n, dual ? c.bn / 2 : c.bn);
        if (t == kT192x192 && (tiles > c.slots || k < 80 * 64)) continue;
        for (int sp : {1, 2, 3, 4, 6, 8}) {
            if (sp > 1 && (!splits_allowed() || t == kT192x192 || k < 256 * sp || tiles * sp > 2 * c.slots || tile_part_bytes(m, n, dual, sp) > std::min(room, kMostPart))) break;
            const double kt = (double)k / 64 / sp, wg = (double)(tiles * sp);
            double us = (double)cdiv(tiles * sp, c.slots) * (c.fixed + c.per_kt * kt) + c.full_kt * kt * wg / 256;
            if (sp > 1) us += c.split + c.split_mb * (double)tile_part_bytes(m, n, dual, sp) / 1e6;
            if (us < least) { least = us; best = {t, sp}; }
        }
    }
    // Two launches: as many whole rows or columns of tiles as fill whole rounds, and the rest, which would leave most of a last round idle,
    // in tiles that fill a round of their own.  Taken where the fit says 7.5 % or more: what it says less about came out level, since a
    // last round that is partly empty runs at a higher clock.  us, weights from memory, measured against the best single launch: pair of
    // 9216 M = 1000 126 -> 119, 2047 238 -> 218, 3000 340 -> 319; N = 6176 M = 3000 135 -> 123; K = 1536, N = 6144 M = 3064 75 -> 71.
    // Over 160 shapes that the rule was tried on first (M = 64 .. 7600, K = 576 .. 9216, N = 768 .. 14336) it gains 8.8 % in the mean; losses of up to
    // 7 % at K of 1024 and less (M = 4758, K = 768, N = 5120 69 -> 74), where the second launch's start counts: those stay whole.  A second launch over
    // a few rows more is bound by the weights, which it reads again, where they are more than the last cache holds: priced without, pairs of
    // K = 9216 .. 14336, N = 14336 lost up to 8 % (M = 563, K = 9216, N = 14432 317 -> 337; M = 270, K = 11008, N = 14336 254 -> 275).  With it they are one launch
    // (317) or are split by columns (M = 352, K = 9216, N = 14432 242, 246, 216; M = 359, K = 14336 378, 376, 332).  Over 180 shapes that take two launches (K up to 14336,
    // N up to 18432) the mean gain is 5.5 %, the largest loss 3 % (M = 2756, K = 14336, N = 6144 442 -> 456: the fit gives 128 x 192 tiles 10 % too much at long K).
    // Left alone too: N = 14432 M = 3064 (5.6 % by the fit, 265 and 262), K = 3072, N = 4096 M = 3064 (5.4 %, 86 and 85).
    if (best.splits == 1 && least > 40.0 && k > 1024) {
        const double one = least;
        // a second launch over further rows reads all weights again; what is left of 256 MB and less is still in the last cache
        const double weights = (double)k * n * (dual ? 2 : 1) * 2, again = weights > 256e6 ? weights / 5.0e6 : 0.0;
        auto cost = [&](int t, int64_t rows, int64_t cols) {
            const TileCost& c = kTileCost[t];
            const int64_t tiles = cdiv(rows, c.bm) * cdiv(cols, dual ? c.bn / 2 : c.bn);
            const double kt = (double)k / 64;
            return (double)cdiv(tiles, c.slots) * (c.fixed + c.per_kt * kt) + c.full_kt * kt * (double)tiles / 256;
        };
        for (int t = 0; t < kTiles; ++t) {
            if ((dual && (t == kT256x192 || t == kT192x192)) || (t == kT192x192 && k < 80 * 64)) continue;
            const TileCost& c = kTileCost[t];
            const int64_t bn = dual ? c.bn / 2 : c.bn, nt = cdiv(n, bn), mt = cdiv(m, c.bm), filled = nt * mt / c.slots * c.slots;
            for (const bool by_columns : {true, false}) {
                const int64_t whole = filled / (by_columns ? mt : nt);   // columns or rows of tiles
                if (whole < 1 || whole >= (by_columns ? nt : mt)) continue;
                TileRegion first, rest;
                (by_columns ? first.cols : first.rows) = whole * (by_columns ? bn : c.bm);
                (by_columns ? rest.col0 : rest.row0) = whole * (by_columns ? bn : c.bm);
                const double us1 = cost(t, by_columns ? m : first.rows, by_columns ? first.cols : n);
                for (int r = 0; us1 < least && r < kTiles; ++r) {
                    if (r == kT192x192 || (dual && r == kT256x192)) continue;
                    const double us = us1 + std::max(cost(r, m - rest.row0, n - rest.col0), by_columns ? 0.0 : again);
                    if (us < least && us < 0.925 * one) { least = us; best = {t, 1, r, first, rest}; }
                }
            }
        }
    }
    return best;
}
int mfma_bf16_regions(int64_t m, int64_t k, int64_t n, bool dual, int64_t* out) {
    const TilePlan p = tile_plan(m, k, n, dual);
    if (p.rest_tile < 0) return 1;
    const int64_t v[8] = {p.first.rows, p.first.cols, p.rest.row0, p.rest.col0, kTileCost[p.tile].bm, dual ? kTileCost[p.tile].bn / 2 : kTileCost[p.tile].bn, p.tile, p.rest_tile};
    for (int i = 0; i < 8; ++i) out[i] = v[i];
    return 2;
}
template <bool DUAL>
static void launch_tile_plan(hipStream_t s, const MfmaLinearArgs& a, TilePlan p, TileRegion at = {}) {
    typedef bf16_t T;
    switch (p.tile) {
        case kT256x256: return launch_tile<T, 4, 4, 2, 4, 4, 2, DUAL>(s, a, p.splits, at);
        case kT256x192: if constexpr (!DUAL) return launch_tile<T, 8, 2, 4, 2, 2, 3, false>(s, a, p.splits, at); else return;
        case kT192x192: if constexpr (!DUAL) return launch_tile<T, 8, 3, 2, 2, 3, 3, false>(s, a, p.splits, at); else return;
        case kT128x256: return launch_tile<T, 8, 3, 2, 4, 2, 2, DUAL>(s, a, p.splits, at);
        case kT128x192: return launch_tile<T, 8, 3, 2, 2, 2, 3, DUAL, 0, 2>(s, a, p.splits, at);
        case kT128x128:
            if constexpr (DUAL) return launch_tile<T, 8, 4, 4, 2, 1, 2, true>(s, a, p.splits, at);
            else return launch_tile<T, 8, 4, 2, 4, 2, 1, false>(s, a, p.splits, at);
        case kT64x256: return launch_tile<T, 8, 3, 2, 4, 1, 2, DUAL>(s, a, p.splits, at);
        default: return launch_tile<T, 8, 3, 2, 2, 1, 2, DUAL>(s, a, p.splits, at);
    }
}

// f32 of up to 128 rows (more: split_plan()): one tile, 64 x 64 outputs in 4 waves of 32 x 32 (a pair: 64 x 64 of each matrix), three workgroups to a CU.  The f32
// products are paced by the matrix pipes alone, 0.43 us for a k tile of 32 on a CU, one wave per SIMD is enough to keep them busy, and the small
// tile divides best among the CUs (64 x 128 takes 44 % longer at M = 400).  Splits over k: rounds of 256 workgroups, a launch more and its bytes.
static int tile_splits_f32(int64_t m, int64_t k, int64_t n, bool dual, size_t room = SIZE_MAX) {
    const int64_t tiles = cdiv(m, 64) * cdiv(n, 64);
    int best = 1;
    double least = 1e300;
    for (int sp : {1, 2, 3, 4, 6, 8}) {
        if (sp > 1 && (!splits_allowed() || k < 128 * sp || tile_part_bytes(m, n, dual, sp) > std::min(room, kMostPart))) break;
        double us = 5.0 + (dual ? 0.88 : 0.44) * ((double)k / 32 / sp) * (double)cdiv(tiles * sp, 256);
        if (sp > 1) us += 3.5 + 0.4 * (double)tile_part_bytes(m, n, dual, sp) / 1e6;
        if (us < least) { least = us; best = sp; }
    }
    return best;
}

// Up to two rows of 64 x 64 tiles the f32 cores keep up on 4 bytes a weight instead of 6 (M = 128, us, f32 and split: K = 768 and N = 2304, 768, 3072 11.8 and 12.9, 9.8 and 10.0,
// 14.0 and 13.4, K = 3072, N = 768 15.1 and 14.6; M = 129: 14.1 and 14.0, 10.6 and 10.4, 17.4 and 16.8, 17.8 and 17.4; M = 200: 17.2 and 16.6,
// 11.0 and 10.9, 18.1 and 17.7, 21.0 and 20.5).
static bool mfma_splits_f32(int64_t m) { return m > 128; }
// The split kernel's tiles and splits, by a cost fitted to measurements at M = 129 .. 8192 of 21 plain layers (K = 64 .. 5120, N = 256 .. 6144) and M = 129 .. 3000 of nine
// pairs (K = 512 .. 4096, N = 768 .. 8192), 1 to 12 splits, weights from memory: rounds of workgroups, at one price where two share a CU and another
// where each has one to itself, x (fixed + per k tile of 16) + what a k tile costs more with the chip full, and for a split the launch that adds them, by their bytes and their
// number (a thread reads one after another).  What it picks is 0.7 % (plain, 233 shapes) and 0.3 % (pairs, 99) slower than the best measured choice in the mean, at most
// 13 %.  (Fitted to four layers alone, and a pair, whose ring leaves room for one workgroup on a CU, priced as if there were two: 2.3 and 8.8 %, and layers of 200 to
// 640 rows, K = N = 768, slower than f32 products.)  A plain layer of 64 x 64 tiles has two workgroups on a CU by its splits only where
// each of them keeps 512 k (K = N = 768, us, 333 rows in 3 and in 6 splits 11.5 and 13.0, 640 rows in 2 and in 4 14.0 and 15.5); no split is under 160 k.
struct SplitCost { int bm, bn, slots; double fixed, per_kt, alone_fixed, alone_per_kt, full_kt, split, split_mb, per_split; };
enum SplitTileId { kS256x96, kS128x96, kS64x64, kSPair, kSTiles };   // a pair: 64 x 64 of each matrix
static const SplitCost kSplitCost[kSTiles] = {
    {256, 96, 256, 6.66, 0.473, 0.0, 0.0, 0.514, 4.14, 0.122, 0.254}, {128, 96, 512, 6.30, 0.558, 4.73, 0.439, 0.242, 4.33, 0.139, 0.225},
    {64, 64, 512, 4.93, 0.295, 4.80, 0.180, 0.090, 2.94, 0.0, 0.131}, {64, 64, 256, 4.96, 0.180, 0.0, 0.0, 0.033, 3.02, 0.0, 0.248},
};
static TilePlan split_plan(int64_t m, int64_t k, int64_t n, bool dual, size_t room = SIZE_MAX) {
    TilePlan best{dual ? kSPair : kS64x64, 1};
    double least = 1e300;
    for (int t = dual ? kSPair : 0; t < (dual ? kSTiles : kSPair); ++t) {
        const SplitCost& c = kSplitCost[t];
        const int64_t tiles = cdiv(m, c.bm) * cdiv(n, c.bn);
        for (int sp : {1, 2, 3, 4, 6, 8, 12}) {
            if (sp > 1 && (!splits_allowed() || k < 160 * sp || tiles * sp > 1024 || tile_part_bytes(m, n, dual, sp) > std::min(room, kMostPart))) break;
            if (sp > 1 && t == kS64x64 && tiles * sp > 256 && k < 512 * sp) break;
            const double kt = (dual ? 2.0 : 1.0) * (double)k / 16 / sp, wg = (double)(tiles * sp);
            const int64_t last = tiles * sp % c.slots;
            const bool alone = c.slots == 512 && last > 0 && last <= 256;   // in the last round
            double us = (double)(cdiv(tiles * sp, c.slots) - alone) * (c.fixed + c.per_kt * kt) + alone * (c.alone_fixed + c.alone_per_kt * kt) + c.full_kt * kt * wg / 256;
            if (sp > 1) us += c.split + c.split_mb * (double)tile_part_bytes(m, n, dual, sp) / 1e6 + c.per_split * sp;
            if (us < least) { least = us; best = {t, sp}; }
        }
    }
    return best;
}
template <int WM, int WN, int TN, int KS, int NST, bool DUAL>
static void launch_split(hipStream_t s, const MfmaLinearArgs& a, int splits) {
    constexpr int BM = 32 * WM, BN = 32 * TN * WN, NREAL = DUAL ? BN / 2 : BN;
    constexpr int ring = NST * KS * (BM * 64 + BN * 96), area = WM * WN * 32 * (32 * (DUAL ? TN / 2 : TN) + 4) * 4, lds_bytes = ring > area ? ring : area;
    auto kern = gemm_split_kernel<WM, WN, TN, KS, NST, DUAL>;
    static bool configured = false;  // the attribute is per function, not per stream or device state
    if (!configured) {
        (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
        configured = true;
    }
    const int64_t nt = cdiv(a.n, NREAL), mt = cdiv(a.m, BM);
    TileEpilogue<float> epi{(const float*)a.bias, a.residual, a.y, a.n, a.act, 0, a.extra};
    const SplitOperands of{(const float*)a.x, (const bf16_t*)a.wk, (const bf16_t*)a.wk2, (int)a.k, (int)mfma_padded_n(a.n), (const float*)a.w, (const float*)a.w2};
    kern<<<(unsigned)(cdiv(nt * mt * splits, 8) * 8), 64 * WM * WN, lds_bytes, s>>>((int)a.m, (int)nt, (int)mt, splits, (float*)a.part, of, epi);
    if (splits > 1) gemm_reduce_kernel<float, DUAL><<<(unsigned)cdiv(a.m * cdiv(a.n, 8), 256), 256, 0, s>>>((const float*)a.part, (int)a.m, splits, epi);
}

// Quantised: which tile converts the codes of which columns.  Every wave converts the B fragments it multiplies, 20 (int8) or
// 23 (int4) vector instructions for 8 codes, so the tiles give a wave as many rows per column as fit: one wave row (128 x 256 in 8
// waves of 128 x 32, 128 x 128 and 64 x 128 in 4) has no column converted twice; a pair, whose waves hold both matrices, has two
// wave rows and runs 256 x 256 where it is large.  Measured with int8 at M = 40 .. 4000 of the 3072-wide layers, fitted as above
// (7 % rms).  Int4 takes the same plan, so that a layer's sums do not depend on its codes: 7 % slower than int8 in the median (-6 .. 16 %), and
// over 60 of those shapes the pick is 2.1 % slower than the best measured choice for int4, 2.8 % for int8; worst for int4 at M = 3000, K =
// 9216 (288 us against 229: a long K's scales leave a CU two workgroups of 64 x 128; counting them so would cost int8 229 -> 255).  Against the
// register-staged tiles that ran here before (64 x 64 below half a chip of 128 x 128), M = 200, int8, us: out and down 65 (mean)
// -> 21 and 29, qkv 35 -> 24, pair 58 -> 58.
enum QuantTileId { kQ256x256, kQ128x256, kQ128x128, kQ64x128, kQTiles };
static const TileCost kQuantCost[2][kQTiles] = {
    {{256, 256, 0, 0, 0, 0, 0, 0}, {128, 256, 256, 4.87, 0.719, 0.337, 5.5, 0.15}, {128, 128, 512, 4.72, 0.486, 0.283, 6.3, 0.12}, {64, 128, 768, 4.25, 0.311, 0.207, 6.3, 0.09}},
    {{256, 256, 256, 3.15, 1.197, 1.059, 0.2, 0.24}, {128, 256, 256, 4.88, 0.870, 0.480, 3.9, 0.17}, {128, 128, 0, 0, 0, 0, 0, 0}, {64, 128, 768, 3.0, 0.524, 0.30, 4.0, 0.0}},
};
static TilePlan quant_plan(int64_t m, int64_t k, int64_t n, bool dual, size_t room = SIZE_MAX) {
    TilePlan best{-1, 1};
    double least = 1e300;
    for (int t = 0; t < kQTiles; ++t) {
        const TileCost& c = kQuantCost[dual][t];
        if (c.slots == 0) continue;
        const int64_t tiles = cdiv(m, c.bm) * cdiv(n, dual ? c.bn / 2 : c.bn);
        for (int sp : {1, 2, 3, 4, 6, 8}) {
            if (sp > 1 && (!splits_allowed() || k < 256 * sp || tiles * sp > 2 * c.slots || tile_part_bytes(m, n, dual, sp) > std::min(room, kMostPart))) break;
            if (int4_lds_bytes(c.bm, c.bn, k, sp) > kTileLds) continue;   // int8 takes the same plan
            const double kt = (double)k / 64 / sp, wg = (double)(tiles * sp);
            double us = (double)cdiv(tiles * sp, c.slots) * (c.fixed + c.per_kt * kt) + c.full_kt * kt * wg / 256;
            if (sp > 1) us += c.split + c.split_mb * (double)tile_part_bytes(m, n, dual, sp) / 1e6;
            if (us < least) { least = us; best = {t, sp}; }
        }
    }
    return best;
}

bool mfma_gemm_supported(int dtype, int64_t m, int64_t k, int64_t n, int quant) {
    if (dtype != 0 && dtype != 2) return false;
    if (quant != 0 && (dtype != 2 || (quant == 2 && k % 128 != 0))) return false;
    const int64_t bk = kKb * kpc_of(dtype);
    return m > 16 && k >= bk && k % bk == 0 && n >= 1 && m < (1ll << 31) && n < (1ll << 31) - kBN && k < (1ll << 31) &&
           cdiv(m, 128) * cdiv(n, 64) < (1ll << 30);   // tile ids are ints
}

// Partial sums of the register-staged kernel's 128 x 128 tiles when they are split.
static size_t staged_part_bytes(int64_t m, int64_t n, bool dual, int splits) {
    return splits > 1 ? (size_t)(cdiv(m, 128) * cdiv(mfma_padded_n(n), dual ? 64 : 128)) * splits * 128 * 128 * sizeof(float) : 0;
}
size_t mfma_workspace_bytes(int dtype, int64_t m, int64_t k, int64_t n, bool dual, int quant) {
    if (!mfma_gemm_supported(dtype, m, k, n, quant)) return 0;
    if (dtype == 0) return tile_part_bytes(m, n, dual, mfma_splits_f32(m) ? split_plan(m, k, n, dual).splits : tile_splits_f32(m, k, n, dual));
    const int qsp = quant_plan(m, k, n, dual).splits;
    return std::max(tile_part_bytes(m, n, dual, quant ? qsp : tile_plan(m, k, n, dual).splits), staged_part_bytes(m, n, dual, qsp));
}

template <typename T, bool DUAL, int QF = 0>
static void launch_staged(hipStream_t s, const MfmaLinearArgs& a, int splits = 1) {
    constexpr int BM = 128, BN = 128, lds_bytes = 2 * kKb * ((BM + 1) * 16 + (BN + 1) * 16);
    auto kern = gemm_mfma_kernel<T, BM, BN, DUAL, QF>;
    static bool configured = false;  // the attribute is per function, not per stream or device state
    if (!configured) {
        (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
        configured = true;
    }
    const int64_t npad = mfma_padded_n(a.n);
    constexpr int nreal = DUAL ? BN / 2 : BN;
    const int64_t nt = cdiv(npad, nreal), mt = cdiv(a.m, BM);
    if (splits > 1 && (!a.part || !a.tickets || nt * mt > (int64_t)kSkinnyTickets || a.part_bytes < staged_part_bytes(a.m, a.n, DUAL, splits))) splits = 1;
    const int64_t full = splits > 1 ? 0 : nt * mt;
    const unsigned grid = (unsigned)(cdiv(full, 8) * 8 + (nt * mt - full) * splits);
    kern<<<grid, 256, lds_bytes, s>>>((const T*)a.x, (const T*)a.wk, (const T*)a.wk2, (const T*)a.bias, (const T*)a.residual, (T*)a.y,
                                      (int)a.m, (int)a.k, (int)a.n, (int)npad, a.act, (int)nt, (int)mt, (const T*)a.scale, (const T*)a.scale2,
                                      (int)full, splits, (float*)a.part, a.tickets, a.dtype == 2 ? a.out_f32 : 0, a.extra);
}

static size_t room_of(const MfmaLinearArgs& a) { return a.part ? a.part_bytes : 0; }
size_t mfma_int4_lds_bytes(int64_t m, int64_t k, int64_t n, bool dual, size_t room) {
    const TilePlan p = quant_plan(m, k, n, dual, room);
    return p.tile < 0 ? 0 : (size_t)int4_lds_bytes(kQuantCost[dual][p.tile].bm, kQuantCost[dual][p.tile].bn, k, p.splits);
}

// The LDS-direct kernels' loads address a k tile with unsigned 32-bit offsets from one scalar base: 256 rows of x (K * 1024 bytes at most), and 8 k-groups of
// 16 bytes of the padded weights, of the split ones 12 in a tile of two k-steps.  The bound is for the 8; the 12 stay under 1.5 * 2^31.
static bool mfma_lds_direct_reach(int64_t k, int64_t n) { return k <= (1 << 21) && (uint64_t)mfma_padded_n(n) * 128 < (1ull << 31); }
bool mfma_takes_split_weights(int dtype, int64_t m, int64_t k, int64_t n, int lds_direct) { return dtype == 0 && lds_direct != 0 && mfma_splits_f32(m) && mfma_lds_direct_reach(k, n); }

template <bool DUAL, int QF>
static void launch_quant(hipStream_t s, const MfmaLinearArgs& a) {
    const TilePlan p = quant_plan(a.m, a.k, a.n, DUAL, room_of(a));
    typedef bf16_t T;
    const int sp = p.splits;
    switch (p.tile) {
        case kQ256x256: if constexpr (DUAL) return launch_tile<T, 8, 3, 2, 4, 4, 2, true, QF>(s, a, sp); else return;
        case kQ128x256:
            if constexpr (DUAL) return launch_tile<T, 8, 3, 2, 4, 2, 2, true, QF>(s, a, sp);
            else return launch_tile<T, 8, 3, 1, 8, 4, 1, false, QF>(s, a, sp);
        case kQ128x128: if constexpr (!DUAL) return launch_tile<T, 8, 3, 1, 4, 4, 1, false, QF>(s, a, sp); else return;
        case kQ64x128:
            if constexpr (DUAL) return launch_tile<T, 8, 3, 2, 2, 1, 2, true, QF>(s, a, sp);
            else return launch_tile<T, 8, 3, 1, 4, 2, 1, false, QF>(s, a, sp);
        default: return launch_staged<T, DUAL, QF>(s, a);   // K too long for the scales of an int4 tile in LDS
    }
}

void mfma_gemm(hipStream_t s, const MfmaLinearArgs& a) {
    const bool dual = a.wk2 != nullptr;
    const bool reach = mfma_lds_direct_reach(a.k, a.n);
    if (a.lds_direct == 0 || !reach) {
        // the splits of a layer of codes of this shape, for them and for the matrix that they stand for: the same sums in the same order
        const int sp = reach && a.dtype == 2 ? quant_plan(a.m, a.k, a.n, dual).splits : 1;
        if (a.dtype == 0) return dual ? launch_staged<float, true>(s, a) : launch_staged<float, false>(s, a);
        if (a.quant == 1) return dual ? launch_staged<bf16_t, true, 1>(s, a, sp) : launch_staged<bf16_t, false, 1>(s, a, sp);
        if (a.quant == 2) return dual ? launch_staged<bf16_t, true, 2>(s, a, sp) : launch_staged<bf16_t, false, 2>(s, a, sp);
        return dual ? launch_staged<bf16_t, true>(s, a, sp) : launch_staged<bf16_t, false>(s, a, sp);
    }
    if (a.quant == 1) return dual ? launch_quant<true, 1>(s, a) : launch_quant<false, 1>(s, a);
    if (a.quant == 2) return dual ? launch_quant<true, 2>(s, a) : launch_quant<false, 2>(s, a);
    if (a.dtype == 0 && mfma_splits_f32(a.m)) {
        const TilePlan p = split_plan(a.m, a.k, a.n, dual, room_of(a));
        if (dual) return launch_split<2, 2, 2, 2, 3, true>(s, a, p.splits);
        if (p.tile == kS256x96) return launch_split<8, 1, 3, 2, 3, false>(s, a, p.splits);
        if (p.tile == kS128x96) return launch_split<4, 1, 3, 1, 4, false>(s, a, p.splits);
        return launch_split<2, 2, 1, 2, 3, false>(s, a, p.splits);
    }
    if (a.dtype == 0) {
        const int sp = tile_splits_f32(a.m, a.k, a.n, dual, room_of(a));
        return dual ? launch_tile<float, 8, 3, 2, 2, 1, 2, true>(s, a, sp) : launch_tile<float, 8, 3, 2, 2, 1, 1, false>(s, a, sp);
    }
    const TilePlan p = tile_plan(a.m, a.k, a.n, dual, room_of(a));
    dual ? launch_tile_plan<true>(s, a, p, p.first) : launch_tile_plan<false>(s, a, p, p.first);
    if (p.rest_tile < 0) return;
    const TilePlan r{p.rest_tile, 1};
    dual ? launch_tile_plan<true>(s, a, r, p.rest) : launch_tile_plan<false>(s, a, r, p.rest);
}

}  // namespace k
}  // namespace gptrs
