// Causal attention kernels for the two sequences the reference emits:
//   * attention_decode_cache (crates/gpt-rs/src/ops/functional/attention.rs:657-779), T = 1
//   * attention without cache (attention.rs:443-522), prefill
// Both compute softmax((q.k) * scale + mask) . v with the additive -1e9 mask replaced by its
// exact f32 effect: masked positions contribute exactly 0 (exp underflows), so only positions
// <= the query position are visited.  GQA: query head h reads kv head h / group.
#include <algorithm>
#include <cstdlib>

#include <type_traits>

#include "kernels.hpp"
#include "device_utils.hpp"

namespace gptrs {
namespace k {

static inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
template <int CTRL> __device__ __forceinline__ float dpp_move(float v) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false)); }

template <typename T> __device__ __forceinline__ float ldf(const T* p, int64_t i);
template <> __device__ __forceinline__ float ldf<float>(const float* p, int64_t i) { return p[i]; }
template <> __device__ __forceinline__ float ldf<bf16_t>(const bf16_t* p, int64_t i) { return bf16_to_f32(p[i]); }
template <typename T> __device__ __forceinline__ void stf(T* p, int64_t i, float v);
template <> __device__ __forceinline__ void stf<float>(float* p, int64_t i, float v) { p[i] = v; }
template <> __device__ __forceinline__ void stf<bf16_t>(bf16_t* p, int64_t i, float v) { p[i] = f32_to_bf16(v); }

template <typename T> struct Vec16;
template <> struct Vec16<float> {
    static constexpr int N = 4;
    static __device__ __forceinline__ void load(const float* p, float (&o)[4]) {
        const float4 v = *reinterpret_cast<const float4*>(p);
        o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    }
};
template <> struct Vec16<bf16_t> {
    static constexpr int N = 8;
    static __device__ __forceinline__ void load(const bf16_t* p, float (&o)[8]) {
        const uint4 v = *reinterpret_cast<const uint4*>(p);
        o[0] = bf16lo(v.x); o[1] = bf16hi(v.x); o[2] = bf16lo(v.y); o[3] = bf16hi(v.y);
        o[4] = bf16lo(v.z); o[5] = bf16hi(v.z); o[6] = bf16lo(v.w); o[7] = bf16hi(v.w);
    }
};

constexpr int kMaxDecodeSplits = 512;

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef float f32x16_v __attribute__((ext_vector_type(16)));
typedef unsigned u32x4_v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int64_t clamp_i64(int64_t v, int64_t lo, int64_t hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Rotate-half RoPE (ops/functional/rotary.rs:430-536) applied while loading VEC consecutive dims
// [c0, c0+VEC) of one head: dims below `half` pair with dim+half, the next `half` dims pair with
// dim-half, dims >= 2*half pass through.  Needs half % VEC == 0 so a chunk never straddles a
// boundary.  The result is rounded to T, the value a stored post-RoPE row would hold.
template <typename T>
__device__ __forceinline__ void load_roped(const T* __restrict__ head, int c0, int half, const T* __restrict__ cs,
                                           const T* __restrict__ sn, float (&out)[Vec16<T>::N]) {
    constexpr int VEC = Vec16<T>::N;
    float own[VEC];
    Vec16<T>::load(head + c0, own);
    if (c0 >= 2 * half) {
#pragma unroll
        for (int v = 0; v < VEC; ++v) out[v] = own[v];
        return;
    }
    const bool first = c0 < half;
    float other[VEC], c[VEC], s[VEC];
    Vec16<T>::load(head + (first ? c0 + half : c0 - half), other);
    const int j0 = first ? c0 : c0 - half;
    Vec16<T>::load(cs + j0, c);
    Vec16<T>::load(sn + j0, s);
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
        // first half: a*cos - b*sin with (a,b) = (own, other); second half: b*cos + a*sin with (b,a) = (own, other)
        const float r = first ? own[v] * c[v] - other[v] * s[v] : own[v] * c[v] + other[v] * s[v];
        T tmp;
        stf(&tmp, 0, r);
        out[v] = ldf(&tmp, 0);
    }
}
template <typename T>
__device__ __forceinline__ T roped_elem(const T* __restrict__ head, int d, int half, const T* __restrict__ cs,
                                        const T* __restrict__ sn) {
    if (d >= 2 * half) return head[d];
    const bool first = d < half;
    const int j = first ? d : d - half;
    const float own = ldf(head, d), other = ldf(head, first ? d + half : d - half);
    const float r = first ? own * ldf(cs, j) - other * ldf(sn, j) : own * ldf(cs, j) + other * ldf(sn, j);
    T tmp;
    stf(&tmp, 0, r);
    return tmp;
}

// ------------------------------------------------------------------------------ decode
// grid (n_kv, nsplit), 256 threads.  A cache row (head_dim elements) is read by LPR lanes with one
// 16-byte load each, so a wave streams 64/LPR positions at a time; every such lane-group keeps
// its own online-softmax state for the G query heads of this kv head.  States are merged by
// shuffles inside the wave, through LDS across the four waves, and across splits by
// attn_decode_combine_kernel.
struct DecodeCaches { void* k[16]; void* v[16]; };   // per-sequence cache pointers of a batched launch (blockIdx.z)

template <typename T, int G>
__global__ __launch_bounds__(256) void attn_decode_kernel(const T* __restrict__ qkv, T* __restrict__ kc,
                                                          T* __restrict__ vc, const int32_t* __restrict__ us,
                                                          const int32_t* __restrict__ qs, T* __restrict__ ctx,
                                                          float* __restrict__ ws, int n_q, int n_kv, int dh,
                                                          int64_t cap, float scale, int64_t chunk, int nsplit,
                                                          const T* __restrict__ cs, const T* __restrict__ sn, int half,
                                                          int batched, DecodeCaches caches) {
    if (batched) {   // sequence blockIdx.z: its row of the stacked projection and of the context, its caches, its records
        const int b = blockIdx.z;
        kc = (T*)caches.k[b];
        vc = (T*)caches.v[b];
        qkv += (int64_t)b * (n_q + 2 * n_kv) * dh;
        ctx += (int64_t)b * n_q * dh;
        ws += (int64_t)b * n_q * nsplit * (dh + 2);
    }
    constexpr int VEC = Vec16<T>::N;
    const int lpr = dh / VEC;          // lanes per cache row (power of two, <= 64)
    const int rpw = 64 / lpr;          // rows per wave-iteration
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int sub = lane / lpr, li = lane % lpr;
    const int nstream = 4 * rpw, sid = wave * rpw + sub;
    const int kvh = blockIdx.x, split = blockIdx.y;

    const int64_t qpos = clamp_i64(qs[0], 0, cap - 1);   // DynamicSlice clamp (cpu.rs:804-820)
    const int64_t upd = clamp_i64(us[1], 0, cap - 1);    // DynamicUpdateSlice clamp on the position axis
    const T* knew = qkv + (int64_t)n_q * dh + (int64_t)kvh * dh;
    const T* vnew = qkv + (int64_t)(n_q + n_kv) * dh + (int64_t)kvh * dh;

    // append this step's row (exactly one block per kv head owns position `upd`)
    if (upd / chunk == split) {
        for (int d = threadIdx.x; d < dh; d += 256) {
            kc[((int64_t)kvh * cap + upd) * dh + d] = cs ? roped_elem<T>(knew, d, half, cs, sn) : knew[d];
            vc[((int64_t)kvh * cap + upd) * dh + d] = vnew[d];
        }
    }

    const int64_t p0 = (int64_t)split * chunk;
    int64_t p1 = p0 + chunk;
    if (p1 > qpos + 1) p1 = qpos + 1;

    float qf[G][VEC];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const T* qh = qkv + (int64_t)(kvh * G + g) * dh;
        if (cs) load_roped<T>(qh, li * VEC, half, cs, sn, qf[g]);
        else Vec16<T>::load(qh + li * VEC, qf[g]);
    }

    float m[G], l[G], o[G][VEC];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        m[g] = -INFINITY; l[g] = 0.f;
#pragma unroll
        for (int v = 0; v < VEC; ++v) o[g][v] = 0.f;
    }

    // Two positions per lane-group are loaded before either is consumed (the kernel is bound by
    // load latency, not bandwidth); a position past the end re-reads a valid row and is skipped.
    for (int64_t base = p0 + sid; base < p1; base += 2 * nstream) {
        float kf2[2][VEC], vf2[2][VEC];
        bool live[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int64_t p = base + (int64_t)j * nstream;
            live[j] = p < p1;
            const int64_t pc = live[j] ? p : base;
            const bool fresh = pc == upd;
            const T* kr = fresh ? knew : kc + ((int64_t)kvh * cap + pc) * dh;
            const T* vr = fresh ? vnew : vc + ((int64_t)kvh * cap + pc) * dh;
            if (cs && fresh) load_roped<T>(knew, li * VEC, half, cs, sn, kf2[j]);
            else Vec16<T>::load(kr + li * VEC, kf2[j]);
            Vec16<T>::load(vr + li * VEC, vf2[j]);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
        if (!live[j]) continue;
        const float (&kf)[VEC] = kf2[j];
        const float (&vf)[VEC] = vf2[j];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float s = 0.f;
#pragma unroll
            for (int v = 0; v < VEC; ++v) s += qf[g][v] * kf[v];
            for (int off = 1; off < lpr; off <<= 1) s += __shfl_xor(s, off, 64);
            s *= scale;
            const float mn = fmaxf(m[g], s);
            const float corr = expf(m[g] - mn);
            const float pe = expf(s - mn);
            l[g] = l[g] * corr + pe;
#pragma unroll
            for (int v = 0; v < VEC; ++v) o[g][v] = o[g][v] * corr + pe * vf[v];
            m[g] = mn;
        }
        }
    }

    // merge the rpw lane-groups of this wave
    for (int off = lpr; off < 64; off <<= 1) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const float om = __shfl_xor(m[g], off, 64);
            const float ol = __shfl_xor(l[g], off, 64);
            const float mn = fmaxf(m[g], om);
            const float ca = mn == -INFINITY ? 0.f : expf(m[g] - mn);
            const float cb = mn == -INFINITY ? 0.f : expf(om - mn);
            l[g] = l[g] * ca + ol * cb;
#pragma unroll
            for (int v = 0; v < VEC; ++v) {
                const float ov = __shfl_xor(o[g][v], off, 64);
                o[g][v] = o[g][v] * ca + ov * cb;
            }
            m[g] = mn;
        }
    }

    // merge the four waves through LDS
    __shared__ float sm[4][G], sl[4][G];
    __shared__ float so[4][G][256];
    if (sub == 0) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            if (li == 0) { sm[wave][g] = m[g]; sl[wave][g] = l[g]; }
#pragma unroll
            for (int v = 0; v < VEC; ++v) so[wave][g][li * VEC + v] = o[g][v];
        }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < G * dh; idx += 256) {
        const int g = idx / dh, d = idx % dh;
        float mn = fmaxf(fmaxf(sm[0][g], sm[1][g]), fmaxf(sm[2][g], sm[3][g]));
        float L = 0.f, O = 0.f;
        if (mn != -INFINITY) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float c = expf(sm[w][g] - mn);
                L += sl[w][g] * c;
                O += so[w][g][d] * c;
            }
        }
        const int h = kvh * G + g;
        if (nsplit == 1) {
            stf(ctx, (int64_t)h * dh + d, O / L);
        } else {
            float* rec = ws + ((int64_t)h * nsplit + split) * (dh + 2);
            if (d == 0) { rec[0] = mn; rec[1] = L; }
            rec[2 + d] = O;
        }
    }
}

// max / sum of a value over the two half-waves, in every lane: v_permlane32_swap leaves the low half's value in one
// register and the high half's in the other (one VALU instruction instead of a round trip through the LDS crossbar)
__device__ __forceinline__ float half_max(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// bf16 decode attention with the scores on the matrix cores.  grid (n_kv, nsplit, batch), 256 threads; wave w of a
// workgroup takes the 32-key tiles w, w+4, ... of the workgroup's share, the rows of its next tile in flight while it works on one.
// Bound by the caches' rows; 8 sequences of 1000 positions of 8 kv heads of 128 (33 MB), capacity 2048: 18.1 -> 14.5 us since the
// attended tiles, not the capacity, are shared out and all workgroups are resident at once; with the merge of the records behind it 18.9 -> 16.8 us (2 x 3000 18.8 -> 17.1, 8 x 30
// 9.3 -> 8.4) with fused multiply-adds, four weights to an LDS read and exchanges that halve the values.  The merge by the workgroup that draws a kv head's last ticket instead of
// a launch: 19.5, 33.1 and 9.7.  Per tile
//   S^T[key, q] = K[key, :] . Q[q, :]   v_mfma_f32_32x32x16_bf16, A = cache rows, read whole and turned in LDS (lane = key row),
//                                       B = the group's G query heads in columns 0..G-1 (other columns repeat them)
// so a lane owns ONE query: its 16 scores, the running maximum and sum (log2 domain) are per-lane values and the
// softmax costs a few instructions per key instead of a cross-lane reduction per key and head.  The probabilities go
// through LDS to the layout of the second product, which stays on the vector ALUs in f32: lane-group `sub` (DH/8
// lanes, 16 bytes of a V row each) accumulates O[g, :] over its keys of the tile.  States are merged across
// lane-groups by shuffles, across waves through LDS, across splits by attn_decode_combine_kernel (same records as
// attn_decode_kernel, maxima in natural-log units).
// Two values of every lane, lane ^ OFF exchanged: the lanes below keep a, those above b, each added up over the pair.
template <int OFF> __device__ __forceinline__ float lane_halves(float a, float b) {
    static_assert(OFF == 16 || OFF == 32, "swaps that the hardware has");
    const auto r = OFF == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false)
                             : __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
template <int DH, int G>
__global__ __launch_bounds__(256, DH * G == 1024 ? 1 : 2) void attn_decode_mfma_kernel(const bf16_t* __restrict__ qkv, bf16_t* __restrict__ kc,
                                                               bf16_t* __restrict__ vc, const int32_t* __restrict__ us,
                                                               const int32_t* __restrict__ qs, bf16_t* __restrict__ ctx,
                                                               float* __restrict__ ws, int n_q, int n_kv, int64_t cap,
                                                               float scale_log2e, int nsplit,
                                                               const bf16_t* __restrict__ cs, const bf16_t* __restrict__ sn,
                                                               int half_rot, int batched, DecodeCaches caches) {
    constexpr int NK = DH / 16;        // k-steps of the score product
    constexpr int LPR = DH / 8;        // lanes per V row
    constexpr int NSUB = 64 / LPR;     // lane-groups per wave
    constexpr int NV = 32 / NSUB;      // keys of a tile per lane-group
    __shared__ __align__(16) float p_lds[4][G][32];
    __shared__ float corr_lds[4][G];
    __shared__ float sm[4][G], sl[4][G];
    __shared__ float so[4][G][DH];
    __shared__ __align__(16) bf16_t q_lds[G][DH], k_lds[DH], kt_lds[4][32][DH];
    if (batched) {
        const int b = blockIdx.z;
        kc = (bf16_t*)caches.k[b];
        vc = (bf16_t*)caches.v[b];
        qkv += (int64_t)b * (n_q + 2 * n_kv) * DH;
        ctx += (int64_t)b * n_q * DH;
        ws += (int64_t)b * n_q * nsplit * (DH + 2);
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, half = lane >> 5;
    const int sub = lane / LPR, li = lane % LPR;
    const int kvh = blockIdx.x, split = blockIdx.y;
    const int64_t qpos = clamp_i64(qs[0], 0, cap - 1);
    const int64_t upd = clamp_i64(us[1], 0, cap - 1);
    const bf16_t* knew = qkv + (int64_t)n_q * DH + (int64_t)kvh * DH;
    const bf16_t* vnew = qkv + (int64_t)(n_q + n_kv) * DH + (int64_t)kvh * DH;
    bf16_t* kbase = kc + (int64_t)kvh * cap * DH;
    bf16_t* vbase = vc + (int64_t)kvh * cap * DH;

    // the tiles that are attended at this position, shared out evenly: shares of the capacity left the workgroups behind the position
    // idle in front of the others (half of the chip at half the capacity)
    const unsigned tiles = (unsigned)(qpos / 32) + 1, share = (tiles + nsplit - 1) / nsplit, own_split = (unsigned)(upd / 32) / share;
    const bool owner = (own_split < (unsigned)nsplit ? own_split : nsplit - 1) == split;
    const int64_t p0 = (int64_t)split * share * 32;
    const int left = qpos + 1 - p0 < (int64_t)share * 32 ? (int)(qpos + 1 - p0) : (int)(share * 32);   // keys of this split
    const int ntiles = left > 0 ? (left + 31) / 32 : 0;
    const int fresh = upd - p0 >= 0 && upd - p0 < left ? (int)(upd - p0) : -1;                        // this step's row among them
    // the cache rows of a wave's first tile are requested before anything else is waited for, whole rows at a time (a lane group to a
    // row).  Rows past the last attended position re-read that position and get probability zero; this step's row, which the caches do
    // not hold yet, comes from LDS (K) and from the projection itself (V)
    const int64_t base = left > 0 ? p0 : 0;
    kbase += base * DH;
    vbase += base * DH;
    u32x4_v kreg[NV], vreg[NV];
    const auto load_k = [&](int k0) {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int r = max(min(k0 + NV * sub + j, left - 1), 0);
            kreg[j] = *reinterpret_cast<const u32x4_v*>(kbase + (unsigned)(r * DH + li * 8));
        }
    };
    const auto load_v = [&](int k0) {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int r = max(min(k0 + NV * sub + j, left - 1), 0);
            vreg[j] = *reinterpret_cast<const u32x4_v*>(r == fresh ? vnew + li * 8 : vbase + (unsigned)(r * DH + li * 8));
        }
    };
    // this step's rows first, since loads are answered in order: LPR threads to each of the group's query heads, to the K row and to the
    // V row.  Dims below half_rot pair with dim + half_rot and the next half_rot with dim - half_rot, a thread's 8 all alike
    const int hd = tid / LPR, c0 = li * 8;
    const bool rot = cs && hd <= G && c0 < 2 * half_rot, first = c0 < half_rot;
    const bf16_t* src = hd < G ? qkv + (int64_t)(kvh * G + hd) * DH : hd == G ? knew : vnew;
    const int other = rot ? (first ? c0 + half_rot : c0 - half_rot) : c0, cj = first ? c0 : c0 - half_rot;
    // every thread loads, and every wave a tile: under a branch the waits for these rows would wait for the caches as well
    u32x4_v own = *reinterpret_cast<const u32x4_v*>(src + c0);
    const u32x4_v oth = *reinterpret_cast<const u32x4_v*>(src + other);
    const u32x4_v cosv = *reinterpret_cast<const u32x4_v*>(rot ? cs + cj : src + c0);
    const u32x4_v sinv = *reinterpret_cast<const u32x4_v*>(rot ? sn + cj : src + c0);
    load_k(wave * 32);
    load_v(wave * 32);
    if (hd < G + 2 && (hd < G || owner)) {
        if (rot) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float a0 = bf16lo(own[e]), a1 = bf16hi(own[e]), b0 = bf16lo(oth[e]), b1 = bf16hi(oth[e]);
                const float x0 = a0 * bf16lo(cosv[e]), x1 = a1 * bf16hi(cosv[e]), y0 = b0 * bf16lo(sinv[e]), y1 = b1 * bf16hi(sinv[e]);
                own[e] = (unsigned)f32_to_bf16(first ? x0 - y0 : x0 + y0) | (unsigned)f32_to_bf16(first ? x1 - y1 : x1 + y1) << 16;
            }
        }
        if (hd <= G) *reinterpret_cast<u32x4_v*>(hd < G ? &q_lds[hd][c0] : &k_lds[c0]) = own;
        // one workgroup per kv head owns position `upd`, and no other reads it
        if (hd >= G) *reinterpret_cast<u32x4_v*>((hd == G ? kbase : vbase) + (upd - base) * DH + c0) = own;
    }
    if (ntiles == 0) {   // a split behind the position: an empty record (split 0 always has a key)
        for (int idx = tid; idx < G * (DH + 2); idx += 256) {
            const int g = idx / (DH + 2), d = idx % (DH + 2);
            ws[((int64_t)(kvh * G + g) * nsplit + split) * (DH + 2) + d] = d == 0 ? -INFINITY : 0.f;
        }
        return;
    }
    __syncthreads();

    float o[G][8];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int e = 0; e < 8; ++e) o[g][e] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    for (int t = wave; t < ntiles; t += 4) {   // waves are on their own: LDS of one wave, in the order of its instructions
        const int k0 = t * 32;
        // 16-byte pieces moved about by their row so that neither side meets bank conflicts
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int r = NV * sub + j;
            *reinterpret_cast<u32x4_v*>(&kt_lds[wave][r][(li ^ (r & (LPR - 1))) * 8]) = kreg[j];
        }
        if ((unsigned)(fresh - k0) < 32u && lane < LPR)
            *reinterpret_cast<u32x4_v*>(&kt_lds[wave][fresh - k0][(lane ^ ((fresh - k0) & (LPR - 1))) * 8]) = *reinterpret_cast<const u32x4_v*>(&k_lds[lane * 8]);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (t + 4 < ntiles) load_k(k0 + 128);
        f32x16_v sc;
#pragma unroll
        for (int v = 0; v < 16; ++v) sc[v] = 0.f;
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) {   // A: key `col`; B: query head col % G, 8 consecutive d per lane and k-step
            const bf16x8_v kf = *reinterpret_cast<const bf16x8_v*>(&kt_lds[wave][col][((2 * kk + half) ^ (col & (LPR - 1))) * 8]);
            const bf16x8_v qf = *reinterpret_cast<const bf16x8_v*>(&q_lds[col % G][16 * kk + 8 * half]);
            sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf, sc, 0, 0, 0);
        }
        float mx = -INFINITY;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const float x = k0 + 8 * (v >> 2) + (v & 3) + 4 * half < left ? sc[v] * scale_log2e : -INFINITY;
            sc[v] = x;
            mx = fmaxf(mx, x);
        }
        mx = half_max(mx);
        const float m_new = fmaxf(m_run, mx);   // finite: the tile holds at least one attended key
        const float corr = __builtin_amdgcn_exp2f(m_run - m_new);
        float ls = 0.f;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            sc[v] = __builtin_amdgcn_exp2f(sc[v] - m_new);
            ls += sc[v];
        }
        ls = half_sum(ls);
        l_run = l_run * corr + ls;
        m_run = m_new;
        if (col < G) {
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
                *reinterpret_cast<float4*>(&p_lds[wave][col][8 * q4 + 4 * half]) =
                    make_float4(sc[4 * q4], sc[4 * q4 + 1], sc[4 * q4 + 2], sc[4 * q4 + 3]);
            if (half == 0) corr_lds[wave][col] = corr;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const float c = corr_lds[wave][g];
#pragma unroll
            for (int e = 0; e < 8; ++e) o[g][e] *= c;
        }
        float pr[G][NV];
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int j = 0; j < NV; j += 4) {
                const float4 p4 = *reinterpret_cast<const float4*>(&p_lds[wave][g][NV * sub + j]);
                pr[g][j] = p4.x; pr[g][j + 1] = p4.y; pr[g][j + 2] = p4.z; pr[g][j + 3] = p4.w;
            }
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const float vf[8] = {bf16lo(vreg[j][0]), bf16hi(vreg[j][0]), bf16lo(vreg[j][1]), bf16hi(vreg[j][1]),
                                 bf16lo(vreg[j][2]), bf16hi(vreg[j][2]), bf16lo(vreg[j][3]), bf16hi(vreg[j][3])};
#pragma unroll
            for (int g = 0; g < G; ++g) {
#pragma unroll
                for (int e = 0; e < 8; ++e) o[g][e] = __builtin_fmaf(pr[g][j], vf[e], o[g][e]);
            }
        }
        if (t + 4 < ntiles) load_v(k0 + 128);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }

    // merge the lane-groups of this wave (they share the wave's maximum), then the four waves through LDS.  The lanes exchanged with go on with half of the values
    // each time (o[g][e] in a row: bits 5, 4 and 3 of the lane say which), so 32 values take 24 exchanges, not 64
    float w0[G * 8], w1[G * 4], w2[G * 2];
#pragma unroll
    for (int i = 0; i < G * 8; ++i) w0[i] = o[i >> 3][i & 7];
#pragma unroll
    for (int i = 0; i < G * 4; ++i) w1[i] = lane_halves<32>(w0[i], w0[i + G * 4]);
#pragma unroll
    for (int i = 0; i < G * 2; ++i) w2[i] = lane_halves<16>(w1[i], w1[i + G * 2]);
    const int first_value = (lane >> 5) * (G * 4) + ((lane >> 4) & 1) * (G * 2);
    if constexpr (NSUB == 4) {
#pragma unroll
        for (int i = 0; i < G * 2; ++i) so[wave][(first_value + i) >> 3][li * 8 + ((first_value + i) & 7)] = w2[i];
    } else {
        const bool up = lane & 8;
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const float keep = up ? w2[i + G] : w2[i], give = up ? w2[i] : w2[i + G];
            const int at = first_value + (up ? G : 0) + i;
            so[wave][at >> 3][li * 8 + (at & 7)] = keep + dpp_move<0x128>(give);   // row_ror:8
        }
    }
    if (lane < G) { sm[wave][lane] = m_run; sl[wave][lane] = l_run; }
    __syncthreads();
    for (int idx = tid; idx < G * DH; idx += 256) {
        const int g = idx / DH, d = idx % DH;
        const float mn = fmaxf(fmaxf(sm[0][g], sm[1][g]), fmaxf(sm[2][g], sm[3][g]));
        float L = 0.f, O = 0.f;
        if (mn != -INFINITY) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float c = exp2f(sm[w][g] - mn);
                L += sl[w][g] * c;
                O += so[w][g][d] * c;
            }
        }
        const int h = kvh * G + g;
        if (nsplit == 1) {
            stf(ctx, (int64_t)h * DH + d, O / L);
        } else {
            float* rec = ws + ((int64_t)h * nsplit + split) * (DH + 2);
            if (d == 0) { rec[0] = mn * 0.6931471805599453f; rec[1] = L; }
            rec[2 + d] = O;
        }
    }
}

template <typename T>
__global__ void attn_decode_combine_kernel(const float* __restrict__ ws, T* __restrict__ ctx, int dh, int nsplit) {
    // grid (n_q, batch): sequence blockIdx.y owns gridDim.x heads of records and of the context
    ws += (int64_t)blockIdx.y * gridDim.x * nsplit * (dh + 2);
    ctx += (int64_t)blockIdx.y * gridDim.x * dh;
    // eight records at a time, all of their loads independent: every thread keeps the running maximum and sum for itself (LDS
    // reductions of the two, with their four barriers and three rounds of dependent loads, took 4.8 us for 16 splits)
    const int h = blockIdx.x;
    const float* base = ws + (int64_t)h * nsplit * (dh + 2);
    for (int d = threadIdx.x; d < dh; d += blockDim.x) {
        float mn = -INFINITY, L = 0.f, O = 0.f;
        for (int s0 = 0; s0 < nsplit; s0 += 8) {
            float m[8], l[8], o[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float* rec = base + (int64_t)(s0 + j < nsplit ? s0 + j : nsplit - 1) * (dh + 2);
                m[j] = rec[0]; l[j] = rec[1]; o[j] = rec[2 + d];
            }
            float mx = mn;
#pragma unroll
            for (int j = 0; j < 8; ++j) if (s0 + j < nsplit) mx = fmaxf(mx, m[j]);
            const float at = mx == -INFINITY ? 0.f : mx;     // nothing but empty records so far: any finite stand-in, for these eight alone
            const float c0 = expf(mn - at);
            L *= c0;
            O *= c0;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (s0 + j < nsplit) {
                    const float c = expf(m[j] - at);
                    L += l[j] * c;
                    O += o[j] * c;
                }
            }
            mn = mx;
        }
        stf(ctx, (int64_t)h * dh + d, O / L);
    }
}

// Launch geometry shared by attn_decode() and attn_decode_workspace_bytes(): chunks of two
// positions per lane-group, capped at kMaxDecodeSplits splits.
static void decode_geometry(int dtype, int64_t dh, int64_t cap, int* nsplit, int64_t* chunk) {
    const int64_t vec = dtype == 0 ? 4 : 8;
    const int64_t lpr = dh / vec > 0 ? dh / vec : 1;
    const int64_t nstream = 4 * (64 / lpr);
    int64_t c = 2 * nstream;
    if (cdiv(cap, c) > kMaxDecodeSplits) c = cdiv(cdiv(cap, kMaxDecodeSplits), 2 * nstream) * 2 * nstream;
    *chunk = c;
    *nsplit = (int)cdiv(cap, c);
}
size_t attn_decode_workspace_bytes(int64_t n_q, int64_t head_dim, int64_t capacity) {
    int ns0, ns2;
    int64_t c;
    decode_geometry(0, head_dim, capacity, &ns0, &c);
    decode_geometry(2, head_dim, capacity, &ns2, &c);
    const int ns = ns0 > ns2 ? ns0 : ns2;
    return (size_t)n_q * (size_t)ns * (size_t)(head_dim + 2) * sizeof(float);
}

// Matrix-core decode path: bf16, head_dim 64 / 128, group sizes 1, 2, 4, 8 (GPTRS_HIP_MFMA_ATTN=0 turns it off).
static bool attn_decode_mfma_ok(const AttnDecodeArgs& a) {
    static const bool use = [] { const char* e = getenv("GPTRS_HIP_MFMA_ATTN"); return !(e && e[0] == '0'); }();
    if (!use || a.dtype != 2 || a.n_kv <= 0 || a.n_q % a.n_kv != 0) return false;
    if (a.head_dim != 64 && a.head_dim != 128) return false;
    if (a.cos && a.rot_half % 8 != 0) return false;
    const int64_t g = a.n_q / a.n_kv;
    return g == 1 || g == 2 || g == 4 || g == 8;
}

static int attn_decode_mfma(hipStream_t s, const AttnDecodeArgs& a) {
    int nsplit;
    int64_t chunk;
    decode_geometry(a.dtype, a.head_dim, a.capacity, &nsplit, &chunk);   // the workspace holds this many splits
    const int nb = a.batch > 1 ? a.batch : 1;
    // at most the two workgroups per CU that its registers hold (one with 8 heads of 128): one round whose waves have their loads in flight together
    const int64_t most = (a.head_dim * a.n_q == 1024 * a.n_kv ? 256 : 512) / ((int64_t)a.n_kv * nb), tiles = cdiv(a.capacity, 32);
    if (nsplit > tiles) nsplit = (int)tiles;
    if (nsplit > most) nsplit = most > 1 ? (int)most : 1;
    dim3 grid((unsigned)a.n_kv, (unsigned)nsplit, (unsigned)nb);
    DecodeCaches caches{};
    for (int b = 0; b < nb && b < 16; ++b) { caches.k[b] = a.k_caches[b]; caches.v[b] = a.v_caches[b]; }
    const float sl = a.scale * 1.44269504088896f;
    const int g = (int)(a.n_q / a.n_kv);
#define GPTRS_LAUNCH(DH, G)                                                                                          \
    attn_decode_mfma_kernel<DH, G><<<grid, 256, 0, s>>>((const bf16_t*)a.qkv, (bf16_t*)a.k_cache, (bf16_t*)a.v_cache, \
        a.update_starts, a.query_start, (bf16_t*)a.ctx, (float*)a.ws, (int)a.n_q, (int)a.n_kv, a.capacity, sl, nsplit, \
        (const bf16_t*)a.cos, (const bf16_t*)a.sin, (int)a.rot_half, a.batch > 1 ? 1 : 0, caches)
#define GPTRS_LAUNCH_G(DH)                                                                                           \
    switch (g) {                                                                                                     \
        case 1: GPTRS_LAUNCH(DH, 1); break;                                                                          \
        case 2: GPTRS_LAUNCH(DH, 2); break;                                                                          \
        case 4: GPTRS_LAUNCH(DH, 4); break;                                                                          \
        default: GPTRS_LAUNCH(DH, 8); break;                                                                         \
    }
    if (a.head_dim == 64) { GPTRS_LAUNCH_G(64) } else { GPTRS_LAUNCH_G(128) }
#undef GPTRS_LAUNCH_G
#undef GPTRS_LAUNCH
    if (nsplit > 1) {
        const int block = a.head_dim <= 64 ? 64 : 128;
        attn_decode_combine_kernel<bf16_t><<<dim3((unsigned)a.n_q, (unsigned)nb), block, 0, s>>>((const float*)a.ws, (bf16_t*)a.ctx, (int)a.head_dim, nsplit);
    }
    return nsplit > 1 ? 2 : 1;
}

template <typename T>
static int attn_decode_t(hipStream_t s, const AttnDecodeArgs& a) {
    int nsplit;
    int64_t chunk;
    decode_geometry(a.dtype, a.head_dim, a.capacity, &nsplit, &chunk);
    const int nb = a.batch > 1 ? a.batch : 1;
    // a batch multiplies the workgroups: longer chunks keep the launch near six workgroups per CU, so the fixed cost
    // of a workgroup (query load, state merges, record) is spread over more positions (fewer splits than the
    // workspace was sized for is always safe)
    const int64_t step = chunk;
    while (nsplit > 1 && (int64_t)a.n_kv * nb * nsplit > 1536) {
        chunk += step;
        nsplit = (int)cdiv(a.capacity, chunk);
    }
    // a short cache is one chunk: the workgroup walks only the positions that are valid (its loop ends at the query
    // position, at most four rounds of loads), stores the context row itself, and the launch of the combine kernel is
    // saved (GPT-2 generate 64 at capacity 128: 1910 -> 1999 tokens/s; at capacity 256 the longer walk costs what the
    // launch saves)
    if (a.capacity <= 128) { chunk = a.capacity; nsplit = 1; }
    dim3 grid((unsigned)a.n_kv, (unsigned)nsplit, (unsigned)nb);
    const int g = (int)(a.n_q / a.n_kv);
    DecodeCaches caches{};
    for (int b = 0; b < nb && b < 16; ++b) { caches.k[b] = a.k_caches[b]; caches.v[b] = a.v_caches[b]; }
#define GPTRS_LAUNCH(G)                                                                                          \
    attn_decode_kernel<T, G><<<grid, 256, 0, s>>>((const T*)a.qkv, (T*)a.k_cache, (T*)a.v_cache, a.update_starts,    \
        a.query_start, (T*)a.ctx, (float*)a.ws, (int)a.n_q, (int)a.n_kv, (int)a.head_dim, a.capacity, a.scale, chunk, nsplit, \
        (const T*)a.cos, (const T*)a.sin, (int)a.rot_half, a.batch > 1 ? 1 : 0, caches)
    switch (g) {
        case 1: GPTRS_LAUNCH(1); break;
        case 2: GPTRS_LAUNCH(2); break;
        case 4: GPTRS_LAUNCH(4); break;
        default: GPTRS_LAUNCH(8); break;
    }
#undef GPTRS_LAUNCH
    if (nsplit > 1) {
        const int block = a.head_dim <= 64 ? 64 : (a.head_dim <= 128 ? 128 : 256);
        attn_decode_combine_kernel<T><<<dim3((unsigned)a.n_q, (unsigned)nb), block, 0, s>>>((const float*)a.ws, (T*)a.ctx, (int)a.head_dim, nsplit);
    }
    return nsplit > 1 ? 2 : 1;
}
int attn_decode(hipStream_t s, const AttnDecodeArgs& a) {
    if (attn_decode_mfma_ok(a)) return attn_decode_mfma(s, a);
    return a.dtype == 0 ? attn_decode_t<float>(s, a) : attn_decode_t<bf16_t>(s, a);
}

// Where the K / V rows of a prefill's sequences lie: in the caches attn_prefill_kv_kernel has put them into, or (no `starts`)
// in the packed rows themselves.
template <typename T> struct PrefillKv {
    const T* k[kAttnBatch];
    const T* v[kAttnBatch];
    const int32_t* starts;
    int64_t capacity;
    const T* cos;
    const T* sin;
};
template <typename T>
__device__ __forceinline__ const T* prefill_rows(const T* const* caches, const PrefillKv<T>& kv, const T* rows, int seq, int kvh, int dh, int t, int64_t row_pitch,
                                                 int64_t col, int64_t& pitch) {
    if (!kv.starts) { pitch = row_pitch; return rows + col; }
    pitch = dh;
    const int64_t at = min(max((int64_t)kv.starts[1], (int64_t)0), kv.capacity - t);
    return caches[seq] + (kvh * kv.capacity + at) * dh;
}

// The K and V columns of stacked packed rows [batch * t, P] -> the sequences' caches [n_kv, capacity, dh] at the row the update
// names, the keys rotated on the way (the arithmetic and rounding of rope_kernel).  One thread per 16 bytes; bound by memory: a
// third of the projection read once and written once, where a rotation of all rows, a copy of every sequence's rows and two
// cache updates per sequence took 164 us a layer at 4 x 2047 tokens of 32 + 2 x 8 heads of 128.
template <typename T>
__global__ __launch_bounds__(256) void attn_prefill_kv_kernel(const T* __restrict__ qkv, int64_t chunks, int t, int n_q, int n_kv, int dh, PrefillKv<T> kv) {
    constexpr int VEC = 16 / sizeof(T);
    typedef T vec_t __attribute__((ext_vector_type(VEC)));
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= chunks) return;
    const int hc = dh / VEC, rc = 2 * n_kv * hc;        // chunks of a head, of a row's K and V
    const int64_t row = id / rc;
    const int c = (int)(id % rc), head = c / hc, d = c % hc * VEC;
    const int seq = (int)(row / t), pos = (int)(row % t);
    const T* src = qkv + row * ((int64_t)(n_q + 2 * n_kv) * dh) + (int64_t)(n_q + head) * dh;
    vec_t x = *reinterpret_cast<const vec_t*>(src + d);
    const bool key = head < n_kv;
    if (key && kv.cos) {
        const int h2 = dh / 2;
        const bool second = d >= h2;
        const int j = second ? d - h2 : d;
        const vec_t y = *reinterpret_cast<const vec_t*>(src + (second ? j : d + h2));
        const vec_t cv = *reinterpret_cast<const vec_t*>(kv.cos + (int64_t)pos * h2 + j), sv = *reinterpret_cast<const vec_t*>(kv.sin + (int64_t)pos * h2 + j);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const T xe = x[e], ye = y[e], ce = cv[e], se = sv[e];
            const float xf = ldf(&xe, 0), yf = ldf(&ye, 0), cf = ldf(&ce, 0), sf = ldf(&se, 0);
            T out;
            stf(&out, 0, second ? xf * cf + yf * sf : xf * cf - yf * sf);
            x[e] = out;
        }
    }
    const int64_t at = min(max((int64_t)kv.starts[1], (int64_t)0), kv.capacity - t) + pos;
    T* to = const_cast<T*>(key ? kv.k[seq] : kv.v[seq]) + ((int64_t)(key ? head : head - n_kv) * kv.capacity + at) * dh + d;
    *reinterpret_cast<vec_t*>(to) = x;
}

// Prompts of one row tile (at most 32 rows where 4 query heads share keys, 128 where one has them alone): the one workgroup of a kv head that sees all
// of its keys puts them into the caches itself, on their way to LDS, and the launch of attn_prefill_kv_kernel is saved.  One 16-byte chunk of
// a K row, rotated as that kernel does it; T: element, `second`: the chunk lies in the rotated half that adds.
template <typename T, typename V>
__device__ __forceinline__ V rotated_chunk(const V& own, const V& other, const V& c, const V& s, bool second) {
    constexpr int VEC = 16 / sizeof(T);
    alignas(16) T x[VEC], y[VEC], cv[VEC], sv[VEC];
    *reinterpret_cast<V*>(x) = own; *reinterpret_cast<V*>(y) = other; *reinterpret_cast<V*>(cv) = c; *reinterpret_cast<V*>(sv) = s;
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
        const float xf = ldf(x, e), yf = ldf(y, e), cf = ldf(cv, e), sf = ldf(sv, e);
        stf(x, e, second ? xf * cf + yf * sf : xf * cf - yf * sf);
    }
    return *reinterpret_cast<const V*>(x);
}

// ------------------------------------------------------------------------------ prefill
// grid (ceil(T/4), n_q), 256 threads: one wave per query row.  Keys are visited 64 at a time
// (one per lane) with an online softmax; the P.V update then walks the chunk with the lanes
// spread over head_dim so V rows are read coalesced.
template <typename T>
__global__ __launch_bounds__(256) void attn_prefill_kernel(const T* __restrict__ qkv, T* __restrict__ ctx, int64_t t,
                                                           int n_q, int n_kv, int dh, float scale) {
    __shared__ float qsm[4][256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t i = (int64_t)blockIdx.x * 4 + wave;
    const int h = blockIdx.y;
    const int kvh = h / (n_q / n_kv);
    const int64_t P = (int64_t)(n_q + 2 * n_kv) * dh;
    const int64_t koff = (int64_t)n_q * dh + (int64_t)kvh * dh;
    const int64_t voff = (int64_t)(n_q + n_kv) * dh + (int64_t)kvh * dh;
    if (i < t)
        for (int d = lane; d < dh; d += 64) qsm[wave][d] = ldf(qkv, i * P + (int64_t)h * dh + d);
    __syncthreads();
    if (i >= t) return;
    float m = -INFINITY, l = 0.f;
    float o[4] = {0.f, 0.f, 0.f, 0.f};
    for (int64_t j0 = 0; j0 <= i; j0 += 64) {
        const int64_t j = j0 + lane;
        float s = -INFINITY;
        if (j <= i) {
            const T* kr = qkv + j * P + koff;
            float acc = 0.f;
            for (int d = 0; d < dh; ++d) acc += qsm[wave][d] * ldf(kr, d);
            s = acc * scale;
        }
        const float mn = fmaxf(m, wave_max(s));
        const float corr = expf(m - mn);
        const float pe = j <= i ? expf(s - mn) : 0.f;
        l = l * corr + wave_sum(pe);
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c] *= corr;
        const int cnt = (int)((i - j0 + 1) < 64 ? (i - j0 + 1) : 64);
        for (int jj = 0; jj < cnt; ++jj) {
            const float pj = __shfl(pe, jj, 64);
            const T* vr = qkv + (j0 + jj) * P + voff;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int d = lane + 64 * c;
                if (d < dh) o[c] += pj * ldf(vr, d);
            }
        }
        m = mn;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int d = lane + 64 * c;
        if (d < dh) stf(ctx, i * (int64_t)n_q * dh + (int64_t)h * dh + d, o[c] / l);
    }
}
// bf16 prefill attention on the matrix cores (flash-attention style, causal, grouped-query).
//
// A workgroup (4 waves) serves one kv head and up to 4 query heads of its group over 32 query rows each, so a key /
// value tile staged in LDS is used by every query head that shares it and all waves see the same causal range.  Per
// tile of 32 keys a wave computes with v_mfma_f32_32x32x16_bf16
//   S^T[key, q] = K[key, :] . Q[q, :]      (A = K rows from LDS, B = Q fragments kept in registers)
//   O^T[d, q]  += V^T[d, key] . P^T[key, q] (A = V^T from LDS, B = the probabilities just computed, from registers)
// Both products are taken transposed so that a lane always owns ONE query (column lane % 32): the 16 scores a lane
// holds belong to its query, the online-softmax state (running maximum and sum, in the log2 domain) is a per-lane
// scalar, the rescaling of O^T is a per-lane multiply, and P^T needs no cross-lane movement to become the B operand:
// the k-slots of the second product are simply numbered in the order the lane holds its keys, and V^T is read out of V's rows in LDS in
// that order by transposing reads.  (Writing V^T into LDS, two bytes at a time, took 16 stores a thread and tile and 53 KB of
// it; without, three workgroups share a CU instead of two.  us a layer, 32 / 8 heads of 128: 4 x 2047 rows 234 -> 199, 1 x 4000 198 -> 176,
// 8 x 1000 137 -> 120, 1 x 1024 37.0 -> 36.2.)
// KG = 2: the workgroup has two groups of four waves; both serve the same queries, group g takes the key tiles
// 2 s + g (it stages them itself, into its own LDS buffers), and the two online-softmax states meet through LDS at the
// end.  A row tile then takes half as many steps, and a SIMD holds two waves whose matrix and vector phases overlap
// (the launch has one wave-sized task per SIMD otherwise).
// KG = 4, HW = 2: four groups of two waves, two query heads to a workgroup: half the steps again, and twice the workgroups, for launches that leave
// most CUs idle (143 KB of LDS, one workgroup to a CU).  What is left of 333 rows' 13.6 us is 9 that two steps also take: the start, the
// first rows' arrival and code that no launch before has brought.  Filling the caches on the way, which saves attn_prefill_kv_kernel's 4.8 us,
// was level at best: keys are turned again by every row tile (13.6 + 4.9 -> 20.8).  Asking for the first tile ahead of turning the queries gave 14.6.
// V^T as the A operand of a 32 x 32 x 16 product, out of 16 rows of V from v on (keys down, 32 d across): lane 32 h + c holds, of d = c, the
// keys 4 h .. 4 h + 3 and 8 + 4 h .. 8 + 4 h + 3, the order in which the scores' lanes hold theirs.  Two transposing reads: lane i of 16 gets
// column i of four rows, lane 4 e + j of the 16 names columns 4 j .. 4 j + 3 of row e.
__device__ __forceinline__ bf16x8_v v_fragment(const bf16_t* v, int stride, int lane) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4* lds_p;
    const int c = lane & 15;
    const bf16_t* p = v + (4 * (lane >> 5) + (c >> 2)) * stride + (lane & 16) + 4 * (c & 3);
    const u32x2_m lo = __builtin_bit_cast(u32x2_m, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_p)(p)));
    const u32x2_m hi = __builtin_bit_cast(u32x2_m, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_p)(p + 8 * stride)));
    u32x4_m r;
    r.x = lo.x; r.y = lo.y; r.z = hi.x; r.w = hi.y;
    return __builtin_bit_cast(bf16x8_v, r);
}

template <int DH, int KG, int HW, bool FILL>
__global__ __launch_bounds__(64 * HW * KG, KG > 1 ? 1 : FILL ? 2 : 3) void attn_prefill_mfma_kernel(const bf16_t* __restrict__ qkv, bf16_t* __restrict__ ctx, int T,
                                                                int n_q, int n_kv, float scale_log2e, int zgroups, PrefillKv<bf16_t> kv) {
    constexpr int KT = 32;            // keys per tile
    constexpr int KS = DH + 8;        // K tile row stride in elements (16 bytes of padding)
    constexpr int VS = DH + 16;       // V tile row stride: four rows of 16 d, which a transposing read takes at a time, lie in 32 different banks
    constexpr int ND = DH / 32;       // 32-row blocks of d in O^T
    constexpr int NK = DH / 16;       // k-steps of the score product
    constexpr int CH = KT * DH / 8;   // 16-byte chunks of a K (or V) tile
    constexpr int TPG = 64 * HW;      // threads of a key group
    constexpr int CPT = (CH + TPG - 1) / TPG;
    __shared__ __align__(16) bf16_t smem[KG * 2 * KT * (KS + VS)];

    static_assert(!FILL || KG == 1, "a workgroup that fills the caches sees every tile once");
    const int kg = KG == 4 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / TPG) : (int)threadIdx.x / TPG;   // key group of this wave
    const int tid = threadIdx.x % TPG, lane = tid & 63, wave = tid >> 6;
    bf16_t (*ksm)[KT * KS] = reinterpret_cast<bf16_t (*)[KT * KS]>(smem + kg * 2 * KT * KS);
    bf16_t (*vsm)[KT * VS] = reinterpret_cast<bf16_t (*)[KT * VS]>(smem + KG * 2 * KT * KS + kg * 2 * KT * VS);
    const int col = lane & 31, half = lane >> 5;
    const int G = n_q / n_kv;
    const int gw = G >= HW ? HW : G;               // query heads of the group in this workgroup
    const int rtpb = HW / gw;                      // 32-row tiles per workgroup
    const XcdTile at = xcd_tile();
    const int kvh = at.y;
    const int seq = at.z / zgroups, zg = at.z % zgroups;
    const int bx = gridDim.x - 1 - at.x;     // rows that see many keys first: the last workgroups to start are the short ones
    const int head = kvh * G + zg * gw + wave % gw;
    const int q0 = (bx * rtpb + wave / gw) * 32;
    const int64_t P = (int64_t)(n_q + 2 * n_kv) * DH;
    qkv += (int64_t)seq * T * P;
    ctx += (int64_t)seq * T * n_q * DH;
    int64_t kpitch;
    const auto* kp = prefill_rows(kv.k, kv, qkv, seq, kvh, DH, T, P, (int64_t)(n_q + kvh) * DH, kpitch);
    const auto* vp = prefill_rows(kv.v, kv, qkv, seq, kvh, DH, T, P, (int64_t)(n_q + n_kv + kvh) * DH, kpitch);
    bf16_t *kout = const_cast<bf16_t*>(kp), *vout = const_cast<bf16_t*>(vp);   // FILL: the caches' rows
    if (FILL) { kp = qkv + (int64_t)(n_q + kvh) * DH; vp = qkv + (int64_t)(n_q + n_kv + kvh) * DH; kpitch = P; }
    const int kend = min(T, (bx * rtpb + rtpb) * 32);   // keys any row of the workgroup may see
    const int ntiles = (kend + KT - 1) / KT;
    const bool active = q0 < T;
    const int my_tiles = active ? min(ntiles, (q0 + 31) / KT + 1) : 0;   // tiles holding a key <= this wave's last row

    // Q fragments (B operand: column = query, 8 consecutive d per lane and k-step)
    bf16x8_v qf[NK];
    {
        const int row = min(q0 + col, T - 1);
        const bf16_t* qp = qkv + (int64_t)row * P + (int64_t)head * DH + 8 * half;
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) qf[kk] = *reinterpret_cast<const bf16x8_v*>(qp + 16 * kk);
        if (kv.cos) {   // the rotated row, rounded to bf16 as the projection's rows are (rope_kernel); partners sit in one lane
#pragma unroll
            for (int kk = 0; kk < NK / 2; ++kk) {
                const bf16x8_v cv = *reinterpret_cast<const bf16x8_v*>(kv.cos + (int64_t)row * (DH / 2) + 16 * kk + 8 * half);
                const bf16x8_v sv = *reinterpret_cast<const bf16x8_v*>(kv.sin + (int64_t)row * (DH / 2) + 16 * kk + 8 * half);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float x = (float)qf[kk][e], y = (float)qf[kk + NK / 2][e], c = (float)cv[e], sn = (float)sv[e];
                    qf[kk][e] = (__bf16)(x * c - y * sn);
                    qf[kk + NK / 2][e] = (__bf16)(y * c + x * sn);
                }
            }
        }
    }
    f32x16_v acc_o[ND];
#pragma unroll
    for (int db = 0; db < ND; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc_o[db][v] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    // native vectors and unconditional loads (the chunk index is clamped instead): with HIP's uint4 struct and a
    // guarded load the compiler keeps these in scratch memory and waits for every load right where it is issued
    typedef uint32_t u32x4_s __attribute__((ext_vector_type(4)));
    u32x4_s kreg[CPT], vreg[CPT], kother[FILL ? CPT : 1], kcos[FILL ? CPT : 1], ksin[FILL ? CPT : 1];
    auto gload = [&](int t) {
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            const int c = min(tid + TPG * j, CH - 1);
            const int r = c / (DH / 8), ch = c % (DH / 8);
            const int64_t key = min(t * KT + r, T - 1);
            kreg[j] = *reinterpret_cast<const u32x4_s*>(kp + key * kpitch + ch * 8);
            vreg[j] = *reinterpret_cast<const u32x4_s*>(vp + key * kpitch + ch * 8);
            if (FILL && kv.cos) {
                const int first = ch % (DH / 16);
                kother[FILL ? j : 0] = *reinterpret_cast<const u32x4_s*>(kp + key * kpitch + (ch < DH / 16 ? ch + DH / 16 : first) * 8);
                kcos[FILL ? j : 0] = *reinterpret_cast<const u32x4_s*>(kv.cos + key * (DH / 2) + first * 8);
                ksin[FILL ? j : 0] = *reinterpret_cast<const u32x4_s*>(kv.sin + key * (DH / 2) + first * 8);
            }
        }
    };
    auto lwrite = [&](int buf, int t) {
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            const int c = tid + TPG * j;
            if (CH % TPG == 0 || c < CH) {
                const int r = c / (DH / 8), ch = c % (DH / 8);
                if (FILL) {
                    if (kv.cos) kreg[j] = rotated_chunk<bf16_t>(kreg[j], kother[FILL ? j : 0], kcos[FILL ? j : 0], ksin[FILL ? j : 0], ch >= DH / 16);
                    if (zg == 0 && t * KT + r < T) {
                        *reinterpret_cast<u32x4_s*>(kout + (int64_t)(t * KT + r) * DH + ch * 8) = kreg[j];
                        *reinterpret_cast<u32x4_s*>(vout + (int64_t)(t * KT + r) * DH + ch * 8) = vreg[j];
                    }
                }
                *reinterpret_cast<u32x4_s*>(&ksm[buf][r * KS + ch * 8]) = kreg[j];
                *reinterpret_cast<u32x4_s*>(&vsm[buf][r * VS + ch * 8]) = vreg[j];
            }
        }
    };

    // group kg visits tiles kg, kg + KG, ...; the step count is uniform over the workgroup (barriers)
    const int nsteps = (ntiles + KG - 1) / KG;
    if (kg < ntiles) { gload(kg); lwrite(0, kg); }
    // The Q fragments are used here, once, so that they have arrived on EVERY path into the step loop.  A workgroup whose
    // group has no first tile skips the wait above; the compiler then assumes the eight Q loads may still be in flight at
    // the loop's head and puts `s_waitcnt vmcnt(7) .. vmcnt(0)` in front of the eight score MFMAs of every step, which in
    // steady state wait for the tile requested at the top of that same step (37.1 -> 34.5 us per layer at 1024 tokens).
    // Two tiles in flight instead of one (a second register set, roles swapped from step to step) gained nothing more.
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) asm volatile("" : : "v"(qf[kk]));
    __syncthreads();
    for (int st = 0; st < nsteps; ++st) {
        const int buf = st & 1;
        const int t = st * KG + kg;
        if (t + KG < ntiles) gload(t + KG);
        if (t < my_tiles) {
            // scores, transposed: rows = keys of the tile, column = this lane's query
            f32x16_v sc;
#pragma unroll
            for (int v = 0; v < 16; ++v) sc[v] = 0.f;
#pragma unroll
            for (int kk = 0; kk < NK; ++kk) {
                const bf16x8_v kf = *reinterpret_cast<const bf16x8_v*>(&ksm[buf][col * KS + 16 * kk + 8 * half]);
                sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[kk], sc, 0, 0, 0);
            }
            const int qrow = q0 + col;
            const int kbase = t * KT + 4 * half;
            // raw scores: the (positive) scale is applied inside the exponent's fma; only a tile that reaches past the
            // wave's first row holds keys to mask
            if (t * KT + KT - 1 > q0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int key = kbase + 8 * (v >> 2) + (v & 3);
                    if (key > qrow) sc[v] = -INFINITY;
                }
            }
            float mx = -INFINITY;
#pragma unroll
            for (int v = 0; v < 16; ++v) mx = fmaxf(mx, sc[v]);
            mx = half_max(mx) * scale_log2e;
            // The reference point of the exponentials follows the running maximum lazily: it moves only when the
            // maximum has grown by more than 2^8 (probabilities then reach 2^8 at most, harmless in bf16 / f32, and
            // the quotient O / l does not depend on the reference point).  Most tiles therefore leave O^T unscaled,
            // and a wave skips the 64 multiplies (the accumulators live in AGPRs: 128 more moves) unless a lane moved.
            const bool move = mx > m_run + 8.0f;    // first tile: m_run = -inf, key 0 is visible to every query
            const float m_new = move ? mx : m_run;
            const float corr = move ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
            float ls = 0.f;
            bf16x8_v pb[2];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[v], scale_log2e, -m_new));
                ls += pv;
                pb[v >> 3][v & 7] = (__bf16)pv;
            }
            ls = half_sum(ls);
            l_run = l_run * corr + ls;
            m_run = m_new;
            if (__builtin_amdgcn_ballot_w64(move) != 0) {
#pragma unroll
                for (int db = 0; db < ND; ++db)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc_o[db][v] *= corr;
            }
#pragma unroll
            for (int db = 0; db < ND; ++db) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const bf16x8_v vf = v_fragment(&vsm[buf][16 * i * VS + db * 32], VS, lane);
                    acc_o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pb[i], acc_o[db], 0, 0, 0);
                }
            }
        }
        if (t + KG < ntiles) lwrite(buf ^ 1, t + KG);
        __syncthreads();
    }
    if (KG == 2) {
        // merge the two groups' states: O = O0 c0 + O1 c1, l = l0 c0 + l1 c1 with c_g = 2^(m_g - max(m0, m1)); a group
        // that saw no tile has m = -inf, l = 0, O = 0 and drops out.  The tiles in LDS are dead (the loop ended on a
        // barrier); the exchange area is 66 floats per lane of the second group.
        float* xch = reinterpret_cast<float*>(smem) + (wave * 64 + lane);
        static_assert(KG != 2 || (ND * 16 + 2) * 256 * 4 <= (int)sizeof(smem), "exchange area fits the tiles");
        if (kg == 1) {
#pragma unroll
            for (int db = 0; db < ND; ++db)
#pragma unroll
                for (int v = 0; v < 16; ++v) xch[(db * 16 + v) * 256] = acc_o[db][v];
            xch[(ND * 16) * 256] = m_run;
            xch[(ND * 16 + 1) * 256] = l_run;
        }
        __syncthreads();
        if (kg == 1) return;
        const float m1 = xch[(ND * 16) * 256], l1 = xch[(ND * 16 + 1) * 256];
        const float mm = fmaxf(m_run, m1);
        const float c0 = __builtin_amdgcn_exp2f(m_run - mm), c1 = __builtin_amdgcn_exp2f(m1 - mm);
        l_run = l_run * c0 + l1 * c1;
#pragma unroll
        for (int db = 0; db < ND; ++db)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc_o[db][v] = acc_o[db][v] * c0 + xch[(db * 16 + v) * 256] * c1;
    }
    if (KG == 4) {
        // four states, likewise; group g finishes the 32 d of block g, so every wave writes and reads as much
        constexpr int SLOTS = ND * 16 + 2;
        static_assert(KG != 4 || (SLOTS * KG * TPG * 4 <= (int)sizeof(smem) && ND <= KG), "exchange area fits the tiles");
        float* xch = reinterpret_cast<float*>(smem) + wave * 64 + lane;
        auto at_slot = [&](int g, int slot) -> float& { return xch[(g * SLOTS + slot) * TPG]; };
#pragma unroll
        for (int db = 0; db < ND; ++db)
            if (db != kg) {
#pragma unroll
                for (int v = 0; v < 16; ++v) at_slot(kg, db * 16 + v) = acc_o[db][v];
            }
        at_slot(kg, ND * 16) = m_run;
        at_slot(kg, ND * 16 + 1) = l_run;
        __syncthreads();
        float mm = m_run, c[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) mm = fmaxf(mm, at_slot(g, ND * 16));
        const float own = __builtin_amdgcn_exp2f(m_run - mm);
        l_run = 0.f;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            c[g] = __builtin_amdgcn_exp2f(at_slot(g, ND * 16) - mm);
            l_run += at_slot(g, ND * 16 + 1) * c[g];
        }
#pragma unroll
        for (int db = 0; db < ND; ++db)
            if (db == kg) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    float o = acc_o[db][v] * own;
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        if (g != db) o = __builtin_fmaf(at_slot(g, db * 16 + v), c[g], o);
                    acc_o[db][v] = o;
                }
            }
    }
    if (active && q0 + col < T) {
        const float inv = 1.0f / l_run;
        bf16_t* op = ctx + (int64_t)(q0 + col) * n_q * DH + (int64_t)head * DH;
#pragma unroll
        for (int db = 0; db < ND; ++db) {
            if (KG == 4 && db != kg) continue;
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int d = db * 32 + 8 * g4 + 4 * half;
                const uint32_t lo = pack_bf16x2(acc_o[db][4 * g4 + 0] * inv, acc_o[db][4 * g4 + 1] * inv);
                const uint32_t hi = pack_bf16x2(acc_o[db][4 * g4 + 2] * inv, acc_o[db][4 * g4 + 3] * inv);
                *reinterpret_cast<uint2*>(op + d) = make_uint2(lo, hi);
            }
        }
    }
}

// The same kernel in f32 on v_mfma_f32_32x32x2_f32: a 16-byte fragment holds 4 consecutive d (scores) or 4 consecutive
// keys (P.V), each fragment feeds four K = 2 products, and the probabilities stay f32.  V^T sits in LDS in plain key
// order: the keys a lane holds of its query in score registers 4 i .. 4 i + 3 are 8 i + 4 (lane / 32) + 0..3, exactly
// what fragment i of the second product covers.
typedef float f32x4_v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x16_v mma_f32x4(const f32x4_v& a, const f32x4_v& b, f32x16_v c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], c, 0, 0, 0);
    return c;
}

template <int DH, bool FILL>
__global__ __launch_bounds__(256, 2) void attn_prefill_mfma_f32_kernel(const float* __restrict__ qkv, float* __restrict__ ctx, int T,
                                                                    int n_q, int n_kv, float scale_log2e, int zgroups, PrefillKv<float> kv) {
    constexpr int KT = 32;            // keys per tile
    constexpr int KS = DH + 4;        // K tile row stride in elements (16 bytes of padding)
    // V^T row stride in elements; row d starts 4 * ((d / 4) % 8) elements in, which spreads the lanes that scatter one
    // key's d-chunks over the banks (as in the bf16 kernel)
    constexpr int VS = KT + 4 + 28;
    constexpr int ND = DH / 32;       // 32-row blocks of d in O^T
    constexpr int NK = DH / 8;        // k-steps of the score product (8 d each)
    constexpr int CH = KT * DH / 4;   // 16-byte chunks of a K (or V) tile
    constexpr int CPT = (CH + 255) / 256;
    __shared__ __align__(16) float ksm[2][KT * KS];
    __shared__ __align__(16) float vsm[2][DH * VS];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, half = lane >> 5;
    const int G = n_q / n_kv;
    const int gw = G >= 4 ? 4 : G;
    const int rtpb = 4 / gw;
    const XcdTile at = xcd_tile();
    const int kvh = at.y;
    const int seq = at.z / zgroups, zg = at.z % zgroups;
    const int bx = gridDim.x - 1 - at.x;     // rows that see many keys first: the last workgroups to start are the short ones
    const int head = kvh * G + zg * gw + wave % gw;
    const int q0 = (bx * rtpb + wave / gw) * 32;
    const int64_t P = (int64_t)(n_q + 2 * n_kv) * DH;
    qkv += (int64_t)seq * T * P;
    ctx += (int64_t)seq * T * n_q * DH;
    int64_t kpitch;
    const auto* kp = prefill_rows(kv.k, kv, qkv, seq, kvh, DH, T, P, (int64_t)(n_q + kvh) * DH, kpitch);
    const auto* vp = prefill_rows(kv.v, kv, qkv, seq, kvh, DH, T, P, (int64_t)(n_q + n_kv + kvh) * DH, kpitch);
    float *kout = const_cast<float*>(kp), *vout = const_cast<float*>(vp);   // FILL: the caches' rows
    if (FILL) { kp = qkv + (int64_t)(n_q + kvh) * DH; vp = qkv + (int64_t)(n_q + n_kv + kvh) * DH; kpitch = P; }
    const int kend = min(T, (bx * rtpb + rtpb) * 32);
    const int ntiles = (kend + KT - 1) / KT;
    const bool active = q0 < T;
    const int my_tiles = active ? min(ntiles, (q0 + 31) / KT + 1) : 0;

    f32x4_v qf[NK];
    {
        const int row = min(q0 + col, T - 1);
        const float* qp = qkv + (int64_t)row * P + (int64_t)head * DH + 4 * half;
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) qf[kk] = *reinterpret_cast<const f32x4_v*>(qp + 8 * kk);
        if (kv.cos) {   // see the bf16 kernel
#pragma unroll
            for (int kk = 0; kk < NK / 2; ++kk) {
                const f32x4_v cv = *reinterpret_cast<const f32x4_v*>(kv.cos + (int64_t)row * (DH / 2) + 8 * kk + 4 * half);
                const f32x4_v sv = *reinterpret_cast<const f32x4_v*>(kv.sin + (int64_t)row * (DH / 2) + 8 * kk + 4 * half);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x = qf[kk][e], y = qf[kk + NK / 2][e];
                    qf[kk][e] = x * cv[e] - y * sv[e];
                    qf[kk + NK / 2][e] = y * cv[e] + x * sv[e];
                }
            }
        }
    }
    f32x16_v acc_o[ND];
#pragma unroll
    for (int db = 0; db < ND; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc_o[db][v] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    f32x4_v kreg[CPT], vreg[CPT], kother[FILL ? CPT : 1], kcos[FILL ? CPT : 1], ksin[FILL ? CPT : 1];
    auto gload = [&](int t) {
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            const int c = min(tid + 256 * j, CH - 1);   // unconditional loads: see the bf16 kernel
            const int r = c / (DH / 4), ch = c % (DH / 4);
            const int64_t key = min(t * KT + r, T - 1);
            kreg[j] = *reinterpret_cast<const f32x4_v*>(kp + key * kpitch + ch * 4);
            vreg[j] = *reinterpret_cast<const f32x4_v*>(vp + key * kpitch + ch * 4);
            if (FILL && kv.cos) {
                const int first = ch % (DH / 8);
                kother[FILL ? j : 0] = *reinterpret_cast<const f32x4_v*>(kp + key * kpitch + (ch < DH / 8 ? ch + DH / 8 : first) * 4);
                kcos[FILL ? j : 0] = *reinterpret_cast<const f32x4_v*>(kv.cos + key * (DH / 2) + first * 4);
                ksin[FILL ? j : 0] = *reinterpret_cast<const f32x4_v*>(kv.sin + key * (DH / 2) + first * 4);
            }
        }
    };
    auto lwrite = [&](int buf, int t) {
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            const int c = tid + 256 * j;
            if (CH % 256 == 0 || c < CH) {
                const int r = c / (DH / 4), ch = c % (DH / 4);
                if (FILL) {
                    if (kv.cos) kreg[j] = rotated_chunk<float>(kreg[j], kother[FILL ? j : 0], kcos[FILL ? j : 0], ksin[FILL ? j : 0], ch >= DH / 8);
                    if (zg == 0 && t * KT + r < T) {
                        *reinterpret_cast<f32x4_v*>(kout + (int64_t)(t * KT + r) * DH + ch * 4) = kreg[j];
                        *reinterpret_cast<f32x4_v*>(vout + (int64_t)(t * KT + r) * DH + ch * 4) = vreg[j];
                    }
                }
                *reinterpret_cast<f32x4_v*>(&ksm[buf][r * KS + ch * 4]) = kreg[j];
#pragma unroll
                for (int e = 0; e < 4; ++e) vsm[buf][(ch * 4 + e) * VS + 4 * (ch & 7) + r] = vreg[j][e];
            }
        }
    };

    gload(0);
    lwrite(0, 0);
    // the Q fragments have arrived before the step loop on every path (see attn_prefill_mfma_kernel)
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) asm volatile("" : : "v"(qf[kk]));
    __syncthreads();
    for (int t = 0; t < ntiles; ++t) {
        const int buf = t & 1;
        if (t + 1 < ntiles) gload(t + 1);
        if (t < my_tiles) {
            f32x16_v sc;
#pragma unroll
            for (int v = 0; v < 16; ++v) sc[v] = 0.f;
#pragma unroll
            for (int kk = 0; kk < NK; ++kk) {
                const f32x4_v kf = *reinterpret_cast<const f32x4_v*>(&ksm[buf][col * KS + 8 * kk + 4 * half]);
                sc = mma_f32x4(kf, qf[kk], sc);
            }
            const int qrow = q0 + col;
            const int kbase = t * KT + 4 * half;
            if (t * KT + KT - 1 > q0) {   // only a tile that reaches past the wave's first row holds keys to mask
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int key = kbase + 8 * (v >> 2) + (v & 3);
                    if (key > qrow) sc[v] = -INFINITY;
                }
            }
            float mx = -INFINITY;
#pragma unroll
            for (int v = 0; v < 16; ++v) mx = fmaxf(mx, sc[v]);
            mx = half_max(mx) * scale_log2e;
            // lazy reference point and wave-wide skip of the rescaling, as in the bf16 kernel
            const bool move = mx > m_run + 8.0f;
            const float m_new = move ? mx : m_run;
            const float corr = move ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
            float ls = 0.f;
            f32x4_v pf[4];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[v], scale_log2e, -m_new));
                ls += pv;
                pf[v >> 2][v & 3] = pv;
            }
            ls = half_sum(ls);
            l_run = l_run * corr + ls;
            m_run = m_new;
            if (__builtin_amdgcn_ballot_w64(move) != 0) {
#pragma unroll
                for (int db = 0; db < ND; ++db)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc_o[db][v] *= corr;
            }
#pragma unroll
            for (int db = 0; db < ND; ++db) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x4_v vf = *reinterpret_cast<const f32x4_v*>(&vsm[buf][(db * 32 + col) * VS + 4 * ((col >> 2) & 7) + 8 * i + 4 * half]);
                    acc_o[db] = mma_f32x4(vf, pf[i], acc_o[db]);
                }
            }
        }
        if (t + 1 < ntiles) lwrite(buf ^ 1, t + 1);
        __syncthreads();
    }
    if (active && q0 + col < T) {
        const float inv = 1.0f / l_run;
        float* op = ctx + (int64_t)(q0 + col) * n_q * DH + (int64_t)head * DH;
#pragma unroll
        for (int db = 0; db < ND; ++db)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int d = db * 32 + 8 * g4 + 4 * half;
                *reinterpret_cast<float4*>(op + d) = make_float4(acc_o[db][4 * g4] * inv, acc_o[db][4 * g4 + 1] * inv,
                                                                 acc_o[db][4 * g4 + 2] * inv, acc_o[db][4 * g4 + 3] * inv);
            }
    }
}

// Prompts of at most 16 f32 rows without rotation: a workgroup a query head and sequence, a wave a row.  All that a wave reads it asks for at once: lane 4 j + p a
// quarter of key j and the same quarter of its query (scores are sums over four lanes), lane d dim d (and d + 64) of every value.  No LDS, no barrier, no matrix
// instruction's 32 x 32 of which 7 rows use a twentieth: bound by its one trip to memory and the launch.  The workgroup of a kv head's first query
// head puts the rows into the caches.  7 rows, 12 heads of 64: 6.6 -> 4.2 us.
constexpr int kShortRows = 16;
template <typename F> __device__ __forceinline__ float quarter_pair(float v, F f) {   // lanes l, l ^ 16, l ^ 32, l ^ 48
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
template <int DH>
__global__ __launch_bounds__(64 * kShortRows) void attn_short_f32_kernel(const float* __restrict__ qkv, float* __restrict__ ctx, int T, int n_q, int n_kv, float scale_log2e,
                                                                         PrefillKv<float> kv) {
    constexpr int QD = DH / 4, ND = DH / 64;
    const int lane = threadIdx.x & 63, row = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int head = blockIdx.x, seq = blockIdx.y, G = n_q / n_kv, kvh = head / G;
    const int64_t P = (int64_t)(n_q + 2 * n_kv) * DH;
    const float* rows = qkv + (int64_t)seq * T * P;
    const float* kp = rows + (int64_t)(n_q + kvh) * DH;
    const float* vp = rows + (int64_t)(n_q + n_kv + kvh) * DH;
    const int j = lane >> 2, part = (lane & 3) * QD;
    f32x4_v q[QD / 4], k[QD / 4];
    float v[kShortRows][ND];
#pragma unroll
    for (int i = 0; i < QD / 4; ++i) {
        q[i] = *reinterpret_cast<const f32x4_v*>(rows + (int64_t)row * P + (int64_t)head * DH + part + 4 * i);
        k[i] = *reinterpret_cast<const f32x4_v*>(kp + (int64_t)min(j, row) * P + part + 4 * i);
    }
#pragma unroll
    for (int t = 0; t < kShortRows; ++t)
        if (t <= row)
#pragma unroll
            for (int e = 0; e < ND; ++e) v[t][e] = vp[(int64_t)t * P + 64 * e + lane];
    const bool fill = kv.starts && head % G == 0;
    float kc[ND], vc[ND];
    if (fill)
#pragma unroll
        for (int e = 0; e < ND; ++e) { kc[e] = kp[(int64_t)row * P + 64 * e + lane]; vc[e] = vp[(int64_t)row * P + 64 * e + lane]; }
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int i = 0; i < QD / 4; ++i) {
        s0 = __builtin_fmaf(q[i].x, k[i].x, s0); s1 = __builtin_fmaf(q[i].y, k[i].y, s1);
        s0 = __builtin_fmaf(q[i].z, k[i].z, s0); s1 = __builtin_fmaf(q[i].w, k[i].w, s1);
    }
    float s = s0 + s1;
    s += dpp_move<0xB1>(s);    // quad_perm [1,0,3,2]
    s += dpp_move<0x4E>(s);    // quad_perm [2,3,0,1]
    s = j <= row ? s * scale_log2e : -INFINITY;
    float m = fmaxf(s, dpp_move<0x141>(s));   // row_half_mirror
    m = fmaxf(m, dpp_move<0x140>(m));         // row_mirror
    m = quarter_pair(m, [](float a, float b) { return fmaxf(a, b); });
    const float p = __builtin_amdgcn_exp2f(s - m);
    float l = p + dpp_move<0x141>(p);
    l += dpp_move<0x140>(l);
    l = quarter_pair(l, [](float a, float b) { return a + b; });
    float o[ND];
#pragma unroll
    for (int e = 0; e < ND; ++e) o[e] = 0.f;
#pragma unroll
    for (int t = 0; t < kShortRows; ++t)
        if (t <= row) {
            const float pt = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), 4 * t));
#pragma unroll
            for (int e = 0; e < ND; ++e) o[e] = __builtin_fmaf(pt, v[t][e], o[e]);
        }
    const float inv = 1.0f / l;
    float* out = ctx + ((int64_t)seq * T + row) * n_q * DH + (int64_t)head * DH;
#pragma unroll
    for (int e = 0; e < ND; ++e) out[64 * e + lane] = o[e] * inv;
    if (fill) {
        const int64_t at = (kvh * kv.capacity + min(max((int64_t)kv.starts[1], (int64_t)0), kv.capacity - T) + row) * DH;
#pragma unroll
        for (int e = 0; e < ND; ++e) {
            const_cast<float*>(kv.k[seq])[at + 64 * e + lane] = kc[e];
            const_cast<float*>(kv.v[seq])[at + 64 * e + lane] = vc[e];
        }
    }
}

static bool attn_prefill_mfma_ok(int dtype, int64_t n_q, int64_t n_kv, int64_t head_dim) {
    static const bool use_mfma = [] { const char* e = getenv("GPTRS_HIP_MFMA_ATTN"); return !(e && e[0] == '0'); }();
    if (!use_mfma || (dtype != 2 && dtype != 0) || n_kv <= 0 || n_q % n_kv != 0) return false;
    if (head_dim != 32 && head_dim != 64 && head_dim != 128) return false;
    const int64_t g = n_q / n_kv;
    return g == 1 || g == 2 || g % 4 == 0;
}
bool attn_prefill_batch_ok(int dtype, int64_t n_q, int64_t n_kv, int64_t head_dim, int64_t rot_half) {
    return attn_prefill_mfma_ok(dtype, n_q, n_kv, head_dim) && (rot_half == 0 || 2 * rot_half == head_dim);
}

template <typename T>
static int attn_prefill_mfma(hipStream_t s, const AttnPrefillArgs& a) {
    PrefillKv<T> kv{};
    for (int b = 0; b < a.batch && a.starts; ++b) { kv.k[b] = (const T*)a.k_caches[b]; kv.v[b] = (const T*)a.v_caches[b]; }
    kv.starts = a.starts;
    kv.capacity = a.capacity;
    if (a.rot_half) { kv.cos = (const T*)a.cos; kv.sin = (const T*)a.sin; }
    // four key groups (bf16) while the launch is one workgroup to a CU at most and rows see more than two tiles.  us, four and two groups (one, under 128
    // rows), 32 / 8 heads of 128: 100 rows 11.3 and 13.5, 128 11.2 and 13.8, 200 11.7 and 14.2, 333 13.6 and 17.1, 512 (256 workgroups) 16.9 and 21.6, 2 x 256
    // 13.7 and 17.1; beyond: 2 x 333 23.5 and 19.0, 1000 37 and 35; 64 rows 12 and 11.  Not where one group's launch is one row tile that fills the caches itself (a query
    // head to a key head, under 128 rows), which saves a launch: us with the rows into the caches, four groups and one, 12 heads of 64: 65 rows 8.0 and 6.6, 100 8.1 and 7.6, 127
    // 8.4 and 7.8; 16 heads of 128: 10.1 and 9.0, 10.7 and 10.5, 11.4 and 11.6; 4 heads of 32: 7.1 and 5.6, 7.2 and 6.4; 32 heads of 128: 10.7 and 9.9, 10.9 and 11.5
    static const bool allow_kg = [] { const char* e = getenv("GPTRS_HIP_ATTN_KEYGROUPS"); return !(e && e[0] == '0'); }();
    const int64_t g = a.n_q / a.n_kv;
    const bool kg4 = std::is_same<T, bf16_t>::value && allow_kg && a.t > 64 && !(a.starts && g == 1 && a.t < 128) && cdiv(cdiv(a.t, 32), g == 1 ? 2 : 1) * a.n_kv * (g == 1 ? 1 : g / 2) * a.batch <= 256;
    const int64_t hw = kg4 ? 2 : 4, gw = std::min(g, hw), zg = g / gw;   // waves of a key group; query heads of a workgroup, workgroups of a key head
    const dim3 grid((unsigned)cdiv(cdiv(a.t, 32), hw / gw), (unsigned)a.n_kv, (unsigned)(zg * a.batch));
    const float sl = a.scale * 1.44269504088896f;
    if constexpr (std::is_same<T, float>::value)
        if (a.t <= kShortRows && !kv.cos && (a.head_dim == 64 || a.head_dim == 128)) {
            const dim3 heads((unsigned)a.n_q, (unsigned)a.batch);
            const auto fn = a.head_dim == 64 ? attn_short_f32_kernel<64> : attn_short_f32_kernel<128>;
            fn<<<heads, 64 * (unsigned)a.t, 0, s>>>((const float*)a.qkv, (float*)a.ctx, (int)a.t, (int)a.n_q, (int)a.n_kv, sl, kv);
            return 1;
        }
    // two key groups per workgroup once the launch is smaller than three workgroups per CU and rows are long
    // enough to split (bf16)
    const bool kg2 = !kg4 && std::is_same<T, bf16_t>::value && allow_kg && a.t >= 128 && (int64_t)grid.x * grid.y * grid.z < 768;
    // one row tile: the attention fills the caches itself (us: 7 rows, 12 heads of 64 in f32 8.9 -> 6.4, 16 x 100 rows 22.7 -> 17.9; 20 rows, 32 / 8 heads of 128 in bf16 11.5 -> 9.4)
    const bool fill = a.starts && grid.x == 1 && !kg2 && !kg4;
    int launches = 1;
    if (a.starts && !fill) {
        const int64_t chunks = a.batch * a.t * 2 * a.n_kv * a.head_dim / (16 / (int64_t)sizeof(T));
        attn_prefill_kv_kernel<T><<<(unsigned)cdiv(chunks, 256), 256, 0, s>>>((const T*)a.qkv, chunks, (int)a.t, (int)a.n_q, (int)a.n_kv, (int)a.head_dim, kv);
        ++launches;
    }
    auto go = [&](auto dh) {
        constexpr int D = decltype(dh)::value;
        auto launch = [&](auto kernel, int threads) { kernel<<<grid, threads, 0, s>>>((const T*)a.qkv, (T*)a.ctx, (int)a.t, (int)a.n_q, (int)a.n_kv, sl, (int)zg, kv); };
        if constexpr (std::is_same<T, float>::value) {
            if (fill) launch(attn_prefill_mfma_f32_kernel<D, true>, 256);
            else launch(attn_prefill_mfma_f32_kernel<D, false>, 256);
        } else {
            if (kg4) launch(attn_prefill_mfma_kernel<D, 4, 2, false>, 512);
            else if (kg2) launch(attn_prefill_mfma_kernel<D, 2, 4, false>, 512);
            else if (fill) launch(attn_prefill_mfma_kernel<D, 1, 4, true>, 256);
            else launch(attn_prefill_mfma_kernel<D, 1, 4, false>, 256);
        }
    };
    if (a.head_dim == 32) go(std::integral_constant<int, 32>{});
    else if (a.head_dim == 64) go(std::integral_constant<int, 64>{});
    else go(std::integral_constant<int, 128>{});
    return launches;
}

int attn_prefill(hipStream_t s, const AttnPrefillArgs& a) {
    if (a.t <= 0) return 0;
    if (attn_prefill_mfma_ok(a.dtype, a.n_q, a.n_kv, a.head_dim) && a.t < (1ll << 30))
        return a.dtype == 0 ? attn_prefill_mfma<float>(s, a) : attn_prefill_mfma<bf16_t>(s, a);
    dim3 grid((unsigned)cdiv(a.t, 4), (unsigned)a.n_q);
    if (a.dtype == 0)
        attn_prefill_kernel<float><<<grid, 256, 0, s>>>((const float*)a.qkv, (float*)a.ctx, a.t, (int)a.n_q, (int)a.n_kv, (int)a.head_dim, a.scale);
    else
        attn_prefill_kernel<bf16_t><<<grid, 256, 0, s>>>((const bf16_t*)a.qkv, (bf16_t*)a.ctx, a.t, (int)a.n_q, (int)a.n_kv, (int)a.head_dim, a.scale);
    return 1;
}

// ------------------------------------------------------------------------------ attention over a growing cache
// k_all / v_all [n_kv, L, dh], L = C + T: positions < C from the caches, the rest from the K / V blocks of packed qkv
template <typename T>
__global__ __launch_bounds__(256) void attn_concat_kv_kernel(const T* __restrict__ qkv, const T* __restrict__ kc, const T* __restrict__ vc,
                                                             T* __restrict__ k_all, T* __restrict__ v_all, int64_t t, int64_t c,
                                                             int n_q, int n_kv, int dh) {
    const int64_t L = c + t, total = (int64_t)n_kv * L * dh;
    const int64_t P = (int64_t)(n_q + 2 * n_kv) * dh;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
        const int d = (int)(e % dh);
        const int64_t pos = (e / dh) % L;
        const int h = (int)(e / ((int64_t)dh * L));
        if (pos < c) {
            const int64_t src = ((int64_t)h * c + pos) * dh + d;
            k_all[e] = kc[src];
            v_all[e] = vc[src];
        } else {
            const int64_t row = (pos - c) * P + (int64_t)h * dh + d;
            k_all[e] = qkv[row + (int64_t)n_q * dh];
            v_all[e] = qkv[row + (int64_t)(n_q + n_kv) * dh];
        }
    }
}
// grid (ceil(T/4), n_q), 256 threads: one wave per query row, as attn_prefill_kernel, over keys 0 .. C + i of the
// combined caches
template <typename T>
__global__ __launch_bounds__(256) void attn_concat_kernel(const T* __restrict__ qkv, const T* __restrict__ k_all, const T* __restrict__ v_all,
                                                          T* __restrict__ ctx, int64_t t, int64_t c, int n_q, int n_kv, int dh, float scale) {
    __shared__ float qsm[4][256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t i = (int64_t)blockIdx.x * 4 + wave;
    const int h = blockIdx.y;
    const int kvh = h / (n_q / n_kv);
    const int64_t P = (int64_t)(n_q + 2 * n_kv) * dh, L = c + t;
    const T* kb = k_all + (int64_t)kvh * L * dh;
    const T* vb = v_all + (int64_t)kvh * L * dh;
    if (i < t)
        for (int d = lane; d < dh; d += 64) qsm[wave][d] = ldf(qkv, i * P + (int64_t)h * dh + d);
    __syncthreads();
    if (i >= t) return;
    const int64_t last = c + i;   // the row's own position
    float m = -INFINITY, l = 0.f;
    float o[4] = {0.f, 0.f, 0.f, 0.f};
    for (int64_t j0 = 0; j0 <= last; j0 += 64) {
        const int64_t j = j0 + lane;
        float s = -INFINITY;
        if (j <= last) {
            const T* kr = kb + j * dh;
            float acc = 0.f;
            for (int d = 0; d < dh; ++d) acc += qsm[wave][d] * ldf(kr, d);
            s = acc * scale;
        }
        const float mn = fmaxf(m, wave_max(s));
        const float corr = expf(m - mn);
        const float pe = j <= last ? expf(s - mn) : 0.f;
        l = l * corr + wave_sum(pe);
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) o[cc] *= corr;
        const int cnt = (int)((last - j0 + 1) < 64 ? (last - j0 + 1) : 64);
        for (int jj = 0; jj < cnt; ++jj) {
            const float pj = __shfl(pe, jj, 64);
            const T* vr = vb + (j0 + jj) * dh;
#pragma unroll
            for (int cc = 0; cc < 4; ++cc) {
                const int d = lane + 64 * cc;
                if (d < dh) o[cc] += pj * ldf(vr, d);
            }
        }
        m = mn;
    }
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) {
        const int d = lane + 64 * cc;
        if (d < dh) stf(ctx, i * (int64_t)n_q * dh + (int64_t)h * dh + d, o[cc] / l);
    }
}
template <typename T>
static void attn_concat_t(hipStream_t s, const AttnConcatArgs& a) {
    const int64_t total = a.n_kv * (a.cache_len + a.t) * a.head_dim;
    const unsigned g = (unsigned)std::min<int64_t>(cdiv(total, 256), 4096);
    attn_concat_kv_kernel<T><<<g, 256, 0, s>>>((const T*)a.qkv, (const T*)a.k_cache, (const T*)a.v_cache, (T*)a.k_all, (T*)a.v_all, a.t,
                                               a.cache_len, (int)a.n_q, (int)a.n_kv, (int)a.head_dim);
    dim3 grid((unsigned)cdiv(a.t, 4), (unsigned)a.n_q);
    attn_concat_kernel<T><<<grid, 256, 0, s>>>((const T*)a.qkv, (const T*)a.k_all, (const T*)a.v_all, (T*)a.ctx, a.t, a.cache_len,
                                               (int)a.n_q, (int)a.n_kv, (int)a.head_dim, a.scale);
}
void attn_concat(hipStream_t s, const AttnConcatArgs& a) {
    if (a.t <= 0) return;
    if (a.dtype == 0) attn_concat_t<float>(s, a);
    else attn_concat_t<bf16_t>(s, a);
}

}  // namespace k
}  // namespace gptrs
