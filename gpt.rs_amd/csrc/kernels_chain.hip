// Decode linear layers as ONE persistent launch per run of consecutive linears ("chain").
//
// A decode step of a transformer block is a dependent sequence of GEMVs (out-proj -> gate/up ->
// down -> next block's qkv ...), each streaming tens of MB of weights once.  Launched one by one,
// every GEMV pays a launch gap, a cold start and a tail; here the whole run executes inside one
// kernel of one workgroup per CU, phases separated by a grid-wide barrier:
//
//   * A layer's output columns, in tiles of 4, are dealt evenly over the workgroups, and a workgroup's words (tile by tile, k by
//     k; a word is 1 KiB, 16 bytes of each lane of a wave) evenly over its 8 compute waves, a run of consecutive words each:
//     every wave finishes a phase at the same time, whatever K and N are.
//   * The compute waves stream their words from HBM straight into LDS (global_load_lds_dwordx4: no registers), each wave into
//     a ring of its own, three words (a step) at a time, in the order they are consumed, phase by phase.  Weights do not
//     depend on activations, so a wave's requests run up to eight steps ahead of its reads across phase boundaries: while the
//     wave stands at the grid barrier or stages the next input, HBM keeps delivering the next phase's first words.  Loads of a
//     wave return in order, so "this step has landed" is a wait on the count of loads in flight: a ring private to the wave
//     needs no flags and no barrier.  The packed copy holds the words in the order of their
//     requests, step by step over all workgroups, so that what the whole chip asks for at one time is one run of memory: a
//     head of 805 MB streams at 6.0 TB/s, where a run of its own for every workgroup streamed at 5.1.  What a wave has
//     beyond the whole steps that all waves have (a step at most where tiles divide evenly) stands behind them.
//   * The compute lanes read their words from the ring and multiply them by the activation vector staged in LDS (v_dot2 for
//     bf16 pairs); at the end of a tile the wave leaves its part of the tile's 4 sums in LDS.
//   * 1 control wave per workgroup adds the parts of a phase's tiles when all waves are done, a lane to each output column,
//     applies the epilogue (SwiGLU pair, bias, GELU, residual), stores through to memory, and runs the grid
//     barrier (16 striped arrival counters, or counters of groups and notes between them; one poll instruction).
//   * Activations cross workgroups through agent-scope (sc1) loads and stores only, so no
//     L2 write-back / invalidate is needed between phases; a phase's input vector is staged into
//     LDS by the 9 compute and control waves together right after the barrier (RMSNorm statistics
//     included).
//   * Phase descriptors are read from the table in memory ahead of the wait that precedes their use (scalar
//     loads in the compute waves, one vector load with a lane per dword in the control wave), so a phase opens
//     the moment its barrier is seen.
//
// Decode attention (T = 1 over the KV cache) runs inside the same launch as two more phase kinds,
// executed by the 8 compute waves of a workgroup together: "partial" (one workgroup per kv head and
// position chunk: append this step's K/V row, online softmax over the chunk for the query heads
// of the group) and "combine" (one workgroup per query head merges the chunk records).
//
// Weight-only quantised linears stream the same 16-byte words with more k per word: int8 codes
// (4 columns x 4 k, stored biased by 128) and int4 codes (4 columns x 8 k, biased by 8, with one bf16
// scale per column and group of 128 k fetched beside the word).  Codes are converted with the
// unsigned-byte converts and accumulated in f32 against the bf16 activations (every product is
// exact); the bias is taken out per word (-128 or -8 times the sum of the word's activations), the
// per-column int8 scale is applied by the control wave.
//
// Every wait is bounded by wall-clock time: a barrier that does not complete raises the abort flag, every
// wave leaves the kernel, and the host reports an execution error.
#include <algorithm>
#include <climits>
#include <cstddef>
#include <cstdlib>
#include <type_traits>

#include "kernels.hpp"
#include "device_utils.hpp"

namespace gptrs {
namespace k {

namespace {

constexpr int NS = 512;          // compute threads
constexpr int NT = NS + 64;      // + control wave: the threads that stage inputs and run attention phases
constexpr int NWS = NS / 64;
constexpr int SW = 3;            // words of a step: what a wave requests and consumes at a time
constexpr int CW = 64;           // lanes, and 16-byte pieces, of a word
constexpr int NC = kChainCounters, NG = kChainGroups, LINE = kChainLine;
constexpr int EPI_MAX = 640;     // output columns of a workgroup, staged values among them: N <= 640 * grid (tiles that do not divide evenly: up to 4 fewer)
constexpr int MAXI = 8;          // 8-byte items per thread in the norm staging: K <= 4*MAXI*NT
constexpr int STEP_BYTES = SW * CW * 16;     // a step of a wave
constexpr int SLOT_BYTES = NWS * STEP_BYTES; // ... of a workgroup
// Steps a compute wave can hold in registers while it waits for a phase to open: bf16, and fewer in the int4 and int8 kernels, whose step arithmetic and staging hold more registers (one step
// more spills), and in f32, whose short phases lose more to a longer text than three parked steps give (GPT-2 call of 64 tokens, us: one 26690, two 27560, three 27720).
constexpr int PARK = 3, PARK_W8 = 2, PARK_W4 = 1, PARK_W32 = 1;
constexpr int RING_MIN = 4, RING_MAX = 5;    // steps a wave's ring holds (its requests run that far ahead of its reads): 5 where the staged activations leave room
// Steps a wave has in flight while it consumes a phase.  What is queued in a CU's memory pipeline stands in front of everything that
// comes later, the control wave's stores, its arrival and its polls of the barrier among it, and more than 48 KiB of a CU under way
// do not make HBM faster: long phases (the head) stream 134 us with two steps, 143 with three, 147 with five; phases of few steps
// are shorter with three (K = 9216, N = 3072: 10.7 us against 11.5), since the next phase's first steps are then under way.
// For the same reason a wave that waits for a phase to open asks for no more than three steps: a ring filled up to its last slot then (five) stood in
// front of the control wave's polls of that very barrier.  The slots that are left are asked for where nobody waits: one as the wave leaves its last
// sums, one when the phase's input has been staged.  157 phases of a 3B model and 61 of GPT-2 small, us, ring filled up in the wait and one step at the end up to
// three, then three in the wait, then with a step behind the staging, then with the ring's last slot at the end too: bf16 1613, 1601, 1559, 1554; int8 1178,
// 1130, 1102, 1102; f32 339, 330, 352, 327; int4 with the last two 1080, 1058.  A freed slot asked for ahead of its step's arithmetic: 1571, 1164, 343.
constexpr int FLIGHT = 3, FLIGHT_LONG = 2, LONG_WORDS = 10 * SW;
constexpr int LDS_BYTES = 160 * 1024;        // per workgroup on gfx950
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
// The thread index behind an opaque barrier: values derived from it are recomputed by the phase that uses them instead of
// being computed once per launch and held in registers (or spilled) across every other phase.
__device__ __forceinline__ int local_tid() { int t = (int)threadIdx.x; asm volatile("" : "+v"(t)); return t; }
template <typename T> __device__ __forceinline__ T* uni_ptr(T* p) {
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32));
    return (T*)(((unsigned long long)hi << 32) | lo);
}
// Pointers read out of the phase table are generic to the compiler; every access goes through an
// explicit global-address-space pointer so it becomes a global_* instruction.  (A flat access counts
// on the LDS counter too, and a wait for an LDS read would then also wait for every weight load in
// flight.)
#define GPTRS_GLOBAL __attribute__((address_space(1)))
#define GPTRS_LDS __attribute__((address_space(3)))
template <typename T> __device__ __forceinline__ const GPTRS_GLOBAL T* as_global(const T* p) { return (const GPTRS_GLOBAL T*)p; }
template <typename T> __device__ __forceinline__ GPTRS_GLOBAL T* as_global(T* p) { return (GPTRS_GLOBAL T*)p; }
template <typename T> __device__ __forceinline__ T gload(const T* p) { return *as_global(p); }   // scalar T
template <typename T> __device__ __forceinline__ void gstore(T* p, const T& v) { *as_global(p) = v; }
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ f32x2 f32_pair(unsigned long long v) { return f32x2{__uint_as_float((unsigned)v), __uint_as_float((unsigned)(v >> 32))}; }
__device__ __forceinline__ uint2 gload2(const void* p) { const u32x2 v = *(const GPTRS_GLOBAL u32x2*)p; return make_uint2(v.x, v.y); }
__device__ __forceinline__ uint4 gload4(const void* p) { const u32x4 v = *(const GPTRS_GLOBAL u32x4*)p; return make_uint4(v.x, v.y, v.z, v.w); }
__device__ __forceinline__ void gstore4(void* p, const uint4& v) { u32x4 w; w.x = v.x; w.y = v.y; w.z = v.z; w.w = v.w; *(GPTRS_GLOBAL u32x4*)p = w; }
// agent-scope accesses: coherent across the XCDs' L2s without cache maintenance
__device__ __forceinline__ unsigned long long cload8(const void* p) {
    return __hip_atomic_load(as_global((const unsigned long long*)p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned cload4(const void* p) {
    return __hip_atomic_load(as_global((const unsigned*)p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void cstore8(void* p, unsigned long long v) {
    __hip_atomic_store(as_global((unsigned long long*)p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void cstore4(void* p, unsigned v) {
    __hip_atomic_store(as_global((unsigned*)p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// bf16 rounding with the hardware converter (v_cvt_pk_bf16_f32, round to nearest even): the staging of a
// normalised row runs these on every wave of the workgroup at once, where each instruction counts three times
// on the SIMD that holds three waves
__device__ __forceinline__ unsigned pack_hw(float lo, float hi) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    f32x2_t f;
    f.x = lo; f.y = hi;
    return __builtin_bit_cast(unsigned, __builtin_convertvector(f, bf16x2));
}
__device__ __forceinline__ float rbf(float v) { return bf16lo(pack_hw(v, 0.f)); }
template <typename P> __device__ __forceinline__ int lds_ld(P p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
template <typename P> __device__ __forceinline__ void lds_st(P p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
#define GPTRS_LDS_RELEASE() __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local")
#define GPTRS_LDS_ACQUIRE() __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local")

struct alignas(16) Shared {
    float part[EPI_MAX / 2 + 2 * NWS][4];   // sums of a tile's 4 columns over a wave's words: tile t of the workgroup by wave w in row t + w (8 rows are read from a tile's first)
    float epi_bias[EPI_MAX];
    float epi_res[EPI_MAX];
    // int8: [0, EPI_MAX) scale of each owned output column (gate of a SwiGLU pair), [EPI_MAX, 2 EPI_MAX) the pair's
    // up column.  (int4 group scales are staged behind the activations, see stage_block.)
    float epi_s[2 * EPI_MAX];
    float ssq[32];   // per-wave sums of the norm statistics (LayerNorm takes two rounds: [0, 16) and [16, 32))
    int go, done, abort, pad;   // done: waves that have left their sums of a linear phase, counted over the launch
};

// The table of phases is read-only for the whole launch: reading it through the constant address space lets the
// compiler use scalar loads (uniform addresses), which do not queue behind a wave's vector memory traffic.
#define GPTRS_CONST __attribute__((address_space(4)))
typedef const GPTRS_CONST ChainPhase* PhaseTable;
static_assert(sizeof(Shared) + (size_t)kChainMaxXsWords * 4 + (size_t)RING_MIN * SLOT_BYTES <= (size_t)LDS_BYTES, "the largest launch fits a CU's LDS");
constexpr int kPhaseDwords = (int)(sizeof(ChainPhase) / 4);
static_assert(kPhaseDwords <= 64, "one lane of the control wave per dword of a phase descriptor");

// Workgroup barrier that waits for this wave's LDS traffic only: the weight loads in flight stay in flight.
__device__ __forceinline__ void wg_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
}

// Uniform copy (scalar registers) of the descriptor fields that the staging and the epilogue read.  The compute waves
// fill it with scalar loads from the table before they wait for the phase to open; the control wave reads the table with
// one vector load (a lane per dword) before it waits for the grid barrier and picks the fields out of the lanes.  Either
// way nothing is fetched between the barrier and the first use.
struct PhaseRegs {
    int K, N, C, tlo, trem, lds_bytes, flags, wfmt;
    float inv_n, eps, glu_limit, glu_alpha, glu_shift;   // (the last three: control wave only)
    const void *x, *gamma, *beta, *bias, *residual, *wscale, *wscale2, *colscale;
    void* y;
    const void *post_gain, *post_res;   // (kChainPostNorm, bf16 weights only)
    float post_mult, post_eps;
};
// (LN: phases of the launch's weight format may read LayerNorm offsets, POST: they may have a residual prologue; a register pair
// that nobody reads is not kept)
template <bool LN, bool POST>
__device__ __forceinline__ void regs_from_table(PhaseRegs& R, const GPTRS_CONST ChainPhase* D) {
    R.K = uni(D->K); R.N = uni(D->N); R.C = uni(D->C); R.tlo = uni(D->tlo); R.trem = uni(D->trem);
    R.lds_bytes = uni(D->lds_bytes); R.flags = uni(D->flags); R.wfmt = uni(D->wfmt);
    R.inv_n = __int_as_float(uni(__float_as_int(D->inv_n))); R.eps = __int_as_float(uni(__float_as_int(D->eps)));
    R.x = uni_ptr(D->x); R.gamma = uni_ptr(D->gamma); R.beta = LN ? uni_ptr(D->beta) : nullptr; R.bias = uni_ptr(D->bias); R.residual = uni_ptr(D->residual);
    R.wscale = uni_ptr(D->wscale); R.wscale2 = uni_ptr(D->wscale2); R.y = uni_ptr(D->y);
    if (POST) {
        R.post_gain = uni_ptr(D->post_gain); R.post_res = uni_ptr(D->post_res);
        R.post_mult = __int_as_float(uni(__float_as_int(D->post_mult))); R.post_eps = __int_as_float(uni(__float_as_int(D->post_eps)));
    }
}
#define GPTRS_PD_INT(field) __builtin_amdgcn_readlane(pd, (int)(offsetof(ChainPhase, field) / 4))
#define GPTRS_PD_PTR(field) ((const void*)(((unsigned long long)(unsigned)__builtin_amdgcn_readlane(pd, (int)(offsetof(ChainPhase, field) / 4) + 1) << 32) | \
                                          (unsigned)__builtin_amdgcn_readlane(pd, (int)(offsetof(ChainPhase, field) / 4))))
template <bool LN, bool POST>
__device__ __forceinline__ void regs_from_lanes(PhaseRegs& R, int pd) {   // pd: dword `lane` of the descriptor
    R.K = GPTRS_PD_INT(K); R.N = GPTRS_PD_INT(N); R.C = GPTRS_PD_INT(C); R.tlo = GPTRS_PD_INT(tlo); R.trem = GPTRS_PD_INT(trem);
    R.lds_bytes = GPTRS_PD_INT(lds_bytes); R.flags = GPTRS_PD_INT(flags); R.wfmt = GPTRS_PD_INT(wfmt);
    R.inv_n = __int_as_float(GPTRS_PD_INT(inv_n)); R.eps = __int_as_float(GPTRS_PD_INT(eps));
    R.x = GPTRS_PD_PTR(x); R.gamma = GPTRS_PD_PTR(gamma); R.beta = LN ? GPTRS_PD_PTR(beta) : nullptr; R.bias = GPTRS_PD_PTR(bias); R.residual = GPTRS_PD_PTR(residual);
    R.wscale = GPTRS_PD_PTR(wscale); R.wscale2 = GPTRS_PD_PTR(wscale2); R.y = const_cast<void*>(GPTRS_PD_PTR(y));
    R.colscale = GPTRS_PD_PTR(colscale); R.glu_limit = __int_as_float(GPTRS_PD_INT(glu_limit));
    R.glu_alpha = __int_as_float(GPTRS_PD_INT(glu_alpha)); R.glu_shift = __int_as_float(GPTRS_PD_INT(glu_shift));
    if (POST) {
        R.post_gain = GPTRS_PD_PTR(post_gain); R.post_res = GPTRS_PD_PTR(post_res);
        R.post_mult = __int_as_float(GPTRS_PD_INT(post_mult)); R.post_eps = __int_as_float(GPTRS_PD_INT(post_eps));
    }
}

// The tiles of a workgroup: the first `trem` workgroups take one more than `tlo`.
__host__ __device__ __forceinline__ int tile_first(int blk, int tlo, int trem) { return blk * tlo + (blk < trem ? blk : trem); }
__host__ __device__ __forceinline__ int tile_count(int blk, int tlo, int trem) { return tlo + (blk < trem ? 1 : 0); }
// The first of a wave's words among the W of its workgroup: words [wave_first(W, w), wave_first(W, w + 1)) are wave w's.
__host__ __device__ __forceinline__ int wave_first(int W, int w) { return (W * w) >> 3; }   // (W < 2^22)
static_assert(NWS == 8, "wave_first");
// A wave asks for a phase's words in two parts: the `whole` steps of three words that every wave of a workgroup with tiles has, which lie in the order in which the
// chip asks for them, [step][workgroup][wave][3], and its rest, a run of words; all workgroups' rests lie one behind the other from word `behind` on.
struct WavePart { int words, at, run, more; };   // words, place of the first, whether they are one run, words of the phase that follow them
__host__ __device__ __forceinline__ WavePart wave_part(int blk, int w, bool rest, int C, int tlo, int trem, int whole, int behind) {
    const int W = tile_count(blk, tlo, trem) * C, f0 = wave_first(W, w), words = wave_first(W, w + 1) - f0, at = SW * (NWS * blk + w), in_steps = words > 0 ? SW * whole : 0;
    const bool run = rest || whole == 0;
    // of a run: the words of the workgroups and waves before, less what they have in whole steps
    return WavePart{run ? words - in_steps : in_steps, run ? behind + tile_first(blk, tlo, trem) * C + f0 - whole * at : at, run, run ? 0 : words - in_steps};
}

// ---------------------------------------------------------------------------- staging (all waves)
// xs[j] = (x[2j], x[2j+1]) as a bf16 pair, zero beyond K; with norm: the value the stand-alone
// RMSNorm kernels store, ((x * inv_rms) * gamma) -> bf16 (normalization.rs:183-217).
// Returns 1 / rms of the sublayer's output where the phase has a residual prologue.
template <int FMT>
__device__ __forceinline__ float stage_block(const PhaseRegs& P, GPTRS_LDS unsigned* xs, GPTRS_LDS float* ssq) {
    const int t = local_tid(), lane = t & 63, wave = uni(t >> 6);
    const int K = P.K;
    const int n = K / 4;                     // 8-byte items holding data (K % 4 == 0)
    const int npad = P.lds_bytes >> 3;  // items to write: the words of every lane read zeros beyond K
    const char* x = (const char*)P.x;
    // int4: the group scales of this workgroup's tiles, one contiguous range of the tile-ordered copy
    // sc[tile][group][4] (bf16, 8 bytes per entry), go behind the activations; the first round of
    // loads is in flight while the activations are staged
    constexpr int SB = 8;
    int sc_n = 0;
    const uint2* sc_src = nullptr;
    GPTRS_LDS u32x2* sc_dst = (GPTRS_LDS u32x2*)(xs + 2 * npad);
    u32x2 sv[SB];
    if (FMT == kChainW4) {   // (every linear phase of a launch has the kernel's weight format)
        const int G = 4 * P.C;
        sc_n = tile_count(blockIdx.x, P.tlo, P.trem) * G;
        sc_src = (const uint2*)P.wscale + (long)tile_first(blockIdx.x, P.tlo, P.trem) * G;
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            const int i = u * NT + t;
            sv[u] = i < sc_n ? *(const GPTRS_GLOBAL u32x2*)(sc_src + i) : u32x2{0u, 0u};
        }
    }
    float post_inv = 0.f;
    if (FMT == kChainW16 && (P.flags & kChainPostNorm)) {
        // r = post_res + mult * rms_norm(x) * post_gain in f32, rounded to bf16 once; with kChainNorm the RMS norm of r instead
        constexpr int MF = MAXI / 2;
        f32x4 v[MF], rr[MF], gg[MF];
#pragma unroll
        for (int u = 0; u < MF; ++u) {
            const int i = u * NT + t;
            v[u] = f32x4{0.f, 0.f, 0.f, 0.f};
            rr[u] = v[u];
            gg[u] = v[u];
            if (u * NT < n && i < n) {
                const unsigned long long a = cload8(x + 16 * (size_t)i), b = cload8(x + 16 * (size_t)i + 8);
                const char* rp = (const char*)P.post_res + 16 * (size_t)i;
                const unsigned long long c = cload8(rp), d = cload8(rp + 8);
                v[u] = f32x4{__uint_as_float((unsigned)a), __uint_as_float((unsigned)(a >> 32)), __uint_as_float((unsigned)b), __uint_as_float((unsigned)(b >> 32))};
                rr[u] = f32x4{__uint_as_float((unsigned)c), __uint_as_float((unsigned)(c >> 32)), __uint_as_float((unsigned)d), __uint_as_float((unsigned)(d >> 32))};
                gg[u] = *(const GPTRS_GLOBAL f32x4*)((const char*)P.post_gain + 16 * (size_t)i);
            }
        }
        float q = 0.f;
#pragma unroll
        for (int u = 0; u < MF; ++u)
            if (u * NT < n) { q += v[u].x * v[u].x; q += v[u].y * v[u].y; q += v[u].z * v[u].z; q += v[u].w * v[u].w; }
        const float ws = wave_sum(q);
        if (lane == 0) ssq[wave] = ws;
        wg_barrier();
        float tot = 0.f;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) tot += ssq[w];
        post_inv = 1.0f / sqrtf(tot * P.inv_n + P.post_eps);
        const float mult = P.post_mult;
#pragma unroll
        for (int u = 0; u < MF; ++u) {   // (padding stays zero)
            rr[u].x += ((v[u].x * post_inv) * gg[u].x) * mult; rr[u].y += ((v[u].y * post_inv) * gg[u].y) * mult;
            rr[u].z += ((v[u].z * post_inv) * gg[u].z) * mult; rr[u].w += ((v[u].w * post_inv) * gg[u].w) * mult;
        }
        if (P.flags & kChainNorm) {
            float q2 = 0.f;
#pragma unroll
            for (int u = 0; u < MF; ++u) {
                const int i = u * NT + t;
                if (u * NT < n) {
                    q2 += rr[u].x * rr[u].x; q2 += rr[u].y * rr[u].y; q2 += rr[u].z * rr[u].z; q2 += rr[u].w * rr[u].w;
                    if (i < n) gg[u] = *(const GPTRS_GLOBAL f32x4*)((const char*)P.gamma + 16 * (size_t)i);
                }
            }
            const float w2 = wave_sum(q2);
            if (lane == 0) ssq[16 + wave] = w2;
            wg_barrier();
            float tot2 = 0.f;
#pragma unroll
            for (int w = 0; w < NT / 64; ++w) tot2 += ssq[16 + w];
            const float inv2 = 1.0f / sqrtf(tot2 * P.inv_n + P.eps);
#pragma unroll
            for (int u = 0; u < MF; ++u) {
                rr[u].x = (rr[u].x * inv2) * gg[u].x; rr[u].y = (rr[u].y * inv2) * gg[u].y;
                rr[u].z = (rr[u].z * inv2) * gg[u].z; rr[u].w = (rr[u].w * inv2) * gg[u].w;
            }
        }
#pragma unroll
        for (int u = 0; u < MF; ++u) {
            const int i = u * NT + t;
            if (u * NT < npad && i < npad) *(GPTRS_LDS u32x2*)&xs[2 * i] = u32x2{pack_hw(rr[u].x, rr[u].y), pack_hw(rr[u].z, rr[u].w)};
        }
    } else if (FMT == kChainW16 && (P.flags & (kChainNorm | kChainXF32 | kChainLayerNorm)) == (kChainNorm | kChainXF32 | kChainLayerNorm)) {
        // LayerNorm of an f32 row (f32 gains and offsets), rounded to bf16 once: mean, then the variance of the centred row
        constexpr int MF = MAXI / 2;
        f32x4 v[MF], gg[MF];
#pragma unroll
        for (int u = 0; u < MF; ++u) {
            const int i = u * NT + t;
            v[u] = f32x4{0.f, 0.f, 0.f, 0.f};
            gg[u] = v[u];
            if (u * NT < n && i < n) {
                const unsigned long long a = cload8(x + 16 * (size_t)i), b = cload8(x + 16 * (size_t)i + 8);
                v[u] = f32x4{__uint_as_float((unsigned)a), __uint_as_float((unsigned)(a >> 32)), __uint_as_float((unsigned)b), __uint_as_float((unsigned)(b >> 32))};
                gg[u] = *(const GPTRS_GLOBAL f32x4*)((const char*)P.gamma + 16 * (size_t)i);
            }
        }
        float s = 0.f;
#pragma unroll
        for (int u = 0; u < MF; ++u)
            if (u * NT < n) { s += v[u].x; s += v[u].y; s += v[u].z; s += v[u].w; }
        const float ws = wave_sum(s);
        if (lane == 0) ssq[wave] = ws;
        wg_barrier();
        float tot = 0.f;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) tot += ssq[w];
        const float mean = tot * P.inv_n;
        float q = 0.f;
#pragma unroll
        for (int u = 0; u < MF; ++u) {
            if (u * NT < n) {
                if (u * NT + t < n) { v[u].x -= mean; v[u].y -= mean; v[u].z -= mean; v[u].w -= mean; }   // (padding stays zero)
                q += v[u].x * v[u].x; q += v[u].y * v[u].y; q += v[u].z * v[u].z; q += v[u].w * v[u].w;
            }
        }
        const float wq = wave_sum(q);
        if (lane == 0) ssq[16 + wave] = wq;
        wg_barrier();
        float var = 0.f;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) var += ssq[16 + w];
        const float inv_std = 1.0f / sqrtf(var * P.inv_n + P.eps);
#pragma unroll
        for (int u = 0; u < MF; ++u) {
            const int i = u * NT + t;
            if (u * NT < npad && i < npad) {
                f32x4 bb = {0.f, 0.f, 0.f, 0.f};
                if (i < n) bb = *(const GPTRS_GLOBAL f32x4*)((const char*)P.beta + 16 * (size_t)i);
                const unsigned o0 = pack_hw((v[u].x * inv_std) * gg[u].x + bb.x, (v[u].y * inv_std) * gg[u].y + bb.y);
                const unsigned o1 = pack_hw((v[u].z * inv_std) * gg[u].z + bb.z, (v[u].w * inv_std) * gg[u].w + bb.w);
                *(GPTRS_LDS u32x2*)&xs[2 * i] = u32x2{o0, o1};
            }
        }
    } else if ((P.flags & (kChainNorm | kChainXF32)) == (kChainNorm | kChainXF32)) {
        // f32 row and gains (a bf16 model whose residual stream is f32): the f32 norm, rounded to bf16 once
        constexpr int MF = MAXI / 2;   // 16-byte items per thread: K <= 4 * MF * NT
        const char* g = (const char*)P.gamma;
        uint4 v[MF], gg[MF];
#pragma unroll
        for (int u = 0; u < MF; ++u) {
            const int i = u * NT + t;
            v[u] = make_uint4(0u, 0u, 0u, 0u);
            gg[u] = make_uint4(0u, 0u, 0u, 0u);
            if (u * NT < n && i < n) {
                const unsigned long long a = cload8(x + 16 * (size_t)i), b = cload8(x + 16 * (size_t)i + 8);
                v[u] = make_uint4((unsigned)a, (unsigned)(a >> 32), (unsigned)b, (unsigned)(b >> 32));
                gg[u] = gload4(g + 16 * (size_t)i);
            }
        }
        float q = 0.f;
#pragma unroll
        for (int u = 0; u < MF; ++u) {
            if (u * NT < n) {
                const float a = __uint_as_float(v[u].x), b = __uint_as_float(v[u].y), c = __uint_as_float(v[u].z), d = __uint_as_float(v[u].w);
                q += a * a; q += b * b; q += c * c; q += d * d;
            }
        }
        const float ws = wave_sum(q);
        if (lane == 0) ssq[wave] = ws;
        wg_barrier();
        float tot = 0.f;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) tot += ssq[w];
        const float inv = 1.0f / sqrtf(tot * P.inv_n + P.eps);
#pragma unroll
        for (int u = 0; u < MF; ++u) {
            const int i = u * NT + t;
            if (u * NT < npad && i < npad) {
                const unsigned o0 = pack_hw((__uint_as_float(v[u].x) * inv) * __uint_as_float(gg[u].x),
                                            (__uint_as_float(v[u].y) * inv) * __uint_as_float(gg[u].y));
                const unsigned o1 = pack_hw((__uint_as_float(v[u].z) * inv) * __uint_as_float(gg[u].z),
                                            (__uint_as_float(v[u].w) * inv) * __uint_as_float(gg[u].w));
                *(GPTRS_LDS u32x2*)&xs[2 * i] = u32x2{o0, o1};
            }
        }
    } else if (P.flags & kChainNorm) {
        const uint2* g = (const uint2*)P.gamma;
        unsigned long long v[MAXI];
        uint2 gg[MAXI];
#pragma unroll
        for (int u = 0; u < MAXI; ++u) {
            const int i = u * NT + t;
            v[u] = 0ull;
            gg[u] = make_uint2(0u, 0u);
            if (u * NT < n && i < n) {
                v[u] = cload8(x + 8 * (size_t)i);
                gg[u] = gload2(g + i);
            }
        }
        // rounds beyond the row (wave-uniform test) are skipped: a short row must not pay for MAXI of them
        float q = 0.f;
#pragma unroll
        for (int u = 0; u < MAXI; ++u) {
            if (u * NT < n) {
                const unsigned lo = (unsigned)v[u], hi = (unsigned)(v[u] >> 32);
                const float a = bf16lo(lo), b = bf16hi(lo), c = bf16lo(hi), d = bf16hi(hi);
                q += a * a; q += b * b; q += c * c; q += d * d;
            }
        }
        const float ws = wave_sum(q);
        if (lane == 0) ssq[wave] = ws;
        wg_barrier();
        float tot = 0.f;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) tot += ssq[w];
        const float inv = 1.0f / sqrtf(tot * P.inv_n + P.eps);
#pragma unroll
        for (int u = 0; u < MAXI; ++u) {
            const int i = u * NT + t;
            if (u * NT < npad && i < npad) {
                const unsigned lo = (unsigned)v[u], hi = (unsigned)(v[u] >> 32);
                // (x * inv) * gamma in f32, rounded to bf16 once: what the stand-alone RMSNorm kernels store
                const unsigned o0 = pack_hw((bf16lo(lo) * inv) * bf16lo(gg[u].x), (bf16hi(lo) * inv) * bf16hi(gg[u].x));
                const unsigned o1 = pack_hw((bf16lo(hi) * inv) * bf16lo(gg[u].y), (bf16hi(hi) * inv) * bf16hi(gg[u].y));
                *(GPTRS_LDS u32x2*)&xs[2 * i] = u32x2{o0, o1};
            }
        }
    } else {
        for (int i0 = 0; i0 < npad; i0 += MAXI * NT) {
            unsigned long long v[MAXI];
#pragma unroll
            for (int u = 0; u < MAXI; ++u) {
                const int i = i0 + u * NT + t;
                v[u] = i < n ? cload8(x + 8 * (size_t)i) : 0ull;
            }
#pragma unroll
            for (int u = 0; u < MAXI; ++u) {
                const int i = i0 + u * NT + t;
                if (i < npad) *(GPTRS_LDS u32x2*)&xs[2 * i] = u32x2{(unsigned)v[u], (unsigned)(v[u] >> 32)};
            }
        }
    }
    if (FMT == kChainW4 && sc_n > 0) {
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            const int i = u * NT + t;
            if (i < sc_n) sc_dst[i] = sv[u];
        }
        for (int i0 = SB * NT; i0 < sc_n; i0 += SB * NT) {
#pragma unroll
            for (int u = 0; u < SB; ++u) {
                const int i = i0 + u * NT + t;
                sv[u] = i < sc_n ? *(const GPTRS_GLOBAL u32x2*)(sc_src + i) : u32x2{0u, 0u};
            }
#pragma unroll
            for (int u = 0; u < SB; ++u) {
                const int i = i0 + u * NT + t;
                if (i < sc_n) sc_dst[i] = sv[u];
            }
        }
    }
    wg_barrier();
    return post_inv;
}


// f32 phases (kChainW32): xs[j] = x[j] as f32, zero beyond K; with norm: LayerNorm as the stand-alone kernel computes it,
// ((x - mean) * inv_std) * gamma + beta with the mean and the variance of the centred row taken in two rounds
// (normalization.rs:36-120).
__device__ __forceinline__ void stage_block_f32(const PhaseRegs& P, GPTRS_LDS unsigned* xs, GPTRS_LDS float* ssq) {
    const int t = local_tid(), lane = t & 63, wave = uni(t >> 6);
    const int n = P.K / 4;                // 16-byte items holding data (K % 4 == 0)
    const int npad = P.lds_bytes >> 4;    // items the readers see
    const char* x = (const char*)P.x;
    constexpr int MF = MAXI / 2;          // items per thread: K <= 4 * MF * NT
    const bool norm = P.flags & kChainNorm;
    if (norm && npad <= 64 * MF) {
        // A short row: each wave that writes a part of it (64 items) reads all of it and finds the mean and the variance by itself, without a word
        // between the waves.  GPT-2's 24 such phases of 768: 1.83 us of staging with two exchanges through LDS,
        // 1.34 so; 61 phases 306 and 292 us.
        if (wave * 64 < npad) {
            f32x4 v[MF], own = {0.f, 0.f, 0.f, 0.f}, gg = own, bb = own;
#pragma unroll
            for (int u = 0; u < MF; ++u) {
                const int i = u * 64 + lane;
                v[u] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (u * 64 < n && i < n) {
                    const unsigned long long a = cload8(x + 16 * (size_t)i), b = cload8(x + 16 * (size_t)i + 8);
                    v[u] = f32x4{__uint_as_float((unsigned)a), __uint_as_float((unsigned)(a >> 32)), __uint_as_float((unsigned)b), __uint_as_float((unsigned)(b >> 32))};
                }
            }
            const int mine = wave * 64 + lane;
            if (mine < n) {
                gg = *(const GPTRS_GLOBAL f32x4*)((const char*)P.gamma + 16 * (size_t)mine);
                bb = *(const GPTRS_GLOBAL f32x4*)((const char*)P.beta + 16 * (size_t)mine);
            }
            float s = 0.f;
#pragma unroll
            for (int u = 0; u < MF; ++u)
                if (u * 64 < n) s += (v[u].x + v[u].y) + (v[u].z + v[u].w);
            const float mean = wave_sum(s) * P.inv_n;
            float q = 0.f;
#pragma unroll
            for (int u = 0; u < MF; ++u) {
                if (u * 64 < n) {
                    f32x4 c = v[u] - mean;
                    if (u * 64 + lane >= n) c = f32x4{0.f, 0.f, 0.f, 0.f};
                    if (u == wave) own = c;
                    q += (c.x * c.x + c.y * c.y) + (c.z * c.z + c.w * c.w);
                }
            }
            const float inv_std = 1.0f / sqrtf(wave_sum(q) * P.inv_n + P.eps);
            own.x = (own.x * inv_std) * gg.x + bb.x; own.y = (own.y * inv_std) * gg.y + bb.y;
            own.z = (own.z * inv_std) * gg.z + bb.z; own.w = (own.w * inv_std) * gg.w + bb.w;
            if (mine < npad) *(GPTRS_LDS f32x4*)&xs[4 * mine] = mine < n ? own : f32x4{0.f, 0.f, 0.f, 0.f};
        }
        wg_barrier();
        return;
    }
    uint4 v[MF], gg[MF], bb[MF];
#pragma unroll
    for (int u = 0; u < MF; ++u) {
        const int i = u * NT + t;
        v[u] = make_uint4(0u, 0u, 0u, 0u);
        gg[u] = make_uint4(0u, 0u, 0u, 0u);
        bb[u] = make_uint4(0u, 0u, 0u, 0u);
        if (u * NT < n && i < n) {
            const unsigned long long a = cload8(x + 16 * (size_t)i), b = cload8(x + 16 * (size_t)i + 8);
            v[u] = make_uint4((unsigned)a, (unsigned)(a >> 32), (unsigned)b, (unsigned)(b >> 32));
            if (norm) {
                gg[u] = gload4((const char*)P.gamma + 16 * (size_t)i);
                bb[u] = gload4((const char*)P.beta + 16 * (size_t)i);
            }
        }
    }
    if (norm) {
        float s = 0.f;
#pragma unroll
        for (int u = 0; u < MF; ++u)
            if (u * NT < n) { s += __uint_as_float(v[u].x); s += __uint_as_float(v[u].y); s += __uint_as_float(v[u].z); s += __uint_as_float(v[u].w); }
        const float ws = wave_sum(s);
        if (lane == 0) ssq[wave] = ws;
        wg_barrier();
        float tot = 0.f;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) tot += ssq[w];
        const float mean = tot * P.inv_n;
        float c[MF][4];
        float q = 0.f;
#pragma unroll
        for (int u = 0; u < MF; ++u) {
            const bool in = u * NT < n && u * NT + t < n;
            c[u][0] = in ? __uint_as_float(v[u].x) - mean : 0.f;
            c[u][1] = in ? __uint_as_float(v[u].y) - mean : 0.f;
            c[u][2] = in ? __uint_as_float(v[u].z) - mean : 0.f;
            c[u][3] = in ? __uint_as_float(v[u].w) - mean : 0.f;
            q += c[u][0] * c[u][0]; q += c[u][1] * c[u][1]; q += c[u][2] * c[u][2]; q += c[u][3] * c[u][3];
        }
        const float wq = wave_sum(q);
        if (lane == 0) ssq[16 + wave] = wq;
        wg_barrier();
        float var = 0.f;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) var += ssq[16 + w];
        const float inv_std = 1.0f / sqrtf(var * P.inv_n + P.eps);
#pragma unroll
        for (int u = 0; u < MF; ++u) {
            v[u].x = __float_as_uint((c[u][0] * inv_std) * __uint_as_float(gg[u].x) + __uint_as_float(bb[u].x));
            v[u].y = __float_as_uint((c[u][1] * inv_std) * __uint_as_float(gg[u].y) + __uint_as_float(bb[u].y));
            v[u].z = __float_as_uint((c[u][2] * inv_std) * __uint_as_float(gg[u].z) + __uint_as_float(bb[u].z));
            v[u].w = __float_as_uint((c[u][3] * inv_std) * __uint_as_float(gg[u].w) + __uint_as_float(bb[u].w));
        }
    }
#pragma unroll
    for (int u = 0; u < MF; ++u) {
        const int i = u * NT + t;
        if (u * NT < npad && i < npad) *(GPTRS_LDS u32x4*)&xs[4 * i] = i < n ? u32x4{v[u].x, v[u].y, v[u].z, v[u].w} : u32x4{0u, 0u, 0u, 0u};
    }
    wg_barrier();
}

// ---------------------------------------------------------------------------- decode attention
__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }
// Waits inside the kernel are bounded by wall-clock time (wall_clock64 ticks at 100 MHz): the control wave's wait for the
// grid barrier by the launch's budget, the waits on it inside the workgroup by a multiple of that, so that the control
// wave is the one to give up and say why.
struct Patience {
    unsigned long long t0, ticks;
    unsigned spins;
    __device__ __forceinline__ Patience(unsigned long long budget) : t0(0), ticks(budget), spins(0) {}
    __device__ __forceinline__ bool spent() {   // call once per poll; reads the clock every 64th time
        if ((++spins & 63u) != 0) return false;
        const unsigned long long now = wall_clock64();
        if (t0 == 0) { t0 = now; return false; }
        return now - t0 > ticks;
    }
};
// compute waves wait here until the control wave has seen the grid barrier of `phase`
template <typename IP>
__device__ __forceinline__ bool wait_go(IP go, IP abort, int phase, unsigned long long budget) {
    Patience pat(8 * budget);
    while (uni(lds_ld(go)) < phase) {
        __builtin_amdgcn_s_sleep(1);
        if (uni(lds_ld(abort)) || pat.spent()) return false;
    }
    return true;
}

// exp through v_exp_f32 (2^x): softmax weights only, about one ulp, exp(-inf) = 0
__device__ __forceinline__ float fast_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896f); }
template <int CTRL> __device__ __forceinline__ float dpp(float v) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false)); }
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_HALF_MIRROR = 0x141, DPP_MIRROR = 0x140, DPP_ROR8 = 0x128;
// sums over the lpr (8, 16 or 32) consecutive lanes of a lane group, in each of them; N values at a time, so that one value's steps stand between another's
template <int N> __device__ __forceinline__ void group_sums(float (&v)[N], int lpr) {
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] += dpp<DPP_XOR1>(v[j]);
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] += dpp<DPP_XOR2>(v[j]);
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] += dpp<DPP_HALF_MIRROR>(v[j]);
    if (lpr >= 16) {
#pragma unroll
        for (int j = 0; j < N; ++j) v[j] += dpp<DPP_MIRROR>(v[j]);
    }
    if (lpr == 32) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const u32x2 sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[j]), __float_as_uint(v[j]), false, false);
            v[j] = __uint_as_float(sw.x) + __uint_as_float(sw.y);
        }
    }
}
// Two values of every lane, lane ^ 32 (16) exchanged: the lanes below keep a, those above b, each added up over the pair.
__device__ __forceinline__ float halves32(float a, float b) {
    const u32x2 sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(sw.x) + __uint_as_float(sw.y);
}
__device__ __forceinline__ float halves16(float a, float b) {
    const u32x2 sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(sw.x) + __uint_as_float(sw.y);
}
__device__ __forceinline__ float pair_max32(float a) {
    const u32x2 sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(a), false, false);
    return fmaxf(__uint_as_float(sw.x), __uint_as_float(sw.y));
}
__device__ __forceinline__ float pair_max16(float a) {
    const u32x2 sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(a), false, false);
    return fmaxf(__uint_as_float(sw.x), __uint_as_float(sw.y));
}

// What a maximum of nothing but hidden scores (-inf) is subtracted as: exp(-inf - 0) = 0, where exp(-inf + inf) is none.
__device__ __forceinline__ float finite_max(float m) { return m == -INFINITY ? 0.f : m; }

// Merge of the records (max m, sum l, N weighted values) of the N_REC waves w = first, first + step, ... of a head, left in LDS.
template <int N_REC>
__device__ __forceinline__ void merge_waves(const GPTRS_LDS float* sm, const GPTRS_LDS float* sl, const GPTRS_LDS float* so, int first, int step, int dh, int d,
                                            float& m, float& l, float& o) {
    float mm[N_REC], ll[N_REC], oo[N_REC];
#pragma unroll
    for (int u = 0; u < N_REC; ++u) { const int w = first + u * step; mm[u] = sm[w]; ll[u] = sl[w]; oo[u] = so[w * dh + d]; }
    m = mm[0];
#pragma unroll
    for (int u = 1; u < N_REC; ++u) m = fmaxf(m, mm[u]);
    const float ref = finite_max(m);
    l = 0.f; o = 0.f;
#pragma unroll
    for (int u = 0; u < N_REC; ++u) { const float c = fast_exp(mm[u] - ref); l += ll[u] * c; o += oo[u] * c; }
}

// The two phases are run by the 8 compute waves.  Nothing in them is long: a phase is a chain of latencies (the query row out of
// other workgroups' hands, scores, softmax, sums over lanes and waves, stores and their acknowledgement), so what counts is how
// many instructions stand behind one another between the barrier and the arrival.  With one online-softmax step for each row, a
// branch on the head's size in every exchange between lanes (1.6 us of two exchanges), 64-bit divisions and the control wave among the
// readers the two phases took, us: bf16 behind 1008 positions of 32 / 8 heads of 128 7.3 + 5.7, in the int8 kernel 7.4 + 4.8, f32 behind 80
// positions of 12 heads of 64 (one phase) 6.2.  With all rows of a lane in one step, one branch for each round of exchanges, and exchanges
// that leave each half of the lanes with half of the values 4.9 + 5.0, 4.6 + 3.9 and 3.3.
//
// unit = kv head * nch + chunk.  Each wave serves ONE query head of the kv head's group (wave w: head w % G, position subset
// w / G of 8 / G), so a lane carries a single softmax state; a cache row is read by head_dim / 8 lanes, 8 values each, and
// the waves of different heads re-read the same rows out of the caches.  Cache rows older than this launch, and the
// RoPE rows, are requested BEFORE the grid barrier is awaited (they do not depend on the previous phase); only the query
// row and this step's K/V row are read after it.
//
// Rows of the chunked design (ROWS == kRowsChunk): the projection's row is f32, queries and the new key are turned pair by pair (f32 angles), brought to unit
// mean square over the head and rounded to bf16 once, a value is rounded once; the caches hold the current chunk.
enum : int { kRowsBf16 = 0, kRowsF32 = 1, kRowsChunk = 2 };
template <int ROWS>
__device__ bool attn_partial(GPTRS_LDS int* go, GPTRS_LDS int* abort, const ChainPhase& P, GPTRS_LDS float* lds, int unit, int phase,
                             unsigned long long budget) {
    constexpr bool F32 = ROWS == kRowsF32, CHUNK = ROWS == kRowsChunk;
    typedef typename std::conditional<F32, float, bf16_t>::type E;       // of the caches
    typedef typename std::conditional<ROWS == kRowsBf16, bf16_t, float>::type X;   // of the projection's row
    constexpr int XW = ROWS == kRowsBf16 ? 1 : 2;                         // 16-byte words of a lane's 8 values there
    constexpr int PP = F32 ? 2 : 5;   // rows of a lane in one step; the first step's are requested ahead of the barrier (32 chunks x 8 lane groups x 5 = 1280 positions)
    constexpr int RW = F32 ? 2 : 1;   // 16-byte words of a lane's 8 values
    const int t = local_tid(), lane = t & 63, wave = uni(t >> 6);
    const int dh = P.head_dim, n_q = P.n_q, n_kv = P.n_kv, nch = P.nch, half = P.rot_half;
    const int G = n_q / n_kv, nparts = NWS / G, cap = P.capacity;   // G = 1, 2, 4 or 8
    const int lpr = dh >> 3, lsh = lpr == 8 ? 3 : lpr == 16 ? 4 : 5, sub = lane >> lsh, li = lane & (lpr - 1);
    const int g = wave & (G - 1), part = wave / G;
    const int stride = nparts * (64 >> lsh), sid = part * (64 >> lsh) + sub;   // position slots of this head's waves
    const int kvh = unit / nch, c = unit - kvh * nch;
    const X* qkv = (const X*)P.x;
    E* kc = (E*)P.k_cache + (long)kvh * cap * dh;
    E* vc = (E*)P.v_cache + (long)kvh * cap * dh;
    const bool rotate = ROWS == kRowsBf16 && P.cos != nullptr;
    int qpos = uni(gload(P.query_start));
    if (CHUNK) qpos = max(qpos, 0) % P.N;                                 // (N: positions of a chunk)
    qpos = clampi(qpos, 0, cap - 1);                                      // DynamicSlice clamp (cpu.rs:804-820)
    const int upd = clampi(uni(gload(P.update_starts + 1)), 0, cap - 1);  // DynamicUpdateSlice clamp
    const float scale = P.scale;
    const int L = qpos + 1, CL = (L + nch - 1) / nch;
    const int p0 = c * CL, p1 = min(L, p0 + CL);
    const bool owner = c == min(upd / CL, nch - 1);
    const int c0 = li * 8;
    u32x4 kraw[PP][RW], vraw[PP][RW];
    auto request_rows = [&](u32x4 (&raw)[PP][RW], const E* cache, int base) {
#pragma unroll
        for (int j = 0; j < PP; ++j) {
            const int p = base + sid + j * stride;
            const bool take = p < p1 && p != upd;
#pragma unroll
            for (int r = 0; r < RW; ++r) raw[j][r] = take ? *(const GPTRS_GLOBAL u32x4*)(cache + (long)p * dh + c0 + 4 * r) : u32x4{0u, 0u, 0u, 0u};
        }
    };
    auto row_values = [&](const u32x4 (&raw)[RW], float (&f)[8]) {
        const unsigned w[8] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w, raw[RW - 1].x, raw[RW - 1].y, raw[RW - 1].z, raw[RW - 1].w};
#pragma unroll
        for (int v = 0; v < 8; ++v) f[v] = F32 ? __uint_as_float(w[v]) : ((v & 1) ? bf16hi(w[v >> 1]) : bf16lo(w[v >> 1]));
    };
    // a row that the phase before has written: agent-scope loads
    auto request_new = [&](const X* p, u32x4 (&raw)[XW]) {
#pragma unroll
        for (int r = 0; r < XW; ++r) {
            const unsigned long long a = cload8(p + (XW == 2 ? 4 : 8) * r), b = cload8(p + (XW == 2 ? 4 : 8) * r + (XW == 2 ? 2 : 4));
            raw[r].x = (unsigned)a; raw[r].y = (unsigned)(a >> 32); raw[r].z = (unsigned)b; raw[r].w = (unsigned)(b >> 32);
        }
    };
    request_rows(kraw, kc, p0);
    request_rows(vraw, vc, p0);
    const bool rot = rotate && c0 < 2 * half, first = c0 < half;
    u32x4 cosr[1], sinr[1];
    const bool turn = CHUNK && c0 < 2 * half;
    if (turn) {   // the angles of a lane's four pairs: [rot / 2] cosines, as many sines
        cosr[0] = *(const GPTRS_GLOBAL u32x4*)((const float*)P.cos + (c0 >> 1));
        sinr[0] = *(const GPTRS_GLOBAL u32x4*)((const float*)P.cos + half + (c0 >> 1));
    }
    if (rot) {
        const int j0 = first ? c0 : c0 - half;
        cosr[0] = *(const GPTRS_GLOBAL u32x4*)((const bf16_t*)P.cos + j0);
        sinr[0] = *(const GPTRS_GLOBAL u32x4*)((const bf16_t*)P.sin + j0);
    }
    if (!wait_go(go, abort, phase, budget)) return false;

    // The wave's query head and, in the first position subset of the workgroup that owns position `upd`, this step's K and V rows
    // (for the first lane group), all requested before any is consumed; RoPE on the fly.
    const bool new_row = owner && part == 0;
    u32x4 qa[XW], qb[XW], ka[XW], kb[XW], va[XW];
    {
        const int co = first ? c0 + half : c0 - half;
        const X* head = qkv + (long)(kvh * G + g) * dh;
        const X* knew = qkv + (long)(n_q + kvh) * dh;
        request_new(head + c0, qa);
        if (rot) request_new(head + co, qb);
        if (new_row) {
            request_new(knew + c0, ka);
            if (rot) request_new(knew + co, kb);
            request_new(knew + (long)n_kv * dh + c0, va);
        }
    }
    auto new_values = [&](const u32x4 (&raw)[XW], float (&f)[8]) {
        const unsigned w[8] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w, raw[XW - 1].x, raw[XW - 1].y, raw[XW - 1].z, raw[XW - 1].w};
#pragma unroll
        for (int v = 0; v < 8; ++v) f[v] = XW == 2 ? __uint_as_float(w[v]) : ((v & 1) ? bf16hi(w[v >> 1]) : bf16lo(w[v >> 1]));
    };
    auto rope = [&](const u32x4 (&own_raw)[XW], const u32x4 (&other_raw)[XW], float (&out)[8]) {
        new_values(own_raw, out);
        if constexpr (CHUNK) {
            const unsigned cw[4] = {cosr[0].x, cosr[0].y, cosr[0].z, cosr[0].w}, sw[4] = {sinr[0].x, sinr[0].y, sinr[0].z, sinr[0].w};
            float q[1] = {0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float a = out[2 * i], b = out[2 * i + 1], cv = __uint_as_float(cw[i]), sv = __uint_as_float(sw[i]);
                if (turn) { out[2 * i] = a * cv - b * sv; out[2 * i + 1] = b * cv + a * sv; }
                q[0] += out[2 * i] * out[2 * i] + out[2 * i + 1] * out[2 * i + 1];
            }
            group_sums(q, lpr);
            const float inv = 1.0f / sqrtf(q[0] / (float)dh + P.eps);
#pragma unroll
            for (int v = 0; v < 8; ++v) out[v] = rbf(out[v] * inv);
        }
        if constexpr (ROWS == kRowsBf16) {
            if (rot) {
                float other[8], cosv[8], sinv[8];
                new_values(other_raw, other);
                new_values(cosr, cosv);
                new_values(sinr, sinv);
#pragma unroll
                for (int v = 0; v < 8; ++v) out[v] = rbf(first ? out[v] * cosv[v] - other[v] * sinv[v] : out[v] * cosv[v] + other[v] * sinv[v]);
            }
        }
    };
    float qf[8], m = -INFINITY, l = 0.f, o[8];
    rope(qa, qb, qf);
#pragma unroll
    for (int v = 0; v < 8; ++v) o[v] = 0.f;
    auto score = [&](const float (&kf)[8]) {
        float s = qf[0] * kf[0];
#pragma unroll
        for (int v = 1; v < 8; ++v) s = __builtin_fmaf(qf[v], kf[v], s);
        return s;
    };
    if (new_row) {   // this step's row: attended to when in range, appended once (by head 0's wave)
        float kf[8], vf[8], s[1];
        rope(ka, kb, kf);
        new_values(va, vf);
        if (CHUNK) {
#pragma unroll
            for (int v = 0; v < 8; ++v) vf[v] = rbf(vf[v]);
        }
        if (sub == 0 && g == 0) {
            E* kd = kc + (long)upd * dh + c0;
            E* vd = vc + (long)upd * dh + c0;
            if constexpr (F32) {
#pragma unroll
                for (int r = 0; r < RW; ++r) { *(GPTRS_GLOBAL u32x4*)(kd + 4 * r) = ka[r]; *(GPTRS_GLOBAL u32x4*)(vd + 4 * r) = va[r]; }
            } else {
                u32x4 kw;
                kw.x = pack_bf16x2(kf[0], kf[1]); kw.y = pack_bf16x2(kf[2], kf[3]); kw.z = pack_bf16x2(kf[4], kf[5]); kw.w = pack_bf16x2(kf[6], kf[7]);
                *(GPTRS_GLOBAL u32x4*)kd = kw;
                u32x4 vw = va[0];
                if constexpr (CHUNK) { vw.x = pack_hw(vf[0], vf[1]); vw.y = pack_hw(vf[2], vf[3]); vw.z = pack_hw(vf[4], vf[5]); vw.w = pack_hw(vf[6], vf[7]); }
                *(GPTRS_GLOBAL u32x4*)vd = vw;
            }
        }
        s[0] = score(kf);
        group_sums(s, lpr);
        if (sub == 0 && upd >= p0 && upd < p1) {
            m = s[0] * scale;
            l = 1.f;
#pragma unroll
            for (int v = 0; v < 8; ++v) o[v] = vf[v];
        }
    }
    for (int base = p0;;) {
        float s[PP], mn = m;
#pragma unroll
        for (int j = 0; j < PP; ++j) {
            float kf[8];
            row_values(kraw[j], kf);
            s[j] = score(kf);
        }
        group_sums(s, lpr);
#pragma unroll
        for (int j = 0; j < PP; ++j) {
            const int p = base + sid + j * stride;
            s[j] = p < p1 && p != upd ? s[j] * scale : -INFINITY;
            mn = fmaxf(mn, s[j]);
        }
        const int next = base + PP * stride;
        const bool more = next < p1;
        if (more) request_rows(kraw, kc, next);
        const float ref = finite_max(mn), corr = fast_exp(m - ref);
        m = mn;
        l *= corr;
#pragma unroll
        for (int v = 0; v < 8; ++v) o[v] *= corr;
#pragma unroll
        for (int j = 0; j < PP; ++j) {
            float vf[8];
            row_values(vraw[j], vf);
            s[j] = fast_exp(s[j] - ref);
            l += s[j];
#pragma unroll
            for (int v = 0; v < 8; ++v) o[v] = __builtin_fmaf(s[j], vf[v], o[v]);
        }
        if (!more) break;
        request_rows(vraw, vc, next);
        base = next;
    }
    // The lane groups of the wave: one maximum, then sums in which each half of the lanes goes on with half of the values.
    // Which of its 8 a lane ends up with: bits 5, 4 and 3 of its number, as many of them as there are lane groups.
    float mw = m;
    if (lpr == 8) mw = fmaxf(mw, dpp<DPP_ROR8>(mw));
    if (lpr <= 16) mw = pair_max16(mw);
    mw = pair_max32(mw);
    const float cw = fast_exp(m - finite_max(mw));
    l *= cw;
    l = halves32(l, l);
#pragma unroll
    for (int v = 0; v < 8; ++v) o[v] *= cw;
    float h4[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) h4[v] = halves32(o[v], o[v + 4]);
    GPTRS_LDS float* sm = lds;
    GPTRS_LDS float* sl = lds + NWS;
    GPTRS_LDS float* so = lds + 2 * NWS;
    GPTRS_LDS float* mine = so + wave * dh + c0 + (lane >> 5) * 4;
    if (lpr == 32) {
        GPTRS_LDS f32x4* d4 = (GPTRS_LDS f32x4*)mine;
        *d4 = f32x4{h4[0], h4[1], h4[2], h4[3]};
    } else {
        l = halves16(l, l);
        const float h0 = halves16(h4[0], h4[2]), h1 = halves16(h4[1], h4[3]);
        mine += ((lane >> 4) & 1) * 2;
        if (lpr == 16) {
            mine[0] = h0;
            mine[1] = h1;
        } else {
            l += dpp<DPP_ROR8>(l);
            const bool up = lane & 8;
            const float keep = up ? h1 : h0, give = up ? h0 : h1;
            mine[up ? 1 : 0] = keep + dpp<DPP_ROR8>(give);
        }
    }
    if (lane == 0) { sm[wave] = mw; sl[wave] = l; }
    wg_barrier();
    // the waves of each head: one record per query head
    const bool final = P.flags & kChainAttnFinal;
    for (int idx = t; idx < G * dh; idx += NS) {
        const int gg = idx >> (lsh + 3), d = idx & (dh - 1);
        float mr, lr, orr;
        if (nparts == 2) merge_waves<2>(sm, sl, so, gg, 4, dh, d, mr, lr, orr);
        else if (nparts == 8) merge_waves<8>(sm, sl, so, gg, 1, dh, d, mr, lr, orr);
        else if (nparts == 4) merge_waves<4>(sm, sl, so, gg, 2, dh, d, mr, lr, orr);
        else merge_waves<1>(sm, sl, so, gg, 8, dh, d, mr, lr, orr);
        if (final) {
            // one chunk per kv head: its record is the whole softmax, and the context row is written here (what the merge of
            // a single record gives: O / L)
            const long at = (long)(kvh * G + gg) * dh + d;
            if (F32) cstore4((float*)P.y + at, __float_as_uint(orr / lr));
            else __hip_atomic_store(as_global((unsigned short*)P.y + at), (unsigned short)pack_bf16x2(orr / lr, 0.f), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            continue;
        }
        float* rec = P.part + ((long)(kvh * G + gg) * nch + c) * (dh + 2);
        cstore4(rec + 2 + d, __float_as_uint(orr));
        if (d == 0) cstore8(rec, (unsigned long long)__float_as_uint(mr) | ((unsigned long long)__float_as_uint(lr) << 32));
    }
    // every lane's stores (record words, the appended cache row) have left the CU before the control wave, which passes
    // this barrier as well, reports the workgroup's arrival
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    wg_barrier();
    return true;
}

// unit = query head: softmax-merge of its nch chunk records into the context row.  A lane has the dims 2 d2, 2 d2 + 1 of the chunks
// wave, wave + 8, ...: all requested at once, merged, and the 8 waves' parts meet in LDS.
template <int N_REC>
__device__ __forceinline__ void merge_chunks(const float* base, int wave, int nch, int dh, int d2, bool act, float& m, float& l, float& o0, float& o1) {
    unsigned long long ml[N_REC], ov[N_REC];
#pragma unroll
    for (int u = 0; u < N_REC; ++u) {
        const int s = wave + u * NWS;
        const bool ok = act && s < nch;
        const float* rec = base + (long)s * (dh + 2);
        ml[u] = ok ? cload8(rec) : 0xff800000ull;   // (-inf, 0)
        ov[u] = ok ? cload8(rec + 2 + 2 * d2) : 0ull;
    }
    m = -INFINITY;
#pragma unroll
    for (int u = 0; u < N_REC; ++u) m = fmaxf(m, __uint_as_float((unsigned)ml[u]));
    const float ref = finite_max(m);
    l = 0.f; o0 = 0.f; o1 = 0.f;
#pragma unroll
    for (int u = 0; u < N_REC; ++u) {
        const float c = fast_exp(__uint_as_float((unsigned)ml[u]) - ref);
        l += __uint_as_float((unsigned)(ml[u] >> 32)) * c;
        o0 += __uint_as_float((unsigned)ov[u]) * c;
        o1 += __uint_as_float((unsigned)(ov[u] >> 32)) * c;
    }
}
template <int ROWS>
__device__ bool attn_combine(GPTRS_LDS int* go, GPTRS_LDS int* abort, const ChainPhase& P, GPTRS_LDS float* lds, int hq, int phase,
                             unsigned long long budget) {
    const int t = local_tid(), wave = uni(t >> 6), lane = t & 63;
    constexpr bool F32 = ROWS == kRowsF32;
    const int dh = P.head_dim, nch = P.nch, h2 = dh / 2;   // nch <= 64
    const float* base = P.part + (long)hq * nch * (dh + 2);
    float sink = 0.f;   // chunked rows: one more term of the head's denominator, and a gate over the head (a value of the projection's row)
    if (ROWS == kRowsChunk) sink = gload((const float*)P.gamma + hq);
    if (!wait_go(go, abort, phase, budget)) return false;
    float gate = 0.f;
    if (ROWS == kRowsChunk) gate = __uint_as_float(cload4((const float*)P.bias + hq));
    for (int d0 = 0; d0 < h2; d0 += 64) {
        const int d2 = d0 + lane;
        const bool act = d2 < h2;
        float m, l, o0, o1;
        if (nch <= 4 * NWS) merge_chunks<4>(base, wave, nch, dh, d2, act, m, l, o0, o1);
        else merge_chunks<8>(base, wave, nch, dh, d2, act, m, l, o0, o1);
        GPTRS_LDS f32x4* rec = (GPTRS_LDS f32x4*)lds;
        rec[wave * 64 + lane] = f32x4{m, l, o0, o1};
        wg_barrier();
        if (wave == 0 && act) {
            f32x4 v[NWS];
#pragma unroll
            for (int w = 0; w < NWS; ++w) v[w] = rec[w * 64 + lane];
            float M = v[0].x;
#pragma unroll
            for (int w = 1; w < NWS; ++w) M = fmaxf(M, v[w].x);
            if (ROWS == kRowsChunk) M = fmaxf(M, sink);
            const float ref = finite_max(M);
            float Lt = 0.f, a0 = 0.f, a1 = 0.f;
#pragma unroll
            for (int w = 0; w < NWS; ++w) {
                const float cw = fast_exp(v[w].x - ref);
                Lt += v[w].y * cw; a0 += v[w].z * cw; a1 += v[w].w * cw;
            }
            if (ROWS == kRowsChunk) { Lt += fast_exp(sink - ref); Lt *= 1.0f + expf(-gate); }   // (times the gate's sigmoid)
            if (F32) cstore8((float*)P.y + (long)hq * dh + 2 * d2, (unsigned long long)__float_as_uint(a0 / Lt) | ((unsigned long long)__float_as_uint(a1 / Lt) << 32));
            else cstore4((bf16_t*)P.y + (long)hq * dh + 2 * d2, pack_bf16x2(a0 / Lt, a1 / Lt));
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the context words are out before the arrival is reported
        wg_barrier();
    }
    return true;
}

// The compute waves of the workgroup: the units blk, blk + grid, ... of an attention phase.  The LDS operands travel as explicit
// local-address-space pointers so their accesses stay ds_* instructions.
// The descriptor comes straight from the table in memory (scalar loads): the waves enter an attention phase, and
// request the cache rows it needs, before the control wave has seen the barrier.
// The control wave only takes part in the workgroup barriers (attn_barriers of them to a unit).
__device__ __forceinline__ int attn_barriers(int kind, int head_dim) { return kind == kChainAttnCombine && head_dim > 128 ? 4 : 2; }
template <int ROWS>
__device__ __forceinline__ bool run_attn_phase(const GPTRS_CONST ChainPhase* php, GPTRS_LDS float* lds, GPTRS_LDS int* go, GPTRS_LDS int* abort, int phase,
                                               unsigned long long budget) {
    ChainPhase P;
    {
        int* dst = reinterpret_cast<int*>(&P);
        const GPTRS_CONST int* src = (const GPTRS_CONST int*)php;
#pragma unroll
        for (int i = 0; i < kPhaseDwords; ++i) dst[i] = uni(src[i]);
    }
    const int kind = P.kind, units = P.units;
    for (int u = blockIdx.x; u < units; u += gridDim.x) {
        const bool ok = kind == kChainAttnCombine ? attn_combine<ROWS>(go, abort, P, lds, u, phase, budget) : attn_partial<ROWS>(go, abort, P, lds, u, phase, budget);
        if (!ok) return false;
    }
    return true;
}

// ---------------------------------------------------------------------------- control wave
__device__ __forceinline__ float finish(float v, int flags, float bias, float res, float colscale) {
    if (flags & kChainBias) v += bias;                                           // tensor_ops.rs:42-56
    if (flags & kChainGelu) v = (v * 0.5f) * (erff(v / 1.41421354f) + 1.0f);     // activation.rs:96-113
    if (flags & kChainColScale) v *= colscale;
    if (flags & kChainResidual) v += res;
    return v;
}

template <int FMT>
// One wave works through this between the barriers that everybody waits at, so its instructions count one by one.  As a function of its own it
// looked the launch's LDS up in memory at every use (what uses dynamic LDS and is no kernel does): outputs of a phase left 0.57 to 0.77 us after the last
// sum for 0.74 to 1.05, GPT-2's 61 phases 356 -> 338 us, 157 of int8 codes 1200 -> 1182, of bf16 1640 either way.
__device__ __forceinline__ void control_wave(GPTRS_LDS Shared& sh, GPTRS_LDS unsigned* xs, const ChainPhase* phases, int nphases, unsigned* bar, int* abort_flag,
                             unsigned long long budget, int stall_phase) {
    PhaseTable table = (PhaseTable)phases;
    const int lane = threadIdx.x & 63;
    // The grid barrier.  Striped: a workgroup adds one to one of NC counters, and everybody polls all of them.  With notes: it adds one to its group's counter and
    // is told how many came before it; the last of a group leaves a note for every group, and everybody polls the eight notes for its own group, which
    // the group's L2 holds between two of them.  Two hops for one, but the arrivals meet nobody's polls.  By themselves 1.72 and 2.10 us (with values out and in 2.53 and 2.91);
    // 61 phases of GPT-2 305 and 327 us, 157 of bf16 1510 and 1545.  Where codes are streamed the wait for the answer costs more than that (int8 1121
    // and 1111, int4 1090 and 1060).  Every access is of agent scope: that a group shares a cache makes the notes fast, not right.
    constexpr bool NOTES = FMT == kChainW16 || FMT == kChainW32;
    const int blk = blockIdx.x, grp = blk % NG;
    const unsigned per = gridDim.x / NC, members = gridDim.x / NG;
    unsigned* const group_count = bar + (NC + grp) * LINE;
    unsigned* const notes = bar + (NC + NG) * LINE;
    unsigned* const counted = bar + (NC + NG + NG * NG) * LINE + (NOTES ? 1 : 0);   // phases that launches with this barrier have had
    const unsigned epoch = gload(counted);   // written by the previous launch, stable during this one
    const GPTRS_GLOBAL unsigned* const word = as_global(NOTES ? notes + (grp * NG + lane) * LINE : bar + lane * LINE);
    int handed = 0;   // arrivals of compute waves that the phases up to this one bring
    for (int ph = 0; ph < nphases; ++ph) {
        // the phase's descriptor is requested before the wait for the barrier and lands in LDS after it, ahead of `go`
        const int pd = lane < kPhaseDwords ? gload(reinterpret_cast<const int*>(phases + ph) + lane) : 0;
        const GPTRS_CONST ChainPhase* D = table + ph;
        const int kind = uni(D->kind);
        const int units = uni(D->units), barriers = attn_barriers(kind, uni(D->head_dim));
        const int T = kind == kChainLinear ? tile_count(blk, uni(D->tlo), uni(D->trem)) : 0;
        if (ph > 0) {
            // stall_phase (a test hook, -1 otherwise): one arrival more than the grid can deliver is expected at that
            // phase, so this wait runs out of time and the give-up path below is taken
            const unsigned target = (epoch + (unsigned)ph) * (NOTES ? 1u : per) + (ph == stall_phase ? 1u : 0u);
            Patience pat(budget);
            bool ok = true;
            for (;;) {
                const unsigned v = lane < (NOTES ? NG : NC) ? __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : target;
                if (__builtin_amdgcn_ballot_w64((int)(v - target) < 0) == 0) break;
                __builtin_amdgcn_s_sleep(1);
                if (pat.spent() || ((pat.spins & 63u) == 0 && __hip_atomic_load(as_global(abort_flag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) { ok = false; break; }
            }
            if (!ok) {
                __hip_atomic_store(as_global(abort_flag), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                lds_st(&sh.abort, 1);
                return;
            }
        }
        // the compute waves hold their own copy of the descriptor: the phase opens the moment the barrier is seen
        if (kind != kChainLinear) {
            if (blk < units) {
                if (lane == 0) lds_st(&sh.go, ph);
                for (int n = barriers * ((units - 1 - blk) / (int)gridDim.x + 1); n > 0; --n) wg_barrier();
            }
        } else if (T > 0) {
            if (lane == 0) lds_st(&sh.go, ph);
            PhaseRegs P;
            regs_from_lanes<FMT == kChainW32 || FMT == kChainW16, FMT == kChainW16>(P, pd);
            const int flags = P.flags, N = P.N;
            const bool dual = flags & kChainDual;
            const int cpt = dual ? 2 : 4;              // output columns per tile
            const int col0 = tile_first(blk, P.tlo, P.trem) * cpt;
            const int ncols = min(T * cpt, EPI_MAX);
            // bias / residual / int8 scales of this workgroup's columns: the first round is requested before the
            // staging loads and written to LDS after the staging, so that its latency hides behind the staging
            // instead of holding up the workgroup's barrier inside it
            const unsigned* bias = (const unsigned*)P.bias;
            const char* resid = (const char*)P.residual;
            constexpr int wfmt = FMT;   // every linear phase of a launch has the kernel's weight format
            const unsigned* sg = wfmt == kChainW8 ? (const unsigned*)P.wscale : nullptr;
            const unsigned* su = wfmt == kChainW8 ? (const unsigned*)P.wscale2 : nullptr;
            const char* cscale = (wfmt == kChainW16 || wfmt == kChainW32) && (flags & kChainColScale) ? (const char*)P.colscale : nullptr;
            unsigned long long e_cs = 0ull;              // two column factors
            const bool out_f32 = flags & kChainOutF32;   // y and the residual are f32
            unsigned long long e_rf = 0ull;              // two f32 residual values
            unsigned long long e_bf = 0ull;              // two f32 bias values (f32 phases)
            auto epi_load = [&](int i, unsigned& bw, unsigned& rw, unsigned& ga, unsigned& gb) {
                const int col = col0 + i;
                const bool in = i < ncols && col < N;
                if (wfmt == kChainW32) {
                    const u32x2 b2 = (bias && in) ? *(const GPTRS_GLOBAL u32x2*)((const char*)bias + 4 * (size_t)col) : u32x2{0u, 0u};
                    e_bf = (unsigned long long)b2.x | ((unsigned long long)b2.y << 32);
                    bw = 0u;
                } else
                bw = (bias && in) ? gload(bias + (col >> 1)) : 0u;
                if (out_f32) e_rf = (resid && in) ? cload8(resid + 4 * (size_t)col) : 0ull;
                rw = (resid && in && !out_f32) ? cload4(resid + 2 * (size_t)col) : 0u;
                if (cscale && in) {
                    const u32x2 c2 = *(const GPTRS_GLOBAL u32x2*)(cscale + 4 * (size_t)col);
                    e_cs = (unsigned long long)c2.x | ((unsigned long long)c2.y << 32);
                }
                ga = (sg && in) ? gload(sg + (col >> 1)) : 0u;
                gb = (su && in) ? gload(su + (col >> 1)) : 0u;
            };
            auto epi_store = [&](int i, unsigned bw, unsigned rw, unsigned ga, unsigned gb) {
                if (i >= ncols) return;
                if (bias || resid) {
                    *(GPTRS_LDS f32x2*)&sh.epi_bias[i] = wfmt == kChainW32 ? f32_pair(e_bf) : f32x2{bf16lo(bw), bf16hi(bw)};
                    *(GPTRS_LDS f32x2*)&sh.epi_res[i] = out_f32 ? f32_pair(e_rf) : f32x2{bf16lo(rw), bf16hi(rw)};
                }
                if (cscale) *(GPTRS_LDS f32x2*)&sh.epi_s[i] = f32_pair(e_cs);
                if (sg) {
                    *(GPTRS_LDS f32x2*)&sh.epi_s[i] = f32x2{bf16lo(ga), bf16hi(ga)};
                    *(GPTRS_LDS f32x2*)&sh.epi_s[EPI_MAX + i] = f32x2{bf16lo(gb), bf16hi(gb)};
                }
            };
            const bool has_epi = bias || resid || sg || cscale;
            unsigned e_bw = 0u, e_rw = 0u, e_ga = 0u, e_gb = 0u;
            if (has_epi) epi_load(lane * 2, e_bw, e_rw, e_ga, e_gb);
            // residual prologue: the workgroups of the phase leave the sum in memory, a share each.  What a lane's first element
            // needs is requested ahead of the staging.
            const bool post = wfmt == kChainW16 && (flags & kChainPostNorm);
            float* post_y = post ? (float*)const_cast<void*>(GPTRS_PD_PTR(post_y)) : nullptr;
            int post_i = 0, post_end = 0;
            float post_v = 0.f, post_r = 0.f, post_g = 0.f;
            auto post_load = [&](int i) {
                post_v = __uint_as_float(cload4((const float*)P.x + i));
                post_r = __uint_as_float(cload4((const float*)P.post_res + i));
                post_g = gload((const float*)P.post_gain + i);
            };
            if (post_y) {
                const int active = P.tlo > 0 ? (int)gridDim.x : P.trem, share = (P.K + active - 1) / active;
                post_i = blk * share + lane;
                post_end = min(blk * share + share, P.K);
                if (post_i < post_end) post_load(post_i);
            }
            float post_inv = 0.f;
            if (wfmt == kChainW32) stage_block_f32(P, xs, &sh.ssq[0]);
            else post_inv = stage_block<FMT>(P, xs, &sh.ssq[0]);
            if (post_y) {
                for (int i = post_i; i < post_end; i += 64) {
                    if (i != post_i) post_load(i);
                    cstore4(post_y + i, __float_as_uint(post_r + ((post_v * post_inv) * post_g) * P.post_mult));
                }
            }
            if (has_epi) {
                epi_store(lane * 2, e_bw, e_rw, e_ga, e_gb);
                for (int i = lane * 2 + 128; i < ncols; i += 128) {
                    epi_load(i, e_bw, e_rw, e_ga, e_gb);
                    epi_store(i, e_bw, e_rw, e_ga, e_gb);
                }
                // below a lane reads what other lanes of the wave have stored (no instruction: LDS serves a wave in order, the compiler has to as well)
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
            char* out = (char*)P.y;
            handed += NWS;
            const int W = T * P.C;
            // A lane's column i: tile i / cpt of the workgroup, whose parts lie in the rows of the waves that hold its words.  All it
            // needs besides the sums is read ahead of the wait for them.
            for (int i0 = 0; i0 < ncols; i0 += 64) {
                const int i = min(i0 + lane, ncols - 1), col = col0 + i;
                const int tl = dual ? i >> 1 : i >> 2, c = dual ? (i & 1) * 2 : i & 3;
                int w0 = 0, w1 = 0;   // the waves of the tile's first and last word
#pragma unroll
                for (int w = 1; w < NWS; ++w) {
                    const int f = wave_first(W, w);
                    w0 += f <= tl * P.C ? 1 : 0;
                    w1 += f <= tl * P.C + P.C - 1 ? 1 : 0;
                }
                const float sc = (wfmt == kChainW8 || cscale) ? sh.epi_s[i] : 1.f;
                const float su2 = (wfmt == kChainW8 && dual) ? sh.epi_s[EPI_MAX + i] : 1.f;
                const bool add = flags & (kChainBias | kChainResidual);   // both arrays are staged when either is present
                const float bi = add ? sh.epi_bias[i] : 0.f, re = add ? sh.epi_res[i] : 0.f;
                const GPTRS_LDS float* first_part = &sh.part[tl + w0][c & 2];
                if (i0 == 0) {
                    Patience pat(8 * budget);
                    while (lds_ld(&sh.done) < handed) {
                        __builtin_amdgcn_s_sleep(1);
                        if (pat.spent()) {
                            lds_st(&sh.abort, 1);
                            __hip_atomic_store(as_global(abort_flag), 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            return;
                        }
                    }
                    GPTRS_LDS_ACQUIRE();
                }
                float s = 0.f, s2 = 0.f;   // s2: the up column of a pair
                // (the parts of a tile by consecutive waves lie in consecutive rows; rows behind the tile's last part are another's and count as nothing)
                auto part = [&](int u) { return *(const GPTRS_LDS f32x2*)&first_part[4 * u]; };
                auto take = [&](int u, f32x2 v) {   // (a pair's c is even)
                    const float vx = w0 + u <= w1 ? v.x : 0.f, vy = w0 + u <= w1 ? v.y : 0.f;
                    s += (c & 1) ? vy : vx;
                    s2 += vy;
                };
                if (T >= NWS) {   // a tile's words are in two waves at most
                    const f32x2 a = part(0), b = part(1);
                    take(0, a); take(1, b);
                } else {
                    f32x2 v[NWS];
#pragma unroll
                    for (int u = 0; u < NWS; ++u) v[u] = part(u);
#pragma unroll
                    for (int u = 0; u < NWS; ++u) take(u, v[u]);
                }
                if (wfmt == kChainW8) { s *= sc; s2 *= su2; }
                float o;
                if (dual) {   // columns interleaved (gate, up, gate, up): activation.rs:141-162
                    const int glu = flags & kChainClampedGlu ? 1 : 0;
                    o = finish(glu_combine(s, s2, glu, P.glu_limit, P.glu_alpha, P.glu_shift), flags, bi, re, 1.0f);
                } else {
                    o = finish(s, flags, bi, re, sc);
                    if (wfmt == kChainW16 && (flags & kChainSoftcap)) o = softcap_f32(o, P.glu_limit);   // (softcap shares the field)
                }
                if (i0 + lane < ncols && col < N) {   // (the last tile of a width that is not a multiple of 4 has columns that do not exist)
                    if (out_f32) cstore4(out + 4 * (size_t)col, __float_as_uint(o));
                    else __hip_atomic_store(as_global((unsigned short*)out + (size_t)col), (unsigned short)pack_hw(o, 0.f), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
        // this workgroup's outputs have left the CU before it arrives at the barrier
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        asm volatile("" ::: "memory");
        if (NOTES) {
            unsigned before = 0u;
            if (lane == 0) before = __hip_atomic_fetch_add(as_global(group_count), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned done = epoch + (unsigned)ph + 1u;
            if ((unsigned)uni((int)before) + 1u == done * members && lane < NG)
                __hip_atomic_store(as_global(notes) + (lane * NG + grp) * LINE, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else if (lane == 0) {
            __hip_atomic_fetch_add(as_global(bar) + (blk % NC) * LINE, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // every launch counts its phases: the next launch starts from there
    if (blk == 0 && lane == 0) gstore(counted, epoch + (unsigned)nphases);
}

// In the bf16 kernel, where requests ahead fill what the barriers leave, the compute waves' registers are dealt better beside a function of its own (157 phases 1542 us,
// 1598 with the text in line).
template <int FMT>
__device__ __noinline__ void control_wave_apart(GPTRS_LDS Shared& sh, GPTRS_LDS unsigned* xs, const ChainPhase* phases, int nphases, unsigned* bar, int* abort_flag,
                                                unsigned long long budget, int stall_phase) {
    control_wave<FMT>(sh, xs, phases, nphases, bar, abort_flag, budget, stall_phase);
}

// Sums each of a wave's 4 per-lane accumulators over its 64 lanes as a reduce-scatter: exchanging half of the values with lane ^ 32
// and then lane ^ 16 leaves every 16-lane row with one value already summed over 4 lanes, which 4 row-wide DPP steps finish.
// Returns the total of accumulator r in every lane of row r.
__device__ __forceinline__ float reduce_tile(const float (&acc)[4]) {
    float h[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {   // lanes < 32 keep values 0 and 1, lanes >= 32 values 2 and 3
        const u32x2 sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[k]), __float_as_uint(acc[k + 2]), false, false);
        h[k] = __uint_as_float(sw.x) + __uint_as_float(sw.y);
    }
    const u32x2 sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(h[0]), __float_as_uint(h[1]), false, false);
    int x = __float_as_int(__uint_as_float(sw.x) + __uint_as_float(sw.y));
#define GPTRS_DPP_ADD(ctrl) x = __float_as_int(__int_as_float(x) + __int_as_float(__builtin_amdgcn_update_dpp(0, x, (ctrl), 0xf, 0xf, false)))
    GPTRS_DPP_ADD(0xB1);    // quad_perm [1,0,3,2]
    GPTRS_DPP_ADD(0x4E);    // quad_perm [2,3,0,1]
    GPTRS_DPP_ADD(0x141);   // row_half_mirror
    GPTRS_DPP_ADD(0x140);   // row_mirror
#undef GPTRS_DPP_ADD
    return __int_as_float(x);
}

// ---------------------------------------------------------------------------- compute waves
// vector memory operations of the wave that are in flight, without waiting: says when it is worth while to look.  That words have
// landed is what the wait below says, and nothing is read out of the ring without it.
__device__ __forceinline__ int vm_in_flight() {
    unsigned v;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_IB_STS)" : "=s"(v) : : "memory");
    return (int)((v & 15u) | ((v >> 18) & 0x30u));
}
// s_waitcnt that waits until at most N vector memory operations of the wave are in flight (and for nothing else); the count is
// an immediate of the instruction
template <int N> __device__ __forceinline__ void wait_vm_imm() { __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14)); }
__device__ __forceinline__ void wait_vm_count(int n) {   // a step of fewer than three words in flight behind the oldest one, or a full ring
    switch (n) {
#define GPTRS_VM(k) case k: wait_vm_imm<k>(); break;
        GPTRS_VM(1) GPTRS_VM(2) GPTRS_VM(3) GPTRS_VM(4) GPTRS_VM(5) GPTRS_VM(6) GPTRS_VM(7) GPTRS_VM(8)
        GPTRS_VM(9) GPTRS_VM(10) GPTRS_VM(11) GPTRS_VM(12)
#undef GPTRS_VM
        default: wait_vm_imm<0>(); break;   // 0, and anything unexpected: wait for everything
    }
    static_assert(3 * (RING_MAX - 1) <= 12, "cases above");
}

// what a lane reads of the staged activations for one word: its k-group's bf16 values, or one f32
template <int FMT> struct Act { typedef unsigned type; };
template <> struct Act<kChainW8> { typedef u32x2 type; };
template <> struct Act<kChainW4> { typedef u32x4 type; };

template <int FMT, int RING_D, int ROWS>
__device__ void compute_waves(Shared& sh, const unsigned* xs, PhaseTable table, int nphases, const unsigned char* ring, unsigned long long budget) {
    const int t = threadIdx.x, lane = t & 63, wave = uni(t >> 6);
    const int blk = blockIdx.x;

    // ---- request side: the wave's next step to ask for, in the order the steps are consumed.  Everything but the lane's offset
    // in a word is uniform.
    int r_part = -1, r_left = 0;      // part of a phase (2 phase: its whole steps, 2 phase + 1: the rest), words of it that are still to be asked for
    unsigned r_step_bytes = 0;
    unsigned long long r_base = 0;    // the next step's first word
    const unsigned lane_off = (unsigned)lane * 16u;
    const unsigned ring_lds = (unsigned)uni((int)((unsigned)(size_t)(GPTRS_LDS unsigned char*)ring + (unsigned)(wave * (RING_D * STEP_BYTES))));
    int r_slot = 0;                   // slot of the ring to fill next
    int inflight = 0;                 // steps requested and not yet read
    unsigned pend = 0u;               // bits 2i, 2i + 1: loads that the i-th oldest of them carries
    int loads = 0;                    // loads in flight
    auto r_seek = [&]() -> bool {     // next part of a linear phase in which this wave has words (an attention phase has no tiles)
        for (;;) {
            ++r_part;
            if (r_part >> 1 >= nphases) return false;
            const GPTRS_CONST ChainPhase* D = table + (r_part >> 1);
            const WavePart p = wave_part(blk, wave, r_part & 1, uni(D->C), uni(D->tlo), uni(D->trem), uni(D->whole), uni(D->behind));
            r_left = p.words;
            if (p.more == 0) r_part |= 1;
            if (r_left == 0) continue;
            r_step_bytes = p.run ? (unsigned)STEP_BYTES : (unsigned)uni(D->step_bytes);
            r_base = (unsigned long long)uni_ptr(D->w) + ((unsigned long long)(unsigned)p.at << 10);
            return true;
        }
    };
    static_assert(CW * 16 == 1 << 10, "bytes of a word");
    bool r_more = r_seek();
    // Asks for one step: a load per word that exists (three but for the last step of a wave's rest).  `pend` records how many loads each step
    // in flight carries, two bits per step, oldest first.  Every load fetches words never fetched before, so all of them take the
    // same way through the memory system and return in the order of issue: a load that re-read words already in a cache was seen
    // to complete ahead of older ones, which a count of loads in flight cannot express.  A step's words lie one behind the other
    // in memory and in LDS, and the instruction's offset counts for both addresses.
    auto request = [&]() {
        const unsigned dst = (unsigned)uni((int)(ring_lds + (unsigned)(r_slot * STEP_BYTES)));
        const unsigned long long base = (unsigned long long)uni_ptr((const char*)r_base);
        int cnt = SW;
        if (__builtin_expect(r_left >= SW, 1)) {
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024\n\tglobal_load_lds_dwordx4 %0, %1 offset:2048"
                         : : "v"(lane_off), "s"(base), "s"(dst) : "memory", "m0");
        } else {
            cnt = r_left;
            if (cnt == 2)
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024"
                             : : "v"(lane_off), "s"(base), "s"(dst) : "memory", "m0");
            else
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(lane_off), "s"(base), "s"(dst) : "memory", "m0");
        }
        static_assert(SW == 3 && CW * 16 == 1024, "offsets above");
        pend |= (unsigned)cnt << (2 * inflight);
        loads += cnt;
        ++inflight;
        if (++r_slot == RING_D) r_slot = 0;
        r_base += r_step_bytes;
        r_left -= cnt;
        if (__builtin_expect(r_left == 0, 0)) r_more = r_seek();
    };
    for (int i = 0; i < RING_D && r_more; ++i) request();

    // ---- read side
    int c_phase = -1, c_left = 0, c_k = 0, c_C = 1, c_row = 0, c_soff = 0, c_stile = 0;
    constexpr int c_fmt = FMT;
    PhaseRegs R;
    // advance to the next linear phase in which this workgroup has tiles, taking part in attention phases on the way
    auto c_seek = [&]() -> bool {
        for (;;) {
            ++c_phase;
            if (c_phase >= nphases) return false;
            const GPTRS_CONST ChainPhase* D = table + c_phase;   // the fields that decide this workgroup's part, before the wait
            if (uni(D->kind) != kChainLinear) {
                if (blk >= uni(D->units)) continue;
                if (!run_attn_phase<ROWS>(table + c_phase, (GPTRS_LDS float*)xs, (GPTRS_LDS int*)&sh.go, (GPTRS_LDS int*)&sh.abort, c_phase,
                                    budget)) return false;
                continue;
            }
            const int T = tile_count(blk, uni(D->tlo), uni(D->trem));
            if (T == 0) continue;
            c_C = uni(D->C);
            const int W = T * c_C, f0 = wave_first(W, wave);
            c_left = wave_first(W, wave + 1) - f0;
            // tile and k of the wave's first word (f0 + 1/2 over C is at least 1 / (2 C) away from a whole number: exact below 2^22 words)
            const int tl = uni((int)(((float)f0 + 0.5f) * __int_as_float(uni(__float_as_int(D->inv_c)))));
            c_k = f0 - tl * c_C;
            c_row = tl + wave;
            c_stile = tl * c_C * 4;             // int4: the tile's first entry in the staged scales ...
            c_soff = uni(D->lds_bytes) >> 2;    // ... which sit behind the activations
            regs_from_table<FMT == kChainW32 || FMT == kChainW16, FMT == kChainW16>(R, D);
            return true;   // (the caller waits for the phase to open and stages its input)
        }
    };

    // two chains per column, words in turn: half as many additions behind one another
    float acc[2][4];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[p][c] = 0.f;
    int slot = 0;
    const GPTRS_LDS u32x4* mine = (const GPTRS_LDS u32x4*)ring + wave * (RING_D * SW * CW) + lane;   // this lane's piece of word 0 in slot 0

    // this lane's activations for word k of a tile
    auto activations = [&](int k) -> typename Act<FMT>::type {
        return *reinterpret_cast<const typename Act<FMT>::type*>(&xs[(k * CW + lane) * (int)(sizeof(typename Act<FMT>::type) / 4)]);
    };
    // word k of its tile times the staged activations
    auto multiply = [&](const u32x4& q4, const typename Act<FMT>::type& act, int k, float (&a)[4]) {
        // element reads go through scalars: __builtin_bit_cast applied directly to `vec.y` of an
        // ext-vector reads element 0 with this compiler
        const unsigned q[4] = {q4.x, q4.y, q4.z, q4.w};
        if constexpr (c_fmt == kChainW16) {
            const unsigned xw = act;
            const bf16x2 xv = __builtin_bit_cast(bf16x2, xw);
#pragma unroll
            for (int c = 0; c < 4; ++c) a[c] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, q[c]), xv, a[c], false);
        } else if constexpr (c_fmt == kChainW32) {
            const float xv = __uint_as_float(act);
#pragma unroll
            for (int c = 0; c < 4; ++c) a[c] = __builtin_fmaf(__uint_as_float(q[c]), xv, a[c]);
        } else if constexpr (c_fmt == kChainW8) {
            const unsigned xa = act.x, xb = act.y;
            const float x0 = bf16lo(xa), x1 = bf16hi(xa), x2 = bf16lo(xb), x3 = bf16hi(xb);
            const float corr = -128.0f * ((x0 + x1) + (x2 + x3));
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                float v = a[c] + corr;
                v = __builtin_fmaf((float)(q[c] & 0xFFu), x0, v);
                v = __builtin_fmaf((float)((q[c] >> 8) & 0xFFu), x1, v);
                v = __builtin_fmaf((float)((q[c] >> 16) & 0xFFu), x2, v);
                v = __builtin_fmaf((float)(q[c] >> 24), x3, v);
                a[c] = v;
            }
        } else {
            const unsigned xa = act.x, xb = act.y, xc = act.z, xd = act.w;
            const float x0 = bf16lo(xa), x1 = bf16hi(xa), x2 = bf16lo(xb), x3 = bf16hi(xb);
            const float x4 = bf16lo(xc), x5 = bf16hi(xc), x6 = bf16lo(xd), x7 = bf16hi(xd);
            const float corr = -8.0f * (((x0 + x1) + (x2 + x3)) + ((x4 + x5) + (x6 + x7)));
            const u32x2 sw = *reinterpret_cast<const u32x2*>(&xs[c_soff + 2 * (c_stile + k * 4 + (lane >> 4))]);
            const unsigned sa = sw.x, sb = sw.y;
            const float sc[4] = {bf16lo(sa), bf16hi(sa), bf16lo(sb), bf16hi(sb)};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                // byte i of a column's dword: k = 2i in the low nibble, k = 2i + 1 in the high one
                const unsigned lo = q[c] & 0x0F0F0F0Fu, hi = (q[c] >> 4) & 0x0F0F0F0Fu;
                float v = corr;
                v = __builtin_fmaf((float)(lo & 0xFFu), x0, v);
                v = __builtin_fmaf((float)(hi & 0xFFu), x1, v);
                v = __builtin_fmaf((float)((lo >> 8) & 0xFFu), x2, v);
                v = __builtin_fmaf((float)((hi >> 8) & 0xFFu), x3, v);
                v = __builtin_fmaf((float)((lo >> 16) & 0xFFu), x4, v);
                v = __builtin_fmaf((float)((hi >> 16) & 0xFFu), x5, v);
                v = __builtin_fmaf((float)(lo >> 24), x6, v);
                v = __builtin_fmaf((float)(hi >> 24), x7, v);
                a[c] = __builtin_fmaf(sc[c], v, a[c]);
            }
        }
    };
    auto leave_tile = [&]() {   // the wave's part of a tile's 4 sums
        float sum[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) { sum[c] = acc[0][c] + acc[1][c]; acc[0][c] = 0.f; acc[1][c] = 0.f; }
        const float v = reduce_tile(sum);
        if ((lane & 15) == 0) sh.part[c_row][lane >> 4] = v;
        ++c_row;
        c_stile += 4 * c_C;
        c_k = 0;
    };

    // A request can hold its wave for a microsecond (the memory pipeline of a CU takes a limited number of requests, and one
    // beyond that waits for an older one to land), so the request that a read frees is made after the step's arithmetic
    // and, at the end of a phase, after the sums are handed over: nothing the workgroup waits for stands behind it.
    while (c_seek()) {
      // Until the phase opens the wave has nothing to do, and what has landed cannot be used yet: the memory system would idle
      // through the barrier.  So the ring is filled up to FLIGHT steps, and then the oldest steps move from the ring into registers (`park`) and
      // the slots they leave are asked to fetch further ahead.  A step is only asked for when nothing of the wave is in flight:
      // the pipeline that the control wave polls the barrier through stays short.  Parked steps are the phase's first ones and
      // are read back first; the registers are free again before the next phase is looked for.
      constexpr int PARKN = FMT == kChainW4 ? PARK_W4 : FMT == kChainW8 ? PARK_W8 : FMT == kChainW32 ? PARK_W32 : PARK;   // (the int4 kernel stages its group scales through registers as well)
      u32x4 park[PARKN][SW];
      int n_parked = 0, park_rd = 0;
      {
        auto closed = [&]() { return uni(lds_ld(&sh.go)) < c_phase && !uni(lds_ld(&sh.abort)); };
        while (r_more && inflight < FLIGHT && closed()) {
            if (vm_in_flight() == 0) request(); else __builtin_amdgcn_s_sleep(1);
        }
        const int want = min(PARKN, min((c_left + SW - 1) / SW, inflight));
#pragma unroll
        for (int i = 0; i < PARKN; ++i) {
            if (i < want) {
                while (vm_in_flight() > 0 && closed()) __builtin_amdgcn_s_sleep(1);
                if (vm_in_flight() == 0 && closed()) {
                    wait_vm_imm<0>();   // (of no length: nothing is in flight)
                    pend = 0u;
                    loads = 0;
                    const GPTRS_LDS u32x4* wp = mine + slot * (SW * CW);
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int p = 0; p < SW; ++p) park[i][p] = wp[p * CW];
                    --inflight;
                    if (++slot == RING_D) slot = 0;
                    __builtin_amdgcn_s_waitcnt(0xC07F);
                    asm volatile("" ::: "memory");
                    if (r_more) request();
                    n_parked = i + 1;
                } else break;
            }
        }
      }
      if (!wait_go(&sh.go, &sh.abort, c_phase, budget)) break;
      if (FMT == kChainW32) stage_block_f32(R, (GPTRS_LDS unsigned*)const_cast<unsigned*>(xs), (GPTRS_LDS float*)sh.ssq);
      else stage_block<FMT>(R, (GPTRS_LDS unsigned*)const_cast<unsigned*>(xs), (GPTRS_LDS float*)sh.ssq);
      // All loads of the wave have landed from here on.  A wave that has staged a part of the row has waited for them with it, since loads return in order; one
      // that has not (f32 rows of 768 take three waves) waits here for the words it has under way.  The compiler is told by it too: left to itself it
      // waited for all loads in flight at the top of each pass of the loop below.
      wait_vm_imm<0>();
      if (r_more && inflight < RING_D) request();
      while (c_left > 0) {
        u32x4 cur[SW];
        if (park_rd < n_parked) {
            switch (park_rd) {
#define GPTRS_PARK(k) case k: _Pragma("unroll") for (int p = 0; p < SW; ++p) cur[p] = park[k < PARKN ? k : 0][p]; break;
                GPTRS_PARK(0) GPTRS_PARK(1)
                default: _Pragma("unroll") for (int p = 0; p < SW; ++p) cur[p] = park[PARKN - 1][p]; break;
#undef GPTRS_PARK
            }
            static_assert(PARKN >= 1 && PARKN <= 3, "cases above");
            ++park_rd;
        } else {
            const GPTRS_LDS u32x4* wp = mine + slot * (SW * CW);
            // the loads of this step are the oldest in flight: they have landed once no more than the younger ones remain
            {
                const int oldest = (int)(pend & 3u), younger = loads - oldest;
                if (oldest) {
                    if (__builtin_expect(younger == SW * (FLIGHT_LONG - 1), 1)) wait_vm_imm<SW * (FLIGHT_LONG - 1)>();
                    else if (__builtin_expect(younger == SW * (FLIGHT - 1), 1)) wait_vm_imm<SW * (FLIGHT - 1)>();
                    else if (__builtin_expect(younger == 0, 1)) wait_vm_imm<0>();
                    else wait_vm_count(younger);
                }
                pend >>= 2;
                loads = younger;
            }
            asm volatile("" ::: "memory");
#pragma unroll
            for (int p = 0; p < SW; ++p) cur[p] = wp[p * CW];
            --inflight;
            if (++slot == RING_D) slot = 0;
        }
        if (__builtin_expect(c_left >= SW && c_k + SW <= c_C, 1)) {   // three words of one tile
            typename Act<FMT>::type x[SW];
#pragma unroll
            for (int p = 0; p < SW; ++p) x[p] = activations(c_k + p);
#pragma unroll
            for (int p = 0; p < SW; ++p) multiply(cur[p], x[p], c_k + p, acc[p & 1]);
            c_k += SW;
            c_left -= SW;
            if (c_k == c_C) leave_tile();
        } else {
#pragma unroll
            for (int p = 0; p < SW; ++p) {
                if (c_left > 0) {
                    multiply(cur[p], activations(c_k), c_k, acc[p & 1]);
                    --c_left;
                    if (++c_k == c_C) leave_tile();
                }
            }
        }
        if (c_left > 0 && r_more && inflight < (c_left > LONG_WORDS ? FLIGHT_LONG : FLIGHT)) request();   // (a parked step's slot was refilled when it was parked)
      }
      if (c_k > 0) leave_tile();
      GPTRS_LDS_RELEASE();
      if (lane == 0) __hip_atomic_fetch_add(&sh.done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (r_more && inflight < RING_D) request();
    }
}

// ROWS: what the launch's attention phases read
template <int FMT, int RING_D, int ROWS = FMT == kChainW32 ? kRowsF32 : kRowsBf16>
__global__ __launch_bounds__(NT, 1) void chain_kernel(const ChainPhase* __restrict__ phases, int nphases, unsigned* bar, int* abort_flag,
                                                        int xs_bytes, unsigned long long budget, int stall_phase) {
    extern __shared__ __align__(16) unsigned char smem[];
    Shared& sh = *reinterpret_cast<Shared*>(smem);
    unsigned* xs = reinterpret_cast<unsigned*>(smem + sizeof(Shared));
    unsigned char* ring = smem + sizeof(Shared) + xs_bytes;
    PhaseTable table = (PhaseTable)phases;
    {
        if (threadIdx.x == 0) { sh.go = -1; sh.done = 0; sh.abort = 0; }
        __syncthreads();
    }
    const int wave = threadIdx.x >> 6;
    if (wave < NWS) {
        compute_waves<FMT, RING_D, ROWS>(sh, xs, table, nphases, ring, budget);
        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): no load may land in LDS after the workgroup has gone
    } else {
        if constexpr (FMT == kChainW16) {
            unsigned at = (unsigned)(size_t)(GPTRS_LDS unsigned char*)smem;
            asm volatile("" : "+s"(at));   // (where the address comes from is hidden: see control_wave)
            control_wave_apart<FMT>(*(GPTRS_LDS Shared*)at, (GPTRS_LDS unsigned*)(at + (unsigned)sizeof(Shared)), phases, nphases, bar, abort_flag, budget, stall_phase);
        } else {
            control_wave<FMT>(*(GPTRS_LDS Shared*)smem, (GPTRS_LDS unsigned*)xs, phases, nphases, bar, abort_flag, budget, stall_phase);
        }
    }
}

// ---------------------------------------------------------------------------- weight layout
// Single: column = 4 * tile + c.  Dual (SwiGLU pair): columns interleaved, c = 0, 2 -> gate column 2 * tile + c / 2, c = 1, 3 -> the
// same column of up, so one tile finishes two outputs.  A word holds 64 k-groups of the tile's 4 columns, lane l (16 bytes) group
// 64 chunk + l: 2 k of each column in bf16, 1 in f32, 4 int8 codes, 8 int4 codes.  Zero (of codes: the biased zero) outside the matrix.
// Every word of the matrix has one place (WavePart), and there is nothing else: with the waves' last steps padded to three words, and room in a step for workgroups
// without tiles, 3072 x 64 took 6.3 MB for 0.39, and the layers of GPT-2 small 528 MB for 340.
struct ChainOrder {
    int64_t ntiles, C, grid, tlo, trem;
    __host__ __device__ int64_t active() const { return tlo > 0 ? grid : trem; }   // workgroups that have tiles
    // Under two steps a wave asks for all of its words at once, whatever their order: they are one run, which saves the second look into the table.
    __host__ __device__ int64_t whole() const {
        const int64_t least = (tlo > 0 ? tlo : 1) * C / NWS;   // words of a wave
        return least < 2 * SW ? 0 : least / SW;
    }
    __host__ __device__ int64_t word(int64_t tile, int64_t chunk) const {
        const int64_t big = trem * (tlo + 1);
        const int64_t b = tile < big ? tile / (tlo + 1) : trem + (tile - big) / tlo;
        const int64_t t0 = b * tlo + (b < trem ? b : trem), W = (tlo + (b < trem ? 1 : 0)) * C, f = (tile - t0) * C + chunk;
        const int64_t w = (8 * f + 7) / W, i = f - wave_first((int)W, (int)w), n = whole();   // word i of wave w
        const WavePart p = wave_part((int)b, (int)w, i >= SW * n, (int)C, (int)tlo, (int)trem, (int)n, (int)behind());
        return p.run ? p.at + i - SW * n : p.at + (i / SW) * active() * (NWS * SW) + i % SW;
    }
    __host__ __device__ int64_t behind() const { return whole() * active() * (NWS * SW); }
    int64_t words() const { return ntiles * C; }
};

__device__ __forceinline__ const void* chain_column(const void* w, const void* w2, int64_t tile, int c, int64_t& col) {
    if (w2) { col = tile * 2 + (c >> 1); return (c & 1) ? w2 : w; }
    col = tile * 4 + c;
    return w;
}
__global__ void chain_pack_kernel(const bf16_t* __restrict__ w, const bf16_t* __restrict__ w2, uint32_t* __restrict__ out,
                                  int64_t K, int64_t N, ChainOrder o) {
    const int64_t total = o.ntiles * o.C * 256;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(idx & 3);
        const int64_t j = (idx >> 2) % (o.C * CW), tile = (idx >> 2) / (o.C * CW);
        int64_t col;
        const bf16_t* src = (const bf16_t*)chain_column(w, w2, tile, c, col);
        uint32_t lo = 0, hi = 0;
        if (col < N) {
            if (2 * j < K) lo = src[(2 * j) * N + col];
            if (2 * j + 1 < K) hi = src[(2 * j + 1) * N + col];
        }
        out[o.word(tile, j / CW) * 256 + (j % CW) * 4 + c] = lo | (hi << 16);
    }
}
__global__ void chain_pack_f32_kernel(const float* __restrict__ w, float* __restrict__ out, int64_t K, int64_t N, ChainOrder o) {
    const int64_t total = o.ntiles * o.C * 256;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(idx & 3);
        const int64_t j = (idx >> 2) % (o.C * CW), tile = (idx >> 2) / (o.C * CW);
        const int64_t col = tile * 4 + c;
        out[o.word(tile, j / CW) * 256 + (j % CW) * 4 + c] = (col < N && j < K) ? w[j * N + col] : 0.f;
    }
}
// Quantised codes: one byte per (column, code row), group j of a tile holds code rows 4j .. 4j+3 of its 4 columns.  int8: a code
// row is one k, bytes stored as q + 128 (flip = 0x80).  int4: a code row is a packed byte (k = 2r low nibble, 2r + 1 high
// nibble), both nibbles stored as q + 8 (flip = 0x88).
__global__ void chain_pack_codes_kernel(const uint8_t* __restrict__ w, const uint8_t* __restrict__ w2, uint32_t* __restrict__ out,
                                        int64_t rows, int64_t N, ChainOrder o, uint32_t flip) {
    const int64_t total = o.ntiles * o.C * 256;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(idx & 3);
        const int64_t j = (idx >> 2) % (o.C * CW), tile = (idx >> 2) / (o.C * CW);
        int64_t col;
        const uint8_t* src = (const uint8_t*)chain_column(w, w2, tile, c, col);
        uint32_t v = 0;
        for (int h = 0; h < 4; ++h) {
            const int64_t r = 4 * j + h;
            const uint32_t b = (col < N && r < rows) ? ((uint32_t)src[r * N + col] ^ flip) : flip;
            v |= b << (8 * h);
        }
        out[o.word(tile, j / CW) * 256 + (j % CW) * 4 + c] = v;
    }
}
// int4 group scales in tile order: sc[tile][g][c] (bf16) for g < 4 C, zero outside the matrix
__global__ void chain_pack_scales_kernel(const bf16_t* __restrict__ sc, const bf16_t* __restrict__ sc2, bf16_t* __restrict__ out,
                                         int64_t groups, int64_t N, int64_t G, int64_t ntiles) {
    const int64_t total = ntiles * G * 4;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(idx & 3);
        const int64_t g = (idx >> 2) % G, tile = (idx >> 2) / G;
        int64_t col;
        const bf16_t* src = (const bf16_t*)chain_column(sc, sc2, tile, c, col);
        out[idx] = (col < N && g < groups) ? src[g * N + col] : (bf16_t)0;
    }
}
// The inverse of the bf16 copy: the row-major [K, N] matrix back, exactly -- the copy is a permutation plus zero padding.  A matrix
// whose packed copy exists need not stay resident in its row-major form; this brings it back when some other kernel family
// asks for it.  second: the up matrix of a pair.
__global__ void chain_unpack_kernel(const uint32_t* __restrict__ packed, bf16_t* __restrict__ w, int64_t K, int64_t N, ChainOrder o, int dual, int second) {
    const int64_t total = (K + 1) / 2 * N;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t col = idx % N, j = idx / N;
        const int64_t tile = dual ? col >> 1 : col >> 2, c = dual ? ((col & 1) << 1) + second : col & 3;
        const uint32_t v = packed[o.word(tile, j / CW) * 256 + (j % CW) * 4 + c];
        w[(2 * j) * N + col] = (bf16_t)(v & 0xFFFFu);
        if (2 * j + 1 < K) w[(2 * j + 1) * N + col] = (bf16_t)(v >> 16);
    }
}

static int g_grid = 0;
static int g_occupancy_ok[10] = {-1, -1, -1, -1, -1, -1, -1, -1, -1, -1};   // per kernel: does a workgroup fit a CU with the LDS it asks for

}  // namespace

int chain_grid() {
    if (g_grid == 0) {
        int dev = 0;
        hipDeviceProp_t prop{};
        if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return 0;
        int g = prop.multiProcessorCount / NC * NC;
        g_grid = g > 0 ? g : -1;
    }
    return g_grid > 0 ? g_grid : 0;
}

static inline int64_t cdiv64(int64_t a, int64_t b) { return (a + b - 1) / b; }
static inline int chain_kpw(int wfmt) { return wfmt == kChainW32 ? 1 : (wfmt == kChainW16 ? 2 : (wfmt == kChainW8 ? 4 : 8)); }   // k per column of a word
// bytes of staged activations per weight word: kpw bf16 values, or one f32
static inline int chain_xbytes(int wfmt) { return wfmt == kChainW32 ? 4 : chain_kpw(wfmt) * 2; }
static inline int64_t chain_chunks(int64_t k, int wfmt) { return cdiv64(k, chain_kpw(wfmt) * CW); }   // words of a tile
static inline int64_t chain_xs_bytes(int64_t k, int wfmt) { return chain_chunks(k, wfmt) * CW * chain_xbytes(wfmt); }   // staged activations

bool chain_supported(int dtype, int64_t m, int64_t k, int64_t n, bool dual, bool norm, int wfmt, bool x_f32, bool plain) {
    if (m != 1 || k < 4 || n < 4) return false;
    // a width that is not a multiple of 4 (GPT-2's head: 50257): the last tile's missing columns are zero in the copy and are not
    // stored; only for an unquantised layer without bias and residual (staged values and scales come in pairs)
    const bool ragged_ok = plain && !dual && (wfmt == kChainW16 || wfmt == kChainW32);
    if (wfmt < kChainW16 || wfmt > kChainW32) return false;
    if (wfmt == kChainW32) {   // f32 weights, activations and output; no SwiGLU pair
        if (dtype != 0 || dual || k % 4 != 0 || (n % 4 != 0 && !ragged_ok) || k > 4 * (MAXI / 2) * NT) return false;
        return chain_xs_bytes(k, wfmt) / 4 <= kChainMaxXsWords;
    }
    if (dtype != 2) return false;
    if (x_f32 && (!norm || k > 4 * (MAXI / 2) * NT)) return false;
    if (k % 4 != 0 || (n % (dual ? 2 : 4) != 0 && !ragged_ok)) return false;
    if (wfmt == kChainW4 && k % 128 != 0) return false;
    if (norm && k > 4 * MAXI * NT) return false;
    if (chain_xs_bytes(k, wfmt) / 4 > kChainMaxXsWords) return false;
    return true;
}

static ChainOrder chain_order(int64_t k, int64_t n, bool dual, int wfmt) {
    ChainOrder o;
    o.ntiles = cdiv64(dual ? 2 * n : n, 4);
    o.C = chain_chunks(k, wfmt);
    o.grid = chain_grid() > 0 ? chain_grid() : 256;
    o.tlo = o.ntiles / o.grid;
    o.trem = o.ntiles % o.grid;
    return o;
}

size_t chain_weight_bytes(int64_t k, int64_t n, bool dual, int wfmt) { return (size_t)(chain_order(k, n, dual, wfmt).words() * CW * 16); }
int chain_wave_words(int64_t k, int64_t n, bool dual, int wfmt, int blk, int wave, int64_t* out, int most) {
    const ChainOrder o = chain_order(k, n, dual, wfmt);
    int got = 0;
    for (int part = 0; part < 2; ++part) {
        const WavePart p = wave_part(blk, wave, part & 1, (int)o.C, (int)o.tlo, (int)o.trem, (int)o.whole(), (int)o.behind());
        if (p.more == 0) part |= 1;
        int64_t base = p.at;
        for (int left = p.words; left > 0; left -= SW, base += p.run ? (int64_t)SW : o.active() * NWS * SW)
            for (int i = 0; i < (left < SW ? left : SW) && got < most; ++i) out[got++] = base + i;
    }
    return got;
}
int64_t chain_weight_word(int64_t k, int64_t n, bool dual, int wfmt, int64_t tile, int64_t chunk) { return chain_order(k, n, dual, wfmt).word(tile, chunk); }

void chain_pack_weights(hipStream_t s, const void* w, const void* w2, void* out, int64_t k, int64_t n, int wfmt) {
    const ChainOrder o = chain_order(k, n, w2 != nullptr, wfmt);
    const int64_t total = o.ntiles * o.C * 256;
    if (total <= 0) return;
    const unsigned g = (unsigned)std::min<int64_t>(cdiv64(total, 256), 65536);
    if (wfmt == kChainW32)
        chain_pack_f32_kernel<<<g, 256, 0, s>>>((const float*)w, (float*)out, k, n, o);
    else if (wfmt == kChainW16)
        chain_pack_kernel<<<g, 256, 0, s>>>((const bf16_t*)w, (const bf16_t*)w2, (uint32_t*)out, k, n, o);
    else
        chain_pack_codes_kernel<<<g, 256, 0, s>>>((const uint8_t*)w, (const uint8_t*)w2, (uint32_t*)out, wfmt == kChainW8 ? k : k / 2, n, o,
                                                  wfmt == kChainW8 ? 0x80u : 0x88u);
}

void chain_unpack_weights(hipStream_t s, const void* packed, void* w, void* w2, int64_t k, int64_t n, bool dual) {
    const int64_t total = (k + 1) / 2 * n;
    if (total <= 0) return;
    const ChainOrder o = chain_order(k, n, dual, kChainW16);
    const unsigned g = (unsigned)std::min<int64_t>(cdiv64(total, 256), 65536);
    if (w) chain_unpack_kernel<<<g, 256, 0, s>>>((const uint32_t*)packed, (bf16_t*)w, k, n, o, dual ? 1 : 0, 0);
    if (w2) chain_unpack_kernel<<<g, 256, 0, s>>>((const uint32_t*)packed, (bf16_t*)w2, k, n, o, dual ? 1 : 0, 1);
}

size_t chain_scale_bytes(int64_t k, int64_t n, bool dual) {
    return (size_t)(cdiv64(dual ? 2 * n : n, 4) * 4 * chain_chunks(k, kChainW4) * 4 * sizeof(bf16_t));
}

void chain_pack_scales_w4(hipStream_t s, int dtype, const void* sc, const void* sc2, void* out, int64_t k, int64_t n) {
    if (dtype != 2) return;   // the chain only takes bf16 activations and scales
    const int64_t ntiles = cdiv64(sc2 ? 2 * n : n, 4), G = 4 * chain_chunks(k, kChainW4);
    const int64_t total = ntiles * G * 4;
    if (total <= 0) return;
    const unsigned g = (unsigned)std::min<int64_t>(cdiv64(total, 256), 65536);
    chain_pack_scales_kernel<<<g, 256, 0, s>>>((const bf16_t*)sc, (const bf16_t*)sc2, (bf16_t*)out, k / 128, n, G, ntiles);
}

bool chain_fill_phase(ChainPhase& p, int64_t k, int64_t n, bool dual, int wfmt) {
    const ChainOrder o = chain_order(k, n, dual, wfmt);
    const int64_t most = o.tlo + (o.trem > 0 ? 1 : 0);   // tiles of a workgroup
    p.K = (int)k;
    p.N = (int)n;
    p.C = (int)o.C;
    p.tlo = (int)o.tlo;
    p.trem = (int)o.trem;
    p.whole = (int)o.whole();
    p.behind = (int)o.behind();
    p.step_bytes = (int)(o.active() * SLOT_BYTES);
    p.inv_c = 1.0f / (float)o.C;
    p.kind = kChainLinear;
    p.wfmt = wfmt;
    p.lds_bytes = (int)chain_xs_bytes(k, wfmt);
    // int4: the workgroup's group scales (8 bytes per tile and group) are staged behind the activations
    const int64_t total = p.lds_bytes + (wfmt == kChainW4 ? most * 4 * o.C * 8 : 0);
    p.lds_total = (int)std::min<int64_t>(total, INT32_MAX);
    if (dual) p.flags |= kChainDual;
    return most * (dual ? 2 : 4) <= EPI_MAX && most * o.C < (1 << 22) && total <= (int64_t)kChainMaxXsWords * 4;
}

bool chain_attn_supported(int dtype, int64_t t, int64_t n_q, int64_t n_kv, int64_t head_dim, int64_t rot_half) {
    static const bool enabled = [] { const char* e = getenv("GPTRS_HIP_CHAIN_ATTN"); return !(e && e[0] == '0'); }();
    if (!enabled) return false;   // GPTRS_HIP_CHAIN_ATTN=0: decode attention keeps its stand-alone kernels
    if ((dtype != 2 && dtype != 0) || t != 1 || n_kv <= 0 || n_q % n_kv != 0) return false;
    if (dtype == 0 && rot_half != 0) return false;   // f32 rows: no RoPE inside the phase
    const int64_t g = n_q / n_kv;
    if (g != 1 && g != 2 && g != 4 && g != 8) return false;
    if (head_dim != 64 && head_dim != 128 && head_dim != 256) return false;
    if (rot_half != 0 && (rot_half % 8 != 0 || 2 * rot_half > head_dim)) return false;
    return chain_grid() > 0;
}
static int chain_attn_nch(int64_t n_kv) {
    const int64_t n = chain_grid() / n_kv;
    return (int)(n < 1 ? 1 : (n > 64 ? 64 : n));
}
size_t chain_attn_part_bytes(int64_t n_q, int64_t n_kv, int64_t head_dim) {
    return (size_t)n_q * (size_t)chain_attn_nch(n_kv) * (size_t)(head_dim + 2) * sizeof(float);
}
int chain_attn_phases(int64_t capacity) { return capacity <= 128 ? 1 : 2; }
void chain_fill_attn(ChainPhase& partial, ChainPhase& combine, int64_t n_q, int64_t n_kv, int64_t head_dim, int64_t capacity,
                     int64_t rot_half, float scale) {
    const bool single = chain_attn_phases(capacity) == 1;
    const int nch = single ? 1 : chain_attn_nch(n_kv);
    if (single) partial.flags |= kChainAttnFinal;
    for (ChainPhase* p : {&partial, &combine}) {
        p->n_q = (int)n_q; p->n_kv = (int)n_kv; p->head_dim = (int)head_dim; p->capacity = (int)capacity;
        p->rot_half = (int)rot_half; p->nch = nch; p->scale = scale;
    }
    partial.kind = kChainAttnPartial;
    partial.units = (int)n_kv * nch;
    partial.lds_bytes = partial.lds_total = (int)((2 * NWS + NWS * head_dim) * sizeof(float));
    combine.kind = kChainAttnCombine;
    combine.units = (int)n_q;
    combine.lds_bytes = combine.lds_total = (int)(NWS * 64 * sizeof(float4));
}

bool chain_chunk_attn_supported(int64_t n_q, int64_t n_kv, int64_t dim, int64_t vdim, int64_t rot) {
    return dim == vdim && rot % 8 == 0 && rot <= dim && chain_attn_supported(2, 1, n_q, n_kv, dim, 0);
}
void chain_fill_chunk_attn(ChainPhase& partial, ChainPhase& combine, int64_t n_q, int64_t n_kv, int64_t dim, int64_t capacity, int64_t rot, int64_t chunk, float scale, float eps) {
    chain_fill_attn(partial, combine, n_q, n_kv, dim, std::max<int64_t>(capacity, 129), rot / 2, scale);   // (two phases whatever the capacity: the merge adds the sink)
    for (ChainPhase* p : {&partial, &combine}) {
        p->capacity = (int)capacity;
        p->N = chunk > 0 ? (int)std::min<int64_t>(chunk, INT32_MAX) : INT32_MAX;
        p->eps = eps;
    }
}

bool chain_launch(hipStream_t s, const ChainPhase* dev_table, int nphases, int lds_bytes, unsigned* bar, int* abort_flag, int wfmt,
                  int stall_phase, bool chunk_rows) {
    const int grid = chain_grid();
    if (grid <= 0 || nphases <= 0 || nphases > kChainMaxPhases || lds_bytes > kChainMaxXsWords * 4) return false;
    if (wfmt < kChainW16 || wfmt > kChainW32 || (chunk_rows && wfmt != kChainW16)) return false;
    const int xs_bytes = (lds_bytes + 1023) / 1024 * 1024;
    static const int max_depth = [] { const char* e = getenv("GPTRS_HIP_CHAIN_RING"); return e ? std::max(RING_MIN, std::min(RING_MAX, atoi(e))) : RING_MAX; }();
    const int depth = sizeof(Shared) + (size_t)xs_bytes + (size_t)max_depth * SLOT_BYTES <= (size_t)LDS_BYTES ? max_depth : RING_MIN;
    const size_t smem = sizeof(Shared) + (size_t)xs_bytes + (size_t)depth * SLOT_BYTES;
    if (smem > (size_t)LDS_BYTES) return false;
    static_assert(RING_MAX == RING_MIN + 1, "two kernels per weight format");
    const int variant = (chunk_rows ? 4 : wfmt) * 2 + (depth - RING_MIN);
    typedef void (*Kernel)(const ChainPhase*, int, unsigned*, int*, int, unsigned long long, int);
    static const Kernel kernels[10] = {chain_kernel<kChainW16, RING_MIN>, chain_kernel<kChainW16, RING_MAX>, chain_kernel<kChainW8, RING_MIN>,
                                      chain_kernel<kChainW8, RING_MAX>,  chain_kernel<kChainW4, RING_MIN>,  chain_kernel<kChainW4, RING_MAX>,
                                      chain_kernel<kChainW32, RING_MIN>, chain_kernel<kChainW32, RING_MAX>,
                                       chain_kernel<kChainW16, RING_MIN, kRowsChunk>, chain_kernel<kChainW16, RING_MAX, kRowsChunk>};
    static_assert(kChainW16 == 0 && kChainW8 == 1 && kChainW4 == 2 && kChainW32 == 3, "index of a kernel");
    const Kernel fn = kernels[variant];
    if (g_occupancy_ok[variant] < 0) {
        // The grid barrier needs every workgroup resident at once: one workgroup per CU, grid <= CUs (chain_grid), and the
        // kernel with the LDS it asks for must fit a CU.  Checked once per kernel.
        int per_cu = 0;
        const bool ok = hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES) == hipSuccess &&
                        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)fn, NT, smem) == hipSuccess && per_cu >= 1;
        g_occupancy_ok[variant] = ok ? 1 : 0;
    }
    if (!g_occupancy_ok[variant]) return false;
    // wall-clock budget of a grid-barrier wait, in ticks of the 100 MHz counter (GPTRS_HIP_CHAIN_WAIT_MS, default 50 ms;
    // a stalled test launch gets 2 ms)
    static const unsigned long long budget = [] {
        const char* e = getenv("GPTRS_HIP_CHAIN_WAIT_MS");
        const long ms = e ? atol(e) : 50;
        return (unsigned long long)std::max<long>(1, std::min<long>(ms, 10000)) * 100000ull;
    }();
    const unsigned long long ticks = stall_phase >= 0 ? 200000ull : budget;
    fn<<<grid, NT, smem, s>>>(dev_table, nphases, bar, abort_flag, xs_bytes, ticks, stall_phase);
    return true;
}

}  // namespace k
}  // namespace gptrs
