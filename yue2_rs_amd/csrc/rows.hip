// rows.hip -- the decode-order forward of many rows at once: what a sequence
// of token steps computes (Model::forward_phase over n ids, src/model.rs:
// 469-477, 523-591), bit for bit, with every weight read once per 32 rows
// instead of once per row.
//
// The order spec fixes every f32 sum (oracle: DOT, softmax sum, PV), and all
// of them are fma chains from +0 combined by fixed trees.  The FP32 matrix
// instructions compute exactly that chain: v_mfma_f32_32x32x2_f32 and
// v_mfma_f32_16x16x4_f32 return fma(a[k+1], b[k+1], fma(a[k], b[k], c))
// rounded to nearest even after every step, denormals kept (self-tests 22 and 23
// hold them to the oracle's chain over normal, wide-range and denormal
// operands).  So the
// order is kept on the matrix cores, 32 rows to a weight read.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../../include/yue2_hip.h"
#include "dev_gemv.h"
#include "dev_mem.h"
#include "dev_mfma.h"
#include "kernels.h"
#include "prefill.h"
#include "rows.h"
#include "runtime.h"
#include "y2_math.h"

using namespace y2;

namespace y2 {

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) const y2_u32x4 lds_u32x4;
typedef unsigned int y2_u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x16 mfma_f32_32(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_f32_16(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// The low (sel kSelLo) or high BF16 of a pair as f32, the choice per lane.
constexpr uint32_t kSelLo = 0x01000c0cu, kSelHi = 0x03020c0cu;
__device__ __forceinline__ float bf16_sel(uint32_t pair, uint32_t sel) {
    return u2f(__builtin_amdgcn_perm(0u, pair, sel));
}

// ---- DOT GEMM --------------------------------------------------------------
//
// DOT(a, b, K): chunk c (8 elements) belongs to chain c mod 64; each chain is
// an fma chain over its chunks in ascending order; the 64 chains are added by
// a butterfly over distances 32, 16, 8, 4, 2, 1.
//
// A workgroup of eight waves computes 32 rows of X against 32 rows of W (the
// gate/up pair: 16 gate and the same 16 up rows).  Wave r takes the chains r
// mod 8 -- of every 128-byte line of K (eight chunks) its own 16 bytes -- so
// the operands stay in their row-major layout and each line is staged once.
// Chain r + 8 i has the lines i, i + 8, ...; the wave runs its eight chains
// in the order i = 0, 4, 2, 6, 1, 5, 3, 7 and adds them as they end: the
// butterfly's distances 32, 16 and 8, with at most three pending sums (4 x 16
// registers).  Distances 4, 2 and 1 add the eight waves' sums through LDS.
//
// Bound: the vector and matrix pipes together.  FP32 MFMAs run at 155
// TFLOP/s from registers, but every vector instruction takes its issue time
// from them (the same loop with the two operands of each MFMA unpacked by
// v_perm: 119), and each value is unpacked once.  Measured: 92 TFLOP/s at
// 2048 x 5120 x 3072, 109 at 2048 x 3072 x 8192, 99 on the gate/up pair at
// 2048 x 8192 x 3072, 95 at 517 x 5120 x 3072 (a prompt token by token: 4).
// Tiles of 32 x 64 unpack a quarter less but leave two waves per SIMD, which
// wait together at every barrier: 87, 104, 95 and 80, with the next tile's
// first stages requested while a tile ends as well.  32 x 32 tiles fit two
// workgroups, four waves per SIMD.  They read 8 KB per line and workgroup,
// 16 bytes per clock and CU, from L2: the tile order gives each XCD 16 row
// tiles x 4 column tiles at a time.  Lines go straight to LDS (global_load_lds), two per stage, 16-byte
// units XOR-swizzled by (row >> 1) & 7 so that the operand reads do not
// conflict.  A lane's operand for K step 2 s + half is the half-word `half`
// of dword s: one byte permute with a per-lane selector.
constexpr int kDotT = 32, kDotThreads = 512;
constexpr int kDotStages = 2;                          // in LDS (a power of two; four measured 1 % slower)
constexpr int kDotLine = 2 * kDotT * 64;               // BF16 elements of a staged line: X rows, then W rows
constexpr int kDotLoads = 2 * kDotLine / 8 / kDotThreads;  // 16-byte loads per lane and stage
constexpr size_t kDotLds = (size_t)kDotStages * 2 * kDotLine * 2;
static_assert(kDotLoads * kDotThreads * 8 == 2 * kDotLine, "whole loads per wave");
static_assert(kDotLds >= 8u * kDotT * kDotT * 4, "the waves' sums fit the stages");

// The order in which the lines of K are taken: chains i = 0, 4, 2, 6, 1, 5,
// 3, 7 (bit-reversed), each chain's lines i, i + 8, ... ascending, two to a
// stage (a chain's last stage may hold one).  Lane l gets the first line of
// stages l and l + 64, so that it is one v_readlane in the loop.
constexpr int kDotLines = 256;  // K up to 16384: at most 128 stages
__device__ __forceinline__ int rev3(int i) { return ((i & 1) << 2) | (i & 2) | ((i >> 2) & 1); }
__device__ __forceinline__ int chain_lines(int nl, int ii) { return max(0, (nl - rev3(ii) + 7) >> 3); }
struct StageOrder {
    int v[2], stages;
    __device__ __forceinline__ explicit StageOrder(int nl) {
        int p = threadIdx.x & 63, q = p + 64;
        v[0] = v[1] = stages = 0;
#pragma unroll
        for (int ii = 0; ii < 8; ++ii) {
            const int n = (chain_lines(nl, ii) + 1) >> 1;
            if (p >= 0 && p < n) v[0] = rev3(ii) + 16 * p;
            if (q >= 0 && q < n) v[1] = rev3(ii) + 16 * q;
            p -= n;
            q -= n;
            stages += n;
        }
    }
    __device__ __forceinline__ int first(int s) const {  // s uniform
        return __builtin_amdgcn_readlane(s < 64 ? v[0] : v[1], s & 63);
    }
};

template <int EPI>
__global__ __launch_bounds__(kDotThreads, 4) void dot_gemm_kernel(const GemmArgs g, int mt, int nt) {
    constexpr bool PAIR = EPI == GEPI_SWIGLU_BF16;
    constexpr int TN = PAIR ? kDotT / 2 : kDotT;  // output columns per tile
    extern __shared__ __align__(16) uint16_t gsm[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroup b runs on XCD b mod 8: each XCD takes a contiguous range of
    // tiles, ordered in groups of sixteen row tiles (2 % faster than eight)
    const int tiles = mt * nt, per = gridDim.x >> 3;
    const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int gsize = 16 * nt, grp = tile / gsize, gm = min(16, mt - 16 * grp), in = tile - grp * gsize;
    const int m0 = (16 * grp + in % gm) * kDotT, n0 = (in / gm) * TN;
    const int nl = g.K / kGemmTK;
    // this lane's source row of each of its loads (rows past the matrices
    // read the last one: they only feed outputs that are not stored); load q
    // of a stage takes eight rows of one of its two lines
    const uint16_t* src[kDotLoads];
#pragma unroll
    for (int j = 0; j < kDotLoads; ++j) {
        const int row = ((wave * kDotLoads + j) & 7) * 8 + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        if (row < kDotT) {
            src[j] = g.x + (size_t)min(m0 + row, g.M - 1) * g.ldx + 8 * c;
        } else {
            int r = row - kDotT;
            const uint16_t* w = g.w;
            if (PAIR && r >= TN) {
                w = g.w2;
                r -= TN;
            }
            src[j] = w + (size_t)min(n0 + r, g.N - 1) * g.ldw + 8 * c;
        }
    }
    const StageOrder order(nl);
    const int stages = order.stages;
    auto issue = [&](int stage) {  // (a missing second line: the first again, never used)
        uint16_t* base = gsm + (size_t)(stage & (kDotStages - 1)) * 2 * kDotLine;
        const int l0 = order.first(stage), l1 = l0 + 8 < nl ? l0 + 8 : l0;
#pragma unroll
        for (int j = 0; j < kDotLoads; ++j) {
            const int q = wave * kDotLoads + j, k0 = (q >= 8 ? l1 : l0) * kGemmTK;
            __builtin_amdgcn_global_load_lds((Y2_GLOBAL void*)(src[j] + k0), (lds_void*)(base + q * 512), 16, 0, 0);
        }
    };
    // this wave's chunk of the staged lines
    const int arow = lane & 31;
    const uint32_t aoff = arow * 64 + ((wave ^ ((arow >> 1) & 7)) * 8);  // (rows 32 apart share the swizzle)
    struct Raw {
        y2_u32x4 a, w;
    };
    auto read = [&](int stage, int half) {
        const uint16_t* base = gsm + (size_t)(stage & (kDotStages - 1)) * 2 * kDotLine + half * kDotLine + aoff;
        return Raw{*(lds_u32x4*)(base), *(lds_u32x4*)(base + kDotT * 64)};
    };
    const uint32_t sel = lane < 32 ? kSelLo : kSelHi;
    // one line into a chain's accumulators (first: the chain starts at +0)
    auto multiply = [&](const Raw& r, f32x16& acc, bool first) {
        f32x16 zero;
#pragma unroll
        for (int i = 0; i < 16; ++i) zero[i] = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            acc = mfma_f32_32(bf16_sel(r.a[e], sel), bf16_sel(r.w[e], sel), first && e == 0 ? zero : acc);
    };
    const int pre = min(stages, kDotStages);
    for (int s = 0; s < pre; ++s) issue(s);
    if (pre == kDotStages) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kDotStages - 1) * kDotLoads) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    Raw r0 = read(0, 0);
    int s = 0;
    auto stage_step = [&](f32x16& acc, bool first, bool both) {
        const Raw r1 = read(s, 1);
        multiply(r0, acc, first);
        ++s;
        if (s < stages) {
            // stage s has landed (its loads are older than those of the later
            // stages in flight) and every wave has read stage s - 1, whose
            // buffer takes the next one
            if (s - 1 + kDotStages <= stages)
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kDotStages - 2) * kDotLoads) : "memory");
            else
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            asm volatile("s_barrier" ::: "memory");
            if (s - 1 + kDotStages < stages) issue(s - 1 + kDotStages);
            r0 = read(s, 0);
        }
        if (both) multiply(r1, acc, false);
    };
    auto chain = [&](int ii, f32x16& acc) {
        const int n = chain_lines(nl, ii);
        if (n == 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
            return;
        }
        stage_step(acc, true, n > 1);
#pragma unroll 1
        for (int l = 2; l < n; l += 2) stage_step(acc, false, l + 1 < n);
    };
    // the chains as they end: distances 32, 16, 8
    f32x16 acc, c0, c1, c2;
#pragma unroll 1
    for (int pair = 0; pair < 4; ++pair) {
        chain(2 * pair, c0);
        chain(2 * pair + 1, acc);
        acc = c0 + acc;
        if (pair & 1) {
            acc = c1 + acc;
            if (pair & 2) acc = c2 + acc;
            else c2 = acc;
        } else {
            c1 = acc;
        }
    }
    // distances 4, 2, 1 across the waves
    const int orow = tid >> 4, ocol = tid & 15;
    float cur[2];
    if constexpr (EPI == GEPI_RESID) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
            cur[c] = g.c[(size_t)min(m0 + orow, g.M - 1) * g.ldc + min(n0 + ocol + 16 * c, g.N - 1)];
    }
    __syncthreads();  // every wave has read the last stage
    // (rows 4-7 mod 8 trade places with their neighbours: the two lane
    // halves' stores then fall in different banks)
    float* ps = reinterpret_cast<float*>(gsm);
    auto place = [](int row) { return (row ^ ((row >> 2) & 1)) * kDotT; };
#pragma unroll
    for (int r = 0; r < 16; ++r)
        ps[wave * kDotT * kDotT + place(acc32_row(lane, r)) + acc32_col(lane)] = acc[r];
    __syncthreads();
    auto total = [&](int c) {
        float p[8];
#pragma unroll
        for (int w = 0; w < 8; ++w) p[w] = ps[w * kDotT * kDotT + place(orow) + c];
        return ((p[0] + p[4]) + (p[2] + p[6])) + ((p[1] + p[5]) + (p[3] + p[7]));
    };
    if (m0 + orow >= g.M) return;
    const size_t at = (size_t)(m0 + orow) * g.ldc + n0 + ocol;
    if constexpr (PAIR) {
        if (n0 + ocol < g.N) g.cb[at] = bf16_bits(rb(silu_rb(rb(total(ocol))) * rb(total(ocol + 16))));
    } else {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if (n0 + ocol + 16 * c >= g.N) continue;
            const float v = total(ocol + 16 * c);
            g.c[at + 16 * c] = EPI == GEPI_RESID ? rb(cur[c] + rb(v)) : rb(v);
        }
    }
}

template <int EPI>
static hipError_t launch_dot_t(hipStream_t s, const GemmArgs& g) {
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&dot_gemm_kernel<EPI>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)kDotLds);
    if (attr != hipSuccess) return attr;
    const int tn = EPI == GEPI_SWIGLU_BF16 ? kDotT / 2 : kDotT;
    const int mt = (g.M + kDotT - 1) / kDotT, nt = (g.N + tn - 1) / tn;
    dot_gemm_kernel<EPI><<<(mt * nt + 7) / 8 * 8, kDotThreads, kDotLds, s>>>(g, mt, nt);
    return hipGetLastError();
}

hipError_t launch_dot_gemm(hipStream_t s, int epi, const GemmArgs& g) {
    if (g.K < kGemmTK || g.K % kGemmTK || g.K > kDotLines * kGemmTK || g.ldx % 8 || g.ldw % 8 || g.M < 1 || g.N < 1)
        return hipErrorInvalidValue;
    if (((uintptr_t)g.x | (uintptr_t)g.w | (uintptr_t)g.w2) & 15) return hipErrorInvalidValue;
    if (epi == GEPI_SWIGLU_BF16 && !g.w2) return hipErrorInvalidValue;
    switch (epi) {
        case GEPI_ROUND: return launch_dot_t<GEPI_ROUND>(s, g);
        case GEPI_RESID: return launch_dot_t<GEPI_RESID>(s, g);
        case GEPI_SWIGLU_BF16: return launch_dot_t<GEPI_SWIGLU_BF16>(s, g);
        default: return hipErrorInvalidValue;
    }
}

// ---- attention -------------------------------------------------------------
//
// The exact softmax normalises by the global maximum and the global sum
// before PV, so the keys are walked three times: maxima, sums (both in
// rows_stats_kernel), then p = e / total and PV (rows_pv_kernel), the scores
// recomputed each time (an f32 score matrix costs as much to write and read
// back, and grows with the square of the context).
//
// Two forms.  Up to kLongKeys keys, and for few rows, the four waves of a
// workgroup share 16 queries (share_*_kernel); for many rows of a longer
// context a workgroup takes 128 rows, a wave 16 of them alone (rows_*_kernel).
// Prompts of two layers through either, ms: 3B class 9.95 against 10.29 at
// 2048 tokens, 37.3 / 38.4 at 6000, 98.4 / 95.7 at 12000, 244 / 215 at 20000
// (the block sums of 313 blocks leave the shared statistics one workgroup per
// CU); a 1B class 6.64 / 6.75, 24.8 / 25.6, 68.5 / 70.2, 108 / 112 at 16000.
// 517 tokens of the YuE2 shape, per layer: 81 us against 236.
//
// The scores are computed transposed, S^T = K Q^T with 16x16x4 MFMAs: lane l has
// query l % 16 and, of the block, keys 16 kt + 4 (l / 16) + r.  A score's
// D / 8 chunk chains (two MFMAs each, from +0) are added as they end, in
// bit-reversed order, which is the butterfly over distances D/16 .. 1.
// PV: stream t of 512 / D takes keys t mod (512 / D) in ascending order.  For
// D = 128 stream r is exactly register r of the score tiles: the four MFMAs
// of kt = 0..3 contract keys 16 kt + 4 j + r in ascending order over j, so P
// feeds the products from the registers it was computed in.  For D = 64 there
// are eight streams, 4 (j & 1) + r: two passes with the other lanes' p zero
// (an fma of zeros leaves a chain that starts at +0 as it is).
//
// Bound: the FP32 MFMAs (4 x 4096 cycles per 16 queries and 64-key block) and
// the vector ALU beside them (unpacking, the trees, the f64 exponentials and
// the divisions: ~6000 cycles), which share their issue time.
constexpr int kRowsQ = 128, kRowsThreads = 512, kRowsWaves = 8, kLongKeys = 255 * kBlockKeys;

template <int D>
__device__ __forceinline__ int key_swz(int key) { return D == 128 ? key & 15 : (key >> 1) & 7; }

// Requests the K rows of block t (keys past last: the last one) into LDS.
template <int D, int NW>
__device__ __forceinline__ void stage_keys(const uint16_t* K, int t, int last, uint16_t* dst) {
    constexpr int U = D / 8, LPW = kBlockKeys * U / (64 * NW);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
        const int q = wave * LPW + j, u = q * 64 + lane, key = u / U, c = (u % U) ^ key_swz<D>(key);
        __builtin_amdgcn_global_load_lds((Y2_GLOBAL void*)(K + (size_t)min(t * kBlockKeys + key, last) * D + 8 * c),
                                         (lds_void*)(dst + q * 512), 16, 0, 0);
    }
}

// V of block t (keys past last: the last one) through registers, transposed, to
// LDS by the NT threads of a workgroup: a unit is a key pair x 8 dims.
template <int D, int NT>
struct ValueStage {
    static constexpr int UNITS = kBlockKeys / 2 * (D / 8), PER = (UNITS + NT - 1) / NT;
    uint4 a[PER], b[PER];
    __device__ __forceinline__ void load(const uint16_t* V, int t, int last) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int u = threadIdx.x + NT * i, k = t * kBlockKeys + 2 * (u % (kBlockKeys / 2));
            const int vd = u / (kBlockKeys / 2) * 8;
            if (UNITS % NT && u >= UNITS) continue;
            a[i] = ldg4(V + (size_t)min(k, last) * D + vd);
            b[i] = ldg4(V + (size_t)min(k + 1, last) * D + vd);
        }
    }
    // row = dim, key 16 kt + 4 j + r at 16 j + 4 kt + r (a lane's keys are 16
    // consecutive halfwords), 16-byte units swizzled
    __device__ __forceinline__ void store(uint16_t* vt) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int u = threadIdx.x + NT * i, vd = u / (kBlockKeys / 2) * 8;
            if (UNITS % NT && u >= UNITS) continue;
            const int k = 2 * (u % (kBlockKeys / 2)), unit = 2 * ((k >> 2) & 3) + (k >> 5), at = ((k >> 4) & 1) * 4 + (k & 3);
            const uint32_t x[4] = {a[i].x, a[i].y, a[i].z, a[i].w}, y[4] = {b[i].x, b[i].y, b[i].z, b[i].w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int d = vd + e;
                const uint32_t w = e & 1 ? (x[e >> 1] >> 16) | (y[e >> 1] & 0xffff0000u)
                                         : (x[e >> 1] & 0xffffu) | (y[e >> 1] << 16);
                *reinterpret_cast<uint32_t*>(&vt[d * kBlockKeys + ((unit ^ ((d >> 1) & 7)) << 3) + at]) = w;
            }
        }
    }
};

// This lane's query values: element 8 c + 4 s + j of query l % 16.
template <int D>
__device__ __forceinline__ void load_query(const uint16_t* q, bool in, float (&qf)[D / 8][2]) {
    const int j = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int c = 0; c < D / 8; ++c)
#pragma unroll
        for (int s = 0; s < 2; ++s) qf[c][s] = in ? bf16(gbl(q)[8 * c + 4 * s + j]) : 0.0f;
}

// The DOTs of 32 staged keys (two 16-key tiles) with the wave's queries.
template <int D>
__device__ __forceinline__ void half_scores(const uint16_t* ks, const float (&qf)[D / 8][2], f32x4 (&s)[2]) {
    constexpr int NC = D / 8, LV = D == 128 ? 4 : 3;
    const int lane = threadIdx.x & 63, j = lane >> 4;
    const uint32_t sel = (j & 1) ? kSelHi : kSelLo;
    typedef __attribute__((address_space(3))) const uint32_t lds_u32;
    const int swz = key_swz<D>(lane & 15);
    const uint16_t* row = ks + (lane & 15) * D + (j >> 1) * 2;
    f32x4 st[LV][2];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ci = 0; ci < NC; ++ci) {
        int c = 0;  // bit-reversed ci
#pragma unroll
        for (int b = 0; b < LV; ++b) c |= ((ci >> b) & 1) << (LV - 1 - b);
        const uint16_t* at = row + ((c ^ swz) << 3);
        f32x4 acc[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t w0 = *(lds_u32*)(at + u * 16 * D), w1 = *(lds_u32*)(at + u * 16 * D + 4);
            const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
            acc[u] = mfma_f32_16(bf16_sel(w0, sel), qf[c][0], zero);
            acc[u] = mfma_f32_16(bf16_sel(w1, sel), qf[c][1], acc[u]);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            bool done = false;
#pragma unroll
            for (int v = 0; v < LV; ++v) {
                if (done) continue;
                if ((ci >> v) & 1) acc[u] = st[v][u] + acc[u];
                else {
                    st[v][u] = acc[u];
                    done = true;
                }
            }
            if (ci == NC - 1) s[u] = acc[u];
        }
    }
}

// The same of 16 staged keys (one tile).
template <int D>
__device__ __forceinline__ void tile_scores(const uint16_t* ks, const float (&qf)[D / 8][2], f32x4& s) {
    constexpr int NC = D / 8;
    const int lane = threadIdx.x & 63, j = lane >> 4;
    const uint32_t sel = (j & 1) ? kSelHi : kSelLo;
    typedef __attribute__((address_space(3))) const uint32_t lds_u32;
    const uint16_t* row = ks + (lane & 15) * D + (j >> 1) * 2;
    f32x4 p[NC];  // the chunk chains, then the butterfly over distances NC / 2 .. 1
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const uint16_t* at = row + ((c ^ key_swz<D>(lane & 15)) << 3);
        const uint32_t w0 = *(lds_u32*)(at), w1 = *(lds_u32*)(at + 4);
        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
        p[c] = mfma_f32_16(bf16_sel(w0, sel), qf[c][0], zero);
        p[c] = mfma_f32_16(bf16_sel(w1, sel), qf[c][1], p[c]);
    }
#pragma unroll
    for (int d = NC / 2; d >= 1; d >>= 1)
#pragma unroll
        for (int c = 0; c < d; ++c) p[c] = p[c] + p[c + d];
    s = p[0];
}

// One block's PV for 16 dims (vrow: this lane's row of the transposed V tile):
// the streams' fma chains over the block's keys, then their butterfly.
template <int D>
__device__ __forceinline__ f32x4 pv_tile(const uint16_t* vrow, const f32x4 (&p)[4]) {
    const int lane = threadIdx.x & 63, j = lane >> 4, swz = (lane & 15) >> 1;
    const y2_u32x4 w0 = *(lds_u32x4*)(vrow + ((2 * j) ^ swz) * 8);
    const y2_u32x4 w1 = *(lds_u32x4*)(vrow + ((2 * j + 1) ^ swz) * 8);
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 acc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float fv[4];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            const uint32_t w = (kt < 2 ? w0 : w1)[(kt & 1) * 2 + (e >> 1)];
            fv[kt] = e & 1 ? bf16_hi(w) : bf16_lo(w);
        }
        if constexpr (D == 128) {
            acc[e] = zero;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) acc[e] = mfma_f32_16(fv[kt], p[kt][e], acc[e]);
        } else {
            f32x4 a0 = zero, a1 = zero;  // streams e and 4 + e
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                a0 = mfma_f32_16(fv[kt], j & 1 ? 0.0f : p[kt][e], a0);
                a1 = mfma_f32_16(fv[kt], j & 1 ? p[kt][e] : 0.0f, a1);
            }
            acc[e] = a0 + a1;
        }
    }
    return (acc[0] + acc[2]) + (acc[1] + acc[3]);
}

// The same over the first `keys` keys of the block alone, on the vector ALU
// (vt: the transposed V tile's first row of these 16 dims).  pv_tile
// multiplies all of the block's keys, those past a query's last one with p =
// 0 and (D = 64) each stream's with 0 in the other's pass, so an infinite or
// NaN value makes NaN of sums that it does not belong to.  What it makes stays
// in the output: the PV kernels walk the blocks a second time, this way, when
// an output is not finite; ordinary values pay for a vote per workgroup and a
// branch per block (2048 tokens, four 3B-class layers: 20.09 -> 20.18 ms).
template <int D>
__device__ __forceinline__ f32x4 pv_exact(const uint16_t* vt, const f32x4 (&p)[4], int keys) {
    constexpr int SETS = D == 64 ? 2 : 1;  // streams e (and 4 + e): keys 16 kt + 4 j + e of every (second) j
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));  // (its addresses are not kept in registers from block to block)
    const int d0 = (lane >> 4) * 4;
    f32x4 part[2];
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int e2 = 0; e2 < 4; e2 += 2) {
            const int e = e2 + half;
            f32x4 sum;
#pragma unroll
            for (int set = 0; set < SETS; ++set) {
                f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) {
                    const float mine = half ? p[kt][e2 + 1] : p[kt][e2];
#pragma unroll
                    for (int j = set; j < 4; j += SETS) {
                        const float pk = __shfl(mine, (lane & 15) + 16 * j);
                        const bool in = 16 * kt + 4 * j + e < keys;
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int d = d0 + r, unit = (2 * j + (kt >> 1)) ^ ((d >> 1) & 7);
                            const float v = bf16(vt[d * kBlockKeys + unit * 8 + (kt & 1) * 4 + e]);
                            acc[r] = in ? __builtin_fmaf(v, pk, acc[r]) : acc[r];
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                sum = set ? sum + acc : acc;
            }
            part[1] = e2 ? part[1] + sum : sum;
        }
        if (half == 0) part[0] = part[1];
    }
    return part[0] + part[1];
}

__device__ __forceinline__ bool finite(const f32x4& v) {
    bool ok = true;
#pragma unroll
    for (int e = 0; e < 4; ++e) ok = ok && __builtin_fabsf(v[e]) <= 3.402823466e38f;
    return ok;
}

// Whether v holds anywhere in a workgroup of NW waves; lds: NW words that no
// wave uses between this call's barriers and the next one.
template <int NW>
__device__ __forceinline__ bool any_wave(bool v, uint16_t* lds) {
    int* votes = reinterpret_cast<int*>(lds);
    const bool mine = __builtin_amdgcn_ballot_w64(v) != 0;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) votes[threadIdx.x >> 6] = mine;
    __syncthreads();
    int any = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) any |= votes[w];
    return any != 0;
}

// The DOTs of a block's 64 keys.
template <int D>
__device__ __forceinline__ void block_scores(const uint16_t* ks, const float (&qf)[D / 8][2], f32x4 (&s)[4]) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        f32x4 t[2];
        half_scores<D>(ks + half * 32 * D, qf, t);
        s[2 * half] = t[0];
        s[2 * half + 1] = t[1];
    }
}

// expf_cr (y2_math.h) of an argument at most 0, without its branches (they
// would end the interleaving of a lane's sixteen exponentials): the same
// operations, the scaling by 2^n through v_ldexp_f64 (exact in f64), and 0
// below -104.  NaN stays NaN.
__device__ __forceinline__ float exp_nonpos(float xf) {
    const double x = (double)(xf < -104.0f ? -104.0f : xf);
    const double n = __builtin_rint(x * 0x1.71547652b82fep+0);
    double r = __builtin_fma(-n, 0x1.62e42fefa3800p-1, x);
    r = __builtin_fma(-n, 0x1.ef35793c76730p-45, r);
    double p = 0x1.6124613a86d09p-33;
    p = __builtin_fma(p, r, 0x1.1eed8eff8d898p-29);
    p = __builtin_fma(p, r, 0x1.ae64567f544e4p-26);
    p = __builtin_fma(p, r, 0x1.27e4fb7789f5cp-22);
    p = __builtin_fma(p, r, 0x1.71de3a556c734p-19);
    p = __builtin_fma(p, r, 0x1.a01a01a01a01ap-16);
    p = __builtin_fma(p, r, 0x1.a01a01a01a01ap-13);
    p = __builtin_fma(p, r, 0x1.6c16c16c16c17p-10);
    p = __builtin_fma(p, r, 0x1.1111111111111p-7);
    p = __builtin_fma(p, r, 0x1.5555555555555p-5);
    p = __builtin_fma(p, r, 0x1.5555555555555p-3);
    p = __builtin_fma(p, r, 0x1.0000000000000p-1);
    p = __builtin_fma(p, r, 1.0);
    p = __builtin_fma(p, r, 1.0);
    const float e = (float)__builtin_ldexp(p, (int)n);
    return xf < -104.0f ? 0.0f : e;
}

struct RowsQuery {
    int h, g, q0, qrow, qpos, wave_first, wave_last, tiles;
    bool in;
};
__device__ __forceinline__ RowsQuery rows_query(const FlashArgs& f) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    RowsQuery r;
    r.h = blockIdx.x;
    r.g = r.h / (f.heads / f.kv_heads);
    r.q0 = (gridDim.y - 1 - blockIdx.y) * kRowsQ;  // the blocks with the most keys first
    r.qrow = r.q0 + wave * 16 + (threadIdx.x & 15);
    r.in = r.qrow < f.rows;
    r.qpos = f.p0 + r.qrow;
    r.wave_first = f.p0 + r.q0 + wave * 16;
    r.wave_last = r.q0 + wave * 16 < f.rows ? min(r.wave_first + 15, f.p0 + f.rows - 1) : -1;
    r.tiles = (min(f.p0 + r.q0 + kRowsQ, f.p0 + f.rows) + kBlockKeys - 1) / kBlockKeys;
    return r;
}

// Contexts past kLongKeys (256 blocks), whose blocks are added in pairs
// (super-blocks of 2): blocks are taken two at a time, a last odd one with an
// empty partner.  A row of fewer blocks beside a longer one adds them singly.
template <int D>
__global__ __launch_bounds__(kRowsThreads, 2) void rows_stats_kernel(const FlashArgs f, float2* stats) {
    __shared__ __align__(16) uint16_t ks[2][kBlockKeys * D];
    const RowsQuery r = rows_query(f);
    const int j = (threadIdx.x & 63) >> 4, last = f.p0 + f.rows - 1;
    const uint16_t* K = f.kv_base + (((size_t)f.layer * 2) * f.kv_heads + r.g) * (size_t)f.cap * D;
    float qf[D / 8][2];
    load_query<D>(f.q + ((size_t)min(r.qrow, f.rows - 1) * f.heads + r.h) * D, r.in, qf);
    const int tiles = (r.tiles + 1) & ~1;
    const bool two = (r.qpos + kBlockKeys) / kBlockKeys >= 256;
    float m = -__builtin_huge_valf(), total = 0.0f, part = 0.0f;
    stage_keys<D, kRowsWaves>(K, 0, last, ks[0]);
    for (int it = 0; it < 2 * tiles; ++it) {
        const bool sums = it >= tiles;
        const int t = sums ? it - tiles : it, kb = t * kBlockKeys;
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        asm volatile("s_barrier" ::: "memory");  // block t is staged, block t - 1 read by every wave
        if (it + 1 < 2 * tiles) stage_keys<D, kRowsWaves>(K, it + 1 < tiles ? it + 1 : it + 1 - tiles, last, ks[(it + 1) & 1]);
        if (it == tiles) m = xor_max<32, 16>(m) * f.scale;  // the scaled maximum (rounding is monotonic)
        float u = 0.0f;
        if (kb <= r.wave_last) {
            f32x4 s[4];
            block_scores<D>(ks[it & 1], qf, s);
            const bool masked = kb + kBlockKeys - 1 > r.wave_first;
            if (!sums) {
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (!masked || kb + kt * 16 + 4 * j + e <= r.qpos) m = fmaxf(m, s[kt][e]);
                continue;
            }
            // the butterfly over the block's keys: distances 32 and 16 are
            // tiles, 8 and 4 lane groups, 2 and 1 registers
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x = exp_nonpos(s[kt][e] * f.scale - m);
                    s[kt][e] = !masked || kb + kt * 16 + 4 * j + e <= r.qpos ? x : 0.0f;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = xor_sum<32, 16>((s[0][e] + s[2][e]) + (s[1][e] + s[3][e]));
            u = (v[0] + v[2]) + (v[1] + v[3]);
        }
        if (!sums) continue;
        if (t & 1) {
            const float pair = part + u;
            total = t == 1 ? pair : two ? total + pair : (total + part) + u;
        } else {
            part = u;
        }
    }
    if (r.in && j == 0) stats[(size_t)r.qrow * f.heads + r.h] = make_float2(m, total);
}

template <int D>
__global__ __launch_bounds__(kRowsThreads, 2) void rows_pv_kernel(const FlashArgs f, const float2* stats) {
    __shared__ __align__(16) uint16_t ks[2][kBlockKeys * D];
    __shared__ __align__(16) uint16_t vt[2][D * kBlockKeys];
    const RowsQuery r = rows_query(f);
    const int tid = threadIdx.x, lane = tid & 63, j = lane >> 4, last = f.p0 + f.rows - 1;
    const uint16_t* K = f.kv_base + (((size_t)f.layer * 2) * f.kv_heads + r.g) * (size_t)f.cap * D;
    const uint16_t* V = f.kv_base + (((size_t)f.layer * 2 + 1) * f.kv_heads + r.g) * (size_t)f.cap * D;
    float qf[D / 8][2];
    load_query<D>(f.q + ((size_t)min(r.qrow, f.rows - 1) * f.heads + r.h) * D, r.in, qf);
    const float2 mt = r.in ? stats[(size_t)r.qrow * f.heads + r.h] : make_float2(0.0f, 1.0f);
    const int tiles = (r.tiles + 1) & ~1;
    const bool two = (r.qpos + kBlockKeys) / kBlockKeys >= 256;
    f32x4 o[D / 16], pend[D / 16];
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt) o[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    ValueStage<D, kRowsThreads> values;
    for (bool exact = false;; exact = true) {
        stage_keys<D, kRowsWaves>(K, 0, last, ks[0]);
        values.load(V, 0, last);
        for (int t = 0; t < tiles; ++t) {
            const int kb = t * kBlockKeys, buf = t & 1;
            values.store(vt[buf]);
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            asm volatile("s_barrier" ::: "memory");  // block t is staged, block t - 1 read by every wave
            if (t + 1 < tiles) {
                stage_keys<D, kRowsWaves>(K, t + 1, last, ks[buf ^ 1]);
                values.load(V, t + 1, last);
            }
            const bool live = kb <= r.wave_last;
            f32x4 p[4];
            if (live) {
                block_scores<D>(ks[buf], qf, p);
                const bool masked = kb + kBlockKeys - 1 > r.wave_first;
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float x = exp_nonpos(p[kt][e] * f.scale - mt.x) / mt.y;
                        p[kt][e] = !masked || kb + kt * 16 + 4 * j + e <= r.qpos ? x : 0.0f;
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int dt = 0; dt < D / 16; ++dt) {
                f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
                if (__builtin_expect(exact, false)) {
                    if (live) v = pv_exact<D>(&vt[buf][dt * 16 * kBlockKeys], p, r.qpos + 1 - kb);
                } else {
                    if (live) v = pv_tile<D>(&vt[buf][(dt * 16 + (lane & 15)) * kBlockKeys], p);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (t & 1) {
                    const f32x4 pair = pend[dt] + v, a = o[dt] + pair, b = (o[dt] + pend[dt]) + v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[dt][e] = t == 1 ? pair[e] : two ? a[e] : b[e];
                } else {
                    pend[dt] = v;
                }
            }
        }
        bool ok = true;
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) ok = ok && finite(o[dt]);
        if (exact || !any_wave<kRowsWaves>(r.in && !ok, vt[1])) break;
    }
    if (r.in) {
        uint16_t* orow = f.out + ((size_t)r.qrow * f.heads + r.h) * D + 4 * j;
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) {
            const uint32_t w0 = (uint32_t)bf16_bits(rb(o[dt][0])) | ((uint32_t)bf16_bits(rb(o[dt][1])) << 16);
            const uint32_t w1 = (uint32_t)bf16_bits(rb(o[dt][2])) | ((uint32_t)bf16_bits(rb(o[dt][3])) << 16);
            *reinterpret_cast<uint2*>(orow + dt * 16) = make_uint2(w0, w1);
        }
    }
}

// The four waves of a workgroup share 16 queries.  A wave of the kernels above
// walks every key block of its queries alone, ~6 us a block in each kernel.
// Here the statistics' blocks are dealt to the waves (maxima and block sums are exchanged through LDS, the
// sums added in block order at the end), and of each PV block a wave computes
// the p of 16 keys and, from everyone's p in LDS, a quarter of the dimensions.
constexpr int kShareWaves = 4, kShareThreads = 64 * kShareWaves;

// LDS of the statistics: each wave's two half-blocks of keys, the block sums.
template <int D>
constexpr size_t share_stats_lds(int tiles) {
    return (size_t)kShareWaves * 2 * 32 * D * 2 + (size_t)tiles * 16 * 4;
}

template <int D, bool LONG>
__global__ __launch_bounds__(kShareThreads, 2) void share_stats_kernel(const FlashArgs f, float2* stats) {
    extern __shared__ __align__(16) uint16_t sm[];
    __shared__ float mx[kShareWaves][16];
    constexpr int U = D / 8, LPH = 32 * U / 64;  // wave loads of a half-block
    const int lane = threadIdx.x & 63, j = lane >> 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = blockIdx.x, g = h / (f.heads / f.kv_heads), q0 = (gridDim.y - 1 - blockIdx.y) * 16;
    const int qrow = q0 + (lane & 15), qpos = f.p0 + qrow, first = f.p0 + q0, last = f.p0 + f.rows - 1;
    const bool in = qrow < f.rows;
    const int tiles = (min(first + 16, f.p0 + f.rows) + kBlockKeys - 1) / kBlockKeys;
    const uint16_t* K = f.kv_base + (((size_t)f.layer * 2) * f.kv_heads + g) * (size_t)f.cap * D;
    uint16_t* ks = sm + wave * 2 * 32 * D;
    float* us = reinterpret_cast<float*>(sm + kShareWaves * 2 * 32 * D);  // [tile][query]
    float qf[D / 8][2];
    load_query<D>(f.q + ((size_t)min(qrow, f.rows - 1) * f.heads + h) * D, in, qf);
    auto stage = [&](int t, int half) {
#pragma unroll
        for (int i = 0; i < LPH; ++i) {
            const int u = i * 64 + lane, key = u / U, c = (u % U) ^ key_swz<D>(key);
            __builtin_amdgcn_global_load_lds(
                (Y2_GLOBAL void*)(K + (size_t)min(t * kBlockKeys + half * 32 + key, last) * D + 8 * c),
                (lds_void*)(ks + half * 32 * D + i * 512), 16, 0, 0);
        }
    };
    const int mine = tiles > wave ? (tiles - wave + kShareWaves - 1) / kShareWaves : 0;  // tiles wave, wave + 4, ..
    float m = -__builtin_huge_valf();
    for (int pass = 0; pass < 2; ++pass) {
        if (mine > 0) stage(wave, 0);
        for (int i = 0; i < mine; ++i) {
            const int t = wave + kShareWaves * i, kb = t * kBlockKeys;
            const bool masked = kb + kBlockKeys - 1 > first;
            f32x4 s[4];
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                // this half has landed, the other one's reads are done
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                if (half == 0) stage(t, 1);
                else if (i + 1 < mine) stage(t + kShareWaves, 0);
                f32x4 v[2];
                half_scores<D>(ks + half * 32 * D, qf, v);
                s[2 * half] = v[0];
                s[2 * half + 1] = v[1];
            }
            if (pass == 0) {
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (!masked || kb + kt * 16 + 4 * j + e <= qpos) m = fmaxf(m, s[kt][e]);
                continue;
            }
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x = exp_nonpos(s[kt][e] * f.scale - m);
                    s[kt][e] = !masked || kb + kt * 16 + 4 * j + e <= qpos ? x : 0.0f;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = xor_sum<32, 16>((s[0][e] + s[2][e]) + (s[1][e] + s[3][e]));
            if (j == 0) us[t * 16 + (lane & 15)] = (v[0] + v[2]) + (v[1] + v[3]);
        }
        if (pass == 0) {
            m = xor_max<32, 16>(m);
            if (j == 0) mx[wave][lane & 15] = m;
            __syncthreads();
            m = mx[0][lane & 15];
#pragma unroll
            for (int w = 1; w < kShareWaves; ++w) m = fmaxf(m, mx[w][lane & 15]);
            m = m * f.scale;  // the scaled maximum (rounding is monotonic)
        }
    }
    __syncthreads();
    if (threadIdx.x < 16 && in) {
        const int nb = (qpos + kBlockKeys) / kBlockKeys;
        const bool two = LONG && nb >= 256;
        float total = us[lane];
        if (two) {
            total = us[lane] + us[16 + lane];
            for (int t = 2; t < nb; t += 2) total = total + (t + 1 < nb ? us[t * 16 + lane] + us[t * 16 + 16 + lane] : us[t * 16 + lane]);
        } else {
            for (int t = 1; t < nb; ++t) total = total + us[t * 16 + lane];
        }
        stats[(size_t)qrow * f.heads + h] = make_float2(m, total);
    }
}

template <int D, bool LONG>
__global__ __launch_bounds__(kShareThreads, D == 64 && !LONG ? 4 : 2) void share_pv_kernel(const FlashArgs f, const float2* stats) {
    constexpr int DW = D / 16 / kShareWaves;  // 16-dim tiles per wave
    static_assert(DW >= 1, "whole tiles");
    __shared__ __align__(16) uint16_t ks[2][kBlockKeys * D];
    __shared__ __align__(16) uint16_t vt[2][D * kBlockKeys];
    __shared__ __align__(16) f32x4 ps[2][kShareWaves][64];    // p of keys 16 kt + 4 j .. + 3, wave kt's lane
    const int tid = threadIdx.x, lane = tid & 63, j = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = blockIdx.x, g = h / (f.heads / f.kv_heads), q0 = (gridDim.y - 1 - blockIdx.y) * 16;
    const int qrow = q0 + (lane & 15), qpos = f.p0 + qrow, last = f.p0 + f.rows - 1;
    const bool in = qrow < f.rows;
    const int nt = (min(f.p0 + q0 + 16, f.p0 + f.rows) + kBlockKeys - 1) / kBlockKeys, tiles = LONG ? (nt + 1) & ~1 : nt;
    const bool two = LONG && (qpos + kBlockKeys) / kBlockKeys >= 256;
    const uint16_t* K = f.kv_base + (((size_t)f.layer * 2) * f.kv_heads + g) * (size_t)f.cap * D;
    const uint16_t* V = f.kv_base + (((size_t)f.layer * 2 + 1) * f.kv_heads + g) * (size_t)f.cap * D;
    float qf[D / 8][2];
    load_query<D>(f.q + ((size_t)min(qrow, f.rows - 1) * f.heads + h) * D, in, qf);
    const float2 mt = in ? stats[(size_t)qrow * f.heads + h] : make_float2(0.0f, 1.0f);
    f32x4 o[DW], pend[DW];
#pragma unroll
    for (int d = 0; d < DW; ++d) o[d] = pend[d] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    ValueStage<D, kShareThreads> values;
    for (bool exact = false;; exact = true) {
        stage_keys<D, kShareWaves>(K, 0, last, ks[0]);
        values.load(V, 0, last);
        for (int t = 0; t < tiles; ++t) {
            const int kb = t * kBlockKeys, buf = t & 1;
            values.store(vt[buf]);
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            asm volatile("s_barrier" ::: "memory");  // block t is staged; block t - 1's scores and p are read
            if (t + 1 < tiles) {
                stage_keys<D, kShareWaves>(K, t + 1, last, ks[buf ^ 1]);
                values.load(V, t + 1, last);
            }
            {
                // the p of this wave's 16 keys (one tile of a half-block's two: the other is another wave's)
                f32x4 s;
                tile_scores<D>(ks[buf] + wave * 16 * D, qf, s);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x = exp_nonpos(s[e] * f.scale - mt.x) / mt.y;
                    s[e] = kb + wave * 16 + 4 * j + e <= qpos ? x : 0.0f;
                }
                ps[buf][wave][lane] = s;
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            asm volatile("s_barrier" ::: "memory");  // every wave's p (the next block's loads stay in flight)
            f32x4 p[4];
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) p[kt] = ps[buf][kt][lane];
            f32x4 vs[DW];
            if (__builtin_expect(exact, false)) {
#pragma unroll
                for (int d = 0; d < DW; ++d) vs[d] = pv_exact<D>(&vt[buf][(wave * DW + d) * 16 * kBlockKeys], p, qpos + 1 - kb);
            } else {
#pragma unroll
                for (int d = 0; d < DW; ++d) vs[d] = pv_tile<D>(&vt[buf][((wave * DW + d) * 16 + (lane & 15)) * kBlockKeys], p);
            }
#pragma unroll
            for (int d = 0; d < DW; ++d) {
                const f32x4 v = vs[d];
                if constexpr (!LONG) {
                    o[d] = t == 0 ? v : o[d] + v;
                } else if (t & 1) {
                    const f32x4 pair = pend[d] + v, a = o[d] + pair, b = (o[d] + pend[d]) + v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[d][e] = t == 1 ? pair[e] : two ? a[e] : b[e];
                } else {
                    pend[d] = v;
                }
            }
        }
        bool ok = true;
#pragma unroll
        for (int d = 0; d < DW; ++d) ok = ok && finite(o[d]);
        if (exact || !any_wave<kShareWaves>(in && !ok, vt[1])) break;
    }
    if (in) {
        uint16_t* orow = f.out + ((size_t)qrow * f.heads + h) * D + 4 * j;
#pragma unroll
        for (int d = 0; d < DW; ++d) {
            const uint32_t w0 = (uint32_t)bf16_bits(rb(o[d][0])) | ((uint32_t)bf16_bits(rb(o[d][1])) << 16);
            const uint32_t w1 = (uint32_t)bf16_bits(rb(o[d][2])) | ((uint32_t)bf16_bits(rb(o[d][3])) << 16);
            *reinterpret_cast<uint2*>(orow + (wave * DW + d) * 16) = make_uint2(w0, w1);
        }
    }
}

template <int D, bool LONG>
static void rows_attention_t(hipStream_t s, const FlashArgs& f, float2* stats) {
    if (LONG && (long)f.heads * ((f.rows + kRowsQ - 1) / kRowsQ) >= 256) {
        const dim3 grid(f.heads, (f.rows + kRowsQ - 1) / kRowsQ);
        rows_stats_kernel<D><<<grid, kRowsThreads, 0, s>>>(f, stats);
        rows_pv_kernel<D><<<grid, kRowsThreads, 0, s>>>(f, stats);
        return;
    }
    const dim3 grid(f.heads, (f.rows + 15) / 16);
    const size_t lds = share_stats_lds<D>((f.p0 + f.rows + kBlockKeys - 1) / kBlockKeys);
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&share_stats_kernel<D, LONG>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
    (void)attr;  // (a refusal shows at the launch)
    share_stats_kernel<D, LONG><<<grid, kShareThreads, lds, s>>>(f, stats);
    share_pv_kernel<D, LONG><<<grid, kShareThreads, 0, s>>>(f, stats);
}

hipError_t launch_rows_attention(hipStream_t s, const FlashArgs& f, float2* stats, int head_dim) {
    const bool lng = f.p0 + f.rows > kLongKeys;
    if (head_dim == 128) lng ? rows_attention_t<128, true>(s, f, stats) : rows_attention_t<128, false>(s, f, stats);
    else if (head_dim == 64) lng ? rows_attention_t<64, true>(s, f, stats) : rows_attention_t<64, false>(s, f, stats);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// ---- self-tests --------------------------------------------------------------

// what 21: exp_nonpos elementwise.  22, 23: eight-term products through two
// 16x16x4 or four 32x32x2 FP32 MFMAs from +0, one wave per group of inputs: A
// [rows][8], then B [columns][8]; out [rows][columns], of the 32 x 32 form the
// rows of the group's parity (a sum of -0 as +0).
__global__ __launch_bounds__(64) void rows_selftest_kernel(int which, const float* in, float* out) {
    const int lane = threadIdx.x, g = blockIdx.x;
    if (which == 21) {
        out[g * 64 + lane] = exp_nonpos(in[g * 64 + lane]);
    } else if (which == 22) {
        const float *a = in + (size_t)g * 256, *b = a + 128;
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int k = lane >> 4; k < 8; k += 4) acc = mfma_f32_16(a[(lane & 15) * 8 + k], b[(lane & 15) * 8 + k], acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) out[(size_t)g * 256 + (4 * (lane >> 4) + r) * 16 + (lane & 15)] = acc[r] + 0.0f;
    } else {
        const float *a = in + (size_t)g * 512, *b = a + 256;
        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
        for (int k = lane >> 5; k < 8; k += 2) acc = mfma_f32_32(a[(lane & 31) * 8 + k], b[(lane & 31) * 8 + k], acc);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = acc32_row(lane, r);
            if ((row & 1) == (g & 1)) out[(size_t)g * 512 + (row >> 1) * 32 + acc32_col(lane)] = acc[r] + 0.0f;
        }
    }
}

hipError_t launch_rows_selftest(hipStream_t s, int which, const float* in, float* out, size_t n) {
    const size_t group = which == 21 ? 64 : which == 22 ? 256 : 512;
    if (which < 21 || which > 23 || n % group || n / group < 1 || n / group > 0x7fffffff) return hipErrorInvalidValue;
    rows_selftest_kernel<<<(unsigned)(n / group), 64, 0, s>>>(which, in, out);
    return hipGetLastError();
}

// ---- host --------------------------------------------------------------------

// Rows per pass through the layers: the GEMMs gain nothing from more, and
// the scratch stays small (4096 rows of the 3B class: 320 MB).
constexpr int kRowsChunk = 4096;

bool rows_supported(const Yue2Model* m, int context, int n) {
    const Yue2Config& c = m->c;
    if (n < 2 || (c.head_dim != 64 && c.head_dim != 128)) return false;
    if (c.hidden_size % kGemmTK || c.intermediate_size % kGemmTK || (c.num_attention_heads * c.head_dim) % kGemmTK)
        return false;
    // A token step costs about the same whatever n is; here few rows cost as
    // much as 32, and their attention walks the context with few workgroups.
    // Measured, four 3B-class layers and the head (us): 880 + 0.38 per cached
    // key against 200 + 230 n (265 n at 8000 keys); two layers of the reduced
    // shape: 200 + 0.11 against 65 + 73 n; four of the YuE2 shape: 770 + 0.36
    // against 240 + 175 n (195 n); four of a 1B class: 720 + 0.24 against
    // 160 + 215 n.  The lines cross at n = 3-4 without a context, 5-7 at 2048
    // keys, 12-17 at 8000.
    return n >= 4 + (context + 299) / 600;
}

int run_rows(Yue2Model* m, Yue2Cache* c, const int32_t* ids, int n, int phase, bool head) {
    const Yue2Config& cf = m->c;
    const int H = cf.hidden_size, D = cf.head_dim, Hq = cf.num_attention_heads, Hkv = cf.num_key_value_heads;
    const int I = cf.intermediate_size, qw = Hq * D, qkvw = (Hq + 2 * Hkv) * D;
    const size_t R = std::min(n, kRowsChunk);
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t o = at;
        at = (at + bytes + 255) / 256 * 256;
        return o;
    };
    const size_t o_x = take(4 * R * H), o_qkv = take(4 * R * qkvw), o_h = take(2 * R * H), o_q = take(2 * R * qw);
    const size_t o_att = take(2 * R * qw), o_act = take(2 * R * I), o_st = take(sizeof(float2) * R * Hq);
    const size_t o_ids = take(sizeof(int32_t) * (size_t)n);
    if (m->scratch.ensure(at) != hipSuccess) {
        (void)hipGetLastError();
        return 1;
    }
    const Scratch& b = m->scratch;
    float *x = reinterpret_cast<float*>(b.p + o_x), *qkv = reinterpret_cast<float*>(b.p + o_qkv);
    uint16_t *h = reinterpret_cast<uint16_t*>(b.p + o_h), *q = reinterpret_cast<uint16_t*>(b.p + o_q);
    uint16_t *att = reinterpret_cast<uint16_t*>(b.p + o_att), *act = reinterpret_cast<uint16_t*>(b.p + o_act);
    float2* stats = reinterpret_cast<float2*>(b.p + o_st);
    int32_t* dids = reinterpret_cast<int32_t*>(b.p + o_ids);
    hipStream_t s = m->stream;
    const float eps = cf.rms_norm_eps;
    // the norms' fallbacks are counted as the token steps of this model count
    // them (the step kernel leaves out the final norm's), and read when asked for
    int32_t* fallbacks = &m->rows_state->norm_fallbacks;
    hipError_t e = hipMemcpyAsync(dids, ids, sizeof(int32_t) * n, hipMemcpyHostToDevice, s);
    for (int p0 = 0; p0 < n && e == hipSuccess; p0 += (int)R) {
        const int rows = std::min((int)R, n - p0), pos = c->length + p0;
        e = launch_embed_rows(s, m->embed, dids + p0, x, rows, H);
        for (int l = 0; l < cf.num_hidden_layers && e == hipSuccess; ++l) {
            const LayerDev& L = m->layers[l];
            const RopeArgs ra{qkv, q, c->kv, c->capacity, l, Hq, Hkv, D, pos, L.q_norm, L.k_norm,
                              m->rope_cos, m->rope_sin, eps};
            const FlashArgs fa{q, c->kv, c->capacity, l, Hq, Hkv, pos, rows, 1.0f / std::sqrt((float)D), att};
            e = launch_norm_rows(s, x, L.in_norm, h, rows, H, eps, fallbacks);
            if (e == hipSuccess)
                e = launch_dot_gemm(s, GEPI_ROUND, GemmArgs{h, H, L.wqkv, nullptr, H, qkv, nullptr, qkvw, rows, qkvw, H});
            if (e == hipSuccess) e = launch_rope_append(s, ra, rows);
            if (e == hipSuccess) e = launch_rows_attention(s, fa, stats, D);
            if (e == hipSuccess)
                e = launch_dot_gemm(s, GEPI_RESID, GemmArgs{att, qw, L.wo, nullptr, qw, x, nullptr, H, rows, H, qw});
            if (e == hipSuccess) e = launch_norm_rows(s, x, L.post_norm, h, rows, H, eps, fallbacks);
            if (e == hipSuccess)
                e = launch_dot_gemm(s, GEPI_SWIGLU_BF16, GemmArgs{h, H, L.wg, L.wu, H, nullptr, act, I, rows, I, H});
            if (e == hipSuccess)
                e = launch_dot_gemm(s, GEPI_RESID, GemmArgs{act, I, L.wd, nullptr, I, x, nullptr, H, rows, H, I});
        }
        if (e == hipSuccess && head && p0 + rows == n)
            if (int rc = enqueue_head(m, m->ws, x + (size_t)(rows - 1) * H, phase, s, 1,
                                      m->step_kernel ? nullptr : m->rows_state)) {
                (void)hipStreamSynchronize(s);
                return rc;
            }
    }
    const hipError_t done = hipStreamSynchronize(s);  // nothing runs over the scratch any more
    m->scratch.trim();
    if (e == hipSuccess) e = done;
    return e == hipSuccess ? YUE2_OK : hip_fail(e, "multi-row forward");
}

}  // namespace y2
