// The lm-head product with the sampler's first statistics in its epilogue,
// for MI355X (gfx950): logits = X W^T in bf16 on the matrix cores (f32
// accumulation), and per (row, block of vocabulary columns) the block's
// argmax (first index), its sum of exponentials against the block max, and
// the logit of the row's draft token when the block holds it. A per-sequence
// finalize then gives each row's argmax and log-normaliser, the draft's
// log-probability and each sequence's acceptance length, so greedy and
// speculative-verify rows need no second read of the logits (and no logits
// at all when the caller does not ask for them).
//
// Reference: the output projection matvec(out_w, norm(x)) per decode token
// (src/locus/model/llama.cpp:512-513, batched at 754-761; Ops::matvec,
// backend/registry.hpp:14-15), then argmax (llama.cpp:1237-1245) and
// logprobs_from with chosen = draft (sampling.cpp:150-170) per row and the
// acceptance rule of engine.cpp:357-383 per sequence.
//
// Up to 64 rows (decode) the weight stream from HBM is the bound; from 256
// rows up (verify) the matrix cores are.
//
// Measured (us a call; the library bf16 GEMM alone 976 at 1024 rows; "before":
// this kernel's predecessor, 64 rows x 256 columns with the weight fragments
// loaded straight into registers and the shared x behind a barrier per step):
//   rows x columns x hidden       before   now
//   64   x 128256 x 4096 (logits)   218    198
//   8    x 32000  x 4096            124     51
//   128  x 128256 x 4096            448    220
//   1024 x 128256 x 4096           2619    886
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "lcs_device.hpp"
#include "lcs_internal.hpp"

namespace lcs {

namespace {
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int kLmThreads = 256;
constexpr float kL2E = 1.4426950408889634f;
constexpr uint32_t kBigHidden = 1u << 22;     // above: 64-bit row offsets

// Waits until at most N vector memory operations are outstanding (and every
// LDS operation is done); the compiler moves no memory access across it.
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vm_lgkm() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// 16 bytes per lane from a buffer (offsets vo per lane + so) to LDS at
// dst + 16 lane (dst is wave-uniform).
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t rs, unsigned char* dst, uint32_t vo, uint32_t so) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)dst, 16, (int)vo, (int)so, 0, 0);
}
// The same from a per-lane address.
__device__ __forceinline__ void dma16_at(const void* src, unsigned char* dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}
// NaN, by its bits: the build's float comparisons and selects assume that there
// are none (the empty asm keeps the compiler from concluding the same here).
__device__ __forceinline__ bool nan_bits(float v) {
    uint32_t u = __float_as_uint(v);
    asm("" : "+v"(u));
    return (u & 0x7fffffffu) > 0x7f800000u;
}
// A workgroup barrier that waits for no memory operation.
__device__ __forceinline__ void block_sync() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

}  // namespace

// A workgroup computes 64 VT columns of BR rows, transposed (columns on the
// MFMA's row side, so that a lane holds many columns of one row and the
// epilogue reduces in registers): NW waves, two over the rows, in
// v_mfma_f32_32x32x16_bf16 tiles (lane l carries 8 consecutive k of row l % 32
// of either operand, k chunk l / 32, and returns rows 8 (e / 4) + 4 (l / 32) +
// e % 4 of column l % 32). The 256 x 256 tile takes eight waves, so that two
// share a SIMD and one's loads, barriers and epilogue leave the matrix cores to
// the other (1024 rows: 990 us with four, 963 with eight).
//
// Both operands go straight from memory into a ring of ST LDS stages of 16 KS k
// with 16-byte DMA loads, so that no register holds data in flight. The loads
// are what holds the matrix cores up (1024 rows: busy 1.03 M of 1.52 M cycles): a
// stage of 64 k reads whole 128-byte lines, half the requests of 32 k, and two
// such stages serve as well as four (1024 rows 963 -> 921 us, 64 rows 209 ->
// 199); narrow and 128-row tiles have too few bytes in flight then (8 x 32000
// 52 -> 69 us, 128 rows 218 -> 229) and keep 32 k. A row's 16-byte chunks are
// permuted by its bits from kSw up: a fragment read's 16 lanes of a phase then
// cover the 64 banks once (0 conflict cycles of 101 M). One barrier per stage, ahead of its last products: each wave has then
// read the stage and its loads of the next one have landed.
//
// The workgroups of a column block are placed on one XCD in consecutive
// dispatch slots (workgroups are dealt to the 8 XCDs in turn): they run
// together, so the block's weight rows come from HBM once and from that XCD's
// L2 for the other row tiles. With one row tile each workgroup starts at its
// own k-step and wraps round, so that those in flight do not all read the same
// offset of their rows (72 rows x 128256 x 4096: 245 -> 225 us); with more the
// row tiles share x through the L2 by running in step (1024 rows: 1013 against
// 1057 us with a start of its own).
template <int VT, int BR, int ST, int NW = 4, int KS = 2, bool BIG = false>
__global__ __launch_bounds__(NW * kWave, 2) void lmhead_tile(LmArgs a) {
    constexpr uint32_t kTV = 64u * VT;        // columns per workgroup
    constexpr int kTK = 16 * KS;              // k per LDS stage
    constexpr uint32_t kTRowB = kTK * 2;      // bytes of a row in a stage
    constexpr uint32_t kStage = (kTV + BR) * kTRowB;
    constexpr int WM = NW / 2;                // waves side by side over the columns, two over the rows
    constexpr int CT = 2 * VT / WM, RT = BR / 64;   // 32-column and 32-row tiles per wave
    constexpr uint32_t kCh = 2 * KS, kLog = KS == 4 ? 3 : 2;   // 16-byte chunks of a row
    constexpr uint32_t kSw = KS == 4 ? 1 : 2;   // the row bits that permute them start here
    constexpr int kLR = 64 / (int)kCh * NW;   // rows that one DMA load of every wave covers
    constexpr int LA = kTV / kLR, LB = BR / kLR;   // DMA loads per wave and stage
    static_assert(KS == 2 || (KS == 4 && ST == 2), "the schedule of the k-loop");
    static_assert(LA * kLR == (int)kTV && LB * kLR == BR && CT * WM == 2 * VT, "tile shape");
    constexpr int LPS = LA + LB;
    __shared__ __attribute__((aligned(128))) unsigned char lds[ST * kStage];
    const uint32_t tid = tid_x();
    const int lane = lane_id(), wv = __builtin_amdgcn_readfirstlane((int)(tid / kWave));
    uint32_t nb = wg_x();
    const uint32_t slot = nb >> 3;
    const uint32_t r0 = (slot % a.nchunks) * BR;
    nb = 8u * (slot / a.nchunks) + (nb & 7u);
    if (nb >= a.nblocks) return;   // (the grid is a multiple of 8 blocks)
    const uint32_t K = a.hidden, V = a.vocab;
    const uint32_t n0 = nb * kTV;
    const uint32_t vrows = min((uint32_t)BR, a.rows - r0), vcols = min(kTV, V - n0);
    const uint32_t wm = (uint32_t)wv % WM, wn = (uint32_t)wv / WM;   // the wave's columns and rows
    const uint16_t* wbase = a.w + (uint64_t)n0 * K;
    const uint16_t* xbase = a.x + (uint64_t)r0 * K;
    const __amdgpu_buffer_rsrc_t wrs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(wbase), 0, (int)(vcols * K * 2u), 0x00020000);
    const __amdgpu_buffer_rsrc_t xrs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(xbase), 0, (int)(vrows * K * 2u), 0x00020000);
    // DMA load i of a wave covers rows kLR i + 16 wv + lane / 4, a 16-byte
    // chunk per lane; rows past the tile read row 0 (masked in the epilogue)
    const uint32_t rr = kWave / kCh * (uint32_t)wv + ((uint32_t)lane >> kLog);
    const uint32_t ch = (((uint32_t)lane & (kCh - 1u)) ^ ((rr >> kSw) & (kCh - 1u))) * 16u;
    uint32_t wo[LA], xo[LB];
#pragma unroll
    for (int i = 0; i < LA; ++i) wo[i] = (kLR * i + rr < vcols ? kLR * i + rr : 0u) * K * 2u + ch;
#pragma unroll
    for (int i = 0; i < LB; ++i) xo[i] = (kLR * i + rr < vrows ? kLR * i + rr : 0u) * K * 2u + ch;
    const uint32_t nsteps = K / kTK;
    const uint32_t rot = a.nchunks == 1u ? nb % nsteps : 0u;
    // (the byte offset of stage t in a row; stages past the end re-read the last)
    auto koff = [&](uint32_t t) -> uint32_t {
        uint32_t q = (t < nsteps ? t : nsteps - 1u) + rot;
        return (q >= nsteps ? q - nsteps : q) * kTRowB;
    };
    auto issue1 = [&](int i, uint32_t ko, uint32_t sl) {   // DMA load i of a stage
        unsigned char* b = lds + sl * kStage + (uint32_t)wv * 1024u + i * (kLR * kTRowB);
        if (BIG) {   // (the row offsets need 64 bits)
            const uint32_t r = kLR * (uint32_t)(i < LA ? i : i - LA) + rr;
            const uint16_t* p = i < LA ? wbase + (uint64_t)(r < vcols ? r : 0u) * K : xbase + (uint64_t)(r < vrows ? r : 0u) * K;
            dma16_at(reinterpret_cast<const unsigned char*>(p) + ko + ch, b);
        } else if (i < LA) {
            dma16(wrs, b, wo[i < LA ? i : 0], ko);
        } else {
            dma16(xrs, b, xo[i >= LA ? i - LA : 0], ko);
        }
    };
    auto issue = [&](uint32_t t, uint32_t sl) {
#pragma unroll
        for (int i = 0; i < LPS; ++i) issue1(i, koff(t), sl);
    };
    f32x16 acc[CT][RT];
#pragma unroll
    for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int j = 0; j < RT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    // fragment s (16 k) of row r: chunk 2 s + lane / 32
    const uint32_t lr = (uint32_t)lane & 31u, lh = (uint32_t)lane >> 5;
    uint32_t fo[KS];
#pragma unroll
    for (uint32_t s = 0; s < KS; ++s) fo[s] = lr * kTRowB + (((2u * s + lh) ^ ((lr >> kSw) & (kCh - 1u))) * 16u);
    struct Frag { bf16x8 w[CT], x[RT]; };
    // read i of a fragment set: x first (every product needs all of it), then w
    constexpr int NR = CT + RT, NP = CT * RT;
    auto read1 = [&](Frag& f, int i, uint32_t sl, int s) {
        const unsigned char* pw = lds + sl * kStage + wm * (kTV / WM * kTRowB) + fo[s];
        const unsigned char* px = lds + sl * kStage + kTV * kTRowB + wn * (BR / 2 * kTRowB) + fo[s];
        if (i < RT) f.x[i < RT ? i : 0] = *reinterpret_cast<const bf16x8*>(px + i * 32 * kTRowB);
        else f.w[i >= RT ? i - RT : 0] = *reinterpret_cast<const bf16x8*>(pw + (i - RT) * 32 * kTRowB);
    };
    auto mul1 = [&](const Frag& f, int k) {   // product k of NP
        const int i = k / RT, j = k % RT;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[i], f.x[j], acc[i][j], 0, 0, 0);
    };
    Frag f0, f1;
#pragma unroll
    for (int t = 0; t < ST; ++t) issue((uint32_t)t, (uint32_t)t);
    wait_vm<(ST - 1) * LPS>();
    block_sync();
#pragma unroll
    for (int i = 0; i < NR; ++i) read1(f0, i, 0u, 0);
    uint32_t sl = 0u;
    // Every LDS read and DMA load is issued behind a product: a wave issues
    // in order, and eight DMA loads in a row hold it for longer than the
    // products queued ahead of them last (1024 rows, four waves: 1022 -> 980 us).
    // (KS 4, two stages: half of a stage's loads go out behind the last products
    // of the stage whose place it takes, half behind the next stage's first)
    uint32_t kn = 0u;   // the offset of the stage whose second half is to be issued
    for (uint32_t t = 0; t < nsteps; ++t) {
        const uint32_t ns = sl + 1u == (uint32_t)ST ? 0u : sl + 1u;
        constexpr int H = LPS / 2;
#pragma unroll
        for (int s = 0; s < KS - 1; ++s) {
            const bool more = KS == 4 && s == 0;
#pragma unroll
            for (int k = 0; k < NP; ++k) {
                mul1(s % 2 == 0 ? f0 : f1, k);
#pragma unroll
                for (int i = k * (NR + (more ? LPS - H : 0)) / NP; i < (k + 1) * (NR + (more ? LPS - H : 0)) / NP; ++i) {
                    if (i < NR) read1(s % 2 == 0 ? f1 : f0, i, sl, s + 1);
                    else if (t != 0u) issue1(H + i - NR, kn, ns);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // stage t is read, stage t + 1 has landed, in every wave
        wait_vm_lgkm<KS == 4 ? 0 : (ST - 2) * LPS>();
        block_sync();
        kn = koff(t + ST);
        constexpr int L = KS == 4 ? H : LPS;
#pragma unroll
        for (int k = 0; k < NP; ++k) {
            mul1(f1, k);
#pragma unroll
            for (int i = k * (NR + L) / NP; i < (k + 1) * (NR + L) / NP; ++i) {
                if (i < NR) read1(f0, i, ns, 0);
                else issue1(i - NR, kn, sl);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        sl = ns;
    }
    wait_vm_lgkm<0>();
    __syncthreads();   // (the last loads have landed: the ring is free)

    // ---- epilogue: acc[i][j][e] is column n0 + kTV / WM wm + 32 i + 8 (e / 4) +
    // 4 lh + e % 4 of row r0 + BR / 2 wn + 32 j + lr ----
    struct Part { float max, sum, draft; uint32_t idx; };
    Part* part = reinterpret_cast<Part*>(lds);   // [WM][BR]: by the wave's columns
    const bool full = vcols == kTV;
    const bool vec = a.logits && (a.ld_logits & 3u) == 0u && (reinterpret_cast<uintptr_t>(a.logits) & 15u) == 0u;
#pragma unroll
    for (int j = 0; j < RT; ++j) {
        const uint32_t rl = wn * (BR / 2) + 32u * j + lr;   // the lane's row in the tile
        const bool rin = rl < vrows;
        const uint32_t cb = kTV / WM * wm + 4u * lh;            // columns cb + 32 i + 8 (e / 4) + e % 4
        if (a.logits && rin) {
            float* out = a.logits + (uint64_t)(r0 + rl) * a.ld_logits + n0;
#pragma unroll
            for (int i = 0; i < CT; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t c = cb + 32u * i + 8u * q;
                    if (vec && c + 4u <= vcols) {
                        *reinterpret_cast<float4*>(out + c) =
                            make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (c + e < vcols) out[c + e] = acc[i][j][4 * q + e];
                    }
                }
        }
        const float NEG = -__builtin_huge_valf();
        if (!full) {
#pragma unroll
            for (int i = 0; i < CT; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (cb + 32u * i + 8u * (e / 4) + e % 4 >= vcols) acc[i][j][e] = NEG;
        }
        // the lane's max, its first column, the draft's logit
        float m = acc[0][j][0];
#pragma unroll
        for (int i = 0; i < CT; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) m = fmaxf(m, acc[i][j][e]);
        const int32_t dr = a.draft && rin ? a.draft[r0 + rl] : -1;
        const uint32_t dc = (uint32_t)dr < V ? (uint32_t)dr - n0 - cb : 0xffffffffu;   // the draft's column, from cb
        uint32_t ci = kTV;
        float dl = 0.0f;
#pragma unroll
        for (int i = CT - 1; i >= 0; --i)
#pragma unroll
            for (int e = 15; e >= 0; --e) {
                const uint32_t c = 32u * i + 8u * (e / 4) + e % 4;
                ci = acc[i][j][e] == m ? c : ci;
            }
        uint32_t found = 0u;
        if (ballot(dc < kTV / WM && (dc & 4u) == 0u) != 0u) {
#pragma unroll
            for (int i = 0; i < CT; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const uint32_t c = 32u * i + 8u * (e / 4) + e % 4;
                    if (dc == c) { dl = acc[i][j][e]; found = kLmDraftBit; }
                }
        }
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < CT; ++i)
#pragma unroll
            for (int e = 0; e < 16; e += 4) {
                float t[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) t[k] = __builtin_amdgcn_exp2f((acc[i][j][e + k] - m) * kL2E);
                s += (t[0] + t[1]) + (t[2] + t[3]);
            }
        if (nan_bits(s)) {
            // a NaN or +inf, or nothing but -inf (columns past the vocabulary
            // too): the max and its first column again, NaNs left out, which
            // keep the sum a NaN; columns of -inf have no term
            bool nan = false;
            m = NEG;
            ci = kTV;
#pragma unroll
            for (int i = 0; i < CT; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float v = acc[i][j][e];
                    const bool n = nan_bits(v), up = !n && (ci == kTV || v > m);
                    nan = nan || n;
                    m = up ? v : m;
                    ci = up ? 32u * i + 8u * (e / 4) + e % 4 : ci;
                }
            s = m == NEG && !nan ? 0.0f : s;
        }
        ci += cb;
        // lanes l and l + 32 share a row
        const float m2 = __shfl_xor(m, 32), s2 = __shfl_xor(s, 32), d2 = __shfl_xor(dl, 32);
        const uint32_t c2 = (uint32_t)__shfl_xor((int)ci, 32), f2 = (uint32_t)__shfl_xor((int)found, 32);
        const float M = fmaxf(m, m2);
        s = (m == NEG ? s : s * __builtin_amdgcn_exp2f((m - M) * kL2E)) +
            (m2 == NEG ? s2 : s2 * __builtin_amdgcn_exp2f((m2 - M) * kL2E));
        ci = m > m2 ? ci : m2 > m ? c2 : min(ci, c2);
        if (lh == 0u) part[wm * BR + rl] = Part{M, s, found ? dl : d2, ci | found | f2};
    }
    __syncthreads();
    if (tid < vrows) {
        const float NEG = -__builtin_huge_valf();
        Part p = part[tid];
#pragma unroll
        for (int w = 1; w < WM; ++w) {
            // (a side of -inf: its sum is 0, or NaN where it holds one)
            const Part q = part[w * BR + tid];
            const float M = fmaxf(p.max, q.max);
            p.sum = (p.max == NEG ? p.sum : p.sum * __builtin_amdgcn_exp2f((p.max - M) * kL2E)) +
                    (q.max == NEG ? q.sum : q.sum * __builtin_amdgcn_exp2f((q.max - M) * kL2E));
            p.draft = (p.idx & kLmDraftBit) ? p.draft : q.draft;
            const uint32_t pc = p.idx & ~kLmDraftBit, qc = q.idx & ~kLmDraftBit;
            p.idx = (p.max > q.max ? pc : q.max > p.max ? qc : min(pc, qc)) | ((p.idx | q.idx) & kLmDraftBit);
            p.max = M;
        }
        LmRec rec;
        rec.max = p.max;
        // (a block of NaNs has no column that equals its max: its first one)
        const uint32_t col = p.idx & ~kLmDraftBit;
        rec.idx = (n0 + (col < vcols ? col : 0u)) | (p.idx & kLmDraftBit);
        rec.sum = p.sum;
        rec.draft = p.draft;
        a.recs[(uint64_t)(r0 + tid) * a.nblocks + nb] = rec;
    }
}

// One workgroup per sequence (rows_per_seq rows; a row is its own sequence
// when rows_per_seq is 0): wave w of NW merges rows w, w + NW, ... from their
// blocks' records (the kernel boundary orders them after the product). A row's
// records (at most 64 PER) are requested together and stay in registers: one
// memory round trip a row (1024 rows of 501 records: 13.2 -> 5.6 us).
template <int NW, uint32_t PER>
__global__ __launch_bounds__(NW * kWave) void lmhead_fin(LmArgs a) {
    __shared__ int32_t am[64];
    const uint32_t tid = tid_x();
    const int lane = lane_id(), wv = (int)(tid / kWave);
    const uint32_t R = a.rows_per_seq ? a.rows_per_seq : 1u;
    const uint32_t seq = wg_x();
    for (uint32_t j = (uint32_t)wv; j < R; j += NW) {
        const uint32_t row = seq * R + j;
        const LmRec* rr = a.recs + (uint64_t)row * a.nblocks;
        LmRec rc[PER];
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) {   // (past the end: block 0 again)
            const uint32_t b = i * kWave + (uint32_t)lane;
            rc[i] = rr[b < a.nblocks ? b : 0u];
        }
        uint64_t best = ~0ull;
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) best = u64_min(best, rank_key(rc[i].max, rc[i].idx & ~kLmDraftBit));
        best = wave_min_u64(best);
        const float M = rank_val(best);
        double z = 0.0;
        float dl = 0.0f;
        bool has = false;
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) {
            const bool in = i * kWave + (uint32_t)lane < a.nblocks;
            z += in ? (double)rc[i].sum * (double)__builtin_amdgcn_exp2f((rc[i].max - M) * kL2E) : 0.0;
            if (in && (rc[i].idx & kLmDraftBit)) { dl = rc[i].draft; has = true; }
        }
        z = wave_sum(z);
        const uint64_t own = ballot(has);
        dl = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dl), own ? __builtin_ctzll(own) : 0));
        const double log_z = log_f64(z) + (double)M;
        if (lane == 0) {
            a.argmax_ids[row] = (int32_t)rank_idx(best);
            if (a.log_z) a.log_z[row] = (float)log_z;
            if (a.draft_lp) a.draft_lp[row] = own ? (float)((double)dl - log_z) : 0.0f;
            if (a.stats) a.stats[row] = lcs_row_stats{log_z, M, (int32_t)rank_idx(best)};
            am[j] = (int32_t)rank_idx(best);
        }
    }
    if (!a.accept_len || !a.draft) return;
    __syncthreads();
    if (tid == 0) {
        uint32_t acc = 0;
        while (acc < R && am[acc] == a.draft[seq * R + acc]) ++acc;
        a.accept_len[seq] = acc;
    }
}

// Column blocks of 64 vt columns that a context's record buffer has to hold for
// a vocabulary (see lmhead_shape's limits).
uint32_t lmhead_max_blocks(uint32_t vocab, uint32_t cus) {
    auto n = [&](uint32_t c) { return (vocab + c - 1u) / c; };
    auto least = [](uint32_t a, uint32_t b) { return a < b ? a : b; };
    const uint32_t n1 = least(n(64u), cus * 2u), n2 = least(n(128u), cus * 4u);
    const uint32_t m = least(n1 > n2 ? n1 : n2, kLmMaxBlocks);
    return m > n(256u) ? m : n(256u);
}

// The tile of a launch. Rows: 64-row tiles up to 64 rows; above, a 128-row tile
// where that leaves out a 256-row tile more than half empty (128 rows: 225
// against 288 us, 384 rows: 479 against 505; 256 rows: 357 against 308).
// Columns: a CU runs its workgroups' columns one after the other, whether two
// are resident or one, so the time goes by ceil(workgroups / CUs) x columns;
// narrow tiles read x more often for the same columns (64 x 128256 x 4096,
// 2 x 256, 4 x 128 and 8 x 64 columns a CU: 209, 227, 276 us), hence the
// weights. 64 rows x 4096, us by 320 / 256 / 128 / 64 columns (the rule's
// first): 20000: 51 (128), 62, 72; 40000: 89 (256), 99, 102; 80000: 131
// (320), 156, 162, 169; 128256: 209 (256), 226, 271; 151936 x 3584: 224 (320),
// 249, 251, 325.
struct LmShape { uint32_t vt, br; };
static LmShape lmhead_shape(uint32_t rows, uint32_t vocab, uint32_t hidden, uint32_t cus) {
    if (hidden > kBigHidden) return {4u, 64u};
    const uint32_t br = rows <= 64u ? 64u : rows <= 128u || (rows > 256u && rows <= 384u) ? 128u : 256u;
    const uint32_t chunks = (rows + br - 1u) / br;
    struct { uint32_t vt, br, weight; } const shapes[] = {   // (widest first; weight in 1/64)
        {5, 64, 64}, {4, 64, 64}, {2, 64, 69}, {1, 64, 85}, {4, 128, 64}, {2, 128, 77}, {4, 256, 64}, {2, 256, 77}};
    LmShape best{4u, br};
    uint64_t least = ~0ull;
    for (const auto& s : shapes) {
        if (s.br != br) continue;
        const uint64_t n = ((uint64_t)vocab + 64u * s.vt - 1u) / (64u * s.vt);
        if ((s.vt == 1u && n > 2u * cus) || (s.vt == 2u && n > 4u * cus) || n > kLmMaxBlocks) continue;   // (lmhead_max_blocks)
        const uint64_t cost = (n * chunks + cus - 1u) / cus * s.vt * s.weight;
        if (cost < least) {
            least = cost;
            best.vt = s.vt;
        }
    }
    return best;
}

hipError_t launch_lmhead(const LmArgs& a0, uint32_t cus, hipStream_t st) {
    LmArgs a = a0;
    const LmShape sh = lmhead_shape(a.rows, a.vocab, a.hidden, cus);
    const uint32_t cols = 64u * sh.vt;
    a.nblocks = (a.vocab + cols - 1u) / cols;
    a.nchunks = (a.rows + sh.br - 1u) / sh.br;
    const dim3 grid(8u * ((a.nblocks + 7u) / 8u) * a.nchunks), block(kLmThreads);
    // (stages: as deep as two workgroups a CU leave room for, or one where
    // there is no second; two of 64 k where two 256-column tiles a CU are all
    // there is: 199 us against 209 with two of 32 k and 212 with three)
    if (a.hidden > kBigHidden) hipLaunchKernelGGL((lmhead_tile<4, 64, 3, 4, 2, true>), grid, block, 0, st, a);
    else if (sh.br == 256u && sh.vt == 4u) hipLaunchKernelGGL((lmhead_tile<4, 256, 2, 8, 4>), grid, dim3(8 * kWave), 0, st, a);
    else if (sh.br == 256u) hipLaunchKernelGGL((lmhead_tile<2, 256, 3>), grid, block, 0, st, a);
    else if (sh.br == 128u && sh.vt == 4u) hipLaunchKernelGGL((lmhead_tile<4, 128, 3>), grid, block, 0, st, a);
    else if (sh.br == 128u) hipLaunchKernelGGL((lmhead_tile<2, 128, 4>), grid, block, 0, st, a);
    else if (sh.vt == 5u) hipLaunchKernelGGL((lmhead_tile<5, 64, 3>), grid, block, 0, st, a);
    else if (sh.vt == 4u && a.nblocks > cus && a.nblocks <= 2u * cus)
        hipLaunchKernelGGL((lmhead_tile<4, 64, 2, 4, 4>), grid, block, 0, st, a);
    else if (sh.vt == 4u) hipLaunchKernelGGL((lmhead_tile<4, 64, 4>), grid, block, 0, st, a);
    else if (sh.vt == 2u) hipLaunchKernelGGL((lmhead_tile<2, 64, 4>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((lmhead_tile<1, 64, 6>), grid, block, 0, st, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const uint32_t nseq = a.rows_per_seq ? a.rows / a.rows_per_seq : a.rows;
    constexpr uint32_t kMost = kLmMaxBlocks / kWave, kHalf = kMost / 2;
    const bool half = a.nblocks <= kHalf * kWave;
    if (a.rows_per_seq > 1u) {
        if (half) hipLaunchKernelGGL((lmhead_fin<8, kHalf>), dim3(nseq), dim3(8 * kWave), 0, st, a);
        else hipLaunchKernelGGL((lmhead_fin<8, kMost>), dim3(nseq), dim3(8 * kWave), 0, st, a);
    } else {
        if (half) hipLaunchKernelGGL((lmhead_fin<1, kHalf>), dim3(nseq), dim3(kWave), 0, st, a);
        else hipLaunchKernelGGL((lmhead_fin<1, kMost>), dim3(nseq), dim3(kWave), 0, st, a);
    }
    return hipGetLastError();
}

}  // namespace lcs
