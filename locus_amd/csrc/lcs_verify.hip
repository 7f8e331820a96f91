// Speculative-decoding verify for MI355X (gfx950).
//
// Per row: greedy argmax with the first-index tie rule (llama.cpp:1237-1245)
// and the natural-distribution log-probability of the row's draft token
// (logprobs_from with chosen = draft, n_top = 0: sampling.cpp:150-170). Per
// sequence: the acceptance length of engine.cpp:357-383 - the number of
// leading rows whose argmax equals the draft they predict.
//
// Two launches on the caller's stream: verify_kernel streams each row once
// (one workgroup per row) and writes the row's argmax and draft logprob;
// accept_kernel then reads each sequence's argmaxes and writes its acceptance
// length. The kernel boundary orders the first launch's stores before the
// second's loads, so no workgroup waits on or signals another.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "lcs_device.hpp"
#include "lcs_internal.hpp"

namespace lcs {

// NT: threads per row. A row's time is its rounds of NT x U 16-byte groups:
// for few rows a memory latency and the round's arithmetic each (20 rows, V
// 128256: 29.3 us a call with the running max moved per group and 256 threads,
// 17.2 with it moved per round, 13.0 with 512 threads), for many the memory
// stream (4096 bf16 rows, V 163840: 246 -> 234 us, 5.7 TB/s).
template <int G, int NT>
__global__ __launch_bounds__(NT) void verify_kernel(VerifyArgs a) {
    constexpr int U = 8;                   // 16-byte groups in flight per thread
    constexpr float kL2E = 1.4426950408889634f;
    __shared__ float redf[NT / kWave];
    __shared__ uint32_t redu[NT / kWave];
    __shared__ double redd[NT / kWave];
    const uint32_t rows = a.n_seq * a.rows_per_seq;
    const uint32_t row = wg_x();
    if (row >= rows) return;
    const uint32_t V = a.vocab;
    const uint32_t esz = a.dtype == LCS_BF16 ? 2u : 4u;
    const void* rowp = static_cast<const char*>(a.logits) + (uint64_t)row * a.row_stride * esz;
    const float NEG = -__builtin_huge_valf();

    // per lane: running max om, the first group bg that reached it, and
    // os = sum exp(v - om) (f32 group sums of exp2 accumulated in f64). The
    // terms are 2^fma(v, K, b) with b = RN(-om K): they share the exponent
    // error e_b = om K + b (exact, by an fma), which corr = 2^-e_b takes out
    // (without it a logit of magnitude 100 would cost ~5e-6 in log z)
    const uint32_t ng = (V + G - 1) / G;
    float om = NEG, b = 0.0f;
    double os = 0.0, corr = 1.0;
    uint32_t bg = 0xffffffffu;
    for (uint32_t g0 = 0; g0 < ng; g0 += NT * U) {
        uint4 r[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t gi = g0 + u * NT + tid_x();
            r[u] = load16(rowp, gi < ng ? gi : 0u);
        }
        // the round's group maxima first, so that the running max moves (and
        // the sum is rescaled) at most once a round
        float v[U][G], gm[U], m = NEG;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t gi = g0 + u * NT + tid_x();
            decode<G>(r[u], v[u]);
            if ((g0 + (u + 1) * NT) * G > V) {   // (uniform: the row's last groups)
#pragma unroll
                for (int k = 0; k < G; ++k) v[u][k] = gi * G + k < V ? v[u][k] : NEG;
            }
            gm[u] = v[u][0];
#pragma unroll
            for (int k = 1; k < G; ++k) gm[u] = fmaxf(gm[u], v[u][k]);
            m = fmaxf(m, gm[u]);
        }
        if (m > om) {
            os = om == NEG ? 0.0 : os * (double)__builtin_amdgcn_exp2f((om - m) * kL2E);
            om = m;
#pragma unroll
            for (int u = U - 1; u >= 0; --u) bg = gm[u] == m ? g0 + u * NT + tid_x() : bg;
            b = -om * kL2E;
            corr = (double)__builtin_amdgcn_exp2f(-fmaf(om, kL2E, b));
        }
        if (om != NEG) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float c[G];
#pragma unroll
                for (int k = 0; k < G; ++k) c[k] = __builtin_amdgcn_exp2f(fmaf(v[u][k], kL2E, b));
#pragma unroll
                for (int w = G / 2; w >= 1; w /= 2)
#pragma unroll
                    for (int k = 0; k < w; ++k) c[k] += c[k + w];
                os += (double)c[0] * corr;
            }
        }
    }
    // first index of the lane max inside its first group
    uint32_t idx = 0xfffffffeu;
    if (bg != 0xffffffffu) {
        float v[G];
        decode<G>(load16(rowp, bg), v);
        uint32_t k = G;
#pragma unroll
        for (int j = G - 1; j >= 0; --j) k = (bg * G + j < V && v[j] == om) ? (uint32_t)j : k;
        idx = bg * G + k;
    }
    float bm = om;
    block_argmax<NT>(bm, idx, redf, redu);
    const double sc = om == NEG ? 0.0 : os * exp((double)om - (double)bm);
    const double z = block_sum<NT>(sc, redd);
    if (tid_x() == 0) {
        const double log_z = log(z) + (double)bm;
        const int32_t d = a.draft[row];
        float lp = 0.0f;
        if (d >= 0 && (uint32_t)d < V) lp = (float)((double)load_elem(rowp, a.dtype, (uint32_t)d) - log_z);
        a.draft_lp[row] = lp;
        a.argmax_ids[row] = (int32_t)(idx < V ? idx : 0u);
    }
}

// Acceptance length per sequence (engine.cpp:366-383): leading rows whose
// argmax equals their draft. A wave per sequence, a row per lane (rows_per_seq
// <= 64): one memory round trip instead of one per accepted row.
constexpr uint32_t kAcceptSeqs = 4;   // sequences per workgroup
__global__ __launch_bounds__(kAcceptSeqs * kWave) void accept_kernel(VerifyArgs a) {
    const uint32_t seq = wg_x() * kAcceptSeqs + tid_x() / kWave;
    if (seq >= a.n_seq) return;
    const uint32_t lane = (uint32_t)lane_id(), R = a.rows_per_seq;
    const uint32_t row = seq * R + (lane < R ? lane : 0u);
    const uint64_t miss = ballot(lane >= R || a.argmax_ids[row] != a.draft[row]);
    const uint32_t acc = miss ? min((uint32_t)__builtin_ctzll(miss), R) : R;
    if (lane == 0u) a.accept_len[seq] = acc;
}

// Threads per row: a row of more than two rounds of 512 threads takes 512 (us
// a call with 256 / 512 / 1024 threads, f32, V 128256: 20 rows 17.2 / 13.0 /
// 13.0, 128 rows 19.6 / 15.6 / 17.2, 2048 rows 187.5 / 187.1 / 189; bf16, V
// 163840, 4096 rows 238.3 / 233.8 / 267), except where about two rows a CU
// make one uneven round of the larger workgroups (512 rows: 51.4 / 52.7, bf16
// 34.9 / 36.6). A shorter row leaves them idle (2048 rows of V 5000: 13.3 /
// 17.1).
template <int G>
static void launch_rows(const VerifyArgs& a, hipStream_t st) {
    const uint32_t rows = a.n_seq * a.rows_per_seq;
    const bool wide = (a.vocab + G - 1u) / G > 8192u && (rows <= 256u || rows > 768u);
    if (wide) hipLaunchKernelGGL((verify_kernel<G, 512>), dim3(rows), dim3(512), 0, st, a);
    else hipLaunchKernelGGL((verify_kernel<G, 256>), dim3(rows), dim3(256), 0, st, a);
}

hipError_t launch_verify(const VerifyArgs& a, hipStream_t st) {
    if (a.dtype == LCS_BF16) launch_rows<8>(a, st);
    else launch_rows<4>(a, st);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(accept_kernel, dim3((a.n_seq + kAcceptSeqs - 1u) / kAcceptSeqs), dim3(kAcceptSeqs * kWave), 0, st, a);
    return hipGetLastError();
}

}  // namespace lcs
