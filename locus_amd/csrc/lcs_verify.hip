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

// ---- a row streamed once by NT threads ----
// Per lane: the running max om, the first group bg that reached it, and os =
// sum exp(v - om) (f32 group sums of exp2 accumulated in f64). The terms are
// 2^fma(v, K, b) with b = RN(-om K): they share the exponent error e_b = om K +
// b (exact, by an fma), which corr = 2^-e_b takes out (without it a logit of
// magnitude 100 would cost ~5e-6 in log z).
//
// A row's time is its rounds of NT x U 16-byte groups: for few rows a memory
// latency and the round's arithmetic each (20 rows, V 128256: 29.3 us a call
// with the running max moved per group and 256 threads, 17.2 with it moved per
// round, 13.0 with 512 threads), for many the memory stream (4096 bf16 rows, V
// 163840: 246 -> 234 us, 5.7 TB/s).
//
// A row's last round takes 1, 2, 3, 4 or 6 groups a thread where the row has no
// more: a short row would spend its time on the terms past its end (2048 bf16
// rows, us a call with eight / as here: V 1000 12.4 / 9.0, V 5000 13.4 / 10.1;
// 1024 rows of V 70000 33.9 / 29.6). Forms of their own: a row without a short
// round keeps its plain loop (the short ones beside it moved 20 f32 rows of V
// 128256 from 13.2 to 13.5), and the registers of eight groups keep short rows
// out (4096 bf16 rows of V 5000 16.3 / 14.5).
constexpr int kRound = 8;
enum RowForm { kRowRounds, kRowTail, kRowShort };   // rounds of kRound groups; and a shorter last one; that one alone
template <int G>
RowForm row_form(uint32_t vocab, uint32_t nt) {
    const uint32_t ng = (vocab + G - 1u) / G, left = ng % (kRound * nt);
    return ng <= 4u * nt ? kRowShort : left != 0u && left <= 6u * nt ? kRowTail : kRowRounds;
}
struct RowLane {
    float om, b;
    double os, corr;
    uint32_t bg;
};
// Rounds of U groups a thread over groups first .. end of a row of ng.
template <int G, int NT, int U>
__device__ __forceinline__ void stream_rounds(const void* rowp, uint32_t V, uint32_t ng, uint32_t first, uint32_t end,
                                              RowLane& l) {
    constexpr float kL2E = 1.4426950408889634f;
    const float NEG = -__builtin_huge_valf();
    float om = l.om, b = l.b;
    double os = l.os, corr = l.corr;
    uint32_t bg = l.bg;
    for (uint32_t g0 = first; g0 < end; g0 += NT * U) {
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
    l = RowLane{om, b, os, corr, bg};
}
template <int G, int NT, RowForm F>
__device__ __forceinline__ RowLane stream_row(const void* rowp, uint32_t V) {
    const uint32_t ng = (V + G - 1) / G;
    RowLane l{-__builtin_huge_valf(), 0.0f, 0.0, 1.0, 0xffffffffu};
    const uint32_t end = F == kRowRounds ? ng : F == kRowTail ? ng / (kRound * NT) * (kRound * NT) : 0u;
    if (F != kRowShort) stream_rounds<G, NT, kRound>(rowp, V, ng, 0u, end, l);
    if (F != kRowRounds) {   // (uniform branches; row_form leaves no more groups than these take)
        const uint32_t n = (ng - end + NT - 1u) / NT;
        if (F == kRowTail && n > 4u) stream_rounds<G, NT, 6>(rowp, V, ng, end, ng, l);
        else if (n > 3u) stream_rounds<G, NT, 4>(rowp, V, ng, end, ng, l);
        else if (n > 2u) stream_rounds<G, NT, 3>(rowp, V, ng, end, ng, l);
        else if (n > 1u) stream_rounds<G, NT, 2>(rowp, V, ng, end, ng, l);
        else stream_rounds<G, NT, 1>(rowp, V, ng, end, ng, l);
    }
    return l;
}

// The block's max and its first index, and the row's sum of exponentials
// against it (NT threads; red*: NT / kWave entries).
template <int G, int NT>
__device__ __forceinline__ double reduce_row(const RowLane& l, const void* rowp, uint32_t V, float& bm, uint32_t& idx,
                                             float* redf, uint32_t* redu, double* redd) {
    // first index of the lane max inside its first group
    idx = 0xfffffffeu;
    if (l.bg != 0xffffffffu) {
        float v[G];
        decode<G>(load16(rowp, l.bg), v);
        uint32_t k = G;
#pragma unroll
        for (int j = G - 1; j >= 0; --j) k = (l.bg * G + j < V && v[j] == l.om) ? (uint32_t)j : k;
        idx = l.bg * G + k;
    }
    bm = l.om;
    block_argmax<NT>(bm, idx, redf, redu);
    const double sc = l.om == -__builtin_huge_valf() ? 0.0 : l.os * exp((double)l.om - (double)bm);
    return block_sum<NT>(sc, redd);
}

template <int G, int NT, RowForm F>
__global__ __launch_bounds__(NT) void verify_kernel(VerifyArgs a) {
    __shared__ float redf[NT / kWave];
    __shared__ uint32_t redu[NT / kWave];
    __shared__ double redd[NT / kWave];
    const uint32_t rows = a.n_seq * a.rows_per_seq;
    const uint32_t row = wg_x();
    if (row >= rows) return;
    const uint32_t V = a.vocab;
    const void* rowp = static_cast<const char*>(a.logits) + (uint64_t)row * a.row_stride * (16u / G);
    const RowLane l = stream_row<G, NT, F>(rowp, V);
    float bm;
    uint32_t idx;
    const double z = reduce_row<G, NT>(l, rowp, V, bm, idx, redf, redu, redd);
    if (tid_x() == 0) {
        const double log_z = log(z) + (double)bm;
        const int32_t d = a.draft[row];
        float lp = 0.0f;
        if (d >= 0 && (uint32_t)d < V) lp = (float)((double)load_elem(rowp, a.dtype, (uint32_t)d) - log_z);
        a.draft_lp[row] = lp;
        a.argmax_ids[row] = (int32_t)(idx < V ? idx : 0u);
    }
}

// ---- logprobs_from over many rows (sampling.cpp:150-190) ----
// A workgroup per row streams it once and writes its argmax, chosen's logprob
// and the top n. The n-th largest of 64 sets of lanes' maxima bounds the row's
// n-th largest value from below, so the candidates lie in the lanes whose max
// reaches it (about n): their groups are read again, a group per lane of a wave,
// and the candidates ranked. A row with more lanes or candidates than fit
// (hundreds of values tied at the top) finds its top n one by one, each the
// best rank key after the last. 1024 bf16
// rows of V 128256, top 5: 99.8 us on the sliced path (85 + 18) -> 55.1, 4.8 TB/s.
constexpr int kLpThreads = 512;
constexpr uint32_t kLpLanes = 64, kLpCand = 256;   // lanes read again, candidates ranked
template <int G, RowForm F>
__global__ __launch_bounds__(kLpThreads) void logprobs_kernel(LogprobArgs a) {
    constexpr int NT = kLpThreads, NW = NT / kWave;
    __shared__ float redf[NW];
    __shared__ uint32_t redu[NW];
    __shared__ double redd[NW];
    __shared__ uint64_t redk[NW];
    __shared__ float lmax[NT];
    __shared__ uint32_t nl, nc, lanes[kLpLanes];
    __shared__ uint64_t ck[kLpCand];
    __shared__ double log_z_s;
    const uint32_t tid = tid_x(), row = wg_x();
    const int lane = lane_id(), wv = __builtin_amdgcn_readfirstlane((int)(tid / kWave));
    if (row >= a.rows) return;
    const uint32_t V = a.vocab, ng = (V + G - 1) / G, ntop = a.n_top;
    const void* rowp = static_cast<const char*>(a.logits) + (uint64_t)row * a.row_stride * (16u / G);
    const RowLane l = stream_row<G, NT, F>(rowp, V);
    lmax[tid] = l.om;
    if (tid == 0) { nl = 0u; nc = 0u; }
    float bm;
    uint32_t idx;
    const double z = reduce_row<G, NT>(l, rowp, V, bm, idx, redf, redu, redd);   // (its barriers order lmax, nl, nc)
    if (tid == 0) {
        const double log_z = log(z) + (double)bm;
        log_z_s = log_z;
        const uint32_t am = idx < V ? idx : 0u;
        if (a.ids) a.ids[row] = (int32_t)am;
        const int32_t d = a.chosen ? a.chosen[row] : (int32_t)am;
        const bool in = d >= 0 && (uint32_t)d < V;
        a.chosen_lp[row] = in ? (float)((double)load_elem(rowp, G == 8 ? LCS_BF16 : LCS_F32, (uint32_t)d) - log_z) : 0.0f;
    }
    if (ntop == 0u) return;   // (uniform)
    float m = lmax[lane];
#pragma unroll
    for (int w = 1; w < NW; ++w) m = fmaxf(m, lmax[lane + w * kWave]);
    // (every wave finds the same bound, the keys cut to 16 bits from below)
    const uint32_t k1 = fkey(m) >> 16;
    uint32_t T = 0;
#pragma unroll
    for (int sh = 14; sh >= 0; sh -= 2) {
        const uint32_t T1 = T | (1u << sh), T2 = T | (2u << sh), T3 = T | (3u << sh);
        const uint32_t c1 = (uint32_t)__builtin_popcountll(ballot(k1 >= T1));
        const uint32_t c2 = (uint32_t)__builtin_popcountll(ballot(k1 >= T2));
        const uint32_t c3 = (uint32_t)__builtin_popcountll(ballot(k1 >= T3));
        T = c3 >= ntop ? T3 : c2 >= ntop ? T2 : c1 >= ntop ? T1 : T;
    }
    const float t = key_to_f(max(T << 16, 0x007fffffu));   // (>= -inf)
    if (l.om >= t) {
        const uint32_t s = atomicAdd(&nl, 1u);
        if (s < kLpLanes) lanes[s] = tid;
    }
    __syncthreads();
    const uint32_t n_lanes = nl;
    if (n_lanes <= kLpLanes) {
        for (uint32_t i = (uint32_t)wv; i < n_lanes; i += NW) {
            for (uint32_t g = lanes[i] + (uint32_t)lane * NT; g < ng; g += kWave * NT) {
                float v[G];
                decode<G>(load16(rowp, g), v);
#pragma unroll
                for (int k = 0; k < G; ++k) {
                    if (v[k] >= t && g * G + k < V) {
                        const uint32_t s = atomicAdd(&nc, 1u);
                        if (s < kLpCand) ck[s] = rank_key(v[k], g * G + k);
                    }
                }
            }
        }
    }
    __syncthreads();
    const double log_z = log_z_s;
    auto put = [&](uint32_t r, uint64_t key) {
        a.top_ids[(uint64_t)row * ntop + r] = (int32_t)rank_idx(key);
        a.top_lp[(uint64_t)row * ntop + r] = (float)((double)rank_val(key) - log_z);
    };
    const uint32_t have = min(ntop, V);   // (past the vocabulary: no key)
    if (n_lanes <= kLpLanes && nc <= kLpCand) {   // (uniform)
        if (wv == 0) {
            uint64_t k[4];
            uint32_t rk[4];
            lds_rank4(ck, nc, k, rk);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if ((uint32_t)lane + (uint32_t)c * kWave < nc && rk[c] < ntop) put(rk[c], k[c]);
            }
        }
    } else {
        uint64_t last = 0ull;
        for (uint32_t r = 0; r < have; ++r) {
            uint64_t best = ~0ull;
            for (uint32_t g = tid; g < ng; g += NT) {
                float v[G];
                decode<G>(load16(rowp, g), v);
#pragma unroll
                for (int k = 0; k < G; ++k) {
                    const uint64_t key = rank_key(v[k], g * G + k);
                    if (g * G + k < V && (r == 0u || key > last)) best = u64_min(best, key);
                }
            }
            last = block_min_u64<NT>(best, redk);
            if (tid == 0) put(r, last);
        }
    }
    if (wv == 0 && (uint32_t)lane >= have && (uint32_t)lane < ntop) put((uint32_t)lane, ~0ull);
}

template <int G>
static void launch_lp(const LogprobArgs& a, hipStream_t st) {
    const dim3 grid(a.rows), block(kLpThreads);
    const RowForm f = row_form<G>(a.vocab, kLpThreads);
    if (f == kRowRounds) hipLaunchKernelGGL((logprobs_kernel<G, kRowRounds>), grid, block, 0, st, a);
    else if (f == kRowTail) hipLaunchKernelGGL((logprobs_kernel<G, kRowTail>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((logprobs_kernel<G, kRowShort>), grid, block, 0, st, a);
}

hipError_t launch_logprobs(const LogprobArgs& a, uint32_t dtype, hipStream_t st) {
    if (dtype == LCS_BF16) launch_lp<8>(a, st);
    else launch_lp<4>(a, st);
    return hipGetLastError();
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

template <int G, int NT>
static void launch_nt(const VerifyArgs& a, uint32_t rows, hipStream_t st) {
    const RowForm f = row_form<G>(a.vocab, NT);
    if constexpr (NT == 256) {   // (512 threads take long rows only)
        if (f == kRowShort) {
            hipLaunchKernelGGL((verify_kernel<G, NT, kRowShort>), dim3(rows), dim3(NT), 0, st, a);
            return;
        }
    }
    if (f == kRowRounds) hipLaunchKernelGGL((verify_kernel<G, NT, kRowRounds>), dim3(rows), dim3(NT), 0, st, a);
    else hipLaunchKernelGGL((verify_kernel<G, NT, kRowTail>), dim3(rows), dim3(NT), 0, st, a);
}

// Threads per row (us a call with 256 / 512 threads). Up to a row a CU, a row
// of more than two rounds of 512 threads takes 512: f32, V 128256, 16 rows 14.3
// / 12.3, 128 rows 19.0 / 15.2, 200 rows 20.2 / 19.9 (256 rows 23.2 / 24.1);
// bf16, V 128256, 128 rows 14.9 / 12.7, 256 rows 16.9 / 15.4, V 70000, 16 rows
// 9.4 / 9.0. Above, smaller workgroups even the CUs out (f32, V 128256, 300 rows
// 27.9 / 32.9, 512 rows 42.7 / 45.2; bf16, V 163840, 300 rows 23.5 / 26.2, 1024
// rows 59.3 / 60.7; 2048 rows of V 5000 10.1 / 16.7), except for thousands of
// long bf16 rows (V 163840, 1536 rows 93.1 / 90.7, 4096 rows 229.7 / 228.8).
template <int G>
static void launch_rows(const VerifyArgs& a, hipStream_t st) {
    const uint32_t rows = a.n_seq * a.rows_per_seq, ng = (a.vocab + G - 1u) / G;
    const bool wide = ng > 8192u && (rows <= 256u || (G == 8 && rows > 1024u && ng > 16384u));
    if (wide) launch_nt<G, 512>(a, rows, st);
    else launch_nt<G, 256>(a, rows, st);
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
