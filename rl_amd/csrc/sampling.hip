// K3: token logprobs under top-k / top-p (nucleus) filtering, forward and backward, for gfx950.
//
// The reference sorts every 151 936-wide row (values + int64 indices).  Here one workgroup of 256
// threads owns a row and never sorts it:
//   pass 1 (HBM)   streams the row keeping 2048 chunk maxima in registers (and, when the caller
//                  wants the unfiltered logprob too, the online log-sum-exp of the full row); a chunk
//                  is a set of whole 128-byte lines, so that what pass 2 re-reads is all used;
//   select         the k-th largest chunk maximum is a lower bound of the k-th largest element
//                  (found two bits per round with wave ballots, the maxima staying in registers);
//                  for top-p alone the bound starts at lse + log((1-p)/V) (everything below it is
//                  dropped whatever the order) and is raised with a 64-bin histogram of probability
//                  over log-probability, filled from the chunk maxima and, only if that is not
//                  enough, from the row read once more;
//   pass 2         re-reads only the chunks whose maximum reaches the bound (about k of 2048) and
//                  appends the elements above the bound to an LDS list;
//   finish         the list put in order by (value, index), top-k threshold with ties kept,
//                  softmax over the kept values, ascending cumulative mass > 1 - top_p, the
//                  renormalised log-sum-exp, the target's logprob (-inf when it was filtered).
// Per row the forward saves (threshold value, tie index, kept log-sum-exp): element v is kept iff
// x_v > thr, or x_v == thr and v >= tie index.  Among exactly tied values at the top-p boundary the
// larger vocabulary indices survive (ascending stable order); all ties at the top-k threshold are
// kept.  The backward streams the row once more: d_v = keep_v * g * (onehot_v - exp(x_v - lse_kept)).
//
// Rows whose candidate list would exceed the LDS capacity (very flat distributions under top-p
// alone, thousands of exact ties, or a top_k in the thousands) are marked and finished by
// topk_topp_wide_kernel, which finds the same predicate by a radix descent over the row's order keys
// (a histogram pass per key digit: two to three passes for 16-bit logits).
//
// bf16 rows under top-p alone take none of this: nucleus_count_kernel counts the elements of every value.

#include <float.h>
#include <math.h>

#include <type_traits>

#include "common.hpp"

namespace nrl {

constexpr int kSelBlock = 256;
constexpr int kSelWaves = kSelBlock / kWave;
constexpr int kMassBins = 64;
constexpr int kLooseHits = 768;  // top-p alone: more hit chunks than this under the chunk maxima's bound -> bound from the row
constexpr int kMassCopies = 8;  // copies of the histogram, by lane: most elements fall into the few lowest bins
constexpr int kWideGrid = 2048;  // workgroups of the kernel that finishes the marked rows
constexpr int32_t kTieUnresolved = -1;  // tie[] marker: the row's kept set did not fit the candidate list
constexpr int32_t kTieNoCut = 0x7fffffff;  // tie[] marker: a bf16 row with +inf under top-p alone, of which nothing falls (its masses are NaN)
constexpr int kSub = 8;                      // chunk maxima per thread
constexpr int kChunks = kSelBlock * kSub;    // 2048
constexpr int kCap = 4096;                   // candidate capacity (LDS); rows under a small top-k use kCapSmall
constexpr int kCapSmall = 2048;              // ... which lets six workgroups share a compute unit instead of three
constexpr int kSmallTopK = 512;

struct Lse2 {
    float m, s;
};
__device__ __forceinline__ Lse2 lse2_merge(Lse2 a, Lse2 b) {
    const float m = fmaxf(a.m, b.m);
    Lse2 r;
    r.m = m;
    r.s = a.s * fast_exp2((a.m - m) * kLog2e) + b.s * fast_exp2((b.m - m) * kLog2e);
    return r;
}

// monotone map float -> uint32 (larger float, larger key)
__device__ __forceinline__ uint32_t order_key(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// maximum over the 8 consecutive lanes (aligned to 8) that read one 128-byte line; every lane returns it
// (written as three hand-placed v_max_f32_dpp the pass has a third fewer vector instructions and takes the same time)
__device__ __forceinline__ float line_max(float v) {
    int x = __float_as_int(v);
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(x, x, 0xB1, 0xF, 0xF, false)));   // quad_perm [1,0,3,2]
    x = __float_as_int(v);
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(x, x, 0x4E, 0xF, 0xF, false)));   // quad_perm [2,3,0,1]
    x = __float_as_int(v);
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(x, x, 0x141, 0xF, 0xF, false)));  // row_half_mirror
}

template <int DT> __device__ __forceinline__ int64_t sel_row_head(const void* row, int64_t vocab) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(row);
    const int64_t h = static_cast<int64_t>(((16 - (a & 15)) & 15) / Row<DT>::BYTES);
    return h < vocab ? h : vocab;
}

template <int CAP> struct SelShared {
    unsigned long long cand[CAP];
    float expv[CAP];
    int sel_cnt[2][kSelWaves * 3];
    Lse2 lse_w[kSelWaves];
    int count;
    float mass_bin[kMassCopies * kMassBins];  // top-p alone: probability mass per log-probability bin
    int n_hit;  // chunks whose maximum reaches the bound (their list lives in expv until the finish phase)
};

// k-th largest (1-based) of the workgroup's kChunks keys (kSub per thread, in registers), or a little less; every thread
// returns it.  Two bits at a time from the top: the answer is the largest v with at least k keys >= v, v a multiple of
// 2^LOW, below which the keys of a 16-bit type are constant (eight and ten rounds for bf16 and fp16).  The 32 bits of fp32 end
// where going on would leave out k / 32 + 2 keys at most: about ten rounds for logits of ordinary size, up to sixteen where
// they share their leading bits (a fixed 20 bits let a whole row pass the bound at logits around 1e4: 1000 rows of V = 151 936,
// top-k 50 110 us, 564 by way of the wide kernel).  A round costs 3 * kSub ballots per wave, three LDS words per wave and one
// barrier (the buffers alternate), with no atomics -- chunk maxima share their high bits, so a histogram would serialise on
// one bin.
template <int DT> constexpr int kSelectLow = DT == NRL_BF16 ? 16 : DT == NRL_F16 ? 12 : 0;
template <int LOW, int CAP>
__device__ __forceinline__ uint32_t select_kth_largest(SelShared<CAP>& sh, const uint32_t (&keys)[kSub], int k) {
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    uint32_t v = 0u;
    // (v = 0 is no answer: it would let -inf through; every key, of chunks without elements too, is above that)
    int at_or_above = 0x7fffffff;
    // two bits per round: three trial values, one barrier
    for (int bit = 30; bit >= LOW && (LOW > 0 || at_or_above > k + k / 32 + 2); bit -= 2) {
        int cnt[3] = {0, 0, 0};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const uint32_t cand = v | (static_cast<uint32_t>(c + 1) << bit);
#pragma unroll
            for (int u = 0; u < kSub; ++u) cnt[c] += __popcll(__ballot(keys[u] >= cand));
        }
        const int par = (bit >> 1) & 1;
        if (lane < 3) sh.sel_cnt[par][wave * 3 + lane] = lane == 0 ? cnt[0] : lane == 1 ? cnt[1] : cnt[2];
        __syncthreads();
        int tot[3] = {0, 0, 0};
#pragma unroll
        for (int w = 0; w < kSelWaves; ++w)
#pragma unroll
            for (int c = 0; c < 3; ++c) tot[c] += sh.sel_cnt[par][w * 3 + c];
        // counts fall as the trial value rises: take the largest trial that still has k keys at or above it
        const uint32_t step = tot[2] >= k ? 3u : tot[1] >= k ? 2u : tot[0] >= k ? 1u : 0u;
        v |= step << bit;
        at_or_above = step == 3u ? tot[2] : step == 2u ? tot[1] : step == 1u ? tot[0] : at_or_above;
    }
    return v;
}

// inclusive sum over the lanes up to this one, by lane moves
__device__ __forceinline__ double wave_scan_double(double v) {
    auto add = [&](auto ctrl, int rows) {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        constexpr int CTRL = decltype(ctrl)::value;
        const int lo = static_cast<int>(u), hi = static_cast<int>(u >> 32);
        uint32_t l, h;  // lanes outside the move bring zero
        if (rows == 0xf) { l = __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xf, 0xf, false); h = __builtin_amdgcn_update_dpp(0, hi, CTRL, 0xf, 0xf, false); }
        else if (rows == 0xa) { l = __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xa, 0xf, false); h = __builtin_amdgcn_update_dpp(0, hi, CTRL, 0xa, 0xf, false); }
        else { l = __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xc, 0xf, false); h = __builtin_amdgcn_update_dpp(0, hi, CTRL, 0xc, 0xf, false); }
        v += __builtin_bit_cast(double, (static_cast<uint64_t>(h) << 32) | l);
    };
    add(std::integral_constant<int, 0x111>{}, 0xf);  // row_shr 1, 2, 4, 8: sums inside the rows of 16 lanes
    add(std::integral_constant<int, 0x112>{}, 0xf);
    add(std::integral_constant<int, 0x114>{}, 0xf);
    add(std::integral_constant<int, 0x118>{}, 0xf);
    add(std::integral_constant<int, 0x142>{}, 0xa);  // row_bcast 15: the row before, to rows 1 and 3
    add(std::integral_constant<int, 0x143>{}, 0xc);  // row_bcast 31: the first two rows, to rows 2 and 3
    return v;
}

// sum of e[0 .. n) in double; called by every lane of one wave, which all return it
__device__ __forceinline__ float wave_sum_list(const float* e, int n) {
    double s = 0.0;
    for (int i = threadIdx.x & (kWave - 1); i < n; i += kWave) s += static_cast<double>(e[i]);
    return static_cast<float>(wave_sum_double(s));
}

// descending bitonic sort of list[0 .. n_pad) in LDS by a workgroup of THREADS; n_pad is a power of two
template <int THREADS> __device__ __forceinline__ void sort_list_desc(unsigned long long* list, int n_pad) {
    const int tid = threadIdx.x;
    for (int size = 2; size <= n_pad; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            __syncthreads();
            for (int i = tid; i < (n_pad >> 1); i += THREADS) {
                const int lo = ((i / stride) * (stride << 1)) + (i % stride);
                const int hi = lo + stride;
                const bool desc = ((lo & size) == 0);
                const unsigned long long a = list[lo], b = list[hi];
                if ((a < b) == desc) { list[lo] = b; list[hi] = a; }
            }
        }
    }
    __syncthreads();
}

// The same for at most THREADS entries, no two of them equal: an entry's place is the number of larger ones.  n LDS reads in a
// row, the same word for all lanes, where a sort takes an LDS round trip or a barrier for each of its steps.  With this, the
// shorter selection above and the target's logit loaded early, forwards under top-k and top-p take (us, before and now): 4095
// rows of V = 151 936 bf16, k 50 213 and 206; 500 rows of 32 000, k 50 26.6 and 20.4; 4000 rows of 32 000, k 100 111 and 86.
template <int THREADS> __device__ __forceinline__ void rank_list_desc(unsigned long long* list, int n) {
    const int tid = threadIdx.x;
    __syncthreads();
    unsigned long long c = 0ull;
    int at = 0;
    if (tid < n) {
        c = list[tid];
#pragma unroll 8
        for (int i = 0; i < n; ++i) at += list[i] > c ? 1 : 0;
    }
    __syncthreads();
    if (tid < n) list[at] = c;
    __syncthreads();
}

struct SelArgs {
    const void* logits;
    int64_t n_inner, vocab, stride_outer, stride_inner;
    const int64_t* targets;  // may be NULL (filter only)
    int64_t ts_outer, ts_inner;
    float tparam;
    int top_k;    // <= 0: off
    float top_p;  // >= 1: off
    float* logprob;      // [rows] or NULL
    float* thr;          // [rows]
    int32_t* tie;        // [rows]
    float* lse_kept;     // [rows]
    float* logprob_full; // [rows] or NULL: unfiltered logprob of the target
    float* lse_full;     // [rows] or NULL
    // the kept set itself, for a backward that does not read the row again (all three NULL: not recorded):
    int32_t* kept_n;     // [rows] number of kept elements, -1 if they do not fit kept_cap (or the row was left to the wide kernel)
    int32_t* kept_idx;   // [rows, kept_cap] their vocabulary indices, in descending (value, index) order
    float* kept_x;       // [rows, kept_cap] their (scaled) logits
    int kept_cap;
};

// PONLY: top-p without top-k (its own instantiation, so that the mass histogram costs the top-k variants
// neither registers nor LDS); otherwise top-k is on, with or without top-p.
template <int DT, int TEMP, bool FULL_LSE, int CAP, bool PONLY = false>
__global__ __launch_bounds__(kSelBlock) void topk_topp_fwd_kernel(SelArgs a) {
    static_assert(!PONLY || FULL_LSE, "top-p alone normalises over the whole row");
    __shared__ SelShared<CAP> sh;
    constexpr int EPV = Row<DT>::EPV;
    const int tid = threadIdx.x;
    const int64_t r = blockIdx.x;
    const uint32_t o = blockIdx.x / static_cast<uint32_t>(a.n_inner);  // (fewer than 2^31 rows)
    const int64_t i_in = blockIdx.x - o * static_cast<uint32_t>(a.n_inner);
    const char* row = static_cast<const char*>(a.logits) + (o * a.stride_outer + i_in * a.stride_inner) * Row<DT>::BYTES;
    const int64_t vocab = a.vocab;
    const int64_t head = sel_row_head<DT>(row, vocab);
    const int64_t nvec = (vocab - head) / EPV;
    const int64_t tail0 = head + nvec * EPV;
    const u32x4* xv = reinterpret_cast<const u32x4*>(row + head * Row<DT>::BYTES);

    // the target's logit, on its way while the row streams
    int64_t tg = -1;
    float x_tg = 0.f;
    if (a.targets && a.logprob) {
        tg = a.targets[o * a.ts_outer + i_in * a.ts_inner];
        if (tg >= 0 && tg < vocab) x_tg = Row<DT>::load1(row, tg);
    }

    // ---- pass 1: chunk maxima (+ full-row online log-sum-exp) ----
    // Without the full-row log-sum-exp only maxima leave this pass, and the temperature scaling (a multiplication or
    // division by a positive number, then rounding to the logits' dtype) is monotone: the maximum of the scaled
    // values is the scaled maximum, so the raw values are compared and each chunk maximum is scaled once at the end.
    constexpr bool LATE_SCALE = !FULL_LSE && TEMP != 0;
    auto scaled = [&](float x) { return LATE_SCALE ? x : scale_logit<DT, TEMP>(x, a.tparam); };
    float mx[kSub];
#pragma unroll
    for (int u = 0; u < kSub; ++u) mx[u] = -FLT_MAX;
    Lse2 acc;
    acc.m = -FLT_MAX;
    acc.s = 0.f;
    // A chunk is a set of whole 128-byte lines: the 8 lanes that read one line together reduce their maxima over
    // the line, and lane j of the 8 keeps the lines of the iterations i with i % 8 == j.  The second pass then
    // re-reads full lines; with a chunk per thread it re-read 16 bytes of a line at a time, and every such piece
    // cost the whole line in HBM traffic.
    const int lane8 = tid & 7;
    int64_t base = 0;
    int iter = 0;
    for (; base + kSub * kSelBlock <= nvec; base += kSub * kSelBlock, ++iter) {
        u32x4 q[kSub];
#pragma unroll
        for (int u = 0; u < kSub; ++u) q[u] = __builtin_nontemporal_load(xv + base + u * kSelBlock + tid);
        const bool mine = (iter & 7) == lane8;
        float v[kSub * EPV];
        float vm_all = -FLT_MAX;
#pragma unroll
        for (int u = 0; u < kSub; ++u) {
            float t[EPV];
            Row<DT>::decode(q[u], t);
            float vm = -FLT_MAX;
#pragma unroll
            for (int k = 0; k < EPV; ++k) {
                t[k] = scaled(t[k]);
                v[u * EPV + k] = t[k];
                vm = fmaxf(vm, t[k]);
            }
            vm_all = fmaxf(vm_all, vm);
            const float lm = line_max(vm);
            mx[u] = fmaxf(mx[u], mine ? lm : -FLT_MAX);
        }
        if (FULL_LSE) {
            const float mn = fmaxf(acc.m, vm_all);
            float part = 0.f;
#pragma unroll
            for (int k = 0; k < kSub * EPV; ++k) part += fast_exp2((v[k] - mn) * kLog2e);
            acc.s = acc.s * fast_exp2((acc.m - mn) * kLog2e) + part;
            acc.m = mn;
        }
    }
    // the ragged end of the row, one more iteration with fewer than kSub vectors per thread: the same chunks
    {
        const bool mine = (iter & 7) == lane8;
#pragma unroll
        for (int u = 0; u < kSub; ++u) {
            const int64_t vi = base + u * kSelBlock + tid;
            float vm = -FLT_MAX;
            if (vi < nvec) {
                float t[EPV];
                Row<DT>::decode(xv[vi], t);
#pragma unroll
                for (int k = 0; k < EPV; ++k) {
                    t[k] = scaled(t[k]);
                    vm = fmaxf(vm, t[k]);
                    if (FULL_LSE) {
                        const float mn = fmaxf(acc.m, t[k]);
                        acc.s = acc.s * fast_exp2((acc.m - mn) * kLog2e) + fast_exp2((t[k] - mn) * kLog2e);
                        acc.m = mn;
                    }
                }
            }
            const float lm = line_max(vm);  // by every lane: lanes past the end bring the identity
            mx[u] = fmaxf(mx[u], mine ? lm : -FLT_MAX);
        }
    }
    {
        const int64_t e0 = tid < head ? tid : -1;
        const int64_t e1 = tail0 + tid < vocab ? tail0 + tid : -1;
        for (int w = 0; w < 2; ++w) {
            const int64_t e = w == 0 ? e0 : e1;
            if (e < 0) continue;
            const float x = scaled(Row<DT>::load1(row, e));
            mx[0] = fmaxf(mx[0], x);
            if (FULL_LSE) {
                const float mn = fmaxf(acc.m, x);
                acc.s = acc.s * fast_exp2((acc.m - mn) * kLog2e) + fast_exp2((x - mn) * kLog2e);
                acc.m = mn;
            }
        }
    }
    if (LATE_SCALE) {
#pragma unroll
        for (int u = 0; u < kSub; ++u) mx[u] = scale_logit<DT, TEMP>(mx[u], a.tparam);
    }
    uint32_t mx_key[kSub];
#pragma unroll
    for (int u = 0; u < kSub; ++u) mx_key[u] = order_key(mx[u]);
    float lse_full = 0.f;
    if (FULL_LSE) {
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) {
            Lse2 other;
            other.m = __shfl_xor(acc.m, off, kWave);
            other.s = __shfl_xor(acc.s, off, kWave);
            acc = lse2_merge(acc, other);
        }
        if ((tid & (kWave - 1)) == 0) sh.lse_w[tid / kWave] = acc;
    }
    if (tid == 0) { sh.count = 0; sh.n_hit = 0; }
    __syncthreads();
    if (FULL_LSE) {
        Lse2 tot = sh.lse_w[0];
#pragma unroll
        for (int w = 1; w < kSelWaves; ++w) tot = lse2_merge(tot, sh.lse_w[w]);
        lse_full = tot.m + logf(tot.s);
    }

    // ---- lower bound of everything that can be kept ----
    constexpr bool use_k = !PONLY;
    const bool use_p = a.top_p < 1.0f;
    uint32_t bound_key = 0u;
    // top-p alone: elements with probability <= (1-p)/V sum to at most 1-p and are the smallest, which puts
    // a first bound b0 under the kept set; but a long tail leaves thousands of elements above b0.  The
    // probability of a set of elements above b0, sorted into kMassBins equal log-probability bins, gives a
    // better one: if the bins from j upwards already hold more than p of the row's mass, everything below
    // bin j weighs less than 1-p and cannot be kept.  First the set is the 2048 chunk maxima (already in
    // registers; enough whenever the kept set is a few hundred tokens), and only if that proves nothing or
    // leaves too many candidates the whole row, read once more.
    const float cut = 1.0f - a.top_p;
    const float span = logf(static_cast<float>(vocab) / cut);  // from probability (1-p)/V up to 1, in nats
    const float b0 = lse_full - span;
    // The bins start a quarter of the span above b0: an edge lower than that would keep thousands of tokens,
    // more than the list holds anyway, and the many elements just above b0 would each cost an LDS atomic.
    const float hb = b0 + 0.25f * span;
    const float to_bin = static_cast<float>(kMassBins) / (0.75f * span);
    auto bin = [&](float x) {
        if (x > hb) {
            const int j = static_cast<int>((x - hb) * to_bin);
            atomicAdd(&sh.mass_bin[(tid & (kMassCopies - 1)) * kMassBins + (j < kMassBins - 1 ? j : kMassBins - 1)], expf(x - lse_full));
        }
    };
    // called by every thread between two barriers around the binning; returns the bound (the same in all)
    auto bound_from_bins = [&]() -> uint32_t {
        // every wave: lane j takes bin j and the mass of the bins from j upwards.  The highest edge whose
        // mass below stays under 1-p (less a margin for the rounding of the sums: the list may hold more
        // than the kept set, never less) bounds the candidates; with none the bound stays at b0.
        static_assert(kMassBins == kWave, "one bin per lane");
        float above = 0.f;
#pragma unroll
        for (int q = 0; q < kMassCopies; ++q) above += sh.mass_bin[q * kMassBins + (tid & (kWave - 1))];
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const float up = __shfl_down(above, off, kWave);
            if ((tid & (kWave - 1)) + off < kWave) above += up;
        }
        const unsigned long long ok = __ballot(1.0f - above <= cut * 0.999f - 1e-5f);
        const int edge = ok ? 63 - __builtin_clzll(ok) : 0;
        // just under the edge, so that an element the rounding of its bin number put into bin `edge` counts
        return ok ? order_key(hb + (static_cast<float>(edge) - 0.01f) / to_bin) : order_key(b0) + 1u;
    };
    auto clear_bins = [&]() {
        for (int i = tid; i < kMassCopies * kMassBins; i += kSelBlock) sh.mass_bin[i] = 0.f;
    };
    auto bound_from_row = [&]() -> uint32_t {
        clear_bins();
        __syncthreads();
        for (int64_t vb = 0; vb < nvec; vb += kSub * kSelBlock) {  // kSub loads in flight per thread
            u32x4 q[kSub];
#pragma unroll
            for (int u = 0; u < kSub; ++u) {
                const int64_t vi = vb + u * kSelBlock + tid;
                if (vi < nvec) q[u] = xv[vi];
            }
#pragma unroll
            for (int u = 0; u < kSub; ++u) {
                if (vb + u * kSelBlock + tid >= nvec) continue;
                float t[EPV];
                Row<DT>::decode(q[u], t);
#pragma unroll
                for (int k = 0; k < EPV; ++k) bin(scale_logit<DT, TEMP>(t[k], a.tparam));
            }
        }
        if (tid < head) bin(scale_logit<DT, TEMP>(Row<DT>::load1(row, tid), a.tparam));
        if (tail0 + tid < vocab) bin(scale_logit<DT, TEMP>(Row<DT>::load1(row, tail0 + tid), a.tparam));
        __syncthreads();
        return bound_from_bins();
    };
    bool whole_row = true;  // top-p alone: the bound already rests on the whole row
    bool force_wide = false;  // top-p alone: the chunk maxima show that the kept set cannot fit the candidate list
    if (use_k) {
        if (a.top_k <= kChunks) bound_key = select_kth_largest<kSelectLow<DT>>(sh, mx_key, a.top_k);
    } else {
        clear_bins();
        // (how many elements the chunks hold whose maxima fall into each bin, and what they would weigh if each
        // weighed as much as its chunk's maximum, is summed too, in integers: see below)
        int* max_cnt = reinterpret_cast<int*>(sh.cand);  // the candidate list is not in use yet
        unsigned long long* max_w = sh.cand + kMassBins;  // 32.32 fixed point
        if (tid <= kMassBins) { max_cnt[tid] = 0; max_w[tid] = 0ull; }
        __syncthreads();
        {
            // this lane's chunks are the lines of the iterations i = lane8, lane8 + 8, ... <= n_full (the ragged last
            // iteration counted whole); chunk 0 also took one element of the unaligned head and of the tail
            const int n_full_iter = static_cast<int>(nvec / (kSub * kSelBlock));
            const int lines = n_full_iter >= lane8 ? (n_full_iter - lane8) / 8 + 1 : 0;
#pragma unroll
            for (int u = 0; u < kSub; ++u) {
                bin(mx[u]);
                const int elems = lines * 8 * EPV + (u == 0 ? 2 : 0);
                int j = kMassBins;  // maxima under the first bin's lower edge
                if (mx[u] > hb) {
                    j = static_cast<int>((mx[u] - hb) * to_bin);
                    j = j < kMassBins - 1 ? j : kMassBins - 1;
                }
                atomicAdd(&max_cnt[j], elems);
                const float w = expf(fminf(mx[u] - lse_full, 0.f)) * 4294967296.0f;  // NaN (no finite row sum) -> 0
                atomicAdd(&max_w[j], static_cast<unsigned long long>(w) * static_cast<unsigned long long>(elems));
            }
        }
        __syncthreads();
        bound_key = bound_from_bins();
        whole_row = bound_key == order_key(b0) + 1u;  // the maxima alone prove nothing: go to the row at once
        if (whole_row) {
            // A row whose kept set cannot fit the candidate list is not worth the two passes that would find that
            // out.  No element outweighs the maximum of its chunk, so the CAP heaviest elements of the row weigh at
            // most what all elements of the chunks with the heaviest maxima would, taken chunk by chunk until CAP
            // elements are reached, each at its chunk's maximum; if even that stays under top_p, more than CAP
            // elements are kept and the row goes to the wide kernel now.  Counts and weights are summed as integers,
            // so the decision does not depend on the order in which atomics arrived (both paths find the same kept
            // set up to near-equal elements at the boundary, but a row should take the same path every time).
            static_assert(kMassBins == kWave, "one bin per lane");
            const int lane_b = tid & (kWave - 1);
            int c_above = max_cnt[lane_b];   // becomes: elements of the chunks whose maxima lie in bins >= lane_b
            unsigned long long w_above = max_w[lane_b];  // their weight, each element at its chunk's maximum
#pragma unroll
            for (int off = 1; off < kWave; off <<= 1) {
                const int cu = __shfl_down(c_above, off, kWave);
                const unsigned long long wu = __shfl_down(w_above, off, kWave);
                if (lane_b + off < kWave) { c_above += cu; w_above += wu; }
            }
            const unsigned long long enough = __ballot(c_above >= CAP);
            const int jstar = enough ? 63 - __builtin_clzll(enough) : 0;
            const float w_star = static_cast<float>(__shfl(w_above, jstar, kWave)) * (1.0f / 4294967296.0f);
            const int c_star = __shfl(c_above, jstar, kWave);
            // chunks whose maxima were not binned lie under hb
            float heaviest = w_star + static_cast<float>(c_star < CAP ? CAP - c_star : 0) * expf(hb - lse_full);
            if (enough) {
                // of bin jstar only as many elements as the list still has room for, each at the bin's upper edge
                const int up = jstar + 1 < kWave ? jstar + 1 : jstar;
                const unsigned long long w_up = __shfl(w_above, up, kWave);
                const int c_up = __shfl(c_above, up, kWave);
                const float w_next = jstar + 1 < kWave ? static_cast<float>(w_up) * (1.0f / 4294967296.0f) : 0.f;
                const int c_next = jstar + 1 < kWave ? c_up : 0;
                const float edge = jstar == kMassBins - 1 ? 0.f : fminf(hb + static_cast<float>(jstar + 1) / to_bin - lse_full, 0.f);
                heaviest = fminf(heaviest, w_next + static_cast<float>(CAP - c_next) * expf(edge));
            }
            force_wide = heaviest < 0.98f * a.top_p;
            if (!force_wide) {
                __syncthreads();  // every wave is done with the bins
                bound_key = bound_from_row();
            }
        }
    }

    // ---- pass 2: collect candidates (top-p alone: once more with the bound from the whole row if the list
    // did not hold what the chunk maxima's bound lets through) ----
    int n = force_wide ? CAP + 1 : 0;
    for (; !force_wide;) {
    // Only the chunks whose maximum reaches the bound can hold candidates (with top-k that is about k of the
    // 2048 chunks, a few percent of the row).
    auto push = [&](uint32_t key, int64_t index) {
        if (key >= bound_key) {
            const int pos = atomicAdd(&sh.count, 1);
            if (pos < CAP) sh.cand[pos] = (static_cast<unsigned long long>(key) << 32) | static_cast<uint32_t>(index);
        }
    };
    auto push_raw = [&](const u32x4& q, int vi) {
        float t[EPV];
        Row<DT>::decode(q, t);
#pragma unroll
        for (int k = 0; k < EPV; ++k) push(order_key(scale_logit<DT, TEMP>(t[k], a.tparam)), head + vi * EPV + k);
    };
    // The hit chunks go to a list and their vectors are then dealt out evenly, a few per thread with the
    // loads in flight together: a thread that re-read only its own hit chunks left most lanes of a wave
    // idle through several thousand instructions, which cost more than the streaming pass.
    static_assert(kChunks <= 65536 && kChunks * 2 <= CAP * 4, "the hit list is 16-bit chunk ids inside expv");
    uint16_t* hit = reinterpret_cast<uint16_t*>(sh.expv);
#pragma unroll
    for (int u = 0; u < kSub; ++u)
        if (mx_key[u] >= bound_key) hit[atomicAdd(&sh.n_hit, 1)] = static_cast<uint16_t>(tid * kSub + u);
    if (mx_key[0] >= bound_key) {  // chunk 0 also took the unaligned head / tail elements
        if (tid < head) push(order_key(scale_logit<DT, TEMP>(Row<DT>::load1(row, tid), a.tparam)), tid);
        if (tail0 + tid < vocab)
            push(order_key(scale_logit<DT, TEMP>(Row<DT>::load1(row, tail0 + tid), a.tparam)), tail0 + tid);
    }
    __syncthreads();
    if (!use_k && !whole_row && sh.n_hit > kLooseHits) {
        // the bound from the chunk maxima lets too many chunks through: the row's own is worth its pass
        __syncthreads();  // every thread has read the hit count
        if (tid == 0) { sh.count = 0; sh.n_hit = 0; }
        whole_row = true;
        bound_key = bound_from_row();
        continue;
    }
    const int n_full = static_cast<int>(nvec / (kSub * kSelBlock));  // whole iterations of pass 1; number n_full is the ragged end
    const int per_chunk = ((n_full + 8) / 8) * 8;  // a line (8 vectors) per iteration the chunk's lane took
    const int n_items = sh.n_hit * per_chunk;
    // vector index of item number `item`, or -1 (an iteration past the end, or a vector past the row's)
    auto item_vec = [&](int item) -> int64_t {
        if (item >= n_items) return -1;
        const int h = item / per_chunk, rem = item - h * per_chunk;
        const int cu = hit[h], t = cu / kSub, u = cu - t * kSub;
        const int i = (t & 7) + (rem & ~7);  // iteration (rem / 8) of those with i % 8 == t % 8
        if (i > n_full) return -1;
        const int64_t vi = i * static_cast<int64_t>(kSub * kSelBlock) + u * kSelBlock + (t & ~7) + (rem & 7);
        return vi < nvec ? vi : -1;
    };
    constexpr int kBatch = 4;
    for (int i0 = tid; i0 < n_items; i0 += kBatch * kSelBlock) {
        // a list that has overflowed is not used (the bound is raised, or the row goes to the wide kernel): stop feeding
        // it -- on a flat row every element would otherwise queue up on the one counter
        if (*reinterpret_cast<volatile int*>(&sh.count) > CAP) break;
        int64_t vi[kBatch];
        u32x4 q[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            vi[j] = item_vec(i0 + j * kSelBlock);
            if (vi[j] >= 0) q[j] = xv[vi[j]];
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j)
            if (vi[j] >= 0) push_raw(q[j], vi[j]);
    }
    __syncthreads();
    n = sh.count;
    if (use_k || whole_row || n <= CAP) break;
    __syncthreads();  // every thread has read the count
    if (tid == 0) { sh.count = 0; sh.n_hit = 0; }
    whole_row = true;
    bound_key = bound_from_row();
    }
    if (n > CAP || n == 0) {
        // the kept set does not fit the candidate list (or the row holds no finite value); the kernel that finishes
        // such a row finds its largest (scaled) logit in thr
        float row_max = mx[0];
#pragma unroll
        for (int u = 1; u < kSub; ++u) row_max = fmaxf(row_max, mx[u]);
        row_max = wave_max(row_max);
        __syncthreads();
        if ((tid & (kWave - 1)) == 0) sh.lse_w[tid / kWave].m = row_max;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kSelWaves; ++q) row_max = fmaxf(row_max, sh.lse_w[q].m);
        if (tid == 0) {
            a.thr[r] = n > CAP ? row_max : __builtin_nanf("");
            a.tie[r] = n > CAP ? kTieUnresolved : 0;  // unresolved rows are finished by topk_topp_wide_kernel
            a.lse_kept[r] = __builtin_nanf("");
            if (a.logprob) a.logprob[r] = __builtin_nanf("");
            if (a.lse_full) a.lse_full[r] = lse_full;
            if (a.logprob_full) a.logprob_full[r] = __builtin_nanf("");
            if (a.kept_n) a.kept_n[r] = -1;
        }
        return;
    }
    if (n <= kSelBlock) {
        rank_list_desc<kSelBlock>(sh.cand, n);
    } else {
        int n_pad = 1;
        while (n_pad < n) n_pad <<= 1;
        for (int i = n + tid; i < n_pad; i += kSelBlock) sh.cand[i] = 0ull;  // sorts last
        sort_list_desc<kSelBlock>(sh.cand, n_pad);
    }

    // ---- top-k threshold (ties kept), softmax over the kept values ----
    int n_k = n;
    if (use_k) {
        const int kk = a.top_k < n ? a.top_k : n;
        const uint32_t thr_key = static_cast<uint32_t>(sh.cand[kk - 1] >> 32);
        int cnt = 0;
        for (int i = tid; i < n; i += kSelBlock) cnt += (static_cast<uint32_t>(sh.cand[i] >> 32) >= thr_key) ? 1 : 0;
        __shared__ int cnt_w[kSelWaves];
        n_k = block_sum<int, kSelWaves>(cnt, cnt_w);
    }
    const float m = key_value(static_cast<uint32_t>(sh.cand[0] >> 32));
    for (int i = tid; i < n_k; i += kSelBlock)
        sh.expv[i] = expf(key_value(static_cast<uint32_t>(sh.cand[i] >> 32)) - m);
    __syncthreads();
    // The masses are summed in double, by the lanes side by side: nearer to the sorted cumulative sum than fp32 in any order, where
    // element by element in fp32 is one dependent addition per element, three times (4000 rows of V = 32 000, top-k 100, top-p
    // 0.9: 86 -> 77 us).
    if (tid < kWave) {  // one wave; every lane computes the same scalars, lane 0 writes them
        int n_keep = n_k;
        if (use_p) {
            float s_k = wave_sum_list(sh.expv, n_k);
            // ascending cumulative probability, smallest kept value first; keep while it exceeds 1 - p
            const float cut = 1.0f - a.top_p;
            double run = 0.0;
            if (!use_k) {
                // top-p alone normalises over the whole row: the elements below the candidate bound
                // come first in ascending order and contribute their (small) mass to the running sum
                const float s_full = expf(lse_full - m);
                run = fmaxf(0.f, (s_full - s_k) / s_full);
                s_k = s_full;
            }
            // Elements fall, smallest first, while the running sum stays <= 1 - p; the sum only grows, so
            // counting the steps that end at or under the cut counts the fallen.  Whole blocks of 64, the last element in lane 0:
            // lanes past the end come first and add nothing (each counts as a step
            // under the cut and is taken off again), index 0 is always kept and never enters the sum.
            const int top_blk = (n_k - 1) / kWave;
            int steps_under = 0;
            for (int blk = top_blk; blk >= 0 && run <= cut; --blk) {  // (also leaves on a NaN)
                const int idx = blk * kWave + kWave - 1 - tid;
                const double v = wave_scan_double((idx >= 1 && idx < n_k) ? static_cast<double>(sh.expv[idx] / s_k) : 0.0);
                steps_under += __popcll(__ballot(run + v <= cut));
                run += lane_double(v, kWave - 1);
            }
            const int fallen = steps_under - ((top_blk + 1) * kWave - n_k);
            n_keep = n_k - fallen;
            if (n_keep < 1) n_keep = 1;
            if (n_keep > n_k) n_keep = n_k;
        }
        const float s = wave_sum_list(sh.expv, n_keep);
        const unsigned long long last = sh.cand[n_keep - 1];
        const uint32_t last_key = static_cast<uint32_t>(last >> 32);
        int tie = 0;
        if (n_keep < n && static_cast<uint32_t>(sh.cand[n_keep] >> 32) == last_key) tie = static_cast<int>(last & 0xffffffffu);
        const float thr = key_value(last_key), lse_kept = m + logf(s);
        if (a.kept_n && n_keep <= a.kept_cap) {
            for (int q = tid; q < n_keep; q += kWave) {
                const unsigned long long c = sh.cand[q];
                a.kept_idx[r * a.kept_cap + q] = static_cast<int32_t>(c & 0xffffffffu);
                a.kept_x[r * a.kept_cap + q] = key_value(static_cast<uint32_t>(c >> 32));
            }
        }
        if (tid == 0) {
            if (a.kept_n) a.kept_n[r] = n_keep <= a.kept_cap ? n_keep : -1;
            a.thr[r] = thr;
            a.tie[r] = tie;
            a.lse_kept[r] = lse_kept;
            if (a.lse_full) a.lse_full[r] = lse_full;
            if (a.targets && a.logprob) {
                float lp = -INFINITY, lpf = 0.f;
                if (tg >= 0 && tg < vocab) {
                    const float xt = scale_logit<DT, TEMP>(x_tg, a.tparam);
                    const bool kept = xt > thr || (xt == thr && tg >= tie);
                    if (kept) lp = xt - lse_kept;
                    lpf = xt - lse_full;
                }
                a.logprob[r] = lp;
                if (a.logprob_full) a.logprob_full[r] = lpf;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// top-p alone over bf16 rows: nothing is sorted and no exponential is taken per element.  A bf16 row has few distinct
// values, so the number of elements per value says everything: one pass over the row counts them in LDS, one bin per
// value, and the bins (count x exp(value - max), in double, walked from the smallest value) give the log-sum-exp, the
// threshold, how many of the elements that tie with it fall, and the kept log-sum-exp.  A second pass, from cache, runs
// only to find the first survivor among such ties or to record a small kept set.
//
// The 16384 bins hold the magnitudes in [2^-31, 2^33), 64 binades of 128 values for either sign.  Smaller magnitudes
// weigh exp(0) to well below an fp32 rounding and share one count; a row whose threshold is among them, or that holds a
// larger value, is left to the wide kernel.  Larger negative values weigh nothing next to any value of the bins.
// Counts are integers and every sum runs in a fixed order, so a row comes out the same every time.
//
// What bounds it: the LDS atomics of the first pass, about 15 cycles per 64 elements and compute unit where these differ
// (lanes that add to one word take turns: see the common value), where the row itself would arrive in 11, and next to them the
// vector unit; then the latency of the steps between two passes, which two workgroups of 1024 threads per compute unit cover
// for each other (workgroups of 512, of which the bins admit two as well: 195 us).  With a kept-set
// record, top_p 0.95, standard deviations 2 - 6, against candidate lists, a sort and the radix descent of the wide kernel:
// 1499 rows of V = 151 936 145 us (62 to read the rows) and 726; 180 rows of V = 205 350 47 and 470; 4000 rows of 32 000
// with a temperature 158 and 408; 800 rows of 9001 37 and 185.  Rows with a common value, 1499 of V = 151 936, against the same
// two and against counting every element in LDS: 99 % of the ids masked with -1e9 148, 216 and 795; 80 % 245, 713 and 650; one
// value 139, 774 and 961; two values of a half each 440, 603 and 688; ordinary rows take 1 - 2 % longer for the look at a sample.
// ---------------------------------------------------------------------------------------------
constexpr int kNucThreads = 1024, kNucWaves = kNucThreads / kWave;
constexpr int kNucLow = 0x3000;                     // bf16 bits of 2^-31, the smallest magnitude with a bin of its own
constexpr int kNucSide = 0x2000;                    // bins per sign: magnitudes 0x3000 .. 0x4fff
constexpr int kNucBins = 2 * kNucSide;
constexpr int kNucChunks = kNucBins / kWave;        // the bins in ascending order of the value, a wave's lanes at a time
constexpr int kNucList = 4096;                      // entries of the list a small kept set is collected in (over the bins)
constexpr int kNucLoads = 4;                        // 16-byte loads in flight per thread
constexpr int kNucCommon = 16;                      // of 64 elements: a value that is counted in registers

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef short i16x2 __attribute__((ext_vector_type(2)));

struct NucShared {
    union {
        uint32_t bin[kNucBins];
        struct {
            unsigned long long list[kNucList];
            uint16_t hit[kNucThreads];  // threads that saw an element of the kept set
        };
        uint32_t block[kNucThreads];  // elements equal to the threshold, per block of indices
    };
    double chunk_mass[kNucChunks];
    int chunk_n[kNucChunks];
    int key_w[kNucWaves];          // largest value of a wave, as a number that ascends with it
    uint32_t block_w[kNucWaves], step_n[3];
    int n_small, odd;
    int n_list, n_hit, tie;
};

// bin number in ascending order of the value -> its place in LDS; -> the value
__device__ __forceinline__ int nuc_bin(int rank) { return rank < kNucSide ? kNucBins - 1 - rank : rank - kNucSide; }
__device__ __forceinline__ float nuc_value(int rank) {
    const uint32_t bits = rank < kNucSide ? 0x8000u | static_cast<uint32_t>(kNucSide - 1 - rank + kNucLow) : static_cast<uint32_t>(rank - kNucSide + kNucLow);
    return bf16_bits_to_f32(bits);
}

// sum and maximum of an int (>= 0) over a wave, by lane moves
template <typename F> __device__ __forceinline__ int wave_fold_int(int v, F f) {
    v = f(v, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, false));   // quad_perm [1,0,3,2]
    v = f(v, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, false));   // quad_perm [2,3,0,1]
    v = f(v, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, false));  // row_half_mirror
    v = f(v, __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, false));  // row_mirror
    return f(f(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)), f(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}
__device__ __forceinline__ int wave_sum_int(int v) { return wave_fold_int(v, [](int p, int q) { return p + q; }); }
__device__ __forceinline__ int wave_max_int(int v) { return wave_fold_int(v, [](int p, int q) { return p > q ? p : q; }); }

constexpr int kOddNan = 1, kOddLarge = 2, kOddInf = 4;  // a NaN; a finite value above the bins; +inf

template <int TEMP> __global__ __launch_bounds__(kNucThreads, 8) void nucleus_count_kernel(SelArgs a) {
    using R = Row<NRL_BF16>;
    __shared__ NucShared sh;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int64_t r = blockIdx.x;
    const uint32_t o = blockIdx.x / static_cast<uint32_t>(a.n_inner);  // (fewer than 2^31 rows)
    const int64_t i_in = blockIdx.x - o * static_cast<uint32_t>(a.n_inner);
    const char* row = static_cast<const char*>(a.logits) + (o * a.stride_outer + i_in * a.stride_inner) * R::BYTES;
    const int64_t vocab = a.vocab;
    const int64_t head = sel_row_head<NRL_BF16>(row, vocab);
    const int64_t nvec = (vocab - head) / R::EPV;
    const int64_t tail0 = head + nvec * R::EPV;
    const u32x4* xv = reinterpret_cast<const u32x4*>(row + head * R::BYTES);

    // a vector of scaled logits, still as bf16 bits
    auto scaled_bits = [&](const u32x4& q) -> u32x4 {
        if constexpr (TEMP == 0) return q;
        float t[R::EPV];
        R::decode(q, t);
#pragma unroll
        for (int k = 0; k < R::EPV; ++k) t[k] = TEMP == 1 ? __fdiv_rn(t[k], a.tparam) : t[k] * a.tparam;
        return R::encode(t);
    };
    auto load_scaled = [&](int64_t e) { return scale_logit<NRL_BF16, TEMP>(R::load1(row, e), a.tparam); };
    // f(scaled vector, its index) over the kNucStep vectors from `base` on, or over the row
    const int n_vec = static_cast<int>(nvec);
    constexpr int kNucStep = kNucLoads * kNucThreads;
    auto for_step = [&](int base, auto f) {
        if (base >= n_vec) return;
        u32x4 q[kNucLoads];
#pragma unroll
        for (int u = 0; u < kNucLoads; ++u) q[u] = xv[base + u * kNucThreads < n_vec ? base + u * kNucThreads : n_vec - 1];
#pragma unroll
        for (int u = 0; u < kNucLoads; ++u)
            if (base + u * kNucThreads < n_vec) f(scaled_bits(q[u]), base + u * kNucThreads);
    };
    auto for_vectors = [&](auto f) {
        for (int base = tid; base < n_vec; base += kNucStep) for_step(base, f);
    };

    // the target's logit, on its way while the row is counted
    int64_t tg = -1;
    float x_tg = 0.f;
    if (a.targets && a.logprob) {
        tg = a.targets[o * a.ts_outer + i_in * a.ts_inner];
        if (tg >= 0 && tg < vocab) x_tg = R::load1(row, tg);
    }

    // and 64 elements from all over the row: lanes that see one value add to one word of LDS, one after the other, so a value of
    // kNucCommon of these elements (of three elements' values the most frequent one) is counted in registers
    const uint32_t sample = f32_to_bf16_bits(load_scaled((static_cast<uint64_t>(lane) * static_cast<uint64_t>(vocab)) >> 6));

    // ---- count the elements of every value ----
#pragma unroll
    for (int i = tid; i < kNucBins / 4; i += kNucThreads) reinterpret_cast<u32x4*>(sh.bin)[i] = u32x4{0u, 0u, 0u, 0u};
    if (tid == 0) { sh.n_small = 0; sh.odd = 0; sh.n_list = 0; sh.n_hit = 0; }
    __syncthreads();
    uint32_t common = 0u;
    int most = 0;
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        const uint32_t v = __builtin_amdgcn_readlane(sample, 21 * l);
        const int n = __popcll(__ballot(sample == v));
        if (n > most) { most = n; common = v; }
    }
    int n_small = 0, odd = 0;
    // the largest of this thread's bits as signed numbers, which is its largest value if that is not negative, and the
    // smallest as unsigned ones, which is its largest value if all are negative; by halves of the words
    i16x2 largest = {-32768, -32768};
    u16x2 least = {65535, 65535};
    // t: bits - kNucLow.  Its top four bits tell the ranges apart: 0, 1 and 8, 9 the bins of either sign, 2 - 4 larger
    // (also NaN), 5 - 7 and 13 - 15 smaller magnitudes, 10 - 12 larger negative ones (also NaN).
    auto count_many = [&](uint32_t t, int n) {
        if (!(t & 0x6000u)) { atomicAdd(&sh.bin[(t & 0x1fffu) | ((t >> 2) & 0x2000u)], static_cast<uint32_t>(n)); return; }
        const uint32_t bits = (t + kNucLow) & 0xffffu, mag = bits & 0x7fffu;
        if (mag > 0x7f80u) odd |= kOddNan;
        else if (bits == 0x7f80u) odd |= kOddInf;
        else if (mag < static_cast<uint32_t>(kNucLow)) n_small += n;
        else if (!(bits & 0x8000u)) odd |= kOddLarge;
    };
    auto count_one = [&](uint32_t t) { count_many(t, 1); };
    auto count_vector = [&](const u32x4& q) {
        uint32_t t[4], outside = 0u;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const uint32_t pair = q[w];  // (__builtin_bit_cast straight from q[w] reads element 0 whatever w is)
            largest = __builtin_elementwise_max(largest, __builtin_bit_cast(i16x2, pair));
            least = __builtin_elementwise_min(least, __builtin_bit_cast(u16x2, pair));
            t[w] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, pair) - u16x2{kNucLow, kNucLow});
            outside |= t[w] & 0x60006000u;
        }
        if (outside == 0u) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const u16x2 up = __builtin_bit_cast(u16x2, t[w]) >> 2;
                const uint32_t at = (t[w] & 0x1fff1fffu) | (__builtin_bit_cast(uint32_t, up) & 0x20002000u);
                atomicAdd(&sh.bin[at & 0xffffu], 1u);
                atomicAdd(&sh.bin[at >> 16], 1u);
            }
        } else {
#pragma unroll
            for (int w = 0; w < 4; ++w) { count_one(t[w] & 0xffffu); count_one(t[w] >> 16); }
        }
    };
    if (most < kNucCommon) {
        for_vectors([&](const u32x4& q, int) { count_vector(q); });
    } else {
        // (an element at a time, in little code: unrolled like the ordinary loop, this one's code made ordinary rows 2 - 7 % slower)
        int n_common = 0;
        for (int vi = tid; vi < n_vec; vi += kNucThreads) {
            u32x4 q = scaled_bits(xv[vi]);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const uint32_t pair = q[w];
                largest = __builtin_elementwise_max(largest, __builtin_bit_cast(i16x2, pair));
                least = __builtin_elementwise_min(least, __builtin_bit_cast(u16x2, pair));
            }
#pragma unroll 1
            for (int k = 0; k < R::EPV; ++k) {
                const uint32_t bits = q.x & 0xffffu;
                q.x = (q.x >> 16) | (q.y << 16);
                q.y = (q.y >> 16) | (q.z << 16);
                q.z = (q.z >> 16) | (q.w << 16);
                q.w >>= 16;
                if (bits == common) ++n_common;
                else count_one((bits - kNucLow) & 0xffffu);
            }
        }
        n_common = wave_sum_int(n_common);
        if (lane == 0 && n_common) count_many((common - kNucLow) & 0xffffu, n_common);
    }
    auto count_scalar = [&](int64_t e) {
        const uint32_t bits = f32_to_bf16_bits(load_scaled(e));
        count_one((bits - kNucLow) & 0xffffu);
        largest.x = static_cast<short>(bits) > largest.x ? static_cast<short>(bits) : largest.x;
        least.x = static_cast<unsigned short>(bits) < least.x ? static_cast<unsigned short>(bits) : least.x;
    };
    if (tid < head) count_scalar(tid);
    if (tail0 + tid < vocab) count_scalar(tail0 + tid);
    if (n_small) atomicAdd(&sh.n_small, n_small);
    if (odd) atomicOr(&sh.odd, odd);
    {
        const int high = largest.x > largest.y ? largest.x : largest.y;
        const int low = least.x < least.y ? least.x : least.y;
        const int key = wave_max_int(high >= 0 ? 0x8000 | high : 0xffff & ~low);  // ascending with the value
        if (lane == 0) sh.key_w[wave] = key;
    }
    __syncthreads();
    n_small = sh.n_small;
    odd = sh.odd;
    uint32_t max_bits;  // of the row
    {
        int key = sh.key_w[0];
#pragma unroll
        for (int w = 1; w < kNucWaves; ++w) key = sh.key_w[w] > key ? sh.key_w[w] : key;
        max_bits = static_cast<uint32_t>(key & 0x8000 ? key & 0x7fff : 0xffff & ~key);
    }
    const uint32_t max_mag = max_bits & 0x7fffu;
    const bool max_binned = max_mag - kNucLow < static_cast<uint32_t>(kNucSide);
    const float m = max_binned ? bf16_bits_to_f32(max_bits) : 0.f;  // (a maximum under the bins counts as 0)
    // (every wave finds the same values from here on: what they rest on is read from LDS by all)
    int pick = -1, n_eq = 0, above = 0;
    float e_thr = 0.f;
    double z = 0.0, below = 0.0, cut = 0.0;
    if (!odd && (max_binned || n_small > 0)) {
        // ---- mass and elements of every chunk of bins, the waves taking turns: what is not empty lies close together ----
#pragma unroll 4
        for (int c = wave; c < kNucChunks; c += kNucWaves) {
            const int rank = c * kWave + lane, n = static_cast<int>(sh.bin[nuc_bin(rank)]);
            double mass = 0.0;
            int elems = 0;
            if (__ballot(n != 0)) {
                if (n) mass = static_cast<double>(n) * static_cast<double>(expf(nuc_value(rank) - m));
                mass = wave_sum_double(mass);
                elems = wave_sum_int(n);
            }
            if (lane == 0) { sh.chunk_mass[c] = mass; sh.chunk_n[c] = elems; }
        }
        __syncthreads();
        // ---- the chunk, then the bin, in which the running sum from the smallest value passes (1 - p) Z ----
        static_assert(kNucChunks == 4 * kWave, "four chunks per lane, the lower half of the lanes has the negative values");
        double four[4];
        double own = 0.0;
#pragma unroll
        for (int k = 0; k < 4; ++k) { four[k] = sh.chunk_mass[4 * lane + k]; own += four[k]; }
        const double upto = wave_scan_double(own);
        const double small = n_small > 0 ? static_cast<double>(n_small) * static_cast<double>(expf(-m)) : 0.0;  // between the two signs
        z = lane_double(upto, kWave - 1) + small;
        cut = static_cast<double>(1.0f - a.top_p) * z;
        double from = upto - own + (lane >= kWave / 2 ? small : 0.0);
        const double next = __shfl_down(from, 1, kWave);
        const double to = lane == kWave / 2 - 1 ? next - small : lane == kWave - 1 ? z : next;  // the next lane starts where this one ends
        const unsigned long long who = __ballot(own > 0.0 && from <= cut && cut < to);
        int chunk = -1;
        if (who) {
            int k_at = -1;
            double k_from = 0.0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                // (the last one with mass stays where rounding leaves the sum just short of the cut)
                if (four[k] > 0.0 && (k_at < 0 || from <= cut)) { k_at = k; k_from = from; }
                from += four[k];
            }
            const int src = __builtin_ctzll(who);
            chunk = 4 * src + __builtin_amdgcn_readlane(k_at, src);
            below = lane_double(k_from, src);
        } else if (!(cut < z) && max_binned) {
            chunk = ((max_bits & 0x8000u) ? kNucSide - 1 - static_cast<int>(max_mag - kNucLow) : kNucSide + static_cast<int>(max_mag - kNucLow)) / kWave;
        }
        if (chunk >= 0) {
            const int rank = chunk * kWave + lane, n = static_cast<int>(sh.bin[nuc_bin(rank)]);
            const float e = n ? expf(nuc_value(rank) - m) : 0.f;
            const double mass = static_cast<double>(n) * static_cast<double>(e), sum = wave_scan_double(mass);
            unsigned long long with = __ballot(mass > 0.0);
            const unsigned long long past = who ? __ballot(mass > 0.0 && below + sum > cut) : 0ull;
            // (none past the cut: rounding again, or nothing at all may fall short of it: the largest value stays)
            const int at = past ? __builtin_ctzll(past) : with ? 63 - __builtin_clzll(with) : -1;
            if (at >= 0) {
                pick = chunk * kWave + at;
                n_eq = __builtin_amdgcn_readlane(n, at);
                e_thr = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(e), at));
                const double eq_mass = static_cast<double>(n_eq) * static_cast<double>(e_thr);
                below = who ? below + (lane_double(sum, at) - eq_mass) : z - eq_mass;
                if (a.kept_n) {
                    above = lane > at ? n : 0;
#pragma unroll
                    for (int k = 0; k < 4; ++k) above += 4 * lane + k > chunk ? sh.chunk_n[4 * lane + k] : 0;
                    above = wave_sum_int(above) + (pick < kNucSide ? n_small : 0);
                }
            }
        }
    }
    if (pick < 0) {
        // NaN and +inf make every result NaN, and so does a row of -inf; the gradient is NaN for +inf alone, 0 for the other two.
        // The wide kernel finishes the other rows, and finds the row's largest (scaled) logit in thr
        const float row_max = bf16_bits_to_f32(max_bits);
        const bool wide = !(odd & (kOddNan | kOddInf)) && row_max > -INFINITY;
        if (tid == 0) {
            const float nan = __builtin_nanf("");
            a.thr[r] = wide ? row_max : nan;
            a.tie[r] = wide ? kTieUnresolved : (odd & kOddNan) || !odd ? 0 : kTieNoCut;
            a.lse_kept[r] = nan;
            if (a.logprob) a.logprob[r] = nan;
            if (a.lse_full) a.lse_full[r] = (odd & (kOddNan | kOddInf)) ? nan : -INFINITY;
            if (a.logprob_full) a.logprob_full[r] = nan;
            if (a.kept_n) a.kept_n[r] = -1;
        }
        return;
    }
    const float thr = nuc_value(pick);
    const double at_or_above = z - below;
    double drop_d = floor((cut - below) / static_cast<double>(e_thr));
    drop_d = drop_d < 0.0 ? 0.0 : drop_d > n_eq - 1 ? n_eq - 1 : drop_d;
    const int drop = static_cast<int>(drop_d);  // elements equal to the threshold that fall: those with the smallest indices
    const float lse_kept = m + logf(static_cast<float>(at_or_above - drop_d * static_cast<double>(e_thr)));
    const float lse_full = m + logf(static_cast<float>(z));
    int tie = 0, n_keep = -1;
    if (a.kept_n && above + n_eq <= kNucList && above + n_eq - drop <= a.kept_cap) n_keep = above + n_eq - drop;
    if (n_keep >= 0) {
        // the kept set and the ties that fall, in descending order of (value, index)
        __syncthreads();
        auto push = [&](float x, int64_t index) {
            if (x < thr) return;
            const int pos = atomicAdd(&sh.n_list, 1);
            if (pos < kNucList) sh.list[pos] = (static_cast<unsigned long long>(order_key(x)) << 32) | static_cast<uint32_t>(index);
        };
        auto push_vector = [&](const u32x4& q, int vi) {
            float t[R::EPV];
            R::decode(q, t);
            float vm = t[0];
#pragma unroll
            for (int k = 1; k < R::EPV; ++k) vm = fmaxf(vm, t[k]);
            if (vm >= thr) {
#pragma unroll
                for (int k = 0; k < R::EPV; ++k) push(t[k], head + static_cast<int64_t>(vi) * R::EPV + k);
            }
        };
        if (thr > 0.f) {
            // only what the threads read that saw such an element is read again, dealt out over all of them
            const int bits = static_cast<int>(f32_to_bf16_bits(thr));
            if (largest.x >= bits || largest.y >= bits) sh.hit[atomicAdd(&sh.n_hit, 1)] = static_cast<uint16_t>(tid);
            __syncthreads();
            const int per = (n_vec + kNucThreads - 1) / kNucThreads, n_items = sh.n_hit * per;
            for (int item = tid; item < n_items; item += 2 * kNucThreads) {
                int vi[2];
                u32x4 q[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int it = item + u * kNucThreads, h = it / per;
                    vi[u] = it < n_items ? sh.hit[h] + (it - h * per) * kNucThreads : n_vec;
                    if (vi[u] < n_vec) q[u] = xv[vi[u]];
                }
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    if (vi[u] < n_vec) push_vector(scaled_bits(q[u]), vi[u]);
            }
        } else {
            for_vectors(push_vector);
        }
        if (tid < head) push(load_scaled(tid), tid);
        if (tail0 + tid < vocab) push(load_scaled(tail0 + tid), tail0 + tid);
        __syncthreads();
        const int n = sh.n_list < kNucList ? sh.n_list : kNucList;
        auto record = [&](unsigned long long c, int at) {
            if (at < n_keep) {
                a.kept_idx[r * a.kept_cap + at] = static_cast<int32_t>(c & 0xffffffffu);
                a.kept_x[r * a.kept_cap + at] = key_value(static_cast<uint32_t>(c >> 32));
            }
            if (at == n_keep - 1) sh.tie = static_cast<int>(c & 0xffffffffu);
        };
        if (n <= kNucThreads) {
            // an element's place is the number of larger ones (no two are equal): n LDS reads in a row, all lanes the same
            // word, where a sort takes a barrier or an LDS round trip for each of its steps
            if (tid < n) {
                const unsigned long long c = sh.list[tid];
                int at = 0;
#pragma unroll 8
                for (int i = 0; i < n; ++i) at += sh.list[i] > c ? 1 : 0;
                record(c, at);
            }
        } else {
            int n_pad = 1;
            while (n_pad < n) n_pad <<= 1;
            for (int i = n + tid; i < n_pad; i += kNucThreads) sh.list[i] = 0ull;
            sort_list_desc<kNucThreads>(sh.list, n_pad);
            for (int q = tid; q < n; q += kNucThreads) record(sh.list[q], q);
        }
        __syncthreads();
        if (drop > 0) tie = sh.tie;
    } else if (drop > 0) {
        // the element with `drop` equal ones before it: equal elements are counted per block of indices, from the front of
        // the row until there are more than that (half of the row on average), then one look at the block that holds it
        const uint32_t want = static_cast<uint32_t>(drop);
        __syncthreads();
        sh.block[tid] = 0u;
        if (tid < 3) sh.step_n[tid] = 0;
        __syncthreads();
        int shift = 0;
        while ((static_cast<int64_t>(kNucThreads) << shift) < vocab) ++shift;
        const uint32_t bits = f32_to_bf16_bits(thr), both = bits | (bits << 16);
        uint32_t seen_n = 0u;
        const bool many = n_eq >= vocab / 8;  // several to a vector, which are added together
        // (steps take turns at three counters: the one cleared in a step was last read two barriers ago)
        for (int base = 0, step = 0; base == 0 || base < n_vec; base += kNucStep, step = step == 2 ? 0 : step + 1) {
            int mine = 0;
            auto count = [&](int64_t index) {
                atomicAdd(&sh.block[index >> shift], 1u);
                ++mine;
            };
            if (base == 0 && tid < head && load_scaled(tid) == thr) count(tid);
            for_step(base + tid, [&](const u32x4& q, int vi) {
                uint32_t differ = 0u;  // elements that are not equal, by halves
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint32_t pair = q[w] ^ both;
                    const u16x2 one = __builtin_elementwise_min(__builtin_bit_cast(u16x2, pair), u16x2{1, 1});
                    differ += __builtin_bit_cast(uint32_t, one);
                }
                if (differ != 0x00040004u) {
                    if (many) {
                        const int64_t index0 = head + static_cast<int64_t>(vi) * R::EPV;
                        if (index0 >> shift == (index0 + R::EPV - 1) >> shift) {
                            const uint32_t equal = R::EPV - (differ & 0xffffu) - (differ >> 16);
                            atomicAdd(&sh.block[index0 >> shift], equal);
                            mine += static_cast<int>(equal);
                            return;
                        }
                    }
#pragma unroll
                    for (int k = 0; k < R::EPV; ++k)
                        if (((q[k >> 1] >> (16 * (k & 1))) & 0xffffu) == bits) count(head + static_cast<int64_t>(vi) * R::EPV + k);
                }
            });
            if (mine) atomicAdd(&sh.step_n[step], static_cast<uint32_t>(mine));
            if (tid == 0) sh.step_n[step == 2 ? 0 : step + 1] = 0;
            __syncthreads();
            seen_n += sh.step_n[step];
            if (seen_n > want) break;
        }
        if (seen_n <= want && tail0 + tid < vocab && load_scaled(tail0 + tid) == thr) atomicAdd(&sh.block[(tail0 + tid) >> shift], 1u);
        __syncthreads();
        const uint32_t here = sh.block[tid];
        uint32_t upto = here;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const uint32_t low = __shfl_up(upto, off, kWave);
            if (lane >= off) upto += low;
        }
        if (lane == kWave - 1) sh.block_w[wave] = upto;
        __syncthreads();
        uint32_t before = upto - here;
        for (int w = 0; w < wave; ++w) before += sh.block_w[w];
        const bool holder = before <= want && want < before + here;
        const unsigned long long who = __ballot(holder);
        if (who) {  // one wave: it walks the block
            const int src = __builtin_ctzll(who);
            uint32_t seen = __builtin_amdgcn_readlane(before, src);
            const int64_t first = static_cast<int64_t>(wave * kWave + src) << shift;
            int64_t stop = first + (int64_t{1} << shift);
            stop = stop < vocab ? stop : vocab;
            for (int64_t j0 = first; j0 < stop && seen <= want; j0 += 4 * kWave) {
                bool eq[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int64_t j = j0 + u * kWave + lane;
                    eq[u] = load_scaled(j < stop ? j : stop - 1) == thr && j < stop;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const unsigned long long bal = __ballot(eq[u]);
                    if (eq[u] && seen + __popcll(bal & ((1ull << lane) - 1ull)) == want) sh.tie = static_cast<int>(j0 + u * kWave + lane);
                    seen += __popcll(bal);
                }
            }
        }
        __syncthreads();
        tie = sh.tie;
    }
    if (tid == 0) {
        if (a.kept_n) a.kept_n[r] = n_keep;
        a.thr[r] = thr;
        a.tie[r] = tie;
        a.lse_kept[r] = lse_kept;
        if (a.lse_full) a.lse_full[r] = lse_full;
        if (a.targets && a.logprob) {
            float lp = -INFINITY, lpf = 0.f;
            if (tg >= 0 && tg < vocab) {
                const float xt = scale_logit<NRL_BF16, TEMP>(x_tg, a.tparam);
                if (xt > thr || (xt == thr && tg >= tie)) lp = xt - lse_kept;
                lpf = xt - lse_full;
            }
            a.logprob[r] = lp;
            if (a.logprob_full) a.logprob_full[r] = lpf;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// rows whose kept set does not fit the on-chip candidate list (top-p alone over a flat distribution, thousands
// of exact ties, or a very large top_k): the same keep predicate found without a sort, by a radix descent over
// the order keys.  A pass streams the row once and fills a histogram over one digit of the keys that share the
// digits chosen so far: the number of elements per bin, which is what top-k descends by (the largest key with at
// least top_k keys at or above it), and their probability mass per bin, which is what top-p descends by (the
// smallest key whose cumulative mass from below exceeds (1 - p) Z).  A 16-bit logit has 16 significant key bits:
// two digits, so top-k and top-p together take three passes (the first histogram serves both), top-p alone two;
// fp16 adds a three-bit digit, fp32 has four digits.  One more pass over the row and a look at one block of it
// find the first survivor among the elements that tie with the top-p threshold.  The row (at most a few hundred
// KB) comes from cache after the first pass.
//
// Masses are summed as 64-bit fixed-point integers (exp(x - max) * 2^S with S chosen from the row length so that a
// whole row cannot overflow): integer addition is associative, so the LDS atomics that fill the histogram give
// the same sums whatever order they arrive in, and the row's result does not depend on scheduling.  The fixed
// point resolves 2^-45 of the largest element's mass at V = 151936; what it drops is below the rounding of the
// reference's fp32 sums by orders of magnitude, and which of two nearly equal neighbours at the top-p boundary
// falls first may differ from a sorted fp32 running sum, as it may between any two summation orders.
// ---------------------------------------------------------------------------------------------
constexpr int kRadixBins = 256;
constexpr int kRadixCopies = 8;   // histogram copies by lane: logits of one magnitude share their leading digit
constexpr int kTieBlocks = kRadixBins * kRadixCopies;  // index blocks of the tie search (they reuse the count bins)

// digits of an order key from the top, by element type: 16-bit types leave the low key bits constant for a given sign
template <int DT> struct KeyDigits;
template <> struct KeyDigits<NRL_F32> {
    static constexpr int N = 4, LOW = 0;
    __device__ static constexpr int shift(int l) { return 24 - 8 * l; }
    __device__ static constexpr int bits(int) { return 8; }
};
template <> struct KeyDigits<NRL_BF16> {
    static constexpr int N = 2, LOW = 16;
    __device__ static constexpr int shift(int l) { return 24 - 8 * l; }
    __device__ static constexpr int bits(int) { return 8; }
};
template <> struct KeyDigits<NRL_F16> {
    static constexpr int N = 3, LOW = 13;
    __device__ static constexpr int shift(int l) { return l == 2 ? 13 : 24 - 8 * l; }
    __device__ static constexpr int bits(int l) { return l == 2 ? 3 : 8; }
};

struct WideShared {
    unsigned long long mass[kRadixBins * kRadixCopies];
    unsigned int cnt[kRadixBins * kRadixCopies];
    unsigned long long scan64[kSelWaves];
    unsigned int scan32[kSelWaves];
    // what the thread that owns the chosen bin tells the others
    unsigned int pick_bin, pick_cnt;
    unsigned long long pick_a, pick_b;
};

template <typename T> __device__ __forceinline__ T wide_scan_excl(T v, T* shm, T& total) {
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    T inc = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const T t = __shfl_up(inc, off, kWave);
        if (lane >= off) inc += t;
    }
    __syncthreads();  // the previous scan's readers are done with shm
    if (lane == kWave - 1) shm[wave] = inc;
    __syncthreads();
    T base = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kSelWaves; ++w) {
        const T part = shm[w];
        if (w < wave) base += part;
        tot += part;
    }
    total = tot;
    return base + inc - v;
}

// exp(x - m) as a fixed-point integer with fx_shift fraction bits (x <= m, 23 <= fx_shift <= 46); zero below its
// resolution.  Without branches: the 24-bit significand is placed where the value 1.0 belongs and moved down by
// the exponent's distance from 1.0's.
__device__ __forceinline__ unsigned long long wide_mass(float x, float m, int fx_shift) {
    const uint32_t b = __float_as_uint(fast_exp2((x - m) * kLog2e)) & 0x7fffffffu;
    const int ex = static_cast<int>(b >> 23);
    const unsigned long long top = static_cast<unsigned long long>((b & 0x7fffffu) | 0x800000u) << (fx_shift - 23);
    int down = 127 - ex;              // 0 for 1.0; 127 for zero and subnormals (flushed); negative never for x <= m
    down = down < 0 ? 0 : down > 63 ? 63 : down;
    return ex == 255 ? 0ull : top >> down;   // (a NaN logit weighs nothing)
}

template <int DT, int TEMP> struct WideRow {
    const char* row;
    const u32x4* xv;
    int64_t vocab, head, nvec, tail0;
    float tparam;
    // f(scaled logit, vocabulary index) for every element of the row, each exactly once
    template <typename F> __device__ __forceinline__ void for_each(F f) const {
        constexpr int EPV = Row<DT>::EPV;
        constexpr int kLoads = 8;  // vector loads in flight per thread: a pass is bound by their latency otherwise
        const int tid = threadIdx.x;
        int64_t vi = tid;
        for (; vi + (kLoads - 1) * kSelBlock < nvec; vi += kLoads * kSelBlock) {
            u32x4 q[kLoads];
#pragma unroll
            for (int u = 0; u < kLoads; ++u) q[u] = xv[vi + u * kSelBlock];
#pragma unroll
            for (int u = 0; u < kLoads; ++u) {
                float t[EPV];
                Row<DT>::decode(q[u], t);
#pragma unroll
                for (int k = 0; k < EPV; ++k) f(scale_logit<DT, TEMP>(t[k], tparam), head + (vi + u * kSelBlock) * EPV + k);
            }
        }
        for (; vi < nvec; vi += kSelBlock) {
            float t[EPV];
            Row<DT>::decode(xv[vi], t);
#pragma unroll
            for (int k = 0; k < EPV; ++k) f(scale_logit<DT, TEMP>(t[k], tparam), head + vi * EPV + k);
        }
        if (tid < head) f(scale_logit<DT, TEMP>(Row<DT>::load1(row, tid), tparam), static_cast<int64_t>(tid));
        if (tail0 + tid < vocab) f(scale_logit<DT, TEMP>(Row<DT>::load1(row, tail0 + tid), tparam), tail0 + tid);
    }
};

// One histogram pass: bin = digit `level` of the keys whose higher digits equal `prefix` (every key at level 0).
// Thread b returns the mass of such elements in bin b and, with CNT, their number (0 otherwise: the top-p descent
// needs counts at its last digit only, and every atomic less shortens the pass).
template <int DT, int TEMP, bool CNT>
__device__ __forceinline__ void wide_hist_pass(const WideRow<DT, TEMP>& w, WideShared& sh, float m, int fx_shift, int level,
                                               uint32_t prefix, unsigned int& my_cnt, unsigned long long& my_mass) {
    const int tid = threadIdx.x;
    const int shift = KeyDigits<DT>::shift(level), bits = KeyDigits<DT>::bits(level);
    const uint32_t mask = (1u << bits) - 1u;
    __syncthreads();  // whoever still reads the bins of the pass before
    for (int i = tid; i < kRadixBins * kRadixCopies; i += kSelBlock) { sh.mass[i] = 0ull; sh.cnt[i] = 0u; }
    __syncthreads();
    const int copy = tid & (kRadixCopies - 1);
    if (level == 0) {
        w.for_each([&](float x, int64_t) {
            const int slot = static_cast<int>((order_key(x) >> shift) & mask) * kRadixCopies + copy;
            if (CNT) atomicAdd(&sh.cnt[slot], 1u);
            atomicAdd(&sh.mass[slot], wide_mass(x, m, fx_shift));
        });
    } else {
        w.for_each([&](float x, int64_t) {
            const uint32_t key = order_key(x);
            if ((key >> (shift + bits)) == prefix) {
                const int slot = static_cast<int>((key >> shift) & mask) * kRadixCopies + copy;
                if (CNT) atomicAdd(&sh.cnt[slot], 1u);
                atomicAdd(&sh.mass[slot], wide_mass(x, m, fx_shift));
            }
        });
    }
    __syncthreads();
    my_cnt = 0u;
    my_mass = 0ull;
#pragma unroll
    for (int q = 0; q < kRadixCopies; ++q) {
        my_cnt += sh.cnt[tid * kRadixCopies + q];
        my_mass += sh.mass[tid * kRadixCopies + q];
    }
}

template <int DT, int TEMP>
__global__ __launch_bounds__(kSelBlock) void topk_topp_wide_kernel(SelArgs a, int64_t n_rows) {
    static_assert(kRadixBins == kSelBlock, "one histogram bin per thread");
    __shared__ WideShared sh;
    using KD = KeyDigits<DT>;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const bool use_p = a.top_p < 1.0f;
    {
        // the usual case is that no row of this workgroup is marked: look at all of them at once and leave
        bool mine = false;
        for (int64_t r = blockIdx.x + static_cast<int64_t>(tid) * gridDim.x; r < n_rows; r += static_cast<int64_t>(kSelBlock) * gridDim.x)
            mine |= a.tie[r] == kTieUnresolved;
        if (!__syncthreads_or(mine)) return;
    }
    int clog2 = 0;
    while ((int64_t{1} << clog2) < a.vocab) ++clog2;
    const int fx_shift = 63 - clog2 < 46 ? 63 - clog2 : 46;  // a row of `vocab` largest elements still fits 63 bits
    for (int64_t r = blockIdx.x; r < n_rows; r += gridDim.x) {
        if (a.tie[r] != kTieUnresolved) continue;  // the same word for every thread of the workgroup
        const int64_t o = r / a.n_inner, i_in = r - o * a.n_inner;
        WideRow<DT, TEMP> w;
        w.row = static_cast<const char*>(a.logits) + (o * a.stride_outer + i_in * a.stride_inner) * Row<DT>::BYTES;
        w.vocab = a.vocab;
        w.head = sel_row_head<DT>(w.row, w.vocab);
        w.nvec = (w.vocab - w.head) / Row<DT>::EPV;
        w.tail0 = w.head + w.nvec * Row<DT>::EPV;
        w.xv = reinterpret_cast<const u32x4*>(w.row + w.head * Row<DT>::BYTES);
        w.tparam = a.tparam;
        const float m = a.thr[r];  // the row's largest (scaled) logit, left here by the kernel that marked the row
        const bool use_k = a.top_k > 0 && a.top_k < w.vocab;

        // ---- first digit, every element: serves the top-k and the top-p descent alike ----
        unsigned int hc[KD::N];         // this thread's bin along the top-k descent (or just level 0), per level
        unsigned long long hm[KD::N];
        uint32_t hprefix[KD::N];
        int h_levels = 1;
        hprefix[0] = 0u;
        if (use_k) wide_hist_pass<DT, TEMP, true>(w, sh, m, fx_shift, 0, 0u, hc[0], hm[0]);
        else wide_hist_pass<DT, TEMP, KD::N == 1>(w, sh, m, fx_shift, 0, 0u, hc[0], hm[0]);
        unsigned long long total_mass = 0ull;
        wide_scan_excl(hm[0], sh.scan64, total_mass);

        // ---- top-k: the largest key with at least top_k keys at or above it (ties at that key are all kept) ----
        uint32_t k_key = 0u;
        unsigned long long mass_below_k = 0ull;
        unsigned int cnt_at_k = 0u;
        if (use_k) {
            unsigned int need = static_cast<unsigned int>(a.top_k);
            uint32_t prefix = 0u;
#pragma unroll
            for (int l = 0; l < KD::N; ++l) {
                if (l > 0) {
                    hprefix[l] = prefix;
                    wide_hist_pass<DT, TEMP, true>(w, sh, m, fx_shift, l, prefix, hc[l], hm[l]);
                    h_levels = l + 1;
                }
                unsigned int tot_c = 0u;
                unsigned long long tot_m = 0ull;
                const unsigned int excl_c = wide_scan_excl(hc[l], sh.scan32, tot_c);
                const unsigned long long excl_m = wide_scan_excl(hm[l], sh.scan64, tot_m);
                const unsigned int at_or_above = tot_c - excl_c, above = at_or_above - hc[l];
                if (at_or_above >= need && above < need) {
                    sh.pick_bin = static_cast<unsigned int>(tid);
                    sh.pick_cnt = hc[l];
                    sh.pick_a = need - above;
                    sh.pick_b = excl_m;
                }
                __syncthreads();
                prefix = (prefix << KD::bits(l)) | sh.pick_bin;
                need = static_cast<unsigned int>(sh.pick_a);
                mass_below_k += sh.pick_b;
                cnt_at_k = sh.pick_cnt;
                __syncthreads();  // everyone has read the pick
            }
            k_key = prefix << KD::LOW;
            if (KD::LOW > 0 && !(k_key >> 31)) k_key |= (1u << KD::LOW) - 1u;  // a negative value's low key bits are ones
        }
        const unsigned long long z = total_mass - mass_below_k;  // mass of the top-k survivors

        uint32_t thr_key = k_key;
        int32_t tie = 0;
        unsigned long long kept_mass = z;
        if (use_p) {
            // ascending cumulative probability over the survivors; elements fall while it stays <= (1 - p) Z.  Counted
            // over the whole row that is: mass below the key <= (1 - p) Z + mass below the top-k threshold.
            const double target_d = static_cast<double>(1.0f - a.top_p) * static_cast<double>(z);
            const unsigned long long target = target_d <= 0.0 ? 0ull : static_cast<unsigned long long>(target_d);
            unsigned long long room = target + mass_below_k;  // what may still lie below the digit being chosen
            unsigned long long below_all = 0ull;
            unsigned int n_eq = 0u;
            uint32_t prefix = 0u;
#pragma unroll
            for (int l = 0; l < KD::N; ++l) {
                unsigned int bc = hc[l];
                unsigned long long bm = hm[l];
                if (l >= h_levels || hprefix[l] != prefix) {
                    if (l == KD::N - 1) wide_hist_pass<DT, TEMP, true>(w, sh, m, fx_shift, l, prefix, bc, bm);
                    else wide_hist_pass<DT, TEMP, false>(w, sh, m, fx_shift, l, prefix, bc, bm);
                }
                unsigned long long tot_m = 0ull;
                const unsigned long long excl_m = wide_scan_excl(bm, sh.scan64, tot_m);
                // the bin in which the cumulative mass first exceeds the room; if it never does (top_p -> 0), the
                // highest bin with any mass, which holds the largest element: that one always survives
                const bool crossing = tot_m > room ? (excl_m + bm > room && excl_m <= room)
                                                   : (bm > 0ull && tot_m - excl_m - bm == 0ull);
                if (crossing) {
                    sh.pick_bin = static_cast<unsigned int>(tid);
                    sh.pick_cnt = bc;
                    sh.pick_a = room - excl_m;
                    sh.pick_b = excl_m;
                }
                __syncthreads();
                prefix = (prefix << KD::bits(l)) | sh.pick_bin;
                room = sh.pick_a;
                below_all += sh.pick_b;
                n_eq = sh.pick_cnt;
                __syncthreads();
            }
            uint32_t c = prefix << KD::LOW;
            if (KD::LOW > 0 && !(c >> 31)) c |= (1u << KD::LOW) - 1u;
            unsigned long long below = 0ull;  // mass of the survivors strictly below the threshold
            if (c <= k_key) { c = k_key; if (use_k) n_eq = cnt_at_k; }
            else below = below_all - mass_below_k;
            thr_key = c;
            // how many of the elements equal to the threshold fall too (the ones with the smallest indices)
            const unsigned long long e_thr = wide_mass(key_value(c), m, fx_shift);
            unsigned long long drop = 0ull;
            if (e_thr > 0ull && n_eq > 1u && target >= below) {
                drop = (target - below) / e_thr;
                if (drop > n_eq - 1u) drop = n_eq - 1u;
            }
            if (drop > 0ull) {
                // index of the first survivor among the equal elements, the one with `drop` equal elements before it:
                // equal elements counted per block of indices, then one look at the block that holds it
                int ishift = clog2 - 11;
                if (ishift < 0) ishift = 0;
                __syncthreads();
                for (int i = tid; i < kTieBlocks; i += kSelBlock) sh.cnt[i] = 0u;
                __syncthreads();
                w.for_each([&](float x, int64_t j) {
                    if (order_key(x) == c) atomicAdd(&sh.cnt[j >> ishift], 1u);
                });
                __syncthreads();
                unsigned int mine8[kRadixCopies], sum8 = 0u;
#pragma unroll
                for (int q = 0; q < kRadixCopies; ++q) { mine8[q] = sh.cnt[tid * kRadixCopies + q]; sum8 += mine8[q]; }
                unsigned int tot_eq = 0u;
                unsigned int before = wide_scan_excl(sum8, sh.scan32, tot_eq);
                if (before <= drop && drop < before + sum8) {
#pragma unroll
                    for (int q = 0; q < kRadixCopies; ++q) {
                        if (before <= drop && drop < before + mine8[q]) {
                            sh.pick_bin = static_cast<unsigned int>(tid * kRadixCopies + q);
                            sh.pick_cnt = static_cast<unsigned int>(drop) - before;
                        }
                        before += mine8[q];
                    }
                }
                __syncthreads();
                const int64_t first = static_cast<int64_t>(sh.pick_bin) << ishift;
                int64_t stop = first + (int64_t{1} << ishift);
                if (stop > w.vocab) stop = w.vocab;
                unsigned int seen = 0u;
                const unsigned int want = sh.pick_cnt;
                for (int64_t j0 = first; j0 < stop; j0 += kSelBlock) {
                    const int64_t j = j0 + tid;
                    const bool eq = j < stop && order_key(scale_logit<DT, TEMP>(Row<DT>::load1(w.row, j), a.tparam)) == c;
                    const unsigned long long bal = __ballot(eq);
                    const unsigned int in_wave = static_cast<unsigned int>(__popcll(bal & ((1ull << lane) - 1ull)));
                    __syncthreads();
                    if (lane == 0) sh.scan32[wave] = static_cast<unsigned int>(__popcll(bal));
                    __syncthreads();
                    unsigned int ahead = seen, chunk = 0u;
#pragma unroll
                    for (int q = 0; q < kSelWaves; ++q) {
                        if (q < wave) ahead += sh.scan32[q];
                        chunk += sh.scan32[q];
                    }
                    if (eq && ahead + in_wave == want) sh.pick_a = static_cast<unsigned long long>(j);
                    seen += chunk;
                }
                __syncthreads();
                tie = static_cast<int32_t>(sh.pick_a);
            }
            kept_mass = z - below - drop * e_thr;
            if (kept_mass == 0ull || kept_mass > z) kept_mass = e_thr;
        }
        const float thr = key_value(thr_key);
        const float unit = __uint_as_float(static_cast<uint32_t>(127 - fx_shift) << 23);  // 2^-fx_shift
        const float lse_kept = m + logf(static_cast<float>(static_cast<double>(kept_mass) * static_cast<double>(unit)));
        const float lse_full = m + logf(static_cast<float>(static_cast<double>(total_mass) * static_cast<double>(unit)));
        __syncthreads();      // every thread has read thr[r] (the row maximum) and tie[r] == unresolved before they are replaced
        if (tid == 0) {
            a.thr[r] = thr;
            a.lse_kept[r] = lse_kept;
            if (a.lse_full) a.lse_full[r] = lse_full;
            if (a.targets && a.logprob) {
                const int64_t tg = a.targets[o * a.ts_outer + i_in * a.ts_inner];
                float lp = -INFINITY, lpf = 0.f;
                if (tg >= 0 && tg < w.vocab) {
                    const float xt = scale_logit<DT, TEMP>(Row<DT>::load1(w.row, tg), a.tparam);
                    const bool kept = xt > thr || (xt == thr && tg >= tie);
                    if (kept) lp = xt - lse_kept;
                    lpf = xt - lse_full;
                }
                a.logprob[r] = lp;
                if (a.logprob_full) a.logprob_full[r] = lpf;
            }
            a.tie[r] = tie;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// backward / materialisation: one streaming pass with the saved keep predicate
// ---------------------------------------------------------------------------------------------
struct SelBwdArgs {
    const void* logits;
    int64_t n_inner, vocab, stride_outer, stride_inner;
    const int64_t* targets;
    int64_t ts_outer, ts_inner;
    float tparam;
    const float* thr;
    const int32_t* tie;
    const float* lse_kept;
    const float* grad;
    int64_t gs_outer, gs_inner;
    void* out;  // dlogits, or filtered logits
    int64_t d_n_inner, ds_outer, ds_inner;
    uint8_t* keep_out;  // [rows, vocab] or NULL (filter mode)
    const int32_t* kept_n;    // the forward's record of the kept sets (see SelArgs), or NULL
    const int32_t* kept_idx;
    const float* kept_x;
    int kept_cap;
    int prefilled;  // the record is in use: rows on record and rows without a gradient were zero-filled before this launch (fill_zero_rows_kernel), rows on record only add their entries
    int parts;      // workgroups per row
};

// The number of kept entries on record for gradient row (o, i), or -1: the row is streamed from the logits.  `g` becomes its
// upstream gradient, 0 for rows that have none (those are zero whatever the record says).
__device__ __forceinline__ int topk_topp_on_record(const SelBwdArgs& a, int64_t o, int64_t i, float& g) {
    const bool real = i < a.n_inner;
    const int n = real ? a.kept_n[o * a.n_inner + i] : 0;  // (on its way together with the gradient)
    g = real ? a.grad[o * a.gs_outer + i * a.gs_inner] : 0.f;
    return g == 0.f ? 0 : n > a.kept_cap ? -1 : n;  // (above the capacity: not a count the forward writes)
}

// MODE 0: gradient, MODE 1: filtered logits (-inf outside the kept set) + keep mask
template <int DT, int TEMP, int MODE>
__device__ __forceinline__ void topk_topp_stream_row(const SelBwdArgs& a, int64_t r, int part) {
    constexpr int EPV = Row<DT>::EPV;
    const int tid = threadIdx.x;
    const int64_t o = r / a.d_n_inner, i_in = r - o * a.d_n_inner;
    char* out = static_cast<char*>(a.out) + (o * a.ds_outer + i_in * a.ds_inner) * Row<DT>::BYTES;
    const int64_t vocab = a.vocab;
    float g = 0.f;
    // With the forward's record of the kept set the gradient row is zeros plus the few kept entries, written
    // without reading the logits again.
    int n_rec = -1;
    if (MODE == 0 && a.prefilled) n_rec = topk_topp_on_record(a, o, i_in, g);
    else if (MODE == 0 && i_in < a.n_inner) g = a.grad[o * a.gs_outer + i_in * a.gs_inner];
    if (MODE == 0 && a.prefilled && n_rec >= 0) {
        if (part > 0) return;
        // the zeros are there already (an earlier launch on the stream): only the kept entries are written
        const int64_t rec = (o * a.n_inner + i_in) * a.kept_cap;
        if (n_rec > 0) {
            const float lse_r = a.lse_kept[o * a.n_inner + i_in];
            const int64_t tg_r = a.targets[o * a.ts_outer + i_in * a.ts_inner];
            for (int q = tid; q < n_rec; q += kSelBlock) {
                const int64_t idx = a.kept_idx[rec + q];
                if (static_cast<uint64_t>(idx) >= static_cast<uint64_t>(vocab)) continue;
                float d = ((idx == tg_r ? 1.f : 0.f) - fast_exp2((a.kept_x[rec + q] - lse_r) * kLog2e)) * g;
                if constexpr (TEMP == 1) d = __fdiv_rn(Row<DT>::round_self(d), a.tparam);
                if constexpr (TEMP == 2) d = Row<DT>::round_self(d) * a.tparam;
                Row<DT>::store1(out, idx, d);
            }
        }
        return;
    }
    if (MODE == 0 && g == 0.f) {  // dropped position or masked token: the gradient row is exactly zero
        const int64_t zh = sel_row_head<DT>(out, vocab);
        const int64_t zn = (vocab - zh) / EPV;
        u32x4* zv = reinterpret_cast<u32x4*>(out + zh * Row<DT>::BYTES);
        const u32x4 z = {0u, 0u, 0u, 0u};
        for (int64_t v = zn * part / a.parts + tid; v < zn * (part + 1) / a.parts; v += kSelBlock) zv[v] = z;
        if (part == 0 && tid < zh) Row<DT>::store1(out, tid, 0.f);
        if (part == 0 && zh + zn * EPV + tid < vocab) Row<DT>::store1(out, zh + zn * EPV + tid, 0.f);
        return;
    }
    const int64_t rr = o * a.n_inner + i_in;
    const char* row = static_cast<const char*>(a.logits) + (o * a.stride_outer + i_in * a.stride_inner) * Row<DT>::BYTES;
    const float thr = a.thr[rr], lse = a.lse_kept[rr];
    const int64_t tie = a.tie[rr];
    int64_t tg = -1;
    if (MODE == 0) tg = a.targets[o * a.ts_outer + i_in * a.ts_inner];
    uint8_t* keep_row = (MODE == 1 && a.keep_out) ? a.keep_out + rr * vocab : nullptr;

    auto elem = [&](float x_raw, int64_t idx, bool& keep) -> float {
        const float x = scale_logit<DT, TEMP>(x_raw, a.tparam);
        keep = x > thr || (x == thr && idx >= tie) || tie == kTieNoCut;
        if (MODE == 1) return keep ? x : -INFINITY;
        if (!keep) return 0.f;
        float d = ((idx == tg ? 1.f : 0.f) - fast_exp2((x - lse) * kLog2e)) * g;
        if constexpr (TEMP == 1) d = __fdiv_rn(Row<DT>::round_self(d), a.tparam);
        if constexpr (TEMP == 2) d = Row<DT>::round_self(d) * a.tparam;
        return d;
    };

    const int64_t head = sel_row_head<DT>(row, vocab);
    if (sel_row_head<DT>(out, vocab) != head) {
        for (int64_t e = vocab * part / a.parts + tid; e < vocab * (part + 1) / a.parts; e += kSelBlock) {
            bool keep;
            Row<DT>::store1(out, e, elem(Row<DT>::load1(row, e), e, keep));
            if (keep_row) keep_row[e] = keep ? 1 : 0;
        }
        return;
    }
    const int64_t nvec = (vocab - head) / EPV;
    const int64_t tail0 = head + nvec * EPV;
    const u32x4* xv = reinterpret_cast<const u32x4*>(row + head * Row<DT>::BYTES);
    u32x4* ov = reinterpret_cast<u32x4*>(out + head * Row<DT>::BYTES);
    // the keep flags of a vector leave as one EPV-byte store where the mask row allows it (one byte store per element
    // made the filter 27 % slower)
    using MaskWord = typename std::conditional<EPV == 8, uint64_t, uint32_t>::type;
    static_assert(sizeof(MaskWord) == EPV, "one mask byte per element of a vector");
    const bool mask_words = keep_row && ((reinterpret_cast<uintptr_t>(keep_row) + head) % EPV) == 0;
    const int64_t end = nvec * (part + 1) / a.parts;
    constexpr int kLoads = 4;  // in flight per thread
    for (int64_t v0 = nvec * part / a.parts + tid; v0 < end; v0 += kLoads * kSelBlock) {
        u32x4 q[kLoads];
#pragma unroll
        for (int u = 0; u < kLoads; ++u)
            if (v0 + u * kSelBlock < end) q[u] = __builtin_nontemporal_load(xv + v0 + u * kSelBlock);
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int64_t vi = v0 + u * kSelBlock;
            if (vi >= end) break;
            float t[EPV];
            Row<DT>::decode(q[u], t);
            MaskWord bits = 0;
#pragma unroll
            for (int k = 0; k < EPV; ++k) {
                bool keep;
                const int64_t idx = head + vi * EPV + k;
                t[k] = elem(t[k], idx, keep);
                bits |= static_cast<MaskWord>(keep ? 1 : 0) << (8 * k);
                if (keep_row && !mask_words) keep_row[idx] = keep ? 1 : 0;
            }
            if (mask_words) *reinterpret_cast<MaskWord*>(keep_row + head + vi * EPV) = bits;
            __builtin_nontemporal_store(Row<DT>::encode(t), ov + vi);
        }
    }
    if (part > 0) return;
    for (int w = 0; w < 2; ++w) {
        const int64_t e = w == 0 ? (tid < head ? tid : -1) : (tail0 + tid < vocab ? tail0 + tid : -1);
        if (e < 0) continue;
        bool keep;
        Row<DT>::store1(out, e, elem(Row<DT>::load1(row, e), e, keep));
        if (keep_row) keep_row[e] = keep ? 1 : 0;
    }
}

// Zero fill of a contiguous gradient by one workgroup per compute unit in 256 KiB spans, 6.0 TB/s, as a memset, where one
// workgroup per row reaches 5.5.  Rows that are streamed from the logits are left out where that pays: a workgroup reads which
// they are for all its spans at once, then clears what lies between them, neighbouring rows as one run (the two loads
// a row waited for in turn before its stores cost more than the stores of a short row: 4096 rows of V = 1024 bf16, all on record,
// 12 -> 70 us for the whole backward).  A 16-byte unit that a streamed row shares with its neighbour is cleared too; the row is
// written later.  1500 rows of V = 151 936, half of them streamed: 57 us when every row is cleared, 17 so.
// Everything is cleared where the flags take longer than what they can save: rows under 8 KiB, buffers of about one span per
// workgroup (4096 rows of V = 8192 on record: 10.4 and 13.0), and records of less than kMixedRecord entries.
constexpr int kFillGrid = 256;
constexpr int64_t kFillSpan = 256 * 1024, kFillShortRow = 8 * 1024, kFillSmall = kFillGrid * kFillSpan * 3 / 2;
// A forward under top-k leaves a record with room for the k: its rows are on record but for those with ties, and flags for the
// fill (4096 rows of V = 32 000: 32.7 us without, 34.5 with them) or several workgroups per row are for nothing.  Top-p alone
// leaves room for this many; nearly flat rows do not fit.
constexpr int kMixedRecord = 128;
constexpr int kFillFlags = 1024, kFillRound = kFillFlags / 2;  // flags, and spans, of a round: a span touches two rows or more
template <int DT> __global__ __launch_bounds__(256) void fill_zero_rows_kernel(SelBwdArgs a, int64_t total_bytes, double row_inverse) {
    __shared__ uint8_t clear[kFillFlags];
    __shared__ uint32_t first_row[kFillRound];  // of a span
    const u32x4 z = {0u, 0u, 0u, 0u};
    char* out = static_cast<char*>(a.out);
    auto clear_run = [&](int64_t b0, int64_t b1) {
        const int64_t v0 = b0 / 16, v1 = b1 / 16;  // whole units, from the one that holds the run's first byte
        const int n = static_cast<int>(v1 - v0);
        u32x4* zv = reinterpret_cast<u32x4*>(out) + v0;
        for (int v = threadIdx.x; v < n; v += 256) zv[v] = z;
        // the run's last bytes: the unit's other bytes are the next row's, or past the buffer's end
        const int64_t b = (v1 * 16 > b0 ? v1 * 16 : b0) + static_cast<int64_t>(threadIdx.x) * Row<DT>::BYTES;
        if (b < b1) Row<DT>::store1(out, b / Row<DT>::BYTES, 0.f);
    };
    const int64_t row_bytes = a.vocab * Row<DT>::BYTES;
    const auto span_end = [&](int64_t s0) { return s0 + kFillSpan < total_bytes ? s0 + kFillSpan : total_bytes; };
    if (row_bytes < kFillShortRow || total_bytes <= kFillSmall || a.kept_cap < kMixedRecord) {
        for (int64_t s0 = blockIdx.x * kFillSpan; s0 < total_bytes; s0 += gridDim.x * kFillSpan) clear_run(s0, span_end(s0));
        return;
    }
    // most rows that a span touches, and spans whose flags are held at a time
    const uint32_t per = static_cast<uint32_t>(kFillSpan) / static_cast<uint32_t>(row_bytes < kFillSpan ? row_bytes : kFillSpan + 1) + 2;
    const uint32_t round = kFillFlags / per;
    for (int64_t base = blockIdx.x * kFillSpan; base < total_bytes; base += round * gridDim.x * kFillSpan) {
        for (uint32_t i = threadIdx.x; i < round * per; i += 256) {
            const uint32_t k = i / per, j = i - k * per;
            const int64_t s0 = base + k * gridDim.x * kFillSpan;
            if (s0 >= total_bytes) break;
            int64_t r = static_cast<int64_t>(static_cast<double>(s0) * row_inverse);  // s0 / row_bytes, or one off
            const int64_t rest = s0 - r * row_bytes;
            r += rest < 0 ? -1 : rest >= row_bytes ? 1 : 0;
            if (j == 0) first_row[k] = static_cast<uint32_t>(r);
            r += j;
            if (r * row_bytes >= span_end(s0)) continue;
            const uint32_t o = static_cast<uint32_t>(r) / static_cast<uint32_t>(a.d_n_inner);  // (fewer than 2^31 rows)
            float g;
            clear[i] = topk_topp_on_record(a, o, r - o * a.d_n_inner, g) >= 0;
        }
        __syncthreads();
        for (uint32_t k = 0; k < round; ++k) {
            const int64_t s0 = base + k * gridDim.x * kFillSpan, s1 = span_end(s0);
            if (s0 >= total_bytes) break;
            const uint8_t* flag = clear + k * per;
            int64_t b0 = -1, b = __builtin_amdgcn_readfirstlane(first_row[k]) * row_bytes;  // a run's first byte; row by row
            for (; b < s1; b += row_bytes, ++flag) {
                const bool yes = __builtin_amdgcn_readfirstlane(*flag);
                if (yes && b0 < 0) b0 = b > s0 ? b : s0;
                if (!yes && b0 >= 0) { clear_run(b0, b); b0 = -1; }
            }
            if (b0 >= 0) clear_run(b0, s1);
        }
        __syncthreads();
    }
}

// One workgroup per row, or several for few rows (a fixed set of 512 workgroups walking the rows, which fills memory
// 10 % faster when it does nothing else, measured no gain here: with few workgroups per compute unit the record staging of a
// row is exposed; workgroups that take a part of each of three rows made an uneven round: 1500 rows of V = 151 936, half of them
// streamed, 157 -> 193 us).
template <int DT, int TEMP, int MODE>
__global__ __launch_bounds__(kSelBlock) void topk_topp_stream_kernel(SelBwdArgs a) {
    const uint32_t r = blockIdx.x / static_cast<uint32_t>(a.parts);
    topk_topp_stream_row<DT, TEMP, MODE>(a, r, static_cast<int>(blockIdx.x - r * a.parts));
}

static int temp_code3(float temperature, int mode, float* tparam) {
    if (temperature == 1.0f) { *tparam = 1.f; return 0; }
    if (mode == NRL_TEMP_DIV) { *tparam = temperature; return 1; }
    *tparam = 1.0f / temperature;
    return 2;
}

static int check_sel_rows(const nrl_rows* r, bool need_targets) {
    if (!r) return fail(NRL_E_INVALID, "rows is NULL");
    if (r->dtype != NRL_F32 && r->dtype != NRL_BF16 && r->dtype != NRL_F16) return fail(NRL_E_INVALID, "unknown logits dtype %d", r->dtype);
    if (r->n_outer < 0 || r->n_inner < 0 || r->vocab <= 0) return fail(NRL_E_INVALID, "bad shape");
    if (r->vocab >= (1ll << 31)) return fail(NRL_E_INVALID, "vocabulary too large");
    if (r->n_outer * r->n_inner > 0 && (!r->logits || (need_targets && !r->targets))) return fail(NRL_E_INVALID, "null logits or targets");
    if (r->vocab_start != 0 || r->vocab_end != r->vocab) return fail(NRL_E_UNSUPPORTED, "top-k/top-p needs the full vocabulary on this GPU");
    if (!(r->temperature > 0.f)) return fail(NRL_E_INVALID, "temperature must be positive");
    if (r->n_outer * r->n_inner >= (1ll << 31)) return fail(NRL_E_INVALID, "more than 2^31 rows in one launch");
    return NRL_OK;
}

#define NRL_SEL_DISPATCH(DT_, TC_, ...)                                                     \
    switch ((DT_) * 3 + (TC_)) {                                                            \
        case NRL_F32 * 3 + 0: { constexpr int DT = NRL_F32, TEMP = 0; __VA_ARGS__; break; }  \
        case NRL_F32 * 3 + 1: { constexpr int DT = NRL_F32, TEMP = 1; __VA_ARGS__; break; }  \
        case NRL_F32 * 3 + 2: { constexpr int DT = NRL_F32, TEMP = 2; __VA_ARGS__; break; }  \
        case NRL_BF16 * 3 + 0: { constexpr int DT = NRL_BF16, TEMP = 0; __VA_ARGS__; break; } \
        case NRL_BF16 * 3 + 1: { constexpr int DT = NRL_BF16, TEMP = 1; __VA_ARGS__; break; } \
        case NRL_BF16 * 3 + 2: { constexpr int DT = NRL_BF16, TEMP = 2; __VA_ARGS__; break; } \
        case NRL_F16 * 3 + 0: { constexpr int DT = NRL_F16, TEMP = 0; __VA_ARGS__; break; }  \
        case NRL_F16 * 3 + 1: { constexpr int DT = NRL_F16, TEMP = 1; __VA_ARGS__; break; }  \
        default: { constexpr int DT = NRL_F16, TEMP = 2; __VA_ARGS__; break; }              \
    }

}  // namespace nrl

using namespace nrl;

extern "C" int nrl_topk_topp_logprob_fwd(const nrl_rows* rows, int64_t top_k, float top_p, float* logprob_out,
                                         float* thr_out, int32_t* tie_out, float* lse_kept_out,
                                         float* logprob_unfiltered_out, float* lse_full_out, int32_t* kept_count_out,
                                         int32_t* kept_index_out, float* kept_value_out, int64_t kept_capacity,
                                         void* stream) {
    if (int e = check_sel_rows(rows, logprob_out != nullptr)) return e;
    const bool use_k = top_k > 0, use_p = top_p < 1.0f;
    if (!use_k && !use_p) return fail(NRL_E_INVALID, "neither top-k nor top-p is active");
    if (use_p && !(top_p > 0.f)) return fail(NRL_E_INVALID, "top_p must be in (0, 1]");
    const int64_t n = rows->n_outer * rows->n_inner;
    if (n == 0) return NRL_OK;
    if (!thr_out || !tie_out || !lse_kept_out) return fail(NRL_E_INVALID, "null state output");
    if (kept_count_out && (!kept_index_out || !kept_value_out || kept_capacity < 1 || kept_capacity > kCapSmall))
        return fail(NRL_E_INVALID, "kept-set record: index and value outputs and a capacity in [1, %d] are needed", kCapSmall);
    SelArgs a;
    a.kept_n = kept_count_out; a.kept_idx = kept_index_out; a.kept_x = kept_value_out; a.kept_cap = static_cast<int>(kept_capacity);
    a.logits = rows->logits; a.n_inner = rows->n_inner; a.vocab = rows->vocab;
    a.stride_outer = rows->stride_outer; a.stride_inner = rows->stride_inner;
    a.targets = rows->targets; a.ts_outer = rows->tgt_stride_outer; a.ts_inner = rows->tgt_stride_inner;
    a.top_k = use_k ? static_cast<int>(top_k > (1ll << 30) ? (1ll << 30) : top_k) : 0;
    a.top_p = use_p ? top_p : 1.0f;
    a.logprob = logprob_out; a.thr = thr_out; a.tie = tie_out; a.lse_kept = lse_kept_out;
    a.logprob_full = logprob_unfiltered_out; a.lse_full = lse_full_out;
    const int tc = temp_code3(rows->temperature, rows->temp_mode, &a.tparam);
    const bool full = !use_k || logprob_unfiltered_out != nullptr || lse_full_out != nullptr;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool small = use_k && a.top_k <= kSmallTopK;
    if (!use_k && rows->dtype == NRL_BF16) {
        // (values of fp16 and fp32 are too many for a bin each)
        if (tc == 0) nucleus_count_kernel<0><<<dim3((unsigned)n), dim3(kNucThreads), 0, s>>>(a);
        else if (tc == 1) nucleus_count_kernel<1><<<dim3((unsigned)n), dim3(kNucThreads), 0, s>>>(a);
        else nucleus_count_kernel<2><<<dim3((unsigned)n), dim3(kNucThreads), 0, s>>>(a);
    } else if (!use_k) {
        NRL_SEL_DISPATCH(rows->dtype, tc, if constexpr (DT != NRL_BF16)
                             topk_topp_fwd_kernel<DT, TEMP, true, kCap, true><<<dim3((unsigned)n), dim3(kSelBlock), 0, s>>>(a));
    } else if (full && small) {
        NRL_SEL_DISPATCH(rows->dtype, tc, topk_topp_fwd_kernel<DT, TEMP, true, kCapSmall><<<dim3((unsigned)n), dim3(kSelBlock), 0, s>>>(a));
    } else if (full) {
        NRL_SEL_DISPATCH(rows->dtype, tc, topk_topp_fwd_kernel<DT, TEMP, true, kCap><<<dim3((unsigned)n), dim3(kSelBlock), 0, s>>>(a));
    } else if (small) {
        NRL_SEL_DISPATCH(rows->dtype, tc, topk_topp_fwd_kernel<DT, TEMP, false, kCapSmall><<<dim3((unsigned)n), dim3(kSelBlock), 0, s>>>(a));
    } else {
        NRL_SEL_DISPATCH(rows->dtype, tc, topk_topp_fwd_kernel<DT, TEMP, false, kCap><<<dim3((unsigned)n), dim3(kSelBlock), 0, s>>>(a));
    }
    if (int e = check_launch("topk_topp_logprob_fwd")) return e;
    // rows the candidate list could not hold are finished here; with none, every workgroup leaves after
    // reading its rows' markers
    const unsigned grid = static_cast<unsigned>(n < kWideGrid ? n : kWideGrid);
    NRL_SEL_DISPATCH(rows->dtype, tc, topk_topp_wide_kernel<DT, TEMP><<<dim3(grid), dim3(kSelBlock), 0, s>>>(a, n));
    return check_launch("topk_topp_logprob_fwd (wide rows)");
}

extern "C" int nrl_topk_topp_logprob_bwd(const nrl_rows* rows, const float* thr, const int32_t* tie,
                                         const float* lse_kept, const float* grad, int64_t grad_stride_outer,
                                         int64_t grad_stride_inner, const int32_t* kept_count, const int32_t* kept_index,
                                         const float* kept_value, int64_t kept_capacity, void* dlogits, int64_t d_n_inner,
                                         int64_t d_stride_outer, int64_t d_stride_inner, void* stream) {
    if (int e = check_sel_rows(rows, true)) return e;
    if (d_n_inner < rows->n_inner) return fail(NRL_E_INVALID, "d_n_inner < n_inner");
    const int64_t n = rows->n_outer * d_n_inner;
    if (n == 0) return NRL_OK;
    if (n >= (1ll << 31)) return fail(NRL_E_INVALID, "more than 2^31 rows in one launch");
    if (!dlogits || (rows->n_outer * rows->n_inner > 0 && (!thr || !tie || !lse_kept || !grad))) return fail(NRL_E_INVALID, "null argument");
    SelBwdArgs a;
    a.logits = rows->logits; a.n_inner = rows->n_inner; a.vocab = rows->vocab;
    a.stride_outer = rows->stride_outer; a.stride_inner = rows->stride_inner;
    a.targets = rows->targets; a.ts_outer = rows->tgt_stride_outer; a.ts_inner = rows->tgt_stride_inner;
    a.thr = thr; a.tie = tie; a.lse_kept = lse_kept; a.grad = grad;
    a.gs_outer = grad_stride_outer; a.gs_inner = grad_stride_inner;
    a.out = dlogits; a.d_n_inner = d_n_inner; a.ds_outer = d_stride_outer; a.ds_inner = d_stride_inner;
    a.keep_out = nullptr;
    if (kept_count && (!kept_index || !kept_value || kept_capacity < 1)) return fail(NRL_E_INVALID, "incomplete kept-set record");
    a.kept_n = kept_count; a.kept_idx = kept_index; a.kept_x = kept_value; a.kept_cap = static_cast<int>(kept_capacity);
    const int tc = temp_code3(rows->temperature, rows->temp_mode, &a.tparam);
    hipStream_t s = static_cast<hipStream_t>(stream);
    // With the kept sets on record nearly every row is zeros plus a few entries.  A gradient buffer that is one
    // contiguous block is then zero-filled flat, which writes faster than row by row, and the row launch only adds
    // the entries (and streams the rows that are not on record).  For a strided buffer the record is left unused.
    const int64_t elt = rows->dtype == NRL_F32 ? 4 : 2;
    a.prefilled = kept_count && d_stride_inner == rows->vocab && d_stride_outer == d_n_inner * rows->vocab &&
                  (reinterpret_cast<uintptr_t>(dlogits) & 15) == 0;
    if (a.prefilled && rows->logits && rows->n_outer * rows->n_inner > 0) {
        // A gradient written over the logits (allowed, as for nrl_logprob_bwd) must not be cleared first: rows that
        // are not on record still stream from the logits.  Such a call takes the row-by-row path, which reads a
        // vector before it overwrites it.
        const uintptr_t d0 = reinterpret_cast<uintptr_t>(dlogits), d1 = d0 + static_cast<uintptr_t>(n * rows->vocab * elt);
        const uintptr_t l0 = reinterpret_cast<uintptr_t>(rows->logits);
        const int64_t so = rows->stride_outer < 0 ? -rows->stride_outer : rows->stride_outer;
        const int64_t si = rows->stride_inner < 0 ? -rows->stride_inner : rows->stride_inner;
        const uintptr_t l1 = l0 + static_cast<uintptr_t>(((rows->n_outer - 1) * so + (rows->n_inner - 1) * si + rows->vocab) * elt);
        if (d0 < l1 && l0 < d1) a.prefilled = 0;
    }
    if (a.prefilled) {
        const int64_t total = n * rows->vocab * elt;
        const double inverse = 1.0 / static_cast<double>(rows->vocab * elt);
        if (rows->dtype == NRL_F32) fill_zero_rows_kernel<NRL_F32><<<dim3(kFillGrid), dim3(256), 0, s>>>(a, total, inverse);
        else fill_zero_rows_kernel<NRL_BF16><<<dim3(kFillGrid), dim3(256), 0, s>>>(a, total, inverse);  // (zeros of two bytes, either type)
    }
    // Parts of at least 32 KiB, as long as the rows alone are too few to keep the chip busy to the end.  1500 rows of V = 151 936 in
    // 1, 2, 3 and 4 parts: half of them streamed 154, 154, 149 and 146 us (medians 176, 164, 172, 157); all on record 5.6, 7.0, 8.0
    // and 10.1, so one part where that is to be expected.
    const int64_t most = a.prefilled && a.kept_cap < kMixedRecord ? 1 : rows->vocab * elt / 32768;
    a.parts = static_cast<int>(6144 / n < most ? 6144 / n : most);
    if (a.parts < 1) a.parts = 1;
    NRL_SEL_DISPATCH(rows->dtype, tc, topk_topp_stream_kernel<DT, TEMP, 0><<<dim3((unsigned)(n * a.parts)), dim3(kSelBlock), 0, s>>>(a));
    return check_launch("topk_topp_logprob_bwd");
}

extern "C" int nrl_topk_topp_filter(const nrl_rows* rows, const float* thr, const int32_t* tie, void* filtered_out,
                                    int64_t f_stride_outer, int64_t f_stride_inner, uint8_t* keep_out, void* stream) {
    if (int e = check_sel_rows(rows, false)) return e;
    const int64_t n = rows->n_outer * rows->n_inner;
    if (n == 0) return NRL_OK;
    if (!thr || !tie || !filtered_out) return fail(NRL_E_INVALID, "null argument");
    SelBwdArgs a;
    a.logits = rows->logits; a.n_inner = rows->n_inner; a.vocab = rows->vocab;
    a.stride_outer = rows->stride_outer; a.stride_inner = rows->stride_inner;
    a.targets = nullptr; a.ts_outer = 0; a.ts_inner = 0;
    a.thr = thr; a.tie = tie; a.lse_kept = thr; a.grad = nullptr; a.gs_outer = 0; a.gs_inner = 0;
    a.out = filtered_out; a.d_n_inner = rows->n_inner; a.ds_outer = f_stride_outer; a.ds_inner = f_stride_inner;
    a.keep_out = keep_out;
    a.kept_n = nullptr; a.kept_idx = nullptr; a.kept_x = nullptr; a.kept_cap = 0; a.prefilled = 0; a.parts = 1;
    const int tc = temp_code3(rows->temperature, rows->temp_mode, &a.tparam);
    hipStream_t s = static_cast<hipStream_t>(stream);
    NRL_SEL_DISPATCH(rows->dtype, tc, topk_topp_stream_kernel<DT, TEMP, 1><<<dim3((unsigned)n), dim3(kSelBlock), 0, s>>>(a));
    return check_launch("topk_topp_filter");
}
