// The single pass over logits rows: log-sum-exp -> token logprob -> d loss / d logprob -> dlogits, with the row held on chip
// (registers plus an LDS slice) between the reduction and the gradient, so the logits are read once and the gradient written
// once (2 * V * sizeof(logit) per token instead of 3).  Valid when d loss / d logprob of a token depends only on that token
// and on per-sequence quantities that do not involve the current logprobs: everything except sequence-level probability
// ratios (GSPO) and the positive-example NLL term.  Tokens whose mask is zero are not evaluated: their gradient row is
// zero-filled without reading the logits and their logprob is reported as 0.
#pragma once

#include <float.h>

#include "grpo_token.hpp"

namespace nrl {

constexpr int kFusedMaxRegVec = 16;  // at most 16 16-byte vectors per lane held in registers ...
constexpr int kFusedLdsVec = 4;      // ... and 4 in LDS
constexpr int kFusedMaxVec = kFusedMaxRegVec + kFusedLdsVec;

// What the pass needs to know about a row, 64 bytes written by fused_prep_kernel: a wave reads it with one load, a word per
// lane, a row ahead of its use.
enum { R_LIVE = 0, R_PREV, R_GEN, R_REF, R_ADV, R_TM, R_SMV, R_XT, R_TLOC, R_SEQ, R_POS, R_WORDS = 16 };

struct FusedArgs {
    nrl_grpo_cfg cfg;
    nrl_grpo_inputs in;  // lp / lpu unused
    const void* logits;
    int64_t n_inner, d_n_inner, vocab, stride_outer, stride_inner;
    const int64_t* targets;
    int64_t ts_outer, ts_inner, vstart, vend;
    float tparam, loss_scale;
    void* dlogits;
    int64_t ds_outer, ds_inner;
    float* lp_out;     // [B, n_inner]
    float* seq_stats;  // [B, 3]: seq_den, seq_w, seq_keep
    uint32_t* rec;     // [B * n_inner, R_WORDS]; packed: [rows, R_WORDS]
    double* parts;     // [B, chunks, P_COUNT]
    // packed mode (cu != NULL): the logits are one row of `total` positions, sequence s occupies
    // [cu[s], cu[s+1]); the loss inputs stay [n_seq, n_inner]
    const int32_t* cu;
    int64_t n_seq;
    int pre_rolled;
    int any_row;       // rows off the 16-byte grid, or longer than the chip holds
    float4* row_grad;  // NULL or [rows]: (d loss / d logprob at loss_scale 1, log-sum-exp, target or -1 as bits, 0) of every row, from
                       // which the gradient can be written again; zeros for rows without a token
};

struct FusedLaunch {
    FusedArgs a;
    int temp;  // 0, 1 (divide), 2 (multiply)
    bool packed;
    int64_t n_rows;
    bool any_row;  // rows off the 16-byte grid, or longer than the chip holds
    int compute_units;
    hipStream_t stream;
};
void launch_fused_f32(const FusedLaunch& l);
void launch_fused_bf16(const FusedLaunch& l);
void launch_fused_f16(const FusedLaunch& l);

template <bool PACKED>
__device__ __forceinline__ int64_t fused_row_offset(const FusedArgs& a, int64_t r, int64_t so, int64_t si) {
    if (PACKED) return r * si;
    const int64_t o = r / a.d_n_inner;
    return o * so + (r - o * a.d_n_inner) * si;
}

// 16 bytes per lane from base + offset (uniform base, `bytes` behind it) to consecutive LDS addresses from dst (uniform) on
__device__ __forceinline__ void load_to_lds(const char* base, int bytes, int offset, u32x4* dst) {
#ifdef __HIP_DEVICE_COMPILE__  // the resource type does not exist for the host pass
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, bytes, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)dst, 16, offset, 0, 0, 0);
#endif
}

// Persistent workgroups: workgroup w walks rows w, w + gridDim.x, ...  A row's gradient goes out as one burst of stores, and
// behind it the loads of the next row this workgroup evaluates (registers by ordinary loads, the LDS slice by direct
// global-to-LDS loads), whose online (max, sum) is advanced as they arrive.  The pass is bound by HBM, and HBM serves long
// runs of reads and of writes better than the two mixed: with every slot refilled right behind its store, 8 x 4096 rows
// of V = 151936 bf16 took 3.65 ms, in runs 3.49 ms (18.4 GB, 5.26 TB/s), although the former overlaps more.
// What lies between two rows is kept short: the row's inputs come in one load a row ahead, every wave evaluates the token
// by itself (no broadcast, no second barrier), and only what the gradient needs is evaluated; the terms of the metrics
// follow in the reduction behind the pass (4 x 1024 rows: 538 -> 520 us for the whole call).
// Slot order q = 0 .. kVec-1: the LDS slots come first (vector NREG + q), then the register slots (vector q - NLDS).
// NREG is the number of register slots the instantiation carries (the row must fit NREG + NLDS
// slots); shorter rows take a smaller instantiation instead of idling through unused slots, and smaller workgroups of which
// several share a compute unit, so that one's stretch between rows is covered by the others' memory operations.
//
// EDGE: rows need not start or end on 16 bytes.  The vectors of a row begin at its first 16-byte boundary; the up to 7 elements
// before it and the tail shorter than a vector are one element each of the first 32 lanes.  (Input and output rows sit alike.)
// LONG (1024 threads): vectors past the on-chip slots are read twice.  They are the last ones read of a row and the first
// ones its gradient needs, in reverse order, so that the second read finds them in the 256 MB cache: at most 256 rows' excess
// lies between the two (72 MB at V = 151936 fp32, 185 MB in the longest rows taken, 1 MiB; gradient stores of other rows pass
// through the same cache meanwhile).  The counters of L2 fills see both reads alike; what speaks for the cache is the rate
// with the second read counted: whole calls at 5.2, 5.6 and 5.85 TB/s for V = 151936, 200000 and 262144 fp32, where rows that
// fit are served at 4.9 - 5.1.
// Both against the three passes (logprobs, loss, gradient) such rows took before, whole calls: 2 x 1024 rows of V = 151936 fp32
// 710 -> 498 us, of V = 262144 bf16 577 -> 478, 2 x 512 of V = 262144 fp32 574 -> 447; 3 x 701 rows of V = 50257 bf16 152 -> 144,
// 4 x 2048 of V = 20001 200 -> 156; 128 rows of V = 262143 fp32 186 -> 105.
template <int DT, int TEMP, int BLOCK, int NREG, int NLDS, bool EDGE, bool LONG, bool PACKED>
__global__ __launch_bounds__(BLOCK, 4) void fused_logits_loss_kernel(FusedArgs a, int64_t n_rows) {
    constexpr int EPV = Row<DT>::EPV;
    constexpr int kVec = NREG + NLDS;
    constexpr int kWavesPerBlock = BLOCK / kWave;
    __shared__ u32x4 stash[NLDS * BLOCK];
    __shared__ Lse sm_l[kWavesPerBlock];
    const nrl_grpo_cfg& c = a.cfg;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    int nvec = static_cast<int>(a.vocab / EPV), head = 0;  // of the row at hand
    const int64_t step = gridDim.x;
    const u32x4 zero = {0u, 0u, 0u, 0u};

    auto out_row = [&](int64_t r) -> char* {
        return static_cast<char*>(a.dlogits) + fused_row_offset<PACKED>(a, r, a.ds_outer, a.ds_inner) * Row<DT>::BYTES;
    };
    auto in_row = [&](int64_t r) -> const char* {
        return static_cast<const char*>(a.logits) + fused_row_offset<PACKED>(a, r, a.stride_outer, a.stride_inner) * Row<DT>::BYTES;
    };
    // Slot q holds vector slot_vec(q) of the row.  Lanes past the end of the row are pointed at the
    // row's last vector instead: they load, compute and store exactly what that vector's own lane does
    // (harmless duplicates), so there is no divergent branch around the memory operations and they stay in flight
    // together.
    auto slot_vec = [&](int q) -> int { return tid + (q < NLDS ? NREG + q : q - NLDS) * BLOCK; };
    // (recomputed at every use from an opaque copy of the lane index: twenty precomputed offsets would
    // not fit in the register file next to the row)
    auto slot_cl = [&](int q) -> int {
        int t = tid;
        asm volatile("" : "+v"(t));
        return min(t + (q < NLDS ? NREG + q : q - NLDS) * BLOCK, nvec - 1);
    };
    auto vec_at = [&](const char* base, int vc) -> const u32x4* {  // uniform base + 32-bit lane offset
        return reinterpret_cast<const u32x4*>(base + static_cast<uint32_t>(vc) * 16u);
    };
    auto place = [&](const char* row) {  // head and nvec of a row, which its output shares
        if (!EDGE) return;
        head = static_cast<int>(((16 - (reinterpret_cast<uintptr_t>(row) & 15)) & 15) / Row<DT>::BYTES);
        nvec = (static_cast<int>(a.vocab) - head) / EPV;
    };
    // this lane's element outside the vectors, or -1
    auto edge_at = [&]() -> int {
        if (tid < head) return tid;
        const int t = head + nvec * EPV + tid - 16;
        return tid >= 16 && t < static_cast<int>(a.vocab) ? t : -1;
    };
    float edge_x = 0.f;
    auto load_rec = [&](int64_t r) -> uint32_t {
        if (r >= n_rows) return 0u;
        if (!PACKED) {  // a record per token: rows behind a sequence's last token have none
            const int64_t o = r / a.d_n_inner, i = r - o * a.d_n_inner;
            if (i >= a.n_inner) return 0u;
            r = o * a.n_inner + i;
        }
        return a.rec[r * R_WORDS + (lane & (R_WORDS - 1))];
    };
    auto word = [&](uint32_t rec, int k) -> uint32_t { return __builtin_amdgcn_readlane(static_cast<int>(rec), k); };
    // First row at or after r (in this workgroup's walk) whose token takes part in the loss, with its record; rec is row
    // r's on entry.  Rows passed over are dropped positions or masked tokens: zero gradient, nothing read.
    auto advance = [&](int64_t r, uint32_t& rec) -> int64_t {
        while (r < n_rows && word(rec, R_LIVE) == 0u) {
            char* out = out_row(r);
            place(out);
            u32x4* ov = reinterpret_cast<u32x4*>(out + head * Row<DT>::BYTES);
            rec = load_rec(r + step);
            for (int v = tid; v < nvec; v += BLOCK) ov[v] = zero;
            if (EDGE && edge_at() >= 0) Row<DT>::store1(out, edge_at(), 0.f);
            r += step;
        }
        return r;
    };
    auto load_stats = [&](uint32_t rec) -> float { return a.seq_stats[static_cast<int64_t>(word(rec, R_SEQ)) * 3 + (lane < 3 ? lane : 0)]; };
    u32x4 regs[NREG];
    Lse acc;
    // LDS slot q of the incoming row: global memory -> LDS without passing through registers; each wave
    // fills the 1 KiB of the slot that its own lanes read back.  (Buffer loads: the compiler counts them like any other
    // memory operation.  global_load_lds it takes for an access that may complete out of order, after which the wait for the
    // first register load is a wait for everything in flight.)
    auto lds_fill = [&](const char* base, int q) {
        u32x4* dst = stash + q * BLOCK + (tid & ~(kWave - 1));
        load_to_lds(base, nvec * 16, slot_cl(q) * 16, dst);
    };
    auto fold_vec = [&](u32x4 raw, int v) {  // vector v of the incoming row -> running sum; lanes past the row add nothing
        if (v >= nvec) raw = u32x4{Row<DT>::NEG_INF_WORD, Row<DT>::NEG_INF_WORD, Row<DT>::NEG_INF_WORD, Row<DT>::NEG_INF_WORD};
        float t[EPV];
        Row<DT>::decode(raw, t);
#pragma unroll
        for (int k = 0; k < EPV; ++k) t[k] = scale_logit<DT, TEMP>(t[k], a.tparam);
        lse_push<EPV>(acc, t);
    };
    auto fold = [&](int q) {
        fold_vec(q < NLDS ? stash[(q < NLDS ? q : 0) * BLOCK + tid] : regs[q < NLDS ? 0 : q - NLDS], slot_vec(q));
    };
    constexpr int kAhead = 4;                    // vectors past the slots in flight per lane
    constexpr int kStride = kAhead * BLOCK;
    const int past = kVec * BLOCK;
    // the direct-to-LDS loads are not tracked against later LDS reads by the compiler: wait for them
    // (and everything older) by hand before the first read of a refilled LDS slot
    auto wait_lds_fill = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };

    auto load_row = [&](const char* row) {  // the row onto the chip, and its (max, sum)
        place(row);
        const char* base = row + head * Row<DT>::BYTES;
#pragma unroll
        for (int q = 0; q < NLDS; ++q) lds_fill(base, q);
#pragma unroll
        for (int q = NLDS; q < kVec; ++q) regs[q - NLDS] = __builtin_nontemporal_load(vec_at(base, slot_cl(q)));
        if (EDGE && edge_at() >= 0) edge_x = Row<DT>::load1(row, edge_at());
        __builtin_amdgcn_sched_barrier(0);  // all loads in flight before the first is waited for
        acc.m = -FLT_MAX;
        acc.s = 0.f;
#pragma unroll
        for (int q = NLDS; q < kVec; ++q) fold(q);
        wait_lds_fill();
#pragma unroll
        for (int q = 0; q < NLDS; ++q) fold(q);
        if (EDGE && edge_at() >= 0) lse_push1(acc, scale_logit<DT, TEMP>(edge_x, a.tparam));
        if (LONG) {
            for (int v0 = past; v0 < nvec; v0 += kStride) {
                u32x4 x[kAhead];
#pragma unroll
                for (int j = 0; j < kAhead; ++j) x[j] = *vec_at(base, min(v0 + j * BLOCK + tid, nvec - 1));
#pragma unroll
                for (int j = 0; j < kAhead; ++j) fold_vec(x[j], v0 + j * BLOCK + tid);
            }
        }
    };

    uint32_t rec = load_rec(blockIdx.x);
    int64_t r = advance(blockIdx.x, rec);
    float stats = 0.f;
    uint32_t ahead = 0u;  // record of row r + step
    if (r < n_rows) {
        stats = load_stats(rec);
        ahead = load_rec(r + step);
        load_row(in_row(r));
    }
    while (r < n_rows) {
        char* const out = out_row(r);
        char* const ov = out + head * Row<DT>::BYTES;
        const Lse tot = block_lse<kWavesPerBlock>(acc, sm_l);
        const int tloc = static_cast<int>(word(rec, R_TLOC));
        const float log_s = logf(tot.s), lse = tot.m + log_s;
        float g;
        {
            auto in = [&](int k) { return __uint_as_float(word(rec, k)); };
            auto stat = [&](int k) { return __uint_as_float(word(__float_as_uint(stats), k)); };
            const float lp = tloc >= 0 ? (in(R_XT) - tot.m) - log_s : 0.f;
            SeqStats st;
            st.seq_den = stat(0); st.seq_ratio = 1.f; st.seq_w = stat(1); st.seq_keep = stat(2);
            TokenIn ti;
            ti.lp = lp; ti.lpu = lp;
            ti.prev = c.force_on_policy_ratio ? lp : in(R_PREV);
            ti.gen = in(R_GEN); ti.ref = in(R_REF); ti.adv = in(R_ADV); ti.tm = in(R_TM); ti.smv = in(R_SMV);
            ti.correct = 0.f;
            ti.den_s = valid_seqs(a.in) + 1e-8f;
            ti.den_t = valid_toks(a.in) + 1e-8f;
            const TokenOut tok = token_eval<false>(c, st, ti);
            const float g1 = tok.d_actor + tok.d_lpu;
            g = g1 * a.loss_scale;
            if (EDGE && tid == 0 && a.row_grad) a.row_grad[r] = make_float4(g1, lse, __int_as_float(tloc), 0.f);
            if (tid == 0) a.lp_out[static_cast<int64_t>(word(rec, R_SEQ)) * a.n_inner + word(rec, R_POS)] = lp;
        }
        const int tvec = tloc >= head ? (tloc - head) / EPV : -1;  // (of a target in the tail: no vector of the row)
        const int tsub = tloc >= head ? (tloc - head) % EPV : -1;
        const RowGrad rg(lse, g, a.tparam);
        if (EDGE && edge_at() >= 0) Row<DT>::store1(out, edge_at(), grad_elem<DT, TEMP>(edge_x, edge_at() == tloc, rg));
        if (LONG) {
            const char* base = in_row(r) + head * Row<DT>::BYTES;
            for (int v0 = past + (nvec - 1 - past) / kStride * kStride; v0 >= past; v0 -= kStride) {
                u32x4 x[kAhead];
#pragma unroll
                for (int j = 0; j < kAhead; ++j) x[j] = __builtin_nontemporal_load(vec_at(base, min(v0 + j * BLOCK + tid, nvec - 1)));
#pragma unroll
                for (int j = 0; j < kAhead; ++j) {
                    const int v = v0 + j * BLOCK + tid;
                    if (v < nvec) __builtin_nontemporal_store(grad_vec<DT, TEMP>(x[j], v == tvec ? tsub : -1, rg), const_cast<u32x4*>(vec_at(ov, v)));
                }
            }
        }
#pragma unroll
        for (int q = 0; q < kVec; ++q) {
            const int vc = slot_cl(q);
            const u32x4 raw = q < NLDS ? stash[(q < NLDS ? q : 0) * BLOCK + tid] : regs[q < NLDS ? 0 : q - NLDS];
            const u32x4 d = grad_vec<DT, TEMP>(raw, vc == tvec ? tsub : -1, rg);
            __builtin_nontemporal_store(d, const_cast<u32x4*>(vec_at(ov, vc)));
        }
        __builtin_amdgcn_sched_barrier(0);  // the stores stay together, and ahead of the loads
        uint32_t rec_n = ahead;
        const int64_t rn = advance(r + step, rec_n);
        const float stats_n = load_stats(rn < n_rows ? rec_n : rec);
        ahead = load_rec(rn + step);
        if (rn < n_rows) load_row(in_row(rn));
        // sm_l is rewritten only behind the first barrier of the next block_lse, which every thread passes after reading it
        r = rn;
        rec = rec_n;
        stats = stats_n;
    }
}

template <int DT, int TEMP, int BLOCK, int NREG, int NLDS = kFusedLdsVec, bool EDGE = false, bool LONG = false> void fused_launch(const FusedLaunch& l) {
    // as many workgroups as are resident together: 1024 threads per compute unit at 128 registers, 64 (LONG: 128) KiB of LDS
    const int64_t resident = static_cast<int64_t>(l.compute_units) * (1024 / BLOCK);
    const dim3 grid(static_cast<unsigned>(l.n_rows < resident ? l.n_rows : resident)), block(BLOCK);
    if (l.packed) fused_logits_loss_kernel<DT, TEMP, BLOCK, NREG, NLDS, EDGE, LONG, true><<<grid, block, 0, l.stream>>>(l.a, l.n_rows);
    else fused_logits_loss_kernel<DT, TEMP, BLOCK, NREG, NLDS, EDGE, LONG, false><<<grid, block, 0, l.stream>>>(l.a, l.n_rows);
}
// Slots past the end of a row are loaded, computed and stored all the same, so a row takes the form with the fewest that
// hold it.  Whole calls of bf16 rows against the 16-slot form of the same workgroup size, on the 16-byte grid and off it:
// 8 register slots, at V = 24576 / 49152 / 98304: 9 and 12 % faster (256 threads), 14 and 21 % (512), 17 and 16 % (1024); 12: 256
// threads 8 and 11 % at V = 25600, 3 and 6 at 28672, 0 and 3 at 30720, 3 and 2 % slower at 32768; 512 threads 1 and 10 % at
// 65536; 1024 threads 4 and 8 % at 131072; 4 at V = 16384: 31 %.
template <int DT, int TEMP, int BLOCK> void fused_launch(const FusedLaunch& l, int64_t slots) {
    if (slots <= 12) fused_launch<DT, TEMP, BLOCK, 8>(l);
    else if (slots <= 16) fused_launch<DT, TEMP, BLOCK, 12>(l);
    else fused_launch<DT, TEMP, BLOCK, 16>(l);
}
template <int DT, int TEMP, int BLOCK> void fused_launch_edge(const FusedLaunch& l, int64_t slots) {
    if (slots <= 12) fused_launch<DT, TEMP, BLOCK, 8, kFusedLdsVec, true>(l);
    else if (slots <= 16) fused_launch<DT, TEMP, BLOCK, 12, kFusedLdsVec, true>(l);
    else fused_launch<DT, TEMP, BLOCK, 16, kFusedLdsVec, true>(l);
}
template <int DT, int TEMP> void fused_launch(const FusedLaunch& l) {
    const int64_t nvec = l.a.vocab / Row<DT>::EPV;
    auto slots = [&](int block) { return (nvec + block - 1) / block; };
    // the smallest workgroup that holds the row
    if (slots(256) <= 8) fused_launch<DT, TEMP, 256, 4>(l);
    else if (slots(256) <= kFusedMaxVec) fused_launch<DT, TEMP, 256>(l, slots(256));
    else if (slots(512) <= kFusedMaxVec) fused_launch<DT, TEMP, 512>(l, slots(512));
    else fused_launch<DT, TEMP, 1024>(l, slots(1024));
}
template <int DT, int TEMP> void fused_launch_edge(const FusedLaunch& l) {
    const int64_t nvec = l.a.vocab / Row<DT>::EPV;
    auto slots = [&](int block) { return (nvec + block - 1) / block; };
    if (slots(256) <= kFusedMaxVec) fused_launch_edge<DT, TEMP, 256>(l, slots(256));
    else if (slots(512) <= kFusedMaxVec) fused_launch_edge<DT, TEMP, 512>(l, slots(512));
    else if (slots(1024) <= kFusedMaxVec) fused_launch_edge<DT, TEMP, 1024>(l, slots(1024));
    else fused_launch<DT, TEMP, 1024, 12, 8, true, true>(l);  // the larger LDS share leaves registers for the vectors past it
}
template <int DT> void fused_launch(const FusedLaunch& l) {
    if (l.any_row) {  // (no divide: the caller's own is a multiplication)
        if (l.temp == 0) fused_launch_edge<DT, 0>(l);
        else fused_launch_edge<DT, 2>(l);
        return;
    }
    if (l.temp == 0) fused_launch<DT, 0>(l);
    else if (l.temp == 1) fused_launch<DT, 1>(l);  // NRL_TEMP_DIV, for direct callers: the wrappers' divide is PyTorch's on the GPU, a multiplication
    else fused_launch<DT, 2>(l);
}

}  // namespace nrl
