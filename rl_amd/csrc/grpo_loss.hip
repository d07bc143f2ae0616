// K4: clipped policy-gradient (GRPO family) loss, its gradient with respect to the token
// logprobs and all metrics, fused.
//
// Launch 1 (one workgroup per sequence row): per-row statistics that the sequence-level modes
// need (token count, mean log-ratio, summed IS log-weight), then every per-token term - ratio,
// clip / dual clip / CISPO, k1-k3 KL with its clamps and importance weight, truncated IS - with
// the analytic gradient written straight to dlp, and per-row partial sums of the loss and of
// every diagnostic in float64.  Launch 2 (one workgroup): fixed-order reduction of the row
// partials, normalisation, and the metrics record the host reads back with a single copy.
// Token arithmetic is fp32 like the PyTorch ops it replaces; only the accumulations are wider.
//
// The data are [B, S-1] fp32 arrays (a few tens of bytes per token), so this stage is launch-
// latency bound; it exists to remove ~40 small kernels and ~15 device->host syncs per call.

#include <float.h>
#include <math.h>

#include <mutex>

#include "common.hpp"
#include "fused_rows.hpp"
#include "grpo_token.hpp"
#include "row_grad.hpp"

namespace nrl {

constexpr int kLossBlock = 256;
constexpr int kLossWaves = kLossBlock / kWave;
// The kernels with one workgroup per sequence have as many workgroups as a microbatch has sequences, 1 - 16: what they cost is
// the number of dependent steps of one workgroup, so a sequence gets the largest there is.  2 sequences of
// 2048 tokens: rows kernel 26.8 -> 16.7 us, 3 of 701: 16.0 -> 11.4 us (256 against 1024 threads).
constexpr int kSeqBlock = 1024;
constexpr int kSeqWaves = kSeqBlock / kWave;

// Sums of N values over a workgroup with two barriers in all; thread k < N returns sum k, waves added in ascending order.
template <int N, int NW> __device__ __forceinline__ double block_sums(const double (&v)[N], double* smem /* [NW * N] */) {
    const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const double s = wave_sum_double(v[k]);
        if (lane == 0) smem[w * N + k] = s;
    }
    __syncthreads();
    double t = 0;
    if (tid < N)
        for (int i = 0; i < NW; ++i) t += smem[i * N + tid];
    return t;
}
// one value, returned by every thread
__device__ __forceinline__ double seq_block_sum(double v, double* smem) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    v = wave_sum_double(v);
    __syncthreads();
    if (lane == 0) smem[w] = v;
    __syncthreads();
    double t = 0;
#pragma unroll
    for (int i = 0; i < kSeqWaves; ++i) t += smem[i];
    return t;
}
constexpr int kSeqSmem = kSeqWaves * P_R_MIN;

// slot k of a sequence's row of partials, from the sum of its tokens' terms
__device__ __forceinline__ double row_part(const nrl_grpo_cfg& c, int k, double sum, const SeqStats& st, float smv) {
    if (!c.token_level_loss && (k == P_ACTOR || k == P_KL))  // sequence-level: masked mean over tokens, then weight by sample_mask
        return static_cast<double>(static_cast<float>(sum) / st.seq_den) * smv;
    if (k == P_SAMPLE_MASK) return smv;
    if (k == P_SEQ_W) {
        double v = c.tis_type == NRL_TIS_SEQ_MASK ? st.seq_w * st.seq_keep : st.seq_w;
        if (c.sequence_level_importance_ratios && c.tis_type == NRL_TIS_TIS) v = clampf(st.seq_w, c.tis_min, c.tis_max);
        if (c.sequence_level_importance_ratios && c.tis_type == NRL_TIS_ICEPOP) v = (st.seq_w >= c.tis_min && st.seq_w <= c.tis_max) ? st.seq_w : 0.f;
        return v;
    }
    if (k == P_OOB && c.tis_type == NRL_TIS_SEQ_MASK) return (1.f - st.seq_keep) * smv;
    return sum;
}

// Workgroup-wide reduction of one sequence's accumulators (or of a share of them) into a row of partials.
template <int NW>
__device__ __forceinline__ void store_parts(double* out, const double (&acc)[P_R_MIN], float r_min, float r_max, float rc_min,
                                            float rc_max, double* sm_d, float* sm_f) {
    const int tid = threadIdx.x;
    const double tot = block_sums<P_R_MIN, NW>(acc, sm_d);
    const float mn = block_min<NW>(r_min, sm_f), mx = block_max<NW>(r_max, sm_f);
    const float cmn = block_min<NW>(rc_min, sm_f), cmx = block_max<NW>(rc_max, sm_f);
    if (tid < P_R_MIN) out[tid] = tot;
    if (tid == 0) { out[P_R_MIN] = mn; out[P_R_MAX] = mx; out[P_RC_MIN] = cmn; out[P_RC_MAX] = cmx; }
}

template <bool GSPO>
__global__ __launch_bounds__(kSeqBlock) void grpo_rows_kernel(GrpoArgs a) {
    __shared__ double sm_d[kSeqSmem];
    __shared__ float sm_f[kSeqWaves];
    const nrl_grpo_cfg& c = a.cfg;
    const nrl_grpo_inputs& in = a.in;
    const int64_t b = blockIdx.x;
    const int tid = threadIdx.x;
    const int64_t n = in.sm1;

    const float* lp_row = in.lp + b * in.lp_stride;
    const float* lpu_row = in.lpu ? in.lpu + b * in.lpu_stride : lp_row;
    const float* prev_row = c.force_on_policy_ratio ? lp_row : in.prev + b * in.prev_stride;
    const float* gen_row = in.gen + b * in.gen_stride;
    const float* ref_row = c.has_kl ? in.ref + b * in.ref_stride : nullptr;
    const float* adv_row = in.adv + b * in.adv_stride;
    const float smv = in.sample_mask[b];
    const float correct = c.has_nll ? in.correct_mask[b] : 0.f;
    const float den_s = valid_seqs(in) + 1e-8f;
    const float den_t = valid_toks(in) + 1e-8f;

    // ---- row statistics ----
    double s_tm = 0, s_lr = 0, s_is = 0, s_geo = 0;
    for (int64_t t = tid; t < n; t += kSeqBlock) {
        const float tm = mask_at(in, b, t);
        const float prev = prev_row[t], gen = gen_row[t];
        s_tm += tm;
        s_lr += (lp_row[t] - prev) * tm;
        s_is += (prev - gen) * (tm * smv);
        s_geo += finite_or_zero(prev - gen) * tm;
    }
    const float n_tm = static_cast<float>(seq_block_sum(s_tm, sm_d));
    const float seq_den = n_tm + 1e-8f;
    float seq_ratio = 1.f, seq_w = 1.f, seq_keep = 1.f;
    if (GSPO) seq_ratio = expf(static_cast<float>(seq_block_sum(s_lr, sm_d)) / seq_den);
    if (c.sequence_level_importance_ratios)
        seq_w = finite_or_zero(expf(static_cast<float>(seq_block_sum(s_is, sm_d))));
    if (c.tis_type == NRL_TIS_SEQ_MASK) {
        const float geo = expf(static_cast<float>(seq_block_sum(s_geo, sm_d)) / seq_den);
        seq_keep = (geo >= c.tis_min && geo <= c.tis_max) ? 1.f : 0.f;
    }
    double acc[P_R_MIN];
#pragma unroll
    for (int k = 0; k < P_R_MIN; ++k) acc[k] = 0;
    float r_min = INFINITY, r_max = -INFINITY, rc_min = INFINITY, rc_max = -INFINITY;
    double gspo_k = 0;  // sum_t coef * w * d clip / d ratio  (GSPO only)

    SeqStats st;
    st.seq_den = seq_den; st.seq_ratio = seq_ratio; st.seq_w = seq_w; st.seq_keep = seq_keep;
    for (int64_t t = tid; t < n; t += kSeqBlock) {
        TokenIn ti;
        ti.lp = lp_row[t]; ti.lpu = lpu_row[t]; ti.prev = prev_row[t]; ti.gen = gen_row[t];
        ti.ref = c.has_kl ? ref_row[t] : 0.f; ti.adv = adv_row[t]; ti.tm = mask_at(in, b, t); ti.smv = smv; ti.correct = correct;
        ti.den_t = den_t; ti.den_s = den_s;
        const TokenOut o = token_eval<GSPO>(c, st, ti);
#pragma unroll
        for (int k = 0; k < P_SAMPLE_MASK; ++k) acc[k] += o.term[k];
        if (o.selected) {
            r_min = fminf(r_min, o.ratio); r_max = fmaxf(r_max, o.ratio);
            rc_min = fminf(rc_min, o.ratio_cl); rc_max = fmaxf(rc_max, o.ratio_cl);
        }
        const float d_actor = o.d_actor, d_lpu = o.d_lpu;
        if (GSPO) {
            gspo_k += d_actor;
            if (a.dlpu) a.dlpu[b * n + t] = d_lpu;
            else a.dlp[b * n + t] = d_lpu;  // KL share; the ratio share is added below
        } else if (a.dlpu) {
            a.dlp[b * n + t] = d_actor;
            a.dlpu[b * n + t] = d_lpu;
        } else {
            a.dlp[b * n + t] = d_actor + d_lpu;
        }
    }

    if (GSPO) {
        // d ratio_b / d lp[b, s] = ratio_b * tm[b, s] / (n_tm + 1e-8)
        const float k_tot = static_cast<float>(seq_block_sum(gspo_k, sm_d));
        for (int64_t t = tid; t < n; t += kSeqBlock) {
            const float share = k_tot * seq_ratio * (mask_at(in, b, t) / seq_den);
            if (a.dlpu) a.dlp[b * n + t] = share;
            else a.dlp[b * n + t] += share;
        }
    }

    double* out = a.parts + b * P_COUNT;
    store_parts<kSeqWaves>(out, acc, r_min, r_max, rc_min, rc_max, sm_d, sm_f);
    if (tid < P_R_MIN) out[tid] = row_part(c, tid, out[tid], st, smv);  // each thread what it has just stored
}

// Fixed-order reduction of the row partials and normalisation into the metrics record, by one workgroup of kSeqBlock threads.
// A wave takes one quantity at a time and sums it over the rows, so the quantities are reduced side by side (one after the
// other by the whole workgroup took 7 - 10 us, this takes 4 - 7).
__device__ __forceinline__ void finish_metrics(const GrpoArgs& a, float* loss_out, float* metrics, double* tot /* shared [P_COUNT] */) {
    const nrl_grpo_cfg& c = a.cfg;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int64_t nb = a.in.batch;
    const int64_t chunks = a.seq_stats ? a.chunks : 1;
    auto final_part = [&](int k, int64_t b, double sum) {
        if (!a.seq_stats) return sum;
        SeqStats st;
        st.seq_den = a.seq_stats[b * 3]; st.seq_ratio = 1.f; st.seq_w = a.seq_stats[b * 3 + 1]; st.seq_keep = a.seq_stats[b * 3 + 2];
        return row_part(c, k, sum, st, a.in.sample_mask[b]);
    };
    for (int k = tid / kWave; k < P_COUNT; k += kSeqWaves) {
        if (k < P_R_MIN) {
            double v = 0;
            if (chunks <= 8) {  // a lane per sequence
                for (int64_t b = lane; b < nb; b += kWave) {
                    double sum = 0;
                    for (int64_t q = 0; q < chunks; ++q) sum += a.parts[(b * chunks + q) * P_COUNT + k];
                    v += final_part(k, b, sum);
                }
                v = wave_sum_double(v);
            } else {  // long sequences, so a microbatch holds few of them: the wave over the shares of one after the other
                for (int64_t b = 0; b < nb; ++b) {
                    double sum = 0;
                    for (int64_t q = lane; q < chunks; q += kWave) sum += a.parts[(b * chunks + q) * P_COUNT + k];
                    v += final_part(k, b, wave_sum_double(sum));
                }
            }
            if (lane == 0) tot[k] = v;
        } else {
            const bool low = k == P_R_MIN || k == P_RC_MIN;
            float v = low ? INFINITY : -INFINITY;
            for (int64_t b = lane; b < nb * chunks; b += kWave) {
                const float p = static_cast<float>(a.parts[b * P_COUNT + k]);
                v = low ? fminf(v, p) : fmaxf(v, p);
            }
            v = low ? wave_min(v) : wave_max(v);
            if (lane == 0) tot[k] = v;
        }
    }
    __syncthreads();
    if (tid != 0) return;
    const float r_min = static_cast<float>(tot[P_R_MIN]), r_max = static_cast<float>(tot[P_R_MAX]);
    const float rc_min = static_cast<float>(tot[P_RC_MIN]), rc_max = static_cast<float>(tot[P_RC_MAX]);

    const double den_s = valid_seqs(a.in) + 1e-8f, den_t = valid_toks(a.in) + 1e-8f;
    const double den_loss = c.token_level_loss ? den_t : den_s;
    const float actor = static_cast<float>(tot[P_ACTOR] / den_loss);
    const float kl = c.has_kl ? static_cast<float>(tot[P_KL] / den_loss) : 0.f;
    float nll = 0.f;
    if (c.has_nll && tot[P_N_CORRECT] > 0) nll = static_cast<float>(tot[P_NLL] / (static_cast<float>(tot[P_N_CORRECT]) + 1e-8f));
    const float loss = (actor + kl) + c.nll_weight * nll;
    loss_out[0] = loss;
    for (int k = 0; k < NRL_GRPO_N_METRICS; ++k) metrics[k] = 0.f;
    metrics[NRL_M_LOSS] = loss;
    metrics[NRL_M_ACTOR_LOSS] = actor;
    metrics[NRL_M_KL] = kl;
    metrics[NRL_M_PROBS_RATIO] = static_cast<float>(tot[P_RATIO] / den_t);
    metrics[NRL_M_PROBS_RATIO_CLAMPED] = static_cast<float>(tot[P_RATIO_CL] / den_t);
    metrics[NRL_M_PROBS_RATIO_MIN] = r_min;
    metrics[NRL_M_PROBS_RATIO_MAX] = r_max;
    metrics[NRL_M_PROBS_RATIO_CLAMPED_MIN] = rc_min;
    metrics[NRL_M_PROBS_RATIO_CLAMPED_MAX] = rc_max;
    metrics[NRL_M_TOKEN_MULT_PROB_ERROR] = static_cast<float>(tot[P_MULT_ERR] / den_t);
    metrics[NRL_M_GEN_KL_ERROR] = static_cast<float>(tot[P_GEN_KL] / den_t);
    metrics[NRL_M_POLICY_KL_ERROR] = static_cast<float>(tot[P_POLICY_KL] / den_t);
    metrics[NRL_M_JS_DIVERGENCE_ERROR] = static_cast<float>(tot[P_JS] / den_t);
    // sequence-level weights: the reference multiplies a [B,1] weight by a [B] mask, which
    // broadcasts to [B,B]; the sum is (sum of weights) * (sum of sample_mask)
    metrics[NRL_M_SAMPLING_IMPORTANCE_RATIO] =
        c.sequence_level_importance_ratios ? static_cast<float>(tot[P_SEQ_W] * tot[P_SAMPLE_MASK] / den_s)
                                           : static_cast<float>(tot[P_SAMPLING] / den_t);
    metrics[NRL_M_NUM_VALID_SAMPLES] = static_cast<float>(tot[P_SAMPLE_MASK]);
    metrics[NRL_M_APPROX_ENTROPY] = -static_cast<float>(tot[P_ENTROPY] / den_t);
    metrics[NRL_M_IS_OOB_RATIO] = static_cast<float>(tot[P_OOB] / (c.tis_type == NRL_TIS_SEQ_MASK ? den_s : den_t));
    metrics[NRL_M_POSITIVE_NLL_LOSS] = nll;
    metrics[NRL_M_N_MASKED_TOKENS] = static_cast<float>(tot[P_N_SELECTED]);
}

__global__ __launch_bounds__(kSeqBlock) void grpo_finish_kernel(GrpoArgs a, float* loss_out, float* metrics) {
    __shared__ double tot[P_COUNT];
    finish_metrics(a, loss_out, metrics, tot);
}

// positive-example NLL: d loss / d lp += -weight * mask * correct / (n_correct + 1e-8)
__global__ void grpo_nll_grad_kernel(GrpoArgs a) {
    const int64_t n = a.in.sm1, total = a.in.batch * n;
    double n_correct = 0;
    for (int64_t b = 0; b < a.in.batch; ++b) n_correct += a.parts[b * P_COUNT + P_N_CORRECT];
    if (!(n_correct > 0)) return;
    const float den = static_cast<float>(n_correct) + 1e-8f;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t b = i / n, t = i - b * n;
        const float cm = mask_at(a.in, b, t) * a.in.sample_mask[b] * a.in.correct_mask[b];
        a.dlp[i] += a.cfg.nll_weight * (-(cm / den));
    }
}

// NLLLossFn: one workgroup per row for the partial sums, then the same finish pattern
__global__ __launch_bounds__(kLossBlock) void nll_rows_kernel(nrl_grpo_inputs in, float* dlp, double* parts) {
    __shared__ double sm_d[kLossWaves];
    const int64_t b = blockIdx.x, n = in.sm1;
    const float smv = in.sample_mask[b];
    const float den_t = valid_toks(in) + 1e-8f;
    double s = 0, cnt = 0;
    for (int64_t t = threadIdx.x; t < n; t += kLossBlock) {
        const float mask = mask_at(in, b, t) * smv;
        s += in.lp[b * in.lp_stride + t] * mask;
        cnt += mask;
        dlp[b * n + t] = -(mask / den_t);
    }
    s = block_sum<double, kLossWaves>(s, sm_d);
    cnt = block_sum<double, kLossWaves>(cnt, sm_d);
    if (threadIdx.x == 0) { parts[b * 3] = s; parts[b * 3 + 1] = cnt; parts[b * 3 + 2] = smv; }
}

__global__ __launch_bounds__(kLossBlock) void nll_finish_kernel(nrl_grpo_inputs in, const double* parts, float* loss_out,
                                                               float* metrics) {
    __shared__ double sm_d[kLossWaves];
    double s = 0, cnt = 0, smv = 0;
    for (int64_t b = threadIdx.x; b < in.batch; b += kLossBlock) { s += parts[b * 3]; cnt += parts[b * 3 + 1]; smv += parts[b * 3 + 2]; }
    s = block_sum<double, kLossWaves>(s, sm_d);
    cnt = block_sum<double, kLossWaves>(cnt, sm_d);
    smv = block_sum<double, kLossWaves>(smv, sm_d);
    if (threadIdx.x == 0) {
        const double den_t = valid_toks(in) + 1e-8f;
        const float loss = -static_cast<float>(s / den_t);
        loss_out[0] = loss;
        metrics[0] = loss; metrics[1] = static_cast<float>(cnt); metrics[2] = static_cast<float>(smv);
    }
}

// ---------------------------------------------------------------------------------------------
// The single pass (fused_rows.hpp): what runs ahead of it and behind it.
// ---------------------------------------------------------------------------------------------
// where a logits row sits in the loss inputs: sequence o, position i (i >= n_inner: the row feeds no token),
// and the index of its target id
struct FusedPos {
    int64_t o, i, tgt;
};
__device__ __forceinline__ FusedPos fused_where_packed(const FusedArgs& a, int64_t r, int64_t total) {
    FusedPos q;
    const int64_t seq = find_seq(a.cu, a.n_seq, r);
    q.o = seq < 0 ? 0 : seq;
    q.i = -1;
    q.tgt = 0;
    if (seq >= 0) {
        const int64_t start = a.cu[seq], len = a.cu[seq + 1] - start, pos = r - start;
        if (pos + 1 < len && pos < a.n_inner) q.i = pos;  // the last position of a sequence predicts nothing
        q.tgt = start + (a.pre_rolled ? pos : (pos + 1 < len ? pos + 1 : 0));
        // (the targets hold at least `total` entries; boundaries that run past the packed row cannot index beyond them)
        if (q.tgt >= total) q.tgt = total - 1;
    }
    return q;
}
template <int DT> __device__ __forceinline__ float fused_target_logit(const FusedArgs& a, const char* row, int64_t i, int temp) {
    const float x = Row<DT>::load1(row, i);
    return temp == 0 ? x : temp == 1 ? scale_logit<DT, 1>(x, a.tparam) : scale_logit<DT, 2>(x, a.tparam);
}

// Everything the pass needs beforehand, in one launch.  The first `batch` workgroups compute the per-sequence statistics, the
// others zero the logprobs (masked tokens and positions without a row keep that) and gather a record per row: where the row
// sits in the loss inputs (in packed mode a search through the boundaries, a chain of dependent loads), the inputs, and its
// target's logit.  (7 packed sequences, 16384 tokens: 10 us; statistics, two fills and row positions as launches of their own 33 us.)
__global__ __launch_bounds__(kSeqBlock) void fused_prep_kernel(FusedArgs a, int64_t n_rows, int dtype, int temp) {
    __shared__ double sm_d[kSeqWaves];
    const nrl_grpo_cfg& c = a.cfg;
    const nrl_grpo_inputs& in = a.in;
    const int64_t b = blockIdx.x, n = in.sm1;
    if (b >= in.batch) {
        const int64_t first = (b - in.batch) * kSeqBlock + threadIdx.x, step = (gridDim.x - in.batch) * kSeqBlock;
        for (int64_t i = first; i < in.batch * n; i += step) a.lp_out[i] = 0.f;
        for (int64_t r = first; r < n_rows; r += step) {
            if (a.row_grad) a.row_grad[r] = make_float4(0.f, 0.f, 0.f, 0.f);
            FusedPos q;
            int64_t off;
            if (a.cu) {
                q = fused_where_packed(a, r, n_rows);
                off = r * a.stride_inner;
            } else {
                q.o = r / a.d_n_inner;
                q.i = r - q.o * a.d_n_inner;
                off = q.o * a.stride_outer + q.i * a.stride_inner;
                if (q.i >= n) continue;  // feeds no token: no record
                q.tgt = q.o * a.ts_outer + q.i * a.ts_inner;
            }
            uint32_t w[R_WORDS];
#pragma unroll
            for (int k = 0; k < R_WORDS; ++k) w[k] = 0u;
            const int64_t o = q.o, i = q.i;
            const float tm = i >= 0 ? mask_at(in, o, i) : 0.f, smv = i >= 0 ? in.sample_mask[o] : 0.f;
            if (tm * smv != 0.f) {
                w[R_LIVE] = 1u;
                if (!c.force_on_policy_ratio) w[R_PREV] = __float_as_uint(in.prev[o * in.prev_stride + i]);
                w[R_GEN] = __float_as_uint(in.gen[o * in.gen_stride + i]);
                if (c.has_kl) w[R_REF] = __float_as_uint(in.ref[o * in.ref_stride + i]);
                w[R_ADV] = __float_as_uint(in.adv[o * in.adv_stride + i]);
                w[R_TM] = __float_as_uint(tm);
                w[R_SMV] = __float_as_uint(smv);
                const int64_t tg = a.targets[q.tgt];
                const bool local = tg >= a.vstart && tg < a.vend;
                w[R_TLOC] = local ? static_cast<uint32_t>(tg - a.vstart) : 0xffffffffu;
                if (local) {
                    const char* row = static_cast<const char*>(a.logits) + off * (dtype == NRL_F32 ? 4 : 2);
                    const float x = dtype == NRL_F32 ? fused_target_logit<NRL_F32>(a, row, tg - a.vstart, temp)
                                    : dtype == NRL_BF16 ? fused_target_logit<NRL_BF16>(a, row, tg - a.vstart, temp)
                                                        : fused_target_logit<NRL_F16>(a, row, tg - a.vstart, temp);
                    w[R_XT] = __float_as_uint(x);
                }
                w[R_SEQ] = static_cast<uint32_t>(o);
                w[R_POS] = static_cast<uint32_t>(i);
            }
            u32x4* out = reinterpret_cast<u32x4*>(a.rec + (a.cu ? r : o * n + i) * R_WORDS);
#pragma unroll
            for (int k = 0; k < R_WORDS / 4; ++k) out[k] = u32x4{w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]};
        }
        return;
    }
    const float smv = in.sample_mask[b];
    double s_tm = 0, s_is = 0, s_geo = 0;
    const bool need_prev = c.sequence_level_importance_ratios || c.tis_type == NRL_TIS_SEQ_MASK;
    for (int64_t t = threadIdx.x; t < n; t += kSeqBlock) {
        const float tm = mask_at(in, b, t);
        s_tm += tm;
        if (need_prev) {
            const float d = in.prev[b * in.prev_stride + t] - in.gen[b * in.gen_stride + t];
            s_is += d * (tm * smv);
            s_geo += finite_or_zero(d) * tm;
        }
    }
    const float seq_den = static_cast<float>(seq_block_sum(s_tm, sm_d)) + 1e-8f;
    float seq_w = 1.f, seq_keep = 1.f;
    if (c.sequence_level_importance_ratios) seq_w = finite_or_zero(expf(static_cast<float>(seq_block_sum(s_is, sm_d))));
    if (c.tis_type == NRL_TIS_SEQ_MASK) {
        const float geo = expf(static_cast<float>(seq_block_sum(s_geo, sm_d)) / seq_den);
        seq_keep = (geo >= c.tis_min && geo <= c.tis_max) ? 1.f : 0.f;
    }
    if (threadIdx.x == 0) {
        a.seq_stats[b * 3] = seq_den;
        a.seq_stats[b * 3 + 1] = seq_w;
        a.seq_stats[b * 3 + 2] = seq_keep;
    }
}

// Logprobs -> the terms of the loss and the metrics, summed over shares of kTermsBlock tokens, one workgroup each and a token
// per thread.  A sequence per workgroup is bound by the chain of one compute unit, 23 us for 7 packed sequences (16384
// tokens); spread out 6 us, 4 sequences of 1024 tokens 9.6 -> 5.7 us.  The shares are added up, in order, by the
// launch that finishes the metrics: done here by the workgroup that arrives last, the device-scope fence in front of its
// arrival waits for the L2 to write back what the pass left there, 13 - 25 us.
constexpr int kTermsBlock = 256, kTermsWaves = kTermsBlock / kWave;
__global__ __launch_bounds__(kTermsBlock) void grpo_terms_reduce_kernel(FusedArgs a, int64_t chunks, int64_t n_rows) {
    __shared__ double sm_d[kTermsWaves * P_R_MIN];
    __shared__ float sm_f[kTermsWaves];
    const nrl_grpo_cfg& c = a.cfg;
    const nrl_grpo_inputs& in = a.in;
    const int64_t b = blockIdx.x / chunks, q = blockIdx.x - b * chunks, t = q * kTermsBlock + threadIdx.x;
    double acc[P_R_MIN];
#pragma unroll
    for (int k = 0; k < P_R_MIN; ++k) acc[k] = 0;
    float r_min = INFINITY, r_max = -INFINITY, rc_min = INFINITY, rc_max = -INFINITY;
    bool live = t < a.n_inner;
    // Packed sequences may hold fewer rows than the loss inputs have columns.  On any_row rows a token of the mask beyond its
    // sequence's rows counts with a logprob of 0 (what lp_out holds there), as the unpacked logprobs of the general path
    // make it count; on aligned rows it does not count.
    if (live && a.cu && !a.any_row) {
        const int64_t start = a.cu[b], len = a.cu[b + 1] - start;
        live = t + 1 < len && start + t >= 0 && start + t < n_rows;
    }
    const float tm = live ? mask_at(in, b, t) : 0.f, smv = in.sample_mask[b];
    if (tm * smv != 0.f) {
        const float lp = a.lp_out[b * a.n_inner + t];
        SeqStats st;
        st.seq_den = a.seq_stats[b * 3]; st.seq_ratio = 1.f; st.seq_w = a.seq_stats[b * 3 + 1]; st.seq_keep = a.seq_stats[b * 3 + 2];
        TokenIn ti;
        ti.lp = lp; ti.lpu = lp;
        ti.prev = c.force_on_policy_ratio ? lp : in.prev[b * in.prev_stride + t];
        ti.gen = in.gen[b * in.gen_stride + t];
        ti.ref = c.has_kl ? in.ref[b * in.ref_stride + t] : 0.f;
        ti.adv = in.adv[b * in.adv_stride + t];
        ti.tm = tm; ti.smv = smv; ti.correct = 0.f;
        ti.den_s = valid_seqs(in) + 1e-8f;
        ti.den_t = valid_toks(in) + 1e-8f;
        const TokenOut out = token_eval<false>(c, st, ti);
#pragma unroll
        for (int k = 0; k < P_SAMPLE_MASK; ++k) acc[k] = out.term[k];
        if (out.selected) { r_min = r_max = out.ratio; rc_min = rc_max = out.ratio_cl; }
    }
    store_parts<kTermsWaves>(a.parts + blockIdx.x * static_cast<int64_t>(P_COUNT), acc, r_min, r_max, rc_min, rc_max, sm_d, sm_f);
}

static int check_inputs(const nrl_grpo_inputs* in, bool need_prev, bool need_ref, bool need_adv) {
    if (!in) return fail(NRL_E_INVALID, "inputs is NULL");
    if (in->token_mask_type < NRL_MASK_F32 || in->token_mask_type > NRL_MASK_U8) return fail(NRL_E_INVALID, "unknown token mask type");
    if (in->batch < 0 || in->sm1 < 0) return fail(NRL_E_INVALID, "bad shape [%lld, %lld]", (long long)in->batch, (long long)in->sm1);
    if (in->batch >= (1ll << 31)) return fail(NRL_E_INVALID, "batch too large");
    if (in->batch * in->sm1 == 0) return NRL_OK;
    if (!in->lp || !in->token_mask || !in->sample_mask || !in->global_valid) return fail(NRL_E_INVALID, "null lp, token_mask, sample_mask or global_valid");
    if (need_adv && (!in->gen || !in->adv)) return fail(NRL_E_INVALID, "null generation_logprobs or advantages");
    if (need_prev && !in->prev) return fail(NRL_E_INVALID, "prev_logprobs is NULL");
    if (need_ref && !in->ref) return fail(NRL_E_INVALID, "reference_policy_logprobs is NULL");
    return NRL_OK;
}

}  // namespace nrl

using namespace nrl;

extern "C" int64_t nrl_grpo_loss_workspace_bytes(int64_t batch) {
    return (batch < 1 ? 1 : batch) * P_COUNT * static_cast<int64_t>(sizeof(double));
}

static int grpo_loss_impl(const nrl_grpo_cfg* cfg, const nrl_grpo_inputs* in, float* loss_out, float* dlp_out, float* dlpu_out,
                          float* metrics_out, double* parts, void* stream, const char* what) {
    const bool split = in->lpu != nullptr && cfg->has_kl;
    GrpoArgs a;
    a.cfg = *cfg;
    a.in = *in;
    if (!cfg->has_kl) a.in.lpu = nullptr;
    a.dlp = dlp_out;
    a.dlpu = split ? dlpu_out : nullptr;
    a.parts = parts;
    a.seq_stats = nullptr; a.chunks = 1;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (in->batch > 0) {
        const bool gspo = cfg->sequence_level_importance_ratios && !cfg->disable_ppo_ratio && !cfg->force_on_policy_ratio;
        if (gspo) grpo_rows_kernel<true><<<dim3((unsigned)in->batch), dim3(kSeqBlock), 0, s>>>(a);
        else grpo_rows_kernel<false><<<dim3((unsigned)in->batch), dim3(kSeqBlock), 0, s>>>(a);
    }
    grpo_finish_kernel<<<dim3(1), dim3(kSeqBlock), 0, s>>>(a, loss_out, metrics_out);
    if (cfg->has_nll && in->batch * in->sm1 > 0) {
        const int64_t total = in->batch * in->sm1;
        const unsigned blocks = (unsigned)((total + 255) / 256 > 1024 ? 1024 : (total + 255) / 256);
        grpo_nll_grad_kernel<<<dim3(blocks), dim3(256), 0, s>>>(a);
    }
    return check_launch(what);
}

// argument checks shared by the two loss entry points (everything except the workspace)
static int grpo_loss_check(const nrl_grpo_cfg* cfg, const nrl_grpo_inputs* in, const float* loss_out, const float* dlp_out,
                           const float* dlpu_out, const float* metrics_out) {
    if (!cfg) return fail(NRL_E_INVALID, "cfg is NULL");
    if (int e = check_inputs(in, !cfg->force_on_policy_ratio, cfg->has_kl != 0, true)) return e;
    if (cfg->kl_type < 1 || cfg->kl_type > 3) return fail(NRL_E_INVALID, "kl_type must be 1, 2 or 3");
    if (cfg->tis_type < 0 || cfg->tis_type > 3) return fail(NRL_E_INVALID, "bad tis_type");
    if (cfg->sequence_level_importance_ratios && cfg->token_level_loss)
        return fail(NRL_E_INVALID, "sequence-level importance ratios need a sequence-level loss");
    if (cfg->has_nll && !in->correct_mask) return fail(NRL_E_INVALID, "correct_mask is NULL");
    if (!loss_out || !metrics_out) return fail(NRL_E_INVALID, "null output");
    const bool split = in->lpu != nullptr && cfg->has_kl;
    if (in->batch * in->sm1 > 0 && (!dlp_out || (split && !dlpu_out))) return fail(NRL_E_INVALID, "null gradient output");
    return NRL_OK;
}

extern "C" int nrl_grpo_loss_fwd_bwd(const nrl_grpo_cfg* cfg, const nrl_grpo_inputs* in, float* loss_out, float* dlp_out,
                                     float* dlpu_out, float* metrics_out, void* workspace, int64_t workspace_bytes,
                                     void* stream) {
    if (int e = grpo_loss_check(cfg, in, loss_out, dlp_out, dlpu_out, metrics_out)) return e;
    if (!workspace) return fail(NRL_E_INVALID, "null workspace");
    if (workspace_bytes < nrl_grpo_loss_workspace_bytes(in->batch)) return fail(NRL_E_WORKSPACE, "workspace too small");
    if (reinterpret_cast<uintptr_t>(workspace) & 7) return fail(NRL_E_INVALID, "workspace must be 8-byte aligned");
    return grpo_loss_impl(cfg, in, loss_out, dlp_out, dlpu_out, metrics_out, static_cast<double*>(workspace), stream,
                          "grpo_loss_fwd_bwd");
}

// ---------------------------------------------------------------------------------------------
// The same loss for callers that cannot allocate: the per-sequence partial sums live in a fixed
// device array instead of a caller workspace.  Every GPU holds its own copy of the array at its own
// address; the name `scratch` is only a host-side handle, the address comes from hipGetSymbolAddress
// once per device and is what the kernels receive.
// ---------------------------------------------------------------------------------------------
namespace nrl {
constexpr int64_t kStaticMaxBatch = NRL_GRPO_STATIC_MAX_BATCH;
constexpr int kStaticMaxDevices = 64;
static __device__ __align__(256) double scratch[kStaticMaxBatch * P_COUNT];  // 1.25 MiB per GPU
static std::mutex scratch_mutex;
static double* scratch_ptr[kStaticMaxDevices] = {nullptr};

// device address of this GPU's `scratch`, resolved on the first call with that GPU current
static int scratch_for_current_device(double** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(NRL_E_LAUNCH, "hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kStaticMaxDevices) return fail(NRL_E_UNSUPPORTED, "device index %d beyond %d", dev, kStaticMaxDevices);
    std::lock_guard<std::mutex> lock(scratch_mutex);
    if (!scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return fail(NRL_E_LAUNCH, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        scratch_ptr[dev] = static_cast<double*>(p);
    }
    *out = scratch_ptr[dev];
    return NRL_OK;
}
}  // namespace nrl

extern "C" int nrl_grpo_loss_fwd_bwd_static(const nrl_grpo_cfg* cfg, const nrl_grpo_inputs* in, float* loss_out,
                                            float* dlp_out, float* dlpu_out, float* metrics_out, void* stream) {
    if (int e = grpo_loss_check(cfg, in, loss_out, dlp_out, dlpu_out, metrics_out)) return e;
    if (in->batch > kStaticMaxBatch)
        return fail(NRL_E_WORKSPACE, "batch %lld exceeds the %lld sequences the static scratch holds; use nrl_grpo_loss_fwd_bwd",
                    (long long)in->batch, (long long)kStaticMaxBatch);
    double* parts = nullptr;
    if (int e = scratch_for_current_device(&parts)) return e;
    // rows 0 .. batch-1 of the scratch are rewritten in full by the first launch before the second reads
    // them, and nothing beyond `batch` rows is read, so a previous call's contents need no clearing
    return grpo_loss_impl(cfg, in, loss_out, dlp_out, dlpu_out, metrics_out, parts, stream, "grpo_loss_fwd_bwd_static");
}

extern "C" int nrl_nll_loss_fwd_bwd(const nrl_grpo_inputs* in, float* loss_out, float* dlp_out, float* metrics_out,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
    if (int e = check_inputs(in, false, false, false)) return e;
    if (!loss_out || !metrics_out || !workspace) return fail(NRL_E_INVALID, "null output or workspace");
    if (workspace_bytes < nrl_grpo_loss_workspace_bytes(in->batch)) return fail(NRL_E_WORKSPACE, "workspace too small");
    if (in->batch * in->sm1 > 0 && !dlp_out) return fail(NRL_E_INVALID, "null gradient output");
    hipStream_t s = static_cast<hipStream_t>(stream);
    double* parts = static_cast<double*>(workspace);
    if (in->batch > 0) nll_rows_kernel<<<dim3((unsigned)in->batch), dim3(kLossBlock), 0, s>>>(*in, dlp_out, parts);
    nll_finish_kernel<<<dim3(1), dim3(kLossBlock), 0, s>>>(*in, parts, loss_out, metrics_out);
    return check_launch("nll_loss_fwd_bwd");
}

// ---------------------------------------------------------------------------------------------
// The two helpers of the loss that the driver also calls on their own (KL in the reward, mean reward):
// calculate_kl element by element, masked_mean row by row.  [B, S]-sized, latency bound.
// ---------------------------------------------------------------------------------------------
struct KlArgs {
    const float* lp;
    const float* ref;
    const float* weight;  // importance sampling weights or NULL
    int64_t n;
    int kl_type, has_in, has_out;
    float in_clamp, out_clamp;
};

struct KlPoint {
    float value, d_logr, d_weight;  // clamped value; d value / d (ref - lp); d value / d weight
};

__device__ __forceinline__ KlPoint kl_point(const KlArgs& a, int64_t i) {
    float logr = a.ref[i] - a.lp[i];
    float in_range = 1.f;
    if (a.has_in) {
        const float cl = clampf(logr, -a.in_clamp, a.in_clamp);
        if (!(logr == cl)) in_range = 0.f;  // a clamped token passes no gradient, neither through the KL nor the weight
        logr = cl;
    }
    const float w = a.weight ? a.weight[i] : 1.f;
    const float k = kl_value(a.kl_type, logr);
    KlPoint o;
    o.value = a.weight ? w * k : k;
    o.d_logr = w * kl_slope(a.kl_type, logr) * in_range;
    o.d_weight = k * in_range;
    if (a.has_out) {
        if (!(o.value >= -a.out_clamp && o.value <= a.out_clamp)) { o.d_logr = 0.f; o.d_weight = 0.f; }
        o.value = clampf(o.value, -a.out_clamp, a.out_clamp);
    }
    return o;
}

__global__ __launch_bounds__(256) void calculate_kl_kernel(KlArgs a, float* out) {
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < a.n; i += gridDim.x * 256ll) out[i] = kl_point(a, i).value;
}

__global__ __launch_bounds__(256) void calculate_kl_bwd_kernel(KlArgs a, const float* g, float* d_lp, float* d_ref, float* d_weight) {
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < a.n; i += gridDim.x * 256ll) {
        const KlPoint p = kl_point(a, i);
        const float t = g[i] * p.d_logr;
        if (d_lp) d_lp[i] = -t;
        if (d_ref) d_ref[i] = t;
        if (d_weight) d_weight[i] = g[i] * p.d_weight;
    }
}

static int kl_args(KlArgs& a, const float* lp, const float* ref, const float* weight, int64_t n, int32_t kl_type,
                   int32_t has_in, float in_clamp, int32_t has_out, float out_clamp) {
    if (n < 0 || (n > 0 && (!lp || !ref))) return fail(NRL_E_INVALID, "calculate_kl: null input");
    if (kl_type < 1 || kl_type > 3) return fail(NRL_E_INVALID, "calculate_kl: kl_type must be 1 (k1), 2 (k2) or 3 (k3)");
    a = KlArgs{lp, ref, weight, n, kl_type, has_in, has_out, in_clamp, out_clamp};
    return NRL_OK;
}

static unsigned small_grid(int64_t n) { return static_cast<unsigned>(n + 255 < 256 * 2048ll ? (n + 255) / 256 : 2048); }

extern "C" int nrl_calculate_kl(const float* logprobs, const float* logprobs_reference, const float* weights, int64_t n,
                                int32_t kl_type, int32_t has_input_clamp, float input_clamp, int32_t has_output_clamp,
                                float output_clamp, float* kl_out, void* stream) {
    KlArgs a;
    if (int e = kl_args(a, logprobs, logprobs_reference, weights, n, kl_type, has_input_clamp, input_clamp,
                        has_output_clamp, output_clamp)) return e;
    if (n == 0) return NRL_OK;
    if (!kl_out) return fail(NRL_E_INVALID, "calculate_kl: null output");
    calculate_kl_kernel<<<dim3(small_grid(n)), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(a, kl_out);
    return check_launch("calculate_kl");
}

extern "C" int nrl_calculate_kl_bwd(const float* grad_kl, const float* logprobs, const float* logprobs_reference,
                                    const float* weights, int64_t n, int32_t kl_type, int32_t has_input_clamp,
                                    float input_clamp, int32_t has_output_clamp, float output_clamp, float* dlogprobs_out,
                                    float* dreference_out, float* dweights_out, void* stream) {
    KlArgs a;
    if (int e = kl_args(a, logprobs, logprobs_reference, weights, n, kl_type, has_input_clamp, input_clamp,
                        has_output_clamp, output_clamp)) return e;
    if (n == 0) return NRL_OK;
    if (!grad_kl) return fail(NRL_E_INVALID, "calculate_kl_bwd: null upstream gradient");
    if (dweights_out && !weights) return fail(NRL_E_INVALID, "calculate_kl_bwd: a weight gradient without weights");
    calculate_kl_bwd_kernel<<<dim3(small_grid(n)), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(
        a, grad_kl, dlogprobs_out, dreference_out, dweights_out);
    return check_launch("calculate_kl_bwd");
}

// one workgroup per row: out[r] = sum_c(values * mask) / (norm + 1e-8), norm = sum_c(mask) unless given
__global__ __launch_bounds__(kLossBlock) void masked_mean_kernel(const float* values, const float* mask, int64_t n_cols,
                                                                 const float* norm_dev, float norm_host, int has_norm,
                                                                 float* out, float* denom_out) {
    __shared__ double red[kLossBlock / kWave];
    const int64_t r = blockIdx.x;
    double sv = 0.0, sm = 0.0;
    for (int64_t c = threadIdx.x; c < n_cols; c += kLossBlock) {
        const float m = mask[r * n_cols + c];
        sv += static_cast<double>(values[r * n_cols + c] * m);
        sm += static_cast<double>(m);
    }
    sv = block_sum<double, kLossBlock / kWave>(sv, red);
    __syncthreads();
    sm = block_sum<double, kLossBlock / kWave>(sm, red);
    if (threadIdx.x == 0) {
        const float norm = has_norm ? (norm_dev ? norm_dev[0] : norm_host) : static_cast<float>(sm);
        const float den = norm + 1e-8f;
        out[r] = static_cast<float>(sv) / den;
        if (denom_out) denom_out[r] = den;
    }
}

__global__ __launch_bounds__(256) void masked_mean_bwd_kernel(const float* g, const float* mask, const float* denom,
                                                              int64_t n_rows, int64_t n_cols, float* d_values) {
    const int64_t n = n_rows * n_cols;
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += gridDim.x * 256ll) {
        const int64_t r = i / n_cols;
        d_values[i] = g[r] * mask[i] / denom[r];
    }
}

extern "C" int nrl_masked_mean(const float* values, const float* mask, int64_t n_rows, int64_t n_cols,
                               const float* norm_device, float norm_host, int32_t has_norm, float* out, float* denom_out,
                               void* stream) {
    if (n_rows < 0 || n_cols < 0) return fail(NRL_E_INVALID, "masked_mean: negative shape");
    if (n_rows == 0) return NRL_OK;
    if (!out || (n_cols > 0 && (!values || !mask))) return fail(NRL_E_INVALID, "masked_mean: null pointer");
    if (n_rows > 0x7fffffffll) return fail(NRL_E_UNSUPPORTED, "masked_mean: more than 2^31 - 1 rows");
    masked_mean_kernel<<<dim3((unsigned)n_rows), dim3(kLossBlock), 0, static_cast<hipStream_t>(stream)>>>(
        values, mask, n_cols, norm_device, norm_host, has_norm, out, denom_out);
    return check_launch("masked_mean");
}

extern "C" int nrl_masked_mean_bwd(const float* grad_out, const float* mask, const float* denom, int64_t n_rows,
                                   int64_t n_cols, float* dvalues_out, void* stream) {
    if (n_rows < 0 || n_cols < 0) return fail(NRL_E_INVALID, "masked_mean_bwd: negative shape");
    if (n_rows * n_cols == 0) return NRL_OK;
    if (!grad_out || !mask || !denom || !dvalues_out) return fail(NRL_E_INVALID, "masked_mean_bwd: null pointer");
    masked_mean_bwd_kernel<<<dim3(small_grid(n_rows * n_cols)), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(
        grad_out, mask, denom, n_rows, n_cols, dvalues_out);
    return check_launch("masked_mean_bwd");
}

// ---------------------------------------------------------------------------------------------
// Positions that are masked out or whose logprob is infinite become 0, with the two counts of the caller's warning, in one
// launch.  The arrays are [B, S]-sized, so what costs is the number of launches: as tensor operations this was 14 of them
// forward and 3 backward, 110 of the 657 us that a filtered microbatch of 2 x 2048 tokens of V = 151936 bf16 took (569 us
// as one kernel each way).  One workgroup per sequence, so the counts need no cleared memory and no atomics.
// ---------------------------------------------------------------------------------------------
struct NegInfArgs {
    const float* lp;
    int64_t lp_stride;
    const void* mask;  // NRL_MASK_* elements
    int mask_type;
    int64_t mask_stride;
    const float* sample_mask;  // [B] or NULL
    int64_t n;
    float* out;        // [B, n]
    uint8_t* keep;     // [B, n]
    double* counts;    // [B, 2]: infinite under the mask, sum of the mask
};
constexpr int kNegInfBlock = 1024;

__global__ __launch_bounds__(kNegInfBlock) void mask_neg_inf_kernel(NegInfArgs a) {
    __shared__ double red[kNegInfBlock / kWave];
    nrl_grpo_inputs in;
    in.token_mask = a.mask; in.token_mask_type = a.mask_type; in.token_mask_stride = a.mask_stride;
    const int64_t b = blockIdx.x;
    const float smv = a.sample_mask ? a.sample_mask[b] : 1.f;
    double hit = 0, total = 0;
    for (int64_t t = threadIdx.x; t < a.n; t += kNegInfBlock) {
        const float x = a.lp[b * a.lp_stride + t];
        const float m = mask_at(in, b, t) * smv;
        const bool inf = fabsf(x) == INFINITY;
        const bool keep = m * (inf ? 0.f : 1.f) != 0.f;
        hit += inf && m != 0.f ? 1.0 : 0.0;
        total += m;
        a.out[b * a.n + t] = keep ? x : 0.f;
        a.keep[b * a.n + t] = keep;
    }
    hit = block_sum<double, kNegInfBlock / kWave>(hit, red);
    total = block_sum<double, kNegInfBlock / kWave>(total, red);
    if (threadIdx.x == 0) { a.counts[2 * b] = hit; a.counts[2 * b + 1] = total; }
}

__global__ __launch_bounds__(256) void mask_neg_inf_bwd_kernel(const float* g, const uint8_t* keep, int64_t n, float* d) {
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += gridDim.x * 256ll) d[i] = keep[i] ? g[i] : 0.f;
}

extern "C" int nrl_mask_neg_inf(const float* logprobs, int64_t lp_stride, const void* mask, int32_t mask_type, int64_t mask_stride,
                                const float* sample_mask, int64_t batch, int64_t n, float* out, uint8_t* keep_out,
                                double* counts_out, void* stream) {
    if (batch < 0 || n < 0) return fail(NRL_E_INVALID, "mask_neg_inf: negative shape");
    if (mask_type < NRL_MASK_F32 || mask_type > NRL_MASK_U8) return fail(NRL_E_INVALID, "mask_neg_inf: unknown mask type");
    if (batch == 0) return NRL_OK;
    if (!counts_out || (n > 0 && (!logprobs || !mask || !out || !keep_out))) return fail(NRL_E_INVALID, "mask_neg_inf: null pointer");
    if (batch > 0x7fffffffll) return fail(NRL_E_UNSUPPORTED, "mask_neg_inf: more than 2^31 - 1 rows");
    const NegInfArgs a{logprobs, lp_stride, mask, mask_type, mask_stride, sample_mask, n, out, keep_out, counts_out};
    mask_neg_inf_kernel<<<dim3((unsigned)batch), dim3(kNegInfBlock), 0, static_cast<hipStream_t>(stream)>>>(a);
    return check_launch("mask_neg_inf");
}

extern "C" int nrl_mask_neg_inf_bwd(const float* grad_out, const uint8_t* keep, int64_t n, float* grad_in, void* stream) {
    if (n < 0) return fail(NRL_E_INVALID, "mask_neg_inf_bwd: negative size");
    if (n == 0) return NRL_OK;
    if (!grad_out || !keep || !grad_in) return fail(NRL_E_INVALID, "mask_neg_inf_bwd: null pointer");
    mask_neg_inf_bwd_kernel<<<dim3(small_grid(n)), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(grad_out, keep, n, grad_in);
    return check_launch("mask_neg_inf_bwd");
}

static int64_t align8(int64_t v) { return (v + 7) / 8 * 8; }

static int64_t terms_chunks(int64_t n) { return n < 1 ? 1 : (n + kTermsBlock - 1) / kTermsBlock; }

// statistics, partial sums, one record per row (16-byte aligned)
static int64_t fused_workspace(int64_t batch, int64_t n_inner, int64_t n_rows) {
    const int64_t b = batch < 1 ? 1 : batch, n = n_inner < 1 ? 1 : n_inner;
    return align8(b * 3 * 4) + b * terms_chunks(n) * P_COUNT * 8 + 16 + (n_rows < 1 ? 1 : n_rows) * R_WORDS * 4;
}
extern "C" int64_t nrl_fused_workspace_bytes(int64_t batch, int64_t n_inner) {
    // (the gradient may have more rows per sequence than the loss has tokens; they have no record)
    return fused_workspace(batch, n_inner, (batch < 1 ? 1 : batch) * (n_inner < 1 ? 1 : n_inner));
}
extern "C" int64_t nrl_fused_packed_workspace_bytes(int64_t n_seq, int64_t n_inner, int64_t total) {
    return fused_workspace(n_seq, n_inner, total);
}

// rows describes the logits; with cu != NULL it is one packed row of rows->n_inner positions (n_outer 1) and
// the loss inputs are [n_seq, in->sm1]
static int fused_impl(const nrl_rows* rows, const nrl_grpo_cfg* cfg, const nrl_grpo_inputs* in, float loss_scale, bool any_row, float* row_grad, void* dlogits,
                      int64_t d_n_inner, int64_t d_stride_outer, int64_t d_stride_inner, float* logprob_out, float* loss_out,
                      float* metrics_out, void* workspace, int64_t workspace_bytes, void* stream, const int32_t* cu,
                      int64_t n_seq, int pre_rolled) {
    if (!rows || !cfg || !in) return fail(NRL_E_INVALID, "null argument");
    if (rows->dtype != NRL_F32 && rows->dtype != NRL_BF16 && rows->dtype != NRL_F16) return fail(NRL_E_INVALID, "unknown logits dtype");
    if (rows->n_outer < 0 || rows->n_inner < 0 || rows->vocab <= 0 || d_n_inner < rows->n_inner) return fail(NRL_E_INVALID, "bad shape");
    if (in->token_mask_type < NRL_MASK_F32 || in->token_mask_type > NRL_MASK_U8) return fail(NRL_E_INVALID, "unknown token mask type");
    if (!cu && (in->batch != rows->n_outer || in->sm1 != rows->n_inner)) return fail(NRL_E_INVALID, "loss inputs and logits rows disagree");
    if (cu && (in->batch != n_seq || rows->n_outer != 1 || n_seq < 0)) return fail(NRL_E_INVALID, "packed loss inputs and cu_seqlens disagree");
    if (rows->vocab_end - rows->vocab_start != rows->vocab) return fail(NRL_E_INVALID, "vocab range does not span the columns");
    if (!(rows->temperature > 0.f)) return fail(NRL_E_INVALID, "temperature must be positive");
    const bool gspo = cfg->sequence_level_importance_ratios && !cfg->disable_ppo_ratio && !cfg->force_on_policy_ratio;
    if (gspo) return fail(NRL_E_UNSUPPORTED, "sequence-level probability ratios need every logprob of a sequence first");
    if (cfg->has_nll) return fail(NRL_E_UNSUPPORTED, "the positive-example NLL term is not fused");
    // sequence-level importance weights are sums over prev - gen; with force_on_policy_ratio prev is the
    // current logprob itself, which does not exist before the pass
    const bool seq_weights = cfg->sequence_level_importance_ratios || cfg->tis_type == NRL_TIS_SEQ_MASK;
    if (seq_weights && cfg->force_on_policy_ratio)
        return fail(NRL_E_UNSUPPORTED, "sequence-level importance weights with force_on_policy_ratio depend on the current logprobs");
    if (seq_weights && in->batch * in->sm1 > 0 && !in->prev) return fail(NRL_E_INVALID, "prev_logprobs is NULL");
    if (cfg->kl_type < 1 || cfg->kl_type > 3 || cfg->tis_type < 0 || cfg->tis_type > 3) return fail(NRL_E_INVALID, "bad kl_type or tis_type");
    const int bytes = rows->dtype == NRL_F32 ? 4 : 2, epv = 16 / bytes;
    const uintptr_t xa = reinterpret_cast<uintptr_t>(rows->logits), da = reinterpret_cast<uintptr_t>(dlogits);
    if (any_row) {
        if (rows->vocab * bytes < NRL_FUSED_ANY_ROW_MIN || rows->vocab * bytes > NRL_FUSED_ANY_ROW_MAX)
            return fail(NRL_E_UNSUPPORTED, "row of %lld bytes", (long long)(rows->vocab * bytes));
        if (((xa - da) & 15) || ((rows->stride_outer - d_stride_outer) * bytes) % 16 || ((rows->stride_inner - d_stride_inner) * bytes) % 16 || xa % bytes)
            return fail(NRL_E_UNSUPPORTED, "logits and gradient rows sit differently on the 16-byte grid");
        if (xa && xa == da) return fail(NRL_E_UNSUPPORTED, "the gradient cannot be written over the logits");
        if (rows->temperature != 1.0f && rows->temp_mode != NRL_TEMP_RCP) return fail(NRL_E_UNSUPPORTED, "temperature as a divide");
        if (reinterpret_cast<uintptr_t>(row_grad) & 15) return fail(NRL_E_INVALID, "row_grad must be 16-byte aligned");
    } else {
        if (rows->vocab % epv || rows->vocab / epv > static_cast<int64_t>(kFusedMaxVec) * 1024)
            return fail(NRL_E_UNSUPPORTED, "row does not fit the on-chip path (vocab %lld)", (long long)rows->vocab);
        if ((xa & 15) || (da & 15) || (rows->stride_outer * bytes) % 16 || (rows->stride_inner * bytes) % 16 ||
            (d_stride_outer * bytes) % 16 || (d_stride_inner * bytes) % 16)
            return fail(NRL_E_UNSUPPORTED, "rows must be 16-byte aligned");
    }
    const int64_t n_rows = rows->n_outer * d_n_inner;
    if (n_rows >= (1ll << 31)) return fail(NRL_E_INVALID, "more than 2^31 rows in one launch");
    if (in->batch * terms_chunks(in->sm1) >= (1ll << 31)) return fail(NRL_E_INVALID, "more than 2^31 shares of sequences");
    if (!loss_out || !metrics_out || !workspace) return fail(NRL_E_INVALID, "null output or workspace");
    const int64_t need = cu ? nrl_fused_packed_workspace_bytes(in->batch, in->sm1, n_rows) : nrl_fused_workspace_bytes(in->batch, in->sm1);
    if (workspace_bytes < need) return fail(NRL_E_WORKSPACE, "workspace too small");
    if (reinterpret_cast<uintptr_t>(workspace) & 7) return fail(NRL_E_INVALID, "workspace must be 8-byte aligned");
    // (empty inputs come without memory: sequences of one token have rows but no token that carries a loss, a microbatch may
    // have no row at all)
    const bool tokens = in->batch * in->sm1 > 0;
    if (!in->global_valid || (in->batch > 0 && !in->sample_mask)) return fail(NRL_E_INVALID, "null sample_mask or global_valid");
    if (n_rows > 0 && (!rows->logits || !dlogits || (any_row && !row_grad))) return fail(NRL_E_INVALID, "null logits, gradient or row_grad");
    if (tokens) {
        if ((n_rows > 0 && !rows->targets) || !logprob_out) return fail(NRL_E_INVALID, "null targets or logprob output");
        if (!in->gen || !in->adv || !in->token_mask) return fail(NRL_E_INVALID, "null loss input");
        if (!cfg->force_on_policy_ratio && !in->prev) return fail(NRL_E_INVALID, "prev_logprobs is NULL");
        if (cfg->has_kl && !in->ref) return fail(NRL_E_INVALID, "reference_policy_logprobs is NULL");
    }
    FusedArgs a;
    a.cfg = *cfg;
    a.in = *in;
    a.in.lp = nullptr; a.in.lpu = nullptr;
    a.cu = cu; a.n_seq = n_seq; a.pre_rolled = pre_rolled;
    a.row_grad = reinterpret_cast<float4*>(row_grad); a.any_row = any_row;
    a.logits = rows->logits; a.n_inner = in->sm1; a.d_n_inner = d_n_inner; a.vocab = rows->vocab;
    a.stride_outer = rows->stride_outer; a.stride_inner = rows->stride_inner;
    a.targets = rows->targets; a.ts_outer = rows->tgt_stride_outer; a.ts_inner = rows->tgt_stride_inner;
    a.vstart = rows->vocab_start; a.vend = rows->vocab_end;
    a.loss_scale = loss_scale;
    a.dlogits = dlogits; a.ds_outer = d_stride_outer; a.ds_inner = d_stride_inner;
    a.lp_out = logprob_out;
    char* ws = static_cast<char*>(workspace);
    a.seq_stats = reinterpret_cast<float*>(ws); ws += align8(in->batch * 3 * 4);
    a.parts = reinterpret_cast<double*>(ws); ws += in->batch * terms_chunks(in->sm1) * P_COUNT * 8;
    a.rec = reinterpret_cast<uint32_t*>(ws + ((16 - (reinterpret_cast<uintptr_t>(ws) & 15)) & 15));
    int tc = 0;
    a.tparam = 1.f;
    if (rows->temperature != 1.0f) {
        if (rows->temp_mode == NRL_TEMP_DIV) { tc = 1; a.tparam = rows->temperature; }
        else { tc = 2; a.tparam = 1.0f / rows->temperature; }
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const unsigned nb = static_cast<unsigned>(in->batch);
    const int64_t items = n_rows > in->batch * in->sm1 ? n_rows : in->batch * in->sm1;
    const unsigned more = static_cast<unsigned>(items < 1024ll * kSeqBlock ? (items + kSeqBlock - 1) / kSeqBlock : 1024);
    if (nb + more > 0) fused_prep_kernel<<<dim3(nb + more), dim3(kSeqBlock), 0, s>>>(a, n_rows, rows->dtype, tc);
    if (n_rows > 0) {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
            return fail(NRL_E_LAUNCH, "cannot read the device's compute-unit count");
        const FusedLaunch l{a, tc, cu != nullptr, n_rows, any_row, cus, s};
        if (rows->dtype == NRL_F32) launch_fused_f32(l);
        else if (rows->dtype == NRL_BF16) launch_fused_bf16(l);
        else launch_fused_f16(l);
    }
    GrpoArgs fa;
    fa.cfg = *cfg;
    fa.in = *in;
    fa.dlp = nullptr; fa.dlpu = nullptr;
    fa.parts = a.parts;
    fa.seq_stats = a.seq_stats; fa.chunks = terms_chunks(in->sm1);
    if (nb > 0) grpo_terms_reduce_kernel<<<dim3((unsigned)(nb * fa.chunks)), dim3(kTermsBlock), 0, s>>>(a, fa.chunks, n_rows);
    grpo_finish_kernel<<<dim3(1), dim3(kSeqBlock), 0, s>>>(fa, loss_out, metrics_out);
    return check_launch("fused_logits_grpo_loss");
}

extern "C" int nrl_fused_logits_grpo_loss(const nrl_rows* rows, const nrl_grpo_cfg* cfg, const nrl_grpo_inputs* in,
                                          float loss_scale, void* dlogits, int64_t d_n_inner, int64_t d_stride_outer,
                                          int64_t d_stride_inner, float* logprob_out, float* loss_out, float* metrics_out,
                                          void* workspace, int64_t workspace_bytes, void* stream) {
    return fused_impl(rows, cfg, in, loss_scale, false, nullptr, dlogits, d_n_inner, d_stride_outer, d_stride_inner, logprob_out, loss_out,
                      metrics_out, workspace, workspace_bytes, stream, nullptr, 0, 0);
}

extern "C" int nrl_fused_packed_logits_grpo_loss(const nrl_rows* rows, int32_t target_is_pre_rolled, const int32_t* cu_seqlens,
                                                 int64_t n_seq, const nrl_grpo_cfg* cfg, const nrl_grpo_inputs* in,
                                                 float loss_scale, void* dlogits, int64_t d_row_stride, float* logprob_out,
                                                 float* loss_out, float* metrics_out, void* workspace, int64_t workspace_bytes,
                                                 void* stream) {
    if (!cu_seqlens) return fail(NRL_E_INVALID, "cu_seqlens is NULL");
    if (rows && rows->tgt_stride_inner != 1) return fail(NRL_E_INVALID, "packed targets must be contiguous");
    return fused_impl(rows, cfg, in, loss_scale, false, nullptr, dlogits, rows ? rows->n_inner : 0, 0, d_row_stride, logprob_out, loss_out,
                      metrics_out, workspace, workspace_bytes, stream, cu_seqlens, n_seq, target_is_pre_rolled);
}

extern "C" int nrl_fused_any_row_grpo_loss(const nrl_rows* rows, int32_t target_is_pre_rolled, const int32_t* cu_seqlens, int64_t n_seq,
                                           const nrl_grpo_cfg* cfg, const nrl_grpo_inputs* in, float loss_scale, float* row_grad_out, void* dlogits,
                                           int64_t d_n_inner, int64_t d_stride_outer, int64_t d_stride_inner, float* logprob_out,
                                           float* loss_out, float* metrics_out, void* workspace, int64_t workspace_bytes, void* stream) {
    if (cu_seqlens && rows && rows->tgt_stride_inner != 1) return fail(NRL_E_INVALID, "packed targets must be contiguous");
    return fused_impl(rows, cfg, in, loss_scale, true, row_grad_out, dlogits, d_n_inner, d_stride_outer, d_stride_inner, logprob_out, loss_out,
                      metrics_out, workspace, workspace_bytes, stream, cu_seqlens, n_seq, target_is_pre_rolled);
}

// The gradient of the rows again, for another upstream factor than the one it was written for (read from the device: with the
// same factor nothing is done).  The factor multiplies d loss / d logprob before the row is formed, so a gradient is rounded
// once whatever it is.
struct RowsGradArgs {
    const void* logits;
    int64_t n_inner, vocab, stride_outer, stride_inner;
    void* d;
    int64_t ds_outer, ds_inner;
    const float4* row_grad;
    const float* factor;
    float written;
    float tparam;
};
template <int DT, int TEMP> __global__ __launch_bounds__(kBlock) void rows_grad_kernel(RowsGradArgs a, int64_t n_rows) {
    const float f = *a.factor;
    if (f == a.written) return;
    for (int64_t r = blockIdx.x; r < n_rows; r += gridDim.x) {
        const int64_t o = r / a.n_inner, i = r - o * a.n_inner;
        char* out = static_cast<char*>(a.d) + (o * a.ds_outer + i * a.ds_inner) * Row<DT>::BYTES;
        const float4 w = a.row_grad[r];
        const float g = w.x * f;
        if (g == 0.f) {
            row_zero<DT>(out, a.vocab);
            continue;
        }
        const char* row = static_cast<const char*>(a.logits) + (o * a.stride_outer + i * a.stride_inner) * Row<DT>::BYTES;
        row_write_grad<DT, TEMP>(row, out, a.vocab, w.y, g, __float_as_int(w.z), a.tparam);
    }
}

extern "C" int nrl_rows_grad(const nrl_rows* rows, const float* row_grad, const float* factor, float written, void* dlogits,
                             int64_t d_stride_outer, int64_t d_stride_inner, void* stream) {
    if (!rows) return fail(NRL_E_INVALID, "rows_grad: null argument");
    if (rows->dtype != NRL_F32 && rows->dtype != NRL_BF16 && rows->dtype != NRL_F16) return fail(NRL_E_INVALID, "unknown logits dtype");
    if (rows->n_outer < 0 || rows->n_inner < 0 || rows->vocab <= 0 || rows->vocab >= (1ll << 31)) return fail(NRL_E_INVALID, "bad shape");
    if (!(rows->temperature > 0.f) || (rows->temperature != 1.0f && rows->temp_mode != NRL_TEMP_RCP))
        return fail(NRL_E_UNSUPPORTED, "rows_grad: temperature must be a positive multiplication");
    const int64_t n_rows = rows->n_outer * rows->n_inner;
    if (n_rows == 0) return NRL_OK;
    if (!rows->logits || !row_grad || !factor || !dlogits) return fail(NRL_E_INVALID, "rows_grad: null pointer");
    const bool temp = rows->temperature != 1.0f;
    const RowsGradArgs a{rows->logits, rows->n_inner, rows->vocab, rows->stride_outer, rows->stride_inner, dlogits, d_stride_outer, d_stride_inner,
                         reinterpret_cast<const float4*>(row_grad), factor, written, temp ? 1.0f / rows->temperature : 1.f};
    const dim3 grid((unsigned)(n_rows < 2048 ? n_rows : 2048)), block(kBlock);
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (rows->dtype * 2 + (temp ? 1 : 0)) {
        case NRL_F32 * 2: rows_grad_kernel<NRL_F32, 0><<<grid, block, 0, s>>>(a, n_rows); break;
        case NRL_F32 * 2 + 1: rows_grad_kernel<NRL_F32, 2><<<grid, block, 0, s>>>(a, n_rows); break;
        case NRL_BF16 * 2: rows_grad_kernel<NRL_BF16, 0><<<grid, block, 0, s>>>(a, n_rows); break;
        case NRL_BF16 * 2 + 1: rows_grad_kernel<NRL_BF16, 2><<<grid, block, 0, s>>>(a, n_rows); break;
        case NRL_F16 * 2: rows_grad_kernel<NRL_F16, 0><<<grid, block, 0, s>>>(a, n_rows); break;
        default: rows_grad_kernel<NRL_F16, 2><<<grid, block, 0, s>>>(a, n_rows); break;
    }
    return check_launch("rows_grad");
}
