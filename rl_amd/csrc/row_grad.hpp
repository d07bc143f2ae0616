// One row's gradient by one workgroup: g * (onehot - softmax), or zeros.
#pragma once

#include "common.hpp"

namespace nrl {

constexpr int kBlock = 256;  // one workgroup of 4 wave64 per row
constexpr int kUnroll = 4;   // 16-byte loads in flight per lane

// rows that are read and written in the same pass stream through non-temporal loads and stores; rows
// that are only written (zero gradients) use plain stores, which a pure write stream sustains faster
template <typename P> __device__ __forceinline__ u32x4 k2_load(const P* p) { return __builtin_nontemporal_load(p); }
template <typename P> __device__ __forceinline__ void k2_store(u32x4 v, P* p) { __builtin_nontemporal_store(v, p); }

template <int DT> __device__ __forceinline__ void row_zero(void* row, int64_t vocab) {
    constexpr int EPV = Row<DT>::EPV;
    const int tid = threadIdx.x;
    const int64_t head = row_head<DT>(row, vocab);
    const int64_t nvec = (vocab - head) / EPV;
    u32x4* ov = reinterpret_cast<u32x4*>(static_cast<char*>(row) + head * Row<DT>::BYTES);
    const u32x4 z = {0u, 0u, 0u, 0u};
    for (int64_t i = tid; i < nvec; i += kBlock) ov[i] = z;
    if (tid < head) Row<DT>::store1(row, tid, 0.f);
    const int64_t tail0 = head + nvec * EPV;
    if (tail0 + tid < vocab) Row<DT>::store1(row, tail0 + tid, 0.f);
}

template <int DT, int TEMP>
__device__ __forceinline__ void row_write_grad(const void* row, void* out, int64_t vocab, float lse, float g,
                                               int64_t tgt, float tparam) {
    constexpr int EPV = Row<DT>::EPV;
    const int tid = threadIdx.x;
    const RowGrad rg(lse, g, tparam);
    const int64_t head = row_head<DT>(row, vocab);
    if (row_head<DT>(out, vocab) != head) {
        // input and output rows are not congruent modulo 16 bytes: element-wise path
        for (int64_t i = tid; i < vocab; i += kBlock)
            Row<DT>::store1(out, i, grad_elem<DT, TEMP>(Row<DT>::load1(row, i), i == tgt, rg));
        return;
    }
    const int64_t nvec = (vocab - head) / EPV;
    const u32x4* xv = reinterpret_cast<const u32x4*>(static_cast<const char*>(row) + head * Row<DT>::BYTES);
    u32x4* ov = reinterpret_cast<u32x4*>(static_cast<char*>(out) + head * Row<DT>::BYTES);
    const int64_t tvec = tgt >= head ? (tgt - head) / EPV : -1;  // vector that holds the target
    const int tsub = tgt >= head ? static_cast<int>((tgt - head) % EPV) : -1;

    int64_t base = 0;
    for (; base + kUnroll * kBlock <= nvec; base += kUnroll * kBlock) {
        u32x4 r[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) r[u] = k2_load(xv + base + u * kBlock + tid);
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int64_t vi = base + u * kBlock + tid;
            k2_store(grad_vec<DT, TEMP>(r[u], vi == tvec ? tsub : -1, rg), ov + vi);
        }
    }
    for (int64_t vi = base + tid; vi < nvec; vi += kBlock)
        k2_store(grad_vec<DT, TEMP>(k2_load(xv + vi), vi == tvec ? tsub : -1, rg), ov + vi);
    if (tid < head) Row<DT>::store1(out, tid, grad_elem<DT, TEMP>(Row<DT>::load1(row, tid), tid == tgt, rg));
    const int64_t tail0 = head + nvec * EPV;
    if (tail0 + tid < vocab) {
        const int64_t i = tail0 + tid;
        Row<DT>::store1(out, i, grad_elem<DT, TEMP>(Row<DT>::load1(row, i), i == tgt, rg));
    }
}

}  // namespace nrl
