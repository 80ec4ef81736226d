// Recurrent gated-delta-rule step (decode, T >= 1) for gfx950.
//
// The reference has no native decode; its decode path is the torch token
// recurrence transformers modeling_qwen3_5.py:331-380
// (torch_recurrent_gated_delta_rule), per token:
//   S <- e^{g} S;  kv = S^T k;  delta = beta (v - kv);  S <- S + k delta^T;
//   o = s S^T q    (o reads the updated state, s = 1/sqrt(DK))
// which this kernel fuses into one read and one write of S per call:
//   a = S^T k,  b = S^T q             (one pass over the old state)
//   delta = beta (v - e^g a)
//   o = s (e^g b + delta (k . q))     (= s S_new^T q)
//   S_new = e^g S + k delta^T         (written back in place)
//
// The state's columns evolve independently, so each (batch, v-head) is split
// over two work-groups of 256 threads, one per half of the columns: thread t
// of half h owns columns 64 h + 4 (t % 16) .. + 3 of rows (t / 16) + 16 m,
// m = 0..7, so every load/store instruction of a wave moves four 256-byte
// half rows.  Two groups of 32 state registers per thread (rather than one of
// 64) leave room for more groups per CU, whose loads overlap each other's
// arithmetic and stores.  Tokens t > 0 reuse the registers; HBM sees the
// state exactly once in each direction.
#include "gdn_common.h"
#include "gdn_hip.h"

#include <math.h>

#include <algorithm>

namespace gdn {
namespace {

constexpr int kDecThreads = 256;
// Work-groups per (batch, v-head), each taking the state's columns
// [c * kDecCols, (c + 1) * kDecCols): 2 measured fastest at B=64 HV=32 (1: 50.2
// us, 2: 47.9 us, 4: 50.4 us), since two halves give 4 groups per CU at 110
// VGPRs where one group per (b, h) holds 190 VGPRs.
constexpr int kDecSplit = 2;
constexpr int kDecCols = kDV / kDecSplit;     // columns per work-group
constexpr int kColBlocks = kDecCols / 4;      // 16 column blocks of 4
constexpr int kRowGroups = kDecThreads / kColBlocks;   // 16
constexpr int kRowsPerThread = kDK / kRowGroups;       // 8
static_assert(kRowGroups * kRowsPerThread == kDK && kRowGroups % 4 == 0, "row groups");

// kNorm: q and k rows are raw and normalised here first, x rsqrt(sum x^2 +
// 1e-6) in fp32 rounded to bf16 (transformers' use_qk_l2norm_in_kernel).
// q, k and v are read where they lie, heads contiguous and batches and tokens
// at the given strides (slices of one conv output, say), and the state may
// go to another buffer than it came from (or come from none: zeros): a
// caller that keeps the old state needs no copy of it, one pass over the
// state instead of two (a B=24 HV=32 layer step with conv and norm: 49.5 ->
// 26 us).  Reading and writing one buffer is safe: a thread reads its
// elements before it writes them, and no other thread touches them.  The
// state is the caller's and may be a view at any float (f32x4_a4; the hardware
// takes 16-byte accesses at 4-byte addresses).
struct DecStrides {   // elements; a batch's T tokens may span more than 31 bits
    int64_t qb, kb, vb;
    int qt, kt, vt;
};

// Elements in front of batch b's token t
__host__ __device__ __forceinline__ size_t dec_row(int b, int64_t bs, int t, int ts) {
    return (size_t)b * (size_t)bs + (size_t)t * (size_t)ts;
}

// kFrom: where the state comes from
constexpr int kFromOut = 0, kFromIn = 1, kFromZero = 2;   // state_out itself, state_in, zeros

template <bool kNorm, int kFrom>
__global__ __launch_bounds__(kDecThreads) void gdn_recurrent_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, const float* __restrict__ g,
    const float* __restrict__ beta, uint16_t* __restrict__ o, const float* __restrict__ state_in,
    float* __restrict__ state_out, int T, int HV, int rep, float scale, DecStrides st) {
    __shared__ float qs[kDK], ks[kDK];
    __shared__ f32x4 part[4][2][kColBlocks];  // [wave][a|b][column block]
    __shared__ float kq;

    // the kernel arguments' cache lines, requested together
    asm volatile("" ::"s"(q), "s"(o), "s"(rep), "s"(st.vt));
    const int tid = threadIdx.x;
    const int cb = tid & (kColBlocks - 1);   // column block: columns c0 + 4cb .. + 3
    const int rg = tid / kColBlocks;         // row group: rows rg + 16m
    const int wave = tid >> 6;
    // grid (kDecSplit HV, batches): one division (by the heads per k-head)
    // stands between the kernel's start and its first load, not three
    const int hv = blockIdx.x / kDecSplit;
    const int c0 = kDecCols * (blockIdx.x % kDecSplit);
    const int b = blockIdx.y;
    const int bh = b * HV + hv;
    const int hk = (unsigned)hv / (unsigned)rep;

    // A token's inputs: this thread's element of q (threads 0..127) or k
    // (128..255), its four v columns, g and beta.  Token 0's are requested
    // before the state, so forming q and k needs only them; each later
    // token's are requested during the previous token's work.
    const uint16_t* qk = tid < kDK ? q + dec_row(b, st.qb, 0, st.qt) + (size_t)hk * kDK + tid
                                   : k + dec_row(b, st.kb, 0, st.kt) + (size_t)hk * kDK + tid - kDK;
    const int qkt = tid < kDK ? st.qt : st.kt;
    const uint16_t* vp = v + dec_row(b, st.vb, 0, st.vt) + (size_t)hv * kDV + c0 + 4 * cb;
    float* qk_dst = tid < kDK ? qs + tid : ks + tid - kDK;
    auto load_token = [&](int t, uint16_t& qkr, uint2& vr, float& gr, float& br) {
        const size_t tk = (size_t)b * T + t;
        qkr = qk[dec_row(0, 0, t, qkt)];
        vr = *reinterpret_cast<const uint2*>(vp + dec_row(0, 0, t, st.vt));
        gr = g[tk * HV + hv];
        br = beta[tk * HV + hv];
    };
    uint16_t qkr;
    uint2 vraw;
    float gt, bt;
    __builtin_assume(T >= 1);   // the launcher returns before T = 0
    load_token(0, qkr, vraw, gt, bt);
    __builtin_amdgcn_sched_barrier(0);   // keeps them ahead of the state loads

    const size_t sb = (size_t)bh * kDK * kDV;
    f32x4 s[kRowsPerThread];
    if constexpr (kFrom != kFromZero) {
        const float* S = (kFrom == kFromOut ? state_out : state_in) + sb;
#pragma unroll
        for (int m = 0; m < kRowsPerThread; ++m)
            s[m] = __builtin_nontemporal_load(
                reinterpret_cast<const f32x4_a4*>(S + (rg + kRowGroups * m) * kDV + c0) + cb);
    } else {
#pragma unroll
        for (int m = 0; m < kRowsPerThread; ++m) s[m] = zero4();
    }

    for (int t = 0; t < T; ++t) {
        const size_t tk = ((size_t)b * T + t);
        *qk_dst = bf16_bits_to_f32(qkr);
        __syncthreads();
        if (kNorm) {
            if (wave == 0) {
                const int l = tid;
                float pq = qs[l] * qs[l] + qs[l + 64] * qs[l + 64];
                float pk = ks[l] * ks[l] + ks[l + 64] * ks[l + 64];
                for (int off = 32; off > 0; off >>= 1) {
                    pq += __shfl_xor(pq, off, 64);
                    pk += __shfl_xor(pk, off, 64);
                }
                const float iq = rsqrtf(pq + 1e-6f), ik = rsqrtf(pk + 1e-6f);
                qs[l] = bf16_bits_to_f32(f32_to_bf16_bits(qs[l] * iq));
                qs[l + 64] = bf16_bits_to_f32(f32_to_bf16_bits(qs[l + 64] * iq));
                ks[l] = bf16_bits_to_f32(f32_to_bf16_bits(ks[l] * ik));
                ks[l + 64] = bf16_bits_to_f32(f32_to_bf16_bits(ks[l + 64] * ik));
            }
            __syncthreads();
        }
        if (wave == 0) {
            float p = qs[tid] * ks[tid] + qs[tid + 64] * ks[tid + 64];
            for (int off = 32; off > 0; off >>= 1) p += __shfl_xor(p, off, 64);
            if (tid == 0) kq = p;
        }
        // partial a = S^T k, b = S^T q over this thread's rows
        f32x4 pa = zero4(), pb = zero4();
#pragma unroll
        for (int m = 0; m < kRowsPerThread; ++m) {
            const int r = rg + kRowGroups * m;
            pa += s[m] * ks[r];
            pb += s[m] * qs[r];
        }
        // the lanes of a wave with one column block (lane % kColBlocks) add up
#pragma unroll
        for (int off = kColBlocks; off < 64; off <<= 1) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pa[i] += __shfl_xor(pa[i], off, 64);
                pb[i] += __shfl_xor(pb[i], off, 64);
            }
        }
        if ((tid & 63) < kColBlocks) {
            part[wave][0][cb] = pa;
            part[wave][1][cb] = pb;
        }
        __syncthreads();
        f32x4 a = part[0][0][cb] + part[1][0][cb] + part[2][0][cb] + part[3][0][cb];
        f32x4 bq = part[0][1][cb] + part[1][1][cb] + part[2][1][cb] + part[3][1][cb];
        const float decay = expf(gt);
        f32x4 vv;
        vv[0] = bf16_bits_to_f32(vraw.x & 0xffffu);
        vv[1] = bf16_bits_to_f32(vraw.x >> 16);
        vv[2] = bf16_bits_to_f32(vraw.y & 0xffffu);
        vv[3] = bf16_bits_to_f32(vraw.y >> 16);
        const f32x4 delta = (vv - a * decay) * bt;
        if (t + 1 < T) load_token(t + 1, qkr, vraw, gt, bt);
        if (rg == 0) {
            const f32x4 ov = (bq * decay + delta * kq) * scale;
            uint2 packed;
            packed.x = (uint32_t)f32_to_bf16_bits(ov[0]) | ((uint32_t)f32_to_bf16_bits(ov[1]) << 16);
            packed.y = (uint32_t)f32_to_bf16_bits(ov[2]) | ((uint32_t)f32_to_bf16_bits(ov[3]) << 16);
            *reinterpret_cast<uint2*>(o + (tk * HV + hv) * kDV + c0 + 4 * cb) = packed;
        }
#pragma unroll
        for (int m = 0; m < kRowsPerThread; ++m) s[m] = s[m] * decay + delta * ks[rg + kRowGroups * m];
        __syncthreads();  // qs/ks/part are rewritten by the next token
    }
    float* S = state_out + sb;
#pragma unroll
    for (int m = 0; m < kRowsPerThread; ++m)
        __builtin_nontemporal_store(
            s[m], reinterpret_cast<f32x4_a4*>(S + (rg + kRowGroups * m) * kDV + c0) + cb);
}

}  // namespace
}  // namespace gdn

using namespace gdn;

namespace {
hipError_t recurrent_launch(const void* q, const void* k, const void* v, const float* g,
                            const float* beta, void* o, const float* state_in, float* state_out,
                            int B, int T, int HV, int HQK, int DK, int DV, const DecStrides& st,
                            hipStream_t stream, bool norm) {
    if (DK != kDK || DV != kDV || B <= 0 || T < 0 || HV <= 0 || HQK <= 0 || HV % HQK != 0)
        return hipErrorInvalidValue;
    if (!state_out) return hipErrorInvalidValue;
    if (T > 0 && (!q || !k || !v || !g || !beta || !o)) return hipErrorInvalidValue;
    if (T == 0) return hipSuccess;
    const int from = state_in == state_out ? kFromOut : state_in ? kFromIn : kFromZero;
    auto kern = norm ? (from == kFromOut ? gdn_recurrent_kernel<true, kFromOut>
                        : from == kFromIn ? gdn_recurrent_kernel<true, kFromIn>
                                          : gdn_recurrent_kernel<true, kFromZero>)
                     : (from == kFromOut ? gdn_recurrent_kernel<false, kFromOut>
                        : from == kFromIn ? gdn_recurrent_kernel<false, kFromIn>
                                          : gdn_recurrent_kernel<false, kFromZero>);
    // a grid's second dimension ends at 65535
    for (int b0 = 0; b0 < B; b0 += 65535) {
        const size_t tk = (size_t)b0 * T, so = (size_t)b0 * HV * kDK * kDV;
        hipLaunchKernelGGL(kern, dim3((unsigned)(kDecSplit * HV), (unsigned)std::min(B - b0, 65535)),
                           dim3(kDecThreads), 0, stream,
                           static_cast<const uint16_t*>(q) + dec_row(b0, st.qb, 0, st.qt),
                           static_cast<const uint16_t*>(k) + dec_row(b0, st.kb, 0, st.kt),
                           static_cast<const uint16_t*>(v) + dec_row(b0, st.vb, 0, st.vt), g + tk * HV,
                           beta + tk * HV, static_cast<uint16_t*>(o) + tk * HV * kDV,
                           state_in ? state_in + so : nullptr, state_out + so, T, HV, HV / HQK,
                           1.0f / sqrtf((float)kDK), st);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    }
    return hipSuccess;
}

// q, k [B][T][HQK][DK] and v [B][T][HV][DV] without gaps
DecStrides packed(int T, int HV, int HQK) {
    const int qt = HQK * kDK, vt = HV * kDV;
    return DecStrides{(int64_t)T * qt, (int64_t)T * qt, (int64_t)T * vt, qt, qt, vt};
}
}  // namespace

extern "C" hipError_t deltanet_recurrent_step(const void* q, const void* k, const void* v,
                                              const float* g, const float* beta, void* o,
                                              float* state, int B, int T, int HV, int HQK,
                                              int DK, int DV, hipStream_t stream) {
    return recurrent_launch(q, k, v, g, beta, o, state, state, B, T, HV, HQK, DK, DV,
                            packed(T, HV, HQK), stream, false);
}

extern "C" hipError_t deltanet_recurrent_step_l2norm(const void* q, const void* k, const void* v,
                                                     const float* g, const float* beta, void* o,
                                                     float* state, int B, int T, int HV,
                                                     int HQK, int DK, int DV,
                                                     hipStream_t stream) {
    return recurrent_launch(q, k, v, g, beta, o, state, state, B, T, HV, HQK, DK, DV,
                            packed(T, HV, HQK), stream, true);
}

extern "C" hipError_t deltanet_recurrent_step_strided(
    const void* q, const void* k, const void* v, const float* g, const float* beta, void* o,
    const float* state_in, float* state_out, int B, int T, int HV, int HQK, int64_t q_batch,
    int64_t q_token, int64_t k_batch, int64_t k_token, int64_t v_batch, int64_t v_token,
    int qk_l2norm, hipStream_t stream) {
    for (int64_t x : {q_batch, q_token, k_batch, k_token, v_batch, v_token})
        if (x < 0 || x > 0x7fffffff) return hipErrorInvalidValue;
    // v is read 8 bytes at a time
    if (reinterpret_cast<uintptr_t>(v) % 8 || v_batch % 4 || v_token % 4)
        return hipErrorInvalidValue;
    if (T == 0) {   // no token: the state as it was
        if (B <= 0 || HV <= 0 || !state_out) return hipErrorInvalidValue;
        if (state_in == state_out) return hipSuccess;
        return hipErrorInvalidValue;
    }
    return recurrent_launch(q, k, v, g, beta, o, state_in, state_out, B, T, HV, HQK, kDK, kDV,
                            DecStrides{q_batch, k_batch, v_batch, (int)q_token, (int)k_token,
                                       (int)v_token},
                            stream, qk_l2norm != 0);
}

extern "C" size_t deltanet_recurrent_row_offset(int T, int heads, int b, int t, int h) {
    const DecStrides st = packed(T, heads, heads);
    return dec_row(b, st.vb, t, st.vt) + (size_t)h * kDV;
}
