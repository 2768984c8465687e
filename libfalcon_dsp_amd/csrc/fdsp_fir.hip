// fdsp_fir.hip -- FIR with complex taps, one stream, on gfx950
// (reference falcon_dsp_fir_filter::apply, src/transform/falcon_dsp_fir_filter.cc:
//  151-243; CUDA __fir_filter, src/transform/falcon_dsp_fir_filter_cuda.cu:102-187).
// y[n] = sum_k h[k] x[n-k], the last M-1 inputs carried from chunk to chunk.
//
//   fir_mfma_kernel  float samples: the convolution as FP32 matrix products
//   fir_seq_kernel   int16 samples: the reference's unfused sums in tap order,
//                    so the truncated outputs are the reference's bit for bit
//   fir_kernel       filters whose window exceeds the LDS of the others
#include <algorithm>
#include <type_traits>

#include "fdsp_internal.h"

namespace fdsp {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// wavefront-uniform taps through the scalar cache
typedef const __attribute__((address_space(4))) float *ctaps_ptr;

constexpr uint32_t kBlock = 256, kWaves = kBlock / 64;
constexpr size_t kLdsMax = 64 * 1024;

// the next history: the last m - 1 samples of [history | chunk] (block 0)
template <typename TI>
__device__ __forceinline__ void carry_history(const TI *in, uint32_t n, uint32_t hlen, const float2 *hist_in,
                                              float2 *hist_out)
{
    for (uint32_t t = threadIdx.x; t < hlen; t += kBlock) {
        const int64_t i = (int64_t)n - hlen + t;
        hist_out[t] = i >= 0 ? sample_f32(in[i]) : hist_in[hlen + i];
    }
}

// sample i of [history | chunk], zero outside them
template <typename TI>
__device__ __forceinline__ float2 sample_at(const TI *in, uint32_t n, uint32_t hlen, const float2 *hist_in, int64_t i)
{
    if (i >= 0)
        return i < n ? sample_f32(in[i]) : make_float2(0.f, 0.f);
    return i >= -(int64_t)hlen ? hist_in[hlen + i] : make_float2(0.f, 0.f);
}

__device__ __forceinline__ bool not_finite(float2 v)
{
    constexpr uint32_t kExp = 0x7f800000u;
    return (__float_as_uint(v.x) & kExp) == kExp || (__float_as_uint(v.y) & kExp) == kExp;
}

// ---------------------------------------------------------------------------
// Float samples. For 16 consecutive outputs y[16b + r] = sum_t H[r][t] W[t][b]
// with H[r][t] = h[t - 15 + r] (a banded Toeplitz matrix of the taps) and
// W[t][b] = x[16b + 15 - t], K = m + 15 rounded up to 16 (kp): real matrix
// products on v_mfma_f32_16x16x4f32, A = H (lane l: row l%16, k l/16), B = W
// (column l%16, k l/16); lane l is left with outputs 4(l/16) .. +3 of block
// l%16. Complex taps take four products a step (yr = Hr Xr - Hi Xi, yi = Hr Xi
// + Hi Xr), real taps (kReal) two.
//
// A product with a zero of H is zero only for a finite sample, so a block
// whose window holds an infinity or a NaN computes its outputs tap by tap.
//
// kSplit: the block's waves share one set of outputs and split its K rounds,
// their sums added through LDS; for chunks too short to give every SIMD a
// wave otherwise.
//
// Bound by the matrix cores on long filters (2^22 samples, 512 complex taps:
// 137 us, 125 of the 153 TFLOP/s that a large FP32 matrix product reaches), by
// staging and launch on short ones. 10^6 samples, 129 complex taps: 14.4 us
// against 34 for one output a thread on the vector ALUs with tap and sample
// each read from LDS. A wave takes 256 outputs: 512 and 1024 a wave (two and
// four B operands per A) were within 4% on 4 x 10^6 samples and 3% to 150%
// slower below 10^6, where they leave SIMDs idle.
// ---------------------------------------------------------------------------
// one padding sample per 16, so the 16 columns of a B read fall in distinct banks
__host__ __device__ __forceinline__ uint32_t pad16(uint32_t q) { return q + (q >> 4); }

// outputs of a block: 256 a wave, or 256 for its four waves together
__host__ __device__ constexpr uint32_t mfma_tile(bool split) { return split ? 256u : kWaves * 256u; }

template <bool kSplit, bool kReal>
__global__ __launch_bounds__(kBlock) void fir_mfma_kernel(const float2 *__restrict__ in, uint32_t n,
                                                          const float2 *__restrict__ taps, uint32_t m, uint32_t kp,
                                                          const float2 *__restrict__ hist_in,
                                                          float2 *__restrict__ hist_out, float2 *__restrict__ out)
{
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr uint32_t kTile = mfma_tile(kSplit);
    float2 *xs = reinterpret_cast<float2 *>(smem);
    const uint32_t span = kTile + kp - 16;
    float2 *hs = xs + ((pad16(span) + 2) & ~1u);  // kp + 16 taps
    const uint32_t tid = threadIdx.x, hlen = m - 1;
    if (blockIdx.x == 0)
        carry_history(in, n, hlen, hist_in, hist_out);
    const uint32_t o0 = blockIdx.x * kTile;
    // window x[lo .. lo + span); W[t][b] at window index 16 b + kp - 1 - t
    const int64_t lo = (int64_t)o0 + 16 - (int64_t)kp;
    for (uint32_t u = tid; u < kp + 16; u += kBlock)
        hs[u] = u >= 15 && u - 15 < m ? taps[u - 15] : make_float2(0.f, 0.f);
    bool odd_value = false;
    constexpr uint32_t kU = 4;
    if (lo >= 0 && lo + span <= n) {
        // the whole window inside the chunk: four loads a thread in flight,
        // their indices clamped into the span
        for (uint32_t t0 = tid; t0 < span; t0 += kBlock * kU) {
            float2 v[kU];
#pragma unroll
            for (uint32_t u = 0; u < kU; ++u)
                v[u] = in[lo + min(t0 + u * kBlock, span - 1)];
#pragma unroll
            for (uint32_t u = 0; u < kU; ++u) {
                odd_value |= not_finite(v[u]);
                if (t0 + u * kBlock < span)
                    xs[pad16(t0 + u * kBlock)] = v[u];
            }
        }
    } else {
        for (uint32_t t = tid; t < span; t += kBlock) {
            const float2 v = sample_at(in, n, hlen, hist_in, lo + t);
            odd_value |= not_finite(v);
            xs[pad16(t)] = v;
        }
    }
    if (__syncthreads_or(odd_value)) {
        // the sample of output o0 + q at distance k: window index q + kp - 16 - k
        for (uint32_t q = tid; q < kTile && o0 + q < n; q += kBlock) {
            float2 acc = make_float2(0.f, 0.f);
            for (uint32_t k = 0; k < m; ++k) {
                const float2 x = xs[pad16(q + kp - 16 - k)], h = hs[k + 15];
                acc.x += x.x * h.x - x.y * h.y;
                acc.y += x.x * h.y + x.y * h.x;
            }
            out[o0 + q] = acc;
        }
        return;
    }
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, kq = lane >> 4, j = lane & 15;
    const uint32_t ob = kSplit ? 0u : wave * 16u;  // the wave's first block of 16 outputs in the tile
    // Eight chains, added at the end: the products of each tap part, even and
    // odd K steps apart. One chain of all of them was 1.4 times further from
    // the sum in 64 bits than the sequential sum is (2.6e-7 against 1.9e-7 of
    // the result at 129 taps).
    const floatx4 zero{0.f, 0.f, 0.f, 0.f};
    floatx4 rr[2] = {zero, zero}, ri[2] = {zero, zero}, ir[2] = {zero, zero}, ii[2] = {zero, zero};
    // Rounds of four K steps, t0 = 16u + 4s. W[t0 + kq][block j] sits at
    // pad16(q0 - t0) = pad16(q0) - e_s - 17u with e_s = 4s + (4s > q0 mod 16);
    // H[j][t0 + kq] at t0 + kq + j.
    const uint32_t first = kSplit ? wave : 0u;
    constexpr uint32_t kStep = kSplit ? kWaves : 1u;
    const uint32_t q0 = 16 * (ob + j) + kp - 1 - kq;
    uint32_t bo[4];
#pragma unroll
    for (uint32_t st = 0; st < 4; ++st)
        bo[st] = pad16(q0) - (4 * st + (4 * st > (q0 & 15) ? 1u : 0u)) - 17 * first;
    uint32_t ao = kq + j + 16 * first;
    for (uint32_t u = first; u < kp / 16; u += kStep) {
#pragma unroll
        for (uint32_t st = 0; st < 4; ++st) {
            const float2 a = hs[ao + 4 * st], b = xs[bo[st]];
            rr[st & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, rr[st & 1], 0, 0, 0);
            ri[st & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.y, ri[st & 1], 0, 0, 0);
            if constexpr (!kReal) {
                ii[st & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, ii[st & 1], 0, 0, 0);
                ir[st & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.x, ir[st & 1], 0, 0, 0);
            }
        }
        ao += 16 * kStep;
#pragma unroll
        for (uint32_t st = 0; st < 4; ++st)
            bo[st] -= 17 * kStep;
    }
    floatx4 dr = rr[0] + rr[1], di = ri[0] + ri[1];
    if constexpr (!kReal) {
        dr -= ii[0] + ii[1];
        di += ir[0] + ir[1];
    }
    if constexpr (kSplit) {
        // the waves' partial sums, [wave][output], over the window (no longer read)
        __syncthreads();
        float4 *p = reinterpret_cast<float4 *>(xs + wave * kTile + 16 * j + 4 * kq);
        p[0] = make_float4(dr[0], di[0], dr[1], di[1]);
        p[1] = make_float4(dr[2], di[2], dr[3], di[3]);
        __syncthreads();
        float2 s = xs[tid];
#pragma unroll
        for (uint32_t w = 1; w < kWaves; ++w) {
            const float2 v = xs[w * kTile + tid];
            s.x += v.x;
            s.y += v.y;
        }
        if (o0 + tid < n)
            out[o0 + tid] = s;
    } else {
        const uint32_t o = o0 + 16 * (ob + j) + 4 * kq;
        if ((reinterpret_cast<uintptr_t>(out) & 15) == 0 && o + 4 <= n) {
            float4 *p = reinterpret_cast<float4 *>(out + o);
            p[0] = make_float4(dr[0], di[0], dr[1], di[1]);
            p[1] = make_float4(dr[2], di[2], dr[3], di[3]);
        } else {
#pragma unroll
            for (uint32_t v = 0; v < 4; ++v)
                if (o + v < n)
                    out[o + v] = make_float2(dr[v], di[v]);
        }
    }
}

size_t mfma_lds(bool split, uint32_t kp)
{
    const uint32_t span = mfma_tile(split) + kp - 16;
    size_t lds = (((size_t)pad16(span) + 2) & ~(size_t)1) * sizeof(float2) + (size_t)(kp + 16) * sizeof(float2);
    if (split)
        lds = std::max(lds, (size_t)kWaves * 256 * sizeof(float2));
    return lds;
}

template <bool kSplit>
hipError_t launch_mfma(const float2 *in, uint32_t n, const float2 *taps, uint32_t m, uint32_t kp, bool real,
                       const float2 *hist_in, float2 *hist_out, float2 *out, hipStream_t s)
{
    const uint32_t tile = mfma_tile(kSplit);
    const dim3 grid((n + tile - 1) / tile), block(kBlock);
    const size_t lds = mfma_lds(kSplit, kp);
    if (real)
        hipLaunchKernelGGL((fir_mfma_kernel<kSplit, true>), grid, block, lds, s, in, n, taps, m, kp, hist_in,
                           hist_out, out);
    else
        hipLaunchKernelGGL((fir_mfma_kernel<kSplit, false>), grid, block, lds, s, in, n, taps, m, kp, hist_in,
                           hist_out, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Int16 samples. The reference rounds each complex product and each sum
// (falcon_dsp_fir_filter.cc:208-230), in tap order. One output a thread, eight
// taps a step: eight window reads from LDS, the taps scalar operands. With
// real taps (kReal) the products with their zero imaginary parts only add
// signed zeros to finite samples and are left out; the carried history is
// float and may hold anything, so the tiles that read it keep all products.
//
// Bound by VALU issue on long chunks (2^20 samples, 256 taps: 42 us complex,
// 32 us real, against 31 and 16 of sums alone), by launch and latency on short
// ones: 2^18 samples, 64 real taps 4.6 us, where one output a thread over
// 2048-output tiles, tap and sample each read from LDS, took 19 us on 128
// blocks. Two or four outputs a thread (fewer LDS reads, fewer waves) took 6.7
// and 8.5 us there and no less on 2^20; taps through LDS, or read one step
// ahead, 5.4 to 5.9 us.
// ---------------------------------------------------------------------------
constexpr uint32_t kSeqT = 8;  // taps a step

template <bool kReal>
__device__ __forceinline__ float2 seq_sum(const float2 *xw, ctaps_ptr h, uint32_t m)
{
#pragma clang fp contract(off)
    float2 acc = make_float2(0.f, 0.f);
    const auto add = [&](float2 x, uint32_t k) {
        float2 p;
        if constexpr (kReal)
            p = make_float2(x.x * h[2 * k], x.y * h[2 * k]);
        else
            p = cmul_ref(x, make_float2(h[2 * k], h[2 * k + 1]));
        acc.x = acc.x + p.x;
        acc.y = acc.y + p.y;
    };
    uint32_t k0 = 0;
    for (; k0 + kSeqT <= m; k0 += kSeqT) {
        float2 w[kSeqT];
#pragma unroll
        for (uint32_t i = 0; i < kSeqT; ++i)
            w[i] = xw[-(int32_t)(k0 + i)];
#pragma unroll
        for (uint32_t i = 0; i < kSeqT; ++i)
            add(w[i], k0 + i);
    }
    for (; k0 < m; ++k0)
        add(xw[-(int32_t)k0], k0);
    return acc;
}

template <bool kReal>
__global__ __launch_bounds__(kBlock) void fir_seq_kernel(const short2 *__restrict__ in, uint32_t n,
                                                         const float2 *__restrict__ taps, uint32_t m,
                                                         const float2 *__restrict__ hist_in,
                                                         float2 *__restrict__ hist_out, short2 *__restrict__ out)
{
    extern __shared__ __align__(16) unsigned char smem[];
    float2 *xs = reinterpret_cast<float2 *>(smem);
    const uint32_t tid = threadIdx.x, hlen = m - 1;
    if (blockIdx.x == 0)
        carry_history(in, n, hlen, hist_in, hist_out);
    const uint32_t o0 = blockIdx.x * kBlock;
    // window x[o0 - hlen .. o0 + kBlock)
    const uint32_t span = kBlock + hlen;
    const int64_t lo = (int64_t)o0 - hlen;
    if (lo >= 0 && lo + span <= n) {
        constexpr uint32_t kU = 2;
        for (uint32_t t0 = tid; t0 < span; t0 += kBlock * kU) {
            short2 v[kU];
#pragma unroll
            for (uint32_t u = 0; u < kU; ++u)
                v[u] = in[lo + min(t0 + u * kBlock, span - 1)];
#pragma unroll
            for (uint32_t u = 0; u < kU; ++u)
                if (t0 + u * kBlock < span)
                    xs[t0 + u * kBlock] = sample_f32(v[u]);
        }
    } else {
        for (uint32_t t = tid; t < span; t += kBlock)
            xs[t] = sample_at(in, n, hlen, hist_in, lo + t);
    }
    __syncthreads();
    const ctaps_ptr h = (ctaps_ptr)(const float *)taps;
    const float2 *xw = xs + hlen + tid;
    const float2 acc = kReal && lo >= 0 ? seq_sum<true>(xw, h, m) : seq_sum<false>(xw, h, m);
    if (o0 + tid < n)
        sample_put(out + o0 + tid, acc);
}

size_t seq_lds(uint32_t m) { return (size_t)(kBlock + m - 1) * sizeof(float2); }

// ---------------------------------------------------------------------------
// Float samples through filters too long for the matrix form's LDS (above 3800
// taps): one output a thread at a time, input window in LDS.
// ---------------------------------------------------------------------------
constexpr uint32_t kLongTile = 2048;

size_t long_lds(uint32_t m) { return (size_t)(kLongTile + m - 1) * sizeof(float2); }

__global__ __launch_bounds__(kBlock) void fir_kernel(const float2 *__restrict__ in, uint32_t n,
                                                     const float2 *__restrict__ taps, uint32_t m,
                                                     const float2 *__restrict__ hist_in,
                                                     float2 *__restrict__ hist_out, float2 *__restrict__ out)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const uint32_t hlen = m - 1;
    if (blockIdx.x == 0)
        carry_history(in, n, hlen, hist_in, hist_out);
    const uint32_t o0 = blockIdx.x * kLongTile;
    const uint32_t nt = min(kLongTile, n - o0);
    float2 *xs = reinterpret_cast<float2 *>(smem);
    const int64_t lo = (int64_t)o0 - hlen;
    for (uint32_t t = threadIdx.x; t < nt + hlen; t += kBlock) {
        const int64_t i = lo + t;
        xs[t] = i >= 0 ? in[i] : hist_in[hlen + i];
    }
    __syncthreads();
    for (uint32_t q = threadIdx.x; q < nt; q += kBlock) {
        const float2 *xw = xs + q + hlen;  // xw[-k] = x[o0 + q - k]
        float2 acc = make_float2(0.f, 0.f);
        for (uint32_t k = 0; k < m; ++k) {
            const float2 x = xw[-(int32_t)k];
            const float2 h = taps[k];
            // complex<float> product added to the accumulator, reference order
            acc.x += x.x * h.x - x.y * h.y;
            acc.y += x.x * h.y + x.y * h.x;
        }
        out[o0 + q] = acc;
    }
}

}  // namespace

template <typename TI, typename TO>
hipError_t launch_fir(const TI *in, uint32_t n, const float2 *taps, uint32_t m, bool real, const float2 *hist_in,
                      float2 *hist_out, TO *out, hipStream_t s)
{
    if (long_lds(m) > kLdsMax)  // 6145 taps at most, whatever the sample type
        return hipErrorInvalidValue;
    if constexpr (std::is_same<TO, short2>::value) {
        const dim3 grid((n + kBlock - 1) / kBlock);
        if (real)
            hipLaunchKernelGGL(fir_seq_kernel<true>, grid, dim3(kBlock), seq_lds(m), s, in, n, taps, m, hist_in,
                               hist_out, out);
        else
            hipLaunchKernelGGL(fir_seq_kernel<false>, grid, dim3(kBlock), seq_lds(m), s, in, n, taps, m, hist_in,
                               hist_out, out);
    } else {
        const uint32_t kp = (m + 15 + 15) / 16 * 16;
        // The split form while its blocks of 256 outputs are at most two a
        // CU: 129 taps take 3.8 us against 6.1 on 4096 to 65536 samples, 6.7
        // against 6.5 on 2^18, 18.9 against 14.4 on 10^6 (each block stages
        // the taps and m samples more than its outputs). Beyond that only for
        // filters whose 1024-output window exceeds the LDS.
        const bool whole = mfma_lds(false, kp) <= kLdsMax, split = mfma_lds(true, kp) <= kLdsMax;
        if (split && (n <= (1u << 17) || !whole))
            return launch_mfma<true>(in, n, taps, m, kp, real, hist_in, hist_out, out, s);
        if (whole)
            return launch_mfma<false>(in, n, taps, m, kp, real, hist_in, hist_out, out, s);
        hipLaunchKernelGGL(fir_kernel, dim3((n + kLongTile - 1) / kLongTile), dim3(kBlock), long_lds(m), s, in, n,
                           taps, m, hist_in, hist_out, out);
    }
    return hipGetLastError();
}
template hipError_t launch_fir<float2, float2>(const float2 *, uint32_t, const float2 *, uint32_t, bool,
                                               const float2 *, float2 *, float2 *, hipStream_t);
template hipError_t launch_fir<short2, short2>(const short2 *, uint32_t, const float2 *, uint32_t, bool,
                                               const float2 *, float2 *, short2 *, hipStream_t);

}  // namespace fdsp
