// Per-token absmax int8 activation quantiser, optionally fused with the operation
// that produces the activations (RMSNorm, relu^2(gate)*up, relu^2(gate)*up followed by
// the FFN sub-norm), and the int8 permute used by the int32 parity entry point.
// The row arithmetic lives in rt_rowquant.h (shared with the decode GEMV prologue).
//
// One workgroup per token row.  The rows that pad the tokens to the matrix kernels' row tiles are
// left as they are: a padding row's bytes reach only that row's accumulators, which no kernel
// stores.  (Zeroing them took more of the launch than the tokens' rows for few tokens: 128
// inputs of 2 tokens in 16-row tiles, 118 -> 99 us for the plan.)
#include <algorithm>

#include "rt_rowquant.h"

// every fp32 operation rounds on its own, as the reference restatement computes them
#pragma clang fp contract(off)

namespace rt {

__device__ __forceinline__ QuantProb select_quant(const QuantArgs& a, int i) { return a.dev ? a.dev[i] : a.p; }

// row m of problem P's activations in their layout (qx_blocked)
__device__ __forceinline__ QxRow qx_row(const QuantProb& P, v4u* qx, int m) {
    const int B = P.blocked;
    if (B == 0) return QxRow{qx + (size_t)m * (P.Kp >> 4), 4, 1};
    return QxRow{qx + (size_t)(m / B) * (P.Kp >> 6) * (4 * B) + m % B, 4 * B, B};
}

__global__ void __launch_bounds__(256) quant_kernel(QuantArgs a) {
    __shared__ RowSmem sm;
    const QuantProb P = select_quant(a, blockIdx.y);
    const int m = blockIdx.x;
    const int K = P.K, Kp = P.Kp, groups = Kp >> 4;
    v4u* const qx = reinterpret_cast<v4u*>(P.qx);
    const QxRow qrow = qx_row(P, qx, m);
    if (P.mode == kPermute) {  // int8 in natural order -> qx
        const int8_t* qr = P.q_in + (size_t)m * K;
        for (int g = threadIdx.x; g < groups; g += blockDim.x) {
            int q[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int k = g * 16 + e;
                q[e] = k < K ? (int)qr[k] : 0;
            }
            qrow[g] = pack_permuted(q);
        }
        if (threadIdx.x == 0 && P.sx) P.sx[m] = 1.0f;
        return;
    }
    int8_t* qn = P.q_nat ? P.q_nat + (size_t)m * K : nullptr;
    float* vo = P.v_out ? P.v_out + (size_t)m * K : nullptr;
    const float s = row_quantize<4>(P, m, qrow, qn, vo, &sm);
    if (threadIdx.x == 0 && P.sx) P.sx[m] = s;
}

// Rows without natural-order / value outputs.  Thread t of T reads float4
// i T + t, i < NV, so a wave's load is one contiguous KiB.  The four lanes of a quad hold the 16
// elements of one group; a 4 x 4 byte transpose within the quad (two DPP exchanges) gives each
// lane one dword of the permuted group, stored directly.  The rows go to the XCDs in
// contiguous ranges: the 16 rows of a block share its lines 16 bytes at a time, and dealt out
// row by row every XCD's L2 wrote back its own part of each.
// Bound by the latency of its two reductions for few rows, by memory and the f64 quotients for
// many.  Measured (launch alone, 10 inputs in rotation; before: 8 or 16 consecutive elements
// per thread, the row assembled in LDS, rows round robin): 2560 wide, plain 5 / 512 / 2048 rows
// 3.6 / 5.6 / 10.5 -> 3.3 / 4.5 / 8.0 us, RMSNorm 4.4 / 6.8 / 13.8 -> 4.4 / 5.8 / 10.6; 6912 wide,
// plain 4.0 / 8.3 / 25.9 -> 3.8 / 6.6 / 19.1, RMSNorm 5.7 / 11.0 / 33.1 -> 5.3 / 9.1 / 25.3.
template <int CTRL>
__device__ __forceinline__ unsigned quad_perm(unsigned v) {
    return (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, true);
}
template <int NV>
__global__ void __launch_bounds__(NV == 4 ? 512 : 256) quant_wide_kernel(QuantArgs a) {
    __shared__ RowSmem sm;
    const QuantProb P = select_quant(a, blockIdx.y);
    const int m = xcd_order((int)blockIdx.x, (int)gridDim.x), t = threadIdx.x, T = (int)blockDim.x, K = P.K;
    const int F4 = P.Kp >> 2;  // (K..Kp: zeros)
    const int nw = T >> 6, wave = t >> 6, lane = t & 63;
    const bool relu2 = has_relu2(P), norm = has_norm(P);
    const float* x = P.x + (size_t)m * K;
    const float* up = P.aux + (relu2 ? (size_t)m * K : 0);
    const float* nwt = norm_weight(P);
    // whole float4s where every row is 16-byte aligned, else element by element; zeros past K
    const bool vec = (K & 3) == 0 && (((uintptr_t)P.x | (uintptr_t)P.aux | (uintptr_t)P.aux2) & 15u) == 0;
    auto load_all = [&](const float* p, float (&z)[NV][4]) {
        if (vec) {
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int f = i * T + t;
                const float4 q = 4 * f < K ? reinterpret_cast<const float4*>(p)[f] : float4{0.0f, 0.0f, 0.0f, 0.0f};
                z[i][0] = q.x;
                z[i][1] = q.y;
                z[i][2] = q.z;
                z[i][3] = q.w;
            }
        } else {
#pragma unroll
            for (int i = 0; i < NV; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int k = 4 * (i * T + t) + j;
                    z[i][j] = k < K ? p[k] : 0.0f;
                }
        }
    };
    float v[NV][4];
    load_all(x, v);
    if (relu2) {
        float u[NV][4];
        load_all(up, u);
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[i][j] = v[i][j] > 0.0f ? (v[i][j] * v[i][j]) * u[i][j] : 0.0f;
    }
    if (norm) {
        float w[NV][4];  // requested before the reduction
        load_all(nwt, w);
        double ss = 0.0;
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) ss += (double)v[i][j] * (double)v[i][j];
        ss = wave_reduce63(ss, 0.0, [](double p, double q) { return p + q; });
        if (lane == 63) sm.d[wave] = ss;
        __syncthreads();
        ss = sm.d[0];
        for (int k = 1; k < nw; ++k) ss += sm.d[k];
        const float nrm = sqrtf((float)(ss / (double)K) + P.eps);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            divide_all<4>(v[i], nrm);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[i][j] = 4 * (i * T + t) + j < K ? v[i][j] * w[i][j] : 0.0f;
        }
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) amax = fmaxf(amax, fabsf(v[i][j]));
    amax = wave_reduce63(amax, 0.0f, [](float p, float q) { return fmaxf(p, q); });
    if (lane == 63) sm.f[wave] = amax;
    __syncthreads();
    amax = sm.f[0];
    for (int k = 1; k < nw; ++k) amax = fmaxf(amax, sm.f[k]);
    const float sc = amax > 0.0f ? amax / 127.0f : 1.0f;
    if (t == 0 && P.sx) P.sx[m] = sc;
    const double rs = 1.0 / (double)sc;  // as scatter_q
    v4u* const qx = reinterpret_cast<v4u*>(P.qx);
    const QxRow qrow = qx_row(P, qx, m);
    const bool odd = t & 1, high = t & 2;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        unsigned d = 0u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float f = rintf((float)((double)v[i][j] * rs));
            d |= ((unsigned)(int)fminf(fmaxf(f, -128.0f), 127.0f) & 0xffu) << (8 * j);
        }
        // byte j of lane b to byte b of lane j
        const unsigned e = quad_perm<0xB1>(d);  // lane ^ 1
        const unsigned p = __builtin_amdgcn_perm(d, e, odd ? 0x07030501u : 0x02060004u);
        const unsigned r = quad_perm<0x4E>(p);  // lane ^ 2
        const unsigned o = high ? (p & 0xFFFF0000u) | (r >> 16) : (p & 0xFFFFu) | (r << 16);
        const int f4 = i * T + t;
        if (f4 < F4) reinterpret_cast<unsigned*>(&qrow[f4 >> 2])[t & 3] = o;
    }
}

__global__ void __launch_bounds__(256) unpermute_kernel(const int8_t* __restrict__ qx, int K, int Kp, int blocked,
                                                        int8_t* __restrict__ q) {
    const int m = blockIdx.y;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= K) return;
    const int g = k >> 4, e = k & 15;  // element e of group g sits at byte 4*(e%4) + e/4
    const int B = blocked;
    const size_t group = B ? ((size_t)(m / B) * (Kp >> 6) + (g >> 2)) * (64 * B) + (m % B + B * (g & 3)) * 16
                           : (size_t)m * Kp + g * 16;
    q[(size_t)m * K + k] = qx[group + 4 * (e & 3) + (e >> 2)];
}

hipError_t launch_unpermute(const int8_t* qx, int M, int K, int Kp, int blocked, int8_t* q, hipStream_t s) {
    hipLaunchKernelGGL(unpermute_kernel, dim3((unsigned)((K + 255) / 256), (unsigned)M), dim3(256), 0, s, qx, K, Kp,
                       blocked, q);
    return hipGetLastError();
}

// quant_wide_kernel's problems: K <= 8192, a row mode (no kPermute / kAttnNorm) and no extra
// outputs; the host checks the single problem it knows of (a.dev == nullptr) or the plan's
// summary.  Widths that are no multiple of 4 and unaligned rows read element by element, still
// well ahead of quant_kernel: 2050 wide, plain 100 / 1000 rows 5.5 / 11.6 -> 3.6 / 6.2 us, RMSNorm
// 9.4 / 21.7 -> 5.0 / 9.6.
bool quant_rows_ok(const QuantProb& P) {
    return P.mode != kPermute && P.mode != kAttnNorm && !P.q_nat && !P.v_out && P.K <= 8192;
}

hipError_t launch_quant(const QuantArgs& a, hipStream_t s, int maxK) {
    if (a.U <= 0 || a.M <= 0) return hipSuccess;
    if (maxK > 0) {  // every problem passed quant_rows_ok; maxK: the largest K
        // float4s per thread: few rows want their reductions over little work per thread (2560
        // wide, RMSNorm, 5 rows: 4 / 8 / 10 a thread 4.4 / 5.4 / 6.1 us; 1024 wide 2 a thread, whose
        // two waves measured 3 % under 4's four); many rows fewer waves each (2560 wide, 2048
        // rows: 11.9 / 13.7 / 10.6, one wave a row with 10; 6912 wide 30.8 / 25.3 / 30.6), the long
        // rows from one a CU on (RMSNorm with 4 / 8, 6912 wide 128 / 300 / 768 rows 6.4 / 8.9 / 13.4
        // against 6.6 / 8.6 / 11.9; 5120 wide 300 / 768 rows 7.7 / 11.6 against 8.0 / 10.8; 4096
        // wide 6.4 / 8.4 against 8.0 / 9.4)
        const long long rows = (long long)a.M * a.U;
        const bool many = rows > 1024;
        const bool eight = (many && maxK > 2560) || (rows > 256 && maxK > 5120);
        const int NV = eight ? 8 : many && maxK > 1536 ? 10 : maxK > 1024 ? 4 : 2;
        const unsigned threads = (unsigned)round_up((round_up(maxK, kChunk) / 4 + NV - 1) / NV, 64);
        const dim3 grid((unsigned)a.M, (unsigned)a.U), block(threads);
        switch (NV) {
            case 2: hipLaunchKernelGGL((quant_wide_kernel<2>), grid, block, 0, s, a); break;
            case 4: hipLaunchKernelGGL((quant_wide_kernel<4>), grid, block, 0, s, a); break;
            case 8: hipLaunchKernelGGL((quant_wide_kernel<8>), grid, block, 0, s, a); break;
            default: hipLaunchKernelGGL((quant_wide_kernel<10>), grid, block, 0, s, a); break;
        }
        return hipGetLastError();
    }
    hipLaunchKernelGGL(quant_kernel, dim3((unsigned)a.M, (unsigned)a.U), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace rt
