// GEMM of some tens of rows over GPTQ int4 weights (single linears and batches on a short prompt):
// y[M,N] = f16(x)[M,K] * f16(W)[N,K]^T (+ bias), fp32 accumulation, W dequantized in the kernel
// bit-identically to the load-time fp16 arena, as gemm_kernel (ql_gemm.hip), for groups of a multiple
// of 128.
//
// x_rows_kernel rounds x to fp16 once, in the order of the MFMA's B fragments: unit (row tile of 16, 32-k
// step, lane (i, kq)) = x[16 tile + i][32 step + 8 kq .. + 7] in dequant order. A workgroup has 64 columns by
// 32 rows; its 8 waves take a part of K each, stream packed words and fragments through registers of
// their own (no barrier), and add up once through LDS in wave order: the scheme of ql_gemv_wave.hip with one
// fp16 part and the weights' scales in fp16. Nothing is split across workgroups, so there are no partial
// sums in memory and no launch that adds them.
//
// What bounds it: latency. A wave loads a 128-k chunk, waits and dequantizes it (about 210 vector instructions
// for 32 MFMAs of 128 k x 64 columns), so its part of K is a serial chain, 1.8 us per 1024 of K with cached
// weights and 2.2 from HBM. 77 rows of 3584 x 3584, 12.7 and 14.5 us: waves wait 57 % of their cycles, the VALU
// is busy 26 % of the launch, the matrix cores 10 %.

#include "ql_device.h"
#include "ql_digits.h"
#include "ql_internal.h"

namespace ql {

namespace {

__device__ const uint32_t kFewSymZeros = 0x77777777u;    // stored zeros of a linear without qzeros

// x [M, K] (fp32, rounded to fp16, or fp16) -> image, a unit per thread; rows up to Mp are zero
template <bool F32>
__device__ __forceinline__ void x_rows(const void* x, u32x4* img, int M, int Mp, int K)
{
    const int i = blockIdx.x * 256 + threadIdx.x, per = K / 8;
    if (i >= Mp * per) return;
    const int m = i / per, u = i - m * per;
    u32x4 r = {0u, 0u, 0u, 0u};
    if (m < M) {
        if (F32) {
            typedef float f32x8 __attribute__((ext_vector_type(8)));
            const f32x4* p = reinterpret_cast<const f32x4*>(static_cast<const float*>(x) + (size_t)m * K) + 2 * u;
            const f32x8 v = __builtin_shufflevector(ld_global(p), ld_global(p + 1), 0, 4, 1, 5, 2, 6, 3, 7);
            r = __builtin_bit_cast(u32x4, __builtin_convertvector(v, f16x8));
        } else {
            const u32x4 v = ld_global(reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(x) + (size_t)m * K) + u);
            r.x = __builtin_amdgcn_perm(v.z, v.x, 0x05040100u);   // k0 | k4
            r.y = __builtin_amdgcn_perm(v.z, v.x, 0x07060302u);   // k1 | k5
            r.z = __builtin_amdgcn_perm(v.w, v.y, 0x05040100u);   // k2 | k6
            r.w = __builtin_amdgcn_perm(v.w, v.y, 0x07060302u);   // k3 | k7
        }
    }
    st_global(img + ((size_t)(m >> 4) * (K / 32) + (u >> 2)) * 64 + (u & 3) * 16 + (m & 15), r);
}

// One input, whose few arguments are in registers when the wave starts (0.35 us less than from the struct), or several.
template <bool F32>
__global__ __launch_bounds__(256) void x_rows_kernel(const void* x, u32x4* img, int M, int Mp, int K)
{
    x_rows<F32>(x, img, M, Mp, K);
}
template <bool F32>
__global__ __launch_bounds__(256) void x_rows_batch_kernel(const XRows a, int Mp)
{
    x_rows<F32>(a.x[blockIdx.y], a.img[blockIdx.y], a.M, Mp, a.K[blockIdx.y]);
}

// Two row tiles keep four waves per SIMD (114 registers), which hide the loads: three or four, in two waves
// per SIMD, took 17.2 and 19.2 us instead of 12.7 for 77 rows of 3584 x 3584 (one: 15.0).
constexpr int MT = 2;
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void gemm_few_kernel(const FewBatch b)
{
    __shared__ f32x4 part[8][16][17];                    // a row tile of every wave: [4-column piece][row]
    // consecutive numbers share an XCD, whose L2 then has a column block's weights for every row block
    const int bid = blockIdx.x, n8 = b.wg_total / 8 * 8;
    const int wg = bid < n8 ? (bid % 8) * (n8 / 8) + bid / 8 : bid;
    int li = 0;
    while (li + 1 < b.count && wg >= b.L[li + 1].wg_begin) li++;
    const FewLinear& L = b.L[li];
    const int N = L.N, K = L.K;
    const int local = wg - L.wg_begin, mi = local % b.mb, n0 = local / b.mb * 64;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15, kq = lane >> 4;
    const int C = K / 128, c0 = wave * C / 8, nc = (wave + 1) * C / 8 - c0;   // 128-k chunks of this wave
    const int cpg = L.group / 128;

    f32x4 acc[MT][4];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < 4; t++) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (nc > 0) {
        // column n0 + 4 i + t is row i of tile t; offsets from addresses that the whole wave shares
        const int c = n0 + 4 * i16, wc = c < N ? c : 0;
        const uint32_t wo = (uint32_t)(kq * N + wc) * 4u, so = (uint32_t)wc * 2u, zo = L.qzeros ? (uint32_t)(wc >> 3) * 4u : 0u;
        const int zs = 4 * (wc & 7);
        const char* qzb = reinterpret_cast<const char*>(L.qzeros ? L.qzeros : &kFewSymZeros);
        const uint32_t zstride = L.qzeros ? (uint32_t)((N + 7) >> 3) * 4u : 0u;
        const uint32_t xo = (uint32_t)lane * 16u;
        const uint64_t tile = (uint64_t)K * 32u;         // bytes of a row tile's image
        uint32_t m0 = 0x000F000Fu, m1 = 0x00F000F0u, magic = 0x64006400u;
        asm volatile("" : "+s"(m0), "+s"(m1));
        asm volatile("" : "+v"(magic));
        for (int q = c0; q < c0 + nc; q++) {
            const char* wb = reinterpret_cast<const char*>(L.qweight) + (uint64_t)q * 64u * (uint32_t)N;
            u32x4 w[4], x[4][MT];
#pragma unroll
            for (int st = 0; st < 4; st++) w[st] = ld_global(reinterpret_cast<const u32x4*>(wb + (uint64_t)(16u * st) * (uint32_t)N + wo));
            const u32x2 sv = ld_global(reinterpret_cast<const u32x2*>(reinterpret_cast<const char*>(L.scales) + (uint64_t)(q / cpg) * 2u * (uint32_t)N + so));
            const uint32_t zv = ld_global(reinterpret_cast<const uint32_t*>(qzb + (uint64_t)(q / cpg) * zstride + zo)) >> zs;
            const char* xb = reinterpret_cast<const char*>(L.img) + (uint64_t)(mi * MT) * tile + (uint64_t)q * 4096u;
#pragma unroll
            for (int st = 0; st < 4; st++)
#pragma unroll
                for (int m = 0; m < MT; m++) x[st][m] = ld_global(reinterpret_cast<const u32x4*>(xb + m * tile + st * 1024 + xo));
            f16x2 za[4], zb[4], sc[4];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                // q - zero, exact in fp16: nibbles at bits 0..3 as 1024 + q - (1024 + zero), at bits 4..7 as
                // (1024 + 16 q) / 16 - (64 + zero)
                const uint32_t zero = ((zv >> (4 * t)) & 15u) + 1u;
                za[t] = as_f16x2((0x6400u + zero) * 0x10001u);
                zb[t] = as_f16x2((0xD400u + (zero << 4)) * 0x10001u);
                sc[t] = as_f16x2((((t < 2 ? sv.x : sv.y) >> (16 * (t & 1))) & 0xFFFFu) * 0x10001u);
            }
            const f16x2 r16 = as_f16x2(0x2C002C00u);     // 1/16
#pragma unroll
            for (int st = 0; st < 4; st++)
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const uint32_t lo = w[st][t], hi = lo >> 8;
                    const f16x2 p0 = (as_f16x2((lo & m0) | magic) - za[t]) * sc[t];
                    const f16x2 p1 = __builtin_elementwise_fma(as_f16x2((lo & m1) | magic), r16, zb[t]) * sc[t];
                    const f16x2 p2 = (as_f16x2((hi & m0) | magic) - za[t]) * sc[t];
                    const f16x2 p3 = __builtin_elementwise_fma(as_f16x2((hi & m1) | magic), r16, zb[t]) * sc[t];
                    const f16x8 wf = f16x8{p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
#pragma unroll
                    for (int m = 0; m < MT; m++) acc[m][t] = mfma_16x16x32_f16(wf, __builtin_bit_cast(f16x8, x[st][m]), acc[m][t]);
                }
        }
    }
    // acc[m][t][r]: row i16 of row tile m, column 4 (4 kq + r) + t
#pragma unroll
    for (int m = 0; m < MT; m++) {
        if (m) __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; r++) part[wave][4 * kq + r][i16] = f32x4{acc[m][0][r], acc[m][1][r], acc[m][2][r], acc[m][3][r]};
        __syncthreads();
        const int c4 = tid & 15, row = (tid >> 4) & 15, at = (mi * MT + m) * 16 + row, n = n0 + 4 * c4;
        if (tid < 256 && at < b.M && n < N) {
            f32x4 v = part[0][c4][row];
#pragma unroll
            for (int k = 1; k < 8; k++) v += part[k][c4][row];
            if (L.bias) v += ld_global(reinterpret_cast<const f32x4*>(L.bias + n));
            st_global(reinterpret_cast<f32x4*>(L.y + (size_t)at * N + n), v);
        }
    }
}

}  // namespace

uint64_t x_rows_bytes(int M, int K) { return (uint64_t)((M + 16 * MT - 1) / (16 * MT) * (16 * MT)) * K * 2; }

hipError_t launch_x_rows(const XRows& a, bool f32, hipStream_t stream)
{
    if (a.count < 1 || a.count > kMaxBatch) return hipErrorInvalidValue;
    const int Mp = (a.M + 16 * MT - 1) / (16 * MT) * (16 * MT);
    int max_k = 0;
    for (int i = 0; i < a.count; i++) max_k = a.K[i] > max_k ? a.K[i] : max_k;
    const dim3 grid(((unsigned)Mp * (max_k / 8) + 255) / 256, a.count);
    if (a.count == 1 && f32) hipLaunchKernelGGL(x_rows_kernel<true>, grid, dim3(256), 0, stream, a.x[0], a.img[0], a.M, Mp, a.K[0]);
    else if (a.count == 1) hipLaunchKernelGGL(x_rows_kernel<false>, grid, dim3(256), 0, stream, a.x[0], a.img[0], a.M, Mp, a.K[0]);
    else if (f32) hipLaunchKernelGGL(x_rows_batch_kernel<true>, grid, dim3(256), 0, stream, a, Mp);
    else hipLaunchKernelGGL(x_rows_batch_kernel<false>, grid, dim3(256), 0, stream, a, Mp);
    return hipGetLastError();
}

hipError_t launch_gemm_few(FewBatch& b, hipStream_t stream)
{
    if (b.count < 1 || b.count > kMaxBatch || b.M < 1) return hipErrorInvalidValue;
    b.mb = (b.M + 16 * MT - 1) / (16 * MT);
    b.wg_total = 0;
    for (int i = 0; i < b.count; i++) {
        b.L[i].wg_begin = b.wg_total;
        b.wg_total += (b.L[i].N + 63) / 64 * b.mb;
    }
    hipLaunchKernelGGL(gemm_few_kernel, dim3(b.wg_total), dim3(512), 0, stream, b);
    return hipGetLastError();
}

}  // namespace ql
