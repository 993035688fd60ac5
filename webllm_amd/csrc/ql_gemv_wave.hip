// Decode product of a few rows (M <= 16) over GPTQ int4 weights of group 128:
// y[M,N] = x[M,K] . W[N,K]^T (+ bias, + res), fp32 x and y, fp32 accumulation.
//
// x comes as an image: per row and quantization group, two fp16 parts per value scaled by a power of
// two (s with max|x| 2^s in [2^14, 2^15): hi = f16(x 2^s), lo = f16(x 2^s - hi), about 22 bits of every
// value), laid out as the B fragments of v_mfma_f32_16x16x32_f16, and the factors 2^-s. Weights are
// never scaled in fp16: q - zero is a small integer, exact, so a group's product
// sum (q - z) x 2^s is one chain of MFMAs from zero, and the VALU adds it into the fp32 sums with the
// fp16 scale and the factor (one rounding: d 2^-s is exact).
//   M > 8: hi and lo are two fragments, lo first; M <= 8: one fragment, hi in columns 0..7 and lo in 8..15,
//   whose sums meet at the end.
// The image is written once (x_image_kernel: rows as they are, RMSNorm, or SiLU-mul of two) instead of
// being formed by every workgroup, which in gemv_mfma_kernel costs more than the product at M > 4.
//
// A workgroup has 16 NT columns; its 8 waves take a part of K each, stream packed words and fragments
// through registers of their own (no barrier), and add up once through LDS in wave
// order. Nothing is split across workgroups, so there are no arrival counters and no partial sums in
// memory: their round trips were most of a small linear's time.
//
// What bounds it: latency. Each wave loads a group, waits and computes, so its part of K is a serial chain
// (gemv_wave_max_k says up to which K that is the faster way); each workgroup reads the image, M <= 8 32 B, M > 8
// 64 B per k beside its 8 NT B of weights. 3584 -> 2 x 18944 at M = 8, 20 us: waves wait 74 % of their cycles,
// the VALU is busy 42 % of the launch, the matrix cores 11 %.
#include <algorithm>
#include <type_traits>

#include "ql_device.h"
#include "ql_digits.h"
#include "ql_internal.h"

namespace ql {

namespace {

__device__ const uint32_t kGwSymZeros = 0x77777777u;     // stored zeros of a linear without qzeros

__device__ __forceinline__ float silu_mul(float g, float u) { return (g / (1.0f + expf(-g))) * u; }

// Image of x [M, K] for BIG (M > 8) or not: per 32-k step, fragment units [part (BIG: hi, lo)][lane],
// lane (column c, quarter kq) = 8 values 32 step + 8 kq .. in dequant order; then factors [group][16].
// KIND 0: x as it is (fp32, or fp16 with F16); 1: RMSNorm of x with weight w; 2: silu(x) * x2.
// Rows past M are zero. KIND 1: a workgroup per row; else (row, 2048 values) each.
template <int KIND, bool F16, bool BIG>
__device__ __forceinline__ void x_image(const XImage& a)
{
    __shared__ float red[4];
    const int tid = threadIdx.x, m = blockIdx.x;
    const int U = a.K / 8;                               // units per row
    const bool live = m < a.M;
    const float* xr = static_cast<const float*>(a.x) + (size_t)m * a.K;
    const float* ur = a.x2 + (size_t)m * a.K;
    auto value = [&](int u, f32x4& p, f32x4& q) {
        p = q = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!live || u >= U) return;
        if (F16) {
            const f16x8 h = __builtin_bit_cast(f16x8, ld_global(reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.x) + (size_t)m * a.K) + u));
#pragma unroll
            for (int e = 0; e < 4; e++) {
                p[e] = (float)h[e];
                q[e] = (float)h[e + 4];
            }
            return;
        }
        p = ld_global(reinterpret_cast<const f32x4*>(xr) + 2 * u);
        q = ld_global(reinterpret_cast<const f32x4*>(xr) + 2 * u + 1);
        if (KIND == 2) {
            const f32x4 s = ld_global(reinterpret_cast<const f32x4*>(ur) + 2 * u), t = ld_global(reinterpret_cast<const f32x4*>(ur) + 2 * u + 1);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                p[e] = silu_mul(p[e], s[e]);
                q[e] = silu_mul(q[e], t[e]);
            }
        }
    };
    auto put = [&](int u, f32x4 p, f32x4 q) {            // every lane of a wave, u consecutive over it
        float mx = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) mx = fmaxf(mx, fmaxf(fabsf(p[e]), fabsf(q[e])));
        // the 16 units of a group are 16 consecutive lanes
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        if (u >= U) return;
        const int sh = (mx > 0.f && mx <= 3.4028235e38f) ? 14 - ilogbf(mx) : 0;
        typedef float f32x8 __attribute__((ext_vector_type(8)));
        const f32x8 v = __builtin_shufflevector(p, q, 0, 4, 1, 5, 2, 6, 3, 7);
        f16x8 hi, lo;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float s = ldexpf(v[e], sh);
            hi[e] = (_Float16)s;
            lo[e] = (_Float16)(s - (float)hi[e]);
        }
        const int step = u >> 2, kq = u & 3;
        u32x4* dst = a.img + (size_t)step * (BIG ? 128 : 64) + kq * 16 + m;
        st_global(dst, __builtin_bit_cast(u32x4, hi));
        st_global(dst + (BIG ? 64 : 8), __builtin_bit_cast(u32x4, lo));
        if ((u & 15) == 0) {
            float* f = a.fac + (size_t)(u >> 4) * 16 + m;
            st_global(f, ldexpf(1.f, -sh));
            if (!BIG) st_global(f + 8, ldexpf(1.f, -sh));
        }
    };
    if (KIND != 1) {
        f32x4 p, q;
        const int u = blockIdx.y * 256 + tid;
        value(u, p, q);
        put(u, p, q);
        return;
    }
    constexpr int KEEP = 2;                              // units a thread keeps: rows up to 4096 values
    f32x4 v[KEEP][2], gw[KEEP][2];                       // and their weights, loaded with them
#pragma unroll
    for (int k = 0; k < KEEP; k++) {
        const int u = min(tid + 256 * k, U - 1);
        gw[k][0] = ld_global(reinterpret_cast<const f32x4*>(a.w) + 2 * u);
        gw[k][1] = ld_global(reinterpret_cast<const f32x4*>(a.w) + 2 * u + 1);
    }
    float ss = 0.f;
    auto add = [&](const f32x4& p, const f32x4& q) {
#pragma unroll
        for (int e = 0; e < 4; e++) ss = fmaf(p[e], p[e], ss);
#pragma unroll
        for (int e = 0; e < 4; e++) ss = fmaf(q[e], q[e], ss);
    };
#pragma unroll
    for (int k = 0; k < KEEP; k++) value(tid + 256 * k, v[k][0], v[k][1]);
#pragma unroll
    for (int k = 0; k < KEEP; k++) add(v[k][0], v[k][1]);
    for (int u = tid + 256 * KEEP; u < U; u += 256) {
        f32x4 p, q;
        value(u, p, q);
        add(p, q);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    const float rstd = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)a.K + a.eps);
    auto norm = [&](int u, f32x4 p, f32x4 q, const f32x4& g, const f32x4& h) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            p[e] = p[e] * rstd * g[e];
            q[e] = q[e] * rstd * h[e];
        }
        if (!live || u >= U) p = q = f32x4{0.f, 0.f, 0.f, 0.f};
        put(u, p, q);
    };
#pragma unroll
    for (int k = 0; k < KEEP; k++)
        if (k * 256 < U) norm(tid + 256 * k, v[k][0], v[k][1], gw[k][0], gw[k][1]);
    for (int k = KEEP; k * 256 < U; k++) {
        const int u = tid + 256 * k, uu = min(u, U - 1);
        f32x4 p, q;
        value(u, p, q);
        norm(u, p, q, ld_global(reinterpret_cast<const f32x4*>(a.w) + 2 * uu), ld_global(reinterpret_cast<const f32x4*>(a.w) + 2 * uu + 1));
    }
}

// One image, or several (blockIdx.z) whose arguments take an index: 0.3 us more.
template <int KIND, bool F16, bool BIG>
__global__ __launch_bounds__(256) void x_image_kernel(const XImage a)
{
    x_image<KIND, F16, BIG>(a);
}
template <int KIND, bool F16, bool BIG>
__global__ __launch_bounds__(256) void x_image_batch_kernel(const XImageBatch b)
{
    x_image<KIND, F16, BIG>(b.im[blockIdx.z]);
}

__device__ __forceinline__ float ror8(float v)           // the value of the lane 8 columns on
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xF, 0xF, false));
}

// NT: 16-column tiles per wave; column n0 + NT i + t is tile t's row i, so a lane's words of a packed row
// are adjacent. One group's loads at a time: 16 waves per CU hide them better than a ring in fewer waves
// (two groups in flight, two waves per SIMD: 16.6 against 15.3 us at N = 18944, K = 3584, M = 8).
template <int NT, bool BIG, int W>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(W)))
void gemv_wave_kernel(const GwBatch b)
{
    static_assert(NT == 1 || NT == 4, "one word or one 16-byte load of a packed row per lane");
    constexpr int P = BIG ? 2 : 1;
    constexpr int C4 = 4 * NT;                           // 4-column pieces per workgroup
    __shared__ f32x4 part[8][C4][17];
    // consecutive numbers share an XCD: neighbours' 64-byte pieces of a packed row are one line of its L2
    const int bid = blockIdx.x, n8 = b.wg_total / 8 * 8;
    const int wg = bid < n8 ? (bid % 8) * (n8 / 8) + bid / 8 : bid;
    int li = 0;
    while (li + 1 < b.count && wg >= b.L[li + 1].wg_begin) li++;
    const GwLinear& L = b.L[li];
    const int N = L.N, K = L.K;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = (wg - L.wg_begin) * (16 * NT);
    const int i16 = lane & 15, kq = lane >> 4;
    const int G = K / 128, g0 = wave * G / 8, ng = (wave + 1) * G / 8 - g0;

    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (ng > 0) {
        // this lane's columns, as a row of the W fragments and (4-column pieces) of the results, as byte
        // offsets from addresses that are the same for the whole wave
        const int c = n0 + NT * i16, wc = c < N ? c : 0;
        const uint32_t wo = (uint32_t)(kq * N + wc) * 4u, zo = L.qzeros ? (uint32_t)(wc >> 3) * 4u : 0u;
        const int zs = 4 * (wc & 7);
        uint32_t so[NT];
#pragma unroll
        for (int q = 0; q < NT; q++) {
            const int n = n0 + 4 * NT * kq + 4 * q;
            so[q] = n < N ? (uint32_t)n * 2u : 0u;
        }
        const char* qzb = reinterpret_cast<const char*>(L.qzeros ? L.qzeros : &kGwSymZeros);
        const uint32_t zstride = L.qzeros ? (uint32_t)((N + 7) >> 3) * 4u : 0u;
        const uint32_t xo = (uint32_t)lane * 16u, fo = (uint32_t)i16 * 4u;
        uint32_t w[4][NT], z;
        u32x4 x[4][P];
        u32x2 s[NT];
        float f;
        auto load = [&](int g) {
            const char* wb = reinterpret_cast<const char*>(L.qweight) + (uint64_t)g * 64u * (uint32_t)N;
#pragma unroll
            for (int st = 0; st < 4; st++) {
                const char* p = wb + (uint64_t)(16u * st) * (uint32_t)N + wo;
                if constexpr (NT == 1) {
                    w[st][0] = ld_global(reinterpret_cast<const uint32_t*>(p));
                } else {
                    const u32x4 v = ld_global(reinterpret_cast<const u32x4*>(p));
#pragma unroll
                    for (int t = 0; t < 4; t++) w[st][t] = v[t];
                }
            }
            const char* xb = reinterpret_cast<const char*>(L.img) + (uint64_t)g * (4096u * P);
#pragma unroll
            for (int st = 0; st < 4; st++)
#pragma unroll
                for (int p = 0; p < P; p++) x[st][p] = ld_global(reinterpret_cast<const u32x4*>(xb + (st * P + p) * 1024 + xo));
            const char* sb = reinterpret_cast<const char*>(L.scales) + (uint64_t)g * 2u * (uint32_t)N;
#pragma unroll
            for (int q = 0; q < NT; q++) s[q] = ld_global(reinterpret_cast<const u32x2*>(sb + so[q]));
            z = ld_global(reinterpret_cast<const uint32_t*>(qzb + (uint64_t)g * zstride + zo));
            f = ld_global(reinterpret_cast<const float*>(reinterpret_cast<const char*>(L.fac) + (uint64_t)g * 64u + fo));
        };
        // constants of the nibble unpacking, in registers (a three-operand instruction takes no literal)
        uint32_t m0 = 0x000F000Fu, m1 = 0x00F000F0u, magic = 0x64006400u;
        asm volatile("" : "+s"(m0), "+s"(m1));
        asm volatile("" : "+v"(magic));
        auto compute = [&]() {
            f32x4 dd[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) {
                // q - zero, exact in fp16: nibbles at bits 0..3 as 1024 + q - (1024 + zero), at bits 4..7 as
                // (1024 + 16 q) / 16 - (64 + zero)
                const uint32_t zero = ((z >> (zs + 4 * t)) & 15u) + 1u;
                const f16x2 za = as_f16x2((0x6400u + zero) * 0x10001u);
                const f16x2 zb = as_f16x2((0xD400u + (zero << 4)) * 0x10001u);   // -(64 + zero): ulp 1/16
                const f16x2 r16 = as_f16x2(0x2C002C00u);                          // 1/16
                f16x8 wf[4];
#pragma unroll
                for (int st = 0; st < 4; st++) {
                    const uint32_t lo = w[st][t], hi = lo >> 8;
                    const f16x2 p0 = as_f16x2((lo & m0) | magic) - za;
                    const f16x2 p1 = __builtin_elementwise_fma(as_f16x2((lo & m1) | magic), r16, zb);
                    const f16x2 p2 = as_f16x2((hi & m0) | magic) - za;
                    const f16x2 p3 = __builtin_elementwise_fma(as_f16x2((hi & m1) | magic), r16, zb);
                    wf[st] = f16x8{p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
                }
                dd[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int p = P - 1; p >= 0; p--)
#pragma unroll
                    for (int st = 0; st < 4; st++) dd[t] = mfma_16x16x32_f16(wf[st], __builtin_bit_cast(f16x8, x[st][p]), dd[t]);
            }
            // dd[t][r]: column NT (4 kq + r) + t of the tile, value t (NT = 1: r) of the scales' piece r (0)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int q = NT == 4 ? r : 0, e = NT == 4 ? t : r;
                    const f16x2 h = as_f16x2(e < 2 ? s[q].x : s[q].y);
                    acc[t][r] = fmaf(dd[t][r] * f, (float)(e & 1 ? h.y : h.x), acc[t][r]);
                }
        };
        for (int g = 0; g < ng; g++) {
            load(g0 + g);
            compute();
        }
    }
    if (!BIG)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[t][r] += ror8(acc[t][r]);
    // 4-column pieces of row i16
#pragma unroll
    for (int q = 0; q < NT; q++) {
        if constexpr (NT == 4) part[wave][4 * kq + q][i16] = f32x4{acc[0][q], acc[1][q], acc[2][q], acc[3][q]};
        else part[wave][kq][i16] = acc[0];
    }
    __syncthreads();
    for (int u = tid; u < C4 * b.M; u += 512) {
        const int c4 = u % C4, m = u / C4, n = n0 + 4 * c4;
        if (n >= N) continue;
        f32x4 v = part[0][c4][m];
#pragma unroll
        for (int k = 1; k < 8; k++) v += part[k][c4][m];
        const size_t at = (size_t)m * N + n;
        if (L.bias) v += ld_global(reinterpret_cast<const f32x4*>(L.bias + n));
        if (L.res) v += ld_global(reinterpret_cast<const f32x4*>(L.res + at));
        st_global(reinterpret_cast<f32x4*>(L.y + at), v);
    }
}

template <int NT>
void launch_nt(const GwBatch& b, hipStream_t stream)
{
    if (b.M > 8) hipLaunchKernelGGL((gemv_wave_kernel<NT, true, 4>), dim3(b.wg_total), dim3(512), 0, stream, b);
    // more workgroups than two per CU: fewer registers, so that a third fits (592 workgroups of 3584 -> 2 x 18944
    // 22.1 -> 20.1 us, where they ran in two rounds; 296 of one of the two 14.5 -> 16.4)
    else if (NT == 4 && b.wg_total > 2 * kPlanCUs) hipLaunchKernelGGL((gemv_wave_kernel<NT, false, 5>), dim3(b.wg_total), dim3(512), 0, stream, b);
    else hipLaunchKernelGGL((gemv_wave_kernel<NT, false, 4>), dim3(b.wg_total), dim3(512), 0, stream, b);
}

}  // namespace

// fragments, then factors
uint64_t x_image_bytes(int M, int K) { return (uint64_t)K / 32 * (M > 8 ? 2048 : 1024) + (uint64_t)K / 128 * 64; }

void x_image_at(XImage* a, void* p)
{
    a->img = static_cast<decltype(a->img)>(p);
    a->fac = reinterpret_cast<float*>(static_cast<char*>(p) + (size_t)a->K / 32 * (a->M > 8 ? 2048 : 1024));
}

hipError_t launch_x_image(const XImageBatch& b, hipStream_t stream)
{
    if (b.count < 1 || b.count > kMaxBatch) return hipErrorInvalidValue;
    const int M = b.im[0].M, kind = b.im[0].kind, f16 = b.im[0].f16;
    int max_k = 0;
    for (int i = 0; i < b.count; i++) {
        if (b.im[i].M != M || b.im[i].kind != kind || b.im[i].f16 != f16) return hipErrorInvalidValue;
        max_k = std::max(max_k, b.im[i].K);
    }
    const dim3 grid(M > 8 ? 16 : 8, kind == 1 ? 1 : (max_k / 8 + 255) / 256, b.count);
    auto go = [&](auto one, auto several) {
        if (b.count == 1) hipLaunchKernelGGL(one, grid, dim3(256), 0, stream, b.im[0]);
        else hipLaunchKernelGGL(several, grid, dim3(256), 0, stream, b);
    };
    auto pick = [&](auto big) {
        constexpr bool B = decltype(big)::value;
        if (kind == 1) go(x_image_kernel<1, false, B>, x_image_batch_kernel<1, false, B>);
        else if (kind == 2) go(x_image_kernel<2, false, B>, x_image_batch_kernel<2, false, B>);
        else if (f16) go(x_image_kernel<0, true, B>, x_image_batch_kernel<0, true, B>);
        else go(x_image_kernel<0, false, B>, x_image_batch_kernel<0, false, B>);
    };
    if (M > 8) pick(std::true_type());
    else pick(std::false_type());
    return hipGetLastError();
}

bool gemv_wave_ok(int M, int N, int K, int group) { return M >= 1 && M <= 16 && N % 4 == 0 && K % 128 == 0 && group == 128; }

// 64 columns a workgroup where that leaves half the chip a workgroup, else 16, which also wins where it
// only fills part of it: measured at M = 8 (us, 16 / 64 columns; 32 lies between them) N = 3584 K = 3584
// 8.3 / 10.4, N = 4096 K = 11008 13.6 / 19.2, 2 x 4864 K = 896 8.9 / 7.2, 2 x 18944 K = 3584 24.8 / 20.7
void gemv_wave_plan(GwBatch* b, int cu_count)
{
    long n = 0;
    for (int i = 0; i < b->count; i++) n += b->L[i].N;
    b->nt = n >= 32L * cu_count ? 4 : 1;
    int wg = 0;
    for (int i = 0; i < b->count; i++) {
        b->L[i].wg_begin = wg;
        wg += (b->L[i].N + 16 * b->nt - 1) / (16 * b->nt);
    }
    b->wg_total = wg;
}

hipError_t launch_gemv_wave(const GwBatch& b, hipStream_t stream)
{
    if (b.count < 1 || b.count > kMaxBatch || b.wg_total < 1 || b.M < 1 || b.M > 16) return hipErrorInvalidValue;
    if (b.nt == 1) launch_nt<1>(b, stream);
    else launch_nt<4>(b, stream);
    return hipGetLastError();
}

}  // namespace ql
