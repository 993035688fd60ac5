// Many-row product over fp16 weights: y[M, N] = x[M, K] . W[N, K]^T (+ bias), x and y fp32, fp32
// accumulation: the tied lm_head over the rows of a prompt (src/model/qwen.ts:488-489 with M = T),
// where the row-per-pass GEMV of ql_f16w.hip would read W once per 16 rows.
//
// Two launches. f16w_split_kernel turns x into the image the GEMM reads: per row and 64-k chunk,
// two fp16 parts per value scaled by a power of two, with s such that max|x[m][64c .. 64c + 63]| 2^s
// lies in [2^14, 2^15), hi = f16(x 2^s), lo = f16(x 2^s - hi) (about 22 bits of every value, as the
// GEMV's parts), laid out as the MFMA's B fragments, and the chunk's factor 2^-s per row.
// f16w_gemm_kernel: a workgroup of 8 waves covers BN columns of y (rows of W) by BM rows of x and walks
// K in 64-k chunks. W and the image go through registers (the chunk after next, or the next one, in
// flight) into double-buffered LDS, one barrier a chunk: an MFMA fragment of W read straight from
// memory takes 16 bytes of 16 rows per quarter wave, and the L1's line lookups then bound the launch
// (219 us at M = 256 below; 193 staged, 8 lanes reading 128 bytes of a row). W's 16-byte pieces are
// xor-swizzled by row, so neither the writes nor the fragment reads conflict. A chunk's four MFMAs per
// tile (lo, hi of two 32-k steps) start from zero and the VALU adds them into fp32 sums as
// fma(d, 2^-s, acc), so the matrix unit never carries the long sum (its chained sums are less exact):
// 1.0e-7 from the 64-bit product at K = 896 where the GEMV is 1.2e-7. Workgroups stay resident and
// their loads run on into the next tile; tiles that share columns go to one XCD at the same time, so W
// comes from HBM once and from its L2 after that.
//
// What bounds it: W from HBM up to about 64 rows. Above, at 256 rows, the matrix cores (two products per
// weight) are busy 35 % of the launch, the VALU 24 %, LDS 23 % without a conflict; the waves wait 43 % of their
// cycles, 8 a CU that meet at every chunk's barrier. 151936 x 896, against the GEMV's pass per 16 rows:
// M = 17 108 -> 58 us, M = 64 215 -> 75 us, M = 256 814 -> 193 us (722 TFLOP/s of products).
#include <algorithm>

#include "ql_device.h"
#include "ql_digits.h"
#include "ql_internal.h"

namespace ql {

namespace {

constexpr int kGcK = 64;                 // k per chunk
constexpr int kTileUnits = 256;          // 16-byte units of a (chunk, 16-row tile): 2 steps x {hi, lo} x 64 lanes
constexpr int kXcds = 8;

// bytes of the image per row of x: both parts and the factor of every chunk
size_t image_row_bytes(int K) { return (size_t)((K + kGcK - 1) / kGcK) * (kGcK * 4 + 4); }

// x rows [M, K] -> image [chunk][row tile of 16][step][part][lane][8 fp16] and factors [chunk][Mp].
// A wave takes 8 rows x one chunk: lane = 8 j + r holds row r's values 8 j .. 8 j + 7. Rows past M
// and values past K are zero.
__global__ __launch_bounds__(256) void f16w_split_kernel(const float* x, u32x4* img, float* scl, int M, int Mp, int K, int C)
{
    const int lane = threadIdx.x & 63;
    const int job = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int rows8 = Mp / 8;
    if (job >= rows8 * C) return;
    const int c = job / rows8, m = (job - c * rows8) * 8 + (lane & 7), j = lane >> 3;
    const int k = c * kGcK + 8 * j;
    f32x4 v0 = {0.f, 0.f, 0.f, 0.f}, v1 = v0;
    if (m < M && k < K) {                // K % 8 == 0: whole units
        const f32x4* src = reinterpret_cast<const f32x4*>(x + (size_t)m * K + k);
        v0 = ld_global(src);
        v1 = ld_global(src + 1);
    }
    float mx = 0.f;
#pragma unroll
    for (int e = 0; e < 4; e++) mx = fmaxf(mx, fmaxf(fabsf(v0[e]), fabsf(v1[e])));
    mx = fmaxf(mx, __shfl_xor(mx, 8));
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    // 0 for an all-zero or non-finite chunk
    const int sh = (mx > 0.f && mx <= 3.4028235e38f) ? 14 - ilogbf(mx) : 0;
    f16x8 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float s = ldexpf(e < 4 ? v0[e & 3] : v1[e & 3], sh);
        hi[e] = (_Float16)s;
        lo[e] = (_Float16)(s - (float)hi[e]);
    }
    const int t = j >> 2, g = j & 3;
    u32x4* dst = img + ((size_t)c * (Mp / 16) + (m >> 4)) * kTileUnits + t * 128 + g * 16 + (m & 15);
    st_global(dst, __builtin_bit_cast(u32x4, hi));
    st_global(dst + 64, __builtin_bit_cast(u32x4, lo));
    if (j == 0) st_global(scl + (size_t)c * Mp + m, ldexpf(1.f, -sh));
}

struct F16wGemm {
    const uint16_t* w;
    const float* bias;
    const u32x4* img;
    const float* scl;
    float* y;
    int M, N, K, C, Mp, mb, nb;          // rows (and padded), chunks, row and column blocks
};

// NT x MT tiles (16 columns x 16 rows) per wave, WN x WM waves, D chunks in flight in registers.
// KFULL: K % 64 == 0 (every unit of W lies inside its row).
template <int NT, int MT, int WN, int WM, int D, bool KFULL>
__global__ __launch_bounds__(512, 2) void f16w_gemm_kernel(const F16wGemm a)
{
    constexpr int BN = 16 * NT * WN, BM = 16 * MT * WM;
    constexpr int WU = BN / 64;                              // units of W per thread and chunk
    constexpr int XU = (BM * 16 + 511) / 512;                // units of the image
    __shared__ u32x4 ws[2][BN * 8];
    __shared__ u32x4 xs[2][BM * 16];
    __shared__ float ss[2][BM];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN, wm = wave / WN;
    const int i16 = lane & 15, g = lane >> 4;
    const int K = a.K, N = a.N, C = a.C;
    // XCD i (workgroups i, i + 8, ...) has the column blocks i, i + 8, ..., each over all row blocks
    const int xcd = blockIdx.x % kXcds, gx = gridDim.x / kXcds;
    const int nbx = (a.nb - xcd + kXcds - 1) / kXcds;        // its column blocks
    const int tiles = nbx * a.mb;
    const int first = blockIdx.x / kXcds;
    if (first >= tiles) return;
    const int njobs = ((tiles - 1 - first) / gx + 1) * C;

    // fetch cursor: the chunk fc of tile ft (past the end it stays on the last job)
    const int wr = tid >> 3, wp = tid & 7;                   // row and 16-byte piece of the thread's units
    int ft = first, fc = 0, fj = 0;
    const char* wb[WU];
    const u32x4* xb;
    const float* sb;
    auto aim = [&]() {
        const int mi = ft % a.mb, ni = ft / a.mb * kXcds + xcd;
#pragma unroll
        for (int u = 0; u < WU; u++)
            wb[u] = reinterpret_cast<const char*>(a.w + (size_t)min(ni * BN + u * 64 + wr, N - 1) * K);
        xb = a.img + (size_t)mi * (BM * 16);
        sb = a.scl + mi * BM;
    };
    aim();
    u32x4 wreg[D][WU], xreg[D][XU];
    float sreg[D];
    auto fetch = [&](int d) {
        const int k = fc * kGcK + 8 * wp;
        const uint32_t off = (uint32_t)(KFULL ? k : min(k, K - 8)) * 2u;
#pragma unroll
        for (int u = 0; u < XU; u++)
            xreg[d][u] = ld_global(xb + (size_t)fc * (a.Mp * 16) + (BM * 16 % 512 ? tid & (BM * 16 - 1) : u * 512 + tid));
        sreg[d] = ld_global(sb + (size_t)fc * a.Mp + (tid & (BM - 1)));
#pragma unroll
        for (int u = 0; u < WU; u++) wreg[d][u] = ld_global(reinterpret_cast<const u32x4*>(wb[u] + off));
        if (!KFULL && k >= K)
#pragma unroll
            for (int u = 0; u < WU; u++) wreg[d][u] = u32x4{0u, 0u, 0u, 0u};
        if (++fj < njobs && ++fc == C) {
            fc = 0;
            ft += gx;
            aim();
        }
    };
    // piece p of W's row r is unit 8 r + (p ^ (r & 7)): the 16 rows a wave reads spread over the banks
    const int wslot = wr * 8 + (wp ^ (wr & 7));
    auto stage = [&](int b, int d) {
#pragma unroll
        for (int u = 0; u < WU; u++) ws[b][u * 512 + wslot] = wreg[d][u];
#pragma unroll
        for (int u = 0; u < XU; u++)
            if (BM * 16 >= 512 || tid < BM * 16) xs[b][u * 512 + tid] = xreg[d][u];
        if (tid < BM) ss[b][tid] = sreg[d];
    };

    f32x4 acc[NT][MT];
#pragma unroll
    for (int u = 0; u < NT; u++)
#pragma unroll
        for (int m = 0; m < MT; m++) acc[u][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bool vec_store = N % 4 == 0;
    int ct = first, cc = 0;                                  // the job computed: chunk cc of tile ct
    auto compute = [&](int b) {
        f16x8 wv[NT][2];
#pragma unroll
        for (int u = 0; u < NT; u++)
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int r = (wn * NT + u) * 16 + i16;
                wv[u][t] = __builtin_bit_cast(f16x8, ws[b][r * 8 + ((4 * t + g) ^ (r & 7))]);
            }
#pragma unroll
        for (int m = 0; m < MT; m++) {
            const u32x4* xt = xs[b] + (wm * MT + m) * kTileUnits + lane;
            const f16x8 h0 = __builtin_bit_cast(f16x8, xt[0]), l0 = __builtin_bit_cast(f16x8, xt[64]);
            const f16x8 h1 = __builtin_bit_cast(f16x8, xt[128]), l1 = __builtin_bit_cast(f16x8, xt[192]);
            const float s = ss[b][(wm * MT + m) * 16 + i16];
            f32x4 p[NT];
#pragma unroll
            for (int u = 0; u < NT; u++) p[u] = mfma_16x16x32_f16(wv[u][0], l0, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int u = 0; u < NT; u++) p[u] = mfma_16x16x32_f16(wv[u][1], l1, p[u]);
#pragma unroll
            for (int u = 0; u < NT; u++) p[u] = mfma_16x16x32_f16(wv[u][0], h0, p[u]);
#pragma unroll
            for (int u = 0; u < NT; u++) p[u] = mfma_16x16x32_f16(wv[u][1], h1, p[u]);
#pragma unroll
            for (int u = 0; u < NT; u++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[u][m][r] = fmaf(p[u][r], s, acc[u][m][r]);
        }
        if (++cc < C) return;
        // lane (i, g): y[row i of each row tile][columns 4 g .. 4 g + 3 of each column tile]
        const int n0 = (ct / a.mb * kXcds + xcd) * BN + wn * NT * 16 + 4 * g;
        const int m0 = ct % a.mb * BM + wm * MT * 16 + i16;
#pragma unroll
        for (int u = 0; u < NT; u++) {
            const int n = n0 + 16 * u;
            f32x4 bv = {0.f, 0.f, 0.f, 0.f};
            if (a.bias)
#pragma unroll
                for (int r = 0; r < 4; r++) bv[r] = ld_global(a.bias + min(n + r, N - 1));
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const f32x4 v = acc[u][m] + bv;
                acc[u][m] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (m0 + 16 * m >= a.M) continue;
                float* yr = a.y + (size_t)(m0 + 16 * m) * N;
                if (vec_store && n + 3 < N) {
                    st_global(reinterpret_cast<f32x4*>(yr + n), v);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (n + r < N) st_global(yr + n + r, v[r]);
                }
            }
        }
        cc = 0;
        ct += gx;
    };

#pragma unroll
    for (int d = 0; d < D; d++) fetch(d);
    stage(0, 0);
    __syncthreads();
    for (int j0 = 0; j0 < njobs; j0 += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            if (j0 + d >= njobs) break;
            fetch(d);                                        // job j + D
            compute((j0 + d) & 1);
            stage((j0 + d + 1) & 1, (d + 1) % D);            // job j + 1
            __syncthreads();
        }
    }
}

template <int NT, int MT, int WN, int WM, int D>
void launch_tile(F16wGemm& g, int slots, hipStream_t stream)
{
    g.mb = g.Mp / (16 * MT * WM);
    g.nb = (g.N + 16 * NT * WN - 1) / (16 * NT * WN);
    // resident workgroups, in whole rounds of the XCDs; each walks its XCD's tiles
    const int per_xcd = std::min((g.nb + kXcds - 1) / kXcds * g.mb, slots / kXcds);
    const dim3 grid(kXcds * per_xcd);
    if (g.K % kGcK == 0) hipLaunchKernelGGL((f16w_gemm_kernel<NT, MT, WN, WM, D, true>), grid, dim3(512), 0, stream, g);
    else hipLaunchKernelGGL((f16w_gemm_kernel<NT, MT, WN, WM, D, false>), grid, dim3(512), 0, stream, g);
}

}  // namespace

// Rows of x whose image fits `ws_bytes`, in whole row blocks (128s, or one of 64, 32 or 16); 0: K too long.
int gemm_f16w_rows(int K, size_t ws_bytes)
{
    const size_t r = ws_bytes / image_row_bytes(K);
    return r >= 128 ? (int)std::min<size_t>(r / 128 * 128, 65536) : r >= 64 ? 64 : r >= 32 ? 32 : r >= 16 ? 16 : 0;
}

hipError_t launch_gemm_f16w(const F16wArgs& a, int cu_count, void* ws, size_t ws_bytes, hipStream_t stream)
{
    const int R = gemm_f16w_rows(a.K, ws_bytes);
    if (R < 16 || a.K % 8) return hipErrorInvalidValue;
    for (int m0 = 0; m0 < a.M; m0 += R) {
        F16wGemm g;
        g.w = a.w;
        g.bias = a.bias;
        g.M = std::min(R, a.M - m0);
        g.N = a.N;
        g.K = a.K;
        g.C = (a.K + kGcK - 1) / kGcK;
        g.y = a.y + (size_t)m0 * a.N;
        // tiles of 128 rows x 256 columns (each fragment of W feeds 8 MFMAs) where they give three CUs of
        // four one, else of up to 64 rows x 128 columns, whose smaller LDS lets 2 or 3 workgroups share a CU
        // (K = 3584, N = 32000, M = 256: 167 us on 250 tiles of the first kind, 182 us on the second)
        const bool big = g.M > 64 && R >= 128 && (size_t)((g.M + 127) / 128) * ((a.N + 255) / 256) * 4 >= (size_t)cu_count * 3;
        const int bm = big ? 128 : g.M <= 16 ? 16 : g.M <= 32 ? 32 : 64;
        g.Mp = (g.M + bm - 1) / bm * bm;
        u32x4* img = static_cast<u32x4*>(ws);
        float* scl = reinterpret_cast<float*>(img + (size_t)g.C * g.Mp * (kTileUnits / 16));
        g.img = img;
        g.scl = scl;
        const int jobs = g.Mp / 8 * g.C;
        hipLaunchKernelGGL(f16w_split_kernel, dim3((jobs + 3) / 4), dim3(256), 0, stream, a.x + (size_t)m0 * a.K, img, scl, g.M, g.Mp, g.K, g.C);
        if (bm == 16) launch_tile<1, 1, 8, 1, 2>(g, 3 * cu_count, stream);
        else if (bm == 32) launch_tile<1, 2, 8, 1, 2>(g, 2 * cu_count, stream);
        else if (bm == 64) launch_tile<1, 4, 8, 1, 2>(g, 2 * cu_count, stream);
        else launch_tile<4, 4, 4, 2, 1>(g, cu_count, stream);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace ql
