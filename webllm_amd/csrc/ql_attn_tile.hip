// Attention of many query rows over the KV cache (prefill: ql_attention_decode with M rows) on the
// matrix cores: the tiled form of attn_kernel (ql_attn.hip), which gives every query row a workgroup
// of its own and re-reads that row's keys.
//
// fp32 in, fp32 out, fp32-grade throughout: every operand enters as two fp16 parts, x 2^s = hi + lo
// (about 22 bits), and a product is lo.hi + hi.lo + hi.hi in fp32 on v_mfma_f32_16x16x32_f16, three of
// which cost 3/16 of the fp32 MFMA's time.
//
// 1. attn_image_kernel splits K and V once, per kv head and block of 64 keys, into the fragments the
//    MFMAs read. K has one exponent per block, V one per block and column d, q one per row. It notes blocks
//    that two parts cannot hold (below).
// 2. attn_tile_kernel: a workgroup has 128 (query row, head) pairs of one kv head, ordered row-major so
//    that their causal limits are close; wave w has 32. Scores are computed transposed, S^T = K Q^T
//    (lane = query column, registers = keys), so that after the exponential a lane already holds the
//    B fragment of O^T = V^T P^T for the keys {4g .. 4g+3} of each 16; V's image has its keys in that
//    order and P never leaves its registers. Per block: K from LDS while V's loads are in flight, then
//    V from LDS while the next K's are, two barriers. Running max and sums in fp32 as in attn_kernel;
//    P's parts are taken of 2^14 P (fp16's range), after the exponential: 14 added to its argument
//    would round away the bits that make it exact. A block's P.V starts
//    from zero and is added to the fp32 output by the VALU, so the matrix unit never carries the long sum.
// 3. Where the row blocks do not fill the chip the keys are split over workgroups and
//    attn_merge_kernel adds the splits.
//
// What bounds it: per block and wave 192 MFMAs, 64 KB of LDS reads and the softmax's vector work (some
// 400 instructions), which overlap only as far as the CU's two workgroups are in different phases. 28 / 4
// heads of 128, 1024 rows after 1024 keys: images 9 us, tiles 95 us (760 TFLOP/s of fp16 products; matrix cores
// 34 % busy, VALU 35 %, LDS 19 % without a conflict; a SIMD's two waves are ready but not issued in 42 % of
// their cycles), merge 9 us; attn_kernel took 630 us.
//
// What two parts cannot hold. A part pair is off by up to 2^-39 of its exponent's range beside its own
// 2^-23, so a value far below another under the same exponent loses bits that fp32 sums keep; and P, a pair
// below 1, loses them where it weighs V far above the other keys'. An infinity or NaN makes 0 * V a NaN for
// rows that must not see the key. A workgroup that meets any of this does its blocks in fp32 from q, K and V
// themselves (tile_f32):
//   a block of K or V that is not finite;
//   a key of K with kFew or more values below kSpan times its block's largest, zeros aside, a column of V below
//   kSpan times its own, a row of q below kSpan times its own;
//   V's largest values of two blocks that the rows see further apart than 1 / kSpan.
// At 2^-16 what is lost is as small as the rounding of an fp32 product. Normally distributed values come that far
// below the largest about once in 20000, three of a key's or column's 64 or 128 hardly ever; looking for
// them costs the images 0.5 us.
#include <algorithm>

#include "ql_device.h"
#include "ql_digits.h"
#include "ql_internal.h"

namespace ql {

namespace {

constexpr int kBlk = 64;                 // keys per block
constexpr int kRows = 128;               // (row, head) pairs per workgroup
constexpr int kWorkgroups = 512;         // two per CU
constexpr float kPScale = 16384.f;       // P enters the MFMA times this, V's factors carry its inverse
constexpr int kSpanLog2 = 16;            // values below 2^-16 of their exponent's largest
constexpr float kSpan = 1.f / (1 << kSpanLog2);
constexpr int kFew = 3;                  // so many of them: fp32
constexpr float kMaxFinite = 3.4028235e38f;
constexpr uint32_t kForFp32 = 1u << 31;

__device__ __forceinline__ float ex2(float x) { return __builtin_amdgcn_exp2f(x); }

// s with |mx| 2^s in [2^14, 2^15); 0 for zero
__device__ __forceinline__ int shift_of(float mx) { return mx > 0.f && mx <= kMaxFinite ? 14 - ilogbf(mx) : 0; }

__device__ __forceinline__ void split8(const float (&x)[8], f16x8& hi, f16x8& lo)
{
#pragma unroll
    for (int e = 0; e < 8; e++) {
        hi[e] = (_Float16)x[e];
        lo[e] = (_Float16)(x[e] - (float)hi[e]);
    }
}

// How many of the N values x(0), x(1), ... lie below mx 2^-kSpanLog2, zeros aside (looked at only where there is one).
template <int N, typename F>
__device__ __forceinline__ int count_small(F x, float mx)
{
    const float t = mx * kSpan;
    int n = 0;
#pragma unroll
    for (int i = 0; i < N; i++) n += fabsf(x(i)) < t;
    if (n) {
        n = 0;
#pragma unroll
        for (int i = 0; i < N; i++) n += fabsf(x(i)) < t && x(i) != 0.f;
    }
    return n;
}

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

struct AttnTile {
    const float *q, *k, *v;
    float *out, *ws;                     // ws: key-split partials, as attn_kernel's
    u32x4 *kimg, *vimg;                  // [KV][blocks][16 D units]
    float *ksc, *vsc;                    // [KV][blocks]: 2^-s; [KV][blocks][D]: 2^-s / kPScale
    uint32_t* note;                      // [KV][blocks][2], K and V: bit 31 the block is for fp32; V: its largest
                                         // value's exponent e as e << 16 | 255 - e (0: none)
    uint32_t* qnote;                     // [KV][rows]: a row tile of q is for fp32
    int M, H, KV, G, past, T, blocks, rows, nsplit;
    float scale;
};

// blockIdx: (block, kv head, 0: K, 1: V, 2: a row tile of q)
template <int ND>
__global__ __launch_bounds__(256) void attn_image_kernel(const AttnTile a)
{
    constexpr int D = 16 * ND, NK = D / 32, LD = D + 1;
    __shared__ float tile[kBlk * LD];
    __shared__ float red[256];
    const int b = blockIdx.x, kv = blockIdx.y, tid = threadIdx.x;
    if (blockIdx.z == 2) {                               // q is only looked at, two threads a row
        const int r = min(b * kRows + (tid >> 1), a.M * a.G - 1), m = r / a.G;
        if (b * kRows >= a.M * a.G) return;
        const f32x4* q = reinterpret_cast<const f32x4*>(a.q + ((size_t)m * a.H + kv * a.G + (r - m * a.G)) * D) + (tid & 1);
        f32x4 x[D / 8];
        float mx = 0.f;
#pragma unroll
        for (int i = 0; i < D / 8; i++) {
            x[i] = ld_global(q + 2 * i);
#pragma unroll
            for (int e = 0; e < 4; e++) mx = fmaxf(mx, fabsf(x[i][e]));
        }
        mx = fmaxf(mx, __shfl_xor(mx, 1));
        int n = count_small<D / 2>([&](int i) { return x[i >> 2][i & 3]; }, mx);
        n += __shfl_xor(n, 1);
        const bool wide = __syncthreads_or(n >= kFew);
        if (tid == 0) a.qnote[(size_t)kv * a.rows + b] = wide;
        return;
    }
    if (b >= a.blocks) return;
    const bool isv = blockIdx.z;
    const int row_len = a.KV * D;
    const float* src = (isv ? a.v : a.k) + (size_t)kv * D;
    bool fin = true;
    for (int i = tid; i < kBlk * (D / 4); i += 256) {
        const int r = i / (D / 4), c = i % (D / 4), key = b * kBlk + r;
        const f32x4 x = key < a.T ? ld_global(reinterpret_cast<const f32x4*>(src + (size_t)key * row_len) + c) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            tile[r * LD + 4 * c + e] = x[e];
            fin = fin && fabsf(x[e]) <= kMaxFinite;
        }
    }
    __syncthreads();
    const size_t blk = (size_t)kv * a.blocks + b;
    // the largest finite value of N in p[0], p[step], ...; they stay in x
    auto largest = [](const float* p, int step, auto& x) {
        float mx = 0.f;
#pragma unroll
        for (int i = 0; i < (int)(sizeof x / sizeof x[0]); i++) {
            x[i] = fabsf(p[i * step]);
            mx = fmaxf(mx, x[i] <= kMaxFinite ? x[i] : 0.f);
        }
        return mx;
    };
    if (!isv) {
        // four threads a key
        float x[D / 4];
        float m = largest(tile + (tid >> 2) * LD + (tid & 3), 4, x);
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) m = fmaxf(m, __shfl_xor(m, o));
        if ((tid & 63) == 0) red[tid >> 6] = m;
        __syncthreads();
        m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        int n = count_small<D / 4>([&](int i) { return x[i]; }, m);
        n += __shfl_xor(n, 1);
        n += __shfl_xor(n, 2);
        const bool wide = __syncthreads_or(!fin || n >= kFew);
        const int sh = shift_of(m);
        if (tid == 0) {
            a.note[2 * blk] = wide ? kForFp32 : 0u;
            a.ksc[blk] = ldexpf(1.f, -sh);
        }
        // unit (kt, t, part, lane (i, g)): K[16 kt + i][32 t + 8 g .. + 7]
        u32x4* dst = a.kimg + blk * (16 * D);
        for (int u = tid; u < 4 * NK * 64; u += 256) {
            const int lane = u & 63, kt_t = u >> 6, kt = kt_t / NK, t = kt_t % NK;
            const float* p = tile + (16 * kt + (lane & 15)) * LD + 32 * t + 8 * (lane >> 4);
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = ldexpf(p[e], sh);
            f16x8 hi, lo;
            split8(x, hi, lo);
            st_global(dst + kt_t * 128 + lane, __builtin_bit_cast(u32x4, hi));
            st_global(dst + kt_t * 128 + 64 + lane, __builtin_bit_cast(u32x4, lo));
        }
    } else {
        // P threads a column
        constexpr int P = 256 / D;
        float x[kBlk / P];
        float m = largest(tile + tid % P * LD + tid / P, P * LD, x);
#pragma unroll
        for (int o = 1; o < P; o <<= 1) m = fmaxf(m, __shfl_xor(m, o));
        int n = count_small<kBlk / P>([&](int i) { return x[i]; }, m);
#pragma unroll
        for (int o = 1; o < P; o <<= 1) n += __shfl_xor(n, o);
        const int sh = shift_of(m);
        if (tid % P == 0) {
            a.vsc[blk * D + tid / P] = ldexpf(1.f / kPScale, -sh);
            red[tid / P] = (float)sh;
        }
#pragma unroll
        for (int o = P; o < 64; o <<= 1) m = fmaxf(m, __shfl_xor(m, o));
        if ((tid & 63) == 0) red[D + (tid >> 6)] = m;
        const bool wide = __syncthreads_or(!fin || n >= kFew);
        if (tid == 0) {
            const uint32_t e = __builtin_bit_cast(uint32_t, fmaxf(fmaxf(red[D], red[D + 1]), fmaxf(red[D + 2], red[D + 3]))) >> 23;
            a.note[2 * blk + 1] = (wide ? kForFp32 : 0u) | (e ? e << 16 | (255u - e) : 0u);
        }
        // unit (dt, ks, part, lane (i, g)): V[32 ks + {4 g + e, 16 + 4 g + e}, e < 4][16 dt + i]
        u32x4* dst = a.vimg + blk * (16 * D);
        for (int u = tid; u < ND * 2 * 64; u += 256) {
            const int lane = u & 63, ks = (u >> 6) & 1, dt = u >> 7;
            const int c = 16 * dt + (lane & 15), r0 = 32 * ks + 4 * (lane >> 4), s = (int)red[c];
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = ldexpf(tile[(r0 + (e & 3) + (e >> 2) * 16) * LD + c], s);
            f16x8 hi, lo;
            split8(x, hi, lo);
            st_global(dst + (u >> 6) * 128 + lane, __builtin_bit_cast(u32x4, hi));
            st_global(dst + (u >> 6) * 128 + 64 + lane, __builtin_bit_cast(u32x4, lo));
        }
    }
}

// The wave's pairs as they end: lane (i, g) has pair i of each row tile, values 16 d + 4 g .. + 3, and its keys' part
// of the sum.
template <int ND>
__device__ __forceinline__ void store_tile(const AttnTile& a, int split, int w0, const size_t (&qrow)[2], const float (&mr)[2],
                                           float (&l)[2], const f32x4 (&acc)[ND][2])
{
    constexpr int D = 16 * ND;
    const int lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int mt = 0; mt < 2; mt++) {
        l[mt] += __shfl_xor(l[mt], 16);
        l[mt] += __shfl_xor(l[mt], 32);
        if (w0 + 16 * mt + i16 >= a.M * a.G) continue;
        if (a.nsplit == 1) {
            const float inv = 1.f / l[mt];
            f32x4* o = reinterpret_cast<f32x4*>(a.out + qrow[mt] * D) + g;
#pragma unroll
            for (int d = 0; d < ND; d++) st_global(o + 4 * d, f32x4{acc[d][mt][0] * inv, acc[d][mt][1] * inv, acc[d][mt][2] * inv, acc[d][mt][3] * inv});
        } else {
            const size_t slot = qrow[mt] * a.nsplit + split;
            f32x4* o = reinterpret_cast<f32x4*>(a.ws + slot * D) + g;
#pragma unroll
            for (int d = 0; d < ND; d++) st_global(o + 4 * d, acc[d][mt]);
            float* stt = a.ws + (size_t)a.M * a.H * a.nsplit * D + 2 * slot;
            if (g < 2) st_global(stt + g, g ? l[mt] : mr[mt]);
        }
    }
}

// The wave's pairs over blocks b0 .. b1 - 1 in fp32 (v_mfma_f32_16x16x4_f32), lanes and results as in the loop below;
// q, K and V as they are, no LDS, no barrier. A lane's four values of a load are four steps of the product, and
// its scores are the B operands of O^T = V^T P^T. A score is a tree of sums of four products each, added by the
// VALU: chained four long in the matrix unit they were less exact (2.24e-7 from 64 bits against 2.15e-7, 1024 rows after
// 1024 keys, 28 / 4 heads of 128; attn_kernel 2.5e-7) and no faster. All blocks there: 590 us, attn_kernel 630.
// A row takes nothing, not even 0 * V, from keys that it does not see: what is not finite in V is left out and
// added by the VALU where it is seen. K and V have images of at most 64 MiB: 32-bit offsets.
template <int ND>
__device__ __forceinline__ void tile_f32(const AttnTile& a, int kvh, int b0, int b1, int split, int w0, const int (&lim)[2],
                                         const size_t (&qrow)[2])
{
    constexpr int D = 16 * ND;
    const int lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
    const f32x4* k4 = reinterpret_cast<const f32x4*>(a.k);
    f32x4 q[2][ND], acc[ND][2];
#pragma unroll
    for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int t = 0; t < ND; t++) q[mt][t] = ld_global(reinterpret_cast<const f32x4*>(a.q + qrow[mt] * D) + 4 * t + g);
    float mr[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};
#pragma unroll
    for (int d = 0; d < ND; d++) acc[d][0] = acc[d][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int b = b0; b < b1; b++) {
        f32x4 s[4][2];
#pragma unroll
        for (int kt = 0; kt < 4; kt++) {
            const uint32_t ko = (uint32_t)(min(b * kBlk + 16 * kt + i16, a.T - 1) * a.KV + kvh) * (D / 4) + g;
            f32x4 k[ND];
#pragma unroll
            for (int t = 0; t < ND; t++) k[t] = ld_global(k4 + (ko + 4 * t));
            f32x4 part[2][5];                            // [.][i]: sums of 2^i products' results
#pragma unroll
            for (int t = 0; t < D / 4; t++) {
                f32x4 c[2];
#pragma unroll
                for (int mt = 0; mt < 2; mt++)
                    c[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[t / 4][t % 4], q[mt][t / 4][t % 4], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                int i = 0;
#pragma unroll
                for (; t >> i & 1; i++)
#pragma unroll
                    for (int mt = 0; mt < 2; mt++) c[mt] = part[mt][i] + c[mt];
#pragma unroll
                for (int mt = 0; mt < 2; mt++) (t + 1 < D / 4 ? part[mt][i] : s[kt][mt]) = c[mt];
            }
        }
#pragma unroll
        for (int mt = 0; mt < 2; mt++) {
            float bm = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < 4; kt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    s[kt][mt][r] = b * kBlk + 16 * kt + 4 * g + r > lim[mt] ? -INFINITY : s[kt][mt][r] * a.scale;
                    bm = fmaxf(bm, s[kt][mt][r]);
                }
            bm = fmaxf(bm, __shfl_xor(bm, 16));
            bm = fmaxf(bm, __shfl_xor(bm, 32));
            const float mn = fmaxf(mr[mt], bm), ref = mn == -INFINITY ? 0.f : mn, al = ex2(mr[mt] - ref);
            mr[mt] = mn;
            float sum = 0.f;
#pragma unroll
            for (int kt = 0; kt < 4; kt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    s[kt][mt][r] = ex2(s[kt][mt][r] - ref);
                    sum += s[kt][mt][r];
                }
            l[mt] = l[mt] * al + sum;
#pragma unroll
            for (int d = 0; d < ND; d++) acc[d][mt] *= al;
        }
        const int key0 = b * kBlk + 4 * g;
        bool fin = true;
#pragma unroll
        for (int d = 0; d < ND; d++) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                float v[2][4];
#pragma unroll
                for (int kt = 0; kt < 2; kt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float x = ld_global(a.v + ((uint32_t)(min(key0 + 16 * (2 * h + kt) + r, a.T - 1) * a.KV + kvh) * D + 16 * d + i16));
                        const bool f = fabsf(x) <= kMaxFinite;
                        v[kt][r] = f ? x : 0.f;
                        fin = fin && f;
                    }
                f32x4 c[2];
#pragma unroll
                for (int mt = 0; mt < 2; mt++) c[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kt = 0; kt < 2; kt++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int mt = 0; mt < 2; mt++) c[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[kt][r], s[2 * h + kt][mt][r], c[mt], 0, 0, 0);
#pragma unroll
                for (int mt = 0; mt < 2; mt++) acc[d][mt] += c[mt];
            }
        }
        if (__all(fin)) continue;
#pragma unroll
        for (int kt = 0; kt < 4; kt++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll 1
                for (int kg = 0; kg < 4; kg++) {
                    const int key = b * kBlk + 16 * kt + 4 * kg + r;
                    const uint32_t vo = (uint32_t)(min(key, a.T - 1) * a.KV + kvh) * (D / 4) + g;
                    float p[2];
#pragma unroll
                    for (int mt = 0; mt < 2; mt++) p[mt] = __shfl(s[kt][mt][r], 16 * kg + i16);
#pragma unroll
                    for (int d = 0; d < ND; d++) {
                        f32x4 x = ld_global(reinterpret_cast<const f32x4*>(a.v) + (vo + 4 * d));
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            if (fabsf(x[e]) <= kMaxFinite) x[e] = 0.f;
#pragma unroll
                            for (int mt = 0; mt < 2; mt++) acc[d][mt][e] = fmaf(p[mt], key > lim[mt] ? 0.f : x[e], acc[d][mt][e]);
                        }
                    }
                }
    }
    store_tile<ND>(a, split, w0, qrow, mr, l, acc);
}

template <int ND>
__global__ __launch_bounds__(256, 2) void attn_tile_kernel(const AttnTile a)
{
    constexpr int D = 16 * ND, NK = D / 32;
    constexpr int U = 16 * D;                            // 16-byte units of a block's K or V image
    constexpr int TU = U / 256;
    __shared__ u32x4 kb[U], vb[U];
    __shared__ float vscale[D];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15, g = lane >> 4;
    // the longest causal ranges first
    const int rb = gridDim.x - 1 - blockIdx.x, split = blockIdx.y, kvh = blockIdx.z;
    const int R = a.M * a.G;
    const int kend = a.past + (min(rb * kRows + kRows, R) - 1) / a.G + 1;
    const int nblk = (kend + kBlk - 1) / kBlk, per = (nblk + a.nsplit - 1) / a.nsplit;
    const int b0 = min(nblk, split * per), b1 = min(nblk, b0 + per);
    const int w0 = rb * kRows + wave * 32;               // the wave's first pair
    const size_t blk0 = (size_t)kvh * a.blocks;
    u32x4 st[TU];
    auto load = [&](const u32x4* img, int b) {           // from an address that the whole wave shares
        const char* p = reinterpret_cast<const char*>(img + (blk0 + b) * U);
#pragma unroll
        for (int u = 0; u < TU; u++) st[u] = ld_global(reinterpret_cast<const u32x4*>(p + u * 4096 + (uint32_t)tid * 16u));
    };
    auto put = [&](u32x4* lds) {
#pragma unroll
        for (int u = 0; u < TU; u++) lds[u * 256 + tid] = st[u];
    };
    if (b0 < b1) load(a.kimg, b0);
    // whether this work is for fp32: its rows of q, K and V of its blocks, V's range over all that its rows see
    bool wide = a.qnote[(size_t)kvh * a.rows + rb] != 0u;
    u16x2 range = {0, 0};
    for (int b = lane; b < nblk; b += 64) {
        const u32x2 w = ld_global(reinterpret_cast<const u32x2*>(a.note) + blk0 + b);
        wide |= b >= b0 && b < b1 && ((w.x | w.y) & kForFp32);
        range = __builtin_elementwise_max(range, __builtin_bit_cast(u16x2, w.y & ~kForFp32));
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
        range = __builtin_elementwise_max(range, __builtin_bit_cast(u16x2, __shfl_xor(__builtin_bit_cast(uint32_t, range), o)));
    wide |= range.x + range.y > 255 + kSpanLog2;

    // Q fragments and exponents: lane (i, g) holds row i's values 32 t + 8 g .. + 7
    f16x8 qh[2][NK], ql[2][NK];
    float qs[2];
    int lim[2];                                          // last visible key
    size_t qrow[2];
#pragma unroll
    for (int mt = 0; mt < 2; mt++) {
        const int r = min(w0 + 16 * mt + i16, R - 1), m = r / a.G;
        lim[mt] = a.past + m;
        qrow[mt] = (size_t)m * a.H + kvh * a.G + (r - m * a.G);
        const f32x4* p = reinterpret_cast<const f32x4*>(a.q + qrow[mt] * D) + 2 * g;
        f32x4 x[NK][2];
        float mx = 0.f;
#pragma unroll
        for (int t = 0; t < NK; t++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                x[t][h] = ld_global(p + 8 * t + h);
#pragma unroll
                for (int e = 0; e < 4; e++) mx = fmaxf(mx, fabsf(x[t][h][e]));
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const int sh = shift_of(mx);
        qs[mt] = ldexpf(a.scale, -sh);
#pragma unroll
        for (int t = 0; t < NK; t++) {
            float y[8];
#pragma unroll
            for (int e = 0; e < 8; e++) y[e] = ldexpf(x[t][e >> 2][e & 3], sh);
            split8(y, qh[mt][t], ql[mt][t]);
        }
    }
    if (__any(wide)) {                                   // the same for every wave of the workgroup
        tile_f32<ND>(a, kvh, b0, b1, split, w0, lim, qrow);
        __builtin_amdgcn_endpgm();
    }
    if (b0 < b1) put(kb);
    const int free_key = a.past + min(w0, R - 1) / a.G;  // keys up to here are visible to the whole wave

    f32x4 acc[ND][2];
    float mr[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};
#pragma unroll
    for (int d = 0; d < ND; d++) acc[d][0] = acc[d][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int b = b0; b < b1; b++) {
        __syncthreads();                                 // K of block b is in LDS; V's buffer is free
        load(a.vimg, b);
        const float vs1 = ld_global(a.vsc + (blk0 + b) * D + (tid & (D - 1)));
        const float ks = ld_global(a.ksc + blk0 + b);
        f32x4 s[4][2];
#pragma unroll
        for (int kt = 0; kt < 4; kt++) {
            s[kt][0] = s[kt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
            // the small products first: the sum takes its full size, and the roundings that go with it,
            // only in the last NK
            f16x8 kh[NK];
#pragma unroll
            for (int t = 0; t < NK; t++) {
                const u32x4* p = kb + (kt * NK + t) * 128 + lane;
                kh[t] = __builtin_bit_cast(f16x8, p[0]);
                const f16x8 kl = __builtin_bit_cast(f16x8, p[64]);
#pragma unroll
                for (int mt = 0; mt < 2; mt++) s[kt][mt] = mfma_16x16x32_f16(kl, qh[mt][t], s[kt][mt]);
#pragma unroll
                for (int mt = 0; mt < 2; mt++) s[kt][mt] = mfma_16x16x32_f16(kh[t], ql[mt][t], s[kt][mt]);
            }
#pragma unroll
            for (int mt = 0; mt < 2; mt++) {
                f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int t = 0; t < NK / 2; t++) s[kt][mt] = mfma_16x16x32_f16(kh[t], qh[mt][t], s[kt][mt]);
#pragma unroll
                for (int t = NK / 2; t < NK; t++) z = mfma_16x16x32_f16(kh[t], qh[mt][t], z);
                s[kt][mt] += z;
            }
        }
        if (b * kBlk + kBlk - 1 > free_key)
#pragma unroll
            for (int kt = 0; kt < 4; kt++)
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int mt = 0; mt < 2; mt++)
                        if (b * kBlk + 16 * kt + 4 * g + r > lim[mt]) s[kt][mt][r] = -INFINITY;
        f16x8 ph[2][2], pl[2][2];                        // [step of 32 keys][row tile]
        float al[2];
#pragma unroll
        for (int mt = 0; mt < 2; mt++) {
            const float f = fmaxf(qs[mt] * ks, 1.17549435e-38f);
            float bm = s[0][mt][0];
#pragma unroll
            for (int kt = 0; kt < 4; kt++)
#pragma unroll
                for (int r = 0; r < 4; r++) bm = fmaxf(bm, s[kt][mt][r]);
            bm = fmaxf(bm, __shfl_xor(bm, 16));
            bm = fmaxf(bm, __shfl_xor(bm, 32));
            const float mn = fmaxf(mr[mt], bm * f);
            const float ref = mn == -INFINITY ? 0.f : mn;         // no visible key yet: every P is 0
            al[mt] = ex2(mr[mt] - ref);
            mr[mt] = mn;
            float sum = 0.f;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                float p[8];
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    p[e] = ex2(fmaf(s[2 * h + (e >> 2)][mt][e & 3], f, -ref));
                    sum += p[e];
                    p[e] *= kPScale;
                }
                split8(p, ph[h][mt], pl[h][mt]);
            }
            l[mt] = l[mt] * al[mt] + sum;
        }
        if (__any(al[0] != 1.f || al[1] != 1.f))
#pragma unroll
            for (int d = 0; d < ND; d++)
#pragma unroll
                for (int mt = 0; mt < 2; mt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[d][mt][r] *= al[mt];
        put(vb);
        if (tid < D) vscale[tid] = vs1;
        __syncthreads();                                 // V of block b is in LDS; K's buffer is free
        load(a.kimg, min(b + 1, b1 - 1));
#pragma unroll
        for (int d = 0; d < ND; d++) {
            const u32x4* p = vb + d * 256 + lane;
            const f16x8 vh0 = __builtin_bit_cast(f16x8, p[0]), vl0 = __builtin_bit_cast(f16x8, p[64]);
            const f16x8 vh1 = __builtin_bit_cast(f16x8, p[128]), vl1 = __builtin_bit_cast(f16x8, p[192]);
            const f32x4 sc = *reinterpret_cast<const f32x4*>(vscale + 16 * d + 4 * g);
            f32x4 o[2];
#pragma unroll
            for (int mt = 0; mt < 2; mt++) o[mt] = mfma_16x16x32_f16(vl0, ph[0][mt], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int mt = 0; mt < 2; mt++) o[mt] = mfma_16x16x32_f16(vl1, ph[1][mt], o[mt]);
#pragma unroll
            for (int mt = 0; mt < 2; mt++) o[mt] = mfma_16x16x32_f16(vh0, pl[0][mt], o[mt]);
#pragma unroll
            for (int mt = 0; mt < 2; mt++) o[mt] = mfma_16x16x32_f16(vh1, pl[1][mt], o[mt]);
#pragma unroll
            for (int mt = 0; mt < 2; mt++) o[mt] = mfma_16x16x32_f16(vh0, ph[0][mt], o[mt]);
#pragma unroll
            for (int mt = 0; mt < 2; mt++) o[mt] = mfma_16x16x32_f16(vh1, ph[1][mt], o[mt]);
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[d][mt][r] = fmaf(o[mt][r], sc[r], acc[d][mt][r]);
        }
        put(kb);
    }

    store_tile<ND>(a, split, w0, qrow, mr, l, acc);
}

// out = sum_i acc_i 2^(m_i - m) / sum_i l_i 2^(m_i - m) over the splits i in order, four values a thread
__global__ __launch_bounds__(256) void attn_merge_kernel(const float* ws, float* out, int rows, int D, int S)
{
    const int i = blockIdx.x * 256 + threadIdx.x, nc = D / 4;
    if (i >= rows * nc) return;
    const int row = i / nc, c = i - row * nc;
    const f32x2* st = reinterpret_cast<const f32x2*>(ws + (size_t)rows * S * D) + (size_t)row * S;
    const f32x4* src = reinterpret_cast<const f32x4*>(ws + (size_t)row * S * D) + c;
    float m = -INFINITY, l = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < S; k++) m = fmaxf(m, ld_global(st + k).x);
#pragma unroll 4
    for (int k = 0; k < S; k++) {
        const f32x2 ml = ld_global(st + k);
        const f32x4 v = ld_global(src + (size_t)k * nc);
        const float w = ml.x == -INFINITY ? 0.f : ex2(ml.x - m);
        l = fmaf(ml.y, w, l);
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = fmaf(v[e], w, o[e]);
    }
    const float inv = 1.f / l;
    st_global(reinterpret_cast<f32x4*>(out + (size_t)row * D) + c, f32x4{o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv});
}

// bytes of the images, exponents and notes, 256-byte aligned pieces
size_t image_bytes(int KV, int D, int blocks, int rows)
{
    const size_t n = (size_t)KV * blocks;
    return 2 * n * kBlk * D * 4 + ((n * D * 4 + 255) & ~(size_t)255) + ((n * 4 + 255) & ~(size_t)255) + ((n * 8 + 255) & ~(size_t)255) +
           (((size_t)KV * rows * 4 + 255) & ~(size_t)255);
}

}  // namespace

// The line between this form and attn_kernel is where both its time and its error against 64 bits are the
// smaller ones: at least 96 rows that see about 900 keys each on average in every key split that attn_kernel
// would take (a: planned; with few rows x heads it splits, and its chains of fp32 sums are then short). Measured (28 / 4
// heads of 128; us and relative error, attn_kernel -> this): 1024 rows after 1024 keys 630 -> 110, 2.5e-7 ->
// 2.1e-7; 128 after 1500 102 -> 41, 2.5e-7 -> 2.1e-7; 1024 after 400 417 -> 90, 2.15e-7 -> 2.0e-7. Beyond the
// line it is mostly still faster but less exact: 1024 rows after none 247 -> 65 us but 1.4e-7 -> 1.5e-7; 14 / 2 heads
// of 64, 96 rows after 912 (three splits) 1.78e-7 -> 1.89e-7, 160 after 880 (two) 1.97e-7 -> 1.99e-7; 28 / 4 of
// 128, 96 after 848 (two) 57 -> 32 us but 1.85e-7 -> 1.89e-7.
bool attention_tile_ok(const AttnArgs& a, size_t ws_bytes, int* nsplit, uint64_t* used)
{
    if (a.D != 64 && a.D != 128) return false;
    if (a.M < 96 || a.past + a.M / 2 < 896 * a.nsplit) return false;
    const int blocks = (a.past + a.M + kBlk - 1) / kBlk;
    const int rows = (a.M * a.G + kRows - 1) / kRows;
    const size_t img = image_bytes(a.KV, a.D, blocks, rows);
    if (img > ws_bytes) return false;                    // so many kv heads: the general kernel
    // key splits up to two workgroups a CU (1 split or 4 instead of 2 at 1024 rows: 144, 138 against 131 us
    // in an earlier form), of at least two blocks, as many as the workspace holds
    const int rb = rows * a.KV;
    int s = std::max(1, std::min(kWorkgroups / rb, (blocks + 1) / 2));
    const size_t one = (size_t)a.M * a.H * (a.D + 2) * sizeof(float);
    *nsplit = (int)std::min<size_t>(std::min(s, 128), std::max<size_t>(1, (ws_bytes - img) / one));
    *used = img + (*nsplit > 1 ? *nsplit * one : 0);
    return true;
}

hipError_t launch_attention_tile(const AttnArgs& a, void* ws, int nsplit, hipStream_t stream)
{
    AttnTile t;
    t.q = a.q;
    t.k = a.k;
    t.v = a.v;
    t.out = a.out;
    t.M = a.M;
    t.H = a.H;
    t.KV = a.KV;
    t.G = a.G;
    t.past = a.past;
    t.T = a.past + a.M;
    t.blocks = (t.T + kBlk - 1) / kBlk;
    t.nsplit = nsplit;
    t.scale = a.scale;
    const size_t n = (size_t)a.KV * t.blocks;
    char* p = static_cast<char*>(ws);
    t.kimg = reinterpret_cast<u32x4*>(p);
    p += n * kBlk * a.D * 4;
    t.vimg = reinterpret_cast<u32x4*>(p);
    p += n * kBlk * a.D * 4;
    t.vsc = reinterpret_cast<float*>(p);
    p += (n * a.D * 4 + 255) & ~(size_t)255;
    t.ksc = reinterpret_cast<float*>(p);
    p += (n * 4 + 255) & ~(size_t)255;
    t.note = reinterpret_cast<uint32_t*>(p);
    p += (n * 8 + 255) & ~(size_t)255;
    t.qnote = reinterpret_cast<uint32_t*>(p);
    t.rows = (a.M * a.G + kRows - 1) / kRows;
    p += ((size_t)a.KV * t.rows * 4 + 255) & ~(size_t)255;
    t.ws = reinterpret_cast<float*>(p);
    const dim3 ig(std::max(t.blocks, t.rows), a.KV, 3), tg(t.rows, nsplit, a.KV);
    if (a.D == 64) {
        hipLaunchKernelGGL(attn_image_kernel<4>, ig, dim3(256), 0, stream, t);
        hipLaunchKernelGGL(attn_tile_kernel<4>, tg, dim3(256), 0, stream, t);
    } else {
        hipLaunchKernelGGL(attn_image_kernel<8>, ig, dim3(256), 0, stream, t);
        hipLaunchKernelGGL(attn_tile_kernel<8>, tg, dim3(256), 0, stream, t);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || nsplit == 1) return e;
    const int rows = a.M * a.H;
    hipLaunchKernelGGL(attn_merge_kernel, dim3((rows * (a.D / 4) + 255) / 256), dim3(256), 0, stream, t.ws, a.out, rows, a.D, nsplit);
    return hipGetLastError();
}

}  // namespace ql
