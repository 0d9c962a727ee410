// Batched GEMM, Y[t] = W . X[t] for ntok token rows, on int8 matrix cores
// (v_mfma_i32_32x32x32_i8; lane l supplies A[l % 32][16*(l/32) .. +15] and
// B[..][l % 32], and holds C[8*(r/4) + 4*(l/32) + r%4][l % 32] in accumulator
// r).  Every sum is the exact integer of the batch-1 GEMV and passes through
// its fp32 expressions, so each row is bit-identical to vgx_gemv on that token
// (the reference's rule for a batched path, docs/prefill-batching.md:98-113).
//
// A workgroup's K groups each walk their k tiles of KS * 32 columns.  A tile's
// operands are converted once into int8 planes in LDS and shared by the
// group's waves: the activations as 256*xh + (xl - 128) + 128, the weights as
// their level (q8, t3) or, for q4, as the exact integer n*s16 + m16 (|w| <=
// 2^19) in three signed bytes.  q4 then needs no per-group work at all: its six
// byte products accumulate over the whole row, where folding a scale and a
// minimum into 16 outputs a lane for each 32 columns was the bound before (512
// x 4608 x 1024 gate 66 -> 41 us).  The 128 of the activations costs each row
// 128 * its weight sum, formed while its bytes are staged.
//
// What the design follows (measured on MI355X): a wave alone issues one
// 16-byte LDS read in 31 clocks, the CU 232 bytes a clock when each group of 16
// lanes covers the 64 banks (the piece swizzle below; by groups of 8 lanes it
// was 127), and writes 75; the next tile is converted between the current one's
// products.  Weight bytes are loaded with neighbouring lanes on neighbouring
// pieces of a row (a lane per row cost an address cycle a lane).  The epilogue
// forms each float by one fused multiply-add of the sum's two halves instead
// of a 64-bit conversion, and the gate's exponential from two tables: a wave's
// epilogue was as long as its products.
#include <algorithm>
#include <type_traits>

#include "vgx_gemm.h"

#pragma clang fp contract(off)

namespace {

// Pins loaded bytes at this point.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void keep(u32x4& x) { asm volatile("" : "+v"(x)); }

constexpr int KS = 2;  // k-steps (32 columns) of a k tile

// 16-byte piece q of LDS row r (of 32 * KS bytes) lies at q ^ swz_row(r): the 16
// rows that one step of a wave's read covers spread over all banks.
__device__ __forceinline__ int swz_row(int r) { return (r >> 2) & 3; }

__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// An offset at or past the end of every buffer (with 16 added, still an int).
constexpr int kPast = 0x7FFFFFE0;

// A buffer over the `total` bytes from p, seen from byte `from` on: reads past
// its end return zero.  Offsets inside a workgroup's rows stay 32-bit.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tail_rsrc(const void* p, size_t from, size_t total) {
    const size_t left = from < total ? total - from : 0;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(static_cast<const uint8_t*>(p) + from), 0,
                                             (int)(left < (size_t)kPast ? left : (size_t)kPast), 0x00020000);
}

// Weight tile of 32 rows from row r0 on.  Loads are not clamped: past the row
// they read the next one, past the matrix zero; columns past the group's
// range meet activations of zero.
template <int KIND>
struct WRows {
    __amdgpu_buffer_rsrc_t body, sm;
    int stride, smstride;
};

template <int KIND>
__device__ __forceinline__ WRows<KIND> w_rows(const MatDev& M, int r0, int K) {
    WRows<KIND> w;
    w.stride = KIND == VGX_Q8 ? K : KIND == VGX_Q4 ? q4_rstride(K) : t3_rstride(K);
    const int f = KIND == VGX_T3 ? r0 >> 1 : r0, nr = KIND == VGX_T3 ? (M.rows + 1) >> 1 : M.rows;
    w.body = tail_rsrc(M.body, (size_t)f * w.stride, (size_t)nr * w.stride);
    if (KIND == VGX_Q4) {
        w.smstride = (K >> 5) * 4;
        w.sm = tail_rsrc(M.sm, (size_t)f * w.smstride, (size_t)nr * w.smstride);
    }
    return w;
}

// 16 columns of one weight row, as the container holds them (t3: of its row pair).
template <int KIND>
struct WChunk {
    u32x4 q8;
    u32x2 d;
    uint32_t sm;
};

template <int KIND>
__device__ __forceinline__ void w_load(const WRows<KIND>& W, int row, int c, WChunk<KIND>& r) {
    if (KIND == VGX_Q8) {
        r.q8 = load16(W.body, row * W.stride + c);
    } else {
        r.d = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_raw_buffer_load_b64(W.body, (KIND == VGX_T3 ? row >> 1 : row) * W.stride + (c >> 1), 0, 0));
        if (KIND == VGX_Q4) r.sm = __builtin_amdgcn_raw_buffer_load_b32(W.sm, row * W.smstride + (c >> 5) * 4, 0, 0);
    }
}

template <int KIND>
__device__ __forceinline__ void w_keep(WChunk<KIND>& r) {
    if (KIND == VGX_Q8) keep(r.q8);
    else asm volatile("" : "+v"(r.d));
    if (KIND == VGX_Q4) asm volatile("" : "+v"(r.sm));
}

// The chunk as int8 operand planes (q8, t3: the level; q4: the exact integer
// weight n*s16 + m16, |w| <= 2^19, as three signed bytes
// w = 65536*w2 + 256*w1 + w0) and its weight sum.
template <int KIND>
__device__ __forceinline__ void w_ops(const WChunk<KIND>& r, int row, Op (&w)[KIND == VGX_Q4 ? 3 : 1], int& wsum) {
    if (KIND == VGX_Q4) {
        const int s = (int16_t)(r.sm & 0xFFFFu), m = (int16_t)(r.sm >> 16);
        const int mo = m + 0x8080;  // w + 0x8080: bytes 0 and 1 hold w0 + 128, w1 + 128
        uint32_t ns = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t dv = r.d[h];  // nibble j = column j
            ns = udot4(dv & 0x0F0F0F0Fu, 0x01010101u, ns);
            ns = udot4((dv >> 4) & 0x0F0F0F0Fu, 0x01010101u, ns);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                uint32_t u[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) u[j] = (uint32_t)(__mul24((int)((dv >> (16 * q + 4 * j)) & 15u), s) + mo);
                const uint32_t p01 = perm(u[1], u[0], 0x05010400u) ^ 0x80808080u;  // b0 b0 b1 b1
                const uint32_t p23 = perm(u[3], u[2], 0x05010400u) ^ 0x80808080u;
                w[0].d[2 * h + q] = perm(p23, p01, 0x05040100u);
                w[1].d[2 * h + q] = perm(p23, p01, 0x07060302u);
                w[2].d[2 * h + q] = perm(perm(u[3], u[2], 0x0c0c0602u), perm(u[1], u[0], 0x0c0c0602u), 0x05040100u);
            }
        }
        wsum = __mul24((int)ns, s) + 16 * m;
        return;
    }
    if (KIND == VGX_Q8) {
#pragma unroll
        for (int k = 0; k < 4; ++k) w[0].d[k] = r.q8[k] ^ 0x80808080u;
    } else {
        // texel: bytes 0, 1 = row 2u columns 8c..8c+7, bytes 2, 3 = row 2u+1
        const int sh = (row & 1) * 16;
        w[0].d[0] = t3_levels((r.d[0] >> sh) & 0xFFu);
        w[0].d[1] = t3_levels((r.d[0] >> (sh + 8)) & 0xFFu);
        w[0].d[2] = t3_levels((r.d[1] >> sh) & 0xFFu);
        w[0].d[3] = t3_levels((r.d[1] >> (sh + 8)) & 0xFFu);
    }
    int s = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) s = sdot4(w[0].d[k], 0x01010101u, s);
    wsum = s;
}

// q16_round with one clamp instruction (the same value for every input, NaN included).
__device__ __forceinline__ int q16_med(float v) {
    return (int)__builtin_amdgcn_fmed3f(floorf(v + 0.5f), -32768.0f, 32767.0f);
}

// gate_value * 2^0 with exp(-g/256) from two 256-entry tables of doubles,
// e[0..255] = exp(128 - i) and e[256..511] = exp(-i/256), and f = 2^(8 - hs).
// The factors and their product are each within 2^-52, and over all 65536 g no
// exp(-g/256) lies within 2^-44 of itself of a float rounding boundary, so the
// float is the one of exp in double.  The quotient: a reciprocal refined once, then
// the quotient corrected by its exact remainder (Markstein), which is the
// correctly rounded one for every g; past 2^100 the factor is cut off, where the
// product rounds to 0 all the same.
__device__ __forceinline__ float gate_value_tab(float v1, float v3, float f, const double* e) {
    const int gi = q16_med(v1);
    const float a = (float)gi * 0.00390625f;
    const float ex = fminf((float)(e[(gi >> 8) + 128] * e[256 + (gi & 255)]), 1.2676506e30f);
    const float dn = 1.0f + ex;
    float y = __builtin_amdgcn_rcpf(dn);
    y = __builtin_fmaf(__builtin_fmaf(-dn, y, 1.0f), y, y);
    const float q = a * y;
    const float r = __builtin_fmaf(__builtin_fmaf(-dn, q, a), y, q);
    return r * ((float)q16_med(v3) * 0.00390625f) * f;
}

// The widest matrix that is uploaded; the bounds of the sums below rest on it.
constexpr int kMaxCols = 32768;

// An output's exact sum: 256 * hi + lo (q8, t3; |hi|, |lo| <= 2^30 at kMaxCols
// columns), or the int64 (q4).
template <int KIND>
struct Sum {
    int hi, lo;
    __device__ __forceinline__ void add(const Sum& o) { hi += o.hi; lo += o.lo; }
    __device__ __forceinline__ float slow() const { return (float)(256LL * hi + (long long)lo); }
    // The same float by one fused multiply-add where both parts are exact
    // floats (each below 2^24); mx collects the largest part.
    __device__ __forceinline__ float fast(float& mx) const {
        const float fh = (float)hi, fl = (float)lo;
        mx = fmaxf(mx, fmaxf(fabsf(fh), fabsf(fl)));
        return __builtin_fmaf(fh, 256.0f, fl);
    }
};
template <>
struct Sum<VGX_Q4> {
    long long v;
    __device__ __forceinline__ void add(const Sum& o) { v += o.v; }
    __device__ __forceinline__ float slow() const { return (float)v; }
    // The high part is an int for every |v| < 2^55: no row reaches past 2^49
    // (kMaxCols columns of 2^15 * 2^19), and from 2^48 on it is no exact float,
    // which mx shows.
    __device__ __forceinline__ float fast(float& mx) const {
        const float fh = (float)(int)(v >> 24), fl = (float)(int)(v & 0xFFFFFF);
        mx = fmaxf(mx, fabsf(fh));
        return __builtin_fmaf(fh, 16777216.0f, fl);
    }
};

// n sums as floats, each rounded once.
template <int KIND, int N>
__device__ __forceinline__ void sums_to_float(const Sum<KIND> (&S)[N], float (&f)[N]) {
    float mx = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i) f[i] = S[i].fast(mx);
    if (__any(mx >= 16777216.0f)) {
#pragma unroll
        for (int i = 0; i < N; ++i) f[i] = S[i].slow();
    }
}

template <int KIND, int EPI, int MT, int NT, int WM, int WN, int WK>
struct Tile {
    static constexpr int threads = 64 * WM * WN * WK, gt = 64 * WM * WN;  // of the block, of a K group
    static constexpr int bm = kTile * MT * WM, bk = kTile * KS, wrows = kTile * NT * WN;
    static constexpr int rt = EPI == BEPI_GATE ? WN * NT / 2 : WN * NT;  // output row tiles
    static constexpr int planes = KIND == VGX_Q4 ? 3 : 1;
    static constexpr int px = bm * 2 * KS / gt, pw = wrows * 2 * KS / gt;  // 16-column chunks a thread stages
    static constexpr bool solo = WM * WN == 1;                // a wave stages its own operands
    static constexpr int buf = bm * bk * 2 + wrows * bk * planes;
    static constexpr int stage = buf * WK * (solo ? 1 : 2);
    // each output's sums (W1's and W3's) lie in one wave: no exchange through LDS
    static constexpr bool direct = WK == 1 && EPI == BEPI_GATE && NT == 2;
    static constexpr int red = direct ? 0 : WM * WN * WK * NT * 16 * 64 * 8;
    static constexpr int lds = (stage > red ? stage : red) + WK * wrows * 8 + (EPI == BEPI_GATE ? 4096 : 0);
    static constexpr bool ok = bm * 2 * KS % gt == 0 && wrows * 2 * KS % gt == 0 && rt * kTile * kTile * WM % threads == 0 &&
                               threads % (rt * kTile > 0 ? rt * kTile : 1) == 0 && lds <= 160 * 1024 &&
                               !(EPI == BEPI_SPLIT && WK % 2) && !(EPI == BEPI_GATE && NT == 1 && WN % 2);
};

// MT x NT: 32-token and 32-row tiles a wave (the gate: NT = 2 holds W1 and W3
// of the same rows, NT = 1 alternates them over the waves).  WM x WN waves a K
// group, WK groups (the split: half of them on each column half).
template <int KIND, int EPI, int MT, int NT, int WM, int WN, int WK>
__global__ void __launch_bounds__(64 * WM * WN * WK, WM* WN* WK <= 4 ? 2 : 1) gemm_tile_kernel(const GemmLaunch G, int ntx, int nty) {
    using T = Tile<KIND, EPI, MT, NT, WM, WN, WK>;
    constexpr int NC = KIND == VGX_Q4 ? 4 : 2;  // int32 accumulators of an output
    constexpr int BK = T::bk, BM = T::bm, RT = T::rt, NTH = T::threads;
    extern __shared__ __align__(16) unsigned char s_dyn[];
    {
        // every argument the launch reads, in scalar registers in one batch of loads
        const uint8_t* b3 = EPI == BEPI_GATE ? G.M3.body : nullptr;
        const float* w3 = EPI == BEPI_GATE ? G.M3.wsr : nullptr;
        const uint32_t* s3 = EPI == BEPI_GATE ? G.M3.sm : nullptr;
        const float p3 = EPI == BEPI_GATE ? G.M3.ps : 0.0f;
        const int hs0 = EPI == BEPI_GATE ? G.hs : 0, sp0 = EPI == BEPI_SPLIT ? G.split : 0;
        asm volatile("" ::"s"(G.M.body), "s"(G.M.wsr), "s"(G.M.sm), "s"(G.M.ps), "s"(G.M.rows), "s"(G.ntok),
                     "s"(G.cols), "s"(G.x), "s"(G.ldx), "s"(G.res), "s"(G.y), "s"(G.ldy), "s"(b3), "s"(w3), "s"(s3),
                     "s"(p3), "s"(hs0), "s"(sp0), "s"(ntx), "s"(nty));
    }
    // XCD-aware tile order: workgroup i runs on XCD i mod 8; an XCD takes every
    // token tile of its row tiles, so a weight row is fetched into one L2.
    const int id = blockIdx.x, xcd = id & 7, idx = id >> 3;
    const int bx = xcd + 8 * (idx / nty), by = idx % nty;
    if (bx >= ntx) return;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave / (WM * WN), wg = wave % (WM * WN), wm = wg / WN, wn = wg % WN;
    const int gtid = tid - wk * T::gt;
    const int half = lane >> 5, li = lane & 31;
    const int n0 = bx * RT * kTile, t0 = by * BM;
    const int K = G.cols, rows = G.M.rows;

    // this group's columns [kb, ke)
    int a0 = 0, a1 = K, gk = wk, gn = WK;
    if (EPI == BEPI_SPLIT) {
        gn = WK / 2;
        if (wk < gn) a1 = G.split;
        else { a0 = G.split; gk = wk - gn; }
    }
    const int tiles = (a1 - a0 + BK - 1) / BK;
    const int tl = tiles * gk / gn, th = tiles * (gk + 1) / gn;
    const int kb = a0 + tl * BK, ke = min(a1, a0 + th * BK);
    // k tiles this wave walks: a block of one-wave groups needs no common
    // count; otherwise the longest run of any group (a shorter one multiplies
    // zeros at its end: columns past ke are masked)
    int nt = th - tl;
    if (!T::solo) {
        const int tm = EPI == BEPI_SPLIT ? (max(G.split, K - G.split) + BK - 1) / BK : tiles;
        nt = (tm + gn - 1) / gn;
    }

    // the weight tile that chunk i of this thread's staging lies in (the
    // chunk's row / 32: one tile a wave instruction)
    WRows<KIND> wrow[T::pw];
#pragma unroll
    for (int i = 0; i < T::pw; ++i) {
        const int wt = __builtin_amdgcn_readfirstlane((gtid + T::gt * i) / (2 * KS) / kTile);
        const int rt = EPI == BEPI_GATE ? wt >> 1 : wt;
        const bool third = EPI == BEPI_GATE && (wt & 1);
        wrow[i] = w_rows<KIND>(third ? G.M3 : G.M, n0 + rt * kTile, K);
    }
    const __amdgpu_buffer_rsrc_t xrs = tail_rsrc(G.x, (size_t)t0 * G.ldx * 2, (size_t)G.ntok * G.ldx * 2);

    i32x16 acc[MT][NT][NC];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int c = 0; c < NC; ++c) acc[m][j][c] = (i32x16){};
    // the weight sum of each staged chunk's row over this thread's chunks (q8, t3: |sum| <= 128 * K)
    using WSum = typename std::conditional<KIND == VGX_Q4, long long, int>::type;
    WSum wsum[T::pw];
#pragma unroll
    for (int i = 0; i < T::pw; ++i) wsum[i] = 0;

    // the next k tile's bytes in flight (two tiles in flight were no faster)
    u32x4 xr[T::px][2];
    WChunk<KIND> wr[T::pw];
    auto load = [&](int t) {
        const int c0 = kb + t * BK;
#pragma unroll
        for (int p = 0; p < T::px; ++p) {
            const int i = gtid + T::gt * p, row = i / (2 * KS), q = i % (2 * KS);
            // a chunk past the group's columns reads past the buffer: zeros,
            // whose products cancel the chunk's part of the weight sum
            const int off = c0 + 16 * q < ke ? (row * G.ldx + c0 + 16 * q) * 2 : kPast;
            xr[p][0] = load16(xrs, off);
            xr[p][1] = load16(xrs, off + 16);
        }
#pragma unroll
        for (int p = 0; p < T::pw; ++p) {
            const int i = gtid + T::gt * p, row = i / (2 * KS) % kTile, q = i % (2 * KS);
            w_load<KIND>(wrow[p], row, c0 + 16 * q, wr[p]);
        }
    };
    // part p of staging the loaded tile: an activation chunk or a weight chunk
    auto stage = [&](int p, unsigned char* xb, bool count) {
        unsigned char* const wb = xb + BM * BK * 2;
        if (p < T::px) {
            keep(xr[p][0]);
            keep(xr[p][1]);
            const int i = gtid + T::gt * p, row = i / (2 * KS), q = i % (2 * KS);
            const uint32_t d[8] = {xr[p][0].x, xr[p][0].y, xr[p][0].z, xr[p][0].w,
                                   xr[p][1].x, xr[p][1].y, xr[p][1].z, xr[p][1].w};
            uint32_t h[4], l[4];
            planes16(d, h, l);
            unsigned char* at = xb + row * BK + ((q ^ swz_row(row)) << 4);
            *reinterpret_cast<uint4*>(at) = make_uint4(h[0], h[1], h[2], h[3]);
            *reinterpret_cast<uint4*>(at + BM * BK) =
                make_uint4(l[0] ^ 0x80808080u, l[1] ^ 0x80808080u, l[2] ^ 0x80808080u, l[3] ^ 0x80808080u);
        } else if (p < T::px + T::pw) {
            const int k = p - T::px;
            w_keep<KIND>(wr[k]);
            const int i = gtid + T::gt * k, row = i / (2 * KS), q = i % (2 * KS);
            Op w[T::planes];
            int ws;
            w_ops<KIND>(wr[k], row, w, ws);
            wsum[k] += count ? ws : 0;
            unsigned char* at = wb + row * BK + ((q ^ swz_row(row)) << 4);
#pragma unroll
            for (int c = 0; c < T::planes; ++c)
                *reinterpret_cast<uint4*>(at + c * T::wrows * BK) = make_uint4(w[c].d[0], w[c].d[1], w[c].d[2], w[c].d[3]);
        }
    };
    auto frag = [&](const unsigned char* plane, int row, int s, Op& o) {
        const uint4 v = *reinterpret_cast<const uint4*>(plane + row * BK + (((2 * s + half) ^ swz_row(row)) << 4));
        o.d[0] = v.x; o.d[1] = v.y; o.d[2] = v.z; o.d[3] = v.w;
    };
    // the tile's products; next: the next tile is staged between them (the
    // matrix cores run while the vector units convert)
    constexpr int PARTS = T::px + T::pw, SLOTS = KS * MT * NT;
    auto compute = [&](const unsigned char* xb, unsigned char* next, bool count) {
        const unsigned char* const wb = xb + BM * BK * 2;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            Op xh[MT], xl[MT], w[NT][T::planes];
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int row = (wm * MT + m) * kTile + li;
                frag(xb, row, s, xh[m]);
                frag(xb + BM * BK, row, s, xl[m]);
            }
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int c = 0; c < T::planes; ++c)
                    frag(wb + c * T::wrows * BK, (wn * NT + j) * kTile + li, s, w[j][c]);
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    if constexpr (KIND == VGX_Q4) {
                        acc[m][j][0] = mfma(xl[m], w[j][0], acc[m][j][0]);
                        acc[m][j][1] = mfma(xh[m], w[j][0], acc[m][j][1]);
                        acc[m][j][2] = mfma(xh[m], w[j][1], acc[m][j][2]);
                        acc[m][j][3] = mfma(xh[m], w[j][2], acc[m][j][3]);
                        acc[m][j][1] = mfma(xl[m], w[j][1], acc[m][j][1]);
                        acc[m][j][2] = mfma(xl[m], w[j][2], acc[m][j][2]);
                    } else {
                        acc[m][j][0] = mfma(xl[m], w[j][0], acc[m][j][0]);
                        acc[m][j][1] = mfma(xh[m], w[j][0], acc[m][j][1]);
                    }
                    if (!T::solo) {
                        const int slot = (s * NT + j) * MT + m;
#pragma unroll
                        for (int p = slot * PARTS / SLOTS; p < (slot + 1) * PARTS / SLOTS; ++p) stage(p, next, count);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
        }
    };

    unsigned char* const s_buf = s_dyn + wk * T::buf * (T::solo ? 1 : 2);
    constexpr int RED = T::stage > T::red ? T::stage : T::red;
    WSum* s_ws = reinterpret_cast<WSum*>(s_dyn + RED);  // [WK][wrows]
    double* s_e = reinterpret_cast<double*>(s_dyn + RED + WK * T::wrows * 8);
    load(0);
    if (EPI == BEPI_GATE)  // the gate's tables, while the first tile arrives
        for (int i = tid; i < 512; i += NTH) s_e[i] = exp(i < 256 ? (double)(128 - i) : (double)(256 - i) / 256.0);
    if (T::solo) {
        for (int t = 0; t < nt; ++t) {
#pragma unroll
            for (int p = 0; p < PARTS; ++p) stage(p, s_buf, true);
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            load(t + 1);
            __builtin_amdgcn_sched_barrier(0);  // (left alone, the loads sink towards their use)
            compute(s_buf, nullptr, true);
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    } else {
#pragma unroll
        for (int p = 0; p < PARTS; ++p) stage(p, s_buf, true);
        load(1);
        lds_barrier();
        auto iter = [&](int t, int par) {  // par = t & 1
            // (the tile staged past the run is not multiplied, nor its weights summed)
            compute(s_buf + par * T::buf, s_buf + (1 - par) * T::buf, t + 1 < nt);
            load(t + 2);
            __builtin_amdgcn_sched_barrier(0);  // (left alone, the loads sink towards their use)
            lds_barrier();
        };
        for (int t = 0; t < nt; t += 2) {
            iter(t, 0);
            if (t + 1 < nt) iter(t + 1, 1);
        }
    }

    // Epilogue.  The weight sums of the group's rows go through LDS first.
#pragma unroll
    for (int p = 0; p < T::pw; ++p) {
        WSum v = wsum[p];
#pragma unroll
        for (int o = 1; o < 2 * KS; o <<= 1) v += __shfl_xor(v, o, 64);
        if (gtid % (2 * KS) == 0) s_ws[wk * T::wrows + (gtid + T::gt * p) / (2 * KS)] = 128 * v;
    }
    const __amdgpu_buffer_rsrc_t rrs =  // (no residual: a buffer of no bytes reads zeros)
        tail_rsrc(G.res, (size_t)t0 * G.ldy * 2, G.res ? (size_t)G.ntok * G.ldy * 2 : 0);
    const __amdgpu_buffer_rsrc_t yrs = tail_rsrc(G.y, (size_t)t0 * G.ldy * 2, (size_t)G.ntok * G.ldy * 2);
    auto sum_of = [&](int m, int j, int r, WSum wt) {
        Sum<KIND> S;
        if constexpr (KIND == VGX_Q4) {
            S.v = (long long)acc[m][j][0][r] + 256LL * acc[m][j][1][r] + 65536LL * acc[m][j][2][r] +
                  16777216LL * acc[m][j][3][r] + wt;
        } else {
            S.hi = acc[m][j][1][r];
            S.lo = acc[m][j][0][r] + wt;
        }
        return S;
    };
    const float gf = EPI == BEPI_GATE ? ldexpf(256.0f, -G.hs) : 0.0f;

    if constexpr (T::direct) {
        // W1's sums and W3's of the same outputs are in this wave's registers
        const int o = n0 + wn * kTile + li, oc = min(o, rows - 1);
        const float sc = KIND == VGX_Q4 ? G.M.ps : G.M.wsr[oc], sc3 = KIND == VGX_Q4 ? G.M3.ps : G.M3.wsr[oc];
        __syncthreads();
        const WSum wt = s_ws[wn * NT * kTile + li], wt3 = s_ws[(wn * NT + 1) * kTile + li];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            float v[16], v3[16];
            Sum<KIND> S[16], S3[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                S[r] = sum_of(m, 0, r, wt);
                S3[r] = sum_of(m, 1, r, wt3);
            }
            sums_to_float<KIND, 16>(S, v);
            sums_to_float<KIND, 16>(S3, v3);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                // token 8*(r/4) + 4*half + r%4 of the tile (a row past the matrix: past the buffer)
                const int t = (wm * MT + m) * kTile + 8 * (r >> 2) + 4 * half + (r & 3);
                __builtin_amdgcn_raw_buffer_store_b16((short)q16_med(gate_value_tab(v[r] * sc, v3[r] * sc3, gf, s_e)), yrs,
                                                      o < rows ? (t * G.ldy + o) * 2 : kPast, 0, 0);
            }
        }
        return;
    }

    // one token tile of each wave row at a time, the groups' sums through LDS
    Sum<KIND>* s_red = reinterpret_cast<Sum<KIND>*>(s_dyn);  // [wave][NT][16][64]
    constexpr int RB = RT * kTile;                  // output rows of the block
    constexpr int OUT = RB * kTile * WM / NTH;      // outputs a thread takes of a pass
    constexpr int NS = EPI == BEPI_STORE ? 1 : 2;   // sums of an output
    const int nl = tid % RB, on = n0 + nl, onc = min(on, rows - 1), rt = nl >> 5;
    const float sc = KIND == VGX_Q4 ? G.M.ps : G.M.wsr[onc];
    const float sc3 = EPI != BEPI_GATE ? sc : KIND == VGX_Q4 ? G.M3.ps : G.M3.wsr[onc];
    // output k of a pass: byte offset of its element
    auto at = [&](int m, int k) {
        const int e = tid / RB + k * (NTH / RB);
        return on < rows ? ((((e >> 5) * MT + m) * kTile + (e & 31)) * G.ldy + on) * 2 : kPast;
    };
    int rs[OUT];
    auto res_load = [&](int m) {
#pragma unroll
        for (int k = 0; k < OUT; ++k)
            rs[k] = EPI == BEPI_GATE ? 0 : (int)(int16_t)__builtin_amdgcn_raw_buffer_load_b16(rrs, at(m, k), 0, 0);
    };
    res_load(0);
    __syncthreads();
    WSum wt[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) wt[j] = s_ws[wk * T::wrows + (wn * NT + j) * kTile + li];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        if (m) __syncthreads();  // the previous pass's sums are read
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) s_red[((wave * NT + j) * 16 + r) * 64 + lane] = sum_of(m, j, r, wt[j]);
        __syncthreads();
        Sum<KIND> S[NS * OUT];
        float v[NS * OUT];
#pragma unroll
        for (int k = 0; k < OUT; ++k) {
            const int e = tid / RB + k * (NTH / RB), ow = e >> 5, tt = e & 31;
            // token tt of the tile: register r, lane half h (8*(r/4) + 4*h + r%4)
            const int r = 4 * (tt >> 3) + (tt & 3), ln = (nl & 31) + 32 * ((tt >> 2) & 1);
#pragma unroll
            for (int a = 0; a < NS; ++a) {
                const int wtile = EPI == BEPI_GATE ? 2 * rt + a : rt;
                const int k0 = EPI == BEPI_SPLIT ? a * (WK / 2) : 0, k1 = EPI == BEPI_SPLIT && a == 0 ? WK / 2 : WK;
                auto part = [&](int q) {
                    return s_red[((((q * WM + ow) * WN + wtile / NT) * NT + wtile % NT) * 16 + r) * 64 + ln];
                };
                Sum<KIND> t = part(k0);
#pragma unroll
                for (int q = 1; q < k1 - k0; ++q) t.add(part(k0 + q));
                S[NS * k + a] = t;
            }
        }
        sums_to_float<KIND, NS * OUT>(S, v);
#pragma unroll
        for (int k = 0; k < OUT; ++k) {
            const float a = v[NS * k] * sc, b = v[NS * k + NS - 1] * sc3, res = (float)rs[k];
            int o;
            if (EPI == BEPI_GATE) o = q16_med(gate_value_tab(a, b, gf, s_e));
            else if (EPI == BEPI_SPLIT) o = q16_med(b + (float)q16_med(a + res));
            else o = q16_med(a + res);  // (no residual: a + 0.0f = a)
            __builtin_amdgcn_raw_buffer_store_b16((short)o, yrs, at(m, k), 0, 0);
        }
        if (m + 1 < MT) res_load(m + 1);
    }
}

using TileFn = void (*)(const GemmLaunch, int, int);
struct TilePlan {
    TileFn fn;
    int bm, rb, threads, lds;
};

template <int KIND, int EPI, int MT, int NT, int WM, int WN, int WK>
TilePlan plan() {
    using T = Tile<KIND, EPI, MT, NT, WM, WN, WK>;
    if constexpr (T::ok && !(KIND == VGX_Q4 && MT * NT > 2))
        return TilePlan{gemm_tile_kernel<KIND, EPI, MT, NT, WM, WN, WK>, T::bm, kTile * T::rt, T::threads, T::lds};
    else return TilePlan{};
}

// The tile plans.  A wave's tile is kept small (32 x 32 to 32 x 64 outputs):
// these launches are a few microseconds, set by the chain of one k tile (LDS
// write, barrier, LDS read, matrix cores) and by the epilogue of a wave, so
// many short waves beat few wide ones until a launch has several tiles a CU.
//   store  0: 32 x 32 outputs a workgroup, K over 8 one-wave groups (no barrier
//             in the loop); 1: 64 x 32, four groups of two waves; 2: 64 x 64, two
//             groups of 2 x 2 waves
//   split  0: 32 x 32, 8 one-wave groups; 1: 64 x 32, the same
//   gate   0: 32 x 32, four groups (W1 and W3 in a wave each); 1: 64 x 32, two
//             groups; 2 (q4): 128 x 32, two groups (three planes of weights a step
//             want more tokens each); 3: 64 x 32, no K groups; 4 (q8, t3): 64 x 64,
//             W1 and W3 in one wave
// us a call, the one-token-tile kernel of vgx_prefill.hip before and the plan after
// (tokens x rows x columns): store 0 q8 512 x 768 x 768 6.9 -> 5.9; 1 q8 256 x 1536
// x 768 6.6 -> 5.8, q4 9.2 -> 7.9; 2 q8 512 x 2048 x 1024 10.9 -> 7.5, q4 17.3 ->
// 11.5; split 0 q8 256 x 768 x 2432 9.4 -> 6.0, q4 14.5 -> 10.4; gate 0 q8 32 x
// 2432 x 768 7.5 -> 5.6; 1 q8 256 x 2432 x 768 13.5 -> 9.1; 2 q4 the same 20.5 ->
// 13.7; 3 q8 256 x 4608 x 1024 25.4 -> 13.3; 4 q8 512 x 4608 x 1024 40.5 -> 20.2.
template <int KIND>
TilePlan plan_of(int epi, int i) {
    constexpr bool q4 = KIND == VGX_Q4;
    if (epi == BEPI_STORE) switch (i) {
        case 0: return plan<KIND, BEPI_STORE, 1, 1, 1, 1, 8>();
        case 1: return plan<KIND, BEPI_STORE, 1, 1, 2, 1, 4>();
        case 2: return plan<KIND, BEPI_STORE, 1, 1, 2, 2, 2>();
    }
    if (epi == BEPI_SPLIT) switch (i) {
        case 0: return plan<KIND, BEPI_SPLIT, 1, 1, 1, 1, 8>();
        case 1: return plan<KIND, BEPI_SPLIT, 2, 1, 1, 1, 8>();
    }
    if (epi == BEPI_GATE) switch (i) {
        case 0: return plan<KIND, BEPI_GATE, 1, 1, 1, 2, 4>();
        case 1: return plan<KIND, BEPI_GATE, 1, 1, 2, 2, 2>();
        case 2: if constexpr (q4) return plan<KIND, BEPI_GATE, 2, 1, 2, 2, 2>(); else break;
        case 3: return plan<KIND, BEPI_GATE, 1, 1, 2, 2, 1>();
        case 4: if constexpr (!q4) return plan<KIND, BEPI_GATE, 1, 2, 2, 2, 1>(); else break;
    }
    return TilePlan{};
}

TilePlan plan_of(int kind, int epi, int i) {
    return kind == VGX_Q8 ? plan_of<VGX_Q8>(epi, i) : kind == VGX_Q4 ? plan_of<VGX_Q4>(epi, i) : plan_of<VGX_T3>(epi, i);
}

// Which plan: the one whose workgroups fill the chip's rounds best.  A CU runs one
// workgroup of 64 x 32 (its operands take half the LDS and a little more) or, for
// q8 and t3, two of 32 x 32, and a second round costs about as much as the first,
// so what decides is each plan's own count of workgroups and not the launch's size
// alone.  us a call at 1,024 columns, the plan's number before each (q8; q4 after
// the bar):
//   96 x 4608 store: 0 6.4, 1 (288 workgroups) 10.9, 2 7.0 | 0 11.9, 1 15.8, 2 10.8
//   200 x 2432 store: 0 8.6, 1 (304) 11.1, 2 7.3 | 0 16.6, 1 15.7, 2 10.9
//   256 x 2048 store: 0 6.7, 1 (256) 6.5, 2 7.2 | 0 11.8, 1 8.8, 2 10.8
//   96 x 4608 gate: 0 8.6, 1 (288) 10.1, 3 10.6, 4 11.2 | 0 19.1, 1 20.9, 2 16.1, 3 17.8
//   256 x 2048 gate: 0 8.9, 1 (256) 7.5, 3 8.9, 4 11.2 | 0 19.5, 1 11.6, 2 16.3, 3 13.4
//   64 x 9600 gate: 0 12.0, 1 (300) 10.2, 3 10.6, 4 13.1 | 0 27.6, 1 20.8, 2 (300) 31.1, 3 17.9
//   200 x 4608 gate: 0 15.1, 1 (576) 14.9, 3 13.0, 4 14.5 | 1 30.2, 2 31.6, 3 24.3
//   256 x 6400 gate: 3 16.4, 4 14.8
// and the two-half residual of 2,432 columns, where a plan-1 workgroup takes as long
// as two rounds of plan 0 (q4, one 32 x 32 workgroup a CU: 1.5 rounds):
//   96 x 4608: 0 9.6, 1 (2 rounds) 16.1 | 0 18.9, 1 26.6
//   384 x 2048: 0 14.3, 1 (2) 16.6 | 0 27.9, 1 26.8
//   512 x 2048: 0 18.4, 1 (2) 17.7 | 0 36.8, 1 27.9
int pick_plan(int kind, int epi, int rows, int ntok, int num_cu) {
    const bool q4 = kind == VGX_Q4;
    auto blocks = [&](int tokens) { return (long)((rows + kTile - 1) / kTile) * ((ntok + tokens - 1) / tokens); };
    auto rounds = [&](int tokens) { return (blocks(tokens) + num_cu - 1) / num_cu; };
    const long b32 = blocks(32), b64 = blocks(64);
    if (b32 <= num_cu) return 0;
    if (epi == BEPI_SPLIT) return q4 ? 3 * rounds(64) <= 2 * rounds(32) : 2 * rounds(64) <= rounds(32);
    if (b64 <= num_cu) return 1;
    if (epi == BEPI_STORE) return !q4 && b32 <= 2L * num_cu ? 0 : 2;
    if (q4) return blocks(128) <= num_cu ? 2 : 3;
    if (b32 <= 2L * num_cu) return 0;
    if (b64 <= 2L * num_cu) return 1;
    return b32 > 6L * num_cu ? 4 : 3;
}

}  // namespace

// LDS past 64 KB is granted per kernel, once a context (not on the launch path).
hipError_t vgx_gemm_tile_init() {
    for (int kind : {VGX_Q8, VGX_Q4, VGX_T3})
        for (int epi : {BEPI_STORE, BEPI_GATE, BEPI_SPLIT})
            for (int i = 0; i < 5; ++i) {
                const TilePlan P = plan_of(kind, epi, i);
                if (P.lds <= 64 * 1024) continue;  // (no such plan: 0)
                const hipError_t e =
                    hipFuncSetAttribute((const void*)P.fn, hipFuncAttributeMaxDynamicSharedMemorySize, P.lds);
                if (e != hipSuccess) return e;
            }
    return hipSuccess;
}

int vgx_gemm_tile_launch(const GemmLaunch& L, int epi, int num_cu, hipStream_t s) {
    // the sums' ranges, and 32-bit offsets within a workgroup's rows
    if (L.cols > kMaxCols || L.M.rows > (1 << 22)) return VGX_ESTATE;
    const int kind = L.M.kind;
    const TilePlan P = plan_of(kind, epi, pick_plan(kind, epi, L.M.rows, L.ntok, num_cu));
    const long ntx = (L.M.rows + P.rb - 1) / P.rb, nty = (L.ntok + P.bm - 1) / P.bm;
    const long blocks = (ntx + 7) / 8 * 8 * nty;
    // (a launch holds less than 2^32 threads along x; the one-tile kernel's grid has a y)
    if (blocks * P.threads > 0xFFFFFFFFL) return VGX_ESTATE;
    hipLaunchKernelGGL(P.fn, dim3((unsigned)blocks), dim3(P.threads), P.lds, s, L, (int)ntx, (int)nty);
    VGX_LAUNCH_CHECK("gemm tile launch");
    return VGX_OK;
}
