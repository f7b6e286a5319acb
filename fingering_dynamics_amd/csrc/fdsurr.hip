// fdsurr.hip - gfx950 BF16 MFMA 3x3 convolutions of the phase-field
// surrogate (declarations and conventions: include/fdsurr.h).
//
// All three passes are GEMMs on v_mfma_f32_16x16x32_bf16 (FP32 accumulate).
// Operand layout of one 16x16x32 MFMA (measured on MI355X):
//   A[i][k] (16 x 32): lane i + 16*(k/8), element k%8
//   B[k][j] (32 x 16): lane j + 16*(k/8), element k%8
//   D[i][j] (16 x 16): lane j + 16*(i/4), element i%4
// so a lane holds 8 consecutive k of one row (A) or column (B): in NHWC
// with C % 8 == 0 those are 8 channels of one pixel and one tap - a single
// 16-byte load.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <string>
#include <type_traits>

#include "fdsurr.h"

namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));
typedef unsigned u2v __attribute__((ext_vector_type(2)));

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}

#define FDS_HIP(call)                                                                     \
    do {                                                                                  \
        hipError_t e_ = (call);                                                           \
        if (e_ != hipSuccess)                                                             \
            return fail(FDS_E_HIP, std::string(#call) + ": " + hipGetErrorString(e_));    \
    } while (0)

__device__ __forceinline__ v8bf bf8(u4v v) { return __builtin_bit_cast(v8bf, v); }

__device__ __forceinline__ uint16_t to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// The bf16 halves of v where the matching halves of m (a ReLU output) are
// > 0 - for bf16 that is the bit pattern read as a positive int16 - and 0
// elsewhere: the ReLU's backward mask applied on load.
__device__ __forceinline__ u4v relu_keep(u4v v, u4v m) {
    u4v r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const unsigned lo = ((int16_t)(m[i] & 0xFFFFu) > 0) ? 0x0000FFFFu : 0u;
        const unsigned hi = ((int16_t)(m[i] >> 16) > 0) ? 0xFFFF0000u : 0u;
        r[i] = v[i] & (lo | hi);
    }
    return r;
}

// ---------------------------------------------------------------- forward
// y[p][co] = act(bias[co] + sum_k A[p][k] w[co][k]), p over N*H*W (NHWC),
// k = tap*Cin + ci with tap = 3*(dh+1) + (dw+1) and A[p][k] = x at pixel
// (n, h+dh, w+dw), channel ci (0 outside the image).  One wave computes
// 16*MP consecutive pixels x 16*NT output channels (MP x NT MFMA tiles, so
// every A fragment is used NT times and every B fragment MP times); the
// four waves of a workgroup take consecutive pixel ranges with the same
// channels, so they share the weight fragments through L1.  The K loop
// takes 32 k per step (one tap and 8 channels per lane, a 16-byte load);
// k beyond 9*Cin and channels beyond Cout load zeros.  With MASK, x is
// multiplied on load by the ReLU mask of xm (the input gradient pass).
// Workgroups of a 1-D grid are dispatched to the 8 XCDs round robin
// (workgroup i runs on XCD i mod 8), and each XCD has its own L2.  The
// logical index returned gives every XCD a contiguous band of logical
// workgroups, so workgroups adjacent in logical order, which read the same
// or overlapping data (the channel blocks of one tile, the taps of one
// pixel slice, neighbouring tiles' halo rows), share an L2.
__device__ __forceinline__ int xcd_band() {
    const int n = (int)gridDim.x, q = n >> 3, rem = n & 7, xcd = (int)blockIdx.x & 7;
    return xcd * q + min(xcd, rem) + ((int)blockIdx.x >> 3);
}

template <int MP, int NT, bool MASK>
__global__ __launch_bounds__(256) void conv_fwd(const uint16_t* __restrict__ x, const uint16_t* __restrict__ xm,
                                                const uint16_t* __restrict__ w, const float* __restrict__ bias,
                                                float* __restrict__ y32, uint16_t* __restrict__ y16, int N, int H,
                                                int W, int Cin, int Cout, int relu) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t P = (int64_t)N * H * W;
    // logical workgroup = pixel block x channel block, channel blocks adjacent
    const int ncb = (Cout + 16 * NT - 1) / (16 * NT);
    const int L = xcd_band();
    const int pb = L / ncb;
    const int64_t pw = ((int64_t)pb * 4 + wave) * (16 * MP);
    const int co0 = (L - pb * ncb) * (16 * NT);
    const int K = 9 * Cin;
    int hq[MP], wq[MP];
    int64_t img[MP];
#pragma unroll
    for (int g = 0; g < MP; ++g) {
        const int64_t pa = pw + 16 * g + (lane & 15);
        hq[g] = -4;  // out of range for every tap: pixels past the end load zeros
        wq[g] = 0;
        img[g] = 0;
        if (pa < P) {
            wq[g] = (int)(pa % W);
            const int64_t t = pa / W;
            hq[g] = (int)(t % H);
            img[g] = (t / H) * H;
        }
    }
    v4f acc[MP][NT];
#pragma unroll
    for (int g = 0; g < MP; ++g)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[g][t] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int kc = 0; kc < K; kc += 32) {
        const int k0 = kc + 8 * (lane >> 4);
        const bool kin = k0 < K;
        const int tap = k0 / Cin, ci = k0 - tap * Cin;
        const int dh = tap / 3 - 1, dw = tap % 3 - 1;
        // every load of the step is issued before any is used, so the
        // waits cover all of them at once
        u4v av[MP], mv[MP], bv[NT];
#pragma unroll
        for (int g = 0; g < MP; ++g) {
            av[g] = u4v{0u, 0u, 0u, 0u};
            mv[g] = u4v{0u, 0u, 0u, 0u};
            const int hh = hq[g] + dh, ww = wq[g] + dw;
            if (kin && hh >= 0 && hh < H && ww >= 0 && ww < W) {
                const int64_t o = ((img[g] + hh) * W + ww) * Cin + ci;
                av[g] = *reinterpret_cast<const u4v*>(x + o);
                if (MASK) mv[g] = *reinterpret_cast<const u4v*>(xm + o);
            }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int co = co0 + 16 * t + (lane & 15);
            bv[t] = u4v{0u, 0u, 0u, 0u};
            if (co < Cout && kin) bv[t] = *reinterpret_cast<const u4v*>(w + (int64_t)co * K + k0);
        }
        if (MASK) {
#pragma unroll
            for (int g = 0; g < MP; ++g) av[g] = relu_keep(av[g], mv[g]);
        }
#pragma unroll
        for (int g = 0; g < MP; ++g)
#pragma unroll
            for (int t = 0; t < NT; ++t)
                acc[g][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf8(av[g]), bf8(bv[t]), acc[g][t], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int co = co0 + 16 * t + (lane & 15);
        if (co >= Cout) continue;
        const float b = bias ? bias[co] : 0.f;
#pragma unroll
        for (int g = 0; g < MP; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t p = pw + 16 * g + 4 * (lane >> 4) + r;
                if (p >= P) continue;
                float v = acc[g][t][r] + b;
                if (relu) v = fmaxf(v, 0.f);
                if (y32) y32[p * Cout + co] = v;
                if (y16) y16[p * Cout + co] = to_bf16(v);
            }
    }
}

// Buffer access to one image or to the weights: a descriptor of `bytes`
// bytes; a load at kOOB (any offset past the end) returns zeros without a
// memory access, which is the convolution's zero padding.
using rsrc_t = __amdgpu_buffer_rsrc_t;
constexpr unsigned kOOB = 0x7FFFFF00u;
constexpr int64_t kMaxBytes = (int64_t)0x7FFFFE00;  // of one descriptor

__device__ __forceinline__ rsrc_t make_rsrc(const void* p, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ u4v load16(rsrc_t r, unsigned voff, unsigned soff) {
    return __builtin_bit_cast(u4v, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
}

__device__ __forceinline__ void store16(rsrc_t r, unsigned voff, u4v v) {
    __builtin_amdgcn_raw_buffer_store_b128(v, r, (int)voff, 0, 0);
}
__device__ __forceinline__ void store8(rsrc_t r, unsigned voff, u2v v) {
    __builtin_amdgcn_raw_buffer_store_b64(v, r, (int)voff, 0, 0);
}

// Tile geometry shared by the two staged convolution kernels below: four
// waves, WP of them stacked over pixel rows and 4 / WP side by side over
// output channels; a wave computes R rows x 16 CT columns x 16 WC output
// channels.  The weights are the MFMA's A operand (rows = output channels)
// and the pixels its B operand, so a lane's results are output channels of
// one pixel.  With WC even, row i of tile t of a pair holds channel
// 8 (i / 4) + 4 (t mod 2) + i mod 4 of the pair's 32, and the lane holds
// eight consecutive channels: one 16-byte store (bf16).  Scattered 2-byte
// stores of the transposed assignment had cost the thin layers as much as
// their MFMAs.
template <int R, int CT, int WC, int WP>
struct Tile {
    static constexpr int WN = 4 / WP;
    static constexpr int BR = WP * R;          // output rows of the block
    static constexpr int BW = 16 * CT;         // output columns
    static constexpr int BC = WN * WC * 16;    // output channels
    static constexpr int HW = BW + 2;          // halo columns
    static constexpr int HP = (BR + 2) * HW;   // halo pixels
    // LDS row (A row) of the block's output channel c
    static __device__ __forceinline__ int wrow(int c) {
        if (WC % 2) return c;
        return (c & ~31) + 16 * ((c >> 2) & 1) + 4 * ((c >> 3) & 3) + (c & 3);
    }
};

struct ConvArgs {
    const uint16_t* x;
    const uint16_t* xm;   // ReLU mask of x applied on load (MASK)
    const uint16_t* w;
    const float* bias;
    float* y32;
    uint16_t* y16;
    int N, H, W, Cin, Cout, relu;
    int hb, wb;           // blocks of an image
    int npx, ncb;         // pixel blocks in all, channel blocks
};

// Results of one wave's tile at rows h0.., columns w0.. and the block's
// channels c0.. (co0 + c0 of the layer).  The stores are predicated by
// offset, without a branch, and the bias comes from LDS: a branch, or a
// load of its own here, makes the wait for the next block's prefetched
// halo cover these stores, or these results wait for that halo.
template <int R, int CT, int WC, bool OUT32>
__device__ __forceinline__ void store_tile(const ConvArgs& a, const v4f (&acc)[R][CT][WC], const float* sbias, int n,
                                           int h0, int w0, int co0, int c0) {
    const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
    constexpr int V = (WC % 2) ? 4 : 8;        // consecutive channels of a lane
    constexpr int G = (WC % 2) ? WC : WC / 2;
    constexpr int ES = OUT32 ? 4 : 2;
    const int64_t img = (int64_t)a.H * a.W * a.Cout * ES;
    const rsrc_t yr = make_rsrc(OUT32 ? (char*)a.y32 + n * img : (char*)a.y16 + n * img, img);
#pragma unroll
    for (int u = 0; u < G; ++u) {
        const int c = c0 + (V == 8 ? 32 : 16) * u + V * q, co = co0 + c;
        float b[V];
#pragma unroll
        for (int e = 0; e < V; ++e) b[e] = sbias[c + e];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int k = 0; k < CT; ++k) {
                const int h = h0 + r, w = w0 + 16 * k + j;
                const bool in = h < a.H && w < a.W && co < a.Cout;
                const unsigned o = in ? (unsigned)(((h * a.W + w) * a.Cout + co) * ES) : kOOB;
                float v[V];
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    v[e] = acc[r][k][V == 8 ? 2 * u + (e >> 2) : u][e & 3] + b[e];
                    if (a.relu) v[e] = fmaxf(v[e], 0.f);
                }
                if constexpr (OUT32) {
#pragma unroll
                    for (int e = 0; e < V; e += 4) store16(yr, o + 4 * e, __builtin_bit_cast(u4v, v4f{v[e], v[e + 1], v[e + 2], v[e + 3]}));
                } else {
                    unsigned p[V / 2];
#pragma unroll
                    for (int e = 0; e < V; e += 2)
                        p[e / 2] = (unsigned)to_bf16(v[e]) | ((unsigned)to_bf16(v[e + 1]) << 16);
                    if constexpr (V == 8)
                        store16(yr, o, u4v{p[0], p[1], p[2], p[3]});
                    else
                        store8(yr, o, u2v{p[0], p[1]});
                }
            }
    }
}

// The block of index t: with one chunk of input channels the channel block
// is the slow index (a workgroup's run of blocks keeps its weights in LDS),
// else the fast one (the channel blocks of a pixel block share its halo
// through L2).
struct BlockPos {
    int n, h0, w0, cb;
};
__device__ __forceinline__ BlockPos block_pos(const ConvArgs& a, int t, bool cb_slow, int BR, int BW) {
    BlockPos p;
    int px;
    if (cb_slow) {
        p.cb = t / a.npx;
        px = t - p.cb * a.npx;
    } else {
        px = t / a.ncb;
        p.cb = t - px * a.ncb;
    }
    const int row = px / a.wb;
    p.w0 = (px - row * a.wb) * BW;
    p.n = row / a.hb;
    p.h0 = (row - p.n * a.hb) * BR;
    return p;
}

// Convolution with input and weights staged in LDS, Cin a multiple of 32.
// A workgroup walks a contiguous run of blocks.  Per block and chunk of 32
// input channels it holds in LDS the block's input halo (zeros outside the
// image) and the nine taps' weights, 64 bytes per pixel or channel, the
// four 16-byte pieces of row p stored at piece ^ ((p / 2) mod 4): the
// fragment reads of eight consecutive rows then cover all 32 banks.  The
// next halo is loaded into registers while this one's MFMAs run (with PFW
// the weights too); with one chunk the weights stay for the whole run.
//
// Bounds: the MFMA needs a fragment (1 KB of LDS reads) per two of its
// 16-cycle issues at most; R = 4, CT = 2, WC = 4 reads 12 fragments per 32
// MFMAs.  The kernel before this one took its weight fragments from global
// memory, 16 rows of 64 bytes per load instruction with consecutive lanes
// in different rows, four times the tag lookups of a contiguous load.
// K order per output: chunk, tap, channel (as that kernel's).
template <int R, int CT, int WC, int WP, int PF, bool MASK, bool OUT32>
__global__ __launch_bounds__(256, 2) void conv_tile(ConvArgs a) {
    using T = Tile<R, CT, WC, WP>;
    constexpr int HPC = T::HP * 4;                 // 16-byte pieces of the halo
    constexpr int PPT = (HPC + 255) / 256;
    constexpr int WPC = 9 * T::BC * 4;             // of the weights
    constexpr int WPT = (WPC + 255) / 256;
    __shared__ __align__(16) u4v halo[HPC];
    __shared__ __align__(16) u4v wlds[WPC];
    __shared__ float sbias[T::BC];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave % WP, wn = wave / WP;
    const int j = lane & 15, q = lane >> 4;
    const int nchunks = a.Cin / 32;
    const int total = a.npx * a.ncb, G = (int)gridDim.x;
    const int L = xcd_band();
    const int tbeg = (int)((int64_t)total * L / G), tend = (int)((int64_t)total * (L + 1) / G);
    if (tbeg >= tend) return;
    const int64_t img_bytes = (int64_t)a.H * a.W * a.Cin * 2;
    const int wbytes = a.Cout * 9 * a.Cin * 2;
    const rsrc_t wres = make_rsrc(a.w, wbytes);
    const rsrc_t bres = make_rsrc(a.bias, a.bias ? a.Cout * 4 : 0);
    const int krow = 9 * a.Cin * 2;

    u4v hv[PPT], mv[MASK ? PPT : 1], wv[PF == 2 ? WPT : 1];
    auto fetch_halo = [&](const BlockPos& p, int c) {
        const rsrc_t xr = make_rsrc(a.x + p.n * (img_bytes / 2), img_bytes);
        const rsrc_t mr = make_rsrc(MASK ? a.xm + p.n * (img_bytes / 2) : a.x, MASK ? img_bytes : 0);
#pragma unroll
        for (int i = 0; i < PPT; ++i) {
            const int s = tid + 256 * i, px = s >> 2, g = s & 3;
            const int hr = px / T::HW, hc = px - hr * T::HW;
            const int hh = p.h0 - 1 + hr, ww = p.w0 - 1 + hc;
            const bool in = s < HPC && (unsigned)hh < (unsigned)a.H && (unsigned)ww < (unsigned)a.W;
            const unsigned vo = in ? (unsigned)(((hh * a.W + ww) * a.Cin + 8 * g) * 2) : kOOB;
            hv[i] = load16(xr, vo, 64 * c);
            if (MASK) mv[i] = load16(mr, vo, 64 * c);
        }
    };
    auto stage_halo = [&]() {
#pragma unroll
        for (int i = 0; i < PPT; ++i) {
            const int s = tid + 256 * i, px = s >> 2, g = s & 3;
            const int hr = px / T::HW, hc = px - hr * T::HW;
            if (s < HPC) halo[px * 4 + (g ^ ((hc >> 1) & 3))] = MASK ? relu_keep(hv[i], mv[i]) : hv[i];
        }
    };
    auto fetch_w = [&](int i, int cb, int c) {
        const int s = tid + 256 * i, tap = s / (T::BC * 4), rem = s - tap * (T::BC * 4), co = rem >> 2, g = rem & 3;
        const bool in = s < WPC && cb * T::BC + co < a.Cout;
        return load16(wres, in ? (unsigned)((cb * T::BC + co) * krow + (tap * a.Cin + 8 * g) * 2) : kOOB, 64 * c);
    };
    auto stage_w = [&](int i, const u4v& v) {
        const int s = tid + 256 * i, tap = s / (T::BC * 4), rem = s - tap * (T::BC * 4), co = rem >> 2, g = rem & 3;
        const int row = T::wrow(co);
        if (s < WPC) wlds[(tap * T::BC + row) * 4 + (g ^ ((row >> 1) & 3))] = v;
    };

    BlockPos p = block_pos(a, tbeg, nchunks == 1, T::BR, T::BW);
    int t = tbeg, c = 0, wcb = -1;  // wcb: channel block whose only chunk is staged
    if (PF) fetch_halo(p, 0);
    if (PF == 2) {
#pragma unroll
        for (int i = 0; i < WPT; ++i) wv[i] = fetch_w(i, p.cb, 0);
    }
    v4f acc[R][CT][WC];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 0; k < CT; ++k)
#pragma unroll
            for (int u = 0; u < WC; ++u) acc[r][k][u] = v4f{0.f, 0.f, 0.f, 0.f};
    // fragment addresses (in 16-byte pieces): pixel row wr R, column j + dw;
    // rows, column tiles and taps are constant offsets from them
    int pa[3];
#pragma unroll
    for (int dw = 0; dw < 3; ++dw) pa[dw] = (wr * R * T::HW + j + dw) * 4 + (q ^ (((j + dw) >> 1) & 3));
    const int wa = (wn * WC * 16 + j) * 4 + (q ^ ((j >> 1) & 3));

    for (;;) {
        if (!PF) fetch_halo(p, c);
        __syncthreads();  // the previous chunk's fragments have been read
        stage_halo();
        if (wcb != p.cb) {
            if (tid < T::BC && c == 0)
                sbias[tid] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(bres, (p.cb * T::BC + tid) * 4, 0, 0));
            if (PF == 2) {
#pragma unroll
                for (int i = 0; i < WPT; ++i) stage_w(i, wv[i]);
            } else {
                u4v v[WPT];
#pragma unroll
                for (int i = 0; i < WPT; ++i) v[i] = fetch_w(i, p.cb, c);
#pragma unroll
                for (int i = 0; i < WPT; ++i) stage_w(i, v[i]);
            }
            wcb = nchunks == 1 ? p.cb : -1;
        }
        __syncthreads();
        // the next chunk (of this block or of the next one)
        const bool last = c + 1 == nchunks;
        const int tn = last ? t + 1 : t, cn = last ? 0 : c + 1;
        BlockPos pn = p;
        if (last && tn < tend) pn = block_pos(a, tn, nchunks == 1, T::BR, T::BW);
        if (PF && tn < tend) {
            fetch_halo(pn, cn);
            if (PF == 2 && wcb != pn.cb) {
#pragma unroll
                for (int i = 0; i < WPT; ++i) wv[i] = fetch_w(i, pn.cb, cn);
            }
        }
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            v8bf wf[WC];
#pragma unroll
            for (int u = 0; u < WC; ++u) wf[u] = bf8(wlds[wa + (tap * T::BC + 16 * u) * 4]);
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int k = 0; k < CT; ++k) {
                    const v8bf pf = bf8(halo[pa[tap % 3] + ((r + tap / 3) * T::HW + 16 * k) * 4]);
#pragma unroll
                    for (int u = 0; u < WC; ++u)
                        acc[r][k][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u], pf, acc[r][k][u], 0, 0, 0);
                }
        }
        if (last) {
            store_tile<R, CT, WC, OUT32>(a, acc, sbias, p.n, p.h0 + wr * R, p.w0, p.cb * T::BC, wn * WC * 16);
            if (tn >= tend) break;
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int k = 0; k < CT; ++k)
#pragma unroll
                    for (int u = 0; u < WC; ++u) acc[r][k][u] = v4f{0.f, 0.f, 0.f, 0.f};
        }
        t = tn;
        c = cn;
        p = pn;
    }
}

// The same for few input channels (Cin = 8 CG, 1 <= CG <= 7): the K index
// k = tap Cin + ci runs over all nine taps in steps of 32, so a lane's
// eight values are channels of tap k / Cin of its pixel; all channels of
// the halo are staged at once, CG pieces per pixel (one more when CG is
// even: an odd stride in 16-byte pieces spreads the banks), and the whole
// weight rows, zero-padded to whole steps.
template <int R, int CT, int WC, int CG, bool MASK, bool OUT32>
__global__ __launch_bounds__(256, 2) void conv_tile_thin(ConvArgs a) {
    using T = Tile<R, CT, WC, 4>;
    constexpr int Cin = 8 * CG, K = 9 * Cin;
    constexpr int S = (K + 31) / 32;               // MFMA steps
    constexpr int PS = CG | 1;                     // pieces per staged pixel
    constexpr int WS = 4 * S + 1;                  // pieces per staged weight row
    constexpr int HPC = T::HP * CG, PPT = (HPC + 255) / 256;
    constexpr int WPC = T::BC * 4 * S;
    __shared__ __align__(16) u4v halo[T::HP * PS];
    __shared__ __align__(16) u4v wlds[T::BC * WS];
    __shared__ float sbias[T::BC];
    const int tid = threadIdx.x, lane = tid & 63, wr = tid >> 6;
    const int j = lane & 15, q = lane >> 4;
    const int total = a.npx * a.ncb, G = (int)gridDim.x;
    const int L = xcd_band();
    const int tbeg = (int)((int64_t)total * L / G), tend = (int)((int64_t)total * (L + 1) / G);
    if (tbeg >= tend) return;
    const int64_t img_bytes = (int64_t)a.H * a.W * Cin * 2;
    const rsrc_t wres = make_rsrc(a.w, (int64_t)a.Cout * K * 2);
    const rsrc_t bres = make_rsrc(a.bias, a.bias ? a.Cout * 4 : 0);

    u4v hv[PPT], mv[MASK ? PPT : 1];
    auto fetch_halo = [&](const BlockPos& p) {
        const rsrc_t xr = make_rsrc(a.x + p.n * (img_bytes / 2), img_bytes);
        const rsrc_t mr = make_rsrc(MASK ? a.xm + p.n * (img_bytes / 2) : a.x, MASK ? img_bytes : 0);
#pragma unroll
        for (int i = 0; i < PPT; ++i) {
            const int s = tid + 256 * i, px = s / CG, g = s - px * CG;
            const int hr = px / T::HW, hc = px - hr * T::HW;
            const int hh = p.h0 - 1 + hr, ww = p.w0 - 1 + hc;
            const bool in = s < HPC && (unsigned)hh < (unsigned)a.H && (unsigned)ww < (unsigned)a.W;
            const unsigned vo = in ? (unsigned)(((hh * a.W + ww) * Cin + 8 * g) * 2) : kOOB;
            hv[i] = load16(xr, vo, 0);
            if (MASK) mv[i] = load16(mr, vo, 0);
        }
    };
    BlockPos p = block_pos(a, tbeg, true, T::BR, T::BW);
    fetch_halo(p);
    int wcb = -1;
    for (int t = tbeg;;) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PPT; ++i) {
            const int s = tid + 256 * i, px = s / CG, g = s - px * CG;
            if (s < HPC) halo[px * PS + g] = MASK ? relu_keep(hv[i], mv[i]) : hv[i];
        }
        if (wcb != p.cb) {
            wcb = p.cb;
            if (tid < T::BC)
                sbias[tid] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(bres, (p.cb * T::BC + tid) * 4, 0, 0));
            for (int s = tid; s < WPC; s += 256) {
                const int co = s / (4 * S), g = s - co * (4 * S);
                const bool in = 8 * g < K && p.cb * T::BC + co < a.Cout;
                wlds[T::wrow(co) * WS + g] =
                    load16(wres, in ? (unsigned)(((p.cb * T::BC + co) * K + 8 * g) * 2) : kOOB, 0);
            }
        }
        __syncthreads();
        BlockPos pn = p;
        if (t + 1 < tend) {
            pn = block_pos(a, t + 1, true, T::BR, T::BW);
            fetch_halo(pn);
        }
        v4f acc[R][CT][WC];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int k = 0; k < CT; ++k)
#pragma unroll
                for (int u = 0; u < WC; ++u) acc[r][k][u] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int k0 = 32 * s + 8 * q;
            const bool kin = k0 < K;
            const int tap = kin ? k0 / Cin : 0, g = kin ? (k0 - tap * Cin) >> 3 : 0;
            const int po = ((wr * R + tap / 3) * T::HW + j + tap % 3) * PS + g;
            v8bf wf[WC];
#pragma unroll
            for (int u = 0; u < WC; ++u) wf[u] = bf8(wlds[(16 * u + j) * WS + 4 * s + q]);
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int k = 0; k < CT; ++k) {
                    u4v v = halo[po + (r * T::HW + 16 * k) * PS];
                    // the padding's pixels are zeros too: what they would
                    // read could be infinite
                    if (32 * s + 32 > K && !kin) v = u4v{0u, 0u, 0u, 0u};
#pragma unroll
                    for (int u = 0; u < WC; ++u)
                        acc[r][k][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u], bf8(v), acc[r][k][u], 0, 0, 0);
                }
        }
        store_tile<R, CT, WC, OUT32>(a, acc, sbias, p.n, p.h0 + wr * R, p.w0, p.cb * T::BC, 0);
        if (++t >= tend) break;
        p = pn;
    }
}

// wt[ci][tap][co] = w[co][8 - tap][ci]
__global__ __launch_bounds__(256) void flip_weights(const uint16_t* __restrict__ w, uint16_t* __restrict__ wt, int Cin,
                                                    int Cout) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t total = (int64_t)Cout * 9 * Cin;
    if (i >= total) return;
    const int ci = (int)(i % Cin);
    const int tap = (int)((i / Cin) % 9);
    const int co = (int)(i / (9 * (int64_t)Cin));
    wt[((int64_t)ci * 9 + (8 - tap)) * Cout + co] = w[i];
}

// The bf16 weights of every layer of a network and their flipped copies
// (flip_weights) from the FP32 master weights in one launch: a step's 15
// layers would otherwise take 30 small launches.  Layer l holds elements
// [start[l], start[l + 1]) of the grid.
constexpr int kCastLayers = 16;
struct CastFlipArgs {
    const float* w[kCastLayers];
    uint16_t* w16[kCastLayers];
    uint16_t* wt[kCastLayers];
    int cin[kCastLayers], cout[kCastLayers];
    int64_t start[kCastLayers + 1];
    int n;
};

__global__ __launch_bounds__(256) void cast_flip(CastFlipArgs a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.start[a.n]) return;
    int l = 0;
    while (l + 1 < a.n && i >= a.start[l + 1]) ++l;
    const int64_t j = i - a.start[l];
    const int Cin = a.cin[l], Cout = a.cout[l];
    const uint16_t v = to_bf16(a.w[l][j]);
    a.w16[l][j] = v;
    if (!a.wt[l]) return;
    const int ci = (int)(j % Cin);
    const int tap = (int)((j / Cin) % 9);
    const int co = (int)(j / (9 * (int64_t)Cin));
    a.wt[l][((int64_t)ci * 9 + (8 - tap)) * Cout + co] = v;
}

// ------------------------------------------------------- weight gradient
// dw[co][tap][ci] = sum_p dy[p][co] x[p + d(tap)][ci]: a GEMM whose
// reduction runs over pixels, the strided dimension of both operands.  Both
// are staged in LDS as they lie in memory, [pixel][channel], and the
// fragments are read with the transposing LDS load (ds_read_b64_tr_b16: the
// 16 lanes of a group address 4 pixels x 4 groups of 4 channels and receive
// 4 pixels of one channel each), two loads for the eight pixels of a lane.
//
// A wave computes 16 ACO output channels x 16 ACI input channels x all nine
// taps.  It marches down the rows of a strip of 32 columns (the 32 k of an
// MFMA step): a row of x meets the three rows of dy whose taps reach it,
// kept as fragments in registers, so a row costs ACO fragments of dy and
// 3 ACI of x (the tap's column shift is the address) for 9 ACO ACI MFMAs:
// 8 for 36, far below what the LDS delivers, and x and dy are read from
// global memory once for all taps.  The kernel before this one had one tap
// per workgroup: nine times the loads, and each of its pixel pairs was
// transposed by 32-bit LDS writes.
//
// The eight waves of a workgroup are WCO x WCI channel tiles x WK groups
// that take different strips (k groups); groups are added through LDS at the
// end in a fixed tree, and the workgroup writes one partial sum, which
// reduce_slices adds in a fixed order.  Work items are (image, run of
// `rows` rows, strip), the strips adjacent (groups that run together read
// neighbouring columns): a run reads its rows and, of x, one row more on
// either side, as zeros outside the image.
//
// A row step has few bytes and few MFMAs (576 cycles of them for 32 x 32
// channels), so what bounds the kernel is how many rows are in flight and
// what else a step issues: rows are loaded straight into LDS (no registers
// are held for them), in a ring of NS stages of RS rows; a lane's offsets
// are formed once per item; the steps that need no masks have a loop of
// their own.  Measured with reduce_slices, us a layer at batch 64, the
// kernels before these in parentheses: 32 -> 32 at 128 x 256 61 (161),
// 96 -> 32 154 (409), 64 -> 64 at 64 x 128 54 (163), 192 -> 64 131 (418),
// 256 -> 128 at 32 x 64 82 (286).  In registers, one row ahead: 83 for the
// first; with the offsets formed per row and every step masked: 73.  The
// 64-channel blocks keep the matrix cores busy 47 % of the time at the
// 2.0 GHz the chip holds there.
//
// A staged row lies in LDS as 16-byte pieces, dy then x (then dy's ReLU
// mask), then the two x columns beside the strip.  Its rows are permuted in
// 32-byte granules so that the four pixels of a transposing load fall on
// different banks: granule g of pixel p is stored at g ^ (p mod 4) with 64
// channels, g ^ (p / 2 mod 2) with 32.
template <int G>
__device__ __forceinline__ int granule(int g, int p) {
    return G >= 4 ? g ^ (p & 3) : (G == 2 ? g ^ ((p >> 1) & 1) : g);
}

typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) v4s lds_v4s;
typedef __attribute__((address_space(3))) char lds_char;

// Fragment of 32 pixels x 16 channels: a and b address this lane's piece of
// the first and second four pixels of its group of eight.
__device__ __forceinline__ v8bf tr_frag(unsigned a, unsigned b) {
    const v4s u = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(lds_char*)(uintptr_t)a);
    const v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(lds_char*)(uintptr_t)b);
    return __builtin_bit_cast(v8bf, v8s{u[0], u[1], u[2], u[3], v[0], v[1], v[2], v[3]});
}

// One 16-byte piece per lane from a buffer straight into LDS at lds + 16 x
// lane (zeros at kOOB).  No register is written, so nothing waits for it but
// wait_loads; the compiler does not see it, and its own waits, which count
// the same counter, only become stricter.
__device__ __forceinline__ void load_lds(u4v rsrc, unsigned voff, unsigned soff, unsigned lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory", "m0");
}
// All but the newest N loads of this wave have arrived, and every LDS read of
// it has returned.  The second is for buffers that later loads land in: that
// the reads' uses come before this point is nothing the compiler has to keep
// (it does; the wait costs nothing).
template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "i"(N) : "memory");
}
// The words of make_rsrc(p, bytes), in scalar registers.
__device__ __forceinline__ u4v rsrc_words(const void* p, int64_t bytes) {
    const uint64_t b = (uint64_t)p;
    return u4v{(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b),
               (unsigned)__builtin_amdgcn_readfirstlane((int)((unsigned)(b >> 32) & 0xFFFFu)), (unsigned)bytes,
               0x00020000u};
}

struct WgradArgs {
    const uint16_t* x;
    const uint16_t* dy;
    const uint16_t* dym;  // ReLU mask of dy (MASK)
    float* part;          // [slice][Cout * 9 * Cin + Cout]
    int with_bias;
    int N, H, W, Cin, Cout;
    int strips, chunks, rows;  // 32-column strips, row runs and their height
    int items, slices, ncb, nib;
};

template <int ACO, int ACI, int WCO, int WCI, int WK, int NS, int RS, bool MASK>
__global__ __launch_bounds__(512, 2) void conv_wgrad(WgradArgs a) {
    static_assert(WCO * WCI * WK == 8, "eight waves");
    constexpr int BCO = 16 * ACO * WCO, BCI = 16 * ACI * WCI;  // channels of the block
    constexpr int WG = WCO * WCI, NT = 64 * WG;                 // waves, threads of a k group
    constexpr int PO = BCO / 8, PI = BCI / 8;                   // 16-byte pieces per pixel
    constexpr int GO = BCO / 16, GI = BCI / 16;                 // granules per pixel
    constexpr int RD = 32 * PO, RX = 32 * PI, RE = 2 * PI;      // pieces of a row: dy, x, x beside the strip
    static_assert(RD % 64 == 0 && RX % 64 == 0 && RE <= 64, "whole waves");
    // loads of a row per wave: dy and x in 64-piece parts dealt to the
    // group's waves, the two edge columns on its first wave
    constexpr int PD = RD / 64, PX = RX / 64;
    constexpr int ND = PD / WG, NX = PX / WG;
    static_assert(PD % WG == 0 && PX % WG == 0, "every wave has as many parts");
    constexpr int ROW = RD + RX + (MASK ? RD : 0) + RE;         // pieces of a staged row
    constexpr int TILES = 9 * ACO * ACI;
    constexpr int NB = NS * RS;                                 // row buffers
    constexpr int RED = 4 * (TILES + ACO) * 64;                 // pieces of the group sums
    constexpr int RING = NB * WK * ROW;
    static_assert(RING * 16 <= 160 * 1024 && RED * 16 <= 160 * 1024, "LDS");
    __shared__ __align__(16) u4v smem[RING > RED ? RING : RED];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave / WG, wt = wave % WG, wco = wt % WCO, wci = wt / WCO;
    const int j = lane & 15, q = lane >> 4;
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_char*)smem + (unsigned)(kg * NB * ROW * 16);  // the group's ring

    // logical workgroup = slice x channel block, the blocks of one slice
    // adjacent (they read the same x and dy)
    const int L = xcd_band(), nblk = a.ncb * a.nib;
    const int slice = L / nblk, blk = L - slice * nblk;
    const int co0 = (blk % a.ncb) * BCO, ci0 = (blk / a.ncb) * BCI;

    // the group's items, and how many every group of the workgroup runs
    const int ngrp = a.slices * WK, gid = slice * WK + kg;
    auto first = [&](int g) { return (int)(((int64_t)a.items * g + ngrp - 1) / ngrp); };  // low groups first
    const int ibeg = first(gid), iend = first(gid + 1);
    const int spi = (a.rows + 2 + RS - 1) / RS * RS;  // row steps of an item
    const int nit = (a.items + ngrp - 1) / ngrp;

    // Loads of the next row.  A lane's byte offsets within a row of the
    // strip are formed once per item; the row is the scalar offset, and a
    // row that is not wanted (outside the run or the image) reads a
    // descriptor of no bytes, i.e. zeros.
    const int64_t xb = (int64_t)a.H * a.W * a.Cin * 2, db = (int64_t)a.H * a.W * a.Cout * 2;
    unsigned dvo[ND], xvo[NX], evo = kOOB;
    int it = ibeg, st = 0, slot = 0;  // item and row to load, its buffer
    int ln = 0, r0 = 0, r1 = 0;       // the item's image and rows
    auto load = [&]() {
        if (st == 0) {
            const int run = it / a.strips, w0 = (it - run * a.strips) * 32;
            const int n = run / a.chunks, chunk = run - n * a.chunks;
            const bool live = it < iend;
            ln = live ? n : 0;
            r0 = live ? chunk * a.rows : a.H + 2;  // rows past the image: none is wanted
            r1 = min(r0 + a.rows, a.H);
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                const int s = (wt + WG * i) * 64 + lane, px = s / PO, g = s % PO;
                const int c = co0 + 8 * (2 * granule<GO>(g >> 1, px) + (g & 1));
                dvo[i] = w0 + px < a.W && c < a.Cout ? (unsigned)(((w0 + px) * a.Cout + c) * 2) : kOOB;
            }
#pragma unroll
            for (int i = 0; i < NX; ++i) {
                const int s = (wt + WG * i) * 64 + lane, px = s / PI, g = s % PI;
                const int c = ci0 + 8 * (2 * granule<GI>(g >> 1, px) + (g & 1));
                xvo[i] = w0 + px < a.W && c < a.Cin ? (unsigned)(((w0 + px) * a.Cin + c) * 2) : kOOB;
            }
            const int ww = lane / PI ? w0 + 32 : w0 - 1, c = ci0 + 8 * (lane % PI);
            evo = lane < RE && ww >= 0 && ww < a.W && c < a.Cin ? (unsigned)((ww * a.Cin + c) * 2) : kOOB;
        }
        const int h = r0 + st, xh = h - 1;
        const bool drow = h < r1, xrow = xh >= 0 && xh < a.H && xh <= r1;
        const u4v dr = rsrc_words((const char*)a.dy + ln * db, drow ? db : 0);
        const u4v xr = rsrc_words((const char*)a.x + ln * xb, xrow ? xb : 0);
        const unsigned ds = drow ? (unsigned)(h * a.W * a.Cout * 2) : 0u, xs = xrow ? (unsigned)(xh * a.W * a.Cin * 2) : 0u;
        const unsigned base = lds0 + (unsigned)(slot * ROW * 16);
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            const unsigned part = (unsigned)(wt + WG * i) * 1024u;
            load_lds(dr, dvo[i], ds, base + part);
            if (MASK)
                load_lds(rsrc_words((const char*)a.dym + ln * db, drow ? db : 0), dvo[i], ds,
                         base + (unsigned)((RD + RX) * 16) + part);
        }
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            load_lds(xr, xvo[i], xs, base + (unsigned)(RD * 16) + (unsigned)(wt + WG * i) * 1024u);
        }
        // columns w0 - 1 and w0 + 32
        if (wt == 0 && lane < RE) load_lds(xr, evo, xs, base + (unsigned)((ROW - RE) * 16));
        slot = slot + 1 == NB ? 0 : slot + 1;
        if (++st == spi) {
            st = 0;
            ++it;
        }
    };
    // the wave's loads of the oldest stage (RS rows) in flight have arrived
    constexpr int LW = ND * (MASK ? 2 : 1) + NX;  // of a wave other than the first
    auto arrived = [&]() {
        if constexpr (WG == 1) {
            wait_loads<(NS - 2) * RS * (LW + 1)>();
            __builtin_amdgcn_wave_barrier();
        } else {
            if (wt == 0) {
                wait_loads<(NS - 2) * RS * (LW + 1)>();
            } else {
                wait_loads<(NS - 2) * RS * LW>();
            }
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
    };

    // fragment addresses in a staged row, bytes: group q of lanes takes
    // pixels 8 q .. 8 q + 7 (x: shifted by the tap), lane j of it addresses
    // pixel j / 4, channels 4 (j mod 4) .. + 3; the pixels -1 and 32 that a
    // shift reaches lie in the edge columns
    unsigned ad[ACO], ax[3][ACI], ax2[ACI];
    const unsigned edge = (unsigned)((ROW - RE) * 16);
#pragma unroll
    for (int i = 0; i < ACO; ++i) {
        const int p = 8 * q + (j >> 2);
        ad[i] = (unsigned)(p * BCO * 2 + granule<GO>(wco * ACO + i, p) * 32 + (j & 3) * 8);
    }
    auto xaddr = [&](int p, int g) {
        if (p < 0 || p > 31) return edge + (unsigned)((p > 31 ? BCI * 2 : 0) + g * 32 + (j & 3) * 8);
        return (unsigned)(RD * 16 + p * BCI * 2 + granule<GI>(g, p) * 32 + (j & 3) * 8);
    };
#pragma unroll
    for (int i = 0; i < ACI; ++i) {
#pragma unroll
        for (int w = 0; w < 3; ++w) ax[w][i] = xaddr(8 * q + (j >> 2) + w - 1, wci * ACI + i);
        ax2[i] = xaddr(8 * q + 4 + (j >> 2) + 1, wci * ACI + i);
    }
    // second four pixels of tap column 0: past the edge column on the lanes
    // that started in it
    unsigned ax0[ACI];
#pragma unroll
    for (int i = 0; i < ACI; ++i) ax0[i] = xaddr(8 * q + 4 + (j >> 2) - 1, wci * ACI + i);

    v4f acc[9][ACO][ACI], accb[ACO];
#pragma unroll
    for (int i = 0; i < ACO; ++i) {
        accb[i] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int k = 0; k < ACI; ++k) acc[t][i][k] = v4f{0.f, 0.f, 0.f, 0.f};
    }
    const bool with_bias = a.with_bias && ci0 == 0 && wci == 0;
    const v8bf ones = bf8(u4v{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
    int cslot = 0;          // buffer being computed
    int rows_i = 0;         // the item's rows of dy
    u4v keep{};             // the pixels of this lane's fragments before the image's edge
    v8bf d1[ACO], d2[ACO];  // dy fragments of the last two rows
#pragma unroll
    for (int i = 0; i < ACO; ++i) d1[i] = d2[i] = bf8(u4v{0u, 0u, 0u, 0u});

    // One row step: row h = first row + t of dy, x row h - 1.
    auto row_step = [&](auto masked, int t) __attribute__((always_inline)) {
        constexpr bool B = decltype(masked)::value;
        const unsigned row = lds0 + (unsigned)(cslot * ROW * 16);
        v8bf d0[ACO];
#pragma unroll
        for (int i = 0; i < ACO; ++i) {
            d0[i] = tr_frag(row + ad[i], row + ad[i] + 4 * BCO * 2);
            if (MASK) {
                const unsigned m = row + (unsigned)((RD + RX) * 16) + ad[i];
                d0[i] = bf8(relu_keep(__builtin_bit_cast(u4v, d0[i]), __builtin_bit_cast(u4v, tr_frag(m, m + 4 * BCO * 2))));
            }
        }
        if (with_bias) {
#pragma unroll
            for (int i = 0; i < ACO; ++i)
                accb[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d0[i], ones, accb[i], 0, 0, 0);
        }
        // x row h - 1 meets dy rows h (its taps of row -1), h - 1 and h - 2,
        // those of the run only.  Where dy is zero beyond the run or the
        // image's edge, x is zeroed too (it could be infinite).
        const unsigned m0 = t < rows_i ? ~0u : 0u, m1 = t >= 1 && t <= rows_i ? ~0u : 0u,
                       m2 = t >= 2 && t <= rows_i + 1 ? ~0u : 0u;
#pragma unroll
        for (int w = 0; w < 3; ++w)
#pragma unroll
            for (int m = 0; m < ACI; ++m) {
                const unsigned p = row + ax[w][m];
                u4v xf = __builtin_bit_cast(
                    u4v, tr_frag(p, w == 0 ? row + ax0[m] : (w == 2 ? row + ax2[m] : p + 4 * BCI * 2)));
                if (B && w == 0) xf &= keep;
                const v8bf x0 = bf8(B ? xf & m0 : xf), x1 = bf8(B ? xf & m1 : xf), x2 = bf8(B ? xf & m2 : xf);
#pragma unroll
                for (int i = 0; i < ACO; ++i) {
                    acc[w][i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d0[i], x0, acc[w][i][m], 0, 0, 0);
                    acc[3 + w][i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d1[i], x1, acc[3 + w][i][m], 0, 0, 0);
                    acc[6 + w][i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d2[i], x2, acc[6 + w][i][m], 0, 0, 0);
                }
            }
#pragma unroll
        for (int i = 0; i < ACO; ++i) {
            d2[i] = d1[i];
            d1[i] = d0[i];
        }
        cslot = cslot + 1 == NB ? 0 : cslot + 1;
    };
    // A stage: RS rows between two barriers.
    auto step = [&](auto masked, int t) __attribute__((always_inline)) {
        arrived();
        // into the buffers read in the stage before (rows past the last one
        // are zeros, so every stage issues the same number of loads)
#pragma unroll
        for (int k = 0; k < RS; ++k) load();
#pragma unroll
        for (int k = 0; k < RS; ++k) row_step(masked, t + k);
    };
#pragma unroll 1
    for (int i = 0; i < NB - RS; ++i) load();
#pragma unroll 1
    for (int i = 0; i < nit; ++i) {
        const int cit = ibeg + i, run = cit / a.strips, chunk = run % a.chunks;
        const int left = a.W - (cit - run * a.strips) * 32;
        rows_i = cit < iend ? min(a.rows, a.H - chunk * a.rows) : 0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            keep[e] = (8 * q + 2 * e < left ? 0x0000FFFFu : 0u) | (8 * q + 2 * e + 1 < left ? 0xFFFF0000u : 0u);
        // the steps that need no mask in a loop of their own (as branches of
        // one loop they would copy the accumulators)
        int t = 0;
#pragma unroll 1
        for (; t < 2; t += RS) step(std::integral_constant<bool, true>(), t);
        if (left >= 32) {
#pragma unroll 1
            for (; t + RS - 1 < rows_i; t += RS) step(std::integral_constant<bool, false>(), t);
        }
#pragma unroll 1
        for (; t < spi; t += RS) step(std::integral_constant<bool, true>(), t);
    }
    // the ring becomes the group sums' memory: no load may land in it later
    wait_loads<0>();
    __syncthreads();

    // sum of the k groups: groups [h, 2 h) hand their tiles to groups [0, h)
    v4f* red = reinterpret_cast<v4f*>(smem);
#pragma unroll
    for (int h = WK / 2; h >= 1; h /= 2) {
        // nothing to add where no group from h on had an item
        if (first(slice * WK + h) == first((slice + 1) * WK)) continue;
        v4f* sl = red + (int64_t)((kg % h) * WG + wt) * (TILES + ACO) * 64 + lane;
        if (kg >= h && kg < 2 * h) {
#pragma unroll
            for (int k = 0; k < 9; ++k)
#pragma unroll
                for (int i = 0; i < ACO; ++i)
#pragma unroll
                    for (int m = 0; m < ACI; ++m) sl[((k * ACO + i) * ACI + m) * 64] = acc[k][i][m];
#pragma unroll
            for (int i = 0; i < ACO; ++i) sl[(TILES + i) * 64] = accb[i];
        }
        __syncthreads();
        if (kg < h) {
#pragma unroll
            for (int k = 0; k < 9; ++k)
#pragma unroll
                for (int i = 0; i < ACO; ++i)
#pragma unroll
                    for (int m = 0; m < ACI; ++m) acc[k][i][m] += sl[((k * ACO + i) * ACI + m) * 64];
#pragma unroll
            for (int i = 0; i < ACO; ++i) accb[i] += sl[(TILES + i) * 64];
        }
        __syncthreads();
    }
    if (kg) return;
    const int64_t K = 9 * (int64_t)a.Cin, nw = a.Cout * K;
    float* out = a.part + slice * (nw + a.Cout);
#pragma unroll
    for (int i = 0; i < ACO; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int co = co0 + 16 * (wco * ACO + i) + 4 * q + r;
            if (co >= a.Cout) continue;
#pragma unroll
            for (int k = 0; k < 9; ++k)
#pragma unroll
                for (int m = 0; m < ACI; ++m) {
                    const int ci = ci0 + 16 * (wci * ACI + m) + j;
                    if (ci < a.Cin) out[co * K + k * a.Cin + ci] = acc[k][i][m][r];
                }
            if (with_bias && j == 0) out[nw + co] = accb[i][r];
        }
}

// The general weight gradient, for operands that conv_wgrad does not
// take (unaligned, or an image beyond its 31-bit offsets) and where it is the
// faster one (bwd_w_general).  Each
// 64-pixel step loads dy (64 px x 64 co) and the shifted x (64 px x 64 ci)
// with 16-byte loads (8 channels of one pixel) and stores them TRANSPOSED
// in LDS, [channel][pixel] with rows padded to 72 elements, so that every
// MFMA fragment (8 consecutive pixels of one channel) is one 16-byte LDS
// read.  Lane l of wave v stages the pixel pair 2(l & 31), 2(l & 31) + 1
// of channel group (l >> 5) + 2v, the pair's two values of a channel in
// one 32-bit write: for a fixed element the 64 lanes write two rows 8
// apart and 32 consecutive pixel pairs (16-bit writes of single pixels
// were 3-6 % slower).  dy is multiplied on load by the ReLU mask of dym
// when given.
// A workgroup owns one tap, 64 co x 64 ci and one slice of pixels; wave
// (wrow, wcol) = (v >> 1, v & 1) computes co 32 wrow .. 32 wrow + 31 x ci
// 32 wcol .. 32 wcol + 31 (2 x 2 tiles of 16 x 16, two 32-pixel MFMA steps per stage: four
// fragment reads per four MFMAs).  LDS holds two stages: the next step is
// written into the other buffer while this one's MFMAs run, one barrier per
// step.  The workgroups of tap 0 and the first ci block also form the bias
// gradient's slice sums, sum_p dy[p][co], on the waves with wcol = 0, with
// one more MFMA per co tile against a ones operand (every column of the
// tile then holds the row sum).  Slices write partial sums that reduce_slices
// adds in a fixed order.
constexpr int kStep = 64;
constexpr int kLds = kStep + 8;

__global__ __launch_bounds__(256) void conv_bwd_w(const uint16_t* __restrict__ x, const uint16_t* __restrict__ dy,
                                                  const uint16_t* __restrict__ dym, float* __restrict__ part,
                                                  int bias, int N, int H, int W, int Cin, int Cout, int64_t chunk) {
    __shared__ __align__(16) uint16_t sdy[2][64][kLds];
    __shared__ __align__(16) uint16_t sx[2][64][kLds];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wrow = wave >> 1, wcol = wave & 1;
    const int ncb = (Cout + 63) / 64;
    // logical workgroup = slice x (ci block, tap, co block), the 9 taps and
    // channel blocks of one slice adjacent (they read the same dy and x)
    const int G = ncb * 9 * ((Cin + 63) / 64);
    const int L = xcd_band();
    const int slice = L / G;
    int gy = L - slice * G;
    const int cb = gy % ncb;
    gy /= ncb;
    const int tap = gy % 9;
    const int ib = gy / 9;
    const int co0 = cb * 64, ci0 = ib * 64, dh = tap / 3 - 1, dw = tap % 3 - 1;
    const int64_t P = (int64_t)N * H * W;
    const int64_t pbeg = (int64_t)slice * chunk;
    const int64_t pend = std::min<int64_t>(P, pbeg + chunk);
    v4f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    v4f accb[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
    const bool with_bias = bias && tap == 0 && ib == 0 && wcol == 0;
    const u4v ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};  // eight bf16 1.0
    // Thread t loads channels g8 .. g8 + 7 (g8 = 8 (t & 7)) of pixels
    // pl = t >> 3 and pl + 32 of the step: eight consecutive lanes read one
    // pixel's 64 channels, 128 contiguous bytes.  Lanes t and t ^ 8 hold
    // adjacent pixels 2m, 2m + 1 (m = pl >> 1); one DPP row rotation by 8
    // swaps half of each one's channels, after which the even lane holds both
    // pixels of channels g8 .. g8 + 3 and the odd lane those of g8 + 4 ..
    // g8 + 7, written as 32-bit pixel pairs.
    const int g8 = (threadIdx.x & 7) * 8, pl = threadIdx.x >> 3;
    const bool odd = pl & 1;
    const bool co_in = co0 + g8 < Cout, ci_in = ci0 + g8 < Cin;
    // the next step's operands are loaded once this step's are in LDS, so
    // the loads run during the barrier and the MFMAs
    u4v ldy[2], lm[2], lx[2];
    // (n, h, wc) of the thread's first pixel of the next load, divided out
    // once and then advanced by kStep pixels per step (64-bit divisions per
    // pixel and step cost more than the step's MFMAs)
    int pn, ph, pwc;
    {
        const int64_t p0 = pbeg + pl, t = p0 / W;
        pwc = (int)(p0 - t * W);
        pn = (int)(t / H);
        ph = (int)(t - (int64_t)pn * H);
    }
    auto advance = [&](int& n, int& h, int& wc, int d) {
        wc += d;
        while (wc >= W) {
            wc -= W;
            if (++h == H) {
                h = 0;
                ++n;
            }
        }
    };
    auto load = [&](int64_t pc) {
        int n = pn, h = ph, wc = pwc;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int64_t p = pc + pl + 32 * k;
            if (k) advance(n, h, wc, 32);
            ldy[k] = u4v{0u, 0u, 0u, 0u};
            lx[k] = u4v{0u, 0u, 0u, 0u};
            lm[k] = u4v{~0u, ~0u, ~0u, ~0u};
            if (p < pend) {
                if (co_in) {
                    ldy[k] = *reinterpret_cast<const u4v*>(dy + p * Cout + co0 + g8);
                    if (dym) lm[k] = *reinterpret_cast<const u4v*>(dym + p * Cout + co0 + g8);
                }
                const int hh = h + dh, ww = wc + dw;
                if (ci_in && hh >= 0 && hh < H && ww >= 0 && ww < W)
                    lx[k] = *reinterpret_cast<const u4v*>(x + (((int64_t)n * H + hh) * W + ww) * Cin + ci0 + g8);
            }
        }
        advance(pn, ph, pwc, kStep);
    };
    // LDS layout [channel R][pixel], the 16-byte chunk c (8 pixels) of row R
    // stored at chunk c ^ (R >> 3): the pair writes of the eight channel
    // groups and the fragment reads of 16 consecutive rows spread over the
    // banks
    auto pair_col = [](int R, int m) { return ((((m >> 2) ^ (R >> 3)) << 2) | (m & 3)) * 2; };
    auto swap8 = [](unsigned v) { return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xF, 0xF, false); };
    auto put = [&](uint16_t (*sb)[kLds], const u4v& v, int k) {
        const unsigned r0 = swap8(odd ? v[0] : v[2]), r1 = swap8(odd ? v[1] : v[3]);
        const unsigned o0 = odd ? v[2] : v[0], o1 = odd ? v[3] : v[1];
        const unsigned e0 = odd ? r0 : o0, e1 = odd ? r1 : o1;  // pixel 2m
        const unsigned d0 = odd ? o0 : r0, d1 = odd ? o1 : r1;  // pixel 2m + 1
        const int m = (pl >> 1) + 16 * k;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int R = g8 + 4 * odd + j, sh = 16 * (j & 1);
            const unsigned ev = j < 2 ? e0 : e1, ov = j < 2 ? d0 : d1;
            *reinterpret_cast<unsigned*>(&sb[R][pair_col(R, m)]) = ((ev >> sh) & 0xFFFFu) | (((ov >> sh) & 0xFFFFu) << 16);
        }
    };
    // LDS stage from the load registers (the ReLU mask applied here)
    auto stage = [&](int buf) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            put(sdy[buf], dym ? relu_keep(ldy[k], lm[k]) : ldy[k], k);
            put(sx[buf], lx[k], k);
        }
    };
    if (pbeg < pend) {
        load(pbeg);
        stage(0);
        if (pbeg + kStep < pend) load(pbeg + kStep);
    }
    __syncthreads();
    int buf = 0;
    for (int64_t pc = pbeg; pc < pend; pc += kStep) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int kc = 4 * kk + (lane >> 4);  // 8-pixel chunk of the fragment
            v8bf a[2], bv[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int ra = 32 * wrow + 16 * i + (lane & 15), rb = 32 * wcol + 16 * i + (lane & 15);
                a[i] = bf8(*reinterpret_cast<const u4v*>(&sdy[buf][ra][8 * (kc ^ (ra >> 3))]));
                bv[i] = bf8(*reinterpret_cast<const u4v*>(&sx[buf][rb][8 * (kc ^ (rb >> 3))]));
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], bv[j], acc[i][j], 0, 0, 0);
            if (with_bias) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    accb[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], bf8(ones), accb[i], 0, 0, 0);
            }
        }
        // the other buffer was last read before the previous barrier
        if (pc + kStep < pend) {
            stage(buf ^ 1);
            if (pc + 2 * kStep < pend) load(pc + 2 * kStep);
        }
        __syncthreads();
        buf ^= 1;
    }
    const int64_t K = 9 * (int64_t)Cin;
    float* out = part + slice * (Cout * K + Cout);   // a slice: the weights' sums, then the bias's
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int ci = ci0 + 32 * wcol + 16 * j + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int co = co0 + 32 * wrow + 16 * i + 4 * (lane >> 4) + r;
                if (co < Cout && ci < Cin) out[co * K + tap * Cin + ci] = acc[i][j][r];
            }
        }
    if (with_bias && (lane & 15) == 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int co = co0 + 32 * wrow + 16 * i + 4 * (lane >> 4) + r;
                if (co < Cout) out[Cout * K + co] = accb[i][r];
            }
    }
}

// out[i] = sum over s of part[s][i]: eight interleaved partial sums a_j
// (slices s = j mod 8 in ascending order, from 0), then a fixed tree of the
// eight; the order is the same on every call.  A workgroup takes 32
// consecutive outputs, thread t the partial sum j = t >> 5 of output t & 31
// (eight times the threads of one per output: the sums are long, the
// outputs few), and the tree runs from LDS.  A slice is `stride` values: n1
// for out, the rest up to n for out2 (weights and bias in one launch).
__global__ __launch_bounds__(256) void reduce_slices(const float* __restrict__ part, int64_t stride, int S, int64_t n,
                                                     float* __restrict__ out, int64_t n1, float* __restrict__ out2) {
    __shared__ float sa[8][33];
    const int j = threadIdx.x >> 5, ii = threadIdx.x & 31;
    const int64_t i = (int64_t)blockIdx.x * 32 + ii;
    float a = 0.f;
    if (i < n) {
#pragma unroll 4
        for (int s = j; s < S; s += 8) a += part[(int64_t)s * stride + i];
    }
    sa[j][ii] = a;
    __syncthreads();
    if (j == 0 && i < n) {
        const float v = ((sa[0][ii] + sa[1][ii]) + (sa[2][ii] + sa[3][ii])) + ((sa[4][ii] + sa[5][ii]) + (sa[6][ii] + sa[7][ii]));
        if (i < n1) out[i] = v; else out2[i - n1] = v;
    }
}

// ------------------------------------------------------ U-Net plumbing
// The decoder input: out[n][h][w][0:C1] = lo[n][h/2][w/2][:] (nearest-
// neighbour upsampling of the coarser level) and out[n][h][w][C1:C1+C2] =
// skip[n][h][w][:] (the skip connection), one pass of 16-byte pieces of 8
// channels (G1 = C1 / 8, G2 = C2 / 8 pieces per pixel); n pieces in all.
__global__ __launch_bounds__(256) void up_cat(const uint16_t* __restrict__ lo, const uint16_t* __restrict__ skip,
                                              uint16_t* __restrict__ out, int H, int W, int G1, int G2, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int G = G1 + G2;
    const int64_t p = i / G;
    const int g = (int)(i - p * G);
    u4v v;
    if (g < G1) {
        const int w = (int)(p % W);
        const int64_t t = p / W;
        const int h = (int)(t % H);
        const int64_t nn = t / H;
        v = reinterpret_cast<const u4v*>(lo)[((nn * (H / 2) + h / 2) * (W / 2) + w / 2) * G1 + g];
    } else {
        v = reinterpret_cast<const u4v*>(skip)[p * G2 + (g - G1)];
    }
    reinterpret_cast<u4v*>(out)[i] = v;
}

__device__ __forceinline__ float bf_lo(unsigned v) { return __builtin_bit_cast(float, v << 16); }
__device__ __forceinline__ float bf_hi(unsigned v) { return __builtin_bit_cast(float, v & 0xFFFF0000u); }

// Backward of up_cat: dlo[n][h][w][c] = the sum of dout[n][2h+a][2w+b][c]
// over the 2 x 2 block, taken in the order of the gradients of the two
// repeats (along w, then along h): the two columns of each row summed and
// rounded to bf16, then the two rows summed and rounded; dskip =
// dout[..., C1:].  With lo_y (lo, the output of a ReLU), dlo is zeroed where
// lo_y is not > 0: that ReLU's backward.  Pieces [0, n_lo) are dlo's,
// [n_lo, n_lo + n_skip) dskip's.
__global__ __launch_bounds__(256) void up_cat_bwd(const uint16_t* __restrict__ dout,
                                                  const uint16_t* __restrict__ lo_y, uint16_t* __restrict__ dlo,
                                                  uint16_t* __restrict__ dskip, int H, int W, int G1, int G2,
                                                  int64_t n_lo, int64_t n_skip) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int G = G1 + G2;
    const u4v* d = reinterpret_cast<const u4v*>(dout);
    if (i < n_lo) {
        const int64_t q = i / G1;
        const int g = (int)(i - q * G1);
        const int w2 = W / 2, h2 = H / 2;
        const int w = (int)(q % w2);
        const int64_t t = q / w2;
        const int h = (int)(t % h2);
        const int64_t nn = t / h2;
        const int64_t p00 = (nn * H + 2 * h) * W + 2 * w;
        const u4v a = d[p00 * G + g], b = d[(p00 + 1) * G + g];
        const u4v c = d[(p00 + W) * G + g], e = d[(p00 + W + 1) * G + g];
        u4v r;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float t0 = bf_lo(to_bf16(bf_lo(a[k]) + bf_lo(b[k]))), t1 = bf_lo(to_bf16(bf_lo(c[k]) + bf_lo(e[k])));
            const float u0 = bf_lo(to_bf16(bf_hi(a[k]) + bf_hi(b[k]))), u1 = bf_lo(to_bf16(bf_hi(c[k]) + bf_hi(e[k])));
            r[k] = (unsigned)to_bf16(t0 + t1) | ((unsigned)to_bf16(u0 + u1) << 16);
        }
        if (lo_y) {
            const u4v m = reinterpret_cast<const u4v*>(lo_y)[i];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                r[k] &= (bf_lo(m[k]) > 0.f ? 0x0000FFFFu : 0u) | (bf_hi(m[k]) > 0.f ? 0xFFFF0000u : 0u);
        }
        reinterpret_cast<u4v*>(dlo)[i] = r;
    } else if (i < n_lo + n_skip) {
        const int64_t j = i - n_lo;
        const int64_t p = j / G2;
        const int g = (int)(j - p * G2);
        reinterpret_cast<u4v*>(dskip)[j] = d[p * G + G1 + g];
    }
}

// out = dy where y > 0 (as a float: -0 and NaN are not), else 0: the
// backward mask of a ReLU whose bf16 output is y; n8 pieces of 8 values.
__global__ __launch_bounds__(256) void relu_mask(const uint16_t* __restrict__ dy, const uint16_t* __restrict__ y,
                                                 uint16_t* __restrict__ out, int64_t n8) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n8) return;
    const u4v v = reinterpret_cast<const u4v*>(dy)[i], m = reinterpret_cast<const u4v*>(y)[i];
    u4v r;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const unsigned lo = bf_lo(m[k]) > 0.f ? 0x0000FFFFu : 0u;
        const unsigned hi = bf_hi(m[k]) > 0.f ? 0xFFFF0000u : 0u;
        r[k] = v[k] & (lo | hi);
    }
    reinterpret_cast<u4v*>(out)[i] = r;
}

// Gradient of a ReLU output s [N][H][W][C] that feeds both a 2 x 2 average
// pool and a skip connection: out = where(s > 0, g, 0) with g = bf16(pool
// gradient + dskip), the pool gradient dp[n][h/2][w/2][c] / 4 rounded to
// bf16 first (the mean's backward), then added to dskip and rounded (the
// sum of a tensor's two gradients), then masked (the ReLU's backward).
// dskip's pixels are Gs pieces of 8 channels apart (a channel slice of a
// wider gradient may be read in place).  One 8-channel piece per thread.
__global__ __launch_bounds__(256) void pool_skip_bwd(const uint16_t* __restrict__ dp,
                                                     const uint16_t* __restrict__ dskip, int Gs,
                                                     const uint16_t* __restrict__ s, uint16_t* __restrict__ out,
                                                     int H, int W, int G, int64_t n8) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n8) return;
    const int64_t p = i / G;
    const int g = (int)(i - p * G);
    const int w = (int)(p % W);
    const int64_t t = p / W;
    const int h = (int)(t % H);
    const int64_t nn = t / H;
    const int64_t q = (nn * (H / 2) + h / 2) * (W / 2) + w / 2;
    const u4v a = reinterpret_cast<const u4v*>(dp)[q * G + g];
    const u4v b = reinterpret_cast<const u4v*>(dskip)[p * Gs + g], m = reinterpret_cast<const u4v*>(s)[i];
    u4v r;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float plo = bf_lo(to_bf16(bf_lo(a[k]) * 0.25f)), phi = bf_lo(to_bf16(bf_hi(a[k]) * 0.25f));
        const unsigned v = (unsigned)to_bf16(plo + bf_lo(b[k])) | ((unsigned)to_bf16(phi + bf_hi(b[k])) << 16);
        r[k] = v & ((bf_lo(m[k]) > 0.f ? 0x0000FFFFu : 0u) | (bf_hi(m[k]) > 0.f ? 0xFFFF0000u : 0u));
    }
    reinterpret_cast<u4v*>(out)[i] = r;
}

// y[n][h][w][c] = the mean of x over each 2 x 2 block: the four values added
// in the order of torch's mean over those two axes (row by row, in float),
// times 1/4, rounded to bf16.  One 8-channel piece per thread; at batch 64
// the three pools of the network take 46 us (torch's mean 97).
__global__ __launch_bounds__(256) void avg_pool2(const uint16_t* __restrict__ x, uint16_t* __restrict__ y, int W, int G,
                                                 int64_t n8) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n8) return;
    const int64_t q = i / G;               // output pixel
    const int g = (int)(i - q * G), w2 = W / 2;
    const int64_t row = q / w2;            // output row of the batch: input rows 2 row, 2 row + 1
    const int w = (int)(q - row * w2);
    const u4v* const d = reinterpret_cast<const u4v*>(x) + (2 * row * W + 2 * w) * G + g;
    const u4v a = d[0], b = d[G], c = d[(int64_t)W * G], e = d[(int64_t)(W + 1) * G];
    u4v r;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float lo = ((bf_lo(a[k]) + bf_lo(b[k])) + bf_lo(c[k])) + bf_lo(e[k]);
        const float hi = ((bf_hi(a[k]) + bf_hi(b[k])) + bf_hi(c[k])) + bf_hi(e[k]);
        r[k] = (unsigned)to_bf16(lo * 0.25f) | ((unsigned)to_bf16(hi * 0.25f) << 16);
    }
    reinterpret_cast<u4v*>(y)[i] = r;
}

// The network's input: per pixel psi, ux s, uy s, solid, lm, th and two
// zeros, each rounded to bf16 (s the reciprocal of the velocity scale, lm and
// th one value per sample or for all).  One 16-byte store per thread, where
// ten tensor operations each made a pass over 4-byte channels.
__global__ __launch_bounds__(256) void net_inputs(const float* __restrict__ psi, const float* __restrict__ ux,
                                                  const float* __restrict__ uy, const float* __restrict__ solid,
                                                  const float* __restrict__ lm, const float* __restrict__ th, float s,
                                                  uint16_t* __restrict__ out, int64_t cells, int64_t solid_n,
                                                  int lm_n, int th_n, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t smp = i / cells;
    const float so = solid[solid_n == n ? i : i - smp * cells];
    auto two = [](float a, float b) { return (unsigned)to_bf16(a) | ((unsigned)to_bf16(b) << 16); };
    reinterpret_cast<u4v*>(out)[i] = u4v{two(psi[i], ux[i] * s), two(uy[i] * s, so),
                                         two(lm[lm_n > 1 ? smp : 0], th[th_n > 1 ? smp : 0]), 0u};
}

// The training loss and its gradient, per pixel with o = the network's output
// (pixels ld floats apart), d = (psi0 + o0) - psi1, x = (v0 + o) - v1:
//   loss = sum d^2 wf / w + lambda (sum |x|^2 wf / w)
// net_loss adds in double (a partial sum per workgroup, added in a fixed
// order by net_loss_sum) and writes d, x0, x1 to res (if given), all that the
// gradient needs: net_loss_bwd forms its products in the order of autograd's
// backward of that expression, so the gradients are its bits.  At batch 64 (2.1 M
// pixels) net_loss takes 24 us and net_loss_bwd 10, bound by memory; forming the
// residuals from the inputs again took 20 and 24, and kept those from changing
// before the backward pass; as some forty tensor operations 250.
struct LossArgs {
    const float *out, *psi0, *psi1, *v0, *v1, *wf;
    float* res;
    int64_t n;
    int ld;
};
constexpr int kLossBlocks = 1024;

__global__ __launch_bounds__(256) void net_loss(LossArgs a, double* __restrict__ part) {
    __shared__ double sh[2][4];
    double p = 0.0, q = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * 256) {
        const float* const o = a.out + i * a.ld;
        const float2 u = reinterpret_cast<const float2*>(a.v0)[i], v = reinterpret_cast<const float2*>(a.v1)[i];
        const float d = (a.psi0[i] + o[0]) - a.psi1[i], x0 = (u.x + o[1]) - v.x, x1 = (u.y + o[2]) - v.y;
        if (a.res) {
            a.res[3 * i] = d;
            a.res[3 * i + 1] = x0;
            a.res[3 * i + 2] = x1;
        }
        const float wf = a.wf[i];
        p += (double)(d * d * wf);
        q += (double)((x0 * x0 + x1 * x1) * wf);
    }
    for (int m = 32; m; m >>= 1) {
        p += __shfl_xor(p, m, 64);
        q += __shfl_xor(q, m, 64);
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        sh[0][wave] = p;
        sh[1][wave] = q;
    }
    __syncthreads();
    if (threadIdx.x < 2)
        part[2 * blockIdx.x + threadIdx.x] =
            (sh[threadIdx.x][0] + sh[threadIdx.x][1]) + (sh[threadIdx.x][2] + sh[threadIdx.x][3]);
}

__global__ __launch_bounds__(64) void net_loss_sum(const double* __restrict__ part, int blocks,
                                                   const float* __restrict__ w, float lambda,
                                                   float* __restrict__ loss) {
    double p = 0.0, q = 0.0;
    for (int i = threadIdx.x; i < blocks; i += 64) {
        p += part[2 * i];
        q += part[2 * i + 1];
    }
    for (int m = 32; m; m >>= 1) {
        p += __shfl_xor(p, m, 64);
        q += __shfl_xor(q, m, 64);
    }
    if (threadIdx.x == 0) *loss = (float)p / *w + lambda * ((float)q / *w);
}

__global__ __launch_bounds__(256) void net_loss_bwd(const float* __restrict__ res, const float* __restrict__ wf,
                                                    const float* __restrict__ w, float lambda,
                                                    const float* __restrict__ g, float* __restrict__ dout, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float gp = *g / *w * wf[i], gu = *g * lambda / *w * wf[i];
    dout[3 * i] = gp * (2.f * res[3 * i]);
    dout[3 * i + 1] = gu * (2.f * res[3 * i + 1]);
    dout[3 * i + 2] = gu * (2.f * res[3 * i + 2]);
}

int check(int N, int H, int W, int Cin, int Cout) {
    if (N < 1 || H < 1 || W < 1 || Cin < 8 || Cout < 1) return fail(FDS_E_ARG, "bad shape");
    if (Cin % 8) return fail(FDS_E_ARG, "Cin must be a multiple of 8");
    if ((int64_t)N * H * W >= ((int64_t)1 << 40)) return fail(FDS_E_ARG, "too many pixels");
    return FDS_OK;
}

// Work split of the weight gradient: the channel block by the layer's
// channels, then row runs and slices, at most one workgroup per CU.  The
// split with the least cost of the busiest k group is taken, in row steps
// (about 1 us each with every CU busy): a run of `rows` rows costs rows + 2,
// and the partial sum of a block, written and read back, 10/256 for 64 x 64
// channels (256 of them, 38 MB: 7 us to write, 2.5 more in reduce_slices).
// Too few slices show: 128 -> 128 channels at 64 x 16 x 32 take 32 us with
// 64 slices of 10 steps and 37 with 32 of 18.
struct BwdWPlan {
    int kind;       // instantiation, launch_wgrad
    int bco, bci, wk;
    int ncb, nib;
    int strips, chunks, rows, items, slices;
    float us;       // what it takes with reduce_slices (below)
};

// The partial sums of S slices, MB.
float partial_mb(int64_t S, int Cin, int Cout) { return (float)(S * Cout * (9 * (int64_t)Cin + 1)) * 4e-6f; }

BwdWPlan bwd_w_plan(int N, int H, int W, int Cin, int Cout) {
    BwdWPlan pl{};
    if (Cout <= 16) pl = BwdWPlan{5, 16, 32, 8};
    else if (Cin <= 16) pl = BwdWPlan{4, 32, 16, 8};
    else if (Cout > 32 && Cin > 32) pl = BwdWPlan{0, 64, 64, 2};
    else if (Cout > 32) pl = BwdWPlan{1, 64, 32, 4};
    else if (Cin > 32 && Cin % 64 == 0) pl = BwdWPlan{2, 32, 64, 4};
    else pl = BwdWPlan{3, 32, 32, 8};
    pl.ncb = (Cout + pl.bco - 1) / pl.bco;
    pl.nib = (Cin + pl.bci - 1) / pl.bci;
    pl.strips = (W + 31) / 32;
    const int64_t nblk = (int64_t)pl.ncb * pl.nib;
    const int64_t cap = std::max<int64_t>(1, 256 / nblk);
    const int64_t sum = nblk * pl.bco * pl.bci * 5 / 8;  // 65536ths of a step per slice
    int64_t best = -1, steps = 0;
    for (int c = 1; c <= H && c <= 256; c = c < 4 ? c + 1 : c + c / 2) {
        const int rows = (H + c - 1) / c, chunks = (H + rows - 1) / rows;
        const int64_t items = (int64_t)N * pl.strips * chunks;
        int64_t per = (items + cap * pl.wk - 1) / (cap * pl.wk);  // items of the busiest group
        for (int k = 0; k < 8; ++k, per += (per + 1) / 2) {
            const int64_t slices = (items + per * pl.wk - 1) / (per * pl.wk);
            const int64_t cost = per * (rows + 2) * 65536 + slices * sum;
            if (best < 0 || cost < best) {
                best = cost;
                pl.chunks = chunks;
                pl.rows = rows;
                pl.items = (int)items;
                pl.slices = (int)slices;
                steps = per * (rows + 2);
            }
            if (slices == 1) break;
        }
    }
    const bool thin = pl.kind >= 4;
    pl.us = (thin ? 10.f : 14.5f) + (thin ? 0.75f : 1.05f) * (float)steps + 3.6f / 256 * (float)(pl.slices * nblk) +
            0.26f * partial_mb(pl.slices, Cin, Cout);
    return pl;
}

// The general kernel's split: pixel slices of whole 64-pixel steps, about
// 2048 workgroups (1..256 slices), at least 64 to 512 pixels each: what takes
// the least time.
//
// Which of the two kernels a layer takes is the smaller of their times, `us`.
// conv_wgrad reads strips of 32 columns and needs some 14 us before its first
// step counts, so narrow images and small problems are the general kernel's:
// 96 -> 96 channels on 67 x 201 x 2 take 79 us there and 159 in conv_wgrad,
// 64 -> 64 on 64 x 16 x 8 16 and 28, 32 -> 32 on 1 x 64 x 64 10 and 18; on
// 64 x 64 x 64 64 -> 64 takes 88 and 40.  Both times
// are fits of 513 measured layers of 256 to 120,000 pixels (19 pairs of
// channels, 27 sizes; the general kernel at four slice heights each) and
// within 6 % of them (rms): steps of a workgroup, rounds of workgroups over
// the CUs, and the bytes of the partial sums.  A narrow image's pixel
// coordinates advance in a loop, hence the terms with 1 / W.
struct BwdWGeneral {
    int64_t chunk;
    int S;
    float us;
};

BwdWGeneral bwd_w_general(int N, int H, int W, int Cin, int Cout) {
    const int64_t P = (int64_t)N * H * W;
    const int64_t per_slice = (int64_t)((Cout + 63) / 64) * 9 * ((Cin + 63) / 64);
    const int64_t want = std::min<int64_t>(256, std::max<int64_t>(1, (2048 + per_slice - 1) / per_slice));
    const int64_t c0 = ((P + want - 1) / want + kStep - 1) / kStep * kStep;
    BwdWGeneral best{0, 0, 0.f};
    for (int64_t least = 64; least <= 512; least *= 2) {
        const int64_t c = std::max(c0, least), S = (P + c - 1) / c;
        const float steps = (float)((std::min(c, P) + kStep - 1) / kStep);
        const float more = std::max(0.f, (float)(S * per_slice) / 256.f - 1.f);   // rounds beyond one
        const float us = 7.3f + steps * (1.07f + 0.29f * more + (3.4f + 0.84f * more) / (float)W) + 0.97f * more +
                         0.4f * partial_mb(S, Cin, Cout);
        if (!best.S || us < best.us) best = BwdWGeneral{c, (int)S, us};
    }
    return best;
}

}  // namespace

namespace {
// Two workgroups per CU.  With one chunk of input channels a launch has about
// that many (the thin kernel, whose LDS is small, twice as many), each with
// an equal run of blocks, so the weights are staged once per run: 51 us
// against 54 for one block per workgroup (32 -> 32 channels, 64 x 128 x
// 256).  With more chunks the weights are staged per chunk anyway, and one
// block per workgroup balances better: 138 us against 154 (96 -> 32).
constexpr int kRun = 512;

template <int R, int CT, int WC, int WP, int PF, bool MASK>
void launch_tile(ConvArgs a, hipStream_t st) {
    using T = Tile<R, CT, WC, WP>;
    a.hb = (a.H + T::BR - 1) / T::BR;
    a.wb = (a.W + T::BW - 1) / T::BW;
    a.npx = a.N * a.hb * a.wb;
    a.ncb = (a.Cout + T::BC - 1) / T::BC;
    const int total = a.npx * a.ncb, per = a.Cin == 32 ? (total + kRun - 1) / kRun : 1;
    const dim3 grid((total + per - 1) / per);
    if (a.y32)
        hipLaunchKernelGGL((conv_tile<R, CT, WC, WP, PF, MASK, true>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((conv_tile<R, CT, WC, WP, PF, MASK, false>), grid, dim3(256), 0, st, a);
}

template <int R, int CT, int WC, int CG, bool MASK>
void launch_thin(ConvArgs a, hipStream_t st) {
    using T = Tile<R, CT, WC, 4>;
    a.hb = (a.H + T::BR - 1) / T::BR;
    a.wb = (a.W + T::BW - 1) / T::BW;
    a.npx = a.N * a.hb * a.wb;
    a.ncb = (a.Cout + T::BC - 1) / T::BC;
    const int total = a.npx * a.ncb, per = (total + 2 * kRun - 1) / (2 * kRun);
    const dim3 grid((total + per - 1) / per);
    if (a.y32)
        hipLaunchKernelGGL((conv_tile_thin<R, CT, WC, CG, MASK, true>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((conv_tile_thin<R, CT, WC, CG, MASK, false>), grid, dim3(256), 0, st, a);
}

// Blocks of one configuration.
template <int R, int CT, int WC, int WP>
int64_t blocks_of(const ConvArgs& a) {
    using T = Tile<R, CT, WC, WP>;
    return (int64_t)a.N * ((a.H + T::BR - 1) / T::BR) * ((a.W + T::BW - 1) / T::BW) * ((a.Cout + T::BC - 1) / T::BC);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Whether images of up to eight columns are conv_fwd's: the staged kernels
// compute 32 columns of them, conv_fwd only the pixels there are.  Estimates
// of both, us (Cout outputs of Cin channels; fits of 336 measured layers of 1
// to 8 columns and 1,000 to 65,536 rows):
//   48 -> 96   on 67 x 201 x 2   25 here, 51 staged    on 64 x 64 x 2    23, 13
//   64 -> 64   on 256 x 256 x 1  28, 135               on 64 x 64 x 4    28, 12
//   16 -> 96   on 67 x 201 x 2   18, 24                on 64 x 256 x 8   38, 25
//   128 -> 128 on 256 x 256 x 4  253, 471              on 64 x 256 x 8   140, 126
bool narrow(int N, int H, int W, int Cin, int Cout, bool mask) {
    if (W > 8) return false;
    const double rows = (double)N * ((H + 7) / 8 * 8), cc = (double)Cin * Cout;
    const double staged = 4. + rows * std::max(cc / (Cin % 32 ? 1.5e6 : 2.3e6), 1. / 3300);
    const double rate = (Cout >= 64 ? 1.2e7 : (Cout >= 32 ? 1e7 : 2.5e6)) * (mask ? 0.5 : 1.);
    const double outputs = (double)N * H * W * Cout;   // few input channels: bound by the stores
    return std::max(15. + 0.19 * Cin, std::max(outputs * Cin / rate, outputs / 3.3e5)) < 0.9 * staged;
}

template <bool MASK>
void launch_fwd(const uint16_t* x, const uint16_t* xm, const uint16_t* w, const float* bias, float* y32, uint16_t* y16,
                int N, int H, int W, int Cin, int Cout, int relu, hipStream_t st) {
    const int64_t P = (int64_t)N * H * W;
    const ConvArgs a{x, xm, w, bias, y32, y16, N, H, W, Cin, Cout, relu, 0, 0, 0, 0};
    // the staged kernels address one image and the weights by 31-bit byte
    // offsets, count blocks in 32 bits and store 16 bytes at once
    const bool staged = !(y32 && y16) && (int64_t)H * W * Cin * 2 < kMaxBytes &&
                        (int64_t)H * W * Cout * (y32 ? 4 : 2) < kMaxBytes && (int64_t)Cout * 9 * Cin * 2 < kMaxBytes &&
                        P < ((int64_t)1 << 28) && P * ((Cout + 15) / 16) < ((int64_t)1 << 31) && aligned16(x) && aligned16(xm) && aligned16(w) && aligned16(y32) &&
                        aligned16(y16) && !narrow(N, H, W, Cin, Cout, MASK);
    if (staged && Cin % 32 == 0) {
        // The block shape, by what was measured at batch 64 on 128 x 256
        // (thin layers) to 32 x 64 (wide ones), us a layer for the shape
        // taken and the next best; the kernel before these in parentheses:
        //   32 -> 8     35.7, 39.7 (110)    96 -> 32    138, 146 (374)
        //   32 -> 32    51, 55 (177)        32 -> 96    137, 162 (512)
        //   32 -> 64    23.5, 26.6 (76)     64 -> 192   113, 117 (359)
        //   192 -> 64   106, 102 (260)      256 -> 128  69, 67 (162)
        // Larger blocks read less LDS per MFMA and less halo; below 512 of
        // them (two per CU; 256, one per CU, for the smaller shapes) CUs
        // stay idle and the next smaller shape is faster, e.g. 128 -> 128
        // on 64 x 16 x 32: 12.4 us against 14.5, and on 1 x 16 x 32: 6 us
        // against 9 (32).  The masked kernels hold the mask in registers
        // too and take the shapes that do not spill with it.
        if (!MASK) {
            if (Cout <= 16 && blocks_of<4, 2, 1, 4>(a) >= kRun) return launch_tile<4, 2, 1, 4, 1, false>(a, st);
            if (Cout <= 32 && Cin >= 96 && blocks_of<4, 2, 2, 4>(a) >= kRun)
                return launch_tile<4, 2, 2, 4, 1, false>(a, st);
            if (Cout % 96 == 0 && blocks_of<2, 2, 6, 4>(a) >= kRun)
                return Cin == 32 ? launch_tile<2, 2, 6, 4, 0, false>(a, st) : launch_tile<2, 2, 6, 4, 1, false>(a, st);
        }
        if (Cout > 32 && blocks_of<2, 2, 4, 4>(a) >= kRun) return launch_tile<2, 2, 4, 4, 1, MASK>(a, st);
        if (blocks_of<2, 2, 2, 4>(a) >= kRun / 2) return launch_tile<2, 2, 2, 4, 2, MASK>(a, st);
        if (!MASK && blocks_of<2, 1, 2, 4>(a) >= kRun / 2) return launch_tile<2, 1, 2, 4, 2, false>(a, st);
        return launch_tile<1, 1, 2, 4, 2, MASK>(a, st);
    }
    if (staged && Cin <= 56) {
        switch (Cin / 8) {
            case 1: launch_thin<2, 2, 2, 1, MASK>(a, st); break;
            case 2: launch_thin<2, 2, 2, 2, MASK>(a, st); break;
            case 3: launch_thin<2, 2, 2, 3, MASK>(a, st); break;
            case 5: launch_thin<2, 2, 2, 5, MASK>(a, st); break;
            case 6: launch_thin<2, 2, 2, 6, MASK>(a, st); break;
            default: launch_thin<2, 2, 2, 7, MASK>(a, st); break;
        }
        return;
    }
    // wave tiles: 64 px x 64 co, 128 px x 32 co, or 128 px x 16 co
    if (Cout >= 64) {
        const dim3 grid((unsigned)((P + 255) / 256) * (unsigned)((Cout + 63) / 64));
        hipLaunchKernelGGL((conv_fwd<4, 4, MASK>), grid, dim3(256), 0, st, x, xm, w, bias, y32, y16, N, H, W, Cin,
                           Cout, relu);
    } else if (Cout >= 32) {
        const dim3 grid((unsigned)((P + 511) / 512) * (unsigned)((Cout + 31) / 32));
        hipLaunchKernelGGL((conv_fwd<8, 2, MASK>), grid, dim3(256), 0, st, x, xm, w, bias, y32, y16, N, H, W, Cin,
                           Cout, relu);
    } else {
        const dim3 grid((unsigned)((P + 511) / 512) * (unsigned)((Cout + 15) / 16));
        hipLaunchKernelGGL((conv_fwd<8, 1, MASK>), grid, dim3(256), 0, st, x, xm, w, bias, y32, y16, N, H, W, Cin,
                           Cout, relu);
    }
}

// conv_wgrad addresses one image of each operand by 31-bit byte offsets and
// counts its work items in 32 bits.
bool wgrad_fits(int N, int H, int W, int Cin, int Cout) {
    return (int64_t)H * W * Cin * 2 < kMaxBytes && (int64_t)H * W * Cout * 2 < kMaxBytes &&
           (int64_t)N * H * ((W + 31) / 32) < ((int64_t)1 << 30) &&
           (int64_t)((Cout + 15) / 16) * ((Cin + 15) / 16) < ((int64_t)1 << 20);
}

template <bool MASK>
void launch_wgrad(const WgradArgs& a, const BwdWPlan& pl, hipStream_t st) {
    const dim3 grid(a.slices * a.ncb * a.nib), block(512);
    switch (pl.kind) {
        case 0: hipLaunchKernelGGL((conv_wgrad<2, 2, 2, 2, 2, MASK ? 3 : 4, 2, MASK>), grid, block, 0, st, a); break;
        case 1: hipLaunchKernelGGL((conv_wgrad<2, 2, 2, 1, 4, 3, MASK ? 1 : 2, MASK>), grid, block, 0, st, a); break;
        case 2: hipLaunchKernelGGL((conv_wgrad<2, 2, 1, 2, 4, MASK ? 4 : 3, MASK ? 1 : 2, MASK>), grid, block, 0, st, a); break;
        case 3: hipLaunchKernelGGL((conv_wgrad<2, 2, 1, 1, 8, MASK ? 3 : 4, 1, MASK>), grid, block, 0, st, a); break;
        case 4: hipLaunchKernelGGL((conv_wgrad<2, 1, 1, 1, 8, MASK ? 3 : 5, 1, MASK>), grid, block, 0, st, a); break;
        default: hipLaunchKernelGGL((conv_wgrad<1, 2, 1, 1, 8, MASK ? 4 : 5, 1, MASK>), grid, block, 0, st, a); break;
    }
}

int conv_fwd_checked(const uint16_t* x, const uint16_t* xm, const uint16_t* w, const float* bias, float* y32,
                     uint16_t* y16, int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout, int32_t relu,
                     void* stream) {
    int rc = check(N, H, W, Cin, Cout);
    if (rc) return rc;
    if (Cout % 8) return fail(FDS_E_ARG, "Cout must be a multiple of 8");
    if (!x || !w || (!y32 && !y16)) return fail(FDS_E_ARG, "NULL pointer");
    if (xm)
        launch_fwd<true>(x, xm, w, bias, y32, y16, N, H, W, Cin, Cout, relu, (hipStream_t)stream);
    else
        launch_fwd<false>(x, nullptr, w, bias, y32, y16, N, H, W, Cin, Cout, relu, (hipStream_t)stream);
    FDS_HIP(hipGetLastError());
    return FDS_OK;
}
// w16 (and, where wt[l] is given, the flipped copy) of n layers.
int cast_layers(int n, const float* const* w, uint16_t* const* w16, uint16_t* const* wt, const int32_t* cin,
                const int32_t* cout, hipStream_t stream) {
    CastFlipArgs a{};
    a.n = n;
    a.start[0] = 0;
    for (int l = 0; l < n; ++l) {
        if (!w[l] || !w16[l]) return fail(FDS_E_ARG, "NULL pointer");
        if (cin[l] < 1 || cout[l] < 1) return fail(FDS_E_ARG, "bad arguments");
        a.w[l] = w[l];
        a.w16[l] = w16[l];
        a.wt[l] = wt ? wt[l] : nullptr;
        a.cin[l] = cin[l];
        a.cout[l] = cout[l];
        a.start[l + 1] = a.start[l] + (int64_t)cout[l] * 9 * cin[l];
    }
    hipLaunchKernelGGL(cast_flip, dim3((unsigned)((a.start[n] + 255) / 256)), dim3(256), 0, stream, a);
    FDS_HIP(hipGetLastError());
    return FDS_OK;
}

// The U-Net's 15 layers in the order of their weights (e0a e0b e1a e1b e2a
// e2b e3a e3b d2a d2b d1a d1b d0a d0b head) for level widths c[0..3].
constexpr int kNetLayers = 15;
struct NetPlan {
    int32_t cin[kNetLayers], cout[kNetLayers];
    // elements (bf16) of the workspace: skips of the three upper levels, two
    // buffers that every other activation alternates between, the weights
    int64_t skip[3], buf, w[kNetLayers], total;
};

int net_plan(int N, int H, int W, const int32_t* c, NetPlan* p) {
    if (!c || N < 1 || H < 8 || W < 8 || (H % 8) || (W % 8)) return fail(FDS_E_ARG, "H and W must be multiples of 8");
    for (int l = 0; l < 4; ++l)
        if (c[l] < 8 || (c[l] % 8)) return fail(FDS_E_ARG, "level widths must be positive multiples of 8");
    if ((int64_t)N * H * W >= ((int64_t)1 << 40)) return fail(FDS_E_ARG, "too many pixels");
    const int32_t in[kNetLayers] = {8,           c[0], c[0],        c[1], c[1],        c[2], c[2], c[3],
                                    c[3] + c[2], c[2], c[2] + c[1], c[1], c[1] + c[0], c[0], c[0]};
    const int32_t out[kNetLayers] = {c[0], c[0], c[1], c[1], c[2], c[2], c[3], c[3],
                                     c[2], c[2], c[1], c[1], c[0], c[0], 8};
    const auto up = [](int64_t n) { return (n + 127) / 128 * 128; };   // 256-byte pieces
    const int64_t P = (int64_t)N * H * W;
    p->total = 0;
    p->buf = 0;
    for (int l = 0; l < 3; ++l) {
        p->skip[l] = p->total;
        p->total += up((P >> (2 * l)) * c[l]);
    }
    for (int l = 0; l < kNetLayers; ++l) {
        p->cin[l] = in[l];
        p->cout[l] = out[l];
        p->w[l] = p->total;
        p->total += up((int64_t)9 * in[l] * out[l]);
        const int lv = l < 8 ? l / 2 : (l < 14 ? 2 - (l - 8) / 2 : 0);
        p->buf = std::max(p->buf, up((P >> (2 * lv)) * std::max(in[l], out[l])));
    }
    return FDS_OK;
}

int pool_launch(const uint16_t* x, uint16_t* y, int N, int H, int W, int C, hipStream_t stream) {
    const int64_t n8 = (int64_t)N * (H / 2) * (W / 2) * (C / 8);
    hipLaunchKernelGGL(avg_pool2, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, stream, x, y, W, C / 8, n8);
    FDS_HIP(hipGetLastError());
    return FDS_OK;
}
}  // namespace

extern "C" {

const char* fds_last_error(void) { return g_err.c_str(); }


int fds_conv3x3_fwd(const uint16_t* x, const uint16_t* w, const float* bias, float* y32, uint16_t* y16, int32_t N,
                    int32_t H, int32_t W, int32_t Cin, int32_t Cout, int32_t relu, void* stream) {
    return conv_fwd_checked(x, nullptr, w, bias, y32, y16, N, H, W, Cin, Cout, relu, stream);
}

int fds_flip_weights(const uint16_t* w, uint16_t* wt, int32_t Cin, int32_t Cout, void* stream) {
    if (!w || !wt || Cin < 1 || Cout < 1) return fail(FDS_E_ARG, "bad arguments");
    const int64_t total = (int64_t)Cout * 9 * Cin;
    hipLaunchKernelGGL(flip_weights, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, w, wt,
                       Cin, Cout);
    FDS_HIP(hipGetLastError());
    return FDS_OK;
}

int fds_cast_flip(int32_t n, const float* const* w, uint16_t* const* w16, uint16_t* const* wt, const int32_t* cin,
                  const int32_t* cout, void* stream) {
    if (n < 1 || n > kCastLayers) return fail(FDS_E_ARG, "1 to 16 layers expected");
    if (!w || !w16 || !wt || !cin || !cout) return fail(FDS_E_ARG, "NULL pointer");
    for (int l = 0; l < n; ++l)
        if (!wt[l]) return fail(FDS_E_ARG, "NULL pointer");
    return cast_layers(n, w, w16, wt, cin, cout, (hipStream_t)stream);
}

int fds_conv3x3_bwd_data(const uint16_t* dy, const uint16_t* wt, const uint16_t* relu_y, float* dx32,
                         uint16_t* dx16, int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout, void* stream) {
    // the transposed convolution is a forward convolution of dy (Cout
    // channels) with the flipped weights (Cin outputs)
    return conv_fwd_checked(dy, relu_y, wt, nullptr, dx32, dx16, N, H, W, Cout, Cin, 0, stream);
}

// The floats of scratch of either kernel: unaligned operands take the general
// one whatever its time.
int64_t fds_bwd_weight_scratch(int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout) {
    int64_t S = bwd_w_general(N, H, W, Cin, Cout).S;
    if (wgrad_fits(N, H, W, Cin, Cout)) S = std::max<int64_t>(S, bwd_w_plan(N, H, W, Cin, Cout).slices);
    return S * Cout * (9 * (int64_t)Cin + 1);
}

int fds_conv3x3_bwd_weight(const uint16_t* x, const uint16_t* dy, const uint16_t* relu_y, float* dw, float* dbias,
                           float* scratch, int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout, void* stream) {
    int rc = check(N, H, W, Cin, Cout);
    if (rc) return rc;
    if (Cout % 8) return fail(FDS_E_ARG, "Cout must be a multiple of 8");
    if (!x || !dy || !dw || !scratch) return fail(FDS_E_ARG, "NULL pointer");
    hipStream_t st = (hipStream_t)stream;
    const int64_t nw = (int64_t)Cout * 9 * Cin, n = dbias ? nw + Cout : nw;
    int S;
    const BwdWGeneral pl = bwd_w_general(N, H, W, Cin, Cout);
    const bool fits = wgrad_fits(N, H, W, Cin, Cout) && aligned16(x) && aligned16(dy) && aligned16(relu_y);
    const BwdWPlan pw = fits ? bwd_w_plan(N, H, W, Cin, Cout) : BwdWPlan{};
    if (fits && pl.us >= 0.98f * pw.us) {
        const WgradArgs a{x, dy, relu_y, scratch, dbias != nullptr, N, H, W, Cin, Cout, pw.strips, pw.chunks, pw.rows,
                          pw.items, pw.slices, pw.ncb, pw.nib};
        if (relu_y) launch_wgrad<true>(a, pw, st);
        else launch_wgrad<false>(a, pw, st);
        S = pw.slices;
    } else {
        S = pl.S;
        const dim3 grid((unsigned)S * (unsigned)(((Cout + 63) / 64) * 9 * ((Cin + 63) / 64)));
        hipLaunchKernelGGL(conv_bwd_w, grid, dim3(256), 0, st, x, dy, relu_y, scratch, dbias != nullptr, N, H, W, Cin,
                           Cout, pl.chunk);
    }
    FDS_HIP(hipGetLastError());
    hipLaunchKernelGGL(reduce_slices, dim3((unsigned)((n + 31) / 32)), dim3(256), 0, st, scratch, nw + Cout, S, n, dw,
                       nw, dbias);
    FDS_HIP(hipGetLastError());
    return FDS_OK;
}

int fds_up_cat(const uint16_t* lo, const uint16_t* skip, uint16_t* out, int32_t N, int32_t H, int32_t W,
               int32_t C1, int32_t C2, void* stream) {
    if (!lo || !skip || !out) return fail(FDS_E_ARG, "NULL pointer");
    if (N < 1 || H < 2 || W < 2 || (H % 2) || (W % 2)) return fail(FDS_E_ARG, "N >= 1 and even H, W >= 2 expected");
    if (C1 < 8 || C2 < 8 || (C1 % 8) || (C2 % 8)) return fail(FDS_E_ARG, "C1, C2 must be positive multiples of 8");
    const int64_t n = (int64_t)N * H * W * ((C1 + C2) / 8);
    hipLaunchKernelGGL(up_cat, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, lo, skip, out, H,
                       W, C1 / 8, C2 / 8, n);
    FDS_HIP(hipGetLastError());
    return FDS_OK;
}

int fds_up_cat_bwd(const uint16_t* dout, uint16_t* dlo, uint16_t* dskip, int32_t N, int32_t H, int32_t W, int32_t C1,
                   int32_t C2, void* stream) {
    if (!dskip) return fail(FDS_E_ARG, "NULL pointer");
    return fds_up_cat_bwd_masked(dout, nullptr, dlo, dskip, N, H, W, C1, C2, stream);
}

int fds_up_cat_bwd_masked(const uint16_t* dout, const uint16_t* lo, uint16_t* dlo, uint16_t* dskip, int32_t N,
                          int32_t H, int32_t W, int32_t C1, int32_t C2, void* stream) {
    if (!dout || !dlo) return fail(FDS_E_ARG, "NULL pointer");
    if (N < 1 || H < 2 || W < 2 || (H % 2) || (W % 2)) return fail(FDS_E_ARG, "N >= 1 and even H, W >= 2 expected");
    if (C1 < 8 || C2 < 8 || (C1 % 8) || (C2 % 8)) return fail(FDS_E_ARG, "C1, C2 must be positive multiples of 8");
    const int64_t n_lo = (int64_t)N * (H / 2) * (W / 2) * (C1 / 8), n_skip = dskip ? (int64_t)N * H * W * (C2 / 8) : 0;
    hipLaunchKernelGGL(up_cat_bwd, dim3((unsigned)((n_lo + n_skip + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       dout, lo, dlo, dskip, H, W, C1 / 8, C2 / 8, n_lo, n_skip);
    FDS_HIP(hipGetLastError());
    return FDS_OK;
}

int fds_relu_mask(const uint16_t* dy, const uint16_t* y, uint16_t* out, int64_t n, void* stream) {
    if (!dy || !y || !out) return fail(FDS_E_ARG, "NULL pointer");
    if (n < 8 || (n % 8)) return fail(FDS_E_ARG, "n must be a positive multiple of 8");
    hipLaunchKernelGGL(relu_mask, dim3((unsigned)((n / 8 + 255) / 256)), dim3(256), 0, (hipStream_t)stream, dy, y,
                       out, n / 8);
    FDS_HIP(hipGetLastError());
    return FDS_OK;
}

int fds_pool_skip_bwd(const uint16_t* dp, const uint16_t* dskip, int32_t dskip_ld, const uint16_t* s, uint16_t* out,
                      int32_t N, int32_t H, int32_t W, int32_t C, void* stream) {
    if (!dp || !dskip || !s || !out) return fail(FDS_E_ARG, "NULL pointer");
    if (N < 1 || H < 2 || W < 2 || (H % 2) || (W % 2)) return fail(FDS_E_ARG, "N >= 1 and even H, W >= 2 expected");
    if (C < 8 || (C % 8)) return fail(FDS_E_ARG, "C must be a positive multiple of 8");
    if (dskip_ld < C || (dskip_ld % 8)) return fail(FDS_E_ARG, "dskip_ld must be a multiple of 8, at least C");
    const int64_t n8 = (int64_t)N * H * W * (C / 8);
    hipLaunchKernelGGL(pool_skip_bwd, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, (hipStream_t)stream, dp,
                       dskip, dskip_ld / 8, s, out, H, W, C / 8, n8);
    FDS_HIP(hipGetLastError());
    return FDS_OK;
}

int fds_avg_pool2(const uint16_t* x, uint16_t* y, int32_t N, int32_t H, int32_t W, int32_t C, void* stream) {
    if (!x || !y) return fail(FDS_E_ARG, "NULL pointer");
    if (N < 1 || H < 2 || W < 2 || (H % 2) || (W % 2)) return fail(FDS_E_ARG, "N >= 1 and even H, W >= 2 expected");
    if (C < 8 || (C % 8)) return fail(FDS_E_ARG, "C must be a positive multiple of 8");
    return pool_launch(x, y, N, H, W, C, (hipStream_t)stream);
}

int fds_net_inputs(const float* psi, const float* ux, const float* uy, const float* solid, int32_t solid_per_sample,
                   const float* lm, int32_t lm_n, const float* th, int32_t th_n, float scale, uint16_t* out, int32_t N,
                   int32_t H, int32_t W, void* stream) {
    if (!psi || !ux || !uy || !solid || !lm || !th || !out) return fail(FDS_E_ARG, "NULL pointer");
    if (N < 1 || H < 1 || W < 1) return fail(FDS_E_ARG, "bad shape");
    if ((lm_n != 1 && lm_n != N) || (th_n != 1 && th_n != N)) return fail(FDS_E_ARG, "one value or one per sample");
    const int64_t cells = (int64_t)H * W, n = N * cells;
    hipLaunchKernelGGL(net_inputs, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, psi, ux, uy,
                       solid, lm, th, scale, out, cells, solid_per_sample ? n : cells, lm_n, th_n, n);
    FDS_HIP(hipGetLastError());
    return FDS_OK;
}

int64_t fds_unet_scratch(int32_t N, int32_t H, int32_t W, const int32_t* c) {
    NetPlan p;
    if (net_plan(N, H, W, c, &p)) return -1;
    return 2 * (p.total + 2 * p.buf);
}

int fds_unet_fwd(const uint16_t* x, const float* const* w, const float* const* bias, float* y, void* scratch,
                 int32_t N, int32_t H, int32_t W, const int32_t* c, void* stream) {
    NetPlan p;
    int rc = net_plan(N, H, W, c, &p);
    if (rc) return rc;
    if (!x || !w || !bias || !y || !scratch) return fail(FDS_E_ARG, "NULL pointer");
    uint16_t* const base = (uint16_t*)scratch;
    uint16_t* const X = base + p.total;
    uint16_t* const Y = X + p.buf;
    uint16_t* w16[kNetLayers];
    for (int l = 0; l < kNetLayers; ++l) w16[l] = base + p.w[l];
    rc = cast_layers(kNetLayers, w, w16, nullptr, p.cin, p.cout, (hipStream_t)stream);
    if (rc) return rc;
    int layer = 0;
    const auto conv = [&](const uint16_t* in, uint16_t* out, int lv) {
        const int l = layer++;
        return conv_fwd_checked(in, nullptr, w16[l], bias[l], l == 14 ? y : nullptr, l == 14 ? nullptr : out, N,
                                H >> lv, W >> lv, p.cin[l], p.cout[l], l == 14 ? 0 : 1, stream);
    };
    const uint16_t* in = x;
    for (int lv = 0; lv < 3; ++lv) {
        uint16_t* const skip = base + p.skip[lv];
        if ((rc = conv(in, X, lv)) || (rc = conv(X, skip, lv)) ||
            (rc = pool_launch(skip, Y, N, H >> lv, W >> lv, c[lv], (hipStream_t)stream)))
            return rc;
        in = Y;
    }
    if ((rc = conv(Y, X, 3)) || (rc = conv(X, Y, 3))) return rc;
    uint16_t *a = Y, *b = X;   // the coarser level's output and a free buffer
    for (int lv = 2; lv >= 0; --lv) {
        if ((rc = fds_up_cat(a, base + p.skip[lv], b, N, H >> lv, W >> lv, c[lv + 1], c[lv], stream)) ||
            (rc = conv(b, a, lv)) || (rc = conv(a, b, lv)))
            return rc;
        std::swap(a, b);
    }
    return conv(a, nullptr, 0);
}

int64_t fds_net_loss_scratch(void) { return 2 * (int64_t)kLossBlocks; }

int fds_net_loss(const float* out, int32_t ld, const float* psi0, const float* psi1, const float* v0, const float* v1,
                 const float* wf, const float* w, float lambda, double* scratch, float* loss, float* res, int64_t n,
                 void* stream) {
    if (!out || !psi0 || !psi1 || !v0 || !v1 || !wf || !w || !scratch || !loss) return fail(FDS_E_ARG, "NULL pointer");
    if (n < 1 || ld < 3 || n > ((int64_t)1 << 38)) return fail(FDS_E_ARG, "bad shape");
    if (((uintptr_t)v0 | (uintptr_t)v1) & 7) return fail(FDS_E_ARG, "v0 and v1 must be 8-byte aligned");
    const LossArgs a{out, psi0, psi1, v0, v1, wf, res, n, ld};
    const int blocks = (int)std::min<int64_t>(kLossBlocks, (n + 255) / 256);
    hipLaunchKernelGGL(net_loss, dim3(blocks), dim3(256), 0, (hipStream_t)stream, a, scratch);
    FDS_HIP(hipGetLastError());
    hipLaunchKernelGGL(net_loss_sum, dim3(1), dim3(64), 0, (hipStream_t)stream, scratch, blocks, w, lambda, loss);
    FDS_HIP(hipGetLastError());
    return FDS_OK;
}

int fds_net_loss_bwd(const float* res, const float* wf, const float* w, float lambda, const float* g, float* dout,
                     int64_t n, void* stream) {
    if (!res || !wf || !w || !g || !dout) return fail(FDS_E_ARG, "NULL pointer");
    if (n < 1 || n > ((int64_t)1 << 38)) return fail(FDS_E_ARG, "bad shape");
    hipLaunchKernelGGL(net_loss_bwd, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, res, wf, w,
                       lambda, g, dout, n);
    FDS_HIP(hipGetLastError());
    return FDS_OK;
}

}  // extern "C"
