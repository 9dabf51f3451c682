// Router and dispatch kernels (engine/ops.cu:137-423): router logits, per-block sigmoid+bias scoring with the
// block expert pool and per-token top-K, routing weights, and the deterministic counting sort of (token, k)
// pairs into expert-major slots with the GEMM work items. All counts stay on the device.
#include <type_traits>

#include "decode_plan.h"

namespace llmoe {

namespace {

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

constexpr int MAXB = 32;    // tokens per routing block (one 32-bit token mask per expert)
constexpr int MAXE = 256;   // experts (one thread each)
constexpr int PLAN_NT = 1024;          // planner threads: 4 per expert
constexpr int MAXB_BLOCKS = 128;       // routing blocks whose masks the planner holds in registers (32 per thread)

// logits partial c: fma chain over k = c H/8 .. (c+1) H/8 - 1 ascending from 0 (the summation order is fixed so
// the CPU checker reproduces it).
// With q != nullptr the workgroups also write the A8 of the x slice (two 128-groups per token, the same operations
// as quant_a8_kernel, spread over the expert slices), so the layer input is quantised without a launch of its own.
__device__ __forceinline__ uint32_t okey(float v) {        // order-preserving unsigned image of a float
    const uint32_t u = __float_as_uint(v);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

constexpr int RKW = 256;                                          // K per chunk (H = 2048)

// Decode (T <= 32): workgroup tile 32 tokens x 8 experts of one K chunk, the chunk's x slice and its Wr slice
// (transposed, k contiguous per expert) staged in LDS; each of the 256 threads runs one chain. grid E/8 x 8 chunks.
// The step is latency-bound: 8 experts per workgroup put 256 workgroups on the chip (7.0 -> 5.8 us against 16 experts
// and two chains per thread).
constexpr int RD_EW = 8;                                          // experts per workgroup
constexpr int RD_STRIDE = RKW + 4;                                // LDS row stride of the x and Wr slices
constexpr int RD_LDS = (32 + RD_EW) * RD_STRIDE * 4;
__global__ void __launch_bounds__(256) router_decode_kernel(const float* __restrict__ x, const float* __restrict__ Wr,
                                                            int T, int H, int E, float* __restrict__ part,
                                                            int8_t* __restrict__ q, float* __restrict__ qs,
                                                            int* __restrict__ qsum) {
    constexpr int RS = RD_STRIDE, K4 = RKW / 4, XV = 32 * K4 / 256, WV = RKW * (RD_EW / 4) / 256;
    extern __shared__ __align__(16) float rl[];
    float* xs = rl;                       // [32][RS]
    float* ws = rl + 32 * RS;             // [8][RS]: Wr slice transposed, k contiguous per expert
    // XCD-aware: workgroups go round-robin over the 8 XCDs by linear workgroup id; slice (id % 8) X/8 + (id / 8) %
    // (X/8) puts the 4 slices of a 128-byte Wr row segment on one XCD (config 1: 0.0545 -> 0.0539 ms per step; chunk
    // per XCD: 0.0540 ms). E % 64 == 0, so X % 8 == 0.
    const int X = gridDim.x, id = blockIdx.x + X * blockIdx.z;
    const int sl = (id % 8) * (X / 8) + (id / 8) % (X / 8), c = id / X;
    const int e0 = sl * RD_EW, kb = c * RKW, tid = threadIdx.x;
    float4 xv[XV], wv[WV];
#pragma unroll
    for (int i = 0; i < XV; ++i) {                                // x: 32 x 256 floats as float4
        const int idx = tid + 256 * i, t = idx / K4, k4 = idx % K4;
        xv[i] = t < T ? *reinterpret_cast<const float4*>(x + size_t(t) * H + kb + 4 * k4)
                      : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
#pragma unroll
    for (int i = 0; i < WV; ++i) {                                // Wr: 256 x 8 floats as float4
        const int idx = tid + 256 * i, k = idx / (RD_EW / 4), e4 = idx % (RD_EW / 4);
        wv[i] = *reinterpret_cast<const float4*>(Wr + size_t(kb + k) * E + e0 + 4 * e4);
    }
#pragma unroll
    for (int i = 0; i < XV; ++i) {
        const int idx = tid + 256 * i, t = idx / K4, k4 = idx % K4;
        *reinterpret_cast<float4*>(xs + t * RS + 4 * k4) = xv[i];
    }
#pragma unroll
    for (int i = 0; i < WV; ++i) {
        const int idx = tid + 256 * i, k = idx / (RD_EW / 4), e4 = idx % (RD_EW / 4);
        ws[(4 * e4 + 0) * RS + k] = wv[i].x;
        ws[(4 * e4 + 1) * RS + k] = wv[i].y;
        ws[(4 * e4 + 2) * RS + k] = wv[i].z;
        ws[(4 * e4 + 3) * RS + k] = wv[i].w;
    }
    __syncthreads();
    // thread (token tid / 8, expert tid % 8)
    const int t = tid / RD_EW, e = tid % RD_EW;
    float acc = 0.0f;
#pragma unroll 4
    for (int k = 0; k < RKW; k += 4) {
        const float4 a = *reinterpret_cast<const float4*>(xs + t * RS + k);
        const float4 b = *reinterpret_cast<const float4*>(ws + e * RS + k);
        acc = __builtin_fmaf(a.x, b.x, acc);
        acc = __builtin_fmaf(a.y, b.y, acc);
        acc = __builtin_fmaf(a.z, b.z, acc);
        acc = __builtin_fmaf(a.w, b.w, acc);
    }
    if (q != nullptr) {
        // A8 of the chunk's x slice (2 groups per token): 32 lanes per token, 2 tokens per wave job; wave w of expert
        // slice b takes jobs w X + b, ...
        const int lane = tid & 63;
        for (int j = (tid >> 6) * X + sl; j < 16; j += 4 * X) {
            const int tt = 2 * j + lane / 32, l = lane % 32;
            const float4 a = *reinterpret_cast<const float4*>(xs + tt * RS + 8 * l);
            const float4 b = *reinterpret_cast<const float4*>(xs + tt * RS + 8 * l + 4);
            const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
            const size_t gi = size_t(tt) * (H / GROUP) + kb / GROUP + (l >> 4);   // (rows beyond T are not written)
            quant_a8_8(v, lane, q + size_t(tt) * H + kb + 8 * l, qs + gi, qsum + gi, tt < T);
        }
    }
    if (t < T) part[(size_t(c) * T + t) * E + e0 + e] = acc;
}

// Above 32 tokens: the chains on the matrix cores. v_mfma_f32_16x16x4_f32 accumulates its four k in ascending order
// with one rounding each -- bit for bit the fma chain (checked on the device against the CPU chain, subnormals
// included; the GPU tests compare the partials' sums with the checker's) -- at twice the vector fma rate: 1024 fma
// in 32 cycles per SIMD. Tile: 32 M tokens x 32 M experts of one K chunk, 4 waves of M x M 16x16 MFMA tiles. The K
// chunk runs in stages of 64 k: the x slice goes through LDS (two buffers) as [token][k % 4][k / 4], so that a lane
// reads the k of four MFMAs (its k are congruent mod 4) as 16 bytes (row stride 68: conflict-free); Wr operands come
// straight from global memory (64 contiguous bytes per k). A stage's loads are in flight during the stage before.
// Experts are the MFMA rows, so a lane ends with four consecutive experts of one token.
// What bounds it: the f32 MFMA issue (28 us of 4096 tokens' 52 at 2.4 GHz; vector work does not overlap f32 MFMAs, so
// the A8 and the addressing add to it). Against vector fma chains on 64 x 64 tiles in LDS, by kernel traces on one box:
// 13.8 -> 9.4 us at 512 tokens, 83 -> 52 us at 4096.
typedef float v4f __attribute__((ext_vector_type(4)));
constexpr int RM_KS = 64, RM_STRIDE = RM_KS + 4;
template <int M>
constexpr int rm_lds() { return 2 * 32 * M * RM_STRIDE * 4; }
template <int M>
__global__ void __launch_bounds__(256, 4) router_mfma_kernel(const float* __restrict__ x, const float* __restrict__ Wr,
                                                             int T, int H, int E, float* __restrict__ part,
                                                             int8_t* __restrict__ q, float* __restrict__ qs,
                                                             int* __restrict__ qsum) {
    constexpr int TT = 32 * M, RS = RM_STRIDE, K4 = RM_KS / 4, XV = TT * K4 / 256, NJ = RM_KS / 4, QS = RM_KS / 4;
    constexpr int NH = RKW / RM_KS;
    static_assert(2 * RM_KS == GROUP && NH % 2 == 0, "a 128-group is two stages");
    extern __shared__ __align__(16) float xs[];                   // [2][TT][RS]: [k % 4][k / 4] per token
    // XCD-aware: workgroups go round-robin over the 8 XCDs by linear id, so K chunk c = id % 8 keeps the chunk's Wr
    // rows and x columns in one XCD's L2
    static_assert(ROUTER_KC == 8, "one K chunk per XCD");
    const int X = gridDim.x, id = blockIdx.x + X * (blockIdx.y + gridDim.y * blockIdx.z);
    const int c = id % ROUTER_KC, sl = (id / ROUTER_KC) % X, ty = id / ROUTER_KC / X;
    const int e0 = sl * TT, t0 = ty * TT;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 15, q4 = lane >> 4;
    const int te = 16 * M * (w & 1), tt0 = 16 * M * (w >> 1);     // the wave's experts and tokens inside the tile
    // this thread's x elements of a stage (rows beyond T read the last row; their outputs are not stored)
    const float* xp[XV];
    float* xl[XV];
#pragma unroll
    for (int i = 0; i < XV; ++i) {
        const int idx = tid + 256 * i, t = idx / K4, k4 = idx % K4;
        xp[i] = x + size_t(min(t0 + t, T - 1)) * H + c * RKW + 4 * k4;
        xl[i] = xs + t * RS + k4;
    }
    const float* wp = Wr + size_t(c * RKW + q4) * E + e0 + te + r;
    float4 xv[XV];
    float wv[2][M][NJ];
    auto load = [&](auto hc) {
        constexpr int h = decltype(hc)::value;
#pragma unroll
        for (int i = 0; i < XV; ++i) xv[i] = *reinterpret_cast<const float4*>(xp[i] + h * RM_KS);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int i = 0; i < M; ++i) wv[h & 1][i][j] = wp[size_t(h * RM_KS + 4 * j) * E + 16 * i];
    };
    v4f acc[M][M];                                                // [expert tile][token tile]
#pragma unroll
    for (int i = 0; i < M; ++i)
#pragma unroll
        for (int j = 0; j < M; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    load(std::integral_constant<int, 0>{});
    static_for<0, NH>([&](auto hc) {
        constexpr int h = decltype(hc)::value;
        float* buf = xs + (h & 1) * TT * RS;
#pragma unroll
        for (int i = 0; i < XV; ++i) {
            float* p = xl[i] + (h & 1) * TT * RS;
            p[0] = xv[i].x;
            p[QS] = xv[i].y;
            p[2 * QS] = xv[i].z;
            p[3 * QS] = xv[i].w;
        }
        __syncthreads();   // (also: the readers of the other buffer, which the next stage overwrites, are done)
        if constexpr (h + 1 < NH) load(std::integral_constant<int, h + 1>{});
#pragma unroll
        for (int j = 0; j < NJ; j += 4) {
            float4 xa[M];
#pragma unroll
            for (int i = 0; i < M; ++i)
                xa[i] = *reinterpret_cast<const float4*>(buf + (tt0 + 16 * i + r) * RS + q4 * QS + j);
#pragma unroll
            for (int jj = 0; jj < 4; ++jj)
#pragma unroll
                for (int i = 0; i < M; ++i)
#pragma unroll
                    for (int n = 0; n < M; ++n) {
                        const float xk = jj == 0 ? xa[n].x : jj == 1 ? xa[n].y : jj == 2 ? xa[n].z : xa[n].w;
                        acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[h & 1][i][j + jj], xk, acc[i][n], 0, 0, 0);
                    }
        }
        if constexpr (h & 1) {
            if (q != nullptr) {
                // A8 of the 128-group now in the two buffers: 16 lanes per token, 4 tokens per wave job; wave w of expert
                // slice b takes jobs w X + b, ...
                const int kb = c * RKW + (h - 1) * RM_KS;
                for (int j = w * X + sl; j < TT / 4; j += 4 * X) {
                    const int tl = 4 * j + q4, t = t0 + tl;
                    const float* v0 = xs + (r >> 3) * TT * RS + tl * RS + 2 * (r & 7);
                    float v[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) v[i] = v0[(i & 3) * QS + (i >> 2)];
                    const size_t gi = size_t(t) * (H / GROUP) + kb / GROUP;   // (rows beyond T are not written)
                    quant_a8_8(v, lane, q + size_t(t) * H + kb + 8 * r, qs + gi, qsum + gi, t < T);
                }
                if constexpr (h + 1 < NH) __syncthreads();   // both buffers have been read
            }
        }
    });
#pragma unroll
    for (int n = 0; n < M; ++n) {
        const int t = t0 + tt0 + 16 * n + r;
        if (t < T)
#pragma unroll
            for (int i = 0; i < M; ++i)
                *reinterpret_cast<v4f*>(part + (size_t(c) * T + t) * E + e0 + te + 16 * i + 4 * q4) = acc[i][n];
    }
}

__device__ __forceinline__ int width_class(int bits) { return bits == 8 ? 0 : bits == 4 ? 1 : bits == 3 ? 2 : 3; }
// decode units, longest first: a streamed unit's time is set by its vector work, and the 2-bit units (4 strips per
// wave) have the most tiles (measured at 32 tokens against the byte order 8, 4, 3, 2 with the shared expert first:
// 0.0623 -> 0.0615 ms per step)

// the units of expert e: items of <= ntok of its c slots starting at slot st, each split into row blocks
__device__ void emit_units(int e, int c, int st, int ntok, int bits, int base_gu, int base_dn, Item* units_gu,
                           Item* units_dn) {
    const int nit = (c + ntok - 1) / ntok, rg = gemm_row_blocks(false, bits), rd = gemm_row_blocks(true, bits);
    for (int j = 0; j < nit; ++j) {
        const int s0 = st + j * ntok, n = min(ntok, c - j * ntok);
        for (int r = 0; r < rg; ++r) units_gu[base_gu + j * rg + r] = Item{e, s0, n, r};
        for (int r = 0; r < rd; ++r) units_dn[base_dn + j * rd + r] = Item{e, s0, n, r};
    }
}

// the shared expert's units (all T tokens, slots T K + t), the first of both lists; strided over the block
__device__ void emit_shared_units(int E, int T, int K, int ntok, int bits, Item* units_gu, Item* units_dn) {
    const int ns = (T + ntok - 1) / ntok, rg = gemm_row_blocks(false, bits), rd = gemm_row_blocks(true, bits);
    for (int u = threadIdx.x; u < ns * rg; u += blockDim.x) {
        const int j = u / rg;
        units_gu[u] = Item{E, T * K + j * ntok, min(ntok, T - j * ntok), u % rg};
    }
    for (int u = threadIdx.x; u < ns * rd; u += blockDim.x) {
        const int j = u / rd;
        units_dn[u] = Item{E, T * K + j * ntok, min(ntok, T - j * ntok), u % rd};
    }
}


// Cost of one row-block task of a chunk with nt 16-slot tiles, in 50 ns units: a per-row-block part (code
// unpacking, the weight stream) plus a per-tile part (MFMAs and the fp32 epilogue), as measured on MI355X for
// each code width (8-bit row blocks have half the rows)
__device__ __forceinline__ int rb_cost(int bits, int nt, bool down) {
    if (down) return bits == 8 ? 73 + 17 * nt : bits == 3 ? 37 + 18 * nt : bits == 4 ? 34 + 19 * nt : 30 + 18 * nt;
    return bits == 8 ? 64 + 35 * nt : bits == 3 ? 134 + 66 * nt : bits == 4 ? 78 + 72 * nt : 70 + 70 * nt;
}
// The activation staging a workgroup does for every chunk it touches (measured: ≈ 4.7 µs for gate_up, 64 slots x
// 2 KiB; ≈ 2.7 µs for down), costed at half weight at each chunk's start, so that workgroups that touch more
// chunks take fewer row blocks. (At full weight config 3 gained 2.6 % but 512-token layers, with under two row
// blocks per workgroup, lost 1.2 %; at half weight config 3 gains 1.8 %, config 4 1 %, and nothing loses.)
constexpr int STAGE_COST_GU = 48, STAGE_COST_DN = 28;
// the chunk's row-block task cost and row-block count of both GEMMs, packed (cost << 8 | count) for the planner
__device__ __forceinline__ void chunk_tasks(int bits, int ntok, uint32_t* gu, uint32_t* dn) {
    const int nt = (ntok + 15) >> 4;
    *gu = uint32_t(rb_cost(bits, nt, false) << 8) | uint32_t(tiled_row_blocks(false, bits));
    *dn = uint32_t(rb_cost(bits, nt, true) << 8) | uint32_t(tiled_row_blocks(true, bits));
}

// floor(x / d) for 0 <= x < 2^53, d > 0: a double quotient corrected by integer products
__device__ __forceinline__ long long floor_div(long long x, long long d) {
    long long q = (long long)(double(x) / double(d));
    while (q > 0 && q * d > x) --q;
    while ((q + 1) * d <= x) ++q;
    return q;
}



// ---- decode routing (one routing block, T <= block <= 32) ------------------------------------------------------
// score_kernel (with the pool), select_token_kernel (one token per workgroup), then dispatch_kernel (one
// workgroup: slots and work units for all tokens; or the gate_up GEMM of a layer forward, which plans for itself).
// DecodeState is zero when a call starts, and whichever kernel consumes it leaves it zero again.

// With qx.x set, the workgroup of token t first writes the A8 of x's row t (H = 2048: wave w takes columns
// 512 w .. 512 w + 511), so routing from given logits needs no launch of its own for it.
__device__ __forceinline__ void row_a8(const QuantX& qx, int t) {
    if (qx.x == nullptr) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const size_t base = size_t(t) * 2048 + 512 * w, gi = size_t(t) * 16 + 4 * w;
    quant_a8_512(qx.x + base, lane, qx.q + base, qx.s + gi, qx.sum + gi);
}

// grid T, 256 threads (thread = expert): logit = partials summed in chunk order; sig[t, e] = sigmoid(logit);
// with the pool, blockmax[e] = max over tokens of the ordered key of sigmoid + bias
template <bool QA8>
__global__ void __launch_bounds__(256) score_kernel(const float* __restrict__ part, int nchunks,
                                                    const float* __restrict__ bias, int T, int E, int block,
                                                    int pool_on, float* __restrict__ sig,
                                                    uint32_t* __restrict__ blockmax, QuantX qx) {
    const int t = blockIdx.x, e = threadIdx.x;
    if constexpr (QA8) row_a8(qx, t);
    if (e >= E) return;
    float p[ROUTER_KC];
#pragma unroll
    for (int c = 0; c < ROUTER_KC; ++c) p[c] = c < nchunks ? part[(size_t(c) * T + t) * E + e] : 0.0f;
    float l = p[0];
#pragma unroll
    for (int c = 1; c < ROUTER_KC; ++c)
        if (c < nchunks) l = l + p[c];
    const float sg = sigmoid_f32(l);
    sig[size_t(t) * E + e] = sg;
    if (pool_on) atomicMax(&blockmax[size_t(t / block) * E + e], okey(sg + bias[e]));
}


// Slots and work units of the decode step (engine/ops.cu:333-370), one workgroup of 256 threads (thread e writes
// expert e's units); the masks and pool maxima are left zero for the next call.
__global__ void __launch_bounds__(256) dispatch_kernel(int T, int E, int K, const int* __restrict__ topk,
                                                       const float* __restrict__ topw, DecodeState ds, DispatchOut d) {
    __shared__ DecodePlan P;
    decode_plan_scan(E, ds.tmask, d.bits, P);
    const int sbits = d.has_shared ? d.bits[E] : 8;
    const int fg = plan_fine(P.tot, false, d.max_gu, T, d.has_shared, sbits);
    const int fd = plan_fine(P.tot, true, d.max_dn, T, d.has_shared, sbits);
    const int e = threadIdx.x;
    if (e < E) {
        ds.tmask[e] = 0u;
        ds.blockmax[e] = 0u;
        decode_plan_write_expert(P, e, 0, 1, fg, fd, d);
    }
    decode_plan_write_rest(P, e, 256, T, E, K, topk, topw, fg, fd, d);
}


// The `want` largest of N keys held V per lane (key v of lane l has index 64 v + l; equal keys: the lower index first),
// by descent over the bits of the threshold: *thr is the largest value t with at least `want` keys >= t -- the want-th
// largest key, or less when the descent stops early at a t with exactly `want` keys >= t. One wave, no LDS, no barrier:
// per bit V compares, each mask counted by the scalar unit. want <= N.
template <int V>
__device__ __forceinline__ uint32_t select_threshold(const uint32_t (&key)[V], int want) {
    uint32_t thr = 0u;
#pragma unroll 1
    for (int bit = 31; bit >= 0; --bit) {
        const uint32_t cand = thr | (1u << bit);
        int n = 0;
#pragma unroll
        for (int v = 0; v < V; ++v) n += __builtin_popcountll(__ballot(key[v] >= cand));
        if (n >= want) {
            thr = cand;
            if (n == want) break;
        }
    }
    return thr;
}
// whether each of the lane's keys is among the `want` largest
template <int V>
__device__ __forceinline__ void select_top(const uint32_t (&key)[V], int want, bool (&in)[V]) {
    const uint32_t thr = select_threshold(key, want);
    int above = 0;
    uint64_t eq[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        above += __builtin_popcountll(__ballot(key[v] > thr));
        eq[v] = __ballot(key[v] == thr);
    }
    int left = want - above;   // keys equal to the threshold that still belong, in index order
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int before = __builtin_amdgcn_mbcnt_hi(uint32_t(eq[v] >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(eq[v]), 0));
        in[v] = key[v] > thr || (key[v] == thr && before < left);
        left -= __builtin_popcountll(eq[v]);
    }
}

// Selection, one token per workgroup (engine/ops.cu:256-327). Thread e scores expert e: without the pool the logit is
// the router partials' sum in chunk order, then the sigmoid; with it score_kernel's sigmoid. Meanwhile the last wave
// finds the block's pool, the C experts with the largest blockmax keys. Then wave 0, four experts per lane, selects the
// token's top-K of the pool, ranks them among each other and writes them with the routing weights
// (engine/ops.cu:298-321) and the token masks. All comparisons are (value desc, index asc). Both selections are bit
// descents over ballots (select_threshold).
// Against bitonic sorts of 64 keys per wave and a merge (for the pool, four sorted lists searched per expert), by kernel
// traces on one box: 11.5 -> 9.8 us at 2048 tokens, 15.2 -> 11.4 at 4096 (2 % of such a layer). At 32 tokens 4.7 us and
// with the pool 5.8 us either way, where the launch and the loads are most of it: there it is the one form for both.
template <bool POOL, bool QA8>
__global__ void __launch_bounds__(256) select_token_kernel(const float* __restrict__ part, int nchunks,
                                                           const float* __restrict__ sig,
                                                           const float* __restrict__ bias, int T, int E, int K,
                                                           int C, int block, float rscale, int* __restrict__ topk,
                                                           float* __restrict__ topw, DecodeState ds, QuantX qx) {
    __shared__ float sig_s[MAXE];
    __shared__ uint32_t key_s[MAXE];
    __shared__ uint32_t pool_s[POOL ? MAXE : 1];
    __shared__ int cand_e[8];
    const int t = blockIdx.x, e = threadIdx.x, lane = e & 63, w = e >> 6;
    if constexpr (QA8) row_a8(qx, t);
    float sv = 0.0f, bv = 0.0f;
    uint32_t pk[4];
    if constexpr (POOL) {
        if (w == 3)
#pragma unroll
            for (int v = 0; v < 4; ++v) pk[v] = 64 * v + lane < E ? ds.blockmax[size_t(t / block) * E + 64 * v + lane] : 0u;
    }
    if (e < E) {
        bv = bias[e];
        if constexpr (POOL) {
            sv = sig[size_t(t) * E + e];
        } else {
            float p[ROUTER_KC];
#pragma unroll
            for (int c = 0; c < ROUTER_KC; ++c) p[c] = c < nchunks ? part[(size_t(c) * T + t) * E + e] : 0.0f;
            float l = p[0];
#pragma unroll
            for (int c = 1; c < ROUTER_KC; ++c)
                if (c < nchunks) l = l + p[c];
            sv = sigmoid_f32(l);
        }
    }
    sig_s[e] = sv;
    // (a key of 0 is no candidate: okey of a number is above it; experts beyond E, and the pool's exclusions below)
    key_s[e] = e < E ? okey(sv + bv) : 0u;
    if constexpr (POOL) {
        if (w == 3) {
            bool in[4];
            select_top<4>(pk, C, in);
#pragma unroll
            for (int v = 0; v < 4; ++v) pool_s[64 * v + lane] = in[v] ? 0xFFFFFFFFu : 0u;
        }
    }
    __syncthreads();
    if (w != 0) return;
    uint32_t key[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        key[v] = key_s[64 * v + lane];
        if constexpr (POOL) key[v] &= pool_s[64 * v + lane];
    }
    bool in[4];
    select_top<4>(key, K, in);
    // the K chosen, in index order, to lanes 0 .. K - 1
    int at = 0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const uint64_t m = __ballot(in[v]);
        const int pos = at + __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0));
        if (in[v]) cand_e[pos] = 64 * v + lane;
        at += __builtin_popcountll(m);
    }
    __builtin_amdgcn_wave_barrier();
    const int ex = lane < K ? cand_e[lane] : 0;
    const float sk = sig_s[ex];
    const uint32_t kk = lane < K ? key_s[ex] : 0u;
    // rank among the chosen (they are in index order, so equal keys rank by lane)
    int rank = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const uint32_t o = __builtin_amdgcn_readlane(kk, k);
        rank += k < K && (o > kk || (o == kk && k < lane)) ? 1 : 0;
    }
    // the sum of the scores in rank order: lane k's score to lane rank(k)
    float wsum = 0.0f;
    const int src = lane < K ? rank : lane;
    const float ranked = __int_as_float(__builtin_amdgcn_ds_permute(4 * src, __float_as_int(sk)));
#pragma unroll
    for (int k = 0; k < 8; ++k)
        if (k < K) wsum = wsum + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ranked), k));
    if (lane < K) {
        topk[size_t(t) * K + rank] = ex;
        topw[size_t(t) * K + rank] = sk / (wsum + 1e-20f) * rscale;
        atomicOr(&ds.tmask[size_t(t / block) * E + ex], 1u << (t % block));
    }
}


// Token masks of externally given routing, and the layer's copy of it (the caller's arrays are free once the call's
// work is done). Bound by launch latency: two copy commands of the runtime took 4.0 us each beside this kernel's 3.9 us;
// with the copies in the kernel it takes 4.6 us (77 tokens). The copies may be the given arrays themselves. grid nb, 256
// threads.
__global__ void __launch_bounds__(256) masks_kernel(const int* topk, const float* topw, int T, int E, int K, int block,
                                                    int* topk_out, float* topw_out, uint32_t* __restrict__ mask) {
    __shared__ uint32_t tmask[MAXE];
    const int b = blockIdx.x, t0 = b * block, tb = min(block, T - t0);
    if (threadIdx.x < E) tmask[threadIdx.x] = 0u;
    __syncthreads();
    for (int p = threadIdx.x; p < tb * K; p += blockDim.x) {
        const size_t i = size_t(t0) * K + p;
        const int e = topk[i];
        const float w = topw[i];
        atomicOr(&tmask[e], 1u << (p / K));
        topk_out[i] = e;
        topw_out[i] = w;
    }
    __syncthreads();
    if (threadIdx.x < E) mask[size_t(b) * E + threadIdx.x] = tmask[threadIdx.x];
}

// Slot ranges and work units (engine/ops.cu:333-370, :384-410): slots expert-major (expert ascending), inside
// an expert block-major then token-ascending. An expert with more than TILED_MIN slots (when `tiled`) gets tiled
// units (chunks of <= TILED_NTOK slots x tiled row blocks), otherwise streamed units (items of <= ntok slots x
// streamed row blocks). Both lists are ordered heaviest first (shared expert, then 8 / 4 / 3 / 2-bit experts).
// One workgroup of four threads per expert: the block masks are split in four contiguous ranges.
__global__ void __launch_bounds__(PLAN_NT) plan_kernel(const uint32_t* __restrict__ mask, int T, int E, int K,
                                                       int block, int has_shared, int ntok, int tiled,
                                                       const int8_t* __restrict__ bits, int* __restrict__ count,
                                                       int* __restrict__ start, int* __restrict__ bpre,
                                                       Item* __restrict__ units_gu, Item* __restrict__ units_dn,
                                                       Item* __restrict__ tunits_gu, Item* __restrict__ tunits_dn,
                                                       int* __restrict__ n_units, int g_gu, int g_dn,
                                                       int* __restrict__ tstart, int max_chunks) {
    constexpr int NP = PLAN_NT / MAXE;         // threads per expert: each takes a contiguous range of blocks
    constexpr int NBR = MAXB_BLOCKS / NP;      // block masks of a range held in registers
    constexpr int NWAVE = PLAN_NT / 64;
    // chunk tables (max_chunks entries): row-block tasks of both GEMMs, then their positions [n_chunks + 1]
    extern __shared__ uint32_t plan_lds[];
    uint32_t* task_gu = plan_lds;
    uint32_t* task_dn = task_gu + max_chunks;
    int* pre_gu = reinterpret_cast<int*>(task_dn + max_chunks);
    int* pre_dn = pre_gu + max_chunks + 1;
    int* owner = pre_dn + max_chunks + 1;      // expert of each chunk
    __shared__ int wt_i[NWAVE], wt_c[NWAVE];
    __shared__ uint64_t wt[4][4];
    __shared__ uint64_t tot[4];
    __shared__ int first_l[MAXE + 1], cnt_l[MAXE + 1], st_l[MAXE + 1], bits_l[MAXE + 1];
    __shared__ int cpart_s[NP][MAXE];          // tokens of expert e in part p's block range
    const int tid = threadIdx.x, e = tid % MAXE, part = tid / MAXE, nb = (T + block - 1) / block;
    const int lane = tid & 63, wv = tid >> 6, w = wv & 3;   // (w: the wave within the expert-scan group)
    const bool g0 = part == 0;                 // the expert's lead thread (scans, units)
    // token masks of the part's block range [b_lo, b_hi): unconditional loads at clamped indices, so that the
    // batch is issued back to back
    const int ec = min(e, E - 1), nbp = (nb + NP - 1) / NP, b_lo = min(nb, part * nbp), b_hi = min(nb, b_lo + nbp);
    // code widths read up front, with the masks: a load after them would expose its own latency
    const int bw_ld = bits[ec], sbits_ld = has_shared ? bits[E] : 8;
    uint32_t mv[NBR];
#pragma unroll
    for (int j = 0; j < NBR; ++j) mv[j] = mask[size_t(min(b_lo + j, nb - 1)) * E + ec];
    int cp = 0;
#pragma unroll
    for (int j = 0; j < NBR; ++j) cp += b_lo + j < b_hi ? __popc(mv[j]) : 0;
    for (int b0 = b_lo + NBR; b0 < b_hi; b0 += 16) {   // ranges longer than the registers hold
        uint32_t m2[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) m2[j] = mask[size_t(min(b0 + j, nb - 1)) * E + ec];
#pragma unroll
        for (int j = 0; j < 16; ++j) cp += b0 + j < b_hi ? __popc(m2[j]) : 0;
    }
    if (e >= E) cp = 0;
    cpart_s[part][e] = cp;
    __syncthreads();
    int c = 0, cbefore = 0;   // the expert's slots; those in the blocks before the part's range
#pragma unroll
    for (int pp = 0; pp < NP; ++pp) {
        const int v = cpart_s[pp][e];
        cbefore += pp < part ? v : 0;
        c += v;
    }
    const bool big = e < E && tiled && c > 0;
    const bool sbig = has_shared && tiled;
    const int nsch = sbig ? tiled_chunks(T) : 0;
    const int bw = e < E ? bw_ld : 2, cls = width_class(bw);
    const int nit = e < E && !big ? (c + ntok - 1) / ntok : 0, nch = big ? tiled_chunks(c) : 0;
    // one pass of inclusive scans over the experts (lead threads): slots, tiled chunks, and per width class
    // (16-bit fields) the streamed units of both lists and the tiled chunks
    int incl = c;
    uint64_t s0 = uint64_t(nit * gemm_row_blocks(false, bw)) << (16 * cls);
    uint64_t s1 = uint64_t(nit * gemm_row_blocks(true, bw)) << (16 * cls);
    uint64_t t0 = uint64_t(nch) << (16 * cls);
    const uint64_t own0 = s0, own1 = s1, ownt = t0;
    incl = wave_incl_scan(incl);
    s0 = wave_incl_scan(s0);
    s1 = wave_incl_scan(s1);
    t0 = wave_incl_scan(t0);
    if (g0 && lane == 63) {
        wt_i[w] = incl;
        wt[w][0] = s0;
        wt[w][1] = s1;
        wt[w][2] = t0;
    }
    __syncthreads();
    for (int i = 0; i < w; ++i) {
        incl += wt_i[i];
        s0 += wt[i][0];
        s1 += wt[i][1];
        t0 += wt[i][2];
    }
    if (tid == MAXE - 1) {
        tot[0] = s0;
        tot[1] = s1;
        tot[2] = t0;
    }
    __syncthreads();
    const int sbits = sbits_ld;
    const int ns = has_shared && !sbig ? (T + ntok - 1) / ntok : 0;
    // offsets: the shared expert's units first, then width classes 0 .. 3 (8, 4, 3, 2 bits), expert ascending
    int bg = ns * gemm_row_blocks(false, sbits), bd = ns * gemm_row_blocks(true, sbits), bt = nsch;
    int og = 0, od = 0, ot = 0;
    for (int k = 0; k < 4; ++k) {
        if (k == cls) {
            og = bg + int(((s0 - own0) >> (16 * k)) & 0xFFFFu);
            od = bd + int(((s1 - own1) >> (16 * k)) & 0xFFFFu);
            ot = bt + int(((t0 - ownt) >> (16 * k)) & 0xFFFFu);
        }
        bg += int((tot[0] >> (16 * k)) & 0xFFFFu);
        bd += int((tot[1] >> (16 * k)) & 0xFFFFu);
        bt += int((tot[2] >> (16 * k)) & 0xFFFFu);
    }
    // (the scans above ran in every part on identical values; only part 0's results are used below)
    const int st = incl - c;
    if (e < E) {
        // slot base of each (block, expert) of the part's range
        int run = st + cbefore;
#pragma unroll
        for (int j = 0; j < NBR; ++j)
            if (b_lo + j < b_hi) {
                bpre[size_t(b_lo + j) * E + e] = run;
                run += __popc(mv[j]);
            }
        for (int b0 = b_lo + NBR; b0 < b_hi; b0 += 16) {
            uint32_t m2[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) m2[j] = mask[size_t(min(b0 + j, nb - 1)) * E + e];
#pragma unroll
            for (int j = 0; j < 16; ++j)
                if (b0 + j < b_hi) {
                    bpre[size_t(b0 + j) * E + e] = run;
                    run += __popc(m2[j]);
                }
        }
    }
    if (g0 && e < E) {
        count[e] = c;
        start[e] = st;
        if (big) {   // the chunks are written below, one thread per chunk
            first_l[e] = ot;
            cnt_l[e] = c;
            st_l[e] = st;
            bits_l[e] = bw;
            for (int j = 0; j < nch; ++j) owner[ot + j] = e;
        } else {
            emit_units(e, c, st, ntok, bw, og, od, units_gu, units_dn);
        }
    }
    if (ns) emit_shared_units(E, T, K, ntok, sbits, units_gu, units_dn);
    if (sbig) {
        if (tid == 0) {
            first_l[E] = 0;
            cnt_l[E] = T;
            st_l[E] = T * K;
            bits_l[E] = sbits;
        }
        for (int j = tid; j < nsch; j += blockDim.x) owner[j] = E;
    }
    if (tid == 0) {
        n_units[0] = bg;
        n_units[1] = bd;
        n_units[2] = bt;
        n_units[3] = bt;
        n_units[4] = bg;   // (streamed units: not split)
        n_units[5] = bd;
    }
    if (!tiled) return;
    // the tiled chunks: tiled_per(c) slots of an expert's c each, the last one shorter (Item.rb unused)
    __syncthreads();
    const int n = bt;
    for (int j = tid; j < n; j += blockDim.x) {
        const int x = owner[j], cx = cnt_l[x], pc = tiled_per(cx), jj = j - first_l[x];
        const Item it{x, st_l[x] + jj * pc, min(pc, cx - jj * pc), 0};
        tunits_gu[j] = it;
        tunits_dn[j] = it;
        chunk_tasks(bits_l[x], it.ntok, &task_gu[j], &task_dn[j]);
    }
    // chunk positions of both GEMMs: scans of the chunk costs (each thread a run of consecutive chunks)
    __syncthreads();
    const int per = (n + blockDim.x - 1) / blockDim.x, j0 = min(n, tid * per), j1 = min(n, j0 + per);
    auto cost = [](uint32_t t, int stage) { return stage + int(t >> 8) * int(t & 255u); };
    int run0 = 0, run1 = 0;
    for (int j = j0; j < j1; ++j) {
        run0 += cost(task_gu[j], STAGE_COST_GU);
        run1 += cost(task_dn[j], STAGE_COST_DN);
    }
    int inc0 = run0, inc1 = run1;
    inc0 = wave_incl_scan(inc0);
    inc1 = wave_incl_scan(inc1);
    if (lane == 63) {
        wt_i[wv] = inc0;
        wt_c[wv] = inc1;
    }
    __syncthreads();
    for (int i = 0; i < wv; ++i) {
        inc0 += wt_i[i];
        inc1 += wt_c[i];
    }
    run0 = inc0 - run0;
    run1 = inc1 - run1;
    for (int j = j0; j < j1; ++j) {
        pre_gu[j] = run0;
        pre_dn[j] = run1;
        run0 += cost(task_gu[j], STAGE_COST_GU);
        run1 += cost(task_dn[j], STAGE_COST_DN);
    }
    if (tid == int(blockDim.x) - 1) {
        pre_gu[n] = inc0;
        pre_dn[n] = inc1;
    }
    __syncthreads();
    // work partition: workgroup q starts at task position lo_q = ceil(q C / G); the chunk j holding it
    // (pre[j] <= lo_q < pre[j + 1]) is found by binary search, and the task inside it is the first row block
    // whose cost span (after the chunk's staging cost) starts at or after lo_q (one past the chunk's last: the
    // next chunk's first)
    // (both GEMMs' partitions at once: thread i takes workgroup i of gate_up, or i - g_gu of down)
    if (tid == 0) {
        tstart[g_gu] = n;
        tstart[g_gu + 1 + g_dn] = n;
    }
    for (int idx = tid; idx < g_gu + g_dn; idx += blockDim.x) {
        const int m = idx >= g_gu, q = m ? idx - g_gu : idx;
        const int G = m ? g_dn : g_gu;
        const int* P = m ? pre_dn : pre_gu;
        const uint32_t* task = m ? task_dn : task_gu;
        int* ts = tstart + (m ? g_gu + 1 : 0);
        const long long C = P[n];
        const long long lo = C == 0 ? 0 : floor_div((long long)q * C + G - 1, G);
        if (lo >= C) {
            ts[q] = n;
            continue;
        }
        int a = 0, b = n;   // P[a] <= lo < P[b]
        while (b - a > 1) {
            const int mid = (a + b) >> 1;
            if (P[mid] <= lo) a = mid;
            else b = mid;
        }
        const int nrb = int(task[a] & 255u), span = int(task[a] >> 8);
        const long long off = lo - P[a] - (m ? STAGE_COST_DN : STAGE_COST_GU);
        const int r = off <= 0 ? 0 : int((off + span - 1) / span);
        ts[q] = r >= nrb ? a + 1 : (a | (r << TASK_RB_SHIFT));
    }
}

// Place every (token, k) pair in its slot; tok_slots[t, K] = the shared slot (or -1). grid nb, 256 threads.
__global__ void __launch_bounds__(256) place_kernel(const int* __restrict__ topk, const float* __restrict__ topw,
                                                    uint32_t* __restrict__ mask, uint32_t* __restrict__ blockmax,
                                                    const int* __restrict__ bpre, int T, int E, int K, int block,
                                                    int has_shared,
                                                    int* __restrict__ slot_token, float* __restrict__ slot_weight,
                                                    int* __restrict__ tok_slots) {
    // the block's masks and slot bases staged in LDS while the (token, k) pairs load, so the slot of a pair
    // costs one global round trip
    __shared__ uint32_t m_s[MAXE];
    __shared__ int bp_s[MAXE];
    const int b = blockIdx.x, t0 = b * block, tb = min(block, T - t0);
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
        m_s[e] = mask[size_t(b) * E + e];
        bp_s[e] = bpre[size_t(b) * E + e];
    }
    __syncthreads();
    for (int p = threadIdx.x; p < tb * K; p += blockDim.x) {
        const int tl = p / K, k = p % K, t = t0 + tl;
        const int ex = topk[size_t(t) * K + k];
        const int sl = bp_s[ex] + __popc(m_s[ex] & ((1u << tl) - 1u));
        slot_token[sl] = t;
        slot_weight[sl] = topw[size_t(t) * K + k];
        tok_slots[size_t(t) * (K + 1) + k] = sl;
    }
    for (int tl = threadIdx.x; tl < tb; tl += blockDim.x) {
        const int t = t0 + tl;
        if (has_shared) {
            slot_token[T * K + t] = t;
            slot_weight[T * K + t] = 1.0f;
        }
        tok_slots[size_t(t) * (K + 1) + K] = has_shared ? T * K + t : -1;
    }
    // the block's token masks and pool maxima are consumed: leave them zero for the next call's atomics
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
        mask[size_t(b) * E + e] = 0u;
        blockmax[size_t(b) * E + e] = 0u;
    }
}

}  // namespace

hipError_t launch_router_logits(const float* x, const float* Wr, int T, int H, int E, float* part, int8_t* q,
                                float* qs, int* qsum, hipStream_t st) {
    if (T <= 32) {
        router_decode_kernel<<<dim3(E / RD_EW, 1, ROUTER_KC), 256, RD_LDS, st>>>(x, Wr, T, H, E, part, q, qs, qsum);
    } else if (T <= 256) {
        // 32 x 32 tiles: with 256 experts 512 workgroups at 256 tokens (64 x 64: 128, half of the CUs). The line was
        // measured at 256 experts only; fewer give fewer workgroups at either size.
        router_mfma_kernel<1><<<dim3(E / 32, (T + 31) / 32, ROUTER_KC), 256, rm_lds<1>(), st>>>(x, Wr, T, H, E, part, q,
                                                                                               qs, qsum);
    } else {
        router_mfma_kernel<2><<<dim3(E / 64, (T + 63) / 64, ROUTER_KC), 256, rm_lds<2>(), st>>>(x, Wr, T, H, E, part, q,
                                                                                               qs, qsum);
    }
    return hipGetLastError();
}

hipError_t launch_route(const float* part, int nchunks, const float* bias, int T, int E, int K, int C, int block,
                        float rscale, float* sig, uint32_t* blockmax, int32_t* topk, float* topw, uint32_t* mask,
                        const QuantX& qx, hipStream_t st) {
    if (E > MAXE || block > MAXB) return hipErrorInvalidValue;
    const DecodeState ds{blockmax, mask};
    if (C < E) {
        if (qx.x) score_kernel<true><<<T, 256, 0, st>>>(part, nchunks, bias, T, E, block, 1, sig, blockmax, qx);
        else score_kernel<false><<<T, 256, 0, st>>>(part, nchunks, bias, T, E, block, 1, sig, blockmax, qx);
        select_token_kernel<true, false><<<T, 256, 0, st>>>(part, nchunks, sig, bias, T, E, K, C, block, rscale,
                                                             topk, topw, ds, QuantX{});
    } else if (qx.x) {
        select_token_kernel<false, true><<<T, 256, 0, st>>>(part, nchunks, sig, bias, T, E, K, C, block, rscale,
                                                             topk, topw, ds, qx);
    } else {
        select_token_kernel<false, false><<<T, 256, 0, st>>>(part, nchunks, sig, bias, T, E, K, C, block, rscale,
                                                              topk, topw, ds, qx);
    }
    return hipGetLastError();
}

hipError_t launch_decode_route(const float* part, int nchunks, const float* bias, int T, int E, int K, int C,
                               float rscale, float* sig, int32_t* topk, float* topw, uint32_t* blockmax,
                               uint32_t* tmask, int has_shared, const int8_t* bits, int32_t* count, int32_t* start,
                               Item* units_gu, Item* units_dn, int* n_units, int32_t* slot_token, float* slot_weight,
                               int32_t* tok_slots, int max_gu, int max_dn, const QuantX& qx, int dispatch,
                               hipStream_t st) {
    if (T > 32 || E > MAXE) return hipErrorInvalidValue;
    const DecodeState ds{blockmax, tmask};
    // (the pool of a block of one token holds that token's best C >= K experts: selecting inside it changes nothing)
    if (C < E && T > 1) {
        if (qx.x) score_kernel<true><<<T, 256, 0, st>>>(part, nchunks, bias, T, E, MAXB, 1, sig, blockmax, qx);
        else score_kernel<false><<<T, 256, 0, st>>>(part, nchunks, bias, T, E, MAXB, 1, sig, blockmax, qx);
        select_token_kernel<true, false><<<T, 256, 0, st>>>(part, nchunks, sig, bias, T, E, K, C, MAXB, rscale, topk,
                                                             topw, ds, QuantX{});
    } else if (qx.x) {
        select_token_kernel<false, true><<<T, 256, 0, st>>>(part, nchunks, sig, bias, T, E, K, C, MAXB, rscale, topk,
                                                             topw, ds, qx);
    } else {
        select_token_kernel<false, false><<<T, 256, 0, st>>>(part, nchunks, sig, bias, T, E, K, C, MAXB, rscale,
                                                              topk, topw, ds, qx);
    }
    const DispatchOut d{has_shared, 16, bits, count, start, units_gu, units_dn, n_units, slot_token, slot_weight,
                        tok_slots, max_gu, max_dn};
    if (dispatch) dispatch_kernel<<<1, 256, 0, st>>>(T, E, K, topk, topw, ds, d);
    return hipGetLastError();
}

__global__ void __launch_bounds__(256) zero_u32_kernel(uint32_t* __restrict__ a, uint32_t* __restrict__ b, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        a[i] = 0u;
        b[i] = 0u;
    }
}

hipError_t launch_zero_decode_state(uint32_t* blockmax, uint32_t* tmask, int E, hipStream_t st) {
    zero_u32_kernel<<<1, 256, 0, st>>>(blockmax, tmask, E);
    return hipGetLastError();
}

hipError_t launch_masks(const int32_t* topk, const float* topw, int T, int E, int K, int block, int32_t* topk_out,
                        float* topw_out, uint32_t* mask, hipStream_t st) {
    const int nb = (T + block - 1) / block;
    masks_kernel<<<nb, 256, 0, st>>>(topk, topw, T, E, K, block, topk_out, topw_out, mask);
    return hipGetLastError();
}

hipError_t launch_plan(const uint32_t* mask, int T, int E, int K, int block, int has_shared, int ntok, int tiled,
                       const int8_t* bits, int32_t* count, int32_t* start, int32_t* bpre, Item* units_gu,
                       Item* units_dn, Item* tunits_gu, Item* tunits_dn, int* n_units, int g_gu, int g_dn,
                       int* tstart, int max_chunks, hipStream_t st) {
    const size_t lds = (5 * size_t(max_chunks) + 2) * sizeof(uint32_t);
    plan_kernel<<<1, PLAN_NT, lds, st>>>(mask, T, E, K, block, has_shared, ntok, tiled, bits, count, start, bpre,
                                     units_gu, units_dn, tunits_gu, tunits_dn, n_units, g_gu, g_dn, tstart,
                                     max_chunks);
    return hipGetLastError();
}

hipError_t launch_place(const int32_t* topk, const float* topw, uint32_t* mask, uint32_t* blockmax,
                        const int32_t* bpre, int T, int E, int K, int block, int has_shared, int32_t* slot_token,
                        float* slot_weight, int32_t* tok_slots, hipStream_t st) {
    const int nb = (T + block - 1) / block;
    place_kernel<<<nb, 256, 0, st>>>(topk, topw, mask, blockmax, bpre, T, E, K, block, has_shared, slot_token,
                                     slot_weight, tok_slots);
    return hipGetLastError();
}

}  // namespace llmoe
