// gemm.hip — BF16-weight Linear for prefill- and MoE-sized M (M > 16):
//   C[m,n] = residual[m,n] + epi( sum_k A[m,k] * W[n,k] + bias[n] )
// with A f32 [M,K], W bf16 [N,K] (the nn.Linear layout, nn/module.go:61-88).
//
// Three kernels on v_mfma_f32_16x16x32_bf16, chosen by estimated time
// (gemm_choice):
//   k_gemm_kw: few tiles (short prompts, narrow weights): the waves of a block
//     split K, each through LDS stages of its own;
//   k_gemm_db: 64-row tiles of 64, 96 or 128 columns on 2 x (2..4) waves of
//     32 x 32, double-buffered LDS filled through registers;
//   k_gemm_pp: many tiles (long prompts): 256 x (32 TN) tiles on 8 waves, the
//     two waves of a SIMD half a step apart.
// k_gemm_db's LDS rows are padded to 160 bytes, which makes the 16-byte
// fragment reads conflict-free on gfx950 (a 144-byte row measured 2-way
// conflicted); the other two load straight to LDS and swizzle instead.
//
// Activation modes:
//   split (default): A = hi + lo in bf16 (two MFMAs per fragment pair),
//     ~2^-16 relative, i.e. f32-activation accuracy like the reference's
//     widen + f32 sgemm (bf16_matmul.go:166-173);
//   bf16 (GORCH_HIP_LINEAR_ACT_BF16): A rounded to bf16 (RNE), one MFMA —
//     the bf16 x bf16 -> f32 MPSGraph path (metal/shim.m:808-857).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "stage_lds.h"

namespace gh {

constexpr int kBK = 64;
constexpr int kLDA = kBK + 16;  // bf16 elements per LDS row (160 bytes: conflict-free 16-byte fragment reads)

// Bias of the wave's TN output columns (column nb + 16 j + r), loaded
// before the main loop; zeros without a bias or past N (a buffer resource
// of size 0 or an out-of-range offset, no branch).
template <int TN>
__device__ __forceinline__ void gemm_bias(const float* bias, int N, int nb, int r, float (&bn)[TN]) {
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(bias, bias ? (long long)N * 4 : 0);
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int n = nb + j * 16 + r;
        bn[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, n < N ? n * 4 : kOutOfRange, 0, 0));
    }
}

// Epilogue kinds (template argument EPI of the GEMM kernels): bit 0 the
// tanh GELU, bit 1 a residual input. A residual decided at run time costs
// ~0.4 us at 512 x 768 x 2304 even when absent, so it is compiled in or out.
constexpr int kEpiGelu = 1, kEpiResidual = 2, kEpiPair = 4;
inline int epi_kind(int epilogue, const float* residual) {
    return (epilogue == GORCH_HIP_EPI_GELU ? kEpiGelu : 0) | (residual ? kEpiResidual : 0);
}

// Epilogue of a wave's TM x TN accumulators (16 x 16 MFMA tiles; lane
// (r, g) holds rows 4g .. 4g+3 of column r of each): out = residual +
// epi(acc + bias), written through the output descriptor. mb / nb: the
// wave's first row relative to the block's m0 and its first column. The
// residual is loaded and every value finished before the first store (a
// load after a store waits for the store's write: both count on vmcnt),
// and the bias is added unconditionally (bn reads zeros without one).
template <int TM, int TN, int EPI>
__device__ __forceinline__ void gemm_epilogue(floatx4 (&acc)[TM][TN], const float (&bn)[TN], const float* residual, const OutDesc& od, int pos, int M, int N,
                                              int m0, int mrows, int mb, int nb, int r, int g) {
    constexpr bool GELU = (EPI & kEpiGelu) != 0, RES = (EPI & kEpiResidual) != 0;
    float res[TM][TN][4];
    if constexpr (RES) {
        const __amdgpu_buffer_rsrc_t rsr = make_rsrc(residual + (size_t)m0 * N, (long long)mrows * N * 4);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int n = nb + j * 16 + r;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int ml = mb + i * 16 + 4 * g + v;
                    const int off = (n < N && ml < mrows) ? (ml * N + n) * 4 : kOutOfRange;
                    res[i][j][v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsr, off, 0, 0));
                }
            }
    }
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                // bn is zero without a bias (a select here costs ~0.2 us)
                float s = acc[i][j][v] + bn[j];
                if constexpr (GELU) s = gelu_gemm(s);
                if constexpr (RES) s = res[i][j][v] + s;
                acc[i][j][v] = s;
            }
    // One output segment without per-sequence rows (every Linear but the
    // fused QKV projection): row m at ptr + (m + pos?) * row_stride. The
    // descriptor's general addressing costs ~1.4 us at 512 x 768 x 2304.
    if (od.nseg == 1 && od.rows_per_seq >= (1 << 30) && od.row_stride[0] < (1ll << 31)) {
        const int rs = __builtin_amdgcn_readfirstlane((int)od.row_stride[0]);
        float* base = od.ptr[0] + (long long)(m0 + (od.use_pos[0] ? pos : 0)) * rs;
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int n = nb + j * 16 + r;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int ml = mb + i * 16 + 4 * g + v;
                    if (ml < mrows && n < N) base[(size_t)ml * rs + n] = acc[i][j][v];
                }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int n = nb + j * 16 + r;
        const OutDesc::Col c = od.col(min(n, N - 1), pos);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int m = m0 + mb + i * 16 + 4 * g + v;
                if (m < M && n < N) *od.row(c, m) = acc[i][j][v];
            }
    }
}

// Linear for a few hundred rows (512 x 768 x {2304, 3072}):
// 64 x BN tiles (BN = 32 * WGN) on 2 x WGN waves, each wave a 32 x 32
// sub-tile of 2 x 2 MFMA accumulators. The block's A and W K-steps (64
// wide) go global -> registers -> one of two LDS stage buffers, so each
// step has a single barrier: step i computes from buffer i & 1 while the
// registers of step i + 1 are written into the other buffer. The loads of
// step i + 2 go out at the top of step i (its register set was emptied
// into LDS during step i - 1), so they have two steps to arrive, and the
// LDS writes of step i + 1 are kept after step i's MFMAs (a wait for their
// loads placed between the MFMAs stalls them). The last two steps issue no
// loads; with KT the K tail and the padding step read zeros.
// EPI = kEpiPair: W is [gate | up] of 2N rows, and output column n is
// silu(gate n) * up n: a tile takes BN / 2 columns, each wave 16 gate rows and
// the same 16 up rows, so both products of an output meet in one lane
// (777 x 1024 x 2 x 3072: 32.8 us, 33.4 and 6.8 for the SwiGLU launch before).
template <int WGN, bool SPLIT, bool KT, int EPI>
__global__ __launch_bounds__(128 * WGN) void k_gemm_db(const float* __restrict__ A, const uint16_t* __restrict__ W,
                                                       const float* __restrict__ bias, const float* residual,
                                                       OutDesc od, int M, int N, int K) {
    constexpr int BM = 64, BN = 32 * WGN, NT = 128 * WGN;
    constexpr int NA = SPLIT ? 2 : 1;
    constexpr int TM = 2, TN = 2;
    constexpr int A_TOT = BM * kBK / 4, W_TOT = BN * kBK / 8;  // float4 / uint4 chunks per step
    constexpr int A_F4 = (A_TOT + NT - 1) / NT, W_U4 = (W_TOT + NT - 1) / NT;
    constexpr int STAGE = (NA * BM + BN) * kLDA;  // bf16 elements per stage buffer
    __shared__ __align__(16) uint16_t lds[2 * STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    constexpr bool PAIR = EPI == kEpiPair;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * (PAIR ? BN / 2 : BN);
    const int mrows = min(BM, M - m0), ncols = min(PAIR ? BN / 2 : BN, N - n0);
    const __amdgpu_buffer_rsrc_t rsa = make_rsrc(A + (size_t)m0 * K, (long long)mrows * K * 4);
    // PAIR: the resource spans the tile's gate rows through its up rows
    const __amdgpu_buffer_rsrc_t rsw = make_rsrc(W + (size_t)n0 * K, (long long)(PAIR ? N + ncols : ncols) * K * 2);
    // W row of the tile's row q: clamped to the valid ones
    auto wrow = [&](int q) {
        return PAIR ? min((q >> 5) * 16 + (q & 15), ncols - 1) + ((q & 16) ? N : 0) : min(q, ncols - 1);
    };
    // Chunk q of a step: A row q / 16, float4 column q % 16; W row q / 8,
    // uint4 column q % 8. Threads past the chunk count (WGN = 3) repeat the
    // last chunk: the same value to the same LDS slot. Rows past M or N are
    // clamped into the tile (computed, never stored).
    float4 ra[2][A_F4];
    uint4 rw[2][W_U4];
    auto gload = [&](int k0, float4 (&a)[A_F4], uint4 (&wv)[W_U4]) {
#pragma unroll
        for (int i = 0; i < A_F4; i++) {
            const int q = min(tid + NT * i, A_TOT - 1), row = q >> 4, k = k0 + 4 * (q & 15);
            const int off = (!KT || k < K) ? (min(row, mrows - 1) * K + k) * 4 : kOutOfRange;
            a[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rsa, off, 0, 0));
        }
#pragma unroll
        for (int i = 0; i < W_U4; i++) {
            const int q = min(tid + NT * i, W_TOT - 1), row = q >> 3, k = k0 + 8 * (q & 7);
            const int off = (!KT || k < K) ? (wrow(row) * K + k) * 2 : kOutOfRange;
            wv[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsw, off, 0, 0));
        }
    };
    auto sstore = [&](int b, const float4 (&a)[A_F4], const uint4 (&wv)[W_U4]) {
        uint16_t* As = lds + b * STAGE;
        uint16_t* Ws = As + NA * BM * kLDA;
#pragma unroll
        for (int i = 0; i < A_F4; i++) {
            const int q = min(tid + NT * i, A_TOT - 1), row = q >> 4, c4 = q & 15;
            const float f[4] = {a[i].x, a[i].y, a[i].z, a[i].w};
            uint16_t hi[4], lo[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (SPLIT) {
                    const uint32_t u = __float_as_uint(f[e]) & 0xffff0000u;
                    hi[e] = (uint16_t)(u >> 16);
                    lo[e] = __builtin_bit_cast(uint16_t, (__bf16)(f[e] - __uint_as_float(u)));
                } else {
                    hi[e] = __builtin_bit_cast(uint16_t, (__bf16)f[e]);
                }
            }
            *reinterpret_cast<uint2*>(&As[row * kLDA + 4 * c4]) =
                make_uint2(hi[0] | ((uint32_t)hi[1] << 16), hi[2] | ((uint32_t)hi[3] << 16));
            if (SPLIT)
                *reinterpret_cast<uint2*>(&As[(BM + row) * kLDA + 4 * c4]) =
                    make_uint2(lo[0] | ((uint32_t)lo[1] << 16), lo[2] | ((uint32_t)lo[3] << 16));
        }
#pragma unroll
        for (int i = 0; i < W_U4; i++) {
            const int q = min(tid + NT * i, W_TOT - 1), row = q >> 3, c8 = q & 7;
            *reinterpret_cast<uint4*>(&Ws[row * kLDA + 8 * c8]) = wv[i];
        }
    };
    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int r = lane & 15, g = lane >> 4;
    auto compute = [&](int b) {
        const uint16_t* As = lds + b * STAGE;
        const uint16_t* Ws = As + NA * BM * kLDA;
#pragma unroll
        for (int kk = 0; kk < kBK; kk += 32) {
            bf16x8 bfr[TN];
#pragma unroll
            for (int j = 0; j < TN; j++)
                bfr[j] = *reinterpret_cast<const bf16x8*>(&Ws[(wn * 32 + j * 16 + r) * kLDA + kk + 8 * g]);
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const bf16x8 ahi = *reinterpret_cast<const bf16x8*>(&As[(wm * 32 + i * 16 + r) * kLDA + kk + 8 * g]);
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = mfma16x16x32(ahi, bfr[j], acc[i][j]);
                if (SPLIT) {
                    const bf16x8 alo =
                        *reinterpret_cast<const bf16x8*>(&As[(BM + wm * 32 + i * 16 + r) * kLDA + kk + 8 * g]);
#pragma unroll
                    for (int j = 0; j < TN; j++) acc[i][j] = mfma16x16x32(alo, bfr[j], acc[i][j]);
                }
            }
        }
    };
    float bn[TN];
    if constexpr (!PAIR) gemm_bias<TN>(bias, N, n0 + wn * 32, r, bn);
    const int pos = __builtin_amdgcn_readfirstlane(od.pos_dev ? *od.pos_dev : 0);
    // steps padded to an even count (a padding step reads zeros, KT)
    const int nk = (K + kBK - 1) / kBK;
    const int nkp = (nk + 1) & ~1;
    gload(0, ra[0], rw[0]);
    __builtin_amdgcn_sched_barrier(0);
    gload(kBK, ra[1], rw[1]);
    __builtin_amdgcn_sched_barrier(0);
    sstore(0, ra[0], rw[0]);
    __syncthreads();
    auto step = [&](int s, int it, bool st, bool ld) {
        if (ld) gload((it + 2) * kBK, ra[s], rw[s]);
        compute(it & 1);
        __builtin_amdgcn_sched_barrier(0);
        if (st) sstore((it + 1) & 1, ra[s ^ 1], rw[s ^ 1]);
        __syncthreads();
    };
    int it0 = 0;
    for (; it0 < nkp - 2; it0 += 2) {
        step(0, it0, true, true);
        step(1, it0 + 1, true, true);
    }
    step(0, it0, true, false);
    step(1, it0 + 1, false, false);

    if constexpr (PAIR) {
        const int n = n0 + wn * 16 + r;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int ml = wm * 32 + i * 16 + 4 * g + v;
                const float gt = acc[i][0][v];
                if (ml < mrows && n < N)
                    od.ptr[0][(size_t)(m0 + ml) * N + n] = gt * sigmoidf_ref(gt) * acc[i][1][v];
            }
    } else {
        gemm_epilogue<TM, TN, EPI>(acc, bn, residual, od, pos, M, N, m0, mrows, wm * 32, n0 + wn * 32, r, g);
    }
}

// ---------------------------------------------------------------------------
// k_gemm_kw and k_gemm_pp stage 32-wide steps (stage_lds.h): A rows stay f32
// (128 bytes, 8 chunks) and are split into their bf16 terms as a fragment is
// read (f32 and hi + lo take the same LDS), W rows are bf16 (64 bytes, 4
// chunks).
constexpr int kStK = 32;

// the bf16 terms of 8 consecutive f32 of an A row: hi (truncated) and lo
// (the remainder rounded), or one rounded term
template <bool SPLIT>
__device__ __forceinline__ void a_terms(const float4& u, const float4& v, bf16x8& hi, bf16x8& lo) {
    const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
    if constexpr (SPLIT) {
        u32x4 h;
#pragma unroll
        for (int q = 0; q < 4; q++)
            h[q] = __builtin_amdgcn_perm(__float_as_uint(f[2 * q + 1]), __float_as_uint(f[2 * q]), 0x07060302u);
        hi = __builtin_bit_cast(bf16x8, h);
#pragma unroll
        for (int e = 0; e < 8; e++)
            lo[e] = (__bf16)(f[e] - __uint_as_float(__float_as_uint(f[e]) & 0xffff0000u));
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) hi[e] = (__bf16)f[e];
    }
}

// Epilogue of 4 consecutive columns n .. n + 3 of one row at a time (the
// accumulator layout of (W fragment) x (A fragment) products). Bias and
// residual come through buffer resources (columns past N or rows past the
// tile read zeros or a neighbour, never stored); `put` writes the columns
// below N through the output descriptor.
struct Out4 {
    typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
    const OutDesc& od;
    __amdgpu_buffer_rsrc_t rb, rr;
    int m0, pos, M, N;
    bool flat, seg4;
    // rows m0 .. m0 + mrows; seg4: every output segment starts at a multiple
    // of 4 columns
    __device__ __forceinline__ Out4(const OutDesc& o, const float* bias, const float* residual, int m0_, int mrows,
                                    int pos_, int M_, int N_, int seg4_)
        : od(o), rb(make_rsrc(bias, bias ? (long long)N_ * 4 : 0)),
          rr(make_rsrc(residual + (residual ? (size_t)m0_ * N_ : 0), residual ? (long long)mrows * N_ * 4 : 0)),
          m0(m0_), pos(pos_), M(M_), N(N_), flat(o.nseg == 1 && o.rows_per_seq >= (1 << 30)), seg4(seg4_ != 0) {}
    __device__ __forceinline__ f4u bias(int n) const {
        return __builtin_bit_cast(f4u, __builtin_amdgcn_raw_buffer_load_b128(rb, n * 4, 0, 0));
    }
    __device__ __forceinline__ f4u res(int m, int n) const {
        return __builtin_bit_cast(f4u, __builtin_amdgcn_raw_buffer_load_b128(rr, ((m - m0) * N + n) * 4, 0, 0));
    }
    __device__ __forceinline__ f4u value(const floatx4& acc, const f4u& b, const f4u& r, int epilogue) const {
        f4u o = {acc[0] + b[0], acc[1] + b[1], acc[2] + b[2], acc[3] + b[3]};
        if (epilogue == GORCH_HIP_EPI_GELU)
#pragma unroll
            for (int v = 0; v < 4; v++) o[v] = gelu_gemm(o[v]);
        return r + o;
    }
    __device__ __forceinline__ void put(int m, int n, const f4u& s) const {
        if (m >= M || n >= N) return;
        float* p;
        if (flat) p = od.ptr[0] + (long long)(m + (od.use_pos[0] ? pos : 0)) * od.row_stride[0] + n;
        else p = od.row(od.col(n, pos), m);
        if (n + 3 < N && (flat || seg4)) {
            *reinterpret_cast<f4u*>(p) = s;
        } else {
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (n + v < N) *od.at_p(m, n + v, pos) = s[v];
        }
    }
};

// The tile of this block when each XCD takes one contiguous run of the tiles
// (blocks are dealt to the 8 XCDs round-robin), walked in bands of `band`
// tile rows: the tiles in flight on an XCD then share their A and W panels in
// its L2.
__device__ __forceinline__ void xcd_tile(int band, int& tx, int& ty) {
    const int gx = gridDim.x, gy = gridDim.y, L = blockIdx.y * gx + blockIdx.x;
    const int items = gx * gy, q8 = items >> 3, rem8 = items & 7, xcd = L & 7;
    const int item = xcd * q8 + min(xcd, rem8) + (L >> 3);
    const int b = item / (band * gx), t = item - b * band * gx;
    const int bh = min(band, gy - b * band);
    ty = b * band + t % bh;
    tx = t / bh;
}

// Linear for few tiles (short prompts, narrow weights): the block's G waves
// share a BM x BN tile of the output and split K: wave w takes the 32-wide
// steps w, w + G, ... through NST LDS stages of its own. Nothing is shared
// until the end, so there is no barrier in the loop: a wave waits for its own
// oldest stage (vmcnt), reads its fragments, and sends the next step's loads
// into the stage it has just read, with NST - 1 steps in flight behind it
// (up to 96 KB per CU). The waves' partial tiles meet in LDS and are added
// in wave order. Products are formed as (W fragment) x (A fragment), which
// leaves each lane 4 consecutive columns of one row.
template <int BM, int BN, int G, int NST, bool SPLIT, bool KT>
__global__ __launch_bounds__(64 * G) void k_gemm_kw(const float* __restrict__ A, const uint16_t* __restrict__ W,
                                                    const float* __restrict__ bias, const float* residual, OutDesc od,
                                                    int M, int N, int K, int epilogue, int seg4) {
    constexpr int TM = BM / 16, TN = BN / 16;
    constexpr int kA = BM * 128, kStage = kA + BN * 64;   // bytes of one wave's stage
    constexpr int kLoads = BM / 8 + BN / 16;
    static_assert(NST == 2 || NST == 3, "stages");
    static_assert((NST - 1) * kLoads < 64, "vmcnt range");
    // one array per stage: reads of one do not wait for loads into another
    __shared__ __align__(16) char st0[G * kStage];
    __shared__ __align__(16) char st1[G * kStage];
    __shared__ __align__(16) char st2[NST > 2 ? G * kStage : 16];
    constexpr int kRed = G * BM * BN * 4;
    static_assert(kRed <= G * kStage * 2, "partial tiles");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int mrows = min(BM, M - m0), ncols = min(BN, N - n0);
    const __amdgpu_buffer_rsrc_t rsa = make_rsrc(A + (size_t)m0 * K, (long long)mrows * K * 4);
    const __amdgpu_buffer_rsrc_t rsw = make_rsrc(W + (size_t)n0 * K, (long long)ncols * K * 2);
    const int pos = __builtin_amdgcn_readfirstlane(od.pos_dev ? *od.pos_dev : 0);

    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int nk = (K + kStK - 1) / kStK;
    const StageLane<8> la(lane, K * 4);
    const StageLane<4> lw(lane, K * 2);
    // chunks of the last step that lie past K
    const int ta = KT && 4 * la.chunk >= K - (nk - 1) * kStK ? kOutOfRange : 0;
    const int tw = KT && 8 * lw.chunk >= K - (nk - 1) * kStK ? kOutOfRange : 0;
    const int wofs = wave * kStage;
    auto issue = [&](char* st, int s) {
        const bool last = KT && s == nk - 1;
        la.issue<BM, KT>(st + wofs, rsa, K * 4, s < nk ? s * 128 : kOutOfRange, last ? ta : 0);
        lw.issue<BN, KT>(st + wofs + kA, rsw, K * 2, s < nk ? s * 64 : kOutOfRange, last ? tw : 0);
    };
    struct Frags {
        float4 a[TM][2];
        bf16x8 w[TN];
    };
    const int ra0 = wofs + r * 128 + 16 * ((2 * g) ^ (r & 7)), ra1 = wofs + r * 128 + 16 * ((2 * g + 1) ^ (r & 7));
    const int rw0 = wofs + kA + r * 64 + 16 * (g ^ ((r >> 1) & 3));
    auto read = [&](const char* st, Frags& f) {
#pragma unroll
        for (int j = 0; j < TN; j++) f.w[j] = *reinterpret_cast<const bf16x8*>(st + (rw0 + j * 1024));
#pragma unroll
        for (int i = 0; i < TM; i++) {
            f.a[i][0] = *reinterpret_cast<const float4*>(st + (ra0 + i * 2048));
            f.a[i][1] = *reinterpret_cast<const float4*>(st + (ra1 + i * 2048));
        }
    };
    auto mul = [&](const Frags& f) {
#pragma unroll
        for (int i = 0; i < TM; i++) {
            bf16x8 hi, lo;
            a_terms<SPLIT>(f.a[i][0], f.a[i][1], hi, lo);
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = mfma16x16x32(f.w[j], hi, acc[i][j]);
            if constexpr (SPLIT)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = mfma16x16x32(f.w[j], lo, acc[i][j]);
        }
    };
    // steps of this wave; the last rounds' missing ones read zeros
    const int rounds = (nk + G - 1) / G;
    issue(st0, wave);
    issue(st1, wave + G);
    if constexpr (NST > 2) issue(st2, wave + 2 * G);
    // one round: wait for the stage (its loads are the oldest NST - 1 stages
    // are newer), read it, refill it, multiply
    constexpr int kWait = (NST - 1) * kLoads;
    auto round = [&](char* st, int it) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(wait_vm(kWait, false));
        asm volatile("" ::: "memory");
        Frags f;
        read(st, f);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(kWaitLgkm0);  // the stage has been read
        asm volatile("" ::: "memory");
        issue(st, wave + (it + NST) * G);
        mul(f);
    };
    int it = 0;
    for (; it + NST <= rounds; it += NST) {
        round(st0, it);
        round(st1, it + 1);
        if constexpr (NST > 2) round(st2, it + 2);
    }
    if (it < rounds) round(st0, it);
    if constexpr (NST > 2)
        if (it + 1 < rounds) round(st1, it + 1);
    // every load has landed before the stages hold the partial tiles
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    float4* p0 = reinterpret_cast<float4*>(st0);
    float4* p1 = reinterpret_cast<float4*>(st1);
    auto part = [&](int w, int f) -> float4* { return (w < G / 2 ? p0 + w * TM * TN * 64 : p1 + (w - G / 2) * TM * TN * 64) + f * 64 + lane; };
    static_assert((G / 2) * TM * TN * 1024 <= G * kStage, "partial tiles fit a stage");
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
            *part(wave, i * TN + j) = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
    __syncthreads();
    const Out4 out(od, bias, residual, m0, mrows, pos, M, N, seg4);
#pragma unroll
    for (int f0 = 0; f0 < TM * TN; f0 += G) {
        const int f = f0 + wave;
        if (TM * TN % G != 0 && f >= TM * TN) break;
        const int m = m0 + (f / TN) * 16 + r, n = n0 + (f % TN) * 16 + 4 * g;
        const Out4::f4u bv = out.bias(n), rv = out.res(m, n);
        floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < G; w++) {
            const float4 v = *part(w, f);
            s = floatx4{s[0] + v.x, s[1] + v.y, s[2] + v.z, s[3] + v.w};
        }
        out.put(m, n, out.value(s, bv, rv, epilogue));
    }
}

// Linear for many tiles (long prompts): 8 waves share a 256 x (32 TN) tile,
// each a 64 x (16 TN) part of it, through three LDS stages.
//
// Two waves run on each SIMD, half a step apart: while waves 0-3 multiply a
// stage (registers only), waves 4-7 read its fragments and send the loads of
// the stage after next, and the other way round in the next half step, so
// the matrix cores wait neither for the fragment reads nor for the barrier.
// 4096^3 runs at 583 TFLOP/s (1,165 on the matrix cores, two terms; this
// card's library bf16 product of that size 1,150-1,240): what is left is the
// loads' share of L2 and LDS (with the loads off 178 us, only the loads 128,
// together 236).
// A wave waits for its own loads (vmcnt, all but the newest stage) before the
// barrier behind which the next stage is first read.
// GELU is compiled in or out: decided at run time, its 64 TN / 4 copies in the
// epilogue cost products without it up to 4% (8192 x 1024 x 6144 192 us, 185 so).
template <int TN, bool SPLIT, bool KT, bool GELU>
__global__ __launch_bounds__(512, 2) void k_gemm_pp(const float* __restrict__ A, const uint16_t* __restrict__ W,
                                                    const float* __restrict__ bias, const float* residual, OutDesc od,
                                                    int M, int N, int K, int seg4, int band) {
    constexpr int TM = 4, BM = 256, BN = 32 * TN, NW = 8;
    constexpr int LA = BM / 8 / NW, LW = (BN / 16 + NW - 1) / NW;  // loads per wave and stage
    constexpr int kA = BM * 128, kStage = kA + LW * NW * 1024;     // bytes (W groups past BN: zeros, unread)
    __shared__ __align__(16) char st0[kStage];
    __shared__ __align__(16) char st1[kStage];
    __shared__ __align__(16) char st2[kStage];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave & 3, wn = wave >> 2, r = lane & 15, g = lane >> 4;
    int tx = blockIdx.x, ty = blockIdx.y;
    if (band) xcd_tile(band, tx, ty);
    const int m0 = ty * BM, n0 = tx * BN;
    const int mrows = min(BM, M - m0), ncols = min(BN, N - n0);
    const __amdgpu_buffer_rsrc_t rsa = make_rsrc(A + (size_t)m0 * K, (long long)mrows * K * 4);
    const __amdgpu_buffer_rsrc_t rsw = make_rsrc(W + (size_t)n0 * K, (long long)ncols * K * 2);
    const int pos = __builtin_amdgcn_readfirstlane(od.pos_dev ? *od.pos_dev : 0);

    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    const int nk = (K + kStK - 1) / kStK;
    const StageLane<8> la(lane, K * 4);
    const StageLane<4> lw(lane, K * 2);
    const int ta = KT && 4 * la.chunk >= K - (nk - 1) * kStK ? kOutOfRange : 0;
    const int tw = KT && 8 * lw.chunk >= K - (nk - 1) * kStK ? kOutOfRange : 0;
    const int awave = wave * LA * 8 * K * 4, wwave = wave * LW * 16 * K * 2;
    auto issue = [&](char* st, int s) {
        const bool last = KT && s == nk - 1;
        la.issue<LA * 8, KT>(st + wave * LA * 1024, rsa, K * 4, s < nk ? s * 128 + awave : kOutOfRange, last ? ta : 0);
        lw.issue<LW * 16, KT>(st + kA + wave * LW * 1024, rsw, K * 2, s < nk ? s * 64 + wwave : kOutOfRange,
                              last ? tw : 0);
    };
    const int ra0 = wm * 8192 + r * 128 + 16 * ((2 * g) ^ (r & 7)), ra1 = wm * 8192 + r * 128 + 16 * ((2 * g + 1) ^ (r & 7));
    const int rw0 = kA + wn * TN * 1024 + r * 64 + 16 * (g ^ ((r >> 1) & 3));
    bf16x8 fw[TN];
    float4 fa[TM][2];
    auto read = [&](const char* st) {
#pragma unroll
        for (int j = 0; j < TN; j++) fw[j] = *reinterpret_cast<const bf16x8*>(st + (rw0 + j * 1024));
#pragma unroll
        for (int i = 0; i < TM; i++) {
            fa[i][0] = *reinterpret_cast<const float4*>(st + (ra0 + i * 2048));
            fa[i][1] = *reinterpret_cast<const float4*>(st + (ra1 + i * 2048));
        }
    };
    auto mul = [&] {
#pragma unroll
        for (int i = 0; i < TM; i++) {
            bf16x8 hi, lo;
            a_terms<SPLIT>(fa[i][0], fa[i][1], hi, lo);
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = mfma16x16x32(fw[j], hi, acc[i][j]);
            if constexpr (SPLIT)
#pragma unroll
                for (int j = 0; j < TN; j++) acc[i][j] = mfma16x16x32(fw[j], lo, acc[i][j]);
        }
    };
    constexpr int kWait = LA + LW;  // the newest stage's loads may stay in flight
    auto meet = [&](auto wait) {
        asm volatile("" ::: "memory");
        if constexpr (decltype(wait)::value != 0) __builtin_amdgcn_s_waitcnt(decltype(wait)::value);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    };
    using C0 = std::integral_constant<int, 0>;
    using CVm = std::integral_constant<int, wait_vm(kWait, false)>;
    using CLgkm = std::integral_constant<int, kWaitLgkm0>;
    using CVmLgkm = std::integral_constant<int, wait_vm(kWait, true)>;
    issue(st0, 0);
    issue(st1, 1);
    meet(CVm{});
    auto run = [&](auto late_tag) {
        constexpr bool LATE = decltype(late_tag)::value;
        auto step = [&](const char* cur, char* nxt, int s) {
            read(cur);
            issue(nxt, s + 2);
            if constexpr (LATE) meet(CVmLgkm{});
            else meet(CLgkm{});
            __builtin_amdgcn_s_setprio(1);
            mul();
            __builtin_amdgcn_s_setprio(0);
            if constexpr (LATE) meet(C0{});
            else meet(CVm{});
        };
        if constexpr (LATE) meet(C0{});
        int s = 0;
        for (; s + 3 <= nk; s += 3) {
            step(st0, st2, s);
            step(st1, st0, s + 1);
            step(st2, st1, s + 2);
        }
        if (s < nk) step(st0, st2, s);
        if (s + 1 < nk) step(st1, st0, s + 1);
        if constexpr (!LATE) meet(C0{});
    };
    if (wave < 4) run(std::false_type{});
    else run(std::true_type{});
    const Out4 out(od, bias, residual, m0, mrows, pos, M, N, seg4);
    const int nw = n0 + wn * TN * 16 + 4 * g, mw = m0 + wm * 64 + r;
    Out4::f4u bv[TN], rv[2][TN];
#pragma unroll
    for (int j = 0; j < TN; j++) {
        bv[j] = out.bias(nw + 16 * j);
        rv[0][j] = out.res(mw, nw + 16 * j);
    }
    // the next 16 rows' residual is requested before this one's stores (a
    // load after a store would wait for the store's write)
#pragma unroll
    for (int i = 0; i < TM; i++) {
        if (i + 1 < TM)
#pragma unroll
            for (int j = 0; j < TN; j++) rv[(i + 1) & 1][j] = out.res(mw + 16 * (i + 1), nw + 16 * j);
#pragma unroll
        for (int j = 0; j < TN; j++)
            out.put(mw + 16 * i, nw + 16 * j,
                    out.value(acc[i][j], bv[j], rv[i & 1][j], GELU ? GORCH_HIP_EPI_GELU : GORCH_HIP_EPI_NONE));
    }
}

// every output segment starts at a multiple of 4 columns
static int segments_by_4(const OutDesc& od) {
    int ok = 1;
    for (int i = 0; i + 1 < od.nseg; i++) ok &= od.n_end[i] % 4 == 0;
    return ok;
}

template <int TN>
static void launch_pp(hipStream_t s, const float* A, const uint16_t* W, const float* bias, const float* residual,
                      const OutDesc& od, int M, int N, int K, int epilogue, bool act_bf16) {
    const dim3 grid((N + 32 * TN - 1) / (32 * TN), (M + 255) / 256);
    const int seg4 = segments_by_4(od);
    // bands of 4 tile rows per XCD: 8192 x 1600 x 6400 347 -> 328 us (8: 333)
    constexpr int band = 4;
#define GH_PP(SP, KTV, GE)                                                                                      \
    hipLaunchKernelGGL((k_gemm_pp<TN, SP, KTV, GE>), grid, dim3(512), 0, s, A, W, bias, residual, od, M, N, K, seg4, band)
#define GH_PP_E(SP, KTV)                                          \
    do {                                                          \
        if (epilogue == GORCH_HIP_EPI_GELU) GH_PP(SP, KTV, true); \
        else GH_PP(SP, KTV, false);                               \
    } while (0)
    if (K % kStK) {
        if (act_bf16) GH_PP_E(false, true);
        else GH_PP_E(true, true);
    } else {
        if (act_bf16) GH_PP_E(false, false);
        else GH_PP_E(true, false);
    }
#undef GH_PP_E
#undef GH_PP
}

template <int BM, int BN, int G, int NST>
static void launch_kw(hipStream_t s, const float* A, const uint16_t* W, const float* bias, const float* residual,
                      const OutDesc& od, int M, int N, int K, int epilogue, bool act_bf16) {
    const dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
    const int seg4 = segments_by_4(od);
#define GH_KW(SP, KTV)                                                                                            \
    hipLaunchKernelGGL((k_gemm_kw<BM, BN, G, NST, SP, KTV>), grid, dim3(64 * G), 0, s, A, W, bias, residual, od, M, N, K, \
                       epilogue, seg4)
    if (K % kStK) {
        if (act_bf16) GH_KW(false, true);
        else GH_KW(true, true);
    } else {
        if (act_bf16) GH_KW(false, false);
        else GH_KW(true, false);
    }
#undef GH_KW
}

static int cu_count() {
    static const int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1)
            n = 256;
        return n;
    }();
    return cus;
}

// Tile width for k_gemm_db: the most 64-row blocks that still fit one
// round on the chip (measured at 512 x 768: N = 2304 on 64 x 96, 192
// blocks, 7.1 us; N = 3072 on 64 x 96, 256 blocks, 7.4 us, against 7.5 /
// 7.6 us on 64 x 128), the widest when every width exceeds it.
static int db_waves(int M, int N) {
    const long long mb = (M + 63) / 64;
    int best = 4;
    long long best_blocks = 0;
    for (int w = 4; w >= 2; w--) {
        const long long blocks = mb * ((N + 32 * w - 1) / (32 * w));
        if (blocks <= cu_count() && blocks > best_blocks) {
            best = w;
            best_blocks = blocks;
        }
    }
    return best;
}

template <int WGN, bool SPLIT>
static void launch_db_t(hipStream_t s, const float* A, const uint16_t* W, const float* bias, const float* residual,
                        const OutDesc& od, int M, int N, int K, int epilogue) {
    dim3 grid((N + 32 * WGN - 1) / (32 * WGN), (M + 63) / 64);
    const int nk = (K + kBK - 1) / kBK;
    const bool kt = K % kBK != 0 || nk % 2 != 0;
#define GH_DB_L(KTV, EV) \
    hipLaunchKernelGGL((k_gemm_db<WGN, SPLIT, KTV, EV>), grid, dim3(128 * WGN), 0, s, A, W, bias, residual, od, M, N, K)
#define GH_DB_E(KTV)                               \
    switch (epi_kind(epilogue, residual)) {        \
        case 0: GH_DB_L(KTV, 0); break;            \
        case kEpiGelu: GH_DB_L(KTV, kEpiGelu); break; \
        case kEpiResidual: GH_DB_L(KTV, kEpiResidual); break; \
        default: GH_DB_L(KTV, kEpiGelu | kEpiResidual); break; \
    }
    if (kt) GH_DB_E(true)
    else GH_DB_E(false)
#undef GH_DB_E
#undef GH_DB_L
}

template <bool SPLIT>
static void launch_db(hipStream_t s, const float* A, const uint16_t* W, const float* bias, const float* residual,
                      const OutDesc& od, int M, int N, int K, int epilogue) {
    switch (db_waves(M, N)) {
        case 2: launch_db_t<2, SPLIT>(s, A, W, bias, residual, od, M, N, K, epilogue); break;
        case 3: launch_db_t<3, SPLIT>(s, A, W, bias, residual, od, M, N, K, epilogue); break;
        default: launch_db_t<4, SPLIT>(s, A, W, bias, residual, od, M, N, K, epilogue); break;
    }
}

// Kernel and tile by estimated time. Each estimate (us) is a sum of terms
// fitted (least squares on the relative error, near the fastest kernel) to
// 1,474 measured launches of every kernel: 17 to 9,000 rows, K 32 to 12,288, N
// 48 to 50,257, both activation modes, weights rotated so that large ones come
// from HBM. n = blocks on the busiest CU, load = blocks per CU, k = K steps:
//   k_gemm_db  a + b k ceil(n / blocks that fit a CU) + c k n + d k load
//   k_gemm_kw  a + b n + c (steps of a wave) n
//   k_gemm_pp  a + b n + c k n + d k load
// each plus e per MB of operands that the XCDs read into their L2s (A once
// per column tile and W once per row tile, 8 at most; k_gemm_pp's bands share
// them) and f per MB written (f2 for k_gemm_db when N is no multiple of 4:
// its rows then start off a 16-byte boundary).
// The choice is on average 1.0% slower than the fastest kernel of a size. It is
// more than 5% slower than k_gemm_db at 16 of 1,126 sizes of less than a round
// of 128 x 128 tiles, 14% at most: the K-split tiles have to be 3% faster by
// estimate. With fewer terms, one set for both activation modes
// and no traffic term the average was 3.4%, and K-split tiles ran where
// k_gemm_db is 1.2 to 1.6 times as fast: 777 x 1600 x 6400 80.6 us against
// 61.5, 1400 x 896 x 4864 62.6 / 48.9, with bf16 activations 79.2 / 50.9 and
// 60.4 / 38.8.
enum GemmKind { kDb, kKw16x32, kKw32x32, kKw32x64, kKw64x64, kPp4, kPp5, kPp6, kPp7, kPp8 };
struct GemmChoice {
    GemmKind kind;
    double us;
};
static GemmChoice gemm_choice(int M, int N, int K, bool act_bf16) {
    auto cdiv = [](long long a, long long b) { return (a + b - 1) / b; };
    const double cus = cu_count(), mb = 1e-6;
    const double out = 4 * mb * M * N;
    auto traffic = [&](int bm, int bn) {
        return mb * ((double)std::min(8ll, cdiv(N, bn)) * 4 * M * K + (double)std::min(8ll, cdiv(M, bm)) * 2 * N * K);
    };
    // the grid's second dimension
    auto rows_ok = [&](int bm) { return cdiv(M, bm) <= 65535; };
    GemmChoice best{kDb, 1e30};
    {
        // a, b, c, d, e, f, f2 for 64, 96 and 128 columns; split, bf16 activations
        constexpr double C[2][3][7] = {{{3.86, 0.241, 0.162, 0, 0.0427, 0.223, 0.287},
                                        {3.88, 0, 0.535, 0.0288, 0.0192, 0.210, 0.250},
                                        {4.01, 0.150, 0.360, 0.0336, 0.0223, 0.179, 0.270}},
                                       {{3.67, 0.123, 0.163, 0, 0.0393, 0.164, 0.212},
                                        {3.71, 0.0467, 0.268, 0, 0.0380, 0.196, 0.268},
                                        {3.85, 0.0941, 0.224, 0, 0.0435, 0.167, 0.237}}};
        constexpr int kFit[2][3] = {{2, 2, 2}, {4, 3, 2}};  // blocks that fit a CU (LDS)
        const int w = db_waves(M, N);
        const double* c = C[act_bf16][w - 2];
        const double blocks = (double)cdiv(M, 64) * cdiv(N, 32 * w), n = std::ceil(blocks / cus), k = (double)cdiv(K, 64);
        if (rows_ok(64))
            best.us = c[0] + k * (c[1] * std::ceil(n / kFit[act_bf16][w - 2]) + c[2] * n + c[3] * blocks / cus) +
                      c[4] * traffic(64, 32 * w) + out * (N % 4 == 0 ? c[5] : c[6]);
    }
    // (`rank` orders the kernels: the estimate, raised for the K-split tiles)
    double rank = best.us;
    auto take = [&](GemmKind kind, double us, double r) {
        if (r >= rank) return;
        rank = r;
        best = {kind, us};
    };
    {
        constexpr int T[4][3] = {{16, 32, 8}, {32, 32, 8}, {32, 64, 4}, {64, 64, 4}};  // rows, columns, waves
        constexpr double C[2][4][5] = {{{2.19, 1.18, 0.390, 0.0110, 0.715},              // a, b, c, e, f
                                        {2.18, 1.74, 0.454, 0.0383, 0.373},
                                        {2.47, 1.52, 0.395, 0.0294, 0.242},
                                        {2.68, 2.47, 0.555, 0.0350, 0.208}},
                                       {{2.17, 1.15, 0.393, 0.0061, 0.793},
                                        {2.20, 1.67, 0.433, 0.0382, 0.406},
                                        {2.42, 1.43, 0.390, 0.0277, 0.286},
                                        {2.66, 2.33, 0.523, 0.0356, 0.125}}};
        double kw = 1e30;
        int at = 0;
        for (int i = 0; i < 4; i++) {
            const double n = std::ceil((double)cdiv(M, T[i][0]) * cdiv(N, T[i][1]) / cus);
            const double* c = C[act_bf16][i];
            const double us = c[0] + n * (c[1] + c[2] * cdiv(cdiv(K, kStK), T[i][2])) +
                              c[3] * traffic(T[i][0], T[i][1]) + c[4] * out;
            if (rows_ok(T[i][0]) && us < kw) {
                kw = us;
                at = i;
            }
        }
        take((GemmKind)(kKw16x32 + at), kw, kw / 0.97);
    }
    // 256 rows of A, and of a residual, behind one 2 GiB resource
    if (256ll * 4 * std::max(K, N) < kOutOfRange && rows_ok(256)) {
        constexpr double C[2][5][5] = {{{3.86, 5.69, 0.520, 0.335, 0.0641},  // a, b, c, d, f for 4 to 8 column groups
                                        {3.73, 5.73, 0.708, 0.309, 0.102},
                                        {3.14, 7.75, 0.794, 0.329, 0.0979},
                                        {2.36, 7.76, 0.971, 0.252, 0.154},
                                        {0.584, 11.3, 1.01, 0.392, 0.139}},
                                       {{4.20, 5.07, 0.520, 0.0783, 0.0775},
                                        {3.83, 6.43, 0.543, 0.0942, 0.0855},
                                        {3.16, 8.15, 0.563, 0.127, 0.0862},
                                        {3.14, 7.53, 0.601, 0.139, 0.126},
                                        {1.93, 10.0, 0.611, 0.185, 0.122}}};
        for (int tn = 4; tn <= 8; tn++) {
            const double* c = C[act_bf16][tn - 4];
            const double blocks = (double)cdiv(M, 256) * cdiv(N, 32 * tn), n = std::ceil(blocks / cus);
            const double k = (double)cdiv(K, kStK);
            const double us = c[0] + n * (c[1] + c[2] * k) + c[3] * k * blocks / cus + c[4] * out;
            take((GemmKind)(kPp4 + tn - 4), us, us);
        }
    }
    return best;
}

// The kernel's name (gorch_hip_kernel_choice).
const char* gemm_choice_name(int M, int N, int K, bool act_bf16) {
    static const char* const kDbName[3] = {"db64x64", "db64x96", "db64x128"};
    static const char* const kName[9] = {"kw16x32",   "kw32x32",   "kw32x64",   "kw64x64",  "pp256x128",
                                         "pp256x160", "pp256x192", "pp256x224", "pp256x256"};
    const GemmKind k = gemm_choice(M, N, K, act_bf16).kind;
    return k == kDb ? kDbName[db_waves(M, N) - 2] : kName[k - kKw16x32];
}

// y[m, n] = silu(x W[n]) * (x W[N + n]) over a [2N, K] weight for more than 16
// rows: k_gemm_db's paired epilogue, where it is estimated faster than the
// Linear of 2N columns and a SwiGLU launch. Both sides are fitted to 220
// measured sizes (17 to 8,192 rows; the choice is on average 0.2% off the
// faster side); the launch's 12 bytes an output mostly come from the Linear's
// output still in cache. The K-split tiles keep few rows (17 x 1024 x 2 x 3072
// 8.4 us against 12.4 paired) and the 256-row tiles long and wide prompts
// (1400 x 2560 x 2 x 9728 278 against 320, 2048 x 4096 x 2 x 12288 690 / 924);
// in between the pair wins (777 x 1024 x 2 x 3072 36.9 / 30.1, 8192 x 896 x 2 x
// 4864 391 / 353).
bool gemm_pair_swiglu_ok(int M, int N, int K) {
    // the resource over the gate and the up rows; the grid's second dimension
    if (M <= 16 || 4ll * N * K >= kOutOfRange || M > 64 * 65535) return false;
    auto cdiv = [](long long a, long long b) { return (a + b - 1) / b; };
    const double cus = cu_count(), out = 4e-6 * M * N, k = (double)cdiv(K, 64);
    const double blocks = (double)cdiv(M, 64) * cdiv(N, 64), n = std::ceil(blocks / cus);
    const double pair = 3.85 + k * (0.165 * std::ceil(n / 2) + 0.418 * n + 0.0344 * blocks / cus) + 0.329 * out;
    return pair < gemm_choice(M, 2 * N, K, false).us + 2.3 + 0.571 * out;
}
int launch_gemm_pair_swiglu(hipStream_t s, const float* A, const uint16_t* W, float* y, int M, int N, int K) {
    const dim3 grid((N + 63) / 64, (M + 63) / 64);
    const int nk = (K + kBK - 1) / kBK;
    const OutDesc od = OutDesc::plain(y, N);
    if (K % kBK != 0 || nk % 2 != 0)
        hipLaunchKernelGGL((k_gemm_db<4, true, true, kEpiPair>), grid, dim3(512), 0, s, A, W, nullptr, nullptr, od, M, N, K);
    else
        hipLaunchKernelGGL((k_gemm_db<4, true, false, kEpiPair>), grid, dim3(512), 0, s, A, W, nullptr, nullptr, od, M, N, K);
    count(CNT_GEMM);
    return check_launch("gemm_pair_swiglu");
}

int launch_gemm_bf16w(hipStream_t s, const float* A, const uint16_t* W, const float* bias,
                      const float* residual, const OutDesc& od, int M, int N, int K, int epilogue,
                      bool act_bf16) {
#define GH_ARGS s, A, W, bias, residual, od, M, N, K, epilogue
    switch (gemm_choice(M, N, K, act_bf16).kind) {
        case kKw16x32: launch_kw<16, 32, 8, 3>(GH_ARGS, act_bf16); break;
        case kKw32x32: launch_kw<32, 32, 8, 3>(GH_ARGS, act_bf16); break;
        case kKw32x64: launch_kw<32, 64, 4, 3>(GH_ARGS, act_bf16); break;
        case kKw64x64: launch_kw<64, 64, 4, 2>(GH_ARGS, act_bf16); break;
        case kPp4: launch_pp<4>(GH_ARGS, act_bf16); break;
        case kPp5: launch_pp<5>(GH_ARGS, act_bf16); break;
        case kPp6: launch_pp<6>(GH_ARGS, act_bf16); break;
        case kPp7: launch_pp<7>(GH_ARGS, act_bf16); break;
        case kPp8: launch_pp<8>(GH_ARGS, act_bf16); break;
        default:
            if (act_bf16) launch_db<false>(GH_ARGS);
            else launch_db<true>(GH_ARGS);
            break;
    }
#undef GH_ARGS
    count(CNT_GEMM);
    return check_launch("gemm_bf16w");
}

}  // namespace gh
