// matmul.hip — the matmul_dt dispatch (metal_mps_matmul_dt's contract,
// metal/shim.h:99-137) and the fused bf16 Linear entry point.
//
// Routing inside gorch_hip_matmul_dt:
//   - f32 A [M,K] x bf16 B stored [N,K] (transB; the nn.Linear layout,
//     ops.go:788-807 -> bf16_matmul.go:159-173): the MFMA weight-streaming
//     kernel in gemv.hip;
//   - every other transpose/dtype combination, and every batch of more than
//     one entry: k_mm, one launch over the batch, a kernel per operand
//     layout and dtype, each operand split into bf16 matrix-core terms.
#include <algorithm>

#include "common.h"

namespace gh {

int launch_gemm_bf16w(hipStream_t s, const float* A, const uint16_t* W, const float* bias,
                      const float* residual, const OutDesc& od, int M, int N, int K, int epilogue,
                      bool act_bf16);

// ---------------------------------------------------------------------------
// k_mm: C[b] = opA(A[b]) @ opB(B[b]) on the matrix cores, one launch for the
// whole batch (blockIdx.z = batch entry), a kernel per operand layout and
// dtype.
//
// Terms: bf16 storage is one exact term; an f32 value is hi (truncated to
// bf16), mid (the remainder truncated) and lo (what is left, rounded): x =
// hi + mid + lo to ~2^-25 relative. The term products with ta + tb <= 2 are
// kept (the rest lie below f32 rounding) and accumulated in f32 by
// v_mfma_f32_16x16x32_bf16: one product for bf16 x bf16, three for f32 x
// bf16, six for f32 x f32.
//
// A block takes a T x T tile of C (4 waves of T/2 x T/2) and steps K by BK.
// Each thread loads a patch of each operand with the widest loads its layout
// allows (8 k of P rows), splits it into terms once, and writes them to LDS
// in [term][row][k] order, 16 bytes at a time, with the 16-byte chunks
// XOR-swizzled so that neither the writes nor the 16-row fragment reads
// conflict. The next step's loads are issued before a step's MFMAs: up to
// 1024^3 the chain of K steps binds (load latency, split, LDS, MFMAs), above
// it the matrix cores (f32 x f32 at 2000^3 runs them at 730 TFLOP/s). Rows
// past the matrix are clamped into it (computed, never stored) and the loads
// need only element alignment, so odd sizes run the same loop; only a last
// step that is ragged in K, or whose row-contiguous loads would run past the
// operand's end, is gathered element by element through a buffer resource
// whose out-of-range reads are zeros.
// The products are formed as (B fragment) x (A fragment), which leaves each
// lane 4 consecutive columns of one row of C: one 16-byte store.
// Tile sizes and what they measured: launch_mm.
template <int T_, int BK_, bool F32>
struct MmOperand {
    static constexpr int T = T_, BK = BK_;
    static constexpr int NT = F32 ? 3 : 1, E = F32 ? 4 : 2;
    static constexpr int CH = BK / 8;           // 16-byte chunks per LDS row
    static constexpr int P = T * BK / 8 / 256;  // rows per thread patch
    static constexpr int ELEMS = NT * T * BK;   // LDS elements per stage
    static_assert(P >= 1 && T % P == 0, "one patch per thread");
    __device__ static __forceinline__ int swz(int row, int c) {
        return CH == 8 ? (c ^ (row & 7)) : (c ^ ((row >> 1) & 3));
    }
    // the 16-byte words of one patch: [row][8 k] of raw storage
    struct Patch {
        uint32_t w[P][8 * E / 4];
    };
    // k-contiguous patches: chunk tid + 256 i of the step (row q / CH, k 8 (q % CH));
    // row-contiguous: rows P (tid % (T / P)) .. +P, k 8 (tid / (T / P)) .. +8
    template <bool KC>
    __device__ static __forceinline__ int row_of(int i) {
        const int tid = threadIdx.x & 255;
        return KC ? (tid + 256 * i) / CH : P * (tid % (T / P)) + i;
    }
    template <bool KC>
    __device__ static __forceinline__ int k_of(int i) {
        const int tid = threadIdx.x & 255;
        return 8 * (KC ? (tid + 256 * i) % CH : tid / (T / P));
    }
    // element loads of a ragged step: zeros past K; rows past the last one are
    // clamped to it, or with SKIP read as zeros too, which costs a compare but
    // no memory traffic (thin outputs: 263 x 1547 x 1 x 28 hh 14.7 -> 12.0 us;
    // but 39 x 29 x 1093 x 80 hh, two steps, 7.1 -> 9.1)
    template <bool KC, bool SKIP>
    __device__ static __forceinline__ void load_edge(const char* base, int r0, int R, int K, int k0, Patch& p) {
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(base, (long long)R * K * E);
#pragma unroll
        for (int i = 0; i < P; i++) {
            const int row = SKIP ? r0 + row_of<KC>(i) : min(r0 + row_of<KC>(i), R - 1);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int k = k0 + k_of<KC>(i) + e;
                const int off = k < K && (!SKIP || row < R) ? (KC ? row * K + k : k * R + row) * E : kOutOfRange;
                if constexpr (F32) {
                    p.w[i][e] = __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0);
                } else {
                    const uint32_t h = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, off, 0, 0);
                    if (e & 1) p.w[i][e / 2] |= h << 16;
                    else p.w[i][e / 2] = h;
                }
            }
        }
    }
    // whole patches: every address inside the operand (the caller sends a
    // step that could leave it to load_edge)
    template <bool KC>
    __device__ static __forceinline__ void load(const char* base, int r0, int R, int K, int k0, Patch& p) {
        typedef uint32_t v4 __attribute__((ext_vector_type(4), aligned(2)));
        if constexpr (KC) {
#pragma unroll
            for (int i = 0; i < P; i++) {
                const int row = min(r0 + row_of<true>(i), R - 1);
                const uint32_t off = ((uint32_t)row * K + k0 + k_of<true>(i)) * E;
#pragma unroll
                for (int q = 0; q < E / 2; q++) {
                    const v4 v = *reinterpret_cast<const v4*>(base + off + 16 * q);
#pragma unroll
                    for (int e = 0; e < 4; e++) p.w[i][4 * q + e] = v[e];
                }
            }
        } else {
            // 8 loads of P consecutive elements, transposed in registers
            constexpr int W = P * E;  // bytes per load
            typedef uint32_t vw __attribute__((ext_vector_type(W >= 4 ? W / 4 : 1), aligned(2)));
            int row = r0 + row_of<false>(0);
            if (row >= R) row = max(R - P, 0);
            uint32_t v[8][W >= 4 ? W / 4 : 1];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const uint32_t off = ((uint32_t)(k0 + k_of<false>(0) + e) * R + row) * E;
                if constexpr (W == 2) {
                    v[e][0] = *reinterpret_cast<const uint16_t*>(base + off);
                } else if constexpr (W == 4) {
                    typedef uint32_t u1 __attribute__((aligned(2)));
                    v[e][0] = *reinterpret_cast<const u1*>(base + off);
                } else {
                    const vw x = *reinterpret_cast<const vw*>(base + off);
#pragma unroll
                    for (int q = 0; q < W / 4; q++) v[e][q] = x[q];
                }
            }
#pragma unroll
            for (int i = 0; i < P; i++) {
                if constexpr (F32) {
#pragma unroll
                    for (int e = 0; e < 8; e++) p.w[i][e] = v[e][i];
                } else {
                    // bf16 i of the load: half i & 1 of word i / 2
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        p.w[i][e] = __builtin_amdgcn_perm(v[2 * e + 1][i / 2], v[2 * e][i / 2],
                                                          (i & 1) ? 0x07060302u : 0x05040100u);
                }
            }
        }
    }
    // terms of the patch into LDS
    template <bool KC>
    __device__ static __forceinline__ void store(uint16_t* lds, const Patch& p) {
#pragma unroll
        for (int i = 0; i < P; i++) {
            const int row = row_of<KC>(i), c = swz(row, k_of<KC>(i) / 8);
            uint16_t* dst = lds + row * BK + 8 * c;
            if constexpr (!F32) {
                *reinterpret_cast<u32x4*>(dst) = u32x4{p.w[i][0], p.w[i][1], p.w[i][2], p.w[i][3]};
            } else {
                u32x4 t[3];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t b0 = p.w[i][2 * q], b1 = p.w[i][2 * q + 1];
                    t[0][q] = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
                    const float r0 = __uint_as_float(b0) - __uint_as_float(b0 & 0xffff0000u);
                    const float r1 = __uint_as_float(b1) - __uint_as_float(b1 & 0xffff0000u);
                    const uint32_t m0 = __float_as_uint(r0), m1 = __float_as_uint(r1);
                    t[1][q] = __builtin_amdgcn_perm(m1, m0, 0x07060302u);
                    const float l0 = r0 - __uint_as_float(m0 & 0xffff0000u);
                    const float l1 = r1 - __uint_as_float(m1 & 0xffff0000u);
                    t[2][q] = (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)l0) |
                              ((uint32_t)__builtin_bit_cast(uint16_t, (__bf16)l1) << 16);
                }
#pragma unroll
                for (int q = 0; q < 3; q++) *reinterpret_cast<u32x4*>(dst + q * T * BK) = t[q];
            }
        }
    }
};

// KA / KB: A stored [M][K] (not transA), B stored [N][K] (transB). G groups
// of 4 waves share a block's tile: group q takes steps q, q + G, ... through
// LDS stages of its own and the groups' sums are added in order at the end.
// ONE: the whole of K is one step (K <= BK). No second stage and no loop, so
// that three to eight blocks fit a CU: such products are bound by their output,
// and their tiles' loads, barriers and stores overlap only across blocks. They are
// formed as A x B, one 4-byte column a lane: 16-byte stores of 16 rows at once
// wrote 8192 x 8192 x 8 hh in 63 us, this in 52.
template <int T, int G, int BK, bool KA, bool FA, bool KB, bool FB, bool ONE = false>
__global__ __launch_bounds__(256 * G, ONE && BK == 32 ? 4 : G <= 2 ? 2 : 1) void k_mm(const void* __restrict__ A, const void* __restrict__ B,
                                                   float* __restrict__ C, int M, int N, int K, int xcd_map) {
    using OA = MmOperand<T, BK, FA>;
    using OB = MmOperand<T, BK, FB>;
    constexpr int TF = T / 32;  // 16-wide fragments per wave and side
    constexpr int STAGE = OA::ELEMS + OB::ELEMS;
    // two LDS stages (one barrier per step) while two blocks still fit a CU
    constexpr int NS = !ONE && 2 * G * STAGE * 2 <= (G > 1 ? 144 : 80) * 1024 ? 2 : 1;
    constexpr size_t kRed = G > 1 ? (size_t)(G - 1) * T * T * 4 : 0;
    constexpr size_t kLds = (size_t)G * NS * STAGE * 2 > kRed ? (size_t)G * NS * STAGE * 2 : kRed;
    __shared__ __align__(16) char smem[kLds];
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3;
    const int grp = G > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
    uint16_t* lds = reinterpret_cast<uint16_t*>(smem) + grp * NS * STAGE;
    const int wm = wave >> 1, wn = wave & 1, r = lane & 15, g = lane >> 4;
    // xcd_map (batches, a one-dimensional grid): blocks are dealt to the 8
    // XCDs round-robin, and XCD k takes the k-th contiguous run of the tiles
    // of all batch entries, so that an entry's tiles share its operands in
    // one L2 (30 x 92 x 725 x 687 ff 46.9 -> 41.7 us; a single product
    // gains nothing and would pay the divisions, 1024^3 hh 9.5 -> 10.0)
    int bz = blockIdx.z, m0 = blockIdx.y * T, n0 = blockIdx.x * T;
    if (xcd_map) {
        const int gx = (N + T - 1) / T, gy = (M + T - 1) / T;
        const int items = gridDim.x, q8 = items >> 3, rem8 = items & 7;
        const int xcd = blockIdx.x & 7;
        const int item = xcd * q8 + min(xcd, rem8) + ((int)blockIdx.x >> 3);
        bz = item / (gx * gy);
        const int t2 = item - bz * (gx * gy);
        m0 = t2 / gx * T;
        n0 = t2 % gx * T;
    }
    const char* Ab = reinterpret_cast<const char*>(A) + (size_t)bz * M * K * OA::E;
    const char* Bb = reinterpret_cast<const char*>(B) + (size_t)bz * K * N * OB::E;

    floatx4 acc[TF][TF];
#pragma unroll
    for (int i = 0; i < TF; i++)
#pragma unroll
        for (int j = 0; j < TF; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    typename OA::Patch pa;
    typename OB::Patch pb;
    auto compute = [&](const uint16_t* buf) {
#pragma unroll
        for (int kk = 0; kk < BK / 32; kk++) {
            bf16x8 af[TF][OA::NT];
#pragma unroll
            for (int i = 0; i < TF; i++) {
                const int row = wm * (T / 2) + 16 * i + r;
#pragma unroll
                for (int t = 0; t < OA::NT; t++)
                    af[i][t] = *reinterpret_cast<const bf16x8*>(buf + (t * T + row) * BK + 8 * OA::swz(row, 4 * kk + g));
            }
#pragma unroll
            for (int j = 0; j < TF; j++) {
                const int row = wn * (T / 2) + 16 * j + r;
                bf16x8 bfr[OB::NT];
#pragma unroll
                for (int t = 0; t < OB::NT; t++)
                    bfr[t] = *reinterpret_cast<const bf16x8*>(buf + OA::ELEMS + (t * T + row) * BK +
                                                              8 * OB::swz(row, 4 * kk + g));
#pragma unroll
                for (int ta = 0; ta < OA::NT; ta++)
#pragma unroll
                    for (int tb = 0; tb < OB::NT; tb++)
                        if (ta + tb <= 2)
#pragma unroll
                            for (int i = 0; i < TF; i++)
                                acc[i][j] = ONE ? mfma16x16x32(af[i][ta], bfr[tb], acc[i][j])
                                                : mfma16x16x32(bfr[tb], af[i][ta], acc[i][j]);
            }
        }
    };
    // steps the whole-patch loads may take: all of K in whole steps, less the
    // last one when a row-contiguous patch can run past the last row's end
    // (by fewer than P elements, so by less than a row), none when a row is
    // shorter than a patch
    int nf = K / BK;
    if (K % BK == 0 && ((!KA && M % OA::P) || (!KB && N % OB::P))) nf--;
    if ((!KA && M < OA::P) || (!KB && N < OB::P)) nf = 0;
    auto store = [&](uint16_t* buf) {
        OA::template store<KA>(buf, pa);
        OB::template store<KB>(buf + OA::ELEMS, pb);
    };
    const int ns = (K + BK - 1) / BK;
    auto load = [&](int s) {
        if (s < nf) {
            OA::template load<KA>(Ab, m0, M, K, s * BK, pa);
            OB::template load<KB>(Bb, n0, N, K, s * BK, pb);
        } else if (s < ns) {
            OA::template load_edge<KA, ONE>(Ab, m0, M, K, s * BK, pa);
            OB::template load_edge<KB, ONE>(Bb, n0, N, K, s * BK, pb);
        }
    };
    float* Cb = C + (size_t)bz * M * N;
    load(grp);
    if constexpr (ONE) {
        static_assert(G == 1, "one step");
        store(lds);
        __syncthreads();
        compute(lds);
        // lane (r, g): column r, rows 4g .. 4g + 3 of each 16 x 16 fragment
#pragma unroll
        for (int i = 0; i < TF; i++)
#pragma unroll
            for (int j = 0; j < TF; j++) {
                const int m = m0 + wm * (T / 2) + 16 * i + 4 * g, n = n0 + wn * (T / 2) + 16 * j + r;
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (m + v < M && n < N) Cb[(size_t)(m + v) * N + n] = acc[i][j][v];
            }
        return;
    }
    if constexpr (NS == 2) {
        if (grp < ns) store(lds);
        __syncthreads();
    }
    for (int s0 = 0, it = 0; s0 < ns; s0 += G, it++) {
        const int s = s0 + grp;
        if constexpr (NS == 2) {
            load(s + G);
            if (s < ns) compute(lds + (it & 1) * STAGE);
            if (s + G < ns) store(lds + ((it + 1) & 1) * STAGE);
            __syncthreads();
        } else {
            if (s < ns) store(lds);
            __syncthreads();
            load(s + G);
            if (s < ns) compute(lds);
            __syncthreads();  // the step's fragments have been read
        }
    }
    if constexpr (G > 1) {
        // (the last step's barrier has passed: the stages are free)
        float4* red = reinterpret_cast<float4*>(smem);
        const int t = threadIdx.x & 255;
        if (grp > 0)
#pragma unroll
            for (int i = 0; i < TF; i++)
#pragma unroll
                for (int j = 0; j < TF; j++)
                    red[((grp - 1) * TF * TF + i * TF + j) * 256 + t] =
                        make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int q = 0; q < G - 1; q++)
#pragma unroll
            for (int i = 0; i < TF; i++)
#pragma unroll
                for (int j = 0; j < TF; j++) {
                    const float4 v = red[(q * TF * TF + i * TF + j) * 256 + t];
                    acc[i][j] += floatx4{v.x, v.y, v.z, v.w};
                }
    }
    // lane (r, g): row r, columns 4g .. 4g + 3 of each 16 x 16 fragment
#pragma unroll
    for (int i = 0; i < TF; i++) {
        const int m = m0 + wm * (T / 2) + 16 * i + r;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TF; j++) {
            const int n = n0 + wn * (T / 2) + 16 * j + 4 * g;
            float* dst = Cb + (size_t)m * N + n;
            typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
            if (n + 3 < N) {
                *reinterpret_cast<f4u*>(dst) = f4u{acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
            } else {
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (n + v < N) dst[v] = acc[i][j][v];
            }
        }
    }
}

// Tile, K groups and step width (BK; 0: 64, 32 for 128 x 128 tiles of f32).
// HALF: two bf16 operands only (4 groups of 64 x 64 stages fit LDS then).
template <int T, int G, int BK = 0, bool ONE = false, bool HALF = false>
static void launch_mm_t(hipStream_t s, const void* A, const void* B, float* C, int M, int N, int K, int batch,
                        bool ka, bool fa, bool kb, bool fb) {
    const unsigned gx = (N + T - 1) / T, gy = (M + T - 1) / T;
    const int xcd_map = batch > 1 && (long long)gx * gy * batch < (1ll << 22);
    const dim3 grid = xcd_map ? dim3(gx * gy * batch) : dim3(gx, gy, batch);
#define GH_MM(KA, FA, KB, FB)                                                                                      \
    hipLaunchKernelGGL((k_mm<T, G, BK ? BK : (T == 128 && (FA || FB) ? 32 : 64), KA, FA, KB, FB, ONE>), grid, dim3(256 * G), \
                       0, s, A, B, C, M, N, K, xcd_map)
#define GH_MM_T(KA, KB)                              \
    do {                                             \
        if constexpr (HALF) GH_MM(KA, false, KB, false); \
        else if (fa && fb) GH_MM(KA, true, KB, true); \
        else if (fa) GH_MM(KA, true, KB, false);     \
        else if (fb) GH_MM(KA, false, KB, true);     \
        else GH_MM(KA, false, KB, false);            \
    } while (0)
    if (ka && kb) GH_MM_T(true, true);
    else if (ka) GH_MM_T(true, false);
    else GH_MM_T(false, false);
#undef GH_MM_T
#undef GH_MM
}

// Tile and K groups, by the number of 64 x 64 tiles n64 of the whole call
// (256 CUs), measured in HIP graphs (us; T/G, f = f32, h = bf16 operands):
//   n64 <= 64: 32 x 32 tiles, 4 groups. Few tiles are bound by the chain of
//     K steps on each: 64 x 64 x 2048 ff 15.1 against 37.6 (64/2), 47.9
//     (64/1); 1103 x 65 x 1699 ff 14.9 / 33.0 / 42.3; 512^3 hh 3.6 / 4.9 /
//     5.2; but 128 tiles (8 x 200^2 x 200 fh) 7.2 / 5.9 / 6.6.
//   n64 <= 256: 64 x 64, 2 groups, one block per CU: 1024^3 ff 23.0 against
//     26.6 (64/1) and 34.6 (32/4); two bf16 operands leave LDS for 4 groups,
//     which pay from a few steps each: hh 8.7 / 9.5 (64/2) / 11.9 / 14.0.
//   else 64 x 64, 1 group: 2048^3 hh 39.6 against 41.4 (64/2), 45.2 (128/1);
//     30 x 92 x 725 x 687 ff 41.7 / 50.3 / 50.9.
//   128 x 128 from 512 such tiles: half the operand traffic, 4096^3 hh 165
//     against 224 (64/1), fh 398 / 598; 48 x 512 x 512 x 64 ff 20.2 / 20.6.
// Up to 64 deep a product is one step (ONE), of 32 up to 32: 192 x 1 x 640 x
// 64 hh 5.1 us, 8.0 in 128 x 128 tiles; 54 x 1869 x 10 x 4 hh 5.4 / 12.8; 16 x
// 16 x 16 3.4, 3.6 on four groups. 128 x 128 tiles stay where they are mostly
// full (three 64 x 64 tiles in each at least) and
//   K > 32: 48 x 1024 x 1024 x 40 ff 0.75 of the time of ONE;
//   K 8 .. 32, 4096 tiles and more: 25 x 1753 x 1946 x 19 fh 90.4 / 123.8 (rows
//     that start off a 64-byte line), 16 x 2048 x 2048 x 8 hh 57.6 / 63.0; but
//     K = 4 8192 x 8192 54 / 43, and below 4096 tiles ONE is even or better
//     (64 x 512 x 512 x 19 fh 18.7 / 17.3).
// The element-wise gather kernel all this replaced: 1024^3 hh 52.4, 48 x 512 x
// 512 x 64 ff 49.2; at 32 deep and less it had 32-wide steps and one stage, and
// the sizes above took 8.5, 5.5, 3.4, 131 and 57 us.
enum MmKind { kMm32x4, kMm64x4, kMm64x2, kMm64x1, kMm128, kMmOne32, kMmOne64, kMmOne64K64, kMm128K32 };
static MmKind mm_kind(int M, int N, int K, int batch, bool half) {
    const long long n64 = (long long)((M + 63) / 64) * ((N + 63) / 64) * batch;
    const long long n128 = (long long)((M + 127) / 128) * ((N + 127) / 128) * batch;
    const bool full128 = n64 >= 3 * n128;
    if (K <= 32) {
        if (n128 >= 4096 && full128 && K >= 8) return kMm128K32;
        return n64 <= 64 ? kMmOne32 : kMmOne64;
    }
    if (K <= 64 && (n128 < 512 || !full128)) return n64 <= 64 ? kMmOne32 : kMmOne64K64;
    if (n64 <= 64) return kMm32x4;
    if (n64 <= 256) return half && K >= 512 ? kMm64x4 : kMm64x2;
    return n128 < 512 ? kMm64x1 : kMm128;
}

// The kernel's name (gorch_hip_kernel_choice).
const char* matmul_choice_name(int M, int N, int K, int batch, bool a_bf16, bool b_bf16) {
    static const char* const kName[] = {"mm32x4",  "mm64x4",  "mm64x2",     "mm64x1",    "mm128",
                                        "mm32one", "mm64one", "mm64one_k64", "mm128_k32"};
    return kName[mm_kind(M, N, K, batch, a_bf16 && b_bf16)];
}

static void launch_mm(hipStream_t s, const void* A, const void* B, float* C, int M, int N, int K, int batch, bool ka,
                      bool fa, bool kb, bool fb) {
#define GH_ARGS s, A, B, C, M, N, K, batch, ka, fa, kb, fb
    switch (mm_kind(M, N, K, batch, !fa && !fb)) {
        case kMm32x4: launch_mm_t<32, 4>(GH_ARGS); break;
        case kMm64x4: launch_mm_t<64, 4, 0, false, true>(GH_ARGS); break;
        case kMm64x2: launch_mm_t<64, 2>(GH_ARGS); break;
        case kMm64x1: launch_mm_t<64, 1>(GH_ARGS); break;
        case kMmOne32: launch_mm_t<32, 1, 64, true>(GH_ARGS); break;
        case kMmOne64: launch_mm_t<64, 1, 32, true>(GH_ARGS); break;
        case kMmOne64K64: launch_mm_t<64, 1, 64, true>(GH_ARGS); break;
        case kMm128K32: launch_mm_t<128, 1, 32>(GH_ARGS); break;
        default: launch_mm_t<128, 1>(GH_ARGS); break;
    }
#undef GH_ARGS
}

static bool linear_fast_ok(const void* x, const void* W, int K) {
    return K % 8 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)W % 16 == 0;
}

}  // namespace gh

using namespace gh;

extern "C" int gorch_hip_linear_bf16_ex(void* stream, const float* x, const uint16_t* W, const float* bias,
                                        const float* residual, float* y, int M, int N, int K, int epilogue,
                                        int flags) {
    GH_REQUIRE(M >= 0 && N >= 0 && K >= 0, "gorch_hip_linear_bf16: negative dimension");
    GH_REQUIRE(epilogue == GORCH_HIP_EPI_NONE || epilogue == GORCH_HIP_EPI_GELU,
               "gorch_hip_linear_bf16: unknown epilogue");
    if (M == 0 || N == 0) return GORCH_HIP_OK;
    GH_REQUIRE(x && W && y, "gorch_hip_linear_bf16: null pointer");
    GH_REQUIRE((const void*)x != (const void*)y, "gorch_hip_linear_bf16: x must not alias y");
    if (!linear_fast_ok(x, W, K)) {
        set_error("gorch_hip_linear_bf16: needs K % 8 == 0 and 16-byte aligned x and W");
        return GORCH_HIP_EUNSUPPORTED;
    }
    GH_REQUIRE((flags & ~GORCH_HIP_LINEAR_ACT_BF16) == 0, "gorch_hip_linear_bf16_ex: unknown flag");
    GH_TRY(bf16_gate(stream_of(stream)));
    if (flags & GORCH_HIP_LINEAR_ACT_BF16)
        return finish(stream, launch_gemm_bf16w(stream_of(stream), x, W, bias, residual, OutDesc::plain(y, N), M, N,
                                                K, epilogue, true));
    return finish(stream, launch_linear_bf16(stream_of(stream), x, W, bias, residual, y, M, N, K, epilogue));
}

extern "C" int gorch_hip_linear_bf16(void* stream, const float* x, const uint16_t* W, const float* bias,
                                     const float* residual, float* y, int M, int N, int K, int epilogue) {
    return gorch_hip_linear_bf16_ex(stream, x, W, bias, residual, y, M, N, K, epilogue, 0);
}

extern "C" size_t gorch_hip_packed_bf16_bytes(int N, int K) {
    if (N <= 0 || K <= 0) return 0;
    return packed_bf16_elems(N, K) * sizeof(uint16_t);
}

extern "C" int gorch_hip_pack_bf16(void* stream, const uint16_t* W, uint16_t* Wp, int N, int K) {
    GH_REQUIRE(N >= 0 && K >= 0, "gorch_hip_pack_bf16: negative dimension");
    if (N == 0 || K == 0) return GORCH_HIP_OK;
    GH_REQUIRE(W && Wp, "gorch_hip_pack_bf16: null pointer");
    GH_REQUIRE(K % 8 == 0 && ((uintptr_t)W | (uintptr_t)Wp) % 16 == 0,
               "gorch_hip_pack_bf16: needs K % 8 == 0 and 16-byte aligned buffers");
    return finish(stream, launch_pack_bf16(stream_of(stream), W, Wp, N, K));
}

extern "C" int gorch_hip_linear_bf16_packed(void* stream, const float* x, const uint16_t* Wp, const float* bias,
                                            const float* residual, float* y, int M, int N, int K, int epilogue) {
    GH_REQUIRE(M >= 0 && N >= 0 && K >= 0, "gorch_hip_linear_bf16_packed: negative dimension");
    GH_REQUIRE(epilogue == GORCH_HIP_EPI_NONE || epilogue == GORCH_HIP_EPI_GELU,
               "gorch_hip_linear_bf16_packed: unknown epilogue");
    if (M == 0 || N == 0) return GORCH_HIP_OK;
    GH_REQUIRE(M <= 16, "gorch_hip_linear_bf16_packed: M must be <= 16 (decode GEMV)");
    GH_REQUIRE(x && Wp && y, "gorch_hip_linear_bf16_packed: null pointer");
    GH_REQUIRE((const void*)x != (const void*)y, "gorch_hip_linear_bf16_packed: x must not alias y");
    GH_REQUIRE(K % 8 == 0 && ((uintptr_t)x | (uintptr_t)Wp) % 16 == 0,
               "gorch_hip_linear_bf16_packed: needs K % 8 == 0 and 16-byte aligned x and Wp");
    GH_TRY(bf16_gate(stream_of(stream)));
    return finish(stream, launch_linear_packed_od(stream_of(stream), x, Wp, bias, residual, OutDesc::plain(y, N), M,
                                                  N, K, epilogue, LinearExtras{}));
}

// C = 0 for an empty contraction (K == 0), as a kernel rather than a memset
// so that a captured graph holds no memset node
__global__ void k_fill_zero(float* __restrict__ c, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        c[i] = 0.f;
}

namespace gh {

// The matmul_dt routing without the probe gate (the probe itself runs
// through it).
int matmul_dt_raw(hipStream_t s, const void* A, const void* B, float* C, uint32_t M, uint32_t N, uint32_t K,
                  uint32_t batch, int transA, int transB, int aBF16, int bBF16) {
    if (transA && transB) {
        set_error("gorch_hip_matmul_dt: transA && transB is not supported");
        return GORCH_HIP_EUNSUPPORTED;
    }
    if (M == 0 || N == 0 || batch == 0) return GORCH_HIP_OK;
    GH_REQUIRE(A && B && C, "gorch_hip_matmul_dt: null pointer");
    GH_REQUIRE(M < (1u << 30) && N < (1u << 30) && K < (1u << 30) && batch < 65536,
               "gorch_hip_matmul_dt: dimension too large");
    if (K == 0) {
        const size_t n = (size_t)batch * M * N;
        const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 4096);
        hipLaunchKernelGGL(k_fill_zero, dim3(blocks), dim3(256), 0, s, C, n);
        count(CNT_ELEMENTWISE);
        return check_launch("fill_zero");
    }
    if (batch == 1 && !transA && transB && !aBF16 && bBF16 && linear_fast_ok(A, B, (int)K)) {
        for (uint32_t b = 0; b < batch; b++) {
            const float* a = reinterpret_cast<const float*>(A) + (size_t)b * M * K;
            const uint16_t* w = reinterpret_cast<const uint16_t*>(B) + (size_t)b * N * K;
            if ((uintptr_t)a % 16 != 0) break;
            GH_TRY(launch_linear_bf16(s, a, w, nullptr, nullptr, C + (size_t)b * M * N, (int)M, (int)N, (int)K,
                                      GORCH_HIP_EPI_NONE));
            if (b + 1 == batch) return GORCH_HIP_OK;
        }
    }
    // the kernel's 32-bit buffer offsets: each batch entry below 2 GiB
    if ((unsigned long long)M * K * (aBF16 ? 2 : 4) >= (1ull << 31) ||
        (unsigned long long)K * N * (bBF16 ? 2 : 4) >= (1ull << 31)) {
        set_error("gorch_hip_matmul_dt: an operand of one batch entry is 2 GiB or more");
        return GORCH_HIP_EUNSUPPORTED;
    }
    launch_mm(s, A, B, C, (int)M, (int)N, (int)K, (int)batch, !transA, !aBF16, transB != 0, !bBF16);
    count(CNT_GENERIC_MATMUL);
    return check_launch("matmul");
}

}  // namespace gh

extern "C" int gorch_hip_matmul_dt(void* stream, const void* A, const void* B, float* C, uint32_t M,
                                   uint32_t N, uint32_t K, int transA, int transB, int aBF16, int bBF16) {
    if (aBF16 || bBF16) GH_TRY(bf16_gate(stream_of(stream)));
    return finish(stream, matmul_dt_raw(stream_of(stream), A, B, C, M, N, K, 1, transA, transB, aBF16, bBF16));
}

extern "C" int gorch_hip_batched_matmul_dt(void* stream, const void* A, const void* B, float* C, uint32_t M,
                                           uint32_t N, uint32_t K, uint32_t batch, int transA, int transB,
                                           int aBF16, int bBF16) {
    if (aBF16 || bBF16) GH_TRY(bf16_gate(stream_of(stream)));
    return finish(stream,
                  matmul_dt_raw(stream_of(stream), A, B, C, M, N, K, batch, transA, transB, aBF16, bBF16));
}
