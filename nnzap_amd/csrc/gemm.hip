// Prefill dequant-GEMM on gfx950 matrix cores.
//
// C[P x M] = A[P x K] . dequant(W[M x K])^T for a prompt of P tokens, where A
// holds the f16 activations of the decode path and W is a Q1 (1-bit, +-s)
// matrix.  The reference has no batched prefill: it runs P sequential decode
// steps (nnmetal/src/transformer.zig:4032-4068), and its only dequant-matmul
// (`qmm`, compute.metal:2975-3083) stores W as [K x N] for the MNIST network.
//
// Three kernels on v_mfma_f32_16x16x32_f16 with fp32 accumulation:
//   * qgemm_kernel, the main one: the presets' weights (1-bit of group size
//     128, 4-bit of group size 64 with bf16 scales) with K a multiple of 512;
//   * dq_gemm_kernel (1-bit) and dq4_gemm_kernel (4-bit): every other K and
//     group size, f16 scales of 4-bit weights, less aligned pointers, short
//     1-bit launches (qgemm_short).
// In all of them a block owns 64 tokens, its waves are 2 W-row halves x KQ
// k-phases (a W fragment expanded in registers feeds 4 MFMAs, an A fragment
// read from LDS feeds 2 or 4, the KQ partial tiles meet in LDS at the end), A
// goes straight into LDS (global_load_lds) with 16-byte piece p of row r at
// slot p ^ (r & 15), so the 16 rows of a fragment read hit distinct banks, and
// there is one barrier per stage.  +-s times an f16 activation is exact in the
// MFMA, so a 1-bit result differs from the decode QMV only in fp32 summation
// order.  Epilogues match the decode kernels: f16 store (Q/K/V), residual +=
// (O, down), silu(a)*b of a gate/up pair stored as f16.
#include "internal.h"

#include <algorithm>

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // register arrays of 16-byte pieces
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <int V> struct IC { static constexpr int value = V; };   // a compile-time index argument

constexpr int BM = 64, BN = 64, BK = 64;

// ---- 1-bit weights of any K and group size (multiples of 64): W staged as
// packed bits, a 16-byte entry per row and k-step (two code words and the
// group scale), expanded in registers to f16 +-s.
// KQ k-phases (2 KQ waves, 128 KQ threads); an LDS stage holds KQ k-steps.
template <int KQ> constexpr int SK = BK * KQ;        // k per LDS stage
template <int KQ> constexpr int PIECES = SK<KQ> / 8; // 16-byte pieces per A row and stage
template <int KQ> constexpr int WROW = KQ + 1;       // W entries per LDS row (one of padding)

// One 16-byte global load per lane straight into LDS: lane l's bytes land
// at LDS address lds + 16 l (lds wave-uniform, in M0).  In asm rather than
// the builtin: for the builtin the compiler waits for every such load in
// flight before any LDS read it cannot prove apart (here: the fragment reads
// of the other stage buffer), which would serialise the pipeline.  Its
// completion is waited for explicitly (load_barrier); the compiler's own
// vmcnt waits stay correct, only more conservative, with these loads
// unknown to it (loads complete in order).  The s_nop is the one wait state
// gfx9 requires between an SALU write of M0 and an LDS DMA reading it (the
// compiler's hazard check does not look into asm).
__device__ __forceinline__ void global_load_lds16(const void *g, uint32_t lds) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(lds) : "memory");
}

// Workgroup barrier for a pipelined loop staging through registers: the
// wave's own LDS stores are waited for, then s_barrier.  __syncthreads()
// would add a release fence, which also waits for the next stage's global
// loads still in flight.  The empty asm statements keep the compiler from
// moving LDS accesses across.
constexpr int LGKM0_IMM = 15 | (3 << 14) | (7 << 4);   // gfx9 waitcnt immediate: lgkmcnt 0 only
__device__ __forceinline__ void step_barrier() {
    __builtin_amdgcn_s_waitcnt(LGKM0_IMM);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Workgroup barrier for a pipelined loop loading A straight into LDS: the
// wave's loads into LDS and its own LDS stores are waited for (vmcnt 0,
// lgkmcnt 0: the data of a global_load_lds is in LDS when it is counted),
// then s_barrier.  The empty asm statements keep the compiler from moving
// LDS accesses across.
constexpr int VM0_LGKM0_IMM = 7 << 4;   // gfx9 waitcnt immediate, expcnt not waited
__device__ __forceinline__ void load_barrier() {
    __builtin_amdgcn_s_waitcnt(VM0_LGKM0_IMM);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Eight weight bits (k ascending from bit 0) -> the B fragment's eight f16
// values: +s where the bit is set, -s where it is clear.  ns2 holds (-s, -s).
// z2 = z | z << 15 carries the byte twice, so one shift by 15 - 2q brings bit
// 2q to position 15 (low half's sign) and bit 2q+1 to position 31.
__device__ __forceinline__ half8 expand_bits(uint32_t z, uint32_t ns2) {
    // z2 is formed in asm so that the compiler does not fold the shifts below
    // into 32-bit multiplies (quarter rate); each dword is then one shift and
    // one three-input bit operation.
    uint32_t z2;
    asm("v_lshl_or_b32 %0, %1, 15, %1" : "=v"(z2) : "v"(z));
    u32x4 e;
    e[0] = ((z2 << 15) & 0x80008000u) ^ ns2;
    e[1] = ((z2 << 13) & 0x80008000u) ^ ns2;
    e[2] = ((z2 << 11) & 0x80008000u) ^ ns2;
    e[3] = ((z2 << 9) & 0x80008000u) ^ ns2;
    return __builtin_bit_cast(half8, e);
}

// silu(c) * u of a gate/up pair, as c / (1 + 2^(-c log2 e)) * u on the
// hardware exponential and reciprocal (each within about one ulp): a few
// float32 ulps from the correctly rounded c / (1 + exp(-c)) * u, well below
// the f16 (or bf16) rounding of the stored result, in 4 instructions where
// expf and the IEEE division take about 20.  c -> -inf: the exponential
// overflows to +inf and the product to -0; c -> +inf: c * u.
__device__ __forceinline__ float silu_mul(float c, float u) {
    const float e = __builtin_amdgcn_exp2f(-c * 1.44269504088896341f);
    return c * __builtin_amdgcn_rcpf(1.f + e) * u;
}

// Rows [0, rows0) of the launch come from matrix 0 (the kernel's codes0 /
// scales0 / out), [rows0, rows0 + rows1) from matrix 1, the rest from
// matrix 2; each writes its own output [P][rows].  n <= 1: one matrix.
struct GemmSegs {
    uint32_t n, rows0, rows1;
    const uint32_t *codes1, *codes2;
    const uint16_t *scales1, *scales2;
    void *out1, *out2;
};

template <int MODE, int NMAT, int KQ, int WN>
__global__ __launch_bounds__(64 * WN * KQ) void dq_gemm_kernel(const f16_t *A, const uint32_t *codes0,
                                                      const uint16_t *scales0,
                                                      const uint32_t *codes1,
                                                      const uint16_t *scales1, void *out,
                                                      uint32_t P, uint32_t M, uint32_t K,
                                                      uint32_t gs_log2, GemmSegs sg) {
    // Two A stages (64 rows x 256 k of f16 each); reused for the k-phase
    // reduction after the main loop.
    constexpr int SK = ::SK<KQ>, PIECES = ::PIECES<KQ>, WROW = ::WROW<KQ>;
    // WN W-row groups x KQ k-phases of waves; a wave's tile is 64 x (64 / WN)
    constexpr int THREADS = 64 * WN * KQ, NJ = 4 / WN, A_LOADS = BM * PIECES / THREADS;
    static_assert(BM * PIECES == A_LOADS * THREADS && 64 * KQ * NMAT <= THREADS, "loader shapes");
    static_assert(PIECES >= 16, "the swizzle p ^ (r & 15) needs 16 pieces per row (KQ >= 2)");
    __shared__ __attribute__((aligned(16))) f16_t As[2][BM * SK];
    // W per stage: for each matrix and row, one 16-byte entry per k-step
    // (code words of its 64 k, scale), rows padded to WROW entries so the 16
    // rows of a fragment read hit distinct banks.
    __shared__ u32x4 Ws[2][NMAT][BN * WROW];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN, kq = wave / WN;

    // Block -> (W tile x, token tile y).  Workgroups are dispatched to the 8
    // XCDs round-robin, so block L runs on XCD L % 8; with the token tiles a
    // multiple of 8, XCD j gets token tiles j, j + 8, ... and all W tiles.
    const uint32_t nx = M / BN, ny = ceil_div(P, BM), L = blockIdx.x;
    uint32_t bx, by;
    if ((ny & 7) == 0) {
        const uint32_t slot = L >> 3;
        by = 8 * (slot / nx) + (L & 7);
        bx = slot % nx;
    } else {
        bx = L % nx;
        by = L / nx;
    }
    const uint32_t p0 = by * BM;
    uint32_t n0 = bx * BN;
    if (sg.n > 1) {   // row segments of up to three matrices, each with its own output
        if (n0 < sg.rows0) {
            M = sg.rows0;
        } else if (n0 < sg.rows0 + sg.rows1 || sg.n == 2) {
            n0 -= sg.rows0;
            codes0 = sg.codes1;
            scales0 = sg.scales1;
            out = sg.out1;
            M = sg.rows1;
        } else {
            n0 -= sg.rows0 + sg.rows1;
            codes0 = sg.codes2;
            scales0 = sg.scales2;
            out = sg.out2;
            M = M - sg.rows0 - sg.rows1;
        }
    }
    const uint32_t words_per_row = K / 32, groups_per_row = K >> gs_log2;
    const uint32_t nk = K / BK, nst = ceil_div(nk, (uint32_t)KQ);

    float4v acc[NMAT][4][NJ];
#pragma unroll
    for (int m = 0; m < NMAT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[m][i][j] = (float4v){0.f, 0.f, 0.f, 0.f};

    // A loader: straight into LDS (global_load_lds_dwordx4: the 64 lanes of
    // a wave instruction fill 64 consecutive 16-byte slots, no registers).
    // Thread tid fills slot lp of rows lr + 16 u, u < A_LOADS, which holds
    // piece lp ^ (r & 15) = lp ^ (lr & 15) of the row, so that is the piece
    // it loads (rows past P re-read row P - 1, discarded at the store;
    // k-steps past the end re-read the last one, never used).
    const int lp = tid & (PIECES - 1), lr = tid / PIECES;
    constexpr int A_ROW_STEP = THREADS / PIECES;   // rows between a thread's pieces
    static_assert(A_ROW_STEP % 16 == 0, "a thread's rows share r & 15");
    const int ap = lp ^ (lr & 15);                 // the piece this thread loads
    const f16_t *arow[A_LOADS];
#pragma unroll
    for (int u = 0; u < A_LOADS; ++u)
        arow[u] = A + (size_t)min(p0 + (uint32_t)(lr + A_ROW_STEP * u), P - 1) * K + (ap & 7) * 8;
    // W loader: thread t < 256 NMAT loads k-step t % 4 of the stage for row
    // (t / 4) % 64 of matrix t / 256: the step's two code words and its scale.
    const int wl_m = tid / (64 * KQ), wl_row = (tid / KQ) & 63, wl_q = tid % KQ;
    const bool wl = wl_m < NMAT;
    const uint32_t *wl_codes = (NMAT == 2 && wl_m == 1 ? codes1 : codes0) +
                               (size_t)(n0 + wl_row) * words_per_row;
    const uint16_t *wl_scales = (NMAT == 2 && wl_m == 1 ? scales1 : scales0) +
                                (size_t)(n0 + wl_row) * groups_per_row;
    const int bsh = 8 * (lane >> 4);   // the lane's byte within a 32-k word

    // One stage in flight: the A pieces land in the other LDS buffer and this
    // thread's W entry in registers (loaded first, so waiting for it leaves
    // the A loads in flight), stored to LDS at the stage's end.
    u32x2 wreg = {0u, 0u};
    uint32_t sreg = 0;
    const int wbase = wave * 64;   // the wave's first 16-byte slot of an instruction
    auto issue = [&](uint32_t st) __attribute__((always_inline)) {
        if (wl) {
            const uint32_t ks = min(st * KQ + (uint32_t)wl_q, nk - 1);
            wreg = *(const u32x2 *)(wl_codes + 2 * ks);
            sreg = wl_scales[(ks * BK) >> gs_log2];
        }
        const uint32_t ka = min(st * KQ + (uint32_t)(ap >> 3), nk - 1) * BK;
        const uint32_t lds = __builtin_amdgcn_readfirstlane(
            (uint32_t)(size_t)(__attribute__((address_space(3))) f16_t *)(As[st & 1] + 8 * wbase));
#pragma unroll
        for (int u = 0; u < A_LOADS; ++u) global_load_lds16(arow[u] + ka, lds + 16u * (uint32_t)(u * THREADS));
    };
    auto stage = [&](uint32_t st) __attribute__((always_inline)) {
        if (wl) Ws[st & 1][wl_m][wl_row * WROW + wl_q] = (u32x4){wreg[0], wreg[1], sreg, 0u};
    };
    auto compute = [&](uint32_t st) __attribute__((always_inline)) {
        if (st * KQ + kq >= nk) return;   // wave-uniform
        const f16_t *buf = As[st & 1];
        uint32_t w[NMAT][NJ][2], ns2[NMAT][NJ];
#pragma unroll
        for (int m = 0; m < NMAT; ++m)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const u32x4 e = Ws[st & 1][m][(16 * NJ * wn + 16 * j + (lane & 15)) * WROW + kq];
                w[m][j][0] = e[0];
                w[m][j][1] = e[1];
                ns2[m][j] = (e[2] | (e[2] << 16)) ^ 0x80008000u;
            }
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int piece = kq * 8 + kk * 4 + (lane >> 4);
            half8 af[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = i * 16 + (lane & 15);
                af[i] = *(const half8 *)(buf + r * SK + 8 * (piece ^ (r & 15)));
            }
#pragma unroll
            for (int m = 0; m < NMAT; ++m)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const half8 bf = expand_bits((w[m][j][kk] >> bsh) & 0xFFu, ns2[m][j]);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc[m][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bf, acc[m][i][j], 0, 0, 0);
                }
        }
    };

    // Stage pipeline: stage st + 1's loads are issued before stage st is
    // computed and stored to the other LDS buffers after it (those were last
    // read in stage st - 1, before the previous barrier).
    issue(0);
    stage(0);
    load_barrier();
    for (uint32_t st = 0; st < nst; ++st) {
        if (st + 1 < nst) issue(st + 1);   // block-uniform
        compute(st);
        if (st + 1 < nst) stage(st + 1);
        load_barrier();
    }

    // k-phase reduction through LDS (the stage buffers are free): phases 2, 3
    // hand their tiles to 0, 1, then phase 1 to phase 0.  Slot layout: one
    // float4 per (fragment, lane), lanes adjacent.
    constexpr int NF = NMAT * 4 * NJ;
    float4v *red = (float4v *)&As[0][0];
    auto put = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < NMAT; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) red[(slot * NF + (m * 4 + i) * NJ + j) * 64 + lane] = acc[m][i][j];
    };
    auto add = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < NMAT; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[m][i][j] += red[(slot * NF + (m * 4 + i) * NJ + j) * 64 + lane];
    };
    static_assert(KQ / 2 * WN * NF * 64 * 16 <= (int)sizeof(As), "reduction slots fit the stage buffers");
    // tree over the k-phases: phases [h, 2h) hand their tiles to [0, h),
    // down to phases 0 and 1
#pragma unroll
    for (int h = KQ / 2; h >= 2; h /= 2) {
        if (kq >= h && kq < 2 * h) put((kq - h) * WN + wn);
        __syncthreads();
        if (kq < h) add(kq * WN + wn);
        __syncthreads();
    }
    // Phases 0 and 1 swap halves and both finish the block: phase 0 the
    // 16-row tiles i = 0, 1, phase 1 the tiles i = 2, 3.  (With phase 0
    // finishing everything, the waves of phase 0 -- the same SIMDs in every
    // block -- carried the whole epilogue.)  Half slots: NF / 2 float4.
    auto put_half = [&](int slot, auto hh) __attribute__((always_inline)) {
        constexpr int H = decltype(hh)::value;
#pragma unroll
        for (int m = 0; m < NMAT; ++m)
#pragma unroll
            for (int ii = 0; ii < 2; ++ii)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    red[(slot * (NF / 2) + (m * 2 + ii) * NJ + j) * 64 + lane] = acc[m][2 * H + ii][j];
    };
    auto add_half = [&](int slot, auto hh) __attribute__((always_inline)) {
        constexpr int H = decltype(hh)::value;
#pragma unroll
        for (int m = 0; m < NMAT; ++m)
#pragma unroll
            for (int ii = 0; ii < 2; ++ii)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    acc[m][2 * H + ii][j] += red[(slot * (NF / 2) + (m * 2 + ii) * NJ + j) * 64 + lane];
    };
    if (kq == 0) put_half(WN + wn, IC<1>{});   // phase 1's tiles
    else if (kq == 1) put_half(wn, IC<0>{});  // phase 0's tiles
    __syncthreads();
    if (kq >= 2) return;   // after the last barrier
    if (kq == 0) add_half(wn, IC<0>{});
    else add_half(WN + wn, IC<1>{});

    // D layout: lane holds rows 4*(lane/16)+r, column lane%16 of each 16x16 tile.
    auto epilogue = [&](auto ti) __attribute__((always_inline)) {
        constexpr int i = decltype(ti)::value;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t p = p0 + i * 16 + 4 * (lane >> 4) + r;
            if (p >= P) continue;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const uint32_t n = n0 + 16 * NJ * wn + 16 * j + (lane & 15);
                const size_t o = (size_t)p * M + n;
                const float c = acc[0][i][j][r];
                if constexpr (MODE == NNZ_GEMM_STORE_F16) ((f16_t *)out)[o] = (f16_t)c;
                else if constexpr (MODE == NNZ_GEMM_STORE_F32) ((float *)out)[o] = c;
                else if constexpr (MODE == NNZ_GEMM_RESADD) ((float *)out)[o] += c;
                else {
                    const float u = acc[NMAT - 1][i][j][r];
                    ((f16_t *)out)[o] = (f16_t)silu_mul(c, u);
                }
            }
        }
    };
    if (kq == 0) {
        epilogue(IC<0>{});
        epilogue(IC<1>{});
    } else {
        epilogue(IC<2>{});
        epilogue(IC<3>{});
    }
}

// ---------------------------------------------------------------------------
// 4-bit (q4_mlx) weights: W = s * n + b per group of >= 64 columns, n a
// nibble, s and b bf16 (or f16).  s * n + b is not exact in f16, so the
// MFMA takes the nibbles themselves, exactly: per 64-k step and W row,
//   sum_k A[p][k] W[r][k] = s_r * (A . n)[p][r] + b_r * (sum_k A[p][k]),
// with (A . n) and the row sums (A against a fragment of ones) on the MFMA
// and the two scalings in fp32 -- the Q4 QMV's arithmetic up to fp32
// summation order.  Nibble pairs become f16 through the exponent trick:
// 0x6400 | n is the f16 value 1024 + n, and subtracting 1024 (v_pk_add_f16)
// leaves n exactly.  Epilogues are the BF16-faithful ones of the Q4 decode
// kernels (q4mv_bf16_specialized.metal:52-57): each result is BF16-truncated
// before the f16 store, the residual += or the SiLU*mul product's store.
// Block: 64 tokens x 64 W rows, 4 waves = 2 W-row halves x 2 k-phases;
// an LDS stage holds 2 k-steps: A (swizzled as above) and, per matrix and
// row, the 16 code words of the two steps plus their (s | b << 16) words,
// rows padded to 20 words so a fragment read of 16 rows hits distinct banks.
// KQ k-phases: 4 KQ waves (2 W-row halves x KQ), LDS stages of KQ k-steps;
// a W row holds 8 code words per step plus one (s | b << 16) word per step,
// padded to a stride of 4 x odd words (20 for KQ = 2, 36 for KQ = 4).
template <int KQ> constexpr int Q4_WROW = KQ == 2 ? 20 : 36;
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float q4_param(uint32_t raw16, int sdt) {
    return sdt == NNZ_BF16 ? bf16_to_f32((uint16_t)raw16) : (float)__builtin_bit_cast(f16_t, (uint16_t)raw16);
}

// The 8 nibbles of one code word (k ascending from bit 0) as f16 values.
__device__ __forceinline__ half8 expand_nibbles(uint32_t w) {
    const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;   // bytes: n[2q], n[2q+1]
    const half2v k1024 = {(_Float16)1024.f, (_Float16)1024.f};
    half8 r;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        // byte q of lo into byte 0, byte q of hi into byte 2, zeros elsewhere
        const uint32_t sel = (uint32_t)q | (0x0Cu << 8) | ((uint32_t)(4 + q) << 16) | (0x0Cu << 24);
        const uint32_t d = __builtin_amdgcn_perm(hi, lo, sel) | 0x64006400u;
        const half2v v = __builtin_bit_cast(half2v, d) - k1024;
        r[2 * q] = v[0];
        r[2 * q + 1] = v[1];
    }
    return r;
}

// At most 256 registers (two waves per SIMD): the pair kernel otherwise
// takes 222 VGPRs + 64 AGPRs, one wave per SIMD, and copies every MFMA
// result out of the AGPRs before its scaling.
template <int MODE, int NMAT, int KQ>
__global__ __launch_bounds__(128 * KQ) __attribute__((amdgpu_waves_per_eu(2))) void dq4_gemm_kernel(const f16_t *A, const uint32_t *codes0,
                                                              const uint16_t *scales0,
                                                              const uint16_t *biases0,
                                                              const uint32_t *codes1,
                                                              const uint16_t *scales1,
                                                              const uint16_t *biases1, void *out,
                                                              uint32_t P, uint32_t M, uint32_t K,
                                                              uint32_t gs_log2, int sdt) {
    constexpr int Q4_KQ = KQ, Q4_SK = BK * KQ, Q4_PIECES = Q4_SK / 8, Q4_THREADS = 128 * KQ;
    constexpr int WR = Q4_WROW<KQ>;
    constexpr int A_LOADS = BM * Q4_PIECES / Q4_THREADS;   // 4
    static_assert(Q4_PIECES >= 16 && 64 * Q4_KQ * NMAT <= Q4_THREADS && WR >= 9 * KQ, "loader shapes");
    __shared__ __attribute__((aligned(16))) f16_t As[2][BM * Q4_SK];
    __shared__ __attribute__((aligned(16))) uint32_t Ws[2][NMAT][BN * WR];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 1, kq = wave >> 1;
    const uint32_t nx = M / BN, ny = ceil_div(P, BM), L = blockIdx.x;
    uint32_t bx, by;
    if ((ny & 7) == 0) {
        const uint32_t slot = L >> 3;
        by = 8 * (slot / nx) + (L & 7);
        bx = slot % nx;
    } else {
        bx = L % nx;
        by = L / nx;
    }
    const uint32_t p0 = by * BM, n0 = bx * BN;
    const uint32_t words_per_row = K / 8, groups_per_row = K >> gs_log2;
    const uint32_t nk = K / BK, nst = ceil_div(nk, (uint32_t)Q4_KQ);

    float4v acc[NMAT][4][2];
#pragma unroll
    for (int m = 0; m < NMAT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[m][i][j] = (float4v){0.f, 0.f, 0.f, 0.f};

    // A through registers (loading it straight into LDS, as dq_gemm_kernel
    // does, measured no faster here: 4-bit down 37.7 -> 38.6 us)
    const int lp = tid & (Q4_PIECES - 1), lr = tid / Q4_PIECES;
    constexpr int A_ROW_STEP = Q4_THREADS / Q4_PIECES;
    const f16_t *arow[A_LOADS];
#pragma unroll
    for (int u = 0; u < A_LOADS; ++u)
        arow[u] = A + (size_t)min(p0 + (uint32_t)(lr + A_ROW_STEP * u), P - 1) * K + (lp & 7) * 8;
    // W loader: thread t < 64 KQ NMAT takes step t % KQ of row (t / KQ) % 64
    // of matrix t / (64 KQ): 8 code words (two 16-byte loads), scale and bias.
    const int wl_m = tid / (64 * KQ), wl_row = (tid / KQ) & 63, wl_q = tid % KQ;
    const bool wl = wl_m < NMAT;
    const uint32_t wrow_g = n0 + wl_row;
    const uint32_t *wl_codes = (NMAT == 2 && wl_m == 1 ? codes1 : codes0) + (size_t)wrow_g * words_per_row;
    const uint16_t *wl_s = (NMAT == 2 && wl_m == 1 ? scales1 : scales0) + (size_t)wrow_g * groups_per_row;
    const uint16_t *wl_b = (NMAT == 2 && wl_m == 1 ? biases1 : biases0) + (size_t)wrow_g * groups_per_row;
    const int gsel = lane >> 4;   // the lane's code word within a 32-k half step

    // scale and bias stay two registers until the stage: joining them at
    // the issue would wait there for their loads, and with them (vmcnt is
    // in order) for the A loads of the stage being prefetched
    u32x4 areg[A_LOADS], wc0 = {0u, 0u, 0u, 0u}, wc1 = {0u, 0u, 0u, 0u};
    uint32_t sreg = 0, breg = 0;
    auto issue = [&](uint32_t st) __attribute__((always_inline)) {
        const uint32_t ka = min(st * Q4_KQ + (uint32_t)(lp >> 3), nk - 1) * BK;
#pragma unroll
        for (int u = 0; u < A_LOADS; ++u) areg[u] = *(const u32x4 *)(arow[u] + ka);
        if (wl) {
            const uint32_t ks = min(st * Q4_KQ + (uint32_t)wl_q, nk - 1);
            wc0 = *(const u32x4 *)(wl_codes + 8 * ks);
            wc1 = *(const u32x4 *)(wl_codes + 8 * ks + 4);
            const uint32_t g = (ks * BK) >> gs_log2;
            sreg = wl_s[g];
            breg = wl_b[g];
        }
    };
    auto stage = [&](uint32_t st) __attribute__((always_inline)) {
        f16_t *buf = As[st & 1];
#pragma unroll
        for (int u = 0; u < A_LOADS; ++u) {
            const int r = lr + A_ROW_STEP * u;
            ((u32x4 *)(buf + r * Q4_SK))[lp ^ (r & 15)] = areg[u];
        }
        if (wl) {
            uint32_t *row = Ws[st & 1][wl_m] + wl_row * WR;
            *(u32x4 *)(row + 8 * wl_q) = wc0;
            *(u32x4 *)(row + 8 * wl_q + 4) = wc1;
            row[8 * KQ + wl_q] = sreg | (breg << 16);
        }
    };
    const half8 ones = {(_Float16)1.f, (_Float16)1.f, (_Float16)1.f, (_Float16)1.f,
                        (_Float16)1.f, (_Float16)1.f, (_Float16)1.f, (_Float16)1.f};
    auto compute = [&](uint32_t st) __attribute__((always_inline)) {
        if (st * Q4_KQ + kq >= nk) return;   // wave-uniform
        const f16_t *buf = As[st & 1];
        half8 af[2][4];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int piece = kq * 8 + kk * 4 + (lane >> 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = i * 16 + (lane & 15);
                af[kk][i] = *(const half8 *)(buf + r * Q4_SK + 8 * (piece ^ (r & 15)));
            }
        }
        // row sums of A over the step: every column of the product with ones
        float4v xs[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            xs[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[0][i], ones, (float4v){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            xs[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[1][i], ones, xs[i], 0, 0, 0);
        }
#pragma unroll
        for (int m = 0; m < NMAT; ++m)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t *row = Ws[st & 1][m] + (32 * wn + 16 * j + (lane & 15)) * WR;
                const uint32_t sb = row[8 * KQ + kq];
                const float sc = q4_param(sb & 0xFFFFu, sdt), bi = q4_param(sb >> 16, sdt);
                const half8 b0 = expand_nibbles(row[8 * kq + gsel]);
                const half8 b1 = expand_nibbles(row[8 * kq + 4 + gsel]);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float4v t = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[0][i], b0, (float4v){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    t = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[1][i], b1, t, 0, 0, 0);
                    // two multiply-adds per element: + b (row sum), then + s (A . n)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[m][i][j][r] = fmaf(sc, t[r], fmaf(bi, xs[i][r], acc[m][i][j][r]));
                }
            }
    };

    issue(0);
    stage(0);
    step_barrier();
    for (uint32_t st = 0; st < nst; ++st) {
        if (st + 1 < nst) issue(st + 1);   // block-uniform
        compute(st);
        if (st + 1 < nst) stage(st + 1);
        step_barrier();
    }

    // k-phase tree through the (free) A buffers: phases [h, 2h) hand their
    // tiles to [0, h), down to phases 0 and 1
    constexpr int NF = NMAT * 8;
    static_assert(KQ / 2 * 2 * NF * 64 * 16 <= (int)sizeof(As), "reduction slots fit the stage buffers");
    float4v *red = (float4v *)&As[0][0];
#pragma unroll
    for (int h = KQ / 2; h >= 2; h /= 2) {
        if (kq >= h && kq < 2 * h) {
#pragma unroll
            for (int m = 0; m < NMAT; ++m)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        red[(((kq - h) * 2 + wn) * NF + (m * 4 + i) * 2 + j) * 64 + lane] = acc[m][i][j];
        }
        __syncthreads();
        if (kq < h) {
#pragma unroll
            for (int m = 0; m < NMAT; ++m)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[m][i][j] += red[((kq * 2 + wn) * NF + (m * 4 + i) * 2 + j) * 64 + lane];
        }
        __syncthreads();
    }
    // Phases 0 and 1 swap halves and both finish the block: phase 0 the
    // 16-row tiles i = 0, 1, phase 1 the tiles i = 2, 3 (half slots of
    // NF / 2 float4).
    auto put_half = [&](int slot, auto hh) __attribute__((always_inline)) {
        constexpr int H = decltype(hh)::value;
#pragma unroll
        for (int m = 0; m < NMAT; ++m)
#pragma unroll
            for (int ii = 0; ii < 2; ++ii)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    red[(slot * (NF / 2) + (m * 2 + ii) * 2 + j) * 64 + lane] = acc[m][2 * H + ii][j];
    };
    auto add_half = [&](int slot, auto hh) __attribute__((always_inline)) {
        constexpr int H = decltype(hh)::value;
#pragma unroll
        for (int m = 0; m < NMAT; ++m)
#pragma unroll
            for (int ii = 0; ii < 2; ++ii)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[m][2 * H + ii][j] += red[(slot * (NF / 2) + (m * 2 + ii) * 2 + j) * 64 + lane];
    };
    if (kq == 0) put_half(2 + wn, IC<1>{});   // phase 1's tiles
    else if (kq == 1) put_half(wn, IC<0>{});  // phase 0's tiles
    __syncthreads();
    if (kq >= 2) return;   // after the last barrier
    if (kq == 0) add_half(wn, IC<0>{});
    else add_half(2 + wn, IC<1>{});

    auto epilogue = [&](auto ti) __attribute__((always_inline)) {
        constexpr int i = decltype(ti)::value;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t p = p0 + i * 16 + 4 * (lane >> 4) + r;
            if (p >= P) continue;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t n = n0 + 32 * wn + 16 * j + (lane & 15);
                const size_t o = (size_t)p * M + n;
                const float c = acc[0][i][j][r];
                if constexpr (MODE == NNZ_GEMM_STORE_F16) ((f16_t *)out)[o] = (f16_t)bf16_trunc(c);
                else if constexpr (MODE == NNZ_GEMM_STORE_F32) ((float *)out)[o] = bf16_trunc(c);
                else if constexpr (MODE == NNZ_GEMM_RESADD) ((float *)out)[o] += bf16_trunc(c);
                else {
                    const float u = acc[NMAT - 1][i][j][r];
                    ((f16_t *)out)[o] = (f16_t)bf16_trunc(silu_mul(c, u));
                }
            }
        }
    };
    if (kq == 0) {
        epilogue(IC<0>{});
        epilogue(IC<1>{});
    } else {
        epilogue(IC<2>{});
        epilogue(IC<3>{});
    }
}

// ---------------------------------------------------------------------------
// The main GEMM kernel: 1-bit weights of group size 128 and 4-bit weights of
// group size 64 with bf16 scales, K a multiple of 512, 16-byte aligned codes.
//
// Block: 64 tokens x NSUB sub-blocks of 64 W rows (a gate/up pair: one of each
// matrix; a single matrix with NSUB = 2: 128 consecutive rows), 2 KQ waves =
// 2 row halves x KQ k-phases.  An LDS stage is KQ steps of 64 k; wave (wn, kq)
// takes step kq of every stage for 32 rows of each sub-block.
//
// dq_gemm_kernel and dq4_gemm_kernel above fetch W and its scales 8 and 2
// bytes per row and step, a 128-byte line each time; with their compute taken
// out they still took two thirds of their time.  Here everything is loaded
// straight into LDS (no registers, no LDS stores) in pieces that use the lines
// they touch: A 128 bytes per row and step, W codes 64 bytes per row (a chunk:
// 512 k of 1-bit, 128 k of 4-bit codes), scales a dword.  A 4-bit weight is
// dequantised exactly into its f16 operand (expand_nibbles_scaled; waves with a
// row whose scales don't allow that take a loop of their own), so its
// accumulators run through K unscaled and only the bias products remain on
// the VALU.  Measured before -> now, weights rotated: 1-bit gate/up 2 x 6144 x
// 2048 at P = 512 33.8 -> 30.5 us (845 TFLOP/s), 2 x 9728 x 2560 at P = 3001
// 295 -> 268 (1113 TFLOP/s; the library's bf16 GEMM of that size without any
// dequantisation 1161); 2560 x 9728 at P = 3001 190 -> 144, 2560 x 4096 82 ->
// 63, 6144 x 2560 120 -> 86; 4-bit gate/up 2 x 6144 x 2048 at P = 512 59.7 ->
// 47, 2 x 9728 x 2560 at P = 1500 290 -> 230.  Bounds now: 1-bit, one round of
// blocks at P = 512 (first loads and epilogue overlap nothing), at large P the
// L2-to-LDS rate of A (8.7 TB/s over the chip) and MFMA issue; 4-bit, VALU
// issue (188 per 40 MFMAs).  Three or four LDS stages in flight instead of
// two: no faster (2048 x 6144, P = 512: 22.4-22.6 us against 21.7).
//
// MFMA k-slot order: lane group q = lane / 16 of the two MFMAs u = 0, 1 of a
// step takes k = 16 q + 8 u .. + 8 of the step (any assignment is right as long
// as A and B agree), so a lane's weights of a step are one aligned piece: 16
// bits (1-bit) or 8 bytes (4-bit).
// Straight-to-LDS loads from a wave-uniform base plus a 32-bit lane offset.
// s_nop 4: gfx9 wants five wait states between a VALU write of an SGPR and a
// memory instruction reading it (the compiler's hazard check does not look
// into asm, and the base may come from a v_readfirstlane).
__device__ __forceinline__ void load_lds_b128(const void *sbase, uint32_t voff, uint32_t lds) {
    asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "{m0}"(lds) : "memory");
}
__device__ __forceinline__ void load_lds_b32(const void *sbase, uint32_t voff, uint32_t lds) {
    asm volatile("s_nop 4\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(sbase), "{m0}"(lds) : "memory");
}
// A wave-uniform pointer as an opaque scalar value: selecting between argument
// fields through it keeps the compiler from selecting between their addresses,
// which would copy the argument block to scratch memory.
template <class T>
__device__ __forceinline__ T *uniform_ptr(T *p) {
    // readfirstlane returns int: through uint32_t, or the low half sign-extends
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (T *)((uint64_t)hi << 32 | lo);
}
// Low half of a lane value times a uniform one, in one register: the compiler's
// multiply-add has a 64-bit result, whose other half would live as long.
__device__ __forceinline__ uint32_t mul_lo(uint32_t v, uint32_t s) {
    uint32_t r;
    asm("v_mul_lo_u32 %0, %1, %2" : "=v"(r) : "v"(v), "s"(s));
    return r;
}
template <class T>
__device__ __forceinline__ uint32_t lds_addr(T *p) {
    return (uint32_t)(size_t)(__attribute__((address_space(3))) T *)p;
}

// 16 weight bits -> the two B fragments' f16 values, +s where the bit is set
// and -s where it is clear.  y carries the bits twice, 15 apart, so that bits
// 2e and 2e + 1 sit 16 apart and one shift brings them to the sign positions.
__device__ __forceinline__ void expand_bits16(uint32_t h, uint32_t ns2, half8 &f0, half8 &f1) {
    uint32_t y;
    asm("v_lshl_or_b32 %0, %1, 15, %1" : "=v"(y) : "v"(h));
    u32x4 e, f;
    e[0] = ((y << 15) & 0x80008000u) ^ ns2;
    e[1] = ((y << 13) & 0x80008000u) ^ ns2;
    e[2] = ((y << 11) & 0x80008000u) ^ ns2;
    e[3] = ((y << 9) & 0x80008000u) ^ ns2;
    f[0] = ((y << 7) & 0x80008000u) ^ ns2;
    f[1] = ((y << 5) & 0x80008000u) ^ ns2;
    f[2] = ((y << 3) & 0x80008000u) ^ ns2;
    f[3] = ((y << 1) & 0x80008000u) ^ ns2;
    f0 = __builtin_bit_cast(half8, e);
    f1 = __builtin_bit_cast(half8, f);
}

// 8 nibbles -> S (n - 8) 2^-20, exact where it is an f16: the nibble in bits 4..7 of a half is
// the (denormal) f16 value n 2^-20, and one fused multiply-add with S and
// c = -8 S 2^-20 scales and centres it.  A bf16 scale has 8 significant bits
// and |n - 8| <= 8 three more, or is a power of two: 11 bits, an f16 down to
// S = 2^3 (below, the last bits fall under the smallest f16).
constexpr int ROW_WIDE = 0x40000000;
__device__ __forceinline__ half8 expand_nibbles_scaled(uint32_t w, half2v S, half2v c) {
    const uint32_t lo = (w << 4) & 0xF0F0F0F0u, hi = w & 0xF0F0F0F0u;   // n[2j], n[2j+1] in byte j
    half8 r;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t sel = (uint32_t)j | (0x0Cu << 8) | ((uint32_t)(4 + j) << 16) | (0x0Cu << 24);
        const half2v v = __builtin_elementwise_fma(__builtin_bit_cast(half2v, __builtin_amdgcn_perm(hi, lo, sel)), S, c);
        r[2 * j] = v[0];
        r[2 * j + 1] = v[1];
    }
    return r;
}

struct GemmMat {
    const void *codes;
    const uint16_t *scales, *biases;   // biases: 4-bit only
    void *out;
    uint32_t rows;
};
// m[0..n): row segments of one launch (Q, K, V), each with its own output; a
// gate/up pair: m[0] and m[1], one output.
struct GemmArgs {
    const f16_t *A;
    GemmMat m0, m1, m2;
    uint32_t n, P, K, nx;   // nx: W tiles of the launch
    float *part;            // split-K: partial sums [splits][P][cols], cols = the launch's rows
    uint32_t splits, cols;
};

// LDS of a block, and the blocks that the shape rules below count on per CU.
template <int BITS, int NSUB, int KQ>
constexpr size_t qgemm_lds() {
    constexpr int cpb = KQ > (BITS == 1 ? 8 : 2) ? KQ / (BITS == 1 ? 8 : 2) : 1;
    return 2 * (size_t)(BM * BK * KQ) * 2 + 2 * (size_t)cpb * (64 * NSUB) * (64 + 8) + (BITS == 4 ? 4 * 64 * NSUB : 4);
}
constexpr size_t LDS_CU = 160 * 1024;
static_assert(qgemm_lds<1, 1, 8>() <= LDS_CU && 2 * qgemm_lds<1, 1, 4>() <= LDS_CU && 3 * qgemm_lds<1, 2, 2>() <= LDS_CU &&
              qgemm_lds<4, 2, 4>() <= LDS_CU && 2 * qgemm_lds<4, 1, 4>() > LDS_CU && 3 * qgemm_lds<4, 2, 2>() <= LDS_CU,
              "blocks per CU");

template <int BITS, int MODE, int NSUB, int KQ, bool SPLIT>
__global__ __launch_bounds__(128 * KQ) __attribute__((amdgpu_waves_per_eu(3))) void qgemm_kernel(GemmArgs ga) {
    constexpr bool PAIR = MODE == NNZ_GEMM_SILU_PAIR;
    static_assert(!PAIR || (NSUB == 2 && !SPLIT), "a pair has two sub-blocks, and is not split");
    constexpr int SK = BK * KQ, PIECES = SK / 8, THREADS = 128 * KQ, A_LOADS = 4, ROWS = 64 * NSUB;
    constexpr int CSTEPS = BITS == 1 ? 8 : 2;                    // 64-k steps per W chunk
    constexpr int CPS = KQ > CSTEPS ? KQ / CSTEPS : 1;           // chunks per buffer
    constexpr int SPC = CSTEPS > KQ ? CSTEPS / KQ : 1;           // stages per buffer
    constexpr bool TWO = BITS == 1 && KQ == 2 && !PAIR;          // two accumulator sets
    constexpr int W_INSTR = 4 * NSUB * CPS, S_INSTR = 2 * NSUB * CPS, WAVES = 2 * KQ;
    __shared__ __attribute__((aligned(16))) f16_t As[2][BM * SK];
    __shared__ __attribute__((aligned(16))) uint32_t Wc[2][CPS][ROWS * 16];
    __shared__ uint32_t Sc[2][CPS][ROWS * 2];
    __shared__ int rowexp[BITS == 4 ? ROWS : 1];
    static_assert(sizeof(As) + sizeof(Wc) + sizeof(Sc) + sizeof(rowexp) == qgemm_lds<BITS, NSUB, KQ>(), "the shape rules' LDS");

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 1, kq = wave >> 1;
    const int q = lane >> 4, r16 = lane & 15;

    // Workgroups go round-robin over the 8 XCDs: XCD j takes the j-th eighth
    // of the tiles, W tile fastest, so its L2 holds the few token tiles it
    // works on and no other XCD reads them.
    const uint32_t ny = ceil_div(ga.P, (uint32_t)BM), nb = ga.nx * ny;
    uint32_t idx = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    uint32_t sp = 0, kb = 0, ke = ga.K;   // the block's k range: whole 512-k pieces
    if constexpr (SPLIT) {
        if (idx >= nb * ga.splits) return;
        sp = idx / nb;
        idx -= sp * nb;
        kb = ga.K / 512 * sp / ga.splits * 512;
        ke = ga.K / 512 * (sp + 1) / ga.splits * 512;
    } else {
        if (idx >= nb) return;
    }
    const uint32_t by = idx / ga.nx, bx = idx % ga.nx, p0 = by * BM;
    const uint32_t K = ga.K, G = K / (BITS == 1 ? 128 : 64), rowbytes = K / 8 * BITS;
    uint32_t n0 = bx * (PAIR ? 64u : (uint32_t)ROWS);
    int seg = 0;
    if (!PAIR && ga.n > 1) {
        if (n0 >= ga.m0.rows) {
            n0 -= ga.m0.rows;
            seg = 1;
            if (ga.n > 2 && n0 >= ga.m1.rows) {
                n0 -= ga.m1.rows;
                seg = 2;
            }
        }
    }
    auto pick = [&](auto f) __attribute__((always_inline)) {
        auto *const v0 = uniform_ptr(f(ga.m0)), *const v1 = uniform_ptr(f(ga.m1)), *const v2 = uniform_ptr(f(ga.m2));
        return seg == 0 ? v0 : (seg == 1 ? v1 : v2);
    };
    const void *const codes = pick([](const GemmMat &m) { return m.codes; });
    const uint16_t *const scales = pick([](const GemmMat &m) { return m.scales; });
    const uint16_t *const biases = pick([](const GemmMat &m) { return m.biases; });
    void *const out = pick([](const GemmMat &m) { return m.out; });
    const uint32_t r0 = ga.m0.rows, r1 = ga.m1.rows, r2 = ga.m2.rows, out_rows = seg == 0 ? r0 : (seg == 1 ? r1 : r2);
    const size_t wat = (size_t)n0 * rowbytes + kb / 8 * BITS, sat = (size_t)n0 * G + kb / (BITS == 1 ? 128 : 64);
    const char *const wbase0 = (const char *)codes + wat;
    const char *const wbase1 = PAIR ? (const char *)ga.m1.codes + wat : wbase0 + (size_t)64 * rowbytes;
    const uint16_t *const sbase0 = scales + sat;
    const uint16_t *const sbase1 = PAIR ? ga.m1.scales + sat : sbase0 + (size_t)64 * G;
    const uint16_t *const bbase0 = BITS == 4 ? biases + sat : nullptr;
    const uint16_t *const bbase1 = BITS == 4 ? (PAIR ? ga.m1.biases + sat : bbase0 + (size_t)64 * G) : nullptr;

    // A: lane's slot lp of rows lr + 16 u holds piece lp ^ (row & 15), so the
    // 16 rows of a fragment read hit distinct banks; rows past P re-read row
    // P - 1, their results are not stored.
    const int lp = tid & (PIECES - 1), lr = tid / PIECES;
    uint32_t avoff[A_LOADS];
#pragma unroll
    for (int u = 0; u < A_LOADS; ++u)
        avoff[u] = mul_lo(min(p0 + (uint32_t)(lr + 16 * u), ga.P - 1) - p0, K * 2u) + (uint32_t)(lp ^ (lr & 15)) * 16u;
    const char *const abase = (const char *)(ga.A + (size_t)p0 * K + kb);
    // W chunk: 64 bytes per row as 4 pieces, piece p of row r at slot
    // p ^ ((r >> 2) & 3); instruction i fills rows 16 i .. 16 i + 15.
    auto issue_a = [&](uint32_t st) __attribute__((always_inline)) {
        const char *const sb = abase + (size_t)st * (SK * 2);
        const uint32_t l0 = __builtin_amdgcn_readfirstlane(lds_addr(As[st & 1] + 8 * (wave * 64)));
#pragma unroll
        for (int u = 0; u < A_LOADS; ++u) load_lds_b128(uniform_ptr(sb), avoff[u], l0 + 16u * (uint32_t)(u * THREADS));
    };
    // buffer b of W: chunks b CPS .. of every row
    // (with two accumulator sets on 128 rows, once in four stages, the lane's
    // number and offsets are computed here each time: three registers fewer in
    // the loop)
    auto issue_w = [&](uint32_t b) __attribute__((always_inline)) {
        uint32_t ln = (uint32_t)lane;
        if constexpr (TWO && NSUB == 2)
            asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
        const uint32_t wvoff = mul_lo(ln >> 2, rowbytes) + ((ln & 3u) ^ (ln >> 4)) * 16u;
        // scales: 2 dwords of a row (1-bit), or one
        const uint32_t svoff = BITS == 1 ? mul_lo(ln >> 1, G * 2u) + (ln & 1u) * 4u : mul_lo(ln, G * 2u);
#pragma unroll
        for (int i0 = 0; i0 < W_INSTR; i0 += WAVES) {
            const int i = i0 + wave;
            if (W_INSTR % WAVES == 0 || i < W_INSTR) {   // wave-uniform
                const int c = i / (4 * NSUB), j = i % (4 * NSUB);
                const char *const sb = (NSUB == 2 && j >= 4 ? wbase1 : wbase0) + (size_t)(j & 3) * 16 * rowbytes +
                                       (size_t)(b * CPS + c) * 64;
                load_lds_b128(uniform_ptr(sb), wvoff, __builtin_amdgcn_readfirstlane(lds_addr(&Wc[b & 1][c][j * 256])));
            }
        }
#pragma unroll
        for (int i0 = 0; i0 < S_INSTR; i0 += WAVES) {
            const int i = i0 + (WAVES - 1 - wave);       // the waves with less W first
            if (S_INSTR % WAVES == 0 || (i >= 0 && i < S_INSTR)) {
                const int c = i / (2 * NSUB), j = i % (2 * NSUB), sub = j >> 1, h = j & 1;
                const uint32_t l0 = __builtin_amdgcn_readfirstlane(lds_addr(&Sc[b & 1][c][sub * 128 + h * 64]));
                if constexpr (BITS == 1) {   // 4 scales of a row = 2 dwords: rows 32 h .. of the sub-block
                    const char *const sb = (const char *)(sub ? sbase1 : sbase0) + (size_t)(32 * h) * G * 2 + (size_t)(b * CPS + c) * 8;
                    load_lds_b32(uniform_ptr(sb), svoff, l0);
                } else {                     // 2 scales (h = 0) or biases (h = 1) of a row = 1 dword
                    const uint16_t *const s0 = uniform_ptr(sbase0), *const s1 = uniform_ptr(sbase1);
                    const uint16_t *const b0 = uniform_ptr(bbase0), *const b1 = uniform_ptr(bbase1);
                    const uint16_t *const t0 = h ? b0 : s0, *const t1 = h ? b1 : s1;
                    const char *const sb = (const char *)(sub ? t1 : t0) + (size_t)(b * CPS + c) * 4;
                    load_lds_b32(uniform_ptr(sb), svoff, l0);
                }
            }
        }
    };

    float4v acc[NSUB][4][2];
#pragma unroll
    for (int s = 0; s < NSUB; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[s][i][j] = (float4v){0.f, 0.f, 0.f, 0.f};
    // 1-bit launches on two k-phases (TWO) keep a second set, for the u = 1
    // MFMAs, so that a float32 chain is no longer than four k-phases make it: with one
    // set the result was 1.4 times as far from float64 (2048 x 6144, P = 1500:
    // 3.5e-7 against 2.5e-7).  Three 128-row blocks per CU leave a lane 168
    // registers, 128 of them these sums: the loop's addresses are held down to
    // that (with spills, or two blocks per CU, it is 1.1 to 1.8 times slower).
    float4v acc1[TWO ? NSUB : 1][4][2];
    if constexpr (TWO) {
#pragma unroll
        for (int t = 0; t < NSUB * 8; ++t) acc1[t / 8][(t / 2) % 4][t % 2] = (float4v){0.f, 0.f, 0.f, 0.f};
    }

    const uint32_t nst = (ke - kb) / SK;
    auto issue = [&](uint32_t st) __attribute__((always_inline)) {   // W before the A of its first stage
        if (st % SPC == 0) issue_w(st / SPC);
        issue_a(st);
    };
    issue(0);
    int ex[NSUB][2];
    bool wide = false;   // wave-uniform: the wave's weights don't fit f16 scaled
    if constexpr (BITS == 4) {
        // Row exponents: S = s 2^e with the row's largest |s| in [2^15, 2^16),
        // so that S (n - 8) 2^-20 is exact in f16 for scales down to 2^-12 of
        // the largest.  A row whose nonzero scales spread further, or whose
        // largest is outside 2^-21 .. 2^12 (where the scaled sums might leave
        // float32's range before the results do: within, that takes results
        // of 2^111), infinite or NaN is wide: its wave multiplies the nibbles
        // as they are and applies scales and biases in float32 per group.  The
        // row's threads scan its scales.
        constexpr int TPR = THREADS / ROWS;   // threads per row
        static_assert(TPR == 2 || TPR == 4 || TPR == 8, "a row's threads are lanes of one octet");
        const int row = tid / TPR, sub = row >> 6;
        const uint16_t *const s0 = uniform_ptr(sbase0), *const s1 = uniform_ptr(sbase1);
        const auto *const rs = (const __attribute__((address_space(1))) u32x4 *)((sub ? s1 : s0) + (size_t)(row & 63) * G);
        typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
        u16x2 mx2 = {0, 0}, mn2 = {0xFFFF, 0xFFFF};   // largest |s|, smallest nonzero |s| less 1 (bits)
        const uint32_t np = (ke - kb) / 512;   // 16-byte pieces of the row's scales
        for (uint32_t p = tid % TPR; p < np; p += 4 * TPR) {
            u32x4 v[4];   // four loads in flight; past the end the last piece again
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = rs[min(p + (uint32_t)(e * TPR), np - 1)];
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const u16x2 a = __builtin_bit_cast(u16x2, v[e / 4][e % 4] & 0x7FFF7FFFu);
                mx2 = __builtin_elementwise_max(mx2, a);
                mn2 = __builtin_elementwise_min(mn2, a - (u16x2){1, 1});
            }
        }
        uint32_t mx = max(mx2[0], mx2[1]), mn1 = min(mn2[0], mn2[1]);
#pragma unroll
        for (int o = 1; o < TPR; o *= 2) {
            mx = max(mx, (uint32_t)__shfl_xor((int)mx, o, 64));
            mn1 = min(mn1, (uint32_t)__shfl_xor((int)mn1, o, 64));
        }
        if (tid % TPR == 0) {
            const uint32_t hi = mx >> 7, lo = (mn1 + 1u) >> 7;   // exponent fields
            // all zero: the sums of the biases as they are
            rowexp[row] = mx == 0 ? 20 : (hi >= 106 && hi < 139 && hi - lo <= 12 ? 142 - (int)hi : ROW_WIDE);   // 15 - (hi - 127)
        }
    }
    load_barrier();
    if constexpr (BITS == 4) {
        bool any = false;
#pragma unroll
        for (int s = 0; s < NSUB; ++s)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                ex[s][j] = rowexp[64 * s + 32 * wn + 16 * j + r16];
                any = any || ex[s][j] == ROW_WIDE;
            }
        wide = __builtin_amdgcn_ballot_w64(any) != 0;
        if (wide) {
#pragma unroll
            for (int s = 0; s < NSUB; ++s)
#pragma unroll
                for (int j = 0; j < 2; ++j) ex[s][j] = 20;
        }
    }

    const half8 ones = {(_Float16)1.f, (_Float16)1.f, (_Float16)1.f, (_Float16)1.f,
                        (_Float16)1.f, (_Float16)1.f, (_Float16)1.f, (_Float16)1.f};
    auto compute = [&](uint32_t st) __attribute__((always_inline)) {
        const f16_t *const buf = As[st & 1];
        const uint32_t wb = (st / SPC) & 1;
        const int step = SPC > 1 ? (int)(st % SPC) * KQ + kq : kq;   // step within the W buffer
        const int c = step / CSTEPS, cs = step % CSTEPS;
        half8 af[2][4];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                af[u][i] = *(const half8 *)(buf + (i * 16 + r16) * SK + 8 * ((kq * 8 + 2 * q + u) ^ r16));
        if constexpr (BITS == 1) {
            // the lane's codes and scale of row 32 wn + r16; its other rows lie
            // at constant offsets (multiples of 16 rows swizzle alike)
            const char *const wp = (const char *)&Wc[wb][c][0] + (32 * wn + r16) * 64 +
                                   (((cs >> 1) ^ ((r16 >> 2) & 3)) << 4) + (cs & 1) * 8 + 2 * q;
            const char *const sp = (const char *)&Sc[wb][c][0] + (32 * wn + r16) * 8 + (cs >> 1) * 2;
#pragma unroll
            for (int s = 0; s < NSUB; ++s)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint32_t h = *(const uint16_t *)(wp + (64 * s + 16 * j) * 64);
                    const uint32_t sc = *(const uint16_t *)(sp + (64 * s + 16 * j) * 8);
                    half8 b0, b1;
                    expand_bits16(h, (sc | (sc << 16)) ^ 0x80008000u, b0, b1);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc[s][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[0][i], b0, acc[s][i][j], 0, 0, 0);
                    auto &a1 = [&]() -> auto & { if constexpr (TWO) return acc1; else return acc; }();
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        a1[s][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[1][i], b1, a1[s][i][j], 0, 0, 0);
                }
        } else {
            const uint16_t *const sp = (const uint16_t *)&Sc[wb][c][0];
            half2v S[NSUB][2];
            float b8[NSUB][2];
#pragma unroll
            for (int s = 0; s < NSUB; ++s)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int at = s * 256 + (32 * wn + 16 * j + r16) * 2 + cs;
                    const float sc = __builtin_ldexpf(bf16_to_f32(sp[at]), ex[s][j]);
                    S[s][j] = __builtin_bit_cast(half2v, __builtin_amdgcn_cvt_pkrtz(sc, sc));
                    // the centred nibbles miss 8 s: bias b + 8 s times the row sum
                    b8[s][j] = fmaf((float)S[s][j][0], 0x1p-17f, __builtin_ldexpf(bf16_to_f32(sp[at + 128]), ex[s][j] - 20));
                }
            // row sums of A over the step's group (every column of A . ones),
            // their bias products
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float4v xs = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[0][i], ones, (float4v){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                xs = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[1][i], ones, xs, 0, 0, 0);
#pragma unroll
                for (int s = 0; s < NSUB; ++s)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[s][i][j][r] = fmaf(b8[s][j], xs[r], acc[s][i][j][r]);
            }
#pragma unroll
            for (int s = 0; s < NSUB; ++s)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int row = 64 * s + 32 * wn + 16 * j + r16;
                    const u32x2 w = *(const u32x2 *)&Wc[wb][c][row * 16 + (((2 * cs + (q >> 1)) ^ ((row >> 2) & 3)) << 2) +
                                                                  (q & 1) * 2];
                    const half2v c8 = S[s][j] * (half2v){(_Float16)-0x1p-17f, (_Float16)-0x1p-17f};
                    const half8 b0 = expand_nibbles_scaled(w[0], S[s][j], c8);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc[s][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[0][i], b0, acc[s][i][j], 0, 0, 0);
                    const half8 b1 = expand_nibbles_scaled(w[1], S[s][j], c8);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc[s][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[1][i], b1, acc[s][i][j], 0, 0, 0);
                }
        }
    };

    // 4-bit, a wide wave: products of the nibbles (as n 2^-5) with A, then s and
    // b per group
    auto compute_wide = [&](uint32_t st) __attribute__((always_inline)) {
        const f16_t *const buf = As[st & 1];
        const uint32_t wb = (st / SPC) & 1;
        const int step = SPC > 1 ? (int)(st % SPC) * KQ + kq : kq;
        const int c = step / CSTEPS, cs = step % CSTEPS;
        const uint16_t *const sp = (const uint16_t *)&Sc[wb][c][0];
        const half2v S = {(_Float16)0x1p15f, (_Float16)0x1p15f}, none = {(_Float16)0.f, (_Float16)0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            half8 af[2];
#pragma unroll
            for (int u = 0; u < 2; ++u)
                af[u] = *(const half8 *)(buf + (i * 16 + r16) * SK + 8 * ((kq * 8 + 2 * q + u) ^ r16));
            float4v xs = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[0], ones, (float4v){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            xs = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[1], ones, xs, 0, 0, 0);
#pragma unroll
            for (int s = 0; s < NSUB; ++s)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int row = 64 * s + 32 * wn + 16 * j + r16, at = s * 256 + (32 * wn + 16 * j + r16) * 2 + cs;
                    const u32x2 w = *(const u32x2 *)&Wc[wb][c][row * 16 + (((2 * cs + (q >> 1)) ^ ((row >> 2) & 3)) << 2) +
                                                                  (q & 1) * 2];
                    float4v t = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[0], expand_nibbles_scaled(w[0], S, none),
                                                                       (float4v){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    t = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[1], expand_nibbles_scaled(w[1], S, none), t, 0, 0, 0);
                    const float sc = bf16_to_f32(sp[at]), bi = bf16_to_f32(sp[at + 128]);
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        acc[s][i][j][r] = fmaf(bi, xs[r], fmaf(sc, t[r] * 0x1p5f, acc[s][i][j][r]));
                }
        }
    };

    // a wide wave in a loop of its own (the same barriers)
    auto stages = [&](auto f) __attribute__((always_inline)) {
        for (uint32_t st = 0; st < nst; ++st) {
            if (st + 1 < nst) issue(st + 1);   // block-uniform
            f(st);
            load_barrier();
        }
    };
    if (BITS == 4 && wide) stages(compute_wide);
    else stages(compute);
    if constexpr (TWO) {
#pragma unroll
        for (int t = 0; t < NSUB * 8; ++t) acc[t / 8][(t / 2) % 4][t % 2] += acc1[t / 8][(t / 2) % 4][t % 2];
    }

    // k-phase reduction through the (free) A buffers: phases [h, 2h) hand
    // their tiles to [0, h) down to phases 0 and 1, which then swap halves
    // and both finish the block (phase 0 the 16-row tiles i = 0, 1).
    constexpr int NF = NSUB * 8;
    float4v *red = (float4v *)&As[0][0];
    static_assert(KQ / 2 * 2 * NF * 64 * 16 <= (int)sizeof(As), "reduction slots fit the stage buffers");
#pragma unroll
    for (int h = KQ / 2; h >= 2; h /= 2) {
        if (kq >= h && kq < 2 * h) {
#pragma unroll
            for (int t = 0; t < NF; ++t) red[(((kq - h) * 2 + wn) * NF + t) * 64 + lane] = acc[t / 8][(t / 2) % 4][t % 2];
        }
        __syncthreads();
        if (kq < h) {
#pragma unroll
            for (int t = 0; t < NF; ++t) acc[t / 8][(t / 2) % 4][t % 2] += red[((kq * 2 + wn) * NF + t) * 64 + lane];
        }
        __syncthreads();
    }
    auto put_half = [&](int slot, auto hh) __attribute__((always_inline)) {
        constexpr int H = decltype(hh)::value;
#pragma unroll
        for (int t = 0; t < NF / 2; ++t)
            red[(slot * (NF / 2) + t) * 64 + lane] = acc[t / 4][2 * H + (t / 2) % 2][t % 2];
    };
    auto add_half = [&](int slot, auto hh) __attribute__((always_inline)) {
        constexpr int H = decltype(hh)::value;
#pragma unroll
        for (int t = 0; t < NF / 2; ++t)
            acc[t / 4][2 * H + (t / 2) % 2][t % 2] += red[(slot * (NF / 2) + t) * 64 + lane];
    };
    if (kq == 0) put_half(2 + wn, IC<1>{});   // phase 1's tiles
    else if (kq == 1) put_half(wn, IC<0>{});  // phase 0's tiles
    __syncthreads();
    if (kq >= 2) return;   // after the last barrier
    if (kq == 0) add_half(wn, IC<0>{});
    else add_half(2 + wn, IC<1>{});

    // D layout: lane holds rows 4 q + r, column r16 of each 16 x 16 tile.
    auto epilogue = [&](auto ti) __attribute__((always_inline)) {
        constexpr int i = decltype(ti)::value;
        auto value = [&](int s, int j, int r) __attribute__((always_inline)) {
            float v = acc[s][i][j][r];
            if constexpr (BITS == 4) v = __builtin_ldexpf(v, 20 - ex[s][j]);
            return v;
        };
        auto rnd = [&](float v) __attribute__((always_inline)) { return BITS == 4 ? bf16_trunc(v) : v; };
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t p = p0 + i * 16 + 4 * q + r;
            if (p >= ga.P) continue;
            if constexpr (SPLIT) {
                float *const row = ga.part + ((size_t)sp * ga.P + p) * ga.cols;
#pragma unroll
                for (int s = 0; s < NSUB; ++s)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        row[bx * ROWS + 64 * s + 32 * wn + 16 * j + r16] = value(s, j, r);
                continue;
            }
#pragma unroll
            for (int s = 0; s < (PAIR ? 1 : NSUB); ++s)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint32_t n = n0 + 64 * s + 32 * wn + 16 * j + r16;
                    const size_t o = (size_t)p * out_rows + n;
                    const float v = value(s, j, r);
                    if constexpr (MODE == NNZ_GEMM_STORE_F16) ((f16_t *)out)[o] = (f16_t)rnd(v);
                    else if constexpr (MODE == NNZ_GEMM_STORE_F32) ((float *)out)[o] = rnd(v);
                    else if constexpr (MODE == NNZ_GEMM_RESADD) ((float *)out)[o] += rnd(v);
                    else ((f16_t *)out)[o] = (f16_t)rnd(silu_mul(v, value(NSUB - 1, j, r)));
                }
        }
    };
    if (kq == 0) {
        epilogue(IC<0>{});
        epilogue(IC<1>{});
    } else {
        epilogue(IC<2>{});
        epilogue(IC<3>{});
    }
}

// Sum of the splits' partial results and the epilogue; a thread takes four
// columns of a token (segments and sub-blocks are multiples of 64 columns).
template <int BITS, int MODE>
__global__ __launch_bounds__(256) void qgemm_reduce_kernel(GemmArgs ga) {
    const uint32_t c4 = ga.cols / 4, e = blockIdx.x * 256 + threadIdx.x;
    if (e >= ga.P * c4) return;
    const uint32_t p = e / c4;
    uint32_t n = e % c4 * 4;
    const float *src = ga.part + (size_t)p * ga.cols + n;
    const size_t stride = (size_t)ga.P * ga.cols;
    float4v v = *(const float4v *)src;
    for (uint32_t s = 1; s < ga.splits; ++s) v += *(const float4v *)(src + s * stride);
    void *out = ga.m0.out;
    uint32_t rows = ga.m0.rows;
    if (ga.n > 1 && n >= rows) {
        n -= rows;
        out = ga.m1.out;
        rows = ga.m1.rows;
        if (ga.n > 2 && n >= rows) {
            n -= rows;
            out = ga.m2.out;
            rows = ga.m2.rows;
        }
    }
    const size_t o = (size_t)p * rows + n;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float y = BITS == 4 ? bf16_trunc(v[r]) : v[r];
        if constexpr (MODE == NNZ_GEMM_STORE_F16) ((f16_t *)out)[o + r] = (f16_t)y;
        else if constexpr (MODE == NNZ_GEMM_STORE_F32) ((float *)out)[o + r] = y;
        else ((float *)out)[o + r] += y;
    }
}

// The forms the main kernel takes.  Others (K not a multiple of 512, other
// group sizes, f16 scales of 4-bit weights, less aligned pointers) run on the
// kernels above.
bool qgemm_weight_ok(const nnz_qweight *w, uint32_t K) {
    return w && K % 512 == 0 && ((uintptr_t)w->codes & 15) == 0 &&
           (w->bits == 1 ? w->group_size == 128 && ((uintptr_t)w->scales & 3) == 0
                         : w->group_size == 64 && w->scale_dtype == NNZ_BF16 && ((uintptr_t)w->scales & 15) == 0 &&
                               ((uintptr_t)w->biases & 3) == 0);
}

// A single 1-bit launch of K <= 2048 and at most one block per CU (of K = 512,
// two) stays on dq_gemm_kernel: too few stages for the main kernel's longer
// first loads.  Measured, dq_gemm_kernel / main: 4096 x 2048, P = 200 (256
// blocks) 8.75 / 9.88 us, P = 320 (320) 12.86 / 12.15; 2048 x 2048, P = 400
// (224) 8.47 / 9.23, P = 512 (256) 9.27 / 9.54, P = 640 (320) 12.85 / 12.01;
// 2048 x 1024, P = 400 5.96 / 6.44, P = 640 8.36 / 8.35; 2048 x 512, P = 1024
// (512) 6.54 / 6.75.  (The one size seen ahead below the line: 1024 x 2048, P =
// 1024, 9.47 / 8.99.)
bool qgemm_short(uint32_t rows, uint32_t P, uint32_t K) {
    const uint32_t g = rows / 64 * ceil_div(P, (uint32_t)BM);
    return K <= 2048 && g <= (K <= 512 ? 512u : 256u);
}

template <int BITS, int MODE, int NSUB, int KQ>
void qgemm_start(nnz_ctx *ctx, GemmArgs ga, uint32_t rows) {
    ga.nx = rows / (MODE == NNZ_GEMM_SILU_PAIR ? 64u : 64u * NSUB);
    const uint32_t nb = ga.nx * ceil_div(ga.P, (uint32_t)BM);
    qgemm_kernel<BITS, MODE, NSUB, KQ, false><<<ceil_div(nb, 8u) * 8u, 128 * KQ, 0, ctx->stream>>>(ga);
}

// Whether a launch may use the context's workspace: not under capture, since
// the graph may be replayed beside the context's own work or after its end.
bool workspace_free(nnz_ctx *ctx) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return ctx->gemm_ws && hipStreamIsCapturing(ctx->stream, &st) == hipSuccess && st == hipStreamCaptureStatusNone;
}

// The same with K split over `splits` blocks per tile, their partial sums
// through the context's workspace (splits x blocks <= 256: it fits).
template <int BITS, int MODE, int NSUB, int KQ>
void qgemm_split(nnz_ctx *ctx, GemmArgs ga, uint32_t rows, uint32_t splits) {
    ga.nx = rows / (64u * NSUB);
    ga.part = ctx->gemm_ws;
    ga.splits = splits;
    ga.cols = rows;
    const uint32_t nb = ga.nx * ceil_div(ga.P, (uint32_t)BM) * splits;
    qgemm_kernel<BITS, MODE, NSUB, KQ, true><<<ceil_div(nb, 8u) * 8u, 128 * KQ, 0, ctx->stream>>>(ga);
    qgemm_reduce_kernel<BITS, MODE><<<ceil_div(ga.P * (rows / 4), 256u), 256, 0, ctx->stream>>>(ga);
}

// Shape of a single-matrix launch (one or more row segments), by how many
// 64-row blocks g it has: a CU holds 3 blocks of KQ = 2 (42 KB of LDS, 51 with
// 128 rows), of KQ = 4 two 1-bit ones (75 KB) or one 4-bit one (84 KB), one of
// KQ = 8 (140 KB).
//   * More than one round of KQ = 2 64-row blocks: 128-row blocks, half the A
//     traffic (1-bit 2560 x 4096, P = 3001: 63 us against 72 with 64 rows; 6144
//     x 2560 86 against 104, P = 768 29.5 against 31.1; 2560 x 9728, P = 1500 74
//     against 104).
//   * Up to 768, from 512 (1-bit) or 256 (4-bit), where KQ = 4 takes a second
//     round: one round of KQ = 2 64-row blocks (2048 x 2048, P = 1500: 18.0 us
//     against 23.7 on KQ = 4; 6144 x 2560, P = 512: 22.6 against 25.0; 4-bit
//     4096 x 2560, P = 400: 21.7 against 26.3, 2560 x 9728, P = 512: 65.8
//     against 79.7, 2048 x 2048, P = 1024: 18.1 against 22.1).
//   * Fewer: KQ = 4, more waves per block (2048 x 6144, P = 1024: 33.5 against
//     38.5 on KQ = 2; 4-bit 2048 x 6144, P = 512: 29.2 against 41.9).
//   * 1-bit, at most one block per CU: KQ = 8 (K > 2048, see qgemm_short; 2048
//     x 6144, P = 512: 21.7 against 25.4 on KQ = 4; the 4-bit stages of KQ = 8
//     do not fit LDS).
template <int BITS, int MODE>
void qgemm_single(nnz_ctx *ctx, const GemmArgs &ga, uint32_t rows, bool rows128) {
    const uint32_t ny = ceil_div(ga.P, (uint32_t)BM);
    const uint32_t g = rows / 64 * ny;   // blocks of 64 rows
    // Few blocks and a long K: split K so that up to 256 blocks run, four ways
    // at most (8 ways: 2560 x 9728, P = 45, 18.9 us against 13.0).  Measured
    // unsplit -> split: 1-bit P = 45 4096 x 12288 29.0 -> 15.9, 2048 x 6144 15.2
    // -> 9.9, 4096 x 4096 11.7 -> 9.8, 2048 x 2048 7.6 -> 7.5 (not split); two
    // ways, P = 128 4096 x 12288 32.0 -> 24.8, 4096 x 4096 13.4 -> 14.2 (not
    // split); 4-bit P = 45 4096 x 12288 46.4 -> 20.2, 2048 x 2048 10.2 -> 8.7,
    // P = 200 2048 x 2048 11.8 -> 12.5 (not split).  KQ = 8 from 2048 k a block
    // (9728 / 4: 13.0 against 14.0; 6144 / 4: 10.2 against 9.9).
    const uint32_t S = std::min(4u, 256u / std::max(g, 1u));
    if (S >= 2 && ga.K >= (BITS == 1 ? (S == 4 ? 4096u : 6144u) : (S == 4 ? 2048u : 4096u)) && workspace_free(ctx)) {
        if constexpr (BITS == 1) {
            if (ga.K / S >= 2048) return qgemm_split<BITS, MODE, 1, 8>(ctx, ga, rows, S);
        }
        return qgemm_split<BITS, MODE, 1, 4>(ctx, ga, rows, S);
    }
    if (g > 768) {
        if (rows128) qgemm_start<BITS, MODE, 2, 2>(ctx, ga, rows);
        else qgemm_start<BITS, MODE, 1, 2>(ctx, ga, rows);
    } else if (g > (BITS == 1 ? 512u : 256u)) {
        qgemm_start<BITS, MODE, 1, 2>(ctx, ga, rows);
    } else {
        if constexpr (BITS == 1) {
            if (g <= 256) return qgemm_start<BITS, MODE, 1, 8>(ctx, ga, rows);
        }
        qgemm_start<BITS, MODE, 1, 4>(ctx, ga, rows);
    }
}

template <int BITS>
int qgemm_launch(nnz_ctx *ctx, const nnz_qweight *wa, const nnz_qweight *wb, const f16_t *A, uint32_t P, void *out,
                 int mode, const nnz_qmv_dims &d) {
    auto mat = [&](const nnz_qweight *w) {
        return GemmMat{w->codes, (const uint16_t *)w->scales, (const uint16_t *)w->biases, out, d.M};
    };
    GemmArgs ga{A, mat(wa), {}, {}, 1, P, d.K, 0, nullptr, 1, 0};
    const bool r128 = d.M % 128 == 0;
    switch (mode) {
    case NNZ_GEMM_STORE_F16: qgemm_single<BITS, NNZ_GEMM_STORE_F16>(ctx, ga, d.M, r128); break;
    case NNZ_GEMM_STORE_F32: qgemm_single<BITS, NNZ_GEMM_STORE_F32>(ctx, ga, d.M, r128); break;
    case NNZ_GEMM_RESADD: qgemm_single<BITS, NNZ_GEMM_RESADD>(ctx, ga, d.M, r128); break;
    case NNZ_GEMM_SILU_PAIR:
        ga.m1 = mat(wb);
        // up to one block per CU: twice the waves per block (2 x 6144 x 2048, P =
        // 45, 96 blocks: 13.0 -> 11.3 us; 2 x 12288 x 4096, 192: 27.5 -> 21.5; 2 x
        // 9728 x 2560, P = 128, 304: 23.4 -> 28.3, KQ = 2 there)
        if (d.M / 64 * ceil_div(P, (uint32_t)BM) <= 256) qgemm_start<BITS, NNZ_GEMM_SILU_PAIR, 2, 4>(ctx, ga, d.M);
        else qgemm_start<BITS, NNZ_GEMM_SILU_PAIR, 2, 2>(ctx, ga, d.M);
        break;
    default: return nnz_fail(ctx, NNZ_EINVAL, "dequant_gemm: unknown mode %d", mode);
    }
    NNZ_LAUNCHED(ctx);
    return NNZ_OK;
}

// k-phases and W-row groups of the single-matrix launches.  Measured at P =
// 512: with a grid of at most one block per CU and K > 2048 (the down
// projection), 8 k-phases (16 waves, 149 KB of LDS) are faster than 4
// (23.4 against 23.5-24.3 us); with A loaded straight into LDS, K = 2048
// does better on 4 (O 11.5 -> 11.3, K/V 9.4 -> 8.8 us); larger grids run 4
// (75 KB: two blocks per CU; the fused Q/K/V launch, 512 blocks: 17.1 us
// against 20.6).
// The gate/up pair runs 2 (4-wave blocks, 44 KB, 88 VGPRs: its 768 blocks
// are all resident at once; 48.7 us with 4 k-phases, 39.5 us with 2).  One
// W-row group (64 x 64 wave tiles, half the A reads from LDS, 8 waves) is
// 7-12 % slower than two.
constexpr int WN1 = 2;
constexpr uint32_t ONE_ROUND_BLOCKS = 256;   // CUs of an MI355X

template <int MODE>
void launch_single(nnz_ctx *ctx, uint32_t grid, const f16_t *A, const uint32_t *c0,
                   const uint16_t *s0, void *out, uint32_t P, uint32_t M, uint32_t K, uint32_t gl,
                   const GemmSegs &sg) {
    if (grid <= ONE_ROUND_BLOCKS && K > 2048)
        dq_gemm_kernel<MODE, 1, 8, WN1><<<grid, 64 * WN1 * 8, 0, ctx->stream>>>(
            A, c0, s0, nullptr, nullptr, out, P, M, K, gl, sg);
    else
        dq_gemm_kernel<MODE, 1, 4, WN1><<<grid, 64 * WN1 * 4, 0, ctx->stream>>>(
            A, c0, s0, nullptr, nullptr, out, P, M, K, gl, sg);
}

}  // namespace

namespace {

// 4-bit weights (every mode; results BF16-faithful, see dq4_gemm_kernel).
int gemm4_launch(nnz_ctx *ctx, const nnz_qweight *wa, const nnz_qweight *wb, const void *a,
                 uint32_t P, void *out, int mode, const nnz_qmv_dims &d) {
    const bool pair = mode == NNZ_GEMM_SILU_PAIR;
    auto ok = [&](const nnz_qweight *w) {
        return w && w->bits == 4 && w->codes && w->scales && w->biases &&
               (uint64_t)w->packed_count == (uint64_t)d.M * d.K && w->group_size == d.group_size &&
               w->scale_dtype == wa->scale_dtype && ((uintptr_t)w->codes & 15) == 0 &&
               ((uintptr_t)w->scales & 1) == 0 && ((uintptr_t)w->biases & 1) == 0;
    };
    NNZ_REQUIRE(ctx, ok(wa) && (!pair || ok(wb)), NNZ_EINVAL,
                "dequant_gemm: 4-bit weights need codes (16-byte aligned), scales and biases "
                "matching the dims");
    NNZ_REQUIRE(ctx, wa->scale_dtype == NNZ_BF16 || wa->scale_dtype == NNZ_F16, NNZ_EINVAL,
                "dequant_gemm: scale dtype must be bf16 or f16");
    NNZ_REQUIRE(ctx, d.M % BN == 0 && d.K % BK == 0 && d.group_size % BK == 0 &&
                         d.K % d.group_size == 0 && (d.group_size & (d.group_size - 1)) == 0,
                NNZ_EUNSUPPORTED,
                "dequant_gemm: need M %% 64 == 0, K %% 64 == 0, power-of-two group size %% 64 == 0");
    NNZ_REQUIRE(ctx, ((uintptr_t)a & 15) == 0, NNZ_EINVAL, "dequant_gemm: A must be 16-byte aligned");
    if (qgemm_weight_ok(wa, d.K) && (!pair || qgemm_weight_ok(wb, d.K)))
        return qgemm_launch<4>(ctx, wa, wb, (const f16_t *)a, P, out, mode, d);
    const uint32_t gl = (uint32_t)__builtin_ctz(d.group_size);
    const uint32_t grid = d.M / BN * ceil_div(P, BM);
    const f16_t *A = (const f16_t *)a;
    const uint32_t *c0 = (const uint32_t *)wa->codes;
    const uint16_t *s0 = (const uint16_t *)wa->scales, *b0 = (const uint16_t *)wa->biases;
    const int sdt = wa->scale_dtype;
    switch (mode) {
    case NNZ_GEMM_STORE_F16:
        if (grid <= ONE_ROUND_BLOCKS)
            dq4_gemm_kernel<NNZ_GEMM_STORE_F16, 1, 4><<<grid, 512, 0, ctx->stream>>>(
                A, c0, s0, b0, nullptr, nullptr, nullptr, out, P, d.M, d.K, gl, sdt);
        else
            dq4_gemm_kernel<NNZ_GEMM_STORE_F16, 1, 2><<<grid, 256, 0, ctx->stream>>>(
                A, c0, s0, b0, nullptr, nullptr, nullptr, out, P, d.M, d.K, gl, sdt);
        break;
    case NNZ_GEMM_STORE_F32:
        if (grid <= ONE_ROUND_BLOCKS)
            dq4_gemm_kernel<NNZ_GEMM_STORE_F32, 1, 4><<<grid, 512, 0, ctx->stream>>>(
                A, c0, s0, b0, nullptr, nullptr, nullptr, out, P, d.M, d.K, gl, sdt);
        else
            dq4_gemm_kernel<NNZ_GEMM_STORE_F32, 1, 2><<<grid, 256, 0, ctx->stream>>>(
                A, c0, s0, b0, nullptr, nullptr, nullptr, out, P, d.M, d.K, gl, sdt);
        break;
    case NNZ_GEMM_RESADD:
        if (grid <= ONE_ROUND_BLOCKS)
            dq4_gemm_kernel<NNZ_GEMM_RESADD, 1, 4><<<grid, 512, 0, ctx->stream>>>(
                A, c0, s0, b0, nullptr, nullptr, nullptr, out, P, d.M, d.K, gl, sdt);
        else
            dq4_gemm_kernel<NNZ_GEMM_RESADD, 1, 2><<<grid, 256, 0, ctx->stream>>>(
                A, c0, s0, b0, nullptr, nullptr, nullptr, out, P, d.M, d.K, gl, sdt);
        break;
    case NNZ_GEMM_SILU_PAIR:
        dq4_gemm_kernel<NNZ_GEMM_SILU_PAIR, 2, 2><<<grid, 256, 0, ctx->stream>>>(
            A, c0, s0, b0, (const uint32_t *)wb->codes, (const uint16_t *)wb->scales,
            (const uint16_t *)wb->biases, out, P, d.M, d.K, gl, sdt);
        break;
    default:
        return nnz_fail(ctx, NNZ_EINVAL, "dequant_gemm: unknown mode %d", mode);
    }
    NNZ_LAUNCHED(ctx);
    return NNZ_OK;
}

}  // namespace

int nnz_gemm_launch(nnz_ctx *ctx, const nnz_qweight *wa, const nnz_qweight *wb, const void *a,
                    uint32_t P, void *out, int mode, const nnz_qmv_dims &d) {
    NNZ_REQUIRE(ctx, wa && a && out && P > 0, NNZ_EINVAL, "dequant_gemm: null argument");
    if (wa->bits == 4) return gemm4_launch(ctx, wa, wb, a, P, out, mode, d);
    NNZ_REQUIRE(ctx, wa->bits == 1 && wa->codes && wa->scales, NNZ_EUNSUPPORTED,
                "dequant_gemm: 1-bit or 4-bit weights");
    NNZ_REQUIRE(ctx, (uint64_t)wa->packed_count == (uint64_t)d.M * d.K && wa->group_size == d.group_size,
                NNZ_EINVAL, "dequant_gemm: descriptor does not match dims");
    NNZ_REQUIRE(ctx, d.M % BN == 0 && d.K % BK == 0 && d.group_size % BK == 0 &&
                         d.K % d.group_size == 0,
                NNZ_EUNSUPPORTED, "dequant_gemm: need M %% 64 == 0, K %% 64 == 0, group size %% 64 == 0");
    NNZ_REQUIRE(ctx, ((uintptr_t)a & 15) == 0, NNZ_EINVAL, "dequant_gemm: A must be 16-byte aligned");
    NNZ_REQUIRE(ctx, ((uintptr_t)wa->codes & 7) == 0 && (!wb || ((uintptr_t)wb->codes & 7) == 0),
                NNZ_EINVAL, "dequant_gemm: codes must be 8-byte aligned");
    const bool pair = mode == NNZ_GEMM_SILU_PAIR;
    if (pair) {
        NNZ_REQUIRE(ctx, wb && wb->bits == 1 && wb->codes && wb->scales &&
                             (uint64_t)wb->packed_count == (uint64_t)d.M * d.K &&
                             wb->group_size == d.group_size,
                    NNZ_EINVAL, "dequant_gemm: bad second weight for SILU_PAIR");
    }
    NNZ_REQUIRE(ctx, (d.group_size & (d.group_size - 1)) == 0, NNZ_EUNSUPPORTED,
                "dequant_gemm: group size must be a power of two");
    if (qgemm_weight_ok(wa, d.K) && (pair ? qgemm_weight_ok(wb, d.K) : !qgemm_short(d.M, P, d.K)))
        return qgemm_launch<1>(ctx, wa, wb, (const f16_t *)a, P, out, mode, d);
    const uint32_t gl = (uint32_t)__builtin_ctz(d.group_size);
    const uint32_t grid = d.M / BN * ceil_div(P, BM);
    const f16_t *A = (const f16_t *)a;
    const uint32_t *c0 = (const uint32_t *)wa->codes;
    const uint16_t *s0 = (const uint16_t *)wa->scales;
    switch (mode) {
    case NNZ_GEMM_STORE_F16:
        launch_single<NNZ_GEMM_STORE_F16>(ctx, grid, A, c0, s0, out, P, d.M, d.K, gl, GemmSegs{});
        break;
    case NNZ_GEMM_STORE_F32:
        launch_single<NNZ_GEMM_STORE_F32>(ctx, grid, A, c0, s0, out, P, d.M, d.K, gl, GemmSegs{});
        break;
    case NNZ_GEMM_RESADD:
        launch_single<NNZ_GEMM_RESADD>(ctx, grid, A, c0, s0, out, P, d.M, d.K, gl, GemmSegs{});
        break;
    case NNZ_GEMM_SILU_PAIR:
        dq_gemm_kernel<NNZ_GEMM_SILU_PAIR, 2, 2, 2><<<grid, 256, 0, ctx->stream>>>(
            A, c0, s0, (const uint32_t *)wb->codes, (const uint16_t *)wb->scales, out, P, d.M, d.K, gl, GemmSegs{});
        break;
    default:
        return nnz_fail(ctx, NNZ_EINVAL, "dequant_gemm: unknown mode %d", mode);
    }
    NNZ_LAUNCHED(ctx);
    return NNZ_OK;
}

// One launch for up to three matrices sharing K and the A operand (the
// prefill's Q, K and V projections), f16 outputs of their own.
int nnz_gemm_segments_launch(nnz_ctx *ctx, const nnz_qweight *const *w, void *const *out, int nw,
                             const void *a, uint32_t P, uint32_t K, uint32_t group_size) {
    NNZ_REQUIRE(ctx, nw >= 1 && nw <= 3 && a && P > 0, NNZ_EINVAL, "gemm_segments: bad arguments");
    NNZ_REQUIRE(ctx, K % BK == 0 && group_size % BK == 0 && K % group_size == 0 &&
                         (group_size & (group_size - 1)) == 0,
                NNZ_EUNSUPPORTED, "gemm_segments: need K %% 64 == 0, power-of-two group size %% 64 == 0");
    NNZ_REQUIRE(ctx, ((uintptr_t)a & 15) == 0, NNZ_EINVAL, "gemm_segments: A must be 16-byte aligned");
    uint32_t rows[3] = {0, 0, 0}, M = 0;
    for (int i = 0; i < nw; ++i) {
        NNZ_REQUIRE(ctx, w[i] && out[i] && w[i]->bits == 1 && w[i]->codes && w[i]->scales &&
                             w[i]->group_size == group_size && w[i]->packed_count % K == 0,
                    NNZ_EINVAL, "gemm_segments: bad weight %d", i);
        NNZ_REQUIRE(ctx, ((uintptr_t)w[i]->codes & 7) == 0, NNZ_EINVAL,
                    "gemm_segments: codes must be 8-byte aligned");
        rows[i] = w[i]->packed_count / K;
        NNZ_REQUIRE(ctx, rows[i] % BN == 0, NNZ_EUNSUPPORTED, "gemm_segments: rows %% 64 != 0");
        M += rows[i];
    }
    bool main_form = true, r128 = true;
    for (int i = 0; i < nw; ++i) {
        main_form = main_form && qgemm_weight_ok(w[i], K);
        r128 = r128 && rows[i] % 128 == 0;
    }
    if (main_form && !qgemm_short(M, P, K)) {
        GemmArgs ga{(const f16_t *)a, {}, {}, {}, (uint32_t)nw, P, K, 0, nullptr, 1, 0};
        GemmMat *const m[3] = {&ga.m0, &ga.m1, &ga.m2};
        for (int i = 0; i < nw; ++i) *m[i] = GemmMat{w[i]->codes, (const uint16_t *)w[i]->scales, nullptr, out[i], rows[i]};
        qgemm_single<1, NNZ_GEMM_STORE_F16>(ctx, ga, M, r128);
        NNZ_LAUNCHED(ctx);
        return NNZ_OK;
    }
    GemmSegs sg{(uint32_t)nw, rows[0], rows[1],
                nw > 1 ? (const uint32_t *)w[1]->codes : nullptr,
                nw > 2 ? (const uint32_t *)w[2]->codes : nullptr,
                nw > 1 ? (const uint16_t *)w[1]->scales : nullptr,
                nw > 2 ? (const uint16_t *)w[2]->scales : nullptr,
                nw > 1 ? out[1] : nullptr, nw > 2 ? out[2] : nullptr};
    const uint32_t grid = M / BN * ceil_div(P, BM);
    launch_single<NNZ_GEMM_STORE_F16>(ctx, grid, (const f16_t *)a, (const uint32_t *)w[0]->codes,
                                      (const uint16_t *)w[0]->scales, out[0], P, M, K,
                                      (uint32_t)__builtin_ctz(group_size), sg);
    NNZ_LAUNCHED(ctx);
    return NNZ_OK;
}

extern "C" int nnz_dispatch_dequant_gemm(nnz_ctx *ctx, const nnz_qweight *wa, const nnz_qweight *wb,
                                         const void *a_f16, uint32_t num_tokens, void *output, int mode,
                                         nnz_qmv_dims dims) {
    NNZ_CHECK_CTX(ctx);
    return nnz_gemm_launch(ctx, wa, wb, a_f16, num_tokens, output, mode, dims);
}
