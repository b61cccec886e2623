// Learned prefilter: the sequence encoder and the candidate proposal.
//
// Encoder of one sequence (codes 0..19, 20 for anything else):
//   x0[p] = E[code[p]]                              E: 22 x 64, rows 20, 21 zero
//   h1    = GELU(conv9(x0; W1: 64 -> 128) + b1)
//   h2    = GELU(conv9(h1; W2: 128 -> 128) + b2)
//   h3    = GELU(conv9(h2; W3: 128 -> 256) + b3)
//   z     = mean over positions of h3,  e = z / |z|      (256-d)
// conv9(x; W)[p][o] = sum_{t<9} sum_i x[p + t - 4][i] * W[t][i][o], zero
// outside the sequence.  The similarity of two sequences is e_q . e_t.
//
// Layout: a batch of sequences is one flat array of rows (positions) with
// four zero "pad" rows before every sequence and after the last one, and
// the row count rounded up to a multiple of 128 with pad rows; mask[p] = 1
// on residue rows, 0 on pad rows.  A layer's input row p + t - 4 of a
// residue row never leaves its sequence and its pads, so a conv layer is
// one GEMM over all rows: C[p][o] = sum_k A[p][k] * Bt[o][k] with
// A[p][k] = X[(p - 4) * Cin + k], k < 9 * Cin -- row p of A is the
// contiguous window of rows p-4 .. p+4 of X -- and Bt the weights as
// [o][t * Cin + i].  Every layer's output is zeroed on pad rows, so pads
// stay zero for the next layer.  The backward pass over the input is the
// same GEMM on dU (gradient before the GELU) with the weights flipped and
// transposed, Bt'[i][t * Cout + o] = W[8 - t][i][o]; the weight gradient
// dW[t * Cin + i][o] = sum_p A[p][t * Cin + i] * dU[p][o] reduces over rows.
//
// bf16 operands, fp32 accumulation on v_mfma_f32_32x32x16_bf16.  The
// proposal scores e_q . e_t of many queries against an FP8 (e4m3) table of
// every database sequence on v_mfma_f32_16x16x32_fp8_fp8.
#include "common.h"

#include <algorithm>
#include <cmath>

namespace sseqs {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline float bf2f(__bf16 v) { return (float)v; }
__device__ inline __bf16 f2bf(float v) { return (__bf16)v; }

// Orders a wave's LDS accesses across its lanes (no barrier between waves):
// wavefront-scope release/acquire fences keep the compiler's memory
// operations on either side, and the hardware runs one wave's LDS
// instructions in order.
__device__ __forceinline__ void lds_wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// GELU, tanh form, and its derivative.
__device__ inline float gelu(float x) {
    const float c = 0.7978845608028654f;  // sqrt(2 / pi)
    const float u = c * (x + 0.044715f * x * x * x);
    return 0.5f * x * (1.f + tanhf(u));
}
__device__ inline float gelu_grad(float x) {
    const float c = 0.7978845608028654f;
    const float u = c * (x + 0.044715f * x * x * x);
    const float t = tanhf(u);
    return 0.5f * (1.f + t) + 0.5f * x * (1.f - t * t) * c * (1.f + 3.f * 0.044715f * x * x);
}

// bf16 of gelu(x0) * m0 and gelu(x1) * m1 (low and high half), equal to the
// functions above bit for bit.  tanhf is a divergent branch of some 40
// instructions, twice the products' own time in the narrow layers.  Here
// tanh u = 2 g - 1 with g = 1 / (1 + exp(-2u)) comes from the hardware's
// exponential and reciprocal, once with g a little too small and once a little
// too large (GELU_EPS).  Each further step is monotonic, so where both ends round
// to one bf16 that is gelu's; where they differ (about 1 in 2000), gelu() itself
// is evaluated.  That the tanhf of gelu() lies between them, its rounding of
// 1 + tanh u for negative u included, is a fact about the installed tanhf: a test
// compares all normal floats.
constexpr float GELU_EPS = 3e-6f;
__device__ inline uint32_t gelu_bf16x2(float x0, float x1, float m0, float m1) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const float x[2] = {x0, x1}, m[2] = {m0, m1};
    bf16x2 lo, hi;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float c = 0.7978845608028654f;  // sqrt(2 / pi)
        const float u = c * (x[i] + 0.044715f * x[i] * x[i] * x[i]);
        const float g =
            __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-2.f * 1.4426950408889634f * u));
        const float h = 0.5f * x[i] * m[i];
        lo[i] = f2bf(h * (1.f + fmaf(g, 2.f - GELU_EPS, -1.f)));
        hi[i] = f2bf(h * (1.f + fmaf(g, 2.f + GELU_EPS, -1.f)));
    }
    uint32_t v = __builtin_bit_cast(uint32_t, lo);
    if (v != __builtin_bit_cast(uint32_t, hi)) {
        lo[0] = f2bf(gelu(x0) * m0);
        lo[1] = f2bf(gelu(x1) * m1);
        v = __builtin_bit_cast(uint32_t, lo);
    }
    return v;
}

// ------------------------------------------------------------- conv GEMM --
//
// A block computes 64 WM - 8 rows x BN columns of C, wave (wm, wn) the rows
// 64 wm .. + 63 (the last wave's last eight are left out) x the BN / WN
// columns of wn, as 2 x BN / (32 WN) MFMA tiles of 32 x 32.  The block's
// 64 WM rows of A are read from memory once and stay in LDS for the nine
// taps, which only shift the row that a lane reads; without the eight rows
// that are left out they and two stages of Bt take half the LDS of a CU
// exactly, so that two blocks share it and one's epilogue and first loads run
// beside the other's products.  K goes by 32 columns of Bt at a time, in
// order: the sums are those of a plain loop over K.  Bt is read two stages
// ahead, into registers; the second half of a stage's operands leaves LDS
// between the products of the first.  Rows of LDS hold their 16-byte pieces
// at piece ^ (row mod 16) (A) and ^ (row / 2 mod 4) (Bt), so that neither the
// row-wise stores nor the operand reads meet in a bank.
//
// MFMA 32x32x16 operands: lane (r = lane % 32, h = lane / 32) supplies
// row r, elements 8h .. 8h+7 of K of both operands.  The weights are the
// first operand: result element e of lane (c, h) is then column
// 8 * (e / 4) + 4 * h + (e % 4) of C in row c, four consecutive columns to a
// lane.
//
// Bound by issue slots: the products take 55 % of them, GELU most of the rest.
// The three layers over 8.6 M rows 16.1 -> 10.0 ms (0.55 -> 0.88 PFLOP/s)
// against 128 x 128 tiles that read every tap's rows from memory, with tanhf
// and two-byte stores; in steps 12.3 (rows kept, wide waves), 10.6
// (gelu_bf16x2) and 10.0 (whole lines out). The backward products of 312 k
// rows 761 -> 466 us.
constexpr int GM = 128, GK = 32;  // granularity of M; columns of Bt of a stage
// Wide blocks when they fill the 512 places of the chip (two a CU) once; with
// fewer, small blocks spread the rows over more CUs.
constexpr int64_t CONV_WIDE = 512;

enum ConvEpi {
    EPI_FWD = 0,      // u = acc + bias; U = u (optional); Y = gelu(u) * mask
    EPI_BWD_GELU = 1, // dUprev = acc * gelu'(Uprev) * mask
    EPI_BWD_F32 = 2,  // dX (fp32) = acc * mask (input of layer 1)
};

struct ConvArgs {
    const __bf16* A;     // A row p at A + (p - 4) * lda (rows -4 .. M + 3 readable)
    int lda;             // elements between consecutive rows of A (Cin or Cout)
    const __bf16* Bt;    // N rows of K
    int64_t M;
    int N, K;
    const float* bias;   // EPI_FWD
    const uint8_t* mask; // [M]
    __bf16* U;           // EPI_FWD: pre-activation out (may be null)
    __bf16* Y;           // EPI_FWD: activation out; EPI_BWD_GELU: gradient out
    const __bf16* Uprev; // EPI_BWD_GELU
    float* Yf;           // EPI_BWD_F32
};

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// 16 bytes at the alignment of their elements (the same instructions)
typedef uint32_t u32x4_el __attribute__((ext_vector_type(4), aligned(2)));
typedef __bf16 bf16x8_el __attribute__((ext_vector_type(8), aligned(2)));

// CIN: lda, K = 9 CIN
template <int CIN, int BN, int EPI, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN, 2) void k_conv_gemm(ConvArgs a) {
    constexpr int NT = BN / (32 * WN);     // MFMA tiles of a wave along N
    constexpr int TH = 64 * WM * WN, ROWS = 64 * WM, OUT = ROWS - 8;
    constexpr int RB = 2 * CIN;            // bytes of a row of A
    constexpr int PA = RB / 16;            // its 16-byte pieces
    constexpr int SW = PA < 16 ? PA - 1 : 15;
    constexpr int APT = ROWS * PA / TH, BPT = BN * 4 / TH;  // pieces per thread
    constexpr int NST = 9 * CIN / GK;      // stages
    __shared__ __align__(16) uint8_t sA[ROWS * RB];
    __shared__ __align__(16) uint8_t sB[2][BN * 64];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm = w / WN, wn = w % WN;
    const int r = lane & 31, h = lane >> 5;
    // the blocks of one row tile are dealt to one XCD (block id mod 8), whose
    // L2 then holds the tile's rows for all of them
    const int nt = a.N / BN, slot = blockIdx.x >> 3;
    const int64_t m0 = ((int64_t)(slot / nt) * 8 + (blockIdx.x & 7)) * OUT;
    const int n0 = slot % nt * BN;
    if (m0 >= a.M) return;

    // Bt through registers: piece tid % 4 of rows tid / 4 + (TH / 4) x
    const int brow = tid >> 2, bc = tid & 3;
    const __bf16* gB = a.Bt + (int64_t)(n0 + brow) * a.K + 8 * bc;
    uint8_t* lB = &sB[0][0] + brow * 64 + 16 * (bc ^ ((brow >> 1) & 3));
    u32x4 rb[2][BPT];
#define CONV_LOAD_B(set, st)                                                               \
    _Pragma("unroll") for (int x = 0; x < BPT; ++x) rb[set][x] =                           \
        *reinterpret_cast<const u32x4*>(gB + (int64_t)(TH / 4 * x) * a.K + (st) * GK)
    // TH / 4 is a multiple of 8, so the swizzle is that of brow
#define CONV_STORE_B(set)                                                                  \
    _Pragma("unroll") for (int x = 0; x < BPT; ++x) *reinterpret_cast<u32x4*>(             \
        lB + (set) * (BN * 64) + TH / 4 * x * 64) = rb[set][x]
    {
        u32x4 ra[APT];
        const int prow = tid / PA, pc = tid % PA;
#pragma unroll
        for (int x = 0; x < APT; ++x) {  // rows m0 - 4 .. , none past M + 3
            int64_t row = m0 - 4 + prow + TH / PA * x;
            row = row < a.M + 3 ? row : a.M + 3;
            ra[x] = *reinterpret_cast<const u32x4*>(a.A + row * CIN + 8 * pc);
        }
        CONV_LOAD_B(0, 0);
        CONV_LOAD_B(1, 1);
#pragma unroll
        for (int x = 0; x < APT; ++x) {
            const int row = prow + TH / PA * x;
            *reinterpret_cast<u32x4*>(sA + row * RB + 16 * (pc ^ (row & SW))) = ra[x];
        }
        CONV_STORE_B(0);
    }
    f32x16 acc[2][NT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    __syncthreads();

    const uint8_t* fB = &sB[0][0] + (BN / WN * wn + r) * 64 + 16 * (h ^ ((r >> 1) & 3));
    const int boff = (int)(fB - &sB[0][0]);
#pragma unroll 1
    for (int t = 0; t < 9; ++t) {
        const int row = 64 * wm + r + t;  // past the block's rows: those left out
        int aoff[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
            aoff[i] = ((row + 32 * i) & (ROWS - 1)) * RB + 16 * (h ^ (row & SW));
#pragma unroll
        for (int c = 0; c < CIN / GK; ++c) {
            const int st = t * (CIN / GK) + c;
            bf16x8 fa[2][2], fb[2][NT];
#define CONV_LOAD_F(s)                                                                     \
    do {                                                                                   \
        _Pragma("unroll") for (int i = 0; i < 2; ++i) fa[s][i] =                           \
            *reinterpret_cast<const bf16x8*>(sA + (aoff[i] ^ (64 * c + 32 * s)));          \
        _Pragma("unroll") for (int j = 0; j < NT; ++j) fb[s][j] =                          \
            *reinterpret_cast<const bf16x8*>(&sB[0][0] + (c & 1) * (BN * 64) +             \
                                             (boff ^ (32 * s)) + 2048 * j);                \
    } while (0)
            CONV_LOAD_F(0);
            // rb[c & 1] went to LDS a stage ago; the last stages read stage NST - 1 again
            CONV_LOAD_B(c & 1, st + 2 < NST ? st + 2 : NST - 1);
            __builtin_amdgcn_sched_barrier(0);  // these loads are on their way first
            CONV_LOAD_F(1);
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[s][j], fa[s][i],
                                                                            acc[i][j], 0, 0, 0);
#pragma unroll
            for (int x = 0; x < 2 + NT; ++x) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // an MFMA
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // an LDS read
            }
            __builtin_amdgcn_sched_barrier(0);
            CONV_STORE_B((c + 1) & 1);  // stage st + 1
            __syncthreads();
        }
    }
#undef CONV_LOAD_B
#undef CONV_STORE_B
#undef CONV_LOAD_F

    // epilogue: lane (r, h) holds columns 32 j + 8 q + 4 h .. + 3 of its row.
    // bf16 rows pass through the wave's part of LDS (free after the last
    // stage's barrier), 32 at a time, so that whole lines of them come and go:
    // 8-byte accesses of 32 rows at once made 16-byte requests.  Row r holds
    // its 16-byte pieces at piece ^ (r mod 16).
    constexpr int WC = BN / WN, PW = 2 * WC / 16;  // the wave's columns, pieces of their row
    static_assert(WM * WN * 32 * 2 * WC <= ROWS * RB, "the waves' rows fit the place of A");
    uint8_t* lw = sA + w * (32 * 2 * WC);
    const int nw = n0 + WC * wn;
    const auto place = [&](int row, int piece) { return row * 2 * WC + 16 * (piece ^ (row & (PW - 1))); };
    // rows 64 wm + 32 i .. + 31 of the block, a whole row to PW lanes
    const auto rows_out = [&](__bf16* out, int i) {
        lds_wave_fence();
#pragma unroll
        for (int x = 0; x < 32 * PW / 64; ++x) {
            const int row = lane / PW + 64 / PW * x, pc = lane % PW;
            const int mr = 64 * wm + 32 * i + row;
            const u32x4 v = *reinterpret_cast<const u32x4*>(lw + place(row, pc));
            if (mr < OUT && m0 + mr < a.M)
                *reinterpret_cast<u32x4*>(out + (m0 + mr) * a.N + nw + 8 * pc) = v;
        }
        lds_wave_fence();
    };
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int mr = 64 * wm + 32 * i + r;
        const int64_t m = m0 + mr;
        const bool in = mr < OUT && m < a.M;
        const float mk = in && a.mask[m] ? 1.f : 0.f;
        if constexpr (EPI == EPI_FWD) {
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 bias =
                        *reinterpret_cast<const float4*>(a.bias + nw + 32 * j + 8 * q + 4 * h);
                    acc[i][j][4 * q] += bias.x;
                    acc[i][j][4 * q + 1] += bias.y;
                    acc[i][j][4 * q + 2] += bias.z;
                    acc[i][j][4 * q + 3] += bias.w;
                }
            if (a.U) {
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        bf16x4 u;
#pragma unroll
                        for (int x = 0; x < 4; ++x) u[x] = f2bf(acc[i][j][4 * q + x]);
                        *reinterpret_cast<bf16x4*>(lw + place(r, 4 * j + q) + 8 * h) = u;
                    }
                rows_out(a.U, i);
            }
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<uint2*>(lw + place(r, 4 * j + q) + 8 * h) = make_uint2(
                        gelu_bf16x2(acc[i][j][4 * q], acc[i][j][4 * q + 1], mk, mk),
                        gelu_bf16x2(acc[i][j][4 * q + 2], acc[i][j][4 * q + 3], mk, mk));
            rows_out(a.Y, i);
        } else if constexpr (EPI == EPI_BWD_GELU) {
#pragma unroll
            for (int x = 0; x < 32 * PW / 64; ++x) {
                const int row = lane / PW + 64 / PW * x, pc = lane % PW;
                const int64_t mu = min(m0 + 64 * wm + 32 * i + row, a.M - 1);
                *reinterpret_cast<u32x4*>(lw + place(row, pc)) =
                    *reinterpret_cast<const u32x4*>(a.Uprev + mu * a.N + nw + 8 * pc);
            }
            lds_wave_fence();
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    bf16x4* at = reinterpret_cast<bf16x4*>(lw + place(r, 4 * j + q) + 8 * h);
                    const bf16x4 up = *at;
                    bf16x4 y;
#pragma unroll
                    for (int x = 0; x < 4; ++x)
                        y[x] = f2bf(acc[i][j][4 * q + x] * gelu_grad(bf2f(up[x])) * mk);
                    *at = y;
                }
            rows_out(a.Y, i);
        } else if (in) {
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<float4*>(a.Yf + m * a.N + nw + 32 * j + 8 * q + 4 * h) =
                        make_float4(acc[i][j][4 * q] * mk, acc[i][j][4 * q + 1] * mk,
                                    acc[i][j][4 * q + 2] * mk, acc[i][j][4 * q + 3] * mk);
        }
    }
}

// Any K and row stride (windows that are not nine whole rows), any alignment
// of the outputs: 128 x 64 tiles, wave (wm, wn) the 64 x 32 share, both
// operands' 32 columns of K through LDS (rows padded to 40 elements) per stage.
constexpr int GPAD = 40;
template <int EPI>
__global__ __launch_bounds__(256) void k_conv_any(ConvArgs a) {
    constexpr int BN = 64, NT = 1;
    __shared__ __align__(16) __bf16 sA[2][GM * GPAD];
    __shared__ __align__(16) __bf16 sB[2][BN * GPAD];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm = w >> 1, wn = w & 1;
    const int r = lane & 31, h = lane >> 5;
    const int64_t m0 = (int64_t)blockIdx.x * GM;
    const int n0 = blockIdx.y * BN;

    // global -> register staging: A tile 128 x 32 = 512 chunks of 8, B tile
    // BN x 32 = BN * 4 chunks; thread i takes chunks i and i + 256
    const int crow = tid >> 2, ccol = (tid & 3) * 8;
    const __bf16* gA0 = a.A + (m0 + crow - 4) * a.lda + ccol;
    const __bf16* gA1 = gA0 + (int64_t)64 * a.lda;
    const __bf16* gB0 = a.Bt + (int64_t)(n0 + crow) * a.K + ccol;
    uint4 ra0, ra1, rb0;
#define CONV_GLOAD(k0)                                                     \
    do {                                                                   \
        ra0 = *reinterpret_cast<const uint4*>(gA0 + (k0));                 \
        ra1 = *reinterpret_cast<const uint4*>(gA1 + (k0));                 \
        rb0 = *reinterpret_cast<const uint4*>(gB0 + (k0));                 \
    } while (0)
#define CONV_SSTORE(b)                                                                   \
    do {                                                                                 \
        *reinterpret_cast<uint4*>(&sA[b][crow * GPAD + ccol]) = ra0;                     \
        *reinterpret_cast<uint4*>(&sA[b][(crow + 64) * GPAD + ccol]) = ra1;              \
        *reinterpret_cast<uint4*>(&sB[b][crow * GPAD + ccol]) = rb0;                     \
    } while (0)

    f32x16 acc[2][NT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    const int nk = a.K / GK;
    CONV_GLOAD(0);
    CONV_SSTORE(0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nk) CONV_GLOAD((kt + 1) * GK);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            bf16x8 fa[2], fb[NT];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                fa[i] = *reinterpret_cast<const bf16x8*>(
                    &sA[buf][(64 * wm + 32 * i + r) * GPAD + 16 * s + 8 * h]);
#pragma unroll
            for (int j = 0; j < NT; ++j)
                fb[j] = *reinterpret_cast<const bf16x8*>(
                    &sB[buf][((BN / 2) * wn + 32 * j + r) * GPAD + 16 * s + 8 * h]);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j],
                                                                        0, 0, 0);
        }
        if (kt + 1 < nk) CONV_SSTORE(buf ^ 1);
        __syncthreads();
    }
#undef CONV_GLOAD
#undef CONV_SSTORE

    // epilogue
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int n = n0 + (BN / 2) * wn + 32 * j + r;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int64_t m = m0 + 64 * wm + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3);
                const float v = acc[i][j][e];
                const float mk = a.mask[m] ? 1.f : 0.f;
                const int64_t o = m * a.N + n;
                if constexpr (EPI == EPI_FWD) {
                    const float u = v + a.bias[n];
                    if (a.U) a.U[o] = f2bf(u);
                    a.Y[o] = f2bf(gelu(u) * mk);
                } else if constexpr (EPI == EPI_BWD_GELU) {
                    a.Y[o] = f2bf(v * gelu_grad(bf2f(a.Uprev[o])) * mk);
                } else {
                    a.Yf[o] = v * mk;
                }
            }
        }
    }
}

// ---------------------------------------------------------- weight grad --
//
// dW[t * Cin + i][o] += sum_p X[p - 4 + t][i] * dU[p][o] over the rows p of
// this block's stages.  A block holds 64 channels i x 64 channels o of all
// nine taps, wave (wm, wn) a 32 x 32 MFMA tile of each tap (144 accumulators),
// so that a stage's 72 rows of X and 64 of dU come from memory once for nine
// products of 64 x 64.  K of the products runs over rows: both operands leave
// LDS through transposing reads, for which a tap is a row offset.  The next
// stage's global loads are issued before the current stage's products.  The
// block's sums are added to dW (fp32) atomically at the end.  Bound by the
// products and those additions (wg_slices).  312 k rows, three layers: 1000 -> 445
// us against 64 x 64 tiles of one tap whose operands were gathered from LDS two
// bytes at a time.
//
// ds_read_b64_tr_b16: of 16 lanes, lane 4 j + q reads the four elements q of
// row j of a 4 x 16 tile, and lane l receives column l: its four rows.
constexpr int WP = 64;           // rows per stage
constexpr int WSTRIDE = 192;     // bytes of a row of 64 channels: rows j .. j + 3 meet in no bank
constexpr int64_t WG_FILL = 512;  // blocks that are resident at once, two to a CU

typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ inline bf16x8 tr_frag(const uint8_t* p) {  // rows 0..3 and 4..7 of 16 columns per 16 lanes
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4 * WSTRIDE));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// TAIL: M is not a multiple of WP.  dU's rows past M - 1 are zeros in LDS, but
// the rows of X that they would meet belong to earlier rows of dU or follow
// the sequence, and 0 times an infinity or NaN is NaN: they are cleared in the
// fragments, by an instance of its own (312 001 rows, 128 -> 256 channels: 228
// us, 312 000 rows 204; the encoder itself always has whole stages).
template <bool TAIL>
__global__ __launch_bounds__(256, 2) void k_conv_wgrad(const __bf16* __restrict__ X, int Cin,
                                                       const __bf16* __restrict__ dU, int Cout,
                                                       int64_t M, int64_t per, float* __restrict__ dW) {
    __shared__ __align__(16) uint8_t sX[2][(WP + 8) * WSTRIDE];
    __shared__ __align__(16) uint8_t sD[2][WP * WSTRIDE];
    const int i0 = blockIdx.x * 64, o0 = blockIdx.y * 64;
    const int64_t s_lo = blockIdx.z * per, s_hi = min(s_lo + per, (M + WP - 1) / WP);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm = w >> 1, wn = w & 1;
    // 16-byte pieces: X's 576 to threads i, i + 256, i + 512, dU's 512 to i, i + 256
    const int prow = tid >> 3, pc = tid & 7;
    u32x4 rx[3], rd[2];
    const auto load = [&](int64_t st) {
        const int64_t p0 = st * WP;
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            int64_t row = p0 - 4 + min(prow + 32 * x, WP + 7);
            row = row < M + 3 ? row : M + 3;
            rx[x] = *reinterpret_cast<const u32x4*>(X + row * Cin + i0 + 8 * pc);
        }
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int64_t row = p0 + prow + 32 * x;
            rd[x] = *reinterpret_cast<const u32x4*>(dU + (row < M ? row : M - 1) * Cout + o0 + 8 * pc);
            if (row >= M) rd[x] = u32x4{0, 0, 0, 0};
        }
    };
    const auto store = [&](int buf) {
#pragma unroll
        for (int x = 0; x < 3; ++x)
            if (x < 2 || prow < 8)
                *reinterpret_cast<u32x4*>(sX[buf] + (prow + 32 * x) * WSTRIDE + 16 * pc) = rx[x];
#pragma unroll
        for (int x = 0; x < 2; ++x)
            *reinterpret_cast<u32x4*>(sD[buf] + (prow + 32 * x) * WSTRIDE + 16 * pc) = rd[x];
    };
    f32x16 acc[9];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[t][e] = 0.f;
    // lane's part of a tile: row 8 h + j, channels 16 (g & 1) + 4 q of the wave's 32
    const int g = lane >> 4, j = (lane >> 2) & 3, q = lane & 3;
    const int lrow = (8 * (g >> 1) + j) * WSTRIDE + 2 * (16 * (g & 1) + 4 * q);
    const int ax = lrow + 64 * wm, ad = lrow + 64 * wn;
    if (s_lo < s_hi) {
        load(s_lo);
        store(0);
    }
    __syncthreads();
    for (int64_t st = s_lo; st < s_hi; ++st) {
        const int buf = (int)(st - s_lo) & 1;
        if (st + 1 < s_hi) load(st + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < WP / 16; ++k) {
            const bf16x8 fb = tr_frag(sD[buf] + ad + 16 * k * WSTRIDE);
            u32x4 keep;
            if constexpr (TAIL) {
                // of the lane's rows, eight from 8 (lane / 32) on, the ones below M
                const int nv = (int)min((int64_t)8, M - (st * WP + 16 * k + 8 * (g >> 1)));
#pragma unroll
                for (int y = 0; y < 4; ++y)
                    keep[y] = nv > 2 * y + 1 ? 0xffffffffu : nv > 2 * y ? 0xffffu : 0u;
            }
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                bf16x8 fa = tr_frag(sX[buf] + ax + (16 * k + t) * WSTRIDE);
                if constexpr (TAIL)
                    fa = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, fa) & keep);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fb, acc[t], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (st + 1 < s_hi) store(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int i = i0 + 32 * wm + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
            const int o = o0 + 32 * wn + (lane & 31);
            atomicAdd(&dW[(int64_t)(t * Cin + i) * Cout + o], acc[t][e]);
        }
}

// db[o] += sum over rows of dU[p][o]: a block sums 1024 rows of 64 channels, a
// thread eight channels of every 32nd row from 16-byte loads (eight in
// flight), then the 32 row classes in LDS and one atomic per channel: blocks
// of 256 rows, with four times as many atomics on the same addresses, took twice as
// long.  312 k rows, three layers: 300 -> 79 us.
constexpr int CS_ROWS = 1024;
__global__ __launch_bounds__(256) void k_colsum(const __bf16* __restrict__ dU, int C, int64_t M,
                                                float* __restrict__ db) {
    __shared__ float s[32][65];
    const int pc = threadIdx.x & 7, ph = threadIdx.x >> 3;
    const int c0 = blockIdx.y * 64;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int q = 0; q < CS_ROWS; q += 256) {
        const int64_t lo = (int64_t)blockIdx.x * CS_ROWS + q;
        if (lo >= M) break;
        u32x4 v[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) {
            const int64_t p = lo + ph + 32 * x;
            v[x] = *reinterpret_cast<const u32x4_el*>(dU + (p < M ? p : M - 1) * C + c0 + 8 * pc);
            if (p >= M) v[x] = u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int x = 0; x < 8; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                acc[2 * y] += __uint_as_float(v[x][y] << 16);
                acc[2 * y + 1] += __uint_as_float(v[x][y] & 0xffff0000u);
            }
    }
#pragma unroll
    for (int y = 0; y < 8; ++y) s[ph][8 * pc + y] = acc[y];
    __syncthreads();
    if (threadIdx.x < 64) {
        float t = 0.f;
#pragma unroll
        for (int x = 0; x < 32; ++x) t += s[x][threadIdx.x];
        atomicAdd(&db[c0 + threadIdx.x], t);
    }
}

// ------------------------------------------------------------ small ops --

// x0[p] = E[code[p]] (bf16 rows of 64)
__global__ void k_embed(const uint8_t* __restrict__ code, int64_t M, const float* __restrict__ E,
                        __bf16* __restrict__ x0) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // one thread: 8 channels
    if (i >= M * 8) return;
    const int64_t p = i >> 3;
    const int c0 = (int)(i & 7) * 8;
    const int cd = code[p];
    bf16x8 v;
#pragma unroll
    for (int x = 0; x < 8; ++x) v[x] = f2bf(E[cd * 64 + c0 + x]);
    *reinterpret_cast<bf16x8*>(x0 + p * 64 + c0) = v;
}

// dE[code][c] += dX0[p][c].  Each wave sums its rows (eight in flight, lane =
// channel) into a table of its own in LDS, without atomics; the block's
// tables are added up and go out as one atomic per entry, from one block per
// CU.  LDS float atomics of one table per block took 117 us for 312 k rows,
// this 21.
constexpr int EG_WAVES = 16, EG_ROWS = 8;
__global__ __launch_bounds__(64 * EG_WAVES) void k_embed_grad(const uint8_t* __restrict__ code,
                                                              int64_t M,
                                                              const float* __restrict__ dx0,
                                                              float* __restrict__ dE) {
    __shared__ float s[EG_WAVES][22 * 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int i = lane; i < 22 * 64; i += 64) s[w][i] = 0.f;
    for (int64_t p0 = ((int64_t)blockIdx.x * EG_WAVES + w) * EG_ROWS; p0 < M;
         p0 += (int64_t)gridDim.x * EG_WAVES * EG_ROWS) {
        const int n = (int)min((int64_t)EG_ROWS, M - p0);
        int cd[EG_ROWS];
        float v[EG_ROWS];
#pragma unroll
        for (int x = 0; x < EG_ROWS; ++x) {
            const int64_t p = p0 + min(x, n - 1);
            cd[x] = code[p];
            v[x] = dx0[p * 64 + lane];
        }
#pragma unroll
        for (int x = 0; x < EG_ROWS; ++x)
            if (x < n) s[w][cd[x] * 64 + lane] += v[x];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 20 * 64; i += 64 * EG_WAVES) {
        float t = 0.f;
#pragma unroll
        for (int x = 0; x < EG_WAVES; ++x) t += s[x][i];
        if (t != 0.f) atomicAdd(&dE[i], t);
    }
}

// Sequence s occupies rows [row0[s], row0[s] + len[s]).  z = mean of h3
// rows, e = z / |z| (|z| = 0 leaves e = 0); one block of 256 threads per
// sequence.  Thread t reads channels 4 (t % 64) .. +3 of rows p = t / 64
// (mod 4), 8 bytes per load and 16 rows of the block in flight per step;
// the four row classes are summed in LDS, in a fixed order.
__global__ __launch_bounds__(256) void k_pool(const __bf16* __restrict__ h3,
                                              const int64_t* __restrict__ row0,
                                              const int32_t* __restrict__ len, int64_t nseq,
                                              float* __restrict__ e, float* __restrict__ znorm) {
    __shared__ float part[4][256];
    __shared__ float red[4];
    const int t = threadIdx.x, c4 = 4 * (t & 63), ph = t >> 6;
    for (int64_t s = blockIdx.x; s < nseq; s += gridDim.x) {
        const int64_t b = row0[s];
        const int L = len[s];
        float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
        int p = ph;
        for (; p + 12 < L; p += 16) {
            uint2 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                v[u] = *reinterpret_cast<const uint2*>(h3 + (b + p + 4 * u) * 256 + c4);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                a0 += __uint_as_float(v[u].x << 16);
                a1 += __uint_as_float(v[u].x & 0xffff0000u);
                a2 += __uint_as_float(v[u].y << 16);
                a3 += __uint_as_float(v[u].y & 0xffff0000u);
            }
        }
        for (; p < L; p += 4) {
            const uint2 v = *reinterpret_cast<const uint2*>(h3 + (b + p) * 256 + c4);
            a0 += __uint_as_float(v.x << 16);
            a1 += __uint_as_float(v.x & 0xffff0000u);
            a2 += __uint_as_float(v.y << 16);
            a3 += __uint_as_float(v.y & 0xffff0000u);
        }
        part[ph][c4] = a0;
        part[ph][c4 + 1] = a1;
        part[ph][c4 + 2] = a2;
        part[ph][c4 + 3] = a3;
        __syncthreads();
        const float acc = (part[0][t] + part[1][t]) + (part[2][t] + part[3][t]);
        const float z = L > 0 ? acc / (float)L : 0.f;
        float sq = z * z;
        for (int off = 32; off > 0; off >>= 1) sq += __shfl_xor(sq, off, 64);
        if ((t & 63) == 0) red[t >> 6] = sq;
        __syncthreads();
        const float nrm = sqrtf(red[0] + red[1] + red[2] + red[3]);
        e[s * 256 + t] = nrm > 0.f ? z / nrm : 0.f;
        if (t == 0 && znorm) znorm[s] = nrm;
        __syncthreads();
    }
}

// Backward of the pool and of layer 3's GELU: dz = (de - e (e . de)) / |z|,
// dU3[p][c] = dz[c] / L * gelu'(U3[p][c]) on the sequence's rows.  Blocks (s, y)
// share a sequence: each works out dz (256 channels) and takes every
// gridDim.y-th group of eight rows, a thread eight channels of one row from
// one 16-byte load.  Bound by gelu' (tanh).  1056 sequences, 312 k rows:
// 553 -> 100 us against one block and one row at a time per sequence.
// A split costs dz once more: at most PG_SPLIT blocks a sequence, and no more than
// make PG_BLOCKS in all (64 sequences of 1000 rows: 1 block 142 us, 8 27; 1056 of
// 300: 102, 4 or 8 81; 5000 of 10: 19, 8 34; 100 000 of 3: 184, 8 588).
constexpr int PG_SPLIT = 8;
constexpr int64_t PG_BLOCKS = 4096;
__global__ __launch_bounds__(256) void k_pool_grad(const float* __restrict__ de,
                                                   const float* __restrict__ e,
                                                   const float* __restrict__ znorm,
                                                   const __bf16* __restrict__ U3,
                                                   const int64_t* __restrict__ row0,
                                                   const int32_t* __restrict__ len, int64_t nseq,
                                                   __bf16* __restrict__ dU3) {
    __shared__ float red[4];
    __shared__ __align__(16) float s_dz[256];
    const int c = threadIdx.x, c8 = 8 * (c & 31), ph = c >> 5;
    for (int64_t s = blockIdx.x; s < nseq; s += gridDim.x) {
        const float ev = e[s * 256 + c], dv = de[s * 256 + c];
        float dot = ev * dv;
        for (int off = 32; off > 0; off >>= 1) dot += __shfl_xor(dot, off, 64);
        if ((c & 63) == 0) red[c >> 6] = dot;
        __syncthreads();
        const float d = red[0] + red[1] + red[2] + red[3];
        const float nrm = znorm[s];
        const int L = len[s];
        s_dz[c] = nrm > 0.f && L > 0 ? (dv - ev * d) / nrm / (float)L : 0.f;
        __syncthreads();
        float dz[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) dz[x] = s_dz[c8 + x];
        const int64_t b = row0[s];
        for (int p = 8 * blockIdx.y + ph; p < L; p += 8 * gridDim.y) {
            const int64_t o = (b + p) * 256 + c8;
            const bf16x8 u = *reinterpret_cast<const bf16x8_el*>(U3 + o);
            bf16x8 v;
#pragma unroll
            for (int x = 0; x < 8; ++x) v[x] = f2bf(dz[x] * gelu_grad(bf2f(u[x])));
            *reinterpret_cast<bf16x8_el*>(dU3 + o) = v;
        }
        __syncthreads();
    }
}

// Pair loss: for pair j, cos = e[qi] . e[ti], loss += (cos - y)^2 / npair;
// de[qi] += 2 (cos - y) / npair * e[ti] and symmetrically.  One wave per
// pair (4 channels per lane).
__global__ __launch_bounds__(256) void k_pair_loss(const float* __restrict__ e, int64_t nseq,
                                                   const int32_t* __restrict__ qi,
                                                   const int32_t* __restrict__ ti,
                                                   const float* __restrict__ y,
                                                   const float* __restrict__ wt, int64_t npair,
                                                   float* __restrict__ de, float* __restrict__ cos_out,
                                                   float* __restrict__ loss) {
    const int lane = threadIdx.x & 63;
    const int64_t j = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (j >= npair) return;
    // pairs naming a sequence outside e are skipped (and counted nowhere)
    if (qi[j] < 0 || qi[j] >= nseq || ti[j] < 0 || ti[j] >= nseq) return;
    const float* a = e + (int64_t)qi[j] * 256;
    const float* b = e + (int64_t)ti[j] * 256;
    float d = 0.f;
#pragma unroll
    for (int x = 0; x < 4; ++x) d += a[lane * 4 + x] * b[lane * 4 + x];
    for (int off = 32; off > 0; off >>= 1) d += __shfl_xor(d, off, 64);
    const float wj = wt ? wt[j] : 1.f;
    const float g = 2.f * wj * (d - y[j]) / (float)npair;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        atomicAdd(&de[(int64_t)qi[j] * 256 + lane * 4 + x], g * b[lane * 4 + x]);
        atomicAdd(&de[(int64_t)ti[j] * 256 + lane * 4 + x], g * a[lane * 4 + x]);
    }
    if (lane == 0) {
        if (cos_out) cos_out[j] = d;
        if (loss) atomicAdd(loss, wj * (d - y[j]) * (d - y[j]) / (float)npair);
    }
}

// Soft-target InfoNCE over a step's sequences: rows 0..nq-1 of e are the
// queries, rows nq..nq+nt-1 the targets.  For query q the logits are
// z_t = e_q . e_t / tau over every target and, with the target distribution
// P[q][.] (a row summing to 1, or all zero to leave the query out), the
// loss is -scale * sum_t P_qt log softmax(z)_t.  With
// G_qt = scale * (softmax(z)_t - P_qt), de_q += sum_t G_qt e_t / tau here and
// de_t += sum_q G_qt e_q / tau in k_infonce_targets.  One block per query;
// the logits live in LDS (nt <= INFONCE_MAX_T).
constexpr int INFONCE_MAX_T = 8192;

__device__ inline float block_reduce_256(float v, float* red, bool is_max) {
    for (int off = 32; off > 0; off >>= 1) {
        const float o = __shfl_xor(v, off, 64);
        v = is_max ? fmaxf(v, o) : v + o;
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return is_max ? fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]))
                  : red[0] + red[1] + red[2] + red[3];
}

__global__ __launch_bounds__(256) void k_infonce(const float* __restrict__ e, int nq, int nt,
                                                 const float* __restrict__ P, float inv_tau,
                                                 float scale, float* __restrict__ G,
                                                 float* __restrict__ de, float* __restrict__ loss) {
    __shared__ float s_q[256];
    __shared__ float s_z[INFONCE_MAX_T];
    __shared__ float red[4];
    const int q = blockIdx.x;
    const int tid = threadIdx.x;
    const float* Pq = P + (int64_t)q * nt;
    float* Gq = G + (int64_t)q * nt;
    s_q[tid] = e[(int64_t)q * 256 + tid];
    __syncthreads();
    float mx = -INFINITY, psum = 0.f;
    for (int t = tid; t < nt; t += 256) {
        const float4* r = reinterpret_cast<const float4*>(e + (int64_t)(nq + t) * 256);
        float d = 0.f;
#pragma unroll 8
        for (int x = 0; x < 64; ++x) {
            const float4 v = r[x];
            d += v.x * s_q[4 * x] + v.y * s_q[4 * x + 1] + v.z * s_q[4 * x + 2] +
                 v.w * s_q[4 * x + 3];
        }
        const float z = d * inv_tau;
        s_z[t] = z;
        mx = fmaxf(mx, z);
        psum += Pq[t];
    }
    mx = block_reduce_256(mx, red, true);
    psum = block_reduce_256(psum, red, false);
    if (!(psum > 0.f)) {  // the query takes no part: zero gradient row
        for (int t = tid; t < nt; t += 256) Gq[t] = 0.f;
        return;
    }
    float se = 0.f;
    for (int t = tid; t < nt; t += 256) se += __expf(s_z[t] - mx);
    se = block_reduce_256(se, red, false);
    const float lse = mx + __logf(se);
    float lsum = 0.f;
    for (int t = tid; t < nt; t += 256) {
        const float pt = Pq[t];
        const float z = s_z[t];
        lsum -= pt * (z - lse);
        const float g = scale * (__expf(z - lse) - pt);
        Gq[t] = g;
        s_z[t] = g;
    }
    lsum = block_reduce_256(lsum, red, false);
    if (tid == 0) atomicAdd(loss, scale * lsum);
    // de_q: thread tid owns channel tid (reads of row t are coalesced)
    float acc = 0.f;
    for (int t = 0; t < nt; ++t) acc += s_z[t] * e[(int64_t)(nq + t) * 256 + tid];
    de[(int64_t)q * 256 + tid] += acc * inv_tau;
}

// de_t += sum_q G_qt e_q / tau: one block per target, one thread per channel.
__global__ __launch_bounds__(256) void k_infonce_targets(const float* __restrict__ e, int nq,
                                                         int nt, const float* __restrict__ G,
                                                         float inv_tau, float* __restrict__ de) {
    const int t = blockIdx.x;
    const int c = threadIdx.x;
    float acc = 0.f;
    for (int q = 0; q < nq; ++q) acc += G[(int64_t)q * nt + t] * e[(int64_t)q * 256 + c];
    de[(int64_t)(nq + t) * 256 + c] += acc * inv_tau;
}

// AdamW step on fp32 parameters.
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, int64_t n, float lr, float b1, float b2, float eps,
                       float wd, float c1, float c2) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * ((mi / c1) / (sqrtf(vi / c2) + eps) + wd * p[i]);
}

// Weight layouts for the GEMMs from W[t][i][o] (fp32): forward
// Bt[o][t * Cin + i], and backward-data Bt'[i][t * Cout + o] = W[8 - t][i][o].
__global__ void k_pack_weights(const float* __restrict__ W, int Cin, int Cout,
                               __bf16* __restrict__ fwd, __bf16* __restrict__ bwd) {
    const int64_t n = (int64_t)9 * Cin * Cout;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    const int o = (int)(idx % Cout);
    const int i = (int)((idx / Cout) % Cin);
    const int t = (int)(idx / ((int64_t)Cout * Cin));
    const __bf16 v = f2bf(W[idx]);
    fwd[(int64_t)o * 9 * Cin + t * Cin + i] = v;
    if (bwd) bwd[(int64_t)i * 9 * Cout + (8 - t) * Cout + o] = v;
}

// ------------------------------------------------------------- table --

// Flat rows of a range of database sequences: codes (0..19, 20 other,
// 21 pad) and mask; sequence s of the range starts at row row0[s].
__global__ void k_db_rows(const uint8_t* __restrict__ packed, const int64_t* __restrict__ off,
                          const int32_t* __restrict__ len, int64_t s_begin, int64_t nseq,
                          const int64_t* __restrict__ row0, int max_len,
                          uint8_t* __restrict__ code, uint8_t* __restrict__ mask) {
    for (int64_t s = blockIdx.x; s < nseq; s += gridDim.x) {
        const int64_t o = off[s_begin + s];
        const int L = min(len[s_begin + s], max_len);
        const int64_t b = row0[s];
        for (int p = threadIdx.x; p < L; p += blockDim.x) {
            const int a = aa_index(packed_sym(packed, o + p));
            code[b + p] = (uint8_t)a;
            mask[b + p] = 1;
        }
    }
}

// Table rows: fp8 (e4m3) of scale * e, 256 bytes per sequence.
__global__ void k_to_fp8(const float* __restrict__ e, int64_t n, float scale,
                         uint8_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // 4 values per thread
    if (i * 4 >= n) return;
    const float4 v = *reinterpret_cast<const float4*>(e + i * 4);
    int w = __builtin_amdgcn_cvt_pk_fp8_f32(scale * v.x, scale * v.y, 0, false);
    w = __builtin_amdgcn_cvt_pk_fp8_f32(scale * v.z, scale * v.w, w, true);
    *reinterpret_cast<int*>(out + i * 4) = w;
}

// ---------------------------------------------------------- proposal --
//
// S[q][s] = sum_c T[s][c] * Q[q][c] over the fp8 table T (n x 256) and G
// query rows Q (G x 256, G a multiple of 16, at most 128), written as fp16
// to S[q * ldS + s].  A block takes PROP_ROWS consecutive table rows per
// step (4 waves x 32 PROP_SUB rows, kept in registers for every query group)
// against all G queries held in LDS.  MFMA 16x16x32 fp8: lane (r = lane %
// 16, g = lane / 16) supplies 8 bytes of row r per 32-byte K slice; result
// element i of lane (c, g) is row 4g + i, column c.  A dot product does not
// depend on the order of its terms, so the K slices are taken in the order
// that lets each lane read 16 bytes at once: slice s of lane (r, g) is bytes
// 64 (s / 2) + 16 g + 8 (s % 2) of its row, for the table and the query
// alike (16-byte loads read the table at 6.2 TB/s where 8-byte loads of the
// natural order reach 4.8).  Each group of 16 queries' 16 x PROP_ROWS scores
// goes through LDS so that the block writes every query's 2 PROP_ROWS
// contiguous bytes with 16-byte stores.
constexpr int PROP_SUB = 2;                // 32-row tiles per wave and step
constexpr int PROP_ROWS = 128 * PROP_SUB;  // table rows per block and step
constexpr int PROP_MAX_SLOTS = 32;         // output rows of a MAXQ launch
static_assert(PROP_ROWS == 256, "the MAXQ fold gives each of 256 threads one table row");

// Output rows of a MAXQ launch, as runs of query rows: query rows lo .. hi-1
// are folded, bit q of starts marks the first row of a run, and output row o
// is the maximum over the rows of run o.
struct PropSlots {
    uint64_t starts;
    int lo, hi;
};

// MAXQ: the kernel writes, per output row, the maximum of its query rows'
// scores (taken in ascending row order, as sseqs_rows_max takes them)
// instead of every query row's scores.  Thread t keeps the running maximum
// of table row t of the step in a register while it walks the query rows in
// order, and stores an output row's maximum to LDS once, when its run of
// query rows ends; no value is read back, so the fold costs one LDS read per
// query row and score.
template <bool MAXQ>
__global__ __launch_bounds__(256) void k_propose(const uint8_t* __restrict__ T, int64_t n,
                                                 const uint8_t* __restrict__ Q, int G,
                                                 PropSlots slots, int nslot,
                                                 _Float16* __restrict__ S, int64_t ldS) {
    constexpr int QROWS = MAXQ ? 64 : 128;
    __shared__ __align__(16) uint8_t sQ[QROWS * 256];
    __shared__ __align__(16) _Float16 sS[16 * PROP_ROWS];
    __shared__ __align__(16) _Float16 sM[MAXQ ? PROP_MAX_SLOTS * PROP_ROWS : 8];
    for (int i = threadIdx.x; i < G * 16; i += 256)
        reinterpret_cast<uint4*>(sQ)[i] = reinterpret_cast<const uint4*>(Q)[i];
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    // the cooperative store: thread -> (row oq of 16, scores 8 oc .. 8 oc + 7
    // of each 128-score part)
    const int oq = threadIdx.x >> 4, oc = threadIdx.x & 15;
    const bool vec = (ldS & 7) == 0 && (reinterpret_cast<uintptr_t>(S) & 15) == 0;
    for (int64_t b0 = (int64_t)blockIdx.x * PROP_ROWS; b0 < n;
         b0 += (int64_t)gridDim.x * PROP_ROWS) {
        const int64_t t0 = b0 + 32 * PROP_SUB * w;
        // this wave's 32 PROP_SUB table rows (two MFMA row tiles per 32), all
        // 8 K slices, kept for every query group
        long fa[PROP_SUB][2][8];
#pragma unroll
        for (int u = 0; u < PROP_SUB; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int64_t row = min(t0 + 32 * u + 16 * i + r, n - 1);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint4 v =
                        *reinterpret_cast<const uint4*>(T + row * 256 + 64 * j + 16 * g);
                    fa[u][i][2 * j] = (long)(((uint64_t)v.y << 32) | v.x);
                    fa[u][i][2 * j + 1] = (long)(((uint64_t)v.w << 32) | v.z);
                }
            }
        int cur_sl = -1;   // MAXQ: the output row of the run being folded
        _Float16 cur = 0;  // and its running maximum (table row threadIdx.x)
        for (int q0 = 0; q0 < G; q0 += 16) {
            f32x4 acc[PROP_SUB][2];
#pragma unroll
            for (int u = 0; u < PROP_SUB; ++u)
#pragma unroll
                for (int i = 0; i < 2; ++i) acc[u][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const long fb = *reinterpret_cast<const long*>(
                    &sQ[(q0 + r) * 256 + 64 * (s >> 1) + 16 * g + 8 * (s & 1)]);
#pragma unroll
                for (int u = 0; u < PROP_SUB; ++u)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        acc[u][i] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(fa[u][i][s], fb,
                                                                               acc[u][i], 0, 0, 0);
            }
            // rows 4g .. 4g+3 of each row tile are consecutive: one 8-byte LDS store
#pragma unroll
            for (int u = 0; u < PROP_SUB; ++u)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    union {
                        _Float16 h[4];
                        uint2 u2;
                    } v;
#pragma unroll
                    for (int x = 0; x < 4; ++x) v.h[x] = (_Float16)acc[u][i][x];
                    *reinterpret_cast<uint2*>(
                        &sS[r * PROP_ROWS + 32 * PROP_SUB * w + 32 * u + 16 * i + 4 * g]) = v.u2;
                }
            // MAXQ: thread t folds table row t, which its own wave wrote (the
            // wave's rows are 32 PROP_SUB w .. + 32 PROP_SUB), and a wave's LDS
            // accesses complete in order: the waves need not wait for each other
            if constexpr (MAXQ)
                lds_wave_fence();
            else
                __syncthreads();
            if constexpr (MAXQ) {
                const int c = threadIdx.x;
                _Float16 x[16];
#pragma unroll
                for (int q = 0; q < 16; ++q) x[q] = sS[q * PROP_ROWS + c];
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const int row = q0 + q;  // the run structure is uniform
                    if (row < slots.lo || row >= slots.hi) continue;
                    if ((slots.starts >> row) & 1) {  // a run starts: the last one is done
                        if (cur_sl >= 0 && cur_sl < PROP_MAX_SLOTS) sM[cur_sl * PROP_ROWS + c] = cur;
                        ++cur_sl;
                        cur = x[q];
                    } else {
                        cur = x[q] > cur ? x[q] : cur;
                    }
                }
            } else {
#pragma unroll
                for (int part = 0; part < PROP_SUB; ++part) {
                    const int64_t row = b0 + 128 * part + 8 * oc;
                    _Float16* dst = S + (int64_t)(q0 + oq) * ldS + row;
                    const _Float16* src = &sS[oq * PROP_ROWS + 128 * part + 8 * oc];
                    if (vec && row + 8 <= n) {
                        *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(src);
                    } else {
                        for (int x = 0; x < 8; ++x)
                            if (row + x < n) dst[x] = src[x];
                    }
                }
            }
            if constexpr (MAXQ)
                lds_wave_fence();  // the fold's reads before the next tile's writes
            else
                __syncthreads();
        }
        if constexpr (MAXQ) {
            if (cur_sl >= 0 && cur_sl < PROP_MAX_SLOTS) sM[cur_sl * PROP_ROWS + threadIdx.x] = cur;
            __syncthreads();
            // every output row's PROP_ROWS scores, 16 bytes per thread and pass
            for (int e = threadIdx.x; e < nslot * (PROP_ROWS / 8); e += 256) {
                const int sl = e / (PROP_ROWS / 8), c8 = e % (PROP_ROWS / 8);
                const int64_t row = b0 + 8 * c8;
                _Float16* dst = S + (int64_t)sl * ldS + row;
                const _Float16* src = &sM[sl * PROP_ROWS + 8 * c8];
                if (vec && row + 8 <= n) {
                    *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(src);
                } else {
                    for (int x = 0; x < 8; ++x)
                        if (row + x < n) dst[x] = src[x];
                }
            }
            __syncthreads();
        }
    }
}

// out[j] = max over r < nrows of S[r * ld + j], j < n (fp16; ld a multiple
// of 8 and S, out 16-byte aligned: 8 scores per thread and step).
__global__ __launch_bounds__(256) void k_rows_max(const _Float16* __restrict__ S, int64_t ld,
                                                  int nrows, int64_t n,
                                                  _Float16* __restrict__ out) {
    const int64_t n8 = n / 8;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c * 8 < n;
         c += (int64_t)gridDim.x * blockDim.x) {
        if (c < n8) {
            uint4 v = *reinterpret_cast<const uint4*>(S + c * 8);
            _Float16* m = reinterpret_cast<_Float16*>(&v);
            for (int r = 1; r < nrows; ++r) {
                uint4 w = *reinterpret_cast<const uint4*>(S + r * ld + c * 8);
                const _Float16* x = reinterpret_cast<const _Float16*>(&w);
#pragma unroll
                for (int e = 0; e < 8; ++e) m[e] = x[e] > m[e] ? x[e] : m[e];
            }
            *reinterpret_cast<uint4*>(out + c * 8) = v;
        } else {
            for (int64_t j = c * 8; j < n; ++j) {
                _Float16 m = S[j];
                for (int r = 1; r < nrows; ++r) m = S[r * ld + j] > m ? S[r * ld + j] : m;
                out[j] = m;
            }
        }
    }
}

}  // namespace sseqs

using namespace sseqs;

// ---------------------------------------------------------------- C ABI --

template <int CIN, int BN, int EPI, int WM, int WN>
static void launch_conv_tiles(const ConvArgs& a, hipStream_t stream) {
    const int64_t slots = ceil_div(ceil_div(a.M, 64 * WM - 8), 8) * (a.N / BN);
    hipLaunchKernelGGL((k_conv_gemm<CIN, BN, EPI, WM, WN>), dim3((unsigned)(8 * slots)),
                       dim3(64 * WM * WN), 0, stream, a);
}

template <int CIN, int EPI>
static void launch_conv_cin(const ConvArgs& a, hipStream_t stream) {
    constexpr int WM = CIN == 256 ? 2 : 4, WN = CIN == 256 ? 2 : 1;  // A: at most 64 KiB
    const int64_t rows = a.M / (64 * WM - 8);
    if (a.N % 128 == 0 && rows * (a.N / 128) >= CONV_WIDE)
        launch_conv_tiles<CIN, 128, EPI, WM, WN>(a, stream);
    else if (CIN != 256 && rows * (a.N / 64) >= CONV_WIDE)
        launch_conv_tiles<CIN, 64, EPI, WM, WN>(a, stream);
    else
        launch_conv_tiles<CIN, 64, EPI, 2, CIN == 256 ? 2 : 1>(a, stream);
}

template <int EPI>
static void launch_conv(const ConvArgs& a, hipStream_t stream) {
    // nine whole rows of the encoder's widths, and outputs that take 16-byte accesses
    const uintptr_t out = (uintptr_t)a.U | (uintptr_t)a.Y | (uintptr_t)a.Uprev |
                          (uintptr_t)a.bias | (uintptr_t)a.Yf;
    const bool whole = a.K == 9 * a.lda && !(out & 15);
    if (whole && a.lda == 64) launch_conv_cin<64, EPI>(a, stream);
    else if (whole && a.lda == 128) launch_conv_cin<128, EPI>(a, stream);
    else if (whole && a.lda == 256) launch_conv_cin<256, EPI>(a, stream);
    else
        hipLaunchKernelGGL((k_conv_any<EPI>), dim3((unsigned)(a.M / GM), (unsigned)(a.N / 64)),
                           dim3(256), 0, stream, a);
}

extern "C" int sseqs_enc_conv(const void* A, int lda, const void* Bt, int64_t M, int N, int K,
                              const float* bias, const uint8_t* mask, void* U, void* Y,
                              const void* Uprev, float* Yf, int epi, hipStream_t stream) {
    if (M <= 0 || M % GM) return fail(-1, "enc_conv: M must be a positive multiple of 128");
    if (K <= 0 || K % GK) return fail(-1, "enc_conv: K must be a positive multiple of 32");
    if (N % 64) return fail(-1, "enc_conv: N must be a multiple of 64");
    if (M / GM > 0x7fffffffLL) return fail(-1, "enc_conv: too many rows");
    if (epi == EPI_FWD && (!Y || !bias)) return fail(-1, "enc_conv: forward needs Y and bias");
    if (epi == EPI_BWD_GELU && (!Y || !Uprev)) return fail(-1, "enc_conv: backward needs Y and Uprev");
    if (epi == EPI_BWD_F32 && !Yf) return fail(-1, "enc_conv: backward to the input needs Yf");
    const ConvArgs a{static_cast<const __bf16*>(A), lda, static_cast<const __bf16*>(Bt), M, N, K,
                     bias, mask, static_cast<__bf16*>(U), static_cast<__bf16*>(Y),
                     static_cast<const __bf16*>(Uprev), Yf};
    switch (epi) {
    case EPI_FWD: launch_conv<EPI_FWD>(a, stream); break;
    case EPI_BWD_GELU: launch_conv<EPI_BWD_GELU>(a, stream); break;
    case EPI_BWD_F32: launch_conv<EPI_BWD_F32>(a, stream); break;
    default: return fail(-1, "enc_conv: unknown epilogue");
    }
    return check_launch("enc_conv");
}

// Blocks along the rows.  A stage takes a block 1.26 us, the blocks' additions
// 0.13 us for each 64 x 64 tile of dW and slice, one slice after the other on the
// same addresses: 1.26 stages / slices + 0.13 tiles slices is least at 3.1
// sqrt(stages / tiles).  128 -> 256 channels, against filling all WG_FILL places for
// any number of rows: 2048 rows 34 -> 14 us, 20 000 rows 70 -> 41, 100 000 rows 104 -> 97;
// from about 220 000 rows on the places are the bound.
static int64_t wg_slices(int64_t stages, int64_t tiles) {
    const int64_t s = (int64_t)(3.1 * sqrt((double)stages / (double)tiles) + 0.5);
    return std::max<int64_t>(1, std::min(s, WG_FILL / tiles));
}

extern "C" int sseqs_enc_wgrad(const void* X, int Cin, const void* dU, int Cout, int64_t M,
                               float* dW, hipStream_t stream) {
    if (M <= 0 || Cin % 64 || Cout % 64) return fail(-1, "enc_wgrad: bad sizes");
    if (ceil_div(M, 2048) > 65535) return fail(-1, "enc_wgrad: at most 65535 * 2048 rows");
    const int64_t tiles = (int64_t)(Cin / 64) * (Cout / 64), stages = ceil_div(M, WP);
    if (tiles == 0) return 0;
    const int64_t per = std::max(ceil_div(stages, wg_slices(stages, tiles)), ceil_div(stages, 65535));
    const dim3 grid((unsigned)(Cin / 64), (unsigned)(Cout / 64), (unsigned)ceil_div(stages, per));
    hipLaunchKernelGGL(M % WP ? k_conv_wgrad<true> : k_conv_wgrad<false>, grid, dim3(256), 0, stream,
                       static_cast<const __bf16*>(X), Cin, static_cast<const __bf16*>(dU), Cout, M, per, dW);
    return check_launch("enc_wgrad");
}

extern "C" int sseqs_enc_bias_grad(const void* dU, int C, int64_t M, float* db,
                                   hipStream_t stream) {
    if (M <= 0) return 0;
    if (C % 64) return fail(-1, "enc_bias_grad: C must be a multiple of 64");
    hipLaunchKernelGGL(k_colsum, dim3((unsigned)ceil_div(M, CS_ROWS), (unsigned)(C / 64)), dim3(256),
                       0, stream, static_cast<const __bf16*>(dU), C, M, db);
    return check_launch("enc_bias_grad");
}

extern "C" int sseqs_enc_embed(const uint8_t* code, int64_t M, const float* E, void* x0,
                               hipStream_t stream) {
    if (M <= 0) return 0;
    hipLaunchKernelGGL(k_embed, dim3((unsigned)ceil_div(M * 8, 256)), dim3(256), 0, stream, code,
                       M, E, static_cast<__bf16*>(x0));
    return check_launch("enc_embed");
}

extern "C" int sseqs_enc_embed_grad(const uint8_t* code, int64_t M, const float* dx0, float* dE,
                                    hipStream_t stream) {
    if (M <= 0) return 0;
    hipLaunchKernelGGL(k_embed_grad, dim3((unsigned)std::min<int64_t>(256, ceil_div(M, EG_WAVES * EG_ROWS))),
                       dim3(64 * EG_WAVES), 0, stream, code, M, dx0, dE);
    return check_launch("enc_embed_grad");
}

extern "C" int sseqs_enc_pool(const void* h3, const int64_t* row0, const int32_t* len,
                              int64_t nseq, float* e, float* znorm, hipStream_t stream) {
    if (nseq <= 0) return 0;
    hipLaunchKernelGGL(k_pool, dim3(grid_cap(nseq, 1)), dim3(256), 0, stream,
                       static_cast<const __bf16*>(h3), row0, len, nseq, e, znorm);
    return check_launch("enc_pool");
}

extern "C" int sseqs_enc_pool_grad(const float* de, const float* e, const float* znorm,
                                   const void* U3, const int64_t* row0, const int32_t* len,
                                   int64_t nseq, void* dU3, hipStream_t stream) {
    if (nseq <= 0) return 0;
    const unsigned split = (unsigned)std::min<int64_t>(PG_SPLIT, ceil_div(PG_BLOCKS, nseq));
    hipLaunchKernelGGL(k_pool_grad, dim3(grid_cap(nseq, 1), split), dim3(256), 0, stream, de, e, znorm,
                       static_cast<const __bf16*>(U3), row0, len, nseq, static_cast<__bf16*>(dU3));
    return check_launch("enc_pool_grad");
}

extern "C" int sseqs_enc_pair_loss(const float* e, int64_t nseq, const int32_t* qi,
                                   const int32_t* ti, const float* y, const float* w,
                                   int64_t npair, float* de, float* cos_out, float* loss,
                                   hipStream_t stream) {
    if (npair <= 0) return 0;
    hipLaunchKernelGGL(k_pair_loss, dim3((unsigned)ceil_div(npair, 4)), dim3(256), 0, stream, e,
                       nseq, qi, ti, y, w, npair, de, cos_out, loss);
    return check_launch("enc_pair_loss");
}

extern "C" int sseqs_enc_infonce(const float* e, int nq, int nt, const float* P, float tau,
                                 float scale, float* G, float* de, float* loss,
                                 hipStream_t stream) {
    if (nq <= 0 || nt <= 0) return fail(-1, "enc_infonce: need at least one query and one target");
    if (nt > INFONCE_MAX_T) return fail(-1, "enc_infonce: more than 8192 targets");
    if (!(tau > 0.f)) return fail(-1, "enc_infonce: tau must be positive");
    hipLaunchKernelGGL(k_infonce, dim3(nq), dim3(256), 0, stream, e, nq, nt, P, 1.f / tau, scale,
                       G, de, loss);
    if (int r = check_launch("enc_infonce")) return r;
    hipLaunchKernelGGL(k_infonce_targets, dim3(nt), dim3(256), 0, stream, e, nq, nt, G, 1.f / tau,
                       de);
    return check_launch("enc_infonce_targets");
}

extern "C" int sseqs_enc_adam(float* p, const float* g, float* m, float* v, int64_t n, float lr,
                              float b1, float b2, float eps, float wd, int step,
                              hipStream_t stream) {
    if (n <= 0) return 0;
    if (step < 1) return fail(-1, "enc_adam: step counts from 1");
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, stream, p, g, m,
                       v, n, lr, b1, b2, eps, wd, c1, c2);
    return check_launch("enc_adam");
}

extern "C" int sseqs_enc_pack_weights(const float* W, int Cin, int Cout, void* fwd, void* bwd,
                                      hipStream_t stream) {
    const int64_t n = (int64_t)9 * Cin * Cout;
    hipLaunchKernelGGL(k_pack_weights, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, stream, W,
                       Cin, Cout, static_cast<__bf16*>(fwd), static_cast<__bf16*>(bwd));
    return check_launch("enc_pack_weights");
}

extern "C" int sseqs_enc_db_rows(const uint8_t* packed, const int64_t* seq_off,
                                 const int32_t* seq_len, int64_t s_begin, int64_t nseq,
                                 const int64_t* row0, int max_len, uint8_t* code, uint8_t* mask,
                                 hipStream_t stream) {
    if (nseq <= 0) return 0;
    hipLaunchKernelGGL(k_db_rows, dim3(grid_cap(nseq, 1)), dim3(256), 0, stream, packed, seq_off,
                       seq_len, s_begin, nseq, row0, max_len, code, mask);
    return check_launch("enc_db_rows");
}

extern "C" int sseqs_enc_to_fp8(const float* e, int64_t n, float scale, uint8_t* out,
                                hipStream_t stream) {
    if (n <= 0) return 0;
    if (n % 4) return fail(-1, "enc_to_fp8: n must be a multiple of 4");
    hipLaunchKernelGGL(k_to_fp8, dim3((unsigned)ceil_div(n / 4, 256)), dim3(256), 0, stream, e, n,
                       scale, out);
    return check_launch("enc_to_fp8");
}

extern "C" int sseqs_rows_max(const void* S, int64_t ld, int nrows, int64_t n, void* out,
                              hipStream_t stream) {
    if (n <= 0) return 0;
    if (nrows < 1) return fail(-1, "rows_max: need at least one row");
    if (ld < n || ld % 8) return fail(-1, "rows_max: ld must be >= n and a multiple of 8");
    if ((reinterpret_cast<uintptr_t>(S) | reinterpret_cast<uintptr_t>(out)) & 15)
        return fail(-1, "rows_max: S and out must be 16-byte aligned");
    hipLaunchKernelGGL(k_rows_max, dim3(grid_cap(ceil_div(n, 8), 256)), dim3(256), 0, stream,
                       static_cast<const _Float16*>(S), ld, nrows, n, static_cast<_Float16*>(out));
    return check_launch("rows_max");
}

extern "C" int sseqs_propose(const uint8_t* table, int64_t n, const uint8_t* q8, int G,
                             void* scores, int64_t ld, hipStream_t stream) {
    if (n <= 0) return 0;
    if (G <= 0 || G % 16 || G > 128) return fail(-1, "propose: G must be 16..128, a multiple of 16");
    if (ld < n) return fail(-1, "propose: ld smaller than n");
    if ((reinterpret_cast<uintptr_t>(table) | reinterpret_cast<uintptr_t>(q8)) & 15)
        return fail(-1, "propose: table and query rows must be 16-byte aligned");
    const unsigned grid =
        (unsigned)(ceil_div(n, PROP_ROWS) < 8192 ? ceil_div(n, PROP_ROWS) : 8192);
    hipLaunchKernelGGL(k_propose<false>, dim3(grid), dim3(256), 0, stream, table, n, q8, G,
                       PropSlots{}, 0, static_cast<_Float16*>(scores), ld);
    return check_launch("propose");
}

extern "C" int sseqs_propose_max(const uint8_t* table, int64_t n, const uint8_t* q8, int G,
                                 const int32_t* row_off, int nslot, void* scores, int64_t ld,
                                 hipStream_t stream) {
    if (n <= 0) return 0;
    if (G <= 0 || G % 16 || G > 64) return fail(-1, "propose_max: G must be 16..64, a multiple of 16");
    if (nslot < 1 || nslot > PROP_MAX_SLOTS) return fail(-1, "propose_max: 1..32 output rows");
    if (!row_off) return fail(-1, "propose_max: no row offsets");
    if (row_off[0] < 0 || row_off[nslot] > G)
        return fail(-1, "propose_max: row offsets outside the G query rows");
    PropSlots sl{0, row_off[0], row_off[nslot]};
    for (int o = 0; o < nslot; ++o) {
        if (row_off[o + 1] <= row_off[o])
            return fail(-1, "propose_max: row offsets must increase (no empty output row)");
        sl.starts |= 1ull << row_off[o];
    }
    if (ld < n) return fail(-1, "propose_max: ld smaller than n");
    if ((reinterpret_cast<uintptr_t>(table) | reinterpret_cast<uintptr_t>(q8)) & 15)
        return fail(-1, "propose_max: table and query rows must be 16-byte aligned");
    const unsigned grid =
        (unsigned)(ceil_div(n, PROP_ROWS) < 8192 ? ceil_div(n, PROP_ROWS) : 8192);
    hipLaunchKernelGGL(k_propose<true>, dim3(grid), dim3(256), 0, stream, table, n, q8, G, sl,
                       nslot, static_cast<_Float16*>(scores), ld);
    return check_launch("propose_max");
}
