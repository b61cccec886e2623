// Affine DP + traceback for a3m rows (replaces the Triton kernels
// sw_diag_batch_affine / backtrack_kernel_batched_affine, sseqs/sw.py:408-768).
//
// DP (i = query 1..Lq, j = target 1..T, zero borders, -5 for non-residues):
//   M  = s + H(i-1,j-1)
//   Ix = max(H(i-1,j)-o, (i-1==0 ? -16384 : Ix(i-1,j)) - e)
//   Iy = max(H(i,j-1)-o, (j-1==0 ? -16384 : Iy(i,j-1)) - e)
//   H  = max(0, M, Ix, Iy)
// The reference stores the three int16 matrices and re-derives the move at
// every traceback cell (H == M -> diagonal, else H == Ix -> up, else
// H == Iy -> left, stop at H == 0).  Those comparisons depend only on the
// cell, so two bits per cell (the move) are stored instead of six bytes.
//
// One wave per target sweeps anti-diagonals of query strips (one row per lane
// in k_backtrack_global, two in k_backtrack) and then follows the moves from
// the end cell, the first cell in row-major order that holds the maximum
// (sseqs/sw.py:620-637).
#include "common.h"

namespace sseqs {

constexpr int BT_NEG = -16384;  // VERY_NEGATIVE_SCORE of sseqs/sw.py:517

// Same DP and traceback for targets too long for k_backtrack's LDS row
// buffer: one move byte per cell and the strip boundary row in global memory.
__global__ __launch_bounds__(64) void k_backtrack_global(
    const uint8_t* __restrict__ query, int Lq, const uint8_t* __restrict__ targets,
    const int64_t* __restrict__ t_off, const int32_t* __restrict__ t_len,
    const int64_t* __restrict__ cell_off, int B, int go, int ge, int A, uint8_t* __restrict__ out_q,
    uint8_t* __restrict__ out_t, int32_t* __restrict__ info, uint8_t* __restrict__ dirs_all,
    int2* __restrict__ rowbuf_all, Blosum bl) {
    __shared__ int8_t s_bl[400];
    const int lane = threadIdx.x;
    for (int i = lane; i < 400; i += 64) s_bl[i] = bl.v[i];
    __syncthreads();
    const int b = blockIdx.x;
    if (b >= B) return;
    const int T = t_len[b];
    const uint8_t* tq = targets + t_off[b];
    uint8_t* dirs = dirs_all + cell_off[b];
    volatile int* rb = reinterpret_cast<int*>(rowbuf_all + (Lq > 0 ? cell_off[b] / Lq : 0));

    int best = 0;
    int64_t bestpos = INT64_MAX;
    if (Lq > 0 && T > 0) {
        for (int i0 = 0; i0 < Lq; i0 += 64) {
            const int i = i0 + lane + 1;  // 1-based row of this lane
            const bool row_ok = i <= Lq;
            const int qa = row_ok ? aa_index(query[i - 1]) : 20;
            int Hleft = 0, Yleft = BT_NEG;   // H(i,0) = 0; Iy(i,0) treated as -16384
            int diagH = 0;                   // H(i-1, j-1), starts at H(i-1, 0) = 0
            int sendH = 0, sendX = BT_NEG;
            const int steps = T + 63;
            for (int s = 0; s < steps; ++s) {
                const int j = s - lane + 1;
                int upH = __shfl_up(sendH, 1, 64);
                int upX = __shfl_up(sendX, 1, 64);
                if (lane == 0) {
                    if (j >= 1 && j <= T && i0 > 0) {
                        upH = rb[2 * (j - 1)];
                        upX = rb[2 * (j - 1) + 1];
                    } else {
                        upH = 0;
                        upX = BT_NEG;
                    }
                }
                if (j >= 1 && j <= T && row_ok) {
                    const int tb = aa_index(tq[j - 1]);
                    const int sc = (qa < 20 && tb < 20) ? (int)s_bl[qa * 20 + tb] : -5;
                    const int m = sc + diagH;
                    const int x = max(upH - go, (i == 1 ? BT_NEG : upX) - ge);
                    const int y = max(Hleft - go, (j == 1 ? BT_NEG : Yleft) - ge);
                    const int h = max(0, max(m, max(x, y)));
                    const uint8_t d = h == 0 ? 0 : (h == m ? 1 : (h == x ? 2 : 3));
                    const int64_t pos = (int64_t)(i - 1) * T + (j - 1);
                    dirs[pos] = d;
                    if (h > best || (h == best && pos < bestpos)) {
                        best = h;
                        bestpos = pos;
                    }
                    Hleft = h;
                    Yleft = y;
                    sendH = h;
                    sendX = x;
                    if (lane == 63) {
                        rb[2 * (j - 1)] = h;
                        rb[2 * (j - 1) + 1] = x;
                    }
                } else if (j < 1) {
                    sendH = 0;
                    sendX = BT_NEG;
                }
                diagH = upH;
            }
            __threadfence();
        }
        // best value, first row-major position among equals
        for (int off = 32; off > 0; off >>= 1) {
            int ob = __shfl_xor(best, off, 64);
            int64_t op = __shfl_xor(bestpos, off, 64);
            if (ob > best || (ob == best && op < bestpos)) {
                best = ob;
                bestpos = op;
            }
        }
    }
    if (lane != 0) return;
    int32_t* inf = info + (int64_t)b * 6;
    int n = 0, ci = -1, cj = -1, ei = -1, ej = -1;
    if (best > 0 && Lq > 0 && T > 0) {
        ei = (int)(bestpos / T) + 1;
        ej = (int)(bestpos % T) + 1;
        int i = ei, j = ej;
        int w = A - 1;
        const volatile uint8_t* vd = dirs;
        while (i > 0 && j > 0 && w >= 0) {
            const uint8_t d = vd[(int64_t)(i - 1) * T + (j - 1)];
            if (d == 0) break;
            uint8_t qc, tc;
            if (d == 1) {
                qc = query[i - 1];
                tc = tq[j - 1];
                --i;
                --j;
            } else if (d == 2) {
                qc = query[i - 1];
                tc = '-';
                --i;
            } else {
                qc = '-';
                tc = tq[j - 1];
                --j;
            }
            out_q[(int64_t)b * A + w] = qc;
            out_t[(int64_t)b * A + w] = tc;
            --w;
            ++n;
        }
        ci = i;
        cj = j;
    }
    if (n > 0) {
        inf[0] = n;
        inf[1] = ci;
        inf[2] = ei - 1;
        inf[3] = cj;
        inf[4] = ej - 1;
    } else {
        inf[0] = 0;
        inf[1] = -1;
        inf[2] = -1;
        inf[3] = -1;
        inf[4] = -1;
    }
    inf[5] = best;
}

// Two 16-bit lanes per register: low half the strip's upper row of a lane,
// high half its lower row.
typedef short bt_i16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short bt_u16x2 __attribute__((ext_vector_type(2)));
__device__ inline bt_i16x2 bt_v(uint32_t u) { return __builtin_bit_cast(bt_i16x2, u); }
__device__ inline uint32_t bt_u(bt_i16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ inline bt_i16x2 bt_max(bt_i16x2 a, bt_i16x2 b) { return __builtin_elementwise_max(a, b); }

// Longest target of k_backtrack (its boundary row and target codes in LDS);
// longer ones take k_backtrack_global.  Cells are 16 bits as in the definition:
// scores wrap past 32767 (11 a residue: from 2979 residues on), as the
// reference's int16 matrices do; k_backtrack_global's 32-bit cells do not.
constexpr int BT_MAX_T = 5416;
constexpr uint32_t BT_NEG2 = 0xC000C000u;  // BT_NEG in both halves
constexpr int BT_LETTERS = 22;             // 20 residues, 20 any other letter, 21 outside the target
constexpr int BT_PAD = 21;
constexpr int BT_TAG_MAX_LEN = 744;   // 4 * 11 * 744 + 3 < 2^15
constexpr int BT_TAG_MAX_GAP = 1024;  // gap parameters of the tagged cells (4 * 1024 above BT_NEG)
// Dynamic LDS of k_backtrack: score pairs | strip boundary | BLOSUM62 |
// target codes.
__host__ __device__ inline int bt_rb_words(int tcap) { return 128 + ((tcap + 7) & ~7) + 144; }
__host__ __device__ inline int bt_lds_bytes(int tcap) {
    return BT_LETTERS * 256 + 4 * bt_rb_words(tcap) + 400 + ((128 + tcap + 160 + 15) & ~15);
}

// Move words of target b start at byte 32 * NS * (cell_off[b] / Lq + 128 b),
// NS = ceil(Lq / 128) strips of 32 * (T + 128) bytes.
//
// One wave per target.  The query is processed in strips of 128 rows; lane l
// owns rows 128k + 2l + 1 (the "a" row, low halves) and 128k + 2l + 2 (the
// "b" row, high halves) and at step s handles column s - 2l + 1 of its a row
// and one column less of its b row, both cells in packed 16-bit arithmetic.
// The a row takes H and Ix of the cell above from lane l-1's b row through one
// DPP wave shift per step, the b row from the lane's own a row one step
// earlier.  Eight steps form a block: the strip's last row (lane 63's b row)
// enters and leaves LDS, and the moves leave for memory, once per block.
//
// The kernel is bound by the instructions of one step, few waves being in
// flight (one per target), so a step does as little as the two cells allow:
// * Scores: tab[letter][lane] holds the scores of both rows of a lane against
//   a letter, written once per strip, so a step reads one word without bank
//   conflicts, a block ahead (the target is known; only H is a recurrence).
// * Moves (TAG): cells hold 4 times the score plus, in the two low bits, the
//   move's rank 3 stop (0), 2 diagonal, 1 up, 0 left, and the maximum picks
//   value and move at once, with the ties of the definition.  A lane keeps
//   the bits of eight steps of both rows in one word and the wave stores 256
//   contiguous bytes per block (word 64 (s / 8) + 63 - l of the strip: the
//   last, partial block holds cells only of the last lanes, so that its words
//   end within the strip's bytes).
// * Borders (TAG): columns outside the target and rows outside the query score
//   BT_NEG.  With gap parameters >= 0 such cells hold 0 before the target and
//   never more than the first valid cell of their value after it, and Iy = -o
//   in column 0 gives column 1 the value of the border, so no cell is masked.
// Without TAG (16 bits do not hold 4 x the scores, or odd gap parameters)
// cells are masked and the moves come from comparisons.  4096 homologs at 200
// residues: 927 -> 289 us against a wave with four ballots, masks and byte reads
// per step.
//
// End cell: the first cell in row-major order that holds the maximum
// (sseqs/sw.py:620-637).  Traceback: lane x reads the move of the cell x
// diagonal steps back, so one round takes the whole run of diagonal moves
// and the gap move that ends it.
// Targets longer than tcap are rejected (info all -2).
template <bool TAG>
__global__ __launch_bounds__(64) void k_backtrack(
    const uint8_t* __restrict__ query, int Lq, const uint8_t* __restrict__ targets,
    const int64_t* __restrict__ t_off, const int32_t* __restrict__ t_len,
    const int64_t* __restrict__ cell_off, int go, int ge, int A, uint8_t* __restrict__ out_q,
    uint8_t* __restrict__ out_t, int32_t* __restrict__ info, uint32_t* __restrict__ moves_all,
    int tcap, Blosum bl) {
    extern __shared__ __align__(16) uint8_t smem[];
    uint32_t* tab = reinterpret_cast<uint32_t*>(smem);
    uint32_t* rb = tab + BT_LETTERS * 64;
    int8_t* s_bl = reinterpret_cast<int8_t*>(rb + bt_rb_words(tcap));
    uint8_t* tq = reinterpret_cast<uint8_t*>(s_bl + 400);
    const int lane = threadIdx.x;
    const int b = blockIdx.x;
    const int T = t_len[b];
    int32_t* inf = info + (int64_t)b * 6;
    if (T > tcap) {
        if (lane < 6) inf[lane] = -2;
        return;
    }
    constexpr int SC = TAG ? 4 : 1;
    constexpr uint32_t XNEG = TAG ? 0xC001u : 0xC000u;
    for (int i = lane; i < 400; i += 64) s_bl[i] = bl.v[i];
    const uint8_t* tg = targets + t_off[b];
    // codes of columns -127 .. T + 160; rb[128 + j - 1]: (H, Ix) of the row
    // above the strip in column j, the border for the first strip
    for (int j = lane; j < 128 + T + 160; j += 64)
        tq[j] = j >= 128 && j < 128 + T ? (uint8_t)aa_index(tg[j - 128]) : (uint8_t)BT_PAD;
    for (int j = lane; j < 128 + ((T + 7) & ~7) + 144; j += 64) rb[j] = XNEG;
    __syncthreads();

    const int NS = (Lq + 127) >> 7;
    const int RS = T + 128;
    const int NB = (T + 127 + 7) >> 3;  // blocks of eight steps
    uint32_t* moves = moves_all + (Lq > 0 ? 8LL * NS * (cell_off[b] / Lq + 128LL * b) : 0);
    const bt_i16x2 GO = bt_v((uint32_t)(uint16_t)(SC * go) * 0x10001u);
    const bt_i16x2 GE = bt_v((uint32_t)(uint16_t)(SC * ge) * 0x10001u);
    const bt_i16x2 GOX = bt_v((uint32_t)(uint16_t)(SC * go - (TAG ? 1 : 0)) * 0x10001u);
    const bt_i16x2 FLOOR = bt_v(TAG ? 0x00030003u : 0u);
    const bt_i16x2 ONE = bt_v(0x00010001u);
    int best = 0, bi = 0, bj = 0;  // this lane's first maximum, in (row, column) order
    if (Lq > 0 && T > 0) {
        for (int k = 0; k < NS; ++k) {
            const int ia = 128 * k + 2 * lane + 1, ib = ia + 1;
            const bool oka = ia <= Lq, okb = ib <= Lq;
            const int qa = oka ? aa_index(query[ia - 1]) : 20;
            const int qb = okb ? aa_index(query[ib - 1]) : 20;
#pragma unroll 2
            for (int t = 0; t < BT_LETTERS; ++t) {
                int va = qa < 20 && t < 20 ? (int)s_bl[qa * 20 + t] : -5;
                int vb = qb < 20 && t < 20 ? (int)s_bl[qb * 20 + t] : -5;
                va = TAG && (t == BT_PAD || !oka) ? BT_NEG : SC * va;
                vb = TAG && (t == BT_PAD || !okb) ? BT_NEG : SC * vb;
                const int rank = TAG ? 2 : 0;
                tab[t * 64 + lane] = ((uint32_t)(va + rank) & 0xffffu) | ((uint32_t)(vb + rank) << 16);
            }
            __syncthreads();
            // state of both rows: H (the cell to the left, and what the next
            // lane sees above), Ix, Iy; the cell above-left (diagonal)
            uint32_t H = 0, X = XNEG * 0x10001u, Y = BT_NEG2, diag = 0;
            uint32_t bv = 0, bs = 0;  // both rows' maxima and the steps they were reached at
            const uint8_t* tl = tq + 128 - 2 * lane;  // code of step s's a-row column
            // the code c of a step gives byte address 256 c + 4 lane of tab
            const uint32_t lane4 = 4u * (uint32_t)lane;
            uint32_t P[8], L[4], R[8];
            uint32_t last = 0;  // score pair of the previous step
#define BT_LETTER_LOAD(q)                                                                        \
    do {                                                                                         \
        _Pragma("unroll") for (int u = 0; u < 4; ++u) L[u] =                                     \
            *reinterpret_cast<const uint16_t*>(tl + 8 * (q) + 2 * u);                            \
    } while (0)
#define BT_SCORE_LOAD(dst)                                                                       \
    do {                                                                                         \
        _Pragma("unroll") for (int u = 0; u < 8; ++u) dst[u] = *reinterpret_cast<const uint32_t*>( \
            smem + __builtin_amdgcn_perm(L[u >> 1], lane4, u & 1 ? 0x0c0c0500u : 0x0c0c0400u));  \
    } while (0)
#define BT_ROW_LOAD(dst, q)                                                                      \
    do {                                                                                         \
        const uint4 r0 = *reinterpret_cast<const uint4*>(rb + 128 + 8 * (q));                    \
        const uint4 r1 = *reinterpret_cast<const uint4*>(rb + 132 + 8 * (q));                    \
        dst[0] = r0.x, dst[1] = r0.y, dst[2] = r0.z, dst[3] = r0.w;                              \
        dst[4] = r1.x, dst[5] = r1.y, dst[6] = r1.z, dst[7] = r1.w;                              \
    } while (0)
            BT_LETTER_LOAD(0);
            BT_SCORE_LOAD(P);
            BT_LETTER_LOAD(1);
            BT_ROW_LOAD(R, 0);
            uint32_t* mv = moves + (int64_t)k * RS * 8 + 63 - lane;
            for (int q = 0; q < NB; ++q) {
                uint32_t Pn[8], Rn[8], O[8], acc = 0;
                BT_SCORE_LOAD(Pn);
                BT_LETTER_LOAD(q + 2);
                BT_ROW_LOAD(Rn, q + 1);
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const uint32_t sc = (P[u] & 0xffffu) | (last & 0xffff0000u);
                    last = P[u];
                    // the cells above: the a row's from lane l-1's b row (lane 0:
                    // the previous strip's last row), the b row's from its a row
                    const uint32_t hin = (uint32_t)__builtin_amdgcn_update_dpp(
                        (int)R[u], (int)H, 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
                    const uint32_t xin = (uint32_t)__builtin_amdgcn_update_dpp(
                        (int)(R[u] << 16), (int)X, 0x138, 0xf, 0xf, false);
                    const uint32_t up = __builtin_amdgcn_alignbit(H, hin, 16);
                    const uint32_t upX = __builtin_amdgcn_alignbit(X, xin, 16);
                    const bt_i16x2 m = bt_v(sc) + bt_v(diag);
                    const bt_i16x2 x = bt_max(bt_v(up) - GOX, bt_v(upX) - GE);
                    const bt_i16x2 y = bt_max(bt_v(H) - GO, bt_v(Y) - GE);
                    const bt_i16x2 h = bt_max(bt_max(m, bt_max(y, FLOOR)), x);
                    const int s = 8 * q + u;
                    if constexpr (TAG) {
                        acc = (acc << 2) | (bt_u(h) & 0x00030003u);
                        H = bt_u(h) & 0xfffcfffcu;
                        X = bt_u(x);
                        Y = bt_u(y);
                    } else {
                        const auto ne = [&](bt_i16x2 v) {  // 1 where h differs
                            const bt_u16x2 d = __builtin_bit_cast(bt_u16x2, h) -
                                               __builtin_bit_cast(bt_u16x2, v);
                            return __builtin_bit_cast(bt_i16x2, __builtin_elementwise_min(
                                d, __builtin_bit_cast(bt_u16x2, ONE)));
                        };
                        const bt_i16x2 nm = ne(m), nx = ne(x), nz = ne(bt_v(0u));
                        const bt_i16x2 code = bt_v(0x00030003u) - nz * (ONE + nm + nm * nx);
                        acc = (acc << 2) | bt_u(code);
                        // rows update only on their valid cells; before a row starts
                        // its state stays (H 0, Ix and Iy BT_NEG), the left boundary
                        const int ja = s - 2 * lane + 1, jb = ja - 1;
                        const uint32_t msk = (ja >= 1 && ja <= T && oka ? 0xffffu : 0u) |
                                             (jb >= 1 && jb <= T && okb ? 0xffff0000u : 0u);
                        H = (bt_u(h) & msk) | (H & ~msk);
                        X = (bt_u(x) & msk) | (X & ~msk);
                        Y = (bt_u(y) & msk) | (Y & ~msk);
                    }
                    O[u] = __builtin_amdgcn_perm(H, X, 0x07060302u);
                    const bt_i16x2 nb = bt_max(bt_v(bv), bt_v(H));
                    uint32_t better;  // 0xffff in the halves that grew (opaque: as a
                                      // compare it becomes two per half)
                    asm("v_pk_ashrrev_i16 %0, 15, %1 op_sel_hi:[0,1]" : "=v"(better) : "v"(bt_v(bv) - nb));
                    bs = (better & ((uint32_t)s * 0x10001u)) | (~better & bs);
                    bv = bt_u(nb);
                    diag = up;
                }
                if (64 * q + 63 - lane < 8 * RS) mv[64 * q] = acc;
                if (lane == 63) {
#pragma unroll
                    for (int u = 0; u < 8; ++u) rb[8 * q + u + 1] = O[u];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    P[u] = Pn[u];
                    R[u] = Rn[u];
                }
            }
#undef BT_LETTER_LOAD
#undef BT_SCORE_LOAD
#undef BT_ROW_LOAD
            // the lane's rows in order: a strictly larger value replaces, so
            // ties keep the earlier row (and the earlier column within a row)
            const int bestA = (int)(bv & 0xffffu) / SC, bestB = (int)(bv >> 16) / SC;
            if (bestA > best) {
                best = bestA;
                bi = ia;
                bj = (int)(bs & 0xffffu) - 2 * lane + 1;
            }
            if (bestB > best) {
                best = bestB;
                bi = ib;
                bj = (int)(bs >> 16) - 2 * lane;
            }
            __syncthreads();  // the strip's last row is in rb
        }
        // best value, then the first cell in row-major order
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const int ob = __shfl_xor(best, off, 64);
            const int oi = __shfl_xor(bi, off, 64);
            const int oj = __shfl_xor(bj, off, 64);
            if (ob > best || (ob == best && (oi < bi || (oi == bi && oj < bj)))) {
                best = ob;
                bi = oi;
                bj = oj;
            }
        }
        __threadfence();  // the moves are visible to the loads below
    }
    int n = 0, ci = -1, cj = -1, ei = -1, ej = -1;
    if (best > 0) {
        ei = bi;
        ej = bj;
        int i = ei, j = ej;
        while (i > 0 && j > 0 && n < A) {
            // the cell `lane` diagonal steps back
            const int ix = i - lane, jx = j - lane;
            int code = 3;
            if (ix > 0 && jx > 0) {
                const int k = (ix - 1) >> 7, r = (ix - 1) & 127;
                const int st = jx - 1 + r;
                const uint32_t v = moves[(int64_t)k * RS * 8 + 64 * (st >> 3) + 63 - (r >> 1)];
                code = (int)(v >> (16 * (r & 1) + 2 * (7 - (st & 7)))) & 3;
            }
            const uint64_t stop = __ballot(code != 2);
            const int run = stop ? __builtin_ctzll(stop) : 64;
            const int end = run < 64 ? __builtin_amdgcn_readlane(code, run) : 2;
            // columns written this round: the run, then the gap move
            const int cols = min(run + (end < 2 ? 1 : 0), A - n);
            if (lane < cols) {
                const int64_t w = (int64_t)b * A + A - 1 - n - lane;
                const bool gap = lane == run;
                out_q[w] = gap && end == 0 ? (uint8_t)'-' : query[ix - 1];
                out_t[w] = gap && end == 1 ? (uint8_t)'-' : tg[jx - 1];
            }
            const int dg = min(run, cols), gp = cols - dg;
            i -= dg + (end == 1 ? gp : 0);
            j -= dg + (end == 0 ? gp : 0);
            n += cols;
            if (end == 3) break;
        }
        ci = i;
        cj = j;
    }
    if (lane != 0) return;
    if (n > 0) {
        inf[0] = n;
        inf[1] = ci;
        inf[2] = ei - 1;
        inf[3] = cj;
        inf[4] = ej - 1;
    } else {
        inf[0] = 0;
        inf[1] = -1;
        inf[2] = -1;
        inf[3] = -1;
        inf[4] = -1;
    }
    inf[5] = best;
}

}  // namespace sseqs

using namespace sseqs;

// Workspace: the move words of k_backtrack or, for targets too long for
// its LDS row buffer, the direction bytes + row buffer of k_backtrack_global.
static size_t bt_records_bytes(int query_len, int64_t total_cells, int B) {
    if (query_len <= 0) return 0;
    const int64_t ns = (query_len + 127) / 128;
    return (size_t)(ns * 32 * (total_cells / query_len + 128LL * B));
}
static size_t bt_global_bytes(int query_len, int64_t total_cells) {
    const int64_t rows = query_len > 0 ? total_cells / query_len : 0;
    return (size_t)((total_cells + 255) & ~255LL) + (size_t)rows * 8;
}

extern "C" size_t sseqs_backtrack_ws_bytes(int query_len, int64_t total_cells, int B) {
    const size_t a = bt_records_bytes(query_len, total_cells, B);
    const size_t g = bt_global_bytes(query_len, total_cells);
    return (a > g ? a : g) + 256;
}

extern "C" int sseqs_backtrack(const uint8_t* query, int query_len, const uint8_t* targets,
                               const int64_t* t_off, const int32_t* t_len, const int64_t* cell_off,
                               int64_t total_cells, int B, int gap_open, int gap_extend,
                               int max_align, uint8_t* out_q, uint8_t* out_t, int32_t* info,
                               void* ws, size_t ws_bytes, hipStream_t stream) {
    if (B < 0 || query_len < 0 || total_cells < 0) return fail(-1, "backtrack: negative size");
    if (B == 0) return 0;
    if (max_align < 1) return fail(-1, "backtrack: max_align must be >= 1");
    if (ws_bytes < sseqs_backtrack_ws_bytes(query_len, total_cells, B))
        return fail(-2, "backtrack: workspace too small");
    // targets are at most max_align - query_len - 1 long (the documented bound)
    const int tcap = max_align - query_len - 1;
    if (tcap >= 1 && tcap <= BT_MAX_T) {
        const bool tag = (query_len < tcap ? query_len : tcap) <= BT_TAG_MAX_LEN && gap_open >= 0 &&
                         gap_open <= BT_TAG_MAX_GAP && gap_extend >= 0 && gap_extend <= BT_TAG_MAX_GAP;
        hipLaunchKernelGGL(tag ? k_backtrack<true> : k_backtrack<false>, dim3((unsigned)B), dim3(64),
                           (size_t)bt_lds_bytes(tcap), stream, query, query_len, targets, t_off, t_len,
                           cell_off, gap_open, gap_extend, max_align, out_q, out_t, info,
                           static_cast<uint32_t*>(ws), tcap, blosum62());
        return check_launch("backtrack");
    }
    uint8_t* dirs = static_cast<uint8_t*>(ws);
    int2* rowbuf = reinterpret_cast<int2*>(dirs + ((total_cells + 255) & ~255LL));
    hipLaunchKernelGGL(k_backtrack_global, dim3((unsigned)B), dim3(64), 0, stream, query,
                       query_len, targets, t_off, t_len, cell_off, B, gap_open, gap_extend,
                       max_align, out_q, out_t, info, dirs, rowbuf, blosum62());
    return check_launch("backtrack");
}
