// Deterministic device top-k.
//
// Used wherever the reference calls torch.topk / torch.sort on the search
// path (sseqs/msa.py:297, 307, 324, 335).  Scores become order-preserving
// 32-bit keys; three histogram passes (11 + 11 + 10 bits, most significant
// first; two, 11 + 8, for fp16 scores, whose keys end in 13 cleared bits) find
// the k-th largest key T and how many keys equal to T are taken;
// a compaction pass then writes every index with key > T plus the first
// ones with key == T, in ascending index order.  The optional sort orders
// them by (key desc, index asc) with a bitonic sort in LDS.  The tie rule
// (smaller index first) is the build's definition; torch.topk leaves it open.
#include <mutex>
#include <string>

#include "common.h"

namespace sseqs {

constexpr int SEL_BINS = 2048;
constexpr int SEL_TILE = 16384;     // elements per block in count/write passes
constexpr int SEL_SORT_MAX = 16384;

// prefix / mask / k_rem: the digits of the k-th largest key fixed so far, as
// an offset from the base key (0, or P in a sampled select), and how many of
// the keys that share them are taken.  P, ncand, maxkey: see "sampled
// select" below (P = 0 when every score is a candidate).
struct SelState {
    uint32_t prefix, mask, k_rem, k;
    uint32_t P, ncand, maxkey, pad;
};

__device__ inline uint32_t key_f32(float x) {
    if (x != x) return 0u;  // NaN ranks lowest
    uint32_t b = __float_as_uint(x);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

template <int DT>
__device__ inline uint32_t load_key(const void* s, int64_t i) {
    if constexpr (DT == SSEQS_F32) return key_f32(static_cast<const float*>(s)[i]);
    // an fp16 value as fp32 has 13 constant low bits (zeros, ones once
    // complemented for a negative value): clearing them keeps the order
    if constexpr (DT == SSEQS_F16)
        return key_f32((float)static_cast<const _Float16*>(s)[i]) & ~0x1FFFu;
    return (uint32_t) static_cast<const int32_t*>(s)[i] ^ 0x80000000u;
}

__global__ void k_sel_init(uint32_t* hist, SelState* st, uint32_t k) {
    for (int i = threadIdx.x; i < SEL_BINS; i += blockDim.x) hist[i] = 0;
    if (threadIdx.x == 0) *st = SelState{0u, 0u, k, k, 0u, 0u, 0u, 0u};
}

// ---- sampled select -------------------------------------------------------
//
// Selecting few of many scores needs the digits of only the largest keys.  A
// strided sample gives a key P that about k + 6 sigma + 8 sample steps of the
// scores reach; one pass over the scores (k_sel_filter) marks every key >= P
// in a bitmap, counts them and takes the largest key; the digit, count and
// write passes then read the bitmap and the few marked scores.  One read of
// the scores instead of five (three digit passes, count, write): 200 M fp32
// scores, top 100 000.
//
// P is only a guess.  If fewer than k keys reach it, or the sample says that
// more than an eighth of them do (ties), the select is done over all scores
// as without a sample: every pass decides that on the device from the state,
// so nothing is read back and the launches can be captured.
//
// Bitmap: tile t of SEL_TILE scores is 64 groups of 256; group g of it has
// four 64-bit words at 32 (64 t + g) bytes, word e, bit l: score 4 l + e of
// the group.  A wave reads a group with one load of four scores per lane, and
// its four ballots are the words; the later passes give a lane a group.
constexpr int SEL_GROUP = 256;
constexpr int SEL_TILE_BITS = SEL_TILE / 8;  // bitmap bytes of a tile
constexpr int SEL_SAMPLE = 32768;            // sampled scores: 8 x 4 per thread of 1024
// blocks of a digit pass over the marked scores: each adds its non-zero bins
// to the histogram with device atomics, which cost more than the marked
// scores' reads (200 M scores, 290 k marked: 4096 blocks 42 us, 1024 26 us,
// 256 50 us)
constexpr int SEL_MARK_BLOCKS = 1024;

// Whether the passes run over all scores.
__device__ inline bool sel_full(const SelState* st) {
    return st->P == 0u || st->ncand < st->k;
}
// Key that digits count from.
__device__ inline uint32_t sel_base(const SelState* st) { return sel_full(st) ? 0u : st->P; }

// Digit of pass p: up to 11 bits below those of the earlier passes, from the
// top of the largest key's offset from the base (bits = 0: nothing is left).
template <int DT>
__device__ inline void sel_digit(const SelState* st, int p, int* shift, int* bits) {
    constexpr int LB = DT == SSEQS_F16 ? 13 : 0;  // constant low bits of a key
    int nb = 32 - LB;
    if (!sel_full(st)) {
        const uint32_t d = (st->maxkey - st->P) >> LB;
        nb = d ? 32 - __clz(d) : 1;
    }
    const int rem = nb - 11 * p;
    *bits = rem > 11 ? 11 : (rem > 0 ? rem : 0);
    *shift = LB + (rem > 0 ? rem - *bits : 0);
}

// Four consecutive scores from i, as loaded (i a multiple of 4, the scores
// at an address aligned to four of them).
template <int DT>
struct Load4 {
    uint4 v;
};
template <>
struct Load4<SSEQS_F16> {
    uint2 v;
};
template <int DT>
__device__ inline Load4<DT> load4(const void* s, int64_t i) {
    Load4<DT> r;
    if constexpr (DT == SSEQS_F16)
        r.v = *reinterpret_cast<const uint2*>(static_cast<const _Float16*>(s) + i);
    else
        r.v = *reinterpret_cast<const uint4*>(static_cast<const uint32_t*>(s) + i);
    return r;
}
// Key of score e of the four.
template <int DT>
__device__ inline uint32_t key4(const Load4<DT>& r, int e) {
    if constexpr (DT == SSEQS_F16) {
        const uint32_t w = e < 2 ? r.v.x : r.v.y;
        const _Float16 h =
            __builtin_bit_cast(_Float16, (uint16_t)((e & 1) ? w >> 16 : w & 0xffffu));
        return key_f32((float)h) & ~0x1FFFu;
    } else {
        const uint32_t w = e == 0 ? r.v.x : e == 1 ? r.v.y : e == 2 ? r.v.z : r.v.w;
        if constexpr (DT == SSEQS_F32) return key_f32(__uint_as_float(w));
        return w ^ 0x80000000u;
    }
}

// One block: clears the state and takes the sample's rank-th largest key as
// P.  n >= 4 SEL_SAMPLE, so the sampled quadruples are distinct.
template <int DT>
__global__ __launch_bounds__(1024) void k_sel_sample(const void* s, int64_t n, uint32_t* hist,
                                                     SelState* st, uint32_t k, int rank) {
    constexpr int PER = SEL_SAMPLE / 4096;
    __shared__ uint32_t lh[SEL_BINS];
    __shared__ uint32_t wsum[16], wmax[16];
    __shared__ uint32_t pick[2];
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    for (int i = t; i < SEL_BINS; i += 1024) hist[i] = 0;
    uint32_t key[PER * 4];
    const int64_t step = n / (SEL_SAMPLE / 4);  // scores per sampled quadruple, >= 16
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int q = j * 1024 + t;
        // a different place in every step, so that no period of the scores is followed
        const int64_t at = (int64_t)q * step + (int64_t)((uint32_t)q * 2654435761u % (uint32_t)min(step - 7, (int64_t)1 << 30));
        const Load4<DT> v = load4<DT>(s, at & ~(int64_t)3);
#pragma unroll
        for (int e = 0; e < 4; ++e) key[4 * j + e] = key4<DT>(v, e);
    }
    // digits from the top of the sample's key range: two of 11 bits resolve it
    // to 2^-22, which is enough for a guess, and spread its keys over the bins
    uint32_t lo = key[0], hi = key[0];
#pragma unroll
    for (int j = 1; j < PER * 4; ++j) {
        lo = min(lo, key[j]);
        hi = max(hi, key[j]);
    }
    for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, (uint32_t)__shfl_xor((int)lo, o, 64));
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, o, 64));
    }
    if (lane == 0) {
        wsum[wid] = lo;
        wmax[wid] = hi;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 16; ++w) {
        lo = min(lo, wsum[w]);
        hi = max(hi, wmax[w]);
    }
    const int nb = hi > lo ? 32 - __clz(hi - lo) : 1;
    uint32_t prefix = 0, mask = 0, need = (uint32_t)rank, got = 0;
    int shift = 0;
    for (int p = 0; p < 2; ++p) {
        const int rem = nb - 11 * p;
        if (rem <= 0) break;
        const int bits = min(rem, 11);
        shift = rem - bits;
        __syncthreads();  // wsum of the step before is read
        for (int i = t; i < SEL_BINS; i += 1024) lh[i] = 0;
        __syncthreads();
        const uint32_t bm = (1u << bits) - 1u;
        // one LDS atomic per run of equal bins (neighbouring scores often tie)
        uint32_t run_bin = 0, run = 0;
#pragma unroll
        for (int j = 0; j < PER * 4; ++j) {
            const uint32_t d = key[j] - lo;
            if ((d & mask) != prefix) continue;
            const uint32_t b = (d >> shift) & bm;
            if (run && b == run_bin) {
                ++run;
            } else {
                if (run) atomicAdd(&lh[run_bin], run);
                run_bin = b;
                run = 1;
            }
        }
        if (run) atomicAdd(&lh[run_bin], run);
        __syncthreads();
        // thread t holds bins 2047 - 2t and 2046 - 2t: a scan from the top
        const uint32_t c_hi = lh[SEL_BINS - 1 - 2 * t], c_lo = lh[SEL_BINS - 2 - 2 * t];
        const uint32_t c = c_hi + c_lo;
        uint32_t inc = c;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t v = __shfl_up(inc, o, 64);
            if (lane >= o) inc += v;
        }
        if (lane == 63) wsum[wid] = inc;
        __syncthreads();
        uint32_t above = inc - c;
        for (int w = 0; w < wid; ++w) above += wsum[w];
        if (above < need && need <= above + c) {
            const bool h = need <= above + c_hi;
            pick[0] = (uint32_t)(SEL_BINS - 1 - 2 * t - (h ? 0 : 1));
            pick[1] = above + (h ? 0u : c_hi);
        }
        __syncthreads();
        prefix |= pick[0] << shift;
        mask |= bm << shift;
        got += pick[1];
        need -= pick[1];
    }
    // sample keys >= P: the ones in the bins above, and those in its last bin
    const uint32_t P = lo + prefix;
    __syncthreads();
    if (t == 0) {
        const uint32_t last = lh[pick[0]];  // the last pass's bins, and its pick
        *st = SelState{0u, 0u, k, k, got + last <= SEL_SAMPLE / 8 ? P : 0u, 0u, 0u, 0u};
    }
}

// The pass over the scores: bitmap of the keys >= P, their count and the
// largest key.  A wave takes a tile in steps of eight groups (eight loads of
// four scores per lane in flight) and stores a step's 32 words together.
template <int DT>
__global__ __launch_bounds__(256) void k_sel_filter(const void* s, int64_t n, int64_t nb,
                                                    SelState* st, uint32_t* bitmap) {
    const uint32_t P = st->P;
    if (P == 0u) return;
    __shared__ uint32_t s_cnt[4], s_max[4];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t cnt = 0, mx = 0;
    for (int64_t tile = (int64_t)blockIdx.x * 4 + wid; tile < nb; tile += (int64_t)gridDim.x * 4) {
        const int64_t base = tile * SEL_TILE;
        for (int g0 = 0; g0 < SEL_TILE / SEL_GROUP; g0 += 8) {
            const int64_t i0 = base + (int64_t)g0 * SEL_GROUP + 4 * lane;
            uint64_t word = 0;  // lane 4 u + e: word e of group g0 + u
            if (base + (int64_t)(g0 + 8) * SEL_GROUP <= n) {
                Load4<DT> v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = load4<DT>(s, i0 + u * SEL_GROUP);
#pragma unroll
                for (int u = 0; u < 8; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t key = key4<DT>(v[u], e);
                        mx = max(mx, key);
                        const uint64_t m = __ballot(key >= P);
                        cnt += (uint32_t)__popcll(m);
                        word = lane == 4 * u + e ? m : word;
                    }
            } else {
#pragma unroll
                for (int u = 0; u < 8; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int64_t i = i0 + u * SEL_GROUP + e;
                        const uint32_t key = i < n ? load_key<DT>(s, i) : 0u;
                        mx = max(mx, key);
                        const uint64_t m = __ballot(key >= P);
                        cnt += (uint32_t)__popcll(m);
                        word = lane == 4 * u + e ? m : word;
                    }
            }
            if (lane < 32)
                reinterpret_cast<uint64_t*>(bitmap)[tile * (SEL_TILE_BITS / 8) + g0 * 4 + lane] = word;
        }
    }
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, (uint32_t)__shfl_xor((int)mx, o, 64));
    if (lane == 0) {
        s_cnt[wid] = cnt;
        s_max[wid] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t c = s_cnt[0] + s_cnt[1] + s_cnt[2] + s_cnt[3];
        const uint32_t m = max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3]));
        if (c) atomicAdd(&st->ncand, c);
        atomicMax(&st->maxkey, m);
    }
}

// A lane's group of a tile: f(index, key) for its marked scores in index order.
template <int DT, class F>
__device__ inline void sel_group(const void* s, const uint32_t* bitmap, int64_t tile, int lane,
                                 F f) {
    const uint4* b = reinterpret_cast<const uint4*>(bitmap) + tile * (SEL_TILE_BITS / 16) + 2 * lane;
    const uint4 lo = b[0], hi = b[1];
    const uint64_t w[4] = {((uint64_t)lo.y << 32) | lo.x, ((uint64_t)lo.w << 32) | lo.z,
                           ((uint64_t)hi.y << 32) | hi.x, ((uint64_t)hi.w << 32) | hi.z};
    const int64_t base = tile * SEL_TILE + lane * SEL_GROUP;
    for (uint64_t any = w[0] | w[1] | w[2] | w[3]; any; any &= any - 1) {
        const int l = __ffsll((unsigned long long)any) - 1;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if ((w[e] >> l) & 1ull) f(base + 4 * l + e, load_key<DT>(s, base + 4 * l + e));
    }
}

// The digit pass over the marked scores (a wave per tile); false when the
// pass runs over all of them.
template <int DT>
__device__ inline bool sel_marked_hist(const void* s, int64_t n, const SelState* st,
                                       uint32_t* hist, int pass, const uint32_t* bitmap,
                                       uint32_t* lh) {
    if (sel_full(st)) return false;
    int shift, bits;
    sel_digit<DT>(st, pass, &shift, &bits);
    const int64_t nb = (n + SEL_TILE - 1) / SEL_TILE;
    const int nblk = min((int)gridDim.x, SEL_MARK_BLOCKS);
    if (bits == 0 || (int)blockIdx.x >= nblk) return true;  // uniform over the block
    for (int i = threadIdx.x; i < SEL_BINS; i += 256) lh[i] = 0;
    __syncthreads();
    const uint32_t prefix = st->prefix, mask = st->mask, bm = (1u << bits) - 1u, P = st->P;
    for (int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); tile < nb;
         tile += (int64_t)nblk * 4)
        sel_group<DT>(s, bitmap, tile, threadIdx.x & 63, [&](int64_t, uint32_t key) {
            const uint32_t d = key - P;
            if ((d & mask) == prefix) atomicAdd(&lh[(d >> shift) & bm], 1u);
        });
    __syncthreads();
    for (int i = threadIdx.x; i < SEL_BINS; i += 256)
        if (lh[i]) atomicAdd(&hist[i], lh[i]);
    return true;
}

template <int DT>
__global__ __launch_bounds__(256) void k_sel_hist(const void* s, int64_t n,
                                                  const SelState* st, uint32_t* hist, int pass,
                                                  const uint32_t* bitmap) {
    __shared__ uint32_t lh[SEL_BINS];
    if (sel_marked_hist<DT>(s, n, st, hist, pass, bitmap, lh)) return;
    int shift, bits;
    sel_digit<DT>(st, pass, &shift, &bits);
    for (int i = threadIdx.x; i < SEL_BINS; i += 256) lh[i] = 0;
    __syncthreads();
    const uint32_t prefix = st->prefix, mask = st->mask, bm = (1u << bits) - 1u;
    // four unconditional (index-clamped) loads in flight per thread
    for (int64_t i0 = (int64_t)blockIdx.x * 1024; i0 < n; i0 += (int64_t)gridDim.x * 1024) {
        uint32_t key[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) key[e] = load_key<DT>(s, min(i0 + e * 256 + threadIdx.x, n - 1));
        __builtin_amdgcn_sched_barrier(0);  // the loads first: the compiler waited for one of them
        // one LDS atomic per run of equal bins: tied scores and constant top
        // digits (int32 scores) would otherwise queue at one address
        uint32_t run_bin = 0, run = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (i0 + e * 256 + threadIdx.x >= n || (key[e] & mask) != prefix) continue;
            const uint32_t b = (key[e] >> shift) & bm;
            if (run && b == run_bin) {
                ++run;
            } else {
                if (run) atomicAdd(&lh[run_bin], run);
                run_bin = b;
                run = 1;
            }
        }
        if (run) atomicAdd(&lh[run_bin], run);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < SEL_BINS; i += 256)
        if (lh[i]) atomicAdd(&hist[i], lh[i]);
}

// One block: fix the next digit of T, clear hist.  The digit is the bin b
// (from the top) where the keys above it fall short of k_rem and the keys
// above plus those in it do not; the counts above every bin come from one
// block-wide scan of the bins in descending order.
template <int DT>
__global__ __launch_bounds__(1024) void k_sel_pick(SelState* st, uint32_t* hist, int pass) {
    __shared__ uint32_t wsum[16];
    __shared__ int pick_b;
    __shared__ uint32_t pick_above, cnt0;
    int shift, bits;
    sel_digit<DT>(st, pass, &shift, &bits);
    if (bits == 0) return;
    const int nb = 1 << bits;
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    // thread t holds bins hi = nb-1-2t and lo = hi-1, so ascending t walks
    // the bins from the top
    const int hi = nb - 1 - 2 * t, lo = hi - 1;
    const uint32_t c_hi = hi >= 0 ? hist[hi] : 0u, c_lo = lo >= 0 ? hist[lo] : 0u;
    if (t == 0) pick_b = -1;
    __syncthreads();
    if (hi >= 0) hist[hi] = 0u;
    if (lo >= 0) hist[lo] = 0u;
    if (lo == 0) cnt0 = c_lo;
    const uint32_t c = c_hi + c_lo;
    uint32_t inc = c;  // inclusive scan over the wave
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t v = __shfl_up(inc, o, 64);
        if (lane >= o) inc += v;
    }
    if (lane == 63) wsum[wid] = inc;
    __syncthreads();
    uint32_t above = inc - c;  // keys in the bins above hi
    for (int w = 0; w < wid; ++w) above += wsum[w];
    const uint32_t need = st->k_rem;
    if (hi >= 0 && above < need && need <= above + c_hi) {
        pick_b = hi;
        pick_above = above;
    } else if (lo >= 0 && above + c_hi < need && need <= above + c) {
        pick_b = lo;
        pick_above = above + c_hi;
    }
    __syncthreads();
    if (t == 0) {
        int b = pick_b;
        uint32_t ab = pick_above;
        if (b < 0) {  // fewer keys than k_rem: bin 0, with every other bin above it
            b = 0;
            ab = 0;
            for (int w = 0; w < 16; ++w) ab += wsum[w];
            ab -= cnt0;
        }
        st->prefix |= (uint32_t)b << shift;
        st->mask |= ((1u << bits) - 1u) << shift;
        st->k_rem = need - ab;
    }
}

// Counts of keys > T and == T per tile from the marked scores (a wave per
// tile); false when the pass runs over all scores.
template <int DT>
__device__ inline bool sel_marked_count(const void* s, int64_t nb, const SelState* st, uint32_t T,
                                        int64_t* cgt, int64_t* ceq, const uint32_t* bitmap) {
    if (sel_full(st)) return false;
    const int lane = threadIdx.x & 63;
    for (int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); tile < nb;
         tile += (int64_t)gridDim.x * 4) {
        int gt = 0, eq = 0;
        sel_group<DT>(s, bitmap, tile, lane, [&](int64_t, uint32_t key) {
            gt += key > T;
            eq += key == T;
        });
        for (int o = 32; o > 0; o >>= 1) {
            gt += __shfl_xor(gt, o, 64);
            eq += __shfl_xor(eq, o, 64);
        }
        if (lane == 0) {
            cgt[tile] = gt;
            ceq[tile] = eq;
        }
    }
    return true;
}

// The write pass over the marked scores (a wave per tile, its lanes' groups
// in index order); false when the pass runs over all scores.
template <int DT>
__device__ inline bool sel_marked_write(const void* s, int64_t nb, const SelState* st, uint32_t T,
                                        const int64_t* bgt, const int64_t* beq, int64_t k,
                                        int64_t* out, const uint32_t* bitmap) {
    if (sel_full(st)) return false;
    const int64_t keq = st->k_rem;
    const int lane = threadIdx.x & 63;
    for (int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); tile < nb;
         tile += (int64_t)gridDim.x * 4) {
        uint32_t c = 0;  // the group's (count > T) << 16 | (count == T), each <= 256
        sel_group<DT>(s, bitmap, tile, lane, [&](int64_t, uint32_t key) {
            c += (key > T ? 0x10000u : 0u) + (key == T ? 1u : 0u);
        });
        uint32_t inc = c;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t v = __shfl_up(inc, o, 64);
            if (lane >= o) inc += v;
        }
        if (c == 0) continue;  // no barrier below
        int64_t gb = bgt[tile] + ((inc - c) >> 16), eb = beq[tile] + ((inc - c) & 0xffffu);
        sel_group<DT>(s, bitmap, tile, lane, [&](int64_t i, uint32_t key) {
            const bool g = key > T, q = key == T;
            const int64_t slot = gb + min(eb, keq);
            if ((g || (q && eb < keq)) && slot < k) out[slot] = i;
            gb += g;
            eb += q;
        });
    }
    return true;
}

template <int DT>
__global__ __launch_bounds__(256) void k_sel_count(const void* s, int64_t n,
                                                   int64_t nb, const SelState* st, int64_t* cgt,
                                                   int64_t* ceq, const uint32_t* bitmap) {
    const uint32_t T = sel_base(st) + st->prefix;
    if (sel_marked_count<DT>(s, nb, st, T, cgt, ceq, bitmap)) return;
    __shared__ int rg[256], re[256];
    for (int64_t tile = blockIdx.x; tile < nb; tile += gridDim.x) {
    const int64_t base = tile * SEL_TILE;
    const int m = (int)min((int64_t)SEL_TILE, n - base);  // the last tile ends early
    int gt = 0, eq = 0;
#pragma unroll 4
    for (int j0 = 0; j0 < m; j0 += 256) {
        const int64_t i = base + j0 + threadIdx.x;
        const uint32_t key = load_key<DT>(s, min(i, n - 1));
        if (i < n) {
            gt += key > T;
            eq += key == T;
        }
    }
    rg[threadIdx.x] = gt;
    re[threadIdx.x] = eq;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            rg[threadIdx.x] += rg[threadIdx.x + o];
            re[threadIdx.x] += re[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        cgt[tile] = rg[0];
        ceq[tile] = re[0];
    }
    __syncthreads();
    }
}

// Exclusive scan of two arrays of nb counts (each at most SEL_TILE), one
// block.  Wave w holds SCAN_ROWS rows of 64 consecutive counts of each array
// in registers per round, so every load is coalesced and all are in flight;
// a row is scanned across the lanes in 32 bits.  (Twelve consecutive counts
// per thread, 12 207 in all, take 35 us.)
constexpr int SCAN_ROWS = 8;

// Inclusive sum over the lanes of a wave: shifts by 1, 2, 4, 8 within the
// rows of 16, then the rows' totals (lane 15 of each row to the next row,
// lane 31 to the upper half).
template <int CTRL, int ROWS>
__device__ inline int scan_dpp(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}
__device__ inline int wave_scan_i32(int v) {
    v += scan_dpp<0x111, 0xf>(v);
    v += scan_dpp<0x112, 0xf>(v);
    v += scan_dpp<0x114, 0xf>(v);
    v += scan_dpp<0x118, 0xf>(v);
    v += scan_dpp<0x142, 0xa>(v);
    v += scan_dpp<0x143, 0xc>(v);
    return v;
}

__global__ __launch_bounds__(1024) void k_sel_scan(int64_t* a, int64_t* b, int64_t nb) {
    __shared__ int wa[16], wb[16];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int64_t ra = 0, rb = 0;  // totals of the rounds before
    for (int64_t r0 = 0; r0 < nb; r0 += 1024 * SCAN_ROWS) {
        // rows per wave of this round (a short round is spread over the waves)
        const int rows = (int)min((int64_t)SCAN_ROWS, (nb - r0 + 1023) / 1024);
        const int64_t w0 = r0 + (int64_t)wid * rows * 64 + lane;
        int va[SCAN_ROWS], vb[SCAN_ROWS];
#pragma unroll
        for (int i = 0; i < SCAN_ROWS; ++i) {  // clamped, so unconditional
            const int64_t at = min(w0 + 64 * min(i, rows - 1), nb - 1);
            va[i] = (int)a[at];
            vb[i] = (int)b[at];
        }
        int ta = 0, tb = 0;  // totals of the wave's rows: at most 64 SCAN_ROWS SEL_TILE
        int ea[SCAN_ROWS], eb[SCAN_ROWS];
#pragma unroll
        for (int i = 0; i < SCAN_ROWS; ++i) {
            const bool in = i < rows && w0 + 64 * i < nb;
            const int ca = in ? va[i] : 0, cb = in ? vb[i] : 0;
            const int ia = wave_scan_i32(ca), ib = wave_scan_i32(cb);
            ea[i] = ta + ia - ca;
            eb[i] = tb + ib - cb;
            ta += __builtin_amdgcn_readlane(ia, 63);
            tb += __builtin_amdgcn_readlane(ib, 63);
        }
        if (lane == 0) {
            wa[wid] = ta;
            wb[wid] = tb;
        }
        __syncthreads();
        int64_t ba = ra, bb = rb;
        for (int w = 0; w < 16; ++w) {
            const int xa = wa[w], xb = wb[w];
            ba += w < wid ? xa : 0;
            bb += w < wid ? xb : 0;
            ra += xa;
            rb += xb;
        }
#pragma unroll
        for (int i = 0; i < SCAN_ROWS; ++i)
            if (i < rows && w0 + 64 * i < nb) {
                a[w0 + 64 * i] = ba + ea[i];
                b[w0 + 64 * i] = bb + eb[i];
            }
        __syncthreads();
    }
}

template <int DT>
__global__ __launch_bounds__(256) void k_sel_write(const void* s, int64_t n,
                                                   int64_t nb, const SelState* st,
                                                   const int64_t* bgt, const int64_t* beq,
                                                   int64_t k, int64_t* out,
                                                   const uint32_t* bitmap) {
    const uint32_t T = sel_base(st) + st->prefix;
    if (sel_marked_write<DT>(s, nb, st, T, bgt, beq, k, out, bitmap)) return;
    const int64_t keq = st->k_rem;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint64_t below = (1ull << lane) - 1ull;
    __shared__ int wg[4][4], we[4][4];  // [step][wave]
    for (int64_t tile = blockIdx.x; tile < nb; tile += gridDim.x) {
        int64_t gt_run = bgt[tile], eq_run = beq[tile];
        const int64_t base = tile * SEL_TILE;
        const int m = (int)min((int64_t)SEL_TILE, n - base);
        // four steps of 256 elements per barrier pair; loads first, in flight together
        for (int j0 = 0; j0 < m; j0 += 1024) {
            uint32_t key[4];
            uint64_t mg[4], me[4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
                key[t] = load_key<DT>(s, min(base + j0 + t * 256 + threadIdx.x, n - 1));
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const bool in = base + j0 + t * 256 + threadIdx.x < n;
                mg[t] = __ballot(in && key[t] > T);
                me[t] = __ballot(in && key[t] == T);
                if (lane == 0) {
                    wg[t][wid] = __popcll(mg[t]);
                    we[t][wid] = __popcll(me[t]);
                }
            }
            __syncthreads();
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                int og = 0, oe = 0, tg = 0, te = 0;
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    if (w < wid) {
                        og += wg[t][w];
                        oe += we[t][w];
                    }
                    tg += wg[t][w];
                    te += we[t][w];
                }
                const bool g = (mg[t] >> lane) & 1ull, e = (me[t] >> lane) & 1ull;
                const int64_t gb = gt_run + og + __popcll(mg[t] & below);  // keys > T before i
                const int64_t eb = eq_run + oe + __popcll(me[t] & below);  // keys == T before i
                const int64_t slot = gb + min(eb, keq);
                if ((g || (e && eb < keq)) && slot < k) out[slot] = base + j0 + t * 256 + threadIdx.x;
                gt_run += tg;
                eq_run += te;
            }
            __syncthreads();
        }
    }
}

// Sort the k selected indices by (key desc, index asc); k <= SEL_SORT_MAX.
// ---- fp16 scores, eight per thread --------------------------------------
//
// The passes above give each thread one 2-byte score per load.  For fp16
// scores at a 16-byte aligned address these variants load eight at once
// (one 16-byte load per thread), and the write pass places a step of 2048
// scores with one block barrier (a wave scan of the threads' packed counts)
// instead of two barriers per 1024.  Same keys, same T, same output.

// Keys of scores i .. i+7 (entries at or past n are flagged invalid).
__device__ inline uint32_t keys8_f16(const _Float16* s, int64_t i, int64_t n, uint32_t key[8]) {
    if (i + 8 <= n) {
        const uint4 v = *reinterpret_cast<const uint4*>(s + i);
        const _Float16* e = reinterpret_cast<const _Float16*>(&v);
#pragma unroll
        for (int x = 0; x < 8; ++x) key[x] = key_f32((float)e[x]) & ~0x1FFFu;
        return 0xFFu;
    }
    uint32_t valid = 0;
#pragma unroll
    for (int x = 0; x < 8; ++x) {
        const bool in = i + x < n;
        key[x] = in ? key_f32((float)s[i + x]) & ~0x1FFFu : 0u;
        valid |= (uint32_t)in << x;
    }
    return valid;
}

__global__ __launch_bounds__(256) void k_sel_hist_h8(const _Float16* __restrict__ s, int64_t n,
                                                     const SelState* st, uint32_t* hist, int pass,
                                                     const uint32_t* bitmap) {
    __shared__ uint32_t lh[SEL_BINS];
    if (sel_marked_hist<SSEQS_F16>(s, n, st, hist, pass, bitmap, lh)) return;
    int shift, bits;
    sel_digit<SSEQS_F16>(st, pass, &shift, &bits);
    for (int i = threadIdx.x; i < SEL_BINS; i += 256) lh[i] = 0;
    __syncthreads();
    const uint32_t prefix = st->prefix, mask = st->mask, bm = (1u << bits) - 1u;
    for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8; i < n;
         i += (int64_t)gridDim.x * 2048) {
        uint32_t key[8];
        const uint32_t valid = keys8_f16(s, i, n, key);
        // neighbouring scores often share a bin: one LDS atomic per run
        uint32_t run_bin = 0, run = 0;
#pragma unroll
        for (int x = 0; x < 8; ++x) {
            if (!((valid >> x) & 1u) || (key[x] & mask) != prefix) continue;
            const uint32_t b = (key[x] >> shift) & bm;
            if (run && b == run_bin) {
                ++run;
            } else {
                if (run) atomicAdd(&lh[run_bin], run);
                run_bin = b;
                run = 1;
            }
        }
        if (run) atomicAdd(&lh[run_bin], run);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < SEL_BINS; i += 256)
        if (lh[i]) atomicAdd(&hist[i], lh[i]);
}

__global__ __launch_bounds__(256) void k_sel_count_h8(const _Float16* __restrict__ s, int64_t n,
                                                      int64_t nb, const SelState* st,
                                                      int64_t* cgt, int64_t* ceq,
                                                      const uint32_t* bitmap) {
    const uint32_t T = sel_base(st) + st->prefix;
    if (sel_marked_count<SSEQS_F16>(s, nb, st, T, cgt, ceq, bitmap)) return;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __shared__ int rg[4], re[4];
    for (int64_t tile = blockIdx.x; tile < nb; tile += gridDim.x) {
        const int64_t base = tile * SEL_TILE;
        int gt = 0, eq = 0;
#pragma unroll 2
        for (int j = 8 * threadIdx.x; j < SEL_TILE; j += 2048) {
            uint32_t key[8];
            const uint32_t valid = keys8_f16(s, base + j, n, key);
#pragma unroll
            for (int x = 0; x < 8; ++x) {
                const bool in = (valid >> x) & 1u;
                gt += in && key[x] > T;
                eq += in && key[x] == T;
            }
        }
        for (int o = 32; o > 0; o >>= 1) {
            gt += __shfl_xor(gt, o, 64);
            eq += __shfl_xor(eq, o, 64);
        }
        if (lane == 0) {
            rg[wid] = gt;
            re[wid] = eq;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            cgt[tile] = rg[0] + rg[1] + rg[2] + rg[3];
            ceq[tile] = re[0] + re[1] + re[2] + re[3];
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void k_sel_write_h8(const _Float16* __restrict__ s, int64_t n,
                                                      int64_t nb, const SelState* st,
                                                      const int64_t* bgt, const int64_t* beq,
                                                      int64_t k, int64_t* out,
                                                      const uint32_t* bitmap) {
    const uint32_t T = sel_base(st) + st->prefix;
    if (sel_marked_write<SSEQS_F16>(s, nb, st, T, bgt, beq, k, out, bitmap)) return;
    const int64_t keq = st->k_rem;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    // wave totals of a step, (count > T) << 16 | (count == T), by step parity:
    // a wave writes a step's slot only after every wave has passed the
    // previous step's barrier, i.e. has read the slot two steps back
    __shared__ uint32_t wt[2][4];
    int par = 0;
    for (int64_t tile = blockIdx.x; tile < nb; tile += gridDim.x) {
        int64_t gt_run = bgt[tile], eq_run = beq[tile];
        const int64_t base = tile * SEL_TILE;
        for (int j0 = 0; j0 < SEL_TILE; j0 += 2048) {
            const int64_t i0 = base + j0 + 8 * threadIdx.x;
            uint32_t key[8];
            const uint32_t valid = keys8_f16(s, i0, n, key);
            uint32_t gm = 0, em = 0;
#pragma unroll
            for (int x = 0; x < 8; ++x) {
                const bool in = (valid >> x) & 1u;
                gm |= (uint32_t)(in && key[x] > T) << x;
                em |= (uint32_t)(in && key[x] == T) << x;
            }
            const uint32_t c = ((uint32_t)__popc(gm) << 16) | (uint32_t)__popc(em);
            uint32_t inc = c;  // inclusive scan over the wave (each field < 2^16)
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t v = __shfl_up(inc, o, 64);
                if (lane >= o) inc += v;
            }
            if (lane == 63) wt[par][wid] = inc;
            __syncthreads();
            uint32_t before = inc - c, total = 0;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const uint32_t t = wt[par][w];
                if (w < wid) before += t;
                total += t;
            }
            par ^= 1;
            if (gm | em) {
                int64_t gb = gt_run + (before >> 16);     // keys > T before score i0
                int64_t eb = eq_run + (before & 0xFFFFu);  // keys == T before score i0
#pragma unroll
                for (int x = 0; x < 8; ++x) {
                    const bool g = (gm >> x) & 1u, e = (em >> x) & 1u;
                    const int64_t slot = gb + min(eb, keq);
                    if ((g || (e && eb < keq)) && slot < k) out[slot] = i0 + x;
                    gb += g;
                    eb += e;
                }
            }
            gt_run += total >> 16;
            eq_run += total & 0xFFFFu;
        }
    }
}

template <int DT>
__global__ __launch_bounds__(1024) void k_sel_sort(const void* s, const int64_t* sel,
                                                   int64_t k, int P, int64_t* out) {
    extern __shared__ uint64_t comp[];
    for (int i = threadIdx.x; i < P; i += 1024) {
        if (i < k) {
            int64_t idx = sel[i];
            uint32_t key = load_key<DT>(s, idx);
            comp[i] = ((uint64_t)(~key) << 32) | (uint64_t)(uint32_t)idx;
        } else {
            comp[i] = ~0ull;
        }
    }
    __syncthreads();
    for (int size = 2; size <= P; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = threadIdx.x; i < P; i += 1024) {
                int j = i ^ stride;
                if (j > i) {
                    bool up = (i & size) == 0;
                    uint64_t a = comp[i], b = comp[j];
                    if ((a > b) == up) {
                        comp[i] = b;
                        comp[j] = a;
                    }
                }
            }
            __syncthreads();
        }
    }
    for (int i = threadIdx.x; i < k; i += 1024) out[i] = (int64_t)(uint32_t)comp[i];
}

// ------------------------------------------------------------------------
// Segmented top-k: the per-batch selects of the reference's cascade
// (sseqs/msa.py:297-310, 324, 335) for every batch of a sweep in one launch.
// One block of SEG_THREADS threads per segment: histogram passes over the
// segment's keys in LDS fix the k-th largest key T, then one pass in index
// order writes the selection (keys > T, then the first keys == T), or the
// selection is staged in LDS and sorted by (key desc, index asc).
//
// The scores of a segment fall into few bins, so a pass over all keys is bound
// by LDS atomics on the same addresses, and a sweep has fewer segments than
// the chip has CUs.  A long segment of which little is taken (seg_guess) is
// therefore first cut down: the R-th largest of SEG_SAMPLE keys, R some
// deviations past the rank that k has among them, is a key that enough of the
// segment reaches, and the keys that reach it go to a list in LDS in index
// order (one pass counts them per wave, one writes them); the passes then
// read the list.  If they are fewer than k or more than the list holds, the
// passes read the segment.  72 segments of 281 000 fp16 scores, k = n / 200:
// 739 -> 283 us.

constexpr int SEG_THREADS = 1024;
constexpr int SEG_WAVES = SEG_THREADS / 64;
constexpr int SEG_SORT_MAX = 4096;
constexpr int SEG_E = 8;  // elements per thread per pass step

// 16-bit order key of an fp16 score (NaN lowest, as key_f32)
__device__ inline uint32_t key_h16(uint16_t h) {
    if ((h & 0x7c00u) == 0x7c00u && (h & 0x03ffu)) return 0u;
    return (h & 0x8000u) ? (~h & 0xffffu) : (h | 0x8000u);
}

// A score as loaded, and its key.
template <int DT>
__device__ inline uint32_t seg_raw(const void* s, int64_t i) {
    if constexpr (DT == SSEQS_F16) return static_cast<const uint16_t*>(s)[i];
    else return static_cast<const uint32_t*>(s)[i];
}
template <int DT>
__device__ inline uint32_t seg_key_of(uint32_t w) {
    if constexpr (DT == SSEQS_F16) return key_h16((uint16_t)w);
    else return load_key<DT>(&w, 0);
}
template <int DT>
__device__ inline uint32_t seg_key(const void* s, int64_t i) {
    return seg_key_of<DT>(seg_raw<DT>(s, i));
}

constexpr int SEG_SAMPLE = SEG_THREADS * SEG_E;
constexpr int SEG_LIST = 12288;     // keys and indices: 96 KiB of LDS
// Selections in index order of at least so many take the instance that can cut
// (a cascade selects 1/200 of segments of some 10^5: 710 of 281 000 fp16 scores,
// k = 1405, 713 us uncut, 371 cut).  Segments that it does not cut take the time
// of the other instance (1000 of 5000 fp32, k = 200: 68 us; 600 of 281 000 fp16,
// k = 20 000: 756 / 697), whose LDS holds the sort instead of the list.
constexpr int SEG_CUT_K = 128;

// The rank among SEG_SAMPLE of n keys to guess at, or 0 where the passes read
// the segment itself: below four samples there is little to save, and a list
// is expected to fill less than seven eighths.
__device__ inline int seg_guess(int n, int k) {
    if (n < 4 * SEG_SAMPLE) return 0;
    const float m = (float)SEG_SAMPLE * (float)k / (float)n;
    const float r = m + 4.f * sqrtf(m) + 8.f;
    return r * (float)n <= 0.875f * SEG_LIST * SEG_SAMPLE ? (int)r : 0;
}

typedef uint32_t seg_u32x4_el __attribute__((ext_vector_type(4), aligned(2)));

// A wave's step: 512 consecutive elements, eight to a lane; U steps' loads are in
// flight together.
template <int DT>
struct SegStep {
    static constexpr int NV = DT == SSEQS_F16 ? 1 : 2, U = 4 / NV;
    uint32_t w[4 * NV];
    __device__ void load(const void* s, int i0) {
        const int i = i0 + 8 * (threadIdx.x & 63);
        const char* p = static_cast<const char*>(s) + (DT == SSEQS_F16 ? 2 : 4) * (int64_t)i;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const seg_u32x4_el x = reinterpret_cast<const seg_u32x4_el*>(p)[v];
#pragma unroll
            for (int y = 0; y < 4; ++y) w[4 * v + y] = x[y];
        }
    }
    // the last, partial step: element by element, past n the last one
    __device__ void load_tail(const void* s, int i0, int n) {
        const int i = i0 + 8 * (threadIdx.x & 63);
#pragma unroll
        for (int y = 0; y < 4 * NV; ++y) {
            if constexpr (DT == SSEQS_F16) {
                const uint16_t* h = static_cast<const uint16_t*>(s);
                w[y] = h[min(i + 2 * y, n - 1)] | (uint32_t)h[min(i + 2 * y + 1, n - 1)] << 16;
            } else {
                w[y] = static_cast<const uint32_t*>(s)[min(i + y, n - 1)];
            }
        }
    }
    __device__ uint32_t key(int e) const {
        if constexpr (DT == SSEQS_F16) return key_h16((uint16_t)(w[e >> 1] >> (16 * (e & 1))));
        else return load_key<DT>(w, e);
    }
    // bit e: element i0 + 8 lane + e is below n and its key at least g
    __device__ uint32_t reach(int i0, int n, uint32_t g) const {
        const int i = i0 + 8 * (threadIdx.x & 63);
        uint32_t in = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) in |= key(e) >= g && i + e < n ? 1u << e : 0u;
        return in;
    }
};

// f(first element, step) over the steps of elements lo .. hi - 1
template <int DT, class F>
__device__ inline void seg_steps(const void* s, int lo, int hi, int n, F f) {
    int i0 = lo;
    constexpr int U = SegStep<DT>::U;
    for (; i0 + 512 * U <= hi; i0 += 512 * U) {
        SegStep<DT> st[U];
#pragma unroll
        for (int u = 0; u < U; ++u) st[u].load(s, i0 + 512 * u);
#pragma unroll
        for (int u = 0; u < U; ++u) f(i0 + 512 * u, st[u]);
    }
    for (; i0 < hi; i0 += 512) {
        SegStep<DT> st;
        if (i0 + 512 <= n) st.load(s, i0);
        else st.load_tail(s, i0, n);
        f(i0, st);
    }
}

template <int DT, bool CUT>
__global__ __launch_bounds__(SEG_THREADS) void k_seg_topk(
    const void* __restrict__ s, const int64_t* __restrict__ seg_begin,
    const int32_t* __restrict__ seg_n, const int32_t* __restrict__ seg_k,
    const int64_t* __restrict__ out_base, int64_t nseg, int sorted, int drop_front,
    int drop_back, int add_begin, int64_t* __restrict__ out) {
    __shared__ uint32_t hist[SEL_BINS];
    __shared__ uint64_t comp[CUT ? 1 : SEG_SORT_MAX];  // sorted output
    __shared__ uint32_t wsum[SEG_WAVES];
    __shared__ uint32_t s_pick[2];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    extern __shared__ uint32_t l_key[];  // CUT: the list, keys, then indices
    uint32_t* l_idx = l_key + SEG_LIST;
    const int npass = DT == SSEQS_F16 ? 2 : 3;
    const int shifts16[2] = {5, 0}, bits16[2] = {11, 5};
    const int shifts32[3] = {21, 10, 0}, bits32[3] = {11, 11, 10};
    for (int64_t j = blockIdx.x; j < nseg; j += gridDim.x) {
        const int64_t beg = seg_begin[j];
        int n = seg_n[j];
        int k = min(seg_k[j], n);
        if (sorted) k = min(k, SEG_SORT_MAX);
        if (k <= 0) continue;  // uniform over the block
        const void* base = DT == SSEQS_F16
                               ? static_cast<const void*>(static_cast<const uint16_t*>(s) + beg)
                           : DT == SSEQS_F32
                               ? static_cast<const void*>(static_cast<const float*>(s) + beg)
                               : static_cast<const void*>(static_cast<const int32_t*>(s) + beg);
        // round 0 (with a guess): the R-th largest key of the sample, and the
        // list of the keys that reach it; round 1: the k-th largest key
        const int R = CUT ? seg_guess(n, k) : 0;
        bool listed = false;
        uint32_t prefix = 0, mask = 0, krem = 0;
        for (int round = CUT && R > 0 ? 0 : 1; round < 2; ++round) {
            const int m = round ? n : SEG_SAMPLE;
            prefix = mask = 0;
            krem = (uint32_t)(round ? k : R);
            for (int p = 0; p < npass; ++p) {
                const int shift = DT == SSEQS_F16 ? shifts16[p] : shifts32[p];
                const int bits = DT == SSEQS_F16 ? bits16[p] : bits32[p];
                const uint32_t bm = (1u << bits) - 1u;
                for (int i = tid; i < SEL_BINS; i += SEG_THREADS) hist[i] = 0;
                __syncthreads();
                const auto count = [&](auto get, auto key_of) {
                    for (int i0 = 0; i0 < m; i0 += SEG_THREADS * SEG_E) {
                        uint32_t w[SEG_E];
                        // SEG_E independent loads in flight per thread: the index is
                        // clamped, so that they are unconditional, and none is moved
                        // to its use
#pragma unroll
                        for (int e = 0; e < SEG_E; ++e) w[e] = get(min(i0 + e * SEG_THREADS + tid, m - 1));
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int e = 0; e < SEG_E; ++e) {
                            const uint32_t key = key_of(w[e]);
                            if ((i0 + e * SEG_THREADS + tid < m) & ((key & mask) == prefix))
                                atomicAdd(&hist[(key >> shift) & bm], 1u);
                        }
                    }
                };
                // a loop of its own for each source of keys: one loop that asked
                // for every key made a pass over a segment half as fast
                const auto key_of = [](uint32_t w) { return seg_key_of<DT>(w); };
                if (CUT && listed)
                    count([&](int i) { return l_key[i]; }, [](uint32_t w) { return w; });
                else if (CUT && round == 0)
                    count([&](int i) { return seg_raw<DT>(base, (int)((int64_t)i * n / SEG_SAMPLE)); }, key_of);
                else
                    count([&](int i) { return seg_raw<DT>(base, i); }, key_of);
                __syncthreads();
                if (wid == 0) {
                    // lane L holds bins 32L..32L+31; the lane whose bins contain
                    // the krem-th largest key walks them from the top
                    uint32_t sum = 0;
                    // (16-byte reads; single words from rotated places, which meet
                    // in no bank, made a launch of short segments 4-8 us longer)
                    for (int t = 0; t < 32; ++t) sum += hist[lane * 32 + t];
                    uint32_t incl = sum;  // keys in bins of lanes >= this one
                    for (int off = 1; off < 64; off <<= 1) {
                        const uint32_t t = __shfl_down(incl, off, 64);
                        if (lane + off < 64) incl += t;
                    }
                    uint32_t above = incl - sum;
                    if (above < krem && krem <= incl) {
                        int b = lane * 32 + 31;
                        for (; b > lane * 32; --b) {
                            if (above + hist[b] >= krem) break;
                            above += hist[b];
                        }
                        s_pick[0] = (uint32_t)b;
                        s_pick[1] = krem - above;
                    }
                }
                __syncthreads();
                prefix |= s_pick[0] << shift;
                mask |= bm << shift;
                krem = s_pick[1];
                __syncthreads();
            }
            if (CUT && round == 0) {
                // wave w takes the w-th sixteenth of the segment, 512 elements a step
                const int per = (n + 512 * SEG_WAVES - 1) / (512 * SEG_WAVES) * 512;
                const int lo = min(n, wid * per), hi = min(n, lo + per);
                int cnt = 0;
                seg_steps<DT>(base, lo, hi, n, [&](int i0, const SegStep<DT>& st) {
                    cnt += __popc(st.reach(i0, n, prefix));
                });
                for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, 64);
                if (lane == 0) wsum[wid] = (uint32_t)cnt;
                __syncthreads();
                int at = 0, total = 0;
#pragma unroll
                for (int w = 0; w < SEG_WAVES; ++w) {
                    at += w < wid ? (int)wsum[w] : 0;
                    total += (int)wsum[w];
                }
                listed = total >= k && total <= SEG_LIST;
                if (listed) {
                    seg_steps<DT>(base, lo, hi, n, [&](int i0, const SegStep<DT>& st) {
                        const uint32_t in = st.reach(i0, n, prefix);
                        if (!__any(in)) return;
                        int inc = __popc(in);
                        for (int o = 1; o < 64; o <<= 1) {
                            const int t = __shfl_up(inc, o, 64);
                            if (lane >= o) inc += t;
                        }
                        int slot = at + inc - __popc(in);
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            if ((in >> e) & 1u) {
                                l_key[slot] = st.key(e);
                                l_idx[slot] = (uint32_t)(i0 + 8 * lane + e);
                                ++slot;
                            }
                        at += __shfl(inc, 63, 64);
                    });
                    n = total;
                }
                __syncthreads();
            }
        }
        // keys > T are all taken, keys == T while fewer than krem came
        // before.  Each thread takes SEG_E consecutive elements of a chunk;
        // a block scan of the per-thread counts (> T, == T), packed as
        // (gt << 16 | eq), gives every element its place in index order.
        const uint32_t T = prefix;
        const int keq = (int)krem;
        const int hi = k - drop_back;
        const int64_t ob = out_base[j] - drop_front;
        const int64_t add = add_begin ? beg : 0;
        int gt_run = 0, eq_run = 0;
        const auto write = [&](auto get, auto index) {
            for (int i0 = 0; i0 < n; i0 += SEG_THREADS * SEG_E) {
                const int ib = i0 + tid * SEG_E;
                uint32_t key[SEG_E];
#pragma unroll
                for (int e = 0; e < SEG_E; ++e)
                    key[e] = get(min(ib + e, n - 1));
                uint32_t cnt = 0;
#pragma unroll
                for (int e = 0; e < SEG_E; ++e) {
                    const bool in = ib + e < n;
                    cnt += (in && key[e] > T) ? 0x10000u : 0u;
                    cnt += (in && key[e] == T) ? 1u : 0u;
                }
                // inclusive scan over the wave, then over the waves
                uint32_t inc = cnt;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const uint32_t t = __shfl_up(inc, o, 64);
                    if (lane >= o) inc += t;
                }
                if (lane == 63) wsum[wid] = inc;
                __syncthreads();
                uint32_t before = inc - cnt, total = 0;
#pragma unroll
                for (int w = 0; w < SEG_WAVES; ++w) {
                    const uint32_t t = wsum[w];
                    before += w < wid ? t : 0u;
                    total += t;
                }
                int gb = gt_run + (int)(before >> 16), eb = eq_run + (int)(before & 0xffffu);
#pragma unroll
                for (int e = 0; e < SEG_E; ++e) {
                    const bool in = ib + e < n;
                    const bool g = in && key[e] > T;
                    const bool q = in && key[e] == T;
                    const int slot = gb + min(eb, keq);
                    if ((g || (q && eb < keq)) && slot < k) {
                        const uint32_t at = index(ib + e);
                        if (!CUT && sorted)
                            comp[slot] = ((uint64_t)(~key[e]) << 32) | (uint64_t)at;
                        else if (slot >= drop_front && slot < hi)
                            out[ob + slot] = add + at;
                    }
                    gb += g;
                    eb += q;
                }
                gt_run += (int)(total >> 16);
                eq_run += (int)(total & 0xffffu);
                __syncthreads();
            }
        };
        if (CUT && listed)
            write([&](int i) { return l_key[i]; }, [&](int i) { return l_idx[i]; });
        else
            write([&](int i) { return seg_key<DT>(base, i); }, [](int i) { return (uint32_t)i; });
        if (!CUT && sorted) {
            int P = 1;
            while (P < k) P <<= 1;
            for (int i = k + tid; i < P; i += SEG_THREADS) comp[i] = ~0ull;
            __syncthreads();
            for (int size = 2; size <= P; size <<= 1) {
                for (int stride = size >> 1; stride > 0; stride >>= 1) {
                    for (int i = tid; i < P; i += SEG_THREADS) {
                        const int m = i ^ stride;
                        if (m > i) {
                            const bool up = (i & size) == 0;
                            const uint64_t a = comp[i], b = comp[m];
                            if ((a > b) == up) {
                                comp[i] = b;
                                comp[m] = a;
                            }
                        }
                    }
                    __syncthreads();
                }
            }
            for (int i = drop_front + tid; i < hi; i += SEG_THREADS)
                out[ob + i] = add + (int64_t)(uint32_t)comp[i];
            __syncthreads();
        }
    }
}

}  // namespace sseqs

using namespace sseqs;

// Launch the instance of a select kernel for the score type `dtype`.
#define SEL_DISPATCH(KERNEL, ...)                                                   \
    do {                                                                          \
        if (dtype == SSEQS_F32)                                                   \
            hipLaunchKernelGGL(KERNEL<SSEQS_F32>, __VA_ARGS__);                   \
        else if (dtype == SSEQS_F16)                                              \
            hipLaunchKernelGGL(KERNEL<SSEQS_F16>, __VA_ARGS__);                   \
        else                                                                      \
            hipLaunchKernelGGL(KERNEL<SSEQS_I32>, __VA_ARGS__);                   \
    } while (0)

// Sampled select: few of many scores, at an address that four of them are
// aligned to.  Top 100 000, sampled against all passes over the scores (us):
// fp32 200 M 298 / 1153, 20 M 115 / 233, 8 M 102 / 137; fp16 200 M 209 / 489,
// 8 M 89 / 109; int32 200 M 274 / 1956.  The marked scores' passes grow with
// k, the others' with n: from 6 M on k = n / 64 is no loss (fp32 6 M 116 / 117,
// 8 M 124 / 131; fp16 6 M 94 / 94); below, at 4 M, fp32 gains up to n / 400 (81 /
// 85; n / 200 90 / 86, n / 64 114 / 95), fp16 up to n / 128 (75 / 77; n / 64
// 85 / 78), and int32 at n / 64 (80 / 111).
constexpr int64_t SEL_SAMPLE_MIN_N = 1 << 22;
constexpr int64_t SEL_SAMPLE_ANY_N = 6000000;
static int64_t sel_sample_ratio(int dtype, int64_t n) {
    if (n >= SEL_SAMPLE_ANY_N || dtype == SSEQS_I32) return 64;
    return dtype == SSEQS_F16 ? 128 : 400;
}
static bool sel_sampled(const void* scores, int dtype, int64_t n, int64_t k) {
    const uintptr_t al = dtype == SSEQS_F16 ? 8 : 16;
    return n >= SEL_SAMPLE_MIN_N && k <= n / sel_sample_ratio(dtype, n) && n <= 0xffffffffLL &&
           (reinterpret_cast<uintptr_t>(scores) & (al - 1)) == 0;
}

static size_t sel_ws_base(int64_t n) {
    int64_t nb = ceil_div(n > 0 ? n : 1, SEL_TILE);
    return (size_t)SEL_BINS * 4 + 64 + (size_t)nb * 16 + (size_t)SEL_SORT_MAX * 8 + 256;
}

extern "C" size_t sseqs_topk_ws_bytes(int64_t n) {
    // plus the bitmap of a sampled select, at a 16-byte aligned address
    return sel_ws_base(n) +
           (n >= SEL_SAMPLE_MIN_N ? (size_t)ceil_div(n, SEL_TILE) * SEL_TILE_BITS + 16 : 0);
}

// bitmap_ok: the workspace holds the bitmap of a sampled select.
static int topk_impl(const void* scores, int dtype, int64_t n, int64_t k, int sorted,
                     int64_t* out_idx, void* ws, bool bitmap_ok, hipStream_t stream) {
    uint8_t* w = static_cast<uint8_t*>(ws);
    uint32_t* hist = reinterpret_cast<uint32_t*>(w);
    SelState* st = reinterpret_cast<SelState*>(w + SEL_BINS * 4);
    const int64_t nb = ceil_div(n, SEL_TILE);
    int64_t* cgt = reinterpret_cast<int64_t*>(w + SEL_BINS * 4 + 64);
    int64_t* ceq = cgt + nb;
    int64_t* tmp = ceq + nb;  // SEL_SORT_MAX entries for the sorted path
    uint32_t* bitmap = nullptr;

    if (bitmap_ok && sel_sampled(scores, dtype, n, k)) {
        bitmap = reinterpret_cast<uint32_t*>(
            (reinterpret_cast<uintptr_t>(w + sel_ws_base(n)) + 15) & ~(uintptr_t)15);
        // expected sample keys among the top k, plus six standard deviations
        // and eight: P then keeps at least k keys unless the sample misleads
        const double mu = (double)k / (double)n * SEL_SAMPLE;
        const int rank = (int)(mu + 6.0 * sqrt(mu) + 8.0) + 1;
        SEL_DISPATCH(k_sel_sample, dim3(1), dim3(1024), 0, stream, scores, n, hist, st,
                     (uint32_t)k, rank);
        if (int r = check_launch("topk sample")) return r;
        const int64_t fb = ceil_div(nb, 4);
        SEL_DISPATCH(k_sel_filter, dim3((unsigned)(fb < 2048 ? fb : 2048)), dim3(256), 0, stream,
                     scores, n, nb, st, bitmap);
        if (int r = check_launch("topk filter")) return r;
    } else {
        hipLaunchKernelGGL(k_sel_init, dim3(1), dim3(256), 0, stream, hist, st, (uint32_t)k);
        if (int r = check_launch("topk init")) return r;
    }
    // digits of 11 bits; keys of fp16 scores have their low 13 bits zero: two
    // passes fix the rest
    const bool half = dtype == SSEQS_F16;
    int64_t hb = ceil_div(n, 256 * 16);
    unsigned hgrid = (unsigned)(hb < 4096 ? (hb > 0 ? hb : 1) : 4096);
    // fp16 scores at a 16-byte aligned address: eight per thread and load
    const bool h8 = half && (reinterpret_cast<uintptr_t>(scores) & 15) == 0;
    const _Float16* sh = static_cast<const _Float16*>(scores);
    for (int p = 0; p < (half ? 2 : 3); ++p) {
        if (h8)
            hipLaunchKernelGGL(k_sel_hist_h8, dim3(hgrid), dim3(256), 0, stream, sh, n, st, hist,
                               p, bitmap);
        else
            SEL_DISPATCH(k_sel_hist, dim3(hgrid), dim3(256), 0, stream, scores, n, st, hist, p,
                         bitmap);
        if (int r = check_launch("topk hist")) return r;
        SEL_DISPATCH(k_sel_pick, dim3(1), dim3(1024), 0, stream, st, hist, p);
        if (int r = check_launch("topk pick")) return r;
    }
    if (h8)
        hipLaunchKernelGGL(k_sel_count_h8, dim3(grid_cap(nb, 1)), dim3(256), 0, stream, sh, n, nb,
                           st, cgt, ceq, bitmap);
    else
        SEL_DISPATCH(k_sel_count, dim3(grid_cap(nb, 1)), dim3(256), 0, stream, scores, n,
                     nb, st, cgt, ceq, bitmap);
    if (int r = check_launch("topk count")) return r;
    hipLaunchKernelGGL(k_sel_scan, dim3(1), dim3(1024), 0, stream, cgt, ceq, nb);
    if (int r = check_launch("topk scan")) return r;
    int64_t* dst = sorted ? tmp : out_idx;
    if (h8)
        hipLaunchKernelGGL(k_sel_write_h8, dim3(grid_cap(nb, 1)), dim3(256), 0, stream, sh, n, nb,
                           st, cgt, ceq, k, dst, bitmap);
    else
        SEL_DISPATCH(k_sel_write, dim3(grid_cap(nb, 1)), dim3(256), 0, stream, scores, n,
                     nb, st, cgt, ceq, k, dst, bitmap);
    if (int r = check_launch("topk write")) return r;
    if (sorted) {
        int P = 1;
        while (P < k) P <<= 1;
        size_t lds = (size_t)P * 8;
        const void* sort_fn = dtype == SSEQS_F32   ? reinterpret_cast<const void*>(&k_sel_sort<SSEQS_F32>)
                              : dtype == SSEQS_F16 ? reinterpret_cast<const void*>(&k_sel_sort<SSEQS_F16>)
                                                   : reinterpret_cast<const void*>(&k_sel_sort<SSEQS_I32>);
        if (lds > 64 * 1024 &&
            hipFuncSetAttribute(sort_fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) !=
                hipSuccess)
            return fail(-3, "topk: cannot enable large LDS for the sort");
        SEL_DISPATCH(k_sel_sort, dim3(1), dim3(1024), lds, stream, scores, tmp, k, P,
                           out_idx);
        if (int r = check_launch("topk sort")) return r;
    }
    return 0;
}

// Checks shared by the two entry points; 1: nothing to do.
static int topk_check(int dtype, int64_t n, int64_t k, int sorted) {
    if (n < 0 || k < 0) return fail(-1, "topk: negative size");
    if (k > n) return fail(-1, "topk: k larger than the number of scores");
    if (dtype != SSEQS_F32 && dtype != SSEQS_F16 && dtype != SSEQS_I32)
        return fail(-1, "topk: unsupported dtype");
    if (k == 0) return 1;
    if (sorted && k > SEL_SORT_MAX) return fail(-1, "topk: sorted output limited to k <= 16384");
    if (sorted && n > 0xffffffffLL) return fail(-1, "topk: sorted output needs n < 2^32");
    return 0;
}

extern "C" int sseqs_topk(const void* scores, int dtype, int64_t n, int64_t k, int sorted,
                          int64_t* out_idx, void* ws, size_t ws_bytes, hipStream_t stream) {
    if (int r = topk_check(dtype, n, k, sorted)) return r < 0 ? r : 0;
    if (ws_bytes < sseqs_topk_ws_bytes(n)) return fail(-2, "topk: workspace too small");
    return topk_impl(scores, dtype, n, k, sorted, out_idx, ws, true, stream);
}

// ------------------------------------------------ sseqs_topk_noalloc --
//
// sseqs_topk on a library-owned scratch array instead of a caller
// workspace, for callers that cannot allocate.  `scratch` lives in device
// memory of every GPU the library runs on (one copy per device, held until
// the process ends).  Host code never passes the array's name to a kernel:
// the name is a host-side stand-in, so each device's address is looked up
// once with hipGetSymbolAddress (with that device current) and kept in
// g_scratch_ptr.  Every call on one device shares its copy; k_sel_init
// clears the histogram and state at the start of each call (a kernel, not
// hipMemsetAsync), and the count pass writes every per-tile counter, so
// nothing depends on the previous call's contents.  Calls that overlap on
// one device (two streams, or two threads) race on the array.

constexpr size_t NOALLOC_SCRATCH_BYTES = 512 * 1024;
static __device__ __align__(256) uint8_t scratch[NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Largest n whose workspace fits the scratch array.
int64_t noalloc_max_n() {
    const size_t fixed = (size_t)SEL_BINS * 4 + 64 + (size_t)SEL_SORT_MAX * 8 + 256;
    return (int64_t)((NOALLOC_SCRATCH_BYTES - fixed) / 16) * SEL_TILE;
}

// Device address of this device's scratch copy (looked up on first use).
int scratch_ptr(void** out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return fail(-4, "topk_noalloc: hipGetDevice failed");
    if (dev < 0 || dev >= kMaxDevices) return fail(-4, "topk_noalloc: device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail((int)(e != hipSuccess ? e : hipErrorInvalidSymbol),
                        std::string("topk_noalloc: hipGetSymbolAddress failed: ") +
                            hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}
}  // namespace

extern "C" int64_t sseqs_topk_noalloc_max_n(void) { return noalloc_max_n(); }

extern "C" int sseqs_topk_noalloc(const void* scores, int dtype, int64_t n, int64_t k, int sorted,
                                  int64_t* out_idx, hipStream_t stream) {
    if (n > noalloc_max_n())
        return fail(-1, "topk_noalloc: n = " + std::to_string(n) + " exceeds the scratch limit of " +
                            std::to_string(noalloc_max_n()) + " scores");
    void* ws = nullptr;
    if (int r = scratch_ptr(&ws)) return r;
    if (int r = topk_check(dtype, n, k, sorted)) return r < 0 ? r : 0;
    return topk_impl(scores, dtype, n, k, sorted, out_idx, ws, false, stream);
}

template <bool CUT, class... Args>
static int launch_segments(int dtype, unsigned grid, hipStream_t stream, Args... args) {
    const auto go = [&](auto kern) -> int {
        const size_t lds = CUT ? (size_t)8 * SEG_LIST : 0;
        if (CUT && hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return fail(-3, "topk_segments: cannot enable large LDS");
        hipLaunchKernelGGL(kern, dim3(grid), dim3(SEG_THREADS), lds, stream, args...);
        return check_launch("topk_segments");
    };
    if (dtype == SSEQS_F32) return go(&k_seg_topk<SSEQS_F32, CUT>);
    if (dtype == SSEQS_F16) return go(&k_seg_topk<SSEQS_F16, CUT>);
    return go(&k_seg_topk<SSEQS_I32, CUT>);
}

extern "C" int sseqs_topk_segments(const void* scores, int dtype, const int64_t* seg_begin,
                                   const int32_t* seg_n, const int32_t* seg_k,
                                   const int64_t* out_base, int64_t nseg, int max_k, int sorted,
                                   int drop_front, int drop_back, int add_begin,
                                   int64_t* out_idx, hipStream_t stream) {
    if (nseg < 0 || max_k < 0 || drop_front < 0 || drop_back < 0)
        return fail(-1, "topk_segments: negative size");
    if (dtype != SSEQS_F32 && dtype != SSEQS_F16 && dtype != SSEQS_I32)
        return fail(-1, "topk_segments: unsupported dtype");
    if (sorted && max_k > SEG_SORT_MAX)
        return fail(-1, "topk_segments: sorted output limited to k <= 4096 per segment");
    if (nseg == 0 || max_k == 0) return 0;
    if (!scores || !seg_begin || !seg_n || !seg_k || !out_base || !out_idx)
        return fail(-1, "topk_segments: null pointer");
    const unsigned grid = (unsigned)(nseg < 8192 ? nseg : 8192);
    if (!sorted && max_k >= SEG_CUT_K)
        return launch_segments<true>(dtype, grid, stream, scores, seg_begin, seg_n, seg_k, out_base, nseg,
                                     sorted, drop_front, drop_back, add_begin, out_idx);
    return launch_segments<false>(dtype, grid, stream, scores, seg_begin, seg_n, seg_k, out_base, nseg,
                                  sorted, drop_front, drop_back, add_begin, out_idx);
}
