// Token sampling on the device: HybridModel::Impl::sample_token
// (nexus/src/model/hybrid_model.cpp:2023-2099) -- temperature softmax,
// top-k, top-p, renormalize, one uniform draw, the first vocabulary index
// whose running sum reaches it -- so the logits never leave HBM.
//
// Three launches: the maximum logit, then e_i = expf((l_i - max) / T) into a
// scratch row with partial sums and the top-k candidates (k up to 64) or
// their counts, each over 64 blocks per sequence (k_sample_max,
// k_sample_exp; a gather launch for larger k up to 1024); then one block of
// 1024 threads per sequence (k_sample) for the selection and the draw.
// Latency bounds all of them: 8 rows of 128256 with k 40 and p 0.9 are 4 MB
// and take 20.9 us (2, 7 and 11), where a gather of its own, a sort with a
// barrier per stage and branching running sums took 47.6.  In k_sample,
// wavefront w owns the contiguous vocabulary chunk [w C, (w + 1) C) and
// walks it 64 consecutive entries at a time (coalesced), so wavefront order
// then iteration order then lane order is vocabulary order; ballots keep
// that order where it matters.  Later passes read p_i = e_i / sum.
//  - top-k (0 < k <= 1024, k < V): the candidates listed by k_sample_exp (k up
//    to 64) or gathered at a threshold; where neither fits, four 8-bit radix
//    passes over the bits of p_i (positive floats order as their bits) find
//    the k-th largest value.  Ties keep the lowest indices (the reference's
//    partial_sort leaves their order unspecified).  The candidates are
//    ordered in LDS (by counting up to 512, else bitonic; ties by index) and
//    the running sum is taken in that order; the renormalization and the
//    draw's scan run over the k survivors in index order, the reference's
//    own summation order.
//  - otherwise (no top-k, or k above 1024; with or without top-p): every
//    entry is a candidate.  A radix selection by counts finds the k-th
//    largest p, a radix selection by probability mass (exact 40-bit
//    fixed-point sums) finds where the running sum in descending order
//    first exceeds top_p; ties at either value keep the lowest indices.
//    The draw's scan runs over the kept entries in wavefront, iteration and
//    lane order with fp32 partial sums in a fixed order.
// The softmax denominator is a fixed-order sum (per block, then the blocks
// in order); the reference's is a sequential fp32 sum, so probabilities
// agree to rounding.
#include "nx_common.h"
#include "nx_kernels.h"

namespace nx {
namespace {

constexpr int kSmpThreads = 1024;
constexpr int kSmpMaxK = 1024;
constexpr int kSmpCand = kSmpCandMax;  // top-k candidates held in LDS
constexpr int kSmpThr = 8;      // candidate thresholds e >= exp(-D)
__constant__ float c_smp_D[kSmpThr] = {24.0f, 16.0f, 12.0f, 8.0f, 5.0f, 3.0f, 2.0f, 1.0f};

constexpr int kSmpWaves = kSmpThreads / 64;
constexpr int kSmpRankMax = 512;  // candidates ordered by counting
constexpr int kSmpPrune = 128;    // listed candidates (k <= 64) ordered without thinning them out first

__device__ inline float smp_wave_max(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}
template <class T>
__device__ inline T smp_wave_sum(T v) {
    for (int o = 32; o > 0; o >>= 1) v = v + __shfl_xor(v, o, 64);
    return v;
}
// inclusive prefix over the 64 lanes (Hillis-Steele, fixed order)
__device__ inline float smp_wave_scan(float x) {
    const int l = threadIdx.x & 63;
    for (int o = 1; o < 64; o <<= 1) {
        const float y = __shfl_up(x, o, 64);
        if (l >= o) x = x + y;
    }
    return x;
}
// lane j: x_0 + x_1 + ... + x_j, added in that order (no branch and no
// memory: 64 steps of a read and an add)
__device__ inline float smp_lane_cum(float x) {
    const int l = threadIdx.x & 63;
    float cum = 0.0f, mine = 0.0f;
#pragma unroll
    for (int j = 0; j < kWave; ++j) {
        cum += readlane_f(x, j);
        mine = l == j ? cum : mine;
    }
    return mine;
}
__device__ inline int popc_below(unsigned long long m, int l) {
    return __popcll(m & ((1ull << l) - 1ull));
}

// Prefix sums of one value per thread in thread order, fixed order of
// additions (a Hillis-Steele scan per wavefront, then the wavefront totals
// in order); wsum holds kSmpWaves + 1 entries.  Returns the exclusive
// prefix; *incl the inclusive one, *total the sum.
template <class T>
__device__ inline T smp_block_scan(T v, T* wsum, T* incl, T* total) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    T x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const T y = __shfl_up(x, o, 64);
        if (l >= o) x = x + y;
    }
    const T xp = __shfl_up(x, 1, 64);
    if (l == 63) wsum[w] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        T acc = T(0);
        for (int i = 0; i < kSmpWaves; ++i) {
            const T t = wsum[i];
            wsum[i] = acc;
            acc = acc + t;
        }
        wsum[kSmpWaves] = acc;
    }
    __syncthreads();
    const T ex = l == 0 ? wsum[w] : wsum[w] + xp;
    *incl = wsum[w] + x;
    *total = wsum[kSmpWaves];
    __syncthreads();
    return ex;
}

// One pass of a wavefront over its chunk [c0, c1): kSmpU loads per lane are
// requested before any is used (a block has only 16 wavefronts to hide the
// memory latency with), then use(i0, valid, value) runs for the 64-entry
// steps i0 in order (entry i0 + lane).  Indices past c1 load c1 - 1 and
// are passed as not valid.
constexpr int kSmpU = 16;
template <class Load, class Use>
__device__ inline void smp_pass(int c0, int c1, Load load, Use use) {
    const int l = threadIdx.x & 63;
    for (int base = c0; base < c1; base += 64 * kSmpU) {
        float v[kSmpU];
#pragma unroll
        for (int u = 0; u < kSmpU; ++u) v[u] = load(min(base + 64 * u + l, c1 - 1));
#pragma unroll
        for (int u = 0; u < kSmpU; ++u) use(base + 64 * u, base + 64 * u + l < c1, v[u]);
    }
}

// The first two passes over the vocabulary, spread over kSmpBlocks blocks
// per sequence (on the one block of k_sample they took 50 of its 85 us).
// k_sample_max writes the maximum logit of the entries of each block, dealt
// in runs of 64 to the blocks in turn; k_sample_exp takes the maximum of
// those (exact in any order).  Its block p = 4 w + q covers quarter q of
// k_sample wavefront w's chunk: it writes e_i = expf((l_i - max) / T) into the
// scratch row and its sum of e (per thread in index order, wavefront tree,
// wavefronts in order) and its candidates, or its counts at each candidate
// threshold.  k_sample adds the sums in block order.
constexpr int kSmpPThreads = 256, kSmpPWaves = kSmpPThreads / 64;
constexpr int kSmpPU = 8;  // entries per thread requested together
static_assert(kSmpBlocks == 4 * kSmpWaves && kSmpBlocks == 64, "four blocks per k_sample wavefront chunk, one per lane");
static_assert(kSmpCandOff == kSmpBlocks * (3 + kSmpThr), "partials: max, sum, counts, listed entries");
__device__ inline void smp_block_range(int V, int p, int& c0, int& c1) {
    const int C = ((V + kSmpWaves - 1) / kSmpWaves + 63) / 64 * 64, Q = C / 4;
    c0 = min((p / 4) * C + (p % 4) * Q, V);
    c1 = min(c0 + Q, V);
}

__global__ __launch_bounds__(kSmpPThreads) void k_sample_max(SampleArgs a) {
    __shared__ float wm[kSmpPWaves];
    const int p = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, l = tid & 63;
    const float* lg = a.logits + (size_t)b * a.ldl;
    float mx = -__builtin_inff();
    for (int i0 = 64 * (p + kSmpBlocks * (tid >> 6)) + l; i0 < a.V; i0 += kSmpPU * kSmpBlocks * kSmpPThreads) {
        float v[kSmpPU];  // requested together
#pragma unroll
        for (int q = 0; q < kSmpPU; ++q) v[q] = lg[min(i0 + q * kSmpBlocks * kSmpPThreads, a.V - 1)];
#pragma unroll
        for (int q = 0; q < kSmpPU; ++q)
            mx = i0 + q * kSmpBlocks * kSmpPThreads < a.V ? fmaxf(mx, v[q]) : mx;
    }
    mx = smp_wave_max(mx);
    if (l == 0) wm[tid >> 6] = mx;
    __syncthreads();
    if (tid == 0) {
        float m = wm[0];
        for (int j = 1; j < kSmpPWaves; ++j) m = fmaxf(m, wm[j]);
        a.part[(size_t)b * kSmpPartFloats + p] = m;
    }
}

// Top-k up to kSmpFastK: the k-th largest of the 64 blocks' maxima (as e) is
// a bound that at least k entries reach, known before this pass, so the pass
// itself lists the entries at or above it (and its ties; an e of 0 is never
// kept), kSmpSlot per block, in no order (k_sample orders them by value and
// index; a row of 128K independent entries lists about 1.6 k of them).  The
// maxima are of entries dealt to the blocks in turn, so that the bound does
// not depend on where the large ids sit (maxima of contiguous ranges, in a
// row whose logits fall with the id, put the bound at the last ranges'
// values).  A block that still holds more than kSmpSlot of them lists its
// own top k instead (smp_block_topk): a row's lists always fit, except
// where more values than that round to ties with a block's k-th.  8 rows of
// 128256, k 40: independent values 21 us; falling with the id 22, half of
// them masked 21, one run of large values over a flat rest 32, 10 finite
// values 17; where a full list sent the row to two passes on one CU 21, 85,
// 83, 73 and 599, and with thresholds and a gather launch for every row 46,
// 43, 47, 39 and 570.
constexpr int kSmpFastK = 64, kSmpSlot = kSmpCandMax / kSmpBlocks;
// The least e whose probability e / sum can round to that of this one (two
// roundings of e below it: quotients of one value lie within one ulp, at most
// 2^-23 of it, and e's steps are at least 2^-24): such entries are ties, which
// the lower index takes, so they are listed with it.
__device__ inline float smp_tie_floor(float e) {
    const uint32_t b = __builtin_bit_cast(uint32_t, e);
    return __builtin_bit_cast(float, b - min(b, 2u));
}
__device__ inline uint32_t smp_tie_bits(uint32_t b) { return b - min(b - 1u, 2u); }  // (b > 0)

// An overfull block's own candidates for the top k: every entry of its
// range that can be among the k largest of the range, ties in rounded
// probability by index.  Entries e[c0 + tid + 256 j] are this thread's (it
// wrote them); positive floats order as their bits.  A bisection over the
// bits finds a value that k to kSmpSlot entries reach, its ties included
// (about 8 counts, one barrier each); where equal values leave none, the
// range's k-th value and the lowest indices of it.  They replace the list
// there is; *nlist is their number, more than kSmpSlot if they do not fit.
constexpr int kSmpSel = 16;  // entries per thread held in registers
constexpr int kSmpProbe = 6; // bisection steps from one probe of a value to the next
__device__ inline void smp_block_topk(const float* e, int c0, int c1, float bound, int k, float* lv, int* li, int* nlist,
                               int (*wc)[kSmpPWaves]) {
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    auto at = [&](int i) {
        const float v = i < c1 ? e[i] : 0.0f;
        return v > 0.0f ? __builtin_bit_cast(uint32_t, v) : 0u;
    };
    uint32_t held[kSmpSel];
#pragma unroll
    for (int q = 0; q < kSmpSel; ++q) held[q] = at(c0 + tid + kSmpPThreads * q);
    int par = 0;
    auto meet = [&](uint32_t c, auto op) {  // over the block; the two buffers alternate, so one barrier is enough
        for (int o = 32; o > 0; o >>= 1) c = op(c, __shfl_xor(c, o, 64));
        if (l == 0) wc[par][w] = (int)c;
        __syncthreads();
        c = (uint32_t)wc[par][0];
        for (int j = 1; j < kSmpPWaves; ++j) c = op(c, (uint32_t)wc[par][j]);
        par ^= 1;
        return c;
    };
    auto each = [&](auto use) {
#pragma unroll
        for (int q = 0; q < kSmpSel; ++q) use(held[q]);
        for (int i = c0 + tid + kSmpPThreads * kSmpSel; i < c1; i += kSmpPThreads) use(at(i));
    };
    auto reach = [&](uint32_t x) {  // entries with bits >= x
        uint32_t c = 0;
        each([&](uint32_t v) { c += v >= x; });
        return (int)meet(c, [](uint32_t p, uint32_t q) { return p + q; });
    };
    auto next_below = [&](uint32_t x) {  // the largest bits < x
        uint32_t c = 0;
        each([&](uint32_t v) { c = v < x ? max(c, v) : c; });
        return meet(c, [](uint32_t p, uint32_t q) { return max(p, q); });
    };
    auto append = [&](uint32_t v, int i) {
        const int n = atomicAdd(nlist, 1);
        if (n < kSmpSlot) {
            lv[n] = __builtin_bit_cast(float, v);
            li[n] = i;
        }
    };
    auto append_from = [&](uint32_t x) {
#pragma unroll
        for (int q = 0; q < kSmpSel; ++q)
            if (held[q] >= x) append(held[q], c0 + tid + kSmpPThreads * q);
        for (int i = c0 + tid + kSmpPThreads * kSmpSel; i < c1; i += kSmpPThreads) {
            const uint32_t v = at(i);
            if (v >= x) append(v, i);
        }
    };
    uint32_t lo = max(__builtin_bit_cast(uint32_t, bound), 1u), hi = 0x3F800001u;  // reached by at least k, by none (e <= 1)
    uint32_t from = 0;
    for (int step = 0; hi - lo > 1u; ++step) {
        // now and then, first of all, the largest value below hi: where few
        // values are far apart, or a flat row's are all one, that is the k-th
        const bool probe = step % kSmpProbe == 0;
        const uint32_t mid = probe ? max(next_below(hi), lo) : lo + (hi - lo) / 2u;
        const int c = reach(mid);
        if (c < k) {
            hi = mid;
        } else if (c > kSmpSlot || reach(smp_tie_bits(mid)) > kSmpSlot) {
            lo = mid;
            if (probe) hi = mid + 1u;
        } else {
            from = smp_tie_bits(mid);
            break;
        }
    }
    if (tid == 0) *nlist = 0;  // (every thread is past a count's barrier, so past reading it)
    __syncthreads();
    if (from) {
        append_from(from);
    } else {
        // lo is the k-th value: the entries above it, and of it and of the
        // two values that may round to its probability the lowest indices
        // (as many as the values that surely have a larger one leave)
        append_from(lo + 1u);
        const int need = k - reach(lo + 3u);
        for (uint32_t x = lo; x >= smp_tie_bits(lo); --x) {
            int run = 0;
            for (int i0 = c0; i0 < c1 && run < need; i0 += kSmpPThreads) {
                const uint32_t v = at(i0 + tid);
                const unsigned long long m = __ballot(v == x);
                if (l == 0) wc[par][w] = __popcll(m);
                __syncthreads();
                int before = run + popc_below(m, l);
                for (int j = 0; j < kSmpPWaves; ++j) {
                    before += j < w ? wc[par][j] : 0;
                    run += wc[par][j];
                }
                par ^= 1;
                if (v == x && before < need) append(v, i0 + tid);
            }
        }
    }
    __syncthreads();
}

__device__ inline bool smp_fast(const SampleArgs& a) { return a.top_k > 0 && a.top_k < a.V && a.top_k <= kSmpFastK; }

template <bool FAST>
__global__ __launch_bounds__(kSmpPThreads) void k_sample_exp(SampleArgs a) {
    __shared__ int nlist;
    __shared__ float wm[kSmpPWaves];
    __shared__ int wc[kSmpThr][kSmpPWaves];
    const int p = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    const float* lg = a.logits + (size_t)b * a.ldl;
    float* e = a.scratch + (size_t)b * a.V;
    float* pt = a.part + (size_t)b * kSmpPartFloats;
    int c0, c1;
    smp_block_range(a.V, p, c0, c1);
    // the first entries are requested with the blocks' maxima, from which
    // every wavefront takes the sequence's
    float lv[kSmpPU];
    auto request = [&](int i0) {
#pragma unroll
        for (int q = 0; q < kSmpPU; ++q) lv[q] = c0 < c1 ? lg[min(i0 + q * kSmpPThreads, c1 - 1)] : 0.0f;
    };
    const float bm = pt[l];
    request(c0 + tid);
    const float mx = smp_wave_max(bm);
    const float T = a.temperature;
    float bound = 0.0f;
    if constexpr (FAST) {
        const float be = expf((bm - mx) / T);
        int rank = 0;
#pragma unroll 16
        for (int j = 0; j < kWave; ++j) {
            const float o = readlane_f(be, j);
            rank += o > be || (o == be && j < l);
        }
        // (no lane has the rank where maxima are NaN: nothing is listed, the
        // count says so)
        const unsigned long long at = __ballot(rank == a.top_k - 1);
        bound = at ? smp_tie_floor(readlane_f(be, __ffsll((long long)at) - 1)) : __builtin_inff();
        if (tid == 0) nlist = 0;
        __syncthreads();
    }
    float sum = 0.0f, thr[kSmpThr];
    int cnt[kSmpThr];
    if constexpr (!FAST)
#pragma unroll
        for (int j = 0; j < kSmpThr; ++j) {
            thr[j] = expf(-c_smp_D[j]);
            cnt[j] = 0;
        }
    float* lp = pt + kSmpCandOff + kSmpSlot * p;  // the block's list
    int* li = reinterpret_cast<int*>(pt + kSmpCandOff + kSmpCandMax) + kSmpSlot * p;
    for (int i0 = c0 + tid; i0 < c1; i0 += kSmpPU * kSmpPThreads) {
        if (i0 != c0 + tid) request(i0);
#pragma unroll
        for (int q = 0; q < kSmpPU; ++q) {
            const int i = i0 + q * kSmpPThreads;
            if (i >= c1) break;
            const float v = expf((lv[q] - mx) / T);
            e[i] = v;
            sum += v;
            if constexpr (FAST) {
                if (v >= bound && v > 0.0f) {
                    const int at = atomicAdd(&nlist, 1);
                    if (at < kSmpSlot) {
                        lp[at] = v;
                        li[at] = i;
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < kSmpThr; ++j) cnt[j] += v >= thr[j];
            }
        }
    }
    sum = smp_wave_sum(sum);
    if constexpr (!FAST)
#pragma unroll
        for (int j = 0; j < kSmpThr; ++j) {
            const int c = smp_wave_sum(cnt[j]);
            if (l == 0) wc[j][w] = c;
        }
    if (l == 0) wm[w] = sum;
    __syncthreads();
    if (tid == 0) {
        float s = 0.0f;
        for (int j = 0; j < kSmpPWaves; ++j) s += wm[j];
        pt[kSmpBlocks + p] = s;
    }
    if constexpr (FAST) {
        if (nlist > kSmpSlot) smp_block_topk(e, c0, c1, bound, a.top_k, lp, li, &nlist, wc);
        if (tid == 0) pt[(2 + kSmpThr) * kSmpBlocks + p] = (float)nlist;
    }
    if (!FAST && tid < kSmpThr) {
        int c = 0;
        for (int j = 0; j < kSmpPWaves; ++j) c += wc[tid][j];
        pt[2 * kSmpBlocks + kSmpThr * p + tid] = (float)c;  // exact: c <= V < 2^24
    }
}

// Top-k (k <= kSmpMaxK) with a candidate threshold that fits kSmpCand: the
// threshold pick of k_sample (the smallest D whose count of e >= exp(-D) is
// at least k), then block p writes the entries of its range at or above it,
// in index order, at the sum of the earlier blocks' counts -- the candidate
// list k_sample would gather with one pass over the row on one CU.
__global__ __launch_bounds__(kSmpPThreads) void k_sample_gather(SampleArgs a) {
    __shared__ int wsum[kSmpPWaves];
    __shared__ int pk[2];
    __shared__ float sm;
    const int p = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    if (!(a.top_k > 0 && a.top_k < a.V && a.top_k <= kSmpMaxK)) return;
    const float* e = a.scratch + (size_t)b * a.V;
    float* pt = a.part + (size_t)b * kSmpPartFloats;
    if (w == 0) {
        // lane q: block q's counts; totals in a fixed order (exact integers)
        int pick = -1, base = 0;
        for (int j = 0; j < kSmpThr; ++j) {
            const int c = (int)pt[2 * kSmpBlocks + kSmpThr * l + j];
            const int tot = smp_wave_sum(c);
            if (tot >= a.top_k) {
                pick = tot <= kSmpCand ? j : -2;
                base = smp_wave_sum(l < p ? c : 0);
            }
        }
        if (l == 0) {
            pk[0] = pick;
            pk[1] = base;
        }
    }
    if (tid == 0) {
        float acc = 0.0f;
        for (int j = 0; j < kSmpBlocks; ++j) acc += pt[kSmpBlocks + j];
        sm = acc;
    }
    __syncthreads();
    const int pick = pk[0];
    if (pick < 0) return;
    int base = pk[1];
    const float sum_e = sm, th = expf(-c_smp_D[pick]);
    float* cp = pt + kSmpCandOff;
    int* ci = reinterpret_cast<int*>(cp + kSmpCandMax);
    int c0, c1;
    smp_block_range(a.V, p, c0, c1);
    for (int i0 = c0; i0 < c1; i0 += kSmpPThreads) {
        const int i = i0 + tid;
        const float ev = i < c1 ? e[i] : 0.0f;
        const bool keep = i < c1 && ev >= th;
        const unsigned long long km = __ballot(keep);
        if (l == 0) wsum[w] = __popcll(km);
        __syncthreads();
        int before = 0, all = 0;
        for (int j = 0; j < kSmpPWaves; ++j) {
            before += j < w ? wsum[j] : 0;
            all += wsum[j];
        }
        if (keep) {
            const int at = base + before + popc_below(km, l);
            cp[at] = ev / sum_e;
            ci[at] = i;
        }
        base += all;
        __syncthreads();
    }
}

// More listed candidates than counting orders (kSmpPrune): those that can
// be among the k <= kSmpFastK largest, at most kSmpPrune, compacted in
// place; returns how many.  A bisection over the values (4 per thread, one
// barrier each) finds one that k to kSmpPrune candidates reach; where equal
// values leave none, another over the indices of the k-th value's ties.
// (Counting the predecessors of 512 takes about 9 us, of 128 one; a bitonic
// sort of 2560, a flat row's, 100: 78 barriers.)
__device__ inline int smp_prune(float* cand_p, int* cand_i, int n, int k, int V, int (*wi)[kSmpWaves + 1]) {
    constexpr int H = kSmpCand / kSmpThreads;
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    uint32_t v[H];  // bits of p, 0 where it is not above 0 (never kept)
    int ix[H];
#pragma unroll
    for (int q = 0; q < H; ++q) {
        const int j = tid + kSmpThreads * q;
        const float p = j < n ? cand_p[j] : 0.0f;
        v[q] = p > 0.0f ? __builtin_bit_cast(uint32_t, p) : 0u;
        ix[q] = j < n ? cand_i[j] : 0;
    }
    int par = 0;
    auto count = [&](auto in) {  // (the two buffers alternate, so one barrier is enough)
        int c = 0;
#pragma unroll
        for (int q = 0; q < H; ++q) c += __popcll(__ballot(in(v[q], ix[q])));
        if (l == 0) wi[par][w] = c;
        __syncthreads();
        int s = 0;
        for (int j = 0; j < kSmpWaves; ++j) s += wi[par][j];
        par ^= 1;
        return s;
    };
    auto reach = [&](uint32_t x) { return count([=](uint32_t b, int) { return b >= x; }); };
    auto next_below = [&](uint32_t x) {  // the largest value < x
        uint32_t c = 0;
#pragma unroll
        for (int q = 0; q < H; ++q) c = v[q] < x ? max(c, v[q]) : c;
        for (int o = 32; o > 0; o >>= 1) c = max(c, (uint32_t)__shfl_xor(c, o, 64));
        if (l == 0) wi[par][w] = (int)c;
        __syncthreads();
        for (int j = 0; j < kSmpWaves; ++j) c = max(c, (uint32_t)wi[par][j]);
        par ^= 1;
        return c;
    };
    uint32_t lo = 1u, hi = 0x3F800001u;  // reached by more than kSmpPrune, by none (p <= 1)
    int below = V;                       // of the entries of value lo, those with a lower index
    if (reach(1u) > kSmpPrune) {
        bool found = false;
        for (int step = 1; hi - lo > 1u && !found; ++step) {
            const bool probe = step % kSmpProbe == 0;  // as in smp_block_topk
            const uint32_t mid = probe ? max(next_below(hi), lo) : lo + (hi - lo) / 2u;
            const int c = reach(mid);
            if (c < k) {
                hi = mid;
            } else {
                lo = mid;
                found = c <= kSmpPrune;
                if (probe) hi = mid + 1u;
            }
        }
        if (!found) {
            const uint32_t t = lo;
            const int above = reach(t + 1u);
            int a0 = 0;  // fewer than k - above ties have a lower index
            while (below - a0 > 1) {
                const int mid = a0 + (below - a0) / 2;
                const int c = above + count([=](uint32_t b, int i) { return b == t && i < mid; });
                if (c < k) {
                    a0 = mid;
                } else {
                    below = mid;
                    if (c <= kSmpPrune) break;
                }
            }
        }
    }
    int m = 0, in = 0, total = 0;
#pragma unroll
    for (int q = 0; q < H; ++q) m += v[q] > lo || (v[q] == lo && ix[q] < below);
    int o = smp_block_scan<int>(m, wi[2], &in, &total);
#pragma unroll
    for (int q = 0; q < H; ++q)
        if (v[q] > lo || (v[q] == lo && ix[q] < below)) {
            cand_p[o] = __builtin_bit_cast(float, v[q]);
            cand_i[o] = ix[q];
            ++o;
        }
    return total;
}

__global__ __launch_bounds__(kSmpThreads) void k_sample(SampleArgs a) {
    __shared__ float wf[kSmpWaves + 1];
    __shared__ int wi[4][kSmpWaves + 1];
    __shared__ int hist[256];
    __shared__ int sel;
    __shared__ __align__(16) float cand_p[kSmpCand];
    __shared__ __align__(16) int cand_i[kSmpCand];
    __shared__ int ord[kSmpCand];
    __shared__ int tcnt[kSmpThr][kSmpWaves + 1];
    const int b = blockIdx.x, tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, V = a.V;
    const float* e = a.scratch + (size_t)b * V;
    const int C = ((V + kSmpWaves - 1) / kSmpWaves + 63) / 64 * 64;
    const int c0 = min(w * C, V), c1 = min(c0 + C, V);

    // the e row and its sum (the blocks' sums in block order, in every
    // wavefront), from k_sample_max / k_sample_exp
    const float* pt = a.part + (size_t)b * kSmpPartFloats;
    const bool fast = smp_fast(a);
    const float bsum = pt[kSmpBlocks + l];
    const int cl = fast ? (int)pt[(2 + kSmpThr) * kSmpBlocks + l] : 0;
    float sum_e = 0.0f;
#pragma unroll
    for (int j = 0; j < kSmpBlocks; ++j) sum_e += readlane_f(bsum, j);
    // per wavefront chunk the entries at or above each candidate threshold
    // exp(-D): from k_sample_exp, or (fast, lists overflowed) counted here
    auto threshold_counts = [&] {
        if (!fast) {
            if (tid < kSmpThr * kSmpWaves) {
                const int j = tid / kSmpWaves, ww = tid % kSmpWaves;
                float c = 0.0f;
                for (int q = 0; q < 4; ++q) c += pt[2 * kSmpBlocks + kSmpThr * (4 * ww + q) + j];
                tcnt[j][ww] = (int)c;
            }
        } else {
            int cnt[kSmpThr];
            float thr[kSmpThr];
#pragma unroll
            for (int j = 0; j < kSmpThr; ++j) {
                cnt[j] = 0;
                thr[j] = expf(-c_smp_D[j]);
            }
            smp_pass(c0, c1, [&](int i) { return e[i]; }, [&](int, bool in, float ev) {
#pragma unroll
                for (int j = 0; j < kSmpThr; ++j) cnt[j] += __popcll(__ballot(in && ev >= thr[j]));
            });
            if (l == 0)
#pragma unroll
                for (int j = 0; j < kSmpThr; ++j) tcnt[j][w] = cnt[j];
        }
        __syncthreads();
    };
    // the draw: fixed, per sequence, or keyed by the sequence's position
    float u = a.u_fixed;
    if (u < 0.0f) {
        if (a.u) {
            u = a.u[b];
        } else {
            const uint32_t x = (uint32_t)rand_at(stream_key(a.key, (uint32_t)b), (uint64_t)a.pos[b]);
            u = (float)x / 4294967296.0f;
            if (u >= 1.0f) u = 0.99999994f;  // the largest float below 1
        }
    }

    bool listed = false;
    int n = 0;
    if (fast) {
        // the lists of k_sample_exp, one after another: block p's at the sum
        // of the earlier blocks' counts (wavefront w copies blocks w, w + 16,
        // ...; every wavefront holds all the counts)
        int in = cl;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(in, o, 64);
            if (l >= o) in += y;
        }
        n = __builtin_amdgcn_readlane(in, 63);
        // (fewer than k are every entry whose e is not 0; none: NaN or
        // infinite maxima)
        listed = !__any(cl > kSmpSlot) && n > 0;
        if (listed) {
            const float* lp = pt + kSmpCandOff;
            const int* li = reinterpret_cast<const int*>(lp + kSmpCandMax);
#pragma unroll
            for (int q = 0; q < kSmpBlocks / kSmpWaves; ++q) {
                const int p = w + kSmpWaves * q, c = __builtin_amdgcn_readlane(cl, p),
                          at = __builtin_amdgcn_readlane(in, p) - c;
                if (l < c) {
                    cand_p[at + l] = lp[kSmpSlot * p + l] / sum_e;
                    cand_i[at + l] = li[kSmpSlot * p + l];
                }
            }
            if (n > kSmpPrune) {
                __syncthreads();
                n = smp_prune(cand_p, cand_i, n, a.top_k, V, wi);
            }
        }
    }

    if (a.top_k > 0 && a.top_k < V && a.top_k <= kSmpMaxK) {
        if (!listed) {
        threshold_counts();
        // candidates: the entries with e >= exp(-D) for the smallest D whose
        // count is at least k (they hold the top k: p orders as e), if that
        // count fits in LDS; otherwise a radix selection over all of p finds
        // exactly k
        if (w == 0) {
            // lane j < kSmpThr: threshold j's exclusive prefix over the
            // wavefronts and its total; D decreases with j, so the pick is
            // the last threshold whose count reaches k (-2 if that count
            // does not fit the candidate list, -1 if none reaches k)
            int tot = 0;
            if (l < kSmpThr) {
                for (int q = 0; q < kSmpWaves; ++q) {
                    const int c = tcnt[l][q];
                    tcnt[l][q] = tot;
                    tot += c;
                }
                tcnt[l][kSmpWaves] = tot;
            }
            const unsigned long long ok = __ballot(l < kSmpThr && tot >= a.top_k);
            const int jm = ok ? 63 - __clzll(ok) : 0;
            const int tj = __shfl(tot, jm, kWave);
            if (l == 0) wi[0][3] = ok ? (tj <= kSmpCand ? jm : -2) : -1;
        }
        __syncthreads();
        const int pick = wi[0][3];
        if (pick >= 0 && fast) {
            // (a row whose lists overflowed) the same candidates, gathered here
            n = tcnt[pick][kSmpWaves];
            const float th = expf(-c_smp_D[pick]);
            int at0 = tcnt[pick][w];
            smp_pass(c0, c1, [&](int i) { return e[i]; }, [&](int i0, bool in, float ev) {
                const bool keep = in && ev >= th;
                const unsigned long long km = __ballot(keep);
                if (keep) {
                    cand_p[at0 + popc_below(km, l)] = ev / sum_e;
                    cand_i[at0 + popc_below(km, l)] = i0 + l;
                }
                at0 += __popcll(km);
            });
        } else if (pick >= 0) {
            // the candidates gathered by k_sample_gather, in index order
            n = tcnt[pick][kSmpWaves];
            const float* cp = a.part + (size_t)b * kSmpPartFloats + kSmpCandOff;
            const int* ci = reinterpret_cast<const int*>(cp + kSmpCandMax);
            for (int j = tid; j < n; j += kSmpThreads) {
                cand_p[j] = cp[j];
                cand_i[j] = ci[j];
            }
        } else {
        // the k-th largest p: radix select over its bits, 8 at a time
        uint32_t prefix = 0, pmask = 0;
        int need = a.top_k;  // still to take at or below the prefix
        for (int sh = 24; sh >= 0; sh -= 8) {
            for (int j = tid; j < 256; j += kSmpThreads) hist[j] = 0;
            __syncthreads();
            smp_pass(c0, c1, [&](int i) { return e[i]; }, [&](int, bool ok, float ev) {
                const uint32_t bits = __builtin_bit_cast(uint32_t, ev / sum_e);
                if (ok && (bits & pmask) == prefix) atomicAdd(&hist[(bits >> sh) & 0xFF], 1);
            });
            __syncthreads();
            if (tid == 0) {
                int bin = 255, above = 0;
                for (; bin > 0; --bin) {
                    if (above + hist[bin] >= need) break;
                    above += hist[bin];
                }
                wi[0][0] = bin;
                wi[0][1] = above;
            }
            __syncthreads();
            prefix |= (uint32_t)wi[0][0] << sh;
            pmask |= 0xFFu << sh;
            need -= wi[0][1];
            __syncthreads();
        }
        // per wavefront: values above the k-th and ties with it
        int nab = 0, ntie = 0;
        smp_pass(c0, c1, [&](int i) { return e[i]; }, [&](int, bool ok, float ev) {
            const uint32_t bits = __builtin_bit_cast(uint32_t, ev / sum_e);
            nab += ok && bits > prefix;
            ntie += ok && bits == prefix;
        });
        nab = smp_wave_sum(nab);
        ntie = smp_wave_sum(ntie);
        if (l == 0) {
            wi[1][w] = nab;
            wi[2][w] = ntie;
        }
        __syncthreads();
        if (tid == 0) {  // ties before each wavefront, and its first output slot
            int tb = 0, ob = 0;
            for (int j = 0; j < kSmpWaves; ++j) {
                const int nt = wi[2][j];
                wi[2][j] = tb;
                wi[3][j] = ob;
                ob += wi[1][j] + max(0, min(nt, need - tb));
                tb += nt;
            }
            wi[0][2] = ob;  // survivors
        }
        __syncthreads();
        // gather the survivors in index order
        int trun = wi[2][w], orun = wi[3][w];
        smp_pass(c0, c1, [&](int i) { return e[i]; }, [&](int i0, bool in, float ev) {
            const float p = ev / sum_e;
            const uint32_t bits = __builtin_bit_cast(uint32_t, p);
            const bool tie = in && bits == prefix;
            const unsigned long long tm = __ballot(tie);
            const bool keep = in && (bits > prefix || (tie && trun + popc_below(tm, l) < need));
            const unsigned long long km = __ballot(keep);
            const int at = orun + popc_below(km, l);
            if (keep && at < kSmpMaxK) {
                cand_p[at] = p;
                cand_i[at] = i0 + l;
            }
            trun += __popcll(tm);
            orun += __popcll(km);
        });
        n = min(wi[0][2], kSmpMaxK);
        }
        }
        __syncthreads();
        // descending order of p (ties by index): up to kSmpRankMax candidates
        // by counting, each thread its candidate's predecessors (45 barriers of
        // a sort over 512 are 11 us, the counts 1); more by a bitonic sort of
        // positions 0..n-1 over the next power of two, padding sorting last.
        // The first k are the top k, then top-p cuts along the same order.
        const int kk = min(a.top_k, n);
        int np2 = 1;
        while (np2 < n) np2 <<= 1;
        if (n > kk || a.top_p < 1.0f || fast) {
            if (n <= kSmpRankMax) {
                if (tid < n) ord[tid] = tid;  // (stands where values are NaN)
                if (tid < 4) cand_p[n + tid] = -1.0f;  // no predecessor of any
                __syncthreads();
                int rank = 0;
                if (tid < n) {
                    const float p = cand_p[tid];
                    const int at = cand_i[tid];
                    for (int x = 0; x < n; x += 4) {
                        const float4 px = *reinterpret_cast<const float4*>(&cand_p[x]);
                        const int4 ix = *reinterpret_cast<const int4*>(&cand_i[x]);
                        rank += px.x > p || (px.x == p && ix.x < at);
                        rank += px.y > p || (px.y == p && ix.y < at);
                        rank += px.z > p || (px.z == p && ix.z < at);
                        rank += px.w > p || (px.w == p && ix.w < at);
                    }
                }
                __syncthreads();
                if (tid < n) ord[rank] = tid;
                __syncthreads();
            } else {
                for (int j = tid; j < np2; j += kSmpThreads) ord[j] = j;
                __syncthreads();
                auto before = [&](int x, int y) {  // x sorts before y
                    if (x >= n) return false;
                    if (y >= n) return true;
                    return cand_p[x] > cand_p[y] || (cand_p[x] == cand_p[y] && cand_i[x] < cand_i[y]);
                };
                for (int k2 = 2; k2 <= np2; k2 <<= 1)
                    for (int j = k2 >> 1; j > 0; j >>= 1) {
                        for (int x = tid; x < np2; x += kSmpThreads) {
                            const int y = x ^ j;
                            if (y > x) {
                                const int ox = ord[x], oy = ord[y];
                                const bool up = (x & k2) == 0;
                                if (up ? before(oy, ox) : before(ox, oy)) {
                                    ord[x] = oy;
                                    ord[y] = ox;
                                }
                            }
                        }
                        __syncthreads();
                    }
            }
            // top-p: the running sum in sorted order by one wavefront (lane
            // j holds entry j, read in order), then the entries past the cut
            // are cleared by the block
            if (w == 0) {
                int cut = kk;
                if (a.top_p < 1.0f) {
                    if (kk <= kWave) {
                        const float pv = l < kk ? cand_p[ord[l]] : 0.0f;
                        const unsigned long long over = __ballot(smp_lane_cum(pv) > a.top_p && l < kk);
                        if (over) cut = __ffsll((long long)over);
                    } else {
                        float cum = 0.0f;
                        for (int j = 0; j < kk; ++j) {
                            cum += cand_p[ord[j]];
                            if (cum > a.top_p) {
                                cut = j + 1;
                                break;
                            }
                        }
                    }
                }
                if (l == 0) wi[0][0] = cut;
            }
            __syncthreads();
            const int cut = wi[0][0];
            if (fast) {
                // at most 64 kept: one wavefront brings them into index order
                // (a value of 0 is not kept), where the code below reads them
                if (w == 0) {
                    const int o = l < cut ? ord[l] : 0;
                    const float pv = l < cut ? cand_p[o] : 0.0f;
                    const int iv = cand_i[o];
                    const bool keep = pv > 0.0f;
                    const unsigned long long km = __ballot(keep);
                    int at = 0;
#pragma unroll 8
                    for (int j = 0; j < kWave; ++j) at += (km >> j & 1) && __builtin_amdgcn_readlane(iv, j) < iv;
                    if (keep) {
                        cand_p[at] = pv;
                        cand_i[at] = iv;
                    }
                    if (l == 0) wi[0][2] = __popcll(km);
                }
            } else {
                for (int j = cut + tid; j < n; j += kSmpThreads) cand_p[ord[j]] = 0.0f;
            }
            __syncthreads();
        }
        // the kept entries (at most k) in index order, compacted in parallel
        // (thread t holds candidates 4t .. 4t+3), then renormalized and drawn
        // from by one lane in that order
        int ktot = wi[0][2];
        if (!fast) {
        int nk = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) nk += 4 * tid + q < n && cand_p[4 * tid + q] > 0.0f;
        int kin = 0;
        const int kat = smp_block_scan<int>(nk, wi[1], &kin, &ktot);
        {
            int o = kat;
            float kp[4];
            int ki[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = 4 * tid + q;
                kp[q] = j < n ? cand_p[j] : 0.0f;
                ki[q] = j < n ? cand_i[j] : 0;
            }
            __syncthreads();  // the candidate arrays are rewritten in place
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (kp[q] > 0.0f) {
                    cand_p[o] = kp[q];
                    cand_i[o] = ki[q];
                    ++o;
                }
        }
        __syncthreads();
        }
        // renormalization and draw by one wavefront, in index order (lane j
        // holds kept entry j when there are at most 64, read in order)
        if (w == 0) {
            const bool lanes = ktot <= kWave;
            const float pv = lanes && l < ktot ? cand_p[l] : 0.0f;
            const int iv = lanes && l < ktot ? cand_i[l] : 0;
            int tok = V - 1;
            if (lanes) {
                const float cum = smp_lane_cum(pv);
                const float sm = readlane_f(cum, 63), r = u * sm;  // (lanes past ktot add zeros)
                const unsigned long long hit = __ballot(cum >= r && l < ktot);
                if (sm <= 0.0f || r <= 0.0f) tok = 0;  // nothing kept, or the running sum reaches r = 0 at index 0
                else if (hit) tok = __builtin_amdgcn_readlane(iv, __ffsll((long long)hit) - 1);
            } else {
                float sm = 0.0f;
                for (int j = 0; j < ktot; ++j) sm += cand_p[j];
                const float r = u * sm;
                if (sm <= 0.0f || r <= 0.0f) {
                    tok = 0;
                } else {
                    float cum = 0.0f;
                    for (int j = 0; j < ktot; ++j) {
                        cum += cand_p[j];
                        if (cum >= r) {
                            tok = cand_i[j];
                            break;
                        }
                    }
                }
            }
            if (l == 0) sel = tok;
        }
        __syncthreads();
    } else {
        // Every entry is a candidate: no top-k, or top-k above the candidate
        // list (kSmpMaxK), each with or without top-p.  A top-k cut keeps the
        // entries above the k-th largest p and, of the entries equal to it,
        // the lowest indices (radix selection of the k-th value by counts).
        // A top-p cut keeps, in descending order of p (ties by index), the
        // entries up to the first whose running sum exceeds top_p (radix
        // selection of that value by probability mass; the masses are summed
        // as 40-bit fixed-point integers, exact and independent of order,
        // where the reference adds fp32 in its sorted order).  The kept
        // entries are renormalized and drawn from in vocabulary order.
        const bool use_k = a.top_k > 0 && a.top_k < V;
        const bool use_p = a.top_p < 1.0f;
        // --- top-k: the k-th largest p (bits kb) and how many of its ties to keep
        uint32_t kb = 0;
        int kneed = 0;
        if (use_k) {
            uint32_t prefix = 0, pmask = 0;
            int need = a.top_k;
            for (int sh = 24; sh >= 0; sh -= 8) {
                for (int j2 = tid; j2 < 256; j2 += kSmpThreads) hist[j2] = 0;
                __syncthreads();
                smp_pass(c0, c1, [&](int i) { return e[i]; }, [&](int, bool ok, float ev) {
                    const uint32_t bits = __builtin_bit_cast(uint32_t, ev / sum_e);
                    if (ok && (bits & pmask) == prefix) atomicAdd(&hist[(bits >> sh) & 0xFF], 1);
                });
                __syncthreads();
                if (tid == 0) {
                    int bin = 255, above = 0;
                    for (; bin > 0; --bin) {
                        if (above + hist[bin] >= need) break;
                        above += hist[bin];
                    }
                    wi[0][0] = bin;
                    wi[0][1] = above;
                }
                __syncthreads();
                prefix |= (uint32_t)wi[0][0] << sh;
                pmask |= 0xFFu << sh;
                need -= wi[0][1];
                __syncthreads();
            }
            kb = prefix;
            kneed = need;
        }
        // tie ranks in vocabulary order: each wavefront's count of ties, then
        // the exclusive prefix over the wavefronts (ranks[w])
        auto wave_base = [&](int cnt, int* base) {
            cnt = smp_wave_sum(cnt);
            if (l == 0) base[w] = cnt;
            __syncthreads();
            if (tid == 0) {
                int acc = 0;
                for (int q = 0; q < kSmpWaves; ++q) {
                    const int c = base[q];
                    base[q] = acc;
                    acc += c;
                }
                base[kSmpWaves] = acc;
            }
            __syncthreads();
            return base[w];
        };
        int ktb = 0;
        if (use_k) {
            int cnt = 0;
            smp_pass(c0, c1, [&](int i) { return e[i]; }, [&](int, bool ok, float ev) {
                cnt += ok && __builtin_bit_cast(uint32_t, ev / sum_e) == kb;
            });
            ktb = wave_base(cnt, wi[1]);
        }
        // keep-by-k of the 64 entries of one step (krun: ties of kb before them)
        auto kept_k = [&](bool ok, uint32_t bits, int& krun) {
            const bool tie = ok && use_k && bits == kb;
            const unsigned long long tm = __ballot(tie);
            const bool keep = ok && (!use_k || bits > kb || (tie && krun + popc_below(tm, l) < kneed));
            krun += __popcll(tm);
            return keep;
        };
        // --- top-p over the entries top-k keeps: the value pb at which the
        // running mass first exceeds top_p, the mass above it, and how many
        // of its ties to keep
        __shared__ unsigned long long hmass[256];
        __shared__ int pinfo[1];
        bool pcut = false;
        uint32_t pb = 0;
        int pneed = 0;
        if (use_p) {
            const unsigned long long tp = (unsigned long long)((double)a.top_p * 1099511627776.0);
            uint32_t prefix = 0, pmask = 0;
            unsigned long long above = 0;
            bool cut = true;
            for (int sh = 24; sh >= 0 && cut; sh -= 8) {
                for (int j2 = tid; j2 < 256; j2 += kSmpThreads) hmass[j2] = 0ull;
                __syncthreads();
                int krun = ktb;
                smp_pass(c0, c1, [&](int i) { return e[i]; }, [&](int, bool ok, float ev) {
                    const float pv = ev / sum_e;
                    const uint32_t bits = __builtin_bit_cast(uint32_t, pv);
                    const bool keep = kept_k(ok, bits, krun);
                    if (keep && (bits & pmask) == prefix)
                        atomicAdd(&hmass[(bits >> sh) & 0xFF], (unsigned long long)(pv * 1099511627776.0f));
                });
                __syncthreads();
                if (tid == 0) {
                    int bin = 255;
                    unsigned long long ab = above;
                    for (; bin >= 0; --bin) {
                        if (ab + hmass[bin] > tp) break;
                        ab += hmass[bin];
                    }
                    pinfo[0] = bin;  // -1: the kept mass never exceeds top_p
                    // mass above the crossing bin, carried in LDS as two words
                    wi[0][1] = (int)(uint32_t)(ab & 0xFFFFFFFFull);
                    wi[0][2] = (int)(uint32_t)(ab >> 32);
                }
                __syncthreads();
                const int bin = pinfo[0];
                if (bin < 0) {
                    cut = false;
                } else {
                    prefix |= (uint32_t)bin << sh;
                    pmask |= 0xFFu << sh;
                    above = (unsigned long long)(uint32_t)wi[0][1] | ((unsigned long long)(uint32_t)wi[0][2] << 32);
                }
                __syncthreads();
            }
            if (cut) {
                pcut = true;
                pb = prefix;
                const unsigned long long unit =
                    (unsigned long long)(__builtin_bit_cast(float, pb) * 1099511627776.0f);
                // smallest m >= 1 with above + m * unit > tp
                pneed = unit > 0 ? (int)min((tp - above) / unit + 1ull, (unsigned long long)V) : V;
            }
        }
        int ptb = 0;
        if (pcut) {
            int cnt = 0, krun = ktb;
            smp_pass(c0, c1, [&](int i) { return e[i]; }, [&](int, bool ok, float ev) {
                const uint32_t bits = __builtin_bit_cast(uint32_t, ev / sum_e);
                const bool keep = kept_k(ok, bits, krun);
                cnt += keep && bits == pb;
            });
            ptb = wave_base(cnt, wi[2]);
        }
        // the kept p of one step's entry (krun, prun: ties before the step)
        auto kept_p = [&](bool ok, float ev, int& krun, int& prun) {
            const float pv = ev / sum_e;
            const uint32_t bits = __builtin_bit_cast(uint32_t, pv);
            const bool keep = kept_k(ok, bits, krun);
            const bool tie = keep && pcut && bits == pb;
            const unsigned long long tm = __ballot(tie);
            const bool kp = keep && (!pcut || bits > pb || (tie && prun + popc_below(tm, l) < pneed));
            prun += __popcll(tm);
            return kp ? pv : 0.0f;
        };
        // --- the draw: running sums per wavefront (64-lane scans, iterations
        // in order), wavefronts in order
        float run = 0.0f;
        {
            int krun = ktb, prun = ptb;
            smp_pass(c0, c1, [&](int i) { return e[i]; }, [&](int, bool ok, float ev) {
                const float x = smp_wave_scan(kept_p(ok, ev, krun, prun));
                run = run + __shfl(x, 63, 64);
            });
        }
        if (l == 0) wf[w] = run;
        __syncthreads();
        if (tid == 0) {
            float acc = 0.0f;
            for (int j2 = 0; j2 < kSmpWaves; ++j2) {
                const float t = wf[j2];
                wf[j2] = acc;
                acc = acc + t;
            }
            wf[kSmpWaves] = acc;
            sel = -1;
        }
        __syncthreads();
        const float base = wf[w], next = w + 1 < kSmpWaves ? wf[w + 1] : wf[kSmpWaves];
        const float r = u * wf[kSmpWaves];
        if (r > 0.0f && base < r && next >= r) {  // this wavefront holds the crossing (exactly one does)
            float rr = 0.0f;
            int tok = -1, lastnz = -1, krun = ktb, prun = ptb;
            smp_pass(c0, c1, [&](int i) { return e[i]; }, [&](int i0, bool ok, float ev) {
                const float p = kept_p(ok, ev, krun, prun);  // every step: the tie counts advance
                if (tok >= 0) return;  // uniform: found in an earlier step
                const float x = smp_wave_scan(p);
                const float it = __shfl(x, 63, 64);
                const unsigned long long nz = __ballot(p > 0.0f);
                if (base + (rr + it) >= r) {
                    const unsigned long long hit = __ballot(base + (rr + x) >= r && p > 0.0f);
                    tok = hit ? i0 + __ffsll((long long)hit) - 1 : (nz ? i0 + 63 - __clzll((long long)nz) : lastnz);
                }
                if (nz) lastnz = i0 + 63 - __clzll((long long)nz);
                rr = rr + it;
            });
            if (l == 0) sel = tok >= 0 ? tok : (lastnz >= 0 ? lastnz : c0);
        }
        __syncthreads();
        if (tid == 0 && sel < 0) sel = r <= 0.0f ? 0 : V - 1;
        __syncthreads();
    }
    if (tid == 0) {
        if (a.out) a.out[b] = sel;
        if (a.best) a.best[b] = 0xFFFFFFFFull - (unsigned long long)(uint32_t)sel;
    }
}

}  // namespace

hipError_t sample_launch(const SampleArgs& a, int batch, hipStream_t st) {
    if (a.V < 1 || a.V >= (1 << 24) || batch < 1 || a.temperature <= 0.0f || a.top_k < 0 || !(a.top_p > 0.0f) ||
        a.top_p > 1.0f || (a.u_fixed < 0.0f && !a.u && !a.pos) || !a.scratch || !a.part)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_sample_max, dim3(kSmpBlocks, batch), dim3(kSmpPThreads), 0, st, a);
    if (a.top_k > 0 && a.top_k < a.V && a.top_k <= kSmpFastK)
        hipLaunchKernelGGL(k_sample_exp<true>, dim3(kSmpBlocks, batch), dim3(kSmpPThreads), 0, st, a);
    else
        hipLaunchKernelGGL(k_sample_exp<false>, dim3(kSmpBlocks, batch), dim3(kSmpPThreads), 0, st, a);
    if (a.top_k > kSmpFastK && a.top_k < a.V && a.top_k <= kSmpMaxK)
        hipLaunchKernelGGL(k_sample_gather, dim3(kSmpBlocks, batch), dim3(kSmpPThreads), 0, st, a);
    hipLaunchKernelGGL(k_sample, dim3(batch), dim3(kSmpThreads), 0, st, a);
    return hipGetLastError();
}

}  // namespace nx
