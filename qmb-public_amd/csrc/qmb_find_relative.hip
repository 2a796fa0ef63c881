// qmb_find_relative.hip -- find_relative as a deterministic radix select on gfx950.
//
// The reference keeps a K-slot min-heap of (weight, config) entries, one entry per contribution
// |sign * coef * psi_i|^2 whose target is not excluded (qmb/_hamiltonian_cpu.cpp:341-405), guarded
// on the GPU by per-node spin locks with racy pre-reads (qmb/_hamiltonian_cuda.cu:276-427); then it
// drops zero weights and returns the distinct configs sorted by bytes (:537-545).
//
// Here the K largest contributions are found without locks, and without looking at most of them.  A
// contribution's weight is at most (|coef| |psi|)^2, so the rows are first put in descending |psi| and
// the terms of every bucket in descending |coef|: the contributions that can reach a weight are then a
// prefix of every bucket's terms for a prefix of the rows, and nothing else is enumerated.  (At 52 spin
// orbitals and 1M rows, K = 100,000, enumerating and weighing all 2.9e10 connections took 64 ms of a
// 73.9 ms call; the whole call takes 4.6 ms this way, 1.9 of them in the digit passes and 1.7 in the
// collecting pass.  At 20 spin orbitals and 10,000 rows, K = 1000: 1.76 -> 0.62 ms.)
//
// Positive doubles order like their bit patterns, so the K-th largest weight is located digit by digit
// (12-bit digits of the weight bits): every pass histograms the next digit of the entries tied with the
// threshold so far, and a one-block kernel picks the digit at which the running count reaches K.  The
// first digit's pass needs a lower bound to be a prefix: it starts from the power of four whose
// products |coef| |psi| (counted from exponent histograms of the two) number some 64 K, and is repeated
// at 16 times as many while it finds fewer than K entries (most connections do not exist or are
// excluded).  Once the tied class fits the candidate buffer, one more pass collects every entry strictly
// above the threshold prefix and the tied candidates; the candidates are ordered by (weight desc,
// config asc) and the first K - above are kept.  A class that does not fit although its weight is settled
// to the last bit (one hopping magnitude and a uniform |psi|, say) is narrowed in the same way by the
// digits of the config, ascending.  All control lives in device memory, so the whole call is enqueued
// without host synchronisation; passes that are not needed return at once.
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include <utility>

#include "qmb_enum.hpp"

namespace qmb {

namespace {

constexpr int kHistBits = 12;
constexpr int kHistBins = 1 << kHistBits;
constexpr int kLevels = 6;  // digits [51,63) [39,51) [27,39) [15,27) [3,15) [0,3)

__host__ __device__ inline int fr_shift(int level) { return level < 5 ? 51 - 12 * level : 0; }
__host__ __device__ inline int fr_width(int level) { return level < 5 ? 12 : 3; }

inline unsigned blocks_for(int64_t n, int block = 256) {
    int64_t b = (n + block - 1) / block;
    return static_cast<unsigned>(b < 1 ? 1 : b);
}

constexpr int kTries = 6;  // lower bounds of the first digit's pass; the last is the least weight

struct FrState {
    int64_t k_rem;
    uint64_t prefix;
    int32_t level;
    int32_t tries;  // bounds tried at level 0
    int32_t done;
    int32_t reserved;
    unsigned long long n_above;
    unsigned long long n_cand;
    int64_t cand_needed;
    uint64_t lo;     // entries with w < lo are not wanted; collect: candidates are lo <= w < hi,
    uint64_t hi;     // entries with w >= hi are selected outright
    double reach;    // |coef| |psi| of an entry with w >= lo is not below this
    int64_t active;  // rows that can reach it: a prefix
    uint64_t bound[kTries];
    // Entries of one weight narrowed by config: those with `key & tie_mask` below tie_key are selected
    // outright, equal to it candidates, above it not wanted (all of them candidates while the mask is 0).
    uint64_t tie_key[kMaxWords];
    uint64_t tie_mask[kMaxWords];
    int32_t ties;  // more entries than the candidate buffer holds are tied on weight and tie_key
    uint32_t tie_blocks;
    unsigned long long least, most;  // weights counted by the pass: equal, the digits below need no passes
};

// Reach of the weight with these bits: no product |coef| |psi| below it gives that weight.  The computed
// weight is within a few roundings of (|coef| |psi|)^2, except at the ends of the range: a product whose
// square overflows (or is NaN) is at least about the root of the largest finite weight, and each square
// of a denormal weight may be rounded up to it.
__device__ __forceinline__ double reach_of(uint64_t lo) {
    constexpr uint64_t kLargest = 0x7fefffffffffffffull;
    const double root = sqrt(__longlong_as_double(static_cast<long long>(lo < kLargest ? lo : kLargest)));
    return root * (lo < (64ull << 52) ? 0.5 : 1.0 - 1e-9);
}

// Rows and terms are ordered by the high word of the bits of |psi| and |coef| (20 bits of mantissa), so
// a later one is at most a factor 1 + 2^-20 above an earlier one or, both denormal, 2^-1042 more: what
// any from there on can have.  NaN orders first and drops nothing.
__device__ __forceinline__ double at_most_from(double a) { return a * (1.0 + 2e-6) + 0x1p-1042; }

__device__ __forceinline__ bool below_reach(double a, double b, double reach) { return a * b < reach; }

struct FrParams {
    EnumSource src;
    const double2* psi;
    const double2* coefs;
    const uint64_t* xkeys;
    const uint64_t* xtable;
    uint64_t xmask;
    const uint64_t* xfilter;
    uint64_t xfmask;
    const uint64_t* xcols;
    const double* aw;  // per term, |coef| at most from there on in its bucket (at_most_from)
    FrState* state;
    unsigned long long* hist;
    uint64_t* sel_c;   // [K][W] selected configs ("above" entries, then the kept candidates)
    uint64_t* cand_w;  // [cap]
    uint64_t* cand_c;  // [cap][W]
    int64_t k;
    int64_t cand_cap;
    int tile_log2;
    int groups;
    int direct;
};

// |sign * coef * psi|^2 with every product and sum rounded separately, so the bits match a plain IEEE
// evaluation of the reference expression (qmb/_hamiltonian_cpu.cpp:388-392) and are the same in every
// kernel: the passes compare the weights that others counted for equality.  (__dmul_rn and __dadd_rn are
// ordinary operators here, which the compiler fuses, each kernel in its own way, unless told not to.)
__device__ __forceinline__ uint64_t weight_bits(const double2 cf, const double2 v) {
#pragma clang fp contract(off)
    const double re = cf.x * v.x - cf.y * v.y;
    const double im = cf.x * v.y + cf.y * v.x;
    const double w = re * re + im * im;
    return static_cast<uint64_t>(__double_as_longlong(w));
}

// Digits of a config's key, the config as one big-endian number (word w of it: bytes 8 w to 8 w + 7), so
// that keys order as configs do.  Digit d is bits [12 d, 12 d + 12) from the top; one may straddle words.
__host__ __device__ inline int tie_levels(int n_qubytes) { return (8 * n_qubytes + kHistBits - 1) / kHistBits; }

// Adds digit `value` of position d to key.
template <int W>
__device__ __forceinline__ void put_digit(uint64_t (&key)[W], int d, uint64_t value) {
    const int first = kHistBits * d >> 6, r = kHistBits * d & 63;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        if (w == first) {
            key[w] |= (value << (64 - kHistBits)) >> r;
        }
        if (w == first + 1 && r > 64 - kHistBits) {
            key[w] |= value << (128 - kHistBits - r);
        }
    }
}

template <int W>
__device__ __forceinline__ uint32_t get_digit(const uint64_t (&key)[W], int d) {
    const int first = kHistBits * d >> 6, r = kHistBits * d & 63;
    uint64_t v = 0ull;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        if (w == first) {
            v |= (key[w] << r) >> (64 - kHistBits);
        }
        if (w == first + 1 && r > 64 - kHistBits) {
            v |= key[w] >> (128 - kHistBits - r);
        }
    }
    return static_cast<uint32_t>(v);
}

template <int W>
struct TieRange {
    uint64_t key[W], mask[W];
    __device__ __forceinline__ explicit TieRange(const FrState* st) {
#pragma unroll
        for (int w = 0; w < W; ++w) {
            key[w] = st->tie_key[w];
            mask[w] = st->tie_mask[w];
        }
    }
    // -1, 0, 1: the config's settled digits below, equal to or above the tied ones.
    __device__ __forceinline__ int side(const Cfg<W>& c) const {
        int s = 0;
#pragma unroll
        for (int w = W - 1; w >= 0; --w) {
            const uint64_t k = bswap64(c.w[w]) & mask[w];
            s = k < key[w] ? -1 : (k > key[w] ? 1 : s);
        }
        return s;
    }
};

// The pruning both passes share: terms whose |coef| with the tile's largest |psi| stays below the reach.
struct PrunedHooks : ActionHooks {
    static constexpr bool kPruned = true;
    const FrParams& p;
    double reach;
    __device__ explicit PrunedHooks(const FrParams& pp) : p(pp), reach(pp.state->reach) {}
    __device__ __forceinline__ double tile_bound(int64_t i0) const { return at_most_from(hypot(p.psi[i0].x, p.psi[i0].y)); }
    __device__ __forceinline__ bool drop(uint32_t t, double bound) const { return below_reach(p.aw[t], bound, reach); }
};

template <int W>
struct HistAction : PrunedHooks {
    uint32_t* hist;
    uint64_t prefix;
    uint64_t lo;
    int shift;
    int width;
    uint64_t least = ~0ull, most = 0ull;  // of the weights this thread counts
    __device__ HistAction(const FrParams& pp, uint32_t* h, uint64_t pre_, int sh, int wd)
        : PrunedHooks(pp), hist(h), prefix(pre_), lo(pp.state->lo), shift(sh), width(wd) {}
    // Only entries still tied with the threshold prefix need the (costly) exclusion lookup.
    __device__ __forceinline__ bool pre(int64_t i, uint32_t t, const Cfg<W>&, int, uint64_t, uint64_t) {
        const uint64_t w = weight_bits(p.coefs[t], p.psi[i]);
        return w >= lo && (w >> (shift + width)) == prefix;
    }
    __device__ __forceinline__ void post(int64_t i, uint32_t t, const Cfg<W>&, int, int64_t j, bool) {
        if (j >= 0) {
            return;  // excluded
        }
        const uint64_t w = weight_bits(p.coefs[t], p.psi[i]);
        least = w < least ? w : least;
        most = w > most ? w : most;
        atomicAdd(&hist[(w >> shift) & ((1u << width) - 1u)], 1u);
    }
};

// The next config digit of the entries with the settled weight and the settled config digits.
template <int W>
struct TieAction : PrunedHooks {
    uint32_t* hist;
    uint64_t weight;
    TieRange<W> range;
    int digit;
    __device__ TieAction(const FrParams& pp, uint32_t* h, int d)
        : PrunedHooks(pp), hist(h), weight(pp.state->prefix), range(pp.state), digit(d) {}
    __device__ __forceinline__ bool pre(int64_t i, uint32_t t, const Cfg<W>& o, int, uint64_t, uint64_t) {
        return weight_bits(p.coefs[t], p.psi[i]) == weight && range.side(o) == 0;
    }
    __device__ __forceinline__ void post(int64_t, uint32_t, const Cfg<W>& o, int, int64_t j, bool) {
        if (j >= 0) {
            return;  // excluded
        }
        uint64_t key[W];
#pragma unroll
        for (int w = 0; w < W; ++w) {
            key[w] = bswap64(o.w[w]);
        }
        atomicAdd(&hist[get_digit<W>(key, digit)], 1u);
    }
};

template <int W>
struct CollectAction : PrunedHooks {
    uint64_t lo;
    uint64_t hi;
    TieRange<W> range;
    __device__ explicit CollectAction(const FrParams& pp) : PrunedHooks(pp), lo(pp.state->lo), hi(pp.state->hi), range(pp.state) {}
    __device__ __forceinline__ bool pre(int64_t i, uint32_t t, const Cfg<W>& o, int, uint64_t, uint64_t) {
        const uint64_t w = weight_bits(p.coefs[t], p.psi[i]);
        return w >= lo && (w >= hi || range.side(o) <= 0);
    }
    __device__ __forceinline__ void post(int64_t i, uint32_t t, const Cfg<W>& o, int, int64_t j, bool) {
        if (j >= 0) {
            return;  // excluded
        }
        const uint64_t w = weight_bits(p.coefs[t], p.psi[i]);
        if (w >= hi || range.side(o) < 0) {
            const unsigned long long s = atomicAdd(&p.state->n_above, 1ull);
            if (s < static_cast<unsigned long long>(p.k)) {
#pragma unroll
                for (int w2 = 0; w2 < W; ++w2) {
                    p.sel_c[s * W + w2] = o.w[w2];
                }
            }
        } else {
            const unsigned long long s = atomicAdd(&p.state->n_cand, 1ull);
            if (s < static_cast<unsigned long long>(p.cand_cap)) {
                p.cand_w[s] = w;
#pragma unroll
                for (int w2 = 0; w2 < W; ++w2) {
                    p.cand_c[s * W + w2] = o.w[w2];
                }
            }
        }
    }
};

// The connections of the rows that can reach the bound, the (tile, bucket group) units dealt over the
// grid's work-groups.
template <int W, typename Action>
__device__ __forceinline__ void fr_enumerate(const FrParams& p, uint64_t* smem, Action& act) {
    const HashIndex ix{p.xtable, p.xkeys, p.xmask, p.xfilter, p.xfmask, p.xcols, false};
    EnumSource src = p.src;
    src.n_i = p.state->active;
    if (p.direct) {
        const int64_t blocks = (src.n_i + kEnumBlock - 1) / kEnumBlock;
        for (int64_t b = blockIdx.x; b < blocks; b += gridDim.x) {
            enumerate_direct<W>(src, ix, b, *reinterpret_cast<DirectLds<W>*>(smem), act);
        }
    } else {
        const int64_t units = ((src.n_i + (1ll << p.tile_log2) - 1) >> p.tile_log2) * p.groups;
        for (int64_t u = blockIdx.x; u < units; u += gridDim.x) {
            enumerate_tile<W>(src, ix, u / p.groups, p.tile_log2, static_cast<int>(u % p.groups), p.groups, smem, act);
            __syncthreads();  // the next unit reuses the tile's LDS
        }
    }
}

template <int W>
__global__ __launch_bounds__(kEnumBlock) void fr_hist_kernel(FrParams p) {
    extern __shared__ uint64_t smem[];
    __shared__ uint32_t s_hist[kHistBins];
    __shared__ unsigned long long s_least, s_most;
    if (p.state->done) {
        return;  // uniform: every thread reads the same flag
    }
    if (threadIdx.x == 0) {
        s_least = ~0ull;
        s_most = 0ull;
    }
    const int level = p.state->level;
    const int shift = fr_shift(level);
    const int width = fr_width(level);
    const uint64_t prefix = p.state->prefix;
    for (int b = threadIdx.x; b < kHistBins; b += kEnumBlock) {
        s_hist[b] = 0;
    }
    __syncthreads();
    HistAction<W> act(p, s_hist, prefix, shift, width);
    fr_enumerate<W>(p, smem, act);
    unsigned long long least = act.least, most = act.most;
    if (__ballot(least != ~0ull) != 0ull) {
        for (int d = 32; d > 0; d >>= 1) {
            const unsigned long long a = __shfl_xor(least, d), b = __shfl_xor(most, d);
            least = a < least ? a : least;
            most = b > most ? b : most;
        }
        if ((threadIdx.x & 63) == 0) {
            atomicMin(&s_least, least);
            atomicMax(&s_most, most);
        }
    }
    __syncthreads();
    // most blocks' weights lie within what others have reported: a look before the atomics
    if (threadIdx.x == 0 && s_least != ~0ull) {
        if (s_least < *const_cast<const volatile unsigned long long*>(&p.state->least)) {
            atomicMin(&p.state->least, s_least);
        }
        if (s_most > *const_cast<const volatile unsigned long long*>(&p.state->most)) {
            atomicMax(&p.state->most, s_most);
        }
    }
    for (int b = threadIdx.x; b < (1 << width); b += kEnumBlock) {
        if (s_hist[b]) {
            atomicAdd(&p.hist[b], static_cast<unsigned long long>(s_hist[b]));
        }
    }
}

template <int W>
__global__ __launch_bounds__(kEnumBlock) void fr_collect_kernel(FrParams p) {
    extern __shared__ uint64_t smem[];
    CollectAction<W> act(p);
    fr_enumerate<W>(p, smem, act);
}

// Entries of one weight that exceed the candidate buffer, digit d of their configs: every block counts, the
// last one to finish picks the digit at which the running count from the lowest reaches what is needed
// (a fence per block, but only where there are such ties; a kernel of its own for the choice would cost
// every other call a launch a digit: the two to five launches without ties are 3 us of 620).  30,000 rows
// of a 32-site Hubbard chain with |psi| = 1 and K = 7500 take 0.70 ms.
template <int W>
__global__ __launch_bounds__(kEnumBlock) void fr_tie_kernel(FrParams p, int d, int levels) {
    extern __shared__ uint64_t smem[];
    __shared__ uint32_t s_hist[kHistBins];
    __shared__ unsigned long long s_wave[kEnumBlock / 64];
    __shared__ bool s_last;
    FrState* st = p.state;
    if (st->ties == 0) {
        return;  // uniform: every thread reads the same flag, which only the last block to finish changes
    }
    for (int b = threadIdx.x; b < kHistBins; b += kEnumBlock) {
        s_hist[b] = 0;
    }
    __syncthreads();
    TieAction<W> act(p, s_hist, d);
    fr_enumerate<W>(p, smem, act);
    __syncthreads();
    for (int b = threadIdx.x; b < kHistBins; b += kEnumBlock) {
        if (s_hist[b]) {
            atomicAdd(&p.hist[b], static_cast<unsigned long long>(s_hist[b]));
        }
    }
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) {
        s_last = atomicAdd(&st->tie_blocks, 1u) == gridDim.x - 1u;
    }
    __syncthreads();
    if (!s_last) {
        return;
    }
    __threadfence();
    constexpr int kPer = kHistBins / kEnumBlock;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long v[kPer], sum = 0ull;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        unsigned long long* bin = &p.hist[kPer * static_cast<int>(threadIdx.x) + q];
        v[q] = __hip_atomic_load(bin, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *bin = 0ull;
        sum += v[q];
    }
    unsigned long long incl = sum;
    for (int k = 1; k < 64; k <<= 1) {
        const unsigned long long o = __shfl_up(incl, k);
        incl += lane >= k ? o : 0ull;
    }
    if (lane == 63) {
        s_wave[wave] = incl;
    }
    __syncthreads();
    unsigned long long cum = incl - sum;
    for (int w = 0; w < wave; ++w) {
        cum += s_wave[w];
    }
    const unsigned long long need = static_cast<unsigned long long>(st->cand_needed);
    __syncthreads();  // every thread has it before one changes it
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        if (cum < need && cum + v[q] >= need) {  // one thread
            uint64_t key[W], mask[W];
#pragma unroll
            for (int w = 0; w < W; ++w) {
                key[w] = st->tie_key[w];
                mask[w] = st->tie_mask[w];
            }
            put_digit<W>(key, d, static_cast<uint64_t>(kPer * static_cast<int>(threadIdx.x) + q));
            put_digit<W>(mask, d, kHistBins - 1);
#pragma unroll
            for (int w = 0; w < W; ++w) {
                st->tie_key[w] = key[w];
                st->tie_mask[w] = mask[w];
            }
            st->cand_needed = static_cast<int64_t>(need - cum);
            // past the last digit the entries left are one config's: any of them will do
            st->ties = v[q] > static_cast<unsigned long long>(p.cand_cap) && d + 1 < levels ? 1 : 0;
            st->tie_blocks = 0u;
        }
        cum += v[q];
    }
}

// Sort keys of the rows: the high word of |psi|'s bits.
__global__ void fr_row_keys_kernel(const double2* __restrict__ psi, int64_t n, uint32_t* __restrict__ keys, uint32_t* __restrict__ idx) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i < n) {
        keys[i] = static_cast<uint32_t>(static_cast<uint64_t>(__double_as_longlong(hypot(psi[i].x, psi[i].y))) >> 32);
        idx[i] = static_cast<uint32_t>(i);
    }
}

__global__ void fr_row_gather_kernel(const uint32_t* __restrict__ order, const uint8_t* __restrict__ configs, const double2* __restrict__ psi,
                                     int64_t n, int nq, uint8_t* __restrict__ out_configs, double2* __restrict__ out_psi) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i < n) {
        const int64_t r = order[i];
        for (int b = 0; b < nq; ++b) {
            out_configs[i * nq + b] = configs[r * nq + b];
        }
        out_psi[i] = psi[r];
    }
}

// Sort keys of the terms (in bucket order): bucket, then descending |coef|.  Terms that never succeed
// stay behind the last bucket.
__global__ void fr_term_keys_kernel(const double2* __restrict__ coefs, const uint32_t* __restrict__ bucket_start, int64_t n_buckets,
                                    int64_t n_terms, uint64_t* __restrict__ keys, uint32_t* __restrict__ idx) {
    const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t < n_terms) {
        int64_t lo = 0, hi = n_buckets;  // last bucket starting at or before t
        while (lo < hi) {
            const int64_t mid = (lo + hi + 1) >> 1;
            if (bucket_start[mid] <= t) {
                lo = mid;
            } else {
                hi = mid - 1;
            }
        }
        const uint64_t bits = static_cast<uint64_t>(__double_as_longlong(hypot(coefs[t].x, coefs[t].y)));
        keys[t] = (static_cast<uint64_t>(lo) << 32) | static_cast<uint32_t>(~(bits >> 32));
        idx[t] = static_cast<uint32_t>(t);
    }
}

__global__ void fr_term_gather_kernel(const uint32_t* __restrict__ order, const uint64_t* __restrict__ recs, const double2* __restrict__ coefs,
                                      int64_t n_terms, uint64_t* __restrict__ out_recs, double2* __restrict__ out_coefs,
                                      double* __restrict__ aw) {
    const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (t < n_terms) {
        const uint32_t o = order[t];
        const double2 c = coefs[o];
        out_recs[t] = recs[o];
        out_coefs[t] = c;
        aw[t] = at_most_from(hypot(c.x, c.y));
    }
}

// The exponent histogram of |v| and the largest |v| (as its bits: NaN above everything).
struct FrExponents {
    uint32_t count[2048];
    unsigned long long most;
};

// Of the rows (exps[0], the first row_blocks blocks) and of the terms (exps[1], the others).
__global__ __launch_bounds__(256) void fr_exponents_kernel(const double2* __restrict__ psi, int64_t n_rows, unsigned row_blocks,
                                                           const double2* __restrict__ coefs, int64_t n_terms, FrExponents* __restrict__ exps) {
    __shared__ uint32_t s_exp[2048];
    unsigned long long most = 0ull;
    const bool rows = blockIdx.x < row_blocks;
    const double2* v = rows ? psi : coefs;
    const int64_t n = rows ? n_rows : n_terms;
    const int64_t block = rows ? blockIdx.x : blockIdx.x - row_blocks, blocks = rows ? row_blocks : gridDim.x - row_blocks;
    exps += rows ? 0 : 1;
    for (int b = threadIdx.x; b < 2048; b += 256) {
        s_exp[b] = 0u;
    }
    __syncthreads();
    for (int64_t i = block * 256 + threadIdx.x; i < n; i += blocks * 256) {
        const unsigned long long a = static_cast<unsigned long long>(__double_as_longlong(hypot(v[i].x, v[i].y)));
        atomicAdd(&s_exp[(a >> 52) & 0x7ffu], 1u);
        most = a > most ? a : most;
    }
    for (int d = 32; d > 0; d >>= 1) {
        const unsigned long long o = __shfl_xor(most, d);
        most = o > most ? o : most;
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMax(&exps->most, most);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < 2048; b += 256) {
        if (s_exp[b] != 0u) {
            atomicAdd(&exps->count[b], s_exp[b]);
        }
    }
}

// exps: of the rows, then of the terms.
__global__ void fr_init_kernel(FrState* st, unsigned long long* hist, FrExponents* exps, int64_t k) {
    for (int b = threadIdx.x; b < kHistBins; b += blockDim.x) {
        hist[b] = 0;
        exps[b >> 11].count[b & 2047] = 0;
    }
    if (threadIdx.x == 0) {
        exps[0].most = 0;
        exps[1].most = 0;
        *st = FrState{};
        st->k_rem = k;
        st->lo = 1;
        st->hi = 1;
        st->least = ~0ull;
    }
}

// Rows (in descending |psi|) that can reach `reach` with the largest |coef|.
__device__ int64_t fr_active(const double2* __restrict__ psi, int64_t n, double amax, double reach) {
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (below_reach(amax, at_most_from(hypot(psi[mid].x, psi[mid].y)), reach)) {
            hi = mid;
        } else {
            lo = mid + 1;
        }
    }
    return lo;
}

__device__ void fr_set_lo(FrState* st, uint64_t lo, const double2* __restrict__ psi, int64_t n, double amax) {
    st->lo = lo < 1ull ? 1ull : lo;
    st->reach = reach_of(st->lo);
    st->active = fr_active(psi, n, amax, st->reach);
}

__device__ __forceinline__ double fr_amax(const FrExponents* exps) {
    return at_most_from(__longlong_as_double(static_cast<long long>(exps[1].most)));
}

// The bounds of the first digit's pass: the products |psi| |coef| whose exponents sum to e or more number
// N(e), from the histograms (zeros and denormals count as the least, non-finite values as the largest
// exponent); bound q is the weight of a product 2^e for the largest e with N(e) >= 64 K 16^q, the last one
// the least weight.  One block.
__global__ __launch_bounds__(1024) void fr_plan_kernel(FrState* st, const double2* __restrict__ psi, int64_t n,
                                                       const FrExponents* __restrict__ exps, int64_t k) {
    __shared__ unsigned long long s_pairs[4096];  // by exponent sum
    __shared__ uint32_t s_rows[2048];
    __shared__ uint32_t s_list[2048];  // exponents that some coefficient has
    __shared__ unsigned long long s_wave[16];
    __shared__ int s_count, s_e[kTries];
    for (int e = threadIdx.x; e < 4096; e += 1024) {
        s_pairs[e] = 0ull;
    }
    if (threadIdx.x == 0) {
        s_count = 0;
    }
    if (threadIdx.x < kTries) {
        s_e[threadIdx.x] = -1;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 2048; e += 1024) {
        s_rows[e] = exps[0].count[e];
        if (exps[1].count[e] != 0u) {
            s_list[atomicAdd(&s_count, 1)] = static_cast<uint32_t>(e);
        }
    }
    __syncthreads();
    for (int l = 0; l < s_count; ++l) {
        const uint32_t a = s_list[l];
        const unsigned long long na = exps[1].count[a];
        for (int b = threadIdx.x; b < 2048; b += 1024) {
            if (s_rows[b] != 0u) {
                atomicAdd(&s_pairs[a + b], na * s_rows[b]);
            }
        }
    }
    __syncthreads();
    // N(e) from the top, four sums a thread
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long v[4], sum = 0ull;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        v[q] = s_pairs[4095 - 4 * static_cast<int>(threadIdx.x) - q];
        sum += v[q];
    }
    unsigned long long incl = sum;
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long o = __shfl_up(incl, d);
        incl += lane >= d ? o : 0ull;
    }
    if (lane == 63) {
        s_wave[wave] = incl;
    }
    __syncthreads();
    unsigned long long cum = incl - sum;
    for (int w = 0; w < wave; ++w) {
        cum += s_wave[w];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        unsigned long long want = 64ull * static_cast<unsigned long long>(k);
        for (int t = 0; t < kTries - 1; ++t, want *= 16ull) {
            if (cum < want && cum + v[q] >= want) {
                s_e[t] = 4095 - 4 * static_cast<int>(threadIdx.x) - q;
            }
        }
        cum += v[q];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int q = 0, last = -1;
        for (int t = 0; t < kTries - 1; ++t) {
            if (s_e[t] >= 0 && s_e[t] != last) {
                // biased exponents summing to e: products from 2^(e - 2046), weights from 2^(2 e - 4092)
                last = s_e[t];
                const int biased = 2 * last - 4092 + 1023;
                st->bound[q++] = biased >= 2046 ? 2046ull << 52 : (biased > 0 ? static_cast<uint64_t>(biased) << 52 : 1ull);
            }
        }
        for (; q < kTries; ++q) {
            st->bound[q] = 1ull;
        }
        fr_set_lo(st, st->bound[0], psi, n, fr_amax(exps));
    }
}

// Chooses the threshold digit of the current level (one block; 4096 bins, four a thread, from the top).
__global__ __launch_bounds__(1024) void fr_select_kernel(FrState* st, unsigned long long* hist, const double2* __restrict__ psi, int64_t n,
                                                         const FrExponents* __restrict__ exps, int64_t cand_cap) {
    __shared__ unsigned long long s_wave[16];
    __shared__ unsigned long long s_cum, s_in;
    __shared__ int s_digit;
    if (st->done) {
        return;  // uniform: every thread reads the same flag
    }
    const int level = st->level;
    const int width = fr_width(level);
    const int bins = 1 << width;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long v[4], sum = 0ull;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int b = bins - 1 - (4 * static_cast<int>(threadIdx.x) + q);
        v[q] = b >= 0 ? hist[b] : 0ull;
        sum += v[q];
        if (b >= 0) {
            hist[b] = 0ull;
        }
    }
    unsigned long long incl = sum;
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long o = __shfl_up(incl, d);
        incl += lane >= d ? o : 0ull;
    }
    if (lane == 63) {
        s_wave[wave] = incl;
    }
    if (threadIdx.x == 0) {
        s_digit = -1;
    }
    __syncthreads();
    unsigned long long total = 0ull, cum = incl - sum;
    for (int w = 0; w < 16; ++w) {
        total += s_wave[w];
        cum += w < wave ? s_wave[w] : 0ull;
    }
    const unsigned long long need = static_cast<unsigned long long>(st->k_rem);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (cum < need && cum + v[q] >= need) {
            s_digit = bins - 1 - (4 * static_cast<int>(threadIdx.x) + q);
            s_cum = cum;
            s_in = v[q];
        }
        cum += v[q];
    }
    __syncthreads();
    if (threadIdx.x != 0) {
        return;
    }
    const double amax = fr_amax(exps);
    const uint64_t least = st->least, most = st->most;
    st->least = ~0ull;
    st->most = 0ull;
    if (level == 0 && total <= need && st->lo > 1ull) {
        // fewer than K above the bound: the next one (K of them exactly: the same selection, found again)
        fr_set_lo(st, st->bound[++st->tries], psi, n, amax);
    } else if (level == 0 && total <= need) {
        st->done = 1;  // every nonzero entry is selected outright
        st->cand_needed = 0;
        st->hi = 1;
    } else if (least == most) {
        // all that were counted weigh the same, so the weight is settled (a uniform |psi| and one coefficient
        // size: four passes less, 20,000 rows of a 50-site Hubbard chain, K = 5000, 1.53 -> 1.01 ms)
        st->prefix = least;
        fr_set_lo(st, least, psi, n, amax);
        st->done = 1;
        st->cand_needed = static_cast<int64_t>(need);
        st->hi = least + 1ull;
        st->ties = total > static_cast<unsigned long long>(cand_cap) ? 1 : 0;
    } else {
        const uint64_t d = static_cast<uint64_t>(s_digit);
        st->k_rem = static_cast<int64_t>(need - s_cum);
        st->prefix = (st->prefix << width) | d;
        const int shift = fr_shift(level);
        const uint64_t tied = st->prefix << shift;  // the tied class and everything above it
        fr_set_lo(st, level == 0 && tied < st->lo ? st->lo : tied, psi, n, amax);
        if (s_in <= static_cast<unsigned long long>(cand_cap) || level == kLevels - 1) {
            st->done = 1;
            st->cand_needed = st->k_rem;
            st->hi = (st->prefix + 1ull) << shift;
            st->ties = s_in > static_cast<unsigned long long>(cand_cap) ? 1 : 0;
        } else {
            st->level = level + 1;
        }
    }
}

template <int W>
__global__ void be_word_gather_kernel(const uint64_t* __restrict__ words, const uint32_t* __restrict__ perm, int64_t n, int w,
                                      uint64_t* __restrict__ out) {
    const int64_t p = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (p < n) {
        out[p] = bswap64(words[static_cast<int64_t>(perm[p]) * W + w]);
    }
}

__global__ void u64_gather_kernel(const uint64_t* __restrict__ v, const uint32_t* __restrict__ perm, int64_t n,
                                  uint64_t* __restrict__ out) {
    const int64_t p = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (p < n) {
        out[p] = v[perm[p]];
    }
}

__global__ void valid_key_kernel(const uint32_t* __restrict__ perm, int64_t n, const FrState* __restrict__ st, int64_t k,
                                 uint64_t* __restrict__ out) {
    const int64_t p = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (p < n) {
        const unsigned long long above = st->n_above < static_cast<unsigned long long>(k) ? st->n_above : k;
        const int64_t n_sel = static_cast<int64_t>(above) + st->cand_needed;
        out[p] = static_cast<int64_t>(perm[p]) < n_sel ? 0ull : 1ull;
    }
}

__global__ void iota_u32_kernel(uint32_t* p, int64_t n) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i < n) {
        p[i] = static_cast<uint32_t>(i);
    }
}

// Appends the first cand_needed candidates (in sorted order) after the "above" entries.
template <int W>
__global__ void fr_take_kernel(const uint32_t* __restrict__ perm, int64_t cap, const uint64_t* __restrict__ cand_c,
                               const FrState* __restrict__ st, int64_t k, uint64_t* __restrict__ sel_c) {
    const int64_t p = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    const unsigned long long above = st->n_above < static_cast<unsigned long long>(k) ? st->n_above : k;
    const int64_t found = static_cast<int64_t>(st->n_cand < static_cast<unsigned long long>(cap) ? st->n_cand : cap);
    const int64_t need = st->cand_needed < found ? st->cand_needed : found;
    if (p < cap && p < need && static_cast<int64_t>(above) + p < k) {
#pragma unroll
        for (int w = 0; w < W; ++w) {
            sel_c[(above + p) * W + w] = cand_c[static_cast<int64_t>(perm[p]) * W + w];
        }
    }
}

template <int W>
__global__ void fr_unique_flag_kernel(const uint32_t* __restrict__ perm, int64_t n, const uint64_t* __restrict__ sel_c,
                                      const FrState* __restrict__ st, int64_t k, uint32_t* __restrict__ flag) {
    const int64_t p = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (p >= n) {
        return;
    }
    const unsigned long long above = st->n_above < static_cast<unsigned long long>(k) ? st->n_above : k;
    const int64_t found = static_cast<int64_t>(st->n_cand);
    const int64_t need = st->cand_needed < found ? st->cand_needed : found;
    int64_t n_sel = static_cast<int64_t>(above) + need;
    if (n_sel > k) {
        n_sel = k;
    }
    const int64_t a = perm[p];
    uint32_t f = a < n_sel ? 1u : 0u;
    if (f && p > 0) {
        const int64_t b = perm[p - 1];
        bool eq = true;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            eq = eq && (sel_c[a * W + w] == sel_c[b * W + w]);
        }
        if (eq) {
            f = 0u;
        }
    }
    flag[p] = f;
}

template <int W>
__global__ void fr_scatter_kernel(const uint32_t* __restrict__ perm, int64_t n, const uint64_t* __restrict__ sel_c,
                                  const uint32_t* __restrict__ flag, const uint32_t* __restrict__ pos, int nq,
                                  uint8_t* __restrict__ out, int64_t* __restrict__ out_rows) {
    const int64_t p = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (p >= n) {
        return;
    }
    if (flag[p]) {
        Cfg<W> c;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            c.w[w] = sel_c[static_cast<int64_t>(perm[p]) * W + w];
        }
        store_row<W>(out + static_cast<int64_t>(pos[p]) * nq, nq, c);
    }
    if (p == n - 1) {
        *out_rows = static_cast<int64_t>(pos[p]) + flag[p];
    }
}

constexpr unsigned kTieGrid = 1024;  // four work-groups a CU: a launch that finds no ties costs 2 us

// Entries tied on the digits so far are collected as candidates up to this many, and narrowed by another
// digit's pass above it (of the weight, then of the config): the candidates are sorted twice in full (1M of them: 1.7 ms), a pass over what
// is left of the connections costs less.
int64_t cand_capacity(int64_t k) {
    const int64_t cap = 2 * k;
    return cap < (1 << 16) ? (1 << 16) : cap;
}

struct FrScratch {
    uint8_t* configs;  // rows in descending |psi|
    double2* psi;
    uint32_t* row_key_a;
    uint32_t* row_key_b;
    uint32_t* row_a;
    uint32_t* row_b;
    uint64_t* recs;  // terms in descending |coef| within each bucket
    double2* coefs;
    double* aw;
    uint64_t* term_key_a;
    uint64_t* term_key_b;
    uint32_t* term_a;
    uint32_t* term_b;
    FrExponents* exps;
    FrState* state;
    unsigned long long* hist;
    uint64_t* sel_c;
    uint64_t* cand_w;
    uint64_t* cand_c;
    uint32_t* perm_a;
    uint32_t* perm_b;
    uint64_t* key_a;
    uint64_t* key_b;
    uint32_t* flag;
    uint32_t* pos;
    void* tmp;
    size_t tmp_bytes;
};

FrScratch fr_layout(Carver& cv, int W, int n_qubytes, int64_t n_i, int64_t k, int64_t n_terms) {
    const int64_t cap = cand_capacity(k);
    const size_t M = static_cast<size_t>(cap > k ? cap : k);
    FrScratch s{};
    const size_t N = static_cast<size_t>(n_i > 0 ? n_i : 1), T = static_cast<size_t>(n_terms > 0 ? n_terms : 1);
    s.configs = cv.take<uint8_t>(N * static_cast<size_t>(n_qubytes));
    s.psi = cv.take<double2>(N);
    s.row_key_a = cv.take<uint32_t>(N);
    s.row_key_b = cv.take<uint32_t>(N);
    s.row_a = cv.take<uint32_t>(N);
    s.row_b = cv.take<uint32_t>(N);
    s.recs = cv.take<uint64_t>(T);
    s.coefs = cv.take<double2>(T);
    s.aw = cv.take<double>(T);
    s.term_key_a = cv.take<uint64_t>(T);
    s.term_key_b = cv.take<uint64_t>(T);
    s.term_a = cv.take<uint32_t>(T);
    s.term_b = cv.take<uint32_t>(T);
    s.exps = cv.take<FrExponents>(2);
    s.state = cv.take<FrState>(1);
    s.hist = cv.take<unsigned long long>(kHistBins);
    s.sel_c = cv.take<uint64_t>(static_cast<size_t>(k) * W);
    s.cand_w = cv.take<uint64_t>(static_cast<size_t>(cap));
    s.cand_c = cv.take<uint64_t>(static_cast<size_t>(cap) * W);
    s.perm_a = cv.take<uint32_t>(M);
    s.perm_b = cv.take<uint32_t>(M);
    s.key_a = cv.take<uint64_t>(M);
    s.key_b = cv.take<uint64_t>(M);
    s.flag = cv.take<uint32_t>(static_cast<size_t>(k));
    s.pos = cv.take<uint32_t>(static_cast<size_t>(k));
    size_t sort_bytes = 0, sort_desc_bytes = 0, scan_bytes = 0, row_bytes = 0, term_bytes = 0;
    (void)rocprim::radix_sort_pairs(nullptr, sort_bytes, s.key_a, s.key_b, s.perm_a, s.perm_b, static_cast<unsigned>(M));
    (void)rocprim::radix_sort_pairs_desc(nullptr, sort_desc_bytes, s.key_a, s.key_b, s.perm_a, s.perm_b, static_cast<unsigned>(M));
    (void)rocprim::exclusive_scan(nullptr, scan_bytes, s.flag, s.pos, 0u, static_cast<size_t>(k), rocprim::plus<uint32_t>());
    (void)rocprim::radix_sort_pairs_desc(nullptr, row_bytes, s.row_key_a, s.row_key_b, s.row_a, s.row_b, N);
    (void)rocprim::radix_sort_pairs(nullptr, term_bytes, s.term_key_a, s.term_key_b, s.term_a, s.term_b, T);
    size_t t = sort_bytes > sort_desc_bytes ? sort_bytes : sort_desc_bytes;
    t = t > scan_bytes ? t : scan_bytes;
    t = t > row_bytes ? t : row_bytes;
    t = t > term_bytes ? t : term_bytes;
    s.tmp = cv.take_bytes(t);
    s.tmp_bytes = t;
    return s;
}

// Sorts perm_a (an index permutation over n entries) stably by config words ascending; perm_b is free.
template <int W>
int sort_by_config(const uint64_t* words, int64_t n, FrScratch& s, hipStream_t stream) {
    for (int w = W - 1; w >= 0; --w) {
        be_word_gather_kernel<W><<<blocks_for(n), 256, 0, stream>>>(words, s.perm_a, n, w, s.key_a);
        QMB_CHECK_LAUNCH();
        size_t need = s.tmp_bytes;
        QMB_HIP_TRY(rocprim::radix_sort_pairs(s.tmp, need, s.key_a, s.key_b, s.perm_a, s.perm_b, static_cast<unsigned>(n), 0, 64,
                                              stream));
        std::swap(s.perm_a, s.perm_b);
    }
    return QMB_OK;
}

template <int W>
int find_relative_impl(const qmb_terms* terms, const qmb_targets* exclude, const uint8_t* configs_i, const double* psi_i,
                       int64_t n_i, int64_t k, uint8_t* out, int64_t* out_rows, void* scratch, size_t scratch_bytes,
                       hipStream_t stream) {
    Carver cv{static_cast<char*>(scratch), 0};
    FrScratch s = fr_layout(cv, W, terms->n_qubytes, n_i, k, terms->n_terms);
    if (cv.off > scratch_bytes) {
        return set_error(QMB_ERR_WORKSPACE, "find_relative scratch too small: need %zu, have %zu", cv.off, scratch_bytes);
    }
    const int64_t cap = cand_capacity(k);
    LaunchShape ls = resolve_launch(nullptr, W, n_i, terms->n_terms);
    if (!ls.direct) {
        // small units: what is enumerated lies in the first tiles' rows and the buckets' first terms
        ls.tile_log2 = 6;
        ls.groups = 16;
    }
    const int64_t T = terms->n_terms;
    FrParams p{};
    p.src = make_source(terms, s.configs, n_i);
    p.src.recs = s.recs;
    p.psi = s.psi;
    p.coefs = s.coefs;
    p.aw = s.aw;
    p.xkeys = exclude->keys;
    p.xtable = exclude->table;
    p.xmask = exclude->capacity - 1;
    p.xfilter = exclude->filter;
    p.xfmask = exclude->filter_words - 1;
    p.xcols = exclude->cols;
    p.state = s.state;
    p.hist = s.hist;
    p.sel_c = s.sel_c;
    p.cand_w = s.cand_w;
    p.cand_c = s.cand_c;
    p.k = k;
    p.cand_cap = cap;
    p.tile_log2 = ls.tile_log2;
    p.groups = ls.groups;
    p.direct = ls.direct ? 1 : 0;
    const int64_t tiles = (n_i + (1ll << ls.tile_log2) - 1) >> ls.tile_log2;
    const int64_t units = n_i <= 0 ? 0 : (ls.direct ? (n_i + kEnumBlock - 1) / kEnumBlock : tiles * ls.groups);
    const unsigned grid = static_cast<unsigned>(units < 4096 ? units : 4096);
    const size_t lds = ls.direct ? direct_lds_bytes(W) : enum_lds_bytes_of(W, terms->n_bits, ls.tile_log2);

    fr_init_kernel<<<1, 256, 0, stream>>>(s.state, s.hist, s.exps, k);
    QMB_CHECK_LAUNCH();
    QMB_TRY(launch_fill_u64(s.cand_w, 0ull, cap, stream));
    if (grid > 0 && T > 0) {
        QMB_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(&fr_hist_kernel<W>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
        QMB_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(&fr_collect_kernel<W>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
        QMB_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(&fr_tie_kernel<W>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
        const auto* psi = reinterpret_cast<const double2*>(psi_i);
        const auto* coefs = reinterpret_cast<const double2*>(terms->coefs);
        fr_row_keys_kernel<<<blocks_for(n_i), 256, 0, stream>>>(psi, n_i, s.row_key_a, s.row_a);
        QMB_CHECK_LAUNCH();
        size_t need = s.tmp_bytes;
        QMB_HIP_TRY(rocprim::radix_sort_pairs_desc(s.tmp, need, s.row_key_a, s.row_key_b, s.row_a, s.row_b, static_cast<size_t>(n_i), 0, 32,
                                                   stream));
        fr_row_gather_kernel<<<blocks_for(n_i), 256, 0, stream>>>(s.row_b, configs_i, psi, n_i, terms->n_qubytes, s.configs, s.psi);
        QMB_CHECK_LAUNCH();
        fr_term_keys_kernel<<<blocks_for(T), 256, 0, stream>>>(coefs, terms->bucket_start, terms->n_buckets, T, s.term_key_a, s.term_a);
        QMB_CHECK_LAUNCH();
        int bits = 33;
        while ((int64_t{1} << (bits - 32)) <= terms->n_buckets) {
            ++bits;
        }
        need = s.tmp_bytes;
        QMB_HIP_TRY(rocprim::radix_sort_pairs(s.tmp, need, s.term_key_a, s.term_key_b, s.term_a, s.term_b, static_cast<size_t>(T), 0,
                                              static_cast<unsigned>(bits), stream));
        fr_term_gather_kernel<<<blocks_for(T), 256, 0, stream>>>(s.term_b, terms->recs, coefs, T, s.recs, s.coefs, s.aw);
        QMB_CHECK_LAUNCH();
        const unsigned row_blocks = blocks_for(n_i) < 512u ? blocks_for(n_i) : 512u;
        const unsigned term_blocks = blocks_for(T) < 512u ? blocks_for(T) : 512u;
        fr_exponents_kernel<<<row_blocks + term_blocks, 256, 0, stream>>>(psi, n_i, row_blocks, coefs, T, s.exps);
        QMB_CHECK_LAUNCH();
        fr_plan_kernel<<<1, 1024, 0, stream>>>(s.state, s.psi, n_i, s.exps, k);
        QMB_CHECK_LAUNCH();
        for (int pass = 0; pass < kTries - 1 + kLevels; ++pass) {
            fr_hist_kernel<W><<<grid, kEnumBlock, lds, stream>>>(p);
            QMB_CHECK_LAUNCH();
            fr_select_kernel<<<1, 1024, 0, stream>>>(s.state, s.hist, s.psi, n_i, s.exps, cap);
            QMB_CHECK_LAUNCH();
        }
        if (n_i > cap / T) {  // else no class can exceed the buffer
            const int digits = tie_levels(terms->n_qubytes);
            for (int d = 0; d < digits; ++d) {
                fr_tie_kernel<W><<<grid < kTieGrid ? grid : kTieGrid, kEnumBlock, lds, stream>>>(p, d, digits);
                QMB_CHECK_LAUNCH();
            }
        }
        fr_collect_kernel<W><<<grid, kEnumBlock, lds, stream>>>(p);
        QMB_CHECK_LAUNCH();
    }
    // Candidates: order by (weight desc, config asc), keep the first cand_needed.
    iota_u32_kernel<<<blocks_for(cap), 256, 0, stream>>>(s.perm_a, cap);
    QMB_CHECK_LAUNCH();
    QMB_TRY(sort_by_config<W>(s.cand_c, cap, s, stream));
    u64_gather_kernel<<<blocks_for(cap), 256, 0, stream>>>(s.cand_w, s.perm_a, cap, s.key_a);
    QMB_CHECK_LAUNCH();
    size_t need = s.tmp_bytes;
    QMB_HIP_TRY(rocprim::radix_sort_pairs_desc(s.tmp, need, s.key_a, s.key_b, s.perm_a, s.perm_b, static_cast<unsigned>(cap), 0, 64,
                                               stream));
    fr_take_kernel<W><<<blocks_for(cap), 256, 0, stream>>>(s.perm_b, cap, s.cand_c, s.state, k, s.sel_c);
    QMB_CHECK_LAUNCH();
    // Selected entries: sort by config (valid entries first), drop repeats, write rows.
    iota_u32_kernel<<<blocks_for(k), 256, 0, stream>>>(s.perm_a, k);
    QMB_CHECK_LAUNCH();
    QMB_TRY(sort_by_config<W>(s.sel_c, k, s, stream));
    valid_key_kernel<<<blocks_for(k), 256, 0, stream>>>(s.perm_a, k, s.state, k, s.key_a);
    QMB_CHECK_LAUNCH();
    need = s.tmp_bytes;
    QMB_HIP_TRY(rocprim::radix_sort_pairs(s.tmp, need, s.key_a, s.key_b, s.perm_a, s.perm_b, static_cast<unsigned>(k), 0, 1, stream));
    fr_unique_flag_kernel<W><<<blocks_for(k), 256, 0, stream>>>(s.perm_b, k, s.sel_c, s.state, k, s.flag);
    QMB_CHECK_LAUNCH();
    need = s.tmp_bytes;
    QMB_HIP_TRY(rocprim::exclusive_scan(s.tmp, need, s.flag, s.pos, 0u, static_cast<size_t>(k), rocprim::plus<uint32_t>(), stream));
    fr_scatter_kernel<W><<<blocks_for(k), 256, 0, stream>>>(s.perm_b, k, s.sel_c, s.flag, s.pos, terms->n_qubytes, out, out_rows);
    QMB_CHECK_LAUNCH();
    return QMB_OK;
}

}  // namespace

size_t find_relative_scratch_bytes(int n_qubytes, int64_t n_i, int64_t count_selected, int64_t n_terms) {
    Carver cv;
    (void)fr_layout(cv, n_words_of(n_qubytes), n_qubytes, n_i, count_selected, n_terms);
    return cv.off + 256;
}

int find_relative_prepared(const qmb_terms* terms, const qmb_targets* exclude, const uint8_t* configs_i, const double* psi_i,
                           int64_t n_i, int64_t count_selected, uint8_t* out, int64_t* out_rows, void* scratch,
                           size_t scratch_bytes, hipStream_t stream) {
    if (count_selected <= 0) {
        return set_error(QMB_ERR_ARGUMENT, "count_selected must be positive, got %lld", static_cast<long long>(count_selected));
    }
    if (count_selected >= (1ll << 31)) {
        return set_error(QMB_ERR_ARGUMENT, "count_selected too large");
    }
    if (terms->n_qubytes != exclude->n_qubytes) {
        return set_error(QMB_ERR_ARGUMENT, "exclude set has a different config width");
    }
    return dispatch_words(terms->n_words, [&](auto wc) -> int {
        constexpr int W = decltype(wc)::value;
        return find_relative_impl<W>(terms, exclude, configs_i, psi_i, n_i, count_selected, out, out_rows, scratch, scratch_bytes,
                                     stream);
    });
}

}  // namespace qmb
