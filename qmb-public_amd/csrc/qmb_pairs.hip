// qmb_pairs.hip -- the pair-excitation path of apply_within on gfx950.
//
// Two configs a, b of one set are connected by a pair excitation (annihilate the pair Pa of a,
// create the pair Pb) exactly when a \ Pa == b \ Pb ("core") and Pa, Pb are disjoint.  So instead
// of generating every (config, term) target and probing the index for it -- the reference's
// scheme, qmb/_hamiltonian_cuda.cu:86-135, which for a molecular Hamiltonian spends ~90% of its
// work on double-excitation targets that are not in the set -- every config emits one entry per
// occupied pair (its cores), the entries are radix-sorted by core hash and dealt into bins by the size
// of their group, and a wave walks the groups of equal cores, combining their rows pairwise with the
// merged coefficient table of qmb_pairs.
// Only connections whose target is in the set are visited; each output row sums in registers and
// reaches HBM with one FP64 atomic per group it belongs to.
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include <vector>

#include "qmb_internal.hpp"

namespace qmb {

namespace {

constexpr int kBlock = 256;
// Sort key of a core entry, 32 bits: the core class (the number of even sites of the core mod 3)
// times kHashRange, plus the 64-bit core hash mod kHashRange.  The class is a function of the core,
// so a group never splits; in a set where every config has the same numbers of even and odd
// occupied sites (spin sectors) it tells the pair class of all the group's entries, so groups come
// in class order and waves running side by side read one block of the coefficient table.  Cores
// with equal keys share a group ("mixed"), where the kernels compare cores exactly; the modulus
// breaks the hash's linearity, so such merges are chance events (about 1 group in 100 at 12M cores
// per class) with no structure.  Unused entries get kKeySentinel and sort last.  A 32-bit key
// sorts in four 8-bit radix passes, with the packed (row, removed sites) value riding along; the
// sort is stable, so inside a group the entries keep the order they were emitted in: by the rank
// of the removed pair (order 1: site) among the row's own, then by row.
constexpr uint32_t kHashRange = 0x55555555u;  // 3 * kHashRange = 2^32 - 1
constexpr uint32_t kKeySentinel = 0xFFFFFFFFu;
constexpr int kKeyBits = 32;
// A packed core entry is one u64: key << kPackedBits | row << sub_bits | sub, sorted on bits
// [kPackedBits, kPackedBits + 32) alone.  The range ends at bit 63, not 64: rocPRIM's radix sort
// takes a merge path for small inputs whose comparison mask is (1 << end_bit) - 1 in the key type,
// which a 64-bit end_bit overflows (it then compared the low bits).
constexpr int kPackedBits = 31;
constexpr int kMaxPairBytes = 16;            // the dense table is n_pairs^2 entries

inline unsigned blocks_for(int64_t n, int block = kBlock) {
    int64_t b = (n + block - 1) / block;
    return static_cast<unsigned>(b < 1 ? 1 : b);
}

// Index of the calling wave among the persistent waves of the grid's first `blocks` blocks, ordered so that
// each XCD holds a contiguous eighth of [0, waves).  Workgroups go to the 8 XCDs round-robin by blockIdx.x, so with
// a grid that divides evenly, waves walking units w, w + waves, ... keep each XCD's L2 on the
// coefficient rows of an eighth of every window of units instead of rows from the whole window.
// Measured: the batch kernel gains (138.9 -> 134 ms on 64 molecular instances); the single-set
// pair and single kernels lose (8.07 -> 8.46 ms at 1M configs), so they keep the plain order.
__device__ __forceinline__ int64_t xcd_wave(uint32_t blocks, int64_t in_block) {
    constexpr int kXcds = 8;
    constexpr int64_t kWavesPerBlock = kBlock / 64;
    if (blocks % kXcds != 0) {
        return static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + in_block;
    }
    const int64_t waves = static_cast<int64_t>(blocks) * kWavesPerBlock;
    return static_cast<int64_t>(blockIdx.x % kXcds) * (waves / kXcds) + static_cast<int64_t>(blockIdx.x / kXcds) * kWavesPerBlock +
           in_block;
}

__global__ void zero_counts_kernel(int64_t* counts) {
    if (threadIdx.x < 4) {
        counts[threadIdx.x] = 0;
    }
}

// ------------------------------------------------------------------------------ coefficients --
// A diagonal term needs every site it touches back in its first state, so each of its sites carries
// an even number of its (at most four) operators: it conditions at most two sites, and its sign is
// the constant (-1)^pconst.  Its indicator prod_s (v_s ? n_s : 1 - n_s) expands into a constant,
// per-site and per-site-pair part: diag[0], diag[1 + p], diag[1 + n_bits + pair_index(p, q)].
__device__ __forceinline__ void add2(double2* d, double sgn, const double2& v) {
    unsafeAtomicAdd(&d->x, sgn * v.x);
    unsafeAtomicAdd(&d->y, sgn * v.y);
}

__device__ void fold_diagonal(uint64_t rec, int particle_cut, int n_bits, const double2& coef, double2* diag) {
    const uint32_t valid = static_cast<uint32_t>(rec >> 32) & 0xf;
    const uint32_t req = static_cast<uint32_t>(rec >> 36) & 0xf;
    const int pconst = particle_cut == 1 ? static_cast<int>((rec >> 48) & 1) : 0;
    const double2 v = pconst ? make_double2(-coef.x, -coef.y) : coef;
    int sites[2], occ[2], ns = 0;
    for (int u = 0; u < 4; ++u) {
        if ((valid >> u) & 1u) {
            if (ns < 2) {
                sites[ns] = static_cast<int>((rec >> (8 * u)) & 0xff);
                occ[ns] = static_cast<int>((req >> u) & 1u);
            }
            ++ns;
        }
    }
    double2* e1 = diag + 1;
    double2* e2 = diag + 1 + n_bits;
    if (ns == 0) {
        add2(diag, 1.0, v);
    } else if (ns == 1) {
        if (occ[0]) {
            add2(e1 + sites[0], 1.0, v);
        } else {
            add2(diag, 1.0, v);
            add2(e1 + sites[0], -1.0, v);
        }
    } else if (ns == 2) {
        const int p = sites[0] < sites[1] ? sites[0] : sites[1];
        const int q = sites[0] < sites[1] ? sites[1] : sites[0];
        const int op = sites[0] < sites[1] ? occ[0] : occ[1];
        const int oq = sites[0] < sites[1] ? occ[1] : occ[0];
        double2* pq = e2 + pair_index(p, q);
        // (op ? n_p : 1 - n_p) (oq ? n_q : 1 - n_q)
        add2(pq, (op == oq) ? 1.0 : -1.0, v);
        if (!oq) {
            add2(e1 + p, op ? 1.0 : -1.0, v);
        }
        if (!op) {
            add2(e1 + q, oq ? 1.0 : -1.0, v);
        }
        if (!op && !oq) {
            add2(diag, 1.0, v);
        }
    }
}

// *counter += the lanes of the wave where `add` holds, as one atomic from the wave's first such lane
// (a same-address atomic per thread serialises: 600k of them took 7 ms).  Every lane must call it.
__device__ __forceinline__ void wave_count(int64_t* counter, bool add) {
    const uint64_t m = __ballot(add);
    if (m != 0ull && static_cast<int>(threadIdx.x & 63u) == __builtin_ctzll(m)) {
        atomicAdd(reinterpret_cast<unsigned long long*>(counter), static_cast<unsigned long long>(__popcll(m)));
    }
}

// The part of pair_parity that the excitation's own sites decide.  The source config is the core
// with {r0, r1}, so popcount(c & ([r0, r1) ^ [c0, c1))) = popcount(core & [r0, r1)) + popcount(core &
// [c0, c1)) + 1 (r0 in its own range) + the sites of {r0, r1} in [c0, c1).  The last two go into the
// table; the first two are one sign per (core, pair), the entry's own, so the group kernels multiply
// two entry signs in and compute no parity per pair.
__device__ __forceinline__ int pair_own_parity(int r0, int r1, int c0, int c1) {
    return 1 ^ static_cast<int>(r0 >= c0 && r0 < c1) ^ static_cast<int>(r1 >= c0 && r1 < c1);
}

// Launched with whole waves: threads past n_terms take part in the counts only.
__global__ void pairs_fill_kernel(const int16_t* __restrict__ site, const uint8_t* __restrict__ kind,
                                  const double2* __restrict__ coef, int64_t n_terms, int particle_cut, int n_bits,
                                  int64_t n_pairs, double2* __restrict__ table, double2* __restrict__ diag,
                                  int64_t* __restrict__ counts) {
    const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    bool is_diag = false, is_pair = false;
    if (t < n_terms) {
        const CompiledTerm c = compile_term(site + 4 * t, kind + 4 * t, particle_cut, n_bits);
        PairExcitation e;
        if (c.status == kCompileOk && c.diagonal) {
            fold_diagonal(c.rec, particle_cut, n_bits, coef[t], diag);
            is_diag = true;
        } else if (c.status == kCompileOk && pair_excitation(c.rec, particle_cut, &e)) {
            const double2 v = coef[t];
            double2* dst = table + pair_slot(e.r0, e.r1, n_bits) * n_pairs + pair_slot(e.c0, e.c1, n_bits);
            const int flip = e.delta ^ (particle_cut == 1 ? pair_own_parity(e.r0, e.r1, e.c0, e.c1) : 0);
            unsafeAtomicAdd(&dst->x, flip ? -v.x : v.x);
            unsafeAtomicAdd(&dst->y, flip ? -v.y : v.y);
            is_pair = true;
        }
    }
    wave_count(&counts[0], is_pair);
    wave_count(&counts[1], is_diag);
}

int pairs_layout(Carver& cv, int n_qubytes, qmb_pairs* out) {
    QMB_TRY(check_qubytes(n_qubytes));
    if (n_qubytes > kMaxPairBytes) {
        return set_error(QMB_ERR_UNSUPPORTED, "the pair-excitation table supports n_qubytes <= %d, got %d", kMaxPairBytes,
                         n_qubytes);
    }
    qmb_pairs p{};
    p.n_qubytes = n_qubytes;
    p.n_bits = 8 * n_qubytes;
    p.n_pairs = static_cast<int64_t>(p.n_bits) * (p.n_bits - 1) / 2;
    p.buffer = cv.base;
    p.counts = cv.take<int64_t>(4);
    p.coef = cv.take<double>(2 * static_cast<size_t>(p.n_pairs) * static_cast<size_t>(p.n_pairs));
    p.coef_re = cv.take<double>(static_cast<size_t>(p.n_pairs) * static_cast<size_t>(p.n_pairs));
    p.diag = cv.take<double>(2 * (1 + static_cast<size_t>(p.n_bits) + static_cast<size_t>(p.n_pairs)));
    p.bytes = cv.off;
    if (out) {
        *out = p;
    }
    return QMB_OK;
}

// Real parts of the merged coefficients; counts[2] += entries with a nonzero imaginary part, counts[3] +=
// entries that are not finite.
__global__ void pairs_real_kernel(const double2* __restrict__ coef, int64_t n, double* __restrict__ re, int64_t* __restrict__ counts) {
    const int64_t k = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (k >= n) {
        return;
    }
    const double2 v = coef[k];
    re[k] = v.x;
    if (v.y != 0.0) {
        atomicAdd(reinterpret_cast<unsigned long long*>(&counts[2]), 1ull);
    }
    if (!(fabs(v.x) < INFINITY)) {
        atomicAdd(reinterpret_cast<unsigned long long*>(&counts[3]), 1ull);
    }
}

// ----------------------------------------------------------------------------------- cores --
template <int W>
__device__ __forceinline__ Cfg<W> load_key(const uint64_t* __restrict__ keys, int64_t i) {
    Cfg<W> c;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        c.w[w] = keys[i * W + w];
    }
    return c;
}

// Sites in [a, b), a <= b: L(a) ^ L(b) with L(s) the sites below s.
template <int W>
__device__ __forceinline__ Cfg<W> range_mask(int a, int b) {
    Cfg<W> m;
    if (W == 1) {
        m.w[0] = (1ull << b) - (1ull << a);  // sites of a one-word config are < 64
    } else {
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const int lo = a - 64 * w, hi = b - 64 * w;
            const uint64_t mh = hi <= 0 ? 0ull : (hi >= 64 ? ~0ull : (1ull << hi) - 1ull);
            const uint64_t ml = lo <= 0 ? 0ull : (lo >= 64 ? ~0ull : (1ull << lo) - 1ull);
            m.w[w] = mh & ~ml;
        }
    }
    return m;
}

template <int W>
__device__ __forceinline__ int masked_parity(const Cfg<W>& c, const Cfg<W>& m) {
    int par = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        par ^= __popcll(c.w[w] & m.w[w]);
    }
    return par & 1;
}

template <int W>
__device__ __forceinline__ void flip_site(Cfg<W>& c, int s) {
#pragma unroll
    for (int w = 0; w < W; ++w) {
        if (w == (s >> 6)) {
            c.w[w] ^= 1ull << (s & 63);
        }
    }
}

__device__ __forceinline__ uint64_t shfl_u64(uint64_t v, int lane) {
    const uint32_t lo = __shfl(static_cast<uint32_t>(v), lane);
    const uint32_t hi = __shfl(static_cast<uint32_t>(v >> 32), lane);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

__device__ __forceinline__ uint32_t core_key(uint64_t h, uint32_t cls) {
    return cls * kHashRange + static_cast<uint32_t>(h % kHashRange);
}

// One thread per config: every occupied pair (x < y) -- ORDER 2 -- or every occupied site x --
// ORDER 1 -- gives the entry (key of the config without those sites, row << 16 | y << 8 | x); unused
// slots of a row with fewer occupied sites get the sentinel key.  Entry k of row i sits at k * n + i,
// so the lanes of a wave store to consecutive addresses.  A row's pairs are emitted in pair_slot
// order (even-even pairs, then odd-odd, each by the higher site first; then even-odd, by the even
// site first) and its sites in ascending order.  Rows of one group share the core, so a pair's rank
// among its row's pairs grows with its slot (ties where no core site lies between two slots), and
// the stable sort leaves each group's entries close to ascending slots: the lanes of a wave then
// read nearby columns of a coefficient table row.
template <int W, int ORDER, typename Emit>
__device__ __forceinline__ void emit_cores(const Cfg<W>& c, const uint64_t* __restrict__ cols, Emit&& emit) {
    constexpr uint64_t kEven = 0x5555555555555555ull;
    const uint64_t h = hash_cfg<W>(c, cols);
    int even = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        even += __popcll(c.w[w] & kEven);
    }
    if (ORDER == 1) {
#pragma unroll
        for (int wx = 0; wx < W; ++wx) {
            uint64_t mx = c.w[wx];
            while (mx) {
                const int x = 64 * wx + __builtin_ctzll(mx);
                mx &= mx - 1;
                emit(core_key(h ^ cols[x], 0u), static_cast<uint32_t>(x));
            }
        }
    } else {
        // same-parity pairs: the core loses two even sites (parity 0) or none (parity 1)
        for (int par = 0; par < 2; ++par) {
            const uint64_t pm = par ? ~kEven : kEven;
            const uint32_t cls = static_cast<uint32_t>((even - (par ? 0 : 2)) % 3);
#pragma unroll
            for (int wy = 0; wy < W; ++wy) {
                uint64_t my = c.w[wy] & pm;
                while (my) {
                    const int y = 64 * wy + __builtin_ctzll(my);
                    my &= my - 1;
                    const uint64_t hy = h ^ cols[y];
#pragma unroll
                    for (int wx = 0; wx < W; ++wx) {
                        if (wx > wy) {
                            continue;
                        }
                        uint64_t mx = c.w[wx] & pm & (wx == wy ? (1ull << (y & 63)) - 1ull : ~0ull);
                        while (mx) {
                            const int x = 64 * wx + __builtin_ctzll(mx);
                            mx &= mx - 1;
                            emit(core_key(hy ^ cols[x], cls), (static_cast<uint32_t>(y) << 8) | static_cast<uint32_t>(x));
                        }
                    }
                }
            }
        }
        // even-odd pairs: the core loses one even site
        const uint32_t cls = static_cast<uint32_t>((even - 1) % 3);
#pragma unroll
        for (int we = 0; we < W; ++we) {
            uint64_t me = c.w[we] & kEven;
            while (me) {
                const int ev = 64 * we + __builtin_ctzll(me);
                me &= me - 1;
                const uint64_t he = h ^ cols[ev];
#pragma unroll
                for (int wo = 0; wo < W; ++wo) {
                    uint64_t mo = c.w[wo] & ~kEven;
                    while (mo) {
                        const int od = 64 * wo + __builtin_ctzll(mo);
                        mo &= mo - 1;
                        const int x = ev < od ? ev : od;
                        const int y = ev < od ? od : ev;
                        emit(core_key(he ^ cols[od], cls), (static_cast<uint32_t>(y) << 8) | static_cast<uint32_t>(x));
                    }
                }
            }
        }
    }
}

template <int W, int ORDER, bool PACKED>
__global__ void core_emit_kernel(const uint64_t* __restrict__ keys, const uint64_t* __restrict__ cols, int64_t n, int n_bits,
                                 int per_config, int sub_bits, uint32_t* __restrict__ okeys, void* __restrict__ ovals,
                                 int64_t* __restrict__ counts) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= n) {
        return;
    }
    int64_t k = 0;
    // the value: row << 16 | y << 8 | x, or packed into 32 bits as row << sub_bits | (pair slot of
    // (x, y), or the site x); the packed value halves what the sort moves per value
    emit_cores<W, ORDER>(load_key<W>(keys, i), cols, [&](uint32_t key, uint32_t sites) {
        if (k < per_config) {
            if (PACKED) {
                const uint32_t sub =
                    ORDER == 2 ? static_cast<uint32_t>(pair_slot(static_cast<int>(sites & 0xff), static_cast<int>(sites >> 8), n_bits)) : sites;
                static_cast<uint64_t*>(ovals)[k * n + i] = (static_cast<uint64_t>(key) << kPackedBits) | ((static_cast<uint32_t>(i) << sub_bits) | sub);
            } else {
                okeys[k * n + i] = key;
                static_cast<uint64_t*>(ovals)[k * n + i] = (static_cast<uint64_t>(i) << 16) | sites;
            }
        }
        ++k;
    });
    if (k > per_config) {
        atomicAdd(reinterpret_cast<unsigned long long*>(&counts[2]), 1ull);
    }
    for (; k < per_config; ++k) {
        if (PACKED) {
            static_cast<uint64_t*>(ovals)[k * n + i] = static_cast<uint64_t>(kKeySentinel) << kPackedBits;
        } else {
            okeys[k * n + i] = kKeySentinel;
            static_cast<uint64_t*>(ovals)[k * n + i] = 0ull;
        }
    }
}

// Start of a build: counts = 0, and (inv non-null) inv[pair_slot(x, y)] = y << 8 | x for every pair
// x < y of n_bits sites.
__global__ void cores_init_kernel(int64_t* __restrict__ counts, int n_bits, uint32_t* __restrict__ inv) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < 4) {
        counts[t] = 0;
    }
    if (inv == nullptr || t >= n_bits * n_bits) {
        return;
    }
    const int x = t % n_bits, y = t / n_bits;
    if (x < y) {
        inv[pair_slot(x, y, n_bits)] = (static_cast<uint32_t>(y) << 8) | static_cast<uint32_t>(x);
    }
}

// Flags of a used sorted core entry: the first entry of its key (a group head, bit 0) and an entry
// whose core differs from the previous entry's under the same key (two cores merged by equal keys,
// kFlagBreak); entries of groups of two or more also carry their sign (kFlagSign): the parity of the
// core's sites in [x, y) (order 2) or below x (order 1), one factor of every element the entry takes
// part in.  One byte per entry.  Unused slots (the sentinel keys, sorted last) get 0; the flag pass writes the number of
// used entries to counts[0] and each wave's number of heads to its chunk's counter; a head's group
// is the heads before its chunk (an exclusive scan of the counters) plus those before it in the chunk.
constexpr uint32_t kFlagHead = 1u;
constexpr uint32_t kFlagSign = 2u;
constexpr uint32_t kFlagBreak = 4u;
// Bit 31 of starts[g] (g < G): group g holds more than one core (its rows' cores are compared exactly).
constexpr uint32_t kGroupMixed = 0x80000000u;
constexpr uint32_t kGroupStart = 0x7FFFFFFFu;

// The core of an entry (row << 16 | y << 8 | x; order 1: row << 16 | x): its row's config without
// the entry's sites.
template <int W, int ORDER>
__device__ __forceinline__ Cfg<W> entry_core(const uint64_t* __restrict__ ckeys, uint64_t v) {
    Cfg<W> c = load_key<W>(ckeys, static_cast<int64_t>(v >> 16));
    flip_site<W>(c, static_cast<int>(v & 0xff));
    if (ORDER == 2) {
        flip_site<W>(c, static_cast<int>((v >> 8) & 0xff));
    }
    return c;
}

template <int ORDER>
__device__ __forceinline__ uint64_t unpack_entry(uint64_t x, int sub_bits, const uint32_t* __restrict__ inv) {
    const uint32_t pv = static_cast<uint32_t>(x & ((uint64_t{1} << kPackedBits) - 1u));
    const uint32_t sub = pv & ((1u << sub_bits) - 1u);
    return (static_cast<uint64_t>(pv >> sub_bits) << 16) | (ORDER == 2 ? inv[sub] : sub);
}

// Flags of kFlagUnroll * 64 consecutive sorted entries per wave: entry base + 64 t + lane in slot t of
// each lane.  A wave loads its entries once (the neighbours' keys come from the lanes beside, across
// slots from lane 63 / lane 0 of the slot beside, and the wave's outer neighbours are read by lanes 0
// and 63).  Only entries of groups of two or more read their config: each compares its core with
// the previous entry's, taken the same way; the slots' config loads are independent, so a lane keeps
// kFlagUnroll of them in flight.  Every lane runs every shuffle.  load(j, k, v) reads entry j < cap.
constexpr int kFlagUnroll = 4;

template <int W, int ORDER, typename Load>
__device__ __forceinline__ void core_flags(const uint64_t* __restrict__ ckeys, int64_t cap, Load load, uint32_t (&f)[kFlagUnroll],
                                           uint32_t (&k)[kFlagUnroll], uint64_t (&v)[kFlagUnroll], int64_t base, int lane,
                                           int64_t* __restrict__ counts) {
    constexpr int U = kFlagUnroll;
#pragma unroll
    for (int t = 0; t < U; ++t) {
        k[t] = kKeySentinel;
        v[t] = 0ull;
        const int64_t e = base + 64 * t + lane;
        if (e < cap) {
            load(e, k[t], v[t]);
        }
    }
    // the wave's outer neighbours
    uint32_t k_before = kKeySentinel, k_after = kKeySentinel;
    uint64_t v_before = 0ull;
    if (lane == 0 && base > 0 && base <= cap) {
        load(base - 1, k_before, v_before);
    }
    if (lane == 63 && base + 64 * U < cap) {
        uint64_t v_after;
        load(base + 64 * U, k_after, v_after);
    }
    uint32_t kp[U], kn[U];
#pragma unroll
    for (int t = 0; t < U; ++t) {
        const uint32_t below = __shfl(k[t], (lane + 63) & 63);
        const uint32_t above = __shfl(k[t], (lane + 1) & 63);
        const uint32_t prev_slot = __shfl(k[t > 0 ? t - 1 : 0], 63);
        const uint32_t next_slot = __shfl(k[t < U - 1 ? t + 1 : U - 1], 0);
        kp[t] = lane != 0 ? below : (t > 0 ? prev_slot : k_before);
        kn[t] = lane != 63 ? above : (t < U - 1 ? next_slot : k_after);
    }
    Cfg<W> core[U];
#pragma unroll
    for (int t = 0; t < U; ++t) {
        const bool used = k[t] != kKeySentinel;
        const bool multi = used && (kp[t] == k[t] || kn[t] == k[t]);
#pragma unroll
        for (int w = 0; w < W; ++w) {
            core[t].w[w] = 0ull;
        }
        if (multi) {
            core[t] = entry_core<W, ORDER>(ckeys, v[t]);
        }
    }
    Cfg<W> core_before{};
    if (lane == 0 && k_before != kKeySentinel && k_before == k[0]) {
        core_before = entry_core<W, ORDER>(ckeys, v_before);
    }
#pragma unroll
    for (int t = 0; t < U; ++t) {
        bool same = true;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const uint64_t below = shfl_u64(core[t].w[w], (lane + 63) & 63);
            const uint64_t prev_slot = shfl_u64(core[t > 0 ? t - 1 : 0].w[w], 63);
            const uint64_t prev = lane != 0 ? below : (t > 0 ? prev_slot : core_before.w[w]);
            same = same & (prev == core[t].w[w]);
        }
        const bool used = k[t] != kKeySentinel;
        const bool head = used && kp[t] != k[t];
        f[t] = !used ? 0u : (head ? kFlagHead : (same ? 0u : kFlagBreak));
        // the core is empty (parity 0) for an entry alone in its group
        const int lo = ORDER == 2 ? static_cast<int>(v[t] & 0xff) : 0;
        const int hi = static_cast<int>((ORDER == 2 ? v[t] >> 8 : v[t]) & 0xff);
        f[t] |= used && masked_parity<W>(core[t], range_mask<W>(lo, hi)) != 0 ? kFlagSign : 0u;
        if (used && kn[t] == kKeySentinel) {
            counts[0] = base + 64 * t + lane + 1;  // the last used entry
        }
    }
}

// out = exclusive sums of in[0, n), by the calling block of kBlock threads.
__device__ __forceinline__ void block_scan(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int64_t n) {
    __shared__ uint32_t s_wave[kBlock / 64];
    constexpr int V = 16;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t carry = 0;
    for (int64_t base = 0; base < n; base += kBlock * V) {
        const int64_t at = base + V * static_cast<int64_t>(threadIdx.x);
        uint32_t v[V], sum = 0;
#pragma unroll
        for (int k = 0; k < V; ++k) {
            v[k] = at + k < n ? in[at + k] : 0u;
            sum += v[k];
        }
        uint32_t incl = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(incl, d);
            incl += lane >= d ? o : 0u;
        }
        if (lane == 63) {
            s_wave[wave] = incl;
        }
        __syncthreads();
        uint32_t run = carry + incl - sum;
#pragma unroll
        for (int w = 0; w < kBlock / 64; ++w) {
            run += w < wave ? s_wave[w] : 0u;
            carry += s_wave[w];
        }
#pragma unroll
        for (int k = 0; k < V; ++k) {
            if (at + k < n) {
                out[at + k] = run;
            }
            run += v[k];
        }
        __syncthreads();
    }
}

// Counters one block scans (16K: four rounds, under 10 us); more go through a device scan.  The kernel
// writing them does not let its last block do it: the device-scope fence that takes writes back the L2
// (the flag kernel of 450,000 entries 7 -> 59 us).
constexpr int64_t kBlockScanMax = 1 << 14;

__global__ __launch_bounds__(kBlock) void block_scan_kernel(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int64_t n) {
    block_scan(in, out, n);
}

// Entries per flag chunk: one wave's kFlagUnroll * 64 consecutive entries.
constexpr int kFlagChunk = 64 * kFlagUnroll;

inline int64_t flag_chunks(int64_t cap) { return static_cast<int64_t>(blocks_for(cap, kBlock * kFlagUnroll)) * (kBlock / 64); }

// chunk_heads[c] = number of group heads among the entries of chunk c (the wave's own).  Every wave
// of the grid writes its chunk, also past the entries.
__device__ __forceinline__ void store_chunk_heads(const uint32_t (&f)[kFlagUnroll], int64_t base, int lane,
                                                  uint32_t* __restrict__ chunk_heads) {
    uint32_t heads = 0;
#pragma unroll
    for (int t = 0; t < kFlagUnroll; ++t) {
        heads += static_cast<uint32_t>(__popcll(__ballot((f[t] & kFlagHead) != 0u)));
    }
    if (lane == 0) {
        chunk_heads[base / kFlagChunk] = heads;
    }
}

// Flags of packed entries (key << 31 | row << sub_bits | sub, sorted on the key); also splits each
// entry into its key and its value in the kernels' form (row << 16 | y << 8 | x), and counts each
// chunk's heads.  Grid: flag_chunks(cap) waves of kFlagChunk entries.
template <int W, int ORDER>
__global__ __launch_bounds__(kBlock) void core_flag_unpack_kernel(const uint64_t* __restrict__ entries, int64_t cap,
                                                                  uint8_t* __restrict__ flag, uint32_t* __restrict__ chunk_heads,
                                                                  int sub_bits, const uint32_t* __restrict__ inv,
                                                                  const uint64_t* __restrict__ ckeys, uint32_t* __restrict__ keys,
                                                                  uint64_t* __restrict__ vals, int64_t* __restrict__ counts) {
    const int lane = threadIdx.x & 63;
    const int64_t base = (blockIdx.x * static_cast<int64_t>(blockDim.x) + (threadIdx.x & ~63)) * kFlagUnroll;
    auto load = [&](int64_t j, uint32_t& kj, uint64_t& vj) {
        const uint64_t xj = entries[j];
        kj = static_cast<uint32_t>(xj >> kPackedBits);
        vj = kj != kKeySentinel ? unpack_entry<ORDER>(xj, sub_bits, inv) : 0ull;
    };
    uint32_t f[kFlagUnroll], k[kFlagUnroll];
    uint64_t v[kFlagUnroll];
    core_flags<W, ORDER>(ckeys, cap, load, f, k, v, base, lane, counts);
    store_chunk_heads(f, base, lane, chunk_heads);
#pragma unroll
    for (int t = 0; t < kFlagUnroll; ++t) {
        const int64_t e = base + 64 * t + lane;
        if (e < cap) {
            flag[e] = static_cast<uint8_t>(f[t]);
            keys[e] = k[t];
            vals[e] = v[t];
        }
    }
}

// Flags of sorted (key, value) pairs and each chunk's heads, as core_flag_unpack_kernel.
template <int W, int ORDER>
__global__ __launch_bounds__(kBlock) void core_flag_kernel(const uint32_t* __restrict__ keys, const uint64_t* __restrict__ vals, int64_t cap,
                                                           const uint64_t* __restrict__ ckeys, uint8_t* __restrict__ flag,
                                                           uint32_t* __restrict__ chunk_heads, int64_t* __restrict__ counts) {
    const int lane = threadIdx.x & 63;
    const int64_t base = (blockIdx.x * static_cast<int64_t>(blockDim.x) + (threadIdx.x & ~63)) * kFlagUnroll;
    auto load = [&](int64_t j, uint32_t& kj, uint64_t& vj) {
        kj = keys[j];
        vj = vals[j];
    };
    uint32_t f[kFlagUnroll], k[kFlagUnroll];
    uint64_t v[kFlagUnroll];
    core_flags<W, ORDER>(ckeys, cap, load, f, k, v, base, lane, counts);
    store_chunk_heads(f, base, lane, chunk_heads);
#pragma unroll
    for (int t = 0; t < kFlagUnroll; ++t) {
        const int64_t e = base + 64 * t + lane;
        if (e < cap) {
            flag[e] = static_cast<uint8_t>(f[t]);
        }
    }
}

// flag[e] = 1 where a sorted key differs from the previous one (the strings index).
__global__ void key_flag_kernel(const uint32_t* __restrict__ keys, int64_t n, uint32_t* __restrict__ flag) {
    const int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (e >= n) {
        return;
    }
    const uint32_t k = keys[e];
    flag[e] = (k != kKeySentinel && (e == 0 || keys[e - 1] != k)) ? 1u : 0u;
}

// starts[g] = first entry of group g, with kGroupMixed when a break lies inside the group;
// starts[G] = number of used entries; counts {entries, G}.  One wave per flag chunk, 64 flags at a
// time: chunk_off[c] = heads before chunk c (the exclusive scan of the chunks' head counts), so a
// head's group is that plus the heads before it in the chunk.  A head finds its group's end (the
// next head or the end of the used entries) and the breaks before it from the wave's ballots; the
// last head of the 64, whose group may run past them, reads on 64 flags at a time with the whole
// wave.  Grid: flag_chunks(capacity) waves.
__global__ __launch_bounds__(kBlock) void core_start_kernel(const uint8_t* __restrict__ flag, const uint32_t* __restrict__ chunk_off,
                                                            uint32_t* __restrict__ starts, int64_t* __restrict__ counts) {
    const int lane = threadIdx.x & 63;
    const int64_t used = counts[0];
    const int64_t chunk = (blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x) >> 6;
    const uint64_t below = (1ull << lane) - 1ull;                    // lanes below this one
    const uint64_t after = lane == 63 ? 0ull : ~0ull << (lane + 1);  // lanes above this one
    if (chunk * kFlagChunk >= used) {
        return;  // the whole wave
    }
    uint32_t g0 = chunk_off[chunk];
    for (int t = 0; t < kFlagUnroll; ++t) {
        const int64_t base = chunk * kFlagChunk + 64 * t;
        if (base >= used) {
            break;  // the whole wave
        }
        const int64_t e = base + lane;
        const uint32_t f = e < used ? flag[e] : 0u;
        const bool head = (f & kFlagHead) != 0u;
        const uint64_t heads = __ballot(head);
        const uint64_t stop = __ballot(e >= used || head);
        const uint64_t brk = __ballot((f & kFlagBreak) != 0u);
        const uint64_t next = stop & after;
        // the group of the 64's last head runs on past them when no stop follows it
        const bool open = head && next == 0ull;
        const uint64_t open_mask = __ballot(open);
        bool tail_break = false;
        int64_t tail_end = 0;
        if (open_mask != 0ull) {
            for (int64_t j0 = base + 64;; j0 += 64) {
                const int64_t j = j0 + lane;
                const uint32_t fj = j < used ? flag[j] : 0u;
                const uint64_t st = __ballot(j >= used || (fj & kFlagHead) != 0u);
                const uint64_t bk = __ballot((fj & kFlagBreak) != 0u);
                if (st != 0ull) {
                    const int nx = __builtin_ctzll(st);
                    tail_break = tail_break || (bk & ((1ull << nx) - 1ull)) != 0ull;
                    tail_end = j0 + nx;
                    break;
                }
                tail_break = tail_break || bk != 0ull;
            }
        }
        if (head) {
            bool mixed;
            int64_t end;
            if (open) {
                mixed = (brk & after) != 0ull || tail_break;
                end = tail_end;
            } else {
                const int nx = __builtin_ctzll(next);
                mixed = (brk & after & ((1ull << nx) - 1ull)) != 0ull;
                end = base + nx;
            }
            const uint32_t g = g0 + static_cast<uint32_t>(__popcll(heads & below));
            starts[g] = static_cast<uint32_t>(e) | (mixed ? kGroupMixed : 0u);
            if (end == used) {
                starts[g + 1] = static_cast<uint32_t>(end);
                counts[1] = static_cast<int64_t>(g) + 1;
            }
        }
        g0 += static_cast<uint32_t>(__popcll(heads));
    }
}

// ------------------------------------------------------------------------------- group bins --
// The groups of two or more entries, dealt into bins by size: one bin per size from 2 to 32, then
// ranges of larger sizes, then what the mixed groups split into (any size).  The entries of a bin's groups are
// copied next to each other in the form the group kernels use (row | slot << 32 | sign << 63, the
// slot pair_slot of the removed pair, order 1 the removed site), so
//   - a wave takes groups of one size: its lane layout is a division by that size, every lane group
//     runs the same number of steps and the entries are one coalesced read (a wave that took 64
//     consecutive groups of every size left half of its lanes idle in the groups of 9 to 32);
//   - the groups of one entry (two thirds of them at 1M molecular configs) are never visited again;
//   - no pair kernel reads a config or counts a bit: the sign is a factor of the entry.
// Binning the 91M entries of 1M configs (52 spin orbitals) costs 0.75 ms once per index; one
// application's pair kernel went from 5.90 to 5.02 ms, the single kernel from 1.57 to 1.12 ms (and 7.6
// to 5.0 ms for the pair kernel of 200,000 two-word configs).
// A mixed group (different cores under one key, about 1 in 100) is split by core when it is binned, so
// the group kernels compare no cores either: its entries move to mvals core by core, and each core's
// group of two or more takes one of the floor(size / 2) slots the mixed group has in the list.
// Within a bin the groups keep the key order up to the order inside a block of bin_groups() groups.
constexpr int kExactMax = 32;
constexpr int kExactBins = kExactMax - 1;
constexpr int kBigBins = 7;                       // up to 48, 64, 96, 128, 192, 256 and above
constexpr int kSplitBin = kExactBins + kBigBins;  // the mixed groups, split by core
constexpr int kBins = kSplitBin + 1;
constexpr int kVarBins = kBins - kExactBins;      // bins whose groups are listed with their size
constexpr int kBinRows = kBins + kVarBins;        // counters per block: groups per bin, entries per listed bin
constexpr int kBinGroupsMax = 4096;               // groups per block of the two binning kernels, at most
constexpr uint32_t kSplitSlots = 16;              // list slots per work unit of the split bin

struct CoreBins {
    uint32_t groups[kBins];
    uint32_t entry_base[kBins];       // first entry of the bin in mvals
    uint32_t list_base[kBins];        // listed bins: first entry of the bin in glist
    uint32_t unit_start[kBins + 1];   // work units before the bin at this position (bins in descending order)
};

__device__ __forceinline__ int group_bin(uint32_t size, bool mixed) {
    if (mixed) {
        return kSplitBin;
    }
    if (size <= kExactMax) {
        return static_cast<int>(size) - 2;
    }
    const int lg = 31 - __clz(size - 1u);                     // 33..64: 5, 65..128: 6, 129..256: 7
    const int half = static_cast<int>(((size - 1u) >> (lg - 1)) & 1u);
    const int k = 2 * (lg - 5) + half;
    return kExactBins + (k < kBigBins ? k : kBigBins - 1);
}

// A group above 64 entries is listed once per 64 of its rows: a wave each, with all its entries.  (With
// one wave for a whole group the few hundred groups of 130 to 700 entries were the kernel's tail: 200,000
// two-word configs 5.0 -> 4.5 ms, a batch of 12 sets 4.1 -> 3.7 ms.)  A list element is
// {first entry, size | tile << 16}; from 2^16 entries on (only with repeated configs) it is
// {first entry, size | kWholeGroup}, for one wave.
constexpr uint32_t kTiledMax = 0xffffu;
constexpr uint32_t kWholeGroup = 0x80000000u;
__device__ __forceinline__ uint32_t group_tiles(uint32_t size) { return size <= kTiledMax ? (size + 63u) / 64u : 1u; }
__device__ __forceinline__ uint2 listed_tile(uint32_t first, uint32_t size, uint32_t tile) {
    return make_uint2(first, size <= kTiledMax ? size | (tile << 16) : size | kWholeGroup);
}
// Elements a group of bin b adds to the bin's count.
__device__ __forceinline__ uint32_t bin_items(int b, uint32_t size) { return b >= kExactBins && b < kSplitBin ? group_tiles(size) : 1u; }

// A work unit of a bin of size g: this many passes of 64 lanes (64 / g groups each), so that a unit of
// small groups is worth its decoding and keeps a few gathers in flight.
__host__ __device__ __forceinline__ int unit_passes(int g, int order) {
    if (order == 1) {
        return g <= 3 ? 2 : 1;
    }
    return g == 2 ? 8 : (g <= 4 ? 4 : (g <= 8 ? 2 : 1));
}

// Groups per block of the binning kernels: the fewest (a wave walks its part of the block's entries one
// after another) that keep the counters within what one block scans.
inline int bin_groups(int64_t cap) {
    int g = 2 * kBlock;
    while (g < kBinGroupsMax && (cap + g - 1) / g * kBinRows >= kBlockScanMax) {
        g <<= 1;
    }
    return g;
}

inline int64_t bin_blocks(int64_t cap) { return (cap + bin_groups(cap) - 1) / bin_groups(cap); }

// Bin table from the bins' groups and entries, thread b of the block calling it with bin b's (every
// thread of the block calls it).
__device__ __forceinline__ void bin_table(int b, uint32_t n, uint32_t entries, int order, CoreBins* __restrict__ bins) {
    __shared__ uint32_t s_entries[kBins], s_units[kBins], s_list[kBins];
    if (b < kBins) {
        const bool listed = b >= kExactBins;
        const int g = b + 2;
        const uint32_t per_unit = listed ? 1u : static_cast<uint32_t>(64 / g * unit_passes(g, order));
        s_entries[b] = entries;
        // the split bin: a slot per two entries of its mixed groups
        const uint32_t slots = b == kSplitBin ? s_entries[b] / 2u : n;
        s_units[b] = b == kSplitBin ? (slots + kSplitSlots - 1u) / kSplitSlots : (n + per_unit - 1u) / per_unit;
        s_list[b] = listed ? slots : 0u;
        bins->groups[b] = slots;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t e = 0, l = 0, u = 0;
        for (int k = 0; k < kBins; ++k) {
            bins->entry_base[k] = e;
            bins->list_base[k] = l;
            e += s_entries[k];
            l += s_list[k];
        }
        for (int p = 0; p < kBins; ++p) {
            bins->unit_start[p] = u;
            u += s_units[kBins - 1 - p];
        }
        bins->unit_start[kBins] = u;
    }
    __syncthreads();
}

// The bin table from the counters, by one block: summed here (hist non-null), or by a device scan.
__global__ __launch_bounds__(kBlock) void bin_table_kernel(const uint32_t* __restrict__ hist, uint32_t* scan, int64_t nblk, int order,
                                                           CoreBins* __restrict__ bins) {
    if (hist != nullptr) {
        block_scan(hist, scan, kBinRows * nblk + 1);
        __threadfence_block();
        __syncthreads();
    }
    const int b = threadIdx.x;
    uint32_t n = 0, entries = 0;
    if (b < kBins) {
        n = scan[(b + 1) * nblk] - scan[b * nblk];
        entries = b >= kExactBins ? scan[(b + kVarBins + 1) * nblk] - scan[(b + kVarBins) * nblk] : n * static_cast<uint32_t>(b + 2);
    }
    bin_table(b, n, entries, order, bins);
}

// hist[r * nblk + block]: groups of bin r among the block's groups (r < kBins), entries of the listed
// bin r - kVarBins (above).  Every block writes its column; the last element is the scan's end.
__global__ __launch_bounds__(kBlock) void bin_count_kernel(const uint32_t* __restrict__ starts, const int64_t* __restrict__ counts,
                                                           int64_t nblk, int per_block, uint32_t* __restrict__ hist) {
    __shared__ unsigned long long s_bin[kBins];
    for (int b = threadIdx.x; b < kBins; b += kBlock) {
        s_bin[b] = 0ull;
    }
    __syncthreads();
    const int64_t groups = counts[1];
    const int64_t g0 = static_cast<int64_t>(blockIdx.x) * per_block;
    for (int t = 0; t < per_block; t += kBlock) {
        const int64_t g = g0 + t + threadIdx.x;
        if (g < groups) {
            const uint32_t s = starts[g];
            const uint32_t size = (starts[g + 1] & kGroupStart) - (s & kGroupStart);
            if (size >= 2u) {
                const int b = group_bin(size, (s & kGroupMixed) != 0u);
                atomicAdd(&s_bin[b], (static_cast<unsigned long long>(bin_items(b, size)) << 32) | size);
            }
        }
    }
    __syncthreads();
    for (int r = threadIdx.x; r < kBinRows; r += kBlock) {
        hist[r * nblk + blockIdx.x] = static_cast<uint32_t>(r < kBins ? s_bin[r] >> 32 : s_bin[r - kVarBins]);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        hist[kBinRows * nblk] = 0u;
    }
}

// Splits the mixed group m (group, place in mvals) by core, by one wave: each core's entries go to the group's place in
// mvals, in the order of their first entries, and take the next size / 2 of the group's list slots; an entry
// alone with its core has no partner and is dropped.  The slots of a group placed `a` entries into the
// bin are [a / 2, (a + size) / 2): disjoint, and at least floor(size / 2) of them.  The rest are empty.
template <int W, int ORDER>
__device__ void split_group(const uint32_t* __restrict__ starts, const uint64_t* __restrict__ vals, const uint64_t* __restrict__ ckeys,
                            const uint2 m, int n_bits, const CoreBins* __restrict__ bins, uint64_t* __restrict__ mvals,
                            uint2* __restrict__ glist, int lane) {
    const uint64_t below = (1ull << lane) - 1ull;
    const auto binned = [&](uint64_t v, const Cfg<W>& core) {
        const int x = static_cast<int>(v & 0xff), y = static_cast<int>((v >> 8) & 0xff);
        const uint64_t slot = ORDER == 2 ? static_cast<uint64_t>(pair_slot(x, y, n_bits)) : static_cast<uint64_t>(x);
        const int odd = ORDER == 2 ? masked_parity<W>(core, range_mask<W>(x, y)) : masked_parity<W>(core, range_mask<W>(0, x));
        return (odd ? 1ull << 63 : 0ull) | (slot << 32) | (v >> 16);
    };
    const auto equal = [](const Cfg<W>& a, const Cfg<W>& b) {
        bool same = true;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            same = same & (a.w[w] == b.w[w]);
        }
        return same;
    };
    const auto of_lane = [](const Cfg<W>& c, int l) {  // l wave-uniform
        Cfg<W> r;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(c.w[w]), l);
            const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(c.w[w] >> 32), l);
            r.w[w] = (static_cast<uint64_t>(hi) << 32) | lo;
        }
        return r;
    };
    const uint32_t s = starts[m.x] & kGroupStart;
    const uint32_t size = (starts[m.x + 1] & kGroupStart) - s;
    const uint32_t a = m.y - bins->entry_base[kSplitBin];
    uint32_t slot = bins->list_base[kSplitBin] + a / 2u;
    const uint32_t slot_end = bins->list_base[kSplitBin] + (a + size) / 2u;
    uint32_t out = m.y;
    for (uint32_t a0 = 0; a0 < size; a0 += 64) {
        const bool in_a = a0 + lane < size;
        const uint64_t va = vals[s + (in_a ? a0 + lane : 0u)];
        const Cfg<W> ca = entry_core<W, ORDER>(ckeys, va);
        // the entries of this chunk that are the first with their core
        bool first = in_a;
        for (uint32_t b0 = 0; b0 <= a0; b0 += 64) {
            const Cfg<W> cb = b0 == a0 ? ca : entry_core<W, ORDER>(ckeys, vals[s + b0 + lane]);
            const int nb = static_cast<int>(size - b0 < 64u ? size - b0 : 64u);
            for (int j = 0; j < nb; ++j) {
                const bool same = equal(of_lane(cb, j), ca);
                first = first & !(same & (b0 + static_cast<uint32_t>(j) < a0 + static_cast<uint32_t>(lane)));
            }
        }
        uint64_t firsts = __ballot(first);
        while (firsts) {
            const int l = __builtin_ctzll(firsts);
            firsts &= firsts - 1;
            const Cfg<W> core = of_lane(ca, l);
            uint32_t n = 0;
            for (uint32_t b0 = a0; b0 < size; b0 += 64) {
                const bool in_b = b0 + lane < size;
                const uint64_t vb = b0 == a0 ? va : vals[s + (in_b ? b0 + lane : 0u)];
                const bool same = in_b & equal(b0 == a0 ? ca : entry_core<W, ORDER>(ckeys, vb), core);
                const uint64_t mask = __ballot(same);
                if (same) {
                    mvals[out + n + static_cast<uint32_t>(__popcll(mask & below))] = binned(vb, core);
                }
                n += static_cast<uint32_t>(__popcll(mask));
            }
            if (n >= 2u) {
                // its tiles, apart so that no two are one unit's (a tile has at least kSplitSlots slots)
                const uint32_t apart = n / 2u / group_tiles(n);
                for (uint32_t k = lane; k < n / 2u; k += 64) {
                    const uint32_t tile = k / apart;
                    const bool here = k % apart == 0u && tile < group_tiles(n);
                    glist[slot + k] = here ? listed_tile(out, n, tile) : make_uint2(0u, 0u);
                }
                slot += n / 2u;
                out += n;
            }
        }
    }
    for (uint32_t k = slot + lane; k < slot_end; k += 64) {
        glist[k] = make_uint2(0u, 0u);
    }
}

// Copies the entries of the groups of two or more into their bins and lists the groups of the listed
// bins (first entry in mvals, size).  A block places its per_block groups, then its waves walk their
// entries with the flags telling where groups start, then split the block's mixed groups, noted in
// msplit as {group, place in mvals}.
template <int W, int ORDER>
__global__ __launch_bounds__(kBlock) void bin_scatter_kernel(const uint32_t* __restrict__ starts, const int64_t* __restrict__ counts,
                                                             const uint8_t* __restrict__ flag, const uint64_t* __restrict__ vals,
                                                             const uint64_t* __restrict__ ckeys, const uint32_t* __restrict__ scan, int64_t nblk, int per_block,
                                                             int n_bits, const CoreBins* __restrict__ bins,
                                                             uint64_t* __restrict__ mvals, uint2* __restrict__ glist,
                                                             uint2* __restrict__ msplit) {
    __shared__ unsigned long long s_rank[kBins];
    __shared__ uint32_t s_group0[kBins], s_entry0[kBins];
    __shared__ uint32_t s_move[kBinGroupsMax];  // binned position minus sorted position, kStay: not copied
    constexpr uint32_t kStay = 0x80000000u;
    const int64_t groups = counts[1];
    const int64_t g0 = static_cast<int64_t>(blockIdx.x) * per_block;
    if (g0 >= groups) {
        return;  // the whole block
    }
    for (int b = threadIdx.x; b < kBins; b += kBlock) {
        s_rank[b] = 0ull;
        s_group0[b] = scan[b * nblk + blockIdx.x] - scan[b * nblk];
        s_entry0[b] = b >= kExactBins ? scan[(b + kVarBins) * nblk + blockIdx.x] - scan[(b + kVarBins) * nblk] : 0u;
    }
    __syncthreads();
    const int here = static_cast<int>(groups - g0 < per_block ? groups - g0 : per_block);
    for (int t = threadIdx.x; t < here; t += kBlock) {
        const uint32_t s = starts[g0 + t];
        const uint32_t first = s & kGroupStart;
        const uint32_t size = (starts[g0 + t + 1] & kGroupStart) - first;
        uint32_t move = kStay;
        if (size >= 2u) {
            const int b = group_bin(size, (s & kGroupMixed) != 0u);
            const unsigned long long r = atomicAdd(&s_rank[b], (static_cast<unsigned long long>(bin_items(b, size)) << 32) | size);
            const uint32_t rank = s_group0[b] + static_cast<uint32_t>(r >> 32);
            if (b < kExactBins) {
                move = bins->entry_base[b] + rank * size - first;
            } else {
                const uint32_t at = bins->entry_base[b] + s_entry0[b] + static_cast<uint32_t>(r);
                if (b == kSplitBin) {
                    msplit[rank] = make_uint2(static_cast<uint32_t>(g0) + static_cast<uint32_t>(t), at);
                } else {
                    for (uint32_t k = 0; k < group_tiles(size); ++k) {
                        glist[bins->list_base[b] + rank + k] = listed_tile(at, size, k);
                    }
                    move = at - first;
                }
            }
        }
        s_move[t] = move;
    }
    __threadfence_block();
    __syncthreads();
    // wave w: the entries of the block's groups [w, w + 1) * per_block / 4
    const int lane = threadIdx.x & 63;
    const int per_wave = per_block / (kBlock / 64);
    const int lo = (threadIdx.x >> 6) * per_wave;
    const int hi = lo + per_wave < here ? lo + per_wave : here;
    const int64_t e0 = lo < here ? starts[g0 + lo] & kGroupStart : 0;
    const int64_t e1 = lo < here ? starts[g0 + hi] & kGroupStart : 0;
    const uint64_t upto = lane == 63 ? ~0ull : (1ull << (lane + 1)) - 1ull;
    int g = lo - 1;  // group of the entry before the 64
    constexpr int U = 4;
    for (int64_t base = e0; base < e1; base += 64 * U) {
        uint32_t f[U];
        uint64_t v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t e = base + 64 * u + lane;
            f[u] = e < e1 ? flag[e] : 0u;
            v[u] = e < e1 ? vals[e] : 0ull;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t e = base + 64 * u + lane;
            const uint64_t heads = __ballot((f[u] & kFlagHead) != 0u);
            if (e < e1) {
                const uint32_t move = s_move[g + __popcll(heads & upto)];
                if (move != kStay) {
                    const int x = static_cast<int>(v[u] & 0xff);
                    const uint64_t slot =
                        ORDER == 2 ? static_cast<uint64_t>(pair_slot(x, static_cast<int>((v[u] >> 8) & 0xff), n_bits)) : static_cast<uint64_t>(x);
                    const uint64_t sign = (f[u] & kFlagSign) != 0u ? 1ull << 63 : 0ull;
                    mvals[static_cast<uint32_t>(e) + move] = sign | (slot << 32) | (v[u] >> 16);
                }
            }
            g += __popcll(heads);
        }
    }
    const uint32_t n_mixed = static_cast<uint32_t>(s_rank[kSplitBin] >> 32);
    for (uint32_t i = threadIdx.x >> 6; i < n_mixed; i += kBlock / 64) {
        split_group<W, ORDER>(starts, vals, ckeys, msplit[s_group0[kSplitBin] + i], n_bits, bins, mvals, glist, lane);
    }
}

// A small set's whole core index in one block: emission, sort, flags, starts and bins, everything
// between in LDS.  The general build is some twenty launches of a few microseconds each, whatever the
// size.  The limit is the LDS: 18 bytes an entry and the sort's power of two.  Entries sort by (key,
// emission index k * n + row), the order the general build's stable sort gives.
constexpr int kSmallCores = 8192;
// Up to this many entries one wave takes all units, in order: the sums of so small a set then come out
// the same in every call (whole units spread over waves add to a row in the order they finish), for
// about the time that the kernel's launch and the call around it take anyway.  Larger ones are worth
// more than the last bit: one wave over the 52 groups that three electrons in 52 sites make takes 235 ms,
// all waves 0.4.
constexpr int kTinyCores = 512;
constexpr int kSmallThreads = 1024;

struct SmallLds {
    uint64_t entry[kSmallCores];    // key << 32 | emission index
    uint16_t sites[kSmallCores];    // by emission index: y << 8 | x
    uint16_t group[kSmallCores];    // by sorted position
    uint16_t start[kSmallCores + 1];
    uint16_t move[kSmallCores];     // by group: place in mvals, kSmallStay: not copied
    uint8_t flag[kSmallCores];
    uint8_t mixed[kSmallCores];     // by group
    uint32_t wave_heads[kSmallThreads / 64];
    unsigned long long rank[kBins];
    uint32_t used, over, n_mixed;
};
static_assert(sizeof(SmallLds) + 3 * kBins * sizeof(uint32_t) <= 160 * 1024, "LDS, with bin_table's");
constexpr uint32_t kSmallStay = 0xffffu;

template <int W, int ORDER>
__global__ __launch_bounds__(kSmallThreads) void cores_small_kernel(const uint64_t* __restrict__ ckeys, const uint64_t* __restrict__ cols,
                                                                    int n, int n_bits, int per_config, uint32_t* __restrict__ keys,
                                                                    uint64_t* __restrict__ vals, uint32_t* __restrict__ starts,
                                                                    int64_t* __restrict__ counts, CoreBins* __restrict__ bins,
                                                                    uint64_t* __restrict__ mvals, uint2* __restrict__ glist,
                                                                    uint2* __restrict__ msplit) {
    extern __shared__ uint64_t smem[];
    SmallLds& L = *reinterpret_cast<SmallLds*>(smem);
    const int tid = threadIdx.x;
    const int cap = n * per_config;
    int p2 = kSmallThreads;
    while (p2 < cap) {
        p2 <<= 1;
    }
    if (tid == 0) {
        L.used = 0u;
        L.over = 0u;
        L.n_mixed = 0u;
    }
    for (int b = tid; b < kBins; b += kSmallThreads) {
        L.rank[b] = 0ull;
    }
    for (int e = cap + tid; e < p2; e += kSmallThreads) {
        L.entry[e] = ~0ull;
    }
    __syncthreads();
    for (int i = tid; i < n; i += kSmallThreads) {
        int k = 0;
        emit_cores<W, ORDER>(load_key<W>(ckeys, i), cols, [&](uint32_t key, uint32_t sites) {
            if (k < per_config) {
                L.entry[k * n + i] = (static_cast<uint64_t>(key) << 32) | static_cast<uint32_t>(k * n + i);
                L.sites[k * n + i] = static_cast<uint16_t>(sites);
            }
            ++k;
        });
        if (k > per_config) {
            atomicAdd(&L.over, 1u);
        }
        atomicAdd(&L.used, static_cast<uint32_t>(k < per_config ? k : per_config));
        for (; k < per_config; ++k) {
            L.entry[k * n + i] = ~0ull;
        }
    }
    // bitonic sort of the p2 entries
    for (int size = 2; size <= p2; size <<= 1) {
        for (int step = size >> 1; step > 0; step >>= 1) {
            __syncthreads();
            for (int t = tid; t < p2 / 2; t += kSmallThreads) {
                const int a = 2 * t - (t & (step - 1));
                const uint64_t x = L.entry[a], y = L.entry[a + step];
                if ((x > y) == ((a & size) == 0)) {
                    L.entry[a] = y;
                    L.entry[a + step] = x;
                }
            }
        }
    }
    __syncthreads();
    const int used = static_cast<int>(L.used);
    const int per = (used + kSmallThreads - 1) / kSmallThreads;  // consecutive entries of a thread
    const int lo = tid * per < used ? tid * per : used;
    const int hi = lo + per < used ? lo + per : used;
    const auto value = [&](int e) {
        const uint32_t at = static_cast<uint32_t>(L.entry[e]);
        return (static_cast<uint64_t>(at % static_cast<uint32_t>(n)) << 16) | L.sites[at];
    };
    uint32_t heads = 0;
    Cfg<W> before{};
    for (int e = lo; e < hi; ++e) {
        const uint32_t key = static_cast<uint32_t>(L.entry[e] >> 32);
        const bool with_prev = e > 0 && static_cast<uint32_t>(L.entry[e - 1] >> 32) == key;
        const bool with_next = e + 1 < used && static_cast<uint32_t>(L.entry[e + 1] >> 32) == key;
        const uint64_t v = value(e);
        uint32_t f = with_prev ? 0u : kFlagHead;
        if (with_prev || with_next) {
            const Cfg<W> core = entry_core<W, ORDER>(ckeys, v);
            if (with_prev && e == lo) {
                before = entry_core<W, ORDER>(ckeys, value(e - 1));
            }
            bool same = true;
#pragma unroll
            for (int w = 0; w < W; ++w) {
                same = same && core.w[w] == before.w[w];
            }
            f |= with_prev && !same ? kFlagBreak : 0u;
            const int a = ORDER == 2 ? static_cast<int>(v & 0xff) : 0;
            const int b = static_cast<int>((ORDER == 2 ? v >> 8 : v) & 0xff);
            f |= masked_parity<W>(core, range_mask<W>(a, b)) != 0 ? kFlagSign : 0u;
            before = core;
        }
        heads += with_prev ? 0u : 1u;
        L.flag[e] = static_cast<uint8_t>(f);
        keys[e] = key;
        vals[e] = v;
    }
    for (int e = used + tid; e < cap; e += kSmallThreads) {
        keys[e] = kKeySentinel;
        vals[e] = 0ull;
    }
    // the heads before each thread's entries
    uint32_t incl = heads;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(incl, d);
        incl += (tid & 63) >= d ? o : 0u;
    }
    if ((tid & 63) == 63) {
        L.wave_heads[tid >> 6] = incl;
    }
    __syncthreads();
    uint32_t g = incl - heads, groups = 0;
    for (int w = 0; w < kSmallThreads / 64; ++w) {
        g += w < (tid >> 6) ? L.wave_heads[w] : 0u;
        groups += L.wave_heads[w];
    }
    for (int e = lo; e < hi; ++e) {
        if ((L.flag[e] & kFlagHead) != 0u) {
            L.start[g] = static_cast<uint16_t>(e);
            L.mixed[g] = 0;
            ++g;
        }
        L.group[e] = static_cast<uint16_t>(g - 1u);
    }
    if (tid == 0) {
        L.start[groups] = static_cast<uint16_t>(used);
        counts[0] = used;
        counts[1] = groups;
        counts[2] = L.over;
        counts[3] = 0;
    }
    __syncthreads();
    for (int e = lo; e < hi; ++e) {
        if ((L.flag[e] & kFlagBreak) != 0u) {
            L.mixed[L.group[e]] = 1;
        }
    }
    __syncthreads();
    const int n_groups = static_cast<int>(groups);
    for (int q = tid; q <= n_groups; q += kSmallThreads) {
        const uint32_t first = L.start[q];
        const bool mixed = q < n_groups && L.mixed[q] != 0;
        starts[q] = first | (mixed ? kGroupMixed : 0u);
        const uint32_t size = q < n_groups ? L.start[q + 1] - first : 0u;
        if (size >= 2u) {
            const int b = group_bin(size, mixed);
            atomicAdd(&L.rank[b], (static_cast<unsigned long long>(bin_items(b, size)) << 32) | size);
        }
    }
    __syncthreads();
    const unsigned long long mine = tid < kBins ? L.rank[tid] : 0ull;
    bin_table(tid, static_cast<uint32_t>(mine >> 32), static_cast<uint32_t>(mine), ORDER, bins);
    if (tid < kBins) {
        L.rank[tid] = 0ull;
    }
    __threadfence_block();
    __syncthreads();
    const int placers = cap <= kTinyCores ? 64 : kSmallThreads;  // one wave: always the same places
    for (int q = tid; tid < placers && q < n_groups; q += placers) {
        const uint32_t first = L.start[q];
        const uint32_t size = L.start[q + 1] - first;
        uint32_t move = kSmallStay;
        if (size >= 2u) {
            const int b = group_bin(size, L.mixed[q] != 0);
            const unsigned long long r = atomicAdd(&L.rank[b], (static_cast<unsigned long long>(bin_items(b, size)) << 32) | size);
            const uint32_t rank = static_cast<uint32_t>(r >> 32);
            move = bins->entry_base[b] + static_cast<uint32_t>(r);
            if (b == kSplitBin) {
                msplit[rank] = make_uint2(static_cast<uint32_t>(q), move);
                atomicAdd(&L.n_mixed, 1u);
                move = kSmallStay;
            } else if (b >= kExactBins) {
                for (uint32_t k = 0; k < group_tiles(size); ++k) {
                    glist[bins->list_base[b] + rank + k] = listed_tile(move, size, k);
                }
            }
        }
        L.move[q] = static_cast<uint16_t>(move);
    }
    __threadfence_block();
    __syncthreads();
    for (int e = lo; e < hi; ++e) {
        const uint32_t q = L.group[e];
        if (L.move[q] != kSmallStay) {
            const uint64_t v = value(e);
            const int x = static_cast<int>(v & 0xff);
            const uint64_t slot =
                ORDER == 2 ? static_cast<uint64_t>(pair_slot(x, static_cast<int>((v >> 8) & 0xff), n_bits)) : static_cast<uint64_t>(x);
            mvals[L.move[q] + static_cast<uint32_t>(e) - L.start[q]] = ((L.flag[e] & kFlagSign) != 0u ? 1ull << 63 : 0ull) | (slot << 32) | (v >> 16);
        }
    }
    for (uint32_t i = tid >> 6; i < L.n_mixed; i += kSmallThreads / 64) {
        split_group<W, ORDER>(starts, vals, ckeys, msplit[i], n_bits, bins, mvals, glist, tid & 63);
    }
}

// Bits of the sub field of a packed core value (order 2: pair slots, order 1: sites) and of the
// row; the 32-bit value applies when both fit.
inline int bits_for(int64_t range) {
    int b = 0;
    while ((int64_t{1} << b) < range) {
        ++b;
    }
    return b;
}
inline int core_sub_bits(int n_bits, int order) {
    return bits_for(order == 2 ? static_cast<int64_t>(n_bits) * (n_bits - 1) / 2 : n_bits);
}
inline bool core_packed(int64_t n, int n_bits, int order) { return bits_for(n) + core_sub_bits(n_bits, order) <= kPackedBits; }

int cores_layout(Carver& cv, int n_qubytes, int64_t n, int max_occupied, int order, qmb_cores* out, void** scratch,
                 size_t* scratch_bytes) {
    QMB_TRY(check_qubytes(n_qubytes));
    if (n < 0) {
        return set_error(QMB_ERR_ARGUMENT, "n must be >= 0");
    }
    if (order != 1 && order != 2) {
        return set_error(QMB_ERR_ARGUMENT, "order must be 1 or 2, got %d", order);
    }
    if (max_occupied < 0 || max_occupied > 8 * n_qubytes) {
        return set_error(QMB_ERR_ARGUMENT, "max_occupied must be in [0, %d], got %d", 8 * n_qubytes, max_occupied);
    }
    qmb_cores c{};
    c.n_qubytes = n_qubytes;
    c.n_words = n_words_of(n_qubytes);
    c.max_occupied = max_occupied;
    c.order = order;
    c.per_config = order == 2 ? max_occupied * (max_occupied - 1) / 2 : max_occupied;
    c.n = n;
    c.capacity = n * c.per_config;
    if (c.capacity >= (1ll << 31)) {
        return set_error(QMB_ERR_UNSUPPORTED, "core index of %lld entries exceeds 2^31 - 1", static_cast<long long>(c.capacity));
    }
    const size_t cap = static_cast<size_t>(c.capacity > 0 ? c.capacity : 1);
    c.buffer = cv.base;
    c.counts = cv.take<int64_t>(4);
    c.keys = cv.take<uint32_t>(cap);
    c.vals = cv.take<uint64_t>(cap);
    c.starts = cv.take<uint32_t>(cap + 1);
    c.bins = cv.take<CoreBins>(1);
    size_t tmp = 0;
    {
        uint64_t* v = nullptr;
        uint32_t* u = nullptr;
        if (rocprim::radix_sort_pairs(nullptr, tmp, u, u, v, v, static_cast<unsigned>(cap), 0, kKeyBits) != hipSuccess) {
            return set_error(QMB_ERR_HIP, "rocprim radix_sort_pairs size query failed");
        }
        size_t packed = 0;
        if (rocprim::radix_sort_keys(nullptr, packed, v, v, static_cast<unsigned>(cap), kPackedBits, kPackedBits + kKeyBits) !=
            hipSuccess) {
            return set_error(QMB_ERR_HIP, "rocprim radix_sort_keys size query failed");
        }
        tmp = tmp > packed ? tmp : packed;
        size_t scan = 0;
        if (rocprim::exclusive_scan(nullptr, scan, u, u, 0u, cap, rocprim::plus<uint32_t>()) != hipSuccess) {
            return set_error(QMB_ERR_HIP, "rocprim exclusive_scan size query failed");
        }
        tmp = tmp > scan ? tmp : scan;
        const size_t bin_counters = static_cast<size_t>(kBinRows * bin_blocks(static_cast<int64_t>(cap)) + 1);
        if (rocprim::exclusive_scan(nullptr, scan, u, u, 0u, bin_counters, rocprim::plus<uint32_t>()) != hipSuccess) {
            return set_error(QMB_ERR_HIP, "rocprim exclusive_scan size query failed");
        }
        tmp = tmp > scan ? tmp : scan;
    }
    const size_t s0 = cv.off;
    const size_t bin_bytes = 2 * static_cast<size_t>(kBinRows * bin_blocks(static_cast<int64_t>(cap)) + 1) * sizeof(uint32_t) + 512;
    const size_t inv_bytes = static_cast<size_t>(8 * n_qubytes) * (8 * n_qubytes) / 2 * sizeof(uint32_t) + 256;
    const size_t chunk_bytes = 2 * static_cast<size_t>(flag_chunks(static_cast<int64_t>(cap))) * sizeof(uint32_t) + 512;
    void* s = cv.take_bytes(2 * cap * sizeof(uint64_t) + cap + chunk_bytes + bin_bytes + inv_bytes + tmp + 4096);
    if (scratch) {
        *scratch = s;
    }
    if (scratch_bytes) {
        *scratch_bytes = cv.off - s0;
    }
    c.bytes = cv.off;
    if (out) {
        *out = c;
    }
    return QMB_OK;
}

// ------------------------------------------------------------------------------ group kernel --
struct PairParams {
    const double2* coef;    // merged pair-excitation coefficients with their own sites' sign, [pair_slot][pair_slot]
    const double* coef_re;  // their real parts when every coefficient is real, else null
    int64_t n_pairs;
    int particle_cut;
    const uint64_t* mvals;  // binned entries
    const uint2* glist;
    const CoreBins* bins;
    const int64_t* counts;
    const double2* in;
    double2* out;
    const double2* in2;  // second input/output of a two-vector pass (NV = 2), else null
    double2* out2;
    const int64_t* table_counts;  // qmb_pairs.counts
    int dense;                    // the bins above 64 entries are pair_dense_kernel's
};

// The lanes' entries as the rows of a group read them, in this wave's LDS: the amplitude with the
// entry's sign and the entry's part of the coefficient index (order 1: its site).
struct GroupStage {
    double2 g[128];
    uint32_t part[128];
};
struct GroupStage2 {
    double2 g[128];
    double2 g2[128];
    uint32_t part[128];
};
template <int NV>
struct StageOf {
    using type = GroupStage;
};
template <>
struct StageOf<2> {
    using type = GroupStage2;
};
template <int NV>
using Stage = typename StageOf<NV>::type;
constexpr int kWavesPerBlock = kBlock / 64;

__device__ __forceinline__ double2 signed_by(const double2& v, uint32_t flip) {
    const int f = static_cast<int>(flip << 31);
    return make_double2(__hiloint2double(__double2hiint(v.x) ^ f, __double2loint(v.x)), __hiloint2double(__double2hiint(v.y) ^ f, __double2loint(v.y)));
}

// A binned entry: row | slot << 32 | sign << 63.
struct Entry {
    uint32_t row;
    uint32_t slot;
    uint32_t sign;
};
__device__ __forceinline__ Entry binned_entry(uint64_t v, bool fermi) {
    return Entry{static_cast<uint32_t>(v), static_cast<uint32_t>(v >> 32) & 0xffffu, fermi ? static_cast<uint32_t>(v >> 63) : 0u};
}

template <int NV, typename P>
__device__ __forceinline__ void stage_lane(const P& p, Stage<NV>& st, int at, bool act, const Entry& e, uint32_t part) {
    double2 g = make_double2(0.0, 0.0), g2 = g;
    if (act) {
        g = signed_by(p.in[e.row], e.sign);
        if constexpr (NV == 2) {
            g2 = signed_by(p.in2[e.row], e.sign);
        }
    }
    st.g[at] = g;
    if constexpr (NV == 2) {
        st.g2[at] = g2;
    }
    st.part[at] = part;
}

// out[row] += sign * (re, im) of the wave's active lanes (every lane calls it).  The sums go through the
// lanes' own stage slots [at0, at0 + 64), so that neighbouring lanes hold the two components of one
// row: their FP64 atomics leave as one 16-byte request instead of two.  The small pair groups are
// bound by these requests: sizes 3 and 4 of 1M molecular configs took 0.96 ms with an instruction per
// component, 0.51 ms so, and 0.31 ms without any atomics.
template <int NV, typename P>
__device__ __forceinline__ void add_rows(const P& p, Stage<NV>& st, int at0, int lane, bool act, const Entry& e, const double (&re)[NV],
                                         const double (&im)[NV]) {
    st.part[at0 + lane] = act ? e.row : ~0u;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        st.g[at0 + lane] = signed_by(make_double2(re[v], im[v]), e.sign);
        __builtin_amdgcn_wave_barrier();
        double* out = reinterpret_cast<double*>(v == 0 ? p.out : p.out2);
        const double* sums = reinterpret_cast<const double*>(st.g + at0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const double x = sums[64 * h + lane];
            const uint32_t row = st.part[at0 + 32 * h + (lane >> 1)];
            if (row != ~0u && x != 0.0) {
                unsafeAtomicAdd(&out[2 * static_cast<int64_t>(row) + (lane & 1)], x);
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

template <bool REAL>
__device__ __forceinline__ double2 pair_coef(const PairParams& p, uint32_t idx) {
    return REAL ? make_double2(p.coef_re[idx], 0.0) : p.coef[idx];
}

// acc += x g (!ADJ) or conj(x) g (ADJ); a real table skips the imaginary part of x.
template <bool ADJ, bool REAL>
__device__ __forceinline__ void pair_madd(const double2& x, const double2& g, double& re, double& im) {
    if (REAL) {
        re = __fma_rn(x.x, g.x, re);
        im = __fma_rn(x.x, g.y, im);
    } else if (ADJ) {
        re = __fma_rn(x.y, g.y, __fma_rn(x.x, g.x, re));
        im = __fma_rn(-x.y, g.x, __fma_rn(x.x, g.y, im));
    } else {
        re = __fma_rn(-x.y, g.y, __fma_rn(x.x, g.x, re));
        im = __fma_rn(x.y, g.x, __fma_rn(x.x, g.y, im));
    }
}

// With the sign split into one factor per entry and a part the table holds (pair_own_parity), a group
// of entries (row_e, slot_e, sign_e) contributes
//   ADJ:  out[row_a] += sign_a sum_b sign_b conj(T[slot_a][slot_b]) in[row_b]
//   !ADJ: out[row_a] += sign_a sum_b sign_b T[slot_b][slot_a] in[row_b]
// T being zero where the two pairs share a site (no pair excitation has fewer than four sites), which
// includes a row with itself.  Per (row, entry) that is an LDS read, one gather and the multiply-adds.

// Groups of G = 2..8 entries, lane = row, PU passes of 64 / G groups side by side.  Each row meets the
// other G - 1 entries in turn (its own left out), all gathers of the lane in flight at once.  A zero
// coefficient adds nothing, so a non-finite amplitude reaches only the rows it is connected to.
template <bool ADJ, bool REAL, int NV, int G, int PU>
__device__ __forceinline__ void pair_small(const PairParams& p, uint32_t e0, uint32_t e_end, int passes, int lane, Stage<NV>& st) {
    constexpr int L = 64 / G * G;
    const bool fermi = p.particle_cut == 1;
    const int ri = lane % G;
    const int lead = lane - ri;
    for (int q0 = 0; q0 < passes; q0 += PU) {
        Entry e[PU];
        bool act[PU];
        uint32_t mine[PU];
        if (e0 + static_cast<uint32_t>(q0 * L) >= e_end) {
            return;  // the whole wave
        }
#pragma unroll
        for (int q = 0; q < PU; ++q) {
            const uint32_t at = e0 + static_cast<uint32_t>((q0 + q) * L + lane);
            act[q] = lane < L && at < e_end;
            e[q] = binned_entry(act[q] ? p.mvals[at] : 0ull, fermi);
        }
#pragma unroll
        for (int q = 0; q < PU; ++q) {
            const uint32_t wide = e[q].slot * static_cast<uint32_t>(p.n_pairs);
            mine[q] = ADJ ? wide : e[q].slot;
            stage_lane<NV>(p, st, 64 * q + lane, act[q], e[q], ADJ ? e[q].slot : wide);
        }
        __builtin_amdgcn_wave_barrier();
        double2 x[PU][G - 1];
        int pl[G - 1];
#pragma unroll
        for (int u = 1; u < G; ++u) {
            const int r = ri + u;
            pl[u - 1] = (lead + (r >= G ? r - G : r)) & 63;
        }
#pragma unroll
        for (int q = 0; q < PU; ++q) {
#pragma unroll
            for (int u = 0; u < G - 1; ++u) {
                x[q][u] = make_double2(0.0, 0.0);
                if (act[q]) {
                    x[q][u] = pair_coef<REAL>(p, st.part[64 * q + pl[u]] + mine[q]);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < PU; ++q) {
            double re[NV] = {}, im[NV] = {};
#pragma unroll
            for (int u = 0; u < G - 1; ++u) {
                if (x[q][u].x != 0.0 || (!REAL && x[q][u].y != 0.0)) {
                    pair_madd<ADJ, REAL>(x[q][u], st.g[64 * q + pl[u]], re[0], im[0]);
                    if constexpr (NV == 2) {
                        pair_madd<ADJ, REAL>(x[q][u], st.g2[64 * q + pl[u]], re[1], im[1]);
                    }
                }
            }
            add_rows<NV>(p, st, 64 * q, lane, act[q], e[q], re, im);
        }
    }
}

// Steps b of a walk over `nb` staged entries from slot `lead`, each lane's row against the same entry
// of its group: the lanes of a group read one table row (!ADJ), their columns ascending.  B gathers
// in flight.  Zero coefficients are multiplied in (a non-finite amplitude reaches the whole group).
template <bool ADJ, bool REAL, int NV, int B>
__device__ __forceinline__ void pair_walk(const PairParams& p, const Stage<NV>& st, int lead, int nb, uint32_t mine, double (&re)[NV],
                                          double (&im)[NV]) {
    for (int u = 0; u < nb; u += B) {
        double2 x[B];
#pragma unroll
        for (int k = 0; k < B; ++k) {
            x[k] = make_double2(0.0, 0.0);
            if (u + k < nb) {  // wave-uniform
                x[k] = pair_coef<REAL>(p, st.part[lead + u + k] + mine);
            }
        }
#pragma unroll
        for (int k = 0; k < B; ++k) {
            if (u + k < nb) {
                pair_madd<ADJ, REAL>(x[k], st.g[lead + u + k], re[0], im[0]);
                if constexpr (NV == 2) {
                    pair_madd<ADJ, REAL>(x[k], st.g2[lead + u + k], re[1], im[1]);
                }
            }
        }
    }
}

// Groups of g = 9..32 entries, lane = row, 64 / g groups to a pass.
template <bool ADJ, bool REAL, int NV, int B>
__device__ __forceinline__ void pair_rows(const PairParams& p, int g, uint32_t e0, uint32_t e_end, int lane, Stage<NV>& st) {
    const bool fermi = p.particle_cut == 1;
    const int lanes = 64 / g * g;
    const uint32_t at = e0 + static_cast<uint32_t>(lane);
    const bool act = lane < lanes && at < e_end;
    const int lead = act ? lane / g * g : 0;
    const Entry e = binned_entry(act ? p.mvals[at] : 0ull, fermi);
    const uint32_t wide = e.slot * static_cast<uint32_t>(p.n_pairs);
    stage_lane<NV>(p, st, lane, act, e, ADJ ? e.slot : wide);
    __builtin_amdgcn_wave_barrier();
    double re[NV] = {}, im[NV] = {};
    pair_walk<ADJ, REAL, NV, B>(p, st, lead, g, ADJ ? wide : e.slot, re, im);
    add_rows<NV>(p, st, 0, lane, act, e, re, im);
}

// Rows [first, last) of one group of any size from mvals[s]: 64 rows at a time against its entries, 64
// staged at a time.
template <bool ADJ, bool REAL, int NV, int B>
__device__ __forceinline__ void pair_big(const PairParams& p, uint32_t s, uint32_t size, uint32_t first, uint32_t last, int lane, Stage<NV>& st) {
    const bool fermi = p.particle_cut == 1;
    const auto wide = [&](const Entry& e) { return e.slot * static_cast<uint32_t>(p.n_pairs); };
    for (uint32_t a0 = first; a0 < last; a0 += 64) {
        const bool act = a0 + lane < size;
        const Entry e = binned_entry(act ? p.mvals[s + a0 + lane] : 0ull, fermi);
        const uint32_t mine = ADJ ? wide(e) : e.slot;
        double re[NV] = {}, im[NV] = {};
        for (uint32_t b0 = 0; b0 < size; b0 += 64) {
            const bool in = b0 + lane < size;
            const Entry b = b0 == a0 ? e : binned_entry(in ? p.mvals[s + b0 + lane] : 0ull, fermi);
            stage_lane<NV>(p, st, lane, in, b, ADJ ? b.slot : wide(b));
            __builtin_amdgcn_wave_barrier();
            pair_walk<ADJ, REAL, NV, B>(p, st, 0, static_cast<int>(size - b0 < 64u ? size - b0 : 64u), mine, re, im);
            __builtin_amdgcn_wave_barrier();
        }
        add_rows<NV>(p, st, 0, lane, act, e, re, im);
    }
}

// The bin and the unit within it of unit u (every lane calls it, u wave-uniform): the last position
// whose first unit is <= u.
__device__ __forceinline__ int unit_bin(const CoreBins* bins, uint32_t u, int lane, uint32_t* local) {
    const uint32_t first = bins->unit_start[lane < kBins ? lane : kBins];
    const uint64_t upto = __ballot(lane < kBins && first <= u);
    const int pos = 63 - __builtin_clzll(upto);
    *local = u - static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(first), pos));
    return kBins - 1 - pos;
}

// The rows of a listed unit: one list element of a bin above 32 entries, or kSplitSlots of the split
// bin, most of them empty.  f(first entry, size, first row, end of the rows) runs for each, wave-uniform.
template <typename P, typename F>
__device__ __forceinline__ void for_listed(const P& p, int bin, uint32_t local, int lane, F&& f) {
    const auto tile = [&](uint32_t s, uint32_t y) {
        const bool whole = (y & kWholeGroup) != 0u;
        const uint32_t size = whole ? y & ~kWholeGroup : y & kTiledMax;
        f(s, size, whole ? 0u : (y >> 16) * 64u, whole ? size : (y >> 16) * 64u + 1u);
    };
    if (bin != kSplitBin) {
        const uint2 group = p.glist[p.bins->list_base[bin] + local];
        tile(group.x, group.y);
        return;
    }
    const uint32_t slot = local * kSplitSlots + static_cast<uint32_t>(lane);
    const bool in = lane < static_cast<int>(kSplitSlots) && slot < p.bins->groups[kSplitBin];
    const uint2 mine = in ? p.glist[p.bins->list_base[kSplitBin] + slot] : make_uint2(0u, 0u);
    uint64_t full = __ballot(mine.y != 0u);
    while (full) {
        const int l = __builtin_ctzll(full);
        full &= full - 1;
        tile(__builtin_amdgcn_readlane(mine.x, l), __builtin_amdgcn_readlane(mine.y, l));
    }
}

// Coefficient gathers in flight per lane of the larger groups.
constexpr int kPairBatch = 8;

// One work unit of the pair bins.
template <bool ADJ, bool REAL, int NV, int B>
__device__ __forceinline__ void pair_unit(const PairParams& p, uint32_t u, int lane, Stage<NV>& st) {
    uint32_t local;
    const int bin = unit_bin(p.bins, u, lane, &local);
    if (bin < kExactBins) {
        const int g = bin + 2;
        const int passes = unit_passes(g, 2);
        const uint32_t base = p.bins->entry_base[bin];
        const uint32_t e0 = base + local * static_cast<uint32_t>(64 / g * g * passes);
        const uint32_t e_end = base + p.bins->groups[bin] * static_cast<uint32_t>(g);
        switch (g) {
            case 2: pair_small<ADJ, REAL, NV, 2, 2>(p, e0, e_end, passes, lane, st); break;
            case 3: pair_small<ADJ, REAL, NV, 3, 2>(p, e0, e_end, passes, lane, st); break;
            case 4: pair_small<ADJ, REAL, NV, 4, 2>(p, e0, e_end, passes, lane, st); break;
            case 5: pair_small<ADJ, REAL, NV, 5, 1>(p, e0, e_end, passes, lane, st); break;
            case 6: pair_small<ADJ, REAL, NV, 6, 1>(p, e0, e_end, passes, lane, st); break;
            case 7: pair_small<ADJ, REAL, NV, 7, 1>(p, e0, e_end, passes, lane, st); break;
            case 8: pair_small<ADJ, REAL, NV, 8, 1>(p, e0, e_end, passes, lane, st); break;
            default: pair_rows<ADJ, REAL, NV, B>(p, g, e0, e_end, lane, st); break;
        }
        return;
    }
    for_listed(p, bin, local, lane, [&](uint32_t s, uint32_t size, uint32_t first, uint32_t last) {
        pair_big<ADJ, REAL, NV, B>(p, s, size, first, last, lane, st);
    });
}

__device__ __forceinline__ void mark_overflow(double2* out) {
    // a row had more occupied sites than the core index was built for
    out[0] = make_double2(__longlong_as_double(0x7ff8000000000000ll), __longlong_as_double(0x7ff8000000000000ll));
}

constexpr int kDenseFirst = kExactBins + 2;  // groups above 64 entries, see pair_dense_kernel
constexpr int kDenseGroups = 8;
constexpr uint32_t kDensePanels = 128;

// List elements of a group of the bin, at least.
__device__ __forceinline__ uint32_t least_tiles(int bin) {
    const int k = bin - kExactBins;
    return k < 2 ? 1u : (k < 4 ? 2u : static_cast<uint32_t>(k) - 1u);
}

// The list elements of a panel of eight groups, and the bin's panels.
__device__ __forceinline__ uint32_t panel_window(int bin) { return kDenseGroups * least_tiles(bin); }
__device__ __forceinline__ uint32_t bin_panels(const CoreBins* bins, int bin) { return (bins->groups[bin] + panel_window(bin) - 1u) / panel_window(bin); }

// Whether the groups above 64 entries go to pair_dense_kernel: a panel takes one CU 20 to 50 us, so that
// a few panels end as a tail (12,000 rows of 52 spin orbitals: 48 us, 100 with their 17 panels; 100,000 rows of
// 40 take 267 us, 286 with 171 panels, which an index of kDenseMin entries no longer notices).
__device__ __forceinline__ bool dense_bins(const CoreBins* bins) {
    uint32_t panels = 0;
#pragma unroll
    for (int bin = kDenseFirst; bin < kSplitBin; ++bin) {
        panels += bin_panels(bins, bin);
    }
    return panels >= kDensePanels;
}

// Persistent waves over the units of the bins.  Every wave leaves when the units are done.
template <bool ADJ, bool REAL, int NV>
__global__ __launch_bounds__(kBlock) void pair_kernel(PairParams p) {
    __shared__ Stage<NV> stages[kWavesPerBlock];
    const int lane = threadIdx.x & 63;
    const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>((blockIdx.x * blockDim.x + threadIdx.x) >> 6)));
    const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
    if (p.counts[2] != 0) {
        if (wave == 0 && lane == 0) {
            mark_overflow(p.out);
        }
        return;
    }
    // the largest bins stand right after the split bin
    const uint32_t skip_at = p.bins->unit_start[1];
    const uint32_t skip = p.dense && dense_bins(p.bins) ? p.bins->unit_start[1 + kSplitBin - kDenseFirst] - skip_at : 0u;
    const uint32_t units = p.bins->unit_start[kBins] - skip;
    for (uint32_t i = wave; i < units; i += nwaves) {
        const uint32_t u = i < skip_at ? i : i + skip;
        pair_unit<ADJ, REAL, NV, NV == 1 ? kPairBatch : kPairBatch / 2>(p, u, lane, stages[threadIdx.x >> 6]);
    }
}

// The groups above 64 entries of a real table, eight at a time as a dense product on the matrix unit.
// A panel is eight groups that follow each other in a bin; its slots are the U pair slots that any of
// them has, and with S the table at these slots and B the [U][16] amplitudes (eight groups, real and imaginary
// part, zero where a group has no such entry) the panel's contributions are S^T B (ADJ: S B).  The
// group kernel gathers one coefficient per pair of entries, a cache line each, and that bounds it;
// here a coefficient is read once for eight groups, in rows.  1M rows of 52 spin orbitals: forward 4.68 ->
// 4.32 ms, adjoint (whose gathers fall in as many rows as lanes) 7.87 -> 5.92; 200,000 rows of 76:
// 3.94 -> 3.27 and 5.44 -> 4.87 (most of its panels are walked; the waves of a work-group then share the rows
// of the table).  The time of a dense panel is half products, half the steps around them.
// A panel is dense where its pairs of entries pay for the products of the slots that a group lacks:
// from kDenseGain pairs per matrix instruction (16 x 16 x 4, eight groups' 512 pairs at most; a local
// energy step of 200,000 sampled rows of 76 spin orbitals: 9.1 ms from 20, 9.2 from 32, 11.1 without panels), U within
// the LDS, and a finite table (a zero amplitude times infinity would reach other groups' rows).  The
// other panels are walked as in pair_kernel.
// Matrix operands: lane l holds S of row slot l % 16 and column slot l / 16 of four, and B of that column slot
// at l % 16; results v = 0..3 are row slot 4 v + l / 16 at l % 16, so that neighbouring lanes add the
// two components of one output row.
constexpr int kDenseThreads = 1024;
constexpr int kDenseWaves = kDenseThreads / 64;
constexpr int kDenseStep = 32;        // column slots whose coefficients are in flight
constexpr int kDenseGain = 20;
constexpr int kDenseSlots = 8192;     // pair slots of 16 bytes of sites: 8128
constexpr int kDenseWindow = 64;      // list elements of a panel, at most
constexpr int kDenseUnion = 960;      // U that fits the LDS
// Entries of the index from which panels are made, forward with / without and adjoint with / without, us:
//   9.1M (52 spin orbitals, 100,000 rows)  317 / 261     432 / 408
//  18.2M (52, 200,000)                     583 / 562     823 / 903
//  23.0M (60, 150,000)                     696 / 625     980 / 976
//  36.4M (52, 400,000)                    1297 / 1347   1807 / 2192
//  61.2M (60, 400,000)                    1717 / 1900   2265 / 2491
constexpr int64_t kDenseMin = 1 << 25;

typedef double f64x4 __attribute__((ext_vector_type(4)));

struct DenseLds {
    double b[kDenseUnion * 16];
    uint32_t rows[kDenseUnion * kDenseGroups];  // row | sign << 31 of a slot in a group, ~0: none
    uint32_t slots[kDenseUnion];
    uint64_t bits[kDenseSlots / 64];
    uint32_t before[kDenseSlots / 64];  // used slots before the word
    uint2 groups[kDenseWindow];         // first entry, size
    uint32_t n_groups;
    uint32_t used;
};

template <bool ADJ, int NV>
__global__ __launch_bounds__(kDenseThreads) void pair_dense_kernel(PairParams p) {
    extern __shared__ uint64_t smem[];
    static_assert(kDenseUnion % kDenseStep == 0 && sizeof(DenseLds) <= 160 * 1024 && sizeof(Stage<NV>) * kDenseWaves <= sizeof(DenseLds::b), "LDS");
    DenseLds& L = *reinterpret_cast<DenseLds*>(smem);
    if (p.counts[2] != 0 || !dense_bins(p.bins)) {
        return;  // pair_kernel marks the overflow, or walks all bins
    }
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool fermi = p.particle_cut == 1;
    const bool finite = p.table_counts[3] == 0;
    const uint32_t np = static_cast<uint32_t>(p.n_pairs);
    const auto place = [&](uint32_t slot) {
        return L.before[slot >> 6] + static_cast<uint32_t>(__popcll(L.bits[slot >> 6] & ((1ull << (slot & 63u)) - 1ull)));
    };
    for (uint32_t panel = blockIdx.x;; panel += gridDim.x) {
        uint32_t local = panel, window = 0;
        int bin = kSplitBin - 1;
        for (; bin >= kDenseFirst; --bin) {
            window = panel_window(bin);
            const uint32_t here = bin_panels(p.bins, bin);
            if (local < here) {
                break;
            }
            local -= here;
        }
        if (bin < kDenseFirst) {
            return;  // the whole work-group
        }
        __syncthreads();  // the previous panel's LDS is done with
        if (tid < kDenseSlots / 64) {
            L.bits[tid] = 0ull;
        }
        if (wave == 0) {
            // the groups that start in the panel's list elements (at most eight, save whole ones)
            const uint32_t at = local * window + static_cast<uint32_t>(lane);
            const bool in = lane < static_cast<int>(window) && at < p.bins->groups[bin];
            const uint2 item = in ? p.glist[p.bins->list_base[bin] + at] : make_uint2(0u, 0u);
            const bool whole = (item.y & kWholeGroup) != 0u;
            const bool start = in && (whole || (item.y >> 16) == 0u);
            const uint64_t starts = __ballot(start);
            if (start) {
                L.groups[__popcll(starts & ((1ull << lane) - 1ull))] = make_uint2(item.x, whole ? item.y & ~kWholeGroup : item.y & kTiledMax);
            }
            if (lane == 0) {
                L.n_groups = static_cast<uint32_t>(__popcll(starts));
            }
        }
        __syncthreads();
        const uint32_t n_groups = L.n_groups;
        const int own_group = wave % kDenseGroups;  // two waves to a group
        const uint32_t own_first = static_cast<uint32_t>(wave / kDenseGroups * 64 + lane);
        const uint2 own = static_cast<uint32_t>(own_group) < n_groups ? L.groups[own_group] : make_uint2(0u, 0u);
        bool dense = finite && n_groups <= kDenseGroups;
        uint64_t pairs = 0;
        for (uint32_t g = 0; g < n_groups; ++g) {
            pairs += static_cast<uint64_t>(L.groups[g].y) * L.groups[g].y;
            dense = dense && L.groups[g].y <= kDenseUnion;
        }
        if (dense) {
            for (uint32_t e = own_first; e < own.y; e += 64 * kDenseWaves / kDenseGroups) {
                const uint32_t slot = binned_entry(p.mvals[own.x + e], fermi).slot;
                atomicOr(reinterpret_cast<unsigned long long*>(&L.bits[slot >> 6]), 1ull << (slot & 63u));
            }
            __syncthreads();
            if (wave == 0) {
                const uint32_t c0 = static_cast<uint32_t>(__popcll(L.bits[2 * lane])), c1 = static_cast<uint32_t>(__popcll(L.bits[2 * lane + 1]));
                uint32_t incl = c0 + c1;
#pragma unroll
                for (int d = 1; d < 64; d <<= 1) {
                    const uint32_t o = __shfl_up(incl, d);
                    incl += lane >= d ? o : 0u;
                }
                L.before[2 * lane] = incl - c0 - c1;
                L.before[2 * lane + 1] = incl - c1;
                if (lane == 63) {
                    L.used = incl;
                }
            }
            __syncthreads();
            const uint64_t tiles = (L.used + 15u) / 16u;
            dense = L.used <= kDenseUnion && pairs >= kDenseGain * tiles * tiles * 4u;
        }
        if (!dense) {
            __syncthreads();
            Stage<NV>& st = reinterpret_cast<Stage<NV>*>(L.b)[wave];
            uint32_t item = 0;
            for (uint32_t g = 0; g < n_groups; ++g) {
                const uint2 group = L.groups[g];
                const bool whole = group.y > kTiledMax;
                for (uint32_t t = 0; t < group_tiles(group.y); ++t, ++item) {
                    if (item % kDenseWaves == static_cast<uint32_t>(wave)) {
                        pair_big<ADJ, true, NV, kPairBatch>(p, group.x, group.y, 64u * t, whole ? group.y : 64u * t + 1u, lane, st);
                    }
                }
            }
            continue;
        }
        const int used = static_cast<int>(L.used);
        const int n_rows = (used + 15) / 16 * 16;
        const int n_cols = (used + kDenseStep - 1) / kDenseStep * kDenseStep;
        {
            const int word = tid >> 3, byte = 8 * (tid & 7);  // kDenseThreads = 8 * words
            const uint64_t bits = L.bits[word];
            uint32_t m = static_cast<uint32_t>(bits >> byte) & 0xffu;
            uint32_t at = L.before[word] + static_cast<uint32_t>(__popcll(bits & ((1ull << byte) - 1ull)));
            while (m) {
                L.slots[at++] = static_cast<uint32_t>(64 * word + byte + __builtin_ctz(m));
                m &= m - 1;
            }
            if (used + tid < n_cols) {
                L.slots[used + tid] = 0u;
            }
        }
        for (int t = tid; t < n_rows * kDenseGroups; t += kDenseThreads) {
            L.rows[t] = ~0u;
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            for (int t = tid; t < n_cols * 16; t += kDenseThreads) {
                L.b[t] = 0.0;
            }
            __syncthreads();
            for (uint32_t i = own_first; i < own.y; i += 64 * kDenseWaves / kDenseGroups) {
                const Entry e = binned_entry(p.mvals[own.x + i], fermi);
                const uint32_t at = place(e.slot);
                const double2 x = signed_by((v == 0 ? p.in : p.in2)[e.row], e.sign);
                L.rows[at * kDenseGroups + own_group] = e.row | (e.sign << 31);
                L.b[16 * at + 2 * own_group] = x.x;
                L.b[16 * at + 2 * own_group + 1] = x.y;
            }
            __syncthreads();
            double* out = reinterpret_cast<double*>(v == 0 ? p.out : p.out2);
            const int quad = lane >> 4, col = lane & 15;
            for (int r0 = 16 * wave; r0 < n_rows; r0 += 16 * kDenseWaves) {
                const uint32_t row_slot = L.slots[r0 + col];
                const auto load = [&](int k) {
                    const uint32_t slot = L.slots[k + quad];
                    return p.coef_re[ADJ ? row_slot * np + slot : slot * np + row_slot];
                };
                f64x4 acc = {0.0, 0.0, 0.0, 0.0};
                double next[kDenseStep / 4];
#pragma unroll
                for (int q = 0; q < kDenseStep / 4; ++q) {
                    next[q] = load(4 * q);
                }
                for (int k0 = 0; k0 < n_cols; k0 += kDenseStep) {
                    double a[kDenseStep / 4];
#pragma unroll
                    for (int q = 0; q < kDenseStep / 4; ++q) {
                        a[q] = next[q];
                    }
                    if (k0 + kDenseStep < n_cols) {
#pragma unroll
                        for (int q = 0; q < kDenseStep / 4; ++q) {
                            next[q] = load(k0 + kDenseStep + 4 * q);
                        }
                    }
#pragma unroll
                    for (int q = 0; q < kDenseStep / 4; ++q) {
                        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], L.b[16 * (k0 + 4 * q + quad) + col], acc, 0, 0, 0);
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t row = L.rows[(r0 + 4 * q + quad) * kDenseGroups + (col >> 1)];
                    if (row != ~0u && acc[q] != 0.0) {
                        const double x = (row >> 31) != 0u ? -acc[q] : acc[q];
                        unsafeAtomicAdd(&out[2 * static_cast<int64_t>(row & 0x7fffffffu) + (lane & 1)], x);
                    }
                }
            }
            if (v + 1 < NV) {
                __syncthreads();
            }
        }
    }
}

// ------------------------------------------------------------------------- single excitations --
// Launched with whole waves: threads past n_terms take part in the counts only.
__global__ void singles_fill_kernel(const int16_t* __restrict__ site, const uint8_t* __restrict__ kind,
                                    const double2* __restrict__ coef, int64_t n_terms, int particle_cut, int n_bits,
                                    double2* __restrict__ a, double2* __restrict__ kd, int64_t* __restrict__ counts) {
    const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    bool is_single = false, is_dressed = false;
    if (t < n_terms) {
        const CompiledTerm c = compile_term(site + 4 * t, kind + 4 * t, particle_cut, n_bits);
        SingleExcitation e;
        if (c.status == kCompileOk && single_excitation(c.rec, particle_cut, &e)) {
            const double2 v0 = coef[t];
            // single_parity(core + r) = popcount(core & (L(r) ^ L(p))) + (r < p): the last part is the
            // table's, the rest a sign per (core, site)
            const int flip = e.delta ^ ((particle_cut == 1 && e.r < e.p) ? 1 : 0);
            const double2 v = flip ? make_double2(-v0.x, -v0.y) : v0;
            const int64_t rp = static_cast<int64_t>(e.r) * n_bits + e.p;
            if (e.k < 0 || !e.kocc) {
                // holds whenever k is empty
                unsafeAtomicAdd(&a[rp].x, v.x);
                unsafeAtomicAdd(&a[rp].y, v.y);
            }
            if (e.k >= 0) {
                double2* dk = kd + rp * n_bits + e.k;
                unsafeAtomicAdd(&dk->x, e.kocc ? v.x : -v.x);
                unsafeAtomicAdd(&dk->y, e.kocc ? v.y : -v.y);
                is_dressed = true;
            }
            is_single = true;
        }
    }
    wave_count(&counts[0], is_single);
    wave_count(&counts[1], is_dressed);
}

int singles_layout(Carver& cv, int n_qubytes, qmb_singles* out) {
    QMB_TRY(check_qubytes(n_qubytes));
    if (n_qubytes > kMaxPairBytes) {
        return set_error(QMB_ERR_UNSUPPORTED, "the single-excitation table supports n_qubytes <= %d, got %d", kMaxPairBytes,
                         n_qubytes);
    }
    qmb_singles g{};
    g.n_qubytes = n_qubytes;
    g.n_bits = 8 * n_qubytes;
    const size_t nb = static_cast<size_t>(g.n_bits);
    g.buffer = cv.base;
    g.counts = cv.take<int64_t>(4);
    g.a = cv.take<double>(2 * nb * nb);
    g.kd = cv.take<double>(2 * nb * nb * nb);
    g.a_re = cv.take<double>(nb * nb);
    g.kd_re = cv.take<double>(nb * nb * nb);
    g.bytes = cv.off;
    if (out) {
        *out = g;
    }
    return QMB_OK;
}

struct SingleParams {
    const double2* a;       // the single-excitation table with the sign of r < p in it
    const double2* kd;
    const double* a_re;   // their real parts when every coefficient is real, else null
    const double* kd_re;
    int n_bits;
    int particle_cut;
    const uint64_t* ckeys;
    const uint64_t* mvals;  // binned entries
    const uint2* glist;
    const CoreBins* bins;
    const int64_t* counts;
    const double2* in;
    double2* out;
    const double2* in2;  // second input/output of a two-vector pass (NV = 2), else null
    double2* out2;
};

// Parity of the sites of c between r and p (core sites: the sign left when the table holds that of
// r < p).
template <int W>
__device__ __forceinline__ int single_parity(const Cfg<W>& c, int r, int p) {
    return masked_parity<W>(c, range_mask<W>(r < p ? r : p, r < p ? p : r));
}

// Sum of row[k] over the set bits k of c, ascending k.  Up to CH indices are taken from the mask
// before their loads are issued, so the loads of one element overlap instead of each waiting for the
// last add (same order of additions, same result as a bit-by-bit walk).  The single-set kernels use
// CH = kSingleLoads (13: the 13 core sites of a 14-electron config in one batch; single kernel 1.68
// -> 1.40 ms at 52 spin orbitals and 7a+7b against 8, while 16 ran 1.67 ms); the batch kernel, held
// to 128 VGPRs, uses 4 (measured on 64 molecular instances: 126.8 ms
// per step against 128.8 ms with 2 and 130.7 ms with the plain walk).  row must hold at least
// 64 * (W - 1) + 1 entries (a lane without an index reads row[64 w] and drops it).
constexpr int kSingleLoads = 13;
__device__ __forceinline__ double zero_like(double) { return 0.0; }
__device__ __forceinline__ double2 zero_like(double2) { return make_double2(0.0, 0.0); }
__device__ __forceinline__ double add_to(double a, double b) { return a + b; }
__device__ __forceinline__ double2 add_to(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }

template <int W, typename T, int CH>
__device__ __forceinline__ T masked_row_sum(const T* __restrict__ row, const Cfg<W>& c, T acc) {
#pragma unroll
    for (int w = 0; w < W; ++w) {
        uint64_t m = c.w[w];
        while (m) {
            T v[CH];
#pragma unroll
            for (int u = 0; u < CH; ++u) {
                const bool have = m != 0ull;
                const int k = 64 * w + (have ? __builtin_ctzll(m) : 0);
                m = have ? m & (m - 1ull) : 0ull;
                const T x = row[k];
                v[u] = have ? x : zero_like(x);
            }
#pragma unroll
            for (int u = 0; u < CH; ++u) {
                acc = add_to(acc, v[u]);
            }
        }
    }
    return acc;
}

// Element of the single excitation (annihilate r, create p) on a source config whose other
// occupied sites are `core`.
template <int W, int CH>
__device__ __forceinline__ double2 single_element(const SingleParams& p, const Cfg<W>& core, int r, int q) {
    const int64_t rq = static_cast<int64_t>(r) * p.n_bits + q;
    if (p.kd_re) {
        // real table: 8-byte reads, the sum kept in one register
        return make_double2(masked_row_sum<W, double, CH>(p.kd_re + rq * p.n_bits, core, p.a_re[rq]), 0.0);
    }
    return masked_row_sum<W, double2, CH>(p.kd + rq * p.n_bits, core, p.a[rq]);
}

// acc += x g (!ADJ) or conj(x) g (ADJ).
template <bool ADJ>
__device__ __forceinline__ void single_madd(const double2& x, const double2& g, double& re, double& im) {
    if (ADJ) {
        re += x.x * g.x + x.y * g.y;
        im += x.x * g.y - x.y * g.x;
    } else {
        re += x.x * g.x - x.y * g.y;
        im += x.x * g.y + x.y * g.x;
    }
}

// Order-1 groups: rows a (config = core + r) against entries b (config = core + q), the sign split into
// one factor per entry (the core's sites below its site) and the table's part:
//   ADJ:  out[a] += sign_a sum_b sign_b conj(M[r][q]) in[b],  M[r][q] = A[r][q] + sum_{k in core} K[r][q][k]
//   !ADJ: out[a] += sign_a sum_b sign_b M[q][r] in[b]
// Groups of g = 2..32 entries, lane = row, 64 / g groups to a pass; each row meets the other g - 1
// entries in turn.
template <int W, bool ADJ, int NV, int CH>
__device__ __forceinline__ void single_rows(const SingleParams& p, int g, uint32_t e0, uint32_t e_end, int lane, Stage<NV>& st) {
    const bool fermi = p.particle_cut == 1;
    const int lanes = 64 / g * g;
    const uint32_t at = e0 + static_cast<uint32_t>(lane);
    const bool act = lane < lanes && at < e_end;
    const int lead = act ? lane / g * g : 0;
    const int ri = lane - lead;
    const Entry e = binned_entry(act ? p.mvals[at] : 0ull, fermi);
    // the group's first row reads its config for the group
    Cfg<W> own;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        own.w[w] = act && ri == 0 ? p.ckeys[static_cast<int64_t>(e.row) * W + w] : 0ull;
    }
    if (act) {
        flip_site<W>(own, static_cast<int>(e.slot));
    }
    stage_lane<NV>(p, st, lane, act, e, e.slot);
    Cfg<W> core;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        core.w[w] = shfl_u64(own.w[w], lead);  // every lane runs every shuffle
    }
    __builtin_amdgcn_wave_barrier();
    double re[NV] = {}, im[NV] = {};
    if (act) {
        const int r = static_cast<int>(e.slot);
        for (int u = 1; u < g; ++u) {
            const int b = lead + (ri + u >= g ? ri + u - g : ri + u);
            const int q = static_cast<int>(st.part[b]);
            const double2 x = ADJ ? single_element<W, CH>(p, core, r, q) : single_element<W, CH>(p, core, q, r);
            single_madd<ADJ>(x, st.g[b], re[0], im[0]);
            if constexpr (NV == 2) {
                single_madd<ADJ>(x, st.g2[b], re[1], im[1]);
            }
        }
    }
    add_rows<NV>(p, st, 0, lane, act, e, re, im);
}

// Rows [first, last) of one group of any size from mvals[s], lane = row.
template <int W, bool ADJ, int NV, int CH>
__device__ __forceinline__ void single_group(const SingleParams& p, uint32_t s, uint32_t size, uint32_t first, uint32_t last, int lane, Stage<NV>& st) {
    const bool fermi = p.particle_cut == 1;
    const Entry head = binned_entry(p.mvals[s], fermi);
    Cfg<W> core = load_key<W>(p.ckeys, static_cast<int64_t>(head.row));
    flip_site<W>(core, static_cast<int>(head.slot));
    for (uint32_t a0 = first; a0 < last; a0 += 64) {
        const bool act = a0 + lane < size;
        const Entry e = binned_entry(p.mvals[s + (act ? a0 + lane : 0u)], fermi);
        const int r = static_cast<int>(e.slot);
        double re[NV] = {}, im[NV] = {};
        for (uint32_t b = 0; b < size; ++b) {
            const Entry eb = binned_entry(p.mvals[s + b], fermi);
            const int q = static_cast<int>(eb.slot);
            if (!act || q == r) {
                continue;
            }
            const double2 x = ADJ ? single_element<W, CH>(p, core, r, q) : single_element<W, CH>(p, core, q, r);
            single_madd<ADJ>(x, signed_by(p.in[eb.row], eb.sign), re[0], im[0]);
            if constexpr (NV == 2) {
                single_madd<ADJ>(x, signed_by(p.in2[eb.row], eb.sign), re[1], im[1]);
            }
        }
        add_rows<NV>(p, st, 0, lane, act, e, re, im);
    }
}

// One work unit of the single bins.
template <int W, bool ADJ, int NV, int CH>
__device__ __forceinline__ void single_unit(const SingleParams& p, uint32_t u, int lane, Stage<NV>& st) {
    uint32_t local;
    const int bin = unit_bin(p.bins, u, lane, &local);
    if (bin < kExactBins) {
        const int g = bin + 2;
        const int passes = unit_passes(g, 1);
        const uint32_t base = p.bins->entry_base[bin];
        const uint32_t e_end = base + p.bins->groups[bin] * static_cast<uint32_t>(g);
        const uint32_t step = static_cast<uint32_t>(64 / g * g);
        for (int k = 0; k < passes; ++k) {
            const uint32_t e0 = base + (local * static_cast<uint32_t>(passes) + static_cast<uint32_t>(k)) * step;
            if (e0 < e_end) {  // wave-uniform
                single_rows<W, ADJ, NV, CH>(p, g, e0, e_end, lane, st);
            }
        }
        return;
    }
    for_listed(p, bin, local, lane, [&](uint32_t s, uint32_t size, uint32_t first, uint32_t last) {
        single_group<W, ADJ, NV, CH>(p, s, size, first, last, lane, st);
    });
}

template <int W, bool ADJ, int NV = 1>
__global__ __launch_bounds__(kBlock) void single_kernel(SingleParams p) {
    __shared__ Stage<NV> stages[kWavesPerBlock];
    const int lane = threadIdx.x & 63;
    const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>((blockIdx.x * blockDim.x + threadIdx.x) >> 6)));
    const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
    if (p.counts[2] != 0) {
        if (wave == 0 && lane == 0) {
            mark_overflow(p.out);
        }
        return;
    }
    const uint32_t units = p.bins->unit_start[kBins];
    for (uint32_t u = wave; u < units; u += nwaves) {
        single_unit<W, ADJ, NV, kSingleLoads>(p, u, lane, stages[threadIdx.x >> 6]);
    }
}

// ----------------------------------------------------------------------------------- hops --
// A single excitation between two sites of one parity (a spin-conserving hop when sites interleave
// spin: even = up, odd = down) leaves the string on the other parity's sites unchanged, so the two
// configs it connects hold equal strings there.  The strings index of parity s groups a set's rows
// by their string on the sites of parity 1 - s: one entry per row, sorted by a 32-bit key of that
// string (a hash of it mod 2^32 - 1).  Inside a group two rows are connected by such a hop iff their
// configs differ in exactly two sites, both of parity s, one occupied in each; rows of different
// strings merged by equal keys fail that test.  Building it sorts n keys, where the order-1 core
// index sorts n per occupied site.
constexpr uint64_t kEvenSites = 0x5555555555555555ull;

__host__ __device__ __forceinline__ uint64_t parity_sites(int parity) { return parity ? ~kEvenSites : kEvenSites; }

// The sites of one parity of a config word, packed into 32 bits (site 2j + parity -> bit j).
__device__ __forceinline__ uint64_t parity_bits(uint64_t x, int parity) {
    x = (parity ? x >> 1 : x) & kEvenSites;
    x = (x | (x >> 1)) & 0x3333333333333333ull;
    x = (x | (x >> 2)) & 0x0F0F0F0F0F0F0F0Full;
    x = (x | (x >> 4)) & 0x00FF00FF00FF00FFull;
    x = (x | (x >> 8)) & 0x0000FFFF0000FFFFull;
    x = (x | (x >> 16)) & 0x00000000FFFFFFFFull;
    return x;
}

// The key of a row: its other-parity string packed (bit 32 w + j = site 64 w + 2 j + 1 - parity),
// mixed by the 64-bit finaliser, mod 2^32 - 1 (the key no entry holds marks nothing here).
template <int W>
__global__ void strings_emit_kernel(const uint64_t* __restrict__ keys, int64_t n, int parity, uint32_t* __restrict__ okeys,
                                    uint32_t* __restrict__ orows) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (i >= n) {
        return;
    }
    const Cfg<W> c = load_key<W>(keys, i);
    uint64_t other = 0ull;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        other |= parity_bits(c.w[w], parity ^ 1) << (32 * w);
    }
    okeys[i] = static_cast<uint32_t>(fmix64(other ^ 0x2545f4914f6cdd1dull) % 0xFFFFFFFFull);
    orows[i] = static_cast<uint32_t>(i);
}

// group[e] holds the inclusive count of group starts up to entry e; turned into the entry's group.
__global__ void strings_start_kernel(const uint32_t* __restrict__ flag, uint32_t* __restrict__ group, int64_t n,
                                     uint32_t* __restrict__ starts, int64_t* __restrict__ counts) {
    const int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (e >= n) {
        return;
    }
    const uint32_t g = group[e] - 1u;
    group[e] = g;
    if (flag[e]) {
        starts[g] = static_cast<uint32_t>(e);
    }
    if (e == n - 1) {
        starts[g + 1] = static_cast<uint32_t>(n);
        counts[0] = n;
        counts[1] = static_cast<int64_t>(g) + 1;
    }
}

// counts[2] = sum of size^2 over the groups of two or more rows (the pairs the hop kernel tests),
// counts[3] = the largest group: a grid-stride pass, one atomic per block.
__global__ __launch_bounds__(kBlock) void strings_stats_kernel(const uint32_t* __restrict__ starts, int64_t* __restrict__ counts) {
    __shared__ unsigned long long s_sq[kBlock / 64], s_mx[kBlock / 64];
    const int64_t groups = counts[1];
    unsigned long long sq = 0ull, mx = 0ull;
    for (int64_t g = blockIdx.x * static_cast<int64_t>(kBlock) + threadIdx.x; g < groups; g += static_cast<int64_t>(gridDim.x) * kBlock) {
        const unsigned long long sz = starts[g + 1] - starts[g];
        sq += sz >= 2ull ? sz * sz : 0ull;
        mx = sz > mx ? sz : mx;
    }
    for (int d = 32; d > 0; d >>= 1) {
        sq += __shfl_down(sq, d);
        const unsigned long long o = __shfl_down(mx, d);
        mx = o > mx ? o : mx;
    }
    if ((threadIdx.x & 63) == 0) {
        s_sq[threadIdx.x >> 6] = sq;
        s_mx[threadIdx.x >> 6] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / 64; ++w) {
            sq += s_sq[w];
            mx = s_mx[w] > mx ? s_mx[w] : mx;
        }
        if (mx != 0ull) {
            atomicAdd(reinterpret_cast<unsigned long long*>(&counts[2]), sq);
            atomicMax(reinterpret_cast<unsigned long long*>(&counts[3]), mx);
        }
    }
}

// mflag[e] = 1 when entry e's group holds two or more rows.
__global__ void strings_multi_kernel(const uint32_t* __restrict__ group, const uint32_t* __restrict__ starts, int64_t n,
                                     uint32_t* __restrict__ mflag) {
    const int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (e >= n) {
        return;
    }
    const uint32_t g = group[e];
    mflag[e] = starts[g + 1] - starts[g] >= 2u ? 1u : 0u;
}

// The entries of groups of two or more rows, in index order, with their config words and hop-parity
// string (site 2j + parity -> bit j) gathered and each entry's group as a range of the compacted
// order (mpos: exclusive scan of mflag); counts[4] = their number.
template <int W>
__global__ void strings_compact_kernel(const uint64_t* __restrict__ ckeys, const uint32_t* __restrict__ rows,
                                       const uint32_t* __restrict__ group, const uint32_t* __restrict__ starts,
                                       const uint32_t* __restrict__ mflag, const uint32_t* __restrict__ mpos, int64_t n, int parity,
                                       uint32_t* __restrict__ mrows, uint2* __restrict__ mrange, uint64_t* __restrict__ mcfg,
                                       uint64_t* __restrict__ mstr, int64_t* __restrict__ counts) {
    const int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (e >= n) {
        return;
    }
    if (e == n - 1) {
        counts[4] = static_cast<int64_t>(mpos[e]) + mflag[e];
    }
    if (!mflag[e]) {
        return;
    }
    const uint32_t p = mpos[e];
    const uint32_t g = group[e];
    const uint32_t lo = mpos[starts[g]];
    const uint32_t row = rows[e];
    mrows[p] = row;
    mrange[p] = make_uint2(lo, lo + (starts[g + 1] - starts[g]));
    uint64_t str = 0ull;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const uint64_t c = ckeys[static_cast<int64_t>(row) * W + w];
        mcfg[static_cast<int64_t>(p) * W + w] = c;
        str |= parity_bits(c, parity) << (32 * w);
    }
    mstr[p] = str;
}

// A compacted group whose rows hold more than one other-parity string (strings merged by equal
// keys): mix[first entry] = 1.
template <int W>
__global__ void strings_mixed_kernel(const uint2* __restrict__ mrange, const uint64_t* __restrict__ mcfg, const int64_t* __restrict__ counts,
                                     int parity, uint32_t* __restrict__ mix) {
    const int64_t p = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (p < 1 || p >= counts[4]) {
        return;
    }
    const uint32_t lo = mrange[p].x;
    if (lo == p) {
        return;
    }
    const uint64_t other = parity_sites(parity ^ 1);
    bool differ = false;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        differ = differ || ((mcfg[p * W + w] ^ mcfg[(p - 1) * W + w]) & other) != 0ull;
    }
    if (differ) {
        mix[lo] = 1u;
    }
}

// Marks the entries of merged groups: bit 31 of their range's end.
__global__ void strings_mark_kernel(const uint32_t* __restrict__ mix, const int64_t* __restrict__ counts, uint2* __restrict__ mrange) {
    const int64_t p = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (p >= counts[4]) {
        return;
    }
    if (mix[mrange[p].x]) {
        mrange[p].y |= 0x80000000u;
    }
}

template <int W>
struct HopStage {
    uint64_t c[W];  // config of the entry's row
    double2 g;      // in[row]
};

struct HopParams {
    SingleParams s;          // the single-excitation tables, in, out and the set's config words
    const int64_t* scounts;  // the tables' counts: [1] = terms with a conditioned site
    uint64_t sites;          // the hop parity's sites, per word
    int parity;
    const uint32_t* mrows;   // the compacted entries (groups of two or more rows): row,
    const uint2* mrange;     // group as a range of the compacted order (bit 31 of the end: merged group),
    const uint64_t* mcfg;    // config words,
    const uint64_t* mstr;    // hop-parity string
    const int64_t* counts;   // [4] = number of compacted entries
};

// One wave per 64 consecutive compacted entries (rows of groups of two or more): lane = row a.  The
// wave walks the entries of the union of its rows' groups (consecutive in the compacted order),
// staged 64 at a time in LDS (amplitudes gathered) and read back as broadcasts, and tests each
// pair: in a wave of unmerged groups only the hop-parity strings of the rows of the lane's own
// group (the other parity's strings are equal there), else the whole configs.  The connections a
// chunk finds (a row may have many: the seed of a star of hops) are then listed in LDS and shared
// out over the lanes, one (row, entry) per lane per round, so their elements and coefficient loads
// run side by side; each row's sum collects in LDS and is added to out[a] without atomics (each row
// has one entry).
//   ADJ:  out[a] += conj(M_ba) in[b],  M_ba = (-1)^single_parity(core; r, q) (A[r][q] + sum_{k in core} K[r][q][k])
//   !ADJ: out[a] += M_ab in[b],        M_ab = (-1)^single_parity(core; q, r) (A[q][r] + sum_{k in core} K[q][r][k])
// with r the site of a, q the site of b (c_a = core + r, c_b = core + q), as in single_rows.
constexpr int kHopList = 256;  // connections listed per round, per wave

template <int W>
struct HopWaveLds {
    HopStage<W> stage[64];
    uint64_t rowc[64][W];      // the lanes' row configs
    double2 acc[64];           // the lanes' row sums
    uint16_t list[kHopList];   // lane << 6 | entry slot
};

template <bool ADJ>
__device__ __forceinline__ void hop_madd(double xr, double xi, const double2& g, double& re, double& im) {
    if (ADJ) {
        re += xr * g.x + xi * g.y;
        im += xr * g.y - xi * g.x;
    } else {
        re += xr * g.x - xi * g.y;
        im += xr * g.y + xi * g.x;
    }
}

template <int W, bool ADJ>
__global__ __launch_bounds__(kBlock) void hop_kernel(HopParams p) {
    __shared__ HopWaveLds<W> lds_all[kBlock / 64];
    const int lane = threadIdx.x & 63;
    HopWaveLds<W>& L = lds_all[threadIdx.x >> 6];
    const int64_t wave = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) >> 6;
    const int64_t nwaves = (static_cast<int64_t>(gridDim.x) * kBlock) >> 6;
    const int64_t entries = p.counts[4];
    const bool fermi = p.s.particle_cut == 1;
    const bool plain = p.scounts[1] == 0;
    for (int64_t base = wave * 64; base < entries; base += nwaves * 64) {
        const int64_t e = base + lane;
        const bool act = e < entries;
        const uint2 range = act ? p.mrange[e] : make_uint2(0xFFFFFFFFu, 0u);
        const uint32_t gs = range.x, ge = range.y & 0x7FFFFFFFu;
        // a wave meeting a merged group compares whole configs; the others compare the hop-parity
        // strings of the rows of their own groups
        const bool merged = __ballot(act && (range.y >> 31) != 0u) != 0ull;
        // the entries any row of the wave can meet: the union of its rows' groups
        uint32_t lo = gs, hi = ge;
        for (int d = 32; d > 0; d >>= 1) {
            const uint32_t ol = __shfl_xor(lo, d);
            const uint32_t oh = __shfl_xor(hi, d);
            lo = ol < lo ? ol : lo;
            hi = oh > hi ? oh : hi;
        }
        lo = __builtin_amdgcn_readfirstlane(lo);
        hi = __builtin_amdgcn_readfirstlane(hi);
        const int64_t ia = act ? static_cast<int64_t>(p.mrows[e]) : 0;
        Cfg<W> ca;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            ca.w[w] = act ? p.mcfg[e * W + w] : 0ull;
            L.rowc[lane][w] = ca.w[w];
        }
        const uint64_t sa = act ? p.mstr[e] : 0ull;
        // the particle count of the wave's first row's string, and whether every row of the wave
        // holds as many (lane 0 always has a row)
        const int pc_ref = __builtin_amdgcn_readfirstlane(__popcll(sa));
        const bool rows_even = __ballot(act && __popcll(sa) != pc_ref) == 0ull;
        L.acc[lane] = make_double2(0.0, 0.0);
        for (uint32_t c0 = lo; c0 < hi; c0 += 64u) {
            const uint32_t b = c0 + static_cast<uint32_t>(lane);
            bool uneven = false;
            if (b < hi) {
                HopStage<W> st;
                if (merged) {
#pragma unroll
                    for (int w = 0; w < W; ++w) {
                        st.c[w] = p.mcfg[static_cast<int64_t>(b) * W + w];
                    }
                } else {
                    st.c[0] = p.mstr[b];
                    uneven = __popcll(st.c[0]) != pc_ref;
                }
                st.g = p.s.in[p.mrows[b]];
                L.stage[lane] = st;
            }
            // every string the chunk's pair tests meet holds pc_ref particles (every lane runs the
            // ballot)
            const bool staged_even = __ballot(uneven) == 0ull;
            const bool even = rows_even && staged_even;
            __builtin_amdgcn_wave_barrier();
            const int nb = static_cast<int>(hi - c0 < 64u ? hi - c0 : 64u);
            // the pair tests: bit u of `hit` marks a connection of this lane's row to entry u.  A row
            // meets only the entries of its own group, so each lane walks its group's part of the
            // chunk: the wave's walk is the longest such part, not the whole union.
            const int ulo = static_cast<int>(gs) - static_cast<int>(c0) > 0 ? static_cast<int>(gs) - static_cast<int>(c0) : 0;
            const int uend = static_cast<int>(ge) - static_cast<int>(c0);
            const int uhi = act ? (uend < nb ? uend : nb) : 0;
            uint64_t hit = 0ull;
            if (merged) {
                for (int u = ulo; u < uhi; ++u) {
                    const HopStage<W>& st = L.stage[u];
                    int pc = 0, pa = 0;
                    uint64_t off = 0ull;
#pragma unroll
                    for (int w = 0; w < W; ++w) {
                        const uint64_t d = ca.w[w] ^ st.c[w];
                        pc += __popcll(d);
                        pa += __popcll(d & ca.w[w]);
                        off |= d & ~p.sites;
                    }
                    // two sites differ, both of the hop parity, one occupied in each config
                    hit |= (pc == 2 && pa == 1 && off == 0ull) ? (1ull << u) : 0ull;
                }
            } else if (even) {
                // rows of one (unmerged) group share the other parity's string, and strings of
                // equal particle counts that differ in two sites hold one of them each: the count
                // of differing sites decides
                for (int u = ulo; u < uhi; ++u) {
                    hit |= static_cast<uint64_t>(__popcll(sa ^ L.stage[u].c[0]) == 2) << u;
                }
            } else {
                // rows of one (unmerged) group share the other parity's string: two hop-parity
                // sites differ, one occupied in each
                for (int u = ulo; u < uhi; ++u) {
                    const uint64_t d = sa ^ L.stage[u].c[0];
                    const bool ok = __popcll(d) == 2 && __popcll(d & sa) == 1;
                    hit |= ok ? (1ull << u) : 0ull;
                }
            }
            hit = act ? hit : 0ull;
            // list the chunk's connections (lane-major) and share them out, kHopList per round
            const int cnt = __popcll(hit);
            int off = cnt;
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(off, d);
                off += lane >= d ? o : 0;
            }
            const int total = __shfl(off, 63);
            off -= cnt;  // exclusive
            for (int r0 = 0; r0 < total; r0 += kHopList) {
                {
                    uint64_t h = hit;
                    int k = off;
                    while (h) {
                        const int u = __builtin_ctzll(h);
                        h &= h - 1ull;
                        if (k >= r0 && k < r0 + kHopList) {
                            L.list[k - r0] = static_cast<uint16_t>((lane << 6) | u);
                        }
                        ++k;
                    }
                }
                __builtin_amdgcn_wave_barrier();
                const int m = total - r0 < kHopList ? total - r0 : kHopList;
                for (int i = lane; i < m; i += 64) {
                    const int item = L.list[i];
                    const int la = item >> 6, u = item & 63;
                    const HopStage<W>& st = L.stage[u];
                    Cfg<W> cx;
#pragma unroll
                    for (int w = 0; w < W; ++w) {
                        cx.w[w] = L.rowc[la][w];
                    }
                    int r = 0, q = 0;
                    if (merged) {
#pragma unroll
                        for (int w = 0; w < W; ++w) {
                            const uint64_t d = cx.w[w] ^ st.c[w];
                            const uint64_t da = d & cx.w[w], db = d & st.c[w];
                            r = da ? 64 * w + __builtin_ctzll(da) : r;
                            q = db ? 64 * w + __builtin_ctzll(db) : q;
                        }
                    } else {
                        // the row's hop-parity string from its config words
                        uint64_t sx = 0ull;
#pragma unroll
                        for (int w = 0; w < W; ++w) {
                            sx |= parity_bits(cx.w[w], p.parity) << (32 * w);
                        }
                        const uint64_t d = sx ^ st.c[0];
                        r = 2 * __builtin_ctzll(d & sx) + p.parity;
                        q = 2 * __builtin_ctzll(d & st.c[0]) + p.parity;
                    }
                    Cfg<W> core = cx;
                    flip_site<W>(core, r);
                    const int sg = fermi ? single_parity<W>(core, r, q) : 0;
                    double2 x;
                    if (plain) {
                        const int64_t rq = ADJ ? static_cast<int64_t>(r) * p.s.n_bits + q : static_cast<int64_t>(q) * p.s.n_bits + r;
                        x = p.s.a_re ? make_double2(p.s.a_re[rq], 0.0) : p.s.a[rq];
                    } else {
                        x = ADJ ? single_element<W, 8>(p.s, core, r, q) : single_element<W, 8>(p.s, core, q, r);
                    }
                    double re = 0.0, im = 0.0;
                    hop_madd<ADJ>(sg ? -x.x : x.x, sg ? -x.y : x.y, st.g, re, im);
                    if (re != 0.0 || im != 0.0) {
                        atomicAdd(&L.acc[la].x, re);
                        atomicAdd(&L.acc[la].y, im);
                    }
                }
                __builtin_amdgcn_wave_barrier();
            }
        }
        __builtin_amdgcn_wave_barrier();
        const double2 acc = L.acc[lane];
        if (act && (acc.x != 0.0 || acc.y != 0.0)) {
            p.s.out[ia].x += acc.x;
            p.s.out[ia].y += acc.y;
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// ------------------------------------------------------------------------------- diagonal --
// d(c) = diag[0] + sum_{p in c} diag[1 + p] + sum_{p < q in c} diag[1 + n_bits + pair_index(p, q)]
template <int W, int CH>
__device__ __forceinline__ double2 diag_value(const Cfg<W>& c, const double2* __restrict__ diag, int n_bits) {
    double2 d = diag[0];
    const double2* e1 = diag + 1;
    const double2* e2 = diag + 1 + n_bits;
#pragma unroll
    for (int wp = 0; wp < W; ++wp) {
        uint64_t mp = c.w[wp];
        while (mp) {
            const int p = 64 * wp + __builtin_ctzll(mp);
            mp &= mp - 1;
            const double2 a = e1[p];
            d.x += a.x;
            d.y += a.y;
#pragma unroll
            for (int wq = 0; wq < W; ++wq) {
                if (wq < wp) {
                    continue;
                }
                uint64_t mq = wq == wp ? mp : c.w[wq];
                // up to CH partners q at a time: their loads go out together (same order of additions)
                while (mq) {
                    double2 v[CH];
#pragma unroll
                    for (int u = 0; u < CH; ++u) {
                        const bool have = mq != 0ull;
                        const int q = 64 * wq + (have ? __builtin_ctzll(mq) : 0);
                        mq = have ? mq & (mq - 1ull) : 0ull;
                        const double2 b = e2[have ? pair_index(p, q) : 0];
                        v[u] = have ? b : make_double2(0.0, 0.0);
                    }
#pragma unroll
                    for (int u = 0; u < CH; ++u) {
                        d.x += v[u].x;
                        d.y += v[u].y;
                    }
                }
            }
        }
    }
    return d;
}

// out[i] += d_i in[i] (conj(d_i) for ADJ)
template <int W, bool ADJ>
__global__ __launch_bounds__(kBlock) void diag_apply_kernel(const uint64_t* __restrict__ ckeys, int64_t n,
                                                            const double2* __restrict__ diag, int n_bits,
                                                            const double2* __restrict__ in, double2* __restrict__ out) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(kBlock) + threadIdx.x;
    if (i >= n) {
        return;
    }
    const double2 d = diag_value<W, 8>(load_key<W>(ckeys, i), diag, n_bits);
    const double im = ADJ ? -d.y : d.y;
    if (d.x != 0.0 || im != 0.0) {
        const double2 g = in[i];
        out[i].x += d.x * g.x - im * g.y;
        out[i].y += d.x * g.y + im * g.x;
    }
}

// The same diagonal on two vectors in one pass (d, or conj(d) for the adjoint): the config words
// and the folded table are read once for both.
template <int W, bool ADJ>
__global__ __launch_bounds__(kBlock) void diag_apply2_kernel(const uint64_t* __restrict__ ckeys, int64_t n,
                                                             const double2* __restrict__ diag, int n_bits,
                                                             const double2* __restrict__ in, double2* __restrict__ out,
                                                             const double2* __restrict__ in2, double2* __restrict__ out2) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(kBlock) + threadIdx.x;
    if (i >= n) {
        return;
    }
    const double2 d = diag_value<W, 8>(load_key<W>(ckeys, i), diag, n_bits);
    const double im = ADJ ? -d.y : d.y;
    if (d.x != 0.0 || im != 0.0) {
        const double2 g = in[i];
        const double2 g2 = in2[i];
        out[i].x += d.x * g.x - im * g.y;
        out[i].y += d.x * g.y + im * g.x;
        out2[i].x += d.x * g2.x - im * g2.y;
        out2[i].y += d.x * g2.y + im * g2.x;
    }
}

// --------------------------------------------------------------------- batched persistent launch --
// Many instances (term tables + config sets) in one pass: the work of every instance is cut into
// units -- those of its core indexes' bins, and 64 diagonal rows -- numbered type-major
// (all pair units, then singles, then diagonal, so the heaviest work is taken first), and
// persistent waves take units round-robin until all are done.  How many units an index makes up is
// known when it is built, on the device, so each application numbers them: a plan, or a graph of
// the launches, stays good when an index is built again in its place.  (Numbered by what the capacities
// allow, the gaps left the waves unevenly loaded: 64 sets of 1000 rows 51 -> 134 us.)
struct BatchItemDev {
    int32_t n_words, particle_cut, has_pairs, has_singles;
    int32_t n_bits, reserved;
    int64_t n;
    const uint64_t* ckeys;
    const double2* diag;
    const double2* pcoef;
    const double* pcoef_re;
    int64_t n_pairs;
    const uint64_t* pmvals;
    const uint2* pglist;
    const CoreBins* pbins;
    const int64_t* pcounts;
    const double2* sa;
    const double2* skd;
    const double* sa_re;
    const double* skd_re;
    const uint64_t* smvals;
    const uint2* sglist;
    const CoreBins* sbins;
    const int64_t* scounts;
    const double2* in;
    double2* out;
    const double2* in2;  // two-vector batches: the second input and output
    double2* out2;
};

constexpr int kBatchMaxItems = 4096;

template <int W, bool ADJ, int NV>
__device__ __forceinline__ void diag_rows(const BatchItemDev& it, int64_t r0, int lane) {
    const int64_t i = r0 + lane;
    if (i >= it.n) {
        return;
    }
    const double2 d = diag_value<W, 4>(load_key<W>(it.ckeys, i), it.diag, it.n_bits);
    const double im = ADJ ? -d.y : d.y;
    if (d.x != 0.0 || im != 0.0) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double2 g = (v == 0 ? it.in : it.in2)[i];
            double2* o = v == 0 ? it.out : it.out2;
            // pair and single units of the same launch add into these rows concurrently
            unsafeAtomicAdd(&o[i].x, d.x * g.x - im * g.y);
            unsafeAtomicAdd(&o[i].y, d.x * g.y + im * g.x);
        }
    }
}

// PART 1: the pair units (type 0); PART 2: the single-excitation (type 1) and diagonal (type 2)
// units.
template <int W, bool ADJ, int NV, int PART>
__device__ __forceinline__ void batch_unit(const BatchItemDev& it, int type, int64_t local, int lane, Stage<NV>& stage) {
    if (PART == 1 && type == 0) {
        PairParams p{};
        p.coef = it.pcoef;
        p.coef_re = it.pcoef_re;
        p.n_pairs = it.n_pairs;
        p.particle_cut = it.particle_cut;
        p.mvals = it.pmvals;
        p.glist = it.pglist;
        p.bins = it.pbins;
        p.counts = it.pcounts;
        p.in = it.in;
        p.out = it.out;
        p.in2 = it.in2;
        p.out2 = it.out2;
        if (it.pcounts[2] == 0) {
            if (p.coef_re != nullptr) {
                pair_unit<ADJ, true, NV, kPairBatch / 2>(p, static_cast<uint32_t>(local), lane, stage);
            } else {
                pair_unit<ADJ, false, NV, kPairBatch / 2>(p, static_cast<uint32_t>(local), lane, stage);
            }
        }
    } else if (PART == 2 && type == 1) {
        SingleParams p{};
        p.a = it.sa;
        p.kd = it.skd;
        p.a_re = it.sa_re;
        p.kd_re = it.skd_re;
        p.n_bits = it.n_bits;
        p.particle_cut = it.particle_cut;
        p.ckeys = it.ckeys;
        p.mvals = it.smvals;
        p.glist = it.sglist;
        p.bins = it.sbins;
        p.counts = it.scounts;
        p.in = it.in;
        p.out = it.out;
        p.in2 = it.in2;
        p.out2 = it.out2;
        if (it.scounts[2] == 0) {
            single_unit<W, ADJ, NV, 4>(p, static_cast<uint32_t>(local), lane, stage);
        }
    } else if (PART == 2 && type == 2) {
        diag_rows<W, ADJ, NV>(it, local * 64, lane);
        if (local == 0 && lane == 0 &&
            ((it.has_pairs && it.pcounts[2] != 0) || (it.has_singles && it.scounts[2] != 0))) {
            mark_overflow(it.out);
            if (NV == 2) {
                mark_overflow(it.out2);
            }
        }
    }
}

// For batches whose waves do not number the units themselves: offsets[type * n_items + item] = first unit of the instance's units of the type, then their number.
// One block; applications of one plan write the same.
constexpr int kOffsetThreads = 1024;
__global__ __launch_bounds__(kOffsetThreads) void batch_offsets_kernel(const BatchItemDev* __restrict__ items, int n_items,
                                                                       int64_t* __restrict__ offsets) {
    __shared__ int64_t s_wave[kOffsetThreads / 64];
    constexpr int kSlots = 3 * kBatchMaxItems / kOffsetThreads;  // of a thread
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int slots = 3 * n_items;
    const int per = (slots + kOffsetThreads - 1) / kOffsetThreads;
    int64_t units[kSlots], sum = 0;
#pragma unroll
    for (int k = 0; k < kSlots; ++k) {
        const int slot = per * static_cast<int>(threadIdx.x) + k;
        units[k] = 0;
        if (k < per && slot < slots) {
            const int type = slot / n_items;
            const BatchItemDev& it = items[slot - type * n_items];
            const CoreBins* bins = type == 0 ? it.pbins : it.sbins;
            units[k] = type == 2 ? (it.n + 63) / 64 : (bins != nullptr ? bins->unit_start[kBins] : 0u);
        }
        sum += units[k];
    }
    int64_t incl = sum;
    for (int d = 1; d < 64; d <<= 1) {
        const int64_t o = __shfl_up(incl, d);
        incl += lane >= d ? o : 0;
    }
    if (lane == 63) {
        s_wave[wave] = incl;
    }
    __syncthreads();
    int64_t run = incl - sum;
    for (int w = 0; w < wave; ++w) {
        run += s_wave[w];
    }
#pragma unroll
    for (int k = 0; k < kSlots; ++k) {
        const int slot = per * static_cast<int>(threadIdx.x) + k;
        if (k < per && slot < slots) {
            offsets[slot] = run;
            run += units[k];
            if (slot == slots - 1) {
                offsets[slots] = run;
            }
        }
    }
}

// One batch application is two persistent launches over the units, the pair units (PART 1), then the
// single and diagonal units (PART 2): each kernel holds only its own unit code, so both keep the
// packed groups within 128 VGPRs (4 waves per SIMD; 3 waves measured ~20% slower).  As one launch
// over all unit types the kernel spilled at that limit and had to walk the 9..32-entry groups one
// per wave (64 molecular instances, forward + backward: 115.0 ms against 108.2 ms split).
__device__ __forceinline__ uint32_t wave_scan(uint32_t v, int lane) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(v, d);
        v += lane >= d ? o : 0u;
    }
    return v;
}

// OWN: every wave numbers the units itself, a lane an instance, and finds a unit's by a ballot, which
// saves the launch of batch_offsets_kernel (3 us; a batch of 200 rows takes 17) but costs the pair units
// of a large batch 2.7% (12 instances, 250,000 rows): for up to kOwnItems instances and kOwnUnits units,
// a pass of some 30 us (16 x 500 rows 18.8 us, 22 with the launch; 64 x 1000 rows 56, 54 with it).
constexpr int kOwnItems = 64;
constexpr int64_t kOwnUnits = 1 << 15;

template <bool ADJ, int NV, int PART, bool OWN>
__global__ __launch_bounds__(kBlock, 4) void batch_kernel(const BatchItemDev* __restrict__ items, const int64_t* __restrict__ offsets,
                                                       int n_items) {
    __shared__ Stage<NV> stages[kWavesPerBlock];
    const int id = threadIdx.x & 63;
    Stage<NV>& stage = stages[threadIdx.x >> 6];
    // the part's units: pair units (PART 1), or `split` single units and then diagonal ones (PART 2)
    uint32_t first_a = 0, first_b = 0, split = 0;
    int64_t first = 0, total;
    if constexpr (OWN) {
        const bool in = id < n_items;
        const BatchItemDev& it = items[in ? id : 0];
        const CoreBins* bins = PART == 1 ? it.pbins : it.sbins;
        const uint32_t a = in && bins != nullptr ? bins->unit_start[kBins] : 0u;
        const uint32_t sum_a = wave_scan(a, id);
        first_a = sum_a - a;
        split = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(sum_a), 63));
        total = split;
        if (PART == 2) {
            const uint32_t b = in ? static_cast<uint32_t>((it.n + 63) / 64) : 0u;
            const uint32_t sum_b = wave_scan(b, id);
            first_b = sum_b - b;
            total += static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(sum_b), 63));
        }
    } else {
        first = PART == 2 ? offsets[n_items] : 0;
        total = offsets[PART == 1 ? n_items : 3 * n_items] - first;
    }
    // as many blocks as there are units for: each XCD then gets an eighth of them
    const uint32_t blocks = total >= static_cast<int64_t>(gridDim.x) * kWavesPerBlock
                                ? gridDim.x
                                : static_cast<uint32_t>((total + kWavesPerBlock - 1) / kWavesPerBlock);
    if (blockIdx.x >= blocks) {
        return;
    }
    const int64_t nwaves = static_cast<int64_t>(blocks) * kWavesPerBlock;
    if constexpr (OWN) {
        for (int64_t u = xcd_wave(blocks, __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6))); u < total; u += nwaves) {
            const bool diagonal = PART == 2 && u >= split;
            // the last instance whose first unit is <= v
            const uint32_t v = static_cast<uint32_t>(u) - (diagonal ? split : 0u);
            const uint32_t from = diagonal ? first_b : first_a;
            const int item = 63 - __builtin_clzll(__ballot(from <= v && id < n_items));
            const int64_t local = v - static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(from), item));
            // made anew for each unit: what every group size derives from the lane would otherwise be computed
            // ahead of the loop (it holds 128 registers and spills)
            int lane = id;
            asm volatile("" : "+v"(lane));
            const int type = PART == 1 ? 0 : (diagonal ? 2 : 1);
            const BatchItemDev& it = items[item];
            if (PART == 1 || it.n_words == 1) {  // the pair units take any width
                batch_unit<1, ADJ, NV, PART>(it, type, local, lane, stage);
            } else {
                batch_unit<2, ADJ, NV, PART>(it, type, local, lane, stage);
            }
        }
    } else {
        const int slots = 3 * n_items;
        const int64_t last = first + total;
        for (int64_t u = first + xcd_wave(blocks, threadIdx.x >> 6); u < last; u += nwaves) {
            // last slot whose first unit is <= u (offsets[slots] > u)
            int lo = 0, hi = slots;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (offsets[mid] <= u) {
                    lo = mid;
                } else {
                    hi = mid;
                }
            }
            const int type = lo / n_items;
            const BatchItemDev& it = items[lo - type * n_items];
            const int64_t local = u - offsets[lo];
            if (PART == 1 || it.n_words == 1) {
                batch_unit<1, ADJ, NV, PART>(it, type, local, id, stage);
            } else {
                batch_unit<2, ADJ, NV, PART>(it, type, local, id, stage);
            }
        }
    }
}

}  // namespace

size_t pairs_bytes(int n_qubytes) {
    Carver cv{nullptr, 0};
    return pairs_layout(cv, n_qubytes, nullptr) == QMB_OK ? cv.off : 0;
}

int pairs_build(int n_qubytes, int particle_cut, const int16_t* site, const uint8_t* kind, const double* coef, int64_t n_terms,
                void* buffer, size_t bytes, qmb_pairs* out, hipStream_t stream) {
    if (particle_cut != 1 && particle_cut != 2) {
        return set_error(QMB_ERR_UNSUPPORTED, "particle_cut must be 1 or 2, got %d", particle_cut);
    }
    Carver cv{static_cast<char*>(buffer), 0};
    qmb_pairs p{};
    QMB_TRY(pairs_layout(cv, n_qubytes, &p));
    if (cv.off > bytes) {
        return set_error(QMB_ERR_WORKSPACE, "pair table buffer too small: need %zu bytes, have %zu", cv.off, bytes);
    }
    p.particle_cut = particle_cut;
    p.bytes = bytes;
    zero_counts_kernel<<<1, 64, 0, stream>>>(p.counts);
    QMB_CHECK_LAUNCH();
    QMB_TRY(launch_zero_f64(p.coef, 2 * p.n_pairs * p.n_pairs, stream));
    QMB_TRY(launch_zero_f64(p.diag, 2 * (1 + p.n_bits + p.n_pairs), stream));
    if (n_terms > 0) {
        pairs_fill_kernel<<<blocks_for(n_terms), kBlock, 0, stream>>>(site, kind, reinterpret_cast<const double2*>(coef), n_terms,
                                                                      particle_cut, p.n_bits, p.n_pairs,
                                                                      reinterpret_cast<double2*>(p.coef),
                                                                      reinterpret_cast<double2*>(p.diag), p.counts);
        QMB_CHECK_LAUNCH();
    }
    *out = p;
    return QMB_OK;
}

int singles_set_real(qmb_singles* singles, int real, hipStream_t stream) {
    if (!singles) {
        return set_error(QMB_ERR_ARGUMENT, "singles must be non-null");
    }
    singles->real = 0;
    if (real) {
        const int64_t nb = singles->n_bits;
        pairs_real_kernel<<<blocks_for(nb * nb), kBlock, 0, stream>>>(reinterpret_cast<const double2*>(singles->a), nb * nb,
                                                                      singles->a_re, singles->counts);
        QMB_CHECK_LAUNCH();
        pairs_real_kernel<<<blocks_for(nb * nb * nb), kBlock, 0, stream>>>(reinterpret_cast<const double2*>(singles->kd),
                                                                           nb * nb * nb, singles->kd_re, singles->counts);
        QMB_CHECK_LAUNCH();
        singles->real = 1;
    }
    return QMB_OK;
}

int pairs_set_real(qmb_pairs* pairs, int real, hipStream_t stream) {
    if (!pairs) {
        return set_error(QMB_ERR_ARGUMENT, "pairs must be non-null");
    }
    pairs->real = 0;
    if (real) {
        const int64_t n = pairs->n_pairs * pairs->n_pairs;
        pairs_real_kernel<<<blocks_for(n), kBlock, 0, stream>>>(reinterpret_cast<const double2*>(pairs->coef), n, pairs->coef_re,
                                                                pairs->counts);
        QMB_CHECK_LAUNCH();
        pairs->real = 1;
    }
    return QMB_OK;
}

size_t cores_bytes(int n_qubytes, int64_t n, int max_occupied, int order) {
    Carver cv{nullptr, 0};
    return cores_layout(cv, n_qubytes, n, max_occupied, order, nullptr, nullptr, nullptr) == QMB_OK ? cv.off : 0;
}

namespace {

int cores_build_small(const qmb_targets* targets, int order, void* scratch, qmb_cores* c, hipStream_t stream) {
    Carver sc{static_cast<char*>(scratch), 0};
    const size_t cap = static_cast<size_t>(c->capacity);
    c->mvals = sc.take<uint64_t>(cap);
    c->glist = sc.take<uint64_t>(cap);
    c->key_bits = kKeyBits;
    auto* glist = reinterpret_cast<uint2*>(c->glist);
    auto go = [&](auto kernel) -> int {
        QMB_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                        static_cast<int>(sizeof(SmallLds))));
        kernel<<<1, kSmallThreads, sizeof(SmallLds), stream>>>(targets->keys, targets->cols, static_cast<int>(c->n), 8 * c->n_qubytes,
                                                               c->per_config, c->keys, c->vals, c->starts, c->counts,
                                                               static_cast<CoreBins*>(c->bins), c->mvals, glist, glist + cap / 2);
        QMB_CHECK_LAUNCH();
        return QMB_OK;
    };
    switch (c->n_words * 2 + (order - 1)) {
        case 2: return go(&cores_small_kernel<1, 1>);
        case 3: return go(&cores_small_kernel<1, 2>);
        case 4: return go(&cores_small_kernel<2, 1>);
        case 5: return go(&cores_small_kernel<2, 2>);
        case 6: return go(&cores_small_kernel<3, 1>);
        case 7: return go(&cores_small_kernel<3, 2>);
        case 8: return go(&cores_small_kernel<4, 1>);
        default: return go(&cores_small_kernel<4, 2>);
    }
}

}  // namespace

int cores_build(const qmb_targets* targets, int max_occupied, int order, void* buffer, size_t bytes, qmb_cores* out,
                hipStream_t stream) {
    if (!targets) {
        return set_error(QMB_ERR_ARGUMENT, "targets must be non-null");
    }
    Carver cv{static_cast<char*>(buffer), 0};
    qmb_cores c{};
    void* scratch = nullptr;
    size_t scratch_bytes = 0;
    QMB_TRY(cores_layout(cv, targets->n_qubytes, targets->n, max_occupied, order, &c, &scratch, &scratch_bytes));
    if (cv.off > bytes) {
        return set_error(QMB_ERR_WORKSPACE, "core index buffer too small: need %zu bytes, have %zu", cv.off, bytes);
    }
    c.bytes = bytes;
    if (c.capacity == 0) {
        cores_init_kernel<<<1, 64, 0, stream>>>(c.counts, 0, nullptr);
        QMB_CHECK_LAUNCH();
    } else if (c.capacity <= kSmallCores) {
        QMB_TRY(cores_build_small(targets, order, scratch, &c, stream));
    } else {
        const size_t cap = static_cast<size_t>(c.capacity);
        Carver sc{static_cast<char*>(scratch), 0};
        // a u64 per entry: the emitted keys (u32) or, packed, the emitted entries
        uint64_t* entries_in = sc.take<uint64_t>(cap);
        uint32_t* keys_in = reinterpret_cast<uint32_t*>(entries_in);
        uint64_t* vals_in = sc.take<uint64_t>(cap);
        uint8_t* flag = sc.take<uint8_t>(cap);
        const int64_t chunks = flag_chunks(c.capacity);
        uint32_t* chunk_heads = sc.take<uint32_t>(static_cast<size_t>(chunks));
        uint32_t* chunk_off = sc.take<uint32_t>(static_cast<size_t>(chunks));
        const int64_t nblk = bin_blocks(c.capacity);
        uint32_t* bin_hist = sc.take<uint32_t>(static_cast<size_t>(kBinRows * nblk + 1));
        uint32_t* bin_scan = sc.take<uint32_t>(static_cast<size_t>(kBinRows * nblk + 1));
        const int n_bits = 8 * c.n_qubytes;
        uint32_t* inv = sc.take<uint32_t>(static_cast<size_t>(n_bits) * n_bits / 2);
        size_t tmp_bytes = scratch_bytes > sc.off + 512 ? scratch_bytes - sc.off - 512 : 0;
        void* tmp = sc.take_bytes(tmp_bytes);
        const unsigned nb = blocks_for(c.n);
        // packed entries (key << 31 | row and pair slot) when row and slot fit in 31 bits: a
        // keys-only sort of one u64 per entry, from entries_in into vals_in
        const bool packed = core_packed(c.n, n_bits, order);
        const int sub_bits = core_sub_bits(n_bits, order);
        auto emit = [&](auto kernel) {
            kernel<<<nb, kBlock, 0, stream>>>(targets->keys, targets->cols, c.n, n_bits, c.per_config, sub_bits, keys_in,
                                              packed ? static_cast<void*>(entries_in) : static_cast<void*>(vals_in), c.counts);
        };
        const int shape = c.n_words * 2 + (order - 1);
        cores_init_kernel<<<blocks_for(static_cast<int64_t>(n_bits) * n_bits), kBlock, 0, stream>>>(c.counts, n_bits,
                                                                                                  packed && order == 2 ? inv : nullptr);
        QMB_CHECK_LAUNCH();
        if (packed) {
            switch (shape) {
                case 2: emit(&core_emit_kernel<1, 1, true>); break;
                case 3: emit(&core_emit_kernel<1, 2, true>); break;
                case 4: emit(&core_emit_kernel<2, 1, true>); break;
                case 5: emit(&core_emit_kernel<2, 2, true>); break;
                case 6: emit(&core_emit_kernel<3, 1, true>); break;
                case 7: emit(&core_emit_kernel<3, 2, true>); break;
                case 8: emit(&core_emit_kernel<4, 1, true>); break;
                default: emit(&core_emit_kernel<4, 2, true>); break;
            }
        } else {
            switch (shape) {
                case 2: emit(&core_emit_kernel<1, 1, false>); break;
                case 3: emit(&core_emit_kernel<1, 2, false>); break;
                case 4: emit(&core_emit_kernel<2, 1, false>); break;
                case 5: emit(&core_emit_kernel<2, 2, false>); break;
                case 6: emit(&core_emit_kernel<3, 1, false>); break;
                case 7: emit(&core_emit_kernel<3, 2, false>); break;
                case 8: emit(&core_emit_kernel<4, 1, false>); break;
                default: emit(&core_emit_kernel<4, 2, false>); break;
            }
        }
        QMB_CHECK_LAUNCH();
        size_t need = tmp_bytes;
        if (packed) {
            QMB_HIP_TRY(rocprim::radix_sort_keys(tmp, need, entries_in, vals_in, static_cast<unsigned>(cap), kPackedBits,
                                                 kPackedBits + kKeyBits, stream));
            auto unpack = [&](auto kernel) {
                kernel<<<blocks_for(c.capacity, kBlock * kFlagUnroll), kBlock, 0, stream>>>(vals_in, c.capacity, flag, chunk_heads, sub_bits,                                                                                         inv, targets->keys, c.keys, c.vals, c.counts);
            };
            switch (shape) {
                case 2: unpack(&core_flag_unpack_kernel<1, 1>); break;
                case 3: unpack(&core_flag_unpack_kernel<1, 2>); break;
                case 4: unpack(&core_flag_unpack_kernel<2, 1>); break;
                case 5: unpack(&core_flag_unpack_kernel<2, 2>); break;
                case 6: unpack(&core_flag_unpack_kernel<3, 1>); break;
                case 7: unpack(&core_flag_unpack_kernel<3, 2>); break;
                case 8: unpack(&core_flag_unpack_kernel<4, 1>); break;
                default: unpack(&core_flag_unpack_kernel<4, 2>); break;
            }
        } else {
            QMB_HIP_TRY(rocprim::radix_sort_pairs(tmp, need, keys_in, c.keys, vals_in, c.vals, static_cast<unsigned>(cap), 0, kKeyBits,
                                                  stream));
            auto flags = [&](auto kernel) {
                kernel<<<blocks_for(c.capacity, kBlock * kFlagUnroll), kBlock, 0, stream>>>(c.keys, c.vals, c.capacity, targets->keys,
                                                                                         flag, chunk_heads, c.counts);
            };
            switch (shape) {
                case 2: flags(&core_flag_kernel<1, 1>); break;
                case 3: flags(&core_flag_kernel<1, 2>); break;
                case 4: flags(&core_flag_kernel<2, 1>); break;
                case 5: flags(&core_flag_kernel<2, 2>); break;
                case 6: flags(&core_flag_kernel<3, 1>); break;
                case 7: flags(&core_flag_kernel<3, 2>); break;
                case 8: flags(&core_flag_kernel<4, 1>); break;
                default: flags(&core_flag_kernel<4, 2>); break;
            }
        }
        QMB_CHECK_LAUNCH();
        if (chunks <= kBlockScanMax) {
            block_scan_kernel<<<1, kBlock, 0, stream>>>(chunk_heads, chunk_off, chunks);
            QMB_CHECK_LAUNCH();
        } else {
            need = tmp_bytes;
            QMB_HIP_TRY(rocprim::exclusive_scan(tmp, need, chunk_heads, chunk_off, 0u, static_cast<size_t>(chunks),
                                                rocprim::plus<uint32_t>(), stream));
        }
        // one wave per flag chunk, as the flag kernel
        core_start_kernel<<<blocks_for(c.capacity, kBlock * kFlagUnroll), kBlock, 0, stream>>>(flag, chunk_off, c.starts, c.counts);
        c.key_bits = kKeyBits;
        QMB_CHECK_LAUNCH();
        // the binned entries and the group list take the place of the sort's buffers, which are no
        // longer read: at most cap / 2 list slots (a slot stands for two or more entries), and as many
        // noted mixed groups behind them
        c.mvals = entries_in;
        c.glist = vals_in;
        auto* bins = static_cast<CoreBins*>(c.bins);
        const bool one_block = kBinRows * nblk + 1 <= kBlockScanMax;
        bin_count_kernel<<<static_cast<unsigned>(nblk), kBlock, 0, stream>>>(c.starts, c.counts, nblk, bin_groups(c.capacity), bin_hist);
        QMB_CHECK_LAUNCH();
        if (!one_block) {
            need = tmp_bytes;
            QMB_HIP_TRY(rocprim::exclusive_scan(tmp, need, bin_hist, bin_scan, 0u, static_cast<size_t>(kBinRows * nblk + 1),
                                                rocprim::plus<uint32_t>(), stream));
        }
        bin_table_kernel<<<1, kBlock, 0, stream>>>(one_block ? bin_hist : nullptr, bin_scan, nblk, order, bins);
        QMB_CHECK_LAUNCH();
        auto* glist = reinterpret_cast<uint2*>(c.glist);
        auto* msplit = glist + cap / 2;
        auto scatter = [&](auto kernel) {
            kernel<<<static_cast<unsigned>(nblk), kBlock, 0, stream>>>(c.starts, c.counts, flag, c.vals, targets->keys, bin_scan, nblk,
                                                                       bin_groups(c.capacity), n_bits, bins, c.mvals, glist, msplit);
        };
        switch (shape) {
            case 2: scatter(&bin_scatter_kernel<1, 1>); break;
            case 3: scatter(&bin_scatter_kernel<1, 2>); break;
            case 4: scatter(&bin_scatter_kernel<2, 1>); break;
            case 5: scatter(&bin_scatter_kernel<2, 2>); break;
            case 6: scatter(&bin_scatter_kernel<3, 1>); break;
            case 7: scatter(&bin_scatter_kernel<3, 2>); break;
            case 8: scatter(&bin_scatter_kernel<4, 1>); break;
            default: scatter(&bin_scatter_kernel<4, 2>); break;
        }
        QMB_CHECK_LAUNCH();
    }
    *out = c;
    return QMB_OK;
}

namespace {

// Persistent waves of a group kernel: enough to fill every CU several times over, never more than the
// entries can need (small sets: a wave per 32 entries).
unsigned group_grid(int64_t capacity) {
    const int64_t want = capacity <= kTinyCores ? 1 : capacity / (32 * kWavesPerBlock) + 1;
    return static_cast<unsigned>(want < 4096 ? want : 4096);
}
unsigned group_block(int64_t capacity) { return capacity <= kTinyCores ? 64u : static_cast<unsigned>(kBlock); }

template <int NV>
int launch_pairs(PairParams p, int64_t capacity, int mode, hipStream_t stream) {
    const unsigned grid = group_grid(capacity);
    if (p.coef_re != nullptr && capacity >= kDenseMin && p.n_pairs <= kDenseSlots) {
        p.dense = 1;
        const auto go = [&](auto kernel) -> int {
            QMB_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, sizeof(DenseLds)));
            kernel<<<256, kDenseThreads, sizeof(DenseLds), stream>>>(p);
            QMB_CHECK_LAUNCH();
            return QMB_OK;
        };
        QMB_TRY(mode == 1 ? go(&pair_dense_kernel<true, NV>) : go(&pair_dense_kernel<false, NV>));
    }
    if (p.coef_re != nullptr) {
        mode == 1 ? pair_kernel<true, true, NV><<<grid, group_block(capacity), 0, stream>>>(p) : pair_kernel<false, true, NV><<<grid, group_block(capacity), 0, stream>>>(p);
    } else {
        mode == 1 ? pair_kernel<true, false, NV><<<grid, group_block(capacity), 0, stream>>>(p) : pair_kernel<false, false, NV><<<grid, group_block(capacity), 0, stream>>>(p);
    }
    QMB_CHECK_LAUNCH();
    return QMB_OK;
}

}  // namespace

int apply_pairs(const qmb_pairs* pairs, const qmb_cores* cores, const qmb_targets* targets, const double* in, double* out,
                int mode, hipStream_t stream) {
    if (!pairs || !cores || !targets) {
        return set_error(QMB_ERR_ARGUMENT, "pairs, cores and targets must be non-null");
    }
    if (pairs->n_qubytes != cores->n_qubytes || cores->n_qubytes != targets->n_qubytes || cores->n != targets->n) {
        return set_error(QMB_ERR_ARGUMENT, "pairs, cores and targets describe different shapes");
    }
    if (mode != 0 && mode != 1) {
        return set_error(QMB_ERR_ARGUMENT, "mode must be 0 (forward) or 1 (adjoint)");
    }
    if (cores->order != 2) {
        return set_error(QMB_ERR_ARGUMENT, "the pair path needs a core index of order 2");
    }
    if (cores->capacity == 0) {
        return QMB_OK;
    }
    PairParams p{};
    p.coef = reinterpret_cast<const double2*>(pairs->coef);
    p.coef_re = pairs->real ? pairs->coef_re : nullptr;
    p.table_counts = pairs->counts;
    p.n_pairs = pairs->n_pairs;
    p.particle_cut = pairs->particle_cut;
    p.mvals = cores->mvals;
    p.glist = reinterpret_cast<const uint2*>(cores->glist);
    p.bins = static_cast<const CoreBins*>(cores->bins);
    p.counts = cores->counts;
    p.in = reinterpret_cast<const double2*>(in);
    p.out = reinterpret_cast<double2*>(out);
    if (cores->n_words > 2) {
        return set_error(QMB_ERR_UNSUPPORTED, "pair path supports n_qubytes <= %d", kMaxPairBytes);
    }
    return launch_pairs<1>(p, cores->capacity, mode, stream);
}

size_t singles_bytes(int n_qubytes) {
    Carver cv{nullptr, 0};
    return singles_layout(cv, n_qubytes, nullptr) == QMB_OK ? cv.off : 0;
}

int singles_build(int n_qubytes, int particle_cut, const int16_t* site, const uint8_t* kind, const double* coef, int64_t n_terms,
                  void* buffer, size_t bytes, qmb_singles* out, hipStream_t stream) {
    if (particle_cut != 1 && particle_cut != 2) {
        return set_error(QMB_ERR_UNSUPPORTED, "particle_cut must be 1 or 2, got %d", particle_cut);
    }
    Carver cv{static_cast<char*>(buffer), 0};
    qmb_singles g{};
    QMB_TRY(singles_layout(cv, n_qubytes, &g));
    if (cv.off > bytes) {
        return set_error(QMB_ERR_WORKSPACE, "single-excitation buffer too small: need %zu bytes, have %zu", cv.off, bytes);
    }
    g.particle_cut = particle_cut;
    g.bytes = bytes;
    const int64_t nb = g.n_bits;
    zero_counts_kernel<<<1, 64, 0, stream>>>(g.counts);
    QMB_CHECK_LAUNCH();
    QMB_TRY(launch_zero_f64(g.a, 2 * nb * nb, stream));
    QMB_TRY(launch_zero_f64(g.kd, 2 * nb * nb * nb, stream));
    if (n_terms > 0) {
        singles_fill_kernel<<<blocks_for(n_terms), kBlock, 0, stream>>>(site, kind, reinterpret_cast<const double2*>(coef), n_terms,
                                                                        particle_cut, g.n_bits, reinterpret_cast<double2*>(g.a),
                                                                        reinterpret_cast<double2*>(g.kd), g.counts);
        QMB_CHECK_LAUNCH();
    }
    *out = g;
    return QMB_OK;
}

int apply_singles(const qmb_singles* singles, const qmb_cores* cores, const qmb_targets* targets, const double* in, double* out,
                  int mode, hipStream_t stream) {
    if (!singles || !cores || !targets) {
        return set_error(QMB_ERR_ARGUMENT, "singles, cores and targets must be non-null");
    }
    if (singles->n_qubytes != cores->n_qubytes || cores->n_qubytes != targets->n_qubytes || cores->n != targets->n) {
        return set_error(QMB_ERR_ARGUMENT, "singles, cores and targets describe different shapes");
    }
    if (cores->order != 1) {
        return set_error(QMB_ERR_ARGUMENT, "the single-excitation path needs a core index of order 1");
    }
    if (mode != 0 && mode != 1) {
        return set_error(QMB_ERR_ARGUMENT, "mode must be 0 (forward) or 1 (adjoint)");
    }
    if (cores->capacity == 0) {
        return QMB_OK;
    }
    SingleParams p{};
    p.a = reinterpret_cast<const double2*>(singles->a);
    p.kd = reinterpret_cast<const double2*>(singles->kd);
    p.a_re = singles->real ? singles->a_re : nullptr;
    p.kd_re = singles->real ? singles->kd_re : nullptr;
    p.n_bits = singles->n_bits;
    p.particle_cut = singles->particle_cut;
    p.ckeys = targets->keys;
    p.mvals = cores->mvals;
    p.glist = reinterpret_cast<const uint2*>(cores->glist);
    p.bins = static_cast<const CoreBins*>(cores->bins);
    p.counts = cores->counts;
    p.in = reinterpret_cast<const double2*>(in);
    p.out = reinterpret_cast<double2*>(out);
    const unsigned grid = group_grid(cores->capacity);
    auto go = [&](auto kernel) -> int {
        kernel<<<grid, group_block(cores->capacity), 0, stream>>>(p);
        QMB_CHECK_LAUNCH();
        return QMB_OK;
    };
    if (cores->n_words == 1) {
        return mode == 1 ? go(&single_kernel<1, true>) : go(&single_kernel<1, false>);
    }
    if (cores->n_words == 2) {
        return mode == 1 ? go(&single_kernel<2, true>) : go(&single_kernel<2, false>);
    }
    return set_error(QMB_ERR_UNSUPPORTED, "single-excitation path supports n_qubytes <= %d", kMaxPairBytes);
}

int apply_diagonal(const qmb_pairs* pairs, const qmb_targets* targets, const double* in, double* out, int mode,
                   hipStream_t stream) {
    if (!pairs || !targets) {
        return set_error(QMB_ERR_ARGUMENT, "pairs and targets must be non-null");
    }
    if (pairs->n_qubytes != targets->n_qubytes) {
        return set_error(QMB_ERR_ARGUMENT, "pairs built for %d bytes, targets for %d", pairs->n_qubytes, targets->n_qubytes);
    }
    if (mode != 0 && mode != 1) {
        return set_error(QMB_ERR_ARGUMENT, "mode must be 0 (forward) or 1 (adjoint)");
    }
    if (targets->n == 0) {
        return QMB_OK;
    }
    const unsigned grid = blocks_for(targets->n);
    const auto* dg = reinterpret_cast<const double2*>(pairs->diag);
    const auto* vi = reinterpret_cast<const double2*>(in);
    auto* vo = reinterpret_cast<double2*>(out);
    const int nb = pairs->n_bits;
    switch (targets->n_words * 2 + mode) {
        case 2: diag_apply_kernel<1, false><<<grid, kBlock, 0, stream>>>(targets->keys, targets->n, dg, nb, vi, vo); break;
        case 3: diag_apply_kernel<1, true><<<grid, kBlock, 0, stream>>>(targets->keys, targets->n, dg, nb, vi, vo); break;
        case 4: diag_apply_kernel<2, false><<<grid, kBlock, 0, stream>>>(targets->keys, targets->n, dg, nb, vi, vo); break;
        default: diag_apply_kernel<2, true><<<grid, kBlock, 0, stream>>>(targets->keys, targets->n, dg, nb, vi, vo); break;
    }
    QMB_CHECK_LAUNCH();
    return QMB_OK;
}

int strings_layout(Carver& cv, int n_qubytes, int64_t n, qmb_strings* out, void** scratch, size_t* scratch_bytes) {
    QMB_TRY(check_qubytes(n_qubytes));
    if (n_qubytes > kMaxPairBytes) {
        return set_error(QMB_ERR_UNSUPPORTED, "the strings index supports n_qubytes <= %d, got %d", kMaxPairBytes, n_qubytes);
    }
    if (n < 0 || n >= (1ll << 31)) {
        return set_error(QMB_ERR_ARGUMENT, "n must be in [0, 2^31), got %lld", static_cast<long long>(n));
    }
    qmb_strings t{};
    t.n_qubytes = n_qubytes;
    t.n_words = n_words_of(n_qubytes);
    t.n = n;
    const size_t cap = static_cast<size_t>(n > 0 ? n : 1);
    t.buffer = cv.base;
    t.counts = cv.take<int64_t>(8);
    t.keys = cv.take<uint32_t>(cap);
    t.rows = cv.take<uint32_t>(cap);
    t.group = cv.take<uint32_t>(cap);
    t.starts = cv.take<uint32_t>(cap + 1);
    t.mrows = cv.take<uint32_t>(cap);
    t.mrange = cv.take<uint32_t>(2 * cap);
    t.mcfg = cv.take<uint64_t>(cap * static_cast<size_t>(t.n_words));
    t.mstr = cv.take<uint64_t>(cap);
    size_t tmp = 0;
    {
        uint32_t* u = nullptr;
        if (rocprim::radix_sort_pairs(nullptr, tmp, u, u, u, u, static_cast<unsigned>(cap), 0, 32) != hipSuccess) {
            return set_error(QMB_ERR_HIP, "rocprim radix_sort_pairs size query failed");
        }
        size_t scan = 0;
        if (rocprim::inclusive_scan(nullptr, scan, u, u, cap, rocprim::plus<uint32_t>()) != hipSuccess) {
            return set_error(QMB_ERR_HIP, "rocprim inclusive_scan size query failed");
        }
        tmp = tmp > scan ? tmp : scan;
        if (rocprim::exclusive_scan(nullptr, scan, u, u, 0u, cap, rocprim::plus<uint32_t>()) != hipSuccess) {
            return set_error(QMB_ERR_HIP, "rocprim exclusive_scan size query failed");
        }
        tmp = tmp > scan ? tmp : scan;
    }
    const size_t s0 = cv.off;
    void* s = cv.take_bytes(4 * cap * sizeof(uint32_t) + tmp + 4096);
    if (scratch) {
        *scratch = s;
    }
    if (scratch_bytes) {
        *scratch_bytes = cv.off - s0;
    }
    t.bytes = cv.off;
    if (out) {
        *out = t;
    }
    return QMB_OK;
}

size_t strings_bytes(int n_qubytes, int64_t n) {
    Carver cv{nullptr, 0};
    return strings_layout(cv, n_qubytes, n, nullptr, nullptr, nullptr) == QMB_OK ? cv.off : 0;
}

int strings_build(const qmb_targets* targets, int parity, void* buffer, size_t bytes, qmb_strings* out, hipStream_t stream) {
    if (!targets || !out) {
        return set_error(QMB_ERR_ARGUMENT, "targets and out must be non-null");
    }
    if (parity != 0 && parity != 1) {
        return set_error(QMB_ERR_ARGUMENT, "parity must be 0 (hops between even sites) or 1 (odd sites), got %d", parity);
    }
    Carver cv{static_cast<char*>(buffer), 0};
    qmb_strings t{};
    void* scratch = nullptr;
    size_t scratch_bytes = 0;
    QMB_TRY(strings_layout(cv, targets->n_qubytes, targets->n, &t, &scratch, &scratch_bytes));
    if (cv.off > bytes) {
        return set_error(QMB_ERR_WORKSPACE, "strings index buffer too small: need %zu bytes, have %zu", cv.off, bytes);
    }
    t.bytes = bytes;
    t.parity = parity;
    QMB_TRY(launch_zero_f64(reinterpret_cast<double*>(t.counts), 8, stream));
    const int64_t n = t.n;
    if (n > 0) {
        const size_t cap = static_cast<size_t>(n);
        Carver sc{static_cast<char*>(scratch), 0};
        uint32_t* keys_in = sc.take<uint32_t>(cap);
        uint32_t* rows_in = sc.take<uint32_t>(cap);
        uint32_t* flag = sc.take<uint32_t>(cap);
        uint32_t* mpos = sc.take<uint32_t>(cap);
        size_t tmp_bytes = scratch_bytes > sc.off + 512 ? scratch_bytes - sc.off - 512 : 0;
        void* tmp = sc.take_bytes(tmp_bytes);
        const unsigned nb = blocks_for(n);
        if (t.n_words == 1) {
            strings_emit_kernel<1><<<nb, kBlock, 0, stream>>>(targets->keys, n, parity, keys_in, rows_in);
        } else {
            strings_emit_kernel<2><<<nb, kBlock, 0, stream>>>(targets->keys, n, parity, keys_in, rows_in);
        }
        QMB_CHECK_LAUNCH();
        size_t need = tmp_bytes;
        QMB_HIP_TRY(rocprim::radix_sort_pairs(tmp, need, keys_in, t.keys, rows_in, t.rows, static_cast<unsigned>(cap), 0, 32, stream));
        key_flag_kernel<<<nb, kBlock, 0, stream>>>(t.keys, n, flag);
        QMB_CHECK_LAUNCH();
        need = tmp_bytes;
        QMB_HIP_TRY(rocprim::inclusive_scan(tmp, need, flag, t.group, cap, rocprim::plus<uint32_t>(), stream));
        strings_start_kernel<<<nb, kBlock, 0, stream>>>(flag, t.group, n, t.starts, t.counts);
        QMB_CHECK_LAUNCH();
        strings_stats_kernel<<<nb < 512u ? nb : 512u, kBlock, 0, stream>>>(t.starts, t.counts);
        QMB_CHECK_LAUNCH();
        strings_multi_kernel<<<nb, kBlock, 0, stream>>>(t.group, t.starts, n, flag);
        QMB_CHECK_LAUNCH();
        need = tmp_bytes;
        QMB_HIP_TRY(rocprim::exclusive_scan(tmp, need, flag, mpos, 0u, cap, rocprim::plus<uint32_t>(), stream));
        auto* mrange = reinterpret_cast<uint2*>(t.mrange);
        if (t.n_words == 1) {
            strings_compact_kernel<1><<<nb, kBlock, 0, stream>>>(targets->keys, t.rows, t.group, t.starts, flag, mpos, n, parity,
                                                                 t.mrows, mrange, t.mcfg, t.mstr, t.counts);
        } else {
            strings_compact_kernel<2><<<nb, kBlock, 0, stream>>>(targets->keys, t.rows, t.group, t.starts, flag, mpos, n, parity,
                                                                 t.mrows, mrange, t.mcfg, t.mstr, t.counts);
        }
        QMB_CHECK_LAUNCH();
        // merged groups (flag is free again: it marks their first entries)
        QMB_TRY(launch_zero_f64(reinterpret_cast<double*>(flag), static_cast<int64_t>((cap + 1) / 2), stream));
        if (t.n_words == 1) {
            strings_mixed_kernel<1><<<nb, kBlock, 0, stream>>>(mrange, t.mcfg, t.counts, parity, flag);
        } else {
            strings_mixed_kernel<2><<<nb, kBlock, 0, stream>>>(mrange, t.mcfg, t.counts, parity, flag);
        }
        QMB_CHECK_LAUNCH();
        strings_mark_kernel<<<nb, kBlock, 0, stream>>>(flag, t.counts, mrange);
        QMB_CHECK_LAUNCH();
    }
    *out = t;
    return QMB_OK;
}

int apply_hops(const qmb_singles* singles, const qmb_strings* strings, const qmb_targets* targets, const double* in, double* out,
               int mode, hipStream_t stream) {
    if (!singles || !strings || !targets || !in || !out) {
        return set_error(QMB_ERR_ARGUMENT, "singles, strings, targets, in and out must be non-null");
    }
    if (singles->n_qubytes != strings->n_qubytes || strings->n_qubytes != targets->n_qubytes || strings->n != targets->n) {
        return set_error(QMB_ERR_ARGUMENT, "singles, strings and targets describe different shapes");
    }
    if (mode != 0 && mode != 1) {
        return set_error(QMB_ERR_ARGUMENT, "mode must be 0 (forward) or 1 (adjoint)");
    }
    if (strings->n == 0) {
        return QMB_OK;
    }
    HopParams p{};
    p.s.a = reinterpret_cast<const double2*>(singles->a);
    p.s.kd = reinterpret_cast<const double2*>(singles->kd);
    p.s.a_re = singles->real ? singles->a_re : nullptr;
    p.s.kd_re = singles->real ? singles->kd_re : nullptr;
    p.s.n_bits = singles->n_bits;
    p.s.particle_cut = singles->particle_cut;
    p.s.ckeys = targets->keys;
    p.s.in = reinterpret_cast<const double2*>(in);
    p.s.out = reinterpret_cast<double2*>(out);
    p.scounts = singles->counts;
    p.sites = parity_sites(strings->parity);
    p.parity = strings->parity;
    p.mrows = strings->mrows;
    p.mrange = reinterpret_cast<const uint2*>(strings->mrange);
    p.mcfg = strings->mcfg;
    p.mstr = strings->mstr;
    p.counts = strings->counts;
    const int64_t want = (strings->n + 64 * 4 - 1) / (64 * 4);
    const unsigned grid = static_cast<unsigned>(want < 8192 ? (want < 1 ? 1 : want) : 8192);
    auto go = [&](auto kernel) -> int {
        kernel<<<grid, kBlock, 0, stream>>>(p);
        QMB_CHECK_LAUNCH();
        return QMB_OK;
    };
    if (strings->n_words == 1) {
        return mode == 1 ? go(&hop_kernel<1, true>) : go(&hop_kernel<1, false>);
    }
    return mode == 1 ? go(&hop_kernel<2, true>) : go(&hop_kernel<2, false>);
}

int apply_structured_dual(const qmb_pairs* pairs, const qmb_singles* singles, const qmb_cores* cores2, const qmb_cores* cores1,
                          const qmb_targets* targets, const double* in, double* out, const double* in2, double* out2, int mode,
                          hipStream_t stream) {
    if (mode != 0 && mode != 1) {
        return set_error(QMB_ERR_ARGUMENT, "mode must be 0 (forward) or 1 (adjoint)");
    }
    if (!pairs || !cores2 || !targets || !in || !out || !in2 || !out2 || (singles && !cores1)) {
        return set_error(QMB_ERR_ARGUMENT, "pairs, cores2, targets, the four vectors (and cores1 with singles) must be non-null");
    }
    if (pairs->n_qubytes != targets->n_qubytes || cores2->n != targets->n || cores2->order != 2 ||
        (singles && (cores1->n != targets->n || cores1->order != 1 || singles->n_qubytes != targets->n_qubytes))) {
        return set_error(QMB_ERR_ARGUMENT, "pairs, singles, cores and targets describe different shapes");
    }
    if (targets->n == 0) {
        return QMB_OK;
    }
    const int W = targets->n_words;
    if (W != 1 && W != 2) {
        return set_error(QMB_ERR_UNSUPPORTED, "the structured path supports n_qubytes <= %d", kMaxPairBytes);
    }
    const auto* vi = reinterpret_cast<const double2*>(in);
    const auto* vi2 = reinterpret_cast<const double2*>(in2);
    auto* vo = reinterpret_cast<double2*>(out);
    auto* vo2 = reinterpret_cast<double2*>(out2);
    const auto* dg = reinterpret_cast<const double2*>(pairs->diag);
    const unsigned dgrid = blocks_for(targets->n);
    if (W == 1) {
        if (mode == 1) {
            diag_apply2_kernel<1, true><<<dgrid, kBlock, 0, stream>>>(targets->keys, targets->n, dg, pairs->n_bits, vi, vo, vi2, vo2);
        } else {
            diag_apply2_kernel<1, false><<<dgrid, kBlock, 0, stream>>>(targets->keys, targets->n, dg, pairs->n_bits, vi, vo, vi2, vo2);
        }
    } else if (mode == 1) {
        diag_apply2_kernel<2, true><<<dgrid, kBlock, 0, stream>>>(targets->keys, targets->n, dg, pairs->n_bits, vi, vo, vi2, vo2);
    } else {
        diag_apply2_kernel<2, false><<<dgrid, kBlock, 0, stream>>>(targets->keys, targets->n, dg, pairs->n_bits, vi, vo, vi2, vo2);
    }
    QMB_CHECK_LAUNCH();
    if (singles && cores1->capacity > 0) {
        SingleParams p{};
        p.a = reinterpret_cast<const double2*>(singles->a);
        p.kd = reinterpret_cast<const double2*>(singles->kd);
        p.a_re = singles->real ? singles->a_re : nullptr;
        p.kd_re = singles->real ? singles->kd_re : nullptr;
        p.n_bits = singles->n_bits;
        p.particle_cut = singles->particle_cut;
        p.ckeys = targets->keys;
        p.mvals = cores1->mvals;
        p.glist = reinterpret_cast<const uint2*>(cores1->glist);
        p.bins = static_cast<const CoreBins*>(cores1->bins);
        p.counts = cores1->counts;
        p.in = vi;
        p.out = vo;
        p.in2 = vi2;
        p.out2 = vo2;
        const unsigned grid = group_grid(cores1->capacity);
        if (W == 1) {
            mode == 1 ? single_kernel<1, true, 2><<<grid, group_block(cores1->capacity), 0, stream>>>(p) : single_kernel<1, false, 2><<<grid, group_block(cores1->capacity), 0, stream>>>(p);
        } else {
            mode == 1 ? single_kernel<2, true, 2><<<grid, group_block(cores1->capacity), 0, stream>>>(p) : single_kernel<2, false, 2><<<grid, group_block(cores1->capacity), 0, stream>>>(p);
        }
        QMB_CHECK_LAUNCH();
    }
    if (cores2->capacity > 0) {
        PairParams p{};
        p.coef = reinterpret_cast<const double2*>(pairs->coef);
        p.coef_re = pairs->real ? pairs->coef_re : nullptr;
        p.table_counts = pairs->counts;
        p.n_pairs = pairs->n_pairs;
        p.particle_cut = pairs->particle_cut;
        p.mvals = cores2->mvals;
        p.glist = reinterpret_cast<const uint2*>(cores2->glist);
        p.bins = static_cast<const CoreBins*>(cores2->bins);
        p.counts = cores2->counts;
        p.in = vi;
        p.out = vo;
        p.in2 = vi2;
        p.out2 = vo2;
        QMB_TRY(launch_pairs<2>(p, cores2->capacity, mode, stream));
    }
    return QMB_OK;
}

int batch_layout(Carver& cv, int n_items, qmb_batch* out) {
    if (n_items < 1 || n_items > kBatchMaxItems) {
        return set_error(QMB_ERR_ARGUMENT, "n_items must be in [1, %d], got %d", kBatchMaxItems, n_items);
    }
    qmb_batch b{};
    b.n_items = n_items;
    b.buffer = cv.base;
    b.items = cv.take<BatchItemDev>(static_cast<size_t>(n_items));
    b.offsets = cv.take<int64_t>(3 * static_cast<size_t>(n_items) + 1);
    b.bytes = cv.off;
    if (out) {
        *out = b;
    }
    return QMB_OK;
}

// Units that the bins of an index of this capacity can make up: none but a bin's last covers fewer than 32
// entries (a group of 65 entries is two; a unit of the split bin is 16 slots of two entries).
inline int64_t unit_bound(int64_t capacity) { return capacity > 0 ? capacity / 32 + kBins : 0; }

size_t batch_bytes(int n_items) {
    Carver cv{nullptr, 0};
    return batch_layout(cv, n_items, nullptr) == QMB_OK ? cv.off : 0;
}

int batch_plan(const qmb_batch_item* items, int n_items, void* buffer, size_t bytes, qmb_batch* out, hipStream_t stream) {
    Carver cv{static_cast<char*>(buffer), 0};
    qmb_batch b{};
    QMB_TRY(batch_layout(cv, n_items, &b));
    if (cv.off > bytes) {
        return set_error(QMB_ERR_WORKSPACE, "batch buffer too small: need %zu bytes, have %zu", cv.off, bytes);
    }
    b.bytes = bytes;
    std::vector<BatchItemDev> dev(static_cast<size_t>(n_items));
    int dual = 0;
    for (int k = 0; k < n_items; ++k) {
        const qmb_batch_item& x = items[k];
        if (!x.pairs || !x.targets) {
            return set_error(QMB_ERR_ARGUMENT, "item %d: pairs and targets must be non-null", k);
        }
        const qmb_targets& tg = *x.targets;
        if (x.pairs->n_qubytes != tg.n_qubytes || tg.n_words > 2) {
            return set_error(QMB_ERR_ARGUMENT, "item %d: pairs / targets shapes differ or n_qubytes > 16", k);
        }
        if (tg.n > 0 && (!x.in || !x.out)) {
            return set_error(QMB_ERR_ARGUMENT, "item %d: in and out must be non-null", k);
        }
        if ((x.pairs && (!x.cores2 || x.cores2->order != 2 || x.cores2->n != tg.n || x.pairs->n_qubytes != tg.n_qubytes)) ||
            (x.singles && (!x.cores1 || x.cores1->order != 1 || x.cores1->n != tg.n || x.singles->n_qubytes != tg.n_qubytes))) {
            return set_error(QMB_ERR_ARGUMENT, "item %d: pair / single tables need matching core indexes of order 2 / 1", k);
        }
        BatchItemDev d{};
        d.n_words = tg.n_words;
        d.particle_cut = x.pairs->particle_cut;
        d.n_bits = 8 * tg.n_qubytes;
        d.n = tg.n;
        d.ckeys = tg.keys;
        d.diag = reinterpret_cast<const double2*>(x.pairs->diag);
        if (x.pairs) {
            d.has_pairs = 1;
            d.pcoef = reinterpret_cast<const double2*>(x.pairs->coef);
            d.pcoef_re = x.pairs->real ? x.pairs->coef_re : nullptr;
            d.n_pairs = x.pairs->n_pairs;
            d.pmvals = x.cores2->mvals;
            d.pglist = reinterpret_cast<const uint2*>(x.cores2->glist);
            d.pbins = x.cores2->capacity > 0 ? static_cast<const CoreBins*>(x.cores2->bins) : nullptr;
            d.pcounts = x.cores2->counts;
            b.total_units += unit_bound(x.cores2->capacity);
        }
        if (x.singles) {
            d.has_singles = 1;
            d.sa = reinterpret_cast<const double2*>(x.singles->a);
            d.skd = reinterpret_cast<const double2*>(x.singles->kd);
            d.sa_re = x.singles->real ? x.singles->a_re : nullptr;
            d.skd_re = x.singles->real ? x.singles->kd_re : nullptr;
            d.smvals = x.cores1->mvals;
            d.sglist = reinterpret_cast<const uint2*>(x.cores1->glist);
            d.sbins = x.cores1->capacity > 0 ? static_cast<const CoreBins*>(x.cores1->bins) : nullptr;
            d.scounts = x.cores1->counts;
            b.total_units += unit_bound(x.cores1->capacity);
        }
        b.total_units += (tg.n + 63) / 64;
        d.in = reinterpret_cast<const double2*>(x.in);
        d.out = reinterpret_cast<double2*>(x.out);
        d.in2 = reinterpret_cast<const double2*>(x.in2);
        d.out2 = reinterpret_cast<double2*>(x.out2);
        const int two = (x.in2 != nullptr && x.out2 != nullptr) ? 1 : 0;
        if ((x.in2 != nullptr) != (x.out2 != nullptr) || (k > 0 && two != dual)) {
            return set_error(QMB_ERR_ARGUMENT, "item %d: in2 and out2 must be given together, for every item or none", k);
        }
        dual = two;
        dev[static_cast<size_t>(k)] = d;
    }
    b.dual = dual;
    QMB_HIP_TRY(hipMemcpyAsync(b.items, dev.data(), dev.size() * sizeof(BatchItemDev), hipMemcpyHostToDevice, stream));
    // the host table above goes out of scope on return
    QMB_HIP_TRY(hipStreamSynchronize(stream));
    *out = b;
    return QMB_OK;
}

int apply_batch(const qmb_batch* batch, int mode, int waves, hipStream_t stream) {
    if (!batch) {
        return set_error(QMB_ERR_ARGUMENT, "batch must be non-null");
    }
    if (mode != 0 && mode != 1) {
        return set_error(QMB_ERR_ARGUMENT, "mode must be 0 (forward) or 1 (adjoint)");
    }
    if (batch->total_units == 0) {
        return QMB_OK;
    }
    int64_t w = waves > 0 ? waves : 8192;
    w = w < 4 ? 4 : w;
    int64_t blocks = (w + 3) / 4;
    const int64_t need = (batch->total_units + 3) / 4;
    blocks = blocks < need ? blocks : need;
    const auto* items = static_cast<const BatchItemDev*>(batch->items);
    const unsigned g = static_cast<unsigned>(blocks);
    const bool own = batch->n_items <= kOwnItems && batch->total_units <= kOwnUnits;
    if (!own) {
        batch_offsets_kernel<<<1, kOffsetThreads, 0, stream>>>(items, batch->n_items, batch->offsets);
        QMB_CHECK_LAUNCH();
    }
    const auto both = [&](auto pair_units, auto other_units) -> int {
        pair_units<<<g, kBlock, 0, stream>>>(items, batch->offsets, batch->n_items);
        QMB_CHECK_LAUNCH();
        other_units<<<g, kBlock, 0, stream>>>(items, batch->offsets, batch->n_items);
        QMB_CHECK_LAUNCH();
        return QMB_OK;
    };
    const auto go = [&](auto wave_numbers) -> int {
        constexpr bool O = decltype(wave_numbers)::value;
        if (batch->dual) {
            return mode == 1 ? both(&batch_kernel<true, 2, 1, O>, &batch_kernel<true, 2, 2, O>)
                             : both(&batch_kernel<false, 2, 1, O>, &batch_kernel<false, 2, 2, O>);
        }
        return mode == 1 ? both(&batch_kernel<true, 1, 1, O>, &batch_kernel<true, 1, 2, O>)
                         : both(&batch_kernel<false, 1, 1, O>, &batch_kernel<false, 1, 2, O>);
    };
    return own ? go(std::true_type{}) : go(std::false_type{});
}

}  // namespace qmb
