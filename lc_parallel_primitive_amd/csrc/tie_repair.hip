// tie_repair.hip — the low digits of 8-byte key sorts, without passes of their
// own.
//
// Reference: device/device_radix_sort.h:187-378 runs a pass for every digit.
//
// MI355X design: a pass over 8-byte keys moves 16 bytes and more per key
// whether or not it still changes the order.  Once keys are sorted by their
// upper digits, those that tie are few and lie side by side wherever the keys
// are spread out (2^23.5 uniform keys: after the top 24 bits every second key
// has a neighbour of equal upper bits, after the top 32 bits one in 360).  So
// the sort stops after the digits that a sample of the keys and the counts of
// their digits ask for (rs_sample and rs_cut_digits in the histogram launch,
// radix_sort.hip) and this kernel orders what ties: one read of the keys, and
// writes where something moves.
//  * A 256-thread workgroup owns the runs that begin in its 2048 keys; 64 more
//    keys cover the runs that begin last.  One bit per key says whether a run
//    begins there and one whether the key ranks below the one before it; with
//    none of the latter every run is in order (equal keys are) and nothing is
//    left to do.  Else the keys that tie with a neighbour are listed; those of a
//    run of up to 32 keys that is not in order count their places in LDS, and
//    those that move are written with their values.
//  * The keys of longer runs that are not in order are ranked against each other
//    by the whole workgroup, up to 256 of them; more are sorted digit by digit
//    between the output and the scratch, by the one workgroup, at a cost linear in
//    their number.
//  * A run that goes on past the 64 keys is followed to its end, and sorted by
//    digits if it is not in order.  Such a run of 60000 among 2^27 keys, u32 values,
//    adds 1270 us to a sort of 3530, one of 5000 among 12 * 10^6 170 to 300.
//    rs_cut_digits bounds it: 1 / 227 of the keys at the most, and n / 2048 and the
//    scatter of even counts where the other keys are spread evenly.
// What bounds it is the read of the keys, and the writes of those that move: 12 *
// 10^6 u64 keys with u32 values, us, after 32 / 24 upper bits: 37 / 75 (one
// thread per run, by insertion in LDS: - / 93; every key looking for its place,
// unlisted: - / 80).  The whole sort: 540 -> 305 us, of u64 keys alone 10^6:
// 125 -> 78; keys that come ten times each 559 -> 330, 60 times 653 -> 304 (with
// every key walking along its run, and the workgroup along each of more than 32:
// 440 and 1135).
// A neighbouring workgroup may read keys of a run while its owner moves them;
// it looks at the upper bits alone, and those are the same wherever they go.
#include "tie_repair.hpp"

namespace lcpp {
namespace {

constexpr int kTrBlock = 256;
constexpr int kTrWaves = kTrBlock / kWave;
constexpr uint32_t kTrTile = 2048, kTrHalo = 64, kTrCap = kTrTile + kTrHalo;
constexpr uint32_t kTrShort = 32;  // longest run whose keys find their places by themselves
constexpr int kTrItems = (int)ceil_div(kTrCap, kTrBlock);
constexpr int kTrWords = kTrItems * kTrWaves;  // bit words, of the 64 keys that a wave holds in one register
// Longest run that the workgroup ranks (L * L / 256 steps of 35 ns); longer ones, and
// those that go on past the halo, are sorted digit by digit (some 40 us, mostly
// beside other workgroups' tiles).  A sort with one run of L among uniform keys, us,
// ranked / by digits: 10^6 u64, L = 300 100 / 90, 600 140 / 92 (79 without); 12 * 10^6
// u64 -> u32 pairs, L = 600 382 / 334, 2100 947 / 340 (300 without).
constexpr uint32_t kTrRanked = 256;
constexpr int kTrRankedItems = kTrRanked / kTrBlock;
constexpr int kTrRadixItems = 4;  // per thread and step of a run sorted by digits
constexpr int kTrFarLoads = 4;    // per thread and step along a run past the halo
// Most workgroups launched per CU; beyond them each takes several tiles.  A sort
// whose digits all have passes pays for this launch's empty workgroups (2^27 u64
// keys of 16 low bits, u32 values: 1673 us with one per tile, 65536 of them, 1661
// with 16384, 1659 with 8192), one that has ties to repair for tiles that
// wait for each other (uniform keys: 3580 / 3578 / 3600; 7 per CU: 3874).
constexpr uint32_t kTrPerCu = 64;
static_assert(kTrHalo > kTrShort, "a run that leaves the halo is longer than kTrShort");

// The LDS of a workgroup.  (The counters of a run sorted digit by digit lie where
// the keys were: 22 KiB, seven workgroups per CU.)
struct TrSmem {
    union {
        uint64_t key[kTrCap];
        struct {
            uint32_t wcnt[kTrWaves][256], dbase[256], wsum[kTrWaves];
        } digit;
    };
    uint16_t place[kTrWaves][kTrItems * kWave];
    uint64_t heads[kTrWords], downs[kTrWords];
    uint32_t longs[kTrTile / kTrShort];  // begin | end << 16
    uint32_t nlong, any_down, end, flag;
};

// Keys [0, L), which tie from bit `cut` on, sorted by the bits below, stably,
// between `keys` and `ktmp`; vals move along.  Every thread of the workgroup calls
// it.
template <class UV, bool PAIRS, bool ZEROS>
__device__ __forceinline__ void tr_by_digits(uint64_t *keys, UV *vals, uint64_t *ktmp, UV *vtmp, uint32_t L,
                                             const KeyCode<uint64_t, ZEROS> &code, uint32_t cut, uint32_t tid,
                                             TrSmem &sm)
{
    const uint32_t lane = tid % kWave, wave = tid / kWave;
    // kTrBlock * kTrRadixItems keys at a time (items of a wave are consecutive:
    // ranked by ballot match, stable)
    auto &wcnt = sm.digit.wcnt;
    uint32_t *dbase = sm.digit.dbase, *wsum = sm.digit.wsum;
    uint64_t *ka = keys, *kb = ktmp;
    UV *va = vals, *vb = vtmp;
#pragma unroll 1
    for (uint32_t shift = 0; shift < cut; shift += 8) {
        __syncthreads();
        dbase[tid] = 0;
        if (tid == 0) sm.flag = 0;
        __syncthreads();
        for (uint32_t i = tid; i < L; i += kTrBlock) atomicAdd(&dbase[code.digit(code.in(ka[i]), shift)], 1u);
        __syncthreads();
        const uint32_t c = dbase[tid];
        if (c == L) sm.flag = 1;
        uint32_t ex = wave_inclusive_scan(c, SumOp());
        if (lane == kWave - 1) wsum[wave] = ex;
        ex -= c;
        __syncthreads();
        for (uint32_t w = 0; w < wave; ++w) ex += wsum[w];
        const bool same = sm.flag != 0;
        dbase[tid] = ex;
        if (same) continue;  // one digit for all: nothing moves
        for (uint32_t s0 = 0; s0 < L; s0 += kTrBlock * kTrRadixItems) {
            for (uint32_t i = tid; i < kTrWaves * 256u; i += kTrBlock) (&wcnt[0][0])[i] = 0;
            __syncthreads();
            uint64_t kk[kTrRadixItems];
            UV w[kTrRadixItems];
            uint32_t r[kTrRadixItems], d[kTrRadixItems];
            const uint32_t p = s0 + wave * (kWave * kTrRadixItems) + lane;
#pragma unroll
            for (int u = 0; u < kTrRadixItems; ++u) {
                const bool ok = p + u * kWave < L;
                kk[u] = ok ? ka[p + u * kWave] : 0;
                if constexpr (PAIRS) w[u] = ok ? va[p + u * kWave] : UV(0);
                d[u] = code.digit(code.in(kk[u]), shift);
                const uint64_t peers = match_any8(d[u]) & ballot(ok);
                const uint32_t below = mask_rank(peers);
                uint32_t b = 0;
                if (ok && below == 0) b = atomicAdd(&wcnt[wave][d[u]], (uint32_t)__builtin_popcountll(peers));
                r[u] = (uint32_t)__shfl((int)b, ok ? (int)__builtin_ctzll(peers) : 0) + below;
            }
            __syncthreads();
            uint32_t at = dbase[tid];
#pragma unroll
            for (int x = 0; x < kTrWaves; ++x) {
                const uint32_t cc = wcnt[x][tid];
                wcnt[x][tid] = at;
                at += cc;
            }
            dbase[tid] = at;
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kTrRadixItems; ++u) {
                if (p + u * kWave < L) {
                    const uint32_t at = wcnt[wave][d[u]] + r[u];
                    kb[at] = kk[u];
                    if constexpr (PAIRS) vb[at] = w[u];
                }
            }
            __syncthreads();
        }
        uint64_t *kx = ka;
        ka = kb;
        kb = kx;
        UV *vx = va;
        va = vb;
        vb = vx;
    }
    __syncthreads();
    if (ka != keys) {
        for (uint32_t i = tid; i < L; i += kTrBlock) {
            keys[i] = ka[i];
            if constexpr (PAIRS) vals[i] = va[i];
        }
    }
}

// The runs that begin in keys [base, base + kTrTile).  Every thread of the
// workgroup calls it.
template <class UV, bool PAIRS, bool ZEROS>
__device__ __forceinline__ void tr_tile(uint64_t *keys, UV *vals, uint64_t *ktmp, UV *vtmp, uint32_t n,
                                        const KeyCode<uint64_t, ZEROS> &code, uint32_t cut, uint32_t base, TrSmem &sm)
{
    uint64_t *sk = sm.key, *heads = sm.heads, *downs = sm.downs;
    uint32_t tid = threadIdx.x;
    // (opaque: what is computed from it is not kept in registers from tile to tile)
    asm volatile("" : "+v"(tid));
    const uint32_t lane = tid % kWave, wave = tid / kWave;
    uint16_t *place = sm.place[wave];
    const uint32_t m = n - base < kTrCap ? n - base : kTrCap;     // keys in LDS
    const uint32_t own = n - base < kTrTile ? n - base : kTrTile;  // those whose runs are this workgroup's
    auto top = [&](uint64_t t) { return code.ranked(t) >> cut; };

    if (tid == 0) sm.nlong = sm.any_down = 0;
    uint64_t k[kTrItems];
#pragma unroll
    for (int u = 0; u < kTrItems; ++u) {
        const uint32_t i = tid + u * kTrBlock;
        k[u] = i < m ? code.in(keys[base + i]) : 0;
    }
    const uint64_t before = base ? top(code.in(keys[base - 1])) : 0;
#pragma unroll
    for (int u = 0; u < kTrItems; ++u) {
        const uint32_t i = tid + u * kTrBlock;
        if (i < m) sk[i] = k[u];
    }
    __syncthreads();

    // bit i of heads: a run begins at key i (or i is past the last key); of
    // downs: key i ties with the one before it and ranks below it.  (What key 0
    // is to the one before it matters to that one's workgroup alone.)
#pragma unroll
    for (int u = 0; u < kTrItems; ++u) {
        const uint32_t w = u * kTrWaves + wave, i = w * kWave + lane;
        const uint64_t l = wave_shr1(k[u], sk[w > 0 && w * kWave < m ? w * kWave - 1 : 0]);
        const bool head = i >= m || (i > 0 ? top(l) != top(k[u]) : base == 0 || before != top(k[u]));
        const uint64_t hw = ballot(head);
        const uint64_t dw = ballot(!head && i > 0 && code.ranked(l) > code.ranked(k[u]));
        if (lane == 0) {
            heads[w] = hw;
            downs[w] = dw;
            if (dw) sm.any_down = 1;
        }
    }
    __syncthreads();
    // where the run of key i begins (~0u: before the tile)
    auto begin_of = [&](uint32_t i) {
        uint32_t w = i / kWave;
        uint64_t x = heads[w] & (~0ull >> (kWave - 1 - i % kWave));
        while (x == 0 && w > 0) x = heads[--w];
        return x ? w * kWave + (uint32_t)(kWave - 1 - __builtin_clzll(x)) : ~0u;
    };
    // the run that holds the last key in LDS may go on
    const uint32_t last = begin_of(m - 1);
    const bool open = last < own && base + m < n;
    if (!sm.any_down && !open) return;  // every run is in order (the same for the whole workgroup)

    // the wave's keys that tie with a neighbour, listed: lane u counts those of its
    // u-th word
    uint64_t tied = 0;
    if (lane < (uint32_t)kTrItems) {
        const uint32_t w = lane * kTrWaves + wave;
        tied = ~heads[w] | ~heads[w] >> 1 | (w + 1 < (uint32_t)kTrWords ? ~heads[w + 1] << (kWave - 1) : 0ull);
    }
    const uint32_t upto = wave_inclusive_scan((uint32_t)__builtin_popcountll(tied), SumOp());
    const uint32_t ties = read_lane(upto, kWave - 1);
#pragma unroll
    for (int u = 0; u < kTrItems; ++u) {
        const uint64_t who = read_lane(tied, u);
        const uint32_t at = read_lane(upto, u) - (uint32_t)__builtin_popcountll(who) + mask_rank(who);
        if (who >> lane & 1u) place[at] = (uint16_t)((u * kTrWaves + wave) * kWave + lane);
    }
    wave_lds_sync();
    // each key of a run that is not in order finds its place in it
    uint32_t to[kTrItems];
    UV v[PAIRS ? kTrItems : 1];
#pragma unroll
    for (int u = 0; u < kTrItems; ++u) {
        to[u] = ~0u;
        const uint32_t q = lane + u * kWave;
        if (q >= ties) continue;
        const uint32_t i = place[q];
        const uint32_t first = begin_of(i);
        // the run is another workgroup's, or goes on past the halo
        if (first >= own || (open && first == last)) continue;
        uint32_t w = first / kWave;
        uint64_t x = heads[w] & (~1ull << first % kWave), d = downs[w] & (~1ull << first % kWave), down = 0;
        for (; x == 0; x = heads[++w], d = downs[w]) down |= d;
        const uint32_t end = w * kWave + (uint32_t)__builtin_ctzll(x);  // (key m counts as a head)
        down |= d & ~(~0ull << end % kWave);
        if (down == 0) continue;
        if (end - first > kTrShort) {
            if (i == first) sm.longs[atomicAdd(&sm.nlong, 1u)] = first | end << 16;
            continue;
        }
        k[u] = sk[i];
        const uint64_t rank = code.ranked(k[u]);
        uint32_t r = first;
        for (uint32_t j = first; j < end; ++j) {
            const uint64_t y = code.ranked(sk[j]);
            r += y < rank || (y == rank && j < i) ? 1u : 0u;
        }
        if (r == i) continue;  // in its place
        to[u] = r;
        if constexpr (PAIRS) v[u] = vals[base + i];
    }
    __syncthreads();  // every key and value that moves has been read
#pragma unroll
    for (int u = 0; u < kTrItems; ++u) {
        if (to[u] != ~0u) {
            keys[base + to[u]] = code.out(k[u]);
            if constexpr (PAIRS) vals[base + to[u]] = v[u];
        }
    }

    // the longer ones, one after the other
    const uint32_t runs = sm.nlong;
    const uint64_t open_top = top(sk[last < m ? last : 0]);
    uint16_t *rank = &sm.place[0][0];
#pragma unroll 1
    for (uint32_t q = 0; q < runs; ++q) {
        const uint32_t b = sm.longs[q] & 0xFFFFu, L = (sm.longs[q] >> 16) - b, g = base + b;
        if (L > kTrRanked) continue;
        __syncthreads();  // `rank` is free
        // each key counts those that go before it
#pragma unroll 1
        for (uint32_t i = tid; i < L; i += kTrBlock) {
            const uint64_t x = code.ranked(sk[b + i]);
            uint32_t r = 0;
#pragma unroll 4
            for (uint32_t j = 0; j < L; ++j) {
                const uint64_t y = code.ranked(sk[b + j]);
                r += y < x || (y == x && j < i) ? 1u : 0u;
            }
            rank[i] = (uint16_t)r;
        }
        if constexpr (PAIRS) {
#pragma unroll
            for (int u = 0; u < kTrRankedItems; ++u) {
                const uint32_t i = tid + u * kTrBlock;
                if (i < L) v[u] = vals[g + i];
            }
            __syncthreads();  // every value has been read
        }
#pragma unroll
        for (int u = 0; u < kTrRankedItems; ++u) {
            const uint32_t i = tid + u * kTrBlock;
            if (i < L) {  // (a thread reads the ranks that it wrote)
                keys[g + rank[i]] = code.out(sk[b + i]);
                if constexpr (PAIRS) vals[g + rank[i]] = v[u];
            }
        }
    }
#pragma unroll 1
    for (uint32_t q = 0; q < runs + (open ? 1u : 0u); ++q) {
        uint32_t L, g;
        if (q < runs) {
            g = base + (sm.longs[q] & 0xFFFFu);
            L = base + (sm.longs[q] >> 16) - g;
            if (L <= kTrRanked) continue;
        } else {
            g = base + last;
            // the first position past the run
            uint32_t end = base + m;
            for (;; end += kTrBlock * kTrFarLoads) {
                __syncthreads();
                if (tid == 0) sm.end = ~0u;
                __syncthreads();
                uint32_t past = ~0u;
#pragma unroll
                for (int u = kTrFarLoads - 1; u >= 0; --u) {
                    const uint32_t i = end + u * kTrBlock + tid;
                    if (i >= n || top(code.in(keys[i])) != open_top) past = u * kTrBlock + tid;
                }
                if (past != ~0u) atomicMin(&sm.end, past);
                __syncthreads();
                if (sm.end != ~0u) break;
            }
            end += sm.end;
            L = end - g;
            __syncthreads();
            if (tid == 0) sm.flag = 0;
            __syncthreads();
            bool down = false;
#pragma unroll 4
            for (uint32_t i = tid; i + 1 < L; i += kTrBlock)
                down |= code.ranked(code.in(keys[g + i])) > code.ranked(code.in(keys[g + i + 1]));
            if (down) sm.flag = 1;
            __syncthreads();
            if (!sm.flag) return;  // the same for the whole workgroup
        }
        tr_by_digits<UV, PAIRS>(keys + g, PAIRS ? vals + g : nullptr, ktmp + g, PAIRS ? vtmp + g : nullptr, L, code, cut,
                                tid, sm);
    }
}

template <class UV, bool PAIRS, bool ZEROS>
__global__ __launch_bounds__(kTrBlock) void tie_repair_kernel(uint64_t *keys, UV *vals, uint64_t *ktmp, UV *vtmp,
                                                              uint32_t n, KeyCode<uint64_t, ZEROS> code,
                                                              const uint32_t *__restrict__ cut_word)
{
    __shared__ TrSmem sm;
    const uint32_t cut = __builtin_amdgcn_readfirstlane(*cut_word);
    if (cut == 0) return;
    for (uint64_t base = (uint64_t)blockIdx.x * kTrTile; base < n; base += (uint64_t)gridDim.x * kTrTile) {
        tr_tile<UV, PAIRS>(keys, vals, ktmp, vtmp, n, code, cut, (uint32_t)base, sm);
        __syncthreads();  // the LDS is free
    }
}

template <class UV, bool PAIRS>
int tr_run(int kind, bool desc, void *keys, void *vals, void *ktmp, void *vtmp, uint32_t n, const uint32_t *cut,
           hipStream_t s)
{
    const uint32_t tiles = (uint32_t)ceil_div(n, kTrTile), most = kTrPerCu * (uint32_t)device_cus();
    const uint32_t grid = (uint32_t)ceil_div(tiles, ceil_div(tiles, most));  // as many tiles for each
    auto go = [&](auto zeros) {
        constexpr bool Z = decltype(zeros)::value;
        LCPP_LAUNCH("rs_tie_repair", s,
                    (tie_repair_kernel<UV, PAIRS, Z><<<grid, kTrBlock, 0, s>>>(
                        static_cast<uint64_t *>(keys), static_cast<UV *>(vals), static_cast<uint64_t *>(ktmp),
                        static_cast<UV *>(vtmp), n, KeyCode<uint64_t, Z>::of(kind, desc), cut)));
    };
    if (kind == kFloat) go(std::true_type{});
    else go(std::false_type{});
    LCPP_CHECK_LAUNCH();
    return LCPP_OK;
}

}  // namespace

int tie_repair_launch(int kind, bool descending, void *keys, void *vals, int val_bytes, void *ktmp, void *vtmp,
                      uint32_t n, const uint32_t *cut, hipStream_t s)
{
    if (!vals) return tr_run<uint32_t, false>(kind, descending, keys, nullptr, ktmp, nullptr, n, cut, s);
    return val_bytes == 4 ? tr_run<uint32_t, true>(kind, descending, keys, vals, ktmp, vtmp, n, cut, s)
                          : tr_run<uint64_t, true>(kind, descending, keys, vals, ktmp, vtmp, n, cut, s);
}

}  // namespace lcpp
