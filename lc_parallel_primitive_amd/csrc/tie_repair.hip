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
// the sort stops after the digits that a sample of the keys asks for
// (rs_sample_kernel, radix_sort.hip) and this kernel orders what
// ties: one read of the keys, and writes where something moves.
//  * A 256-thread workgroup owns the runs that begin in its 2048 keys; 64 more
//    keys cover the runs that begin last.  Keys that tie with a neighbour are
//    listed; each counts its place among its run in LDS (runs of up to 32 keys),
//    and those that move are written with their values.
//  * Longer runs are found to the end by the whole workgroup, skipped if in
//    order already (equal keys are), ranked against each other in LDS up to
//    2112 keys, and else sorted digit by digit between the output and the
//    scratch, by the one workgroup, at a cost linear in their length.
// What bounds it is the read of the keys, and the writes of those that move: 12 *
// 10^6 u64 keys with u32 values, us, after 32 / 24 upper bits: 37 / 75 (one
// thread per run, by insertion in LDS: - / 93; every key looking for its place,
// unlisted: - / 80).  The whole sort: 540 -> 315 us, of u64 keys alone 10^6:
// 125 -> 78.
// A neighbouring workgroup may read keys of a run while its owner moves them;
// it looks at the upper bits alone, and those are the same wherever they go.
#include "tie_repair.hpp"

namespace lcpp {
namespace {

constexpr int kTrBlock = 256;
constexpr int kTrWaves = kTrBlock / kWave;
constexpr uint32_t kTrTile = 2048, kTrHalo = 64, kTrCap = kTrTile + kTrHalo;
constexpr uint32_t kTrShort = 32;  // longest run for one thread
constexpr int kTrItems = (int)ceil_div(kTrCap, kTrBlock);
constexpr int kTrRadixItems = 4;  // per thread and step of a run longer than kTrCap
static_assert(kTrHalo > kTrShort, "a run that begins in the tile is known to its first 33 keys");

template <class UV, bool PAIRS, bool ZEROS>
__global__ __launch_bounds__(kTrBlock) void tie_repair_kernel(uint64_t *keys, UV *vals, uint64_t *ktmp, UV *vtmp,
                                                              uint32_t n, KeyCode<uint64_t, ZEROS> code,
                                                              const uint32_t *__restrict__ cut_word)
{
    __shared__ uint64_t sk[kTrCap];
    __shared__ uint16_t place[kTrCap];
    __shared__ uint32_t longs[kTrTile / kTrShort];
    __shared__ uint32_t nlong, nties, s_end, s_flag;
    __shared__ uint32_t wcnt[kTrWaves][256], dbase[256], wsum[kTrWaves];

    const uint32_t cut = __builtin_amdgcn_readfirstlane(*cut_word);
    if (cut == 0) return;
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    const uint32_t base = blockIdx.x * kTrTile;
    const uint32_t m = n - base < kTrCap ? n - base : kTrCap;     // keys in LDS
    const uint32_t own = n - base < kTrTile ? n - base : kTrTile;  // those whose runs are this workgroup's
    auto top = [&](uint64_t t) { return code.ranked(t) >> cut; };

    if (tid == 0) nlong = nties = 0;
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

    // the keys that tie with a neighbour, listed
#pragma unroll
    for (int u = 0; u < kTrItems; ++u) {
        const uint32_t i = tid + u * kTrBlock;
        const uint64_t t = top(k[u]);
        const uint64_t l = top(sk[i > 0 && i < m ? i - 1 : 0]), r = top(sk[i + 1 < m ? i + 1 : 0]);
        const bool tie = i < m && ((i > 0 && l == t) || (i + 1 < m && r == t));
        const uint64_t who = ballot(tie);
        if (who == 0) continue;
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(&nties, (uint32_t)__builtin_popcountll(who));
        at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) + mask_rank(who);
        if (tie) place[at] = (uint16_t)i;
    }
    __syncthreads();
    // each finds its place in its run by itself: the keys to its left that do
    // not rank above it and those to its right that rank below it
    const uint32_t ties = nties;
    uint32_t to[kTrItems];
    UV v[PAIRS ? kTrItems : 1];
#pragma unroll
    for (int u = 0; u < kTrItems; ++u) {
        to[u] = ~0u;
        const uint32_t q = tid + u * kTrBlock;
        if (q >= ties) continue;
        const uint32_t i = place[q];
        k[u] = sk[i];
        const uint64_t x = code.ranked(k[u]), t = x >> cut;
        uint32_t left = 0, right = 0, r = 0;
        while (left <= kTrShort && left < i) {
            const uint64_t y = code.ranked(sk[i - 1 - left]);
            if (y >> cut != t) break;
            r += y <= x ? 1u : 0u;
            ++left;
        }
        while (left + right <= kTrShort && i + 1 + right < m) {
            const uint64_t y = code.ranked(sk[i + 1 + right]);
            if (y >> cut != t) break;
            r += y < x ? 1u : 0u;
            ++right;
        }
        const uint32_t first = i - left;
        // the run is another workgroup's, or goes to the whole workgroup
        if (first >= own || (first == 0 && base && before == t)) continue;
        if (left + 1 + right > kTrShort) {
            if (left == 0) longs[atomicAdd(&nlong, 1u)] = base + i;
            continue;
        }
        if (r == left) continue;  // in its place
        to[u] = first + r;
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
    __syncthreads();

    const uint32_t runs = nlong;
#pragma unroll 1
    for (uint32_t q = 0; q < runs; ++q) {
        const uint32_t g0 = longs[q];
        const uint64_t t = top(code.in(keys[g0]));
        // the first position past the run
        uint32_t end = g0 + kTrShort + 1;
        for (;; end += kTrBlock) {
            __syncthreads();
            if (tid == 0) s_end = ~0u;
            __syncthreads();
            const uint64_t i = (uint64_t)end + tid;
            if (i >= n || top(code.in(keys[i])) != t) atomicMin(&s_end, tid);
            __syncthreads();
            if (s_end != ~0u) break;
        }
        end = end + s_end < n ? end + s_end : n;
        const uint32_t L = end - g0;
        __syncthreads();
        if (tid == 0) s_flag = 0;
        __syncthreads();
        bool down = false;
        for (uint32_t i = tid; i + 1 < L; i += kTrBlock)
            down |= code.ranked(code.in(keys[g0 + i])) > code.ranked(code.in(keys[g0 + i + 1]));
        if (down) s_flag = 1;
        __syncthreads();
        if (!s_flag) continue;  // the same for the whole workgroup
        if (L <= kTrCap) {
            for (uint32_t i = tid; i < L; i += kTrBlock) sk[i] = code.in(keys[g0 + i]);
            if constexpr (PAIRS) {
#pragma unroll
                for (int u = 0; u < kTrItems; ++u) {
                    const uint32_t i = tid + u * kTrBlock;
                    if (i < L) v[u] = vals[g0 + i];
                }
            }
            __syncthreads();
            for (int u = 0; u < kTrItems; ++u) {
                const uint32_t i = tid + u * kTrBlock;
                if (i >= L) break;
                const uint64_t x = code.ranked(sk[i]);
                uint32_t r = 0;
                for (uint32_t j = 0; j < L; ++j) {
                    const uint64_t y = code.ranked(sk[j]);
                    r += y < x || (y == x && j < i) ? 1u : 0u;
                }
                place[i] = (uint16_t)r;
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kTrItems; ++u) {
                const uint32_t i = tid + u * kTrBlock;
                if (i < L) {
                    keys[g0 + place[i]] = code.out(sk[i]);
                    if constexpr (PAIRS) vals[g0 + place[i]] = v[u];
                }
            }
            continue;
        }
        // digit by digit, kTrBlock * kTrRadixItems keys at a time (items of a
        // wave are consecutive: ranked by ballot match, stable)
        uint64_t *ka = keys + g0, *kb = ktmp + g0;
        UV *va = PAIRS ? vals + g0 : nullptr, *vb = PAIRS ? vtmp + g0 : nullptr;
#pragma unroll 1
        for (uint32_t shift = 0; shift < cut; shift += 8) {
            __syncthreads();
            dbase[tid] = 0;
            if (tid == 0) s_flag = 0;
            __syncthreads();
            for (uint32_t i = tid; i < L; i += kTrBlock) atomicAdd(&dbase[code.digit(code.in(ka[i]), shift)], 1u);
            __syncthreads();
            const uint32_t c = dbase[tid];
            if (c == L) s_flag = 1;
            uint32_t ex = wave_inclusive_scan(c, SumOp());
            if (lane == kWave - 1) wsum[wave] = ex;
            ex -= c;
            __syncthreads();
            for (uint32_t w = 0; w < wave; ++w) ex += wsum[w];
            const bool same = s_flag != 0;
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
        if (ka != keys + g0) {
            for (uint32_t i = tid; i < L; i += kTrBlock) {
                keys[g0 + i] = ka[i];
                if constexpr (PAIRS) vals[g0 + i] = va[i];
            }
        }
        __syncthreads();
    }
}

template <class UV, bool PAIRS>
int tr_run(int kind, bool desc, void *keys, void *vals, void *ktmp, void *vtmp, uint32_t n, const uint32_t *cut,
           hipStream_t s)
{
    const uint32_t grid = (uint32_t)ceil_div(n, kTrTile);
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
