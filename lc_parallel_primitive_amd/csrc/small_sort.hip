// small_sort.hip — DeviceRadixSort of inputs that fit one workgroup.
//
// Reference: device/device_radix_sort.h:129-184 (the same entry points).
//
// MI355X design: the onesweep pipeline (init, histogram, one launch per digit)
// costs six or ten dependent launches of one busy workgroup each, 52-118 us
// however few the keys.  Here one 1024-thread workgroup keeps the keys in
// registers and runs every digit pass through LDS: rank in the wave with the
// per-wave digit counters of the onesweep, one digit scan, scatter to LDS,
// read back in order.
//  * Keys are held wave-striped (wave w, item u, lane l: position
//    w*64*IPT + u*64 + l), so the ranks are stable as in the onesweep; there
//    are no pad keys, positions past n take no part.
//  * A digit that is the same in every key is skipped (one OR over the
//    workgroup of the bits in which the keys differ from the first one).
//  * Values do not ride along: a 16-bit source position does, and the values
//    are gathered once, after the last pass.
//  * Key types differ in what is XORed in and out, so the kernel takes the
//    masks as arguments and is compiled per key size only.
// What bounds it is one CU's LDS and VALU: a full pass of 16384 u32 keys takes
// about 4 us, with a payload 6 us.  Measured (us per call, onesweep pipeline
// -> here): SortKeys u32 of 1023 keys 96 -> 8.6, 8192: 88 -> 11.8, 16384: 59 ->
// 19.2; SortKeys u64 of 8192: 87 -> 25.4; SortPairs u32 -> u32 of 16384: 52 ->
// 29.5 (31.8 with the key and its source position as two LDS words and a
// branch around each counter update).
#include "small_sort.hpp"

namespace lcpp {
namespace {

constexpr int kSsBlock = 1024;
constexpr int kSsWaves = kSsBlock / kWave;
constexpr int kSsRadix = 256;

// A 4-byte key travels with its source position in one 8-byte LDS word.
template <int IPT, class UK, bool PAIRS>
struct SsSmem {
    static constexpr int N = kSsBlock * IPT;
    static constexpr bool kSplit = PAIRS && sizeof(UK) == 8;
    std::conditional_t<PAIRS, uint64_t, UK> item[N];
    uint16_t src[kSplit ? N : 2];
    uint32_t cnt[kSsWaves][kSsRadix];
    uint32_t wsum[kSsRadix / kWave];
    uint32_t diff[kSsWaves][sizeof(UK) / 4];
};

template <int IPT, class UK, bool PAIRS, bool ZEROS, bool MATCH>
__global__ __launch_bounds__(kSsBlock) void small_sort_kernel(const UK *kin, UK *kout, const void *vin, void *vout,
                                                              int val_bytes, uint32_t n, KeyCode<UK, ZEROS> code,
                                                              uint32_t *status)
{
    extern __shared__ __align__(16) unsigned char s_raw[];
    SsSmem<IPT, UK, PAIRS> &sm = *reinterpret_cast<SsSmem<IPT, UK, PAIRS> *>(s_raw);
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    const uint32_t p0 = wave * (kWave * IPT) + lane;  // position of item 0; item u: + u * 64
    if (tid == 0) *status = 0;

    UK tk[IPT];
    uint32_t src[PAIRS ? IPT : 1];
    const UK first = code.ranked(code.in(kin[0]));
    UK diff = 0;
#pragma unroll
    for (int u = 0; u < IPT; ++u) {
        const uint32_t p = p0 + u * kWave;
        tk[u] = p < n ? code.in(kin[p]) : UK(0);
        if constexpr (PAIRS) src[u] = p;
    }
#pragma unroll
    for (int u = 0; u < IPT; ++u)
        if (p0 + u * kWave < n) diff |= code.ranked(tk[u]) ^ first;
    auto or_op = [](uint32_t a, uint32_t b) { return a | b; };
#pragma unroll
    for (int h = 0; h < (int)sizeof(UK) / 4; ++h) {
        const uint32_t w = wave_allreduce((uint32_t)(diff >> (UK)(32 * h)), or_op);
        if (lane == 0) sm.diff[wave][h] = w;
    }
    for (uint32_t i = tid; i < (uint32_t)(kSsWaves * kSsRadix); i += kSsBlock) (&sm.cnt[0][0])[i] = 0;
    __syncthreads();
    diff = 0;
#pragma unroll
    for (int w = 0; w < kSsWaves; ++w)
#pragma unroll
        for (int h = 0; h < (int)sizeof(UK) / 4; ++h) diff |= (UK)sm.diff[w][h] << (UK)(32 * h);

    uint32_t *cnt = sm.cnt[wave];
    const bool busy = wave * (kWave * IPT) < n;  // wave-uniform: the wave holds keys
#pragma unroll 1
    for (uint32_t shift = 0; shift < sizeof(UK) * 8; shift += 8) {
        if (((uint32_t)(diff >> shift) & 255u) == 0) continue;  // the same for the whole workgroup
        uint32_t rank[IPT];
        if (busy) {
#pragma unroll
            for (int u = 0; u < IPT; ++u) {
                // (no branch: positions past n add 0 to a counter per lane)
                const bool ok = p0 + u * kWave < n;
                const uint32_t d = code.digit(tk[u], shift);
                if constexpr (MATCH) {
                    const uint64_t peers = match_any8(d) & ballot(ok);
                    const uint32_t below = mask_rank(peers);
                    uint32_t b = 0;
                    if (ok && below == 0) b = atomicAdd(&cnt[d], (uint32_t)__builtin_popcountll(peers));
                    rank[u] = (uint32_t)__shfl((int)b, ok ? (int)__builtin_ctzll(peers) : 0) + below;
                } else {
                    rank[u] = atomicAdd(&cnt[ok ? d : lane], ok ? 1u : 0u);
                }
            }
        }
        __syncthreads();
        // threads 0..255: one digit each, its counts turned into the position
        // of each wave's first key of that digit
        uint32_t pre[kSsWaves], total = 0;
        if (tid < (uint32_t)kSsRadix) {
#pragma unroll
            for (int w = 0; w < kSsWaves; ++w) pre[w] = sm.cnt[w][tid];
#pragma unroll
            for (int w = 0; w < kSsWaves; ++w) {
                const uint32_t c = pre[w];
                pre[w] = total;
                total += c;
            }
        }
        uint32_t at = wave_inclusive_scan(total, SumOp());
        if (lane == kWave - 1 && wave < (uint32_t)(kSsRadix / kWave)) sm.wsum[wave] = at;
        at -= total;
        __syncthreads();
        if (tid < (uint32_t)kSsRadix) {
#pragma unroll
            for (int w = 0; w < kSsRadix / kWave; ++w)
                if ((uint32_t)w < wave) at += sm.wsum[w];
#pragma unroll
            for (int w = 0; w < kSsWaves; ++w) sm.cnt[w][tid] = at + pre[w];
        }
        __syncthreads();
        if (busy) {
#pragma unroll
            for (int u = 0; u < IPT; ++u) rank[u] += cnt[code.digit(tk[u], shift)];
#pragma unroll
            for (int u = 0; u < IPT; ++u)
                if (p0 + u * kWave < n) {
                    if constexpr (!PAIRS) sm.item[rank[u]] = tk[u];
                    else if constexpr (sizeof(UK) == 4) sm.item[rank[u]] = (uint64_t)src[u] << 32 | tk[u];
                    else {
                        sm.item[rank[u]] = tk[u];
                        sm.src[rank[u]] = (uint16_t)src[u];
                    }
                }
        }
        __syncthreads();
        // (reads past n give stale words that nothing uses)
#pragma unroll
        for (int u = 0; u < IPT; ++u) {
            const auto w = sm.item[p0 + u * kWave];
            tk[u] = (UK)w;
            if constexpr (PAIRS) {
                if constexpr (sizeof(UK) == 4) src[u] = (uint32_t)(w >> 32);
                else src[u] = sm.src[p0 + u * kWave];
            }
        }
        for (uint32_t i = tid; i < (uint32_t)(kSsWaves * kSsRadix); i += kSsBlock) (&sm.cnt[0][0])[i] = 0;
        __syncthreads();
    }
    // every load from the inputs is issued before the barrier, so outputs that
    // alias them are written after
    if constexpr (PAIRS) {
        if (val_bytes == 4) {
            uint32_t v[IPT];
#pragma unroll
            for (int u = 0; u < IPT; ++u)
                if (p0 + u * kWave < n) v[u] = static_cast<const uint32_t *>(vin)[src[u]];
            __syncthreads();
#pragma unroll
            for (int u = 0; u < IPT; ++u)
                if (p0 + u * kWave < n) static_cast<uint32_t *>(vout)[p0 + u * kWave] = v[u];
        } else {
            uint64_t v[IPT];
#pragma unroll
            for (int u = 0; u < IPT; ++u)
                if (p0 + u * kWave < n) v[u] = static_cast<const uint64_t *>(vin)[src[u]];
            __syncthreads();
#pragma unroll
            for (int u = 0; u < IPT; ++u)
                if (p0 + u * kWave < n) static_cast<uint64_t *>(vout)[p0 + u * kWave] = v[u];
        }
    }
#pragma unroll
    for (int u = 0; u < IPT; ++u)
        if (p0 + u * kWave < n) kout[p0 + u * kWave] = code.out(tk[u]);
}

template <int IPT, class UK, bool PAIRS, bool ZEROS, bool MATCH>
int ss_run(const KeyCode<UK, ZEROS> &code, const void *kin, void *kout, const void *vin, void *vout, int val_bytes,
           uint32_t n, uint32_t *status, hipStream_t s)
{
    constexpr size_t lds = sizeof(SsSmem<IPT, UK, PAIRS>);
    static_assert(lds <= 160 * 1024, "one workgroup's LDS");
    if (lds > 64 * 1024) {
        static DeviceCache lds_set;
        if (device_cached(lds_set, [] {
                return hipFuncSetAttribute(reinterpret_cast<const void *>(&small_sort_kernel<IPT, UK, PAIRS, ZEROS, MATCH>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess
                           ? 1
                           : -1;
            }) < 0)
            return LCPP_ERR_HIP;
    }
    LCPP_LAUNCH("rs_small", s,
                (small_sort_kernel<IPT, UK, PAIRS, ZEROS, MATCH><<<1, kSsBlock, lds, s>>>(
                    static_cast<const UK *>(kin), static_cast<UK *>(kout), vin, vout, val_bytes, n, code, status)));
    LCPP_CHECK_LAUNCH();
    return LCPP_OK;
}

template <class UK, bool PAIRS, bool ZEROS, bool MATCH>
int ss_size(const KeyCode<UK, ZEROS> &code, const void *kin, void *kout, const void *vin, void *vout, int vb, uint32_t n,
            uint32_t *status, hipStream_t s)
{
    // items per thread: the fewest that hold n
    if (n <= 2 * kSsBlock) return ss_run<2, UK, PAIRS, ZEROS, MATCH>(code, kin, kout, vin, vout, vb, n, status, s);
    if (n <= 8 * kSsBlock) return ss_run<8, UK, PAIRS, ZEROS, MATCH>(code, kin, kout, vin, vout, vb, n, status, s);
    if constexpr (sizeof(UK) == 4) return ss_run<16, UK, PAIRS, ZEROS, MATCH>(code, kin, kout, vin, vout, vb, n, status, s);
    return LCPP_ERR_INVALID_ARG;
}

template <class UK, bool ZEROS>
int ss_key(int kind, bool desc, bool match, const void *kin, void *kout, const void *vin, void *vout, int vb,
           uint32_t n, uint32_t *status, hipStream_t s)
{
    const KeyCode<UK, ZEROS> c = KeyCode<UK, ZEROS>::of(kind, desc);
    if (vin)
        return match ? ss_size<UK, true, ZEROS, true>(c, kin, kout, vin, vout, vb, n, status, s)
                     : ss_size<UK, true, ZEROS, false>(c, kin, kout, vin, vout, vb, n, status, s);
    return match ? ss_size<UK, false, ZEROS, true>(c, kin, kout, vin, vout, vb, n, status, s)
                 : ss_size<UK, false, ZEROS, false>(c, kin, kout, vin, vout, vb, n, status, s);
}

}  // namespace

int small_sort_launch(int key_bytes, int kind, bool descending, bool match, const void *keys_in, void *keys_out,
                      const void *vals_in, void *vals_out, int val_bytes, uint32_t n, uint32_t *status,
                      hipStream_t s)
{
    auto go = [&](auto uk) {
        using UK = decltype(uk);
        return kind == kFloat ? ss_key<UK, true>(kind, descending, match, keys_in, keys_out, vals_in, vals_out,
                                                 val_bytes, n, status, s)
                              : ss_key<UK, false>(kind, descending, match, keys_in, keys_out, vals_in, vals_out,
                                                  val_bytes, n, status, s);
    };
    return key_bytes == 4 ? go(uint32_t()) : go(uint64_t());
}

}  // namespace lcpp
