// by_key.hpp — tile machinery shared by ScanByKey and ReduceByKey (gfx950).
//
// Reference: device/details/scan_by_key.h:77-258 and
// device/details/reduce_by_key.h:61-258 (BlockLoad of keys and values,
// BlockDiscontinuity::FlagHeads, a BlockScan of (flag, value) pairs with
// ScanBySegmentOp / ReduceBySegmentOp, TilePrefixCallbackOp look-back).
//
// MI355X design: one 256-thread workgroup per tile of 8 x 16-byte value
// vectors per thread (8192 4-byte or 4096 8-byte values).  Thread t, vector
// k holds elements k*256*VP + t*VP + j (VP = 16 / sizeof(V), j < VP), so every
// load and store instruction covers contiguous memory; its keys sit at the
// same element indices.  Segment heads (key != previous key, compared in the
// key type) are one bit per element.  The tile is processed reduce-then-
// rescan: pass 1 folds each thread's elements into (has-head, value since
// the last head) pairs, a wave64 segmented scan of those pairs per vector,
// the wave totals through LDS; one wave runs the decoupled look-back
// (lookback.hpp), where a tile containing a head publishes INCLUSIVE at
// once; pass 2 rescans each thread's elements seeded with its exact prefix.
#pragma once

#include "lookback.hpp"

namespace lcpp {
namespace {

constexpr int kBkBlock = 256;
constexpr int kBkWaves = kBkBlock / kWave;
constexpr int kBkVecs = 8;

template <class V>
constexpr int bk_vp()
{
    return 16 / (int)sizeof(V);
}
template <class V>
constexpr uint32_t bk_tile()
{
    return (uint32_t)(kBkBlock * kBkVecs * bk_vp<V>());
}
template <class V>
uint64_t bk_tiles(uint64_t n)
{
    return n ? ceil_div(n, bk_tile<V>()) : 0;
}

// Binary operators with their identities (common/thread_operators.h:49-74).
template <class Op, class T>
__device__ __forceinline__ T op_identity()
{
    return Op::template identity<T>();
}

// Segment-pair fold (ScanBySegmentOp / ReduceBySegmentOp,
// common/thread_operators.h:85-127): (fa, a) then (fb, b).
template <class T, class Op>
__device__ __forceinline__ void seg_fold(bool &fa, T &a, bool fb, T b, Op op)
{
    a = fb ? b : op(a, b);
    fa = fa || fb;
}

// Inclusive wave64 segmented scan of (f, s) over lanes (lane order).
template <class T, class Op>
__device__ __forceinline__ void wave_seg_scan(bool &f, T &s, Op op)
{
    // the DPP steps of wave_inclusive_scan over (flag, value) pairs; lanes
    // with no source take (false, identity)
    const T id = op_identity<Op, T>();
    auto step = [&](int fu, T su) {
        s = f ? s : op(su, s);
        f = f || fu != 0;
    };
    step(dpp_move<kDppRowShr + 1>((int)f, 0), dpp_move<kDppRowShr + 1>(s, id));
    step(dpp_move<kDppRowShr + 2>((int)f, 0), dpp_move<kDppRowShr + 2>(s, id));
    step(dpp_move<kDppRowShr + 4>((int)f, 0), dpp_move<kDppRowShr + 4>(s, id));
    step(dpp_move<kDppRowShr + 8>((int)f, 0), dpp_move<kDppRowShr + 8>(s, id));
    step(dpp_move<kDppRowBcast15, 0xA>((int)f, 0), dpp_move<kDppRowBcast15, 0xA>(s, id));
    step(dpp_move<kDppRowBcast31, 0xC>((int)f, 0), dpp_move<kDppRowBcast31, 0xC>(s, id));
}

// Keys and values of one thread.
template <class K, class V>
struct BkRegs {
    static constexpr int VP = bk_vp<V>();
    K key[kBkVecs][VP];
    V val[kBkVecs][VP];
};

// Element offset (within the tile) of item (k, j) of thread t.
template <class V>
__device__ __forceinline__ uint32_t bk_elem(int k, uint32_t t, int j)
{
    return (uint32_t)k * kBkBlock * bk_vp<V>() + t * bk_vp<V>() + (uint32_t)j;
}

// Loads one tile.  `fast`: full tile and 16-byte aligned pointers; otherwise
// element-wise raw-buffer loads whose offsets (all in the VGPR operand) are
// range-checked against `valid` elements, returning 0 past it.  KEYS_FIRST
// issues every key load before the value loads, so that work on the keys
// alone can start while the values are still in flight (loads complete in
// issue order).
template <bool KEYS_FIRST = false, class K, class V>
__device__ __forceinline__ void bk_load(BkRegs<K, V> &r, const K *keys, const V *vals, uint64_t base,
                                        uint32_t valid, bool fast, uint32_t tid)
{
    constexpr int VP = bk_vp<V>();
    constexpr uint32_t KB = VP * sizeof(K);  // key bytes per thread and vector
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(keys + base, valid * (uint32_t)sizeof(K));
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(vals + base, valid * (uint32_t)sizeof(V));
    if (fast) {
#pragma unroll
        for (int k = 0; k < kBkVecs; ++k) {
            if constexpr (!KEYS_FIRST) unpack16<V>(buf_ld16_nt(rv, tid * 16 + (uint32_t)k * kBkBlock * 16, 0), r.val[k]);
            const uint32_t ko = tid * KB + (uint32_t)k * kBkBlock * KB;
            if constexpr (KB == 16) {
                unpack16<K>(buf_ld16_nt(rk, ko, 0), r.key[k]);
            } else if constexpr (KB == 32) {
                K lo[2], hi[2];
                unpack16<K>(buf_ld16_nt(rk, ko, 0), lo);
                unpack16<K>(buf_ld16_nt(rk, ko + 16, 0), hi);
                r.key[k][0] = lo[0];
                r.key[k][1] = lo[1];
                r.key[k][2] = hi[0];
                r.key[k][3] = hi[1];
            } else {
                static_assert(KB == 8, "4-byte keys with 8-byte values");
                const auto w = __builtin_amdgcn_raw_buffer_load_b64(rk, (int)ko, 0, kPolicyNT);
                const uint32_t a = w[0], b = w[1];
                r.key[k][0] = __builtin_bit_cast(K, a);
                r.key[k][1] = __builtin_bit_cast(K, b);
            }
        }
        if constexpr (KEYS_FIRST) {
#pragma unroll
            for (int k = 0; k < kBkVecs; ++k)
                unpack16<V>(buf_ld16_nt(rv, tid * 16 + (uint32_t)k * kBkBlock * 16, 0), r.val[k]);
        }
    } else {
#pragma unroll
        for (int k = 0; k < kBkVecs; ++k)
#pragma unroll
            for (int j = 0; j < VP; ++j) {
                const uint32_t e = bk_elem<V>(k, tid, j);
                r.val[k][j] = buf_ld_elem<V>(rv, e * (uint32_t)sizeof(V), 0);
                r.key[k][j] = buf_ld_elem<K>(rk, e * (uint32_t)sizeof(K), 0);
            }
    }
}

// Segment-head bits: bit k*VP + j is set when item (k, j) starts a segment
// (element 0 of the input, or key != previous key in the key type).  The
// previous key of a thread's first item comes from lane - 1 (a shuffle), the
// last lane of the previous wave or vector (LDS), or the key just before the
// tile.  prev0[k] receives the previous key of item (k, 0).  Contains a
// workgroup barrier.
template <class K, int VP>
__device__ __forceinline__ uint32_t bk_heads(const K (&key)[kBkVecs][VP], K (&prev0)[kBkVecs],
                                             K (&s_last)[kBkVecs][kBkWaves], K &s_pred, const K *keys,
                                             uint64_t base, uint32_t tile, uint32_t tid)
{
    const uint32_t lane = lane_id(), wave = tid / kWave;
    if (lane == kWave - 1) {
#pragma unroll
        for (int k = 0; k < kBkVecs; ++k) s_last[k][wave] = key[k][VP - 1];
    }
    if (tid == 0) s_pred = tile > 0 ? keys[base - 1] : K(0);
    __syncthreads();
    uint32_t fl = 0;
#pragma unroll
    for (int k = 0; k < kBkVecs; ++k) {
        const K up = shfl_up(key[k][VP - 1], 1);
        const K prev = lane > 0 ? up : wave > 0 ? s_last[k][wave - 1] : k > 0 ? s_last[k - 1][kBkWaves - 1] : s_pred;
        prev0[k] = prev;
        bool h = key[k][0] != prev;
        if (k == 0 && tid == 0 && tile == 0) h = true;
        fl |= (uint32_t)h << (k * VP);
#pragma unroll
        for (int j = 1; j < VP; ++j) fl |= (uint32_t)(key[k][j] != key[k][j - 1]) << (k * VP + j);
    }
    return fl;
}

// Pass 1 of one vector: (has-head, fold since the last head) of a thread's
// VP items.
template <class V, class Op, int VP>
__device__ __forceinline__ void bk_thread_pair(const V (&x)[VP], uint32_t bits, Op op, bool &f, V &s)
{
    f = false;
    s = op_identity<Op, V>();
#pragma unroll
    for (int j = 0; j < VP; ++j) seg_fold(f, s, ((bits >> j) & 1u) != 0, x[j], op);
}

// ---------------------------------------------------------------- small inputs
// They take one launch without look-back state: every 1024-thread workgroup (4
// consecutive elements per thread) looks for the run that enters its tile by
// itself, back to that run's head, and ReduceByKey counts the heads before its
// tile as well.  What bounds it is the last workgroup's read of the keys before
// it, from L2.  Measured (us per call, C calls back to back, int32 keys, f32
// values, n = 2^15 / 2^16, look-back form 8.8 and 13.3): InclusiveSumByKey, runs of
// 128: 4.8 / 4.9, all keys equal 7.9 / 11.2; ReduceByKey 6.8 / 9.8 (all equal
// 7.2 / 10.6).  Without 16-byte loads, at 2^14: 6.8, 9.9; 9.0, 10.0.  The lines
// lie where every kind of run still gains.
constexpr int kBkAloneBlock = 1024;
constexpr int kBkAloneWaves = kBkAloneBlock / kWave;
constexpr int kBkAloneItems = 4;
constexpr uint32_t kBkAloneTile = kBkAloneBlock * kBkAloneItems;
constexpr uint64_t bk_alone_max(bool reduce, bool vec) { return (reduce ? 1u << 16 : 1u << 15) >> (vec ? 0 : 2); }

template <class V>
struct BkAloneSmem {
    uint32_t cnt[kBkAloneWaves], last[kBkAloneWaves];
    V fold[kBkAloneWaves], S[kBkAloneWaves];
    uint32_t F, C[kBkAloneWaves];  // F bit w: wave w has a head
};

// A thread's items [i0, i0 + 4) of `p`, those below `end` (the others: `fill`);
// `vec`: p is 16-byte aligned.
template <class T>
__device__ __forceinline__ void bk_alone_load(const T *p, uint32_t i0, uint32_t end, bool vec, T fill,
                                              T (&x)[kBkAloneItems])
{
    if (vec && i0 + kBkAloneItems <= end) {
        constexpr int V = 16 / (int)sizeof(T);
#pragma unroll
        for (int q = 0; q < kBkAloneItems / V; ++q) {
            T e[V];
            unpack16<T>(*reinterpret_cast<const u32x4 *>(p + i0 + q * V), e);
#pragma unroll
            for (int j = 0; j < V; ++j) x[q * V + j] = e[j];
        }
    } else {
#pragma unroll
        for (int j = 0; j < kBkAloneItems; ++j) x[j] = i0 + j < end ? p[i0 + j] : fill;
    }
}

// Heads of a thread's items below `end`: bit j for item j.
template <class K>
__device__ __forceinline__ uint32_t bk_alone_heads(const K *keys, uint32_t i0, uint32_t end, bool vec,
                                                   K (&key)[kBkAloneItems], K &prev)
{
    uint32_t fl = 0;
    prev = i0 > 0 && i0 < end ? keys[i0 - 1] : K(0);
    bk_alone_load(keys, i0, end, vec, K(0), key);
#pragma unroll
    for (int j = 0; j < kBkAloneItems; ++j) {
        const bool h = i0 + j == 0 || key[j] != (j ? key[j - 1] : prev);
        fl |= (uint32_t)(h && i0 + j < end) << j;
    }
    return fl;
}

// What lies before the tile at `base` (> 0): `fold` over the values from the
// last head before it on, and (COUNT) the number of heads.  Contains barriers;
// every thread gets both.
template <bool COUNT, class K, class V, class Op>
__device__ __forceinline__ void bk_alone_before(const K *keys, const V *vals, uint32_t base, bool vec, Op op, V &fold,
                                                uint32_t &heads, BkAloneSmem<V> &sm)
{
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    uint32_t head = 0, count = 0;  // head: the last one's position + 1
    auto look = [&](uint32_t lo, uint32_t hi) {  // both multiples of the tile
        uint32_t last = 0, c = 0;
#pragma unroll 4
        for (uint32_t i0 = lo + tid * kBkAloneItems; i0 < hi; i0 += kBkAloneTile) {
            K key[kBkAloneItems], prev;
            const uint32_t fl = bk_alone_heads(keys, i0, hi, vec, key, prev);
            last = fl ? i0 + (uint32_t)(32 - __builtin_clz(fl)) : last;
            if constexpr (COUNT) c += (uint32_t)__builtin_popcount(fl);
        }
        last = wave_allreduce(last, MaxOp());
        if constexpr (COUNT) c = wave_allreduce(c, SumOp());
        __syncthreads();
        if (lane == 0) {
            sm.last[wave] = last;
            sm.cnt[wave] = c;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kBkAloneWaves; ++w) {
            head = sm.last[w] > head ? sm.last[w] : head;
            if constexpr (COUNT) count += sm.cnt[w];
        }
    };
    // a run is most often found in the tile before; then all that is left
    if (!COUNT) look(base - kBkAloneTile, base);
    if (head == 0) look(0, COUNT ? base : base - kBkAloneTile);
    V acc = op_identity<Op, V>();
#pragma unroll 8
    for (uint32_t i = head - 1 + tid; i < base; i += kBkAloneBlock) acc = op(acc, vals[i]);  // element 0 is a head
    acc = wave_allreduce(acc, op);
    if (lane == 0) sm.fold[wave] = acc;
    __syncthreads();
    fold = sm.fold[0];
#pragma unroll
    for (int w = 1; w < kBkAloneWaves; ++w) fold = op(fold, sm.fold[w]);
    heads = count;
}

// The fold since the last head before this thread's first item.  f, s: the
// thread's (has-head, fold since its last head) pair.  Contains a barrier.
template <class V, class Op>
__device__ __forceinline__ V bk_alone_prefix(bool f, V s, V before, Op op, BkAloneSmem<V> &sm)
{
    const uint32_t lane = lane_id(), wave = threadIdx.x / kWave;
    wave_seg_scan(f, s, op);
    const int fu = __shfl_up((int)f, 1);
    const V su = shfl_up(s, 1);
    if (lane == kWave - 1) {
        sm.S[wave] = s;
        if (f) atomicOr(&sm.F, 1u << wave);
    }
    __syncthreads();
    V p = before;
#pragma unroll
    for (int w = 0; w < kBkAloneWaves; ++w)
        if ((uint32_t)w < wave) p = ((sm.F >> w) & 1u) ? sm.S[w] : op(p, sm.S[w]);
    return lane == 0 ? p : fu ? su : op(p, su);
}

// Whether [a, a + an) and [b, b + bn) share bytes.
inline bool bk_overlap(const void *a, uint64_t an, const void *b, uint64_t bn)
{
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x < y + bn && y < x + an;
}

}  // namespace
}  // namespace lcpp
