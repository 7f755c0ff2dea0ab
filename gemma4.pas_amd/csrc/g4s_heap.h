/*
 * g4s_heap.h -- exact replay of the reference's min-heap pass
 * (DoSelectTopKIndices, src/Gemma4.Model.pas:2632-2664) over a whole row, for
 * rows whose K-th value is tied in a way the heap's layout decides (bf16
 * logits: nearly every row).  Used by the launch that follows a bf16 top-k
 * select (g4s_topk.hip) and by the wide select (g4s_full.hip).
 *
 * About K (1 + ln(V / K)) elements enter the heap, each after the one before,
 * so the replay is bound by the latency of one insertion.  Without NaNs the
 * heap's root only rises, so screening against an older root keeps a superset:
 * waves 1.. screen the next stretch of the row into LDS (as long as what
 * precedes it, less where the segments would overflow; read 16 bytes a lane,
 * several loads in flight) while wave 0 inserts from the stretch before.  The
 * first stretches admit one segment each (every element passes the first root),
 * so 100,003 elements with K = 40 take nine phases.  Wave 0 inserts in one of
 * two ways:
 *
 *  - K <= 64: node j of the heap lives in lane j (node 64 in lane 0).  The
 *    smaller child of every node is known before the value is: its ballot
 *    gives each lane whether it lies on the path of smaller children, and the
 *    lanes of the path that are below the value take their child, or the
 *    value.  One insertion is one round of cross-lane reads.
 *  - larger K: the nodes are 8-byte LDS entries, a node's children one
 *    16-byte read, and insertions two levels apart run down the heap at the
 *    same time, one per lane: a new one enters every second step, whatever
 *    the depth.
 *
 * A NaN passes every screen and breaks the heap's order: later insertions can
 * lift it to the root, whatever follows is then accepted, and the root falls.
 * So from the stretch that holds the row's first NaN on each element is compared
 * with the root that it meets, and inserted through the LDS form, which makes
 * the reference's comparisons one by one.
 *
 * bf16 rows of 262,144 logits, whole calls, before (one lane inserting step by
 * step, tiles of the block's size) and now: K = 64, one row 713 -> 135 us;
 * K = 200, eight rows 2,050 -> 473; K = 1,000, four rows 15,200 -> 1,743; K =
 * 1,100, one row 23,300 -> 1,804 (its heap was in device memory).  An insertion
 * takes about 0.11 us in the lanes and 0.26 us through LDS.
 */
#ifndef G4S_HEAP_H
#define G4S_HEAP_H

#include "g4s_device.h"

namespace g4s {

constexpr int kHeapExtra = 4;   /* entries beyond K: node 0 and the children past the last node */
constexpr int kHeapMaxWaves = 16;
constexpr int kHeapNan = 1 << 20; /* above any number of entries */

/* two entries; may_alias: the same memory is written as single entries */
typedef uint64_t HeapPair __attribute__((ext_vector_type(2), may_alias));

struct HeapCtl {
    int cnt[2][kHeapMaxWaves];  /* entries of each screening wave's segment, kHeapNan if NaNs passed */
    int stop[2][kHeapMaxWaves]; /* first element that found its segment full, -1: none */
    float root[2];              /* NaN: there is one in the stretch */
};

__device__ __forceinline__ uint64_t heap_pack(float v, int32_t i)
{
    return ((uint64_t)(uint32_t)i << 32) | __float_as_uint(v);
}
__device__ __forceinline__ float heap_val(uint64_t e) { return __uint_as_float((uint32_t)e); }
__device__ __forceinline__ int32_t heap_idx(uint64_t e) { return (int32_t)(e >> 32); }

/* The elements of a 16-byte load. */
template <int DT>
__device__ __forceinline__ void heap_unpack(const uint4 q, float (&v)[Elem<DT>::VW])
{
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (DT == 0) {
            v[i] = __uint_as_float(w[i]);
        } else {
            v[2 * i] = __uint_as_float(w[i] << 16);
            v[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
        }
    }
}

/* Wave 0's side.  heap: nodes 1..K, K + kHeapExtra entries, 16-byte aligned
 * (LDS, or device memory for the largest K). */
struct HeapWave {
    uint64_t* heap;
    int K, lane;
    float root;
    bool regs; /* the heap is in the lanes */
    /* lanes */
    float kv;
    int32_t ki;
    float lv, rv;
    int32_t li, ri;
    uint32_t anc, dir; /* parents of the lane's node, and those whose right side it is on */
    int lc, rc;        /* byte addresses of the children's lanes */
    bool leaf;
    /* pipeline: the insertion of this lane, at node sp (0: none) */
    int sp, slot;
    float sv, nv;
    int32_t si;

    __device__ __forceinline__ void children()
    {
        lv = __int_as_float(__builtin_amdgcn_ds_bpermute(lc, __float_as_int(kv)));
        rv = __int_as_float(__builtin_amdgcn_ds_bpermute(rc, __float_as_int(kv)));
        li = __builtin_amdgcn_ds_bpermute(lc, ki);
        ri = __builtin_amdgcn_ds_bpermute(rc, ki);
    }
    __device__ __forceinline__ void init(uint64_t* h, int k, int ln)
    {
        heap = h;
        K = k;
        lane = ln;
        root = -1e30f;
        regs = K <= 64;
        sp = 0;
        slot = 0;
        sv = nv = 0.0f;
        si = 0;
        const int n = lane == 0 ? 64 : lane;
        /* a missing right child reads the left one (never smaller than it), a
         * lane without a node is never below a value */
        leaf = 2 * n > K;
        lc = ((2 * n) & 63) * 4;
        rc = 2 * n + 1 <= K ? ((2 * n + 1) & 63) * 4 : lc;
        anc = dir = 0;
        for (int c = n; c > 1; c >>= 1) {
            if (c == 64) continue; /* node 32 of 64 has no right child */
            anc |= 1u << (c >> 1);
            if (c & 1) dir |= 1u << (c >> 1);
        }
        kv = n <= K ? -1e30f : __builtin_inff(); /* Model.pas:2634-2638 */
        ki = -1;
        for (int i = lane; i < K + kHeapExtra; i += 64)
            heap[i] = heap_pack(i <= K ? -1e30f : __builtin_inff(), -1);
        if (regs) children();
    }
    /* the lanes' heap to memory */
    __device__ __forceinline__ void spill()
    {
        const int n = lane == 0 ? 64 : lane;
        if (n <= K) heap[n] = heap_pack(kv, ki);
        __builtin_amdgcn_wave_barrier();
        regs = false;
    }
    /* one level of every running insertion (:2647-2661) */
    __device__ __forceinline__ void step()
    {
        if (sp) {
            /* everything but the children is known before they arrive */
            const int last = K / 2 + 1; /* a pair past the last node */
            const float lim = 2 * sp > K ? -__builtin_inff() : sv; /* no child: stop */
            const HeapPair c =
                *reinterpret_cast<const HeapPair*>(heap + 2 * (sp < last ? sp : last));
            const bool right = heap_val(c.y) < heap_val(c.x);
            const float cv = right ? heap_val(c.y) : heap_val(c.x);
            const int32_t ci = right ? heap_idx(c.y) : heap_idx(c.x);
            const bool stop = cv >= lim;
            nv = stop ? sv : cv;
            heap[sp] = heap_pack(nv, stop ? si : ci);
            const int child = right ? 2 * sp + 1 : 2 * sp;
            sp = stop ? 0 : child;
        }
        __builtin_amdgcn_wave_barrier();
    }
    __device__ __forceinline__ void insert_lanes(float v, int32_t vi)
    {
        const bool right = rv < lv;
        const uint32_t pm = (uint32_t)__builtin_amdgcn_ballot_w64(right);
        const float cv = right ? rv : lv;
        const int32_t ci = right ? ri : li;
        const bool stop = cv >= v || leaf;
        const float nk = stop ? v : cv;
        const int32_t ni = stop ? vi : ci;
        const bool moves = kv < v && (pm & anc) == dir;
        kv = moves ? nk : kv;
        ki = moves ? ni : ki;
        children();
        root = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(kv), 1));
    }
    __device__ __forceinline__ void insert_pipe(float v, int32_t vi)
    {
        slot = (slot + 1) & 15;
        if (lane == slot) {
            sp = 1;
            sv = v;
            si = vi;
        }
        step();
        root = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(nv), slot));
        step();
    }
    /* up to 64 screened elements, one per lane, in index order */
    __device__ __forceinline__ void take(uint64_t e, bool valid)
    {
        const float qv = heap_val(e);
        const int32_t qi = heap_idx(e);
        uint64_t mask = __builtin_amdgcn_ballot_w64(valid && !(qv <= root)); /* :2643-2644 */
        if (regs) {
            while (mask) {
                const int l = (int)__builtin_ctzll(mask);
                insert_lanes(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(qv), l)),
                             __builtin_amdgcn_readlane(qi, l));
                mask = (mask & (mask - 1)) & __builtin_amdgcn_ballot_w64(!(qv <= root));
            }
        } else {
            /* the loop's place in the 32-byte windows of instruction fetch: K =
             * 1,100 takes 1,836 us (four rows of 262,144) where it ends up with five
             * s_nop, 1,849 with two or three, 1,862 with four, 1,910 with six and
             * 1,938 with none or eight; without this it moves with any change */
            asm volatile(".p2align 6\ns_nop 0\ns_nop 0\ns_nop 0\ns_nop 0\ns_nop 0");
            while (mask) {
                const int l = (int)__builtin_ctzll(mask);
                insert_pipe(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(qv), l)),
                            __builtin_amdgcn_readlane(qi, l));
                mask = (mask & (mask - 1)) & __builtin_amdgcn_ballot_w64(!(qv <= root));
            }
        }
    }
    /* n elements of the row; the root may fall, so those behind an insertion are
     * compared again */
    __device__ __forceinline__ void follow(const uint64_t* e, int n)
    {
        if (regs) spill();
        for (int i = lane; i - lane < n; i += 64) {
            const uint64_t x = i < n ? e[i] : 0ull;
            uint64_t mask = __builtin_amdgcn_ballot_w64(i < n && !(heap_val(x) <= root));
            while (mask) {
                const int l = (int)__builtin_ctzll(mask);
                insert_pipe(
                    __int_as_float(__builtin_amdgcn_readlane(__float_as_int(heap_val(x)), l)),
                    __builtin_amdgcn_readlane(heap_idx(x), l));
                mask = __builtin_amdgcn_ballot_w64(i < n && lane > l && !(heap_val(x) <= root));
            }
        }
    }
    __device__ __forceinline__ void finish()
    {
        if (regs) spill();
        while (__builtin_amdgcn_ballot_w64(sp != 0)) step();
    }
};

/* Replays the row.  On return (after a barrier) heap[1..K] hold the heap
 * (heap_val, heap_idx; index -1: an entry never filled).  q: qn entries of
 * LDS, at least 2 * (BLOCK / 64 - 1). */
template <int BLOCK, int DT>
__device__ __forceinline__ void heap_replay(const char* row, int V, int K, uint64_t* heap, uint64_t* q, int qn,
                            HeapCtl& ctl)
{
    constexpr int VW = Elem<DT>::VW;
    constexpr int NP = BLOCK / 64 - 1; /* screening waves */
    constexpr int STEP = 64 * VW;
    constexpr int U = BLOCK > 512 ? 4 : 8; /* loads in flight */
    static_assert(NP >= 1 && NP <= kHeapMaxWaves, "screening waves");
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cap = qn / (2 * NP);
    HeapWave hw;
    __syncthreads(); /* the areas are free */
    if (wid == 0) hw.init(heap, K, lane);
    float root = -1e30f;
    int pos = 0, from = 0, nseg = 0;
    for (int ph = 0;; ++ph) {
        const int buf = ph & 1;
        const bool more = pos < V;
        const int t0 = pos - pos % VW;
        /* steps per wave: as much as precedes, less where that would overfill
         * the segments (about K * length / pos elements pass) */
        int64_t len = pos;
        if (cap * NP < K) len = len * (cap * NP) / K;
        int n = (int)(len / (NP * STEP));
        n = n < 1 ? 1 : n;
        if (wid == 0) {
            /* the segments one after another, 64 elements at a time */
            const uint64_t* seg = q + (buf ^ 1) * NP * cap;
            int first[NP], total = 0, nan = 0; /* a segment's first element in that order */
#pragma unroll
            for (int s = 0; s < NP; ++s) {
                first[s] = total;
                const int c =
                    __builtin_amdgcn_readfirstlane(s < nseg ? ctl.cnt[buf ^ 1][s] : 0);
                nan |= c;
                total += c;
            }
            nan &= kHeapNan;
            if (nan) total = 0;
            for (int i = 0; i < total; i += 64) {
                const int f = i + lane;
                int at = f;
#pragma unroll
                for (int s = 1; s < NP; ++s) at = f >= first[s] ? s * cap + f - first[s] : at;
                hw.take(f < total ? seg[at] : 0ull, f < total);
            }
            if (!more && !nan) hw.finish();
            if (lane == 0) ctl.root[buf] = nan ? __builtin_nanf("") : hw.root;
        } else if (more) {
            const int pw = wid - 1;
            uint64_t* seg = q + (buf * NP + pw) * cap;
            const int64_t w0 = t0 + (int64_t)pw * n * STEP + lane * VW;
            int total = 0;
            bool nan = false;
            if (lane == 0) ctl.stop[buf][pw] = -1;
            const auto screen = [&](const float(&x)[VW], int64_t e0) __attribute__((always_inline)) {
                uint32_t in = 0;
#pragma unroll
                for (int i = 0; i < VW; ++i)
                    if (e0 + i >= pos && e0 + i < V && !(x[i] <= root)) in |= 1u << i;
                if (!__builtin_amdgcn_ballot_w64(in != 0) || total > cap) return; /* uniform */
                const int incl = wave_inclusive_scan(__popc(in));
                int at = total + incl - __popc(in);
#pragma unroll
                for (int i = 0; i < VW; ++i) {
                    if ((in >> i) & 1u) {
                        nan |= !(x[i] > root);
                        if (at < cap)
                            seg[at] = heap_pack(x[i], (int32_t)(e0 + i));
                        else if (at == cap)
                            ctl.stop[buf][pw] = (int)(e0 + i);
                        ++at;
                    }
                }
                total += __builtin_amdgcn_readlane(incl, 63);
            };
            for (int s = 0; s < n && total <= cap; s += U) {
                const int64_t last = t0 + ((int64_t)pw * n + (s + U < n ? s + U : n)) * STEP;
                if (last <= V) { /* uniform: whole steps, their loads in flight together */
                    uint4 raw[U];
#pragma unroll
                    for (int t = 0; t < U; ++t)
                        if (s + t < n)
                            raw[t] = *reinterpret_cast<const uint4*>(
                                row + (w0 + (int64_t)(s + t) * STEP) * Elem<DT>::SIZE);
#pragma unroll
                    for (int t = 0; t < U; ++t) {
                        if (s + t < n) {
                            float x[VW];
                            heap_unpack<DT>(raw[t], x);
                            screen(x, w0 + (int64_t)(s + t) * STEP);
                        }
                    }
                } else {
                    for (int t = s; t < n && t < s + U; ++t) {
                        float x[VW];
                        load_vec<DT>(row, w0 + (int64_t)t * STEP, V, x);
                        screen(x, w0 + (int64_t)t * STEP);
                    }
                }
            }
            const int bad = __builtin_amdgcn_ballot_w64(nan) ? kHeapNan : 0;
            if (lane == 0) ctl.cnt[buf][pw] = (total < cap ? total : cap) | bad;
        }
        __syncthreads();
        root = ctl.root[buf];
        if (!more || root != root) break;
        nseg = 0;
        int64_t next = t0 + (int64_t)NP * n * STEP;
        while (nseg < NP) {
            const int stop = ctl.stop[buf][nseg++];
            if (stop >= 0) {
                next = stop;
                break;
            }
        }
        from = pos; /* what the next phase inserts begins here */
        pos = next < V ? (int)next : V;
    }
    if (__builtin_expect(root != root, 0)) {
        for (int base = from; base < V; base += qn) {
            const int n = V - base < qn ? V - base : qn;
            for (int i = threadIdx.x; i < n; i += BLOCK)
                q[i] = heap_pack(load_elem<DT>(row, base + i), base + i);
            __syncthreads();
            if (wid == 0) hw.follow(q, n);
            __syncthreads();
        }
        if (wid == 0) hw.finish();
        __syncthreads();
    }
}

}  // namespace g4s

#endif
