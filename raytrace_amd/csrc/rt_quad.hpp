// rt_quad.hpp — walks of short queues: four lanes per ray.
//
// A wave that walks 64 rays takes about a microsecond a step whatever else the
// GPU does: a node's loads, then the tests of its four children one after
// another, and it runs as long as its slowest ray.  Where a level holds fewer
// rays than the GPU has lanes (the deep levels of a frame, small frames and
// batches) that chain is the kernel's time.  Here four neighbouring lanes (a
// quad) share a ray: each tests one child of a node, or one primitive of the
// two leaves it postponed, and the results meet in cross-lane moves.  A wave
// holds 16 rays, so it waits for the slowest of 16, and a short queue spreads
// over four times the waves.
//
// The results are trace_closest's and trace_any's: the same child tests
// (Node4Test), primitive tests and winner (the least (t, key)), which depend
// on neither the order of the walk nor on who tests what.
#pragma once
#include <type_traits>

#include "rt_devstack.hpp"
#include "rt_trace.hpp"

namespace rtg {

constexpr int kQuadLanes = 4;
// Queues of up to this many rays per CU are walked by quads: what a CU holds
// of them at once, 24 waves (k_extend's 6 per SIMD) of 16 rays; 98,304 on 256
// CUs.  Longer queues keep every lane busy with a ray of its own, and a quad
// spends about half the instructions of a whole ray on a quarter of its lanes.
// Limits of 8k / 32k / 64k / 128k / 256k / 600k rays measured (us a call, no
// quads first): 64x64 frame 271 / 217 / 218 / 217 / 217 / 218 / 217; 12
// thumbnails in a batch 2586 / 2324 / 2000 / 1962 / 1977 / 1958 / 1950; 1080p
// frame 2120 / 2122 / 2051 / 2013 / 2012 / 2075 / 2126; 640x480 frame 609 /
// 614 / 619 / 625 / 622 / 707 / 851.
constexpr int kQuadRaysPerCu = 24 * 16;
static_assert(kLdsStack * kQuadLanes + kStackMax - kLdsStack >= kStackMax, "a quad's stack holds any walk");

// Move across the quad: lane k reads lane (k ^ 1), (k ^ 2) or (k ^ 3) of its
// quad.  Quads are active or inactive as a whole.
template <int kXor>
__device__ inline int quad_xor(int v) {
    constexpr int ctrl = kXor == 1 ? 0xB1 : kXor == 2 ? 0x4E : 0x1B;
    return __builtin_amdgcn_update_dpp(v, v, ctrl, 0xF, 0xF, true);
}
template <int kXor>
__device__ inline float quad_xor(float v) {
    return as_float(quad_xor<kXor>(as_int(v)));
}
__device__ inline int quad_or(int v) {
    v |= quad_xor<1>(v);
    return v | quad_xor<2>(v);
}
__device__ inline float quad_min(float v) {
    v = fminf(v, quad_xor<1>(v));
    return fminf(v, quad_xor<2>(v));
}

// One stack per quad, in the stack memory of its own four lanes and no other
// (waves of a block may walk rays by quads and by lanes at the same time):
// entry e in row e / 4, column e % 4 of their LDS columns, 64 entries; the
// rest in the first lane's spill column.  An entry is written by the lane that
// holds the child and read by all four; a wave's accesses to LDS, and to one
// global address, are done in order, and the fences keep the compiler from
// moving them.
struct QuadStack {
    int *lds;
    int *spill;
    int gstride;
    int sp;
    const Bvh4Node *top;
    static constexpr int kLds = kLdsStack * kQuadLanes;
    __device__ explicit QuadStack(const DevStack &st, int *lds_base)
        : lds(lds_base + (threadIdx.x & ~(kQuadLanes - 1))), spill(st.spill - (threadIdx.x & (kQuadLanes - 1))),
          gstride(st.gstride), sp(0), top(st.top) {}
    __device__ static void order() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    static __device__ unsigned at(unsigned e) { return (e / kQuadLanes) * kBlockThreads + e % kQuadLanes; }
    // Entry 0 is kWalkDone (see DevStack).  Every lane of the quad calls it.
    __device__ void reset() {
        put_lds(0, kWalkDone);
        sp = 1;
    }
    __device__ void put_lds(int e, int v) {
#if defined(__HIP_DEVICE_COMPILE__)
        typedef int __attribute__((address_space(3))) LdsInt;
        ((LdsInt *)lds)[at(e)] = v;
        __asm__ volatile("" ::: "memory");
#endif
    }
    // The lanes with `mine` put their v into their entry e, at most sp + 2.
    __device__ void put(bool mine, int e, int v) {
        if (__ballot(sp > kLds - 3) == 0ull) {
            if (mine) put_lds(e, v);
        } else if (mine) {
            if (e < kLds)
                put_lds(e, v);
            else
                spill[(e - kLds) * gstride] = v;
        }
    }
    __device__ int pop() {
        --sp;
        int v = 0;
        order();
#if defined(__HIP_DEVICE_COMPILE__)
        typedef const int __attribute__((address_space(3))) LdsInt;
        if (__ballot(sp >= kLds) == 0ull) {
            v = ((LdsInt *)lds)[at(sp)];
            __asm__ volatile("" ::: "memory");  // not merged with the spill read into a flat load
        } else if (sp < kLds) {
            v = ((LdsInt *)lds)[at(sp)];
            __asm__ volatile("" ::: "memory");
        } else {
            v = spill[(sp - kLds) * gstride];
        }
#endif
        order();
        return v;
    }
    template <int N, int D>
    __device__ bool lanes_at_least(bool v) const {
        return D * __popcll(__ballot(v)) >= N * __popcll(__ballot(true));
    }
    // Node i's bounds, and the link of its child k.
    __device__ Bvh4Node node(const SceneView &S, int i, int k, int &link) const {
        Bvh4Node n{};
#if defined(__HIP_DEVICE_COMPILE__)
        typedef const Bvh4Node __attribute__((address_space(3))) LdsNode;
        typedef const int __attribute__((address_space(3))) LdsInt;
        if (top != nullptr && i < kTopNodes) {
            n.org = ((LdsNode *)top)[i].org, n.qxy = ((LdsNode *)top)[i].qxy, n.qz = ((LdsNode *)top)[i].qz;
            link = ((LdsInt *)top)[i * (int)(sizeof(Bvh4Node) / 4) + 12 + k];
            __asm__ volatile("" ::: "memory");
            return n;
        }
#endif
        const Bvh4Node &g = S.nodes[i];
        n.org = g.org, n.qxy = g.qxy, n.qz = g.qz;
        link = (&g.link.x)[k];
        return n;
    }
};

// bvh_walk<true, kOrdered> with a quad per ray: the same postponed leaves and
// wave-wide exit of the node loop.  test(primitive) -> true to stop (any-hit).
template <bool kOrdered, class Test>
__device__ inline void quad_walk(const SceneView &S, const Ray &r, float &tmax, QuadStack &st, Test &&test) {
    if (S.n_prims == 0) return;
    st.reset();
    const int k = threadIdx.x & (kQuadLanes - 1);
    const V3 inv = safe_inv(r.d);
    int node = S.root;
    auto step = [&](int nd) -> int {
        int link;
        const Bvh4Node n = st.node(S, nd, k, link);
        const Node4Test nt(n, r.o, inv);
        float t;
        const bool h = nt.child(k, tmax, t) & (k < node4_count(n));
        int rank, hits;  // children reached that come before this lane's, and all of them
        if constexpr (kOrdered) {
            // by entry distance; the two lowest bits make the keys distinct
            const uint32_t key = h ? ((__builtin_bit_cast(uint32_t, t > 0.0f ? t : 0.0f) & ~3u) | (uint32_t)k) : ~0u;
            const uint32_t a = (uint32_t)quad_xor<1>((int)key), b = (uint32_t)quad_xor<2>((int)key),
                           c = (uint32_t)quad_xor<3>((int)key);
            rank = (a < key) + (b < key) + (c < key);
            hits = h + (a != ~0u) + (b != ~0u) + (c != ~0u);
        } else {
            const uint32_t m = (uint32_t)(__ballot(h) >> (__lane_id() & ~3)) & 15u;
            rank = __popc(m & ((1u << k) - 1u));
            hits = __popc(m);
        }
        const int next = quad_or(h && rank == 0 ? link : 0);
        st.put(h && rank > 0, st.sp + hits - 1 - rank, link);
        if (hits == 0) return st.pop();
        st.sp += hits - 1;
        return next;
    };
    int leaf = 0, leaf2 = 0;  // postponed leaves (< 0), or 0
    for (;;) {
        while (node >= 0) {
            node = step(node);
            if (node < 0 && node != kWalkDone && leaf2 == 0) {
                (leaf == 0 ? leaf : leaf2) = node;
                node = st.pop();
            }
            if (kOrdered ? st.template lanes_at_least<1, 2>(leaf != 0) : st.template lanes_at_least<3, 4>(leaf != 0))
                break;
        }
        if (leaf == 0 && node < 0 && node != kWalkDone) {
            leaf = node;
            node = st.pop();
        }
        while (leaf < 0) {
            // lanes 0 and 1 take the first leaf's primitives, 2 and 3 the second's
            const int mine = (k & 2) ? leaf2 : leaf;
            int stop = 0;
            if (mine < 0) {
                const int first = leaf_first(mine), count = leaf_count(mine);
                for (int i = k & 1; i < count; i += 2) stop |= test(first + i) ? 1 : 0;
            }
            if constexpr (kOrdered)
                tmax = quad_min(tmax);
            else if (quad_or(stop))
                return;
            leaf = leaf2 = 0;
            if (node < 0 && node != kWalkDone) {
                leaf = node;
                node = st.pop();
            }
        }
        if (node == kWalkDone) return;
    }
}

// trace_closest<false, true>; every lane of the quad gets the hit.
__device__ inline Hit quad_closest(const SceneView &S, const TraceRay &q, QuadStack &st, int before) {
    Hit best{kMiss, HIT_NONE, -1, -1, 0, 0, 0};
    brute_objects(S, q, false, 0.0f, best, before);
    uint64_t bkey = best.kind != HIT_NONE ? hit_key(best.obj, best.prim) : ~0ull;
    float tmax = best.t;
    int self = 0;  // 1 + slot of the source triangle, where the ray hits it
    quad_walk<true>(S, q.r, tmax, st, [&](int pi) -> bool {
        Hit h;
        if (!closest_prim(q, load_prim(S, pi), before, h)) return false;
        if (h.kind == HIT_TRI && is_source_tri(q, h.obj, h.prim)) {
            self = pi + 1;
            return false;
        }
        const uint64_t key = hit_key(h.obj, h.prim);
        if (h.t < best.t || (h.t == best.t && key < bkey)) best = h, bkey = key, tmax = fminf(tmax, h.t);
        return false;
    });
    auto take = [&](const Hit &h, uint64_t key) {
        if (h.t < best.t || (h.t == best.t && key < bkey)) best = h, bkey = key;
    };
    auto from = [&](auto x) {
        constexpr int X = decltype(x)::value;
        const Hit h{quad_xor<X>(best.t), quad_xor<X>(best.kind), quad_xor<X>(best.obj), quad_xor<X>(best.prim),
                    quad_xor<X>(best.w), quad_xor<X>(best.u), quad_xor<X>(best.v)};
        const uint64_t key = (uint64_t)(uint32_t)quad_xor<X>((int)(bkey >> 32)) << 32 |
                             (uint32_t)quad_xor<X>((int)(uint32_t)bkey);
        take(h, key);
    };
    from(std::integral_constant<int, 1>());
    from(std::integral_constant<int, 2>());
    self = quad_or(self);  // one slot: the triangle is in one leaf
    if (self) take_source_hit(S, q, self - 1, before, best, bkey);
    return best;
}

// trace_any; every lane of the quad gets the answer.
__device__ inline bool quad_any(const SceneView &S, const TraceRay &q, float dis, QuadStack &st) {
    Hit dummy{kMiss, HIT_NONE, -1, -1, 0, 0, 0};
    if (brute_objects(S, q, true, dis, dummy)) return true;
    int blocked = 0, self = 0;
    float tmax = dis;
    quad_walk<false>(S, q.r, tmax, st, [&](int pi) -> bool {
        if (any_prim(q, load_prim(S, pi), dis, self)) blocked = 1;
        return blocked != 0;
    });
    if (quad_or(blocked)) return true;
    return quad_or(self) && self_testable(S, q.r, q.src, dis);
}

}  // namespace rtg
