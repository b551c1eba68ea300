// rt_quad.hpp — a wave's rays walked together: a lane per ray, then four lanes
// per ray, then every idle lane on the rays that are left.
//
// A wave that walks 64 rays takes about a microsecond a step whatever else the
// GPU does: a node's loads, then the tests of its four children one after
// another, and it runs as long as its slowest ray.  Where a level holds fewer
// rays than the GPU has lanes (the deep levels of a frame, small frames and
// batches), and at the end of longer levels, that chain is the kernel's time.
// So four neighbouring lanes (a quad) share a ray: each tests one child of a
// node, or one primitive of the two leaves it postponed, and the results meet in
// cross-lane moves.  A short queue starts with quads, 16 rays a wave; a wave of
// 64 rays goes on with quads once 16 are left; and quads whose rays are done
// take over subtrees of those still walking.
//
// us a call, lane by lane and short queues by quads -> this: 12 thumbnails in a
// batch 1273 -> 895, burst of 32 requests 1861 -> 1479, 60 mixed requests 6765 ->
// 5704, 801x451 frame at 4 samples 1854 -> 1762, 1080p frame 1962 -> 1909,
// 1280x720 normal view 423 -> 405, 64x64 frame unchanged.
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
// Queues of up to this many rays per CU are walked by quads from the start
// (98,304 on 256 CUs): a quad spends about half the instructions of a whole ray
// on a quarter of its lanes, so longer queues keep every lane busy with a ray of
// its own first.  Limits of 48k / 96k / 192k rays (us a call, against the same
// start): 64x64 frame 208 of 203 / 197 of 198 / 196 of 196; 1080p frame 1776 of
// 1838 / 1909 of 1962 / 1786 of 1827; 801x451 at 4 samples 1796 of 1881 / 1762
// of 1854 / 1928 of 1832; burst of 32 requests 1568 of 1954 / 1479 of 1861 /
// 1532 of 1845.
constexpr int kQuadRaysPerCu = 24 * 16;
// Queues of up to this many rays per CU (4,096 on 256 CUs) go four to a wave, a
// wave on every SIMD, and its twelve other quads take subtrees over from the
// second round on.  Limits of 4k / 16k / 32k rays, against quads alone: 64x64
// frame 1.06 / 1.03 / 1.05x, 12 thumbnails in a batch 1.10 / 1.05 / 1.01x, burst
// of 32 requests 1.04 / 1.02 / 0.96x, 1080p frame 1.00 / 1.00 / 0.99x.
constexpr int kFewRaysPerCu = 16;

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
// entry e in row e / 4, column e % 4 of their LDS columns; past kLds entries in
// the first lane's spill column.  The last kRec words are the record of the
// quad's own ray (QuadRec).  An entry is written by the lane that holds the
// child and read by all four; a wave's accesses to LDS, and to one global
// address, are done in order, and the fences keep the compiler from moving
// them.  Entry `base` is kWalkDone (see DevStack): helpers take entries from
// the bottom.
enum QuadRec { REC_BOUND, REC_SELF, REC_CLAIM, REC_T, REC_OBJ, REC_PRIM, REC_KIND, REC_W, REC_U, REC_V, REC_GIVER };
struct QuadStack {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef int __attribute__((address_space(3))) LdsInt;
#else
    typedef int LdsInt;
#endif
    LdsInt *lds;   // this quad's columns
    LdsInt *wave;  // the wave's columns
    int *spill;
    int gstride;
    int sp, base;
    const Bvh4Node *top;
    static constexpr int kRec = 12, kLds = kLdsStack * kQuadLanes - kRec;
    __device__ explicit QuadStack(const DevStack &st, int *lds_base)
        : lds((LdsInt *)(lds_base + (threadIdx.x & ~(kQuadLanes - 1)))), wave((LdsInt *)(lds_base + (threadIdx.x & ~63))),
          spill(st.spill - (threadIdx.x & (kQuadLanes - 1))), gstride(st.gstride), sp(0), base(0), top(st.top) {}
    __device__ static void order() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    static __device__ unsigned at(unsigned e) { return (e / kQuadLanes) * kBlockThreads + e % kQuadLanes; }
    // Word w of the record of the wave's quad r.
    __device__ LdsInt &rec(int r, int w) const { return wave[r * kQuadLanes + at(kLds + w)]; }
    // Entry e of the wave's quad r.
    __device__ LdsInt &entry(int r, int e) const { return wave[r * kQuadLanes + at(e)]; }
    // Every lane of the quad calls it.
    __device__ void reset() {
        put_lds(0, kWalkDone);
        sp = 1, base = 0;
    }
    __device__ void put_lds(int e, int v) {
        lds[at(e)] = v;
        __asm__ volatile("" ::: "memory");
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
        if (__ballot(sp >= kLds) == 0ull) {
            v = lds[at(sp)];
            __asm__ volatile("" ::: "memory");  // not merged with the spill read into a flat load
        } else if (sp < kLds) {
            v = lds[at(sp)];
            __asm__ volatile("" ::: "memory");
        } else {
            v = spill[(sp - kLds) * gstride];
        }
        order();
        return v;
    }
    template <int N, int D>
    __device__ bool lanes_at_least(bool v) const {
        return D * __popcll(__ballot(v)) >= N * __popcll(__ballot(true));
    }
    // Node i's bounds, and the link of its child k.
    __device__ Bvh4Node node(const Bvh4Node *nodes, int i, int k, int &link) const {
        Bvh4Node n{};
#if defined(__HIP_DEVICE_COMPILE__)
        typedef const Bvh4Node __attribute__((address_space(3))) LdsNode;
        typedef const int __attribute__((address_space(3))) LdsConst;
        if (top != nullptr && i < kTopNodes) {
            n.org = ((LdsNode *)top)[i].org, n.qxy = ((LdsNode *)top)[i].qxy, n.qz = ((LdsNode *)top)[i].qz;
            link = ((LdsConst *)top)[i * (int)(sizeof(Bvh4Node) / 4) + 12 + k];
            __asm__ volatile("" ::: "memory");
            return n;
        }
#endif
        const Bvh4Node &g = nodes[i];
        n.org = g.org, n.qxy = g.qxy, n.qz = g.qz;
        link = (&g.link.x)[k];
        return n;
    }
};
static_assert(REC_GIVER < QuadStack::kRec, "the record fits");
static_assert(QuadStack::kLds + (kStackMax - kLdsStack) >= kStackMax, "a quad's stack holds any walk");

// Hit a is nearer than b, or as near and of the lower key (no hit is as near
// as HIT_NONE's kMiss).
__device__ inline bool closer(const Hit &a, const Hit &b) {
    return a.t < b.t || (a.t == b.t && hit_key(a.obj, a.prim) < hit_key(b.obj, b.prim));
}

// Idle quads of a wave take work over once there are this many of them, after
// this many rounds of the wave: earlier, and for fewer, the hand-over (some 200
// instructions of the whole wave) costs rays that would soon be done (from 4
// quads after 6 rounds, 64x64 frame 207.7 -> 209.5 us; from 8 after 8, 208.7 ->
// 208.5; 12 thumbnails gain 1.2-1.4x with either).
constexpr int kHelpFrom = 8, kHelpAfter = 8;
// A wave's last 16 rays go on as quads, after this many rounds (4 and 12: 60
// mixed requests 1.04x and 0.96x, 801x451 at 4 samples 1.016x and 1.003x of the
// walk without it).
constexpr int kTailAfter = 4;

// The walks of a wave's 1 << lg rays, bvh_walk<true, kOrdered> with a lane
// (lg 6) or a quad per ray: the same postponed leaves and wave-wide exit of the
// node loop.  Every lane of the wave calls it; lanes without a ray come with
// root kWalkDone.
//
// A wave runs as long as its slowest ray, and a level as long as the slowest
// of all: a few rays that graze a surface visit a thousand nodes where the
// others visit thirty.  So a quad whose own walk is over takes the bottom
// entry, the largest subtree left, off the stack of a quad that still walks,
// and walks it with that quad's ray.  Once a wave does so, its rays' results
// meet in their records in LDS: REC_BOUND is the closest distance found by any
// of a ray's quads (closest hit), or -1 once one found a blocker (any hit), and
// is read before every round; a finished quad whose hit is that close leaves it
// in REC_T.. unless an equal hit of lower key is there.  Subtrees are disjoint
// and the winner is the least (t, key), so the result does not depend on who
// walks what.
//
// Closest hit: `best` comes as the closest hit outside the BVH and leaves as
// the closest of all; `self` leaves as 1 + slot of the source triangle where
// the ray hits it.  Any hit: best.t comes as the segment's length; returns
// whether the segment is blocked.
template <bool kOrdered, bool kOneScene>
__device__ inline bool wave_rays(int lg, const SceneView &S0, const Bvh4Node *nodes, const float4 *prims, int root,
                                 TraceRay q, int before, DevStack &ds, int *lds_base, Hit &best, int &self) {
    const bool quads = lg < 6;
    const int lane = __lane_id(), k = lane & (kQuadLanes - 1), me = lane / kQuadLanes;
    const int help_after = lg < 4 ? 1 : kHelpAfter;
    const unsigned long long leaders = 0x1111111111111111ull;
    V3 inv = safe_inv(q.r.d);
    float tmax = best.t;
    int node = root, leaf = 0, leaf2 = 0;  // postponed leaves (< 0), or 0
    int blocked = 0;
    self = 0;
    QuadStack st(ds, lds_base);
    // One primitive of the lane's ray; true: it blocks the segment (any hit).
    auto test = [&](int pi, bool shared_bound, int owner) -> bool {
        const PrimRec R = load_prim(kOneScene ? S0.prims : prims, pi);
        if constexpr (!kOrdered) {
            return any_prim(q, R, tmax, self);
        } else {
            Hit h;
            if (!closest_prim(q, R, before, h)) return false;
            if (h.kind == HIT_TRI && is_source_tri(q, h.obj, h.prim)) {
                self = pi + 1;
                return false;
            }
            if (closer(h, best)) {
                best = h, tmax = fminf(tmax, h.t);
                if (shared_bound)  // (hits are at t > 0, where floats order as their bits do)
                    __hip_atomic_fetch_min(&st.rec(owner, REC_BOUND), as_int(h.t), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WAVEFRONT);
            }
            return false;
        }
    };
    // ---- a lane per ray (bvh_walk<true, kOrdered>), until a quad per ray will do
    unsigned long long rest = 0ull;  // the lanes whose rays go on as quads
    Hit lane_best = best;
    int lane_self = 0, lane_blocked = 0;
    if (!quads) {
        ds.reset();
        for (int round = 0;; ++round) {
            const bool busy = node != kWalkDone || leaf < 0;
            rest = __ballot(busy);
            if (rest == 0ull) return blocked != 0;
            if (round >= kTailAfter && __popcll(rest) <= 64 / kQuadLanes && __ballot(busy && ds.sp > kLdsStack) == 0ull)
                break;
            while (node >= 0) {
                node = node_step<kOrdered>(kOneScene ? S0.nodes : nodes, node, q.r.o, inv, tmax, ds);
                if (node < 0 && node != kWalkDone && leaf2 == 0) {
                    (leaf == 0 ? leaf : leaf2) = node;
                    node = ds.pop();
                }
                if (kOrdered ? ds.template lanes_at_least<1, 2>(leaf != 0) : ds.template lanes_at_least<3, 4>(leaf != 0))
                    break;
            }
            if (leaf == 0 && node < 0 && node != kWalkDone) {
                leaf = node;
                node = ds.pop();
            }
            // one loop over the primitives of every held leaf, so that a lane
            // with a short leaf goes on with its next one
            if (leaf < 0) {
                int pi = leaf_first(leaf), end = pi + leaf_count(leaf);
                for (;;) {
                    if (test(pi, false, 0)) {
                        blocked = 1;
                        node = kWalkDone;
                        break;
                    }
                    if (++pi < end) continue;
                    leaf = leaf2, leaf2 = 0;
                    if (leaf == 0 && node < 0 && node != kWalkDone) {
                        leaf = node;
                        node = ds.pop();
                    }
                    if (leaf == 0) break;
                    pi = leaf_first(leaf), end = pi + leaf_count(leaf);
                }
                leaf = leaf2 = 0;
            }
        }
        // Ray r of the rest moves to quad r, with its stack (all in LDS).
        lane_best = best, lane_self = self, lane_blocked = blocked;
        int src = lane;
        unsigned long long m = rest;
        for (int r = 0; m != 0ull; ++r, m &= m - 1ull)
            if (r == me) src = __builtin_ctzll(m);
        const bool moved = me < __popcll(rest);
        QuadStack::order();
        int e[kLdsStack / kQuadLanes];
#pragma unroll
        for (int j = 0; j < kLdsStack / kQuadLanes; ++j) e[j] = st.wave[src + (j * kQuadLanes + k) * kBlockThreads];
        QuadStack::order();
#pragma unroll
        for (int j = 0; j < kLdsStack / kQuadLanes; ++j) st.wave[lane + j * kBlockThreads] = e[j];
        QuadStack::order();
        auto move = [&](auto &x) { x = __shfl(x, src, 64); };
        auto move64 = [&](auto &x) {
            x = (std::remove_reference_t<decltype(x)>)__shfl((unsigned long long)x, src, 64);
        };
        move(q.r.o.x), move(q.r.o.y), move(q.r.o.z), move(q.r.d.x), move(q.r.d.y), move(q.r.d.z);
        move(inv.x), move(inv.y), move(inv.z), move(q.inside), move(q.src.obj), move(q.src.prim);
        move(tmax), move(node), move(leaf), move(leaf2), move(self);
        if constexpr (kOrdered) {
            move(best.t), move(best.kind), move(best.obj), move(best.prim), move(best.w), move(best.u), move(best.v);
            move(before);
        }
        if constexpr (!kOneScene) move64(nodes), move64(prims);
        st.sp = __shfl(ds.sp, src, 64), st.base = 0;
        blocked = 0;
        if (!moved) node = kWalkDone, leaf = leaf2 = 0;
    } else {
        st.reset();
    }
    // ---- a quad per ray
    int owner = me;       // the quad whose ray this quad walks
    bool helped = false;  // (wave-uniform) a quad took over work: the records are in use
    bool saved = false;   // the owner's record has this quad's result
    auto step = [&](int nd) -> int {
        int link;
        const Bvh4Node n = st.node(kOneScene ? S0.nodes : nodes, nd, k, link);
        const Node4Test nt(n, q.r.o, inv);
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
            const uint32_t m = (uint32_t)(__ballot(h) >> (lane & ~3)) & 15u;
            rank = __popc(m & ((1u << k) - 1u));
            hits = __popc(m);
        }
        const int next = quad_or(h && rank == 0 ? link : 0);
        st.put(h && rank > 0, st.sp + hits - 1 - rank, link);
        if (hits == 0) return st.pop();
        st.sp += hits - 1;
        return next;
    };
    // The closest of the four lanes' hits, in all of them.
    auto join_lanes = [&]() {
        auto from = [&](auto x) {
            constexpr int X = decltype(x)::value;
            const Hit h{quad_xor<X>(best.t),    quad_xor<X>(best.kind), quad_xor<X>(best.obj),
                        quad_xor<X>(best.prim), quad_xor<X>(best.w),    quad_xor<X>(best.u),
                        quad_xor<X>(best.v)};
            if (closer(h, best)) best = h;
        };
        from(std::integral_constant<int, 1>());
        from(std::integral_constant<int, 2>());
    };
    // Quads with `save` leave their results in their owners' records.
    auto save_results = [&](bool save) {
        save = save && !saved;
        saved = saved || save;
        if (save && self) st.rec(owner, REC_SELF) = self;  // (one slot: the triangle is in one leaf)
        if constexpr (kOrdered) {
            if (save) join_lanes();
            for (;;) {
                bool mine = save && best.kind != HIT_NONE && best.t == as_float(st.rec(owner, REC_BOUND));
                if (mine) {
                    const float rt = as_float(st.rec(owner, REC_T));
                    mine = best.t < rt || hit_key(best.obj, best.prim) < hit_key(st.rec(owner, REC_OBJ), st.rec(owner, REC_PRIM));
                }
                if (__ballot(mine) == 0ull) break;
                // of several quads with one owner, one at a time
                if (mine && k == 0) st.rec(owner, REC_CLAIM) = me;
                QuadStack::order();
                if (mine && st.rec(owner, REC_CLAIM) == me) {
                    st.rec(owner, REC_T) = as_int(best.t), st.rec(owner, REC_KIND) = best.kind;
                    st.rec(owner, REC_OBJ) = best.obj, st.rec(owner, REC_PRIM) = best.prim;
                    st.rec(owner, REC_W) = as_int(best.w), st.rec(owner, REC_U) = as_int(best.u);
                    st.rec(owner, REC_V) = as_int(best.v);
                    save = false;
                }
                QuadStack::order();
            }
        }
    };
    for (int round = 0;; ++round) {
        const bool busy = node != kWalkDone || leaf < 0;
        const unsigned long long idle = ~__ballot(busy) & leaders;
        if (idle == leaders) break;
        if (round >= help_after && __popcll(idle) >= kHelpFrom) {
            const bool spare = busy && st.sp - st.base > 1 && st.base + 1 < QuadStack::kLds;
            const unsigned long long give = __ballot(spare) & leaders;
            if (give != 0ull) {
                QuadStack::order();
                if (!helped) {
                    helped = true;
                    if (k == 0) {
                        st.rec(me, REC_BOUND) = as_int(blocked ? -1.0f : tmax);
                        st.rec(me, REC_SELF) = 0, st.rec(me, REC_T) = as_int(kMiss), st.rec(me, REC_KIND) = HIT_NONE;
                    }
                    QuadStack::order();
                }
                const unsigned long long below = (1ull << (lane & ~(kQuadLanes - 1))) - 1ull;
                const int pairs = min(__popcll(give), __popcll(idle));
                const int rank = __popcll((busy ? give : idle) & below);  // among the givers, or the takers
                const bool takes = !busy && rank < pairs;
                save_results(takes);
                if (spare && rank < pairs && k == 0) st.rec(rank, REC_GIVER) = me;
                QuadStack::order();
                const int from = takes ? st.rec(rank, REC_GIVER) : me;
                const int src = from * kQuadLanes + k;  // (every lane reads its own values unless it takes over)
                const int gbase = __shfl(st.base, src, 64);
                q.r.o = V3{__shfl(q.r.o.x, src, 64), __shfl(q.r.o.y, src, 64), __shfl(q.r.o.z, src, 64)};
                q.r.d = V3{__shfl(q.r.d.x, src, 64), __shfl(q.r.d.y, src, 64), __shfl(q.r.d.z, src, 64)};
                inv = V3{__shfl(inv.x, src, 64), __shfl(inv.y, src, 64), __shfl(inv.z, src, 64)};
                q.inside = __shfl(q.inside, src, 64);
                q.src.obj = __shfl(q.src.obj, src, 64), q.src.prim = __shfl(q.src.prim, src, 64);
                owner = __shfl(owner, src, 64);
                if constexpr (kOrdered) before = __shfl(before, src, 64);
                if constexpr (!kOneScene) {
                    nodes = reinterpret_cast<const Bvh4Node *>(__shfl(reinterpret_cast<unsigned long long>(nodes), src, 64));
                    prims = reinterpret_cast<const float4 *>(__shfl(reinterpret_cast<unsigned long long>(prims), src, 64));
                }
                if (takes) {
                    node = st.entry(from, gbase + 1);
                    if constexpr (kOrdered) best = Hit{kMiss, HIT_NONE, -1, -1, 0, 0, 0};
                    self = blocked = 0, saved = false;
                }
                QuadStack::order();
                if (takes) st.reset();
                if (spare && rank < pairs) {
                    ++st.base;
                    st.put_lds(st.base, kWalkDone);
                }
                QuadStack::order();
            }
        }
        if (helped) {
            QuadStack::order();
            tmax = as_float(st.rec(owner, REC_BOUND));
            if (!kOrdered && tmax < 0.0f) {  // blocked
                node = kWalkDone, leaf = leaf2 = 0;
                st.sp = st.base;
            }
        }
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
                for (int i = k & 1; i < count; i += 2) stop |= test(first + i, helped, owner) ? 1 : 0;
            }
            if constexpr (kOrdered) {
                tmax = quad_min(tmax);
            } else if (quad_or(stop)) {
                blocked = 1;
                if (helped && k == 0) st.rec(owner, REC_BOUND) = as_int(-1.0f);
                node = kWalkDone, leaf = leaf2 = 0;
                st.sp = st.base;
                break;
            }
            leaf = leaf2 = 0;
            if (node < 0 && node != kWalkDone) {
                leaf = node;
                node = st.pop();
            }
        }
    }
    if (!helped) {
        self = quad_or(self);
        if constexpr (kOrdered) join_lanes();
    } else {
        QuadStack::order();
        save_results(true);
        QuadStack::order();
        self = st.rec(me, REC_SELF);
        if constexpr (kOrdered) {
            const int kind = st.rec(me, REC_KIND);
            best = Hit{kMiss, HIT_NONE, -1, -1, 0, 0, 0};
            if (kind != HIT_NONE)
                best = Hit{as_float(st.rec(me, REC_T)), kind, st.rec(me, REC_OBJ), st.rec(me, REC_PRIM),
                           as_float(st.rec(me, REC_W)), as_float(st.rec(me, REC_U)), as_float(st.rec(me, REC_V))};
        }
        blocked = as_float(st.rec(me, REC_BOUND)) < 0.0f;
        QuadStack::order();
    }
    if (quads) return blocked != 0;
    // ---- back to the lanes
    const bool mine = (rest >> lane) & 1ull;
    const int src = mine ? __popcll(rest & ((1ull << lane) - 1ull)) * kQuadLanes : lane;
    auto back = [&](auto &x, auto kept) {
        const auto v = __shfl(x, src, 64);
        x = mine ? v : kept;
    };
    back(self, lane_self), back(blocked, lane_blocked);
    if constexpr (kOrdered) {
        back(best.t, lane_best.t), back(best.kind, lane_best.kind), back(best.obj, lane_best.obj);
        back(best.prim, lane_best.prim), back(best.w, lane_best.w), back(best.u, lane_best.u);
        back(best.v, lane_best.v);
    }
    return blocked != 0;
}

// trace_closest<false, true> and trace_any of the wave's 1 << lg rays (those of
// lanes with `valid`), a lane or, with lg < 6, a quad per ray.  All lanes of the
// wave call it; every lane of a quad gets its ray's answer.
template <bool kOneScene>
__device__ inline Hit wave_closest(int lg, const SceneView &S, const TraceRay &q, DevStack &st, int *lds, int before,
                                   bool valid) {
    Hit best{kMiss, HIT_NONE, -1, -1, 0, 0, 0};
    int root = kWalkDone, self;
    const Bvh4Node *nodes = nullptr;
    const float4 *prims = nullptr;
    if (valid) {
        brute_objects(S, q, false, 0.0f, best, before);
        if (S.n_prims > 0) root = S.root, nodes = S.nodes, prims = S.prims;
    }
    wave_rays<true, kOneScene>(lg, S, nodes, prims, root, q, before, st, lds, best, self);
    if (self) take_source_hit(S, q, self - 1, before, best, best.kind != HIT_NONE ? hit_key(best.obj, best.prim) : ~0ull);
    return best;
}
template <bool kOneScene>
__device__ inline bool wave_any(int lg, const SceneView &S, const TraceRay &q, float dis, DevStack &st, int *lds,
                                bool valid) {
    Hit best{dis, HIT_NONE, -1, -1, 0, 0, 0};
    int root = kWalkDone, self;
    const Bvh4Node *nodes = nullptr;
    const float4 *prims = nullptr;
    bool blocked = false;
    if (valid) {
        Hit dummy{kMiss, HIT_NONE, -1, -1, 0, 0, 0};
        blocked = brute_objects(S, q, true, dis, dummy);
        if (S.n_prims > 0 && !blocked) root = S.root, nodes = S.nodes, prims = S.prims;
    }
    if (wave_rays<false, kOneScene>(lg, S, nodes, prims, root, q, 0, st, lds, best, self)) blocked = true;
    return blocked || (self && self_testable(S, q.r, q.src, dis));
}

}  // namespace rtg
