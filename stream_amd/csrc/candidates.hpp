// Candidate search of the alpha-shapes (DirectAlphaShape2D.cpp:310-357,
// DirectAlphaShape3D.cpp:310-363): the nodes within 2 delta min(alpha_i,
// alpha_j) of a node, in the order in which a depth-first walk of the LBVH
// meets them.  The walk pushes the hit children of a visited node in order and
// visits the last one pushed next; leaf children are tested at the visit.
#pragma once
#include "lbvh.hpp"

namespace stream_amd {

template <class S, int D> struct CandTree {
    uint32_t n;
    const Sph4<S>* P;        // Morton order
    const uint32_t* node;    // internal nodes: sep | child_is_leaf << 30
    const BoxD<S, D>* ibox;  // internal boxes
};

// Internal child c: its word, and whether its box reaches into the ball of
// radius rs around the node's centre.
template <class S, int D>
__device__ __forceinline__ bool cand_hit_box(const CandTree<S, D>& t, const Sph4<S>& si, S rs, uint32_t c,
                                             uint32_t* word) {
    const BoxD<S, D> bb = t.ibox[c];
    *word = t.node[c];
    S d = (S)0;
#pragma unroll
    for (int k = 0; k < D; ++k) {
        const S hi = fmax(si.c[k] - bb.hi[k], (S)0), lo = fmax(bb.lo[k] - si.c[k], (S)0);
        d = k == 0 ? hi * hi + lo * lo : d + hi * hi + lo * lo;
    }
    return d < rs * rs;
}
// Leaf child c.
template <class S, int D>
__device__ __forceinline__ bool cand_hit_leaf(const CandTree<S, D>& t, const Sph4<S>& si, S two_delta, uint32_t c) {
    const Sph4<S> sj = t.P[c];
    const S ma = fmin(si.r, sj.r);
    S sq = (S)0;
#pragma unroll
    for (int k = 0; k < D; ++k) {
        const S d = si.c[k] - sj.c[k];
        sq = k == 0 ? d * d : sq + d * d;
    }
    return sq < (two_delta * ma) * (two_delta * ma);
}

// The walk by one lane (for what cand_group leaves).  take(c) receives the
// candidates and returns false to end the walk after this visit.  A full stack
// (64 deep with the register) raises the capacity error, drops the second
// child and visits the first.
template <class S, int D, class Take>
__device__ void cand_walk(const CandTree<S, D>& t, uint32_t tid, const Sph4<S>& si, S two_delta, uint32_t* flags,
                          Take&& take) {
    const S rs = two_delta * si.r;
    uint32_t stack[63];
    int ss = 0;
    bool live = t.n >= 2;
    uint32_t w = live ? t.node[0] : 0u;
    // a valid tree has n - 1 internal nodes: the visit cap only guards a
    // malformed topology
    for (uint32_t visits = 0; live; ++visits) {
        if (visits >= t.n) {
            raise_flag(flags, kErrCapacity);
            return;
        }
        const uint32_t sep = w & 0x3fffffffu, cl = w >> 30;
        bool hit[2] = {false, false}, more = true;
        uint32_t wc[2] = {0u, 0u};
#pragma unroll
        for (uint32_t ch = 0; ch < 2; ++ch) {
            const uint32_t c = sep + ch;
            if (!(cl & (ch + 1)))
                hit[ch] = cand_hit_box(t, si, rs, c, &wc[ch]);
            else if (tid != c && cand_hit_leaf(t, si, two_delta, c))
                more &= take(c);
        }
        if (!more) return;
        if (hit[0] && hit[1]) {
            if (ss < 63) {
                stack[ss++] = wc[0];
                w = wc[1];
            } else {
                raise_flag(flags, kErrCapacity);
                w = wc[0];
            }
        } else if (hit[0] || hit[1]) {
            w = hit[1] ? wc[1] : wc[0];
        } else if (ss != 0) {
            w = stack[--ss];
        } else {
            live = false;
        }
    }
}

// The same by G lanes (8 or 16, aligned in the wavefront).  The stack holds
// what the walk has still to visit, next on top, and candidates behind it.
// Each round the top G entries are replaced by what a visit leaves of each, in
// order: its leaf candidates, then its hit internal children, the last first.
// Candidates with nothing to visit before them leave through out(j, c).  So
// the order is the walk's, while a round trip to memory serves G visits
// instead of one.  Bound: that round trip.  One lane per node -> 16, 3D: 20,102
// FP32 nodes (79 blocks before) 313 -> 51 us, 100,000 FP32 263 -> 150 us,
// 299,000 FP64 1.50 -> 0.81 ms.
// Returns false, with candidates already written, when the stack overflows or
// when a visit is 63 or more levels deep (only there the walk's own stack can
// overflow, an error of its own).  *count is the number found; the search ends
// early, with the first ones right, once it exceeds `limit`.
template <int CAP> struct CandStack {
    uint32_t w[CAP];  // node word, or leaf
    uint8_t t[CAP];   // level, kCandLeaf for a leaf
};
constexpr uint32_t kCandLeaf = 128u;
template <int G> __device__ __forceinline__ uint32_t cand_bits(bool b, uint32_t grp) {
    const uint64_t m = __builtin_amdgcn_ballot_w64(b);
    constexpr uint32_t per = 32 / G;
    const uint32_t h = grp >= per ? (uint32_t)(m >> 32) : (uint32_t)m;
    return (h >> ((grp % per) * G)) & ((1u << G) - 1u);
}
__device__ __forceinline__ void cand_sync() {
    // one wavefront: program order is execution order for LDS
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
template <class S, int D, int G, int CAP, class Out>
__device__ bool cand_group(const CandTree<S, D>& t, uint32_t tid, const Sph4<S>& si, S two_delta, uint32_t sub,
                           uint32_t grp, CandStack<CAP>& L, uint32_t limit, uint32_t* count, Out&& out) {
    const S rs = two_delta * si.r;
    uint32_t top = t.n >= 2 ? 1u : 0u, found = 0;
    if (sub == 0 && top) {
        L.w[0] = t.node[0];
        L.t[0] = 0;
    }
    cand_sync();
    const uint32_t below = (1u << sub) - 1u;
    bool ok = true;
    while (top && ok && found <= limit) {
        const uint32_t take = min(top, (uint32_t)G), bottom = top - take;
        uint32_t v0 = 0, v1 = 0, level = 0;
        bool e0 = false, e1 = false, l0 = false, l1 = false;  // outputs: present, leaf
        if (sub < take) {
            const uint32_t w = L.w[top - 1 - sub], tag = L.t[top - 1 - sub];
            if (tag & kCandLeaf) {
                e0 = l0 = true;
                v0 = w;
            } else {
                level = tag + 1;
                const uint32_t sep = w & 0x3fffffffu, cl = w >> 30;
                const bool leaf0 = cl & 1u, leaf1 = cl & 2u;
                uint32_t w0 = sep, w1 = sep + 1;
                const bool h0 = leaf0 ? tid != sep && cand_hit_leaf(t, si, two_delta, sep)
                                      : cand_hit_box(t, si, rs, sep, &w0);
                const bool h1 = leaf1 ? tid != sep + 1 && cand_hit_leaf(t, si, two_delta, sep + 1)
                                      : cand_hit_box(t, si, rs, sep + 1, &w1);
                // leaves before internal children, of two internal ones the second
                e0 = leaf0 ? h0 : h1;
                v0 = leaf0 ? w0 : w1;
                l0 = leaf0 ? true : leaf1;
                e1 = leaf0 ? h1 : h0;
                v1 = leaf0 ? w1 : w0;
                l1 = leaf0 ? leaf1 : false;
            }
        }
        if (!e0) {
            e0 = e1;
            v0 = v1;
            l0 = l1;
            e1 = false;
        }
        const uint32_t b0 = cand_bits<G>(e0, grp), b1 = cand_bits<G>(e1, grp);
        const uint32_t bl = cand_bits<G>(e0 && l0, grp), bi = cand_bits<G>((e0 && !l0) || (e1 && !l1), grp);
        const uint32_t off = __popc(b0 & below) + __popc(b1 & below), m = __popc(b0) + __popc(b1);
        uint32_t first = m;  // outputs before the first one to visit
        if (bi) {
            const uint32_t k = (uint32_t)__builtin_ctz(bi), bk = (1u << k) - 1u;
            first = __popc(b0 & bk) + __popc(b1 & bk) + ((bl >> k) & 1u);
        }
        top = bottom + (m - first);
        ok = top <= (uint32_t)CAP && !cand_bits<G>(level >= 63, grp);
        cand_sync();
        if (ok) {
            auto put = [&](uint32_t q, uint32_t v, bool leaf) {
                if (q < first) {
                    out(found + q, v);
                } else {
                    const uint32_t at = bottom + (m - 1 - q);
                    L.w[at] = v;
                    L.t[at] = (uint8_t)(leaf ? kCandLeaf : level);
                }
            };
            if (e0) put(off, v0, l0);
            if (e1) put(off + 1, v1, l1);
        }
        found += first;
        cand_sync();
    }
    *count = found;
    return ok;
}

}  // namespace stream_amd
