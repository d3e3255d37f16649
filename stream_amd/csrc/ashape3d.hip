// 3D alpha-shape kernels and the AlphaShape3D C-ABI (see ashape3d.hpp).
#include <chrono>
#include <vector>

#include "ashape3d.hpp"
#include "candidates.hpp"
#include "predicates.hpp"

namespace stream_amd {

template <class S> struct Consts3D;
template <> struct Consts3D<float> {
    // 2*delta (DirectAlphaShape3D.cpp:196,335): 2 + 2^-21 in float
    static constexpr float two_delta = 2.0000004768371866248429007339848490744624f;
};
template <> struct Consts3D<double> {
    static constexpr double two_delta = 2.0 + 0x1p-50;
};

template <class S> struct Ash3Args {
    uint32_t n;
    const Sph4<S>* P;        // Morton-ordered points + infinity nodes
    const uint32_t* node;    // LBVH internal nodes
    const BoxD<S, 3>* ibox;  // LBVH internal boxes
    uint32_t* cand;
    uint32_t* tet;
    uint8_t* active;
    uint32_t* nineig;
    uint32_t* nfneig;
    uint8_t* node_is_bnd;
    uint8_t* nelem;
    uint8_t* nelem_out;
    uint32_t* queue;
    uint32_t* flags;
};

namespace {

constexpr uint32_t kEmpty = 255u;

__device__ __forceinline__ uint32_t pack_tet(uint32_t a, uint32_t b, uint32_t c) { return a | (b << 8) | (c << 16); }

// Infinity nodes (cpp:144-170) from the global sphere box, radius 1.
template <class S> __global__ void infinity3_kernel(const BoxD<S, 3>* gbox, Sph4<S>* P, uint32_t n) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const BoxD<S, 3> g = *gbox;
    S avg[3], range[3];
    for (int a = 0; a < 3; ++a) {
        avg[a] = (S)0.5 * (g.hi[a] + g.lo[a]);
        range[a] = g.hi[a] - g.lo[a];
    }
    const S mr = fmax(range[0], fmax(range[1], range[2]));
    Sph4<S> p;
    p.r = (S)1;
    p.c[0] = avg[0] - 2 * mr; p.c[1] = avg[1] - 2 * mr; p.c[2] = avg[2] - 2 * mr;
    P[n] = p;
    p.c[0] = avg[0] + 2 * mr; p.c[1] = avg[1] - 2 * mr; p.c[2] = avg[2] - 2 * mr;
    P[n + 1] = p;
    p.c[0] = avg[0] + 2 * mr; p.c[1] = avg[1] + 2 * mr; p.c[2] = avg[2] - 2 * mr;
    P[n + 2] = p;
    p.c[0] = avg[0]; p.c[1] = avg[1]; p.c[2] = avg[2] + 2 * mr;
    P[n + 3] = p;
}

// Candidate search (candidates.hpp), 16 lanes per node.  The first 124
// candidates are kept (the reference clamps its list to 128 entries including
// the 4 infinity nodes and warns), queue[1] counts clamped nodes.
constexpr int kFillLanes3D = 16, kFillStack3D = 192;
constexpr uint32_t kFillBlock = 256;
template <class S> __global__ __launch_bounds__(kFillBlock) void fill3_kernel(Ash3Args<S> a, uint32_t blocks_per_xcd) {
    constexpr uint32_t G = kFillLanes3D, NPB = kFillBlock / G;
    __shared__ CandStack<kFillStack3D> lds[NPB];
    const uint32_t sub = threadIdx.x % G, slot = threadIdx.x / G, grp = slot % (64 / G);
    const uint32_t tid = ((blockIdx.x & 7u) * blocks_per_xcd + (blockIdx.x >> 3)) * NPB + slot;
    if (tid >= a.n) return;
    const CandTree<S, 3> t{a.n, a.P, a.node, a.ibox};
    const Sph4<S> si = a.P[tid];
    const S two_delta = Consts3D<S>::two_delta;
    auto store = [&](uint32_t j, uint32_t c) {
        if (j < kCand3D) a.cand[slab3(tid, j, kCand3D)] = c;
    };
    uint32_t found = 0;
    if (!cand_group<S, 3, (int)G>(t, tid, si, two_delta, sub, grp, lds[slot], kCand3D, &found, store) && sub == 0) {
        found = 0;
        cand_walk(t, tid, si, two_delta, a.flags, [&](uint32_t c) {
            store(found++, c);
            return found <= kCand3D;
        });
    }
    if (sub != 0) return;
    if (found > kCand3D) atomicAdd(&a.queue[1], 1u);
    a.nineig[tid] = kNInf3D + min(found, kCand3D);
}

template <class S> __device__ __forceinline__ void load3(const Sph4<S>* P, uint32_t i, S* p) {
    const Sph4<S> s = P[i];
    p[0] = s.c[0];
    p[1] = s.c[1];
    p[2] = s.c[2];
}

// LDS written by other lanes of this wavefront: program order is execution
// order there, so only the compiler has to be held.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// Boundary of the R removed tetrahedra at positions Tlast .. Tlast + R - 1 of
// T (cpp:497-580): Ray et al.'s cycle walk, C(v) = next vertex of v on the
// cycle (kEmpty off it).  C must be kEmpty for every vertex of the star.
// Returns true when the 100-step cap stopped the walk (an open star);
// *first_out is the vertex that the re-triangulation starts from.
template <class TF, class CF>
__device__ __forceinline__ bool cavity_walk(TF&& T, CF&& C, uint32_t Tlast, uint32_t Rsize, uint32_t* first_out) {
    --Rsize;
    const uint32_t tlst = T(Tlast + Rsize);
    const uint32_t ta = tlst & 255u, tb = (tlst >> 8) & 255u, tc3 = (tlst >> 16) & 255u;
    C(ta) = tb;
    C(tb) = tc3;
    C(tc3) = ta;
    uint32_t cur = Tlast;
    uint32_t first = ta;
    int swap_with = (int)(Tlast + Rsize) - 1;
    uint32_t failed = 0;
    int niter = 0;
    while (Rsize && niter++ < 100) {
        const uint32_t tw = T(cur);
        const uint32_t tcv[3] = {tw & 255u, (tw >> 8) & 255u, (tw >> 16) & 255u};
        const uint32_t ty[3] = {C(tcv[0]), C(tcv[1]), C(tcv[2])};
        bool inb[3], opp[3];
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            inb[e] = ty[e] != kEmpty;
            opp[e] = ty[(e + 1) % 3] == tcv[e];
        }
        bool simple = opp[0] || opp[1] || opp[2];
#pragma unroll
        for (int e = 0; e < 3; ++e) simple &= (opp[e] || opp[(e + 1) % 3] || !inb[(e + 1) % 3]);
        if (!simple) {
            // a pass in which all fail leaves the rest of the steps to fail too
            if (++failed == Rsize) break;
            ++cur;
            continue;
        }
        failed = 0;
#pragma unroll
        for (int e = 0; e < 3; ++e)
            if (!opp[e]) C(tcv[e]) = tcv[(e + 1) % 3];
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            if (opp[e] && opp[(e + 1) % 3]) {
                if (first == tcv[(e + 1) % 3]) first = ty[(e + 1) % 3];
                C(tcv[(e + 1) % 3]) = kEmpty;
            }
        }
        T(cur) = T((uint32_t)swap_with);
        T((uint32_t)swap_with) = tw;
        --swap_with;
        --Rsize;
        cur = Tlast;
    }
    *first_out = first;
    return Rsize != 0;
}

// Minimum over the wavefront.
__device__ __forceinline__ uint32_t wave_min(uint32_t v) {
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x111, 0xf, 0xf, false));  // row_shr:1
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x112, 0xf, 0xf, false));  // row_shr:2
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x114, 0xf, 0xf, false));  // row_shr:4
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x118, 0xf, 0xf, false));  // row_shr:8
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x142, 0xa, 0xf, false));  // row_bcast:15
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x143, 0xc, 0xf, false));  // row_bcast:31
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// cavity_walk by a whole wavefront, one removed triangle per lane (R <= 64):
// every remaining triangle is tried at once, and the one at the lowest
// position joins, as the scan would find it after one failed step per position
// before.  T keeps its order (only the new tetrahedra follow).
template <class TF, class CF>
__device__ __forceinline__ bool wave_walk(TF&& T, CF&& C, uint32_t m, uint32_t R, uint32_t* first_out) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t tw = lane < R ? T(m + lane) : 0u, tl = T(m + R - 1);
    const uint32_t x = tw & 255u, y = (tw >> 8) & 255u, z = (tw >> 16) & 255u;
    const uint32_t ta = tl & 255u, tb = (tl >> 8) & 255u, tc = (tl >> 16) & 255u;
    C(ta) = tb;
    C(tb) = tc;
    C(tc) = ta;
    wave_lds_sync();
    uint32_t first = ta, left = R - 1, steps = 0;
    uint32_t pos = lane < R - 1 ? lane : ~0u;  // position behind m; ~0: in the cycle already
    while (left) {
        const uint32_t cx = C(x), cy = C(y), cz = C(z);
        const bool o0 = cy == x, o1 = cz == y, o2 = cx == z;
        const bool simple = (o0 || o1 || o2) && (o0 || o1 || cy == kEmpty) && (o1 || o2 || cz == kEmpty) &&
                            (o2 || o0 || cx == kEmpty);
        const uint32_t best = wave_min(simple ? pos : ~0u);
        steps += best + 1;
        if (best == ~0u || steps > 100) break;
        const bool mine = pos == best;
        uint32_t nf = first;  // another start when the first corner goes inside
        wave_lds_sync();
        if (mine) {
            if (!o0) C(x) = y;
            if (!o1) C(y) = z;
            if (!o2) C(z) = x;
            if (o0 && o1) {
                nf = nf == y ? cy : nf;
                C(y) = kEmpty;
            }
            if (o1 && o2) {
                nf = nf == z ? cz : nf;
                C(z) = kEmpty;
            }
            if (o2 && o0) {
                nf = nf == x ? cx : nf;
                C(x) = kEmpty;
            }
        }
        const uint64_t chg = __builtin_amdgcn_ballot_w64(nf != first);
        if (chg) first = (uint32_t)__builtin_amdgcn_readlane((int)nf, __builtin_ctzll(chg));
        --left;
        pos = mine ? ~0u : (pos == left ? best : pos);
        wave_lds_sync();
    }
    *first_out = first;
    return left != 0;
}

// The alpha filter of the tetrahedron (tid, i2, i3, i4) (cpp:590-682): kept
// when its squared circumradius is at most every corner's alpha^2; *own when
// tid is its lowest id.
template <class S>
__device__ __forceinline__ bool alpha_keep(const Sph4<S>* P, uint32_t tid, uint32_t i2, uint32_t i3, uint32_t i4,
                                           bool* own) {
    uint32_t i1 = tid, t;
    if (i1 > i3) { t = i3; i3 = i1; i1 = t; }
    if (i2 > i4) { t = i4; i4 = i2; i2 = t; }
    if (i1 > i2) { t = i2; i2 = i1; i1 = t; }
    if (i3 > i4) { t = i4; i4 = i3; i3 = t; }
    if (i2 > i3) { t = i3; i3 = i2; i2 = t; }
    const Sph4<S> qa = P[i1], qb = P[i2], qc = P[i3], qd = P[i4];
    const S tv[3] = {qa.c[0] - qd.c[0], qa.c[1] - qd.c[1], qa.c[2] - qd.c[2]};
    const S uv[3] = {qb.c[0] - qd.c[0], qb.c[1] - qd.c[1], qb.c[2] - qd.c[2]};
    const S vv[3] = {qc.c[0] - qd.c[0], qc.c[1] - qd.c[1], qc.c[2] - qd.c[2]};
    const S d2t = tv[0] * tv[0] + tv[1] * tv[1] + tv[2] * tv[2];
    const S d2u = uv[0] * uv[0] + uv[1] * uv[1] + uv[2] * uv[2];
    const S d2v = vv[0] * vv[0] + vv[1] * vv[1] + vv[2] * vv[2];
    const S vol = tv[2] * (uv[0] * vv[1] - vv[0] * uv[1]) - uv[2] * (tv[0] * vv[1] - vv[0] * tv[1]) +
                  vv[2] * (tv[0] * uv[1] - uv[0] * tv[1]);
    S w[3];
    {
        const S x0 = uv[1] * vv[2] - uv[2] * vv[1], x1 = uv[2] * vv[0] - uv[0] * vv[2],
                x2 = uv[0] * vv[1] - uv[1] * vv[0];
        w[0] = d2t * x0;
        w[1] = d2t * x1;
        w[2] = d2t * x2;
    }
    {
        const S x0 = vv[1] * tv[2] - vv[2] * tv[1], x1 = vv[2] * tv[0] - vv[0] * tv[2],
                x2 = vv[0] * tv[1] - vv[1] * tv[0];
        w[0] += d2u * x0;
        w[1] += d2u * x1;
        w[2] += d2u * x2;
    }
    {
        const S x0 = tv[1] * uv[2] - tv[2] * uv[1], x1 = tv[2] * uv[0] - tv[0] * uv[2],
                x2 = tv[0] * uv[1] - tv[1] * uv[0];
        w[0] += d2v * x0;
        w[1] += d2v * x1;
        w[2] += d2v * x2;
    }
    const S wn = w[0] * w[0] + w[1] * w[1] + w[2] * w[2];
    const S rc = wn / ((S)4 * vol * vol);
    *own = tid == i1;
    return rc <= qa.r * qa.r && rc <= qb.r * qb.r && rc <= qc.r * qc.r && rc <= qd.r * qd.r;
}

// Outputs of a node with fewer than three candidates.
template <class S> __device__ __forceinline__ void empty_star(const Ash3Args<S>& a, uint32_t tid) {
    a.node_is_bnd[tid] = 1;
    a.nelem_out[tid] = 0;
    a.nelem[tid] = 0;
    a.nfneig[tid] = 0;
}

// Local Delaunay of node tid's star + alpha filter (cpp:380-682) by one
// wavefront, what the FP64 filter leaves undecided through the exact stage
// (queue[2] counts the nodes that need it; the others are here for space).  A
// lane tests the tetrahedra at its positions (each is tested once per insertion,
// and its result depends on it and the point alone, so the order is free); lane 0
// evaluates the undecided ones, with the expansion in LDS.  Removal and
// re-triangulation run on the flags, on every lane alike.
template <class S> struct Exact3Lds {
    double ws[kExactWs3D];
    S x[kCycle3D][3];  // candidates
    uint32_t t[kTet3D];
    uint32_t c[kCycle3D];
};
template <class S> __device__ void local_delaunay3_exact(const Ash3Args<S>& a, uint32_t tid, Exact3Lds<S>& L) {
    const uint32_t n = a.n, lane = threadIdx.x & 63u;
    const Sph4<S>* P = a.P;
    const uint32_t ncand = a.nineig[tid];
    auto neig = [&](uint32_t j) -> uint32_t { return j < kNInf3D ? n + j : a.cand[slab3(tid, j - kNInf3D, kCand3D)]; };
    auto T = [&](uint32_t ti) -> uint32_t& { return L.t[ti]; };
    auto C = [&](uint32_t v) -> uint32_t& { return L.c[v]; };

    T(0) = pack_tet(0, 2, 1);
    T(1) = pack_tet(1, 2, 3);
    T(2) = pack_tet(0, 1, 3);
    T(3) = pack_tet(0, 3, 2);
    for (uint32_t j = lane; j < ncand; j += 64) load3(P, neig(j), L.x[j]);
    wave_lds_sync();
    S pa0[3];
    load3(P, tid, pa0);
    auto corner = [&](uint32_t j, S* p) {
        p[0] = L.x[j][0];
        p[1] = L.x[j][1];
        p[2] = L.x[j][2];
    };
    uint32_t Tlast = 4;
    bool over = false, needed = false;
    for (uint32_t pi = kNInf3D; pi < ncand; ++pi) {
        S pe0[3];
        corner(pi, pe0);
        uint64_t f[4] = {0, 0, 0, 0};
#pragma unroll 1
        for (uint32_t q = 0; q * 64 < Tlast; ++q) {
            const uint32_t ti = q * 64 + lane;
            S pb[3], pc[3], pd[3];
            uint32_t tl = 0;
            S det = (S)0;
            bool undecided = false;
            if (ti < Tlast) {
                tl = T(ti);
                corner(tl & 255u, pb);
                corner((tl >> 8) & 255u, pc);
                corner((tl >> 16) & 255u, pd);
                S err;
                det = -insphere_filter(pa0, pb, pc, pd, pe0, &err);
                undecided = !((det > err) || (-det > err));
                if constexpr (sizeof(S) == sizeof(float)) {
                    if (undecided) {
                        double q[5][3];
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            q[0][k] = pa0[k];
                            q[1][k] = pb[k];
                            q[2][k] = pc[k];
                            q[3][k] = pd[k];
                            q[4][k] = pe0[k];
                        }
                        double e2;
                        const double d2 = -insphere_filter(q[0], q[1], q[2], q[3], q[4], &e2);
                        undecided = !((d2 > e2) || (-d2 > e2));
                        det = d2 > 0.0 ? (S)1 : (S)-1;
                    }
                }
            }
            // one undecided lane after the other: the workspace is shared
            uint64_t u = __builtin_amdgcn_ballot_w64(undecided);
            needed |= u != 0;
            for (; u; u &= u - 1) {
                if (lane == (uint32_t)__builtin_ctzll(u)) {
                    double* ws = L.ws;
                    uint32_t i1 = tid, i2 = neig(tl & 255u), i3 = neig((tl >> 8) & 255u),
                             i4 = neig((tl >> 16) & 255u), i5 = neig(pi);
                    S qa[3] = {pa0[0], pa0[1], pa0[2]}, qe[3] = {pe0[0], pe0[1], pe0[2]};
                    S* p1 = qa;
                    S* p2 = pb;
                    S* p3 = pc;
                    S* p4 = pd;
                    S* p5 = qe;
                    bool swap = false;
                    auto cs = [&](uint32_t& x, uint32_t& y, S*& px, S*& py) {
                        if (x > y) {
                            const uint32_t t = x;
                            x = y;
                            y = t;
                            S* u = px;
                            px = py;
                            py = u;
                            swap = !swap;
                        }
                    };
                    cs(i1, i5, p1, p5);
                    cs(i2, i4, p2, p4);
                    cs(i1, i3, p1, p3);
                    cs(i3, i5, p3, p5);
                    cs(i1, i2, p1, p2);
                    cs(i3, i4, p3, p4);
                    cs(i2, i5, p2, p5);
                    cs(i2, i3, p2, p3);
                    cs(i4, i5, p4, p5);
                    det = (S)-insphere_exact(p1, p2, p3, p4, p5, ws, (int)kExactWs3D, &over);
                    int depth = 0;
                    while (det == (S)0) {
                        ++depth;
                        if (depth == 1) {
                            bool c1;
                            det = orient3d_filter(p2, p3, p4, p5, &c1);
                            if (!c1) det = (S)orient3d_exact(p2, p3, p4, p5, ws, (int)kExactWs3D, &over);
                        } else if (depth == 2) {
                            bool c2;
                            det = orient3d_filter(p1, p3, p4, p5, &c2);
                            if (!c2) det = (S)orient3d_exact(p1, p3, p4, p5, ws, (int)kExactWs3D, &over);
                            det = -det;
                        } else {
                            det = swap ? (S)1 : (S)-1;
                        }
                    }
                    if (swap) det = -det;
                }
                wave_lds_sync();
            }
            const uint64_t m = __builtin_amdgcn_ballot_w64(det > (S)0);
            f[0] = q == 0 ? m : f[0];
            f[1] = q == 1 ? m : f[1];
            f[2] = q == 2 ? m : f[2];
            f[3] = q == 3 ? m : f[3];
        }
        // the cavity: the sequential order of cpp:421-495 (a conflicting
        // tetrahedron is swapped with the last one, which is tested next at
        // the same position)
        auto flag = [&](uint32_t k) -> bool {
            const uint64_t w = k < 64 ? f[0] : (k < 128 ? f[1] : (k < 192 ? f[2] : f[3]));
            return (w >> (k & 63u)) & 1u;
        };
        // first flagged position >= k (256 when none)
        auto next_flag = [&](uint32_t k) -> uint32_t {
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                if (k < q * 64 + 64) {
                    const uint64_t m = k > q * 64 ? f[q] & (~0ull << (k - q * 64)) : f[q];
                    if (m) return q * 64 + (uint32_t)__builtin_ctzll(m);
                }
            }
            return 256u;
        };
        uint32_t Rsize = 0;
        wave_lds_sync();
        for (uint32_t ti = next_flag(0); ti < Tlast; ti = next_flag(ti)) {
            ++Rsize;
            --Tlast;
            const uint32_t tl = T(ti), te = T(Tlast);
            T(ti) = te;
            T(Tlast) = tl;
            const bool fl = flag(Tlast);
            const uint64_t bit = 1ull << (ti & 63u);
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q)
                if (ti >> 6 == q) f[q] = fl ? f[q] | bit : f[q] & ~bit;
        }
        if (Rsize) {
            for (uint32_t v = lane; v < kCycle3D; v += 64) C(v) = kEmpty;
            wave_lds_sync();
            uint32_t first;
            if (Rsize <= 64)
                wave_walk(T, C, Tlast, Rsize, &first);
            else
                cavity_walk(T, C, Tlast, Rsize, &first);
            uint32_t c = first;
            int guard = 0;
            bool bad = false;
            do {
                bad = c >= kCycle3D || ++guard > 255 || Tlast >= kTet3D;
                if (bad) break;
                const uint32_t nx = C(c);
                T(Tlast++) = pack_tet(pi, c, nx);
                c = nx;
            } while (c != first);
            if (bad) {
                raise_flag(a.flags, kErrCapacity);
                Tlast = 0;
                break;
            }
        }
        wave_lds_sync();
    }
    if (over) raise_flag(a.flags, kErrCapacity);
    if (needed && lane == 0) atomicAdd(&a.queue[2], 1u);
    // alpha filter (cpp:590-682): kept tetrahedra count at their corners; this
    // node's own ones come first, a dropped or foreign one giving its position
    // to the last one that is left
    for (uint32_t v = lane; v < ncand; v += 64) C(v) = 0;
    wave_lds_sync();
    uint32_t nloc = 0;
#pragma unroll 1
    for (uint32_t q = 0; q * 64 < Tlast; ++q) {
        const uint32_t ti = q * 64 + lane;
        bool keep = false, own = false;
        if (ti < Tlast) {
            const uint32_t tl = T(ti);
            const uint32_t la = tl & 255u, lb = (tl >> 8) & 255u, lc = (tl >> 16) & 255u;
            if (la >= kNInf3D && lb >= kNInf3D && lc >= kNInf3D)
                keep = alpha_keep(P, tid, neig(la), neig(lb), neig(lc), &own);
            if (keep) {
                atomicAdd(&C(la), 1u);
                atomicAdd(&C(lb), 1u);
                atomicAdd(&C(lc), 1u);
            }
            T(ti) = tl | (keep && own ? 1u << 24 : 0u);
        }
        nloc += __popcll(__builtin_amdgcn_ballot_w64(keep));
    }
    wave_lds_sync();
    // per candidate, the number of kept tetrahedra using it (the infinity
    // nodes are in no kept tetrahedron)
    uint32_t nf = 0;
    for (uint32_t v0 = kNInf3D; v0 < ncand; v0 += 64) {
        const uint32_t v = v0 + lane, c = v < ncand ? C(v) : 0u;
        if (v < ncand) a.active[slab3(tid, v - kNInf3D, kCand3D)] = (uint8_t)c;
        nf += __popcll(__builtin_amdgcn_ballot_w64(c != 0));
    }
    if (lane != 0) return;
    uint32_t nout = 0, left = Tlast;
    for (uint32_t ti = 0; ti < left;) {
        const uint32_t tl = T(ti);
        if (tl >> 24) {
            a.tet[slab3(tid, nout++, kTet3D)] = tl & 0xffffffu;
            ++ti;
        } else {
            T(ti) = T(--left);
        }
    }
    a.node_is_bnd[tid] = nloc != Tlast;
    a.nelem_out[tid] = (uint8_t)nout;
    a.nelem[tid] = (uint8_t)nloc;
    a.nfneig[tid] = nf;
}

// Local Delaunay + alpha filter of every node, 16 lanes per node.
//
// A star holds about 23 tetrahedra while 34 to 80 candidates go in, two of
// three of which open a cavity of about 5.  One lane per node spent its time
// gathering three corners for each of the ~1,500 insphere tests of a node (a
// cache line per lane and load).  Here 16 lanes hold the star: lane l the
// tetrahedra at positions l, l + 16, ... in registers, the ids also in LDS.
//
//   test    The sphere test of predicates.hpp: 7 FP32 operations on one LDS
//           read and what is kept per tetrahedron, in both node types.  What
//           it cannot certify goes to the FP64 filter on the node's own
//           coordinates, and a node where that fails too to the exact kernel.
//           A certified sign is the exact sign, so all three give the same
//           decisions.
//   remove  The sequential swap with the last (cpp:421-495) fills the flagged
//           positions below m (the number kept), in order, with the kept ones
//           from the end backwards.  With j flagged positions below p, a
//           flagged p takes the j-th of these, and a kept p >= m is the
//           (m - 1 - p + j)-th.  The removed ones end up from m on: the
//           flagged one at q > m at q - 1, the j-th other one right below
//           where the (j-1)-th moved one came from.
//   cycle   One removed triangle per lane, a set of lanes per corner: the
//           lanes that hold both ends of an edge are its two triangles, so an
//           edge whose other triangle stays is on the boundary cycle.  The
//           reference's walk ends on the same cycle, and starts there from the
//           first removed triangle's first corner, unless that corner ends
//           inside: then the start is, as often as needed, the corner before
//           it in the triangle that closes the fan around it.  Which one that
//           is depends on the order of the walk, so the walk runs, on sets of
//           lanes: a triangle can join the disc when it shares two edges with
//           it, or one and the third corner is not in it yet, and the scan
//           takes the one at the lowest position, after one failed step per
//           position before.  A cavity of 14 or fewer is done in at most 91
//           steps (at most one fails per remaining triangle), so the cap of
//           100 plays no part.  One of up to 32 has two triangles per lane;
//           where its walk meets the cap, in larger ones and in stars that the
//           cap left open, the reference's own walk runs.
//   new     One lane per new tetrahedron computes its W, V and bounds; the
//           lane that holds the position picks them up through LDS.
//
// A star that outgrows 64 positions goes to the exact kernel.
//
// Bound: instruction issue (364 vector and 264 scalar instructions per
// insertion of a wavefront's four nodes, three quarters of the vector issue
// slots at 4 wavefronts per SIMD).  5 wavefronts (96 registers) spill and are
// a third slower.  From one lane per node to this: 1,996,920 FP64 nodes 68.7 ->
// 24.6 ms, 100,000 FP32 ones 2.50 -> 0.68 ms, 20,102 FP32 ones (79 blocks of
// one lane per node left most of the chip idle) 3.96 -> 0.43 ms.
constexpr int kStarLanes = 16;
constexpr uint32_t kStarTets = 64;
constexpr int kStarSlots = (int)kStarTets / kStarLanes;
constexpr uint32_t kWalkFree = 14;  // R (R - 1) / 2 <= 100, and R + 2 new ones on 16 lanes

// Candidates of the four nodes of a wavefront together (LDS); a node that does
// not fit beside the others waits for a second pass.  34 to 85 candidates per
// node are usual; 448 bring a wavefront's LDS to 10 KB, four per SIMD.
constexpr uint32_t kStarPool = 448;

// Consecutive nodes share candidates and slab lines, so an XCD (the blocks go to
// the 8 in turn) takes runs of this many blocks, 256 nodes.  One contiguous eighth
// of the nodes each left the XCDs unequal loads: 20,000 nodes of 124 candidates in
// a dense cluster beside 20,000 ordinary ones 7.8 ms (4.9 now), a tank of 299,000
// 4.05 (3.72), the 2M one 26.6 (24.6).  Shorter runs share less (100,000 uniform
// nodes 0.68 ms, as before; 0.69 with 16 blocks).
constexpr uint32_t kStarRun = 64;

struct alignas(16) SphRec {
    SphReg r;
    uint32_t pos;  // where it comes from
};
struct Star3Lds {
    union {
        uint32_t c[kCycle3D];    // per local id: set of lanes, next on the cycle, count
        SphRec rec[kStarLanes];  // tetrahedra on their way to another lane
    };
    uint32_t t[kStarTets];  // ids: removed ones; the whole star for a large cavity
};

__device__ __forceinline__ uint64_t ballot(bool b) { return __builtin_amdgcn_ballot_w64(b); }
// Bits of this lane's group of 16 in a wavefront ballot.
__device__ __forceinline__ uint32_t group_bits(uint64_t m, uint32_t grp) {
    const uint32_t h = grp >= 2 ? (uint32_t)(m >> 32) : (uint32_t)m;
    return (h >> ((grp & 1u) * 16u)) & 0xffffu;
}
// Two ballots' bits of this lane's group, the second one's in the upper half.
__device__ __forceinline__ uint32_t group_bits2(uint64_t m0, uint64_t m1, uint32_t grp) {
    const uint32_t h0 = grp >= 2 ? (uint32_t)(m0 >> 32) : (uint32_t)m0;
    const uint32_t h1 = grp >= 2 ? (uint32_t)(m1 >> 32) : (uint32_t)m1;
    return __builtin_amdgcn_perm(h1, h0, (grp & 1u) ? 0x07060302u : 0x05040100u);
}
// Minimum over the 16 lanes of the group (a DPP row).
__device__ __forceinline__ uint32_t group_min(uint32_t v) {
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x128, 0xf, 0xf, false));  // row_ror:8
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x124, 0xf, 0xf, false));  // row_ror:4
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x122, 0xf, 0xf, false));  // row_ror:2
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x121, 0xf, 0xf, false));  // row_ror:1
    return v;
}
// A set of up to 64 positions.
struct PosSet {
    uint32_t lo, hi;
};

// The FP64 filter's sign of the insphere test of e against the tetrahedron
// (a, b, c, d): 1 inside, -1 outside, 0 undecided.
template <class S>
__device__ __forceinline__ int insphere_side_f64(const Sph4<S>* P, uint32_t ia, uint32_t ib, uint32_t ic, uint32_t id,
                                              uint32_t ie) {
    const Sph4<S> q[5] = {P[ia], P[ib], P[ic], P[id], P[ie]};
    double x[5][3];
#pragma unroll
    for (int v = 0; v < 5; ++v)
#pragma unroll
        for (int k = 0; k < 3; ++k) x[v][k] = q[v].c[k];
    double err;
    const double det = -insphere_filter(x[0], x[1], x[2], x[3], x[4], &err);
    return det > err ? 1 : (-det > err ? -1 : 0);
}

template <class S>
__device__ __forceinline__ void star3_node(const Ash3Args<S>& a, uint32_t tid, uint32_t ncand, uint32_t sub,
                                           uint32_t grp, float4* E, Star3Lds& L) {
    constexpr int G = kStarLanes, NS = kStarSlots;
    const uint32_t n = a.n;
    const Sph4<S>* P = a.P;
    auto neig = [&](uint32_t j) -> uint32_t { return j < kNInf3D ? n + j : a.cand[slab3(tid, j - kNInf3D, kCand3D)]; };
    const Sph4<S> self = P[tid];
    {
        const double scale = sph_scale((double)self.r);
        for (uint32_t j = sub; j < ncand; j += G) {
            const Sph4<S> q = P[neig(j)];
            E[j] = sph_point(((double)q.c[0] - (double)self.c[0]) * scale, ((double)q.c[1] - (double)self.c[1]) * scale,
                             ((double)q.c[2] - (double)self.c[2]) * scale);
        }
    }
    wave_lds_sync();
    uint32_t Tl = 4;
    SphReg rec[NS];
    auto load_rec = [&](uint32_t w) { return sph_rec(w, E[w & 255u], E[(w >> 8) & 255u], E[(w >> 16) & 255u]); };
    if (sub < 4) {
        const uint32_t w = sub == 0   ? pack_tet(0, 2, 1)
                           : sub == 1 ? pack_tet(1, 2, 3)
                           : sub == 2 ? pack_tet(0, 1, 3)
                                      : pack_tet(0, 3, 2);
        rec[0] = load_rec(w);
    }
    const uint32_t below[2] = {(1u << sub) - 1u, (1u << (sub + 16)) - 1u};
    auto has = [&](const PosSet& F, int s) -> bool { return ((s < 2 ? F.lo : F.hi) >> ((s & 1) * 16 + sub)) & 1u; };
    auto rank = [&](const PosSet& F, int s) -> uint32_t {  // members of F below this lane's position in slot s
        return s < 2 ? __popc(F.lo & below[s & 1]) : __popc(F.hi & below[s & 1]) + __popc(F.lo);
    };
    auto members = [](const PosSet& F) -> uint32_t { return __popc(F.lo) + __popc(F.hi); };
    auto word = [&](uint32_t s) -> uint32_t {
        return s == 0 ? rec[0].w : (s == 1 ? rec[1].w : (s == 2 ? rec[2].w : rec[3].w));
    };
    bool open_star = false;
    uint32_t redo = 0;  // 1: undecided sign, 2: too many tetrahedra or a broken cycle
    for (uint32_t pi = kNInf3D; pi < ncand; ++pi) {
        const float4 e = E[pi];
        const float ee = e.w * e.w;
        // lane constants are cheaper to form again than to hold
        asm volatile("" : "+v"(sub));
        const bool wide = ballot(Tl > 32) != 0;  // some node of the wavefront uses slots 2 and 3
        uint64_t in_m[NS];
        bool un[NS];
        auto test = [&](int s) {
            float err;
            const float det = sph_test(rec[s], e, ee, &err);
            const bool in = (uint32_t)(s * G) + sub < Tl;
            in_m[s] = ballot(in && det > err);
            un[s] = in && !(fabsf(det) > err);
        };
        test(0);
        test(1);
        PosSet F;
        F.lo = group_bits2(in_m[0], in_m[1], grp);
        F.hi = 0;
        uint64_t un_m = ballot(un[0] || un[1]);
        un[2] = un[3] = false;
        if (wide) {
            test(2);
            test(3);
            F.hi = group_bits2(in_m[2], in_m[3], grp);
            un_m |= ballot(un[2] || un[3]);
        }
        if (__builtin_expect(un_m != 0, 0)) {
            const uint32_t unsure = un[0] | (un[1] << 1) | (un[2] << 2) | (un[3] << 3);
            bool undecided = false;
            // the FP64 test needs the records' registers
            volatile SphReg save[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                save[s].wx = rec[s].wx;
                save[s].wy = rec[s].wy;
                save[s].wz = rec[s].wz;
                save[s].v = rec[s].v;
                save[s].wp = rec[s].wp;
                save[s].vp = rec[s].vp;
                save[s].w = rec[s].w;
            }
#pragma unroll 1
            for (uint32_t k = 0; k < (uint32_t)NS; ++k) {
                bool pos = false;
                if ((unsure >> k) & 1u) {
                    const uint32_t tw = save[k].w;
                    const int side = insphere_side_f64(P, tid, neig(tw & 255u), neig((tw >> 8) & 255u),
                                                       neig((tw >> 16) & 255u), neig(pi));
                    pos = side > 0;
                    undecided |= side == 0;
                }
                const uint32_t bits = group_bits(ballot(pos), grp) << ((k & 1u) * 16u);
                F.lo |= k < 2 ? bits : 0u;
                F.hi |= k < 2 ? 0u : bits;
            }
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                rec[s].wx = save[s].wx;
                rec[s].wy = save[s].wy;
                rec[s].wz = save[s].wz;
                rec[s].v = save[s].v;
                rec[s].wp = save[s].wp;
                rec[s].vp = save[s].vp;
                rec[s].w = save[s].w;
            }
            if (group_bits(ballot(undecided), grp)) {
                redo = 1;
                break;
            }
        }
        const uint32_t R = members(F);
        if (R == 0) continue;
        const uint32_t m = Tl - R;
        uint32_t end = m;
        if (__builtin_expect(R <= kWalkFree && !open_star, 1)) {
            // moved and removed tetrahedra
            auto move_out = [&](int s) {
                const uint32_t p = (uint32_t)(s * G) + sub;
                if (p >= m && p < Tl && !has(F, s)) L.rec[m - 1 - p + rank(F, s)] = SphRec{rec[s], p};
            };
            auto move_in = [&](int s) {
                const uint32_t p = (uint32_t)(s * G) + sub;
                if (has(F, s)) {
                    const uint32_t j = rank(F, s), w = rec[s].w;
                    const uint32_t at = p > m ? p : (j ? L.rec[j - 1].pos : Tl);
                    L.t[at - 1 - m] = w;
                    if (p < m) rec[s] = L.rec[j].r;
                }
            };
            move_out(0);
            move_out(1);
            if (wide) {
                move_out(2);
                move_out(3);
            }
            wave_lds_sync();
            move_in(0);
            move_in(1);
            if (wide) {
                move_in(2);
                move_in(3);
            }
            wave_lds_sync();
            const uint32_t tw = L.t[sub], ta = L.t[R - 1] & 255u;  // (lanes from R on: any valid or stale ids)
            const uint32_t x = tw & 127u, y = (tw >> 8) & 127u, z = (tw >> 16) & 127u;
            if (sub < R) {
                L.c[x] = 0;
                L.c[y] = 0;
                L.c[z] = 0;
            }
            wave_lds_sync();
            if (sub < R) {
                atomicOr(&L.c[x], 1u << sub);
                atomicOr(&L.c[y], 1u << sub);
                atomicOr(&L.c[z], 1u << sub);
            }
            wave_lds_sync();
            uint32_t first = ta;
            const uint32_t mx = L.c[x], my = L.c[y], mz = L.c[z], others = ~(1u << sub);
            const uint32_t n0 = mx & my & others, n1 = my & mz & others, n2 = mz & mx & others;
            const bool b0 = sub < R && n0 == 0, b1 = sub < R && n1 == 0, b2 = sub < R && n2 == 0;
            auto on_cycle = [&](uint32_t v) -> bool {
                return group_bits(ballot((b0 && x == v) || (b1 && y == v) || (b2 && z == v)), grp) != 0;
            };
            if (!on_cycle(first)) {
                uint32_t disc = 1u << (R - 1), fan = L.c[first], left = R - 1;
                uint32_t key = sub < R - 1 ? sub << 4 | sub : ~0u;  // position and lane; ~0: in the disc
                while (left) {
                    const bool o0 = n0 & disc, o1 = n1 & disc, o2 = n2 & disc;
                    const bool joins = (o0 && (o1 || o2 || !(mz & disc))) || (o1 && (o2 || !(mx & disc))) ||
                                       (o2 && !(my & disc));
                    const uint32_t best = group_min(joins ? key : ~0u);
                    if (best == ~0u) {
                        first = kEmpty;  // no disc: refused below
                        break;
                    }
                    const uint32_t win = best & 15u;
                    disc |= 1u << win;
                    --left;
                    // the last position's triangle takes the winner's
                    key = key >> 4 == left ? (best & ~15u) | sub : key;
                    key = sub == win ? ~0u : key;
                    if ((fan & ~disc) == 0) {
                        const uint32_t before = x == first ? z : (y == first ? x : y);
                        first = (uint32_t)__shfl((int)before, (int)(grp * G + win), 64);
                        if (on_cycle(first)) break;
                        fan = L.c[first];
                    }
                }
            }
            wave_lds_sync();
            if (b0) L.c[x] = y;
            if (b1) L.c[y] = z;
            if (b2) L.c[z] = x;
            wave_lds_sync();
            // around the cycle (and on, until the wavefront's longest one is
            // closed); lane b keeps the start of the b-th edge
            uint32_t c = first, mc = first;
            uint64_t open_m = ballot(true);
            for (uint32_t k = 1; k < (uint32_t)G && open_m; ++k) {
                c = L.c[c & (kCycle3D - 1)];
                mc = sub == k ? c : mc;
                open_m &= ballot(c != first);
            }
            const uint32_t mn = L.c[mc & (kCycle3D - 1)];
            const uint32_t again = group_bits(ballot(sub != 0 && mc == first), grp) & ~1u;
            const uint32_t nb = again ? (uint32_t)__builtin_ctz(again) : (uint32_t)G;
            end = m + nb;
            // (a proper boundary has R + 2 edges, less two per corner inside, and
            // its corners went in before pi: what a broken one reads is no id)
            if (group_bits(ballot(sub < nb && (mc >= pi || (sub + 1 == nb && mn != first))), grp) || nb > R + 2 ||
                ((nb ^ R) & 1u) || end > kStarTets) {
                redo = 2;
                break;
            }
            wave_lds_sync();
            if (sub < nb) L.rec[sub] = SphRec{sph_rec(pack_tet(pi, mc, mn), e, E[mc], E[mn]), 0};
            wave_lds_sync();
            auto take = [&](int s) {
                const uint32_t p = (uint32_t)(s * G) + sub;
                if (p >= m && p < end) rec[s] = L.rec[p - m].r;
            };
            take(0);
            take(1);
            if (ballot(end > 32)) {
                take(2);
                take(3);
            }
            wave_lds_sync();
        } else {
            auto T = [&](uint32_t k) -> uint32_t& { return L.t[k]; };
            auto C = [&](uint32_t k) -> uint32_t& { return L.c[k]; };
            // as above for the ids alone; L.t becomes the whole star, the
            // removed ones from m on
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const uint32_t p = (uint32_t)(s * G) + sub;
                if (p >= m && p < Tl && !has(F, s)) L.c[m - 1 - p + rank(F, s)] = rec[s].w | p << 24;
            }
            wave_lds_sync();
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const uint32_t p = (uint32_t)(s * G) + sub;
                if (has(F, s)) {
                    const uint32_t j = rank(F, s);
                    const uint32_t at = p > m ? p : (j ? L.c[j - 1] >> 24 : Tl);
                    T(at - 1) = rec[s].w;
                    if (p < m) T(p) = L.c[j] & 0xffffffu;
                } else if (p < m) {
                    T(p) = rec[s].w;
                }
            }
            wave_lds_sync();
            // every lane of the group runs what follows on the same words
            uint32_t first = T(Tl - 1) & 255u;
            bool walk = open_star || R > 2 * (uint32_t)G;
            if (!walk) {
                // as above with two triangles per lane, at sub and sub + 16
                uint32_t x[2], y[2], z[2], n0[2], n1[2], n2[2], mx[2], my[2], mz[2], key[2];
                bool b0[2], b1[2], b2[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t i = sub + h * G, tw = i < R ? T(m + i) : 0u;
                    x[h] = tw & 255u;
                    y[h] = (tw >> 8) & 255u;
                    z[h] = (tw >> 16) & 255u;
                    if (i < R) {
                        C(x[h]) = 0;
                        C(y[h]) = 0;
                        C(z[h]) = 0;
                    }
                }
                wave_lds_sync();
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t i = sub + h * G;
                    if (i < R) {
                        atomicOr(&C(x[h]), 1u << i);
                        atomicOr(&C(y[h]), 1u << i);
                        atomicOr(&C(z[h]), 1u << i);
                    }
                }
                wave_lds_sync();
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t i = sub + h * G, others = ~(1u << i);
                    mx[h] = C(x[h]);
                    my[h] = C(y[h]);
                    mz[h] = C(z[h]);
                    n0[h] = mx[h] & my[h] & others;
                    n1[h] = my[h] & mz[h] & others;
                    n2[h] = mz[h] & mx[h] & others;
                    b0[h] = i < R && n0[h] == 0;
                    b1[h] = i < R && n1[h] == 0;
                    b2[h] = i < R && n2[h] == 0;
                    key[h] = i < R - 1 ? i << 5 | i : ~0u;
                }
                auto on_cycle = [&](uint32_t v) -> bool {
                    bool on = false;
#pragma unroll
                    for (int h = 0; h < 2; ++h) on |= (b0[h] && x[h] == v) || (b1[h] && y[h] == v) || (b2[h] && z[h] == v);
                    return group_bits(ballot(on), grp) != 0;
                };
                uint32_t disc = 1u << (R - 1), left = R - 1, steps = 0;
                while (left) {
                    uint32_t k = ~0u;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const bool o0 = n0[h] & disc, o1 = n1[h] & disc, o2 = n2[h] & disc;
                        const bool joins = (o0 && (o1 || o2 || !(mz[h] & disc))) || (o1 && (o2 || !(mx[h] & disc))) ||
                                           (o2 && !(my[h] & disc));
                        k = joins ? min(k, key[h]) : k;
                    }
                    const uint32_t best = group_min(k);
                    steps += (best >> 5) + 1;
                    if (best == ~0u || steps > 100) break;
                    const uint32_t win = best & 31u;
                    disc |= 1u << win;
                    --left;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        key[h] = key[h] >> 5 == left ? (best & ~31u) | (sub + h * G) : key[h];
                        key[h] = sub + h * G == win ? ~0u : key[h];
                    }
                    if (!on_cycle(first) && (C(first) & ~disc) == 0) {
                        const bool up = win >= (uint32_t)G;
                        const uint32_t vx = up ? x[1] : x[0], vy = up ? y[1] : y[0], vz = up ? z[1] : z[0];
                        const uint32_t before = vx == first ? vz : (vy == first ? vx : vy);
                        first = (uint32_t)__shfl((int)before, (int)(grp * G + (win & 15u)), 64);
                    }
                }
                walk = left != 0;
                wave_lds_sync();
                if (!walk) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        if (b0[h]) C(x[h]) = y[h];
                        if (b1[h]) C(y[h]) = z[h];
                        if (b2[h]) C(z[h]) = x[h];
                    }
                }
            }
            if (walk) {
                for (uint32_t v = sub; v < kCycle3D; v += G) C(v) = kEmpty;
                wave_lds_sync();
                open_star |= cavity_walk(T, C, m, R, &first);
            }
            wave_lds_sync();
            uint32_t c = first;
            do {
                if (c >= pi || end >= kStarTets) {
                    redo = 2;
                    break;
                }
                const uint32_t nx = C(c);
                T(end++) = pack_tet(pi, c, nx);
                c = nx;
            } while (c != first);
            if (redo) break;
            wave_lds_sync();
#pragma unroll 1
            for (uint32_t k = 0; k * G < end; ++k) {
                const uint32_t p = k * G + sub;
                if (p < end) {
                    const SphReg r = load_rec(T(p));
                    if (k == 0) rec[0] = r;
                    if (k == 1) rec[1] = r;
                    if (k == 2) rec[2] = r;
                    if (k == 3) rec[3] = r;
                }
            }
            wave_lds_sync();
        }
        Tl = end;
    }
    if (redo) {
        if (sub == 0) a.queue[kQueueIds + atomicAdd(&a.queue[0], 1u)] = tid;
        return;
    }
    // alpha filter: kept tetrahedra count at their corners; this node's own
    // ones come first, in the order the sequential filter leaves them in
    for (uint32_t v = sub; v < ncand; v += G) L.c[v] = 0;
    wave_lds_sync();
    uint64_t own_m = 0;
    uint32_t nloc = 0;
#pragma unroll 1
    for (uint32_t p0 = 0; p0 < Tl; p0 += G) {
        const uint32_t p = p0 + sub;
        bool keep = false, own = false;
        if (p < Tl) {
            const uint32_t tw = word(p0 / G);
            const uint32_t la = tw & 255u, lb = (tw >> 8) & 255u, lc = (tw >> 16) & 255u;
            if (la >= kNInf3D && lb >= kNInf3D && lc >= kNInf3D)
                keep = alpha_keep(P, tid, neig(la), neig(lb), neig(lc), &own);
            if (keep) {
                atomicAdd(&L.c[la], 1u);
                atomicAdd(&L.c[lb], 1u);
                atomicAdd(&L.c[lc], 1u);
            }
        }
        nloc += __popc(group_bits(ballot(keep), grp));
        own_m |= (uint64_t)group_bits(ballot(keep && own), grp) << p0;
    }
    const uint32_t nout = __popcll(own_m);
#pragma unroll 1
    for (uint32_t p0 = 0; p0 < Tl; p0 += G) {
        const uint32_t p = p0 + sub;
        if (!((own_m >> p) & 1u)) continue;
        // below nout they stay; the others fill the gaps from the end
        uint32_t q = p;
        if (p >= nout) {
            uint32_t k = __popcll(own_m >> p) - 1;
            uint64_t gaps = ~own_m;
            while (k--) gaps &= gaps - 1;
            q = __builtin_ctzll(gaps);
        }
        a.tet[slab3(tid, q, kTet3D)] = word(p0 / G);
    }
    uint32_t nf = 0;
    for (uint32_t v0 = kNInf3D; v0 < ncand; v0 += G) {
        const uint32_t v = v0 + sub;
        const uint32_t c = v < ncand ? L.c[v] : 0u;
        if (v < ncand) a.active[slab3(tid, v - kNInf3D, kCand3D)] = (uint8_t)c;
        nf += __popc(group_bits(ballot(c != 0), grp));
    }
    if (sub == 0) {
        a.node_is_bnd[tid] = nloc != Tl;
        a.nelem_out[tid] = (uint8_t)nout;
        a.nelem[tid] = (uint8_t)nloc;
        a.nfneig[tid] = nf;
    }
}


template <class S>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 4))) void star3_kernel(Ash3Args<S> a) {
    constexpr uint32_t G = kStarLanes;
    constexpr uint32_t NPW = 64 / G;
    __shared__ float4 pool[kStarPool];
    __shared__ Star3Lds lds[NPW];
    const uint32_t sub = threadIdx.x % G, grp = threadIdx.x / G;
    const uint32_t q = blockIdx.x >> 3;  // of this XCD's blocks
    const uint32_t blk = (q / kStarRun * 8 + (blockIdx.x & 7u)) * kStarRun + q % kStarRun;
    const uint32_t tid = blk * NPW + grp;
    const uint32_t n = a.n;
    const uint32_t ncand = tid < n ? a.nineig[tid] : 0u;
    if (tid < n && ncand - kNInf3D < 3) {
        if (sub < ncand - kNInf3D) a.active[slab3(tid, sub, kCand3D)] = 0;
        if (sub == 0) empty_star(a, tid);
    }
    // share of the pool: the nodes that fit, in order; the first one always does
    uint32_t want = tid < n && ncand - kNInf3D >= 3 ? ncand : 0u;
    while (ballot(want != 0)) {
        uint32_t off = 0, mine = ~0u;
#pragma unroll
        for (uint32_t g = 0; g < NPW; ++g) {
            const uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)want, (int)(g * G));
            if (k && off + k <= kStarPool) {
                if (grp == g) mine = off;
                off += k;
            }
        }
        if (mine != ~0u) {
            star3_node<S>(a, tid, ncand, sub, grp, pool + mine, lds[grp]);
            want = 0;
        }
        wave_lds_sync();
    }
}

template <class S> void launch_star3(const Ash3Args<S>& a, hipStream_t s) {
    constexpr uint32_t round = 8 * kStarRun;
    const uint32_t blocks = (a.n + 64 / kStarLanes - 1) / (64 / kStarLanes);
    hipLaunchKernelGGL((star3_kernel<S>), dim3((blocks + round - 1) / round * round), dim3(64), 0, s, a);
}

// One queued node per wavefront (the block is one wavefront): the exact
// evaluations of different nodes happen at different points of their
// insertions, so nodes sharing a wavefront would run their exact stages one
// after another.  Bound: the latency of one node's chain.  A single open star
// that outgrew 64 tetrahedra (tank, 299,000 nodes): 1.94 ms by one lane, star
// and coordinates in global memory; 0.23 ms by the wavefront, both in LDS.
template <class S> __global__ __launch_bounds__(64) void delaunay3_exact_kernel(Ash3Args<S> a) {
    __shared__ Exact3Lds<S> lds;
    const uint32_t cnt = a.queue[0];
    for (uint32_t k = blockIdx.x; k < cnt; k += gridDim.x) {
        local_delaunay3_exact<S>(a, a.queue[kQueueIds + k], lds);
        wave_lds_sync();
    }
}

// Slab -> CSR (cpp:692-735): edges with count <= 3 are boundary edges; the
// first nelem_out local tetrahedra are the ones this node owns.
template <class S>
__global__ __launch_bounds__(256) void compress3_kernel(Ash3Args<S> a, const uint32_t* __restrict__ row,
                                                        const uint32_t* __restrict__ elemrow,
                                                        uint32_t* __restrict__ neig, uint8_t* __restrict__ edge_is_bnd,
                                                        uint32_t* __restrict__ elem) {
    const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= a.n) return;
    const uint32_t n = a.n;
    auto gneig = [&](uint32_t j) -> uint32_t { return j < kNInf3D ? n + j : a.cand[slab3(tid, j - kNInf3D, kCand3D)]; };
    uint32_t put = row[tid];
    const uint32_t nn = a.nineig[tid];
    for (uint32_t i = kNInf3D; i < nn; ++i) {
        const uint8_t ec = a.active[slab3(tid, i - kNInf3D, kCand3D)];
        if (ec) {
            edge_is_bnd[put] = (ec <= 3);
            neig[put] = gneig(i);
            ++put;
        }
    }
    uint32_t t = 0;
    for (uint32_t k = elemrow[tid]; k < elemrow[tid + 1]; ++k, ++t) {
        const uint32_t tl = a.tet[slab3(tid, t, kTet3D)];
        elem[4ull * k] = tid;
        elem[4ull * k + 1] = gneig(tl & 255u);
        elem[4ull * k + 2] = gneig((tl >> 8) & 255u);
        elem[4ull * k + 3] = gneig((tl >> 16) & 255u);
    }
}

template <class S> Ash3Args<S> make_args3(Ash3D<S>& A) {
    Ash3Args<S> a;
    a.n = A.n;
    a.P = A.lbvh.obj_m.p;
    a.node = A.lbvh.node.p;
    a.ibox = A.lbvh.ibox.p;
    a.cand = A.cand.p;
    a.tet = A.tet.p;
    a.active = A.active.p;
    a.nineig = A.nineig.p;
    a.nfneig = A.nfneig.p;
    a.node_is_bnd = A.node_is_bnd.p;
    a.nelem = A.nelem.p;
    a.nelem_out = A.nelem_out.p;
    a.queue = A.queue.p;
    a.flags = ctx().d_flags;
    return a;
}

}  // namespace

template <class S> void Ash3D<S>::set_nodes_host(uint32_t n_, const S* xyz, const S* alpha) {
    std::vector<Sph4<S>> h(n_);
    for (uint32_t i = 0; i < n_; ++i) {
        h[i].c[0] = xyz[3ull * i];
        h[i].c[1] = xyz[3ull * i + 1];
        h[i].c[2] = xyz[3ull * i + 2];
        h[i].r = alpha[i];
    }
    n = n_;
    coords.resize(n ? n : 1);
    h2d(coords.p, h.data(), n);
    inited = computed = false;
}

template <class S> void Ash3D<S>::set_nodes_device(uint32_t n_, const Sph4<S>* d) {
    n = n_;
    coords.resize(n ? n : 1);
    d2d(coords.p, d, n);
    inited = computed = false;
}

template <class S> void Ash3D<S>::init(hipStream_t s) {
    if (n < 4) throw std::invalid_argument("AlphaShape3D needs at least 4 nodes");
    lbvh.build(coords.p, n, bits, kLeafCentre, kNInf3D, s);
    hipLaunchKernelGGL((infinity3_kernel<S>), dim3(1), dim3(64), 0, s, lbvh.gbox.p, lbvh.obj_m.p, n);
    cand.resize(slab3_words(n, kCand3D));
    tet.resize(slab3_words(n, kTet3D));
    active.resize(slab3_words(n, kCand3D));
    nineig.resize(n);
    nfneig.resize(n);
    node_is_bnd.resize(n);
    nelem.resize(n);
    nelem_out.resize(n);
    row.resize(n + 1);
    elemrow.resize(n + 1);
    queue.resize((size_t)n + kQueueIds);
    scan_ws.resize(scan_workspace_words(n));
    inited = true;
    computed = false;
}

template <class S> void Ash3D<S>::compute(hipStream_t s) {
    if (!inited) throw std::invalid_argument("AlphaShape3D_compute called before init");
    Ash3Args<S> a = make_args3(*this);
    section_mark(s, kMarkCompute0);
    fill<uint32_t>(queue.p, kQueueIds, 0u, s);
    constexpr uint32_t fill_nodes = kFillBlock / kFillLanes3D;
    const uint32_t fill_xcd = ((n + fill_nodes - 1) / fill_nodes + 7) / 8;
    hipLaunchKernelGGL((fill3_kernel<S>), dim3(8 * fill_xcd), dim3(kFillBlock), 0, s, a, fill_xcd);
    section_mark(s, kMarkFill);
    launch_star3(a, s);
    section_mark(s, kMarkDelaunayMain);
    hipLaunchKernelGGL((delaunay3_exact_kernel<S>), dim3(kExactWaves3D), dim3(64), 0, s, a);
    section_mark(s, kMarkDelaunay);
    exclusive_scan_u8(nelem_out.p, elemrow.p, n, scan_ws.p, s);
    exclusive_scan_u32(nfneig.p, row.p, n, scan_ws.p, s);
    section_mark(s, kMarkScans);
    n_elems_ = read_scalar(elemrow.p + n);
    n_edges_ = read_scalar(row.p + n);
    neig.resize(n_edges_ ? n_edges_ : 1);
    edge_is_bnd.resize(n_edges_ ? n_edges_ : 1);
    elemglob.resize(4ull * (n_elems_ ? n_elems_ : 1));
    a = make_args3(*this);
    section_mark(s, kMarkCompress0);
    hipLaunchKernelGGL((compress3_kernel<S>), dim3(grid_for(n, 256)), dim3(256), 0, s, a, row.p, elemrow.p, neig.p,
                       edge_is_bnd.p, elemglob.p);
    section_mark(s, kMarkCompress);
    computed = true;
}

template <class S> uint32_t Ash3D<S>::n_exact_nodes() {
    return computed ? read_scalar(queue.p + 2) : 0u;
}
template <class S> uint32_t Ash3D<S>::n_over_cap() { return computed ? read_scalar(queue.p + 1) : 0u; }

template struct Ash3D<float>;
template struct Ash3D<double>;

}  // namespace stream_amd

// ---------------------------------------------------------------------------
// C-ABI: the reference's AlphaShape3D_* surface (DirectAlphaShape3D.cpp:
// 743-814) plus FP64 and query extensions, as for AlphaShape2D.
// ---------------------------------------------------------------------------
using namespace stream_amd;

struct AlphaShape3D {
    int bits = 21;
    bool f64 = false;
    Ash3D<float> a32;
    Ash3D<double> a64;
    int32_t status = 0;
};

namespace {
template <class F> void run_void3(AlphaShape3D* h, F&& f) {
    if (!h) {
        set_last_error("null AlphaShape3D handle");
        return;
    }
    h->status = guarded(f);
}
template <class F> int32_t run_status3(AlphaShape3D* h, F&& f) {
    if (!h) {
        set_last_error("null AlphaShape3D handle");
        return kErrArgument;
    }
    h->status = guarded(f);
    return h->status;
}
void check_flags3() {
    const uint32_t f = read_scalar(ctx().d_flags + kFlagError);
    if (f) {
        fill<uint32_t>(ctx().d_flags, 1, 0u, ctx().stream);
        throw std::runtime_error(f == kErrCapacity ? "device capacity overflow (3D alpha-shape)"
                                                   : "device error flag raised");
    }
}
}  // namespace

extern "C" {

AlphaShape3D* AlphaShape3D_create(void) {
    try {
        (void)ctx();
        return new AlphaShape3D();
    } catch (const std::exception& e) {
        set_last_error(e.what());
        return nullptr;
    }
}

void AlphaShape3D_destroy(AlphaShape3D* h) { delete h; }

// Morton resolution (bits per axis, 1..21) of the next init.
int32_t AlphaShape3D_set_morton_bits(AlphaShape3D* h, int32_t bits) {
    return run_status3(h, [&] {
        if (bits < 1 || bits > 21) throw std::invalid_argument("3D Morton bits per axis must be in [1, 21]");
        h->bits = bits;
    });
}

// FP32 nodes: coords row-major [3N], alpha [N] (reference signature).
void AlphaShape3D_set_nodes(AlphaShape3D* h, uint32_t nnodes, const float* coords, const float* alpha) {
    run_void3(h, [&] {
        h->f64 = false;
        h->a32.set_nodes_host(nnodes, coords, alpha);
    });
}

int32_t AlphaShape3D_set_nodes_f64(AlphaShape3D* h, uint32_t nnodes, const double* coords, const double* alpha) {
    return run_status3(h, [&] {
        h->f64 = true;
        h->a64.set_nodes_host(nnodes, coords, alpha);
    });
}

// FP64 nodes already in device memory, rows (x, y, z, alpha).
int32_t AlphaShape3D_set_nodes_device_f64(AlphaShape3D* h, uint32_t nnodes, const double* d_xyzr) {
    return run_status3(h, [&] {
        h->f64 = true;
        h->a64.set_nodes_device(nnodes, reinterpret_cast<const Sph4<double>*>(d_xyzr));
    });
}

void AlphaShape3D_init(AlphaShape3D* h) {
    run_void3(h, [&] {
        if (h->f64) {
            h->a64.bits = h->bits;
            h->a64.init(ctx().stream);
        } else {
            h->a32.bits = h->bits;
            h->a32.init(ctx().stream);
        }
    });
}

void AlphaShape3D_compute(AlphaShape3D* h) {
    run_void3(h, [&] {
        if (h->f64)
            h->a64.compute(ctx().stream);
        else
            h->a32.compute(ctx().stream);
        check_flags3();
    });
}

uint32_t AlphaShape3D_get_nelem(const AlphaShape3D* hc) {
    AlphaShape3D* h = const_cast<AlphaShape3D*>(hc);
    uint32_t r = 0;
    run_void3(h, [&] { r = h->f64 ? h->a64.n_elems() : h->a32.n_elems(); });
    return r;
}

// Tetrahedra [4*nelem], Morton ids, each output by its lowest id.
void AlphaShape3D_get_elem(const AlphaShape3D* hc, uint32_t* elems) {
    AlphaShape3D* h = const_cast<AlphaShape3D*>(hc);
    run_void3(h, [&] {
        const uint32_t ne = h->f64 ? h->a64.n_elems() : h->a32.n_elems();
        d2h(elems, h->f64 ? h->a64.elemglob.p : h->a32.elemglob.p, 4ull * ne);
    });
}

void AlphaShape3D_get_ordered_nodes(AlphaShape3D* h, float* nodes) {
    run_void3(h, [&] {
        if (h->f64) throw std::invalid_argument("handle holds FP64 nodes: use AlphaShape3D_get_ordered_nodes_f64");
        std::vector<Sph4<float>> v(h->a32.n);
        d2h(v.data(), h->a32.lbvh.obj_m.p, h->a32.n);
        for (uint32_t i = 0; i < h->a32.n; ++i)
            for (int c = 0; c < 3; ++c) nodes[3 * i + c] = v[i].c[c];
    });
}

int32_t AlphaShape3D_get_ordered_nodes_f64(AlphaShape3D* h, double* nodes) {
    return run_status3(h, [&] {
        if (!h->f64) throw std::invalid_argument("handle holds FP32 nodes");
        std::vector<Sph4<double>> v(h->a64.n);
        d2h(v.data(), h->a64.lbvh.obj_m.p, h->a64.n);
        for (uint32_t i = 0; i < h->a64.n; ++i)
            for (int c = 0; c < 3; ++c) nodes[3 * i + c] = v[i].c[c];
    });
}

uint32_t AlphaShape3D_get_nedge(const AlphaShape3D* hc) {
    AlphaShape3D* h = const_cast<AlphaShape3D*>(hc);
    uint32_t r = 0;
    run_void3(h, [&] { r = h->f64 ? h->a64.n_edges() : h->a32.n_edges(); });
    return r;
}

// Edge CSR (AlphaShape3D::getEdge, cpp:90-98), edge flags (count <= 3) and
// node flags (getBoundaryNodes, cpp:101-105); any pointer may be null.
int32_t AlphaShape3D_get_edges(const AlphaShape3D* hc, uint32_t* row, uint32_t* neig, uint8_t* edge_is_bnd,
                               uint8_t* node_is_bnd) {
    AlphaShape3D* h = const_cast<AlphaShape3D*>(hc);
    return run_status3(h, [&] {
        auto go = [&](auto& A) {
            const uint32_t ne = A.n_edges();
            if (row) d2h(row, A.row.p, A.n + 1);
            if (neig) d2h(neig, A.neig.p, ne);
            if (edge_is_bnd) d2h(edge_is_bnd, A.edge_is_bnd.p, ne);
            if (node_is_bnd) d2h(node_is_bnd, A.node_is_bnd.p, A.n);
        };
        if (h->f64)
            go(h->a64);
        else
            go(h->a32);
    });
}

// perm[i] = input index of Morton slot i (getPermutation, cpp:75-80).
int32_t AlphaShape3D_get_permutation(const AlphaShape3D* hc, uint32_t* perm) {
    AlphaShape3D* h = const_cast<AlphaShape3D*>(hc);
    return run_status3(h, [&] {
        if (h->f64)
            d2h(perm, h->a64.lbvh.perm, h->a64.n);
        else
            d2h(perm, h->a32.lbvh.perm, h->a32.n);
    });
}

// Nodes that needed the exact stage; nodes whose candidate list was clamped.
uint32_t AlphaShape3D_get_nexact(const AlphaShape3D* hc) {
    AlphaShape3D* h = const_cast<AlphaShape3D*>(hc);
    uint32_t r = 0;
    run_void3(h, [&] { r = h->f64 ? h->a64.n_exact_nodes() : h->a32.n_exact_nodes(); });
    return r;
}
uint32_t AlphaShape3D_get_nclamped(const AlphaShape3D* hc) {
    AlphaShape3D* h = const_cast<AlphaShape3D*>(hc);
    uint32_t r = 0;
    run_void3(h, [&] { r = h->f64 ? h->a64.n_over_cap() : h->a32.n_over_cap(); });
    return r;
}

int32_t AlphaShape3D_last_status(const AlphaShape3D* h) { return h ? h->status : kErrArgument; }


// Nodal fields between input order and Morton order (permuteForward /
// permuteBackward, include/mesh/DirectAlphaShape3D.hpp): forward out[i] =
// in[perm[i]] gives the field in the Morton order of the outputs, backward
// out[perm[i]] = in[i] returns it to input order.  n elements of
// elem_bytes each; host arrays (copied) or device buffers (_device, on the
// library stream, not synchronised).  Needs init (the permutation).
}  // extern "C"

namespace {
template <class F> int32_t permute_call(const AlphaShape3D* hc, F&& f) {
    AlphaShape3D* h = const_cast<AlphaShape3D*>(hc);
    return run_status3(h, [&] {
        const bool ok = h->f64 ? h->a64.inited : h->a32.inited;
        if (!ok) throw std::invalid_argument("AlphaShape3D: permutation needs init (set_nodes)");
        const uint32_t* perm = h->f64 ? h->a64.lbvh.perm : h->a32.lbvh.perm;
        const uint32_t n = h->f64 ? h->a64.n : h->a32.n;
        f(perm, n);
    });
}
}  // namespace

extern "C" {

int32_t AlphaShape3D_permute_forward(const AlphaShape3D* h, const void* in, void* out, uint32_t elem_bytes) {
    return permute_call(h, [&](const uint32_t* perm, uint32_t n) {
        permute_host_elements(in, out, perm, n, elem_bytes, true);
    });
}
int32_t AlphaShape3D_permute_backward(const AlphaShape3D* h, const void* in, void* out, uint32_t elem_bytes) {
    return permute_call(h, [&](const uint32_t* perm, uint32_t n) {
        permute_host_elements(in, out, perm, n, elem_bytes, false);
    });
}
int32_t AlphaShape3D_permute_forward_device(const AlphaShape3D* h, const void* d_in, void* d_out, uint32_t elem_bytes) {
    return permute_call(h, [&](const uint32_t* perm, uint32_t n) {
        permute_elements(d_in, d_out, perm, n, elem_bytes, true, ctx().stream);
    });
}
int32_t AlphaShape3D_permute_backward_device(const AlphaShape3D* h, const void* d_in, void* d_out, uint32_t elem_bytes) {
    return permute_call(h, [&](const uint32_t* perm, uint32_t n) {
        permute_elements(d_in, d_out, perm, n, elem_bytes, false, ctx().stream);
    });
}


// One init + compute timed as testcases/IMR26/uniform3d.cpp times them:
// ms[0] tlbvh (LBVH build), ms[1] tashape (candidate search, local
// Delaunay + filter, element/edge scans), ms[2] tcompress (compaction to
// CSR), ms[3] the host wall time of both calls, ms[4] the GPU time from the
// build's start to the compaction's end; within tashape, ms[5] the
// candidate search, ms[6] the local Delaunay + filter of every node, ms[7]
// the exact redo of the nodes whose filters could not decide a sign.  GPU times come from HIP events
// on the library stream between the launches.
int32_t AlphaShape3D_timed_run(AlphaShape3D* h, double* ms) {
    return run_status3(h, [&] {
        if (!ms) throw std::invalid_argument("AlphaShape3D_timed_run: null ms");
        struct Disarm {
            ~Disarm() { sections_arm(false); }
        } disarm;
        sections_arm(true);
        const auto t0 = std::chrono::steady_clock::now();
        if (h->f64) {
            h->a64.init(ctx().stream);
            h->a64.compute(ctx().stream);
        } else {
            h->a32.init(ctx().stream);
            h->a32.compute(ctx().stream);
        }
        SA_HIP(hipStreamSynchronize(ctx().stream));
        const auto t1 = std::chrono::steady_clock::now();
        ms[0] = sections_elapsed(kMarkBuild0, kMarkRefit);
        ms[1] = sections_elapsed(kMarkCompute0, kMarkScans);
        ms[2] = sections_elapsed(kMarkCompress0, kMarkCompress);
        ms[3] = std::chrono::duration<double, std::milli>(t1 - t0).count();
        ms[4] = sections_elapsed(kMarkBuild0, kMarkCompress);
        ms[5] = sections_elapsed(kMarkCompute0, kMarkFill);
        ms[6] = sections_elapsed(kMarkFill, kMarkDelaunayMain);
        ms[7] = sections_elapsed(kMarkDelaunayMain, kMarkDelaunay);
        sections_arm(false);
        check_flags3();
    });
}

}  // extern "C"
