// Constraint-segment recovery on gfx950.
//
// Reference: addConstraints (addConstraints.cu:1723-1835) locates each
// segment, collects the triangles it crosses, builds the upper/lower vertex
// chains and retriangulates each chain (formPolygon_s1/s2, calDistance,
// makeTree, reTriangle, :1491-1721).  It drops segments that pass through a
// vertex (:962-965).  Here:
//   1. split pass: every segment is walked through the Delaunay mesh and cut
//      at the vertices lying exactly on it into pieces (a, b) with no vertex
//      in their open interior; pieces that already are edges are marked
//      constrained at once;
//   2. rounds: every pending piece walks its crossed triangles and claims
//      them (atomicMin of a per-round key, smallest piece id wins); a piece
//      that owns all its crossed triangles retriangulates its cavity in
//      place: the left and right pseudo-polygons are triangulated by the
//      recursive Delaunay-vertex rule (for base (A,B) pick the chain vertex
//      C whose circle through A,B contains no other chain vertex, recurse on
//      (A,C) and (C,B)), which reuses exactly the crossed slots (k crossing
//      edges -> k+1 triangles before and after);
//   3. outer adjacency is resolved after all cavities of the round are
//      written (a neighbour rewritten in the same round is found in its
//      cavity's slot list);
// and the caller finishes with constrained flips.
#include <algorithm>
#include <climits>

#include "cons_bodies.hpp"
#include "mesh.hpp"

namespace gcdt {

__global__ __launch_bounds__(kBlock) void k_split_count(Cons c, const int2* cons, int C, int nmax, int* cnt)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < C; i += (long long)gridDim.x * blockDim.x) {
        int2 e = cons[i];
        if (e.x < 0 || e.y < 0 || e.x >= nmax || e.y >= nmax || e.x == e.y) {
            atomicOr(c.err, MERR_INVALID);
            cnt[i] = 0;
            continue;
        }
        cnt[i] = split_walk(c, e.x, e.y, nullptr);
    }
}

__global__ __launch_bounds__(kBlock) void k_split_emit(Cons c, const int2* cons, int C, const int* off, int2* pieces)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < C; i += (long long)gridDim.x * blockDim.x) {
        int2 e = cons[i];
        if (off[i + 1] == off[i]) continue;
        split_walk(c, e.x, e.y, pieces + off[i]);
    }
}

__global__ __launch_bounds__(kBlock) void k_build_vt(const int3* tri, int T, int* vt)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < T; i += (long long)gridDim.x * blockDim.x) {
        int3 t = tri[i];
        vt[t.x] = (int)i;
        vt[t.y] = (int)i;
        vt[t.z] = (int)i;
    }
}

// queue of pieces that need a cavity (first vertex >= 0)
__global__ __launch_bounds__(kBlock) void k_piece_queue(const int2* pieces, int np, int* q, int* nq)
{
    WAVE_LOOP(i, np)
    {
        bool want = i < np && pieces[i].x >= 0;
        int slot = wave_alloc(want ? 1 : 0, nq);
        if (want) q[slot] = (int)i;
    }
}

// ---------------------------------------------------------------- rounds

__device__ inline unsigned cell_morton(unsigned x, unsigned y)
{
    x = (x | (x << 8)) & 0x00FF00FFu;
    x = (x | (x << 4)) & 0x0F0F0F0Fu;
    x = (x | (x << 2)) & 0x33333333u;
    x = (x | (x << 1)) & 0x55555555u;
    y = (y | (y << 8)) & 0x00FF00FFu;
    y = (y | (y << 4)) & 0x0F0F0F0Fu;
    y = (y | (y << 2)) & 0x33333333u;
    y = (y | (y << 1)) & 0x55555555u;
    return x | (y << 1);
}

// wave_alloc on a 64-bit counter: the triangles that all pieces cross may be
// more than an int counts
__device__ inline long long wave_alloc_64(int k, unsigned long long* counter)
{
    int total;
    const int ex = wave_excl_scan(k, total);
    unsigned long long base = 0;
    if (__lane_id() == 0 && total > 0) base = atomicAdd(counter, (unsigned long long)total);
    return (long long)__shfl(base, 0, 64) + ex;
}

// R1: claim crossed triangles; pieces that became edges are retired.  One
// thread per piece: a walk that collects the crossed triangles in LDS, then
// the claims and the path for the later steps (paths[] at ppos[i], room
// permitting: the cursor counts on, and the caller repeats the launch with a
// larger buffer).  A piece that crosses more than CAV_WAVE_K triangles goes
// to the long list.
__global__ __launch_bounds__(kBlock) void k_cav_claim(Cons c, const int2* pieces, const int* q, const int* nq,
                                                      unsigned epoch, int* ncross, int* paths, int pcap,
                                                      unsigned long long* pcur, int* ppos, int* longq, int* nlong)
{
    constexpr int KEEP = CAV_WAVE_K | 1;  // odd stride: no bank conflicts
    __shared__ int s_keep[kBlock * KEEP];
    int* mine = s_keep + threadIdx.x * KEEP;
    int n = *nq;
    WAVE_LOOP(i, n)
    {
        int k = 0;
        bool lng = false;
        if (i < n) {
            const int pi = q[i];
            const int2 pc = pieces[pi];
            int m = 0;
            k = cav_walk(c, pc.x, pc.y, true, nullptr, [&](int t) { mine[m++] = t; }, CAV_WAVE_K);
            lng = k == -3;
            // steiner mode: a piece that crosses a recovered one is deferred
            // and claims nothing (its claims would block others)
            if (k == -2) c.defer[pi] = 1;
            if (k == -1) atomicOr(c.err, MERR_WALK);
            if (k < 0) k = 0;
            ncross[i] = k;
            const unsigned long long key = cav_key(epoch, pi);
            for (int j = 0; j < k; j++) atomicMin(&c.owner[mine[j]], key);
        }
        const long long off = wave_alloc_64(k, pcur);
        if (k > 0) ppos[i] = (int)off;
        if (k > 0 && off + k <= pcap)
            for (int j = 0; j < k; j++) paths[off + j] = mine[j];
        const int l = wave_alloc(lng ? 1 : 0, nlong);
        if (lng) longq[l] = (int)i;
    }
}

// steps of a seed's walk (a neighbour in Morton order is a few triangles away,
// or far; every lane of the wave waits for the longest walk)
constexpr int SEED_STEPS = 20;

// A triangle that piece (A, B) crosses near its point X, for a lane that walks
// a part of the piece: from a vertex near X in the points' Morton order, an
// edge-to-edge walk to the triangle that holds X.  It serves when its
// vertices lie strictly on both sides of the line and the edge (r, l) by which
// the piece leaves it -- from right to left in its counter-clockwise order --
// is crossed between A and B.  False when there is none (the piece is then
// walked on from the lane before).
__device__ inline bool cav_seed(const Cons& c, int2 A, int2 B, int2 X, const int* cell_end, int& t, int& r, int& l)
{
    const Mesh& m = c.m;
    const unsigned cell = cell_morton((unsigned)X.x >> 20, (unsigned)X.y >> 20);
    const int n = cell_end[(1 << 20) - 1], e = cell_end[cell];
    const int v0 = e > 0 ? e - 1 : 0, v1 = e < n ? e : v0;
    const int2 P0 = m.pts[v0], P1 = m.pts[v1];
    const long long d0 = (long long)abs(P0.x - X.x) + abs(P0.y - X.y), d1 = (long long)abs(P1.x - X.x) + abs(P1.y - X.y);
    t = c.vt[d0 <= d1 ? v0 : v1];
    for (int g = 0; g < SEED_STEPS && t >= 0; g++) {
        const int3 tv = m.tri[t], ta = m.adj[t];
        const int2 P[3] = {m.pts[tv.x], m.pts[tv.y], m.pts[tv.z]};
        int out = -1;
#pragma unroll
        for (int k = 0; k < 3; k++)
            if (out < 0 && orient2d(P[(k + 1) % 3], P[(k + 2) % 3], X) < 0) out = k;
        if (out < 0) {
            const int s0 = orient2d(A, B, P[0]), s1 = orient2d(A, B, P[1]), s2 = orient2d(A, B, P[2]);
            if (s0 == 0 || s1 == 0 || s2 == 0) return false;
            // the directed edge from a right vertex to a left one
            const int k = s1 < 0 && s2 > 0 ? 0 : (s2 < 0 && s0 > 0 ? 1 : (s0 < 0 && s1 > 0 ? 2 : -1));
            if (k < 0) return false;
            r = get3(tv, nx3(k));
            l = get3(tv, pv3(k));
            const int2 R = k == 0 ? P[1] : (k == 1 ? P[2] : P[0]), L = k == 0 ? P[2] : (k == 1 ? P[0] : P[1]);
            return orient2d(R, L, A) * orient2d(R, L, B) < 0;
        }
        t = get3(ta, out);
    }
    return false;
}

// R1 for the long list, one wave per piece.  With the points' Morton cells
// (cell_end) every lane finds a triangle of its own along the piece and walks
// from it until it meets another lane's, so a piece is walked in 64 parts at
// once; the parts that follow one another from the first endpoint give the
// crossed triangles in order; they are claimed and kept in paths[].
// Bound by the chain of loads of the longest part and of the slowest seed.
// 1,000 rows over 100,000 points (350 crossed triangles on average), per
// round: two whole walks on one thread, 380 + 330 us -> 25 us for the short
// walk that finds the piece long and 43 us here.
constexpr int WALK_HASH = 256;
constexpr int WALK_KEEP = 32;  // triangles of a part kept in LDS (longer parts are walked twice)

__global__ __launch_bounds__(64) void k_cav_walk_long(Cons c, const int2* pieces, const int* q, const int* longq,
                                                      const int* nlong, const int* cell_end, unsigned epoch,
                                                      int* ncross, int* total, int* paths, int pcap,
                                                      unsigned long long* pcur, int* ppos)
{
    __shared__ int s_tag[WALK_HASH], s_lane[WALK_HASH];
    __shared__ int s_next[64], s_sum[64], s_st[64], s_on[64];
    __shared__ int s_keep[64 * WALK_KEEP];
    __shared__ int s_off;
    const int lane = threadIdx.x;
    const int n = *nlong;
    for (int w = blockIdx.x; w < n; w += gridDim.x) {
        const int i = longq[w], pi = q[i];
        const int2 pc = pieces[pi];
        const int b = pc.y;
        const int2 A = c.m.pts[pc.x], B = c.m.pts[b];
        for (int h = lane; h < WALK_HASH; h += 64) s_tag[h] = -1;
        __syncthreads();
        // ---- the lanes' first triangles, each kept by one lane
        int t0 = -1, r0 = -1, l0 = -1;
        bool mine = false;
        int st = 0;  // 1 walk failed, 2 met a constrained edge
        if (lane == 0) {
            int s;
            if (find_wedge(c, pc.x, b, t0, s) == 0) {
                const int3 tv = c.m.tri[t0];
                r0 = get3(tv, nx3(s));
                l0 = get3(tv, pv3(s));
                mine = true;
            } else {
                st = 1;
            }
        } else if (cell_end) {
            const int2 X = make_int2(A.x + (int)(((long long)B.x - A.x) * lane / 64),
                                     A.y + (int)(((long long)B.y - A.y) * lane / 64));
            mine = cav_seed(c, A, B, X, cell_end, t0, r0, l0);
        }
        if (mine) {
            for (unsigned h = hash32((uint32_t)t0);; h++) {  // at most 64 tags in 256 places
                const int g = atomicCAS(&s_tag[h % WALK_HASH], -1, t0);
                if (g == -1) {
                    s_lane[h % WALK_HASH] = lane;
                    break;
                }
                if (g == t0) {
                    mine = false;
                    break;
                }
            }
        }
        __syncthreads();
        // ---- each lane's part: up to another lane's first triangle, or b
        int cnt = 0, next = 64;
        if (mine) {
            int rr = r0, ll = l0;
            Cross wk;
            wk.start(c.m, t0);
            s_keep[lane * WALK_KEEP] = t0;
            cnt = 1;
            for (int g = 0; g < (1 << 26); g++) {
                int nb, v;
                int2 PV;
                if (wk.step(c.m, rr, ll, nb, v, PV)) {
                    st = 2;
                    break;
                }
                if (nb < 0) {
                    st = 1;
                    break;
                }
                int found = -1;
                for (unsigned h = hash32((uint32_t)nb);; h++) {
                    const int tag = s_tag[h % WALK_HASH];
                    if (tag == nb) found = s_lane[h % WALK_HASH];
                    if (tag == nb || tag == -1) break;
                }
                if (found >= 0) {
                    next = found;
                    break;
                }
                if (cnt < WALK_KEEP) s_keep[lane * WALK_KEEP + cnt] = nb;
                cnt++;
                if (v == b) break;
                const int o = orient2d(A, B, PV);
                if (o == 0) {
                    st = 1;
                    break;
                }
                if (o > 0) ll = v;
                else rr = v;
            }
        }
        // ---- the chain of parts from lane 0: sums to the end, members
        s_next[lane] = next;
        s_sum[lane] = cnt;
        s_st[lane] = st;
        s_on[lane] = lane == 0;
        __syncthreads();
        int jump = next, sum = cnt;
        for (int d = 0; d < 6; d++) {
            int js = 0, jn = 64, jst = 0;
            const bool on = s_on[lane] != 0;
            if (jump < 64) {
                js = s_sum[jump];
                jn = s_next[jump];
                jst = s_st[jump];
            }
            __syncthreads();
            if (jump < 64) {
                if (on) s_on[jump] = 1;
                sum += js;
                st |= jst;
                jump = jn;
            }
            s_sum[lane] = sum;
            s_next[lane] = jump;
            s_st[lane] = st;
            __syncthreads();
        }
        const int K = s_sum[0], bad = s_st[0];
        const bool on = s_on[lane] != 0;
        if (lane == 0) {
            s_off = -1;
            if (bad & 1) atomicOr(c.err, MERR_WALK);
            else if (bad && c.steiner) c.defer[pi] = 1;
            else if (bad) atomicOr(c.err, MERR_CROSSING | MERR_WALK);
            if (bad) {
                ncross[i] = 0;
            } else {
                const long long off = (long long)atomicAdd(pcur, (unsigned long long)K);
                ncross[i] = K;
                ppos[i] = (int)off;
                atomicAdd(total, K);
                if (off + K <= pcap) s_off = (int)off;
            }
        }
        __syncthreads();
        const int off = s_off;
        if (off >= 0 && on && cnt > 0) {
            const unsigned long long key = cav_key(epoch, pi);
            int* out = paths + off + (K - sum);
            const int kept = cnt < WALK_KEEP ? cnt : WALK_KEEP;
            for (int j = 0; j < kept; j++) {
                const int t = s_keep[lane * WALK_KEEP + j];
                out[j] = t;
                atomicMin(&c.owner[t], key);
            }
            if (cnt > kept) {
                int rr = r0, ll = l0;
                Cross wk;
                wk.start(c.m, t0);
                for (int j = 1; j < cnt; j++) {
                    int nb, v;
                    int2 PV;
                    wk.step(c.m, rr, ll, nb, v, PV);
                    if (j >= kept) {
                        out[j] = nb;
                        atomicMin(&c.owner[nb], key);
                    }
                    if (orient2d(A, B, PV) > 0) ll = v;
                    else rr = v;
                }
            }
        }
        __syncthreads();
    }
}

// R2: a piece that owns every triangle it crosses wins (its path goes to its
// scratch); the others stay queued.
__global__ __launch_bounds__(kBlock) void k_cav_check(Cons c, const int* q, const int* nq, const int* ncross,
                                                      const int* paths, const int* ppos, unsigned epoch, int* q2,
                                                      int* nq2, Win* wins, int* nwin, int* scr, int* scr_cursor,
                                                      long long scr_cap)
{
    int n = *nq;
    WAVE_LOOP(i, n)
    {
        int pi = -1, K = 0;
        const int* path = nullptr;
        bool win = false, keep = false;
        if (i < n) {
            pi = q[i];
            K = ncross[i];
            if (K > 0 && K <= CAV_WAVE_K) {
                path = paths + ppos[i];
                const unsigned long long key = cav_key(epoch, pi);
                bool all = true;
                for (int j = 0; j < K; j++) all &= c.owner[path[j]] == key;
                win = all;
                keep = !all;
            }
        }
        int need = win ? K : 0;
        int off = wave_alloc(need, scr_cursor);
        if (win && off + (long long)need > scr_cap) {
            win = false;  // defer to a later round
            keep = true;
        }
        int ws = wave_alloc(win ? 1 : 0, nwin);
        if (win) {
            wins[ws] = Win{pi, path[0], K, off};
            for (int j = 0; j < K; j++) scr[off + j] = path[j];
        }
        int qs = wave_alloc(keep ? 1 : 0, nq2);
        if (keep) q2[qs] = pi;
    }
}

// one wave per long piece: its path against the claims, and a winner's path
// to the head of its scratch; longw lists the winners, big ones from the end
__global__ __launch_bounds__(kBlock) void k_cav_check_long(Cons c, const int* q, const int* longq, const int* nlong,
                                                           const int* ncross, const int* paths, const int* ppos,
                                                           unsigned epoch, int* q2, int* nq2, Win* wins, int* nwin,
                                                           int* scr, int* scr_cursor, long long scr_cap, int* longw,
                                                           int* nmid, int* nbig, int big_k)
{
    const int lane = __lane_id();
    const int n = *nlong;
    for (int w = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6); w < n; w += (int)((gridDim.x * blockDim.x) >> 6)) {
        const int i = longq[w], pi = q[i], K = ncross[i];
        if (K <= 0) continue;  // deferred, or an error is flagged
        const int* path = paths + ppos[i];
        const unsigned long long key = cav_key(epoch, pi);
        bool ok = true;
        for (int j = lane; j < K; j += 64) ok &= c.owner[path[j]] == key;
        bool win = __ballot(!ok) == 0;
        int off = 0;
        if (win) {
            const int need = (int)cav_block_ints(K);
            if (lane == 0) off = atomicAdd(scr_cursor, need);
            off = __shfl(off, 0, 64);
            win = off + (long long)need <= scr_cap;  // else defer to a later round
        }
        if (win)
            for (int j = lane; j < K; j += 64) scr[off + j] = path[j];
        if (lane == 0) {
            if (win) {
                const int ws = atomicAdd(nwin, 1);
                wins[ws] = Win{pi, path[0], K, off};
                if (K > big_k) longw[n - 1 - atomicAdd(nbig, 1)] = ws;
                else longw[atomicAdd(nmid, 1)] = ws;
            } else {
                q2[atomicAdd(nq2, 1)] = pi;
            }
        }
    }
}

// R3: collect the cavity and retriangulate it in place (one thread per cavity
// of up to CAV_WAVE_K triangles, its arrays in LDS: a batch of 32
// small instances took 24 us per round with them in global memory, 17 us so).
constexpr int RETRI_BS = 64;

__global__ __launch_bounds__(RETRI_BS) void k_cav_retri(Cons c, const int2* pieces, const Win* wins, const int* nwin,
                                                        unsigned epoch)
{
    constexpr int INTS = (13 * CAV_WAVE_K + 20) | 1;  // cav_scratch_ints, an odd stride
    __shared__ int s_scr[RETRI_BS * INTS];
    int nw = *nwin;
    for (long long wi = (long long)blockIdx.x * blockDim.x + threadIdx.x; wi < nw; wi += (long long)gridDim.x * blockDim.x)
        if (wins[wi].K <= CAV_WAVE_K)
            cav_retri_one(c, pieces, wins, (int)wi, s_scr, epoch, s_scr + threadIdx.x * INTS);
}

// Delaunay vertex found by the 64 lanes of a wave: each scans every 64th
// candidate as DvScan does, then a butterfly keeps the better of two
// candidates -- the one strictly inside the other's circle, the lower index
// when cocircular -- which is the vertex DvScan returns.
struct DvWave {
    __device__ static int find(const int* PX, const int* PY, int lo, int hi, int2 PA, int2 PB)
    {
        const int lane = __lane_id();
        int ci = -1;
        int2 PC = make_int2(0, 0);
        for (int i = lo + lane; i < hi; i += 64) {
            const int2 PI = make_int2(PX[i], PY[i]);
            if (ci < 0 || incircle(PA, PB, PC, PI) > 0) {
                ci = i;
                PC = PI;
            }
        }
        for (int d = 32; d > 0; d >>= 1) {
            const int oi = __shfl(ci, lane ^ d, 64);
            const int ox = __shfl(PC.x, lane ^ d, 64), oy = __shfl(PC.y, lane ^ d, 64);
            if (oi < 0) continue;
            const int2 PO = make_int2(ox, oy);
            bool take = ci < 0;
            if (!take) {
                const int r = incircle(PA, PB, PC, PO);
                take = r > 0 || (r == 0 && oi < ci);
            }
            if (take) {
                ci = oi;
                PC = PO;
            }
        }
        return ci;
    }
};

// Cavities of up to this many crossed triangles keep their arrays in LDS (the
// larger block's; the smaller one's is CAV_MID_K).
#ifndef GCDT_CAV_MID_K
#define GCDT_CAV_MID_K 128
#endif
#ifndef GCDT_CAV_FEW
#define GCDT_CAV_FEW 1024  // long pieces of a round
#endif
#ifndef GCDT_CAV_LDS_K
#define GCDT_CAV_LDS_K 2048
#endif
constexpr int CAV_MID_K = GCDT_CAV_MID_K;
constexpr int CAV_FEW = GCDT_CAV_FEW;
constexpr int CAV_LDS_K = GCDT_CAV_LDS_K;
// nodes of up to this many candidates are scanned by as many lanes, several
// nodes at once; larger ones by a wave each
constexpr int CAV_SCAN = 16;
constexpr int cav_lds_ints(int K) { return 7 * K + 10; }

// The cavity of `path` retriangulated by a workgroup: the same triangles in
// the same slots as cav_retri_one.  The recursive Delaunay-vertex rule fixes
// the tree, and its order (right part before left) fixes the slot of every
// node: node (lo, hi) at slot e has its right part (ci + 1, hi) at e + 1 and
// its left part (lo, ci) at e + hi - ci.  So all nodes of one depth, of both
// pseudo-polygons, are done at once.  Bound by the tree's depth times a scan's chain of in-circle
// tests.  One wave doing node after node took 1.6 us a node: 1,000 rows over
// 100,000 points 1,080 -> 103 us per round.
// buf: cav_lds_ints(K) ints (LDS, or the cavity's scratch).  s_list, s_ctl:
// LDS of 64 and 4 ints.
template <int BS>
__device__ void cav_block_retri(const Cons& c, int a, int b, const int* slots, int K, int* newown, int wi,
                                unsigned epoch, int* buf, int* s_list, int* s_ctl)
{
    const Mesh& m = c.m;
    int* V = buf;            // K: chain vertices, left then right, in polygon order
    int* PK = V + K;         // K + 2: boundary edges by place: neighbour + 1, low bit the constraint bit
    int* PX = PK + K + 2;    // K + 4: polygon coordinates, left 0..nl+1 then right 0..nr+1
    int* PY = PX + K + 4;    // K + 4
    int* MS = PY + K + 4;    // K: size of the node that starts here, bit 30 its depth's parity; 0 none
    int* E0 = MS + K;        // K: its slot index
    int* PAR = E0 + K;       // K: the triangle across its base
    const int2 PA = m.pts[a], PB = m.pts[b];
    const int lane = __lane_id();
    // ---- collect: every crossed triangle's entry edge and apex follow from
    // its vertices' sides of the piece
    int carry = 0;  // left vertices added by the middle triangles so far
    bool bad = false;
    for (int j0 = 0; j0 < K; j0 += BS) {
        const int j = j0 + (int)threadIdx.x;
        int side = 0;  // +1 / -1: a middle triangle that adds a left / right vertex
        int t = -1, v = -1, nb = -1, cf = 0;
        int2 PV = make_int2(0, 0);
        int3 tv, ta;
        int k = -1;
        if (j < K) {
            t = slots[j];
            tv = m.tri[t];
            ta = m.adj[t];
            cf = m.cflag[t];
            if (j == 0) {
                k = slot_of(tv, a);
            } else if (j == K - 1) {
                k = slot_of(tv, b);
            } else {
                const int s0 = orient2d(PA, PB, m.pts[tv.x]), s1 = orient2d(PA, PB, m.pts[tv.y]),
                          s2 = orient2d(PA, PB, m.pts[tv.z]);
                // the entry edge runs from a left vertex to a right one
                k = s1 > 0 && s2 < 0 ? 0 : (s2 > 0 && s0 < 0 ? 1 : (s0 > 0 && s1 < 0 ? 2 : -1));
                if (k >= 0) side = k == 0 ? s0 : (k == 1 ? s1 : s2);
                if (side == 0) k = -1;
            }
            if (k < 0) bad = true;
        }
        int tot;
        const int before = carry + block_excl_prefix<BS>(side > 0 ? 1 : 0, &tot);
        carry += tot;
        if (k >= 0) {
            const int kn = nx3(k), kp = pv3(k);  // left and right vertex of the entry edge (of the exit edge for j = 0: right, left)
            int place;
            if (j == 0) {
                const int r = get3(tv, kn), l = get3(tv, kp);
                const int2 PR = m.pts[r], PL = m.pts[l];
                V[0] = l;
                PX[1] = PL.x;
                PY[1] = PL.y;
                PK[0] = ((get3(ta, kn) + 1) << 1) | ((cf >> kn) & 1);
                V[K - 1] = r;
                PX[K + 2] = PR.x;
                PY[K + 2] = PR.y;
                PK[K + 1] = ((get3(ta, kp) + 1) << 1) | ((cf >> kp) & 1);
                place = 0;
            } else if (j == K - 1) {
                const int nl = 1 + before;  // no middle triangle follows
                PK[nl] = ((get3(ta, kp) + 1) << 1) | ((cf >> kp) & 1);
                PK[nl + 1] = ((get3(ta, kn) + 1) << 1) | ((cf >> kn) & 1);
                place = nl;
            } else {
                v = get3(tv, k);
                PV = m.pts[v];
                const int L = 1 + before;  // left vertices before this triangle
                const int R = j + 1 - L;   // right ones
                if (side > 0) {
                    nb = get3(ta, kp);
                    cf = (cf >> kp) & 1;
                    place = L;
                    V[L] = v;
                    PX[L + 1] = PV.x;
                    PY[L + 1] = PV.y;
                } else {
                    nb = get3(ta, kn);
                    cf = (cf >> kn) & 1;
                    place = K + 1 - R;
                    V[K - 1 - R] = v;
                    PX[K + 2 - R] = PV.x;
                    PY[K + 2 - R] = PV.y;
                }
                PK[place] = ((nb + 1) << 1) | cf;
            }
            c.owner[t] = cav_place(place);
        }
    }
    const int nl = 1 + carry, nr = K - nl;
    if (threadIdx.x == 0) {
        PX[0] = PA.x;
        PY[0] = PA.y;
        PX[nl + 1] = PB.x;
        PY[nl + 1] = PB.y;
        PX[nl + 2] = PB.x;
        PY[nl + 2] = PB.y;
        PX[K + 3] = PA.x;
        PY[K + 3] = PA.y;
        s_ctl[0] = 0;  // large nodes listed
        s_ctl[1] = 0;  // nodes done at this depth
        s_ctl[2] = 0;  // inconsistent
    }
    for (int g = threadIdx.x; g < K; g += BS) MS[g] = 0;
    __syncthreads();
    if (bad) s_ctl[2] = 1;
    if (threadIdx.x == 0) {
        MS[0] = nl;
        E0[0] = 0;
        PAR[0] = slots[nl < K ? nl : 0];  // the two top triangles share the piece
        if (nr > 0) {
            MS[nl] = nr;
            E0[nl] = nl;
            PAR[nl] = slots[0];
        }
    }
    __syncthreads();
    if (s_ctl[2] || nr < 1) {  // block-uniform
        if (threadIdx.x == 0) at_or(c.err, MERR_CAVITY);
        __syncthreads();
        return;
    }
    // node at position g of size sz: its triangle is written, its parts start
    auto emit = [&](int g, int sz, int ci_off, int par_bit) {
        const bool right = g >= nl;
        const int M = right ? nr : nl, base = right ? nl : 0;
        const int lo = g - base + 1, hi = lo + sz, ci = lo + ci_off;
        auto vtx = [&](int i) -> int { return i == 0 ? (right ? b : a) : (i == M + 1 ? (right ? a : b) : V[base + i - 1]); };
        const int e0 = E0[g], par = PAR[g];
        const int T = slots[e0];
        const int vA = vtx(lo - 1), vB = vtx(hi), vC = vtx(ci);
        const int nleft = ci - lo, nright = hi - ci - 1;
        int3 na;
        int cf = sz == M ? 4 : 0;  // the whole polygon: its base is the piece
        na.z = par;
        if (nleft > 0) {
            na.y = slots[e0 + 1 + nright];
            MS[g] = nleft | ((par_bit ^ 1) << 30);
            E0[g] = e0 + 1 + nright;
            PAR[g] = T;
        } else {
            const int p = (right ? nl + 1 : 0) + lo - 1, x = PK[p];
            na.y = adj_mark((x >> 1) - 1);
            cf |= (x & 1) << 1;
            newown[p] = T;
            MS[g] = 0;
        }
        if (nright > 0) {
            na.x = slots[e0 + 1];
            const int h = g + ci_off + 1;
            E0[h] = e0 + 1;
            PAR[h] = T;
            MS[h] = nright | ((par_bit ^ 1) << 30);
        } else {
            const int p = (right ? nl + 1 : 0) + ci, x = PK[p];
            na.x = adj_mark((x >> 1) - 1);
            cf |= x & 1;
            newown[p] = T;
        }
        m.tri[T] = make_int3(vA, vB, vC);
        m.adj[T] = na;
        m.cflag[T] = cf;
        c.stamp[T] = (int)epoch;
        c.cavof[T] = wi;
        c.vt[vA] = T;
        c.vt[vB] = T;
        c.vt[vC] = T;
    };
    // coordinates of node (g, sz): first candidate, and the base's ends
    auto first = [&](int g) { return g >= nl ? g + 3 : g + 1; };
    for (int par_bit = 0;; par_bit ^= 1) {
        bool did = false;
        for (int g0 = (int)(threadIdx.x & ~63u); g0 < K; g0 += BS) {
            // 64 positions per wave: their nodes of up to CAV_SCAN candidates are
            // scanned together, one candidate per lane
            const int g = g0 + lane;
            const int x = g < K ? MS[g] : 0;
            const bool head = x != 0 && ((x >> 30) & 1) == par_bit;
            const int sz = x & ((1 << 30) - 1);
            const bool small = head && sz <= CAV_SCAN && lane + sz <= 64;
            did |= head;
            if (head && !small) {
                const int s = atomicAdd(&s_ctl[0], 1);
                if (s < 64) s_list[s] = g;  // the others wait for the next depth of this parity
            }
            const unsigned long long heads = __ballot(small);
            if (heads == 0) continue;
            const unsigned long long upto = heads & ((2ull << lane) - 1);
            const int hl = upto ? 63 - __clzll(upto) : lane;
            const int hsz = __shfl(sz, hl, 64);
            const bool in = upto != 0 && lane - hl < hsz;
            const int f = first(g0 + hl), end = hl + hsz;
            int2 NA = make_int2(0, 0), NB = NA, PC = NA;
            if (in) {
                NA = make_int2(PX[f - 1], PY[f - 1]);
                NB = make_int2(PX[f + hsz], PY[f + hsz]);
                PC = make_int2(PX[f + lane - hl], PY[f + lane - hl]);
            }
            int ci = lane - hl;
            for (int d = 1; d < CAV_SCAN; d <<= 1) {
                // a lane holds the best of d candidates: the lower one stays on a
                // tie, as in DvScan
                const int oi = __shfl_down(ci, d, 64);
                const int ox = __shfl_down(PC.x, d, 64), oy = __shfl_down(PC.y, d, 64);
                const bool pair = in && lane + d < end;
                if (__ballot(pair) == 0) break;
                if (pair && incircle(NA, NB, PC, make_int2(ox, oy)) > 0) {
                    ci = oi;
                    PC = make_int2(ox, oy);
                }
            }
            if (small) emit(g, sz, ci, par_bit);
        }
        if (did) s_ctl[1] = 1;
        __syncthreads();
        const int nbig = min(s_ctl[0], 64);
        if (s_ctl[1] == 0) break;  // block-uniform
        __syncthreads();
        if (threadIdx.x == 0) {
            s_ctl[0] = 0;
            s_ctl[1] = 0;
        }
        for (int s = (int)(threadIdx.x >> 6); s < nbig; s += BS / 64) {
            const int g = s_list[s];
            const int sz = MS[g] & ((1 << 30) - 1);
            const int f = first(g);
            const int ci = DvWave::find(PX, PY, f, f + sz, make_int2(PX[f - 1], PY[f - 1]),
                                        make_int2(PX[f + sz], PY[f + sz]));
            if (__lane_id() == 0) emit(g, sz, ci - f, par_bit);
        }
        __syncthreads();
    }
    __syncthreads();
}

// R3 for long pieces, a workgroup per cavity: BIG takes those above CAV_MID_K.
template <int BS, int CAP, bool BIG>
__global__ __launch_bounds__(BS) void k_cav_retri_block(Cons c, const int2* pieces, const Win* wins, const int* longw,
                                                        const int* nw, const int* nlong, int* scr, unsigned epoch,
                                                        int* rew, int* nrew)
{
    __shared__ int s_buf[cav_lds_ints(CAP)];
    __shared__ int s_list[64], s_ctl[4];
    __shared__ int s_base;
    const int n = *nw, nl = *nlong;
    for (int q = blockIdx.x; q < n; q += gridDim.x) {
        const int wi = longw[BIG ? nl - 1 - q : q];
        const Win w = wins[wi];
        const int2 pc = pieces[w.piece];
        int* slots = scr + w.off;
        int* newown = slots + w.K;
        if (w.K <= CAP)
            cav_block_retri<BS>(c, pc.x, pc.y, slots, w.K, newown, wi, epoch, s_buf, s_list, s_ctl);
        else
            cav_block_retri<BS>(c, pc.x, pc.y, slots, w.K, newown, wi, epoch, newown + w.K + 2, s_list, s_ctl);
        if (threadIdx.x == 0) s_base = atomicAdd(nrew, w.K);
        __syncthreads();
        for (int j = threadIdx.x; j < w.K; j += BS) rew[s_base + j] = slots[j];
        __syncthreads();
    }
}

// R4: resolve the marked outer adjacency of rewritten triangles, a thread per
// triangle: FIX_LANES lanes per cavity of up to CAV_WAVE_K, the others listed
constexpr int FIX_LANES = 16;
static_assert(CAV_WAVE_K <= FIX_LANES, "lanes per short cavity");

// (touched != nullptr: every rewritten triangle is flagged there, and listed
// the first time)
__global__ __launch_bounds__(kBlock) void k_cav_fix(Cons c, const Win* wins, const int* nwin, const int* scr,
                                                    const int* rew, const int* nrew, unsigned epoch, int* touched,
                                                    int* tlist, int* ntlist, int tcap)
{
    __shared__ int s_buf[STAGE_CAP];
    __shared__ int s_base;
    Staged<STAGE_CAP> sl(s_buf, &s_base, tlist, ntlist, tcap, c.err, MERR_CAPACITY);
    const long long nw = *nwin, ns = nw * FIX_LANES;
    const int n = *nrew;
    // short cavities first, then the listed triangles, in whole tiles
    const long long s0 = (ns + kBlock - 1) / kBlock * kBlock;
    TILE_LOOP(base, s0 + n, kBlock)
    {
        const long long i = base + threadIdx.x;
        int t = -1;
        if (i < ns) {
            const Win w = wins[i / FIX_LANES];
            const int j = (int)(i % FIX_LANES);
            if (w.K <= CAV_WAVE_K && j < w.K) t = scr[w.off + j];
        } else if (i >= s0 && i < s0 + n) {
            t = rew[i - s0];
        }
        bool first = false;
        if (t >= 0) {
            cav_fix_one(c, wins, scr, t, epoch, true);
            if (touched && !touched[t]) {
                touched[t] = 1;
                first = tlist != nullptr;
            }
        }
        const int at = sl.reserve(first ? 1 : 0);
        if (first) s_buf[at] = t;
    }
    sl.flush();
}

// move: the pieces left by the round before are the queue
__global__ void k_cav_begin(int* cnt, int move)
{
    if (move) {
        cnt[C_NQ] = cnt[C_NQ2];
        cnt[C_STUCK] = cnt[C_NQ2] > 0 && cnt[C_NWIN] == 0;
    }
    cnt[C_NQ2] = 0;
    cnt[C_NWIN] = 0;
    cnt[C_SCR] = 0;
    cnt[C_NREW] = 0;
    cnt[C_TOTAL] = 0;
    cnt[C_NLONG] = 0;
    cnt[C_PATH] = 0;
    cnt[C_PATH + 1] = 0;
    cnt[C_NMID] = 0;
    cnt[C_NBIGW] = 0;
}

// ---------------------------------------------------------------- split by cells
//
// The split pass above walks each segment on one thread, vertex by vertex: a
// segment that runs through many collinear vertices (the lattice's diagonals:
// about 190 each) is a long chain of dependent loads on a single thread.  When
// the points are in Morton order of their 1024^2 cells (the single solve), the
// vertices on a segment are found instead by testing the points of every cell
// the segment touches, a wave per segment; they are then sorted along it in
// LDS, and each piece between two
// consecutive ones is checked for being an existing edge on a thread of its
// own.  The pieces are the same as the walk's: in order along the segment,
// existing edges marked constrained and stored with a negative first vertex.
// Segments with more than SEG_SORT_MAX vertices on them keep the walk.

constexpr int SEG_SORT_MAX = 1024;

// A segment is cut into strips one cell wide along the axis it extends furthest
// on: columns, or rows where |dy| > |dx| (a strip then meets at most a few
// cells; walked by columns, a steep segment's cells were one thread's work).
struct SegStrips {
    int u0, u1, v0, v1;  // major / minor coordinates of the ends, u0 <= u1
    bool rows;
    double m;            // dv / du, |m| <= 1
    __device__ SegStrips(int2 A, int2 B)
    {
        const int ax = A.x < B.x ? B.x - A.x : A.x - B.x, ay = A.y < B.y ? B.y - A.y : A.y - B.y;
        rows = ay > ax;
        u0 = rows ? A.y : A.x;
        v0 = rows ? A.x : A.y;
        u1 = rows ? B.y : B.x;
        v1 = rows ? B.x : B.y;
        if (u0 > u1) {
            int t = u0;
            u0 = u1;
            u1 = t;
            t = v0;
            v0 = v1;
            v1 = t;
        }
        m = u1 > u0 ? (double)(v1 - v0) / (double)(u1 - u0) : 0.0;
    }
    __device__ int first() const { return u0 >> 20; }
    __device__ int last() const { return u1 >> 20; }
    // Cells [lo, hi] of strip s that the closed segment can touch.  A superset
    // serves (each cell's points are tested exactly): the line is evaluated in
    // double, off by less than 2^-18 here, and widened by one unit.
    __device__ void cells(int s, int& lo, int& hi) const
    {
        const int a = max(u0, s << 20), b = min(u1, (s << 20) + ((1 << 20) - 1));
        const double va = v0 + (double)(a - u0) * m, vb = v0 + (double)(b - u0) * m;
        const int l = (int)(va < vb ? va : vb) - 2, h = (int)(va < vb ? vb : va) + 2;
        lo = max(l, min(v0, v1)) >> 20;
        hi = min(h, max(v0, v1)) >> 20;
    }
};

__device__ inline bool seg_valid(int2 e, int nmax) { return e.x >= 0 && e.y >= 0 && e.x < nmax && e.y < nmax && e.x != e.y; }

// Vertices strictly inside each segment, one wave per segment: its lanes share
// the strips, test the points of every cell and collect the vertices on
// the segment in LDS, where they are sorted along it.  They leave at hpos[i]
// of hits[] (room permitting: the cursor counts on and the caller repeats the
// launch with more), np[i] = pieces of the segment.  A segment with more than
// SEG_SORT_MAX vertices on it goes to the walk list (its count comes later).
// Bound by the latency of a strip's chain (cell ends, points); the passes of
// one thread per segment and strip that this replaces took 155 + 186 us for
// 12 segments over 300 points and 864 + 1,024 us for 1,000 rows over 100,000.
// A segment of up to 32 strips has several lanes to a strip, which stride over
// the points of its cells: a short segment lies in one or two cells, and with
// a lane to a strip 20,000 of them in one cell of 200,000 points took 222 ms
// (the two passes before 56; so 4.8), 20,000 of them in 100 cells 2.7 ms (1.2;
// so 0.4).  Constraint recovery of 100,000 segments among 1M points all over
// the square takes 0.6 ms either way.
__global__ __launch_bounds__(64) void k_seg_find(const int2* pts, const int* cell_end, const int2* cons, int C, int nmax,
                                                 int* np, int* hcnt, int* hpos, int* hits, int hcap, int* hcur,
                                                 int* walk_list, int* nwalk, int* err)
{
    __shared__ long long s_key[SEG_SORT_MAX];
    __shared__ int s_val[SEG_SORT_MAX];
    __shared__ int s_n, s_at;
    const int lane = threadIdx.x;
    for (int i = blockIdx.x; i < C; i += gridDim.x) {
        const int2 e = cons[i];
        if (!seg_valid(e, nmax)) {  // block-uniform
            if (lane == 0) {
                atomicOr(err, MERR_INVALID);
                np[i] = 0;
                hcnt[i] = 0;
            }
            continue;
        }
        if (lane == 0) s_n = 0;
        __syncthreads();
        const int2 A = pts[e.x], B = pts[e.y];
        const long long dx = (long long)B.x - A.x, dy = (long long)B.y - A.y;
        const SegStrips g(A, B);
        const int first = g.first(), last = g.last();
        int per = 1;  // lanes to a strip
        while (2 * per * (last - first + 1) <= 64) per <<= 1;
        const int sub = lane & (per - 1);
        for (int st = first + lane / per; st <= last; st += 64 / per) {
            int lo, hi;
            g.cells(st, lo, hi);
            for (int v = lo; v <= hi; v++) {
                const unsigned cell = g.rows ? cell_morton((unsigned)v, (unsigned)st) : cell_morton((unsigned)st, (unsigned)v);
                const int p1 = cell_end[cell];
                for (int p = (cell ? cell_end[cell - 1] : 0) + sub; p < p1; p += per) {
                    if (p == e.x || p == e.y) continue;
                    const int2 P = pts[p];
                    if (orient2d(A, B, P) != 0 || !strictly_between(A, B, P)) continue;
                    const int k = atomicAdd(&s_n, 1);
                    if (k < SEG_SORT_MAX) {
                        s_key[k] = ((long long)P.x - A.x) * dx + ((long long)P.y - A.y) * dy;
                        s_val[k] = p;
                    }
                }
            }
        }
        __syncthreads();
        const int h = s_n;
        if (h > 1 && h <= SEG_SORT_MAX) {
            int m = 2;
            while (m < h) m <<= 1;
            for (int k = h + lane; k < m; k += 64) {
                s_key[k] = LLONG_MAX;
                s_val[k] = -1;
            }
            __syncthreads();
            for (int size = 2; size <= m; size <<= 1) {
                for (int stride = size >> 1; stride > 0; stride >>= 1) {
                    for (int k = lane; k < (m >> 1); k += 64) {
                        const int a = 2 * k - (k & (stride - 1)), b = a + stride;
                        const bool up = (a & size) == 0;
                        const long long ka = s_key[a], kb = s_key[b];
                        if ((ka > kb) == up) {
                            s_key[a] = kb;
                            s_key[b] = ka;
                            const int t = s_val[a];
                            s_val[a] = s_val[b];
                            s_val[b] = t;
                        }
                    }
                    __syncthreads();
                }
            }
        }
        if (lane == 0) {
            hcnt[i] = h;
            np[i] = h <= SEG_SORT_MAX ? h + 1 : 0;
            s_at = -1;
            if (h > SEG_SORT_MAX) {
                walk_list[atomicAdd(nwalk, 1)] = i;
            } else if (h > 0) {
                const int at = atomicAdd(hcur, h);
                hpos[i] = at;
                if (at >= 0 && h <= hcap - at) s_at = at;
            }
        }
        __syncthreads();
        if (s_at >= 0)
            for (int k = lane; k < h; k += 64) hits[s_at + k] = s_val[k];
        __syncthreads();
    }
}

__device__ inline int upper_bound_seg(const int* a, int n, long long x)
{
    int lo = 0, hi = n;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (a[mid] <= x) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// one thread per piece of the sorted segments: (previous vertex, next vertex)
// along the segment; an existing edge is marked constrained and stored with
// a negative first vertex, any other piece is queued for the rounds
__global__ __launch_bounds__(kBlock) void k_seg_pieces(Cons c, const int2* cons, int C, const int* poff,
                                                       const int* hcnt, const int* hpos, const int* hits,
                                                       long long total, int2* pieces, int* queue, int* nq)
{
    const Mesh& m = c.m;
    WAVE_LOOP(j, total)
    {
        bool want = false;
        const int sg = j < total ? upper_bound_seg(poff, C + 1, j) - 1 : 0;
        const int h = j < total ? hcnt[sg] : 0;
        if (j < total && h <= SEG_SORT_MAX) {  // else the walk writes this segment's pieces
            const int k = (int)(j - poff[sg]);
            const int2 e = cons[sg];
            // the q-th vertex from e.x (hits are sorted from e.x towards e.y)
            auto vtx = [&](int q) { return q == 0 ? e.x : (q == h + 1 ? e.y : hits[hpos[sg] + q - 1]); };
            const int u = vtx(k), v = vtx(k + 1);
            int t, s;
            const int r = find_wedge(c, u, v, t, s);
            if (r < 0) at_or(c.err, MERR_WALK);
            if (r == 1 && get3(m.tri[t], nx3(s)) == v) {
                mark_pair(c, t, pv3(s));
                pieces[j] = make_int2(-(u + 1), v);
            } else {
                pieces[j] = make_int2(u, v);
                want = true;
            }
        }
        const int at = wave_alloc(want ? 1 : 0, nq);
        if (want) queue[at] = (int)j;
    }
}

// the walk's pieces for the listed (long) segments: counted into np, then
// written at their offsets
__global__ __launch_bounds__(kBlock) void k_seg_counts(const int2* cons, int C, int nmax, const int* hcnt, int* np)
{
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < C; i += (long long)gridDim.x * blockDim.x)
        np[i] = seg_valid(cons[i], nmax) && hcnt[i] <= SEG_SORT_MAX ? hcnt[i] + 1 : 0;
}

__global__ __launch_bounds__(kBlock) void k_seg_walk(Cons c, const int2* cons, const int* list, const int* nlist,
                                                     int* np, const int* poff, int2* pieces)
{
    int n = *nlist;
    for (long long w = (long long)blockIdx.x * blockDim.x + threadIdx.x; w < n; w += (long long)gridDim.x * blockDim.x) {
        int sg = list[w];
        int2 e = cons[sg];
        if (poff) split_walk(c, e.x, e.y, pieces + poff[sg]);
        else np[sg] = split_walk(c, e.x, e.y, nullptr);
    }
}

// Cells that the closed segments can touch, column by column (a superset): what
// the solve on a fixed array bounds its inputs by (split_limit).
__global__ __launch_bounds__(64) void k_seg_demand(const int2* pts, const int2* cons, int C, int nmax, int* total)
{
    for (int i = blockIdx.x; i < C; i += gridDim.x) {
        const int2 e = cons[i];
        if (!seg_valid(e, nmax)) continue;
        int2 A = pts[e.x], B = pts[e.y];
        if (A.x > B.x) {
            const int2 t = A;
            A = B;
            B = t;
        }
        const long long dx = (long long)B.x - A.x, dy = (long long)B.y - A.y;
        int k = 0;
        for (int cx = (A.x >> 20) + (int)threadIdx.x; cx <= B.x >> 20; cx += 64) {
            int lo = min(A.y, B.y) >> 20, hi = max(A.y, B.y) >> 20;
            if (dx > 0) {
                const long long xl = max((long long)A.x, (long long)cx << 20),
                                xr = min((long long)B.x, ((long long)(cx + 1) << 20) - 1);
                const long long nl = A.y * dx + (xl - A.x) * dy, nr = A.y * dx + (xr - A.x) * dy;
                // all within the square, so neither numerator is negative
                lo = (int)((min(nl, nr) / dx) >> 20);
                hi = (int)(((max(nl, nr) + dx - 1) / dx) >> 20);
                hi = min(hi, 1023);
            }
            k += hi - lo + 1;
        }
        wave_alloc(k, total);
    }
}

// Bytes that the solve on a fixed array counts for a split of C segments with
// nh vertices on them and `pairs` touched cells, whatever it takes: offsets,
// counts, positions and pieces by segment, two lists of segments, the
// vertices, and each touched cell with its segment.
static size_t split_limit(size_t C, size_t nh, size_t pairs)
{
    return 4 * Arena::size(4 * (C + 1)) + 2 * Arena::size(4 * C) + Arena::size(4 * std::max<size_t>(nh, 1)) +
           2 * Arena::size(4 * std::max<size_t>(pairs, 1));
}

// Pieces of the segments, from the points' cells; *queued: those that need a
// cavity are in queue already (C_NQ, C_NREW and C_NQ2 were cleared by the
// caller).  pad: the rest of split_limit, held while the constraints are
// inserted.
static int split_pieces_cells(Ctx& cx, const Cons& c, const int* cell_end, const int2* cons, int C, int nmax,
                              DBuf<int2>& pieces, DBuf<int>& queue, bool* queued, DBuf<int>& pad)
{
    const int2* pts = c.m.pts;
    int* cnt = cx.dcnt.p;
    const size_t top0 = g_arena ? g_arena->top : 0;
    if (g_arena) {
        cx.set(C_STUCK, 0);
        k_seg_demand<<<std::min(C, 16384), 64, 0, cx.st>>>(pts, cons, C, nmax, cnt + C_STUCK);
        GCDT_LAUNCH_CHECK();
    }
    DBuf<int> np((size_t)C + 1), hcnt(C), hpos(C), wlist(C), hits((size_t)2 * C + 1024);
    for (int tries = 0;; tries++) {
        const int hcap = (int)std::min<size_t>(hits.n, INT_MAX);
        k_seg_find<<<std::min(C, 16384), 64, 0, cx.st>>>(pts, cell_end, cons, C, nmax, np.p, hcnt.p, hpos.p, hits.p, hcap,
                                                         cnt + C_NREW, wlist.p, cnt + C_NQ2, c.err);
        GCDT_LAUNCH_CHECK();
        scan_excl_total(cx, np.p, np.p, C);
        cx.read(0, C_NUM);
        if (cx.hcnt[C_ERR]) cx.check_err();
        const long long nh = cx.hcnt[C_NREW];
        if (nh < 0) throw Error(GCDT_ERR_SCRATCH, "too many vertices on the constraints");
        if (nh <= (long long)hits.n) break;
        if (tries) throw Error(GCDT_ERR_INTERNAL, "constraint split changed between two passes");
        hits.ensure((size_t)nh);
        cx.set(C_NREW, 0);
        cx.set(C_NQ2, 0);
    }
    int total = cx.hcnt[C_TOTAL];
    const int nwalk = cx.hcnt[C_NQ2];
    DBuf<int> cnts;
    if (nwalk > 0) cnts.alloc((size_t)C + 1);
    if (g_arena) hold_to(pad, top0 + split_limit(C, cx.hcnt[C_NREW], cx.hcnt[C_STUCK]));
    if (nwalk > 0) {
        // segments with many vertices keep the walk: their counts, and the
        // offsets again (from the counts of the others)
        k_seg_counts<<<grid_for(C), kBlock, 0, cx.st>>>(cons, C, nmax, hcnt.p, cnts.p);
        GCDT_LAUNCH_CHECK();
        k_seg_walk<<<grid_for(nwalk), kBlock, 0, cx.st>>>(c, cons, wlist.p, cnt + C_NQ2, cnts.p, nullptr, nullptr);
        GCDT_LAUNCH_CHECK();
        scan_excl_total(cx, cnts.p, np.p, C);
        cx.read(0, C_NUM);
        if (cx.hcnt[C_ERR]) cx.check_err();
        total = cx.hcnt[C_TOTAL];
    }
    pieces.alloc(total > 0 ? total : 1);
    queue.alloc(total > 0 ? total : 1);
    if (total > 0) {
        k_seg_pieces<<<grid_for(total), kBlock, 0, cx.st>>>(c, cons, C, np.p, hcnt.p, hpos.p, hits.p, total, pieces.p,
                                                            queue.p, cnt + C_NQ);
        GCDT_LAUNCH_CHECK();
    }
    *queued = nwalk == 0;
    if (nwalk > 0) {
        k_seg_walk<<<grid_for(nwalk), kBlock, 0, cx.st>>>(c, cons, wlist.p, cnt + C_NQ2, nullptr, np.p, pieces.p);
        GCDT_LAUNCH_CHECK();
        cx.check_err();
    }
    return total;
}

// Split pass: pieces of every constraint (existing edges marked constrained
// and stored with a negative first vertex).  Returns the piece count.
static int split_pieces(Ctx& cx, const Cons& c, const int2* cons, int C, int nmax, DBuf<int2>& pieces)
{
    DBuf<int> cnt((size_t)C + 1);
    k_split_count<<<grid_for(C), kBlock, 0, cx.st>>>(c, cons, C, nmax, cnt.p);
    GCDT_LAUNCH_CHECK();
    scan_excl_total(cx, cnt.p, cnt.p, C);
    cx.read(0, C_NUM);
    if (cx.hcnt[C_ERR]) cx.check_err();
    int np = cx.hcnt[C_TOTAL];
    pieces.alloc(np > 0 ? np : 1);
    k_split_emit<<<grid_for(C), kBlock, 0, cx.st>>>(c, cons, C, cnt.p, pieces.p);
    GCDT_LAUNCH_CHECK();
    cx.check_err();
    return np;
}

long long mark_constraint_chains(Ctx& cx, const Mesh& m, int T, int nv, int nmax, const int2* cons, int C)
{
    if (C <= 0) return 0;
    DBuf<int> vt(nv);
    fill_i32(cx, vt.p, -1, nv);
    k_build_vt<<<grid_for(T), kBlock, 0, cx.st>>>(m.tri, T, vt.p);
    GCDT_LAUNCH_CHECK();
    Cons c;
    c.m = m;
    c.vt = vt.p;
    c.owner = nullptr;
    c.stamp = nullptr;
    c.cavof = nullptr;
    c.err = cx.dcnt.p + C_ERR;
    DBuf<int2> pieces;
    return split_pieces(cx, c, cons, C, nmax, pieces);
}

ConsResult insert_constraints(Ctx& cx, const Mesh& m, int T, int nv, int nmax, const int2* cons, int C,
                              int* touched, int* tlist, const int* cell_end, ConsDefer* defer)
{
    ConsResult res;
    if (C <= 0) return res;
    DBuf<int> vt(nv);
    DBuf<unsigned long long> owner(T);
    DBuf<int> stamp(T), cavof(T);
    FillJobs f;
    f.add(vt.p, -1, nv);
    f.add(owner.p, -1, 2LL * T);
    f.add(stamp.p, 0, T);
    f.add(m.cflag, 0, T);
    f.add(touched, 0, T);
    f.add(cx.dcnt.p + C_NPIECE, 0, C_NWIN - C_NPIECE + 1);
    fill_jobs(cx, f);
    k_build_vt<<<grid_for(T), kBlock, 0, cx.st>>>(m.tri, T, vt.p);
    GCDT_LAUNCH_CHECK();
    Cons c;
    c.m = m;
    c.vt = vt.p;
    c.owner = owner.p;
    c.stamp = stamp.p;
    c.cavof = cavof.p;
    c.err = cx.dcnt.p + C_ERR;
    c.steiner = defer != nullptr;
    // 1. split into pieces
    DBuf<int2> pieces;
    DBuf<int> qa;
    bool queued = false;
    DBuf<int> pad;
    int np = cell_end ? split_pieces_cells(cx, c, cell_end, cons, C, nmax, pieces, qa, &queued, pad)
                      : split_pieces(cx, c, cons, C, nmax, pieces);
    res.pieces = np;
    DBuf<int> dflag;
    if (defer) {
        dflag.alloc(np > 0 ? np : 1);
        fill_i32(cx, dflag.p, 0, np);
        c.defer = dflag.p;
    }
    // 2. rounds over pieces that need a cavity
    DBuf<int> qb(np > 0 ? np : 1), ncross(np > 0 ? np : 1);
    DBuf<Win> wins(np > 0 ? np : 1);
    if (!queued) {
        qa.ensure(np > 0 ? np : 1);
        cx.set(C_NQ, 0);
        k_piece_queue<<<grid_for(np), kBlock, 0, cx.st>>>(pieces.p, np, qa.p, cx.dcnt.p + C_NQ);
        GCDT_LAUNCH_CHECK();
    }
    int nq = np;  // at most; the first round's counters tell
    int* Q = qa.p;
    int* Q2 = qb.p;
    DBuf<int> scr, rew;
    DBuf<int> longq, longw, ppos, paths, round_pad;
    const size_t round_top = g_arena ? g_arena->top : 0;
    int r = 0;
    int* cnt = cx.dcnt.p;
    while (nq > 0) {
        if (++r > 100000) throw Error(GCDT_ERR_NOT_CONVERGED, "constraint rounds did not converge");
        unsigned ep = cx.next_epoch();
        longq.ensure(nq);
        longw.ensure(nq);
        ppos.ensure(nq);
        paths.ensure((size_t)4 * nq + (size_t)64 * std::min(nq, 2048));
        const int g = grid_for(nq);
        long long npath = 0;
        for (int tries = 0;; tries++) {
            const int pcap = (int)std::min<size_t>(paths.n, INT_MAX);
            unsigned long long* pcur = (unsigned long long*)(cnt + C_PATH);
            k_cav_begin<<<1, 1, 0, cx.st>>>(cnt, r > 1 && tries == 0);
            GCDT_LAUNCH_CHECK();
            k_cav_claim<<<g, kBlock, 0, cx.st>>>(c, pieces.p, Q, cnt + C_NQ, ep, ncross.p, paths.p, pcap, pcur, ppos.p,
                                                 longq.p, cnt + C_NLONG);
            GCDT_LAUNCH_CHECK();
            k_cav_walk_long<<<std::min(nq, 2048), 64, 0, cx.st>>>(c, pieces.p, Q, longq.p, cnt + C_NLONG, cell_end, ep,
                                                                  ncross.p, cnt + C_TOTAL, paths.p, pcap, pcur, ppos.p);
            GCDT_LAUNCH_CHECK();
            cx.read(0, C_NUM);
            if (cx.hcnt[C_ERR]) cx.check_err();
            if (r > 1 && cx.hcnt[C_STUCK]) throw Error(GCDT_ERR_INTERNAL, "constraint round without progress");
            nq = cx.hcnt[C_NQ];
            npath = ((long long)cx.hcnt[C_PATH + 1] << 32) | (unsigned)cx.hcnt[C_PATH];
            if (npath > INT_MAX) throw Error(GCDT_ERR_SCRATCH, "constraints cross too many triangles");
            if (npath <= (long long)paths.n) break;
            // the paths did not fit: a larger buffer, and the walks again (their
            // claims are the same)
            if (tries) throw Error(GCDT_ERR_INTERNAL, "constraint paths changed between two walks");
            paths.ensure((size_t)npath);
        }
        if (nq == 0) {  // every piece was an edge already, or the round before inserted the last
            res.rewritten = cx.hcnt[C_NPIECE];
            r--;
            break;
        }
        const int nlong = cx.hcnt[C_NLONG];
        // scratch of every queued piece: cav_block_ints(K) (9 K + 16) for the
        // long ones, which C_TOTAL counts, K for the others
        const long long npl = cx.hcnt[C_TOTAL];
        long long cap = (npath - npl) + 9 * npl + 16LL * nlong + 1024;
        if (cap > (1LL << 30)) cap = 1LL << 30;
        rew.ensure((size_t)npl + 1);
        scr.ensure((size_t)cap);
        // a fixed array counts 13 words per crossed triangle and 20 per piece here,
        // and a word per triangle for the list of them, whatever the round takes
        if (r == 1 && g_arena)
            hold_to(round_pad, round_top + Arena::size(sizeof(int) * (size_t)std::min(13 * npath + 20LL * nq + 1024, 1LL << 30)) +
                                   Arena::size(sizeof(int) * (size_t)(npath + 1)));
        k_cav_check<<<g, kBlock, 0, cx.st>>>(c, Q, cnt + C_NQ, ncross.p, paths.p, ppos.p, ep, Q2, cnt + C_NQ2, wins.p,
                                             cnt + C_NWIN, scr.p, cnt + C_SCR, (long long)scr.n);
        GCDT_LAUNCH_CHECK();
        // Few long pieces, or very long ones: the larger workgroup for all of them, in
        // one launch (two in turn last as long as their longest cavities
        // together).  Many of up to CAV_MID_K triangles on average: a wave each for
        // those below it, as the larger workgroup's LDS admits two to a CU.  Solves
        // with c segments that cross k triangles each, one workgroup size / both:
        //   n 100,000  c 1,000  k 350        4.36 / 5.27 ms
        //   n 100,000  c 4,000  k 300        7.72 / 9.24
        //   n 1M       c 4,000  k 1,000     13.03 / 14.20
        //   n 1M       c 8,000  k 200        7.10 / 7.87
        //   n 1M       c 2,000  k 80         3.74 / 3.70
        //   n 1M       c 8,000  k 80         5.44 / 5.12
        //   n 4M       c 32,000  k 80       14.25 / 12.52
        const bool many = nlong > CAV_FEW && npl <= (long long)CAV_MID_K * nlong;
        const int mid_k = many ? CAV_MID_K : CAV_WAVE_K;
        if (nlong > 0) {
            k_cav_check_long<<<grid_for(64LL * nlong), kBlock, 0, cx.st>>>(
                c, Q, longq.p, cnt + C_NLONG, ncross.p, paths.p, ppos.p, ep, Q2, cnt + C_NQ2, wins.p, cnt + C_NWIN,
                scr.p, cnt + C_SCR, (long long)scr.n, longw.p, cnt + C_NMID, cnt + C_NBIGW, mid_k);
            GCDT_LAUNCH_CHECK();
        }
        if (nlong < nq) {
            k_cav_retri<<<std::min((nq + RETRI_BS - 1) / RETRI_BS, 16384), RETRI_BS, 0, cx.st>>>(c, pieces.p, wins.p,
                                                                                           cnt + C_NWIN, ep);
            GCDT_LAUNCH_CHECK();
        }
        if (nlong > 0 && many) {
            k_cav_retri_block<64, CAV_MID_K, false><<<std::min(nlong, 8192), 64, 0, cx.st>>>(
                c, pieces.p, wins.p, longw.p, cnt + C_NMID, cnt + C_NLONG, scr.p, ep, rew.p, cnt + C_NREW);
            GCDT_LAUNCH_CHECK();
        }
        if (nlong > 0) {
            k_cav_retri_block<256, CAV_LDS_K, true><<<std::min(nlong, 1024), 256, 0, cx.st>>>(
                c, pieces.p, wins.p, longw.p, cnt + C_NBIGW, cnt + C_NLONG, scr.p, ep, rew.p, cnt + C_NREW);
            GCDT_LAUNCH_CHECK();
        }
        k_cav_fix<<<grid_for(std::max<long long>((long long)FIX_LANES * (nq - nlong), npl)), kBlock, 0, cx.st>>>(
            c, wins.p, cnt + C_NWIN, scr.p, rew.p, cnt + C_NREW, ep, touched, tlist, cnt + C_NPIECE, tlist ? T : 0);
        GCDT_LAUNCH_CHECK();
        std::swap(Q, Q2);
        // After the first round, which is often the only one, the host looks
        // whether it was the last; a later one is followed by the next round's
        // claims at once, whose counters tell (a wait is 10 us, and the claims of
        // an empty queue as much).
        if (r == 1) {
            cx.read(0, C_NUM);
            if (cx.hcnt[C_ERR]) cx.check_err();
            nq = cx.hcnt[C_NQ2];
            if (nq > 0 && cx.hcnt[C_NWIN] == 0) throw Error(GCDT_ERR_INTERNAL, "constraint round without progress");
            res.rewritten = cx.hcnt[C_NPIECE];
        }
    }
    res.rounds = r;
    if (defer) {
        defer->pieces = std::move(pieces);
        defer->flag = std::move(dflag);
        defer->np = np;
    }
    return res;
}

}  // namespace gcdt
