// pm_trace.hip -- kd-restart, short-stack and brute-force traversal for
// gfx950 (wave64).  One lane per ray; the short stack lives in LDS,
// interleaved by lane so a wave's 64 accesses hit 64 different banks.
//
// Semantics (first hit of each ray):
//   kd-restart   Raytracer.cu:57-106 (TraceNode), :165-262 (KDRestart)
//   short-stack  ShortStack.cu:58-94 (TraceNode), :96-194, ShortStack.h:43-98
//   brute force  BruteTracer.cu:54-96 (Exhaustive)
//
// The tracers read a trace view built once per tree (build_trace_view):
//   packed[node]   int4 {split bits | prim index, left | bitmap lo,
//                        right | bitmap hi, axis}: one 16-byte load per visit;
//                        a child that is a leaf has its sign bit set
//   leaf_rec[2n]   a leaf's box, first slot and low bitmap word: one 32-byte
//                  load, issued as soon as its parent names it
//   leaf_tris[3k]  float4 v0 (w = triangle id bits), e1 = v1 - v0,
//                  e2 = v2 - v0 for leaf slot k: a leaf's triangles are
//                  contiguous and need no prim-index indirection.
// e1/e2 are the same IEEE subtractions Moller-Trumbore performs, so hits are
// bit-identical to testing the original vertices.
#include <algorithm>
#include <climits>

#include "pm_device.h"
#include "pm_internal.h"


namespace pmkd {

namespace {

constexpr int TB = 256;   // threads per block (4 waves)

__device__ __forceinline__ pm_hit miss_record() {
    pm_hit h;
    h.id = -1; h.t = __int_as_float(0x7f800000); h.u = 0.0f; h.v = 0.0f;
    return h;
}

// Moller-Trumbore (IRayTracer.h:111-145) from precomputed edges.  The same
// values (t = inv (q.e2), u = inv (p.T), v = inv (q.d), inv = 1/det) and the
// same acceptance (0 <= t <= th, u >= 0, v >= 0, u + v <= 1), tested in the
// order that rejects soonest: u first (u <= 1 is implied by v >= 0 and
// u + v <= 1, since rounding is monotonic), then v, then t.  Rays of a wave
// that test the same triangle mostly agree, so the wave skips the rest.
__device__ __forceinline__ bool mt_edges(f3 v0, f3 e1, f3 e2, f3 o, f3 d, float &th, float &tu,
                                         float &tv) {
    const f3 p = cross3(d, e2);
    const f3 t = sub3(o, v0);
    const float inv = rcp_rn(dot3(p, e1));
    const float hy = inv * dot3(p, t);
    if (!(hy >= 0.0f && hy <= 1.0f)) return false;
    const f3 q = cross3(t, e1);
    const float hz = inv * dot3(q, d);
    if (!(hz >= 0.0f && hy + hz <= 1.0f)) return false;
    const float hx = inv * dot3(q, e2);
    if (!(0.0f <= hx && hx <= th)) return false;
    th = hx; tu = hy; tv = hz;
    return true;
}

// A child or root as the tracers carry it: the node index, with the sign bit
// set for a leaf, so that a descent knows a leaf before it loads anything of
// it and then loads the whole leaf record (box, first slot, bitmap) at once.
// A round of the tracers is a chain of dependent loads (about 0.2 us each);
// without the bit it loaded the leaf's node record to see that it is one, then
// the box from two more arrays: three cache lines and one more wait per leaf.
// With it, 16.8M rays over a 256-mesh forest 7.8 -> 5.7 ms, four photon passes
// of 12M rays 6.66 -> 6.1 ms, 2M camera rays over a terrain 2.65 -> 2.25 ms.
constexpr int LEAF_CODE = INT_MIN;

__device__ __forceinline__ int root_code(const TreeDev &T, int root) {
    return T.packed[(unsigned)root].w == LEAF ? root | LEAF_CODE : root;
}

struct LeafRec {
    f3 bmin, bmax;
    int first;                  // the leaf's first slot
    unsigned long long bitmap;
};

__device__ __forceinline__ LeafRec load_leaf(const TreeDev &T, int code) {
    const unsigned node = (unsigned)code & 0x7fffffffu;
    const float4 a = T.leaf_rec[2ull * node], b = T.leaf_rec[2ull * node + 1];
    LeafRec r;
    r.bmin = mk3(a); r.bmax = mk3(b);
    r.first = __float_as_int(a.w);
    r.bitmap = (unsigned)__float_as_int(b.w);
    if (T.wide) r.bitmap |= (unsigned long long)(unsigned)T.packed[node].z << 32;
    return r;
}

// Leaf test (Raytracer.cu:194-216): optional box test, then Moller-Trumbore
// over the leaf bitmap in ascending bit order; the next triangle's data is
// loaded before the current one is tested.
template <bool SKIP, bool COUNT, bool WOOP>
__device__ __forceinline__ int test_leaf(const TreeDev &T, int code, f3 o, f3 d,
                                         f3 inv, float &th, float &tu, float &tv, int4 &cnt) {
    if (COUNT) cnt.y++;
    const LeafRec lf = load_leaf(T, code);
    if (SKIP) {
        if (COUNT) cnt.w++;
        if (!ray_box(o, inv, lf.bmin, lf.bmax)) return -1;
    }
    unsigned long long bm = lf.bitmap;
    if (!bm) return -1;
    if (WOOP) {   // the slot's Woop matrices; the id comes from the prim indices
        const float4 *W = T.leaf_woop + 3ll * lf.first;
        int slot = -1;
        for (; bm; bm &= bm - 1) {
            const int i = __builtin_ctzll(bm);
            if (COUNT) cnt.z++;
            if (woop_test(W[3 * i], W[3 * i + 1], W[3 * i + 2], o, d, th, tu, tv)) slot = i;
        }
        return slot < 0 ? -1 : T.prim_indices[lf.first + slot];
    }
    // two register sets, A and B, alternate: the next triangle loads while
    // the current one is tested.  The loads are unconditional (past the last
    // triangle they re-read the first one) so that a test waits for its own
    // loads only.
    const float4 *L = T.leaf_tris + 3ll * lf.first;
    const int first = __builtin_ctzll(bm);
    bm &= bm - 1;
    float4 a0 = L[3 * first], a1 = L[3 * first + 1], a2 = L[3 * first + 2];
    int hit = -1;
    for (;;) {
        const bool more_b = bm != 0;
        const int j = more_b ? __builtin_ctzll(bm) : first;
        bm &= bm - 1;
        const float4 b0 = L[3 * j], b1 = L[3 * j + 1], b2 = L[3 * j + 2];
        __builtin_amdgcn_sched_barrier(0);         // issue the loads before the test
        if (COUNT) cnt.z++;
        if (mt_edges(mk3(a0), mk3(a1), mk3(a2), o, d, th, tu, tv)) hit = __float_as_int(a0.w);
        if (!more_b) break;
        const bool more_a = bm != 0;
        const int k = more_a ? __builtin_ctzll(bm) : first;
        bm &= bm - 1;
        a0 = L[3 * k]; a1 = L[3 * k + 1]; a2 = L[3 * k + 2];
        __builtin_amdgcn_sched_barrier(0);
        if (COUNT) cnt.z++;
        if (mt_edges(mk3(b0), mk3(b1), mk3(b2), o, d, th, tu, tv)) hit = __float_as_int(b0.w);
        if (!more_a) break;
    }
    return hit;
}

// Traversal state of one ray between passes of the outer loop.
struct RayState {
    f3 o, d, inv;
    float th, tu, tv;
    int root_id;
    int nxt, count;            // short stack: ring position (slot * TB) and fill
    int visits;
};

__device__ __forceinline__ RayState ray_start(const TreeDev &T, int root_id, f3 o, f3 d) {
    RayState R;
    R.o = o;
    R.d = d;
    R.inv = {1.0f / d.x, 1.0f / d.y, 1.0f / d.z};
    R.th = 0.0f; R.tu = 0.0f; R.tv = 0.0f;
    R.root_id = root_id;
    R.nxt = 0; R.count = 0;
    R.visits = 0;
    return R;
}

__device__ __forceinline__ pm_hit ray_record(const RayState &R, int hit) {
    if (hit == -1) return miss_record();
    pm_hit h;
    h.id = hit; h.t = R.th; h.u = R.tu; h.v = R.tv;
    return h;
}

// One pass of the tracers' outer loop: start at the root (kd-restart, or
// short stack with an empty stack) or at the popped far child, descend to
// the leaf the ray is in at t = th, move th to the leaf's exit, test the
// leaf.
//   kd-restart   Raytracer.cu:57-106 (TraceNode), :165-262 (KDRestart)
//   short stack  ShortStack.cu:58-194, ShortStack.h:43-98: a ring of the S
//                most recent far children in LDS (interleaved by lane),
//                restart from the root when it runs empty
// descend() is the inner-node half: it returns false when the ray is done
// (a miss) before it reaches a leaf; else node/nd are the leaf and R.th its
// exit.  trace_step() is the whole pass: it returns true when the ray is
// done, `hit` being its triangle or -1.
// The ring lives in one LDS array int[2 * SMAX][TB]: rows 0..SMAX-1 hold the
// far nodes, rows SMAX.. their tNext bits; `stk` points at this lane's column
// and R.nxt counts in rows of TB, so a slot's two words are one register
// offset apart by a constant.
// The descent is split in two so that the cooperative kernel can spread it
// over several loop iterations: pass_start picks the pass's first node (the
// root or the popped far child; false: the visit bound is spent, a miss),
// descend_steps walks at most `cap` inner nodes from `node` (1: a leaf, nd
// its record and R.th its exit; 0: still inner, node/tNext/steps carry on;
// -1: the descent bound is spent, a miss).
// RESUME: kd-restart with a ring of its own.  A restart's descent at the new th
// makes the decisions of the last one down to the deepest node X whose far
// child was pushed, as long as th is below every plane above X that sent the
// ray to its lower side, that is below the tNext saved with the entry; there it
// turns to X's far child with that tNext, since th is X's plane or past it.  So
// the pass goes on from the entry, its steps as if counted from the root (the
// descent bound), and where th has passed the saved tNext too, from the root.
// The passes, their leaves and limits are those of restarting every time, with a
// third to a fifth of the inner nodes: 2,073,600 camera rays over a 2,093,058-
// triangle terrain 3.93 -> 3.10 ms (step cap 4: 6.45 -> 2.55), 65,536 in a 5,316-
// triangle room 194 -> 139 us (400 -> 149), 300,007 probes in a 50,001-triangle
// soup, whose time is in its leaves, 378 -> 372 us (600 -> 364).
enum StackMode { RESTART = 0, SHORT_RING = 1, RESUME = 2 };

// a lane's ring: node rows, then tNext rows, then (RESUME) 16-bit step rows
template <int SMAX, int MODE>
__device__ __forceinline__ unsigned short *ring_steps(int *stk) {
    return reinterpret_cast<unsigned short *>(stk - threadIdx.x + 2 * SMAX * TB) + threadIdx.x;
}
template <int SMAX, int MODE>
constexpr int ring_rows() { return MODE == RESTART ? 2 : MODE == RESUME ? 2 * SMAX + SMAX / 2 : 2 * SMAX; }

template <int SMAX, int MODE>
__device__ __forceinline__ bool pass_start(const TreeDev &T, RayState &R, int S, int *stk, int &node,
                                           float &tNext, int &steps) {
    if (R.visits++ > T.num_nodes) return false;
    steps = 0;
    if (MODE == RESTART || R.count == 0) {
        node = R.root_id; tNext = F_INF;
    } else {                                     // Pop, ShortStack.h:68-72
        R.nxt = (R.nxt == 0 ? S * TB : R.nxt) - TB;
        R.count--;
        node = stk[R.nxt];
        tNext = __int_as_float(stk[R.nxt + SMAX * TB]);
        if (MODE == RESUME) {
            steps = ring_steps<SMAX, MODE>(stk)[R.nxt];
            if (!(R.th < tNext)) {
                R.count = 0;
                steps = 0;
                node = R.root_id; tNext = F_INF;
            }
        }
    }
    return true;
}

template <int SMAX, int MODE, bool COUNT>
__device__ __forceinline__ int descend_steps(const TreeDev &T, RayState &R, int S, int *stk, int4 &cnt, int &node,
                                             float &tNext, int &steps, int cap) {
    for (int k = 0; node >= 0; ++k) {
        if (k == cap) return 0;
        if (++steps > MAX_DESCENT) return -1;
        if (COUNT) cnt.x++;
        const int4 nd = T.packed[(unsigned)node];   // child indices are in [0, num_nodes)
        const float s = __int_as_float(nd.x);
        const float ori = comp3(R.o, nd.w), dd = comp3(R.inv, nd.w);
        const float tSplit = (s - ori) * dd;
        const int lower = 0 < dd ? nd.y : nd.z;
        const int upper = 0 < dd ? nd.z : nd.y;
        if (R.th < tSplit) {
            node = lower;
            // here tSplit > th >= 0, and tNext (the sentinel or an earlier
            // tSplit) is never NaN: the select is exactly fminf(tSplit, tNext)
            const bool nearer = tSplit < tNext;
            if (MODE != RESTART && nearer) {         // Push, ShortStack.h:57-62
                stk[R.nxt] = upper;
                stk[R.nxt + SMAX * TB] = __float_as_int(tNext);
                if (MODE == RESUME) ring_steps<SMAX, MODE>(stk)[R.nxt] = (unsigned short)steps;
                R.nxt = R.nxt == (S - 1) * TB ? 0 : R.nxt + TB;
                R.count = min(R.count + 1, S);       // count <= S: count == S ? S : count + 1
            }
            tNext = nearer ? tSplit : tNext;
        } else {
            node = upper;
        }
    }
    R.th = tNext * 1.00001f;
    return 1;
}

template <int SMAX, int MODE, bool COUNT>
__device__ __forceinline__ bool descend(const TreeDev &T, RayState &R, int S, int *stk, int4 &cnt, int &node) {
    float tNext;
    int steps;
    if (!pass_start<SMAX, MODE>(T, R, S, stk, node, tNext, steps)) return false;
    return descend_steps<SMAX, MODE, COUNT>(T, R, S, stk, cnt, node, tNext, steps, INT_MAX) > 0;
}

template <int SMAX, bool SHORT, bool SKIP, bool COUNT, bool WOOP>
__device__ __forceinline__ bool trace_step(const TreeDev &T, RayState &R, int S, int *stk, int4 &cnt,
                                           int &hit) {
    hit = -1;
    int node;
    if (!descend<SMAX, SHORT ? SHORT_RING : RESTART, COUNT>(T, R, S, stk, cnt, node)) return true;
    hit = test_leaf<SKIP, COUNT, WOOP>(T, node, R.o, R.d, R.inv, R.th, R.tu, R.tv, cnt);
    return hit != -1 || !(R.th < F_INF);
}

// the whole traversal of one ray (the canvas shading's per-bounce trace)
template <bool SKIP, bool COUNT, bool WOOP>
__device__ __forceinline__ pm_hit kd_restart_ray(const TreeDev &T, int root_id, f3 o, f3 d, int4 &cnt) {
    RayState R = ray_start(T, root_id, o, d);
    int hit;
    while (!trace_step<1, false, SKIP, COUNT, WOOP>(T, R, 1, nullptr, cnt, hit)) {
    }
    return ray_record(R, hit);
}

template <int SMAX, bool SKIP, bool COUNT, bool WOOP>
__device__ __forceinline__ pm_hit short_stack_ray(const TreeDev &T, int root_id, f3 o, f3 d, int S,
                                                  int *stk, int4 &cnt) {
    RayState R = ray_start(T, root_id, o, d);
    int hit;
    while (!trace_step<SMAX, true, SKIP, COUNT, WOOP>(T, R, S, stk, cnt, hit)) {
    }
    return ray_record(R, hit);
}

// The first-hit kernels (kd-restart and short stack): persistent waves.
// A wave takes CHUNK consecutive rays at a time from a global counter
// (*work, zero at launch); once REFILL_MIN of its lanes are done, they take
// the next rays of the wave's chunk, so the wave's lanes stay busy while its
// longest rays finish.  Lane state: the ray's index q and its traversal
// state; one loop iteration = one pass of trace_step for every busy lane.
// The rays are handed out in the order `order` lists them (input order
// without one); ray q reads org[q], dir[q], ray_root[q] and writes out[q].
// Every wave leaves the loop once the counter has
// passed n and its lanes are idle; every ray ends (trace_step's visit and
// descent bounds), so every wave does.
constexpr int CHUNK = 64;        // rays a wave takes from the counter at a time
constexpr int REFILL_MIN = 16;   // idle lanes that make a wave take new rays

__device__ __forceinline__ bool ray_root_valid(const TreeDev &T, const int *ray_root, int r, int &root_id) {
    root_id = ray_root ? ray_root[r] : 0;
    // no such mesh, or (captured batch) the build before this trace failed: a miss
    if (root_id < 0 || root_id >= T.num_roots || (T.fail && *T.fail)) return false;
    root_id = root_code(T, root_id);
    return true;
}

template <int SMAX, bool SHORT, bool SKIP, bool COUNT, bool WOOP>
__global__ __launch_bounds__(TB) void trace_kernel(TreeDev T, const float4 *__restrict__ org,
                                                   const float4 *__restrict__ dir,
                                                   const int *__restrict__ ray_root,
                                                   const unsigned *__restrict__ order, int n, int S,
                                                   pm_hit *__restrict__ out, int4 *__restrict__ counters,
                                                   int *__restrict__ work) {
    __shared__ int stk_rows[2 * (SHORT ? SMAX : 1)][TB];   // short stack: node rows, then tNext rows
    int *const stk = &stk_rows[0][threadIdx.x];
    const int lane = threadIdx.x & 63;
    const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;
    int next = 0, end = 0;          // the wave's chunk (same in every lane)
    bool exhausted = false;
    int q = -1;                     // this lane's ray, -1 = idle
    RayState R;
    int4 cnt = make_int4(0, 0, 0, 0);
    for (;;) {
        const unsigned long long idle = __ballot(q < 0);
        // refill once a quarter of the lanes are idle: new rays start at
        // the root while the others are deep in the tree, so refilling
        // single lanes costs more than it gains
        if (__popcll(idle) >= REFILL_MIN && !exhausted) {
            if (next >= end) {
                int base = 0;
                if (lane == 0) base = atomicAdd(work, CHUNK);
                base = __builtin_amdgcn_readfirstlane(__shfl(base, 0, 64));
                if (base >= n || base < 0) {
                    exhausted = true;
                } else {
                    next = base;
                    end = n - base < CHUNK ? n : base + CHUNK;
                }
            }
            if (!exhausted) {
                const int avail = end - next;
                const int rank = __popcll(idle & below);
                if (q < 0 && rank < avail) {
                    q = order ? (int)order[next + rank] : next + rank;
                    int root_id;
                    if ((unsigned)q >= (unsigned)n) {
                        q = -1;                  // not a ray index (never for a valid order)
                    } else if (ray_root_valid(T, ray_root, q, root_id)) {
                        R = ray_start(T, root_id, mk3(org[q]), adjust_dir(mk3(dir[q])));
                        cnt = make_int4(0, 0, 0, 0);
                    } else {
                        out[q] = miss_record();
                        if (COUNT) counters[q] = make_int4(0, 0, 0, 0);
                        q = -1;
                    }
                }
                const int took = __popcll(idle);
                next = __builtin_amdgcn_readfirstlane(next + (took < avail ? took : avail));
            }
        }
        const bool busy = q >= 0;
        if (__ballot(busy) == 0) {
            if (exhausted) break;
            continue;
        }
        if (busy) {
            int hit;
            if (trace_step<SMAX, SHORT, SKIP, COUNT, WOOP>(T, R, S, stk, cnt, hit)) {
                out[q] = ray_record(R, hit);
                if (COUNT) counters[q] = cnt;
                q = -1;
            }
        }
    }
}

// ---- cooperative leaf test (Moller-Trumbore, and Woop on the slots' matrices)
//
// After a wave's lanes have descended to their leaves, lane i holds a leaf
// with k_i triangles; tested lane by lane the wave would loop max k_i times
// with most lanes idle.  Instead the wave lists all (lane, triangle) pairs
// in LDS (COOP_WIN at a time) and every lane tests the next pair, with the
// owner's ray and leaf exit th (read from the owner, see CoopLds).  An
// owner's first hit is the pair with the smallest t, and among equal t the
// triangle latest in bitmap order -- exactly what the sequential leaf loop
// (accept 0 <= t <= th, then th = t) ends with -- so each accepted pair
// offers the key (t bits, ~slot) to its owner's 64-bit LDS minimum, and the
// owner recomputes its winning triangle itself for t, u, v and the id.
// The key's low word is ~(byte offset of the slot's record): slots of one
// leaf grow with the bit index, so it orders ties like the bitmap does; t >=
// 0 here (-0 keyed as +0).  Record offsets are 32-bit (48 bytes per slot):
// trees with 2^32 / 48 slots or more take the lane-per-ray kernel.
constexpr int COOP_WIN = 512;
static_assert(COOP_WIN % 64 == 0, "a wave reads pair[r + lane] for r < COOP_WIN, r a multiple of 64");

// The tester reads the owner's ray, leaf exit and first slot either from
// LDS records the owners write (RECS) or straight from the owner's registers
// (ds_bpermute, whole wave active).  The short-stack kernel takes the second:
// its LDS, not its registers, caps its occupancy, and the records' 2 KiB a
// wave is what brings a block under a sixth of the CU's LDS.
template <bool RECS>
struct CoopLds {
    alignas(8) unsigned short pair[COOP_WIN];   // bit << 8 | 4 * owner lane
    unsigned long long key[64];
    float4 org[RECS ? 64 : 1];           // owner's origin, w = its leaf's first record offset (bits)
    float4 dir[RECS ? 64 : 1];           // owner's direction, w = its leaf exit th
};

// inclusive prefix sum over the wave's 64 lanes (every lane active): DPP
// row shifts within each row of 16 lanes, then row broadcasts of lanes 15
// and 31 into the rows after them (disabled lanes add the old value, 0)
__device__ __forceinline__ int wave_incl_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15, rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31, rows 2 and 3
    return v;
}

// lane src4 / 4's value of x (every lane of the wave active)
__device__ __forceinline__ float lane_read(float x, int src4) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(src4, __float_as_int(x)));
}

// orders this lane's LDS accesses with the other lanes' of the wave (a
// wave's LDS instructions execute in order; this keeps the compiler from
// moving them across)
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One (lane, triangle) pair: the owner's ray against the slot whose record
// starts `off` bytes into the leaf triangles; an accepted hit offers its key
// to the owner.  mt_edges' values without its early exits (the lanes test
// different triangles, so a wave never skips a part) and the same
// acceptance, written as min(hx, hy, hz) >= 0, hx <= th, hy + hz <= 1 (fminf
// returns the other operand of a NaN; a NaN hx fails hx <= th, a NaN hy or
// hz fails hy + hz <= 1).
// WOOP: the slot's record is its matrix m0, m1, m2 and the test woop_test's
// (the lane-per-ray loop waited for each lane's own matrices, one triangle
// after another: 100,003 probe rays over a 20,011-triangle soup 505 -> 186 us).
template <bool WOOP>
__device__ __forceinline__ void coop_pair(const float4 *__restrict__ L, unsigned long long *key, unsigned off,
                                          f3 ro, f3 rd, float rth) {
    const float4 *R3 = reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(L) + off);
    const float4 a0 = R3[0], a1 = R3[1], a2 = R3[2];
    if constexpr (WOOP) {
        float t = rth, u, v;
        if (woop_test(a0, a1, a2, ro, rd, t, u, v))
            atomicMin(key, ((unsigned long long)__float_as_uint(t + 0.0f) << 32) | (unsigned)~off);
        return;
    }
    const f3 v0 = mk3(a0), e1 = mk3(a1), e2 = mk3(a2);
    const f3 p = cross3(rd, e2);
    const f3 t = sub3(ro, v0);
    const f3 q = cross3(t, e1);
    const float inv = rcp_rn(dot3(p, e1));
    const float hx = inv * dot3(q, e2);
    const float hy = inv * dot3(p, t);
    const float hz = inv * dot3(q, rd);
    if (fminf(fminf(hx, hy), hz) >= 0.0f && hx <= rth && hy + hz <= 1.0f)
        atomicMin(key, ((unsigned long long)__float_as_uint(hx + 0.0f) << 32) | (unsigned)~off);
}

// every lane of the wave calls it with the byte offset of its leaf's first
// record (3 float4 per slot; every offset fits 32 bits); returns the byte
// offset of the lane's winning record, or -1
template <bool RECS, bool WOOP>
__device__ __forceinline__ long long coop_leaf(const float4 *__restrict__ L, CoopLds<RECS> &C,
                                               unsigned long long bm, unsigned base48, f3 o, f3 d, float th) {
    const int lane = threadIdx.x & 63;
    C.key[lane] = ~0ull;
    if (RECS) {
        C.org[lane] = make_float4(o.x, o.y, o.z, __uint_as_float(base48));
        C.dir[lane] = make_float4(d.x, d.y, d.z, th);
    }
    // k <= 64 pairs per lane: the wave's prefix sum of k (this lane's first
    // pair) and its total (the wave's pairs)
    const int k = __popcll(bm);
    const int incl = wave_incl_scan(k);
    const int excl = incl - k;
    const int W = __builtin_amdgcn_readlane(incl, 63);
    int pos = excl;
    // a pair is bit << 8 | 4 * owner lane (the owner's ds_bpermute address);
    // a run of bits b0 .. b0+k-1 (every leaf the upper stage makes) is listed
    // four pairs to a 64-bit store; other bitmaps bit by bit
    const int lane4 = lane << 2;
    const int b0 = bm ? __builtin_ctzll(bm) : 0;
    const unsigned long long run = bm >> b0;
    const bool contig = (run & (run + 1)) == 0ull;
    unsigned lo = contig ? 0u : (unsigned)bm, hi = contig ? 0u : (unsigned)(bm >> 32);
    unsigned long long *pair4 = reinterpret_cast<unsigned long long *>(C.pair);
    for (int wbase = 0; wbase < W; wbase += COOP_WIN) {
        const int wn = W - wbase < COOP_WIN ? W - wbase : COOP_WIN;
        wave_sync();
        // list this lane's pairs of the window, bits in ascending order
        if (contig) {
            int i = wbase - excl > 0 ? wbase - excl : 0;
            const int iend = wbase + wn - excl < k ? wbase + wn - excl : k;
            int p = excl + i - wbase;
            while (i < iend && (p & 3)) {
                C.pair[p++] = (unsigned short)((b0 + i) << 8 | lane4);
                ++i;
            }
            unsigned long long v = (unsigned long long)((b0 + i) << 8 | lane4) * 0x0001000100010001ull +
                                   0x0300020001000000ull;
            while (i + 4 <= iend) {
                pair4[p >> 2] = v;
                v += 1024ull * 0x0001000100010001ull;
                p += 4;
                i += 4;
            }
            while (i < iend) {
                C.pair[p++] = (unsigned short)((b0 + i) << 8 | lane4);
                ++i;
            }
        }
        while (lo && pos < wbase + wn) {
            const int b = __builtin_ctz(lo);
            lo &= lo - 1;
            C.pair[pos++ - wbase] = (unsigned short)(b << 8 | lane4);
        }
        while (hi && pos < wbase + wn) {
            const int b = __builtin_ctz(hi) + 32;
            hi &= hi - 1;
            C.pair[pos++ - wbase] = (unsigned short)(b << 8 | lane4);
        }
        wave_sync();
        // the owner's ray, leaf exit and first record offset, for pair pr
        auto pair_at = [&](int e, f3 &ro, f3 &rd, float &rth, unsigned &off, int &ow4) {
            const int pr = C.pair[e];   // e < COOP_WIN: stale past wn, used only for an in-range lane
            ow4 = pr & 255;
            unsigned rbase;
            if (RECS) {
                const float4 a = C.org[ow4 >> 2], b = C.dir[ow4 >> 2];
                ro = mk3(a); rd = mk3(b); rth = b.w; rbase = __float_as_uint(a.w);
            } else {
                ro = {lane_read(o.x, ow4), lane_read(o.y, ow4), lane_read(o.z, ow4)};
                rd = {lane_read(d.x, ow4), lane_read(d.y, ow4), lane_read(d.z, ow4)};
                rth = lane_read(th, ow4);
                rbase = (unsigned)__builtin_amdgcn_ds_bpermute(ow4, (int)base48);
            }
            off = (unsigned)(pr >> 8) * 48u + rbase;
        };
        // full rounds of 64 pairs, then the window's tail
        const int full = wn & ~63;
        int r = 0;
        for (; r < full; r += 64) {
            f3 ro, rd;
            float rth;
            unsigned off;
            int ow4;
            pair_at(r + lane, ro, rd, rth, off, ow4);
            coop_pair<WOOP>(L, &C.key[ow4 >> 2], off, ro, rd, rth);
        }
        if (r < wn) {
            f3 ro, rd;
            float rth;
            unsigned off;
            int ow4;
            pair_at(r + lane, ro, rd, rth, off, ow4);
            if (r + lane < wn) coop_pair<WOOP>(L, &C.key[ow4 >> 2], off, ro, rd, rth);
        }
    }
    wave_sync();
    const unsigned long long best = C.key[lane];
    return best == ~0ull ? -1ll : (long long)(unsigned)~(unsigned)(best & 0xffffffffu);
}

// ---- canvas shading: ColorKernels.h:15-85 in the tracers' shading loops
// (Raytracer.cu:165-262, ShortStack.cu:96-194, BruteTracer.cu:54-96); the
// specular power is the correctly rounded float of the double power
struct Light { f3 pos, ambient, diffuse, specular; };

__device__ __forceinline__ f3 scale3(f3 a, float s) { return {a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ f3 add3(f3 a, f3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ f3 mul3(f3 a, f3 b) { return {a.x * b.x, a.y * b.y, a.z * b.z}; }
__device__ __forceinline__ float saturate(float x) { return x > 1.0f ? 1.0f : (x > 0.0f ? x : 0.0f); }
__device__ __forceinline__ float clamp01(float x) { return fmaxf(0.0f, fminf(x, 1.0f)); }

// PhongLighting, ColorKernels.h:15-45, shadow = 1 (the reference's shadow
// rays are disabled, Raytracer.cu:219-226)
__device__ __forceinline__ float4 phong(const float4 c, f3 normal, f3 point, f3 origin, const Light &L) {
    const f3 lightDir = normalize3(sub3(L.pos, point));
    const float diffuse = saturate(dot3(lightDir, normal) * 1.0f);
    f3 refl = sub3(scale3(normal, 2.0f * dot3(normal, lightDir)), lightDir);
    refl = normalize3(refl);
    const float stemp = saturate(dot3(normalize3(sub3(origin, point)), refl));
    const float specProp = 1.0f - c.w;
    const float specular = specProp * (float)pow((double)stemp, (double)(128.0f * specProp));
    const f3 base = {c.x, c.y, c.z};
    const f3 light = add3(mul3(base, add3(L.ambient, scale3(L.diffuse, diffuse))),
                          scale3(scale3(scale3(L.specular, specular), 10.0f), 1.0f));
    const float alpha = c.w < specular ? specular : c.w;
    return make_float4(clamp01(light.x), clamp01(light.y), clamp01(light.z), alpha);
}

// Lighting, ColorKernels.h:47-77: shade the hit, turn the ray into its
// mirror reflection from the hit point
__device__ __forceinline__ float4 lighting(const pm_hit &h, f3 &origin, f3 &dir, const float4 *__restrict__ n0,
                                           const float4 *__restrict__ n1, const float4 *__restrict__ n2,
                                           const uchar4 *__restrict__ c0, const Light &L) {
    const f3 point = add3(origin, scale3(dir, h.t));
    const float w = 1.0f - h.u - h.v;
    f3 normal = add3(add3(scale3(mk3(n0[h.id]), w), scale3(mk3(n1[h.id]), h.u)), scale3(mk3(n2[h.id]), h.v));
    normal = normalize3(normal);
    const uchar4 cc = c0[h.id];
    const float4 col = make_float4(cc.x / 255.0f, cc.y / 255.0f, cc.z / 255.0f, cc.w / 255.0f);
    dir = add3(scale3(normal, 2.0f * dot3(normal, scale3(dir, -1.0f))), dir);
    dir = normalize3(dir);
    const float4 out = phong(col, normal, point, origin, L);
    origin = add3(point, scale3(dir, 0.00001f));
    return out;
}

// BlendColor, ColorKernels.h:79-84
__device__ __forceinline__ float4 blend(const float4 o, float4 n) {
    const float a = n.w;
    n.w = 1.0f;
    const float k = (1.0f - o.w) * a;
    return make_float4(o.x + k * n.x, o.y + k * n.y, o.z + k * n.z, o.w + k * n.w);
}

// What the cooperative kernel needs to turn first hits into a canvas (CANVAS):
// a lane keeps its pixel over all bounces, so the mirror rays of some lanes are
// traced in the same rounds as the first rays of others.  Against the
// lane-per-ray loop (a lane's leaf triangles one after another, most lanes
// idle), 1280 x 720 in a 5,316-triangle room: 605 -> 359 us.  The launch has no
// ray counter: canvas calls on one context share no memory of it, and handing a
// block's rays out to its waves as lanes fall idle measured slower (542 us with
// runs of 450 rays, 370 with 256: neighbouring pixels are of like cost, and a
// refilled lane falls out of step with them).
struct CanvasArgs {
    const float4 *n0, *n1, *n2;
    const uchar4 *c0;
    Light light;
    int max_bounces;
    uchar4 *canvas;
};

__device__ __forceinline__ uchar4 canvas_pixel(const float4 col) {
    return make_uchar4((unsigned char)(col.x * 255.0f), (unsigned char)(col.y * 255.0f),
                       (unsigned char)(col.z * 255.0f), (unsigned char)(col.w * 255.0f));
}

// the persistent kernel of trace_kernel with the leaf test done by the wave.
// Lanes below `width` take rays (launch_coop's rule); a wave's first chunk is
// the one its index names, so that a launch's thousands of waves do not start
// by queueing on one counter (8,192 fetches of it take 0.13 ms), and later
// ones come from *work past those; work == nullptr: there are no later ones.
// CAPPED: a lane's descent walks at most `cap` inner nodes per iteration and
// goes on in the next (pm_trace_params.step_cap); the nodes visited, and so
// records and counters, are the same.
template <int SMAX, int MODE, bool SKIP, bool COUNT, bool CAPPED, bool WOOP, bool CANVAS = false>
__global__ __launch_bounds__(TB) void trace_coop_kernel(TreeDev T, const float4 *__restrict__ org,
                                                        const float4 *__restrict__ dir,
                                                        const int *__restrict__ ray_root,
                                                        const unsigned *__restrict__ order, int n, int S,
                                                        pm_hit *__restrict__ out,
                                                        int4 *__restrict__ counters, int *__restrict__ work,
                                                        int cap, int width, CanvasArgs V) {
    __shared__ int stk_rows[ring_rows<SMAX, MODE>()][TB];
    int *const stk = &stk_rows[0][threadIdx.x];
    __shared__ CoopLds<MODE == RESTART> coop[TB / 64];
    const int lane = threadIdx.x & 63;
    CoopLds<MODE == RESTART> &C = coop[threadIdx.x >> 6];
    const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;
    int next = 0, end = 0;          // the wave's chunk (same in every lane)
    bool exhausted = false;
    // lanes that take rays, and the idle ones that make the wave take more
    const bool taker = lane < width;
    const int refill = width < 4 * REFILL_MIN ? (width + 3) >> 2 : REFILL_MIN;
    const int first = (int)(gridDim.x * (TB / 64)) * width;   // rays the waves' first chunks take
    int q = -1;                     // this lane's ray, -1 = idle
    // a descent in progress (mid): its node, the far limit tNext, its steps
    bool mid = false;
    int cur = 0, steps = 0;
    float tnext = 0.0f;
    RayState R;
    R.o = {0.0f, 0.0f, 0.0f}; R.d = R.o; R.th = 0.0f;
    int4 cnt = make_int4(0, 0, 0, 0);
    float4 col = make_float4(0.0f, 0.0f, 0.0f, 0.0f);   // CANVAS: the ray's colour and bounces so far
    int bounce = 0;
    for (;;) {
        const unsigned long long idle = __ballot(taker && q < 0);
        if (__popcll(idle) >= refill && !exhausted) {
            if (next >= end) {
                int b = 0;
                if (end == 0) {                  // a wave's first chunk is its own
                    b = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * TB + threadIdx.x) >> 6) * width);
                } else if (work) {
                    if (lane == 0) b = atomicAdd(work, width);
                    b = first + __builtin_amdgcn_readfirstlane(b);
                } else {
                    b = n;
                }
                if (b >= n || b < 0) {
                    exhausted = true;
                } else {
                    next = b;
                    end = n - b < width ? n : b + width;
                }
            }
            if (!exhausted) {
                const int avail = end - next;
                const int rank = __popcll(idle & below);
                if (taker && q < 0 && rank < avail) {
                    q = order ? (int)order[next + rank] : next + rank;
                    int root_id;
                    if ((unsigned)q >= (unsigned)n) {
                        q = -1;                  // not a ray index (never for a valid order)
                    } else if (ray_root_valid(T, ray_root, q, root_id)) {
                        R = ray_start(T, root_id, mk3(org[q]), adjust_dir(mk3(dir[q])));
                        cnt = make_int4(0, 0, 0, 0);
                        if (CANVAS) {
                            col = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                            bounce = 0;
                        }
                    } else {
                        if (CANVAS) V.canvas[q] = make_uchar4(0, 0, 0, 0);
                        else out[q] = miss_record();
                        if (COUNT) counters[q] = make_int4(0, 0, 0, 0);
                        q = -1;
                    }
                }
                const int took = __popcll(idle);
                next = __builtin_amdgcn_readfirstlane(next + (took < avail ? took : avail));
            }
        }
        if (__ballot(q >= 0) == 0) {
            if (exhausted) break;
            continue;
        }
        // inner nodes, lane by lane (CAPPED: at most `cap` per iteration)
        bool done = false, at_leaf = false;
        unsigned long long bm = 0;
        int base = 0;
        if (q >= 0) {
            int r = 0;
            if (!CAPPED) {
                r = descend<SMAX, MODE, COUNT>(T, R, S, stk, cnt, cur) ? 1 : -1;
            } else {
                if (!mid) {
                    if (pass_start<SMAX, MODE>(T, R, S, stk, cur, tnext, steps)) mid = true;
                    else r = -1;
                }
                if (mid) r = descend_steps<SMAX, MODE, COUNT>(T, R, S, stk, cnt, cur, tnext, steps, cap);
                if (r != 0) mid = false;
            }
            if (r < 0) {
                done = true;
            } else if (r > 0) {
                const LeafRec lf = load_leaf(T, cur);
                at_leaf = true;
                if (COUNT) cnt.y++;
                bool enter = true;
                if (SKIP) {
                    if (COUNT) cnt.w++;
                    enter = ray_box(R.o, R.inv, lf.bmin, lf.bmax);
                }
                if (enter) {
                    bm = lf.bitmap;
                    base = lf.first;
                    if (COUNT) cnt.z += __popcll(bm);
                }
            }
        }
        // the leaves, by the whole wave
        const float4 *const recs = WOOP ? T.leaf_woop : T.leaf_tris;
        const long long win = coop_leaf<MODE == RESTART, WOOP>(recs, C, bm, (unsigned)base * 48u, R.o, R.d, R.th);
        if (q >= 0 && at_leaf) {
            int hit = -1;
            if (win >= 0) {             // the owner's own test of its winner
                const float4 *W = reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(recs) +
                                                                   (unsigned)win);
                const float4 a0 = W[0];
                if constexpr (WOOP) {
                    if (woop_test(a0, W[1], W[2], R.o, R.d, R.th, R.tu, R.tv))
                        hit = T.prim_indices[(unsigned)win / 48u];
                } else {
                    if (mt_edges(mk3(a0), mk3(W[1]), mk3(W[2]), R.o, R.d, R.th, R.tu, R.tv))
                        hit = __float_as_int(a0.w);
                }
            }
            done = hit != -1 || !(R.th < F_INF);
            if (CANVAS && hit != -1) {
                // shade the hit; the mirror ray goes on in this lane
                f3 o = R.o, d = R.d;
                col = blend(col, lighting(ray_record(R, hit), o, d, V.n0, V.n1, V.n2, V.c0, V.light));
                done = !(col.w < 0.97f) || ++bounce >= V.max_bounces;
                R = ray_start(T, R.root_id, o, adjust_dir(d));
            }
            if (done) {
                if (CANVAS) V.canvas[q] = canvas_pixel(col);
                else out[q] = ray_record(R, hit);
                if (COUNT) counters[q] = cnt;
                q = -1;
            }
        } else if (q >= 0 && done) {    // done before a leaf: a miss
            if (CANVAS) V.canvas[q] = canvas_pixel(col);
            else out[q] = miss_record();
            if (COUNT) counters[q] = cnt;
            q = -1;
        }
    }
}

// ---- brute force
// Every ray against every triangle; the record is the one the sequential loop
// ends with (accept 0 <= t <= th, then th = t): the smallest t, ties to the
// highest index, so hits are offered as keys (t bits, ~index) to the ray's
// 64-bit LDS minimum and the winner is tested once more for t, u, v.
//
// Moller-Trumbore: nearly all of the work is to find that a ray passes a
// triangle by, and that is a contraction.  With w = o x d and N = e1 x e2,
//   det = -d.N,  f1 = det u = d.(v0 x e2) + w.e2,
//   f2 = det v = -d.(v0 x e1) - w.e1,  f3 = det - f1 - f2,
// so the three edge values of 32 triangles and 32 rays are three 32x32x8
// matrix products of (d, w) with the triangles' vectors.  A pair the exact
// test accepts has f1, f2, f3 of one sign up to rounding; pairs that do not
// (beyond a bound E on every rounding involved) are dropped, the others are
// listed and tested exactly, 64 at a time.
//
// The bound.  Coordinates are taken relative to c, a vertex (exact to half an
// ulp of the differences), and scaled by S > 0:
//   ray       (S d, w) / alpha,          alpha = |d| (S + |o|)
//   triangle  (g / S, h) / beta,         beta = em (S + V) / S,
//             em = |e1| + |e2|, V = |v0| + em, g / h its d and w vectors
// The halves of the ray's vector then have norms S / (S + |o|) and |o| / (S +
// |o|), the triangle's at most V / (S + V) and S / (S + V), so the sum of the
// absolute products of a value is at most S (|o| + V) / ((S + |o|) (S + V)) <=
// 1, and alpha beta >= |d| em (|o| + V).  Rounding the entries to 16 bits moves
// a value by at most 2^-10 (2^-11 of an entry on either side) and, where
// entries are tiny or flushed (2^-14 of each), by 2 sqrt(3) 2^-14 = 0.00021;
// the exact test's own rounding of f1, f2, det (a few 2^-24 of |d| em (|o| +
// V)), of u + v <= 1 and of these vectors is below 2^-18.  E = 0.00122 covers
// their sum, 0.00119.
// A ray or triangle whose alpha or beta is not in [2^-40, 2^40] (NaN,
// infinite, degenerate or out of range) gets the zero vector: always listed.  So
// does one whose |d| or em is below 2^-60: squared, a length below about 2^-70
// is a few multiples of 2^-149, off by up to a third, and products of the exact
// test that small round by more than a part of their size.  (From 2^-60 on a
// square is exact to 2^-24, and |d| em >= 2^-120 keeps the exact test's products
// above what 2^-149 roundings change.)
//
constexpr int BRUTE_WAVES = 16;          // waves of a block, each with its share of the triangles
constexpr int BRUTE_T = 64 * BRUTE_WAVES;
constexpr float BRUTE_E = 0x1.4p-10f;

typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float norm3(f3 a) { return sqrtf(dot3(a, a)); }
__device__ __forceinline__ bool brute_scale_ok(float x) { return x >= 0x1p-40f && x <= 0x1p40f; }
__device__ __forceinline__ bool brute_length_ok(float x) { return x >= 0x1p-60f; }
__device__ __forceinline__ half4 to_half4(f3 a) {
    half4 h;
    h.x = (_Float16)a.x; h.y = (_Float16)a.y; h.z = (_Float16)a.z; h.w = (_Float16)0.0f;
    return h;
}

__device__ __forceinline__ unsigned long long hit_key(float t, int id) {
    return ((unsigned long long)__float_as_uint(t + 0.0f) << 32) | (unsigned)~id;
}

// the record of a ray whose best key is k: the winner's own test again
template <bool WOOP>
__device__ __forceinline__ pm_hit brute_record(unsigned long long k, const float4 *__restrict__ A,
                                               const float4 *__restrict__ B, const float4 *__restrict__ C, f3 o,
                                               f3 d) {
    pm_hit res = miss_record();
    if (k == ~0ull) return res;
    const int id = (int)~(unsigned)(k & 0xffffffffu);
    float th = F_INF, tu = 0.0f, tv = 0.0f;
    const bool h = WOOP ? woop_test(A[id], B[id], C[id], o, d, th, tu, tv)
                        : moller_trumbore(mk3(A[id]), mk3(B[id]), mk3(C[id]), o, d, th, tu, tv);
    if (h && th < F_INF) { res.id = id; res.t = th; res.u = tu; res.v = tv; }
    return res;
}

// RT: 32-ray tiles of a block (the same rays for its 16 waves, which take the
// triangle tiles w, w + 16, ...)
template <int RT, bool COUNT>
__global__ __launch_bounds__(BRUTE_T) void brute_kernel(const float4 *__restrict__ P0, const float4 *__restrict__ P1,
                                                        const float4 *__restrict__ P2, int ntris,
                                                        const float4 *__restrict__ org,
                                                        const float4 *__restrict__ dir, int n,
                                                        pm_hit *__restrict__ out, int4 *__restrict__ counters) {
    constexpr int NR = 32 * RT;
    __shared__ unsigned long long key[NR];
    __shared__ int list_tri[BRUTE_WAVES][128];
    __shared__ unsigned short list_ray[BRUTE_WAVES][128];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 31;
    const bool wpart = lane >= 32;         // lanes 32..63 hold the operands' w half (k = 4..7)
    const int r0 = blockIdx.x * NR;
    for (int j = threadIdx.x; j < NR; j += BRUTE_T) key[j] = ~0ull;
    __syncthreads();
    if (ntris > 0) {
        // the frame: c a vertex, S the size of a sample of the triangles
        // (any c and any S > 0 are right; these keep E small in the scene)
        const f3 first = mk3(P0[0]);
        const bool fin = fabsf(first.x) < 0x1p40f && fabsf(first.y) < 0x1p40f && fabsf(first.z) < 0x1p40f;
        const f3 c = fin ? first : f3{0.0f, 0.0f, 0.0f};
        float S;
        {
            const int k = (int)((long long)lane * ntris / 64);
            float v = norm3(sub3(mk3(P0[k]), c));
            v = brute_scale_ok(v) ? v : 0.0f;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
            S = v > 0.0f ? v : 1.0f;
        }
        half4 rays[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const int r = min(r0 + 32 * t + col, n - 1);
            const f3 o = sub3(mk3(org[r]), c), d = mk3(dir[r]);
            const float len = norm3(d), alpha = len * (S + norm3(o));
            const f3 x = wpart ? cross3(o, d) : f3{d.x * S, d.y * S, d.z * S};
            const float k = 1.0f / alpha;
            const bool ok = brute_scale_ok(alpha) && brute_length_ok(len);
            rays[t] = to_half4(ok ? f3{x.x * k, x.y * k, x.z * k} : f3{0.0f, 0.0f, 0.0f});
        }
        int pending = 0;
        // tests the list's first m pairs exactly
        auto flush = [&](int m) {
            if (lane < m) {
                const int tri = list_tri[w][lane], j = list_ray[w][lane];
                float th = F_INF, tu, tv;
                if (moller_trumbore(mk3(P0[tri]), mk3(P1[tri]), mk3(P2[tri]), mk3(org[r0 + j]), mk3(dir[r0 + j]), th,
                                    tu, tv))
                    atomicMin(&key[j], hit_key(th, tri));
            }
        };
        const int tiles = (ntris + 31) >> 5;
        auto load_tri = [&](int tile, float4 &a, float4 &b, float4 &e) {
            const int k = min(32 * tile + col, ntris - 1);
            a = P0[k]; b = P1[k]; e = P2[k];
        };
        float4 na, nb, ne;
        if (w < tiles) load_tri(w, na, nb, ne);
        for (int tile = w; tile < tiles; tile += BRUTE_WAVES) {
            const f3 p0 = mk3(na), p1 = mk3(nb), p2 = mk3(ne);
            if (tile + BRUTE_WAVES < tiles) load_tri(tile + BRUTE_WAVES, na, nb, ne);
            half4 t1, t2, t3;
            {
                const f3 v0 = sub3(p0, c), e1 = sub3(p1, p0), e2 = sub3(p2, p0);
                const float em = norm3(e1) + norm3(e2);
                const float beta = em * (S + norm3(v0) + em) / S;
                const bool ok = brute_scale_ok(beta) && brute_length_ok(em);
                f3 g1, g2, g3;
                float k = 1.0f / beta;
                if (wpart) {
                    g1 = e2; g2 = {-e1.x, -e1.y, -e1.z}; g3 = sub3(e1, e2);
                } else {
                    k = k / S;
                    g1 = cross3(v0, e2);
                    g2 = cross3(e1, v0);
                    const f3 m = cross3(e2, e1);
                    g3 = sub3(sub3(m, g1), g2);
                }
                k = ok ? k : 0.0f;
                auto scaled = [&](f3 g) {
                    return to_half4(ok ? f3{g.x * k, g.y * k, g.z * k} : f3{0.0f, 0.0f, 0.0f});
                };
                t1 = scaled(g1); t2 = scaled(g2); t3 = scaled(g3);
            }
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                const f32x16 zero = {0};
                const f32x16 f1 = __builtin_amdgcn_mfma_f32_32x32x8f16(t1, rays[t], zero, 0, 0, 0);
                const f32x16 f2 = __builtin_amdgcn_mfma_f32_32x32x8f16(t2, rays[t], zero, 0, 0, 0);
                const f32x16 f3_ = __builtin_amdgcn_mfma_f32_32x32x8f16(t3, rays[t], zero, 0, 0, 0);
                // max over the tile of max(min f, -max f): a pair is listed at >= -E
                float best = -1.0f;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float lo = fminf(fminf(f1[r], f2[r]), f3_[r]), hi = fmaxf(fmaxf(f1[r], f2[r]), f3_[r]);
                    best = fmaxf(fmaxf(best, lo), -hi);
                }
                if (__ballot(best >= -BRUTE_E) == 0ull) continue;
                const bool ray_in = r0 + 32 * t + col < n;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float lo = fminf(fminf(f1[r], f2[r]), f3_[r]), hi = fmaxf(fmaxf(f1[r], f2[r]), f3_[r]);
                    const int tri = 32 * tile + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    const bool cand = fmaxf(lo, -hi) >= -BRUTE_E && ray_in && tri < ntris;
                    const unsigned long long m = __ballot(cand);
                    if (m == 0ull) continue;
                    if (cand) {
                        const int at = pending + __popcll(m & (lane ? ~0ull >> (64 - lane) : 0ull));
                        list_tri[w][at] = tri;
                        list_ray[w][at] = (unsigned short)(32 * t + col);
                    }
                    pending += __popcll(m);
                    if (pending >= 64) {
                        wave_sync();
                        flush(64);
                        wave_sync();
                        pending -= 64;
                        if (lane < pending) {
                            list_tri[w][lane] = list_tri[w][64 + lane];
                            list_ray[w][lane] = list_ray[w][64 + lane];
                        }
                        wave_sync();
                    }
                }
            }
        }
        wave_sync();
        flush(pending);
    }
    __syncthreads();
    for (int j = threadIdx.x; j < NR; j += BRUTE_T) {
        const int r = r0 + j;
        if (r >= n) continue;
        out[r] = brute_record<false>(key[j], P0, P1, P2, mk3(org[r]), mk3(dir[r]));
        if (COUNT) counters[r] = make_int4(0, 0, ntris, 0);
    }
}

// Woop: P0/P1/P2 hold the matrices m0/m1/m2.  64 rays a block, every wave
// with its share of the triangles (w, w + 16, ...), read through the scalar
// cache: one triangle for the 64 lanes.  (The matrices come out of a float
// inversion, so no bound of their test's rounding is small enough to filter by.)
template <bool COUNT>
__global__ __launch_bounds__(BRUTE_T) void brute_woop_kernel(const float4 *__restrict__ W0,
                                                             const float4 *__restrict__ W1,
                                                             const float4 *__restrict__ W2, int ntris,
                                                             const float4 *__restrict__ org,
                                                             const float4 *__restrict__ dir, int n,
                                                             pm_hit *__restrict__ out, int4 *__restrict__ counters) {
    __shared__ unsigned long long key[64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (threadIdx.x < 64) key[threadIdx.x] = ~0ull;
    __syncthreads();
    const int r = blockIdx.x * 64 + lane;
    const f3 o = mk3(org[min(r, n - 1)]), d = mk3(dir[min(r, n - 1)]);
    float th = F_INF, tu = 0.0f, tv = 0.0f;
    int hit = -1;
#pragma unroll 2
    for (int k = w; k < ntris; k += BRUTE_WAVES)
        if (woop_test(W0[k], W1[k], W2[k], o, d, th, tu, tv)) hit = k;
    if (hit >= 0) atomicMin(&key[lane], hit_key(th, hit));
    __syncthreads();
    if (w == 0 && r < n) {
        out[r] = brute_record<true>(key[lane], W0, W1, W2, o, d);
        if (COUNT) counters[r] = make_int4(0, 0, ntris, 0);
    }
}

// A lane per ray through every triangle in index order, the triangles staged
// through LDS (TB at a time): for few triangles and many rays (see
// brute_lane_per_ray).
template <bool COUNT, bool WOOP>
__global__ __launch_bounds__(TB) void brute_lanes_kernel(const float4 *__restrict__ P0,
                                                         const float4 *__restrict__ P1,
                                                         const float4 *__restrict__ P2, int ntris,
                                                         const float4 *__restrict__ org,
                                                         const float4 *__restrict__ dir, int n,
                                                         pm_hit *__restrict__ out, int4 *__restrict__ counters) {
    __shared__ float4 s0[TB], s1[TB], s2[TB];
    const int r = blockIdx.x * TB + threadIdx.x;
    const bool live = r < n;
    f3 o = {0.0f, 0.0f, 0.0f}, d = {0.0f, 0.0f, 1.0f};
    if (live) { o = mk3(org[r]); d = mk3(dir[r]); }
    float th = F_INF, tu = 0.0f, tv = 0.0f;
    int hit = -1;
    for (int base = 0; base < ntris; base += TB) {
        const int k = base + threadIdx.x;
        __syncthreads();
        if (k < ntris) { s0[threadIdx.x] = P0[k]; s1[threadIdx.x] = P1[k]; s2[threadIdx.x] = P2[k]; }
        __syncthreads();
        const int m = min(TB, ntris - base);
        if (live) {
            for (int j = 0; j < m; ++j) {
                const bool h = WOOP ? woop_test(s0[j], s1[j], s2[j], o, d, th, tu, tv)
                                    : moller_trumbore(mk3(s0[j]), mk3(s1[j]), mk3(s2[j]), o, d, th, tu, tv);
                if (h) hit = base + j;
            }
        }
    }
    if (!live) return;
    pm_hit res = miss_record();
    if (th < F_INF && hit != -1) { res.id = hit; res.t = th; res.u = tu; res.v = tv; }
    out[r] = res;
    if (COUNT) counters[r] = make_int4(0, 0, ntris, 0);
}

// ---- trace view
// n = n_dev ? *n_dev : n_host (a captured build passes its device node count)
__global__ __launch_bounds__(TB) void pack_nodes_kernel(const int8_t *__restrict__ info,
                                                        const float *__restrict__ split,
                                                        const int2 *__restrict__ children,
                                                        const int *__restrict__ prim_index,
                                                        const long long *__restrict__ bitmap,
                                                        const float4 *__restrict__ bmin,
                                                        const float4 *__restrict__ bmax, int n_host,
                                                        const int *n_dev, int4 *__restrict__ out,
                                                        float4 *__restrict__ leaf_rec) {
    const int n = n_dev ? *n_dev : n_host;
    for (int i = blockIdx.x * TB + threadIdx.x; i < n; i += gridDim.x * TB) {
        const int ax = info[i] & 3;
        if (ax) {
            const int2 c = children[i];
            // (a captured build that failed leaves nodes with any children)
            const bool ll = (unsigned)c.x < (unsigned)n && !(info[c.x] & 3);
            const bool rl = (unsigned)c.y < (unsigned)n && !(info[c.y] & 3);
            out[i] = make_int4(__float_as_int(split[i]), ll ? c.x | LEAF_CODE : c.x, rl ? c.y | LEAF_CODE : c.y, ax);
        } else {
            const unsigned long long b = (unsigned long long)bitmap[i];
            const int first = prim_index[i], lo = (int)(unsigned)(b & 0xffffffffull);
            out[i] = make_int4(first, lo, (int)(unsigned)(b >> 32), LEAF);
            const float4 mn = bmin[i], mx = bmax[i];
            leaf_rec[2ll * i] = make_float4(mn.x, mn.y, mn.z, __int_as_float(first));
            leaf_rec[2ll * i + 1] = make_float4(mx.x, mx.y, mx.z, __int_as_float(lo));
        }
    }
}

// leaf slot k -> v0 (w = id bits), e1, e2; an index outside the triangles
// sets *bad
__global__ __launch_bounds__(TB) void leaf_tris_kernel(const int *__restrict__ prim_indices, int m,
                                                       const float4 *__restrict__ P0,
                                                       const float4 *__restrict__ P1,
                                                       const float4 *__restrict__ P2, int ntris,
                                                       float4 *__restrict__ out, int *bad) {
    const int k = blockIdx.x * TB + threadIdx.x;
    if (k >= m) return;
    const int t = prim_indices[k];
    if (t < 0 || t >= ntris) {
        atomicOr(bad, 1);
        const float nan = __int_as_float(0x7fc00000);
        out[3ll * k] = make_float4(nan, nan, nan, __int_as_float(-1));
        out[3ll * k + 1] = make_float4(nan, nan, nan, 0.0f);
        out[3ll * k + 2] = make_float4(nan, nan, nan, 0.0f);
        return;
    }
    const f3 v0 = mk3(P0[t]), v1 = mk3(P1[t]), v2 = mk3(P2[t]);
    const f3 e1 = sub3(v1, v0), e2 = sub3(v2, v0);
    out[3ll * k] = make_float4(v0.x, v0.y, v0.z, __int_as_float(t));
    out[3ll * k + 1] = make_float4(e1.x, e1.y, e1.z, 0.0f);
    out[3ll * k + 2] = make_float4(e2.x, e2.y, e2.z, 0.0f);
}

// A build's leaf slots from its final refs (the triangle index is in their
// min.w, ExtractIndexFromAabb, TriangleUpper.h:43-52): the slot's prim index,
// its triangle's record by one contiguous 48-byte gather, and (areas) its
// triangle's area 0.5 |e1 x e2| (CalcSurfaceArea, LowerTriangleMap.h:24-38, the
// same operations tri_area performs).  The indices are
// not written by a pass of their own and read back here (1,000,002 triangles:
// 105 -> 103 us and a launch less).
__global__ __launch_bounds__(TB) void leaf_slots_kernel(const float4 *__restrict__ refs, const Lvl *__restrict__ L,
                                                        const float4 *__restrict__ rec,
                                                        int *__restrict__ prim_indices, float4 *__restrict__ out,
                                                        float *__restrict__ areas) {
    const int m = L->status ? 0 : L->final_refs;
    for (int k = blockIdx.x * TB + threadIdx.x; k < m; k += gridDim.x * TB) {
        const int t = __float_as_int(refs[k].w);
        const float4 r0 = rec[3ll * t], r1 = rec[3ll * t + 1], r2 = rec[3ll * t + 2];
        prim_indices[k] = t;
        out[3ll * k] = r0;
        out[3ll * k + 1] = r1;
        out[3ll * k + 2] = r2;
        if (areas) {
            const f3 c = cross3(mk3(r1), mk3(r2));
            areas[k] = 0.5f * sqrtf(dot3(c, c));
        }
    }
}

// brute-force first hit for one ray (Exhaustive, BruteTracer.cu:54-96),
// straight from global memory
template <bool WOOP>
__device__ __forceinline__ pm_hit brute_ray(const float4 *__restrict__ A, const float4 *__restrict__ B,
                                            const float4 *__restrict__ C, int ntris, f3 o, f3 d) {
    float th = F_INF, tu = 0.0f, tv = 0.0f;
    int hit = -1;
    for (int k = 0; k < ntris; ++k) {
        const bool h = WOOP ? woop_test(A[k], B[k], C[k], o, d, th, tu, tv)
                            : moller_trumbore(mk3(A[k]), mk3(B[k]), mk3(C[k]), o, d, th, tu, tv);
        if (h) hit = k;
    }
    pm_hit res = miss_record();
    if (th < F_INF && hit != -1) { res.id = hit; res.t = th; res.u = tu; res.v = tv; }
    return res;
}

// IRayTracer::Trace(canvas): per ray, first hit -> Lighting -> BlendColor
// until a miss, alpha >= 0.97 or max_bounces; one uchar4 per ray
template <int ALGO, bool SKIP, bool WOOP>
__global__ __launch_bounds__(TB) void canvas_kernel(TreeDev T, const float4 *__restrict__ A,
                                                    const float4 *__restrict__ B,
                                                    const float4 *__restrict__ C, int ntris,
                                                    const float4 *__restrict__ org,
                                                    const float4 *__restrict__ dir, int n, int S,
                                                    const float4 *__restrict__ n0,
                                                    const float4 *__restrict__ n1,
                                                    const float4 *__restrict__ n2,
                                                    const uchar4 *__restrict__ c0, Light L, int max_bounces,
                                                    uchar4 *__restrict__ canvas) {
    __shared__ int stk_rows[2 * (ALGO == PM_TRACE_SHORT_STACK ? 16 : 1)][TB];   // node rows, then tNext rows
    int *const stk = &stk_rows[0][threadIdx.x];
    const int r = blockIdx.x * TB + threadIdx.x;
    if (r >= n) return;
    f3 o = mk3(org[r]), d = mk3(dir[r]);
    if (ALGO != PM_TRACE_BRUTE) d = adjust_dir(d);
    float4 col = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    int4 cnt = make_int4(0, 0, 0, 0);
    const int root = ALGO != PM_TRACE_BRUTE ? root_code(T, 0) : 0;
    for (int b = 0; b < max_bounces; ++b) {
        pm_hit h;
        if constexpr (ALGO == PM_TRACE_BRUTE) {
            h = brute_ray<WOOP>(A, B, C, ntris, o, d);
        } else if constexpr (ALGO == PM_TRACE_KD_RESTART) {
            h = kd_restart_ray<SKIP, false, WOOP>(T, root, o, d, cnt);
        } else {
            h = short_stack_ray<16, SKIP, false, WOOP>(T, root, o, d, S, stk, cnt);
        }
        if (h.id < 0) break;
        col = blend(col, lighting(h, o, d, n0, n1, n2, c0, L));
        if (ALGO != PM_TRACE_BRUTE) d = adjust_dir(d);
        if (!(col.w < 0.97f)) break;
    }
    canvas[r] = canvas_pixel(col);
}

// CreateWoopValues (GeometryList.cu:80-101): matrices of (p1, p2, p0) for
// every triangle (W0/W1/W2 arrays) or for every leaf slot (3 per slot)
__global__ __launch_bounds__(TB) void woop_tris_kernel(const float4 *__restrict__ P0,
                                                       const float4 *__restrict__ P1,
                                                       const float4 *__restrict__ P2, int n,
                                                       float4 *__restrict__ W0, float4 *__restrict__ W1,
                                                       float4 *__restrict__ W2) {
    const int k = blockIdx.x * TB + threadIdx.x;
    if (k >= n) return;
    float4 m0, m1, m2;
    woop_matrix(mk3(P1[k]), mk3(P2[k]), mk3(P0[k]), m0, m1, m2);
    W0[k] = m0; W1[k] = m1; W2[k] = m2;
}

__global__ __launch_bounds__(TB) void woop_slots_kernel(const int *__restrict__ prim_indices, int m,
                                                        const float4 *__restrict__ P0,
                                                        const float4 *__restrict__ P1,
                                                        const float4 *__restrict__ P2, int ntris,
                                                        float4 *__restrict__ W) {
    const int k = blockIdx.x * TB + threadIdx.x;
    if (k >= m) return;
    const int t = prim_indices[k];
    float4 m0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), m1 = m0, m2 = m0;
    if (t >= 0 && t < ntris) woop_matrix(mk3(P1[t]), mk3(P2[t]), mk3(P0[t]), m0, m1, m2);
    W[3ll * k] = m0; W[3ll * k + 1] = m1; W[3ll * k + 2] = m2;
}

__global__ void clear_int_kernel(int *p) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p = 0;
}

// the rays of one trace call
struct RayBatch {
    const float4 *org, *dir;
    const int *root;            // per-ray root (forest) or null
    const unsigned *order;      // the order the rays are traced in, or null
    int n;
};

// persistent grid: at most as many blocks as the device holds at once
struct Launch {
    int num_cus;
    int *work;
    int step_cap;   // pm_trace_params.step_cap (cooperative kernels)
};

template <class K>
long long resident_blocks(K kernel, const Launch &L) {
    int b = 0;
    PM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, kernel, TB, 0));
    return (long long)(b > 0 ? b : 1) * L.num_cus;
}

void clear_work(int *work, hipStream_t s) {
    clear_int_kernel<<<1, 64, 0, s>>>(work);
    PM_LAUNCH_CHECK();
}

// The cooperative kernel's launch.  A wave that holds 64 rays waits for the
// slowest of them in every round, and a trace of fewer rays than the device
// holds lanes leaves SIMDs without a wave; the leaf test needs its 64 lanes
// for the pairs, not for 64 rays.  So a trace takes the narrowest waves (a
// power of two of rays) whose number still fits the device at once: 65,536
// camera rays in a 5,316-triangle room take 103 us with 16 rays a wave, 115
// with 32, 130 with 64; 1,000 probe rays in a 50,000-triangle soup 80 us with
// 1 and 228 with 64; past the line (30,000 probes: 143 us with 8 rays a wave,
// 190 with 4) the extra waves queue.  When every wave's first chunk covers
// all rays the counter is neither cleared nor read; a launch without a counter
// always does that, its later blocks starting as earlier ones end.
template <class K>
void launch_coop(K k, const TreeDev &T, const RayBatch &R, int S, pm_hit *out, int4 *cnt, const Launch &L, int cap,
                 hipStream_t s, const CanvasArgs &V = CanvasArgs{}) {
    const long long resident = resident_blocks(k, L);
    constexpr int WAVES = TB / 64;
    int width = 64;
    while (width > 1 && R.n <= resident * WAVES * (width / 2)) width /= 2;
    const long long blocks = ((long long)R.n + WAVES * width - 1) / (WAVES * width);
    const bool one_chunk = !L.work || blocks <= resident;
    if (!one_chunk) clear_work(L.work, s);
    k<<<(int)(one_chunk ? blocks : resident), TB, 0, s>>>(T, R.org, R.dir, R.root, R.order, R.n, S, out, cnt,
                                                    one_chunk ? nullptr : L.work, cap, width, V);
}

template <int SMAX, bool SHORT, bool SKIP, bool COUNT, bool WOOP>
void launch_trace(const TreeDev &T, const RayBatch &R, int S, pm_hit *out, int4 *cnt, const Launch &L,
                  hipStream_t s) {
    if (48ll * T.num_slots < (1ll << 32)) {
        // kd-restart's counters count the nodes of every restart; without
        // them it resumes (a ring of 8)
        constexpr int MODE = SHORT ? SHORT_RING : COUNT ? RESTART : RESUME, RING = MODE == RESUME ? 8 : SMAX;
        const int ring = MODE == RESUME ? RING : S;
        if (L.step_cap > 0) {
            auto k = trace_coop_kernel<RING, MODE, SKIP, COUNT, true, WOOP>;
            launch_coop(k, T, R, ring, out, cnt, L, L.step_cap, s);
        } else {
            auto k = trace_coop_kernel<RING, MODE, SKIP, COUNT, false, WOOP>;
            launch_coop(k, T, R, ring, out, cnt, L, 0, s);
        }
    } else {
        auto k = trace_kernel<SMAX, SHORT, SKIP, COUNT, WOOP>;
        clear_work(L.work, s);
        const long long blocks = std::min(((long long)R.n + TB - 1) / TB, resident_blocks(k, L));
        k<<<(int)blocks, TB, 0, s>>>(T, R.org, R.dir, R.root, R.order, R.n, S, out, cnt, L.work);
    }
}

template <bool SKIP, bool COUNT, bool WOOP>
void dispatch(const TreeDev &T, int algo, const RayBatch &R, int S, pm_hit *out, int4 *cnt, const Launch &L,
              hipStream_t s) {
    if (algo == PM_TRACE_KD_RESTART) {
        launch_trace<1, false, SKIP, COUNT, WOOP>(T, R, 1, out, cnt, L, s);
    } else {
        if (S <= 4) launch_trace<4, true, SKIP, COUNT, WOOP>(T, R, S, out, cnt, L, s);
        else if (S <= 8) launch_trace<8, true, SKIP, COUNT, WOOP>(T, R, S, out, cnt, L, s);
        else launch_trace<16, true, SKIP, COUNT, WOOP>(T, R, S, out, cnt, L, s);
    }
}

template <bool WOOP>
void dispatch_flags(const TreeDev &T, bool skip, bool count, int algo, const RayBatch &R, int S, pm_hit *out,
                    int4 *cnt, const Launch &L, hipStream_t s) {
    if (skip) {
        if (count) dispatch<true, true, WOOP>(T, algo, R, S, out, cnt, L, s);
        else dispatch<true, false, WOOP>(T, algo, R, S, out, cnt, L, s);
    } else {
        if (count) dispatch<false, true, WOOP>(T, algo, R, S, out, cnt, L, s);
        else dispatch<false, false, WOOP>(T, algo, R, S, out, cnt, L, s);
    }
}

}  // namespace

void build_node_view(pm_ctx *ctx, hipStream_t s, const int *n_dev) {
    const int n = ctx->num_nodes;
    ctx->packed.reserve((size_t)n + 1, s);
    ctx->leaf_rec.reserve(2 * (size_t)n + 2, s);
    if (n > 0) {
        const int blocks = std::min((n + TB - 1) / TB, n_dev ? 4096 : INT_MAX);
        pack_nodes_kernel<<<blocks, TB, 0, s>>>(ctx->nodes.info.ptr, ctx->nodes.split.ptr, ctx->nodes.children.ptr,
                                                ctx->nodes.prim_index.ptr, ctx->nodes.bitmap.ptr,
                                                ctx->nodes.bmin.ptr, ctx->nodes.bmax.ptr, n, n_dev, ctx->packed.ptr,
                                                ctx->leaf_rec.ptr);
        PM_LAUNCH_CHECK();
    }
}

void build_leaf_slots(pm_ctx *ctx, const float4 *refs, const float4 *rec, float *areas, const Lvl *L, hipStream_t s) {
    const int m = ctx->num_prim_indices;
    ctx->leaf_tris.reserve(3 * (size_t)m + 3, s);
    if (m == 0) return;
    leaf_slots_kernel<<<std::min((m + TB - 1) / TB, 1 << 16), TB, 0, s>>>(refs, L, rec, ctx->prim_indices.ptr,
                                                                         ctx->leaf_tris.ptr, areas);
    PM_LAUNCH_CHECK();
}

namespace {

// an uploaded tree's leaf slots, from its prim indices, which are checked
void build_leaf_view(pm_ctx *ctx, hipStream_t s) {
    const int m = ctx->num_prim_indices;
    ctx->leaf_tris.reserve(3 * (size_t)m + 3, s);
    if (m == 0) return;
    BuildScratch &sc = ctx->scratch;
    sc.totals.reserve(8, s);
    sc.host.ensure(8);
    clear_int_kernel<<<1, 64, 0, s>>>(sc.totals.ptr);
    PM_LAUNCH_CHECK();
    leaf_tris_kernel<<<(m + TB - 1) / TB, TB, 0, s>>>(ctx->prim_indices.ptr, m, ctx->p0, ctx->p1, ctx->p2, ctx->ntris,
                                                      ctx->leaf_tris.ptr, sc.totals.ptr);
    PM_LAUNCH_CHECK();
    PM_HIP(hipMemcpyAsync(sc.host.ptr, sc.totals.ptr, sizeof(int), hipMemcpyDeviceToHost, s));
    PM_HIP(hipStreamSynchronize(s));
    if (sc.host.ptr[0]) throw Error{PM_ERR_ARG, "prim index outside the triangle array"};
}

}  // namespace


void build_trace_view(pm_ctx *ctx, hipStream_t s) {
    ctx->wide_leaves = true;   // an uploaded tree's bitmaps are not looked through
    build_node_view(ctx, s);
    build_leaf_view(ctx, s);
}

namespace {

TreeDev tree_dev(pm_ctx *ctx) {
    TreeDev T;
    T.prim_indices = ctx->prim_indices.ptr;
    T.packed = ctx->packed.ptr;
    T.leaf_rec = ctx->leaf_rec.ptr;
    T.wide = ctx->wide_leaves;
    T.leaf_tris = ctx->leaf_tris.ptr;
    T.leaf_woop = nullptr;
    T.num_nodes = ctx->num_nodes;
    T.num_roots = ctx->num_roots;
    T.num_slots = ctx->num_prim_indices;
    T.fail = ctx->trace_fail;
    return T;
}

// GetWoopValues, computed per call: per leaf slot for the tree tracers
const float4 *woop_slots(pm_ctx *ctx, hipStream_t s) {
    const int m = ctx->num_prim_indices;
    ctx->woop.reserve(3 * (size_t)m + 3, s);
    if (m > 0) {
        woop_slots_kernel<<<(m + TB - 1) / TB, TB, 0, s>>>(ctx->prim_indices.ptr, m, ctx->p0, ctx->p1, ctx->p2,
                                                           ctx->ntris, ctx->woop.ptr);
        PM_LAUNCH_CHECK();
    }
    return ctx->woop.ptr;
}

// ... and per triangle (W0 | W1 | W2) for brute force
float4 *woop_tris(pm_ctx *ctx, int tris, hipStream_t s) {
    ctx->woop.reserve(3 * (size_t)tris + 3, s);
    float4 *W = ctx->woop.ptr;
    if (tris > 0) {
        woop_tris_kernel<<<(tris + TB - 1) / TB, TB, 0, s>>>(ctx->p0, ctx->p1, ctx->p2, tris, W, W + tris,
                                                             W + 2ll * tris);
        PM_LAUNCH_CHECK();
    }
    return W;
}

void query_cus(pm_ctx *ctx);

// More rays a block mean fewer conversions of the triangles' vectors per pair,
// fewer rays more blocks: the most that still give every CU a block.  65,536
// rays x 5,316 triangles: 109 us with 128 rays a block, 134 with 64, 187 with
// 32 (256 need more registers than four waves a SIMD leave); a lane per ray
// through every triangle 1,440.  Bound by VALU issue: three instructions per
// pair and matrix tile row.
//
// A block costs some 6 us before its first pair, so where there are many of
// them and few triangles the lane-per-ray kernel is the better one.  Its time is
// 0.27 us a triangle (0.3 Woop) until the device is full and grows with the rays
// then; the others' grows with the rays at once.  Lane per ray / matrix filter,
// us: 32,768 rays x 24 triangles 9/10, x 48 16/11; 131,072 x 96 29/35, x 192
// 55/37; 262,144 x 1 9/50, x 128 51/68, x 256 100/73; 2M x 1 16/390, x 192
// 410/569, x 384 811/676.  Woop's split kernel (64 rays a block): 262,144 x 32
// 17/20, x 96 39/36; 1M x 1 12/42, x 192 214/221, x 512 557/557; 131,072 and fewer
// within 1 us up to 24 triangles, slower with more.  So the limits are 30
// triangles (Woop 8) per 128 rays of a CU, up to the line from which the filter
// wins at any number of rays (192; Woop: 384, the two are equal from there).
bool brute_lane_per_ray(const pm_ctx *ctx, int tris, int n, bool woop) {
    const long long limit = (long long)(woop ? 8 : 30) * n / (128ll * ctx->num_cus);
    return tris <= std::min<long long>(limit, woop ? 384 : 192);
}

template <bool COUNT>
void brute_rays(pm_ctx *ctx, int tris, bool woop, const float4 *org, const float4 *dir, int n, pm_hit *out,
                int4 *counters, hipStream_t s) {
    query_cus(ctx);
    const float4 *A = ctx->p0, *B = ctx->p1, *C = ctx->p2;
    if (woop) {
        A = woop_tris(ctx, tris, s);
        B = A + tris;
        C = B + tris;
    }
    auto launch = [&](auto k, int rays, int threads) {
        k<<<(int)(((long long)n + rays - 1) / rays), threads, 0, s>>>(A, B, C, tris, org, dir, n, out, counters);
    };
    if (brute_lane_per_ray(ctx, tris, n, woop)) {
        if (woop) launch(brute_lanes_kernel<COUNT, true>, TB, TB);
        else launch(brute_lanes_kernel<COUNT, false>, TB, TB);
        return;
    }
    if (woop) return launch(brute_woop_kernel<COUNT>, 64, BRUTE_T);
    const long long per_cu = (long long)n / ctx->num_cus;
    if (per_cu >= 128) launch(brute_kernel<4, COUNT>, 128, BRUTE_T);
    else if (per_cu >= 64) launch(brute_kernel<2, COUNT>, 64, BRUTE_T);
    else launch(brute_kernel<1, COUNT>, 32, BRUTE_T);
}

void query_cus(pm_ctx *ctx) {
    if (ctx->num_cus) return;
    int v = 0;
    PM_HIP(hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, ctx->device));
    ctx->num_cus = v > 0 ? v : 1;
}

template <int SMAX, bool SHORT, bool SKIP, bool WOOP>
void launch_canvas_coop(const TreeDev &T, const RayBatch &R, int S, const Launch &L, hipStream_t s,
                        const CanvasArgs &V) {
    // (kd-restart does not resume here: 394 us with the ring and 378 without for
    // 1280 x 720 in a 5,316-triangle room)
    auto k = trace_coop_kernel<SMAX, SHORT ? SHORT_RING : RESTART, SKIP, false, false, WOOP, true>;
    launch_coop(k, T, R, S, nullptr, nullptr, L, 0, s, V);
}

template <bool SKIP, bool WOOP>
void dispatch_canvas(const TreeDev &T, int algo, const RayBatch &R, int S, const Launch &L, hipStream_t s,
                     const CanvasArgs &V) {
    if (algo == PM_TRACE_KD_RESTART) launch_canvas_coop<1, false, SKIP, WOOP>(T, R, 1, L, s, V);
    else if (S <= 4) launch_canvas_coop<4, true, SKIP, WOOP>(T, R, S, L, s, V);
    else if (S <= 8) launch_canvas_coop<8, true, SKIP, WOOP>(T, R, S, L, s, V);
    else launch_canvas_coop<16, true, SKIP, WOOP>(T, R, S, L, s, V);
}

template <int ALGO>
void launch_canvas(bool skip, bool woop, int blocks, hipStream_t s, const TreeDev &T, const float4 *A,
                   const float4 *B, const float4 *C, int ntris, const float4 *org, const float4 *dir, int n,
                   int S, const float4 *n0, const float4 *n1, const float4 *n2, const uchar4 *c0,
                   const Light &L, int maxb, uchar4 *canvas) {
    if (skip && woop)
        canvas_kernel<ALGO, true, true><<<blocks, TB, 0, s>>>(T, A, B, C, ntris, org, dir, n, S, n0, n1, n2, c0, L, maxb, canvas);
    else if (skip)
        canvas_kernel<ALGO, true, false><<<blocks, TB, 0, s>>>(T, A, B, C, ntris, org, dir, n, S, n0, n1, n2, c0, L, maxb, canvas);
    else if (woop)
        canvas_kernel<ALGO, false, true><<<blocks, TB, 0, s>>>(T, A, B, C, ntris, org, dir, n, S, n0, n1, n2, c0, L, maxb, canvas);
    else
        canvas_kernel<ALGO, false, false><<<blocks, TB, 0, s>>>(T, A, B, C, ntris, org, dir, n, S, n0, n1, n2, c0, L, maxb, canvas);
}

}  // namespace

void trace_rays(pm_ctx *ctx, int algo, const float4 *org, const float4 *dir, int nrays,
                const int *ray_mesh, pm_hit *out, const pm_trace_params &prm, int4 *counters,
                hipStream_t s, int *ext_work) {
    if (nrays == 0) return;
    const bool woop = prm.intersection == PM_INTERSECT_WOOP;
    if (algo == PM_TRACE_BRUTE) {
        const int tris = prm.brute_cap > 0 ? std::min(ctx->ntris, prm.brute_cap) : ctx->ntris;
        if (counters) brute_rays<true>(ctx, tris, woop, org, dir, nrays, out, counters, s);
        else brute_rays<false>(ctx, tris, woop, org, dir, nrays, out, counters, s);
        PM_LAUNCH_CHECK();
        return;
    }
    TreeDev T = tree_dev(ctx);
    if (woop) T.leaf_woop = woop_slots(ctx, s);
    const bool skip = prm.leaf_skipping && ctx->has_boxes;
    const int S = prm.stack_size;
    RayBatch R{org, dir, ray_mesh, nullptr, nrays};
    if (ray_order_used(prm, nrays, T.num_slots))
        R.order = ray_order(ctx, org, dir, ray_mesh, nrays, s);
    query_cus(ctx);
    int *work = ext_work;
    if (!work) {
        ctx->scratch.trace_work.reserve(1, s);
        work = ctx->scratch.trace_work.ptr;
    }
    const Launch L{ctx->num_cus, work, prm.step_cap};
    if (woop) dispatch_flags<true>(T, skip, counters != nullptr, algo, R, S, out, counters, L, s);
    else dispatch_flags<false>(T, skip, counters != nullptr, algo, R, S, out, counters, L, s);
    PM_LAUNCH_CHECK();
}

void trace_canvas(pm_ctx *ctx, int algo, const float4 *org, const float4 *dir, int nrays, const float4 *n0,
                  const float4 *n1, const float4 *n2, const uchar4 *c0, const pm_light &light, int max_bounces,
                  uchar4 *canvas, const pm_trace_params &prm, hipStream_t s) {
    if (nrays == 0) return;
    const bool woop = prm.intersection == PM_INTERSECT_WOOP;
    const Light L = {{light.position[0], light.position[1], light.position[2]},
                     {light.ambient[0], light.ambient[1], light.ambient[2]},
                     {light.diffuse[0], light.diffuse[1], light.diffuse[2]},
                     {light.specular[0], light.specular[1], light.specular[2]}};
    const int blocks = (nrays + TB - 1) / TB;
    TreeDev T = tree_dev(ctx);
    const float4 *A = ctx->p0, *B = ctx->p1, *C = ctx->p2;
    int tris = 0;
    if (algo == PM_TRACE_BRUTE) {
        tris = prm.brute_cap > 0 ? std::min(ctx->ntris, prm.brute_cap) : ctx->ntris;
        if (woop) {
            const float4 *W = woop_tris(ctx, tris, s);
            A = W; B = W + tris; C = W + 2ll * tris;
        }
        launch_canvas<PM_TRACE_BRUTE>(false, woop, blocks, s, T, A, B, C, tris, org, dir, nrays, 1, n0, n1, n2, c0,
                                      L, max_bounces, canvas);
    } else {
        if (woop) T.leaf_woop = woop_slots(ctx, s);
        const bool skip = prm.leaf_skipping && ctx->has_boxes;
        if (48ll * T.num_slots < (1ll << 32)) {
            query_cus(ctx);
            const Launch W{ctx->num_cus, nullptr, 0};
            const RayBatch R{org, dir, nullptr, nullptr, nrays};
            const CanvasArgs V{n0, n1, n2, c0, L, max_bounces, canvas};
            if (skip && woop) dispatch_canvas<true, true>(T, algo, R, prm.stack_size, W, s, V);
            else if (skip) dispatch_canvas<true, false>(T, algo, R, prm.stack_size, W, s, V);
            else if (woop) dispatch_canvas<false, true>(T, algo, R, prm.stack_size, W, s, V);
            else dispatch_canvas<false, false>(T, algo, R, prm.stack_size, W, s, V);
        } else if (algo == PM_TRACE_KD_RESTART)
            launch_canvas<PM_TRACE_KD_RESTART>(skip, woop, blocks, s, T, A, B, C, 0, org, dir, nrays, 1, n0, n1, n2,
                                               c0, L, max_bounces, canvas);
        else
            launch_canvas<PM_TRACE_SHORT_STACK>(skip, woop, blocks, s, T, A, B, C, 0, org, dir, nrays,
                                                prm.stack_size, n0, n1, n2, c0, L, max_bounces, canvas);
    }
    PM_LAUNCH_CHECK();
}

}  // namespace pmkd
