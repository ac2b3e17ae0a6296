// walk.hip -- device dual-tree walk emitting interaction lists grouped by target.
//
// The reference walks (target, source) cell pairs depth-first from (root, root)
// and emits P2P and M2L tasks (src/fmm.c:406-712 for the home box,
// src/remotes.c:213-552 against each of the 26 shifted, pruned copies of the tree
// built by prepare_sendtree2, src/remotes.c:60-169).  Which pairs it emits depends
// only on the rule applied to each pair, so any traversal that applies the same
// rules emits the same set.
//
// MI355X formulation: one launch per depth of the target tree, one workgroup per target
// at a time.  A pair (A, B) whose rule opens the target A passes the source B on to both
// children of A (a node paired with itself passes its two children): a node's down list
// is the source list of its two children.  A workgroup takes up to a window of its
// target's sources into LDS, applies the rule to all of them at once, replaces the opened
// ones by their children, level by level, and finally numbers the settled ones along the
// tree of replacements: the outputs of a target come out in the reference's order (shift,
// depth-first rank of the source) without a sort and without a second pass over the
// cells.  The space for a target's outputs is taken off a common counter when their
// number is known, so where a target lies in the lists varies from run to run; its
// entries and their order do not.

// Image walks: a shifted node keeps no children when its box is rc or more from
// the domain box or when 0.95*theta*distance exceeds its largest width
// (src/remotes.c:145-158); the rule is evaluated on the fly, no copy is built.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <stdexcept>

#include "engine.h"
#include "fmm_math.h"

namespace photons {

__host__ __device__ inline void shift_of(int sid, double L, double &sx, double &sy, double &sz)
{
    // ids 1..26: (mi, mj, mk) over {-1,0,1}^3 without (0,0,0), mi slowest
    if (sid <= 0) {
        sx = sy = sz = 0.0;
        return;
    }
    int k = sid <= 13 ? sid - 1 : sid;  // skip the centre (index 13 of the 27)
    sx = (double)(k / 9 - 1) * L;
    sy = (double)((k / 3) % 3 - 1) * L;
    sz = (double)(k % 3 - 1) * L;
}

__device__ __forceinline__ bool let_pruned(const CellGeom &root, const CellGeom &g, double sx, double sy, double sz,
                                           double rc, double theta)
{
    double s[3] = {sx, sy, sz};
    double dr = 0.0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        double d = root.c[i] - g.c[i] - s[i];
        if (d < 0.0) d = -d;
        d -= (root.w[i] + g.w[i]) * 0.5;
        if (d > 0.0) dr += d * d;
    }
    dr = sqrt(dr);
    double wmax = g.w[0];
    if (wmax < g.w[1]) wmax = g.w[1];
    if (wmax < g.w[2]) wmax = g.w[2];
    if (dr >= rc) return true;
    return wmax < 0.95 * theta * dr;
}

// what the rule does with one pair
enum : int {
    kActNone = 0,  // pruned
    kActP2P,       // a leaf with itself, or two leaves: P2P, whatever the acceptance says
    kActSelfNode,  // a node with itself: its children pass down
    kActM2L,       // accepted (or a target leaf against a pruned image node): M2L
    kActOpenA,     // open the target: the source passes down
    kActOpenB      // open the source
};

// by cell: what the rule needs of it, as a target or as a source, in one 64-byte record
struct alignas(16) WalkRec {
    CellGeom g;
    int32_t kid[2];  // a node's children, first and second in depth-first order; a leaf's parent (-1: none)
    int32_t swap;    // the second one is son 0
    int32_t box;
};
static_assert(sizeof(WalkRec) == 64, "one 64-byte record per cell");

enum : int { kP2P = 0, kM2L = 1, kDown = 2, kOut = 3 };  // what a walk writes
constexpr int kLeaves = -1;        // the step of the leaves
constexpr int kXcds = 8;           // workgroups go to the XCDs in turn, each with its own L2
constexpr int kWalkBlocks = 4096;  // workgroups of a launch, at most
constexpr int kCountSlots = 16;    // adders of a depth's counts

// The walk's own state in device memory, zeroed by k_walk_records
struct WalkState {
    unsigned long long next[kOut][16];               // list entries handed out (128 bytes apart)
    unsigned long long count[2][kOut][kCountSlots];  // outputs written, outputs counted ahead (ordinary evaluations)
    int heavy[kMaxDepth + 2][2], taken[kMaxDepth + 2][2];  // targets put off by step (0: leaves), counting and writing; those begun
    int overflow, pad;
    int64_t chunk[kWalkBlocks][kOut][2];             // the list space a workgroup holds: next entry, end
};

struct WalkArgs {
    const WalkRec *rec;      // by cell
    const DevSizes *sz;
    WalkState *st;
    const double *box_len;
    double theta, theta2, rc, rc2;
    int step;                // kLeaves, or 0: the start targets; d + 1: the node children of the nodes of depth d
    bool heavy_only;         // the targets of this step that were put off
    int tile;                // consecutive targets per XCD
    const int32_t *nodes;    // the nodes by depth, in depth-first order: those of depth d at
    const int *level;        // level[d * nblk] .. level[(d + 1) * nblk]
    int nblk;
    const int32_t *start;    // step 0: the boxes' roots, or null: the target `target`
    const int32_t *start_list;  // and their sources, nshift each
    int target, nstart, nshift;
    int64_t *dspan;          // per node, its down list
    int2 *heavy;             // targets put off to a launch of their own, and their parents; null: none are
    int32_t *out[kOut];      // P2P, M2L and down lists
    int64_t room[kOut];      // entries they hold
    int64_t chunk[kOut];     // list space taken at a time (0: a target's outputs exactly)
    int64_t *p2p_span, *m2l_span;  // per leaf / cell
};

// The room a list of n entries needs where it is handed out in chunks: a chunk is left
// with at most an eighth of it unused (take), and every workgroup may hold one
static int64_t list_room(int64_t n, int64_t chunk) { return chunk ? n + n / 7 + kWalkBlocks * chunk + 1 : n; }

struct Target {
    CellGeom g;
    double L;  // its box's length
    int cell, nleaf;
    bool leaf;
};

__device__ __forceinline__ int decide(const WalkArgs &a, const Target &t, const CellGeom &R, int cell, int sid)
{
    const bool bleaf = cell < t.nleaf;
    if (sid == 0 && cell == t.cell) return t.leaf ? kActP2P : kActSelfNode;
    if (t.leaf && bleaf) return kActP2P;  // leaf-leaf pairs are always P2P
    double sx = 0.0, sy = 0.0, sz = 0.0;
    if (sid != 0) shift_of(sid, t.L, sx, sy, sz);
    const double d0 = t.g.c[0] - (R.c[0] + sx);
    const double d1 = t.g.c[1] - (R.c[1] + sy);
    const double d2 = t.g.c[2] - (R.c[2] + sz);
    const int flag = mac(t.g.w, R.w, d0, d1, d2, a.theta2, a.rc2);
    if (flag < 0) return kActNone;
    bool pruned = false;
    if (sid != 0 && !bleaf) {
        const double L = t.L;
        const CellGeom box = {{0.5 * L, 0.5 * L, 0.5 * L}, {L, L, L}};
        pruned = let_pruned(box, R, sx, sy, sz, a.rc, a.theta);
    }
    // accepted; in the image walk a target leaf against a pruned node takes M2L whatever
    // the acceptance says (src/remotes.c:442)
    if (flag == 1 || (t.leaf && pruned)) return kActM2L;
    if (t.leaf) return kActOpenB;
    if (bleaf) return kActOpenA;
    const bool bigger = (t.g.w[0] + t.g.w[1] + t.g.w[2]) > (R.w[0] + R.w[1] + R.w[2]);
    return (bigger || pruned) ? kActOpenA : kActOpenB;  // ties open the source
}

// A window of a target's sources in LDS.  Items 0 .. cnt - 1 are the sources, the ones
// after them the children of opened items, level by level, two and two.  A settled item
// has one output or none: a list entry of kind X (P2P for a target leaf, down for a target
// node: a target has only one of them) or M2L.  An item's word holds its kind in the top 4
// bits and below it, 14 bits each, X and M2L: the outputs of the item and its children,
// then the position of the first.
enum : uint32_t { kKindNone = 0u, kKindX = 1u, kKindM2L = 2u, kForced = 3u, kOpened = 4u };  // kForced: X before any rule
constexpr int kPosBits = 14;
constexpr uint32_t kPosMask = (1u << kPosBits) - 1u, kOutMask = (1u << 2 * kPosBits) - 1u;
__device__ __forceinline__ uint32_t item_kind(uint32_t w) { return w >> 28; }

template <int NW, int CAP>
struct Window {
    static constexpr int TH = 64 * NW;
    static constexpr int WIN = CAP / 2;  // sources taken at a time
    static_assert(CAP < 1 << kPosBits, "a window's items, and so its outputs, fit their fields");
    int32_t entry[CAP];  // an opened item's: its first child
    uint32_t word[CAP];
    uint16_t level[kMaxDepth + 8];  // first item of each level
    int added[3];        // children of the current level (by level modulo 3)
    uint32_t wsum[NW];
    int32_t pend[kMaxDepth + 8];  // sources taken apart, the next one last
    int64_t at[2], left[2];  // where the target's outputs go (X, M2L); the room there
    int unit;            // the next target that was put off
    int64_t held[kOut][2];  // list space held: next entry, end
};
// a value that is the same in every lane, in scalar registers
__device__ __forceinline__ int64_t scalar(int64_t v)
{
    return (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)v) |
                     (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32);
}
__device__ __forceinline__ double scalar(double v) { return __longlong_as_double(scalar((int64_t)__double_as_longlong(v))); }

struct Found {
    int items, levels;
};

// Items 0 .. cnt - 1 (stored, not yet visible to the other threads) settled, with all that
// opening them brings in; false: more items than fit
template <int NW, int CAP>
__device__ __forceinline__ bool expand(const WalkArgs &a, const Target &t, Window<NW, CAP> &w, int cnt, Found &f)
{
    constexpr int TH = Window<NW, CAP>::TH;
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const uint64_t below = (1ull << lane) - 1ull;
    if (tid == 0) w.added[0] = 0;
    __syncthreads();
    int lo = 0, hi = cnt;
    for (int l = 0; lo < hi; l++) {
        if (tid == 0) {
            w.level[l] = (uint16_t)lo;
            w.level[l + 1] = (uint16_t)hi;
            w.added[(l + 1) % 3] = 0;  // the last level read [(l - 1) % 3]
        }
        for (int i0 = lo + 64 * wave; i0 < hi; i0 += TH) {  // the same for the whole wavefront
            const int i = i0 + lane;
            int act = kActNone, sid = 0;
            int4 k{};
            if (i < hi) {
                const int32_t e = w.entry[i];
                const int cell = entry_cell(e);
                sid = entry_shift(e);
                if (item_kind(w.word[i]) == kForced) {
                    act = kActOpenA;
                } else if (t.leaf && cell < t.nleaf) {
                    act = kActP2P;
                } else {
                    const WalkRec *R = a.rec + cell;
                    const CellGeom g = R->g;
                    k = *reinterpret_cast<const int4 *>(R->kid);
                    act = decide(a, t, g, cell, sid);
                }
            }
            const bool self = act == kActSelfNode, open = act == kActOpenB || self;
            const uint64_t bo = __ballot(open);
            int slot = 0;
            if (bo) {
                if (lane == 0) slot = atomicAdd(&w.added[l % 3], 2 * __popcll(bo));
                slot = hi + __builtin_amdgcn_readfirstlane(slot) + 2 * __popcll(bo & below);
            }
            if (i < hi) {
                const bool x = act == kActP2P || act == kActOpenA, m = act == kActM2L;
                if (open) {
                    if (slot + 2 <= CAP) {
                        // a node with itself passes its sons down, the first one first
                        const bool sw = self && k.z != 0;
                        w.entry[slot] = pack_entry(sw ? k.y : k.x, sid);
                        w.entry[slot + 1] = pack_entry(sw ? k.x : k.y, sid);
                        w.word[slot] = w.word[slot + 1] = self ? kForced << 28 : 0u;
                        w.entry[i] = slot;
                    }
                    w.word[i] = kOpened << 28;
                } else {
                    w.word[i] = x ? kKindX << 28 | 1u : m ? kKindM2L << 28 | 1u << kPosBits : 0u;
                }
            }
        }
        __syncthreads();
        lo = hi;
        hi += w.added[l % 3];
        f.levels = l + 1;
        if (hi > CAP) {
            __syncthreads();  // (the caller writes what is still read here)
            return false;
        }
    }
    f.items = hi;
    return true;
}

// The window's outputs (packed): every item's added up over its children, the sources' then
// numbered in turn
template <int NW, int CAP>
__device__ __forceinline__ uint32_t count(Window<NW, CAP> &w, int cnt, const Found &f)
{
    constexpr int TH = Window<NW, CAP>::TH;
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    for (int l = f.levels - 2; l >= 0; l--) {
        for (int i = w.level[l] + tid; i < w.level[l + 1]; i += TH)
            if (item_kind(w.word[i]) == kOpened) {
                const int c = w.entry[i];
                w.word[i] = kOpened << 28 | ((w.word[c] & kOutMask) + (w.word[c + 1] & kOutMask));
            }
        __syncthreads();
    }
    // each thread numbers K consecutive sources (an odd number: no two lanes in one bank)
    const int K = ((cnt + TH - 1) / TH) | 1, i0 = min(tid * K, cnt), i1 = min(i0 + K, cnt);
    uint32_t sum = 0;
    for (int i = i0; i < i1; i++) sum += w.word[i] & kOutMask;
    uint32_t incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(incl, o, 64);
        if (lane >= o) incl += y;
    }
    if (lane == 63) w.wsum[wave] = incl;
    __syncthreads();
    uint32_t run = incl - sum, all = 0;
#pragma unroll
    for (int k = 0; k < NW; k++) {
        const uint32_t s = w.wsum[k];
        run += k < wave ? s : 0u;
        all += s;
    }
    for (int i = i0; i < i1; i++) {
        const uint32_t word = w.word[i];
        w.word[i] = (word & ~kOutMask) | run;
        run += word & kOutMask;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(all);
}

// The settled items' positions, from their sources', and their entries stored there (after
// count): in the order of the walk from x and m on (null: not stored)
template <int NW, int CAP>
__device__ __forceinline__ void emit(Window<NW, CAP> &w, const Found &f, int32_t *__restrict__ x, int32_t *__restrict__ m)
{
    for (int l = 0; l < f.levels; l++) {
        for (int i = w.level[l] + (int)threadIdx.x; i < w.level[l + 1]; i += Window<NW, CAP>::TH) {
            const uint32_t k = item_kind(w.word[i]), p = w.word[i] & kOutMask;
            const int32_t entry = w.entry[i];
            if (k == kOpened) {
                const uint32_t c0 = w.word[entry], c1 = w.word[entry + 1];
                w.word[entry] = (c0 & ~kOutMask) | p;
                w.word[entry + 1] = (c1 & ~kOutMask) | (p + (c0 & kOutMask));
            } else if (k == kKindX) {
                if (x) x[p & kPosMask] = entry;
            } else if (k == kKindM2L) {
                if (m) m[p >> kPosBits] = entry;
            }
        }
        if (l + 1 < f.levels) __syncthreads();
    }
}

// n entries of list space (one thread), or -1: there is none left
__device__ __forceinline__ int64_t take(const WalkArgs &a, int list, int64_t n)
{
    if (n == 0) return 0;
    const int64_t at = (int64_t)atomicAdd(&a.st->next[list][0], (unsigned long long)n);
    if (at + n <= a.room[list]) return at;
    atomicOr(&a.st->overflow, (int)(list == kP2P ? kOvfP2P : list == kM2L ? kOvfM2L : kOvfDown));
    return -1;
}

// One step of the walk, a workgroup of NW wavefronts per target: the start targets, the
// nodes of a depth, or all leaves.  A leaf passes nothing down, so that the leaves wait for
// the last depth and are taken in one launch: the ones beside a dense cluster, with
// thousands of entries each, are then waited for once and not at every depth (128^3
// clustered particles: walk 15.4 -> 6.4 ms).  Targets of long lists, and those whose items
// do not fit, are put off to a launch of wider workgroups (heavy_only).  XCD x takes every
// eighth tile of targets (in depth-first order: neighbours share their sources).
// STORE = false counts the step's outputs (an ordinary evaluation sizes its lists by them).
//
// What bounds it: a box of few cells, the chain of dependent loads and barriers of one step
// (12 us) times the depths; a large one, latency too: 65% of the wavefronts' cycles are
// waits.  The windows leave a CU 18 wavefronts of the narrow workgroups (17 KB each) and 24 of
// the wide ones (two of half the LDS).  Against the walk it replaces (two passes over the
// traversals of single lanes, a dozen launches per depth): 16^3 clustered particles 0.68 ->
// 0.20 ms, 64^3 1.56 -> 0.71, 10^6 uniform ones 1.39 -> 0.65, 128^3 clustered 6.1 -> 3.3, 256^3
// 35.8 -> 23.1 ms.
template <int NW, int CAP, int EU, bool STORE>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(EU))) k_walk_step(WalkArgs a)
{
    constexpr int WIN = Window<NW, CAP>::WIN, TH = Window<NW, CAP>::TH;
    __shared__ Window<NW, CAP> w;
    if (a.sz->overflow) return;  // not written by this kernel: the same for every thread
    const int tid = threadIdx.x;
    const int nleaf = a.sz->nleaf;
    const int first = a.step > 0 ? a.level[(a.step - 1) * a.nblk] : 0;
    const int nunit = a.step > 0 ? 2 * (a.level[a.step * a.nblk] - first)
                                 : a.step == kLeaves ? nleaf : a.nstart;
    const int slot = max(a.step, 0);
    const int nheavy = a.heavy_only ? a.st->heavy[slot][STORE] : 0;
    const int x0 = (int)(blockIdx.x % kXcds);
    if (STORE && tid < 2 * kOut) w.held[tid / 2][tid % 2] = a.st->chunk[blockIdx.x][tid / 2][tid % 2];
    wave_sync();  // (thread 0 reads them)
    uint64_t total[kOut] = {};  // thread 0's
    for (int i = (int)(blockIdx.x / kXcds);; i += (int)(gridDim.x / kXcds)) {
        int u;
        if (a.heavy_only) {
            __syncthreads();
            if (tid == 0) w.unit = atomicAdd(&a.st->taken[slot][STORE], 1);
            __syncthreads();
            u = __builtin_amdgcn_readfirstlane(w.unit);
            if (u >= nheavy) break;
        } else {
            const int64_t at = ((int64_t)(i / a.tile) * kXcds + x0) * a.tile;  // the tile's first target
            if (at >= nunit) break;
            u = (int)at + i % a.tile;
            if (u >= nunit) continue;
        }
        Target t;
        int parent = -1;
        int64_t b, e;
        const int32_t *src = a.out[kDown];
        if (a.step == 0) {
            t.cell = a.start ? a.start[u] : a.target;
            src = a.start_list;
            b = (int64_t)u * a.nshift;
            e = b + a.nshift;
        } else {
            int v;
            if (a.heavy_only) {
                t.cell = a.heavy[u].x;
                v = a.heavy[u].y;
            } else if (a.step > 0) {
                v = a.nodes[first + u / 2];
                t.cell = a.rec[v].kid[u % 2];
                if (t.cell < nleaf) continue;
            } else {
                t.cell = u;
                v = a.rec[t.cell].kid[0];
                if (v < 0) continue;
            }
            parent = v;
            b = a.dspan[2 * (size_t)(v - nleaf)];
            e = a.dspan[2 * (size_t)(v - nleaf) + 1];
        }
        if (b >= e) continue;
        b = scalar(b);
        e = scalar(e);
        t.cell = __builtin_amdgcn_readfirstlane(t.cell);
        const WalkRec *R = a.rec + t.cell;
        for (int k = 0; k < 3; k++) {
            t.g.c[k] = scalar(R->g.c[k]);
            t.g.w[k] = scalar(R->g.w[k]);
        }
        t.L = scalar(a.box_len[R->box]);
        t.nleaf = nleaf;
        t.leaf = t.cell < nleaf;
        const int X = t.leaf ? kP2P : kDown;
        const bool once = a.heavy && !a.heavy_only && a.step != 0;
        // the outputs go to the list space the workgroup holds, if they fit it; an eighth of a
        // chunk left is given up for a new one
        bool ahead = STORE && a.chunk[X] > 0;
        if (ahead && tid == 0)
            for (int k = 0; k < 2; k++) {
                const int list = k ? (int)kM2L : X;
                int64_t (&held)[2] = w.held[list];
                if (8 * (held[1] - held[0]) < a.chunk[list]) {
                    held[0] = take(a, list, a.chunk[list]);
                    held[1] = held[0] + a.chunk[list];
                    if (held[0] < 0) held[0] = held[1] = 0;  // none left
                }
                w.at[k] = held[0];
                w.left[k] = held[1] - held[0];
            }
        uint64_t nx = 0, nm = 0;
        bool put_off = once && e - b > (a.step == kLeaves ? 4 : 1) * WIN;
        for (int pass = 0; pass < 2 && !put_off; pass++) {
            // Windows of the list.  One whose items do not fit is halved, and the next one is
            // as wide as its items would then fill three quarters of the space; a single
            // source whose items do not fit is taken apart, its two children taking its
            // place.
            int64_t b0 = b;
            int win = WIN, np = 0;
            int32_t *x = nullptr, *m = nullptr;
            if (pass) {
                x = w.at[0] < 0 ? nullptr : a.out[X] + w.at[0];
                m = w.at[1] < 0 ? nullptr : a.out[kM2L] + w.at[1];
            }
            bool whole = false;
            Found f;
            while (np > 0 || b0 < e) {
                int cnt = 1;
                if (np > 0) {
                    if (tid == 0) {
                        w.entry[0] = w.pend[np - 1];
                        w.word[0] = 0u;
                    }
                } else {
                    cnt = (int)min((int64_t)win, e - b0);
                    for (int k = tid; k < cnt; k += TH) {
                        w.entry[k] = src[b0 + k];
                        w.word[k] = 0u;
                    }
                }
                if (!expand<NW, CAP>(a, t, w, cnt, f)) {
                    put_off = once;
                    if (put_off) break;
                    if (cnt > 1) {
                        win = cnt / 2;
                        continue;
                    }
                    // (its item holds a child by now)
                    const int32_t s = np > 0 ? w.pend[np - 1] : src[b0];
                    const WalkRec *S = a.rec + entry_cell(s);
                    if (np > 0) np--;
                    else b0++;
                    __syncthreads();
                    if (tid == 0) {
                        w.pend[np] = pack_entry(S->kid[1], entry_shift(s));
                        w.pend[np + 1] = pack_entry(S->kid[0], entry_shift(s));
                    }
                    np += 2;
                    __syncthreads();
                    continue;
                }
                const uint32_t n = count<NW, CAP>(w, cnt, f);
                const uint32_t wx = n & kPosMask, wm = n >> kPosBits;
                whole = np == 0 && cnt == e - b;
                if (pass) {
                    emit<NW, CAP>(w, f, x, m);
                    if (x) x += wx;
                    if (m) m += wm;
                } else {
                    if (ahead) {
                        ahead = (int64_t)(nx + wx) <= w.left[0] && (int64_t)(nm + wm) <= w.left[1];
                        if (ahead) emit<NW, CAP>(w, f, a.out[X] + w.at[0] + nx, a.out[kM2L] + w.at[1] + nm);
                    }
                    nx += wx;
                    nm += wm;
                }
                if (np > 0) {
                    np--;
                } else {
                    b0 += cnt;
                    win = max(min(3 * CAP / 4 * cnt / f.items, WIN), 1);
                }
                if (!whole) __syncthreads();  // the window is used again
            }
            if (put_off || !STORE || pass) break;
            // the target's list space: what it filled already, or its outputs exactly
            __syncthreads();  // (w.at is read above)
            if (tid == 0) {
                const int64_t n[2] = {(int64_t)nx, (int64_t)nm};
                for (int k = 0; k < 2; k++) {
                    if (ahead) w.held[k ? (int)kM2L : X][0] += n[k];
                    else w.at[k] = take(a, k ? (int)kM2L : X, n[k]);
                    int64_t *span = k ? a.m2l_span + 2 * (size_t)t.cell
                                      : t.leaf ? a.p2p_span + 2 * (size_t)t.cell : a.dspan + 2 * (size_t)(t.cell - nleaf);
                    span[0] = max(w.at[k], (int64_t)0);
                    span[1] = w.at[k] < 0 ? 0 : w.at[k] + n[k];
                }
            }
            if (ahead) break;
            __syncthreads();
            if (whole) {  // still in its window
                emit<NW, CAP>(w, f, w.at[0] < 0 ? nullptr : a.out[X] + w.at[0], w.at[1] < 0 ? nullptr : a.out[kM2L] + w.at[1]);
                break;
            }
        }
        if (tid == 0) {
            if (put_off) {
                a.heavy[atomicAdd(&a.st->heavy[slot][STORE], 1)] = int2{t.cell, parent};
            } else {
                total[kM2L] += nm;
                if (t.leaf) total[kP2P] += nx;
                else total[kDown] += nx;
            }
        }
        __syncthreads();  // the window is used again
    }
    __syncthreads();
    if (STORE && tid < 2 * kOut) a.st->chunk[blockIdx.x][tid / 2][tid % 2] = w.held[tid / 2][tid % 2];
    if (tid == 0)
        for (int k = 0; k < kOut; k++)
            if (total[k]) atomicAdd(&a.st->count[STORE ? 0 : 1][k][blockIdx.x % kCountSlots], (unsigned long long)total[k]);
}

// After the last step: the lists' lengths, and what exceeds the capacities.
__global__ void k_walk_end(DevSizes *sz, const WalkState *__restrict__ st, int64_t p2p_cap, int64_t m2l_cap,
                           int64_t dl_cap)
{
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const int64_t cap[kOut] = {p2p_cap, m2l_cap, dl_cap};
    const int bit[kOut] = {kOvfP2P, kOvfM2L, kOvfDown};
    int64_t n[kOut] = {};
    int ovf = sz->overflow | st->overflow;
#pragma unroll
    for (int k = 0; k < kOut; k++) {
#pragma unroll
        for (int i = 0; i < kCountSlots; i++) n[k] += (int64_t)st->count[0][k][i];
        if (n[k] > cap[k]) ovf |= bit[k];
    }
    sz->overflow = ovf;
    sz->n_p2p = ovf ? 0 : n[kP2P];
    sz->n_m2l = ovf ? 0 : n[kM2L];
}

// The cells' records; every span empty (cells a walk from a given pair never reaches keep
// no entries); the walk's state cleared; the nodes of each depth counted per block of 256
// cells (hist[depth][block]).  n: the launch bound of the cells, nl, nn: of leaves and nodes.
constexpr int kLevelTile = 256;

__global__ void __launch_bounds__(kLevelTile) k_walk_records(DevSizes *__restrict__ sz, const CellInfo *__restrict__ info,
                                                             const CellGeom *__restrict__ geom,
                                                             const int *__restrict__ cell_box, int n, int nl, int nn,
                                                             WalkRec *__restrict__ rec, int64_t *__restrict__ p2p_span,
                                                             int64_t *__restrict__ m2l_span,
                                                             int64_t *__restrict__ dspan, uint64_t *__restrict__ state,
                                                             int ndepth, int *__restrict__ hist)
{
    __shared__ int cnt[256];
    const int c = blockIdx.x * kLevelTile + threadIdx.x;
    cnt[threadIdx.x] = 0;
    for (size_t i = (size_t)c; i < sizeof(WalkState) / 8; i += (size_t)gridDim.x * kLevelTile) state[i] = 0;
    if (c < n) {
        m2l_span[2 * (size_t)c] = m2l_span[2 * (size_t)c + 1] = 0;
        if (c < nl) p2p_span[2 * (size_t)c] = p2p_span[2 * (size_t)c + 1] = 0;
        if (c < nn) dspan[2 * (size_t)c] = dspan[2 * (size_t)c + 1] = 0;
    }
    __syncthreads();
    // an overflowed tree's cells were not written, and nothing is read of them
    if (!sz->overflow && c < sz->ncell) {
        const CellInfo I = info[c];
        WalkRec R;
        R.g = geom[c];
        R.box = cell_box[c];
        R.kid[0] = R.kid[1] = -1;
        R.swap = 0;
        if (I.son0 >= 0) {
            const bool first0 = info[I.son0].dfs == I.dfs + 1;
            R.kid[0] = first0 ? I.son0 : I.son1;
            R.kid[1] = first0 ? I.son1 : I.son0;
            R.swap = first0 ? 0 : 1;
            if (I.depth < ndepth) atomicAdd(&cnt[I.depth], 1);
        } else {
            R.kid[0] = I.parent;
        }
        rec[c] = R;
    }
    __syncthreads();
    if ((int)threadIdx.x < ndepth) hist[threadIdx.x * gridDim.x + blockIdx.x] = cnt[threadIdx.x];
    if (blockIdx.x == 0 && threadIdx.x == 0) hist[ndepth * gridDim.x] = 0;
}

// The nodes by depth, each depth's in the order of their numbers (depth-first); a node of a
// depth that the plan has no step for overflows it.  The start lists: every box's root
// (box_root given) or the source B, once per shift in [shift_lo, shift_hi).
__global__ void __launch_bounds__(kLevelTile) k_walk_levels(const DevSizes *__restrict__ sz, const CellInfo *__restrict__ info,
                                                            int ndepth, const int *__restrict__ base,
                                                            int32_t *__restrict__ nodes, WalkState *__restrict__ st,
                                                            int32_t *__restrict__ start, const int *__restrict__ box_root,
                                                            int nbox, int B, int shift_lo, int nshift)
{
    __shared__ int wcnt[kLevelTile / 64][256];
    if (sz->overflow) return;
    const int c = blockIdx.x * kLevelTile + threadIdx.x, lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    for (int i = c; i < nbox * nshift; i += gridDim.x * kLevelTile)
        start[i] = pack_entry(box_root ? box_root[i / nshift] : B, shift_lo + i % nshift);
    for (int k = 0; k < kLevelTile / 64; k++) wcnt[k][threadIdx.x] = 0;
    __syncthreads();
    int depth = -1;
    if (c < sz->ncell && c >= sz->nleaf) depth = info[c].depth;
    if (depth >= ndepth) {
        atomicOr(&st->overflow, (int)kOvfDepths);
        depth = -1;
    }
    uint64_t same = __ballot(depth >= 0);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const uint64_t bk = __ballot((depth >> k) & 1);
        same &= (depth >> k) & 1 ? bk : ~bk;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    if (depth >= 0 && rank == 0) wcnt[wave][depth] = __popcll(same);
    __syncthreads();
    if (depth < 0) return;
    int at = base[depth * gridDim.x + blockIdx.x] + rank;
    for (int k = 0; k < wave; k++) at += wcnt[k][depth];
    nodes[at] = c;
}
static_assert(kMaxDepth <= 256, "a block counts 256 depths");

// ---------------------------------------------------------------------------- host side

// grow to `need` bytes keeping the first `keep` bytes
static void *grow_keep(DevBuf &b, size_t need, size_t keep, hipStream_t st)
{
    if (need <= b.cap) return b.p;
    const size_t want = need + need / (arena_active() ? 4 : 2);
    void *nw = dev_alloc(want);
    if (b.p && keep) PH_CHECK(hipMemcpyAsync(nw, b.p, keep, hipMemcpyDeviceToDevice, st));
    PH_CHECK(hipStreamSynchronize(st));
    dev_free(b.p);
    b.p = nw;
    b.cap = want;
    return nw;
}

// The workgroups of a step of at most `units` targets.  A step of few targets is bound by
// the latency of one after the other, and takes workgroups of 8 wavefronts; one of many by
// the number of loads in flight, and takes 2 wavefronts per target (nodes of 256^3
// clustered particles with 1, 2 and 4 wavefronts: 15.8, 10.7 and 12.1 ms), up to
// kWalkBlocks workgroups of them.  What those put off goes to 12 wavefronts with half a
// CU's LDS each: a list taken in one window is expanded once, in several often twice (100,003
// particles in leaves of 8, half of them in one cluster, with 4096, 6144, 7680 and 9408
// items: walk 4.5, 3.0, 2.5 and 2.2 ms).
constexpr int kWideUnits = 512, kHeavyBlocks = 512;
// Walks of more cells put heavy targets off and take list space by chunks
constexpr int kSmallWalk = 8192;

template <bool STORE>
static void launch_step(WalkArgs &a, int step, int64_t units, hipStream_t st)
{
    a.step = step;
    a.heavy_only = false;
    const int grid = (int)std::min<int64_t>(kWalkBlocks, (units + 2 * kXcds - 1) / (2 * kXcds) * (2 * kXcds));
    a.tile = units <= kWalkBlocks ? 2 : 64;
    if (units <= kWideUnits) {
        int2 *const heavy = a.heavy;
        a.heavy = nullptr;  // none put off
        k_walk_step<8, 4096, 4, STORE><<<grid, 512, 0, st>>>(a);
        a.heavy = heavy;
        return;
    }
    k_walk_step<2, 1920, 5, STORE><<<grid, 128, 0, st>>>(a);
    if (!a.heavy || step == 0) return;  // (of the start targets none are put off)
    a.heavy_only = true;
    k_walk_step<12, 9408, 6, STORE><<<kHeavyBlocks, 768, 0, st>>>(a);
}

// The walk from the pair (start_target, start_source) over the shifts [shift_lo, shift_hi),
// or from every box's (root, root) when start_target < 0.  One step for the start targets,
// one per depth of nodes for their children; an ordinary evaluation counts each step's
// outputs first and reads the three totals to size the lists.
void run_walk_from(Ctx &c, int shift_lo, int shift_hi, int start_target, int start_source)
{
    hipStream_t st = c.stream;
    const bool planned = c.plan.active;
    const int nlb = nleaf_bound(c), ncb = ncell_bound(c), nnb = std::max(1, nnode_bound(c));
    if (ncb >= (1 << 27)) throw std::runtime_error("more than 2^27 cells");
    need(c.cell_box, sizeof(int) * (size_t)ncb, "cell boxes");
    const bool forest = start_target < 0;
    if (planned && !forest) throw std::runtime_error("a planned walk starts from the roots");
    const int nshift = shift_hi - shift_lo, nstart = forest ? c.nbox : 1;
    const int64_t n0 = (int64_t)nstart * nshift;
    if (forest) need(c.d_box_root, sizeof(int) * (size_t)c.nbox, "box roots");
    // depths that hold nodes: the plan's, or the tree's
    const int ndepth = planned ? c.plan.depths - 1 : c.nlevel;

    DevSizes *sz = dptr<DevSizes>(c.sizes);
    WalkArgs a{};
    a.sz = sz;
    a.box_len = dptr<double>(c.d_box_len);
    a.theta = c.prm.theta;
    a.theta2 = c.prm.theta * c.prm.theta;
    a.rc = c.prm.rc;
    a.rc2 = c.prm.rc * c.prm.rc;
    a.nblk = (ncb + kLevelTile - 1) / kLevelTile;
    const int nhist = ndepth * a.nblk + 1;
    WalkRec *rec = static_cast<WalkRec *>(ctx_buf(c, c.walk_rec, sizeof(WalkRec) * (size_t)ncb, "walk records"));
    a.p2p_span = static_cast<int64_t *>(ctx_buf(c, c.p2p_off, sizeof(int64_t) * 2 * (size_t)std::max(1, nlb), "P2P list"));
    a.m2l_span = static_cast<int64_t *>(ctx_buf(c, c.m2l_off, sizeof(int64_t) * 2 * (size_t)ncb, "M2L list"));
    a.dspan = static_cast<int64_t *>(ctx_buf(c, c.walk_dspan, sizeof(int64_t) * 2 * (size_t)nnb, "walk spans"));
    a.st = static_cast<WalkState *>(ctx_buf(c, c.walk_state, sizeof(WalkState), "walk state"));
    int *hist = static_cast<int *>(ctx_buf(c, c.walk_hist, sizeof(int) * 2 * (size_t)nhist, "walk levels"));
    int32_t *nodes = static_cast<int32_t *>(ctx_buf(c, c.walk_nodes, sizeof(int32_t) * (size_t)nnb, "walk levels"));
    k_walk_records<<<a.nblk, kLevelTile, 0, st>>>(sz, dptr<CellInfo>(c.info), dptr<CellGeom>(c.geom),
                                                  dptr<int>(c.cell_box), ncb, nlb, nnb, rec, a.p2p_span, a.m2l_span,
                                                  a.dspan, reinterpret_cast<uint64_t *>(a.st), ndepth, hist);
    {
        size_t bytes = 0;
        PH_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, hist, hist + nhist, nhist, st));
        void *tmp = scan_storage(c, bytes);
        PH_CHECK(hipcub::DeviceScan::ExclusiveSum(tmp, bytes, hist, hist + nhist, nhist, st));
    }
    // List space by chunks: a small box's targets take theirs exactly (some thousand
    // additions to one counter take some 10 us), larger ones in proportion to their cells
    int64_t chunk = 0;
    if (ncb > kSmallWalk && !arena_active())
        for (chunk = 1024; chunk < 16384 && 16 * chunk < ncb; chunk *= 2) {}
    a.chunk[kP2P] = chunk;
    a.chunk[kM2L] = chunk / 4;
    a.chunk[kDown] = chunk / 4;
    int32_t *start = static_cast<int32_t *>(ctx_buf(c, c.walk_start, sizeof(int32_t) * (size_t)n0, "walk start"));
    if (ncb > kSmallWalk)
        a.heavy = static_cast<int2 *>(ctx_buf(c, c.walk_heavy, sizeof(int2) * (size_t)std::max(nlb, nnb), "walk targets"));
    const int *roots = forest ? dptr<int>(c.d_box_root) : nullptr;
    k_walk_levels<<<a.nblk, kLevelTile, 0, st>>>(sz, dptr<CellInfo>(c.info), ndepth, hist + nhist, nodes, a.st, start,
                                                 roots, nstart, start_source, shift_lo, nshift);
    a.rec = rec;
    a.nodes = nodes;
    a.level = hist + nhist;
    a.start = roots;
    a.start_list = start;
    a.target = start_target;
    a.nstart = nstart;
    a.nshift = nshift;

    DevBuf *list[kOut] = {&c.p2p_src, &c.m2l_src, &c.walk_down};
    int64_t cap[kOut] = {c.plan.p2p_cap, c.plan.m2l_cap, c.plan.dl_cap};  // an ordinary walk's: what it counts
    if (!planned)
        for (int k = 0; k < kOut; k++) cap[k] = 0;
    // makes room for cap[] entries; an ordinary walk's lists keep what they hold (held[])
    auto make_room = [&](const int64_t (&held)[kOut]) {
        for (int k = 0; k < kOut; k++) {
            a.room[k] = list_room(cap[k], a.chunk[k]);
            const size_t bytes = 4 * (size_t)std::max<int64_t>(a.room[k], 1);
            if (planned) ctx_buf(c, *list[k], bytes, k == kP2P ? "P2P list" : k == kM2L ? "M2L list" : "down lists");
            else grow_keep(*list[k], bytes, held[k] ? 4 * (size_t)list_room(held[k], a.chunk[k]) : 0, st);
            a.out[k] = dptr<int32_t>(*list[k]);
        }
    };
    make_room({0, 0, 0});
    // a step's outputs counted ahead (by `count`) and room made for them
    auto count_ahead = [&](auto count) {
        count();
        constexpr size_t words = kOut * kCountSlots;
        unsigned long long *pin = reinterpret_cast<unsigned long long *>(c.pinned.p);
        PH_CHECK(hipMemcpyAsync(pin, a.st->count[1], 8 * words, hipMemcpyDeviceToHost, st));
        PH_CHECK(hipEventRecord(c.counts_ready, st));
        PH_CHECK(hipEventSynchronize(c.counts_ready));
        int64_t held[kOut];
        for (int k = 0; k < kOut; k++) {
            held[k] = cap[k];
            cap[k] = 0;
        }
        for (size_t k = 0; k < words; k++) cap[k / kCountSlots] += (int64_t)pin[k];
        make_room(held);
    };
    // a walk from a given cell: its children's depth is the next one with targets
    int next = 1;
    if (!forest) {
        CellInfo *pin = reinterpret_cast<CellInfo *>(c.pinned.p);
        PH_CHECK(hipMemcpyAsync(pin, dptr<CellInfo>(c.info) + start_target, sizeof(CellInfo), hipMemcpyDeviceToHost, st));
        PH_CHECK(hipStreamSynchronize(st));
        next = pin->depth + 1;
    }
    for (int d = 0; d <= ndepth; d = d == 0 ? next : d + 1) {
        const int64_t units = d == 0 ? nstart
                                     : 2 * std::min<int64_t>(nnb, d < 32 ? (int64_t)nstart << (d - 1) : (int64_t)nnb);
        const int64_t down = cap[kDown];
        if (!planned) count_ahead([&] { launch_step<false>(a, d, units, st); });
        launch_step<true>(a, d, units, st);
        if (!planned && cap[kDown] == down) break;  // nothing passed down: no targets below
    }
    if (planned || cap[kDown] > 0) {
        if (!planned) count_ahead([&] { launch_step<false>(a, kLeaves, nlb, st); });
        launch_step<true>(a, kLeaves, nlb, st);
    }
    k_walk_end<<<1, 1, 0, st>>>(sz, a.st, cap[kP2P], cap[kM2L], cap[kDown]);
    if (!planned) {
        c.n_p2p = cap[kP2P];
        c.n_m2l = cap[kM2L];
        if (forest) {
            Measure &m = c.meas;
            m.depths = ndepth + 1;
            m.dl = cap[kDown];
            m.p2p = c.n_p2p;
            m.m2l = c.n_m2l;
        }
    }
    c.lists_valid = true;
    PH_CHECK(hipGetLastError());
}

void run_walk(Ctx &c, int shift_lo, int shift_hi) { run_walk_from(c, shift_lo, shift_hi, -1, -1); }

}  // namespace photons
