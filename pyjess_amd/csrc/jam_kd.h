// jam_kd.h -- kd-tree leaf order of every candidate set, on gfx950.
//
// The reference builds one kd-tree per candidate set (KdTree_create,
// patches/KdTree.c.patch:348-451): the root splits the set at its median on
// x, the children on y, then z, ..., each median found by QuickSelect
// (qselect_r, patches/qselect.h.patch:50-116): median-of-three pivot at
// mid = (l + r + 1) / 2 moved to r, Lomuto partition sending "<= pivot" to the
// left, pivot swapped into place, repeat on the side holding the median. The
// Join walks the tree depth first, right child first, so the order in which
// candidates are met -- and therefore the order of the hits -- is the tree's
// leaf order read backwards. The kernels here compute that order for every
// set and store the set in it (32-byte entries: x, y, z, chain, resSeq; and
// the atom index) with one bounding box per 64 consecutive entries, which the
// join uses for pruning.
//
// Two algorithms, both exact:
//   fast   when no range of the tree has equal coordinates on both sides of
//          its split point, the left half of every range is its n/2 smallest
//          elements whatever the arrangement, and the leaf order follows from
//          memberships alone: sort every axis once, then at level d cut each
//          range of axis d%3 in half and stably partition the two other axes
//          by side. Detects a tie across a split point and then gives up.
//   exact  all ranges of a tree level run their QuickSelect together, one
//          partition round at a time, and each Lomuto partition is computed
//          without its serial scan: the "<= pivot" elements keep their order
//          (a stable compaction), the others move as a FIFO queue (each is
//          pushed when scanned, and each "<=" element scanned after the first
//          ">" one pops the front and pushes it back), whose final contents
//          are found by following each push back to the element it started
//          as. Nearly as fast as the fast path's sorts, so only sets that
//          seldom have a tie (up to 128 entries of many molecules, and those
//          too large for LDS unless a sample of them has one) try the fast path first.
//
// Fast path: sets of up to 64 entries in one wave's registers, up to 128
// with one position per thread, above KD_LDS_MAX in global scratch. Exact
// path: up to KD_LDS_MAX entries in LDS, larger ones in global scratch. Every
// loop of an exact pass whose length depends on the data has a bound that a
// correct run never reaches; a pass that reaches it sets st.kd_err, and the
// query reports an error.
#pragma once

#include <hip/hip_runtime.h>

#include "jam_common.h"
#include "jam_wave.h"

namespace jam {

#define KD_BIG 1024
#define KD_TIERS 6
#ifndef KD_THREADS
#define KD_THREADS 256
#endif
// threads of the exact pass over a set larger than KD_LDS_MAX: its rounds are
// latency-bound loops over the positions, so more threads per set
#define KD_EXACT_THREADS 1024
// global scratch of sets larger than KD_LDS_MAX, per set entry (padded to a power
// of two for the fast path's sorts: 3 doubles, 9 ints and 1 byte per padded
// entry, at most 2 * 61 bytes per entry)
#define KD_SCRATCH_BYTES_PER_ENTRY 128

// size tier of a set: (0,64], (64,128], (128,256], (256,512], (512,1024],
// larger; -1 for an empty set
__host__ __device__ static inline int kd_tier(int n)
{
    if (n <= 0) return -1;
    if (n <= 64) return 0;
    if (n <= 128) return 1;
    if (n <= 256) return 2;
    if (n <= 512) return 3;
    if (n <= KD_BIG) return 4;
    return 5;
}

__device__ static inline int shfl_int(int v, int src) { return __shfl(v, src, JAM_WAVE); }

// lane `dst` receives v from this lane (ds_permute: push)
__device__ static inline int push_int(int v, int dst) { return __builtin_amdgcn_ds_permute(dst << 2, v); }

__device__ static inline bool key_less(double a, int ia, double b, int ib)
{
    return a < b || (a == b && ia < ib);
}

// Buckets the sets by size tier: bucket[k * n_sets + i] is the i-th set of
// tier k (in no particular order), nb[k] their number. Each workgroup takes
// one contiguous span of sets: it counts its sets per tier in LDS (one LDS
// atomic per wave and tier), reserves room in each tier's list with one
// global atomic per tier, then places its sets there.
#define KD_BUCKET_SPAN 4096
__global__ void __launch_bounds__(256) k_kdbucket(DevSets st, int *bucket, unsigned int *nb)
{
    __shared__ unsigned int cnt[KD_TIERS], base[KD_TIERS];
    const int lane = lane_id();
    const int t = threadIdx.x;
    for (long long s0 = (long long)blockIdx.x * KD_BUCKET_SPAN; s0 < st.n_sets;
         s0 += (long long)gridDim.x * KD_BUCKET_SPAN) {
        const long long s1 = min(s0 + (long long)KD_BUCKET_SPAN, (long long)st.n_sets);
        if (t < KD_TIERS) cnt[t] = 0u;
        __syncthreads();
        for (long long s = s0 + t; s - lane < s1; s += blockDim.x) {
            const int tier = s < s1 ? kd_tier(st.cnt[s]) : -1;
            for (int k = 0; k < KD_TIERS; k++) {
                const unsigned long long mask = ballot(tier == k);
                if (mask != 0ull && lane == first_bit(mask)) atomicAdd(&cnt[k], (unsigned int)__popcll(mask));
            }
        }
        __syncthreads();
        if (t < KD_TIERS) {
            base[t] = cnt[t] ? atomicAdd(&nb[t], cnt[t]) : 0u;
            cnt[t] = 0u;
        }
        __syncthreads();
        for (long long s = s0 + t; s - lane < s1; s += blockDim.x) {
            const int tier = s < s1 ? kd_tier(st.cnt[s]) : -1;
            for (int k = 0; k < KD_TIERS; k++) {
                const unsigned long long mask = ballot(tier == k);
                if (mask == 0ull) continue;
                const int leader = first_bit(mask);
                unsigned int off = 0u;
                if (lane == leader) off = atomicAdd(&cnt[k], (unsigned int)__popcll(mask));
                off = (unsigned int)shfl_int((int)off, leader);
                if (tier == k) bucket[(size_t)k * st.n_sets + base[k] + off + rank_below(mask)] = (int)s;
            }
        }
        __syncthreads();
    }
}

// Writes position p of set s (element e of its candidate list, p < n) and,
// with the other lanes of the wave holding positions p & ~63 ... p | 63, the
// bounding boxes of that 64-entry block and of its JAM_SUB-entry sub-blocks.
// Every lane of the wave calls it.
__device__ static inline void kd_emit_lane(const DevMols &ms, const DevSets &st, int s, int n, int64_t off,
                                           int abase, int p, int e)
{
    const bool ok = p < n;
    double x = 0.0, y = 0.0, z = 0.0;
    if (ok) {
        const int atom = st.list[off + e];
        const size_t g = (size_t)(abase + atom);
        x = ms.xyz[3 * g + 0];
        y = ms.xyz[3 * g + 1];
        z = ms.xyz[3 * g + 2];
        SetEnt en;
        en.x = x;
        en.y = y;
        en.z = z;
        en.ch = ms.chain[g];
        en.res = ms.resseq[g];
        st.kent[off + p] = en;
        st.katom[off + p] = atom;
        st.kidx[off + p] = e;
        st.l2k[off + e] = p;
    }
    double blo[3] = {ok ? x : INFINITY, ok ? y : INFINITY, ok ? z : INFINITY};
    double bhi[3] = {ok ? x : -INFINITY, ok ? y : -INFINITY, ok ? z : -INFINITY};
    // the box of each JAM_SUB entries, then of the 64
    for (int sh = JAM_SUB / 2; sh >= 1; sh >>= 1) {
#pragma unroll
        for (int q = 0; q < 3; q++) {
            blo[q] = fmin(blo[q], __shfl_xor(blo[q], sh, JAM_WAVE));
            bhi[q] = fmax(bhi[q], __shfl_xor(bhi[q], sh, JAM_WAVE));
        }
    }
    if ((p & (JAM_SUB - 1)) == 0 && p < n) {
        double *sb = st.sbox + 6 * (off / JAM_SUB + s + p / JAM_SUB);
        sb[0] = blo[0];
        sb[1] = blo[1];
        sb[2] = blo[2];
        sb[3] = bhi[0];
        sb[4] = bhi[1];
        sb[5] = bhi[2];
    }
    for (int sh = JAM_WAVE / 2; sh >= JAM_SUB; sh >>= 1) {
#pragma unroll
        for (int q = 0; q < 3; q++) {
            blo[q] = fmin(blo[q], __shfl_xor(blo[q], sh, JAM_WAVE));
            bhi[q] = fmax(bhi[q], __shfl_xor(bhi[q], sh, JAM_WAVE));
        }
    }
    const int b0 = p & ~(JAM_WAVE - 1);
    if ((p & (JAM_WAVE - 1)) == 0 && b0 < n) {
        double *bb = st.bbox + 6 * (off / JAM_WAVE + s + b0 / JAM_WAVE);
        bb[0] = blo[0];
        bb[1] = blo[1];
        bb[2] = blo[2];
        bb[3] = bhi[0];
        bb[4] = bhi[1];
        bb[5] = bhi[2];
    }
}

// ---------------------------------------------------------------------------
// fast path, sets of at most 64 entries: one wave, one element per lane,
// everything in registers
// ---------------------------------------------------------------------------

// Returns true (nothing written) when a tie straddles a split point.
__device__ static bool kd_wave64(const DevMols &ms, const DevSets &st, int s, int n, int64_t off, int abase)
{
    const int lane = lane_id();
    double c[3] = {INFINITY, INFINITY, INFINITY};
    if (lane < n) {
        const size_t g = (size_t)(abase + st.list[off + lane]);
        c[0] = ms.xyz[3 * g + 0];
        c[1] = ms.xyz[3 * g + 1];
        c[2] = ms.xyz[3 * g + 2];
    }
    // per axis: element at each position, sorted by (coordinate, element)
    int perm[3];
    for (int a = 0; a < 3; a++) {
        double key = c[a];
        int id = lane;
        for (int k = 2; k <= JAM_WAVE; k <<= 1) {
            for (int j = k >> 1; j > 0; j >>= 1) {
                const double ok = __shfl_xor(key, j, JAM_WAVE);
                const int oi = __shfl_xor(id, j, JAM_WAVE);
                const bool up = (lane & k) == 0;
                const bool lower = (lane & j) == 0;
                const bool other_less = key_less(ok, oi, key, id);
                // the lower lane of an ascending pair keeps the smaller key
                const bool take = (lower == up) ? other_less : !other_less;
                if (take) {
                    key = ok;
                    id = oi;
                }
            }
        }
        perm[a] = id;
    }
    int sb = 0, se = n;
    for (int d = 0;; d++) {
        const int a = d % 3;
        const bool act = lane < n && se - sb >= 2;
        const int m = sb + (se - sb) / 2;
        const bool split = act && lane == m;
        if (ballot(act) == 0ull) break;
        // tie across the split point: compare with the previous position
        const int pa = (a == 0) ? perm[0] : (a == 1) ? perm[1] : perm[2];
        const double ca = (a == 0) ? c[0] : (a == 1) ? c[1] : c[2];
        const double here = __shfl(ca, pa & 63, JAM_WAVE);
        const double prev = __shfl_up(here, 1, JAM_WAVE);
        if (ballot(split && prev == here) != 0ull) return true;
        // side of every element, delivered to the lane of the element id
        const int left_pos = act && lane < m ? 1 : 0;
        const int side_by_elem = push_int(left_pos, pa & 63);
        for (int b = 0; b < 3; b++) {
            if (b == a) continue;
            const int pb = (b == 0) ? perm[0] : (b == 1) ? perm[1] : perm[2];
            const int sd = shfl_int(side_by_elem, pb & 63);
            const unsigned long long lm = ballot(act && sd);
            int np = lane;
            if (act) {
                const unsigned long long below = (1ull << lane) - (1ull << sb);
                const int lc = __popcll(lm & below);
                np = sd ? sb + lc : m + (lane - sb - lc);
            }
            const int moved = push_int(pb, np);
            if (b == 0) perm[0] = lane < n ? moved : perm[0];
            else if (b == 1) perm[1] = lane < n ? moved : perm[1];
            else perm[2] = lane < n ? moved : perm[2];
        }
        if (act) {
            if (lane < m) se = m;
            else sb = m;
        }
    }
    // DFS order: position p holds element perm[n-1-p]
    const int src = n - 1 - lane;
    const int e = shfl_int(perm[0], src < 0 ? 0 : src);
    kd_emit_lane(ms, st, s, n, off, abase, lane, e);
    return false;
}

__global__ void __launch_bounds__(JAM_WAVE) k_kdwave(DevMols ms, DevTpls tp, DevSets st, const int *list,
                                                     const unsigned int *count, int *tied, unsigned int *n_tied)
{
    if (*st.total > st.cap) return;
    const int cnt = (int)*count;
    for (int q = blockIdx.x; q < cnt; q += gridDim.x) {
        const int s = list[q];
        const int n = st.cnt[s];
        const int64_t off = st.off[s];
        const int abase = ms.atom_off[s / tp.n_types];
        if (kd_wave64(ms, st, s, n, off, abase) && lane_id() == 0) tied[atomicAdd(n_tied, 1u)] = s;
    }
}

// ---------------------------------------------------------------------------
// fast path, sets of (NT/2, NT] entries (NT = 128 ... KD_BIG): one position
// per thread, the arrangement of every axis held in registers (position t:
// key and element); bitonic stages less than 64 positions apart by shuffles,
// the others through LDS; side flags and the stable partitions' prefix counts
// by ballots and one LDS word per wave
// ---------------------------------------------------------------------------

template <int NT>
__global__ void __launch_bounds__(NT) k_kdblock(DevMols ms, DevTpls tp, DevSets st, const int *list,
                                                const unsigned int *count, int *tied, unsigned int *n_tied)
{
    constexpr int NW = NT / JAM_WAVE;
    // the two axes other than a level's are partitioned together: one
    // exchange buffer and prefix array each
    __shared__ double xkey[NT], xkey2[NT];
    __shared__ int xid[NT], xid2[NT];
    __shared__ int xpre[NT], xpre2[NT];
    __shared__ int side[NT];
    __shared__ int wsum[NW], wsum2[NW];
    const int t = threadIdx.x;
    const int lane = lane_id();
    const int wv = t / JAM_WAVE;
    if (*st.total > st.cap) return;
    const int cnt = (int)*count;
    for (int q = blockIdx.x; q < cnt; q += gridDim.x) {
        const int s = list[q];
        const int n = st.cnt[s];
        const int64_t off = st.off[s];
        const int abase = ms.atom_off[s / tp.n_types];
        double c[3] = {INFINITY, INFINITY, INFINITY};
        if (t < n) {
            const size_t g = (size_t)(abase + st.list[off + t]);
            c[0] = ms.xyz[3 * g + 0];
            c[1] = ms.xyz[3 * g + 1];
            c[2] = ms.xyz[3 * g + 2];
        }
        // per axis: (key, element) at position t, sorted by (key, element);
        // positions n ... NT-1 hold padding elements with infinite keys
        double key[3];
        int id[3];
        // exchanges across waves go through LDS, the steps taking the two
        // buffer pairs in turn: a buffer is written again only after a
        // barrier that every read of it precedes, so one barrier a step
        bool second = false;
#pragma unroll
        for (int a = 0; a < 3; a++) {
            double k0 = c[a];
            int i0 = t;
            for (int k = 2; k <= NT; k <<= 1) {
                for (int j = k >> 1; j > 0; j >>= 1) {
                    double ok;
                    int oi;
                    if (j >= JAM_WAVE) {
                        double *bk = second ? xkey2 : xkey;
                        int *bi = second ? xid2 : xid;
                        second = !second;
                        bk[t] = k0;
                        bi[t] = i0;
                        __syncthreads();
                        ok = bk[t ^ j];
                        oi = bi[t ^ j];
                    } else {
                        ok = __shfl_xor(k0, j, JAM_WAVE);
                        oi = __shfl_xor(i0, j, JAM_WAVE);
                    }
                    const bool up = (t & k) == 0;
                    const bool lower = (t & j) == 0;
                    const bool other_less = key_less(ok, oi, k0, i0);
                    const bool take = (lower == up) ? other_less : !other_less;
                    if (take) {
                        k0 = ok;
                        i0 = oi;
                    }
                }
            }
            key[a] = k0;
            id[a] = i0;
        }
        // Per level, five barriers: the split side of every element; the tie
        // test folded into the publication of both axes' ballot counts;
        // their prefix counts; their stable partitions; and whether any
        // range is still open folded into the last.
        int sb = 0, se = n;
        bool tie = false;
        bool open = __syncthreads_or(t < n && n >= 2);
        for (int d = 0; open; d++) {
            const int a = d % 3;
            const int b1 = a == 0 ? 1 : 0, b2 = a == 2 ? 1 : 2;   // the two other axes
            const bool act = t < n && se - sb >= 2;
            const int m = sb + (se - sb) / 2;
            const double ka = (a == 0) ? key[0] : (a == 1) ? key[1] : key[2];
            const int ia = (a == 0) ? id[0] : (a == 1) ? id[1] : id[2];
            xkey[t] = ka;
            side[ia] = (act && t < m) ? 1 : 0;
            __syncthreads();
            const bool my_tie = act && t == m && xkey[t - 1] == ka;
            const int i1 = (b1 == 0) ? id[0] : id[1];
            const int i2 = (b2 == 1) ? id[1] : id[2];
            const double k1 = (b1 == 0) ? key[0] : key[1];
            const double k2 = (b2 == 1) ? key[1] : key[2];
            const int sd1 = side[i1], sd2 = side[i2];
            const unsigned long long bal1 = ballot(act && sd1), bal2 = ballot(act && sd2);
            if (lane == 0) {
                wsum[wv] = __popcll(bal1);
                wsum2[wv] = __popcll(bal2);
            }
            if (__syncthreads_or(my_tie)) {
                tie = true;
                break;
            }
            int pre1 = rank_below(bal1), pre2 = rank_below(bal2);
            for (int w = 0; w < wv; w++) {
                pre1 += wsum[w];
                pre2 += wsum2[w];
            }
            xpre[t] = pre1;
            xpre2[t] = pre2;
            __syncthreads();
            int np1 = t, np2 = t;
            if (act) {
                const int lc1 = pre1 - xpre[sb], lc2 = pre2 - xpre2[sb];
                np1 = sd1 ? sb + lc1 : m + (t - sb - lc1);
                np2 = sd2 ? sb + lc2 : m + (t - sb - lc2);
            }
            xkey[np1] = k1;
            xid[np1] = i1;
            xkey2[np2] = k2;
            xid2[np2] = i2;
            __syncthreads();
            const double n1 = xkey[t], n2 = xkey2[t];
            const int j1 = xid[t], j2 = xid2[t];
            if (b1 == 0) {
                key[0] = n1;
                id[0] = j1;
            } else {
                key[1] = n1;
                id[1] = j1;
            }
            if (b2 == 1) {
                key[1] = n2;
                id[1] = j2;
            } else {
                key[2] = n2;
                id[2] = j2;
            }
            if (act) {
                if (t < m) se = m;
                else sb = m;
            }
            open = __syncthreads_or(t < n && se - sb >= 2);
        }
        if (tie) {
            if (t == 0) tied[atomicAdd(n_tied, 1u)] = s;
            __syncthreads();
            continue;
        }
        // DFS order: position p holds element arrangement[n-1-p]
        xid[t] = id[0];
        __syncthreads();
        const int e = t < n ? xid[n - 1 - t] : 0;
        kd_emit_lane(ms, st, s, n, off, abase, t, e);
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// exact path, sets of at most KD_LDS_MAX entries
//
// One partition step of a window [l, r] (pivot moved to r) in the reference's
// order: the k "<=" elements keep their order at the front, the pivot goes to
// pos = l + k. The ">" elements are a queue that lies in place behind the
// "<=" ones and rotates by one whenever a "<=" element is scanned: after the
// scan position q > pos holds what was pushed when q was scanned -- its own
// element if that is a ">" one, else the queue's front of that moment, which
// is what lies s positions earlier, s being the number of ">" elements before
// q (the queue's length). Following q -> q - s until a ">" element is met
// names the source of every position behind pos; the queue's front (position
// pos) goes to r in the pivot's swap. Inside a run of "<=" elements s does not
// change, so a run is left in one hop of a multiple of s; every hop then
// passes a ">" element, s shrinks by at least one and a hop is at least s
// long: at most about sqrt(2 * width) hops (and one per 64 positions, as runs
// are looked at one flag word at a time).
//
// Windows of more than 64 positions take rounds of the whole workgroup: the
// "<=" flags as one 64-bit word per 64 positions in LDS, prefix counts by
// popcounts, two barriers a round. Windows of at most 64 positions, and from
// the depth on where every range has at most 64 positions whole subtrees, are
// finished by one wave each with its positions in lanes: no barrier, flags
// and queue chains in one ballot word. What bounds it is the chain of
// dependent rounds (18 of the workgroup and 50 of a wave for 1,000 entries, 40
// and 70 for 4,000), each a few thousand cycles of dependent LDS reads and of
// the VALU work of up to 16 waves. Against one round of the whole workgroup
// per partition at all sizes, with the queues resolved by pointer jumping
// through LDS (a barrier per jump): a set of 1,000 entries 224 -> 94 us, 4,000
// entries 891 -> 442 us, 8,000 entries 1,370 -> 928 us; 2,000 sets of 800
// entries 1,191 -> 353 us, 1,000 sets of 2,000 entries 1,606 -> 885 us.
// ---------------------------------------------------------------------------

// ceil(log2(n)) for n >= 1
__host__ __device__ constexpr int kd_log2_ceil(int n) { return n <= 1 ? 0 : 1 + kd_log2_ceil((n + 1) / 2); }

// Bounds of the exact passes' data-dependent loops. A window of w elements
// needs at most w partition rounds, a tree of n elements fewer than
// n * (ceil(log2 n) + 1) in all; a chain of the queue has at most n links, and
// pointer jumping (each round halves every open chain) ends within
// ceil(log2 n) + 1 rounds. Reaching a bound means a broken invariant: the pass
// stops and reports it instead of looping.
#define KD_JUMP_BOUND(n) (kd_log2_ceil(n) + 2)
#ifndef KD_WAVE_ROUNDS
#define KD_WAVE_ROUNDS JAM_WAVE
#endif
#ifndef KD_WAVE_JUMPS
#define KD_WAVE_JUMPS KD_JUMP_BOUND(JAM_WAVE)
#endif
#define KD_ROUND_BOUND(n) ((long long)(n) * (kd_log2_ceil(n) + 2) + 64)

#if defined(__HIP_DEVICE_COMPILE__)
#define KD_RCP(x) __builtin_amdgcn_rcpf(x)
#else
#define KD_RCP(x) (1.0f / (x))
#endif

// bits [0, x) of a word, x < 64
__device__ static inline unsigned long long kd_below(int x) { return (1ull << x) - 1ull; }

// Range i (of 2^d, in position order) of depth d of a tree of n elements: [lo, hi).
__device__ static inline void kd_range(int n, int d, int i, int &lo, int &hi)
{
    lo = 0;
    hi = n;
    for (int b = d - 1; b >= 0; b--) {
        const int m = lo + (hi - lo) / 2;
        if ((i >> b) & 1) lo = m;
        else hi = m;
    }
}

// The range of depth d that position p lies in.
__device__ static inline int kd_range_of(int n, int d, int p)
{
    int lo = 0, hi = n, i = 0;
    for (; d > 0; d--) {
        const int m = lo + (hi - lo) / 2;
        i = 2 * i + (p < m ? 0 : 1);
        if (p < m) hi = m;
        else lo = m;
    }
    return i;
}

// Hops out of the run of "<=" positions that ends at position q, given the
// "<=" flags of q's word shifted up so that q's is the top bit (t) and the
// number s > 0 of ">" positions before q: as many hops of s as the run's part
// in this word takes. run / s by reciprocal: run < 64, and the half keeps the
// quotient further from the integers than the reciprocal's error reaches.
__device__ static inline int kd_hop(int q, unsigned long long t, int s)
{
    const int run = __clzll((long long)~t) - 1;
    return q - s * (1 + (int)(((float)run + 0.5f) * KD_RCP((float)s)));
}

// The QuickSelects of the windows [lw, rw] of a wave, lane = position (rw < 0:
// no window; lanes of one window agree on lw, rw and K, and are all there),
// until each has its element K in place. id and v (the key) move along. False
// where a window is left open, at the bound of the rounds; where a chain of the
// queue is not followed to its end, at the bound of the jumps, a lane's element
// is taken twice (kd_wave_whole).
__device__ static inline bool kd_wave_select(int &id, double &v, int lw, int rw, int K)
{
    const int lane = lane_id();
    // every round shortens every open window
    for (int round = 0; round < KD_WAVE_ROUNDS; round++) {
        const bool open = rw >= 0;
        if (ballot(open) == 0ull) break;
        const int l = open ? lw : lane, r = open ? rw : lane;
        const int mid = (l + r + 1) >> 1;
        // pivot: median of three, swapped with the window's right end
        const double vl = __shfl(v, l, JAM_WAVE), vm = __shfl(v, mid, JAM_WAVE), vr = __shfl(v, r, JAM_WAVE);
        int piv = r;
        double pv = vr;
        if ((vl > vm) != (vl > vr)) {
            piv = l;
            pv = vl;
        } else if ((vm < vl) != (vm < vr)) {
            piv = mid;
            pv = vm;
        }
        const bool in = lane >= l && lane < r;
        const bool le = in && (lane == piv ? vr : v) <= pv;
        const unsigned long long bl = kd_below(l);
        const unsigned long long L = ballot(le) & kd_below(r) & ~bl;
        const unsigned long long G = ~(L | bl);   // ">" from l on
        const int pos = l + __popcll(L);
        const int ones = __popcll(L & kd_below(lane));
        // the stable partition is a permutation of the lanes: every "<="
        // lane tells its new place
        const int part = push_int(lane, in ? (le ? l + ones : pos + (lane - l - ones)) : lane);
        // the queue: one hop of every "<=" lane behind the first ">" one,
        // then pointer doubling until every lane from pos on names a ">" one;
        // lane r takes what pos names
        const int before = lane - l - ones;       // ">" before this lane
        int from = le && before > 0 ? kd_hop(lane, L << (JAM_WAVE - 1 - lane), before) : lane;
        if (lane == r && open) from = pos;
        for (int jump = 0; jump < KD_WAVE_JUMPS; jump++) {
            from = __shfl(from, from, JAM_WAVE);
            from = __shfl(from, from, JAM_WAVE);
            if (ballot(open && lane > pos && lane <= r && ((G >> from) & 1ull) == 0ull) == 0ull) break;
        }
        int src = lane < pos ? part : (lane == pos ? r : from);
        src = src == piv ? r : (src == r ? piv : src);
        if (!(open && lane >= l && lane <= r)) src = lane;
        id = __shfl(id, src, JAM_WAVE);
        v = __shfl(v, src, JAM_WAVE);
        if (open) {
            // the next window of the QuickSelect
            if (pos == K) rw = -1;
            else if (K < pos) rw = pos - 1;
            else lw = pos + 1;
            if (rw >= 0 && lw == rw) rw = -1;
        }
    }
    return ballot(rw >= 0) == 0ull;
}

// Whether id, which the selects moved, still names every lane once.
__device__ static inline bool kd_wave_whole(int id) { return ballot(push_int(1, id) != 1) == 0ull; }

// The whole subtree of n <= 64 elements whose root splits axis d % 3: lane k
// holds the element at position k (coordinates c0, c1, c2) and returns the
// lane that held the element which ends there; ok: false where a loop bound
// was reached.
__device__ static inline int kd_wave_tree(int n, int d, double c0, double c1, double c2, bool &ok)
{
    const int lane = lane_id();
    int id = lane, R = 0, H = n;
    for (int h = n; h >= 2; h -= h / 2, d++) {
        const int ax = d % 3;
        double v = __shfl(ax == 0 ? c0 : (ax == 1 ? c1 : c2), id, JAM_WAVE);
        const bool open = lane < n && H - R >= 2;
        const int K = R + (H - R) / 2;
        ok &= kd_wave_select(id, v, R, open ? H - 1 : -1, K);
        if (open) {
            if (lane < K) H = K;
            else R = K;
        }
    }
    ok &= kd_wave_whole(id);
    return id;
}

// largest set of the LDS exact pass (1,024 threads, eight positions each);
// larger ones run in global scratch
#define KD_LDS_MAX 8192

template <int NT, int P>
struct KdExactLds {
    static constexpr int N = NT * P;
    static constexpr int NW = NT / JAM_WAVE;
    static constexpr int NWORDS = N / JAM_WAVE;
    // all three axes of small sets; of larger ones the axis of the depth
    // (loaded again at every depth)
    static constexpr int AXES = N <= KD_BIG ? 3 : 1;
    double cc[AXES][N];                   // coordinates by element
    unsigned long long le[N / JAM_WAVE];  // "<=" flags by position
    int pre[2][N / JAM_WAVE];             // "<=" flags of the words before (rounds take turns)
    int wbig[NW];                         // whether a wave has a window of more than 64 positions
    int winl[N / JAM_WAVE], winr[N / JAM_WAVE];   // windows of a depth's ranges
    unsigned short xa[2][N];              // arrangement: element at each position (rounds take turns)
};

// Arranges set s (n <= NT * P entries) in the reference's leaf order; the
// index of the xa buffer that holds it, or -1 when a loop bound was reached.
// P positions per thread: wave w holds positions w * 64P ... (w + 1) * 64P - 1,
// its lane l positions w * 64P + k * 64 + l (k < P), so that the lanes of a
// wave touch consecutive LDS entries. A thread keeps the element, range and
// window of each of its positions in registers; its positions in one range
// share the range's pivot and prefix reads.
template <int NT, int P>
__device__ static inline int kd_exact_set(const DevMols &ms, const DevSets &st, KdExactLds<NT, P> &S, int n,
                                          int64_t off, int abase)
{
    using Lds = KdExactLds<NT, P>;
    constexpr int N = Lds::N, NW = Lds::NW;
    const int t = threadIdx.x;
    const int lane = lane_id();
    const int wv = t / JAM_WAVE;
    const int p0 = wv * JAM_WAVE * P + lane;   // position of slice k: p0 + k * JAM_WAVE
#pragma unroll
    for (int k = 0; k < P; k++) {
        const int e = t + k * NT;
        if (e < n) {
            const size_t g = (size_t)(abase + st.list[off + e]);
#pragma unroll
            for (int q = 0; q < Lds::AXES; q++) S.cc[q][e] = ms.xyz[3 * g + q];
            S.xa[0][e] = (unsigned short)e;
        }
    }
    for (int i = t; i < 2 * Lds::NWORDS; i += NT) S.pre[i / Lds::NWORDS][i % Lds::NWORDS] = 0;
    __syncthreads();
    int cur = 0, par = 0, d = 0, hmax = n;   // hmax: the largest range of this depth
    if (n > JAM_WAVE) {
        // per position: element, range [R, H), window [lw, rw] (pairs of
        // 16-bit halves; rw < 0: no window)
        int a[P], range[P], win[P];
#pragma unroll
        for (int k = 0; k < P; k++) {
            a[k] = p0 + k * JAM_WAVE;
            range[k] = p0 + k * JAM_WAVE < n ? n << 16 : 0;
        }
        const long long round_bound = KD_ROUND_BOUND(n);
        long long rounds = 0;
        for (; hmax > JAM_WAVE; d++, hmax -= hmax / 2) {
            const double *c = S.cc[Lds::AXES == 3 ? d % 3 : 0];
#pragma unroll
            for (int k = 0; k < P; k++) win[k] = range[k] - (1 << 16);
            // rounds of the workgroup while a window has more than 64 positions
            for (;;) {
                if (++rounds > round_bound) return -1;   // the same for every thread
                const unsigned short *xc = S.xa[cur];
                unsigned short *xn = S.xa[cur ^ 1];
                // per position: the pivot of its window, the "<=" lanes before it
                int pp[P];
                unsigned lem = 0u;                       // bit k: position k is "<=" in its window
                unsigned long long word = 0ull;
                int wtot = 0, before = 0;
                {
                    int cR = -1, c_piv = 0, c_er = 0, c_ep = 0;
                    double c_pv = 0.0;
#pragma unroll
                    for (int k = 0; k < P; k++) {
                        const int p = p0 + k * JAM_WAVE;
                        const int l = win[k] & 0xFFFF, r = win[k] >> 16;
                        const bool big = r - l >= JAM_WAVE;
                        pp[k] = 0;
                        if (ballot(big) == 0ull) continue;   // no large window in this slice
                        if (big && range[k] != cR) {
                            // pivot: median of three, swapped with the window's right end
                            const int mid = (l + r + 1) / 2;
                            const int el = xc[l], em = xc[mid];
                            c_er = xc[r];
                            const double kl = c[el], km = c[em], kr = c[c_er];
                            const bool at_l = (kl > km) != (kl > kr), at_m = (km < kl) != (km < kr);
                            c_piv = at_l ? l : (at_m ? mid : r);
                            c_ep = at_l ? el : (at_m ? em : c_er);
                            c_pv = at_l ? kl : (at_m ? km : kr);
                            cR = range[k];
                        }
                        if (big) a[k] = p == c_piv ? c_er : (p == r ? c_ep : a[k]);
                        const bool le = big && p >= l && p < r && c[a[k]] <= c_pv;
                        const unsigned long long bal = ballot(le);
                        if (le) lem |= 1u << k;
                        pp[k] = c_piv | rank_below(bal) << 16;
                        if (lane == (wv * P + k) % JAM_WAVE) word = bal;
                        if (lane > (wv * P + k) % JAM_WAVE) before += __popcll(bal);
                        wtot += __popcll(bal);
                    }
                }
                // the wave's flag words, and its counts added to the prefix
                // counts of every later word
#pragma unroll
                for (int i = lane; i < Lds::NWORDS; i += JAM_WAVE) {
                    const bool own = i >= wv * P && i < wv * P + P;
                    if (own) S.le[i] = word;
                    const int add = own ? before : wtot;
                    if (i >= wv * P && add != 0) atomicAdd(&S.pre[par][i], add);
                }
                __syncthreads();
                for (int i = t; i < Lds::NWORDS; i += NT) S.pre[par ^ 1][i] = 0;
                const int *pre = S.pre[par];
                // "<=" flags before position q
                auto prefix = [&](int q) {
                    const int w = q / JAM_WAVE;
                    return pre[w] + __popcll(S.le[w] & kd_below(q % JAM_WAVE));
                };
                bool big = false;
                {
                    int cR = -1, c_pl = 0, c_pos = 0;
#pragma unroll
                    for (int k = 0; k < P; k++) {
                        const int p = p0 + k * JAM_WAVE;
                        int l = win[k] & 0xFFFF, r = win[k] >> 16;
                        const bool mine = r - l >= JAM_WAVE;
                        if (ballot(mine) == 0ull) {
                            if (p < n) xn[p] = (unsigned short)a[k];
                            continue;
                        }
                        if (mine && range[k] != cR) {
                            c_pl = prefix(l);
                            c_pos = l + prefix(r) - c_pl;
                            cR = range[k];
                        }
                        // "<=" elements in order, the pivot after them; the
                        // places behind pos look for what the queue leaves there
                        const bool in = mine && p >= l && p <= r, le = (lem >> k) & 1u;
                        const int to = !in ? p : (p == r ? c_pos : l + pre[wv * P + k] + (pp[k] >> 16) - c_pl);
                        if (in ? (le || p == r) : p < n) xn[to] = (unsigned short)a[k];
                        const bool behind = in && p > c_pos;
                        int q = behind && p == r ? c_pos : p;
                        for (int hops = 0;; hops++) {
                            const int w = q / JAM_WAVE;
                            const unsigned long long t = S.le[w] << (JAM_WAVE - 1 - q % JAM_WAVE);
                            const bool hop = behind && (long long)t < 0;
                            if (ballot(hop) == 0ull) break;
                            if (hops > N) {   // cannot happen: every hop goes towards the first ">" position
                                atomicOr(st.kd_err, 1u);
                                break;
                            }
                            const int s = q - (l - c_pl - 1) - (pre[w] + __popcll(t));   // ">" before q
                            const int next = kd_hop(q, t, max(s, 1));
                            q = hop ? next : q;
                        }
                        if (behind) xn[p] = xc[q == (pp[k] & 0xFFFF) ? r : q];
                        if (!mine) continue;
                        // the next window of the range's QuickSelect
                        const int lo = range[k] & 0xFFFF, hi = range[k] >> 16, kk = lo + (hi - lo) / 2;
                        if (c_pos == kk) r = -1;
                        else if (kk < c_pos) r = c_pos - 1;
                        else l = c_pos + 1;
                        if (l == r) r = -1;
                        win[k] = l | r << 16;
                        big |= r - l >= JAM_WAVE;
                    }
                }
                const unsigned long long bigs = ballot(big);
                if (lane == 0) S.wbig[wv] = bigs != 0ull;
                __syncthreads();
                cur ^= 1;
                par ^= 1;
#pragma unroll
                for (int k = 0; k < P; k++)
                    if (p0 + k * JAM_WAVE < n) a[k] = xn[p0 + k * JAM_WAVE];
                if (ballot(lane < NW && S.wbig[lane] != 0) == 0ull) break;
            }
            // the windows left, of at most 64 positions, one wave each
#pragma unroll
            for (int k = 0; k < P; k++)
                if (p0 + k * JAM_WAVE < n && p0 + k * JAM_WAVE == (range[k] & 0xFFFF)) {
                    const int i = kd_range_of(n, d, range[k] & 0xFFFF);
                    S.winl[i] = win[k] & 0xFFFF;
                    S.winr[i] = win[k] >> 16;
                }
            __syncthreads();
            for (int i = wv; i < (1 << d); i += NW) {
                const int l = S.winl[i], r = S.winr[i];
                if (r < 0) continue;   // the same for the whole wave
                int lo, hi;
                kd_range(n, d, i, lo, hi);
                const int K = lo + (hi - lo) / 2;
                const int p = l + lane;
                const bool in = p <= r;
                int e = in ? (int)S.xa[cur][p] : 0, id = lane;
                double v = in ? c[e] : 0.0;
                const bool closed = kd_wave_select(id, v, 0, in ? r - l : -1, K - l);
                if (!(kd_wave_whole(id) && closed) && lane == 0) atomicOr(st.kd_err, 1u);
                e = shfl_int(e, id);
                if (in) S.xa[cur][p] = (unsigned short)e;
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < P; k++) {
                const int p = p0 + k * JAM_WAVE;
                if (p >= n) continue;
                a[k] = S.xa[cur][p];
                const int lo = range[k] & 0xFFFF, hi = range[k] >> 16, m = lo + (hi - lo) / 2;
                range[k] = p < m ? (lo | m << 16) : (m | hi << 16);
            }
            if (Lds::AXES == 1 && hmax - hmax / 2 > JAM_WAVE) {
                const int ax = (d + 1) % 3;
#pragma unroll
                for (int k = 0; k < P; k++)
                    if (t + k * NT < n)
                        S.cc[0][t + k * NT] = ms.xyz[3 * (size_t)(abase + st.list[off + t + k * NT]) + ax];
                __syncthreads();
            }
        }
    }
    // ranges of at most 64 positions: one wave each
    for (int i = wv; i < (1 << d); i += NW) {
        int lo, hi;
        kd_range(n, d, i, lo, hi);
        const int m = hi - lo;
        int e = 0;
        double x[3] = {0.0, 0.0, 0.0};
        if (lane < m) {
            e = S.xa[cur][lo + lane];
            if (Lds::AXES == 3) {
#pragma unroll
                for (int q = 0; q < 3; q++) x[q] = S.cc[q % Lds::AXES][e];
            } else {
                const size_t g = (size_t)(abase + st.list[off + e]);
#pragma unroll
                for (int q = 0; q < 3; q++) x[q] = ms.xyz[3 * g + q];
            }
        }
        bool ok = true;
        const int id = kd_wave_tree(m, d, x[0], x[1], x[2], ok);
        if (!ok && lane == 0) atomicOr(st.kd_err, 1u);
        e = shfl_int(e, id);
        if (lane < m) S.xa[cur][lo + lane] = (unsigned short)e;
    }
    __syncthreads();
    return cur;
}

template <int NT, int P>
__device__ static inline void kd_exact_emit(const DevMols &ms, const DevSets &st, KdExactLds<NT, P> &S, int s, int n,
                                            int64_t off, int abase)
{
    const int lane = lane_id();
    const int cur = kd_exact_set<NT, P>(ms, st, S, n, off, abase);
    if (cur < 0) {
        if (threadIdx.x == 0) atomicOr(st.kd_err, 1u);
    } else {
        // DFS order: position p holds element arrangement[n-1-p]
        for (int b0 = (threadIdx.x / JAM_WAVE) * JAM_WAVE; b0 < n; b0 += NT) {
            const int p = b0 + lane;
            kd_emit_lane(ms, st, s, n, off, abase, p, p < n ? (int)S.xa[cur][n - 1 - p] : 0);
        }
    }
    __syncthreads();
}

// every set of `list` (at most NT entries each), one position per thread
template <int NT>
__global__ void __launch_bounds__(NT, 8) k_kdexact(DevMols ms, DevTpls tp, DevSets st, const int *list,
                                                const unsigned int *count)
{
    __shared__ KdExactLds<NT, 1> S;
    if (*st.total > st.cap) return;
    const int cnt = (int)*count;
    for (int q = blockIdx.x; q < cnt; q += gridDim.x) {
        const int s = list[q];
        kd_exact_emit<NT, 1>(ms, st, S, s, st.cnt[s], st.off[s], ms.atom_off[s / tp.n_types]);
    }
}

// the sets of `list` (every set of the query where there is none) of min_n + 1
// ... NT * P entries, P positions per thread
template <int NT, int P>
__global__ void __launch_bounds__(NT, 4) k_kdexact_lds(DevMols ms, DevTpls tp, DevSets st, const int *list,
                                                    const unsigned int *count, int min_n)
{
    static_assert(NT * P <= KD_LDS_MAX && KD_LDS_MAX <= 65536, "16-bit elements");
    __shared__ KdExactLds<NT, P> S;
    if (*st.total > st.cap) return;
    const int cnt = list ? (int)*count : st.n_sets;
    for (int q = blockIdx.x; q < cnt; q += gridDim.x) {
        const int s = list ? list[q] : q;
        const int n = st.cnt[s];
        if (n <= min_n || n > NT * P) continue;
        kd_exact_emit<NT, P>(ms, st, S, s, n, st.off[s], ms.atom_off[s / tp.n_types]);
    }
}

// ---------------------------------------------------------------------------
// sets larger than KD_LDS_MAX: both paths on work arrays in global scratch
// (scr + off * KD_SCRATCH_BYTES_PER_ENTRY), KD_THREADS threads looping over
// the positions
// ---------------------------------------------------------------------------

// in-place exclusive block scan of v[0, n)
template <int NT>
__device__ static void kd_scan(int *v, int n, int *partial)
{
    const int tid = threadIdx.x;
    const int per = (n + NT - 1) / NT;
    const int b0 = tid * per, b1 = min(n, b0 + per);
    int cnt = 0;
    for (int p = b0; p < b1; p++) cnt += v[p];
    partial[tid] = cnt;
    __syncthreads();
    if (tid < JAM_WAVE) {
        int x[NT / JAM_WAVE], sum = 0;
#pragma unroll
        for (int q = 0; q < NT / JAM_WAVE; q++) {
            x[q] = partial[(NT / JAM_WAVE) * tid + q];
            sum += x[q];
        }
        int incl = sum;
        for (int sh = 1; sh < JAM_WAVE; sh <<= 1) {
            int o = __shfl_up(incl, sh, JAM_WAVE);
            if (tid >= sh) incl += o;
        }
        int run = incl - sum;
#pragma unroll
        for (int q = 0; q < NT / JAM_WAVE; q++) {
            partial[(NT / JAM_WAVE) * tid + q] = run;
            run += x[q];
        }
    }
    __syncthreads();
    int run = partial[tid];
    for (int p = b0; p < b1; p++) {
        const int x = v[p];
        v[p] = run;
        run += x;
    }
    __syncthreads();
}

// Writes the kd arrays of set s from its arrangement `order` (element ids =
// list positions): position p of the DFS visit order is element n-1-p.
template <int NT>
__device__ static void kd_emit_order(const DevMols &ms, const DevSets &st, int s, int n, int64_t off, int abase,
                                     const int *order)
{
    const int lane = lane_id();
    for (int b0 = (threadIdx.x / JAM_WAVE) * JAM_WAVE; b0 < n; b0 += NT) {
        const int p = b0 + lane;
        kd_emit_lane(ms, st, s, n, off, abase, p, p < n ? order[n - 1 - p] : 0);
    }
}

struct KdFast {
    double *c;               // coordinates, axis-major, stride entries per axis
    int *perm;               // 3 axes x 2 buffers, stride entries each
    int *pre;                // prefix of left sides
    int *sb, *se;            // range of each position
    unsigned char *side;     // by element
    int stride;
};

template <int NT>
__device__ static void kdf_sort(const double *c, int *perm, int n, int n2)
{
    const int tid = threadIdx.x;
    for (int i = tid; i < n2; i += NT) perm[i] = i;
    __syncthreads();
    for (int k = 2; k <= n2; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = tid; i < n2; i += NT) {
                const int ixj = i ^ j;
                if (ixj > i) {
                    const int x = perm[i], y = perm[ixj];
                    const double kx = x < n ? c[x] : INFINITY, ky = y < n ? c[y] : INFINITY;
                    const bool y_less = key_less(ky, y, kx, x);
                    const bool up = (i & k) == 0;
                    if (y_less == up) {
                        perm[i] = y;
                        perm[ixj] = x;
                    }
                }
            }
            __syncthreads();
        }
    }
}

// fast path; returns true (nothing written to out) on a split tie
template <int NT>
__device__ static bool kd_fast(const KdFast &w, int n, int *out, int *partial, int *flag)
{
    const int tid = threadIdx.x;
    int n2 = 1;
    while (n2 < n) n2 <<= 1;
    const int S = w.stride;
    for (int a = 0; a < 3; a++) kdf_sort<NT>(w.c + a * S, w.perm + 2 * a * S, n, n2);
    for (int p = tid; p < n; p += NT) {
        w.sb[p] = 0;
        w.se[p] = n;
    }
    int cur[3] = {0, 0, 0};
    __syncthreads();
    for (int d = 0;; d++) {
        const int a = d % 3;
        if (tid == 0) {
            flag[0] = 0;
            flag[1] = 0;
        }
        __syncthreads();
        const int *pa = w.perm + (2 * a + cur[a]) * S;
        const double *ca = w.c + a * S;
        for (int p = tid; p < n; p += NT) {
            const int sb = w.sb[p], se = w.se[p];
            if (se - sb < 2) continue;
            const int m = sb + (se - sb) / 2;
            w.side[pa[p]] = p < m ? 1 : 0;
            if (p == m) {
                flag[0] = 1;
                if (ca[pa[m - 1]] == ca[pa[m]]) flag[1] = 1;
            }
        }
        __syncthreads();
        const int splits = flag[0], tie = flag[1];
        __syncthreads();
        if (tie) return true;
        if (!splits) break;
        for (int b = 0; b < 3; b++) {
            if (b == a) continue;
            const int *src = w.perm + (2 * b + cur[b]) * S;
            int *dst = w.perm + (2 * b + (cur[b] ^ 1)) * S;
            for (int p = tid; p < n; p += NT) w.pre[p] = w.side[src[p]];
            __syncthreads();
            kd_scan<NT>(w.pre, n, partial);
            for (int p = tid; p < n; p += NT) {
                const int sb = w.sb[p], se = w.se[p];
                int np = p;
                if (se - sb >= 2) {
                    const int m = sb + (se - sb) / 2;
                    const int lc = w.pre[p] - w.pre[sb];
                    np = w.side[src[p]] ? sb + lc : m + (p - sb - lc);
                }
                dst[np] = src[p];
            }
            __syncthreads();
            cur[b] ^= 1;
        }
        for (int p = tid; p < n; p += NT) {
            const int sb = w.sb[p], se = w.se[p];
            if (se - sb < 2) continue;
            const int m = sb + (se - sb) / 2;
            if (p < m) w.se[p] = m;
            else w.sb[p] = m;
        }
        __syncthreads();
    }
    const int *fin = w.perm + cur[0] * S;
    for (int p = tid; p < n; p += NT) out[p] = fin[p];
    __syncthreads();
    return false;
}

struct KdWork {
    double *c;               // coordinates: axis a of element e at c[a * stride + e]
    int *arr;                // arrangement, double buffered at arr and arr + stride
    int *pre1, *pre2;        // exclusive prefixes: "<=" flags, re-push flags
    int *src;                // push -> element (>= 0) or -(push index) - 1
    int *rlo, *rhi;          // range of each position at the current level
    int *wl, *wr;            // QuickSelect window of the range starting here; wr < 0: done
    int stride;
};

__device__ static inline int kd_cmp3(const double *c, int x, int y)
{
    const double u = c[x], v = c[y];
    return u < v ? -1 : (u > v ? 1 : 0);
}

// exact path: arranges elements 0..n-1 into the reference's leaf order;
// false when a loop bound was reached (out is then not written)
template <int NT>
__device__ static bool kd_exact(const KdWork &w, int n, int *out, int *partial, int *flag)
{
    const int tid = threadIdx.x;
    const int jump_bound = KD_JUMP_BOUND(n);
    const long long round_bound = KD_ROUND_BOUND(n);
    long long rounds = 0;
    int cur = 0;
    for (int p = tid; p < n; p += NT) {
        w.arr[p] = p;
        w.rlo[p] = 0;
        w.rhi[p] = n;
    }
    __syncthreads();
    for (int d = 0;; d++) {
        const double *c = w.c + (d % 3) * w.stride;
        if (tid == 0) flag[0] = 0;
        __syncthreads();
        for (int p = tid; p < n; p += NT) {
            if (w.rlo[p] != p) continue;
            const int hi = w.rhi[p];
            if (hi - p >= 2) {
                w.wl[p] = p;
                w.wr[p] = hi - 1;
                flag[0] = 1;
            } else {
                w.wr[p] = -1;
            }
        }
        __syncthreads();
        if (!flag[0]) break;
        for (;;) {
            if (++rounds > round_bound) return false;
            int *a = w.arr + cur * w.stride;
            int *an = w.arr + (cur ^ 1) * w.stride;
            // pivot: median of three, moved to the right end of the window
            for (int p = tid; p < n; p += NT) {
                if (w.rlo[p] != p || w.wr[p] < 0) continue;
                const int l = w.wl[p], r = w.wr[p], mid = (l + r + 1) / 2;
                int piv;
                if ((kd_cmp3(c, a[l], a[mid]) > 0) != (kd_cmp3(c, a[l], a[r]) > 0)) piv = l;
                else if ((kd_cmp3(c, a[mid], a[l]) < 0) != (kd_cmp3(c, a[mid], a[r]) < 0)) piv = mid;
                else piv = r;
                const int t = a[r];
                a[r] = a[piv];
                a[piv] = t;
            }
            __syncthreads();
            // "<= pivot" flags of the windows
            for (int i = tid; i < n; i += NT) {
                const int R = w.rlo[i];
                const int r = w.wr[R];
                int b = 0;
                if (r >= 0 && i >= w.wl[R] && i < r) b = c[a[i]] <= c[a[r]] ? 1 : 0;
                w.pre1[i] = b;
            }
            __syncthreads();
            kd_scan<NT>(w.pre1, n, partial);
            // re-push flags: a "<=" element after the first ">" one
            for (int i = tid; i < n; i += NT) {
                const int R = w.rlo[i];
                const int l = w.wl[R], r = w.wr[R];
                int rot = 0;
                if (r >= 0 && i >= l && i < r && c[a[i]] <= c[a[r]]) {
                    const int zeros = (i - l) - (w.pre1[i] - w.pre1[l]);
                    rot = zeros > 0 ? 1 : 0;
                }
                w.pre2[i] = rot;
            }
            __syncthreads();
            kd_scan<NT>(w.pre2, n, partial);
            // pushes: ">" elements are new pushes, re-pushes point to push q
            for (int i = tid; i < n; i += NT) {
                const int R = w.rlo[i];
                const int l = w.wl[R], r = w.wr[R];
                if (r < 0 || i < l || i >= r) continue;
                const int ones = w.pre1[i] - w.pre1[l];
                const int zeros = (i - l) - ones;
                const int rots = w.pre2[i] - w.pre2[l];
                const int slot = l + zeros + rots;      // push number - 1, absolute
                if (!(c[a[i]] <= c[a[r]])) w.src[slot] = a[i];
                else if (zeros > 0) w.src[slot] = -(l + rots) - 1;
            }
            __syncthreads();
            // pointer jumping until every push names an element
            for (int jumps = 0;; jumps++) {
                if (jumps > jump_bound) return false;
                if (tid == 0) flag[1] = 0;
                __syncthreads();
                for (int i = tid; i < n; i += NT) {
                    const int R = w.rlo[i];
                    const int l = w.wl[R], r = w.wr[R];
                    if (r < 0 || i < l || i >= r) continue;
                    // only the m + nrot pushes of this round are valid; each
                    // re-push points to a lower push, so the chains end
                    const int pushes = (r - l) - (w.pre1[r] - w.pre1[l]) + (w.pre2[r] - w.pre2[l]);
                    if (i - l >= pushes) continue;
                    const int v = w.src[i];
                    if (v < 0) {
                        const int u = w.src[-v - 1];
                        w.src[i] = u;
                        if (u < 0) flag[1] = 1;
                    }
                }
                __syncthreads();
                const int again = flag[1];
                __syncthreads();
                if (!again) break;
            }
            // scatter into the other buffer
            for (int i = tid; i < n; i += NT) {
                const int R = w.rlo[i];
                const int l = w.wl[R], r = w.wr[R];
                if (r < 0 || i < l || i > r) {
                    an[i] = a[i];
                    continue;
                }
                const int k1 = w.pre1[r] - w.pre1[l];
                const int m = (r - l) - k1;
                const int nrot = w.pre2[r] - w.pre2[l];
                if (i == r) {
                    an[l + k1] = a[r];                  // the pivot
                    continue;
                }
                if (c[a[i]] <= c[a[r]]) an[l + (w.pre1[i] - w.pre1[l])] = a[i];
                const int j = i - l;                    // queue slot j+1
                if (j < m) an[j == 0 ? r : l + k1 + j] = w.src[l + nrot + j];
            }
            __syncthreads();
            cur ^= 1;
            // next window of each QuickSelect
            if (tid == 0) flag[1] = 0;
            __syncthreads();
            for (int p = tid; p < n; p += NT) {
                if (w.rlo[p] != p || w.wr[p] < 0) continue;
                const int l = w.wl[p], r = w.wr[p];
                const int pos = l + (w.pre1[r] - w.pre1[l]);
                const int k = p + (w.rhi[p] - p) / 2;
                int nl = l, nr = r;
                if (pos == k) nr = -1;
                else if (k < pos) nr = pos - 1;
                else nl = pos + 1;
                if (nr >= 0 && nl == nr) nr = -1;
                w.wl[p] = nl;
                w.wr[p] = nr;
                if (nr >= 0) flag[1] = 1;
            }
            __syncthreads();
            const int more = flag[1];
            __syncthreads();
            if (!more) break;
        }
        // split every range at its median position
        for (int p = tid; p < n; p += NT) {
            const int lo = w.rlo[p], hi = w.rhi[p];
            if (hi - lo < 2) continue;
            const int m = lo + (hi - lo) / 2;
            if (p < m) w.rhi[p] = m;
            else w.rlo[p] = m;
        }
        __syncthreads();
    }
    const int *fin = w.arr + cur * w.stride;
    for (int p = tid; p < n; p += NT) out[p] = fin[p];
    __syncthreads();
    return true;
}

__device__ static void kd_load_global(const DevMols &ms, const DevSets &st, int n, int64_t off, int abase,
                                      double *c, size_t stride)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const size_t g = (size_t)(abase + st.list[off + i]);
        c[i] = ms.xyz[3 * g + 0];
        c[stride + i] = ms.xyz[3 * g + 1];
        c[2 * stride + i] = ms.xyz[3 * g + 2];
    }
    __syncthreads();
}

// Whether the fast path is not worth trying: equal coordinates among (up to)
// KD_SAMPLE elements of an axis, or a coordinate that is not a number
// anywhere. The fast path finds a split tie only after its sorts, and has then
// cost as much as the exact path (9,000 entries on 0.001 A coordinates: 7 ms
// each); on such coordinates 2,048 of them hold equal ones for sure (21
// pairs an axis in 100 A, 2 in 1,000 A), on unrounded ones they do not.
#define KD_SAMPLE 2048
__device__ static bool kd_repeats(const double *c, size_t stride, int n, unsigned long long *slot, int *flag)
{
    constexpr int SLOTS = 2 * KD_SAMPLE;
    constexpr unsigned long long EMPTY = ~0ull;   // the bits of a NaN
    const int every = max(n / KD_SAMPLE, 1), sampled = min(n / every, KD_SAMPLE);
    if (threadIdx.x == 0) flag[0] = 0;
    for (int a = 0; a < 3; a++) {
        const double *x = c + a * stride;
        for (int i = threadIdx.x; i < SLOTS; i += blockDim.x) slot[i] = EMPTY;
        __syncthreads();
        bool stop = false;
        for (int i = threadIdx.x; i < n; i += blockDim.x) stop |= x[i] != x[i];
        for (int i = threadIdx.x; i < sampled && !stop; i += blockDim.x) {
            const double v = x[i * every] + 0.0;   // one zero
            unsigned long long bits;
            __builtin_memcpy(&bits, &v, sizeof(bits));
            unsigned int h = (unsigned int)((bits * 0x9E3779B97F4A7C15ull) >> 40);
            for (int probe = 0; probe < SLOTS; probe++, h++) {
                const unsigned long long old = atomicCAS(&slot[h % SLOTS], EMPTY, bits);
                if (old == EMPTY) break;
                stop |= old == bits;
                if (stop) break;
            }
        }
        if (stop) flag[0] = 1;
        __syncthreads();
        if (flag[0]) break;
    }
    const bool found = flag[0] != 0;
    __syncthreads();
    return found;
}

// fast path of the sets of `list` (every set of the query where there is none)
// larger than min_n; sets with a split tie go to `tied`, and so do those that
// are likely to have one
__global__ void __launch_bounds__(KD_THREADS) k_kdbig(DevMols ms, DevTpls tp, DevSets st, unsigned char *scr,
                                                      const int *list, const unsigned int *count, int *tied,
                                                      unsigned int *n_tied, int min_n)
{
    __shared__ int partial[KD_THREADS];
    __shared__ int flag[2];
    __shared__ unsigned long long slot[2 * KD_SAMPLE];
    if (*st.total > st.cap) return;
    const int cnt = list ? (int)*count : st.n_sets;
    for (int q = blockIdx.x; q < cnt; q += gridDim.x) {
        const int s = list ? list[q] : q;
        const int n = st.cnt[s];
        if (n <= min_n) continue;
        const int64_t off = st.off[s];
        const int abase = ms.atom_off[s / tp.n_types];
        int n2 = 1;
        while (n2 < n) n2 <<= 1;
        double *cb = (double *)(scr + (size_t)off * KD_SCRATCH_BYTES_PER_ENTRY);
        int *ib = (int *)(cb + 3 * (size_t)n2);
        KdFast w;
        w.c = cb;
        w.perm = ib;
        w.pre = ib + 6 * n2;
        w.sb = ib + 7 * n2;
        w.se = ib + 8 * n2;
        w.side = (unsigned char *)(ib + 9 * n2);
        w.stride = n2;
        kd_load_global(ms, st, n, off, abase, w.c, (size_t)n2);
        // the arrangement after the work arrays: 61 * n2 + 4 * n <= 128 * n bytes
        int *order = (int *)((unsigned char *)(ib + 9 * n2) + n2);
        if (!kd_repeats(w.c, (size_t)n2, n, slot, flag) && !kd_fast<KD_THREADS>(w, n, order, partial, flag))
            kd_emit_order<KD_THREADS>(ms, st, s, n, off, abase, order);
        else if (threadIdx.x == 0) tied[atomicAdd(n_tied, 1u)] = s;
        __syncthreads();
    }
}

// exact path of the sets of `list` (every set of the query where there is none)
// larger than min_n
__global__ void __launch_bounds__(KD_EXACT_THREADS) k_kdbig_exact(DevMols ms, DevTpls tp, DevSets st,
                                                                  unsigned char *scr, const int *list,
                                                                  const unsigned int *count, int min_n)
{
    __shared__ int partial[KD_EXACT_THREADS];
    __shared__ int flag[2];
    if (*st.total > st.cap) return;
    const int cnt = list ? (int)*count : st.n_sets;
    for (int q = blockIdx.x; q < cnt; q += gridDim.x) {
        const int s = list ? list[q] : q;
        const int n = st.cnt[s];
        if (n <= min_n) continue;
        const int64_t off = st.off[s];
        const int abase = ms.atom_off[s / tp.n_types];
        double *cb = (double *)(scr + (size_t)off * KD_SCRATCH_BYTES_PER_ENTRY);
        int *ib = (int *)(cb + 3 * (size_t)n);
        const size_t stride = (size_t)n;
        KdWork w;
        w.c = cb;
        w.arr = ib;
        w.pre1 = ib + 2 * stride;
        w.pre2 = ib + 3 * stride;
        w.src = ib + 4 * stride;
        w.rlo = ib + 5 * stride;
        w.rhi = ib + 6 * stride;
        w.wl = ib + 7 * stride;
        w.wr = ib + 8 * stride;
        w.stride = (int)stride;
        kd_load_global(ms, st, n, off, abase, w.c, stride);
        int *order = ib + 9 * stride;   // the arrangement after the work arrays (64 * n bytes)
        if (kd_exact<KD_EXACT_THREADS>(w, n, order, partial, flag))
            kd_emit_order<KD_EXACT_THREADS>(ms, st, s, n, off, abase, order);
        else if (threadIdx.x == 0)
            atomicOr(st.kd_err, 1u);
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// launches
// ---------------------------------------------------------------------------

// clears the kd passes' per-tier counts
__global__ void __launch_bounds__(64) k_kd_setup(unsigned int *counts, int n)
{
    if ((int)threadIdx.x < n) counts[threadIdx.x] = 0u;
}

// The kd passes over the candidate sets of `st`. Sets of up to
// KD_LDS_MAX entries are mostly left to the exact QuickSelect pass alone: on
// 0.001 A coordinates a set of a few hundred entries often has equal values at
// one of its n-1 split points, and the exact pass costs no more than the sorts
// of the fast pass (2,000 sets of 800 entries: 0.35 ms against 0.46 ms).
//
// One molecule (a few hundred sets, bound by the latency of the longest chain
// of rounds and by launches): every set of up to KD_BIG entries in one launch
// of 1,024-thread workgroups, one position per thread -- two of them per CU,
// so all sets run at once -- and the larger ones beside it on side streams:
// one of them where the molecule is too small for more than an odd set of
// that size (KD_ONE_STREAM_ATOMS), three, by size, in larger ones. Sets beyond
// KD_LDS_MAX get a fast and an exact pass in global scratch, as below (without
// equal coordinates, one set of 40,000 entries: 40 ms against 55 by the exact
// pass alone).
//
// Several molecules: the sets are bucketed by size tier, and every tier gets
// a stream of its own. Tiers 0 and 1 (<= 128 entries, mostly without ties)
// get a fast pass on the main stream and the exact pass over the sets that it lists;
// tiers 2-4 the exact pass alone, two positions per thread above 256 entries
// (throughput: 0.35 ms for 2,000 sets of 800 entries against 0.51 ms with one
// position per thread, which is the faster form for a single set); tier 5 the
// exact pass in LDS up to KD_LDS_MAX entries, and above that a fast and an
// exact pass in global scratch.
//
// q: q.run(k, slot, kernel, threads, args...) launches on side stream k (or
// KD_MAIN) over a grid of at most n_sets workgroups (slot: the kernel's place
// among the grids that q keeps), q.run_grid over as many as given; grids are
// upper bounds, every kernel loops over its own list. q.fork(k, from): side
// stream k goes on from where the main stream is at fork(from, from);
// q.joined(k): nothing more on side stream k. Every set is written once all
// side streams that were joined, and the main stream, are through.
#define KD_MAIN (-1)
#define KD_SIDES (KD_TIERS + 1)   // a side stream per tier, and one more for the smallest sets of the largest
#define KD_GRIDS 13
constexpr int64_t KD_ONE_STREAM_ATOMS = 16384;

// bucket, tied: KD_TIERS * n_sets each; count: 2 * KD_TIERS
template <class Q>
static void kd_launches(Q &q, const DevMols &ms, const DevTpls &tp, const DevSets &st, unsigned char *scr, int *bucket,
                        int *tied, unsigned int *count, bool one_molecule, int64_t n_atoms)
{
    typedef const int *List;
    typedef const unsigned int *Count;
    const size_t ns = (size_t)st.n_sets;
    unsigned int *nb = count, *nt = count + KD_TIERS;
    // the passes over `list` (every set where there is none) of the sets beyond
    // KD_BIG entries, by size
    auto lds2 = [&](int k, List list, Count n) { q.run(k, 9, k_kdexact_lds<1024, 2>, 1024, ms, tp, st, list, n, KD_BIG); };
    auto lds4 = [&](int k, List list, Count n) {
        q.run(k, 10, k_kdexact_lds<1024, 4>, 1024, ms, tp, st, list, n, KD_LDS_MAX / 4);
    };
    auto lds8 = [&](int k, List list, Count n) {
        q.run(k, 11, k_kdexact_lds<1024, 8>, 1024, ms, tp, st, list, n, KD_LDS_MAX / 2);
    };
    auto big_fast = [&](int k, List list, Count n, int *out, unsigned int *n_out) {
        q.run(k, 2, k_kdbig, KD_THREADS, ms, tp, st, scr, list, n, out, n_out, KD_LDS_MAX);
    };
    auto big_exact = [&](int k, List list, Count n) {
        q.run(k, 12, k_kdbig_exact, KD_EXACT_THREADS, ms, tp, st, scr, list, n, KD_LDS_MAX);
    };
    static_assert(KD_LDS_MAX == 8 * 1024, "the sizes of the LDS passes");
    if (one_molecule) {
        // the side streams start before the main stream's pass, which is the
        // longest, and goes first, where sets as large as theirs are odd ones
        const bool sides = n_atoms > KD_BIG, spread = n_atoms > KD_ONE_STREAM_ATOMS;
        auto main_pass = [&] {
            q.run(KD_MAIN, 8, k_kdexact_lds<KD_BIG, 1>, KD_BIG, ms, tp, st, (List)nullptr, (Count)nullptr, 0);
        };
        if (sides)
            for (int k = 5; k >= (spread ? 3 : 5); k--) q.fork(k, 5);
        if (!spread) main_pass();
        if (sides) {
            lds8(5, nullptr, nullptr);
            lds4(spread ? 4 : 5, nullptr, nullptr);
            lds2(spread ? 3 : 5, nullptr, nullptr);
        }
        if (spread) main_pass();
        if (sides) {
            if (n_atoms > KD_LDS_MAX) {
                int *list = tied + 5 * ns;
                q.run_grid(5, 1, k_kd_setup, 64, nt + 5, 1);
                big_fast(5, nullptr, nullptr, list, nt + 5);
                big_exact(5, list, nt + 5);
            }
            for (int k = 5; k >= (spread ? 3 : 5); k--) q.joined(k);
        }
        return;
    }
    q.run_grid(KD_MAIN, 1, k_kd_setup, 64, nb, 2 * KD_TIERS);
    q.run_grid(KD_MAIN, max(1, min((st.n_sets + KD_BUCKET_SPAN - 1) / KD_BUCKET_SPAN, 1024)), k_kdbucket, 256, st,
               bucket, nb);
    // largest tier first: its exact passes, the longest, start earliest
    for (int k = KD_TIERS - 1; k >= 0; k--) {
        List all = bucket + (size_t)k * ns;
        int *list = tied + (size_t)k * ns;
        Count n_all = nb + k;
        unsigned int *n_list = nt + k;
        switch (k) {
        case 5:
            big_fast(KD_MAIN, all, n_all, list, n_list);
            q.fork(5, 5);
            q.fork(6, 5);
            lds2(6, all, n_all);
            q.joined(6);
            lds8(5, all, n_all);
            lds4(5, all, n_all);
            big_exact(5, list, n_list);
            break;
        case 4:
            q.fork(k, k);
            q.run(k, 7, k_kdexact_lds<512, 2>, 512, ms, tp, st, all, n_all, 0);
            break;
        case 3:
            q.fork(k, k);
            q.run(k, 6, k_kdexact_lds<256, 2>, 256, ms, tp, st, all, n_all, 0);
            break;
        case 2:
            q.fork(k, k);
            q.run(k, 5, k_kdexact<256>, 256, ms, tp, st, all, n_all);
            break;
        case 1:
            q.run(KD_MAIN, 1, k_kdblock<128>, 128, ms, tp, st, all, n_all, list, n_list);
            q.fork(k, k);
            q.run(k, 4, k_kdexact<128>, 128, ms, tp, st, (List)list, (Count)n_list);
            break;
        default:
            q.run(KD_MAIN, 0, k_kdwave, JAM_WAVE, ms, tp, st, all, n_all, list, n_list);
            q.fork(k, k);
            q.run(k, 3, k_kdexact<64>, 64, ms, tp, st, (List)list, (Count)n_list);
            break;
        }
        q.joined(k);
    }
}

}  // namespace jam
