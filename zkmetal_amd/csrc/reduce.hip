// Bucket merge, bucket reduction and window combine: the additions that follow
// the accumulation.  All of them are chains of dependent point additions, so
// they run on lane teams (team29.hpp): 64 G1 teams or 32 G2 teams per block.
//
//   k_merge_runs / k_merge_lists / k_merge_spans   bucket partials that
//                     crossed lane boundaries
//   k_br_rowcol / k_br_bits  bucket reduction: window sum = U + sum_b 2^b Q_b,
//                     Q_b bit-plane sums of the bucket index (replaces the
//                     running sums of msm_kernels.metal:152-248)
//   k_tail_windows / k_tail_combine   window combine on the device
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "kernels.hpp"
#include "plan.hpp"
#include "segments.hpp"
#include "team29.hpp"

namespace zk {

// the call's last kernel, block 0: err and counts to pinned host memory
__device__ __forceinline__ void write_back(const CallBack& b) {
    if (blockIdx.x != 0 || !b.out) return;
    if (threadIdx.x < 5) b.out[threadIdx.x] = b.err[threadIdx.x];
    for (uint32_t i = threadIdx.x; i < b.nseg; i += blockDim.x) b.out[8 + i] = b.seg_valid[i];
}

// sum over aligned groups of P teams of a wave (P a power of two, uniform):
// a butterfly, so every team ends with the group's total
template <class T>
__device__ __forceinline__ void wave_tree(typename T::Pt& acc, uint32_t P) {
#pragma unroll 1
    for (uint32_t s = 1; s < P; s <<= 1) T::add(acc, T::xor_team(acc, s));
}

// the same over groups of up to a block's teams: the waves of a group meet in
// LDS (lds: four points).  P uniform over the block; every thread calls it,
// but those that tree_idle excuses.
template <class T>
__device__ __forceinline__ void block_tree(typename T::Pt& acc, uint32_t P, uint4* lds) {
    wave_tree<T>(acc, min(P, T::kPerWave));
    const uint32_t nw = P / T::kPerWave;  // waves per group
    if (nw <= 1) return;
    const uint32_t w = threadIdx.x >> 6;
#pragma unroll 1
    for (uint32_t k = 1; k < nw; k <<= 1) {
        if ((threadIdx.x & 63u) < T::kLanes) T::store(lds, w, acc);
        __syncthreads();
        const typename T::Pt o = T::load(lds, w ^ k);
        T::add(acc, o);
        __syncthreads();  // the slots are written again
    }
}

// ------------------------------------------------------ partial merging
// Records with equal key are contiguous (a bucket's partials come from
// consecutive lanes; the padding of empty lanes carries key 0x7fffffff): a
// run.  A run of at most kMergeShort payload records (and three times as many
// records in all) is summed by the team that sees its first record; one of at
// most kMergeMid records goes to the mid list (a wave each); a longer one is
// cut at record indices divisible by kMergeSpan into spans of at most that
// many records (a block each).  A run of several spans leaves a partial sum
// per span, and its entry in the run list has k_merge_spans add those up: a
// heavy bucket's thousands of records are summed by as many blocks as they
// fill, 4 + 6 additions deep, instead of one block walking them all.
// Measured against one lane per addition (and one block per long run):
// 150,001 witness-like scalars 303 -> 69 us, 2^16 points 218 -> 95, 2^22
// points 98 -> 73.  What is left at 2^22 points is issue: 16 waves per SIMD
// of one or two additions each.
constexpr uint32_t kMergeShort = 8;
constexpr uint32_t kMergeMid = 64;
constexpr uint32_t kMergeSpan = 256;

// the lists' device memory: counters, then the lists (caps in MergeCaps)
struct MergeLists {
    uint32_t* counts;  // mid runs, spans, span partials, runs of several spans
    uint32_t* mid;     // first record
    uint2* spans;      // first record, partial slot (or none: the run's only span)
    uint4* runs;       // first partial slot, spans, bucket
    uint4* part;       // partial sums
};

template <class T>
__global__ __launch_bounds__(256) void k_merge_runs(const uint32_t* __restrict__ keys,
                                                    const uint4* __restrict__ pts, uint64_t nrec,
                                                    uint4* __restrict__ dest, MergeLists L, MergeCaps cap) {
    // team i looks at records 2i and 2i+1 (one accumulation lane's head and
    // tail slots); at most one of them starts a run with a payload
    const uint64_t i2 = 2 * (((uint64_t)blockIdx.x * 256 + threadIdx.x) / T::kLanes);
    if (i2 >= nrec) return;
    const bool lead = T::lane() == 0;
    // the usual run -- it starts here, ends within the next records and has at
    // most three payloads -- from one batch of key loads and one of payloads
    constexpr uint32_t kAhead = 8;
    uint32_t kw[kAhead + 1];  // keys i2 - 1 .. i2 + 7
#pragma unroll
    for (uint32_t t = 0; t <= kAhead; t++) {
        const uint64_t x = i2 + t;
        kw[t] = x > 0 && x <= nrec ? keys[x - 1] : ~0u;
    }
    // bit t: record i2 + t starts a run of a real key
    uint32_t starts = 0;
#pragma unroll
    for (uint32_t t = 0; t < 2; t++)
        if ((kw[t + 1] & ZK_REC_KEYMASK) != ZK_REC_KEYMASK && (kw[t] & ZK_REC_KEYMASK) != (kw[t + 1] & ZK_REC_KEYMASK))
            starts |= 1u << t;
    if (starts == 0) return;
    {
        const uint32_t t0 = (starts & 2u) ? 1u : 0u;
        const uint32_t k = (t0 ? kw[2] : kw[1]) & ZK_REC_KEYMASK;
        uint32_t mask = 0, inside = 0;  // payload records and records of the run among kw[1..]
#pragma unroll
        for (uint32_t t = 0; t < kAhead; t++) {
            inside |= ((kw[t + 1] & ZK_REC_KEYMASK) == k) ? 1u << t : 0u;
            mask |= kw[t + 1] == k ? 1u << t : 0u;
        }
        // (an earlier run that starts here too, t0 = 1, ended at once: it has
        // a payload only if its one record is)
        const bool other = starts == 3u && !(kw[1] & ZK_REC_INVALID);
        if (!other && !(inside >> (kAhead - 1)) && __popc(mask) <= 3) {
            if (mask == 0) return;
            const uint32_t b0 = __ffs(mask) - 1;
            mask &= mask - 1;
            const uint32_t b1 = mask ? __ffs(mask) - 1 : b0;
            const uint32_t more = mask & (mask - 1);
            const uint32_t b2 = more ? __ffs(more) - 1 : b0;
            typename T::Pt acc = T::load(pts, i2 + b0);
            if (mask) {
                const typename T::Pt q = T::load(pts, i2 + b1);
                typename T::Pt q2 = T::load(pts, i2 + b2);
                T::add(acc, q);
                if (more) T::add(acc, q2);
            }
            T::store(dest, k, acc);
            return;
        }
    }
    for (uint64_t i = i2; i < i2 + 2 && i < nrec; i++) {
        const uint32_t k = keys[i] & ZK_REC_KEYMASK;
        if (k == ZK_REC_KEYMASK) continue;  // padding
        if (i > 0 && (keys[i - 1] & ZK_REC_KEYMASK) == k) continue;
        uint64_t j = i;
        uint32_t valid = 0;
        while (j < nrec && valid <= kMergeShort && j - i <= 3 * kMergeShort) {
            const uint32_t kj = keys[j];
            if ((kj & ZK_REC_KEYMASK) != k) break;
            valid += (kj & ZK_REC_INVALID) ? 0u : 1u;
            j++;
        }
        auto same = [&](uint64_t x) { return x < nrec && (keys[x] & ZK_REC_KEYMASK) == k; };
        if (valid > kMergeShort || (j - i > 3 * kMergeShort && same(j))) {
            if (!lead) continue;
            if (!same(i + kMergeMid)) {
                const uint32_t slot = atomicAdd(&L.counts[0], 1u);
                if (slot < cap.mid) L.mid[slot] = (uint32_t)i;
                continue;
            }
            // spans: [i, first boundary), then one per boundary inside the run
            const uint64_t w0 = i / kMergeSpan;
            uint64_t lo = 0, hi = 1;  // boundary w0 + lo is inside (or lo = 0), w0 + hi is not
            while (same((w0 + hi) * kMergeSpan)) {
                lo = hi;
                hi *= 2;
            }
            while (hi - lo > 1) {
                const uint64_t mid = (lo + hi) / 2;
                if (same((w0 + mid) * kMergeSpan)) lo = mid;
                else hi = mid;
            }
            const uint32_t ns = (uint32_t)lo + 1;
            uint32_t p0 = ~0u;
            if (ns > 1) {
                p0 = atomicAdd(&L.counts[2], ns);
                if (p0 + ns > cap.parts) continue;  // never: the caps are true bounds
                const uint32_t r = atomicAdd(&L.counts[3], 1u);
                if (r < cap.runs) L.runs[r] = make_uint4(p0, ns, k, 0);
            }
            const uint32_t s0 = atomicAdd(&L.counts[1], ns);
            for (uint32_t s = 0; s < ns; s++)
                if (s0 + s < cap.spans)
                    L.spans[s0 + s] = make_uint2(s ? (uint32_t)((w0 + s) * kMergeSpan) : (uint32_t)i,
                                                 ns > 1 ? p0 + s : ~0u);
            continue;
        }
        bool has = false;
        typename T::Pt acc = T::identity();
        for (uint64_t p = i; p < j; p++) {
            if (!(keys[p] & ZK_REC_INVALID)) {
                const typename T::Pt q = T::load(pts, p);
                if (has) T::add(acc, q);
                else acc = q;
                has = true;
            }
        }
        if (has) T::store(dest, k, acc);
    }
}

// payload records of key k in [b, e), one after another; true if there are any
template <class T>
__device__ __forceinline__ bool sum_records(const uint32_t* keys, const uint4* pts, uint64_t b, uint64_t e,
                                            uint32_t k, typename T::Pt& acc) {
    bool has = false;
    acc = T::identity();
    for (uint64_t p = b; p < e; p++) {
        if (keys[p] != k) continue;  // another run's, or no payload
        const typename T::Pt q = T::load(pts, p);
        if (has) T::add(acc, q);
        else acc = q;
        has = true;
    }
    return has;
}

template <class T>
__global__ __launch_bounds__(256) void k_merge_lists(const uint32_t* __restrict__ keys,
                                                     const uint4* __restrict__ pts, uint64_t nrec,
                                                     uint4* __restrict__ dest, MergeLists L, MergeCaps cap) {
    __shared__ uint4 lds[4 * T::kPtBytes / 16];
    constexpr uint32_t kTeams = 256 / T::kLanes;
    const uint32_t team = threadIdx.x / T::kLanes, wteam = team % T::kPerWave;
    // the spans: a block each, consecutive records per team
    const uint32_t nspan = min(L.counts[1], cap.spans);
    for (uint32_t s = blockIdx.x; s < nspan; s += gridDim.x) {  // uniform per block
        const uint2 sp = L.spans[s];
        const uint64_t start = sp.x, end = min(nrec, (start / kMergeSpan + 1) * kMergeSpan);
        const uint32_t k = keys[start] & ZK_REC_KEYMASK;
        constexpr uint32_t kEach = kMergeSpan / kTeams;
        const uint64_t b = min(start + (uint64_t)team * kEach, end), e = min(b + kEach, end);
        typename T::Pt acc;
        (void)sum_records<T>(keys, pts, b, e, k, acc);
        block_tree<T>(acc, kTeams, lds);
        // (a run of more than kMergeMid records holds payloads: a lane inside
        // a bucket leaves one in its first record)
        if (team == 0) T::store(sp.y == ~0u ? dest : L.part, sp.y == ~0u ? k : sp.y, acc);
    }
    // the mid runs: a wave each
    const uint32_t nmid = min(L.counts[0], cap.mid);
    constexpr uint32_t kEach = kMergeMid / T::kPerWave;
    for (uint64_t r = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6); r < nmid; r += (uint64_t)gridDim.x * 4) {
        const uint64_t start = L.mid[r], end = min(nrec, start + kMergeMid);
        const uint32_t k = keys[start] & ZK_REC_KEYMASK;
        const uint64_t b = min(start + (uint64_t)wteam * kEach, end), e = min(b + kEach, end);
        typename T::Pt acc;
        const bool has = sum_records<T>(keys, pts, b, e, k, acc);
        wave_tree<T>(acc, T::kPerWave);
        if (__any(has) && wteam == 0) T::store(dest, k, acc);
    }
}

template <class T>
__global__ __launch_bounds__(256) void k_merge_spans(uint4* __restrict__ dest, MergeLists L, MergeCaps cap) {
    __shared__ uint4 lds[4 * T::kPtBytes / 16];
    constexpr uint32_t kTeams = 256 / T::kLanes;
    const uint32_t team = threadIdx.x / T::kLanes;
    const uint32_t nruns = min(L.counts[3], cap.runs);
    for (uint32_t r = blockIdx.x; r < nruns; r += gridDim.x) {  // uniform per block
        const uint4 run = L.runs[r];
        typename T::Pt acc = T::identity();
        if (team < run.y) acc = T::load(L.part, run.x + team);
        for (uint32_t s = team + kTeams; s < run.y; s += kTeams) {
            const typename T::Pt q = T::load(L.part, run.x + s);
            T::add(acc, q);
        }
        uint32_t P = 1;
        while (P < kTeams && P < run.y) P <<= 1;
        block_tree<T>(acc, P, lds);
        if (team == 0) T::store(dest, run.z, acc);
    }
}

// ------------------------------------------------------ bucket reduction
// Window sum S = sum_k (k+1) B_k over bucket keys k < 2^(c-1).  Write
// k = hi * 2^g + lo (g = (c-1)/2 low bits, h = c-1-g high bits).  Then
//   S = U + sum_{b<g} 2^b Pl_b + sum_{b<h} 2^(g+b) Ph_b,
//   U = sum_lo C_lo,  Pl_b = sum_{lo: bit b} C_lo,  Ph_b = sum_{hi: bit b} R_hi,
// with row sums R_hi = sum_lo B_{hi,lo} and column sums C_lo = sum_hi B_{hi,lo}
// (two additions per bucket in all).  k_br_rowcol: a row of 2^g buckets is
// summed by reduce_teams(2^g, per) teams (about `per` buckets each, then a
// tree), a column of 2^h buckets likewise; the rows and the columns of a
// segment start on block boundaries, so the tree's width is block-uniform.
// k_br_bits: one block per output point j of segment s: j = 0 -> U, 1..g ->
// Pl_{j-1}, g+1..c-1 -> Ph_{j-1-g}.  The host (bits[s*16 + j]) or
// k_tail_windows (plane j over the segment's bucket j, whose sums are taken by
// then: c planes, 2^(c-1) buckets) applies the powers of 2.  Small calls are bound by the depth of the two
// kernels' chains: 256 points (16 windows of 128 buckets) 79 us with one lane
// per addition, 26 us with teams.

__device__ __forceinline__ void seg_shape(uint32_t nbk, uint32_t& g, uint32_t& h) {
    const uint32_t cb = 31 - __clz(nbk);  // c - 1
    g = cb >> 1;
    h = cb - g;
}

template <class T>
__global__ __launch_bounds__(256) void k_br_rowcol(const SegDesc* __restrict__ segs,
                                                   const uint64_t* __restrict__ seg_blk0,
                                                   const uint64_t* __restrict__ seg_rc0, uint32_t nseg,
                                                   uint32_t per, const uint4* __restrict__ buckets,
                                                   uint4* __restrict__ rc) {
    __shared__ uint4 lds[4 * T::kPtBytes / 16];
    constexpr uint32_t kTeams = 256 / T::kLanes;
    const uint32_t s = upper_index(seg_blk0, nseg, blockIdx.x);
    const SegDesc sg = segs[s];
    uint32_t g, h;
    seg_shape(sg.nbk, g, h);
    const uint32_t nrow = 1u << h, ncol = 1u << g;
    const uint32_t Pr = reduce_teams(ncol, per, kTeams), Pc = reduce_teams(nrow, per, kTeams);
    const uint32_t row_blocks = (nrow * Pr + kTeams - 1) / kTeams;
    uint32_t blk = blockIdx.x - (uint32_t)seg_blk0[s];
    const bool rows = blk < row_blocks;
    if (!rows) blk -= row_blocks;
    const uint32_t P = rows ? Pr : Pc;
    const uint32_t li = blk * kTeams + threadIdx.x / T::kLanes;
    const uint32_t nitem = rows ? nrow : ncol;
    const uint32_t item = min(li / P, nitem - 1), part = li % P;  // past the end: the last item again
    const uint32_t len = rows ? ncol : nrow;  // buckets per item
    const uint32_t cnt = len / P;  // buckets this team sums
    auto bucket = [&](uint32_t e) {
        const uint32_t x = part * cnt + e;
        return T::load(buckets, sg.bkt0 + (rows ? ((uint64_t)item << g) + x : ((uint64_t)x << g) + item));
    };
    // the next bucket is loaded while this one is added (one wave per SIMD has
    // nothing else to hide the load behind)
    typename T::Pt acc = bucket(0), q = bucket(min(1u, cnt - 1));
#pragma unroll 1
    for (uint32_t e = 1; e < cnt; e++) {
        const typename T::Pt next = bucket(min(e + 1, cnt - 1));
        T::add(acc, q);
        q = next;
    }
    block_tree<T>(acc, P, lds);
    if (li / P < nitem && part == 0) T::store(rc, seg_rc0[s] + (rows ? item : nrow + item), acc);
}

// One lane per addition, for the points that fill the chip this way
template <class F>
struct LaneG1 {
    using Pt = QXyzz;
    using Team = TeamG1<F>;
    static __device__ __forceinline__ Pt load(const uint4* b, uint64_t i) { return load_qxyzz(b, i); }
    static __device__ __forceinline__ void store(uint4* b, uint64_t i, const Pt& p) { store_qxyzz(b, i, p); }
    static __device__ __forceinline__ void add(Pt& a, const Pt& b) { Arith<F>::qxyzz_add(a, b); }
};
struct LaneG2 {
    using Pt = QXyzz2;
    using Team = TeamG2;
    static __device__ __forceinline__ Pt load(const uint4* b, uint64_t i) { return load_qxyzz2(b, i); }
    static __device__ __forceinline__ void store(uint4* b, uint64_t i, const Pt& p) { store_qxyzz2(b, i, p); }
    static __device__ __forceinline__ void add(Pt& a, const Pt& b) { G2Arith::add(a, b); }
};

// k_br_rowcol for bucket sets that give every SIMD a wave of one-lane chains:
// a row or column is split over P lanes (`per` buckets each); their sums meet
// in LDS, where teams add four each and a tree finishes.  A full wave of
// one-lane additions takes less per addition than four waves of teams (squares
// and merged reductions, no exchanges), the tree of teams less than a tree of
// lanes: at 2^22 points (262,144 buckets) 107 us with both by lanes, 100 us
// with both by teams, 76 us this way; 64 MSMs of 2^15 buckets 547, 637, 453;
// G2 at 2^20 points (524,288 buckets) 599, 486, 372.  Bound by the issue of
// the additions: 8 x 7 us of the 76 at 2^22 points.
template <class C>
__global__ __launch_bounds__(256) void k_br_rowcol_lanes(const SegDesc* __restrict__ segs,
                                                         const uint64_t* __restrict__ seg_blk0,
                                                         const uint64_t* __restrict__ seg_rc0, uint32_t nseg,
                                                         uint32_t per, const uint4* __restrict__ buckets,
                                                         uint4* __restrict__ rc) {
    using T = typename C::Team;
    __shared__ uint4 lds[256 * T::kPtBytes / 16];
    constexpr uint32_t kTeams = 256 / T::kLanes;
    const uint32_t s = upper_index(seg_blk0, nseg, blockIdx.x);
    const SegDesc sg = segs[s];
    uint32_t g, h;
    seg_shape(sg.nbk, g, h);
    const uint32_t nrow = 1u << h, ncol = 1u << g;
    const uint32_t Pr = reduce_teams(ncol, per, kTeams), Pc = reduce_teams(nrow, per, kTeams);
    const uint32_t row_blocks = (nrow * Pr + 255) / 256;
    uint32_t blk = blockIdx.x - (uint32_t)seg_blk0[s];
    const bool rows = blk < row_blocks;
    if (!rows) blk -= row_blocks;
    const uint32_t P = rows ? Pr : Pc;
    const uint32_t li = blk * 256 + threadIdx.x;
    const uint32_t nitem = rows ? nrow : ncol;
    const uint64_t rc0 = seg_rc0[s] + (rows ? 0 : nrow);
    const uint32_t cnt = (rows ? ncol : nrow) / P;  // buckets this lane sums
    if (li < nitem * P) {
        const uint32_t item = li / P, part = li % P;
        auto bucket = [&](uint32_t e) {
            const uint32_t x = part * cnt + e;
            return C::load(buckets, sg.bkt0 + (rows ? ((uint64_t)item << g) + x : ((uint64_t)x << g) + item));
        };
        typename C::Pt acc = bucket(0), q = bucket(min(1u, cnt - 1));
#pragma unroll 1
        for (uint32_t e = 1; e < cnt; e++) {
            const typename C::Pt next = bucket(min(e + 1, cnt - 1));
            C::add(acc, q);
            q = next;
        }
        if (P == 1) C::store(rc, rc0 + item, acc);
        else C::store(lds, threadIdx.x, acc);
    }
    if (P == 1) return;
    __syncthreads();
    // the block's 256 / P items: tpi teams each, of up to four partials
    const uint32_t each = min(P, 4u), tpi = P / each, item0 = blk * (256 / P);
    for (uint32_t t = threadIdx.x / T::kLanes; t < 256 / each; t += kTeams) {
        if (item0 + t / tpi >= nitem) break;  // whole waves or groups: tpi <= kPerWave
        typename T::Pt acc = T::load(lds, t * each);
#pragma unroll 1
        for (uint32_t e = 1; e < each; e++) {
            const typename T::Pt q = T::load(lds, t * each + e);
            T::add(acc, q);
        }
        wave_tree<T>(acc, tpi);
        if (t % tpi == 0) T::store(rc, rc0 + item0 + t / tpi, acc);
    }
}

// index of the i-th value with bit b set: insert a 1 at bit position b
__device__ __forceinline__ uint32_t with_bit(uint32_t i, uint32_t b) {
    return ((i >> b) << (b + 1)) | (1u << b) | (i & ((1u << b) - 1u));
}

// (blockDim.x: a wave per point where the segments' points fill the chip,
// else up to four)
template <class T>
__global__ __launch_bounds__(256) void k_br_bits(const SegDesc* __restrict__ segs,
                                                 const uint64_t* __restrict__ seg_rc0,
                                                 const uint4* __restrict__ rc, uint4* __restrict__ bits,
                                                 int host_form, CallBack back) {
    __shared__ uint4 lds[4 * T::kPtBytes / 16];
    write_back(back);
    const uint32_t s = blockIdx.x >> 4, j = blockIdx.x & 15u;
    const SegDesc sg = segs[s];
    uint32_t g, h;
    seg_shape(sg.nbk, g, h);
    if (j > g + h) return;
    const uint64_t R0 = seg_rc0[s], C0 = R0 + (1u << h);
    // element list: U -> all columns; Pl_b -> columns with bit b; Ph_b -> rows with bit b
    uint64_t base;
    uint32_t count, b = 0;
    bool masked;
    if (j == 0) {
        base = C0; count = 1u << g; masked = false;
    } else if (j <= g) {
        base = C0; b = j - 1; count = 1u << (g - 1); masked = true;
    } else {
        base = R0; b = j - 1 - g; count = 1u << (h - 1); masked = true;
    }
    // count is a power of 2: teams take elements team, team + P, ...; teams past
    // P repeat the first ones'
    const uint32_t P = min(count, blockDim.x / T::kLanes), team = threadIdx.x / T::kLanes;
    if (tree_idle(P, team, T::kPerWave)) return;
    auto element = [&](uint32_t i) { return T::load(rc, base + (masked ? with_bit(i, b) : i)); };
    typename T::Pt acc = element(team & (P - 1));
#pragma unroll 1
    for (uint32_t i = team + P; i < count; i += P) T::add(acc, element(i));
    block_tree<T>(acc, P, lds);
    if (threadIdx.x < T::kLanes) {
        if (host_form) T::store_host(bits, blockIdx.x, acc);  // for the host tail
        else T::store(bits, sg.bkt0 + j, acc);                // for k_tail_windows
    }
}

// ------------------------------------------------ window combine on the device
// The device form of the call's tail (the host form is Engine::run's
// host_tail): result_j = sum_w 2^(cstep w) S_w over the MSM's segments w,
// S_w = U_w + sum_{t < c-1} 2^t Q_{w,t}, the planes k_br_bits stored over the
// segment's first buckets (U, then Q_t), then the affine normalisation;
// cstep = c for plain windows, 0 for window-shifted segments (a plain sum).
// The reference does its window combine on the host
// (Sources/zkMetal/MSM/MSMEngine.swift:899-904); on the device it lets a
// captured graph end with one sum per MSM.  The doubling chain is inherently
// serial (2^127 S_top needs 127 doublings): sixteen teams per segment compute
// S_w, then one team per MSM runs the Horner over segments.

// k_tail_windows: sixteen teams per segment: team t < c - 1 doubles plane Q_t
// t times, team 15 holds U, then a tree sums the sixteen.  The longest chain
// is c - 2 doublings and four additions (64 segments: 104 us with one lane
// per plane, 43 us with teams).
template <class T>
__global__ __launch_bounds__(16 * T::kLanes) void k_tail_windows(const SegDesc* __restrict__ segs,
                                                                const MsmDesc* __restrict__ msms,
                                                                const uint4* __restrict__ bits,
                                                                uint4* __restrict__ wins, int host_form,
                                                                CallBack back) {
    __shared__ uint4 lds[4 * T::kPtBytes / 16];
    write_back(back);
    const uint32_t s = blockIdx.x, t = threadIdx.x / T::kLanes;
    const uint32_t c = msms[segs[s].msm].c;
    const uint64_t b0 = segs[s].bkt0;
    // plane t (c - 1 <= 15 of them) or U; the identity in between
    const bool plane = t + 1 < c, has = plane || t == 15;
    typename T::Pt v = T::load(bits, has ? b0 + (plane ? 1 + t : 0) : b0);
    v = T::select(has, v, T::identity());
    const uint32_t n = plane ? t : 0;
#pragma unroll 1
    for (uint32_t i = 0; i < n; i++) v = T::dbl(v);
    block_tree<T>(v, 16, lds);
    if (t != 0) return;
    if (host_form) T::store_host(wins, s, v);
    else T::store(wins, s, v);
}

// one team per MSM: the MSM's sum in the host form (128 B) into out, or (norm)
// in the stored form over its first segment's sum, for k_tail_normalise.  An
// inversion here costs 150-205 us, its chain of products in one lane; the host
// shares one among 64 sums.
template <class T>
__global__ __launch_bounds__(64) void k_tail_combine(const MsmDesc* __restrict__ msms, uint32_t nmsm,
                                                     uint4* __restrict__ wins, uint4* __restrict__ out,
                                                     int norm, CallBack back) {
    if (!norm) write_back(back);
    const uint32_t j = (blockIdx.x * 64 + threadIdx.x) / T::kLanes;
    if (j >= nmsm) return;
    const MsmDesc m = msms[j];
    typename T::Pt acc = T::load(wins, m.seg0 + m.nseg - 1);
#pragma unroll 1
    for (int w = (int)m.nseg - 2; w >= 0; w--) {
        // 2^cstep acc (window-shifted segments: cstep = 0, their sums already
        // carry the window weights)
#pragma unroll 1
        for (uint32_t i = 0; i < m.cstep; i++) acc = T::dbl(acc);
        T::add(acc, T::load(wins, m.seg0 + w));
    }
    if (norm) T::store(wins, m.seg0, acc);
    else T::store_host(out, j, acc);
}

// result slot j (96 B): the normalised Jacobian X | Y | Z in the 2^256
// Montgomery form, canonical: (x, y, 1), the identity (1, 1, 0).  One lane per
// MSM, one inversion each (150 us whatever their number).
template <class F>
__global__ __launch_bounds__(64) void k_tail_normalise(const MsmDesc* __restrict__ msms, uint32_t nmsm,
                                                       const uint4* __restrict__ wins,
                                                       uint4* __restrict__ out, CallBack back) {
    using A = Arith<F>;
    write_back(back);
    const uint32_t j = blockIdx.x * 64 + threadIdx.x;
    if (j >= nmsm) return;
    const QXyzz p = load_qxyzz(wins, msms[j].seg0);
    const Fq one = A::fq_one();
    Fp x = A::fq_to_fp(one), y = x, z = fp_zero();
    if (!A::qxyzz_is_id(p)) {
        // 1/ZZ = ZZZ / (ZZ ZZZ), 1/ZZZ = ZZ / (ZZ ZZZ): one inversion
        const Fq inv = A::fq_inv(A::fq_mul(p.ZZ, p.ZZZ));
        z = x;
        x = A::fq_to_fp(A::fq_mul(p.X, A::fq_mul(p.ZZZ, inv)));
        y = A::fq_to_fp(A::fq_mul(p.Y, A::fq_mul(p.ZZ, inv)));
    }
    uint4* o = out + (uint64_t)j * 6;
    store_fp(o, x);
    store_fp(o + 2, y);
    store_fp(o + 4, z);
}

// ------------------------------------------------------ test entry point
// out[i] = p[i] + q[i] (dbl: 2 p[i]) on host-form points, by teams
template <class T>
__global__ __launch_bounds__(64) void k_test_team(int dbl, const uint4* __restrict__ p, const uint4* __restrict__ q,
                                                  uint4* __restrict__ out, uint64_t n) {
    const uint64_t i = ((uint64_t)blockIdx.x * 64 + threadIdx.x) / T::kLanes;
    if (i >= n) return;
    using F = typename T::Field;
    auto coord = [&](const uint4* b) {
        return T::A::fq_from_fp_canon(canon32<F>(load_fp(b + (i * T::kLanes + T::lane()) * 2)));
    };
    typename T::Pt a = coord(p);
    const typename T::Pt b = coord(q);
    if (dbl) a = T::dbl(a);
    else T::add(a, b);
    T::store_host(out, i, a);
}

// ------------------------------------------------------------ launchers

void launch_test_team(CurveId cv, bool dbl, const void* p, const void* q, void* out, uint64_t n, hipStream_t st) {
    if (!n) return;
    const unsigned blocks = (unsigned)((n * team_lanes(cv) + 63) / 64);
    const uint4 *a = (const uint4*)p, *b = (const uint4*)q;
    if (cv == CurveId::Grumpkin)
        hipLaunchKernelGGL(k_test_team<TeamG1<Bn254Fr>>, dim3(blocks), dim3(64), 0, st, dbl, a, b, (uint4*)out, n);
    else if (cv == CurveId::Bn254G2)
        hipLaunchKernelGGL(k_test_team<TeamG2>, dim3(blocks), dim3(64), 0, st, dbl, a, b, (uint4*)out, n);
    else
        hipLaunchKernelGGL(k_test_team<TeamG1<Bn254Fp>>, dim3(blocks), dim3(64), 0, st, dbl, a, b, (uint4*)out, n);
}

template <class T>
static void merge_t(const uint32_t* keys, const void* pts, uint64_t nrec, void* dest, const MergeLists& L,
                    const MergeCaps& cap, hipStream_t st) {
    const uint64_t teams = (nrec + 1) / 2, per_block = 256 / T::kLanes;
    hipLaunchKernelGGL(k_merge_runs<T>, dim3((unsigned)((teams + per_block - 1) / per_block)), dim3(256), 0, st, keys,
                       (const uint4*)pts, nrec, (uint4*)dest, L, cap);
    // grid-stride over the lists (their lengths are known on the device only)
    hipLaunchKernelGGL(k_merge_lists<T>, dim3(std::min<uint32_t>(cap.spans + cap.mid / 4, 1024)), dim3(256), 0, st,
                       keys, (const uint4*)pts, nrec, (uint4*)dest, L, cap);
    hipLaunchKernelGGL(k_merge_spans<T>, dim3(std::min<uint32_t>(cap.runs, 256)), dim3(256), 0, st, (uint4*)dest, L,
                       cap);
}

MergeCaps merge_caps(uint64_t nrec) {
    // a mid run has more than kMergeShort records, a long run more than
    // kMergeMid; every boundary inside a run adds a span, and a run with one
    // inside is in the run list
    const uint64_t bounds = nrec / kMergeSpan + 1;
    MergeCaps c;
    c.mid = (uint32_t)(nrec / (kMergeShort + 1) + 1);
    c.spans = (uint32_t)(nrec / (kMergeMid + 1) + 1 + bounds);
    c.runs = (uint32_t)bounds;
    c.parts = (uint32_t)(2 * bounds);
    return c;
}

// the lists in one allocation: runs and partials (16-byte records), spans, mid
uint64_t merge_lists_bytes(uint64_t nrec, CurveId cv) {
    const MergeCaps c = merge_caps(nrec);
    return (uint64_t)c.parts * point_bytes(cv) + (uint64_t)c.runs * 16 + (uint64_t)c.spans * 8 + (uint64_t)c.mid * 4;
}

void launch_merge_runs(CurveId cv, const uint32_t* keys, const void* pts, uint64_t nrec, void* dest,
                       uint32_t* counts, void* lists, hipStream_t st) {
    if (!nrec) return;
    const MergeCaps cap = merge_caps(nrec);
    uint8_t* p = (uint8_t*)lists;
    MergeLists L;
    L.counts = counts;
    L.part = (uint4*)p;
    p += (uint64_t)cap.parts * point_bytes(cv);
    L.runs = (uint4*)p;
    p += (uint64_t)cap.runs * 16;
    L.spans = (uint2*)p;
    p += (uint64_t)cap.spans * 8;
    L.mid = (uint32_t*)p;
    if (cv == CurveId::Grumpkin) merge_t<TeamG1<Bn254Fr>>(keys, pts, nrec, dest, L, cap, st);
    else if (cv == CurveId::Bn254G2) merge_t<TeamG2>(keys, pts, nrec, dest, L, cap, st);
    else merge_t<TeamG1<Bn254Fp>>(keys, pts, nrec, dest, L, cap, st);
}

template <class C>
static void bucket_reduce_t(const SegDesc* segs, const uint64_t* seg_blk0, const uint64_t* seg_rc0,
                            uint32_t nseg, uint64_t blocks, uint32_t per, bool by_lanes, const void* buckets,
                            void* rc, void* bits, bool host_form, const CallBack& back, hipStream_t st) {
    using T = typename C::Team;
    if (by_lanes)
        hipLaunchKernelGGL(k_br_rowcol_lanes<C>, dim3((unsigned)blocks), dim3(256), 0, st, segs, seg_blk0, seg_rc0,
                           nseg, per, (const uint4*)buckets, (uint4*)rc);
    else
        hipLaunchKernelGGL(k_br_rowcol<T>, dim3((unsigned)blocks), dim3(256), 0, st, segs, seg_blk0, seg_rc0, nseg,
                           per, (const uint4*)buckets, (uint4*)rc);
    const uint32_t waves = nseg > 32 ? 1 : nseg > 16 ? 2 : 4;  // of one of ~1000 points
    hipLaunchKernelGGL(k_br_bits<T>, dim3(nseg * 16), dim3(64 * waves), 0, st, segs, seg_rc0, (const uint4*)rc,
                       (uint4*)bits, host_form ? 1 : 0, back);
}

void launch_bucket_reduce(CurveId cv, const SegDesc* segs, const uint64_t* seg_blk0, const uint64_t* seg_rc0,
                          uint32_t nseg, uint64_t blocks, uint32_t per, bool by_lanes, const void* buckets, void* rc,
                          void* bits, bool host_form, const CallBack& back, hipStream_t st) {
    if (!blocks || !nseg) return;
    if (cv == CurveId::Grumpkin)
        bucket_reduce_t<LaneG1<Bn254Fr>>(segs, seg_blk0, seg_rc0, nseg, blocks, per, by_lanes, buckets, rc, bits,
                                             host_form, back, st);
    else if (cv == CurveId::Bn254G2)
        bucket_reduce_t<LaneG2>(segs, seg_blk0, seg_rc0, nseg, blocks, per, by_lanes, buckets, rc, bits, host_form,
                                back, st);
    else
        bucket_reduce_t<LaneG1<Bn254Fp>>(segs, seg_blk0, seg_rc0, nseg, blocks, per, by_lanes, buckets, rc, bits,
                                             host_form, back, st);
}

template <class F>
static void tail_t(const SegDesc* segs, const MsmDesc* msms, uint32_t nseg, uint32_t nmsm, const void* bits,
                   void* wins, void* out, bool norm, const CallBack& back, hipStream_t st) {
    using T = TeamG1<F>;
    hipLaunchKernelGGL(k_tail_windows<T>, dim3(nseg), dim3(16 * T::kLanes), 0, st, segs, msms, (const uint4*)bits,
                       (uint4*)wins, 0, CallBack{});
    hipLaunchKernelGGL(k_tail_combine<T>, dim3((nmsm + T::kPerWave - 1) / T::kPerWave), dim3(64), 0, st, msms, nmsm,
                       (uint4*)wins, (uint4*)out, norm ? 1 : 0, back);
    if (norm)
        hipLaunchKernelGGL(k_tail_normalise<F>, dim3((nmsm + 63) / 64), dim3(64), 0, st, msms, nmsm,
                           (const uint4*)wins, (uint4*)out, back);
}

void launch_tail(CurveId cv, const SegDesc* segs, const MsmDesc* msms, uint32_t nseg, uint32_t nmsm,
                 const void* bits, void* wins, void* out, bool norm, const CallBack& back, hipStream_t st) {
    if (!nseg || !nmsm) return;
    if (cv == CurveId::Grumpkin) tail_t<Bn254Fr>(segs, msms, nseg, nmsm, bits, wins, out, norm, back, st);
    else if (cv == CurveId::Bn254) tail_t<Bn254Fp>(segs, msms, nseg, nmsm, bits, wins, out, norm, back, st);
}

void launch_g2_windows(const SegDesc* segs, const MsmDesc* msms, uint32_t nseg, const void* bits, void* out,
                       const CallBack& back, hipStream_t st) {
    if (!nseg) return;
    hipLaunchKernelGGL(k_tail_windows<TeamG2>, dim3(nseg), dim3(16 * TeamG2::kLanes), 0, st, segs, msms,
                       (const uint4*)bits, (uint4*)out, 1, back);
}

}  // namespace zk
