// kgmt_kernels.hip — HIP kernels of the KGMT per-iteration expansion path (gfx950).
//
// One iteration of the planner is two launches over a table of queries, three
// over more than 256:
//   k_propagate  persistent over tiles of children: Philox draws, per-wave
//                sort by step count, RK4 rollout, AABB test against the
//                obstacles staged in LDS (candidate boxes per wave), region
//                and next-frontier flag of every child, the row of each
//                flagged child (dense per 32-child segment), region counters
//                and new subregion bits summed per tile in LDS, per-chunk
//                flag counts.
//                (KGMT.cu:218-299, statePropagator.cu, collisionCheck.cu)
//   k_update     one workgroup per 1024-element job, old-node chunks then
//                child chunks: region scores with a fixed pairwise summation
//                order (each re-activation job for itself), re-activation of
//                old nodes, compaction of the flagged children, tree append
//                and goal test, and the next expansion list (segmented
//                repeat) at offsets found by a decoupled look-back.
//                (Graph.cu:207-358, KGMT.cu:170-181, 305-403, Planner.cu:52-80)
//   k_finish     (more than 256 queries) one workgroup: closes the iteration of every query (tree
//                size, stop rules, next launch regime; KGMT.cu:84-95, 183-201,
//                399-402) and builds the next iteration's work lists.
// Per plan: k_init (scene build and first iteration's state) before the first
// iteration, and k_paths
// (goal path walk, KGMT.cu:342-361) after the last.
// All sizes stay on the device: the host only polls a completion word that
// the kernels write into host memory.
#include "kgmt_launch.hpp"

#include <utility>

namespace kgmt
{

// ---------------------------------------------------------------------------
// shared helpers
// ---------------------------------------------------------------------------
// total[key]++ for lanes with `has`, valid[key]++ for lanes with `has && ok`:
// one atomic per distinct key held by several lanes (leader loop over the
// ballot; children of one parent share regions, and atomics of every lane on
// a shared counter serialise in the L2). The leader rounds stop at the first key that only one lane holds: the
// remaining lanes then add their own counts (their keys are spread, so
// contention is low). Integer sums: the result is the same either way.
__device__ __forceinline__ void wave_count(int32_t* total, int32_t* validc, int key, bool has, bool ok)
{
    uint64_t pending = __ballot(has);
    while(pending)
        {
            const int leader    = __ffsll((unsigned long long)pending) - 1;
            const int k         = __builtin_amdgcn_readlane(key, leader);
            const uint64_t same = __ballot(has && key == k);
            const uint64_t good = __ballot(has && ok && key == k);
            if((int)lane_id() == leader)
                {
                    atomicAdd(&total[k], (int32_t)__popcll(same));
                    if(good) atomicAdd(&validc[k], (int32_t)__popcll(good));
                }
            pending &= ~same;
            if(__popcll(same) < 2) break;
        }
    if((pending >> lane_id()) & 1ull)
        {
            atomicAdd(&total[key], 1);
            if(ok) atomicAdd(&validc[key], 1);
        }
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_or(uint32_t v)
{
    return v | (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}

// OR of v over the 64 lanes (all active), as a wave-uniform value: DPP within
// each row of 16 lanes, then the four rows' lane 0 read into scalars.
__device__ __forceinline__ uint32_t wave_or(uint32_t v)
{
    v = dpp_or<0xB1>(v);   // quad_perm [1,0,3,2]
    v = dpp_or<0x4E>(v);   // quad_perm [2,3,0,1]
    v = dpp_or<0x141>(v);  // row_half_mirror
    v = dpp_or<0x140>(v);  // row_mirror
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 0) | (uint32_t)__builtin_amdgcn_readlane((int)v, 16) |
           (uint32_t)__builtin_amdgcn_readlane((int)v, 32) | (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
}

// Sets bit `bit` of `words` for every lane with `want`: one atomicOr per
// distinct word per wave, with the OR of that word's lane masks (a wave's
// children come from few parents and mostly fall in the same few words; one
// atomic per lane on a shared word serialises in the L2). Call with every
// lane of the wave.
__device__ __forceinline__ void wave_set_bits(uint32_t* words, uint32_t bit, bool want)
{
    const uint32_t w = bit >> 5, m = 1u << (bit & 31u);
    uint64_t pending = __ballot(want);
    while(pending)
        {
            const int leader    = __ffsll((unsigned long long)pending) - 1;
            const uint32_t k    = (uint32_t)__builtin_amdgcn_readlane((int)w, leader);
            const bool mine     = want && w == k;
            const uint64_t same = __ballot(mine);
            const uint32_t v    = wave_or(mine ? m : 0u);
            if((int)lane_id() == leader) atomicOr(&words[k], v);
            pending &= ~same;
            if(__popcll(same) < 2) break;  // spread words: one atomic per lane below
        }
    if((pending >> lane_id()) & 1ull) atomicOr(&words[w], m);
}

constexpr int kScoreThreads = 1024;
constexpr int kMaxRegions   = 8192;

// v of lane + C (C <= 8: row_shl, only lanes whose source stays in the row
// are used; C >= 16: shuffle)
template <int C>
__device__ __forceinline__ float lane_down(float v)
{
    if constexpr(C <= 8)
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x100 + C, 0xF, 0xF, false));
    else
        return __shfl_down(v, C, 64);
}

// Active subregions of region r (bits r P .. r P + P - 1 of the bitset): one
// word when P divides 32 (the bits never straddle a word), else count_bits.
__device__ __forceinline__ uint32_t region_active(const uint32_t* __restrict__ act, uint32_t r, uint32_t P)
{
    if(P <= 32u && 32u % P == 0u)
        {
            const uint32_t b = r * P;
            const uint32_t m = P == 32u ? 0xffffffffu : ((1u << P) - 1u) << (b & 31u);
            return (uint32_t)__popc(act[b >> 5] & m);
        }
    return count_bits(act, r * P, P);
}

// Raw score of a region with vc > 0 valid children of tc, cnt of its P
// subregions active (Graph.cu:239-257, Q6: fv^4 = (fv*fv)*(fv*fv))
__device__ __forceinline__ float region_raw_score(const QueryDesc& qd, int32_t vc, int32_t tc, uint32_t cnt)
{
    const float eps = qd.cfg.epsilon;
    // cnt / P, as the product with 1 / P when that is exact (same bits)
    const float cov = qd.invP != 0.0f ? (float)cnt * qd.invP : (float)cnt / (float)qd.P;
    const float vf  = (float)vc;
    const float fv  = (eps + vf) / ((eps + vf) + (float)(tc - vc)) * qd.vol;
    const float f2  = fv * fv;
    const float f4  = f2 * f2;
    const float tt  = (float)tc;
    return f4 / ((1.0f + cov) * (1.0f + tt * tt));
}

// Region scores of one query (block of NT threads, R1 <= kMaxRegions). Q6
// semantics: closed formula, then the pairwise sum a[i] += a[i + st] for
// st = P2/2, ..., 1 over the scores padded with zeros to P2 = pow2(R1). Thread
// t owns regions t + k NT: its inputs are loaded together, and the levels with
// st >= NT add a thread's own registers (i and i + st differ by a multiple of
// NT). The NT partial sums then go through LDS once (a: at least NT floats,
// not read after the call): lane l of the first wave takes sums l + 64 j, so
// the levels 64 <= st < NT add the lane's own registers too, and the last six
// levels pair lanes l and l + st within the wave. Every level adds the same
// two partial sums as the plain tree, so the total has the same bits.
template <int NT>
struct ScoreInputs
{
    static constexpr int KR = kMaxRegions / NT;
    int32_t vc[KR], tc[KR];  // valid and total children of regions t + k NT
    uint32_t cnt[KR];        // their active subregions
};

// the inputs of score_regions_sum for thread t (regions t + k NT), loaded
// together; a caller may issue them before it knows whether it needs them
template <int NT>
__device__ __forceinline__ void score_load(const QueryDesc& qd, const int32_t* __restrict__ total,
                                           const int32_t* __restrict__ validc, const uint32_t* __restrict__ act,
                                           ScoreInputs<NT>& in)
{
    const int R1     = qd.R1;
    const uint32_t P = (uint32_t)qd.P;
    const int t      = (int)threadIdx.x;
#pragma unroll
    for(int k = 0; k < ScoreInputs<NT>::KR; ++k)
        {
            const int r = t + k * NT;
            in.vc[k]    = r < R1 ? validc[r] : 0;
            in.tc[k]    = r < R1 ? total[r] : 0;
            in.cnt[k]   = r < R1 ? region_active(act, (uint32_t)r, P) : 0u;
        }
}

template <int NT>
__device__ void score_regions_sum(const QueryDesc& qd, const ScoreInputs<NT>& in, float* __restrict__ score,
                                  float* a);

template <int NT>
__device__ void score_regions(const QueryDesc& qd, const int32_t* __restrict__ total,
                              const int32_t* __restrict__ validc, const uint32_t* __restrict__ act,
                              float* __restrict__ score, float* a)
{
    ScoreInputs<NT> in;
    score_load<NT>(qd, total, validc, act, in);
    score_regions_sum<NT>(qd, in, score, a);
}

template <int NT>
__device__ void score_regions_sum(const QueryDesc& qd, const ScoreInputs<NT>& in, float* __restrict__ score,
                                  float* a)
{
    static_assert(NT % 64 == 0 && NT <= 1024, "score block");
    constexpr int KR = ScoreInputs<NT>::KR;
    const int R1     = qd.R1;
    const float eps  = qd.cfg.epsilon;
    int P2           = 1;
    while(P2 < R1) P2 <<= 1;
    const int t = (int)threadIdx.x;
    const int32_t* vc   = in.vc;
    const int32_t* tc   = in.tc;
    const uint32_t* cnt = in.cnt;
    float s0[KR], sv[KR];
#pragma unroll
    for(int k = 0; k < KR; ++k)
        {
            const float s = vc[k] > 0 ? region_raw_score(qd, vc[k], tc[k], cnt[k]) : 0.0f;
            s0[k] = sv[k] = s;
        }
    int st = P2 / 2;
    for(; st >= NT; st >>= 1)
        {
            const int m = st / NT;
#pragma unroll
            for(int k = 0; k < KR; ++k)
                if(k < m && k + m < KR) sv[k] = sv[k] + sv[k + m];
        }
    // a[i] for i < NT: the thread's own partial sum (zero past P2)
    a[t] = t < P2 ? sv[0] : 0.0f;
    __syncthreads();
    if(t < 64)
        {
            constexpr int NJ = NT / 64;
            float x[NJ];
#pragma unroll
            for(int j = 0; j < NJ; ++j) x[j] = a[t + 64 * j];
            // levels st = 64 m < min(P2, NT): slot j += slot j + m
#pragma unroll
            for(int m = NJ / 2; m >= 1; m >>= 1)
                if(64 * m < P2)
                    {
#pragma unroll
                        for(int j = 0; j < m; ++j) x[j] = x[j] + x[j + m];
                    }
            float v = x[0];
            if(32 < P2) v = v + lane_down<32>(v);
            if(16 < P2) v = v + lane_down<16>(v);
            if(8 < P2) v = v + lane_down<8>(v);
            if(4 < P2) v = v + lane_down<4>(v);
            if(2 < P2) v = v + lane_down<2>(v);
            if(1 < P2) v = v + lane_down<1>(v);
            if(t == 0) a[0] = v;  // after this wave's reads of a
        }
    __syncthreads();
    const float sum = a[0];
#pragma unroll
    for(int k = 0; k < KR; ++k)
        {
            const int r = t + k * NT;
            if(r < R1) score[r] = vc[k] == 0 ? 1.0f : eps + s0[k] / sum;
        }
}

// fAccept (KGMT.cu:387-388): the host computes (itr * EPSILON) * pow(a, 5)
// with a and the first factor in float and pow's double result, and stores
// the product as float; here the fifth power is (a^2)^2 * a in double (a^2
// is exact) and the product is rounded to float once
__device__ __forceinline__ float faccept(const QueryDesc& qd, uint32_t itr, uint32_t tree, uint32_t next)
{
    const float a   = 1.0f - (float)(tree + next) / (float)qd.cap;
    const double ad = (double)a;
    const double a2 = ad * ad;
    const double a5 = (a2 * a2) * ad;
    return (float)((double)((float)itr * qd.cfg.epsilon) * a5);
}

// children per expansion entry and child count (KGMT.cu:183-201, Q9)
__device__ __forceinline__ void launch_regime(const QueryDesc& qd, uint32_t R, uint32_t tree, uint32_t& per,
                                              uint32_t& nChildren)
{
    const uint32_t B     = qd.cfg.children_per_entry;
    const uint32_t avail = qd.cap - tree;
    if((uint64_t)R * B <= avail)
        per = B;
    else
        {
            const uint32_t qv = avail / R;
            per               = qv > B ? B : qv;
            if(per == 0) per = 1;
        }
    const uint64_t nc = (uint64_t)R * per;
    nChildren         = nc > qd.cap ? qd.cap : (uint32_t)nc;
}

// children per tile of a query: a workgroup's lanes, or twice as many for a
// quadcopter query whose children fill the chip anyway
__device__ __forceinline__ uint32_t tile_children(const QueryDesc& qd, const WorkLists& W, uint32_t nC)
{
    return W.refill && qd.cfg.model == KGMT_MODEL_QUADCOPTER && nC >= W.refill ? 2u * W.tile : W.tile;
}

// Work lists of the next iteration into buffer `parity` (block of NT threads,
// run by the last workgroup to arrive).
template <int NT>
__device__ void build_worklists(const QueryDesc* __restrict__ qds, const QueryState* sts, const WorkLists& W,
                                uint32_t parity, uint32_t* sbuf)
{
    const uint32_t nq = W.nq;
    uint32_t* tileStart = W.tileStart + parity * (nq + 1);
    uint32_t* jobStart  = W.jobStart + parity * (nq + 1);
    uint32_t carryT = 0, carryJ = 0, carryA = 0;
    for(uint32_t base = 0; base < nq; base += NT)
        {
            const uint32_t q = base + threadIdx.x;
            uint32_t tiles = 0, jobs = 0, alive = 0;
            if(q < nq)
                {
                    const uint32_t done = __hip_atomic_load(&sts[q].doneN, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if(!done)
                        {
                            const uint32_t nc = __hip_atomic_load(&sts[q].nChildrenN, __ATOMIC_RELAXED,
                                                                  __HIP_MEMORY_SCOPE_AGENT);
                            const uint32_t tr = __hip_atomic_load(&sts[q].treeSizeN, __ATOMIC_RELAXED,
                                                                  __HIP_MEMORY_SCOPE_AGENT);
                            const uint32_t tc = tile_children(qds[q], W, nc);
                            tiles             = (nc + tc - 1) / tc;
                            jobs              = (nc + kChunk - 1) / kChunk + (tr + kChunk - 1) / kChunk;
                            alive             = 1;
                        }
                }
            uint32_t tT, tJ, tA;
            const uint32_t eT = block_excl_scan<NT>(tiles, sbuf, tT);
            const uint32_t eJ = block_excl_scan<NT>(jobs, sbuf, tJ);
            block_excl_scan<NT>(alive, sbuf, tA);
            if(q < nq)
                {
                    tileStart[q] = carryT + eT;
                    jobStart[q]  = carryJ + eJ;
                }
            carryT += tT, carryJ += tJ, carryA += tA;
        }
    if(threadIdx.x == 0)
        {
            tileStart[nq]     = carryT;
            jobStart[nq]      = carryJ;
            *W.counter        = 0;
            __hip_atomic_store(W.allDone, carryA == 0 ? 1u : 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
}

// One more iteration closed in this plan: the count for the host, which
// stays a few launch units ahead of it (one thread per iteration: the closing
// job of a single query, k_finish for many queries)
__device__ __forceinline__ void count_closed(const WorkLists& W)
{
    const uint32_t n = *W.closedDev + 1u;
    *W.closedDev     = n;
    __hip_atomic_store(W.closed, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The same for a few queries, whose iterations no one thread closes: the next
// propagate counts the one before it as it starts.
__device__ __forceinline__ void count_started(const WorkLists& W)
{
    const uint32_t n = *W.closedDev;
    *W.closedDev     = n + 1u;
    __hip_atomic_store(W.closed, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Tiles and jobs of a query's next iteration as one word (0 once it is done).
__device__ __forceinline__ uint64_t query_work(const QueryDesc& qd, const QueryState& st, const WorkLists& W)
{
    if(st.doneN) return 0ull;
    const uint32_t nc = st.nChildrenN, tr = st.treeSizeN, tc = tile_children(qd, W, nc);
    return (uint64_t)((nc + kChunk - 1) / kChunk + (tr + kChunk - 1) / kChunk) << 32 | (nc + tc - 1) / tc;
}

// Starts of the queries' items (tiles: shift 0, jobs: 32) into list (nq + 1
// words of LDS) by a block of NT threads; returns their number.
template <int NT>
__device__ __forceinline__ uint32_t few_starts(const WorkLists& W, uint32_t parity, uint32_t shift, uint32_t* list,
                                               uint32_t* sbuf)
{
    constexpr uint32_t I = kFewQueries > NT ? kFewQueries / NT : 1;
    const uint32_t nq    = W.nq;
    const uint64_t* work = W.work + parity * nq;
    uint32_t v[I], sum = 0;
#pragma unroll
    for(uint32_t i = 0; i < I; ++i)
        {
            const uint32_t q = threadIdx.x * I + i;
            v[i]             = q < nq ? (uint32_t)(work[q] >> shift) : 0u;
            sum += v[i];
        }
    uint32_t tot;
    uint32_t at = block_excl_scan<NT>(sum, sbuf, tot);
#pragma unroll
    for(uint32_t i = 0; i < I; ++i)
        {
            const uint32_t q = threadIdx.x * I + i;
            if(q < nq) list[q] = at;
            at += v[i];
        }
    __syncthreads();
    return tot;
}

// Returns true in every thread of the last workgroup to arrive (all writes of
// the earlier ones are visible to it afterwards).
__device__ __forceinline__ bool last_arrival(uint32_t* counter, uint32_t expected, uint32_t* sflag)
{
    __threadfence();
    __syncthreads();
    if(threadIdx.x == 0)
        {
            const uint32_t prev = atomicAdd(counter, 1u);
            const bool last     = prev == expected - 1;
            // every workgroup has arrived: the counter starts at zero for the
            // next launch
            if(last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *sflag = last ? 1u : 0u;
        }
    __syncthreads();
    const bool last = *sflag != 0;
    if(last) __threadfence();
    return last;
}

// ---------------------------------------------------------------------------
// init (KGMT.cu:50-81): per-query part of k_init, defined after the scene build
// ---------------------------------------------------------------------------
// the cleared region counters, scores, subregion bits, chunk counts and
// job words of one query: thread `rank` of `ranks` clears every ranks-th word
__device__ void clear_query(const QueryDesc& qd, const Pools& P, uint32_t rank, uint32_t ranks)
{
    for(uint32_t r = rank; r < 16u << qd.regShift; r += ranks)
        {
            P.cnt[qd.regOff + r]   = 0ull;
            P.score[qd.regOff + r] = 0.0f;
        }
    for(uint32_t w = rank; w < (uint32_t)qd.R2words; w += ranks)
        {
            P.actPrev[qd.subOff + w] = 0u;
            P.actNext[qd.subOff + w] = 0u;
        }
    for(uint32_t c = rank; c <= qd.nChunks; c += ranks) P.partA[qd.chunkOff + c] = 0u;
    for(uint32_t i = rank; i < 4 * (qd.nChunks + 1); i += ranks) P.look[4 * (size_t)qd.chunkOff + i] = 0ull;
}

// root and the first iteration's state of one query (one workgroup)
__device__ void root_query(const QueryDesc& qd, QueryState& st, const Pools& P)
{
    const uint32_t rootRep = qd.cfg.root_repeat < qd.cap ? qd.cfg.root_repeat : qd.cap;
    for(uint32_t k = threadIdx.x; k < rootRep; k += kBlock) P.repIdx[qd.nodeOff + k] = 0u;
    for(int d = threadIdx.x; d < qd.D; d += kBlock) P.treeS[qd.sampleOff + (size_t)d * qd.cap] = qd.start[d];
    if(threadIdx.x == 0)
        {
            P.parent[qd.nodeOff]   = -1;
            P.grand[qd.nodeOff]    = -1;
            P.anc[qd.nodeOff]      = make_int4(-1, -1, -1, -1);
            P.cost[qd.nodeOff]     = 0.0f;
            P.frontier[qd.nodeOff] = 1;
            int ix, iy, iz;
            P.r1node[qd.nodeOff] = region_of(qd, qd.start[0], qd.start[1], qd.start[2], ix, iy, iz);
            st.itr               = 1;
            st.treeSize          = 1;
            st.R                 = qd.cfg.root_repeat;
            uint32_t per, nc;
            launch_regime(qd, st.R, 1, per, nc);
            st.per       = per;
            st.nChildren = nc;
            st.nAcc = 0, st.next = 0;
            st.fAccept = 0.0f;
            st.done = 0, st.success = 0;
            st.goalIdx  = kNoGoal;
            st.pathRows = 0;
            st.pathCost = 0.0f, st.pathLen = 0.0f;
            st.expanded  = 0;
            st.flagged   = 0;
            st.finishItr = 0;
            st.itrN = st.itr, st.treeSizeN = st.treeSize, st.nChildrenN = st.nChildren, st.perN = st.per;
            st.doneN = 0, st.successN = 0, st.finishItrN = 0, st.padN = 0;
            st.expandedN = 0, st.flaggedN = 0;
        }
}

// ---------------------------------------------------------------------------
// propagate: persistent over 256-child tiles
// ---------------------------------------------------------------------------
// LDS of one propagate tile: the draws of its NT / K children and the order
// in which the lanes take them. The per-wave candidate lists of the two-phase
// check exist only with one lane per child (the only shape that runs it), so
// they take no LDS, and no occupancy, from the other shapes.
template <int NT, int K>
struct TileLds
{
    static constexpr int kCandWaves = K == 1 ? NT / 64 : 1;
    static constexpr int kCandBoxes = K == 1 ? kCand : 1;
    uint32_t hist[NT];      // children per step bucket, then bucket offsets
    uint16_t slot[NT];      // lane -> child of the tile
    float ctrl[KGMT_MAX_CONTROL][NT];
    int32_t steps[NT];
    float ufront[NT];
    uint32_t sbuf[NT / 64 + 1];
    float4 cand[kCandWaves][2 * kCandBoxes];  // per-wave candidate boxes (two-phase check)
    // per-tile sums of the region counters and ORs of the subregion bitset
    // words, flushed with one global atomic per distinct key (open addressing,
    // key -1 = empty; at most NT distinct keys per tile, so a probe always ends)
    int32_t rkey[NT];
    uint32_t rtot[NT], rval[NT];
    int32_t wkey[NT];
    uint32_t wmask[NT];
    // flagged children of the tile, one bit per child, by 32-child segment;
    // two buffers alternating by tile, so a tile empties the other one
    uint32_t fbits[2][NT / 32];
};

// empties thread t's slot of both tables and of flag buffer `fb`
template <int NT, int K>
__device__ __forceinline__ void clear_tables(TileLds<NT, K>& L, uint32_t fb)
{
    const uint32_t t = threadIdx.x;
    L.rkey[t] = -1, L.rtot[t] = 0, L.rval[t] = 0;
    L.wkey[t] = -1, L.wmask[t] = 0;
    if(t < NT / 32) L.fbits[fb][t] = 0;
}

// slot of `key` in an NT-entry open-addressing table of LDS keys (claimed by
// compare-and-swap); the table holds fewer than NT other keys
template <int NT>
__device__ __forceinline__ uint32_t tab_slot(int32_t* keys, int32_t key)
{
    uint32_t slot = ((uint32_t)key * 2654435761u) & (uint32_t)(NT - 1);
    for(;;)
        {
            const int32_t old = atomicCAS(&keys[slot], -1, key);
            if(old == -1 || old == key) return slot;
            slot = (slot + 1) & (uint32_t)(NT - 1);
        }
}

// row v of flagged children: parent and grandparent bits, sample, zero
// padding, in whole float4 stores
template <int S, int C>
__device__ __forceinline__ void store_row(float* rows, uint32_t v, int32_t p, int32_t gp, const float* s,
                                          const float* uc, float dur)
{
    constexpr int D = S + C + 1, RW = row_words(D);
    float w[RW];
    w[0] = __int_as_float(p);
    w[1] = __int_as_float(gp);
#pragma unroll
    for(int d = 0; d < S; ++d) w[2 + d] = s[d];
#pragma unroll
    for(int k = 0; k < C; ++k) w[2 + S + k] = uc[k];
    w[D + 1] = dur;
#pragma unroll
    for(int e = D + 2; e < RW; ++e) w[e] = 0.0f;
    float4* row = reinterpret_cast<float4*>(rows + (size_t)v * RW);
#pragma unroll
    for(int j = 0; j < RW / 4; ++j) row[j] = make_float4(w[4 * j], w[4 * j + 1], w[4 * j + 2], w[4 * j + 3]);
}

// word and bit of subregion r2 (r1 P + local) in the planner's bitsets
__device__ __forceinline__ void subregion_bit(const QueryDesc& qd, int r1, int r2, uint32_t& word, uint32_t& bit)
{
    const uint32_t sub = (uint32_t)(r2 - r1 * qd.P);
    word               = region_word((uint32_t)r1, qd.regShift, qd.actW) + (sub >> 5);
    bit                = 1u << (sub & 31u);
}

// a tile's children and valid children of region r, one atomic for both
// (the low word would carry past 2^32 children of one region in a plan)
__device__ __forceinline__ void count_region(const QueryDesc& qd, const Pools& P, uint32_t r, uint32_t total,
                                             uint32_t valid)
{
    atomicAdd(reinterpret_cast<unsigned long long*>(P.cnt + qd.regOff + region_slot(r, qd.regShift)),
              (unsigned long long)valid << 32 | total);
}

// One tile of TC = NT / K children u = base .. base + TC - 1 of a query (TC
// divides kChunk, so a tile never straddles two chunks), K lanes per child.
// Every child writes its flag and region; a flagged child (the only ones the
// tree append reads) also writes its row and parent, at the next free slot of
// its 32-child segment (segment start + flagged children before it in the
// segment), so the rows of a segment are dense. fb: this tile's flag buffer.
// The children are drawn in tile order, then handed to the lane groups
// longest-first (counting sort on the step count) so that each wave's groups
// integrate about the same number of steps. The K lanes of a group integrate
// the same edge (same operations, same bits) and split its box tests; the
// group's first lane writes the child. Each child still writes only its own
// slot and the counters are integer atomics, so the outputs do not depend on
// the order or on K.
template <int MODEL, int NT, int K>
__device__ __forceinline__ void child_tile(const QueryDesc& qd, const QueryState& st, uint32_t base,
                                           const Pools& P, float4* sObs, TileLds<NT, K>& L, uint32_t fb,
                                           bool stage)
{
    constexpr int S = ModelDims<MODEL>::S, C = ModelDims<MODEL>::C;
    static_assert(K > 1 || MODEL != KGMT_MODEL_QUADCOPTER, "one lane per child: quad_tile");
    constexpr uint32_t TC = NT / K;
    const uint32_t nC  = st.nChildrenN;
    const uint32_t cap = qd.cap;
    const size_t nodeO = qd.nodeOff;
    const uint32_t t   = threadIdx.x;
    const uint32_t per = st.perN;
    const float* T     = P.treeS + qd.sampleOff;
    // K == 1: the parent of child t (tile order) and its state, loaded while
    // the draws and the sort run; after the sort the wave passes them to the
    // lanes that take the children, through its candidate area (written
    // again only by the two-phase check)
    static_assert(K > 1 || (2 + S) * 64 <= 8 * TileLds<NT, K>::kCandBoxes, "parent stage fits a wave's candidates");
    uint32_t pp = 0;
    int32_t pg  = -1;
    float ps[S];
#pragma unroll
    for(int d = 0; d < S; ++d) ps[d] = 0.0f;
    const bool pre = K == 1 && t < TC && base + t < nC;
    if(pre) pp = P.repIdx[nodeO + (base + t) / per];
    // the query's scene into LDS on the workgroup's first tile of it (its
    // loads in flight with the parent index)
    if(stage)
        {
            stage_scene(P.obs, qd.obsOff, qd.nGrp, sObs);
            __syncthreads();
        }
    // draws of the child in tile order
    {
        const uint32_t un = base + t;
        float uc[C];
        int32_t steps = 0;
        float uf      = 0.0f;
        // K == 1: each wave sorts its own 64 children (they come from one or
        // two parents, so the wave's edges stay close together and share few
        // candidate boxes); K > 1: the whole tile is sorted
        constexpr uint32_t BW = K == 1 ? 64u : (uint32_t)NT;  // buckets per sorted group
        const uint32_t g0     = K == 1 ? (t / 64u) * 64u : 0u;
        uint32_t bucket       = g0 + BW - 1;                  // past the end: last
        if(t < TC && un < nC)
            {
                draw_child<C>(qd.cfg, qd.cfg.query_id, st.itrN, un, uc, steps, uf);
                const int32_t k = steps - qd.cfg.steps_min;
                bucket = g0 + (BW - 2) - (uint32_t)(k < (int32_t)BW - 2 ? k : (int32_t)BW - 2);
            }
        L.hist[t] = 0;
        if constexpr(K == 1)
            {
                // The wave's 64 buckets hold exactly its 64 lanes, so its
                // offsets are a wave scan from g0, and every LDS word written
                // here is read only by this wave: no workgroup barrier (the
                // LDS runs one wave's operations in order; the wave barriers
                // keep the compiler from reordering them).
                wave_sync();
                const uint32_t rank = atomicAdd(&L.hist[bucket], 1u);
                wave_sync();
                const uint32_t h = L.hist[t];
                L.hist[t]        = g0 + wave_incl_scan(h) - h;
                wave_sync();
                L.slot[L.hist[bucket] + rank] = (uint16_t)t;
#pragma unroll
                for(int k = 0; k < C; ++k) L.ctrl[k][t] = uc[k];
                L.steps[t]  = steps;
                L.ufront[t] = uf;
                if(pre)
                    {
#pragma unroll
                        for(int d = 0; d < S; ++d) ps[d] = T[(size_t)d * cap + pp];
                        pg = P.parent[nodeO + pp];
                    }
                // parent, grandparent and state of child t at word j * 64 + t % 64
                float* stg          = reinterpret_cast<float*>(L.cand[t / 64]);
                const uint32_t l    = t % 64u;
                stg[l]              = __uint_as_float(pp);
                stg[64 + l]         = __int_as_float(pg);
#pragma unroll
                for(int d = 0; d < S; ++d) stg[(2 + d) * 64 + l] = ps[d];
                wave_sync();
            }
        else
            {
                __syncthreads();
                uint32_t rank = 0;
                if(t < TC) rank = atomicAdd(&L.hist[bucket], 1u);
                __syncthreads();
                uint32_t tot;
                const uint32_t off = block_excl_scan<NT>(L.hist[t], L.sbuf, tot);
                L.hist[t]          = off;
                __syncthreads();
                if(t < TC)
                    {
                        L.slot[L.hist[bucket] + rank] = (uint16_t)t;
#pragma unroll
                        for(int k = 0; k < C; ++k) L.ctrl[k][t] = uc[k];
                        L.steps[t]  = steps;
                        L.ufront[t] = uf;
                    }
                __syncthreads();
            }
    }
    const uint32_t i    = L.slot[t / K];
    const uint32_t u    = base + i;
    const bool has      = u < nC;
    const bool lead     = K == 1 || t % K == 0;
    int r1              = 0;
    bool ok = false, fn = false;
    bool setBit   = false;  // valid child in a subregion unseen at iteration start
    uint32_t word = 0, bit = 0;  // of the subregion
    uint32_t p         = 0;
    int32_t gp         = -1;  // parent of the parent
    float s[S], uc[C];
    int32_t steps = 0;
    float uf      = 0.0f;
#pragma unroll
    for(int d = 0; d < S; ++d) s[d] = 0.0f;
#pragma unroll
    for(int k = 0; k < C; ++k) uc[k] = 0.0f;
    if(has)
        {
            if constexpr(K == 1)
                {
                    // child i is one of this wave's 64
                    const float* stg = reinterpret_cast<const float*>(L.cand[t / 64]);
                    const uint32_t l = i % 64u;
                    p                = __float_as_uint(stg[l]);
                    gp               = __float_as_int(stg[64 + l]);
#pragma unroll
                    for(int d = 0; d < S; ++d) s[d] = stg[(2 + d) * 64 + l];
                }
            else
                {
                    p = P.repIdx[nodeO + u / per];
#pragma unroll
                    for(int d = 0; d < S; ++d) s[d] = T[(size_t)d * cap + p];
                    gp = P.parent[nodeO + p];
                }
#pragma unroll
            for(int k = 0; k < C; ++k) uc[k] = L.ctrl[k][i];
            steps = L.steps[i];
            uf    = L.ufront[i];
        }
    if constexpr(K == 1) wave_sync();  // the stage is read before the check writes candidates
    const Scene sc{sObs, (int)qd.nGrp, (int)(t % K)};
    if constexpr(K == 1)
        ok = propagate_two_phase<MODEL>(qd, s, uc, steps, sc, L.cand[t / 64], has);  // every lane
    else if(has)
        ok = propagate<MODEL, K>(qd, s, uc, steps, sc);
    if(has)
        {
            if(lead)
                {
                    // region ids and the loads they need first: a load issued
                    // after the stores would wait for them (one in-order counter)
                    int ix, iy, iz;
                    r1 = region_of(qd, s[0], s[1], s[2], ix, iy, iz);
                    if(ok)
                        {
                            const int r2 = subregion_of(qd, s[0], s[1], s[2], r1, ix, iy, iz);
                            subregion_bit(qd, r1, r2, word, bit);
                            const bool seen = (P.actPrev[qd.subOff + word] & bit) != 0u;
                            fn              = (uf < P.score[qd.regOff + r1]) || !seen;
                            setBit          = !seen;
                        }
                    if(u % per == 0) P.frontier[nodeO + p] = 0;
                    P.r1child[nodeO + u] = r1;
                    P.fnext[nodeO + u]   = fn ? 1 : 0;
                    if(fn) atomicOr(&L.fbits[fb][i >> 5], 1u << (i & 31u));
                }
        }
    // region counters and new subregion bits: summed per tile in LDS, then
    // one global atomic per distinct region / bitset word
    if(has && lead)
        {
            const uint32_t e = tab_slot<NT>(L.rkey, r1);
            atomicAdd(&L.rtot[e], 1u);
            if(ok) atomicAdd(&L.rval[e], 1u);
        }
    if(setBit)
        {
            const uint32_t e = tab_slot<NT>(L.wkey, (int32_t)word);
            atomicOr(&L.wmask[e], bit);
        }
    // the tile lies inside one 1024-element chunk
    const uint64_t fm = __ballot(fn);
    if(lane_id() == 0 && fm) atomicAdd(&P.partA[qd.chunkOff + base / kChunk], (uint32_t)__popcll(fm));
    __syncthreads();
    if(fn)
        {
            // row slot: segment start + flagged children before it
            const uint32_t v = !dense_rows(MODEL) ? u
                               : base + (i & ~31u) +
                                   (uint32_t)__popc(L.fbits[fb][i >> 5] & ((1u << (i & 31u)) - 1u));
            store_row<S, C>(P.childR + qd.rowOffC, v, (int32_t)p, gp, s, uc, qd.cfg.dt * (float)steps);
        }
    {
        const int32_t rk = L.rkey[t];
        if(rk >= 0) count_region(qd, P, (uint32_t)rk, L.rtot[t], L.rval[t]);
        const int32_t wk = L.wkey[t];
        if(wk >= 0) atomicOr(&P.actNext[qd.subOff + (uint32_t)wk], L.wmask[t]);
        // empty for the next tile, which uses the other flag buffer (this
        // tile's is emptied by the next one, after the barrier below)
        clear_tables(L, fb ^ 1u);
    }
    __syncthreads();  // L is reused by the next tile
}

// ---------------------------------------------------------------------------
// quadcopter tiles, one lane per child
// ---------------------------------------------------------------------------
// Most edges of a quadcopter end long before their drawn 10 to 50 steps (out
// of the workspace, past a speed bound, in a box: 8 to 16 steps on average on
// the configured queries), and a step is about 1090 instructions, so a wave
// that runs until its longest edge ends leaves more than half of its lanes
// idle (2.0 to 2.5 times the steps needed). A tile's lanes are therefore
// looked over every kQuadSteps steps: with children left, once 64 lanes are
// free they take new ones; with none left, the lanes still running move out
// of the last wave as soon as the waves before it have room, and the wave
// idles (its SIMD goes to other workgroups): 1.3 to 1.6 times the steps needed.
// The last 64 children take a quad of lanes each: a lone wave's step costs the
// launch its whole length (160 children: 50 steps). Where each child runs does
// not change its result. With the mask check in place of the group bounds:
// three configured quadcopter queries 29.2 -> 19.9 ms a plan, the mixed batch
// of 512 queries 112 -> 35.7 ms (propagate launches 444 -> 295 and 1154 ->
// about 340 us, 239 and 295 with quad_ode's shorter divisions and roots, 211 and
// 268 with the longest edges first); bound by vector issue, then by the length
// of the longest edge.
constexpr int kQuadSteps = 4;
constexpr int kMoveWords = 20;  // a running child: state, controls, frontier uniform, steps left, index and steps, parent

template <int NT>
struct QuadRunLds
{
    float move[kMoveWords][64];
    uint32_t order[64];        // slots of the last children, most steps left first
    uint32_t cnt[2][NT / 64];  // running lanes per wave, alternating
};

// A child of a quadcopter tile
struct QuadChild
{
    float s[12], u[4], uf;  // state (at the start, then at the end of the edge), controls, frontier uniform
    int left;               // steps left; 0: the edge ended valid; -1: invalid
    uint32_t meta;          // index in the tile | steps << 10
    uint32_t p;             // parent
};

// Runs the children 0 .. count - 1 (at most 2 NT) of a workgroup of NT threads:
// steps(i) tells a child's steps, take(i, ch) fills it (state, controls, steps
// into left), done(ch) takes the finished one; take and done are called once
// per child, in any order and lane. More children than lanes start in the
// order of their steps, the longest first, so that no long edge begins when
// the others end (a quadcopter plan's propagate launches 240 to 211 us).
// Barriers inside, the last before the last calls of done: call uniformly.
template <int NT, class STEPS, class TAKE, class DONE>
__device__ __forceinline__ void quad_run(const QueryDesc& qd, uint32_t count, const MaskScene& sc, QuadRunLds<NT>& L,
                                         STEPS steps, TAKE take, DONE done)
{
    constexpr int S = 12, C = 4, NW = NT / 64;
    // children left when a quad of lanes takes each: a quad's step costs half
    // an instruction more per child than half a wave of single lanes
    constexpr int kTail = NT / 4 < 64 ? NT / 4 : 64;
    const int t    = (int)threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(t / 64);
    QuadChild ch;
    bool held = false, run = false;  // a child in this lane; still running
    MaskWalk walk{0, 0, 0};
#pragma unroll
    for(int d = 0; d < S; ++d) ch.s[d] = 0.0f;
#pragma unroll
    for(int k = 0; k < C; ++k) ch.u[k] = 0.0f;
    ch.uf = 0.0f, ch.left = 0, ch.meta = 0u, ch.p = 0u;
    // the child's words into / out of slot m of L.move
    auto put = [&](uint32_t m) {
#pragma unroll
        for(int d = 0; d < S; ++d) L.move[d][m] = ch.s[d];
#pragma unroll
        for(int k = 0; k < C; ++k) L.move[S + k][m] = ch.u[k];
        L.move[16][m] = ch.uf, L.move[17][m] = __int_as_float(ch.left);
        L.move[18][m] = __uint_as_float(ch.meta), L.move[19][m] = __uint_as_float(ch.p);
    };
    auto get = [&](uint32_t m) {
#pragma unroll
        for(int d = 0; d < S; ++d) ch.s[d] = L.move[d][m];
#pragma unroll
        for(int k = 0; k < C; ++k) ch.u[k] = L.move[S + k][m];
        ch.uf = L.move[16][m], ch.left = __float_as_int(L.move[17][m]);
        ch.meta = __float_as_uint(L.move[18][m]), ch.p = __float_as_uint(L.move[19][m]);
    };
    // The order of the children, by a counting sort over 64 ranges of steps; in
    // the words of L.move, which hold running children only once all are taken.
    // (Children that all start at once gain nothing by it: 100003 edges and the
    // mixed batch 1 % slower.)
    uint16_t* order = reinterpret_cast<uint16_t*>(L.move);
    uint32_t* hist  = reinterpret_cast<uint32_t*>(L.move) + NT;
    static_assert(NT + 64 <= kMoveWords * 64, "the order of 2 NT children and the ranges fit");
    const bool sorted = count > NT;
    if(sorted)
    {
        const kgmt_config& k = qd.cfg;
        const float scale    = 64.0f / (float)(k.steps_max - k.steps_min + 1);
        if(t < 64) hist[t] = 0u;
        __syncthreads();
        uint32_t b[2], r[2];
#pragma unroll
        for(int j = 0; j < 2; ++j)
            {
                const uint32_t i = (uint32_t)t + (uint32_t)j * NT;
                if(i >= count) continue;
                const float f = fminf(fmaxf((float)(k.steps_max - steps(i)) * scale, 0.0f), 63.0f);
                b[j] = (uint32_t)f, r[j] = atomicAdd(&hist[b[j]], 1u);
            }
        __syncthreads();
        if(t < 64)
            {
                const uint32_t h = hist[t];
                hist[t]          = wave_incl_scan(h) - h;
            }
        __syncthreads();
#pragma unroll
        for(int j = 0; j < 2; ++j)
            {
                const uint32_t i = (uint32_t)t + (uint32_t)j * NT;
                if(i < count) order[hist[b[j]] + r[j]] = (uint16_t)i;
            }
    }
    uint32_t next = 0;   // children taken
    uint32_t rest = 0;   // children left to the quads of lanes
    int W         = NW;  // waves that may hold running lanes
    uint32_t par  = 0;
    while(true)
        {
            // running lanes of every wave (the first round's barrier also
            // covers what the caller staged)
            const uint64_t mine = __ballot(run);
            if(lane_id() == 0) L.cnt[par][wave] = (uint32_t)__popcll(mine);
            __syncthreads();
            const uint32_t* now = L.cnt[par];
            uint32_t cw[NW], total = 0;
#pragma unroll
            for(int k = 0; k < NW; ++k) cw[k] = now[k], total += cw[k];
            par ^= 1u;
            const bool more = next < count;
            const bool fill = more && (NT - total >= 64u);
            while(!more && W > 1 && now[W - 1] == 0u) --W;
            const bool end  = !more && total <= (uint32_t)kTail;
            const bool drop = !end && !more && W > 1 && total <= 64u * (uint32_t)(W - 1);
            if(fill || drop || end)
                {
                    if(held && !run)
                        {
                            held = false;
                            done(ch);
                        }
                    const uint64_t lower = (1ull << lane_id()) - 1ull;
                    if(end)
                        {
                            // the children still running, to the quads below
                            uint32_t rank = (uint32_t)__popcll(mine & lower);
#pragma unroll
                            for(int k = 0; k < NW; ++k) rank += k < wave ? cw[k] : 0u;
                            if(run) put(rank);
                            rest = total;
                            break;
                        }
                    // rank among the lanes that take something
                    uint32_t rank = (uint32_t)__popcll(~mine & lower);
#pragma unroll
                    for(int k = 0; k < NW; ++k) rank += k < wave ? 64u - cw[k] : 0u;
                    if(fill)
                        {
                            if(!run && next + rank < count)
                                {
                                    const uint32_t i = sorted ? order[next + rank] : next + rank;
                                    take(i, ch);
                                    walk.start(qd, ch.s[0], ch.s[1], ch.s[2]);
                                    ch.meta = i | (uint32_t)ch.left << 10;
                                    held    = true;
                                    run     = ch.left > 0;
                                }
                            next = next + (NT - total) < count ? next + (NT - total) : count;
                        }
                    else
                        {
                            // the last wave's lanes to the free lanes before it
                            --W;
                            const uint32_t movers = now[W];
                            if(wave == W && run)
                                {
                                    put((uint32_t)__popcll(mine & lower));
                                    held = run = false;
                                }
                            __syncthreads();
                            if(wave < W && !run && rank < movers)
                                {
                                    get(rank);
                                    walk.start(qd, ch.s[0], ch.s[1], ch.s[2]);
                                    held = run = true;
                                }
                        }
                }
            for(int k = 0; k < kQuadSteps; ++k)
                {
                    if(!__any(run)) break;
                    if(run)
                        {
                            const float px = ch.s[0], py = ch.s[1], pz = ch.s[2];
                            quad_step(qd, ch.s, ch.u);
                            const bool out = quad_out(qd.cfg, ch.s);
                            const bool hit = walk.hit(qd, sc, px, py, pz, ch.s[0], ch.s[1], ch.s[2], !out);
                            ch.left        = (out | hit) ? -1 : ch.left - 1;
                            run            = ch.left > 0;
                        }
                }
        }
    if(!rest) return;
    // the last children, a quad of lanes each, until they end; the longest
    // first, so that a wave's 16 end together
    __syncthreads();
    const uint32_t m = (uint32_t)t / 4u;
    const int c      = (t & 3) < 3 ? (t & 3) : 2;
    run              = m < rest;
    if(run)
        {
            // children before child m: more steps left, or as many and a lower slot
            const int own   = __float_as_int(L.move[17][m]);
            uint32_t before = 0;
            for(uint32_t k = (uint32_t)t & 3u; k < rest; k += 4)
                {
                    const int o = __float_as_int(L.move[17][k]);
                    before += o > own || (o == own && k < m) ? 1u : 0u;
                }
            before += quad_perm<0xB1>(before);
            before += quad_perm<0x4E>(before);
            L.order[before] = m;
        }
    __syncthreads();
    const uint32_t r = run ? L.order[m] : 0u;
    QuadLane ql;
    ql.c = c;
    ql.x = L.move[c][r], ql.a = L.move[3 + c][r], ql.v = L.move[6 + c][r], ql.w = L.move[9 + c][r];
    ql.qa  = c == 0 ? qd.qax : c == 1 ? qd.qay : qd.qaz;
    ql.qb  = c == 0 ? qd.qbx : c == 1 ? qd.qby : qd.qbz;
    ql.thr = qd.qminv * L.move[12][r], ql.tor = ql.qb * L.move[13 + c][r];
    int left = __float_as_int(L.move[17][r]);
    int i    = slab_of(ql.x, qd.cfg.ws_min, qd.slabScale);
    while(__any(run))
        {
            if(run)
                {
                    const float px = ql.x;
                    ql.step(qd);
                    left = ql.ends(qd, sc, px, i) ? -1 : left - 1;
                    run  = left > 0;
                }
        }
    if(m < rest)
        {
            if((t & 3) < 3)
                L.move[c][r] = ql.x, L.move[3 + c][r] = ql.a, L.move[6 + c][r] = ql.v, L.move[9 + c][r] = ql.w;
            else
                L.move[17][r] = __int_as_float(left);
        }
    wave_sync();  // a child's words stay within its quad
    if(m < rest && (t & 3) == 0)
        {
            get(r);
            done(ch);
        }
}

template <int NT>
struct QuadLds
{
    static constexpr int kTile = 2 * NT;  // most children of a tile
    // sums per region and bitset word, as in TileLds
    int32_t rkey[kTile];
    uint32_t rtot[kTile], rval[kTile];
    int32_t wkey[kTile];
    uint32_t wmask[kTile];
    QuadRunLds<NT> run;
};

template <int NT>
__device__ __forceinline__ void quad_tile(const QueryDesc& qd, const QueryState& st, uint32_t base, uint32_t tile,
                                          const Pools& P, float4* sObs, QuadLds<NT>& L, bool stage)
{
    constexpr int S = 12, C = 4;
    constexpr int kT   = QuadLds<NT>::kTile;
    const uint32_t nC  = st.nChildrenN, per = st.perN, itr = st.itrN;
    const uint32_t cap = qd.cap;
    const size_t nodeO = qd.nodeOff;
    const float* T     = P.treeS + qd.sampleOff;
    for(int k = (int)threadIdx.x; k < kT; k += NT)
        {
            L.rkey[k] = -1, L.rtot[k] = 0, L.rval[k] = 0;
            L.wkey[k] = -1, L.wmask[k] = 0;
        }
    const MaskScene sc = stage_masks(P.obs, qd.obsOff, qd.nGrp, qd.nObs, sObs, stage);
    quad_run<NT>(
      qd, nC - base < tile ? nC - base : tile, sc, L.run,
      [&](uint32_t i) { return draw_steps<C>(qd.cfg, qd.cfg.query_id, itr, base + i); },
      [&](uint32_t i, QuadChild& ch) {
          const uint32_t u = base + i;
          ch.p             = P.repIdx[nodeO + u / per];
          draw_child<C>(qd.cfg, qd.cfg.query_id, itr, u, ch.u, ch.left, ch.uf);
#pragma unroll
          for(int d = 0; d < S; ++d) ch.s[d] = T[(size_t)d * cap + ch.p];
      },
      [&](const QuadChild& ch) {
          const uint32_t u = base + (ch.meta & 1023u);
          const bool ok    = ch.left == 0;
          bool fn = false, setBit = false;
          uint32_t word = 0, bit = 0;
          int ix, iy, iz;
          const int r1 = region_of(qd, ch.s[0], ch.s[1], ch.s[2], ix, iy, iz);
          if(ok)
              {
                  const int r2 = subregion_of(qd, ch.s[0], ch.s[1], ch.s[2], r1, ix, iy, iz);
                  subregion_bit(qd, r1, r2, word, bit);
                  const bool seen = (P.actPrev[qd.subOff + word] & bit) != 0u;
                  fn              = (ch.uf < P.score[qd.regOff + r1]) || !seen;
                  setBit          = !seen;
              }
          if(u % per == 0) P.frontier[nodeO + ch.p] = 0;
          P.r1child[nodeO + u] = r1;
          P.fnext[nodeO + u]   = fn ? 1 : 0;
          const uint32_t e     = tab_slot<kT>(L.rkey, r1);
          atomicAdd(&L.rtot[e], 1u);
          if(ok) atomicAdd(&L.rval[e], 1u);
          if(setBit)
              {
                  const uint32_t f = tab_slot<kT>(L.wkey, (int32_t)word);
                  atomicOr(&L.wmask[f], bit);
              }
          // the tile lies inside one 1024-element chunk
          const uint64_t fm = __ballot(fn);
          if(fn)
              {
                  if((int)lane_id() == __ffsll((unsigned long long)fm) - 1)
                      atomicAdd(&P.partA[qd.chunkOff + base / kChunk], (uint32_t)__popcll(fm));
                  store_row<S, C>(P.childR + qd.rowOffC, u, (int32_t)ch.p, P.parent[nodeO + ch.p], ch.s, ch.u,
                                  qd.cfg.dt * (float)(ch.meta >> 10));
              }
      });
    __syncthreads();
    for(int k = (int)threadIdx.x; k < kT; k += NT)
        {
            const int32_t rk = L.rkey[k];
            if(rk >= 0) count_region(qd, P, (uint32_t)rk, L.rtot[k], L.rval[k]);
            const int32_t wk = L.wkey[k];
            if(wk >= 0) atomicOr(&P.actNext[qd.subOff + (uint32_t)wk], L.wmask[k]);
        }
}

// LDS of a propagate workgroup: its model's tile state
template <int MODEL, int NT, int K>
union PropagateLds
{
    TileLds<NT, K> tile;
    QuadLds<NT> quad;
};
template <int NT>
union PropagateLds<KGMT_MODEL_QUADCOPTER, NT, 1>
{
    QuadLds<NT> quad;
};
template <int MODEL, int NT, int K>
constexpr bool kUseTile = !(MODEL == KGMT_MODEL_QUADCOPTER && K == 1);
template <int MODEL, int NT, int K>
constexpr bool kUseQuad = (MODEL == KGMT_MODEL_QUADCOPTER || MODEL < 0) && K == 1;

template <int MODEL, int NT, int K>
__global__ __launch_bounds__(NT, 4) void k_propagate(const QueryDesc* __restrict__ qds,
                                                  QueryState* __restrict__ sts, Pools P, WorkLists W,
                                                  uint32_t parity)
{
    static_assert(NT % 64 == 0 && kChunk % (NT / K) == 0, "tile size");
    extern __shared__ float4 sObs[];
    __shared__ PropagateLds<MODEL, NT, K> L;
    const uint32_t nq        = W.nq;
    // the first workgroup commits the next-state fields (written when the
    // last iteration closed) to the current ones, which the update kernel
    // reads; propagate itself reads only the next-state fields
    // (a done query's word for the iteration after the next stays empty)
    const bool few = W.few();
    if(blockIdx.x == 0)
        {
            for(uint32_t q = threadIdx.x; q < nq; q += NT)
                {
                    commit_state(sts[q]);
                    if(few && sts[q].doneN) W.work[(parity ^ 1u) * nq + q] = 0ull;
                }
            if(few && threadIdx.x == 0) count_started(W);
        }
    // the tiles: one query's straight from its state, a few queries' scanned
    // by every workgroup, more queries' from the list
    const uint32_t* starts = W.tiles(parity);
    uint32_t nTiles;
    if(nq == 1)
        {
            const uint32_t nc = sts[0].nChildrenN, tc = tile_children(qds[0], W, nc);
            nTiles            = sts[0].doneN ? 0u : (nc + tc - 1) >> __builtin_ctz(tc);  // a power of two
        }
    else if(few)
        {
            __shared__ uint32_t sbuf[NT / 64];
            uint32_t* list = reinterpret_cast<uint32_t*>(sObs) + W.listOff;
            nTiles         = few_starts<NT>(W, parity, 0u, list, sbuf);
            starts         = list;
        }
    else
        nTiles = starts[nq];
    uint32_t staged          = 0xffffffffu;
    uint32_t fb              = 0;  // flag buffer of the next tile
    // the tables and both flag buffers start empty (each tile empties them
    // again after its flush; the first tile's staging barrier comes before
    // any insert); used: by a quadcopter tile's state since
    bool used = false;
    if constexpr(kUseTile<MODEL, NT, K>) clear_tables(L.tile, 0u), clear_tables(L.tile, 1u);
    // Workgroup j takes tile j, then, with more tiles than workgroups, every
    // gridDim.x-th tile; where quadcopter tiles are among them (they differ
    // several times in length), the next from a counter instead, fetched while
    // a tile runs (the mixed batch: 45.6 to 41.0 ms a plan; the other models'
    // tiles are short and even, and the fetch at their start cost them 2 to
    // 4 %). The other parity's counter starts at zero for the next launch.
    constexpr bool claim = kUseQuad<MODEL, NT, K>;
    __shared__ uint32_t sNext[2];
    if(claim && blockIdx.x == 0 && threadIdx.x == 0) W.tileClaim[parity ^ 1u] = 0u;
    uint32_t turn = 0;
    for(uint32_t t = blockIdx.x; t < nTiles; t = claim ? sNext[turn] : t + gridDim.x, turn ^= 1u)
        {
            if(claim && threadIdx.x == 0)
                sNext[turn] = nTiles > gridDim.x ? gridDim.x + __hip_atomic_fetch_add(W.tileClaim + parity, 1u,
                                                                                      __ATOMIC_RELAXED,
                                                                                      __HIP_MEMORY_SCOPE_AGENT)
                                                 : nTiles;
            const uint32_t q     = nq == 1 ? 0u : locate(starts, nq, t);
            const uint32_t first = nq == 1 ? 0u : (uint32_t)__builtin_amdgcn_readfirstlane((int)starts[q]);
            if(sts[q].doneN)
                {
                    if(claim) __syncthreads();
                    continue;  // stale list entry of a finished query
                }
            const QueryDesc& qd = qds[q];
            // a new query's scene: the tile stages it (after the barrier
            // that ends the last tile, so no wave still reads the old one)
            const bool stage = q != staged;
            staged           = q;
            const int model  = MODEL >= 0 ? MODEL : qd.cfg.model;
            if constexpr(kUseQuad<MODEL, NT, K>)
                if(model == KGMT_MODEL_QUADCOPTER)
                    {
                        const uint32_t tile = tile_children(qd, W, sts[q].nChildrenN);
                        quad_tile<NT>(qd, sts[q], (t - first) * tile, tile, P, sObs, L.quad, stage);
                        used = true;
                        continue;
                    }
            if constexpr(kUseTile<MODEL, NT, K>)
                {
                    if(used)
                        {
                            __syncthreads();
                            clear_tables(L.tile, 0u), clear_tables(L.tile, 1u);
                            __syncthreads();
                            used = false;
                        }
                    const uint32_t base = (t - first) * (NT / K);
                    if constexpr(MODEL >= 0)
                        child_tile<MODEL, NT, K>(qd, sts[q], base, P, sObs, L.tile, fb, stage);
                    else
                        {
                            // (a batch never mixes planar and 3D queries, so
                            // a mixed batch holds no unicycle)
                            if(model == KGMT_MODEL_DOUBLE_INTEGRATOR)
                                child_tile<KGMT_MODEL_DOUBLE_INTEGRATOR, NT, K>(qd, sts[q], base, P, sObs, L.tile, fb, stage);
                            else if(model == KGMT_MODEL_DUBINS_AIRPLANE)
                                child_tile<KGMT_MODEL_DUBINS_AIRPLANE, NT, K>(qd, sts[q], base, P, sObs, L.tile, fb, stage);
                            else if(model == KGMT_MODEL_DUBINS_5D)
                                child_tile<KGMT_MODEL_DUBINS_5D, NT, K>(qd, sts[q], base, P, sObs, L.tile, fb, stage);
                            else if constexpr(!kUseQuad<MODEL, NT, K>)
                                child_tile<KGMT_MODEL_QUADCOPTER, NT, K>(qd, sts[q], base, P, sObs, L.tile, fb, stage);
                        }
                    fb ^= 1u;
                }
        }
}

// ---------------------------------------------------------------------------
// closing an iteration
// ---------------------------------------------------------------------------
// End of an iteration for one query (one thread): tree size, stop rules,
// next launch regime. The goal path is walked once the plan has ended
// (k_paths).
__device__ void finish_query(const QueryDesc& qd, QueryState& st, uint32_t R)
{
    const uint32_t tree = st.treeSize + st.next;
    uint32_t itr = st.itr, per = st.per, nc = st.nChildren, done = 0, success = 0, fin = st.finishItr;
    if(st.goalIdx != kNoGoal)
        {
            success = 1;
            done    = 1;
            fin     = itr;
        }
    else if(itr >= qd.cfg.max_iter || tree == qd.cap)
        {
            // out of iterations, or a full tree that can take no further node
            done = 1;
            fin  = itr;
        }
    else
        {
            launch_regime(qd, R, tree, per, nc);
            itr = itr + 1;
        }
    st.treeSizeN  = tree;
    st.expandedN  = st.expanded + st.nChildren;
    st.flaggedN   = st.flagged + st.nAcc;
    st.itrN       = itr;
    st.perN       = per;
    st.nChildrenN = nc;
    st.doneN      = done;
    st.successN   = success;
    st.finishItrN = fin;
}

// f(0), .., f(N - 1) with constant indices from the start: an array that only
// they index is split into registers before anything takes it for a vector
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// goal -> root rows of a solved query by one wave (every lane): the chain is
// followed six levels per round of loads (parent, grandparent and the
// ancestors at 3..6), lane l takes the row of the l-th node, and kWaveRows rows
// go out together, the first ones to `first`, those after them to `out` (both
// as if they held the whole path); cost and length (of the edge durations and
// of the segments between node positions) are summed in walk order. stage:
// null, or LDS for kWaveRows rows, through which they go out as whole lines.
__device__ __forceinline__ void walk_path_wave(const QueryDesc& qd, QueryState& st, const Pools& P, float* first,
                                               float* out, float* stage, int32_t goal)
{
    const uint32_t lane    = lane_id();
    const uint32_t cap     = qd.cap;
    const int D            = qd.D;
    const uint32_t maxRows = qd.cfg.max_iter + 2;
    const int32_t* par     = P.parent + qd.nodeOff;
    const int32_t* gpar    = P.grand + qd.nodeOff;
    const int4* anc        = P.anc + qd.nodeOff;
    const float* __restrict__ T = P.treeS + qd.sampleOff;
    uint32_t rows = 0;  // rows out
    int32_t head  = goal;
    float pc = 0.0f, pl = 0.0f, px = 0.0f, py = 0.0f, pz = 0.0f;
    while(true)
        {
            const uint32_t lim = maxRows - rows < kWaveRows ? maxRows - rows : kWaveRows;
            int32_t mine = lane == 0 ? head : -1;  // this lane's node
            int32_t f    = head;                    // the last node found
            uint32_t cnt = 1;                       // nodes found
            bool root    = false;                   // the chain ended at the root
            while(!root && cnt < lim)
                {
                    const int32_t p = par[f], g = gpar[f];
                    const int4 a    = anc[f];
                    const int32_t up[6] = {p, g, a.x, a.y, a.z, a.w};
#pragma unroll
                    for(int j = 0; j < 6; ++j)
                        if(!root && cnt < lim)
                            {
                                if(up[j] < 0 || (uint32_t)up[j] >= cap)  // -1: past the root
                                    root = true;
                                else
                                    {
                                        if(lane == cnt) mine = up[j];
                                        f = up[j];
                                        ++cnt;
                                    }
                            }
                }
            if(!root)
                {
                    head = par[f];
                    root = head < 0 || (uint32_t)head >= cap;
                }
            // a dimension past the sample's repeats the first (never stored)
            float r[KGMT_MAX_SAMPLE];
            const uint32_t node = mine < 0 ? (uint32_t)f : (uint32_t)mine;
            static_for<KGMT_MAX_SAMPLE>([&](auto K) { r[K] = T[(size_t)(K < D ? K : 0) * cap + node]; });
            const float dn = T[(size_t)(D - 1) * cap + node];
            float* to = rows == 0u ? first : out + rows * D;
            if(lane < cnt)
                static_for<KGMT_MAX_SAMPLE>([&](auto K) {
                    if(K < D) (stage ? stage : to)[lane * D + K] = r[K];
                });
            if(stage)
                {
                    // (one wave: its LDS writes come before its reads)
                    __builtin_amdgcn_wave_barrier();
                    for(uint32_t i = lane; i < cnt * (uint32_t)D; i += 64u) to[i] = stage[i];
                    __builtin_amdgcn_wave_barrier();
                }
            // segment length from the row before (lane l - 1, or the last of
            // the rows before) to this one
            float qx = __shfl_up(r[0], 1, 64), qy = __shfl_up(r[1], 1, 64), qz = __shfl_up(r[2], 1, 64);
            if(lane == 0) qx = px, qy = py, qz = pz;
            const float e = pos_dist(qd, qx, qy, qz, r[0], r[1], r[2]);
            // a node's edge duration counts when it has a parent: every node
            // but the root
            for(uint32_t l = 0; l < cnt; ++l)
                {
                    const float dl = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dn), l));
                    if(!(root && l == cnt - 1)) pc = pc + dl;
                    if(rows + l > 0) pl = pl + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e), l));
                }
            rows += cnt;
            if(root || rows >= maxRows) break;
            px = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r[0]), cnt - 1));
            py = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r[1]), cnt - 1));
            pz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r[2]), cnt - 1));
        }
    if(lane == 0)
        {
            st.pathRows = rows;
            st.pathCost = pc;
            st.pathLen  = pl;
        }
}

// How a single-query plan ended.
struct Outcome
{
    uint32_t success, iterations, treeSize;
    int32_t goal;
    uint64_t expanded, flagged;
};

// End of a single-query plan (one thread; a solved plan's path rows are out
// already, walk_path_wave): the result into host-mapped memory, then the
// completion word, so the host can return without waiting for the launches it
// queued past the last iteration (they find the query done and exit). Without
// a host result buffer only the completion word is set.
__device__ __forceinline__ void publish_single(const QueryState& st, const WorkLists& W, const Outcome& r)
{
    if(!W.result)
        {
            __hip_atomic_store(W.allDone, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            return;
        }
    HostResult* h = W.result;
    h->success    = r.success;
    h->iterations = r.iterations;
    h->treeSize   = r.treeSize;
    h->pathRows   = r.success ? st.pathRows : 0u;
    h->goalIdx    = r.success ? r.goal : -1;
    h->pathCost   = r.success ? st.pathCost : 0.0f;
    h->pathLen    = r.success ? st.pathLen : 0.0f;
    h->expanded   = r.expanded;
    h->flagged    = r.flagged;
    __threadfence_system();
    __hip_atomic_store(W.allDone, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------------------
// update: the rest of an iteration in one launch: region scores, tree
// append, goal test, re-activation and the next expansion list
// (Graph.cu:207-358, KGMT.cu:305-403)
// ---------------------------------------------------------------------------
// A query's jobs, in the order of their entries in the next expansion list:
// its old-node chunks (one entry per re-activated node, ascending), then its
// child chunks (each appended node repeated 15 or 1 times). A job finds the
// entries before it by a decoupled look-back (Merrill and Garland,
// "Single-pass Parallel Prefix Scan with Decoupled Look-back", 2016) over one
// 64-bit word per job (two sets, by iteration parity; each launch empties
// the other set for the next): it publishes its own count and smallest goal
// node (aggregate) as soon as it has them, reads the words before it until
// one holds a prefix that includes its job (inclusive), and then publishes
// its own inclusive word. A job waits only for jobs held by workgroups that
// are running, and those publish their aggregates without waiting, so every
// wait ends: with no more jobs than workgroups, workgroup j does job j (the
// dispatcher starts the workgroups of an XCD in index order, so a workgroup
// whose predecessor has not started leaves that predecessor's XCD slots to
// lower-index workgroups or to other kernels, all of which finish); with
// more, workgroups take jobs from a counter in order. The wait is bounded all
// the same (kLookBackPolls); a job that runs out sets the error word, which
// the host reports, and goes on with what it has.
// Every job derives the iteration's totals it needs itself rather than
// waiting for a launch that computes them once: the flagged children of all
// chunks (and of the chunks before its own) from the chunk counts, and, for
// a re-activation job, the region scores (their sum is one fixed pairwise
// tree, so every job gets the same bits). Job 0 stores the scores and the
// subregion snapshot that the next propagate reads.
// update workgroups: kUpd threads, each taking kPer consecutive slots of a
// job's chunk (one slot: one block scan covers the chunk, and a thread's
// flag byte is one load), and all of them the region scores
constexpr uint32_t kUpd = 4 * kBlock;
constexpr uint32_t kPer = kChunk / kUpd;
static_assert(kPer == 1, "one slot per thread");
constexpr uint32_t kLbNone        = (1u << 27) - 1;  // no goal node (node indices stay below 2^26)
constexpr uint64_t kLbAggregate   = 1ull << 62;
constexpr uint64_t kLbInclusive   = 2ull << 62;
constexpr uint32_t kLookBackPolls = 1u << 20;

// Arguments of k_update; read in place (fresh), not copied into registers.
struct UpdateArgs
{
    const QueryDesc* qds;
    QueryState* sts;
    Pools P;
    WorkLists W;
    uint32_t parity, own;
};

// v, in constant memory (kernel arguments, a descriptor), as a reference whose
// fields are loaded where they are used after this point. Without it the
// compiler loads every field that a job needs anywhere before the job loop,
// runs out of scalar registers and moves them through vector lanes: 87 writes
// in front of the loop and some 150 reads a job, each issued by all 16 waves
// (k_update: 33 Dubins queries 11.4 to 10.1 us a launch, one 11.6 to 10.9,
// one double integrator 10.0 to 9.1, 512 mixed queries 30.0 to 27.7).
template <class T>
__device__ __forceinline__ const T& fresh(const T& v)
{
    const __attribute__((address_space(4))) T* p = (const __attribute__((address_space(4))) T*)&v;
    asm volatile("" : "+s"(p));
    return *(const T*)p;
}

// Place of a region's raw score in LDS: rows of 16 counter slots, padded to 17
// words, so that threads in slot order (the counters' loads) and threads in
// region order (the score tree) both spread over the banks
__device__ __forceinline__ uint32_t raw_index(uint32_t r, uint32_t shift)
{
    return (r & ((1u << shift) - 1u)) * 17u + (r >> shift);
}

// LDS of an update workgroup
struct UpdateLds
{
    union
    {
        float raw[17 * (kMaxRegions / 16)];  // raw region scores (-1: no valid child), at raw_index
        uint32_t stage[kMaxRegions];         // then the job's expansion-list entries
    };
    float part[kUpd];                   // the score tree's partial sums
    uint32_t sbuf[3 * (kUpd / 64)];     // block scans
    uint32_t job, before, goalBefore, nAcc;
    float sum;
};

// word: flag (bits 62-63), smallest goal node (32-58), entries (0-31)
__device__ __forceinline__ uint64_t lb_word(uint64_t flag, uint32_t entries, uint32_t goal)
{
    return flag | ((uint64_t)goal << 32) | entries;
}

__device__ __forceinline__ uint32_t wave_min_u(uint32_t v)
{
#pragma unroll
    for(int o = 32; o > 0; o >>= 1)
        {
            const uint32_t t = (uint32_t)__shfl_xor((int)v, o, 64);
            v                = t < v ? t : v;
        }
    return v;
}

// Entries and smallest goal node of the jobs before job li (words: the
// query's job words); every lane of one wave. A round reads the 256 words
// before `base` (lane l, slot k: word base - 1 - l - 64 k), all loads in
// flight together, so the jobs of one launch (every aggregate published at
// about the same time) find their prefix in one or two round trips. False if
// a word did not appear within the poll bound (the sums then cover the words
// seen).
__device__ bool look_back(const uint64_t* words, uint32_t li, uint32_t& entries, uint32_t& goal)
{
    constexpr int KL   = 4;
    const int32_t lane = (int32_t)lane_id();
    uint32_t c = 0, g = kLbNone, polls = 0;
    int32_t base = (int32_t)li;
    while(true)
        {
            uint64_t w[KL];
#pragma unroll
            for(int k = 0; k < KL; ++k)
                {
                    const int32_t idx = base - 1 - lane - 64 * k;
                    // before the first job: an inclusive word of nothing
                    w[k] = idx >= 0 ? __hip_atomic_load(words + idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                    : lb_word(kLbInclusive, 0u, kLbNone);
                }
            // per slot, the lanes up to and including the nearest inclusive
            // word (none past the slot that holds it)
            uint64_t need[KL];
            bool found = false, wait = false;
#pragma unroll
            for(int k = 0; k < KL; ++k)
                {
                    const uint32_t flag = (uint32_t)(w[k] >> 62);
                    const uint64_t incl = __ballot(flag == 2u);
                    const uint64_t none = __ballot(flag == 0u);
                    need[k] = found ? 0ull : incl ? ((incl & (~incl + 1ull)) << 1) - 1ull : ~0ull;
                    wait    = wait || (none & need[k]) != 0ull;
                    found   = found || incl != 0ull;
                }
            if(wait)
                {
                    if(++polls >= kLookBackPolls)
                        {
                            entries = c, goal = g;
                            return false;
                        }
                    __builtin_amdgcn_s_sleep(1);
                    continue;
                }
            uint32_t wc = 0u, wg = kLbNone;
#pragma unroll
            for(int k = 0; k < KL; ++k)
                if((need[k] >> lane) & 1ull)
                    {
                        wc += (uint32_t)w[k];
                        const uint32_t gk = (uint32_t)(w[k] >> 32) & kLbNone;
                        wg                = gk < wg ? gk : wg;
                    }
            c += (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan(wc), 63);
            const uint32_t gm = wave_min_u(wg);
            g = gm < g ? gm : g;
            if(found)
                {
                    entries = c, goal = g;
                    return true;
                }
            base -= 64 * KL;
        }
}

// Exclusive scan of v and minimum of m over a block of NT threads, one
// barrier pair; sbuf: 2 * NT/64 words. Call uniformly.
template <int NT>
__device__ __forceinline__ uint32_t block_excl_scan_min(uint32_t v, uint32_t m, uint32_t* sbuf, uint32_t& total,
                                                        uint32_t& mmin)
{
    constexpr int NW = NT / 64;
    static_assert(NW >= 2 && NW <= 16, "block of 128 to 1024 threads");
    const uint32_t incl = wave_incl_scan(v);
    const uint32_t lane = lane_id();
    const int wave      = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64));
    if(__ballot(m != kLbNone)) m = wave_min_u(m);
    if(lane == 63) sbuf[wave] = incl, sbuf[NW + wave] = m;
    __syncthreads();
    const uint32_t w  = row_incl_scan(lane < (uint32_t)NW ? sbuf[lane] : 0u);
    const uint32_t pw = wave == 0 ? 0u : (uint32_t)__builtin_amdgcn_readlane((int)w, wave - 1);
    total             = (uint32_t)__builtin_amdgcn_readlane((int)w, NW - 1);
    uint32_t mm       = kLbNone;
#pragma unroll
    for(int i = 0; i < NW; ++i) mm = sbuf[NW + i] < mm ? sbuf[NW + i] : mm;
    mmin = mm;
    __syncthreads();
    return pw + incl - v;
}

// Region scores for a re-activation job (Graph.cu:239-257 per region,
// :297-304 and :349-357 for the sum): raw scores into L.raw (-1 for a region
// without valid children), their sum by the pairwise tree of
// score_regions_sum, here over all kMaxRegions leaves (the levels above the
// query's own padded size add zeros, which leave every partial sum's bits
// unchanged), into L.sum; with the flagged children of the iteration
// (nAcc, acc: this thread's share of the chunk counts) into L.nAcc.
// KB regions per thread (KB kUpd cover the query's). Barriers inside: call
// uniformly.
template <int KB>
__device__ __forceinline__ void job_scores(const QueryDesc& qd, const Pools& P, uint32_t acc, UpdateLds& L)
{
    const uint32_t R1    = (uint32_t)qd.R1;
    const int t          = (int)threadIdx.x;
    const uint32_t sh    = qd.regShift, actW = qd.actW;
    const uint32_t slots = 16u << sh;
    const uint64_t* cnt  = P.cnt + qd.regOff;
    const uint32_t* act  = P.actNext + qd.subOff;
    // KB counter slots per thread, every load issued before any is used
    // (indices clamped into the query's slots, so no load sits behind a
    // branch); up to 64 subregion bits per region lie at the same slots
    uint64_t c[KB];
    uint32_t n[KB];  // active subregions
#pragma unroll
    for(int k = 0; k < KB; ++k)
        {
            const uint32_t i = (uint32_t)t + (uint32_t)k * kUpd;
            c[k]             = cnt[i < slots ? i : slots - 1u];
        }
    auto bits = [&](auto x) {  // x: a region's bits
        using T = decltype(x);
#pragma unroll
        for(int k = 0; k < KB; ++k)
            {
                const uint32_t i = (uint32_t)t + (uint32_t)k * kUpd;
                n[k]             = (uint32_t)__popcll(reinterpret_cast<const T*>(act)[i < slots ? i : slots - 1u]);
            }
    };
    if(actW == 1u)
        bits(uint32_t{});
    else if(actW == 2u)
        bits(uint64_t{});
    else
        {
            // more (in region order): their counts at the places of this
            // thread's raw scores, where the regions with a valid child are
            // marked first: the others' words are not read (8000 regions of
            // 1000 subregions, three iterations: a plan 0.55 to 0.28 ms)
#pragma unroll
            for(int k = 0; k < KB; ++k)
                {
                    const uint32_t i = (uint32_t)t + (uint32_t)k * kUpd;
                    if(i < slots) L.raw[(i >> 4) * 17u + (i & 15u)] = __uint_as_float((int32_t)(c[k] >> 32) > 0 ? 1u : 0u);
                }
#pragma unroll 1
            for(int k = 0; k < KB; ++k)
                {
                    const uint32_t i = (uint32_t)t + (uint32_t)k * kUpd, r = slot_region(i, sh);
                    if(i >= slots || r >= R1) continue;
                    float& raw = L.raw[(i >> 4) * 17u + (i & 15u)];
                    if(__float_as_uint(raw) == 0u) continue;
                    uint32_t m = 0u;
                    for(uint32_t w = 0; w < actW; ++w) m += (uint32_t)__popc(act[(size_t)r * actW + w]);
                    raw = __uint_as_float(m);
                }
        }
#pragma unroll
    for(int k = 0; k < KB; ++k)
        {
            const uint32_t i = (uint32_t)t + (uint32_t)k * kUpd;
            const uint32_t r = slot_region(i, sh);
            const int32_t vc = (int32_t)(c[k] >> 32), tc = (int32_t)(uint32_t)c[k];
            float& raw       = L.raw[(i >> 4) * 17u + (i & 15u)];  // raw_index(r)
            if(i < slots && r < R1)
                raw = vc > 0 ? region_raw_score(qd, vc, tc, actW > 2u ? __float_as_uint(raw) : n[k]) : -1.0f;
        }
    // the flagged children of the iteration, per wave (used after the tree)
    const uint32_t lane    = lane_id();
    const int wave         = __builtin_amdgcn_readfirstlane(t / 64);
    const uint32_t waveAcc = (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan(acc), 63);
    if(lane == 0) L.sbuf[wave] = waveAcc;
    __syncthreads();
    // the thread's leaves t + k kUpd; the levels with stride >= kUpd add
    // the thread's own registers
    float sv[KB];
#pragma unroll
    for(int k = 0; k < KB; ++k)
        {
            const uint32_t r = (uint32_t)t + (uint32_t)k * kUpd;
            const float x    = r < R1 ? L.raw[raw_index(r, sh)] : 0.0f;
            sv[k]            = x < 0.0f ? 0.0f : x;
        }
#pragma unroll
    for(int m = KB / 2; m >= 1; m >>= 1)
        {
#pragma unroll
            for(int k = 0; k < m; ++k) sv[k] = sv[k] + sv[k + m];
        }
    L.part[t] = sv[0];
    __syncthreads();
    if(t < 64)
        {
            // lane l holds partial sums l + 64 j; then the last six levels
            // pair lanes within the wave (as score_regions_sum)
            constexpr int NJ = (int)kUpd / 64;
            float x[NJ];
#pragma unroll
            for(int j = 0; j < NJ; ++j) x[j] = L.part[t + 64 * j];
#pragma unroll
            for(int m = NJ / 2; m >= 1; m >>= 1)
                {
#pragma unroll
                    for(int j = 0; j < m; ++j) x[j] = x[j] + x[j + m];
                }
            float v = x[0];
            v       = v + lane_down<32>(v);
            v       = v + lane_down<16>(v);
            v       = v + lane_down<8>(v);
            v       = v + lane_down<4>(v);
            v       = v + lane_down<2>(v);
            v       = v + lane_down<1>(v);
            if(t == 0)
                {
                    L.sum       = v;
                    uint32_t na = 0;
#pragma unroll
                    for(int w = 0; w < NJ; ++w) na += L.sbuf[w];
                    L.nAcc = na;
                }
        }
    __syncthreads();
}

// score of a region from its raw score and the sum (-1: no valid child)
__device__ __forceinline__ float region_score(const QueryDesc& qd, float raw, float sum)
{
    return raw < 0.0f ? 1.0f : qd.cfg.epsilon + raw / sum;
}

// Old-node chunk o: the nodes not in the frontier whose draw u is at most
// their region's score plus fA join it again (KGMT.cu:364-376); scores from
// L.raw and sum (own) or from P.score; entries: one per re-activated node
// (node[k] = its index, rep[k] = 1)
__device__ __forceinline__ void react_job(const QueryDesc& qd, const QueryState& st, uint32_t o, const Pools& P,
                                          uint32_t fw, const int32_t rr, const float (&u)[kPer], bool own,
                                          const float* raw, float sum, float fA, uint32_t (&node)[kPer],
                                          uint32_t (&rep)[kPer])
{
    const uint32_t tree = st.treeSize;
    const size_t nodeO  = qd.nodeOff;
    const uint32_t i0   = o * kChunk + kPer * threadIdx.x;
#pragma unroll
    for(uint32_t k = 0; k < kPer; ++k) node[k] = i0 + k, rep[k] = 0u;
    if(i0 >= tree) return;
    const int32_t r[kPer] = {rr};
    float sc[kPer];
#pragma unroll
    for(uint32_t k = 0; k < kPer; ++k)
        {
            const bool cand = i0 + k < tree && ((fw >> (8 * k)) & 0xffu) == 0;
            sc[k] = !cand ? 0.0f : own ? region_score(qd, raw[raw_index((uint32_t)r[k], qd.regShift)], sum) : P.score[qd.regOff + r[k]];
        }
    uint32_t rw = 0;
#pragma unroll
    for(uint32_t k = 0; k < kPer; ++k)
        {
            const bool cand = i0 + k < tree && ((fw >> (8 * k)) & 0xffu) == 0;
            if(cand && u[k] <= sc[k] + fA)
                {
                    // byte store: the new nodes' flags past the tree are
                    // written concurrently by the child chunk jobs
                    P.frontier[nodeO + i0 + k] = 1;
                    rw |= 1u << (8 * k);
                    rep[k] = 1u;
                }
        }
    P.react[nodeO + i0] = (uint8_t)rw;
}

// Child chunk c: the flagged children whose rank (flagged children before
// them) is below `next` (nAcc clamped to the free capacity) are appended at
// tree + rank with their distance to the goal (KGMT.cu:305-345); entries:
// each appended node repeated 15 or 1 times by its region's valid count
// (KGMT.cu:336-339); goal: this thread's smallest appended index within
// goal_thresh (kLbNone if none). pAll / pBefore: this thread's share of the
// chunk counts of all chunks / of the chunks before c.
template <bool QUADS>
__device__ __forceinline__ void append_job(const QueryDesc& qd, const QueryState& st, uint32_t c, const Pools& P,
                                           uint32_t pAll, uint32_t pBefore, uint32_t* sbuf, uint32_t (&node)[kPer],
                                           uint32_t (&rep)[kPer], uint32_t& goal, uint32_t& nAcc, int32_t& apar)
{
    const uint32_t cap = qd.cap, nC = st.nChildren, tree = st.treeSize;
    const size_t nodeO    = qd.nodeOff;
    float* __restrict__ T = P.treeS + qd.sampleOff;
    const int D           = qd.D;
    const uint32_t u0     = c * kChunk + kPer * threadIdx.x;
    uint32_t fl           = 0;
    int32_t r1[kPer]      = {0};
    int32_t vcount[kPer]  = {0};
    constexpr int kRowMax = row_words(KGMT_MAX_SAMPLE);
    const int RW          = row_words(D);
    float v[kPer][kRowMax];  // rows as stored: parent and grandparent bits, then the sample
    if(u0 < nC)
        {
            // flags and regions together
            const uint32_t w = P.fnext[nodeO + u0];
            r1[0]            = P.r1child[nodeO + u0];
#pragma unroll
            for(uint32_t k = 0; k < kPer; ++k)
                if(u0 + k < nC && ((w >> (8 * k)) & 0xffu)) fl |= 1u << k;
        }
    // Before the rank scan: the regions' valid counts for the repeat count
    // and the rows of the flagged children (appended unless the tree fills
    // up). A flagged child's row sits at its 32-child segment's start plus
    // the flagged children before it in the segment (the 32 threads of half
    // a wave).
    const uint32_t nf = (uint32_t)__popc(fl);
    uint32_t slot     = half_incl_scan(nf) - nf;
    slot              = QUADS && !dense_rows(qd.cfg.model) ? u0 : (u0 & ~31u) + slot;
#pragma unroll
    for(uint32_t k = 0; k < kPer; ++k)
        if((fl >> k) & 1u)
            {
                vcount[k] = reinterpret_cast<const int32_t*>(
                  P.cnt + qd.regOff)[2 * region_slot((uint32_t)r1[k], qd.regShift) + 1];  // valid children
                const float4* row = reinterpret_cast<const float4*>(P.childR + qd.rowOffC + (size_t)slot * RW);
                static_for<kRowMax / 4>([&](auto J) {
                    constexpr int j = J;
                    if(4 * j < RW)
                        {
                            const float4 x = row[j];
                            v[k][4 * j] = x.x, v[k][4 * j + 1] = x.y, v[k][4 * j + 2] = x.z, v[k][4 * j + 3] = x.w;
                        }
                });
                ++slot;
            }
    // one scan: ranks inside the chunk, flagged children of all chunks and
    // of the chunks before this one
    const uint32_t in3[3] = {nf, pAll, pBefore};
    uint32_t ex3[3], tot3[3];
    block_excl_scan_n<kUpd, 3>(in3, ex3, tot3, sbuf);
    nAcc                = tot3[1];
    const uint32_t next = nAcc < cap - tree ? nAcc : cap - tree;
    uint32_t rank       = tot3[2] + ex3[0];
    goal                = kLbNone;
    apar                = -1;
    uint32_t t          = tree + rank;
#pragma unroll
    for(uint32_t k = 0; k < kPer; ++k)
        {
            rep[k]  = 0u;
            node[k] = t;
            if((fl >> k) & 1u)
                {
                    if(rank < next)
                        {
                            static_for<KGMT_MAX_SAMPLE>([&](auto I) {
                                constexpr int d = I;
                                if(d < D) T[(size_t)d * cap + t] = v[k][2 + d];
                            });
                            P.parent[nodeO + t]   = __float_as_int(v[k][0]);
                            P.grand[nodeO + t]    = __float_as_int(v[k][1]);
                            apar                  = __float_as_int(v[k][0]);
                            const float dg        = goal_dist(qd, v[k][2], v[k][3], v[k][4]);
                            P.cost[nodeO + t]     = dg;
                            P.frontier[nodeO + t] = 1;
                            P.r1node[nodeO + t]   = r1[k];
                            rep[k] = vcount[k] < qd.cfg.sparse_valid_below ? qd.cfg.repeat_sparse : qd.cfg.repeat_dense;
                            if(dg < qd.cfg.goal_thresh && goal == kLbNone) goal = t;
                        }
                    ++rank;
                    ++t;
                }
        }
}

// One job of query q (li: its index among the query's jobs). own: the
// scores come from the region counts (the planner); otherwise from P.score
// (the stage entry, which is given them).
template <bool QUADS>
__device__ __forceinline__ void update_job(const UpdateArgs& A0, uint32_t q, uint32_t li, UpdateLds& L)
{
    const UpdateArgs& A = fresh(A0);
    QueryState& st      = A.sts[q];
    const QueryDesc& qd = fresh(A.qds[q]);
    const WorkLists& W  = A.W;
    const Pools& P      = A.P;
    const bool own      = A.own != 0u;
    const uint32_t parity = A.parity;
    const uint32_t nq   = W.nq;
    const uint32_t tree = st.treeSize, nC = st.nChildren, cap = qd.cap;
    const uint32_t nOC  = (tree + kChunk - 1) / kChunk;
    const uint32_t nCC  = (nC + kChunk - 1) / kChunk;
    const uint32_t nJ   = nOC + nCC;
    const uint32_t* pa  = P.partA + qd.chunkOff;  // flagged children per child chunk
    const size_t wpq    = 2 * ((size_t)qd.nChunks + 1);  // words of one parity
    uint64_t* words     = P.look + 4 * (size_t)qd.chunkOff + parity * wpq;
    uint64_t* wordsNext = P.look + 4 * (size_t)qd.chunkOff + (parity ^ 1u) * wpq;
    const uint32_t c    = li - nOC;  // child chunk of a child job
    // this thread's share of the chunk counts: the first without a branch
    // (the index clamped into the query's chunks), the rest past kUpd chunks
    const uint32_t i0c = threadIdx.x < qd.nChunks ? threadIdx.x : qd.nChunks;
    const uint32_t x0  = pa[i0c];
    uint32_t pAll      = threadIdx.x < nCC ? x0 : 0u;
    uint32_t pBefore   = threadIdx.x < nCC && threadIdx.x < c ? x0 : 0u;
    for(uint32_t i = threadIdx.x + kUpd; i < nCC; i += kUpd)
        {
            const uint32_t x = pa[i];
            pAll += x;
            pBefore += i < c ? x : 0u;
        }
    uint32_t node[kPer], rep[kPer], goal = kLbNone, nAcc;
    int32_t apar = -1;  // parent of the node this thread appends
    if(li < nOC)
        {
            // the job's nodes first, then the totals (their loads overlap)
            const uint32_t i0 = li * kChunk + kPer * threadIdx.x;
            uint32_t fw       = 0;
            int32_t rr        = 0;
            if(i0 < tree)
                {
                    fw = P.frontier[qd.nodeOff + i0];
                    rr = P.r1node[qd.nodeOff + i0];
                }
            // the draws need neither loads nor scores: computed while they come
            float u[kPer];
#pragma unroll
            for(uint32_t k = 0; k < kPer; ++k) u[k] = draw_react(qd.cfg, qd.cfg.query_id, st.itr, i0 + k);
            // one round of loads: 4 regions per thread up to 4096 regions, 8 above
            if(own && qd.R1 <= 4 * (int)kUpd)
                job_scores<4>(qd, P, pAll, L);
            else if(own)
                job_scores<8>(qd, P, pAll, L);
            else
                {
                    uint32_t tot;
                    block_excl_scan<kUpd>(pAll, L.sbuf, tot);
                    if(threadIdx.x == 0) L.nAcc = tot, L.sum = 0.0f;
                    __syncthreads();
                }
            nAcc                = L.nAcc;
            const uint32_t next = nAcc < cap - tree ? nAcc : cap - tree;
            react_job(qd, st, li, P, fw, rr, u, own, L.raw, L.sum, faccept(qd, st.itr, tree, next), node, rep);
        }
    else
        append_job<QUADS>(qd, st, c, P, pAll, pBefore, L.sbuf, node, rep, goal, nAcc, apar);
    uint32_t total, jobGoal;
    const uint32_t ex = block_excl_scan_min<kUpd>(rep[0], goal, L.sbuf, total, jobGoal);
    if(threadIdx.x == 0)
        {
            __hip_atomic_store(words + li, lb_word(li == 0 ? kLbInclusive : kLbAggregate, total, jobGoal),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            L.before = 0u, L.goalBefore = kLbNone;
        }
    // the aggregate goes out before the look-back's loads
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    // the appended node's ancestors at distances 3..6 are its parent's at
    // 2..5, for the path walk (no job of this launch reads them): written
    // while the look-back runs, by wave 0 after it
    auto link = [&]() {
        if(apar >= 0 && (uint32_t)apar < cap)
            {
                const int32_t g = P.grand[qd.nodeOff + apar];
                const int4 a    = P.anc[qd.nodeOff + apar];
                P.anc[qd.nodeOff + node[0]] = make_int4(g, a.x, a.y, a.z);
            }
    };
    if(threadIdx.x >= 64) link();
    // the job's entries into LDS while the look-back runs (written out below
    // as whole rows; a job with more entries than the stage holds, and job 0,
    // whose region scores stay in L.raw, write them directly)
    const bool staged = total <= (uint32_t)kMaxRegions && !(li == 0 && own);
    if(staged && threadIdx.x >= 64)
        {
            uint32_t p = ex;
#pragma unroll
            for(uint32_t k = 0; k < kPer; ++k)
                {
                    for(uint32_t m = 0; m < rep[k]; ++m) L.stage[p + m] = node[k];
                    p += rep[k];
                }
        }
    if(li > 0 && threadIdx.x < 64)
        {
            uint32_t pc, pg;
            const bool ok = look_back(words, li, pc, pg);
            if(threadIdx.x == 0)
                {
                    if(!ok) __hip_atomic_store(W.error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    __hip_atomic_store(words + li, lb_word(kLbInclusive, pc + total, jobGoal < pg ? jobGoal : pg),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    L.before = pc, L.goalBefore = pg;
                }
        }
    if(threadIdx.x < 64) link();
    if(staged && threadIdx.x < 64)
        {
            uint32_t p = ex;
#pragma unroll
            for(uint32_t k = 0; k < kPer; ++k)
                {
                    for(uint32_t m = 0; m < rep[k]; ++m) L.stage[p + m] = node[k];
                    p += rep[k];
                }
        }
    // (work that no job of this launch reads) the other parity's words start
    // empty for the next launch; job 0 stores the scores and the subregion
    // snapshot for the next propagate (four loads in flight a thread)
    for(size_t i = (size_t)li * kUpd + threadIdx.x; i < wpq; i += (size_t)nJ * kUpd) wordsNext[i] = 0ull;
    if(li == 0 && own)
        {
            const uint32_t* act  = P.actNext + qd.subOff;
            uint32_t* prev       = P.actPrev + qd.subOff;
            const uint32_t words = (uint32_t)qd.R2words;
            for(uint32_t w0 = threadIdx.x; w0 < words; w0 += 4 * kUpd)
                {
                    uint32_t x[4];
#pragma unroll
                    for(uint32_t k = 0; k < 4; ++k) x[k] = act[w0 + k * kUpd < words ? w0 + k * kUpd : w0];
#pragma unroll
                    for(uint32_t k = 0; k < 4; ++k)
                        if(w0 + k * kUpd < words) prev[w0 + k * kUpd] = x[k];
                }
            for(int r = threadIdx.x; r < qd.R1; r += kUpd)
                P.score[qd.regOff + r] = region_score(qd, L.raw[raw_index((uint32_t)r, qd.regShift)], L.sum);
        }
    __syncthreads();
    const uint32_t before = L.before, goalBefore = L.goalBefore;
    // the job's entries of the expansion list at before.., its first
    // capacity entries kept
    uint32_t* out = P.repIdx + qd.nodeOff;
    if(staged)
        {
            for(uint32_t e = threadIdx.x; e < total; e += kUpd)
                if(before + e < cap) out[before + e] = L.stage[e];
        }
    else
        {
            uint32_t pos = before + ex;
#pragma unroll
            for(uint32_t k = 0; k < kPer; ++k)
                {
                    for(uint32_t m = 0; m < rep[k]; ++m)
                        if(pos + m < cap) out[pos + m] = node[k];
                    pos += rep[k];
                }
        }
    const uint32_t next = nAcc < cap - tree ? nAcc : cap - tree;
    const bool last     = li == nJ - 1;
    // the first goal of a single query's iteration: wave 0 walks its path
    // into host memory before its first lane publishes the result
    if(nq == 1 && jobGoal != kLbNone && goalBefore == kLbNone && W.result != nullptr && threadIdx.x < 64 &&
       st.pathRows == 0u)
        walk_path_wave(qd, st, P, W.hostPath, W.hostPath, nullptr, (int32_t)jobGoal);
    // The last job's look-back has seen a word of every other job, each
    // published after that job read the chunk counts: they start at zero
    // again for the next propagate.
    if(last)
        for(uint32_t i = threadIdx.x; i < nCC; i += kUpd) P.partA[qd.chunkOff + i] = 0u;
    if(threadIdx.x == 0)
        {
            const uint32_t goalAll = jobGoal < goalBefore ? jobGoal : goalBefore;
            // a single query's job holding the smallest goal node publishes
            // the solved plan: the goal row was written by this workgroup,
            // the rest of its path by earlier launches
            if(nq == 1 && jobGoal != kLbNone && goalBefore == kLbNone)
                {
                    const Outcome r{1u, st.itr, tree + next, (int32_t)jobGoal, st.expanded + nC, st.flagged + nAcc};
                    publish_single(st, W, r);
                }
            // the last job knows the list size and the goal: it closes the
            // iteration of a single query (the next-state fields and work
            // lists, read from the next kernel on), and that of each of a few
            // queries; k_finish those of more
            if(last)
                {
                    const uint32_t R = before + total;
                    st.R             = R;
                    st.goalIdx       = goalAll == kLbNone ? kNoGoal : (int32_t)goalAll;
                    st.nAcc          = nAcc;
                    st.next          = next;
                    st.fAccept       = faccept(qd, st.itr, tree, next);
                    if(W.few())
                        {
                            finish_query(qd, st, R);
                            W.work[(parity ^ 1u) * nq + q] = query_work(qd, st, W);
                            if(st.doneN && atomicAdd(W.ended, 1u) == nq - 1u)
                                __hip_atomic_store(W.allDone, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                        }
                    if(nq == 1)
                        {
                            finish_query(qd, st, R);
                            count_closed(W);
                            if(st.doneN && !st.successN)
                                {
                                    const Outcome r{0u, st.finishItrN, st.treeSizeN, -1, st.expandedN, st.flaggedN};
                                    publish_single(st, W, r);
                                }
                        }
                }
        }
}

// QUADS: some query is a quadcopter's
template <bool QUADS>
__global__ __launch_bounds__(kUpd) void k_update(UpdateArgs)
{
    __shared__ UpdateLds L;
    const UpdateArgs& A = *(const UpdateArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    const WorkLists& W           = A.W;
    QueryState* __restrict__ sts = A.sts;
    const uint32_t parity        = A.parity;
    const uint32_t nq            = W.nq;
    // the jobs: one query's straight from its state, a few queries' scanned by
    // every workgroup, more queries' from the list
    __shared__ uint32_t list[kFewQueries + 1];
    const QueryState& st0  = sts[0];
    const uint32_t* starts = W.jobs(parity);
    uint32_t nJobs;
    if(nq == 1)
        nJobs = st0.done ? 0u : (st0.treeSize + kChunk - 1) / kChunk + (st0.nChildren + kChunk - 1) / kChunk;
    else if(W.few())
        {
            nJobs  = few_starts<kUpd>(W, parity, 32u, list, L.sbuf);
            starts = list;
        }
    else
        nJobs = starts[nq];
    // with no more jobs than workgroups, workgroup j does job j; with more,
    // every job comes from the counter (the other parity's counter starts at
    // zero for the next launch)
    if(blockIdx.x >= nJobs) return;
    if(blockIdx.x == 0 && threadIdx.x == 0) W.claim[parity ^ 1u] = 0u;
    const bool more = nJobs > gridDim.x;
    while(true)
        {
            uint32_t j = blockIdx.x;
            if(more)
                {
                    if(threadIdx.x == 0)
                        L.job = __hip_atomic_fetch_add(W.claim + parity, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __syncthreads();
                    j = L.job;
                    if(j >= nJobs) return;
                }
            const uint32_t q     = nq == 1 ? 0u : locate(starts, nq, j);
            const uint32_t first = nq == 1 ? 0u : (uint32_t)__builtin_amdgcn_readfirstlane((int)starts[q]);
            // (a stale list entry of a finished query has nothing to do)
            if(!sts[q].done) update_job<QUADS>(A, q, j - first, L);
            if(!more) return;
            __syncthreads();  // L is rewritten by the next job
        }
}

// ---------------------------------------------------------------------------
// finish: one workgroup closes the iteration of every query and builds the
// next iteration's work lists
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_finish(const QueryDesc* __restrict__ qds, QueryState* __restrict__ sts,
                                                   WorkLists W, uint32_t parity)
{
    __shared__ uint32_t sbuf[kBlock / 64 + 1];
    for(uint32_t q = threadIdx.x; q < W.nq; q += kBlock)
        if(!sts[q].done) finish_query(qds[q], sts[q], sts[q].R);
    __syncthreads();
    build_worklists<kBlock>(qds, sts, W, parity ^ 1u, sbuf);
    if(threadIdx.x == 0) count_closed(W);
}

// ---------------------------------------------------------------------------
// paths: goal -> root rows of every solved query, exact depth (Q13), one wave
// per query (512 mixed queries: 40.4 us with one thread per query and two
// levels a round)
// ---------------------------------------------------------------------------
// hostPaths: the host-mapped pool of the first kWaveRows rows of every path,
// which the host reads without a copy (null: all rows go to the device pool)
__global__ __launch_bounds__(64) void k_paths(const QueryDesc* __restrict__ qds, QueryState* __restrict__ sts,
                                              Pools P, uint32_t nq, float* __restrict__ hostPaths)
{
    __shared__ float stage[kWaveRows * KGMT_MAX_SAMPLE];
    const uint32_t q = blockIdx.x;
    QueryState& st   = sts[q];
    if(threadIdx.x == 0) commit_state(st);  // the closed last iteration
    if(!st.successN || st.pathRows) return;
    const QueryDesc& qd = qds[q];
    float* rows         = P.path + qd.pathOff;
    walk_path_wave(qd, st, P, hostPaths ? hostPaths + qd.hostPathOff : rows, rows, stage, st.goalIdx);
}

// ---------------------------------------------------------------------------
// scene build: one workgroup per scene. Boxes sorted along a Morton curve of
// their centres (10 bits per axis over the bounds of the finite centres; ties
// by input order), grouped by kGroup; each group's bounds are the min/max of
// its boxes per axis, or NaN on an axis where a member has a NaN face (such a
// group is never skipped); groups past the boxes hold lo = +inf, hi = -inf and
// are never near. Output: nGrp group (lo, hi) pairs, then nGrp * kGroup boxes.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t morton10(uint32_t x, uint32_t y, uint32_t z)
{
    uint32_t code = 0;
    for(int b = 9; b >= 0; --b) code = (code << 3) | (((x >> b) & 1u) << 2) | (((y >> b) & 1u) << 1) | ((z >> b) & 1u);
    return code;
}

// The masks of n boxes (device.hpp, kSlabs) by a workgroup of kBlock threads;
// face(k, d): face d (0..2 low, 3..5 high) of box k. 64 boxes per wave and
// round: the ballot of "low face in slab g or lower" is their two words of row
// (axis, 0, g), "high face in slab g or higher" of row (axis, 1, g); a NaN
// face belongs to every row of its side.
template <class FACE>
__device__ __forceinline__ void box_masks(uint32_t n, float wsMin, float slabScale, uint32_t* mask, FACE face)
{
    const uint32_t nw = mask_row(n), lane = lane_id();
    for(uint32_t wp = threadIdx.x / 64; wp < nw / 2; wp += kBlock / 64)
        {
            const uint32_t k = 64 * wp + lane;
            for(int d = 0; d < 3; ++d)
                {
                    int lo = (int)kSlabs, hi = -1;
                    if(k < n)
                        {
                            const float h = face(k, 3 + d);
                            lo            = slab_of(face(k, d), wsMin, slabScale);  // NaN: 0
                            hi            = h == h ? slab_of(h, wsMin, slabScale) : (int)kSlabs - 1;
                        }
                    uint64_t keep = 0;
#pragma unroll
                    for(int g = 0; g < (int)kSlabs; ++g)
                        {
                            const uint64_t a = __ballot(lo <= g), b = __ballot(hi >= g);
                            keep             = (int)lane == g ? a : (int)lane == (int)kSlabs + g ? b : keep;
                        }
                    if(lane < 2 * kSlabs)
                        *reinterpret_cast<uint64_t*>(mask + (size_t)(2 * kSlabs * d + lane) * nw + 2 * wp) = keep;
                }
        }
}

struct SceneLds
{
    float box[kMaxObs][6];
    alignas(16) uint32_t key[kMaxObs];
    float red[6][kBlock / 64];
};

// Face k (0..2 min x y z, 3..5 max x y z) of box i of rows of 2 * W floats; a
// planar box (W = 2) spans z [-1, 1], which holds the planar positions' z = 0.
template <int W>
__device__ __forceinline__ float row_face(const float* __restrict__ rows, uint32_t i, int k)
{
    if constexpr(W == 3)
        return rows[6 * (size_t)i + k];
    else
        return k == 2 ? -1.0f : k == 5 ? 1.0f : rows[4 * (size_t)i + (k < 3 ? k : k - 1)];
}

// mask (null: none): the box masks too, for a workspace from wsMin with
// slabScale slabs per unit.
template <int W, bool MASKS = false>
__device__ __forceinline__ void build_scene_wg(const float* __restrict__ rows, uint32_t n, uint32_t nGrp, float4* __restrict__ out,
                               SceneLds& L, uint32_t* __restrict__ mask = nullptr, float wsMin = 0.0f,
                               float slabScale = 0.0f)
{
    // bounds of the finite centres
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for(uint32_t i = threadIdx.x; i < n; i += kBlock)
        for(int d = 0; d < 3; ++d)
            {
                const float c = 0.5f * (row_face<W>(rows, i, d) + row_face<W>(rows, i, 3 + d));
                if(__builtin_isfinite(c)) lo[d] = c < lo[d] ? c : lo[d], hi[d] = c > hi[d] ? c : hi[d];
            }
    for(int d = 0; d < 3; ++d)
        {
            for(int o = 32; o > 0; o >>= 1)
                {
                    const float a = __shfl_xor(lo[d], o, 64), b = __shfl_xor(hi[d], o, 64);
                    lo[d] = a < lo[d] ? a : lo[d], hi[d] = b > hi[d] ? b : hi[d];
                }
            if(lane_id() == 0) L.red[d][threadIdx.x / 64] = lo[d], L.red[3 + d][threadIdx.x / 64] = hi[d];
        }
    __syncthreads();
    for(int d = 0; d < 3; ++d)
        {
            lo[d] = INFINITY, hi[d] = -INFINITY;
            for(int w = 0; w < kBlock / 64; ++w)
                {
                    const float a = L.red[d][w], b = L.red[3 + d][w];
                    lo[d] = a < lo[d] ? a : lo[d], hi[d] = b > hi[d] ? b : hi[d];
                }
        }
    // Morton keys
    for(uint32_t i = threadIdx.x; i < n; i += kBlock)
        {
            uint32_t q[3];
            for(int d = 0; d < 3; ++d)
                {
                    const float c = 0.5f * (row_face<W>(rows, i, d) + row_face<W>(rows, i, 3 + d));
                    float t       = hi[d] > lo[d] ? (c - lo[d]) / (hi[d] - lo[d]) : 0.0f;
                    if(!(t >= 0.0f)) t = 0.0f;
                    if(t > 1.0f) t = 1.0f;
                    q[d] = (uint32_t)(t * 1023.0f);
                }
            L.key[i] = morton10(q[0], q[1], q[2]);
        }
    if(threadIdx.x < 3 && n + threadIdx.x < kMaxObs) L.key[n + threadIdx.x] = 0xffffffffu;
    __syncthreads();
    // rank = position in (key, index) order; box i goes to slot rank. Four keys
    // a read, the ones past the last box after every box (333 boxes: k_init_one
    // 26.6 to 21.7 us)
    static_assert(kMaxObs % 4 == 0, "keys read in fours");
    for(uint32_t i = threadIdx.x; i < n; i += kBlock)
        {
            const uint32_t ki = L.key[i];
            uint32_t rank     = 0;
#pragma unroll 4
            for(uint32_t j = 0; j < n; j += 4)
                {
                    const uint4 k = reinterpret_cast<const uint4*>(L.key)[j / 4];
                    rank += (k.x < ki + (j < i)) + (k.y < ki + (j + 1 < i)) + (k.z < ki + (j + 2 < i)) +
                            (k.w < ki + (j + 3 < i));
                }
            for(int d = 0; d < 6; ++d) L.box[rank][d] = row_face<W>(rows, i, d);
        }
    __syncthreads();
    float4* box = out + 2 * nGrp;
    for(uint32_t k = threadIdx.x; k < nGrp * kGroup; k += kBlock)
        {
            if(k < n)
                {
                    box[2 * k]     = make_float4(L.box[k][0], L.box[k][1], L.box[k][2], 0.0f);
                    box[2 * k + 1] = make_float4(L.box[k][3], L.box[k][4], L.box[k][5], 0.0f);
                }
            else
                {
                    box[2 * k]     = make_float4(INFINITY, INFINITY, INFINITY, 0.0f);
                    box[2 * k + 1] = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
                }
        }
    for(uint32_t g = threadIdx.x; g < nGrp; g += kBlock)
        {
            float gl[3] = {INFINITY, INFINITY, INFINITY}, gh[3] = {-INFINITY, -INFINITY, -INFINITY};
            bool nanAxis[3] = {false, false, false};
            const uint32_t b1 = n < (g + 1) * kGroup ? n : (g + 1) * kGroup;
            for(uint32_t k = g * kGroup; k < b1; ++k)
                for(int d = 0; d < 3; ++d)
                    {
                        const float l = L.box[k][d], h = L.box[k][3 + d];
                        if(l != l || h != h) nanAxis[d] = true;
                        gl[d] = l < gl[d] ? l : gl[d];  // a NaN member leaves the bound as is
                        gh[d] = gh[d] < h ? h : gh[d];
                    }
            for(int d = 0; d < 3; ++d)
                if(nanAxis[d]) gl[d] = gh[d] = NAN;
            out[2 * g]     = make_float4(gl[0], gl[1], gl[2], 0.0f);
            out[2 * g + 1] = make_float4(gh[0], gh[1], gh[2], 0.0f);
        }
    if(!MASKS || !mask) return;
    box_masks(n, wsMin, slabScale, mask, [&](uint32_t k, int d) { return L.box[k][d]; });
}

// a query's scene from its rows, with its masks where MASKS and it has them
template <bool MASKS>
__device__ __forceinline__ void build_query_scene(const QueryDesc& qd, const float* __restrict__ rows, const Pools& P, SceneLds& L)
{
    float4* out    = P.obs + 2 * (size_t)qd.obsOff;
    uint32_t* mask = MASKS && qd.masks ? reinterpret_cast<uint32_t*>(out + 2 * (size_t)qd.nGrp * (1 + kGroup)) : nullptr;
    if(qd.wdim == 2)
        build_scene_wg<2, MASKS>(rows + 4 * (size_t)qd.rowOff, qd.nObs, qd.nGrp, out, L, mask, qd.cfg.ws_min,
                                 qd.slabScale);
    else
        build_scene_wg<3, MASKS>(rows + 6 * (size_t)qd.rowOff, qd.nObs, qd.nGrp, out, L, mask, qd.cfg.ws_min,
                                 qd.slabScale);
}

// ---------------------------------------------------------------------------
// init: one workgroup per query (KGMT.cu:50-81): the query's scene from the
// caller's obstacle rows (rows null: no obstacles), then the root, cleared
// counters and the first iteration's state; the last workgroup to arrive
// builds the first work lists.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_init(const QueryDesc* __restrict__ qds, QueryState* __restrict__ sts,
                                                 Pools P, WorkLists W, uint32_t nq, const float* __restrict__ rows)
{
    __shared__ SceneLds L;
    __shared__ uint32_t sbuf[kBlock / 64 + 1];
    __shared__ uint32_t sflag;
    const uint32_t q    = blockIdx.x;
    const QueryDesc& qd = qds[q];
    if(rows && qd.nObs) build_query_scene<true>(qd, rows, P, L);
    clear_query(qd, P, threadIdx.x, kBlock);
    root_query(qd, sts[q], P);
    if(q == 0 && threadIdx.x < 2) W.claim[threadIdx.x] = W.tileClaim[threadIdx.x] = 0u;
    if(q == 0 && threadIdx.x == 0) *W.closedDev = 0u;
    if(q == 0 && threadIdx.x == 0) *W.ended = 0u;
    if(W.few())
        {
            // (the first thread wrote the state)
            if(threadIdx.x == 0) W.work[q] = query_work(qd, sts[q], W);
            return;
        }
    if(last_arrival(W.counter, nq, &sflag)) build_worklists<kBlock>(qds, sts, W, 0, sbuf);
}

// k_init of a single query, its descriptor a kernel argument that the first
// thread stores for the kernels after it (no upload before the launch):
// workgroup 0 builds the scene, the root, the state and the first work
// lists (no hand-off between workgroups), workgroups 1.. clear the counters
template <bool MASKS>
__global__ __launch_bounds__(kBlock) void k_init_one(const QueryDesc qd, QueryDesc* __restrict__ dq,
                                                     QueryState* __restrict__ sts, Pools P, WorkLists W,
                                                     const float* __restrict__ rows)
{
    __shared__ SceneLds L;
    if(blockIdx.x > 0)
        {
            clear_query(qd, P, (blockIdx.x - 1) * kBlock + threadIdx.x, (gridDim.x - 1) * kBlock);
            return;
        }
    if(threadIdx.x == 0) *dq = qd;
    if(rows && qd.nObs) build_query_scene<MASKS>(qd, rows, P, L);
    root_query(qd, sts[0], P);
    if(threadIdx.x < 2) W.claim[threadIdx.x] = W.tileClaim[threadIdx.x] = 0u;
    if(threadIdx.x == 0) *W.closedDev = 0u;
}

template <int W>
__global__ __launch_bounds__(kBlock) void k_build_scene(const float* __restrict__ rows, uint32_t n, uint32_t nGrp,
                                                        float4* __restrict__ out)
{
    __shared__ SceneLds L;
    build_scene_wg<W>(rows, n, nGrp, out, L);
}

// a caller's boxes as the planner's scene of a query with box masks
__global__ __launch_bounds__(kBlock) void k_build_mask_scene(const QueryDesc* __restrict__ qdp,
                                                             const float* __restrict__ rows, uint32_t n, uint32_t nGrp,
                                                             float4* __restrict__ out)
{
    __shared__ SceneLds L;
    build_scene_wg<3, true>(rows, n, nGrp, out, L, reinterpret_cast<uint32_t*>(out + 2 * (size_t)nGrp * (1 + kGroup)),
                            qdp->cfg.ws_min, qdp->slabScale);
}

// ---------------------------------------------------------------------------
// a query's tree in the reference's layout: rows of D floats
// (d_treeSamples_), parents and costs; entries past the tree are 0, -1, 0 as
// the reference's fills leave them (KGMT.cu:62-64)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_tree_rows(const float* __restrict__ treeS,
                                                      const int32_t* __restrict__ parent,
                                                      const float* __restrict__ cost, uint32_t cap, uint32_t n, int D,
                                                      uint32_t treeSize, float* __restrict__ rows,
                                                      int32_t* __restrict__ parents, float* __restrict__ costs)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if(i >= n) return;
    const bool in = i < treeSize;
    for(int d = 0; d < D; ++d) rows[(size_t)i * D + d] = in ? treeS[(size_t)d * cap + i] : 0.0f;
    if(!parents) return;
    parents[i] = in ? parent[i] : -1;
    costs[i]   = in ? cost[i] : 0.0f;
}

// ---------------------------------------------------------------------------
// stage-level kernels (single query, caller buffers)
// ---------------------------------------------------------------------------
template <int C>
__global__ __launch_bounds__(kBlock) void k_stage_draw(const QueryDesc* __restrict__ qd, uint32_t query,
                                                       uint32_t itr, uint32_t u0, uint32_t n, float* controls,
                                                       int32_t* steps, float* ufront)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if(i >= n) return;
    float uc[C];
    int32_t st;
    float uf;
    draw_child<C>(qd->cfg, query, itr, u0 + i, uc, st, uf);
#pragma unroll
    for(int k = 0; k < C; ++k) controls[(size_t)k * n + i] = uc[k];
    steps[i]  = st;
    ufront[i] = uf;
}

// Segment check of the dynamics by box masks
struct MaskCheck
{
    const QueryDesc& qd;
    const MaskScene& sc;
    MaskWalk walk;
    __device__ __forceinline__ bool operator()(float px, float py, float pz, float x, float y, float z)
    {
        return !walk.hit(qd, sc, px, py, pz, x, y, z, true);
    }
};

// LDS pairs of a stage's scene: its boxes in the caller's order, their masks
static uint32_t stage_pairs(uint32_t nObs)
{
    return nObs + mask_pairs(nObs);
}

template <int W>
__device__ __forceinline__ MaskScene stage_scene_masks(const QueryDesc& qd, const float* __restrict__ rows, uint32_t n,
                                                       float4* sObs)
{
    float4 *lo = sObs, *hi = sObs + n;
    uint32_t* mask = reinterpret_cast<uint32_t*>(sObs + 2 * n);
    for(uint32_t i = threadIdx.x; i < n; i += kBlock)
        {
            lo[i] = make_float4(row_face<W>(rows, i, 0), row_face<W>(rows, i, 1), row_face<W>(rows, i, 2), 0.0f);
            hi[i] = make_float4(row_face<W>(rows, i, 3), row_face<W>(rows, i, 4), row_face<W>(rows, i, 5), 0.0f);
        }
    __syncthreads();
    box_masks(n, qd.cfg.ws_min, qd.slabScale, mask, [&](uint32_t k, int d) {
        const float4& f = d < 3 ? lo[k] : hi[k];
        const int e     = d < 3 ? d : d - 3;
        return e == 0 ? f.x : e == 1 ? f.y : f.z;
    });
    __syncthreads();
    return MaskScene{lo, hi, mask, (int)mask_row(n), (int)n};
}

// A caller's edges: parent, control and steps in, child, verdict and regions
// out.
template <int MODEL>
struct StageEdges
{
    static constexpr int S = ModelDims<MODEL>::S, C = ModelDims<MODEL>::C, D = S + C + 1;
    const int32_t* __restrict__ parentIdx;
    const float* __restrict__ parentStates;
    uint32_t nParents;
    const float* __restrict__ controls;
    const int32_t* __restrict__ steps;
    uint32_t n;
    float* __restrict__ child;
    uint8_t* __restrict__ valid;
    int32_t* __restrict__ r1o;
    int32_t* __restrict__ r2o;

    // -1: out of range
    __device__ __forceinline__ int32_t parent(uint32_t i) const
    {
        const int32_t p = parentIdx[i];
        return p >= 0 && (uint32_t)p < nParents ? p : -1;
    }
    // start state and control of edge i
    __device__ __forceinline__ void read(uint32_t i, int32_t p, float* s, float* u) const
    {
#pragma unroll
        for(int d = 0; d < S; ++d) s[d] = p < 0 ? 0.0f : parentStates[(size_t)d * nParents + p];
#pragma unroll
        for(int k = 0; k < C; ++k) u[k] = controls[(size_t)k * n + i];
    }
    __device__ __forceinline__ void write(const QueryDesc& qd, uint32_t i, int32_t p, const float* s, const float* u,
                                          bool ok) const
    {
        if(p < 0)
            {
                // caller index out of range: no state is read; flagged by r1 = r2 = -1
                for(int d = 0; d < D; ++d) child[(size_t)d * n + i] = 0.0f;
                valid[i] = 0;
                r1o[i]   = -1;
                r2o[i]   = -1;
                return;
            }
#pragma unroll
        for(int d = 0; d < S; ++d) child[(size_t)d * n + i] = s[d];
#pragma unroll
        for(int k = 0; k < C; ++k) child[(size_t)(S + k) * n + i] = u[k];
        child[(size_t)(D - 1) * n + i] = qd.cfg.dt * (float)steps[i];
        int ix, iy, iz;
        const int r1 = region_of(qd, s[0], s[1], s[2], ix, iy, iz);
        valid[i]     = ok ? 1 : 0;
        r1o[i]       = r1;
        r2o[i]       = subregion_of(qd, s[0], s[1], s[2], r1, ix, iy, iz);
    }
};

// Quadcopter edges base .. base + count - 1 as a planner's tile of NT threads
// (at most 2 NT edges; barriers inside).
template <int NT>
__device__ __forceinline__ void stage_quad_tile(const QueryDesc& qd, const StageEdges<KGMT_MODEL_QUADCOPTER>& E,
                                                uint32_t base, uint32_t count, const MaskScene& sc, QuadRunLds<NT>& L)
{
    quad_run<NT>(
      qd, count, sc, L, [&](uint32_t k) { return E.steps[base + k]; },
      [&](uint32_t k, QuadChild& ch) {
          const uint32_t i = base + k;
          const int32_t p  = E.parent(i);
          ch.p             = (uint32_t)p;
          E.read(i, p, ch.s, ch.u);
          const int32_t st = E.steps[i];
          ch.uf            = 0.0f;
          ch.left          = p < 0 || st < 0 ? 0 : st;
      },
      [&](const QuadChild& ch) { E.write(qd, base + (ch.meta & 1023u), (int32_t)ch.p, ch.s, ch.u, ch.left == 0); });
}

// kgmt_propagate_collide: one launch. Every workgroup builds the scene's
// masks in its LDS (about 2 us for 200 boxes; a scene kernel before this one
// took 10.6 and the sort its group bounds need grows with the square of the
// boxes) and takes every gridDim.x-th tile of kBlock children: one per lane,
// or, for the quadcopter, as the planner's tiles do. 100003 quadcopter edges
// among 200 boxes: kernels 539 + 10.6 -> 235 us, the call 580 -> 233; 100003 of
// the other models 102 to 246 -> 22 to 47 us, 1000 of them 55 to 65 -> 12 to 20.
template <int MODEL>
__global__ __launch_bounds__(kBlock, 4) void k_stage_propagate(const QueryDesc qd, const int32_t* __restrict__ parentIdx,
                                                               const float* __restrict__ parentStates,
                                                               uint32_t nParents, const float* __restrict__ controls,
                                                               const int32_t* __restrict__ steps, uint32_t n,
                                                               const float* __restrict__ rows, uint32_t nObs,
                                                               float* __restrict__ child, uint8_t* __restrict__ valid,
                                                               int32_t* __restrict__ r1o, int32_t* __restrict__ r2o)
{
    constexpr int S = ModelDims<MODEL>::S, C = ModelDims<MODEL>::C;
    extern __shared__ float4 sObs[];
    const MaskScene sc = stage_scene_masks<MODEL == KGMT_MODEL_UNICYCLE ? 2 : 3>(qd, rows, nObs, sObs);
    const StageEdges<MODEL> E{parentIdx, parentStates, nParents, controls, steps, n, child, valid, r1o, r2o};
    if constexpr(MODEL == KGMT_MODEL_QUADCOPTER)
        {
            __shared__ QuadRunLds<kBlock> L;
            // (64 bits: the turn after the last can pass 2^32)
            for(uint64_t at = blockIdx.x * kBlock; at < n; at += gridDim.x * kBlock)
                {
                    const uint32_t base = (uint32_t)at;
                    stage_quad_tile<kBlock>(qd, E, base, n - base < kBlock ? n - base : kBlock, sc, L);
                    __syncthreads();  // L is used again
                }
        }
    else
        for(uint64_t at = blockIdx.x * kBlock + threadIdx.x; at < n; at += gridDim.x * kBlock)
            {
                const uint32_t i = (uint32_t)at;
                const int32_t p  = E.parent(i);
                float s[S], u[C];
                bool ok = false;
                E.read(i, p, s, u);
                if(p >= 0)
                    {
                        MaskCheck chk{qd, sc, MaskWalk{0, 0, 0}};
                        chk.walk.start(qd, s[0], s[1], pos_z<MODEL>(s));
                        ok = propagate_with<MODEL>(qd, s, u, steps[i], chk);
                    }
                E.write(qd, i, p, s, u, ok);
            }
}

// The planner's per-child path on caller buffers: children in waves of 64
// consecutive indices, handed to the wave's lanes longest-first by the same
// counting sort child_tile runs with one lane per child, then
// propagate_two_phase called by every lane of the wave as child_tile calls it
// (lanes without a child take part with an empty box). check / box (optional)
// receive the check that decided each child and its edge box.
template <int MODEL>
__global__ __launch_bounds__(kBlock) void k_stage_propagate_planner(
  const QueryDesc* __restrict__ qdp, const int32_t* __restrict__ parentIdx, const float* __restrict__ parentStates,
  uint32_t nParents, const float* __restrict__ controls, const int32_t* __restrict__ steps, uint32_t n,
  const float4* __restrict__ obs, uint32_t nGrp, float* child, uint8_t* valid, int32_t* r1o, int32_t* r2o,
  uint8_t* checkOut, float* boxOut)
{
    constexpr int S = ModelDims<MODEL>::S, C = ModelDims<MODEL>::C;
    extern __shared__ float4 sObs[];
    __shared__ float4 cand[kBlock / 64][2 * kCand];
    __shared__ uint32_t hist[kBlock];
    __shared__ uint16_t slot[kBlock];
    const QueryDesc& qd = *qdp;
    stage_scene(obs, 0, nGrp, sObs);
    __syncthreads();
    const uint32_t t    = threadIdx.x;
    const uint32_t base = blockIdx.x * kBlock;
    // counting sort of the wave's 64 children by step count, longest first
    // (bucket 63 of the wave: lanes past the end)
    {
        const uint32_t g0 = (t / 64u) * 64u;
        uint32_t bucket   = g0 + 63u;
        if(base + t < n)
            {
                int32_t k = steps[base + t] - qd.cfg.steps_min;
                k         = k < 0 ? 0 : (k > 62 ? 62 : k);
                bucket    = g0 + 62u - (uint32_t)k;
            }
        hist[t] = 0;
        wave_sync();
        const uint32_t rank = atomicAdd(&hist[bucket], 1u);
        wave_sync();
        const uint32_t h = hist[t];
        hist[t]          = g0 + wave_incl_scan(h) - h;
        wave_sync();
        slot[hist[bucket] + rank] = (uint16_t)t;
        wave_sync();
    }
    const StageEdges<MODEL> E{parentIdx, parentStates, nParents, controls, steps, n, child, valid, r1o, r2o};
    const uint32_t i = base + slot[t];
    const int32_t p  = i < n ? E.parent(i) : -1;
    const bool has   = p >= 0;
    float s[S] = {}, uc[C] = {};
    int32_t st = 0;
    if(has) E.read(i, p, s, uc), st = steps[i];
    const Scene sc{sObs, (int)nGrp, 0};
    TwoPhaseTrace tr{KGMT_CHECK_SCENE, {0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
    const bool ok = propagate_two_phase<MODEL>(qd, s, uc, st, sc, cand[t / 64], has, &tr);  // every lane
    if(i >= n) return;
    E.write(qd, i, p, s, uc, ok);
    if(!has) return;
    if(checkOut) checkOut[i] = (uint8_t)tr.path;
    if(boxOut)
        for(int d = 0; d < 3; ++d) boxOut[(size_t)d * n + i] = tr.lo[d], boxOut[(size_t)(3 + d) * n + i] = tr.hi[d];
}

// The same for the quadcopter: tiles of the planner's workgroup with one lane
// per child (quad_run) on the planner's scene, in turn a tile of twice as many
// children as lanes (sorted, refilled) and one of as many.
__global__ __launch_bounds__(kTile, 4) void k_stage_quad_planner(
  const QueryDesc* __restrict__ qdp, const int32_t* __restrict__ parentIdx, const float* __restrict__ parentStates,
  uint32_t nParents, const float* __restrict__ controls, const int32_t* __restrict__ steps, uint32_t n,
  const float4* __restrict__ obs, uint32_t nGrp, uint32_t nObs, float* __restrict__ child, uint8_t* __restrict__ valid,
  int32_t* __restrict__ r1o, int32_t* __restrict__ r2o, uint8_t* __restrict__ checkOut)
{
    extern __shared__ float4 sObs[];
    __shared__ QuadRunLds<kTile> L;
    const QueryDesc& qd = *qdp;
    const StageEdges<KGMT_MODEL_QUADCOPTER> E{parentIdx, parentStates, nParents, controls, steps, n,
                                              child,     valid,        r1o,      r2o};
    const MaskScene sc  = stage_masks(obs, 0, nGrp, nObs, sObs, true);
    const uint32_t two  = blockIdx.x & 1u ? 0u : kTile;
    const uint32_t base = (blockIdx.x >> 1) * 3u * kTile + (two ? 0u : 2u * kTile);
    if(base >= n) return;
    const uint32_t count = n - base < kTile + two ? n - base : kTile + two;
    stage_quad_tile<kTile>(qd, E, base, count, sc, L);
    if(checkOut)
        for(uint32_t k = threadIdx.x; k < count; k += kTile)
            if(E.parent(base + k) >= 0) checkOut[base + k] = KGMT_CHECK_ONE_PASS;
}

// Frontier update stage: the caller's tree and children staged into a
// one-query pool the way the iteration's propagate and score kernels leave
// it, so that the planner's own k_append and k_expand run on it. Per tree
// node its region (the reference's getRegion of the node, KGMT.cu:369); per
// child its region, its flag and, when flagged, its row (parent, parent's
// parent, sample) at the next free slot of its 32-child segment.
__global__ __launch_bounds__(kBlock) void k_stage_fu_nodes(const QueryDesc* __restrict__ qdp, Pools P, uint32_t tree,
                                                           const float* __restrict__ child,
                                                           const int32_t* __restrict__ childParent,
                                                           const uint8_t* __restrict__ fnext, uint32_t nC,
                                                           const int32_t* __restrict__ valid)
{
    const QueryDesc& qd = *qdp;
    const uint32_t i    = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t cap  = qd.cap;
    int ix, iy, iz;
    if(i < (uint32_t)qd.R1) P.cnt[region_slot(i, qd.regShift)] = (uint64_t)(uint32_t)valid[i] << 32;
    if(i < tree)
        P.r1node[i] = region_of(qd, P.treeS[i], P.treeS[(size_t)cap + i], P.treeS[2 * (size_t)cap + i], ix, iy, iz);
    if(i >= nC) return;
    const bool f = fnext[i] != 0;
    P.fnext[i]   = f ? 1 : 0;
    P.r1child[i] = region_of(qd, child[i], child[(size_t)nC + i], child[2 * (size_t)nC + i], ix, iy, iz);
    if(!f) return;
    const uint32_t s0 = dense_rows(qd.cfg.model) ? i & ~31u : i;
    uint32_t before   = 0;
    for(uint32_t k = s0; k < i; ++k) before += fnext[k] ? 1u : 0u;
    const int32_t p  = childParent[i];
    const int32_t gp = p >= 0 && (uint32_t)p < tree ? P.parent[p] : -1;
    const int D      = qd.D, RW = row_words(D);
    float* row       = P.childR + (size_t)(s0 + before) * RW;
    row[0]           = __int_as_float(p);
    row[1]           = __int_as_float(gp);
    for(int d = 0; d < D; ++d) row[2 + d] = child[(size_t)d * nC + i];
    for(int e = D + 2; e < RW; ++e) row[e] = 0.0f;
}

// flagged children per chunk, the state an iteration's propagate leaves
// (accepted count and fAccept for the info output) and the work lists of the
// update jobs (one workgroup)
__global__ __launch_bounds__(kBlock) void k_stage_fu_state(const QueryDesc* __restrict__ qdp, QueryState* st,
                                                           Pools P, WorkLists W, uint32_t itr, uint32_t tree,
                                                           uint32_t nC)
{
    __shared__ uint32_t cnt[1024];
    const QueryDesc& qd = *qdp;
    const uint32_t nCC  = (nC + kChunk - 1) / kChunk;
    for(uint32_t c = threadIdx.x; c < nCC; c += kBlock)
        {
            uint32_t n = 0;
            for(uint32_t u = c * kChunk; u < nC && u < (c + 1) * kChunk; ++u) n += P.fnext[u];
            cnt[c] = n;
        }
    __syncthreads();
    if(threadIdx.x != 0) return;
    uint32_t acc = 0;
    for(uint32_t c = 0; c < nCC; ++c)
        {
            P.partA[c] = cnt[c];
            acc += cnt[c];
        }
    const uint32_t avail = qd.cap - tree;
    const uint32_t next  = acc < avail ? acc : avail;
    QueryState s{};
    s.itr = s.itrN = itr;
    s.treeSize = s.treeSizeN = tree;
    s.nChildren = s.nChildrenN = nC;
    s.nAcc      = acc;
    s.next      = next;
    s.fAccept   = faccept(qd, itr, tree, next);
    s.goalIdx   = kNoGoal;
    *st         = s;
    const uint32_t jobs = nCC + (tree + kChunk - 1) / kChunk;
    for(uint32_t i = 0; i < jobs; ++i) P.look[i] = 0ull;  // parity 0's words
    W.claim[0] = W.claim[1] = 0u;
    *W.error   = 0u;
}

// info[4] = {appended, expansion multiset size, goal node or -1, re-activated}
__global__ void k_stage_fu_info(const QueryDesc* __restrict__ qdp, const QueryState* st, Pools P, uint32_t tree,
                                int32_t* info)
{
    if(threadIdx.x != 0) return;
    // the inclusive entries of the last old-node job: the re-activated count
    const uint32_t nOC   = (tree + kChunk - 1) / kChunk;
    const uint32_t react = (uint32_t)P.look[nOC - 1];
    info[0] = (int32_t)st->next;
    info[1] = (int32_t)st->R;
    info[2] = st->goalIdx == kNoGoal ? -1 : st->goalIdx;
    info[3] = (int32_t)react;
}

__global__ __launch_bounds__(kBlock) void k_stage_region_update(const QueryDesc* __restrict__ qdp,
                                                                const int32_t* __restrict__ r1,
                                                                const int32_t* __restrict__ r2,
                                                                const uint8_t* __restrict__ valid,
                                                                const float* __restrict__ ufront, uint32_t n,
                                                                const float* __restrict__ score,
                                                                const uint32_t* __restrict__ actPrev,
                                                                uint32_t* actNext, int32_t* total, int32_t* validc,
                                                                uint8_t* fnext)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    const QueryDesc& qd = *qdp;
    int key             = i < n ? r1[i] : 0;
    const int sub       = i < n ? r2[i] : 0;
    // children with a region id out of range are ignored
    const bool has = i < n && key >= 0 && key < qd.R1 && sub >= 0 && sub < qd.R2;
    if(!has) key = 0;
    const bool ok = has && valid[i] != 0;
    bool fn       = false;
    bool setBit   = false;
    if(ok)
        {
            const bool seen = test_bit(actPrev, (uint32_t)sub);
            fn              = (ufront[i] < score[key]) || !seen;
            setBit          = !seen;
        }
    if(i < n) fnext[i] = fn ? 1 : 0;
    wave_set_bits(actNext, has ? (uint32_t)sub : 0u, setBit);
    wave_count(total, validc, key, has, ok);
}

__global__ __launch_bounds__(kScoreThreads) void k_stage_score(const QueryDesc* __restrict__ qd,
                                                               const int32_t* __restrict__ total,
                                                               const int32_t* __restrict__ validc,
                                                               const uint32_t* __restrict__ act, float* score)
{
    __shared__ float a[kScoreThreads];
    score_regions<kScoreThreads>(*qd, total, validc, act, score, a);
}

// compaction: chunk counts -> one-workgroup scan -> scatter
__global__ __launch_bounds__(kBlock) void k_stage_count(const uint8_t* __restrict__ flags, uint32_t n, uint32_t* tmp)
{
    __shared__ uint32_t sbuf[kBlock / 64 + 1];
    const uint32_t c = blockIdx.x;
    uint32_t cnt     = 0;
    for(uint32_t k = 0; k < kChunk / kBlock; ++k)
        {
            const uint32_t i = c * kChunk + k * kBlock + threadIdx.x;
            cnt += (i < n && flags[i]) ? 1u : 0u;
        }
    uint32_t tot;
    block_excl_scan<kBlock>(cnt, sbuf, tot);
    if(threadIdx.x == 0) tmp[c] = tot;
}

__global__ __launch_bounds__(kScoreThreads) void k_stage_scan(uint32_t* tmp, uint32_t m, uint32_t* total)
{
    __shared__ uint32_t sbuf[kScoreThreads / 64 + 1];
    const uint32_t t = block_scan_array<kScoreThreads>(tmp, m, sbuf);
    if(threadIdx.x == 0) *total = t;
}

__global__ __launch_bounds__(kBlock) void k_stage_scatter(const uint8_t* __restrict__ flags, uint32_t n,
                                                          const uint32_t* __restrict__ tmp, uint32_t* out)
{
    __shared__ uint32_t sbuf[kBlock / 64 + 1];
    const uint32_t c = blockIdx.x;
    uint32_t run     = tmp[c];
    for(uint32_t k = 0; k < kChunk / kBlock; ++k)
        {
            const uint32_t i = c * kChunk + k * kBlock + threadIdx.x;
            const bool f     = i < n && flags[i] != 0;
            uint32_t tot;
            const uint32_t ex = block_excl_scan<kBlock>(f ? 1u : 0u, sbuf, tot);
            if(f) out[run + ex] = i;
            run += tot;
        }
}

// segmented repeat: chunk sums -> scan -> write
__global__ __launch_bounds__(kBlock) void k_stage_sum(const uint32_t* __restrict__ counts, uint32_t n, uint32_t* tmp)
{
    __shared__ uint32_t sbuf[kBlock / 64 + 1];
    const uint32_t c = blockIdx.x;
    uint32_t sum     = 0;
    for(uint32_t k = 0; k < kChunk / kBlock; ++k)
        {
            const uint32_t i = c * kChunk + k * kBlock + threadIdx.x;
            sum += i < n ? counts[i] : 0u;
        }
    uint32_t tot;
    block_excl_scan<kBlock>(sum, sbuf, tot);
    if(threadIdx.x == 0) tmp[c] = tot;
}

__global__ __launch_bounds__(kBlock) void k_stage_repeat(const uint32_t* __restrict__ ids,
                                                         const uint32_t* __restrict__ counts, uint32_t n,
                                                         const uint32_t* __restrict__ tmp, uint32_t* out,
                                                         uint32_t outCap)
{
    __shared__ uint32_t sbuf[kBlock / 64 + 1];
    const uint32_t c = blockIdx.x;
    uint32_t run     = tmp[c];
    for(uint32_t k = 0; k < kChunk / kBlock; ++k)
        {
            const uint32_t i   = c * kChunk + k * kBlock + threadIdx.x;
            const uint32_t cnt = i < n ? counts[i] : 0u;
            uint32_t tot;
            const uint32_t ex = block_excl_scan<kBlock>(cnt, sbuf, tot);
            for(uint32_t m = 0; m < cnt; ++m)
                if(run + ex + m < outCap) out[run + ex + m] = ids[i];
            run += tot;
        }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t launch_init(const QueryDesc* qds, QueryState* sts, const Pools& P, const WorkLists& W, const float* rows,
                       hipStream_t s)
{
    hipLaunchKernelGGL(k_init, dim3(W.nq), dim3(kBlock), 0, s, qds, sts, P, W, W.nq, rows);
    return hipGetLastError();
}

hipError_t launch_init_one(const QueryDesc& qd, QueryDesc* dq, QueryState* sts, const Pools& P, const WorkLists& W,
                           const float* rows, hipStream_t s)
{
    // about 4 K words to clear per clearing workgroup
    const uint32_t words = (48u << qd.regShift) + 2u * (uint32_t)qd.R2words + 9u * (qd.nChunks + 1u);
    const uint32_t clear = std::min(32u, std::max(1u, (words + 4095u) / 4096u));
    if(qd.masks)
        hipLaunchKernelGGL(k_init_one<true>, dim3(1 + clear), dim3(kBlock), 0, s, qd, dq, sts, P, W, rows);
    else
        hipLaunchKernelGGL(k_init_one<false>, dim3(1 + clear), dim3(kBlock), 0, s, qd, dq, sts, P, W, rows);
    return hipGetLastError();
}

template <int NT, int K>
static hipError_t launch_propagate_nt(int model, const QueryDesc* qds, QueryState* sts, const Pools& P,
                                      WorkLists W, uint32_t parity, uint32_t maxPairs, const Launch& L, hipStream_t s)
{
    const size_t scene = (size_t)maxPairs * 2 * sizeof(float4);
    const size_t lds   = scene + (W.few() ? (kFewQueries + 1) * sizeof(uint32_t) : 0u);
    W.listOff          = (uint32_t)(scene / sizeof(uint32_t));
    const dim3 g(L.propGrid), b(NT);
    switch(model)
        {
            case KGMT_MODEL_DOUBLE_INTEGRATOR:
                hipLaunchKernelGGL((k_propagate<KGMT_MODEL_DOUBLE_INTEGRATOR, NT, K>), g, b, lds, s, qds, sts, P, W,
                                   parity);
                break;
            case KGMT_MODEL_DUBINS_AIRPLANE:
                hipLaunchKernelGGL((k_propagate<KGMT_MODEL_DUBINS_AIRPLANE, NT, K>), g, b, lds, s, qds, sts, P, W,
                                   parity);
                break;
            case KGMT_MODEL_DUBINS_5D:
                hipLaunchKernelGGL((k_propagate<KGMT_MODEL_DUBINS_5D, NT, K>), g, b, lds, s, qds, sts, P, W, parity);
                break;
            case KGMT_MODEL_QUADCOPTER:
                hipLaunchKernelGGL((k_propagate<KGMT_MODEL_QUADCOPTER, NT, K>), g, b, lds, s, qds, sts, P, W, parity);
                break;
            case KGMT_MODEL_UNICYCLE:
                hipLaunchKernelGGL((k_propagate<KGMT_MODEL_UNICYCLE, NT, K>), g, b, lds, s, qds, sts, P, W, parity);
                break;
            default: hipLaunchKernelGGL((k_propagate<-1, NT, K>), g, b, lds, s, qds, sts, P, W, parity); break;
        }
    return hipGetLastError();
}

bool launch_supported(uint32_t block, uint32_t lanes)
{
    return (lanes == 1 && (block == 128 || block == 256 || block == 512)) ||
           (block == 256 && (lanes == 2 || lanes == 4));
}

hipError_t launch_propagate(int model, const QueryDesc* qds, QueryState* sts, const Pools& P, const WorkLists& W,
                            uint32_t parity, uint32_t maxPairs, const Launch& L, hipStream_t s)
{
    if(!launch_supported(L.propBlock, L.lanes) || W.tile != L.propBlock / L.lanes) return hipErrorInvalidValue;
    if(L.lanes == 2) return launch_propagate_nt<256, 2>(model, qds, sts, P, W, parity, maxPairs, L, s);
    if(L.lanes == 4) return launch_propagate_nt<256, 4>(model, qds, sts, P, W, parity, maxPairs, L, s);
    switch(L.propBlock)
        {
            case 128: return launch_propagate_nt<128, 1>(model, qds, sts, P, W, parity, maxPairs, L, s);
            case 256: return launch_propagate_nt<256, 1>(model, qds, sts, P, W, parity, maxPairs, L, s);
            default: return launch_propagate_nt<512, 1>(model, qds, sts, P, W, parity, maxPairs, L, s);
        }
}

hipError_t launch_update(const QueryDesc* qds, QueryState* sts, const Pools& P, const WorkLists& W,
                         uint32_t parity, const Launch& L, bool own, hipStream_t s)
{
    const dim3 g(L.chunkGrid), b(kUpd);
    const UpdateArgs a{qds, sts, P, W, parity, own ? 1u : 0u};
    if(W.quads)
        hipLaunchKernelGGL(k_update<true>, g, b, 0, s, a);
    else
        hipLaunchKernelGGL(k_update<false>, g, b, 0, s, a);
    return hipGetLastError();
}

hipError_t launch_build_scene(const float* rows, uint32_t n, uint32_t nGrp, float4* out, int wdim, hipStream_t s)
{
    if(n == 0) return hipSuccess;
    if(wdim == 2)
        hipLaunchKernelGGL(k_build_scene<2>, dim3(1), dim3(kBlock), 0, s, rows, n, nGrp, out);
    else
        hipLaunchKernelGGL(k_build_scene<3>, dim3(1), dim3(kBlock), 0, s, rows, n, nGrp, out);
    return hipGetLastError();
}

hipError_t launch_build_mask_scene(const QueryDesc* qd, const float* rows, uint32_t n, uint32_t nGrp, float4* out,
                                   hipStream_t s)
{
    if(n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_build_mask_scene, dim3(1), dim3(kBlock), 0, s, qd, rows, n, nGrp, out);
    return hipGetLastError();
}

hipError_t launch_finish(const QueryDesc* qds, QueryState* sts, const WorkLists& W, uint32_t parity, hipStream_t s)
{
    hipLaunchKernelGGL(k_finish, dim3(1), dim3(kBlock), 0, s, qds, sts, W, parity);
    return hipGetLastError();
}

hipError_t launch_paths(const QueryDesc* qds, QueryState* sts, const Pools& P, uint32_t nq, float* hostPaths,
                        hipStream_t s)
{
    if(nq == 0) return hipSuccess;
    hipLaunchKernelGGL(k_paths, dim3(nq), dim3(64), 0, s, qds, sts, P, nq, hostPaths);
    return hipGetLastError();
}

hipError_t launch_tree_rows(const float* treeS, const int32_t* parent, const float* cost, uint32_t cap, uint32_t n,
                            int D, uint32_t treeSize, float* rows, int32_t* parents, float* costs, hipStream_t s)
{
    if(n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_tree_rows, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, treeS, parent, cost, cap, n,
                       D, treeSize, rows, parents, costs);
    return hipGetLastError();
}

hipError_t launch_stage_draw(const QueryDesc* qd, int C, uint32_t query, uint32_t itr, uint32_t u0, uint32_t n,
                             float* controls, int32_t* steps, float* ufront, hipStream_t s)
{
    const dim3 g((n + kBlock - 1) / kBlock), b(kBlock);
    if(n == 0) return hipSuccess;
    switch(C)
        {
            case 2: hipLaunchKernelGGL(k_stage_draw<2>, g, b, 0, s, qd, query, itr, u0, n, controls, steps, ufront); break;
            case 3: hipLaunchKernelGGL(k_stage_draw<3>, g, b, 0, s, qd, query, itr, u0, n, controls, steps, ufront); break;
            case 4: hipLaunchKernelGGL(k_stage_draw<4>, g, b, 0, s, qd, query, itr, u0, n, controls, steps, ufront); break;
            default: return hipErrorInvalidValue;
        }
    return hipGetLastError();
}

hipError_t launch_stage_propagate(int model, const QueryDesc& qd, const int32_t* parentIdx, const float* parentStates,
                                  uint32_t nParents, const float* controls, const int32_t* steps, uint32_t n,
                                  const float* rows, uint32_t nObs, float* child, uint8_t* valid, int32_t* r1,
                                  int32_t* r2, hipStream_t s)
{
    if(n == 0) return hipSuccess;
    // more workgroups than the chip holds would build the masks again
    const uint32_t most = model == KGMT_MODEL_QUADCOPTER ? 1024u : 2048u;
    const dim3 g(std::min((n - 1) / kBlock + 1, most)), b(kBlock);
    const size_t lds = (size_t)std::max<uint32_t>(stage_pairs(nObs), 1) * 2 * sizeof(float4);
#define KGMT_STAGE_PROP(M)                                                                                     \
    hipLaunchKernelGGL(k_stage_propagate<M>, g, b, lds, s, qd, parentIdx, parentStates, nParents, controls, steps, \
                       n, rows, nObs, child, valid, r1, r2)
    switch(model)
        {
            case KGMT_MODEL_DOUBLE_INTEGRATOR: KGMT_STAGE_PROP(KGMT_MODEL_DOUBLE_INTEGRATOR); break;
            case KGMT_MODEL_DUBINS_AIRPLANE: KGMT_STAGE_PROP(KGMT_MODEL_DUBINS_AIRPLANE); break;
            case KGMT_MODEL_DUBINS_5D: KGMT_STAGE_PROP(KGMT_MODEL_DUBINS_5D); break;
            case KGMT_MODEL_QUADCOPTER: KGMT_STAGE_PROP(KGMT_MODEL_QUADCOPTER); break;
            case KGMT_MODEL_UNICYCLE: KGMT_STAGE_PROP(KGMT_MODEL_UNICYCLE); break;
            default: return hipErrorInvalidValue;
        }
#undef KGMT_STAGE_PROP
    return hipGetLastError();
}

hipError_t launch_stage_propagate_planner(int model, const QueryDesc* qd, const int32_t* parentIdx,
                                          const float* parentStates, uint32_t nParents, const float* controls,
                                          const int32_t* steps, uint32_t n, const float4* obs, uint32_t nGrp,
                                          uint32_t nObs, float* child, uint8_t* valid, int32_t* r1, int32_t* r2,
                                          uint8_t* check, float* box, hipStream_t s)
{
    if(n == 0) return hipSuccess;
    if(model == KGMT_MODEL_QUADCOPTER)
        {
            const size_t ldsQ = (size_t)std::max<uint32_t>(nGrp * kGroup + mask_pairs(nObs), 1) * 2 * sizeof(float4);
            hipLaunchKernelGGL(k_stage_quad_planner, dim3(2 * ((n - 1) / (3 * kTile) + 1)), dim3(kTile), ldsQ, s, qd,
                               parentIdx, parentStates, nParents, controls, steps, n, obs, nGrp, nObs, child, valid, r1,
                               r2, check);
            return hipGetLastError();
        }
    const dim3 g((n - 1) / kBlock + 1), b(kBlock);
    const size_t lds = (size_t)(nGrp ? nGrp * (1 + kGroup) : 1) * 2 * sizeof(float4);
#define KGMT_STAGE_PROP(M)                                                                                        \
    hipLaunchKernelGGL(k_stage_propagate_planner<M>, g, b, lds, s, qd, parentIdx, parentStates, nParents, controls, \
                       steps, n, obs, nGrp, child, valid, r1, r2, check, box)
    switch(model)
        {
            case KGMT_MODEL_DOUBLE_INTEGRATOR: KGMT_STAGE_PROP(KGMT_MODEL_DOUBLE_INTEGRATOR); break;
            case KGMT_MODEL_DUBINS_AIRPLANE: KGMT_STAGE_PROP(KGMT_MODEL_DUBINS_AIRPLANE); break;
            case KGMT_MODEL_DUBINS_5D: KGMT_STAGE_PROP(KGMT_MODEL_DUBINS_5D); break;
            case KGMT_MODEL_UNICYCLE: KGMT_STAGE_PROP(KGMT_MODEL_UNICYCLE); break;
            default: return hipErrorInvalidValue;
        }
#undef KGMT_STAGE_PROP
    return hipGetLastError();
}

hipError_t launch_stage_frontier_update(const QueryDesc* qd, QueryState* st, const Pools& P, const WorkLists& W,
                                        uint32_t R1, uint32_t itr, uint32_t tree, const float* child,
                                        const int32_t* childParent, const uint8_t* fnext, uint32_t nC,
                                        const int32_t* valid, int32_t* info, hipStream_t s)
{
    const uint32_t n = std::max(std::max(tree, nC), R1);
    hipLaunchKernelGGL(k_stage_fu_nodes, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, qd, P, tree, child,
                       childParent, fnext, nC, valid);
    hipLaunchKernelGGL(k_stage_fu_state, dim3(1), dim3(kBlock), 0, s, qd, st, P, W, itr, tree, nC);
    Launch L;
    L.chunkGrid = 256;
    const hipError_t e = launch_update(qd, st, P, W, 0, L, false, s);
    if(e != hipSuccess) return e;
    hipLaunchKernelGGL(k_stage_fu_info, dim3(1), dim3(64), 0, s, qd, st, P, tree, info);
    return hipGetLastError();
}

hipError_t launch_stage_region_update(const QueryDesc* qd, const int32_t* r1, const int32_t* r2, const uint8_t* valid,
                                      const float* ufront, uint32_t n, const float* score, const uint32_t* actPrev,
                                      uint32_t* actNext, int32_t* total, int32_t* validc, uint8_t* fnext,
                                      hipStream_t s)
{
    if(n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_stage_region_update, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, qd, r1, r2, valid,
                       ufront, n, score, actPrev, actNext, total, validc, fnext);
    return hipGetLastError();
}

hipError_t launch_stage_score(const QueryDesc* qd, const int32_t* total, const int32_t* validc, const uint32_t* act,
                              float* score, hipStream_t s)
{
    hipLaunchKernelGGL(k_stage_score, dim3(1), dim3(kScoreThreads), 0, s, qd, total, validc, act, score);
    return hipGetLastError();
}

hipError_t launch_stage_compact(const uint8_t* flags, uint32_t n, uint32_t* out, uint32_t* count, uint32_t* tmp,
                                hipStream_t s)
{
    const uint32_t m = (n + kChunk - 1) / kChunk;
    if(m) hipLaunchKernelGGL(k_stage_count, dim3(m), dim3(kBlock), 0, s, flags, n, tmp);
    hipLaunchKernelGGL(k_stage_scan, dim3(1), dim3(kScoreThreads), 0, s, tmp, m, count);
    if(m) hipLaunchKernelGGL(k_stage_scatter, dim3(m), dim3(kBlock), 0, s, flags, n, tmp, out);
    return hipGetLastError();
}

hipError_t launch_stage_repeat(const uint32_t* ids, const uint32_t* counts, uint32_t n, uint32_t* out,
                               uint32_t outCap, uint32_t* total, uint32_t* tmp, hipStream_t s)
{
    const uint32_t m = (n + kChunk - 1) / kChunk;
    if(m) hipLaunchKernelGGL(k_stage_sum, dim3(m), dim3(kBlock), 0, s, counts, n, tmp);
    hipLaunchKernelGGL(k_stage_scan, dim3(1), dim3(kScoreThreads), 0, s, tmp, m, total);
    if(m) hipLaunchKernelGGL(k_stage_repeat, dim3(m), dim3(kBlock), 0, s, ids, counts, n, tmp, out, outCap);
    return hipGetLastError();
}

}  // namespace kgmt
