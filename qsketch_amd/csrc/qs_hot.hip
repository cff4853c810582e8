// qs_hot.hip -- hot-key filter of a plain insert of 32-bit keys.
//
// Under skew most of a stream belongs to a few thousand keys, and once such a
// key's bucket is linked every insert of it is the same commutative update:
// g[w][j] += 1 for the three counters j of its mask (v3:111-129).  Only the
// inserts into unlinked buckets depend on their order (the promotion point,
// v3:160-190).  So a long insert call runs as:
//   1. the candidates: the keys occurring at least HOT_MIN_RUN times among the
//      first HOT_SAMPLE keys, the HOT_MAX most frequent of them; on a second stream, at
//      the same time as
//   2. the first keys of the call (hot_prefix) through the ordinary pipeline
//      (qs_insert.hip), which links the buckets of the hot keys;
//   3. the hot set: the candidates whose bucket is linked now, in a table of
//      HOT_BUCKETS buckets of 2 slots where each key may sit in one of two
//      buckets (the emptier one when it is placed), so that a lookup is two
//      8-byte reads and no loop; a key that finds both buckets full is left
//      out of the set (it then takes the ordered path, which is always exact);
//   4. the rest of the call in one pass: a hot key is counted in LDS (per
//      persistent block, summed over blocks at the end and added to its high
//      row once), every other key is written, in stream order, to a cold
//      array (packed per chunk, then moved together after a scan);
//   5. the cold array through the ordinary pipeline.
// The result is the sequential one: the hot keys' inserts commute with
// everything after their bucket is linked, and the cold keys keep their
// stream order (so the allocation ids, given in stream order of the
// promoting inserts, are unchanged).  A call whose sample shows no skew
// (candidates covering less than HOT_MIN_COVER of it) runs the rest of the
// call after the prefix through the ordinary pipeline.
//
// qs_hot_split_keys serves a sink whose inserts all commute (the SF sketch,
// qs_sf.hip): no prefix and no link condition; every candidate enters the
// table, and the caller gets the cold keys and the per-slot counts.
#include "qs_internal.h"

#include <cstring>

#define CK(x)                                                                                    \
    do {                                                                                         \
        hipError_t e__ = (x);                                                                    \
        if (e__ != hipSuccess)                                                                   \
            return QS_ERR_HIP;                                                                   \
    } while (0)

#define HOT_SAMPLE (1u << 20)              // candidates come from the first HOT_SAMPLE keys
#define HOT_MIN_RUN 8u                     // a candidate occurs at least this often there
#define HOT_CAND_MAX (HOT_SAMPLE / HOT_MIN_RUN)
static_assert(HOT_CAND_MAX % 1024u == 0, "blocks of k_samp_select");
#define HOT_MAX 8192u                      // hot keys at most
#define HOT_BUCKETS 8192u                  // buckets of 2 slots (load at most 1/2)
#define HOT_SLOTS (HOT_BUCKETS * 2u)
#define HOT_FIRST_RUN 64u                  // candidates this frequent are placed before the others
#define HOT_EMPTY 0xffffffffu              // empty slot (that key is never hot)
#define HOT_THREADS 1024
#define HOT_IPT 16u                        // rows of 64 keys per chunk
#define HOT_CHUNK (64u * HOT_IPT)          // keys per chunk (one wavefront's unit of work)
#define HOT_MIN_KEYS (1ull << 26)          // shorter calls are not filtered
#define HOT_MIN_COVER_NUM 3u               // filter when the candidates cover at least
#define HOT_MIN_COVER_DEN 10u              //   3/10 of the sample

// Keys inserted the ordinary way first: a sixteenth of the call, 2^22 to 2^24.
// A longer prefix links more of the candidates' buckets, but its keys all go
// through the sort.  2^26 keys, Zipf 1.1: 1461 us with 2^24, 1381 with 2^23, 1336
// with 2^22, 1359 with 2^21; 2^27: 2215, 2173, 2186, 2260; 2^28: 4072, 4173, 4310.
// At Zipf 1.5 2^26 keys take 719 us with 2^22 and 868 with 2^24.
static uint64_t hot_prefix(uint64_t n)
{
    const uint64_t p = n / 16;
    return p < (1ull << 22) ? 1ull << 22 : p > (1ull << 24) ? 1ull << 24 : p;
}

// device control words
#define HC_NCAND 0   // candidates (at most HOT_MAX)
#define HC_COVER 1   // sample keys they cover
#define HC_NHOT 2    // keys in the hot table
#define HC_FOUND 3   // keys of the sample that occur often enough
#define HC_TIES 4    // of those, the ones with the least count taken that were looked at
#define HC_WORDS 5

struct qs_hot {
    uint32_t *samp;            // the sample grouped by bin
    uint32_t *scnt;            // its keys per tile and bin, then the bins' starts
    uint32_t *ccount;          // histogram of the counts of its frequent keys
    uint32_t *ck, *cv;         // those keys and their counts
    uint32_t *cand, *ccnt;     // the candidates and their counts
    uint32_t *ctl;             // HC_* words
    uint32_t *h_ctl;           // pinned copy
    uint32_t *tkey;            // hot table: key per slot
    uint32_t *tinfo;           // its link id
    uint32_t *tmask;           // its mask
    uint32_t *tfill;           // entries claimed per bucket while placing
    uint32_t *part;            // per persistent block and slot: hot inserts counted
    uint32_t nblk;             // persistent blocks (rows of part)
    uint32_t *ccold;           // cold keys per chunk, scanned in place (+ total)
    uint32_t *stage;           // per chunk of HOT_CHUNK slots: its cold keys, packed at the front
    uint32_t *bsum;            // block sums of the chunk-count scan (+ total)
    uint64_t chunk_cap;
    uint32_t *cold;            // the cold keys of the call, in stream order
    uint64_t cold_cap;
    uint32_t seq;              // sequence number of the last publication to h_ctl
    hipStream_t side;          // the candidate phase of a plain insert runs here (default priority)
    hipEvent_t ev_fork;        // the caller's stream up to the call
    hipEvent_t ev_cand;        // the candidate phase done
    bool prev_flat;            // the previous call's sample showed no skew
};

// The host reads a few device words without a copy or a synchronisation
// call: one wavefront writes them into coherent pinned host memory and then,
// after a system-scope fence, a new sequence number into the last word; the
// host polls that word.  (The filter's two waits sit between launches; going
// through the runtime's copy and completion path there left the GPU idle for
// milliseconds in some calls.)
#define HOT_PUB_WORDS 8u // h_ctl[0 .. 7) data, h_ctl[7] sequence

__global__ void k_hot_publish(const uint32_t *__restrict__ src, uint32_t nwords, uint32_t *dst, uint32_t seq)
{
    const uint32_t i = threadIdx.x;
    if (i < nwords)
        __hip_atomic_store(dst + i, src[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();
    __syncthreads();
    if (i == 0)
        __hip_atomic_store(dst + HOT_PUB_WORDS - 1, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// publish nwords (< HOT_PUB_WORDS) device words to h->h_ctl and wait for them
static int hot_read(qs_hot *h, const uint32_t *d_src, uint32_t nwords, hipStream_t st)
{
    const uint32_t seq = ++h->seq;
    hipLaunchKernelGGL(k_hot_publish, dim3(1), dim3(64), 0, st, d_src, nwords, h->h_ctl, seq);
    CK(hipGetLastError());
    for (uint64_t it = 1; __atomic_load_n(h->h_ctl + HOT_PUB_WORDS - 1, __ATOMIC_ACQUIRE) != seq; ++it) {
        if ((it & 0xfffffu) == 0) { // now and then: has the stream failed, or finished without it?
            const hipError_t e = hipStreamQuery(st);
            if (e != hipErrorNotReady &&
                __atomic_load_n(h->h_ctl + HOT_PUB_WORDS - 1, __ATOMIC_ACQUIRE) != seq)
                return QS_ERR_HIP;
        }
    }
    return QS_OK;
}

// The two buckets a key may sit in (now and then the same one): two fields of
// one 24-bit product, a full-rate instruction where a 32-bit product takes four
// times as long.
__device__ static inline void hot_buckets(uint32_t key, uint32_t &b1, uint32_t &b2)
{
    const uint32_t h = __umul24(key ^ (key >> 15), 0x9E3779u);
    b1 = h >> 19; // HOT_BUCKETS = 2^13
    b2 = (h >> 6) & (HOT_BUCKETS - 1u);
}

// ---------------------------------------------------------------------------
// Candidates: the sample's keys are split by hash into SAMP_BINS bins, one block
// counts each bin's keys in an LDS table, and the HOT_MAX most frequent of
// those that occur at least HOT_MIN_RUN times are selected by a histogram
// of the counts.  Which keys become candidates moves time only, never the
// result, so a key that finds the LDS table crowded is simply left out.
// (The sample was sorted before, and the candidates sorted again by count:
// 29 launches, about 270 us with their gaps; these four kernels take 65 us at
// Zipf 1.1 over 2^24 keys, 43 of them the block whose bin holds the hottest key.
// On the second stream k_samp_count shares the chip with the prefix: its launch spans
// 50 us in one trace of a 2^28-key call and 228 in another, within the prefix's time.)
// ---------------------------------------------------------------------------
#define SAMP_TILE 8192u // sample keys per block of the split
#define SAMP_TILES (HOT_SAMPLE / SAMP_TILE)
#define SAMP_IPT (SAMP_TILE / 1024u)
#define SAMP_BINS 256u
#define SAMP_SLOTS 8192u   // LDS table of one bin (about 4096 keys)
#define SAMP_PROBES 32u
#define SAMP_ROWS 8u
#define SAMP_COUNTS 4096u  // histogram of candidate counts (the last one holds all above)

__device__ static inline uint32_t samp_hash(uint32_t k)
{
    return k * 0x9E3779B1u;
}
__device__ static inline uint32_t samp_bin(uint32_t k)
{
    return samp_hash(k) >> 24;
}

// keys per bin of each tile; also clears the control words and the histogram
__global__ __launch_bounds__(1024) void k_samp_hist(const uint32_t *__restrict__ keys, uint32_t *__restrict__ cnt,
                                                    uint32_t *__restrict__ ccount, uint32_t *__restrict__ ctl)
{
    __shared__ uint32_t s_cnt[SAMP_BINS];
    const uint32_t t = threadIdx.x, i0 = blockIdx.x * SAMP_TILE + t;
    if (t < SAMP_BINS)
        s_cnt[t] = 0;
    if (blockIdx.x < SAMP_COUNTS / 1024u)
        ccount[blockIdx.x * 1024u + t] = 0;
    if (blockIdx.x == 0 && t < HC_WORDS)
        ctl[t] = 0;
    uint32_t k[SAMP_IPT];
#pragma unroll
    for (uint32_t r = 0; r < SAMP_IPT; ++r)
        k[r] = keys[i0 + r * 1024u];
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < SAMP_IPT; ++r)
        atomicAdd(&s_cnt[samp_bin(k[r])], 1u);
    __syncthreads();
    if (t < SAMP_BINS)
        cnt[blockIdx.x * SAMP_BINS + t] = s_cnt[t];
}

// the keys grouped by bin (any order within one); bin b is
// out[start[b] .. start[b + 1])
__global__ __launch_bounds__(1024) void k_samp_split(const uint32_t *__restrict__ keys,
                                                     const uint32_t *__restrict__ cnt, uint32_t *__restrict__ out,
                                                     uint32_t *__restrict__ start)
{
    __shared__ uint32_t s_pre[4][SAMP_BINS], s_tot[4][SAMP_BINS], s_pos[SAMP_BINS], s_red[4];
    const uint32_t t = threadIdx.x, b = t & (SAMP_BINS - 1u), part = t / SAMP_BINS;
    const uint32_t i0 = blockIdx.x * SAMP_TILE + t;
    uint32_t k[SAMP_IPT];
#pragma unroll
    for (uint32_t r = 0; r < SAMP_IPT; ++r)
        k[r] = keys[i0 + r * 1024u];
    uint32_t pre = 0, tot = 0;
#pragma unroll 8
    for (uint32_t u = 0; u < SAMP_TILES / 4u; ++u) {
        const uint32_t tile = part * (SAMP_TILES / 4u) + u, v = cnt[tile * SAMP_BINS + b];
        tot += v;
        pre += tile < blockIdx.x ? v : 0u;
    }
    s_pre[part][b] = pre;
    s_tot[part][b] = tot;
    __syncthreads();
    uint32_t x = 0;
    if (t < SAMP_BINS) {
        tot = s_tot[0][t] + s_tot[1][t] + s_tot[2][t] + s_tot[3][t];
        pre = s_pre[0][t] + s_pre[1][t] + s_pre[2][t] + s_pre[3][t];
        x = tot;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)x, o, 64);
            x += (t & 63u) >= (uint32_t)o ? y : 0u;
        }
        if ((t & 63u) == 63u)
            s_red[t >> 6] = x;
    }
    __syncthreads();
    if (t < SAMP_BINS) {
        for (uint32_t w = 0; w < t >> 6; ++w)
            x += s_red[w];
        s_pos[t] = x - tot + pre;
        if (blockIdx.x == 0) {
            start[t] = x - tot;
            if (t == SAMP_BINS - 1u)
                start[SAMP_BINS] = x;
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < SAMP_IPT; ++r)
        out[atomicAdd(&s_pos[samp_bin(k[r])], 1u)] = k[r];
}

// counts one bin's keys; those with HOT_MIN_RUN or more are appended to (ck, cv),
// their counts to the histogram
__global__ __launch_bounds__(1024) void k_samp_count(const uint32_t *__restrict__ bins,
                                                     const uint32_t *__restrict__ start, uint32_t *__restrict__ ck,
                                                     uint32_t *__restrict__ cv, uint32_t *__restrict__ ccount,
                                                     uint32_t *__restrict__ ctl)
{
    __shared__ uint32_t s_key[SAMP_SLOTS], s_cnt[SAMP_SLOTS], s_h[SAMP_COUNTS];
    __shared__ uint32_t s_n, s_base;
    const uint32_t t = threadIdx.x, lane = t & 63u;
    for (uint32_t e = t; e < SAMP_SLOTS; e += 1024u) {
        s_key[e] = HOT_EMPTY;
        s_cnt[e] = 0;
    }
    for (uint32_t e = t; e < SAMP_COUNTS; e += 1024u)
        s_h[e] = 0;
    if (t == 0)
        s_n = 0;
    __syncthreads();
    const uint32_t b0 = start[blockIdx.x], b1 = start[blockIdx.x + 1];
    // adds w to key k's count, if there is room for it
    auto add = [&](uint32_t k, uint32_t w) {
        uint32_t sl = (samp_hash(k) >> 11) & (SAMP_SLOTS - 1u);
        for (uint32_t pr = 0; pr < SAMP_PROBES; ++pr, sl = (sl + 1u) & (SAMP_SLOTS - 1u)) {
            uint32_t cur = s_key[sl];
            if (cur == HOT_EMPTY)
                cur = atomicCAS(&s_key[sl], HOT_EMPTY, k);
            if (cur == HOT_EMPTY || cur == k) {
                atomicAdd(&s_cnt[sl], w);
                break;
            }
        }
    };
    // A hot key's bin can hold most of the sample, nearly all of it that key:
    // one block walks 113 rows of the default workload's.  Each wavefront keeps one
    // key and its count in scalar registers (the key that its latest row shared
    // most, or was led by), so such a row costs a compare and a population count,
    // and the LDS table only sees the other lanes: 95 -> 50 us with the default
    // workload, 52 -> 43 with Zipf 1.1 over 2^24 keys.  The loads of SAMP_ROWS rows
    // are in flight together.
    uint32_t hk = HOT_EMPTY, hc = 0; // uniform
    for (uint32_t i0 = b0; i0 < b1; i0 += 1024u * SAMP_ROWS) {
        uint32_t kk[SAMP_ROWS];
#pragma unroll
        for (uint32_t r = 0; r < SAMP_ROWS; ++r) {
            const uint32_t i = i0 + r * 1024u + t;
            kk[r] = bins[i < b1 ? i : b1 - 1u];
        }
#pragma unroll
        for (uint32_t r = 0; r < SAMP_ROWS; ++r) {
            const uint32_t i = i0 + r * 1024u + t, k = kk[r];
            uint64_t left = __ballot(i < b1 && k != HOT_EMPTY); // (the empty marker is never hot)
            const uint64_t kept = __ballot(k == hk) & left;
            hc += (uint32_t)__popcll(kept);
            left &= ~kept;
            if (left == 0)
                continue;
            // the lanes with the first remaining lane's key are added by one lane,
            // or take the kept key's place
            const uint32_t first = (uint32_t)__builtin_ctzll(left);
            const uint32_t fk = (uint32_t)__builtin_amdgcn_readlane((int)k, (int)first);
            const uint64_t same = __ballot(k == fk) & left;
            const uint32_t ns = (uint32_t)__popcll(same);
            uint32_t w = (left >> lane) & 1ull;
            if ((same >> lane) & 1ull)
                w = lane == first ? ns : 0u;
            uint32_t ak = k;
            if (ns > (uint32_t)__popcll(kept)) {
                // the first lane hands the old key's count over instead of its own
                if (lane == first) {
                    ak = hk;
                    w = hc;
                }
                hk = fk;
                hc = ns;
            }
            if (w)
                add(ak, w);
        }
    }
    if (lane == 0 && hc)
        add(hk, hc);
    __syncthreads();
    uint32_t mine = 0;
    for (uint32_t e = t; e < SAMP_SLOTS; e += 1024u)
        if (s_cnt[e] >= HOT_MIN_RUN) {
            ++mine;
            atomicAdd(&s_h[min(s_cnt[e], SAMP_COUNTS - 1u)], 1u);
        }
    uint32_t at = mine ? atomicAdd(&s_n, mine) : 0u;
    __syncthreads();
    if (t == 0)
        s_base = s_n ? atomicAdd(ctl + HC_FOUND, s_n) : 0u;
    __syncthreads();
    at += s_base;
    for (uint32_t e = t; e < SAMP_SLOTS; e += 1024u)
        if (s_cnt[e] >= HOT_MIN_RUN) { // (at most HOT_SAMPLE / HOT_MIN_RUN in all bins)
            ck[at] = s_key[e];
            cv[at] = s_cnt[e];
            ++at;
        }
    for (uint32_t e = t; e < SAMP_COUNTS; e += 1024u)
        if (s_h[e])
            atomicAdd(ccount + e, s_h[e]);
}

// The HOT_MAX most frequent candidates (of those with the least count among
// them, as many as there is room for) to cand, their number and the sample keys
// they cover to the control words.
__global__ __launch_bounds__(1024) void k_samp_select(const uint32_t *__restrict__ ck, const uint32_t *__restrict__ cv,
                                                      const uint32_t *__restrict__ ccount, uint32_t *__restrict__ cand,
                                                      uint32_t *__restrict__ ccnt, uint32_t *__restrict__ ctl)
{
    __shared__ uint32_t s_w[16], s_least, s_room, s_take, s_base, s_cover;
    const uint32_t n = ctl[HC_FOUND];
    if (blockIdx.x * 1024u >= n) // uniform
        return;
    const uint32_t t = threadIdx.x, lane = t & 63u, wv = t >> 6;
    if (t == 0) {
        s_least = 0; // every candidate is taken, unless found otherwise below
        s_room = 0;
        s_take = 0;
        s_cover = 0;
    }
    // thread t holds the four counts from the top: 4095 - 4 t and the three below
    uint32_t h[4], sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        h[k] = ccount[SAMP_COUNTS - 1u - (4u * t + k)];
        sum += h[k];
    }
    uint32_t x = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)x, o, 64);
        x += lane >= (uint32_t)o ? y : 0u;
    }
    if (lane == 63u)
        s_w[wv] = x;
    __syncthreads();
    uint32_t above = x - sum; // candidates with larger counts than h[0]'s
    for (uint32_t w = 0; w < wv; ++w)
        above += s_w[w];
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        if (above <= HOT_MAX && above + h[k] > HOT_MAX) { // one count at most
            s_least = SAMP_COUNTS - 1u - (4u * t + k);
            s_room = HOT_MAX - above;
        }
        above += h[k];
    }
    __syncthreads();
    const uint32_t i = blockIdx.x * 1024u + t;
    const uint32_t c = i < n ? cv[i] : 0u, cl = min(c, SAMP_COUNTS - 1u);
    bool take = i < n && cl > s_least;
    if (i < n && s_least && cl == s_least)
        take = atomicAdd(ctl + HC_TIES, 1u) < s_room;
    const uint64_t m = __ballot(take);
    uint32_t at = 0;
    if (lane == 0 && m)
        at = atomicAdd(&s_take, (uint32_t)__popcll(m));
    at = (uint32_t)__shfl((int)at, 0, 64) + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    if (take)
        atomicAdd(&s_cover, c);
    __syncthreads();
    if (t == 0 && s_take) {
        s_base = atomicAdd(ctl + HC_NCAND, s_take);
        atomicAdd(ctl + HC_COVER, s_cover);
    }
    __syncthreads();
    if (take && s_base + at < HOT_MAX) {
        cand[s_base + at] = ck[i];
        ccnt[s_base + at] = c;
    }
}

__global__ void k_hot_clear(uint32_t *__restrict__ tkey, uint32_t *__restrict__ tfill, uint32_t *__restrict__ ctl)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < HOT_SLOTS)
        tkey[i] = HOT_EMPTY;
    if (i < HOT_BUCKETS)
        tfill[i] = 0;
    if (i == 0)
        ctl[HC_NHOT] = 0;
}

// The candidates whose bucket is linked now enter the hot table, those that the
// sample holds at least lo and fewer than hi times (a key that finds both its
// buckets full stays out, so the most frequent go first: with 8192 keys
// about 1 % of the last placed do).
__global__ void k_hot_build(const uint32_t *__restrict__ cand, const uint32_t *__restrict__ ccnt, uint32_t lo,
                            uint32_t hi, qs_sdesc d0, const uint32_t *__restrict__ low,
                            const uint32_t *__restrict__ masks, uint32_t *__restrict__ tkey,
                            uint32_t *__restrict__ tinfo, uint32_t *__restrict__ tmask, uint32_t *tfill,
                            uint32_t *ctl)
{
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= min(ctl[HC_NCAND], HOT_MAX))
        return;
    const uint32_t k = cand[c];
    if (k == HOT_EMPTY || ccnt[c] < lo || ccnt[c] >= hi)
        return;
    const uint32_t h = k * d0.seed;
    const uint32_t b = qs_fastmod(h, d0.fd_low);
    const uint32_t w = low[(size_t)b * 8u + 7u];
    if (w <= QS_LINK_START)
        return;
    const uint32_t M = masks[qs_fastmod(h, d0.fd_masks)];
    uint32_t b1, b2;
    hot_buckets(k, b1, b2);
    // the emptier bucket first (a racy look: only the placement depends on it)
    if (__hip_atomic_load(tfill + b2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <
        __hip_atomic_load(tfill + b1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        const uint32_t t = b1;
        b1 = b2;
        b2 = t;
    }
    uint32_t pos = atomicAdd(tfill + b1, 1u), hb = b1;
    if (pos >= 2u) {
        pos = atomicAdd(tfill + b2, 1u);
        hb = b2;
    }
    if (pos >= 2u)
        return; // both full: the key stays on the ordered path
    const uint32_t slot = hb * 2u + pos;
    tkey[slot] = k;
    tinfo[slot] = w;
    tmask[slot] = M;
    atomicAdd(ctl + HC_NHOT, 1u);
}

// every candidate enters the hot table (a sink whose inserts all commute)
__global__ void k_hot_build_any(const uint32_t *__restrict__ cand, const uint32_t *__restrict__ ccnt, uint32_t lo,
                                uint32_t hi, uint32_t *__restrict__ tkey, uint32_t *tfill, uint32_t *ctl)
{
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= min(ctl[HC_NCAND], HOT_MAX))
        return;
    const uint32_t k = cand[c];
    if (k == HOT_EMPTY || ccnt[c] < lo || ccnt[c] >= hi)
        return;
    uint32_t b1, b2;
    hot_buckets(k, b1, b2);
    if (__hip_atomic_load(tfill + b2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <
        __hip_atomic_load(tfill + b1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        const uint32_t t = b1;
        b1 = b2;
        b2 = t;
    }
    uint32_t pos = atomicAdd(tfill + b1, 1u), hb = b1;
    if (pos >= 2u) {
        pos = atomicAdd(tfill + b2, 1u);
        hb = b2;
    }
    if (pos >= 2u)
        return; // both full: the key stays cold
    tkey[hb * 2u + pos] = k;
    atomicAdd(ctl + HC_NHOT, 1u);
}

// slot of key k in the LDS copy of the hot table, or -1: both buckets read
// at once, no loop (the empty marker is never looked up: it is never hot)
__device__ static inline int hot_find(const uint2 *skey2, uint32_t k)
{
    uint32_t b1, b2;
    hot_buckets(k, b1, b2);
    const uint2 p = skey2[b1], q = skey2[b2];
    int s = -1;
    s = p.x == k ? (int)(b1 * 2u) : s;
    s = p.y == k ? (int)(b1 * 2u + 1u) : s;
    s = q.x == k ? (int)(b2 * 2u) : s;
    s = q.y == k ? (int)(b2 * 2u + 1u) : s;
    return k == HOT_EMPTY ? -1 : s;
}

// Pass 1 over the keys after the prefix.  A wavefront owns chunks of
// HOT_CHUNK consecutive keys (HOT_IPT rows of 64), loads the next chunk while
// it works on this one, counts hot keys per slot in LDS and writes the
// chunk's cold keys, in stream order, to the front of the chunk's own
// HOT_CHUNK slots of `stage`, and their number to ccold.  Persistent blocks
// (one per CU: the two LDS arrays take 128 KB) take chunks in turn and write
// their row of per-slot counts at the end.
// Bound by VALU issue (55 instructions per 64 keys kept it 80 % busy) and LDS
// conflicts (the two 16-byte reads of a table with 4-slot buckets): buckets of two
// slots, the cheaper hash and addresses from scalar bases took 252 M keys of a
// 2^28-key Zipf 1.1 call from 435 us to 321.
__global__ __launch_bounds__(HOT_THREADS) void k_hot_count(const uint32_t *__restrict__ keys, uint64_t n,
                                                           uint32_t nchunks, const uint32_t *__restrict__ tkey,
                                                           uint32_t *__restrict__ part,
                                                           uint32_t *__restrict__ stage,
                                                           uint32_t *__restrict__ ccold)
{
    __shared__ uint2 skey2[HOT_BUCKETS];
    __shared__ uint32_t scnt[HOT_SLOTS];
    for (uint32_t e = threadIdx.x; e < HOT_BUCKETS; e += HOT_THREADS)
        skey2[e] = reinterpret_cast<const uint2 *>(tkey)[e];
    for (uint32_t e = threadIdx.x; e < HOT_SLOTS; e += HOT_THREADS)
        scnt[e] = 0;
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t nw = gridDim.x * (HOT_THREADS / 64);
    // the chunk number and what follows from it stay in scalar registers
    uint32_t c = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * (HOT_THREADS / 64) + (threadIdx.x >> 6)));
    uint32_t k[HOT_IPT], kn[HOT_IPT];
    auto load = [&](uint32_t ch, uint32_t *v) {
        const uint64_t base = (uint64_t)ch * HOT_CHUNK;
        const uint32_t *src = keys + base;
        if (ch < nchunks && base + HOT_CHUNK <= n) { // uniform: a whole chunk
#pragma unroll
            for (uint32_t r = 0; r < HOT_IPT; ++r)
                v[r] = __builtin_nontemporal_load(src + (r * 64u + lane));
        } else {
            const uint32_t left = ch < nchunks ? (uint32_t)(n - base) : 0u;
#pragma unroll
            for (uint32_t r = 0; r < HOT_IPT; ++r)
                v[r] = r * 64u + lane < left ? __builtin_nontemporal_load(src + (r * 64u + lane)) : HOT_EMPTY;
        }
    };
    load(c, k);
    for (; c < nchunks; c += nw) {
        load(c + nw, kn); // the next chunk, loaded while this one is probed
        const uint64_t base = (uint64_t)c * HOT_CHUNK;
        const uint32_t left = n - base < HOT_CHUNK ? (uint32_t)(n - base) : HOT_CHUNK; // keys of this chunk
        uint32_t cold = 0;
        uint32_t *dst = stage + base;
#pragma unroll
        for (uint32_t r = 0; r < HOT_IPT; ++r) {
            const int s = hot_find(skey2, k[r]); // the key past the end is HOT_EMPTY: -1
            if (s >= 0)
                atomicAdd(&scnt[s], 1u);
            const bool is_cold = (r * 64u + lane < left) & (s < 0);
            const uint64_t m = __ballot(is_cold); // every lane, outside any branch
            if (is_cold)
                dst[cold + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] =
                    k[r];
            cold += (uint32_t)__popcll(m);
        }
        if (lane == 0)
            ccold[c] = cold;
#pragma unroll
        for (uint32_t r = 0; r < HOT_IPT; ++r)
            k[r] = kn[r];
    }
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < HOT_SLOTS; e += HOT_THREADS)
        part[(size_t)blockIdx.x * HOT_SLOTS + e] = scnt[e];
}

// Pass 2: every chunk moves its packed cold keys from `stage` to its scanned
// offset (coff[c] .. coff[c + 1]), so the cold keys end up contiguous in
// stream order.  Only the cold keys are read again, not the whole stream.
__global__ __launch_bounds__(256) void k_hot_move(const uint32_t *__restrict__ stage, uint32_t nchunks,
                                                  const uint32_t *__restrict__ coff, uint32_t *__restrict__ cold)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t nw = gridDim.x * 4u;
    for (uint32_t c = blockIdx.x * 4u + (threadIdx.x >> 6); c < nchunks; c += nw) {
        const uint32_t off = coff[c], cnt = coff[c + 1] - off; // cnt <= HOT_CHUNK
        const uint32_t *src = stage + (size_t)c * HOT_CHUNK;
        uint32_t v[HOT_IPT];
#pragma unroll
        for (uint32_t r = 0; r < HOT_IPT; ++r)
            v[r] = r * 64u + lane < cnt ? __builtin_nontemporal_load(src + r * 64u + lane) : 0u;
#pragma unroll
        for (uint32_t r = 0; r < HOT_IPT; ++r)
            if (r * 64u + lane < cnt)
                cold[(size_t)off + r * 64u + lane] = v[r];
    }
}

// Exclusive scan of the per-chunk cold counts, in place, with the total after
// them: block sums over SCAN_SPAN entries, one block scans those, and every
// block scans its span again from its offset.
#define SCAN_SPAN 8192u // entries per block: 1024 threads x 8

__device__ static inline uint32_t block_excl_scan(uint32_t x, uint32_t *s_w, uint32_t &total)
{
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    uint32_t inc = x;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)inc, o, 64);
        inc += lane >= (uint32_t)o ? y : 0u;
    }
    if (lane == 63)
        s_w[wv] = inc;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
    for (uint32_t w = 0; w < blockDim.x / 64u; ++w) {
        before += w < wv ? s_w[w] : 0u;
        total += s_w[w];
    }
    __syncthreads();
    return before + inc - x;
}

__global__ __launch_bounds__(1024) void k_scan_reduce(const uint32_t *__restrict__ a, uint32_t n,
                                                      uint32_t *__restrict__ bsum)
{
    __shared__ uint32_t s_w[16];
    const uint32_t i0 = blockIdx.x * SCAN_SPAN + threadIdx.x * 8u;
    uint32_t x = 0;
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k)
        x += i0 + k < n ? a[i0 + k] : 0u;
    uint32_t total;
    block_excl_scan(x, s_w, total);
    if (threadIdx.x == 0)
        bsum[blockIdx.x] = total;
}

// one block: exclusive scan of the nb block sums (nb <= 8192), the total to bsum[nb]
__global__ __launch_bounds__(1024) void k_scan_top(uint32_t *__restrict__ bsum, uint32_t nb)
{
    __shared__ uint32_t s_w[16];
    const uint32_t i0 = threadIdx.x * 8u;
    uint32_t v[8], x = 0;
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k) {
        v[k] = i0 + k < nb ? bsum[i0 + k] : 0u;
        x += v[k];
    }
    uint32_t total;
    uint32_t run = block_excl_scan(x, s_w, total);
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k) {
        if (i0 + k < nb)
            bsum[i0 + k] = run;
        run += v[k];
    }
    if (threadIdx.x == 0)
        bsum[nb] = total;
}

__global__ __launch_bounds__(1024) void k_scan_apply(uint32_t *__restrict__ a, uint32_t n,
                                                     const uint32_t *__restrict__ bsum, uint32_t nb)
{
    __shared__ uint32_t s_w[16];
    const uint32_t i0 = blockIdx.x * SCAN_SPAN + threadIdx.x * 8u;
    uint32_t v[8], x = 0;
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k) {
        v[k] = i0 + k < n ? a[i0 + k] : 0u;
        x += v[k];
    }
    uint32_t total;
    uint32_t run = bsum[blockIdx.x] + block_excl_scan(x, s_w, total);
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k) {
        if (i0 + k < n)
            a[i0 + k] = run;
        run += v[k];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0)
        a[n] = bsum[nb];
}

// the hot counts summed over the persistent blocks and added to the high
// rows: a block takes 64 slots, its wavefronts a share of the rows each
#define FLUSH_WAVES 16u // wavefronts per block, each summing every 16th row of part
__global__ __launch_bounds__(64 * FLUSH_WAVES) void k_hot_flush(const uint32_t *__restrict__ part, uint32_t nblk,
                                                                const uint32_t *__restrict__ tkey,
                                                                const uint32_t *__restrict__ tinfo,
                                                                const uint32_t *__restrict__ tmask,
                                                                uint32_t *__restrict__ high)
{
    __shared__ uint32_t s_sum[FLUSH_WAVES][64];
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const uint32_t s = blockIdx.x * 64u + lane;
    uint32_t c = 0;
    for (uint32_t b = wv; b < nblk; b += FLUSH_WAVES)
        c += part[(size_t)b * HOT_SLOTS + s];
    s_sum[wv][lane] = c;
    __syncthreads();
    if (wv != 0)
        return;
    c = 0;
#pragma unroll
    for (uint32_t w = 0; w < FLUSH_WAVES; ++w)
        c += s_sum[w][lane];
    if (!c || tkey[s] == HOT_EMPTY)
        return;
    uint32_t *g = high + (size_t)(tinfo[s] - QS_LINK_START) * 32u;
    for (uint32_t M = tmask[s]; M; M &= M - 1u)
        atomicAdd(g + __builtin_ctz(M), c);
}

// ===========================================================================
// host
// ===========================================================================
uint64_t qs_scan_sums(uint64_t n)
{
    return (n + SCAN_SPAN - 1) / SCAN_SPAN + 1;
}

void qs_scan_u32(uint32_t *a, uint32_t n, uint32_t *bsum, hipStream_t stream)
{
    const uint32_t nb = (uint32_t)(((uint64_t)n + SCAN_SPAN - 1) / SCAN_SPAN); // <= 8192
    hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(1024), 0, stream, a, n, bsum);
    hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, stream, bsum, nb);
    hipLaunchKernelGGL(k_scan_apply, dim3(nb), dim3(1024), 0, stream, a, n, bsum, nb);
}

void qs_hot_state_free(void *state)
{
    qs_hot *h = (qs_hot *)state;
    if (!h)
        return;
    (void)hipFree(h->samp); // and the candidate buffers after it
    (void)hipFree(h->ctl);
    (void)hipFree(h->tkey);
    (void)hipFree(h->tinfo);
    (void)hipFree(h->tmask);
    (void)hipFree(h->tfill);
    (void)hipFree(h->part);
    (void)hipFree(h->ccold);
    (void)hipFree(h->stage);
    (void)hipFree(h->bsum);
    (void)hipFree(h->cold);
    if (h->h_ctl)
        (void)hipHostFree(h->h_ctl);
    if (h->ev_fork)
        (void)hipEventDestroy(h->ev_fork);
    if (h->ev_cand)
        (void)hipEventDestroy(h->ev_cand);
    if (h->side)
        (void)hipStreamDestroy(h->side);
    free(h);
}

void qs_hot_free(qs_sketch *s)
{
    qs_hot_state_free(s->hot);
    s->hot = nullptr;
}

// the filter's scratch in *state (created on first use), sized for `rest`
// keys after the part inserted the ordinary way
static int hot_alloc(void **state, uint64_t rest)
{
    qs_hot *h = (qs_hot *)*state;
    if (!h) {
        h = (qs_hot *)calloc(1, sizeof(qs_hot));
        if (!h)
            return QS_ERR_NOMEM;
        int dev = 0, cu = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cu <= 0)
            cu = 256;
        h->nblk = (uint32_t)cu;
        const uint64_t words = HOT_SAMPLE + (SAMP_TILES + 2u) * SAMP_BINS + SAMP_COUNTS + 2ull * HOT_CAND_MAX +
                               2ull * HOT_MAX;
        bool ok = hipMalloc(&h->samp, 4ull * words) == hipSuccess &&
             hipMalloc(&h->ctl, 4ull * HC_WORDS) == hipSuccess &&
             hipMalloc(&h->tkey, 4ull * HOT_SLOTS) == hipSuccess &&
             hipMalloc(&h->tinfo, 4ull * HOT_SLOTS) == hipSuccess &&
             hipMalloc(&h->tmask, 4ull * HOT_SLOTS) == hipSuccess &&
             hipMalloc(&h->tfill, 4ull * HOT_BUCKETS) == hipSuccess &&
             hipMalloc(&h->part, 4ull * HOT_SLOTS * h->nblk) == hipSuccess &&
             hipHostMalloc(&h->h_ctl, 4ull * HOT_PUB_WORDS, hipHostMallocCoherent) == hipSuccess &&
             hipStreamCreateWithFlags(&h->side, hipStreamNonBlocking) == hipSuccess &&
             hipEventCreateWithFlags(&h->ev_fork, hipEventDisableTiming) == hipSuccess &&
             hipEventCreateWithFlags(&h->ev_cand, hipEventDisableTiming) == hipSuccess;
        if (!ok) { // nothing half built is kept: a later call starts over
            qs_hot_state_free(h);
            return qs_alloc_failed();
        }
        h->scnt = h->samp + HOT_SAMPLE;
        h->ccount = h->scnt + (SAMP_TILES + 2u) * SAMP_BINS;
        h->ck = h->ccount + SAMP_COUNTS;
        h->cv = h->ck + HOT_CAND_MAX;
        h->cand = h->cv + HOT_CAND_MAX;
        h->ccnt = h->cand + HOT_MAX;
        memset(h->h_ctl, 0, 4ull * HOT_PUB_WORDS);
        h->seq = 0;
        *state = h;
    }
    const uint64_t chunks = (rest + HOT_CHUNK - 1) / HOT_CHUNK;
    if (h->chunk_cap < chunks) {
        (void)hipFree(h->ccold);
        (void)hipFree(h->stage);
        (void)hipFree(h->bsum);
        h->ccold = nullptr;
        h->stage = nullptr;
        h->bsum = nullptr;
        h->chunk_cap = 0;
        if (hipMalloc(&h->ccold, 4ull * (chunks + 1)) != hipSuccess ||
            hipMalloc(&h->stage, 4ull * HOT_CHUNK * chunks) != hipSuccess ||
            hipMalloc(&h->bsum, 4ull * ((chunks + SCAN_SPAN - 1) / SCAN_SPAN + 1)) != hipSuccess)
            return qs_alloc_failed();
        h->chunk_cap = chunks;
    }
    if (h->cold_cap < rest) {
        (void)hipFree(h->cold);
        h->cold = nullptr;
        h->cold_cap = 0;
        if (hipMalloc(&h->cold, 4ull * rest) != hipSuccess)
            return qs_alloc_failed();
        h->cold_cap = rest;
    }
    return QS_OK;
}

// Candidates from the first HOT_SAMPLE keys (step 1), queued on `stream`, to
// h->cand.  hot_cand_result then waits for their cover.
static int hot_cand_launch(qs_hot *h, const uint32_t *keys, hipStream_t stream)
{
    uint32_t *start = h->scnt + SAMP_TILES * SAMP_BINS; // SAMP_BINS + 1 words
    hipLaunchKernelGGL(k_samp_hist, dim3(SAMP_TILES), dim3(1024), 0, stream, keys, h->scnt, h->ccount, h->ctl);
    hipLaunchKernelGGL(k_samp_split, dim3(SAMP_TILES), dim3(1024), 0, stream, keys, h->scnt, h->samp, start);
    hipLaunchKernelGGL(k_samp_count, dim3(SAMP_BINS), dim3(1024), 0, stream, h->samp, start, h->ck, h->cv, h->ccount,
                       h->ctl);
    hipLaunchKernelGGL(k_samp_select, dim3(HOT_CAND_MAX / 1024u), dim3(1024), 0, stream, h->ck, h->cv, h->ccount,
                       h->cand, h->ccnt, h->ctl);
    CK(hipGetLastError());
    return QS_OK;
}

// *skewed = whether the candidates cover at least HOT_MIN_COVER of the
// sample (read after the candidate kernels queued on `stream`)
static int hot_cand_result(qs_hot *h, hipStream_t stream, bool *skewed)
{
    *skewed = false;
    const int rc = hot_read(h, h->ctl, HC_WORDS, stream);
    if (rc)
        return rc;
    const uint64_t cover = h->h_ctl[HC_COVER];
    *skewed = h->h_ctl[HC_NCAND] != 0 && cover * HOT_MIN_COVER_DEN >= (uint64_t)HOT_SAMPLE * HOT_MIN_COVER_NUM;
    return QS_OK;
}

// Blocking insert of n 32-bit keys into a plain sketch through the hot-key
// filter.  *used = 0 (and nothing inserted) when the call is too short, its sample
// shows too little skew or the device has no room for the filter's buffers: the
// caller then runs the ordinary insert.
int qs_insert_hot(qs_sketch *s, const void *d_keys, uint64_t n, hipStream_t stream, int *used)
{
    *used = 0;
    if (s->nsk != 1 || s->key_bytes != 4 || n < HOT_MIN_KEYS || n - hot_prefix(n) > 0xffffffffull)
        return QS_OK;
    const uint32_t *keys = (const uint32_t *)d_keys;
    const uint64_t prefix = hot_prefix(n), rest = n - prefix;
    // The filter only saves time, so no call is refused for its memory (8 bytes per
    // key beside the insert's scratch): without room for both it is given back.
    auto no_room = [&]() -> int {
        qs_hot_free(s);
        return QS_OK; // *used = 0: the caller runs the ordinary insert
    };
    int rc = hot_alloc(&s->hot, rest);
    if (rc)
        return rc == QS_ERR_NOMEM ? no_room() : rc;
    qs_hot *h = (qs_hot *)s->hot;
    const qs_sdesc d0 = s->h_desc[0];
    qs_evpair e1, e2;
    const bool timed = s->timing != 0;

    // The insert scratch is sized before the prefix is queued, for the whole
    // call (at least every key after the prefix, the most the cold part can
    // hold): the cold count varies a little between calls (the hot table's
    // placement races), and a call without skew after one with skew runs as
    // one chunk; growing the scratch between launches, or in the next call,
    // would free and allocate.
    auto size_scratch = [&]() -> int {
        const uint64_t offs_n[2] = {0, n};
        const uint64_t cap = qs_chunk_keys(s, offs_n);
        return qs_ensure_scratch(s, n < cap ? n : cap);
    };
    const uint64_t offs_p[2] = {0, prefix};
    bool skewed = false;
    if (!h->prev_flat) {
        // 2. the prefix goes through the ordinary pipeline on the caller's
        // stream while 1. the candidates run on the side stream, from the
        // point the caller's stream had reached at this call (the two share
        // no memory but the keys, which both only read).  The prefix is
        // queued first: its launches are what keeps the GPU busy while the
        // host queues the candidates' short kernels.  The prefix is inserted
        // whatever the sample shows: a prefix and then the rest is the
        // sequential result, as for any call split into chunks.
        rc = size_scratch();
        if (rc)
            return rc == QS_ERR_NOMEM ? no_room() : rc;
        CK(hipEventRecord(h->ev_fork, stream));
        *used = 1;
        rc = qs_insert_set(s, keys, offs_p, nullptr, stream, false, false);
        if (rc)
            return rc;
        CK(hipStreamWaitEvent(h->side, h->ev_fork, 0));
        rc = hot_cand_launch(h, keys, h->side);
        if (rc)
            return rc;
        CK(hipEventRecord(h->ev_cand, h->side));
        rc = hot_cand_result(h, h->side, &skewed); // the GPU runs the prefix meanwhile
        if (rc)
            return rc;
        h->prev_flat = !skewed;
        if (!skewed) { // not skewed enough to pay for the filter: the rest the ordinary way
            CK(hipStreamWaitEvent(stream, h->ev_cand, 0));
            const uint64_t offs_r[2] = {0, rest};
            return qs_insert_set(s, keys + prefix, offs_r, nullptr, stream, true, false);
        }
    } else {
        // The previous call showed no skew: 1. the candidates first, on the
        // caller's stream, so that a call without skew again runs the
        // ordinary pipeline as one chunk (split at the prefix, every bucket
        // the prefix touches would be read and written once more: 0.7 ms
        // of a 2^28-key Zipf 0.8 call).  Either order gives the same state.
        // The candidates are timed with the filter here: the call waits for
        // them.
        qs_evpair e0;
        if (timed)
            qs_tim_begin(s, e0, QS_TK_HOT, 0, stream);
        rc = hot_cand_launch(h, keys, stream);
        if (timed)
            qs_tim_end(s, e0, stream);
        if (rc)
            return rc;
        rc = hot_cand_result(h, stream, &skewed);
        if (rc)
            return rc;
        h->prev_flat = !skewed;
        if (!skewed)
            return QS_OK; // *used = 0: the caller runs the ordinary insert
        rc = size_scratch();
        if (rc)
            return rc == QS_ERR_NOMEM ? no_room() : rc;
        *used = 1;
        rc = qs_insert_set(s, keys, offs_p, nullptr, stream, false, false); // 2. the prefix
        if (rc)
            return rc;
        CK(hipEventRecord(h->ev_cand, stream)); // (the wait below is then already met)
    }
    // 3. the hot set, 4. the filter
    const uint32_t nchunks = (uint32_t)((rest + HOT_CHUNK - 1) / HOT_CHUNK);
    if (timed)
        qs_tim_begin(s, e1, QS_TK_HOT, 0, stream); // a wait for the candidates counts here
    CK(hipStreamWaitEvent(stream, h->ev_cand, 0));
    hipLaunchKernelGGL(k_hot_clear, dim3(HOT_SLOTS / 256), dim3(256), 0, stream, h->tkey, h->tfill, h->ctl);
    for (int first = 1; first >= 0; --first)
        hipLaunchKernelGGL(k_hot_build, dim3(HOT_MAX / 256), dim3(256), 0, stream, h->cand, h->ccnt,
                           first ? HOT_FIRST_RUN : 0u, first ? ~0u : HOT_FIRST_RUN, d0, s->d_low, s->d_masks, h->tkey,
                           h->tinfo, h->tmask, h->tfill, h->ctl);
    hipLaunchKernelGGL(k_hot_count, dim3(h->nblk), dim3(HOT_THREADS), 0, stream, keys + prefix, rest,
                       nchunks, h->tkey, h->part, h->stage, h->ccold);
    qs_scan_u32(h->ccold, nchunks, h->bsum, stream);
    hipLaunchKernelGGL(k_hot_move, dim3(h->nblk * 8u), dim3(256), 0, stream, h->stage, nchunks, h->ccold, h->cold);
    hipLaunchKernelGGL(k_hot_flush, dim3(HOT_SLOTS / 64), dim3(64 * FLUSH_WAVES), 0, stream, h->part, h->nblk, h->tkey,
                       h->tinfo, h->tmask, s->d_high);
    CK(hipGetLastError());
    if (timed)
        qs_tim_end(s, e1, stream);
    rc = hot_read(h, h->ccold + nchunks, 1, stream);
    if (rc)
        return rc;
    const uint64_t ncold = h->h_ctl[0];
    const uint64_t nhot = rest - ncold;
    s->hot_keys += nhot;
    s->keys_inserted += nhot;
    if (timed) { // the filtered keys count as inserted keys of the timed path
        qs_tim_begin(s, e2, QS_TIMING_KERNELS, nhot, stream);
        qs_tim_end(s, e2, stream);
    }

    // 5. the cold keys the ordinary way (blocking: reports a pool error)
    if (ncold == 0) {
        CK(hipMemcpyAsync(s->h_st, s->d_st, sizeof(qs_dev_state), hipMemcpyDeviceToHost, stream));
        CK(hipStreamSynchronize(stream));
        if (s->h_st->err) {
            s->sticky_err = qs_err_code(s->h_st->err);
            return s->sticky_err;
        }
        return QS_OK;
    }
    const uint64_t offs_c[2] = {0, ncold};
    return qs_insert_set(s, h->cold, offs_c, nullptr, stream, true, false);
}

// For a sink whose inserts all commute (the SF sketch): the n keys split into
// hot keys, counted per table slot and persistent block, and cold keys in
// stream order.  out->split = 0 (nothing done) when n < HOT_MIN_KEYS or the
// sample shows too little skew.
int qs_hot_split_keys(void **state, const uint32_t *keys, uint64_t n, hipStream_t stream, qs_hot_split *out)
{
    memset(out, 0, sizeof(*out));
    if (n < HOT_MIN_KEYS || n > 0xffffffffull)
        return QS_OK;
    int rc = hot_alloc(state, n);
    if (rc)
        return rc;
    qs_hot *h = (qs_hot *)*state;
    bool skewed = false;
    rc = hot_cand_launch(h, keys, stream);
    if (rc)
        return rc;
    rc = hot_cand_result(h, stream, &skewed);
    if (rc || !skewed)
        return rc;
    const uint32_t nchunks = (uint32_t)((n + HOT_CHUNK - 1) / HOT_CHUNK);
    hipLaunchKernelGGL(k_hot_clear, dim3(HOT_SLOTS / 256), dim3(256), 0, stream, h->tkey, h->tfill, h->ctl);
    for (int first = 1; first >= 0; --first)
        hipLaunchKernelGGL(k_hot_build_any, dim3(HOT_MAX / 256), dim3(256), 0, stream, h->cand, h->ccnt,
                           first ? HOT_FIRST_RUN : 0u, first ? ~0u : HOT_FIRST_RUN, h->tkey, h->tfill, h->ctl);
    hipLaunchKernelGGL(k_hot_count, dim3(h->nblk), dim3(HOT_THREADS), 0, stream, keys, n, nchunks, h->tkey, h->part,
                       h->stage, h->ccold);
    qs_scan_u32(h->ccold, nchunks, h->bsum, stream);
    hipLaunchKernelGGL(k_hot_move, dim3(h->nblk * 8u), dim3(256), 0, stream, h->stage, nchunks, h->ccold, h->cold);
    CK(hipGetLastError());
    rc = hot_read(h, h->ccold + nchunks, 1, stream);
    if (rc)
        return rc;
    out->split = 1;
    out->cold = h->cold;
    out->ncold = h->h_ctl[0];
    out->part = h->part;
    out->nblk = h->nblk;
    out->tkey = h->tkey;
    out->nslots = HOT_SLOTS;
    return QS_OK;
}
