// Batching request-loop simulation for gfx950, one simulation to a wavefront.
//
// The same loop as sim_batching.hip (simulate_requests_mixed_batching, alpa_serve/simulator/controller.py:631-798), for
// batches that leave the chip room for a wavefront per simulation.  There is one flow of control, so what it turns on is
// scalar, and the lanes hold what it looks things up in, in registers:
//
//   lane e  event slot e: time and group of a pending idle event (:728, :739-740).  The earliest is found by comparing
//           all lanes with the earliest time, which is kept exact (one minimum over the wavefront when an event is
//           taken, none when one is added).
//   lane g  the models of group g, a bit per model (up to 512 of them in ascending order; other batches keep lists).  Which
//           models have waiting requests is a scalar mask, so whether a group that became idle has anything to do is one
//           AND, and only when several of its models wait are the ranks of their heads looked at (:654-664).
//   lane j  entry j of the queue a batch is taken from, sixteen of them, and latency column j (:666-704).
//
// Latency sums are kept by place in the queue, as the octets there keep them, so that they are equal bit for bit (but where simulations are
// cut into runs: add_latency).
//
// Arrivals are looked at eight at a time, one to an octet of lanes (lane 8 i + j: the j-th replica of arrival i's model):
// those at which nothing happens but a place in a queue cost no more than that.  Events that are due are seen to before
// an arrival is looked at, since the clocks it is judged by may change.
//
// What bounds it: one dependent chain per event or arrival.  A wavefront that has its SIMD to itself pays for instructions
// (4 cycles each, whatever they do), taken branches (20 to 30 cycles until the instructions at the target are there), two
// trips to LDS and one to memory per batch; five of them on a SIMD pay for scalar instructions (one in four cycles for all
// of them).  Hence masks in scalars and look-ups in registers instead of lists in LDS, clocks of the window's replicas kept
// in registers as they change, conditions of a window's octets as bits of one mask, and paths laid out so that what happens
// most falls through.
//
// Measured.  30000 requests, 48 models on 24 devices, 128 placements: 25.0 ms with the octets of sim_batching.hip each
// looking at an arrival of its own (per arrival 226 instructions, 18 of them branches, 1746 cycles), 14.2 ms here (117, 11,
// 939).  150000 requests, 96 models on 48 devices, 2048 placements on 4 streams: 161 ms with octets, 90 ms here; of these
// 34 ms since conditions are masks (44 scalar instructions per arrival -> 28), joins of a window's models one reduction
// (octets_or), dropped requests a loop of its own, the next window's rows in LDS.  Tried, no gain: the queue entries of
// arrivals touched a window ahead; the batch's times worked out beside the look at its deadline (14.2 -> 14.6, 90 -> 97 ms: its
// writes by one lane cost more than the chain); six wavefronts to a SIMD.
//
// Counts of groups are in the lanes' registers and counts of models beside the queues until the end: added to global memory where
// a batch is run, each was a load that the batch waited for (128 placements 21.8 -> 16.6 ms with both, scores 14.9; one
// placement with all outputs 18.0 -> 14.5 ms).  Tried, no gain: the next sixteen entries of every queue in LDS, fetched when the batch before
// them was run (14.8 -> 15.0 ms: the wait for entries of a queue is not what a lone wavefront's time goes to).
//
// Few simulations of long streams without per-request outputs are cut into runs (SPANS), as sim_window.hip cuts its own: a run starts a span
// with idle clocks and empty queues, and ends where its clocks, the queues of the models that some group lists and its idle events equal those that
// the next run had there (or its clocks differ where nothing looks any more).  30000 requests, 128 placements, runs agree after 192 requests in the median, 704 at most of 24: 24 runs
// each, 15.4 -> 1.76 ms.  This instance is 3 to 5 % slower by itself (scalar registers that are kept in vector registers), and runs that never agree cost
// up to 13 % (105000 requests of 10 models on 30 single devices, 309 placements, 259 -> 270 ms): runs_agree_early says where the line is.
//
// LDS: the latency table (per workgroup, if it fits), and per wavefront the stage clocks and, per model, its queue: places of
// its head and of its next arrival in the stream's lists, rank of the head, requests accepted; up to 128 models also their replicas; without
// masks the groups' lists of models, if they fit.
#include "mmsim_internal.h"
#include "runs.h"

namespace mmsim {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <typename T>
__device__ __forceinline__ T lds_get(uint32_t addr) {
    return *reinterpret_cast<const __attribute__((address_space(3))) T *>(addr);
}
template <typename T>
__device__ __forceinline__ void lds_put(uint32_t addr, T v) {
    *reinterpret_cast<__attribute__((address_space(3))) T *>(addr) = v;
}
// Marks the places where the lanes' LDS accesses depend on one another (a wavefront's LDS accesses are carried out in
// order; no instruction).
__device__ __forceinline__ void wave_order() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ bool rarely(bool p) { return __builtin_expect(p, 0); }  // (a branch that is not taken costs little)
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }
__device__ __forceinline__ int first_of(uint64_t lanes) { return __builtin_ctzll(lanes); }  // (lanes: not 0)
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ double uni(double v) { return __hiloint2double(uni(__double2hiint(v)), uni(__double2loint(v))); }
__device__ __forceinline__ int lane_value(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ uint32_t lane_value(uint32_t v, int l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, l); }
__device__ __forceinline__ float lane_value(float v, int l) { return __uint_as_float(lane_value(__float_as_uint(v), l)); }
__device__ __forceinline__ double lane_value(double v, int l) {
    return __hiloint2double(lane_value(__double2hiint(v), l), lane_value(__double2loint(v), l));
}
__device__ __forceinline__ uint64_t lane_value(uint64_t v, int l) {
    return (uint64_t)lane_value((uint32_t)(v >> 32), l) << 32 | lane_value((uint32_t)v, l);
}
__device__ __forceinline__ double max_nn(double x, double y) {  // neither is NaN: no input quieting
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    return r;
}
// whether this lane's bit is set (a scalar mask used as a condition: no instruction)
__device__ __forceinline__ bool in_mask(uint64_t lanes) { return __builtin_amdgcn_inverse_ballot_w64(lanes); }
constexpr uint64_t kFirstOfOctets = 0x0101010101010101ull;
// of each octet, the first of its lanes that are in the mask
__device__ __forceinline__ uint64_t first_of_octets(uint64_t lanes) { return lanes & ~((lanes | kFirstOfOctets << 7) - kFirstOfOctets); }
__device__ __forceinline__ int ilog2i(int v) { return 31 - __clz(v); }

// Smallest value of the octet, in all of its lanes; of the wavefront, as a scalar.  A DPP operand needs two wait states
// after the write of its register (s_nop 1).  All lanes must be active.
__device__ __forceinline__ uint32_t oct_min(uint32_t v) {
    asm("s_nop 1\n"
        "v_min_u32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "s_nop 1\n"
        "v_min_u32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
        "s_nop 1\n"
        "v_min_u32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n"
        : "+v"(v));
    return v;
}
__device__ __forceinline__ uint32_t wave_min(uint32_t v) {
    asm volatile(
        "s_nop 1\n"
        "v_min_u32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
        "s_nop 1\n"
        "v_min_u32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
        "s_nop 1\n"
        "v_min_u32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n"
        "s_nop 1\n"
        "v_min_u32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0xf\n"
        "s_nop 1\n"
        "v_min_u32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n"
        "s_nop 1\n"
        "v_min_u32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n"
        "s_nop 1\n"
        : "+v"(v));
    return lane_value(v, 63);
}
// Each word or'ed over the octets (whose lanes hold the same).  All lanes must be active.
#define MMSIM_OR(W, HOW) "v_or_b32_dpp %" #W ", %" #W ", %" #W " " HOW " bank_mask:0xf\n"
#define MMSIM_OR2(HOW) MMSIM_OR(0, HOW) MMSIM_OR(1, HOW) "s_nop 0\n"
#define MMSIM_OR4(HOW) MMSIM_OR(0, HOW) MMSIM_OR(1, HOW) MMSIM_OR(2, HOW) MMSIM_OR(3, HOW)
__device__ __forceinline__ void octets_or(uint32_t (&v)[2]) {
    asm volatile("s_nop 1\n" MMSIM_OR2("row_shr:8 row_mask:0xf") MMSIM_OR2("row_bcast:15 row_mask:0xa") MMSIM_OR2("row_bcast:31 row_mask:0xc")
                 : "+v"(v[0]), "+v"(v[1]));
    for (uint32_t &x : v) x = lane_value(x, 63);
}
__device__ __forceinline__ void octets_or(uint32_t (&v)[4]) {
    asm volatile("s_nop 1\n" MMSIM_OR4("row_shr:8 row_mask:0xf") MMSIM_OR4("row_bcast:15 row_mask:0xa") MMSIM_OR4("row_bcast:31 row_mask:0xc")
                 : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
    for (uint32_t &x : v) x = lane_value(x, 63);
}
#undef MMSIM_OR4
#undef MMSIM_OR2
#undef MMSIM_OR
// Doubles that are never negative nor NaN order as their bit patterns do: the smallest high word, then the smallest low
// word among the lanes that have it (clocks and event times start at +0 and only grow; +inf is allowed).
__device__ __forceinline__ double oct_min(double v) {
    const uint32_t hi = (uint32_t)__double2hiint(v), mh = oct_min(hi);
    const uint32_t ml = oct_min(hi == mh ? (uint32_t)__double2loint(v) : 0xFFFFFFFFu);
    return __hiloint2double((int)mh, (int)ml);
}
__device__ __forceinline__ double wave_min(double v) {
    const uint32_t hi = (uint32_t)__double2hiint(v), lo = (uint32_t)__double2loint(v), mh = wave_min(hi);
    const uint64_t at = ballot(hi == mh);
    uint32_t ml = lane_value(lo, first_of(at));
    if (rarely((at & (at - 1)) != 0)) ml = wave_min(hi == mh ? lo : 0xFFFFFFFFu);
    return __hiloint2double((int)mh, (int)ml);
}

// LATLDS: the latency table is in LDS.  UNIF: every (model,
// configuration) has the same latencies in all of its stages, held once.  OUTPUTS: anything beyond the scores (a.flags
// says what).  MW: 64-bit words that hold a bit per model; 0: any number of models, and groups that list them in any order.
// Then who waits is read from the queues, and the group's list is gone through 64 entries at a time (LDS if it fits): the first of
// the earliest heads by its place in the list.
// SPANS: a simulation is cut into a.spans runs (MW not 0, no per-request outputs).
template <bool LATLDS, bool UNIF, bool OUTPUTS, int MW, bool SPANS>
__global__ __launch_bounds__(kMaxWavesPerBlockBatching *kWave) void sim_batching_solo_kernel(const BatchingArgs a) {
    const int lane = (int)(threadIdx.x & 63), oct = lane >> 3;
    const int wv = uni((int)(threadIdx.x >> 6));
    const unsigned grid_seeds = a.paired ? 1u : (unsigned)a.n_seeds;
    int tile = (int)(blockIdx.x / grid_seeds) * (int)(blockDim.x >> 6) + wv, seed_row = (int)(blockIdx.x % grid_seeds);
    int own = 0;  // the run
    if constexpr (SPANS) {  // (first runs first)
        const int at = (int)blockIdx.x * (int)(blockDim.x >> 6) + wv, sims = a.tiles * (int)grid_seeds;
        own = uni(at / sims);
        const int sim = at - own * sims;
        seed_row = uni(sim / a.tiles);
        tile = sim - seed_row * a.tiles;
    }
    const int M = a.M, NB = a.NB;
    if (LATLDS) {
        const int n = M * a.lat_row * NB;
        for (int i = (int)threadIdx.x; i < n; i += (int)blockDim.x) lds_put<float>((uint32_t)i * 4u, a.lat[i]);
        __syncthreads();
    }
    if (tile >= a.tiles || (SPANS && own >= a.spans)) return;
    // paired batches: the tile's own stream; otherwise every tile on every stream
    const int seed = a.paired ? a.tile_seed[tile] : seed_row;
    const bool want_model = OUTPUTS && (a.flags & MMSIM_WANT_MODEL_COUNTS) != 0;
    const bool want_group = OUTPUTS && (a.flags & MMSIM_WANT_GROUP_COUNTS) != 0;
    const bool want_req = OUTPUTS && !SPANS && (a.flags & MMSIM_WANT_PER_REQUEST) != 0;
    const uint32_t clk = (uint32_t)a.lat_lds_bytes + (uint32_t)wv * (uint32_t)a.wave_lds_bytes;
    const uint32_t queues = clk + (uint32_t)((a.nslots + 4) & ~1) * 8u;  // [M] {requests accepted, head, behind the last arrival so far: places in the stream's lists; rank of the head}

    const int wave = a.paired ? tile : seed * a.tiles + tile;  // where this (tile, stream) pair's results go
    const int64_t off = a.stream_off[seed], R = a.stream_off[seed + 1] - off;
    const Req *__restrict__ reqs = a.streams + off;
    const int64_t *__restrict__ mo = a.mq_off + (size_t)seed * (M + 1);
    const MqEntry *__restrict__ mq = a.mq + mo[0];
    const uint32_t *__restrict__ rows = reinterpret_cast<const uint32_t *>(a.rep8) + (size_t)tile * M * 8;
    constexpr bool ROWSLDS = MW != 0 && 64 * MW <= kSoloRowsInLds;
    const uint32_t rows16 = queues + (uint32_t)M * 16u;  // [M][8] the descriptors' low halves, if they are in LDS
    const uint8_t *__restrict__ more_replicas = a.repx + (size_t)tile * M * a.rep_extra;
    const uint32_t *__restrict__ ginfo = a.ginfo + (size_t)tile * (a.Gmax + 1);
    double *fin_out = a.finish + (size_t)wave * a.Rmax;
    uint8_t *good_out = a.good + (size_t)wave * a.Rmax;
    const double overhead = a.fixed_overhead, inf = __builtin_inf();
    auto lat_at = [&](uint32_t i) -> float { return LATLDS ? lds_get<float>(i * 4u) : a.lat[i]; };

    // ---- state
    for (int s = lane; s < a.nslots; s += kWave) lds_put<double>(clk + (uint32_t)s * 8u, 0.0);
    const int64_t start = SPANS ? (int64_t)own * a.span_blocks * kWave : 0;
    for (int m = lane; m < M; m += kWave) {
        uint32_t at = (uint32_t)(mo[m] - mo[0]);
        if (SPANS && own > 0)  // the model's first arrival in the span
            for (uint32_t end = (uint32_t)(mo[m + 1] - mo[0]); at < end;) {
                const uint32_t mid = (at + end) >> 1;
                if (mq[mid].idx < start) at = mid + 1;
                else end = mid;
            }
        lds_put<u32x4>(queues + (uint32_t)m * 16u, u32x4{0u, at, at, (uint32_t)mq[at].rank});
    }
    if constexpr (ROWSLDS)
        for (int x = lane; x < M * 8; x += kWave) lds_put<uint16_t>(rows16 + (uint32_t)x * 2u, (uint16_t)((rows[x] & 0x1FFFu) | (rows[x] >> 16 & 0x8000u)));
    constexpr int W = MW != 0 ? MW : 1;
    uint64_t members[W] = {};  // lane g: models of group g
    uint32_t list_begin = 0, list_end = 0;  // MW 0, lane g: their places in the lists
    const uint16_t *__restrict__ lists = a.g2m_idx + (size_t)tile * a.members_max;
    const uint32_t lists16 = clk + (uint32_t)batching_solo_bytes(a.nslots, M);
    if (MW == 0 && a.g2m_in_lds)
        for (int x = lane; x < a.members_max; x += kWave) lds_put<uint16_t>(lists16 + (uint32_t)x * 2u, lists[x]);
    if (lane < a.Gmax) {
        const uint16_t *first = a.g2m_off + (size_t)tile * (a.Gmax + 1) + lane;
        list_begin = first[0];
        list_end = first[1];
        if constexpr (MW != 0)
            for (uint32_t x = list_begin; x < list_end; ++x) {
                const int m = lists[x];
#pragma unroll
                for (int i = 0; i < W; ++i) members[i] |= m >> 6 == i ? 1ull << (m & 63) : 0ull;
            }
    }
    const uint32_t group = lane < a.Gmax ? ginfo[lane] : kEmpty;  // lane g: descriptor of group g
    const uint64_t groups = ballot((int32_t)group >= 0);  // (a group that lists no model may still be some model's replica)
    uint64_t waiting[W] = {};  // models with waiting requests
    double ev_t = inf;          // lane e: event slot e
    uint32_t ev_d = 0;
    uint64_t used = 0;          // event slots that hold an event
    const uint64_t slots = ~0ull >> (64 - a.heap_cap);
    double next_due = inf;      // the earliest event's time
    int32_t requests_of_group = 0, good_of_group = 0;  // lane g (a count in global memory would be waited for in every batch)
    int32_t n_good = 0;
    // Of the batch members this lane accounts for.  SPANS: and what its roundings left out (Knuth's two-sum).  Where one run takes over from
    // another depends on which marks were there in time, and so does the order of the additions: with 106 bits the sum of all of them comes out the same
    // wherever that was (unless what lat_rest itself leaves out decides a rounding, which no launch has shown).  It is the exact sum, rounded once, but for that;
    // that of a simulation that is not cut has its own roundings, so the last bits of a sum depend on how many placements there are beside it.
    double lat_sum = 0.0, lat_rest = 0.0;
    auto add_latency = [&](double x) {
        const double sum = lat_sum + x;
        if constexpr (SPANS) {
            const double of_x = sum - lat_sum;
            lat_rest += (lat_sum - (sum - of_x)) + (x - of_x);
        }
        lat_sum = sum;
    };
    int dead = 0;
    const int cand = a.batch_sizes[lane < NB ? lane : NB - 1], cand_col = ilog2i(cand);  // lane q: batch size q and its latency column
    const bool sizes_pow2 = ballot(lane < NB && cand != 1 << lane) == 0ull;
    wave_order();

    // The window of arrivals being looked at: where the lane's replica has its clocks of the last and of the first stage,
    // and these clocks, kept as they change.  (Lanes without a replica: slot 0, not used.)
    uint32_t last = clk;
    double c_last = 0.0, c_first = 0.0;
    uint64_t here = 0;  // octets that hold an arrival; none from when a simulation is given up

    auto set_waiting = [&](int m, bool on) {
#pragma unroll
        for (int i = 0; i < MW; ++i) {
            uint64_t bit = 1ull << (m & 63);
            if (MW > 1) asm("s_cmp_eq_u32 %1, %2\ns_cselect_b64 %0, %3, 0" : "=s"(bit) : "s"(m >> 6), "n"(i), "s"(bit) : "scc");
            waiting[i] = on ? waiting[i] | bit : waiting[i] & ~bit;
        }
    };

    // the models m of these octets wait
    auto add_waiting = [&](int m, uint64_t lanes) {
        if constexpr (MW == 0) {
        } else if constexpr (MW <= 2) {
            uint32_t bits[2 * MW];
#pragma unroll
            for (int i = 0; i < 2 * MW; ++i) bits[i] = in_mask(lanes & ballot(m >> 5 == i)) ? 1u << (m & 31) : 0u;
            octets_or(bits);
#pragma unroll
            for (int i = 0; i < MW; ++i) waiting[i] |= (uint64_t)bits[2 * i + 1] << 32 | bits[2 * i];
        } else {
            for (lanes &= kFirstOfOctets; lanes != 0ull; lanes &= lanes - 1) set_waiting(lane_value(m, first_of(lanes)), true);
        }
    };

    // :654-664 -- among the models of group g with a waiting request, the one whose head arrived first; of several that
    // arrived at the same time the first of the list (which ascends, unless MW is 0)
    auto select_model = [&](uint32_t g) -> int {
        if constexpr (MW == 0) {
            const uint32_t end = lane_value(list_end, (int)g);
            uint32_t best = 0xFFFFFFFFu;
            int pick = -1;
            for (uint32_t x = lane_value(list_begin, (int)g); x < end; x += kWave) {
                const uint32_t at = x + (uint32_t)lane < end ? x + (uint32_t)lane : end - 1u;  // (the last one again: comes later)
                const int m = a.g2m_in_lds ? lds_get<uint16_t>(lists16 + at * 2u) : lists[at];
                const u32x4 queue = lds_get<u32x4>(queues + (uint32_t)m * 16u);
                const uint32_t rank = queue.z != queue.y ? queue.w : 0xFFFFFFFFu, least = wave_min(rank);
                if (least < best) {
                    best = least;
                    pick = lane_value(m, first_of(ballot(rank == least)));
                }
            }
            return pick;
        }
        uint64_t cand[W];
        int n = 0, only = -1;
#pragma unroll
        for (int i = 0; i < MW; ++i) {
            cand[i] = waiting[i] & lane_value(members[i], (int)g);
            n += __builtin_popcountll(cand[i]);
            if (cand[i] != 0ull) only = 64 * i + first_of(cand[i]);
        }
        if (n <= 1) return only;
        uint32_t rank[W], least = 0xFFFFFFFFu;
#pragma unroll
        for (int i = 0; i < MW; ++i) {
            rank[i] = 0xFFFFFFFFu;
            if (in_mask(cand[i])) rank[i] = lds_get<uint32_t>(queues + (uint32_t)(64 * i + lane) * 16u + 12u);
            least = rank[i] < least ? rank[i] : least;
        }
        least = wave_min(least);
        int pick = -1;
#pragma unroll
        for (int i = MW - 1; i >= 0; --i) {
            const uint64_t at = ballot(rank[i] == least);
            if (at != 0ull) pick = 64 * i + first_of(at);
        }
        return pick;
    };

    // takes the lexicographically smallest (time, group) event, which is due at time T == next_due: its descriptor, which
    // orders like the group's index
    auto take_event = [&](double T) -> uint32_t {
        uint64_t at = ballot(ev_t == T) & used;
        int slot = first_of(at);
        uint32_t d = lane_value(ev_d, slot);
        for (at &= at - 1; rarely(at != 0ull); at &= at - 1) {  // several at that time
            const int s2 = first_of(at);
            const uint32_t d2 = lane_value(ev_d, s2);
            if (d2 < d) {
                d = d2;
                slot = s2;
            }
        }
        if (lane == slot) ev_t = inf;
        used &= ~(1ull << slot);
        next_due = wave_min(ev_t);
        return d;
    };

    // :706-732 with :674-704 inlined; the reference's recursion on "nothing servable" is the outer loop
    auto handle = [&](double t0, int m, uint32_t d) {
        const uint32_t g = desc_group(d);
        const int stages = (int)desc_stages_m1(d) + 1;
        const uint32_t gclk = clk + (desc_last_slot(d) - desc_stages_m1(d)) * 8u;
        double c0[4];  // clocks of the group's first four stages (or of what lies behind a shallower group's)
#pragma unroll
        for (int u = 0; u < 4; ++u) c0[u] = lds_get<double>(gclk + (uint32_t)u * 8u);
        // fn(k, clock) for the stages in turn.  Nested, so that a shallow group leaves with one branch taken.
        // (The number of stages anew, or the compiler keeps each comparison as a mask of lanes.)
        auto walk = [&](auto &&fn) {
            int n = stages;
            asm("" : "+s"(n));
            fn(0, c0[0]);
            if (n > 1) {
                fn(1, c0[1]);
                if (n > 2) {
                    fn(2, c0[2]);
                    if (n > 3) {
                        fn(3, c0[3]);
                        for (int k = 4; k < n; ++k) fn(k, lds_get<double>(gclk + (uint32_t)k * 8u));
                    }
                }
            }
        };
        for (;;) {
            const uint32_t lat_mg = ((uint32_t)m * (uint32_t)a.lat_row + desc_lat_off(d)) * (uint32_t)NB;
            const u32x4 queue = lds_get<u32x4>(queues + (uint32_t)m * 16u);
            const int col_j = (lane & 7) < NB ? lane & 7 : NB - 1;
            const float lu = UNIF ? lat_at(lat_mg + (uint32_t)col_j) : 0.0f;
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t arr = uni(queue.z);
            uint32_t h = uni(queue.y);  // arr - h > 0: the caller saw a waiting request
            // lane j takes entry j from the head of the queue on, whether it has arrived yet or not
            const MqEntry *ep = mq + (size_t)h + (lane & 15);
            double2 hv = *reinterpret_cast<const double2 *>(ep);
            int rank = ep->rank, idx = want_req ? ep->idx : 0;
            __builtin_amdgcn_sched_barrier(0);
            // when a batch started now leaves the last stage, lane j: latency column j (:666-672)
            double tcol = t0;
            walk([&](int k, double c) { tcol = max_nn(c, tcol) + (double)(UNIF ? lu : lat_at(lat_mg + (uint32_t)(k * NB + col_j))); });
            tcol += overhead;
            const double alone = lane_value(tcol, 0);
            // drop heads that cannot meet their deadline even alone (:677-686): up to eight at a time
            auto first_that_can = [&](int avail) -> int {  // avail: none of them
                const uint64_t pass = ballot(lane < avail) & ballot(alone <= hv.y);
                const int k = pass != 0ull ? first_of(pass) : avail;
                if (want_req && lane < k) {
                    fin_out[idx] = hv.x;
                    good_out[idx] = 0;
                }
                if (want_group) requests_of_group += lane == (int)g ? k : 0;
                return k;
            };
            auto waiting_heads = [&]() -> int { return (int)(arr - h) < 8 ? (int)(arr - h) : 8; };
            int avail = waiting_heads(), kfirst = first_that_can(avail);  // kfirst: place of the one that leads the batch, among the entries fetched
            while (kfirst == avail) {
                h += (uint32_t)avail;
                if (h == arr) break;  // (else there are more than eight)
                ep = mq + (size_t)h + (lane & 15);
                hv = *reinterpret_cast<const double2 *>(ep);
                rank = ep->rank;
                if (want_req) idx = ep->idx;
                avail = waiting_heads();
                kfirst = first_that_can(avail);
            }
            if (h == arr) {  // none of them (:709-713)
                const int32_t next_rank = lane_value(rank, avail);  // (behind those of the entries fetched last that were looked at)
                set_waiting(m, false);
                if (MW == 0) {  // (select_model looks at it)
                    lds_put<uint32_t>(queues + (uint32_t)m * 16u + 4u, h);
                    wave_order();
                }
                const int m_next = select_model(g);
                lds_put<uint32_t>(queues + (uint32_t)m * 16u + 4u, h);
                lds_put<uint32_t>(queues + (uint32_t)m * 16u + 12u, (uint32_t)next_rank);
                wave_order();
                m = m_next;
                if (m < 0) return;
                continue;
            }
            const uint32_t first = h + (uint32_t)kfirst;  // its place in the model's list
            const double deadline = lane_value(hv.y, kfirst);
            // grow the batch while the first request still meets its deadline (:693-702): lane b tests batch size b, the
            // batch is the last size before the first one that fails
            double tc = tcol;
            if (rarely(!sizes_pow2)) tc = __hiloint2double(__shfl(__double2hiint(tcol), cand_col), __shfl(__double2loint(tcol), cand_col));
            const uint64_t fits = ballot(lane < NB) & ballot(cand <= (int)(arr - first)) & ballot(tc <= deadline);
            const int sizes = first_of(~(fits | 1ull));  // (NB < 64)
            const int bs = lane_value(cand, sizes - 1), col = lane_value(cand_col, sizes - 1);
            // run it (:715-732)
            const int kb = kfirst + bs;  // the rank of the arrival after the batch
            uint32_t next_rank = (uint32_t)lane_value(rank, kb & 15);
            if (rarely(kb >= 16)) next_rank = uni((uint32_t)mq[(size_t)first + (uint32_t)bs].rank);
            double t = t0 + overhead, idle_at = 0.0;
            const float lb = UNIF ? lane_value(lu, col) : 0.0f;
            walk([&](int k, double c) {
                t = max_nn(t, c) + (double)(UNIF ? lb : lat_at(lat_mg + (uint32_t)(k * NB + col)));
                lds_put<double>(gclk + (uint32_t)k * 8u, t);
                if (k == 0) idle_at = uni(t);
            });
            const bool of_group = last == clk + desc_last_slot(d) * 8u;
            c_last = of_group ? t : c_last;
            c_first = of_group ? idle_at : c_first;
            const uint32_t left = first + (uint32_t)bs;  // the batch is the arrivals first .. first+bs-1 of the model
            lds_put<uint32_t>(queues + (uint32_t)m * 16u + 4u, left);
            lds_put<uint32_t>(queues + (uint32_t)m * 16u + 12u, next_rank);
            wave_order();
            if (left == arr) set_waiting(m, false);
            // (sums by place in the queue, see above)
            if (lane >= kfirst && lane < kfirst + bs && lane < 8) add_latency(t - hv.x);
            for (int k = 8; rarely(k < kb); ++k) {
                const double at = k < 16 ? lane_value(hv.x, k) : mq[(size_t)first + (uint32_t)(k - kfirst)].t;
                if (lane == 0) add_latency(t - at);
            }
            if (want_req) {
                if (lane >= kfirst && lane < kb && lane < 16) {
                    fin_out[idx] = t;
                    good_out[idx] = 1;
                }
                for (int k = 16 + lane; k < kb; k += kWave) {
                    const int32_t r = mq[(size_t)first + (uint32_t)(k - kfirst)].idx;
                    fin_out[r] = t;
                    good_out[r] = 1;
                }
            }
            n_good += bs;
            if (want_group) {
                requests_of_group += lane == (int)g ? bs : 0;
                good_of_group += lane == (int)g ? bs : 0;
            }
            if (want_model && lane == 0)
                __hip_atomic_fetch_add(reinterpret_cast<__attribute__((address_space(3))) uint32_t *>(queues + (uint32_t)m * 16u), (uint32_t)bs,
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            if (rarely(used == slots)) {  // given up: no event is due, no arrival left (`dead` is looked at once a window)
                dead = MMSIM_E_OVERFLOW;
                used = 0ull;
                next_due = inf;
                here = 0ull;
                return;
            }
            const int slot = first_of(~used);
            used |= 1ull << slot;
            if (lane == slot) {
                ev_t = idle_at;
                ev_d = d;
            }
            next_due = idle_at < next_due ? idle_at : next_due;
            return;
        }
    };

    // idle events that are due at time tstamp (:739-744)
    auto due_events = [&](double tstamp) {
        while (next_due <= tstamp) {
            if (rarely(used == 0ull)) break;  // (tstamp: +inf)
            const double T = next_due;
            const uint32_t d = take_event(T);
            const int m = select_model(desc_group(d));
            if (m < 0) break;  // the popped event is dropped, later due events stay (:742-743)
            handle(T, m, d);
        }
    };

    // ---- the arrivals: windows of eight.  Requests are fetched a block of 64 ahead, replica rows a window ahead.
    auto fetch_block = [&](int64_t i) -> Req {
        Req r = {0.0, -1, 0.0f};
        if (i + lane < R) r = reqs[i + lane];
        return r;
    };
    auto row_word = [&](int m) -> uint32_t {
        const uint32_t at = (uint32_t)(m < 0 ? 0 : m) * 8u + (uint32_t)(lane & 7);
        if constexpr (ROWSLDS) return (uint32_t)(int32_t)lds_get<int16_t>(rows16 + at * 2u);
        return rows[at];
    };
    auto time_of = [&](const Req &r, int l) -> double { return __hiloint2double(__shfl(__double2hiint(r.t), l), __shfl(__double2loint(r.t), l)); };
    Req block, block_next;
    // of the next window, and the models of the one after it
    int m1, m2;
    uint32_t d1;
    double t1;
    auto start_at = [&](int64_t w) {  // (a multiple of 64)
        block = fetch_block(w);
        block_next = fetch_block(w + kWave);
        m1 = __shfl(block.m, oct);
        m2 = __shfl(block.m, 8 + oct);
        d1 = row_word(m1);
        t1 = time_of(block, oct);
    };

    // ---- SPANS: this wavefront's run and the simulation's others.  What they agree in: clocks, queues of the models that some group lists
    // (what no group turns to waits for ever), and the idle events, in whichever slots.
    typedef const __attribute__((address_space(4))) BatchingArgs ColdArgs;
    Runs runs;
    uint64_t hosted_models[W] = {};
    uint64_t peeked = 0;
    if constexpr (SPANS) {
        runs.start(cold_args<BatchingArgs>(), own);
        for (int g = 0; g < a.Gmax; ++g)
#pragma unroll
            for (int i = 0; i < W; ++i) hosted_models[i] |= lane_value(members[i], g);
    }
    // A state, 64-bit words: accepted requests, event slots in use, clocks, queues {head, behind the last arrival}; a lane each: time and
    // group of the events, latency sums and what they left out; with counts groups {requests, accepted} (lanes) and models
    auto marked = [&](int r, int i) {
        ColdArgs *q = cold_args<BatchingArgs>();
        return q->mark_state + (((size_t)wave * q->spans + r) * q->marks + i) * (size_t)q->state_words;
    };
    auto ended = [&](int r) {
        ColdArgs *q = cold_args<BatchingArgs>();
        return q->end_state + ((size_t)wave * q->spans + r) * (size_t)(q->state_words + kEndWords);
    };
    auto published = [&](int r) {
        ColdArgs *q = cold_args<BatchingArgs>();
        return q->span_sync + (size_t)wave * (q->spans + kSyncWords) + r;
    };
    const int at_queues = 2 + a.nslots, at_lanes = at_queues + M;  // where the queues and the lanes' words begin
    auto save = [&](uint64_t *st) {
        if (lane == 0) {
            tell(st, (uint64_t)(uint32_t)n_good);
            tell(st + 1, used);
        }
        for (int k = lane; k < a.nslots; k += kWave) tell(st + 2 + k, lds_get<uint64_t>(clk + (uint32_t)k * 8u));
        for (int m = lane; m < M; m += kWave) {
            const u32x4 queue = lds_get<u32x4>(queues + (uint32_t)m * 16u);
            tell(st + at_queues + m, (uint64_t)queue.z << 32 | queue.y);
            if (OUTPUTS) tell(st + at_lanes + 5 * kWave + m, (uint64_t)queue.x);
        }
        uint64_t *mine = st + at_lanes + lane;
        tell(mine, (uint64_t)__double_as_longlong(ev_t));
        tell(mine + kWave, (uint64_t)ev_d);
        tell(mine + 2 * kWave, (uint64_t)__double_as_longlong(lat_sum));
        tell(mine + 3 * kWave, (uint64_t)__double_as_longlong(lat_rest));
        if (OUTPUTS) tell(mine + 4 * kWave, (uint64_t)(uint32_t)good_of_group << 32 | (uint32_t)requests_of_group);
    };
    // Clocks that are equal, or that differ before anything that happens from here on (sim_window.hip): arrivals and idle events.
    auto alike = [](uint64_t x, uint64_t y, double before) -> bool {
        return x == y || (__longlong_as_double((long long)x) < before && __longlong_as_double((long long)y) < before);
    };
    auto agree = [&](const uint64_t *st, double unseen) -> bool {
        const uint64_t their_used = (uint64_t)uni((uint32_t)(told(st + 1) >> 32)) << 32 | uni((uint32_t)told(st + 1));
        if (__builtin_popcountll(their_used) != __builtin_popcountll(used)) return false;
        bool same = true, differ = false;
        for (int k = lane; k < a.nslots; k += kWave) {
            const uint64_t theirs = told(st + 2 + k), mine = lds_get<uint64_t>(clk + (uint32_t)k * 8u);
            differ = differ || theirs != mine;
            same = same && alike(theirs, mine, unseen);
        }
#pragma unroll
        for (int i = 0; i < W; ++i) {
            const int m = 64 * i + lane;
            if (in_mask(hosted_models[i]) && m < M) {
                const u32x4 queue = lds_get<u32x4>(queues + (uint32_t)m * 16u);
                same = same && told(st + at_queues + m) == ((uint64_t)queue.z << 32 | queue.y);
            }
        }
        if (ballot(!same) != 0ull) return false;
        if (ballot(differ) != 0ull) {  // the groups' last clocks in the same order
            const uint32_t slot = in_mask(groups) ? desc_last_slot(group) : 0u;
            const double mine = lds_get<double>(clk + slot * 8u), theirs = __longlong_as_double((long long)told(st + 2 + slot));
            for (uint64_t left = groups; left != 0ull; left &= left - 1)
                same = same && (mine < lane_value(mine, first_of(left))) == (theirs < lane_value(theirs, first_of(left)));
            if ((ballot(!same) & groups) != 0ull) return false;
        }
        const double their_t = __longlong_as_double((long long)told(st + at_lanes + lane));
        const uint32_t their_d = (uint32_t)told(st + at_lanes + kWave + lane);
        for (uint64_t left = used; left != 0ull; left &= left - 1) {  // as often there as here
            const double t = lane_value(ev_t, first_of(left));
            const uint32_t d = lane_value(ev_d, first_of(left));
            if (__builtin_popcountll(ballot(ev_t == t) & ballot(ev_d == d) & used) != __builtin_popcountll(ballot(their_t == t) & ballot(their_d == d) & their_used))
                return false;
        }
        return true;
    };
    // Something happens before block `at`: a mark of this run, one of a later run or the block ahead of it, the end of the run (true).
    auto event = [&](uint32_t at) -> bool {
        ColdArgs *q = cold_args<BatchingArgs>();
        if (at >= runs.limit(q)) return true;
        uint64_t *st = marked(runs.in, runs.mark);
        if (runs.in == runs.own) {
            save(st);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (stores of device scope have been carried out then)
            if (lane == 0) tell(published(runs.in), (uint32_t)runs.mark + 1u);
        } else if (!runs.looked) {
            if (uni(told(published(runs.in))) > (uint32_t)runs.mark) {
                asm volatile("" ::: "memory");
                peeked = told(st + 2 + (lane < a.nslots ? lane : 0));
                runs.looked = true;
                runs.next = at + 1u;
                return false;
            }
        } else {
            const double next = lane_value(t1, 0), unseen = q->alike == 0 ? -1.0 : next_due < next ? next_due : next;
            if (ballot(lane < a.nslots && !alike(peeked, lds_get<uint64_t>(clk + (uint32_t)lane * 8u), unseen)) == 0ull) {
                runs.met = agree(st, unseen);
                if (runs.met) return true;
            }
        }
        runs.go_on(q, at);
        return false;
    };
    int64_t from_w = start, w0 = start;
    bool last_one = false;  // this wavefront puts the simulation together
    uint32_t met_again = 0;
    for (;;) {
        bool cut = false;
        if (from_w < R) start_at(from_w);
        for (w0 = from_w; w0 < R && !dead; w0 += 8) {
            if constexpr (SPANS)
                if ((w0 & 63) == 0 && (uint32_t)(w0 >> 6) == runs.next && event((uint32_t)(w0 >> 6))) {
                    cut = true;
                    break;
                }
            const int from = (int)(w0 & 63) + oct;  // the lane that holds this octet's request
            const int n = R - w0 < 8 ? (int)(R - w0) : 8;
            const int m = m1;
            const uint32_t dj = d1;
            const double t = t1;
            last = clk + desc_last_slot(dj) * 8u;
            c_last = lds_get<double>(last);
            c_first = lds_get<double>(last - desc_stages_m1(dj) * 8u);
            if ((w0 & 63) == 56) {
                block = block_next;
                block_next = fetch_block(w0 + 8 + kWave);
            }
            m1 = m2;
            d1 = row_word(m1);  // (past the end of the stream: -1)
            t1 = time_of(block, (from + 8) & 63);
            m2 = __shfl((w0 & 63) == 48 ? block_next.m : block.m, (from + 16) & 63);
            const bool valid = ((int32_t)dj >= 0) & (m >= 0);
            const uint64_t valids = ballot((int32_t)dj >= 0) & ballot(m >= 0), known = ballot(m >= 0);
            const uint64_t hosted = valids & kFirstOfOctets, longer = valids >> 7 & kFirstOfOctets;  // longer: the list may go on
            here = ~0ull >> (64 - 8 * n);
            int cur = 0;             // arrivals before this one are settled
            uint64_t unseen = ~0ull;  // arrivals whose due events have not been seen to
            while (cur < n) {
                uint64_t due = ballot(next_due <= t) & unseen;
                if ((due >> (cur * 8) & 1ull) != 0ull) {  // events first (:739-744)
                    due_events(lane_value(t, cur * 8));
                    unseen = ~0xFFull << (cur * 8);
                    due = ballot(next_due <= t) & unseen;
                }
                const double mn = oct_min(valid ? c_last : inf);
                const uint64_t found = ballot(mn < 1e100);
                // the first listed of those with the smallest last-stage clock
                const uint64_t selected = first_of_octets(ballot(c_last == mn) & valids);
                const uint64_t idle = selected & found & ballot(t >= c_first), special = hosted & (~found | longer);
                const uint64_t left = here & ~0ull << (cur * 8), happens = left & (due | idle | special);
                // those before the first at which something happens join their queues, and that one unless it has events first
                uint64_t joining = left;
                int f = n;
                if (happens != 0ull) {
                    f = first_of(happens) >> 3;
                    joining &= (((due >> (f * 8) & 1ull) != 0ull ? 1ull : 0x100ull) << (f * 8)) - 1ull;
                }
                if (in_mask(joining & known & kFirstOfOctets))
                    __hip_atomic_fetch_add(reinterpret_cast<__attribute__((address_space(3))) uint32_t *>(queues + (uint32_t)m * 16u + 8u), 1u,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                if (want_req && in_mask(joining & kFirstOfOctets & ~hosted)) {
                    fin_out[w0 + oct] = t;
                    good_out[w0 + oct] = 0;
                }
                wave_order();
                add_waiting(m, joining & known);
                cur = f;
                if (happens == 0ull) break;
                const int fl = f * 8;
                if ((due >> fl & 1ull) != 0ull) continue;
                // its group turns to the arrival if it is idle (:746-778)
                cur = f + 1;
                const double tf = lane_value(t, fl);
                const int mf = lane_value(m, fl);
                uint32_t dsel = lane_value(dj, first_of(selected >> fl) + fl);
                if (ROWSLDS) dsel = lane_value(group, first_of(ballot((group & 0x1FFFu) == (dsel & 0x1FFFu)) & groups));
                bool ready = (idle >> fl & 0xFFull) != 0ull;
                if (rarely((special >> fl & 1ull) != 0ull)) {
                    double best = lane_value(mn, fl);
                    if (!(best < 1e100)) {
                        best = 1e100;
                        dsel = kEmpty;
                        ready = false;
                    }
                    if ((longer >> fl & 1ull) != 0ull)
                        for (int x = 0; x < a.rep_extra; ++x) {
                            const uint32_t g = more_replicas[(size_t)mf * a.rep_extra + x];
                            if (g == (uint32_t)a.Gmax) break;
                            const uint32_t d2 = ginfo[g];
                            const double c2 = uni(lds_get<double>(clk + desc_last_slot(d2) * 8u));
                            if (c2 < best) {
                                best = c2;
                                dsel = d2;
                                ready = tf >= uni(lds_get<double>(clk + (desc_last_slot(d2) - desc_stages_m1(d2)) * 8u));
                            }
                        }
                    dsel = uni(dsel);
                    if (rarely(dsel == kEmpty)) {  // every replica's clock is infinite (sim_batching.hip says when)
                        dead = MMSIM_E_UNSUPPORTED;
                        used = 0ull;
                        break;
                    }
                }
                if (ready) handle(tf, mf, dsel);
            }
        }
        // ---- drain (:781-787)
        while (used != 0ull && !dead && !cut) {
            const double T = next_due;
            const uint32_t d = take_event(T);
            const int m = select_model(desc_group(d));
            if (m >= 0) handle(T, m, d);
        }
        if constexpr (!SPANS) break;
        // ---- the end of a run
        ColdArgs *q = cold_args<BatchingArgs>();
        int first = 0, first_mark = -1;
        if (!last_one) {
            uint64_t *e = ended(own);
            save(e);
            if (lane == 0) {
                tell(e + q->state_words, (uint64_t)(uint32_t)dead << 32 | (cut ? (uint32_t)(w0 >> 6) : 0xFFFFFFFFu));
                tell(e + q->state_words + 1, runs.met ? (uint64_t)(uint32_t)runs.in | (uint64_t)(uint32_t)runs.mark << 32 : ~0ull);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            uint32_t before_me = 0;
            if (lane == 0) before_me = __hip_atomic_fetch_add(published(q->spans), 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
            if (uni(before_me) + 1u != (uint32_t)q->spans) return;
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            // All runs have ended: this wavefront follows them from the first on.
            last_one = true;
            n_good = requests_of_group = good_of_group = 0;
            lat_sum = lat_rest = 0.0;
            for (int m = lane; m < M; m += kWave) lds_put<uint32_t>(queues + (uint32_t)m * 16u, 0u);
        } else {
            if (!runs.met) break;
            met_again += 1;
            first = runs.in;
            first_mark = runs.mark;
        }
        const uint64_t *e = nullptr;
        for (int r = first, mark = first_mark;;) {  // run r from that mark of its (-1: from its beginning) to its end
            e = ended(r);
            const uint64_t *b = marked(r, mark < 0 ? 0 : mark);
            const bool whole = mark < 0;
            n_good += (int32_t)uni((uint32_t)(e[0] - (whole ? 0ull : b[0])));
            const int l = at_lanes + 2 * kWave + lane;
            // (A sum that was infinite at the mark: so was a clock, and whoever came to agree with it has an infinite sum as well.)
            const double sum_before = whole ? 0.0 : __longlong_as_double((long long)b[l]);
            add_latency(__longlong_as_double((long long)e[l]));
            if (sum_before < inf) add_latency(-sum_before);
            lat_rest += __longlong_as_double((long long)e[l + kWave]) - (whole ? 0.0 : __longlong_as_double((long long)b[l + kWave]));
            if constexpr (OUTPUTS) {
                const uint64_t v = e[l + 2 * kWave] - (whole ? 0ull : b[l + 2 * kWave]);
                requests_of_group += (int32_t)(uint32_t)v;
                good_of_group += (int32_t)(v >> 32);
                for (int m = lane; m < M; m += kWave) {
                    const int w = at_lanes + 5 * kWave + m;
                    const uint32_t at = queues + (uint32_t)m * 16u;
                    lds_put<uint32_t>(at, lds_get<uint32_t>(at) + (uint32_t)(e[w] - (whole ? 0ull : b[w])));
                }
            }
            const uint64_t to = e[q->state_words + 1];
            if (to == ~0ull) break;
            r = uni((int)(uint32_t)to);
            mark = uni((int)(uint32_t)(to >> 32));
        }
        const uint32_t end = uni((uint32_t)e[q->state_words]);
        dead = uni((int)(uint32_t)(e[q->state_words] >> 32));
        if (dead != 0 || end == 0xFFFFFFFFu) break;
        // The last of them was given up: on from there.
        for (int k = lane; k < a.nslots; k += kWave) lds_put<uint64_t>(clk + (uint32_t)k * 8u, e[2 + k]);
        for (int i = 0; i < W; ++i) {
            const int m = 64 * i + lane;
            uint64_t queue = 0;
            if (m < M) {
                queue = e[at_queues + m];
                const uint32_t at = queues + (uint32_t)m * 16u, head = (uint32_t)queue;
                lds_put<uint32_t>(at + 4u, head);
                lds_put<uint32_t>(at + 8u, (uint32_t)(queue >> 32));
                lds_put<uint32_t>(at + 12u, (uint32_t)mq[head].rank);
            }
            const uint64_t some = ballot((uint32_t)queue != (uint32_t)(queue >> 32));
#pragma unroll
            for (int k = 0; k < W; ++k) waiting[k] = k == i ? some : waiting[k];
        }
        ev_t = __longlong_as_double((long long)e[at_lanes + lane]);
        ev_d = (uint32_t)e[at_lanes + kWave + lane];
        used = (uint64_t)uni((uint32_t)(e[1] >> 32)) << 32 | uni((uint32_t)e[1]);
        next_due = wave_min(ev_t);
        wave_order();
        runs.resume(q, end);
        from_w = (int64_t)end * kWave;
    }
    if constexpr (SPANS) {
        // For the next launch; not before: a run that is taken up again looks at the marks.
        ColdArgs *q = cold_args<BatchingArgs>();
        for (int k = lane; k <= q->spans; k += kWave) tell(published(k), 0u);
        if (lane == 0) tell(published(q->spans + 1), met_again);
    }

    for (int k = 1; k < 8; k *= 2) {
        auto theirs = [&](double x) -> double { return __hiloint2double(__shfl_xor(__double2hiint(x), k), __shfl_xor(__double2loint(x), k)); };
        if constexpr (SPANS) lat_rest += theirs(lat_rest);
        add_latency(theirs(lat_sum));
    }
    if constexpr (SPANS) lat_sum += lat_sum < inf ? lat_rest : 0.0;
    if (lane == 0) {
        const size_t out = (size_t)wave;
        a.n_good[out] = n_good;
        a.lat_sum[out] = lat_sum;
        a.status[out] = dead;
    }
    if (want_group && lane < a.Gmax) {
        a.group_req[(size_t)wave * a.Gmax + lane] = requests_of_group;
        a.group_good[(size_t)wave * a.Gmax + lane] = good_of_group;
    }
    if (want_model) {
        wave_order();
        for (int m = lane; m < M; m += kWave) a.model_good[(size_t)wave * M + m] = lds_get<int32_t>(queues + (uint32_t)m * 16u);
    }
}

#ifdef MMSIM_SOLO_RUNS
constexpr bool kRuns = true;  // the file is compiled once more for simulations cut into runs
#else
constexpr bool kRuns = false;
#endif
template <bool LATLDS, bool UNIF, bool OUTPUTS, int MW>
constexpr auto solo_kernel = sim_batching_solo_kernel<LATLDS, UNIF, OUTPUTS, kRuns && MW == 0 ? 1 : MW, kRuns>;

bool solo_outputs(const BatchingArgs &a) {
    return (a.flags & (MMSIM_WANT_MODEL_COUNTS | MMSIM_WANT_GROUP_COUNTS | MMSIM_WANT_PER_REQUEST)) != 0;
}

}  // namespace

template <>
hipError_t launch_sim_batching_solo<kRuns>(const BatchingArgs &args, int wpb, size_t lds_bytes, hipStream_t stream) {
    const bool ll = args.lat_lds_bytes > 0, unif = args.uniform_stages != 0, outputs = solo_outputs(args);
    if (wpb < 1 || wpb > kMaxWavesPerBlockBatching || args.tile_sims != 1 || !batching_solo_fits(args.NB, args.heap_cap, args.Gmax) || (args.solo == 1 && args.M > kSoloMasks)) return hipErrorInvalidValue;
    if (kRuns && (args.solo != 1 || (args.flags & MMSIM_WANT_PER_REQUEST))) return hipErrorInvalidValue;
    void (*kern)(const BatchingArgs) = nullptr;
#define MMSIM_PICK3(L, U, O)                                       \
    (args.solo == 2  ? solo_kernel<L, U, O, 0>          \
     : args.M <= 64  ? solo_kernel<L, U, O, 1>          \
     : args.M <= 128 ? solo_kernel<L, U, O, 2>          \
     : args.M <= 256 ? solo_kernel<L, U, O, 4>          \
                     : solo_kernel<L, U, O, 8>)
#define MMSIM_PICK2(L, U) (outputs ? MMSIM_PICK3(L, U, true) : MMSIM_PICK3(L, U, false))
#define MMSIM_PICK(L) (unif ? MMSIM_PICK2(L, true) : MMSIM_PICK2(L, false))
    kern = ll ? MMSIM_PICK(true) : MMSIM_PICK(false);
#undef MMSIM_PICK3
#undef MMSIM_PICK2
#undef MMSIM_PICK
    // The kernel takes LDS addresses as numbers from 0 on: its dynamic LDS starts there as long as nothing static lies
    // before it.
    hipFuncAttributes attr;
    hipError_t e = hipFuncGetAttributes(&attr, reinterpret_cast<const void *>(kern));
    if (e != hipSuccess) return e;
    if (attr.sharedSizeBytes != 0) return hipErrorInvalidKernelFile;
    if (lds_bytes > 64 * 1024) {
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
        if (e != hipSuccess) return e;
    }
    const unsigned seeds = (unsigned)(args.paired ? 1 : args.n_seeds);
    const unsigned groups = kRuns ? (unsigned)(((int64_t)args.tiles * seeds * args.spans + wpb - 1) / wpb) : (unsigned)((args.tiles + wpb - 1) / wpb) * seeds;
    hipLaunchKernelGGL(kern, dim3(groups), dim3(wpb * kWave), lds_bytes, stream, args);
    return hipGetLastError();
}

#ifndef MMSIM_SOLO_RUNS
std::string sim_batching_solo_kernel_name(const BatchingArgs &args) {
    return std::string("sim_batching_solo_kernel<") + (args.lat_lds_bytes > 0 ? "true, " : "false, ") +
           (args.uniform_stages != 0 ? "true, " : "false, ") + (solo_outputs(args) ? "true, " : "false, ") + (args.solo == 2 ? "0" : args.M <= 64 ? "1" : args.M <= 128 ? "2" : args.M <= 256 ? "4" : "8") + (args.spans > 1 ? ", true>" : ">");
}
#endif

}  // namespace mmsim
