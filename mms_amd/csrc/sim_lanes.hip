// Plain (non-batching) request-loop simulation for gfx950, large batches of bursty streams: lanes at their own pace.
//
// sim_mixed.hip simulates 64 placements of a wavefront on the same request at the same time.  On an overloaded bursty
// stream a placement accepts one request in ten, and the wavefront walks the stages of nearly every request because one
// or another of its lanes accepts it: ten lanes of 64 are at work (configuration 4: 0.71 requests simulated per
// request of the stream, 6.4 lanes accept one).  Here every lane goes through the stream by itself: it stays with a run
// of equal requests (same model, same SLO, one after the other in the stream) as long as it can accept some of it, and then takes
// the next run whose model it hosts.  A step of the wavefront is one request for each lane, whatever requests these are:
//
//   scan    clocks of the last stages of the run's replicas, tournament for the strictly smallest (controller.py:590-598)
//   walk    stage walk, SLO decision, commit (:605-619): the block of walk_asm.inc
//   on      accepted, or rejected and perhaps not the rest of the run: the next request of the run;
//           rejected with all that is left of the run, or the run is over: the next run that the lane hosts.
//
// "All that is left": a lane's clocks change only when it accepts, so while it rejects it keeps its choice, a last-stage clock c
// and a latency l, and a later request at t <= c is rejected if fl(fl(fl(c + l) + overhead) - t) > slo, as the walk's
// finish time is never below that (t >= arrival at every stage and rounding is monotone).  The left side falls with t,
// so the latest arrival of the run decides for the rest of it.  On configuration 4 a wavefront takes about 0.18 steps per request of its stream.
//
// Every lane makes the decisions of the serial loop in the serial loop's order, with the same fp64 operations: results
// equal it bit for bit.
//
// The stream is cut into blocks (MixedArgs::run_block requests); the lanes of a wavefront finish a block before any of
// them starts the next, so that what they read stays together (without the cut they drift apart by a tenth of the stream;
// blocks of 8192 cost 1.5 % more steps, of 4096 3 %, of 1024 12 %).  The runs of a block are listed ahead (list_runs_kernel).  A lane has the
// run that it is at in registers, with up to eight replicas; the next one that it hosts, whose latencies are on their way; and the
// run after that, which is on its way with its entries.  The arrival of the next request of its run is fetched a step ahead.
// Everything is asked for at the end of a step and looked at at the end of the next one: where it comes from L2, a step waits for nothing but
// LDS.  Only replicas beyond the eighth are read where they are looked at, each in two dependent loads.
//
// What bounds it (configuration 4, 131072 simulations, two wavefronts to a SIMD): a step is about 290 instructions, 160 of them vector
// instructions, in 2300 cycles; 56 % of a wavefront's cycles issue, 30 % wait (LDS, and memory where an XCD's L2 misses), the rest wait for the SIMD.
// 506 ms with all lanes at the same request (102 instructions and 978 cycles for each of the stream's), 208 ms here.  On the way:
// entries and latencies as 8 bytes a replica, 2 KB to a row, 338 ms; without the copies for which the compiler waits at the end of a step 261
// (rows of all tiles of an XCD 8.4 MB, 20 % of its L2 requests miss); entries of 16 bits, 512 bytes to a row, and the latencies from a table 226
// (misses 3 %); branch targets on 64-byte boundaries and max-ilp scheduling 212; blocks of 8192 instead of 4096 requests 208.  A wavefront that has a CU to
// itself takes 178 ms for the stream: what is left is the length of one wavefront's step.  All items are on the
// chip from the start, so the time is that of the slowest: half of them end 33 ms before it.  Without effect: tiles composed by the steps that
// their lanes take, items dealt by what they cost, a higher issue priority for the large items' wavefronts, a run of a model with one replica
// left in the step that accepts the last of it (4 % fewer steps; -3.6 to +1.9 % over 18 batches, 0.5 % here): all within 0.5 %.
//
// LDS, the schedule of items and segments and the clocks' layout are those of the loop over runs in sim_mixed.hip.
#include "mmsim_internal.h"
#include "sched.h"
#include "walk_asm.inc"

namespace mmsim {

namespace {

__device__ __forceinline__ double vmax(double x, double y) {  // neither is NaN: no input quieting
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    return r;
}
__device__ __forceinline__ double vmin(double x, double y) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    return r;
}
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }
__device__ __forceinline__ bool in_mask(uint64_t lanes) { return __builtin_amdgcn_inverse_ballot_w64(lanes); }
__device__ __forceinline__ double lds_f64(uint32_t addr) {
    return *reinterpret_cast<const __attribute__((address_space(3))) double *>(addr);
}
__device__ __forceinline__ void lds_set_f64(uint32_t addr, double v) {
    *reinterpret_cast<__attribute__((address_space(3))) double *>(addr) = v;
}
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u32x2 load2(const void *p) {
    return *reinterpret_cast<const __attribute__((address_space(1))) u32x2 *>(reinterpret_cast<uintptr_t>(p));
}
// p, the same in every lane, as a scalar
__device__ __forceinline__ const unsigned char *uniform(const void *p) {
    const uintptr_t v = reinterpret_cast<uintptr_t>(p);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32));
    return reinterpret_cast<const unsigned char *>((uintptr_t)hi << 32 | lo);
}
__device__ __forceinline__ double load_f64(const void *p) {
    return *reinterpret_cast<const __attribute__((address_space(1))) double *>(reinterpret_cast<uintptr_t>(p));
}
__device__ __forceinline__ u32x4 load4(const void *p) {
    return *reinterpret_cast<const __attribute__((address_space(1))) u32x4 *>(reinterpret_cast<uintptr_t>(p));
}
// to = from, here and nowhere else: what follows can overwrite `from` in place.  (A copy of a word that is on its way, as the
// compiler makes them where a value moves up in a loop, would wait for it.)
__device__ __forceinline__ void move(double &to, const u32x2 &from) {
    asm volatile("v_mov_b64 %0, %1" : "+v"(to) : "v"(__builtin_bit_cast(double, from)) : "memory");
}
__device__ __forceinline__ void move(double &to0, double &to1, const u32x4 &from) {
    const f64x2 v = __builtin_bit_cast(f64x2, from);
    asm volatile("v_mov_b64 %0, %2\nv_mov_b64 %1, %3" : "+v"(to0), "+v"(to1) : "v"(v.x), "v"(v.y) : "memory");
}

// Entry of a replica, 16 bits, so that the rows that the wavefronts of an XCD read stay in its L2: clock slot of the group's last
// stage and configuration; what the configuration means for the model is in `stage` ({last-stage latency, stages - 1}, 12 KB for
// 128 models and 11 configurations).
constexpr uint32_t kEntryMore = 1u << 14;   // fourth entry: there are more than four; eighth: more than eight
constexpr uint32_t kEntryNone = 1u << 15;   // first entry: the lane does not host the model
__device__ __forceinline__ uint32_t make_entry(uint32_t d) {
    return rep_addr(d) / kSlotBytes | rep_lat_last(d) << 8 | ((d & kEmpty) ? kEntryNone : 0u);
}

// rep16[tile][model][2][64]: four entries to a word of 8 bytes, from rep32[tile][model][2][64].
__global__ __launch_bounds__(256) void entries_kernel(const MixedArgs a, uint2 *rep16, int64_t rows) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = (int)(i & 63);
    const int64_t row = i >> 6;  // tile * M + model
    if (row >= rows) return;
    for (int h = 0; h < 2; ++h) {
        const uint4 v = a.rep32[(row * 2 + h) * kWave + lane];
        const bool more = h == 0 ? (int32_t)a.rep32[(row * 2 + 1) * kWave + lane].x >= 0
                                 : a.rep_extra > 0 && (int32_t)a.repx32[row * a.rep_extra * kWave + lane] >= 0;
        rep16[(row * 2 + h) * kWave + lane] =
            make_uint2(make_entry(v.x) | make_entry(v.y) << 16, make_entry(v.z) | (make_entry(v.w) | (more ? kEntryMore : 0u)) << 16);
    }
}

// One wavefront per block of requests.  runs == null: how many runs the block has.  Otherwise its runs, from
// runs[off[block]] on.  A run is a row of neighbours in the block with one model and one SLO; requests of no model are in none.
__global__ __launch_bounds__(64) void list_runs_kernel(const Req *streams, const int64_t *stream_off, const int32_t *block_stream,
                                                       const int64_t *block_first, int32_t run_block, const uint32_t *off, Run *runs,
                                                       double *times, uint32_t *counts) {
    const int lane = (int)threadIdx.x;
    const int64_t seed = block_stream[blockIdx.x];
    const int64_t first = block_first[blockIdx.x];  // within the stream
    const int64_t left = stream_off[seed + 1] - stream_off[seed] - first;
    const uint32_t n = (uint32_t)(left < run_block ? left : run_block);
    const Req *reqs = streams + stream_off[seed] + first;
    uint32_t listed = 0;
    for (uint32_t i0 = 0; i0 < n; i0 += 64) {
        const uint32_t i = i0 + (uint32_t)lane;
        bool starts = false;
        Req r{};
        auto same = [&](const Req &x) { return x.m == r.m && __float_as_uint(x.slo) == __float_as_uint(r.slo); };
        if (i < n) {
            r = reqs[i];
            starts = r.m >= 0 && (i == 0 || !same(reqs[i - 1]));
            if (runs) times[stream_off[seed] + first + i] = r.t;
        }
        const uint64_t lanes = ballot(starts);
        if (runs && starts) {
            double latest = r.t;
            uint32_t end = i + 1, next = 0;  // next: model of the next run of the block, if there is one
            for (; end < n; ++end) {
                const Req x = reqs[end];
                if (!same(x)) break;
                latest = x.t > latest ? x.t : latest;
            }
            for (uint32_t k = end; k < n; ++k)
                if (reqs[k].m >= 0) {
                    next = (uint32_t)reqs[k].m;
                    break;
                }
            float bound = (float)latest;
            if ((double)bound < latest) bound = nextafterf(bound, __builtin_inff());
            Run out{r.t, bound, r.slo, i * 8 | (end - 1) * 8 << 16, (uint32_t)r.m | next << 16, {0u, 0u}};
            runs[off[blockIdx.x] + listed + (uint32_t)__popcll(lanes & ((1ull << lane) - 1ull))] = out;
        }
        listed += (uint32_t)__popcll(lanes);
    }
    if (!runs && lane == 0) counts[blockIdx.x] = listed;
}

// SMAX: most stages of a group (bucket).  POW2: every group has 1, 2, 4, 8 or 16 stages.
template <int SMAX, bool POW2>
__global__ __launch_bounds__(kMaxWavesPerBlock *kWave) void sim_lanes_kernel(const MixedArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63);
    if (lds_addr(lds_raw) != 0u) {  // the entries assume that the dynamic LDS starts at address 0
        if (threadIdx.x == 0) *a.error = 1;
        return;
    }
    SchedLds *sched = reinterpret_cast<SchedLds *>(lds_raw);
    const int item0 = a.wg_off[blockIdx.x], n_items = a.wg_off[blockIdx.x + 1] - item0;
    const int part_off = a.part_off[(size_t)blockIdx.x * kMaxWavesPerBlock + wv];
    const int part_bytes = a.part_bytes[(size_t)blockIdx.x * kMaxWavesPerBlock + wv];
    for (int k = (int)threadIdx.x; k < n_items; k += (int)blockDim.x) sched->item[k] = 0u;
    __syncthreads();
    if (part_off < 0) return;
    const uint32_t clk_off = (uint32_t)(a.sched_lds_bytes + part_off) + mixed_clock_offset(a.rmax_lds_bytes, true);
    double *clk = reinterpret_cast<double *>(lds_raw + clk_off) + lane;
    const double overhead = a.fixed_overhead;

    for (int spins = 0;;) {
        const int item_k = sched_claim(sched, a, item0, n_items, part_bytes, lane);
        if (item_k == -1) break;
        if (item_k == -2) {
            __builtin_amdgcn_s_sleep(127);
            if (++spins > a.sched_spin_limit) break;
            continue;
        }
        spins = 0;
        const int tile = a.item_tile[item0 + item_k], seed = a.item_seed[item0 + item_k];
        const int nslots = a.item_nslots[item0 + item_k];
        const int seg = sched_segment(sched, item_k);
        const int wave = a.paired ? tile : seed * a.tiles + tile;
        const size_t out = (size_t)wave * kWave + lane;
        const int64_t off = a.stream_off[seed], R = a.stream_off[seed + 1] - off;
        const int64_t r0 = (int64_t)seg * a.seg_requests, r1 = r0 + a.seg_requests < R ? r0 + a.seg_requests : R;
        const bool last_seg = r1 >= R;
        double *saved = a.state + (size_t)wave * a.state_rows * kWave + lane;
        int32_t n_good = 0;
        double lat_sum = 0.0;
        if (seg > 0) {
            for (int s = 0; s < nslots; ++s) clk[s * kWave] = saved[(size_t)s * kWave];
            n_good = a.n_good[out];
            lat_sum = a.lat_sum[out];
        } else {
            for (int s = 0; s < nslots; ++s) clk[s * kWave] = 0.0;
        }
        const unsigned char *entry_rows = uniform(a.rep16 + (size_t)tile * a.M * 2 * kWave);
        const uint32_t *repx_tile = a.repx32 + (size_t)tile * a.M * a.rep_extra * kWave + lane;
        const uint32_t lane_clk = clk_off + (uint32_t)lane * 8u;
        const uint32_t stage_row = (uint32_t)a.lat_row * 8u;
        const unsigned char *stage = uniform(a.stage);
        auto load_entries = [&](uint32_t m, int half) { return load2(entry_rows + (m * (2u * kWave * 8u) + (uint32_t)lane * 8u) + half * kWave * 8); };
        // {latency, stages - 1} of the entry in the lower (upper) half of w, model m
        auto load_stage = [&](uint32_t w, int upper, uint32_t m) { return load2(stage + ((__builtin_amdgcn_ubfe(w, upper ? 24 : 8, 6) << 3) + m * stage_row)); };

        int64_t bi = a.run_base[seed] + r0 / a.run_block;
        for (int64_t blk = r0; blk < r1; blk += a.run_block, ++bi) {
            const uint32_t run0 = a.run_off[bi], n_runs = (uint32_t)__builtin_amdgcn_readfirstlane((int)(a.run_off[bi + 1] - run0));
            if (n_runs == 0) continue;
            const unsigned char *runs = uniform(a.run_list + run0);
            const unsigned char *times = uniform(a.run_times + off + blk);
            // ---- the lane's run
            uint64_t act = 0;                 // lanes that have one
            uint64_t last = 0;                // ... and are at its last request
            uint64_t more4 = 0, more8 = 0;    // ... whose model has more than four (eight) replicas
            uint32_t at = 0, end = 0, model = 0;  // byte offsets of the arrivals of its present and of its last request
            double t = 0.0, t_next = 0.0;
            float latest = 0.0f, slo = 0.0f;
            uint32_t ca[kPackedReplicas] = {}, word[kPackedReplicas] = {};  // LDS address of the last-stage clock; the same with stages - 1 from bit 20 on
            float l[kPackedReplicas] = {};                                  // last-stage latency
            auto set_entry = [&](int k, uint32_t w, int upper, const u32x2 &st) {
                ca[k] = (__builtin_amdgcn_ubfe(w, upper ? 16 : 0, 8) << 9) + lane_clk;  // (slots are 512 bytes)
                word[k] = ca[k] | st.y << 20;
                l[k] = __uint_as_float(st.x);
            };
            // ---- the next one that it hosts: asked for are its latencies
            uint64_t full = 0;                // lanes that have one
            uint64_t many = 0, lacks = 0;     // ... whose model has more than four replicas, and where entries 4-7 or their latencies are not asked for yet
            uint64_t asked = 0;               // ... where the entries are
            double b_t0 = 0.0, b_limits = 0.0, b_where = 0.0, b_entries = 0.0;  // (all but the first: two words each)
            u32x2 bs[kPackedReplicas] = {}, b_second{};
            // ---- the one after that: it and its entries are asked for
            uint64_t valid = ~0ull;           // lanes that have one
            uint32_t ia = 0;                  // its place in the list
            // (as the words that they come in: loads go straight to the registers that are read a step later)
            u32x4 ahead = load4(runs);
            u32x2 ahead2 = load2(runs + 16);
            u32x2 ahead_entries = load_entries(__builtin_amdgcn_readfirstlane((int)ahead2.y) & 0xFFFFu, 0);

            for (;;) {
                struct Cand {
                    double c;
                    uint32_t w;
                    float l;
                };
                auto first_min = [](const Cand &x, const Cand &y) {  // (the left one wins ties)
                    const bool right = y.c < x.c;
                    return Cand{vmin(x.c, y.c), right ? y.w : x.w, right ? y.l : x.l};
                };
                auto scan = [&](auto J0) {
                    constexpr int j0 = decltype(J0)::value;
                    Cand k[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) k[j] = Cand{lds_f64(ca[j0 + j]), word[j0 + j], l[j0 + j]};
                    return first_min(first_min(k[0], k[1]), first_min(k[2], k[3]));
                };
                Cand win = scan(std::integral_constant<int, 0>{});
                if (__builtin_expect((more4 & act) != 0, 0)) {
                    const Cand x = scan(std::integral_constant<int, 4>{});
                    if (in_mask(more4)) win = first_min(win, x);
                    const uint64_t beyond = more8 & more4;  // (more8 keeps a lane's bit until it takes a run of more than four again)
                    if (__builtin_expect((beyond & act) != 0, 0))
                        if (in_mask(beyond)) {
                            const uint32_t *row = repx_tile + (size_t)model * a.rep_extra * kWave;
                            for (int j = 0; j < a.rep_extra; ++j) {
                                const uint32_t d = row[(size_t)j * kWave];
                                if ((int32_t)d < 0) break;
                                const uint32_t at = rep_addr(d) + clk_off;
                                win = first_min(win, Cand{lds_f64(at), at | rep_stages_m1(d) << 20, a.lat[(size_t)model * a.lat_row + rep_lat_last(d)]});
                            }
                        }
                }
                const uint32_t last_addr = win.w & 0xFFFFFu;
                const int sm1 = (int)(win.w >> 20);
                const uint32_t first_addr = last_addr - (uint32_t)sm1 * kSlotBytes;
                const double l_last = (double)win.l, slo_d = (double)slo;
                const uint64_t found = ballot(win.c < 1e100) & act;  // a clock that is infinite is never chosen (:590-598)
                uint64_t acc = 0;
                if constexpr (SMAX == 4 || SMAX == 16) {
                    const int walk = in_mask(found) ? sm1 : -1;
                    uint64_t saved_exec, mask1, mask2, mask4, mask8;
                    int accepted;
                    double latency, finish_time;
#define MMSIM_WALK(NAME)                                                                                                 \
    asm volatile(NAME##_LEAN_TEXT                                                                                        \
                 : [sv] "=&s"(saved_exec), [acc] "=&v"(accepted), [fin] "=&v"(finish_time), [lat] "=&v"(latency),        \
                   [ng] "+v"(n_good), [ls] "+v"(lat_sum), [m1] "=&s"(mask1), [m2] "=&s"(mask2), [m4] "=&s"(mask4),       \
                   [m8] "=&s"(mask8), [am] "=&s"(acc)                                                                    \
                 : [walk] "v"(walk), [cb] "v"(first_addr), [lc] "v"(l_last), [ts] "v"(t), [slo] "v"(slo_d),              \
                   [oh] "s"(overhead)                                                                                    \
                 : "vcc", "scc", "memory", NAME##_LEAN_CLOBBERS)
                    if constexpr (POW2) {
                        if constexpr (SMAX == 4)
                            MMSIM_WALK(MMSIM_WALK_PU4);
                        else
                            MMSIM_WALK(MMSIM_WALK_PU16);
                    } else {
                        if constexpr (SMAX == 4)
                            MMSIM_WALK(MMSIM_WALK_U4);
                        else
                            MMSIM_WALK(MMSIM_WALK_U16);
                    }
#undef MMSIM_WALK
                } else {
                    const int walk = in_mask(found) ? sm1 : -1;
                    double cv[SMAX], x = t;
#pragma unroll
                    for (int k = 0; k < SMAX; ++k)
                        if (k <= walk) {
                            cv[k] = lds_f64(first_addr + (uint32_t)k * kSlotBytes);
                            x = vmax(x, cv[k]) + l_last;
                            cv[k] = x;
                        }
                    const double latency = (x + overhead) - t;
                    acc = ballot(latency <= slo_d) & found;
                    if (in_mask(acc)) {
                        n_good += 1;
                        lat_sum += latency;
#pragma unroll
                        for (int k = 0; k < SMAX; ++k)
                            if (k <= walk) lds_set_f64(first_addr + (uint32_t)k * kSlotBytes, cv[k]);
                    }
                }
                // ---- what is left of the run
                const double c_fin = (win.c + l_last) + overhead;
                const uint64_t rejects = ballot((double)latest <= win.c) & ballot(c_fin - (double)latest > slo_d) & act & ~acc;
                const uint64_t fin = (last & act) | rejects;
                act &= ~fin;
                at += in_mask(act) ? 8u : 0u;
                t = in_mask(act) ? t_next : t;
                // ---- lanes without a run take the next one, if all of it is here
                const uint64_t take = full & ~lacks & ~act;
                if (in_mask(take)) {
                    t = b_t0;
                    latest = __int_as_float(__double2loint(b_limits));
                    slo = __int_as_float(__double2hiint(b_limits));
                    at = (uint32_t)__double2loint(b_where) & 0xFFFFu;
                    end = (uint32_t)__double2loint(b_where) >> 16;
                    model = (uint32_t)__double2hiint(b_where) & 0xFFFFu;
#pragma unroll
                    for (int k = 0; k < 4; ++k) set_entry(k, (uint32_t)(k < 2 ? __double2loint(b_entries) : __double2hiint(b_entries)), k & 1, bs[k]);
                }
                act |= take;
                more4 &= ~take;
                uint64_t ask1 = 0, ask2 = 0;  // lanes whose next run's entries 4-7 (their latencies) are to be asked for
                if (__builtin_expect(many != 0, 0)) {
                    const uint64_t take2 = many & take;
                    if (in_mask(take2)) {
#pragma unroll
                        for (int k = 4; k < kPackedReplicas; ++k) set_entry(k, k < 6 ? b_second.x : b_second.y, k & 1, bs[k]);
                    }
                    more4 |= take2;
                    more8 = (more8 & ~take) | (ballot((b_second.y & kEntryMore << 16) != 0) & take2);
                    many &= ~take;
                    ask1 = lacks & ~asked;
                    ask2 = lacks & asked;
                    asked |= ask1;
                    lacks &= ~ask2;
                }
                last = ballot(at >= end);
                // ---- where it was taken the one after it moves up, if the lane hosts its model; if it does not, it is passed over
                full &= ~take;
                const uint64_t hosted = ballot((ahead_entries.x & kEntryNone) == 0);
                const uint64_t up = valid & hosted & ~full, on = valid & (up | ~hosted);
                const uint32_t next_model = ahead2.y >> 16;
                if (in_mask(up)) {
                    move(b_t0, b_limits, ahead);
                    move(b_where, ahead2);
                    move(b_entries, ahead_entries);
                }
                // ---- what the next step reads is asked for.  (Behind everything that was: a load that something waits for has all those
                // before it to wait for as well.)
                const uint32_t b_model = (uint32_t)__double2hiint(b_where) & 0xFFFFu;
                if (in_mask(act & ~last)) t_next = load_f64(times + at + 8);
                if (in_mask(up)) {
                    const uint32_t w0 = (uint32_t)__double2loint(b_entries), w1 = (uint32_t)__double2hiint(b_entries);
                    bs[0] = load_stage(w0, 0, b_model);
                    bs[1] = load_stage(w0, 1, b_model);
                    if ((w1 & kEntryNone) == 0) {  // (without a third replica the entries repeat the first and are never chosen)
                        bs[2] = load_stage(w1, 0, b_model);
                        bs[3] = load_stage(w1, 1, b_model);
                    }
                }
                if (__builtin_expect((ask1 | ask2) != 0, 0)) {
                    if (in_mask(ask2)) {
#pragma unroll
                        for (int k = 4; k < kPackedReplicas; ++k) bs[k] = load_stage(k < 6 ? b_second.x : b_second.y, k & 1, b_model);
                    }
                    if (in_mask(ask1)) b_second = load_entries(b_model, 1);
                }
                full |= up;
                const uint64_t many_up = up & ballot(((uint32_t)__double2hiint(b_entries) & kEntryMore << 16) != 0);
                many |= many_up;
                lacks |= many_up;
                asked &= ~up;
                if (in_mask(on)) {
                    ++ia;
                    const unsigned char *run = runs + ia * (uint32_t)sizeof(Run);
                    ahead_entries = load_entries(next_model, 0);
                    ahead = load4(run);  // (the list has a run more than there are)
                    ahead2 = load2(run + 16);
                }
                valid &= ~(on & ballot(ia >= n_runs));
                if ((act | full | valid) == 0) break;
            }
        }

        a.n_good[out] = n_good;
        a.lat_sum[out] = lat_sum;
        if (!last_seg)
            for (int s = 0; s < nslots; ++s) saved[(size_t)s * kWave] = clk[s * kWave];
        sched_hand_back(sched, a, item_k, seg, last_seg, lane);
    }
}

using Kernel = void (*)(const MixedArgs);
template <int SMAX>
Kernel pick_depths(bool pow2) {
    return pow2 ? sim_lanes_kernel<SMAX, true> : sim_lanes_kernel<SMAX, false>;
}

}  // namespace

std::string sim_lanes_kernel_name(const MixedArgs &args, int sb) {
    return "sim_lanes_kernel<" + std::to_string(sb) + (sb != 32 && args.pow2_depths ? ", true>" : ", false>");
}

hipError_t launch_sim_lanes(const MixedArgs &args, int sb, int wpb, size_t lds_bytes, hipStream_t stream, std::string *err) {
    const Kernel kern = sb == 4 ? pick_depths<4>(args.pow2_depths) : sb == 16 ? pick_depths<16>(args.pow2_depths) : sim_lanes_kernel<32, false>;
    hipError_t e = wpb < 1 || wpb > kMaxWavesPerBlock || (sb != 4 && sb != 16 && sb != 32) ? hipErrorInvalidValue : hipSuccess;
    if (e == hipSuccess && lds_bytes > 64 * 1024)
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(kern, dim3((unsigned)args.sched_groups), dim3(wpb * kWave), lds_bytes, stream, args);
        e = hipGetLastError();
    }
    if (e != hipSuccess && err) *err = std::string("sim_lanes launch: ") + hipGetErrorString(e);
    return e;
}

hipError_t launch_entries(const MixedArgs &args, uint2 *rep16, hipStream_t stream) {
    const int64_t rows = (int64_t)args.tiles * args.M;
    hipLaunchKernelGGL(entries_kernel, dim3((unsigned)((rows * kWave + 255) / 256)), dim3(256), 0, stream, args, rep16, rows);
    return hipGetLastError();
}

hipError_t launch_list_runs(const Req *streams, const int64_t *stream_off, const int32_t *block_stream, const int64_t *block_first,
                            int32_t blocks, int32_t run_block, const uint32_t *off, Run *runs, double *times, uint32_t *counts, hipStream_t stream) {
    hipLaunchKernelGGL(list_runs_kernel, dim3((unsigned)blocks), dim3(kWave), 0, stream, streams, stream_off, block_stream, block_first,
                       run_block, off, runs, times, counts);
    return hipGetLastError();
}

}  // namespace mmsim
