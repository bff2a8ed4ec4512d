// Plain (non-batching) request-loop simulation for gfx950, small and middle-sized batches: requests side by side.
//
// The request loop of the reference (simulate_requests_mixed, alpa_serve/simulator/controller.py:561-628) is serial
// in its requests, and sim_mixed.hip walks it that way, 64 placements to a wavefront: the fastest form when there
// are enough placements to fill the chip (a hundred thousand simulations), and one wavefront's 470 cycles per
// request when there are not -- a search step of a thousand candidates keeps 16 of the 1024 SIMDs busy.  Here the
// lanes of a wavefront hold W consecutive REQUESTS of one placement (W = 64, 32, 16 or 8; 64 / W placements to a
// wavefront), and a block of W requests takes as many steps as its longest chain of requests that really depend on
// one another, not W.
//
// A step evaluates every pending request of the block against the clocks as they are: choice of the group, stage
// walk, SLO decision.  Which of these verdicts are what the serial loop would find?
//
//   Clocks only ever grow, and only when a request is accepted.  Take a pending request j that chose group h, and
//   let no earlier pending request i that is accepted, or whose verdict is open, list h among its replicas.  Then
//   whatever the earlier ones do, the clocks of h are the same when j's turn comes, and those of the other groups on
//   j's list have not become smaller: j still chooses h (ties go to the group listed first, and h won its ties
//   already) and finds the same times.  Its verdict is final.  A request that does meet such an i waits for the next
//   step, and counts as open for those behind it.
//
// The earliest pending request never waits, so every step settles at least one.  What is left of the dependences of a
// training workload is about 7 to 17 steps for 64 requests, since bursts that overload a model are mostly rejects,
// and a run of rejects is settled in one step.
//
// "Lists h among its replicas" is a bit mask per (request, replica): before the first step of a block every request
// sets its bit in the masks of its groups (gm[slot] in LDS), reads back those of its own replicas and keeps the bits
// of the requests before it.  The tournament that picks the group carries the mask along, so a step decides who has
// to wait with one ballot ("accepted") and one AND, without another trip to LDS.  Requests that wait and are not
// accepted so far, and list several groups, may still be accepted by another of their groups: only these can hold up
// requests that the accepted ones do not hold up (the loop behind the ballot; rare).
//
// Times are the same fp64 operations in the reference's order as in sim_mixed.hip; the latency sum is accumulated in
// arrival order (ordered_sum), so every result equals the serial loop's bit for bit.
//
// What bounds it: a lone wavefront per SIMD is one dependent chain per step, LDS read of the replicas' clocks ->
// tournament -> walk -> ballot -> commit; when several share a SIMD, instruction issue.  Per placement all state is a
// few KB of LDS and nothing in a step touches global memory; requests are fetched two blocks ahead, replica entries
// one block ahead.  Measured, 120280 requests on single-device groups, 64 side by side: 256 placements 2.57 ms, 2902 cycles a
// block, 64 % of them issuing (275 vector, 98 scalar, 35 LDS instructions) and 36 % waiting; 4096 placements, four wavefronts
// to a SIMD, 5.32 ms, 4464 cycles a block, 42 % issuing, 33 % waiting to issue, 25 % for LDS.  (One request after the other, 64 placements to
// a wavefront: 24 ms either way.)
// Few instructions to a step count most where a wavefront is alone.  That a block's second four replicas are in registers like
// the first, instead of being fetched for every step, and that the words that the walk needs are ready for it took, 108000
// requests: 700 placements of single-device groups, a model in 25 on more than four of them, 6.1 -> 5.3 ms, 1025 placements of
// groups up to 16 deep 15.5 -> 13.1 ms, 600 of four-stage pipelines 10.4 -> 9.65 ms.  Batches of up to eight wavefronts to a CU
// whose models have more than eight replicas keep sixteen in registers (EXT 2; 150 to 180 of them) and fetch the others: 12000
// requests, 6 models on 20 devices, up to 12 replicas, 1 / 64 / 700 / 1500 placements 2.7 / 3.3 / 3.9 / 4.4 -> 1.85 / 2.0 / 2.2 /
// 3.1 ms; 12 models on 33 devices, up to 17, 5.7 / 5.9 / 7.1 / 7.6 -> 3.7 / 3.8 / 4.7 / 5.7 ms.
//
// Few simulations of long streams leave most of the chip idle, and a simulation is one chain of blocks.  It is cut into spans then
// (SPANS): a run, a wavefront of its own, starts at the beginning of every span with all clocks at zero, as if nothing had come before.
// That is wrong at first.  But what a simulation does next depends on its clocks alone, and clocks forget: a group that was
// idle finishes its next request at a time that does not depend on what it did before, and one that rejected until it had caught up
// agrees soon after.  So a run goes on behind its span and compares its clocks with those that the next run had at the same places
// (marks: it left them in memory on its way).  Where all clocks are equal, bit for bit, or differ in ways that no request can see (event), both runs do the same for ever, and the one
// that started further on has done it already: the run ends.  The first run is what the simulation does; where it ended
// the run that it met takes over, and so on: the results are the serial loop's.  A run that meets nobody within half a span (48 blocks
// at least) is given up; the wavefront that ends last follows the runs, takes up again one that was given up where
// it is needed, and the first run never gives up: runs that never agree cost what they take from the first one, not the result.
// Counts are differences between a run's end and the mark at which it was taken over; latencies are kept per request and added in their
// order by a second kernel (LatencySum).  Runs agree after 200 to 2000 requests of bursty streams (of 108000 requests at 0.6 accepted, 32 models
// on 32 single devices: 1000 in the median, 4000 at most of 180; eight four-stage pipelines: 400, 430), or never: steady overload, or groups
// that are all idle most of the time, whose requests go round in the order the groups were used.
// Kernels, 108000 requests: 700 placements of single devices, four runs each, 5.2 -> 2.9 + 0.2 ms (three wavefronts to a SIMD take 1.9 times
// as long as one: issue); 600 of four-stage pipelines, five, 9.6 -> 3.4 + 0.3; 1025 up to 16 deep, three, 13.1 -> 8.4 + 0.3; one placement, 30000
// requests, 24 runs, 1.85 -> 0.21 + 0.10 ms.  A run that is taken up again looks for the marks of the others as the first one does (five even streams of 82000 requests
// at load 0.4, three replicas to a model, 20 such meetings: 4.9 -> 1.4 and 5.5 -> 3.1 ms, and 30 % slower with more wavefronts to a SIMD: runs_agree_early).  Where no
// runs agree ten placements of 115532 requests, cut into 2 to 64 runs, take 4.7 -> 5.0 to 5.2 ms: this instance keeps scalar registers in vector registers and is up to 8 %
// slower by itself; the wavefronts' priorities (s_setprio for the first run and one taken up again) change nothing.
//
// LDS of one placement (byte offsets in WindowArgs, built by the wavefront itself from the packed placement):
//   clk  [slots+SMAX] f64   stage clocks, a placement's groups laid end to end, and SMAX slots for what does not count
//   gm   [slots+SMAX] u64   mask of the block's requests that list the group whose last slot this is
//   cnt  [slots+SMAX] u64   requests (low half) and accepted requests (high half) of that group  (OUTPUTS)
//   rep  [M][4] {u32, f32}  entry word and last-stage latency of the first four replicas, in group order
//   ext  [..][4] {u32, f32} further replicas, four to a chunk; xi[M]: first chunk | chunks << 16
//   bits [M][GW] u32        which groups host the model (used while the entries are made)
//   gd   [Gmax] u32         entry word of every group
//   mcnt [M] u32            accepted requests per model  (OUTPUTS)
// Entry word: bits 0-14 LDS address / 8 of the group's last-stage clock, 15-19 stages - 1, 20-29 index of its
// last-stage latency in the model's row of the latency table, 30 "there are more" (fourth entry), "than eight" (third), "than sixteen" (second), 31 "no such replica":
// the word then repeats the first replica's (which wins every tie against its copies) or, without any replica, the
// placement's first slot.
#include "mmsim_internal.h"
#include "runs.h"

namespace mmsim {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63); }
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }
// whether this lane's bit is set (a scalar mask used as a condition: no instruction)
__device__ __forceinline__ bool in_mask(uint64_t lanes) { return __builtin_amdgcn_inverse_ballot_w64(lanes); }
// a request of the stream: a load that only counts as global (through a generic pointer it would be waited for with
// the LDS accesses)
__device__ __forceinline__ u32x4 load_global(const Req *p) {
    return *reinterpret_cast<const __attribute__((address_space(1))) u32x4 *>(reinterpret_cast<uintptr_t>(p));
}
__device__ __forceinline__ Req as_req(const u32x4 &v) { return Req{__hiloint2double((int)v.y, (int)v.x), (int32_t)v.z, __uint_as_float(v.w)}; }
// Marks the places where the lanes' LDS accesses depend on one another: the compiler keeps them on their side (a
// wavefront's LDS accesses are carried out in order; no instruction).
__device__ __forceinline__ void wave_order() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}
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
template <typename T>
__device__ __forceinline__ T lds_get(uint32_t addr) {
    return *reinterpret_cast<const __attribute__((address_space(3))) T *>(addr);
}
template <typename T>
__device__ __forceinline__ void lds_put(uint32_t addr, T v) {
    *reinterpret_cast<__attribute__((address_space(3))) T *>(addr) = v;
}
// waits for a request on its way here, not inside the loops that follow
__device__ __forceinline__ void arrived(u32x4 &r) { asm volatile("" : "+v"(r)); }
// keeps the compiler from merging what made v with what uses it
__device__ __forceinline__ void pin(uint32_t &v) { asm volatile("" : "+v"(v)); }
// LDS atomics whose result nobody waits for
__device__ __forceinline__ void lds_or_u32(uint32_t addr, uint32_t v) { asm volatile("ds_or_b32 %0, %1" : : "v"(addr), "v"(v) : "memory"); }
__device__ __forceinline__ void lds_or_u64(uint32_t addr, uint64_t v) { asm volatile("ds_or_b64 %0, %1" : : "v"(addr), "v"(v) : "memory"); }
__device__ __forceinline__ void lds_add_u32(uint32_t addr, uint32_t v) { asm volatile("ds_add_u32 %0, %1" : : "v"(addr), "v"(v) : "memory"); }
__device__ __forceinline__ void lds_add_u64(uint32_t addr, uint64_t v) { asm volatile("ds_add_u64 %0, %1" : : "v"(addr), "v"(v) : "memory"); }
__device__ __forceinline__ uint32_t lds_fetch_add_u32(uint32_t addr, uint32_t v) {
    return __hip_atomic_fetch_add(reinterpret_cast<__attribute__((address_space(3))) uint32_t *>(addr), v, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_WAVEFRONT);
}
template <int W>
__device__ __forceinline__ int shfl_up(int v, int d) { return __shfl_up(v, (unsigned)d, W); }
template <int W>
__device__ __forceinline__ int shfl_last(int v) { return __shfl(v, W - 1, W); }
template <int W>
__device__ __forceinline__ int shfl_xor(int v, int d) { return __shfl_xor(v, d, W); }
__device__ __forceinline__ int lane_value(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ double lane_value(double v, int l) { return __hiloint2double(lane_value(__double2hiint(v), l), lane_value(__double2loint(v), l)); }

// S + x of lane 0 of the W lanes, + x of lane 1, ...: one addition after the other, as the serial loop adds.  In and
// out S is the same in all W lanes.  v_fmac_f64 with a DPP operand that a lane of the row broadcasts computes
// fma(x_k, 1, S) = S + x_k, one instruction an addition (rows are 16 lanes; 64-bit DPP knows this pattern only), for
// all placements of the wavefront at once; rows of one placement follow one another.  Lanes outside `lanes` hold zero.  A DPP operand needs two wait
// states after its register is written (s_nop).
#define MMSIM_ADD1(K, ROWS) "v_fmac_f64_dpp %0, %1, %2 row_newbcast:" #K " row_mask:" ROWS " bank_mask:0xf\n"
#define MMSIM_ADD16(ROWS)                                                                                      \
    MMSIM_ADD1(0, ROWS) MMSIM_ADD1(1, ROWS) MMSIM_ADD1(2, ROWS) MMSIM_ADD1(3, ROWS) MMSIM_ADD1(4, ROWS)          \
    MMSIM_ADD1(5, ROWS) MMSIM_ADD1(6, ROWS) MMSIM_ADD1(7, ROWS) MMSIM_ADD1(8, ROWS) MMSIM_ADD1(9, ROWS)          \
    MMSIM_ADD1(10, ROWS) MMSIM_ADD1(11, ROWS) MMSIM_ADD1(12, ROWS) MMSIM_ADD1(13, ROWS) MMSIM_ADD1(14, ROWS)     \
    MMSIM_ADD1(15, ROWS)
#define MMSIM_ADD2(K, K2)                                                            \
    "v_fmac_f64_dpp %0, %2, %3 row_newbcast:" #K " row_mask:0xf bank_mask:0xf\n"     \
    "v_fmac_f64_dpp %1, %2, %3 row_newbcast:" #K2 " row_mask:0xf bank_mask:0xf\n"
#define MMSIM_ADD_ROWS(ROWS) \
    asm("s_nop 1\n" MMSIM_ADD16(ROWS) "s_nop 1" : "+v"(s) : "v"(x), "v"(one))
// what lane 15 of a row holds, into all lanes of the next row (rows named by ROWS)
template <int ROWS>
__device__ __forceinline__ double row_carry(double s) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(s), __double2loint(s), 0x142 /* row_bcast:15 */, ROWS, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(s), __double2hiint(s), 0x142, ROWS, 0xF, false);
    return __hiloint2double(hi, lo);
}
template <int W>
__device__ __forceinline__ double ordered_sum(double s, double x, uint64_t lanes) {
    const double one = 1.0;
    if constexpr (W == 64) {
        if (lanes & 0xFFFFull) MMSIM_ADD_ROWS("0x1");
        s = row_carry<0x2>(s);
        if (lanes & 0xFFFF0000ull) MMSIM_ADD_ROWS("0x2");
        s = row_carry<0x4>(s);
        if (lanes & 0xFFFF00000000ull) MMSIM_ADD_ROWS("0x4");
        s = row_carry<0x8>(s);
        if (lanes & 0xFFFF000000000000ull) MMSIM_ADD_ROWS("0x8");
        return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(s), 63), __builtin_amdgcn_readlane(__double2loint(s), 63));
    } else if constexpr (W == 32) {
        MMSIM_ADD_ROWS("0x5");
        s = row_carry<0xA>(s);
        MMSIM_ADD_ROWS("0xa");
        return __hiloint2double(__shfl(__double2hiint(s), 31, 32), __shfl(__double2loint(s), 31, 32));
    } else if constexpr (W == 16) {
        MMSIM_ADD_ROWS("0xf");
        return s;
    } else {  // two placements to a row: lanes 0-7 are the first one's, lanes 8-15 the second one's
        double s2 = s;
        asm("s_nop 1\n" MMSIM_ADD2(0, 8) MMSIM_ADD2(1, 9) MMSIM_ADD2(2, 10) MMSIM_ADD2(3, 11) MMSIM_ADD2(4, 12) MMSIM_ADD2(5, 13)
                MMSIM_ADD2(6, 14) MMSIM_ADD2(7, 15) "s_nop 1"
            : "+v"(s), "+v"(s2)
            : "v"(x), "v"(one));
        return (lane_id() & 8) ? s2 : s;
    }
}
#undef MMSIM_ADD_ROWS
#undef MMSIM_ADD2
#undef MMSIM_ADD16
#undef MMSIM_ADD1

// x of this lane + x of all others, in lane 63
template <int CTRL, int ROWS>
__device__ __forceinline__ double plus_moved(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xF, false);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double sum_of_lanes(double v) {
    v = plus_moved<0x111 /* row_shr:1 */, 0xF>(v);
    v = plus_moved<0x112, 0xF>(v);
    v = plus_moved<0x114, 0xF>(v);
    v = plus_moved<0x118, 0xF>(v);
    v = plus_moved<0x142 /* row_bcast:15 */, 0xA>(v);
    v = plus_moved<0x143 /* row_bcast:31 */, 0xC>(v);
    return __hiloint2double(lane_value(__double2hiint(v), 63), lane_value(__double2loint(v), 63));
}

// The sum S of the accepted requests' latencies, added up in the order of their arrival: what S + x1 + x2 + ... gives with a
// rounding behind every addition, without the chain of additions.  While S stays in [2^k, 2^(k+1)) it is a multiple of
// u = 2^(k-52), and an addition adds x rounded to a multiple of u, r(x), whatever S is: unless x is half-way between two of them, where
// S/u must come out even.  (That is common: times are multiples of 2^-43 or so.)  Whether S/u is odd before a request is how many odd
// r(x) there were since the last half-way one, behind which it is even.  So the r(x) of 64 requests are found side by side, and
// several blocks are added exactly, in any order.  Blocks that take S to 2^(k+1) or beyond (then their sum does as well, however it is
// rounded), or have a negative x, go through ordered_sum one by one: S doubles a dozen times in a stream.
struct LatencySum {
    double s, base, half;  // base: 2^k, half: u / 2
    int odd;               // whether s / u is odd, or s and what was taken since
    double first_tie = 0.0;
    __device__ __forceinline__ explicit LatencySum(double v) { set(v); }
    __device__ __forceinline__ void set(double v) {
        s = v;
        odd = __double2loint(v) & 1;
        const int hi = __double2hiint(v) & 0x7FF00000;
        base = __hiloint2double(hi, 0);
        half = __hiloint2double(hi > (53 << 20) ? hi - (53 << 20) : 0, 0);
    }
    // What the lanes add for their x.
    __device__ __forceinline__ double take(double x) {
        const double up = base + x, r = up - base, off = x - r;
        const bool half_way = __builtin_fabs(off) == half;
        const uint64_t ties = ballot(half_way), odds = ballot((__double2loint(up) & 1) != 0);  // (half-way ones came out even)
        // Whether S / u is odd before a half-way request: as many odd ones came since the half-way one before it, or since the
        // beginning and S / u was odd then.  since: whether the number of odd ones up to that one was odd, carried through the
        // requests between them by an addition.
        const uint64_t odd_below = ballot((__builtin_amdgcn_mbcnt_hi((uint32_t)(odds >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)odds, 0u)) & 1u) != 0u);
        const uint64_t at_ties = odd_below & ties;
        uint64_t since;
        const bool out1 = __builtin_add_overflow(~ties, at_ties << 1, &since), out2 = __builtin_add_overflow(since, (uint64_t)odd, &since);
        const uint64_t others = (odd_below ^ since) & ties;
        odd = (__builtin_popcountll(odds) ^ (out1 || out2 ? 1 : 0) ^ (int)(at_ties >> 63)) & 1;
        if (first_tie == 0.0 && ties != 0ull) {
            const int l = __builtin_ctzll(ties);
            first_tie = 2.0 * __hiloint2double(lane_value(__double2hiint(off), l), lane_value(__double2loint(off), l));
            if ((others >> l & 1ull) != 0ull) first_tie = -first_tie;
        }
        const bool other = in_mask(others);
        return other ? x + off : r;
    }
    // What N blocks' latencies add to a sum in [2^k, 2^(k+1)), if it is even, and how much more if it is odd: only the first
    // half-way one comes out differently then.  negative: they must be added one by one.
    template <int N>
    __device__ __forceinline__ void look(const double (&x)[N], double *added, double *more_if_odd, bool *negative) const {
        LatencySum even = *this;
        even.odd = 0;
        even.first_tie = 0.0;
        double lanes = 0.0;
        bool neg = false;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            lanes += even.take(x[i]);
            neg = neg || x[i] < 0.0;
        }
        *added = sum_of_lanes(lanes);
        *more_if_odd = even.first_tie;
        *negative = ballot(neg) != 0ull;
    }
    // Adds what look() found, unless the sum leaves [2^k, 2^(k+1)).
    __device__ __forceinline__ bool add(double added, double more_if_odd, bool negative) {
        const double sum = added + (odd != 0 ? more_if_odd : 0.0);
        if (negative || !(sum <= 2.0 * base - s)) return false;
        set(s + sum);
        return true;
    }
    __device__ __forceinline__ void add_block(double x) {
        const double one[1] = {x};
        const uint64_t some = ballot(x != 0.0);
        double added, more;
        bool negative;
        look(one, &added, &more, &negative);
        if (some != 0ull && !add(added, more, negative)) set(ordered_sum<kWave>(s, x, some));
    }
};

struct Entry {  // a replica, as rep and ext hold it
    uint32_t d;
    float l;
};
struct Entry4 {
    Entry e[4];
};
__device__ __forceinline__ float as_float(uint32_t v) { return __uint_as_float(v); }
__device__ __forceinline__ Entry4 load_entries(uint32_t addr) {  // two 16-byte reads
    const u32x4 a = lds_get<u32x4>(addr), b = lds_get<u32x4>(addr + 16u);
    return Entry4{{{a.x, as_float(a.y)}, {a.z, as_float(a.w)}, {b.x, as_float(b.y)}, {b.z, as_float(b.w)}}};
}
__device__ __forceinline__ int max2(int x, int y) { return x > y ? x : y; }
constexpr uint32_t kAddrMask8 = 0x7FFFu;
constexpr uint32_t kEntryMore = 1u << 30;
__device__ __forceinline__ uint32_t entry_addr(uint32_t d) { return (d & kAddrMask8) << 3; }
__device__ __forceinline__ int entry_stages_m1(uint32_t d) { return (int)(d >> 15) & 0x1F; }
__device__ __forceinline__ uint32_t entry_lat(uint32_t d) { return (d >> 20) & 0x3FFu; }
__device__ __forceinline__ bool entry_none(uint32_t d) { return (int32_t)d < 0; }

template <int I>
struct Int {
    static constexpr int value = I;
};
// Where a run's latencies are (finish times, if wanted), by place in the stream.  Run 0 adds up its own and writes its outputs.  One
// that is taken up again puts them where the run of the span that it is in has its own: if anybody takes over from that one, then behind
// where the two meet.
typedef const __attribute__((address_space(4))) WindowArgs ColdArgs;
__device__ __forceinline__ double *values_of(ColdArgs *q, int sim, int r) {
    return q->run_vals + ((int64_t)sim * (q->spans - 1) + (r - 1)) * q->run_cap - (int64_t)r * q->span_blocks * kWave;
}

// Wavefronts of a SIMD that the registers have to leave room for, with simulations cut into runs.
constexpr int least_waves(int smax, bool outputs, int ext) {
    return ext > 1 || (smax == 32 && (outputs || ext > 0)) ? 2 : outputs || smax == 32 || (smax == 16 && ext > 0) ? 3 : 4;
}

// W: requests (lanes) of one placement.  SMAX: most stages of a group (bucket).  OUTPUTS: anything beyond the scores
// (a.flags says what).  EXT: 1, some model has more than four replicas; 2, and up to sixteen are kept in registers, not eight.  POW2: every group has 1, 2, 4, ... stages.
// UNIFORM: one latency per (model, configuration).
// SPANS: a simulation is cut into a.spans runs (W == 64).
template <int W, int SMAX, bool OUTPUTS, int EXT, bool POW2, bool UNIFORM, bool SPANS>
__global__ __launch_bounds__(kMaxWindowWaves *kWave, SPANS ? least_waves(SMAX, OUTPUTS, EXT) : 1) void sim_window_kernel(const WindowArgs a) {
    constexpr int P = kWave / W;
    const int lane = lane_id(), j = lane % W, sub = W == 64 ? 0 : lane / W;
    const int wv = SMAX >= 16 || SPANS ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : (int)(threadIdx.x >> 6);
    // latency table for the per-stage latencies of the walk (general tables only), shared by the workgroup
    if (!UNIFORM && a.lat_lds_bytes > 0) {
        for (int i = (int)threadIdx.x; i < a.M * a.lat_row; i += (int)blockDim.x) lds_put<float>((uint32_t)i * 4u, a.lat[i]);
        __syncthreads();
    }
    int64_t unit = (int64_t)blockIdx.x * (blockDim.x >> 6) + wv;  // (seed, tile of P placements)
    int own = 0;                                                  // the run
    if constexpr (SPANS) {
        // First runs first, each workgroup's on another SIMD than those of the workgroups that share its CU.
        const int waves = (int)(blockDim.x >> 6), sims = a.tiles * a.out_seeds;
        const int at = __builtin_amdgcn_readfirstlane((wv + (int)(blockIdx.x >> 8)) % waves) * (int)gridDim.x + (int)blockIdx.x;
        own = __builtin_amdgcn_readfirstlane(at / sims);
        if (own >= a.spans) return;
        unit = at - own * sims;
    }
    if (unit >= (int64_t)a.tiles * a.out_seeds) return;
    const int seed_row = SPANS ? __builtin_amdgcn_readfirstlane((int)unit / a.tiles) : (int)(unit / a.tiles);
    const int b = SPANS ? (int)unit - seed_row * a.tiles : (int)(unit % a.tiles) * P + sub;
    const bool mine = b < a.B;
    // (with a stream of its own for every placement there is one placement to a wavefront: the host sees to that)
    const int seed = a.stream_of ? lane_value(a.stream_of[mine ? b : 0], 0) : seed_row;
    const Req *__restrict__ reqs = a.stream_ptr[seed];
    const uint32_t R = (uint32_t)a.stream_len[seed];

    // LDS: [latency table][per wavefront: two chunks of 64 requests (W < 64)][per placement: its tables and state]
    const uint32_t ring = (uint32_t)a.lat_lds_bytes + (uint32_t)wv * (uint32_t)window_ring_bytes(W);
    const uint32_t base = (uint32_t)a.lat_lds_bytes + (blockDim.x >> 6) * (uint32_t)window_ring_bytes(W) +
                          (uint32_t)(wv * P + sub) * (uint32_t)a.place_bytes;
    const uint32_t clk = base, rep = base + a.o_rep, ext = base + a.o_ext, xi = base + a.o_xi;
    const uint32_t bits = base + a.o_bits, gd = base + a.o_gd, mcnt = base + a.o_mcnt;
    const uint32_t gm_rel = (uint32_t)(a.nslots + SMAX) * 8u, cnt_rel = gm_rel * 2u;  // from a clock to its mask and its counter
    const uint32_t spare = clk + (uint32_t)a.nslots * 8u;  // SMAX slots for writes that do not count
    const int M = a.M, GW = a.group_words, Gmax = a.Gmax;

    // ---- the placement's tables
    for (int k = j; k < (a.nslots + SMAX) * (OUTPUTS ? 3 : 2); k += W) lds_put<uint64_t>(clk + (uint32_t)k * 8u, 0ull);
    for (int k = j; k < M * GW; k += W) lds_put<uint32_t>(bits + (uint32_t)k * 4u, 0u);
    if (OUTPUTS)
        for (int k = j; k < M; k += W) lds_put<uint32_t>(mcnt + (uint32_t)k * 4u, 0u);
    const int ng = mine ? (int)a.num_groups[b] : 0;
    {
        const uint8_t *cfg = a.group_cfg + (size_t)(mine ? b : 0) * Gmax;
        int slot = 0;
        for (int g0 = 0; g0 < Gmax; g0 += W) {
            const int g = g0 + j;
            int pp = 0, c = 0;
            if (g < ng) {
                c = cfg[g];
                pp = a.cfg_pp[c];
            }
            int upto = pp;
            for (int d = 1; d < W; d *= 2) {
                const int v = shfl_up<W>(upto, d);
                if (j >= d) upto += v;
            }
            if (g < ng) {
                const uint32_t last = (uint32_t)(slot + upto - 1);
                const uint32_t lat_last = (uint32_t)a.lat_off[c] + (UNIFORM ? 0u : (uint32_t)(pp - 1));
                lds_put<uint32_t>(gd + (uint32_t)g * 4u, (clk + last * 8u) >> 3 | (uint32_t)(pp - 1) << 15 | lat_last << 20);
            }
            slot += shfl_last<W>(upto);
        }
    }
    uint32_t ext_used = base + a.o_gd + (uint32_t)Gmax * 4u;  // a word behind gd: chunks of ext given out
    if (j == 0) lds_put<uint32_t>(ext_used, 0u);
    wave_order();
    if (mine)
        for (uint32_t e = a.entry_off[b] + (uint32_t)j; e < a.entry_off[b + 1]; e += W) {
            const uint32_t v = a.entries[e], m = v & 0xFFFFu, g = v >> 16;
            lds_or_u32(bits + (m * (uint32_t)GW + (g >> 5)) * 4u, 1u << (g & 31u));
        }
    wave_order();
    for (int m = j; m < M; m += W) {
        const uint32_t mb = bits + (uint32_t)(m * GW) * 4u;
        int n = 0;
        for (int w = 0; w < GW; ++w) n += __popc(lds_get<uint32_t>(mb + (uint32_t)w * 4u));
        uint32_t chunk0 = 0;
        if constexpr (EXT > 0) {
            const uint32_t chunks = n > 4 ? (uint32_t)(n - 1) / 4u : 0u;
            if (chunks > 0) chunk0 = lds_fetch_add_u32(ext_used, chunks);
            lds_put<uint32_t>(xi + (uint32_t)m * 4u, chunk0 | chunks << 16);
        }
        Entry first{(clk >> 3) | kEmpty, __builtin_inff()};
        int k = 0;
        auto put = [&](const Entry &e) {
            const uint32_t at = k < 4 ? rep + (uint32_t)(m * 4 + k) * 8u : ext + (chunk0 * 4u + (uint32_t)(k - 4)) * 8u;
            lds_put<uint32_t>(at, (k == 3 && n > 4) || (k == 2 && n > 8) || (k == 1 && n > 16) ? e.d | kEntryMore : e.d);
            lds_put<float>(at + 4u, e.l);
            ++k;
        };
        for (int w = 0; w < GW; ++w)
            for (uint32_t v = lds_get<uint32_t>(mb + (uint32_t)w * 4u); v != 0u; v &= v - 1u) {
                const uint32_t d = lds_get<uint32_t>(gd + (uint32_t)(w * 32 + __ffs((int)v) - 1) * 4u);
                const Entry e{d, a.lat[(size_t)m * a.lat_row + entry_lat(d)]};
                if (k == 0) first = Entry{d | kEmpty, e.l};
                put(e);
            }
        while (k < 4 || (k & 3) != 0) put(first);
    }
    wave_order();

    const double overhead = a.fixed_overhead;
    const uint64_t my_bit = 1ull << lane;
    // bits of this placement's requests before this one
    const uint64_t before = (my_bit - 1ull) & ~((1ull << (sub * W)) - 1ull);
    int32_t n_good = 0;
    double lat_sum = 0.0;
    const size_t row = (size_t)seed_row * a.B + (size_t)(mine ? b : 0);  // where the results go
    double *fin_out = a.finish + row * (size_t)a.Rmax;
    uint8_t *good_out = a.good + row * (size_t)a.Rmax;
    const bool want_req = OUTPUTS && (a.flags & MMSIM_WANT_PER_REQUEST) != 0;

    auto load_req = [&](uint32_t i) -> u32x4 {
        u32x4 r{0u, 0u, ~0u, 0u};
        if (i < R) r = load_global(reqs + i);
        return r;
    };
    auto load_rep = [&](int m) -> Entry4 { return load_entries(rep + (uint32_t)(m < 0 ? 0 : m) * 32u); };
    // Requests come 64 at a time, one to a lane.  W == 64: that is a block, fetched two blocks ahead.  Otherwise the
    // chunks pass through LDS, which deals them to the placements' lanes; the chunk after the one a block is of is in
    // LDS as well, and the one after that on its way.
    u32x4 far, nxt;
    Req cur;
    auto store_ring = [&](uint32_t chunk) { lds_put<u32x4>(ring + (chunk & 1u) * 1024u + (uint32_t)lane * 16u, far); };
    auto load_ring = [&](uint32_t i) -> u32x4 { return lds_get<u32x4>(ring + (i & 127u) * 16u); };
    Entry4 q;
    // What a block is like: requests that can be served at all, that list several groups, more than two, more than
    // four; how deep their groups are.  Worked out a block ahead (a scalar that depends on vector compares is slow to come).
    uint64_t pend, multis, fours, mores, eights, sixteens, deep_a, deep_b;
    auto look = [&]() {
        pend = ballot(cur.m >= 0 && !entry_none(q.e[0].d));  // (past the end of the stream: m is -1)
        multis = ballot(!entry_none(q.e[1].d)) & pend;
        fours = ballot(!entry_none(q.e[2].d)) & pend;
        if constexpr (EXT > 0) {
            mores = ballot((q.e[3].d & kEntryMore) != 0u) & pend;
            eights = ballot((q.e[2].d & kEntryMore) != 0u) & pend;
            if constexpr (EXT > 1) sixteens = ballot((q.e[1].d & kEntryMore) != 0u) & pend;
        }
        if constexpr (SMAX > 1) {
            const int deep = max2(max2(entry_stages_m1(q.e[0].d), entry_stages_m1(q.e[1].d)),
                                  max2(entry_stages_m1(q.e[2].d), entry_stages_m1(q.e[3].d)));
            deep_a = ballot(deep >= (SMAX == 4 ? 2 : SMAX == 16 ? 8 : 16)) & pend;
            if constexpr (SMAX == 16) deep_b = ballot(deep >= 4) & pend;
            if constexpr (EXT > 0) {  // (the groups behind the fourth are not looked at: as deep as any of the batch)
                if (a.smax > (SMAX == 4 ? 2 : SMAX == 16 ? 8 : 16)) deep_a |= mores;
                if (SMAX == 16 && a.smax > 4) deep_b |= mores;
            }
        }
    };
    auto start_at = [&](uint32_t first) {  // (a multiple of 64)
        far = load_req(first + (uint32_t)lane);
        if constexpr (W == 64) {
            nxt = load_req(first + 64u + (uint32_t)lane);
            arrived(far);  // (here, or the first step of every block waits for what is on its way then)
            arrived(nxt);
            cur = as_req(far);
        } else {
            store_ring(0u);
            far = load_req(64u + (uint32_t)lane);
            store_ring(1u);
            far = load_req(128u + (uint32_t)lane);
            wave_order();
            cur = as_req(load_ring((uint32_t)j));
            nxt = load_ring((uint32_t)(W + j));
        }
        q = load_rep(cur.m);
        look();
    };

    // What a step needs of an entry word, ready for it: the address of the group's first clock and, from bit 18 on, stages - 1;
    // of a single stage the address, of several latencies the word itself.
    auto walk_word = [](uint32_t d) -> uint32_t {
        if constexpr (SMAX > 1 && !UNIFORM) return d;
        return SMAX == 1 ? entry_addr(d) : (entry_addr(d) - (uint32_t)entry_stages_m1(d) * 8u) | (uint32_t)entry_stages_m1(d) << 18;
    };
    auto first_clock = [](uint32_t w) -> uint32_t {
        if constexpr (SMAX > 1 && !UNIFORM) return entry_addr(w) - (uint32_t)entry_stages_m1(w) * 8u;
        return SMAX == 1 ? w : w & 0x3FFFFu;
    };
    auto stages_m1 = [](uint32_t w) -> int { return SMAX == 1 ? 0 : UNIFORM ? (int)(w >> 18) : entry_stages_m1(w); };
    // ---- SPANS: this wavefront's run, and the simulation's others
    const int sim = (int)unit;
    Runs runs;
    if constexpr (SPANS) {
        runs.start(cold_args<WindowArgs>(), own);
    }
    auto marked = [&](int r, int i) {
        ColdArgs *q = cold_args<WindowArgs>();
        return q->mark_state + (((size_t)sim * q->spans + r) * q->marks + i) * (size_t)q->state_words;
    };
    auto ended = [&](int r) {
        ColdArgs *q = cold_args<WindowArgs>();
        return q->end_state + ((size_t)sim * q->spans + r) * (size_t)(q->state_words + kEndWords);
    };
    // state: accepted requests, clocks; counts of the slots and of the models
    auto for_state = [&](auto f) {
        const int nslots = cold_args<WindowArgs>()->nslots;
        for (int k = j; k < nslots; k += W) f(1 + k, clk + (uint32_t)k * 8u, false);
        if constexpr (OUTPUTS) {
            for (int k = j; k < nslots; k += W) f(1 + nslots + k, clk + (uint32_t)k * 8u + cnt_rel, false);
            for (int m = j; m < M; m += W) f(1 + 2 * nslots + m, mcnt + (uint32_t)m * 4u, true);
        }
    };
    auto get_word = [&](uint32_t at, bool half) -> uint64_t { return half ? (uint64_t)lds_get<uint32_t>(at) : lds_get<uint64_t>(at); };
    // Something happens before block `at`: a mark of this run, one of a later run or the block ahead of it, the end of the run (true).
    auto published = [&](int r) {
        ColdArgs *q = cold_args<WindowArgs>();
        return q->span_sync + (size_t)sim * (q->spans + kSyncWords) + r;
    };
    uint64_t peeked = 0;
    auto event = [&](uint32_t at) -> bool {
        ColdArgs *q = cold_args<WindowArgs>();
        if (at >= runs.limit(q)) return true;
        uint64_t *st = marked(runs.in, runs.mark);
        if (runs.in == runs.own) {
            if (lane == 0) tell(st, (uint64_t)(uint32_t)n_good);
            for_state([&](int w, uint32_t addr, bool half) { tell(st + w, get_word(addr, half)); });
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (stores of device scope have been carried out then)
            if (lane == 0) tell(published(runs.in), (uint32_t)runs.mark + 1u);
        } else if (!runs.looked) {
            if (__builtin_amdgcn_readfirstlane(told(published(runs.in))) > (uint32_t)runs.mark) {
                asm volatile("" ::: "memory");
                peeked = told(st + 1 + (lane < q->nslots ? lane : 0));
                runs.looked = true;
                runs.next = at + 1u;
                return false;
            }
        } else {
            // Equal clocks, or alike: what differs lies before the next arrival in both (limit; never, if a.alike is 0), so no walk sees it,
            // and the groups' last clocks are in the same order, so every choice is the same.  That lasts: a clock that is written comes out the same in
            // both, and not before that arrival.
            const double limit = q->alike != 0 ? lane_value(cur.t, 0) : -1.0;
            bool differ = false, same = true;
            auto compare = [&](uint64_t theirs, uint32_t addr) {
                const uint64_t mine = lds_get<uint64_t>(addr);
                const bool other = theirs != mine;
                differ = differ || other;
                same = same && (!other || (__longlong_as_double((long long)theirs) < limit && __longlong_as_double((long long)mine) < limit));
            };
            if (lane < q->nslots) compare(peeked, clk + (uint32_t)lane * 8u);
            if (ballot(!same) == 0ull) {
                for (int k = j + W; k < q->nslots; k += W) compare(told(st + 1 + k), clk + (uint32_t)k * 8u);
                if (ballot(differ) != 0ull && ballot(!same) == 0ull) {
                    uint32_t slot = 0;  // lane g: the last one of group g (of others the first group's)
                    if (q->Gmax > 0) slot = (entry_addr(lds_get<uint32_t>(gd + (uint32_t)(lane < ng ? lane : 0) * 4u)) - clk) >> 3;
                    const double mine = lds_get<double>(clk + slot * 8u), theirs = __longlong_as_double((long long)told(st + 1 + slot));
                    for (int g = 0; g < ng; ++g) same = same && (mine < lane_value(mine, g)) == (theirs < lane_value(theirs, g));
                }
                runs.met = ballot(!same) == 0ull;
                if (runs.met) return true;
            }
        }
        runs.go_on(q, at);
        return false;
    };
    auto q_pieces = [&](int of) { return cold_args<WindowArgs>()->pieces + (size_t)of * kPieceWords; };
    auto piece = [&](uint32_t at, uint32_t first, uint32_t end, int src) {
        uint32_t *w = q_pieces(sim) + at * 4u;
        w[0] = first;
        w[1] = end;
        w[2] = (uint32_t)src;
    };
    uint32_t from = SPANS ? (uint32_t)own * (uint32_t)a.span_blocks * 64u : 0u, blk = from;
    double *run_vals = SPANS ? values_of(cold_args<WindowArgs>(), sim, own) : nullptr;  // by place in the stream
    uint32_t num_pieces = 0;
    bool last = false;  // this wavefront puts the simulation together
    uint32_t met_again = 0;
    for (;;) {
        if (from < R) start_at(from);
        for (blk = from; blk < R; blk += W) {
            if constexpr (SPANS)
                if (blk / 64u == runs.next && event(blk / 64u)) break;
            const int m = cur.m;
            const double arr = cur.t, slo = (double)cur.slo;
            uint32_t ca[4], word[4];  // what the tournament carries of an entry word
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                ca[k] = entry_addr(q.e[k].d);
                word[k] = walk_word(q.e[k].d);
            }
            Entry4 nrep;
            u32x4 nn;
            double best = 0.0, t = 0.0, latency = 0.0;
            uint32_t chosen = SMAX > 1 && !UNIFORM ? clk >> 3 : clk;  // the chosen group's walk word
            // The block, for requests that list at most NC groups (2, 4, 8, 16, or 0: any number).
            auto block = [&](auto NCv) {
                constexpr int NC = decltype(NCv)::value, N4 = NC == 2 ? 2 : 4;
                // Further ones kept in registers.  (Not beside the fetched ones with 16 stages and counts: 133 registers instead of 126, three
                // wavefronts to a SIMD instead of four.)
                constexpr int NX = NC > 4 ? NC - 4 : NC == 0 ? (EXT > 1 ? 12 : SMAX < 16 ? 4 : 0) : 0;
                constexpr bool MORE = NC != 2 && NC != 4, ANY = NC == 0;                // ANY: and others are fetched in every step
                double c[N4];
#pragma unroll
                for (int k = 0; k < N4; ++k) c[k] = lds_get<double>(ca[k]);
                // ---- the masks of the block's requests.  (Copies of the first replica set its bit again: harmless.)
                uint64_t gm[N4];
                uint32_t x0 = 0, xn = 0;  // chunks of further replicas
                if constexpr (MORE) {
                    const uint32_t v = lds_get<uint32_t>(xi + (uint32_t)(m < 0 ? 0 : m) * 4u);
                    x0 = ext + (v & 0xFFFFu) * 32u;
                    xn = in_mask(pend) ? v >> 16 : 0u;
                }
                // the further ones in registers, like the first four (of a request without: copies of its first, which never beat it)
                constexpr int NA = NX > 0 ? NX : 1;
                uint32_t xa[NA], xword[NA];
                float xl[NA];
                double cx[NA];
#pragma unroll
                for (int x = 0; x < NX / 4; ++x) {
                    Entry4 more;
                    if (xn > (uint32_t)x) more = load_entries(x0 + (uint32_t)x * 32u);
                    else more.e[0] = more.e[1] = more.e[2] = more.e[3] = q.e[0];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        xa[4 * x + k] = entry_addr(more.e[k].d);
                        xword[4 * x + k] = walk_word(more.e[k].d);
                        xl[4 * x + k] = more.e[k].l;
                        cx[4 * x + k] = lds_get<double>(xa[4 * x + k]);
                    }
                }
                uint32_t ga[N4];
#pragma unroll
                for (int k = 0; k < N4; ++k) {
                    ga[k] = ca[k] + gm_rel;
                    pin(ga[k]);
                }
                if (in_mask(pend)) {
#pragma unroll
                    for (int k = 0; k < N4; ++k) lds_or_u64(ga[k], my_bit);
                    if constexpr (NX > 0) {
#pragma unroll
                        for (int x = 0; x < NX / 4; ++x)
                            if (xn > (uint32_t)x) {
#pragma unroll
                                for (int k = 0; k < 4; ++k) lds_or_u64(xa[4 * x + k] + gm_rel, my_bit);
                            }
                    }
                    if constexpr (ANY)
                        for (uint32_t x = NX / 4; x < xn; ++x) {
                            const Entry4 e = load_entries(x0 + x * 32u);
#pragma unroll
                            for (int k = 0; k < 4; ++k) lds_or_u64(entry_addr(e.e[k].d) + gm_rel, my_bit);
                        }
                }
                wave_order();
#pragma unroll
                for (int k = 0; k < N4; ++k) gm[k] = lds_get<uint64_t>(ga[k]) & before;
                uint64_t gm_ext = 0;  // requests before this one that share any of the groups: holds for every further replica
                if constexpr (MORE) {
                    if constexpr (NX > 0) {
#pragma unroll
                        for (int k = 0; k < NX; ++k) gm_ext |= lds_get<uint64_t>(xa[k] + gm_rel);
                    }
                    if constexpr (ANY) {
                        for (uint32_t x = NX / 4; x < xn; ++x) {
                            const Entry4 e = load_entries(x0 + x * 32u);
#pragma unroll
                            for (int k = 0; k < 4; ++k) gm_ext |= lds_get<uint64_t>(entry_addr(e.e[k].d) + gm_rel);
                        }
                    }
                    gm_ext = (gm_ext & before) | gm[0] | gm[1] | gm[2] | gm[3];
                }
                wave_order();
#pragma unroll
                for (int k = 0; k < N4; ++k) lds_put<uint64_t>(ga[k], 0);  // for the next block
                if constexpr (NX > 0) {
#pragma unroll
                    for (int k = 0; k < NX; ++k) lds_put<uint64_t>(xa[k] + gm_rel, 0);
                }
                if constexpr (ANY)
                    for (uint32_t x = NX / 4; x < xn; ++x) {
                        const Entry4 e = load_entries(x0 + x * 32u);
#pragma unroll
                        for (int k = 0; k < 4; ++k) lds_put<uint64_t>(entry_addr(e.e[k].d) + gm_rel, 0);
                    }
                // ---- fetched ahead: the requests of the block after the next, the replicas of the next
                if constexpr (W == 64) {
                    nn = load_req(blk + 128u + (uint32_t)j);
                } else {
                    if ((blk & 63u) == 0u && blk != 0u) {  // a chunk begins: the one after it takes the place of the one before
                        store_ring(blk / 64u + 1u);
                        far = load_req(blk + 128u + (uint32_t)lane);
                        wave_order();
                    }
                    nn = load_ring(blk + 2u * W + (uint32_t)j);
                }
                wave_order();
                // ---- the steps.  Each lane stays in the loop until its verdict is final and leaves with what it found.
                // D: most stages of a group.
                auto steps = [&](auto Dv) {
                    constexpr int D = decltype(Dv)::value;
                    // The stages behind the first NEAR are read, walked and written by the lanes that chose a group with
                    // so many, in a branch that most steps skip.  A wavefront on its own (W == 64) takes up to eight
                    // without a branch, as the stages are a shorter chain than the branch; wavefronts that share a
                    // SIMD (W < 64) gain from four stages on, as they share its issue slots.  20000 requests, against
                    // all stages in every lane: 4096 placements of groups up to 16 deep 6.44 -> 5.11 ms, up to 8 deep
                    // 5.02 -> 4.81 ms; 1025 placements, W == 64, up to 16 deep 3.60 -> 3.20 ms (2.88 -> 2.98 ms up to 8
                    // deep, where only the registers of the unused deep path differ).
                    constexpr int NEAR = W == 64 ? 8 : 4;
                    struct Cand {
                        double c;
                        uint32_t d;
                        float l;
                        uint64_t g;
                    };
                    auto first_min = [](const Cand &x, const Cand &y) {
                        const bool right = y.c < x.c;
                        return Cand{vmin(x.c, y.c), right ? y.d : x.d, right ? y.l : x.l, right ? y.g : x.g};
                    };
                    bool waits;
                    do {
                        // ---- choose the replica group: strictly smallest last-stage clock, first listed wins ties (:590-598)
                        Cand win = first_min(Cand{c[0], word[0], q.e[0].l, gm[0]}, Cand{c[1], word[1], q.e[1].l, gm[1]});
                        if constexpr (NC != 2)
                            win = first_min(win, first_min(Cand{c[2], word[2], q.e[2].l, gm[2]}, Cand{c[3], word[3], q.e[3].l, gm[3]}));
                        if constexpr (NX > 0) {
#pragma unroll
                            for (int x = 0; x < NX; x += 4) {
                                Cand y[4];
#pragma unroll
                                for (int k = 0; k < 4; ++k) y[k] = Cand{cx[x + k], xword[x + k], xl[x + k], gm_ext};
                                win = first_min(win, first_min(first_min(y[0], y[1]), first_min(y[2], y[3])));
                            }
                        }
                        if constexpr (ANY)
                            for (uint32_t x = NX / 4; x < xn; ++x) {
                                const Entry4 e = load_entries(x0 + x * 32u);
                                Cand y[4];
#pragma unroll
                                for (int k = 0; k < 4; ++k) {
                                    const uint32_t at = entry_addr(e.e[k].d);
                                    y[k] = Cand{lds_get<double>(at), e.e[k].d, e.e[k].l, gm_ext};
                                }
                                Cand z = first_min(first_min(y[0], y[1]), first_min(y[2], y[3]));
                                z.d = walk_word(z.d);
                                win = first_min(win, z);
                            }
                        best = win.c;
                        chosen = win.d;
                        const double l_last = (double)win.l;
                        // ---- walk the stages and decide (:605-613).  All requests read and walk the near stages from their group's first
                        // on and take the time after their last one (what lies behind a shallower group's slots does not matter).
                        double cv[D];
                        const int sm1 = stages_m1(win.d);
                        const uint32_t gclk = first_clock(win.d);
                        if constexpr (SMAX == 1) {
                            t = vmax(arr, best) + l_last;
                            cv[0] = t;
                        } else {
                            const uint32_t lrow = (uint32_t)m * (uint32_t)a.lat_row + entry_lat(win.d) - (uint32_t)sm1;
                            float l[UNIFORM ? 1 : D];
                            auto read = [&](int k) {
                                cv[k] = lds_get<double>(gclk + (uint32_t)k * 8u);
                                if constexpr (!UNIFORM)
                                    l[k] = a.lat_lds_bytes > 0 ? lds_get<float>((lrow + (uint32_t)k) * 4u) : a.lat[lrow + (uint32_t)k];
                            };
                            auto pass = [&](int k) {
                                cv[k] = vmax(k == 0 ? arr : cv[k > 0 ? k - 1 : 0], cv[k]) + (UNIFORM ? l_last : (double)l[UNIFORM ? 0 : k]);
                                if (k == 0)
                                    t = cv[0];
                                else if (!POW2 || (k & (k + 1)) == 0)
                                    t = sm1 >= k ? cv[k] : t;
                            };
#pragma unroll
                            for (int k = 0; k < (D < 8 ? D : 8); ++k) read(k);
#pragma unroll
                            for (int k = 0; k < (D < NEAR ? D : NEAR); ++k) pass(k);
                            if constexpr (D > NEAR) {
                                if (sm1 >= NEAR) {
#pragma unroll
                                    for (int k = NEAR; k < (D < 8 ? D : 8); ++k) pass(k);
                                    if constexpr (D > 8) {
                                        if (sm1 >= 8) {
#pragma unroll
                                            for (int k = 8; k < (D < 16 ? D : 16); ++k) read(k);
#pragma unroll
                                            for (int k = 8; k < (D < 16 ? D : 16); ++k) pass(k);
                                            if constexpr (D > 16) {
                                                if (sm1 >= 16) {
#pragma unroll
                                                    for (int k = 16; k < D; ++k) read(k);
#pragma unroll
                                                    for (int k = 16; k < D; ++k) pass(k);
                                                }
                                            }
                                        }
                                    }
                                }
                            }
                        }
                        latency = (t + overhead) - arr;
                        const uint64_t accs = ballot(latency <= slo) & ballot(best < 1e100);  // a clock that is infinite is never chosen (:590-598)
                        // ---- whose verdict is final
                        const uint64_t blockers = win.g & accs;
                        waits = blockers != 0ull;
                        uint64_t waiting = ballot(waits);
                        // requests that wait, are not accepted so far and list several groups: they hold up others too
                        for (uint64_t open = waiting & multis & ~accs; __builtin_expect(open != 0ull, 0);) {
                            waits = (win.g & (accs | waiting)) != 0ull;
                            const uint64_t w2 = ballot(waits);
                            open = w2 & ~waiting & multis & ~accs;
                            waiting = w2;
                        }
                        // accepted and final: the clocks (:614-619).  Everybody writes the near stages, the others where it does
                        // not matter.
                        uint32_t to = in_mask(accs) ? gclk : spare;
                        pin(to);
                        to = waits ? spare : to;
                        pin(to);
                        auto commit = [&](int k) {
                            if (k > 0 && (!POW2 || (k & (k - 1)) == 0)) {
                                to = sm1 >= k ? to : spare;
                                pin(to);
                            }
                            lds_put<double>(to + (uint32_t)k * 8u, cv[k]);
                        };
#pragma unroll
                        for (int k = 0; k < (D < NEAR ? D : NEAR); ++k) commit(k);
                        if constexpr (D > NEAR) {
                            if (to == gclk && sm1 >= NEAR) {
#pragma unroll
                                for (int k = NEAR; k < (D < 8 ? D : 8); ++k) commit(k);
                                if constexpr (D > 8) {
                                    if (sm1 >= 8) {
#pragma unroll
                                        for (int k = 8; k < D; ++k) commit(k);
                                    }
                                }
                            }
                        }
                        wave_order();
#pragma unroll
                        for (int k = 0; k < N4; ++k) c[k] = lds_get<double>(ca[k]);
#pragma unroll
                        for (int k = 0; k < NX; ++k) cx[k] = lds_get<double>(xa[k]);
                    } while (waits);
                };
                if (in_mask(pend)) {
                    if constexpr (SMAX == 1) {
                        steps(Int<1>{});
                    } else if constexpr (SMAX == 4) {
                        if (deep_a == 0ull) steps(Int<2>{});
                        else steps(Int<4>{});
                    } else if constexpr (SMAX == 16) {
                        if (deep_a != 0ull) steps(Int<16>{});
                        else if (deep_b != 0ull) steps(Int<8>{});
                        else steps(Int<4>{});
                    } else {
                        if (deep_a == 0ull) steps(Int<16>{});
                        else steps(Int<32>{});
                    }
                }
            };
            if constexpr (EXT > 0) {
                if ((EXT > 1 ? sixteens : eights) != 0ull) block(Int<0>{});
                else if (EXT > 1 && eights != 0ull) block(Int<(EXT > 1 ? 16 : 8)>{});
                else if (mores != 0ull) block(Int<8>{});
                else if (fours != 0ull) block(Int<4>{});
                else block(Int<2>{});
            } else {
                if (fours != 0ull) block(Int<4>{});
                else block(Int<2>{});
            }
            wave_order();
            const uint64_t found = ballot(best < 1e100) & pend, accepted = ballot(latency <= slo) & found;
            const bool good = in_mask(accepted);
            const double took = good ? latency : 0.0;
            n_good += SPANS ? __popcll(accepted) : good ? 1 : 0;
            if constexpr (OUTPUTS) {
                if (in_mask(found)) lds_add_u64(first_clock(chosen) + (uint32_t)stages_m1(chosen) * 8u + cnt_rel, good ? 0x100000001ull : 1ull);  // :611, :618
                if (good) lds_add_u32(mcnt + (uint32_t)m * 4u, 1u);
            }
            if constexpr (OUTPUTS)
                if (want_req && mine && blk + (uint32_t)j < R && (!SPANS || runs.own == 0)) {
                    fin_out[blk + (uint32_t)j] = good ? t + overhead : arr;
                    good_out[blk + (uint32_t)j] = good ? 1 : 0;
                }
            nrep = load_rep((int)nxt.z);
            if constexpr (W == 64) arrived(nn);
            cur = as_req(nxt);
            nxt = nn;
            q = nrep;
            look();
            if (SPANS && runs.own != 0) {
                if (runs.own < 0) run_vals = values_of(cold_args<WindowArgs>(), sim, (int)(blk / 64u / (uint32_t)cold_args<WindowArgs>()->span_blocks));
                run_vals[blk + (uint32_t)j] = OUTPUTS && want_req ? (good ? t + overhead : __builtin_nan("")) : took;
            } else if (accepted != 0ull) lat_sum = ordered_sum<W>(lat_sum, took, accepted);
        }
        if constexpr (!SPANS) break;
        // ---- the end of a run
        ColdArgs *q = cold_args<WindowArgs>();
        int first = 0, first_mark = -1;
        if (!last) {
            uint64_t *e = ended(own);
            for_state([&](int w, uint32_t addr, bool half) { e[w] = get_word(addr, half); });
            if (lane == 0) {
                if (own == 0) q->lat_sum[sim] = lat_sum;
                e[0] = (uint64_t)(uint32_t)n_good;
                e[q->state_words] = (uint64_t)(blk < R ? blk / 64u : (R + 63u) / 64u);
                e[q->state_words + 1] = runs.met ? (uint64_t)(uint32_t)runs.in | (uint64_t)(uint32_t)runs.mark << 32 : ~0ull;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            uint32_t before_me = 0;
            if (lane == 0)
                before_me = __hip_atomic_fetch_add(published(q->spans), 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
            if (__builtin_amdgcn_readfirstlane(before_me) + 1u != (uint32_t)q->spans) return;
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            // All runs have ended: this wavefront follows them from the first on.
            last = true;
            n_good = 0;
            if constexpr (OUTPUTS) {
                for (int k = j; k < q->nslots; k += W) lds_put<uint64_t>(clk + (uint32_t)k * 8u + cnt_rel, 0ull);
                for (int m = j; m < M; m += W) lds_put<uint32_t>(mcnt + (uint32_t)m * 4u, 0u);
            }
        } else {
            const uint32_t span = (uint32_t)q->span_blocks, stop = blk < R ? blk / 64u : (R + 63u) / 64u;
            for (uint32_t at = from / 64u; at < stop;) {
                const uint32_t in = at / span, next = (in + 1u) * span < stop ? (in + 1u) * span : stop;
                if (lane == 0) piece(num_pieces, at, next, (int)in);
                num_pieces += 1;
                at = next;
            }
            if (!runs.met) break;
            met_again += 1;
            first = runs.in;
            first_mark = runs.mark;
        }
        // Lane k: where run k ended, which it met and at which mark, and at which mark it is taken over (-1: from its beginning).
        int ends = 0, met = -1, met_mark = 0, taken_at = first_mark;
        uint32_t count = 0;
        if (lane < q->spans) {
            const uint64_t *e = ended(lane);
            count = (uint32_t)e[0];
            ends = (int)(uint32_t)e[q->state_words];
            met = (int)(uint32_t)e[q->state_words + 1];
            met_mark = (int)(uint32_t)(e[q->state_words + 1] >> 32);
        }
        uint64_t followed = 0;
        int tail = first;
        for (;;) {
            followed |= 1ull << tail;
            const int to = lane_value(met, tail);
            if (to < 0) break;
            if (lane == to) taken_at = lane_value(met_mark, tail);
            tail = to;
        }
        if (!in_mask(followed)) count = 0;
        else if (taken_at >= 0) count -= (uint32_t)marked(lane, taken_at)[0];
        for (int d = 1; d < kWave; d *= 2) count += (uint32_t)shfl_xor<kWave>((int)count, d);
        n_good += __builtin_amdgcn_readfirstlane((int)count);
        if constexpr (OUTPUTS) {
            auto counts = [&](int w) -> uint64_t {
                uint64_t v = 0;
#pragma unroll 2
                for (uint64_t left = followed; left != 0ull; left &= left - 1ull) {
                    const int r = __builtin_ctzll(left), m = lane_value(taken_at, r);
                    v += ended(r)[w] - (m < 0 ? 0ull : marked(r, m)[w]);
                }
                return v;
            };
            for (int k = j; k < q->nslots; k += W) {
                const uint32_t at = clk + (uint32_t)k * 8u + cnt_rel;
                lds_put<uint64_t>(at, lds_get<uint64_t>(at) + counts(1 + q->nslots + k));
            }
            for (int m = j; m < M; m += W) {
                const uint32_t at = mcnt + (uint32_t)m * 4u;
                lds_put<uint32_t>(at, lds_get<uint32_t>(at) + (uint32_t)counts(1 + 2 * q->nslots + m));
            }
        }
        if (in_mask(followed))
            piece(num_pieces + (uint32_t)__popcll(followed & ((1ull << lane) - 1ull)), (uint32_t)(lane * q->span_blocks + (taken_at < 0 ? 0 : span_mark(taken_at))),
                  (uint32_t)ends, lane);
        num_pieces += (uint32_t)__popcll(followed);
        const uint32_t end = (uint32_t)lane_value(ends, tail);
        if ((uint64_t)end * 64u >= R) break;
        // The last of them was given up: on from there.
        const uint32_t resume = end;
        for (int k = j; k < q->nslots; k += W) lds_put<uint64_t>(clk + (uint32_t)k * 8u, ended(tail)[1 + k]);
        wave_order();
        runs.resume(q, resume);
        from = resume * 64u;
    }

    if constexpr (SPANS) {
        // For the next launch; not before: a run that is taken up again looks at the marks.
        ColdArgs *q = cold_args<WindowArgs>();
        for (int k = j; k <= q->spans; k += W) tell(published(k), 0u);
        if (j == 0) tell(published(q->spans + 1), met_again);
    } else {
        for (int d = 1; d < W; d *= 2) n_good += shfl_xor<W>(n_good, d);
    }
    if (!mine) return;
    if (j == 0) {
        a.n_good[row] = n_good;
        if constexpr (SPANS) q_pieces(sim)[kPieceWords - 1] = num_pieces;
        else a.lat_sum[row] = lat_sum;
    }
    if constexpr (OUTPUTS) {
        if (a.flags & MMSIM_WANT_MODEL_COUNTS)
            for (int m = j; m < M; m += W) a.model_good[row * (size_t)M + (size_t)m] = (int32_t)lds_get<uint32_t>(mcnt + (uint32_t)m * 4u);
        if (a.flags & MMSIM_WANT_GROUP_COUNTS)
            for (int g = j; g < Gmax; g += W) {
                uint64_t v = 0ull;
                if (g < ng) v = lds_get<uint64_t>(entry_addr(lds_get<uint32_t>(gd + (uint32_t)g * 4u)) + cnt_rel);
                a.group_req[row * (size_t)Gmax + (size_t)g] = (int32_t)(uint32_t)v;
                a.group_good[row * (size_t)Gmax + (size_t)g] = (int32_t)(v >> 32);
            }
    }
}

#ifdef MMSIM_WINDOW_SPANS
// What the runs of a simulation come to: a workgroup adds up the latencies of the pieces that are followed, in their order, and writes
// the per-request outputs.  Sixteen blocks to a wavefront and round: all look at theirs side by side, for the sum as it is at the
// beginning of the round, and add in turn; one that takes the sum across a power of two is looked at again, block by block.
// One wavefront to a placement and lanes that worked out 64-bit masks each, against this: 700 placements of 108000 requests, three quarters of them
// here, 0.23 -> 0.22 ms (450 MB of latencies; a copy reads them in 0.1), 600 placements 0.34 -> 0.24, five of 82000 0.20 -> 0.12, one of 30000 with outputs 0.10 -> 0.08.
__global__ __launch_bounds__(kSumWaves *kWave) void window_sum_kernel(const WindowArgs a) {
    constexpr int N = 16;
    __shared__ uint32_t pieces[kPieceWords];
    __shared__ double added[kSumWaves], more_if_odd[kSumWaves], exact;
    __shared__ int negative[kSumWaves];
    const int lane = lane_id(), wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), waves = (int)(blockDim.x >> 6), sim = (int)blockIdx.x;
    ColdArgs *q = cold_args<WindowArgs>();
    for (int k = (int)threadIdx.x; k < kPieceWords; k += (int)blockDim.x) pieces[k] = a.pieces[(size_t)sim * kPieceWords + k];
    __syncthreads();
    const int num = __builtin_amdgcn_readfirstlane((int)pieces[kPieceWords - 1]);
    const bool want_req = (a.flags & MMSIM_WANT_PER_REQUEST) != 0;
    const int seed = __builtin_amdgcn_readfirstlane(a.stream_of ? a.stream_of[sim] : sim / a.tiles);
    const Req *__restrict__ reqs = a.stream_ptr[seed];
    const uint32_t R = (uint32_t)a.stream_len[seed], blocks = (R + 63u) / 64u;
    double *fin_out = a.finish + (size_t)sim * (size_t)a.Rmax;
    uint8_t *good_out = a.good + (size_t)sim * (size_t)a.Rmax;
    if (num < 2) return;  // (the first run went through the whole stream)
    const uint32_t begin = (uint32_t)__builtin_amdgcn_readfirstlane((int)pieces[1]);  // where the first run ends
    int p = 0;
    uint32_t p_end = begin;
    const double *v = nullptr;
    auto load = [&](uint32_t first, double *x, double *arr) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint32_t at = first + i < blocks ? first + i : blocks - 1;
            while (at >= p_end && p + 1 < num) {
                ++p;
                p_end = (uint32_t)__builtin_amdgcn_readfirstlane((int)pieces[4 * p + 1]);
                v = values_of(q, sim, __builtin_amdgcn_readfirstlane((int)pieces[4 * p + 2]));
            }
            const uint32_t pos = at * (uint32_t)kWave + (uint32_t)lane;
            x[i] = v[pos];
            if (want_req) arr[i] = as_req(load_global(reqs + (pos < R ? pos : R - 1u))).t;
        }
    };
    LatencySum sum(a.lat_sum[sim]);  // (the same in all wavefronts)
    double x[N], y[N], arr[N];
    const uint32_t round = (uint32_t)(waves * N);
    uint32_t mine = begin + (uint32_t)(wv * N);
    load(mine, y, arr);
    for (uint32_t at = begin; at < blocks; at += round, mine += round) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint32_t pos = (mine + i) * (uint32_t)kWave + (uint32_t)lane;
            const bool in = mine + i < blocks && pos < R;
            x[i] = y[i];
            if (want_req) {  // finish times, NaN of the requests that are not accepted
                const bool good = x[i] == x[i];
                if (in) {
                    fin_out[pos] = good ? x[i] : arr[i];
                    good_out[pos] = good ? 1 : 0;
                }
                x[i] = good ? x[i] - arr[i] : 0.0;
            }
            if (!in) x[i] = 0.0;
        }
        if (mine + round < blocks) load(mine + round, y, arr);
        double mine_added, mine_more;
        bool mine_negative;
        sum.look(x, &mine_added, &mine_more, &mine_negative);
        if (lane == 0) {
            added[wv] = mine_added;
            more_if_odd[wv] = mine_more;
            negative[wv] = mine_negative ? 1 : 0;
        }
        __syncthreads();
        const double base = sum.base;  // what they were looked at for
        for (int k = 0; k < waves; ++k) {
            if (sum.base == base && sum.add(added[k], more_if_odd[k], negative[k] != 0)) continue;
            if (wv == k) {
                sum.look(x, &mine_added, &mine_more, &mine_negative);
                if (!sum.add(mine_added, mine_more, mine_negative))
#pragma unroll 1
                for (int i = 0; i < N; ++i) {
                    double w = x[0];
#pragma unroll
                    for (int l = 1; l < N; ++l) w = i == l ? x[l] : w;
                    sum.add_block(w);
                }
                if (lane == 0) exact = sum.s;
            }
            __syncthreads();
            sum.set(exact);
            __syncthreads();
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) a.lat_sum[sim] = sum.s;
}
#endif

constexpr int W_ = MMSIM_WINDOW_LANES;  // the file is compiled once for each number of requests side by side
#ifdef MMSIM_WINDOW_SPANS
constexpr bool kSpans = true;           // and for simulations cut into runs
#else
constexpr bool kSpans = false;
#endif

template <int SMAX, bool OUTPUTS, bool POW2, bool UNIFORM>
WindowKernel pick_ext(int ext) {
    if (W_ == 64 && ext > 1) return sim_window_kernel<W_, SMAX, OUTPUTS, W_ == 64 ? 2 : 1, POW2, UNIFORM, kSpans>;
    return ext > 0 ? sim_window_kernel<W_, SMAX, OUTPUTS, 1, POW2, UNIFORM, kSpans> : sim_window_kernel<W_, SMAX, OUTPUTS, 0, POW2, UNIFORM, kSpans>;
}
template <int SMAX, bool POW2, bool UNIFORM>
WindowKernel pick_out(bool outputs, int ext) {
    return outputs ? pick_ext<SMAX, true, POW2, UNIFORM>(ext) : pick_ext<SMAX, false, POW2, UNIFORM>(ext);
}
template <int SMAX>
WindowKernel pick_depths(bool outputs, int ext, bool pow2, bool uniform) {
    if (pow2) return uniform ? pick_out<SMAX, true, true>(outputs, ext) : pick_out<SMAX, true, false>(outputs, ext);
    return uniform ? pick_out<SMAX, false, true>(outputs, ext) : pick_out<SMAX, false, false>(outputs, ext);
}

}  // namespace

#ifdef MMSIM_WINDOW_SPANS
WindowKernel window_sum() { return window_sum_kernel; }
#endif

template <>
WindowKernel window_kernel<MMSIM_WINDOW_LANES, kSpans>(int smax, bool outputs, int ext, bool pow2, bool uniform) {
    switch (smax) {
        case 1: return pick_out<1, true, true>(outputs, ext);  // one stage: its latency is the configuration's
        case 4: return pick_depths<4>(outputs, ext, pow2, uniform);
        case 16: return pick_depths<16>(outputs, ext, pow2, uniform);
        case 32: return pick_depths<32>(outputs, ext, pow2, uniform);
        default: return nullptr;
    }
}

}  // namespace mmsim
