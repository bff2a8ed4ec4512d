// Host side of the kernel that simulates requests side by side (sim_window.hip): which batches it is for, how many
// requests of a placement share a wavefront, packing, launch, results.
//
// The placements travel as they were given, a few bytes per replica: the wavefronts build their own tables (the other
// kernels' descriptor tables are a kilobyte per placement and model of a tile).  One buffer holds every input and one
// every output, so a call is one copy in, one launch and one copy out, through the context's pinned staging memory
// (mmsim_eval_batch_static, which must not call the runtime's allocators: through ordinary memory).
#include <cstring>

#include "mmsim_host.h"

namespace mmsim {
namespace {

size_t up16(size_t v) { return (v + 15) & ~(size_t)15; }

// Bump layout of a buffer: offset of the next array.
struct Layout {
    size_t used = 0;
    size_t take(size_t bytes) {
        const size_t at = used;
        used += (bytes + 255) & ~(size_t)255;
        return at;
    }
};

bool has_outputs(uint32_t flags) {
    return (flags & (MMSIM_WANT_PER_REQUEST | MMSIM_WANT_MODEL_COUNTS | MMSIM_WANT_GROUP_COUNTS)) != 0;
}

hipError_t launch_window(const WindowArgs &a, int waves_per_block, size_t lds_bytes, hipStream_t stream) {
    const int ext = a.has_ext;
    const bool out = has_outputs(a.flags), pow2 = a.pow2_depths != 0, uniform = a.uniform_stages != 0;
    const WindowKernel kern = a.spans > 1     ? window_kernel<64, true>(a.smax_bucket, out, ext, pow2, uniform)
                              : a.lanes == 64 ? window_kernel<64, false>(a.smax_bucket, out, ext, pow2, uniform)
                              : a.lanes == 32 ? window_kernel<32, false>(a.smax_bucket, out, ext, pow2, uniform)
                              : a.lanes == 16 ? window_kernel<16, false>(a.smax_bucket, out, ext, pow2, uniform)
                                              : window_kernel<8, false>(a.smax_bucket, out, ext, pow2, uniform);
    if (!kern || waves_per_block < 1 || waves_per_block > kMaxWindowWaves) return hipErrorInvalidValue;
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
    const int64_t units = (int64_t)a.tiles * a.out_seeds * a.spans;
    hipLaunchKernelGGL(kern, dim3((unsigned)((units + waves_per_block - 1) / waves_per_block)), dim3((unsigned)waves_per_block * kWave),
                       lds_bytes, stream, a);
    if (a.spans > 1)
        hipLaunchKernelGGL(window_sum(), dim3((unsigned)(a.tiles * a.out_seeds)), dim3(kWave * kSumWaves), 0, stream, a);
    return hipGetLastError();
}

struct Shape {
    int32_t nslots = 1, smax = 1, rmax = 1, ext_cap = 0;
    bool pow2 = true;  // every group has 1, 2, 4, ... stages
    int64_t depths = 0;  // stages of the group of every replica, added up
};

}  // namespace

int build_window(mmsim_ctx *ctx, const mmsim_workload *const *wls, int32_t n_seeds, const mmsim_tables *t,
                 const mmsim_placements *p, const int32_t *stream_of, uint32_t flags, const mmsim_options &o, bool events,
                 mmsim_batch **out) {
    constexpr int kOther = 1;  // the batch is for the other kernels, or they will say what is wrong with it
    if (o.window_lanes < 0 || (flags & (MMSIM_BATCHING | MMSIM_WANT_OP_COUNT))) return kOther;
    if (o.window_lanes == 0 && (o.request_loop >= 0 || o.waves_per_cu > 0 || o.counts_in_lds >= 0 || o.tile_order_by_slots >= 0 ||
                                o.sched_groups > 0 || o.segment_requests > 0 || o.sched_spin_limit >= 0 || o.skip_ahead >= 0 || o.xcd_map >= 0))
        return kOther;
    if (!p || !p->num_groups || !p->group_cfg || !p->gm_off || p->B < 1 || p->Gmax < 1 || p->Gmax > MMSIM_MAX_GROUPS) return kOther;
    if (n_seeds < 1 || !wls || t->M > 65535) return kOther;
    for (int s = 0; s < n_seeds; ++s)
        if (!wls[s] || wls[s]->ctx != ctx || wls[s]->M != t->M) return kOther;
    const int32_t B = p->B, M = t->M, Gmax = p->Gmax, C = t->C;
    const int32_t out_seeds = stream_of ? 1 : n_seeds;
    const int64_t sims = (int64_t)B * out_seeds;
    if (o.window_lanes == 0 && sims > kMaxWindowSims) return kOther;
    if (stream_of)
        for (int32_t b = 0; b < B; ++b)
            if (stream_of[b] < 0 || stream_of[b] >= n_seeds) return kOther;
    CompactLatency cl;
    if (compact_latency(t, false, &cl) != MMSIM_OK) return kOther;

    // Beyond what the chip's LDS holds at once in any case (see below): known before anything is packed.
    const size_t lds = (size_t)ctx->max_lds;
    const int group_words = (Gmax + 31) / 32;
    const int64_t cus = std::max(1, ctx->prop.multiProcessorCount);
    const size_t place_least = (size_t)M * 32 + (size_t)M * group_words * 4;
    if (place_least > lds) return kOther;
    // A call that evaluates a batch once packs it for the other kernel at about 18 ns per placement and model, and for this
    // one at a tenth of that; the other kernel runs 0.5 us per request.  Where that is the faster one (the lines below), it is
    // by a quarter of its time or so and worth its packing with streams of more than a sixth of placements x models.  Whole
    // calls, 3000 / 12000 / 50000 requests, against the other kernel: 12288 placements in groups of 2 to 16 devices, 32
    // models, 2.4 / 7.8 / 29 against 8.3 / 12.9 / 32 ms; 5000 16-stage pipelines, 16 models, 2.0 / 7.3 / 29 against 4.2 /
    // 7.8 / 26; 12288 placements of 128 models, twice what LDS holds, 2.7 / 7.1 / 25 against 29 / 34 / 53.
    // In the static scratch the batch stays here too: the other kernel's tables are a hundred times as large.
    int64_t longest = 0;
    for (int s = 0; s < n_seeds; ++s) longest = std::max(longest, wls[s]->R);
    const bool packing_counts = g_arena || (!events && (int64_t)B * M >= 6 * longest);
    const int64_t most_in_rounds = packing_counts ? kMaxWindowSims : 8192;  // simulations that LDS does not hold at once
    if (o.window_lanes == 0 && sims > most_in_rounds && sims > cus * (int64_t)(lds / place_least)) return kOther;

    // ---- inputs: one buffer
    Layout in;
    int64_t replicas = 0;
    for (int32_t b = 0; b < B; ++b) {
        const int32_t G = p->num_groups[b];
        if (G < 0 || G > Gmax) return kOther;
        const int64_t *off = p->gm_off + (size_t)b * (Gmax + 1);
        if (off[G] < off[0] || (off[G] > off[0] && !p->gm_idx) || off[G] - off[0] > (int64_t)M * MMSIM_MAX_REPLICAS) return kOther;
        replicas += off[G] - off[0];
        if (replicas > 0x7FFFFFFF) return kOther;
    }
    const size_t at_ptr = in.take(sizeof(void *) * (size_t)n_seeds), at_len = in.take(sizeof(int64_t) * (size_t)n_seeds);
    const size_t at_so = in.take(stream_of ? sizeof(int32_t) * (size_t)B : 0);
    const size_t at_ng = in.take((size_t)B), at_cfg = in.take((size_t)B * Gmax), at_off = in.take(sizeof(uint32_t) * ((size_t)B + 1));
    const size_t at_ent = in.take(sizeof(uint32_t) * (size_t)replicas), at_pp = in.take((size_t)C), at_loff = in.take(sizeof(uint16_t) * (size_t)C);
    const size_t at_lat = in.take(sizeof(float) * (cl.lat.size() + MMSIM_MAX_STAGES));  // (the walk reads past a shallow group's row)
    const int64_t blocks = (longest + kWave - 1) / kWave;
    const bool may_cut = !g_arena && (o.window_lanes > 0 ? o.segment_requests > 0 : blocks >= 6 * kLeastSpan);
    const size_t at_sync = in.take(may_cut ? sizeof(uint32_t) * (size_t)(sims * kSyncWords + std::min<int64_t>(kMaxRuns, sims * kMaxSpans)) : 0);
    HIP_TRY(hipSetDevice(ctx->device));
    std::vector<unsigned char> plain;  // (read until the wait below)
    if (g_arena)
        plain.resize(in.used);
    else
        HIP_TRY(ctx->staging.ensure(in.used));
    struct Trim {  // the memory of a batch that is not made after all
        Staging *staging;
        hipStream_t stream;
        ~Trim() {
            if (!staging) return;
            if (staging->n > Staging::kMost) (void)hipStreamSynchronize(stream);  // (the inputs may be on their way out of it)
            staging->trim();
        }
    } unless_made{g_arena ? nullptr : &ctx->staging, ctx->stream};
    unsigned char *host = g_arena ? plain.data() : ctx->staging.p;
    uint8_t *h_ng = host + at_ng, *h_cfg = host + at_cfg;
    uint32_t *h_off = reinterpret_cast<uint32_t *>(host + at_off), *h_ent = reinterpret_cast<uint32_t *>(host + at_ent);
    {
        uint32_t at = 0;
        for (int32_t b = 0; b < B; ++b) {
            const int64_t *off = p->gm_off + (size_t)b * (Gmax + 1);
            h_off[b] = at;
            at += (uint32_t)(off[p->num_groups[b]] - off[0]);
        }
        h_off[B] = at;
    }
    std::atomic<bool> bad{false};
    std::mutex shape_mutex;
    Shape shape;
    parallel_slices(B, 1024, [&](int64_t b0, int64_t b1) {
        Shape mine;
        std::vector<uint8_t> count((size_t)M, 0);
        for (int64_t b = b0; b < b1; ++b) {
            const int32_t G = p->num_groups[b];
            const int64_t *off = p->gm_off + (size_t)b * (Gmax + 1);
            const int32_t *cfg = p->group_cfg + (size_t)b * Gmax;
            uint32_t *ent = h_ent + h_off[b];  // (room for off[G] - off[0])
            int32_t slots = 0, chunks = 0;
            h_ng[b] = (uint8_t)G;
            for (int32_t g = 0; g < Gmax; ++g) {
                h_cfg[(size_t)b * Gmax + g] = g < G ? (uint8_t)cfg[g] : 0;
                if (g >= G) continue;
                if (cfg[g] < 0 || cfg[g] >= C || off[g + 1] < off[g] || off[g + 1] > off[G]) {
                    bad = true;
                    return;
                }
                const int32_t pp = t->cfg_pp[cfg[g]];
                slots += pp;
                mine.pow2 = mine.pow2 && (pp & (pp - 1)) == 0;
                mine.smax = std::max(mine.smax, pp);
                mine.depths += (off[g + 1] - off[g]) * pp;
                for (int64_t x = off[g]; x < off[g + 1]; ++x) {
                    const int32_t m = p->gm_idx[x];
                    if (m < 0 || m >= M || count[m] >= MMSIM_MAX_REPLICAS) {
                        bad = true;
                        return;
                    }
                    *ent++ = (uint32_t)m | (uint32_t)g << 16;
                    chunks += count[m] >= 4 && (count[m] & 3) == 0;
                    count[m] += 1;
                    mine.rmax = std::max<int32_t>(mine.rmax, count[m]);
                }
            }
            if (slots > MMSIM_MAX_SLOTS) {
                bad = true;
                return;
            }
            mine.nslots = std::max(mine.nslots, slots);
            mine.ext_cap = std::max(mine.ext_cap, chunks);
            for (const uint32_t *e = h_ent + h_off[b]; e < ent; ++e) count[*e & 0xFFFFu] = 0;
        }
        std::lock_guard<std::mutex> lock(shape_mutex);
        shape.nslots = std::max(shape.nslots, mine.nslots);
        shape.smax = std::max(shape.smax, mine.smax);
        shape.pow2 = shape.pow2 && mine.pow2;
        shape.rmax = std::max(shape.rmax, mine.rmax);
        shape.ext_cap = std::max(shape.ext_cap, mine.ext_cap);
        shape.depths += mine.depths;
    });
    if (bad) return kOther;

    // ---- LDS of one placement, lanes per placement, wavefronts per workgroup
    WindowArgs a{};
    a.smax = shape.smax;
    a.smax_bucket = smax_bucket_for(shape.smax);
    if (a.smax_bucket < 0) return kOther;
    const bool uniform = cl.uniform || a.smax_bucket == 1;
    const bool counts = has_outputs(flags);
    // (behind the clocks as many slots as a walk has stages, for reads and writes that do not count)
    size_t place = up16(((size_t)shape.nslots + a.smax_bucket) * 8 * (counts ? 3 : 2));
    a.o_rep = (int32_t)place;
    place += (size_t)M * 32;
    a.o_ext = (int32_t)place;
    place += (size_t)shape.ext_cap * 32;
    a.o_xi = (int32_t)place;
    place = up16(place + (shape.ext_cap > 0 ? (size_t)M * 4 : 0));
    a.o_bits = (int32_t)place;
    place = up16(place + (size_t)M * group_words * 4);
    a.o_gd = (int32_t)place;
    place = up16(place + ((size_t)Gmax + 1) * 4);
    a.o_mcnt = (int32_t)place;
    place = up16(place + (counts ? (size_t)M * 4 : 0));
    const size_t lat_bytes = uniform ? 0 : up16(cl.lat.size() * sizeof(float));
    if (place > lds) return kOther;
    const size_t lat_lds = lat_bytes + place <= lds ? lat_bytes : 0;
    auto wave_lds = [&](int lanes) { return place * (size_t)(kWave / lanes) + (size_t)window_ring_bytes(lanes); };
    auto fits = [&](int lanes) { return lat_lds + wave_lds(lanes) <= lds; };
    auto waves_for = [&](int l) {  // wavefronts of a workgroup
        const int64_t units = (B + kWave / l - 1) / (kWave / l) * out_seeds;
        int waves = (int)std::min<int64_t>(kMaxWindowWaves, std::max<int64_t>(1, (units + cus - 1) / cus));
        while (waves > 1 && lat_lds + wave_lds(l) * (size_t)waves > lds) --waves;
        return waves;
    };
    auto at_once = [&](int l) {  // placements on the chip at once, in workgroups of so many wavefronts
        const int waves = waves_for(l);
        return cus * (int64_t)(lds / (lat_lds + wave_lds(l) * (size_t)waves)) * waves * (kWave / l);
    };
    int lanes = o.window_lanes;
    if (lanes == 0) {
        // Up to how many simulations, and how many requests side by side.  Measured on some 500 batches (12000 or 20000
        // requests at 1 to 12 a second and model; 1025 to 12288 placements of 16 to 300 models on 16 to 64 devices, in
        // groups of 1 to 32 stages); below: milliseconds at 64 / 32 / 16 / 8 lanes against 64 placements to a wavefront.
        //
        // A step is longer the deeper the groups are, while with 64 placements to a wavefront the depth costs little; what
        // counts is between the mean and the deepest.  Groups of 2 to 16 devices (3.5 and 16 stages), 8192: 7.1 / 6.7 / 5.3
        // / 5.8 against 6.0, 12288: 9.4 / 8.8 / 6.8 / 10.7; 16-stage pipelines, 4096: 7.8 / 5.6 / 4.9 / 5.3 against 5.7,
        // 8192: 14.7 / 9.9 / 7.1 / 5.9; 1 to 8 stages (3.2), 12288: 7.5 / 6.3 / 5.1 / 8.7 against 5.7.  Depths other than
        // 1, 2, 4, 8 and 16 are slow in the other kernel (6.4 and 12 stages, 12288: 11.7 / 9.7 / 7.7 / 12.2 against 10.7),
        // and paired batches fill its tiles with what one stream has.
        const double mean = replicas > 0 ? (double)shape.depths / (double)replicas : 1.0, depth = (shape.smax + mean) / 2;
        const bool any_depth = packing_counts || stream_of || !shape.pow2 || shape.smax > 16;
        if (sims > (any_depth || depth <= 6 ? kMaxWindowSims : depth <= 10 ? 8192 : 4096)) return kOther;
        // More than LDS holds at once: the wavefronts with one placement each, which follow one another freely (8192 of 300
        // models: 2.1 / 3.0 / 4.8 / 7.7 against 4.6; of 128 models, at worst, 5.7 / 5.1 / 5.8 / 7.3 against 5.2; 12288: 3.0 to
        // 8.5 against 4.5 to 6.1), but narrower ones with deep groups, whose steps are long.
        lanes = kWave;
        const bool rounds = sims > at_once(kWave);
        if (rounds && (sims > most_in_rounds || !fits(kWave))) return kOther;
        // (12288 16-stage pipelines of 64 models: 3000 requests 2.7 against 9.1 with the packing, 12000: 9.7 / 13.5, 50000: 37 / 31)
        if (rounds && depth > 10 && shape.pow2 && shape.smax <= 16 && !g_arena && (int64_t)B * M < 20 * longest) return kOther;
        if (!rounds || depth > 10) {
            // As many requests side by side as leave three wavefronts to a SIMD (the registers of the kernels for up to 16
            // stages hold three or four), four of the single-stage kernel, two of deep groups.  Four-stage pipelines, 3000:
            // 3.6 / 4.2 / 4.5 / 5.6, 6000: 5.6 / 4.9 / 5.7 / 6.2, 12288: 10.2 / 9.3 / 7.2 / 7.8; single stages, 4096: 2.6 / 2.8
            // / 3.8 / 5.0, 8192: 4.5 / 4.2 / 4.4 / 5.7; eight-stage pipelines, 12288: 14.8 / 10.0 / 6.9 / 6.1; 32-stage ones 45 / 29
            // / 19 / 15.  A narrower wavefront needs more LDS, for its placements and for the requests on their way to them:
            // where it would take two rounds instead of one, up to twice as many wavefronts stay (5000 placements of 128
            // models, 5.1 / 6.4).  Streams that ask twice what the groups can do are mostly runs of rejects, which the widest
            // blocks settle in the fewest steps: four to a SIMD there (4096 placements of groups of 1 to 16 stages, 64 / 32 lanes,
            // load 0.4: 26.8 / 23.7, 3.4: 14.6 / 14.6, single devices or 16 stages: load 0.9 263 / 264, 3.5 144 / 157; four-stage
            // pipelines 0.4: 18.9 / 18.1, 1.7: 13.7 / 14.4, 3.4: 9.4 / 10.4; streams of a few blocks take microseconds either way).
            int64_t most = (a.smax_bucket == 1 ? 16 : mean > 7 ? 8 : 12) * cus;
            if (most == 12 * cus && sims > most && sims <= 16 * cus && longest >= 1024 && offered_load(wls, n_seeds, t, B, Gmax, p->num_groups, p->group_cfg) >= 2.0)
                most = 16 * cus;
            while (lanes > 8 && sims * lanes / kWave > most && fits(lanes / 2) &&
                   (sims <= at_once(lanes / 2) || sims * lanes / kWave > 2 * most || (depth > 10 && sims > at_once(lanes))))
                lanes /= 2;
        }
    }
    if (stream_of) lanes = kWave;  // (the placements of a wavefront share a stream)
    while (lanes < kWave && !fits(lanes)) lanes *= 2;
    if (!fits(lanes)) return kOther;
    const int per_wave = kWave / lanes;
    const int64_t tiles = (B + per_wave - 1) / per_wave, units = tiles * out_seeds;

    // ---- runs
    a.state_words = 1 + shape.nslots + (counts ? shape.nslots + M : 0);
    Layout runs;
    size_t at_ends = 0, at_pieces = 0, at_vals = 0;
    auto cut = [&](int64_t spans) {
        a.span_blocks = (int32_t)std::max<int64_t>((blocks + spans - 1) / spans, 1);
        a.spans = (int32_t)std::max<int64_t>((blocks + a.span_blocks - 1) / a.span_blocks, 1);
        a.ext_blocks = std::max(a.span_blocks / 2, kLeastExt);
        a.run_cap = (int64_t)kWave * (a.span_blocks + a.ext_blocks);
        for (a.marks = 0; span_mark(a.marks) < a.span_blocks;) ++a.marks;
        const size_t n = a.spans > 1 ? (size_t)(units * a.spans) : 0;
        runs = Layout{};
        runs.take(8 * n * (size_t)a.marks * (size_t)a.state_words);
        at_ends = runs.take(8 * n * (size_t)(a.state_words + kEndWords));
        at_pieces = runs.take(4 * (n > 0 ? (size_t)units : 0) * kPieceWords);
        at_vals = runs.take(n > 0 ? 8 * (size_t)units * (size_t)((a.spans - 1) * a.run_cap) : 0);
    };
    // sixteen replicas in registers, which leaves two or three wavefronts to a SIMD: sim_window.hip has both sides
    const bool sixteen = lanes == kWave && shape.rmax > 8 && units <= 8 * cus;
    int64_t spans = 1;
    if (lanes == kWave && may_cut) {
        // As many runs as leave three wavefronts to a SIMD (a few more than that wait for their turn; 2.9 ms of kernel with two
        // to a SIMD, 700 placements and 108000 requests, are 4.3, and four do not fit with counts: 6.0), of 20 blocks at least (30000 requests of one placement: 16 and 24
        // are level, 8 a third slower, as runs are given up).  Streams of less than 384 blocks have them while every run has a SIMD to itself: where runs
        // do not agree the first one shares issue with the others for a span and a half (393 placements, 5844 requests: 2.0 ms not cut, 2.6
        // with four runs); below 120 blocks there is little to gain (5757 requests 155 us, with a second kernel 190).
        const int64_t per_cu = blocks < 384 ? 4 : sixteen || a.smax_bucket == 32 ? 8 : 12;
        spans = std::min((per_cu * cus + cus / 2) / units, blocks / kLeastSpan);
        if (o.window_lanes == 0 && spans > 1 &&
            !runs_agree_early(wls, n_seeds, offered_load(wls, n_seeds, t, B, Gmax, p->num_groups, p->group_cfg), replicas_of_a_request(wls, n_seeds, p, M), 1.0))
            spans = 1;
        if (o.window_lanes > 0) spans = blocks / std::max<int64_t>(8, o.segment_requests / kWave);
    }
    cut(std::max<int64_t>(1, std::min<int64_t>(spans, std::min<int64_t>(kMaxSpans, kMaxRuns / units))));
    if (a.spans > 1 && !ctx->runs.fits(runs.used)) cut(1);
    spans = a.spans;
    a.alike = Gmax <= kWave ? 1 : 0;
    for (int s = 0; s < n_seeds; ++s)
        if (!wls[s]->sorted) a.alike = 0;
    for (const float l : cl.lat)
        if (!(l >= 0.0f)) a.alike = 0;
    const int64_t wave_units = units * spans;
    int waves = spans > 1 ? (int)std::min<int64_t>(kMaxWindowWaves, std::max<int64_t>(1, (wave_units + cus - 1) / cus)) : waves_for(lanes);
    while (spans > 1 && waves > 1 && lat_lds + wave_lds(lanes) * (size_t)waves > lds) --waves;

    std::unique_ptr<mmsim_batch> b(new (std::nothrow) mmsim_batch);
    if (!b) return fail(MMSIM_E_NOMEM, "host allocation failed");
    b->ctx = ctx;
    b->opt = o;
    b->window = true;
    b->flags = flags;
    b->n_seeds = n_seeds;
    b->B = B;
    b->M = M;
    b->Gmax = Gmax;
    b->paired = stream_of != nullptr;
    b->out_seeds = out_seeds;
    b->tiles = (int32_t)tiles;
    b->waves = (int32_t)wave_units;
    b->smax_bucket = a.smax_bucket;
    b->rmax_all = shape.rmax;
    b->nslots = shape.nslots;
    b->waves_per_block = waves;
    b->lds_bytes = lat_lds + wave_lds(lanes) * (size_t)waves;
    if (stream_of) b->stream_of.assign(stream_of, stream_of + B);
    const Req **h_ptr = reinterpret_cast<const Req **>(host + at_ptr);
    int64_t *h_len = reinterpret_cast<int64_t *>(host + at_len);
    for (int s = 0; s < n_seeds; ++s) {
        b->wl_R.push_back(wls[s]->R);
        b->wl_id.push_back(wls[s]->id);
        b->wl_model_requests.push_back(wls[s]->model_num_requests);
        b->win_streams.push_back(wls[s]->reqs);  // (the workload may be destroyed before the batch)
        h_ptr[s] = wls[s]->reqs->p;
        h_len[s] = wls[s]->R;
        b->Rmax = std::max(b->Rmax, wls[s]->R);
        b->Rtotal += wls[s]->R;
    }
    if (stream_of) std::memcpy(host + at_so, stream_of, sizeof(int32_t) * (size_t)B);
    for (int32_t c = 0; c < C; ++c) {
        (host + at_pp)[c] = (uint8_t)t->cfg_pp[c];
        reinterpret_cast<uint16_t *>(host + at_loff)[c] = (uint16_t)cl.off[c];
    }
    std::memcpy(host + at_lat, cl.lat.data(), sizeof(float) * cl.lat.size());

    std::memset(host + at_sync, 0, spans > 1 ? sizeof(uint32_t) * (size_t)(units * (spans + kSyncWords)) : 0);

    // ---- outputs: one buffer, laid out as the caller's arrays
    Layout res;
    const size_t L = (size_t)sims;
    res.take(sizeof(int32_t) * L);
    b->win_lat_sum = res.take(sizeof(double) * L);
    b->win_model = res.take((flags & MMSIM_WANT_MODEL_COUNTS) ? sizeof(int32_t) * L * M : 0);
    b->win_group = res.take((flags & MMSIM_WANT_GROUP_COUNTS) ? 2 * sizeof(int32_t) * L * Gmax : 0);
    b->win_finish = res.take((flags & MMSIM_WANT_PER_REQUEST) ? sizeof(double) * L * (size_t)b->Rmax : 0);
    b->win_good = res.take((flags & MMSIM_WANT_PER_REQUEST) ? L * (size_t)b->Rmax : 0);

    HIP_TRY(b->win_in.alloc(in.used));
    HIP_TRY(b->win_out.alloc(res.used));
    HIP_TRY(hipMemcpyAsync(b->win_in.p, host, in.used, hipMemcpyHostToDevice, ctx->stream));
    if (events) {
        if (g_arena) {
            b->own_events = false;
            b->in_scratch = true;
            b->ev_start = ctx->ev_static[0];
            b->ev_stop = ctx->ev_static[1];
        } else {
            HIP_TRY(hipEventCreate(&b->ev_start));
            HIP_TRY(hipEventCreate(&b->ev_stop));
        }
        HIP_TRY(hipStreamSynchronize(ctx->stream));  // a batch that is kept: the staging memory serves other calls before its run
        if (!g_arena) ctx->staging.trim();
    }
    uint8_t *d = b->win_in.p;
    a.span_sync = reinterpret_cast<uint32_t *>(d + at_sync);
    a.stream_ptr = reinterpret_cast<const Req *const *>(d + at_ptr);
    a.stream_len = reinterpret_cast<const int64_t *>(d + at_len);
    a.stream_of = stream_of ? reinterpret_cast<const int32_t *>(d + at_so) : nullptr;
    a.num_groups = d + at_ng;
    a.group_cfg = d + at_cfg;
    a.entry_off = reinterpret_cast<const uint32_t *>(d + at_off);
    a.entries = reinterpret_cast<const uint32_t *>(d + at_ent);
    a.cfg_pp = d + at_pp;
    a.lat_off = reinterpret_cast<const uint16_t *>(d + at_loff);
    a.lat = reinterpret_cast<const float *>(d + at_lat);
    a.M = M;
    a.lat_row = cl.row;
    a.B = B;
    a.Gmax = Gmax;
    a.group_words = group_words;
    a.nslots = shape.nslots;
    a.tiles = (int32_t)tiles;
    a.out_seeds = out_seeds;
    a.lanes = lanes;
    a.pow2_depths = shape.pow2 ? 1 : 0;
    a.uniform_stages = uniform ? 1 : 0;
    a.has_ext = shape.ext_cap > 0 ? (sixteen ? 2 : 1) : 0;
    a.lat_lds_bytes = (int32_t)lat_lds;
    a.place_bytes = (int32_t)place;
    a.Rmax = b->Rmax;
    a.fixed_overhead = t->fixed_overhead;
    a.flags = flags;
    uint8_t *r = b->win_out.p;
    a.n_good = reinterpret_cast<int32_t *>(r);
    a.lat_sum = reinterpret_cast<double *>(r + b->win_lat_sum);
    a.model_good = reinterpret_cast<int32_t *>(r + b->win_model);
    a.group_req = reinterpret_cast<int32_t *>(r + b->win_group);
    a.group_good = a.group_req + L * Gmax;
    a.finish = reinterpret_cast<double *>(r + b->win_finish);
    a.good = r + b->win_good;
    b->wargs = a;
    if (spans > 1) {
        b->run_bytes = runs.used;
        b->run_ends = at_ends;
        b->run_pieces = at_pieces;
        b->run_vals = at_vals;
        if (events) b->run_again(&ctx->runs);
    }
    unless_made.staging = nullptr;
    *out = b.release();
    return MMSIM_OK;
}

std::string sim_window_kernel_name(const WindowArgs &a) {
    auto tf = [](bool v) { return v ? ", true" : ", false"; };
    return "sim_window_kernel<" + std::to_string(a.lanes) + ", " + std::to_string(a.smax_bucket) + tf(has_outputs(a.flags)) + ", " + std::to_string(a.has_ext) +
           tf(a.pow2_depths != 0) + tf(a.uniform_stages != 0) + (a.spans > 1 ? ", true>" : ">");
}

int run_window(mmsim_batch *b) {
    WindowArgs &a = b->wargs;
    if (a.spans > 1) {
        if (uint8_t *at = b->ctx->runs.ensure(b->run_bytes, b->ctx->stream)) {
            a.mark_state = reinterpret_cast<uint64_t *>(at);
            a.end_state = reinterpret_cast<uint64_t *>(at + b->run_ends);
            a.pieces = reinterpret_cast<uint32_t *>(at + b->run_pieces);
            a.run_vals = reinterpret_cast<double *>(at + b->run_vals);
        } else {  // not cut from here on
            b->waves /= a.spans;
            a.spans = 1;
        }
    }
    if (b->ev_start) HIP_TRY(hipEventRecord(b->ev_start, b->ctx->stream));
    const hipError_t e = launch_window(b->wargs, b->waves_per_block, b->lds_bytes, b->ctx->stream);
    if (e == hipErrorInvalidKernelFile) return fail(MMSIM_E_HIP, "simulation kernel: dynamic LDS does not start at address 0");
    if (e != hipSuccess) return hip_fail(e, "sim_window launch");
    if (b->ev_stop) HIP_TRY(hipEventRecord(b->ev_stop, b->ctx->stream));
    b->ran = true;
    return MMSIM_OK;
}

int fetch_window(mmsim_batch *b, mmsim_result *out) {
    const bool wm = b->flags & MMSIM_WANT_MODEL_COUNTS, wg = b->flags & MMSIM_WANT_GROUP_COUNTS,
               wr = (b->flags & MMSIM_WANT_PER_REQUEST) && out->finish && out->good;
    hipStream_t st = b->ctx->stream;
    const size_t L = (size_t)b->B * b->out_seeds, M = (size_t)b->M, G = (size_t)b->Gmax, Rm = (size_t)b->Rmax;
    Staging &stage = b->ctx->staging;
    std::vector<unsigned char> plain;
    if (b->in_scratch) {
        plain.resize(b->win_finish);
    } else {
        if (b->win_finish > stage.n) HIP_TRY(hipStreamSynchronize(st));  // the inputs may still be on their way out of it
        HIP_TRY(stage.ensure(b->win_finish));
    }
    unsigned char *host = b->in_scratch ? plain.data() : stage.p;
    StreamWait copies(st);
    HIP_TRY(hipMemcpyAsync(host, b->win_out.p, b->win_finish, hipMemcpyDeviceToHost, st));
    if (wr && Rm > 0) {
        HIP_TRY(hipMemcpyAsync(out->finish, b->win_out.p + b->win_finish, sizeof(double) * L * Rm, hipMemcpyDeviceToHost, st));
        HIP_TRY(hipMemcpyAsync(out->good, b->win_out.p + b->win_good, L * Rm, hipMemcpyDeviceToHost, st));
    }
    HIP_TRY(copies.now());
    const int32_t *ng = reinterpret_cast<const int32_t *>(host);
    for (size_t l = 0; l < L; ++l) out->n_good[l] = ng[l];
    std::memcpy(out->latency_sum, host + b->win_lat_sum, sizeof(double) * L);
    if (out->status) std::memset(out->status, 0, sizeof(int32_t) * L);
    if (wm) {
        std::memcpy(out->model_num_good, host + b->win_model, sizeof(int32_t) * L * M);
        for (size_t l = 0; l < L; ++l)
            std::memcpy(out->model_num_requests + l * M,
                        b->wl_model_requests[(size_t)(b->paired ? b->stream_of[l] : (int32_t)(l / (size_t)b->B))].data(), sizeof(int32_t) * M);
    }
    if (wg) {
        std::memcpy(out->group_num_requests, host + b->win_group, sizeof(int32_t) * L * G);
        std::memcpy(out->group_num_good, host + b->win_group + sizeof(int32_t) * L * G, sizeof(int32_t) * L * G);
    }
    if (!b->in_scratch) stage.trim();
    return MMSIM_OK;
}

}  // namespace mmsim
