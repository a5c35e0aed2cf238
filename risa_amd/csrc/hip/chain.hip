// The whole per-frame chain on one device:
//   Attenuation -> Fan2Para -> Filter -> Backprojection (+ fused Masking)
// as RISA/example/main.cpp:95-134 wires the stages, without the per-stage
// host synchronisation of the reference (each stage there syncs its stream
// before handing the frame on, e.g. Backprojection.cu:203): launches are
// stream-ordered, and a captured hipGraph replays the launch sequence.
//
// PLAIN: frame by frame, FP32 in and out of every stage (FFT filter, FP32
//        backprojector; on the matrix cores its products are of FP16 hi + lo
//        operands, 22 bits, its sums FP32).  Groups of `per` consecutive
//        frames (up to 16, or 32; each stage runs once per group) are dealt
//        round-robin to `lanes` streams (own scratch buffers each) forked from
//        and joined back into the caller's stream, so lanes x per frames are in
//        flight -- the way the reference overlaps frames across its per-stage
//        threads.  Chains of at least 64
//        frames take groups of 32 and backproject a call on the matrix cores
//        (bp_split_kernel) where timing both at creation says that this is the
//        faster way for its number of frames: 256 frames of 512^2 x 1000 angles
//        4.29 ms a call, 6.67 with bp_linear_kernel; 256^2 x 500 stays with
//        the latter (125 us per 32 slices against 179).
// MIXED: groups of `per` consecutive frames (a multiple of 4, up to 32) dealt
//        to `lanes` streams the same way; per group the DFT-GEMM filter on
//        MFMA writes the FP16 sinogram in the 4-slice interleaved layout and
//        the FP16-sinogram / FP32-accumulate backprojection runs the group in
//        one launch, so one lane's front stages overlap the other's
//        backprojection.  Chains of at least 128 frames take groups of 64 and
//        backproject those of at least split_min frames on the matrix cores
//        (bp_f16_mfma_kernel, the same bits), where timing both at creation
//        finds that the faster way: 512 frames of 512^2 x 1000 angles 8.00 ms
//        a call, 8.95 with bp_linear_f16_kernel.
#include "device_common.h"

#include <cmath>
#include <map>
#include <tuple>
#include <vector>

int risa_filter_run_oop(risa_filter_t h, const float* in, float* out, long rows, hipStream_t s);
double risa_filter_l1(risa_filter_t h);
int risa_fan2para_gain(risa_fan2para_t h, double* gain);
extern "C" size_t risa_bp_split_bytes(risa_bp_t h);
extern "C" int risa_bp_autotune_f16_tile(risa_bp_t h, int slices);
extern "C" size_t risa_bp_f16_pack_bytes(risa_bp_t h);
extern "C" int risa_bp_tune_f16_packed(risa_bp_t h, hipStream_t s, int slices, int* min_slices);
extern "C" int risa_bp_run_f16_packed(risa_bp_t h, const uint16_t* sino_x4, float in_scale, int slices, void* packed,
                                      float* img, hipStream_t s);
extern "C" int risa_bp_tune_split(risa_bp_t h, hipStream_t s, int* shape, float cost[2]);
extern "C" int risa_bp_run_split(risa_bp_t h, int shape, const float* sino, float scale, int slices, void* packed, float* img,
                      hipStream_t s);

namespace {
constexpr float kF16SinoScale = 256.0f;   // FP16 filtered sinogram stores 256 * value
constexpr int kPlainLanes = 2;            // streams in PLAIN mode
constexpr int kPlainMaxPer = 16;          // frames per lane step of a PLAIN chain below 64 frames, at most
constexpr int kSplitPer = 32;             // and of 64 frames or more (also the split backprojector's slices)
constexpr int kMixedLanes = 2;            // streams in MIXED mode
constexpr int kMixedMaxPer = 32;          // frames per lane step in MIXED mode, at most (a multiple of 4)
constexpr int kPackPer = 64;              // and of a MIXED chain that backprojects groups on the matrix cores
}  // namespace

// Graph executables a chain keeps (one per buffer set and call shape); the
// least recently replayed one is released beyond this.
constexpr size_t kMaxGraphs = 128;

struct ChainGraph {
    hipGraphExec_t exec = nullptr;
    unsigned long long last_use = 0;
};

struct risa_chain_s {
    int device = 0;
    int mode = 0;
    int max_frames = 0;
    int lanes = 1;
    int per = 1;   // frames per lane step
    risa_geom g{};
    risa_attenuation_t att = nullptr;
    risa_fan2para_t f2p = nullptr;
    risa_filter_t filt = nullptr;
    risa_bp_t bp = nullptr;
    risa::DeviceBuffer<float> att_buf, par_buf, filt_buf;   // `per` frame slots per lane
    risa::DeviceBuffer<uint16_t> f16_buf;                   // MIXED: `per` slots per lane, x4 layout
    // Backprojection on the matrix cores (split_shape -1: none).  PLAIN: all
    // groups of a call or none (split_call), so that a frame's bits do not depend
    // on its place in the call, with tile shape split_shape and FP16 hi + lo
    // operands that hold filtered sample * split_scale, until the caller sets a
    // variant; split_cost: of a group of up to 16 and up to 32 frames, in frames of
    // the FP32 variant.  MIXED: groups of at least split_min frames, while the
    // FP16 variant is one whose bits that kernel has
    int split_shape = -1, split_min = 0;
    float split_cost[2] = {0.0f, 0.0f};
    float split_scale = 0.0f;
    risa::DeviceBuffer<char> split_buf;                     // packed sinograms, one launch per lane
    size_t split_bytes = 0;
    std::vector<hipStream_t> lane_streams;
    std::vector<hipEvent_t> lane_events;   // [0] fork, [1..lanes] joins
    std::map<std::tuple<const void*, const void*, int, std::vector<int32_t>>, ChainGraph> graphs;
    unsigned long long uses = 0;

    // A graph executable, event or stream must not be released while work
    // that uses it may still run: hipGraphLaunch returns before the replay
    // ends, and the caller's stream is not known here, so the whole device
    // is drained first.
    void drain() const
    {
        int prev = -1;
        if (hipGetDevice(&prev) != hipSuccess) return;
        if (prev != device) (void)hipSetDevice(device);
        (void)hipDeviceSynchronize();
        if (prev != device) (void)hipSetDevice(prev);
    }
    bool split_call(int frames) const;
    bool packed_group(int n) const;
    void release_graphs()
    {
        for (auto& kv : graphs) (void)hipGraphExecDestroy(kv.second.exec);
        graphs.clear();
    }
    ~risa_chain_s()
    {
        drain();
        release_graphs();
        for (hipEvent_t e : lane_events) (void)hipEventDestroy(e);
        for (hipStream_t s : lane_streams) (void)hipStreamDestroy(s);
        if (bp) risa_hip_bp_destroy(bp);
        if (filt) risa_hip_filter_destroy(filt);
        if (f2p) risa_hip_fan2para_destroy(f2p);
        if (att) risa_hip_attenuation_destroy(att);
    }
};

using namespace risa;

// Whether a plain call takes no longer on the matrix cores, tail included, than
// with the FP32 variant.  512^2 x 1000 angles, 32 / 48 / 65 frames on the matrix
// cores 630 / 1030 / 1580 us, 32 / 33 with the variant 890 / 1060; with only the
// full groups on the matrix cores 65 took 1370.
bool risa_chain_s::split_call(int frames) const
{
    if (mode != RISA_CHAIN_PLAIN || split_shape < 0) return false;
    const int tail = frames % kSplitPer;
    const float last = tail == 0 ? 0.0f : split_cost[tail > kSplitPer / 2];
    return (float)(frames / kSplitPer) * split_cost[1] + last <= (float)frames;
}
bool risa_chain_s::packed_group(int n) const
{
    return mode == RISA_CHAIN_MIXED && split_shape >= 0 && n >= split_min && risa_bp_f16_pack_bytes(bp) > 0;
}

static void ok(int rc)
{
    if (rc != RISA_OK) fail(rc, "%s", risa_last_error());
}

// The power of two that brings every filtered sample of the chain into the
// FP16 range, from what the stages can produce: counts of 0 .. 65535 over the
// given references, the rebinning's weights and the filter's absolute sum.
// 0 when there is none (references that are not finite).
static float split_scale(risa_chain_t h, const float* avg_ref, const float* avg_dark)
{
    const risa_geom& g = h->g;
    const long Df = g.numberOfFanDetectors, n = Df * g.numberOfFanProjections;
    const float tiny = 1.0e-5f;
    float lo = INFINITY, hi = 0.0f, num = tiny;   // the denominators' range, the largest numerator
    for (int k = 0; k < g.numberOfPlanes; k++)
        for (long e = 0; e < n; e++) {
            const float dark = avg_dark[k * Df + e % Df], den = std::max(avg_ref[k * n + e] - dark, tiny);
            if (!(std::fabs(dark) <= 1e30f) || !(den <= 1e30f) || std::isnan(avg_ref[k * n + e])) return 0.0f;
            lo = std::min(lo, den);
            hi = std::max(hi, den);
            num = std::max(num, 65535.0f - dark);
        }
    double gain = 0.0;
    ok(risa_fan2para_gain(h->f2p, &gain));
    const double att = std::max(std::fabs(std::log((double)num / lo)), std::fabs(std::log((double)tiny / hi)));
    const double bound = 1.001 * att * gain * risa_filter_l1(h->filt);
    // counts over a flat field give 10 .. 100; with a bound of 4000 the operands'
    // step (2^-25 / scale) is still 2e-6 of samples of 1e-3, far below the error
    // of their sums, beyond it is not
    if (!(bound > 0.0) || !(bound < 4000.0)) return 0.0f;
    return (float)std::exp2(std::floor(std::log2(65000.0 / bound)));
}

extern "C" int risa_hip_chain_create(const risa_geom* g, const float* avg_ref, const float* avg_dark, int device,
                                     int mode, int max_frames, risa_chain_t* out)
{
    return guarded("risa_hip_chain_create", [&] {
        if (!g || !avg_ref || !avg_dark || !out || max_frames <= 0) fail(RISA_ERR_ARG, "bad argument");
        if (mode != RISA_CHAIN_PLAIN && mode != RISA_CHAIN_MIXED) fail(RISA_ERR_ARG, "unknown chain mode");
        DeviceGuard dg(device);
        auto h = new risa_chain_s();
        try {
            h->device = device;
            h->mode = mode;
            h->max_frames = max_frames;
            h->g = *g;
            ok(risa_hip_attenuation_create(g, avg_ref, avg_dark, device, &h->att));
            ok(risa_hip_fan2para_create(g, device, &h->f2p));
            ok(risa_hip_filter_create(g, device, mode == RISA_CHAIN_MIXED ? RISA_FILTER_MODE_GEMM_SPLIT : RISA_FILTER_MODE_FFT32,
                                      &h->filt));
            ok(risa_hip_bp_create(g, device, &h->bp));
            const size_t fan = (size_t)g->numberOfFanDetectors * g->numberOfFanProjections;
            const size_t par = (size_t)g->numberOfParallelDetectors * g->numberOfParallelProjections;
            if (mode == RISA_CHAIN_PLAIN) {
                // one group while it holds every frame (8 frames of 256^2 x 500 /
                // 384^2 x 700 / 512^2 x 1000 / 560^2 x 300: 96 / 181 / 305 / 129
                // us, 124 / 237 / 321 / 132 as two groups of 4 in two lanes; 2 to
                // 16 frames of these 1.02 to 1.64 times faster), 32 to a group
                // from 64 frames on (100 frames of 256^2 x 500 539 us, 588 with 16)
                h->lanes = max_frames > kPlainMaxPer ? kPlainLanes : 1;
                h->per = std::min(max_frames >= kPlainLanes * kSplitPer ? kSplitPer : kPlainMaxPer, max_frames);
                if (max_frames >= kPlainLanes * kSplitPer && (h->split_bytes = risa_bp_split_bytes(h->bp)) > 0 &&
                    (h->split_scale = split_scale(h, avg_ref, avg_dark)) > 0.0f) {
                    ok(risa_hip_bp_autotune_batch(h->bp, kPlainLanes * kPlainMaxPer, nullptr));
                    ok(risa_bp_tune_split(h->bp, nullptr, &h->split_shape, h->split_cost));
                    if (h->split_cost[1] <= (float)kSplitPer) {
                        h->split_bytes = (h->split_bytes + 255) / 256 * 256;
                        h->split_buf.resize(h->split_bytes * h->lanes);
                    } else {
                        h->split_shape = -1;
                    }
                }
                const size_t slots = (size_t)h->lanes * h->per;
                h->att_buf.resize(fan * slots);
                h->par_buf.resize(par * slots);
                h->filt_buf.resize(par * slots);
            } else {
                // groups of a multiple of 4 frames: whole x4 slice groups per
                // lane; as few as hold the frames (512^2 x 1000, 8 frames: one
                // group 245 us, two of 4 in two lanes 292; 48 frames as 32 + 16
                // 978, as 24 + 24 1160)
                h->per = std::min(kMixedMaxPer, (max_frames + 3) / 4 * 4);
                // the tile shape (and with it the results) as timed for half of the
                // frames per lane, the variant for the group
                const int half = (max_frames + kMixedLanes - 1) / kMixedLanes;
                ok(risa_hip_bp_autotune_f16(h->bp, std::min(kMixedMaxPer, (half + 3) / 4 * 4), nullptr));
                ok(risa_bp_autotune_f16_tile(h->bp, h->per));
                if (max_frames >= kMixedLanes * kPackPer) {
                    ok(risa_bp_tune_f16_packed(h->bp, nullptr, h->per, &h->split_min));
                    if (h->split_min <= kPackPer) {
                        h->per = kPackPer;
                        h->split_shape = 0;
                        h->split_bytes = (risa_bp_f16_pack_bytes(h->bp) + 255) / 256 * 256;
                        h->split_buf.resize(h->split_bytes * kMixedLanes);
                    }
                }
                h->lanes = std::min(kMixedLanes, (max_frames + h->per - 1) / h->per);
                const size_t slots = (size_t)h->lanes * h->per;
                h->att_buf.resize(fan * slots);
                h->par_buf.resize(par * slots);
                h->f16_buf.resize(par * slots);   // x4 layout: per / 4 groups of 4 slices per lane
            }
            for (int k = 0; k < h->lanes; k++) {
                hipStream_t s;
                RISA_HIP_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
                h->lane_streams.push_back(s);
            }
            for (int k = 0; k <= h->lanes; k++) {
                hipEvent_t e;
                RISA_HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
                h->lane_events.push_back(e);
            }
            // backprojector tile shape, timed at the frames the chain keeps
            // in flight (plain: lanes x per slices, two-slice tiles included
            // when per > 1) or at a lane step's batch (mixed); timing the chain
            // itself per variant, eagerly, proved too noisy to rank the closest
            // shapes
            if (mode == RISA_CHAIN_PLAIN) {
                if (h->split_cost[1] > 0.0f) {
                    // tuned above
                } else if (h->per > 1) ok(risa_hip_bp_autotune_batch(h->bp, std::min(kPlainLanes * kPlainMaxPer, h->lanes * h->per), nullptr));
                else ok(risa_hip_bp_autotune_slices(h->bp, h->lanes, nullptr));
            }
            RISA_HIP_CHECK(hipDeviceSynchronize());
        } catch (...) {
            delete h;
            throw;
        }
        *out = h;
    });
}

static void enqueue(risa_chain_t h, const uint16_t* raw, const int32_t* planes, int frames, float* img, hipStream_t s)
{
    const risa_geom& g = h->g;
    const size_t fan = (size_t)g.numberOfFanDetectors * g.numberOfFanProjections;
    const size_t par = (size_t)g.numberOfParallelDetectors * g.numberOfParallelProjections;
    const size_t out = (size_t)g.numberOfPixels * g.numberOfPixels;
    const int per = h->per;
    const int groups = (frames + per - 1) / per;
    const int lanes = std::min(h->lanes, groups);
    const bool matrix = h->split_call(frames);
    RISA_HIP_CHECK(hipEventRecord(h->lane_events[0], s));
    for (int k = 0; k < lanes; k++) RISA_HIP_CHECK(hipStreamWaitEvent(h->lane_streams[k], h->lane_events[0], 0));
    for (int q = 0; q < groups; q++) {
        const int k = q % lanes, f = q * per, n = std::min(per, frames - f);
        hipStream_t ls = h->lane_streams[k];
        float* att = h->att_buf.ptr + (size_t)k * per * fan;
        float* pb = h->par_buf.ptr + (size_t)k * per * par;
        if (h->mode == RISA_CHAIN_PLAIN) {
            float* fb = h->filt_buf.ptr + (size_t)k * per * par;
            if (n == 1) {
                ok(risa_hip_attenuation_run(h->att, raw + f * fan, planes[f], att, ls));
                ok(risa_hip_fan2para_run(h->f2p, att, planes[f], pb, ls));
            } else {
                ok(risa_hip_attenuation_run_batch(h->att, raw + f * fan, planes + f, n, att, ls));
                ok(risa_hip_fan2para_run_batch(h->f2p, att, planes + f, n, pb, ls));
            }
            ok(risa_filter_run_oop(h->filt, pb, fb, (long)n * g.numberOfParallelProjections, ls));
            if (matrix)
                ok(risa_bp_run_split(h->bp, h->split_shape, fb, h->split_scale, n, h->split_buf.ptr + k * h->split_bytes,
                                     img + f * out, ls));
            else if (n == 1)
                ok(risa_hip_bp_run(h->bp, fb, img + f * out, ls));
            else
                ok(risa_hip_bp_run_batch(h->bp, fb, n, img + f * out, ls));
        } else {
            uint16_t* hb = h->f16_buf.ptr + (size_t)k * per * par;
            ok(risa_hip_attenuation_run_batch(h->att, raw + f * fan, planes + f, n, att, ls));
            ok(risa_hip_fan2para_run_batch(h->f2p, att, planes + f, n, pb, ls));
            ok(risa_hip_filter_run_f16x4(h->filt, pb, hb, n, kF16SinoScale, ls));
            if (h->packed_group(n))
                ok(risa_bp_run_f16_packed(h->bp, hb, kF16SinoScale, n, h->split_buf.ptr + k * h->split_bytes,
                                          img + f * out, ls));
            else
                ok(risa_hip_bp_run_f16x4(h->bp, hb, kF16SinoScale, n, img + f * out, ls));
        }
    }
    for (int k = 0; k < lanes; k++) {
        RISA_HIP_CHECK(hipEventRecord(h->lane_events[k + 1], h->lane_streams[k]));
        RISA_HIP_CHECK(hipStreamWaitEvent(s, h->lane_events[k + 1], 0));
    }
}

extern "C" int risa_hip_chain_run(risa_chain_t h, const uint16_t* raw, const int32_t* planes, int frames, float* img,
                                  int use_graph, void* stream)
{
    return guarded("risa_hip_chain_run", [&] {
        if (!h || !raw || !planes || !img || frames < 0) fail(RISA_ERR_ARG, "bad argument");
        if (frames > h->max_frames) fail(RISA_ERR_ARG, "frames (%d) exceeds max_frames (%d)", frames, h->max_frames);
        if (frames == 0) return;
        for (int f = 0; f < frames; f++)
            if (planes[f] < 0 || planes[f] >= h->g.numberOfPlanes) fail(RISA_ERR_ARG, "plane out of range");
        hipStream_t s = as_stream(stream);
        if (!use_graph) {
            enqueue(h, raw, planes, frames, img, s);
            return;
        }
        if (!s) fail(RISA_ERR_ARG, "graph replay needs a non-null stream");
        auto key = std::make_tuple((const void*)raw, (const void*)img, frames, std::vector<int32_t>(planes, planes + frames));
        auto it = h->graphs.find(key);
        if (it == h->graphs.end()) {
            if (h->graphs.size() >= kMaxGraphs) {
                // release the least recently replayed executable, once no
                // replay of it can still be running
                auto lru = h->graphs.begin();
                for (auto jt = h->graphs.begin(); jt != h->graphs.end(); ++jt)
                    if (jt->second.last_use < lru->second.last_use) lru = jt;
                DeviceGuard dg(h->device);
                RISA_HIP_CHECK(hipDeviceSynchronize());
                RISA_HIP_CHECK(hipGraphExecDestroy(lru->second.exec));
                h->graphs.erase(lru);
            }
            hipGraph_t graph;
            RISA_HIP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
            try {
                enqueue(h, raw, planes, frames, img, s);
            } catch (...) {
                hipGraph_t dummy = nullptr;
                if (hipStreamEndCapture(s, &dummy) == hipSuccess && dummy) (void)hipGraphDestroy(dummy);
                throw;
            }
            RISA_HIP_CHECK(hipStreamEndCapture(s, &graph));
            hipGraphExec_t exec;
            const hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
            (void)hipGraphDestroy(graph);
            RISA_HIP_CHECK(ie);
            it = h->graphs.emplace(key, ChainGraph{exec, 0}).first;
        }
        it->second.last_use = ++h->uses;
        RISA_HIP_CHECK(hipGraphLaunch(it->second.exec, s));
    });
}

extern "C" int risa_hip_chain_intermediate(risa_chain_t h, int which, const void** ptr)
{
    return guarded("risa_hip_chain_intermediate", [&] {
        if (!h || !ptr) fail(RISA_ERR_ARG, "null argument");
        switch (which) {
            case 0: *ptr = h->att_buf.ptr; break;
            case 1: *ptr = h->par_buf.ptr; break;
            case 2: *ptr = h->mode == RISA_CHAIN_PLAIN ? (const void*)h->filt_buf.ptr : (const void*)h->f16_buf.ptr; break;
            default: fail(RISA_ERR_ARG, "which must be 0, 1 or 2");
        }
    });
}

// Captured graphs hold the launches of the layout and variant they were
// captured with: a change drains the device, releases them, and the next
// graph run captures anew.
extern "C" int risa_hip_chain_set_input_layout(risa_chain_t h, int layout)
{
    return guarded("risa_hip_chain_set_input_layout", [&] {
        if (!h) fail(RISA_ERR_ARG, "null handle");
        int cur = 0;
        ok(risa_hip_attenuation_get_input_layout(h->att, &cur));
        if (cur == layout) return;
        h->drain();
        h->release_graphs();
        ok(risa_hip_attenuation_set_input_layout(h->att, layout));
    });
}

extern "C" int risa_hip_chain_set_variant(risa_chain_t h, int variant)
{
    return guarded("risa_hip_chain_set_variant", [&] {
        if (!h) fail(RISA_ERR_ARG, "null handle");
        int cur = 0;
        ok(risa_hip_bp_get_variant(h->bp, &cur));
        // a plain chain runs a variant that was set for every group, also one
        // that it reported itself
        const bool pins = h->mode == RISA_CHAIN_PLAIN && h->split_shape >= 0;
        if (cur == variant && !pins) return;
        h->drain();
        h->release_graphs();
        ok(risa_hip_bp_set_variant(h->bp, variant));
        if (pins) h->split_shape = -1;
    });
}

extern "C" int risa_hip_chain_on_matrix_cores(risa_chain_t h, int frames, int* yes)
{
    return guarded("risa_hip_chain_on_matrix_cores", [&] {
        if (!h || !yes || frames < 1) fail(RISA_ERR_ARG, "bad argument");
        *yes = h->split_call(frames) || h->packed_group(std::min(frames, h->per)) ? 1 : 0;
    });
}

/* Graph executables the chain holds (tooling; no reference counterpart). */
extern "C" int risa_hip_chain_graph_count(risa_chain_t h, int* count)
{
    return guarded("risa_hip_chain_graph_count", [&] {
        if (!h || !count) fail(RISA_ERR_ARG, "null argument");
        *count = (int)h->graphs.size();
    });
}

extern "C" int risa_hip_chain_get_variant(risa_chain_t h, int* variant)
{
    return guarded("risa_hip_chain_get_variant", [&] {
        if (!h || !variant) fail(RISA_ERR_ARG, "null argument");
        ok(risa_hip_bp_get_variant(h->bp, variant));
    });
}

extern "C" int risa_hip_chain_destroy(risa_chain_t h)
{
    return guarded("risa_hip_chain_destroy", [&] { delete h; });
}
