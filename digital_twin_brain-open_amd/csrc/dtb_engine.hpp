// dtb_engine.hpp -- C++ host runtime: device buffers, instances and the
// step engine that drives the gfx950 kernels.
//
// Vocabulary follows the reference host library:
//   DataAllocator<T>  include/data_allocator.hpp:8-38 (device buffer + host
//                     mirror, zero-filled, explicit copies)
//   Weights/DataType  include/weights.hpp:14-94 (two values per synapse)
//   Instance          one BrainBlock<float,float2> (include/block.hpp:21-889)
//   Engine            the per-GPU step loop of snn_run
//                     (tools/dist_simulator.cpp:2072-2315), here able to step
//                     many instances in one launch pair.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <memory>
#include <stdexcept>
#include <string>
#include <unordered_set>
#include <vector>

#include "dtb_kernels.hpp"
#include "dtb_types.hpp"

namespace dtb {

// Status codes: 0-5 are protos/snn.proto:44-51 SnnStatus.
enum StatusCode : int {
    kOk = 0,
    kInvalidParameter = 1,
    kUnsetSampleFailure = 2,
    kUnsupported = 3,
    kNotEnableMetric = 4,
    kInvalidNetwork = 5,
    kHipError = 100,
    kOutOfMemory = 101,
    kNoDevice = 102,
    kInternal = 103,
};

struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

void hip_check(hipError_t e, const char *what, const char *file, int line);
#define DTB_HIP(x) ::dtb::hip_check((x), #x, __FILE__, __LINE__)

// Property-matrix columns (src/configuration.cpp:1778-2156).
enum Col : int {
    kColNoiseRate = 0,
    kColBlocked = 1,
    kColIExt = 2,
    kColSubIdx = 3,
    kColC = 4,
    kColTRef = 5,
    kColGLeak = 6,
    kColVLeak = 7,
    kColVTh = 8,
    kColVReset = 9,
    kColGU = 10,
    kColVU = 14,
    kColTauU = 18,
    kNumCols = 22,
};

// include/stage.hpp:320-341 == protos/snn.proto:94-115.
enum PropType : int {
    EXT_STIMULI_I = 0,
    MEMBRANE_C = 1,
    REF_T = 2,
    LEAKAGE_G = 3,
    LEAKAGE_V = 4,
    THRESHOLD_V = 5,
    RESET_V = 6,
    CONDUCT_G_AMPA = 7,
    CONDUCT_G_NMDA = 8,
    CONDUCT_G_GABAa = 9,
    CONDUCT_G_GABAb = 10,
    MEMBRANE_V_AMPA = 11,
    MEMBRANE_V_NMDA = 12,
    MEMBRANE_V_GABAa = 13,
    MEMBRANE_V_GABAb = 14,
    TAO_AMPA = 15,
    TAO_NMDA = 16,
    TAO_GABAa = 17,
    TAO_GABAb = 18,
    NOISE_RATE = 19,
    kNumPropTypes = 20,
};

int prop_type_column(int prop);   // PropType -> property column, -1 if unknown

// include/weights.hpp:14-21
enum DataType : int { DOUBLE = 0, FLOAT = 1, FLOAT16 = 2, INT32 = 3, INT8 = 4 };
size_t data_size(DataType t);

// Device memory that stays with the library once freed (dtb_devmem.cpp).
namespace devmem {
void *alloc(size_t bytes);           // on the current device
void release(void *p);               // block from alloc; may still be in use by queued work
void reserve(size_t bytes);          // keeps at least this much for blocks of 1 MB and more
void trim();                         // returns all unused memory to the runtime
size_t cached_bytes(int device);     // bytes held in the cache
// While one is alive on a thread, alloc on that thread (and HostStage::reserve)
// throws instead of taking memory (the entry points that promise not to
// allocate).
struct NoAlloc {
    NoAlloc();
    ~NoAlloc();
    static bool active();   // on this thread
    NoAlloc(const NoAlloc &) = delete;
    NoAlloc &operator=(const NoAlloc &) = delete;
};
}  // namespace devmem

// The static device array of dtb_run_noalloc (kScratchBytes) on the current
// device: its address, looked up once per device (dtb_noalloc.hip).
void *scratch_address(int device);
// Zeroes `bytes` (a multiple of 4) at p with a fill kernel.
hipError_t launch_zero_words(void *p, size_t bytes, hipStream_t stream);
// Per-population means of a recording: cnt[q] = non-blocked neurons of
// population q (counted on the device from the instance's blocked flags and
// population table), then out[k][r][q] = (float)((double)sums[r][q][k] *
// 2^-24 / cnt[q]) for every field k with out[k] != null.
hipError_t launch_stat_means(const uint8_t *blocked, const PopDev *pops, uint32_t npop, const long long *sums,
                             uint32_t rows, unsigned long long *cnt, float *const *out, hipStream_t stream);

// Device buffer with a lazily created, zero-filled host mirror.
template <typename T>
class DataAllocator {
public:
    explicit DataAllocator(size_t count = 0) { resize(count); }
    ~DataAllocator() { release(); }
    DataAllocator(const DataAllocator &) = delete;
    DataAllocator &operator=(const DataAllocator &) = delete;

    void resize(size_t count)
    {
        if (count == count_)
            return;
        release();
        count_ = count;
    }
    size_t count() const { return count_; }
    size_t size() const { return count_ * sizeof(T); }

    const T *gpu_data() { return mutable_gpu_data(); }
    T *mutable_gpu_data()
    {
        if (gpu_ == nullptr && count_ > 0) {
            gpu_ = static_cast<T *>(devmem::alloc(size()));
            // The zero fill runs on the null stream, which does not order
            // with the engine's non-blocking stream: wait for it here so a
            // later upload on the engine stream cannot be overwritten.
            DTB_HIP(hipMemsetAsync(gpu_, 0, size(), nullptr));
            DTB_HIP(hipStreamSynchronize(nullptr));
        }
        return gpu_;
    }
    // The device memory, not cleared when it is taken: for a buffer of which
    // nothing is read that a kernel has not written.
    T *gpu_uncleared()
    {
        if (gpu_ == nullptr && count_ > 0)
            gpu_ = static_cast<T *>(devmem::alloc(size()));
        return gpu_;
    }
    const T *cpu_data() { return mutable_cpu_data(); }
    T *mutable_cpu_data()
    {
        if (cpu_.size() != count_)
            cpu_.assign(count_, T{});
        return cpu_.data();
    }
    void to_gpu(hipStream_t s)
    {
        if (count_ == 0)
            return;
        DTB_HIP(hipMemcpyAsync(mutable_gpu_data(), mutable_cpu_data(), size(), hipMemcpyHostToDevice, s));
    }
    void to_cpu(hipStream_t s)
    {
        if (count_ == 0)
            return;
        DTB_HIP(hipMemcpyAsync(mutable_cpu_data(), mutable_gpu_data(), size(), hipMemcpyDeviceToHost, s));
    }
    void upload(const T *src, size_t n, hipStream_t s)
    {
        if (n > count_)
            throw Error(kInvalidParameter, "upload larger than buffer");
        if (n == 0)
            return;
        DTB_HIP(hipMemcpyAsync(mutable_gpu_data(), src, n * sizeof(T), hipMemcpyHostToDevice, s));
    }
    void download(T *dst, size_t n, hipStream_t s)
    {
        if (n > count_)
            throw Error(kInvalidParameter, "download larger than buffer");
        if (n == 0)
            return;
        DTB_HIP(hipMemcpyAsync(dst, mutable_gpu_data(), n * sizeof(T), hipMemcpyDeviceToHost, s));
    }
    void release_cpu() { std::vector<T>().swap(cpu_); }

private:
    void release()
    {
        devmem::release(gpu_);
        gpu_ = nullptr;
        std::vector<T>().swap(cpu_);
        count_ = 0;
    }
    size_t count_ = 0;
    T *gpu_ = nullptr;
    std::vector<T> cpu_;
};

// Pinned host memory that kernels read and write in place: what a call
// uploads (its tables) and returns (its records, a small state), without a
// copy call each.  Grows; freed with its owner.
class HostStage {
public:
    HostStage() = default;
    ~HostStage() { release(); }
    HostStage(const HostStage &) = delete;
    HostStage &operator=(const HostStage &) = delete;
    // At least `bytes`; what it held before is lost when it grows, so no
    // kernel may be using it.  Under NoAlloc it throws instead of growing (a
    // caller inside a capture may make no allocating runtime call).
    unsigned char *reserve(size_t bytes)
    {
        if (bytes > cap_) {
            if (devmem::NoAlloc::active())
                throw Error(kInvalidParameter, "this call allocates no memory, but needs " + std::to_string(bytes) +
                                                   " bytes of pinned host memory first (build the tables with one "
                                                   "dtb_run or dtb_engine_run)");
            release();
            DTB_HIP(hipHostMalloc(&p_, bytes, hipHostMallocDefault));
            cap_ = bytes;
        }
        return static_cast<unsigned char *>(p_);
    }

private:
    void release()
    {
        if (p_ != nullptr)
            (void)hipHostFree(p_);
        p_ = nullptr;
        cap_ = 0;
    }
    void *p_ = nullptr;
    size_t cap_ = 0;
};
// A call's results are taken through at most this much pinned memory at a time.
constexpr size_t kCallStageBytes = (size_t)1 << 20;

// Host description of a network in the reference layout: property matrix
// [n][22] and a presynaptic-major CSR whose synapses carry a weight pair and a
// channel bit (0: AMPA/NMDA pair, 1: GABA_A/GABA_B pair), bit-packed in
// 32-bit words as in presynaptic_voltage.cpp:152.
struct NetworkHost {
    int64_t n = 0;
    const float *props = nullptr;
    int64_t nsyn = 0;
    const int64_t *rowptr = nullptr;
    const uint32_t *col = nullptr;
    const void *w = nullptr;            // [nsyn][2] in format wfmt
    const uint32_t *kind_bits = nullptr;  // [ceil(nsyn/32)]
    uint32_t wfmt = kWeightF32;         // kWeightF32 / kWeightF16 / kWeightU8
};

// Per-run options (protos/snn.proto:63-77 RunRequest).
struct RunOptions {
    int32_t t_steps = 1;
    bool use_ou = true;
    bool record_freq = false;
    bool record_samples = false;
};

class Engine;

// One simulated block.
// A fan-out network generated on the device (gen_fanout / launch_gen_fanout).
struct FanoutSpec {
    int64_t n = 0;
    uint32_t K = 0;
    uint64_t net_seed = 0;
    float g_ui[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t sub_base = 0;
};

class Instance {
public:
    Instance(const NetworkHost &net, float dt, uint64_t seed, hipStream_t stream);
    // The network is generated in device memory (no host copy of the
    // synapses, nothing crosses PCIe but the property matrix).
    Instance(const FanoutSpec &spec, float dt, uint64_t seed, hipStream_t stream);
    ~Instance();

    uint32_t n() const { return n_; }
    int64_t nsyn() const { return nsyn_; }
    uint32_t weight_format() const { return wfmt_; }
    uint32_t npop() const { return (uint32_t)pop_ids_.size(); }
    const std::vector<uint32_t> &pop_ids() const { return pop_ids_; }
    const std::vector<uint32_t> &pop_begin() const { return pop_begin_; }
    float dt() const { return dt_; }
    uint64_t seed() const { return seed_; }
    int32_t t_steps() const { return t_steps_; }
    bool use_ou() const { return use_ou_; }

    // extern_stimuli.cpp / block.cpp:222-281 (set_I_ou_current_param).
    void set_ou(const uint32_t *brain_ids, const float *mean, const float *sigma, const float *tau, size_t n,
                hipStream_t s);
    // property.cpp:57-466 (update_props / assign_prop_cols / update_prop_cols).
    void update_props(const uint32_t *neuron_ids, const uint32_t *prop_ids, const float *vals, size_t n,
                      hipStream_t s);
    void update_prop_cols(const uint32_t *prop_ids, const uint32_t *brain_ids, const float *vals, size_t n,
                          bool assign, hipStream_t s);
    // Per-population Gamma(concentration, rate) resampling of properties:
    // draw stream = (seed, call count of this instance, neuron).
    void gamma_prop_cols(const uint32_t *prop_ids, const uint32_t *brain_ids, const float *alpha, const float *beta,
                         size_t n, hipStream_t s);
    // The [n][22] property matrix as updated so far.
    void read_props(float *out) const;
    void set_samples(const uint32_t *ids, size_t n);
    const std::vector<uint32_t> &samples() const { return samples_; }

    // Configure t_steps / OU mode for the next run (recomputes substep decays).
    bool configure_run(int32_t t_steps, bool use_ou, hipStream_t s);
    // Recording window of `steps` rows starting at the current step;
    // stat_mask selects per-population means (kStatV | kStatI | kStatReceptor).
    // step0: the step index (step()).
    void begin_record(int64_t step0, int64_t steps, bool freq, bool samples, uint32_t stat_mask, hipStream_t s);
    // The same window recorded into caller-provided device buffers (no
    // allocation): counts [steps][npop] and sums [steps][npop][kStatFields]
    // are zeroed here; the sample rows [steps][nsample] need no clearing.
    struct RecordBuffers {
        uint32_t *counts;
        long long *stat;
        uint8_t *spike;
        float *v, *isyn, *iou;
    };
    void begin_record_at(int64_t steps, bool freq, bool samples, uint32_t stat_mask, const RecordBuffers &b,
                         hipStream_t s);
    void end_record();
    // Device descriptors the statistics need (the instance's blocked flags
    // and population table).
    const uint8_t *blocked_dev() { return blocked_.gpu_data(); }
    const PopDev *pops_dev() { return pops_.gpu_data(); }
    uint32_t stat_mask() const { return rec_stat_mask_; }
    // means: [6] arrays [steps][npop] (vmean, imean, AMPA, NMDA, GABA_A,
    // GABA_B), any may be null.
    void fetch_record(HostStage &stage, uint32_t *freq, uint8_t *spike, float *v, float *isyn, float *iou, float *const *means,
                      hipStream_t s);

    // Reference-visible state after the last completed step: V, refractory
    // counter, spike flag, emitted flag, i_ou, J[4] (pending delta folded
    // in), I_syn (without i_ou).
    void read_state(HostStage &stage, float *V, int32_t *t, uint8_t *f, uint8_t *emitted, float *iou, float *J, float *isyn,
                    hipStream_t s);
    void write_state(HostStage &stage, const float *V, const int32_t *t, const uint8_t *f, const float *iou, const float *J,
                     hipStream_t s);
    // The step index is kept in two device slots (read and written by
    // alternating launch parities); the current step is the larger one.
    int64_t step(hipStream_t s);
    void set_step(int64_t step, hipStream_t s);
    void counters(int64_t *step, uint64_t *events, uint64_t *spikes, hipStream_t s);

    // Kernel descriptor; `gather`: propagate by gather (ensure_gather first);
    // `direct`: by direct propagation (ensure_direct first);
    // defer_min > 0 with the in-edges built: pull propagation (a tile with
    // at least defer_min emitted rows defers them to the pull).
    // `passes`: binning by k_bin (ensure_passes first).
    InstDev dev(uint32_t tile_base, bool gather, bool direct, bool pull, uint32_t defer_min, bool passes);
    // Descriptor of tile t for the step kernels; inst: the device address of
    // the instance's descriptor `d`, idx its index; pop0: population of the
    // tile's first neuron; qoff, qcap: its queue.
    TileDesc tile_desc(uint32_t t, const InstDev &d, const InstDev *inst, uint32_t idx, uint32_t pop0, uint64_t qoff,
                       uint32_t qcap);
    // Distinct parameter records (classes); n() when stored per neuron.
    uint32_t param_classes() const { return (uint32_t)prm_.count(); }
    SampleRecDev sample_rec();
    // Synapses whose target lies in tile `tile` (2^kTileBits neurons): the
    // exact queue bound of the binning.
    uint32_t tile_synapses(uint32_t tile) const;
    // Zeroes both spill accumulators (the queues of this instance were
    // cleared).
    void clear_spill(hipStream_t s);
    // Propagation queues of `slots` entries per parity (grow-only; the
    // contents need no initialisation: only the first `count` entries of a
    // tile's queue are ever read).
    void ensure_queue(uint64_t slots);
    // Mean over rows of the fraction of this instance's tiles that the row's
    // synapses reach (tile segments of the row / tiles).
    double row_coverage() const { return row_coverage_; }
    // (Row, tile) pairs of all rows that the row kSharingDistance neurons on
    // reaches too, estimated from kSharingRows rows.
    double shared_segments() const { return shared_segments_; }

    // Gather propagation (k_gather): possible when every row is ordered by
    // target group, no row is longer than kGatherMaxRow and the group offsets
    // ([n][ngroups + 1] x 2 bytes) are no larger than the synapse arrays.
    bool gather_allowed() const { return gather_ok_; }
    // Mean over rows of the fraction of the groups of 2^kGroupBits neurons
    // that the row reaches.
    double group_coverage() const { return group_coverage_; }
    uint32_t ngroups(uint32_t bits = kGroupBits) const { return (n_ + (1u << bits) - 1) >> bits; }
    // Neurons per group of k_gather (log2): 2^kGroupBits, or fewer to get
    // kGatherGroups groups, where rows are ordered by tile and the offsets of
    // the smaller groups keep to the same limit.
    uint32_t gather_bits() const { return gather_bits_; }
    // Rows per fired list (the tiles of one list hold at most this many).
    uint32_t fired_capacity() const;
    // Builds the group offsets and fired lists if not built yet.
    void ensure_gather(hipStream_t s);
    // Returns them (no table may still reference them).
    void release_gather();
    bool gather_built() const { return gather_built_; }
    // Empties both fired lists (checkpoint restore).
    void clear_fired(hipStream_t s);

    // Pull propagation: a copy of the synapses grouped by target tile (the
    // in-edges, 12 bytes per synapse), through which a tile whose queue
    // overflowed, or whose sources deferred their rows, takes its input.
    // Possible for instances of at most kPullMaxNeurons neurons.
    bool pull_allowed() const { return n_ <= kPullMaxNeurons && nsyn_ > 0; }
    // Device bytes ensure_pull allocates.
    uint64_t pull_bytes() const;
    uint64_t direct_bytes() const { return (uint64_t)n_ * ((n_ + kBlock - 1) / kBlock + 1u) * sizeof(uint16_t); }
    uint64_t pass_bytes() const { return (uint64_t)kFiredLists * passcap_ * sizeof(unsigned long long); }
    void ensure_pull(hipStream_t s);
    void release_pull();
    bool pull_built() const { return pull_built_; }
    // Forgets emitted and deferred rows (after the pending input was folded
    // or dropped).
    void clear_deferred(hipStream_t s);
    CopyWords deferred_words();   // the same as a launch_copy_words segment
    const int64_t *step_words() { return step_.gpu_data(); }   // [2], the larger one is the step index

    // Direct propagation: possible when every row is ordered by tile and at
    // most kGatherMaxRow long, the instance has at most kDirectMaxNeurons
    // neurons, the tile offsets ([n][ntiles + 1] x 2 bytes) are no larger
    // than the synapse arrays and a row has enough synapses for its lookups.
    bool direct_allowed() const { return direct_ok_; }
    void ensure_direct(hipStream_t s);
    // Pass lists of k_bin (InstDev::passes), long enough for a step in which
    // every neuron fires.
    void ensure_passes();
    void release_passes();
    bool passes_built() const { return passes_.count() != 0; }
    CopyWords pass_count_words();   // to clear the lists
    void release_direct() { tidx_.resize(0); }
    bool direct_built() const { return tidx_.count() != 0; }

private:
    void init_common(const float *props, float dt, uint64_t seed, hipStream_t s);
    void init_common(std::vector<float> &&props, float dt, uint64_t seed, hipStream_t s);
    void derive_params(hipStream_t s);
    void derive_pops(hipStream_t s);     // population table (OU factors) only
    void init_state(hipStream_t s);
    StateView state_view();
    // Plain device arrays for `count` neurons' state (read_state,
    // write_state), as many neurons as device memory holds, at most `count`.
    struct StateStage;
    void count_tile_synapses(const NetworkHost &net);
    uint32_t find_pop(uint32_t brain_id) const;

    uint32_t n_ = 0;
    int64_t nsyn_ = 0;
    float dt_ = 0.1f;
    uint64_t seed_ = 0;
    int32_t t_steps_ = 1;
    bool use_ou_ = true;

    std::vector<float> props_;           // host property matrix [n][22]
    std::vector<uint32_t> pop_ids_;      // brain id per population
    std::vector<uint32_t> pop_begin_;    // [npop+1]
    std::vector<uint8_t> ou_on_;
    std::vector<float> ou_mean_, ou_sigma_, ou_tau_;
    std::vector<uint32_t> samples_;

    DataAllocator<ParamRec> prm_;                      // parameter records per class
    DataAllocator<uint16_t> cls_;                      // parameter class per neuron
    bool dense_params_ = false;                        // one class per neuron
    DataAllocator<uint8_t> blocked_;
    DataAllocator<unsigned char> state_;               // [ntiles][kStateBytes]
    DataAllocator<float4> dlt_;
    DataAllocator<unsigned long long> spill_;      // [2][n][4] Q23.40
    DataAllocator<QSyn> queue_;                    // [2][qslots_] + kQueuePrefetch
    uint64_t qslots_ = 0;
    DataAllocator<int64_t> rowptr_;
    DataAllocator<uint32_t> col_;
    DataAllocator<uint8_t> w_;                     // [nsyn] weight pairs in format wfmt_
    uint32_t wfmt_ = kWeightF32;
    DataAllocator<PopDev> pops_;
    // [2] step index, [2] deferral stamps, padded to 16 words; then the
    // emitted and deferred rows, [2][ntiles][kBitWords]
    DataAllocator<int64_t> step_;
    static constexpr size_t kStepPad = 16;
    DataAllocator<unsigned long long> counters_;   // per wave: events, spikes
    // Records of the run, [steps][rec_slots_][stride]: counts per population,
    // and its sums ([npop][kStatFields]); the slots of a row are added up
    // when it is fetched.
    DataAllocator<uint32_t> rec_counts_;
    DataAllocator<long long> rec_stat_;
    size_t count_slots() const { return (size_t)rec_len_ * rec_slots_ * rec_cstride_; }
    size_t stat_slots() const { return (size_t)rec_len_ * rec_slots_ * rec_sstride_; }
    uint32_t rec_slots_ = 1, rec_cstride_ = 0, rec_sstride_ = 0;
    void layout_record(int64_t steps, bool freq, bool stat, bool slots);
    uint32_t rec_stat_mask_ = 0;
    DataAllocator<uint8_t> rec_spike_;
    DataAllocator<float> rec_v_, rec_isyn_, rec_iou_;
    int64_t rec_step0_ = 0;
    int64_t rec_len_ = 0;
    bool rec_freq_ = false, rec_samples_ = false;
    bool rec_ext_on_ = false;            // recording into rec_ext_ (begin_record_at)
    RecordBuffers rec_ext_{};
    std::vector<uint32_t> tile_syn_;      // synapses per target tile
    double row_coverage_ = 0.0;           // mean fraction of the tiles one row reaches
    double shared_segments_ = 0.0;        // shared_segments()
    void sample_sharing(const NetworkHost &net);
    double group_coverage_ = 0.0;         // mean fraction of the gather groups one row reaches
    bool gather_ok_ = false;              // gather_allowed()
    uint32_t gather_bits_ = kGroupBits;   // gather_bits()
    void choose_groups(bool by_tile);     // sets gather_bits_
    bool gather_built_ = false;           // segidx_, fired_, fcount_ built
    bool direct_ok_ = false;              // direct_allowed()
    bool direct_fits() const;             // its conditions on the sizes
    DataAllocator<uint16_t> tidx_;        // [n][ntiles + 1] tile offsets (direct propagation)
    std::vector<uint32_t> src_pass_;      // per tile: binning passes of all its rows
    uint64_t passcap_ = 0;
    DataAllocator<unsigned long long> passes_;   // [kFiredLists][passcap_]
    DataAllocator<uint32_t> pass_count_;  // [2][kFiredLists][kFiredCountStride]
    DataAllocator<uint16_t> segidx_;      // [n][ngroups + 1] group offsets (built on demand)
    DataAllocator<uint32_t> grec_;        // [nsyn][grec_words] gather records (built with segidx_)
    DataAllocator<uint32_t> fired_;       // [2][kFiredLists][fired_capacity()] fired rows
    DataAllocator<uint32_t> fcount_;      // [2][kFiredLists][kFiredCountStride]
    bool pull_built_ = false;             // crec_, cptr_, bitmaps built
    DataAllocator<uint32_t> crec_;        // [nsyn][grec_words] in-edges: key (source row | target in tile |
                                          // channel bit), weight pair bits
    DataAllocator<int64_t> cptr_;         // [ntiles + 1] first in-edge of each target tile
    uint32_t gamma_calls_ = 0;            // gamma draw streams used
    std::vector<uint32_t> tile_cls_;      // per tile: 1 + shared parameter class, or 0
};

// Steps a set of instances together.  One launch per step covers every
// neuron of every active instance (one workgroup per tile of 256 neurons),
// preceded by one k_gather launch when some instance gathers.  The step
// loop can be captured into HIP graphs (one per starting parity).
class Engine {
public:
    explicit Engine(int device);
    ~Engine();

    int device() const { return device_; }
    hipStream_t stream() const { return stream_; }

    int add(std::unique_ptr<Instance> inst);
    std::unique_ptr<Instance> remove(int id);
    Instance *get(int id);
    size_t active() const;

    // Runs `steps` steps of every active instance.  graph_chunk > 1 captures
    // that many steps into one HIP graph and replays it.
    void run(int64_t steps, int graph_chunk);
    // Since the engine was made: synapses past a queue's capacity (spilled,
    // or dropped and taken by the pull; not an error), tiles that deferred
    // their rows, tiles that pulled.
    CtlTotals propagation_stats();
    uint64_t spilled() { return propagation_stats().spilled; }
    // Step-kernel schedule: synapses per lane in a binning pass (1, 2, 4) and
    // the propagation layout: queues with dense or spread counts
    // (kLayoutAuto: by row coverage), or gather (kLayoutGather: every
    // instance that allows it; the others use dense queues).  Every schedule
    // gives the same results.
    void set_schedule(uint32_t pass_k, int layout);
    // Whether instance p propagates by gather under the current layout.
    bool use_gather(const Instance &p) const;
    uint32_t pass_k() const { return pass_k_; }
    int count_layout() const { return count_layout_; }
    uint32_t count_shift() const { return cshift_; }
    // Times every schedule on about `trial_steps` real steps of all
    // instances, in turns of kAutotuneWindow steps (each preceded by 2 steps
    // that apply it, and one untimed turn first), keeps the fastest; us[7] =
    // mean microseconds per step, [dense, spread] x [K = 1, 2, 4], then
    // gather (K = 2; a candidate only when some instance allows it, else its
    // turns run the default schedule and us[6] = 0).  Steps run:
    // autotune_steps(trial_steps).
    static constexpr int64_t kAutotuneWindow = 4;
    static int64_t autotune_steps(int64_t trial_steps)
    {
        const int64_t rounds = (trial_steps + kAutotuneWindow - 1) / kAutotuneWindow;
        return 7 * (2 + rounds * (2 + kAutotuneWindow));
    }
    // Some instance allows gather propagation.
    bool gather_possible() const;
    // Some instance propagates by gather under the current layout.
    bool any_gather() const;
    void autotune(int64_t trial_steps, uint32_t *best_k, int *best_layout, float *us);
    // Pull propagation: on = every instance that allows it gets its
    // in-edges (when added, or at the next table build) and propagates
    // through them where queues overflow or tiles defer; defer_min = emitted
    // rows from which a tile defers (0: tiles never defer, overflowing
    // queues still pull).  Off: queues only, past-capacity synapses through
    // the spill accumulators.  Every setting gives the same results.
    void set_pull(bool on, uint32_t defer_min);
    // Split binning: the fired rows are binned by a second launch per step
    // (k_bin) in equal shares, instead of by the tiles whose neurons fired;
    // off, large engines do so (kBinLaunchTiles).  Results never depend on it,
    // and nothing on cap.
    void set_split(bool on, uint32_t cap)
    {
        if (on != split_ || cap != split_cap_) {
            split_ = on;
            split_cap_ = cap;
            routes_changed();
        }
    }
    bool split() const { return split_; }
    uint32_t split_cap() const { return split_cap_; }
    bool pull_on() const { return pull_on_; }
    uint32_t defer_min() const { return defer_min_; }
    // (a direct instance pulls the steps whose emitted rows are many)
    bool uses_pull(const Instance &p) const { return pull_on_ && p.pull_built() && !use_gather(p); }
    // How the tables of the last build step (gathers(): some of their
    // instances gather), and how often an instance's tile offsets or pass
    // lists were built.
    StepMode step_mode() const { return mode_; }
    bool gathers() const { return ngroups_ > 0; }
    uint64_t tables_built() const { return tables_built_; }
    // Queue capacity per tile: min(synapses targeting it, floor +
    // (synapses >> shift)); shift 0 keeps the exact worst case.
    void set_queue_capacity(uint32_t floor, uint32_t shift);
    uint32_t queue_capacity(uint32_t synapses) const;
    // Queue slots per parity of instance p at the current capacity.
    uint64_t queue_slots(const Instance &p) const;
    void sync();
    void mark_dirty() { dirty_ = true; }
    // Stream for building instances: their set-up runs beside the steps of
    // the instances already in the tables.
    hipStream_t admit_stream() const { return admit_stream_; }
    // Instances added since the last table build do not step yet: changing
    // them needs no settle, and their uploads go on the admission stream.
    bool staged(int id) const { return staged_.count(id) != 0; }
    void settle_for(int id)
    {
        if (!staged(id))
            settle();
    }
    hipStream_t stream_for(int id) const { return staged(id) ? admit_stream_ : stream_; }
    // Writes the pending delta of every instance into its dlt buffer (the
    // queues are left for the next step), then waits.
    void materialize();
    // Drops the pending delta of one instance (checkpoint restore).
    void clear_queues(int id);
    // Records the I_syn-based statistics of the last step run (imean,
    // receptor imeans), which the next step's launch would otherwise take.
    // wait: until it is done; else only enqueued on stream().
    void stat_tail(bool wait = true);
    // Folds every pending delta into J with the current tables and
    // parameters.  Must run before parameters, samples, recording or the
    // instance set change (a table rebuild empties the queues).
    // wait: until it is done; else only enqueued on stream().
    void settle(bool wait = true);
    // settle(), and the step index of instance p.
    int64_t settled_step(Instance &p);
    // Pinned memory for one call's results.
    HostStage &call_stage() { return call_stage_; }

    // Kernel-time measurement: events recorded around every step kernel
    // (total in ms over `steps` steps).
    void run_timed(int64_t steps, float *ms_step);
    // run(steps, graph_chunk) between two events on the engine stream; *ms =
    // the GPU time between them (the step kernels and the gaps between).
    void run_span(int64_t steps, int graph_chunk, float *ms);
    // run(steps, graph_chunk) with an event after every unit (a step run
    // eagerly or a replayed graph chunk); *ms = the GPU time from before the
    // first unit to after the last, ms_steps[steps] (optional) = each step's
    // share of its unit's time (a chunk's time divided by its steps).
    void run_span_units(int64_t steps, int graph_chunk, float *ms, float *ms_steps);

private:
    void rebuild();
    void launch_step();        // one step at parity par_, then par_ ^= 1
    void launch_step_k(hipEvent_t *ev = nullptr);   // ev: 6 events (start and stop of up to three kernels)
    void launch_aux();         // materialize + sample after a step, if samples are set
    void drop_graphs();
    QueueSet queues();

    int device_ = 0;
    hipStream_t stream_ = nullptr;
    std::vector<std::unique_ptr<Instance>> insts_;
    std::vector<uint32_t> tile_base_;      // per instance slot, first tile in the engine table
    bool dirty_ = true;
    hipStream_t admit_stream_ = nullptr;
    std::unordered_set<int> staged_;
    bool pending_ = false;                 // queues may hold an unfolded delta
    uint32_t par_ = 0;                     // parity of the next step launch (= pending queue set)
    uint32_t ninst_ = 0, nsamples_ = 0, ntiles_ = 0;
    uint32_t cshift_ = kCountShiftDense;   // queue count layout (count_slot)
    int count_layout_ = kLayoutAuto;       // requested layout
    uint32_t pass_k_ = kPassKDefault;      // synapses per lane in a binning pass
    uint32_t wfmt_ = kWeightF32;           // weight format of every instance in the tables, or kWeightAny
    bool stat_ = false;                    // some instance in the tables records population statistics
    static constexpr uint32_t kQueueFloorDefault = 4096, kQueueShiftDefault = 3;
    uint32_t queue_floor_ = kQueueFloorDefault, queue_shift_ = kQueueShiftDefault;   // queue_capacity
    bool tuning_ = false;                  // autotune running: gather buffers are kept
    bool pull_on_ = true;                  // pull propagation where in-edges fit
    bool split_ = false;                   // split binning (k_bin)
    uint32_t split_cap_ = 0;               // as given to set_split
    DataAllocator<BinDesc> d_bins_;        // k_bin's workgroups
    uint32_t nbins_ = 0, bin_tiles_ = 0;   // their number (0: tiles bin their own rows), tiles of the largest queue instance
    bool want_bin_launch();   // and builds the pass lists; false if they do not fit
    uint64_t tables_built_ = 0;            // tables_built()
    uint32_t defer_min_ = kDeferMinDefault;
    void try_pull(Instance &p, hipStream_t s);   // builds p's in-edges if on and they fit
    DataAllocator<InstDev> d_insts_;
    DataAllocator<StepCtl> d_ctl_;
    DataAllocator<SampleDev> d_samples_;
    DataAllocator<SampleRecDev> d_recs_;
    DataAllocator<TileDesc> d_tiles_;
    DataAllocator<QueueTile> d_qtiles_;
    DataAllocator<QueueSet> d_queues_;     // queues() of the tables, as k_step reads it
    DataAllocator<uint32_t> d_qcnt_;       // count_words(2 * ntiles)
    DataAllocator<GroupDesc> d_groups_;    // gather groups of the gather instances
    uint32_t ngroups_ = 0;
    void launch_gather_k(uint32_t par);    // k_gather of parity par, if any instance gathers
    // Whether instance p takes its input by direct propagation: the automatic
    // layout (or the autotuner's pick of it) with no propagation setting of
    // the user's own, and p allows it.  (It then needs its in-edges, which
    // volleys are taken through: without them 200k neurons' volley from rest
    // takes 7.0 ms, by queues and spill 2.2.)
    bool wants_direct(const Instance &p) const
    {
        return (count_layout_ == kLayoutAuto || tuned_ == Tuned::automatic) && !split_ && pull_on_ && queue_floor_ == kQueueFloorDefault &&
               queue_shift_ == kQueueShiftDefault && defer_min_ == kDeferMinDefault && p.direct_allowed();
    }
    bool try_direct(Instance &p, hipStream_t s);   // builds p's tile offsets if they fit
    // Whether the engine's instances, and `joining` with them, should step by
    // direct propagation, all of them (an engine with both kinds steps in two
    // launches, one after the other): all want it, and they have at most
    // kDirectTiles tiles together (kDirectTilesStay while it steps so).
    bool direct_by_rules(const Instance *joining = nullptr) const;
    bool want_direct();                    // direct_by_rules(), and builds what it needs
    // Offsets or pass lists did not fit: not tried again (each table build
    // would build and return those that do fit) before the instances or the
    // propagation settings change, or as much memory as was missing is given
    // back to the library.
    struct Short {
        bool on = false, base_set = false;
        size_t need = 0, base = 0;

        void failed(size_t bytes) { *this = Short{true, false, bytes, 0}; }
        // Whether it still holds, at a table build with `cached` bytes free in
        // the library (the first one after the failure sets the base).
        bool holds(size_t cached)
        {
            if (on && !base_set) {
                base_set = true;
                base = cached;
            }
            on = on && cached < base + need;
            return on;
        }
    };
    Short direct_short_, passes_short_;
    void routes_changed()
    {
        dirty_ = true;
        direct_short_.on = passes_short_.on = false;
    }
    StepMode mode_ = StepMode::tile_bin;   // of every tile in the tables
    // A schedule of the autotuner's: its (dense, default pass) candidate
    // stands for the automatic choice among direct propagation, the binning
    // launch and binning in the tiles; the other queue candidates are what
    // they name, with the rows binned in the tiles (a binning launch knows no
    // pass size, so they would all time the same kernels).
    enum class Tuned { no, automatic, named };
    Tuned tuned_ = Tuned::no;
    HostStage tables_stage_, call_stage_;
    // Everything a captured step's launches take from the engine: graphs stay
    // as long as it does (what changes from run to run is in the tables).
    struct GraphKey {
        const void *tiles, *insts, *queues, *qtiles, *qcnt, *bins, *groups, *samples, *recs;
        uint32_t ntiles, mode, nbins, bin_tiles, ngroups, nsamples, cshift, pass_k, wfmt, stat;
    };
    GraphKey graph_key_{};
    hipGraphExec_t graph_[2] = {nullptr, nullptr};   // by starting parity
    int graph_steps_[2] = {0, 0};
};

}  // namespace dtb
