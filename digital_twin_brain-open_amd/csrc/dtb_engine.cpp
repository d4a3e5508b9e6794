// dtb_engine.cpp -- host runtime of the DTB step (see dtb_engine.hpp).
//
// Host arithmetic that produces kernel inputs (1/C, refractory steps,
// exp(-dt/tau), OU factors, V0) is done here once per run configuration, in
// the order the CPU oracle uses, with contraction disabled, so that the GPU
// and the oracle start from bit-identical parameters.
#include "dtb_engine.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <thread>
#include <unordered_map>
#include <unordered_set>

#include "dtb_devgen.hpp"
#include "dtb_gen.hpp"
#include "dtb_kernels.hpp"
#include "dtb_parts.hpp"

namespace dtb {

void hip_check(hipError_t e, const char *what, const char *file, int line)
{
    if (e == hipSuccess)
        return;
    std::string msg = std::string(hipGetErrorString(e)) + " in " + what + " (" + file + ":" + std::to_string(line) + ")";
    if (e == hipErrorOutOfMemory)
        throw Error(kOutOfMemory, msg);
    if (e == hipErrorNoDevice || e == hipErrorInvalidDevice)
        throw Error(kNoDevice, msg);
    throw Error(kHipError, msg);
}

int prop_type_column(int prop)
{
    // dist_blockwrapper.py:32-33 maps columns to PropType with
    // [19, -1, 0, -1, 1, 2, ..., 18]; this is the inverse.
    static const int kCol[kNumPropTypes] = {kColIExt,  kColC,      kColTRef,   kColGLeak, kColVLeak,
                                            kColVTh,   kColVReset, kColGU + 0, kColGU + 1, kColGU + 2,
                                            kColGU + 3, kColVU + 0, kColVU + 1, kColVU + 2, kColVU + 3,
                                            kColTauU + 0, kColTauU + 1, kColTauU + 2, kColTauU + 3, kColNoiseRate};
    if (prop < 0 || prop >= kNumPropTypes)
        return -1;
    return kCol[prop];
}

size_t data_size(DataType t)
{
    switch (t) {
    case DOUBLE:
        return 8;
    case FLOAT:
    case INT32:
        return 4;
    case FLOAT16:
        return 2;
    case INT8:
        return 1;
    }
    return 0;
}

// ---------------------------------------------------------------------------
// Host-side parameter derivation.  Mirrors the oracle exactly.

static inline float host_expf(float x)
{
    return (float)std::exp((double)x);
}

static inline int32_t refractory_substeps(float t_ref, float dt, int32_t t_steps)
{
    // property.cpp:45-53 (t_ref / dt at init, block.cpp:150) and
    // membrane_voltage.cpp:177 ((int)t_ref * t_steps).
    const float steps = t_ref / dt;
    return (int32_t)steps * t_steps;
}

static inline void ou_factors(float dt_sub, float tau, float sigma, float *f1, float *f2s)
{
    // extern_stimuli.cpp:87-91
    const float factor = (-dt_sub) / tau;
    const float a = 1.0f - host_expf(factor);
    const float b = std::sqrt(1.0f - host_expf(2.0f * factor));
    *f1 = a;
    *f2s = b * sigma;
}

static inline float bits_as_float(int32_t v)
{
    float f;
    std::memcpy(&f, &v, 4);
    return f;
}

// ---------------------------------------------------------------------------

Instance::Instance(const NetworkHost &net, float dt, uint64_t seed, hipStream_t s)
{
    if (net.n <= 0 || net.n > (int64_t)kColMask)
        throw Error(kInvalidNetwork, "neuron count out of range");
    if (net.props == nullptr || net.rowptr == nullptr)
        throw Error(kInvalidParameter, "props and rowptr are required");
    if (net.nsyn < 0 || (net.nsyn > 0 && (net.col == nullptr || net.w == nullptr || net.kind_bits == nullptr)))
        throw Error(kInvalidParameter, "synapse arrays are required");
    if (net.wfmt != kWeightF32 && net.wfmt != kWeightF16 && net.wfmt != kWeightU8)
        throw Error(kInvalidParameter, "unknown weight format");
    n_ = (uint32_t)net.n;
    nsyn_ = net.nsyn;
    wfmt_ = net.wfmt;

    // CSR validation (rows ascending, columns in range).
    if (net.rowptr[0] != 0 || net.rowptr[net.n] != net.nsyn)
        throw Error(kInvalidNetwork, "rowptr must start at 0 and end at nsyn");
    if (net.nsyn >= kMaxSynapses)
        throw Error(kInvalidNetwork, "too many synapses for one block");
    for (int64_t i = 0; i < net.n; ++i)
        if (net.rowptr[i + 1] < net.rowptr[i] || net.rowptr[i + 1] - net.rowptr[i] >= kMaxRowLength)
            throw Error(kInvalidNetwork, "rowptr must be non-decreasing with rows below 2^31 synapses");
    for (int64_t j = 0; j < net.nsyn; ++j)
        if (net.col[j] >= n_)
            throw Error(kInvalidNetwork, "column index out of range");

    init_common(net.props, dt, seed, s);

    rowptr_.upload(net.rowptr, (size_t)n_ + 1, s);
    // Pack the channel bit into bit 31 of the column index so that one
    // 4-byte load per synapse carries both.
    const int64_t chunk = (int64_t)1 << 24;
    std::vector<uint32_t> stage((size_t)std::min<int64_t>(std::max<int64_t>(nsyn_, 1), chunk));
    for (int64_t base = 0; base < nsyn_; base += chunk) {
        const int64_t m = std::min<int64_t>(chunk, nsyn_ - base);
        for (int64_t j = 0; j < m; ++j) {
            const int64_t g = base + j;
            const uint32_t kind = (net.kind_bits[g >> 5] >> (g & 31)) & 1u;
            stage[(size_t)j] = net.col[g] | (kind ? kKindBit : 0u);
        }
        DTB_HIP(hipMemcpyAsync(col_.mutable_gpu_data() + base, stage.data(), (size_t)m * sizeof(uint32_t),
                               hipMemcpyHostToDevice, s));
        DTB_HIP(hipStreamSynchronize(s));
    }
    if (nsyn_ > 0)
        w_.upload(static_cast<const uint8_t *>(net.w), (size_t)nsyn_ * weight_bytes(wfmt_), s);
    count_tile_synapses(net);
    DTB_HIP(hipStreamSynchronize(s));
}

void Instance::init_common(const float *props, float dt, uint64_t seed, hipStream_t s)
{
    init_common(std::vector<float>(props, props + (size_t)n_ * kNumCols), dt, seed, s);
}

void Instance::init_common(std::vector<float> &&props, float dt, uint64_t seed, hipStream_t s)
{
    if (!(dt > 0.0f))
        throw Error(kInvalidParameter, "dt must be positive");
    dt_ = dt;
    seed_ = seed;
    props_ = std::move(props);

    // Populations: contiguous runs of the sub-block column
    // (configuration.cpp:1902-1930 requires each sub-block to be contiguous).
    std::unordered_set<uint32_t> seen;
    for (uint32_t i = 0; i < n_; ++i) {
        const float v = props_[(size_t)i * kNumCols + kColSubIdx];
        if (!(v >= 0.0f) || v > 4294967040.0f)
            throw Error(kInvalidNetwork, "sub-block id must be a non-negative integer");
        const uint32_t id = (uint32_t)v;
        if (i == 0 || id != pop_ids_.back()) {
            if (!seen.insert(id).second)
                throw Error(kInvalidNetwork, "sub-block ids must form contiguous ranges");
            pop_ids_.push_back(id);
            pop_begin_.push_back(i);
        }
    }
    pop_begin_.push_back(n_);
    const size_t np = pop_ids_.size();
    ou_on_.assign(np, 0);
    ou_mean_.assign(np, 0.0f);
    ou_sigma_.assign(np, 0.0f);
    ou_tau_.assign(np, 1.0f);

    blocked_.resize(n_);
    state_.resize((size_t)((n_ + kBlock - 1) / kBlock) * kStateBytes);
    dlt_.resize(n_);
    spill_.resize((size_t)n_ * 8);
    rowptr_.resize((size_t)n_ + 1);
    col_.resize((size_t)std::max<int64_t>(nsyn_, 1));
    w_.resize((size_t)std::max<int64_t>(nsyn_, 1) * weight_bytes(wfmt_));
    pops_.resize(np);
    step_.resize(kStepPad + 2 * (size_t)((n_ + kBlock - 1) / kBlock) * kBitWords);
    counters_.resize(2 * (size_t)((n_ + kWave - 1) / kWave));

    derive_params(s);
    init_state(s);

}

Instance::Instance(const FanoutSpec &f, float dt, uint64_t seed, hipStream_t s)
{
    if (f.n < 2 || f.n > (int64_t)kColMask || f.K == 0 || f.K > 8192)
        throw Error(kInvalidParameter, "fan-out network: need n >= 2 and 1 <= K <= 8192");
    if (f.n * (int64_t)f.K >= kMaxSynapses)
        throw Error(kInvalidNetwork, "too many synapses for one block");
    n_ = (uint32_t)f.n;
    nsyn_ = f.n * (int64_t)f.K;
    // The synapses are generated on the device while the host builds the
    // property matrix and parameter records (init_common's uploads follow
    // the generation on the same stream).
    rowptr_.resize((size_t)n_ + 1);
    col_.resize((size_t)nsyn_);
    wfmt_ = kWeightF32;
    w_.resize((size_t)nsyn_ * weight_bytes(wfmt_));
    const uint32_t ntile = (n_ + (1u << kTileBits) - 1) >> kTileBits;
    DataAllocator<uint32_t> tsyn(ntile);
    DTB_HIP(launch_gen_fanout(n_, f.K, f.net_seed, rowptr_.mutable_gpu_data(), col_.mutable_gpu_data(),
                              reinterpret_cast<float2 *>(w_.mutable_gpu_data()), tsyn.mutable_gpu_data(), s));
    std::vector<float> props((size_t)n_ * kNumCols);
    gen_default_props(f.n, f.g_ui, f.sub_base, props.data());
    init_common(std::move(props), dt, seed, s);
    tile_syn_.assign(ntile, 0u);
    tsyn.download(tile_syn_.data(), ntile, s);
    DTB_HIP(hipStreamSynchronize(s));
    // expected distinct tiles (groups) among K uniform targets, as a fraction
    row_coverage_ = 1.0 - std::pow(1.0 - 1.0 / ntile, (double)f.K);
    group_coverage_ = 1.0 - std::pow(1.0 - 1.0 / ngroups(), (double)f.K);
    shared_segments_ = row_coverage_ * row_coverage_ * (double)ntile * (double)n_;
    // rows are ordered by target, K <= 8192
    gather_ok_ = (double)n_ * (ngroups() + 1.0) * 2.0 <= 12.0 * (double)nsyn_;
    src_pass_.assign(ntile, 0u);
    for (uint32_t t = 0; t < ntile; ++t)
        src_pass_[t] = std::min<uint32_t>(kBlock, n_ - t * kBlock) * (((uint32_t)f.K + kBinPass - 1u) / kBinPass);
    choose_groups(true);
    direct_ok_ = direct_fits();
}

Instance::~Instance() = default;

void Instance::count_tile_synapses(const NetworkHost &net)
{
    // Synapses per target tile: a tile's queue holds at most one entry per
    // synapse that targets it (every row fires at most once per step), so
    // these counts are its exact capacity.
    const uint32_t nfine = (n_ + (1u << kTileBits) - 1) >> kTileBits;
    tile_syn_.assign(nfine, 0u);
    src_pass_.assign(nfine, 0u);
    for (uint32_t r = 0; r < n_; ++r)
        src_pass_[r >> kTileBits] += (uint32_t)((net.rowptr[r + 1] - net.rowptr[r] + kBinPass - 1) / kBinPass);
    unsigned hw = std::thread::hardware_concurrency();
    const int nt = (int)std::max<int64_t>(1, std::min<int64_t>(std::min(hw ? hw : 4u, 16u), nsyn_ / (1 << 20)));
    std::vector<std::vector<uint32_t>> part(nt, std::vector<uint32_t>(nfine, 0u));
    std::vector<uint64_t> segs(nt, 0), gsegs(nt, 0);
    std::vector<char> sorted(nt, 1), tile_sorted(nt, 1);
    std::vector<std::thread> th;
    for (int t = 0; t < nt; ++t) {
        th.emplace_back([&, t]() {
            const int64_t a = (int64_t)n_ * t / nt, b = (int64_t)n_ * (t + 1) / nt;
            uint32_t *c = part[t].data();
            uint64_t sg = 0, gs = 0;
            bool ordered = true, by_tile = true;
            for (int64_t r = a; r < b; ++r) {
                uint32_t prev = 0xffffffffu, gprev = 0xffffffffu;
                for (int64_t j = net.rowptr[r]; j < net.rowptr[r + 1]; ++j) {
                    const uint32_t tl = net.col[j] >> kTileBits;
                    const uint32_t gr = net.col[j] >> kGroupBits;
                    ++c[tl];
                    sg += tl != prev;
                    gs += gr != gprev;
                    ordered = ordered && (gprev == 0xffffffffu || gr >= gprev);
                    by_tile = by_tile && (prev == 0xffffffffu || tl >= prev);
                    prev = tl;
                    gprev = gr;
                }
                ordered = ordered && net.rowptr[r + 1] - net.rowptr[r] <= kGatherMaxRow;
            }
            segs[t] = sg;
            gsegs[t] = gs;
            sorted[t] = ordered ? 1 : 0;
            tile_sorted[t] = ordered && by_tile ? 1 : 0;
        });
    }
    for (auto &x : th)
        x.join();
    uint64_t sg = 0, gs = 0;
    bool ordered = true, by_tile = true;
    for (int t = 0; t < nt; ++t) {
        sg += segs[t];
        gs += gsegs[t];
        ordered = ordered && sorted[t];
        by_tile = by_tile && tile_sorted[t];
        for (uint32_t k = 0; k < nfine; ++k)
            tile_syn_[k] += part[t][k];
    }
    row_coverage_ = (double)sg / ((double)n_ * (double)nfine);
    group_coverage_ = (double)gs / ((double)n_ * (double)ngroups());
    gather_ok_ = ordered && nsyn_ > 0 && (double)n_ * (ngroups() + 1.0) * 2.0 <= 12.0 * (double)nsyn_;
    choose_groups(by_tile);
    sample_sharing(net);
    direct_ok_ = by_tile && direct_fits();
}

void Instance::sample_sharing(const NetworkHost &net)
{
    const uint32_t ntile = (n_ + kBlock - 1) / kBlock;
    const uint32_t rows = std::min(n_, kSharingRows);
    std::vector<uint32_t> mark(ntile, 0u);   // 2 k + 1: reached by the k-th sampled row, 2 k + 2: and counted
    uint64_t shared = 0, seen = 0;
    uint32_t k = 0;
    for (; k < rows && seen < ((uint64_t)1 << 20); ++k) {   // (rows of tens of thousands: fewer of them)
        const uint32_t r = (uint32_t)((uint64_t)n_ * k / rows);
        const uint32_t s = (uint32_t)(((uint64_t)r + kSharingDistance) % n_);
        for (int64_t j = net.rowptr[r]; j < net.rowptr[r + 1]; ++j)
            mark[(net.col[j] & kColMask) >> kTileBits] = 2u * k + 1u;
        for (int64_t j = net.rowptr[s]; j < net.rowptr[s + 1]; ++j) {
            uint32_t &m = mark[(net.col[j] & kColMask) >> kTileBits];
            if (m == 2u * k + 1u) {
                ++m;
                ++shared;
            }
        }
        seen += (uint64_t)(net.rowptr[r + 1] - net.rowptr[r]) + (uint64_t)(net.rowptr[s + 1] - net.rowptr[s]);
    }
    shared_segments_ = k > 0 ? (double)shared / k * n_ : 0.0;
}

void Instance::choose_groups(bool by_tile)
{
    gather_bits_ = kGroupBits;
    while (by_tile && gather_bits_ > kGroupBitsMin && ngroups(gather_bits_) < kGatherGroups &&
           (double)n_ * (ngroups(gather_bits_ - 1u) + 1.0) * 2.0 <= 12.0 * (double)nsyn_)
        --gather_bits_;
}

uint32_t Instance::fired_capacity() const
{
    const uint32_t ntile = (n_ + kBlock - 1) / kBlock;
    return (ntile + kFiredLists - 1) / kFiredLists * kBlock;
}

void Instance::ensure_gather(hipStream_t s)
{
    if (!gather_ok_)
        throw Error(kInvalidParameter, "this network does not allow gather propagation");
    if (gather_built_)
        return;
    try {
        fcount_.resize(2 * (size_t)kFiredLists * kFiredCountStride);
        fcount_.mutable_gpu_data();
        fired_.resize(2 * (size_t)kFiredLists * fired_capacity());
        fired_.mutable_gpu_data();
        grec_.resize((size_t)nsyn_ * grec_words(wfmt_));
        DTB_HIP(launch_build_grec(col_.gpu_data(), w_.gpu_data(), wfmt_, (uint64_t)nsyn_, grec_.mutable_gpu_data(),
                                  s));
        for (;;) {
            segidx_.resize((size_t)n_ * (ngroups(gather_bits_) + 1u));
            try {
                segidx_.mutable_gpu_data();
                break;
            } catch (const Error &e) {
                // without device memory for the offsets of smaller groups:
                // larger ones
                if (e.code != kOutOfMemory || gather_bits_ == kGroupBits)
                    throw;
                ++gather_bits_;
            }
        }
        DTB_HIP(launch_build_segidx(rowptr_.gpu_data(), col_.gpu_data(), n_, ngroups(gather_bits_), gather_bits_,
                                    segidx_.mutable_gpu_data(), s));
        DTB_HIP(hipStreamSynchronize(s));
    } catch (...) {
        // out of device memory (or a failed build): nothing half-built stays
        release_gather();
        throw;
    }
    gather_built_ = true;
}

// The lookups of an emitted row (one per tile) against the queue entries it
// would make.  Voxel networks, rows emitted per step: time of a step by
// queues / direct: 130k neurons x 150 synapses (4 T / k = 14): 66: 7.2 / 7.2
// us, 749: 17.4 / 11.7; 200k x 150 (21): 98: 8.2 / 8.5, 677: 14.5 / 13.6;
// 260k x 300 (14): 78: 9.8 / 9.1, 1465: 25.5 / 23.4.  Rows that reach many
// tiles cost the queues more: uniform 200k x 150 (coverage 0.17), 99: 10.0 /
// 8.1, 1920: 74.5 / 26.3.
bool Instance::direct_fits() const
{
    const double ntile = (double)((n_ + kBlock - 1) / kBlock);
    return nsyn_ > 0 && nsyn_ < ((int64_t)1 << 32) && n_ <= kDirectMaxNeurons &&
           (double)n_ * (ntile + 1.0) * 2.0 <= 12.0 * (double)nsyn_ &&
           ((double)n_ * ntile <= 4.0 * (double)nsyn_ || row_coverage_ >= 0.125);
}

void Instance::ensure_direct(hipStream_t s)
{
    if (!direct_ok_)
        throw Error(kInvalidParameter, "this network does not allow direct propagation");
    if (direct_built())
        return;
    const uint32_t ntile = (n_ + kBlock - 1) / kBlock;
    try {
        tidx_.resize((size_t)n_ * (ntile + 1u));
        // (every word is written; up to 500 MB to clear otherwise)
        DTB_HIP(launch_build_segidx(rowptr_.gpu_data(), col_.gpu_data(), n_, ntile, kTileBits, tidx_.gpu_uncleared(),
                                    s));
        DTB_HIP(hipStreamSynchronize(s));
    } catch (...) {
        tidx_.resize(0);
        throw;
    }
}

void Instance::ensure_passes()
{
    if (passes_built())
        return;
    // list l takes the tiles t with t * kFiredLists / ntiles == l
    const uint64_t nt = src_pass_.size();
    std::vector<uint64_t> cap(kFiredLists, 0);
    for (uint64_t t = 0; t < nt; ++t)
        cap[t * kFiredLists / nt] += src_pass_[t];
    passcap_ = std::max<uint64_t>(1, *std::max_element(cap.begin(), cap.end()));
    try {
        pass_count_.resize(2 * (size_t)kFiredLists * kFiredCountStride);
        pass_count_.mutable_gpu_data();
        passes_.resize((size_t)(kFiredLists * passcap_));
        passes_.gpu_uncleared();   // (entries past a list's count are not read)
    } catch (...) {
        release_passes();
        throw;
    }
}

void Instance::release_passes()
{
    passes_.resize(0);
    pass_count_.resize(0);
}

CopyWords Instance::pass_count_words()
{
    return CopyWords{pass_count_.mutable_gpu_data(), nullptr, pass_count_.count()};
}

void Instance::release_gather()
{
    segidx_.resize(0);
    grec_.resize(0);
    fired_.resize(0);
    fcount_.resize(0);
    gather_built_ = false;
}

void Instance::clear_fired(hipStream_t s)
{
    if (gather_built_)
        DTB_HIP(hipMemsetAsync(fcount_.mutable_gpu_data(), 0, fcount_.size(), s));
}

uint64_t Instance::pull_bytes() const
{
    const uint64_t ntile = (n_ + kBlock - 1) / kBlock;
    return (uint64_t)nsyn_ * sizeof(uint32_t) * grec_words(wfmt_) + (ntile + 1) * sizeof(int64_t);
}

void Instance::ensure_pull(hipStream_t s)
{
    if (!pull_allowed())
        throw Error(kInvalidParameter, "this network does not allow pull propagation");
    if (pull_built_)
        return;
    const uint32_t ntile = (n_ + kBlock - 1) / kBlock;
    try {
        // first in-edge of every target tile: prefix sums of the synapses
        // targeting the tiles
        std::vector<int64_t> ptr((size_t)ntile + 1, 0);
        for (uint32_t t = 0; t < ntile; ++t)
            ptr[t + 1] = ptr[t] + tile_syn_.at(t);
        if (ptr[ntile] != nsyn_)
            throw Error(kInternal, "tile synapse counts do not add up to the synapses");
        cptr_.resize((size_t)ntile + 1);
        cptr_.upload(ptr.data(), ptr.size(), s);
        crec_.resize((size_t)nsyn_ * grec_words(wfmt_));
        DataAllocator<uint32_t> cursor(ntile);
        DTB_HIP(hipMemsetAsync(cursor.mutable_gpu_data(), 0, (size_t)ntile * sizeof(uint32_t), s));
        DTB_HIP(launch_build_pull(rowptr_.gpu_data(), col_.gpu_data(), w_.gpu_data(), wfmt_, n_, cptr_.gpu_data(),
                                  cursor.mutable_gpu_data(), crec_.mutable_gpu_data(), s));
        DTB_HIP(hipStreamSynchronize(s));
    } catch (...) {
        release_pull();
        throw;
    }
    pull_built_ = true;
}

void Instance::release_pull()
{
    crec_.resize(0);
    cptr_.resize(0);
    pull_built_ = false;
}

CopyWords Instance::deferred_words()
{
    return CopyWords{step_.mutable_gpu_data() + 2, nullptr, (step_.size() - 2 * sizeof(int64_t)) / 4};
}

void Instance::clear_deferred(hipStream_t s)
{
    const CopyWords w = deferred_words();
    DTB_HIP(launch_copy_words(&w, 1, s));
}

uint32_t Instance::tile_synapses(uint32_t tile) const
{
    return tile_syn_.at(tile);
}

namespace {

bool same_bits(const ParamRec &x, const ParamRec &y)
{
    return std::memcmp(&x, &y, sizeof(ParamRec)) == 0;
}

struct ParamRecHash {
    size_t operator()(const ParamRec &r) const
    {
        uint32_t w[sizeof(ParamRec) / 4];
        std::memcpy(w, &r, sizeof(ParamRec));
        uint64_t h = 0x9e3779b97f4a7c15ull;
        for (uint32_t x : w)
            h = (h ^ x) * 0x100000001b3ull;
        return (size_t)(h ^ (h >> 29));
    }
};

struct ParamRecEq {
    bool operator()(const ParamRec &x, const ParamRec &y) const { return same_bits(x, y); }
};

}  // namespace

void Instance::derive_params(hipStream_t s)
{
    const float dt_sub = dt_ / (float)t_steps_;
    // A thread's derivation, in neuron order.
    struct Derive {
        const float *props;
        float dt, dt_sub;
        int32_t t_steps;
        const float *prev = nullptr;
        ParamRec cur{};

        const ParamRec &operator()(uint32_t i)
        {
            const float *p = props + (size_t)i * kNumCols;
            if (prev != nullptr && std::memcmp(p, prev, sizeof(float) * kNumCols) == 0)
                return cur;   // same property row as the neuron before
            prev = p;
            cur.a = make_float4(p[kColVReset], p[kColVTh], dt_sub * (1.0f / p[kColC]), p[kColVLeak]);
            cur.b = make_float4(p[kColGLeak], p[kColIExt], p[kColNoiseRate],
                                bits_as_float(refractory_substeps(p[kColTRef], dt, t_steps)));
            cur.g = make_float4(p[kColGU + 0], p[kColGU + 1], p[kColGU + 2], p[kColGU + 3]);
            cur.v = make_float4(p[kColVU + 0], p[kColVU + 1], p[kColVU + 2], p[kColVU + 3]);
            // property.cpp:19-29: exp(-dt / tau)
            cur.d = make_float4(host_expf((-dt_sub) / p[kColTauU + 0]), host_expf((-dt_sub) / p[kColTauU + 1]),
                                host_expf((-dt_sub) / p[kColTauU + 2]), host_expf((-dt_sub) / p[kColTauU + 3]));
            return cur;
        }
    };
    const Derive fresh{props_.data(), dt_, dt_sub, t_steps_};

    // Deduplicate the records: class per neuron + one record per class, by
    // ranges of whole tiles; a range's classes, in the order in which it
    // meets them, then join those of the ranges before it (the same numbers
    // as in one pass).
    const uint32_t ntile = (n_ + kBlock - 1) / kBlock;
    const uint32_t parts = host_parts(n_);
    struct Part {
        std::vector<ParamRec> recs;
        std::vector<uint32_t> cls;   // of its own classes
        bool dense = false;
    };
    std::vector<Part> part(parts);
    auto range = [&](uint32_t k) {
        return std::pair<uint32_t, uint32_t>(
            std::min<uint32_t>(n_, (uint32_t)((uint64_t)ntile * k / parts) * kBlock),
            std::min<uint32_t>(n_, (uint32_t)((uint64_t)ntile * (k + 1) / parts) * kBlock));
    };
    cls_.resize(n_);
    uint16_t *cls = cls_.mutable_cpu_data();
    uint8_t *bl = blocked_.mutable_cpu_data();
    for_parts(parts, [&](uint32_t k) {
        Part &p = part[k];
        Derive derive = fresh;
        std::unordered_map<ParamRec, uint32_t, ParamRecHash, ParamRecEq> index;
        const auto [b, e] = range(k);
        for (uint32_t i = b; i < e; ++i) {
            bl[i] = props_[(size_t)i * kNumCols + kColBlocked] != 0.0f;
            if (p.dense)
                continue;
            const ParamRec &r = derive(i);
            if (i > b && same_bits(r, p.recs[cls[i - 1]])) {
                cls[i] = cls[i - 1];
                continue;
            }
            auto it = index.find(r);
            if (it == index.end()) {
                if (p.recs.size() == kMaxParamClasses) {
                    p.dense = true;
                    continue;
                }
                it = index.emplace(r, (uint32_t)p.recs.size()).first;
                p.recs.push_back(r);
            }
            cls[i] = (uint16_t)it->second;
        }
    });
    std::vector<ParamRec> recs;
    bool dense = false;
    {
        std::unordered_map<ParamRec, uint32_t, ParamRecHash, ParamRecEq> index;
        for (Part &p : part) {
            dense = dense || p.dense;
            for (const ParamRec &r : p.recs) {
                if (dense)
                    break;
                auto it = index.find(r);
                if (it == index.end()) {
                    if (recs.size() == kMaxParamClasses) {
                        dense = true;
                        break;
                    }
                    it = index.emplace(r, (uint32_t)recs.size()).first;
                    recs.push_back(r);
                }
                p.cls.push_back(it->second);
            }
        }
    }
    dense_params_ = dense;
    prm_.resize(dense ? n_ : recs.size());
    ParamRec *rec = prm_.mutable_cpu_data();
    if (!dense)
        std::copy(recs.begin(), recs.end(), rec);
    tile_cls_.assign(ntile, 0u);
    for_parts(parts, [&](uint32_t k) {
        Derive derive = fresh;
        const auto [b, e] = range(k);
        for (uint32_t t0 = b; t0 < e; t0 += kBlock) {
            const uint32_t t1 = std::min<uint32_t>(e, t0 + kBlock);
            bool same = true;
            for (uint32_t i = t0; i < t1; ++i) {
                if (dense) {
                    rec[i] = derive(i);
                    cls[i] = (uint16_t)(i & (kBlock - 1));
                } else {
                    cls[i] = (uint16_t)part[k].cls[cls[i]];
                    same = same && cls[i] == cls[t0];
                }
            }
            if (!dense)
                tile_cls_[t0 / kBlock] = same ? (uint32_t)cls[t0] + 1u : 0u;
        }
    });
    prm_.to_gpu(s);
    cls_.to_gpu(s);
    blocked_.to_gpu(s);
    derive_pops(s);
}

void Instance::derive_pops(hipStream_t s)
{
    // extern_stimuli.cpp:84-110: per-population OU factors at the substep dt.
    const float dt_sub = dt_ / (float)t_steps_;
    PopDev *pd = pops_.mutable_cpu_data();
    for (size_t q = 0; q < pop_ids_.size(); ++q) {
        PopDev r{};
        r.begin = pop_begin_[q];
        r.end = pop_begin_[q + 1];
        r.ou_on = ou_on_[q];
        if (ou_on_[q]) {
            ou_factors(dt_sub, ou_tau_[q], ou_sigma_[q], &r.f1, &r.f2s);
            r.mu = ou_mean_[q];
        }
        pd[q] = r;
    }
    pops_.to_gpu(s);
    DTB_HIP(hipStreamSynchronize(s));
}

void Instance::init_state(hipStream_t s)
{
    // block.cpp:136-179 and membrane_voltage.cpp:18.
    DTB_HIP(hipMemsetAsync(state_.mutable_gpu_data(), 0, state_.size(), s));
    DTB_HIP(launch_init_state(state_view(), s));
    DTB_HIP(hipMemsetAsync(dlt_.mutable_gpu_data(), 0, dlt_.size(), s));
    DTB_HIP(hipMemsetAsync(spill_.mutable_gpu_data(), 0, spill_.size(), s));
    DTB_HIP(hipMemsetAsync(step_.mutable_gpu_data(), 0, step_.size(), s));
    DTB_HIP(hipMemsetAsync(counters_.mutable_gpu_data(), 0, counters_.size(), s));
    DTB_HIP(hipStreamSynchronize(s));
}

StateView Instance::state_view()
{
    return StateView{state_.mutable_gpu_data(), prm_.gpu_data(), cls_.gpu_data(), dlt_.mutable_gpu_data(),
                     dense_params_ ? ~(uint32_t)(kBlock - 1) : 0u, n_};
}

uint32_t Instance::find_pop(uint32_t brain_id) const
{
    for (size_t q = 0; q < pop_ids_.size(); ++q)
        if (pop_ids_[q] == brain_id)
            return (uint32_t)q;
    return UINT32_MAX;
}

void Instance::set_ou(const uint32_t *brain_ids, const float *mean, const float *sigma, const float *tau,
                      size_t n, hipStream_t s)
{
    // block.cpp:222-281.  A population seen for the first time has its OU
    // current reset to the mean (reset_partial_gpu); a known one only has its
    // parameters replaced.  Ids that are not in this block are skipped.
    for (size_t k = 0; k < n; ++k) {
        if (!(tau[k] > 0.0f))
            throw Error(kInvalidParameter, "OU correlation time must be positive");
    }
    for (size_t k = 0; k < n; ++k) {
        const uint32_t q = find_pop(brain_ids[k]);
        if (q == UINT32_MAX)
            continue;
        const bool first = !ou_on_[q];
        ou_on_[q] = 1;
        ou_mean_[q] = mean[k];
        ou_sigma_[q] = sigma[k];
        ou_tau_[q] = tau[k];
        if (first) {
            DTB_HIP(launch_fill_iou(state_view(), pop_begin_[q], pop_begin_[q + 1], mean[k], s));
        }
    }
    derive_pops(s);   // the neurons' parameter records do not involve the OU current
}

void Instance::update_props(const uint32_t *neuron_ids, const uint32_t *prop_ids, const float *vals, size_t n,
                            hipStream_t s)
{
    // property.cpp:57-183 sets one property of one neuron; the columns of the
    // host property matrix are updated and the kernel inputs re-derived.
    for (size_t k = 0; k < n; ++k) {
        if (prop_type_column((int)prop_ids[k]) < 0)
            throw Error(kInvalidParameter, "unknown property id");
    }
    for (size_t k = 0; k < n; ++k) {
        if (neuron_ids[k] >= n_)
            continue;   // property.cpp:73 ignores out-of-range neurons
        props_[(size_t)neuron_ids[k] * kNumCols + prop_type_column((int)prop_ids[k])] = vals[k];
    }
    derive_params(s);
}

void Instance::update_prop_cols(const uint32_t *prop_ids, const uint32_t *brain_ids, const float *vals, size_t n,
                                bool assign, hipStream_t s)
{
    // property.cpp:185-466: per-population assign (=) or multiply (*=).
    for (size_t k = 0; k < n; ++k) {
        if (prop_type_column((int)prop_ids[k]) < 0)
            throw Error(kInvalidParameter, "unknown property id");
    }
    struct Set {
        uint32_t begin, end;
        int col;
        float val;
    };
    std::vector<Set> sets;
    for (size_t k = 0; k < n; ++k) {
        const uint32_t q = find_pop(brain_ids[k]);
        if (q != UINT32_MAX)
            sets.push_back(Set{pop_begin_[q], pop_begin_[q + 1], prop_type_column((int)prop_ids[k]), vals[k]});
    }
    const uint32_t parts = host_parts(n_);
    for_parts(parts, [&](uint32_t k) {
        const uint32_t b = (uint32_t)((uint64_t)n_ * k / parts), e = (uint32_t)((uint64_t)n_ * (k + 1) / parts);
        for (const Set &v : sets)   // in the caller's order
            for (uint32_t i = std::max(b, v.begin); i < std::min(e, v.end); ++i) {
                float &x = props_[(size_t)i * kNumCols + v.col];
                x = assign ? v.val : x * v.val;
            }
    });
    derive_params(s);
}

void Instance::gamma_prop_cols(const uint32_t *prop_ids, const uint32_t *brain_ids, const float *alpha,
                               const float *beta, size_t n, hipStream_t s)
{
    // block.cpp:1472-1536, property.cpp:470-640: every neuron of the
    // population gets its own Gamma(alpha, rate beta) draw as the property.
    for (size_t k = 0; k < n; ++k) {
        if (prop_type_column((int)prop_ids[k]) < 0)
            throw Error(kInvalidParameter, "unknown property id");
        if (!(alpha[k] >= 0.0f) || !(beta[k] > 0.0f) || !std::isfinite(alpha[k]) || !std::isfinite(beta[k]))
            throw Error(kInvalidParameter, "gamma needs concentration >= 0 and rate > 0");
    }
    std::vector<float> draws;
    for (size_t k = 0; k < n; ++k) {
        const uint32_t call = gamma_calls_++;
        const uint32_t q = find_pop(brain_ids[k]);
        if (q == UINT32_MAX)
            continue;
        const int c = prop_type_column((int)prop_ids[k]);
        const uint32_t b = pop_begin_[q], e = pop_begin_[q + 1];
        draws.resize(e - b);
        gen_gamma(seed_, call, b, e - b, alpha[k], beta[k], draws.data());
        for (uint32_t i = b; i < e; ++i)
            props_[(size_t)i * kNumCols + c] = draws[i - b];
    }
    derive_params(s);
}

void Instance::read_props(float *out) const
{
    std::memcpy(out, props_.data(), sizeof(float) * props_.size());
}

void Instance::set_samples(const uint32_t *ids, size_t n)
{
    for (size_t k = 0; k < n; ++k)
        if (ids[k] >= n_)
            throw Error(kInvalidParameter, "sample id out of range");
    samples_.assign(ids, ids + n);
}

bool Instance::configure_run(int32_t t_steps, bool use_ou, hipStream_t s)
{
    if (t_steps < 1)
        throw Error(kInvalidParameter, "t_steps must be >= 1");
    if (t_steps > 1 && !use_ou)
        throw Error(kInvalidParameter, "t_steps > 1 requires the OU background");   // dist_simulator.cpp:3225-3234
    const bool changed = t_steps != t_steps_ || use_ou != use_ou_;
    use_ou_ = use_ou;
    if (t_steps != t_steps_) {
        t_steps_ = t_steps;
        derive_params(s);
    }
    return changed;
}

// Slots and strides of the next record; slots = false: one slot (records in
// caller buffers).
void Instance::layout_record(int64_t steps, bool freq, bool stat, bool slots)
{
    const uint32_t np = npop(), tiles = (n_ + kBlock - 1) / kBlock;
    rec_slots_ = 1;
    rec_cstride_ = np;
    rec_sstride_ = np * kStatFields;
    if (!slots)
        return;
    // whole 128-byte lines per slot
    const uint32_t cs = (np + 31u) / 32u * 32u, ss = (np * kStatFields + 15u) / 16u * 16u;
    const uint64_t slot_bytes = (uint64_t)steps * ((freq ? cs * sizeof(uint32_t) : 0) + (stat ? ss * sizeof(long long) : 0));
    uint32_t k = 1;
    while ((uint64_t)steps * tiles >= kRecMinMeets * np && k < kRecMaxSlots &&
           (uint64_t)k * kRecTilesPerSlot * np < tiles && 2 * k * slot_bytes <= kRecMaxBytes)
        k *= 2;
    if (k > 1) {
        rec_slots_ = k;
        rec_cstride_ = cs;
        rec_sstride_ = ss;
    }
}

void Instance::begin_record(int64_t step0, int64_t steps, bool freq, bool samples, uint32_t stat_mask, hipStream_t s)
{
    if (samples && samples_.empty())
        throw Error(kUnsetSampleFailure, "samples requested but not set");
    rec_step0_ = step0;
    rec_len_ = steps;
    rec_freq_ = freq;
    rec_samples_ = samples;
    rec_stat_mask_ = stat_mask;
    // The samples first: the sums' slots can do with less.
    auto take_samples = [&] {
        const size_t m = (size_t)steps * samples_.size();
        rec_spike_.resize(m);
        rec_v_.resize(m);
        rec_isyn_.resize(m);
        rec_iou_.resize(m);
        rec_spike_.mutable_gpu_data();
        rec_v_.mutable_gpu_data();
        rec_isyn_.mutable_gpu_data();
        rec_iou_.mutable_gpu_data();
    };
    auto allocate = [&](bool slots) {
        layout_record(steps, freq, stat_mask != 0, slots);
        if (stat_mask != 0) {
            rec_stat_.resize(stat_slots());
            rec_stat_.mutable_gpu_data();
        }
        if (freq) {
            rec_counts_.resize(count_slots());
            rec_counts_.mutable_gpu_data();
        }
    };
    try {
        if (samples) {
            try {
                take_samples();
            } catch (const Error &e) {
                if (e.code != kOutOfMemory)
                    throw;
                rec_stat_.resize(0);   // an earlier record's slots
                rec_counts_.resize(0);
                take_samples();
            }
        }
        try {
            allocate(true);
        } catch (const Error &e) {
            // no device memory for the slots: one per row, as without them
            if (e.code != kOutOfMemory || rec_slots_ == 1)
                throw;
            allocate(false);
        }
    } catch (...) {
        end_record();   // no step may write a record whose buffers are not there
        throw;
    }
    const CopyWords clear[2] = {{stat_mask != 0 ? rec_stat_.mutable_gpu_data() : nullptr, nullptr,
                                 stat_mask != 0 ? rec_stat_.size() / 4 : 0},
                                {freq ? rec_counts_.mutable_gpu_data() : nullptr, nullptr,
                                 freq ? rec_counts_.size() / 4 : 0}};
    DTB_HIP(launch_copy_words(clear, 2, s));
}

void Instance::begin_record_at(int64_t steps, bool freq, bool samples, uint32_t stat_mask, const RecordBuffers &b,
                               hipStream_t s)
{
    if (samples && samples_.empty())
        throw Error(kUnsetSampleFailure, "samples requested but not set");
    if ((freq && !b.counts) || (stat_mask != 0 && !b.stat) || (samples && !(b.spike && b.v && b.isyn && b.iou)))
        throw Error(kInvalidParameter, "record buffer missing");
    rec_step0_ = step(s);
    rec_len_ = steps;
    rec_freq_ = freq;
    rec_samples_ = samples;
    rec_stat_mask_ = stat_mask;
    rec_ext_ = b;
    rec_ext_on_ = true;
    layout_record(steps, freq, stat_mask != 0, false);
    if (stat_mask != 0)
        DTB_HIP(launch_zero_words(b.stat, (size_t)steps * npop() * kStatFields * sizeof(long long), s));
    if (freq)
        DTB_HIP(launch_zero_words(b.counts, (size_t)steps * npop() * sizeof(uint32_t), s));
}

void Instance::end_record()
{
    rec_ext_on_ = false;
    rec_ext_ = RecordBuffers{};
    rec_freq_ = rec_samples_ = false;
    rec_stat_mask_ = 0;
    rec_len_ = 0;
}

void Instance::fetch_record(HostStage &stage, uint32_t *freq, uint8_t *spike, float *v, float *isyn, float *iou,
                            float *const *means, hipStream_t s)
{
    if (rec_ext_on_)
        throw Error(kInternal, "the recording is in caller buffers");
    const uint32_t np = npop();
    const bool stats = means != nullptr && rec_stat_mask_ != 0, counts = freq && rec_freq_;
    if (stats || counts) {
        RecordRows r{};
        r.stat = rec_stat_.gpu_data();
        r.counts = rec_counts_.gpu_data();
        r.slots = rec_slots_;
        r.sstride = rec_sstride_;
        r.cstride = rec_cstride_;
        r.swidth = stats ? np * kStatFields : 0u;
        r.cwidth = counts ? np : 0u;
        std::vector<double> cnt(np, 0.0);
        if (stats) {
            const uint8_t *bl = blocked_.cpu_data();
            for (uint32_t q = 0; q < np; ++q)
                cnt[q] = (double)std::count(bl + pop_begin_[q], bl + pop_begin_[q + 1], (uint8_t)0);
        }
        const size_t row_bytes = (size_t)r.swidth * sizeof(long long) + (size_t)r.cwidth * sizeof(uint32_t);
        const int64_t most = (int64_t)std::max<size_t>(1, kCallStageBytes / row_bytes);
        unsigned char *p = stage.reserve(std::max(kCallStageBytes, row_bytes));
        for (int64_t r0 = 0; r0 < rec_len_; r0 += most) {
            const int64_t m = std::min(most, rec_len_ - r0);
            r.out_stat = reinterpret_cast<long long *>(p);
            r.out_counts = reinterpret_cast<uint32_t *>(p + (size_t)m * r.swidth * sizeof(long long));
            DTB_HIP(launch_fetch_rows(r, (uint64_t)r0, (uint64_t)m, s));
            DTB_HIP(hipStreamSynchronize(s));
            // stat_result.cpp:266-391 divides by the population size minus its
            // blocked neurons: mean = (double) sum * 2^-24 / count, as float.
            for (int k = 0; stats && k < kStatFields; ++k) {
                if (means[k] == nullptr)
                    continue;
                for (int64_t t = 0; t < m; ++t)
                    for (uint32_t q = 0; q < np; ++q)
                        means[k][(size_t)(r0 + t) * np + q] =
                            (float)((double)r.out_stat[((size_t)t * np + q) * kStatFields + k] * 0x1p-24 / cnt[q]);
            }
            if (counts)
                std::memcpy(freq + (size_t)r0 * np, r.out_counts, (size_t)m * np * sizeof(uint32_t));
        }
    }
    if (rec_samples_) {
        if (spike)
            rec_spike_.download(spike, rec_spike_.count(), s);
        if (v)
            rec_v_.download(v, rec_v_.count(), s);
        if (isyn)
            rec_isyn_.download(isyn, rec_isyn_.count(), s);
        if (iou)
            rec_iou_.download(iou, rec_iou_.count(), s);
    }
    DTB_HIP(hipStreamSynchronize(s));
}

int64_t Instance::step(hipStream_t s)
{
    int64_t v[2] = {0, 0};
    step_.download(v, 2, s);
    DTB_HIP(hipStreamSynchronize(s));
    return std::max(v[0], v[1]);
}

void Instance::set_step(int64_t step, hipStream_t s)
{
    const int64_t v[2] = {step, step};
    step_.upload(v, 2, s);
    DTB_HIP(hipStreamSynchronize(s));
}

void Instance::counters(int64_t *step, uint64_t *events, uint64_t *spikes, hipStream_t s)
{
    std::vector<unsigned long long> w(counters_.count());
    int64_t st[2] = {0, 0};
    counters_.download(w.data(), w.size(), s);
    step_.download(st, 2, s);
    DTB_HIP(hipStreamSynchronize(s));
    if (step)
        *step = std::max(st[0], st[1]);
    unsigned long long c[2] = {0, 0};
    for (size_t k = 0; k < w.size(); k += 2) {
        c[0] += w[k];
        c[1] += w[k + 1];
    }
    if (events)
        *events = c[0];
    if (spikes)
        *spikes = c[1];
}

// The state lives in tile blocks; callers have plain arrays.  A kernel
// gathers (scatters) the fields and folds the pending delta, in device
// arrays of as many neurons as fit (usually all), and each field is one copy:
// 2M neurons read in 6 ms, 28 ms with the fold on the host.
struct Instance::StateStage {
    unsigned char *base = nullptr;   // device memory, or null: the arrays are pinned host memory
    uint32_t cap = 0;
    StateArrays a{};

    static constexpr size_t kPerNeuron = 4 + 4 + 4 + 16 + 4 + 1 + 1;
    // A small state goes through the call's pinned memory, which the kernel
    // reads or writes itself: a copy per field of 10k neurons was 250 us.
    StateStage(HostStage &host, uint32_t count)
    {
        unsigned char *p = nullptr;
        constexpr uint32_t kHostNeurons = kCallStageBytes / kPerNeuron;
        // at most 1M neurons (34 MB) at a time; fewer when memory is short,
        // and in the end the pinned memory's
        for (cap = std::min<uint32_t>(count, 1u << 20); cap > kHostNeurons && p == nullptr;) {
            try {
                p = base = static_cast<unsigned char *>(devmem::alloc((size_t)cap * kPerNeuron));
            } catch (const Error &e) {
                if (e.code != kOutOfMemory && !devmem::NoAlloc::active())
                    throw;
                cap /= 2;
            }
        }
        if (p == nullptr) {
            cap = std::min(count, kHostNeurons);
            p = host.reserve(kCallStageBytes);
        }
        a.J = reinterpret_cast<float4 *>(p);
        a.V = reinterpret_cast<float *>(p + (size_t)cap * 16);
        a.t = reinterpret_cast<int32_t *>(p + (size_t)cap * 20);
        a.iou = reinterpret_cast<float *>(p + (size_t)cap * 24);
        a.isyn = reinterpret_cast<float *>(p + (size_t)cap * 28);
        a.f = p + (size_t)cap * 32;
        a.emitted = p + (size_t)cap * 33;
    }
    ~StateStage() { devmem::release(base); }
    StateStage(const StateStage &) = delete;
    StateStage &operator=(const StateStage &) = delete;
};

void Instance::read_state(HostStage &stage, float *V, int32_t *t, uint8_t *f, uint8_t *emitted, float *iou, float *J, float *isyn,
                          hipStream_t s)
{
    StateStage st(stage, n_);
    StateArrays a = st.a;
    a.V = V ? a.V : nullptr;
    a.t = t ? a.t : nullptr;
    a.iou = iou ? a.iou : nullptr;
    a.J = J ? a.J : nullptr;
    a.isyn = isyn ? a.isyn : nullptr;
    a.f = f ? a.f : nullptr;
    a.emitted = emitted ? a.emitted : nullptr;
    for (uint32_t b = 0; b < n_; b += st.cap) {
        const size_t m = std::min(st.cap, n_ - b);
        DTB_HIP(launch_read_state(state_view(), b, (uint32_t)m, a, s));
        if (st.base == nullptr)
            DTB_HIP(hipStreamSynchronize(s));
        auto copy = [&](auto *dst, const auto *src, size_t per) {
            if (dst != nullptr && st.base == nullptr)
                std::memcpy(dst + (size_t)b * per, src, m * per * sizeof(*dst));
            else if (dst != nullptr)
                DTB_HIP(hipMemcpyAsync(dst + (size_t)b * per, src, m * per * sizeof(*dst), hipMemcpyDeviceToHost, s));
        };
        copy(V, a.V, 1);
        copy(t, a.t, 1);
        copy(f, a.f, 1);
        copy(emitted, a.emitted, 1);
        copy(iou, a.iou, 1);
        copy(J, reinterpret_cast<const float *>(a.J), 4);
        copy(isyn, a.isyn, 1);
    }
    DTB_HIP(hipStreamSynchronize(s));
}

void Instance::write_state(HostStage &stage, const float *V, const int32_t *t, const uint8_t *f, const float *iou, const float *J,
                           hipStream_t s)
{
    if (!V && !t && !f && !iou && !J)
        return;
    StateStage st(stage, n_);
    StateArrays a = st.a;
    a.V = V ? a.V : nullptr;
    a.t = t ? a.t : nullptr;
    a.iou = iou ? a.iou : nullptr;
    a.J = J ? a.J : nullptr;
    a.f = f ? a.f : nullptr;
    for (uint32_t b = 0; b < n_; b += st.cap) {
        const size_t m = std::min(st.cap, n_ - b);
        auto copy = [&](auto *dst, const auto *src, size_t per) {
            if (src != nullptr && st.base == nullptr)
                std::memcpy(dst, src + (size_t)b * per, m * per * sizeof(*src));
            else if (src != nullptr)
                DTB_HIP(hipMemcpyAsync(dst, src + (size_t)b * per, m * per * sizeof(*src), hipMemcpyHostToDevice, s));
        };
        copy(a.V, V, 1);
        copy(a.t, t, 1);
        copy(a.f, f, 1);
        copy(a.iou, iou, 1);
        copy(reinterpret_cast<float *>(a.J), J, 4);
        DTB_HIP(launch_write_state(state_view(), b, (uint32_t)m, a, s));
        if (st.base == nullptr)
            DTB_HIP(hipStreamSynchronize(s));   // the next neurons go into the same memory
    }
    DTB_HIP(hipStreamSynchronize(s));
}

void Instance::ensure_queue(uint64_t slots)
{
    slots = std::max<uint64_t>(slots, 1);
    if (slots > qslots_ || queue_.count() == 0) {
        queue_.resize((size_t)(2 * slots + kQueuePrefetch));
        queue_.mutable_gpu_data();
        qslots_ = slots;
    }
}

void Instance::clear_spill(hipStream_t s)
{
    DTB_HIP(hipMemsetAsync(spill_.mutable_gpu_data(), 0, spill_.size(), s));
}

InstDev Instance::dev(uint32_t tile_base, bool gather, bool direct, bool pull, uint32_t defer_min, bool passes)
{
    InstDev d{};
    if (passes) {
        if (!passes_built() || gather || direct)
            throw Error(kInternal, "binning by a launch of its own needs the pass lists and queues");
        d.passes = passes_.mutable_gpu_data();
        d.pass_count = pass_count_.mutable_gpu_data();
        d.passcap = passcap_;
    }
    if (direct) {
        if (!direct_built() || gather || !pull)
            throw Error(kInternal, "direct propagation needs the tile offsets, the in-edges and no gather");
        d.tidx = tidx_.gpu_data();
    }
    if (pull) {
        if (!pull_built_ || gather)
            throw Error(kInternal, "pull propagation needs the in-edges and no gather");
        d.crec = crec_.gpu_data();
        d.cptr = cptr_.gpu_data();
        d.defer_min = defer_min;
    }
    if (gather) {
        if (!gather_built_)
            throw Error(kInvalidParameter, "gather buffers not built");
        d.segidx = segidx_.gpu_data();
        d.grec = grec_.gpu_data();
        d.fired = fired_.mutable_gpu_data();
        d.fcount = fcount_.mutable_gpu_data();
        d.ngroups = ngroups(gather_bits_);
        d.fcap = fired_capacity();
    }
    d.prm = prm_.gpu_data();
    d.cls = cls_.gpu_data();
    d.pmask = dense_params_ ? ~(uint32_t)(kBlock - 1) : 0u;
    d.blocked = blocked_.gpu_data();
    d.state = state_.mutable_gpu_data();
    d.bits = reinterpret_cast<unsigned long long *>(step_.mutable_gpu_data() + kStepPad);
    d.dlt = dlt_.mutable_gpu_data();
    d.spill = spill_.mutable_gpu_data();
    d.queue = queue_.mutable_gpu_data();
    d.qslots = qslots_;
    d.rowptr = rowptr_.gpu_data();
    d.col = col_.gpu_data();
    d.w = w_.gpu_data();
    d.wfmt = wfmt_;
    d.pops = pops_.gpu_data();
    d.rec_counts = (rec_freq_ && rec_len_ > 0) ? (rec_ext_on_ ? rec_ext_.counts : rec_counts_.mutable_gpu_data())
                                                : nullptr;
    d.rec_stat = (rec_stat_mask_ != 0 && rec_len_ > 0) ? (rec_ext_on_ ? rec_ext_.stat : rec_stat_.mutable_gpu_data())
                                                       : nullptr;
    d.stat_mask = rec_stat_mask_;
    d.rec_slots = rec_slots_;
    d.rec_cstride = rec_cstride_;
    d.rec_sstride = rec_sstride_;
    d.wave_ctr = counters_.mutable_gpu_data();
    d.step = step_.mutable_gpu_data();
    d.seed = seed_;
    d.rec_step0 = rec_step0_;
    d.n = n_;
    d.npop = npop();
    d.rec_len = (uint32_t)rec_len_;
    d.t_steps = t_steps_;
    d.use_ou = use_ou_ ? 1 : 0;
    d.tile_base = tile_base;
    d.ntiles = (n_ + kBlock - 1) / kBlock;
    return d;
}

TileDesc Instance::tile_desc(uint32_t t, const InstDev &d, const InstDev *inst, uint32_t idx, uint32_t pop0,
                             uint64_t qoff, uint32_t qcap)
{
    TileDesc r{};
    r.begin = t * kBlock;
    r.count = std::min<uint32_t>(kBlock, n_ - r.begin);
    r.state = d.state + (size_t)t * kStateBytes;
    r.cls = d.cls + r.begin;
    r.inst = inst;
    r.inst_idx = idx;
    r.step = d.step;
    r.bits = d.bits + (size_t)t * kBitWords;
    r.rowptr = d.rowptr + r.begin;
    r.seed = d.seed;
    r.queue = d.queue + qoff;
    r.qslots = d.qslots;
    r.qcap = qcap;
    r.dlt = d.dlt + r.begin;
    r.pop0 = pop0;
    r.ntiles = d.ntiles;
    r.flags = (d.use_ou ? kTileOu : 0u) | (d.crec ? kTilePull : 0u) | (d.segidx ? kTileGather : 0u) |
              (d.t_steps == 1 ? kTileOneSub : 0u) | (d.rec_stat ? kTileStat : 0u);
    if (tile_cls_[t] != 0u) {
        r.flags |= kTileUniform;
        r.prm = d.prm + (tile_cls_[t] - 1u);
    } else {
        r.prm = d.prm + (r.begin & d.pmask);
    }
    if (r.begin + r.count <= pop_begin_[pop0 + 1]) {
        r.flags |= kTileOnePop;
        if (d.use_ou && ou_on_[pop0]) {
            r.flags |= kTileOuOn;
            const PopDev &pop = pops_.cpu_data()[pop0];
            r.f1 = pop.f1;
            r.f2s = pop.f2s;
            r.mu = pop.mu;
        }
    }
    return r;
}

SampleRecDev Instance::sample_rec()
{
    SampleRecDev r{};
    if (rec_samples_ && rec_len_ > 0 && rec_ext_on_) {
        r.spike = rec_ext_.spike;
        r.v = rec_ext_.v;
        r.isyn = rec_ext_.isyn;
        r.iou = rec_ext_.iou;
        r.nsample = (uint32_t)samples_.size();
    } else if (rec_samples_ && rec_len_ > 0) {
        r.spike = rec_spike_.mutable_gpu_data();
        r.v = rec_v_.mutable_gpu_data();
        r.isyn = rec_isyn_.mutable_gpu_data();
        r.iou = rec_iou_.mutable_gpu_data();
        r.nsample = (uint32_t)samples_.size();
    }
    return r;
}

// ---------------------------------------------------------------------------

}  // namespace dtb
