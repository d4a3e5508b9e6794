// dtb_engine_loop.cpp -- the step engine: instance tables, launch sequence,
// HIP-graph replay and kernel timing (tools/dist_simulator.cpp:2072-2315 is
// the reference per-step loop this replaces for one GPU).
#include <algorithm>
#include <cstring>
#include <vector>

#include "dtb_engine.hpp"
#include "dtb_kernels.hpp"

namespace dtb {

Engine::Engine(int device) : device_(device)
{
    int count = 0;
    DTB_HIP(hipGetDeviceCount(&count));
    if (device < 0 || device >= count)
        throw Error(kNoDevice, "device index out of range");
    DTB_HIP(hipSetDevice(device));
    DTB_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
    DTB_HIP(hipStreamCreateWithFlags(&admit_stream_, hipStreamNonBlocking));
    d_ctl_.resize(1);
    d_ctl_.mutable_gpu_data();
    d_queues_.resize(1);
    d_queues_.mutable_gpu_data();
}

Engine::~Engine()
{
    drop_graphs();
    insts_.clear();
    if (stream_)
        (void)hipStreamDestroy(stream_);
    if (admit_stream_)
        (void)hipStreamDestroy(admit_stream_);
}

int Engine::add(std::unique_ptr<Instance> inst)
{
    // The instance's queues are allocated now, so that running out of device
    // memory shows up when it is added, not in the middle of a later run.
    DTB_HIP(hipSetDevice(device_));
    inst->ensure_queue(queue_slots(*inst));
    if (use_gather(*inst))
        inst->ensure_gather(admit_stream_);
    else
        try_pull(*inst, admit_stream_);
    // Beside the steps of the others, like the in-edges (a table build would
    // do it on their stream).
    if (inst->pull_built() && direct_by_rules(inst.get()))
        try_direct(*inst, admit_stream_);
    for (size_t i = 0; i < insts_.size(); ++i)
        if (!insts_[i]) {
            insts_[i] = std::move(inst);
            routes_changed();
            staged_.insert((int)i);
            return (int)i;
        }
    insts_.push_back(std::move(inst));
    routes_changed();
    staged_.insert((int)insts_.size() - 1);
    return (int)insts_.size() - 1;
}

std::unique_ptr<Instance> Engine::remove(int id)
{
    if (id < 0 || (size_t)id >= insts_.size() || !insts_[id])
        throw Error(kInvalidParameter, "no such instance");
    settle();
    sync();
    routes_changed();
    staged_.erase(id);
    return std::move(insts_[id]);
}

Instance *Engine::get(int id)
{
    if (id < 0 || (size_t)id >= insts_.size() || !insts_[id])
        throw Error(kInvalidParameter, "no such instance");
    return insts_[id].get();
}

size_t Engine::active() const
{
    size_t k = 0;
    for (auto &p : insts_)
        k += p ? 1 : 0;
    return k;
}

void Engine::set_schedule(uint32_t pass_k, int layout)
{
    if (pass_k != 1 && pass_k != 2 && pass_k != 4)
        throw Error(kInvalidParameter, "pass size must be 1, 2 or 4 synapses per lane");
    if (layout != kLayoutAuto && layout != kLayoutDense && layout != kLayoutSpread && layout != kLayoutGather)
        throw Error(kInvalidParameter, "unknown propagation layout");
    if (pass_k != pass_k_ || layout != count_layout_ || tuned_ != Tuned::no) {
        pass_k_ = pass_k;
        count_layout_ = layout;
        tuned_ = Tuned::no;
        routes_changed();   // graphs hold the old kernel; counts move to the new layout
    }
}

bool Engine::use_gather(const Instance &p) const
{
    return p.gather_allowed() && count_layout_ == kLayoutGather;
}

bool Engine::try_direct(Instance &p, hipStream_t s)
{
    if (p.direct_built())
        return true;
    if (devmem::NoAlloc::active())
        return false;
    try {
        p.ensure_direct(s);
        ++tables_built_;
        return true;
    } catch (const Error &e) {
        // without device memory for the offsets the instance keeps queues
        // (same results)
        if (e.code != kOutOfMemory)
            throw;
        return false;
    }
}

bool Engine::direct_by_rules(const Instance *joining) const
{
    uint64_t tiles = 0;
    auto wanted = [&](const Instance &p) {
        tiles += (p.n() + kBlock - 1) / kBlock;
        return wants_direct(p);
    };
    if (joining && !wanted(*joining))
        return false;
    for (auto &p : insts_)
        if (p && !wanted(*p))
            return false;
    return tiles <= (step_mode() == StepMode::direct ? kDirectTilesStay : kDirectTiles);
}

bool Engine::want_direct()
{
    if (!direct_by_rules() || direct_short_.holds(devmem::cached_bytes(device_)))
        return false;
    // an engine holds offsets or pass lists, not both (the old tables,
    // settled by the caller, were the last to use the lists)
    for (auto &p : insts_)
        if (p && !tuning_ && !devmem::NoAlloc::active())
            p->release_passes();
    for (auto &p : insts_) {
        if (!p)
            continue;
        try_pull(*p, stream_);
        if (!p->pull_built() || !try_direct(*p, stream_)) {
            if (!devmem::NoAlloc::active())
                direct_short_.failed(p->pull_built() ? p->direct_bytes() : p->pull_bytes());
            return false;
        }
    }
    return true;
}

bool Engine::want_bin_launch()
{
    uint64_t tiles = 0;
    double segments = 0.0, synapses = 0.0, shared = 0.0;   // tile segments of all rows, their synapses, shared ones
    auto queued = [&](size_t i) { return insts_[i] && !use_gather(*insts_[i]); };
    for (size_t i = 0; i < insts_.size(); ++i)
        if (queued(i)) {
            const double t = (insts_[i]->n() + kBlock - 1) / kBlock;
            tiles += (uint64_t)t;
            segments += insts_[i]->row_coverage() * t * insts_[i]->n();
            synapses += (double)insts_[i]->nsyn();
            shared += insts_[i]->shared_segments();
        }
    const bool rules = tiles >= kBinLaunchTiles && 2.0 * segments <= synapses && shared >= kBinLaunchShared;
    const bool want = tiles > 0 && (split_ || (rules && tuned_ != Tuned::named)) &&
                      !passes_short_.holds(devmem::cached_bytes(device_));
    for (size_t i = 0; i < insts_.size() && want; ++i) {
        if (!queued(i) || insts_[i]->passes_built())
            continue;
        if (devmem::NoAlloc::active())
            return false;
        try {
            insts_[i]->ensure_passes();
            ++tables_built_;
        } catch (const Error &e) {
            // without device memory for the lists the tiles bin their own
            // rows (same results)
            if (e.code != kOutOfMemory)
                throw;
            for (auto &p : insts_)
                if (p)
                    p->release_passes();
            passes_short_.failed(insts_[i]->pass_bytes());
            return false;
        }
    }
    return want;
}

bool Engine::any_gather() const
{
    for (auto &p : insts_)
        if (p && use_gather(*p))
            return true;
    return false;
}

bool Engine::gather_possible() const
{
    for (auto &p : insts_)
        if (p && p->gather_allowed())
            return true;
    return false;
}

void Engine::autotune(int64_t trial_steps, uint32_t *best_k, int *best_layout, float *us)
{
    if (trial_steps < 1)
        throw Error(kInvalidParameter, "autotune needs at least one step per trial");
    if (active() == 0)
        throw Error(kInvalidParameter, "autotune needs an instance to step");
    static const uint32_t ks[7] = {1, 2, 4, 1, 2, 4, kPassKDefault};
    static const int layouts[7] = {kLayoutDense, kLayoutDense, kLayoutDense, kLayoutSpread,
                                   kLayoutSpread, kLayoutSpread, kLayoutGather};
    // Without an instance that allows gather (or device memory for its
    // buffers) the seventh turn runs the default schedule and is not a
    // candidate, so the number of steps does not depend on the networks.
    int nc = gather_possible() ? 7 : 6;
    auto set_candidate = [&](int s) {
        set_schedule(ks[s], layouts[s]);
        const Tuned t = layouts[s] == kLayoutDense && ks[s] == kPassKDefault ? Tuned::automatic : Tuned::named;
        if (t != tuned_) {
            tuned_ = t;
            routes_changed();
        }
    };
    // The cost of a step follows the network's activity, which drifts and
    // bursts; so the schedules take turns in short windows (kAutotuneWindow
    // timed steps, after 2 steps that apply the schedule) over the whole
    // tuning period, and their totals are compared.  A first untimed turn
    // loads every kernel variant (and builds the gather offsets).
    const int64_t rounds = (trial_steps + kAutotuneWindow - 1) / kAutotuneWindow;
    double t_sum[7] = {0, 0, 0, 0, 0, 0, 0};
    // The gather buffers, tile offsets and pass lists stay built between their
    // turns (a table build would otherwise return them at every other turn
    // and build them again); the first table build after the tuning returns
    // what the winner does not use.
    struct Tuning {
        bool &flag;
        explicit Tuning(bool &f) : flag(f) { flag = true; }
        ~Tuning() { flag = false; }
    } tuning(tuning_);
    for (int64_t r = -1; r < rounds; ++r) {
        for (int s = 0; s < 7; ++s) {
            if (s < nc)
                set_candidate(s);
            else
                set_schedule(kPassKDefault, kLayoutDense);
            try {
                run(2, 0);   // applies the schedule (rebuild) outside the timed span
            } catch (const Error &e) {
                // the gather buffers did not fit: drop the candidate (the
                // failed table build is redone by the next run)
                if (e.code != kOutOfMemory || layouts[s] != kLayoutGather || s >= nc)
                    throw;
                nc = 6;
                set_schedule(kPassKDefault, kLayoutDense);
                run(2, 0);
            }
            if (r < 0)
                continue;
            float ms = 0.0f;
            run_span(kAutotuneWindow, 0, &ms);
            t_sum[s] += ms;
        }
    }
    int bi = 0;
    for (int i = 1; i < nc; ++i)
        if (t_sum[i] < t_sum[bi])
            bi = i;
    if (us)
        for (int i = 0; i < 7; ++i)
            us[i] = i < nc ? (float)(t_sum[i] * 1e3 / (double)(rounds * kAutotuneWindow)) : 0.0f;
    const uint32_t bk = ks[bi];
    const int bl = layouts[bi];
    set_candidate(bi);
    dirty_ = true;   // the next table build returns what is no longer used
    if (best_k)
        *best_k = bk;
    if (best_layout)
        *best_layout = bl;
}

void Engine::set_pull(bool on, uint32_t defer_min)
{
    if (on != pull_on_ || defer_min != defer_min_) {
        pull_on_ = on;
        defer_min_ = defer_min;
        routes_changed();
    }
}

void Engine::try_pull(Instance &p, hipStream_t s)
{
    if (!pull_on_ || p.pull_built() || !p.pull_allowed())
        return;
    try {
        p.ensure_pull(s);
    } catch (const Error &e) {
        // without device memory for the in-edges the instance keeps queues
        // with spill accumulators (same results, slower volleys)
        if (e.code != kOutOfMemory)
            throw;
    }
}

CtlTotals Engine::propagation_stats()
{
    StepCtl c{};
    d_ctl_.download(&c, 1, stream_);
    DTB_HIP(hipStreamSynchronize(stream_));
    CtlTotals t{};
    for (uint32_t k = 0; k < kCtlSlots; ++k) {
        t.spilled += c.slot[k].spilled;
        t.deferred += c.slot[k].deferred;
        t.pulled += c.slot[k].pulled;
    }
    return t;
}

uint64_t Engine::queue_slots(const Instance &p) const
{
    uint64_t slots = 0;
    for (uint32_t b = 0, t = 0; b < p.n(); b += kBlock, ++t)
        slots += queue_capacity(p.tile_synapses(t));
    return slots;
}

void Engine::set_queue_capacity(uint32_t floor, uint32_t shift)
{
    if (shift > 31)
        throw Error(kInvalidParameter, "queue capacity shift must be at most 31");
    queue_floor_ = floor;
    queue_shift_ = shift;
    routes_changed();
}

uint32_t Engine::queue_capacity(uint32_t synapses) const
{
    // Every row fires at most once per step, so `synapses` entries always
    // suffice; fewer keep the queues small, and the synapses past the
    // capacity take the spill path.
    const uint64_t c = (uint64_t)queue_floor_ + (synapses >> queue_shift_);
    return (uint32_t)std::min<uint64_t>(std::min<uint64_t>(synapses, c), 0x7fffffffull);
}

void Engine::drop_graphs()
{
    for (int p = 0; p < 2; ++p)
        if (graph_[p]) {
            (void)hipGraphExecDestroy(graph_[p]);
            graph_[p] = nullptr;
            graph_steps_[p] = 0;
        }
}

QueueSet Engine::queues()
{
    QueueSet q{};
    q.tile = d_qtiles_.gpu_data();
    q.ctl = d_ctl_.mutable_gpu_data();
    q.count = d_qcnt_.mutable_gpu_data();
    q.ntiles = ntiles_;
    q.cshift = cshift_;
    return q;
}

namespace {
// Workgroups of k_bin for an instance of nt tiles.
uint32_t bin_parts(uint32_t nt)
{
    return std::min(kBinGroups, (nt + kBinTiles - 1) / kBinTiles);
}

// Place in the launch of direct tile j of n.  Workgroups are dealt to the 8
// XCDs by index mod 8: each XCD gets a contiguous range of the tiles, so tiles
// that share cache lines of a row's offsets and synapses meet in one L2.
size_t dealt(size_t j, size_t n)
{
    const size_t q = n >> 3, r = n & 7u;   // the first r ranges have q + 1 tiles
    const size_t x = j < r * (q + 1) ? j / (q + 1) : r + (j - r * (q + 1)) / q;
    return (j - (x * q + std::min(x, r))) * 8 + x;
}
}  // namespace

void Engine::rebuild()
{
    settle();   // the queues are reallocated below; nothing pending may be lost
    DTB_HIP(hipStreamSynchronize(stream_));   // the last tables have left their staging memory
    staged_.clear();
    std::vector<InstDev> table;
    size_t ninst = 0, ntile = 0, sample_set = 0, group_max = 0, bin_max = 0;
    for (auto &p : insts_)
        if (p) {
            const uint32_t nt = (p->n() + kBlock - 1) / kBlock;
            ++ninst;
            ntile += nt;
            sample_set += p->samples().size();
            bin_max += bin_parts(nt);
            if (use_gather(*p))
                group_max += p->ngroups(p->gather_bits());
        }
    // The tables only grow (the kernels get their lengths as arguments), so
    // a rebuild after the largest set so far allocates nothing.
    auto grow = [](auto &buf, size_t n) {
        if (buf.count() < std::max<size_t>(n, 1))
            buf.resize(std::max<size_t>(n, 1));
    };
    grow(d_insts_, ninst);
    // The tables go to the device from pinned memory.  The tiles' are written
    // there at once (by way of vectors, 2M neurons' 1.1 MB made a rebuild
    // 60-100 us longer); it holds every sample that is set, recorded or not,
    // so a recording that follows takes no pinned memory (dtb_run_noalloc).
    TileDesc *tiles = reinterpret_cast<TileDesc *>(
        tables_stage_.reserve(ntile * (sizeof(TileDesc) + sizeof(QueueTile)) + ninst * (sizeof(InstDev) + sizeof(SampleRecDev)) +
                              sizeof(QueueSet) + group_max * sizeof(GroupDesc) + bin_max * sizeof(BinDesc) +
                              sample_set * sizeof(SampleDev)));
    QueueTile *qtiles = reinterpret_cast<QueueTile *>(tiles + ntile);
    size_t tile = 0;   // written so far
    std::vector<GroupDesc> groups;
    std::vector<SampleDev> samples;
    std::vector<SampleRecDev> recs;
    tile_base_.assign(insts_.size(), 0u);
    stat_ = false;
    uint64_t total = 0;
    double coverage = 0.0;
    std::vector<BinDesc> bins;
    bin_tiles_ = 0;
    uint32_t fmt = kWeightAny + 1;   // the instances' common weight format (kWeightAny: mixed)
    const bool dir = want_direct();   // every instance, or none
    const bool bin_launch = !dir && want_bin_launch();
    std::vector<CopyWords> put;   // the tables' copies, below
    for (size_t slot = 0; slot < insts_.size(); ++slot) {
        Instance *p = insts_[slot].get();
        if (!p)
            continue;
        const uint32_t idx = (uint32_t)table.size();
        tile_base_[slot] = (uint32_t)tile;
        stat_ = stat_ || p->stat_mask() != 0;
        fmt = fmt == kWeightAny + 1 || fmt == p->weight_format() ? p->weight_format() : kWeightAny;
        uint64_t qtotal = 0;   // this instance's queue slots per parity
        for (uint32_t b = 0, t = 0; b < p->n(); b += kBlock, ++t) {
            const uint32_t cap = queue_capacity(p->tile_synapses(t));
            qtiles[tile + t] = QueueTile{qtotal, cap, 0u};
            qtotal += cap;
        }
        // Each instance owns its queues (both parities and the read-ahead
        // slack), so instances of any size come and go without one large
        // engine-wide block.
        p->ensure_queue(qtotal);
        const bool gat = use_gather(*p);
        if (gat) {
            p->ensure_gather(stream_);
            const uint32_t gb = p->gather_bits();
            for (uint32_t g = 0; g < p->ngroups(gb); ++g)
                groups.push_back(GroupDesc{idx, g, std::min<uint32_t>(1u << gb, p->n() - (g << gb)), gb});
        } else if (p->gather_built() && !tuning_) {
            // the old tables (settled above) were the last to use them;
            // device memory returns to the cache
            p->release_gather();
        }
        if (!gat)
            try_pull(*p, stream_);
        const bool pl = !gat && pull_on_ && p->pull_built();
        if (!dir && !tuning_)
            p->release_direct();   // (the old tables, settled above, were the last to use it)
        const bool passes = bin_launch && !gat;
        if (!passes && !tuning_ && !devmem::NoAlloc::active())
            p->release_passes();
        table.push_back(p->dev(tile_base_[slot], gat, dir, pl, defer_min_, passes));
        if (passes)
            put.push_back(p->pass_count_words());
        const auto &pb = p->pop_begin();
        uint32_t q = 0;
        for (uint32_t b = 0, t = 0; b < p->n(); b += kBlock, ++t) {
            while (pb[q + 1] <= b)
                ++q;
            const QueueTile &qt = qtiles[tile];
            tiles[dir ? dealt(tile, ntile) : tile] =
                p->tile_desc(t, table.back(), d_insts_.gpu_data() + idx, idx, q, qt.off, qt.cap);
            ++tile;
        }
        recs.push_back(p->sample_rec());
        if (recs.back().nsample > 0) {
            const auto &ids = p->samples();
            for (uint32_t k = 0; k < ids.size(); ++k)
                samples.push_back(SampleDev{idx, ids[k], k, 0});
        }
        if (!gat && !dir) {
            total += p->n();
            coverage += p->row_coverage() * p->n();
            if (passes) {
                const uint32_t nt = (p->n() + kBlock - 1) / kBlock;
                bin_tiles_ = std::max(bin_tiles_, nt);
                const uint32_t parts = bin_parts(nt);
                for (uint32_t k = 0; k < parts; ++k)
                    bins.push_back(BinDesc{d_insts_.gpu_data() + idx, k, parts});
            }
        }
    }
    if (total > 0xffffffffull || ntile > 0xffffffffull)
        throw Error(kInvalidParameter, "too many neurons in one engine");
    ninst_ = (uint32_t)table.size();
    wfmt_ = fmt > kWeightAny ? kWeightF32 : fmt;
    ntiles_ = (uint32_t)ntile;
    ngroups_ = (uint32_t)groups.size();
    nsamples_ = (uint32_t)samples.size();
    grow(d_groups_, groups.size());
    grow(d_tiles_, ntile);
    grow(d_qtiles_, ntile);
    // sized by the samples set, recorded or not: a recording run then finds
    // the table built
    grow(d_samples_, sample_set);
    grow(d_recs_, recs.size());
    // Auto: dense, unless rows reach most of their instance's tiles (the
    // reservations of many waves then meet on the same lines).  Measured with
    // the tile's passes dealt to all its waves, dense was as fast or faster
    // up to a coverage of 0.92 (in-degree 5000 on 500k neurons), so the
    // threshold sits above that; the autotuner measures instead of guessing.
    if (count_layout_ == kLayoutDense || count_layout_ == kLayoutGather)
        cshift_ = kCountShiftDense;
    else if (count_layout_ == kLayoutSpread)
        cshift_ = kCountShiftSpread;
    else
        cshift_ = (total > 0 && coverage / (double)total > kSpreadCoverage) ? kCountShiftSpread : kCountShiftDense;
    grow(d_qcnt_, count_words(2 * std::max<size_t>(ntile, 1), cshift_));
    nbins_ = (uint32_t)bins.size();
    mode_ = dir && ntiles_ > 0 ? StepMode::direct : nbins_ > 0 ? StepMode::bin_launch : StepMode::tile_bin;
    grow(d_bins_, bins.size());
    d_bins_.mutable_gpu_data();
    // Allocate (zero-filled) everything the step kernels touch before any
    // capture: no allocation may happen while a graph is being recorded.
    d_qcnt_.mutable_gpu_data();
    d_samples_.mutable_gpu_data();
    d_recs_.mutable_gpu_data();
    d_groups_.mutable_gpu_data();
    // All tables in one launch: a copy call each and the wait for the last
    // were 60 of a short call's 240 us.
    const std::vector<QueueSet> qset(1, queues());
    unsigned char *at = reinterpret_cast<unsigned char *>(qtiles + ntile);
    auto put_table = [&](auto &buf, const auto *src, size_t n) {
        static_assert(sizeof(src[0]) % 4 == 0, "tables are whole words");
        if (n > 0)
            put.push_back(CopyWords{buf.mutable_gpu_data(), src, n * sizeof(src[0]) / 4});
    };
    auto stage_table = [&](auto &buf, const auto &v) {
        std::memcpy(at, v.data(), v.size() * sizeof(v[0]));
        put_table(buf, reinterpret_cast<decltype(v.data())>(at), v.size());
        at += v.size() * sizeof(v[0]);
    };
    put_table(d_tiles_, tiles, ntile);
    put_table(d_qtiles_, qtiles, ntile);
    stage_table(d_insts_, table);
    stage_table(d_bins_, bins);
    stage_table(d_queues_, qset);
    stage_table(d_groups_, groups);
    stage_table(d_samples_, samples);
    stage_table(d_recs_, recs);
    put.push_back(CopyWords{d_qcnt_.mutable_gpu_data(), nullptr, d_qcnt_.size() / 4});
    DTB_HIP(launch_copy_words(put.data(), (int)put.size(), stream_));
    GraphKey key{};
    key.tiles = d_tiles_.gpu_data();
    key.insts = d_insts_.gpu_data();
    key.queues = d_queues_.gpu_data();
    key.qtiles = d_qtiles_.gpu_data();
    key.qcnt = d_qcnt_.gpu_data();
    key.bins = d_bins_.gpu_data();
    key.groups = d_groups_.gpu_data();
    key.samples = d_samples_.gpu_data();
    key.recs = d_recs_.gpu_data();
    key.ntiles = ntiles_;
    key.mode = (uint32_t)mode_;
    key.nbins = nbins_;
    key.bin_tiles = bin_tiles_;
    key.ngroups = ngroups_;
    key.nsamples = nsamples_;
    key.cshift = cshift_;
    key.pass_k = pass_k_;
    key.wfmt = wfmt_;
    key.stat = stat_;
    if (std::memcmp(&key, &graph_key_, sizeof(key)) != 0) {
        // (capturing and instantiating 64 steps takes 0.3-0.5 ms)
        drop_graphs();
        graph_key_ = key;
    }
    dirty_ = false;
}

void Engine::launch_gather_k(uint32_t par)
{
    DTB_HIP(launch_gather(d_groups_.gpu_data(), ngroups_, d_insts_.gpu_data(), par, wfmt_, nullptr, nullptr, stream_));
}

void Engine::launch_step_k(hipEvent_t *ev)
{
    // start and stop events of the i-th kernel, or none
    auto e = [&](int i) { return ev ? ev[i] : nullptr; };
    DTB_HIP(launch_gather(d_groups_.gpu_data(), ngroups_, d_insts_.gpu_data(), par_, wfmt_, e(0), e(1), stream_));
    DTB_HIP(launch_step_kernel(d_tiles_.gpu_data(), ntiles_, mode_, pass_k_, d_queues_.gpu_data(), par_, wfmt_, stat_,
                               e(2), e(3), stream_));
    DTB_HIP(launch_bin_kernel(d_bins_.gpu_data(), nbins_, bin_tiles_, d_queues_.gpu_data(), par_, wfmt_, e(4), e(5),
                              stream_));
}

void Engine::launch_aux()
{
    // par_ has already advanced: the step just run had parity par_ ^ 1 and
    // its spikes are queued in set par_.
    if (nsamples_ > 0) {
        launch_gather_k(par_);
        DTB_HIP(launch_materialize(d_tiles_.gpu_data(), ntiles_, d_insts_.gpu_data(), queues(), par_, stream_));
        DTB_HIP(launch_sample(d_insts_.gpu_data(), d_samples_.gpu_data(), nsamples_, d_recs_.gpu_data(), par_ ^ 1u,
                              stream_));
    }
}

void Engine::launch_step()
{
    launch_step_k();
    par_ ^= 1u;
    launch_aux();
}

void Engine::run(int64_t steps, int graph_chunk)
{
    if (steps < 0)
        throw Error(kInvalidParameter, "negative step count");
    DTB_HIP(hipSetDevice(device_));
    if (dirty_)
        rebuild();
    if (ninst_ == 0 || steps == 0)
        return;
    pending_ = true;
    if (graph_chunk > 1 && steps >= graph_chunk) {
        int64_t done = 0;
        while (steps - done >= graph_chunk) {
            const uint32_t p0 = par_;
            if (!graph_[p0] || graph_steps_[p0] != graph_chunk) {
                if (graph_[p0]) {
                    DTB_HIP(hipGraphExecDestroy(graph_[p0]));
                    graph_[p0] = nullptr;
                }
                hipGraph_t g = nullptr;
                DTB_HIP(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal));
                for (int k = 0; k < graph_chunk; ++k)
                    launch_step();
                DTB_HIP(hipStreamEndCapture(stream_, &g));
                DTB_HIP(hipGraphInstantiate(&graph_[p0], g, nullptr, nullptr, 0));
                DTB_HIP(hipGraphDestroy(g));
                graph_steps_[p0] = graph_chunk;
                par_ = p0;   // capture recorded the launches without running them
            }
            DTB_HIP(hipGraphLaunch(graph_[p0], stream_));
            par_ = p0 ^ (uint32_t)(graph_chunk & 1);
            done += graph_chunk;
        }
        for (; done < steps; ++done)
            launch_step();
    } else {
        for (int64_t k = 0; k < steps; ++k)
            launch_step();
    }
}

int64_t Engine::settled_step(Instance &p)
{
    DTB_HIP(hipSetDevice(device_));
    settle(false);
    int64_t *v = reinterpret_cast<int64_t *>(call_stage_.reserve(kCallStageBytes));
    const CopyWords c{v, p.step_words(), 4};
    DTB_HIP(launch_copy_words(&c, 1, stream_));
    DTB_HIP(hipStreamSynchronize(stream_));
    return std::max(v[0], v[1]);
}

void Engine::settle(bool wait)
{
    if (!pending_)
        return;
    DTB_HIP(hipSetDevice(device_));
    launch_gather_k(par_);
    DTB_HIP(launch_settle(d_tiles_.gpu_data(), ntiles_, d_insts_.gpu_data(), queues(), par_, stream_));
    // the deferred rows were folded with the rest of the pending input
    std::vector<CopyWords> clear;
    for (auto &p : insts_)
        if (p)
            clear.push_back(p->deferred_words());
    DTB_HIP(launch_copy_words(clear.data(), (int)clear.size(), stream_));
    if (wait)
        DTB_HIP(hipStreamSynchronize(stream_));
    pending_ = false;
}

void Engine::materialize()
{
    DTB_HIP(hipSetDevice(device_));
    if (dirty_)
        rebuild();
    launch_gather_k(par_);
    DTB_HIP(launch_materialize(d_tiles_.gpu_data(), ntiles_, d_insts_.gpu_data(), queues(), par_, stream_));
    DTB_HIP(hipStreamSynchronize(stream_));
}

void Engine::clear_queues(int id)
{
    get(id);
    DTB_HIP(hipSetDevice(device_));
    if (dirty_)
        rebuild();
    const uint32_t ntile = (get(id)->n() + kBlock - 1) / kBlock;
    for (uint32_t p = 0; p < 2; ++p) {
        // the counts of these tiles and the unused words between them
        const size_t first = count_slot((size_t)p * ntiles_ + tile_base_[(size_t)id], cshift_);
        const size_t last = count_slot((size_t)p * ntiles_ + tile_base_[(size_t)id] + ntile - 1, cshift_);
        DTB_HIP(hipMemsetAsync(d_qcnt_.mutable_gpu_data() + first, 0, (last + 1 - first) * sizeof(uint32_t), stream_));
    }
    get(id)->clear_spill(stream_);
    get(id)->clear_fired(stream_);
    get(id)->clear_deferred(stream_);
    DTB_HIP(hipStreamSynchronize(stream_));
}

void Engine::stat_tail(bool wait)
{
    DTB_HIP(hipSetDevice(device_));
    if (dirty_)
        rebuild();
    if (ninst_ == 0)
        return;
    launch_gather_k(par_);
    DTB_HIP(launch_materialize(d_tiles_.gpu_data(), ntiles_, d_insts_.gpu_data(), queues(), par_, stream_));
    DTB_HIP(launch_stat_tail(d_tiles_.gpu_data(), ntiles_, d_insts_.gpu_data(), par_, stream_));
    if (wait)
        DTB_HIP(hipStreamSynchronize(stream_));
}

void Engine::run_timed(int64_t steps, float *ms_step)
{
    DTB_HIP(hipSetDevice(device_));
    if (dirty_)
        rebuild();
    if (ninst_ == 0 || steps <= 0)
        return;
    pending_ = true;
    // Every kernel of a step (k_gather, k_step, k_bin: those with a grid)
    // records its own start and stop events at the dispatch boundaries, on
    // the engine stream; they are read back once per chunk so the launch
    // pipeline is not drained every step.
    const uint32_t grid[3] = {ngroups_, ntiles_, nbins_};
    const int last = nbins_ > 0 ? 2 : 1;
    const int64_t chunk = 256;
    std::vector<hipEvent_t> ev((size_t)(6 * chunk));
    for (auto &e : ev)
        DTB_HIP(hipEventCreate(&e));
    double ts = 0.0;
    for (int64_t base = 0; base < steps; base += chunk) {
        const int64_t m = std::min<int64_t>(chunk, steps - base);
        for (int64_t k = 0; k < m; ++k) {
            launch_step_k(&ev[(size_t)(6 * k)]);
            par_ ^= 1u;
            launch_aux();
        }
        DTB_HIP(hipEventSynchronize(ev[(size_t)(6 * (m - 1) + 2 * last + 1)]));
        for (int64_t k = 0; k < m; ++k)
            for (int i = 0; i < 3; ++i) {
                if (grid[i] == 0)
                    continue;
                float a = 0.0f;
                DTB_HIP(hipEventElapsedTime(&a, ev[(size_t)(6 * k + 2 * i)], ev[(size_t)(6 * k + 2 * i + 1)]));
                ts += a;
            }
    }
    for (auto &e : ev)
        DTB_HIP(hipEventDestroy(e));
    if (ms_step)
        *ms_step = (float)ts;
}

void Engine::run_span(int64_t steps, int graph_chunk, float *ms)
{
    DTB_HIP(hipSetDevice(device_));
    if (dirty_)
        rebuild();
    hipEvent_t e0 = nullptr, e1 = nullptr;
    DTB_HIP(hipEventCreate(&e0));
    DTB_HIP(hipEventCreate(&e1));
    DTB_HIP(hipEventRecord(e0, stream_));
    run(steps, graph_chunk);
    DTB_HIP(hipEventRecord(e1, stream_));
    DTB_HIP(hipEventSynchronize(e1));
    float t = 0.0f;
    DTB_HIP(hipEventElapsedTime(&t, e0, e1));
    DTB_HIP(hipEventDestroy(e0));
    DTB_HIP(hipEventDestroy(e1));
    if (ms)
        *ms = t;
}

void Engine::run_span_units(int64_t steps, int graph_chunk, float *ms, float *ms_steps)
{
    DTB_HIP(hipSetDevice(device_));
    if (dirty_)
        rebuild();
    if (steps <= 0) {
        if (ms)
            *ms = 0.0f;
        return;
    }
    // one event before the first step and one after every unit: a step run
    // eagerly, or a replayed graph chunk
    std::vector<hipEvent_t> ev;
    std::vector<int64_t> len;
    auto mark = [&]() {
        hipEvent_t e = nullptr;
        DTB_HIP(hipEventCreate(&e));
        ev.push_back(e);
        DTB_HIP(hipEventRecord(e, stream_));
    };
    try {
        mark();
        for (int64_t done = 0; done < steps;) {
            const bool chunk = graph_chunk > 1 && steps - done >= graph_chunk;
            const int64_t u = chunk ? graph_chunk : 1;
            run(u, chunk ? graph_chunk : 0);
            mark();
            len.push_back(u);
            done += u;
        }
        DTB_HIP(hipEventSynchronize(ev.back()));
        float total = 0.0f;
        int64_t k = 0;
        for (size_t i = 0; i < len.size(); ++i) {
            float t = 0.0f;
            DTB_HIP(hipEventElapsedTime(&t, ev[i], ev[i + 1]));
            total += t;
            for (int64_t j = 0; j < len[i]; ++j)
                if (ms_steps)
                    ms_steps[k++] = t / (float)len[i];
        }
        if (ms)
            *ms = total;
    } catch (...) {
        for (auto e : ev)
            (void)hipEventDestroy(e);
        throw;
    }
    for (auto e : ev)
        DTB_HIP(hipEventDestroy(e));
}

void Engine::sync()
{
    DTB_HIP(hipSetDevice(device_));
    DTB_HIP(hipStreamSynchronize(stream_));
}

}  // namespace dtb
