// dtb_types.hpp -- device-visible data layout of a simulation instance.
//
// One instance is one reference "block" (BrainBlock<float,float2>,
// include/block.hpp:782-885).  Its per-neuron state and parameters are
// structure-of-arrays in HBM; parameters that the step reads together are
// packed into float4 records so that one 64-lane wave issues 16-byte loads
// over a contiguous 1 KiB.  Many instances can be stepped by one launch: the
// kernels find their instance through small descriptor tables.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dtb {

constexpr int kBlock = 256;            // threads per workgroup (4 wave64)
constexpr int kWave = 64;
constexpr uint32_t kKindBit = 0x80000000u;   // channel-pair bit packed into the column index
constexpr uint32_t kColMask = 0x7fffffffu;
constexpr uint32_t kTileBits = 8;            // target tile = one step workgroup = 256 neurons
static_assert((1 << kTileBits) == kBlock, "a tile is one workgroup of neurons");

// Flag byte per neuron: bit 0 = membrane spike flag f (reference
// f_inner_actives_), bit 1 = spike emitted to the synapses in the last step
// (f_inner_actives_ or f_recorded_inner_actives_, dist_simulator.cpp:2118-2131).
constexpr uint8_t kFlagSpike = 1u;
constexpr uint8_t kFlagEmit = 2u;
// bit 2: J already holds the reference-visible J of the last step (set when a
// checkpoint is restored or pending input is settled); the next step uses it
// without the decay-and-delta fold.
constexpr uint8_t kFlagFolded = 4u;

// Per-population record (reference sub-block, sub_bcounts_ ranges and the
// OU_Background_Current_Param map, include/stage.hpp:14-19).
struct alignas(16) PopDev {
    uint32_t begin;     // first neuron (instance-local)
    uint32_t end;       // one past the last neuron
    float mu;           // OU mean
    float f1;           // 1 - exp(-dt/tau)
    float f2s;          // sqrt(1 - exp(-2 dt/tau)) * sigma
    uint32_t ou_on;     // OU configured for this population
    uint32_t pad0, pad1;
};

// One delivered synapse queued for its target tile: the target's index in
// the tile (bits 0..7), the channel pair (bit 8: 0 AMPA/NMDA, 1
// GABA_A/GABA_B) and the weight pair.
struct QSyn {
    uint32_t key;
    float w0, w1;
};
constexpr uint32_t kQSynKind = 1u << 8;
constexpr int64_t kMaxSynapses = (int64_t)1 << 40;
constexpr int64_t kMaxRowLength = (int64_t)1 << 31;

// Per-population statistics (stat_result.cpp:266-391): which sums a run
// records.  Each neuron's value enters as the exact integer rint(x * 2^24),
// so the sums do not depend on the order of the additions.
constexpr uint32_t kStatV = 1u;          // membrane potential (vmean)
constexpr uint32_t kStatI = 2u;          // synaptic current (imean)
constexpr uint32_t kStatReceptor = 4u;   // per-receptor currents (receptor imeans)
constexpr int kStatFields = 6;           // V, I_syn, AMPA, NMDA, GABA_A, GABA_B
// Slots of a record: one for every kRecTilesPerSlot tiles of a population (a
// line then serves about 8 x 6 atomics of 8 ns per step), at most
// kRecMaxSlots, and fewer where the slots of a record would pass kRecMaxBytes.
constexpr uint32_t kRecTilesPerSlot = 8, kRecMaxSlots = 64;
// Atomics that must meet on one line, over the record, before it has slots
// (8 ns each).
constexpr uint64_t kRecMinMeets = 1024;
constexpr uint64_t kRecMaxBytes = (uint64_t)64 << 20;

// Largest number of distinct parameter records kept as classes (2-byte class
// index per neuron); beyond it the records are stored per neuron.
constexpr size_t kMaxParamClasses = 65536;

// Parameter record of a class of neurons (80 bytes, so a tile of one class
// reads its record with two scalar loads):
//   a = (v_reset, v_th, dt_sub / C, v_leak)
//   b = (g_leak, i_ext, noise_rate, bits(refractory substeps))
//   g, v, d = g_u, V_u and the decay of (AMPA, NMDA, GABA_A, GABA_B)
struct alignas(16) ParamRec {
    float4 a, b, g, v, d;
};

// State block of a tile of 256 neurons, one after the other in memory, so a
// workgroup reaches all of its state from one base address: V, refractory
// counter (reference t_actives_), OU current (i_ou_background_stimuli_),
// flags (kFlagSpike | kFlagEmit | kFlagFolded) and J_u after the previous
// step's decay (delta pending).  The offsets fit the immediate field of a
// global load.
constexpr uint32_t kStV = 0, kStT = 1024, kStIou = 2048, kStFlag = 3072, kStJ = 3328;
constexpr uint32_t kStateBytes = 3328 + 256 * 16;   // 7424: whole 128-byte lines

// Everything a kernel needs about one instance.
struct alignas(16) InstDev {
    // Parameter records by class.  Neurons with bit-identical records share a
    // class (in practice one per population), so the step reads 2 bytes of
    // class per neuron at most instead of 80 bytes of parameters.  The record
    // of neuron i is (i & pmask) + cls[i]: pmask = 0 with shared classes; when
    // the records have more than 65536 values every neuron has its own
    // (pmask = ~0xff, cls[i] = i & 0xff, record = i).
    const ParamRec *prm;
    const uint16_t *cls;        // [n] parameter class
    const uint8_t *blocked;     // excluded from population statistics
    unsigned char *state;       // [ntiles][kStateBytes]
    float4 *dlt;                // materialised pending delta (gather, sampling, read-back)
    unsigned long long *spill;  // [2][n][4] Q23.40 sums of the synapses past a queue's capacity
    QSyn *queue;                // [2][qslots] propagation queues (+ read-ahead slack)
    uint64_t qslots;            // queue slots per parity (tile t's start: TileDesc::qoff)
    // connectivity: presynaptic-major CSR, 64-bit row offsets
    const int64_t *rowptr;      // [n+1]
    const uint32_t *col;        // [S] postsynaptic id | kKindBit
    const void *w;              // [S] weight pair in format wfmt (kWeightF32 / F16 / U8)
    // Gather propagation (null: queue propagation).  segidx[r][g] = offset in
    // row r of its first synapse whose target lies in group g or later
    // (segidx[r][ngroups] = row length).  The rows with synapses fired by the
    // launch of parity p ^ 1 are in the kFiredLists lists of set p: list s
    // takes the rows of tiles t with t % kFiredLists == s, so it never holds
    // more than fcap rows; its count is word (p * kFiredLists + s) *
    // kFiredCountStride of fcount (one cache line per count).
    const uint16_t *segidx;     // [n][ngroups + 1]
    // The synapses again as one record each (column, then the weight pair's
    // raw bits: grec_words(wfmt) 32-bit words), so a gathered segment is one
    // contiguous stream instead of two.
    const uint32_t *grec;       // [S][grec_words(wfmt)]
    uint32_t *fired;            // [2][kFiredLists][fcap]
    uint32_t *fcount;           // [2][kFiredLists][kFiredCountStride]
    // Direct propagation (null tidx: off; never together with gather).
    // tidx[r][t] = offset in row r of its first synapse whose target lies in
    // tile t or later (tidx[r][ntiles] = row length).  A tile takes its input
    // straight from the rows of the step before: it reads the emitted bits of
    // every tile and, per emitted row, the row's segment for itself.
    const uint16_t *tidx;       // [n][ntiles + 1]
    // Binning by k_bin (null passes: the tiles bin their rows): the passes of
    // a step's rows, (first synapse << 8) | (synapses - 1), in kFiredLists
    // lists of passcap entries, tile t's on list t * kFiredLists / ntiles;
    // their counts at pass_count[(set * kFiredLists + list) * kFiredCountStride].
    unsigned long long *passes;
    uint32_t *pass_count;
    uint64_t passcap;
    // Pull propagation (null crec: off; never together with gather).  The
    // in-edges of target tile t are records [cptr[t], cptr[t + 1]) of crec,
    // grec_words(wfmt) words each: key = source row (bits 0..22) | target's
    // index in the tile (bits 23..30) | channel pair (bit 31), then the
    // weight pair's raw bits, so one load brings both.  bits: per set and
    // tile, the 256 rows emitted by the launch that filled the set (4 words
    // of 64), then those of them whose tile deferred its propagation to the
    // pull (4 words).  step[2 + s] (the deferral stamp of set s) = 1 + the
    // step index of the launch that consumes set s when some tile deferred
    // into it (0: none; a stale stamp never equals a later consumer's).  A
    // consuming tile pulls when its queue overflowed (then it ignores the
    // queue and takes every emitted row through its in-edges) or when rows
    // were deferred (then it adds the deferred rows to its queue).
    const uint32_t *crec;       // [S][grec_words(wfmt)]
    const int64_t *cptr;        // [ntiles + 1]
    unsigned long long *bits;   // [2][ntiles][kBitWords]
    const PopDev *pops;         // [npop]
    // recording (device buffers, row = step - rec_step0)
    // Sums spread over rec_slots slots (a power of two) per row, a tile's
    // into slot (tile % rec_slots); with one slot the strides are npop and
    // npop * 6.
    uint32_t *rec_counts;       // [rec_len][rec_slots][rec_cstride] spikes per population
    long long *rec_stat;        // [rec_len][rec_slots][rec_sstride]: [npop][6] sums of V, I_syn, 4 receptor currents (x 2^24)
    // counters
    // per wave of 64 neurons: (synaptic events delivered = sum of fired
    // out-degrees, spikes emitted); each slot is updated only by the wave
    // that owns those neurons, so no atomics are needed
    unsigned long long *wave_ctr;   // [ceil(n/64)][2]
    int64_t *step;              // [0..1] step index by launch parity: the launch of
                                // parity p reads step[p] and writes step[p^1] = step[p] + 1;
                                // [2..3] deferral stamps by queue set
    // scalars
    uint64_t seed;
    int64_t rec_step0;
    uint32_t n;
    uint32_t npop;
    uint32_t rec_len;
    int32_t t_steps;
    int32_t use_ou;
    uint32_t tile_base;         // engine-wide index of this instance's first tile
    uint32_t stat_mask;         // kStatV | kStatI | kStatReceptor: statistics recorded in rec_stat
    uint32_t pmask;             // parameter record of neuron i: (i & pmask) + cls[i]
    uint32_t ngroups;           // gather groups of the instance
    uint32_t fcap;              // rows per fired list
    uint32_t defer_min;         // pull: a tile with this many emitted rows defers them (0: never)
    uint32_t wfmt;              // weight pair format of w and cw
    uint32_t rec_slots, rec_cstride, rec_sstride;   // layout of rec_counts and rec_stat
    uint32_t ntiles;
};

// Words per tile and set of InstDev::bits: 4 of emitted rows, 4 of deferred
// rows; with direct propagation, in place of the deferred rows, one word with
// the count of emitted rows (2 bytes) and, up to kDirectIds, the rows
// themselves (a byte each).
constexpr uint32_t kBitWords = 8;
constexpr uint32_t kDirectIds = 6;
// Direct propagation: neurons an instance may have (every tile reads the
// emitted rows of every tile, up to kDirectRounds words per thread, all in
// registers: built for 2^20 neurons the kernel spilled 27 of them and every
// size was slower), the emitted rows a tile lists in LDS at a time (with 1024
// a 200k-neuron step of 1143 rows took 25.5 us, in two rounds, with 2048 18.2;
// with 4096 five workgroups fit a CU and eight instances in one engine took
// 14.7 us instead of 12.7), and the synapses a lane has in flight (4: 66k
// neurons x 250 6.63 us, 2: 6.53).
constexpr uint32_t kDirectMaxNeurons = 1u << 18;
// Tiles of an engine up to which it takes direct propagation: it shortens the
// chain of one tile's waits, and past a few rounds of resident workgroups what
// counts is their work.  Uniform networks of 20k-200k neurons, steps direct /
// by queues: 1672 tiles 11.8 / 20.0 us, 4853 36.4 / 42.1, 10330 67.1 / 69.7,
// 20345 128.9 / 119.6.  Served networks of 10k-1M neurons, the small ones
// direct in a launch of their own: 1.24e10 synaptic events per second, all by
// queues 1.35e10.
constexpr uint32_t kDirectTiles = 8192;
// An engine that steps directly goes on to here (10330 tiles, above, are still
// no slower), so instances that come and go around the limit do not make it
// build and return every instance's offsets at each change.
constexpr uint32_t kDirectTilesStay = kDirectTiles + kDirectTiles / 4u;
constexpr uint32_t kDirectRows = 2048, kDirectItems = 2;
constexpr uint32_t kDirectRounds = (kDirectMaxNeurons / kBlock + kBlock - 1) / kBlock;   // tiles per thread

// Weight pair formats kept on the device (include/weights.hpp:14-21 and the
// decode of presynaptic_voltage.cpp:153-176): two fp32 (8 bytes), two fp16
// (4 bytes, converted exactly) or two uint8 codes u (2 bytes, weight
// (float)u / 255.f, correctly rounded).  Double weights are stored as fp32,
// the type the reference's float block converts them to.
enum : uint32_t { kWeightF32 = 0, kWeightF16 = 1, kWeightU8 = 2 };
// Kernel specialisation for launches whose instances hold different formats
// (each weight pair is then decoded by its instance's format at run time).
constexpr uint32_t kWeightAny = 3;
__host__ __device__ inline uint32_t weight_bytes(uint32_t fmt)
{
    return fmt == kWeightF32 ? 8u : fmt == kWeightF16 ? 4u : 2u;
}

// 32-bit words of a gather record: the column and the weight pair (fp32
// pairs 2 words; fp16 pairs and uint8 codes 1 word).
__host__ __device__ inline uint32_t grec_words(uint32_t fmt)
{
    return fmt == kWeightF32 ? 3u : 2u;
}

// Pull propagation limits: source rows are 23-bit fields of the in-edge key.
constexpr uint32_t kPullRowBits = 23;
constexpr uint32_t kPullRowMask = (1u << kPullRowBits) - 1u;
constexpr uint32_t kPullMaxNeurons = 1u << kPullRowBits;
// Default deferral threshold: a tile whose step emitted at least this many
// rows leaves them to the consumers' pull instead of binning them.
constexpr uint32_t kDeferMinDefault = 16;

// One tile = one workgroup of the step kernel: up to 256 consecutive neurons
// of one instance.  The descriptor holds all that a step without spikes
// needs, resolved for the tile, in 128 bytes: a workgroup issues its state,
// parameter and queue loads after one scalar round trip (the instance's
// descriptor behind it is only read by tiles that fire, pull or record).
// Fields are read where a phase needs them (again() in the kernel): held in
// scalar registers from the start, they cost about 100 spilled scalars, each
// a vector instruction to store and one to load back.
constexpr uint32_t kTileUniform = 1u;    // one parameter class (prm is its record)
constexpr uint32_t kTileOnePop = 2u;     // one population (mu, f1, f2s are its OU factors)
constexpr uint32_t kTileOu = 4u;         // the instance runs with the OU background
constexpr uint32_t kTileOuOn = 8u;       // and the tile's one population has it configured
constexpr uint32_t kTilePull = 16u;      // pull propagation
constexpr uint32_t kTileGather = 32u;    // gather propagation
constexpr uint32_t kTileOneSub = 64u;    // one substep per step
constexpr uint32_t kTileStat = 128u;     // population statistics are recorded
struct alignas(128) TileDesc {
    unsigned char *state;    // the tile's state block
    const QSyn *queue;       // its queue of set 0
    uint64_t qslots;         // entries between the sets
    int64_t *step;           // InstDev::step
    uint32_t begin;          // first instance-local neuron
    uint32_t count;          // neurons in the tile (<= 256)
    uint32_t flags;
    uint32_t qcap;           // queue capacity: synapses of all rows targeting this tile, at most
    const ParamRec *prm;     // its record (kTileUniform), else record of class 0 for its neurons
    uint64_t seed;
    float mu, f1, f2s;       // OU of its population (kTileOnePop)
    uint32_t pop0;           // population of the first neuron
    const uint16_t *cls;     // classes of its neurons
    const float4 *dlt;       // gather: its neurons' delta
    const InstDev *inst;
    unsigned long long *bits;   // its words of set 0 (pull)
    const int64_t *rowptr;   // rows of its neurons
    uint32_t ntiles;         // tiles of the instance (words between the sets of bits: ntiles * kBitWords)
    uint32_t inst_idx;       // index of inst
};
static_assert(sizeof(TileDesc) == 128, "two scalar loads of 64 bytes");

// Queue of a target tile as the binning sees it (a set's first slot within
// the instance's queue, capacity).
struct alignas(16) QueueTile {
    uint64_t off;
    uint32_t cap;
    uint32_t pad;
};

// Gather propagation: one workgroup of kGatherBlock threads gathers the
// synapses of every fired row that target one group of consecutive neurons
// (at most 2^kGroupBits; Instance::gather_bits) into LDS, then writes their
// delta.
constexpr uint32_t kGroupBits = kTileBits + 3, kGroupBitsMin = kTileBits;
// Groups below which an instance is cut into smaller ones: one workgroup per
// group, 256 CUs.  Steps with groups of 2^kGroupBits neurons / by the rule:
// 20k neurons x 2000 synapses 67 / 18 us, 60k x 3000 49 / 17, 120k x 3000
// 39 / 22, 200k x 5000 42 / 31 (98 / 196 groups); past it halving the group
// costs more (every group looks every row up) than it fills: 300k x 2000, 147
// groups 30.8 us, 293 35.4.
constexpr uint32_t kGatherGroups = 128;
constexpr int kGatherBlock = 1024;
// Synapses each lane of k_gather loads before it adds them (in flight together).
constexpr uint32_t kGatherItems = 8;
// Longest row the 16-bit group offsets can index.
constexpr int64_t kGatherMaxRow = 65535;
// Fired lists per set (appends spread over this many counters, one wave of
// k_gather reads one count per lane) and the words between their counts.
constexpr uint32_t kFiredLists = 64;
constexpr uint32_t kFiredCountStride = 32;
static_assert(kFiredLists == 64, "k_gather reads one list count per lane");

struct alignas(16) GroupDesc {
    uint32_t inst;
    uint32_t g;         // group index within the instance (first neuron g << bits)
    uint32_t count;     // neurons in the group
    uint32_t bits;      // Instance::gather_bits()
};

// Queues of both parities: the launch of parity p drains set p and fills set
// p ^ 1.
// Queue entries per tile that the step kernel reads ahead together with the
// count; the queue buffer has this many slots of slack after both sets.
constexpr uint32_t kQueuePrefetch = 128;

// Word of queue count i (i = set * ntiles + tile): groups of 2^shift
// consecutive counts share one 128-byte line (32 words).  shift = 5 packs the
// counts densely: the reservations of one wave, which mostly hit neighbouring
// tiles, touch few lines.  shift = 0 gives every count a line of its own:
// when every fired row reaches most tiles, many waves reserve in the same
// counts at once, and counts sharing a line would serialise on it.
constexpr uint32_t kCountLineWords = 32;
// Synapses per lane in a binning pass of the step kernel: 1, 2 or 4 (passes
// of 64, 128 or 256 synapses).  Every value gives the same results.
constexpr uint32_t kPassKDefault = 2;

// Row coverage (tile segments per row / tiles) above which the automatic
// layout spreads the counts.
constexpr double kSpreadCoverage = 0.95;

// Requested layout of an engine's queue counts.
// kLayoutGather: instances that allow it propagate by gather (the others
// keep dense queues); it is chosen explicitly or by the autotuner.
enum : int { kLayoutAuto = 0, kLayoutDense = 1, kLayoutSpread = 2, kLayoutGather = 3 };
constexpr uint32_t kCountShiftDense = 5;
constexpr uint32_t kCountShiftSpread = 0;

__host__ __device__ inline size_t count_slot(size_t i, uint32_t shift)
{
    return ((i >> shift) * kCountLineWords) + (i & ((1u << shift) - 1u));
}

__host__ __device__ inline size_t count_words(size_t n, uint32_t shift)
{
    return ((n + (1u << shift) - 1u) >> shift) * kCountLineWords;
}

// Binning by a launch of its own (k_bin): passes of kBinPass synapses, taken
// by workgroups of kBinBlock threads, each wave kBinDeep passes per round and
// each lane kBinItems synapses of a pass.
constexpr int kBinBlock = 1024;
constexpr uint32_t kBinItems = 4, kBinDeep = 1;
constexpr uint32_t kBinPass = kWave * kBinItems;
static_assert(kBinPass == 256, "a pass entry holds its length less one in 8 bits");
constexpr uint32_t kBinMaxTiles = 16384;   // LDS counts of target tiles (64 KB)
// Workgroups: one per kBinTiles source tiles, at most kBinGroups (two per CU)
// per instance.
constexpr uint32_t kBinTiles = 16, kBinGroups = 512;
// Queue tiles from which an engine bins by k_bin instead of in the tiles that
// fired: its launch and its chain of waits are 8 us of a step, its atomics a
// third as many.  Steps in the tiles / by k_bin, voxel networks at 10, 16 and
// 33 spikes per second: 400k neurons (1563 tiles) 13.5 / 15.3, 15.7 / 16.0 and
// 22.9 / 20.7 us; 600k (2344) 16.3 / 18.0, 19.5 / 19.6 and 28.8 / 25.9; 900k
// (3516) 22.9 / 23.1, 27.5 / 25.9 and 38.1 / 33.8; 2M (7813) at 6, 11 and 21
// 40.6 / 38.4, 49.5 / 43.5 and 69.1 / 59.8.  And only where rows have two
// synapses per tile they reach (voxel networks: three; neighbouring rows then
// reach the same tiles): with uniformly drawn targets there is little to add
// up first, 900k x 300 35.9 / 44.0, 2M x 300 53.8 / 63.2.
constexpr uint32_t kBinLaunchTiles = 3072u;
// And only where the rows that fire in one step share tiles: the (row, tile)
// pairs of all rows that a row 512 neurons on reaches too (about the distance
// of two rows at 20 spikes per second).  Voxels of 10k neurons have 4.5e7 and
// more from 800k neurons and 150 synapses on; of 200 neurons they have none,
// and steps in the tiles / by k_bin are 1M x 60 21.6 / 27.0 us, 1M x 200 24.3 /
// 29.6, 800k x 100 19.1 / 25.4, 2M x 200 41.9 / 44.9; of 1000 neurons 1M x 200
// (1.2e7) 23.6 / 27.5, of 2500 (2.5e7) 23.3 / 26.1, of 1500 2M x 300 (4.2e7)
// 40.9 / 40.9, at 16 spikes per second 47.8 / 45.9.
constexpr double kBinLaunchShared = 3.5e7;
constexpr uint32_t kSharingDistance = 512, kSharingRows = 64;
struct alignas(16) BinDesc {
    const InstDev *inst;
    uint32_t part, parts;   // takes part `part` of `parts` of the step's passes
};

struct StepCtl;
struct alignas(16) QueueSet {
    const QueueTile *tile;   // [ntiles]
    uint32_t *count;    // [2][ntiles], tile t of set p at word count_slot(p * ntiles + t, cshift)
    StepCtl *ctl;
    uint32_t ntiles;
    uint32_t cshift;    // kCountShiftDense or kCountShiftSpread
};

// Sample request (reference stat_samples_kernel, stat_result.cpp:393-433).
struct alignas(16) SampleDev {
    uint32_t inst;
    uint32_t neuron;
    uint32_t slot;      // column in the instance's sample record
    uint32_t pad;
};

// Per-instance sample records, row = step - rec_step0.
struct alignas(16) SampleRecDev {
    uint8_t *spike;
    float *v;
    float *isyn;
    float *iou;
    uint32_t nsample;
    uint32_t pad[3];
};

// Size of the static device array that holds the per-step records of one
// dtb_run_noalloc call (one copy per GPU, kept until the process ends).
constexpr size_t kScratchBytes = (size_t)64 << 20;

// Shared per-engine diagnostics in device memory.
// Diagnostic counters of the step launches.  Each is spread over kCtlSlots
// cache lines, a workgroup adding into slot blockIdx.x % kCtlSlots: atomics
// from every tile of a launch on one address would be serialised by the
// memory and hold the launch's end (a volley step defers or pulls in all
// 7,813 tiles of the 2M-neuron block).
constexpr uint32_t kCtlSlots = 64;
struct alignas(128) CtlSlot {
    unsigned long long spilled;   // synapses past a queue's capacity (spilled, or taken by the pull)
    unsigned long long deferred;  // tiles that left their emitted rows to the pull
    unsigned long long pulled;    // tiles that took input through their in-edges (step launches)
    unsigned long long pad[13];
};
struct StepCtl {
    CtlSlot slot[kCtlSlots];
};
// The counters summed over their slots.
struct CtlTotals {
    unsigned long long spilled, deferred, pulled;
};

}  // namespace dtb
