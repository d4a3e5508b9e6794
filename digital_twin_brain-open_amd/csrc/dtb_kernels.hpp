// dtb_kernels.hpp -- host-callable launchers of the gfx950 step kernels.
#pragma once

#include "dtb_types.hpp"

namespace dtb {

// How a k_step launch's tiles take their input and pass on their rows: queues
// (or gather), binned by the tiles themselves or by a launch_bin_kernel after
// it; or direct propagation.
enum class StepMode { tile_bin, bin_launch, direct };

// One step of every tile, launch parity `par` (input of set par + fold + OU +
// LIF; the emitted rows into set par ^ 1).  pass_k: synapses per lane in a
// binning pass (tile_bin: 1, 2 or 4).  wfmt: the weight format of every
// instance in the tables, or kWeightAny (each launch's kernels are
// specialised for it).  stat: some instance records population statistics.
// start / stop (may be null): recorded at the kernel's own dispatch
// boundaries (kernel time without launch gaps).
hipError_t launch_step_kernel(const TileDesc *tiles, uint32_t ntiles, StepMode mode, uint32_t pass_k,
                              const QueueSet *qs, uint32_t par, uint32_t wfmt, bool stat, hipEvent_t start,
                              hipEvent_t stop, hipStream_t stream);

// Bins the rows emitted by the k_step launch of parity `par` into queue set
// par ^ 1 (groups of source tiles; max_tiles: tiles of the largest instance).
hipError_t launch_bin_kernel(const BinDesc *groups, uint32_t ngroups, uint32_t max_tiles, const QueueSet *qs,
                             uint32_t par, uint32_t wfmt, hipEvent_t start, hipEvent_t stop, hipStream_t stream);

// Gather propagation: delta of fired list `par` into InstDev::dlt for every
// group (runs before the k_step launch of parity `par`, and before
// materialize / settle of set `par`); empties fired list par ^ 1.
hipError_t launch_gather(const GroupDesc *groups, uint32_t ngroups, const InstDev *insts, uint32_t par, uint32_t wfmt,
                         hipEvent_t start, hipEvent_t stop, hipStream_t stream);

// Gather records ([nsyn][grec_words(wfmt)]: column, weight pair bits).
hipError_t launch_build_grec(const uint32_t *col, const void *w, uint32_t wfmt, uint64_t nsyn, uint32_t *rec,
                             hipStream_t stream);

// Offsets per target group of 2^shift neurons ([n][ngroups + 1], rows ordered
// by target group; tiles: shift kTileBits).
hipError_t launch_build_segidx(const int64_t *rowptr, const uint32_t *col, uint32_t n, uint32_t ngroups,
                               uint32_t shift, uint16_t *segidx, hipStream_t stream);

// In-edges of the pull propagation from the presynaptic-major CSR: cptr
// [ntiles + 1] holds each target tile's first in-edge; cursor [ntiles] is
// zeroed and counts the records placed per tile.
hipError_t launch_build_pull(const int64_t *rowptr, const uint32_t *col, const void *w, uint32_t wfmt, uint32_t n,
                             const int64_t *cptr, uint32_t *cursor, uint32_t *rec, hipStream_t stream);

// Pending delta of queue set `set` into InstDev::dlt (queues left intact).
hipError_t launch_materialize(const TileDesc *tiles, uint32_t ntiles, const InstDev *insts, const QueueSet &qs,
                              uint32_t set, hipStream_t stream);

// Pending delta of queue set `set` folded into J now, that set emptied
// (before parameter changes).
hipError_t launch_settle(const TileDesc *tiles, uint32_t ntiles, const InstDev *insts, const QueueSet &qs,
                         uint32_t set, hipStream_t stream);

// I_syn-based statistics of the last step run into the recording (after
// launch_materialize of the pending set); `par` = parity of the next launch.
hipError_t launch_stat_tail(const TileDesc *tiles, uint32_t ntiles, const InstDev *insts, uint32_t par,
                            hipStream_t stream);

// Copies `words` 4-byte words of src (null: zeros) to dst; either may be
// pinned host memory.
struct CopyWords {
    void *dst;
    const void *src;
    uint64_t words;
};
// All of segs[n] (kCopySegs per launch).
constexpr int kCopySegs = 10;
hipError_t launch_copy_words(const CopyWords *segs, int n, hipStream_t stream);

// Rows [row0, row0 + rows) of a record, each row's slots added up, as plain
// arrays: sums [rows][swidth] and counts [rows][cwidth] (width 0: none).
// The outputs may be pinned host memory.
struct RecordRows {
    const long long *stat;
    const uint32_t *counts;
    uint32_t slots, sstride, cstride, swidth, cwidth;
    long long *out_stat;
    uint32_t *out_counts;
};
hipError_t launch_fetch_rows(const RecordRows &r, uint64_t row0, uint64_t rows, hipStream_t stream);

// Samples of the step run by the k_step launch of parity `par`.
hipError_t launch_sample(const InstDev *insts, const SampleDev *samples, uint32_t nsamples,
                         const SampleRecDev *recs, uint32_t par, hipStream_t stream);

// State of one instance (its blocks and what reading them needs), and plain
// arrays of it.
struct StateView {
    unsigned char *state;
    const ParamRec *prm;
    const uint16_t *cls;
    float4 *dlt;
    uint32_t pmask, n;
};
struct StateArrays {
    float *V;
    int32_t *t;
    float *iou;
    float4 *J;
    float *isyn;
    uint8_t *f, *emitted;
};
// V of a fresh state (the blocks zeroed before); OU current of a range of
// neurons; state of neurons [first, first + count) into / from plain device
// arrays (null: not read / kept).
hipError_t launch_init_state(const StateView &v, hipStream_t stream);
hipError_t launch_fill_iou(const StateView &v, uint32_t begin, uint32_t end, float value, hipStream_t stream);
hipError_t launch_read_state(const StateView &v, uint32_t first, uint32_t count, const StateArrays &out,
                             hipStream_t stream);
hipError_t launch_write_state(const StateView &v, uint32_t first, uint32_t count, const StateArrays &in,
                              hipStream_t stream);

hipError_t launch_normals(uint64_t seed, uint32_t neuron0, uint64_t substep, uint32_t count, float *out,
                          hipStream_t stream);

}  // namespace dtb
