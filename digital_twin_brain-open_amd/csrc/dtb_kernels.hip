// dtb_kernels.hip -- gfx950 kernels of the DTB single-block step.
//
// Reference stage order for one step with t_steps substeps
// (tools/dist_simulator.cpp:2072-2315):
//   substeps: OU current (extern_stimuli.cpp:39-112) -> LIF membrane update
//             (membrane_voltage.cpp:114-195) -> [t_steps > 1: OR fired flags,
//             J decay, I_syn]
//   propagation of the fired rows into the delta buffers
//             (presynaptic_voltage.cpp:122-225)
//   J = J * decay + delta (presynaptic_voltage.cpp:46-120), I_syn
//             (synaptic_current.cpp:7-105)
//
// One launch per step here (k_step; see the end of this comment for the
// second launches of the gather schedule and of large engines).  Every workgroup of 256 threads owns a
// tile of 256 consecutive neurons of one instance, and per tile:
//   1. reads the tile's queue (the synapses delivered to it: target index,
//      channel pair, weight pair; contiguous, so the reads coalesce) and adds
//      the weights into exact Q23.40 accumulators in LDS (64-bit integer LDS
//      atomics, so the sum does not depend on the order);
//   2. folds the delta into J (J = J * decay + delta), computes I_syn, runs
//      OU + LIF for every substep;
//   3. lists the tile's fired rows in LDS and deals their passes of 128
//      synapses round-robin to its four waves; a wave reads a pass (synapses
//      ordered by target), reserves one contiguous segment per target tile
//      with an atomic add on that tile's count and writes each synapse's
//      entry into the target tile's queue for the next launch (12 bytes per
//      synapse).
// The queues are double-buffered: the launch of parity p drains set p and
// fills set p ^ 1, so step k consumes exactly the synapses queued from the
// spikes of step k - 1.  No global atomics touch the delta.
//   With the gather schedule (instances with group offsets) a k_gather
//   launch precedes each k_step: per group of target neurons it gathers
//   the last step's fired rows into the same exact LDS sums and writes the
//   delta, which k_step folds instead of draining a queue; k_step lists its
//   fired rows for the next k_gather instead of binning them.
//   Small engines propagate directly: no queues, a tile reads the rows that
//   every tile emitted in the step before (direct_tile).  Large ones bin in a
//   launch of their own (k_bin) in place of 3.
//   k_materialize writes the pending delta of every neuron (without consuming
//   the queues) for sampling and state read-back; k_sample gathers samples.
#include <hip/hip_ext.h>

#include <type_traits>

#include "dtb_kernels.hpp"
#include "dtb_rng.hpp"

namespace dtb {

// Pointers read from the instance descriptors are generic; accessing them
// through the global address space lets the compiler emit global (not flat)
// memory instructions, which do not share the LDS wait counter.
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T *gp(T *p)
{
    return (__attribute__((address_space(1))) T *)p;
}

typedef float gfloat4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float4 ld4(const float4 *p, size_t i)
{
    const gfloat4 v = *(const __attribute__((address_space(1))) gfloat4 *)(p + i);
    return make_float4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ void st4(float4 *p, size_t i, const float4 v)
{
    gfloat4 g;
    g.x = v.x;
    g.y = v.y;
    g.z = v.z;
    g.w = v.w;
    *(__attribute__((address_space(1))) gfloat4 *)(p + i) = g;
}

// Memory that no launch reading it changes (descriptors, parameters, the step
// index of the launch's parity), read through the scalar unit where the
// address is uniform.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T *cp(const T *p)
{
    return (const __attribute__((address_space(4))) T *)p;
}
typedef const __attribute__((address_space(4))) InstDev *InstPtr;
typedef const __attribute__((address_space(4))) TileDesc *TilePtr;
typedef const __attribute__((address_space(4))) QueueSet *QueuePtr;

__device__ __forceinline__ float4 ld4c(const float4 *p)
{
    const gfloat4 v = *(const __attribute__((address_space(4))) gfloat4 *)p;
    return make_float4(v.x, v.y, v.z, v.w);
}

// The same address, opaque to the compiler: what is read through it is read
// again (scalar cache hits) instead of kept in scalar registers from an
// earlier phase of the kernel.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T *again(
    const __attribute__((address_space(4))) T *p)
{
    asm volatile("" : "+s"(p));
    return p;
}

// Device-scope add on global memory (no flat access).
template <typename T>
__device__ __forceinline__ T gadd(T *p, T v)
{
    return __hip_atomic_fetch_add(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// (float)((double)q * 2^-40): the two halves meet in one rounded double, as
// the conversion of q does; the scaling is exact on either side of the float
// rounding (|q| >= 1 keeps the result normal).
__device__ __forceinline__ float q40_to_f32(long long q)
{
    const double d = fma((double)(int32_t)(q >> 32), 0x1p32, (double)(uint32_t)q);
    return (float)d * 0x1p-40f;
}

__device__ __forceinline__ unsigned long long f32_to_q40(float w)
{
    return (unsigned long long)(long long)rintf(w * 0x1p40f);
}


// uint8 weight codes: u -> (float)u / 255.f, the correctly rounded quotient
// (presynaptic_voltage.cpp:171-176), folded at compile time (IEEE division).
struct U8Weights {
    float v[256];
};
constexpr U8Weights make_u8_weights()
{
    U8Weights t{};
    for (int u = 0; u < 256; ++u)
        t.v[u] = (float)u / 255.0f;
    return t;
}
__constant__ U8Weights c_u8_weight = make_u8_weights();

// Weight pairs (presynaptic_voltage.cpp:153-176): raw bits of pair j of an
// array in format fmt (at most 64 bits) and the pair they encode.
__device__ __forceinline__ unsigned long long w_raw(const void *w, size_t j, uint32_t fmt)
{
    if (fmt == kWeightF32)
        return gp(static_cast<const unsigned long long *>(w))[j];
    if (fmt == kWeightF16)
        return gp(static_cast<const uint32_t *>(w))[j];
    return gp(static_cast<const uint16_t *>(w))[j];
}

__device__ __forceinline__ float2 w_decode(unsigned long long b, uint32_t fmt)
{
    if (fmt == kWeightF32)
        return make_float2(__uint_as_float((uint32_t)b), __uint_as_float((uint32_t)(b >> 32)));
    if (fmt == kWeightF16)
        return make_float2((float)__builtin_bit_cast(_Float16, (uint16_t)b),
                           (float)__builtin_bit_cast(_Float16, (uint16_t)(b >> 16)));
    // uchar2 codes over 255
    return make_float2(c_u8_weight.v[b & 0xffu], c_u8_weight.v[(b >> 8) & 0xffu]);
}

// K weight pairs at indices jj[] of array w (one branch on the format for
// all K loads, so they are in flight together).
template <uint32_t K, typename Idx>
__device__ __forceinline__ void w_load(unsigned long long (&out)[K], const void *w, const Idx (&jj)[K],
                                       uint32_t fmt)
{
    if (fmt == kWeightF32) {
        const auto p = gp(static_cast<const unsigned long long *>(w));
#pragma unroll
        for (uint32_t k = 0; k < K; ++k)
            out[k] = p[jj[k]];
    } else if (fmt == kWeightF16) {
        const auto p = gp(static_cast<const uint32_t *>(w));
#pragma unroll
        for (uint32_t k = 0; k < K; ++k)
            out[k] = p[jj[k]];
    } else {
        const auto p = gp(static_cast<const uint16_t *>(w));
#pragma unroll
        for (uint32_t k = 0; k < K; ++k)
            out[k] = p[jj[k]];
    }
}

__device__ __forceinline__ const void *w_row(const void *w, int64_t first, uint32_t fmt)
{
    return static_cast<const char *>(w) + (size_t)first * weight_bytes(fmt);
}

// Parameter record of neuron li.
__device__ __forceinline__ const ParamRec *param_of(const InstDev &I, uint32_t li)
{
    return I.prm + ((li & I.pmask) + (uint32_t)gp(I.cls)[li]);
}

// Neuron i of a state block: field at byte offset kOff, one T per neuron.
template <uint32_t kOff, typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T *st_at(unsigned char *block, uint32_t i)
{
    return (__attribute__((address_space(1))) T *)(gp(block) + (size_t)(i * (uint32_t)sizeof(T)) + kOff);
}

__device__ __forceinline__ float4 ld_J(unsigned char *block, uint32_t i)
{
    const gfloat4 v = *st_at<kStJ, gfloat4>(block, i);
    return make_float4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ void st_J(unsigned char *block, uint32_t i, const float4 v)
{
    gfloat4 g;
    g.x = v.x;
    g.y = v.y;
    g.z = v.z;
    g.w = v.w;
    *st_at<kStJ, gfloat4>(block, i) = g;
}

// State block of the tile that holds neuron li.
__device__ __forceinline__ unsigned char *block_of(const InstDev &I, uint32_t li)
{
    return I.state + (size_t)(li >> kTileBits) * kStateBytes;
}

// synaptic_current.cpp:39-43 in source order, no contraction.
__device__ __forceinline__ float syn_current(const float4 g, const float4 vu, const float4 J, const float V)
{
    const float a = g.x * (vu.x - V) * J.x;
    const float b = g.y * (vu.y - V) * J.y;
    const float c = g.z * (vu.z - V) * J.z;
    const float d = g.w * (vu.w - V) * J.w;
    return a + b + c + d;
}

// presynaptic_voltage.cpp:62-73: J = J * decay + delta (fused multiply-add).
__device__ __forceinline__ float4 fold_delta(const float4 J, const float4 dc, const float4 dl)
{
    float4 r;
    r.x = fmaf(J.x, dc.x, dl.x);
    r.y = fmaf(J.y, dc.y, dl.y);
    r.z = fmaf(J.z, dc.z, dl.z);
    r.w = fmaf(J.w, dc.w, dl.w);
    return r;
}

// v plus the value that DPP control kCtrl brings from another lane (0 where it
// brings none), as two 32-bit moves and one 64-bit add.
template <int kCtrl, int kRowMask>
__device__ __forceinline__ unsigned long long dpp_add_u64(unsigned long long v)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, kCtrl, kRowMask, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), kCtrl, kRowMask, 0xf, false);
    return v + (((unsigned long long)hi << 32) | lo);
}

// Sum over the 64 lanes (all of them active): an inclusive scan with DPP, no
// LDS round trips; lane 63 holds the total.
__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v)
{
    v = dpp_add_u64<0x111, 0xf>(v);   // row_shr:1
    v = dpp_add_u64<0x112, 0xf>(v);   // row_shr:2
    v = dpp_add_u64<0x114, 0xf>(v);   // row_shr:4
    v = dpp_add_u64<0x118, 0xf>(v);   // row_shr:8
    v = dpp_add_u64<0x142, 0xa>(v);   // row_bcast:15
    v = dpp_add_u64<0x143, 0xc>(v);   // row_bcast:31
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, kWave - 1);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), kWave - 1);
    return ((unsigned long long)hi << 32) | lo;
}

// Inclusive sum over the 64 lanes with DPP: shifts by 1, 2, 4, 8 within each
// row of 16 lanes (lanes shifted in from outside the row read 0), then the
// last lane of row 0 / 2 into rows 1 / 3 and the last lane of row 1 into rows
// 2 and 3.
__device__ __forceinline__ uint32_t wave_add_scan(uint32_t v)
{
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);   // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);   // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);   // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);   // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);   // row_bcast:15
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);   // row_bcast:31
    return v;
}

// The LDS sums are channel-major: channel c of row i at acc[c * rows + i].
// A wave's 64-bit atomics go to random rows; with the rows 8 bytes apart
// (not 32, as row-major would put them) they spread over twice as many LDS
// banks.
__device__ __forceinline__ uint32_t acc_at(uint32_t row, uint32_t chan, uint32_t rows)
{
    return chan * rows + row;
}

__device__ __forceinline__ QSyn ld_entry(const QSyn *q, size_t k)
{
    const auto p = gp(reinterpret_cast<const uint32_t *>(q)) + k * 3u;
    QSyn e;
    e.key = p[0];
    e.w0 = __uint_as_float(p[1]);
    e.w1 = __uint_as_float(p[2]);
    return e;
}

__device__ __forceinline__ void st_entry(QSyn *q, size_t k, uint32_t key, float w0, float w1)
{
    const auto p = gp(reinterpret_cast<uint32_t *>(q)) + k * 3u;
    p[0] = key;
    p[1] = __float_as_uint(w0);
    p[2] = __float_as_uint(w1);
}

// Adds the queued synapses of one tile into acc[4][256] (Q23.40, LDS): every
// thread takes every 256th entry of the tile's queue (contiguous, so the
// reads coalesce) and adds its weight pair with 64-bit integer LDS atomics,
// so the sum does not depend on the order.  Threads tid < npre already hold
// entry tid in `pre`.
__device__ __forceinline__ void accumulate_tile(unsigned long long *acc, const QSyn *__restrict__ q, uint32_t cnt,
                                                const QSyn &pre, uint32_t npre, uint32_t tid)
{
    for (uint32_t k = tid; k < cnt; k += kBlock) {
        const QSyn e = (k < npre) ? pre : ld_entry(q, k);
        const uint32_t row = e.key & 0xffu, c0 = (e.key & kQSynKind) ? 2u : 0u;
        atomicAdd(&acc[acc_at(row, c0, kBlock)], f32_to_q40(e.w0));
        atomicAdd(&acc[acc_at(row, c0 + 1u, kBlock)], f32_to_q40(e.w1));
    }
}

// Zeroes row tid of a tile's sums (every row by the whole workgroup).
__device__ __forceinline__ void clear_row(unsigned long long *acc, uint32_t tid)
{
#pragma unroll
    for (uint32_t c = 0; c < 4; ++c)
        acc[acc_at(tid, c, kBlock)] = 0ull;
}

// Adds neuron li's spill accumulator of queue set `set` into the neuron's own
// LDS sums (row tid of acc); `consume` clears it for the set's next use.
// Called by the neuron's thread after the queue accumulation.
__device__ __forceinline__ void take_spill(unsigned long long *acc, unsigned long long *spill, uint32_t n,
                                           uint32_t set, uint32_t li, uint32_t tid, bool consume)
{
    const auto s = gp(spill) + ((size_t)set * n + li) * 4u;
#pragma unroll
    for (uint32_t c = 0; c < 4; ++c) {
        acc[acc_at(tid, c, kBlock)] += s[c];
        if (consume)
            s[c] = 0ull;
    }
}

// Pull propagation: adds into acc (the tile's Q23.40 LDS sums) the weight
// pairs of tile t's in-edges whose source row was emitted by the launch that
// filled set `set`: every emitted row (`all`: the queue overflowed and is
// ignored) or only the rows of tiles that deferred them.  An in-edge
// is one record (key, then the weight pair's bits: kW words), read
// coalesced; the source's bit comes from the per-tile bitmaps (n / 4 bytes,
// cache resident; read as 32-bit words), so a batch is two dependent loads
// (records, bit words); each thread keeps kPullItems in-edges in flight.
// Called by the whole workgroup.
constexpr uint32_t kPullItems = 4;
template <uint32_t kFmt>
__device__ __forceinline__ void pull_loop(unsigned long long *acc, const uint32_t *rec,
                                          const unsigned long long *bits, uint32_t len, uint32_t tid)
{
    constexpr uint32_t U = kPullItems;
    constexpr uint32_t kW = kFmt == kWeightF32 ? 3u : 2u;   // grec_words(kFmt)
    // uniform bases and 32-bit byte offsets (a tile's in-edges span less
    // than 4 GB; the bitmaps less than 3 MB): one VGPR per address
    using gbyte = const __attribute__((address_space(1))) unsigned char;
    gbyte *rb = reinterpret_cast<gbyte *>(gp(rec));
    gbyte *bb = reinterpret_cast<gbyte *>(gp(reinterpret_cast<const uint32_t *>(bits)));
    for (uint32_t k0 = tid; k0 < len; k0 += kBlock * U) {
        uint32_t kv[U];
        unsigned long long wr[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t j = k0 + u * kBlock;
            const auto r = reinterpret_cast<const __attribute__((address_space(1))) uint32_t *>(
                rb + (j < len ? j : len - 1u) * (kW * 4u));
            kv[u] = r[0];
            wr[u] = kW == 3u ? ((unsigned long long)r[1] | ((unsigned long long)r[2] << 32)) : r[1];
        }
        uint32_t bw[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            bw[u] = *reinterpret_cast<const __attribute__((address_space(1))) uint32_t *>(
                bb + ((kv[u] & kPullRowMask) >> kTileBits) * (kBitWords * 8u) + ((kv[u] >> 3) & 0x1cu));
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            if (k0 + u * kBlock < len && ((bw[u] >> (kv[u] & 31u)) & 1u) != 0u) {
                const float2 wp = w_decode(wr[u], kFmt);
                const uint32_t row = (kv[u] >> kPullRowBits) & 0xffu, c0 = (kv[u] & kKindBit) ? 2u : 0u;
                atomicAdd(&acc[acc_at(row, c0, kBlock)], f32_to_q40(wp.x));
                atomicAdd(&acc[acc_at(row, c0 + 1u, kBlock)], f32_to_q40(wp.y));
            }
        }
    }
}

// The pull of tile t; kFmt: the launch's weight format (kWeightAny: the
// instance's, at run time).
template <uint32_t kFmt, typename Inst>
__device__ __forceinline__ void pull_tile(unsigned long long *acc, const Inst &I, uint32_t set, uint32_t t, bool all,
                                          uint32_t tid)
{
    const unsigned long long *bits = I.bits + (size_t)set * I.ntiles * kBitWords + (all ? 0u : 4u);
    const int64_t b = gp(I.cptr)[t];
    const uint32_t len = (uint32_t)(gp(I.cptr)[t + 1] - b);   // a tile has fewer than 2^32 in-edges
    const uint32_t fmt = kFmt != kWeightAny ? kFmt : I.wfmt;
    const uint32_t *rec = I.crec + (size_t)b * grec_words(fmt);
    if (fmt == kWeightF32)
        pull_loop<kWeightF32>(acc, rec, bits, len, tid);
    else if (fmt == kWeightF16)
        pull_loop<kWeightF16>(acc, rec, bits, len, tid);
    else
        pull_loop<kWeightU8>(acc, rec, bits, len, tid);
}

// LDS of a tile's direct propagation.
struct DirectList {
    uint32_t row[kDirectRows];      // emitted rows
    uint32_t first[2 * kBlock];     // of two rows per lane: first synapse of the row's segment,
    uint32_t off[2 * kBlock];       // and items of its wave before it
    uint16_t item[kDirectItems * kBlock];   // per synapse of a wave's window: its row's slot
    uint32_t n;
    uint32_t wave[kBlock / kWave];
};

// Orders a wave's LDS accesses before and after it (the wave's lanes hand
// each other values through LDS).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Adds the listed rows' segments for tile t into acc.  The rows are dealt to
// the four waves in turn, and each wave works by itself, without a barrier
// (with the segments shared by the whole workgroup, and two barriers per
// round, 130k neurons x 150 took 8.30 us a step instead of 8.07, 200k x 500
// 8.19 instead of 7.85): a lane looks up two rows (offsets and start), the
// wave's segments (mostly none to a few synapses) are laid end to end, and
// consecutive lanes take consecutive synapses, kDirectItems each in flight.
template <uint32_t kFmt, typename Inst>
__device__ __forceinline__ void direct_rows(unsigned long long *acc, const Inst &I, DirectList &ls, uint32_t n,
                                            uint32_t t, uint32_t tid)
{
    const uint32_t wfmt = kFmt != kWeightAny ? kFmt : I.wfmt;
    const uint32_t stride = I.ntiles + 1u;
    const uint32_t lane = tid & (kWave - 1u), w = tid / kWave;
    constexpr uint32_t kWaves = kBlock / kWave, kWin = kDirectItems * kWave;
    uint32_t *first = ls.first + 2u * kWave * w, *off = ls.off + 2u * kWave * w;
    uint16_t *item = ls.item + kWin * w;
    const auto col = gp(I.col);
    const void *wt = I.w;
    for (uint32_t k0 = w; k0 < n; k0 += 2u * kBlock) {
        uint32_t len[2];
#pragma unroll
        for (uint32_t i = 0; i < 2u; ++i) {
            len[i] = 0u;
            const uint32_t k = k0 + i * kBlock + lane * kWaves;
            if (k < n) {
                const uint32_t r = ls.row[k];
                const auto sg = gp(I.tidx) + ((size_t)r * stride + t);
                const uint32_t a = sg[0], e = sg[1];
                first[i * kWave + lane] = (uint32_t)gp(I.rowptr)[r] + a;   // (fewer than 2^32 synapses)
                len[i] = e - a;
            }
        }
        const uint32_t incl = wave_add_scan(len[0] + len[1]);
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        const uint32_t before = incl - len[0] - len[1];
        off[lane] = before;
        off[kWave + lane] = before + len[0];
        for (uint32_t w0 = 0; w0 < total; w0 += kWin) {
            // the items of this lane's segments that fall into the window
#pragma unroll
            for (uint32_t i = 0; i < 2u; ++i) {
                const uint32_t b = before + (i ? len[0] : 0u);
                for (uint32_t k = max(b, w0); k < min(b + len[i], w0 + kWin); ++k)
                    item[k - w0] = (uint16_t)(i * kWave + lane);
            }
            wave_sync();
            const uint32_t m = min(total - w0, kWin);
            uint32_t cv[kDirectItems];
            unsigned long long wv[kDirectItems];
#pragma unroll
            for (uint32_t u = 0; u < kDirectItems; ++u) {
                const uint32_t k = u * kWave + lane;
                if (k < m) {
                    const uint32_t slot = item[k];
                    const uint32_t at = first[slot] + (w0 + k - off[slot]);
                    cv[u] = col[at];
                    wv[u] = w_raw(wt, (size_t)at, wfmt);
                }
            }
#pragma unroll
            for (uint32_t u = 0; u < kDirectItems; ++u)
                if (u * kWave + lane < m) {
                    const float2 wp = w_decode(wv[u], wfmt);
                    const uint32_t row = cv[u] & 0xffu, c0 = (cv[u] & kKindBit) ? 2u : 0u;
                    atomicAdd(&acc[acc_at(row, c0, kBlock)], f32_to_q40(wp.x));
                    atomicAdd(&acc[acc_at(row, c0 + 1u, kBlock)], f32_to_q40(wp.y));
                }
            wave_sync();
        }
    }
}

// The emitted rows of a thread's source tiles, all rounds in flight together:
// per tile, after its 4 words of bits, a word of the count and the first ids.
struct DirectIds {
    unsigned long long b[kDirectRounds];

    // bits: the instance's words of the set
    __device__ __forceinline__ DirectIds(const unsigned long long *bits, uint32_t T, uint32_t tid)
    {
#pragma unroll
        for (uint32_t i = 0; i < kDirectRounds; ++i)
            if (i * kBlock < T) {
                const uint32_t src = i * kBlock + tid;
                b[i] = src < T ? gp(bits)[(size_t)src * kBitWords + 4u] : 0ull;
            }
    }
};

// Direct propagation: adds into acc (zeroed, as ls.n is; both visible) the
// synapses onto tile t of every row emitted into set `set`.  Each thread
// reads the emitted rows of up to kDirectRounds source tiles (the count and
// the first ids; their bits where there are more) and lists them in LDS.  More rows than the list holds are taken in rounds, by rank; where
// reading the tile's in-edges is cheaper than one segment lookup per row
// (volleys), the tile pulls.  Called by the whole workgroup; ends without a
// barrier.  Returns whether the tile pulled.
template <uint32_t kFmt, typename Inst>
__device__ __forceinline__ bool direct_tile(unsigned long long *acc, DirectList &ls, const Inst &I,
                                            const DirectIds &ids, uint32_t set, uint32_t t, uint32_t tid)
{
    const uint32_t T = I.ntiles;
    typedef unsigned long long u64x4 __attribute__((ext_vector_type(4)));
    const auto bits = (const __attribute__((address_space(1))) u64x4 *)gp(I.bits + (size_t)set * T * kBitWords);
    const unsigned long long(&b4)[kDirectRounds] = ids.b;
    // places in the list: one LDS add per wave
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t i = 0; i < kDirectRounds; ++i)
        if (i * kBlock < T)
            mine += (uint32_t)b4[i] & 0xffffu;
    const uint32_t incl = wave_add_scan(mine);
    uint32_t at = 0;
    if ((tid & (kWave - 1u)) == kWave - 1u)
        at = atomicAdd(&ls.n, incl);
    at = (uint32_t)__builtin_amdgcn_readlane((int)at, kWave - 1) + incl - mine;
#pragma unroll
    for (uint32_t i = 0; i < kDirectRounds; ++i) {
        if (i * kBlock >= T)
            continue;
        unsigned long long b = b4[i];
        const uint32_t c = (uint32_t)b & 0xffffu, src = i * kBlock + tid, r0 = src * kBlock;
        const uint32_t last = min(at + c, kDirectRows);   // rows past the list are taken in rounds, below
        if (c <= kDirectIds) {
            // the usual case: ids in bytes 2..7
            for (uint32_t k = at; k < last; ++k) {
                b >>= 8;
                ls.row[k] = r0 + ((uint32_t)(b >> 8) & 0xffu);
            }
        } else {
            const u64x4 e = bits[2u * src];
            uint32_t k = at;
#pragma unroll
            for (uint32_t q = 0; q < 4u; ++q)
                for (unsigned long long m = e[q]; m != 0ull && k < last; m &= m - 1ull, ++k)
                    ls.row[k] = r0 + q * kWave + (uint32_t)__ffsll((long long)m) - 1u;
        }
        at += c;
    }
    __syncthreads();
    const uint32_t n = ls.n;
    if (n <= kDirectRows) {
        direct_rows<kFmt>(acc, I, ls, n, t, tid);
        return false;
    }
    // Bytes either way: a lookup touches a line of offsets, and a short
    // segment a line of columns and one of weights per few synapses; the
    // in-edges are one stream (a volley step of 200k x 150 pulls in 110-146
    // us, with every row in rounds 7 ms).
    const uint64_t in_edges = (uint64_t)(gp(I.cptr)[t + 1] - gp(I.cptr)[t]);
    if ((uint64_t)n * (64u * (uint64_t)I.n + 24u * in_edges) > 12u * in_edges * (uint64_t)I.n) {
        pull_tile<kFmt>(acc, I, set, t, true, tid);
        return true;
    }
    // ranks: rows of the threads before, then a thread's own in tile order
    const uint32_t lane = tid & (kWave - 1u), w = tid / kWave;
    if (lane == kWave - 1)
        ls.wave[w] = incl;
    __syncthreads();
    uint32_t rank0 = incl - mine;
    for (uint32_t k = 0; k < w; ++k)
        rank0 += ls.wave[k];
    for (uint32_t first = 0; first < n; first += kDirectRows) {
        if (rank0 < first + kDirectRows && rank0 + mine > first) {
            uint32_t at = rank0;
            for (uint32_t src = tid; src < T; src += kBlock) {
                const u64x4 b = bits[2u * src];
#pragma unroll
                for (uint32_t q = 0; q < 4u; ++q)
                    for (unsigned long long m = b[q]; m != 0ull; m &= m - 1ull, ++at)
                        if (at >= first && at < first + kDirectRows)
                            ls.row[at - first] = src * kBlock + q * kWave + (uint32_t)__ffsll((long long)m) - 1u;
            }
        }
        __syncthreads();
        direct_rows<kFmt>(acc, I, ls, min(n - first, kDirectRows), t, tid);
        __syncthreads();
    }
    return false;
}

// A statistic's value as the exact integer rint(x * 2^24).
__device__ __forceinline__ long long stat_q(float x)
{
    return (long long)rintf(x * 0x1p24f);
}

// Receptor currents g_u (V_u - V) J_u (synaptic_current.cpp:39-42 terms).
__device__ __forceinline__ float4 receptor_currents(const float4 g, const float4 vu, const float4 J, const float V)
{
    float4 r;
    r.x = g.x * (vu.x - V) * J.x;
    r.y = g.y * (vu.y - V) * J.y;
    r.z = g.z * (vu.z - V) * J.z;
    r.w = g.w * (vu.w - V) * J.w;
    return r;
}

// Recorded sums of step row `row` (counts and statistics): the tile's slot.
// Atomics on one 128-byte line are served one after the other (about 8 ns
// each: a block of two populations and 469 tiles took 97 us per step with
// one line per step, 9 us without statistics), so a record has rec_slots
// slots of whole lines, a tile adding into slot (tile % slots); k_fetch_rows
// adds the slots up when the record is fetched.
template <typename Inst>
__device__ __forceinline__ uint32_t *rec_count_row(const Inst &I, int64_t row, uint32_t begin)
{
    const size_t slot = (begin >> kTileBits) & (I.rec_slots - 1u);
    return I.rec_counts + ((size_t)row * I.rec_slots + slot) * I.rec_cstride;
}

template <typename Inst>
__device__ __forceinline__ long long *rec_stat_row(const Inst &I, int64_t row, uint32_t begin)
{
    const size_t slot = (begin >> kTileBits) & (I.rec_slots - 1u);
    return I.rec_stat + ((size_t)row * I.rec_slots + slot) * I.rec_sstride;
}

// The statistics selected by kmask of a tile whose neurons share one
// population: the wave's sums into the tile's LDS sums (one global atomic
// per tile and field follows, instead of one per wave).
__device__ __forceinline__ void wave_tile_stats(unsigned long long *s_stat, bool valid, const long long *v,
                                                uint32_t kmask, uint32_t lane)
{
#pragma unroll
    for (int k = 0; k < kStatFields; ++k) {
        if (!(kmask & (1u << k)))
            continue;
        const unsigned long long s = wave_sum_u64(valid ? (unsigned long long)v[k] : 0ull);
        if (lane == 0)
            atomicAdd(&s_stat[k], s);
    }
}

// Adds this wave's per-population sums of the statistics selected by kmask
// (bit k: field k of kStatFields) of the lanes with `valid` into
// row[pop * kStatFields + k]: one 64-bit atomic per population present in
// the wave and field.  Called by the whole wave.
__device__ __forceinline__ void wave_pop_stats(long long *row, bool valid, uint32_t p, const long long *v,
                                               uint32_t kmask, uint32_t lane)
{
    unsigned long long rest = __ballot(valid);
    while (rest != 0ull) {
        const int src = __ffsll((long long)rest) - 1;
        const uint32_t ps = __shfl(p, src, kWave);
        const bool mine = valid && p == ps;
        rest &= ~__ballot(mine);
#pragma unroll
        for (int k = 0; k < kStatFields; ++k) {
            if (!(kmask & (1u << k)))
                continue;
            const unsigned long long s = wave_sum_u64(mine ? (unsigned long long)v[k] : 0ull);
            if ((int)lane == src)
                atomicAdd(reinterpret_cast<unsigned long long *>(row + (size_t)ps * kStatFields + k), s);
        }
    }
}

// Field mask of wave_pop_stats for the I_syn-based statistics of stat_mask.
__device__ __forceinline__ uint32_t current_fields(uint32_t stat_mask)
{
    return ((stat_mask & kStatI) ? 2u : 0u) | ((stat_mask & kStatReceptor) ? 0x3cu : 0u);
}

__device__ __forceinline__ float4 acc_to_delta(const unsigned long long *acc, uint32_t i, uint32_t rows = kBlock)
{
    float4 r;
    r.x = q40_to_f32((long long)acc[acc_at(i, 0u, rows)]);
    r.y = q40_to_f32((long long)acc[acc_at(i, 1u, rows)]);
    r.z = q40_to_f32((long long)acc[acc_at(i, 2u, rows)]);
    r.w = q40_to_f32((long long)acc[acc_at(i, 3u, rows)]);
    return r;
}

// Lane l gets lane l - 1's value (lane 0: fill), within the wave (DPP
// wave_shr:1, no LDS round trip).
__device__ __forceinline__ uint32_t wave_shr1(uint32_t v, uint32_t fill)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)fill, (int)v, 0x138, 0xf, 0xf, false);
}

// Lane l gets lane l + 1's value (lane 63: fill) (DPP wave_shl:1).
__device__ __forceinline__ uint32_t wave_shl1(uint32_t v, uint32_t fill)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)fill, (int)v, 0x130, 0xf, 0xf, false);
}

// Inclusive max-scan over the 64 lanes with DPP: shifts by 1, 2, 4, 8 within
// each row of 16 lanes (lanes shifted in from outside the row read 0, the
// identity), then the last lane of row 0 / 2 into rows 1 / 3 and the last
// lane of row 1 into rows 2 and 3.
__device__ __forceinline__ uint32_t wave_max_scan(uint32_t v)
{
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));   // row_shr:1
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));   // row_shr:2
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));   // row_shr:4
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));   // row_shr:8
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));   // row_bcast:15
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));   // row_bcast:31
    return v;
}

// Adds the wave's synapses past their queue's capacity (`over` per lane) to
// the engine's diagnostic count: one atomic per wave, and none when no lane
// has any (the usual case).
__device__ __forceinline__ void count_over(StepCtl *__restrict__ ctl, uint32_t over, uint32_t lane)
{
    if (__ballot(over != 0u) != 0ull) {
        const unsigned long long s = wave_sum_u64((unsigned long long)over);
        if (lane == 0)
            atomicAdd(&ctl->slot[blockIdx.x & (kCtlSlots - 1u)].spilled, s);
    }
}

// bin_pass with the loads and reservations of a lane's synapses one after the
// other (measured faster for one synapse per lane).
template <uint32_t K, uint32_t kFmt>
__device__ __forceinline__ void bin_pass_serial(const uint32_t *__restrict__ col_all, const void *w_all, uint32_t wfmt,
                                        int64_t row_begin, uint32_t len, uint32_t c0, uint32_t tile_base,
                                        const QueueTile *__restrict__ qtab, uint32_t *__restrict__ qcnt, size_t qset, uint32_t cshift,
                                        QSyn *__restrict__ queue, unsigned long long *__restrict__ spill,
                                        StepCtl *__restrict__ ctl, unsigned long long *seg_dst, uint32_t *seg_room,
                                        uint32_t lane)
{
    if (kFmt != kWeightAny)
        wfmt = kFmt;   // the launch's instances share one format: decoded without branches
    constexpr uint32_t kNone = 0xffffffffu;   // "no start" marker for positions
    const auto col = gp(col_all) + row_begin;
    const void *wt = w_row(w_all, row_begin, wfmt);
    {
        const uint32_t j0 = c0 + lane * K;
        uint32_t cv[K], tl[K];
        float2 wv[K];
#pragma unroll
        for (uint32_t k = 0; k < K; ++k) {
            if (j0 + k < len) {
                cv[k] = col[j0 + k];
                wv[k] = w_decode(w_raw(wt, j0 + k, wfmt), wfmt);
                tl[k] = (cv[k] & kColMask) >> kTileBits;
            } else {
                cv[k] = 0u;
                wv[k] = make_float2(0.0f, 0.0f);
                tl[k] = 0xfffffff0u + k;
            }
        }
        // neighbours across lanes; the pass boundaries end segments
        const uint32_t prev0 = wave_shr1(tl[K - 1], 0xffffffe0u);
        const uint32_t nextK = wave_shl1(tl[0], 0xffffffe1u);
        uint32_t last_start = kNone;
#pragma unroll
        for (uint32_t k = 0; k < K; ++k) {
            const uint32_t pv = (k == 0) ? prev0 : tl[k - 1];
            if (j0 + k < len && tl[k] != pv)
                last_start = j0 + k;
        }
        // exclusive max-scan over lanes of last_start (kNone counts as -1)
        const uint32_t sc = wave_max_scan((last_start == kNone) ? 0u : last_start + 1u);
        const uint32_t before = wave_shr1(sc, 0u);
        uint32_t open = (before != 0u) ? before - 1u : c0;   // segment open at the lane's first synapse
        uint32_t st[K];
        uint32_t over = 0;   // synapses of this lane's segments past their queue's capacity
#pragma unroll
        for (uint32_t k = 0; k < K; ++k) {
            const uint32_t j = j0 + k;
            const uint32_t pv = (k == 0) ? prev0 : tl[k - 1];
            const uint32_t nx = (k == K - 1) ? nextK : tl[k + 1];
            if (j < len && tl[k] != pv)
                open = j;
            st[k] = open;
            if (j < len && tl[k] != nx) {
                const uint32_t tg = tile_base + tl[k];
                const uint32_t n = j + 1u - open;
                const uint32_t base = gadd(&qcnt[count_slot(qset + tg, cshift)], n);
                const QueueTile td = qtab[tg];
                const uint32_t room = td.cap > base ? min(n, td.cap - base) : 0u;
                over += n - room;
                seg_dst[open - c0] = td.off + base;
                seg_room[open - c0] = room;
            }
        }
        count_over(ctl, over, lane);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (uint32_t k = 0; k < K; ++k) {
            const uint32_t j = j0 + k;
            if (j < len) {
                const uint32_t at = j - st[k];
                if (at < seg_room[st[k] - c0]) {
                    st_entry(queue, seg_dst[st[k] - c0] + at,
                             (cv[k] & 0xffu) | ((cv[k] & kKindBit) ? kQSynKind : 0u), wv[k].x, wv[k].y);
                } else if (spill != nullptr) {
                    unsigned long long *a = spill + (size_t)(cv[k] & kColMask) * 4u + ((cv[k] & kKindBit) ? 2u : 0u);
                    gadd(a, f32_to_q40(wv[k].x));
                    gadd(a + 1, f32_to_q40(wv[k].y));
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}


// Queues synapses c0 .. c0 + 64 K - 1 of one fired row (one pass) for the next
// launch: each synapse's target index within its tile, channel pair and
// weight pair go into the target tile's queue.  The row's synapses are
// ordered by target, so the synapses of one tile form segments; each segment
// reserves its slots with one atomic add on the tile's count and its
// synapses are stored contiguously.  Called by a whole wave with
// wave-uniform arguments.  Lane l holds synapses c0 + K l .. c0 + K l + K - 1
// of the row (segments end at pass boundaries).  A synapse's segment start is
// the last start at or before it (within the lane, else from a wave max-scan
// of the lanes' last starts); the lane holding the segment's last synapse
// reserves and publishes the destination and the number of the segment's
// synapses that fit the queue in seg_dst / seg_room (this wave's 64 K LDS
// entries, indexed by segment start within the pass).  Synapses past the
// queue's capacity add their weights into the target's spill accumulator
// instead (64-bit integer atomics, Q23.40 like the LDS sums, so the total
// does not depend on which path a synapse took).
template <uint32_t K, uint32_t kFmt>
__device__ __forceinline__ void bin_pass(const uint32_t *__restrict__ col_all, const void *w_all, uint32_t wfmt,
                                        int64_t row_begin, uint32_t len, uint32_t c0, uint32_t tile_base,
                                        const QueueTile *__restrict__ qtab, uint32_t *__restrict__ qcnt, size_t qset, uint32_t cshift,
                                        QSyn *__restrict__ queue, unsigned long long *__restrict__ spill,
                                        StepCtl *__restrict__ ctl, unsigned long long *seg_dst, uint32_t *seg_room,
                                        uint32_t lane)
{
    if (kFmt != kWeightAny)
        wfmt = kFmt;   // the launch's instances share one format: decoded without branches
    constexpr uint32_t kNone = 0xffffffffu;   // "no start" marker for positions
    const auto col = gp(col_all) + row_begin;
    const void *wt = w_row(w_all, row_begin, wfmt);
    const uint32_t j0 = c0 + lane * K;
    // Every lane loads K synapses without a branch (past the row's end it
    // re-reads the last one and marks it invalid), so all loads are in
    // flight together.
    uint32_t cv[K], tl[K], jj[K];
    float2 wv[K];
    bool ok[K];
    unsigned long long wr[K];
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
        ok[k] = j0 + k < len;
        jj[k] = ok[k] ? j0 + k : len - 1u;
        cv[k] = col[jj[k]];
    }
    w_load<K, uint32_t>(wr, wt, jj, wfmt);
#pragma unroll
    for (uint32_t k = 0; k < K; ++k)
        wv[k] = w_decode(wr[k], wfmt);
#pragma unroll
    for (uint32_t k = 0; k < K; ++k)
        tl[k] = ok[k] ? (cv[k] & kColMask) >> kTileBits : 0xfffffff0u + k;
    // neighbours across lanes; the pass boundaries end segments
    const uint32_t prev0 = wave_shr1(tl[K - 1], 0xffffffe0u);
    const uint32_t nextK = wave_shl1(tl[0], 0xffffffe1u);
    uint32_t last_start = kNone;
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
        const uint32_t pv = (k == 0) ? prev0 : tl[k - 1];
        if (ok[k] && tl[k] != pv)
            last_start = j0 + k;
    }
    // exclusive max-scan over lanes of last_start (kNone counts as -1)
    const uint32_t sc = wave_max_scan((last_start == kNone) ? 0u : last_start + 1u);
    const uint32_t before = wave_shr1(sc, 0u);
    uint32_t open = (before != 0u) ? before - 1u : c0;   // segment open at the lane's first synapse
    uint32_t st[K];
    bool end[K];
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
        const uint32_t pv = (k == 0) ? prev0 : tl[k - 1];
        const uint32_t nx = (k == K - 1) ? nextK : tl[k + 1];
        if (ok[k] && tl[k] != pv)
            open = j0 + k;
        st[k] = open;
        end[k] = ok[k] && tl[k] != nx;
    }
    // Reservations: every segment-end synapse issues its atomic and its
    // tile's queue range before any result is used, so they overlap.
    uint32_t base[K];
    unsigned long long qoff[K];
    uint32_t qcap[K];
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
        base[k] = 0u;
        qoff[k] = 0ull;
        qcap[k] = 0u;
        if (end[k]) {
            const uint32_t tg = tile_base + tl[k];
            base[k] = gadd(&qcnt[count_slot(qset + tg, cshift)], j0 + k + 1u - st[k]);
            qoff[k] = qtab[tg].off;
            qcap[k] = qtab[tg].cap;
        }
    }
    uint32_t over = 0;   // synapses of this lane's segments past their queue's capacity
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
        if (end[k]) {
            const uint32_t n = j0 + k + 1u - st[k];
            const uint32_t room = qcap[k] > base[k] ? min(n, qcap[k] - base[k]) : 0u;
            over += n - room;
            seg_dst[st[k] - c0] = qoff[k] + base[k];
            seg_room[st[k] - c0] = room;
        }
    }
    count_over(ctl, over, lane);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
        if (ok[k]) {
            const uint32_t at = j0 + k - st[k];
            if (at < seg_room[st[k] - c0]) {
                st_entry(queue, seg_dst[st[k] - c0] + at,
                         (cv[k] & 0xffu) | ((cv[k] & kKindBit) ? kQSynKind : 0u), wv[k].x, wv[k].y);
            } else if (spill != nullptr) {
                unsigned long long *a = spill + (size_t)(cv[k] & kColMask) * 4u + ((cv[k] & kKindBit) ? 2u : 0u);
                gadd(a, f32_to_q40(wv[k].x));
                gadd(a + 1, f32_to_q40(wv[k].y));
            }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}


// A tile's recorded sums in LDS (tiles of one population).
struct TileRec {
    unsigned long long stat[kStatFields];
    uint32_t count;   // emitted neurons that population counts include
};

// Neuron state of one lane.
struct Lane {
    float4 J;
    float V, iou;
    int32_t t;
    uint32_t fl;
};

__device__ __forceinline__ Lane load_lane(unsigned char *state, uint32_t i)
{
    Lane x;
    x.J = ld_J(state, i);
    x.V = *st_at<kStV, float>(state, i);
    x.t = *st_at<kStT, int32_t>(state, i);
    x.fl = *st_at<kStFlag, uint8_t>(state, i);
    x.iou = *st_at<kStIou, float>(state, i);
    return x;
}

// The tile's parameter record: of the tile (scalar loads), or of the lane's
// class.
template <bool kUniform>
__device__ __forceinline__ ParamRec load_params(TilePtr d, uint32_t i)
{
    ParamRec r;
    if (kUniform) {
        r.a = ld4c(&d->prm->a);
        r.b = ld4c(&d->prm->b);
        r.g = ld4c(&d->prm->g);
        r.v = ld4c(&d->prm->v);
        r.d = ld4c(&d->prm->d);
    } else {
        const float4 *p = &d->prm[gp(d->cls)[i]].a;
        r.a = ld4(p, 0);
        r.b = ld4(p, 1);
        r.g = ld4(p, 2);
        r.v = ld4(p, 3);
        r.d = ld4(p, 4);
    }
    return r;
}

// LIF update of one substep (membrane_voltage.cpp:114-195): a.z = dt_sub / C.
__device__ __forceinline__ bool lif(Lane &x, uint32_t &f, const ParamRec &q, float Ieff)
{
    float cvi = q.b.x * (q.a.w - x.V);
    cvi = cvi + Ieff;
    cvi = cvi + q.b.y;
    const float Vn = x.V + q.a.z * cvi;
    const bool held = x.t < 0;
    const bool spk = !held && Vn >= q.a.y;
    const float Vh = f ? q.a.x : x.V;   // refractory: reset once after the spike
    x.V = held ? Vh : (spk ? q.a.y : Vn);
    x.t = held ? x.t + 1 : (spk ? 1 - __float_as_int(q.b.w) : x.t);
    f = spk ? 1u : 0u;
    return spk;
}

// One OU step (extern_stimuli.cpp:39-112).
__device__ __forceinline__ float ou_step(float iou, float mu, float f1, float f2s, float xi)
{
    return iou + (f1 * (mu - iou) + f2s * xi);
}

// The step's normal draw of a tile with one population, one substep and the
// OU current on.  Taken while the tile's loads are in flight: its 100
// instructions wait for nothing but the step index (with the emitted rows'
// words read as early: 200k x 250 9.8 -> 9.6 us a step, 10k 5.25 -> 5.10,
// eight instances 12.7 -> 11.9).
__device__ __forceinline__ float ou_draw(TilePtr d, uint32_t tid, int64_t step)
{
    constexpr uint32_t kOne = kTileOnePop | kTileOneSub | kTileOuOn;
    return (d->flags & kOne) == kOne ? ou_normal(d->seed, d->begin + tid, (uint64_t)step) : 0.0f;
}

// Every substep of a tile whose neurons share one population, with one
// substep per step (the usual case: straight-line code, the OU factors in
// scalar registers).  Returns whether the lane's neuron emitted.
__device__ __forceinline__ bool step_lane_one(TilePtr d, Lane &x, const ParamRec &q, float isyn, uint32_t li,
                                              int64_t step, float xi)
{
    uint32_t f = x.fl & kFlagSpike;
    float Ieff = isyn;
    if (d->flags & kTileOuOn) {
        x.iou = ou_step(x.iou, d->mu, d->f1, d->f2s, xi);
        Ieff = isyn + x.iou;
    }
    bool emit = lif(x, f, q, Ieff);
    if (!(d->flags & kTileOu))   // spike.cpp:55-62: f_rec = f | (U < noise_rate)
        emit = f || (noise_uniform(d->seed, li, (uint64_t)step) < q.b.z);
    x.fl = f;
    return emit;
}

// The same for any number of substeps and populations: p is the lane's
// population.
__device__ __forceinline__ bool step_lane_any(TilePtr d, InstPtr I, Lane &x, const ParamRec &q, float isyn,
                                              uint32_t li, int64_t step, uint32_t p)
{
    const auto pop = gp(I->pops) + p;
    const float mu = pop->mu, f1 = pop->f1, f2s = pop->f2s;
    const bool ou = (d->flags & kTileOu) != 0u && pop->ou_on != 0u;
    const int32_t T = I->t_steps;
    uint32_t f = x.fl & kFlagSpike;
    bool emit = false;
    for (int32_t s = 0; s < T; ++s) {
        float Ieff = isyn;
        if (ou) {
            x.iou = ou_step(x.iou, mu, f1, f2s, ou_normal(d->seed, li, (uint64_t)step * (uint64_t)T + (uint64_t)s));
            Ieff = isyn + x.iou;
        }
        emit = lif(x, f, q, Ieff) || emit;
        if (s < T - 1) {
            x.J.x = x.J.x * q.d.x;
            x.J.y = x.J.y * q.d.y;
            x.J.z = x.J.z * q.d.z;
            x.J.w = x.J.w * q.d.w;
            isyn = syn_current(q.g, q.v, x.J, x.V);
        }
    }
    if (!(d->flags & kTileOu))
        emit = f || (noise_uniform(d->seed, li, (uint64_t)step) < q.b.z);
    x.fl = f;
    return emit;
}

// Fold of the delta, the recorded statistics, and every substep of OU + LIF
// (or of the noise mode) of the tile's neurons; returns whether the lane's
// neuron emitted a spike and writes the state back.  xi: the step's normal
// draw, where the tile has one (ou_draw).
template <bool kStat>
__device__ __forceinline__ bool step_lane(TilePtr d, Lane &x, const ParamRec &q, const float4 dl, bool active,
                                          uint32_t tid, uint32_t lane, int64_t step, float xi, uint32_t &p,
                                          TileRec &rec)
{
    const bool one_pop = (d->flags & kTileOnePop) != 0u;
    const uint32_t li = d->begin + tid;
    const InstPtr I = cp(d->inst);
    p = d->pop0;
    float isyn = 0.0f;
    if (active) {
        if (!(x.fl & kFlagFolded))
            x.J = fold_delta(x.J, q.d, dl);
        isyn = syn_current(q.g, q.v, x.J, x.V);
        if (!one_pop) {
            // the population of neuron li (populations in order of their ends)
            const auto pops = gp(I->pops);
            const uint32_t npop = I->npop;
            while (p + 1 < npop && li >= pops[p].end)
                ++p;
        }
    }
    // stat_result.cpp:266-391: population sums, blocked neurons excluded.
    // The I_syn-based statistics belong to the previous step (its J is
    // complete only now: J folded, V before this step's update); the V
    // statistic (after the update, below) to this one.
    const bool stat_on = kStat && (d->flags & kTileStat) != 0u;
    int64_t row_v = 0;
    bool stat_valid = false;
    if (stat_on) {
        row_v = step - I->rec_step0;
        stat_valid = active && !gp(I->blocked)[active ? li : d->begin];
        const uint32_t cf = current_fields(I->stat_mask);
        if (cf != 0u && row_v - 1 >= 0 && row_v - 1 < (int64_t)I->rec_len) {
            long long stv[kStatFields] = {};
            const float4 rc = receptor_currents(q.g, q.v, x.J, x.V);
            stv[1] = stat_q(isyn);
            stv[2] = stat_q(rc.x);
            stv[3] = stat_q(rc.y);
            stv[4] = stat_q(rc.z);
            stv[5] = stat_q(rc.w);
            if (one_pop)
                wave_tile_stats(rec.stat, stat_valid, stv, cf, lane);
            else
                wave_pop_stats(rec_stat_row(*I, row_v - 1, d->begin), stat_valid, p, stv, cf, lane);
        }
    }
    bool emit = false;
    if (active) {
        if ((d->flags & (kTileOnePop | kTileOneSub)) == (kTileOnePop | kTileOneSub))
            emit = step_lane_one(d, x, q, isyn, li, step, xi);
        else
            emit = step_lane_any(d, I, x, q, isyn, li, step, p);
        *st_at<kStV, float>(d->state, tid) = x.V;
        *st_at<kStT, int32_t>(d->state, tid) = x.t;
        *st_at<kStFlag, uint8_t>(d->state, tid) = (uint8_t)(x.fl | (emit ? kFlagEmit : 0u));
        *st_at<kStIou, float>(d->state, tid) = x.iou;
        st_J(d->state, tid, x.J);
    }
    if (stat_on && (I->stat_mask & kStatV) && row_v >= 0 && row_v < (int64_t)I->rec_len) {
        long long stv[kStatFields] = {};
        stv[0] = stat_q(x.V);
        if (one_pop)
            wave_tile_stats(rec.stat, stat_valid, stv, 1u, lane);
        else
            wave_pop_stats(rec_stat_row(*I, row_v, d->begin), stat_valid, p, stv, 1u, lane);
    }
    return emit;
}

// Per-population counts of a wave with emitted neurons
// (stat_result.cpp:161-206; blocked neurons are not counted): one LDS add
// per wave in a tile of one population, else one atomic per population
// present in the wave.
__device__ __forceinline__ void count_wave(TilePtr d, InstPtr I, bool emit, uint32_t tid, uint32_t lane,
                                           int64_t step, uint32_t p, TileRec &rec)
{
    const int64_t row = step - I->rec_step0;
    if (row < 0 || row >= (int64_t)I->rec_len)
        return;
    const bool counted = emit && !gp(I->blocked)[d->begin + tid];
    unsigned long long rest = __ballot(counted);
    if (d->flags & kTileOnePop) {
        if (lane == 0 && rest != 0ull)
            atomicAdd(&rec.count, (uint32_t)__popcll(rest));
        return;
    }
    while (rest != 0ull) {
        const int src = __ffsll((long long)rest) - 1;
        const uint32_t ps = __shfl(p, src, kWave);
        const unsigned long long same = __ballot(counted && p == ps);
        if ((int)lane == src)
            gadd(rec_count_row(*I, row, d->begin) + ps, (uint32_t)__popcll(same));
        rest &= ~same;
    }
}

// The recorded sums of a tile of one population, after the barrier that
// follows the waves' LDS adds.
template <bool kStat>
__device__ __forceinline__ void put_tile_rec(TilePtr d, InstPtr I, uint32_t tid, int64_t step,
                                             const TileRec &rec)
{
    if (!(d->flags & kTileOnePop))
        return;
    // rec.count is nonzero only inside the recorded rows
    if (tid == 0 && rec.count != 0u)
        gadd(rec_count_row(*I, step - I->rec_step0, d->begin) + d->pop0, rec.count);
    if (kStat && (d->flags & kTileStat) && tid < (uint32_t)kStatFields) {
        // fields of the current step (V) and of the step before (I_syn)
        const int64_t r = step - I->rec_step0 - (tid == 0 ? 0 : 1);
        const uint32_t on = ((I->stat_mask & kStatV) ? 1u : 0u) | current_fields(I->stat_mask);
        if (((on >> tid) & 1u) && r >= 0 && r < (int64_t)I->rec_len)
            gadd(reinterpret_cast<unsigned long long *>(rec_stat_row(*I, r, d->begin)) +
                     (size_t)d->pop0 * kStatFields + tid,
                 rec.stat[tid]);
    }
}

// How the tiles of a k_step launch get their input and pass on their rows:
// from queues (or gather's delta, a flag of the tile), the emitted rows binned
// by the tile itself (kTileBin) or left to a k_bin launch (kQueues); or from
// the emitted rows directly (kDirect).
enum : int { kQueues = 0, kDirect = 1, kTileBin = 2 };

// What a tile's step reads before its queue.
template <bool kUniform, int kMode>
struct StepIn {
    TilePtr d;
    QueuePtr q;
    uint32_t cnt, lc;
    int64_t step, stamp;
    Lane x;
    ParamRec prm;
    bool active;

    __device__ __forceinline__ StepIn(TilePtr tp, QueuePtr qp, uint32_t par, uint32_t tid)
    {
        d = tp;
        q = qp;
        if (kMode != kDirect)
            cnt = *cp(count(par));
        step = cp(d->step)[par];
        stamp = cp(d->step)[2u + par];
        active = tid < d->count;
        lc = active ? tid : 0u;   // in-range index for idle lanes
        x = load_lane(d->state, lc);
        if (kUniform)
            prm = load_params<true>(d, lc);
    }
    __device__ __forceinline__ uint32_t *count(uint32_t par) const
    {
        return q->count + count_slot((size_t)par * q->ntiles + blockIdx.x, q->cshift);
    }
    __device__ __forceinline__ const QSyn *queue(uint32_t par) const { return d->queue + (size_t)par * d->qslots; }
};

// The wave's own counters: events (sum of the fired rows' lengths) and
// spikes, added without waiting for a read.
// Returns the fired lane's row.
struct RowSpan {
    int64_t first;
    uint32_t len;
};

__device__ __forceinline__ RowSpan count_fired(TilePtr d, InstPtr I, bool emit, unsigned long long m, uint32_t tid,
                                               uint32_t lane, uint32_t w)
{
    RowSpan r{0, 0u};
    if (emit) {
        r.first = gp(d->rowptr)[tid];
        r.len = (uint32_t)(gp(d->rowptr)[tid + 1] - r.first);
    }
    const unsigned long long ev = wave_sum_u64((unsigned long long)r.len);
    if (lane == 0) {
        unsigned long long *c = I->wave_ctr + 2u * ((d->begin >> 6) + w);
        gadd(c, ev);
        gadd(c + 1, (unsigned long long)__popcll(m));
    }
    return r;
}

// Gather propagation: the wave's fired rows with synapses go to the tile's
// fired list of set par ^ 1 for the next launch's k_gather (one atomic per
// wave, on a count shared with 1/64 of the tiles).
__device__ __forceinline__ void list_fired(TilePtr d, InstPtr I, bool emit, uint32_t par, uint32_t tid, uint32_t lane)
{
    const uint32_t len = emit ? (uint32_t)(gp(d->rowptr)[tid + 1] - gp(d->rowptr)[tid]) : 0u;
    const bool has = emit && len != 0u;
    const unsigned long long mg = __ballot(has);
    if (mg != 0ull) {
        const uint32_t list = (par ^ 1u) * kFiredLists + ((d->begin >> kTileBits) & (kFiredLists - 1u));
        const int lg = __ffsll((long long)mg) - 1;
        uint32_t gb = 0;
        if ((int)lane == lg)
            gb = gadd(I->fcount + (size_t)list * kFiredCountStride, (uint32_t)__popcll(mg));
        gb = (uint32_t)__builtin_amdgcn_readlane((int)gb, lg);
        if (has)
            gp(I->fired)[(size_t)list * I->fcap + gb + (uint32_t)__popcll(mg & ((1ull << lane) - 1ull))] =
                d->begin + tid;
    }
}

// LDS of a tile that bins its own rows: the rows, and per wave the segments
// of one pass.
template <uint32_t K>
struct TileRows {
    unsigned long long seg_dst[4 * kWave * K];
    uint32_t seg_room[4 * kWave * K];
    long long rb[kBlock];    // fired rows of the tile: first synapse
    uint32_t len[kBlock];    // and length
    uint32_t n;
};

// The pass list of tile t of nt: contiguous ranges of tiles, so a list's rows
// share target tiles.
__device__ __forceinline__ uint32_t pass_list(uint32_t t, uint32_t nt)
{
    return (uint32_t)(((uint64_t)t * kFiredLists) / nt);
}

// One tile's step (the body of k_step).  kUniform: every neuron of the tile
// has the same parameter class, so the parameter record is read once per
// tile through the scalar unit instead of per lane.  kStat: some instance
// records population statistics (their code costs registers that a launch
// without them does not spend).
// kMode: kQueues, kDirect or kTileBin; K: with kTileBin, synapses per lane in
// a binning pass (a pass is 64 K synapses).
template <bool kUniform, uint32_t kFmt, bool kStat, int kMode, uint32_t K>
__device__ __forceinline__ void step_tile(TilePtr tp, QueuePtr qp, uint32_t par, unsigned long long *acc,
                                          unsigned long long *s_bits, TileRec &rec, DirectList *ls,
                                          TileRows<K> *rows)
{
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = __lane_id();
    const uint32_t w = tid / kWave;
    bool emit, pull;
    uint32_t p;
    int64_t step;
    {
        // Everything a silent step reads is addressed from the descriptor, so
        // all of it is in flight before anything waits: the queue count, the
        // step index and deferral stamp, the neuron state, the parameter
        // record and the queue head (the queue is complete when the launch
        // starts; entries past the count are ignored, and the queue buffer has
        // kQueuePrefetch slots of slack at its end, so the read needs no
        // branch).
        StepIn<kUniform, kMode> e(tp, qp, par, tid);
        // One register quad for both: the delta that k_gather wrote (gather
        // propagation), or the queue entry.
        float4 ahead = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (kMode == kDirect) {
        } else if (e.d->flags & kTileGather) {
            ahead = ld4(e.d->dlt, e.lc);
        } else {
            const QSyn h = ld_entry(e.queue(par), min(tid, kQueuePrefetch - 1u));
            ahead = make_float4(__uint_as_float(h.key), h.w0, h.w1, 0.0f);
        }
        // A tile pulls (the pull propagation, never with gather) when its
        // queue overflowed or rows were deferred into this set: rare (volleys).
        const bool gat = kMode == kDirect || (e.d->flags & kTileGather) != 0u;   // no queue
        bool over = !gat && e.cnt > e.d->qcap;
        uint32_t cnt = gat ? 0u : min(e.cnt, e.d->qcap);
        pull = !gat && (e.d->flags & kTilePull) && (over || e.stamp == e.step + 1);
        const uint32_t begin_word = kMode == kDirect ? (e.d->begin >> kTileBits) * kBitWords : 0u;
        DirectIds ids(kMode == kDirect ? e.d->bits - begin_word + (size_t)par * e.d->ntiles * kBitWords : nullptr,
                      kMode == kDirect ? e.d->ntiles : 0u, tid);
        clear_row(acc, tid);
        const float xi = ou_draw(e.d, tid, e.step);
        if (tid == 0) {
            rec.count = 0u;
            if (kMode == kDirect)
                ls->n = 0u;
            if (kMode == kTileBin)
                rows->n = 0u;
        }
        if (kStat && tid < (uint32_t)kStatFields)
            rec.stat[tid] = 0ull;
        __syncthreads();
        if (pull) {
            // An overflowed queue is ignored: every emitted row then comes
            // through the in-edges.
            accumulate_tile(acc, e.queue(par), over ? 0u : cnt, QSyn{}, 0u, tid);
            pull_tile<kFmt>(acc, *cp(e.d->inst), par, e.d->begin >> kTileBits, over, tid);
            if (tid == 0)
                gadd(&again(qp)->ctl->slot[blockIdx.x & (kCtlSlots - 1u)].pulled, 1ull);
            // Everything again: nothing loaded above is live across the call
            // (what is, the compiler keeps in spilled registers from the
            // kernel's start, in every tile).
            e = StepIn<kUniform, kMode>(again(tp), again(qp), par, tid);
            pull = true;
            over = false;
            cnt = 0u;
        }
        if (kMode == kDirect) {
            if (direct_tile<kFmt>(acc, *ls, *cp(e.d->inst), ids, par, e.d->begin >> kTileBits, tid) && tid == 0) {
                // the tile pulled; and its own rows, if any, went by the pull
                CtlSlot &c = qp->ctl->slot[blockIdx.x & (kCtlSlots - 1u)];
                gadd(&c.pulled, 1ull);
                const auto b = gp(e.d->bits) + (size_t)par * e.d->ntiles * kBitWords;
                if ((b[0] | b[1] | b[2] | b[3]) != 0ull)
                    gadd(&c.deferred, 1ull);
            }
        } else {
            accumulate_tile(acc, e.queue(par), cnt, QSyn{__float_as_uint(ahead.x), ahead.y, ahead.z}, kQueuePrefetch,
                            tid);
        }
        __syncthreads();
        if (!kUniform)   // a rare tile: its lanes' records do not wait in registers
            e.prm = load_params<false>(e.d, e.lc);
        step = e.step;
        if (over && e.active) {   // (a tile that pulls took everything)
            const InstPtr I = cp(e.d->inst);
            take_spill(acc, I->spill, I->n, par, e.d->begin + tid, tid, true);   // synapses past the queue's capacity
        }
        if (tid == 0) {
            if (kMode != kDirect)
                *gp(e.count(par)) = 0u;   // this launch consumed the queue
            if (e.d->begin == 0)
                gp(e.d->step)[par ^ 1u] = step + 1;   // no tile of this launch reads this slot
        }
        const float4 dl = kMode != kDirect && (e.d->flags & kTileGather) ? ahead : acc_to_delta(acc, tid);
        emit = step_lane<kStat>(e.d, e.x, e.prm, dl, e.active, tid, lane, step, xi, p, rec);
    }

    const TilePtr d = again(tp);
    const InstPtr I = cp(d->inst);
    const bool gat = (d->flags & kTileGather) != 0u;
    // Spike propagation (presynaptic_voltage.cpp:122-225): with gather the
    // fired rows go to lists for the next k_gather; else they are binned by
    // the tile (below) or listed as passes for the k_bin launch that follows,
    // or left as bits and ids (direct).
    const unsigned long long m = __ballot(emit);
    if (lane == 0)
        s_bits[w] = m;
    RowSpan span{0, 0u};
    if (m != 0ull) {
        span = count_fired(d, I, emit, m, tid, lane, w);
        if (kMode == kTileBin && !gat) {
            uint32_t base = 0;
            if (lane == 0)
                base = atomicAdd(&rows->n, (uint32_t)__popcll(m));
            base = (uint32_t)__builtin_amdgcn_readlane((int)base, 0);
            if (emit) {
                const uint32_t k = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
                rows->rb[k] = span.first;
                rows->len[k] = span.len;
            }
        }
        if (gat)
            list_fired(d, I, emit, par, tid, lane);
        if (I->rec_counts != nullptr)
            count_wave(d, I, emit, tid, lane, step, p, rec);
    }
    __syncthreads();
    if (kMode == kDirect) {
        // the tile's rows: their bits, then the count and the first ids
        if (w == 0) {
            unsigned long long word = s_bits[lane & 3u];
            uint32_t c = (uint32_t)__popcll(word);
            unsigned long long first = 0ull;
            c = (uint32_t)__builtin_amdgcn_readlane((int)c, 0) + (uint32_t)__builtin_amdgcn_readlane((int)c, 1) +
                (uint32_t)__builtin_amdgcn_readlane((int)c, 2) + (uint32_t)__builtin_amdgcn_readlane((int)c, 3);
            if (c != 0u && c <= kDirectIds) {
                uint32_t k = 2u;
                for (uint32_t q = 0; q < 4u; ++q)
                    for (unsigned long long r = s_bits[q]; r != 0ull; r &= r - 1ull, ++k)
                        first |= (unsigned long long)(q * kWave + (uint32_t)__ffsll((long long)r) - 1u) << (8u * k);
            }
            if (lane < 5u)
                gp(d->bits)[(size_t)(par ^ 1u) * d->ntiles * kBitWords + lane] = lane < 4u ? word : (first | c);
        }
    }
    put_tile_rec<kStat>(d, I, tid, step, rec);
    if (kMode == kDirect || gat)
        return;
    // A tile with many emitted rows (a synchronous volley) leaves them to
    // the consumers' pull: binning them would overflow the queues.  A tile
    // that pulls in this launch (the volley is under way) defers only from
    // four times the count: the volley's tail, where a few tiles still emit
    // that many, would otherwise cost the next step a pull of every in-edge.
    bool defer = false;
    const unsigned long long b = s_bits[lane & 3u];
    if (d->flags & kTilePull) {
        const uint32_t c = (uint32_t)__popcll(b);
        const uint32_t nr = (uint32_t)__builtin_amdgcn_readlane((int)c, 0) +
                            (uint32_t)__builtin_amdgcn_readlane((int)c, 1) +
                            (uint32_t)__builtin_amdgcn_readlane((int)c, 2) +
                            (uint32_t)__builtin_amdgcn_readlane((int)c, 3);
        if (nr != 0u) {
            const uint32_t dm = I->defer_min;
            defer = dm != 0u && nr >= (pull ? 4u * dm : dm);
            if (defer && tid == 0) {
                gp(d->step)[2u + (par ^ 1u)] = step + 2;   // consumer's step + 1 (0: none)
                gadd(&again(qp)->ctl->slot[blockIdx.x & (kCtlSlots - 1u)].deferred, 1ull);
            }
        }
    }
    // the tile's emitted and deferred rows, one 64-byte store
    if (tid < kBitWords && (d->flags & kTilePull))
        gp(d->bits)[(size_t)(par ^ 1u) * d->ntiles * kBitWords + tid] = (tid < 4u || defer) ? b : 0ull;
    if (kMode == kQueues && m != 0ull && !defer) {
        // The wave's passes onto its list: one atomic on a count shared with
        // 1/64 of the tiles.
        const uint32_t np = (span.len + kBinPass - 1u) / kBinPass;
        const uint32_t incl = wave_add_scan(np);
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        if (total != 0u) {
            const uint32_t list = pass_list(d->begin >> kTileBits, d->ntiles);
            uint32_t at = 0;
            if (lane == 0)
                at = gadd(I->pass_count + ((par * kFiredLists + list) * kFiredCountStride), total);
            at = (uint32_t)__builtin_amdgcn_readlane((int)at, 0) + incl - np;
            const auto out = gp(I->passes) + ((size_t)list * I->passcap + at);
            for (uint32_t k = 0; k < np; ++k)
                out[k] = ((unsigned long long)(span.first + (int64_t)(k * kBinPass)) << 8) |
                         (min(span.len - k * kBinPass, kBinPass) - 1u);
        }
    }
    if constexpr (kMode == kTileBin) {
        // The passes of the tile's rows, dealt round-robin to its four waves,
        // so one long row does not keep a single wave busy while the others
        // idle.
        const uint32_t nbin = defer ? 0u : rows->n;
        if (nbin == 0u)
            return;
        const QueuePtr qs = again(qp);
        unsigned long long *spill_out =
            (d->flags & kTilePull) ? nullptr : I->spill + (size_t)(par ^ 1u) * I->n * 4u;
        QSyn *q_out = I->queue + (size_t)(par ^ 1u) * d->qslots;
        uint32_t pass = 0;
        for (uint32_t r = 0; r < nbin; ++r) {
            const long long rb_s = rows->rb[r];
            const uint32_t len_s = rows->len[r];
            for (uint32_t c0 = 0; c0 < len_s; c0 += kWave * K, ++pass) {
                if ((pass & 3u) != w)
                    continue;
                if constexpr (K == 1)
                    bin_pass_serial<K, kFmt>(I->col, I->w, I->wfmt, (int64_t)rb_s, len_s, c0, I->tile_base, qs->tile,
                                             qs->count, (size_t)(par ^ 1u) * qs->ntiles, qs->cshift, q_out, spill_out,
                                             qs->ctl, rows->seg_dst + w * kWave * K, rows->seg_room + w * kWave * K,
                                             lane);
                else
                    bin_pass<K, kFmt>(I->col, I->w, I->wfmt, (int64_t)rb_s, len_s, c0, I->tile_base, qs->tile,
                                      qs->count, (size_t)(par ^ 1u) * qs->ntiles, qs->cshift, q_out, spill_out, qs->ctl,
                                      rows->seg_dst + w * kWave * K, rows->seg_room + w * kWave * K, lane);
            }
        }
    }
}

// The step of launch parity `par`: takes the input of set par, passes its
// emitted rows on into set par ^ 1, reads the step index from step[par] and advances it into step[par ^ 1].
// Seven waves per SIMD: at eight the compiler spills up to 14 registers, and
// the 2M-neuron step takes 42.3 us instead of 40.5 (1200 rows per step), a
// 10k-neuron step by direct propagation 5.7 instead of 5.3.
template <uint32_t kFmt, bool kStat, int kMode, uint32_t K>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(K == 4 ? 6 : 7))) void k_step(const TileDesc *tiles,
                                                                                         const QueueSet *queues,
                                                                                         uint32_t par)
{
    __shared__ unsigned long long acc[kBlock * 4];
    __shared__ unsigned long long s_bits[4];   // emitted rows per wave
    __shared__ TileRec rec;
    DirectList *ls = nullptr;
    if constexpr (kMode == kDirect) {
        __shared__ DirectList list;
        ls = &list;
    }

    TileRows<K> *rows = nullptr;
    if constexpr (kMode == kTileBin) {
        __shared__ TileRows<K> r;
        rows = &r;
    }

    const TilePtr tp = cp(tiles + blockIdx.x);
    if (tp->flags & kTileUniform)
        step_tile<true, kFmt, kStat, kMode, K>(tp, cp(queues), par, acc, s_bits, rec, ls, rows);
    else
        step_tile<false, kFmt, kStat, kMode, K>(tp, cp(queues), par, acc, s_bits, rec, ls, rows);
}

// Binning of the passes listed by the k_step launch of parity `par` into
// queue set par ^ 1.  A workgroup takes an equal share of them, consecutive
// ones: rows of neighbouring neurons reach the same target tiles (a voxel's
// rows share theirs), so it counts its synapses per target tile in LDS,
// reserves each tile's share with one device atomic, and writes every
// synapse's entry to its tile's queue at reserved start + rank.
// Without it (one reservation per row and target tile, in the tiles whose
// neurons fired) binning is 22 of 50 us of the 2M-neuron block's step:
// returning atomics on single counts are served at about 2.7e10 per second,
// and a row of 500 synapses makes 160-190 of them; with it 14.5 of 43.5.
// Groups of 32 source tiles instead of equal shares of the passes took 19 us:
// the fullest group's time.
// The counts of a round live in min(ntiles, kBinMaxTiles) LDS words;
// instances with more tiles are binned in windows of that many target tiles.
// Also empties the lists of set par ^ 1 (the next k_step's; their last reader
// was the previous k_bin).
template <uint32_t kFmt>
__global__ __launch_bounds__(kBinBlock) void k_bin(const BinDesc *__restrict__ groups, const QueueSet *queues,
                                                   uint32_t par)
{
    constexpr uint32_t kWaves = kBinBlock / kWave;
    extern __shared__ uint32_t hist[];               // min(ntiles, kBinMaxTiles)
    __shared__ uint32_t s_list[kFiredLists];         // passes of the lists before
    __shared__ uint16_t s_touch[kWaves * kBinDeep * kBinPass];   // target tiles of a round, each once
    __shared__ uint32_t s_ntouch;
    const uint32_t tid = threadIdx.x, lane = __lane_id(), w = tid / kWave;
    const auto bd = cp(groups + blockIdx.x);
    const InstPtr I = cp(bd->inst);
    const uint32_t T = I->ntiles, set = par ^ 1u;
    const uint32_t cnt = gp(I->pass_count)[(par * kFiredLists + lane) * kFiredCountStride];
    const uint32_t incl = wave_add_scan(cnt);
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
    if (w == 0)
        s_list[lane] = incl - cnt;
    if (bd->part == 0u && tid < kFiredLists)
        gp(I->pass_count)[(set * kFiredLists + tid) * kFiredCountStride] = 0u;
    const uint32_t lo = (uint32_t)((uint64_t)total * bd->part / bd->parts);
    const uint32_t hi = (uint32_t)((uint64_t)total * (bd->part + 1u) / bd->parts);
    if (lo == hi)
        return;
    for (uint32_t t = tid; t < min(T, (uint32_t)kBinMaxTiles); t += kBinBlock)
        hist[t] = 0u;
    if (tid == 0)
        s_ntouch = 0u;
    const QueuePtr qs = cp(queues);
    const uint32_t wfmt = kFmt != kWeightAny ? kFmt : I->wfmt;
    const uint32_t tb = I->tile_base;
    uint32_t *count = qs->count;
    const size_t cset = (size_t)set * qs->ntiles + tb;
    const uint32_t cshift = qs->cshift;
    const QueueTile *qtab = qs->tile + tb;
    QSyn *q_out = I->queue + (size_t)set * I->qslots;
    const bool pull_on = I->crec != nullptr;
    for (uint32_t t0 = 0; t0 < T; t0 += kBinMaxTiles) {
        const uint32_t tw = min(T - t0, (uint32_t)kBinMaxTiles);
        for (uint32_t p0 = lo; p0 < hi; p0 += kWaves * kBinDeep) {
            __syncthreads();   // s_list is written, hist is zero
            constexpr uint32_t N = kBinDeep * kBinItems;
            uint32_t cv[N], rank[N];
            unsigned long long wv[N];
            bool ok[N];
            unsigned long long pe[kBinDeep];
#pragma unroll
            for (uint32_t q = 0; q < kBinDeep; ++q) {
                const uint32_t p = p0 + q * kWaves + w;
                if (p < hi) {
                    // the list holding pass p: the last one with at most p passes before it
                    uint32_t l = 0;
#pragma unroll
                    for (uint32_t st = kFiredLists / 2; st > 0; st >>= 1)
                        if (s_list[l + st] <= p)
                            l += st;
                    pe[q] = gp(I->passes)[(size_t)l * I->passcap + (p - s_list[l])];
                }
            }
#pragma unroll
            for (uint32_t q = 0; q < kBinDeep; ++q) {
                const bool any = p0 + q * kWaves + w < hi;
                const uint64_t first = any ? pe[q] >> 8 : 0ull;
                const uint32_t n = any ? (uint32_t)(pe[q] & 0xffull) + 1u : 0u;
#pragma unroll
                for (uint32_t v = 0; v < kBinItems; ++v) {
                    const uint32_t u = q * kBinItems + v, j = v * kWave + lane;
                    ok[u] = j < n;
                    if (ok[u]) {
                        cv[u] = gp(I->col)[first + j];
                        wv[u] = w_raw(I->w, (size_t)(first + j), wfmt);
                    }
                }
            }
#pragma unroll
            for (uint32_t u = 0; u < N; ++u)
                if (ok[u]) {
                    const uint32_t t = ((cv[u] & kColMask) >> kTileBits) - t0;
                    ok[u] = t < tw;
                    if (ok[u]) {
                        rank[u] = atomicAdd(&hist[t], 1u);
                        if (rank[u] == 0u)
                            s_touch[atomicAdd(&s_ntouch, 1u)] = (uint16_t)t;
                    }
                }
            __syncthreads();
            const uint32_t nt = s_ntouch;
            uint32_t over = 0;   // synapses of this thread's tiles past their queue's capacity
            for (uint32_t k = tid; k < nt; k += kBinBlock) {
                const uint32_t t = s_touch[k];
                const uint32_t c = hist[t];
                const uint32_t b = gadd(&count[count_slot(cset + t0 + t, cshift)], c);
                const uint32_t cap = gp(qtab)[t0 + t].cap;
                const uint64_t off = gp(qtab)[t0 + t].off;
                const uint32_t room = cap > b ? min(c, cap - b) : 0u;
                over += c - room;
                // the segment's first slot; bit 31: it does not fit whole
                // (or the slot takes more than 31 bits), then its start
                // within the tile's queue
                hist[t] = room == c && off + b + c < 0x80000000ull ? (uint32_t)(off + b)
                                                                  : 0x80000000u | min(b, 0x7fffffffu);
            }
            if (over != 0u)
                gadd(&qs->ctl->slot[blockIdx.x & (kCtlSlots - 1u)].spilled, (unsigned long long)over);
            __syncthreads();
#pragma unroll
            for (uint32_t u = 0; u < N; ++u) {
                if (!ok[u])
                    continue;
                const uint32_t tile = (cv[u] & kColMask) >> kTileBits;
                const uint32_t h = hist[tile - t0];
                const uint32_t key = (cv[u] & 0xffu) | ((cv[u] & kKindBit) ? kQSynKind : 0u);
                const float2 wp = w_decode(wv[u], wfmt);
                if (!(h & 0x80000000u)) {
                    st_entry(q_out, h + rank[u], key, wp.x, wp.y);
                } else {
                    const uint64_t at = (uint64_t)(h & 0x7fffffffu) + rank[u];
                    if (at < gp(qtab)[tile].cap) {
                        st_entry(q_out, gp(qtab)[tile].off + at, key, wp.x, wp.y);
                    } else if (!pull_on) {
                        // past the capacity: the target's spill accumulator
                        // (Q23.40 integers like the LDS sums); with the pull
                        // the tile takes every row through its in-edges
                        unsigned long long *a = I->spill + ((size_t)set * I->n + (cv[u] & kColMask)) * 4u +
                                                ((cv[u] & kKindBit) ? 2u : 0u);
                        gadd(a, f32_to_q40(wp.x));
                        gadd(a + 1, f32_to_q40(wp.y));
                    }
                }
            }
            __syncthreads();
            for (uint32_t k = tid; k < nt; k += kBinBlock)
                hist[s_touch[k]] = 0u;
            if (tid == 0)
                s_ntouch = 0u;
        }
    }
}

// Gather propagation (instances with InstDev::segidx; their k_step reads
// the delta from dlt): the delta of the rows fired by the last launch (the
// fired lists of set `par`) for one group of consecutive neurons (GroupDesc),
// written into dlt.  A wave takes 64 fired rows at a time: lane l reads row l's segment bounds for the group
// from the row's group offsets, a wave prefix sum lays the segments end to
// end, and the wave then reads them with consecutive lanes on consecutive
// synapses (a segment is contiguous in the row), adding each weight pair
// into the group's Q23.40 LDS sums (64-bit integer atomics, so the result
// does not depend on the order); each lane has kGatherItems synapses in
// flight.  Segments of about 20 synapses (in-degree 5000, 2048 neurons of
// 500k, 1024 of 200k) coalesce the reads; one 1024-thread workgroup per group,
// and smaller groups where those of 2048 leave CUs idle.  Also empties the fired lists
// of set par ^ 1 (the ones the k_step launch after this one fills; their
// last reader was the previous k_gather).  Consecutive groups go to one XCD (workgroups
// are dealt to the 8 XCDs round-robin by index), so the segments of
// neighbouring groups, which share cache lines, meet in one L2.
template <uint32_t kFmt>
__global__ __launch_bounds__(kGatherBlock) __attribute__((amdgpu_waves_per_eu(8))) void k_gather(const GroupDesc *__restrict__ groups,
                                                         const InstDev *__restrict__ insts, uint32_t par)
{
    constexpr uint32_t kWaves = kGatherBlock / kWave;
    constexpr uint32_t kNeurons = 1u << kGroupBits;
    __shared__ unsigned long long acc[kNeurons * 4];
    __shared__ uint32_t s_off[kWaves][kWave];             // per wave: first item of each row's segment
    __shared__ unsigned long long s_base[kWaves][kWave];  // and the segment's first synapse
    __shared__ uint32_t s_list[kWaves][kWave];            // per wave: first row of each fired list
    const uint32_t nb = gridDim.x, x = blockIdx.x & 7u, slot = blockIdx.x >> 3;
    const GroupDesc d = groups[x * (nb >> 3) + min(x, nb & 7u) + slot];
    const InstDev &I = insts[d.inst];
    const uint32_t nn = 1u << d.bits;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = __lane_id();
    const uint32_t wv = tid / kWave;
    for (uint32_t i = tid; i < nn; i += kGatherBlock)
#pragma unroll
        for (uint32_t c = 0; c < 4u; ++c)
            acc[acc_at(i, c, kNeurons)] = 0ull;
    // the fired lists of set par laid end to end: lane l holds list l's count
    const uint32_t lcnt = gp(I.fcount)[((size_t)par * kFiredLists + lane) * kFiredCountStride];
    uint32_t lincl = lcnt;
#pragma unroll
    for (uint32_t o = 1; o < (uint32_t)kWave; o <<= 1) {
        const uint32_t v = __shfl_up(lincl, o, kWave);
        if (lane >= o)
            lincl += v;
    }
    const uint32_t nf = (uint32_t)__builtin_amdgcn_readlane((int)lincl, kWave - 1);
    s_list[wv][lane] = lincl - lcnt;
    if (d.g == 0 && tid < kFiredLists)
        gp(I.fcount)[((size_t)(par ^ 1u) * kFiredLists + tid) * kFiredCountStride] = 0u;
    __syncthreads();
    const auto fired = gp(I.fired) + (size_t)par * kFiredLists * I.fcap;
    const uint32_t wfmt = kFmt != kWeightAny ? kFmt : I.wfmt;
    const uint32_t stride = I.ngroups + 1u;
    const uint32_t first = d.g << d.bits;
    for (uint32_t c0 = wv * kWave; c0 < nf; c0 += kGatherBlock) {
        const uint32_t k = c0 + lane;
        const bool valid = k < nf;
        const uint32_t kc = valid ? k : nf - 1u;
        // the list holding row kc: the last list starting at or before it
        uint32_t ls = 0;
#pragma unroll
        for (uint32_t st = kWave / 2; st > 0; st >>= 1)
            if (s_list[wv][ls + st] <= kc)
                ls += st;
        const uint32_t r = fired[(size_t)ls * I.fcap + (kc - s_list[wv][ls])];
        const auto sg = gp(I.segidx) + (size_t)r * stride + d.g;
        const uint32_t a = sg[0];
        const uint32_t e = sg[1];
        const int64_t rb = gp(I.rowptr)[r];
        const uint32_t len = (valid && e > a) ? e - a : 0u;
        uint32_t incl = len;
#pragma unroll
        for (uint32_t o = 1; o < (uint32_t)kWave; o <<= 1) {
            const uint32_t v = __shfl_up(incl, o, kWave);
            if (lane >= o)
                incl += v;
        }
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        s_off[wv][lane] = incl - len;
        s_base[wv][lane] = (unsigned long long)(rb + (int64_t)a);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (uint32_t it = 0; it < total; it += kGatherItems * kWave) {
            uint32_t cv[kGatherItems];
            size_t jw[kGatherItems];
            unsigned long long wb[kGatherItems];
            bool ok[kGatherItems];
#pragma unroll
            for (uint32_t u = 0; u < kGatherItems; ++u) {
                const uint32_t item = it + u * kWave + lane;
                ok[u] = item < total;
                const uint32_t ic = ok[u] ? item : total - 1u;
                // the row whose segment holds item: the last lane whose
                // segment starts at or before it (empty segments before a
                // non-empty one start at the same item and lose to it)
                uint32_t lo = 0;
#pragma unroll
                for (uint32_t st = kWave / 2; st > 0; st >>= 1)
                    if (s_off[wv][lo + st] <= ic)
                        lo += st;
                jw[u] = (size_t)s_base[wv][lo] + (ic - s_off[wv][lo]);
            }
            // one record per synapse: column and weight pair side by side
            // (3 or 2 words at a word stride of grec_words(wfmt))
            const auto rec = gp(I.grec);
            if (wfmt == kWeightF32) {
#pragma unroll
                for (uint32_t u = 0; u < kGatherItems; ++u) {
                    const auto r = rec + jw[u] * 3u;
                    cv[u] = r[0];
                    wb[u] = (unsigned long long)r[1] | ((unsigned long long)r[2] << 32);
                }
            } else {
#pragma unroll
                for (uint32_t u = 0; u < kGatherItems; ++u) {
                    const auto r = rec + jw[u] * 2u;
                    cv[u] = r[0];
                    wb[u] = r[1];
                }
            }
#pragma unroll
            for (uint32_t u = 0; u < kGatherItems; ++u) {
                if (ok[u]) {
                    const float2 wp = w_decode(wb[u], wfmt);
                    const uint32_t row = (cv[u] & kColMask) - first, c0 = (cv[u] & kKindBit) ? 2u : 0u;
                    atomicAdd(&acc[acc_at(row, c0, kNeurons)], f32_to_q40(wp.x));
                    atomicAdd(&acc[acc_at(row, c0 + 1u, kNeurons)], f32_to_q40(wp.y));
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __syncthreads();
    for (uint32_t i = tid; i < d.count; i += kGatherBlock)
        st4(I.dlt, first + i, acc_to_delta(acc, i, kNeurons));
}

// Gather records: synapse j's column and weight-pair bits side by side.
__global__ __launch_bounds__(kBlock) void k_build_grec(const uint32_t *__restrict__ col, const void *__restrict__ w,
                                                       uint32_t wfmt, uint64_t nsyn, uint32_t *__restrict__ rec)
{
    const uint32_t nw = grec_words(wfmt);
    for (uint64_t j = (uint64_t)blockIdx.x * kBlock + threadIdx.x; j < nsyn; j += (uint64_t)gridDim.x * kBlock) {
        const unsigned long long b = w_raw(w, j, wfmt);
        uint32_t *r = rec + j * nw;
        r[0] = col[j];
        r[1] = (uint32_t)b;
        if (nw == 3u)
            r[2] = (uint32_t)(b >> 32);
    }
}

// Offsets per target group of 2^shift neurons (gather groups, or tiles for
// the direct propagation), one wave per row: segidx[r][g] = offset in row r
// of the first synapse whose target lies in group g or a later one, segidx[r][ngroups] = row length.  Rows must be ordered by
// target group (checked on the host).
__global__ __launch_bounds__(kBlock) void k_build_segidx(const int64_t *__restrict__ rowptr,
                                                         const uint32_t *__restrict__ col, uint32_t n,
                                                         uint32_t ngroups, uint32_t shift,
                                                         uint16_t *__restrict__ segidx)
{
    const uint32_t r = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    const uint32_t lane = __lane_id();
    if (r >= n)
        return;
    const int64_t rb = rowptr[r];
    const uint32_t len = (uint32_t)(rowptr[r + 1] - rb);
    uint16_t *s = segidx + (size_t)r * (ngroups + 1u);
    for (uint32_t j = lane; j < len; j += kWave) {
        const uint32_t gc = (col[rb + j] & kColMask) >> shift;
        const uint32_t g0 = j == 0 ? 0u : ((col[rb + j - 1] & kColMask) >> shift) + 1u;
        for (uint32_t g = g0; g <= gc; ++g)
            s[g] = (uint16_t)j;
    }
    const uint32_t tail = len == 0 ? 0u : ((col[rb + len - 1] & kColMask) >> shift) + 1u;
    for (uint32_t g = tail + lane; g <= ngroups; g += kWave)
        s[g] = (uint16_t)len;
}

// In-edges of the pull propagation: every synapse of source row r goes to
// its target tile t's range of records (from cptr[t]) as (key = source row |
// target in tile | channel bit, weight pair bits).  A workgroup takes
// kBuildRows consecutive rows: it counts their synapses per target tile in
// LDS, reserves each tile's share with one atomic on the tile's cursor
// (cursor[t]: records placed so far, from 0), then reads the rows again and
// places every record at its tile's reserved range, ranked by an LDS
// atomic.  One device atomic per (workgroup, target tile) instead of one
// per synapse: on the 2M-neuron voxel block a voxel's rows share their
// target tiles, and per-synapse atomics on the same cursors serialised.
// The order within a tile follows the atomics; the pull's sums are exact
// integers, so it does not matter.  Instances of more than kBuildMaxTiles
// tiles are built in windows of that many target tiles (the rows are read
// again for each window).
constexpr uint32_t kBuildBlock = 1024, kBuildRows = 256, kBuildMaxTiles = 16384;
__global__ __launch_bounds__(kBuildBlock) void k_build_pull(const int64_t *__restrict__ rowptr,
                                                            const uint32_t *__restrict__ col,
                                                            const void *__restrict__ w, uint32_t wfmt, uint32_t n,
                                                            uint32_t ntiles, const int64_t *__restrict__ cptr,
                                                            uint32_t *__restrict__ cursor, uint32_t *__restrict__ rec)
{
    extern __shared__ uint32_t hist[];   // min(ntiles, kBuildMaxTiles) words
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = __lane_id();
    const uint32_t wv = tid / kWave;
    constexpr uint32_t kWaves = kBuildBlock / kWave;
    const uint32_t r0 = blockIdx.x * kBuildRows;
    const uint32_t r1 = min(n, r0 + kBuildRows);
    const uint32_t nw = grec_words(wfmt);
    for (uint32_t t0 = 0; t0 < ntiles; t0 += kBuildMaxTiles) {
        const uint32_t tw = min(kBuildMaxTiles, ntiles - t0);
        for (uint32_t t = tid; t < tw; t += kBuildBlock)
            hist[t] = 0u;
        __syncthreads();
        for (uint32_t r = r0 + wv; r < r1; r += kWaves) {
            const int64_t rb = rowptr[r];
            const uint32_t len = (uint32_t)(rowptr[r + 1] - rb);
            for (uint32_t j = lane; j < len; j += kWave) {
                const uint32_t t = ((col[rb + j] & kColMask) >> kTileBits) - t0;
                if (t < tw)
                    atomicAdd(&hist[t], 1u);
            }
        }
        __syncthreads();
        for (uint32_t t = tid; t < tw; t += kBuildBlock) {
            const uint32_t h = hist[t];
            if (h != 0u)
                hist[t] = atomicAdd(&cursor[t0 + t], h);
        }
        __syncthreads();
        for (uint32_t r = r0 + wv; r < r1; r += kWaves) {
            const int64_t rb = rowptr[r];
            const uint32_t len = (uint32_t)(rowptr[r + 1] - rb);
            for (uint32_t j = lane; j < len; j += kWave) {
                const uint32_t c = col[rb + j];
                const uint32_t t = ((c & kColMask) >> kTileBits) - t0;
                if (t >= tw)
                    continue;
                const uint32_t off = atomicAdd(&hist[t], 1u);
                const unsigned long long b = w_raw(w, (size_t)(rb + j), wfmt);
                uint32_t *e = rec + ((size_t)cptr[t0 + t] + off) * nw;
                e[0] = r | ((c & (kBlock - 1u)) << kPullRowBits) | (c & kKindBit);
                e[1] = (uint32_t)b;
                if (nw == 3u)
                    e[2] = (uint32_t)(b >> 32);
            }
        }
        __syncthreads();   // the window's last ranks are taken before the next window zeroes the counts
    }
}

// Writes the pending delta (the runs queued in queue set `set` for the next
// k_step) of every neuron of every tile without consuming the queues: used
// before sampling I_syn and before reading the state back.
__global__ __launch_bounds__(kBlock) void k_materialize(const TileDesc *__restrict__ tiles,
                                                        const InstDev *__restrict__ insts,
                                                        QueueSet qs,
                                                        uint32_t set)
{
    __shared__ unsigned long long acc[kBlock * 4];
    __shared__ DirectList ls;
    const TileDesc &d = tiles[blockIdx.x];
    const InstDev &I = insts[d.inst_idx];
    if (I.segidx != nullptr)
        return;   // gather propagation: k_gather has written dlt
    const uint32_t tid = threadIdx.x;
    clear_row(acc, tid);
    if (I.tidx != nullptr) {
        if (tid == 0)
            ls.n = 0u;
        __syncthreads();
        const DirectIds ids(I.bits + (size_t)set * I.ntiles * kBitWords, I.ntiles, tid);
        direct_tile<kWeightAny>(acc, ls, I, ids, set, d.begin >> kTileBits, tid);
        __syncthreads();
        if (tid < d.count)
            st4(I.dlt, d.begin + tid, acc_to_delta(acc, tid));
        return;
    }
    const uint32_t cnt_raw = qs.count[count_slot((size_t)set * qs.ntiles + blockIdx.x, qs.cshift)];
    const bool over = cnt_raw > d.qcap;
    const bool pull_on = I.crec != nullptr;
    const bool pull = pull_on && (over || gp(I.step)[2u + set] == gp(I.step)[set] + 1);
    const uint32_t cnt = (pull_on && over) ? 0u : min(cnt_raw, d.qcap);
    __syncthreads();
    accumulate_tile(acc, d.queue + (size_t)set * d.qslots, cnt, QSyn{}, 0u, tid);
    if (pull)
        pull_tile<kWeightAny>(acc, I, set, d.begin >> kTileBits, over, tid);
    __syncthreads();
    if (tid < d.count) {
        if (!pull_on && over)
            take_spill(acc, I.spill, I.n, set, d.begin + tid, tid, false);
        st4(I.dlt, d.begin + tid, acc_to_delta(acc, tid));
    }
}

// Folds the pending delta of queue set `set` into J now (J = J * decay +
// delta, with the decay of the step that produced it), marks J as folded and
// empties the queues.  Runs before any change of parameters or of the
// instance set, so no pending spike is lost or folded with a later decay.
__global__ __launch_bounds__(kBlock) void k_settle(const TileDesc *__restrict__ tiles,
                                                   const InstDev *__restrict__ insts,
                                                   QueueSet qs,
                                                   uint32_t set)
{
    __shared__ unsigned long long acc[kBlock * 4];
    __shared__ DirectList ls;
    const TileDesc &d = tiles[blockIdx.x];
    const InstDev &I = insts[d.inst_idx];
    const uint32_t tid = threadIdx.x;
    if (I.segidx != nullptr) {
        // gather propagation: k_gather has written the pending delta into
        // dlt; after the fold the fired list of this set is empty
        if (tid < d.count) {
            const uint32_t li = d.begin + tid;
            const auto flag = st_at<kStFlag, uint8_t>(d.state, tid);
            const uint32_t fl = *flag;
            if (!(fl & kFlagFolded)) {
                st_J(d.state, tid, fold_delta(ld_J(d.state, tid), ld4(&param_of(I, li)->d, 0), ld4(I.dlt, li)));
                *flag = (uint8_t)(fl | kFlagFolded);
            }
        }
        if (d.begin == 0 && tid < kFiredLists)
            gp(I.fcount)[((size_t)set * kFiredLists + tid) * kFiredCountStride] = 0u;
        return;
    }
    const bool direct = I.tidx != nullptr;
    uint32_t *cnt_p = qs.count + count_slot((size_t)set * qs.ntiles + blockIdx.x, qs.cshift);
    clear_row(acc, tid);
    if (direct) {
        if (tid == 0)
            ls.n = 0u;
        __syncthreads();
        const DirectIds ids(I.bits + (size_t)set * I.ntiles * kBitWords, I.ntiles, tid);
        direct_tile<kWeightAny>(acc, ls, I, ids, set, d.begin >> kTileBits, tid);
    }
    const uint32_t cnt_raw = direct ? 0u : *cnt_p;
    const bool over = cnt_raw > d.qcap;
    const bool pull_on = !direct && I.crec != nullptr;
    const bool pull = pull_on && (over || gp(I.step)[2u + set] == gp(I.step)[set] + 1);
    const uint32_t cnt = (pull_on && over) ? 0u : min(cnt_raw, d.qcap);
    __syncthreads();
    accumulate_tile(acc, d.queue + (size_t)set * d.qslots, cnt, QSyn{}, 0u, tid);
    if (pull)
        pull_tile<kWeightAny>(acc, I, set, d.begin >> kTileBits, over, tid);
    __syncthreads();
    if (tid < d.count) {
        const uint32_t li = d.begin + tid;
        if (!pull_on && over)
            take_spill(acc, I.spill, I.n, set, li, tid, true);
        const auto flag = st_at<kStFlag, uint8_t>(d.state, tid);
        const uint32_t fl = *flag;
        if (!(fl & kFlagFolded)) {
            st_J(d.state, tid, fold_delta(ld_J(d.state, tid), ld4(&param_of(I, li)->d, 0), acc_to_delta(acc, tid)));
            *flag = (uint8_t)(fl | kFlagFolded);
        }
    }
    if (tid == 0 && !direct)
        *cnt_p = 0u;
}

// I_syn-based statistics (imean, receptor imeans) of the last step run: the
// k_step launch of the next step would record them, so after the last step
// they are taken here from the materialised pending delta.  `par` is the
// parity of the next launch (its step slot holds the next step index).
__global__ __launch_bounds__(kBlock) void k_stat_tail(const TileDesc *__restrict__ tiles,
                                                      const InstDev *__restrict__ insts,
                                                      uint32_t par)
{
    __shared__ unsigned long long s_stat[kStatFields];
    const TileDesc &d = tiles[blockIdx.x];
    const InstDev &I = insts[d.inst_idx];
    const uint32_t cf = current_fields(I.stat_mask);
    if (I.rec_stat == nullptr || cf == 0u)
        return;
    const int64_t row = gp(I.step)[par] - 1 - I.rec_step0;
    if (row < 0 || row >= (int64_t)I.rec_len)
        return;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = __lane_id();
    const uint32_t li = d.begin + tid;
    const bool active = tid < d.count;
    long long stv[kStatFields];
    uint32_t p = d.pop0;
    bool valid = false;
    if (active) {
        while (p + 1 < I.npop && li >= I.pops[p].end)
            ++p;
        const ParamRec *c = param_of(I, li);
        const float V = *st_at<kStV, float>(d.state, tid);
        float4 J = ld_J(d.state, tid);
        if (!(*st_at<kStFlag, uint8_t>(d.state, tid) & kFlagFolded))
            J = fold_delta(J, ld4(&c->d, 0), ld4(I.dlt, li));
        const float4 g = ld4(&c->g, 0), vu = ld4(&c->v, 0);
        const float4 rc = receptor_currents(g, vu, J, V);
        stv[1] = stat_q(syn_current(g, vu, J, V));
        stv[2] = stat_q(rc.x);
        stv[3] = stat_q(rc.y);
        stv[4] = stat_q(rc.z);
        stv[5] = stat_q(rc.w);
        valid = !gp(I.blocked)[li];
    }
    if (!(d.flags & kTileOnePop)) {
        wave_pop_stats(rec_stat_row(I, row, d.begin), valid, p, stv, cf, lane);
        return;
    }
    if (tid < (uint32_t)kStatFields)
        s_stat[tid] = 0ull;
    __syncthreads();
    wave_tile_stats(s_stat, valid, stv, cf, lane);
    __syncthreads();
    if (tid < (uint32_t)kStatFields && ((cf >> tid) & 1u))
        atomicAdd(reinterpret_cast<unsigned long long *>(rec_stat_row(I, row, d.begin)) +
                      (size_t)d.pop0 * kStatFields + tid,
                  s_stat[tid]);
}

// Rows [row0, row0 + rows) of a record with each row's slots added up
// (integers, so the order does not matter), statistics first.  The outputs
// are the call's pinned host memory, so a small record costs one launch and
// no copy: two folds and two copies were 45 us of a 240 us call.
__global__ __launch_bounds__(kBlock) void k_fetch_rows(RecordRows r, uint64_t row0, uint64_t rows)
{
    const uint64_t ns = rows * r.swidth, nc = rows * r.cwidth;
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < ns + nc; i += (uint64_t)gridDim.x * kBlock) {
        if (i < ns) {
            const uint64_t row = i / r.swidth;
            const long long *p = r.stat + (row0 + row) * r.slots * r.sstride + (i - row * r.swidth);
            long long s = 0;
            for (uint32_t k = 0; k < r.slots; ++k)
                s += p[(size_t)k * r.sstride];
            r.out_stat[i] = s;
        } else {
            const uint64_t c = i - ns, row = c / r.cwidth;
            const uint32_t *p = r.counts + (row0 + row) * r.slots * r.cstride + (c - row * r.cwidth);
            uint32_t s = 0;
            for (uint32_t k = 0; k < r.slots; ++k)
                s += p[(size_t)k * r.cstride];
            r.out_counts[c] = s;
        }
    }
}

// Several small copies and fills in one launch: the tables of a run (up to
// nine) from pinned host memory, and the words a call clears.  One hipMemcpy
// or hipMemset each cost 3-20 us of host time, most of a short call's.
struct CopyList {
    CopyWords seg[kCopySegs];
    int n;
};

__global__ __launch_bounds__(kBlock) void k_copy_words(CopyList l)
{
    for (int k = 0; k < l.n; ++k) {
        uint32_t *dst = static_cast<uint32_t *>(l.seg[k].dst);
        const uint32_t *src = static_cast<const uint32_t *>(l.seg[k].src);
        for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < l.seg[k].words;
             i += (uint64_t)gridDim.x * kBlock)
            dst[i] = src != nullptr ? src[i] : 0u;
    }
}

// stat_result.cpp:393-433 (sampled spike flag, V, I_syn, i_ou) of the step
// just run by the k_step launch of parity `par`.  Runs after k_materialize
// (dlt holds that step's delta, folded in exactly as the next k_step will
// fold it).
__global__ __launch_bounds__(kBlock) void k_sample(const InstDev *__restrict__ insts,
                                                   const SampleDev *__restrict__ samples,
                                                   uint32_t nsamples,
                                                   const SampleRecDev *__restrict__ recs,
                                                   uint32_t par)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= nsamples)
        return;
    const SampleDev s = samples[i];
    const InstDev &I = insts[s.inst];
    const SampleRecDev R = recs[s.inst];
    const int64_t row = gp(I.step)[par] - I.rec_step0;
    if (row < 0 || row >= (int64_t)I.rec_len)
        return;
    const uint32_t li = s.neuron;
    const size_t o = (size_t)row * R.nsample + s.slot;
    unsigned char *block = block_of(I, li);
    const uint32_t k = li & (kBlock - 1u);
    const float V = *st_at<kStV, float>(block, k);
    if (R.spike)
        R.spike[o] = (*st_at<kStFlag, uint8_t>(block, k) & kFlagEmit) ? 1 : 0;
    if (R.v)
        R.v[o] = V;
    if (R.isyn) {
        const ParamRec *c = param_of(I, li);
        const float4 J = fold_delta(ld_J(block, k), ld4(&c->d, 0), ld4(I.dlt, li));   // flag bit 2 is clear here
        R.isyn[o] = syn_current(ld4(&c->g, 0), ld4(&c->v, 0), J, V);
    }
    if (R.iou)
        R.iou[o] = *st_at<kStIou, float>(block, k);
}

// Fresh state (block.cpp:136-179, membrane_voltage.cpp:18): V0 = (V_th +
// V_reset) / 2; the rest of the blocks is zeroed before.
__global__ __launch_bounds__(kBlock) void k_init_state(StateView v)
{
    const uint32_t li = blockIdx.x * kBlock + threadIdx.x;
    if (li >= v.n)
        return;
    const float4 a = ld4(&v.prm[(li & v.pmask) + (uint32_t)gp(v.cls)[li]].a, 0);
    *st_at<kStV, float>(v.state + (size_t)blockIdx.x * kStateBytes, threadIdx.x) = (a.y + a.x) / 2.0f;
}

// OU current of neurons [begin, end) set to `value`.
__global__ __launch_bounds__(kBlock) void k_fill_iou(StateView v, uint32_t begin, uint32_t end, float value)
{
    const uint32_t li = begin + blockIdx.x * kBlock + threadIdx.x;
    if (li < end)
        *st_at<kStIou, float>(v.state + (size_t)(li >> kTileBits) * kStateBytes, li & (kBlock - 1u)) = value;
}

// Reference-visible state of `count` neurons from `first` on into plain
// arrays (any may be null): the pending delta folded exactly as the next
// step will fold it, I_syn of the folded J.
__global__ __launch_bounds__(kBlock) void k_read_state(StateView v, uint32_t first, uint32_t count, StateArrays out)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= count)
        return;
    const uint32_t li = first + i, k = li & (kBlock - 1u);
    unsigned char *block = v.state + (size_t)(li >> kTileBits) * kStateBytes;
    const float V = *st_at<kStV, float>(block, k);
    const uint32_t fl = *st_at<kStFlag, uint8_t>(block, k);
    if (out.V)
        out.V[i] = V;
    if (out.t)
        out.t[i] = *st_at<kStT, int32_t>(block, k);
    if (out.iou)
        out.iou[i] = *st_at<kStIou, float>(block, k);
    if (out.f)
        out.f[i] = fl & kFlagSpike;
    if (out.emitted)
        out.emitted[i] = (fl & kFlagEmit) ? 1 : 0;
    if (out.J || out.isyn) {
        const ParamRec *c = v.prm + ((li & v.pmask) + (uint32_t)gp(v.cls)[li]);
        float4 J = ld_J(block, k);
        if (!(fl & kFlagFolded))
            J = fold_delta(J, ld4(&c->d, 0), ld4(v.dlt, li));
        if (out.J)
            st4(out.J, i, J);
        if (out.isyn)
            out.isyn[i] = syn_current(ld4(&c->g, 0), ld4(&c->v, 0), J, V);
    }
}

// Checkpoint restore of `count` neurons from `first` on (null arrays keep
// their field).  J is the reference-visible J of the last step: the pending
// delta is cleared and the flag byte marks J as folded, so the next step
// uses it as is.
__global__ __launch_bounds__(kBlock) void k_write_state(StateView v, uint32_t first, uint32_t count, StateArrays in)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= count)
        return;
    const uint32_t li = first + i, k = li & (kBlock - 1u);
    unsigned char *block = v.state + (size_t)(li >> kTileBits) * kStateBytes;
    if (in.V)
        *st_at<kStV, float>(block, k) = in.V[i];
    if (in.t)
        *st_at<kStT, int32_t>(block, k) = in.t[i];
    if (in.iou)
        *st_at<kStIou, float>(block, k) = in.iou[i];
    if (in.f || in.J) {
        uint32_t fl = *st_at<kStFlag, uint8_t>(block, k);
        if (in.f)
            fl = (fl & ~(uint32_t)kFlagSpike) | (in.f[i] ? kFlagSpike : 0u);
        if (in.J)
            fl |= kFlagFolded;
        *st_at<kStFlag, uint8_t>(block, k) = (uint8_t)fl;
    }
    if (in.J) {
        st_J(block, k, ld4(in.J, i));
        st4(v.dlt, li, make_float4(0.0f, 0.0f, 0.0f, 0.0f));
    }
}

// Verification entry: normals of the OU stream for a range of neurons at one
// substep (checks CPU/GPU bit identity of the generator).
__global__ __launch_bounds__(kBlock) void k_normals(uint64_t seed, uint32_t neuron0, uint64_t substep,
                                                    uint32_t count, float *__restrict__ out)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < count)
        out[i] = ou_normal(seed, neuron0 + i, substep);
}

// ---- launchers ----------------------------------------------------------

namespace {
// Calls f with the weight format as a constant (a format of every launched
// instance, or kWeightAny).
template <typename F>
hipError_t with_format(uint32_t wfmt, F f)
{
    switch (wfmt) {
    case kWeightF32: f(std::integral_constant<uint32_t, kWeightF32>{}); break;
    case kWeightF16: f(std::integral_constant<uint32_t, kWeightF16>{}); break;
    case kWeightU8: f(std::integral_constant<uint32_t, kWeightU8>{}); break;
    case kWeightAny: f(std::integral_constant<uint32_t, kWeightAny>{}); break;
    default: return hipErrorInvalidValue;
    }
    return hipSuccess;
}
}  // namespace

namespace {
typedef void (*StepKernel)(const TileDesc *, const QueueSet *, uint32_t);

template <uint32_t kF, bool kStat>
StepKernel step_kernel(StepMode mode, uint32_t pass_k)
{
    if (mode == StepMode::direct)
        return k_step<kF, kStat, kDirect, 1>;
    if (mode == StepMode::bin_launch)
        return k_step<kF, kStat, kQueues, 1>;
    return pass_k == 1 ? k_step<kF, kStat, kTileBin, 1>
           : pass_k == 4 ? k_step<kF, kStat, kTileBin, 4>
                         : k_step<kF, kStat, kTileBin, 2>;
}
}  // namespace

hipError_t launch_step_kernel(const TileDesc *tiles, uint32_t ntiles, StepMode mode, uint32_t pass_k,
                              const QueueSet *qs, uint32_t par, uint32_t wfmt, bool stat, hipEvent_t start,
                              hipEvent_t stop, hipStream_t stream)
{
    if (ntiles == 0)
        return hipSuccess;
    const hipError_t e = with_format(wfmt, [&](auto fmt) {
        constexpr uint32_t kF = decltype(fmt)::value;
        const StepKernel kern = stat ? step_kernel<kF, true>(mode, pass_k) : step_kernel<kF, false>(mode, pass_k);
        if (start != nullptr)
            hipExtLaunchKernelGGL(kern, dim3(ntiles), dim3(kBlock), 0, stream, start, stop, 0, tiles, qs, par);
        else
            hipLaunchKernelGGL(kern, dim3(ntiles), dim3(kBlock), 0, stream, tiles, qs, par);
    });
    return e != hipSuccess ? e : hipGetLastError();
}

hipError_t launch_bin_kernel(const BinDesc *groups, uint32_t ngroups, uint32_t max_tiles, const QueueSet *qs,
                             uint32_t par, uint32_t wfmt, hipEvent_t start, hipEvent_t stop, hipStream_t stream)
{
    if (ngroups == 0)
        return hipSuccess;
    const uint32_t lds = std::min(max_tiles, kBinMaxTiles) * (uint32_t)sizeof(uint32_t);
    const hipError_t e = with_format(wfmt, [&](auto fmt) {
        auto kern = k_bin<decltype(fmt)::value>;
        if (start != nullptr)
            hipExtLaunchKernelGGL(kern, dim3(ngroups), dim3(kBinBlock), lds, stream, start, stop, 0, groups, qs, par);
        else
            hipLaunchKernelGGL(kern, dim3(ngroups), dim3(kBinBlock), lds, stream, groups, qs, par);
    });
    return e != hipSuccess ? e : hipGetLastError();
}

hipError_t launch_gather(const GroupDesc *groups, uint32_t ngroups, const InstDev *insts, uint32_t par, uint32_t wfmt,
                         hipEvent_t start, hipEvent_t stop, hipStream_t stream)
{
    if (ngroups == 0)
        return hipSuccess;
    const hipError_t e = with_format(wfmt, [&](auto fmt) {
        auto kern = k_gather<decltype(fmt)::value>;
        if (start != nullptr)
            hipExtLaunchKernelGGL(kern, dim3(ngroups), dim3(kGatherBlock), 0, stream, start, stop, 0, groups, insts, par);
        else
            hipLaunchKernelGGL(kern, dim3(ngroups), dim3(kGatherBlock), 0, stream, groups, insts, par);
    });
    return e != hipSuccess ? e : hipGetLastError();
}

hipError_t launch_build_grec(const uint32_t *col, const void *w, uint32_t wfmt, uint64_t nsyn, uint32_t *rec,
                             hipStream_t stream)
{
    if (nsyn == 0)
        return hipSuccess;
    const uint64_t nb = std::min<uint64_t>((nsyn + kBlock - 1) / kBlock, 65536);
    hipLaunchKernelGGL(k_build_grec, dim3((uint32_t)nb), dim3(kBlock), 0, stream, col, w, wfmt, nsyn, rec);
    return hipGetLastError();
}

hipError_t launch_build_segidx(const int64_t *rowptr, const uint32_t *col, uint32_t n, uint32_t ngroups,
                               uint32_t shift, uint16_t *segidx, hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    const uint32_t rows_per_block = kBlock / kWave;
    const uint32_t nb = (n + rows_per_block - 1) / rows_per_block;
    hipLaunchKernelGGL(k_build_segidx, dim3(nb), dim3(kBlock), 0, stream, rowptr, col, n, ngroups, shift, segidx);
    return hipGetLastError();
}

hipError_t launch_build_pull(const int64_t *rowptr, const uint32_t *col, const void *w, uint32_t wfmt, uint32_t n,
                             const int64_t *cptr, uint32_t *cursor, uint32_t *rec, hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    const uint32_t ntiles = (n + kBlock - 1) / kBlock;
    const uint32_t nb = (n + kBuildRows - 1) / kBuildRows;
    hipLaunchKernelGGL(k_build_pull, dim3(nb), dim3(kBuildBlock), min(ntiles, kBuildMaxTiles) * sizeof(uint32_t),
                       stream, rowptr, col, w, wfmt, n, ntiles, cptr, cursor, rec);
    return hipGetLastError();
}

hipError_t launch_materialize(const TileDesc *tiles, uint32_t ntiles, const InstDev *insts, const QueueSet &qs,
                              uint32_t set, hipStream_t stream)
{
    if (ntiles == 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_materialize, dim3(ntiles), dim3(kBlock), 0, stream, tiles, insts, qs, set);
    return hipGetLastError();
}

hipError_t launch_settle(const TileDesc *tiles, uint32_t ntiles, const InstDev *insts, const QueueSet &qs,
                         uint32_t set, hipStream_t stream)
{
    if (ntiles == 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_settle, dim3(ntiles), dim3(kBlock), 0, stream, tiles, insts, qs, set);
    return hipGetLastError();
}

hipError_t launch_stat_tail(const TileDesc *tiles, uint32_t ntiles, const InstDev *insts, uint32_t par,
                            hipStream_t stream)
{
    if (ntiles == 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_stat_tail, dim3(ntiles), dim3(kBlock), 0, stream, tiles, insts, par);
    return hipGetLastError();
}

hipError_t launch_fetch_rows(const RecordRows &r, uint64_t row0, uint64_t rows, hipStream_t stream)
{
    const uint64_t cells = rows * ((uint64_t)r.swidth + r.cwidth);
    if (cells == 0)
        return hipSuccess;
    const uint64_t nb = std::min<uint64_t>((cells + kBlock - 1) / kBlock, 4096);
    hipLaunchKernelGGL(k_fetch_rows, dim3((uint32_t)nb), dim3(kBlock), 0, stream, r, row0, rows);
    return hipGetLastError();
}

hipError_t launch_copy_words(const CopyWords *segs, int n, hipStream_t stream)
{
    while (n > 0) {
        CopyList l{};
        uint64_t most = 0;
        for (l.n = 0; l.n < kCopySegs && n > 0; --n, ++segs)
            if (segs->words > 0) {
                l.seg[l.n++] = *segs;
                most = std::max(most, segs->words);
            }
        if (l.n == 0)
            continue;
        const uint64_t nb = std::min<uint64_t>((most + kBlock - 1) / kBlock, 1024);
        hipLaunchKernelGGL(k_copy_words, dim3((uint32_t)nb), dim3(kBlock), 0, stream, l);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

hipError_t launch_sample(const InstDev *insts, const SampleDev *samples, uint32_t nsamples,
                         const SampleRecDev *recs, uint32_t par, hipStream_t stream)
{
    if (nsamples == 0)
        return hipSuccess;
    const uint32_t nb = (nsamples + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(k_sample, dim3(nb), dim3(kBlock), 0, stream, insts, samples, nsamples, recs, par);
    return hipGetLastError();
}

hipError_t launch_init_state(const StateView &v, hipStream_t stream)
{
    hipLaunchKernelGGL(k_init_state, dim3((v.n + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, v);
    return hipGetLastError();
}

hipError_t launch_fill_iou(const StateView &v, uint32_t begin, uint32_t end, float value, hipStream_t stream)
{
    if (begin >= end)
        return hipSuccess;
    hipLaunchKernelGGL(k_fill_iou, dim3((end - begin + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, v, begin, end,
                       value);
    return hipGetLastError();
}

hipError_t launch_read_state(const StateView &v, uint32_t first, uint32_t count, const StateArrays &out,
                             hipStream_t stream)
{
    hipLaunchKernelGGL(k_read_state, dim3((count + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, v, first, count,
                       out);
    return hipGetLastError();
}

hipError_t launch_write_state(const StateView &v, uint32_t first, uint32_t count, const StateArrays &in,
                              hipStream_t stream)
{
    hipLaunchKernelGGL(k_write_state, dim3((count + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, v, first, count,
                       in);
    return hipGetLastError();
}

hipError_t launch_normals(uint64_t seed, uint32_t neuron0, uint64_t substep, uint32_t count, float *out,
                          hipStream_t stream)
{
    if (count == 0)
        return hipSuccess;
    const uint32_t nb = (count + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(k_normals, dim3(nb), dim3(kBlock), 0, stream, seed, neuron0, substep, count, out);
    return hipGetLastError();
}

}  // namespace dtb
