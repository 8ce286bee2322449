// tpamd_internal.h -- declarations shared by the library's translation units:
// the opaque handle types of the C ABI, the error helper, the chunk record of
// batched launches, and the launch entry points each kernel family's unit
// defines (one unit per family, so they compile in parallel).
#pragma once

#include "tpamd_device.h"
#include "tpamd_adjoint.h"
#include "tpamd.h"

#include <hip/hip_runtime.h>

#include <string>

struct tpamd_field {
    tpamd::DevField d;
    void* dev_data;          // owned device buffer (grids)
    void* cells_data;        // owned cell-replicated copy (grids, optional)
    bool cells_off;          // the caller dropped the copy: no solve builds it again
    bool cells_auto;         // a solve built it and the caller has not asked for it: no batch uses it,
                             // and it may go between calls (relieve)
    double cells_owed;       // ns that solves since the last offer would have saved on a copy (offer_cells)
    tpamd_ctx* owner;        // the context whose calls use the field
    const tpamd_field* src;  // UxB: the B field it was built from
    size_t bytes;
    tpamd::MeshGrid mesh_host;      // Mesh: host copy of the descriptor (device pointers)
};

struct tpamd_ctx {
    int device;
    hipStream_t stream;
    hipEvent_t ev0, ev1, ev2;
    std::string err;
    // device buffer of the calls that stage or need workspace (ctx_buffer)
    void* d_buf;
    size_t d_buf_bytes;
    size_t keep_bytes;                      // what of it may stay between calls (ctx_trim)
    unsigned long long* d_steps;
    // pinned host memory of kPinSlots pieces, with one event per piece
    // (stage_in, stage_out), and behind them a word for a step count
    char* h_pin;
    hipEvent_t pin_ev[4];                   // kPinSlots
    // the device address of this device's copy of the allocation-free
    // entry point's scratch array (looked up at tpamd_init; null if that failed)
    unsigned char* scratch;
};

namespace tpamd {

// tpamd_sort.hip: radix sort of (key, record) pairs on key bits [begin, end)
template <typename R>
hipError_t adj_sort_records(void* d_temp, size_t& temp_bytes, const unsigned* keys_in,
                            unsigned* keys_out, const AdjRec<R>* vals_in, AdjRec<R>* vals_out,
                            long long n, int begin_bit, int end_bit, hipStream_t stream);

// tpamd_sort.hip: the bin sums over the reverse kernel's blocks of records
// (tot: nbins words of workspace)
template <typename R>
hipError_t adj_bins_seg(const unsigned* keys, const AdjRec<R>* vals, const unsigned* seg, unsigned* tot, int nblk,
                        unsigned nbins, unsigned ncell, double* G, hipStream_t stream);

// The context's device buffer, grown to `bytes` (contents are lost): for use
// within one call, which the caller serialises and which ends synchronised.
// A failure leaves no buffer and no error for the next launch to report.
hipError_t ctx_buffer(tpamd_ctx* ctx, size_t bytes, void** out);
// Releases it when it has grown past what is kept between calls: 1/16 of the
// device's memory, as a cell copy may take, or 4 GiB.
void ctx_trim(tpamd_ctx* ctx);

// Host arrays and the span of the context's device buffer that holds them: a
// part is the array `host` of `bytes` bytes at offset `off` of the span, parts
// in rising order.
struct HostPart {
    void* host;
    size_t off, bytes;
};
// A pageable copy waits for each of its pieces and costs 10-20 us of host
// time for even a few bytes; these go through the context's pinned memory
// instead, a span at a time.  Measured, microseconds (pageable -> staged):
//   out of 5 arrays of a small solve, 40 KB          75 -> 21 (both ways)
//   to the host   64 KB 34 -> 18   256 KB 113 -> 27   9 MB 549 -> 380   96 MB 5843 -> 3826
//   to the device 64 KB 33 -> 17   256 KB 108 -> 23   1 MB 60 -> 71     9 MB 333 -> 368
// so spans to the device above kStageIn are copied part by part as they lie.
// (Several threads emptying the pieces gained nothing on memory that is
// already mapped.)  stage_in only enqueues: the host arrays stay until the
// stream has been waited for.  stage_out returns with everything before it on
// the stream done.
constexpr int kPinSlots = 4;
constexpr size_t kPinPiece = (size_t)1 << 20;
constexpr size_t kPinBytes = kPinSlots * kPinPiece + 4096;
constexpr size_t kStageIn = (size_t)512 << 10;
hipError_t stage_in(tpamd_ctx* ctx, char* dev, size_t span, const HostPart* parts, int n, hipStream_t st);
hipError_t stage_out(tpamd_ctx* ctx, const char* dev, size_t span, const HostPart* parts, int n, hipStream_t st);

// records the message on ctx (or as the last tpamd_init error) and returns code
int fail(tpamd_ctx* ctx, int code, const char* fmt, ...);

// ---------------------------------------------------------------------------
// Batched ensembles: a persistent grid of waves pulls chunks of particles from
// an atomic queue.  A chunk never straddles a field instance, so the
// instance's parameter block is wave-uniform; within a chunk the 64 lanes
// stride over its particles (particles per thread = chunk size / 64), which
// evens out uneven lifetimes.  Every wave leaves once the queue is drained.
// ---------------------------------------------------------------------------
// The batched kernel's chunk list is cut into kQueues slices of neighbouring
// chunks, each with its own claim counter on its own 128-B line.  A wave
// starts on the slice of its block's XCD (blocks are dispatched to the 8 XCDs
// round-robin) and moves on to the others when it is drained, so all waves
// finish; one shared counter serialised ~8 claims per microsecond.
// Neighbouring chunks are mostly of one instance: a wave's next chunk seldom
// makes it wait, and few instances' cells are in use at a time.  Dealt one by
// one instead, or in 64 slices, 4 M particles of 24 instances took 1.38 and
// 1.15 ms against 1.28 (FP64) and 1.05 and 0.99 against 1.04 (FP32C), 16 M of
// 32 instances 2.53 and 2.74 against 2.49.
constexpr int kQueues = 8;
static_assert(64 % kQueues == 0, "a lane for each counter");
constexpr int kQueueStride = 32;   // unsigned words between counters (128 B)

struct Chunk {
    int inst;
    int pad;
    long long begin, end;
};

// one launch of a solve kernel: a thread per particle (batch == false, over
// *p) or the persistent chunk-queue kernel over a parameter table (with
// `occ` set, only the kernel's resident blocks per CU are reported)
struct LaunchReq {
    bool batch;
    int adaptive;
    dim3 g, b;
    hipStream_t st;
    const KParams* p;
    const KParams* table;
    const Chunk* chunks;
    int nchunks;
    unsigned* counter;
    unsigned long long* steps;
    int* occ;
    bool rec;                 // records carry E, B or work columns
};

// generic kernels, FP64 and FP32C, per field-kind class: analytic fields
// (tpamd_gen64a/32a.hip), + grids (nodes tpamd_gen64/32.hip, cells
// tpamd_gen64c/32c.hip), + meshes (tpamd_gen64m/32m.hip)
void launch_generic64_analytic(const LaunchReq& r, int alg, bool special);
void launch_generic32_analytic(const LaunchReq& r, int alg, bool special);
void launch_generic64(const LaunchReq& r, int alg);
void launch_generic32(const LaunchReq& r, int alg);
void launch_generic64_cells(const LaunchReq& r, int alg);
void launch_generic32_cells(const LaunchReq& r, int alg);
void launch_generic64_mesh(const LaunchReq& r, int alg);
void launch_generic32_mesh(const LaunchReq& r, int alg);
// specialised gridded-B kernels (tpamd_spec64/32.hip): emode kEUniform /
// kEUxB, ns the subcycle class, per a periodic grid, f32 float storage,
// cells the cell-replicated layout
void launch_spec64(const LaunchReq& r, int emode, int ns, bool per, bool f32, bool cells);
void launch_spec32(const LaunchReq& r, int emode, int ns, bool per, bool cells);
// the reference-form multistep classes (ns = kRefBase + n)
void launch_spec64r(const LaunchReq& r, int emode, int ns, bool per, bool f32, bool cells);
void launch_spec32r(const LaunchReq& r, int emode, int ns, bool per, bool cells);
// fixed-step Boris with two gathers a step (tpamd_pair64/32.hip): gridded E
// and B on one geometry, or (time) B a sequence of snapshots
void launch_pair64(const LaunchReq& r, bool time, bool uxb, bool per, bool f32, bool cells);
void launch_pair32(const LaunchReq& r, bool time, bool uxb, bool per, bool cells);
// full-orbit segments of the hybrid solver (tpamd_hybrid.hip)
struct FoArgs {
    double* state;       // [N][8] x, v, t, dt
    long long* iters;    // [N][2] it, steps
    int* flags;          // [N] in: TPAMD_FO_ENTER | TPAMD_FO_CHECKED; out: status
    double* sync;        // [N][6]
    double dtmin, dtmax, safety;
    long long check_interval, maxiters;
};
void launch_fo_segment(const KParams& p, const FoArgs& a, int fk, hipStream_t st);
// the checkpointed adjoint (tpamd_adj.hip)
int adjoint_launch(tpamd_ctx* ctx, const KParams& p, const tpamd_field* B, const double* xv0,
                   int64_t N, const double* targets, int K, int64_t nt, double* loss,
                   double* dL_dB, double* dL_dxv0, tpamd_stats* stats, bool f32, bool bf32,
                   bool per, bool cells, bool bycomp, bool ckpt);

}  // namespace tpamd

#define HIP_TRY(ctx, expr)                                                                   \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess)                                                                \
            return tpamd::fail((ctx), e_ == hipErrorOutOfMemory ? TPAMD_ERR_OOM : TPAMD_ERR_DEVICE, \
                               "%s failed: %s", #expr, hipGetErrorString(e_));               \
    } while (0)
