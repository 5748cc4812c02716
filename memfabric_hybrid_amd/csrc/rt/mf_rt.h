// Thin C layer over HIP.  Host C++ above this line never sees a HIP type:
// streams, events and device pointers travel as void*, sizes as integers.
// mfrt_* = runtime services, mfk_* = kernel launchers (enqueue only).
// Every int return is 0 on success or the hipError_t value.
#ifndef MF_RT_H
#define MF_RT_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* The plugin library keeps the runtime layer private so that it can share a
 * process with the data-plane library. */
#ifndef MF_RT_HIDDEN
#pragma GCC visibility push(default)
#endif

#define MFRT_ROUTE_HBM 0        /* source and destination in HBM            */
#define MFRT_ROUTE_TO_HOST 1    /* destination in pinned, mapped host DRAM  */
#define MFRT_ROUTE_FROM_HOST 2  /* source in pinned, mapped host DRAM       */

#define MFRT_PTR_PAGEABLE 0     /* ordinary host memory the GPU cannot address */
#define MFRT_PTR_DEVICE 1
#define MFRT_PTR_PINNED_HOST 2

/* ---- runtime ------------------------------------------------------------ */
int mfrt_init(int device);
int mfrt_current_device(void);          /* device current on the calling thread, -1 on error */
int mfrt_bind_thread(void);             /* make the initialised device current on this thread */
void mfrt_shutdown(void);
int mfrt_is_initialised(void);
int mfrt_device_id(void);
uint32_t mfrt_cu_count(void);
const char *mfrt_error_string(int err);

void *mfrt_alloc_device(uint64_t bytes);
int mfrt_free_device(void *p);
void *mfrt_alloc_host(uint64_t bytes);  /* pinned + device-mapped + portable */
int mfrt_free_host(void *p);
int mfrt_pointer_kind(const void *p);

/* Address windows: reserve virtual addresses first, back pieces of them with HBM later
 * (hipMemAddressReserve / hipMemCreate / hipMemMap).  Sizes and offsets are multiples of
 * mfrt_window_granularity().  A mapping is named by the handle mfrt_window_map returns;
 * [accessBase, +accessBytes) is the contiguous mapped run that ends with the new piece. */
uint64_t mfrt_window_granularity(void);
void *mfrt_window_reserve(uint64_t bytes);
int mfrt_window_release(void *base, uint64_t bytes);
void *mfrt_window_map(void *addr, uint64_t bytes, void *accessBase, uint64_t accessBytes);  /* handle, NULL on failure */
int mfrt_window_unmap(void *addr, uint64_t bytes, void *handle);
int mfrt_window_last_error(void);                       /* failed step (1 create, 2 map, 3 access) * 10000 + hipError_t */

void *mfrt_stream_create(void);
int mfrt_stream_destroy(void *stream);
int mfrt_stream_sync(void *stream);
int mfrt_stream_done(void *stream);                     /* 1 nothing left to run, 0 pending, <0 error */
int mfrt_stream_capturing(void *stream);                /* 1: launches on the stream become nodes of a HIP graph */
int mfrt_device_sync(void);

void *mfrt_event_create(void);
int mfrt_event_destroy(void *event);
int mfrt_event_record(void *event, void *stream);
int mfrt_event_sync(void *event);
int mfrt_stream_wait_event(void *stream, void *event);   /* work queued on `stream` afterwards waits for the event */
/* 1: launches on the two (idle) streams run one after the other because the streams share a hardware queue; 0: they
 * run side by side; -1: not known.  About 50 us. */
int mfrt_streams_share_queue(void *a, void *b);
int mfrt_event_done(void *event);       /* 1 finished, 0 pending, <0 error */
float mfrt_event_elapsed_ms(void *start, void *stop);

int mfrt_memcpy(void *dst, const void *src, uint64_t bytes);  /* blocking hipMemcpy, direction inferred */
int mfrt_memset(void *dst, int value, uint64_t bytes);
int mfrt_memcpy_async(void *dst, const void *src, uint64_t bytes, void *stream);  /* the runtime's own DMA path */

/* ---- xcopy launchers (kernels/xcopy.hip) --------------------------------- */
/* anyOrder != 0: the launch does not wait for launches queued before it on `stream` (it carries no barrier);
 * launches queued after it without that option still wait for it. */
/* holdNanos != 0: every wave keeps its loaded data until that long after its own start (see HoldNanosFor in
 * kernels/xcopy_plan.h); honoured only by a launch of one chunk per workgroup, the chunk being 4 KiB or
 * mfk_xcopy_window_units() units (16 KiB, copied by single waves with sixteen loads per lane in flight). */
int mfk_xcopy_inline(const void *inlinePlan, int route, uint32_t grid, void *mask, uint32_t maskValue, void *stream,
                     int anyOrder, uint32_t holdNanos);
/* A copy by `grid` workgroups, few or short-lived ones, that stores `value` into `word` (pinned host memory) itself once every
 * byte it moved is in memory, without a launch behind it.  `counter` is a word of device memory, 0 before the launch and 0
 * again when `word` has been stored: launches that share it follow one another on a stream. */
int mfk_xcopy_done(const void *inlinePlan, int route, uint32_t grid, void *word, uint32_t value, void *counter, void *stream);
/* HBM to HBM copies of hundreds of MiB: the plan's chunks are mfk_xcopy_window_units() units (16 KiB), copied by up to
 * 6144 single-wave workgroups that alternate, chip-wide and by the clock, between a read half and a
 * write half of a period cut for `windowMBps` MB/s of HBM traffic, whatever the addresses (see XcopyWindowKernel). */
int mfk_xcopy_windows_available(void);   /* 1 when the current device's constant-rate clock is known, which the period is cut by */
uint32_t mfk_xcopy_window_units(void);
int mfk_xcopy_windowed(const void *inlinePlan, uint32_t windowMBps, void *mask, uint32_t maskValue, void *stream);
/* tablePlan: a mf::TablePlan (kernels/xcopy_plan.h).  Under a pattern its triples may live in pinned host
 * memory and neither prefix nor group map is read. */
int mfk_xcopy_table(const void *tablePlan, int route, uint32_t grid, void *mask, uint32_t maskValue, void *stream);
/* HBM to HBM: `count` mf::Piece (kernels/xcopy_plan.h) in pinned host memory, of together `bytes` bytes and up to `units` (256, 512
 * or 1024) units each.  holdNanos: as for mfk_xcopy_inline; it is what a table of as many chunks would wait.
 * event (may be NULL): completes with the launch.  The stream must not be one that records a graph, whose launches cannot carry one. */
int mfk_xcopy_pieces(const void *pieces, uint32_t count, uint64_t bytes, uint32_t units, void *mask, uint32_t maskValue, void *stream,
                     uint32_t holdNanos, void *event);
/* The same pieces; the launch stores `value` into `word` (pinned host memory) once `pieces` may be rewritten.  Without a counter when
 * it has started: the launches before it on `stream` have then ended, and theirs may be.  With one (kDoneCounterBytes of device memory,
 * 0 between launches that follow one another) when every wave has its descriptor.  windowMBps != 0, which takes no counter: in
 * windows, as mfk_xcopy_pieces_windowed. */
int mfk_xcopy_pieces_reported(const void *pieces, uint32_t count, uint64_t bytes, uint32_t units, uint32_t holdNanos, uint32_t windowMBps,
                              uint32_t reading, void *word, uint32_t value, void *counter, void *stream);
/* The same pieces, of 4 KiB each; the launch stores `value` into `word` once every byte is in memory.  `counter`: as for
 * mfk_xcopy_done. */
int mfk_xcopy_pieces_done(const void *pieces, uint32_t count, void *word, uint32_t value, void *counter, void *stream);
/* The same pieces, of up to mfk_xcopy_window_units() units, whatever their addresses (those off cache lines hold a lower rate), in read and
 * write windows cut for `windowMBps` MB/s of HBM traffic.  reading: 64ths of a period that are its read part, 0 = half of it. */
int mfk_xcopy_pieces_windowed(const void *pieces, uint32_t count, uint64_t bytes, uint32_t windowMBps, uint32_t reading, void *mask, uint32_t maskValue,
                              void *stream, void *event);
/* Launches every copy kernel once on empty plans (a kernel's first launch is not capturable into a HIP graph). */
int mfk_xcopy_prelaunch(void *stream);
/* Times the calibration workloads on `stream` with HIP events, in 1 GiB of device memory it allocates and frees:
 * out[0 .. 3] = us per 2196-chunk batch without a hold and held for holdNanos[0 .. 2]; out[4 .. 7] = us per 512 MiB
 * copy without windows and in windows cut for windowMBps[0 .. 2].  0, or a HIP error number. */
int mfk_xcopy_calibrate(void *stream, const uint32_t *holdNanos, const uint32_t *windowMBps, float *out);
/* One lane stores `value` (as a 64-bit word, released at system scope) into `word` once everything queued on
 * `stream` before it has finished. */
int mfk_xcopy_signal(void *word, uint32_t value, void *stream);
/* A triple table in device memory, copied without a plan (kernels/xcopy_plan.h says how): `grid` workgroups walk its segments,
 * `restGrid` those of the second launch what is left of the long segments that the first has listed in `rest`, a mf::RestList in
 * device memory with room for `capacity` segments whose counts are 0 before and after.  One call at a time may use a list.
 * event: as for mfk_xcopy_pieces; NULL on a stream that records a graph.  windowMBps: as for mfk_xcopy_planned, for longer tables
 * between HBM addresses whose segments, as far as they are looked at, are pages of one length; 0: they go as all others. */
int mfk_xcopy_direct(const void *triples, uint32_t nseg, uint32_t units, int route, uint32_t grid, uint32_t restGrid, void *rest,
                     uint32_t capacity, uint32_t windowMBps, void *mask, uint32_t maskValue, void *stream, void *event);
/* A triple table in device memory of up to kPlannedSegments (kernels/xcopy_plan.h) segments between HBM addresses, in one launch that
 * reads and plans it.  Waves that are resident together hold their stores for holdNanos and holdMoreNanos per 64 MiB; what is more goes
 * in read and write windows cut for `windowMBps`.  0: not held, no windows. */
int mfk_xcopy_planned(const void *triples, uint32_t nseg, uint32_t holdNanos, uint32_t holdMoreNanos, uint32_t windowMBps, void *mask,
                      uint32_t maskValue, void *stream);
/* Makes `count` mf::RestList in device memory, `stride` bytes apart, empty. */
int mfk_xcopy_clear_lists(void *lists, uint32_t count, uint64_t stride, void *stream);
/* The same with the list in a statically allocated device array instead of memory the engine allocates: no allocation
 * anywhere, at most MFK_STATIC_TABLE_SEGMENTS segments, one call at a time per GPU.  mfk_xcopy_static_setup looks the
 * array's address up for the current device (once per device, at start-up); mfk_xcopy_table_static returns -2 when that has
 * not happened. */
#define MFK_STATIC_TABLE_SEGMENTS 32768u
int mfk_xcopy_static_setup(void);
int mfk_xcopy_table_static(const void *triples, uint32_t nseg, uint32_t units, int route, uint32_t grid, uint32_t restGrid, void *stream);

/* ---- staged copies (kernels/staging.hip) ---------------------------------- */
/* `count` mf::StreamChunk (kernels/staging.h) in pinned host memory, chunk c between HBM and slot c % slots, of kStreamChunkBytes, of a ring
 * in pinned host memory, where it begins `at` % kStreamLine bytes in; the launch runs while the CPU fills (toHost 0) or empties the slots.  hostWords and
 * gpuWords: a 64-bit word per slot, kStreamWordBytes apart, in which the CPU and the GPU say base + c + 1 when they are done with chunk c
 * there.  A workgroup that waits limitMillis for the CPU leaves, and the chunks it has left are not copied.  To the host it waits for
 * nothing, and count is at most slots.  The second form does not wait for launches queued before it on `stream` (it carries no barrier). */
int mfk_stream_chunks(int toHost, void *ring, const void *chunks, void *hostWords, void *gpuWords, uint64_t base, uint32_t count, uint32_t slots,
                      uint32_t limitMillis, void *stream);
int mfk_stream_chunks_beside(int toHost, void *ring, const void *chunks, void *hostWords, void *gpuWords, uint64_t base, uint32_t count,
                             uint32_t slots, uint32_t limitMillis, void *stream);

/* Every kernel of theirs once, on nothing. */
int mfk_stream_prelaunch(void *stream);

/* ---- MoE launchers (kernels/moe.hip) ---------------------------------------- */
uint64_t mfk_moe_workspace_bytes(uint32_t tokens, uint32_t topK, uint32_t experts);
int mfk_moe_dispatch(const void *x, const void *topk, uint32_t tokens, uint32_t hidden, uint32_t topK, uint32_t experts,
                     void *out, void *counts, void *offsets, void *rowOf, void *srcOf, void *workspace, void *stream);
/* paced != 0: the form whose waves stay and alternate between reading and writing may be used (see mfk_moe_combine_windows) */
int mfk_moe_combine(const void *rows, const void *rowOf, const void *weights, uint32_t tokens, uint32_t hidden,
                    uint32_t topK, void *y, void *stream, int paced);
/* once after the GPU is bound: finds out whether consecutive workgroups go to the eight XCDs in turn (the tile permute
 * of the dispatch needs it); mfk_moe_xcd_streams() is 1 if they do */
int mfk_moe_setup(void);
int mfk_moe_xcd_streams(void);
/* 1 where mfk_moe_dispatch with rows is the one launch in which every workgroup counts all ids */
int mfk_moe_dispatch_counts(uint32_t tokens, uint32_t hidden, uint32_t topK, uint32_t experts);
/* 1 where mfk_moe_combine takes the form that keeps reads and writes apart in time, if it may pace itself */
int mfk_moe_combine_stays(uint32_t tokens, uint32_t hidden, uint32_t topK);
/* pace of that form, MB/s for its read and write parts; 0 = never */
void mfk_moe_combine_windows(uint32_t readMBps, uint32_t writeMBps);

/* ---- 2-D copy launcher (kernels/copy2d.hip) ----------------------------------- */
int mfk_copy2d(const void *rectPlan, uint32_t grid, void *stream);
/* rectChunkPlan: mf::RectChunkPlan; in read and write windows cut for windowMBps over chunks of kRectWindowUnits units, or with 0 in
 * chunks of 64 * kRectChunkDepth.  Between HBM addresses. */
int mfk_copy2d_chunks(const void *rectChunkPlan, uint32_t windowMBps, void *stream);
/* Every rectangle kernel once on an empty plan. */
int mfk_copy2d_prelaunch(void *stream);

#ifndef MF_RT_HIDDEN
#pragma GCC visibility pop
#endif

#ifdef __cplusplus
}
#endif

#endif /* MF_RT_H */
