// Kernel argument block of the generator kernels (host and device).
#pragma once
#if !defined( __HIPCC_RTC__ )
#include <stdint.h>
#endif
#include "fn2_program.h"

namespace fn2
{
    // A range record: the output range of one call as ordered-int keys.
    // With rangeSlots > 0 it is kept in `slots` {min, max} pairs `stride` ints apart (GenArgs::rangeSlots,
    // a power of two, and GenArgs::rangeStride). A block (or a wave)
    // publishes to the slot of its index, so that its atomics do not queue
    // behind every other block's on one address: device-wide atomics on one
    // 128-byte line complete one after another, about 11 ns each on MI355X.
    // The range is the smallest min key and the largest max key over the
    // slots. Measured (1 slot -> 16 compact slots -> 16 slots on their own
    // lines): Perlin 64^3 15.0 -> 9.1 -> 4.4 us, a 1 M-point 4D call 56 ->
    // 41 -> 40 us; 512 blocks storing 1 MB took 3.22 us with 16 lines, 2.69
    // with 64 and 2.64 with 256 (2.22 without a record). The entry point that
    // allocates nothing takes kCallRangeSlots slots, the persistent serving
    // mode kRangeSlots per request.
    //
    // With rangeSlots = kRangePerBlock the record is a {min, max} pair per
    // block instead (rangeStride of them): block b of the call (of a batched
    // request: of its job) stores its pair at 2 b. Nothing is reset before
    // and no atomics queue up. Up to kRangeDirectBlocks blocks store their
    // pairs to pinned host memory, and the host reads them when the kernel
    // has ended; more blocks store them to device memory, and a reduction
    // launch after the kernel (fn2_launch_range_reduce) leaves one pair per
    // job in pinned memory. Against a reset launch, atomics and a copy of the
    // record of slots (MI355X, whole calls with their range): 16^3 Perlin 21.4
    // -> 16.4 us, 64^3 22.8 -> 20.5, 1 M-point 4D 51.7 -> 50.1. A small
    // store over PCIe costs about 2 ns, one after the other: with pinned
    // pairs for every launch, a 1.8 M-point call of 6,900 blocks took 55.7
    // us instead of 50.1; between 512 and 2048 blocks both ways are equal.
    constexpr int kRangeSlots = 16;
    constexpr int kCallRangeSlots = 64;
    constexpr int kRangePerBlock = 0;
    constexpr int kRangeDirectBlocks = 512;
    constexpr int kRangeStrideSpread = 32;    // a slot per 128-byte line

    // Blocks of a single call at most (its record holds a pair for each):
    // twice the 8 resident blocks of 256 threads per CU times 4 rounds that
    // such a call is launched with on 256 CUs
    constexpr int kMaxCallBlocks = 16384;

    // A work-queue launch's counters: kQueueCounters of them, each on its own
    // 128-byte line (kQueueCounterStride uint32 apart); counter c hands out
    // the c-th sixteenth of the items beyond the first one per wave.
    constexpr int kQueueCounters = 16;
    constexpr int kQueueCounterStride = 32;
    constexpr int kQueueCounterInts = kQueueCounters * kQueueCounterStride;

    // The work-queue partition of a launch of `waves` waves over `items`
    // items: wave g runs item g first; the items beyond the first round are
    // split into min(waves, kQueueCounters) contiguous parts, one per
    // counter, and wave g pulls the items of part g % parts, [first, end),
    // from that part's counter. Every part has a wave for any grid size.
    struct QueuePart
    {
        uint32_t part, first, end;
    };
#if defined( __HIPCC__ ) || defined( __HIPCC_RTC__ )
    __host__ __device__
#endif
    inline QueuePart queuePart( uint32_t g, uint32_t waves, uint32_t items )
    {
        const uint32_t parts = waves < (uint32_t)kQueueCounters ? waves : (uint32_t)kQueueCounters;
        const uint32_t extra = items > waves ? items - waves : 0;
        const uint32_t chunk = ( extra + parts - 1 ) / parts;
        QueuePart q;
        q.part = g % parts;
        q.first = waves + q.part * chunk;
        q.end = q.first + chunk < items ? q.first + chunk : items;
        return q;
    }

    struct GenArgs
    {
        const Ins* ins;          // device program
        const float* konst;      // device constant pool
        int32_t nIns;
        int32_t resultReg;
        int32_t dims;            // dimensionality of the starting position
        int32_t kind;            // SourceKind
        int32_t seed;
        int32_t total;           // points (the reference counts in int)
        float* out;              // device output, `total` floats
        int32_t* minmax;         // range record (ordered-int keys), or null
        FastDiv div[3];          // grid: divisors by x, y, z count; tileable: div[0] = x size
        float offset[4];
        float step[4];
        const float* pos[4];     // position arrays (device); tileable: cos x, cos y, sin x, sin y tables
        int32_t ppt;             // batched kernel: points per lane of each block of this job
        int32_t regs;            // registers the program uses (the interpreter's file holds as many)
        int32_t tables;          // LDS tables the program reads (kTable* bits)
        int32_t rangeStride;     // ints between the slots of the range record (kRangePerBlock: its pairs)
        int32_t rangeSlots;      // slots of the range record (a power of two), or kRangePerBlock
        // index of this job's first point in its request: a request split
        // into several jobs evaluates points base + [0, total) of the whole
        // grid or image (position arrays are offset by the host instead)
        uint32_t base;
    };
}
