// Host-side launchers of the kernels in fn2_kernels.hip (C linkage; each
// returns a hipError_t). fn2_kernels.hip includes this header too, so a
// definition that drifts from its declaration fails to compile.
#pragma once
#include <stdint.h>
#include <hip/hip_runtime_api.h>
#include "fn2_kernel_args.h"

namespace fn2
{
    // A range record of a pair per block
    struct RangeRecord
    {
        const int32_t* pairs;
        int32_t count;
    };

    // Density blocks of one face-count launch, passed by value, and the
    // { quads, solid } entries its blocks write at most
    // (fn2_face_blocks( n, gen ) per chunk, n <= kFaceJobs)
    constexpr int kFaceJobs = 64;
    constexpr int kFaceEntries = 2048;
    struct FaceJobs
    {
        const float* density[kFaceJobs];
    };
}

extern "C" {
// one interpreter launch over args->total points. `blocks` (may be null)
// receives the launch's blocks; with at most kRangeDirectBlocks of them their
// range pairs go to `direct` (unless null) instead of args->minmax
int fn2_launch_generate( const fn2::GenArgs* args, int dimMask, int featMask, hipStream_t stream, int32_t* direct, unsigned* blocks );
// blocks of a single-call launch over `total` points (also used for the
// run-time specialised kernels), at most kMaxCallBlocks
unsigned fn2_grid_for( int64_t total, int blocksPerCU );
// the same for grid requests of cheap programs (JitKernel::wide); at most
// kMaxCallBlocks when the call has a range record
unsigned fn2_wide_grid_for( int64_t total, int ranged );
// interpreter launch over a batch of jobs (block b runs job dBlockJob[b])
int fn2_launch_generate_batch( const fn2::GenArgs* dJobs, const int32_t* dBlockJob, const uint32_t* dBlockBase, int nBlocks, int dimMask, int featMask,
                               int regs, hipStream_t stream );
// interpreter work-queue launch over nTiles tiles of a batch
int fn2_launch_generate_queue( const fn2::GenArgs* dJobs, const int32_t* dTileJob, const uint32_t* dTileBase, int nTiles, int dimMask, int featMask,
                               int regs, uint32_t* dCounter, hipStream_t stream );
// reduces n per-block range records (those of dJobs, or `one` when dJobs is
// null) to a pair each at out + 2 j
int fn2_launch_range_reduce( const fn2::GenArgs* dJobs, fn2::RangeRecord one, int n, int32_t* out, hipStream_t stream );
// resets n consecutive range records of `slots` slots, `stride` ints apart
int fn2_launch_minmax_init( int32_t* keys, int n, int slots, int stride, hipStream_t stream );
// the same, also zeroing nc work-queue counters
int fn2_launch_batch_init( int32_t* keys, int n, int slots, int stride, uint32_t* counters, int nc, hipStream_t stream );
// threads per block of the batched interpreter kernel
int fn2_batch_block_threads( void );
// device-side checks of the math helpers
int fn2_launch_selftest_math( int op, const float* in, float* out, int n, hipStream_t stream );
// faces of the bloxel meshes of n gen^3 density blocks (divS divides by
// gen - 2): fn2_face_blocks( n, gen ) entries of { quads, solid } per block,
// chunk after chunk, into `partials`
int fn2_face_blocks( int n, int gen );
int fn2_launch_bloxel_faces( const fn2::FaceJobs* jobs, int n, int gen, fn2::FastDiv divS, float iso, uint32_t* partials, hipStream_t stream );
}
