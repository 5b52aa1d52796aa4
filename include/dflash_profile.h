/*
 * dflash_profile.h -- measurement hooks of libdflash_hip.so.
 *
 * NOT part of the drop-in surface (include/dflash_hip.h, include/dflash_cache.h): nothing the reference's call
 * sites need is declared here, the module map does not export this header, and a host that only serves requests
 * never includes it.  The benchmark and the profiles use these entries to time single kernels and to price
 * launches that do no work.
 */
#ifndef DFLASH_PROFILE_H
#define DFLASH_PROFILE_H

#ifdef __cplusplus
extern "C" {
#endif

/* ------------------------------------------------------------------------
 * Measurement hook (no counterpart in the reference, whose bench times whole
 * calls from the host: Sources/DFlashKernelBench/main.swift:33-57).  Arms the
 * calling thread so that the NEXT launch of the named kernel carries the two
 * events on its own dispatch (hipExtLaunchKernelGGL): their elapsed time is the
 * kernel's begin-to-end duration on the launch stream, as a profiler's kernel
 * trace reports it.  The arming is consumed by that launch.  Events are
 * hipEvent_t passed as void*, created and read by the caller.
 * ---------------------------------------------------------------------- */
#define DFLASH_KERNEL_SDPA_PARTIAL 0
#define DFLASH_KERNEL_SDPA_COMBINE 1
#define DFLASH_KERNEL_GDN_FORWARD 2
#define DFLASH_KERNEL_TAPE_REPLAY 3
#define DFLASH_KERNEL_GREEDY_PARTIAL 4
#define DFLASH_KERNEL_GDN_PREPARE 5
#define DFLASH_KERNEL_EMPTY 6
#define DFLASH_KERNEL_GDN_LAYER 7
#define DFLASH_KERNEL_GDN_FINISH 8
#define DFLASH_KERNEL_COUNT 9
int dflash_profile_next_launch(int kernel_id, void* start_event, void* stop_event);

/* Launches a kernel that does nothing, with the given grid, block size (a multiple of 64, at most
 * 1024) and dynamic LDS size (at most 160 KB): the cost of a launch of that shape before any work,
 * i.e. the floor under each kernel of a verify step.  No counterpart in the reference.  Kernel id
 * DFLASH_KERNEL_EMPTY for dflash_profile_next_launch. */
int dflash_profile_empty_launch(void* stream, int grid_x, int grid_y, int grid_z, int threads, int lds_bytes);

/* What dflash_sdpa_block_causal* launches for a batch whose sequences all have N keys (with lengths on the device the
 * workgroups may be dealt, or the splits more than fit at once, which changes the first grid): kernel names and launch
 * shapes, in launch order, for pricing and labelling a step's launches.  Returns how many there are (1 or 2), or 0 for a
 * call that those entries refuse.  No counterpart in the reference. */
typedef struct {
    const char* kernel;
    int grid_x, grid_y, grid_z, threads, lds_bytes;
} dflash_launch_shape;
int dflash_profile_sdpa_launches(int dtype, int B, int Hq, int Hk, int N, int D, dflash_launch_shape shapes[2]);

/* What dflash_gdn_layer launches first for rows aligned to 16 bytes and the gated norm in the same launch.  Returns 1, or 0 for
 * sizes that it refuses.  No counterpart in the reference. */
int dflash_profile_gdn_layer_launch(int in_dtype, int B, int Hv, int Dk, int Dv, dflash_launch_shape* shape);

#ifdef __cplusplus
}
#endif
#endif /* DFLASH_PROFILE_H */
