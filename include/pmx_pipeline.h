/*
 * pmx_pipeline.h — C ABI of a pipeline library generated by the MI355X
 * PolyMage backend (polymage_amd/host_stub.py writes it; runtime.build
 * links it as lib<name>.so against libpmx_rt.so).
 *
 * For a pipeline named <name> with parameters P..., input images I... and
 * live-out outputs O... (each list sorted by name, the reference's order,
 * sandbox/codegen.py:957-999 and sandbox/utils.py:98-115), the library
 * exports the functions below.  Parameters are passed by value with their
 * DSL C type (Int -> int, Float -> float, ...).  Images are dense,
 * row-major arrays over their declared extents; outputs cover the
 * bounding box of their domain; points no Case defines keep the bytes the
 * caller put there.
 *
 * All int-returning functions return 0 on success, or a negative /
 * hipError_t code with the message in pmx_last_error() (pmx_rt.h).
 * Errors: a parameter set for which some unconditional access falls
 * outside the producer's declared extent (the reference raises this at
 * compile time for its fixed estimates, sandbox/bounds.py:36-118), an
 * extent above INT_MAX points, or a group whose per-tile region outgrows
 * its planned scratch box (device status word, pipeline_<name>_status).
 */
#ifndef PMX_PIPELINE_H
#define PMX_PIPELINE_H

#ifdef __cplusplus
extern "C" {
#endif

/* ---- generic form (macro only documents the shapes) ------------------------
 *
 * Replaces the reference's generated entry point
 *   void pipeline_<name>(P..., void* I..., void* O...)
 * (sandbox/codegen.py:957-999; loaded by sandbox/apps/python/loader.py:4-21,
 * called by sandbox/tuner.py:525 and the apps' exec_pipe.py files):
 *
 *   void pipeline_<name>(P..., void* I..., void* O...);
 *       host pointers, synchronous; prints pmx_last_error() on failure.
 *   int  pipeline_<name>_host(P..., void* I..., void* O...);
 *       same, returns the status instead of printing.
 *   int  pipeline_<name>_dev(P..., const void* I_dev..., void* O_dev...,
 *                            void* stream);
 *       device pointers, enqueued on `stream` (NULL = null stream), no
 *       synchronisation; intermediates live in the device arena.
 *   int  pipeline_<name>_status(void);
 *       synchronises the device and reports the device overflow guard of
 *       the last launches (0 = fine), of both _dev and _dev_noalloc calls.
 *   int  pipeline_<name>_dev_noalloc(P..., const void* I_dev..., void* O_dev...,
 *                                    void* stream);
 *       No counterpart in the reference.  For callers that cannot allocate
 *       device memory (code under HIP graph capture, tight serving loops,
 *       harnesses that forbid hipMalloc): the launches of _dev, with the
 *       status word, constant tables and intermediates carved from the
 *       runtime's static device scratch (PMX_SCRATCH_BYTES per GPU,
 *       pmx_rt.h) instead of the arena.  After its first call on a device
 *       (which loads the code object and looks the scratch address up) it
 *       allocates nothing.  Sizes needing more than the scratch holds
 *       return -12 before anything is launched.  Every such call on a GPU
 *       shares that GPU's scratch: calls that overlap on one GPU race.
 *
 * Batched frames (no reference counterpart; one launch per kernel
 * for many small or uneven frames):
 *
 *   int pipeline_<name>_batch_create(int n, const P* P_arr...,
 *                                    void* const* I_arr..., void* const* O_arr...,
 *                                    void** handle);
 *       n frames; per-frame parameters and device pointers; validates every
 *       frame and builds the frame tables on the device.
 *   int pipeline_<name>_batch_run(void* handle, void* stream);
 *       one launch per kernel over all frames' tiles (a workgroup each).
 *   int pipeline_<name>_batch_run_graph(void* handle, void* stream);
 *       the same launches captured once into a hipGraph, replayed.
 *   int pipeline_<name>_batch_run_frames(void* handle, void* stream);
 *       the per-frame path (pipeline_<name>_dev for each frame), for
 *       comparison.
 *   int pipeline_<name>_batch_destroy(void* handle);
 */

/* ---- the five benchmark pipelines ------------------------------------------ */

/* Harris corner response, sandbox/apps/python/img_proc/harris/polymage_harris.py:13-78.
 * img: float[R+2][C+2], harris: float[R+2][C+2] (interior written). */
void pipeline_harris(int C, int R, void* img, void* harris);
int pipeline_harris_dev(int C, int R, const void* img_dev, void* harris_dev, void* stream);
int pipeline_harris_dev_noalloc(int C, int R, const void* img_dev, void* harris_dev, void* stream);

/* Unsharp mask, sandbox/apps/python/img_proc/unsharp_mask/polymage_unsharp_mask.py:16-77.
 * img: float[3][R+4][C+4], mask: float[3][R][C]. */
void pipeline_unsharp(int C, int R, float threshold, float weight, void* img, void* mask);
int pipeline_unsharp_dev(int C, int R, float threshold, float weight,
                         const void* img_dev, void* mask_dev, void* stream);
int pipeline_unsharp_dev_noalloc(int C, int R, float threshold, float weight,
                                 const void* img_dev, void* mask_dev, void* stream);

/* Bilateral grid, sandbox/apps/python/img_proc/bilateral_grid/polymage_bilateral_grid.py:16-130.
 * input: float[rows][cols], filtered: float[rows][cols]. */
void pipeline_bilateral(int cols, int rows, void* input, void* filtered);
int pipeline_bilateral_dev(int cols, int rows, const void* input_dev, void* filtered_dev,
                           void* stream);
int pipeline_bilateral_dev_noalloc(int cols, int rows, const void* input_dev, void* filtered_dev,
                                   void* stream);

/* Local Laplacian filter (uint16, K = 8 intensity levels, J = 4 pyramid
 * levels), restated from sandbox/video_demo/laplacian_naive.cpp:10-931.
 * R, C are the padded sizes: img_colour: uint16[R - p][C - p][3] with
 * p = 3*2^J - 4 (edge padding 2^J - 1 before, 2^(J+1) - 3 after),
 * laplacian: uint16[R - p][C - p][3]. */
void pipeline_laplacian(int C, int R, float alpha, float beta, void* img_colour, void* laplacian);
int pipeline_laplacian_dev(int C, int R, float alpha, float beta,
                           const void* img_colour_dev, void* laplacian_dev, void* stream);
int pipeline_laplacian_dev_noalloc(int C, int R, float alpha, float beta,
                                   const void* img_colour_dev, void* laplacian_dev, void* stream);

/* Camera raw pipeline, sandbox/apps/python/img_proc/campipe/polymage_campipe.py:13-304
 * (batched benchmark variant: 10-bit input, 1024-entry curve, 3x3 sharpen).
 * img: uint16[R][C] raw Bayer, matrix_3200/7000: float[3][4],
 * process: uint8[3][R-48][C-64]. */
void pipeline_campipe(int C, int R, float colour_temp, float contrast, float gamma,
                      void* img, void* matrix_3200, void* matrix_7000, void* process);
int pipeline_campipe_dev(int C, int R, float colour_temp, float contrast, float gamma,
                         const void* img_dev, const void* matrix_3200_dev,
                         const void* matrix_7000_dev, void* process_dev, void* stream);
int pipeline_campipe_dev_noalloc(int C, int R, float colour_temp, float contrast, float gamma,
                                 const void* img_dev, const void* matrix_3200_dev,
                                 const void* matrix_7000_dev, void* process_dev, void* stream);
int pipeline_campipe_batch_create(int n, const int* C_arr, const int* R_arr,
                                  const float* colour_temp_arr, const float* contrast_arr,
                                  const float* gamma_arr, void* const* img_arr,
                                  void* const* matrix_3200_arr, void* const* matrix_7000_arr,
                                  void* const* process_arr, void** handle);
int pipeline_campipe_batch_run(void* handle, void* stream);
int pipeline_campipe_batch_run_graph(void* handle, void* stream);
int pipeline_campipe_batch_run_frames(void* handle, void* stream);
int pipeline_campipe_batch_destroy(void* handle);

#ifdef __cplusplus
}
#endif
#endif /* PMX_PIPELINE_H */
