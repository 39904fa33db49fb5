// The thin extern "C" HIP layer underneath the host API: one function per
// kernel launch, nothing but pointers and ints, no validation (the host API
// has checked the shapes these grids assume).
#ifndef FLASHLLM_AMD_SPMM_LAUNCH_H
#define FLASHLLM_AMD_SPMM_LAUNCH_H

#include "flashllm_spmm.h"

#include <stddef.h>

// size of the library-owned slab storage behind flashllm_hip_static_workspace: the limit the public header states
#define FLASHLLM_STATIC_WORKSPACE_BYTES FLASHLLM_STATIC_WORKSPACE_MAX_BYTES

#ifdef __cplusplus
extern "C" {
#endif

// *ptr = device address, on the current device, of the library's own fixed slab storage
// (FLASHLLM_STATIC_WORKSPACE_BYTES, 256-byte aligned).  Resolved once per device; allocates nothing.
int flashllm_hip_static_workspace(void** ptr);

// How a launch of the products below stores its sums.
enum {
    kStorePlain = 0,  // C, or slab s as M*N halfs at s*M*N, laid out like C (for flashllm_hip_launch_reduce)
    kStorePages = 1,  // split_k > 1: each workgroup's 128 x 16 blocks of partial sums as 4 KB pages in workgroup order
                      // (for flashllm_hip_launch_reduce_pages; needs out 16-byte aligned)
    kStoreRelu = 2    // split_k == 1: C through max(., 0), the activation between FFN1 and FFN2
};

// out: C when split_k == 1, else the slab workspace (split_k * M * N halfs).
// ldb: halfs between consecutive columns of B (>= K, a multiple of 8; K for a dense column-major B).
// k_waves: 1, 2, 4 or 8 waves per workgroup divide each (row tile, slice) among themselves along K (ignored by a
// launch that takes eight row tiles per workgroup, below).  0, for n = 64: four waves with a quarter of the slice each
// (spmm_quarter_kernel; pages only with one row tile per workgroup).
// Requires M % 128 == 0, K % 64 == 0, N in {8,16,32,64} or N % 64 == 0.
int flashllm_hip_launch_spmm(void*       stream,
                             const void* compressed_a,
                             const int*  tile_offsets,
                             const void* b,
                             int         ldb,
                             void*       out,
                             int         m,
                             int         n,
                             int         k,
                             int         split_k,
                             int         store,
                             int         k_waves);

// Row tiles per workgroup of flashllm_hip_launch_spmm for n columns, m rows and split_k slices: 8 for n = 64
// when m / 128 is a multiple of 8 and (m / 1024) * split_k lies in 192 .. 256, otherwise 1.
// flashllm_hip_set_rows_per_workgroup is a measuring and testing aid, process-wide: 1 forces 1, 8 forces 8
// wherever m / 128 is a multiple of 8, anything else restores the rule.  The launch of the partial products and
// the reduction of its pages must see the same setting.
void flashllm_hip_set_rows_per_workgroup(int rows);
int  flashllm_hip_rows_per_workgroup(int n, int m, int split_k);

// The same product for wide B (n % 128 == 0).  runs 1: by workgroups of four waves that share each scattered tile, 128
// or 256 columns each (a rule of n, m and split_k, which the reduction of its pages follows too).  Any other value: by
// workgroups of four waves, 128 columns each, that divide the slice along K among themselves and add up at the end (pages
// only where the rule says 128).
int flashllm_hip_launch_spmm_group(void*       stream,
                                   const void* compressed_a,
                                   const int*  tile_offsets,
                                   const void* b,
                                   int         ldb,
                                   void*       out,
                                   int         m,
                                   int         n,
                                   int         k,
                                   int         split_k,
                                   int         store,
                                   int         runs);

int flashllm_hip_columns_per_workgroup(int n, int m, int split_k);

// The product and the reduction for wide B (n % 128 == 0) with the k tiles of all (row tile, 128 columns) divided evenly
// among 256 workgroups, share = tiles of each, at least a 256th of them.  ws: (kt - 1) / share + 2 slabs of M*N halfs, kt = K / 64.
int flashllm_hip_launch_spmm_even(void*       stream,
                                  const void* compressed_a,
                                  const int*  tile_offsets,
                                  const void* b,
                                  int         ldb,
                                  void*       c,
                                  void*       ws,
                                  int         m,
                                  int         n,
                                  int         k,
                                  int         share,
                                  int         relu);

// Time of such a launch per k tile of a slice, in us, with one group per workgroup: what Split_K is chosen by.
double flashllm_hip_wide_b_step(int n, int m, int split_k);

// c[e] = rn16(sum_s float(ws[s*mn + e])), through max(., 0) first when relu != 0; requires mn % 4 == 0.
int flashllm_hip_launch_reduce(void* stream, void* c, const void* ws, long mn, int split_k, int relu);

// The same sums over the pages a launch with kStorePages left for this (m, n, split_k): one workgroup per
// 128 x 16 block of C, on the XCD that stored the block's pages.  Requires M % 128 == 0, N as above, ws 16-byte
// and c 8-byte aligned.
int flashllm_hip_launch_reduce_pages(void* stream, void* c, const void* ws, int m, int n, int split_k, int relu);

// out[w] = id of the XCD workgroup w ran on, for a launch of `workgroups` one-wave workgroups shaped like the
// SpMM launches (a three-dimensional grid, eight wide, w counted x first, then y, then z): shows whether the
// round-robin hand-out in that order, which the placement above counts on, holds on this machine.
int flashllm_hip_launch_xcd_probe(void* stream, unsigned* out, int workgroups);

// dst[j*rows + i] = src[j*src_ld + i] for i < rows, j < cols (rows % 8 == 0, src_ld % 8 == 0).
int flashllm_hip_launch_take_rows(void* stream, void* dst, const void* src, int rows, int cols, int src_ld);

// offs[0..tiles+1] = TileOffsets of the device-resident dense matrix a (M x K halfs, 16-byte aligned,
// M % 128 == 0, K % 64 == 0): a count kernel and an in-place prefix sum, which also stores the sum of all counts at
// vectors (host memory the GPU can write, or null).
int flashllm_hip_launch_tile_offsets(void* stream, const void* a, int m, int k, int* offs, int* vectors);

// out[offs[t]*4 ...] = the packed nonzeros of tile t in the reference's reordered layout.
int flashllm_hip_launch_encode(void* stream, const void* a, int m, int k, const int* offs, void* out);

// The same in scan order (the layout of the reference's compressor without reordering).
int flashllm_hip_launch_encode_scan(void* stream, const void* a, int m, int k, const int* offs, void* out);

// A testing aid: takes all free words that a compression's size reaches the host through (64 in the process), so that calls copy it
// instead, or gives them back.  Returns how many.
int flashllm_hip_hold_host_words(int take);

// A weight on its way to the GPU without its zeros, in pieces of 65536 halfs: the index of the first value of each of its 32 groups
// (4 bytes), a bit per half, the values whose bits are not all zero, and room for what a 16-byte store writes beyond them.
enum {
    kPackPiece  = 65536,
    kPackGroup  = 2048,
    kPackBits   = kPackPiece / kPackGroup * 4,
    kPackValues = kPackBits + kPackPiece / 8,
    kPackStride = kPackValues + kPackPiece * 2 + 128
};

// One piece of n halfs (at most kPackPiece, a multiple of kPackGroup) at src, at dst.  Host only.
void flashllm_pack_piece(const unsigned short* src, size_t n, unsigned char* dst);
// The same in the way of processors without SSSE3, whatever this one has.
void flashllm_pack_piece_plain(const unsigned short* src, size_t n, unsigned char* dst);

// Whether n halfs at src reach the GPU sooner by way of packed pieces than as they are.
int flashllm_packing_pays(const unsigned short* src, size_t n);

// Threads that the host compressor would take for so many pieces of work.
int flashllm_compress_workers(size_t pieces);

// The same matrix at dst (device memory, 16-byte aligned) as flashllm_hip_upload leaves there, by way of packed pieces in stage (pinned
// host memory, 16-byte aligned, at least flashllm_hip_upload_stage(n) bytes: at most 30 MB) that a kernel fetches and expands.  n halfs, a
// multiple of kPackGroup.  Waits for it.
int    flashllm_hip_upload_packed(void* stream, void* dst, const void* src, size_t n, void* stage);
size_t flashllm_hip_upload_stage(size_t n);

// Copies ordinary host memory to the GPU and waits for it.
int flashllm_hip_upload(void* stream, void* dst, const void* src, size_t bytes);

// Waits for the stream, then *status = the FLASHLLM_ENCODE_* bits the encoder has recorded on the current device
// since they were last read, and clears them.
int flashllm_hip_encode_status(void* stream, unsigned int* status);

#ifdef __cplusplus
}
#endif
#endif
