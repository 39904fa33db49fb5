// Tiled-CSL compression on the GPU, for weights that are already device-resident.
//
// Produces the bytes of the reference's host-side InitSparseMatrixA_API
// (csrc/SpMM_API.cu:163-360).  Its per-tile procedure is sequential (bucket the
// nonzeros by LDS bank, pad, then pop the fullest bank item by item,
// csrc/SpMM_API.cu:248-346), but its result has a closed form that every item
// can evaluate on its own:
//
//   * An item's height h in its bank is 1 + the number of nonzeros before it in
//     the bank's scan order (row-major over the tile; a bank owns two adjacent
//     columns of every row).  Padding items sit on top.
//   * "Pop the fullest bank, lowest index on ties" removes items in order of
//     (height descending, bank ascending), so the item (bank b, height h) is
//     pop number  j = sum_b' max(fill[b'] - h, 0) + #{b' < b : fill[b'] >= h}.
//   * The drain's tail-then-main fill and its last-in-first-out write-out
//     (csrc/SpMM_API.cu:306-346) map j to one output index.
//
// Three kernels: vectors per tile, an in-place prefix sum (TileOffsets), the encoder.
//
// The path has to read A twice (the caller allocates Compressed_A between the two passes) and to write Compressed_A
// once: 1.2 GB at 27648 x 9216 and 80 %, HBM-bound when every access is a whole line.  So the count reads 1 KB of a
// row per load, and the encoder sorts a tile into output order in LDS and stores it as consecutive 16-byte vectors:
// with every item storing its own 4 bytes at its destination (a line of its own per lane) and one wave counting 128-byte
// pieces of eight rows at a time the call took 550 us; as it is now 222 (count 76, encoder 122, i.e. 6.7 and 5.9 TB/s).  About 25 us are a fixed cost: launches, the prefix sum
// and the host's wait for its total, which the kernel stores to host memory itself (2048 x 4096: 35.8 us; 44.1 with a copy
// of it).  Encoding the tiles last counted first, while they may still be in the Infinity Cache, gains nothing (27648 x
// 9216: 122 us either way, with cached loads in either kernel or both too).
#include "spmm_launch.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

namespace {

constexpr int kTileRows = 128;
constexpr int kTileCols = 64;
constexpr int kBanks    = 32;
constexpr int kLanes    = 64;
constexpr int kMaxFill  = kTileRows * kTileCols / kBanks + 3;  // 256 positions of a tile map to one bank; at most three padding items

// What the encoder found wrong since the word was last read (FLASHLLM_ENCODE_* bits), one word per GPU.  The host
// compressor returns an error in these cases; a kernel cannot, so it records them here and carries on.
__device__ unsigned int g_encode_status;

__device__ __forceinline__ void report(unsigned int what)
{
    atomicOr(&g_encode_status, what);
}

// |x| > 0 in the reference's float compare (csrc/SpMM_API.cu:183: drops +0, -0 and NaN) of both halfs of a word at
// once, as bits 0 and 16
__device__ __forceinline__ uint32_t keeps_pair(uint32_t w)
{
    using ushort2v          = uint16_t __attribute__((ext_vector_type(2)));
    const ushort2v below    = __builtin_bit_cast(ushort2v, w & 0x7fff7fffu) - ushort2v{1, 1};  // +-0 becomes 0xffff
    const ushort2v distance = __builtin_elementwise_sub_sat(ushort2v{0x7c00, 0x7c00}, below);  // 0 for +-0 and NaN
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(distance, ushort2v{1, 1}));
}

// The kernels here read and write each line once: non-temporal loads and stores, but for the loads of the scan-order encoder.
using uintx4 = uint32_t __attribute__((ext_vector_type(4)));

// Reductions over the 32 lanes of each half wave, the result in all of them: rotations inside the rows of sixteen
// lanes, then the other row of the half.
template<int CTRL>
__device__ __forceinline__ int dpp(int x)
{
    return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, true);
}

template<typename F>
__device__ __forceinline__ int over_half_wave(int x, F&& f)
{
    x = f(x, dpp<0x128>(x));  // row_ror:8, 4, 2, 1
    x = f(x, dpp<0x124>(x));
    x = f(x, dpp<0x122>(x));
    x = f(x, dpp<0x121>(x));
    return f(x, __builtin_amdgcn_ds_swizzle(x, 0x401f));  // lane ^ 16
}

__device__ __forceinline__ int half_sum(int x)
{
    return over_half_wave(x, [](int a, int b) { return a + b; });
}
__device__ __forceinline__ int half_min(int x)
{
    return over_half_wave(x, [](int a, int b) { return a < b ? a : b; });
}
__device__ __forceinline__ int half_max(int x)
{
    return over_half_wave(x, [](int a, int b) { return a > b ? a : b; });
}

__device__ __forceinline__ const uint16_t* tile_base(const uint16_t* a, int k, int tiles_per_row, int t)
{
    const int ti = t / tiles_per_row, tj = t % tiles_per_row;
    return a + static_cast<size_t>(ti) * kTileRows * k + static_cast<size_t>(tj) * kTileCols;
}

__device__ __forceinline__ int keeps_count(const uintx4 (&v)[16])
{
    uint32_t both = 0;
#pragma unroll
    for (int i = 0; i < 16; i++)  // at most 64 per half: the two counts do not meet
        both += keeps_pair(v[i][0]) + keeps_pair(v[i][1]) + keeps_pair(v[i][2]) + keeps_pair(v[i][3]);
    return static_cast<int>((both & 0xffffu) + (both >> 16));
}

// A wave counts a tile on its own, eight rows of 128 bytes per load: for matrices of at most 4096 tiles, where the latency of
// a workgroup counts and not how much of a row a load takes.  With the prefix sum, this way / by whole rows of eight tiles:
// 1024 x 1024 6.5 / 7.5 us, 1152 x 1088 (17 tiles in a row: the last row piece is one tile) 6.5 / 11.6, 2048 x 8192 8.2 /
// 11.2, 4096 x 8192 16.1 / 17.3; 7168 x 7168 22.1 / 21.7, 27648 x 9216 102 / 82.
constexpr int kCountAlone = 4096;

__global__ __launch_bounds__(kLanes) void count_tile_kernel(const uint16_t* __restrict__ a, int k, int tiles_per_row, int* __restrict__ offs)
{
    const int       lane = threadIdx.x;
    const uint16_t* base = tile_base(a, k, tiles_per_row, blockIdx.x) + static_cast<size_t>(lane >> 3) * k + (lane & 7) * 8;
    uintx4          v[16];
#pragma unroll
    for (int i = 0; i < 16; i++)
        v[i] = *reinterpret_cast<const uintx4*>(base + static_cast<size_t>(i) * 8 * k);
    int n = keeps_count(v);
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1)
        n += __shfl_xor(n, s);
    if (lane == 0)
        offs[blockIdx.x + 1] = (n + 3) / 4;
}

// offs[t + 1] = 16-byte vectors of tile t (nonzeros rounded up to a multiple of four, over four).
// A workgroup counts eight tiles side by side: a load takes 1 KB of a row (eight lanes per tile), wave w the rows
// 16w .. 16w + 15, all of them in flight at once.
constexpr int kCountWaves = 8;
constexpr int kCountTiles = kLanes * 8 / kTileCols;

__global__ __launch_bounds__(kLanes* kCountWaves) void count_tiles_kernel(
    const uint16_t* __restrict__ a, int k, int tiles_per_row, int strips, int* __restrict__ offs)
{
    constexpr int  kRows = kTileRows / kCountWaves;
    __shared__ int part[kCountWaves][kCountTiles];
    const int      lane  = threadIdx.x & (kLanes - 1), wave = threadIdx.x / kLanes;
    const int      ti    = blockIdx.x / strips, strip = blockIdx.x % strips;
    const int      tj    = strip * kCountTiles + lane / 8;  // this lane's tile
    int            n     = 0;
    if (tj < tiles_per_row) {
        const uint16_t* base = a + (static_cast<size_t>(ti) * kTileRows + wave * kRows) * k + static_cast<size_t>(strip) * (kLanes * 8) + lane * 8;
        uintx4          v[kRows];
#pragma unroll
        for (int i = 0; i < kRows; i++)
            v[i] = __builtin_nontemporal_load(reinterpret_cast<const uintx4*>(base + static_cast<size_t>(i) * k));
        n = keeps_count(v);
    }
#pragma unroll
    for (int s = 4; s >= 1; s >>= 1)
        n += __shfl_xor(n, s);
    if ((lane & 7) == 0)
        part[wave][lane / 8] = n;
    __syncthreads();
    const int t = strip * kCountTiles + threadIdx.x;
    if (threadIdx.x < kCountTiles && t < tiles_per_row) {
        int sum = 0;
#pragma unroll
        for (int w = 0; w < kCountWaves; w++)
            sum += part[w][threadIdx.x];
        offs[static_cast<size_t>(ti) * tiles_per_row + t + 1] = (sum + 3) / 4;
    }
}

// in place: offs[0] = 0, offs[t + 1] = sum of the counts up to tile t, offs[tiles + 1] = offs[tiles].
// One workgroup, latency-bound: up to 16 x 1024 counts are loaded in one round trip (wave w a contiguous run, 64 at a
// time), scanned across lanes with DPP and across waves in LDS.
constexpr int kScanWaves = 16;
constexpr int kScanRuns  = 16;

__device__ __forceinline__ int wave_scan(int x)  // inclusive
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1, 2, 4, 8
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
    return x;
}

// vectors: where the host reads the sum of all counts (host memory), or null.
__global__ __launch_bounds__(kLanes* kScanWaves) void scan_offsets_kernel(int* __restrict__ offs, int tiles, int* vectors)
{
    __shared__ int total[kScanWaves];
    const int      lane  = threadIdx.x & (kLanes - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    int            carry = 0;
    for (int first = 0; first < tiles;) {
        const int left = tiles - first, most = (left - 1) / (kLanes * kScanWaves) + 1;
        const int runs = most < kScanRuns ? most : kScanRuns;
        const int mine = wave * runs * kLanes + lane;  // counted from `first`
        int       x[kScanRuns];
#pragma unroll
        for (int r = 0; r < kScanRuns; r++) {
            x[r] = 0;
            if (r < runs && mine + r * kLanes < left)
                x[r] = offs[first + mine + r * kLanes + 1];
        }
        int sum = 0;
#pragma unroll
        for (int r = 0; r < kScanRuns; r++) {
            x[r] = wave_scan(x[r]) + sum;
            sum  = __builtin_amdgcn_readlane(x[r], kLanes - 1);
        }
        if (lane == 0)
            total[wave] = sum;
        __syncthreads();
        int before = carry;
#pragma unroll
        for (int w = 0; w < kScanWaves; w++) {
            const int s = total[w];
            before += w < wave ? s : 0;
            carry += s;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kScanRuns; r++)
            if (r < runs && mine + r * kLanes < left)
                offs[first + mine + r * kLanes + 1] = x[r] + before;
        first += left < runs * kLanes * kScanWaves ? left : runs * kLanes * kScanWaves;
    }
    if (threadIdx.x == 0) {
        offs[0]         = 0;
        offs[tiles + 1] = carry;
        if (vectors)
            __hip_atomic_store(vectors, carry, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// the reference's compare, as above, of one half of a word: finite or infinite and no zero.  By class, with the classes out of the
// compiler's sight, which makes an ordered compare with zero of them and then, under a ballot, one that NaN passes.
__device__ __forceinline__ bool keeps_half(uint32_t word, int half)
{
    using half2v = _Float16 __attribute__((ext_vector_type(2)));
    int classes  = 0x39c;
    asm("" : "+s"(classes));
    return __builtin_amdgcn_classh(__builtin_bit_cast(half2v, word)[half], classes);
}

__device__ __forceinline__ uint32_t lds_address(const void* p)
{
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)(p)));
}

// Four items to LDS, each at `at` in the lanes of its mask, which step on by STEP bytes: two vector instructions an item, where a branch
// on a lane's own bit takes five.  For whole waves.  lds_done() waits for these stores, which the compiler does not count.
template<int STEP>
__device__ __forceinline__ void store_and_step(uint32_t& at, const uint32_t (&item)[4], const uint64_t (&mask)[4])
{
    asm volatile("s_mov_b64 exec, %5\n\tds_write_b32 %0, %1\n\tv_add_u32_e32 %0, %9, %0\n\t"
                 "s_mov_b64 exec, %6\n\tds_write_b32 %0, %2\n\tv_add_u32_e32 %0, %9, %0\n\t"
                 "s_mov_b64 exec, %7\n\tds_write_b32 %0, %3\n\tv_add_u32_e32 %0, %9, %0\n\t"
                 "s_mov_b64 exec, %8\n\tds_write_b32 %0, %4\n\tv_add_u32_e32 %0, %9, %0\n\t"
                 "s_mov_b64 exec, -1"
                 : "+v"(at)
                 : "v"(item[0]), "v"(item[1]), "v"(item[2]), "v"(item[3]), "s"(mask[0]), "s"(mask[1]), "s"(mask[2]), "s"(mask[3]), "n"(STEP)
                 : "memory");
}

__device__ __forceinline__ void store_where(uint32_t at, uint32_t item, uint64_t mask)
{
    asm volatile("s_mov_b64 exec, %2\n\tds_write_b32 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(at), "v"(item), "s"(mask) : "memory");
}

__device__ __forceinline__ uint32_t min_pair(uint32_t a, uint32_t b)
{
    using ushort2v = uint16_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(ushort2v, a), __builtin_bit_cast(ushort2v, b)));
}

__device__ __forceinline__ void lds_done()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// The encoder: one workgroup of four waves per tile.
//
// Element (m, n) lives at swizzled column sw = n ^ ((m % 8) << 3) (csrc/SpMM_API.cu:252-256); bank sw / 2 owns the word
// sw / 2 of every swizzled row.  Thread (bank, segment) loads its bank's words of rows 16*segment .. +15 (32 lanes take
// one 128-byte line), i.e. 32 elements of the bank in scan order, and keeps them in registers.  Then
//   1. counts of all (bank, segment) meet in LDS: fills, heights, padding (every wave works it out for itself);
//   2. every thread lists its nonzeros by (height, bank) in LDS;
//   3. level by level: an item of the level is pop number  (items on higher levels) + (banks before it that reach the
//      level), a sum over the banks and a ballot over the half wave that holds the level; the items move to that place, through
//      registers because the list and the pops share their LDS;
//   4. vector v of the tile gathers its four items, which lie 32 pops apart, and is stored whole.
// Every element passes through a dozen vector instructions, and those, not memory, were the bound (685 per wave, the units busy all of
// the time; scalar ones 335): now a compare per half, whose mask the store goes by, two more instructions for the store itself, the sums of
// all levels at once in 16 lanes, row addresses in scalar registers; 493 and 349.  27648 x 9216, 80 %: 133.8 -> 121.7 us (5.9 TB/s;
// without its stores 104), 90 % 120 -> 106, 70 % 149 -> 142, 7168 x 7168 32.2 -> 28.9.  Seven or eight workgroups per CU instead of six,
// with fewer masks held: 3 % faster at 90 %, 4 to 7 % slower at 70 %.
// The list holds 128 levels (16 KB; the registers, 75, allow six workgroups per CU).  A tile in which a bank holds more
// (beyond about 45 % of all its elements) takes each item's pop number from a table of the levels instead, and the list in
// two parts: the pops that fit, up to the end of a pass of four, then the rest.  27648 x 9216, both calls: 320 us at 50 %
// and 366 at 20 % sparsity (589 and 818 when every nonzero stored itself to its place in memory; 244 at 70 %).
constexpr int kEncodeThreads = 256;
constexpr int kFarColumns    = 1 << 26;  // FAR: from here on; the other half of a wave is 16 rows on, 32 * k bytes, less than 2^31 for fewer
constexpr int kSegments      = kEncodeThreads / kBanks;
constexpr int kRowsOfThread  = kTileRows / kSegments;
constexpr int kLevels        = 128;
constexpr int kLevelsAtOnce  = kEncodeThreads / kBanks;

template<bool FAR>
__global__ __launch_bounds__(kEncodeThreads, 6) void encode_tiles_kernel(const uint16_t* __restrict__ a,
                                                                       int k,
                                                                       int tiles_per_row,
                                                                       const int* __restrict__ offs,
                                                                       uint32_t* __restrict__ out)
{
    __shared__ uint32_t list[kLevels * kBanks];            // [height - 1][bank]; then the pops in order
    __shared__ __attribute__((aligned(8))) uint8_t count_s[kBanks][kSegments];
    __shared__ __attribute__((aligned(16))) uint16_t fill_s[kBanks];
    __shared__ uint2 level[kMaxFill + 1];                  // only for tiles beyond the list: items higher than h, over all banks; banks holding at least h

    const int       t    = blockIdx.x;
    const int       tid  = threadIdx.x;
    const int       bank = tid & (kBanks - 1), segment = tid / kBanks;

    uint32_t word[kRowsOfThread];
    if constexpr (!FAR) {  // an offset of 32 bits from an address of the wave's, one vector instruction a row instead of three
        const uint16_t* base = tile_base(a, k, tiles_per_row, t) + static_cast<size_t>(__builtin_amdgcn_readfirstlane(tid / kLanes)) * (2 * kRowsOfThread) * k;
        const uint32_t  from = (tid & 32) * static_cast<uint32_t>(k);
#pragma unroll
        for (int i = 0; i < kRowsOfThread; i++)
            word[i] = __builtin_nontemporal_load(
                reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(base + static_cast<size_t>(i) * k) + (from + ((bank * 4u) ^ ((i & 7) * 16u)))));
    }
    else {
        const uint16_t* base = tile_base(a, k, tiles_per_row, t) + static_cast<size_t>(segment) * kRowsOfThread * k;
#pragma unroll
        for (int i = 0; i < kRowsOfThread; i++)
            word[i] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(base + static_cast<size_t>(i) * k + (((bank >> 2) ^ (i & 7)) * 4 + (bank & 3)) * 2));
    }
    const int first = offs[t], room = (offs[t + 1] - first) * 4;

    // The lanes that keep half e of row i.  There are scalar registers to hold those of six rows; the others are compared once more.
    constexpr int kHeldRows = 6;
    uint64_t      keeps[2 * kHeldRows];
    int           mine = 0;
#pragma unroll
    for (int i = 0; i < kRowsOfThread; i++) {
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const bool kept  = keeps_half(word[i], e);
            if (i < kHeldRows)
                keeps[2 * i + e] = __builtin_amdgcn_ballot_w64(kept);
            mine += kept;
        }
    }
    count_s[bank][segment] = static_cast<uint8_t>(mine);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kRowsOfThread; i++)
        asm volatile("" : "+v"(word[i]));  // compared again where the masks are wanted, not kept in spilled registers

    // this thread's bank: its fill (both halves of every wave hold all banks) and the items below this segment
    int         fill, below;
    const uint2 c = *reinterpret_cast<const uint2*>(&count_s[bank][0]);
    {
        const uint32_t low  = segment < 4 ? (1u << (8 * segment)) - 1u : 0xffffffffu;
        const uint32_t high = segment < 4 ? 0u : (1u << (8 * (segment - 4))) - 1u;
        fill  = static_cast<int>(__builtin_amdgcn_sad_u8(c.y, 0u, __builtin_amdgcn_sad_u8(c.x, 0u, 0u)));
        below = static_cast<int>(__builtin_amdgcn_sad_u8(c.y & high, 0u, __builtin_amdgcn_sad_u8(c.x & low, 0u, 0u)));
    }
    // Padding to a multiple of four: each padding item goes on top of the emptiest bank (lowest index on ties) at that
    // bank's first zero position, value 0 (csrc/SpMM_API.cu:274-287).
    const int unpadded = fill;
    const int nnz      = __builtin_amdgcn_readfirstlane(half_sum(fill));
    const int pad      = (4 - nnz % 4) % 4;
    for (int p = 0; p < pad; p++)
        fill += (half_min((fill << 5) | bank) & (kBanks - 1)) == bank;
    // The thread whose segment has that position puts the bank's padding items there.
    uint32_t pad_item = 0;
    bool     pads     = false;
    if (fill > unpadded) {
        const uint64_t full = (static_cast<uint64_t>(c.y) << 32 | c.x) ^ 0x0101010101010101ull * (2 * kRowsOfThread);
        if (full == 0) {  // cannot happen: the emptiest bank holds fewer than 256 items
            if (segment == 0)
                report(FLASHLLM_ENCODE_NO_ZERO);
        }
        else if (__builtin_ctzll(full) / 8 == segment) {
            pads       = true;
            int z      = 0;
#pragma unroll
            for (int i = 2 * kRowsOfThread - 1; i >= 0; i--)
                z = keeps_half(word[i / 2], i % 2) ? z : i;
            pad_item = static_cast<uint32_t>((segment * kRowsOfThread + (z >> 1)) * kTileCols + 2 * bank + (z & 1)) << 16;
        }
    }
#pragma unroll
    for (int i = 0; i < kRowsOfThread; i++)
        asm volatile("" : "+v"(word[i]));
    const int count = nnz + pad;
    const int top   = __builtin_amdgcn_readfirstlane(half_max(fill));

    const int vectors    = count >> 2;
    const int rep        = vectors >> 5, rem = vectors & (kBanks - 1);
    const int tail_items = rem * 4;
    uint32_t* out_tile   = out + static_cast<size_t>(first) * 4;
    // Never write outside this tile's range of Compressed_A, whatever TileOffsets says: with offsets that were
    // not computed from this very matrix the output is meaningless, but it stays inside the caller's buffer.
    const int space = count < room ? count : room;
    if (room != count && tid == 0)
        report(FLASHLLM_ENCODE_OFFSETS);
    // positions of the two halves of this thread's first row; a row further each is 64 more
    const uint32_t first_positions = static_cast<uint32_t>(segment * kRowsOfThread * kTileCols + 2 * bank) * 0x10001u + 0x10000u;
    auto           item_of         = [&](int i, int e, uint32_t positions) {
        return __builtin_amdgcn_perm(positions, word[i], e ? 0x07060302u : 0x05040100u);
    };

    // vector v out of the list, which holds the pops from `from` on
    auto store_vector = [&](int v, int from) {
        // a vector of the main part: pops of four passes, last pass first; of the tail (drained first): every rem-th
        const bool main = v < rep * kBanks;
        const int  step = main ? kBanks : rem;
        const int  last = (main ? tail_items + (rep - 1 - (v >> 5)) * (4 * kBanks) + (v & (kBanks - 1)) : v - rep * kBanks) - from;
        __builtin_nontemporal_store(uintx4{list[last + 3 * step], list[last + 2 * step], list[last + step], list[last]}, reinterpret_cast<uintx4*>(out_tile) + v);
    };

    if (top <= kLevels) {
        uint32_t       at        = lds_address(list) + (below * kBanks + bank) * 4;
        uint32_t       positions = first_positions;
#pragma unroll
        for (int i = 0; i < kRowsOfThread; i += 2) {
            uint32_t item[4];
            uint64_t mask[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                item[j] = item_of(i + j / 2, j % 2, positions + j / 2 * (kTileCols * 0x10001u));
                mask[j] = i < kHeldRows ? keeps[2 * (i % kHeldRows) + j] : __builtin_amdgcn_ballot_w64(keeps_half(word[i + j / 2], j % 2));
            }
            store_and_step<kBanks * 4>(at, item, mask);
            positions += 2 * kTileCols * 0x10001u;
        }
        if (tid < kBanks)
            fill_s[tid] = static_cast<uint16_t>(fill);
        if (pads)
            for (int h = unpadded; h < fill; h++)
                list[h * kBanks + bank] = pad_item;
        lds_done();
        __syncthreads();

        // Two levels at a time by the halves of a wave, 8i + 2w + 1 and + 2 in step i of wave w.  An item of a level comes after
        // those of the levels above it, which are all items but those up to this level.  Lane l of each sixteen works out how many
        // lie below step l's two levels, sum_b min(fill[b], 8l + 2w): eight banks to a lane, which go together in pairs and quarters.
        const int      wave  = __builtin_amdgcn_readfirstlane(tid / kLanes);
        const uint32_t half  = tid & 32 ? ~0u : 0u;
        const int      high  = fill + static_cast<int>(half);
        int            under = 0;
        {
            const uintx4   fills = *reinterpret_cast<const uintx4*>(&fill_s[(tid & (kLanes - 1)) / 16 * 8]);
            const uint32_t most  = ((tid & 15) * kLevelsAtOnce + 2 * wave) * 0x10001u;
            uint32_t       sum   = 0;  // two halfs of at most 4 * 128
#pragma unroll
            for (int j = 0; j < 4; j++)
                sum += min_pair(fills[j], most);
            under = static_cast<int>((sum & 0xffffu) + (sum >> 16));
            under += __builtin_amdgcn_ds_swizzle(under, 0x401f);  // lane ^ 16
        }
        uint32_t item[kLevels / kLevelsAtOnce];
        uint32_t pop[kLevels / kLevelsAtOnce];
        uint64_t here[kLevels / kLevelsAtOnce];
        uint64_t beyond = 0;
#pragma unroll
        for (int i = 0; i < kLevels / kLevelsAtOnce; i++) {
            here[i] = 0;
            if (i * kLevelsAtOnce < top) {
                item[i] = list[(i * kLevelsAtOnce + segment) * kBanks + bank];
                const int      lower = __builtin_amdgcn_readlane(under, i) + __builtin_amdgcn_readlane(under, 32 + i);
                const uint64_t have  = __builtin_amdgcn_ballot_w64(high > i * kLevelsAtOnce + 2 * wave);
                const uint32_t lo    = static_cast<uint32_t>(have), hi = static_cast<uint32_t>(have >> 32);
                // the upper half's lanes count those of the lower level as before them, and its own are not before them
                const uint32_t above = count - lower - __builtin_popcount(lo);
                const uint32_t base  = above - (half & __builtin_popcountll(have));
                pop[i]               = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, base));
                here[i]              = have & __builtin_amdgcn_ballot_w64(pop[i] < static_cast<uint32_t>(count));
                beyond |= have ^ here[i];
            }
        }
        if (beyond && tid % kLanes == 0)  // cannot happen while the closed form is right
            report(FLASHLLM_ENCODE_RANGE);
        __syncthreads();
        const uint32_t to = lds_address(list);
#pragma unroll
        for (int i = 0; i < kLevels / kLevelsAtOnce; i++)
            if (i * kLevelsAtOnce < top)
                store_where(to + pop[i] * 4, item[i], here[i]);
        lds_done();
        __syncthreads();
        for (int v = tid; v < space / 4; v += kEncodeThreads)
            store_vector(v, 0);
        return;
    }

    if (tid < kBanks)
        fill_s[bank] = static_cast<uint16_t>(fill);
    __syncthreads();
    for (int h = tid; h <= top; h += kEncodeThreads) {
        int      g = 0;
        uint32_t r = 0;
        for (int b = 0; b < kBanks; b++) {
            const int f = fill_s[b];
            g += f > h ? f - h : 0;
            r |= f >= h ? 1u << b : 0u;
        }
        level[h] = uint2{static_cast<uint32_t>(g), r};
    }
    // the pops up to the end of a pass of four (a pass of four is 32 whole vectors) that the list holds, and the rest
    const int fit   = (kLevels * kBanks - tail_items) / (4 * kBanks);
    const int early = rep < fit ? rep : fit;                       // passes of four in the first part
    const int split = tail_items + early * (4 * kBanks);
    bool beyond = false;
#pragma unroll 1
    for (int part = 0; part < (early < rep ? 2 : 1); part++) {
        const uint32_t from = part == 0 ? 0 : split, size = part == 0 ? split : count - split;
        auto           place = [&](int h, uint32_t item) {
            const uint2    l = level[h];
            const uint32_t j = l.x + __builtin_popcount(l.y & ((1u << bank) - 1u));
            beyond |= j >= static_cast<uint32_t>(count);
            if (j - from < size)
                list[j - from] = item;
        };
        __syncthreads();  // the table is complete / the first part is out of the list
        int      h         = below;
        uint32_t positions = first_positions;
        asm volatile("" : "+v"(positions));  // made here, not kept in registers for both parts; nor are the compares
#pragma unroll
        for (int i = 0; i < kRowsOfThread; i++)
            asm volatile("" : "+v"(word[i]));
#pragma unroll
        for (int i = 0; i < kRowsOfThread; i++) {
#pragma unroll
            for (int e = 0; e < 2; e++)
                if (keeps_half(word[i], e))
                    place(++h, item_of(i, e, positions));
            positions += kTileCols * 0x10001u;
        }
        if (pads)
            for (int p = unpadded; p < fill; p++)
                place(p + 1, pad_item);
        __syncthreads();
        // the first part ends the tile: the main part's last vectors (its passes are emitted last first) and the tail
        const int begin = part == 0 ? (rep - early) * kBanks : 0, end = part == 0 ? vectors : (rep - early) * kBanks;
        for (int v = begin + tid; v < end && v < space / 4; v += kEncodeThreads)
            store_vector(v, static_cast<int>(from));
    }
    if (beyond)  // cannot happen while the closed form is right
        report(FLASHLLM_ENCODE_RANGE);
}

// The encoder without reordering (csrc/SpMM_API.cu:363-489): a tile's items in scan order, row by row; the padding to a
// multiple of four takes the first zeros of the tile as they are (-0 and NaN among them), each in its place in the order.
// One workgroup of four waves per tile, half a row (64 bytes) to a thread: the items before it are the nonzeros before it, by
// a scan over the workgroup, and of the zeros before it at most as many as the tile is padded with.  The tile is put
// together in LDS and stored as consecutive 16-byte vectors.  32 KB of LDS, four workgroups per CU;
// bound by HBM like the encoder above (27648 x 9216 with the count 251 us, reordered 225; 36864 x 9216 326 and 292).
constexpr int kHalfRow = kTileCols / 2;

__global__ __launch_bounds__(kEncodeThreads) void encode_tiles_scan_kernel(const uint16_t* __restrict__ a,
                                                                         int k,
                                                                         int tiles_per_row,
                                                                         const int* __restrict__ offs,
                                                                         uint32_t* __restrict__ out)
{
    __shared__ __attribute__((aligned(16))) uint32_t list[kTileRows * kTileCols];
    __shared__ int total[kEncodeThreads / kLanes];
    const int       t    = blockIdx.x;
    const int       tid  = threadIdx.x, lane = tid & (kLanes - 1), wave = tid / kLanes;
    const int       row  = tid / 2, col = tid % 2 * kHalfRow;
    const uint16_t* base = tile_base(a, k, tiles_per_row, t) + static_cast<size_t>(row) * k + col;
    uint32_t        word[kHalfRow / 2];
#pragma unroll
    for (int i = 0; i < kHalfRow / 8; i++) {
        const uintx4 v = *reinterpret_cast<const uintx4*>(base + i * 8);
#pragma unroll
        for (int e = 0; e < 4; e++)
            word[4 * i + e] = v[e];
    }
    const int first = offs[t], room = (offs[t + 1] - first) * 4;

    int mine = 0;
#pragma unroll
    for (int i = 0; i < kHalfRow / 2; i++) {
        const uint32_t both = keeps_pair(word[i]);
        mine += static_cast<int>((both & 1u) + (both >> 16));
    }
    const int inclusive = wave_scan(mine);
    if (lane == kLanes - 1)
        total[wave] = inclusive;
    __syncthreads();
    int before = inclusive - mine, nnz = 0;
#pragma unroll
    for (int w = 0; w < kEncodeThreads / kLanes; w++) {
        before += w < wave ? total[w] : 0;
        nnz += total[w];
    }
    const int pad   = (4 - nnz % 4) % 4;
    const int count = nnz + pad;
    int       zeros = tid * kHalfRow - before;  // before this half row
    int       at    = before + (zeros < pad ? zeros : pad);
    if (room != count && tid == 0)
        report(FLASHLLM_ENCODE_OFFSETS);
    const uint32_t flip = static_cast<uint32_t>(row & 7) << 3, row_position = static_cast<uint32_t>(row * kTileCols);
#pragma unroll
    for (int i = 0; i < kHalfRow / 2; i++) {
        const uint32_t both = keeps_pair(word[i]);
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const bool     kept     = (both >> (16 * e)) & 1u;
            const uint32_t position = row_position + (static_cast<uint32_t>(col + 2 * i + e) ^ flip);
            if (kept || zeros < pad)
                list[at++] = ((word[i] >> (16 * e)) & 0xffffu) | (position << 16);
            zeros += kept ? 0 : 1;
        }
    }
    __syncthreads();
    // never outside this tile's range of Compressed_A, whatever TileOffsets says
    const int vectors = (count < room ? count : room) / 4;
    uintx4*   to      = reinterpret_cast<uintx4*>(out) + first;
    for (int v = tid; v < vectors; v += kEncodeThreads)
        __builtin_nontemporal_store(reinterpret_cast<const uintx4*>(list)[v], to + v);
}

// Packed pieces (spmm_launch.h) in pinned host memory -> the dense matrix.  One workgroup per group of 2048 halfs, a byte of the bits and
// eight halfs to a thread; the group's values come through LDS, so that what crosses the link is whole 16-byte vectors.  The kernel fetches
// them itself because the pieces lie a full piece apart (a copy would carry that) and 25 launches do for 7168 x 7168.  Bound by the
// link and the threads that pack: 27 of its 103 MB at 80 %, 0.92 ms; a launch for 32 pieces takes 26.5 us, i.e. 41 GB/s.
constexpr int kExpandThreads = kPackGroup / 8;

__global__ __launch_bounds__(kExpandThreads) void expand_kernel(const unsigned char* __restrict__ pieces, uintx4* __restrict__ dst)
{
    __shared__ uintx4 values[kExpandThreads + 1];
    __shared__ int    total[kExpandThreads / kLanes];
    constexpr int        kGroups = kPackPiece / kPackGroup;
    const int            tid = threadIdx.x, lane = tid & (kLanes - 1), wave = tid / kLanes;
    const unsigned char* piece = pieces + static_cast<size_t>(blockIdx.x / kGroups) * kPackStride;
    const int            group = blockIdx.x % kGroups;
    const uint32_t       first = reinterpret_cast<const uint32_t*>(piece)[group];
    const uint32_t       bits  = piece[kPackBits + group * (kPackGroup / 8) + tid];
    const int            mine = __builtin_popcount(bits), inclusive = wave_scan(mine);
    if (lane == kLanes - 1)
        total[wave] = inclusive;
    __syncthreads();
    int before = inclusive - mine, all = 0;
#pragma unroll
    for (int w = 0; w < kExpandThreads / kLanes; w++) {
        before += w < wave ? total[w] : 0;
        all += total[w];
    }
    const uint32_t skip    = first & 7;  // values in front of the group's in its first vector
    const int      vectors = (static_cast<int>(skip) + all + 7) / 8;
    const uintx4*  from    = reinterpret_cast<const uintx4*>(piece + kPackValues) + first / 8;
    if (tid < vectors)
        values[tid] = from[tid];
    if (tid == 0 && vectors > kExpandThreads)
        values[kExpandThreads] = from[kExpandThreads];
    __syncthreads();
    const uint16_t* at = reinterpret_cast<const uint16_t*>(values) + skip + before;
    uintx4          v;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const uint32_t lo = bits >> (2 * e) & 1, hi = bits >> (2 * e + 1) & 1;
        const uint32_t a = lo ? *at : 0;
        at += lo;
        const uint32_t b = hi ? *at : 0;
        at += hi;
        v[e] = a | b << 16;
    }
    dst[static_cast<size_t>(blockIdx.x) * kExpandThreads + tid] = v;
}

// The pinned memory is a ring of parts, each of them one launch: while the GPU fetches one part, the threads pack the ones after it.
// 7168 x 7168, 80 %, whole load, with 12 threads as long as there could be so many: 4 parts of 32 pieces 1.29 ms, 8 of 16 1.22, 16 of 16 1.22, 8 of 32 1.04; seven of 32
// stay below 32 MB, to which torch rounds up.
constexpr int kPartPieces = 32;
constexpr int kParts      = 7;

}  // namespace

extern "C" int flashllm_hip_launch_tile_offsets(void* stream, const void* a, int m, int k, int* offs, int* vectors)
{
    const int   tiles_per_row = k / kTileCols;
    const int   tiles         = (m / kTileRows) * tiles_per_row;
    hipStream_t s             = static_cast<hipStream_t>(stream);
    const int   strips        = (tiles_per_row - 1) / kCountTiles + 1;
    if (tiles <= kCountAlone)
        hipLaunchKernelGGL(count_tile_kernel, dim3(tiles), dim3(kLanes), 0, s, static_cast<const uint16_t*>(a), k, tiles_per_row, offs);
    else
        hipLaunchKernelGGL(count_tiles_kernel, dim3((m / kTileRows) * strips), dim3(kLanes * kCountWaves), 0, s, static_cast<const uint16_t*>(a),
                       k, tiles_per_row, strips, offs);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return static_cast<int>(e);
    hipLaunchKernelGGL(scan_offsets_kernel, dim3(1), dim3(kLanes * kScanWaves), 0, s, offs, tiles, vectors);
    return static_cast<int>(hipGetLastError());
}

// 28 GB/s from pageable memory: 7168 x 7168 in 3.6 ms.
extern "C" int flashllm_hip_upload(void* stream, void* dst, const void* src, size_t bytes)
{
    hipStream_t      s = static_cast<hipStream_t>(stream);
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
    return static_cast<int>(e == hipSuccess ? hipStreamSynchronize(s) : e);
}

extern "C" size_t flashllm_hip_upload_stage(size_t n)
{
    const size_t pieces = (n + kPackPiece - 1) / kPackPiece, most = static_cast<size_t>(kParts) * kPartPieces;
    return (pieces < most ? pieces : most) * kPackStride;
}

// The host's threads leave the zeros out (they read the matrix faster than the link carries it), and what is left crosses the link once,
// read by the kernel that expands it.  Only the calling thread talks to the runtime.
extern "C" int flashllm_hip_upload_packed(void* stream, void* dst, const void* src, size_t n, void* stage)
{
    hipStream_t  s      = static_cast<hipStream_t>(stream);
    const size_t pieces = (n + kPackPiece - 1) / kPackPiece, parts = (pieces + kPartPieces - 1) / kPartPieces;
    const auto*  from   = static_cast<const unsigned short*>(src);
    auto*        ring   = static_cast<unsigned char*>(stage);
    if (n == 0 || n % kPackGroup)
        return static_cast<int>(hipErrorInvalidValue);
    // where the GPU finds it: memory that was pinned after it was allocated may have another address there, and other memory has none
    void*      ring_there = nullptr;
    hipError_t e          = hipHostGetDevicePointer(&ring_there, stage, 0);
    if (e != hipSuccess)
        return static_cast<int>(e);
    hipEvent_t free_again[kParts];
    int        events = 0;
    while (events < kParts && (e = hipEventCreateWithFlags(&free_again[events], hipEventDisableTiming)) == hipSuccess)
        events++;

    std::atomic<size_t> next{0}, allowed{kParts};  // the next piece to pack; parts that have a place in the ring
    std::atomic<int>    packed[kParts];            // pieces of the part in that place that are ready
    std::atomic<bool>   stop{e != hipSuccess};
    for (auto& p : packed)
        p.store(0, std::memory_order_relaxed);
    auto pack_one = [&]() {  // false: nothing to do now
        size_t piece = next.load(std::memory_order_relaxed);
        do
            if (piece >= pieces || piece / kPartPieces >= allowed.load(std::memory_order_acquire))
                return false;
        while (!next.compare_exchange_weak(piece, piece + 1, std::memory_order_relaxed));
        const size_t first = piece * kPackPiece, slot = piece % (kParts * kPartPieces);
        flashllm_pack_piece(from + first, n - first < kPackPiece ? n - first : kPackPiece, ring + slot * kPackStride);
        packed[slot / kPartPieces].fetch_add(1, std::memory_order_release);
        return true;
    };
    // A thread that finds no place in the ring looks again for as long as the GPU usually takes over a part (40 us), then sleeps: the stream
    // may have other work before this (7168 x 7168 behind 320 ms of it took 2560 ms of the host's cores instead of 320, the wait's own).
    std::mutex              door;
    std::condition_variable place_free;
    auto                    pack_all = [&]() {
        int in_vain = 0;
        while (!stop.load(std::memory_order_relaxed) && next.load(std::memory_order_relaxed) < pieces)
            if (pack_one())
                in_vain = 0;
            else if (++in_vain < 500)
                std::this_thread::yield();
            else {
                std::unique_lock<std::mutex> lock(door);
                place_free.wait(lock, [&]() {
                    return stop.load(std::memory_order_relaxed) || next.load(std::memory_order_relaxed) / kPartPieces < allowed.load(std::memory_order_relaxed);
                });
                in_vain = 0;
            }
    };
    std::vector<std::thread> pool;
    try {  // a thread that cannot be created is left out
        // a thread for eight pieces (2048 x 2048 0.21 ms with 6 threads, 0.36 with 16), and at most eight: 16 took 4 % off 7168 x 7168 for twice the cores
        const int workers = flashllm_compress_workers(pieces / 8 < 8 ? pieces / 8 : 8);
        pool.reserve(workers);
        for (int w = 1; w < workers; w++)
            pool.emplace_back(pack_all);
    }
    catch (...) {
    }
    for (size_t p = 0; p < parts && e == hipSuccess; p++) {
        const size_t first = p * kPartPieces, count = pieces - first < kPartPieces ? pieces - first : kPartPieces;
        const int    place = static_cast<int>(p % kParts);
        while (packed[place].load(std::memory_order_acquire) < static_cast<int>(count))
            if (!pack_one())
                std::this_thread::yield();
        packed[place].store(0, std::memory_order_relaxed);
        const size_t start = first * kPackPiece, halfs = n - start < count * kPackPiece ? n - start : count * kPackPiece;
        hipLaunchKernelGGL(expand_kernel, dim3(static_cast<unsigned>(halfs / kPackGroup)), dim3(kExpandThreads), 0, s,
                           static_cast<const unsigned char*>(ring_there) + static_cast<size_t>(place) * kPartPieces * kPackStride,
                           static_cast<uintx4*>(dst) + start / 8);
        e = hipGetLastError();
        if (e == hipSuccess)
            e = hipEventRecord(free_again[place], s);
        if (e == hipSuccess && p + 2 >= kParts) {  // part p + 2 follows part p + 2 - kParts
            e = hipEventSynchronize(free_again[(p + 2) % kParts]);
            {
                const std::lock_guard<std::mutex> lock(door);
                allowed.store(p + 3, std::memory_order_release);
            }
            place_free.notify_all();
        }
    }
    {
        const std::lock_guard<std::mutex> lock(door);
        stop.store(true, std::memory_order_relaxed);
    }
    place_free.notify_all();
    for (auto& t : pool)
        t.join();
    const hipError_t done = hipStreamSynchronize(s);  // the ring is the caller's again
    for (int i = 0; i < events; i++)
        static_cast<void>(hipEventDestroy(free_again[i]));
    return static_cast<int>(e == hipSuccess ? done : e);
}

extern "C" int flashllm_hip_encode_status(void* stream, unsigned int* status)
{
    hipStream_t   s = static_cast<hipStream_t>(stream);
    unsigned int* word = nullptr;
    hipError_t    e = hipGetSymbolAddress(reinterpret_cast<void**>(&word), HIP_SYMBOL(g_encode_status));
    if (e == hipSuccess)
        e = hipStreamSynchronize(s);
    if (e == hipSuccess)
        e = hipMemcpy(status, word, sizeof(unsigned int), hipMemcpyDeviceToHost);
    const unsigned int zero = 0;
    if (e == hipSuccess && *status)
        e = hipMemcpy(word, &zero, sizeof(unsigned int), hipMemcpyHostToDevice);
    return static_cast<int>(e);
}

extern "C" int flashllm_hip_launch_encode(void* stream, const void* a, int m, int k, const int* offs, void* out)
{
    const int tiles_per_row = k / kTileCols;
    const int tiles         = (m / kTileRows) * tiles_per_row;
    hipLaunchKernelGGL(k < kFarColumns ? encode_tiles_kernel<false> : encode_tiles_kernel<true>,
                       dim3(tiles),
                       dim3(kEncodeThreads),
                       0,
                       static_cast<hipStream_t>(stream),
                       static_cast<const uint16_t*>(a),
                       k,
                       tiles_per_row,
                       offs,
                       static_cast<uint32_t*>(out));
    return static_cast<int>(hipGetLastError());
}

extern "C" int flashllm_hip_launch_encode_scan(void* stream, const void* a, int m, int k, const int* offs, void* out)
{
    const int tiles_per_row = k / kTileCols;
    const int tiles         = (m / kTileRows) * tiles_per_row;
    hipLaunchKernelGGL(encode_tiles_scan_kernel,
                       dim3(tiles),
                       dim3(kEncodeThreads),
                       0,
                       static_cast<hipStream_t>(stream),
                       static_cast<const uint16_t*>(a),
                       k,
                       tiles_per_row,
                       offs,
                       static_cast<uint32_t*>(out));
    return static_cast<int>(hipGetLastError());
}
