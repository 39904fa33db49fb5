// gfx950 kernels of the Flash-LLM hot path and their launch functions.
//
// spmm_stream_kernel: load-as-sparse / compute-as-dense, redesigned around a
// wave64 that works alone (the reference uses four cooperating 32-lane
// warps and two barriers per k tile, csrc/SpMM_Kernel.cuh:179-386):
//
//   * A wave owns one 128-row tile row of A, one K slice (or, with several
//     waves per slice, one run of its k tiles) and one group of output
//     columns.  The slice's packed nonzeros are one contiguous range
//     of Compressed_A (tiles of a tile row are stored back to back), so the
//     wave streams it as 1 KB chunks (64 lanes x 16 B, coalesced, aligned,
//     non-temporal) through a ring of DEPTH register slots that stays DEPTH
//     chunks ahead, whatever the tile boundaries are.
//   * Each chunk is scattered into the wave's private 128x64 fp16 tile in LDS
//     at the position stored in the item (the format's XOR-swizzled layout,
//     reference csrc/SpMM_API.cu:252-261).  When the running vector index
//     passes TileOffsets[t+1] the tile is complete: the wave takes it out of
//     LDS as 16 MFMA operands of 16 bytes per lane with ds_wrxchg2_rtn_b64,
//     which returns the operand and leaves zeros behind in one LDS instruction
//     (the swizzle makes every group of eight lanes hit 32 distinct banks), so
//     the tile is empty again for the next one without a separate clearing
//     pass, and issues v_mfma_f32_16x16x32_f16 against the B fragments of that
//     k tile (column-major B already is the MFMA operand layout: 8 consecutive
//     k per lane).  Any number of tiles may end inside one chunk (empty tiles,
//     tiles of a single vector).
//   * One wave, in-order LDS: no barrier in the loop over the tiles.
//   * Two, four or eight such waves form a workgroup where the launch leaves CUs short of waves: they divide the
//     slice along K and meet only at the end, to add their sums up in LDS (KS in the kernel's own comment).
//   * For N = 64 the same wave program runs eight to a workgroup, one row tile each over the same K slice, and
//     the workgroup stages B in LDS once for all eight (see the kernel's own comment); the waves meet at one
//     barrier per two k tiles and are otherwise as independent as before.
//
// Waiting for memory.  Every path through a ring stage issues exactly one
// ring load, so the compiler's wait before a slot is used is the exact
// vmcnt(DEPTH-1).  The B fragments of a k tile (column-major B already is the
// MFMA operand layout, 16 bytes per lane per fragment) are loaded straight
// into registers when the tile is opened and first used when it completes;
// the compiler places those waits as well.  Staging B through LDS instead
// (global_load_lds_dwordx4) measured the same at N <= 32 and slower at
// N = 64, where its 8 KB per wave cost two resident waves per CU.
// The operand exchanges are inline assembly (the compiler has no 16-byte LDS
// exchange) and carry their own lgkmcnt(0) inside the same statement.
//
// Placement.  The GPU has eight accelerator dies (XCDs), each with its own L2, and hands the
// workgroups of a launch to them round-robin in launch order: workgroup w runs on XCD w % 8.  The
// SpMM kernels therefore give the Split_K slices of one (row tile, column group) unit to workgroups
// eight apart, and each XCD a contiguous block of units: the partial sums of a unit all land in one L2.
//
// splitk_reduce_pages_kernel: the separate reduction (reference csrc/Reduction_Kernel.cuh:24-45) over
// slabs stored by workgroup (store_pages below), one workgroup per 128 x 16 block of C on the XCD that
// stored the block's pages, 16 bytes per lane per slice, eight slices in flight.  Where a workgroup runs
// only decides where its loads hit; the sums do not depend on it.
// splitk_reduce_kernel: the same sums over plain slabs (slab s = M*N halfs laid out like C), the
// reference's workspace layout.
#include "spmm_launch.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <type_traits>

namespace {

using half8   = _Float16 __attribute__((ext_vector_type(8)));
using half4   = _Float16 __attribute__((ext_vector_type(4)));
using floatx4 = float __attribute__((ext_vector_type(4)));
using uintx4  = uint32_t __attribute__((ext_vector_type(4)));

constexpr int kTileRows  = 128;
constexpr int kTileCols  = 64;
constexpr int kTileHalfs = kTileRows * kTileCols;
constexpr int kLanes     = 64;
constexpr int kNoTile    = 0x7fffffff;
constexpr int kXcds      = 8;  // accelerator dies of an MI355X, each with its own L2

// Workgroup w of a launch <-> (unit, part), part in [0, parts): the parts of one unit go to workgroups kXcds
// apart (one XCD under round-robin hand-out), XCD x takes the units x*per_xcd .. (x+1)*per_xcd-1 with
// per_xcd = units / kXcds:  w = ((unit % per_xcd)*parts + part)*kXcds + unit / per_xcd;  the units beyond a
// multiple of kXcds are laid out plainly behind them, w = unit*parts + part.
// The launches are three-dimensional grids (kXcds, parts, layers), whose workgroups the dispatcher hands out in
// the order x fastest, then y, then z, so that w = x + kXcds*(y + parts*z) and unit and part fall out of the
// workgroup's coordinates without a division: layer z < per_xcd holds unit x*per_xcd + z, part y.  One more
// layer holds the units beyond a multiple of kXcds (and a few workgroups that find nothing to do).
struct Place {
    int      unit, part;
    unsigned w;      // position in the launch order described above
    bool     valid;  // false: a workgroup of the last layer beyond the last unit
};

__device__ __forceinline__ Place place_of_workgroup(unsigned units, unsigned parts)
{
    const unsigned per_xcd = units / kXcds;
    Place          p;
    if (blockIdx.z < per_xcd) {
        p.unit  = static_cast<int>(blockIdx.x * per_xcd + blockIdx.z);
        p.part  = static_cast<int>(blockIdx.y);
        p.w     = blockIdx.x + kXcds * (blockIdx.y + parts * blockIdx.z);
        p.valid = true;
    }
    else {
        const unsigned i = blockIdx.x + kXcds * blockIdx.y;
        p.unit           = static_cast<int>(per_xcd * kXcds + i / parts);
        p.part           = static_cast<int>(i % parts);
        p.w              = per_xcd * kXcds * parts + i;
        p.valid          = static_cast<unsigned>(p.unit) < units;
    }
    return p;
}

inline dim3 grid_of(unsigned units, unsigned parts)
{
    return dim3(kXcds, parts, units / kXcds + (units % kXcds ? 1 : 0));
}

// Slab storage by workgroup ("pages").  A page is one 128-row x 16-column block of partial sums (4 KB; 128 x 8
// and 2 KB when N == 8), kept in the order the matrix cores leave it in registers: 16-byte piece
// q*(4*cols) + g*cols + r16 holds rows 32q + 4g .. +3 and 32q + 16 + 4g .. +3 of column r16.  Page b of
// workgroup w (its position in the launch order above) of a launch of G workgroups is page b*G + w of the workspace.  Under round-robin hand-out the
// XCD that writes and later sums a page is (page index) % 8 whenever G is a multiple of 8, whatever the shape
// of the product: a workspace shared by the linears of a layer keeps every line in one L2, where stores to
// lines already present stay readable for the reduction kernel (stores that miss go to memory and do not).
template<int NBLK>
__device__ __forceinline__ void store_pages(_Float16* ws, const floatx4 (&acc)[NBLK][8], int first_page, int N, int lane, unsigned w, unsigned launch)
{
    const int    cols  = N < 16 ? 8 : 16;
    const int    r16   = lane & 15, g = lane >> 4;
    const size_t pitch = static_cast<size_t>(launch) * (cols * 16);  // uint4 between consecutive pages of a workgroup
    uint4*       page  = reinterpret_cast<uint4*>(ws) + (static_cast<size_t>(first_page) * launch + w) * (cols * 16);
    if (r16 >= cols)
        return;
#pragma unroll
    for (int nb = 0; nb < NBLK; nb++) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            half8 h;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                h[e]     = static_cast<_Float16>(acc[nb][2 * q][e]);
                h[4 + e] = static_cast<_Float16>(acc[nb][2 * q + 1][e]);
            }
            page[nb * pitch + q * (4 * cols) + g * cols + r16] = __builtin_bit_cast(uint4, h);
        }
    }
}

// `store` here and in the kernels is how the launch stores its sums (kStorePlain, kStorePages, kStoreRelu: spmm_launch.h)
__device__ __forceinline__ half4 to_half4(const floatx4& x, int store)
{
    half4 h;
#pragma unroll
    for (int e = 0; e < 4; e++)
        h[e] = static_cast<_Float16>(store == kStoreRelu && !(x[e] > 0.f) ? 0.f : x[e]);  // NaN -> 0 like max(x, 0)
    return h;
}

// spmm_stream_kernel's 128 x 16*NBLK block of C, or of a plain slab: o is row 4*g of column 0.  The activation is a branch
// round the whole block: as a select in every conversion it cost the stores without it up to 0.8 us (36608 x 448, Split_K
// 1, one wave per slice: N = 64 17.8 -> 17.0, N = 8 11.1 -> 10.8).  The kernels for wide B are faster with the selects
// (the same weight, N = 128: 18.5 us, 18.8 with a branch).
template<int STORE, int NBLK>
__device__ __forceinline__ void store_block_as(_Float16* o, const floatx4 (&acc)[NBLK][8], int M, int N, int col0, int r16)
{
#pragma unroll
    for (int nb = 0; nb < NBLK; nb++) {
        const int n = col0 + nb * 16 + r16;
        if (n < N) {
#pragma unroll
            for (int rb = 0; rb < 8; rb++)
                *reinterpret_cast<half4*>(o + static_cast<size_t>(n) * M + rb * 16) = to_half4(acc[nb][rb], STORE);
        }
    }
}

template<int NBLK>
__device__ __forceinline__ void store_block(_Float16* o, const floatx4 (&acc)[NBLK][8], int M, int N, int col0, int r16, int store)
{
    if (store == kStoreRelu)
        store_block_as<kStoreRelu>(o, acc, M, N, col0, r16);
    else
        store_block_as<kStorePlain>(o, acc, M, N, col0, r16);
}

__device__ __forceinline__ void clear_tile(uint16_t* tile, int lane)
{
    const uint4 zero = {0u, 0u, 0u, 0u};
    uint4*      t    = reinterpret_cast<uint4*>(tile);
#pragma unroll
    for (int i = 0; i < kTileHalfs * 2 / 16 / kLanes; i++)
        t[i * kLanes + lane] = zero;
}

// low 16 bits: fp16 value; high 16 bits: position in the swizzled tile.
__device__ __forceinline__ void scatter_item(uint16_t* tile, uint32_t item)
{
    tile[(item >> 16) & (kTileHalfs - 1)] = static_cast<uint16_t>(item);
}

__device__ __forceinline__ void scatter_vector(uint16_t* tile, const uint4& v)
{
    scatter_item(tile, v.x);
    scatter_item(tile, v.y);
    scatter_item(tile, v.z);
    scatter_item(tile, v.w);
}

// streaming load of one 16-byte vector: the weights are read once, keep them out of the caches' way
__device__ __forceinline__ uint4 load_stream(const uint4* p)
{
    const uintx4 x = __builtin_nontemporal_load(reinterpret_cast<const uintx4*>(p));
    return uint4{x[0], x[1], x[2], x[3]};
}

__device__ __forceinline__ uint32_t lds_offset(const void* p)
{
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)(p)));
}

// Takes eight 16-byte operands out of LDS (one per 16-row block, at addr[0..7]) and leaves zeros behind:
// ds_wrxchg2_rtn_b64 returns the operand and stores the zeros in one LDS instruction.  The compiler does not
// track the LDS returns of inline assembly, so the exchanges and the wait for them sit in ONE statement, with
// early-clobber outputs: no register of a[] can be read, moved or spilled while its exchange is in flight.
using uintx2 = uint32_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void take_8_and_wait(uintx4 (&a)[8], const uint32_t (&addr)[8])
{
    const uintx2 zero = {0u, 0u};
    asm volatile(
        "ds_wrxchg2_rtn_b64 %0, %8, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %1, %9, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %2, %10, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %3, %11, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %4, %12, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %5, %13, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %6, %14, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %7, %15, %16, %16 offset1:1\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]), "=&v"(a[4]), "=&v"(a[5]), "=&v"(a[6]), "=&v"(a[7])
        : "v"(addr[0]), "v"(addr[1]), "v"(addr[2]), "v"(addr[3]), "v"(addr[4]), "v"(addr[5]), "v"(addr[6]), "v"(addr[7]), "v"(zero)
        : "memory");
}

// An operand by two exchanges that the compiler knows of: the products of the first row blocks run while the operands of the later ones are
// on their way.  For eight row tiles per workgroup (N = 64), whose waves are in step and would all exchange and then all multiply: 36864
// x 9216, Split_K 7, at 70, 80 and 90 % 89.3 -> 88.1, 72.4 -> 68.2 and 65.3 -> 60.7 us, 49152 x 12288, 5 142 -> 140, 116.9 -> 113.6 and 105.2 ->
// 96.8.  Waves that run freely fill each other's gaps, and lose by 16 more instructions per tile: 11392 x 18112, N = 64, Split_K 11 46.5
// and 48.0, 36864 x 9216, N = 16 52.3 and 53.8, 49152 x 12288, N = 32 93.7 and 95.8.  By loads and, behind them, stores of zeros the first
// took 75.4 at 80 % instead of 67.9, 9216 x 36864, N = 64, 90 % 70 instead of 66: 1 KB takes the LDS of a CU 5.7 ns to store, 5.4 to
// exchange and 1.8 to load.
__device__ __forceinline__ uintx4 take(uint32_t addr)
{
    using Half = __attribute__((address_space(3), may_alias)) uint64_t;
    const uint64_t lo = __hip_atomic_exchange(reinterpret_cast<Half*>(addr), uint64_t{0}, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    const uint64_t hi = __hip_atomic_exchange(reinterpret_cast<Half*>(addr + 8), uint64_t{0}, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    return uintx4{static_cast<uint32_t>(lo), static_cast<uint32_t>(lo >> 32), static_cast<uint32_t>(hi), static_cast<uint32_t>(hi >> 32)};
}

// Sixteen operands (both 32-wide k steps): all sixteen exchanges are issued back to back, then one wait.
// Two statements, because one statement takes at most thirty operands: the first issues eight exchanges,
// the second, directly behind it, the other eight and the wait, and carries the first eight as in/out
// operands so that they cannot be used before that wait.
__device__ __forceinline__ void take_16_and_wait(uintx4 (&a0)[8], uintx4 (&a1)[8], const uint32_t (&addr0)[8], const uint32_t (&addr1)[8])
{
    const uintx2 zero = {0u, 0u};
    asm volatile(
        "ds_wrxchg2_rtn_b64 %0, %8, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %1, %9, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %2, %10, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %3, %11, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %4, %12, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %5, %13, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %6, %14, %16, %16 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %7, %15, %16, %16 offset1:1"
        : "=&v"(a0[0]), "=&v"(a0[1]), "=&v"(a0[2]), "=&v"(a0[3]), "=&v"(a0[4]), "=&v"(a0[5]), "=&v"(a0[6]), "=&v"(a0[7])
        : "v"(addr0[0]), "v"(addr0[1]), "v"(addr0[2]), "v"(addr0[3]), "v"(addr0[4]), "v"(addr0[5]), "v"(addr0[6]), "v"(addr0[7]), "v"(zero)
        : "memory");
    asm volatile(
        "ds_wrxchg2_rtn_b64 %0, %16, %24, %24 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %1, %17, %24, %24 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %2, %18, %24, %24 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %3, %19, %24, %24 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %4, %20, %24, %24 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %5, %21, %24, %24 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %6, %22, %24, %24 offset1:1\n\t"
        "ds_wrxchg2_rtn_b64 %7, %23, %24, %24 offset1:1\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a1[0]), "=&v"(a1[1]), "=&v"(a1[2]), "=&v"(a1[3]), "=&v"(a1[4]), "=&v"(a1[5]), "=&v"(a1[6]), "=&v"(a1[7]),
          "+v"(a0[0]), "+v"(a0[1]), "+v"(a0[2]), "+v"(a0[3]), "+v"(a0[4]), "+v"(a0[5]), "+v"(a0[6]), "+v"(a0[7])
        : "v"(addr1[0]), "v"(addr1[1]), "v"(addr1[2]), "v"(addr1[3]), "v"(addr1[4]), "v"(addr1[5]), "v"(addr1[6]), "v"(addr1[7]), "v"(zero)
        : "memory");
}

// One 1 KB piece of B (eight columns x the 64 k of a k tile, i.e. eight whole 128-byte lines) from global memory
// straight into LDS, without passing through registers: lane l delivers its 16 bytes at lds + 16*l.  The wave's
// vector-memory counter counts it like any load; the compiler does not know of it.
__device__ __forceinline__ void load_to_lds_16(const void* src, uint32_t lds)
{
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %2\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, off\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved)
        : "v"(src), "s"(lds)
        : "memory");
}

// The same with the lanes' byte offsets from a common address.
__device__ __forceinline__ void load_to_lds_16(const void* base, uint32_t offset, uint32_t lds)
{
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %3\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %2\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved)
        : "v"(offset), "s"(base), "s"(lds)
        : "memory");
}

// The end of a workgroup whose KS waves share a slice: every wave leaves its accumulators in its own 16 KB of LDS
// (its tile, no longer needed; NB = 4 in two halves), then the waves divide the blocks of 32 rows x 16 columns among
// themselves, add the KS contributions to each in the order of k and store it like the one-wave form does.
template<int NB, int KS>
__device__ __forceinline__ void add_up_and_store(
    floatx4* lds, const floatx4 (&acc)[NB][8], _Float16* out, int store, int M, int N, int col0, int rowtile, int slice, int wave, int lane, unsigned w, unsigned launch)
{
    constexpr int kAtOnce  = NB < 2 ? NB : 2;             // column blocks whose sums fit the LDS of a wave at once
    constexpr int kPerWave = kTileHalfs * 2 / 16;         // 16-byte places per wave
    const int     cols = N < 16 ? 8 : 16, r16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int part = 0; part < NB / kAtOnce; part++) {
        if (part > 0)
            __syncthreads();
#pragma unroll
        for (int i = 0; i < kAtOnce; i++)
#pragma unroll
            for (int rb = 0; rb < 8; rb++)
                lds[wave * kPerWave + (i * 8 + rb) * kLanes + lane] = acc[part * kAtOnce + i][rb];
        __syncthreads();
        for (int u = wave; u < kAtOnce * 4; u += KS) {  // rows 32q .. +31 of column block nb
            const int i = u / 4, q = u % 4, nb = part * kAtOnce + i;
            floatx4   lo = lds[(i * 8 + 2 * q) * kLanes + lane], hi = lds[(i * 8 + 2 * q + 1) * kLanes + lane];
#pragma unroll
            for (int v = 1; v < KS; v++) {
                lo += lds[v * kPerWave + (i * 8 + 2 * q) * kLanes + lane];
                hi += lds[v * kPerWave + (i * 8 + 2 * q + 1) * kLanes + lane];
            }
            const half4 l = to_half4(lo, store), h = to_half4(hi, store);
            if (r16 >= cols)
                continue;
            if (store == kStorePages) {
                uint4* page = reinterpret_cast<uint4*>(out) + (static_cast<size_t>(nb) * launch + w) * (cols * 16);
                const uint2 a = __builtin_bit_cast(uint2, l), b = __builtin_bit_cast(uint2, h);
                page[q * (4 * cols) + g * cols + r16] = uint4{a.x, a.y, b.x, b.y};
            }
            else {
                _Float16* o = out + static_cast<size_t>(slice) * M * N + static_cast<size_t>(col0 + nb * 16 + r16) * M
                              + static_cast<size_t>(rowtile) * kTileRows + q * 32 + g * 4;
                *reinterpret_cast<half4*>(o)      = l;
                *reinterpret_cast<half4*>(o + 16) = h;
            }
        }
    }
}

// NB: 16-column blocks per wave (1 for N <= 16, 2 for N = 32, 4 for N >= 64).
// DEPTH: ring slots = 1 KB chunks in flight per wave.
// W: waves per workgroup that share B.  W == 1: every wave fetches its own B fragments from L2.
//
// W > 1 (N = 32 and 64, where the 2*NB fragment loads per tile and wave are what holds the one-wave form back):
// the W waves of a workgroup take the SAME K slice of W consecutive row tiles, so they need the same B, and B
// is staged in LDS once per workgroup, as the reference stages one B tile per thread block for all of its
// warps (csrc/MatMulUtilities.cuh:39-75).  Every wave keeps its private tile and its own stream and runs
// freely; the waves meet once per window of G k tiles:
//   * the window's B (G k tiles x 16*NB columns x 128 bytes) is fetched as whole 128-byte lines by
//     load_to_lds_16, each wave two of the window's 1 KB pieces; piece (l % 8) ^ (l / 8) of a line goes to
//     slot l % 8 of its column, so the operand reads below are free of bank conflicts;
//   * two windows of LDS alternate.  Before a wave reads the first fragment of window w it makes sure its own
//     pieces of w have landed (they were requested a whole window earlier: after DEPTH younger ring loads the
//     ring's own waits have already covered them, otherwise it drains) and meets the others at a barrier;
//     past the barrier everybody has finished reading window w-1, whose LDS then receives window w+1;
//   * a tile's fragments are 2*NB plain 16-byte LDS reads issued with the operand exchanges.
// A wave without nonzeros in the slice, or beyond the last row tile, still fetches its pieces and attends
// every barrier.
//
// KS: waves of a workgroup that share one (row tile, slice) (W == 1 only).  They take the slice's k tiles in KS
// consecutive runs, each with a tile and a stream of its own and without meeting, and at the end add their
// accumulators up in fp32 through LDS, in the order of k.  The slab they store is that of the whole slice: to the
// workspace and the reduction a workgroup of KS waves is a workgroup.
template<int NB, int DEPTH, int W, int G, int KS>
__global__ __launch_bounds__(kLanes* W* KS) void spmm_stream_kernel(const uint4* __restrict__ comp,
                                                                const int* __restrict__ offs,
                                                                const _Float16* __restrict__ B,
                                                                int ldb,
                                                                _Float16* __restrict__ out,
                                                                int M,
                                                                int N,
                                                                int K,
                                                                int split_k,
                                                                int col_groups,
                                                                int store,
                                                                unsigned units)
{
    constexpr int kBTile  = NB * 2048;                     // bytes of B per k tile in LDS: 16*NB columns x 128
    constexpr int kBBytes = W > 1 ? 2 * G * kBTile : 0;    // two windows
    constexpr int kPieces = W > 1 ? G * 2 * NB / W : 0;    // 1 KB pieces of a window each wave fetches
    static_assert(W == 1 || (G * 2 * NB) % W == 0, "the pieces of a window must divide among the waves");
    static_assert((G & (G - 1)) == 0, "G must be a power of two");
    static_assert(W == 1 || KS == 1, "waves share either B or a slice");
    // the windows of B first (the LDS address of a direct load travels in M0 and stays small), then the waves' tiles
    __shared__ __attribute__((aligned(16))) unsigned char lds[kBBytes + W * KS * kTileHalfs * 2];

    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = W * KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes) : 0;
    uint16_t* const tile = reinterpret_cast<uint16_t*>(lds + kBBytes) + wave * kTileHalfs;
    const int r16  = lane & 15;  // row inside a 16-row block / output column
    const int g    = lane >> 4;  // which 8-wide k chunk of a 32-wide k step
    const int kt   = K / kTileCols;
    // W == 1: unit = (row tile, column group), column group fastest: the column groups of a row tile read the
    // same weights and meet in one L2.  W > 1: unit = W consecutive row tiles, all 16*NB columns.
    const Place place = place_of_workgroup(units, split_k);
    if (!place.valid)
        return;
    const int  unit = place.unit, slice = place.part;
    const int  rowtile   = W > 1 ? unit * W + wave : unit / col_groups;
    const int  col0      = W > 1 ? 0 : (unit % col_groups) * (16 * NB);
    const bool have_rows = W == 1 || rowtile < M / kTileRows;
    // HW_ID.wave_id: which of the SIMD's wave slots this wave sits in (bit 0 tells the two apart)
    const int wave_slot = __builtin_amdgcn_s_getreg(4 | (0 << 6) | (3 << 11)) & 1;

    // the reference's slicing (csrc/SpMM_Kernel.cuh:196-204), clamped to K
    const int avg = (kt - 1) / split_k + 1;
    int       kb  = slice * avg;
    kb            = kb < kt ? kb : kt;
    int ke        = kb + avg;
    ke            = ke < kt ? ke : kt;
    if constexpr (KS > 1) {  // this wave's run of the slice's tiles
        const int tiles = ke - kb, base = kb;
        kb = base + tiles * wave / KS;
        ke = base + tiles * (wave + 1) / KS;
    }

    floatx4 acc[NB][8];
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
#pragma unroll
        for (int rb = 0; rb < 8; rb++)
            acc[nb][rb] = floatx4{0.f, 0.f, 0.f, 0.f};

    const int* toff = offs + static_cast<size_t>(have_rows ? rowtile : 0) * kt;
    const int  vbeg = toff[kb];
    const int  vend = have_rows ? toff[ke] : vbeg;

    // ---- the shared B windows (W > 1 only) ----
    const uint32_t bwin_lds = lds_offset(&lds[0]);
    int            since    = 0;  // ring loads this wave has issued since it last requested pieces of B
    // this wave's pieces of window w: piece j is k tile j / (2*NB) of the window, columns 8*(j % (2*NB)) .. +7
    auto fetch_window = [&](int w) {
#pragma unroll
        for (int i = 0; i < kPieces; i++) {
            const int j  = wave * kPieces + i;
            int       tk = kb + w * G + j / (2 * NB);
            tk           = tk < ke ? tk : ke - 1;  // past the slice's end: any valid lines, nobody reads them
            const int c  = 8 * (j % (2 * NB)) + (lane >> 3);
            load_to_lds_16(B + static_cast<size_t>(c) * ldb + tk * kTileCols + (((lane & 7) ^ (lane >> 3)) << 3),
                           bwin_lds + (w & 1) * (G * kBTile) + j * 1024);
        }
        since = 0;
    };
    // before the first read of window w
    auto open_window = [&](int w) {
        // At most DEPTH loads still in flight: with DEPTH ring loads younger than this wave's pieces of window w
        // those have landed (loads complete in order); the ring itself is rarely touched by this wait, a slot is
        // only refilled after the wait for its previous contents.  With fewer younger loads: drain.
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DEPTH) : "memory");
        if (since < DEPTH)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("s_barrier" ::: "memory");
        if (kb + (w + 1) * G < ke)
            fetch_window(w + 1);
    };
    if constexpr (W > 1) {
        if (kb < ke)
            fetch_window(0);
    }

    if (vend > vbeg) {
        // operand addresses: row r16 of a row block, 16-byte chunk (ks*4+g) ^ (row%8)
        const int       a_off0 = r16 * (kTileCols * 2) + ((g ^ (r16 & 7)) << 4);
        const int       a_off1 = a_off0 ^ 64;
        const _Float16* bptr[NB];
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
            int n    = col0 + nb * 16 + r16;
            n        = n < N ? n : N - 1;  // N == 8: lanes 8..15 compute columns nobody stores
            bptr[nb] = B + static_cast<size_t>(n) * ldb + g * 8;
        }
        const uint32_t tile_lds = lds_offset(tile);
        uint32_t       a_addr0[8], a_addr1[8];  // LDS byte addresses of this lane's operands: k step 0 / 1 of row block rb
#pragma unroll
        for (int rb = 0; rb < 8; rb++) {
            a_addr0[rb] = tile_lds + rb * (16 * kTileCols * 2) + a_off0;
            a_addr1[rb] = tile_lds + rb * (16 * kTileCols * 2) + a_off1;
        }
        half8          bfrag[2][NB];  // B fragments of the open tile (W == 1) / of the tile being multiplied
        auto           load_b = [&](int t) {
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int nb = 0; nb < NB; nb++)
                    bfrag[ks][nb] = *reinterpret_cast<const half8*>(bptr[nb] + t * kTileCols + ks * 32);
        };
        // W > 1: the fragments of k step ks of tile t out of its window: column 16*nb + r16 holds piece
        // (4*ks + g) at slot (4*ks + g) ^ (r16 % 8), the same offsets as an operand of A inside a row block
        auto read_b = [&](int t, int ks) {
            const int            i    = t - kb;
            const unsigned char* base = lds + ((i / G) & 1) * (G * kBTile) + (i % G) * kBTile + (ks ? a_off1 : a_off0);
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
                bfrag[ks][nb] = *reinterpret_cast<const half8*>(base + nb * 2048);
        };

        clear_tile(tile, lane);

        const int cbase   = vbeg & ~(kLanes - 1);
        const int nchunks = (vend - cbase + kLanes - 1) / kLanes;
        const int vlast   = vend - 1;
        uint4     ring[DEPTH];
#pragma unroll
        for (int d = 0; d < DEPTH; d++)
            ring[d] = uint4{0u, 0u, 0u, 0u};

        int t = kb, tile_lo = vbeg, tile_hi = toff[kb + 1], next_hi = toff[kb + 2];
        if constexpr (W == 1)
            load_b(t);

        // Chunks -DEPTH .. -1 only fill the ring: none of their lanes reaches tile_lo, and a tile can
        // only "end" there when it is empty.
        for (int c0 = -DEPTH; c0 < nchunks; c0 += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; d++) {
                const int v  = cbase + (c0 + d) * kLanes + lane;  // this lane's vector
                const int ve = cbase + (c0 + d + 1) * kLanes;     // end of the chunk
                {
                    const uint4 cur = ring[d];
                    if (v >= tile_lo && v < tile_hi)
                        scatter_vector(tile, cur);
                    while (tile_hi <= ve) {  // a tile ends inside, or exactly at the end of, this chunk
                        if constexpr (W > 1) {
                            if (((t - kb) & (G - 1)) == 0)
                                open_window((t - kb) / G);
                        }
                        if (tile_hi > tile_lo) {
                            // NB <= 2: all 16 operands in one batch.  NB == 4: one 32-wide k step at a time, which
                            // keeps the kernel within 256 VGPRs (two waves per SIMD).
                            if constexpr (NB >= 4) {
                                if constexpr (W > 1)
                                    asm volatile("" ::: "memory");  // the items are in the tile
#pragma unroll
                                for (int ks = 0; ks < 2; ks++) {
                                    uintx4 a[8];
                                    if constexpr (W > 1) {
                                        read_b(t, ks);
#pragma unroll
                                        for (int rb = 0; rb < 8; rb++)
                                            a[rb] = take((ks ? a_addr1 : a_addr0)[rb]);
                                    }
                                    else
                                        take_8_and_wait(a, ks ? a_addr1 : a_addr0);
#pragma unroll
                                    for (int rb = 0; rb < 8; rb++)
#pragma unroll
                                        for (int nb = 0; nb < NB; nb++)
                                            acc[nb][rb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                                __builtin_bit_cast(half8, a[rb]), bfrag[ks][nb], acc[nb][rb], 0, 0, 0);
                                    // This wave's reads of the window have ended here, before the barrier that gives its LDS to other
                                    // loads: products that use them could sink below that barrier, and their wait with them.
                                    if constexpr (W > 1)
#pragma unroll
                                        for (int nb = 0; nb < NB; nb++)
                                            asm volatile("" ::"v"(bfrag[ks][nb]));
                                }
                                if constexpr (W > 1)
                                    asm volatile("" ::: "memory");  // the next tile's come after
                            }
                            else {
                                uintx4 a0[8], a1[8];
                                if constexpr (W > 1) {
                                    read_b(t, 0);
                                    read_b(t, 1);
                                }
                                take_16_and_wait(a0, a1, a_addr0, a_addr1);
#pragma unroll
                                for (int rb = 0; rb < 8; rb++)
#pragma unroll
                                    for (int nb = 0; nb < NB; nb++)
                                        acc[nb][rb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                            __builtin_bit_cast(half8, a0[rb]), bfrag[0][nb], acc[nb][rb], 0, 0, 0);
#pragma unroll
                                for (int rb = 0; rb < 8; rb++)
#pragma unroll
                                    for (int nb = 0; nb < NB; nb++)
                                        acc[nb][rb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                            __builtin_bit_cast(half8, a1[rb]), bfrag[1][nb], acc[nb][rb], 0, 0, 0);
                            }
                        }
                        t++;
                        tile_lo = tile_hi;
                        // The SIMD's arbiter serves its older wave first, which leaves the younger of the two
                        // resident waves about 17 % slower; taking turns at raised priority, one tile each,
                        // evens their finishing times.  The tile counters of the two waves are not in step:
                        // the younger wave's raised level is the higher one, so it wins when both are raised
                        // as the older one wins when neither is.
                        if ((t ^ wave_slot) & 1) {
                            if (wave_slot)
                                __builtin_amdgcn_s_setprio(2);
                            else
                                __builtin_amdgcn_s_setprio(1);
                        }
                        else
                            __builtin_amdgcn_s_setprio(0);
                        if (t < ke) {
                            if constexpr (W == 1)
                                load_b(t);
                            tile_hi = next_hi;
                            next_hi = toff[t + 2];
                            if (v >= tile_lo && v < tile_hi)  // the rest of this chunk opens the next tile
                                scatter_vector(tile, cur);
                        }
                        else {  // nothing left: the remaining stages are no-ops
                            tile_lo = kNoTile;
                            tile_hi = kNoTile;
                        }
                    }
                }
                {
                    int vn  = v + DEPTH * kLanes;
                    vn      = vn < vlast ? vn : vlast;
                    ring[d] = load_stream(comp + vn);
                    if constexpr (W > 1)
                        since++;
                }
            }
        }
    }
    else if constexpr (W > 1) {
        // nothing to multiply: this wave's part in the windows remains
        for (int w = 0; w * G < ke - kb; w++)
            open_window(w);
    }

    if (!have_rows)
        return;
    if constexpr (KS > 1) {
        add_up_and_store<NB, KS>(reinterpret_cast<floatx4*>(lds), acc, out, store, M, N, col0, rowtile, slice, wave, lane, place.w, units * split_k);
        return;
    }
    // D layout of the 16x16 MFMA: lane holds column r16, rows 4*g .. 4*g+3 of each 16-row block.
    if (store == kStorePages) {  // a workgroup's pages: wave by wave, NB each
        store_pages<NB>(out, acc, wave * NB, N, lane, place.w, units * split_k);
        return;
    }
    store_block(out + static_cast<size_t>(slice) * M * N + static_cast<size_t>(rowtile) * kTileRows + g * 4, acc, M, N, col0, r16, store);
}

// ------------------------------------------------------------------------------------------------
// spmm_group_kernel: the kernel for wide B (N a multiple of 128).  The one-wave kernel above pays the whole
// cost of a tile (scatter, take it out of LDS, clear it) once per 64 output columns; here four waves share it,
// as the reference's four warps share one A tile for its wide-N configurations (csrc/SpMM_API.cu:97-112).
// A workgroup of four waves owns (row tile, K slice, group of 4*16*NBW columns):
//   * all four stream and scatter: round r of a tile gives wave w the 64 vectors (r*4 + w)*64 .. of the
//     tile's range of Compressed_A; the vectors of the next kAhead tiles are in flight per wave;
//   * each wave multiplies the whole tile by its own 16*NBW columns: 16 plain 16-byte operand reads
//     (no clearing: the tile has four readers), 16*NBW MFMAs; its B operands are fetched a tile ahead as
//     whole 128-byte lines and turned into the MFMA layout through LDS (stage_b);
//   * three tile buffers rotate, so one barrier per tile is enough: in step t a wave reads tile t from one
//     buffer (complete since the previous barrier), scatters its part of tile t+1 into the second and clears
//     its quarter of the third (read by everybody before the previous barrier).
// Every step issues the same number of global loads in the same order (R stream loads and 2*NBW loads of B
// lines, addresses clamped instead of skipped) and every round has all three steps, so the waits the compiler
// places are exact counts that never drain the stream, and the accumulators stay where they are (with early
// exits from the unrolled round the register allocation more than doubled).  A tile with more than R*256
// vectors takes its remaining rounds on a slow path.
constexpr int kGroupWaves   = 4;
constexpr int kGroupThreads = kGroupWaves * kLanes;
constexpr int kAhead        = 3;  // tiles of the stream in flight per wave = the three buffers' rotation

template<int NBW, int R>
__device__ __forceinline__ void spmm_group_body(uint16_t (*const tiles)[kTileHalfs],
                                                const uint4* __restrict__ comp,
                                                const int* __restrict__ toff,
                                                const _Float16* __restrict__ B,
                                                int ldb,
                                                _Float16* __restrict__ o,
                                                int M,
                                                int N,
                                                int K,
                                                int kb,
                                                int ke,
                                                int col0,
                                                int vmax,
                                                int store,
                                                unsigned w,
                                                unsigned launch)
{
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = threadIdx.x / kLanes;

    floatx4 acc[NBW][8];
#pragma unroll
    for (int nb = 0; nb < NBW; nb++)
#pragma unroll
        for (int rb = 0; rb < 8; rb++)
            acc[nb][rb] = floatx4{0.f, 0.f, 0.f, 0.f};

    // B is fetched whole 128-byte lines at a time: load i of a tile takes the 64 k of columns col0 + 8i .. + 7,
    // eight lanes per column.  (A load of 16 columns x 64 bytes, which is what the MFMA operand layout asks
    // for, takes twice the requests for the same bytes and measured slower.)  Lane l fetches 16-byte piece
    // (l % 8) ^ (l / 8) of its column, so that the staging below reads back without bank conflicts.
    const _Float16* bptr = B + static_cast<size_t>(col0 + (lane >> 3)) * ldb + (((lane & 7) ^ (lane >> 3)) << 3);
    // operand of this lane inside a 16-row block: row r16 = lane % 16, 16-byte chunk (ks*4 + lane/16) ^ (row%8)
    const int a_off0 = (lane & 15) * (kTileCols * 2) + (((lane >> 4) ^ (lane & 7)) << 4);
    const int a_off1 = a_off0 ^ 64;

    uint4 ring[kAhead][R];  // ring[p][r]: this wave's vectors of round r of the tile in slot p
    int   slot_lo[kAhead], slot_n[kAhead];
    uintx4 braw[2 * NBW];  // braw[i]: columns col0 + 8i .. + 7 of B for the next tile, as loaded
    half8  bfrag[2][NBW];  // the MFMA B operands of the current tile

    auto tile_range = [&](int t, int& lo, int& n) {  // tiles at or beyond ke are empty
        const int a = t < ke ? t : ke, b = t + 1 < ke ? t + 1 : ke;
        lo          = toff[a];
        n           = toff[b] - lo;
    };
    int  ahead_lo, ahead_n;  // range of the tile the next request is for, fetched one request earlier
    auto request = [&](auto pp, int t) {  // this wave's R loads of tile t into slot p, always issued
        constexpr int p = decltype(pp)::value;
        slot_lo[p]      = ahead_lo;
        slot_n[p]       = ahead_n;
        tile_range(t + 1, ahead_lo, ahead_n);  // requests go tile by tile, so the next one is for t + 1
#pragma unroll
        for (int r = 0; r < R; r++) {
            int v      = slot_lo[p] + (r * kGroupWaves + wave) * kLanes + lane;
            v          = v < vmax ? v : vmax;
            ring[p][r] = load_stream(comp + v);
        }
    };
    auto load_b = [&](int t) {  // always issued: past the end the last tile's lines are fetched again
        const int tc = t < ke ? t : ke - 1;
#pragma unroll
        for (int i = 0; i < 2 * NBW; i++)
            braw[i] = *reinterpret_cast<const uintx4*>(bptr + static_cast<size_t>(i) * 8 * ldb + tc * kTileCols);
    };
    // The lines go to LDS as they are (lane l -> piece l of load i, i.e. column 8i + l/8 at 128 bytes per
    // column) and are read back at once in the operand layout of the MFMA: lane (r16, g) takes piece
    // (4*ks + g) ^ (r16 % 8) of column 16*nb + r16.  The 4 KB this needs are the wave's own quarter of the
    // tile buffer it is about to clear (nobody else touches that quarter between two meetings).  One wave,
    // in-order LDS: no barrier between write, read and the clearing that follows.
    // blank: a tile past the slice's end multiplies by zeros, whatever B holds
    auto stage_b = [&](uint16_t* buf, bool blank) {
        uintx4* mine = reinterpret_cast<uintx4*>(buf) + wave * (kTileHalfs * 2 / 16 / kGroupWaves);
        static_assert(2 * NBW * kLanes <= kTileHalfs * 2 / 16 / kGroupWaves, "a wave's B lines must fit its quarter of a tile buffer");
#pragma unroll
        for (int i = 0; i < 2 * NBW; i++)
            mine[i * kLanes + lane] = blank ? uintx4{0u, 0u, 0u, 0u} : braw[i];
#pragma unroll
        for (int ks = 0; ks < 2; ks++)
#pragma unroll
            for (int nb = 0; nb < NBW; nb++)
                bfrag[ks][nb] = __builtin_bit_cast(half8, mine[(nb * 16 + (lane & 15)) * 8 + ((ks * 4 + (lane >> 4)) ^ (lane & 7))]);
    };
    auto scatter_slot = [&](auto pp, uint16_t* buf) {
        constexpr int p = decltype(pp)::value;
#pragma unroll
        for (int r = 0; r < R; r++)
            if ((r * kGroupWaves + wave) * kLanes + lane < slot_n[p])
                scatter_vector(buf, ring[p][r]);
        // a tile longer than R rounds: the rest straight from memory
        for (int r = R; r * kGroupThreads < slot_n[p]; r++) {
            const int i = (r * kGroupWaves + wave) * kLanes + lane;
            if (i < slot_n[p])
                scatter_vector(buf, load_stream(comp + slot_lo[p] + i));
        }
    };
    auto clear_quarter = [&](uint16_t* buf) {
        uint4 zero = {0u, 0u, 0u, 0u};
        asm volatile("" : "+v"(zero.x), "+v"(zero.y), "+v"(zero.z), "+v"(zero.w));  // made here, not kept in registers round the loop
        uint4* q = reinterpret_cast<uint4*>(buf) + wave * (kTileHalfs * 2 / 16 / kGroupWaves);
#pragma unroll
        for (int i = 0; i < kTileHalfs * 2 / 16 / kGroupThreads; i++)
            q[i * kLanes + lane] = zero;
    };
    constexpr int kAtOnce = 8;
    auto          multiply = [&](const half8 (&bf)[2][NBW], const uint16_t* buf) {
        const char* base = reinterpret_cast<const char*>(buf);
#pragma unroll
        for (int ks = 0; ks < 2; ks++)
#pragma unroll
            for (int part = 0; part < 8 / kAtOnce; part++) {  // a few row blocks at a time keeps the operand registers few
                half8 a[kAtOnce];
#pragma unroll
                for (int i = 0; i < kAtOnce; i++)
                    a[i] = *reinterpret_cast<const half8*>(base + (part * kAtOnce + i) * (16 * kTileCols * 2) + (ks ? a_off1 : a_off0));
#pragma unroll
                for (int i = 0; i < kAtOnce; i++)
#pragma unroll
                    for (int nb = 0; nb < NBW; nb++)
                        // in place (the accumulator is an in/out operand): left to itself the compiler gives the
                        // unrolled steps accumulators of their own and runs out of registers moving between them
                        asm("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(acc[nb][part * kAtOnce + i]) : "v"(a[i]), "v"(bf[ks][nb]));
            }
    };
    // all LDS traffic of this wave has landed, then everybody meets: nothing here waits for global memory
    auto meet = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // prologue: request kAhead tiles, clear the buffers, scatter the first tile
    tile_range(kb, ahead_lo, ahead_n);
    request(std::integral_constant<int, 0>{}, kb + 0);
    request(std::integral_constant<int, 1>{}, kb + 1);
    request(std::integral_constant<int, 2>{}, kb + 2);
    load_b(kb);
    clear_quarter(tiles[0]);
    clear_quarter(tiles[1]);
    meet();
    scatter_slot(std::integral_constant<int, 0>{}, tiles[0]);
    request(std::integral_constant<int, 0>{}, kb + kAhead);
    clear_quarter(tiles[2]);
    meet();

    // step j of a round of three: tile t sits in buffer j and came from slot j; its B lines were requested a
    // step ago and go through LDS first.  The MFMAs (their A operands have been complete since the last
    // meeting) run while the wave requests the next tile's B lines and scatters the next tile.
    // Rounds are always whole: a step past the slice's end finds an empty (all-zero) buffer, scatters nothing,
    // and multiplies zeros by zeros (its fragments are blanked, so that an Inf or NaN in B cannot leak in).
    auto step = [&](auto jj, int t) {
        constexpr int j = decltype(jj)::value, next = (j + 1) % kAhead;
        stage_b(tiles[(j + 2) % 3], t >= ke);
        multiply(bfrag, tiles[j]);
        load_b(t + 1);
        scatter_slot(std::integral_constant<int, next>{}, tiles[next]);  // tile t + 1 (empty past the end)
        request(std::integral_constant<int, next>{}, t + 1 + kAhead);
        clear_quarter(tiles[(j + 2) % 3]);
        meet();
    };
    for (int t = kb; t < ke; t += kAhead) {
        step(std::integral_constant<int, 0>{}, t);
        step(std::integral_constant<int, 1>{}, t + 1);
        step(std::integral_constant<int, 2>{}, t + 2);
    }

    // the MFMAs came from inline assembly, where the compiler does not pad for the matrix core's write-back
    // latency: give the last ones time before the accumulators are read
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    // D layout of the 16x16 MFMA: lane holds column r16, rows 4*g .. 4*g+3 of each 16-row block.  The lane's
    // coordinates are derived afresh (through an opaque statement) so that nothing is carried round the loop for this.
    int lane_again = threadIdx.x & (kLanes - 1);
    asm volatile("" : "+v"(lane_again));
    if (store == kStorePages) {  // o is the workspace itself here; this wave's NBW pages follow those of the waves before it
        store_pages<NBW>(o, acc, static_cast<int>(threadIdx.x / kLanes) * NBW, N, lane_again, w, launch);
        return;
    }
    const int r16 = lane_again & 15, g = lane_again >> 4;
#pragma unroll
    for (int nb = 0; nb < NBW; nb++) {
        const int n = col0 + nb * 16 + r16;
        if (n < N) {
#pragma unroll
            for (int rb = 0; rb < 8; rb++) {
                *reinterpret_cast<half4*>(o + static_cast<size_t>(n) * M + g * 4 + rb * 16) = to_half4(acc[nb][rb], store);
            }
        }
    }
}

template<int NBW>
__global__ __launch_bounds__(kGroupThreads, 3) void spmm_group_kernel(const uint4* __restrict__ comp,
                                                                  const int* __restrict__ offs,
                                                                  const _Float16* __restrict__ B,
                                                                  int ldb,
                                                                  _Float16* __restrict__ out,
                                                                  int M,
                                                                  int N,
                                                                  int K,
                                                                  int split_k,
                                                                  int col_groups,
                                                                  int store,
                                                                  unsigned units)
{
    __shared__ __attribute__((aligned(16))) uint16_t tiles[3][kTileHalfs];
    const int   kt    = K / kTileCols;
    const Place place = place_of_workgroup(units, split_k);
    if (!place.valid)
        return;
    const int unit = place.unit, slice = place.part;
    const int rowtile = unit / col_groups;
    const int col0    = (unit % col_groups) * (kGroupWaves * 16 * NBW) + (threadIdx.x / kLanes) * (16 * NBW);
    // the reference's slicing (csrc/SpMM_Kernel.cuh:196-204), clamped to K
    const int avg = (kt - 1) / split_k + 1;
    int       kb  = slice * avg;
    kb            = kb < kt ? kb : kt;
    int ke        = kb + avg;
    ke            = ke < kt ? ke : kt;
    const int* toff = offs + static_cast<size_t>(rowtile) * kt;
    _Float16*  o    = store == kStorePages ? out : out + static_cast<size_t>(slice) * M * N + static_cast<size_t>(rowtile) * kTileRows;
    // last vector any load of this slice may touch (clamped loads re-read it)
    int vmax = toff[ke] - 1;
    vmax     = vmax > 0 ? vmax : 0;
    // rounds held in registers per tile: two cover 512 vectors (8 KB, tiles up to a quarter full), three 768
    const int whole = offs[static_cast<size_t>(M / kTileRows) * kt];  // vectors in the matrix
    // An empty matrix has no vector 0: its callers allocate one 4-byte element (reference
    // kernel_benchmark/spmm_test.cu:258-260).  The always-issued loads then read the first 16 bytes of B
    // instead (always there, 16-byte aligned); nothing of them is scattered, every tile has zero vectors.
    if (whole == 0)
        comp = reinterpret_cast<const uint4*>(B);
    if (whole <= 440LL * (M / kTileRows) * kt)
        spmm_group_body<NBW, 2>(tiles, comp, toff, B, ldb, o, M, N, K, kb, ke, col0, vmax, store, place.w, units * split_k);
    else
        spmm_group_body<NBW, 3>(tiles, comp, toff, B, ldb, o, M, N, K, kb, ke, col0, vmax, store, place.w, units * split_k);
}

// ------------------------------------------------------------------------------------------------
// spmm_wide_kernel: four waves share every scattered tile as above, but each multiplies it by 64 columns, 256 per
// workgroup (N a multiple of 256).  The 16 KB of operands a wave reads out of LDS per tile then feed 64 MFMAs instead
// of 32, and the scatter and the clearing are paid once per 256 columns.  128 accumulator registers leave room for two
// waves per SIMD, and no room to hold B a tile ahead in registers: a tile's lines of B (whole 128-byte lines, piece
// (l % 8) ^ (l / 8) of a line to slot l % 8) go straight from memory to 8 KB of LDS that belong to the wave, requested
// as soon as the previous tile's have been read out, i.e. a whole step ahead, and without a meeting.  Fetched in the
// operand layout instead, where neighbouring lanes hold neighbouring columns, the loads themselves are the bound: 9.7
// TB/s out of L2 against 32 with neighbouring lanes on one line (256 columns x 7168, all CUs; 231 against 206 us in an
// earlier form of this kernel at 28672 x 7168, N = 512).
// A wave's tile is taken in quarters, the reads of one ahead of the MFMAs of the one before, in an order that scheduling
// barriers fix (left alone the reads sink to their first use).  What a step asks of global memory is waited for at the
// head of the next: the lines of B right after this tile's are out of LDS (the statement that names every fragment),
// then, behind the first quarter's MFMAs, the wave's part of the stream two tiles on.  Both are asked for early and
// needed a step later, so the wait is for everything and the scatter waits for nothing; the stream behind B, because B
// is the longer fetch (the other order 213 us where this one takes 206, and with the stream asked for at the end of a
// step and waited for in the scatter of the next, which then waits for the younger B too, 202).  28672 x 7168, N = 512, Split_K 1
// with the requests of the stream one quarter earlier / later: 195 / 189 us, B asked for before / after the second
// quarter's reads 188 / 186, clearing or scattering before the third quarter 198 .. 209.
// 80 KB of LDS, two workgroups per CU.  A step takes 1.15 us alone on a CU and 1.65 us for two, where the four-wave
// kernel above takes 0.79 / 1.13 / 1.62 us for one / two / three workgroups with half the columns.  The bound is LDS (144
// KB to and from registers per tile and workgroup, about 0.6 us) beside the MFMAs (0.43 us), which the meetings keep
// from overlapping fully.  Whole calls with the four-wave kernel and this one at the same Split_K, 80 %: 28672 x 7168, N =
// 512, Split_K 1 247 -> 186 us, 21504 x 7168, N = 512, 3 191 -> 154, 36864 x 9216, N = 256, 5 223 -> 176, 7168 x 28672, N
// = 512, 4 259 -> 201.
constexpr int kWideWaves = 4;
constexpr int kWideCols  = kWideWaves * 64;

template<int R>
__device__ __forceinline__ void spmm_wide_body(unsigned char* lds,
                                               const uint4* __restrict__ comp,
                                               const int* __restrict__ toff,
                                               const _Float16* __restrict__ B,
                                               int ldb,
                                               _Float16* __restrict__ o,
                                               int M,
                                               int kb,
                                               int ke,
                                               int col0,
                                               int vmax,
                                               int store,
                                               unsigned w,
                                               unsigned launch)
{
    constexpr int NW = kWideWaves, NBW = 4;
    constexpr int kThreads   = NW * kLanes;
    constexpr int kTileBytes = kTileHalfs * 2;
    const int     lane = threadIdx.x & (kLanes - 1);
    const int     wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    const int     r16 = lane & 15, g = lane >> 4;
    unsigned char* const tiles = lds + NW * NBW * 2048;

    floatx4 acc[NBW][8];
#pragma unroll
    for (int nb = 0; nb < NBW; nb++)
#pragma unroll
        for (int rb = 0; rb < 8; rb++)
            acc[nb][rb] = floatx4{0.f, 0.f, 0.f, 0.f};

    // operand of this lane inside a 16-row block: row r16, 16-byte chunk (ks*4 + g) ^ (row%8)
    const int      a_off0 = r16 * (kTileCols * 2) + ((g ^ (r16 & 7)) << 4);
    const int      a_off1 = a_off0 ^ 64;
    // this wave's columns of B
    const _Float16* bwave  = B + static_cast<size_t>(col0 + wave * (16 * NBW)) * ldb;
    const unsigned  b_voff = (static_cast<unsigned>(lane >> 3) * static_cast<unsigned>(ldb) + (((lane & 7) ^ (lane >> 3)) << 3)) * 2;
    unsigned char* const bwin = lds + wave * (NBW * 2048);
    const uint32_t  bwin_lds  = __builtin_amdgcn_readfirstlane(lds_offset(bwin));
    auto fetch_b = [&](int t) {  // past the end the last tile's lines are fetched again
        const _Float16* p = bwave + (t < ke ? t : ke - 1) * kTileCols;
#pragma unroll
        for (int i = 0; i < 2 * NBW; i++)
            load_to_lds_16(p + static_cast<size_t>(i) * 8 * ldb, b_voff, bwin_lds + i * 1024);
    };
    half8 bfrag[2][NBW];
    auto  read_b = [&](int ks) {
#pragma unroll
        for (int nb = 0; nb < NBW; nb++)
            bfrag[ks][nb] = *reinterpret_cast<const half8*>(bwin + nb * 2048 + (ks ? a_off1 : a_off0));
    };
    struct Ring {
        uintx4 v[R];
        int    lo, n;
    };
    Ring  here, coming;
    int   ahead_lo = toff[kb], ahead_hi = toff[kb + 1 < ke ? kb + 1 : ke];  // range of the tile the next request is for
    auto  request = [&](Ring& ring) {  // this wave's part of that tile (empty past the end), always issued
        ring.lo           = ahead_lo;
        ring.n            = ahead_hi - ahead_lo;
#pragma unroll
        for (int r = 0; r < R; r++) {
            int v     = ring.lo + (r * NW + wave) * kLanes + lane;
            v         = v < vmax ? v : vmax;
            ring.v[r] = __builtin_bit_cast(uintx4, load_stream(comp + v));
        }
    };
    auto look_ahead = [&](int t) {  // behind the request for tile t
        ahead_lo = ahead_hi;
        ahead_hi = toff[t + 2 < ke ? t + 2 : ke];
    };
    auto landed = [&](Ring& ring) {  // the compiler's wait for these loads goes here instead of to their first use
#pragma unroll
        for (int r = 0; r < R; r++)
            asm volatile("" : "+v"(ring.v[r])::"memory");
    };
    auto scatter = [&](int buf, const Ring& ring) {
        uint16_t* tile = reinterpret_cast<uint16_t*>(tiles + buf);
#pragma unroll
        for (int r = 0; r < R; r++)
            if ((r * NW + wave) * kLanes + lane < ring.n)
                scatter_vector(tile, __builtin_bit_cast(uint4, ring.v[r]));
        for (int r = R; r * kThreads < ring.n; r++) {  // a tile longer than R rounds: the rest straight from memory
            const int i = (r * NW + wave) * kLanes + lane;
            if (i < ring.n)
                scatter_vector(tile, load_stream(comp + ring.lo + i));
        }
    };
    auto clear_part = [&](int buf) {
        const uint4 zero = {0u, 0u, 0u, 0u};
        uint4*      q    = reinterpret_cast<uint4*>(tiles + buf) + wave * (kTileBytes / 16 / NW);
#pragma unroll
        for (int i = 0; i < kTileBytes / 16 / kThreads; i++)
            q[i * kLanes + lane] = zero;
    };
    half8 a[2][4];
    auto  read_a = [&](auto cc, int buf) {  // quarter c of the tile: k step c / 2, row blocks 4*(c % 2) .. +3
        constexpr int        c    = decltype(cc)::value;
        const unsigned char* base = tiles + buf + (c / 2 ? a_off1 : a_off0) + (c % 2) * (64 * kTileCols * 2);
#pragma unroll
        for (int i = 0; i < 4; i++)
            a[c % 2][i] = *reinterpret_cast<const half8*>(base + i * (16 * kTileCols * 2));
    };
    auto multiply = [&](auto cc) {
        constexpr int c = decltype(cc)::value;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int nb = 0; nb < NBW; nb++)
                acc[nb][4 * (c % 2) + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[c % 2][i], bfrag[c / 2][nb], acc[nb][4 * (c % 2) + i], 0, 0, 0);
    };
    constexpr std::integral_constant<int, 0> q0{};
    constexpr std::integral_constant<int, 1> q1{};
    constexpr std::integral_constant<int, 2> q2{};
    constexpr std::integral_constant<int, 3> q3{};
    auto meet = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        asm volatile("" ::"s"(ahead_hi));  // here the wait for a scalar load, which shares the counter of LDS, costs nothing
    };
    auto keep_in_order = [&]() { __builtin_amdgcn_sched_barrier(0); };

    int cur = 0, next = kTileBytes, old = 2 * kTileBytes;
    request(here);
    look_ahead(kb);
    fetch_b(kb);
    clear_part(cur);
    clear_part(next);
    meet();
    scatter(cur, here);
    request(coming);
    look_ahead(kb + 1);
    meet();
    for (int t = kb; t < ke; t++) {
        // this tile's lines of B and the stream's part of the next tile were requested a step ago
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        landed(coming);
        here = coming;
        read_b(0);
        read_b(1);
        read_a(q0, cur);
        keep_in_order();
        // ... and are in registers before the next tile's may overwrite them
        asm volatile("" ::"v"(bfrag[0][0]), "v"(bfrag[0][1]), "v"(bfrag[0][2]), "v"(bfrag[0][3]), "v"(bfrag[1][0]), "v"(bfrag[1][1]), "v"(bfrag[1][2]), "v"(bfrag[1][3]) : "memory");
        read_a(q1, cur);
        keep_in_order();
        if (t + 1 < ke)
            fetch_b(t + 1);
        keep_in_order();
        multiply(q0);
        keep_in_order();
        request(coming);  // tile t + 2
        keep_in_order();
        read_a(q2, cur);
        keep_in_order();
        multiply(q1);
        keep_in_order();
        read_a(q3, cur);
        keep_in_order();
        clear_part(old);
        keep_in_order();
        multiply(q2);
        keep_in_order();
        scatter(next, here);  // tile t + 1 (empty past the end)
        keep_in_order();
        look_ahead(t + 2);
        keep_in_order();
        multiply(q3);
        meet();
        const int done = cur;
        cur  = next;
        next = old;
        old  = done;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may land in LDS that is no longer this workgroup's

    if (store == kStorePages) {
        store_pages<NBW>(o, acc, wave * NBW, 16 * NBW, lane, w, launch);
        return;
    }
#pragma unroll
    for (int nb = 0; nb < NBW; nb++) {
        const int n = col0 + (wave * NBW + nb) * 16 + r16;
#pragma unroll
        for (int rb = 0; rb < 8; rb++) {
            *reinterpret_cast<half4*>(o + static_cast<size_t>(n) * M + g * 4 + rb * 16) = to_half4(acc[nb][rb], store);
        }
    }
}

__global__ __launch_bounds__(kWideWaves* kLanes, 2) void spmm_wide_kernel(const uint4* __restrict__ comp,
                                                                 const int* __restrict__ offs,
                                                                 const _Float16* __restrict__ B,
                                                                 int ldb,
                                                                 _Float16* __restrict__ out,
                                                                 int M,
                                                                 int N,
                                                                 int K,
                                                                 int split_k,
                                                                 int col_groups,
                                                                 int store,
                                                                 unsigned units)
{
    __shared__ __attribute__((aligned(16))) unsigned char lds[kWideWaves * 8192 + 3 * kTileHalfs * 2];
    const int   kt    = K / kTileCols;
    const Place place = place_of_workgroup(units, split_k);
    if (!place.valid)
        return;
    const int unit = place.unit, slice = place.part;
    const int rowtile = unit / col_groups;
    const int col0    = (unit % col_groups) * kWideCols;
    // slices, the last vector a load may touch and the empty matrix as in spmm_group_kernel
    const int avg = (kt - 1) / split_k + 1;
    int       kb  = slice * avg;
    kb            = kb < kt ? kb : kt;
    int ke        = kb + avg;
    ke            = ke < kt ? ke : kt;
    const int* toff = offs + static_cast<size_t>(rowtile) * kt;
    _Float16*  o    = store == kStorePages ? out : out + static_cast<size_t>(slice) * M * N + static_cast<size_t>(rowtile) * kTileRows;
    int vmax = toff[ke] - 1;
    vmax     = vmax > 0 ? vmax : 0;
    const int whole = offs[static_cast<size_t>(M / kTileRows) * kt];
    if (whole == 0)
        comp = reinterpret_cast<const uint4*>(B);
    if (whole <= 440LL * (M / kTileRows) * kt)
        spmm_wide_body<2>(lds, comp, toff, B, ldb, o, M, kb, ke, col0, vmax, store, place.w, units * split_k);
    else
        spmm_wide_body<3>(lds, comp, toff, B, ldb, o, M, kb, ke, col0, vmax, store, place.w, units * split_k);
}

// ------------------------------------------------------------------------------------------------
// spmm_quarter_kernel: N a multiple of 128, for slices that are long and launches that leave the two kernels above with one
// or two workgroups per CU.  Both are bound by LDS: a tile of 128 columns takes about 1200 clocks of it in the four-wave kernel, of which
// the four waves' reads of the same 16 KB of operands are 512, and their meetings keep the MFMAs from filling the gaps.
// Here a workgroup's four waves divide the slice along K and never meet before the end: a wave scatters its own tiles and
// multiplies each by all 128 columns, 4 x 4 blocks of 32 x 32 in 256 accumulation registers, so that an operand is read
// once and feeds four MFMAs.  One wave per SIMD has to do by itself what others do by turns: everything that is not an
// MFMA is dealt out between them in program order, at most about one LDS instruction (a 16-byte store takes a lone wave 30
// clocks to issue, a 2-byte store 14) per 32-clock MFMA, and scheduling barriers keep it there.  The MFMAs are inline
// assembly on accumulators that may not move.
//   * Four phases of sixteen MFMAs per tile: columns 0-63 with k steps 0, 1 and 2, 3 of the tile's four, then columns
//     64-127.  Phases 3 and 0 take the operands of the next tile / the tile's second half out of LDS and clear behind the
//     reads, phases 1 and 2 scatter the next tile, and ask for the part of the stream two tiles later.
//   * B comes as whole 128-byte lines straight into LDS, 64 columns at a time into three rotating windows; what is asked
//     for in phase 1 (3) of a tile is read from phase 1 (3) of the next one.  A wait leaves as
//     many loads in flight as have been asked for since at the least; what came between by chance of the depth (the last
//     requests of the phase, those of a long tile) is waited for with the rest.
//   * The ring holds two tiles of the stream, R vectors per lane each, by the average tile of the slice: rows of uneven density
//     make row tiles whose tiles are all longer than the matrix's average, which costs the path below every time.
//   * A tile longer than that has the X vectors per lane behind those of the ring asked for before its first phase and scattered after its
//     last, each later one when the one X before it has been; asked for where they were scattered, one at a time, every one
//     cost a round trip to memory.  Whole calls so, with R by the slice and up to 12 (64 columns: 13, evenly: 11, as many as there
//     are registers for), and with the kernels that shared slices before there were quarters: 10880 x 14144, N = 64, 70 %, rows of uneven density, Split_K 1 139.5 -> 87.1
//     (97.8), 6272 x 21184, N = 128, 30 %, Split_K 5 166 -> 103 (101), 1664 x 3712, N = 640, 90 % with each sixteenth row tile
//     dense 205 -> 73 (101).  With R at most
//     10, 70 % and uneven rows lost 9 %: 14080 x 14656, N = 128, Split_K 4 83.0 -> 90.4.  What N = 64 still loses to eight waves per
//     slice, at most 22 %, are matrices outside 50 ... 90 % and with whole tiles dense: a lone wave issues every store of a dense
//     tile itself, and a nearly empty tile costs it the same clears.  Scattered before the next request instead, which spares the compiler's too strict wait (below): 4 %
//     slower at 70 % and 12 % at N = 64, 80 %, where no tile is long.
//   * With one tile in the ring the compiler's wait before a vector is used, which does not know of B's loads, also waits for B
//     asked for half a tile ago: 7168 x 28672, N = 512, Split_K 1, as first built 240 us, 213 with two.
//     The loop body is therefore two tiles; an early exit between them makes the compiler move accumulators and spill, so
//     runs are whole pairs of tiles and an odd one ends with an empty tile, whose B is zeros.
//   * Lanes past a tile's end load its last vector again and store the same items once more: no masks.
//   * A lone wave issues an instruction in four to five clocks, so that seven fit beside an MFMA and every one more delays the next.
//     An item's address is a mask, which keeps a position that no compressor writes inside the wave's tile, and one instruction on it
//     (v_mad_u32_u16 takes the upper half), M0 is set for every fourth request for B, requests are two slots apart, and scalar work is
//     not left to the phases' ends, where nothing covers it.  Calls in turn, before and after: 7168 x 28672, N = 512 214 -> 206 us, 21504
//     x 7168, N = 384 126 -> 121, 36864 x 9216, N = 128, Split_K 3 at 80 and 90 % 108 -> 106 and 99 -> 94, 28672 x 7168, N = 64 45.2 ->
//     44.0.  The mask is 1 % of that (21504 x 7168, N = 384 118.4 us without, 120.0 with it), with 64 columns up to 2.5 % (6528 x 18240, Split_K
//     5, 78 % 30.5 and 31.2).
//   * The stream is loaded as other data is: the column groups of a row tile sit on one XCD and share its L2 (7168 x 28672, N =
//     512, Split_K 1 210.7 us with non-temporal loads, 202.3).
// With 64 columns (N = 64) a tile is two such phases and one window of B, so that B is asked for two tiles ahead; a tile without
// vectors takes zeros for B, as the other kernels for N <= 64 leave it out altogether.
// 160 KB of LDS and up to 510 registers (64 columns 380): one workgroup per CU.  Calls over copies of A that no cache holds, 80 %, Split_K
// 1, with the kernels before (four waves on every tile, where a launch had at most one workgroup per CU three groups of four; 256
// columns) and this one: 7168 x 28672, N = 512 244 -> 202 us, 7168 x 7168, N = 512 70.5 -> 55.9, N = 128 69.6 -> 52.2, 21504 x 7168, N =
// 384 132.8 -> 117.0, N = 512 180.1 -> 166.8, 1664 x 27200, N = 128 232 -> 169, 28672 x 7168, N = 64 47.5 -> 42.6.  21504 x 7168, N = 384 under counters:
// matrix cores busy half of the time that a workgroup runs, LDS 43 %, 19 % of the waves' time waiting for memory and 17 % for LDS, 83 LDS
// instructions per tile.  As first built (213 us on the first) it took 161 without loads from memory and 128 with nothing but the
// MFMAs; with B through registers and LDS stores 238, with B's windows by halves of k instead of columns, i.e. 64-byte pieces of lines,
// 261.
constexpr int kQuarters      = 4;
constexpr int kQuarterWindow = 64 * kTileCols * 2;                       // 64 columns of B for one k tile
constexpr int kQuarterLds    = kTileHalfs * 2 + 3 * kQuarterWindow;      // a wave's: its tile and three windows of B
using floatx16 = float __attribute__((ext_vector_type(16)));

// what a tile without vectors reads: an item that stores 0 at position 0; and a tile without B, whose requests are up to 3 KB apart
__device__ uint4 g_zeros[256];

template<int NJ, int R, int X>
__device__ __forceinline__ void spmm_quarter_body(unsigned char* lds,
                                                  const uint4* __restrict__ comp,
                                                  const int* __restrict__ toff,
                                                  const _Float16* __restrict__ B,
                                                  int ldb,
                                                  _Float16* __restrict__ o,
                                                  int M,
                                                  int kb,
                                                  int ke,
                                                  int col0,
                                                  int store,
                                                  unsigned w,
                                                  unsigned launch)
{
    using Lds16 = __attribute__((address_space(3))) uint16_t;
    using Lds128 = __attribute__((address_space(3))) uintx4;
    using Global = const __attribute__((address_space(1))) char;
    const int      lane   = threadIdx.x & (kLanes - 1);
    const int      wave   = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    unsigned char* mine   = lds + wave * (kTileHalfs * 2);
    const uint32_t tile_l = __builtin_amdgcn_readfirstlane(lds_offset(mine));
    const uint32_t bwin_l = __builtin_amdgcn_readfirstlane(lds_offset(lds)) + kQuarters * (kTileHalfs * 2) + wave * (3 * kQuarterWindow);

    floatx16 acc[4][NJ];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int e = 0; e < 16; e++)
                acc[i][j][e] = 0.f;

    if (kb < ke) {
        const int r32 = lane & 31, hi = lane >> 5;
        // operand of this lane in k step 0 of a block of 32 rows of the tile, or columns of a window of B; step s: ^ 32 s
        const uint32_t off   = r32 * (kTileCols * 2) + ((hi ^ (r32 & 7)) << 4);
        const uint32_t a_off = tile_l + off;
        uint32_t       b_lane[4];  // where this lane's 16 bytes of 8i columns of B lie, from the first column of the 32
#pragma unroll
        for (int i = 0; i < 4; i++)
            b_lane[i] = (static_cast<unsigned>(8 * i + (lane >> 3)) * static_cast<unsigned>(ldb) + (((lane & 7) ^ (lane >> 3)) << 3)) * 2 - 1024 * i;
        const _Float16* bcols = B + static_cast<size_t>(col0) * ldb;

        half8    a[4][4], b[2][4];
        uintx4   ring[2][R];
        uintx4   rest[X];     // of a tile longer than the ring
        Global*  nothing = (Global*)g_zeros;
        asm volatile("" : "+s"(nothing));  // its address stays in registers
        Global*  from;        // the tile that requests are at
        uint32_t from_last;   // byte of its last vector
        int      lo[3], n[3]; // first vector and vectors of that tile (2), the one before (1) and the one to scatter (0)
        int      ahead_lo = toff[kb], ahead_hi = toff[kb + 1];

        auto keep = [&]() { __builtin_amdgcn_sched_barrier(0); };
        auto next_tile = [&](int t) {  // requests are at tile t from here on; past the end it is empty
            lo[0] = lo[1], n[0] = n[1];
            lo[1] = lo[2], n[1] = n[2];
            lo[2]     = ahead_lo;
            n[2]      = ahead_hi - ahead_lo;
            from      = n[2] > 0 ? (Global*)(comp + ahead_lo) : nothing;
            from_last = n[2] > 0 ? (n[2] - 1) * 16u : 0u;
            ahead_lo  = ahead_hi;
            ahead_hi  = toff[t + 2 < ke ? t + 2 : ke];
        };
        // Lanes past the tile's end load its last vector again, and store the same items to the same places.
        auto request = [&](uintx4& slot, int r) {
            const uint32_t at = lane * 16u + r * (kLanes * 16u);
            slot = *reinterpret_cast<const __attribute__((address_space(1))) uintx4*>(from + (at < from_last ? at : from_last));
        };
        uint32_t in_tile = (kTileHalfs << 16) - 1u;
        asm volatile("" : "+s"(in_tile));  // a register, not a literal of every instruction
        auto scatter = [&](uint32_t item) {
            const uint32_t inside = item & in_tile;  // whatever the item says, it stays in the wave's own tile
            uint32_t       at;                       // 2 * position + tile_l
            asm("v_mad_u32_u16 %0, %1, 2, %2 op_sel:[1,0,0,0]" : "=v"(at) : "v"(inside), "s"(tile_l));
            *reinterpret_cast<Lds16*>(at) = static_cast<uint16_t>(item);
        };
        // a tile of more than R chunks: chunks R .. R + X - 1 of it; lanes past its end as above
        auto request_rest = [&](int r, int chunk) {
            const uint32_t at = lane * 16u + chunk * (kLanes * 16u), last = (n[0] - 1) * 16u;
            rest[r] = *reinterpret_cast<const __attribute__((address_space(1))) uintx4*>((Global*)(comp + lo[0]) + (at < last ? at : last));
        };
        auto expect_rest = [&]() {
            if (n[0] > R * kLanes)
#pragma unroll
                for (int r = 0; r < X; r++)
                    request_rest(r, R + r);
            keep();
        };
        auto scatter_rest = [&]() {
            int chunk = R;
            for (; n[0] > (chunk + X) * kLanes; chunk += X)
#pragma unroll
                for (int r = 0; r < X; r++) {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        scatter(rest[r][e]);
                    request_rest(r, chunk + X + r);
                }
#pragma unroll
            for (int r = 0; r < X; r++)
                if (n[0] > (chunk + r) * kLanes)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        scatter(rest[r][e]);
        };
        auto read_lds = [&](uint32_t at) { return *reinterpret_cast<const __attribute__((address_space(3))) half8*>(at); };
        auto read_a   = [&](int s, int i) { a[s][i] = read_lds((a_off ^ (s * 32)) + i * 4096); };
        auto clear_a  = [&](int s, int i) { *reinterpret_cast<Lds128*>((a_off ^ (s * 32)) + i * 4096) = uintx4{0u, 0u, 0u, 0u}; };
        // operands of phase p out of its half's window: k step 2 (p % 2) + m / 2, columns 32 (m % 2) .. +31 of the 64
        auto read_b = [&](int p, uint32_t window, int m) { b[p & 1][m] = read_lds(((off ^ ((2 * (p & 1) + m / 2) * 32)) + window) + (m % 2) * 4096); };
        // a half: 64 of the 128 columns of a tile's B, as whole lines of eight columns
        struct Half {
            Global*  first;
            size_t   step;  // bytes between 32 columns
            uint32_t lanes;
        };
        auto half_of_b = [&](int half) {  // past the end: zeros (a run of an odd number of tiles ends with an empty one, and Inf and NaN stay out)
            const bool there = NJ == 4 ? half < 2 * ke : n[2] > 0;  // NJ == 2: asked where requests are at the same tile
            return Half{there ? (Global*)(NJ == 4 ? bcols + (half & 1) * (64 * static_cast<size_t>(ldb)) + (half >> 1) * kTileCols : bcols + half * kTileCols) : nothing,
                        there ? 64 * static_cast<size_t>(ldb) : 0, there ? ~0u : 0u};
        };
        // eight requests in a row: M0 is set for every fourth, between them the instruction's offset counts in LDS and in memory.  It is an
        // operand of all four, so that the compiler knows it to be in use (carried so it costs no copy: the same instructions)
        uint32_t m0;
        auto fetch_b = [&](const Half& half, uint32_t window, int i) {
            const uint32_t at    = b_lane[i % 4] & half.lanes;
            Global* const  first = half.first + (i / 4) * half.step;
            if (i % 4 == 0)
                asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : "={m0}"(m0) : "v"(at), "s"(first), "s"(window + i * 1024) : "memory");
            else if (i % 4 == 1)
                asm volatile("global_load_lds_dwordx4 %0, %1 offset:1024" ::"v"(at), "s"(first), "{m0}"(m0) : "memory");
            else if (i % 4 == 2)
                asm volatile("global_load_lds_dwordx4 %0, %1 offset:2048" ::"v"(at), "s"(first), "{m0}"(m0) : "memory");
            else
                asm volatile("global_load_lds_dwordx4 %0, %1 offset:3072" ::"v"(at), "s"(first), "{m0}"(m0) : "memory");
        };
        auto multiply = [&](int p, int m) {
            const int s = 2 * (p & 1) + m / 8, i = m / 2 % 4, j = 2 * (p / 2) + m % 2;
            asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(a[s][i]), "v"(b[p & 1][m / 8 * 2 + m % 2]));
        };
        // windows: w0 holds half 0 of the current tile, w1 half 1, w2 half 0 of the next
        uint32_t w0 = bwin_l, w1 = bwin_l + kQuarterWindow, w2 = bwin_l + 2 * kQuarterWindow;

        // prologue: tile kb in LDS, tiles kb + 1 and kb + 2 in slots 1 and 0 of the ring
        lo[1] = lo[2] = n[1] = n[2] = 0;
        next_tile(kb);
#pragma unroll
        for (int r = 0; r < R; r++)
            request(ring[0][r], r);
        keep();
        Half first = half_of_b(NJ / 2 * kb);
#pragma unroll
        for (int i = 0; i < 8; i++)
            fetch_b(first, w0, i);
        next_tile(kb + 1);
        keep();
#pragma unroll
        for (int r = 0; r < R; r++)
            request(ring[1][r], r);
        keep();
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                clear_a(s, i);
        first = half_of_b(NJ / 2 * kb + 1);
#pragma unroll
        for (int i = 0; i < 8; i++)
            fetch_b(first, w1, i);
        next_tile(kb + 2);
        expect_rest();
#pragma unroll
        for (int r = 0; r < R; r++) {
#pragma unroll
            for (int e = 0; e < 4; e++)
                scatter(ring[0][r][e]);
            request(ring[0][r], r);
            keep();
        }
        if (n[0] > R * kLanes)
            scatter_rest();
        keep();
        first = half_of_b(NJ / 2 * kb + 2);
#pragma unroll
        for (int i = 0; i < 8; i++)
            fetch_b(first, w2, i);
        next_tile(kb + 3);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(R + 16) : "memory");
        keep();
#pragma unroll
        for (int m = 0; m < 4; m++)
            read_b(0, w0, m);
#pragma unroll
        for (int i = 0; i < 8; i++)
            read_a(i / 4, i % 4);
        keep();
#pragma unroll
        for (int i = 0; i < 8; i++)
            clear_a(i / 4, i % 4);
        keep();

        constexpr int R0 = (R + 1) / 2, R1 = R - R0;
        auto clear_some = [&](int m, int s) {  // k steps s and s + 1, behind their reads
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (m == 5 + i * 11 / 8)
                    clear_a(s + i / 4, i % 4);
        };
        auto tile_of_128 = [&](auto slot, int t) {
            uintx4(&next)[R] = ring[decltype(slot)::value];
            expect_rest();
            Half b_half1, b_half0;  // what phases 1 and 3 ask for
            // phase 0: half 0 of B, k steps 0 and 1
#pragma unroll
            for (int m = 0; m < 16; m++) {
                multiply(0, m);
                if (m == 5)
                    b_half1 = half_of_b(2 * t + 3);
                if (m < 4)
                    read_b(1, w0, m);
                else if (m < 12)
                    read_a(2 + (m - 4) / 4, m % 4);
                clear_some(m, 2);
                keep();
            }
            // phase 1: half 0, k steps 2 and 3.  Half 1 has landed; half 0 is out of LDS
            asm volatile("" ::"v"(b[1][0]), "v"(b[1][1]), "v"(b[1][2]), "v"(b[1][3]) : "memory");
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 + R1) : "memory");
            keep();
#pragma unroll
            for (int m = 0; m < 16; m++) {
                multiply(1, m);
                if (m < 4)
                    read_b(2, w1, m);
                if (m % 2 == 0)
                    fetch_b(b_half1, w0, m / 2);
#pragma unroll
                for (int i = m * R0 * 4 / 16; i < (m + 1) * R0 * 4 / 16; i++) {
                    scatter(next[i / 4][i % 4]);
                    if (i % 4 == 3)
                        request(next[i / 4], i / 4);
                }
                keep();
            }
            // phase 2: half 1, k steps 0 and 1
#pragma unroll
            for (int m = 0; m < 16; m++) {
                multiply(2, m);
                if (m < 4)
                    read_b(3, w1, m);
                if (m == 4)
                    b_half0 = half_of_b(2 * t + 4);
#pragma unroll
                for (int i = m * R1 * 4 / 16; i < (m + 1) * R1 * 4 / 16; i++) {
                    scatter(next[R0 + i / 4][i % 4]);
                    if (i % 4 == 3)
                        request(next[R0 + i / 4], R0 + i / 4);
                }
                keep();
            }
            if (n[0] > R * kLanes)
                scatter_rest();
            keep();
            // phase 3: half 1, k steps 2 and 3.  Half 0 of the next tile has landed; this tile's B is out of LDS
            asm volatile("" ::"v"(b[1][0]), "v"(b[1][1]), "v"(b[1][2]), "v"(b[1][3]) : "memory");
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 + R) : "memory");
            keep();
#pragma unroll
            for (int m = 0; m < 16; m++) {
                multiply(3, m);
                if (m < 4)
                    read_b(0, w2, m);
                else if (m < 12)
                    read_a((m - 4) / 4, m % 4);
                clear_some(m, 0);
                if (m % 2 == 0)
                    fetch_b(b_half0, w1, m / 2);
                if (m == 13)
                    next_tile(t + 4);
                keep();
            }
            // next tile: half 0 is in w2, half 1 on its way to w0, the half 0 after it on its way to w1
            const uint32_t old = w0;
            w0 = w2;
            w2 = w1;
            w1 = old;
        };
        // 64 columns: phases 0 and 1 are all there is, and B's windows hold three tiles.  w0 holds the current one's.
        auto tile_of_64 = [&](auto slot, int t) {
            uintx4(&next)[R] = ring[decltype(slot)::value];
            auto scatter_part = [&](int m) {  // m of 16
#pragma unroll
                for (int i = m * R * 4 / 16; i < (m + 1) * R * 4 / 16; i++) {
                    scatter(next[i / 4][i % 4]);
                    if (i % 4 == 3)
                        request(next[i / 4], i / 4);
                }
            };
            expect_rest();
#pragma unroll
            for (int m = 0; m < 16; m++) {
                multiply(0, m);
                if (m < 4)
                    read_b(1, w0, m);
                if (m < 8)
                    read_a(2 + m / 4, m % 4);
                if (m >= 4 && m < 12)
                    clear_a(2 + (m - 4) / 4, m % 4);
                if (m >= 12) {
                    scatter_part(2 * (m - 12));
                    scatter_part(2 * (m - 12) + 1);
                }
                keep();
            }
            // this tile's B is out of LDS, the next one's has landed
            asm volatile("" ::"v"(b[1][0]), "v"(b[1][1]), "v"(b[1][2]), "v"(b[1][3]) : "memory");
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 + R) : "memory");
            const Half b_next = half_of_b(t + 3);
            keep();
#pragma unroll
            for (int m = 0; m < 16; m++) {
                multiply(1, m);
                if (m < 4)
                    read_b(0, w1, m);
                if (m < 8) {
                    scatter_part(8 + m);
                    fetch_b(b_next, w0, m);
                }
                if (m == 7) {
                    if (n[0] > R * kLanes)
                        scatter_rest();
                    keep();
                    next_tile(t + 4);
                }
                if (m >= 8) {
                    read_a((m - 8) / 4, m % 4);
                    clear_a((m - 8) / 4, m % 4);
                }
                keep();
            }
            const uint32_t old = w0;
            w0 = w1;
            w1 = w2;
            w2 = old;
        };
        auto tile = [&](auto slot, int t) {
            if constexpr (NJ == 4)
                tile_of_128(slot, t);
            else
                tile_of_64(slot, t);
        };
        for (int t = kb; t < ke; t += 2) {
            tile(std::integral_constant<int, 1>{}, t);
            tile(std::integral_constant<int, 0>{}, t + 1);
        }
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");  // nothing may land in LDS that other data goes to now; the matrix cores have written back
    }
    __syncthreads();

    // Add up: each wave leaves two column blocks of 32 at a time in its own LDS; wave i sums rows 32i .. +31 in the order of k
    int lane_again = threadIdx.x & (kLanes - 1);
    asm volatile("" : "+v"(lane_again));
    const int r32 = lane_again & 31, hi = lane_again >> 5;
    floatx4*  sums = reinterpret_cast<floatx4*>(lds);
    constexpr int kPerWave = kQuarterLds / 16;
#pragma unroll
    for (int part = 0; part < NJ / 2; part++) {
        if (part)
            __syncthreads();
#pragma unroll
        for (int jj = 0; jj < 2; jj++)
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    sums[wave * kPerWave + ((jj * 4 + i) * 4 + q) * kLanes + lane_again] =
                        floatx4{acc[i][2 * part + jj][4 * q], acc[i][2 * part + jj][4 * q + 1], acc[i][2 * part + jj][4 * q + 2], acc[i][2 * part + jj][4 * q + 3]};
        __syncthreads();
#pragma unroll
        for (int jj = 0; jj < 2; jj++) {
            floatx4 x[4];
#pragma unroll
            for (int q = 0; q < 4; q++)
                x[q] = sums[((jj * 4 + wave) * 4 + q) * kLanes + lane_again];
#pragma unroll
            for (int v = 1; v < kQuarters; v++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    x[q] += sums[v * kPerWave + ((jj * 4 + wave) * 4 + q) * kLanes + lane_again];
            const int col = (2 * part + jj) * 32 + r32;  // of the 128; x[q]: rows 32*wave + 8q + 4*hi .. +3
            if (store == kStorePages) {
                uint4* page = reinterpret_cast<uint4*>(o) + (static_cast<size_t>(col / 16) * launch + w) * 256 + wave * 64 + (col & 15);
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const uint2 l = __builtin_bit_cast(uint2, to_half4(x[q], store)), h = __builtin_bit_cast(uint2, to_half4(x[q + 2], store));
                    page[(2 * q + hi) * 16] = uint4{l.x, l.y, h.x, h.y};
                }
            }
            else {
                _Float16* at = o + static_cast<size_t>(col0 + col) * M + wave * 32 + hi * 4;
#pragma unroll
                for (int q = 0; q < 4; q++)
                    *reinterpret_cast<half4*>(at + 8 * q) = to_half4(x[q], store);
            }
        }
    }
}

template<int NJ>
__global__ __launch_bounds__(kQuarters* kLanes, 1) void spmm_quarter_kernel(const uint4* __restrict__ comp,
                                                                   const int* __restrict__ offs,
                                                                   const _Float16* __restrict__ B,
                                                                   int ldb,
                                                                   _Float16* __restrict__ out,
                                                                   int M,
                                                                   int N,
                                                                   int K,
                                                                   int split_k,
                                                                   int col_groups,
                                                                   int store,
                                                                   unsigned units)
{
    __shared__ __attribute__((aligned(16384))) unsigned char lds[kQuarters * kQuarterLds];
    const int   kt    = K / kTileCols;
    const Place place = place_of_workgroup(units, split_k);
    if (!place.valid)
        return;
    const int unit = place.unit, slice = place.part;
    const int rowtile = unit / col_groups;
    const int col0    = (unit % col_groups) * (32 * NJ);
    // slices as in spmm_group_kernel
    const int avg = (kt - 1) / split_k + 1;
    int       kb  = slice * avg;
    kb            = kb < kt ? kb : kt;
    int ke        = kb + avg;
    ke            = ke < kt ? ke : kt;
    // the waves' runs: whole pairs of tiles, but for the last one of an odd slice
    const int pairs = (ke - kb + 1) / 2, base = kb, end = ke;
    const int run = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    kb            = base + pairs * run / kQuarters * 2;
    ke            = base + pairs * (run + 1) / kQuarters * 2;
    ke            = ke < end ? ke : end;
    const int* toff = offs + static_cast<size_t>(rowtile) * kt;
    _Float16*  o    = store == kStorePages ? out : out + static_cast<size_t>(slice) * M * N + static_cast<size_t>(rowtile) * kTileRows;
    // 64 columns pay for every chunk of a ring that a tile does not fill, and have finer steps: with 4, 7, 10 and 13 rows of uneven
    // density at 80 % take 0.98 x the time of eight waves per slice, at most 1.05 x; with these 0.92 x, at most 0.99 x
    constexpr int X       = NJ == 4 ? 4 : 8;
    const int     vectors = toff[end] - toff[base], tiles = end - base;  // of the slice: all waves take the same depth
    const auto    with    = [&](auto depth) {
        spmm_quarter_body<NJ, decltype(depth)::value, X>(lds, comp, toff, B, ldb, o, M, kb, ke, col0, store, place.w, units * split_k);
    };
    if (vectors <= 236 * tiles)
        with(std::integral_constant<int, 4>{});
    else if (NJ == 2 && vectors <= 300 * tiles)
        with(std::integral_constant<int, NJ == 2 ? 5 : 4>{});
    else if (vectors <= 428 * tiles)
        with(std::integral_constant<int, 7>{});
    else if (NJ == 2 && vectors <= 492 * tiles)
        with(std::integral_constant<int, NJ == 2 ? 8 : 4>{});
    else if (vectors <= 620 * tiles)
        with(std::integral_constant<int, 10>{});
    else if (NJ == 2 && vectors <= 684 * tiles)
        with(std::integral_constant<int, NJ == 2 ? 11 : 4>{});
    else
        with(std::integral_constant<int, NJ == 2 ? 13 : 12>{});
}

// spmm_even_kernel: the same program for launches of several rounds, or of one that leaves CUs idle: the k tiles of all units
// (row tile, 128 columns) in a row are divided evenly among 256 workgroups, one per CU, `share` tiles each.  A workgroup
// takes what it has of one unit after the other, and leaves the sums of each as eight pages in the workspace: the i-th
// workgroup that has a part of unit u at page 8 * (i * units + u).  splitk_reduce_even_kernel adds the parts up.
// The ranges of a die's workgroups follow one another, so that the parts of a unit meet in one L2.  252 + 256 registers.  Calls, 80 %: 36864
// x 9216, N = 128, Split_K 3 117.0 -> 102.8 us (the four-wave kernel, 864 workgroups of which 768 run at once), 17152 x 9536, N = 256, 2
// 124.5 -> 99.7.
constexpr int kEvenWorkgroups = 256;

__global__ __launch_bounds__(kQuarters* kLanes, 1) void spmm_even_kernel(const uint4* __restrict__ comp,
                                                                const int* __restrict__ offs,
                                                                const _Float16* __restrict__ B,
                                                                int ldb,
                                                                _Float16* __restrict__ ws,
                                                                int M,
                                                                int K,
                                                                int col_groups,
                                                                int units,
                                                                int share)
{
    __shared__ __attribute__((aligned(16384))) unsigned char lds[kQuarters * kQuarterLds];
    const int       kt    = K / kTileCols;
    const long long all   = static_cast<long long>(units) * kt;
    const int       range = blockIdx.x * (kEvenWorkgroups / kXcds) + blockIdx.y;
    long long       at    = static_cast<long long>(range) * share;
    const long long end   = at + share < all ? at + share : all;
    const int       run   = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
    while (at < end) {
        const int       unit  = __builtin_amdgcn_readfirstlane(static_cast<int>(at / kt));
        const long long first = static_cast<long long>(unit) * kt;
        const int       base  = __builtin_amdgcn_readfirstlane(static_cast<int>(at - first));
        const int       stop  = __builtin_amdgcn_readfirstlane(static_cast<int>((end - first < kt ? end - first : kt)));
        const int       pairs = (stop - base + 1) / 2;
        const int       kb    = base + pairs * run / kQuarters * 2;
        const int       ke    = base + pairs * (run + 1) / kQuarters * 2;
        const int       part  = __builtin_amdgcn_readfirstlane(static_cast<int>(range - first / share));
        const int*      toff  = offs + static_cast<size_t>(unit / col_groups) * kt;
        const int       vectors = toff[stop] - toff[base], tiles = stop - base;
        const int       col0  = unit % col_groups * 128, end_of_run = ke < stop ? ke : stop;
        const unsigned  page  = 8u * (static_cast<unsigned>(part) * units + unit);
        __syncthreads();  // everybody is done with the sums of the unit before
        if (vectors <= 236 * tiles)
            spmm_quarter_body<4, 4, 4>(lds, comp, toff, B, ldb, ws, 0, kb, end_of_run, col0, kStorePages, page, 1u);
        else if (vectors <= 428 * tiles)
            spmm_quarter_body<4, 7, 4>(lds, comp, toff, B, ldb, ws, 0, kb, end_of_run, col0, kStorePages, page, 1u);
        else if (vectors <= 620 * tiles)
            spmm_quarter_body<4, 10, 4>(lds, comp, toff, B, ldb, ws, 0, kb, end_of_run, col0, kStorePages, page, 1u);
        else
            spmm_quarter_body<4, 11, 4>(lds, comp, toff, B, ldb, ws, 0, kb, end_of_run, col0, kStorePages, page, 1u);
        at = first + stop;
    }
}

__device__ __forceinline__ void add_slab(float (&s)[4], const uint2 v)
{
    const half4 h = __builtin_bit_cast(half4, v);
#pragma unroll
    for (int j = 0; j < 4; j++)
        s[j] += static_cast<float>(h[j]);
}

// C[e] = rn16(sum over slabs, in slab order, of float(ws[s*MN + e])).  Eight bytes per lane and up to
// eight slabs in flight per lane: the slabs are small (M*N halfs), so the kernel is latency bound and
// wants many independent loads rather than wide ones.
// RELU: the sums go through max(x, 0) before rounding (the activation after FFN1, saving a pass over C)
template<bool RELU>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(uint2* __restrict__ c,
                                                           const uint2* __restrict__ ws,
                                                           long n4,
                                                           int  split_k)
{
    const long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n4)
        return;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    int   k    = 0;
    for (; k + 8 <= split_k; k += 8) {
        uint2 v[8];
#pragma unroll
        for (int j = 0; j < 8; j++)
            v[j] = ws[(k + j) * n4 + i];
#pragma unroll
        for (int j = 0; j < 8; j++)
            add_slab(s, v[j]);
    }
    if (k + 4 <= split_k) {
        uint2 v[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            v[j] = ws[(k + j) * n4 + i];
#pragma unroll
        for (int j = 0; j < 4; j++)
            add_slab(s, v[j]);
        k += 4;
    }
    {
        uint2 v[3];
        const int left = split_k - k;  // 0..3
#pragma unroll
        for (int j = 0; j < 3; j++)
            if (j < left)
                v[j] = ws[(k + j) * n4 + i];
#pragma unroll
        for (int j = 0; j < 3; j++)
            if (j < left)
                add_slab(s, v[j]);
    }
    half4 h;
#pragma unroll
    for (int j = 0; j < 4; j++)
        h[j] = static_cast<_Float16>(RELU && !(s[j] > 0.f) ? 0.f : s[j]);
    c[i] = __builtin_bit_cast(uint2, h);
}

// The same sums over slabs stored by workgroup (store_pages), one workgroup per 128-row x 16-column block of C.
// pages_per_unit: pages one workgroup of the SpMM launch stores (its NB, or 4*NBW in the four-wave kernel);
// spmm_grid: workgroups of that launch.  The workgroup order mirrors the SpMM kernel's, so a block is summed
// on the XCD that stored its pages.  Thread t takes 16-byte piece t of each slice's page.
template<bool RELU>
__global__ __launch_bounds__(256) void splitk_reduce_pages_kernel(_Float16* __restrict__ c,
                                                                 const uint4* __restrict__ ws,
                                                                 int M,
                                                                 int N,
                                                                 int split_k,
                                                                 int pages_per_unit,
                                                                 int rows_per_unit,
                                                                 int col_groups,
                                                                 unsigned units)
{
    const int cols = N < 16 ? 8 : 16;
    const int t    = threadIdx.x;
    if (t >= cols * 16)  // N == 8: half a block
        return;
    const Place place = place_of_workgroup(units, pages_per_unit);
    if (!place.valid)
        return;
    const int      unit = place.unit, sub = place.part;
    const unsigned spmm_grid = units * split_k;
    const uint4* first = ws + static_cast<size_t>(sub) * spmm_grid * (cols * 16) + t;
    // the SpMM launch's workgroup of (unit, slice) is base_w + slice*step_w (the launch order above is linear in
    // the part); for a unit of the XCDs' own blocks its two coordinates are this workgroup's x and z
    const bool     own    = blockIdx.z < units / kXcds;
    const unsigned base_w = own ? blockIdx.z * split_k * kXcds + blockIdx.x : static_cast<unsigned>(unit) * split_k;
    const unsigned step_w = own ? kXcds : 1;
    float          s[8]   = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < split_k; k0 += 8) {
        uint4 v[8];
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (k0 + j < split_k)
                v[j] = first[static_cast<size_t>(base_w + (k0 + j) * step_w) * (cols * 16)];
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (k0 + j < split_k) {
                const half8 h = __builtin_bit_cast(half8, v[j]);
#pragma unroll
                for (int e = 0; e < 8; e++)
                    s[e] += static_cast<float>(h[e]);
            }
    }
    half4 lo, hi;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        lo[e] = static_cast<_Float16>(RELU && !(s[e] > 0.f) ? 0.f : s[e]);
        hi[e] = static_cast<_Float16>(RELU && !(s[4 + e] > 0.f) ? 0.f : s[4 + e]);
    }
    // piece t = q*(4*cols) + g*cols + r16: rows 32q + 4g .. +3 and 16 further on, column r16 of the block
    // a unit's pages: rows_per_unit row tiles, one after the other, each with the unit's 16-column blocks in order
    const int lg = N < 16 ? 3 : 4;  // cols = 1 << lg
    const int q = t >> (lg + 2), g = (t >> lg) & 3, r16 = t & (cols - 1);
    const int blocks  = pages_per_unit / rows_per_unit;
    const int n       = ((unit % col_groups) * blocks + sub % blocks) * 16 + r16;
    const int rowtile = (unit / col_groups) * rows_per_unit + sub / blocks;
    _Float16* o = c + static_cast<size_t>(n) * M + static_cast<size_t>(rowtile) * kTileRows + q * 32 + g * 4;
    *reinterpret_cast<half4*>(o)      = lo;
    *reinterpret_cast<half4*>(o + 16) = hi;
}

// The sums over what spmm_even_kernel left: one workgroup per 128-row x 16-column block of C, mostly on the XCD that stored it.
template<bool RELU>
__global__ __launch_bounds__(256) void splitk_reduce_even_kernel(_Float16* __restrict__ c,
                                                                const uint4* __restrict__ ws,
                                                                int M,
                                                                int kt,
                                                                int col_groups,
                                                                unsigned units,
                                                                int share)
{
    const Place place = place_of_workgroup(units, 8);
    if (!place.valid)
        return;
    const int       unit  = place.unit, t = threadIdx.x;
    const long long first = static_cast<long long>(unit) * kt;
    const int       parts = static_cast<int>((first + kt - 1) / share - first / share) + 1;
    const uint4*    from  = ws + (static_cast<size_t>(unit) * 8 + place.part) * 256 + t;
    const size_t    step  = static_cast<size_t>(units) * 8 * 256;
    float           s[8]  = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < parts; k0 += 4) {
        uint4 v[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (k0 + j < parts)
                v[j] = from[(k0 + j) * step];
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (k0 + j < parts) {
                const half8 h = __builtin_bit_cast(half8, v[j]);
#pragma unroll
                for (int e = 0; e < 8; e++)
                    s[e] += static_cast<float>(h[e]);
            }
    }
    half4 lo, hi;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        lo[e] = static_cast<_Float16>(RELU && !(s[e] > 0.f) ? 0.f : s[e]);
        hi[e] = static_cast<_Float16>(RELU && !(s[4 + e] > 0.f) ? 0.f : s[4 + e]);
    }
    const int q = t >> 6, g = (t >> 4) & 3, r16 = t & 15;  // as in splitk_reduce_pages_kernel
    _Float16* o = c + (static_cast<size_t>(unit % col_groups) * 128 + place.part * 16 + r16) * M + static_cast<size_t>(unit / col_groups) * kTileRows + q * 32 + g * 4;
    *reinterpret_cast<half4*>(o)      = lo;
    *reinterpret_cast<half4*>(o + 16) = hi;
}

// out[w] = id of the XCD that workgroup w of this launch ran on, w = x + 8*(y + 3*z) in a grid (8, 3, layers):
// the order in which the launches above count on their workgroups being handed out
__global__ __launch_bounds__(kLanes) void xcd_probe_kernel(unsigned* __restrict__ out, unsigned workgroups)
{
    const unsigned w = blockIdx.x + kXcds * (blockIdx.y + 3 * blockIdx.z);
    if (threadIdx.x == 0 && w < workgroups)
        out[w] = __builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11));  // XCC_ID, bits 3:0
}

__global__ __launch_bounds__(256) void take_rows_kernel(uint4* __restrict__ dst, const uint4* __restrict__ src, int rows8, int cols, int ld8)
{
    const long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= static_cast<long>(rows8) * cols)
        return;
    const int j = static_cast<int>(i / rows8), r = static_cast<int>(i % rows8);
    dst[i] = src[static_cast<long>(j) * ld8 + r];
}

template<int NB, int DEPTH, int W, int G, int KS>
int launch_spmm(hipStream_t stream, const void* comp, const int* offs, const void* b, int ldb, void* out, int m, int n, int k, int split_k, int col_groups, int store)
{
    const unsigned units = (static_cast<unsigned>(m / kTileRows) + W - 1) / W * col_groups;
    hipLaunchKernelGGL((spmm_stream_kernel<NB, DEPTH, W, G, KS>),
                       grid_of(units, split_k),
                       dim3(kLanes * W * KS),
                       0,
                       stream,
                       static_cast<const uint4*>(comp),
                       offs,
                       static_cast<const _Float16*>(b),
                       ldb,
                       static_cast<_Float16*>(out),
                       m,
                       n,
                       k,
                       split_k,
                       col_groups,
                       store,
                       units);
    return static_cast<int>(hipGetLastError());
}

template<int KS>
int launch_by_columns(hipStream_t s, const void* comp, const int* offs, const void* b, int ldb, void* out, int m, int n, int k, int split_k, int store)
{
    if (n <= 16)
        return launch_spmm<1, 8, 1, 1, KS>(s, comp, offs, b, ldb, out, m, n, k, split_k, 1, store);
    if (n == 32)
        return launch_spmm<2, 8, 1, 1, KS>(s, comp, offs, b, ldb, out, m, n, k, split_k, 1, store);
    return launch_spmm<4, 6, 1, 1, KS>(s, comp, offs, b, ldb, out, m, n, k, split_k, n / 64, store);
}

// Row tiles per workgroup of the launch for B of n columns, A of m rows and split_k slices: 8 (a CU's eight waves
// share each staged window of B) for n = 64 when the row tiles come in whole groups of eight (the slabs of whole
// workgroups then fill Split_K*M*N halfs exactly, and the callers' workspaces hold no more) and the launch's
// workgroups, each of which fills a CU, number between 192 and 256: one round on at least three quarters of the
// 256 CUs.  Otherwise 1: fewer, larger workgroups would leave CUs idle (7168 x 7168 at its best Split_K: 23.8 us
// with one row tile per workgroup, 29.6 us with eight), more would run in two rounds.
// Calls at n = 64, Split_K 7, 80 %: 36864 x 9216 68.2 us, with one row tile per workgroup 84.6, 36864 x 12288 88.6 and 109.8; at 70 and
// 90 % the first 88.1 and 100.3, 60.7 and 68.0.  At n = 32 52.4
// against 51.7 (the four fragment loads a tile costs there are no more than the meeting and the LDS reads that
// replace them), and workgroups of four row tiles meeting at every tile gain nothing at n = 64 (72.9 us, eight 62 to 64 then).
// The lines at 192 and 256 are from then; fewer workgroups have not been measured since the form takes 2 to 8 % less.
// g_rows_override (a measuring and testing aid): 1 forces 1, 8 forces 8 wherever the row tiles allow it.
std::atomic<int> g_rows_override{0};

int rows_per_workgroup(int n, int m, int split_k)
{
    const int forced = g_rows_override.load(std::memory_order_relaxed);
    const int tiles  = m / kTileRows;
    if (n != 64 || forced == 1 || tiles % 8)
        return 1;
    if (forced == 8)
        return 8;
    const long workgroups = static_cast<long>(tiles / 8) * split_k;
    return workgroups >= 192 && workgroups <= 256 ? 8 : 1;
}

// Columns per workgroup of a launch at N a multiple of 128: 128 (spmm_group_kernel, three workgroups per CU) or 256
// (spmm_wide_kernel, two), by the time of a step with the workgroups that share a CU, beyond a full round the whole
// rounds and what the rest of the last one adds (us).  Fitted to whole-call times of 25 weight shapes (1024 x 1024 ..
// 36864 x 14336, among them the reference's twelve) x N = 128, 256, 384, 512, 640 x Split_K 1 .. 24, 80 %.  At a given Split_K
// the 256-column kernel takes 0.83 x the time of the four-wave kernel on average where it is chosen, at most 1.04 x
// (22016 x 1984, N = 256, Split_K 3: 45.5 / 47.4 us).  Closest is one round and up to a quarter more, 513 .. 640 workgroups of
// 256 columns: 0.89 .. 0.96 x on slices of 4 tiles, 0.98 x of 16, 1.02 x of 36 and more (50 .. 97 % sparsity).
double group_step(long workgroups)
{
    if (workgroups <= 768)
        return workgroups <= 256 ? 0.79 : workgroups <= 512 ? 1.13 : 1.62;
    const long rest = workgroups % 768;
    return 1.62 * (workgroups / 768 + (rest == 0 ? 0.0 : rest <= 256 ? 0.37 : rest <= 512 ? 0.69 : 1.0));
}

double wide_step(long workgroups)
{
    if (workgroups <= 512)
        return workgroups <= 256 ? 1.15 : 1.65;
    const long rest = workgroups % 512;
    return 1.65 * (workgroups / 512 + (rest == 0 ? 0.0 : rest <= 256 ? 0.61 : 1.0));
}

int columns_per_workgroup(int n, int m, int split_k)
{
    const long workgroups = static_cast<long>(m / kTileRows) * (n / 128) * split_k;
    return n % kWideCols == 0 && wide_step(workgroups / 2) < group_step(workgroups) ? kWideCols : 128;
}

constexpr int      kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

}  // namespace

// Library-owned slab storage for callers that cannot provide (or allocate) a Reduction_Workspace: a fixed
// array in the code object's own device memory, one copy per GPU the library runs on, held until the
// process ends.  In host code the array's name is only a handle: the device address comes from
// hipGetSymbolAddress, once per device, and that pointer is what kernels receive.
static __device__ __align__(256) unsigned char scratch[FLASHLLM_STATIC_WORKSPACE_BYTES];

extern "C" int flashllm_hip_static_workspace(void** ptr)
{
    int        dev = -1;
    hipError_t e   = hipGetDevice(&dev);
    if (e != hipSuccess)
        return static_cast<int>(e);
    if (dev < 0 || dev >= kMaxDevices)
        return static_cast<int>(hipErrorInvalidDevice);
    void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {  // first call on this device (two threads racing here resolve the same address)
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess)
            return static_cast<int>(e);
        if (!p)
            return static_cast<int>(hipErrorInvalidSymbol);
        g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
    *ptr = p;
    return 0;
}

// kStorePages only with a Split_K > 1, kStoreRelu only with Split_K == 1
extern "C" int flashllm_hip_launch_spmm(
    void* stream, const void* comp, const int* offs, const void* b, int ldb, void* out, int m, int n, int k, int split_k, int store, int k_waves)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    store         = split_k > 1 ? store == kStorePages : store & kStoreRelu;
    if (n == 64 && k_waves == 0) {
        const unsigned units = static_cast<unsigned>(m / kTileRows);
        hipLaunchKernelGGL(spmm_quarter_kernel<2>, grid_of(units, split_k), dim3(kQuarters * kLanes), 0, s, static_cast<const uint4*>(comp), offs,
                           static_cast<const _Float16*>(b), ldb, static_cast<_Float16*>(out), m, n, k, split_k, 1, store, units);
        return static_cast<int>(hipGetLastError());
    }
    if (n == 64 && rows_per_workgroup(n, m, split_k) == 8)
        return launch_spmm<4, 8, 8, 2, 1>(s, comp, offs, b, ldb, out, m, n, k, split_k, 1, store);
    if (k_waves == 8)
        return launch_by_columns<8>(s, comp, offs, b, ldb, out, m, n, k, split_k, store);
    if (k_waves == 4)
        return launch_by_columns<4>(s, comp, offs, b, ldb, out, m, n, k, split_k, store);
    if (k_waves == 2)
        return launch_by_columns<2>(s, comp, offs, b, ldb, out, m, n, k, split_k, store);
    return launch_by_columns<1>(s, comp, offs, b, ldb, out, m, n, k, split_k, store);
}

extern "C" void flashllm_hip_set_rows_per_workgroup(int rows)
{
    g_rows_override.store(rows, std::memory_order_relaxed);
}

extern "C" int flashllm_hip_rows_per_workgroup(int n, int m, int split_k)
{
    return rows_per_workgroup(n, m, split_k);
}

extern "C" int flashllm_hip_columns_per_workgroup(int n, int m, int split_k)
{
    return columns_per_workgroup(n, m, split_k);
}

extern "C" double flashllm_hip_wide_b_step(int n, int m, int split_k)
{
    const long workgroups = static_cast<long>(m / kTileRows) * (n / 128) * split_k;
    return columns_per_workgroup(n, m, split_k) == kWideCols ? wide_step(workgroups / 2) : group_step(workgroups);
}

extern "C" int flashllm_hip_launch_spmm_group(
    void* stream, const void* comp, const int* offs, const void* b, int ldb, void* out, int m, int n, int k, int split_k, int store, int runs)
{
    const int       cols  = runs > 1 ? 128 : columns_per_workgroup(n, m, split_k);
    const unsigned  units = static_cast<unsigned>(m / kTileRows) * (n / cols);
    const dim3      grid  = grid_of(units, split_k);
    hipStream_t     s     = static_cast<hipStream_t>(stream);
    const uint4*    cp    = static_cast<const uint4*>(comp);
    const _Float16* bp    = static_cast<const _Float16*>(b);
    _Float16*       op    = static_cast<_Float16*>(out);
    store                 = split_k > 1 ? store == kStorePages : store & kStoreRelu;
    if (cols == kWideCols)
        hipLaunchKernelGGL(spmm_wide_kernel, grid, dim3(kWideWaves * kLanes), 0, s, cp, offs, bp, ldb, op, m, n, k, split_k, n / cols, store, units);
    else if (runs > 1)
        hipLaunchKernelGGL(spmm_quarter_kernel<4>, grid, dim3(kQuarters * kLanes), 0, s, cp, offs, bp, ldb, op, m, n, k, split_k, n / 128, store, units);
    else
        hipLaunchKernelGGL(spmm_group_kernel<2>, grid, dim3(kGroupThreads), 0, s, cp, offs, bp, ldb, op, m, n, k, split_k, n / 128, store, units);
    return static_cast<int>(hipGetLastError());
}

extern "C" int flashllm_hip_launch_spmm_even(
    void* stream, const void* comp, const int* offs, const void* b, int ldb, void* c, void* ws, int m, int n, int k, int share, int relu)
{
    const unsigned units = static_cast<unsigned>(m / kTileRows) * (n / 128);
    hipStream_t    s     = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(spmm_even_kernel, dim3(kXcds, kEvenWorkgroups / kXcds), dim3(kQuarters * kLanes), 0, s, static_cast<const uint4*>(comp), offs,
                       static_cast<const _Float16*>(b), ldb, static_cast<_Float16*>(ws), m, k, n / 128, static_cast<int>(units), share);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return static_cast<int>(e);
    const auto reduce = relu ? splitk_reduce_even_kernel<true> : splitk_reduce_even_kernel<false>;
    hipLaunchKernelGGL(reduce, grid_of(units, 8), dim3(256), 0, s, static_cast<_Float16*>(c), static_cast<const uint4*>(ws), m, k / kTileCols, n / 128,
                       units, share);
    return static_cast<int>(hipGetLastError());
}

extern "C" int flashllm_hip_launch_reduce(void* stream, void* c, const void* ws, long mn, int split_k, int relu)
{
    const long     n4 = mn / 4;
    const dim3     grid(static_cast<unsigned>((n4 + 255) / 256));
    hipStream_t    s  = static_cast<hipStream_t>(stream);
    uint2*         cp = static_cast<uint2*>(c);
    const uint2*   wp = static_cast<const uint2*>(ws);
    if (relu)
        hipLaunchKernelGGL(splitk_reduce_kernel<true>, grid, dim3(256), 0, s, cp, wp, n4, split_k);
    else
        hipLaunchKernelGGL(splitk_reduce_kernel<false>, grid, dim3(256), 0, s, cp, wp, n4, split_k);
    return static_cast<int>(hipGetLastError());
}

extern "C" int flashllm_hip_launch_reduce_pages(void* stream, void* c, const void* ws, int m, int n, int split_k, int relu)
{
    // the units of the SpMM launch for this N: `rows` row tiles x 16*blocks columns (a wave's columns in
    // spmm_stream_kernel, a workgroup's 128 or 256 at n % 128 == 0)
    const bool     group      = n % 128 == 0;
    const int      rows       = group ? 1 : rows_per_workgroup(n, m, split_k);
    const int      cols       = group ? columns_per_workgroup(n, m, split_k) : (n <= 16 ? 16 : n == 32 ? 32 : 64);
    const int      blocks     = cols / 16;
    const int      col_groups = n <= 64 ? 1 : n / cols;
    const unsigned units      = (static_cast<unsigned>(m / kTileRows) + rows - 1) / rows * col_groups;
    const int      pages_per_unit = blocks * rows;
    const dim3     grid = grid_of(units, pages_per_unit);
    hipStream_t    s  = static_cast<hipStream_t>(stream);
    _Float16*      cp = static_cast<_Float16*>(c);
    const uint4*   wp = static_cast<const uint4*>(ws);
    if (relu)
        hipLaunchKernelGGL(splitk_reduce_pages_kernel<true>, grid, dim3(256), 0, s, cp, wp, m, n, split_k, pages_per_unit, rows, col_groups, units);
    else
        hipLaunchKernelGGL(splitk_reduce_pages_kernel<false>, grid, dim3(256), 0, s, cp, wp, m, n, split_k, pages_per_unit, rows, col_groups, units);
    return static_cast<int>(hipGetLastError());
}

extern "C" int flashllm_hip_launch_xcd_probe(void* stream, unsigned* out, int workgroups)
{
    if (workgroups <= 0)
        return static_cast<int>(hipErrorInvalidValue);
    const dim3 grid(kXcds, 3, (static_cast<unsigned>(workgroups) + 3 * kXcds - 1) / (3 * kXcds));
    hipLaunchKernelGGL(xcd_probe_kernel, grid, dim3(kLanes), 0, static_cast<hipStream_t>(stream), out, static_cast<unsigned>(workgroups));
    return static_cast<int>(hipGetLastError());
}

extern "C" int flashllm_hip_launch_take_rows(void* stream, void* dst, const void* src, int rows, int cols, int src_ld)
{
    const long n8 = static_cast<long>(rows / 8) * cols;
    hipLaunchKernelGGL(take_rows_kernel, dim3(static_cast<unsigned>((n8 + 255) / 256)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), static_cast<uint4*>(dst), static_cast<const uint4*>(src),
                       rows / 8, cols, src_ld / 8);
    return static_cast<int>(hipGetLastError());
}
