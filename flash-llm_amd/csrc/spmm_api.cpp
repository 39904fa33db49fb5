// Host API: argument checks, Split_K policy and the two launches behind
// SpMM_SplitK_API (reference csrc/SpMM_API.cu:55-130), plus the C++ wrappers
// that keep the reference's compressor signatures (build/SpMM_API.cuh:51-58).
#include "SpMM_API.h"
#include "flashllm_spmm.h"
#include "spmm_launch.h"

#include <cmath>
#include <cstdio>
#include <cstdlib>

namespace {

// The N values the reference dispatches on (csrc/SpMM_API.cu:79-118).
bool supported_n(int n)
{
    return n == 8 || n == 16 || n == 32 || n == 64 || (n > 0 && n % 128 == 0);
}

int check_shape(const void* comp, const int* offs, const void* b, const void* c, int m, int n, int k, const void* ws, int split_k)
{
    if (!comp || !offs || !b || !c)
        return hipErrorInvalidValue;
    if (m <= 0 || k <= 0 || m % 128 || k % 64 || split_k < 1)
        return hipErrorInvalidValue;
    if (!supported_n(n)) {
        std::printf("MM_Sparse_API Error: Unsupported N dimension %d!\n", n);
        return hipErrorUnknown;
    }
    if (split_k > 1 && !ws)
        return hipErrorInvalidValue;
    if (reinterpret_cast<uintptr_t>(comp) % 16 || reinterpret_cast<uintptr_t>(b) % 16 || reinterpret_cast<uintptr_t>(c) % 8
        || reinterpret_cast<uintptr_t>(ws) % 16)
        return hipErrorInvalidValue;
    return hipSuccess;
}

// What a call at N <= 64 takes with k_waves waves on each (row tile, slice), in units of about 0.2 us:
//     k tiles of the longest wave x (a + waves on its CU)  +  adding up k_waves sums  +  a second launch and its slabs.
// A wave needs a fixed time per tile plus what its neighbours on the CU take from it (LDS and issue slots are
// shared), so more waves only help while they shorten the longest run faster than they crowd the CU.  A CU holds
// eight waves; workgroups beyond one round of the GPU wait for a whole round.  The waves on a CU count as a mean of
// their average and, more so, of the fullest CU's (workgroups of eight waves fill CUs unevenly, e.g. 288 of them).
// Fitted to whole-call times of nineteen weight shapes (1024 x 1024 .. 49152 x 12288, among them the reference's,
// kernel_benchmark/benchmark.sh:13-14) x N in {8, 16, 32, 64} x Split_K 1..32 x 1 / 2 / 4 / 8 waves at 70, 80 and
// 90 % sparsity: N <= 32 the best (Split_K, waves) by this cost is on average 0.4 %, at most 4.3 % above the best
// measured, N = 64 0.2 % and 2.2 %; the number of waves at a given Split_K is 0.1 % above the best on average.
double stream_cost(int m, int n, int k, int split_k, int k_waves)
{
    const int    units   = m / 128;  // N <= 64: one column group
    const int    slice   = (k / 64 - 1) / split_k + 1;
    const double scale   = n / 16.0 * m / 36864.0;
    const double average = static_cast<double>(units) * split_k / 256.0;  // workgroups per CU
    if (flashllm_hip_rows_per_workgroup(n, m, split_k) == 8)  // eight row tiles per workgroup sharing B
        return 1.18 * slice * (3.15 + 0.94 * average) + (split_k > 1 ? 7.8 + split_k * (0.46 + 0.37 * scale) : 0.0);
    const double resident = 8 / k_waves;
    const double fullest  = std::ceil(average) < resident ? std::ceil(average) : resident;
    const double typical  = average < resident ? average : resident;
    const double rounds   = std::ceil(average / resident);
    const int    longest  = (slice - 1) / k_waves + 1;
    const double adding   = k_waves > 1 ? 0.15 * k_waves : 0.0;
    if (n < 64)
        return longest * (3.67 + k_waves * (0.7 * fullest + 0.3 * typical)) * rounds + adding + (split_k > 1 ? 18.0 + split_k * (0.84 + 0.22 * scale) : 0.0);
    return longest * (4.0 + k_waves * (0.86 * fullest + 0.14 * typical)) * rounds + adding + (split_k > 1 ? 7.8 + split_k * (0.46 + 0.37 * scale) : 0.0);
}

// Whether the GPU (256 CUs of eight waves) holds all workgroups of such a call at once.
bool one_round(int m, int split_k, int k_waves)
{
    return static_cast<long>(m / 128) * split_k <= 256L * (8 / k_waves);
}

// Waves that share one (row tile, slice) of a call at N <= 64: 1, 2, 4 or 8, by the cost above.  With a Split_K that
// leaves CUs idle this is most of the call's parallelism (4736 x 5184, N = 32, Split_K 4: 35.9 us with one wave per
// slice, 13.8 with eight); with a Split_K of the library's choice it replaces slabs, whose reduction costs a launch
// and about 3 us, by sums in LDS (28672 x 7168, N = 16: Split_K 8 33.1 us, Split_K 1 with eight waves 32.1;
// 7168 x 7168, N = 64: Split_K 16 23.8, Split_K 4 with eight waves 20.8).  N = 64 keeps one wave on slices of fewer
// than twelve tiles: there its sums are those of the kernel for wide B, bit for bit.
int waves_per_slice(int m, int n, int k, int split_k)
{
    const int slice = (k / 64 - 1) / split_k + 1;
    int       best  = 1;
    if (n > 64 || flashllm_hip_rows_per_workgroup(n, m, split_k) == 8 || (n == 64 && slice < 12))
        return 1;
    double best_cost = stream_cost(m, n, k, split_k, 1);
    for (int w = 2; w <= 8 && w <= slice && one_round(m, split_k, w); w *= 2) {
        const double cost = stream_cost(m, n, k, split_k, w);
        if (cost < best_cost) {
            best_cost = cost;
            best      = w;
        }
    }
    return best;
}

// Groups of four waves that divide a slice of a call at N % 128 == 0: three where the launch gives a CU at most one
// workgroup and the runs are long enough to pay for their own fill and the sum (measured in us with one / three:
// 7168 x 7168, N = 128, slices of 112 tiles 90.6 / 71.6, of 56 50.2 / 44.7, of 28 31.4 / 31.7; 2048 x 8192, N = 384, of 32
// 33.0 / 30.9; 9216 x 36864, N = 128, of 192 152.9 / 123.9), otherwise one.
int runs_per_slice(int m, int n, int k, int split_k)
{
    const int slice = (k / 64 - 1) / split_k + 1;
    return static_cast<long>(m / 128) * (n / 128) * split_k <= 256 && slice >= 32 ? 3 : 1;
}

bool known_order(int slab_order)
{
    return slab_order == FLASHLLM_SLABS_PLAIN || slab_order == FLASHLLM_SLABS_BY_WORKGROUP;
}

int launch_partials(void* stream, const void* comp, const int* offs, const void* b, int ldb, void* c, int m, int n, int k, void* ws, int split_k, int slab_order, int relu)
{
    // with one slice the sums are final: the activation belongs to them
    const int pages = split_k == 1 ? 2 * relu : slab_order == FLASHLLM_SLABS_BY_WORKGROUP;
    // wide B: four waves share every scattered tile; otherwise each wave has its own (row tile, run of k tiles)
    if (n % 128 == 0)
        return flashllm_hip_launch_spmm_group(stream, comp, offs, b, ldb, split_k == 1 ? c : ws, m, n, k, split_k, pages, runs_per_slice(m, n, k, split_k));
    return flashllm_hip_launch_spmm(stream, comp, offs, b, ldb, split_k == 1 ? c : ws, m, n, k, split_k, pages, waves_per_slice(m, n, k, split_k));
}

// SpMM_SplitK_API with B's columns ldb halfs apart (the public entry points take a dense column-major B: ldb = K)
// relu: C through max(., 0)
int spmm_splitk_ldb(void* stream, const void* comp, const int* offs, const void* b, int ldb, void* c, int m, int n, int k, void* ws, int split_k, int relu)
{
    int rc = check_shape(comp, offs, b, c, m, n, k, ws, split_k);
    if (rc)
        return rc;
    if (ldb < k || ldb % 8)
        return hipErrorInvalidValue;
    rc = launch_partials(stream, comp, offs, b, ldb, c, m, n, k, ws, split_k, FLASHLLM_SLABS_BY_WORKGROUP, relu);
    if (rc || split_k == 1)
        return rc;
    return flashllm_hip_launch_reduce_pages(stream, c, ws, m, n, split_k, relu);
}

// The reduction behind launch_partials with the same slab_order.
int reduce_slabs(void* stream, void* c, const void* ws, int m, int n, int split_k, int slab_order)
{
    if (slab_order == FLASHLLM_SLABS_BY_WORKGROUP)
        return flashllm_hip_launch_reduce_pages(stream, c, ws, m, n, split_k, 0);
    return flashllm_hip_launch_reduce(stream, c, ws, static_cast<long>(m) * n, split_k, 0);
}

}  // namespace

extern "C" {

int flashllm_spmm_partials(void*       stream,
                           const void* comp,
                           const int*  offs,
                           const void* b,
                           void*       c,
                           int         m,
                           int         n,
                           int         k,
                           void*       ws,
                           int         split_k,
                           int         slab_order)
{
    const int bad = check_shape(comp, offs, b, c, m, n, k, ws, split_k);
    if (bad)
        return bad;
    if (!known_order(slab_order))
        return hipErrorInvalidValue;
    return launch_partials(stream, comp, offs, b, k, c, m, n, k, ws, split_k, slab_order, 0);
}

int flashllm_splitk_reduce(void* stream, void* c, const void* ws, int m, int n, int split_k, int slab_order)
{
    if (!c || !ws || m <= 0 || n <= 0 || split_k < 1 || (static_cast<long>(m) * n) % 4 || !known_order(slab_order)
        || reinterpret_cast<uintptr_t>(c) % 8 || reinterpret_cast<uintptr_t>(ws) % 8)
        return hipErrorInvalidValue;
    // pages exist only for shapes the SpMM kernels take
    if (slab_order == FLASHLLM_SLABS_BY_WORKGROUP && (m % 128 || !supported_n(n) || reinterpret_cast<uintptr_t>(ws) % 16))
        return hipErrorInvalidValue;
    return reduce_slabs(stream, c, ws, m, n, split_k, slab_order);
}

int flashllm_spmm_splitk(void*       stream,
                         const void* /*A: unused, as in the reference*/,
                         const void* comp,
                         const int*  offs,
                         const void* b,
                         void*       c,
                         int         m,
                         int         n,
                         int         k,
                         void*       ws,
                         int         split_k)
{
    // the workspace is this call's own business between its two kernels: slabs by workgroup
    int rc = flashllm_spmm_partials(stream, comp, offs, b, c, m, n, k, ws, split_k, FLASHLLM_SLABS_BY_WORKGROUP);
    if (rc || split_k == 1)
        return rc;
    return reduce_slabs(stream, c, ws, m, n, split_k, FLASHLLM_SLABS_BY_WORKGROUP);
}

// SpMM_SplitK_API for callers that must not allocate and hold no workspace: the slabs go to the
// library's fixed device array.
int flashllm_spmm_splitk_static(void*       stream,
                                const void* a,
                                const void* comp,
                                const int*  offs,
                                const void* b,
                                void*       c,
                                int         m,
                                int         n,
                                int         k,
                                int         split_k)
{
    void* ws = nullptr;
    if (split_k > 1) {
        // sizes first: no launch and no symbol lookup for a call that cannot fit
        if (m <= 0 || n <= 0)
            return hipErrorInvalidValue;
        const size_t need = flashllm_workspace_bytes(m, n, split_k);
        if (need > FLASHLLM_STATIC_WORKSPACE_BYTES) {
            std::fprintf(stderr,
                         "flashllm_spmm_splitk_static: Split_K*M*N*2 = %zu bytes exceeds the library's fixed slab storage of %u bytes; "
                         "use a smaller Split_K or flashllm_spmm_splitk with a workspace of your own\n",
                         need, FLASHLLM_STATIC_WORKSPACE_BYTES);
            return hipErrorInvalidValue;
        }
        const int rc = flashllm_hip_static_workspace(&ws);
        if (rc)
            return rc;
    }
    return flashllm_spmm_splitk(stream, a, comp, offs, b, c, m, n, k, ws, split_k);
}

int flashllm_device_tile_offsets(void* stream, const void* a, int m, int k, int* offs, long long* nnz_padded)
{
    if (!a || !offs || (reinterpret_cast<uintptr_t>(a) & 15u))
        return FLASHLLM_E_ARG;
    if (m <= 0 || k <= 0 || m % 128 || k % 64)
        return FLASHLLM_E_SHAPE;
    int rc = flashllm_hip_launch_tile_offsets(stream, a, m, k, offs);
    if (rc || !nnz_padded)
        return rc;
    const size_t tiles   = static_cast<size_t>(m / 128) * (k / 64);
    int          vectors = 0;
    hipStream_t  s       = static_cast<hipStream_t>(stream);
    hipError_t   e       = hipMemcpyAsync(&vectors, offs + tiles, sizeof(int), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess)
        e = hipStreamSynchronize(s);
    if (e != hipSuccess)
        return static_cast<int>(e);
    *nnz_padded = 4LL * vectors;
    return 0;
}

int flashllm_device_compress(void* stream, const void* a, int m, int k, const int* offs, void* comp)
{
    if (!a || !offs || !comp || (reinterpret_cast<uintptr_t>(a) & 15u) || (reinterpret_cast<uintptr_t>(comp) & 15u))
        return FLASHLLM_E_ARG;
    if (m <= 0 || k <= 0 || m % 128 || k % 64)
        return FLASHLLM_E_SHAPE;
    return flashllm_hip_launch_encode(stream, a, m, k, offs, comp);
}

int flashllm_device_compress_status(void* stream, unsigned int* status)
{
    if (!status)
        return hipErrorInvalidValue;
    return flashllm_hip_encode_status(stream, status);
}

size_t flashllm_workspace_bytes(int m, int n, int split_k)
{
    if (split_k <= 1 || m <= 0 || n <= 0)
        return 0;
    return static_cast<size_t>(split_k) * m * n * sizeof(uint16_t);
}

int flashllm_splitk_heuristic(int m, int n, int k)
{
    if (m <= 0 || k <= 0 || n <= 0 || m % 128 || k % 64)
        return 1;
    const int kt = k / 64;
    if (n % 128 == 0) {
        // Wide B: the slice's tiles at the time of a step, and what a slab costs: M*N halfs written and read at about
        // 6 TB/s, beside the second launch (3 us).
        const double slab_cost = 4e-6 / 6.0 * m * n;
        int          best      = 1;
        double       best_cost = 1e30;
        for (int s = 1; s <= 32 && s <= kt; s++) {
            const int    longest = (kt - 1) / s + 1;
            const double step    = runs_per_slice(m, n, k, s) == 1 ? flashllm_hip_wide_b_step(n, m, s) : 0.6;
            const double cost    = longest * step + (s > 1 ? 3.0 + s * slab_cost : 0.0);
            if (cost < best_cost) {
                best_cost = cost;
                best      = s;
            }
        }
        return best;
    }
    int    best      = 1;
    double best_cost = 1e30;
    for (int s = 1; s <= 32 && s <= kt; s++) {  // workspace sizes in existing callers assume at most 32 slabs
        if (s > 1 && !one_round(m, s, 1))
            break;
        const double cost = stream_cost(m, n, k, s, waves_per_slice(m, n, k, s));
        if (cost < best_cost) {
            best_cost = cost;
            best      = s;
        }
    }
    return best;
}

// The four pruned linears of a decoder layer, in the order and with the Split_K fallbacks of the
// reference's FasterTransformer call sites (third_party/ft.patch:512-525, :615-633, :1247-1261,
// :1328-1340, :1444-1456, :1508-1521).
int flashllm_decoder_layer_linears(void*                         stream,
                                   const flashllm_decoder_layer* layer,
                                   const void*                   x,
                                   void*                         qkv_out,
                                   void*                         attn_in,
                                   void*                         attn_out,
                                   void*                         ffn_mid,
                                   void*                         y,
                                   int                           tokens,
                                   void*                         ws)
{
    if (!layer || !x || !qkv_out || !attn_out || !ffn_mid || !y)
        return hipErrorInvalidValue;
    const flashllm_sparse_weight& q = layer->qkv;
    const flashllm_sparse_weight& o = layer->attn_out;
    const flashllm_sparse_weight& f1 = layer->ffn1;
    const flashllm_sparse_weight& f2 = layer->ffn2;
    const int hidden = q.k;
    if (o.k != hidden || q.m < hidden || f1.k != o.m || f2.k != f1.m || hidden % 8 || q.m % 8)
        return hipErrorInvalidValue;
    auto split = [&](const flashllm_sparse_weight& w, int limit) {
        if (tokens > limit)
            return 1;
        return w.split_k > 0 ? w.split_k : flashllm_splitk_heuristic(w.m, tokens, w.k);
    };
    auto linear = [&](const flashllm_sparse_weight& w, const void* in, int ld_in, void* out, int limit, int relu) {
        return spmm_splitk_ldb(stream, w.nz_weights, w.tile_offsets, in, ld_in, out, w.m, tokens, w.k, ws, split(w, limit), relu);
    };
    int rc = linear(q, x, hidden, qkv_out, 64, 0);
    if (rc)
        return rc;
    // The attention-output linear multiplies the first `hidden` rows of every column of qkv_out: it reads them
    // where they are (columns q.m halfs apart).  A caller that also wants them contiguous passes attn_in.
    if (attn_in) {
        rc = flashllm_hip_launch_take_rows(stream, attn_in, qkv_out, hidden, tokens, q.m);
        if (rc)
            return rc;
    }
    rc = linear(o, qkv_out, q.m, attn_out, 64, 0);
    if (rc)
        return rc;
    // FFN1's ReLU rides in whatever stores its sums: the reduction, or the product itself when there is none
    rc = linear(f1, attn_out, f1.k, ffn_mid, 128, 1);
    if (rc)
        return rc;
    return linear(f2, ffn_mid, f2.k, y, 128, 0);
}

}  // extern "C"

hipError_t SpMM_SplitK_API(hipStream_t  stream,
                           const half*  A,
                           const uint4* Compressed_A,
                           const int*   TileOffsets,
                           const half*  B,
                           half*        C,
                           const int    M_Global,
                           const int    N_Global,
                           const int    K_Global,
                           half*        Reduction_Workspace,
                           int          Split_K)
{
    return static_cast<hipError_t>(flashllm_spmm_splitk(
        stream, A, Compressed_A, TileOffsets, B, C, M_Global, N_Global, K_Global, Reduction_Workspace, Split_K));
}

namespace {
int init_or_exit(int rc)
{
    if (rc == FLASHLLM_E_NOMEM) {
        std::printf("InitSparseMatrixA: Error in malloc memory from host memory!\n");
        std::exit(-1);
    }
    if (rc < 0)
        std::fprintf(stderr, "InitSparseMatrixA: rejected (code %d): M must be a multiple of 128 and K of 64\n", rc);
    return rc;
}
}  // namespace

int InitSparseMatrixA_API(half* A_h, int M, int /*N*/, int K, uint32_t** Compressed_A, int** TileOffsets)
{
    return init_or_exit(
        flashllm_init_sparse_matrix_a(reinterpret_cast<const uint16_t*>(A_h), M, K, Compressed_A, TileOffsets));
}

int InitSparseMatrixA_API_NoReorder(half* A_h, int M, int /*N*/, int K, uint32_t** Compressed_A, int** TileOffsets)
{
    return init_or_exit(flashllm_init_sparse_matrix_a_noreorder(
        reinterpret_cast<const uint16_t*>(A_h), M, K, Compressed_A, TileOffsets));
}
