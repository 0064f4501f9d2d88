// C ABI of the gfx950 GPT-2 ops around the attention path (declared in
// include/gpt_hip_ops.h): argument validation, launches of the matrix products
// (ops_gemm.hip; the BLAS libraries for the shapes it does not take) and of the
// element-wise / normalisation / reduction kernels (ops_kernels.hip), the
// workspaces, status codes.
//
// The reference's op methods return void and abort on any runtime error
// (src/backend/cuda/utils/cuda_utils.cuh:21-34); here every entry point returns
// a status and keeps a per-thread message.
#include "../../include/gpt_hip_ops.h"
#include "ops_internal.h"

#include <hip/hip_runtime.h>
#include <hipblaslt/hipblaslt.h>
#include <rocblas/rocblas.h>

#include <atomic>
#include <math.h>
#include <mutex>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

int check_device(const char *op)
{
    int n = 0;
    const hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n <= 0)
        return fail(GPT_HIP_OPS_ENODEV, "%s: no HIP device (%s)", op,
                    e != hipSuccess ? hipGetErrorString(e) : "device count is 0");
    return 0;
}

int launched(const char *op, hipError_t e)
{
    if (e != hipSuccess)
        return fail(GPT_HIP_OPS_ELAUNCH, "%s: launch failed: %s", op, hipGetErrorString(e));
    return 0;
}

// Rows (B * T) of a [B, T, n] tensor, validated: non-negative, grid- and
// index-sized (rows < 2^31, rows * n < 2^40).
int check_rows(const char *op, int B, int T, long long n, long *rows)
{
    if (B < 0 || T < 0 || n <= 0)
        return fail(GPT_HIP_OPS_EINVAL, "%s: invalid shape B=%d T=%d width=%lld", op, B, T, n);
    const long long r = (long long)B * T;
    if (r >= (1LL << 31) || r * n >= (1LL << 40))
        return fail(GPT_HIP_OPS_ERANGE, "%s: tensor too large (B=%d T=%d width=%lld)", op, B, T, n);
    *rows = (long)r;
    return 0;
}

// ---------------------------------------------------------------- rocBLAS

constexpr int kMaxDevices = 64;
std::mutex g_blas_mu;
rocblas_handle g_blas[kMaxDevices] = {};

// One rocBLAS handle per device, created on first use with that device
// current; atomics are disallowed so that every GEMM is deterministic.
int blas_for(const char *op, hipStream_t st, rocblas_handle *out)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
        return fail(GPT_HIP_OPS_ENODEV, "%s: no current HIP device", op);
    std::lock_guard<std::mutex> lock(g_blas_mu);
    if (!g_blas[dev])
    {
        rocblas_handle h = nullptr;
        if (rocblas_create_handle(&h) != rocblas_status_success)
            return fail(GPT_HIP_OPS_ELAUNCH, "%s: rocblas_create_handle failed", op);
        if (rocblas_set_atomics_mode(h, rocblas_atomics_not_allowed) != rocblas_status_success)
            return fail(GPT_HIP_OPS_ELAUNCH, "%s: rocblas_set_atomics_mode failed", op);
        g_blas[dev] = h;
    }
    if (rocblas_set_stream(g_blas[dev], st) != rocblas_status_success)
        return fail(GPT_HIP_OPS_ELAUNCH, "%s: rocblas_set_stream failed", op);
    *out = g_blas[dev];
    return 0;
}

// Row-major C[M x N] = alpha op(A) op(B) + beta C, op(A) [M x K], op(B)
// [K x N], leading dimensions in elements of the row-major storage. rocBLAS
// is column-major: the row-major product is the column-major C^T = op(B)^T
// op(A)^T, i.e. the same call with the operands swapped.
int gemm_rm(const char *op, rocblas_handle h, bool ta, bool tb, int M, int N, int K, float alpha, const float *A,
            int lda, const float *B, int ldb, float beta, float *C, int ldc)
{
    const rocblas_status s =
        rocblas_sgemm(h, tb ? rocblas_operation_transpose : rocblas_operation_none,
                      ta ? rocblas_operation_transpose : rocblas_operation_none, N, M, K, &alpha, B, ldb, A, lda,
                      &beta, C, ldc);
    if (s != rocblas_status_success)
        return fail(GPT_HIP_OPS_ELAUNCH, "%s: rocblas_sgemm failed: %s", op, rocblas_status_to_string(s));
    return 0;
}

// ---------------------------------------------------------------- workspace

// hipMalloc is refused, and ends the capture, while any stream is captured in
// the default mode, but for a thread in this one.
struct RelaxedCapture
{
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// Workspaces, one buffer per (device, stream) and purpose, kept until
// gpt_hip_ops_release_workspaces or the process's end. Calls on one stream run
// in order, so they can share its buffers; calls on different streams get
// different ones. (A stream-ordered hipMallocAsync / hipFreeAsync pair per call
// measured ~10 us of GPU time per call here, more than the reductions it
// serves.) Reduction partials (at most 256 partial rows, a few MB) grow when a
// call needs more; at most kMaxWorkspaces of them. A graph holds the address that
// its calls were captured with: a buffer that a capture got is not freed any more
// (nothing tells when the graph is destroyed).
struct Workspace
{
    int dev;
    hipStream_t st;
    float *p;
    size_t floats;
    bool captured;
};
constexpr int kMaxWorkspaces = 64;
std::mutex g_ws_mu;
Workspace g_ws[kMaxWorkspaces];
int g_ws_n = 0;

int ws_get(const char *op, float **out, size_t floats, hipStream_t st)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess)
        return fail(GPT_HIP_OPS_ENODEV, "%s: no current HIP device", op);
    std::lock_guard<std::mutex> lock(g_ws_mu);
    Workspace *w = nullptr;
    for (int i = 0; i < g_ws_n; ++i)
        if (g_ws[i].dev == dev && g_ws[i].st == st)
            w = &g_ws[i];
    if (!w)
    {
        if (g_ws_n == kMaxWorkspaces)
            return fail(GPT_HIP_OPS_ENOMEM, "%s: more than %d (device, stream) workspaces", op, kMaxWorkspaces);
        w = &g_ws[g_ws_n++];
        *w = Workspace{dev, st, nullptr, 0, false};
    }
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess)
        (void)hipGetLastError();
    const bool capturing = cs != hipStreamCaptureStatusNone;
    if (w->floats < floats)
    {
        const RelaxedCapture relaxed;
        if (w->p && (w->captured || capturing))
        {
            // left to the graph, or to work queued before a capture that cannot
            // wait for it; at least twice the size takes its place, so that all
            // that are left come to less than the last
            floats = floats > 2 * w->floats ? floats : 2 * w->floats;
        }
        else if (w->p)
        {
            // the old buffer may still be read by work queued on this stream
            if (hipStreamSynchronize(st) != hipSuccess || hipFree(w->p) != hipSuccess)
                return fail(GPT_HIP_OPS_ELAUNCH, "%s: workspace release failed", op);
        }
        w->p = nullptr;
        w->floats = 0;
        w->captured = false;
        void *q = nullptr;
        const hipError_t e = hipMalloc(&q, floats * sizeof(float));
        if (e != hipSuccess)
            return fail(GPT_HIP_OPS_ENOMEM, "%s: workspace of %zu bytes: %s", op, floats * sizeof(float),
                        hipGetErrorString(e));
        w->p = static_cast<float *>(q);
        w->floats = floats;
    }
    w->captured |= capturing;
    *out = w->p;
    return 0;
}

// A split product's tickets and partial tiles, 32 MB that never grow, for the
// eager calls of a stream or for one capture on it. A graph has one of its own,
// since it may be replayed on any stream, beside eager calls on the one that it
// was captured on, and keeps it: nothing tells when it is destroyed. At most
// kMaxSplit of either kind on a device, in a table of their own.
struct SplitWorkspace
{
    hipStream_t st;
    unsigned long long capture;
    float *p;
};
constexpr int kMaxSplit = 16;
SplitWorkspace g_split[2][kMaxDevices][kMaxSplit];  // [captured] (g_ws_mu); p = null: free

// A new one, its tickets cleared on *st, or where st is null (a captured stream,
// whose graph would clear them again on every replay, 5 us) by work that has
// ended. Null where there is no memory.
float *new_split_workspace(const hipStream_t *st)
{
    const RelaxedCapture relaxed;
    void *q = nullptr;
    hipError_t e = hipMalloc(&q, (gpt_ops::gemm::kMaxTickets + gpt_ops::gemm::kPartFloats) * sizeof(float));
    if (e != hipSuccess)
    {
        (void)hipGetLastError();
        return nullptr;
    }
    hipStream_t own = nullptr;
    if (!st)
        e = hipStreamCreateWithFlags(&own, hipStreamNonBlocking);
    if (e == hipSuccess)
        e = gpt_ops::launch_fill_const(static_cast<float *>(q), gpt_ops::gemm::kMaxTickets, 0.f, st ? *st : own);
    if (own)
    {
        const hipError_t sync = hipStreamSynchronize(own);
        e = e == hipSuccess ? sync : e;
        (void)hipStreamDestroy(own);
    }
    if (e == hipSuccess)
        return static_cast<float *>(q);
    (void)hipGetLastError();
    (void)hipFree(q);
    return nullptr;
}

// Tickets and partial tiles for a split product on `st`; false where there are
// none to be had: on hipStreamPerThread, whose handle names a stream of each
// thread, or when memory or table entries have run out. *capturing: whether the
// stream is being captured.
bool split_workspace(float **part, int **ticket, bool *capturing, hipStream_t st)
{
    using namespace gpt_ops::gemm;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    *capturing = true;
    if (hipStreamGetCaptureInfo(st, &cs, &id) != hipSuccess)
    {
        (void)hipGetLastError();
        return false;
    }
    *capturing = cs != hipStreamCaptureStatusNone;
    int dev = 0;
    if ((!*capturing && st == hipStreamPerThread) || hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
        return false;
    std::lock_guard<std::mutex> lock(g_ws_mu);
    SplitWorkspace *w = nullptr, *free = nullptr;
    for (SplitWorkspace &e : g_split[*capturing][dev])
    {
        if (e.p && e.st == st && (!*capturing || e.capture == id))
            w = &e;
        if (!e.p && !free)
            free = &e;
    }
    if (!w)
    {
        if (!free)
            return false;
        float *const q = new_split_workspace(*capturing ? nullptr : &st);
        if (!q)
            return false;
        w = free;
        *w = SplitWorkspace{st, id, q};
    }
    *ticket = reinterpret_cast<int *>(w->p);
    *part = w->p + kMaxTickets;
    return true;
}

// ---------------------------------------------------------------- hipBLASLt

// The library's own kernels (ops_gemm.hip) take every product whose rows are
// 16-byte aligned multiples of 4 floats and that they finish first by their
// time model, against 7 us plus 7.2 us per GFLOP, but 10.5 us at least except for
// weight gradients, for the BLAS libraries. The 10.5 us are the libraries' host
// time: a call takes 12 us on the host, here 5 to 6, and the first one of every new
// row count, as each step of generating makes them, 212 us on hipBLASLt for its
// plan. In a captured graph, where that time is paid once, small products are
// faster on the libraries (77 x 768 x 768: the kernels alone 6 us, here 8.6).
// With the host time counted, over 224 sizes of each form from 1 to 4096 rows, the
// rule's choices take 0.73 (forward), 0.81 (grad_y w^T) and 0.89 (x^T grad_y) of
// the libraries' time in the geometric mean, and are more than 8 % slower in 14, 10
// and 23 of them: mostly between the sizes of gemm_rows_kernel and those that fill
// the card with tiles (384 x 768 x 2304 31 against 19 us, 1024 rows of 3072 x 768
// 53 against 43, x^T grad_y of 1024 x 1024 over 1536 rows 47 against 29). At 4096
// rows: 768 x 3072 110 against 152 us. The model is of operands in cache.
// Weights that come from memory, as while generating, cost the libraries more (77
// rows, GPT-2's four linear layers: 57 us and 8 for bias and GELU passes, against
// 50), so up to 128 rows this library's kernel may be modelled 1.3 times slower;
// weight gradients of few rows are modelled low, so there it has to be 0.95 times.
// Between the two libraries a fixed rule decides (use_lt): hipBLASLt's fp32
// kernels win where the row-major product has at most 1024 columns and for the
// weight gradients x^T grad_y, and fuse the linear layer's bias (and GELU) into
// their epilogue; rocBLAS wins on the wide products. Every algorithm is fixed
// per shape, so results are bitwise reproducible. One hipBLASLt plan
// (descriptor, layouts, heuristic algorithm) per (device, shape, transposes,
// epilogue), built on first use and kept; rocBLAS takes any shape hipBLASLt has
// no plan for. (A product that splits k takes another kernel, and with it other
// bits, where it gets no split workspace.)
struct LtPlan
{
    int dev;
    bool ta, tb;
    int M, N, K, lda, ldb, ldc;
    int epi;  // 0 none, 1 + bias, 2 + bias with GELU (pre-activation to aux)
    bool ok;
    hipblasLtMatmulDesc_t desc;
    hipblasLtMatrixLayout_t la, lb, lc;
    hipblasLtMatmulAlgo_t algo;
    size_t ws;  // always 0: only workspace-free algorithms are planned
};
constexpr int kMaxPlans = 256;
std::mutex g_lt_mu;
hipblasLtHandle_t g_lt[kMaxDevices] = {};
LtPlan g_plans[kMaxPlans];
int g_nplans = 0;

// Plan for row-major C[M x N] = op(A) op(B) (+ bias, GELU) on the current
// device, or nullptr when hipBLASLt has none (the caller falls back to
// rocBLAS). Called with g_lt_mu held.
LtPlan *lt_plan(int dev, bool ta, bool tb, int M, int N, int K, int lda, int ldb, int ldc, int epi)
{
    for (int i = 0; i < g_nplans; ++i)
    {
        LtPlan &q = g_plans[i];
        if (q.dev == dev && q.ta == ta && q.tb == tb && q.M == M && q.N == N && q.K == K && q.lda == lda &&
            q.ldb == ldb && q.ldc == ldc && q.epi == epi)
            return q.ok ? &q : nullptr;
    }
    if (g_nplans == kMaxPlans || dev < 0 || dev >= kMaxDevices)
        return nullptr;
    if (!g_lt[dev])
    {
        if (hipblasLtCreate(&g_lt[dev]) != HIPBLAS_STATUS_SUCCESS)
        {
            g_lt[dev] = nullptr;
            return nullptr;
        }
    }
    LtPlan &q = g_plans[g_nplans++];
    q = LtPlan{dev, ta, tb, M, N, K, lda, ldb, ldc, epi, false, nullptr, nullptr, nullptr, nullptr, {}, 0};
    // column-major view: C^T [N x M] = op(B)^T [N x K] op(A)^T [K x M]
    const hipblasOperation_t opa = tb ? HIPBLAS_OP_T : HIPBLAS_OP_N, opb = ta ? HIPBLAS_OP_T : HIPBLAS_OP_N;
    const uint32_t ep = epi == 0 ? HIPBLASLT_EPILOGUE_DEFAULT
                                 : epi == 1 ? HIPBLASLT_EPILOGUE_BIAS : HIPBLASLT_EPILOGUE_GELU_AUX_BIAS;
    const int32_t f32 = HIP_R_32F;
    const int64_t ld_aux = ldc;
    if (hipblasLtMatmulDescCreate(&q.desc, HIPBLAS_COMPUTE_32F, HIP_R_32F) != HIPBLAS_STATUS_SUCCESS ||
        hipblasLtMatmulDescSetAttribute(q.desc, HIPBLASLT_MATMUL_DESC_TRANSA, &opa, sizeof(opa)) ||
        hipblasLtMatmulDescSetAttribute(q.desc, HIPBLASLT_MATMUL_DESC_TRANSB, &opb, sizeof(opb)) ||
        hipblasLtMatmulDescSetAttribute(q.desc, HIPBLASLT_MATMUL_DESC_EPILOGUE, &ep, sizeof(ep)))
        return nullptr;
    if (epi >= 1 && hipblasLtMatmulDescSetAttribute(q.desc, HIPBLASLT_MATMUL_DESC_BIAS_DATA_TYPE, &f32, sizeof(f32)))
        return nullptr;
    if (epi == 2 &&
        (hipblasLtMatmulDescSetAttribute(q.desc, HIPBLASLT_MATMUL_DESC_EPILOGUE_AUX_LD, &ld_aux, sizeof(ld_aux)) ||
         hipblasLtMatmulDescSetAttribute(q.desc, HIPBLASLT_MATMUL_DESC_EPILOGUE_AUX_DATA_TYPE, &f32, sizeof(f32))))
        return nullptr;
    if (hipblasLtMatrixLayoutCreate(&q.la, HIP_R_32F, tb ? K : N, tb ? N : K, ldb) ||
        hipblasLtMatrixLayoutCreate(&q.lb, HIP_R_32F, ta ? M : K, ta ? K : M, lda) ||
        hipblasLtMatrixLayoutCreate(&q.lc, HIP_R_32F, N, M, ldc))
        return nullptr;
    hipblasLtMatmulPreference_t pref;
    if (hipblasLtMatmulPreferenceCreate(&pref))
        return nullptr;
    // Only algorithms that need no workspace: the split-K / stream-K kinds
    // that do were seen to fail at launch with an internal error on some
    // shapes, and their cross-workgroup reductions need not be reproducible.
    size_t wmax = 0;
    constexpr int kAsk = 32;
    hipblasLtMatmulHeuristicResult_t res[kAsk];
    int n = 0;
    const bool asked =
        !hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &wmax, sizeof(wmax)) &&
        !hipblasLtMatmulAlgoGetHeuristic(g_lt[dev], q.desc, q.la, q.lb, q.lc, q.lc, pref, kAsk, res, &n);
    hipblasLtMatmulPreferenceDestroy(pref);
    if (!asked)
        return nullptr;
    int pick = -1;  // the heuristic's first workspace-free choice
    for (int i = 0; i < n && pick < 0; ++i)
        if (res[i].state == HIPBLAS_STATUS_SUCCESS && res[i].workspaceSize == 0)
            pick = i;
    if (pick < 0)
        return nullptr;
    q.algo = res[pick].algo;
    q.ws = 0;
    q.ok = true;
    return &q;
}

// Row-major C[M x N] = alpha op(A) op(B) + beta C, with the epilogue: epi 1
// adds bias[n] to every row; epi 2 also writes GELU of that to D and the
// biased product to aux. Returns 1 when hipBLASLt has no plan (nothing was
// enqueued), 0 on success, a GPT_HIP_OPS_E* code on failure.
int lt_gemm(const char *op, hipStream_t st, bool ta, bool tb, int M, int N, int K, float alpha, const float *A,
            int lda, const float *B, int ldb, float beta, float *C, int ldc, int epi, const float *bias, float *aux)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess)
        return fail(GPT_HIP_OPS_ENODEV, "%s: no current HIP device", op);
    std::lock_guard<std::mutex> lock(g_lt_mu);
    LtPlan *q = lt_plan(dev, ta, tb, M, N, K, lda, ldb, ldc, epi);
    if (!q)
        return 1;
    if (epi >= 1 &&
        hipblasLtMatmulDescSetAttribute(q->desc, HIPBLASLT_MATMUL_DESC_BIAS_POINTER, &bias, sizeof(bias)))
        return fail(GPT_HIP_OPS_ELAUNCH, "%s: hipBLASLt bias attribute", op);
    if (epi == 2 &&
        hipblasLtMatmulDescSetAttribute(q->desc, HIPBLASLT_MATMUL_DESC_EPILOGUE_AUX_POINTER, &aux, sizeof(aux)))
        return fail(GPT_HIP_OPS_ELAUNCH, "%s: hipBLASLt aux attribute", op);
    const hipblasStatus_t s = hipblasLtMatmul(g_lt[dev], q->desc, &alpha, B, q->la, A, q->lb, &beta, C, q->lc, C,
                                              q->lc, &q->algo, nullptr, 0, st);
    if (s != HIPBLAS_STATUS_SUCCESS)
    {
        q->ok = false;  // this shape goes to rocBLAS from now on
        // An accumulating product (beta != 0) is not run again on rocBLAS:
        // if the failed call had enqueued any work, a second run would add
        // the product twice. An overwriting one (beta = 0) is safe to redo.
        if (beta != 0.f)
            return fail(GPT_HIP_OPS_ELAUNCH, "%s: hipblasLtMatmul failed (%d) on an accumulating product", op,
                        (int)s);
        return 1;
    }
    return 0;
}

bool use_lt(bool ta, int N) { return ta || N <= 1024; }

// Shapes that the library's own kernel has been considered for, with their launch
// choices, and whether one has been launched. Entries stay where they are; past
// kOwnFull shapes choices are made anew for each call, and not counted.
struct OwnPlan
{
    int M, N, K;
    bool ta, tb;
    std::atomic<bool> ran;
    gpt_ops::gemm::Choice c, plain;  // plain: the best without a split
};
constexpr int kOwnPlans = 1024, kOwnFull = 768;
std::mutex g_own_mu;
OwnPlan g_own[kOwnPlans];  // K = 0: free; a shape's entry is at its hash or after
int g_nown = 0;
std::atomic<int> g_own_ran{0};

// The plan of a shape; `spare` where the table is full.
OwnPlan *own_plan(int M, int N, int K, bool ta, bool tb, OwnPlan *spare)
{
    std::lock_guard<std::mutex> lock(g_own_mu);
    unsigned h = ((unsigned)M * 0x9E3779B1u) ^ ((unsigned)N * 0x85EBCA77u) ^ ((unsigned)K * 0xC2B2AE3Du) ^ (ta ? 1u : 0u) ^ (tb ? 2u : 0u);
    h = (h ^ h >> 15) % kOwnPlans;
    for (; g_own[h].K; h = (h + 1) % kOwnPlans)
    {
        OwnPlan &p = g_own[h];
        if (p.M == M && p.N == N && p.K == K && p.ta == ta && p.tb == tb)
            return &p;
    }
    OwnPlan *p = spare;
    if (g_nown < kOwnFull)
    {
        p = &g_own[h];
        ++g_nown;
    }
    p->M = M, p->N = N, p->K = K, p->ta = ta, p->tb = tb;
    p->ran = p == spare;
    p->c = gpt_ops::gemm::choose(M, N, K, ta, tb, true);
    p->plain = p->c.splits > 1 ? gpt_ops::gemm::choose(M, N, K, ta, tb, false) : p->c;
    return p;
}

// Whether the handle is there that a product on the libraries takes: they cannot
// make one while a stream is captured.
bool library_ready(bool ta, int N)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
        return false;
    if (use_lt(ta, N))
    {
        std::lock_guard<std::mutex> lock(g_lt_mu);
        return g_lt[dev];
    }
    std::lock_guard<std::mutex> lock(g_blas_mu);
    return g_blas[dev];
}

// Row-major C [M x N] = op(A) op(B) (+ bias, act = GELU(C)), or C += op(A)
// op(B), on the library's own kernel. Returns 1 when it does not take the
// operands or would be slower (nothing was enqueued), 0 or a GPT_HIP_OPS_E* code.
int own_gemm(const char *op, hipStream_t st, bool ta, bool tb, int M, int N, int K, const float *A, const float *B,
             bool add, float *C, const float *bias = nullptr, float *act = nullptr)
{
    if (!gpt_ops::gemm::fits(A, B, C, act, M, N, K, ta, tb))
        return 1;
    OwnPlan spare;
    OwnPlan *const plan = own_plan(M, N, K, ta, tb, &spare);
    gpt_ops::gemm::Choice c = plan->c;
    // (rocBLAS, on the wide products, needs a pass of its own for the bias)
    float library_us = 7.f + 7.2e-9f * 2.f * M * N * K;
    if (!ta && library_us < 10.5f)
        library_us = 10.5f;
    library_us += bias && !use_lt(ta, N) ? 3.f : 0.f;
    const float limit_us = library_us * (ta ? 0.95f : M <= 128 ? 1.3f : 1.f);
    if (c.us > limit_us)
        return 1;
    float *part = nullptr;
    int *ticket = nullptr;
    bool capturing = false;
    if (c.splits > 1 && !split_workspace(&part, &ticket, &capturing, st))
    {
        // unsplit, unless the libraries are faster then (x^T grad_y of 768 x 768
        // over 4096 rows: 125 us against 42)
        c = plan->plain;
        if (c.us > limit_us && (!capturing || library_ready(ta, N)))
            return 1;
    }
    const int rc = launched(op, gpt_ops::gemm::run(A, B, C, bias, act, M, N, K, ta, tb, add, c, part, ticket, st));
    if (rc == 0 && !plan->ran.exchange(true))
        ++g_own_ran;
    return rc;
}

// Row-major C = op(A) op(B), or C +=: this library's kernel, or hipBLASLt
// where use_lt says so and it has a plan, or rocBLAS.
int gemm(const char *op, hipStream_t st, bool ta, bool tb, int M, int N, int K, const float *A, const float *B,
         bool add, float *C)
{
    int rc = own_gemm(op, st, ta, tb, M, N, K, A, B, add, C);
    if (rc != 1)
        return rc;
    const int lda = ta ? M : K, ldb = tb ? K : N;
    const float beta = add ? 1.f : 0.f;
    if (use_lt(ta, N))
    {
        rc = lt_gemm(op, st, ta, tb, M, N, K, 1.f, A, lda, B, ldb, beta, C, N, 0, nullptr, nullptr);
        if (rc != 1)
            return rc;
    }
    rocblas_handle h;
    if (int r = blas_for(op, st, &h))
        return r;
    return gemm_rm(op, h, ta, tb, M, N, K, 1.f, A, lda, B, ldb, beta, C, N);
}

hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

}  // namespace

extern "C" {

int gpt_hip_embedding_forward_f32(float *y, const float *wte, const float *wpe, const int *input_tokens,
                                  int batch_size, int seq_len, int hidden_size, int vocab_rows, void *stream)
{
    static const char *op = "gpt_hip_embedding_forward_f32";
    long rows = 0;
    if (int rc = check_rows(op, batch_size, seq_len, hidden_size, &rows))
        return rc;
    if (rows == 0)
        return 0;
    if (!y || !wte || !wpe || !input_tokens)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    return launched(op, gpt_ops::launch_embedding_fwd(y, wte, wpe, input_tokens, batch_size, seq_len, hidden_size,
                                                      vocab_rows, as_stream(stream)));
}

int gpt_hip_embedding_backward_f32(float *grad_wte, float *grad_wpe, const float *grad_y, const int *input_tokens,
                                   int batch_size, int seq_len, int hidden_size, int vocab_rows, void *stream)
{
    static const char *op = "gpt_hip_embedding_backward_f32";
    long rows = 0;
    if (int rc = check_rows(op, batch_size, seq_len, hidden_size, &rows))
        return rc;
    if (rows == 0)
        return 0;
    if (!grad_wte || !grad_wpe || !grad_y || !input_tokens)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    return launched(op, gpt_ops::launch_embedding_bwd(grad_wte, grad_wpe, grad_y, input_tokens, batch_size, seq_len,
                                                      hidden_size, vocab_rows, as_stream(stream)));
}

int gpt_hip_unembedding_forward_f32(float *y, const float *x, const float *wte, int batch_size, int seq_len,
                                    int hidden_size, int vocab_size_padded, void *stream)
{
    static const char *op = "gpt_hip_unembedding_forward_f32";
    long rows = 0;
    if (int rc = check_rows(op, batch_size, seq_len, (long long)hidden_size + vocab_size_padded, &rows))
        return rc;
    if (hidden_size <= 0 || vocab_size_padded <= 0)
        return fail(GPT_HIP_OPS_EINVAL, "%s: hidden_size %d, vocab_size_padded %d", op, hidden_size,
                    vocab_size_padded);
    if (rows == 0)
        return 0;
    if (!y || !x || !wte)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    // y [M x Vp] = x [M x C] wte^T
    return gemm(op, as_stream(stream), false, true, (int)rows, vocab_size_padded, hidden_size, x, wte, false, y);
}

int gpt_hip_unembedding_backward_f32(float *grad_x, float *grad_wte, const float *grad_y, const float *x,
                                     const float *wte, int batch_size, int seq_len, int hidden_size,
                                     int vocab_size_padded, void *stream)
{
    static const char *op = "gpt_hip_unembedding_backward_f32";
    long rows = 0;
    if (int rc = check_rows(op, batch_size, seq_len, (long long)hidden_size + vocab_size_padded, &rows))
        return rc;
    if (hidden_size <= 0 || vocab_size_padded <= 0)
        return fail(GPT_HIP_OPS_EINVAL, "%s: hidden_size %d, vocab_size_padded %d", op, hidden_size,
                    vocab_size_padded);
    if (rows == 0)
        return 0;
    if (!grad_x || !grad_wte || !grad_y || !x || !wte)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    const hipStream_t st = as_stream(stream);
    const int M = (int)rows, C = hidden_size, V = vocab_size_padded;
    // grad_x [M x C] = grad_y [M x V] wte [V x C]
    if (int rc = gemm(op, st, false, false, M, C, V, grad_y, wte, false, grad_x))
        return rc;
    // grad_wte [V x C] += grad_y^T [V x M] x [M x C]
    return gemm(op, st, true, false, V, C, M, grad_y, x, true, grad_wte);
}

int gpt_hip_layernorm_residual_forward_f32(float *y, float *means, float *vars, float *x, const float *residual,
                                           const float *gamma, const float *beta, int batch_size, int seq_len,
                                           int hidden_size, void *stream)
{
    static const char *op = "gpt_hip_layernorm_residual_forward_f32";
    long rows = 0;
    if (int rc = check_rows(op, batch_size, seq_len, hidden_size, &rows))
        return rc;
    if (rows == 0)
        return 0;
    if (!y || !means || !vars || !x || !gamma || !beta)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    return launched(op, gpt_ops::launch_layernorm_fwd(y, means, vars, x, residual, gamma, beta, rows, hidden_size,
                                                      as_stream(stream)));
}

int gpt_hip_layernorm_residual_backward_f32(float *grad_x, float *grad_gamma, float *grad_beta, const float *grad_y,
                                            const float *grad_residual, const float *x, const float *means,
                                            const float *vars, const float *gamma, int batch_size, int seq_len,
                                            int hidden_size, void *stream)
{
    static const char *op = "gpt_hip_layernorm_residual_backward_f32";
    long rows = 0;
    if (int rc = check_rows(op, batch_size, seq_len, hidden_size, &rows))
        return rc;
    if (rows == 0)
        return 0;
    if (!grad_x || !grad_gamma || !grad_beta || !grad_y || !x || !means || !vars || !gamma)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    const hipStream_t st = as_stream(stream);
    float *ws = nullptr;
    if (int rc = ws_get(op, &ws, (size_t)gpt_ops::colsum_parts(rows) * 2 * hidden_size, st))
        return rc;
    return launched(op, gpt_ops::launch_layernorm_bwd(grad_x, grad_gamma, grad_beta, grad_y, grad_residual, x, means,
                                                      vars, gamma, rows, hidden_size, ws, st));
}

int gpt_hip_linear_activation_forward_f32(float *y, float *act, const float *x, const float *w, const float *b,
                                          int activation, int batch_size, int seq_len, int input_size,
                                          int output_size, void *stream)
{
    static const char *op = "gpt_hip_linear_activation_forward_f32";
    long rows = 0;
    if (int rc = check_rows(op, batch_size, seq_len, (long long)input_size + output_size, &rows))
        return rc;
    if (input_size <= 0 || output_size <= 0)
        return fail(GPT_HIP_OPS_EINVAL, "%s: input_size %d, output_size %d", op, input_size, output_size);
    if (rows == 0)
        return 0;
    if (!y || !x || !w || !b || (activation && !act))
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    const hipStream_t st = as_stream(stream);
    const int M = (int)rows, K = input_size, N = output_size;
    // y [M x N] = x [M x K] w [K x N] + b, bias and GELU in the epilogue of
    // this library's kernel or (use_lt) hipBLASLt's (D = act, pre-activation y
    // as the auxiliary output); on rocBLAS one pass adds the bias and writes
    // the GELU.
    int rc = own_gemm(op, st, false, false, M, N, K, x, w, false, y, b, activation ? act : nullptr);
    if (rc != 1)
        return rc;
    if (use_lt(false, N))
    {
        rc = activation ? lt_gemm(op, st, false, false, M, N, K, 1.f, x, K, w, N, 0.f, act, N, 2, b, y)
                        : lt_gemm(op, st, false, false, M, N, K, 1.f, x, K, w, N, 0.f, y, N, 1, b, nullptr);
        if (rc != 1)
            return rc;
    }
    // no hipBLASLt plan: rocBLAS GEMM, then + b (and GELU) in one pass
    rocblas_handle h;
    if (int rc = blas_for(op, st, &h))
        return rc;
    if (int rc = gemm_rm(op, h, false, false, M, N, K, 1.f, x, K, w, N, 0.f, y, N))
        return rc;
    return launched(op, gpt_ops::launch_bias_gelu(y, activation ? act : nullptr, b, rows, N, st));
}

int gpt_hip_linear_backward_f32(float *grad_x, float *grad_w, float *grad_b, const float *grad_y, const float *x,
                                const float *w, int batch_size, int seq_len, int input_size, int output_size,
                                void *stream)
{
    static const char *op = "gpt_hip_linear_backward_f32";
    long rows = 0;
    if (int rc = check_rows(op, batch_size, seq_len, (long long)input_size + output_size, &rows))
        return rc;
    if (input_size <= 0 || output_size <= 0)
        return fail(GPT_HIP_OPS_EINVAL, "%s: input_size %d, output_size %d", op, input_size, output_size);
    if (rows == 0)
        return 0;
    if (!grad_x || !grad_w || !grad_b || !grad_y || !x || !w)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    const hipStream_t st = as_stream(stream);
    const int M = (int)rows, K = input_size, N = output_size;
    // grad_x [M x K] = grad_y [M x N] w^T [N x K]
    if (int rc = gemm(op, st, false, true, M, K, N, grad_y, w, false, grad_x))
        return rc;
    // grad_w [K x N] += x^T [K x M] grad_y [M x N]
    if (int rc = gemm(op, st, true, false, K, N, M, x, grad_y, true, grad_w))
        return rc;
    float *ws = nullptr;
    if (int rc = ws_get(op, &ws, (size_t)gpt_ops::colsum_parts(rows) * N, st))
        return rc;
    return launched(op, gpt_ops::launch_bias_grad(grad_b, grad_y, rows, N, ws, st));
}

int gpt_hip_activation_backward_f32(float *grad_x, const float *grad_y, const float *x, int batch_size,
                                    int seq_len, int output_size, void *stream)
{
    static const char *op = "gpt_hip_activation_backward_f32";
    long rows = 0;
    if (int rc = check_rows(op, batch_size, seq_len, output_size, &rows))
        return rc;
    if (rows == 0)
        return 0;
    if (!grad_x || !grad_y || !x)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    return launched(op, gpt_ops::launch_gelu_bwd(grad_x, grad_y, x, rows * output_size, as_stream(stream)));
}

int gpt_hip_softmax_forward_f32(float *y, const float *x, int batch_size, int seq_len, int vocab_size,
                                int vocab_size_padded, void *stream)
{
    static const char *op = "gpt_hip_softmax_forward_f32";
    long rows = 0;
    if (int rc = check_rows(op, batch_size, seq_len, vocab_size_padded, &rows))
        return rc;
    if (vocab_size <= 0 || vocab_size > vocab_size_padded)
        return fail(GPT_HIP_OPS_EINVAL, "%s: vocab_size %d, vocab_size_padded %d", op, vocab_size,
                    vocab_size_padded);
    if (rows == 0)
        return 0;
    if (!y || !x)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    return launched(op, gpt_ops::launch_softmax_fwd(y, x, rows, vocab_size, vocab_size_padded, as_stream(stream)));
}

int gpt_hip_cross_entropy_softmax_backward_f32(float *grad_x, const float *y_softmax, const int *tokens_labels,
                                               int batch_size, int seq_len, int vocab_size, int vocab_size_padded,
                                               void *stream)
{
    static const char *op = "gpt_hip_cross_entropy_softmax_backward_f32";
    long rows = 0;
    if (int rc = check_rows(op, batch_size, seq_len, vocab_size_padded, &rows))
        return rc;
    if (vocab_size <= 0 || vocab_size > vocab_size_padded)
        return fail(GPT_HIP_OPS_EINVAL, "%s: vocab_size %d, vocab_size_padded %d", op, vocab_size,
                    vocab_size_padded);
    if (rows == 0)
        return 0;
    if (!grad_x || !y_softmax || !tokens_labels)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    return launched(op, gpt_ops::launch_ce_bwd(grad_x, y_softmax, tokens_labels, rows, vocab_size,
                                               vocab_size_padded, as_stream(stream)));
}

int gpt_hip_cross_entropy_loss_f32(float *loss, const float *y_softmax, const int *tokens_labels, int batch_size,
                                   int seq_len, int vocab_size_padded, void *stream)
{
    static const char *op = "gpt_hip_cross_entropy_loss_f32";
    long rows = 0;
    if (int rc = check_rows(op, batch_size, seq_len, vocab_size_padded, &rows))
        return rc;
    if (!loss)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (rows == 0)
        return 0;
    if (!y_softmax || !tokens_labels)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    return launched(op, gpt_ops::launch_ce_loss(loss, y_softmax, tokens_labels, rows, vocab_size_padded,
                                                as_stream(stream)));
}

int gpt_hip_adamw_step_f32(float *params, float *g, float *m, float *v, int size, float lr, float beta1,
                           float beta2, float eps, float weight_decay, int step, void *stream)
{
    static const char *op = "gpt_hip_adamw_step_f32";
    if (size < 0)
        return fail(GPT_HIP_OPS_EINVAL, "%s: size %d", op, size);
    if (size == 0)
        return 0;
    if (!params || !g || !m || !v)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    // bias corrections exactly as the CPU backend forms them (cpu_backend.cpp:519-520, 526-527)
    const float one_m_b1p = 1.0f - powf(beta1, (float)step);
    const float one_m_b2p = 1.0f - powf(beta2, (float)step);
    return launched(op, gpt_ops::launch_adamw(params, g, m, v, size, lr, beta1, beta2, eps, weight_decay, one_m_b1p,
                                              one_m_b2p, as_stream(stream)));
}

int gpt_hip_scale_and_clip_grad_f32(float *g, int size, float max_norm, int accum_steps, void *stream)
{
    static const char *op = "gpt_hip_scale_and_clip_grad_f32";
    if (size < 0 || accum_steps < 1)
        return fail(GPT_HIP_OPS_EINVAL, "%s: size %d, accum_steps %d", op, size, accum_steps);
    if (size == 0)
        return 0;
    if (!g)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    const hipStream_t st = as_stream(stream);
    float *ws = nullptr;
    if (int rc = ws_get(op, &ws, (size_t)gpt_ops::clip_parts(), st))
        return rc;
    return launched(op, gpt_ops::launch_scale_clip(g, size, max_norm, (float)accum_steps, ws, st));
}

int gpt_hip_fill_normal_f32(float *ptr, float mean, float stddev, size_t size, unsigned long long seed,
                            void *stream)
{
    static const char *op = "gpt_hip_fill_normal_f32";
    if (size == 0)
        return 0;
    if (!ptr)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    return launched(op, gpt_ops::launch_fill_normal(ptr, size, mean, stddev, seed, as_stream(stream)));
}

int gpt_hip_fill_const_f32(float *ptr, float value, size_t size, void *stream)
{
    static const char *op = "gpt_hip_fill_const_f32";
    if (size == 0)
        return 0;
    if (!ptr)
        return fail(GPT_HIP_OPS_ENULL, "%s: NULL pointer", op);
    if (int rc = check_device(op))
        return rc;
    return launched(op, gpt_ops::launch_fill_const(ptr, size, value, as_stream(stream)));
}

const char *gpt_hip_ops_last_error(void) { return g_err; }

int gpt_hip_ops_gemm_info(int *plans, int *tuned, int *blaslt_version)
{
    if (!plans || !tuned || !blaslt_version)
        return fail(GPT_HIP_OPS_ENULL, "gpt_hip_ops_gemm_info: NULL output");
    std::lock_guard<std::mutex> lock(g_lt_mu);
    int np = 0;
    for (int i = 0; i < g_nplans; ++i)
        np += g_plans[i].ok ? 1 : 0;
    *tuned = g_own_ran;
    *plans = np + *tuned;
    *blaslt_version = 0;
    for (int d = 0; d < kMaxDevices; ++d)
        if (g_lt[d])
        {
            int v = 0;
            if (hipblasLtGetVersion(g_lt[d], &v) == HIPBLAS_STATUS_SUCCESS)
                *blaslt_version = v;
            break;
        }
    return 0;
}

int gpt_hip_ops_release_workspaces(void)
{
    static const char *op = "gpt_hip_ops_release_workspaces";
    if (int rc = check_device(op))
        return rc;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess)
        return fail(GPT_HIP_OPS_ENODEV, "%s: no current HIP device", op);
    std::lock_guard<std::mutex> lock(g_ws_mu);
    const hipError_t e = hipDeviceSynchronize();
    if (e != hipSuccess)
        return fail(GPT_HIP_OPS_ELAUNCH, "%s: %s", op, hipGetErrorString(e));
    int keep = 0;
    for (int i = 0; i < g_ws_n; ++i)
    {
        if (g_ws[i].dev == dev && !g_ws[i].captured)
            (void)hipFree(g_ws[i].p);
        else
            g_ws[keep++] = g_ws[i];
    }
    g_ws_n = keep;
    if (dev >= 0 && dev < kMaxDevices)
        for (SplitWorkspace &w : g_split[0][dev])  // (a graph's may be replayed yet)
        {
            (void)hipFree(w.p);
            w = SplitWorkspace{};
        }
    return 0;
}

}  // extern "C"
