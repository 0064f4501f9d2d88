// Causal attention for any head size 1..256, any row length and any pointer
// alignment, forward and backward, on v_mfma_f32_16x16x4_f32. (head_dim 64 has
// kernels of its own, attn_fwd.hip and attn_bwd*.hip; it comes here for rows
// beyond their buffer ranges, for misaligned pointers and as path 1.)
//
// One workgroup per (b, h, 16 rows), 4 waves that take the 16-row blocks of the
// other operand in turn (keys for the forward and dQ, queries for dK and dV),
// operands straight from memory into registers, no barrier until the waves'
// partial results are merged through LDS in wave order. Rows of 16 and a
// 4-way split keep the card busy where (b, h) and rows are few, which is where
// these sizes are called (B = 2, T = 250, H = 6, d = 128: 192 workgroups of at
// most 4 blocks a wave); each block's operands are read by T / 32 workgroups
// on average, from the XCD's L2. No workspace, no atomics: results are bitwise
// reproducible. The backward recomputes S once for dQ and once for dK and dV (7
// products where a workspace of dS tiles would take 5).
//
// What bounds it: a wave's chain of memory round trips and MFMAs, 2048 cycles
// a block of the forward at d = 128. B = 2, T = 250, H = 6, d = 128, forward
// and backward: 19.2 ms with one thread per row, now 50 us (forward 11, dQ and D 16, dK and
// dV 22). A full card, B = 8, T = 1024, H = 6, d = 128: 142 and 622 us (91 TFLOP/s and,
// of five products, 52).
// Rows off 16 bytes (4-byte loads) past d = 128 spill up to 450 registers a lane: B = 2,
// T = 250, H = 6, d = 130 58 and 405 us, where d = 132 takes 14.6 and 44, and one thread
// per row took 6.8 and 25 ms.
#include "attn_common.h"
#include "attn_kernels.h"

#include <float.h>
#include <type_traits>

namespace gpt_attn {
namespace {

float softmax_scale(int d) { return 1.0f / sqrtf((float)d); }

constexpr int kRows = 16, kWaves = 4;

// Operand layouts for a head padded to 16 ND dimensions. Row fragment: lane
// (l16, kc) holds dimensions 16 u + 4 kc + e of row l16 (u < ND, e < 4): the
// A or B operand of MFMA (u, e), whose k index kc is dimension 16 u + 4 kc + e
// in both operands. Column fragment: lane (l16, kc) holds, of row 4 kc + r,
// the NU consecutive dimensions 16 NU g + NU l16 + u: the A operand of the
// product that sums over rows, whose B operand is a 16 x 16 result in its
// accumulator layout (row 4 kc + r of column l16 in register r).
template <int ND> struct Head
{
    static constexpr int NU = ND % 4 == 0 ? 4 : ND % 2 == 0 ? 2 : 1;
    // dimension of accumulator n, register r, lane group kc
    static __device__ __forceinline__ int dim(int n, int r, int kc) { return 16 * NU * (n / NU) + NU * (4 * kc + r) + n % NU; }
};

// 16 rows from `row` < T on of a [T][W] matrix whose head starts at `p`; rows
// past T read as zeros. The vector form reads through a buffer range, whose
// offsets have 31 bits (the host takes it where 16 rows fit); the scalar form
// has 64-bit addresses and reads row `row`'s first element where it would read
// nothing.
struct Rows
{
    rsrc_t r;
    const float *p;
    long W;
    int left;
    __device__ __forceinline__ float at(int row, int e, int d) const
    {
        const bool ok = row < left && e < d;
        const float v = p[ok ? row * W + e : 0];
        return ok ? v : 0.f;
    }
};
__device__ __forceinline__ Rows rows_of(const float *p, int row, int T, long W, int d)
{
    const int left = T - row < kRows ? T - row : kRows;
    const float *const first = p + (long)row * W;
    return Rows{make_rsrc(first, (uint32_t)(((left - 1) * W + d) * 4)), first, W, left};
}

template <int ND, bool VEC>
__device__ __forceinline__ void load_rows(float (&f)[ND][4], const Rows &rs, int d, int l16, int kc)
{
#pragma unroll
    for (int u = 0; u < ND; ++u)
    {
        const int e = 16 * u + 4 * kc;
        if (VEC)  // d is a multiple of 4
        {
            const uint32_t off = ((uint32_t)l16 * (uint32_t)rs.W + (uint32_t)e) * 4u;
            const float4 v = bload4(rs.r, e < d ? off : kNoBlock);
            f[u][0] = v.x, f[u][1] = v.y, f[u][2] = v.z, f[u][3] = v.w;
        }
        else
        {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                f[u][q] = rs.at(l16, e + q, d);
        }
    }
}

template <int ND, bool VEC>
__device__ __forceinline__ void load_cols(float (&f)[4][ND], const Rows &rs, int d, int l16, int kc)
{
    constexpr int NU = Head<ND>::NU;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int g = 0; g < ND / NU; ++g)
        {
            const int e = 16 * NU * g + NU * l16;
            const uint32_t off = ((uint32_t)(4 * kc + r) * (uint32_t)rs.W + (uint32_t)e) * 4u;
            float *const o = &f[r][g * NU];
            if (VEC && NU == 4)
            {
                const float4 v = bload4(rs.r, e < d ? off : kNoBlock);
                o[0] = v.x, o[1] = v.y, o[2] = v.z, o[3] = v.w;
            }
            else if (VEC && NU == 2)
            {
                const float2 v = bload2(rs.r, e < d ? off : kNoBlock);
                o[0] = v.x, o[1] = v.y;
            }
            else
            {
#pragma unroll
                for (int u = 0; u < NU; ++u)
                    o[u] = VEC ? bload1(rs.r, e + u < d ? off + 4u * u : kNoBlock) : rs.at(4 * kc + r, e + u, d);
            }
        }
}

// D[16 x 16] = A B over the head's dimensions, from row fragments; two chains.
template <int ND> __device__ __forceinline__ v4f dot_rows(const float (&a)[ND][4], const float (&b)[ND][4])
{
    v4f x = zero4(), y = zero4();
#pragma unroll
    for (int u = 0; u < ND; ++u)
    {
        x = mfma16(a[u][0], b[u][0], x);
        y = mfma16(a[u][1], b[u][1], y);
        x = mfma16(a[u][2], b[u][2], x);
        y = mfma16(a[u][3], b[u][3], y);
    }
    return x + y;
}

// acc += cols^T w, w a 16 x 16 result in its accumulator layout.
template <int ND> __device__ __forceinline__ void add_cols(v4f (&acc)[ND], const float (&c)[4][ND], v4f w)
{
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int n = 0; n < ND; ++n)
            acc[n] = mfma16(c[r][n], w[r], acc[n]);
}

// Merges the waves' accumulators (each times `mine`, its factor for the lane's
// row l16) through `red` (kMerge floats), wave w writing register w of every
// accumulator to out[row l16][dimension]. Returns whether a value that this
// lane stored is not finite.
constexpr int kMergeN = 8, kMerge = kWaves * kMergeN * 4 * 64;
template <int ND, bool VEC>
__device__ __forceinline__ bool merge_store(const v4f (&acc)[ND], float mine, float *red, float *out, long W, int d,
                                            bool row_ok, int w, int lane)
{
    constexpr int NU = Head<ND>::NU;
    const int l16 = lane & 15, kc = lane >> 4;
    bool bad = false;
#pragma unroll
    for (int n0 = 0; n0 < ND; n0 += kMergeN)
    {
        const int cnt = ND - n0 < kMergeN ? ND - n0 : kMergeN;
        __syncthreads();
#pragma unroll
        for (int n = 0; n < kMergeN; ++n)
            if (n < cnt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    red[((w * kMergeN + n) * 4 + r) * 64 + lane] = acc[(n0 + n) % ND][r] * mine;
        __syncthreads();
#pragma unroll
        for (int n = 0; n < kMergeN; n += NU)
            if (n < cnt)
            {
                float o[NU];
#pragma unroll
                for (int u = 0; u < NU; ++u)
                {
                    o[u] = red[((0 * kMergeN + n + u) * 4 + w) * 64 + lane];
#pragma unroll
                    for (int q = 1; q < kWaves; ++q)
                        o[u] += red[((q * kMergeN + n + u) * 4 + w) * 64 + lane];
                }
                const int e = Head<ND>::dim(n0 + n, w, kc);
                float *const dst = out + l16 * W + e;
                if (row_ok)
                {
#pragma unroll
                    for (int u = 0; u < NU; ++u)
                        bad |= !__builtin_isfinite(o[u]);
                    if (VEC && NU == 4)
                    {
                        if (e < d)
                            *reinterpret_cast<float4 *>(dst) = make_float4(o[0], o[1 % NU], o[2 % NU], o[3 % NU]);
                    }
                    else
                    {
#pragma unroll
                        for (int u = 0; u < NU; ++u)
                            if (e + u < d)
                                dst[u] = o[u];
                    }
                }
            }
    }
    return bad;
}

// Whether x holds in any lane of the workgroup (through red: __syncthreads_or has
// LDS of its own, with which five backward workgroups no longer fit a CU).
__device__ __forceinline__ bool any_lane(bool x, float *red, int w, int lane)
{
    x = __any(x);
    __syncthreads();
    if (lane == 0)
        red[w] = x ? 1.f : 0.f;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3] != 0.f;
}

// The matrix products above multiply a masked pair's weight of 0 with what
// stands in its rows: an infinity or NaN in V or K of a key after the query, or in
// Q or dO of a query before the key, would reach results of the same diagonal
// block, and a wave whose blocks hold no score but -inf has no maximum to take them
// against. A workgroup with an output that is not finite therefore works its rows
// out again, pair by pair: 16 lanes a row, lane p dimensions p + 16 u, over the
// row's own keys (or queries) alone.
template <int ND> struct Pairs
{
    int g, p;  // row of the block, lane of the row
    int d;
    __device__ __forceinline__ explicit Pairs(int dims) : d(dims)
    {
        int t = (int)threadIdx.x;
        asm volatile("" : "+v"(t));  // shares nothing with the first pass, whose registers it would hold
        g = t >> 4;
        p = t & 15;
    }
    __device__ __forceinline__ void load(float (&f)[ND], const float *row) const
    {
#pragma unroll
        for (int u = 0; u < ND; ++u)
            f[u] = p + 16 * u < d ? row[p + 16 * u] : 0.f;
    }
    __device__ __forceinline__ void store(float *row, const float (&f)[ND], float scale) const
    {
#pragma unroll
        for (int u = 0; u < ND; ++u)
            if (p + 16 * u < d)
                row[p + 16 * u] = f[u] * scale;
    }
    static __device__ __forceinline__ float dot(const float (&a)[ND], const float (&b)[ND])
    {
        float x = 0.f;
#pragma unroll
        for (int u = 0; u < ND; ++u)
            x += a[u] * b[u];
        return row16_sum(x);
    }
    static __device__ __forceinline__ void add(float (&acc)[ND], float w, const float (&b)[ND])
    {
#pragma unroll
        for (int u = 0; u < ND; ++u)
            acc[u] += w * b[u];
    }
};

template <int ND>
__device__ __forceinline__ void fwd_pairs(float *y, float *lse, const float *x, int T, long C, int H, int b, int h, int q0, int d,
                                          float qscale)
{
    const Pairs<ND> pr(d);
    const int i = q0 + pr.g;
    if (i >= T)
        return;
    const float *const base = x + (long)b * T * 3 * C + (long)h * d;
    float q[ND], o[ND] = {}, m = -FLT_MAX, l = 0.f;
    pr.load(q, base + (long)i * 3 * C);
#pragma unroll 1
    for (int j = 0; j <= i; ++j)
    {
        float k[ND], v[ND];
        pr.load(k, base + (long)j * 3 * C + C);
        pr.load(v, base + (long)j * 3 * C + 2 * C);
        const float s = Pairs<ND>::dot(q, k) * qscale, mn = fmaxf(m, s), corr = fast_exp2(m - mn), e = fast_exp2(s - mn);
        m = mn;
        l = l * corr + e;
#pragma unroll
        for (int u = 0; u < ND; ++u)
            o[u] = o[u] * corr + e * v[u];
    }
    pr.store(y + ((long)b * T + i) * C + (long)h * d, o, 1.f / l);
    if (pr.p == 0)
        lse[((long)b * T + i) * H + h] = (m + fast_log2(l)) * kLn2;
}

template <int ND>
__device__ __forceinline__ void dq_pairs(float *gx, const float *lse, const float *dy, const float *y, const float *x, int T,
                                         long C, int H, int b, int h, int q0, int d, float scale, float qscale)
{
    const Pairs<ND> pr(d);
    const int i = q0 + pr.g;
    if (i >= T)
        return;
    const float *const base = x + (long)b * T * 3 * C + (long)h * d;
    const long at = ((long)b * T + i) * C + (long)h * d;
    float q[ND], g[ND], acc[ND] = {}, D;
    pr.load(q, base + (long)i * 3 * C);
    pr.load(g, dy + at);
    {
        float o[ND];
        pr.load(o, y + at);
        D = Pairs<ND>::dot(g, o);
    }
    const float L = lse[((long)b * T + i) * H + h] * kLog2e;
#pragma unroll 1
    for (int j = 0; j <= i; ++j)
    {
        float k[ND], v[ND];
        pr.load(k, base + (long)j * 3 * C + C);
        pr.load(v, base + (long)j * 3 * C + 2 * C);
        const float e = fast_exp2(Pairs<ND>::dot(q, k) * qscale - L);
        Pairs<ND>::add(acc, e * (Pairs<ND>::dot(g, v) - D), k);
    }
    pr.store(gx + ((long)b * T + i) * 3 * C + (long)h * d, acc, scale);
}

template <int ND>
__device__ __forceinline__ void dkdv_pairs(float *gx, const float *lse, const float *D, const float *dy, const float *x, int T,
                                           long C, int H, int b, int h, int k0, int d, float scale, float qscale)
{
    const Pairs<ND> pr(d);
    const int j = k0 + pr.g;
    if (j >= T)
        return;
    const float *const base = x + (long)b * T * 3 * C + (long)h * d;
    float k[ND], v[ND], dk[ND] = {}, dv[ND] = {};
    pr.load(k, base + (long)j * 3 * C + C);
    pr.load(v, base + (long)j * 3 * C + 2 * C);
#pragma unroll 1
    for (int i = j; i < T; ++i)
    {
        float q[ND], g[ND];
        pr.load(q, base + (long)i * 3 * C);
        pr.load(g, dy + ((long)b * T + i) * C + (long)h * d);
        const long at = ((long)b * T + i) * H + h;
        const float e = fast_exp2(Pairs<ND>::dot(q, k) * qscale - lse[at] * kLog2e);
        Pairs<ND>::add(dk, e * (Pairs<ND>::dot(g, v) - D[at]), q);
        Pairs<ND>::add(dv, e, g);
    }
    float *const out = gx + ((long)b * T + j) * 3 * C + (long)h * d;
    pr.store(out + C, dk, scale);
    pr.store(out + 2 * C, dv, 1.f);
}

// Workgroup -> (b, h) and row block: (b, h) fastest, so that with B H a
// multiple of 8 one (b, h) stays on one XCD, and heaviest blocks first. The
// last row of a two-dimensional grid may reach past the items (past(it)).
struct Item
{
    int b, h, blk;
};
__device__ __forceinline__ Item item(int H, int BH, int n_blk, bool last_first)
{
    const unsigned i = blockIdx.y * gridDim.x + blockIdx.x;
    const int bh = (int)(i % (unsigned)BH), k = (int)(i / (unsigned)BH);
    return Item{bh / H, bh % H, last_first ? n_blk - 1 - k : k};
}
__device__ __forceinline__ bool past(const Item &it, int n_blk) { return it.blk < 0 || it.blk >= n_blk; }

// y and lse of 16 queries. S^T is formed (lane: query l16, keys 4 kc + r), so
// that P feeds the second product as it stands.
template <int ND, bool VEC>
__global__ __launch_bounds__(64 * kWaves, ND <= 8 ? 2 : 1) void fwd_general_kernel(float *__restrict__ y, float *__restrict__ lse,
                                                                                const float *__restrict__ qkv, int T, int C,
                                                                                int H, int BH, int n_blk, int d, float qscale)
{
    __shared__ float red[kMerge];
    __shared__ float sm[kWaves][kRows], sl[kWaves][kRows];
    const int lane = threadIdx.x & 63, l16 = lane & 15, kc = lane >> 4, w = wave_id();
    const Item it = item(H, BH, n_blk, true);
    if (past(it, n_blk))
        return;
    const long W = 3L * C;
    const float *const base = qkv + (long)it.b * T * W + (long)it.h * d;
    const int q0 = kRows * it.blk;
    // What a second pass would need, for the 4-byte form, whose loops spill scalar
    // registers as it is (B = 2, T = 200, H = 4, d = 129: 50.9 us, 55.1 with them held).
    struct Held
    {
        float *y, *lse;
        const float *qkv;
        int T, C, H, b, h, q0, d;
        float qscale;
    };
    __shared__ Held held;
    if (!VEC && threadIdx.x == 0)
        held = Held{y, lse, qkv, T, C, H, it.b, it.h, q0, d, qscale};

    float q[ND][4];
    load_rows<ND, VEC>(q, rows_of(base, q0, T, W, d), d, l16, kc);
#pragma unroll
    for (int u = 0; u < ND; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            q[u][e] *= qscale;
    v4f acc[ND];
#pragma unroll
    for (int n = 0; n < ND; ++n)
        acc[n] = zero4();
    float m = -INFINITY, l = 0.f;
    for (int j = w; j <= it.blk; j += kWaves)
    {
        float k[ND][4], v[4][ND];
        load_rows<ND, VEC>(k, rows_of(base + C, kRows * j, T, W, d), d, l16, kc);
        load_cols<ND, VEC>(v, rows_of(base + 2L * C, kRows * j, T, W, d), d, l16, kc);
        v4f s = dot_rows<ND>(k, q);
        if (j == it.blk)
        {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (4 * kc + r > l16)
                    s[r] = -INFINITY;
        }
        const float mb = rows16_max(halves_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
        const float mn = fmaxf(m, mb);
        if (__any(mn > m))
        {
            const float corr = fast_exp2(m - mn);
            l *= corr;
#pragma unroll
            for (int n = 0; n < ND; ++n)
                acc[n] *= corr;
            m = mn;
        }
        v4f p;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            p[r] = fast_exp2(s[r] - m);
        l += (p[0] + p[1]) + (p[2] + p[3]);
        add_cols<ND>(acc, v, p);
    }
    l = rows16_sum(halves_sum(l));
    if (kc == 0)
    {
        sm[w][l16] = m;
        sl[w][l16] = l;
    }
    __syncthreads();
    float M = sm[0][l16], L = 0.f;
#pragma unroll
    for (int k = 1; k < kWaves; ++k)
        M = fmaxf(M, sm[k][l16]);
#pragma unroll
    for (int k = 0; k < kWaves; ++k)
        L += sl[k][l16] * fast_exp2(sm[k][l16] - M);
    const int row = q0 + l16;
    const bool bad = merge_store<ND, VEC>(acc, fast_exp2(m - M) / L, red, y + ((long)it.b * T + q0) * C + (long)it.h * d, C, d,
                                         row < T, w, lane);
    if (w == 0 && kc == 0 && row < T)
        lse[((long)it.b * T + row) * H + it.h] = (M + fast_log2(L)) * kLn2;
    if (any_lane(bad, red, w, lane))
    {
        if (VEC)
            fwd_pairs<ND>(y, lse, qkv, T, C, H, it.b, it.h, q0, d, qscale);
        else
            fwd_pairs<ND>(held.y, held.lse, held.qkv, held.T, held.C, held.H, held.b, held.h, held.q0, held.d, held.qscale);
    }
}

// D and dQ of 16 queries (lane: query l16, keys 4 kc + r).
template <int ND, bool VEC>
__global__ __launch_bounds__(64 * kWaves, 1) void bwd_dq_general_kernel(float *__restrict__ grad_x, float *__restrict__ D,
                                                                        const float *__restrict__ lse,
                                                                        const float *__restrict__ dy,
                                                                        const float *__restrict__ y,
                                                                        const float *__restrict__ qkv, int T, int C, int H,
                                                                        int BH, int n_blk, int d, float scale, float qscale)
{
    __shared__ float red[kMerge];
    const int lane = threadIdx.x & 63, l16 = lane & 15, kc = lane >> 4, w = wave_id();
    const Item it = item(H, BH, n_blk, true);
    if (past(it, n_blk))
        return;
    const long W = 3L * C;
    const float *const base = qkv + (long)it.b * T * W + (long)it.h * d;
    const int q0 = kRows * it.blk, row = q0 + l16;

    float q[ND][4], g[ND][4];
    load_rows<ND, VEC>(q, rows_of(base, q0, T, W, d), d, l16, kc);
    load_rows<ND, VEC>(g, rows_of(dy + (long)it.b * T * C + (long)it.h * d, q0, T, C, d), d, l16, kc);
    const long at = ((long)it.b * T + (row < T ? row : T - 1)) * H + it.h;
    const float L = lse[at] * kLog2e;
    // D = rowsum(dO * O), every wave its own copy
    float Dr = 0.f;
    {
        float o[ND][4];
        load_rows<ND, VEC>(o, rows_of(y + (long)it.b * T * C + (long)it.h * d, q0, T, C, d), d, l16, kc);
#pragma unroll
        for (int u = 0; u < ND; ++u)
            Dr += (g[u][0] * o[u][0] + g[u][1] * o[u][1]) + (g[u][2] * o[u][2] + g[u][3] * o[u][3]);
        Dr = rows16_sum(halves_sum(Dr));
    }
    if (w == 0 && kc == 0 && row < T)
        D[at] = Dr;
#pragma unroll
    for (int u = 0; u < ND; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            q[u][e] *= qscale;
    v4f acc[ND];
#pragma unroll
    for (int n = 0; n < ND; ++n)
        acc[n] = zero4();
    for (int j = w; j <= it.blk; j += kWaves)
    {
        float k[ND][4], v[ND][4], kt[4][ND];
        const Rows rk = rows_of(base + C, kRows * j, T, W, d);
        load_rows<ND, VEC>(k, rk, d, l16, kc);
        load_rows<ND, VEC>(v, rows_of(base + 2L * C, kRows * j, T, W, d), d, l16, kc);
        load_cols<ND, VEC>(kt, rk, d, l16, kc);
        const v4f s = dot_rows<ND>(k, q), dp = dot_rows<ND>(v, g);
        v4f ds;
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const float p = j == it.blk && 4 * kc + r > l16 ? 0.f : fast_exp2(s[r] - L);
            ds[r] = p * (dp[r] - Dr);
        }
        add_cols<ND>(acc, kt, ds);
    }
    const bool bad =
        merge_store<ND, VEC>(acc, scale, red, grad_x + ((long)it.b * T + q0) * W + (long)it.h * d, W, d, row < T, w, lane);
    if (any_lane(bad, red, w, lane))
        dq_pairs<ND>(grad_x, lse, dy, y, qkv, T, C, H, it.b, it.h, q0, d, scale, qscale);
}

// dK and dV of 16 keys (lane: key l16, queries 4 kc + r). The keys' own rows
// stay in registers while they leave room (ND <= 8) and are read again for
// every block beyond.
template <int ND, bool VEC>
__global__ __launch_bounds__(64 * kWaves, 1) void bwd_dkdv_general_kernel(float *__restrict__ grad_x, const float *__restrict__ lse,
                                                                          const float *__restrict__ D,
                                                                          const float *__restrict__ dy,
                                                                          const float *__restrict__ qkv, int T, int C, int H,
                                                                          int BH, int n_blk, int d, float scale, float qscale)
{
    __shared__ float red[kMerge];
    const int lane = threadIdx.x & 63, l16 = lane & 15, kc = lane >> 4, w = wave_id();
    const Item it = item(H, BH, n_blk, false);
    if (past(it, n_blk))
        return;
    const long W = 3L * C;
    const float *const base = qkv + (long)it.b * T * W + (long)it.h * d;
    const float *const dyb = dy + (long)it.b * T * C + (long)it.h * d;
    const int k0 = kRows * it.blk;
    constexpr bool kKeep = ND <= 8;

    const Rows rk = rows_of(base + C, k0, T, W, d), rv = rows_of(base + 2L * C, k0, T, W, d);
    float k[ND][4], v[ND][4];
    if (kKeep)
    {
        load_rows<ND, VEC>(k, rk, d, l16, kc);
        load_rows<ND, VEC>(v, rv, d, l16, kc);
    }
    v4f dk[ND], dv[ND];
#pragma unroll
    for (int n = 0; n < ND; ++n)
        dk[n] = dv[n] = zero4();
    for (int i = it.blk + w; i < n_blk; i += kWaves)
    {
        const Rows rq = rows_of(base, kRows * i, T, W, d), rg = rows_of(dyb, kRows * i, T, C, d);
        v4f s, dp;
        {
            float q[ND][4];
            load_rows<ND, VEC>(q, rq, d, l16, kc);
            if (!kKeep)
                load_rows<ND, VEC>(k, rk, d, l16, kc);
            s = dot_rows<ND>(q, k);
        }
        {
            float g[ND][4];
            load_rows<ND, VEC>(g, rg, d, l16, kc);
            if (!kKeep)
                load_rows<ND, VEC>(v, rv, d, l16, kc);
            dp = dot_rows<ND>(g, v);
        }
        v4f p, ds;
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const int row = kRows * i + 4 * kc + r;
            const long at = ((long)it.b * T + (row < T ? row : T - 1)) * H + it.h;
            const bool ok = row < T && row >= k0 + l16;
            p[r] = ok ? fast_exp2(s[r] * qscale - lse[at] * kLog2e) : 0.f;
            ds[r] = p[r] * (dp[r] - D[at]);
        }
        {
            float gt[4][ND];
            load_cols<ND, VEC>(gt, rg, d, l16, kc);
            add_cols<ND>(dv, gt, p);
        }
        {
            float qt[4][ND];
            load_cols<ND, VEC>(qt, rq, d, l16, kc);
            add_cols<ND>(dk, qt, ds);
        }
    }
    float *const out = grad_x + ((long)it.b * T + k0) * W + (long)it.h * d;
    bool bad = merge_store<ND, VEC>(dk, scale, red, out + C, W, d, k0 + l16 < T, w, lane);
    bad |= merge_store<ND, VEC>(dv, 1.f, red, out + 2L * C, W, d, k0 + l16 < T, w, lane);
    if (any_lane(bad, red, w, lane))
        dkdv_pairs<ND>(grad_x, lse, D, dy, qkv, T, C, H, it.b, it.h, k0, d, scale, qscale);
}

bool vec_ok(const Shape &s, const void *a, const void *b, const void *c, const void *e = nullptr)
{
    return s.d % 4 == 0 && s.C % 4 == 0 && 3LL * kRows * s.C * 4 < (1LL << 31) &&
           ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(c) |
             reinterpret_cast<uintptr_t>(e)) & 15u) == 0;
}

// One workgroup per item. A launch holds below 2^32 threads along a dimension,
// so more than 2^23 workgroups take rows of 2^23 (calls of up to 2^31 rows).
dim3 items_grid(const Shape &s)
{
    const long n = (long)s.B * s.H * ((s.T + kRows - 1) / kRows), row = 1L << 23;
    return n <= row ? dim3((unsigned)n) : dim3((unsigned)row, (unsigned)((n + row - 1) / row));
}

// Calls f with the padded head size (in 16 dimensions) and the vector form as
// template arguments. Heads that are no multiple of 4 floats, or misaligned
// ones, take 4-byte loads and every other padding.
template <class F> void with_head(const Shape &s, bool vec, F f)
{
    const int nd = (s.d + 15) / 16;
#define HEAD(N) f(std::integral_constant<int, N>(), std::true_type())
#define HEAD1(N) f(std::integral_constant<int, N>(), std::false_type())
    if (vec)
        nd <= 1 ? HEAD(1) : nd <= 2 ? HEAD(2) : nd <= 3 ? HEAD(3) : nd <= 4 ? HEAD(4) : nd <= 5 ? HEAD(5) : nd <= 6 ? HEAD(6)
        : nd <= 8 ? HEAD(8) : nd <= 10 ? HEAD(10) : nd <= 12 ? HEAD(12) : HEAD(16);
    else
        nd <= 1 ? HEAD1(1) : nd <= 2 ? HEAD1(2) : nd <= 4 ? HEAD1(4) : nd <= 8 ? HEAD1(8) : HEAD1(16);
#undef HEAD
#undef HEAD1
}

}  // namespace

hipError_t launch_fwd_general(float *y, float *lse, const float *qkv, const Shape &s, hipStream_t st)
{
    const int n_blk = (s.T + kRows - 1) / kRows, BH = s.B * s.H;
    const dim3 grid = items_grid(s), block(64 * kWaves);
    const float qscale = softmax_scale(s.d) * kLog2e;
    timer_begin(kKindOther, st);
    with_head(s, vec_ok(s, y, qkv, qkv), [&](auto nd, auto vec) {
        hipLaunchKernelGGL((fwd_general_kernel<decltype(nd)::value, decltype(vec)::value>), grid, block, 0, st, y, lse, qkv,
                           s.T, s.C, s.H, BH, n_blk, s.d, qscale);
    });
    timer_end(st);
    return hipGetLastError();
}

hipError_t launch_bwd_general(float *grad_x, float *D, const float *lse, const float *dy, const float *y,
                              const float *qkv, const Shape &s, hipStream_t st)
{
    const int n_blk = (s.T + kRows - 1) / kRows, BH = s.B * s.H;
    const dim3 grid = items_grid(s), block(64 * kWaves);
    const float scale = softmax_scale(s.d), qscale = scale * kLog2e;
    timer_begin(kKindOther, st);
    with_head(s, vec_ok(s, grad_x, dy, y, qkv), [&](auto nd, auto vec) {
        constexpr int ND = decltype(nd)::value;
        constexpr bool VEC = decltype(vec)::value;
        hipLaunchKernelGGL((bwd_dq_general_kernel<ND, VEC>), grid, block, 0, st, grad_x, D, lse, dy, y, qkv, s.T, s.C, s.H,
                           BH, n_blk, s.d, scale, qscale);
        hipLaunchKernelGGL((bwd_dkdv_general_kernel<ND, VEC>), grid, block, 0, st, grad_x, lse, D, dy, qkv, s.T, s.C, s.H,
                           BH, n_blk, s.d, scale, qscale);
    });
    timer_end(st);
    return hipGetLastError();
}

}  // namespace gpt_attn
