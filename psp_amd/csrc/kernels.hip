// HIP kernels for gfx950 (MI355X): front assembly, multifrontal LDL^T,
// front solves, sweep couplings, the PML 7-point operator and the GMRES
// vector primitives.  All kernels use 256-thread workgroups (4 wave64).
#include "kernels.hpp"

#include <algorithm>
#include <type_traits>

namespace psp_amd {

namespace {

constexpr int kThreads = 256;

// --------------------------------------------------------------------------
// Complex arithmetic (interleaved re, im).
// --------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ cx<T> mk(T r, T i) { return cx<T>{r, i}; }
template <typename T>
__device__ __forceinline__ cx<T> operator+(cx<T> a, cx<T> b) { return {a.r + b.r, a.i + b.i}; }
template <typename T>
__device__ __forceinline__ cx<T> operator-(cx<T> a, cx<T> b) { return {a.r - b.r, a.i - b.i}; }
template <typename T>
__device__ __forceinline__ cx<T> operator-(cx<T> a) { return {-a.r, -a.i}; }
template <typename T>
__device__ __forceinline__ cx<T> operator*(cx<T> a, cx<T> b)
{
    return {a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r};
}
template <typename T>
__device__ __forceinline__ cx<T> operator*(cx<T> a, T s) { return {a.r * s, a.i * s}; }
// acc + a*b
template <typename T>
__device__ __forceinline__ cx<T> cfma(cx<T> a, cx<T> b, cx<T> acc)
{
    acc.r = fma(a.r, b.r, acc.r);
    acc.r = fma(-a.i, b.i, acc.r);
    acc.i = fma(a.r, b.i, acc.i);
    acc.i = fma(a.i, b.r, acc.i);
    return acc;
}
// acc - a*b
template <typename T>
__device__ __forceinline__ cx<T> cfms(cx<T> a, cx<T> b, cx<T> acc)
{
    acc.r = fma(-a.r, b.r, acc.r);
    acc.r = fma(a.i, b.i, acc.r);
    acc.i = fma(-a.r, b.i, acc.i);
    acc.i = fma(-a.i, b.r, acc.i);
    return acc;
}
// Smith's complex division a / b.
template <typename T>
__device__ __forceinline__ cx<T> cdiv(cx<T> a, cx<T> b)
{
    if (fabs(b.r) >= fabs(b.i)) {
        const T rr = b.i / b.r, den = b.r + b.i * rr;
        return {(a.r + a.i * rr) / den, (a.i - a.r * rr) / den};
    }
    const T rr = b.r / b.i, den = b.i + b.r * rr;
    return {(a.r * rr + a.i) / den, (a.i * rr - a.r) / den};
}
template <typename T>
__device__ __forceinline__ cx<T> cinv(cx<T> b) { return cdiv(cx<T>{T(1), T(0)}, b); }
template <typename T>
__device__ __forceinline__ cx<T> cdivr(cx<T> a, T s) { return {a.r / s, a.i / s}; }

template <typename To, typename Ti>
__device__ __forceinline__ cx<To> cvt(cx<Ti> a) { return {To(a.r), To(a.i)}; }

// Two reals of one type (a pre-swizzled LDS operand pair).
template <typename T>
struct T2 {
    T x, y;
};

template <typename T>
__device__ __forceinline__ cx<T> czero() { return {T(0), T(0)}; }

// --------------------------------------------------------------------------
// PML 7-point stencil: FormGlobalRow (initialize_finalize.hpp:527-587) and
// FormLowerColumnOfNode (:589-640).  out[0] centre, out[1..6] the values of
// the x-1, x+1, y-1, y+1, v-1, v+1 couplings.
// --------------------------------------------------------------------------
__device__ __forceinline__ void Stencil(c128 s1L, c128 s1M, c128 s1R, c128 s2L, c128 s2M,
                                        c128 s2R, c128 s3L, c128 s3M, c128 s3R, c128 k2,
                                        double hx, double hy, double hz, c128 out[7])
{
    const c128 xTop = s2M * s3M;
    const c128 xTempL = cdiv(xTop, s1L), xTempM = cdiv(xTop, s1M), xTempR = cdiv(xTop, s1R);
    const c128 xTermL = cdivr(xTempL + xTempM, 2 * hx * hx);
    const c128 xTermR = cdivr(xTempR + xTempM, 2 * hx * hx);
    const c128 yTop = s1M * s3M;
    const c128 yTempL = cdiv(yTop, s2L), yTempM = cdiv(yTop, s2M), yTempR = cdiv(yTop, s2R);
    const c128 yTermL = cdivr(yTempL + yTempM, 2 * hy * hy);
    const c128 yTermR = cdivr(yTempR + yTempM, 2 * hy * hy);
    const c128 zTop = s1M * s2M;
    const c128 vTempL = cdiv(zTop, s3L), vTempM = cdiv(zTop, s3M), vTempR = cdiv(zTop, s3R);
    const c128 vTermL = cdivr(vTempL + vTempM, 2 * hz * hz);
    const c128 vTermR = cdivr(vTempR + vTempM, 2 * hz * hz);
    out[0] = (xTermL + xTermR + yTermL + yTermR + vTermL + vTermR) - k2 * s1M * s2M * s3M;
    out[1] = -xTermL;
    out[2] = -xTermR;
    out[3] = -yTermL;
    out[4] = -yTermR;
    out[5] = -vTermL;
    out[6] = -vTermR;
}

// Global operator row at (x, y, v): undamped frequency, physical PML.
__device__ __forceinline__ void GlobalRow(const StencilArgs& st, double alpha, int x, int y,
                                          int v, c128 out[7])
{
    const double wa = st.omega / alpha;
    const c128 k2 = {wa * wa, 0.0};
    Stencil(st.s1[x], st.s1[x + 1], st.s1[x + 2], st.s2[y], st.s2[y + 1], st.s2[y + 2],
            st.s3[v], st.s3[v + 1], st.s3[v + 2], k2, st.hx, st.hy, st.hz, out);
}

// The same row from per-axis tables: xTermL = (s2 s3) (1/s1(x-1) + 1/s1(x))
// / (2 hx^2) etc., i.e. FormGlobalRow's terms with the divisions hoisted into
// host tables (equal up to rounding).
__device__ __forceinline__ void GlobalRowFast(const StencilArgs& st, double alpha, int x, int y,
                                              int v, c128 out[7])
{
    const c128 s1M = st.s1[x + 1], s2M = st.s2[y + 1], s3M = st.s3[v + 1];
    const c128 xTop = s2M * s3M, yTop = s1M * s3M, zTop = s1M * s2M;
    const c128 xL = xTop * st.ax[2 * x], xR = xTop * st.ax[2 * x + 1];
    const c128 yL = yTop * st.ay[2 * y], yR = yTop * st.ay[2 * y + 1];
    const c128 vL = zTop * st.av[2 * v], vR = zTop * st.av[2 * v + 1];
    const double wa = st.omega / alpha;
    out[0] = (xL + xR + yL + yR + vL + vR) - (zTop * s3M) * (wa * wa);
    out[1] = -xL;
    out[2] = -xR;
    out[3] = -yL;
    out[4] = -yR;
    out[5] = -vL;
    out[6] = -vR;
}

// --------------------------------------------------------------------------
// Fill
// --------------------------------------------------------------------------
__global__ void k_fill_zero(uint4* p, int64_t n16)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride)
        p[i] = make_uint4(0, 0, 0, 0);
}

// rows ranges of n8 8-byte words, range r at p + r * stride8
__global__ void k_fill_zero_rows(uint2* p, int64_t n8, int64_t stride8)
{
    uint2* q = p + (int64_t)blockIdx.y * stride8;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8; i += stride)
        q[i] = make_uint2(0, 0);
}

__global__ void k_fill_zero_bytes(unsigned char* p, int64_t n)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = 0;
}

// --------------------------------------------------------------------------
// Front assembly of the original panel operator (FillPanelFronts,
// initialize_finalize.hpp:1284-1337): one thread per padded unknown of one
// panel of the batch; writes the diagonal and the strictly-lower couplings
// of its column into its front.
// --------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kThreads) void k_scatter_orig(
    int n, int vsize, const int32_t* qxy, const int32_t* qv, const int32_t* qnode,
    const int32_t* qcol, const int32_t* qrows, const int64_t* nodeL, const int32_t* nodeS,
    const int32_t* nodeU, const int32_t* panelVOff, const c128* s3art, StencilArgs st,
    const double* vel, double damping, cx<T>* L, int64_t fstore)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const int b = blockIdx.y;
    const int x = qxy[q] & 0xffff, y = qxy[q] >> 16, vl = qv[q];
    const int vOffset = panelVOff[b];
    const int v = vOffset + vl;
    const int z = st.nz - 1 - v;
    const double alpha = vel[x + (int64_t)y * st.nx + (int64_t)z * st.nx * st.ny];
    const c128* s3 = s3art + (int64_t)b * (vsize + 2);
    const c128 so = {st.omega / alpha, damping / alpha};  // (omega + i damping)/alpha
    const c128 k2 = so * so;
    c128 e[7];
    Stencil(st.s1[x], st.s1[x + 1], st.s1[x + 2], st.s2[y], st.s2[y + 1], st.s2[y + 2],
            s3[vl], s3[vl + 1], s3[vl + 2], k2, st.hx, st.hy, st.hz, e);
    const int t = qnode[q], j = qcol[q];
    const int64_t fs = nodeS[t] + nodeU[t];
    cx<T>* col = L + (int64_t)b * fstore + nodeL[t] + (int64_t)j * fs;
    col[j] = cvt<T>(e[0]);
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const int row = qrows[(int64_t)q * 6 + k];
        if (row >= 0) col[row] = cvt<T>(e[k + 1]);
    }
}

// --------------------------------------------------------------------------
// Extend-add of a child's Schur complement into its parent front.
// --------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kThreads) void k_extend_add(const ExtAddItem* items, int start,
                                                          const int32_t* relinds, cx<T>* L,
                                                          int64_t fstore, cx<T>* U,
                                                          int64_t ustore)
{
    const ExtAddItem it = items[start + blockIdx.x];
    const int b = blockIdx.y;
    const cx<T>* Uc = U + (int64_t)b * ustore + it.uChild;
    cx<T>* Lp = L + (int64_t)b * fstore + it.lParent;
    cx<T>* Up = U + (int64_t)b * ustore + it.uParent;
    const int32_t* rel = relinds + it.relStart;
    const int ldp = it.sp + it.up;
    for (int cb = it.col0; cb < it.col1; ++cb) {
        const int rb = rel[cb];
        for (int a = cb + threadIdx.x; a < it.uc; a += blockDim.x) {
            const cx<T> val = Uc[a + (int64_t)cb * it.uc];
            const int ra = rel[a];
            if (rb < it.sp) {
                cx<T>* p = Lp + ra + (int64_t)rb * ldp;
                *p = *p + val;
            } else {
                cx<T>* p = Up + (ra - it.sp) + (int64_t)(rb - it.sp) * it.up;
                *p = *p + val;
            }
        }
    }
}

// --------------------------------------------------------------------------
// Blocked LDL^T, step 1: unpivoted LDL^T of the diagonal block in LDS.
// --------------------------------------------------------------------------
template <typename T, int NB>
__global__ __launch_bounds__(kThreads) void k_ldl_diag(const LdlItem* items, int start, cx<T>* L,
                                                        int64_t fstore)
{
    const LdlItem it = items[start + blockIdx.x];
    cx<T>* F = L + (int64_t)blockIdx.y * fstore + it.l;
    const int ld = it.ld, j0 = it.j0, m = it.j1 - it.j0;
    static_assert(NB == 32 && kThreads == 256, "each thread owns 2 x 2 elements of the block");
    __shared__ cx<T> A[NB][NB + 1];  // A[col][row]
    // thread (tx, ty) owns rows tx, tx + 16 and columns ty, ty + 16
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int r = tx + 16 * a, c = ty + 16 * b;
            if (r < m && c <= r) A[c][r] = F[(j0 + r) + (int64_t)(j0 + c) * ld];
        }
    __syncthreads();
    // Step j updates the trailing block with column j (unscaled) and scales
    // column j - 1, which step j no longer reads: one barrier per column.
    for (int j = 0; j < m; ++j) {
        const cx<T> dinv = cinv(A[j][j]);
        if (j > 0 && ty == 0) {
            const cx<T> dp = cinv(A[j - 1][j - 1]);
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int r = tx + 16 * a;
                if (r > j - 1 && r < m) A[j - 1][r] = A[j - 1][r] * dp;
            }
        }
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int r = tx + 16 * a, c = ty + 16 * b;
                if (c > j && r >= c && r < m) A[c][r] = cfms(A[j][r] * dinv, A[j][c], A[c][r]);
            }
        __syncthreads();  // no global loads are in flight here
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int r = tx + 16 * a, c = ty + 16 * b;
            if (r < m && c <= r) F[(j0 + r) + (int64_t)(j0 + c) * ld] = A[c][r];
        }
}

// Blocked LDL^T, step 2: rows below the diagonal block,
// L21 = F21 L11^{-T} D1^{-1}, one thread per row.
template <typename T, int NB>
__global__ __launch_bounds__(kThreads) void k_ldl_trsm(const LdlItem* items, int start, cx<T>* L,
                                                        int64_t fstore)
{
    const LdlItem it = items[start + blockIdx.x];
    cx<T>* F = L + (int64_t)blockIdx.y * fstore + it.l;
    const int ld = it.ld, j0 = it.j0, m = it.j1 - it.j0;
    __shared__ cx<T> W[NB][NB];  // W[c][q] = d_q L11(c, q), q < c
    __shared__ cx<T> dinv[NB];
    for (int e = threadIdx.x; e < m * m; e += blockDim.x) {
        const int c = e / m, q = e % m;
        if (q < c)
            W[c][q] = F[(j0 + q) + (int64_t)(j0 + q) * ld] * F[(j0 + c) + (int64_t)(j0 + q) * ld];
    }
    for (int c = threadIdx.x; c < m; c += blockDim.x)
        dinv[c] = cinv(F[(j0 + c) + (int64_t)(j0 + c) * ld]);
    __syncthreads();
    const int r = it.r0 + threadIdx.x;
    if (r >= it.r1) return;
    cx<T> x[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) x[c] = c < m ? F[r + (int64_t)(j0 + c) * ld] : czero<T>();
#pragma unroll
    for (int c = 0; c < NB; ++c) {
        if (c < m) {
            cx<T> acc = x[c];
#pragma unroll
            for (int q = 0; q < c; ++q) acc = cfms(x[q], W[c][q], acc);
            x[c] = acc * dinv[c];
        }
    }
#pragma unroll
    for (int c = 0; c < NB; ++c)
        if (c < m) F[r + (int64_t)(j0 + c) * ld] = x[c];
}

// Inverse of one unit-lower diagonal block in place (strict lower part).
template <typename T, int NB>
__global__ __launch_bounds__(kThreads) void k_inv_diag(const InvItem* items, cx<T>* L,
                                                        int64_t fstore)
{
    const InvItem it = items[blockIdx.x];
    cx<T>* F = L + (int64_t)blockIdx.y * fstore + it.l;
    const int ld = it.ld, j0 = it.j0, m = it.j1 - it.j0;
    __shared__ cx<T> A[NB][NB + 1];  // A[col][row] strictly lower
    __shared__ cx<T> X[NB][NB + 1];  // X[col][row] inverse
    for (int e = threadIdx.x; e < m * m; e += blockDim.x) {
        const int r = e % m, c = e / m;
        A[c][r] = r > c ? F[(j0 + r) + (int64_t)(j0 + c) * ld] : czero<T>();
    }
    __syncthreads();
    const int c = threadIdx.x;
    if (c < m) {
        X[c][c] = cx<T>{T(1), T(0)};
        for (int r = c + 1; r < m; ++r) {
            cx<T> acc = czero<T>();
            for (int q = c; q < r; ++q) acc = cfms(A[q][r], X[c][q], acc);
            X[c][r] = acc;
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < m * m; e += blockDim.x) {
        const int r = e % m, cc = e / m;
        if (r > cc) F[(j0 + r) + (int64_t)(j0 + cc) * ld] = X[cc][r];
    }
}

// Workgroup barrier for LDS traffic only: waits for this wave's LDS
// operations but not for its outstanding global loads, so loads issued
// before the barrier (the next operands) stay in flight across it.  Used
// wherever a barrier only orders LDS accesses.
__device__ __forceinline__ void LdsBarrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// --------------------------------------------------------------------------
// Front solves on the padded panel vector Xp (rows x k, interleaved), with
// the factors in the solve layout (rows < s of L: Linv with a stored unit
// diagonal; rows >= s: -L_BL Linv; LT: [Linv^T D^-1 | (-L_BL Linv)^T]).
// Per node, with g = [Xp_own; 0] + the children's update vectors (read from
// per-slot copies of the node's front rows that the children write):
//   forward  F: W_top = Linv g_top; the update g_bot + (-L_BL Linv) g_top
//               goes into the parent's slot copy;
//   backward B: Xp_own = LT [W_top; x_struct].
// Each is one product over the node's factor block, split into row tiles
// (and, near the root, inner slices summed by a reduce launch).
// --------------------------------------------------------------------------
enum { PH_F = 0, PH_B = 1 };

// The children's update rows: each child writes its rows straight into a
// per-slot copy of its parent's front rows (slot 0: first child, slot 1:
// second child), at the parent rows given by relinds.  Rows a child does not
// touch stay zero from the workspace's allocation (each slot copy belongs to
// one panel class, and a class writes the same rows in every solve), so a
// parent reads its gathered input with plain loads.
template <typename T>
struct Slots {
    cx<T>* G;                // slot 0; slot 1 at G + half
    int64_t half;            // work rows of the class * k
    const int32_t* relinds;  // row in the parent's front of each update row
};

// Raw loads of a staged operand element, combined after they have arrived.
template <typename T>
struct Raw2 {
    cx<T> a, b;
};
// The value v, passed through an empty asm: the compiler must hold it in a
// register at this point, so a load that produced it is not sunk into the
// arm of a later select (where its wait would sit inside a branch, one
// round trip per element).
template <class X>
__device__ __forceinline__ X Opaque(X v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// An empty asm that reads v: every load that may still write v is waited for
// here, so its register is free of pending writes on every path that
// follows (without it, a register whose load result is used on one branch
// only can be reused on the other while the load is still in flight, and
// the reuse then waits for every outstanding load).
template <class X>
__device__ __forceinline__ void Sink(const X& v)
{
    asm volatile("" ::"v"(v));
}

// Branch-free staging of inner operands, in two steps so that a thread's
// index loads (B: the struct rows of the update columns) are all in flight
// together before the value loads that depend on them.  Every load is issued
// unconditionally from a valid address (F: col < s, the forward inner range;
// B: the struct list carries a sentinel entry, so structs[ustart] exists at a
// root).
template <int PH>
__device__ __forceinline__ int32_t StageIndex(const NodeDev& nd, const int32_t* structs, int col)
{
    return PH == PH_F ? 0 : structs[nd.ustart + max(col - nd.s, 0)];
}

template <typename T, int PH>
__device__ __forceinline__ cx<T> StageValue(const NodeDev& nd, const Slots<T>& gs, const cx<T>* Xp,
                                            const cx<T>* W, int col, int rr, int k, int32_t srow)
{
    if (PH == PH_F) {
        const int64_t g = (nd.w + col) * k + rr;
        return gs.G[g] + gs.G[gs.half + g] + Xp[(int64_t)(nd.off + col) * k + rr];
    }
    const cx<T>* p = col < nd.s ? W + (nd.w + col) * k + rr : Xp + (int64_t)srow * k + rr;
    return *p;
}

// N staged elements of a thread; at(q) gives element q's (inner index,
// right-hand side) as an int2.
template <typename T, int PH, int N, class AT>
__device__ __forceinline__ void StageBatch(const NodeDev& nd, const int32_t* structs,
                                           const Slots<T>& gs, const cx<T>* Xp, const cx<T>* W,
                                           int k, const AT& at, cx<T> (&sv)[N])
{
    int32_t sx[N];
#pragma unroll
    for (int q = 0; q < N; ++q) sx[q] = StageIndex<PH>(nd, structs, at(q).x);
    if (PH == PH_B) {
#pragma unroll
        for (int q = 0; q < N; ++q) sx[q] = Opaque(sx[q]);
    }
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const int2 p = at(q);
        sv[q] = StageValue<T, PH>(nd, gs, Xp, W, p.x, p.y, k, sx[q]);
    }
}

// Finish of output row `row`, right-hand side r, product a.  F: top rows
// are y (into W); a bottom row is g + a, with g the gathered value of that
// row, written into the parent's slot copy at parent row `prow`.  B: the
// node's Xp rows.
template <typename T, int PH>
__device__ __forceinline__ void Finish(const NodeDev& nd, const Slots<T>& gs, cx<T>* Xp, cx<T>* W,
                                       int row, int r, int k, cx<T> a, cx<T> g, int prow)
{
    if (PH == PH_F) {
        if (row < nd.s)
            W[(nd.w + row) * k + r] = a;
        else if (nd.cslot >= 0)
            gs.G[nd.cslot * gs.half + (int64_t)(nd.pw + prow) * k + r] = g + a;
    } else {
        Xp[(int64_t)(nd.off + row) * k + r] = a;
    }
}

template <typename T, int PH>
__device__ __forceinline__ void FinishGather(const NodeDev& nd, const Slots<T>& gs, cx<T>* Xp,
                                             cx<T>* W, int row, int r, int k, cx<T> a)
{
    if (PH == PH_F && row >= nd.s) {
        const int64_t g = (nd.w + row) * k + r;
        Finish<T, PH>(nd, gs, Xp, W, row, r, k, a, gs.G[g] + gs.G[gs.half + g],
                      gs.relinds[nd.ustart + row - nd.s]);
    } else {
        Finish<T, PH>(nd, gs, Xp, W, row, r, k, a, czero<T>(), 0);
    }
}

// --------------------------------------------------------------------------
// Front-solve products on the matrix cores (k >= 8 right-hand sides).
//
// One 16x16x4 real MFMA computes D(16x16) += A(16x4) B(4x16).  A complex
// product out = M v (M: rows x inner, v: inner x k) maps onto two of them by
// splitting the 16 output columns into the real parts (j < 8) and imaginary
// parts (j >= 8) of 8 right-hand sides:
//     D += Re(M) [Re v | Im v]  +  Im(M) [-Im v | Re v],
// which is exactly 8 real flops per complex multiply-add, all on the MFMA
// units (no 3M recombination).  Lane l of a wave holds A(l % 16, l / 16) and
// B(l / 16, l % 16); its accumulator register q holds D(row, l % 16) with
// row = 4 (l / 16) + q for the f32 instruction and l / 16 + 4 q for f64.
// --------------------------------------------------------------------------
typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v4d __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma;
template <>
struct Mfma<float> {
    typedef v4f acc;
    static __device__ __forceinline__ acc step(float a, float b, acc c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lk, int q) { return 4 * lk + q; }
};
template <>
struct Mfma<double> {
    typedef v4d acc;
    static __device__ __forceinline__ acc step(double a, double b, acc c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lk, int q) { return lk + 4 * q; }
};

// Factor loads in flight per lane of the level and fused-subtree kernels, and
// staged elements (columns x right-hand sides) per chunk by front precision:
// smaller chunks keep fewer staging registers, so more workgroups fit on a CU.
constexpr int PSP_MVM_U = 8, PSP_MVM_CHUNK32 = 1024, PSP_MVM_CHUNK64 = 512;

// --------------------------------------------------------------------------
// Hand-offs between workgroups of one XCD.  Workgroups are dealt to the 8
// XCDs round-robin (blockIdx % 8 == XCC_ID, checked at device set-up), and
// the XCDs' L2 caches are not coherent with each other, so a hand-off that
// stays on one XCD needs no L2 write-back: the producer waits for its
// stores and raises a device-scope counter, the consumer sees the counter
// and reads the data with loads that miss the L1 (L2Buf).
// --------------------------------------------------------------------------
__device__ __forceinline__ int XccId()
{
    return __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20);  // HW_REG_XCC_ID, bits 3:0
}

__device__ __forceinline__ int LoadAgent(const int32_t* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int AddAgent(int32_t* p, int v)
{
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// This wave's stores (and loads) have completed: s_waitcnt vmcnt(0).
__device__ __forceinline__ void WaitVmem() { __builtin_amdgcn_s_waitcnt(0xF70); }

// Loads of vectors that another workgroup of the XCD wrote during this
// launch: buffer loads with the device-scope cache policy (sc1), which miss
// the CU's L1 and read the L2, where the producer's stores are.  They are
// ordinary loads to the compiler (scheduled and batched like any other).
// Measured on MI355X: with sc0 loads (workgroup scope), or with an L1
// invalidate after the wait, results went wrong whenever a vector row was
// not a whole number of 128-byte lines (a line then holds rows of two nodes,
// and the L1 can keep or regain a copy read before the other node was
// written); with sc1 loads every case is exact, and so are full
// device-scope release/acquire fences, which also write back and
// invalidate the L2.  A buffer spans at most 4 GiB (the host checks).
template <typename T>
struct L2Buf {
    __amdgpu_buffer_rsrc_t r;
    __device__ explicit L2Buf(const void* base)
        : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, -1, 0x00020000))
    {
    }
    __device__ cx<T> operator[](int64_t i) const
    {
        constexpr int kSc1 = 16;  // cache policy: SC1 set (device scope)
        const uint32_t off = (uint32_t)(i * (int64_t)sizeof(cx<T>));
        cx<T> v;
        if constexpr (sizeof(T) == 4) {
            const auto x = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, kSc1);
            __builtin_memcpy(&v, &x, 8);
        } else {
            const auto x = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kSc1);
            __builtin_memcpy(&v, &x, 16);
        }
        return v;
    }
};

__global__ void k_xcc_probe(int32_t* out)
{
    if (threadIdx.x == 0) out[blockIdx.x] = XccId();
}

// Matrix-core path (k >= 8).  One workgroup per tile; wave w owns rows
// 16 (w / WK) .. +16 of the tile and every WK-th 4-column step of its inner
// range.  The inner range streams through LDS in chunks of CC columns (all
// KB right-hand sides of a pass); the factor loads of the next U steps are
// issued before the current ones are consumed.  Waves that share rows sum
// their partial tiles in a fixed order through LDS.  Loads that do not
// depend on the products (the first factor batch, the staged vector, and
// for single-pass blocks the gathered bottom rows of F) are issued right
// after the tile record arrives, so a workgroup waits for few memory round
// trips.
//
// Inner slices of a split row block (slot >= 0) write partial sums to their
// slots.  With redc given, the host has placed the slices of each row block
// at launch positions that are equal mod 8, so they all run on one XCD: each
// slice waits for its partial stores and counts itself in redc[red], and the
// last to arrive sums the block's slots in slot order (the sums of
// k_mv_reduce, bit for bit), finishes the rows and clears the counter.
// Without redc a reduce launch follows.  Tiles with no rows are holes in that
// placement and exit at once.
//
// MvmTile is the work of one workgroup on tile tl (nrows > 0).
template <typename T, int PH, int RT, int KB>
__device__ __forceinline__ void MvmTile(const SolveTile tl, const int32_t* structs,
                                        const Slots<T> gs, const cx<T>* L, const cx<T>* LT,
                                        cx<T>* Xp, cx<T>* W, cx<T>* P, int k, int32_t* redc,
                                        const SolveTile* reds);

template <typename T, int PH, int RT, int KB>
__global__ __launch_bounds__(256) void k_mvm(const SolveTile* tiles, int start,
                                                     const int32_t* structs,
                                                     Slots<T> gs, const cx<T>* L,
                                                     const cx<T>* LT, cx<T>* Xp, cx<T>* W,
                                                     cx<T>* P, int k, int32_t* redc,
                                                     const SolveTile* reds)
{
    const SolveTile tl = tiles[start + blockIdx.x];
    if (tl.nrows <= 0) return;
    MvmTile<T, PH, RT, KB>(tl, structs, gs, L, LT, Xp, W, P, k, redc, reds);
}

template <typename T, int PH, int RT, int KB>
__device__ __forceinline__ void MvmTile(const SolveTile tl, const int32_t* structs,
                                        const Slots<T> gs, const cx<T>* L, const cx<T>* LT,
                                        cx<T>* Xp, cx<T>* W, cx<T>* P, int k, int32_t* redc,
                                        const SolveTile* reds)
{
    typedef typename Mfma<T>::acc acc_t;
    constexpr int NWV = 4, NT = 64 * NWV, WR = RT / 16, WK = NWV / WR, NB = KB / 8;
    constexpr int U = PSP_MVM_U;  // factor loads in flight per lane
    // staged inner columns per chunk
    constexpr int CC = (sizeof(T) == 4 ? PSP_MVM_CHUNK32 : PSP_MVM_CHUNK64) / KB;
    constexpr bool PRE = KB <= 16 && PH == PH_F;
    static_assert(WR * WK == NWV && CC % 4 == 0 && U >= 1, "tile shape");
    static_assert(WK == 1 || 2 * CC * KB >= WR * (WK / 2) * NB * 256,
                  "reduction scratch must fit in vs");
    const NodeDev nd = tl.nd;
    const int s = nd.s, fs = nd.s + nd.u;
    const cx<T>* Lf = L + nd.l;
    const cx<T>* Lt = LT + nd.l;
    __shared__ cx<T> vs[CC][KB];
    __shared__ int arrived;
    T* red = reinterpret_cast<T*>(&vs[0][0]);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave / WK, wk = wave % WK;
    const int li = lane & 15, lk = lane >> 4;
    // Finishing lanes: wk == 0, li < 8; element (b, q) is row
    // 16 wr + row(lk, q) of the tile and right-hand side 8 b + li of the pass.
    const bool fin = wk == 0 && li < 8 && tl.slot < 0;
    cx<T> pre[PRE ? NB : 1][4];
    int prow[4] = {0, 0, 0, 0};
    if (PRE && fin && k <= KB) {
        // branch-free: rows clamped into the node's front (the relinds list
        // carries a sentinel entry), unused values dropped at the finish
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int row = min(tl.row0 + 16 * wr + Mfma<T>::row(lk, q), fs - 1);
            prow[q] = gs.relinds[nd.ustart + max(row - s, 0)];
        }
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = min(tl.row0 + 16 * wr + Mfma<T>::row(lk, q), fs - 1);
                const int64_t o = (nd.w + row) * k + min(8 * b + li, k - 1);
                pre[PRE ? b : 0][q] = gs.G[o] + gs.G[gs.half + o];
            }
    }
    for (int r0 = 0; r0 < k; r0 += KB) {
        const int kc = min(KB, k - r0);
        acc_t acc[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = acc_t{0, 0, 0, 0};
        for (int cb = tl.col0; cb < tl.col1; cb += CC) {
            const int ncol = min(CC, tl.col1 - cb);
            const int nsteps = (ncol + 3) >> 2;
            const int mine = nsteps > wk ? (nsteps - wk + WK - 1) / WK : 0;
            cx<T> m[U];
            // Factor entries from a scalar base and a per-lane offset, rows
            // clamped into the tile, unmasked: the unused triangles of the
            // solve storage are zero, and a wave reads at most 3 columns past
            // the chunk (inside the storage's zero padding), against zeros
            // in the staged vector.  Steps past the wave's share reload its
            // last one and are not multiplied.
            const int fa = PH == PH_F ? fs : s;
            const cx<T>* Ab = (PH == PH_F ? Lf : Lt) + tl.row0 + (int64_t)cb * fa;
            const uint32_t la = (uint32_t)(min(16 * wr + li, tl.nrows - 1) + (4 * wk + lk) * fa);
            const int64_t ustep = (int64_t)(4 * WK) * fa;
            const int ulast = max(mine - 1, 0);
            auto load = [&](cx<T>* dst, int u0) {
#pragma unroll
                for (int u = 0; u < U; ++u) dst[u] = (Ab + min(u0 + u, ulast) * ustep)[la];
            };
            // staging loads first, then the first factor batch, all in flight
            // together; the LDS stores wait only for the staging loads
            // (columns up to the next multiple of 4 are written, as zeros
            // past the range)
            constexpr int SPT = CC * KB / NT;
            const int nst = min(CC, 4 * nsteps);
            cx<T> sv[SPT];
            StageBatch<T, PH>(nd, structs, gs, Xp, W, k, [&](int q) {
                const int e = tid + NT * q, c = e / KB, r = e % KB;
                return int2{cb + min(c, ncol - 1), min(r0 + r, k - 1)};
            }, sv);
            load(m, 0);
            LdsBarrier();  // the previous chunk's (or pass's) readers are done with vs
#pragma unroll
            for (int q = 0; q < SPT; ++q) {
                const int e = tid + NT * q, c = e / KB, r = e % KB;
                if (c < nst) vs[c][r] = (r < kc && c < ncol) ? sv[q] : czero<T>();
            }
            LdsBarrier();
            for (int u0 = 0; u0 < mine; u0 += U) {
                cx<T> mn[U];
                if (u0 + U < mine) load(mn, u0 + U);
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (u0 + u < mine) {
                        const int c = 4 * (wk + WK * (u0 + u)) + lk;
#pragma unroll
                        for (int b = 0; b < NB; ++b) {
                            const cx<T> v = vs[c][8 * b + (li & 7)];
                            const T b1 = li < 8 ? v.r : v.i;
                            const T b2 = li < 8 ? -v.i : v.r;
                            acc[b] = Mfma<T>::step(m[u].r, b1, acc[b]);
                            acc[b] = Mfma<T>::step(m[u].i, b2, acc[b]);
                        }
                    }
                }
                if (u0 + U < mine) {
#pragma unroll
                    for (int u = 0; u < U; ++u) m[u] = mn[u];
                }
            }
        }
        // waves that share rows sum their partial tiles by a fixed tree
        if (WK > 1) {
            for (int h = WK / 2; h >= 1; h >>= 1) {
                LdsBarrier();
                if (wk >= h && wk < 2 * h) {
#pragma unroll
                    for (int b = 0; b < NB; ++b)
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            red[(((wr * h + wk - h) * NB + b) * 64 + lane) * 4 + q] = acc[b][q];
                }
                LdsBarrier();
                if (wk < h) {
#pragma unroll
                    for (int b = 0; b < NB; ++b)
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            acc[b][q] += red[(((wr * h + wk) * NB + b) * 64 + lane) * 4 + q];
                }
            }
        }
        if (wk == 0) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const T val = acc[b][q];
                    const T other = __shfl_xor(val, 8, 64);
                    const int rl = 16 * wr + Mfma<T>::row(lk, q);  // row within the tile
                    const int rr = 8 * b + li;                      // right-hand side within the pass
                    if (li < 8 && rl < tl.nrows && rr < kc) {
                        const cx<T> a{val, other};
                        const int row = tl.row0 + rl;
                        if (tl.slot >= 0)
                            P[((int64_t)tl.slot * 64 + rl) * k + r0 + rr] = a;
                        else if (PRE && k <= KB)
                            Finish<T, PH>(nd, gs, Xp, W, row, rr, k, a, pre[PRE ? b : 0][q],
                                          prow[q]);
                        else
                            FinishGather<T, PH>(nd, gs, Xp, W, row, r0 + rr, k, a);
                    }
                }
            }
        }
    }
    if (redc != nullptr && tl.slot >= 0) {
        const int rix = tl.pad_;
        WaitVmem();
        LdsBarrier();  // every wave's partial sums have reached the L2
        if (tid == 0) arrived = AddAgent(redc + rix, 1);
        LdsBarrier();
        const SolveTile it = reds[rix];  // row block: first slot, slot count
        if (__builtin_amdgcn_readfirstlane(arrived) == it.col1 - 1) {
            const L2Buf<T> lP(P);
            constexpr int kS = 16;  // slots loaded together (more: in groups)
            for (int e = tid; e < it.nrows * k; e += NT) {
                const int rl = e / k, r = e % k;
                cx<T> a = czero<T>();
                for (int j0 = 0; j0 < it.col1; j0 += kS) {
                    // all of a group's loads in flight at once, then summed in
                    // slot order (slots past the block add nothing)
                    cx<T> v[kS];
#pragma unroll
                    for (int j = 0; j < kS; ++j)
                        v[j] = lP[((int64_t)(it.col0 + min(j0 + j, it.col1 - 1)) * 64 + rl) * k + r];
#pragma unroll
                    for (int j = 0; j < kS; ++j)
                        if (j0 + j < it.col1) a = a + v[j];
                }
                FinishGather<T, PH>(it.nd, gs, Xp, W, it.row0 + rl, r, k, a);
            }
            if (tid == 0) redc[rix] = 0;  // no slice of this launch counts any more
        }
    }
}

// --------------------------------------------------------------------------
// Fused subtree solves (8 <= k <= KB).  One persistent launch runs every
// level of a phase from the class's cut depth down (forward: deepest level
// first; backward: the cut level first).  The subtrees under the cut nodes
// are split over nqueues queues, one per XCD: a workgroup reads the XCD it
// runs on (hardware register XCC_ID), serves queue XCC_ID (if there is
// one; no two XCDs ever serve one queue), takes its tiles in
// queue order (an atomic head), and before reading a tile's inputs waits
// until the nodes the tile depends on have all their row blocks done
// (per-node counters; forward: the node's children, backward: its nearest
// ancestor with pivots).  Producer and consumer of every hand-off then
// share one XCD and its L2, and the hand-off is the cross-CU one of the
// memory model, with no L2 write-back:
//   producer: its stores; s_waitcnt vmcnt(0) (the stores have reached the
//             L2); barrier; one lane increments the node's counter;
//   consumer: polls the counter; barrier; reads what the launch wrote with
//             loads that miss the L1 and read the L2 (sc1, L2Buf).
// Counters and heads are device-scope atomics.  Near the cut a row block
// is cut into inner slices: slices write partial sums to their slots, and
// the slice that arrives last (a counter per row block) sums the slots in
// slot order and finishes the rows, so sums have a fixed order.
//
// No workgroup waits forever: a tile's dependencies come earlier in its
// queue, and the earliest tile not yet done is held by a running workgroup
// whose own earlier tiles are done, so it proceeds.  A queue that no
// workgroup serves (fewer XCDs than queues) is run, tile by tile, by the
// last workgroup to leave (an exit counter).  The per-tile body is that of
// k_mvm: waves own 16-row blocks and every WK-th 4-column step, the inner
// range streams through LDS, factor loads run U steps ahead; the first
// factor batch of a tile is issued before its dependency wait.  The launch
// state (counters, heads) is cleared by the copy-in or zero-set launch
// that precedes each panel solve.
// --------------------------------------------------------------------------
// The fused launch's buffers read through the L2: slot copies, work vectors,
// panel vector, partial sums.
template <typename T>
struct L2Bufs {
    L2Buf<T> G, W, X, P;
};

// StageBatch of the fused launch: the same operand (the same sums in the
// same order) with the vectors written in this launch read from the L2.
// Backward: both the work-vector and the panel-vector element are loaded
// (a buffer per vector, so no per-lane choice of descriptor) and one kept.
template <typename T, int PH, int N, class AT>
__device__ __forceinline__ void StageBatchL2(const NodeDev& nd, const int32_t* structs,
                                             const Slots<T>& gs, const L2Bufs<T>& lb,
                                             const cx<T>* Xp, int k, const AT& at,
                                             cx<T> (&sv)[N])
{
    int32_t sx[N];
#pragma unroll
    for (int q = 0; q < N; ++q) sx[q] = StageIndex<PH>(nd, structs, at(q).x);
    if (PH == PH_B) {
#pragma unroll
        for (int q = 0; q < N; ++q) sx[q] = Opaque(sx[q]);
    }
    // all loads first, combined once they have arrived
    cx<T> ra[N], rb[N], rc[N];
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const int2 p = at(q);
        const int col = p.x, rr = p.y;
        if (PH == PH_F) {
            const int64_t g = (nd.w + col) * k + rr;
            ra[q] = (lb.G[g]);
            rb[q] = (lb.G[gs.half + g]);
            rc[q] = (Xp[(int64_t)(nd.off + col) * k + rr]);
        } else {
            ra[q] = (lb.W[(nd.w + min(col, nd.s - 1)) * k + rr]);
            rb[q] = (lb.X[(int64_t)sx[q] * k + rr]);
        }
    }
#pragma unroll
    for (int q = 0; q < N; ++q) {
        if (PH == PH_F)
            sv[q] = ra[q] + rb[q] + rc[q];
        else
            sv[q] = at(q).x < nd.s ? ra[q] : rb[q];
    }
}

template <typename T, int PH, int RT, int KB>
__global__ __launch_bounds__(256) void k_mvq(const QTile* tiles, const int32_t* qstart,
                                             const QRed* reds, const int4* dep,
                                             const NodeDev* nodes, int32_t* sync, int nnodes,
                                             int nqueues, const int32_t* structs, Slots<T> gs,
                                             const cx<T>* L, const cx<T>* LT, cx<T>* Xp,
                                             cx<T>* W, cx<T>* P, int k)
{
    typedef typename Mfma<T>::acc acc_t;
    constexpr int NWV = 4, NT = 256, WR = RT / 16, WK = NWV / WR, NB = KB / 8;
    constexpr int U = PSP_MVM_U;
    constexpr int CC = (sizeof(T) == 4 ? PSP_MVM_CHUNK32 : PSP_MVM_CHUNK64) / KB;
    constexpr int SPT = CC * KB / NT;
    constexpr bool PRE = PH == PH_F;
    static_assert(WR * WK == NWV && CC % 4 == 0 && SPT >= 1, "tile shape");
    static_assert(WK == 1 || 2 * CC * KB >= WR * (WK / 2) * NB * 256,
                  "reduction scratch must fit in vs");
    int32_t* done = sync;
    int32_t* head = sync + nnodes;
    int32_t* exitc = head + nqueues;
    int32_t* redc = exitc + 1;
    const L2Bufs<T> lb{L2Buf<T>(gs.G), L2Buf<T>(W), L2Buf<T>(Xp), L2Buf<T>(P)};
    __shared__ cx<T> vs[CC][KB];
    __shared__ int bc[4];
    T* red = reinterpret_cast<T*>(&vs[0][0]);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave / WK, wk = wave % WK;
    const int li = lane & 15, lk = lane >> 4;

    // One queue tile: wait for its dependencies, the products, the finish
    // (or the partial sums and, for the last slice, the row block's sum and
    // finish), then the node's counter.
    auto runTile = [&](int idx) {
        const QTile qt = tiles[idx];
        const NodeDev nd = nodes[qt.node];
        const int s = nd.s, fs = nd.s + nd.u;
        const int fa = PH == PH_F ? fs : s;
        const cx<T>* Ab0 = (PH == PH_F ? L : LT) + nd.l + qt.row0;
        const uint32_t la = (uint32_t)(min(16 * wr + li, qt.nrows - 1) + (4 * wk + lk) * fa);
        const int64_t ustep = (int64_t)(4 * WK) * fa;
        // the first factor batch (independent of the dependencies)
        const int ncol0 = min(CC, qt.col1 - qt.col0);
        const int nsteps0 = (max(ncol0, 0) + 3) >> 2;
        const int mine0 = nsteps0 > wk ? (nsteps0 - wk + WK - 1) / WK : 0;
        cx<T> m[U];
        {
            const cx<T>* Ab = Ab0 + (int64_t)qt.col0 * fa;
            const int ulast = max(mine0 - 1, 0);
#pragma unroll
            for (int u = 0; u < U; ++u) m[u] = (Ab + min(u, ulast) * ustep)[la];
        }
        int prow[4] = {0, 0, 0, 0};
        const bool fin = wk == 0 && li < 8 && qt.red < 0;
        if (PRE && fin) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = min(qt.row0 + 16 * wr + Mfma<T>::row(lk, q), fs - 1);
                prow[q] = gs.relinds[nd.ustart + max(row - s, 0)];
            }
        }
        // dependencies
        {
            const int4 dp = dep[qt.node];
            if (tid == 0) {
                if (dp.x >= 0)
                    while (LoadAgent(done + dp.x) < dp.z) __builtin_amdgcn_s_sleep(1);
                if (dp.y >= 0)
                    while (LoadAgent(done + dp.y) < dp.w) __builtin_amdgcn_s_sleep(1);
            }
            LdsBarrier();
        }
        cx<T> pre[PRE ? NB : 1][4], pre1[PRE ? NB : 1][4];
        if (PRE && fin) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int row = min(qt.row0 + 16 * wr + Mfma<T>::row(lk, q), fs - 1);
                    const int64_t o = (nd.w + row) * k + min(8 * b + li, k - 1);
                    pre[PRE ? b : 0][q] = (lb.G[o]);
                    pre1[PRE ? b : 0][q] = (lb.G[gs.half + o]);
                }
        }
        acc_t acc[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = acc_t{0, 0, 0, 0};
        for (int cb = qt.col0; cb < qt.col1; cb += CC) {
            const int ncol = min(CC, qt.col1 - cb);
            const int nsteps = (ncol + 3) >> 2;
            const int mine = nsteps > wk ? (nsteps - wk + WK - 1) / WK : 0;
            const cx<T>* Ab = Ab0 + (int64_t)cb * fa;
            const int ulast = max(mine - 1, 0);
            auto load = [&](cx<T>* dst, int u0) {
#pragma unroll
                for (int u = 0; u < U; ++u) dst[u] = (Ab + min(u0 + u, ulast) * ustep)[la];
            };
            const int nst = min(CC, 4 * nsteps);
            cx<T> sv[SPT];
            StageBatchL2<T, PH>(nd, structs, gs, lb, Xp, k, [&](int q) {
                const int e = tid + NT * q, c = e / KB, r = e % KB;
                return int2{cb + min(c, ncol - 1), min(r, k - 1)};
            }, sv);
            if (cb != qt.col0) load(m, 0);
            LdsBarrier();  // the previous chunk's readers are done with vs
#pragma unroll
            for (int q = 0; q < SPT; ++q) {
                const int e = tid + NT * q, c = e / KB, r = e % KB;
                if (c < nst) vs[c][r] = (r < k && c < ncol) ? sv[q] : czero<T>();
            }
            LdsBarrier();
            for (int u0 = 0; u0 < mine; u0 += U) {
                cx<T> mn[U];
                if (u0 + U < mine) load(mn, u0 + U);
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (u0 + u < mine) {
                        const int c = 4 * (wk + WK * (u0 + u)) + lk;
#pragma unroll
                        for (int b = 0; b < NB; ++b) {
                            const cx<T> v = vs[c][8 * b + (li & 7)];
                            const T b1 = li < 8 ? v.r : v.i;
                            const T b2 = li < 8 ? -v.i : v.r;
                            acc[b] = Mfma<T>::step(m[u].r, b1, acc[b]);
                            acc[b] = Mfma<T>::step(m[u].i, b2, acc[b]);
                        }
                    }
                }
                if (u0 + U < mine) {
#pragma unroll
                    for (int u = 0; u < U; ++u) m[u] = mn[u];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) Sink(m[u].r), Sink(m[u].i);
        if (WK > 1) {  // waves that share rows sum their partial tiles by a fixed tree
            for (int h = WK / 2; h >= 1; h >>= 1) {
                LdsBarrier();
                if (wk >= h && wk < 2 * h) {
#pragma unroll
                    for (int b = 0; b < NB; ++b)
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            red[(((wr * h + wk - h) * NB + b) * 64 + lane) * 4 + q] = acc[b][q];
                }
                LdsBarrier();
                if (wk < h) {
#pragma unroll
                    for (int b = 0; b < NB; ++b)
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            acc[b][q] += red[(((wr * h + wk) * NB + b) * 64 + lane) * 4 + q];
                }
            }
        }
        if (wk == 0) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const T val = acc[b][q];
                    const T other = __shfl_xor(val, 8, 64);
                    const int rl = 16 * wr + Mfma<T>::row(lk, q);
                    const int rr = 8 * b + li;
                    if (li < 8 && rl < qt.nrows && rr < k) {
                        const cx<T> a{val, other};
                        if (qt.red >= 0)
                            P[((int64_t)qt.slot * 64 + rl) * k + rr] = a;
                        else if (PRE)
                            Finish<T, PH>(nd, gs, Xp, W, qt.row0 + rl, rr, k, a,
                                          pre[PRE ? b : 0][q] + pre1[PRE ? b : 0][q], prow[q]);
                        else
                            Finish<T, PH>(nd, gs, Xp, W, qt.row0 + rl, rr, k, a, czero<T>(), 0);
                    }
                }
            }
        }
        WaitVmem();
        LdsBarrier();
        bool rowsDone = qt.red < 0;
        if (!rowsDone) {
            const QRed rd = reds[qt.red];
            if (tid == 0) bc[2] = AddAgent(redc + qt.red, 1);
            LdsBarrier();
            if (__builtin_amdgcn_readfirstlane(bc[2]) == rd.nslots - 1) {
                // the last slice: every other slice's partials are in L2
                for (int e = tid; e < rd.nrows * k; e += NT) {
                    const int rl = e / k, r = e % k;
                    cx<T> a = czero<T>();
                    for (int j = 0; j < rd.nslots; ++j)
                        a = a + lb.P[((int64_t)(rd.slot0 + j) * 64 + rl) * k + r];
                    if (PH == PH_F && rd.row0 + rl >= nd.s) {
                        const int row = rd.row0 + rl;
                        const int64_t g = (nd.w + row) * k + r;
                        Finish<T, PH>(nd, gs, Xp, W, row, r, k, a, lb.G[g] + lb.G[gs.half + g],
                                      gs.relinds[nd.ustart + row - nd.s]);
                    } else {
                        Finish<T, PH>(nd, gs, Xp, W, rd.row0 + rl, r, k, a, czero<T>(), 0);
                    }
                }
                WaitVmem();
                LdsBarrier();
                rowsDone = true;
            }
        }
        if (rowsDone && tid == 0) AddAgent(done + qt.node, 1);
    };

    // queue x is served by the workgroups of XCD x only (none of another XCD
    // ever shares it); XCDs without a queue go straight to the exit
    const int q = __builtin_amdgcn_readfirstlane(XccId());
    int cur = 0, qs = 0, qn = 0;
    if (q < nqueues) {
        qs = qstart[q];
        qn = qstart[q + 1] - qs;
        if (tid == 0) bc[0] = AddAgent(head + q, 1);
        LdsBarrier();
        cur = __builtin_amdgcn_readfirstlane(bc[0]);
    }
    while (cur < qn) {
        int nxt = 0;
        if (tid == 0) nxt = AddAgent(head + q, 1);  // the tile after this one
        runTile(qs + cur);
        if (tid == 0) bc[1] = nxt;
        LdsBarrier();
        cur = __builtin_amdgcn_readfirstlane(bc[1]);
    }
    // the last workgroup out runs the queues no workgroup served
    if (tid == 0) bc[3] = AddAgent(exitc, 1);
    LdsBarrier();
    if (__builtin_amdgcn_readfirstlane(bc[3]) != (int)gridDim.x - 1) return;
    for (int qq = 0; qq < nqueues; ++qq) {
        if (tid == 0) bc[0] = LoadAgent(head + qq);
        LdsBarrier();
        const int served = __builtin_amdgcn_readfirstlane(bc[0]);
        LdsBarrier();
        if (served != 0) continue;
        for (int i = qstart[qq]; i < qstart[qq + 1]; ++i) runTile(i);
    }
}


// --------------------------------------------------------------------------
// Complex tile engine on the matrix cores: one 256-thread workgroup computes
// an RT x 64 complex tile C = A B over an inner range, K staged through LDS
// 16 columns at a time with two buffers (the global loads of stage s + 1
// are in flight while stage s is multiplied).  Waves split the tile into
// WRW x WCW parts; each wave holds RB x CB accumulator blocks of 16 rows x 8
// complex columns (16 real MFMA columns: real parts, then imaginary parts).
// A and B are read through policy objects: a(i, k) and b(k, j) return the
// complex entry or zero outside the operand.
// --------------------------------------------------------------------------
template <int RT, int CT = 64>
struct TileShape {
    static constexpr int WRW = RT >= 64 ? 2 : 1;       // waves along rows
    static constexpr int WCW = 4 / WRW;                // waves along columns
    static constexpr int RB = RT / 16 / WRW;           // 16-row blocks per wave
    static constexpr int CB = CT / 8 / WCW;            // 8-column blocks per wave
};

constexpr int kBK = 16;  // inner columns per LDS stage (solve tiles)

// la(i, k) / lb(k, j) return the raw loads of one A / B element and must be
// safe to call for every i < RT, j < CT and k in [kbeg, kend) (loaders clamp
// their own indices, so a stage's loads are issued without branches);
// fa(i, k, raw) / fb(k, j, raw) turn them into the operand value, masks and
// scaling included.  The transforms run when the next stage is written to
// LDS, after this stage's matrix-core steps, so the loads of stage s + 1 are
// in flight while stage s computes.
// skipAbove: (lower-triangular results) a 16-row x 8-column block whose
// rows all lie above its columns, i + skipAbove < j for tile coordinates
// (i, j), is not multiplied; its accumulators stay zero.  1 << 30: none.
template <typename T, int RT, bool BJFAST, int BK = kBK, int CT = 64, class LA, class FA, class LB,
          class FB>
__device__ __forceinline__ void MmaTile(const LA& la, const FA& fa, const LB& lb, const FB& fb,
                                        int kbeg, int kend, cx<T> (*As)[BK][RT + 1],
                                        cx<T> (*Bs)[BK][CT + 1],
                                        typename Mfma<T>::acc (&acc)[TileShape<RT, CT>::RB]
                                                                   [TileShape<RT, CT>::CB],
                                        int skipAbove = 1 << 30)
{
    typedef TileShape<RT, CT> S;
    constexpr int kBK = BK;
    constexpr int NA = RT * kBK / 256, NBL = CT * kBK / 256;  // loads per thread per stage
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave / S::WCW, wc = wave % S::WCW;
    const int li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int a = 0; a < S::RB; ++a)
#pragma unroll
        for (int b = 0; b < S::CB; ++b) acc[a][b] = typename Mfma<T>::acc{0, 0, 0, 0};
    if (kend <= kbeg) return;
    decltype(la(0, kbeg)) ra[NA];
    decltype(lb(kbeg, 0)) rb[NBL];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int q = 0; q < NA; ++q) {
            const int e = tid + 256 * q, i = e % RT, kk = e / RT;
            ra[q] = la(i, min(k0 + kk, kend - 1));
        }
#pragma unroll
        for (int q = 0; q < NBL; ++q) {
            const int e = tid + 256 * q;
            const int j = BJFAST ? e % CT : e / kBK, kk = BJFAST ? e / CT : e % kBK;
            rb[q] = lb(min(k0 + kk, kend - 1), j);
        }
    };
    auto put = [&](int buf, int k0) {
#pragma unroll
        for (int q = 0; q < NA; ++q) {
            const int e = tid + 256 * q, i = e % RT, kk = e / RT;
            As[buf][kk][i] = k0 + kk < kend ? fa(i, k0 + kk, ra[q]) : czero<T>();
        }
#pragma unroll
        for (int q = 0; q < NBL; ++q) {
            const int e = tid + 256 * q;
            const int j = BJFAST ? e % CT : e / kBK, kk = BJFAST ? e / CT : e % kBK;
            Bs[buf][kk][j] = k0 + kk < kend ? fb(k0 + kk, j, rb[q]) : czero<T>();
        }
    };
    const int nst = (kend - kbeg + kBK - 1) / kBK;
    fetch(kbeg);
    LdsBarrier();  // the caller's previous use of As / Bs is over
    put(0, kbeg);
    LdsBarrier();
    for (int st = 0; st < nst; ++st) {
        const int buf = st & 1;
        if (st + 1 < nst) fetch(kbeg + (st + 1) * kBK);
#pragma unroll
        for (int k4 = 0; k4 < kBK / 4; ++k4) {
            cx<T> av[S::RB];
#pragma unroll
            for (int a = 0; a < S::RB; ++a) av[a] = As[buf][4 * k4 + lk][16 * (wr * S::RB + a) + li];
#pragma unroll
            for (int b = 0; b < S::CB; ++b) {
                const int c0 = 8 * (wc * S::CB + b);  // the block's first column (wave-uniform)
                if (16 * (wr * S::RB + S::RB - 1) + 15 + skipAbove < c0) continue;
                const cx<T> v = Bs[buf][4 * k4 + lk][c0 + (li & 7)];
                const T b1 = li < 8 ? v.r : v.i;
                const T b2 = li < 8 ? -v.i : v.r;
#pragma unroll
                for (int a = 0; a < S::RB; ++a) {
                    if (16 * (wr * S::RB + a) + 15 + skipAbove < c0) continue;
                    acc[a][b] = Mfma<T>::step(av[a].r, b1, acc[a][b]);
                    acc[a][b] = Mfma<T>::step(av[a].i, b2, acc[a][b]);
                }
            }
        }
        if (st + 1 < nst) put(buf ^ 1, kbeg + (st + 1) * kBK);
        LdsBarrier();
    }
}

// Epilogue over the tile elements this lane finishes, one 16-row block at a
// time: ld(i, j) is called for every element of the block first (it must be
// safe for any i < RT, j < CT: the loads of the block are all in flight
// together), then st(i, j, value, loaded) for the elements of lanes with
// l % 16 < 8, after pairing the real and imaginary halves.
template <typename T, int RT, int CT = 64, class LD, class ST>
__device__ __forceinline__ void MmaEpilogue(const typename Mfma<T>::acc (&acc)[TileShape<RT, CT>::RB]
                                                                             [TileShape<RT, CT>::CB],
                                            const LD& ld, const ST& st)
{
    typedef TileShape<RT, CT> S;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wr = wave / S::WCW, wc = wave % S::WCW;
    const int li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int a = 0; a < S::RB; ++a) {
        decltype(ld(0, 0)) old[S::CB][4];
#pragma unroll
        for (int b = 0; b < S::CB; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                old[b][q] = ld(16 * (wr * S::RB + a) + Mfma<T>::row(lk, q), 8 * (wc * S::CB + b) + (li & 7));
#pragma unroll
        for (int b = 0; b < S::CB; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const T val = acc[a][b][q];
                const T other = __shfl_xor(val, 8, 64);
                if (li < 8)
                    st(16 * (wr * S::RB + a) + Mfma<T>::row(lk, q), 8 * (wc * S::CB + b) + li,
                       cx<T>{val, other}, old[b][q]);
            }
    }
}

// Calls f(i, j, value) for every tile element this lane finishes (lanes with
// l % 16 < 8 after pairing the real and imaginary halves).
template <typename T, int RT, int CT = 64, class F>
__device__ __forceinline__ void MmaForEach(const typename Mfma<T>::acc (&acc)[TileShape<RT, CT>::RB]
                                                                            [TileShape<RT, CT>::CB],
                                           const F& f)
{
    typedef TileShape<RT, CT> S;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wr = wave / S::WCW, wc = wave % S::WCW;
    const int li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int a = 0; a < S::RB; ++a)
#pragma unroll
        for (int b = 0; b < S::CB; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const T val = acc[a][b][q];
                const T other = __shfl_xor(val, 8, 64);
                if (li < 8)
                    f(16 * (wr * S::RB + a) + Mfma<T>::row(lk, q), 8 * (wc * S::CB + b) + li,
                      cx<T>{val, other});
            }
}

// Batched tile GEMM on the matrix cores: C (+)= +/- opA(A) diag(D) opB(B)
// over a list of 64x64 tiles (see GemmFlags), through the tile engine.
// 8-column LDS stages keep the registers low enough for 5 waves per SIMD in
// FP32 and 3 in FP64 without spills; on the factorization's many short-K
// Schur updates that occupancy is worth more than deeper stages.
template <typename T>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 5 : 3) void k_gemm_mma(const GemmDesc* descs, const GemmTile* tiles,
                                                  int tileStart, cx<T>* b0, int64_t st0,
                                                  cx<T>* b1, int64_t st1, cx<T>* b2,
                                                  int64_t st2, cx<T>* b3)
{
    constexpr int BK = 8;  // inner columns per stage
    constexpr int TS = 64;   // 128x128 tiles measured slower on the Schur updates
    __shared__ cx<T> As[2][BK][TS + 1];
    __shared__ cx<T> Bs[2][BK][TS + 1];
    const GemmTile tl = tiles[tileStart + blockIdx.x];
    const GemmDesc g = descs[tl.desc];
    const int bt = blockIdx.y;
    cx<T>* bases[4] = {b0 + (int64_t)bt * st0, b1 + (int64_t)bt * st1, b2 + (int64_t)bt * st2,
                       b3 + (int64_t)bt * st0};  // b3 (LT) has L's stride
    const cx<T>* A = bases[g.abuf] + g.a;
    const cx<T>* B = bases[g.bbuf] + g.b;
    cx<T>* Cm = bases[g.cbuf] + g.c;
    const cx<T>* D = bases[g.dbuf] + g.d;
    const int tm = tl.tm, tn = tl.tn, f = g.flags;
    int kbeg = 0, kend = g.K;
    if (f & G_BUNIT) kbeg = tn;
    if (f & G_AUNIT) kend = min(kend, tm + TS);
    // Every loader reads from a clamped index inside the operand's rectangle
    // (always allocated), so a stage's loads go out without branches; the
    // masks, the unit diagonals and the diag(D) scaling are applied when the
    // stage is written to LDS.  Without G_HASD the D load reads A's first
    // element (a broadcast) and is ignored.
    const bool hasd = f & G_HASD;
    const cx<T>* Dv = hasd ? D : A;
    const int64_t dinc = hasd ? g.dinc : 0;
    auto la = [&](int i, int k) {
        return Raw2<T>{A[min(tm + i, g.M - 1) + (int64_t)k * g.lda], Dv[(int64_t)k * dinc]};
    };
    auto fa = [&](int i, int k, const Raw2<T>& r) {
        const int gi = tm + i;
        cx<T> v = r.a;
        if (f & G_AUNIT) v = gi > k ? v : (gi == k ? cx<T>{T(1), T(0)} : czero<T>());
        if (hasd) v = v * r.b;
        return gi < g.M ? v : czero<T>();
    };
    typename Mfma<T>::acc acc[TileShape<TS, TS>::RB][TileShape<TS, TS>::CB];
    // lower-triangular results: blocks above the diagonal are not computed
    // (only tiles that cross the diagonal have any)
    const int skip = (f & G_CLOWER) ? tm - tn : 1 << 30;
    if (f & G_BTRANS) {
        auto lb = [&](int k, int j) { return B[min(tn + j, g.N - 1) + (int64_t)k * g.ldb]; };
        auto fb = [&](int, int j, cx<T> v) { return tn + j < g.N ? v : czero<T>(); };
        MmaTile<T, TS, true, BK, TS>(la, fa, lb, fb, kbeg, kend, As, Bs, acc, skip);
    } else {
        auto lb = [&](int k, int j) { return B[k + (int64_t)min(tn + j, g.N - 1) * g.ldb]; };
        auto fb = [&](int k, int j, cx<T> v) {
            const int gj = tn + j;
            if (f & G_BUNIT) v = k > gj ? v : (k == gj ? cx<T>{T(1), T(0)} : czero<T>());
            return gj < g.N ? v : czero<T>();
        };
        MmaTile<T, TS, false, BK, TS>(la, fa, lb, fb, kbeg, kend, As, Bs, acc, skip);
    }
    auto offset = [&](int gi, int gj) {
        return (f & G_CTRANS) ? gj + (int64_t)gi * g.ldc : gi + (int64_t)gj * g.ldc;
    };
    auto keep = [&](int gi, int gj) {
        return gi < g.M && gj < g.N && !((f & G_CLOWER) && gi < gj);
    };
    if (f & G_BETA0) {
        MmaForEach<T, TS, TS>(acc, [&](int i, int j, cx<T> v) {
            const int gi = tm + i, gj = tn + j;
            if (keep(gi, gj)) Cm[offset(gi, gj)] = (f & G_NEG) ? -v : v;
        });
    } else {
        // C is read for a whole row block before the first store goes out.
        auto ld = [&](int i, int j) { return Cm[offset(min(tm + i, g.M - 1), min(tn + j, g.N - 1))]; };
        MmaEpilogue<T, TS, TS>(acc, ld, [&](int i, int j, cx<T> v, cx<T> c) {
            const int gi = tm + i, gj = tn + j;
            if (keep(gi, gj)) Cm[offset(gi, gj)] = c + ((f & G_NEG) ? -v : v);
        });
    }
}

// Sum of the inner slices of split row blocks, in slot order, then the
// phase's finish.  One workgroup per row block.
template <typename T, int PH>
__device__ __forceinline__ void MvReduceItem(const SolveTile& it, const Slots<T>& gs, cx<T>* Xp,
                                             cx<T>* W, const cx<T>* P, int k)
{
    const NodeDev nd = it.nd;
    for (int e = threadIdx.x; e < it.nrows * k; e += kThreads) {
        const int rl = e / k, r = e % k;
        cx<T> a = czero<T>();
        for (int j = 0; j < it.col1; ++j) a = a + P[((int64_t)(it.col0 + j) * 64 + rl) * k + r];
        FinishGather<T, PH>(nd, gs, Xp, W, it.row0 + rl, r, k, a);
    }
}

template <typename T, int PH>
__global__ __launch_bounds__(kThreads) void k_mv_reduce(const SolveTile* items, int start,
                                                        Slots<T> gs, cx<T>* Xp,
                                                        cx<T>* W, const cx<T>* P, int k)
{
    MvReduceItem<T, PH>(items[start + blockIdx.x], gs, Xp, W, P, k);
}

// --------------------------------------------------------------------------
// Merged solves: F in blocks of 16 x 16 (see BlockTile), one launch per depth
// group and direction, for any number of right-hand sides.
//
// A workgroup has 4 waves; wave q owns output block ob0 + q of its tile and
// runs over the tile's inner blocks.  Factor blocks go straight from HBM into
// the A operands: forward, lane l of a step t loads row l % 16 of column
// 4 t + l / 16; backward the block is used transposed, and lane l loads rows
// 4 (l / 16) .. + 4 of column l % 16 (the four steps then take the inner
// index in the order t, 4 + t, 8 + t, 12 + t, which the staged vector
// follows).  Either way a wave reads whole blocks, 2 or 4 KB, contiguous.
// The inner vector is shared by the waves through LDS, CB blocks at a time.  Up
// to 16 right-hand sides (BlockTileWork) a chunk has one buffer and two barriers:
// its vector is loaded once the chunk before is multiplied, the first chunk's
// before anything is waited for, and a ring of U factor blocks a wave is in flight
// throughout, across chunks.  Passes of 32 (BlockTileWide) have two buffers and one
// barrier a chunk, with two chunks of vector and factor blocks in flight.
//
// What bounds it: for k <= 16 the factor stream (HBM) and, on small launches,
// the dependent round trips record -> (indices ->) operands -> stores; for
// k >= 32 the matrix cores.
// --------------------------------------------------------------------------
template <typename T>
struct BlockBufs {
    const cx<T>* F;      // one panel's blocks
    cx<T>* V;            // the class's solve vector (VecRows)
    const int32_t* bsrc;
    const int32_t* blist;
    const int32_t* udst;
    cx<T>* P;            // partial sums, 64 rows per slot
    int64_t w, g0, g1;   // VecRows
    int32_t xrows, zero; // zero: a block of zeros in F
};

typedef const __attribute__((address_space(4))) int32_t* ConstInts;
__device__ __forceinline__ ConstInts Const(const void* p) { return (ConstInts)(uintptr_t)p; }

__device__ __forceinline__ int Uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Vector rows of an update row: where it is written, and what is added (the
// children's contributions to it, and what a pivot row of the parent holds).
template <typename T>
__device__ __forceinline__ cx<T> UpdateBase(const BlockBufs<T>& a, int u, int work, int leaf,
                                            int dst, int r, int k)
{
    cx<T> g = czero<T>();
    if (!leaf) g = a.V[(a.g0 + u) * k + r] + a.V[(a.g1 + work) * k + r];
    if (dst < a.xrows) g = g + a.V[(int64_t)dst * k + r];
    return g;
}

// Output row `row` of a merged front (product v), right-hand side r.
template <typename T, int PH>
__device__ __forceinline__ void BlockFinish(const BlockBufs<T>& a, int x0, int w0, int u0, int s,
                                            int u, int sb, int leaf, int row, int r, int k, cx<T> v)
{
    if (PH == PH_B) {
        if (row < s) a.V[(int64_t)(x0 + row) * k + r] = v;
    } else if (row < s) {
        a.V[(a.w + x0 + row) * k + r] = v;
    } else if (row >= kBlk * sb && row - kBlk * sb < u) {
        const int ur = u0 + row - kBlk * sb, dst = a.udst[ur];
        a.V[(int64_t)dst * k + r] = UpdateBase(a, ur, w0 + row, leaf, dst, r, k) + v;
    }
}

template <typename T, int KB>
struct BlockShape {
    static constexpr int NB = KB / 8;
    // blocks in flight per wave: 32 registers, so that 4 to 7 workgroups fit on
    // a CU (twice as many in flight and half the workgroups: 5% slower)
    static constexpr int U = sizeof(T) == 4 ? 4 : 2;
    // inner blocks per chunk of the staged vector
    static constexpr int CB = 16 / (KB / 8) / (sizeof(T) == 8 ? 2 : 1);
    static constexpr int SPT = CB * kBlk * KB / 256;  // staged elements per thread
    // accumulators that a block's products are dealt to (BlockSum)
    static constexpr int NA = KB == 8 ? (sizeof(T) == 4 ? 4 : 2) : 1;
    // steps whose vector operands are read ahead: a whole block of them would
    // take 64 more registers in FP64 with KB = 16
    static constexpr int OS = sizeof(T) == 4 ? 4 : 2;
    static_assert(CB % U == 0 || U % CB == 0, "chunk shape");
};

// Fields of a tile (scalar loads).
struct TileRec {
    int x0, w0, u0, s, u, sb, leaf, ob0, nob, ib0, nib, lst, slot, red;
    int base, lo, hi;  // forward: of wave q's output block
    __device__ TileRec(ConstInts t, int q)
        : x0(t[0]), w0(t[1]), u0(t[2]), s(t[3]), u(t[4]), sb(t[5]), leaf(t[6]), ob0(t[7]),
          nob(t[8]), ib0(t[9]), nib(t[10]), lst(t[11]), slot(t[12]), red(t[13]),
          base(t[16 + q]), lo(t[20 + q]), hi(t[24 + q])
    {
    }
};

// An output element of a sliced tile (row rl of the tile, right-hand side r) and
// the operands that finish it.
template <typename T, int PH>
struct SliceElement {
    int rl, r, dst;
    cx<T> x, ga, gb;
    __device__ __forceinline__ void Load(const BlockBufs<T>& a, const TileRec& t, int e, int r0,
                                         int kc, int k)
    {
        rl = e / kc;
        r = r0 + e % kc;
        if constexpr (PH == PH_F) {
            const int row = kBlk * t.ob0 + rl, ur = row - kBlk * t.sb;
            dst = 0;
            ga = gb = czero<T>();
            if (ur >= 0) {
                dst = a.udst[t.u0 + ur];
                if (!t.leaf) {
                    ga = a.V[(a.g0 + t.u0 + ur) * k + r];
                    gb = a.V[(a.g1 + t.w0 + row) * k + r];
                }
                x = a.V[(int64_t)dst * k + r];
            }
        }
    }
    __device__ __forceinline__ void Store(const BlockBufs<T>& a, const TileRec& t, int k, cx<T> v)
    {
        const int row = kBlk * t.ob0 + rl;
        if constexpr (PH == PH_B) {
            if (row < t.s) a.V[(int64_t)(t.x0 + row) * k + r] = v;
        } else if (row < t.s) {
            a.V[(a.w + t.x0 + row) * k + r] = v;
        } else if (row >= kBlk * t.sb && row - kBlk * t.sb < t.u) {
            cx<T> g = czero<T>();
            if (!t.leaf) g = ga + gb;
            if (dst < a.xrows) g = g + x;
            a.V[(int64_t)dst * k + r] = g + v;
        }
    }
};

// Inner slices of a tile: each wave's partial sums are in P; the slice that
// arrives last sums the slots in slot order and finishes the rows.  That is the
// end of a launch's longest chain (7 to 10 us of 24 at 144 x 128 x 80, k = 16 in
// FP64, one element after another), so a thread's elements go together: all
// their operands and slots are in flight at once, as far as registers allow
// (8 or 16 values).  Operands loaded before the arrival count gained nothing.
template <typename T, int PH, int KB>
__device__ __forceinline__ void SumSlices(const TileRec& t, const BlockBufs<T>& a, int k, int r0,
                                          int kc, int32_t* redc, const BlockRed* reds)
{
    __shared__ int arrived;
    const int tid = threadIdx.x;
    constexpr int E = 64 * KB / 256, G = E < 4 ? E : 4;  // elements per thread, at a time
    constexpr int kS = (PH == PH_F || sizeof(T) == 4 ? 16 : 8) / G;  // slots loaded together
    WaitVmem();
    LdsBarrier();  // every wave's partial sums have reached the L2
    if (tid == 0) arrived = AddAgent(redc + t.red, 1);
    LdsBarrier();
    const ConstInts rd = Const(reds + t.red);
    const int slot0 = rd[9], nslots = rd[10];
    if (Uni(arrived) != nslots - 1) return;
    const L2Buf<T> lP(a.P);
    const int ne = t.nob * kBlk * kc;
    for (int e0 = 0; e0 + Uni(tid & ~63) < ne; e0 += 256 * G) {
        // (elements past the end are not loaded or repeat the last)
        SliceElement<T, PH> el[G];
        cx<T> v[G];
#pragma unroll
        for (int i = 0; i < G; ++i) {
            v[i] = czero<T>();
            if (i == 0 || e0 + 256 * i < ne)
                el[i].Load(a, t, min(e0 + 256 * i + tid, ne - 1), r0, kc, k);
        }
        for (int j0 = 0; j0 < nslots; j0 += kS) {
            cx<T> pv[G][kS];
#pragma unroll
            for (int i = 0; i < G; ++i)
                if (i == 0 || e0 + 256 * i < ne) {
#pragma unroll
                    for (int j = 0; j < kS; ++j) {
                        const int64_t slot = slot0 + min(j0 + j, nslots - 1);
                        pv[i][j] = lP[(slot * 64 + el[i].rl) * k + el[i].r];
                    }
                }
#pragma unroll
            for (int i = 0; i < G; ++i)
#pragma unroll
                for (int j = 0; j < kS; ++j)
                    if (j0 + j < nslots) v[i] = v[i] + pv[i][j];
        }
#pragma unroll
        for (int i = 0; i < G; ++i)
            if (e0 + 256 * i + tid < ne) el[i].Store(a, t, k, v[i]);
    }
    if (tid == 0) redc[t.red] = 0;  // no slice of this launch counts any more
}

// Where a lane's 4 rows (rows row(lk, p) of output block ob) go, if they are
// update rows.
template <typename T>
struct FinishOps {
    int32_t dst[4];
    __device__ void Load(const BlockBufs<T>& a, const TileRec& t, int ob, int lk)
    {
        if (ob < t.sb) return;
        const int32_t* p = a.udst + t.u0 + kBlk * (ob - t.sb);
#pragma unroll
        for (int i = 0; i < 4; ++i) dst[i] = p[Mfma<T>::row(lk, i)];
    }
};

// Stores a wave's output block: products of right-hand sides r0 + 8 n + li
// (li < 8, below r0 + kc), as partial sums of a slice or finished.  The loads
// of an update block are issued together for each n.
template <typename T, int PH, int NB, class SUM>
__device__ __forceinline__ void StoreBlock(const BlockBufs<T>& a, const TileRec& t, int q, int k,
                                           int r0, int kc, const FinishOps<T>& fo,
                                           const SUM (&sum)[NB])
{
    typedef typename SUM::real S;
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int ob = t.ob0 + q;
    cx<S> o[NB][4];
#pragma unroll
    for (int n = 0; n < NB; ++n) {
        const typename SUM::vec v = sum[n].Value();
#pragma unroll
        for (int p = 0; p < 4; ++p) o[n][p] = cx<S>{S(v[p]), S(__shfl_xor(v[p], 8, 64))};
    }
    auto each = [&](auto&& f) {
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int p = 0; p < 4; ++p) f(n, p, Mfma<T>::row(lk, p), 8 * n + li);
    };
    if (t.slot >= 0) {
        cx<T>* out = a.P + ((int64_t)t.slot * 64 + kBlk * q) * k + r0;
        each([&](int n, int p, int row, int r) {
            if (li < 8 && r < kc) out[row * k + r] = cvt<T>(o[n][p]);
        });
    } else if (PH == PH_B) {
        cx<T>* out = a.V + (int64_t)(t.x0 + kBlk * ob) * k + r0;
        each([&](int n, int p, int row, int r) {
            if (li < 8 && r < kc && kBlk * ob + row < t.s) out[row * k + r] = cvt<T>(o[n][p]);
        });
    } else if (ob < t.sb) {
        cx<T>* out = a.V + (a.w + t.x0 + kBlk * ob) * k + r0;
        each([&](int n, int p, int row, int r) {
            if (li < 8 && r < kc && kBlk * ob + row < t.s) out[row * k + r] = cvt<T>(o[n][p]);
        });
    } else {
        // an update row: the children's contributions to it and, for a pivot
        // row of the parent, what that holds
        const int ru = kBlk * (ob - t.sb);
        const cx<T>* g0 = a.V + (a.g0 + t.u0 + ru) * k + r0;
        const cx<T>* g1 = a.V + (a.g1 + t.w0 + kBlk * ob) * k + r0;
        cx<T>* out[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) out[p] = a.V + (int64_t)fo.dst[p] * k + r0;
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const int r = 8 * n + li, rc = min(r, kc - 1);
            cx<T> x[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) x[p] = out[p][rc];
            if (!t.leaf) {
                cx<T> ga[4], gb[4];
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    ga[p] = g0[Mfma<T>::row(lk, p) * k + rc];
                    gb[p] = g1[Mfma<T>::row(lk, p) * k + rc];
                }
#pragma unroll
                for (int p = 0; p < 4; ++p) o[n][p] = cvt<S>(ga[p]) + cvt<S>(gb[p]) + o[n][p];
            }
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const cx<T> v = cvt<T>(fo.dst[p] < a.xrows ? cvt<S>(x[p]) + o[n][p] : o[n][p]);
                if (li < 8 && r < kc && ru + Mfma<T>::row(lk, p) < t.u) out[p][r] = v;
            }
        }
    }
}

// The sum of an output block over the inner blocks.  A block's products run
// through accumulators of their own, from zero, and are added here: one
// accumulator through a whole slice (up to 768 columns) rounds two to four times
// as much as the sums need, and GMRES with FP32 fronts then stalls before its
// tolerance (40^3, k = 1, to 1e-5: 21 steps, 18 so).  TWICE: in twice the
// precision of T (FP64: a value and what its additions rounded off, by the
// Moller-Knuth sum of two numbers), for few right-hand sides, where nothing else
// of a launch takes the time.  What a sweep of u + v differs from those of u and
// of v by, the rounding of its vectors and sums, k = 1, with one accumulator and
// so: 40^3 FP32 3.7e-7 and 1.2e-7, FP64 7.0e-16 and 2.5e-16; 61 x 47 x 83 FP32
// 5.4e-7 and 1.1e-7, FP64 8.4e-16 and 2.5e-16; k = 32 at 100^3 FP32 7.2e-7 and
// 2.1e-7, FP64 1.3e-15 and 4.0e-16.
template <typename T, bool TWICE>
struct BlockSum {
    typedef typename Mfma<T>::acc vec;
    typedef T real;
    vec v{0, 0, 0, 0};
    __device__ __forceinline__ void Add(const vec& z) { v += z; }
    __device__ __forceinline__ vec Value() const { return v; }
};
template <>
struct BlockSum<float, true> {
    typedef Mfma<double>::acc vec;
    typedef double real;
    vec v{0, 0, 0, 0};
    __device__ __forceinline__ void Add(const Mfma<float>::acc& z)
    {
        v += __builtin_convertvector(z, vec);
    }
    __device__ __forceinline__ vec Value() const { return v; }
};
template <>
struct BlockSum<double, true> {
    typedef Mfma<double>::acc vec;
    typedef double real;
    vec v{0, 0, 0, 0}, off{0, 0, 0, 0};
    __device__ __forceinline__ void Add(const vec& z)
    {
        const vec s = v + z, d = s - v;
        off += (v - (s - d)) + (z - d);
        v = s;
    }
    __device__ __forceinline__ vec Value() const { return v + off; }
};

// One workgroup: up to KB = 8 or 16 right-hand sides of a tile (shared by
// k_block and k_block_batch).  Reads of the vector and of the index lists may
// run past the tile's inner range (up to a chunk; the buffers are padded);
// those rows are not multiplied.
template <typename T, int PH, int KB>
__device__ __forceinline__ void BlockTileWork(const BlockTile* tp, const BlockBufs<T>& a, int k,
                                              int32_t* redc, const BlockRed* reds)
{
    typedef typename Mfma<T>::acc acc_t;
    typedef BlockShape<T, KB> S;
    constexpr int NB = S::NB, CB = S::CB, SPT = S::SPT, U = S::U, NA = S::NA, OS = S::OS;
    constexpr int RP = 256 / KB;  // rows staged by one load of the workgroup
    __shared__ cx<T> vs[CB * kBlk][KB];
    const int tid = threadIdx.x, lane = tid & 63, q = Uni(tid >> 6);
    const int li = lane & 15, lk = lane >> 4;
    const TileRec t(Const(tp), q);
    const uint32_t loff = PH == PH_F ? lk * kBlk + li : li * kBlk + 4 * lk;
    const uint32_t rk = min(tid % KB, k - 1);           // staged right-hand side
    const uint32_t voff = (tid / KB) * k + rk;

    // backward: lane l holds the block at inner index c CB + l
    int list = 0;
    auto loadList = [&](int c) {
        if constexpr (PH == PH_B)
            list = a.blist[4 * (int64_t)(t.lst + t.ib0 + min(c * CB + lane, t.nib - 1)) + q];
    };
    // loads of the wave's block at inner index c CB + i (the zero block where
    // it has none)
    cx<T> m[U][4];
    int id[U];
    auto issue = [&](int u, int c, int i) {
        int blk;
        if constexpr (PH == PH_F) {
            const int j = t.ib0 + c * CB + i;
            blk = j >= t.lo && j < t.hi ? t.base + j : a.zero;
        } else {
            blk = __builtin_amdgcn_readlane(list, i);
        }
        if (c * CB + i >= t.nib) blk = a.zero;
        id[u] = blk;
        const cx<T>* p = a.F + (int64_t)blk * (kBlk * kBlk);
#pragma unroll
        for (int st = 0; st < 4; ++st) m[u][st] = (p + (PH == PH_F ? 4 * kBlk * st : st))[loff];
    };
    cx<T> sa[SPT], sg[PH == PH_F ? SPT : 1];
    auto stage = [&](int c) {
        if constexpr (PH == PH_F) {
            const int row0 = kBlk * (t.ib0 + c * CB);
            const cx<T>* x = a.V + (int64_t)(t.x0 + row0) * k;
            const cx<T>* g = a.V + (a.g1 + t.w0 + row0) * k;
#pragma unroll
            for (int p = 0; p < SPT; ++p) sa[p] = (x + p * RP * k)[voff];
            if (!t.leaf) {
#pragma unroll
                for (int p = 0; p < SPT; ++p) sg[p] = (g + p * RP * k)[voff];
            } else {
#pragma unroll
                for (int p = 0; p < SPT; ++p) sg[p] = czero<T>();
            }
        } else {
            const int32_t* ix = a.bsrc + (int64_t)kBlk * (t.lst + t.ib0 + c * CB);
            uint32_t sx[SPT];
#pragma unroll
            for (int p = 0; p < SPT; ++p) sx[p] = (uint32_t)(ix + p * RP)[tid / KB];
#pragma unroll
            for (int p = 0; p < SPT; ++p) sa[p] = a.V[sx[p] * (uint32_t)k + rk];
        }
    };
    auto put = [&]() {
#pragma unroll
        for (int p = 0; p < SPT; ++p) {
            const int c = tid / KB + RP * p;
            // backward: inner index 4 a + b of a block sits at 4 b + a
            const int row = PH == PH_F ? c : (c & ~15) | ((c & 3) << 2) | ((c >> 2) & 3);
            cx<T> v = sa[p];
            if constexpr (PH == PH_F) v = v + sg[p];
            vs[row][tid % KB] = mk(v.r, v.i);
        }
    };
    acc_t acc[NA][NB];
    BlockSum<T, KB == 8> sum[NB];
    auto clear = [&]() {
#pragma unroll
        for (int h = 0; h < NA; ++h)
#pragma unroll
            for (int n = 0; n < NB; ++n) acc[h][n] = acc_t{0, 0, 0, 0};
    };
    auto fold = [&]() {
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            if constexpr (NA == 4)
                sum[n].Add((acc[0][n] + acc[1][n]) + (acc[2][n] + acc[3][n]));
            else if constexpr (NA == 2)
                sum[n].Add(acc[0][n] + acc[1][n]);
            else
                sum[n].Add(acc[0][n]);
        }
        clear();
    };
    // vector operands of OS steps from step st of the block at inner index i of
    // the chunk
    struct Operand {
        cx<T> v[OS][NB];
    };
    auto operand = [&](int i, int st) {
        Operand o;
#pragma unroll
        for (int j = 0; j < OS; ++j)
#pragma unroll
            for (int n = 0; n < NB; ++n)
                o.v[j][n] = vs[kBlk * i + 4 * (st + j) + lk][8 * n + (li & 7)];
        return o;
    };
    auto multiply = [&](int u, int st, const Operand& o) {
#pragma unroll
        for (int j = 0; j < OS; ++j)
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                const cx<T> v = o.v[j][n];
                const T b1 = li < 8 ? v.r : v.i;
                const T b2 = li < 8 ? -v.i : v.r;
                const int h1 = NA == 4 ? 2 * ((st + j) & 1) : 0, h2 = NA > 1 ? h1 + 1 : 0;
                acc[h1][n] = Mfma<T>::step(m[u][st + j].r, b1, acc[h1][n]);
                acc[h2][n] = Mfma<T>::step(m[u][st + j].i, b2, acc[h2][n]);
            }
    };
    // the chunk's products, half a ring at a time, each register group refilled
    // as soon as it is used; blocks that the tile does not have (3 to 38% of a
    // launch) are skipped: 11.8 to 11.3 ms a sweep at 100^3 k = 16 in FP32
    auto run = [&](int c) {
        const int left = t.nib - c * CB;
        constexpr int H = U / 2;
        Operand o = operand(0, 0);
        for (int i0 = 0;; i0 += U) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int u = H * h; u < H * h + H; ++u) {
                    const int i1 = min(i0 + u + 1, CB - 1);
                    if (id[u] == a.zero) {
                        o = operand(i1, 0);
                        continue;
                    }
#pragma unroll
                    for (int st = 0; st < 4; st += OS) {
                        const Operand o1 =
                            st + OS < 4 ? operand(i0 + u, st + OS) : operand(i1, 0);
                        multiply(u, st, o);
                        o = o1;
                    }
                    fold();
                }
                if (i0 + H * h + H >= left) return;
#pragma unroll
                for (int u = H * h; u < H * h + H; ++u) issue(u, c, i0 + u + U);
            }
            if (i0 + U >= CB) return;
        }
    };
    // the first loads all go out before the first wait
    loadList(0);
    stage(0);
#pragma unroll
    for (int u = 0; u < U; ++u) issue(u, 0, u);
    __builtin_amdgcn_sched_barrier(0);
    const bool own = q < t.nob;
    FinishOps<T> fo;
    if (PH == PH_F && own && t.slot < 0) fo.Load(a, t, t.ob0 + q, lk);
    clear();
    put();
    LdsBarrier();
    run(0);
    const int nch = (t.nib + CB - 1) / CB;
    for (int c = 1; c < nch; ++c) {
        loadList(c);
        stage(c);
        LdsBarrier();  // the previous chunk's readers are done
        put();
        LdsBarrier();
        run(c);
    }
    if (own) StoreBlock<T, PH, NB>(a, t, q, k, 0, k, fo, sum);
    if (redc != nullptr && t.slot >= 0) SumSlices<T, PH, KB>(t, a, k, 0, k, redc, reds);
}

// The same for one pass (right-hand sides KB pass .. + KB) of a wide block.
// Bound by the matrix cores and by waiting for loads, so the vector and the
// factor blocks of the next two chunks of CB inner blocks are in flight, each in
// its own registers, while one is multiplied from LDS (two buffers), and blocks
// that a tile does not have are skipped.  The passes are workgroups of one
// launch: a loop over them in one workgroup, on one staged chunk ahead, took
// 41.7 ms a sweep at 100^3 k = 64 FP32 and 66.0 in FP64 (28.5 and 50.4 now);
// 15.8 ms at 120 x 96 x 60 k = 32 FP32 (11.3).  CB = 4 and three workgroups a CU
// spill registers and were slower.  A block's sums for 8 right-hand sides run from
// zero at a time (BlockSum): accumulators of all four, kept beside their sums,
// took 29.0 and 52.0 ms.
template <typename T, int KB>
struct WideShape {
    static constexpr int NB = KB / 8;
    static constexpr int CB = 2;
    static constexpr int SPT = CB * kBlk * KB / 256;  // staged elements per thread
};

template <typename T, int PH, int KB>
__device__ __forceinline__ void BlockTileWide(const BlockTile* tp, const BlockBufs<T>& a, int k,
                                              int pass, int32_t* redc, const BlockRed* reds)
{
    typedef typename Mfma<T>::acc acc_t;
    typedef WideShape<T, KB> S;
    constexpr int NB = S::NB, CB = S::CB, SPT = S::SPT;
    __shared__ cx<T> vs[2][CB * kBlk][KB];
    const int tid = threadIdx.x, lane = tid & 63, q = Uni(tid >> 6);
    const int li = lane & 15, lk = lane >> 4;
    const uint32_t loff = PH == PH_F ? lk * kBlk + li : li * kBlk + 4 * lk;
    struct Chunk {
        int blk[CB];  // wave-uniform
        cx<T> m[CB][4];
    };
    const int r0 = KB * pass, kc = min(KB, k - r0);
    constexpr int RP = 256 / KB;  // rows staged by one load of the workgroup
    const int rr = r0 + min(tid % KB, kc - 1);
    const uint32_t voff = (tid / KB) * k + rr;
    struct Stage {
        cx<T> a[SPT], g[PH == PH_F ? SPT : 1];
    };
    const TileRec t(Const(tp), q);
    const ConstInts bl = Const(a.blist) + 4 * (int64_t)(t.lst + t.ib0) + q;
    const int32_t* src = a.bsrc + (int64_t)kBlk * (t.lst + t.ib0);
    const int nch = (t.nib + CB - 1) / CB;
    auto factor = [&](int c, Chunk& d) {
#pragma unroll
        for (int b = 0; b < CB; ++b) {
            const int i = c * CB + b;
            int blk = a.zero;
            if (i < t.nib) {
                if constexpr (PH == PH_F) {
                    const int j = t.ib0 + i;
                    if (j >= t.lo && j < t.hi) blk = t.base + j;
                } else {
                    blk = bl[4 * i];
                }
            }
            if (q >= t.nob) blk = a.zero;
            d.blk[b] = blk;
            const cx<T>* p = a.F + (int64_t)blk * (kBlk * kBlk);
#pragma unroll
            for (int st = 0; st < 4; ++st) d.m[b][st] = (p + (PH == PH_F ? 4 * kBlk * st : st))[loff];
        }
    };
    BlockSum<T, false> sum[NB];
    // (stages past the end read the last chunk again, unused)
    int32_t sx[PH == PH_B ? SPT : 1];
    auto indices = [&](int c) {
        if constexpr (PH == PH_B) {
            const int32_t* ix = src + min(c, nch - 1) * CB * kBlk;
#pragma unroll
            for (int p = 0; p < SPT; ++p) sx[p] = (ix + p * RP)[tid / KB];
        }
    };
    auto stage = [&](int c, Stage& d) {
        if constexpr (PH == PH_F) {
            const int row0 = kBlk * (t.ib0 + min(c, nch - 1) * CB);
            const cx<T>* x = a.V + (int64_t)(t.x0 + row0) * k;
            const cx<T>* g = a.V + (a.g1 + t.w0 + row0) * k;
#pragma unroll
            for (int p = 0; p < SPT; ++p) d.a[p] = (x + p * RP * k)[voff];
            if (!t.leaf) {
#pragma unroll
                for (int p = 0; p < SPT; ++p) d.g[p] = (g + p * RP * k)[voff];
            } else {
#pragma unroll
                for (int p = 0; p < SPT; ++p) d.g[p] = czero<T>();
            }
        } else {
#pragma unroll
            for (int p = 0; p < SPT; ++p) d.a[p] = a.V[(int64_t)sx[p] * k + rr];
        }
    };
    auto put = [&](int buf, const Stage& d) {
#pragma unroll
        for (int p = 0; p < SPT; ++p) {
            const int c = tid / KB + RP * p;
            const int row = PH == PH_F ? c : (c & ~15) | ((c & 3) << 2) | ((c >> 2) & 3);
            cx<T> v = d.a[p];
            if constexpr (PH == PH_F) v = v + d.g[p];
            vs[buf][row][tid % KB] = mk(v.r, v.i);
        }
    };
    Chunk d0, d1;
    Stage s0, s1;
    indices(0);
    stage(0, s0);
    indices(1);
    stage(1, s1);
    indices(2);
    factor(0, d0);
    factor(1, d1);
    auto step = [&](int c, Chunk& d, Stage& sv) {
        put(c & 1, sv);
        stage(c + 2, sv);
        indices(c + 3);
        LdsBarrier();
#pragma unroll
        for (int b = 0; b < CB; ++b) {
            if (d.blk[b] == a.zero) continue;
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                acc_t acc{0, 0, 0, 0};
#pragma unroll
                for (int st = 0; st < 4; ++st) {
                    const cx<T> v = vs[c & 1][kBlk * b + 4 * st + lk][8 * n + (li & 7)];
                    const T b1 = li < 8 ? v.r : v.i;
                    const T b2 = li < 8 ? -v.i : v.r;
                    acc = Mfma<T>::step(d.m[b][st].r, b1, acc);
                    acc = Mfma<T>::step(d.m[b][st].i, b2, acc);
                }
                sum[n].Add(acc);
            }
        }
        factor(c + 2, d);
    };
    for (int c = 0; c < nch; c += 2) {
        step(c, d0, s0);
        if (c + 1 >= nch) break;
        step(c + 1, d1, s1);
    }
    if (q < t.nob) {
        FinishOps<T> fo;
        if (PH == PH_F && t.slot < 0) fo.Load(a, t, t.ob0 + q, lk);
        StoreBlock<T, PH, NB>(a, t, q, k, r0, kc, fo, sum);
    }
    if (redc != nullptr && t.slot >= 0) SumSlices<T, PH, KB>(t, a, k, r0, kc, redc, reds);
}

// One tile, right-hand sides KB pass .. + KB (KB 8 and 16: one pass).
template <typename T, int PH, int KB>
__device__ __forceinline__ void BlockWork(const BlockTile* tp, const BlockBufs<T>& a, int k,
                                          int pass, int32_t* redc, const BlockRed* reds)
{
    if constexpr (KB <= 16)
        BlockTileWork<T, PH, KB>(tp, a, k, redc, reds);
    else
        BlockTileWide<T, PH, KB>(tp, a, k, pass, redc, reds);
}

// Workgroups per CU the register budget allows for (the most without spills).
template <typename T, int PH, int KB>
constexpr int BlockOccupancy()
{
    if (KB > 16) return 2;
    const int wide = KB == 16, f64 = sizeof(T) == 8;
    return PH == PH_B ? 6 - f64 - wide : 4 - wide;
}

// Workgroup g of a launch of `count` tiles and `passes` passes: the passes of
// a tile are 8 workgroups apart, so they run on one XCD at about the same time
// and the later ones find the factor blocks in its L2.  redc: counters, one
// set of nreds per pass.
template <typename T, int PH, int KB>
__global__ __launch_bounds__(256, (BlockOccupancy<T, PH, KB>())) void k_block(
    const BlockTile* tiles, BlockBufs<T> a, int k, int count, int passes, int32_t* redc, int nreds,
    const BlockRed* reds)
{
    int tile = blockIdx.x, pass = 0;
    if (KB > 16) {
        tile = blockIdx.x / (8 * passes) * 8 + blockIdx.x % 8;
        pass = blockIdx.x / 8 % passes;
        if (tile >= count) return;
        if (redc != nullptr) redc += pass * nreds;
    }
    const BlockTile* tp = tiles + tile;
    if (Const(tp)[8] <= 0) return;  // a hole of the XCD placement
    BlockWork<T, PH, KB>(tp, a, k, pass, redc, reds);
}

// Sum of the slices of one tile in slot order, then the finish (where the
// product launch does not do it).
template <typename T, int PH>
__device__ __forceinline__ void BlockReduceItem(const BlockRed& it, const BlockBufs<T>& a, int k)
{
    for (int e = threadIdx.x; e < it.nob * kBlk * k; e += kThreads) {
        const int rl = e / k, r = e % k;
        cx<T> v = czero<T>();
        for (int j = 0; j < it.nslots; ++j)
            v = v + a.P[((int64_t)(it.slot0 + j) * 64 + rl) * k + r];
        BlockFinish<T, PH>(a, it.x0, it.w0, it.u0, it.s, it.u, it.sb, it.leaf, kBlk * it.ob0 + rl,
                           r, k, v);
    }
}

template <typename T, int PH>
__global__ __launch_bounds__(kThreads) void k_block_reduce(const BlockRed* reds, BlockBufs<T> a,
                                                           int k)
{
    BlockReduceItem<T, PH>(reds[blockIdx.x], a, k);
}

// --------------------------------------------------------------------------
// Fold: the merged fronts' F from the factored fine fronts (L after the
// selective inversion: Linv below the diagonal, D on it, L_BL below; E =
// -L_BL Linv from a batched product).  Pivot rows are scaled by D^-1/2, so that F
// serves both directions without a product by D^-1 between them, whose rounding
// would come on top of theirs.
// --------------------------------------------------------------------------
// Address of (row, column) of a merged front in F.
__device__ __forceinline__ int64_t BlockAt(int browBase, int row, int col)
{
    return (int64_t)(browBase + (col >> 4)) * (kBlk * kBlk) + (col & 15) * kBlk + (row & 15);
}

// A square root of z, by the half-angle formulas (F's scale is used twice, so
// either root will do).
__device__ __forceinline__ c128 csqrt(c128 z)
{
    const double m = sqrt(0.5 * (hypot(z.r, z.i) + fabs(z.r)));
    const double o = m > 0.0 ? 0.5 * fabs(z.i) / m : 0.0;
    return z.r >= 0.0 ? c128{m, z.i < 0.0 ? -o : o} : c128{o, z.i < 0.0 ? -m : m};
}

// Copies a 32 x 32 piece of a node's front: its own lower triangle (row i of the
// unit lower Linv times D_i^-1/2), or rows of E of a group's top node.
// Entries of F outside every piece stay zero from its allocation.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_pack(const TransItem* items, const FoldNode* nodes,
                                                   const int32_t* browBase, const cx<T>* L,
                                                   int64_t fstore, const cx<T>* E, int64_t estride,
                                                   cx<T>* F, int64_t fentries)
{
    const TransItem it = items[blockIdx.x];
    const FoldNode f = nodes[it.node];
    const cx<T>* Lf = L + (int64_t)blockIdx.y * fstore + f.l;
    const cx<T>* Ef = E + (int64_t)blockIdx.y * estride + f.e;
    cx<T>* Fp = F + (int64_t)blockIdx.y * fentries;
    const int fs = f.s + f.u, i = it.i0 + (threadIdx.x & 31);
    const bool own = it.i0 < f.s;
    if (i >= (own ? f.s : fs)) return;
    const int row = own ? f.mcol + i : f.urow + i - f.s;
    const int bb = browBase[f.br0 + (row >> 4)];
    c128 scale{1.0, 0.0};
    if (own) scale = csqrt(cinv(cvt<double>(Lf[i + (int64_t)i * fs])));
    for (int j = it.j0 + (threadIdx.x >> 5); j < min(it.j0 + 32, f.s); j += 8) {
        if (own && i < j) break;
        cx<T> v;
        if (!own)
            v = Ef[i - f.s + (int64_t)j * f.u];
        else if (i == j)
            v = cvt<T>(scale);
        else
            v = cvt<T>(scale * cvt<double>(Lf[i + (int64_t)j * fs]));
        Fp[BlockAt(bb, row, f.mcol + j)] = v;
    }
}

// Columns of a node below its group's top: F_c = F_A P + ext(E_c) (see
// ComposeDesc), one 64 x 64 tile per workgroup through the tile engine.
template <typename T>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 4 : 2) void k_compose(
    const GemmTile* tiles, const ComposeDesc* descs, const int32_t* flist, const int32_t* fsrc,
    const ComposeKey* fkeys, const int32_t* browBase, const cx<T>* E, int64_t estride, cx<T>* F, int64_t fentries)
{
    constexpr int BK = 8, TS = 64;
    __shared__ cx<T> As[2][BK][TS + 1];
    __shared__ cx<T> Bs[2][BK][TS + 1];
    __shared__ int rowOf[TS], baseOf[TS], srcOf[TS];
    const GemmTile tl = tiles[blockIdx.x];
    const ComposeDesc g = descs[tl.desc];
    const cx<T>* Ec = E + (int64_t)blockIdx.y * estride + g.e;
    cx<T>* Fp = F + (int64_t)blockIdx.y * fentries;
    const int tm = tl.tm, tn = tl.tn;
    if (threadIdx.x < TS) {
        const int i = min(tm + (int)threadIdx.x, g.rows - 1);
        const int row = flist[g.list + i];
        rowOf[threadIdx.x] = row;
        baseOf[threadIdx.x] = browBase[g.br0 + (row >> 4)];
        srcOf[threadIdx.x] = fsrc[g.src + i];
    }
    __syncthreads();
    const ComposeKey* keys = fkeys + g.kl;
    // F_A is lower triangular: entries past a pivot row are not stored, and
    // the row's diagonal is read instead, unused
    struct RawA {
        cx<T> v;
        int pos;
    };
    auto la = [&](int i, int k) {
        const ComposeKey key = keys[k];
        const int col = tm + i >= key.pos ? key.col : rowOf[i];
        return RawA{Fp[BlockAt(baseOf[i], rowOf[i], col)], key.pos};
    };
    auto fa = [&](int i, int, const RawA& a) {
        return tm + i < g.rows && tm + i >= a.pos ? a.v : czero<T>();
    };
    auto lb = [&](int k, int j) {
        return Ec[keys[k].row + (int64_t)min(tn + j, g.n - 1) * g.lde];
    };
    auto fb = [&](int, int j, cx<T> v) { return tn + j < g.n ? v : czero<T>(); };
    typename Mfma<T>::acc acc[TileShape<TS, TS>::RB][TileShape<TS, TS>::CB];
    MmaTile<T, TS, false, BK, TS>(la, fa, lb, fb, 0, tl.pad_, As, Bs, acc);
    auto ld = [&](int i, int j) {
        return Ec[max(srcOf[i], 0) + (int64_t)min(tn + j, g.n - 1) * g.lde];
    };
    MmaEpilogue<T, TS, TS>(acc, ld, [&](int i, int j, cx<T> v, cx<T> e) {
        if (tm + i >= g.rows || tn + j >= g.n) return;
        if (tm + i >= g.piv && srcOf[i] >= 0) v = v + e;
        Fp[BlockAt(baseOf[i], rowOf[i], g.ccol + tn + j)] = v;
    });
}

// --------------------------------------------------------------------------
// Batched panel solves: one launch runs the same step (a tree level's
// products or reduce, a panel copy) of the sweeps of many independent
// problems.  Every workgroup reads its BatchBlock: the tile or reduce item it
// works on (tiles of the problems' own lists, unchanged), the segment (one
// problem's panel solve: buffers, factors of that panel, k) and the problem,
// whose flag in `active` is zero once its solve has finished (its
// workgroups then exit at once).  The work of a workgroup is that of the
// single-problem kernels, with the same summation order.
// --------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ BlockBufs<T> SegBufs(const BatchSolveSeg& sg)
{
    return BlockBufs<T>{(const cx<T>*)sg.F, (cx<T>*)sg.V, sg.bsrc, sg.blist, sg.udst,
                        (cx<T>*)sg.P, sg.w, sg.g0, sg.g1, sg.xrows,
                        sg.zero};
}

template <typename T, int PH, int KB>
__global__ __launch_bounds__(256, (BlockOccupancy<T, PH, KB>())) void k_block_batch(const BatchBlock* blocks,
                                                     const BatchSolveSeg* segs,
                                                     const int32_t* active)
{
    const BatchBlock bb = blocks[blockIdx.x];
    const BlockTile* tp = (const BlockTile*)bb.item;
    const BatchSolveSeg sg = segs[bb.seg];
    // (holes of the XCD placement: no tile, or one without output blocks)
    if (!active[bb.problem] || tp == nullptr || Const(tp)[8] <= 0) return;
    int32_t* redc = sg.redc == nullptr ? nullptr : sg.redc + bb.blk * sg.nreds;
    BlockWork<T, PH, KB>(tp, SegBufs<T>(sg), sg.k, bb.blk, redc, sg.reds);
}

template <typename T, int PH>
__global__ __launch_bounds__(kThreads) void k_block_reduce_batch(const BatchBlock* blocks,
                                                                 const BatchSolveSeg* segs,
                                                                 const int32_t* active)
{
    const BatchBlock bb = blocks[blockIdx.x];
    const BatchSolveSeg sg = segs[bb.seg];
    if (!active[bb.problem]) return;
    BlockReduceItem<T, PH>(*(const BlockRed*)bb.item, SegBufs<T>(sg), sg.k);
}

// LT[:, :s] = Linv^T D^-1 per front (upper triangle; D^-1 on the diagonal),
// through a 32x32 LDS tile of L_TL (strictly lower part: Linv; diagonal: D).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_transpose_scale(const TransItem* items,
                                                               const NodeDev* nodes,
                                                               cx<T>* L, cx<T>* LT,
                                                               int64_t fstore)
{
    const TransItem it = items[blockIdx.x];
    const NodeDev nd = nodes[it.node];
    const int s = nd.s, fs = nd.s + nd.u;
    cx<T>* Lf = L + (int64_t)blockIdx.y * fstore + nd.l;
    cx<T>* Lt = LT + (int64_t)blockIdx.y * fstore + nd.l;
    __shared__ cx<T> tile[32][33];
    __shared__ cx<T> dinv[32];
    const int t32 = threadIdx.x & 31, q = threadIdx.x >> 5;
    if (threadIdx.x < 32) {
        const int i = it.i0 + t32;
        dinv[t32] = i < s ? cinv(Lf[i + (int64_t)i * fs]) : czero<T>();
    }
    for (int jj = q; jj < 32; jj += 8) {
        const int i = it.i0 + t32, j = it.j0 + jj;
        if (i < s && j < s) tile[jj][t32] = Lf[i + (int64_t)j * fs];
    }
    __syncthreads();
    // LT's block, with zeros below its diagonal; L's block is read by now,
    // and its part above the diagonal (which no solve uses) becomes zero
    for (int il = q; il < 32; il += 8) {
        const int j = it.j0 + t32, i = it.i0 + il;
        if (i < s && j < s)
            Lt[j + (int64_t)i * s] =
                i > j ? tile[t32][il] * dinv[il] : (i == j ? dinv[il] : czero<T>());
    }
    for (int jj = q; jj < 32; jj += 8) {
        const int i = it.i0 + t32, j = it.j0 + jj;
        if (i < s && j < s && j > i) Lf[i + (int64_t)j * fs] = czero<T>();
    }
}

// L_BL = (LT[:, s:])^T, i.e. -L_BL Linv back in column-major L, and the unit
// diagonal of Linv stored in L (items with i0 == 0 of each column block).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_fold_back(const TransItem* items,
                                                         const NodeDev* nodes, cx<T>* L,
                                                         const cx<T>* LT, int64_t fstore)
{
    const TransItem it = items[blockIdx.x];
    const NodeDev nd = nodes[it.node];
    const int s = nd.s, u = nd.u, fs = nd.s + nd.u;
    cx<T>* Lf = L + (int64_t)blockIdx.y * fstore + nd.l;
    const cx<T>* Lt = LT + (int64_t)blockIdx.y * fstore + nd.l;
    __shared__ cx<T> tile[32][33];
    const int t32 = threadIdx.x & 31, q = threadIdx.x >> 5;
    for (int il = q; il < 32; il += 8) {
        const int i = it.i0 + il, j = it.j0 + t32;  // LT(j, s + i)
        if (i < u && j < s) tile[il][t32] = Lt[j + (int64_t)(s + i) * s];
    }
    __syncthreads();
    for (int jj = q; jj < 32; jj += 8) {
        const int i = it.i0 + t32, j = it.j0 + jj;  // L(s + i, j)
        if (i < u && j < s) Lf[s + i + (int64_t)j * fs] = tile[t32][jj];
    }
    if (it.i0 == 0 && threadIdx.x < 32) {
        const int j = it.j0 + threadIdx.x;
        if (j < s) Lf[j + (int64_t)j * fs] = cx<T>{T(1), T(0)};
    }
}

// --------------------------------------------------------------------------
// Natural-order vector <-> padded panel vector (SolvePanel's copies,
// solve.hpp:756-778 and :825-847).
// --------------------------------------------------------------------------
// Panel copies, element e = (panel row q, right-hand side r) of a panel
// vector; the kernels below run them on one panel (k_copy_in, k_copy_out,
// k_zero_set_plane) or on panels of many problems (k_copy_batch).
template <typename T>
__device__ __forceinline__ void CopyInElem(int64_t e, int n, int k, const int32_t* qxy,
                                           const int32_t* qv, const c128* B, cx<T>* Xp, int nx,
                                           int ny, int nz, int vOffset, int padding)
{
    if (e >= (int64_t)n * k) return;
    const int q = (int)(e / k), r = (int)(e - (int64_t)q * k);
    const int vl = qv[q];
    if (vl < padding) {
        Xp[e] = czero<T>();
        return;
    }
    const int x = qxy[q] & 0xffff, y = qxy[q] >> 16;
    const int z = nz - 1 - (vOffset + vl);
    const int64_t nat = x + (int64_t)y * nx + (int64_t)z * nx * ny;
    Xp[e] = cvt<T>(B[nat * k + r]);
}

template <typename T>
__global__ __launch_bounds__(kThreads) void k_copy_in(int n, int k, const int32_t* qxy,
                                                       const int32_t* qv, const c128* B,
                                                       cx<T>* Xp, int nx, int ny, int nz,
                                                       int vOffset, int padding,
                                                       int32_t* sync, int nsync)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    // the fused-launch state of the panel solve that follows starts at zero
    for (int64_t j = e; j < nsync; j += (int64_t)gridDim.x * blockDim.x) sync[j] = 0;
    CopyInElem<T>(e, n, k, qxy, qv, B, Xp, nx, ny, nz, vOffset, padding);
}

template <typename T>
__device__ __forceinline__ void CopyOutElem(int64_t e, int n, int k, const int32_t* qxy,
                                            const int32_t* qv, c128* B, const cx<T>* Xp, int nx,
                                            int ny, int nz, int vOffset, int padding, int mode,
                                            const StencilArgs& st, const double* vel, int v1);

template <typename T>
__global__ __launch_bounds__(kThreads) void k_copy_out(int n, int k, const int32_t* qxy,
                                                        const int32_t* qv, c128* B,
                                                        const cx<T>* Xp, int nx, int ny, int nz,
                                                        int vOffset, int padding, int mode,
                                                        StencilArgs st, const double* vel, int v1)
{
    CopyOutElem<T>((int64_t)blockIdx.x * blockDim.x + threadIdx.x, n, k, qxy, qv, B, Xp, nx, ny,
                   nz, vOffset, padding, mode, st, vel, v1);
}

template <typename T>
__device__ __forceinline__ void CopyOutElem(int64_t e, int n, int k, const int32_t* qxy,
                                            const int32_t* qv, c128* B, const cx<T>* Xp, int nx,
                                            int ny, int nz, int vOffset, int padding, int mode,
                                            const StencilArgs& st, const double* vel, int v1)
{
    if (e >= (int64_t)n * k) return;
    const int q = (int)(e / k), r = (int)(e - (int64_t)q * k);
    const int vl = qv[q];
    if (vl < padding) return;
    const int x = qxy[q] & 0xffff, y = qxy[q] >> 16;
    const int z = nz - 1 - (vOffset + vl);
    const int64_t nat = x + (int64_t)y * nx + (int64_t)z * nx * ny;
    const c128 v = cvt<double>(Xp[e]);
    if (mode == 0)
        B[nat * k + r] = v;
    else
        B[nat * k + r] = B[nat * k + r] + v;
    // forward sweep: the subdiagonal coupling into the next panel's first
    // plane v1 (k_subdiag's update), applied by the thread that wrote the
    // value it reads: row (x,y,v1) couples to (x,y,v1-1) with value c[5]
    if (v1 >= 0 && vOffset + vl == v1 - 1) {
        const int64_t natN = nat - (int64_t)nx * ny;
        c128 c[7];
        GlobalRowFast(st, vel[natN], x, y, v1, c);
        B[natN * k + r] = B[natN * k + r] - c[5] * v;
    }
}

// --------------------------------------------------------------------------
// Sweep couplings between consecutive panels (solve.hpp:884-1047).
// --------------------------------------------------------------------------
// Backward sweep (ExtractPanel + MultiplySuperdiagonal): the panel vector is
// zero except on its last local plane vlLast (global plane v2), which holds
// -A(v2, v2+1) B(plane v2+1), i.e. row (x,y,v2) times its coupling c[6] to
// (x,y,v2+1) = natural z-1; one pass over the panel vector.  The forward
// sweep's subdiagonal coupling is applied by k_copy_out.
template <typename T>
__device__ __forceinline__ void ZeroSetPlaneElem(int64_t e, int n, int k, const int32_t* qxy,
                                                 const int32_t* qv, const StencilArgs& st,
                                                 const double* vel, const c128* B, cx<T>* Xp,
                                                 int v2, int vlLast);

template <typename T>
__global__ __launch_bounds__(kThreads) void k_zero_set_plane(int n, int k, const int32_t* qxy,
                                                              const int32_t* qv, StencilArgs st,
                                                              const double* vel, const c128* B,
                                                              cx<T>* Xp, int v2, int vlLast,
                                                              int32_t* sync, int nsync)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (int64_t j = e; j < nsync; j += (int64_t)gridDim.x * blockDim.x) sync[j] = 0;
    ZeroSetPlaneElem<T>(e, n, k, qxy, qv, st, vel, B, Xp, v2, vlLast);
}

// A panel's copy out, with its coupling, and the next panel's copy in as one
// launch: both are small (5 us each, mostly latency, and a sweep of P panels had
// 4 P - 2 of them; now 2 P), and a value that couples stays in a register.  A
// thread owns a column (x, y, r) of both panels, so it has read every row of the
// old vector that it writes in the new one.  The arithmetic is CopyOutElem's,
// CopyInElem's and ZeroSetPlaneElem's.  Bound by its chain of loads (6 us at 24 x
// 20, k = 3), so the first U planes of both panels are loaded together.  ms a
// sweep, before and after: 100^3 k = 8 FP32 8.87 -> 8.68, k = 16 11.26 -> 10.9,
// k = 64 28.4 -> 27.6; 120 x 96 x 60 k = 32 FP32 11.4 -> 11.15; 24 x 20 x 26 and
// 40^3 as before.
template <typename T, int U>
__global__ __launch_bounds__(kThreads) void k_pass_on(StencilArgs st, const double* vel, c128* B,
                                                       int k, PassPanel o, PassPanel i, int mode,
                                                       int dir)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t plane = (int64_t)st.nx * st.ny;
    if (e >= plane * k) return;
    const int xy = (int)(e / k), r = (int)(e - (int64_t)xy * k);
    const int y = xy / st.nx, x = xy - y * st.nx;
    // grid point of (x, y) on plane vl of a panel
    auto at = [&](const PassPanel& p, int vl) {
        return xy + plane * (st.nz - 1 - (p.vOffset + vl));
    };
    const cx<T>* Xo = (const cx<T>*)o.X;
    cx<T>* Xi = (cx<T>*)i.X;
    const int edgeIn = dir == 0 ? 0 : i.depth - 1;
    const double velIn = vel[at(i, i.padding + edgeIn)];
    int32_t ro[U], ri[U];
    cx<T> v[U];
    c128 bo[U], bi[U];
    auto rows = [&](const PassPanel& p, int j0, int32_t (&row)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            row[u] = p.row[(p.padding + min(j0 + u, p.depth - 1)) * plane + xy];
    };
    auto outs = [&](int j0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            v[u] = Xo[(int64_t)ro[u] * k + r];
            if (mode != 0) bo[u] = B[at(o, o.padding + min(j0 + u, o.depth - 1)) * k + r];
        }
    };
    auto ins = [&](int j0) {
        if (dir == 0) {
#pragma unroll
            for (int u = 0; u < U; ++u)
                bi[u] = B[at(i, i.padding + min(j0 + u, i.depth - 1)) * k + r];
        }
    };
    rows(o, 0, ro);
    rows(i, 0, ri);
    ins(0);
    outs(0);
    const int edgeOut = dir == 0 ? o.depth - 1 : 0;  // the plane that couples
    c128 ev{0.0, 0.0};
    for (int j0 = 0;;) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (j0 + u >= o.depth) break;
            const c128 w = cvt<double>(v[u]);
            const c128 out = mode == 0 ? w : bo[u] + w;
            B[at(o, o.padding + j0 + u) * k + r] = out;
            if (j0 + u == edgeOut) ev = out;
        }
        if ((j0 += U) >= o.depth) break;
        rows(o, j0, ro);
        outs(j0);
    }
    for (int vl = 0; vl < i.padding; ++vl)
        Xi[(int64_t)i.row[vl * plane + xy] * k + r] = czero<T>();
    // row (x, y, v) couples to the plane below with c[5], above with c[6]
    c128 c[7];
    GlobalRowFast(st, velIn, x, y, i.vOffset + i.padding + edgeIn, c);
    for (int j0 = 0;;) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = j0 + u;
            if (j >= i.depth) break;
            c128 in = dir == 0 ? bi[u] : c128{0.0, 0.0};
            if (j == edgeIn) in = dir == 0 ? in - c[5] * ev : -(c[6] * ev);
            Xi[(int64_t)ri[u] * k + r] = cvt<T>(in);
        }
        if ((j0 += U) >= i.depth) break;
        rows(i, j0, ri);
        ins(j0);
    }
}

// One batched panel copy: op BATCH_COPY_IN, BATCH_COPY_OUT (mode and
// coupling plane v1 per segment) or BATCH_ZERO_SET_PLANE, with the segment's
// elements split into whole workgroups (BatchBlock.item unused, blk: the
// workgroup's index inside its segment).
template <typename T>
__global__ __launch_bounds__(kBatchCopyThreads) void k_copy_batch(int op, const BatchBlock* blocks,
                                                                  const BatchCopySeg* segs,
                                                                  const int32_t* active)
{
    const BatchBlock bb = blocks[blockIdx.x];
    const BatchCopySeg sg = segs[bb.seg];
    if (!active[bb.problem]) return;
    const int64_t e = (int64_t)bb.blk * kBatchCopyThreads + threadIdx.x;
    if (op == BATCH_COPY_IN)
        CopyInElem<T>(e, sg.n, sg.k, sg.qxy, sg.qv, sg.B, (cx<T>*)sg.Xp, sg.st.nx, sg.st.ny,
                      sg.st.nz, sg.vOffset, sg.padding);
    else if (op == BATCH_COPY_OUT)
        CopyOutElem<T>(e, sg.n, sg.k, sg.qxy, sg.qv, sg.B, (const cx<T>*)sg.Xp, sg.st.nx,
                       sg.st.ny, sg.st.nz, sg.vOffset, sg.padding, sg.mode, sg.st, sg.vel, sg.v1);
    else
        ZeroSetPlaneElem<T>(e, sg.n, sg.k, sg.qxy, sg.qv, sg.st, sg.vel, sg.B, (cx<T>*)sg.Xp,
                            sg.v2, sg.vlLast);
}

template <typename T>
__device__ __forceinline__ void ZeroSetPlaneElem(int64_t e, int n, int k, const int32_t* qxy,
                                                 const int32_t* qv, const StencilArgs& st,
                                                 const double* vel, const c128* B, cx<T>* Xp,
                                                 int v2, int vlLast)
{
    if (e >= (int64_t)n * k) return;
    const int q = (int)(e / k), r = (int)(e - (int64_t)q * k);
    cx<T> out = czero<T>();
    if (qv[q] == vlLast) {
        const int x = qxy[q] & 0xffff, y = qxy[q] >> 16;
        const int64_t plane = (int64_t)st.nx * st.ny;
        const int64_t nat = x + (int64_t)y * st.nx + (int64_t)(st.nz - 1 - v2) * plane;
        c128 c[7];
        GlobalRowFast(st, vel[nat], x, y, v2, c);
        out = cvt<T>(-(c[6] * B[(nat - plane) * k + r]));
    }
    Xp[e] = out;
}

// --------------------------------------------------------------------------
// Multiply (solve.hpp:613-679) in natural order: y = A x or y = b - A x.
// --------------------------------------------------------------------------
// Bound by memory: a block is read and written once if its neighbours in y and
// z are found in L2.  Workgroups in the order of memory go to the 8 XCDs in turn,
// so each XCD's L2 fetched the lines of its neighbours too.  Order of the work
// here: strips of `rows` lines of y, in each all planes z, so that a plane of a
// strip, read as z + 1, is still in L2 as z and z - 1; workgroup b takes place
// b / 8 in the part b % 8 of that order, so an XCD has its own part.
// kStripBytes: 128 KiB, 256 KiB and no strips were up to 7, 4 and 13% slower.  us
// a call on blocks that no cache holds, before and after: 100^3 k = 8 137 -> 129,
// k = 64 915 -> 745; 144 x 128 x 80 k = 16 355 -> 308; 120 x 96 x 60 k = 32
// 336 -> 276; 61 x 47 x 83 k = 5 38.6 -> 36.5.  Now the L1s' loads bound it (seven
// of 16 bytes for each 32 moved).
struct SpmvOrder {
    int rows, strips, per;   // lines per strip, strips, workgroups per strip plane
    int64_t part;            // workgroups per part
};
constexpr int kStripBytes = 512 << 10;
constexpr unsigned kSpmvGrid = 1u << 22;  // most workgroups of a launch (more: several turns)

// V: right-hand sides of a point per thread (V divides k), which share its
// stencil row (four needed more registers: 15% slower than two).
// LOOP: more workgroups than a launch takes.
template <int V, bool LOOP>
__global__ __launch_bounds__(kThreads) void k_spmv(StencilArgs st, const double* vel,
                                                    const c128* X, const c128* Bv, c128* Y, int k,
                                                    int mode, SpmvOrder o)
{
    for (int64_t i = blockIdx.x >> 3; LOOP ? i < o.part : true; i += gridDim.x >> 3) {
        const int64_t g = (int64_t)(blockIdx.x & 7) * o.part + i;
        const int64_t sp = g / o.per;
        const int strip = (int)(sp / st.nz), z = (int)(sp - (int64_t)strip * st.nz);
        if (strip >= o.strips) return;
        const int y0 = strip * o.rows, rows = min(o.rows, st.ny - y0);
        const uint32_t nx = st.nx, kk = k / V;
        const uint32_t t = (uint32_t)(g - sp * o.per) * kThreads + threadIdx.x;
        if (t >= rows * nx * kk) {
            if (LOOP) continue;
            return;
        }
        const uint32_t q = t / kk, r = (t - q * kk) * V, yl = q / nx;
        const int x = (int)(q - yl * nx), y = y0 + (int)yl, v = st.nz - 1 - z;
        const int64_t p = ((int64_t)z * st.ny + y0) * nx + q;
        const int64_t line = (int64_t)st.nx * k, plane = line * st.ny;
        const c128* Xe = X + p * k + r;
        c128 c[7];
        GlobalRowFast(st, vel[p], x, y, v, c);
        c128 acc[V];
        auto term = [&](bool on, int64_t d, int j) {
            if (on) {
#pragma unroll
                for (int n = 0; n < V; ++n) acc[n] = cfma(c[j], Xe[d + n], acc[n]);
            }
        };
#pragma unroll
        for (int n = 0; n < V; ++n) acc[n] = Xe[n] * c[0];
        term(x > 0, -k, 1);
        term(x + 1 < st.nx, k, 2);
        term(y > 0, -line, 3);
        term(y + 1 < st.ny, line, 4);
        term(v > 0, plane, 5);
        term(v + 1 < st.nz, -plane, 6);
#pragma unroll
        for (int n = 0; n < V; ++n) {
            const int64_t e = p * k + r + n;
            Y[e] = mode == 0 ? acc[n] : (Bv[e] - acc[n]);
        }
        if (!LOOP) return;
    }
}

// dL/dm_i = sum_s Re(omega^2 s1 s2 s3 lambda_s(i) u_s(i)).
__global__ __launch_bounds__(kThreads) void k_adjoint_grad(StencilArgs st, const c128* U,
                                                            const c128* Lam, int k, double* grad,
                                                            int accumulate)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t plane = (int64_t)st.nx * st.ny;
    if (p >= plane * st.nz) return;
    const int x = (int)(p % st.nx);
    const int y = (int)((p / st.nx) % st.ny);
    const int z = (int)(p / plane);
    const int v = st.nz - 1 - z;
    const c128 s = st.s1[x + 1] * st.s2[y + 1] * st.s3[v + 1];
    double g = 0.0;
    for (int r = 0; r < k; ++r) {
        const c128 t = Lam[p * k + r] * U[p * k + r];
        const c128 w = s * t;
        g += w.r;
    }
    g *= st.omega * st.omega;
    grad[p] = accumulate ? grad[p] + g : g;
}

// --------------------------------------------------------------------------
// Column reductions (Norms / InnerProducts, environment.hpp:177-211).
// Each workgroup reduces a contiguous point range; thread t < lanes owns
// column t % k; partials are summed in a fixed order (deterministic).
// --------------------------------------------------------------------------
constexpr int kReduceBlocks = 512;

__global__ __launch_bounds__(kThreads) void k_colnorm_part(const c128* X, int64_t np, int k,
                                                            double* part)
{
    __shared__ double sh[kThreads];
    const int lanes = (kThreads / k) * k, per = kThreads / k;
    const int t = threadIdx.x;
    const int64_t chunk = (np + gridDim.x - 1) / gridDim.x;
    const int64_t p0 = (int64_t)blockIdx.x * chunk, p1 = min(np, p0 + chunk);
    double acc = 0.0;
    if (t < lanes) {
        const int r = t % k;
        for (int64_t p = p0 + t / k; p < p1; p += per) {
            const c128 v = X[p * k + r];
            acc = fma(v.r, v.r, acc);
            acc = fma(v.i, v.i, acc);
        }
    }
    sh[t] = acc;
    __syncthreads();
    if (t < k) {
        double s = 0.0;
        for (int i = 0; i < per; ++i) s += sh[t + i * k];
        part[(int64_t)blockIdx.x * k + t] = s;
    }
}

// One workgroup per column: fixed-order tree sum of the block partials.
__global__ __launch_bounds__(kThreads) void k_colnorm_final(const double* part, int nblk, int k,
                                                             double* out)
{
    __shared__ double sh[kThreads];
    const int r = blockIdx.x;
    double s = 0.0;
    for (int b = threadIdx.x; b < nblk; b += kThreads) s += part[(int64_t)b * k + r];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int o = kThreads / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[r] = sqrt(sh[0]);
}

__global__ __launch_bounds__(kThreads) void k_coldot_part(const c128* __restrict__ V,
                                                           const c128* __restrict__ W,
                                                           int64_t np, int k,
                                                           c128* __restrict__ part)
{
    __shared__ c128 sh[kThreads];
    const int lanes = (kThreads / k) * k, per = kThreads / k;
    const int t = threadIdx.x;
    const int64_t chunk = (np + gridDim.x - 1) / gridDim.x;
    const int64_t p0 = (int64_t)blockIdx.x * chunk, p1 = min(np, p0 + chunk);
    c128 acc = {0.0, 0.0};
    if (t < lanes) {
        const int r = t % k;
#pragma unroll 4
        for (int64_t p = p0 + t / k; p < p1; p += per) {
            const c128 v = V[p * k + r], w = W[p * k + r];
            // conj(v) * w
            acc.r = fma(v.r, w.r, acc.r);
            acc.r = fma(v.i, w.i, acc.r);
            acc.i = fma(v.r, w.i, acc.i);
            acc.i = fma(-v.i, w.r, acc.i);
        }
    }
    sh[t] = acc;
    __syncthreads();
    if (t < k) {
        c128 s = {0.0, 0.0};
        for (int i = 0; i < per; ++i) s = s + sh[t + i * k];
        part[(int64_t)blockIdx.x * k + t] = s;
    }
}

// Modified Gram-Schmidt, two steps in one pass: W -= alpha V (step i's
// update) and the partial sums of conj(Vn) W for step i + 1, with the
// block partition and summation order of k_coldot_part.
__global__ __launch_bounds__(kThreads) void k_axpy_dot_part(const c128* __restrict__ alpha,
                                                             const c128* __restrict__ V,
                                                             const c128* __restrict__ Vn,
                                                             c128* __restrict__ W, int64_t np,
                                                             int k, c128* __restrict__ part)
{
    __shared__ c128 sh[kThreads];
    const int lanes = (kThreads / k) * k, per = kThreads / k;
    const int t = threadIdx.x;
    const int64_t chunk = (np + gridDim.x - 1) / gridDim.x;
    const int64_t p0 = (int64_t)blockIdx.x * chunk, p1 = min(np, p0 + chunk);
    c128 acc = {0.0, 0.0};
    if (t < lanes) {
        const int r = t % k;
        const c128 a = alpha[r];
        // unrolled so a thread has several elements' loads in flight (the
        // sums still run in element order)
#pragma unroll 4
        for (int64_t p = p0 + t / k; p < p1; p += per) {
            const int64_t e = p * k + r;
            const c128 w = cfms(a, V[e], W[e]), v = Vn[e];
            W[e] = w;
            acc.r = fma(v.r, w.r, acc.r);
            acc.r = fma(v.i, w.i, acc.r);
            acc.i = fma(v.r, w.i, acc.i);
            acc.i = fma(-v.i, w.r, acc.i);
        }
    }
    sh[t] = acc;
    __syncthreads();
    if (t < k) {
        c128 s = {0.0, 0.0};
        for (int i = 0; i < per; ++i) s = s + sh[t + i * k];
        part[(int64_t)blockIdx.x * k + t] = s;
    }
}

__global__ __launch_bounds__(kThreads) void k_coldot_final(const c128* part, int nblk, int k,
                                                            c128* out)
{
    __shared__ c128 sh[kThreads];
    const int r = blockIdx.x;
    c128 s = {0.0, 0.0};
    for (int b = threadIdx.x; b < nblk; b += kThreads) s = s + part[(int64_t)b * k + r];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int o = kThreads / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[r] = sh[0];
}

// Modified Gram-Schmidt with two passes over the basis.  Step by step it is
// h_a = v_a^H (w - sum_{b<a} h_b v_b) = d_a - sum_{b<a} (v_a^H v_b) h_b, so all
// d_a = v_a^H w and the Gram row v_a^H v_j of the newest vector come from one
// pass (k_arnoldi_dots), h from a triangular solve with the Gram rows of the
// cycle (k_arnoldi_solve), and w - V h with its norm from a second pass
// (k_arnoldi_update): 2.25 j vectors moved instead of 4 j, 4 launches instead of
// 2 j + 4.  The rounding error is that of the steps one by one.  Bound by memory
// for wide blocks.  ms a solve, before and after: 120 x 96 x 60 k = 32 501 -> 465,
// 44 x 36 x 48 k = 16 with its adjoint 141 -> 137, 61 x 47 x 83 k = 5 57.4 -> 56.8,
// 40^3 k = 1 19.9 -> 19.5.  Cycles past 64 (the solve is one wave) go step by step.
constexpr int kDotGroup = 8;  // basis vectors per workgroup (16 sums in registers)

// Block partials of group blockIdx.y: part[(q grid.x + block) k + r], q = i for
// v_i^H w and j + 1 + i for v_i^H v_j.
__global__ __launch_bounds__(kThreads) void k_arnoldi_dots(const c128* __restrict__ V, int64_t n,
                                                            int j, const c128* __restrict__ W,
                                                            int64_t np, int k,
                                                            c128* __restrict__ part)
{
    __shared__ c128 sh[kThreads];
    const int lanes = (kThreads / k) * k, per = kThreads / k;
    const int t = threadIdx.x, i0 = blockIdx.y * kDotGroup, cnt = min(kDotGroup, j + 1 - i0);
    const int64_t chunk = (np + gridDim.x - 1) / gridDim.x;
    const int64_t p0 = (int64_t)blockIdx.x * chunk, p1 = min(np, p0 + chunk);
    const c128 *Vi = V + i0 * n, *Vj = V + j * n;
    c128 acc[2 * kDotGroup];
#pragma unroll
    for (int u = 0; u < 2 * kDotGroup; ++u) acc[u] = c128{0.0, 0.0};
    auto add = [](c128& s, const c128& v, const c128& w) {  // s += conj(v) w
        s.r = fma(v.r, w.r, s.r);
        s.r = fma(v.i, w.i, s.r);
        s.i = fma(v.r, w.i, s.i);
        s.i = fma(-v.i, w.r, s.i);
    };
    if (t < lanes) {
        const int r = t % k;
        for (int64_t p = p0 + t / k; p < p1; p += per) {
            const int64_t e = p * k + r;
            const c128 w = W[e], vj = Vj[e];
            c128 v[kDotGroup];
#pragma unroll
            for (int u = 0; u < kDotGroup; ++u)
                if (u < cnt) v[u] = Vi[u * n + e];
#pragma unroll
            for (int u = 0; u < kDotGroup; ++u)
                if (u < cnt) {
                    add(acc[2 * u], v[u], w);
                    add(acc[2 * u + 1], v[u], vj);
                }
        }
    }
#pragma unroll
    for (int u = 0; u < 2 * kDotGroup; ++u) {
        if (u / 2 >= cnt) break;
        sh[t] = acc[u];
        __syncthreads();
        if (t < k) {
            c128 s = {0.0, 0.0};
            for (int q = 0; q < per; ++q) s = s + sh[t + q * k];
            const int64_t q = (u & 1) * (j + 1) + i0 + u / 2;
            part[(q * gridDim.x + blockIdx.x) * k + t] = s;
        }
        __syncthreads();
    }
}

// Column r = blockIdx.x: sums the partials (a wave per sum, in a fixed order),
// stores the Gram row j, gram[(j m + i) k + r] = v_j^H v_i, and solves for h.
constexpr int kSolveThreads = 512, kMaxGram = 64;  // the longest cycle this form takes
__global__ __launch_bounds__(kSolveThreads) void k_arnoldi_solve(const c128* part, int nblk, int j,
                                                                  int m, int k, c128* gram, c128* h)
{
    __shared__ c128 d[kMaxGram], row[kMaxGram];
    const int r = blockIdx.x, lane = threadIdx.x & 63;
    for (int q = threadIdx.x >> 6; q < 2 * (j + 1); q += kSolveThreads / 64) {
        c128 s = {0.0, 0.0};
        for (int b = lane; b < nblk; b += 64) s = s + part[((int64_t)q * nblk + b) * k + r];
        for (int o = 32; o > 0; o >>= 1) {
            s.r += __shfl_xor(s.r, o, 64);
            s.i += __shfl_xor(s.i, o, 64);
        }
        if (lane == 0) {
            if (q <= j)
                d[q] = s;
            else
                row[q - j - 1] = c128{s.r, -s.i};  // v_j^H v_i
        }
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    // one wave: lane a holds row a (j < kMaxGram = 64)
    if (lane < j) gram[((int64_t)j * m + lane) * k + r] = row[lane];
    c128 da = lane <= j ? d[lane] : c128{0.0, 0.0};
    for (int b = 0; b < j; ++b) {
        const c128 hb{__shfl(da.r, b, 64), __shfl(da.i, b, 64)};
        if (lane > b && lane <= j) {
            const c128 g = lane == j ? row[b] : gram[((int64_t)lane * m + b) * k + r];
            da = cfms(g, hb, da);
        }
    }
    if (lane <= j) h[lane * k + r] = da;
}

// W -= V h, and the partial sums of its norms (k_colnorm_part's partition).
__global__ __launch_bounds__(kThreads) void k_arnoldi_update(const c128* __restrict__ V, int64_t n,
                                                              int j, const c128* __restrict__ h,
                                                              c128* __restrict__ W, int64_t np,
                                                              int k, double* __restrict__ part)
{
    __shared__ double sh[kThreads];
    const int lanes = (kThreads / k) * k, per = kThreads / k;
    const int t = threadIdx.x;
    const int64_t chunk = (np + gridDim.x - 1) / gridDim.x;
    const int64_t p0 = (int64_t)blockIdx.x * chunk, p1 = min(np, p0 + chunk);
    double acc = 0.0;
    if (t < lanes) {
        const int r = t % k;
        for (int64_t p = p0 + t / k; p < p1; p += per) {
            const int64_t e = p * k + r;
            c128 w = W[e];
            int i = 0;
            for (; i + 4 <= j + 1; i += 4) {
                c128 v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = V[(i + u) * n + e];
#pragma unroll
                for (int u = 0; u < 4; ++u) w = cfms(h[(i + u) * k + r], v[u], w);
            }
            for (; i <= j; ++i) w = cfms(h[i * k + r], V[i * n + e], w);
            W[e] = w;
            acc = fma(w.r, w.r, acc);
            acc = fma(w.i, w.i, acc);
        }
    }
    sh[t] = acc;
    __syncthreads();
    if (t < k) {
        double s = 0.0;
        for (int i = 0; i < per; ++i) s += sh[t + i * k];
        part[(int64_t)blockIdx.x * k + t] = s;
    }
}

__global__ __launch_bounds__(kThreads) void k_axpy_cols(const c128* alpha, int sign,
                                                         const c128* V, c128* W, int64_t n, int k)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const int r = (int)(e % k);
    const c128 a = alpha[r];
    W[e] = sign > 0 ? cfma(a, V[e], W[e]) : cfms(a, V[e], W[e]);
}

__global__ __launch_bounds__(kThreads) void k_scale_cols(const double* delta, const c128* W,
                                                          c128* V, int64_t n, int k)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const int r = (int)(e % k);
    const double inv = 1.0 / delta[r];
    V[e] = W[e] * inv;
}

__global__ __launch_bounds__(kThreads) void k_update_x(const c128* X0, const c128* V,
                                                        const c128* Y, int j, int64_t n, int k,
                                                        int64_t vstride, c128* X)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const int r = (int)(e % k);
    c128 acc = X0[e];
    for (int i = 0; i <= j; ++i) acc = cfma(Y[i * k + r], V[i * vstride + e], acc);
    X[e] = acc;
}

__global__ __launch_bounds__(kThreads) void k_neg(const c128* X, c128* W, int64_t n)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n) W[e] = -X[e];
}

inline unsigned Blocks(int64_t n) { return (unsigned)((n + kThreads - 1) / kThreads); }

}  // namespace

// ==========================================================================
// Launch wrappers
// ==========================================================================
bool XcdRoundRobin(hipStream_t s)
{
    constexpr int kBlocks = 64;
    int32_t* d = nullptr;
    if (hipMalloc(&d, sizeof(int32_t) * kBlocks) != hipSuccess) return false;
    int32_t h[kBlocks] = {};
    bool ok = hipMemsetAsync(d, 0xff, sizeof(h), s) == hipSuccess;
    if (ok) {
        hipLaunchKernelGGL(k_xcc_probe, dim3(kBlocks), dim3(64), 0, s, d);
        ok = hipGetLastError() == hipSuccess &&
             hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, s) == hipSuccess &&
             hipStreamSynchronize(s) == hipSuccess;
    }
    (void)hipFree(d);
    for (int b = 0; ok && b < kBlocks; ++b) ok = h[b] == b % 8;
    return ok;
}

void LaunchFillZeroRows(void* p, int64_t bytes, int rows, int64_t strideBytes, hipStream_t s)
{
    if (bytes <= 0 || rows <= 0) return;
    const int64_t n8 = bytes / 8;
    const unsigned g = (unsigned)std::min<int64_t>(Blocks(n8), 4096);
    hipLaunchKernelGGL(k_fill_zero_rows, dim3(g, rows), dim3(kThreads), 0, s, (uint2*)p, n8,
                       strideBytes / 8);
}

void LaunchFillZero(void* p, int64_t bytes, hipStream_t s)
{
    if (bytes <= 0) return;
    const int64_t n16 = bytes / 16;
    if (n16 > 0) {
        const unsigned g = (unsigned)std::min<int64_t>(Blocks(n16), 65535 * 4);
        hipLaunchKernelGGL(k_fill_zero, dim3(g), dim3(kThreads), 0, s, (uint4*)p, n16);
    }
    const int64_t rem = bytes - n16 * 16;
    if (rem > 0)
        hipLaunchKernelGGL(k_fill_zero_bytes, dim3(1), dim3(kThreads), 0, s,
                           (unsigned char*)p + n16 * 16, rem);
}

template <typename T>
void LaunchScatterOrig(const ClassDev& c, const StencilArgs& st, const double* vel,
                       double damping, hipStream_t s)
{
    hipLaunchKernelGGL((k_scatter_orig<T>), dim3(Blocks(c.n), c.npanels), dim3(kThreads), 0, s,
                       c.n, c.vsize, c.qxy, c.qv, c.qnode, c.qcol, c.qrows, c.nodeL, c.nodeS,
                       c.nodeU, c.panelVOff, c.s3art, st, vel, damping, (cx<T>*)c.L, c.fstore);
}

template <typename T>
void LaunchExtendAdd(const ClassDev& c, int start, int count, hipStream_t s)
{
    if (count <= 0) return;
    hipLaunchKernelGGL((k_extend_add<T>), dim3(count, c.npanels), dim3(kThreads), 0, s,
                       c.extadd, start, c.relinds, (cx<T>*)c.L, c.fstore, (cx<T>*)c.U, c.ustore);
}

template <typename T>
void LaunchLdlDiag(const ClassDev& c, int start, int count, int nb, hipStream_t s)
{
    if (count <= 0) return;
    (void)nb;
    hipLaunchKernelGGL((k_ldl_diag<T, 32>), dim3(count, c.npanels), dim3(kThreads), 0, s, c.ldl,
                       start, (cx<T>*)c.L, c.fstore);
}

template <typename T>
void LaunchLdlTrsm(const ClassDev& c, int start, int count, int nb, hipStream_t s)
{
    if (count <= 0) return;
    (void)nb;
    hipLaunchKernelGGL((k_ldl_trsm<T, 32>), dim3(count, c.npanels), dim3(kThreads), 0, s, c.ldl,
                       start, (cx<T>*)c.L, c.fstore);
}

template <typename T>
void LaunchGemm(const ClassDev& c, int tileStart, int tileCount, hipStream_t s)
{
    if (tileCount <= 0) return;
    hipLaunchKernelGGL((k_gemm_mma<T>), dim3(tileCount, c.npanels), dim3(256), 0, s, c.gemms,
                       c.tiles, tileStart, (cx<T>*)c.L, c.fstore, (cx<T>*)c.U, c.ustore,
                       (cx<T>*)c.T, c.tstore, (cx<T>*)c.LT);
}

template <typename T>
void LaunchInvDiag(const ClassDev& c, int nb, hipStream_t s)
{
    if (c.ninv <= 0) return;
    (void)nb;
    hipLaunchKernelGGL((k_inv_diag<T, 32>), dim3(c.ninv, c.npanels), dim3(kThreads), 0, s, c.inv,
                       (cx<T>*)c.L, c.fstore);
}

// Workgroups of a fused launch: as many as fit on the device at once.
template <typename T, int PH, int RT, int KB>
int MvqGrid(int cus)
{
    static const int perCU = [] {
        int b = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k_mvq<T, PH, RT, KB>, 256, 0) !=
                hipSuccess ||
            b < 1)
            b = 1;
        return b;
    }();
    return perCU * std::max(cus, 1);
}

void PrimeSolveOccupancy()
{
    auto prime = [](auto t) {
        typedef decltype(t) T;
        (void)MvqGrid<T, PH_F, 64, 8>(1), (void)MvqGrid<T, PH_F, 32, 8>(1);
        (void)MvqGrid<T, PH_F, 16, 8>(1), (void)MvqGrid<T, PH_F, 64, 16>(1);
        (void)MvqGrid<T, PH_F, 32, 16>(1), (void)MvqGrid<T, PH_F, 16, 16>(1);
        (void)MvqGrid<T, PH_B, 64, 8>(1), (void)MvqGrid<T, PH_B, 32, 8>(1);
        (void)MvqGrid<T, PH_B, 16, 8>(1), (void)MvqGrid<T, PH_B, 64, 16>(1);
        (void)MvqGrid<T, PH_B, 32, 16>(1), (void)MvqGrid<T, PH_B, 16, 16>(1);
    };
    prime(float());
    prime(double());
}

// Start and end of a timed product launch, and its algorithmic work.
static void ProfBegin(MvProfile* prof, hipStream_t s)
{
    if (prof) (void)hipEventRecord(prof->a, s);
}

static void ProfEnd(MvProfile* prof, hipStream_t s, double bytes, double flops)
{
    if (!prof) return;
    (void)hipEventRecord(prof->b, s);
    (void)hipEventSynchronize(prof->b);
    float ms = 0;
    (void)hipEventElapsedTime(&ms, prof->a, prof->b);
    prof->launches += 1;
    prof->seconds += ms * 1e-3;
    prof->bytes += bytes;
    prof->flops += flops;
}

int32_t* SliceCounters(const ClassDev& c, const ClassPlan& plan, int k, int entryBytes)
{
    // the partial sums are read through a buffer of at most 4 GiB, and each
    // pass needs counters of its own
    const bool fits = (int64_t)entryBytes * k * 64 * plan.bslots < ((int64_t)1 << 32) &&
                      k <= kPassRhs * kMaxPasses;
    return fits ? c.bredc : nullptr;
}

template <typename T>
void LaunchPanelSolve(const ClassDev& c, const ClassPlan& plan, int b, void* V, void* P, int k,
                      hipStream_t s, MvProfile* prof, int onlyGroup, int onlyPhase)
{
    const VecRows vr(plan);
    const BlockBufs<T> bufs{(const cx<T>*)c.F + (int64_t)b * c.fentries,
                            (cx<T>*)V,
                            c.bsrc,
                            c.blist,
                            c.udst,
                            (cx<T>*)P,
                            vr.w,
                            vr.g0,
                            vr.g1,
                            c.xrows,
                            plan.nblocks};
    int32_t* rc = SliceCounters(c, plan, k, sizeof(cx<T>));
    auto go = [&](auto ph, int g) {
        constexpr int PH = decltype(ph)::value;
        const ClassPlan::BlockLevel& L = plan.blevels[g];
        if (L.count[PH] <= 0) return;
        auto run = [&](auto kb) {
            constexpr int KB = decltype(kb)::value;
            const int passes = KB <= 16 ? 1 : (k + KB - 1) / KB;
            const int grid = KB <= 16 ? L.count[PH] : (L.count[PH] + 7) / 8 * 8 * passes;
            hipLaunchKernelGGL((k_block<T, PH, KB>), dim3(grid), dim3(256), 0, s,
                               c.btiles + L.start[PH], bufs, k, L.count[PH], passes, rc, c.nbreds,
                               c.breds);
        };
        ProfBegin(prof, s);
        if (k <= 8)
            run(std::integral_constant<int, 8>());
        else if (k <= 16)
            run(std::integral_constant<int, 16>());
        else
            run(std::integral_constant<int, kPassRhs>());
        ProfEnd(prof, s, sizeof(cx<T>) * (L.entries[PH] + L.vecRows[PH] * k),
                8.0 * L.entries[PH] * k);
        if (L.rcount[PH] > 0 && !rc)
            hipLaunchKernelGGL((k_block_reduce<T, PH>), dim3(L.rcount[PH]), dim3(kThreads), 0, s,
                               c.breds + L.rstart[PH], bufs, k);
    };
    const int ng = (int)plan.blevels.size();
    const std::integral_constant<int, PH_F> F;
    const std::integral_constant<int, PH_B> B;
    if (onlyGroup >= 0) {  // one launch, for tuning
        if (onlyPhase == PH_F)
            go(F, onlyGroup);
        else
            go(B, onlyGroup);
        return;
    }
    for (int g = ng - 1; g >= 0; --g) go(F, g);
    for (int g = 0; g < ng; ++g) go(B, g);
}

bool FusedApplies(const ClassDev& c, const ClassPlan& plan, int k, int64_t eb)
{
    // the fused kernel reads its vectors through buffer descriptors: each
    // buffer must span less than 4 GiB
    const int64_t span = (int64_t)1 << 32;
    return c.nqueues > 0 && plan.qcut >= 0 && k >= 8 && k <= 16 &&
           eb * k * (2 * c.wstore + kSolvePad + 2) < span &&
           eb * k * (int64_t)(c.n + kSolvePad + 2) < span &&
           eb * k * 64 * (int64_t)plan.maxSlots < span;
}

template <typename T>
void LaunchPanelSolveFused(const ClassDev& c, const ClassPlan& plan, int b, void* Xpv, void* Wv,
                           void* Pv, void* Gv, int k, hipStream_t s, MvProfile* prof, int32_t* sync)
{
    const cx<T>* L = (const cx<T>*)c.L + (int64_t)b * c.fstore;
    const cx<T>* LT = (const cx<T>*)c.LT + (int64_t)b * c.fstore;
    cx<T>* Xp = (cx<T>*)Xpv;
    cx<T>* W = (cx<T>*)Wv;
    cx<T>* P = (cx<T>*)Pv;
    const Slots<T> gs{(cx<T>*)Gv, c.wstore * k, c.relinds};
    const double eb = sizeof(cx<T>);
    auto byKb = [&](int rows, const auto& go) {
        auto byRows = [&](auto kb) {
            if (rows == 64)
                go(std::integral_constant<int, 64>(), kb);
            else if (rows == 32)
                go(std::integral_constant<int, 32>(), kb);
            else
                go(std::integral_constant<int, 16>(), kb);
        };
        if (k <= 8)
            byRows(std::integral_constant<int, 8>());
        else
            byRows(std::integral_constant<int, 16>());
    };
    // one level above the cut; split row blocks are summed in the launch
    // where their slices were placed per XCD
    auto level = [&](auto ph, int d) {
        constexpr int PH = decltype(ph)::value;
        const ClassPlan::SolveLevel& lv = plan.solveLevels[d];
        const ClassPlan::Range& r = PH == PH_F ? lv.f : lv.b;
        if (r.count <= 0) return;
        int32_t* rc = r.xcd ? c.redc : nullptr;
        ProfBegin(prof, s);
        byKb(r.rows, [&](auto rt, auto kb) {
            hipLaunchKernelGGL((k_mvm<T, PH, decltype(rt)::value, decltype(kb)::value>),
                               dim3(r.count), dim3(256), 0, s, c.mv, r.start, c.structs, gs, L, LT,
                               Xp, W, P, k, rc, c.mvred);
        });
        ProfEnd(prof, s, eb * (lv.entries[PH] + lv.vecRows[PH] * k), 8.0 * lv.entries[PH] * k);
        if (r.rcount > 0 && !rc)
            hipLaunchKernelGGL((k_mv_reduce<T, PH>), dim3(r.rcount), dim3(kThreads), 0, s,
                               c.mvred, r.rstart, gs, Xp, W, P, k);
    };
    auto subtrees = [&](auto ph) {
        constexpr int PH = decltype(ph)::value;
        const int nt = c.nqtiles[PH];
        if (nt <= 0) return;
        int32_t* st = sync + (PH == PH_F ? 0 : QueueSyncInts(c.nnodes, c.nqueues, c.nqreds[0]));
        ProfBegin(prof, s);
        byKb(c.queueRows, [&](auto rt, auto kb) {
            constexpr int RT = decltype(rt)::value, KB = decltype(kb)::value;
            const int G = std::max(1, std::min(nt, MvqGrid<T, PH, RT, KB>(c.cus)));
            hipLaunchKernelGGL((k_mvq<T, PH, RT, KB>), dim3(G), dim3(256), 0, s, c.qtiles[PH],
                               c.qstart[PH], c.qreds[PH], c.qdep[PH], c.nodes, st, c.nnodes,
                               c.nqueues, c.structs, gs, L, LT, Xp, W, P, k);
        });
        const ClassPlan::QueuePhase& Q = plan.queue[PH];
        ProfEnd(prof, s, eb * (Q.entries + Q.vecRows * k), 8.0 * Q.entries * k);
    };
    const std::integral_constant<int, PH_F> F;
    const std::integral_constant<int, PH_B> B;
    subtrees(F);
    for (int d = std::min(plan.maxDepth, plan.qcut - 1); d >= 0; --d) level(F, d);
    for (int d = 0; d < std::min(plan.maxDepth + 1, plan.qcut); ++d) level(B, d);
    subtrees(B);
}

template <typename T>
void LaunchPack(const ClassDev& c, int start, int count, hipStream_t s)
{
    if (count <= 0) return;
    hipLaunchKernelGGL((k_pack<T>), dim3(count, c.npanels), dim3(kThreads), 0, s, c.packs + start,
                       c.foldNodes, c.browBase, (const cx<T>*)c.L, c.fstore, (const cx<T>*)c.U,
                       c.ustore, (cx<T>*)c.F, c.fentries);
}

template <typename T>
void LaunchCompose(const ClassDev& c, int tileStart, int tileCount, hipStream_t s)
{
    if (tileCount <= 0) return;
    hipLaunchKernelGGL((k_compose<T>), dim3(tileCount, c.npanels), dim3(256), 0, s,
                       c.composeTiles + tileStart, c.compose, c.flist, c.fsrc, c.fkeys, c.browBase,
                       (const cx<T>*)c.U, c.ustore, (cx<T>*)c.F, c.fentries);
}

template <typename T>
void LaunchTransposeScale(const ClassDev& c, hipStream_t s)
{
    if (c.ntrans <= 0) return;
    hipLaunchKernelGGL((k_transpose_scale<T>), dim3(c.ntrans, c.npanels), dim3(kThreads), 0, s,
                       c.trans, c.nodes, (cx<T>*)c.L, (cx<T>*)c.LT, c.fstore);
}

template <typename T>
void LaunchFoldBack(const ClassDev& c, hipStream_t s)
{
    if (c.nfold <= 0) return;
    hipLaunchKernelGGL((k_fold_back<T>), dim3(c.nfold, c.npanels), dim3(kThreads), 0, s,
                       c.foldBack, c.nodes, (cx<T>*)c.L, (const cx<T>*)c.LT, c.fstore);
}

template <typename T>
void LaunchCopyIn(const PanelMap& m, const c128* B, void* Xp, int k, int nx, int ny, int nz,
                  int vOffset, int padding, hipStream_t s, int32_t* sync, int nsync)
{
    hipLaunchKernelGGL((k_copy_in<T>), dim3(Blocks((int64_t)m.n * k)), dim3(kThreads), 0, s, m.n,
                       k, m.xy, m.v, B, (cx<T>*)Xp, nx, ny, nz, vOffset, padding, sync,
                       sync ? nsync : 0);
}

template <typename T>
void LaunchCopyOut(const PanelMap& m, c128* B, const void* Xp, int k, int nx, int ny, int nz,
                   int vOffset, int padding, int mode, hipStream_t s, const StencilArgs* st,
                   const double* vel, int v1)
{
    const StencilArgs none{};
    hipLaunchKernelGGL((k_copy_out<T>), dim3(Blocks((int64_t)m.n * k)), dim3(kThreads), 0, s, m.n,
                       k, m.xy, m.v, B, (const cx<T>*)Xp, nx, ny, nz, vOffset, padding, mode,
                       st ? *st : none, vel, st ? v1 : -1);
}

template <typename T>
void LaunchPassOn(const StencilArgs& st, const double* vel, c128* B, int k, const PassPanel& o,
                  const PassPanel& i, int mode, int dir, hipStream_t s)
{
    // few columns: small workgroups, so that they are on more CUs, and more
    // loads at a time
    const int64_t n = (int64_t)st.nx * st.ny * k;
    if (n < 256 * kThreads)
        hipLaunchKernelGGL((k_pass_on<T, 8>), dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, st,
                           vel, B, k, o, i, mode, dir);
    else
        hipLaunchKernelGGL((k_pass_on<T, 4>), dim3(Blocks(n)), dim3(kThreads), 0, s, st, vel, B, k,
                           o, i, mode, dir);
}

template <typename T>
void LaunchZeroSetPlane(const PanelMap& m, const StencilArgs& st, const double* vel,
                        const c128* B, void* Xp, int k, int v2, int vlLast, hipStream_t s,
                        int32_t* sync, int nsync)
{
    hipLaunchKernelGGL((k_zero_set_plane<T>), dim3(Blocks((int64_t)m.n * k)), dim3(kThreads), 0, s,
                       m.n, k, m.xy, m.v, st, vel, B, (cx<T>*)Xp, v2, vlLast, sync,
                       sync ? nsync : 0);
}

template <typename T>
void LaunchSolveBatch(int ph, int kb, const BatchBlock* blocks, int nblocks,
                      const BatchSolveSeg* segs, const int32_t* active, hipStream_t s)
{
    if (nblocks <= 0) return;
    auto go = [&](auto phc) {
        constexpr int PH = decltype(phc)::value;
        auto run = [&](auto kbc) {
            hipLaunchKernelGGL((k_block_batch<T, PH, decltype(kbc)::value>), dim3(nblocks),
                               dim3(256), 0, s, blocks, segs, active);
        };
        if (kb <= 8)
            run(std::integral_constant<int, 8>());
        else if (kb <= 16)
            run(std::integral_constant<int, 16>());
        else
            run(std::integral_constant<int, kPassRhs>());
    };
    if (ph == PH_F)
        go(std::integral_constant<int, PH_F>());
    else
        go(std::integral_constant<int, PH_B>());
}

template <typename T>
void LaunchReduceBatch(int ph, const BatchBlock* blocks, int nblocks, const BatchSolveSeg* segs,
                       const int32_t* active, hipStream_t s)
{
    if (nblocks <= 0) return;
    if (ph == PH_F)
        hipLaunchKernelGGL((k_block_reduce_batch<T, PH_F>), dim3(nblocks), dim3(kThreads), 0, s,
                           blocks, segs, active);
    else
        hipLaunchKernelGGL((k_block_reduce_batch<T, PH_B>), dim3(nblocks), dim3(kThreads), 0, s,
                           blocks, segs, active);
}

template <typename T>
void LaunchCopyBatch(int op, const BatchBlock* blocks, int nblocks, const BatchCopySeg* segs,
                     const int32_t* active, hipStream_t s)
{
    if (nblocks <= 0) return;
    hipLaunchKernelGGL((k_copy_batch<T>), dim3(nblocks), dim3(kBatchCopyThreads), 0, s, op,
                       blocks, segs, active);
}

void LaunchSpmv(const StencilArgs& st, const double* vel, const c128* x, const c128* b, c128* y,
                int k, int mode, hipStream_t s)
{
    auto run = [&](auto vc) {
        constexpr int V = decltype(vc)::value;
        SpmvOrder o;
        const int64_t line = (int64_t)st.nx * k * (int64_t)sizeof(c128);
        o.rows = (int)std::min<int64_t>(st.ny, std::max<int64_t>(1, kStripBytes / line));
        o.strips = (st.ny + o.rows - 1) / o.rows;
        o.per = (int)Blocks((int64_t)o.rows * st.nx * (k / V));
        o.part = ((int64_t)o.strips * st.nz * o.per + 7) / 8;
        const unsigned grid = (unsigned)std::min<int64_t>(8 * o.part, kSpmvGrid);
        if (8 * o.part <= kSpmvGrid)
            hipLaunchKernelGGL((k_spmv<V, false>), dim3(grid), dim3(kThreads), 0, s, st, vel, x, b,
                               y, k, mode, o);
        else
            hipLaunchKernelGGL((k_spmv<V, true>), dim3(grid), dim3(kThreads), 0, s, st, vel, x, b,
                               y, k, mode, o);
    };
    if (k % 2 == 0)
        run(std::integral_constant<int, 2>());
    else
        run(std::integral_constant<int, 1>());
}

int ReducePartials(int64_t npoints)
{
    return (int)std::max<int64_t>(1, std::min<int64_t>(kReduceBlocks, (npoints + 255) / 256));
}

void LaunchColNorm2(const c128* x, int64_t np, int k, double* part, double* out, hipStream_t s)
{
    const int g = ReducePartials(np);
    hipLaunchKernelGGL(k_colnorm_part, dim3(g), dim3(kThreads), 0, s, x, np, k, part);
    hipLaunchKernelGGL(k_colnorm_final, dim3(k), dim3(kThreads), 0, s, part, g, k, out);
}

void LaunchColDot(const c128* v, const c128* w, int64_t np, int k, c128* part, c128* out,
                  hipStream_t s)
{
    const int g = ReducePartials(np);
    hipLaunchKernelGGL(k_coldot_part, dim3(g), dim3(kThreads), 0, s, v, w, np, k, part);
    hipLaunchKernelGGL(k_coldot_final, dim3(k), dim3(kThreads), 0, s, part, g, k, out);
}

int64_t ArnoldiPartials(int64_t np, int k, int m)
{
    return 2 * (int64_t)std::min(m, kMaxGram) * ReducePartials(np) * k;
}

int64_t ArnoldiGram(int k, int m)
{
    const int64_t g = std::min(m, kMaxGram);
    return g * g * k;
}

void LaunchArnoldi(const c128* V, int j, int m, c128* w, int64_t np, int k, c128* part, c128* gram,
                   double* npart, c128* h, double* norms, hipStream_t s)
{
    const int64_t n = np * k;
    const int g = ReducePartials(np);
    if (m <= kMaxGram) {
        hipLaunchKernelGGL(k_arnoldi_dots, dim3(g, (j + kDotGroup) / kDotGroup), dim3(kThreads), 0, s,
                           V, n, j, w, np, k, part);
        hipLaunchKernelGGL(k_arnoldi_solve, dim3(k), dim3(kSolveThreads), 0, s, part, g, j, m, k,
                           gram, h);
        hipLaunchKernelGGL(k_arnoldi_update, dim3(g), dim3(kThreads), 0, s, V, n, j, h, w, np, k,
                           npart);
    } else {
        // step i's update of w and step i + 1's dot product share a pass
        LaunchColDot(V, w, np, k, part, h, s);
        for (int i = 0; i < j; ++i)
            LaunchAxpyDot(h + (int64_t)i * k, V + i * n, V + (i + 1) * n, w, np, k, part,
                          h + (int64_t)(i + 1) * k, s);
        LaunchAxpyCols(h + (int64_t)j * k, -1, V + j * n, w, np, k, s);
        hipLaunchKernelGGL(k_colnorm_part, dim3(g), dim3(kThreads), 0, s, w, np, k, npart);
    }
    hipLaunchKernelGGL(k_colnorm_final, dim3(k), dim3(kThreads), 0, s, npart, g, k, norms);
}

void LaunchAxpyDot(const c128* alpha, const c128* v, const c128* vn, c128* w, int64_t np, int k,
                   c128* part, c128* out, hipStream_t s)
{
    const int g = ReducePartials(np);
    hipLaunchKernelGGL(k_axpy_dot_part, dim3(g), dim3(kThreads), 0, s, alpha, v, vn, w, np, k, part);
    hipLaunchKernelGGL(k_coldot_final, dim3(k), dim3(kThreads), 0, s, part, g, k, out);
}

void LaunchAxpyCols(const c128* alpha, int sign, const c128* v, c128* w, int64_t np, int k,
                    hipStream_t s)
{
    const int64_t n = np * k;
    hipLaunchKernelGGL(k_axpy_cols, dim3(Blocks(n)), dim3(kThreads), 0, s, alpha, sign, v, w, n,
                       k);
}

void LaunchScaleCols(const double* delta, const c128* w, c128* v, int64_t np, int k,
                     hipStream_t s)
{
    const int64_t n = np * k;
    hipLaunchKernelGGL(k_scale_cols, dim3(Blocks(n)), dim3(kThreads), 0, s, delta, w, v, n, k);
}

void LaunchUpdateX(const c128* x0, const c128* V, const c128* y, int j, int64_t np, int k,
                   c128* x, hipStream_t s)
{
    const int64_t n = np * k;
    hipLaunchKernelGGL(k_update_x, dim3(Blocks(n)), dim3(kThreads), 0, s, x0, V, y, j, n, k, n,
                       x);
}

void LaunchNeg(const c128* x, c128* w, int64_t n, hipStream_t s)
{
    hipLaunchKernelGGL(k_neg, dim3(Blocks(n)), dim3(kThreads), 0, s, x, w, n);
}

void LaunchAdjointGrad(const StencilArgs& st, const c128* u, const c128* lam, int k, double* grad,
                       int accumulate, hipStream_t s)
{
    const int64_t n = (int64_t)st.nx * st.ny * st.nz;
    hipLaunchKernelGGL(k_adjoint_grad, dim3(Blocks(n)), dim3(kThreads), 0, s, st, u, lam, k, grad,
                       accumulate);
}

// Explicit instantiations for complex double and complex float fronts.
#define PSP_INST(T)                                                                               \
    template void LaunchScatterOrig<T>(const ClassDev&, const StencilArgs&, const double*, double, \
                                       hipStream_t);                                              \
    template void LaunchExtendAdd<T>(const ClassDev&, int, int, hipStream_t);                     \
    template void LaunchLdlDiag<T>(const ClassDev&, int, int, int, hipStream_t);                  \
    template void LaunchLdlTrsm<T>(const ClassDev&, int, int, int, hipStream_t);                  \
    template void LaunchGemm<T>(const ClassDev&, int, int, hipStream_t);                          \
    template void LaunchInvDiag<T>(const ClassDev&, int, hipStream_t);                            \
    template void LaunchPanelSolve<T>(const ClassDev&, const ClassPlan&, int, void*, void*, int,   \
                                      hipStream_t, MvProfile*, int, int);                         \
    template void LaunchPanelSolveFused<T>(const ClassDev&, const ClassPlan&, int, void*, void*,  \
                                           void*, void*, int, hipStream_t, MvProfile*, int32_t*); \
    template void LaunchPack<T>(const ClassDev&, int, int, hipStream_t);                          \
    template void LaunchCompose<T>(const ClassDev&, int, int, hipStream_t);                       \
    template void LaunchTransposeScale<T>(const ClassDev&, hipStream_t);                          \
    template void LaunchFoldBack<T>(const ClassDev&, hipStream_t);                                \
    template void LaunchCopyIn<T>(const PanelMap&, const c128*, void*, int, int, int, int, int,   \
                                  int, hipStream_t, int32_t*, int);                               \
    template void LaunchCopyOut<T>(const PanelMap&, c128*, const void*, int, int, int, int, int,  \
                                   int, int, hipStream_t, const StencilArgs*, const double*,      \
                                   int);                                                          \
    template void LaunchPassOn<T>(const StencilArgs&, const double*, c128*, int,                  \
                                  const PassPanel&, const PassPanel&, int, int, hipStream_t);     \
    template void LaunchZeroSetPlane<T>(const PanelMap&, const StencilArgs&, const double*,       \
                                        const c128*, void*, int, int, int, hipStream_t, int32_t*, \
                                        int);                                                     \
    template void LaunchSolveBatch<T>(int, int, const BatchBlock*, int, const BatchSolveSeg*,     \
                                      const int32_t*, hipStream_t);                               \
    template void LaunchReduceBatch<T>(int, const BatchBlock*, int, const BatchSolveSeg*,         \
                                       const int32_t*, hipStream_t);                              \
    template void LaunchCopyBatch<T>(int, const BatchBlock*, int, const BatchCopySeg*,            \
                                     const int32_t*, hipStream_t);
PSP_INST(double)
PSP_INST(float)
#undef PSP_INST

}  // namespace psp_amd
