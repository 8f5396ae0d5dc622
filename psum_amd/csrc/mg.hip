// Geometric-transfer Galerkin multigrid for the FD Poisson problem on
// MI355X, served through PSuM's field-solver plugin ABI.
//
// Algorithm (the reference's, restated; PSuM paths):
//   transfers  P = tensor product of 1-D linear interpolation on index axes
//              that keep every other node and the last one; R = P^T scaled
//              by fine/coarse lumped volumes
//              (field_solver/implements/multigrid/multigrid_utilities.hpp:28-104)
//   setup      A0^ = D0^-1 A, A(l+1)^ = D(l+1)^-1 (R A(l)^ P), relax = I - 2/3 A^,
//              dense inverse of the coarsest A^      (multigrid_core.hpp:49-150)
//   V-cycle    weighted Jacobi pre/post smoothing, residual, restrict + D^-1,
//              prolong-add, coarse dense solve        (multigrid_core.hpp:163-272)
//   backends   sycl_multigrid_gpu.cpp:22-230 (FP64) and
//              sycl_multigrid32f_gpu.cpp:23-266 (FP32 V-cycles inside an FP64
//              residual refinement loop; here the coarse solve stays FP64)
//
// MI355X form: the levels' matrices never exist on the device (only the
// coarse end, as the dense matrix of its V-cycle).  Every level is a
// structured node grid (n0 x n1 [x n2], last dimension fastest) whose rows
// are 3^D-point stencils; rows with identical coefficients share a class,
// so a level is a uint16 class id per node plus a small coefficient table.
// Level 0 of a 5/7-point matrix uses the compact (axis-only) stencil kernel.
// Transfers are per-axis weight tables (<= 3 fine nodes per coarse node and
// <= 2 coarse nodes per fine node along each axis).

#include <algorithm>
#include <array>
#include <type_traits>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <memory>
#include <sstream>
#include <stdexcept>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>

#include "common.hpp"
#include "mg_batch.hpp"
#include "psum_field_solver.h"

using namespace psum_hip;

namespace {

constexpr int kMgThreads = 256;
// right-hand sides hold this many zeros beyond their nodes (the dense product
// reads whole 16-byte vectors of its operator's rows)
constexpr int kOpPad = 2;

#define MG_HIP(expr)                                                                        \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess)                                                               \
            throw std::runtime_error(std::string("hip_multigrid: ") + #expr + ": " +       \
                                     hipGetErrorString(e_));                                \
    } while (0)

template <typename F>
void parallel_for(int64_t n, F&& f)
{
    unsigned nt = std::max(1u, std::min(32u, std::thread::hardware_concurrency()));
    if (n < 4096 || nt == 1) {
        for (int64_t i = 0; i < n; ++i) f(i);
        return;
    }
    const int64_t chunk = (n + nt - 1) / nt;
    host_threads(nt, [&](unsigned t) {
        const int64_t b = (int64_t)t * chunk, e = std::min(n, b + chunk);
        for (int64_t i = b; i < e; ++i) f(i);
    });
}

// ------------------------------------------------------------ device data

struct DevLevel {
    int n[3];
    int wrap[3];
    int64_t N;
    const uint16_t* cls;
};

template <typename T>
struct DevTable {
    const T* coef;    // ncls * KS
    const T* dinv;    // ncls
};

template <typename T>
struct DevTransfer {
    const int* pc[3];     // fine f -> lower coarse index
    const T* pw[3];       // fine f -> weights (2 per f)
    const int* rf[3];     // coarse c -> first fine index
    const int* rn[3];     // coarse c -> number of fine nodes (1..3)
    const T* rw[3];       // coarse c -> weights (3 per c)
    int wrap[3];          // periodic axis: indices wrap modulo the axis length
};

__device__ __forceinline__ int wrap_index(int i, int n, int wrap)
{
    if (!wrap) return i;
    return i < 0 ? i + n : (i >= n ? i - n : i);
}

// node coordinates of linear index i (row-major, last axis fastest); 32-bit
// unsigned division when the level has fewer than 2^32 nodes (64-bit
// division is a long software sequence on the GPU)
template <int D>
__device__ __forceinline__ void node_coords(const DevLevel& L, int64_t i, int* c)
{
    if (L.N <= (int64_t)0xffffffffll) {
        uint32_t u = (uint32_t)i;
        if (D == 3) {
            const uint32_t q = u / (uint32_t)L.n[2];
            c[2] = (int)(u - q * (uint32_t)L.n[2]);
            u = q;
        }
        const uint32_t q = u / (uint32_t)L.n[1];
        c[1] = (int)(u - q * (uint32_t)L.n[1]);
        c[0] = (int)q;
        return;
    }
    if (D == 3) {
        c[2] = (int)(i % L.n[2]);
        i /= L.n[2];
    }
    c[1] = (int)(i % L.n[1]);
    c[0] = (int)(i / L.n[1]);
}

__device__ __forceinline__ int nb_index(int c, int o, int n, int wrap)
{
    int q = c + o;
    if (q < 0) q = wrap ? q + n : 0;
    else if (q >= n) q = wrap ? q - n : n - 1;
    return q;
}

// Workgroups are dealt to the eight XCDs round-robin (workgroup b runs on
// XCD b % 8).  xcd_block() renumbers them so that each XCD works through one
// contiguous eighth of the index range: on 3D levels the neighbour planes a
// stencil reads (n1*n2 nodes apart) then stay in the same XCD's L2.  Blocks
// of an incomplete last round keep their index, so the map is a bijection
// for any grid size.
constexpr unsigned kXcds = 8;
__device__ __forceinline__ int64_t xcd_block()
{
    const unsigned g = gridDim.x, b = blockIdx.x;
    const unsigned full = g / kXcds * kXcds;
    if (b >= full) return b;
    return (int64_t)(b % kXcds) * (full / kXcds) + b / kXcds;
}

template <int D>
__device__ __forceinline__ int64_t level_block()
{
    return D == 3 ? xcd_block() : (int64_t)blockIdx.x;
}

// sum_k coef[k] * x[nb_k], k ascending over the 3^D offsets (o0 slowest),
// COMPACT: only the 2D+1 axis offsets (all other coefficients are zero).
template <typename T, int D, bool COMPACT>
__device__ __forceinline__ T stencil_apply(const DevLevel& L, const T* __restrict__ coef,
                                          const T* __restrict__ x, const int* c)
{
    T s = (T)0;
    if (D == 2) {
        const int n0 = L.n[0], n1 = L.n[1];
#pragma unroll
        for (int a = -1; a <= 1; ++a)
#pragma unroll
            for (int b = -1; b <= 1; ++b) {
                if (COMPACT && a != 0 && b != 0) continue;
                const int k = (a + 1) * 3 + (b + 1);
                const int q0 = nb_index(c[0], a, n0, L.wrap[0]);
                const int q1 = nb_index(c[1], b, n1, L.wrap[1]);
                s = s + coef[k] * x[(int64_t)q0 * n1 + q1];
            }
    } else {
        const int n0 = L.n[0], n1 = L.n[1], n2 = L.n[2];
#pragma unroll
        for (int a = -1; a <= 1; ++a)
#pragma unroll
            for (int b = -1; b <= 1; ++b)
#pragma unroll
                for (int e = -1; e <= 1; ++e) {
                    if (COMPACT && ((a != 0) + (b != 0) + (e != 0)) > 1) continue;
                    const int k = (a + 1) * 9 + (b + 1) * 3 + (e + 1);
                    const int q0 = nb_index(c[0], a, n0, L.wrap[0]);
                    const int q1 = nb_index(c[1], b, n1, L.wrap[1]);
                    const int q2 = nb_index(c[2], e, n2, L.wrap[2]);
                    s = s + coef[k] * x[((int64_t)q0 * n1 + q1) * n2 + q2];
                }
    }
    return s;
}

// x_out = relax x_in + b * (2/3)   (multiply_add(relax, x, b, buf, 2/3, 1));
// ACC: also xacc += x_out in FP64 (the mixed refinement's x += e, fused into
// the last level-0 sweep)
template <typename T, int D, bool COMPACT, bool ACC>
__device__ __forceinline__ void smooth_node(const DevLevel& L, const DevTable<T>& relax,
                                            const T* __restrict__ xin, const T* __restrict__ b,
                                            T* __restrict__ xout, T two3, double* __restrict__ xacc,
                                            int64_t i)
{
    int c[3];
    node_coords<D>(L, i, c);
    const T* coef = relax.coef + (int64_t)L.cls[i] * (D == 2 ? 9 : 27);
    const T t = stencil_apply<T, D, COMPACT>(L, coef, xin, c);
    const T v = t * (T)1 + b[i] * (two3 * (T)1);
    xout[i] = v;
    if (ACC) xacc[i] += (double)v;
}

template <typename T, int D, bool COMPACT, bool ACC = false>
__global__ __launch_bounds__(kMgThreads) void k_smooth(DevLevel L, DevTable<T> relax,
                                                       const T* __restrict__ xin,
                                                       const T* __restrict__ b,
                                                       T* __restrict__ xout, T two3,
                                                       double* __restrict__ xacc = nullptr)
{
    const int64_t i = level_block<D>() * kMgThreads + threadIdx.x;
    if (i >= L.N) return;
    smooth_node<T, D, COMPACT, ACC>(L, relax, xin, b, xout, two3, xacc, i);
}

// r = (A^ x)*(-1) + b*((-1)*(-1))   (multiply_add(A, x, b, buf, -1, -1))
template <typename T, int D, bool COMPACT>
__device__ __forceinline__ void residual_node(const DevLevel& L, const DevTable<T>& A, const T* __restrict__ x,
                                              const T* __restrict__ b, T* __restrict__ r, int64_t i)
{
    int c[3];
    node_coords<D>(L, i, c);
    const T* coef = A.coef + (int64_t)L.cls[i] * (D == 2 ? 9 : 27);
    const T t = stencil_apply<T, D, COMPACT>(L, coef, x, c);
    r[i] = t * (T)-1 + b[i] * (T)1;
}

template <typename T, int D, bool COMPACT>
__global__ __launch_bounds__(kMgThreads) void k_residual(DevLevel L, DevTable<T> A,
                                                         const T* __restrict__ x,
                                                         const T* __restrict__ b,
                                                         T* __restrict__ r)
{
    const int64_t i = level_block<D>() * kMgThreads + threadIdx.x;
    if (i >= L.N) return;
    residual_node<T, D, COMPACT>(L, A, x, b, r, i);
}

// ---- 3D levels in chunks of kLine consecutive nodes ------------------------
// On a 3D level nearly every node lies inside the box and carries the same
// stencil class.  A chunk of kLine nodes (linear indices kLine*t ..
// kLine*t + kLine-1) all on one grid line, strictly inside the box, all of
// that class, is updated by one thread with the class row in registers and
// vector loads of the line and its neighbour lines (four for a 7-point
// level, eight for a 27-point one): no coordinate division per node, no
// clamping, no per-node table reads.  The per-node terms and their order
// are stencil_apply's, so the result is bit-identical to k_smooth /
// k_residual.  The other nodes (box faces, line ends, other classes, the
// tail) are listed when the level is built and updated by the per-node
// kernels over that list.
constexpr int kLine = 4;

struct LineGeom {
    int n0, n1, n2;
    uint32_t nchunks;          // full chunks: N / kLine
    const uint16_t* cls;
    int cls_in;                // the class the chunk kernels handle
};

// the chunk of nodes i .. i+kLine-1 (i = kLine*t) is a chunk-kernel chunk
// (the host lists the others with line_chunk_fast_host, the same test)
__device__ __forceinline__ bool line_chunk_fast(const LineGeom& G, uint32_t i)
{
    const uint32_t q = i / (uint32_t)G.n2;
    const uint32_t z = i - q * (uint32_t)G.n2;
    const uint32_t x = q / (uint32_t)G.n1;
    const uint32_t y = q - x * (uint32_t)G.n1;
    if (z < 1u || z + kLine > (uint32_t)G.n2 - 1u || y < 1u || y + 2u > (uint32_t)G.n1 || x < 1u ||
        x + 2u > (uint32_t)G.n0)
        return false;
    unsigned long long c4;
    __builtin_memcpy(&c4, G.cls + i, sizeof c4);
    const unsigned long long in = (unsigned long long)(uint16_t)G.cls_in;
    return c4 == (in | in << 16 | in << 32 | in << 48);
}

template <typename T>
__device__ __forceinline__ void ld_line(const T* __restrict__ p, T* v)
{
    struct alignas(sizeof(T)) Q { T a[kLine]; } q;
    __builtin_memcpy(&q, p, sizeof q);
#pragma unroll
    for (int k = 0; k < kLine; ++k) v[k] = q.a[k];
}

template <typename T>
__device__ __forceinline__ void st_line(T* __restrict__ p, const T* v)
{
    struct alignas(sizeof(T)) Q { T a[kLine]; } q;
#pragma unroll
    for (int k = 0; k < kLine; ++k) q.a[k] = v[k];
    __builtin_memcpy(p, &q, sizeof q);
}

// stencil_apply<T, 3, COMPACT> at the chunk's nodes: the 7-point sum in
// offset order x-1, y-1, z-1, centre, z+1, y+1, x+1, or the 27-point sum
// with offsets (a, b, e) in x, y, z ascending, z fastest
template <typename T, bool COMPACT>
__device__ __forceinline__ void line_apply(const LineGeom& G, const T* __restrict__ row,
                                           const T* __restrict__ x, uint32_t i, T* s)
{
    const uint32_t sy = (uint32_t)G.n2, sx = (uint32_t)G.n1 * (uint32_t)G.n2;
    if constexpr (COMPACT) {
        const T cxm = row[4], cym = row[10], czm = row[12], cc = row[13], czp = row[14], cyp = row[16],
                cxp = row[22];
        T xm[kLine], ym[kLine], zz[kLine + 2], yp[kLine], xp[kLine];
        ld_line(x + (i - sx), xm);
        ld_line(x + (i - sy), ym);
        zz[0] = x[i - 1];
        ld_line(x + i, zz + 1);
        zz[kLine + 1] = x[i + kLine];
        ld_line(x + (i + sy), yp);
        ld_line(x + (i + sx), xp);
#pragma unroll
        for (int k = 0; k < kLine; ++k) {
            T t = (T)0;
            t = t + cxm * xm[k];
            t = t + cym * ym[k];
            t = t + czm * zz[k];
            t = t + cc * zz[k + 1];
            t = t + czp * zz[k + 2];
            t = t + cyp * yp[k];
            t = t + cxp * xp[k];
            s[k] = t;
        }
    } else {
#pragma unroll
        for (int k = 0; k < kLine; ++k) s[k] = (T)0;
#pragma unroll
        for (int a = -1; a <= 1; ++a)
#pragma unroll
            for (int b = -1; b <= 1; ++b) {
                const T* ln = x + (i + (uint32_t)((int)sx * a + (int)sy * b));
                T zz[kLine + 2];
                zz[0] = ln[-1];
                ld_line(ln, zz + 1);
                zz[kLine + 1] = ln[kLine];
#pragma unroll
                for (int e = -1; e <= 1; ++e) {
                    const T c = row[(a + 1) * 9 + (b + 1) * 3 + (e + 1)];
#pragma unroll
                    for (int k = 0; k < kLine; ++k) s[k] = s[k] + c * zz[k + 1 + e];
                }
            }
    }
}

// A launch takes nbc blocks of chunks and nblk(n) blocks of listed nodes
// (one per thread, with the per-node kernels' code).  Workgroup b runs on
// XCD x = b % kXcds as that XCD's j = b / kXcds-th: j < lb takes listed block
// x*lb + j, later ones chunk block x*cb + (j - lb) (lb, cb: the listed and
// chunk blocks per XCD, rounded up; indexes past the end exit).  Every XCD
// thus gets an eighth of the listed nodes, whose per-node path is slower,
// started first, and a contiguous eighth of the chunks.
struct LineList {
    const uint32_t* list;
    uint32_t n;
    uint32_t nbc;              // blocks of chunks
};

__host__ __device__ __forceinline__ uint32_t line_listed_blocks(const LineList& LL)
{
    return (LL.n + kMgThreads - 1) / kMgThreads;
}
__host__ __device__ __forceinline__ uint32_t line_grid(const LineList& LL)
{
    const uint32_t lb = (line_listed_blocks(LL) + kXcds - 1) / kXcds, cb = (LL.nbc + kXcds - 1) / kXcds;
    return kXcds * (lb + cb);
}
// this workgroup's block: listed (true) or chunk, and its index (-1: none)
__device__ __forceinline__ int64_t line_block(const LineList& LL, bool* listed)
{
    const uint32_t nbl = line_listed_blocks(LL);
    const uint32_t lb = (nbl + kXcds - 1) / kXcds, cb = (LL.nbc + kXcds - 1) / kXcds;
    const uint32_t x = blockIdx.x % kXcds, j = blockIdx.x / kXcds;
    if (j < lb) {
        *listed = true;
        const uint32_t k = x * lb + j;
        return k < nbl ? (int64_t)k : -1;
    }
    *listed = false;
    const uint32_t k = x * cb + (j - lb);
    return k < LL.nbc ? (int64_t)k : -1;
}

template <typename T, bool COMPACT, bool ACC>
__global__ __launch_bounds__(kMgThreads) void k_smooth_line(LineGeom G, LineList LL, DevLevel L, DevTable<T> relax,
                                                            const T* __restrict__ row,
                                                            const T* __restrict__ xin,
                                                            const T* __restrict__ b,
                                                            T* __restrict__ xout, T two3,
                                                            double* __restrict__ xacc)
{
    bool listed;
    const int64_t blk = line_block(LL, &listed);
    if (blk < 0) return;
    if (listed) {
        const int64_t t = blk * kMgThreads + threadIdx.x;
        if (t < (int64_t)LL.n) smooth_node<T, 3, COMPACT, ACC>(L, relax, xin, b, xout, two3, xacc, (int64_t)LL.list[t]);
        return;
    }
    const int64_t t = blk * kMgThreads + threadIdx.x;
    if (t >= (int64_t)G.nchunks) return;
    const uint32_t i = (uint32_t)t * kLine;
    if (!line_chunk_fast(G, i)) return;
    T s[kLine], bb[kLine], v[kLine];
    line_apply<T, COMPACT>(G, row, xin, i, s);
    ld_line(b + i, bb);
#pragma unroll
    for (int k = 0; k < kLine; ++k) v[k] = s[k] * (T)1 + bb[k] * (two3 * (T)1);
    st_line(xout + i, v);
    if (ACC) {
        double a[kLine];
        ld_line(xacc + i, a);
#pragma unroll
        for (int k = 0; k < kLine; ++k) a[k] += (double)v[k];
        st_line(xacc + i, a);
    }
}

template <typename T, bool COMPACT>
__global__ __launch_bounds__(kMgThreads) void k_residual_line(LineGeom G, LineList LL, DevLevel L, DevTable<T> A,
                                                              const T* __restrict__ row,
                                                              const T* __restrict__ x,
                                                              const T* __restrict__ b, T* __restrict__ r)
{
    bool listed;
    const int64_t blk = line_block(LL, &listed);
    if (blk < 0) return;
    if (listed) {
        const int64_t t = blk * kMgThreads + threadIdx.x;
        if (t < (int64_t)LL.n) residual_node<T, 3, COMPACT>(L, A, x, b, r, (int64_t)LL.list[t]);
        return;
    }
    const int64_t t = blk * kMgThreads + threadIdx.x;
    if (t >= (int64_t)G.nchunks) return;
    const uint32_t i = (uint32_t)t * kLine;
    if (!line_chunk_fast(G, i)) return;
    T s[kLine], bb[kLine], v[kLine];
    line_apply<T, COMPACT>(G, row, x, i, s);
    ld_line(b + i, bb);
#pragma unroll
    for (int k = 0; k < kLine; ++k) v[k] = s[k] * (T)-1 + bb[k] * (T)1;
    st_line(r + i, v);
}

// b_c = (R r) o D_c^-1 ; x_c = 0, or, when the coarse level is pre-smoothed,
// the first Jacobi sweep from x_c = 0 fused in: relax*0 + b_c*(2/3) is
// exactly b_c * (2/3) (first_sweep = 2/3; 0 means plain x_c = 0).
template <typename T, int D>
__global__ __launch_bounds__(kMgThreads) void k_restrict(DevLevel F, DevLevel Cl,
                                                         DevTransfer<T> tr, DevTable<T> Ac,
                                                         const T* __restrict__ r,
                                                         T* __restrict__ bc, T* __restrict__ xc,
                                                         T first_sweep)
{
    const int64_t i = level_block<D>() * kMgThreads + threadIdx.x;
    if (i >= Cl.N) return;
    int c[3];
    node_coords<D>(Cl, i, c);
    T s = (T)0;
    const int f0 = tr.rf[0][c[0]], m0 = tr.rn[0][c[0]];
    const int f1 = tr.rf[1][c[1]], m1 = tr.rn[1][c[1]];
    if (D == 2) {
        for (int a = 0; a < m0; ++a) {
            const T w0 = tr.rw[0][3 * c[0] + a];
            const int i0 = wrap_index(f0 + a, F.n[0], tr.wrap[0]);
            for (int b = 0; b < m1; ++b) {
                const T w = w0 * tr.rw[1][3 * c[1] + b];
                const int i1 = wrap_index(f1 + b, F.n[1], tr.wrap[1]);
                s = s + w * r[(int64_t)i0 * F.n[1] + i1];
            }
        }
    } else {
        const int f2 = tr.rf[2][c[2]], m2 = tr.rn[2][c[2]];
        for (int a = 0; a < m0; ++a) {
            const T w0 = tr.rw[0][3 * c[0] + a];
            const int i0 = wrap_index(f0 + a, F.n[0], tr.wrap[0]);
            for (int b = 0; b < m1; ++b) {
                const T w01 = w0 * tr.rw[1][3 * c[1] + b];
                const int i1 = wrap_index(f1 + b, F.n[1], tr.wrap[1]);
                const int64_t row = ((int64_t)i0 * F.n[1] + i1) * F.n[2];
                for (int e = 0; e < m2; ++e) {
                    const T w = w01 * tr.rw[2][3 * c[2] + e];
                    s = s + w * r[row + wrap_index(f2 + e, F.n[2], tr.wrap[2])];
                }
            }
        }
    }
    const T bv = s * Ac.dinv[Cl.cls[i]];
    bc[i] = bv;
    xc[i] = first_sweep != (T)0 ? bv * (first_sweep * (T)1) : (T)0;
}

// x_f = (P x_c)*1 + x_f*(1*1)
template <typename T, int D>
__global__ __launch_bounds__(kMgThreads) void k_prolong_add(DevLevel F, DevLevel Cl,
                                                            DevTransfer<T> tr,
                                                            const T* __restrict__ xc,
                                                            T* __restrict__ xf)
{
    const int64_t i = level_block<D>() * kMgThreads + threadIdx.x;
    if (i >= F.N) return;
    int c[3];
    node_coords<D>(F, i, c);
    T s = (T)0;
    const int p0 = tr.pc[0][c[0]], p1 = tr.pc[1][c[1]];
    const T* w0 = tr.pw[0] + 2 * c[0];
    const T* w1 = tr.pw[1] + 2 * c[1];
    if (D == 2) {
        for (int a = 0; a < 2; ++a) {
            if (w0[a] == (T)0) continue;
            const int i0 = wrap_index(p0 + a, Cl.n[0], tr.wrap[0]);
            for (int b = 0; b < 2; ++b) {
                if (w1[b] == (T)0) continue;
                const int i1 = wrap_index(p1 + b, Cl.n[1], tr.wrap[1]);
                s = s + (w0[a] * w1[b]) * xc[(int64_t)i0 * Cl.n[1] + i1];
            }
        }
    } else {
        const int p2 = tr.pc[2][c[2]];
        const T* w2 = tr.pw[2] + 2 * c[2];
        for (int a = 0; a < 2; ++a) {
            if (w0[a] == (T)0) continue;
            const int i0 = wrap_index(p0 + a, Cl.n[0], tr.wrap[0]);
            for (int b = 0; b < 2; ++b) {
                if (w1[b] == (T)0) continue;
                const T w01 = w0[a] * w1[b];
                const int i1 = wrap_index(p1 + b, Cl.n[1], tr.wrap[1]);
                for (int e = 0; e < 2; ++e) {
                    if (w2[e] == (T)0) continue;
                    const int i2 = wrap_index(p2 + e, Cl.n[2], tr.wrap[2]);
                    s = s + (w01 * w2[e]) * xc[((int64_t)i0 * Cl.n[1] + i1) * Cl.n[2] + i2];
                }
            }
        }
    }
    xf[i] = s * (T)1 + xf[i] * (T)1;
}

// ---- 3D transfers over planes ---------------------------------------------
// k_prolong_add / k_restrict on 3D levels with a two-dimensional launch:
// blockIdx.y is the output node's slowest coordinate, so its transfer table
// entries are uniform across the block, and one division splits the rest of
// the index.  Each node's terms and their order are the per-node kernels',
// so the bits are the same.
// index p + o on an axis of n nodes, wrapped on a periodic axis, else kept
// in range (the caller selects the term away when p + o is outside)
__device__ __forceinline__ uint32_t axis_index(int p, int n, int wrap)
{
    int q = wrap_index(p, n, wrap);
    q = q < 0 ? 0 : (q >= n ? n - 1 : q);
    return (uint32_t)q;
}

template <typename T>
__global__ __launch_bounds__(kMgThreads) void k_prolong_add_plane(DevLevel F, DevLevel Cl, DevTransfer<T> tr,
                                                                  const T* __restrict__ xc, T* __restrict__ xf)
{
    const uint32_t j = blockIdx.x * kMgThreads + threadIdx.x;
    const uint32_t plane = (uint32_t)F.n[1] * (uint32_t)F.n[2];
    if (j >= plane) return;
    const int c0 = blockIdx.y;
    const int c1 = (int)(j / (uint32_t)F.n[2]);
    const int c2 = (int)(j - (uint32_t)c1 * (uint32_t)F.n[2]);
    const int64_t i = (int64_t)c0 * plane + j;
    const int p0 = tr.pc[0][c0], p1 = tr.pc[1][c1], p2 = tr.pc[2][c2];
    T w0[2], w1[2], w2[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        w0[a] = tr.pw[0][2 * c0 + a];
        w1[a] = tr.pw[1][2 * c1 + a];
        w2[a] = tr.pw[2][2 * c2 + a];
    }
    // all eight coarse values are loaded before any is used (addresses kept
    // in range); a term whose weight is zero is then skipped by a select, so
    // the sum is k_prolong_add's, term for term
    const uint32_t cs1 = (uint32_t)Cl.n[2], cs0 = (uint32_t)Cl.n[1] * (uint32_t)Cl.n[2];
    uint32_t q0[2], q1[2], q2[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        q0[a] = axis_index(p0 + a, Cl.n[0], tr.wrap[0]) * cs0;
        q1[a] = axis_index(p1 + a, Cl.n[1], tr.wrap[1]) * cs1;
        q2[a] = axis_index(p2 + a, Cl.n[2], tr.wrap[2]);
    }
    T v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = xc[q0[k >> 2] + q1[(k >> 1) & 1] + q2[k & 1]];
    const T xo = xf[i];
    T s = (T)0;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const T w01 = w0[a] * w1[b];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const bool use = w0[a] != (T)0 && w1[b] != (T)0 && w2[e] != (T)0;
                const T t = s + (w01 * w2[e]) * v[a * 4 + b * 2 + e];
                s = use ? t : s;
            }
        }
    xf[i] = s * (T)1 + xo * (T)1;
}

// k_restrict on 3D levels: the slowest coarse coordinate in blockIdx.y and
// all (up to 27) fine residuals loaded before any is used; a term outside
// the node's support (a >= m0, ...) is skipped by a select, so the sum is
// k_restrict's, term for term.
template <typename T>
__global__ __launch_bounds__(kMgThreads) void k_restrict_plane(DevLevel F, DevLevel Cl, DevTransfer<T> tr,
                                                               DevTable<T> Ac, const T* __restrict__ r,
                                                               T* __restrict__ bc, T* __restrict__ xc,
                                                               T first_sweep)
{
    const uint32_t j = blockIdx.x * kMgThreads + threadIdx.x;
    const uint32_t plane = (uint32_t)Cl.n[1] * (uint32_t)Cl.n[2];
    if (j >= plane) return;
    const int c0 = blockIdx.y;
    const int c1 = (int)(j / (uint32_t)Cl.n[2]);
    const int c2 = (int)(j - (uint32_t)c1 * (uint32_t)Cl.n[2]);
    const int64_t i = (int64_t)c0 * plane + j;
    const int f0 = tr.rf[0][c0], m0 = tr.rn[0][c0];
    const int f1 = tr.rf[1][c1], m1 = tr.rn[1][c1];
    const int f2 = tr.rf[2][c2], m2 = tr.rn[2][c2];
    T w0[3], w1[3], w2[3];
    uint32_t g0[3], g1[3], g2[3];
    const uint32_t fs1 = (uint32_t)F.n[2], fs0 = (uint32_t)F.n[1] * (uint32_t)F.n[2];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        w0[a] = tr.rw[0][3 * c0 + a];
        w1[a] = tr.rw[1][3 * c1 + a];
        w2[a] = tr.rw[2][3 * c2 + a];
        g0[a] = axis_index(f0 + a, F.n[0], tr.wrap[0]) * fs0;
        g1[a] = axis_index(f1 + a, F.n[1], tr.wrap[1]) * fs1;
        g2[a] = axis_index(f2 + a, F.n[2], tr.wrap[2]);
    }
    T v[27];
#pragma unroll
    for (int k = 0; k < 27; ++k) v[k] = r[g0[k / 9] + g1[(k / 3) % 3] + g2[k % 3]];
    const uint16_t ci = Cl.cls[i];
    T s = (T)0;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const T w01 = w0[a] * w1[b];
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                const bool use = a < m0 && b < m1 && e < m2;
                const T t = s + (w01 * w2[e]) * v[a * 9 + b * 3 + e];
                s = use ? t : s;
            }
        }
    const T bv = s * Ac.dinv[ci];
    bc[i] = bv;
    xc[i] = first_sweep != (T)0 ? bv * (first_sweep * (T)1) : (T)0;
}

// ---- batched launches ------------------------------------------------------
// A batched launch runs one kernel body for several independent solver
// instances: instance i owns blocks first[i] .. first[i+1]-1 of the grid and
// reads its arguments from args[i].  The bodies below take the block index
// as a parameter, so a single-instance launch (block = blockIdx.x) and a
// batched one execute identical arithmetic.
__device__ __forceinline__ int batch_instance(const unsigned* __restrict__ first, int n)
{
    int lo = 0, hi = n - 1;
    const unsigned b = blockIdx.x;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first[mid] <= b) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// ---- fused 2D kernels: a tile of the level in LDS -------------------------
// A block works on 64 columns (one wave per row) of a tile held in LDS with a
// halo as wide as the operations need: h Jacobi sweeps (sweep k updates the
// region shrunk by k, so the output nodes hold exactly what h launches of
// k_smooth produce, same operations in the same order), and in k_down_tile
// one more node for the residual.  A thread owns one column and RPT
// consecutive rows: its right-hand side and class rows stay in registers and the 3 x 3 window slides down its rows, so a
// sweep reads 3 (RPT + 2) LDS values per thread instead of 9 values and 9
// coefficients per node.  The iterate ping-pongs between two LDS planes;
// class tables of up to kMaxClsLds classes are staged in LDS.  Halo nodes
// beyond a non-wrapped edge are clamped copies: the stencils of real nodes
// give them zero coefficients, as in k_smooth's clamped neighbour.
//
// Everything a block reads is asked for in one run of unconditional loads
// before its first barrier (transfer tables, coarse values, weights of the
// restriction): on small levels a launch is a chain of memory round trips and
// of instruction fetches, not bandwidth.  128^2 and 64^2 FP64 levels of 256
// threads a block: 6.7-7.9 us a launch with copy loops and conditional loads,
// 5.7-6.7 us so; 1024^2 FP32: 19.7 and 20.0 -> 17.3 and 18.8 us.  Two
// geometries per precision: large tiles, 1024 threads over 32 rows (16 coarse
// rows) in FP32 and 512 threads over 16 rows (7 coarse rows) in FP64, and 256
// threads over 8 rows (3 coarse rows) for levels that large tiles would leave
// mostly idle (small_tiles()).  All of a block's waves wait for the same
// barriers, so a compute unit with two blocks of 1024 threads moves nothing
// meanwhile: on large FP64 levels, which are bound by bandwidth, four blocks
// of 512 threads are faster (walls, 2049^2: prolongation and sweep 58 -> 45
// us, downward half 78 -> 71 us; 1025^2: 20 -> 15 and 25 -> 23 us).
constexpr int kTileX = 64;
constexpr int kMaxFuse = 3;
constexpr int kMaxClsLds = 32;

template <typename T, bool SMALL>
struct TileGeom {
    static constexpr int threads = SMALL ? 256 : (sizeof(T) == 8 ? 512 : 1024);
    static constexpr int groups = threads / kTileX;     // waves, one row group each
    static constexpr int rpt = SMALL ? 4 : 3;           // consecutive rows per thread
    static constexpr int rows = SMALL ? 8 : (sizeof(T) == 8 ? 16 : 32);   // output rows of a smoothing tile
    static constexpr int crows = SMALL ? 3 : (sizeof(T) == 8 ? 7 : 16);   // coarse rows of a k_down_tile tile
    // one guard row on each side, one guard value before and after: tile row
    // i, column tx at at(i, tx)
    static constexpr int plane = (groups * rpt + 2) * kTileX + 2;
    // values of a class table, and of the coarse values a prolongation reads
    // (cw columns, ch rows), each thread brings into LDS
    static constexpr int tab_per = (kMaxClsLds * 9 + threads - 1) / threads;
    static constexpr int cw = kTileX / 2 + 2, ch = (groups * rpt) / 2 + 2;
    static constexpr int xc_per = (cw * ch + threads - 1) / threads;
    static __device__ __forceinline__ int at(int i, int tx) { return (i + 1) * kTileX + tx + 1; }
    static_assert(rows + 2 * kMaxFuse <= groups * rpt, "smoothing tile exceeds its planes");
    static_assert(2 * crows + 1 + 2 + 2 * kMaxFuse <= groups * rpt, "k_down_tile tile exceeds its planes");
    static_assert(crows <= groups, "one coarse row per wave");
};

// The thread's share of a class table, loaded to registers and stored to LDS
// later: a loop that copies global to LDS waits for memory in every turn, so
// the tile's other loads would only be asked for after it (a round trip is
// 0.5-1 us on lines that another XCD wrote).
template <bool SMALL, typename T>
__device__ __forceinline__ void tab_load(const T* __restrict__ coef, int n, T* v)
{
#pragma unroll
    for (int q = 0; q < TileGeom<T, SMALL>::tab_per; ++q) {
        const int i = threadIdx.x + q * TileGeom<T, SMALL>::threads;
        v[q] = coef[i < n ? i : 0];
    }
}
template <bool SMALL, typename T>
__device__ __forceinline__ void tab_store(T* lds, int n, const T* v)
{
#pragma unroll
    for (int q = 0; q < TileGeom<T, SMALL>::tab_per; ++q) {
        const int i = threadIdx.x + q * TileGeom<T, SMALL>::threads;
        if (i < n) lds[i] = v[q];
    }
}

// wrapped (periodic axis) or clamped node coordinate; g is less than two
// tiles outside [0, n).  Without loops or branches (they were a third of the
// tile kernels' code): the float quotient is off by at most one below 2^23
// periods, which the selects mend.
__device__ __forceinline__ int tile_coord(int g, int n, int wrap)
{
    const int q = (int)floorf((float)g * __builtin_amdgcn_rcpf((float)n));
    int m = g - q * n;
    m = m < 0 ? m + n : m;
    m = m >= n ? m - n : m;
    const int w = wrap ? -1 : 0;
    return (m & w) | (min(max(g, 0), n - 1) & ~w);
}

template <typename T, bool COMPACT>
struct TileRow {
    static constexpr int n = COMPACT ? 5 : 9;
    T c[n];
    __device__ __forceinline__ void load(const T* __restrict__ row)
    {
        if (COMPACT) {
            c[0] = row[1]; c[1] = row[3]; c[2] = row[4]; c[3] = row[5]; c[4] = row[7];
        } else {
#pragma unroll
            for (int q = 0; q < n; ++q) c[q] = row[q];
        }
    }
    // u, m, d: the rows above, at and below the node (columns -1, 0, 1)
    __device__ __forceinline__ T apply(const T* u, const T* m, const T* d) const
    {
        T t = (T)0;
        if (COMPACT) {
            t = t + c[0] * u[1];
            t = t + c[1] * m[0];
            t = t + c[2] * m[1];
            t = t + c[3] * m[2];
            t = t + c[4] * d[1];
        } else {
#pragma unroll
            for (int q = 0; q < 3; ++q) t = t + c[q] * u[q];
#pragma unroll
            for (int q = 0; q < 3; ++q) t = t + c[3 + q] * m[q];
#pragma unroll
            for (int q = 0; q < 3; ++q) t = t + c[6 + q] * d[q];
        }
        return t;
    }
};

// f(k, sum) for the thread's rows k: sum = the class row applied to the plane
// (p: the thread's column in the row above its first)
template <typename T, bool COMPACT, bool SMALL, typename R, typename F>
__device__ __forceinline__ void tile_stencil(const T* p, R&& row, F&& f)
{
    constexpr int RPT = TileGeom<T, SMALL>::rpt;
    T w[3][3];
    // a compact row reads only column 0 of the rows above and below
    auto get = [&](int r, T* q, bool side) {
        const T* a = p + r * kTileX;
        q[1] = a[0];
        if (side) {
            q[0] = a[-1];
            q[2] = a[1];
        }
    };
    get(0, w[0], !COMPACT);
    get(1, w[1], true);
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        T* u = w[k % 3];
        T* m = w[(k + 1) % 3];
        T* d = w[(k + 2) % 3];
        get(k + 2, d, !COMPACT || k + 1 < RPT);
        f(k, row(k).apply(u, m, d));
    }
}

// h sweeps of the thread's rows between the planes; returns the plane that
// holds the result.  i0: the thread's first tile row, R: tile rows in use.
template <typename T, bool COMPACT, bool SMALL, typename R, typename P>
__device__ __forceinline__ int tile_sweeps(P& sx, int tx, int i0, int nrows, int h, const T* breg, T two3, R&& row)
{
    int cur = 0;
    for (int sw = 1; sw <= h; ++sw) {
        const T* xs = &sx[cur][TileGeom<T, SMALL>::at(i0 - 1, tx)];
        T* xn = &sx[cur ^ 1][TileGeom<T, SMALL>::at(i0, tx)];
        const bool colok = tx >= sw && tx < kTileX - sw;
        tile_stencil<T, COMPACT, SMALL>(xs, row, [&](int k, T t) {
            const int i = i0 + k;
            if (colok && i >= sw && i < nrows - sw) xn[k * kTileX] = t * (T)1 + breg[k] * (two3 * (T)1);
        });
        __syncthreads();
        cur ^= 1;
    }
    return cur;
}

template <typename T>
struct SmoothTileArgs {
    DevLevel L;
    DevTable<T> relax;
    int ncls;
    const T* xin;
    const T* b;
    T* xout;
    T two3;
    int h;
    DevLevel Cl;
    DevTransfer<T> tr;
    int half;            // both axes halve: the tile's coarse values are staged in LDS
    const T* xc;
    double* xacc;
};

// Up to kMaxFuse sweeps of one level.  PROLONG adds P x_c to every loaded
// node first (k_prolong_add's arithmetic), fusing the coarse-grid correction
// with the post-sweeps; ACC adds the result into an FP64 iterate (the mixed
// refinement's x += e, fused into the last level-0 sweep).
template <typename T, bool COMPACT, bool PROLONG, bool ACC, bool SMALL>
__device__ __forceinline__ void smooth_tile_body(const SmoothTileArgs<T>& A, unsigned bid)
{
    using G = TileGeom<T, SMALL>;
    constexpr int RPT = G::rpt;
    constexpr int CW = G::cw, CH = G::ch;   // staged coarse values
    const DevLevel& L = A.L;
    const DevTable<T>& relax = A.relax;
    const int h = A.h;
    const DevLevel& Cl = A.Cl;
    const DevTransfer<T>& tr = A.tr;
    const T* __restrict__ xc = A.xc;
    __shared__ T sx[2][G::plane];
    __shared__ T ctab[kMaxClsLds * 9];
    __shared__ T sxc[PROLONG ? CW * CH : 1];
    const int tx = threadIdx.x & (kTileX - 1), ty = threadIdx.x / kTileX, i0 = ty * RPT;
    const int n0 = L.n[0], n1 = L.n[1];
    const int ostep = kTileX - 2 * h;
    const int ntc = (n1 + ostep - 1) / ostep;
    const int t0 = (int)(bid / ntc) * G::rows, t1 = (int)(bid % ntc) * ostep;
    const int R = G::rows + 2 * h;
    const bool lds_tab = A.ncls <= kMaxClsLds;
    // coordinates first, then every load in one straight run (a load under a
    // condition is waited for where the paths join); rows beyond the tile
    // repeat its last.  Waves of large FP64 tiles without a row (2 of 8 with
    // one sweep) load none: those launches are bound by these loads (walls,
    // 2049^2: 237 -> 230 us a cycle).  In FP32 and in small tiles they are
    // not, and the branch costs more (1024^2 FP32 3 us a cycle)
    const int g1 = tile_coord(t1 - h + tx, n1, L.wrap[1]);
    int g0[RPT];
#pragma unroll
    for (int k = 0; k < RPT; ++k) g0[k] = tile_coord(t0 - h + min(i0 + k, R - 1), n0, L.wrap[0]);
    // coarse rows and columns lo .. lo + CH - 1, CW - 1 hold every value the
    // tile interpolates from when both axes halve
    const int lo0 = (t0 - h) >> 1, lo1 = (t1 - h) >> 1;
    const bool staged = PROLONG && A.half;
    int64_t ic[G::xc_per];
    if (staged)
#pragma unroll
        for (int k = 0; k < G::xc_per; ++k) {
            const int i = threadIdx.x + k * G::threads;
            const int r = i / CW, q = i - r * CW;
            ic[k] = (int64_t)tile_coord(lo0 + min(r, CH - 1), Cl.n[0], tr.wrap[0]) * Cl.n[1] +
                    tile_coord(lo1 + q, Cl.n[1], tr.wrap[1]);
        }
    T tab[G::tab_per], cv[G::xc_per];
    if (staged)
#pragma unroll
        for (int k = 0; k < G::xc_per; ++k) cv[k] = xc[ic[k]];
    if (lds_tab) tab_load<SMALL>(relax.coef, A.ncls * 9, tab);
    T breg[RPT], xv[RPT];
    int creg[RPT] = {};      // (waves that load no row index the tables with it)
    double xa[RPT];
    int p0[RPT], p1 = 0;
    T w0[RPT][2], w1[2] = {(T)0, (T)0};
    if (PROLONG) {
        p1 = tr.pc[1][g1];
        w1[0] = tr.pw[1][2 * g1];
        w1[1] = tr.pw[1][2 * g1 + 1];
    }
    const int g1o = t1 + tx - h;
    const bool colout = tx >= h && tx < kTileX - h && g1o < n1;
    if (SMALL || sizeof(T) == 4 || i0 < R)
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const int64_t gi = (int64_t)g0[k] * n1 + g1;
            xv[k] = A.xin[gi];
            breg[k] = A.b[gi];
            creg[k] = L.cls[gi];
            if (PROLONG) {
                p0[k] = tr.pc[0][g0[k]];
                w0[k][0] = tr.pw[0][2 * g0[k]];
                w0[k][1] = tr.pw[0][2 * g0[k] + 1];
            }
            if (ACC) xa[k] = A.xacc[gi];
        }
    if (lds_tab) tab_store<SMALL>(ctab, A.ncls * 9, tab);
    if (PROLONG) {
        if (staged) {
#pragma unroll
            for (int k = 0; k < G::xc_per; ++k) {
                const int i = threadIdx.x + k * G::threads;
                if (i < CW * CH) sxc[i] = cv[k];
            }
            __syncthreads();
        }
        int q1[2];
        if (staged) {
            q1[0] = (tr.wrap[1] ? (t1 - h + tx) >> 1 : p1) - lo1;
            q1[1] = q1[0] + 1;
        } else {
            q1[0] = wrap_index(p1, Cl.n[1], tr.wrap[1]);
            q1[1] = wrap_index(p1 + 1, Cl.n[1], tr.wrap[1]);
        }
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const int i = i0 + k;
            if (i >= R) continue;
            // k_prolong_add's sum: a over the row factor, b over the column factor
            const int r0 = (tr.wrap[0] ? (t0 - h + i) >> 1 : p0[k]) - lo0;
            T s = (T)0;
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                if (w0[k][a] == (T)0) continue;
                const int j0 = staged ? 0 : wrap_index(p0[k] + a, Cl.n[0], tr.wrap[0]);
#pragma unroll
                for (int bb = 0; bb < 2; ++bb) {
                    if (w1[bb] == (T)0) continue;
                    const T v = staged ? sxc[(r0 + a) * CW + q1[bb]] : xc[(int64_t)j0 * Cl.n[1] + q1[bb]];
                    s = s + (w0[k][a] * w1[bb]) * v;
                }
            }
            xv[k] = s * (T)1 + xv[k] * (T)1;
        }
    }
#pragma unroll
    for (int k = 0; k < RPT; ++k)
        if (i0 + k < R) sx[0][G::at(i0 + k, tx)] = xv[k];
    __syncthreads();
    TileRow<T, COMPACT> rows[RPT];
#pragma unroll
    for (int k = 0; k < RPT; ++k) rows[k].load(lds_tab ? &ctab[creg[k] * 9] : relax.coef + (int64_t)creg[k] * 9);
    const int cur = tile_sweeps<T, COMPACT, SMALL>(sx, tx, i0, R, h, breg, A.two3, [&](int k) { return rows[k]; });
    if (!colout) return;
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        const int i = i0 + k;
        const int g0 = t0 + i - h;
        if (i < h || i >= h + G::rows || g0 >= n0) continue;
        const int64_t gi = (int64_t)g0 * n1 + g1o;
        const T v = sx[cur][G::at(i, tx)];
        A.xout[gi] = v;
        if (ACC) A.xacc[gi] = xa[k] + (double)v;
    }
}

template <typename T, bool COMPACT, bool PROLONG, bool ACC, bool SMALL>
__global__ __launch_bounds__((TileGeom<T, SMALL>::threads)) void k_smooth_tile(SmoothTileArgs<T> a)
{
    smooth_tile_body<T, COMPACT, PROLONG, ACC, SMALL>(a, blockIdx.x);
}

template <typename T, bool COMPACT, bool PROLONG, bool ACC>
__global__ __launch_bounds__((TileGeom<T, false>::threads)) void k_smooth_tile_many(const SmoothTileArgs<T>* __restrict__ a,
                                                                               const unsigned* __restrict__ first, int n)
{
    const int i = batch_instance(first, n);
    smooth_tile_body<T, COMPACT, PROLONG, ACC, false>(a[i], blockIdx.x - first[i]);
}

template <typename T>
struct ResidRestrictArgs {
    DevLevel F, Cl;
    DevTransfer<T> tr;
    DevTable<T> Af;
    int ncls;
    DevTable<T> Ac;
    const T* x;
    const T* bf;
    T* bc;
    T* xc;
    T first_sweep;
};

// The downward half of a level in one launch (2D): h = 0 .. kMaxFuse last
// pre-sweeps, the residual, its restriction.  A block restricts to crows x CC
// coarse nodes (CC from h, so that their fine support, the residual's and
// the sweeps' halos fit 64 columns); it stores the swept iterate on the fine
// nodes of its tile (h > 0), evaluates the residuals of the support in LDS
// (k_residual's arithmetic), and one thread sums each coarse node's support
// (k_restrict's order).  The fine support of coarse nodes lo..hi-1 lies in
// [st lo - (st - 1), st (hi - 1) + st - 1], st = 2 on a halved axis and 1 on
// one kept as it is (the host checks the transfer tables, down_fits()).
template <typename T>
struct DownTileArgs {
    ResidRestrictArgs<T> r;
    DevTable<T> relax;
    T* xout;
    T two3;
    int h;
    int st[2];
};

__host__ __device__ inline int down_cols(int h, int st) { return (kTileX - 2 - 2 * h - (st - 1)) / st; }

template <typename T, bool COMPACT, bool SMALL>
__device__ __forceinline__ void down_tile_body(const DownTileArgs<T>& A, unsigned bid)
{
    using G = TileGeom<T, SMALL>;
    constexpr int RPT = G::rpt;
    const DevLevel& F = A.r.F;
    const DevLevel& Cl = A.r.Cl;
    const DevTransfer<T>& tr = A.r.tr;
    const int h = A.h;
    __shared__ T sx[2][G::plane];
    __shared__ T rtab[kMaxClsLds * 9], atab[kMaxClsLds * 9];
    const int CC = down_cols(h, A.st[1]);
    const int ntc = (Cl.n[1] + CC - 1) / CC;
    const int c0lo = (int)(bid / ntc) * G::crows, c1lo = (int)(bid % ntc) * CC;
    const int c0hi = min(c0lo + G::crows, Cl.n[0]), c1hi = min(c1lo + CC, Cl.n[1]);
    // fine coordinates (before wrapping) of the tile's first row and column
    const int u0 = A.st[0] * c0lo - A.st[0] - h, u1 = A.st[1] * c1lo - A.st[1] - h;
    const int R = A.st[0] * (c0hi - c0lo) + (A.st[0] - 1) + 2 + 2 * h;
    const int W = A.st[1] * (c1hi - c1lo) + (A.st[1] - 1) + 2 + 2 * h;
    const bool lds_tab = A.r.ncls <= kMaxClsLds;
    const int tx = threadIdx.x & (kTileX - 1), ty = threadIdx.x / kTileX, i0 = ty * RPT;
    const int n0 = F.n[0], n1 = F.n[1];
    // as in smooth_tile_body: coordinates, then the loads in one run
    const int g1 = tile_coord(u1 + tx, n1, F.wrap[1]);
    int g0[RPT];
#pragma unroll
    for (int k = 0; k < RPT; ++k) g0[k] = tile_coord(u0 + min(i0 + k, R - 1), n0, F.wrap[0]);
    T ta[G::tab_per], tb[G::tab_per];
    if (lds_tab) {
        tab_load<SMALL>(A.r.Af.coef, A.r.ncls * 9, ta);
        tab_load<SMALL>(A.relax.coef, A.r.ncls * 9, tb);
    }
    T breg[RPT], xv[RPT];
    int creg[RPT] = {};      // (waves that load no row index the tables with it)
    if (SMALL || sizeof(T) == 4 || i0 < R)
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const int64_t gi = (int64_t)g0[k] * n1 + g1;
            xv[k] = A.r.x[gi];
            breg[k] = A.r.bf[gi];
            creg[k] = F.cls[gi];
        }
    // the coarse node this thread sums: its support and weights
    const int c0 = c0lo + ty, c1 = c1lo + tx;
    const bool coarse = ty < G::crows && tx < CC && c0 < c0hi && c1 < c1hi;
    const int c0r = min(c0, Cl.n[0] - 1), c1r = min(c1, Cl.n[1] - 1);
    const int f0 = tr.rf[0][c0r], m0 = tr.rn[0][c0r], f1 = tr.rf[1][c1r], m1 = tr.rn[1][c1r];
    T rw0[3], rw1[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        rw0[q] = tr.rw[0][3 * c0r + q];
        rw1[q] = tr.rw[1][3 * c1r + q];
    }
    const int cc = Cl.cls[(int64_t)c0r * Cl.n[1] + c1r];
    if (lds_tab) {
        tab_store<SMALL>(atab, A.r.ncls * 9, ta);
        tab_store<SMALL>(rtab, A.r.ncls * 9, tb);
    }
#pragma unroll
    for (int k = 0; k < RPT; ++k)
        if (i0 + k < R) sx[0][G::at(i0 + k, tx)] = xv[k];
    const T dinv = A.r.Ac.dinv[cc];
    __syncthreads();
    auto row_of = [&](const T* lds, const T* coef, int k) {
        TileRow<T, COMPACT> r;
        r.load(lds_tab ? lds + creg[k] * 9 : coef + (int64_t)creg[k] * 9);
        return r;
    };
    int cur = 0;
    if (h > 0) {
        TileRow<T, COMPACT> rows[RPT];
#pragma unroll
        for (int k = 0; k < RPT; ++k) rows[k] = row_of(rtab, A.relax.coef, k);
        cur = tile_sweeps<T, COMPACT, SMALL>(sx, tx, i0, R, h, breg, A.two3, [&](int k) { return rows[k]; });
        // the tile's own fine nodes
        const int e0 = c0hi == Cl.n[0] ? n0 : A.st[0] * c0hi, e1 = c1hi == Cl.n[1] ? n1 : A.st[1] * c1hi;
        const int o1 = u1 + tx;
        if (o1 >= A.st[1] * c1lo && o1 < e1)
#pragma unroll
            for (int k = 0; k < RPT; ++k) {
                const int o0 = u0 + i0 + k;
                if (o0 >= A.st[0] * c0lo && o0 < e0)
                    A.xout[(int64_t)o0 * n1 + o1] = sx[cur][G::at(i0 + k, tx)];
            }
    }
    // residuals on the support, into the other plane
    {
        const bool colok = tx >= h + 1 && tx < W - h - 1;
        T* rn = &sx[cur ^ 1][G::at(i0, tx)];
        tile_stencil<T, COMPACT, SMALL>(&sx[cur][G::at(i0 - 1, tx)], [&](int k) { return row_of(atab, A.r.Af.coef, k); },
                                        [&](int k, T t) {
            const int i = i0 + k;
            if (colok && i >= h + 1 && i < R - h - 1) rn[k * kTileX] = t * (T)-1 + breg[k] * (T)1;
        });
    }
    __syncthreads();
    if (!coarse) return;
    const T* sr = &sx[cur ^ 1][G::at(f0 - u0, f1 - u1)];
    T s = (T)0;
#pragma unroll
    for (int a = 0; a < 3; ++a)
        if (a < m0)
#pragma unroll
            for (int b = 0; b < 3; ++b)
                if (b < m1) s = s + (rw0[a] * rw1[b]) * sr[a * kTileX + b];
    const int64_t ci = (int64_t)c0 * Cl.n[1] + c1;
    const T bv = s * dinv;
    A.r.bc[ci] = bv;
    A.r.xc[ci] = A.r.first_sweep != (T)0 ? bv * (A.r.first_sweep * (T)1) : (T)0;
}

template <typename T, bool COMPACT, bool SMALL>
__global__ __launch_bounds__((TileGeom<T, SMALL>::threads)) void k_down_tile(DownTileArgs<T> a)
{
    down_tile_body<T, COMPACT, SMALL>(a, blockIdx.x);
}

template <typename T, bool COMPACT>
__global__ __launch_bounds__((TileGeom<T, false>::threads)) void k_down_tile_many(const DownTileArgs<T>* __restrict__ a,
                                                                             const unsigned* __restrict__ first, int n)
{
    const int i = batch_instance(first, n);
    down_tile_body<T, COMPACT, false>(a[i], blockIdx.x - first[i]);
}

// k_residual fused into k_restrict (2D): the restriction evaluates the fine
// residual b - A^ x at each of its fine support nodes with k_residual's
// arithmetic instead of reading a stored residual.
template <typename T, bool COMPACT>
__device__ __forceinline__ void resid_restrict_body(const ResidRestrictArgs<T>& A, unsigned bid)
{
    const DevLevel& F = A.F;
    const DevLevel& Cl = A.Cl;
    const DevTransfer<T>& tr = A.tr;
    const DevTable<T>& Af = A.Af;
    const DevTable<T>& Ac = A.Ac;
    const T* __restrict__ x = A.x;
    const T* __restrict__ bf = A.bf;
    T* __restrict__ bc = A.bc;
    T* __restrict__ xc = A.xc;
    const T first_sweep = A.first_sweep;
    const int64_t i = (int64_t)bid * kMgThreads + threadIdx.x;
    if (i >= Cl.N) return;
    int c[3];
    node_coords<2>(Cl, i, c);
    T s = (T)0;
    const int f0 = tr.rf[0][c[0]], m0 = tr.rn[0][c[0]];
    const int f1 = tr.rf[1][c[1]], m1 = tr.rn[1][c[1]];
    for (int a = 0; a < m0; ++a) {
        const T w0 = tr.rw[0][3 * c[0] + a];
        const int i0 = wrap_index(f0 + a, F.n[0], tr.wrap[0]);
        for (int b = 0; b < m1; ++b) {
            const T w = w0 * tr.rw[1][3 * c[1] + b];
            const int i1 = wrap_index(f1 + b, F.n[1], tr.wrap[1]);
            const int64_t fi = (int64_t)i0 * F.n[1] + i1;
            const int fc[3] = {i0, i1, 0};
            const T t = stencil_apply<T, 2, COMPACT>(F, Af.coef + (int64_t)F.cls[fi] * 9, x, fc);
            const T r = t * (T)-1 + bf[fi] * (T)1;
            s = s + w * r;
        }
    }
    const T bv = s * Ac.dinv[Cl.cls[i]];
    bc[i] = bv;
    xc[i] = first_sweep != (T)0 ? bv * (first_sweep * (T)1) : (T)0;
}

template <typename T, bool COMPACT>
__global__ __launch_bounds__(kMgThreads) void k_resid_restrict(ResidRestrictArgs<T> a)
{
    resid_restrict_body<T, COMPACT>(a, blockIdx.x);
}

template <typename T, bool COMPACT>
__global__ __launch_bounds__(kMgThreads) void k_resid_restrict_many(const ResidRestrictArgs<T>* __restrict__ a,
                                                                    const unsigned* __restrict__ first, int n)
{
    const int i = batch_instance(first, n);
    resid_restrict_body<T, COMPACT>(a[i], blockIdx.x - first[i]);
}

// b0 = b o D0^-1  (hadamard_to)
template <typename T>
struct HadamardArgs {
    DevLevel L;
    DevTable<T> A;
    const T* b;
    T* out;
};

template <typename T>
__device__ __forceinline__ void hadamard_body(const HadamardArgs<T>& a, unsigned bid)
{
    const int64_t i = (int64_t)bid * kMgThreads + threadIdx.x;
    if (i < a.L.N) a.out[i] = a.b[i] * a.A.dinv[a.L.cls[i]];
}

template <typename T>
__global__ __launch_bounds__(kMgThreads) void k_hadamard(HadamardArgs<T> a)
{
    hadamard_body<T>(a, blockIdx.x);
}

template <typename T>
__global__ __launch_bounds__(kMgThreads) void k_hadamard_many(const HadamardArgs<T>* __restrict__ a,
                                                              const unsigned* __restrict__ first, int n)
{
    const int i = batch_instance(first, n);
    hadamard_body<T>(a[i], blockIdx.x - first[i]);
}

// x = M b with the dense coarse-end operator M (row-major, rows padded to ld
// values; M is the V-cycle from the level down, or the coarsest inverse): one
// wave per row, 16-byte loads of the row, products summed in FP64 in a fixed
// order (lane partials, then a butterfly).  Bound by reading M: up to the
// 32 MB of the eight L2s (a block's rows stay on its XCD from launch to
// launch) n = 1024 takes 2.6 us and 2025 4.3 us, launch included; beyond it
// the Infinity Cache gives about 6 TB/s (2856: 11 us, 4913: 28 us).  Two or
// four rows per wave, or a block per row pair, were no faster.  M is FP64 for
// FP32 vectors too, as the coarsest inverse is: in FP32 it would be read in
// half the time, but where the terms of a row cancel (the singular system of
// a periodic box, a pair of far charges) a V-cycle's error grew from 1.0e-7
// to 3.7e-7.  b holds ld values (zeros beyond n).
template <typename T>
struct CoarseArgs {
    const double* op;
    int n, ld;
    const T* b;
    T* x;
};

template <typename T>
__device__ __forceinline__ void coarse_solve_body(const CoarseArgs<T>& a, unsigned bid)
{
    constexpr int V = 2;
    typedef double vec __attribute__((ext_vector_type(2)));
    const int row = (int)(((int64_t)bid * kMgThreads + threadIdx.x) >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= a.n) return;
    const double* __restrict__ m = a.op + (int64_t)row * a.ld;
    const T* __restrict__ b = a.b;
    double s = 0.0;
#pragma unroll 4
    for (int j = lane * V; j < a.ld; j += 64 * V) {
        const vec v = *reinterpret_cast<const vec*>(m + j);
#pragma unroll
        for (int k = 0; k < V; ++k) s += v[k] * (double)b[j + k];
    }
    s = wave_sum_full(s);
    if (lane == 0) a.x[row] = (T)s;
}

template <typename T>
__global__ __launch_bounds__(kMgThreads) void k_coarse_solve(CoarseArgs<T> a)
{
    coarse_solve_body<T>(a, blockIdx.x);
}

template <typename T>
__global__ __launch_bounds__(kMgThreads) void k_coarse_solve_many(const CoarseArgs<T>* __restrict__ a,
                                                                  const unsigned* __restrict__ first, int n)
{
    const int i = batch_instance(first, n);
    coarse_solve_body<T>(a[i], blockIdx.x - first[i]);
}

// ---- building the dense coarse-end operator --------------------------------
// The V-cycle from level l down, started from zero, is linear in its
// right-hand side: its matrix is built column by column in FP64 with the
// level kernels' terms.  An N x N matrix of columns is stored row-major, so
// row i holds node i's value in every column; blockIdx.y is the row (its
// class and neighbours are uniform), threads run over the columns.

// Y = beta (coef X) + gamma I  (X == nullptr: X = 0)
template <int D>
__global__ __launch_bounds__(kMgThreads) void k_dense_stencil(DevLevel L, const double* __restrict__ coef,
                                                              const double* __restrict__ X, double* __restrict__ Y,
                                                              double beta, double gamma)
{
    const int j = (int)(blockIdx.x * kMgThreads + threadIdx.x);
    const int64_t i = blockIdx.y, N = L.N;
    if (j >= N) return;
    constexpr int KS = D == 2 ? 9 : 27;
    double s = 0.0;
    if (X) {
        int c[3] = {0, 0, 0};
        node_coords<D>(L, i, c);
        const double* row = coef + (int64_t)L.cls[i] * KS;
        for (int k = 0; k < KS; ++k) {
            const double v = row[k];
            if (v == 0.0) continue;
            const int o[3] = {D == 2 ? k / 3 - 1 : k / 9 - 1, D == 2 ? k % 3 - 1 : (k / 3) % 3 - 1, D == 2 ? 0 : k % 3 - 1};
            int64_t q = 0;
            for (int d = 0; d < D; ++d) q = q * L.n[d] + nb_index(c[d], o[d], L.n[d], L.wrap[d]);
            s = s + v * X[q * N + j];
        }
    }
    Y[i * N + j] = beta * s + (i == j ? gamma : 0.0);
}

// B = (R r) o D_c^-1 for every column
template <int D>
__global__ __launch_bounds__(kMgThreads) void k_dense_restrict(DevLevel F, DevLevel Cl, DevTransfer<double> tr,
                                                               const double* __restrict__ dinv,
                                                               const double* __restrict__ r, double* __restrict__ B)
{
    const int j = (int)(blockIdx.x * kMgThreads + threadIdx.x);
    const int64_t i = blockIdx.y, N = F.N;
    if (j >= N) return;
    int c[3] = {0, 0, 0};
    node_coords<D>(Cl, i, c);
    double s = 0.0;
    for (int a = 0; a < tr.rn[0][c[0]]; ++a)
        for (int b = 0; b < tr.rn[1][c[1]]; ++b)
            for (int e = 0; e < (D == 3 ? tr.rn[2][c[2]] : 1); ++e) {
                double w = tr.rw[0][3 * c[0] + a] * tr.rw[1][3 * c[1] + b];
                int64_t q = (int64_t)wrap_index(tr.rf[0][c[0]] + a, F.n[0], tr.wrap[0]) * F.n[1] +
                            wrap_index(tr.rf[1][c[1]] + b, F.n[1], tr.wrap[1]);
                if (D == 3) {
                    w = w * tr.rw[2][3 * c[2] + e];
                    q = q * F.n[2] + wrap_index(tr.rf[2][c[2]] + e, F.n[2], tr.wrap[2]);
                }
                s = s + w * r[q * N + j];
            }
    B[i * N + j] = s * dinv[Cl.cls[i]];
}

// X += P E for every column
template <int D>
__global__ __launch_bounds__(kMgThreads) void k_dense_prolong(DevLevel F, DevLevel Cl, DevTransfer<double> tr,
                                                              const double* __restrict__ E, double* __restrict__ X)
{
    const int j = (int)(blockIdx.x * kMgThreads + threadIdx.x);
    const int64_t i = blockIdx.y, N = F.N;
    if (j >= N) return;
    int c[3] = {0, 0, 0};
    node_coords<D>(F, i, c);
    double s = 0.0;
    for (int h = 0; h < (1 << D); ++h) {
        double w = 1.0;
        int64_t q = 0;
        for (int d = 0; d < D; ++d) {
            const int o = (h >> (D - 1 - d)) & 1;
            const double f = tr.pw[d][2 * c[d] + o];
            w = w * f;
            // a zero weight's node may lie outside the axis: not read
            q = q * Cl.n[d] + (f == 0.0 ? 0 : wrap_index(tr.pc[d][c[d]] + o, Cl.n[d], tr.wrap[d]));
        }
        if (w != 0.0) s = s + w * E[q * N + j];
    }
    X[i * N + j] += s;
}

// E (m x n) = A (m x m) B (m x n), 32 x 32 tiles through LDS, FP64
__global__ __launch_bounds__(kMgThreads) void k_dense_product(int m, int n, const double* __restrict__ A,
                                                              const double* __restrict__ B, double* __restrict__ E)
{
    __shared__ double sa[32][33], sb[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;     // 32 x 8
    const int r0 = (int)blockIdx.y * 32, c0 = (int)blockIdx.x * 32;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < m; k0 += 32) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = ty + 8 * q;
            sa[r][tx] = (r0 + r < m && k0 + tx < m) ? A[(int64_t)(r0 + r) * m + k0 + tx] : 0.0;
            sb[r][tx] = (k0 + r < m && c0 + tx < n) ? B[(int64_t)(k0 + r) * n + c0 + tx] : 0.0;
        }
        __syncthreads();
        for (int k = 0; k < 32; ++k)
#pragma unroll
            for (int q = 0; q < 4; ++q) s[q] += sa[ty + 8 * q][k] * sb[k][tx];
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (r0 + ty + 8 * q < m && c0 + tx < n) E[(int64_t)(r0 + ty + 8 * q) * n + c0 + tx] = s[q];
}

// rows of n values -> rows of ld values, zeros beyond n
__global__ __launch_bounds__(kMgThreads) void k_dense_pad(int n, int ld, const double* __restrict__ A, double* __restrict__ out)
{
    const int j = (int)(blockIdx.x * kMgThreads + threadIdx.x);
    if (j < ld) out[(int64_t)blockIdx.y * ld + j] = j < n ? A[(int64_t)blockIdx.y * n + j] : 0.0;
}

// FP64 residual of the unscaled operator: r = b - A x, partial sums of r^2
// and of b^2 per block; when OUTF32 also emit (float)r o D0^-1 (the mixed
// backend's residual_to + hadamard_to).
// FP64 residual r = b - A x of the unscaled level-0 operator; partial sums
// of r^2 (skipping row `pin` of a pinned-periodic system, which the gauge
// shift satisfies exactly) and of bn^2 (the caller's right-hand side).
struct OuterArgs {
    DevLevel L;
    DevTable<double> K;
    const double* x;
    const double* b;
    const double* bn;
    int64_t pin;
    const float* dinv32;
    float* b0;
    double* part;
    float* e0;
    // 3D 7-point level 0: the dominant class and its row (K.coef +
    // cls_in * 27), read as uniform values; -1: every node reads its row
    int cls_in;
    const double* row_in;
};

template <int D, bool COMPACT, bool OUTF32, bool NORMS>
__device__ __forceinline__ void outer_residual_body(const OuterArgs& A, int64_t blk)
{
    const DevLevel& L = A.L;
    const DevTable<double>& K = A.K;
    const double* __restrict__ x = A.x;
    const double* __restrict__ b = A.b;
    const double* __restrict__ bn = A.bn;
    const int64_t pin = A.pin;
    const float* __restrict__ dinv32 = A.dinv32;
    float* __restrict__ b0 = A.b0;
    double* __restrict__ part = A.part;
    float* __restrict__ e0 = A.e0;
    __shared__ double ws[kMgThreads / 64][2];
    const int64_t i = blk * kMgThreads + threadIdx.x;
    double rr = 0.0, bb = 0.0;
    if (i < L.N) {
        int c[3];
        node_coords<D>(L, i, c);
        const uint16_t ci = L.cls[i];
        double ax;
        if (D == 3 && COMPACT && (int)ci == A.cls_in) {
            ax = stencil_apply<double, D, COMPACT>(L, A.row_in, x, c);
        } else {
            const double* coef = K.coef + (int64_t)ci * (D == 2 ? 9 : 27);
            ax = stencil_apply<double, D, COMPACT>(L, coef, x, c);
        }
        const double r = b[i] - ax;
        if (NORMS) {
            rr = i == pin ? 0.0 : r * r;
            bb = bn[i] * bn[i];
        }
        if (OUTF32) {
            const float bv = (float)r * dinv32[L.cls[i]];
            b0[i] = bv;
            // first Jacobi sweep of the correction from e = 0: relax*0 + b*(2/3)
            if (e0) e0[i] = bv * (2.0f / 3.0f * 1.0f);
        }
    }
    if (!NORMS) return;
    rr = wave_sum(rr);
    bb = wave_sum(bb);
    if ((threadIdx.x & 63) == 0) {
        ws[threadIdx.x >> 6][0] = rr;
        ws[threadIdx.x >> 6][1] = bb;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double s = 0.0;
        for (int w = 0; w < kMgThreads / 64; ++w) s += ws[w][threadIdx.x];
        part[2 * blk + threadIdx.x] = s;
    }
}

template <int D, bool COMPACT, bool OUTF32, bool NORMS>
__global__ __launch_bounds__(kMgThreads) void k_outer_residual(OuterArgs a)
{
    outer_residual_body<D, COMPACT, OUTF32, NORMS>(a, level_block<D>());
}

template <int D, bool COMPACT, bool OUTF32, bool NORMS>
__global__ __launch_bounds__(kMgThreads) void k_outer_residual_many(const OuterArgs* __restrict__ a,
                                                                    const unsigned* __restrict__ first, int n)
{
    const int i = batch_instance(first, n);
    outer_residual_body<D, COMPACT, OUTF32, NORMS>(a[i], (int64_t)(blockIdx.x - first[i]));
}

// The outer residual without norms on a chunked 7-point 3D level: the
// FP32 right-hand side (and first sweep) of outer_residual_body at the
// chunk kernels' nodes (line_apply in FP64 over the unscaled class row),
// the listed nodes one per thread; same terms and order, same bits.
__device__ __forceinline__ void outer_node_f32(const OuterArgs& A, int64_t i)
{
    const DevLevel& L = A.L;
    int c[3];
    node_coords<3>(L, i, c);
    const double* coef = A.K.coef + (int64_t)L.cls[i] * 27;
    const double ax = stencil_apply<double, 3, true>(L, coef, A.x, c);
    const double r = A.b[i] - ax;
    const float bv = (float)r * A.dinv32[L.cls[i]];
    A.b0[i] = bv;
    if (A.e0) A.e0[i] = bv * (2.0f / 3.0f * 1.0f);
}

__global__ __launch_bounds__(kMgThreads) void k_outer_line(LineGeom G, LineList LL, OuterArgs A,
                                                           const double* __restrict__ row, float dinv_in)
{
    bool listed;
    const int64_t blk = line_block(LL, &listed);
    if (blk < 0) return;
    if (listed) {
        const int64_t t = blk * kMgThreads + threadIdx.x;
        if (t < (int64_t)LL.n) outer_node_f32(A, (int64_t)LL.list[t]);
        return;
    }
    const int64_t t = blk * kMgThreads + threadIdx.x;
    if (t >= (int64_t)G.nchunks) return;
    const uint32_t i = (uint32_t)t * kLine;
    if (!line_chunk_fast(G, i)) return;
    double ax[kLine], bb[kLine];
    line_apply<double, true>(G, row, A.x, i, ax);
    ld_line(A.b + i, bb);
    float bv[kLine], e[kLine];
#pragma unroll
    for (int k = 0; k < kLine; ++k) {
        const double r = bb[k] - ax[k];
        bv[k] = (float)r * dinv_in;
        e[k] = bv[k] * (2.0f / 3.0f * 1.0f);
    }
    st_line(A.b0 + i, bv);
    if (A.e0) st_line(A.e0 + i, e);
}

// Squared norms of a residual and its right-hand side in pinned host memory.
// The kernel that sums them stores them there and then, at system scope, the
// number of norms stored so far (kept in *count on the device), which the host
// waits for: a copy and a stream synchronisation after it left the GPU idle
// for 25 us per check of a small problem.
struct NormBox {
    double rr, bb;
    unsigned long long seq;
};

// (x non-null: also shift = x_pin - bn_pin, the gauge of a pinned system)
__global__ __launch_bounds__(kMgThreads) void k_reduce2(const double* __restrict__ part, int64_t nb,
                                                        NormBox* __restrict__ box,
                                                        unsigned long long* __restrict__ count,
                                                        const double* __restrict__ x,
                                                        const double* __restrict__ bn, int64_t pin,
                                                        double* __restrict__ shift)
{
    if (x && threadIdx.x == 2) shift[0] = x[pin] - bn[pin];
    __shared__ double sh[2][kMgThreads];
    double s0 = 0.0, s1 = 0.0;
    // thread t sums pairs 8t .. 8t+7, then 8(t + 256) .., in order; the eight
    // pairs of a round are loaded before they are added
    constexpr int kU = 8;
    for (int64_t b0 = (int64_t)threadIdx.x * kU; b0 < nb; b0 += (int64_t)kMgThreads * kU) {
        double v[2 * kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const bool in = b0 + u < nb;
            v[2 * u] = in ? part[2 * (b0 + u)] : 0.0;
            v[2 * u + 1] = in ? part[2 * (b0 + u) + 1] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            s0 += v[2 * u];
            s1 += v[2 * u + 1];
        }
    }
    sh[0][threadIdx.x] = s0;
    sh[1][threadIdx.x] = s1;
    __syncthreads();
    for (int w = kMgThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + w];
            sh[1][threadIdx.x] += sh[1][threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const unsigned long long c = *count + 1;
        *count = c;
        box->rr = sh[0][0];
        box->bb = sh[1][0];
        __threadfence_system();
        __hip_atomic_store(&box->seq, c, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// per-block sums of x (part[b]), then a fixed-order single-block total
__global__ __launch_bounds__(kMgThreads) void k_psum(const double* __restrict__ x, int64_t n,
                                                     double* __restrict__ part)
{
    __shared__ double ws[kMgThreads / 64];
    const int64_t i = (int64_t)blockIdx.x * kMgThreads + threadIdx.x;
    double v = wave_sum(i < n ? x[i] : 0.0);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < kMgThreads / 64; ++w) s += ws[w];
        part[blockIdx.x] = s;
    }
}

// the total of the block sums, in every thread of the block
__device__ __forceinline__ double block_fsum(const double* __restrict__ part, int64_t nb)
{
    __shared__ double sh[kMgThreads];
    double s = 0.0;
    for (int64_t b = threadIdx.x; b < nb; b += kMgThreads) s += part[b];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = kMgThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    return sh[0];
}

__global__ __launch_bounds__(kMgThreads) void k_fsum(const double* __restrict__ part, int64_t nb,
                                                     double* __restrict__ out)
{
    const double s = block_fsum(part, nb);
    if (threadIdx.x == 0) out[0] = s;
}

// The right-hand side of a pinned system in two launches: between the solves
// of small problems every launch costs its 5 us, and the eight that subtract
// the mean, replace, copy, sum (twice), set the pin and scale took a tenth of
// a 128^2 step.  k_pin_rhs: b (less the mean whose block sums are mean_part),
// replaced nodes set, copied to bp and, scaled by dinv, to b0 (FP64 cycles;
// null in the mixed solve), summed per block.  Every block adds the mean's
// sums itself, so there are at most kPinBlocks.  k_pin_set: the total, and the
// pin's entries.  Operations and orders are those of the single kernels.
constexpr unsigned kPinBlocks = 512;
constexpr int kPinReplace = 4;
struct PinArgs {
    double* b;
    int64_t n;
    const double* mean_part;
    const unsigned long long* idx;
    const double* val;
    int nrep, zero;
    double *bp, *part, *b0;
    const double* dinv;
    const uint16_t* cls;
    int64_t pin;
    double* sum;
};

__global__ __launch_bounds__(kMgThreads) void k_pin_rhs(PinArgs a)
{
    __shared__ double ws[kMgThreads / 64];
    const int64_t i = (int64_t)blockIdx.x * kMgThreads + threadIdx.x;
    double v = 0.0, dinv = 0.0;
    if (i < a.n) {
        v = a.b[i];
        if (a.b0) dinv = a.dinv[a.cls[i]];
    }
    if (a.mean_part) {
        const double mean = block_fsum(a.mean_part, gridDim.x) / (double)a.n;
        if (i < a.n) v = v - mean;
    }
    if (i < a.n) {
        for (int r = 0; r < a.nrep; ++r)
            if ((int64_t)a.idx[r] == i) v = a.zero ? 0.0 : a.val[r];
        a.b[i] = v;
        a.bp[i] = v;
        if (a.b0) a.b0[i] = v * dinv;
    }
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < kMgThreads / 64; ++w) s += ws[w];
        a.part[blockIdx.x] = s;
    }
}

__global__ __launch_bounds__(kMgThreads) void k_pin_set(PinArgs a, int64_t nb)
{
    const double s = block_fsum(a.part, nb);
    if (threadIdx.x == 0) {
        const double v = a.b[a.pin] - s;
        a.sum[0] = s;
        a.bp[a.pin] = v;
        if (a.b0) a.b0[a.pin] = v * a.dinv[a.cls[a.pin]];
    }
}

// b'_p = b_p - sum(b): the consistent right-hand side of the singular system
__global__ void k_set_pin(double* __restrict__ bp, const double* __restrict__ b,
                          const double* __restrict__ sum, int64_t p)
{
    if (threadIdx.x == 0) bp[p] = b[p] - sum[0];
}

// gauge: shift = x_p - b_p ; x -= shift
__global__ void k_gauge_read(const double* __restrict__ x, const double* __restrict__ b, int64_t p,
                             double* __restrict__ shift)
{
    if (threadIdx.x == 0) shift[0] = x[p] - b[p];
}

__global__ __launch_bounds__(kMgThreads) void k_gauge_apply(double* __restrict__ x, int64_t n,
                                                            const double* __restrict__ shift)
{
    const int64_t i = (int64_t)blockIdx.x * kMgThreads + threadIdx.x;
    if (i < n) x[i] = x[i] - shift[0];
}

// Element-wise level-0 vector operations: x = 0 (FP32), x += e (FP64 +=
// FP32) and x = y (FP64 copy).
struct VecArgs {
    void* x;
    const void* y;
    int64_t n;
};

template <int OP>
__device__ __forceinline__ void vec_body(const VecArgs& a, unsigned bid)
{
    const int64_t i = (int64_t)bid * kMgThreads + threadIdx.x;
    if (i >= a.n) return;
    if (OP == 0) static_cast<float*>(a.x)[i] = 0.0f;
    else if (OP == 1) static_cast<double*>(a.x)[i] += (double)static_cast<const float*>(a.y)[i];
    else static_cast<double*>(a.x)[i] = static_cast<const double*>(a.y)[i];
}

template <int OP>
__global__ __launch_bounds__(kMgThreads) void k_vec(VecArgs a)
{
    vec_body<OP>(a, blockIdx.x);
}

template <int OP>
__global__ __launch_bounds__(kMgThreads) void k_vec_many(const VecArgs* __restrict__ a,
                                                        const unsigned* __restrict__ first, int n)
{
    const int i = batch_instance(first, n);
    vec_body<OP>(a[i], blockIdx.x - first[i]);
}

__global__ __launch_bounds__(kMgThreads) void k_zero_f32(float* __restrict__ x, int64_t n)
{
    vec_body<0>(VecArgs{x, nullptr, n}, blockIdx.x);
}

__global__ __launch_bounds__(kMgThreads) void k_addback(double* __restrict__ b,
                                                        const unsigned long long* __restrict__ idx,
                                                        const double* __restrict__ v, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * kMgThreads + threadIdx.x;
    if (i < n) b[idx[i]] += v[i];
}

__global__ __launch_bounds__(kMgThreads) void k_replace(double* __restrict__ b,
                                                        const unsigned long long* __restrict__ idx,
                                                        const double* __restrict__ v, int64_t n,
                                                        int zero)
{
    const int64_t i = (int64_t)blockIdx.x * kMgThreads + threadIdx.x;
    if (i < n) b[idx[i]] = zero ? 0.0 : v[i];
}

inline unsigned nblk(int64_t n) { return (unsigned)((n + kMgThreads - 1) / kMgThreads); }

// ------------------------------------------------------------ host levels

struct Axis {
    std::vector<double> x;
};

Axis coarsen(const Axis& f)
{
    Axis c;
    for (size_t i = 0; i < f.x.size(); i += 2) c.x.push_back(f.x[i]);
    if (c.x.back() != f.x.back()) c.x.push_back(f.x.back());
    return c;
}

std::vector<double> volumes(const Axis& a)
{
    std::vector<double> w(a.x.size(), 1.0);
    if (a.x.size() == 1) return w;
    for (size_t i = 0; i < a.x.size(); ++i)
        w[i] = ((i ? a.x[i] - a.x[i - 1] : 0.0) + (i + 1 < a.x.size() ? a.x[i + 1] - a.x[i] : 0.0)) * 0.5;
    return w;
}

struct AxisTransfer {
    std::vector<int> pc;        // per fine f
    std::vector<double> pw;     // 2 per fine f (w_lo, w_hi); exact node: (1, 0)
    std::vector<int> rf, rn;    // per coarse c
    std::vector<double> rw;     // 3 per coarse c
    int wrap = 0;               // periodic axis: fine/coarse indices wrap
};

// Periodic axis of even length nf >= 4: coarse node c is fine node 2c; an odd
// fine node interpolates its two coarse neighbours (wrapping); volumes are
// uniform, so R = P^T / 2 = {1/4, 1/2, 1/4} around 2c.
AxisTransfer axis_transfer_periodic(int nf)
{
    AxisTransfer t;
    const int nc = nf / 2;
    t.wrap = 1;
    t.pc.resize(nf);
    t.pw.resize(2 * nf);
    for (int i = 0; i < nf; ++i) {
        if (i % 2 == 0) { t.pc[i] = i / 2; t.pw[2 * i] = 1.0; t.pw[2 * i + 1] = 0.0; }
        else { t.pc[i] = (i - 1) / 2; t.pw[2 * i] = 0.5; t.pw[2 * i + 1] = 0.5; }
    }
    t.rf.resize(nc);
    t.rn.assign(nc, 3);
    t.rw.resize(3 * nc);
    for (int c = 0; c < nc; ++c) {
        t.rf[c] = 2 * c - 1;
        t.rw[3 * c] = 0.25;
        t.rw[3 * c + 1] = 0.5;
        t.rw[3 * c + 2] = 0.25;
    }
    return t;
}

AxisTransfer axis_transfer_identity(int n, int wrap)
{
    AxisTransfer t;
    t.wrap = wrap;
    t.pc.resize(n);
    t.pw.assign(2 * n, 0.0);
    t.rf.resize(n);
    t.rn.assign(n, 1);
    t.rw.assign(3 * n, 0.0);
    for (int i = 0; i < n; ++i) {
        t.pc[i] = i;
        t.pw[2 * i] = 1.0;
        t.rf[i] = i;
        t.rw[3 * i] = 1.0;
    }
    return t;
}

AxisTransfer axis_transfer(const Axis& f, const Axis& c)
{
    AxisTransfer t;
    const int nf = (int)f.x.size(), nc = (int)c.x.size();
    t.pc.resize(nf);
    t.pw.resize(2 * nf);
    for (int i = 0; i < nf; ++i) {
        const double x = f.x[i];
        int hi = (int)(std::lower_bound(c.x.begin(), c.x.end(), x) - c.x.begin());
        if (hi >= nc) throw std::runtime_error("hip_multigrid: point outside coarse grid");
        if (c.x[hi] == x) {
            t.pc[i] = hi;
            t.pw[2 * i] = 1.0;
            t.pw[2 * i + 1] = 0.0;
        } else {
            if (hi == 0) throw std::runtime_error("hip_multigrid: point outside coarse grid");
            const double tt = (x - c.x[hi - 1]) / (c.x[hi] - c.x[hi - 1]);
            t.pc[i] = hi - 1;
            t.pw[2 * i] = 1.0 - tt;
            t.pw[2 * i + 1] = tt;
        }
    }
    const std::vector<double> vol = volumes(f);
    std::vector<double> cvol(nc, 0.0);
    for (int i = 0; i < nf; ++i) {
        cvol[t.pc[i]] += t.pw[2 * i] * vol[i];
        if (t.pw[2 * i + 1] != 0.0) cvol[t.pc[i] + 1] += t.pw[2 * i + 1] * vol[i];
    }
    t.rf.assign(nc, -1);
    t.rn.assign(nc, 0);
    t.rw.assign(3 * nc, 0.0);
    for (int i = 0; i < nf; ++i)
        for (int h = 0; h < 2; ++h) {
            const double p = t.pw[2 * i + h];
            if (p == 0.0) continue;
            const int cc = t.pc[i] + h;
            if (t.rf[cc] < 0) t.rf[cc] = i;
            const int k = i - t.rf[cc];
            if (k < 0 || k > 2) throw std::runtime_error("hip_multigrid: restriction support > 3");
            t.rw[3 * cc + k] = p * (vol[i] / cvol[cc]);
            t.rn[cc] = std::max(t.rn[cc], k + 1);
        }
    return t;
}

struct RowKey {
    const double* v;
    int ks;
};

struct HostLevel {
    int D = 2;
    int n[3] = {1, 1, 1};
    int wrap[3] = {0, 0, 0};
    int64_t N = 0;
    int KS = 9;
    bool compact = false;
    std::vector<uint16_t> cls;
    std::vector<double> K;     // unscaled class rows
    std::vector<double> dinv;  // per class
    std::vector<double> Ah;    // scaled rows
    std::vector<double> Rx;    // relax rows
};

// Dedupe rows (bitwise) into classes.  rows: N * KS doubles.
void classify(HostLevel& L, const std::vector<double>& rows)
{
    const int KS = L.KS;
    std::unordered_map<std::string, int> map;
    L.cls.resize(L.N);
    L.K.clear();
    for (int64_t i = 0; i < L.N; ++i) {
        std::string key(reinterpret_cast<const char*>(&rows[i * KS]), sizeof(double) * KS);
        auto it = map.find(key);
        int id;
        if (it == map.end()) {
            id = (int)map.size();
            if (id >= 65535) throw std::runtime_error("hip_multigrid: more than 65535 distinct stencil rows");
            map.emplace(std::move(key), id);
            L.K.insert(L.K.end(), rows.begin() + i * KS, rows.begin() + (i + 1) * KS);
        } else {
            id = it->second;
        }
        L.cls[i] = (uint16_t)id;
    }
    const int ncls = (int)map.size();
    const int center = (KS - 1) / 2;
    L.dinv.resize(ncls);
    L.Ah.resize((size_t)ncls * KS);
    L.Rx.resize((size_t)ncls * KS);
    L.compact = true;
    for (int c = 0; c < ncls; ++c) {
        const double diag = L.K[(size_t)c * KS + center];
        L.dinv[c] = 1 / diag;
        for (int k = 0; k < KS; ++k) {
            const double a = L.K[(size_t)c * KS + k] * L.dinv[c];
            L.Ah[(size_t)c * KS + k] = a;
            const double s = a * 2.0 / 3;
            L.Rx[(size_t)c * KS + k] = (k == center) ? 1.0 - s : 0.0 - s;
            if (a != 0.0) {
                int nz = 0;
                int kk = k;
                for (int d = 0; d < L.D; ++d) {
                    if (kk % 3 != 1) ++nz;
                    kk /= 3;
                }
                if (nz > 1) L.compact = false;
            }
        }
    }
}

// offset of column (cc) from row (rc) along an axis of n nodes; wrapped
// offsets flag the axis periodic.  Returns false if not a 3-point neighbour.
bool axis_offset(int rc, int cc, int n, int& off, int& wrapped)
{
    const int d = cc - rc;
    if (d >= -1 && d <= 1) {
        off = d;
        return true;
    }
    if (d == n - 1) {
        off = -1;
        wrapped = 1;
        return true;
    }
    if (d == -(n - 1)) {
        off = 1;
        wrapped = 1;
        return true;
    }
    return false;
}

inline int dims_n(const HostLevel& L, int d) { return L.n[d]; }

// Pinned-periodic detection on the level-0 rows (N x KS): every axis of
// size > 1 wrapped, exactly one identity row p, zero row sums elsewhere.
// Returns p, or -1.
int64_t detect_pinned_periodic(const HostLevel& L, const std::vector<double>& R)
{
    for (int d = 0; d < 3; ++d)
        if (L.n[d] > 1 && !L.wrap[d]) return -1;
    const int KS = L.KS, center = (KS - 1) / 2;
    int64_t pin = -1;
    for (int64_t i = 0; i < L.N; ++i) {
        const double* r = &R[(size_t)i * KS];
        bool ident = r[center] == 1.0;
        double s = 0.0, m = 0.0;
        for (int k = 0; k < KS; ++k) {
            if (k != center && r[k] != 0.0) ident = false;
            s += r[k];
            m += std::fabs(r[k]);
        }
        if (ident) {
            if (pin >= 0) return -1;
            pin = i;
        } else if (std::fabs(s) > 1e-12 * m) {
            return -1;
        }
    }
    return pin;
}

// Row p of the singular periodic operator from column p (the FD matrix is
// symmetric): A[p][p+o] = A[p+o][p]; the diagonal closes the zero row sum.
void restore_pinned_row(const HostLevel& L, std::vector<double>& R, int64_t p)
{
    const int KS = L.KS, center = (KS - 1) / 2, D = L.D;
    int c[3];
    int64_t t = p;
    c[2] = (int)(t % L.n[2]); t /= L.n[2]; c[1] = (int)(t % L.n[1]); c[0] = (int)(t / L.n[1]);
    double off = 0.0;
    for (int k = 0; k < KS; ++k) {
        if (k == center) continue;
        int o[3] = {0, 0, 0};
        if (D == 2) { o[0] = k / 3 - 1; o[1] = k % 3 - 1; }
        else { o[0] = k / 9 - 1; o[1] = (k / 3) % 3 - 1; o[2] = k % 3 - 1; }
        int g[3];
        for (int d = 0; d < 3; ++d) {
            g[d] = c[d] + o[d];
            if (g[d] < 0) g[d] += L.n[d];
            else if (g[d] >= L.n[d]) g[d] -= L.n[d];
        }
        const int64_t j = ((int64_t)g[0] * L.n[1] + g[1]) * L.n[2] + g[2];
        const double v = R[(size_t)j * KS + (KS - 1 - k)];
        R[(size_t)p * KS + k] = v;
        off += v;
    }
    R[(size_t)p * KS + center] = -off;
}

HostLevel level_from_coo(int I, int J, int K, unsigned long long n_row, unsigned long long nnz,
                         const unsigned long long* rows, const unsigned long long* cols,
                         const double* vals, bool periodic_aware, int64_t* pin_out,
                         std::vector<double>* pinned_rows)
{
    HostLevel L;
    L.D = K > 1 ? 3 : 2;
    L.n[0] = I;
    L.n[1] = J;
    L.n[2] = K;
    L.N = (int64_t)I * J * K;
    L.KS = L.D == 2 ? 9 : 27;
    if ((unsigned long long)L.N != n_row)
        throw std::runtime_error("hip_multigrid: I*J*K does not match the matrix size");
    std::vector<double> R((size_t)L.N * L.KS, 0.0);
    int wrapped[3] = {0, 0, 0};
    for (unsigned long long q = 0; q < nnz; ++q) {
        const unsigned long long r = rows[q], c = cols[q];
        if (r >= n_row || c >= n_row) throw std::runtime_error("hip_multigrid: index out of range");
        int rc[3], cc[3];
        unsigned long long a = r, b = c;
        rc[2] = (int)(a % K); a /= K; rc[1] = (int)(a % J); rc[0] = (int)(a / J);
        cc[2] = (int)(b % K); b /= K; cc[1] = (int)(b % J); cc[0] = (int)(b / J);
        int off[3] = {0, 0, 0};
        const int dims[3] = {I, J, K};
        for (int d = 0; d < 3; ++d)
            if (!axis_offset(rc[d], cc[d], dims[d], off[d], wrapped[d]))
                throw std::runtime_error("hip_multigrid: matrix is not a 3^D-point stencil on the I x J x K node grid");
        int k;
        if (L.D == 2) k = (off[0] + 1) * 3 + (off[1] + 1);
        else k = (off[0] + 1) * 9 + (off[1] + 1) * 3 + (off[2] + 1);
        R[(size_t)r * L.KS + k] += vals[q];
    }
    for (int d = 0; d < 3; ++d) L.wrap[d] = (dims_n(L, d) >= 3) ? wrapped[d] : 0;
    *pin_out = -1;
    if (periodic_aware) {
        *pin_out = detect_pinned_periodic(L, R);
        if (*pin_out >= 0) {
            if (pinned_rows) *pinned_rows = R;
            restore_pinned_row(L, R, *pin_out);
        }
    }
    classify(L, R);
    return L;
}

// Galerkin coarse level: rows of R A^ P with A^ the scaled fine operator.
HostLevel galerkin(const HostLevel& F, const AxisTransfer* tr, const int* nc)
{
    HostLevel C;
    C.D = F.D;
    C.KS = F.KS;
    for (int d = 0; d < 3; ++d) {
        C.n[d] = nc[d];
        C.wrap[d] = F.wrap[d];
    }
    C.N = (int64_t)nc[0] * nc[1] * nc[2];
    const int D = F.D, KS = F.KS;
    std::vector<double> rows((size_t)C.N * KS, 0.0);
    std::atomic<int> bad{0};
    parallel_for(C.N, [&](int64_t ci) {
        int c[3];
        int64_t t = ci;
        c[2] = (int)(t % nc[2]); t /= nc[2]; c[1] = (int)(t % nc[1]); c[0] = (int)(t / nc[1]);
        double* out = &rows[(size_t)ci * KS];
        const int m0 = tr[0].rn[c[0]], m1 = tr[1].rn[c[1]], m2 = D == 3 ? tr[2].rn[c[2]] : 1;
        for (int a = 0; a < m0; ++a)
            for (int b = 0; b < m1; ++b)
                for (int e = 0; e < m2; ++e) {
                    int f[3] = {tr[0].rf[c[0]] + a, tr[1].rf[c[1]] + b, D == 3 ? tr[2].rf[c[2]] + e : 0};
                    for (int d = 0; d < 3; ++d)
                        if (tr[d].wrap) f[d] = f[d] < 0 ? f[d] + F.n[d] : (f[d] >= F.n[d] ? f[d] - F.n[d] : f[d]);
                    double rw = tr[0].rw[3 * c[0] + a] * tr[1].rw[3 * c[1] + b];
                    if (D == 3) rw = rw * tr[2].rw[3 * c[2] + e];
                    const int64_t fi = ((int64_t)f[0] * F.n[1] + f[1]) * F.n[2] + f[2];
                    const double* arow = &F.Ah[(size_t)F.cls[fi] * KS];
                    for (int k = 0; k < KS; ++k) {
                        const double av = arow[k];
                        if (av == 0.0) continue;
                        int o[3] = {0, 0, 0};
                        if (D == 2) { o[0] = k / 3 - 1; o[1] = k % 3 - 1; }
                        else { o[0] = k / 9 - 1; o[1] = (k / 3) % 3 - 1; o[2] = k % 3 - 1; }
                        int g[3];
                        for (int d = 0; d < 3; ++d) {
                            g[d] = f[d] + o[d];
                            if (g[d] < 0) g[d] += F.n[d];
                            else if (g[d] >= F.n[d]) g[d] -= F.n[d];
                        }
                        const double ra = rw * av;
                        const int hm2 = D == 3 ? 2 : 1;
                        for (int h0 = 0; h0 < 2; ++h0) {
                            const double p0 = tr[0].pw[2 * g[0] + h0];
                            if (p0 == 0.0) continue;
                            for (int h1 = 0; h1 < 2; ++h1) {
                                const double p1 = tr[1].pw[2 * g[1] + h1];
                                if (p1 == 0.0) continue;
                                for (int h2 = 0; h2 < hm2; ++h2) {
                                    double p = p0 * p1;
                                    int cc[3] = {tr[0].pc[g[0]] + h0, tr[1].pc[g[1]] + h1, 0};
                                    if (D == 3) {
                                        const double p2 = tr[2].pw[2 * g[2] + h2];
                                        if (p2 == 0.0) continue;
                                        p = p * p2;
                                        cc[2] = tr[2].pc[g[2]] + h2;
                                    }
                                    for (int d = 0; d < 3; ++d)
                                        if (tr[d].wrap && cc[d] == nc[d]) cc[d] = 0;
                                    int oo[3] = {0, 0, 0};
                                    for (int d = 0; d < D; ++d) {
                                        int dd = cc[d] - c[d];
                                        if (C.wrap[d]) {
                                            if (dd > 1) dd -= nc[d];
                                            else if (dd < -1) dd += nc[d];
                                        }
                                        if (dd < -1 || dd > 1) { bad = 1; dd = 0; }
                                        oo[d] = dd;
                                    }
                                    const int kk = D == 2 ? (oo[0] + 1) * 3 + (oo[1] + 1)
                                                          : (oo[0] + 1) * 9 + (oo[1] + 1) * 3 + (oo[2] + 1);
                                    out[kk] += ra * p;
                                }
                            }
                        }
                    }
                }
    });
    if (bad) throw std::runtime_error("hip_multigrid: Galerkin operator wider than 3 nodes");
    classify(C, rows);
    return C;
}

void dense_inverse(const HostLevel& L, std::vector<double>& inv, bool pin0)
{
    const int64_t n = L.N;
    std::vector<double> m((size_t)(n * n), 0.0);
    inv.assign((size_t)(n * n), 0.0);
    const int D = L.D, KS = L.KS;
    for (int64_t i = 0; i < n; ++i) {
        int c[3];
        int64_t t = i;
        c[2] = (int)(t % L.n[2]); t /= L.n[2]; c[1] = (int)(t % L.n[1]); c[0] = (int)(t / L.n[1]);
        const double* row = &L.Ah[(size_t)L.cls[i] * KS];
        for (int k = 0; k < KS; ++k) {
            if (row[k] == 0.0) continue;
            int o[3] = {0, 0, 0};
            if (D == 2) { o[0] = k / 3 - 1; o[1] = k % 3 - 1; }
            else { o[0] = k / 9 - 1; o[1] = (k / 3) % 3 - 1; o[2] = k % 3 - 1; }
            int g[3];
            for (int d = 0; d < 3; ++d) {
                g[d] = c[d] + o[d];
                if (g[d] < 0) g[d] += L.n[d];
                else if (g[d] >= L.n[d]) g[d] -= L.n[d];
            }
            const int64_t j = ((int64_t)g[0] * L.n[1] + g[1]) * L.n[2] + g[2];
            m[(size_t)(i * n + j)] += row[k];
        }
        inv[(size_t)(i * n + i)] = 1.0;
    }
    if (pin0) {
        // singular coarsest operator: pin coarse node 0 (identity row)
        for (int64_t j = 0; j < n; ++j) m[(size_t)j] = 0.0;
        m[0] = 1.0;
    }
    for (int64_t col = 0; col < n; ++col) {
        int64_t p = col;
        for (int64_t r = col + 1; r < n; ++r)
            if (std::fabs(m[(size_t)(r * n + col)]) > std::fabs(m[(size_t)(p * n + col)])) p = r;
        if (m[(size_t)(p * n + col)] == 0.0) throw std::runtime_error("hip_multigrid: singular coarsest operator");
        if (p != col)
            for (int64_t j = 0; j < n; ++j) {
                std::swap(m[(size_t)(col * n + j)], m[(size_t)(p * n + j)]);
                std::swap(inv[(size_t)(col * n + j)], inv[(size_t)(p * n + j)]);
            }
        const double d = m[(size_t)(col * n + col)];
        for (int64_t j = 0; j < n; ++j) {
            m[(size_t)(col * n + j)] /= d;
            inv[(size_t)(col * n + j)] /= d;
        }
        parallel_for(n, [&](int64_t r) {
            if (r == col) return;
            const double f = m[(size_t)(r * n + col)];
            if (f == 0.0) return;
            for (int64_t j = 0; j < n; ++j) {
                m[(size_t)(r * n + j)] -= f * m[(size_t)(col * n + j)];
                inv[(size_t)(r * n + j)] -= f * inv[(size_t)(col * n + j)];
            }
        });
    }
    // with node 0 pinned its right-hand side entry is ignored (b_0 -> 0)
    if (pin0)
        for (int64_t i = 0; i < n; ++i) inv[(size_t)(i * n)] = 0.0;
}

// ------------------------------------------------------------ device buffers

template <typename T>
T* dev_copy(const std::vector<T>& v)
{
    T* p = nullptr;
    MG_HIP(hipMalloc(&p, std::max<size_t>(1, v.size()) * sizeof(T)));
    if (!v.empty()) MG_HIP(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return p;
}

template <typename T>
std::vector<T> cast_vec(const std::vector<double>& v)
{
    return std::vector<T>(v.begin(), v.end());
}

struct DevLevelBuf {
    uint16_t* cls = nullptr;
    // chunked 7-point 3D level: nodes the chunk kernels leave to the
    // per-node kernels, and the class the chunk kernels handle
    uint32_t* line_list = nullptr;
    uint32_t line_n = 0;
    int line_cls = -1;
    double *K = nullptr, *Ah = nullptr, *Rx = nullptr, *dinv = nullptr;
    float *Ah32 = nullptr, *Rx32 = nullptr, *dinv32 = nullptr;
    // vectors: FP64 x/b/t and FP32 x/b/t
    double *x = nullptr, *b = nullptr, *t = nullptr;
    float *xf = nullptr, *bf = nullptr, *tf = nullptr;
};

struct DevTransferBuf {
    int *pc[3] = {nullptr, nullptr, nullptr}, *rf[3] = {nullptr, nullptr, nullptr},
        *rn[3] = {nullptr, nullptr, nullptr};
    double *pw[3] = {nullptr, nullptr, nullptr}, *rw[3] = {nullptr, nullptr, nullptr};
    float *pw32[3] = {nullptr, nullptr, nullptr}, *rw32[3] = {nullptr, nullptr, nullptr};
};

}  // namespace

// ================================================================= solver

namespace psum_hip {

// kernel kinds of recorded ops (base + template variant bits)
constexpr uint16_t kKindSmooth = 0;      // + (FP64 << 3 | compact << 2 | prolong << 1 | acc), large tiles
constexpr uint16_t kKindDown = 16;       // + (FP64 << 1 | compact), large tiles
constexpr uint16_t kKindRR = 20;         // + (FP64 << 1 | compact)
constexpr uint16_t kKindCoarse = 24;     // + FP64
constexpr uint16_t kKindOuter = 26;      // + (norms << 2 | compact << 1 | emit FP32), 2D
constexpr uint16_t kKindVec = 34;        // + op (0 zero, 1 add correction, 2 copy)
constexpr uint16_t kKindHadamard = 37;   // FP64
constexpr uint16_t kKindCount = 38;

class HipMultigrid {
public:
    explicit HipMultigrid(bool mixed) : mixed_(mixed) {}
    ~HipMultigrid() { release(); }

    // options (sycl_multigrid_gpu.cpp:134-162, sycl_multigrid32f_gpu.cpp:162-196)
    void set_options(const char* options)
    {
        std::istringstream iss(options ? options : "");
        std::string key;
        bool k_provided = false;
        const int pre0 = pre_, post0 = post_;
        while (iss >> key) {
            if (key == "I") iss >> I_;
            else if (key == "J") iss >> J_;
            else if (key == "K") { iss >> K_; k_provided = true; }
            else if (key == "depth") iss >> depth_;
            else if (key == "pre_relax") iss >> pre_;
            else if (key == "post_relax") iss >> post_;
            else if (key == "max_cycles") iss >> max_cycles_;
            else if (key == "correction_interval") {
                int v = 0;
                if (!(iss >> v) || v < 1) throw std::invalid_argument("correction_interval must be positive");
                corr_ = v;
            } else if (key == "tol") iss >> tol_;
            else if (key == "periodic_mode") iss >> periodic_mode_;
            else if (key == "fuse") iss >> fuse_;
            else if (key == "line") iss >> line_;
            else if (key == "graph") iss >> use_graph_;
            else if (key == "num_conv_mask" || key == "num_conv_mask_relax" ||
                     key == "num_conv_mask_restrict" || key == "num_conv_mask_interpolate" ||
                     key == "num_conv_mask_a" || key == "tail") {
                int ignored;
                iss >> ignored;
            }
        }
        if (!k_provided) K_ = 1;
        if (!host_.empty() && (pre_ != pre0 || post_ != post0)) {
            drop_graphs();
            build_operator();
        }
    }

    // Kernel-shape options that may change after set_matrix: "fuse 0|1"
    // (2D fused tile kernels) and "line 0|1" (chunked sweeps and residuals on
    // 7-point 3D levels).  "tail 0|1" is accepted and has no effect: the
    // coarse end is one dense product (build_operator).  Other keys are
    // rejected.
    void set_tuning(const char* options)
    {
        std::istringstream iss(options ? options : "");
        std::string key;
        while (iss >> key) {
            int v = 0;
            if (!(iss >> v)) throw std::invalid_argument("hip_multigrid: tuning option " + key + " needs a value");
            if (key == "tail") continue;
            else if (key == "fuse") fuse_ = v;
            else if (key == "line") line_ = v;
            else throw std::invalid_argument("hip_multigrid: unknown tuning option " + key);
        }
        tile_fit_.clear();
        drop_graphs();   // captured cycles hold the previous kernel shapes
    }

    // Smoothing sweeps per level before and after the coarse correction
    // (pre_relax / post_relax), changed after set-up; captured cycles are
    // dropped.
    void set_smoothing(int pre, int post)
    {
        if (pre < 0 || post < 0 || pre > 64 || post > 64 || pre + post < 1)
            throw std::invalid_argument("hip_multigrid: smoothing sweeps need 0 <= pre, post <= 64, pre + post >= 1");
        pre_ = pre;
        post_ = post;
        tile_fit_.clear();
        drop_graphs();
        if (!host_.empty()) build_operator();
    }

    void set_stream(hipStream_t s) { stream_ = s; }

    void set_matrix(unsigned long long n_row, unsigned long long n_col, unsigned long long nnz,
                    const unsigned long long* rows, const unsigned long long* cols, const double* vals)
    {
        if (n_row != n_col) throw std::runtime_error("hip_multigrid: matrix must be square");
        if (I_ < 1 || J_ < 1 || K_ < 1 || depth_ < 1)
            throw std::invalid_argument("multigrid: positive grid dimensions and depth required");
        release();
        std::vector<HostLevel> L;
        int64_t pin = -1;
        L.push_back(level_from_coo(I_, J_, K_, n_row, nnz, rows, cols, vals, periodic_mode_ != 0,
                                   &pin, nullptr));
        pin_ = pin;
        std::vector<std::array<AxisTransfer, 3>> T;
        Axis ax[3];
        const int sz[3] = {I_, J_, K_};
        int per[3];
        for (int d = 0; d < 3; ++d) {
            for (int i = 0; i < sz[d]; ++i) ax[d].x.push_back(i);
            per[d] = periodic_mode_ != 0 && L[0].wrap[d];
        }
        for (int level = 0; level < depth_; ++level) {
            Axis co[3];
            int nc[3];
            bool same = true;
            std::array<AxisTransfer, 3> tr;
            for (int d = 0; d < 3; ++d) {
                const int nf = (int)ax[d].x.size();
                if (per[d]) {
                    // periodic axis: halve while even and >= 4, else keep
                    if (nf % 2 == 0 && nf >= 4) {
                        tr[d] = axis_transfer_periodic(nf);
                        for (int i = 0; i < nf; i += 2) co[d].x.push_back(ax[d].x[i]);
                    } else {
                        tr[d] = axis_transfer_identity(nf, 1);
                        co[d] = ax[d];
                    }
                } else {
                    co[d] = coarsen(ax[d]);
                }
                nc[d] = (int)co[d].x.size();
                if (co[d].x.size() != ax[d].x.size()) same = false;
            }
            if (same) break;   // endpoints cannot be coarsened further
            for (int d = 0; d < 3; ++d)
                if (!per[d]) tr[d] = axis_transfer(ax[d], co[d]);
            L.push_back(galerkin(L.back(), tr.data(), nc));
            T.push_back(tr);
            for (int d = 0; d < 3; ++d) ax[d] = co[d];
        }
        if (T.empty()) throw std::invalid_argument("multigrid: grid cannot be coarsened while retaining endpoints");
        if (L.back().N > 8192)
            throw std::runtime_error("hip_multigrid: coarse matrix too large (" + std::to_string(L.back().N) +
                                     " > 8192); increase depth");
        dense_inverse(L.back(), cinv_host_, pin_ >= 0);
        host_ = std::move(L);
        tr_host_ = std::move(T);
        tile_fit_.clear();
        upload();
        build_operator();
    }

    void set_source_replace(unsigned long long n, const unsigned long long* idx, const double* v)
    {
        // unique indices; the last value of a repeated index wins
        std::map<unsigned long long, double> m;
        for (unsigned long long i = 0; i < n; ++i) m[idx[i]] = v[i];
        upload_pairs(m, rep_idx_, rep_val_, rep_n_);
    }

    void set_source_addback(unsigned long long n, const unsigned long long* idx, const double* v)
    {
        // repeated indices accumulate (in argument order) before the device add
        std::map<unsigned long long, double> m;
        for (unsigned long long i = 0; i < n; ++i) m[idx[i]] += v[i];
        upload_pairs(m, add_idx_, add_val_, add_n_);
    }

    // solve(b, x): device pointers, b modified in place (addback, replace)
    // homogeneous: no addback and zero replace values (the linear part of the
    // solve, used by the adjoint)
    void solve(double* b, double* x, bool sync = true, bool homogeneous = false)
    {
        const double* bs = solve_begin(b, homogeneous);
        solve_core(b, bs, x);
        solve_end(b, x, sync);
    }

    // The three parts of solve(): begin (addback, replace, the consistent
    // right-hand side of a pinned periodic system; returns the right-hand
    // side the V-cycles see), core (the cycles) and end (gauge, sync).
    //
    // mean_part: b still holds the charge whose block sums (kMgThreads nodes
    // each) these are; its mean is taken off first (takes_mean() only).
    bool takes_mean() const
    {
        return pin_ >= 0 && nblk(N0()) <= kPinBlocks && add_n_ == 0 && rep_n_ <= kPinReplace;
    }
    const double* solve_begin(double* b, bool homogeneous = false, const double* mean_part = nullptr)
    {
        if (host_.empty()) throw std::runtime_error("hip_multigrid: solve before set_matrix");
        build_operator();     // nothing to do, unless a call that set the sweeps failed
        hipStream_t st = stream_;
        scaled_ = false;
        if (takes_mean()) {
            const PinArgs a{b, N0(), mean_part, rep_idx_, rep_val_, (int)rep_n_, homogeneous ? 1 : 0, bprime_, part_,
                            mixed_ ? nullptr : dev_[0].b, table<double>(0, false).dinv, dl(0).cls, pin_, shift_};
            hipLaunchKernelGGL(k_pin_rhs, dim3(nblk(N0())), dim3(kMgThreads), 0, st, a);
            hipLaunchKernelGGL(k_pin_set, dim3(1), dim3(kMgThreads), 0, st, a, (int64_t)nblk(N0()));
            MG_HIP(hipGetLastError());
            scaled_ = !mixed_;
            return bprime_;
        }
        if (add_n_ && !homogeneous) hipLaunchKernelGGL(k_addback, dim3(nblk(add_n_)), dim3(kMgThreads), 0, st, b, add_idx_, add_val_, add_n_);
        if (rep_n_) hipLaunchKernelGGL(k_replace, dim3(nblk(rep_n_)), dim3(kMgThreads), 0, st, b, rep_idx_, rep_val_, rep_n_, homogeneous ? 1 : 0);
        MG_HIP(hipGetLastError());
        const int64_t N = N0();
        if (pin_ >= 0) {
            // consistent singular form: b' = b, b'_p = b_p - sum(b)
            MG_HIP(hipMemcpyAsync(bprime_, b, (size_t)N * sizeof(double), hipMemcpyDeviceToDevice, st));
            hipLaunchKernelGGL(k_psum, dim3(nblk(N)), dim3(kMgThreads), 0, st, b, N, part_);
            hipLaunchKernelGGL(k_fsum, dim3(1), dim3(kMgThreads), 0, st, part_, (int64_t)nblk(N), shift_);
            hipLaunchKernelGGL(k_set_pin, dim3(1), dim3(64), 0, st, bprime_, b, shift_, pin_);
            MG_HIP(hipGetLastError());
            return bprime_;
        }
        return b;
    }

    void solve_core(const double* b, const double* bs, double* x)
    {
        last_cycles_ = 0;
        last_rel_ = NAN;
        rec_iter_ = 1;                 // iteration 0 is the residual before the first cycle
        const bool use_tol = tol_ > 0.0;
        // With a tolerance, the first check comes after the number of cycles
        // the previous solve needed minus one (warm-started solves of a
        // time-stepping loop need similar counts); after that every cycle is
        // checked.  A check reads ||b - A x||^2 and ||b||^2 back to the host.
        const int first_check = std::max(1, std::min(max_cycles_, predicted_ - 1));
        if (!mixed_) {
            rec_phase(0, kStageOuter, 0);
            if (!scaled_ || rec_) scale_rhs_f64(bs);
            if (!use_tol) {
                vcycles_f64(x, max_cycles_);
                last_cycles_ = max_cycles_;
            } else {
                double rr, bb;
                const bool chain = chained(b, x);
                cycles_f64(b, x, first_check - 1, chain);
                last_cycles_ = first_check - 1;
                do {
                    checked_cycle_f64(bs, b, x, chain);
                    ++last_cycles_;
                    read_norms(&rr, &bb);
                    last_rel_ = bb > 0 ? std::sqrt(rr / bb) : 0.0;
                } while (!(last_rel_ <= tol_) && last_cycles_ < max_cycles_);
            }
        } else {
            // refinement iteration: r = b - A x (FP64) -> FP32 V-cycles on A e = r -> x += e
            double rr, bb;
            const bool fm = fused_mixed();
            rec_phase(0, kStageOuter, 0);
            outer_residual(bs, b, x, true, fm, false);
            int cycle = 0;
            if (use_tol) {
                // the iterations before the first whose norms are read
                cycle = std::max(0, std::min(first_check, max_cycles_) - 1);
                iterations_f32(bs, b, x, cycle, chained(b, x));
                last_cycles_ = cycle;
            }
            while (cycle < max_cycles_) {
                if (use_tol && cycle >= first_check) {
                    read_norms(&rr, &bb);
                    last_rel_ = bb > 0 ? std::sqrt(rr / bb) : 0.0;
                    if (last_rel_ <= tol_) break;
                }
                if (use_tol) {
                    // the check before iteration cycle+1 reads this iteration's norms
                    iteration_f32(bs, b, x);
                    cycle += 1;
                    last_cycles_ += 1;
                    continue;
                }
                // fixed count (the reference 32f backend): batches of
                // correction_interval V-cycles between FP64 residuals, no
                // host check (so the whole solve can be captured in a graph)
                const int batch = std::min(corr_, max_cycles_ - cycle);
                vcycles_f32(batch, fm, x);
                cycle += batch;
                last_cycles_ += batch;
                if (cycle < max_cycles_) {
                    rec_phase(rec_iter_ - 1, kStageOuter, 0);
                    outer_residual(bs, b, x, true, fm, false);
                }
            }
            if (use_tol) {
                if (last_cycles_ == 0) {
                    outer_residual(bs, b, x, false, false, true);
                    ++norm_seq_;
                }
                read_norms(&rr, &bb);
                last_rel_ = bb > 0 ? std::sqrt(rr / bb) : 0.0;
            }
        }
        if (use_tol) predicted_ = last_cycles_;
    }

    void solve_end(const double* b, double* x, bool sync)
    {
        hipStream_t st = stream_;
        if (const double* shift = gauge(b, x)) {
            hipLaunchKernelGGL(k_gauge_apply, dim3(nblk(N0())), dim3(kMgThreads), 0, st, x, N0(), shift);
            MG_HIP(hipGetLastError());
        }
        if (sync) MG_HIP(hipStreamSynchronize(st));
    }
    // the device value to take off x after the cycles, or null
    const double* gauge(const double* b, const double* x)
    {
        if (pin_ < 0) return nullptr;
        // (with a tolerance, the last check has left it)
        if (!(tol_ > 0.0)) {
            hipLaunchKernelGGL(k_gauge_read, dim3(1), dim3(64), 0, stream_, x, b, pin_, shift_ + 1);
            MG_HIP(hipGetLastError());
        }
        return shift_ + 1;
    }

    // ---- batched fixed-cycle solves --------------------------------------
    // An op of the core of a fixed-cycle solve, recorded instead of launched:
    // the kernel body and variant (kind), its block count and its argument
    // struct.  Ops of different solvers with equal keys are independent and
    // run as one batched launch; keys grow along each solver's sequence.
    using RecOp = MgRecOp;

    // whether the core of a solve can be recorded: a fixed cycle count on a
    // 2D hierarchy through the fused tile kernels, with pre- and post-sweeps
    bool recordable() const
    {
        if (host_.empty() || tol_ > 0.0 || host_[0].D != 2 || !fuse_ || pre_ < 1 || post_ < 1) return false;
        for (const auto& h : host_)
            if (h.D != 2) return false;
        return true;
    }

    // The ops of solve_core(b, bs, x), in order, without launching anything
    // (solve_begin must have produced bs; solve_end follows the ops).
    void record_core(const double* b, const double* bs, double* x, std::vector<RecOp>& ops)
    {
        if (!recordable()) throw std::logic_error("hip_multigrid: this solve cannot be batched");
        build_operator();
        ops.clear();
        rec_ = &ops;
        try {
            solve_core(b, bs, x);
        } catch (...) {
            rec_ = nullptr;
            throw;
        }
        rec_ = nullptr;
    }

    double* pin_rhs() const { return pin_ >= 0 ? bprime_ : nullptr; }

    // fixed V-cycle count, one per refinement iteration, no host checks and
    // no graphs of its own: the solve can be captured into a caller's graph
    void set_fixed_cycles(int cycles)
    {
        if (cycles < 1) throw std::invalid_argument("hip_multigrid: fixed cycle count must be >= 1");
        tol_ = 0.0;
        max_cycles_ = cycles;
        corr_ = 1;
        use_graph_ = 0;
        drop_graphs();
        fixed_mode_ = true;
    }

    int last_cycles() const { return last_cycles_; }
    int predicted() const { return predicted_; }
    void set_predicted(int p) { predicted_ = p; }
    double last_rel() const { return last_rel_; }
    int64_t N0() const { return host_.empty() ? 0 : host_[0].N; }
    int levels() const { return (int)host_.size(); }

private:
    // ---- recording of batched solves (see record_core)
    static constexpr uint32_t kStageInit = 0, kStageDown = 1, kStageCoarse = 2, kStageUp = 3,
                              kStageCorr = 4, kStageOuter = 5;
    std::vector<RecOp>* rec_ = nullptr;
    uint32_t rec_iter_ = 0, rec_key_ = 0, rec_seq_ = 0;

    // key of the ops that follow: iteration, stage, level (ascending for the
    // downward pass, descending for the upward one), then emission order
    void rec_phase(uint32_t it, uint32_t stage, uint32_t lvl)
    {
        rec_key_ = (it << 20) | (stage << 16) | (lvl << 8);
        rec_seq_ = 0;
    }

    template <typename A>
    void emit(uint16_t kind, unsigned nb, const A& a)
    {
        RecOp op;
        op.key = rec_key_ | (rec_seq_ & 0xffu);
        ++rec_seq_;
        op.kind = kind;
        op.nblocks = nb;
        op.args.resize(sizeof(A));
        std::memcpy(op.args.data(), &a, sizeof(A));
        rec_->push_back(std::move(op));
    }

    template <typename T>
    static constexpr int tbit() { return std::is_same<T, double>::value ? 1 : 0; }

    template <typename T, bool C, bool P, bool A>
    void run_smooth_tile(bool small, unsigned nb, const SmoothTileArgs<T>& a)
    {
        if (rec_) { emit((uint16_t)(kKindSmooth + ((tbit<T>() << 3) | (C << 2) | (P << 1) | (A ? 1 : 0))), nb, a); return; }
        if (small) hipLaunchKernelGGL((k_smooth_tile<T, C, P, A, true>), dim3(nb), dim3(TileGeom<T, true>::threads), 0, stream_, a);
        else hipLaunchKernelGGL((k_smooth_tile<T, C, P, A, false>), dim3(nb), dim3(TileGeom<T, false>::threads), 0, stream_, a);
    }

    template <typename T, bool C>
    void run_down(bool small, unsigned nb, const DownTileArgs<T>& a)
    {
        if (rec_) { emit((uint16_t)(kKindDown + ((tbit<T>() << 1) | (C ? 1 : 0))), nb, a); return; }
        if (small) hipLaunchKernelGGL((k_down_tile<T, C, true>), dim3(nb), dim3(TileGeom<T, true>::threads), 0, stream_, a);
        else hipLaunchKernelGGL((k_down_tile<T, C, false>), dim3(nb), dim3(TileGeom<T, false>::threads), 0, stream_, a);
    }

    template <typename T, bool C>
    void run_rr(unsigned nb, const ResidRestrictArgs<T>& a)
    {
        if (rec_) { emit((uint16_t)(kKindRR + ((tbit<T>() << 1) | (C ? 1 : 0))), nb, a); return; }
        hipLaunchKernelGGL((k_resid_restrict<T, C>), dim3(nb), dim3(kMgThreads), 0, stream_, a);
    }

    template <typename T>
    void run_coarse(unsigned nb, const CoarseArgs<T>& a)
    {
        if (rec_) { emit((uint16_t)(kKindCoarse + tbit<T>()), nb, a); return; }
        hipLaunchKernelGGL((k_coarse_solve<T>), dim3(nb), dim3(kMgThreads), 0, stream_, a);
    }

    template <int D, bool C, bool F32, bool NORMS>
    void run_outer(unsigned nb, const OuterArgs& a)
    {
        if (rec_) {
            if (D != 2) throw std::logic_error("hip_multigrid: only 2D solves are batched");
            emit((uint16_t)(kKindOuter + ((NORMS ? 4 : 0) | (C ? 2 : 0) | (F32 ? 1 : 0))), nb, a);
            return;
        }
        hipLaunchKernelGGL((k_outer_residual<D, C, F32, NORMS>), dim3(nb), dim3(kMgThreads), 0, stream_, a);
    }

    template <int OP>
    void run_vec(const VecArgs& a)
    {
        const unsigned nb = nblk(a.n);
        if (rec_) { emit((uint16_t)(kKindVec + OP), nb, a); return; }
        hipLaunchKernelGGL((k_vec<OP>), dim3(nb), dim3(kMgThreads), 0, stream_, a);
    }

    void run_hadamard(const HadamardArgs<double>& a)
    {
        const unsigned nb = nblk(a.L.N);
        if (rec_) { emit((uint16_t)kKindHadamard, nb, a); return; }
        hipLaunchKernelGGL((k_hadamard<double>), dim3(nb), dim3(kMgThreads), 0, stream_, a);
    }

    bool mixed_;
    int I_ = 0, J_ = 0, K_ = 0, depth_ = 3, pre_ = 2, post_ = 1, max_cycles_ = 10, corr_ = 4;
    int fuse_ = 1;   // 2D: fused multi-sweep tile smoothing and residual+restriction
    int line_ = 1;   // 3D 7-point levels: chunk kernels (k_smooth_line, k_residual_line)
    // the coarse end as one dense operator: levels `level` and below (the
    // coarsest alone when nothing is merged)
    struct Operator {
        double* m = nullptr;
        int level = 0, ld = 0;
    };
    Operator op_, op_fixed_;           // op_fixed_: fixed-cycle solves (may be op_'s matrix)
    int op_pre_ = -1, op_post_ = -1;   // sweeps they were built for
    bool fixed_mode_ = false;          // set_fixed_cycles was called
    std::vector<int> tile_fit_;
    double tol_ = 0.0;
    int predicted_ = 1;                // cycles the previous solve needed
    int periodic_mode_ = 1;
    int64_t pin_ = -1;                 // pinned node of a pinned-periodic matrix
    double* bprime_ = nullptr;         // consistent singular right-hand side
    bool scaled_ = false;              // dev_[0].b holds the scaled right-hand side
    double* shift_ = nullptr;          // device scalar for the gauge shift / sums
    hipStream_t stream_ = nullptr;
    std::vector<HostLevel> host_;
    std::vector<std::array<AxisTransfer, 3>> tr_host_;
    std::vector<double> cinv_host_;
    std::vector<DevLevelBuf> dev_;
    std::vector<DevTransferBuf> dtr_;
    double* part_ = nullptr;
    unsigned long long* norm_count_ = nullptr;   // norms stored, on the device
    NormBox* norms_ = nullptr;                   // pinned host memory
    unsigned long long norm_seq_ = 0;            // norms asked for
    unsigned long long *rep_idx_ = nullptr, *add_idx_ = nullptr;
    double *rep_val_ = nullptr, *add_val_ = nullptr;
    int64_t rep_n_ = 0, add_n_ = 0, rep_cap_ = 0, add_cap_ = 0;
    int last_cycles_ = 0;
    double last_rel_ = NAN;

    void upload_pairs(const std::map<unsigned long long, double>& m, unsigned long long*& di,
                      double*& dv, int64_t& n)
    {
        std::vector<unsigned long long> hi;
        std::vector<double> hv;
        for (auto& kv : m) {
            if (!host_.empty() && kv.first >= (unsigned long long)host_[0].N)
                throw std::runtime_error("hip_multigrid: source index out of range");
            hi.push_back(kv.first);
            hv.push_back(kv.second);
        }
        if (di) (void)hipFree(di);
        if (dv) (void)hipFree(dv);
        di = nullptr;
        dv = nullptr;
        n = (int64_t)hi.size();
        if (n) {
            di = dev_copy(hi);
            dv = dev_copy(hv);
        }
    }

    void release()
    {
        for (auto& c : cap64_.e) drop_graph(c);
        for (auto& c : cap32_.e) drop_graph(c);
        for (auto& d : dev_) {
            for (void* p : {(void*)d.cls, (void*)d.line_list, (void*)d.K, (void*)d.Ah, (void*)d.Rx, (void*)d.dinv,
                            (void*)d.Ah32, (void*)d.Rx32, (void*)d.dinv32, (void*)d.t, (void*)d.bf,
                            (void*)d.xf, (void*)d.tf, (void*)d.b, (void*)d.x})
                if (p) (void)hipFree(p);
        }
        dev_.clear();
        for (auto& t : dtr_)
            for (int d = 0; d < 3; ++d)
                for (void* p : {(void*)t.pc[d], (void*)t.rf[d], (void*)t.rn[d], (void*)t.pw[d],
                                (void*)t.rw[d], (void*)t.pw32[d], (void*)t.rw32[d]})
                    if (p) (void)hipFree(p);
        dtr_.clear();
        release_operator();
        if (part_) (void)hipFree(part_);
        if (norm_count_) (void)hipFree(norm_count_);
        if (norms_) (void)hipHostFree(norms_);
        if (shift_) (void)hipFree(shift_);
        if (bprime_) (void)hipFree(bprime_);
        shift_ = nullptr;
        bprime_ = nullptr;
        part_ = nullptr;
        norm_count_ = nullptr;
        norms_ = nullptr;
        norm_seq_ = 0;
    }

    void upload()
    {
        const int nl = (int)host_.size();
        dev_.resize(nl);
        for (int l = 0; l < nl; ++l) {
            const HostLevel& h = host_[l];
            DevLevelBuf& d = dev_[l];
            d.cls = dev_copy(h.cls);
            build_line_list(h, d);
            d.K = dev_copy(h.K);
            d.Ah = dev_copy(h.Ah);
            d.Rx = dev_copy(h.Rx);
            d.dinv = dev_copy(h.dinv);
            d.Ah32 = dev_copy(cast_vec<float>(h.Ah));
            d.Rx32 = dev_copy(cast_vec<float>(h.Rx));
            d.dinv32 = dev_copy(cast_vec<float>(h.dinv));
            const size_t N = (size_t)h.N;
            if (!mixed_) {
                if (l > 0) MG_HIP(hipMalloc(&d.x, N * sizeof(double)));
                MG_HIP(hipMalloc(&d.b, (N + kOpPad) * sizeof(double)));
                MG_HIP(hipMemset(d.b + N, 0, kOpPad * sizeof(double)));   // read beyond N by the dense product
                MG_HIP(hipMalloc(&d.t, N * sizeof(double)));
            } else {
                MG_HIP(hipMalloc(&d.xf, N * sizeof(float)));
                MG_HIP(hipMalloc(&d.bf, (N + kOpPad) * sizeof(float)));
                MG_HIP(hipMemset(d.bf + N, 0, kOpPad * sizeof(float)));
                MG_HIP(hipMalloc(&d.tf, N * sizeof(float)));
            }
        }
        dtr_.resize(tr_host_.size());
        for (size_t l = 0; l < tr_host_.size(); ++l)
            for (int d = 0; d < 3; ++d) {
                const AxisTransfer& t = tr_host_[l][d];
                dtr_[l].pc[d] = dev_copy(t.pc);
                dtr_[l].rf[d] = dev_copy(t.rf);
                dtr_[l].rn[d] = dev_copy(t.rn);
                dtr_[l].pw[d] = dev_copy(t.pw);
                dtr_[l].rw[d] = dev_copy(t.rw);
                dtr_[l].pw32[d] = dev_copy(cast_vec<float>(t.pw));
                dtr_[l].rw32[d] = dev_copy(cast_vec<float>(t.rw));
            }
        const int64_t nb = (int64_t)nblk(host_[0].N);
        MG_HIP(hipMalloc(&part_, (size_t)nb * 2 * sizeof(double)));
        MG_HIP(hipMalloc(&norm_count_, sizeof *norm_count_));
        MG_HIP(hipMemset(norm_count_, 0, sizeof *norm_count_));
        MG_HIP(hipMalloc(&shift_, 4 * sizeof(double)));
        if (pin_ >= 0) MG_HIP(hipMalloc(&bprime_, (size_t)host_[0].N * sizeof(double)));
        MG_HIP(hipHostMalloc(&norms_, sizeof *norms_, hipHostMallocCoherent));
        *norms_ = NormBox{0.0, 0.0, 0};
        MG_HIP(hipStreamSynchronize(nullptr));   // the clears above, before work on other streams
    }

    // A 3D level of at least 2^16 nodes (and fewer than 2^32) runs its
    // smoothing sweeps and residuals in chunks of kLine nodes: the class that
    // covers most nodes goes to the chunk kernels, and every node of a chunk
    // they skip (by the same test as line_chunk_fast) is listed.
    static bool line_chunk_fast_host(const HostLevel& h, uint32_t i, int cls_in)
    {
        const uint32_t n0 = (uint32_t)h.n[0], n1 = (uint32_t)h.n[1], n2 = (uint32_t)h.n[2];
        const uint32_t q = i / n2, z = i - q * n2, x = q / n1, y = q - x * n1;
        if (z < 1u || z + kLine > n2 - 1u || y < 1u || y + 2u > n1 || x < 1u || x + 2u > n0) return false;
        for (int k = 0; k < kLine; ++k)
            if ((int)h.cls[i + k] != cls_in) return false;
        return true;
    }
    void build_line_list(const HostLevel& h, DevLevelBuf& d)
    {
        d.line_cls = -1;
        d.line_n = 0;
        if (h.D != 3 || h.N < (1 << 16) || h.N >= (int64_t)0xffffffffll) return;
        std::vector<int64_t> count(h.dinv.size(), 0);
        for (int64_t i = 0; i < h.N; ++i) ++count[h.cls[i]];
        const int cls_in = (int)(std::max_element(count.begin(), count.end()) - count.begin());
        std::vector<uint32_t> list;
        const uint32_t nchunks = (uint32_t)(h.N / kLine);
        for (uint32_t t = 0; t < nchunks; ++t)
            if (!line_chunk_fast_host(h, t * kLine, cls_in))
                for (int k = 0; k < kLine; ++k) list.push_back(t * kLine + k);
        for (int64_t i = (int64_t)nchunks * kLine; i < h.N; ++i) list.push_back((uint32_t)i);
        d.line_cls = cls_in;
        d.line_n = (uint32_t)list.size();
        if (!list.empty()) d.line_list = dev_copy(list);
    }
    // dinv of class k of level l as the FP32 table holds it
    float host_dinv32(int l, int k) const { return (float)host_[l].dinv[k]; }

    // 3D transfers writing level l over planes (k_prolong_add_plane,
    // k_restrict_plane): planes of at least a wave, since a launch is a chain
    // of memory round trips and the per-node kernels' are longer (a term's
    // load waits for the one before).  Restriction to 26 x 23 x 31 and
    // 14 x 12 x 16 nodes in FP64: 11.9 -> 4.9 us.
    bool planar(int l) const
    {
        const HostLevel& h = host_[l];
        return line_ && h.D == 3 && (int64_t)h.n[1] * h.n[2] >= 64 && h.n[0] <= 65535 &&
               h.N < (int64_t)0xffffffffll && (l == 0 || host_[l - 1].N < (int64_t)0xffffffffll);
    }

    LineList line_list(int l) const
    {
        LineList ll;
        ll.list = dev_[l].line_list;
        ll.n = dev_[l].line_n;
        ll.nbc = nblk(host_[l].N / kLine);
        return ll;
    }
    LineGeom line_geom(int l) const
    {
        LineGeom g;
        g.n0 = host_[l].n[0];
        g.n1 = host_[l].n[1];
        g.n2 = host_[l].n[2];
        g.nchunks = (uint32_t)(host_[l].N / kLine);
        g.cls = dev_[l].cls;
        g.cls_in = dev_[l].line_cls;
        return g;
    }

    DevLevel dl(int l) const
    {
        DevLevel d;
        for (int q = 0; q < 3; ++q) {
            d.n[q] = host_[l].n[q];
            d.wrap[q] = host_[l].wrap[q];
        }
        d.N = host_[l].N;
        d.cls = dev_[l].cls;
        return d;
    }

    template <typename T>
    DevTable<T> table(int l, bool relax) const
    {
        DevTable<T> t;
        if constexpr (std::is_same<T, double>::value) {
            t.coef = relax ? dev_[l].Rx : dev_[l].Ah;
            t.dinv = dev_[l].dinv;
        } else {
            t.coef = relax ? dev_[l].Rx32 : dev_[l].Ah32;
            t.dinv = dev_[l].dinv32;
        }
        return t;
    }

    template <typename T>
    DevTransfer<T> transfer(int l) const
    {
        DevTransfer<T> t;
        for (int d = 0; d < 3; ++d) {
            t.wrap[d] = tr_host_[l][d].wrap;
            t.pc[d] = dtr_[l].pc[d];
            t.rf[d] = dtr_[l].rf[d];
            t.rn[d] = dtr_[l].rn[d];
            if constexpr (std::is_same<T, double>::value) {
                t.pw[d] = dtr_[l].pw[d];
                t.rw[d] = dtr_[l].rw[d];
            } else {
                t.pw[d] = dtr_[l].pw32[d];
                t.rw[d] = dtr_[l].rw32[d];
            }
        }
        return t;
    }

    template <typename T>
    void smooth(int l, T*& x, T*& buf, const T* b, double* acc = nullptr)
    {
        const DevLevel L = dl(l);
        const T two3 = (T)(2.0 / 3);
        const unsigned nb = nblk(L.N);
#define SMOOTH(DIM, CMP) \
        if (acc) hipLaunchKernelGGL((k_smooth<T, DIM, CMP, true>), dim3(nb), dim3(kMgThreads), 0, stream_, L, table<T>(l, true), x, b, buf, two3, acc); \
        else hipLaunchKernelGGL((k_smooth<T, DIM, CMP, false>), dim3(nb), dim3(kMgThreads), 0, stream_, L, table<T>(l, true), x, b, buf, two3, nullptr)
        if (line_ && dev_[l].line_cls >= 0) {
            const LineGeom G = line_geom(l);
            const LineList LL = line_list(l);
            const DevTable<T> tb = table<T>(l, true);
            const T* row = tb.coef + (int64_t)G.cls_in * 27;
            const unsigned nb = line_grid(LL);
#define SLINE(CMP, ACC, A) hipLaunchKernelGGL((k_smooth_line<T, CMP, ACC>), dim3(nb), dim3(kMgThreads), 0, stream_, G, LL, L, tb, row, x, b, buf, two3, A)
            if (host_[l].compact) { if (acc) SLINE(true, true, acc); else SLINE(true, false, nullptr); }
            else { if (acc) SLINE(false, true, acc); else SLINE(false, false, nullptr); }
#undef SLINE
        } else if (host_[l].D == 2) {
            if (host_[l].compact) { SMOOTH(2, true); } else { SMOOTH(2, false); }
        } else {
            if (host_[l].compact) { SMOOTH(3, true); } else { SMOOTH(3, false); }
        }
#undef SMOOTH
        std::swap(x, buf);
    }

    template <typename T>
    void residual(int l, const T* x, const T* b, T* r)
    {
        const DevLevel L = dl(l);
        const unsigned nb = nblk(L.N);
        if (line_ && dev_[l].line_cls >= 0) {
            const LineGeom G = line_geom(l);
            const LineList LL = line_list(l);
            const DevTable<T> tb = table<T>(l, false);
            const T* row = tb.coef + (int64_t)G.cls_in * 27;
            if (host_[l].compact) hipLaunchKernelGGL((k_residual_line<T, true>), dim3(line_grid(LL)), dim3(kMgThreads), 0, stream_, G, LL, L, tb, row, x, b, r);
            else hipLaunchKernelGGL((k_residual_line<T, false>), dim3(line_grid(LL)), dim3(kMgThreads), 0, stream_, G, LL, L, tb, row, x, b, r);
            return;
        }
        if (host_[l].D == 2) {
            if (host_[l].compact) hipLaunchKernelGGL((k_residual<T, 2, true>), dim3(nb), dim3(kMgThreads), 0, stream_, L, table<T>(l, false), x, b, r);
            else hipLaunchKernelGGL((k_residual<T, 2, false>), dim3(nb), dim3(kMgThreads), 0, stream_, L, table<T>(l, false), x, b, r);
        } else {
            if (host_[l].compact) hipLaunchKernelGGL((k_residual<T, 3, true>), dim3(nb), dim3(kMgThreads), 0, stream_, L, table<T>(l, false), x, b, r);
            else hipLaunchKernelGGL((k_residual<T, 3, false>), dim3(nb), dim3(kMgThreads), 0, stream_, L, table<T>(l, false), x, b, r);
        }
    }

    // `count` sweeps on level l: 2D levels in fused tile launches of up to
    // kMaxFuse sweeps (PROLONG: the first launch also applies x += P x_c)
    // acc (FP32 levels only): the last launch also adds its result into the
    // FP64 array acc; returns whether it did (only the fused 2D path can)
    template <typename T>
    bool smooth_n(int l, T*& x, T*& buf, const T* b, int count, const T* xc = nullptr,
                  double* acc = nullptr)
    {
        if (host_[l].D != 2 || !fuse_ || count == 0) {
            if (xc) prolong(l, xc, x);
            for (int s = 0; s < count; ++s) smooth<T>(l, x, buf, b, s == count - 1 ? acc : nullptr);
            return acc != nullptr && count > 0;
        }
        const DevLevel L = dl(l);
        const T two3 = (T)(2.0 / 3);
        const DevLevel C = xc ? dl(l + 1) : L;
        const DevTransfer<T> tr = xc ? transfer<T>(l) : DevTransfer<T>{};
        const bool cmp = host_[l].compact;
        const int ncls = (int)host_[l].dinv.size();
        const int half = xc && tile_steps(l, true) == 22 ? 1 : 0;
        bool accd = false;
        while (count > 0) {
            const int k = std::min(count, kMaxFuse);
            const int ostep = kTileX - 2 * k;
            const int64_t ntc = (L.n[1] + ostep - 1) / ostep;
            const bool small = small_tiles<T>(((L.n[0] + TileGeom<T, false>::rows - 1) / TileGeom<T, false>::rows) * ntc);
            const int rows = small ? TileGeom<T, true>::rows : TileGeom<T, false>::rows;
            const unsigned nb = (unsigned)(((L.n[0] + rows - 1) / rows) * ntc);
            double* a = (k == count) ? acc : nullptr;
            const SmoothTileArgs<T> ta{L, table<T>(l, true), ncls, x, b, buf, two3, k, C, tr, half, xc, a};
#define TILE(CMP, PRO, ACC) run_smooth_tile<T, CMP, PRO, ACC>(small, nb, ta)
            if constexpr (std::is_same<T, float>::value) {
                if (a) {
                    if (xc) { if (cmp) TILE(true, true, true); else TILE(false, true, true); }
                    else { if (cmp) TILE(true, false, true); else TILE(false, false, true); }
                    accd = true;
                }
            }
            if (!accd) {
                if (xc) { if (cmp) TILE(true, true, false); else TILE(false, true, false); }
                else { if (cmp) TILE(true, false, false); else TILE(false, false, false); }
            }
#undef TILE
            std::swap(x, buf);
            xc = nullptr;
            count -= k;
        }
        return accd;
    }

    // Tiles of 256 threads and 8 rows where the large ones would cover the
    // level with fewer blocks than this.  FP32: 128 blocks of 1024 threads,
    // half the compute units (1024^2 with small tiles 0.5-2 % slower).  FP64:
    // 512 blocks of 512 threads, two a compute unit: the small tiles' launches
    // take 10.4 and 12.1 us on 513^2 nodes (297 large blocks: 11.2 and 12.4),
    // 17.3 and 25.7 on 1025^2 (1105 large blocks: 15.6 and 23.0).  V(2,1)
    // cycles of 128^2 FP64 take 16 % less time with them (13.6 against 16.0 ms
    // per 20 steps of the Langmuir run).  Recorded solves share their launches
    // with other solvers, whose blocks fill the chip: always the large ones
    // (12 instances of 64^2..256^2: 27.3 against 28.2 ms).
    template <typename T>
    bool small_tiles(int64_t large_blocks) const
    {
        return !rec_ && large_blocks < (sizeof(T) == 8 ? 512 : 128);
    }

    // How the transfers between levels l and l + 1 step along the two axes,
    // 10 st[0] + st[1] with 2 for a halved axis and 1 for one kept as it is,
    // or 0 where the tables go beyond what the tiles hold (k_down_tile,
    // prolongation: the staged coarse values).  Checked once per level.
    int tile_steps(int l, bool prolongation)
    {
        if (tile_fit_.size() != 2 * host_.size()) tile_fit_.assign(2 * host_.size(), -1);
        int& fit = tile_fit_[2 * (size_t)l + (prolongation ? 1 : 0)];
        if (fit >= 0) return fit;
        int code = 0;
        bool ok = true;
        for (int d = 0; d < 2; ++d) {
            const AxisTransfer& t = tr_host_[l][d];
            const int nf = host_[l].n[d], nc = host_[l + 1].n[d];
            const int st = nf == nc ? 1 : 2;
            code = 10 * code + st;
            // a wrapped axis with transfers that do not wrap (periodic_mode 0):
            // a halo node's coarse nodes are not next to its tile's
            if (prolongation && (host_[l].wrap[d] != 0) != (t.wrap != 0)) ok = false;
            for (int c = 0; c < nc && !prolongation; ++c)
                if (t.rn[c] > 3 || t.rf[c] < st * c - (st - 1) || t.rf[c] + t.rn[c] > st * c + st) ok = false;
            for (int i = 0; i < nf && prolongation; ++i) {
                const int q = st == 2 ? i >> 1 : i;
                // (the last node of an even count is a coarse node itself)
                if (t.pc[i] != q && (t.wrap || t.pc[i] != q + 1 || t.pw[2 * i + 1] != 0.0)) ok = false;
                if (t.wrap && st == 2 && nf % 2 != 0) ok = false;
            }
        }
        fit = ok ? code : 0;
        return fit;
    }

    template <typename T>
    void prolong(int l, const T* xc, T* x)
    {
        const DevLevel F = dl(l), C = dl(l + 1);
        if (host_[l].D == 2)
            hipLaunchKernelGGL((k_prolong_add<T, 2>), dim3(nblk(F.N)), dim3(kMgThreads), 0, stream_, F, C, transfer<T>(l), xc, x);
        else if (planar(l))
            hipLaunchKernelGGL((k_prolong_add_plane<T>), dim3(nblk((int64_t)F.n[1] * F.n[2]), F.n[0]), dim3(kMgThreads), 0, stream_, F, C, transfer<T>(l), xc, x);
        else
            hipLaunchKernelGGL((k_prolong_add<T, 3>), dim3(nblk(F.N)), dim3(kMgThreads), 0, stream_, F, C, transfer<T>(l), xc, x);
    }

    // ---- the coarse end as one dense operator -----------------------------
    // The V-cycle from a level l >= 1 down starts from zero, so it is the
    // product of its right-hand side with a fixed N_l x N_l matrix (built once
    // per matrix and smoothing counts, k_dense_*).  One product replaces every
    // launch of the levels it covers: 3 per 2D level (5-7 us each), 2 + pre +
    // post per 3D level (3.7-11 us each).  The level taken is the finest whose
    // matrix is small enough to beat those launches:
    //   2D  33 MB: 2048 nodes 4.3 us (16-18 us for the level's launches), 4096
    //       nodes 21 us, no faster than the launches
    //   3D  200 MB: 17^3 nodes 28 us against 45-60 us
    // Fixed-cycle solves (batches of many solvers, whose matrices share the
    // caches) take at most 1089 nodes.  Their matrix is one of those that the
    // other is built from, so both are kept and a solver that switches to a
    // fixed cycle count builds nothing again.
    int operator_level(bool fixed) const
    {
        const int Lc = (int)host_.size() - 1;
        const int64_t limit = host_[0].D == 3 ? 200000000 : 33600000;
        for (int l = 1; l < Lc; ++l) {
            const int64_t n = host_[l].N;
            if (fixed ? n <= 1089 : (n < 32768 && n * n * 8 <= limit)) return l;
        }
        return Lc;
    }

    void release_operator()
    {
        if (op_.m) (void)hipFree(op_.m);
        if (op_fixed_.m && op_fixed_.m != op_.m) (void)hipFree(op_fixed_.m);
        op_ = op_fixed_ = Operator{};
        op_pre_ = op_post_ = -1;
    }

    // the operators for the current hierarchy and smoothing counts; without
    // memory for a merged one, the coarsest inverse alone
    void build_operator()
    {
        if (op_.m && pre_ == op_pre_ && post_ == op_post_) return;
        const int Lc = (int)host_.size() - 1;
        drop_graphs();
        release_operator();
        try {
            build_operators_at(operator_level(false), operator_level(true));
        } catch (const std::runtime_error&) {
            (void)hipGetLastError();
            release_operator();
            build_operators_at(Lc, Lc);
        }
        op_pre_ = pre_;
        op_post_ = post_;
    }

    // op_ at level `target`, op_fixed_ at `fixed` (target <= fixed).  One
    // allocation for everything but the results: a hipMalloc and a hipFree of
    // their own for each matrix of each level were most of the set-up's time
    // on small grids.
    void build_operators_at(int target, int fixed)
    {
        const int Lc = (int)host_.size() - 1;
        struct Scope {
            hipStream_t st = nullptr;
            double* mem = nullptr;
            ~Scope()
            {
                if (mem) (void)hipFree(mem);
                if (st) (void)hipStreamDestroy(st);
            }
        } own;
        MG_HIP(hipStreamCreateWithFlags(&own.st, hipStreamNonBlocking));
        hipStream_t st = own.st;
        size_t sq = (size_t)host_[Lc].N * host_[Lc].N, rect = 0;
        for (int l = target; l < Lc; ++l) {
            sq = std::max(sq, (size_t)host_[l].N * host_[l].N);
            rect = std::max(rect, (size_t)host_[l].N * host_[l + 1].N);
        }
        // the next level's operator and two n x n matrices, two m x n ones
        MG_HIP(hipMalloc(&own.mem, ((target < Lc ? 3 : 1) * sq + 2 * rect) * sizeof(double)));
        double *M = own.mem, *X = M + sq, *Y = X + sq, *B = Y + sq, *E = B + rect;
        MG_HIP(hipMemcpy(M, cinv_host_.data(), cinv_host_.size() * sizeof(double), hipMemcpyHostToDevice));
        for (int l = Lc;; --l) {
            if (l == fixed && l != target) keep_operator(op_fixed_, l, M, st);
            if (l == target) break;
            if (host_[l - 1].D == 2) operator_columns<2>(l - 1, M, X, Y, B, E, st);
            else operator_columns<3>(l - 1, M, X, Y, B, E, st);
            std::swap(M, X);
        }
        keep_operator(op_, target, M, st);
        if (fixed == target) op_fixed_ = op_;
        MG_HIP(hipStreamSynchronize(st));
    }

    void keep_operator(Operator& op, int level, const double* M, hipStream_t st)
    {
        const int n = (int)host_[level].N;
        op.level = level;
        op.ld = (n + 1) / 2 * 2;
        MG_HIP(hipMalloc(&op.m, (size_t)n * op.ld * sizeof(double)));
        hipLaunchKernelGGL(k_dense_pad, dim3(nblk(op.ld), n), dim3(kMgThreads), 0, st, n, op.ld, M, op.m);
        MG_HIP(hipGetLastError());
    }

    // X = the V-cycle from level l down applied to every unit vector:
    // pre-sweeps from zero, residual, restriction, the next level's operator M,
    // prolongation, post-sweeps (X and Y are exchanged as the sweeps go)
    template <int D>
    void operator_columns(int l, const double* M, double*& X, double*& Y, double* B, double* E, hipStream_t st)
    {
        const DevLevel F = dl(l), C = dl(l + 1);
        const int n = (int)F.N, m = (int)C.N;
        const double two3 = 2.0 / 3;
        const DevTable<double> rx{dev_[l].Rx, dev_[l].dinv}, ah{dev_[l].Ah, dev_[l].dinv};
        const dim3 th(kMgThreads), gf(nblk(n), n), gc(nblk(n), m);
        // sweep from zero: (2/3) I; no pre-sweeps: 0
        hipLaunchKernelGGL(k_dense_stencil<D>, gf, th, 0, st, F, rx.coef, (const double*)nullptr, X, 0.0, pre_ > 0 ? two3 : 0.0);
        for (int k = 1; k < pre_; ++k) {
            hipLaunchKernelGGL(k_dense_stencil<D>, gf, th, 0, st, F, rx.coef, X, Y, 1.0, two3);
            std::swap(X, Y);
        }
        hipLaunchKernelGGL(k_dense_stencil<D>, gf, th, 0, st, F, ah.coef, X, Y, -1.0, 1.0);
        hipLaunchKernelGGL(k_dense_restrict<D>, gc, th, 0, st, F, C, transfer<double>(l), dev_[l + 1].dinv, Y, B);
        hipLaunchKernelGGL(k_dense_product, dim3((n + 31) / 32, (m + 31) / 32), th, 0, st, m, n, M, B, E);
        hipLaunchKernelGGL(k_dense_prolong<D>, gf, th, 0, st, F, C, transfer<double>(l), E, X);
        for (int k = 0; k < post_; ++k) {
            hipLaunchKernelGGL(k_dense_stencil<D>, gf, th, 0, st, F, rx.coef, X, Y, 1.0, two3);
            std::swap(X, Y);
        }
        MG_HIP(hipGetLastError());
    }

    // One or more V-cycles on level-0 arrays (b0 scaled, x0 warm start).
    // xs[l] / ts[l] are the ping-pong pair of level l, bs[l] its rhs.
    // first_swept: xs[0] already holds the first level-0 sweep from zero.
    // acc: the last cycle's final level-0 sweep adds its result into acc
    // (returns whether that happened).
    template <typename T>
    bool vcycles(std::vector<T*>& xs, std::vector<T*>& ts, std::vector<T*>& bs, int cycles,
                 bool first_swept = false, double* acc = nullptr)
    {
        const T two3 = (T)(2.0 / 3);
        bool accd = false;
        const Operator& op = fixed_mode_ ? op_fixed_ : op_;
        const int ld = op.level;                 // this level and those below: one dense product
        for (int cyc = 0; cyc < cycles; ++cyc) {
            const uint32_t it = rec_iter_ + (uint32_t)cyc;
            for (int l = 0; l < ld; ++l) {
                rec_phase(it, kStageDown, (uint32_t)l);
                // coarse levels received their first sweep from the restriction
                const bool swept = (l > 0 || (cyc == 0 && first_swept)) && pre_ > 0;
                const int sweeps = swept ? pre_ - 1 : pre_;
                const DevLevel F = dl(l), C = dl(l + 1);
                const T fs = (l + 1 < ld && pre_ > 0) ? two3 : (T)0;
                if (host_[l].D == 2 && fuse_) {
                    const int steps = tile_steps(l, false);
                    const int h = steps ? std::min(sweeps, kMaxFuse) : 0;
                    smooth_n<T>(l, xs[l], ts[l], bs[l], sweeps - h);
                    const ResidRestrictArgs<T> ra{F, C, transfer<T>(l), table<T>(l, false), (int)host_[l].dinv.size(), table<T>(l + 1, false), xs[l], bs[l], bs[l + 1], xs[l + 1], fs};
                    if (steps) {
                        const int st[2] = {steps / 10, steps % 10};
                        const int64_t ntc = (C.n[1] + down_cols(h, st[1]) - 1) / down_cols(h, st[1]);
                        const bool small = small_tiles<T>(((C.n[0] + TileGeom<T, false>::crows - 1) / TileGeom<T, false>::crows) * ntc);
                        const int rows = small ? TileGeom<T, true>::crows : TileGeom<T, false>::crows;
                        const DownTileArgs<T> da{ra, table<T>(l, true), ts[l], two3, h, {st[0], st[1]}};
                        const unsigned nb = (unsigned)(((C.n[0] + rows - 1) / rows) * ntc);
                        if (host_[l].compact) run_down<T, true>(small, nb, da);
                        else run_down<T, false>(small, nb, da);
                        if (h > 0) std::swap(xs[l], ts[l]);
                    } else {
                        if (host_[l].compact) run_rr<T, true>(nblk(C.N), ra);
                        else run_rr<T, false>(nblk(C.N), ra);
                    }
                    continue;
                }
                smooth_n<T>(l, xs[l], ts[l], bs[l], sweeps);
                residual<T>(l, xs[l], bs[l], ts[l]);
                if (host_[l].D == 2)
                    hipLaunchKernelGGL((k_restrict<T, 2>), dim3(nblk(C.N)), dim3(kMgThreads), 0, stream_, F, C, transfer<T>(l), table<T>(l + 1, false), ts[l], bs[l + 1], xs[l + 1], fs);
                else if (planar(l + 1))
                    hipLaunchKernelGGL((k_restrict_plane<T>), dim3(nblk((int64_t)C.n[1] * C.n[2]), C.n[0]), dim3(kMgThreads), 0, stream_, F, C, transfer<T>(l), table<T>(l + 1, false), ts[l], bs[l + 1], xs[l + 1], fs);
                else
                    hipLaunchKernelGGL((k_restrict<T, 3>), dim3(nblk(C.N)), dim3(kMgThreads), 0, stream_, F, C, transfer<T>(l), table<T>(l + 1, false), ts[l], bs[l + 1], xs[l + 1], fs);
            }
            rec_phase(it, kStageCoarse, 0);
            const int n = (int)host_[ld].N;
            const unsigned nb = (unsigned)(((int64_t)n * 64 + kMgThreads - 1) / kMgThreads);
            run_coarse<T>(nb, CoarseArgs<T>{op.m, n, op.ld, bs[ld], xs[ld]});
            for (int l = ld - 1; l >= 0; --l) {
                rec_phase(it, kStageUp, 255u - (uint32_t)l);
                if (post_ > 0) {
                    double* a = (l == 0 && cyc == cycles - 1) ? acc : nullptr;
                    accd = smooth_n<T>(l, xs[l], ts[l], bs[l], post_, xs[l + 1], a) || accd;
                } else {
                    prolong<T>(l, xs[l + 1], xs[l]);
                }
            }
        }
        rec_iter_ += (uint32_t)cycles;
        MG_HIP(hipGetLastError());
        return accd;
    }

    // b0 = b o D0^-1 into dev_[0].b (once per solve: the V-cycles read it)
    void scale_rhs_f64(const double* b)
    {
        run_hadamard(HadamardArgs<double>{dl(0), table<double>(0, false), b, dev_[0].b});
    }

    // FP64 V-cycles on x with the scaled right-hand side in dev_[0].b
    void vcycles_f64(double* x, int cycles)
    {
        const int nl = (int)host_.size();
        std::vector<double*> xs(nl), ts(nl), bs(nl);
        for (int l = 0; l < nl; ++l) {
            xs[l] = l == 0 ? x : dev_[l].x;
            ts[l] = dev_[l].t;
            bs[l] = dev_[l].b;
        }
        vcycles<double>(xs, ts, bs, cycles);
        rec_phase(rec_iter_ - 1, kStageCorr, 0);
        if (xs[0] != x) run_vec<2>(VecArgs{x, xs[0], N0()});
    }

    // The mixed iteration fuses work into its neighbours when the level-0
    // smoothing runs through the 2D tile kernels: the outer residual also
    // writes the first sweep of e from zero, and the last post-sweep adds e
    // into x.
    // the mixed solve's first level-0 sweep from e = 0 taken from the FP64
    // outer residual (2D with the fused tile kernels, 3D with the chunk
    // kernels; "fuse 0" / "line 0" run it as a sweep of its own)
    bool fused_mixed() const { return (host_[0].D == 2 ? fuse_ : line_) && pre_ > 0 && post_ > 0; }

    // FP32 V-cycles on dev_[0].bf (already scaled) for the correction e from
    // e = 0.  first_swept: dev_[0].xf already holds the first level-0 sweep.
    // x != nullptr: x += e is applied (fused when possible).  Otherwise e
    // ends in dev_[0].xf (a fixed buffer, so the sequence can be captured).
    void vcycles_f32(int cycles, bool first_swept, double* x)
    {
        const int nl = (int)host_.size();
        std::vector<float*> xs(nl), ts(nl), bs(nl);
        for (int l = 0; l < nl; ++l) {
            xs[l] = dev_[l].xf;
            ts[l] = dev_[l].tf;
            bs[l] = dev_[l].bf;
        }
        rec_phase(rec_iter_, kStageInit, 0);
        if (!first_swept)
            run_vec<0>(VecArgs{xs[0], nullptr, N0()});
        const bool accd = vcycles<float>(xs, ts, bs, cycles, first_swept, x);
        rec_phase(rec_iter_ - 1, kStageCorr, 0);
        if (x && !accd) {
            run_vec<1>(VecArgs{x, xs[0], N0()});
        } else if (!x && xs[0] != dev_[0].xf) {
            MG_HIP(hipMemcpyAsync(dev_[0].xf, xs[0], (size_t)N0() * sizeof(float), hipMemcpyDeviceToDevice, stream_));
        }
    }

    // V-cycles (FP64) or refinement iterations (mixed: FP32 V-cycle, x += e,
    // next residual), replayed from captured hipGraphs when the solver runs on
    // its own stream.  Graphs are keyed on (b, x) (the caller's b: the checks
    // read it) and what they hold; a few are kept so that a stepper
    // alternating between solves on different buffers (a forward and an
    // adjoint solve) does not re-capture each time.
    //
    // Between two graph launches the GPU idles for 8 us (nodes of one graph
    // follow each other without a gap), as long as one and a half launches of
    // a small level: the cycles before the first check run in graphs of 8, 4,
    // 2 and 1, and the checked cycle's graph holds its residual and norms.
    // Langmuir 128^2 FP64, 16 cycles a step: 610 -> 581 us a step.  The
    // longer graphs are captured from the second solve on a pair (b, x) on: a
    // caller with new buffers each time replays one-cycle graphs.
    struct Captured {
        hipGraphExec_t exec = nullptr;
        const void* b = nullptr;
        const void* x = nullptr;
        int flag = 0;
    };
    static constexpr int kGraphs = 32, kPairs = 4, kChain = 8, kChecked = 1 << 16;
    struct GraphCache {
        Captured e[kGraphs];
        int next = 0;
    };
    GraphCache cap64_, cap32_;
    int use_graph_ = 1;
    // the latest pairs solved on
    struct Pair {
        const void* b = nullptr;
        const void* x = nullptr;
    };
    Pair pairs_[kPairs];
    int pair_next_ = 0;

    // whether the pair was solved on before (and note it)
    bool chained(const void* b, const void* x)
    {
        for (const auto& p : pairs_)
            if (p.b == b && p.x == x) return true;
        pairs_[pair_next_] = Pair{b, x};
        pair_next_ = (pair_next_ + 1) % kPairs;
        return false;
    }

    void drop_graph(Captured& c)
    {
        if (c.exec) {
            // (the host saw its norms, not yet its end)
            (void)hipStreamSynchronize(stream_);
            (void)hipGraphExecDestroy(c.exec);
        }
        c = Captured{};
    }
    void drop_graphs()
    {
        for (auto* gc : {&cap64_, &cap32_})
            for (auto& e : gc->e) drop_graph(e);
    }

    template <typename F>
    void replay(GraphCache& gc, const void* b, const void* x, int flag, F&& body)
    {
        if (!use_graph_ || stream_ == nullptr) {
            body();
            return;
        }
        Captured* c = nullptr;
        for (auto& e : gc.e)
            if (e.exec && e.b == b && e.x == x && e.flag == flag) c = &e;
        if (!c) {
            c = &gc.e[gc.next];
            gc.next = (gc.next + 1) % kGraphs;
            drop_graph(*c);
            MG_HIP(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal));
            CaptureGuard guard(stream_);
            body();
            hipGraph_t graph = nullptr;
            guard.release();
            MG_HIP(hipStreamEndCapture(stream_, &graph));
            MG_HIP(hipGraphInstantiate(&c->exec, graph, nullptr, nullptr, 0));
            (void)hipGraphDestroy(graph);
            c->b = b;
            c->x = x;
            c->flag = flag;
        }
        MG_HIP(hipGraphLaunch(c->exec, stream_));
    }

    // body(m) for n = sum m, m a power of two up to kChain (chain) or 1
    template <typename F>
    void replay_runs(GraphCache& gc, const void* b, const void* x, int n, bool chain, F&& body)
    {
        for (int m = chain ? kChain : 1; n > 0; m = std::max(1, m / 2))
            for (; n >= m; n -= m) replay(gc, b, x, m, [&]() { body(m); });
    }

    void cycles_f64(const double* b, double* x, int n, bool chain)
    {
        replay_runs(cap64_, b, x, n, chain, [&](int m) { vcycles_f64(x, m); });
    }

    // one V-cycle, ||b - A x||^2 and ||b||^2 on their way to the host
    void checked_cycle_f64(const double* bs, const double* b, double* x, bool chain)
    {
        auto check = [&]() { outer_residual(bs, b, x, false, false, true); };
        if (chain) {
            replay(cap64_, b, x, 1 | kChecked, [&]() {
                vcycles_f64(x, 1);
                check();
            });
        } else {
            cycles_f64(b, x, 1, false);
            check();
        }
        ++norm_seq_;
    }

    // refinement iterations: FP32 V-cycle on A e = r, x += e, next residual
    // r = b - A x (FP64); norms: also reduce ||r||^2, ||b||^2 for a host check
    void iterate_f32(const double* bs, const double* b, double* x, bool norms)
    {
        const bool fm = fused_mixed();
        vcycles_f32(1, fm, x);
        outer_residual(bs, b, x, true, fm, norms);
    }
    void iterations_f32(const double* bs, const double* b, double* x, int n, bool chain)
    {
        replay_runs(cap32_, b, x, n, chain, [&](int m) {
            for (int i = 0; i < m; ++i) iterate_f32(bs, b, x, false);
        });
    }
    void iteration_f32(const double* bs, const double* b, double* x)
    {
        replay(cap32_, b, x, 1 | kChecked, [&]() { iterate_f32(bs, b, x, true); });
        ++norm_seq_;
    }

    // The residual b - A x.  emit_f32: scaled and in FP32 into dev_[0].bf;
    // first_sweep: and the first sweep of e from zero into dev_[0].xf; norms:
    // ||b - A x||^2 and ||bn||^2 into norms_ (the caller counts them in
    // norm_seq_ once per launch or replay, read_norms waits).
    void outer_residual(const double* b, const double* bn, const double* x, bool emit_f32,
                        bool first_sweep, bool norms)
    {
        const DevLevel L = dl(0);
        const unsigned nb = nblk(L.N);
        DevTable<double> K;
        K.coef = dev_[0].K;
        K.dinv = dev_[0].dinv;
        const bool c = host_[0].compact;
        float* b0 = emit_f32 ? dev_[0].bf : nullptr;
        const float* d32 = dev_[0].dinv32;
        float* e0 = (emit_f32 && first_sweep) ? dev_[0].xf : nullptr;
        const bool dom = line_ && host_[0].D == 3 && c && dev_[0].line_cls >= 0;
        const OuterArgs oa{L, K, x, b, bn, pin_, d32, b0, part_, e0, dom ? dev_[0].line_cls : -1,
                           dom ? K.coef + (int64_t)dev_[0].line_cls * 27 : nullptr};
        if (!norms && emit_f32 && !rec_ && line_ && dev_[0].line_cls >= 0 && host_[0].compact) {
            const LineGeom G = line_geom(0);
            const LineList LL = line_list(0);
            hipLaunchKernelGGL(k_outer_line, dim3(line_grid(LL)), dim3(kMgThreads), 0, stream_, G, LL, oa,
                               K.coef + (int64_t)G.cls_in * 27, host_dinv32(0, G.cls_in));
            MG_HIP(hipGetLastError());
            return;
        }
        // the squared norms only when they are read (norms); otherwise the
        // kernel skips bn and the reductions
#define OUTER(DIM, CMP, F32) \
        do { if (norms) run_outer<DIM, CMP, F32, true>(nb, oa); else run_outer<DIM, CMP, F32, false>(nb, oa); } while (0)
        if (host_[0].D == 2) {
            if (c) { if (emit_f32) OUTER(2, true, true); else OUTER(2, true, false); }
            else { if (emit_f32) OUTER(2, false, true); else OUTER(2, false, false); }
        } else {
            if (c) { if (emit_f32) OUTER(3, true, true); else OUTER(3, true, false); }
            else { if (emit_f32) OUTER(3, false, true); else OUTER(3, false, false); }
        }
#undef OUTER
        MG_HIP(hipGetLastError());
        if (!norms) return;
        hipLaunchKernelGGL(k_reduce2, dim3(1), dim3(kMgThreads), 0, stream_, part_, (int64_t)nb, norms_, norm_count_,
                           pin_ >= 0 ? x : nullptr, bn, pin_, shift_ + 1);
        MG_HIP(hipGetLastError());
    }

    void read_norms(double* rr, double* bb)
    {
        // a short wait watches the box, giving way to the host's other
        // threads between looks (steppers on more threads than cores); a
        // longer one, and one for norms that a failed launch never stored,
        // synchronises
        const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(2000);
        while (__atomic_load_n(&norms_->seq, __ATOMIC_ACQUIRE) < norm_seq_) {
            if (std::chrono::steady_clock::now() > until) {
                MG_HIP(hipStreamSynchronize(stream_));
                norm_seq_ = __atomic_load_n(&norms_->seq, __ATOMIC_ACQUIRE);
                break;
            }
            std::this_thread::yield();
        }
        *rr = norms_->rr;
        *bb = norms_->bb;
    }
};

// ---- batched launches of recorded solves -----------------------------------
// Ops of all solvers are ordered by (key, kind, solver); each run of equal
// (key, kind) becomes one launch of the kind's batched kernel over the
// concatenated blocks of its solvers.  Every solver's ops keep their own
// order (keys grow along each solver's sequence), and ops sharing a launch
// belong to different, independent solvers.
struct MgBatchGroup {
    uint16_t kind;
    unsigned blocks;
    int n;
    size_t args_off, first_off;
};

struct MgBatchPlan {
    std::vector<MgBatchGroup> groups;
    void* dev = nullptr;
    size_t bytes = 0;
    int64_t ops = 0;
    ~MgBatchPlan() { release(); }
    void release()
    {
        if (dev) (void)hipFree(dev);
        dev = nullptr;
        bytes = 0;
        groups.clear();
        ops = 0;
    }
};

void mg_batch_build(const std::vector<const std::vector<MgRecOp>*>& per, MgBatchPlan& plan)
{
    plan.release();
    struct E {
        uint32_t key;
        uint16_t kind;
        int inst;
        const MgRecOp* op;
    };
    std::vector<E> all;
    for (int i = 0; i < (int)per.size(); ++i)
        for (const auto& op : *per[i]) {
            if (op.kind >= kKindCount) throw std::logic_error("hip_multigrid: unknown recorded kind");
            all.push_back(E{op.key, op.kind, i, &op});
        }
    std::stable_sort(all.begin(), all.end(), [](const E& a, const E& b) {
        if (a.key != b.key) return a.key < b.key;
        if (a.kind != b.kind) return a.kind < b.kind;
        return a.inst < b.inst;
    });
    std::vector<unsigned char> host;
    auto align16 = [&]() { host.resize((host.size() + 15) & ~(size_t)15, 0); };
    for (size_t a = 0; a < all.size();) {
        size_t b = a;
        while (b < all.size() && all[b].key == all[a].key && all[b].kind == all[a].kind) ++b;
        MgBatchGroup g{};
        g.kind = all[a].kind;
        g.n = (int)(b - a);
        const size_t asz = all[a].op->args.size();
        align16();
        g.args_off = host.size();
        for (size_t k = a; k < b; ++k) {
            if (all[k].op->args.size() != asz) throw std::logic_error("hip_multigrid: argument size mismatch");
            host.insert(host.end(), all[k].op->args.begin(), all[k].op->args.end());
        }
        align16();
        g.first_off = host.size();
        uint64_t blocks = 0;
        for (size_t k = a; k < b; ++k) {
            const unsigned f = (unsigned)blocks;
            const unsigned char* q = reinterpret_cast<const unsigned char*>(&f);
            host.insert(host.end(), q, q + sizeof(unsigned));
            blocks += all[k].op->nblocks;
        }
        if (blocks > 0x7fffffffull) throw std::runtime_error("hip_multigrid: batched launch too large");
        g.blocks = (unsigned)blocks;
        if (g.blocks > 0) plan.groups.push_back(g);
        a = b;
    }
    plan.ops = (int64_t)all.size();
    plan.bytes = std::max<size_t>(host.size(), 16);
    MG_HIP(hipMalloc(&plan.dev, plan.bytes));
    if (!host.empty()) MG_HIP(hipMemcpy(plan.dev, host.data(), host.size(), hipMemcpyHostToDevice));
}

void mg_batch_launch(const MgBatchPlan& plan, hipStream_t st)
{
    const unsigned char* base = static_cast<const unsigned char*>(plan.dev);
    for (const auto& g : plan.groups) {
        const void* a = base + g.args_off;
        const unsigned* f = reinterpret_cast<const unsigned*>(base + g.first_off);
        const dim3 grid(g.blocks);
        const uint16_t k = g.kind;
        if (k < kKindDown) {
#define SMT(T, C, P, A)                                                                                                   \
    hipLaunchKernelGGL((k_smooth_tile_many<T, C, P, A>), grid, dim3(TileGeom<T, false>::threads), 0, st,                     \
                       static_cast<const SmoothTileArgs<T>*>(a), f, g.n)
            switch (k - kKindSmooth) {
            case 0: SMT(float, false, false, false); break;
            case 1: SMT(float, false, false, true); break;
            case 2: SMT(float, false, true, false); break;
            case 3: SMT(float, false, true, true); break;
            case 4: SMT(float, true, false, false); break;
            case 5: SMT(float, true, false, true); break;
            case 6: SMT(float, true, true, false); break;
            case 7: SMT(float, true, true, true); break;
            case 8: SMT(double, false, false, false); break;
            case 10: SMT(double, false, true, false); break;
            case 12: SMT(double, true, false, false); break;
            case 14: SMT(double, true, true, false); break;
            default: throw std::logic_error("hip_multigrid: unknown recorded kind");
            }
#undef SMT
        } else if (k < kKindRR) {
#define DWN(T, C)                                                                                                         \
    hipLaunchKernelGGL((k_down_tile_many<T, C>), grid, dim3(TileGeom<T, false>::threads), 0, st,                             \
                       static_cast<const DownTileArgs<T>*>(a), f, g.n)
            switch (k - kKindDown) {
            case 0: DWN(float, false); break;
            case 1: DWN(float, true); break;
            case 2: DWN(double, false); break;
            default: DWN(double, true); break;
            }
#undef DWN
        } else if (k < kKindCoarse) {
#define RRL(T, C) hipLaunchKernelGGL((k_resid_restrict_many<T, C>), grid, dim3(kMgThreads), 0, st, static_cast<const ResidRestrictArgs<T>*>(a), f, g.n)
            switch (k - kKindRR) {
            case 0: RRL(float, false); break;
            case 1: RRL(float, true); break;
            case 2: RRL(double, false); break;
            default: RRL(double, true); break;
            }
#undef RRL
        } else if (k < kKindOuter) {
            if (k - kKindCoarse)
                hipLaunchKernelGGL((k_coarse_solve_many<double>), grid, dim3(kMgThreads), 0, st,
                                   static_cast<const CoarseArgs<double>*>(a), f, g.n);
            else
                hipLaunchKernelGGL((k_coarse_solve_many<float>), grid, dim3(kMgThreads), 0, st,
                                   static_cast<const CoarseArgs<float>*>(a), f, g.n);
        } else if (k < kKindVec) {
            const OuterArgs* oa = static_cast<const OuterArgs*>(a);
#define OUT(C, F, N) hipLaunchKernelGGL((k_outer_residual_many<2, C, F, N>), grid, dim3(kMgThreads), 0, st, oa, f, g.n)
            switch (k - kKindOuter) {
            case 0: OUT(false, false, false); break;
            case 1: OUT(false, true, false); break;
            case 2: OUT(true, false, false); break;
            case 3: OUT(true, true, false); break;
            case 4: OUT(false, false, true); break;
            case 5: OUT(false, true, true); break;
            case 6: OUT(true, false, true); break;
            default: OUT(true, true, true); break;
            }
#undef OUT
        } else if (k < kKindHadamard) {
            const VecArgs* va = static_cast<const VecArgs*>(a);
            switch (k - kKindVec) {
            case 0: hipLaunchKernelGGL((k_vec_many<0>), grid, dim3(kMgThreads), 0, st, va, f, g.n); break;
            case 1: hipLaunchKernelGGL((k_vec_many<1>), grid, dim3(kMgThreads), 0, st, va, f, g.n); break;
            default: hipLaunchKernelGGL((k_vec_many<2>), grid, dim3(kMgThreads), 0, st, va, f, g.n); break;
            }
        } else {
            hipLaunchKernelGGL((k_hadamard_many<double>), grid, dim3(kMgThreads), 0, st,
                               static_cast<const HadamardArgs<double>*>(a), f, g.n);
        }
    }
    MG_HIP(hipGetLastError());
}

}  // namespace psum_hip

// ============================================================ plugin ABI

namespace {

std::map<std::string, func_table>& registry()
{
    static std::map<std::string, func_table> r;
    return r;
}

template <bool MIXED>
psum_field_solver_handle mg_init()
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n < 1)
        throw std::runtime_error(MIXED ? "hip_multigrid32f_gpu: no GPU device available"
                                       : "hip_multigrid_gpu: no GPU device available");
    return new HipMultigrid(MIXED);
}

void mg_set_matrix(psum_field_solver_handle h, unsigned long long n_row, unsigned long long n_col,
                   unsigned long long nnz, unsigned long long* rows, unsigned long long* cols,
                   double* vals)
{
    static_cast<HipMultigrid*>(h)->set_matrix(n_row, n_col, nnz, rows, cols, vals);
}

void mg_solve(psum_field_solver_handle h, double* b, double* x)
{
    static_cast<HipMultigrid*>(h)->solve(b, x, true);
}

void mg_set_options(psum_field_solver_handle h, const char* o)
{
    static_cast<HipMultigrid*>(h)->set_options(o);
}

void mg_set_replace(psum_field_solver_handle h, unsigned long long n, unsigned long long* i, double* v)
{
    static_cast<HipMultigrid*>(h)->set_source_replace(n, i, v);
}

void mg_set_addback(psum_field_solver_handle h, unsigned long long n, unsigned long long* i, double* v)
{
    static_cast<HipMultigrid*>(h)->set_source_addback(n, i, v);
}

void mg_free(psum_field_solver_handle h) { delete static_cast<HipMultigrid*>(h); }

const int registered = []() {
    func_table t64{mg_init<false>, mg_set_matrix, mg_solve, mg_set_options, mg_set_replace, mg_set_addback, mg_free};
    func_table t32{mg_init<true>, mg_set_matrix, mg_solve, mg_set_options, mg_set_replace, mg_set_addback, mg_free};
    registry()["hip_multigrid_gpu"] = t64;
    registry()["hip_multigrid32f_gpu"] = t32;
    return 0;
}();

template <typename F>
int guarded(F&& f)
{
    try {
        f();
        return PSUM_OK;
    } catch (const std::invalid_argument& e) {
        set_error(e.what());
        return PSUM_ERR_ARG;
    } catch (const std::exception& e) {
        set_error(e.what());
        return PSUM_ERR_UNSUPPORTED;
    }
}

}  // namespace

namespace psum_hip {

// in-library access for the step engine
HipMultigrid* mg_create(bool mixed) { return new HipMultigrid(mixed); }
void mg_destroy(HipMultigrid* h) { delete h; }
void mg_set_options(HipMultigrid* h, const char* o) { h->set_options(o); }
void mg_set_tuning(HipMultigrid* h, const char* o) { h->set_tuning(o); }
void mg_set_smoothing(HipMultigrid* h, int pre, int post) { h->set_smoothing(pre, post); }
void mg_set_matrix(HipMultigrid* h, unsigned long long n, unsigned long long nnz,
                   const unsigned long long* r, const unsigned long long* c, const double* v)
{
    h->set_matrix(n, n, nnz, r, c, v);
}
void mg_set_replace(HipMultigrid* h, unsigned long long n, const unsigned long long* i, const double* v)
{
    h->set_source_replace(n, i, v);
}
void mg_set_stream(HipMultigrid* h, hipStream_t s) { h->set_stream(s); }
void mg_solve(HipMultigrid* h, double* b, double* x, bool sync) { h->solve(b, x, sync); }
void mg_solve_homogeneous(HipMultigrid* h, double* b, double* x) { h->solve(b, x, false, true); }
int mg_predicted(HipMultigrid* h) { return h->predicted(); }
void mg_set_fixed_cycles(HipMultigrid* h, int cycles) { h->set_fixed_cycles(cycles); }
void mg_set_predicted(HipMultigrid* h, int p) { h->set_predicted(p); }
int mg_last_cycles(HipMultigrid* h) { return h->last_cycles(); }
double mg_last_rel(HipMultigrid* h) { return h->last_rel(); }
const double* mg_solve_begin(HipMultigrid* h, double* b, const double* mean_part)
{
    return h->solve_begin(b, false, mean_part);
}
bool mg_takes_mean(HipMultigrid* h) { return h->takes_mean(); }
void mg_solve_core(HipMultigrid* h, const double* b, const double* bs, double* x) { h->solve_core(b, bs, x); }
const double* mg_gauge(HipMultigrid* h, const double* b, const double* x) { return h->gauge(b, x); }
bool mg_recordable(HipMultigrid* h) { return h->recordable(); }
const double* mg_core_rhs(HipMultigrid* h, double* b)
{
    double* p = h->pin_rhs();
    return p ? p : b;
}
void mg_record_core(HipMultigrid* h, const double* b, const double* bs, double* x,
                    std::vector<MgRecOp>& ops)
{
    h->record_core(b, bs, x, ops);
}
MgBatchPlan* mg_batch_plan_create() { return new MgBatchPlan(); }
void mg_batch_plan_destroy(MgBatchPlan* p) { delete p; }
void mg_batch_plan_build(MgBatchPlan* p, const std::vector<const std::vector<MgRecOp>*>& per)
{
    mg_batch_build(per, *p);
}
void mg_batch_plan_launch(const MgBatchPlan* p, hipStream_t st) { mg_batch_launch(*p, st); }
int64_t mg_batch_plan_launches(const MgBatchPlan* p) { return (int64_t)p->groups.size(); }
int64_t mg_batch_plan_ops(const MgBatchPlan* p) { return p->ops; }

}  // namespace psum_hip

extern "C" {

void register_solver(const char* name, func_table table) { registry()[name] = table; }

func_table get_solver_funcs(const char* name)
{
    func_table ans{};
    ans.init = nullptr;
    auto& reg = registry();
    auto it = reg.find(name ? name : "");
    if (it != reg.end()) return it->second;
    return ans;
}

void* psum_solver_create(const char* kind)
{
    func_table t = get_solver_funcs(kind);
    if (!t.init) {
        set_error(std::string("psum_solver_create: unknown backend ") + (kind ? kind : "(null)"));
        return nullptr;
    }
    void* h = nullptr;
    if (guarded([&]() { h = t.init(); }) != PSUM_OK) return nullptr;
    return h;
}

int psum_solver_set_options(void* h, const char* options)
{
    if (!h) { set_error("psum_solver_set_options: null handle"); return PSUM_ERR_ARG; }
    return guarded([&]() { static_cast<HipMultigrid*>(h)->set_options(options); });
}

int psum_solver_set_matrix(void* h, unsigned long long n_row, unsigned long long n_col,
                           unsigned long long nnz, unsigned long long* rows,
                           unsigned long long* cols, double* vals)
{
    if (!h) { set_error("psum_solver_set_matrix: null handle"); return PSUM_ERR_ARG; }
    return guarded([&]() { static_cast<HipMultigrid*>(h)->set_matrix(n_row, n_col, nnz, rows, cols, vals); });
}

int psum_solver_set_source_replace(void* h, unsigned long long n, unsigned long long* idxs, double* vals)
{
    if (!h) { set_error("null handle"); return PSUM_ERR_ARG; }
    return guarded([&]() { static_cast<HipMultigrid*>(h)->set_source_replace(n, idxs, vals); });
}

int psum_solver_set_source_addback(void* h, unsigned long long n, unsigned long long* idxs, double* vals)
{
    if (!h) { set_error("null handle"); return PSUM_ERR_ARG; }
    return guarded([&]() { static_cast<HipMultigrid*>(h)->set_source_addback(n, idxs, vals); });
}

int psum_solver_solve(void* h, double* b_dev, double* x_dev)
{
    if (!h) { set_error("null handle"); return PSUM_ERR_ARG; }
    return guarded([&]() { static_cast<HipMultigrid*>(h)->solve(b_dev, x_dev, true); });
}

int psum_solver_stats(void* h, int* cycles, double* rel_res)
{
    if (!h) { set_error("null handle"); return PSUM_ERR_ARG; }
    auto* m = static_cast<HipMultigrid*>(h);
    if (cycles) *cycles = m->last_cycles();
    if (rel_res) *rel_res = m->last_rel();
    return PSUM_OK;
}

void psum_solver_free(void* h) { delete static_cast<HipMultigrid*>(h); }

}  // extern "C"
