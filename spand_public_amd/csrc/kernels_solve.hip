// Preconditioner-apply sweeps and FP64 Krylov vector kernels for gfx950.
//
// Tree::solve (src/tree.cpp:1610-1635) replays the recorded operations forward then
// backward on per-cluster segments of one vector; here the ops of one ND level run as three
// launches per direction (tasks.hpp) on a block of nrhs right-hand sides stored interleaved,
// x[(xoff + i) * nrhs + r]. They replace
//   E      ScalingLLT fwd/bwd             src/operations.cpp:95-103 (cblas_dtrsv)
//   G      GemmSymmOut/In fwd/bwd         src/operations.cpp:55-93  (cblas_dgemv)
//   W      ScalingLLT, Orthogonal, Merge  src/operations.cpp:95-103,149-158,166-192
// The Krylov kernels back cg (src/is.cpp:39-121): CSR SpMV and deterministic two-pass dots.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "kernels.hpp"
#include "tasks.hpp"

namespace spand {

// Device-memory pointers that the task records carry as plain pointers: accessed through a
// pointer in the global address space, the compiler emits global_* instead of flat_*
// instructions (a flat access also holds the LDS wait counter).
template <typename X>
using gptr = __attribute__((address_space(1))) X*;
template <typename X>
__device__ __attribute__((always_inline)) inline gptr<X> gp(X* p) {
    return (gptr<X>)p;
}

constexpr int NT = 256;
// Segments are FP64 whatever the factor's element type T: an FP32 factor is read as FP32 and
// applied in FP64 arithmetic, so the preconditioner stays one fixed linear operator.
using VT = double;
static inline int grid_for(size_t n) {
    size_t g = (n + NT - 1) / NT;
    return (int)(g > 65536 ? 65536 : (g == 0 ? 1 : g));
}

// ---------------------------------------------------------------------------------------
// Element (i, r) of the caller's vector block lives at b[i * sx + r * sr] (column-major:
// sx = 1, sr = ld; interleaved: sx = nrhs, sr = 1).
template <typename T>
__global__ void __launch_bounds__(NT) k_perm_in(const double* b, size_t sx, size_t sr, int nrhs, const int* perm,
                                                int N, VT* ws) {
    size_t n = (size_t)N * nrhs;
    for (size_t idx = (size_t)blockIdx.x * NT + threadIdx.x; idx < n; idx += (size_t)gridDim.x * NT) {
        int i = (int)(idx / nrhs), r = (int)(idx % nrhs);
        ws[idx] = b[(size_t)perm[i] * sx + (size_t)r * sr];
    }
}
template <typename T>
__global__ void __launch_bounds__(NT) k_perm_out(const VT* ws, const int* perm, int N, int nrhs, double* x, size_t sx,
                                                 size_t sr) {
    size_t n = (size_t)N * nrhs;
    for (size_t idx = (size_t)blockIdx.x * NT + threadIdx.x; idx < n; idx += (size_t)gridDim.x * NT) {
        int i = (int)(idx / nrhs), r = (int)(idx % nrhs);
        x[(size_t)perm[i] * sx + (size_t)r * sr] = ws[idx];
    }
}

// column-major (ld) <-> interleaved conversions of an N x nrhs block
__global__ void __launch_bounds__(NT) k_cm2il(const double* src, int ld, int N, int nrhs, double* dst) {
    size_t n = (size_t)N * nrhs;
    for (size_t idx = (size_t)blockIdx.x * NT + threadIdx.x; idx < n; idx += (size_t)gridDim.x * NT) {
        int i = (int)(idx / nrhs), r = (int)(idx % nrhs);
        dst[idx] = src[(size_t)i + (size_t)r * ld];
    }
}
__global__ void __launch_bounds__(NT) k_il2cm(const double* src, int N, int nrhs, double* dst, int ld) {
    size_t n = (size_t)N * nrhs;
    for (size_t idx = (size_t)blockIdx.x * NT + threadIdx.x; idx < n; idx += (size_t)gridDim.x * NT) {
        int i = (int)(idx / nrhs), r = (int)(idx % nrhs);
        dst[(size_t)i + (size_t)r * ld] = src[idx];
    }
}

// ---------------------------------------------------------------------------------------
// mv phases (task layouts in tasks.hpp), on the FP64 matrix cores whatever the factor's type.
// A chunk is 16 outputs; its inner positions are taken 16 at a time (a step), and step s of
// the chunk belongs to wavefront s % nw of the nw that share the chunk.
//   * Each wavefront reads the chunk's term records itself, one lane per term, scans their
//     step counts, and finds a step's term by a ballot over the lanes: the records cost one
//     memory round trip whatever their number, and no LDS.
//   * A step's matrix entries are loaded straight into the operand layout (lane l: output
//     l % 16, inner positions 4 (l / 16) + q, q = 0..3), with no staging: along a column of A
//     when not transposed (16 contiguous entries a column), along 4 contiguous entries a lane
//     when transposed. The next step's loads are issued before a step's products.
//   * Up to 4 right-hand sides use v_mfma_f64_4x4x4 (four blocks of 4 outputs; a quarter of
//     the 16x16x4's cycles), up to 16 one v_mfma_f64_16x16x4 tile, up to 32 two.
// The matrix instructions add their four products in inner order by fused multiply-adds, so
// an output's sum does not depend on the number of right-hand sides.
// Bound by the launch and the chain chunk -> terms -> entries for most phases (a level holds
// few outputs), by the factor's bytes for the largest. 16 outputs a chunk and 16 positions a
// step keep the padding of short clusters (10 to 60 rows at the lower levels) small.
// Measured against six phases per level and direction staged through LDS with partial sums
// added by second launches: 64^3 Laplacian, FP64 factor (619 MB), 4 columns 2.92 -> 0.81 ms;
// 512^2, 32 columns 4.98 -> 1.00 ms; 40^2, one column 273 -> 89 us.
constexpr int WAVE = 64;
using d4 = double __attribute__((ext_vector_type(4)));

template <typename T>
struct MvStep {  // one step's operands
    T a[4];
    double x[2][4];
};

// Records of a wavefront's terms, one lane each, and where each term's steps start.
struct MvLane {
    const void* A;
    const int* perm;
    int ld, lo, hi, xsrc, trans, off;
};

__device__ inline int rl(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
template <typename X>
__device__ inline X* rlp(X* p, int lane) {
    const unsigned long long u = (unsigned long long)p;
    const unsigned lo = (unsigned)rl((int)(unsigned)u, lane), hi = (unsigned)rl((int)(unsigned)(u >> 32), lane);
    return (X*)(((unsigned long long)hi << 32) | lo);
}

// Operands of step s: term t of the lanes, inner positions [j, j + 16) clipped to hi. Rows past
// the chunk's outputs read its last row (their sums are not stored); positions past hi are
// zero in both operands.
template <typename T, int CT>
__device__ inline void mv_load(const MvLane& L, unsigned long long m, int s, int o0, int no, const double* ws, int nrhs,
                               int r0, MvStep<T>& st) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int t = __popcll(m) - 1;
    const int j = rl(L.lo, t) + (s - rl(L.off, t)) * MV_STEP;
    const int nv = min(MV_STEP, rl(L.hi, t) - j);
    const int ld = rl(L.ld, t), xs = rl(L.xsrc, t);
    const gptr<const T> A = gp(reinterpret_cast<const T*>(rlp(L.A, t)));
    const int row = o0 + min(lane & 15, no - 1), kk = 4 * (lane >> 4);
    if (rl(L.trans, t)) {
        const gptr<const T> p = A + (size_t)row * ld + j;
        if (nv == MV_STEP) {
#pragma unroll
            for (int q = 0; q < 4; q++) st.a[q] = p[kk + q];
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const T v = p[min(kk + q, nv - 1)];
                st.a[q] = kk + q < nv ? v : T(0);
            }
        }
    } else {
        const gptr<const T> p = A + row + (size_t)j * ld;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const T v = p[(size_t)min(kk + q, nv - 1) * ld];
            st.a[q] = kk + q < nv ? v : T(0);
        }
    }
    const gptr<const int> perm = gp(rlp(L.perm, t));
    const gptr<const double> x = gp(ws);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int k = j + min(kk + q, nv - 1);
        const size_t e = (size_t)(xs + (perm ? perm[k] : k)) * nrhs;
#pragma unroll
        for (int c = 0; c < (CT == 0 ? 1 : CT); c++) {
            const int r = min(r0 + (CT == 0 ? lane & 3 : 16 * c + (lane & 15)), nrhs - 1);
            const double v = x[e + r];
            st.x[c][q] = kk + q < nv ? v : 0.0;
        }
    }
}

// One chunk by the nw wavefronts of a group (sub: this one's place in it); red holds the
// group's (nw - 1) x 64 lanes x NACC partial sums. Every wavefront of the workgroup calls it
// (live: the group has a chunk) because the sums meet at workgroup barriers.
template <typename T, int CT>
__device__ inline void mv_chunk(const MvDevPhase& ph, int ci, bool live, int sub, double* red, double* ws, int nrhs,
                                int r0) {
    constexpr int NACC = CT == 0 ? 1 : 4 * CT;
    const int lane = threadIdx.x & (WAVE - 1), nw = ph.nw;
    double acc1 = 0.0;
    d4 acc[2] = {};
    MvChunk ch{};
    if (live) {
        ch = ph.chunks[ci];
        for (int kb = ch.k0; kb < ch.k1; kb += WAVE) {
            const int nt = min(WAVE, ch.k1 - kb);
            MvLane L{};
            int n = 0;
            if (lane < nt) {
                const MvTerm tm = ph.terms[kb + lane];
                L.A = tm.A;
                L.perm = tm.perm;
                L.ld = tm.ld;
                L.xsrc = tm.xsrc;
                L.trans = tm.flags & MV_TRANS;
                L.lo = (tm.flags & MV_TRI_UP) ? min(tm.len, ch.o0) : 0;
                L.hi = (tm.flags & MV_TRI_LO) ? min(tm.len, ch.o0 + MV_ROWS) : tm.len;
                n = (max(0, L.hi - L.lo) + MV_STEP - 1) / MV_STEP;
            }
            int incl = n;  // inclusive scan over the wavefront
#pragma unroll
            for (int d = 1; d < WAVE; d <<= 1) {
                const int v = __shfl_up(incl, d);
                if (lane >= d) incl += v;
            }
            L.off = incl - n;
            const int total = rl(incl, WAVE - 1);
            // the term of step s: the last one starting at or before it
            auto at = [&](int s) { return __ballot(lane < nt && L.off <= s); };
            MvStep<T> cur, nxt;
            if (sub < total) mv_load<T, CT>(L, at(sub), sub, ch.o0, ch.no, ws, nrhs, r0, cur);
            for (int s = sub; s < total; s += nw) {
                const int s1 = s + nw;
                if (s1 < total) mv_load<T, CT>(L, at(s1), s1, ch.o0, ch.no, ws, nrhs, r0, nxt);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const double a = (double)cur.a[q];
                    if (CT == 0) {
                        acc1 = __builtin_amdgcn_mfma_f64_4x4x4f64(a, cur.x[0][q], acc1, 0, 0, 0);
                    } else {
#pragma unroll
                        for (int c = 0; c < CT; c++)
                            acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, cur.x[c][q], acc[c], 0, 0, 0);
                    }
                }
                cur = nxt;
            }
        }
    }
    if (nw > 1) {
        double* mine = red + (size_t)(sub - 1) * WAVE * NACC + lane;
        if (sub > 0) {
            if (CT == 0) mine[0] = acc1;
#pragma unroll
            for (int u = 0; u < (CT == 0 ? 0 : NACC); u++) mine[u * WAVE] = acc[u / 4][u % 4];
        }
        __syncthreads();
        if (sub == 0)
            for (int w = 0; w < nw - 1; w++) {
                const double* p = red + (size_t)w * WAVE * NACC + lane;
                if (CT == 0) acc1 += p[0];
#pragma unroll
                for (int u = 0; u < (CT == 0 ? 0 : NACC); u++) acc[u / 4][u % 4] += p[u * WAVE];
            }
    }
    if (live && sub == 0) {
        auto put = [&](int i, int r, double v) {  // output i of the chunk, right-hand side r
            if (i >= ch.no || r >= nrhs) return;
            const int o = ch.o0 + i;
            const gptr<double> y = gp(ws) + (size_t)(ch.xdst + (ch.dperm ? gp(ch.dperm)[o] : o)) * nrhs + r;
            *y = ch.mode == MV_SUB ? *y - v : v;
        };
        if (CT == 0) {  // 4x4x4: lane l holds output 4 ((l % 16) / 4) + l / 16, right-hand side l % 4
            put(4 * ((lane & 15) >> 2) + (lane >> 4), lane & 3, acc1);
        } else {  // 16x16x4: register v of lane l holds output l / 16 + 4 v, right-hand side l % 16
#pragma unroll
            for (int u = 0; u < NACC; u++)
                put((lane >> 4) + 4 * (u % 4), r0 + 16 * (u / 4) + (lane & 15), acc[u / 4][u % 4]);
        }
    }
}

// Consecutive workgroups run on different XCDs (block b on XCD b % 8): chunk ranges are dealt
// out so that neighbouring chunks, which share sources and the cache lines of A's columns,
// meet in one L2. Grid: (8 x workgroups per XCD, blocks of 16 CT right-hand sides).
constexpr int XCDS = 8;
template <typename T, int CT>
__global__ void __launch_bounds__(1024) k_mv(MvDevPhase ph, double* ws, int nrhs) {
    extern __shared__ double mv_red[];
    constexpr int NACC = CT == 0 ? 1 : 4 * CT;
    const int groups = blockDim.x / WAVE / ph.nw;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int blk = (blockIdx.x % XCDS) * (gridDim.x / XCDS) + blockIdx.x / XCDS;
    const int g = wv / ph.nw, ci = blk * groups + g;
    mv_chunk<T, CT>(ph, ci, ci < ph.nchunks, wv % ph.nw, mv_red + (size_t)g * (ph.nw - 1) * WAVE * NACC, ws, nrhs,
                    blockIdx.y * (CT == 0 ? 4 : 16 * CT));
}

// Consecutive phases of little work in one workgroup, a barrier between them instead of a
// launch (about 4.5 us each in a replayed graph, against 2-3 us for such a phase here).
template <typename T, int CT>
__global__ void __launch_bounds__(1024) k_mv_tail(MvTail tail, double* ws, int nrhs) {
    extern __shared__ double mv_red[];
    constexpr int NACC = CT == 0 ? 1 : 4 * CT;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    for (int p = 0; p < tail.n; p++) {
        const MvDevPhase ph = tail.ph[p];
        const int groups = MV_NW_MAX / ph.nw, g = wv / ph.nw;
        for (int r0 = 0; r0 < nrhs; r0 += (CT == 0 ? 4 : 16 * CT))
            for (int c0 = 0; c0 < ph.nchunks; c0 += groups) {
                mv_chunk<T, CT>(ph, c0 + g, c0 + g < ph.nchunks, wv % ph.nw,
                                mv_red + (size_t)g * (ph.nw - 1) * WAVE * NACC, ws, nrhs, r0);
                if (ph.nw > 1) __syncthreads();  // the partial sums are read before the next chunk's
            }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------------------
// Compact-WY factors of the Orthogonal ops (task layout in tasks.hpp): Ve = V with its unit
// diagonal and zeros above; S = -diag(1 / tau) - stril(Ve^T Ve).
template <typename T>
__global__ void __launch_bounds__(NT) k_wy_explicit(const WyTask* tasks) {
    const WyTask t = tasks[blockIdx.x];
    const T* V = reinterpret_cast<const T*>(t.V);
    double* Ve = t.Ve;
    const size_t n = (size_t)t.m * t.k;
    for (size_t idx = (size_t)blockIdx.y * NT + threadIdx.x; idx < n; idx += (size_t)gridDim.y * NT) {
        const int i = (int)(idx % t.m), c = (int)(idx / t.m);
        Ve[idx] = i == c ? 1.0 : (i > c ? (double)V[idx] : 0.0);
    }
    // S on and above the diagonal
    const T* tau = reinterpret_cast<const T*>(t.tau);
    double* S = t.S;
    const size_t kk = (size_t)t.k * t.k;
    for (size_t idx = (size_t)blockIdx.y * NT + threadIdx.x; idx < kk; idx += (size_t)gridDim.y * NT) {
        const int a = (int)(idx % t.k), c = (int)(idx / t.k);
        if (a <= c) S[idx] = a == c ? -(1.0 / (double)tau[a]) : 0.0;
    }
}

// one workgroup per 32 x 32 tile (a0, c0), a0 <= c0, of one op's Gram matrix; entry
// (a, c), a < c, goes to S(c, a)
__global__ void __launch_bounds__(NT) k_wy_gram(const WyTask* tasks, const int4* tiles) {
    constexpr int GT = 32;  // tile edge (the host plans 32 x 32 tiles)
    __shared__ double As[GT][GT + 1], Cs[GT][GT + 1];
    const int4 tl = tiles[blockIdx.x];  // (task, a0, c0, unused)
    const WyTask t = tasks[tl.x];
    const int a0 = tl.y, c0 = tl.z, m = t.m, k = t.k;
    const double* Ve = t.Ve;
    const int tid = threadIdx.x;
    // thread -> 4 outputs: a = a0 + tid % 32, c = c0 + (tid / 32) * 4 + q
    const int ta = tid % GT, tc0 = (tid / GT) * 4;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i0 = c0; i0 < m; i0 += GT) {  // Ve(i, c) = 0 for i < c
        const int ni = min(GT, m - i0);
        for (int idx = tid; idx < GT * GT; idx += NT) {
            const int ii = idx % GT, cc = idx / GT;
            As[ii][cc] = (ii < ni && a0 + cc < k) ? Ve[(i0 + ii) + (size_t)(a0 + cc) * m] : 0.0;
            Cs[ii][cc] = (ii < ni && c0 + cc < k) ? Ve[(i0 + ii) + (size_t)(c0 + cc) * m] : 0.0;
        }
        __syncthreads();
        for (int ii = 0; ii < ni; ii++) {
            const double a = As[ii][ta];
#pragma unroll
            for (int q = 0; q < 4; q++) acc[q] += a * Cs[ii][tc0 + q];
        }
        __syncthreads();
    }
    double* S = t.S;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int a = a0 + ta, c = c0 + tc0 + q;
        if (a < k && c < k && a < c) S[c + (size_t)a * k] = -acc[q];
    }
}

template <typename T>
__global__ void __launch_bounds__(NT) k_merge(const MergeTask* tasks, const int2* children, VT* ws, int nrhs, int fwd) {
    const MergeTask t = tasks[blockIdx.x];
    int k = 0;
    for (int c = t.c0; c < t.c1; c++) {
        const int2 ch = children[c];  // (xoff, size)
        const int n = ch.y * nrhs;
        VT* P = ws + (size_t)(t.pxoff + k) * nrhs;
        VT* Cx = ws + (size_t)ch.x * nrhs;
        if (fwd)
            for (int i = threadIdx.x; i < n; i += NT) P[i] = Cx[i];
        else
            for (int i = threadIdx.x; i < n; i += NT) Cx[i] = P[i];
        k += ch.y;
    }
}

// ---------------------------------------------------------------------------------------
// FP64 Krylov kernels
__global__ void __launch_bounds__(NT) k_spmv(int N, const int* rowptr, const int* colidx, const double* val,
                                             const double* x, double* y, int nrhs) {
    size_t n = (size_t)N * nrhs;
    for (size_t idx = (size_t)blockIdx.x * NT + threadIdx.x; idx < n; idx += (size_t)gridDim.x * NT) {
        int i = (int)(idx / nrhs), r = (int)(idx % nrhs);
        double acc = 0.0;
        for (int k = rowptr[i]; k < rowptr[i + 1]; k++) acc += val[k] * x[(size_t)colidx[k] * nrhs + r];
        y[idx] = acc;
    }
}

// Sampled outer product on A's pattern: for stored entry p = (i, j) (CSR position, row i),
// out[csc_of[p]] = alpha * sum over r of u(i, r) v(j, r), the right-hand sides in
// increasing r; u, v column-major with leading dimension ld. OUTER_LANES lanes per row, one
// stored entry each at a time (a row of a grid's matrix holds 5 or 7): one thread per row
// walked them in turn, a chain of entries times right-hand sides with too few wavefronts to
// hide it. OUTER_R right-hand sides' loads are in flight together. 300 x 300 grid, 16 right-hand
// sides: 43.5 -> 26.8 us.
constexpr int OUTER_LANES = 8, OUTER_R = 8;
__global__ void __launch_bounds__(NT) k_sampled_outer(int N, const int* rowptr, const int* colidx, const int* csc_of,
                                                      const double* u, const double* v, int nrhs, int ld,
                                                      double alpha, double* out) {
    const int sub = threadIdx.x % OUTER_LANES, rows = NT / OUTER_LANES;
    for (int i = blockIdx.x * rows + threadIdx.x / OUTER_LANES; i < N; i += gridDim.x * rows) {
        const int end = rowptr[i + 1];
        for (int p = rowptr[i] + sub; p < end; p += OUTER_LANES) {
            const int j = colidx[p], at = csc_of[p];
            double acc = 0.0;
            int r = 0;
            for (; r + OUTER_R <= nrhs; r += OUTER_R) {
                double a[OUTER_R], b[OUTER_R];
#pragma unroll
                for (int q = 0; q < OUTER_R; q++) {
                    a[q] = u[i + (size_t)(r + q) * ld];
                    b[q] = v[j + (size_t)(r + q) * ld];
                }
#pragma unroll
                for (int q = 0; q < OUTER_R; q++) acc = fma(a[q], b[q], acc);
            }
            for (; r < nrhs; r++) acc = fma(u[i + (size_t)r * ld], v[j + (size_t)r * ld], acc);
            out[at] = alpha * acc;
        }
    }
}

constexpr int DOT_BLOCKS = 1024;
__global__ void __launch_bounds__(NT) k_dot_partial(int N, int nrhs, const double* a, const double* b,
                                                    double* partial) {
    __shared__ double red[NT];
    int nrp = 1;
    while (nrp < nrhs) nrp <<= 1;
    const int groups = NT / nrp;
    const int tid = threadIdx.x, r = tid % nrp, g = tid / nrp;
    double s = 0.0;
    if (r < nrhs) {
        for (size_t i = (size_t)blockIdx.x * groups + g; i < (size_t)N; i += (size_t)gridDim.x * groups)
            s += a[i * nrhs + r] * b[i * nrhs + r];
    }
    red[tid] = s;
    __syncthreads();
    for (int off = groups / 2; off > 0; off >>= 1) {
        if (g < off) red[tid] += red[tid + off * nrp];
        __syncthreads();
    }
    if (g == 0 && r < nrhs) partial[(size_t)blockIdx.x * nrhs + r] = red[tid];
}
__global__ void __launch_bounds__(NT) k_dot_final(int nblocks, int nrhs, const double* partial, double* out) {
    __shared__ double red[NT];
    for (int r = 0; r < nrhs; r++) {
        double s = 0.0;
        for (int b = threadIdx.x; b < nblocks; b += NT) s += partial[(size_t)b * nrhs + r];
        red[threadIdx.x] = s;
        __syncthreads();
        for (int off = NT / 2; off > 0; off >>= 1) {
            if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
            __syncthreads();
        }
        if (threadIdx.x == 0) out[r] = red[0];
        __syncthreads();
    }
}

__global__ void __launch_bounds__(NT) k_axpby(int N, int nrhs, const double* x, const double* ax, double sgn,
                                              double* y, const double* by) {
    size_t n = (size_t)N * nrhs;
    for (size_t idx = (size_t)blockIdx.x * NT + threadIdx.x; idx < n; idx += (size_t)gridDim.x * NT) {
        int r = (int)(idx % nrhs);
        double a = sgn * (ax ? ax[r] : 1.0);
        double b = by ? by[r] : 1.0;
        y[idx] = a * x[idx] + b * y[idx];
    }
}

// GMRES kernels. V holds Householder vectors as interleaved N x nrhs blocks (block j at
// V + j * N * nrhs). out = base + [ye; 0] - sum_{j<k} V_j z_j, per column (base may be
// nullptr = 0; ye holds ny rows, or nullptr).
__global__ void __launch_bounds__(NT) k_gm_comb(int N, int nrhs, const double* base, const double* ye, int ny,
                                               const double* V, int k, const double* z, double* out) {
    const size_t n = (size_t)N * nrhs, blk = (size_t)N * nrhs;
    for (size_t idx = (size_t)blockIdx.x * NT + threadIdx.x; idx < n; idx += (size_t)gridDim.x * NT) {
        const int i = (int)(idx / nrhs), r = (int)(idx % nrhs);
        double acc = base ? base[idx] : 0.0;
        if (ye && i < ny) acc += ye[idx];
        for (int j = 0; j < k; j++) acc -= V[(size_t)j * blk + idx] * z[(size_t)j * nrhs + r];
        out[idx] = acc;
    }
}
// partial[(b * k + j) * nrhs + r] = sum over block b of V_j[i, r] * v[i, r]; grid (blocks, k)
__global__ void __launch_bounds__(NT) k_gm_multidot_partial(int N, int nrhs, const double* V, const double* v,
                                                            double* partial) {
    __shared__ double red[NT];
    int nrp = 1;
    while (nrp < nrhs) nrp <<= 1;
    const int groups = NT / nrp;
    const int tid = threadIdx.x, r = tid % nrp, g = tid / nrp, j = blockIdx.y;
    const double* Vj = V + (size_t)j * N * nrhs;
    double s = 0.0;
    if (r < nrhs)
        for (size_t i = (size_t)blockIdx.x * groups + g; i < (size_t)N; i += (size_t)gridDim.x * groups)
            s += Vj[i * nrhs + r] * v[i * nrhs + r];
    red[tid] = s;
    __syncthreads();
    for (int off = groups / 2; off > 0; off >>= 1) {
        if (g < off) red[tid] += red[tid + off * nrp];
        __syncthreads();
    }
    if (g == 0 && r < nrhs) partial[((size_t)blockIdx.x * gridDim.y + j) * nrhs + r] = red[tid];
}
// out[j * nrhs + r] = sum over blocks; one workgroup per (j, r)
__global__ void __launch_bounds__(NT) k_gm_multidot_final(int nblocks, int k, int nrhs, const double* partial,
                                                          double* out) {
    __shared__ double red[NT];
    const int jr = blockIdx.x;  // j * nrhs + r
    double s = 0.0;
    for (int b = threadIdx.x; b < nblocks; b += NT) s += partial[(size_t)b * k * nrhs + jr];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int off = NT / 2; off > 0; off >>= 1) {
        if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[jr] = red[0];
}
// Householder vector of step k from v: u[i] = 0 (i < k), 1 (i = k), v[i] / d[r] (i > k);
// d[r] = 0 means a zero essential part (tau = 0).
__global__ void __launch_bounds__(NT) k_gm_householder(int N, int nrhs, int k, const double* v, const double* d,
                                                       double* u) {
    const size_t n = (size_t)N * nrhs;
    for (size_t idx = (size_t)blockIdx.x * NT + threadIdx.x; idx < n; idx += (size_t)gridDim.x * NT) {
        const int i = (int)(idx / nrhs), r = (int)(idx % nrhs);
        u[idx] = i < k ? 0.0 : (i == k ? 1.0 : (d[r] != 0.0 ? v[idx] / d[r] : 0.0));
    }
}

__global__ void k_ratio(int nrhs, const double* num, const double* den, const int* active, double* out) {
    int r = threadIdx.x;
    if (r < nrhs) out[r] = (active == nullptr || active[r]) ? num[r] / den[r] : 0.0;
}

__global__ void __launch_bounds__(NT) k_copy_f64(double* dst, const double* src, size_t n) {
    for (size_t i = (size_t)blockIdx.x * NT + threadIdx.x; i < n; i += (size_t)gridDim.x * NT) dst[i] = src[i];
}

// dst[k] = src[idx[k]]: values of a fixed pattern moved from the caller's order to a stored one
template <typename I>
__global__ void __launch_bounds__(NT) k_gather_f64(const I* idx, const double* src, long long n, double* dst) {
    for (long long k = (long long)blockIdx.x * NT + threadIdx.x; k < n; k += (long long)gridDim.x * NT)
        dst[k] = src[idx[k]];
}

// ---------------------------------------------------------------------------------------
template <typename T>
hipError_t launch_perm_in(const double* b, size_t sx, size_t sr, int nrhs, const int* perm, int N, double* ws,
                          hipStream_t st) {
    k_perm_in<T><<<grid_for((size_t)N * nrhs), NT, 0, st>>>(b, sx, sr, nrhs, perm, N, ws);
    return hipGetLastError();
}
template <typename T>
hipError_t launch_perm_out(const double* ws, const int* perm, int N, int nrhs, double* x, size_t sx, size_t sr,
                           hipStream_t st) {
    k_perm_out<T><<<grid_for((size_t)N * nrhs), NT, 0, st>>>(ws, perm, N, nrhs, x, sx, sr);
    return hipGetLastError();
}
hipError_t launch_cm2il(const double* src, int ld, int N, int nrhs, double* dst, hipStream_t st) {
    k_cm2il<<<grid_for((size_t)N * nrhs), NT, 0, st>>>(src, ld, N, nrhs, dst);
    return hipGetLastError();
}
hipError_t launch_il2cm(const double* src, int N, int nrhs, double* dst, int ld, hipStream_t st) {
    k_il2cm<<<grid_for((size_t)N * nrhs), NT, 0, st>>>(src, N, nrhs, dst, ld);
    return hipGetLastError();
}
// Right-hand sides per pass of a phase: 4, 16 or 32 (more run as several passes).
template <typename F>
static hipError_t mv_width(int nrhs, F&& f) {
    if (nrhs <= 4) return f(std::integral_constant<int, 0>());
    if (nrhs <= 16) return f(std::integral_constant<int, 1>());
    return f(std::integral_constant<int, 2>());
}
template <typename T>
hipError_t launch_mv(const MvDevPhase& ph, double* ws, int nrhs, hipStream_t st) {
    if (ph.nchunks == 0) return hipSuccess;
    return mv_width(nrhs, [&](auto ct) {
        constexpr int CT = decltype(ct)::value, NACC = CT == 0 ? 1 : 4 * CT, W = CT == 0 ? 4 : 16 * CT;
        const int waves = std::max(4, ph.nw), groups = waves / ph.nw;
        const int nb = (ph.nchunks + groups - 1) / groups;
        const dim3 grid((nb + XCDS - 1) / XCDS * XCDS, (nrhs + W - 1) / W);
        const size_t lds = (size_t)groups * (ph.nw - 1) * WAVE * NACC * sizeof(double);
        k_mv<T, CT><<<grid, waves * WAVE, lds, st>>>(ph, ws, nrhs);
        return hipGetLastError();
    });
}
template <typename T>
hipError_t launch_mv_tail(const MvTail& tail, double* ws, int nrhs, hipStream_t st) {
    if (tail.n == 0) return hipSuccess;
    return mv_width(nrhs, [&](auto ct) {
        constexpr int CT = decltype(ct)::value, NACC = CT == 0 ? 1 : 4 * CT;
        size_t lds = 0;
        for (int p = 0; p < tail.n; p++)
            lds = std::max(lds, (size_t)(MV_NW_MAX - MV_NW_MAX / tail.ph[p].nw) * WAVE * NACC * sizeof(double));
        k_mv_tail<T, CT><<<1, MV_NW_MAX * WAVE, lds, st>>>(tail, ws, nrhs);
        return hipGetLastError();
    });
}
template <typename T>
hipError_t launch_wy(const WyTask* d_tasks, int ntasks, const int4* d_tiles, int ntiles, hipStream_t st) {
    if (ntasks == 0) return hipSuccess;
    k_wy_explicit<T><<<dim3(ntasks, 16), NT, 0, st>>>(d_tasks);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || ntiles == 0) return e;
    k_wy_gram<<<ntiles, NT, 0, st>>>(d_tasks, d_tiles);
    return hipGetLastError();
}
template <typename T>
hipError_t launch_merge(const MergeTask* d_tasks, int ntasks, const int2* d_children, double* ws, int nrhs, int fwd,
                        hipStream_t st) {
    if (ntasks == 0) return hipSuccess;
    k_merge<T><<<ntasks, NT, 0, st>>>(d_tasks, d_children, ws, nrhs, fwd);
    return hipGetLastError();
}

hipError_t launch_spmv(int N, const int* rowptr, const int* colidx, const double* val, const double* x, double* y,
                       int nrhs, hipStream_t st) {
    k_spmv<<<grid_for((size_t)N * nrhs), NT, 0, st>>>(N, rowptr, colidx, val, x, y, nrhs);
    return hipGetLastError();
}
hipError_t launch_sampled_outer(int N, const int* rowptr, const int* colidx, const int* csc_of, const double* u,
                                const double* v, int nrhs, int ld, double alpha, double* out, hipStream_t st) {
    if (N == 0) return hipSuccess;
    k_sampled_outer<<<grid_for((size_t)N * OUTER_LANES), NT, 0, st>>>(N, rowptr, colidx, csc_of, u, v, nrhs, ld, alpha, out);
    return hipGetLastError();
}
hipError_t launch_dot(int N, int nrhs, const double* a, const double* b, double* partial, double* out,
                      hipStream_t st) {
    k_dot_partial<<<DOT_BLOCKS, NT, 0, st>>>(N, nrhs, a, b, partial);
    k_dot_final<<<1, NT, 0, st>>>(DOT_BLOCKS, nrhs, partial, out);
    return hipGetLastError();
}
hipError_t launch_axpby(int N, int nrhs, const double* x, const double* ax, double sgn_ax, double* y,
                        const double* by, hipStream_t st) {
    k_axpby<<<grid_for((size_t)N * nrhs), NT, 0, st>>>(N, nrhs, x, ax, sgn_ax, y, by);
    return hipGetLastError();
}
hipError_t launch_gm_comb(int N, int nrhs, const double* base, const double* ye, int ny, const double* V, int k,
                          const double* z, double* out, hipStream_t st) {
    k_gm_comb<<<grid_for((size_t)N * nrhs), NT, 0, st>>>(N, nrhs, base, ye, ny, V, k, z, out);
    return hipGetLastError();
}
hipError_t launch_gm_multidot(int N, int nrhs, int k, const double* V, const double* v, double* partial, double* out,
                              hipStream_t st) {
    if (k == 0) return hipSuccess;
    constexpr int MB = 256;
    k_gm_multidot_partial<<<dim3(MB, k), NT, 0, st>>>(N, nrhs, V, v, partial);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    k_gm_multidot_final<<<k * nrhs, NT, 0, st>>>(MB, k, nrhs, partial, out);
    return hipGetLastError();
}
hipError_t launch_gm_householder(int N, int nrhs, int k, const double* v, const double* d, double* u, hipStream_t st) {
    k_gm_householder<<<grid_for((size_t)N * nrhs), NT, 0, st>>>(N, nrhs, k, v, d, u);
    return hipGetLastError();
}
hipError_t launch_ratio(int nrhs, const double* num, const double* den, const int* active, double* out,
                        hipStream_t st) {
    k_ratio<<<1, 64, 0, st>>>(nrhs, num, den, active, out);
    return hipGetLastError();
}
hipError_t launch_copy_f64(double* dst, const double* src, size_t n, hipStream_t st) {
    k_copy_f64<<<grid_for(n), NT, 0, st>>>(dst, src, n);
    return hipGetLastError();
}
hipError_t launch_gather_f64(const long long* idx, const double* src, long long n, double* dst, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    k_gather_f64<long long><<<grid_for((size_t)n), NT, 0, st>>>(idx, src, n, dst);
    return hipGetLastError();
}
hipError_t launch_gather_f64(const int* idx, const double* src, long long n, double* dst, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    k_gather_f64<int><<<grid_for((size_t)n), NT, 0, st>>>(idx, src, n, dst);
    return hipGetLastError();
}

#define SPAND_SOLVE_INST(T)                                                                                  \
    template hipError_t launch_perm_in<T>(const double*, size_t, size_t, int, const int*, int, double*, hipStream_t); \
    template hipError_t launch_perm_out<T>(const double*, const int*, int, int, double*, size_t, size_t, hipStream_t); \
    template hipError_t launch_mv<T>(const MvDevPhase&, double*, int, hipStream_t);                          \
    template hipError_t launch_mv_tail<T>(const MvTail&, double*, int, hipStream_t);                         \
    template hipError_t launch_wy<T>(const WyTask*, int, const int4*, int, hipStream_t);                    \
    template hipError_t launch_merge<T>(const MergeTask*, int, const int2*, double*, int, int, hipStream_t);
SPAND_SOLVE_INST(float)
SPAND_SOLVE_INST(double)

}  // namespace spand
