// Task descriptors shared by the host level planner (tree.cpp) and the level-batched HIP
// kernels (kernels.hip). Every kernel launch processes an array of these, one workgroup per
// task (or per task tile), so one launch covers every cluster / edge of one ND level, of
// uneven sizes. Blocks are column-major with ld = rows, in the element type of the
// factorization (float or double); pointers are device addresses in the block arena.
#pragma once
#include <cstdint>

namespace spand {

// In-place lower Cholesky of an n x n pivot block (reference: potf, src/util.cpp:158-165).
struct PotrfTask {
    void* A;
    int n;
    int cluster;  // reported through the info array on a non-SPD pivot
    void* dbuf;   // pivots above POTRF_SMALL_MAX: the factored 32 x 32 diagonal block of the
                  // current panel, handed from k_potrf_panel to k_potrf_trail
};

// Triangular solve of (a 64-wide chunk of) an edge block against a pivot factor L
// (n x n, lower, ld n):
//   side 0: B (n x m, ld ldb) := L^{-1} B      (trsm_left,  src/util.cpp:266-274)
//   side 1: B (m x n, ld ldb) := B L^{-T}      (trsm_right, src/util.cpp:256-264)
// m <= 64: the host splits wide blocks into independent column (left) / row (right) chunks.
// A left solve may read its right-hand side from another block: B := L^{-1} P^T src, row i
// of P^T src being row perm[i] of src (perm nullptr: the identity), the row interchanges of
// an LU pivot applied to an in-edge (trsm_getf_edgeIn, src/tree.cpp:668-677).
struct TrsmTask {
    const void* L;
    void* B;
    int n;
    int m;
    int side;
    int ldb;
    const void* src;  // nullptr: in place
    const int* perm;
};

// LU with partial pivoting of an n x n pivot block (getf, src/util.cpp:184-199, in dgetf2
// order) followed by split_LU (src/util.cpp:213-227). On return A holds L (lower, diagonal
// sqrt|d_j|, zero above), Ut holds U^T (lower, zero above) and perm the row permutation p
// with P^T A = L U (row i of P^T A is row p[i] of A).
struct GetrfTask {
    void* A;
    void* Ut;
    int* perm;
    int n;
    int cluster;  // reported through the info array on a zero pivot
    void* diag;   // panel launches: the n pivots, for split_LU
    int* moves;   // and the current panel's row interchanges (GETRF_MOVES)
};
// moves: the row that each of the panel's GETRF_NB top positions takes, the number of the
// other rows that moved, and (to, from) of each, all counted from the panel's first row.
constexpr int GETRF_NB = 32;
constexpr int GETRF_MOVES = 3 * GETRF_NB + 1;

// One Schur-complement target tile: C[r0:r0+tm, c0:c0+tn] of a block C (ldc rows) receives
// contributions [k0, k1) in order, each C -= opA(A) opB(B) (gemm / syrk, src/util.cpp:122-156).
// SCHUR_LOWER restricts the update to the lower triangle (syrk on a diagonal block);
// SCHUR_CLEAR takes C as zero before the first contribution, whatever it holds.
enum SchurFlags { SCHUR_LOWER = 1, SCHUR_CLEAR = 2 };
struct SchurTile {
    void* C;
    int ldc;
    int r0, c0, tm, tn;
    int lower;   // SCHUR_LOWER, SCHUR_CLEAR
    int k0, k1;
};
struct SchurContrib {
    const void* A;  // opA(A) is m x k: ta ? A^T (A is k x m, ld lda) : A (m x k, ld lda)
    const void* B;  // opB(B) is k x n: tb ? B^T (B is n x k, ld ldb) : B (k x n, ld ldb)
    int k;
    int lda, ldb;
    int ta, tb;
    int pad;
};

// Column-pivoted QR sparsification of one cluster (sparsify_adaptive_only,
// src/tree.cpp:1292-1347). Its Asn = [A_sn(in edges) | A_ns^T(out edges)] is gathered
// from segs[seg0:seg0+nseg] using the live sizes in dsize[], factored (dgeqp3 order),
// truncated by choose_rank and scattered back into the edge blocks.
struct RrqrTask {
    int cluster;
    int seg0, nseg;
    int max_rows, max_cols;  // capacity of the scratch (rows x cols) and Q (rows x rows)
    int pad;
    void* scratch;     // T[max_rows * max_cols]
    double* norms;     // double[2 * max_cols]
    int* jpvt;         // int[max_cols]
    void* Q;           // T[max_rows * min(max_rows, max_cols)] (Householder vectors)
    void* tau;         // T[min(max_rows, max_cols)]
};
struct RrqrSeg {
    void* E;   // edge block
    int nbr;   // neighbour cluster (its live size gives the segment width)
    int out;   // 0: in-edge, block is s x n; 1: out-edge, block is n x s (transposed)
};

// Large clusters use the stepped RRQR (one launch per pivot step, columns split into
// 64-wide slabs, one wavefront each). Columns never move: a double-buffered
// position <-> column map reproduces LAPACK's column swaps and its first-max tie-break.
struct RrqrBig {
    RrqrTask t;      // scratch holds A (rows x cols, ld rows); norms holds vn1 | vn2 by column
    int* map;        // p2c[2][max_cols] then c2p[2][max_cols]
    double* cand_v;  // [2][nslab] per-slab best partial norm for the next step, then |R_00|
    int* cand_p;     // [2][nslab] its position
    int* dims;       // rows, cols, min(rows, cols), steps to run (the rank once it is known),
                     // 1 once every kept reflector is stored
    void* vbuf;      // nullptr, or [nslab][2][max_rows] pivot column / reflector buffers
                     // (per-step launches), or the relay words of the persistent launch
                     // (relay = 1): candidates [2][nsub][4], then candidate columns
                     // [2][nsub][max_rows * sizeof(T) / 4], 64 bits each
    long long* done; // host-visible flag, or nullptr: set to 1 by the last step that does
                     // work (rank reached or all min(rows, cols) steps taken)
    int nslab;
    int relay;       // 1: vbuf holds relay words (k_rrqr_init clears them)
    int nsub;        // slabs of the persistent launch (narrower than 64 columns for long ones)
};
struct RrqrSlab {
    int big;   // index into the RrqrBig array
    int slab;  // columns [64 * slab, 64 * slab + 64)
};

// Merge copy of one child block into a parent block (update_edges, src/tree.cpp:1133-1184), or
// an identity block.
struct CopyTask {
    const void* src;  // nullptr => identity block
    void* dst;
    int rows, cols;
    int ldd;
    int c0;           // identity block: the row of its first column's one
};

// ---------------------------------------------------------------------------------------
// Preconditioner apply (Tree::solve, src/tree.cpp:1610-1635). Vectors are stored
// interleaved: element i of right-hand side r lives at x[(xoff + i) * nrhs + r].
//
// The recorded ops of a level run as three mv phases per direction, each a set of groups
// x[dst] (op)= sum_k op(A_k) x[src_k] whose destinations are never sources of the same
// phase, so one launch covers a phase whatever the order of its workgroups:
//   E   ScalingLLT / ScalingPLUQ of the eliminated clusters (src/operations.cpp:95-121):
//       xe := Linv x[perm] into a segment of its own, back x := Linv^T xe or (U^{-T})^T xe
//   G   Gemm* (src/operations.cpp:31-93): x_n -= A xe, back xe -= A^T x_n
//   W   the scaling and the Orthogonal op of a remaining cluster in one matrix
//       (src/operations.cpp:95-121,149-158), W = Q^T Linv: its first r outputs (the kept
//       rank) go to the cluster's place in its parent's segment (Merge,
//       src/operations.cpp:166-192), the rest to the sibling's segment; back x := W^T y
struct MvTerm {
    const void* A;     // op(A)'s element (output o, inner j): A[o + j ld], transposed A[j + o ld]
    const int* perm;   // not transposed: inner index j reads source element perm[j]
    int ld, len;       // column stride of A, inner positions
    int xsrc;          // source segment
    int flags;         // MV_TRANS, and the inner-range clip of a triangular A for the outputs
                       // [o0, o0 + 16): MV_TRI_LO inner < o0 + 16, MV_TRI_UP inner >= o0
};
enum MvFlags { MV_TRANS = 1, MV_TRI_LO = 2, MV_TRI_UP = 4 };
enum MvMode { MV_SUB = 0, MV_SET = 1 };  // x -= s, x = s
struct MvChunk {       // up to MV_ROWS outputs of one group
    int k0, k1;        // terms of the group
    int o0, no;        // outputs [o0, o0 + no)
    int xdst, mode;
    const int* dperm;  // nullptr, or output o goes to xdst + dperm[o]
};
// One mv phase: its chunks, and the wavefronts that share a chunk's inner positions.
struct MvDevPhase {
    const MvChunk* chunks;
    const MvTerm* terms;
    int nchunks, nw;
};
// Explicit Householder vectors V (unit diagonal, zeros above) and the compact-WY factor of
// one Orthogonal op, built at factorization. Q = H_0 H_1 ... H_{k-1} = I - V T V^T with T
// upper triangular and T^{-1} = diag(1 / tau) + striu(V^T V) (the UT transform), so
// W = Q^T Linv = Linv - V Z with Z = S^{-1} V^T Linv, S = diag(1 / tau) + stril(V^T V).
// Stored is -S: Y = -V^T Linv is what the Schur kernel leaves in a cleared block, and the
// triangular solve (-S) Z = Y gives Z.
struct WyTask {
    const void* V;    // m x k reflectors as stored by the QR (R on and above the diagonal)
    const void* tau;
    double* Ve;       // m x k explicit V
    double* S;        // k x k lower: -diag(1 / tau) - stril(V^T V)
    int m, k;
};
struct MergeTask {  // Merge (src/operations.cpp:166-192) of children without a W phase
    int pxoff;
    int c0, c1;  // range into (child xoff, child size) pairs
    int pad;
};

}  // namespace spand
