// Host-side symbolic analysis for the MI355X sweep solver: PSP's panel
// split, analytic nested dissection, elimination tree and front structures,
// plus the static device work lists (front assembly, blocked LDL^T steps,
// Schur GEMMs, diagonal-block inversion, per-level solve phases).
//
// Everything here is integer work done once per DistHelmholtz object
// (PSP's constructor, dist_helmholtz/main.hpp:12-436).
#pragma once

#include <cstdint>
#include <string>
#include <array>
#include <vector>

#include "psp_hip.h"

namespace psp_amd {

// ---------------------------------------------------------------------------
// Panel geometry (dist_helmholtz/main.hpp:35-57, 728-821).
// ---------------------------------------------------------------------------
struct Geometry {
    int nx = 0, ny = 0, nz = 0, bz = 0, P = 0, cutoff = 0;
    bool topPML = true;
    int bottomDepth = 0, topOrigDepth = 0, innerDepth = 0, leftoverDepth = 0;
    int numFullInner = 0, numPanels = 0;
    bool haveLeftover = false;

    // Returns PSP_HIP_OK or PSP_HIP_ERR_SHALLOW.
    int init(const psp_hip_desc& d);
    int padding(int p) const { return p == 0 ? 0 : bz; }
    int depth(int p) const;
    int panelV(int p) const;
    int cls(int p) const;  // 0 bottom/full inner, 1 leftover, 2 top
    int vOffset(int p) const { return panelV(p) - padding(p); }
    int classVSize(int c) const;
};

// In-panel nested-dissection index (ReorderedIndexRecursion,
// dist_helmholtz/main.hpp:1425-1477, one process).
int NestedIndex(int x, int y, int vLocal, int xSize, int ySize, int vSize,
                int cutoff);

// ---------------------------------------------------------------------------
// Device work-list records.  All offsets are element offsets inside one
// panel's slice of the named buffer; the kernels add batch * stride.
// ---------------------------------------------------------------------------
enum BufId : int16_t { BUF_L = 0, BUF_U = 1, BUF_T = 2, BUF_LT = 3 };

enum GemmFlags : int32_t {
    G_BTRANS = 1,   // B(k,n) = Bp[n + k*ldb]
    G_AUNIT = 2,    // A is unit lower triangular (square)
    G_BUNIT = 4,    // B is unit lower triangular (square)
    G_CLOWER = 8,   // only C(i,j) with i >= j is touched
    G_HASD = 16,    // multiply by diag(D) between A and B
    G_NEG = 32,     // C -= ...
    G_BETA0 = 64,   // C is overwritten instead of accumulated
    G_CTRANS = 128, // C(i,j) is stored at Cp[j + i*ldc]
};

struct GemmDesc {
    int64_t a, b, c, d;
    int32_t lda, ldb, ldc, dinc;
    int32_t M, N, K;
    int16_t abuf, bbuf, cbuf, dbuf;
    int32_t flags;
    int32_t pad_;
};

struct GemmTile {
    int32_t desc;
    int32_t tm, tn;
    int32_t pad_;
};

// Extend-add of one child's Schur complement column range into its parent.
struct ExtAddItem {
    int64_t uChild;     // child's U offset (BUF_U)
    int64_t lParent;    // parent's L offset (BUF_L)
    int64_t uParent;    // parent's U offset (BUF_U)
    int32_t relStart;   // into relinds
    int32_t uc;         // child's update size
    int32_t sp, up;     // parent's pivot and update sizes
    int32_t col0, col1; // child's U column range handled by this item
};

// One block column step of the blocked LDL^T on one front: either the
// factorization of the diagonal block [j0,j1)^2 (r0 == r1 == -1) or the
// triangular solve of rows [r0, r1) against the factored diagonal block.
struct LdlItem {
    int64_t l;          // front's L offset
    int32_t ld;         // s + u
    int32_t j0, j1;     // block columns [j0, j1)
    int32_t r0, r1;     // rows [r0, r1) below the diagonal block
};

// Inversion of one diagonal block of a unit lower triangular L_TL.
struct InvItem {
    int64_t l;
    int32_t ld;
    int32_t j0, j1;
    int32_t pad_;
};

// One row block of a matrix-vector product of one node in a front solve:
// output rows [row0, row0 + nrows) (nrows <= 64), inner indices [col0, col1).
// slot >= 0: the tile is one inner slice of its row block and writes its
// partial sums to that slot of the partial buffer.  As a reduce item (same
// struct): col0 = first slot, col1 = number of slots.
struct MvTile {
    int32_t node;
    int32_t row0, nrows;  // nrows 0: a hole of the XCD placement (no work)
    int32_t col0, col1;
    int32_t slot;
    int32_t red = -1;     // reduce item of a slice's row block (into mvred), -1 if none
};

// Fused subtree solves: one persistent launch per phase runs every level of
// a panel's tree from the cut depth down, the subtrees under the cut split
// over kQueues queues (one per XCD of the device, each queue's tiles in
// dependency order).  A queue tile names its node (the node's fields come
// from the per-node records); red >= 0: the tile is one inner slice
// (partial sums in slot `slot`) of the split row block QRed[red].
constexpr int kQueues = 8;
struct QTile {
    int32_t node, row0, nrows, col0, col1, slot, red, pad_;
};
struct QRed {
    int32_t node, row0, nrows, slot0, nslots, pad_[3];
};
static_assert(sizeof(QTile) == 32 && sizeof(QRed) == 32, "queue records");

// Shape of the tiles of one (level, phase) of the front solves.
struct SolveShape {
    int rows = 64;  // output rows per tile: 64, 32 or 16
    int split = 1;  // inner slices per row block (partial sums + reduce)
};

// 32x32 block (rows i0.., columns j0..) of a per-front copy between L and
// LT (see the solve layout in ClassPlan).
struct TransItem {
    int32_t node, i0, j0, pad_;
};

struct Node {
    int off = 0, size = 0, usize = 0, parent = -1;
    int child[2] = {-1, -1};
    int nchild = 0;
    int depth = 0;
    int64_t ustart = 0;   // into structs / relinds
    int64_t loff = 0;     // factor storage (BUF_L), (s+u) x s column-major
    int64_t uoff = 0;     // Schur complement workspace (BUF_U), u x u
    int64_t toff = 0;     // inversion temporary (BUF_T)
    int64_t woff = 0;     // solve work vector rows (s+u)
};

struct GemmLaunch {
    int32_t tileStart = 0, tileCount = 0;
};

// ---------------------------------------------------------------------------
// Merged solves.  The tree levels are cut into groups of consecutive depths;
// the nodes of one group under a common ancestor (the group's top node) form
// one merged front, solved with the explicit inverse of its whole pivot
// block, so a panel solve takes one launch per group and direction instead
// of one per level.  A merged front's factor F has the group's pivots as
// columns and, as rows, the same pivots (D^-1/2 Linv, lower triangular) followed
// by the top node's update rows (-L_BL Linv), in blocks of 16 x 16.  Blocks are
// stored once, row of blocks by row of blocks, and serve both directions:
//   forward   [y; w] = F g
//   backward  x = F^T [y; x_struct].
// Pivots keep their post-order, so the pivots under a node are contiguous
// and row i of F has its entries in one column range: from the first pivot
// below i's node to i.  Blocks of siblings that do not meet are not stored.
// ---------------------------------------------------------------------------
constexpr int kBlk = 16;

struct BlockNode {
    int top = -1;            // the group's top node (fine tree)
    int group = 0;
    int s = 0, u = 0;        // pivots, update rows
    int sb = 0, ub = 0;      // the same in blocks
    int x0 = 0;              // first panel-vector row (solve order, multiple of 16)
    int w0 = 0;              // first work row; rows [0, 16 sb) pivots, then the update rows
    int u0 = 0;              // first entry of udst / usrc (16 ub entries)
    int br0 = 0;             // first block row (browBase, browLo); sb + ub of them
    int parent = -1;         // merged parent
    bool leaf = true;        // no merged children
};

// One workgroup of a merged solve: up to 4 output blocks (one per wave) and
// a range of inner blocks.  128 bytes, read once.
struct BlockTile {
    int32_t x0, w0, u0, s;      // of the node
    int32_t u, sb, leaf, ob0;   // first output block (row of blocks forward, column backward)
    int32_t nob, ib0, nib, lst; // inner blocks [ib0, ib0 + nib); lst: first entry of blist / bsrc (backward)
    int32_t slot, red;          // partial-sum slot and reduce item of an inner slice, -1 if none
    int32_t pad_[2];
    int32_t base[4];            // forward: block (row ob0 + q, column j) is base[q] + j
    int32_t lo[4], hi[4];       // forward: its columns [lo, hi)
    int32_t pad2_[4];
};
static_assert(sizeof(BlockTile) == 128, "BlockTile is one 128-byte record");

// A split set of output blocks: the tile's fields with its slots.
struct BlockRed {
    int32_t x0, w0, u0, s;
    int32_t u, sb, leaf, ob0;
    int32_t nob, slot0, nslots, pad_[5];
};
static_assert(sizeof(BlockRed) == 64, "BlockRed is one 64-byte record");

// Fold of one fine node into its merged front.
struct FoldNode {
    int64_t l;           // factor offset (BUF_L), (s + u) x s
    int64_t e;           // E = -L_BL Linv, u x s (in the update scratch, of its depth group)
    int32_t s, u;
    int32_t mcol;        // first pivot within the merged front
    int32_t br0;         // the merged front's first block row
    int32_t x0;          // panel-vector row of the node's first pivot
    int32_t urow;        // merged row of the first update row (group tops), -1 otherwise
};

// Columns of a node below its group's top: F_c = F_A P + ext(E_c), with A the
// node's ancestors in the group (their columns already folded), P the rows of
// E_c at their pivots and ext its rows at the top node's update rows.
// flist[list ..] are the merged rows involved: the pivots of A, nearest
// ancestor first, then the update rows; F_A is lower triangular in this order.
// Only the k pivots that E_c has a row for (the node's ring) enter the product.
struct ComposeDesc {
    int64_t e;
    int32_t lde, list, rows, br0;
    int32_t k, ccol, n;
    int32_t src;         // fsrc[src ..]: E_c's row at each entry of flist, -1 if none
    int32_t kl, piv;     // fkeys[kl ..]: the k pivots; entries of flist that are pivots
};
struct ComposeKey {      // a pivot of F_A: column of F, entry of flist, E_c's row
    int32_t col, pos, row, pad_;
};
static_assert(sizeof(FoldNode) == 40 && sizeof(ComposeDesc) == 48, "fold records");

struct ClassPlan {
    int cls = 0;
    int vsize = 0;
    int n = 0;          // padded unknowns nx*ny*vsize
    int maxDepth = 0;
    std::vector<Node> nodes;            // post-order, root last
    std::vector<int> structs;           // sorted lower structures
    std::vector<int> relinds;           // row of each struct entry in parent
    std::vector<std::vector<int>> levels;  // node ids per depth
    int64_t fstore = 0, ustore = 0, tstore = 0, wstore = 0;

    // Front assembly: per padded unknown q: packed x | y<<16, vLocal,
    // node, column within node, and six front rows (x-1,x+1,y-1,y+1,v-1,v+1)
    // or -1 when the coupling is absent or above the diagonal.
    std::vector<int32_t> qxy, qv, qnode, qcol;
    std::vector<int32_t> qrows;  // 6 per q

    // Factorization schedule.
    struct LevelSteps {
        int64_t uoff = 0, ucount = 0;                // the level's updates in BUF_U
        std::vector<std::pair<int, int>> extadd[2];  // item range per child slot
        std::vector<std::pair<int, int>> ldlDiag;    // per block step: item range
        std::vector<std::pair<int, int>> ldlTrsm;    // per block step: item range
        std::vector<GemmLaunch> trail;               // per block step
        GemmLaunch schur;
    };
    std::vector<ExtAddItem> extadd;
    std::vector<LdlItem> ldl;
    std::vector<GemmDesc> gemms;
    std::vector<GemmTile> tiles;
    std::vector<LevelSteps> steps;        // per depth (deepest first order)
    std::vector<InvItem> inv;
    std::vector<GemmLaunch> invGemm;      // alternating T = C*Ainv, X = -Binv*T

    // Layout of the fused launches, made after the selective inversion when they
    // are on:
    //   L  ((s+u) x s, ld s+u): rows < s hold Linv (unit lower, ones stored
    //      on the diagonal), rows >= s hold -L_BL Linv;
    //   LT (s x (s+u), ld s):   columns < s hold Linv^T D^-1 (upper),
    //      columns >= s hold (-L_BL Linv)^T.
    // The forward solve of a node is then one product [y; W_bot] =
    // L g_top + [0; g_bot] and the backward solve one product
    // x = LT [y; x_struct]: one launch per level and direction.
    GemmLaunch fold;                 // LT[:, s:] = (-L_BL Linv)^T
    std::vector<TransItem> foldBack; // L_BL <- LT[:, s:]^T, diag(L) <- 1

    // Solve schedule.  Per depth: forward product (F) and backward product
    // (B).
    std::vector<MvTile> mv;
    std::vector<MvTile> mvred;  // reduce items of split row blocks
    int maxSlots = 0;           // partial slots of the largest (level, phase)
    std::vector<std::array<SolveShape, 2>> shapes;  // per depth, per phase (F, B)
    struct Range {
        int start = 0, count = 0;    // tiles
        int rows = 64;               // output rows per tile (64, 32 or 16)
        int persist = 0;             // always 0: a workgroup has one tile
        int rstart = 0, rcount = 0;  // reduce items
        int xcd = 0;                 // tiles placed so each row block's slices share an XCD
    };
    struct SolveLevel {
        Range f, b;
        // per phase (F, B): factor entries read and vector rows (inner
        // inputs + outputs) moved, for algorithmic bytes and flops
        double entries[2] = {0, 0};
        double vecRows[2] = {0, 0};
    };
    std::vector<SolveLevel> solveLevels;  // index = depth
    std::vector<TransItem> trans;

    // Fused subtree solves (qcut < 0: none; every level is its own launch).
    // Per phase: the tiles of queue q are tiles[qstart[q] .. qstart[q+1]),
    // forward deepest level first, backward the cut level first; dep[t] =
    // {dep0, dep1, row blocks of dep0, of dep1} names the nodes whose row
    // blocks must be done before node t's tiles read their inputs (forward:
    // its children; backward: its nearest ancestor with pivots, when that
    // is inside the fused levels), -1 for none.
    int qcut = -1;
    int queueRows = 32;  // output rows per queue tile (64, 32 or 16)
    int nqueues = 0;
    struct QueuePhase {
        std::vector<QTile> tiles;
        std::vector<int32_t> qstart;
        std::vector<QRed> reds;
        std::vector<std::array<int32_t, 4>> dep;
        double entries = 0, vecRows = 0;  // algorithmic work of the launch
    };
    QueuePhase queue[2];

    // Merged solves (BuildMerged, BuildBlockTiles).
    std::vector<std::array<int, 2>> groups;  // first and last depth of each group, top group first
    std::vector<BlockNode> bnodes;
    std::vector<int> bnodeOf;        // merged front of each fine node (-1: no pivots in it)
    int xrows = 0;                   // panel-vector rows in solve order, padding included
    int wrows = 0;                   // work rows
    int nblocks = 0;                 // 16 x 16 blocks of one panel's factor; block nblocks is zero
    int64_t estore = 0;              // entries of all E of one panel, of the largest group
    std::vector<int32_t> sxy, sv;    // qxy, qv per panel-vector row (sv -1: padding)
    std::vector<int32_t> browBase, browLo;
    std::vector<int32_t> udst;       // vector row an update row is added into, see VecRows
    std::vector<int32_t> usrc;       // panel-vector row of an update row (backward input)
    std::vector<FoldNode> foldNodes;
    std::vector<TransItem> packs;    // 32 x 32 pieces copied into F: node, row, column of its front
    std::vector<ComposeDesc> compose;
    std::vector<ComposeKey> fkeys;
    std::vector<GemmTile> composeTiles;    // pad_: keys that meet the tile's rows
    std::vector<GemmLaunch> composeSteps;  // per group by depth below its top, 1, 2, ...
    std::vector<int32_t> flist, fsrc;
    // The fold goes group by group, so that the update scratch holds the E of
    // one group at a time: all of them at once were more than the updates of a
    // level (7.8 against 7.3 GB at 100^3 in FP64, 39 against 33 at 200 x 200 x 100).
    struct FoldGroup {
        GemmLaunch e;                // E = -L_BL Linv
        int packStart = 0, packCount = 0, stepStart = 0, stepCount = 0;
    };
    std::vector<FoldGroup> foldGroups;   // per depth group
    struct BlockLevel {              // one group: tiles and reduce items per direction
        int start[2] = {0, 0}, count[2] = {0, 0};
        int rstart[2] = {0, 0}, rcount[2] = {0, 0};
        double entries[2] = {0, 0}, vecRows[2] = {0, 0};
    };
    std::vector<std::array<int, 2>> slices;  // per group and direction: inner blocks per tile
    std::vector<BlockLevel> blevels;
    std::vector<BlockTile> btiles;
    std::vector<BlockRed> breds;
    std::vector<int32_t> blist;      // backward: 4 blocks per inner block (nblocks: not stored)
    std::vector<int32_t> bsrc;       // backward: 16 vector rows per inner block
    int bslots = 0;

    // Algorithmic work per panel.
    double flops = 0, schurFlops = 0, solveFlopsPerRhs = 0;
    double factorEntries = 0;
};

struct Plan {
    Geometry geo;
    ClassPlan cls[3];
    bool present[3] = {false, false, false};
    int blockNb = 32;      // LDL^T block width
    int tile = 64;         // GEMM tile
    int minTiles = 256;    // solve tiles wanted per launch (default shapes)
    int maxSplit = 8;      // inner slices per row block at most (default shapes)
    bool persist = true;   // without effect
    bool fused = false;    // fused subtree launches (8 <= k <= 16)
    int fusedCut = -1;     // cut depth of the fused launches (-1: the first with
                           // at least kQueues nodes)
    int fusedRows = 32;    // output rows per queue tile
    int fusedQueues = kQueues;  // queues (more than the device's XCDs leaves
                                // queues that the last workgroup runs alone)
    int fusedWgPerQueue = 64;   // workgroups a queue expects (inner slices are
                                // cut so a level has about that many tiles)
};

// Rows (of the solve vector) and entries (of bsrc) a workgroup may read past
// its tile's inner range, unused.
constexpr int kStagePad = 256;

// Rows of a class's solve vector, one buffer: the panel vector (xrows rows
// and 16 zero rows), the forward results (xrows), and two copies of what
// children add to a front: g0, its update rows (at their u0), and g1, all its
// work rows (at w0).  A child adds into its parent's pivot rows in place
// (panel-vector rows) when it is the first to touch them, and to its parent's
// update rows in g0; the second child to touch a row writes it in g1.  No row
// is touched by more than two children.
struct VecRows {
    int64_t w, g0, g1, total;
    explicit VecRows(const ClassPlan& C)
        : w(C.xrows + kBlk), g0(w + C.xrows), g1(g0 + (int64_t)C.udst.size()),
          total(g1 + C.wrows + kStagePad)
    {
    }
};

// Depth groups of the merged solves, the merged fronts and the fold's work
// lists.  entryBytes: bytes of a factor entry.
void BuildMerged(ClassPlan& C, int entryBytes);
// Inner blocks per tile: as many as give about `minTiles` workgroups a launch,
// in at most maxSplit slices.
void DefaultSlices(ClassPlan& C, int minTiles, int maxSplit);
// (Re)builds the merged solves' tiles from C.slices.
void BuildBlockTiles(ClassPlan& C);

// Builds everything; returns PSP_HIP_OK or an error code with `msg` set.
int BuildPlan(const psp_hip_desc& desc, Plan& plan, std::string& msg);

// Solve tile shapes: the default per (level, phase) is the largest row
// block of 64, 32, 16 rows that gives minTiles tiles, and otherwise inner
// slices (at most maxSplit) to reach minTiles.
void DefaultSolveShapes(ClassPlan& C, int minTiles, int maxSplit);
// (Re)builds the solve tiles, reduce items and their accounting from
// C.shapes.
void BuildSolveTiles(ClassPlan& C);
// (Re)builds the fused subtree launches of a class (after BuildSolveTiles:
// uses its per-level accounting and raises maxSlots to cover the queues'
// partial slots).  nqueues <= 0 or a tree with no level of nqueues nodes
// leaves qcut = -1.
void BuildQueues(ClassPlan& C, int nqueues, int rows, int cut, int wgPerQueue);

}  // namespace psp_amd
