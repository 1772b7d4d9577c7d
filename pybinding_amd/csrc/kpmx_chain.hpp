// Launch interface of the chained diagonal recurrence (kpmx_chain.hip): several Chebyshev steps per
// launch on row tiles whose vectors stay in LDS.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace kpmx {

constexpr int CHAIN_MAX_STEPS = 12;      // steps per launch at most
constexpr int CHAIN_MAX_HALO = 6144;     // halo rows of a tile at most
constexpr int CHAIN_CANDIDATES = 8;      // tile heights whose halos one chain_sample measures
constexpr int CHAIN_SAMPLES = 32;        // tiles it looks at per height

// Matrix entries of a plan: every stored value (standard SELL), 1-byte codes into a value table,
// or one value for all off-diagonal entries; the last two keep the diagonal as a dense vector.
enum { CHAIN_STD = 0, CHAIN_TABLE = 1, CHAIN_UNIFORM = 2 };

// The SELL-64 matrix a plan is built from: with codes the off-diagonal entries and the diagonal.
struct ChainMatrix {
    int scalar = 1;
    int64_t n = 0;
    // row order of the plan's tiles: perm[plan row] = matrix row, place[matrix row] = plan row (null:
    // the matrix's own).  The work vectors are in plan order, the first launch's x, weights and marks in
    // matrix order; panels need the matrix's own.
    const int32_t* perm = nullptr;
    const int32_t* place = nullptr;
    bool adjoint = false;  // for the backward recurrence: two vectors in LDS, standard form
    int max_width = 0;
    const int64_t* slice_ptr = nullptr;
    const int32_t* slice_width = nullptr;
    const int32_t* indices = nullptr;
    const void* vals = nullptr;      // standard form
    const uint8_t* codes = nullptr;  // value-table form
    const void* diag = nullptr;
    const void* table = nullptr;     // zero first; several systems' tables one after another
    int table_size = 0;
    int table_most = 0;              // entries of the largest of them
    // value-table form of 32-bit types: the standard SELL of the same rows, whose entry order (diagonal
    // in its place) the plan keeps
    const int64_t* row_ptr = nullptr;
    const int32_t* row_width = nullptr;
    const int32_t* row_indices = nullptr;
    const void* row_vals = nullptr;
    int row_max_width = 0;
    __host__ __device__ bool ordered() const { return codes && (scalar == 0 || scalar == 2); }
    __host__ __device__ int width() const { return ordered() ? row_max_width : max_width; }  // entries of a plan's rows
    __host__ __device__ int form() const { return !codes ? CHAIN_STD : table_most <= 2 ? CHAIN_UNIFORM : CHAIN_TABLE; }
};

// Device arrays of a plan.  Tile t owns rows [tile_begin[t], tile_begin[t + 1]); its local rows are
// those, then its halo: the rows at distance 1, 2, ..., `steps` from them in the matrix's graph
// (ext, ascending inside a ring).  ring[t * (CHAIN_MAX_STEPS + 1) + j] counts the local rows up to
// distance j.  Entries are kept for the local rows up to distance steps - 1.
struct ChainPlan {
    int64_t ntiles = 0, tile_rows = 0;
    int steps = 0;      // steps per launch the entries reach for
    int width = 0;      // entries per row
    int groups = 0;     // ceil(width / 4)
    int rows_x = 0;     // most local rows of a tile (distance <= steps)
    int rows_y = 0;     // row stride of the entry arrays (rows at distance <= steps - 1, padded)
    int row_items = 1;  // items of a row
    int64_t ext_stride = 0;
    int32_t* tile_begin = nullptr;
    int32_t* tile_table = nullptr;  // first entry of the tile's value table (null: 0)
    int32_t* ring = nullptr;
    int32_t* ext = nullptr;
    ushort4* lidx = nullptr;    // [tile][group][row], first item of the column's local row (none: the zero row)
    uint32_t* codes = nullptr;  // [tile][group][row], four 1-byte codes
    void* vals = nullptr;       // [tile][entry][row]
    void* diag = nullptr;       // [tile][row]
};

// (launches return 0, or -1 where the device refuses)
// local rows (distance <= j) of sampled tiles of each candidate height: out[(c * CHAIN_SAMPLES + s)
// * (CHAIN_MAX_STEPS + 1) + j], -1 where they exceed `capacity` rows
int chain_sample(const ChainMatrix& m, const int* heights, int count, int capacity, int32_t* out, hipStream_t s);
// ring counts and halo rows (at most P.ext_stride) of every tile (P.tile_begin set; P.ring, P.ext
// allocated)
int chain_rings(const ChainMatrix& m, const ChainPlan& P, int max_steps, hipStream_t s);
// entry arrays of every tile (P.steps, rows_x, rows_y set and the arrays allocated)
int chain_entries(const ChainMatrix& m, const ChainPlan& P, hipStream_t s);

// Reverse steps j, j - 1, ..., j - steps + 1 of the adjoint (kpmx_chain_adjoint.hip) on `cols` columns:
// reads v_j, v_j+1, lambda_j+1, lambda_j+2 (lam null: both zero) and writes the same four `steps` lower
// (v_out null: no v, lam_next_out null: lambda_j+1-steps only); grad[4 row + k] of every stored entry is
// updated.  The outputs are no inputs.
struct AdjointChainLaunch {
    ChainMatrix m;  // standard form
    const ChainPlan* plan = nullptr;
    int cols = 4, steps = 1;
    int64_t ldv = 0, ldlam = 0;  // row strides of v and v_next, of lam_out in scalars (the others: cols)
    const void* v = nullptr;
    const void* v_next = nullptr;
    const void* lam = nullptr;
    const void* lam_next = nullptr;
    void* v_out = nullptr;
    void* v_next_out = nullptr;
    void* lam_out = nullptr;
    void* lam_next_out = nullptr;
    double* grad = nullptr;
    double ca[CHAIN_MAX_STEPS], chv[CHAIN_MAX_STEPS], cg[CHAIN_MAX_STEPS];  // of step j - i
};
int chain_adjoint_cols(int scalar, int vw);  // columns of a group of blocks of vw >= 4
// local rows, own rows and row padding of its tiles (-1: no such layout); at most 4 entries per row
int chain_adjoint_capacity(int scalar, int cols);
int chain_adjoint_own_rows(int scalar, int cols);
int chain_adjoint_row_pad(int scalar, int cols);
int launch_adjoint_chain(const AdjointChainLaunch& L, hipStream_t s);
// grad (SELL order, every stored entry) from the row-major sums
void launch_adjoint_chain_grad(const ChainMatrix& m, const double* rows, double* grad, hipStream_t s);

// What a step leaves beside the vectors: the diagonal sums, the dots with a weight vector, panel rows
// of the new vector, panel rows of an operator applied to the vector before, or the new vector at
// marked rows.
enum { CHAIN_SUMS = 0, CHAIN_DOTS = 1, CHAIN_PANEL = 2, CHAIN_PANEL_OP = 3, CHAIN_MARKS = 4 };

// An operator's entries on a plan's tiles (their own rows only).
struct ChainOp {
    int groups = 0, rows = 0;  // groups of four entries per row; row stride
    ushort4* lidx = nullptr;
    void* vals = nullptr;
};
// fills op (allocated for groups and rows) from the operator's SELL arrays (standard form); *missing
// is set to 1 where an entry's column is no local row of its tile
int chain_op_entries(const ChainMatrix& op, const ChainPlan& P, const ChainOp& o, int32_t* missing, hipStream_t s);

struct ChainLaunch {
    int mode = CHAIN_SUMS;
    ChainMatrix m;
    const ChainPlan* plan = nullptr;
    int cols = 8;              // vectors per row of the work blocks
    int steps = 1;             // steps of this launch (<= plan->steps)
    bool first = false;        // the first step is 0.5 H2 x
    const void* x = nullptr;   // r_k, rows of ldx scalars
    int64_t ldx = 0;
    const void* xprev = nullptr;  // r_{k-1}, rows of `cols` scalars (not read by a first launch)
    void* out1 = nullptr;         // r_{k+steps-1} (not written by a one-step launch)
    void* out2 = nullptr;         // r_{k+steps}
    int64_t ldprev = 0, ldout = 0;  // row strides of xprev and of out1 and out2 in scalars (0: cols)
    double* partials = nullptr;   // [steps][ntiles][chain_partial_width] (sums and dots)
    // sums: groups of `cols` columns in one launch, and the strides between them of x, of xprev, out1 and
    // out2 (in scalars) and of the partials
    int col_groups = 1;
    int64_t x_group = 0, w_group = 0, partials_group = 0;
    const void* w = nullptr;      // dots (one column): n weights
    // panels: column q of r_{k+j} (of the operator on r_{k+j-1}) goes to panel + q panel_col + p panel_step
    // + row (scalars) with p = j (p = j - 1), step j = 1 ... steps; the operator's first row is halved
    // in a first launch
    void* panel = nullptr;
    int64_t panel_col = 0, panel_step = 0;
    const ChainOp* op = nullptr;
    // marks (one column): r_{k+j} of row i goes to mark_out[mark[i] mark_stride + j] where mark[i] >= 0
    const int32_t* mark = nullptr;
    void* mark_out = nullptr;
    int64_t mark_stride = 0;
};
// widest supported column tile of a scalar type
int chain_max_cols(int scalar);
// local rows one workgroup's LDS holds
int chain_row_capacity(const ChainMatrix& m, int cols);
// items of a row (see kpmx_chain_step.hpp); the row stride of the entry arrays is a multiple of pad
int chain_row_items(int scalar, int cols);
int chain_row_pad(const ChainMatrix& m, int cols);
int chain_partial_width(int scalar, int cols, int mode = CHAIN_SUMS);
int launch_chain(const ChainLaunch& L, hipStream_t s);
int launch_chain_f32(const ChainLaunch& L, hipStream_t s);
int launch_chain_f64(const ChainLaunch& L, hipStream_t s);
int launch_chain_c64(const ChainLaunch& L, hipStream_t s);
int launch_chain_c128(const ChainLaunch& L, hipStream_t s);
// sums[step][system][4 vw] of the columns [c0, c0 + cols) of a vw-column block from the partials of
// nsteps steps; system_tiles (num_systems + 1) null: one system over all tiles
void launch_chain_reduce(int scalar, int mode, const double* partials, int64_t ntiles, int cols, int64_t nsteps,
                         const int32_t* system_tiles, int64_t num_systems, int vw, int c0, double* sums, hipStream_t s);

}  // namespace kpmx
