// FP64 geometric multigrid for the cut-domain 5-point Poisson operator of
// PoissonSolver::cutoffStencil (PoissonSolver.cpp:678-766).
//
// Operator on an nx x ny node grid (callers' arrays row-major, x fastest),
// spacings hx (already multiplied by gamma for the boosted frame) and hy:
//   unknown rows:   2(cx+cy) phi_ij - cx (phi_i-1,j + phi_i+1,j) - cy (phi_i,j-1 + phi_i,j+1) = b_ij
//                   with cx = 1/hx^2, cy = 1/hy^2; neighbours that are not
//                   unknowns contribute zero (Dirichlet) unless they are
//                   "known" nodes, whose value b moves to the right-hand side;
//   other rows:     identity, phi = b.
// For gamma >> 1 the x coupling is weaker than the y coupling by
// (hy / (gamma hx))^2, so the smoother is an exact y-line solve (red/black
// column order) and coarsening halves x only.  That pairing converges at a rate
// that does not depend on the anisotropy.
//
// Inside the solver a level's arrays are column by column, in the order in
// which one wave solves a line: lane l holds rows l M .. l M + M - 1, and
// row_pos() puts row pair t of all lanes side by side, so that every load and
// store of the wave is one contiguous kilobyte.  With plain columns a lane's
// 16 rows lie 128 bytes from the next lane's and each load took 64 cache lines:
// a half sweep, averaged over the levels of a 2048 x 1024 grid, took 8.7 us and
// takes 4.7 us (15.8 us with parallel cyclic reduction over row-major arrays).  Callers' arrays are brought into this order once on the way
// in and back once on the way out.  Values at nodes that are not unknowns are
// zero on every level.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "hip_util.h"

namespace pmg {

enum NodeClass : uint8_t { kFixed = 0, kUnknown = 1, kKnown = 2 };

constexpr int kMaxLane = 32;      // rows of a line per lane; longer lines run in chunks of 64 kLongLane rows
constexpr int kLongLane = 16;

// place of row j in a column of M rows per lane
__host__ __device__ inline int row_pos(int j, int M)
{
    const int N = 64 * M, c = j / N, r = j - c * N, lane = r / M, t = r - lane * M;
    return c * N + (t >> 1) * 128 + lane * 2 + (t & 1);
}

// The unknowns of a level-0 column: rows lo <= j < hi, or several runs of rows
// (hi = -1), or none (lo = hi).  tab: the table of elimination factors for runs
// that start at lo, or -1.  Coarsening keeps every second column, so column I
// of level l has the unknowns of column I << l of level 0.
struct alignas(16) ColRows {
    int lo, hi, tab, pad;
};

struct Level {
    int nx = 0, ny = 0, pitch = 0;
    int lane = 0;                    // rows per lane (M)
    int shift = 0;                   // column I of this level is column I << shift of level 0
    double cx = 0, cy = 0;
    const ColRows *rows = nullptr;   // of level 0
    const uint8_t *act = nullptr;    // of level 0: 1 = unknown
    const double *g = nullptr;       // elimination factors of the k-th row of a run
    const double *gt = nullptr;      // tables of them in column order, `pitch` apart, one per run start
    double *phi = nullptr, *rhs = nullptr;
    double *res = nullptr;           // level 0 only
    // where row j of column i lies
    __host__ __device__ size_t at(int i, int j) const { return (size_t)i * pitch + row_pos(j, lane); }
};

struct Stats {
    int cycles = 0;
    double resid0 = 0, resid = 0, bnorm = 0;   // ||r|| at start and end, ||b|| (unknown rows)
};

struct Tail;

class Solver {
public:
    Solver() = default;
    Solver(const Solver &) = delete;
    Solver &operator=(const Solver &) = delete;
    ~Solver();
    // cls: device array of NodeClass, nx*ny.  Allocates the level hierarchy.
    void setup(int nx, int ny, double hx, double hy, const uint8_t *cls, hipStream_t s);
    // b: device, nx*ny right-hand side of every row; phi: device, in = initial
    // guess, out = solution (identity rows set to b).  Iterates V(2,2) cycles
    // until ||b - A phi|| <= tol ||b|| over unknown rows, maxit cycles, or
    // three cycles in a row that reduce the residual by less than 5% (the
    // round-off floor of the grid).
    Stats solve(const double *b, double *phi, double tol, int maxit);
    // residual norm of phi (device) against b without iterating
    double residual(const double *b, const double *phi);
    // Step-wise use (a caller that acts on the iterate between V-cycles):
    // begin() loads b and the guess phi0 (device) and returns ||b||; resnorm()
    // computes the level-0 residual (level0().res) and returns its norm over
    // the unknowns; cycle() runs one V-cycle on level0().phi; store() writes
    // the solution (identity rows phi = b) to phi (device).
    double begin(const double *b, const double *phi0);
    double resnorm();
    void cycle();
    void store(const double *b, double *phi);
    const Level &level0() const { return lv_[0]; }
    size_t level0_size() const { return (size_t)nx_ * lv_[0].pitch; }   // elements of a level-0 array
    hipStream_t stream() const { return s_; }
    int nx() const { return nx_; }
    int ny() const { return ny_; }
    int levels() const { return (int)lv_.size(); }

private:
    double read_norm();
    int nx_ = 0, ny_ = 0;
    hipStream_t s_ = nullptr;
    const uint8_t *cls_ = nullptr;
    std::vector<Level> lv_;
    hu::DBuf<uint8_t> cols_, mem_;   // the columns' unknowns; everything else
    double *partial_ = nullptr;
    Tail *tail_ = nullptr;           // the coarse levels that one workgroup takes: t0_ and below
    int t0_ = 0, coarse_ = 0;        // coarse_: sweeps on the coarsest level
    double *hnorm_ = nullptr;        // pinned host memory: the norm's last kernel writes it
    int npart_ = 0;
};

// Between a caller's row-major image (x fastest) and a level-0 array: the
// workgroup's 32 x 32 tile with its origin at column i0, row j0.  Callers
// read the image with x across the lanes, keep the tile in LDS, and write the
// level with y across the lanes (or the reverse); the odd LDS pitch keeps both
// passes free of bank conflicts.  The tiles are a flat grid: a grid's y dimension
// ends at 65535, and a grid may have more columns, or rows of tiles, than that.
constexpr int kTile = 32;
inline unsigned num_tiles(int nx, int rows)
{
    return (unsigned)((nx + kTile - 1) / kTile) * (unsigned)((rows + kTile - 1) / kTile);
}
__device__ __forceinline__ void tile_origin(int nx, int &i0, int &j0)
{
    const unsigned across = (unsigned)(nx + kTile - 1) / kTile;
    i0 = (int)(blockIdx.x % across) * kTile;
    j0 = (int)(blockIdx.x / across) * kTile;
}

}  // namespace pmg
