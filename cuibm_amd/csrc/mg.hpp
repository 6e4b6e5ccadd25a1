// Multigrid preconditioner of the pressure-Poisson operator in stencil form (plain and Luo
// solvers), in place of a stored hierarchy.
//
// The operator is a tensor sum A0 = Tx (+) Ty of two tridiagonal matrices (finite volumes,
// per cell volume: off-diagonals -dt / (w_I (w_I + w_{I+1}) / 2)) plus the doubled diagonal
// of cell 0 and, for the plain solver, of the centre cell. Every level here is such a tensor
// sum too, on a grid whose cells are unions of the finer level's: 1-D arrays of O(nx + ny)
// values describe it, so no level but the finest vector moves more than its unknowns.
//
//  - Coarsening by cell width. A stretched grid's point smoother leaves errors that oscillate
//    along the wide side of flat cells, and aggregates that merge cells whatever their shape
//    cannot represent them: the aggregation hierarchy of the 1024 x 1024 cylinder took 27-38
//    BiCGSTAB iterations. Here two neighbours of an axis merge while their joint width stays
//    below a threshold (MG_WIDTH times the level's smallest cell), so flat cells coarsen along
//    their narrow side only until they are square: 3 iterations, of the same cost.
//  - Restriction is the volume average of the residual over an aggregate, prolongation linear
//    interpolation between the aggregates' centres; the coarse operator is the same finite-
//    volume formula on the coarse widths.
//  - Smoothing: three weighted-Jacobi sweeps before and after, with the weights of a
//    Chebyshev polynomial on the upper part of D^-1 A's spectrum.
//  - The level whose axes both have at most MG_FDM_MAX cells is solved exactly by fast
//    diagonalisation (Lynch, Rice & Thomas 1964): Tx and Ty have full sets of eigenvectors
//    (a diagonal scaling makes them symmetric), so the pseudo-inverse of A0 is four dense
//    products with the 1-D eigenvector matrices, on the matrix cores.
//  - A grid of at most MG_DIRECT_MAX cells an axis is that level itself, in FP64: the
//    preconditioner is then the exact inverse of A, pins included, and BiCGSTAB leaves after
//    its first half step.
//  - The constant mode, fixed only by the pins, is carried in FP64 around the cycle: with
//    the cell areas w, w^T A0 = 0 and w^T A = (w o a)^T with a = A 1 nonzero only at the pins;
//    for the input r, c = w^T r / w^T a and A^-1 r = A^-1 (r - c a) + c 1.
#pragma once
#include <memory>
#include <vector>

#include "krylov.hpp"

namespace cuibm {

// Sizes at which a level is solved directly: below the finest level, 224 cells an axis (14 tiles
// of 16), where three more levels and a dense solve took 28 us of a cycle against 12 for the
// four products (a cycle with 128, 224, 320: 336^2 46, 38, 28 us; 498^2 59, 52, 46; 1024^2 87, 79,
// 78, the steps within 1% from 224 up); as the finest level, 320, where the exact inverse saves the
// Krylov iterations (its products grow as n^3: 25 us at 200^2, 37 at 300^2, 55 at 390^2). The line
// could lie higher: a 336^2 cylinder's FP32 step takes 0.44 ms solved directly and 0.74 with levels,
// but from 336^2 on solves are to run on three levels or more, which the tests check.
constexpr int MG_FDM_MAX = 224, MG_DIRECT_MAX = 320;
// width threshold of the coarsening, in smallest cells of the level. Time steps of the 1024^2,
// 498^2 and 336^2 cylinders with 4, 5, 6, 7 (FP32 levels): 1.56, 1.59, 1.47, 1.54 ms; 1.60,
// 1.66, 1.65, 1.87; 1.11, 1.19, 1.02, 1.19. Twice the iterations at 12.
constexpr double MG_WIDTH = 6.0;

// one smoothed level as the kernels see it; the arrays have nx or ny entries
template <class T>
struct MgLevelDev {
    int nx = 0, ny = 0;
    int ld = 0;                         // row stride of the level's vectors
    int ldc = 0;                        // row stride of the next coarser level's
    const T *cE, *cW, *cN, *cS;         // coupling magnitudes, 0 towards a missing neighbour
    const T *rx, *ry;                   // w_I / (width of I's aggregate)
    const T *tx, *ty;                   // interpolation weight of the other aggregate
    const int *ax, *ay, *ox, *oy;       // own and other aggregate
};

// a directly solved level; F = Q^T W^(1/2) and B = W^(-1/2) Q of each axis, row-major with
// rows and columns padded by zeros to multiples of 16
template <class T>
struct FdmDev {
    int nx = 0, ny = 0, px = 0, py = 0;
    const T *Fx, *Fy, *Bx, *By, *lx, *ly;  // l: eigenvalues
    int zx = 0, zy = 0;                    // the axes' zero modes
    T *t1, *t2;                            // scratch, px py values each
};

// the pins and the constant mode's constants (see above)
struct MgPins {
    int centre = -1;             // second pinned cell or -1
    double a0 = 0, ac = 0;       // A 1 at cell 0 and at the centre
    double inv_wa = 0;           // 1 / w^T a
    const double *part = nullptr;  // npart partial sums of w_i r_i
    int npart = 0;
    double *c = nullptr;         // the constant of the last input
    // direct solves with two pins: A0^+ (a0 e_0 - (w_0 a0 / w_c) e_centre), and
    // 1 / (1 + w_0 a0 / (w_c ac) + H(0) - H(centre))
    const double *H = nullptr;
    double hq = 0;
};

// One case's arguments of the level kernels (in a batch: one per case of the level). The
// finest level's vectors are the Krylov vectors, FP64; coarser ones are of type T.
template <class T>
struct MgTask {
    MgLevelDev<T> L;
    const T *b;          // right-hand side (levels below the finest)
    T *x3, *rc;          // smoothed iterate, restricted residual
    const T *e;          // the coarser level's solution
    T *x;                // result (levels below the finest)
    T w[3];              // sweep weights, ascending
    MgPins pins;         // finest level
    long off;            // offset of the case in the Krylov vectors
    const double *stop;  // Krylov stop code: the kernels return at once while it is set
};

template <class T>
struct FdmTask {
    FdmDev<T> F;
    const T *b;    // right-hand side (below the finest level), row stride px
    T *x;          // result, row stride px
    MgPins pins;   // finest level
    long off;
    const double *stop;
};

// host description of one level (mg_setup.cpp)
struct MgHostLevel {
    std::vector<double> dx, dy;
    std::vector<int> ax, ay, ox, oy;    // towards the next level (empty on the last)
    std::vector<double> tx, ty;
};
// the levels of a grid: coarsened until both axes have at most `cap` cells and the level at
// most `most` unknowns (most <= 0: no such limit)
std::vector<MgHostLevel> mg_levels(const std::vector<double> &dx, const std::vector<double> &dy, int cap, long most);
// eigenvalues lam and eigenvectors (row k of q) of the symmetric tridiagonal matrix with
// diagonal d and off-diagonal e
void tridiagonal_eigen(std::vector<double> d, std::vector<double> e, std::vector<double> &lam, std::vector<double> &q);
// coupling magnitudes of one axis: towards the next and the previous cell
void axis_couplings(const std::vector<double> &w, double dt, std::vector<double> &next, std::vector<double> &prev);
// F, B (padded row-major) and eigenvalues of one axis, and its zero mode
struct AxisModes {
    int n = 0, pad = 0, zero = 0;
    std::vector<double> F, B, lam;
};
AxisModes axis_modes(const std::vector<double> &w, double dt);

// whether the widths of an axis can be coarsened: finite, none zero, all of one sign (the
// operator holds products of two widths, so an axis may run downwards)
bool mg_axis(const std::vector<double> &w);

// the preconditioner of one case, on axes that mg_axis() accepts; `precision` 64, 32 (levels in FP32) or 3264 (level
// coefficients rounded to FP32, vectors and arithmetic in FP64)
class TensorMg {
  public:
    TensorMg(const std::vector<double> &dx, const std::vector<double> &dy, double dt, int centre, int precision,
             int coarse_max, const double *dx_dev, const double *dy_dev, hipStream_t s);
    ~TensorMg();
    void apply(const double *r, double *z, hipStream_t s, bool weighted);
    InputWeights weights() const { return w_; }
    void set_stop(const double *stop);
    // cells of each level; the last is the directly solved one
    const std::vector<std::pair<int, int>> &sizes() const { return sizes_; }
    std::vector<double> launch_bytes() const;  // per launch of one apply, in order
    KernelProbe &probe() { return probe_; }
    // the first and the last finest-level kernel alone (timing), and their bytes
    void fine_first(const double *b, hipStream_t s);
    void fine_last(const double *b, double *z, hipStream_t s);
    double fine_first_bytes() const { return launch_bytes().front(); }
    double fine_last_bytes() const { return launch_bytes().back(); }

  private:
    friend class BatchMg;
    template <class T>
    struct Levels;
    InputWeights w_;
    P5Dev wdot_{};
    std::vector<std::pair<int, int>> sizes_;
    std::unique_ptr<Levels<double>> d_;
    std::unique_ptr<Levels<float>> f_;
    KernelProbe probe_;
};

}  // namespace cuibm
