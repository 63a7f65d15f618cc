// Smoothed-aggregation multigrid (lh_amg.hip): the preconditioner of the
// linear solves on large systems (FP64) and of the block eigensolver (FP32
// blocks, as its Chebyshev polynomial's arithmetic).
#pragma once
#include "lh_dense.hpp"

namespace lh {

// one level's operators in the precision T of the cycle
template <typename T>
struct AmgOps {
    const T* kv = nullptr;    // K (the level's CSR slots; level 0 with an ELL copy: its slots)
    const T* dinv = nullptr;  // 1 / diag K, smaller in the guarded rows (0 on a zero row)
    const T* pv = nullptr;    // P
    const T* rv = nullptr;    // P^T
};

struct AmgLevel {
    int64_t n = 0, nnz = 0;
    const int32_t* rp = nullptr;  // K: CSR
    const int32_t* cl = nullptr;
    int W = 0;  // level 0 with an ELL copy: slots per row; 0: CSR
    const int32_t* ecl = nullptr;
    const double* ekv = nullptr;
    const float* ekv32 = nullptr;
    double bmax = 2.0;  // upper end of the smoother's interval
    // transfer to the next level (absent on the last one)
    int64_t nc = 0, pnnz = 0;
    const int32_t *pp = nullptr, *pc = nullptr;  // P (n x nc), CSR
    const int32_t *tp = nullptr, *tc = nullptr;  // P^T (nc x n), CSR
    AmgOps<double> d;
    AmgOps<float> f;  // the block cycle's
    const AmgOps<double>& ops(double) const { return d; }
    const AmgOps<float>& ops(float) const { return f; }
};

struct Amg {
    // Hierarchy of the n x n operator with CSR slots (rp, cl, kv); symmetric,
    // diagonal positive except on zero rows.  ell_w > 0: an ELL copy (ecl,
    // ekv) for the products of the finest level.  Returns false (nothing to
    // free) when no useful hierarchy exists: a negative diagonal, coarsening
    // that stalls, or a coarsest matrix that does not factorise.
    // coarse_shift: what raises the unit diagonal of the equilibrated
    // coarsest matrix, kShiftF64 or kShiftBlocks.
    bool setup(lh_ctx* ctx, int64_t n, int64_t nnz, const int32_t* rp, const int32_t* cl, const double* kv, int ell_w,
               const int32_t* ecl, const double* ekv, double coarse_shift);
    static constexpr double kShiftF64 = 1e-9, kShiftBlocks = 1e-5;
    // work blocks for m columns in double precision
    void prepare(int m);
    // Z <- M R, row-major n x m; a set status[0] makes every launch return at
    // once.  part (not null; m <= 4): dot_blocks() partial sums of each
    // column of R . Z, part[block * m + column]
    void apply(const double* R, double* Z, double* part, const int* status);
    int dot_blocks() const;  // 0: more than four columns

    // the block cycle for at most m columns: FP32 copies and work blocks.
    // ell_w == 8: the columns of an ELL copy of the finest level's pattern
    void prepare_blocks(int m, int ell_w, const int32_t* ecl);
    // columns perm[0 .. cols - 1] of W (leading dimension ldw; null: the first
    // cols) <- p(M K) M times them, in FP32; columns perm[cols .. total - 1] <-
    // D^-1 times them
    template <typename WT>  // double or float
    void apply_blocks(WT* W, int ldw, int cols, int total, const int32_t* perm);

    // products with the finest K in one application: four a cycle, one between two
    int block_products() const { return 5 * cycles - 1; }

    std::vector<AmgLevel> levels;

   private:
    lh_ctx* ctx = nullptr;
    int m = 0;
    int tail = 0;  // first level of the one-launch tail
    std::vector<DevBuf> keep;  // every level's arrays
    DevBuf ginv;               // inverse of the coarsest matrix (nl x nl)
    DevBuf work;
    DevBuf tail_desc;          // the tail's levels, for its kernel
    std::vector<double*> wb, wx, wy, wr;  // per level: right-hand side, iterate, second iterate, residual
    double rough = 0.0;        // the finest level's estimate of lambda_max(D^-1 K)
    int ld = 0;                // block cycle: columns rounded up to 4
    int cycles = 2;            // combined in one application
    float *bin = nullptr, *bx1 = nullptr, *bx2 = nullptr;
    std::vector<float*> fb, fx, fy, fr;
    template <typename T> void describe_tail();
    template <int MODE> void blk_step(int l, int w, const float* b, const float* x, float* out, float w0, float w1, float g);
    void cycle_blocks(int l, int w, const float* b, float* x);
    template <typename X> X* own(size_t count);
    void cycle(int l, const double* b, double* x, double* part, const int* status);
};

// 2 tr(D) / 1^T K 1: a lower bound of the condition number of D^-1 K for an
// operator with a mass term (close to it when the mass is spread evenly)
double amg_condition(lh_ctx* ctx, int64_t n, const int32_t* rp, const int32_t* cl, const double* kv,
                     const double* dinv);

}  // namespace lh
