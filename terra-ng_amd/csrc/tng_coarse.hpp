// Solvers on the coarsest multigrid level (kernels_coarse.hip): direct, and PCG on
// the assembled operator.
#pragma once

#include <cstdint>

#include "tng_internal.hpp"

namespace tng {

struct CoarseDirect {
    static constexpr int kMaxUnknowns = 6000;  // 288 MB of FP64 inverse at most
    int nu = 0, n = 0;                          // unique nodes, unknowns (3 nu)
    int64_t ncopies = 0;
    bool ready = false;
    DevBuf d_uid, d_rep, d_M, d_row, d_col, d_b, d_x;
    void numbering(const tng_domain &m);
    // the inverse of A over the unique node components; x, y: FP64 work vectors on A's mesh
    // (fp32_levels: the V-cycle's other levels are FP32; with the fs/fs penalty
    // the rotations are then projected out, see project_rotations)
    void build(tng_operator &A, tng_vector &x, tng_vector &y, bool fp32_levels, hipStream_t s);
    // e0 = A^{-1} r0 on every node copy (r0 consistent over the copies)
    void solve(tng_vector &e0, const tng_vector &r0, hipStream_t s);
    // M <- P M P, P the projection off the three rigid rotations (fs/fs penalty)
    void project_rotations(const tng_domain &m, hipStream_t s);
};

// PCG with the identity preconditioner on the assembled coarsest operator
// (linalg/solvers/pcg.hpp:81-170 from a zero guess): 3 x 3 blocks over the
// unique nodes, boundary rows included, two kernels per iteration.
struct CoarsePcg {
    static constexpr int kMaxNodes = 8192, kWidth = 24;  // unique nodes; blocks per row (at most 21 are used)
    static constexpr int kMaxSlots = 72;                 // 12 wedges x 6 nodes around a node copy
    int nu = 0;
    int64_t ncopies = 0;
    bool ready = false;
    DevBuf d_uid, d_rep, d_slot, d_col, d_copy_begin, d_copy_list, d_A, d_vec, d_state;
    // the operator is a plain one (no rotation penalty) on a mesh of this size
    static bool accepts(const tng_operator &A);
    void numbering(const tng_domain &m);
    void build(tng_operator &A, hipStream_t s);  // after every change of the coefficient
    // e0 = the iterate after at most max_it steps, on every node copy (r0 consistent over the copies)
    void solve(tng_vector &e0, const tng_vector &r0, int max_it, double rtol, double atol, hipStream_t s);
    // iterations since the last call (synchronises)
    long take_iterations(hipStream_t s);
};

}  // namespace tng
