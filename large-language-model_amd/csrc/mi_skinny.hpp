// mi_skinny.hpp -- plan and launch interface of the skinny GEMM kernels (mi_skinny.hip):
// products of a few rows, called by the dispatch in mi_gemm.hip.
#pragma once
#include "mi_gemm_device.hpp"

namespace mig {

// Rows that the kernels take.  Above 32 rows only while B is at most SKINNY_WIDE_BYTES: a lane
// then issues as many loads of A as of B, and a larger B fills the chip with 128-row tiles
// anyway (64 rows, bf16: a layer of width 2048, whose largest B has 23 MB, 103 -> 84 us; the
// logits of a 131 MB table with their two gradients 150 -> 167 us).
// Taller fp32 NN products whose 64-row x 32-column blocks fill at least half of the CUs and at
// most all of them, K up to 1024, take them too: each block on a workgroup of 8 waves that
// share K.  A tile kernel leaves them the choice between idle CUs and a second launch (512 x
// 768 x 768 with bias: 64x128 tiles split 5 16.0 us, 64x64 tiles 16.9, here 12.1).  The NT
// form would read A again for every 16 columns.
constexpr int SKINNY_MAX_M = 64;
constexpr int64_t SKINNY_WIDE_BYTES = (int64_t)24 << 20;

struct SkinnyPlan {
  bool take;   // false: a tile kernel is the better one (the rest is not set)
  int mb;      // blocks of 16 rows of a workgroup: 1, 2 or 4
  int blocks;  // workgroups along M: 1 up to 64 rows
  int cols;    // output columns of a workgroup's strip
  int strips;
  int splits;  // workgroups along K
  bool part;   // workgroups of 4 waves on wide strips (else whole K, narrow strips, no partials)
  bool dual_parts;  // part of a dual product: gate and up on workgroups of their own, whose
                    // partials the reduction gates
};

// Plan for C[M, N] = A[M, K] op(B) on a chip of `cus` compute units.  ws_elems: fp32 partials
// the workspace holds.
SkinnyPlan skinny_plan(bool bf16, bool transB, bool dual, int64_t M, int64_t N, int64_t K, int64_t ws_elems,
                       int cus);

// p as for the GEMM kernels (op(A) not transposed, one problem, one K segment, no causal
// structure, p.splits set to the plan's); dual: p.B2 holds the second B of the SiLU gate.
hipError_t launch_skinny(const Params& p, const SkinnyPlan& pl, bool bf16, bool transB, bool dual,
                         hipStream_t stream);

}  // namespace mig
