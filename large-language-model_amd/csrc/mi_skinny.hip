// mi_skinny.hip -- GEMM of a few rows (token generation, short batches): C[M, N] with
// M <= 64 and op(A) not transposed, bf16 or fp32, optionally with the dual-B SiLU gate; and
// small fp32 products in blocks of 64 rows (mi_skinny.hpp).
//
// Bound: the weights B are read once from HBM and everything else is small, so a call
// takes the time of streaming K x N elements plus a memory latency per launch.  What that
// rate depends on, measured with a kernel that only reads B (2048 x 2048 bf16, cold): a CU
// draws 20 to 45 GB/s however many loads it has in flight, so all CUs must read, and rows
// must be read in long pieces: 64 workgroups on 64-byte pieces of every row 8.4 us, 256
// workgroups on the same 4.6, 256 workgroups on 256-byte pieces 3.2 (5632 x 2048: 20.0, 8.2
// and 6.1 us, 3.8 TB/s).  Hence:
//   * a workgroup of 4 waves owns a strip of 128 columns (64 of fp32) and a part of K;
//     each wave a part of that part.  The waves' sums meet in LDS, the workgroups' as fp32
//     partials in the workspace, added in order by a second kernel (deterministic);
//   * where the second launch would cost more than the longer pieces save, and without a
//     workspace, a workgroup of up to 16 waves takes the whole of K on a strip of 32
//     columns (16 rows of a K-contiguous B): skinny_plan weighs the two;
//   * operands go from memory straight to MFMA registers: a lane loads 16 bytes (8
//     columns of bf16) of each of the 8 k rows that one 16x16x32 MFMA wants of it, and byte
//     permutes turn them into the operands of 8 MFMAs, one per column; neither LDS nor a
//     barrier is on the way.  fp32 takes 4 columns of 4 k rows and feeds them as they are;
//   * an operand that is K-contiguous in memory (A, and B of the NT form) is loaded with
//     four neighbouring lanes on the 64 bytes that a step takes of a row, and moved to the
//     MFMA's lanes (row = lane mod 16) through the LDS crossbar: loaded in the MFMA's lane
//     order, neighbouring lanes would touch different rows and the address unit would
//     take 64 cycles a load instead of 16;
//   * B is the first MFMA operand, so a lane ends up with consecutive columns of one row.
// Strips next to each other go to the same XCD, whose L2 then holds the lines they share.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "mi_skinny.hpp"

namespace mig {
namespace {

// A 16-row x 64-byte block loaded by lane as (row lane / 4, chunk lane mod 4), to the MFMA's
// (row lane mod 16, chunk lane / 16).
__device__ __forceinline__ u32x4_t to_mfma_lanes(u32x4_t v) {
  const int src = ((threadIdx.x & 15) * 4 + ((threadIdx.x & 63) >> 4)) * 4;
  u32x4_t o;
#pragma unroll
  for (int q = 0; q < 4; ++q) o[q] = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)v[q]);
  return o;
}

template <int DW>
struct Words {  // DW dwords of one lane's load
  uint32_t w[DW];
};
template <int DW>
__device__ __forceinline__ Words<DW> buf_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  Words<DW> o;
  if constexpr (DW == 4) {
    const u32x4_t v = buf_load16(r, off);
#pragma unroll
    for (int i = 0; i < 4; ++i) o.w[i] = v[i];
  } else if constexpr (DW == 2) {
    const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0);
    o.w[0] = v[0];
    o.w[1] = v[1];
  } else {
    o.w[0] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
  }
  return o;
}

// Waves of a workgroup that takes the whole of K (as many as the LDS sums allow), and of one
// that takes a part.
constexpr int whole_waves(int mb, int nd) { return mb * nd <= 2 ? 16 : 8; }
constexpr int PART_WAVES = 4;

// Dwords of B that a lane loads of one k row (row-contiguous B), or 16-row groups of a strip
// (K-contiguous B).  K parts: 16 bytes, or half as many where the accumulators are many.
constexpr int lane_dwords(bool part, bool bkc, int es, int mb) {
  return part ? (mb >= 4 ? 2 : 4) : (bkc || es == 2 ? 1 : 2);
}

// MB: blocks of 16 rows; ND: B matrices of a workgroup (2: both of a dual product, PART
// false only); PART: the workgroup takes a part of K, as do the waves of one that does not.
template <typename T, bool BKC, int MB, int ND, bool PART>
__global__ void __launch_bounds__(64 * (PART ? PART_WAVES : whole_waves(MB, ND)))
    skinny_kernel(Params p, int dual_parts) {
  constexpr int NW = PART ? PART_WAVES : whole_waves(MB, ND);
  constexpr int ES = (int)sizeof(T);
  constexpr int KL = 16 / ES;                    // k of one lane per step
  constexpr int SK = 4 * KL;                     // k of a step
  constexpr int DW = lane_dwords(PART, BKC, ES, MB);
  constexpr int CB = BKC ? DW : DW * 4 / ES;     // 16-column accumulators of a strip
  constexpr int STRIP = 16 * CB, PITCH = STRIP + 4;
  constexpr int U = MB * ND >= 4 ? 1 : PART || ND * MB == 2 ? 2 : 4;  // steps whose loads go out together
  __shared__ __attribute__((aligned(16))) float red[NW][ND][MB * 16][PITCH];

  const int lane = threadIdx.x & 63, wave = uniform((int)threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;    // MFMA lanes
  const int cr = lane >> 2, gr = lane & 3;   // lanes of a K-contiguous load
  // work item: strips innermost, then the matrix of a dual product, then the K part; the
  // items of one XCD (block id mod 8) are consecutive
  const int nb = gridDim.x, x = blockIdx.x & 7, q8 = nb >> 3, r8 = nb & 7;
  const int item = x * q8 + (x < r8 ? x : r8) + ((int)blockIdx.x >> 3);
  const int strips = (p.N + STRIP - 1) / STRIP;
  const int strip = uniform(item % strips), rest = uniform(item / strips);
  const int parts = dual_parts ? 2 : 1;
  const int which = uniform(rest % parts), outer = uniform(rest / parts);
  // the K part, or of an unsplit product the block of rows
  const int split = PART ? outer : 0, m0 = PART ? 0 : outer * (16 * MB);
  const int n0 = strip * STRIP;

  const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.A, p.extA);
  const __amdgpu_buffer_rsrc_t rb1 = make_rsrc(which ? p.B2 : p.B, p.extB);
  __amdgpu_buffer_rsrc_t rb2 = rb1;
  if constexpr (ND == 2) rb2 = make_rsrc(p.B2, p.extB);
  const int lda = (int)p.lda * ES, ldb = (int)p.ldb * ES;
  // byte offsets at k = 0; rows of A past M lie past its extent
  uint32_t ao[MB], bo[BKC ? CB : 1];
#pragma unroll
  for (int i = 0; i < MB; ++i) ao[i] = (uint32_t)((m0 + 16 * i + cr) * lda + gr * 16);
  if constexpr (BKC) {
#pragma unroll
    for (int j = 0; j < CB; ++j)
      bo[j] = n0 + 16 * j + cr < p.N ? (uint32_t)((n0 + 16 * j + cr) * ldb + gr * 16) : kBufOOB;
  } else {
    // the columns past N of a lane that straddles it are not stored
    bo[0] = n0 + CB * c < p.N ? (uint32_t)((n0 + CB * c) * ES + g * KL * ldb) : kBufOOB;
  }

  f32x4_t acc[ND][MB][CB];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) acc[d][i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  struct Step {
    u32x4_t a[MB];
    u32x4_t bk[BKC ? ND : 1][BKC ? CB : 1];   // K-contiguous B: 16 bytes of each group's row
    Words<DW> br[BKC ? 1 : ND][BKC ? 1 : KL];  // row-contiguous B: columns of the lane's k rows
  };
  auto load = [&](Step& s, int step) __attribute__((always_inline)) {
    const int k0 = step * SK;
    // a lane whose k lie past K reads zeros from both operands (K is whole 16-byte chunks)
    const bool in = k0 + g * KL < p.K, inr = k0 + gr * KL < p.K;
#pragma unroll
    for (int i = 0; i < MB; ++i) s.a[i] = buf_load16(ra, inr ? ao[i] + (uint32_t)(k0 * ES) : kBufOOB);
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      const __amdgpu_buffer_rsrc_t r = d ? rb2 : rb1;
      if constexpr (BKC) {
#pragma unroll
        for (int j = 0; j < CB; ++j) s.bk[d][j] = buf_load16(r, inr ? bo[j] + (uint32_t)(k0 * ES) : kBufOOB);
      } else {
        const uint32_t b = in ? bo[0] + (uint32_t)(k0 * ldb) : kBufOOB;
#pragma unroll
        for (int e = 0; e < KL; ++e) s.br[d][e] = buf_load<DW>(r, b + (uint32_t)(e * ldb));
      }
    }
  };
  auto compute = [&](const Step& s) __attribute__((always_inline)) {
    u32x4_t a[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) a[i] = to_mfma_lanes(s.a[i]);
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        u32x4_t w;  // the lane's KL values of k for column group j
        if constexpr (BKC) {
          w = to_mfma_lanes(s.bk[d][j]);
        } else if constexpr (ES == 2) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            w[q] = __builtin_amdgcn_perm(s.br[d][2 * q + 1].w[j / 2], s.br[d][2 * q].w[j / 2],
                                         (j & 1) ? 0x07060302u : 0x05040100u);
        } else {
#pragma unroll
          for (int t = 0; t < 4; ++t) w[t] = s.br[d][t].w[j];
        }
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          if constexpr (ES == 2) {
            acc[d][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, a[i]), acc[d][i][j], 0, 0, 0);
          } else {
#pragma unroll
            for (int t = 0; t < 4; ++t)  // value t of both operands is k = 4g + t
              acc[d][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w[t]), __uint_as_float(a[i][t]),
                                                                  acc[d][i][j], 0, 0, 0);
          }
        }
      }
  };

  // this wave's steps: its part of the workgroup's part of K, consecutive
  const int steps = (p.K + SK - 1) / SK;
  const int share = p.splits * NW, mine = split * NW + wave;
  int s = uniform((int)((int64_t)steps * mine / share));
  const int s_end = uniform((int)((int64_t)steps * (mine + 1) / share));
  for (; s + U <= s_end; s += U) {
    Step st[U];
#pragma unroll
    for (int u = 0; u < U; ++u) load(st[u], s + u);
#pragma unroll
    for (int u = 0; u < U; ++u) compute(st[u]);
  }
  for (; U > 1 && s < s_end; ++s) {
    Step st;
    load(st, s);
    compute(st);
  }

  // acc[d][i][j][e]: row m0 + 16i + c, column n0 + CB * (4g + e) + j (K-contiguous B: 16j + 4g + e)
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      float* dst = &red[wave][d][16 * i + c][0];
#pragma unroll
      for (int h = 0; h < CB; ++h) {
        if constexpr (BKC) {
          *reinterpret_cast<f32x4_t*>(dst + 16 * h + 4 * g) = acc[d][i][h];
        } else {
          f32x4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[d][i][(4 * h + e) % CB][(4 * h + e) / CB];
          *reinterpret_cast<f32x4_t*>(dst + 4 * CB * g + 4 * h) = v;
        }
      }
    }
  __syncthreads();
  constexpr int QPR = STRIP / 4;  // 4-column groups per row
  const int rows = p.M - m0 < MB * 16 ? p.M - m0 : MB * 16;
  const bool partial = p.splits > 1 || dual_parts;
  for (int t = threadIdx.x; t < rows * QPR; t += 64 * NW) {
    const int m = t / QPR, nq = (t - m * QPR) * 4, n = n0 + nq;
    f32x4_t sum[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      sum[d] = *reinterpret_cast<const f32x4_t*>(&red[0][d][m][nq]);
#pragma unroll
      for (int w = 1; w < NW; ++w) sum[d] += *reinterpret_cast<const f32x4_t*>(&red[w][d][m][nq]);
    }
    if (partial) {
      float* W = p.ws + ((int64_t)(split * parts + which) * p.M + m) * p.N + n;
      if ((p.N & 3) == 0 && n + 3 < p.N) {
        *reinterpret_cast<f32x4_t*>(W) = sum[0];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < p.N) W[e] = sum[0][e];
      }
      continue;
    }
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = ND == 2 ? silu_f(p.alpha * sum[0][e]) * (p.alpha * sum[ND - 1][e]) : p.alpha * sum[0][e];
    epilogue4(p, p.C, p.R, m0 + m, n, v);
  }
}

// C = epilogue(alpha * sum of the K parts), in order; PARTS = 2: SiLU(gate) * up.  Bound by
// one trip to the partials, so all loads of 16 parts are issued before their sum, on
// single-wave workgroups that reach every CU.
template <int PARTS>
__global__ void __launch_bounds__(64) skinny_reduce_kernel(Params p) {
  const int qpr = (p.N + 3) / 4;
  const int t = blockIdx.x * 64 + threadIdx.x;
  if (t >= p.M * qpr) return;
  const int m = t / qpr, n = (t - m * qpr) * 4;
  const int64_t slab = (int64_t)p.M * p.N;
  const float* W = p.ws + (int64_t)m * p.N + n;
  const bool vec = (p.N & 3) == 0;
  f32x4_t sum[PARTS];
#pragma unroll
  for (int d = 0; d < PARTS; ++d) sum[d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  constexpr int FLY = 16 / PARTS;
  for (int s = 0; s < p.splits; s += FLY) {
    f32x4_t v[FLY][PARTS];
#pragma unroll
    for (int u = 0; u < FLY; ++u)
#pragma unroll
      for (int d = 0; d < PARTS; ++d) {
        v[u][d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (s + u < p.splits) {
          const float* w = W + (int64_t)((s + u) * PARTS + d) * slab;
          if (vec) {
            v[u][d] = *reinterpret_cast<const f32x4_t*>(w);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e < p.N) v[u][d][e] = w[e];
          }
        }
      }
#pragma unroll
    for (int u = 0; u < FLY; ++u)
#pragma unroll
      for (int d = 0; d < PARTS; ++d) sum[d] += v[u][d];
  }
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    v[e] = PARTS == 2 ? silu_f(p.alpha * sum[0][e]) * (p.alpha * sum[PARTS - 1][e]) : p.alpha * sum[0][e];
  epilogue4(p, p.C, p.R, m, n, v);
}

template <typename T, bool BKC, int MB, int ND, bool PART>
void launch_one(const Params& p, const SkinnyPlan& pl, hipStream_t st) {
  const dim3 grid((unsigned)(pl.strips * pl.splits * pl.blocks * (pl.dual_parts ? 2 : 1)));
  const dim3 block((unsigned)(64 * (PART ? PART_WAVES : whole_waves(MB, ND))));
  hipLaunchKernelGGL((skinny_kernel<T, BKC, MB, ND, PART>), grid, block, 0, st, p, (int)pl.dual_parts);
}

template <typename T, bool BKC>
void launch_rows(const Params& p, const SkinnyPlan& pl, bool both, hipStream_t st) {
  auto go = [&](auto mb_c) {
    constexpr int MB = decltype(mb_c)::value;
    if (pl.part) launch_one<T, BKC, MB, 1, true>(p, pl, st);
    else if (both) launch_one<T, BKC, MB, 2, false>(p, pl, st);
    else launch_one<T, BKC, MB, 1, false>(p, pl, st);
  };
  if (pl.mb == 1) go(std::integral_constant<int, 1>{});
  else if (pl.mb == 2) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 4>{});
}

}  // namespace

SkinnyPlan skinny_plan(bool bf16, bool transB, bool dual, int64_t M, int64_t N, int64_t K, int64_t ws_elems,
                       int cus) {
  SkinnyPlan pl{};
  const int64_t es = bf16 ? 2 : 4, nd = dual ? 2 : 1;
  pl.blocks = (int)((M + 63) / 64);
  if (M > SKINNY_MAX_M) {
    const int64_t blocks = pl.blocks * ((N + 31) / 32);
    if (bf16 || transB || dual || K > 1024 || 2 * blocks < cus || blocks > cus) return pl;
  } else if (M > 32 && N * K * es > SKINNY_WIDE_BYTES) {
    return pl;
  }
  pl.mb = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  const int64_t steps = std::max<int64_t>(1, (K * es + 63) / 64);
  auto cols_of = [&](bool part) {
    const int dw = lane_dwords(part, transB, (int)es, pl.mb);
    return 16 * (transB ? dw : dw * 4 / (int)es);
  };
  auto strips_of = [&](bool part) { return (N + cols_of(part) - 1) / cols_of(part); };
  // K parts: up to two workgroups a CU, each wave at least one step, and the partials (written
  // and read back) at most half the bytes of B
  const int64_t groups = strips_of(true) * nd;
  const int64_t sp = std::min<int64_t>({2 * cus / groups, steps / PART_WAVES, K * es / (16 * M),
                                        ws_elems / std::max<int64_t>(1, nd * M * N), 64});
  // Time of either form in us, fitted to the rates above, to 4758 products with B cold and to whole
  // decoder layers, whose weights the last-level cache holds: a whole-K workgroup takes 1 us
  // and 24 GB/s of its strip and half of A (which the L2 holds), at most 2.3 TB/s over the
  // chip; K parts run at 3.5 TB/s from 5 workgroups on 8 CUs on, and their second launch takes
  // 4.5 us (cold products prefer 6.5, by 1 %: 16 x 768 x 768 fp32 parts 6.3 us, whole 5.9; a
  // layer of 8 rows, all whole / all parts / by this rule: width 2048 68.5 / 56.7 / 57.0 us,
  // with 6.5 59.7; width 768 all whole 36.0, all parts 41.6).
  const double bytes = (double)(nd * N * K * es);
  const double whole = (double)((nd * cols_of(false) + 8 * pl.mb) * K * es);
  const double t_whole = 1.0 + std::max(whole / 24e3 * (double)((strips_of(false) + cus - 1) / cus), bytes / 2.3e6);
  const double t_part = bytes / 3.5e6 * std::max(1.0, 0.625 * cus / (double)(groups * std::max<int64_t>(sp, 1))) +
                        (sp > 1 || dual ? 4.5 + 8.0 * (double)(sp * nd * M * N) / 3.5e6 : 0.0);
  pl.part = sp >= 1 && t_part < t_whole && pl.blocks == 1;
  pl.splits = pl.part ? (int)sp : 1;
  pl.dual_parts = pl.part && dual;
  pl.cols = cols_of(pl.part);
  pl.strips = (int)strips_of(pl.part);
  // Strips past two or three to a CU are short work for a workgroup each, and 128-row tiles
  // leave no CU idle either.  Where whole-K workgroups then have the lower time, by bytes of a
  // row of K, skinny over tile with B in the caches and cold: M <= 16 NN bf16 1.31 / 1.39 at
  // 256, 0.96 / 1.07 at 2048, fp32 1.19 / - at 256, 0.79 / 0.77 at 1024; NT past 4 strips a CU
  // bf16 1.37 / 1.14 at 1024, 0.94 / 0.80 at 4096, fp32 1.11 at 1024, 0.90 / 0.98 at 2048;
  // M <= 32 NN 1.0 / 1.2 at 256, 0.8 / 1.0 at 1024, 1.03 / 1.2 at 8192 (fp32 0.72 / 0.94), NT
  // past 4 strips 1.4 at 512, 1.0 / 1.35 at 2048; M <= 64 NT bf16 0.85 / 0.96 at 512, 0.8 / 0.93
  // to 4 strips at 1024, else past 1.1 (2 x 32000 x 112 bf16 NT 11.5 us, tile 6.6; 26 x 32000 x
  // 2424 fp32 NT 119 and 84; 20 x 32000 x 768 fp32 NN 20.6 and 27.5).
  const int64_t row = K * es, s = pl.strips, big = (int64_t)1 << 40;
  auto within = [&](int64_t lo, int64_t hi) { return lo <= row && row <= hi; };
  if (pl.part || M > SKINNY_MAX_M) pl.take = true;
  else if (M > 32)
    pl.take = s <= (dual && !transB ? cus : 2 * cus) ||
              (bf16 && transB && !dual && within(0, s <= 4 * cus ? 1024 : 512));
  else if (s <= 3 * cus) pl.take = true;
  else if (transB && s > 4 * cus) pl.take = M <= 16 && !(bf16 && dual) && within(bf16 ? 4096 : 1536, big);
  else if (transB) pl.take = within(768, big);
  else if (bf16) pl.take = M <= 16 ? !dual && within(2048, big) : within(512, 4096);
  else pl.take = within(512, M <= 16 ? big : 8192);
  return pl;
}

hipError_t launch_skinny(const Params& p, const SkinnyPlan& pl, bool bf16, bool transB, bool dual,
                         hipStream_t stream) {
  const bool both = dual && !pl.part;
  if (bf16)
    transB ? launch_rows<__bf16, true>(p, pl, both, stream) : launch_rows<__bf16, false>(p, pl, both, stream);
  else
    transB ? launch_rows<float, true>(p, pl, both, stream) : launch_rows<float, false>(p, pl, both, stream);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || (pl.splits == 1 && !pl.dual_parts)) return e;
  const dim3 grid((unsigned)((p.M * ((p.N + 3) / 4) + 63) / 64));
  if (pl.dual_parts)
    hipLaunchKernelGGL((skinny_reduce_kernel<2>), grid, dim3(64), 0, stream, p);
  else
    hipLaunchKernelGGL((skinny_reduce_kernel<1>), grid, dim3(64), 0, stream, p);
  return hipGetLastError();
}

}  // namespace mig
