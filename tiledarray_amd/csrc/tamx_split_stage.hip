// Grouped split GEMM on 64 x 64 macro tiles, chunks multiplied out of
// registers (the default for BF16 and INT8 limbs).
//
// Per tile pair the limb products s + t < S run on the 16-row MFMA (BF16
// 16x16x32, INT8 16x16x64) into one accumulator per level (BF16: P_0, P_1
// and P_T), folded into FP64 at pair ends and every FOLD chunks; the folds
// and the order of the sums are those of the other split kernels, so the
// results are the same bit for bit.
//
// What bounds it: the matrix cores reach 4.75 INT8 POP/s on 16x16x64 in a
// register-only loop, and 60 of these MFMAs a wave and chunk (five limbs) are
// no longer than what surrounds them: 40 KB of limbs to land in LDS (about 30
// TB/s out of L2 over the card, 7.5 from beyond it), 20 fragment reads, the
// fold, and waiting for the slowest wave.  So
//  - a wave reads all fragments of a chunk into registers and multiplies
//    while the last ones arrive; a second barrier after the first S products
//    frees the stage, and the loads of the chunk after next go out between
//    the other products.  Almost two chunks are in flight at all times out of
//    two stages, and neither reads nor loads hold up the MFMAs;
//  - the loads are 16-byte buffer_load ... lds with an offset per thread that
//    is fixed for a pair; rows past the tile's padded rows and the second half
//    of a chunk that holds only k padding carry an offset outside the
//    descriptor and fetch nothing;
//  - the 16 x 16 blocks of a macro tile go to the waves in turn along each
//    direction, so a ragged edge leaves them nearly equal work;
//  - pair descriptors come 64 at a time, one per lane;
//  - the first MFMAs after a fold start from a zero operand, and INT8 levels
//    are joined as integers, so a fold is seven instructions per result.
// Against the kernel with one chunk in flight and fragments read between the
// MFMAs (GEMM alone): block-sparse 16384^3 in five INT8 limbs 1.90 -> 1.62 ms,
// 8192^3 in three BF16 limbs 955 -> 720 us, ladder at 20 x 150 in four INT8
// limbs 2.65 -> 2.33 ms.
#include <type_traits>

#include "tamx_internal.hpp"
#include "tamx_split.hpp"

namespace {

using namespace tamx::split;

constexpr int kTile = 64;              // macro tile rows and columns
constexpr int kPlaneUnits = kTile * 4;  // 16-byte units of one plane of a chunk
constexpr int kBandRows = 8;  // macro tiles are taken column by column in bands of these rows
// buffer descriptor word 3 (raw 32-bit format) and an offset outside every range
[[maybe_unused]] constexpr int kBufFlags = 0x00020000;
constexpr uint32_t kOutside = 0x80000000u;

// vmcnt(n), the other counters left alone (gfx9 encoding)
constexpr int wait_vm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

template <int N>
using ic = std::integral_constant<int, N>;

// The fold of INT8 levels joins up to five of them as a 64-bit integer,
// x = sum lvl[g] 2^(7 (n - 1 - g)), on top of the bits of 1.5 * 2^52: while
// |x| < 2^51 the sum is the bits of the double 1.5 * 2^52 + x, so one
// subtraction gives x exactly.  With |l_0| <= 127 and |l_s| <= 64 that holds
// up to 448 k; after more than that the levels are converted one by one.
// (Both are exact, so the results do not depend on it.  Converting, scaling
// and adding the levels one by one and clearing them afterwards took 24% of
// the kernel on block-sparse 16384^3 in five limbs, where a pair has three
// chunks on average.)
constexpr int kJoinChunks = 7;
constexpr double kJoin = 6755399441055744.0;  // 1.5 * 2^52
constexpr int64_t kJoinBits = 0x4338000000000000;

// kJoinBits + a, and x + a * b, one v_mad_i64_i32 each: a factor the compiler
// cannot see through keeps it from shifting and adding instead.  (The
// instruction is the compiler's, not inline asm: a vector instruction has to
// keep its distance from the MFMA whose result it reads, which the hardware
// does not check and the compiler sees to for its own instructions only.)
__device__ __forceinline__ int64_t join_next(int a, int b, int64_t x) {
#ifdef __HIP_DEVICE_COMPILE__
  asm("" : "+s"(b));
#endif
  return x + (int64_t)a * b;
}
__device__ __forceinline__ int64_t join_first(int a) { return join_next(a, 1, kJoinBits); }

// The LDS unit of a plane that holds unit q of row r.  BF16: lds_unit.  INT8:
// the 32-k blocks of the limb layout one after the other: each group of four lanes then loads 64 consecutive
// bytes, which the vector cache serves in one step (with four units a row,
// two of each block, every group touched two cache lines, and the loads
// alone took 1.51 of 1.76 ms on block-sparse 16384^3 in five limbs).  A
// fragment read takes sixteen lanes at a time, rows 0-3 and 12-15 of one unit
// with rows 4-11 of the next, which fall in distinct banks in both layouts.
template <bool I8>
__device__ inline int stage_unit(int r, int q) {
  if constexpr (I8) return (q >> 1) * (2 * kTile) + 2 * r + (q & 1);
  return lds_unit(r, q);
}

// workgroups per CU: two stages of 8 S KB each
constexpr int staged_occupancy(int s) { return s <= 2 ? 4 : (s == 3 ? 3 : (s <= 5 ? 2 : 1)); }

template <int S, bool I8>
__global__ __launch_bounds__(kThreads, staged_occupancy(S)) void split_gemm_staged_kernel(
    SplitParams p) {
  constexpr int NG = I8 ? S : (S >= 3 ? 3 : S);  // accumulators per block
  constexpr int CK = I8 ? SBK8 : SBK;            // k per chunk
  constexpr int FOLD = I8 ? kFoldChunks8 : kFoldChunks;
  constexpr int EB = I8 ? 1 : 2;                 // bytes per limb
  constexpr int NEXT = I8 ? 64 : 128;            // units from a wave's block to its next
  using lvl_t = std::conditional_t<I8, i4_t, f4_t>;
  // one variable per stage: the compiler then knows that loads landing in
  // one stage do not alias reads of the other
  __shared__ bf8_t stage0[2][S][kPlaneUnits];
  __shared__ bf8_t stage1[2][S][kPlaneUnits];
  // the grabbed item passes through the first word of stage 0 while the
  // stages are idle between items
  int* s_item = reinterpret_cast<int*>(&stage0[0][0][0]);
  auto stage = [&](auto X) -> bf8_t(&)[2][S][kPlaneUnits] {
    if constexpr (decltype(X)::value == 0) return stage0; else return stage1;
  };

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = uni(tid >> 6);
  const int lrow = lane & 15, lq = lane >> 4;  // MFMA: row lrow, k unit lq
  const int wr = (wave >> 1) * 16, wc = (wave & 1) * 16;  // the wave's first block
  // staging: thread tid writes LDS unit tid of every plane, which holds unit
  // st_q of row st_r
  const int st_r = I8 ? (tid >> 1) & (kTile - 1) : tid >> 2;
  const int st_q = I8 ? (tid >> 7) * 2 + (tid & 1) : (tid & 3) ^ ((st_r >> 1) & 3);
  const int fa = stage_unit<I8>(wr + lrow, lq), fb = stage_unit<I8>(wc + lrow, lq);

  int64_t ntasks64 = p.counters[TAMX_WL_NTASKS];
  if (ntasks64 < 0 || ntasks64 > p.task_capacity || p.counters[TAMX_WL_STATUS] != 0)
    ntasks64 = 0;
  const int32_t ntasks = uni((int32_t)ntasks64);
  const int32_t total = uni(p.prefix[ntasks > 0 ? ntasks : 0]);
  tamx::ItemQueue queue(p.queue, total);  // used by thread 0 only
  auto barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  // The parameters are read again where they are used, rather than kept in
  // scalar registers across the main loop.
  auto args = [&]() {
#ifdef __HIP_DEVICE_COMPILE__
    const auto* q = (const __attribute__((address_space(4))) SplitParams*)
        __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(q));
    return q;
#else
    return &p;
#endif
  };
  for (;;) {
    if (tid == 0) *s_item = queue.next();
    __syncthreads();
    const int item = uni(*s_item);
    __syncthreads();
    if (item < 0) break;
    int lo;
    if (total <= args()->item_capacity) {
      lo = uni(tamx::scalar_ptr(args()->item_task)[item]);
    } else {
      lo = 0;
      int hi = ntasks - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (uni(args()->prefix[mid]) <= item) lo = mid; else hi = mid - 1;
      }
    }
    const auto* tp = tamx::scalar_ptr(args()->tasks) + lo;
    const int t_m = uni(tp->m), t_n = uni(tp->n);
    int lp = uni(tp->pair_begin);
    const int pend = lp + uni(tp->pair_count);
    const int local = item - uni(tamx::scalar_ptr(args()->prefix)[lo]);
    const int tiles_n = (t_n + kTile - 1) / kTile, tiles_m = (t_m + kTile - 1) / kTile;
    const int band = local / (kBandRows * tiles_n), in_band = local - band * kBandRows * tiles_n;
    const int band_rows = min(kBandRows, tiles_m - band * kBandRows);
    const int r0 = uni(band * kBandRows + in_band % band_rows) * kTile;
    const int c0 = uni(in_band / band_rows) * kTile;
    const int mrem = min(kTile, t_m - r0), nrem = min(kTile, t_n - c0);
    // the wave's 16-row (column) blocks inside the tile
    const int ni = uni(min(2, max(0, (mrem - wr + 31) >> 5)));
    const int nj = uni(min(2, max(0, (nrem - wc + 31) >> 5)));

    // The descriptors of 64 pairs from pair `tb` on, one pair per lane: limb
    // addresses of the macro tile's first row (column) in plane 0, padded rows,
    // contracted extent and scale exponent.  (Read pair by pair through the
    // scalar unit, every pair waited for three dependent loads: block-sparse
    // 16384^3 in five INT8 limbs, 11% of the kernel.)
    int tb = lp;
    int64_t t_a = 0, t_b = 0;
    int t_arows = 0, t_brows = 0, t_k = 0, t_exp = 0;
    auto fill_table = [&](int first) {
      tb = first;
      const auto* pr = tamx::global_ptr(args()->pairs) + min(first + lane, pend - 1);
      const auto* A = tamx::global_ptr(args()->ta) + pr->a_tile;
      const auto* B = tamx::global_ptr(args()->tb) + pr->b_tile;
      const int step = I8 ? kI8Block : A->k_pad * EB;  // bytes from a row to the next
      t_a = (int64_t)args()->LA + A->limb_off * EB + (int64_t)r0 * step;
      t_b = (int64_t)args()->LB + B->limb_off * EB + (int64_t)c0 * step;
      t_arows = A->rows_pad;
      t_brows = B->rows_pad;
      t_k = A->out_k;
      t_exp = A->sigma + B->sigma - (I8 ? 14 : 16);
      // (used here, so that no wait for these loads is left to the main loop)
      asm volatile("" : "+v"(t_a), "+v"(t_b), "+v"(t_arows), "+v"(t_brows), "+v"(t_k), "+v"(t_exp));
    };
    auto lane_of = [&](int x, int l) { return __builtin_amdgcn_readlane(x, l); };
    auto lane_of64 = [&](int64_t x, int l) {
      const uint32_t u = lane_of((int)x, l), v = lane_of((int)(x >> 32), l);
      return (int64_t)(((uint64_t)v << 32) | u);
    };

    // Load cursor: pair lp, chunk at k lk0.  next_chunk() sets what the 2 S
    // loads of the cursor's chunk need and moves the cursor on; past the last
    // pair every load lies outside and writes zeros nobody reads, so every
    // step issues the same loads and the wait counts are exact.
    int lk0 = 0, out_k = 0, a_rows = 0, b_rows = 0, expo = 0;
    [[maybe_unused]] int64_t a_base = 0, b_base = 0;
    uint32_t a_vo = kOutside, b_vo = kOutside;
    [[maybe_unused]] uint32_t va = kOutside, vb = kOutside;
    // (unsigned: past a chunk's last plane they may reach 2^31)
    [[maybe_unused]] uint32_t a_so = 0, b_so = 0, a_plane = 0, b_plane = 0;
    // per stage: whether it holds a chunk, whether that ends a pair, and the
    // pair's scale exponent
    bool valid0 = false, valid1 = false;
    bool ends0 = false, ends1 = false;
    int exp0 = 0, exp1 = 0;
    auto next_chunk = [&](auto X) {
      const bool valid = lp < pend;
      if constexpr (decltype(X)::value == 0) valid0 = valid; else valid1 = valid;
      if (!valid) {
        va = vb = kOutside;
        // (the range check takes the scalar offset from the descriptor's
        // size: left where the last chunk's loads ended, plane by plane
        // beyond the tile, it passes 2^31 for tiles with 0.7 GB of limbs)
        a_so = b_so = 0;
        if (tid == 0) queue.prefetch();
        return;
      }
      if (lk0 == 0) {
        if (lp - tb == 64) fill_table(lp);
        const int l = lp - tb;
        a_base = lane_of64(t_a, l);
        b_base = lane_of64(t_b, l);
        a_rows = lane_of(t_arows, l);
        b_rows = lane_of(t_brows, l);
        out_k = lane_of(t_k, l);
        expo = lane_of(t_exp, l);
        const int k_pad = max(CK, (out_k + CK - 1) / CK * CK);
        a_plane = a_rows * k_pad * EB;
        b_plane = b_rows * k_pad * EB;
        auto offset = [&](int rows, int first) -> uint32_t {
          const uint32_t o = I8 ? (uint32_t)((st_q >> 1) * (rows * kI8Block) + st_r * kI8Block +
                                             (st_q & 1) * 16)
                                : (uint32_t)(st_r * (k_pad * EB) + st_q * 16);
          return first + st_r < rows ? o : kOutside;
        };
        a_vo = offset(a_rows, r0);
        b_vo = offset(b_rows, c0);
      }
      a_so = I8 ? lk0 * a_rows : lk0 * EB;  // (INT8: 32 bytes a row and 32 k)
      b_so = I8 ? lk0 * b_rows : lk0 * EB;
      const bool half = I8 && out_k - lk0 <= kI8Block && st_q >= 2;
      va = half ? kOutside : a_vo;
      vb = half ? kOutside : b_vo;
      lk0 += CK;
      const bool ends = lk0 >= out_k;
      if constexpr (decltype(X)::value == 0) { ends0 = ends; exp0 = expo; }
      else { ends1 = ends; exp1 = expo; }
      if (ends) {
        ++lp;
        lk0 = 0;
      }
    };
    // load e (of 2 S) of the chunk next_chunk() has set, into stage X
    auto load = [&]([[maybe_unused]] auto X, [[maybe_unused]] int e) {
#ifdef __HIP_DEVICE_COMPILE__  // (the host pass does not accept the LDS load builtin)
      const bool is_a = e < S;
      const int s = is_a ? e : e - S;
      const auto d = __builtin_amdgcn_make_buffer_rsrc((void*)(is_a ? a_base : b_base), (short)0,
                                                       (int)(kOutside - 1), kBufFlags);
      int w = wave;
      asm volatile("" : "+s"(w));  // (else the 4 S destinations stay in registers)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          d, (__attribute__((address_space(3))) void*)(&stage(X)[is_a ? 0 : 1][s][w * 64]), 16,
          is_a ? va : vb, is_a ? a_so : b_so, 0, 0);
      if (is_a) a_so += a_plane;
      else b_so += b_plane;
#endif
    };

    const bool have = lp < pend;
    // The item with NI x NJ blocks in this wave (the waves of a workgroup may
    // differ; all pass the same barriers and issue the same loads).
    auto run_item = [&](auto NI_, auto NJ_) {
      constexpr int NI = decltype(NI_)::value, NJ = decltype(NJ_)::value;
      constexpr bool ACTIVE = NI > 0 && NJ > 0;
      constexpr int AI = ACTIVE ? NI : 1, AJ = ACTIVE ? NJ : 1;
      d4_t acc[AI][AJ];
      lvl_t lvl[NG][AI][AJ];
#pragma unroll
      for (int i = 0; i < AI; ++i)
#pragma unroll
        for (int j = 0; j < AJ; ++j) acc[i][j] = d4_t{0.0, 0.0, 0.0, 0.0};
      int since_fold = 0;

      // The products of a chunk.  After the first MID of them every fragment
      // has been read: a barrier frees the stage, and the loads of the chunk
      // after next go out between the others.
      constexpr int NP = S * (S + 1) / 2, MID = S + (S > 3 ? 1 : 0) - 1;
      auto products = [&](auto X, const bf8_t (&af)[S][AI], const bf8_t (&bf)[S][AJ], auto FIRST) {
        int n = 0, e = 0;
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
          for (int t = 0; t < S - s; ++t) {
            const int g = I8 ? s + t : (s + t < 2 ? s + t : 2);
            // the first product of its level (of P_T: of level 2) in this order
            const bool zero = decltype(FIRST)::value && s == 0 && (I8 || t < 3);
            if constexpr (ACTIVE) {
#pragma unroll
              for (int i = 0; i < AI; ++i)
#pragma unroll
                for (int j = 0; j < AJ; ++j) {
                  const lvl_t c = zero ? lvl_t{0, 0, 0, 0} : lvl[g][i][j];
                  if constexpr (I8)
                    lvl[g][i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                        __builtin_bit_cast(i4_t, af[s][i]), __builtin_bit_cast(i4_t, bf[t][j]), c,
                        0, 0, 0);
                  else
                    lvl[g][i][j] =
                        __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[s][i], bf[t][j], c, 0, 0, 0);
                }
            }
            ++n;
            if (n == MID) barrier();
            // loads spread over the products from MID on
            const int upto = n < MID ? 0 : 2 * S * (n - MID + 1) / (NP - MID + 1);
#pragma unroll
            for (; e < upto; ++e) load(X, e);
            __builtin_amdgcn_sched_barrier(0);
          }
      };
      auto fold = [&](int e) {
        if constexpr (I8) {
          if (__builtin_expect(since_fold > kJoinChunks || e < -900 || e > 1000, 0)) {
            const double scale = ldexp(1.0, e);
#pragma unroll
            for (int i = 0; i < AI; ++i)
#pragma unroll
              for (int j = 0; j < AJ; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                  double t = 0.0;
#pragma unroll
                  for (int g = NG - 1; g >= 0; --g) {
                    int x = lvl[g][i][j][v];
                    asm volatile("" : "+v"(x));  // (kept out of the common path)
                    t = fma((double)x, 1.0 / (double)(1LL << (7 * g)), t);
                  }
                  acc[i][j][v] = fma(t, scale, acc[i][j][v]);
                }
            return;
          }
        }
        const double scale = ldexp(1.0, e - (I8 && S <= 5 ? 7 * (S - 1) : 0));
#pragma unroll
        for (int i = 0; i < AI; ++i)
#pragma unroll
          for (int j = 0; j < AJ; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              double t;
              if constexpr (I8) {
                // (six limbs: level 0 is added to the other five, which
                // rounds once, as the sum level by level does)
                constexpr int G0 = S > 5 ? 1 : 0;
                int64_t x = join_first(lvl[S - 1][i][j][v]);
#pragma unroll
                for (int g = S - 2; g >= G0; --g)
                  x = join_next(lvl[g][i][j][v], 1 << (7 * (S - 1 - g)), x);
                t = __longlong_as_double(x) - kJoin;
                if (G0) t = fma(t, 1.0 / (double)(1LL << 35), (double)lvl[0][i][j][v]);
              } else {
                t = (double)lvl[NG - 1][i][j][v];
#pragma unroll
                for (int g = NG - 2; g >= 0; --g) t += (double)lvl[g][i][j][v];
              }
              acc[i][j][v] = fma(t, scale, acc[i][j][v]);
            }
      };
      // One chunk out of stage X, chunk c + 2 into its place.
      auto step = [&](auto X) {
        __builtin_amdgcn_s_waitcnt(wait_vm(2 * S));
        barrier();
        bf8_t af[S][AI], bf[S][AJ];
        if constexpr (ACTIVE) {
#pragma unroll
          for (int s = 0; s < S; ++s) {
#pragma unroll
            for (int i = 0; i < AI; ++i)
              if (s == 0) af[s][i] = stage(X)[0][s][fa + i * NEXT];
#pragma unroll
            for (int j = 0; j < AJ; ++j) bf[s][j] = stage(X)[1][s][fb + j * NEXT];
          }
#pragma unroll
          for (int s = 1; s < S; ++s)
#pragma unroll
            for (int i = 0; i < AI; ++i) af[s][i] = stage(X)[0][s][fa + i * NEXT];
        }
        const bool ends = decltype(X)::value == 0 ? ends0 : ends1;
        const int e = decltype(X)::value == 0 ? exp0 : exp1;
        next_chunk(X);
        // (a wave that multiplies goes first: the other workgroup's reads and
        // loads fit between; 2% on the INT8 cases)
        __builtin_amdgcn_s_setprio(2);
        if (since_fold == 0) products(X, af, bf, ic<1>{});
        else products(X, af, bf, ic<0>{});
        __builtin_amdgcn_s_setprio(0);
        ++since_fold;
        if (ends || since_fold == FOLD) {
          if constexpr (ACTIVE) fold(e);
          since_fold = 0;
        }
      };
      if (have) {
        for (;;) {
          step(ic<0>{});
          if (!valid1) break;
          step(ic<1>{});
          if (!valid0) break;
        }
        // the loads that lie outside land before the stages are used again
        __builtin_amdgcn_s_waitcnt(wait_vm(0));
      }

      if constexpr (ACTIVE) {
        const int64_t t_coff = uni64(tp->c_off);
        const int t_ldc = uni(tp->ldc), t_flags = uni(tp->flags);
        const bool beta1 = (t_flags & TAMX_TASK_BETA1) != 0;
        const double alpha = args()->alpha;
        double* __restrict__ c = args()->C + t_coff;
        tamx::with_result_index(args()->c_scatter, args()->task_tile, lo, t_flags, t_ldc,
                                [&](auto cidx) {
#pragma unroll
          for (int i = 0; i < AI; ++i)
#pragma unroll
            for (int j = 0; j < AJ; ++j)
#pragma unroll
              for (int v = 0; v < 4; ++v) {
                // 16x16 MFMA output: row 4 * (lane / 16) + v, column lane % 16
                const int row = wr + i * 32 + lq * 4 + v;
                const int col = wc + j * 32 + lrow;
                if (row < mrem && col < nrem) {
                  const int64_t idx = cidx(r0 + row, c0 + col);
                  double val = alpha * acc[i][j][v];
                  if (beta1) val += c[idx];
                  c[idx] = val;
                }
              }
        });
      }
    };  // run_item

    if (have) {
      fill_table(lp);
      next_chunk(ic<0>{});
#pragma unroll
      for (int e = 0; e < 2 * S; ++e) load(ic<0>{}, e);
      next_chunk(ic<1>{});
#pragma unroll
      for (int e = 0; e < 2 * S; ++e) load(ic<1>{}, e);
    }
    if (ni == 2 && nj == 2) run_item(ic<2>{}, ic<2>{});
    else if (ni == 0 || nj == 0) run_item(ic<0>{}, ic<0>{});
    else if (ni == 2) run_item(ic<2>{}, ic<1>{});
    else if (nj == 2) run_item(ic<1>{}, ic<2>{});
    else run_item(ic<1>{}, ic<1>{});
  }
}

template <int S, bool I8>
int launch_staged(tamx_context* ctx, tamx_worklist* wl, const SplitParams& prm, hipStream_t s) {
  auto kern = split_gemm_staged_kernel<S, I8>;
  int occ = 0;
  TAMX_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kern, kThreads, 0));
  if (occ < 1) occ = 1;
  if (int rc = tamx::plan_items(wl, kTile, kTile, s)) return rc;
  kern<<<ctx->num_cus * occ, kThreads, 0, s>>>(prm);
  TAMX_LAUNCH_CHECK();
  return TAMX_OK;
}

}  // namespace

int tamx::split::launch_split_gemm_staged(int limb_type, int nslices, tamx_context* ctx,
                                          tamx_worklist* wl, const SplitParams& prm,
                                          hipStream_t s) {
  if (limb_type == TAMX_LIMB_I8) {
    switch (nslices) {
      case 2: return launch_staged<2, true>(ctx, wl, prm, s);
      case 3: return launch_staged<3, true>(ctx, wl, prm, s);
      case 4: return launch_staged<4, true>(ctx, wl, prm, s);
      case 5: return launch_staged<5, true>(ctx, wl, prm, s);
      default: return launch_staged<6, true>(ctx, wl, prm, s);
    }
  }
  switch (nslices) {
    case 2: return launch_staged<2, false>(ctx, wl, prm, s);
    case 3: return launch_staged<3, false>(ctx, wl, prm, s);
    case 4: return launch_staged<4, false>(ctx, wl, prm, s);
    case 5: return launch_staged<5, false>(ctx, wl, prm, s);
    default: return launch_staged<6, false>(ctx, wl, prm, s);
  }
}
