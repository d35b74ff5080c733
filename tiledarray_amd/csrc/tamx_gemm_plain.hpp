// The persistent grouped GEMM kernel for plain operands (row-major tiles,
// FP64 and FP32 MFMA).
//
// Work division as in tamx_gemm.hpp: a result tile of m x n is cut into
// BM x BN macro tiles ("items"); a workgroup of 2 x 2 waves takes items from
// a device queue, walks the item's tile pairs in order, K in chunks of BK,
// and writes the result once.  The 16 x 16 blocks of a macro tile go to the
// waves in turn along each direction (wave w has blocks w, w + 2, ...), so a
// ragged edge leaves the waves with nearly equal work.
//
// Chunks travel from global memory straight into LDS (16-byte
// buffer_load ... lds, no registers and no LDS store instructions), one
// chunk ahead of the MFMAs, through two stage buffers with one barrier per
// chunk.
//
// What bounds it: an FP64 MFMA holds its SIMD for 64 cycles and overlaps with
// no VALU instruction, and under this load the clock falls from 2.4 to about
// 2.0 GHz, so what costs is everything but the MFMAs: VALU instructions,
// bytes moved through LDS and bytes fetched from L2 (a 64 x 64 tile asks for
// 16 bytes per cycle and CU, about 10 TB/s).  Staging through registers took
// four times as many load instructions (8 bytes each) and as many LDS stores;
// with direct loads and offsets that are fixed per pair a chunk costs no
// vector arithmetic but the fragment addresses.  GEMM against it, 64 x 64 macro
// tiles on one card: FP64 ladder at 32 x 192 53.4 -> 48.3 ms, block-sparse
// 16384^3 3.41 -> 3.13 ms, 5000^3 700 -> 631 us.
#pragma once

#include "tamx_gemm.hpp"

namespace {

// Buffer descriptor word 3 for raw 32-bit-format buffers on this family, and
// the offset that lies outside every range.
constexpr int kBufFlags = 0x00020000;
constexpr uint32_t kOutside = 0x80000000u;

// what the units outside a tile load where they have 64-bit addresses
__device__ __align__(16) const unsigned char g_zero_unit[16] = {};

// Where the elements of one operand's chunk (R rows or columns of the
// macro tile, BK k) lie in its LDS stage.  The stage is an array of 16-byte
// units in the order the loads write them: unit g of the stage is fetched by
// thread g % NT with its load g / NT.  KF: k is the contiguous index of the
// stored tile, the stage holds R rows of BK k; otherwise BK rows of R.
//
// Loads write lanes in order, so rows cannot be padded; instead the lane of
// unit position `pos` in row r fetches source unit pos ^ swz(r), with swz
// chosen so that the 64 lanes of a fragment read (16 rows or columns times
// 4 k) fall on distinct banks of a 256-byte window.
template <typename T, int R, int BK, bool KF, int NT>
struct StageMap {
  static constexpr int EPU = 16 / (int)sizeof(T);     // elements per unit
  static constexpr int UPR = (KF ? BK : R) / EPU;     // units per stage row
  static constexpr int UNITS = R * BK / EPU;
  static constexpr int LOADS = (UNITS + NT - 1) / NT;
  static_assert(UNITS % 64 == 0 && UPR >= 1, "chunk split over the waves");
  // the largest leading dimension for which a chunk's rows lie within
  // kOutside bytes (2^22 for 64 rows of FP64)
  static constexpr int MAX_LD = (int)(kOutside / ((KF ? R : BK) * sizeof(T)));
  static constexpr int RPW = UPR * 16 >= 256 ? 1 : 256 / (UPR * 16);  // rows per window
  __device__ static inline int swz(int r) {
    // KF: 16 rows read the same unit column; else 16 / EPU consecutive units
    // of 4 rows (k) are read, which need distinct shares of the window
    if constexpr (KF) return (r / RPW) & (UPR - 1);
    constexpr int G = EPU / RPW;  // EPU: 16-column shares of a window
    static_assert(EPU % RPW == 0, "stage rows per window");
    return ((r / RPW) % G) * (16 / EPU);
  }
  // stage row and source unit of this thread's load e
  __device__ static inline int row(int tid, int e) { return (e * NT + tid) / UPR; }
  __device__ static inline int unit(int tid, int e) {
    const int g = e * NT + tid;
    return (g % UPR) ^ swz(g / UPR);
  }
  // whether the wave has a load e (a small chunk leaves some without)
  __device__ static inline bool has(int wave, int e) {
    return UNITS % NT == 0 || e * NT + wave * 64 < UNITS;
  }
  // byte offset of element (x, k): x the row or column of the macro tile
  __device__ static inline int at(int x, int k) {
    const int r = KF ? x : k, c = KF ? k : x;
    return (r * UPR + ((c / EPU) ^ swz(r))) * 16 + (c % EPU) * (int)sizeof(T);
  }
};

// LDS byte offsets of a wave's fragments, W waves along the direction: at(s,
// i) is element (x0 + 16 W i, k 4 s + lk) of the stage, x0 the lane's row
// (column) in the wave's first block.  With k contiguous the swizzle mixes s
// into the offset (one register per step), else it mixes at most i.
template <typename T, int R, int BK, bool KF, int NT, int W>
struct FragMap {
  using S = StageMap<T, R, BK, KF, NT>;
  static constexpr int STEP = 16 * W;  // from one block of the wave to its next
  static constexpr int N = KF ? BK / 4 : (STEP / S::EPU % 16 == 0 ? 1 : R / STEP);
  int o[N];
  __device__ FragMap(int x0, int lk) {
#pragma unroll
    for (int n = 0; n < N; ++n) o[n] = KF ? S::at(x0, 4 * n + lk) : S::at(x0 + STEP * n, lk);
  }
  __device__ inline int at(int s, int i) const {
    if constexpr (KF) return o[s] + i * STEP * S::UPR * 16;
    return o[N == 1 ? 0 : i] + (N == 1 ? i * STEP * (int)sizeof(T) : 0) + s * 4 * S::UPR * 16;
  }
};

// Macro tiles of a result tile are taken column by column in bands of this
// many rows: the items in flight on an XCD then share both operands' panels
// in its L2 (row by row, a result tile of 256 x 4096 kept one A panel and 64
// B panels in flight, and every B panel was fetched again for each of its
// four rows: FP64 ladder at 32 x 192, 52.1 ms row by row, 48.3 in bands).
constexpr int kBandRows = 8;

// vmcnt(0), the other counters left alone (gfx9 encoding)
constexpr int kWaitVm0 = (7 << 4) | (15 << 8);

// One operand's chunk into its stage `dst`: rem rows (columns) and kc k from
// element `org` of the pool, vo the byte offsets of this thread's units.
// With k contiguous the chunk is cut at kc by marking the units past it; the
// rest of a unit that kc cuts is cleared once the loads have landed.
template <class S, typename T, int BK, bool KF, int NT>
__device__ __forceinline__ void load_operand(const T* base, int64_t org, int ld, int rem, int kc,
                                             const uint32_t (&vo)[S::LOADS], unsigned char* dst,
                                             int tid, int wave) {
#ifdef __HIP_DEVICE_COMPILE__  // (the host pass does not accept the LDS load builtin)
  const int rng =
      kc > 0 ? uni((KF ? (rem - 1) * ld + kc : (kc - 1) * ld + rem) * (int)sizeof(T)) : 0;
  const auto d = __builtin_amdgcn_make_buffer_rsrc((void*)(base + uni64(org)), (short)0, rng,
                                                   kBufFlags);
  const bool cut = KF && kc < BK;
  asm volatile("" : "+s"(wave));  // (else every load's destination stays in a register)
#pragma unroll
  for (int e = 0; e < S::LOADS; ++e) {
    if (!S::has(wave, e)) continue;
    uint32_t o = vo[e];
    if (cut && S::unit(tid, e) * S::EPU >= kc) o = kOutside;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        d, (__attribute__((address_space(3))) void*)(dst + (e * NT + wave * 64) * 16), 16, o, 0, 0,
        0);
  }
#endif
}

// The same with 64-bit addresses, for any leading dimension.  Units outside
// the tile load zeros; the elements of a unit that the end of its row cuts
// are copied one by one, so that nothing past the row is read.
template <class S, typename T, bool KF, int NT>
__device__ __forceinline__ void load_operand_far(const T* base, int64_t org, int ld, int rem,
                                                 int kc, unsigned char* dst, int tid, int wave) {
#ifdef __HIP_DEVICE_COMPILE__
  const int rows = KF ? rem : kc, cols = KF ? kc : rem;
#pragma unroll
  for (int e = 0; e < S::LOADS; ++e) {
    if (!S::has(wave, e)) continue;
    const int r = S::row(tid, e), c = S::unit(tid, e) * S::EPU;
    const T* src = base + org + ((int64_t)r * ld + c);
    const bool whole = r < rows && c + S::EPU <= cols;
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) void*)(whole ? (const void*)src
                                                              : (const void*)g_zero_unit),
        (__attribute__((address_space(3))) void*)(dst + (e * NT + wave * 64) * 16), 16, 0, 0);
    if (cols % S::EPU != 0 && r < rows && c < cols && !whole) {
      T* unit = reinterpret_cast<T*>(dst + (e * NT + tid) * 16);
      T v[S::EPU];
#pragma unroll
      for (int x = 0; x < S::EPU; ++x) v[x] = c + x < cols ? src[x] : T(0);
      __builtin_amdgcn_s_waitcnt(kWaitVm0);  // (the zeros have landed)
#pragma unroll
      for (int x = 0; x < S::EPU; ++x) unit[x] = v[x];
    }
  }
#endif
}

template <typename T, int BM, int BN, int BK, int WM, int WN, bool TA, bool TB, int OCC>
__global__ __launch_bounds__(64 * WM * WN, OCC) void plain_gemm_kernel(GemmParams<T> p) {
  using M = Mfma<T>;
  using acc_t = typename M::acc_t;
  constexpr int NT = 64 * WM * WN;                         // threads
  constexpr int FM = BM / (16 * WM), FN = BN / (16 * WN);  // 16x16 blocks per wave
  constexpr int NS = BK / 4;                               // MFMA steps per chunk
  using SA = StageMap<T, BM, BK, !TA, NT>;
  using SB = StageMap<T, BN, BK, TB, NT>;
  constexpr int EPU = SA::EPU;
  constexpr int A_BYTES = BM * BK * (int)sizeof(T), B_BYTES = BN * BK * (int)sizeof(T);
  static_assert(BM % (16 * WM) == 0 && BN % (16 * WN) == 0 && BK % 4 == 0, "tile shape");

  // one variable per stage: the compiler then knows that loads landing in
  // one stage do not alias reads of the other
  __shared__ __align__(256) unsigned char stage0[A_BYTES + B_BYTES];
  __shared__ __align__(256) unsigned char stage1[A_BYTES + B_BYTES];
  __shared__ int s_item;
  auto stage = [&](auto X) -> unsigned char* {
    if constexpr (decltype(X)::value == 0) return stage0; else return stage1;
  };
  using zero = std::integral_constant<int, 0>;
  using one = std::integral_constant<int, 1>;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = uni(tid >> 6);
  const int lrow = lane & 15, lk = lane >> 4;

  const int wr = (wave / WN) * 16, wc = (wave % WN) * 16;  // the wave's first block
  const FragMap<T, BM, BK, !TA, NT, WM> fa(wr + lrow, lk);
  const FragMap<T, BN, BK, TB, NT, WN> fb(wc + lrow, lk);

  int64_t ntasks64 = p.counters[TAMX_WL_NTASKS];
  // same validation as the planner: an invalid list has no items
  if (ntasks64 < 0 || ntasks64 > p.task_capacity || p.counters[TAMX_WL_STATUS] != 0)
    ntasks64 = 0;
  const int32_t ntasks = uni((int32_t)ntasks64);
  int32_t total = uni(p.prefix[ntasks > 0 ? ntasks : 0]);
  if (p.choice != nullptr && uni(*p.choice) != BM) total = 0;  // the other macro tile runs

  tamx::ItemQueue queue(p.queue, total);  // used by thread 0 only
  for (;;) {
    if (tid == 0) s_item = queue.next();
    __syncthreads();
    const int item = uni(s_item);
    __syncthreads();
    if (item < 0) break;

    int lo;
    if (total <= p.item_capacity) {
      lo = uni(tamx::scalar_ptr(p.item_task)[item]);
    } else {
      lo = 0;
      int hi = ntasks - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (uni(p.prefix[mid]) <= item) lo = mid; else hi = mid - 1;
      }
    }
    const auto* tp = tamx::scalar_ptr(p.tasks) + lo;
    const int64_t t_coff = uni64(tp->c_off);
    const int t_m = uni(tp->m), t_n = uni(tp->n), t_ldc = uni(tp->ldc);
    const int t_pb = uni(tp->pair_begin), t_pc = uni(tp->pair_count);
    const int t_flags = uni(tp->flags);
    const int local = item - uni(tamx::scalar_ptr(p.prefix)[lo]);
    const int tiles_n = (t_n + BN - 1) / BN;
    const int tiles_m = (t_m + BM - 1) / BM;
    const int band = local / (kBandRows * tiles_n), in_band = local - band * kBandRows * tiles_n;
    const int band_rows = min(kBandRows, tiles_m - band * kBandRows);
    const int r0 = uni(band * kBandRows + in_band % band_rows) * BM;
    const int c0 = uni(in_band / band_rows) * BN;
    const int mrem = min(BM, t_m - r0), nrem = min(BN, t_n - c0);
    // the wave's 16-row (column) blocks inside the tile
    const int ni = uni(min(FM, max(0, (mrem - wr + 16 * WM - 1) / (16 * WM))));
    const int nj = uni(min(FN, max(0, (nrem - wc + 16 * WN - 1) / (16 * WN))));

    // (not __syncthreads: its release fence would also wait for the loads
    // of the next chunk; LDS stores of this thread are waited for here)
    auto barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // The item's sum, with loads through 32-bit offsets, or (FAR) 64-bit
    // addresses where these do not do; false where a pair would need the latter.
    //
    // Load cursor: pair lp at k lk0.  Per pair every staged unit has a
    // 32-bit byte offset from the chunk's origin, fixed for the pair; the
    // descriptor of a chunk starts at the macro tile's first row (column)
    // and the chunk's first k and ends with the last valid element, so what
    // lies past it (rows past the tile, k past the pair's end where k is the
    // slow index) loads zero.  Units wholly past the row's end carry
    // kOutside.  With a leading dimension above MAX_LD the offsets of a chunk
    // could pass 2^31: the item is then summed anew with 64-bit addresses, in
    // a loop of its own, for the mere presence of those loads in this one
    // costs it up to 5%.  (Figures in FP64, NN and NT, against a descriptor
    // for every single stage row above a leading dimension of 2^20, eight
    // masked loads in place of each where k is contiguous: M and N 1024 over K
    // of 2^20 + 4096 in one tile 121 and 197 ms, now 49 and 55; M and N 256
    // over K of 2^22 + 64 483 and 786, now 229 and 248.)
    acc_t acc[FM][FN];
    auto sum_item = [&](auto FAR_) -> bool {
      constexpr bool FAR = decltype(FAR_)::value;
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[i][j][v] = T(0);

      int64_t a_base = 0, b_base = 0;
      int a_ld = 0, b_ld = 0, pk = 0;
      uint32_t a_vo[SA::LOADS], b_vo[SB::LOADS];
      const int pend = t_pb + t_pc;
      int lp = t_pb, lk0 = 0;
      bool far = false;  // a pair that needs 64-bit addresses, which ends this loop
      auto set_pair = [&](int pi) {
        const auto& pp = tamx::scalar_ptr(p.pairs)[pi];
        a_base = uni64(pp.a_off);
        b_base = uni64(pp.b_off);
        pk = uni(pp.k);
        a_ld = uni(pp.lda);
        b_ld = uni(pp.ldb);
        if (!FAR && __builtin_expect(a_ld > SA::MAX_LD || b_ld > SB::MAX_LD, 0)) {
          far = true;
          lp = pend;
        }
#pragma unroll
        for (int e = 0; e < SA::LOADS; ++e) {
          const int r = SA::row(tid, e), c = SA::unit(tid, e) * EPU;
          a_vo[e] = (!TA || c < mrem) ? ((uint32_t)r * a_ld + c) * (uint32_t)sizeof(T) : kOutside;
        }
#pragma unroll
        for (int e = 0; e < SB::LOADS; ++e) {
          const int r = SB::row(tid, e), c = SB::unit(tid, e) * EPU;
          b_vo[e] = (TB || c < nrem) ? ((uint32_t)r * b_ld + c) * (uint32_t)sizeof(T) : kOutside;
        }
      };

      if (lp < pend) set_pair(lp);
      // loads the cursor's chunk and advances the cursor; returns the number
      // of k in the chunk
      auto load_chunk = [&](auto X) -> int {
        const int kc = min(BK, pk - lk0);
        unsigned char* st = stage(X);
        const int64_t a_org = a_base + (TA ? (int64_t)lk0 * a_ld + r0 : (int64_t)r0 * a_ld + lk0);
        const int64_t b_org = b_base + (TB ? (int64_t)c0 * b_ld + lk0 : (int64_t)lk0 * b_ld + c0);
        if (FAR && a_ld > SA::MAX_LD)
          load_operand_far<SA, T, !TA, NT>(p.A, a_org, a_ld, mrem, kc, st, tid, wave);
        else
          load_operand<SA, T, BK, !TA, NT>(p.A, a_org, a_ld, mrem, kc, a_vo, st, tid, wave);
        if (FAR && b_ld > SB::MAX_LD)
          load_operand_far<SB, T, TB, NT>(p.B, b_org, b_ld, nrem, kc, st + A_BYTES, tid, wave);
        else
          load_operand<SB, T, BK, TB, NT>(p.B, b_org, b_ld, nrem, kc, b_vo, st + A_BYTES, tid,
                                          wave);
        lk0 += BK;
        if (lk0 >= pk) {
          ++lp;
          lk0 = 0;
          if (lp < pend) set_pair(lp);
        }
        return kc;
      };
      // Waits for this thread's loads of a chunk of kc k, and clears what they
      // brought from past the k end in the unit that kc cuts (the other
      // operand holds zeros there, but zero times an infinity is not zero).
      auto landed = [&](auto X, int kc) {
        __builtin_amdgcn_s_waitcnt(kWaitVm0);
        if ((!TA || TB) && (kc % EPU) != 0) {
          unsigned char* st = stage(X);
          auto clear = [&](auto map, unsigned char* dst) {
            using S = decltype(map);
#pragma unroll
            for (int e = 0; e < S::LOADS; ++e)
              if (S::has(wave, e) && S::unit(tid, e) == kc / EPU)
                for (int x = kc % EPU; x < EPU; ++x)
                  *reinterpret_cast<T*>(dst + (e * NT + tid) * 16 + x * (int)sizeof(T)) = T(0);
          };
          if constexpr (!TA) clear(SA{}, st);
          if constexpr (TB) clear(SB{}, st + A_BYTES);
        }
      };
      // nks MFMA steps of a chunk; the fragments of step s + 1 are read while
      // the MFMAs of step s run (reads of blocks past a ragged edge stay inside
      // the stage and are not used)
      auto compute_chunk = [&](auto X, int kc) {
        if (ni == 0 || nj == 0) return;
        const int nks = (kc + 3) >> 2;
        const unsigned char* st = stage(X);
        T af[2][FM], bf[2][FN];
        auto frag = [&](int s, T (&a)[FM], T (&b)[FN]) {
#pragma unroll
          for (int i = 0; i < FM; ++i) a[i] = *reinterpret_cast<const T*>(st + fa.at(s, i));
#pragma unroll
          for (int j = 0; j < FN; ++j)
            b[j] = *reinterpret_cast<const T*>(st + A_BYTES + fb.at(s, j));
        };
        frag(0, af[0], bf[0]);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          if (s < nks) {
            if (s + 1 < NS) frag(s + 1, af[(s + 1) & 1], bf[(s + 1) & 1]);
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
              for (int j = 0; j < FN; ++j)
                // (the rare loop has no conditions, for they would be held in
                // scalar registers through the other)
                if (FAR || (i < ni && j < nj))
                  acc[i][j] = M::op(af[s & 1][i], bf[s & 1][j], acc[i][j]);
          }
        }
      };

      // Pipeline: while chunk c is multiplied out of one stage, chunk c + 1
      // lands in the other.
      if (lp < pend) {
        int k0c = load_chunk(zero{}), k1c = 0;
        for (;;) {
          landed(zero{}, k0c);
          barrier();
          bool more = lp < pend;
          if (more) k1c = load_chunk(one{});
          compute_chunk(zero{}, k0c);
          if (!more) break;
          landed(one{}, k1c);
          barrier();
          more = lp < pend;
          if (more) k0c = load_chunk(zero{});
          compute_chunk(one{}, k1c);
          if (!more) break;
        }
      }
      return !far;
    };  // sum_item

    if (__builtin_expect(!sum_item(std::false_type{}), 0)) {
      barrier();  // every wave is done with the stages
      (void)sum_item(std::true_type{});
    }

    const bool beta1 = (t_flags & TAMX_TASK_BETA1) != 0;
    T* __restrict__ c = p.C + t_coff;
    tamx::with_result_index(p.c_scatter, p.task_tile, lo, t_flags, t_ldc, [&](auto cidx) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int row = wr + i * 16 * WM + M::row(lk, v);
            const int col = wc + j * 16 * WN + lrow;
            if (row < mrem && col < nrem) {
              const int64_t idx = cidx(r0 + row, c0 + col);
              T val = p.alpha * acc[i][j][v];
              if (beta1) val += c[idx];
              c[idx] = val;
            }
          }
    });
  }
}

// workgroups per CU that the registers are budgeted for (FP32 stages of 32 k
// are half the size of FP64's, so four of them fit)
template <typename T>
constexpr int plain_occupancy(int bm, int bn, int bk) {
  if (bm * bn <= 64 * 64) return bk > 16 && sizeof(T) == 8 ? 2 : 4;
  return bm * bn >= 128 * 128 ? 2 : (bk > 16 ? 1 : 3);
}
template <typename T, int BM, int BN, int BK, bool TA, bool TB>
struct GemmKernel<T, BM, BN, BK, TA, TB, 0> {
  static constexpr auto get() {
    return plain_gemm_kernel<T, BM, BN, BK, 2, 2, TA, TB, plain_occupancy<T>(BM, BN, BK)>;
  }
  static constexpr int threads() { return kThreads; }
};

}  // namespace
