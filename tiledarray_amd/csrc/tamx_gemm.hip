// Plain entry points of the grouped GEMM and its item planner (the kernel
// is in tamx_gemm.hpp).
#include "tamx_gemm_plain.hpp"
#include "tamx_queue.hpp"
#include "tamx_scan.hpp"

namespace {

// Item planner: prefix[t] = number of BM x BN macro tiles of tasks 0..t-1,
// and the item -> task map when it fits in item_capacity entries.  Three
// launches (chunk sums over kScanBlocks workgroups, one-workgroup scan of the
// sums, chunk rescans), each walking the task list once.  The last one also
// clears the item queue for the GEMM that follows.
//
// A launch may leave the macro tile, 64 x 64 or 128 x 128, to the planner: the
// first two kernels then add up items and cost for both, and the choice goes
// by the tasks that are really there, which the host does not know.
__device__ inline int64_t planned_tasks(const int64_t* counters, int64_t capacity) {
  const int64_t n = counters[TAMX_WL_NTASKS];
  return (n < 0 || n > capacity || counters[TAMX_WL_STATUS] != 0) ? 0 : n;
}
__device__ inline int32_t task_items(const tamx_gemm_task* tasks, int64_t i, int bm,
                                     int bn) {
  const tamx_gemm_task t = tasks[i];
  return ((t.m + bm - 1) / bm) * ((t.n + bn - 1) / bn);
}

constexpr int kPlanThreads = 256;

__global__ __launch_bounds__(kPlanThreads) void plan_items_sum_kernel(
    const tamx_gemm_task* __restrict__ tasks, const int64_t* __restrict__ counters,
    int bm, int bn, int64_t capacity, int32_t* __restrict__ partial) {
  __shared__ int32_t red[kPlanThreads];
  const int64_t n = planned_tasks(counters, capacity);
  tamx::scan_phase1<kPlanThreads, int32_t>(
      n, red, [&](int64_t i) { return task_items(tasks, i, bm, bn); }, partial);
}

__global__ __launch_bounds__(1024) void plan_items_offsets_kernel(int32_t* partial) {
  __shared__ int32_t part[1024];
  tamx::scan_phase2<1024, int32_t>(tamx::kScanBlocks, part, partial);
}

// Items and their cost in 64 x 64 (0) and 128 x 128 (1) macro tiles.
struct PlanSums {
  int32_t items[2];
  float cost[2];
  PlanSums() = default;
  __device__ explicit PlanSums(int x) : items{x, x}, cost{(float)x, (float)x} {}
  __device__ PlanSums& operator+=(const PlanSums& o) {
    for (int i = 0; i < 2; ++i) {
      items[i] += o.items[i];
      cost[i] += o.cost[i];
    }
    return *this;
  }
};

// The cost of a task in units of a whole item: half of an item's is the same
// however little of the macro tile it fills (its chunks and barriers), half
// goes with the 16 x 16 blocks of its busiest wave (of two in each
// direction).  Result tiles narrower than 192 cost a quarter more in 128 x
// 128.  The halves, the quarter and the rule below are what agrees with the
// GEMM times of both macro tiles on 65 products: uniform tiles of 160 to 4096,
// flat ones of 16 x 8192 to 4096 x 36, block-sparse ones of 128 to 900 and
// ladders of 8 to 24 occupied orbitals a tile.
__device__ inline void add_macro_tiles(PlanSums& s, int i, int m, int n) {
  const int b = i ? 128 : 64;
  // items in one direction, and their blocks in quarters of an item
  auto items = [&](int x) { return (x + b - 1) / b; };
  auto quarters = [&](int x) {
    const int rest = ((x % b + 15) / 16 + 1) / 2;  // blocks of the busiest wave
    return x / b * 4 + rest * (i ? 1 : 2);
  };
  const int count = items(m) * items(n);
  s.items[i] = count;
  s.cost[i] = 0.5f * (float)count + 0.5f / 16.0f * ((float)quarters(m) * (float)quarters(n));
  if (i && min(m, n) < 192) s.cost[i] *= 1.25f;
}

__global__ __launch_bounds__(kPlanThreads) void plan_sums_kernel(
    const tamx_gemm_task* __restrict__ tasks, const int64_t* __restrict__ counters,
    int64_t capacity, PlanSums* __restrict__ partial) {
  __shared__ PlanSums red[kPlanThreads];
  const int64_t n = planned_tasks(counters, capacity);
  tamx::scan_phase1<kPlanThreads, PlanSums>(
      n, red,
      [&](int64_t i) {
        const tamx_gemm_task t = tasks[i];
        PlanSums s(0);
        for (int k = 0; k < 2; ++k) add_macro_tiles(s, k, t.m, t.n);
        return s;
      },
      partial);
}

// Picks the macro tile and scans its items.  128 x 128 reads half the operand
// bytes per MFMA, from LDS and from L2, which gives 2 to 9% where everything
// else is equal (17% at most), but wants full macro tiles and several of them
// for each CU: a load of L items a CU is taken to last as long as L and a
// quarter of what is missing to the next whole number.  On the products above
// it picks 128 x 128 for 26, none of them slower with it, and leaves out four
// that would gain 3 to 7%.
__global__ __launch_bounds__(1024) void plan_choose_kernel(const PlanSums* sums, int32_t* partial,
                                                           int num_cus, int32_t* choice) {
  __shared__ int32_t part[1024];
  __shared__ PlanSums red[tamx::kScanBlocks];
  const int t = threadIdx.x;
  static_assert(tamx::kScanBlocks <= 1024, "one thread per chunk");
  if (t < tamx::kScanBlocks) red[t] = sums[t];
  __syncthreads();
  for (int w = tamx::kScanBlocks / 2; w > 0; w >>= 1) {
    if (t < w) red[t] += red[t + w];
    __syncthreads();
  }
  auto lasts = [](float l) { return l + 0.25f * (ceilf(l) - l); };
  const float l64 = red[0].cost[0] / num_cus, l128 = red[0].cost[1] / num_cus;
  const int pick = l128 >= 3.5f && 0.97f * 4.0f * lasts(l128) < lasts(l64);
  if (t == 0) choice[0] = pick ? 128 : 64;
  if (t < tamx::kScanBlocks) partial[t] = sums[t].items[pick];
  __syncthreads();
  tamx::scan_phase2<1024, int32_t>(tamx::kScanBlocks, part, partial);
}

// choice: the macro tile's width where the planner picked it (else null)
__global__ __launch_bounds__(kPlanThreads) void plan_items_fill_kernel(
    const tamx_gemm_task* __restrict__ tasks, const int64_t* __restrict__ counters,
    int bm, int bn, const int32_t* __restrict__ choice, int64_t capacity,
    const int32_t* __restrict__ partial, int32_t* __restrict__ prefix,
    int32_t* __restrict__ item_task, int64_t item_capacity, int32_t* __restrict__ queue) {
  if (choice) bm = bn = choice[0];
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < tamx::kQueueInts; i += kPlanThreads) queue[i] = 0;
  __shared__ int32_t part[kPlanThreads];
  const int64_t n = planned_tasks(counters, capacity);
  const int32_t total = partial[tamx::kScanBlocks];
  const bool map = total <= item_capacity;
  auto count = [&](int64_t i) { return task_items(tasks, i, bm, bn); };
  tamx::scan_phase3<kPlanThreads, int32_t>(
      n, part, count,
      [&](int64_t i, int32_t q0) {
        prefix[i] = q0;
        if (map) {
          const int32_t q1 = q0 + count(i);
          for (int32_t q = q0; q < q1; ++q) item_task[q] = (int32_t)i;
        }
      },
      partial);
  if (blockIdx.x == 0 && threadIdx.x == 0) prefix[n] = total;
}

}  // namespace

int tamx::plan_items(tamx_worklist* wl, int bm, int bn, hipStream_t s) {
  auto* partial = static_cast<int32_t*>(wl->scan_partials);
  plan_items_sum_kernel<<<tamx::kScanBlocks, kPlanThreads, 0, s>>>(
      wl->tasks, wl->counters, bm, bn, wl->task_capacity, partial);
  TAMX_LAUNCH_CHECK();
  plan_items_offsets_kernel<<<1, 1024, 0, s>>>(partial);
  TAMX_LAUNCH_CHECK();
  plan_items_fill_kernel<<<tamx::kScanBlocks, kPlanThreads, 0, s>>>(
      wl->tasks, wl->counters, bm, bn, nullptr, wl->task_capacity, partial, wl->item_prefix,
      wl->item_task, wl->item_capacity, wl->queue);
  TAMX_LAUNCH_CHECK();
  return TAMX_OK;
}

int tamx::plan_items_choosing(tamx_context* ctx, tamx_worklist* wl, hipStream_t s) {
  // (the sums of both macro tiles, then the chosen one's in the usual place)
  auto* partial = static_cast<int32_t*>(wl->scan_partials);
  auto* sums = reinterpret_cast<PlanSums*>(partial + tamx::kScanBlocks + 4);
  static_assert(sizeof(PlanSums) == 16 &&
                    (kScanBlocks + 4) * 4 + kScanBlocks * sizeof(PlanSums) <= 32 * kScanBlocks,
                "both fit the scan scratch");
  plan_sums_kernel<<<tamx::kScanBlocks, kPlanThreads, 0, s>>>(wl->tasks, wl->counters,
                                                              wl->task_capacity, sums);
  TAMX_LAUNCH_CHECK();
  plan_choose_kernel<<<1, 1024, 0, s>>>(sums, partial, ctx->num_cus, wl->choice);
  TAMX_LAUNCH_CHECK();
  plan_items_fill_kernel<<<tamx::kScanBlocks, kPlanThreads, 0, s>>>(
      wl->tasks, wl->counters, 0, 0, wl->choice, wl->task_capacity, partial, wl->item_prefix,
      wl->item_task, wl->item_capacity, wl->queue);
  TAMX_LAUNCH_CHECK();
  return TAMX_OK;
}

extern "C" {

int tamx_gemm_config_count(void) { return (int)(sizeof(kConfigs) / sizeof(kConfigs[0])); }

int tamx_gemm_config_get(int index, tamx_gemm_config* cfg) {
  TAMX_REQUIRE(cfg != nullptr, "null config");
  TAMX_REQUIRE(index >= 0 && index < tamx_gemm_config_count(), "config index out of range");
  cfg->bm = kConfigs[index][0];
  cfg->bn = kConfigs[index][1];
  cfg->bk = kConfigs[index][2];
  cfg->wgs_per_cu = 0;
  return TAMX_OK;
}

int tamx_gemm_macro_tile(const tamx_worklist* wl, tamx_gemm_config* cfg) {
  TAMX_REQUIRE(wl != nullptr && cfg != nullptr, "null argument");
  TAMX_REQUIRE(wl->last.bm != 0, "no grouped GEMM was launched on this work list");
  *cfg = wl->last;
  if (wl->last_chosen) {
    if (int rc = tamx::activate(wl->ctx)) return rc;
    int32_t width = 0;
    TAMX_CHECK_HIP(hipDeviceSynchronize());
    TAMX_CHECK_HIP(hipMemcpy(&width, wl->choice, sizeof(width), hipMemcpyDeviceToHost));
    cfg->bm = cfg->bn = width;
  }
  return TAMX_OK;
}

}  // extern "C"

int tamx::plain_gemm_f64(tamx_context* ctx, tamx_worklist* wl, int op_a, int op_b,
                         double alpha, const double* A, const double* B, double* C,
                         const tamx_gemm_config* cfg, const GatherTile* c_scatter,
                         void* stream) {
  return grouped_gemm<double, 0>(ctx, wl, op_a, op_b, alpha, A, B, C, stream, cfg, nullptr,
                                 nullptr, c_scatter);
}

int tamx::plain_gemm_f32(tamx_context* ctx, tamx_worklist* wl, int op_a, int op_b,
                         float alpha, const float* A, const float* B, float* C,
                         const tamx_gemm_config* cfg, const GatherTile* c_scatter,
                         void* stream) {
  return grouped_gemm<float, 0>(ctx, wl, op_a, op_b, alpha, A, B, C, stream, cfg, nullptr,
                                nullptr, c_scatter);
}

extern "C" {

int tamx_grouped_gemm_f64_config(tamx_context* ctx, tamx_worklist* wl, int op_a,
                                 int op_b, double alpha, const double* A,
                                 const double* B, double* C,
                                 const tamx_gemm_config* cfg, void* stream) {
  return grouped_gemm<double, 0>(ctx, wl, op_a, op_b, alpha, A, B, C, stream, cfg);
}

int tamx_grouped_gemm_f32_config(tamx_context* ctx, tamx_worklist* wl, int op_a,
                                 int op_b, float alpha, const float* A,
                                 const float* B, float* C,
                                 const tamx_gemm_config* cfg, void* stream) {
  return grouped_gemm<float, 0>(ctx, wl, op_a, op_b, alpha, A, B, C, stream, cfg);
}

int tamx_grouped_gemm_f64(tamx_context* ctx, tamx_worklist* wl, int op_a,
                          int op_b, double alpha, const double* A,
                          const double* B, double* C, void* stream) {
  return grouped_gemm<double, 0>(ctx, wl, op_a, op_b, alpha, A, B, C, stream, nullptr);
}

int tamx_grouped_gemm_f32(tamx_context* ctx, tamx_worklist* wl, int op_a,
                          int op_b, float alpha, const float* A,
                          const float* B, float* C, void* stream) {
  return grouped_gemm<float, 0>(ctx, wl, op_a, op_b, alpha, A, B, C, stream, nullptr);
}

}  // extern "C"
