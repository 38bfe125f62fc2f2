// afft_queue_long.hip -- the long jobs of an uneven batch (afft_queue.hip) when
// there are enough of them to fill the GPU.
//
//   rows   a job of 2^13, 2^14 or 2^15 complex points (c2c n, real n = twice
//          that) is one row, transformed by one work-group in LDS: the data
//          crosses memory once, where a chain of tiles takes it through a
//          scratch buffer (and a real job through its real pass as well).
//   pairs  a 2^16-point complex job takes the two passes of a four-step, each
//          a launch over the tiles of a group of such jobs.
//
// What bounds them: memory.  Of 10,000 jobs of 2^6..2^16 points (MI355X) 909
// rows of 2^15 take 183 us (2.6 TB/s: one group per CU, 3.6 rounds of it, loads
// and butterflies of a row in turn), 1818 rows of 2^13 and 2^14 111 us (3.2
// TB/s), 636 pairs 240 us (5.5 TB/s over both passes); as chains they took 0.85
// ms.  The whole batch: 906 -> 609 us.  With the three kinds of row in one
// kernel queue_row15_kernel spills 38 VGPRs (132 B a lane), queue_row14_kernel
// 10; the plans' own kernels of 2^15 points 2 to 14.
//
// Every kernel reads its list's length on the device and strides over it, so a
// captured launch runs the lists of the latest prepare on the grid of the one it
// was captured with.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "afft_queue_tasks.h"

namespace afgpu {

// What these kernels need of a task.
struct QRec {
  int kind, lg;
  unsigned long long src, dst;
};
__device__ __forceinline__ QRec q_rec(const QArgs& a, int i) {
  const QConst<QTask> t = q_const(a.tasks) + i;
  auto pair = [](int lo, int hi) AFGPU_INLINE { return (unsigned long long)(unsigned)hi << 32 | (unsigned)lo; };
  return {t->kind, t->lg, pair(t->first, t->job), pair(t->tile, t->need)};
}

// One row of 2^lg points, addressed through buffer resources.
template <int L, int SV, int EPI>
__device__ __forceinline__ void q_row(const QArgs& a, const QRec& tk, int tid, cx<float>* lds) {
  constexpr bool REAL = EPI != EPI_PLAIN;
  PassParams<float> p{};
  p.in_re = q_global<const float>(tk.src);
  p.out_re = q_global<float>(tk.dst);
  p.in_js = 1;
  p.out_ks = 1;
  p.n_col = 1;
  p.col_tiles = 1;
  p.n_blo = 1;
  p.in_il = p.out_il = 1;
  p.in_bytes = 8u * (EPI == EPI_C2R ? L + 1 : L);
  p.out_bytes = 8u * (EPI == EPI_R2C ? L + 1 : L);
  // rows of L + 1 bins start off line boundaries: partial lines merge in the L2
  p.in_nt = p.out_nt = !REAL;
  p.swap_in = p.swap_out = EPI == EPI_C2R || tk.kind == afft_gpu_ci;
  p.stage_tw = q_global(q_const(a.tab)->stage[tk.lg]);
  fft_tile<float, L, 1, false, EPI, false, true, SV, true>(p, 0, tid, lds);
}

template <int L, int SV>
__device__ __forceinline__ void q_row_any(const QArgs& a, const QRec& tk, int tid, cx<float>* lds) {
  if (tk.kind == afft_gpu_r)
    q_row<L, SV, EPI_R2C>(a, tk, tid, lds);
  else if (tk.kind == afft_gpu_ri)
    q_row<L, SV, EPI_C2R>(a, tk, tid, lds);
  else
    q_row<L, SV, EPI_PLAIN>(a, tk, tid, lds);
}

// The tasks blockIdx.x, blockIdx.x + gridDim.x, ... of one list, f(task, thread)
// for each.  The next task's record is read while the present one runs: popped
// from a counter, a task began with three dependent reads (counter, record,
// buffer addresses) in front of its first load.
template <typename F>
__device__ __forceinline__ void q_each(const QArgs& a, int list, F&& f) {
  const int off = q_const(a.hdr)->list_off[list];
  const int n = q_const(a.hdr)->list_off[list + 1] - off;
  int i = blockIdx.x;
  if (i >= n) return;
  QRec tk = q_rec(a, off + i);
  for (;;) {
    const int nx = i + gridDim.x;
    const QRec next = q_rec(a, off + (nx < n ? nx : i));
    // the thread id is opaque to the compiler in every turn: the tile bodies'
    // addresses, hoisted out of the loop, held 120 to 200 registers' worth
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    f(tk, tid);
    if (nx >= n) return;
    i = nx;
    tk = next;
    __syncthreads();
  }
}

// 2^15 points: 1024 threads, one group per CU (the half-LDS tile takes 136 KiB).
__global__ void __launch_bounds__(1024, 4) queue_row15_kernel(QArgs a) {
  extern __shared__ __align__(16) unsigned char q_smem[];
  cx<float>* lds = reinterpret_cast<cx<float>*>(q_smem);
  q_each(a, QL_ROW15, [&](const QRec& tk, int tid) AFGPU_INLINE { q_row_any<32768, 0>(a, tk, tid, lds); });
}

// 2^13 and 2^14 points: 512 threads, two groups per CU (68 KiB).
__global__ void __launch_bounds__(512, 4) queue_row14_kernel(QArgs a) {
  extern __shared__ __align__(16) unsigned char q_smem[];
  cx<float>* lds = reinterpret_cast<cx<float>*>(q_smem);
  q_each(a, QL_ROW14, [&](const QRec& tk, int tid) AFGPU_INLINE {
    if (tk.lg == 14)
      q_row_any<16384, 1>(a, tk, tid, lds);
    else
      q_row_any<8192, 0>(a, tk, tid, lds);
  });
}

// ---- 2^16-point complex jobs: 64 x 1024 ----------------------------------------
// The shapes of the batched plan of that length: 64-point columns, 64 per tile
// (512-byte row segments), then 1024-point rows, 8 per tile.
constexpr int kPairN1 = 64, kPairN2 = 1024;
constexpr int kPairCols = 64, kPairRows = 8;

__device__ __forceinline__ PassParams<float> q_pair_params(const QArgs& a, const QRec& tk, int lg_len) {
  PassParams<float> p{};
  p.n_blo = 1;
  p.in_il = p.out_il = 1;
  p.in_bytes = p.out_bytes = 8u << 16;
  p.stage_tw = q_global(q_const(a.tab)->stage[lg_len]);
  return p;
}

__device__ __forceinline__ float* q_pair_scratch(const QArgs& a, int job) {
  return q_global<float>((unsigned long long)(q_const(a.hdr)->pair_scratch + ((idx_t)job << 16)));
}

// Group `group` of the pair list in `ngroups` equal ones: its first task and its
// number of jobs (read from the list, so a captured launch splits whichever list
// is prepared when it is replayed).
__device__ __forceinline__ void q_pair_group(const QArgs& a, int group, int ngroups, int& off, int& n) {
  const int all = q_const(a.hdr)->list_off[QL_PAIR + 1] - q_const(a.hdr)->list_off[QL_PAIR];
  const int per = (all + ngroups - 1) / ngroups;
  off = q_const(a.hdr)->list_off[QL_PAIR] + group * per;
  n = min(per, all - group * per);
}

__global__ void __launch_bounds__((PassShape<kPairN1, kPairCols>::NT)) queue_pair_a_kernel(QArgs a, int group, int ngroups) {
  extern __shared__ __align__(16) unsigned char q_smem[];
  int off, n;
  q_pair_group(a, group, ngroups, off, n);
  constexpr int TILES = kPairN2 / kPairCols;
  for (int i = blockIdx.x; i < n * TILES; i += gridDim.x) {
    const QRec tk = q_rec(a, off + i / TILES);
    PassParams<float> p = q_pair_params(a, tk, 6);
    p.in_re = q_global<const float>(tk.src);
    p.out_re = q_pair_scratch(a, i / TILES);
    p.in_js = p.out_ks = kPairN2;
    p.in_cs = p.out_cs = 1;
    p.n_col = kPairN2;
    p.in_nt = 1;
    p.swap_in = tk.kind == afft_gpu_ci;
    p.tw4_log2n = 16;
    p.col_tiles = TILES;
    fft_tile<float, kPairN1, kPairCols, true, EPI_TW4, false, true>(p, i % TILES, threadIdx.x,
                                                                   reinterpret_cast<cx<float>*>(q_smem));
    __syncthreads();
  }
}

__global__ void __launch_bounds__((PassShape<kPairN2, kPairRows>::NT), 4) queue_pair_b_kernel(QArgs a, int group, int ngroups) {
  extern __shared__ __align__(16) unsigned char q_smem[];
  int off, n;
  q_pair_group(a, group, ngroups, off, n);
  constexpr int TILES = kPairN1 / kPairRows;
  for (int i = blockIdx.x; i < n * TILES; i += gridDim.x) {
    const QRec tk = q_rec(a, off + i / TILES);
    PassParams<float> p = q_pair_params(a, tk, 10);
    p.in_re = q_pair_scratch(a, i / TILES);
    p.out_re = q_global<float>(tk.dst);
    p.in_js = 1;
    p.in_cs = kPairN2;
    p.out_ks = kPairN1;
    p.out_cs = 1;
    p.n_col = kPairN1;
    p.out_nt = 1;
    p.swap_out = tk.kind == afft_gpu_ci;
    p.col_tiles = TILES;
    fft_tile<float, kPairN2, kPairRows, false, EPI_PLAIN, true, true, 0, true>(p, i % TILES, threadIdx.x,
                                                                              reinterpret_cast<cx<float>*>(q_smem));
    __syncthreads();
  }
}

template <auto K, typename... Args>
static hipError_t launch_long(size_t lds, int grid, int threads, hipStream_t st, Args... args) {
  static PerDevice attr;
  if (hipError_t e = allow_lds(attr, (const void*)K, lds); e != hipSuccess) return e;
  hipLaunchKernelGGL(K, dim3(grid), dim3(threads), lds, st, args...);
  return hipGetLastError();
}

hipError_t queue_rows(const QArgs& a, int list, int ncu, hipStream_t st) {
  constexpr size_t l15 = tile_lds_bytes<float, 32768, 1, false, false, 0, true>();
  constexpr size_t l14 = tile_lds_bytes<float, 16384, 1, false, false, 1, true>();
  if (list == QL_ROW15) return launch_long<queue_row15_kernel>(l15, ncu, 1024, st, a);
  return launch_long<queue_row14_kernel>(l14, 2 * ncu, 512, st, a);
}

// Jobs per pass pair: 448 x 512 KiB of scratch, so that pass B still finds most
// of what pass A wrote in the 256 MB Infinity Cache and little of it is written
// back in between.  636 jobs of 2^16: 2 groups 0.230 ms, one 0.311; of 10,000
// mixed jobs: groups of at most 64, 100, 160, 220, 320 jobs and one group 716,
// 676, 668, 629, 629, 664 us; 381 jobs of 6000: 471, 441, 430, 423, 422, 407.
constexpr int kPairGroup = 448;

int queue_pair_groups(int njobs) { return (njobs + kPairGroup - 1) / kPairGroup; }

hipError_t queue_pairs(const QArgs& a, int njobs, hipStream_t st) {
  using SA = PassShape<kPairN1, kPairCols>;
  using SB = PassShape<kPairN2, kPairRows>;
  constexpr size_t la = tile_lds_bytes<float, kPairN1, kPairCols, true, false, 0, false>();
  constexpr size_t lb = tile_lds_bytes<float, kPairN2, kPairRows, false, true, 0, true>();
  const int groups = queue_pair_groups(njobs), per = (njobs + groups - 1) / groups;
  for (int g = 0; g < groups; g++) {
    hipError_t e = launch_long<queue_pair_a_kernel>(la, per * (kPairN2 / kPairCols), SA::NT, st, a, g, groups);
    if (e == hipSuccess)
      e = launch_long<queue_pair_b_kernel>(lb, per * (kPairN1 / kPairRows), SB::NT, st, a, g, groups);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace afgpu
