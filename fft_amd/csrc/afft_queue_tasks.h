// afft_queue_tasks.h -- what the kernels of an uneven batch share: the task
// record, the tables and the lists a prepared queue holds on the device.
#pragma once

#include "../../include/afft_gpu.h"
#include "afft_pass.h"

namespace afgpu {

// (the row and pair kernels go by their lists; a record names its type all the same)
enum { QT_GROUP = 0, QT_RPRE = 1, QT_BIGA = 2, QT_BIGB = 3, QT_RPOST = 4, QT_ROW = 5, QT_PAIR = 6 };
constexpr int kQMaxLog2 = 16;
constexpr int kXcd = 8;   // XCDs of an MI355X: one chain list each
constexpr int kCtr = 16;  // ints between counters (one 64-byte line each)

// Task lists: kXcd chain lists, the shared group list, whole rows of 2^15
// points, whole rows of 2^13 and 2^14 points, 2^16-point pass pairs.
enum { QL_GROUP = kXcd, QL_ROW15 = kXcd + 1, QL_ROW14 = kXcd + 2, QL_PAIR = kXcd + 3, kQLists = kXcd + 4 };

struct QTask {
  int type;
  int lg;     // log2 of the complex length (group: L, chain: m)
  int kind;   // afft_gpu_c / ci / r / ri
  int count;  // group: jobs; chain: index of this step within the job
  int first;  // first (src, dst) pair in the pointer table; a chain's scratch follows
  int job;    // chain: job index (dependency counters)
  int tile;   // chain: tile index within the step
  int need;   // chain: tiles of the previous step to wait for (0: none)

  // rows and pairs: the job's buffers take the place of the last four fields, so
  // a record stays 32 bytes (padded to 48, 610 jobs of 2^7..2^16 take the same:
  // 70.6 us)
  void set_buffers(unsigned long long src, unsigned long long dst) {
    first = (int)(unsigned)src;
    job = (int)(unsigned)(src >> 32);
    tile = (int)(unsigned)dst;
    need = (int)(unsigned)(dst >> 32);
  }
};

struct QTables {
  const cx<float>* stage[kQMaxLog2 + 1];  // stage twiddles of an L-point tile, by log2 L
  const cx<float>* tw4[kQMaxLog2 + 1];    // four-step hi table (lo follows), by log2 m
  const cx<float>* real[kQMaxLog2 + 1];   // W_{2L}^k, by log2 L
};

// Written by prepare, read by every launch: a launch (or a replay of a captured
// one) runs the task list of the latest prepare.
struct QListHdr {
  int list_off[kQLists + 1];
  int ndeps;  // step counters to clear (4 per chain job)
  cx<float>* pair_scratch;  // 2^16 entries per job of a pair group
};

struct QArgs {
  const QTask* tasks;  // the lists, one after the other
  const unsigned long long* ptrs;
  int* counter;        // list l pops through counter[l * kCtr]
  const QListHdr* hdr;
  int* deps;       // 4 step counters per chain job
  int* status;     // set to 1 when a dependency wait hits the spin limit
  long long spin_limit;
  const QTables* tab;  // device copy: indexed by log2 length at run time
};

// A pointer read from device memory, as what it is: an address in global
// memory (without the cast the compiler emits flat accesses, which count as LDS
// operations as well).
template <typename X>
__device__ __forceinline__ X* q_global(unsigned long long a) {
  return (X*)(__attribute__((address_space(1))) X*)a;
}
template <typename X>
__device__ __forceinline__ X* q_global(X* p) {
  return q_global<X>((unsigned long long)p);
}
// Reads that no kernel of a launch writes (lists, records, tables): scalar
// loads, so the values are the same in every lane by construction (a buffer
// resource made from an address that could differ costs a loop per access).
template <typename X>
using QConst = __attribute__((address_space(4))) const X*;
template <typename X>
__device__ __forceinline__ QConst<X> q_const(const X* p) {
  return (QConst<X>)(unsigned long long)p;
}

// afft_queue_long.hip: the jobs longer than a group tile, without waits
// between work-groups (each launch follows the previous one on the stream).
hipError_t queue_rows(const QArgs& a, int list, int ncu, hipStream_t st);
// Pass pairs in queue_pair_groups(njobs) groups, njobs = those prepared now.
int queue_pair_groups(int njobs);
hipError_t queue_pairs(const QArgs& a, int njobs, hipStream_t st);

}  // namespace afgpu
