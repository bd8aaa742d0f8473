// What the launches that keep several rounds resident share: the barrier of a group of workgroups on
// one XCD, the row reads behind it, and the reduction of the four-row tiles' accumulators.
#ifndef CAVS_CSRC_ROUND_SYNC_H_
#define CAVS_CSRC_ROUND_SYNC_H_

#include "round_common.h"

namespace cavs {

// The sync block: word 1 = status (all groups); group g owns the 128 words from 128 (g + 1): how often each
// of its workgroups has arrived (a word each), then the XCDs they saw (bit mask) and how many have left.
constexpr int kSyncGroups = 128;  // groups a sync block has room for (H = 32: two workgroups each, one to a CU)
enum { TAIL_STATUS = 1, TAIL_GROUP_WORDS = 128, TAIL_FLAGS = 0, TAIL_XCC = 64, TAIL_LEFT = 65 };

__device__ inline int xcc_id() { return __builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11)) & 15; }  // HW_REG_XCC_ID[3:0]

// The barrier of a group.  A workgroup arrives by an ordinary store to a word of its own, which like its
// rows is in the XCD's L2 once acknowledged; every wavefront waits by itself, with one load over all the
// words (agent scope: past the L1).  On 8, 16 and 32 workgroups of one XCD, a store before and a load
// after included, 0.66, 0.67 and 0.69 us a round; with one counter added to atomically and polled by one
// thread 1.05, 1.03 and 1.25, with words stored at agent scope 0.96, 1.14 and 1.30, with a word per
// wavefront 0.87, 1.18 and 1.65.

// This workgroup's results of a round are written: tell the others of the group.
__device__ inline void tail_arrive(unsigned *gsync, int wg, unsigned arrivals) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's stores are acknowledged by the L2
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(gsync + TAIL_FLAGS + wg, arrivals, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The words of the group's first `expect` (at most 64) workgroups, a lane's each (the others': as if there): asked for here,
// looked at by who has done something else in between.
__device__ inline unsigned tail_ask(const unsigned *gsync, int expect) {
  const int lane = threadIdx.x & 63;
  const unsigned v = __hip_atomic_load(gsync + TAIL_FLAGS + (lane < expect ? lane : 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return lane < expect ? v : ~0u;
}

// Waits until the group's first `expect` (at most 64) workgroups have arrived `target` times; no barrier of the
// workgroup.  Where the wait gives up (spin_max polls, or another workgroup already did, or the group's
// workgroups turned out to sit on more than one XCD: the status word says why) *s_bail is set, and the
// workgroup leaves behind its next barrier.  `whole_lines`: see ld_row.
__device__ inline void tail_wait(unsigned *status, unsigned *gsync, unsigned target, int expect, int spin_max, bool check_xcc, bool whole_lines,
                                 int *s_bail) {
  const int lane = threadIdx.x & 63;
  unsigned why = 0;
  bool in = false;
  for (int tries = 1; !in && !why; tries++) {
    const unsigned v = lane < expect ? __hip_atomic_load(gsync + TAIL_FLAGS + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : target;
    in = __all(v >= target);
    if (!in && tries > spin_max) why = CAVS_TAIL_TIMEOUT;
    if (!in && !why && (tries & 15) == 0) why = __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (check_xcc && !why && (in || (tries & 15) == 0)) {
      const unsigned seen = __hip_atomic_load(gsync + TAIL_XCC, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (seen & (seen - 1)) why = CAVS_TAIL_SPREAD;  // the L2 is not shared: nothing read here can be trusted
    }
  }
  if (why && lane == 0) {
    __hip_atomic_store(status, why, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *s_bail = 1;
  }
  if (!whole_lines) asm volatile("buffer_inv sc1" ::: "memory");
  asm volatile("" ::: "memory");  // (what the others wrote is read after this)
}

// This workgroup waits no more (behind a barrier of its own).  The last of the group's `wgs` to say so leaves
// the group's words as the next launch expects them: zero.  So a workgroup's own arrivals, stored by its first
// wavefront (the last list arrives too), have to be in the L2 before it counts as gone -- one still under way
// then would land on top of the zero, and the next launch's waits would pass early.  Stores and atomics of
// a wavefront are not ordered by themselves: the wait (once a launch) does it.
__device__ inline void tail_leave(unsigned *gsync, int wgs) {
  if (threadIdx.x >= 64) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  unsigned old = 0;
  if (threadIdx.x == 0) old = __hip_atomic_fetch_add(gsync + TAIL_LEFT, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (__builtin_amdgcn_readfirstlane(old) + 1 != (unsigned)wgs) return;
  __hip_atomic_store(gsync + TAIL_FLAGS + threadIdx.x, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (threadIdx.x < 2) __hip_atomic_store(gsync + TAIL_XCC + threadIdx.x, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A row another workgroup of the group wrote in an earlier round, by an ordinary load, which may be served by
// this CU's L1.  A line that is in there is not updated by another CU's store, and what the workgroups share is
// the L2; so no line of such a row may have been loaded before the barrier that follows the row's round:
//   * the L1 starts a kernel empty, and a store does not leave its line in there;
//   * a row is read only behind that barrier: loads for a missing child, which are issued all the same and
//     masked, go to the weights (to row 0 of the pool they could meet a row of this launch);
//   * rows are whole lines of 128 bytes, so that no row's line holds a piece of one written in another round.
//     The launching side looks (whole_lines: pointers and row strides); where they are not, every wait drops
//     the L1's lines (buffer_inv sc1, about 15 us a round for 32 workgroups).
// Measured, a line loaded, stored to by another CU of the XCD, loaded again: the old value by an ordinary load, by
// a load with sc0, and by one behind buffer_inv sc0; the new one behind buffer_inv sc1, by a load with sc1, and
// after a store of one's own to the line.  Loads that bypass the L1 by scope (agent-scope atomic loads) cost
// about sixty cycles per wavefront and access here, one request per lane: three times the MFMA time of a tile.
constexpr int kLineBytes = 128;
inline bool line_rows(const void *p, long ld_floats) { return reinterpret_cast<uintptr_t>(p) % kLineBytes == 0 && ld_floats * 4 % kLineBytes == 0; }
__device__ inline float ld_row(const float *p) { return *p; }

// The four k slots of an element added up across the wavefront, for the four rows of NP products
// at once: afterwards the lanes of k slot s hold, in r[p][0], the sum of row s of product p --
// (v[x] + v[x+16]) + (v[x+32] + v[x+48]) with v = that row's accumulator, the order in which the
// per-round kernels add the slots up.  v_permlane16_swap exchanges the odd 16-lane rows of its first
// operand with the even rows of its second, v_permlane32_swap the upper half of the first with the
// lower half of the second; swapping two rows' accumulators and adding puts both partial sums into
// one register, a butterfly of three swaps and three adds per product on the vector ALU (a shuffle
// through the LDS crossbar costs eight cycles of a unit all eight wavefronts share).  Spelled out
// as instructions, which change both operands where they are, in the order that is wanted between
// other work.  The compiler does not look inside such a statement, so the waits an instruction needs after the
// one that produced its operand are the caller's: all() carries its own (twelve cycles cover the
// six a two-pass MFMA asks for before a vector-ALU read, two between an add and the swap that reads
// it); the stages are for callers that put at least that many instructions between them.
template <int NP>
struct SlotSums;
template <>
struct SlotSums<5> {
  float r[5][4];
  __device__ inline void take(const floatx4 (&acc)[5]) {
#pragma unroll
    for (int p = 0; p < 5; p++)
#pragma unroll
      for (int k = 0; k < 4; k++) r[p][k] = acc[p][k];
  }
  // the stages one at a time, for a caller that puts other work (MFMAs of the next tile) between them
  __device__ inline void stage_a() {
    asm volatile(
        "v_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\t"
        "v_permlane16_swap_b32 %4, %5\n\tv_permlane16_swap_b32 %6, %7\n\t"
        "v_permlane16_swap_b32 %8, %9\n\tv_permlane16_swap_b32 %10, %11\n\t"
        "v_permlane16_swap_b32 %12, %13\n\tv_permlane16_swap_b32 %14, %15\n\t"
        "v_permlane16_swap_b32 %16, %17\n\tv_permlane16_swap_b32 %18, %19"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]), "+v"(r[1][2]), "+v"(r[1][3]), "+v"(r[2][0]), "+v"(r[2][1]), "+v"(r[2][2]), "+v"(r[2][3]), "+v"(r[3][0]), "+v"(r[3][1]), "+v"(r[3][2]), "+v"(r[3][3]), "+v"(r[4][0]), "+v"(r[4][1]), "+v"(r[4][2]), "+v"(r[4][3]));
  }
  __device__ inline void stage_b() {
    asm volatile(
        "v_add_f32 %0, %0, %1\n\tv_add_f32 %2, %2, %3\n\t"
        "v_add_f32 %4, %4, %5\n\tv_add_f32 %6, %6, %7\n\t"
        "v_add_f32 %8, %8, %9\n\tv_add_f32 %10, %10, %11\n\t"
        "v_add_f32 %12, %12, %13\n\tv_add_f32 %14, %14, %15\n\t"
        "v_add_f32 %16, %16, %17\n\tv_add_f32 %18, %18, %19"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]), "+v"(r[1][2]), "+v"(r[1][3]), "+v"(r[2][0]), "+v"(r[2][1]), "+v"(r[2][2]), "+v"(r[2][3]), "+v"(r[3][0]), "+v"(r[3][1]), "+v"(r[3][2]), "+v"(r[3][3]), "+v"(r[4][0]), "+v"(r[4][1]), "+v"(r[4][2]), "+v"(r[4][3]));
  }
  __device__ inline void stage_c() {
    asm volatile(
        "v_permlane32_swap_b32 %0, %2\n\t"
        "v_permlane32_swap_b32 %4, %6\n\t"
        "v_permlane32_swap_b32 %8, %10\n\t"
        "v_permlane32_swap_b32 %12, %14\n\t"
        "v_permlane32_swap_b32 %16, %18"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]), "+v"(r[1][2]), "+v"(r[1][3]), "+v"(r[2][0]), "+v"(r[2][1]), "+v"(r[2][2]), "+v"(r[2][3]), "+v"(r[3][0]), "+v"(r[3][1]), "+v"(r[3][2]), "+v"(r[3][3]), "+v"(r[4][0]), "+v"(r[4][1]), "+v"(r[4][2]), "+v"(r[4][3]));
  }
  __device__ inline void stage_d() {
    asm volatile(
        "v_add_f32 %0, %0, %2\n\t"
        "v_add_f32 %4, %4, %6\n\t"
        "v_add_f32 %8, %8, %10\n\t"
        "v_add_f32 %12, %12, %14\n\t"
        "v_add_f32 %16, %16, %18"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]), "+v"(r[1][2]), "+v"(r[1][3]), "+v"(r[2][0]), "+v"(r[2][1]), "+v"(r[2][2]), "+v"(r[2][3]), "+v"(r[3][0]), "+v"(r[3][1]), "+v"(r[3][2]), "+v"(r[3][3]), "+v"(r[4][0]), "+v"(r[4][1]), "+v"(r[4][2]), "+v"(r[4][3]));
  }
  // all of it at once, right after the MFMAs that produced the accumulators
  __device__ inline void all() {
    asm volatile(
      "s_nop 7\n\ts_nop 3\n\t"
      "v_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\t"
      "v_permlane16_swap_b32 %4, %5\n\tv_permlane16_swap_b32 %6, %7\n\t"
      "v_permlane16_swap_b32 %8, %9\n\tv_permlane16_swap_b32 %10, %11\n\t"
      "v_permlane16_swap_b32 %12, %13\n\tv_permlane16_swap_b32 %14, %15\n\t"
      "v_permlane16_swap_b32 %16, %17\n\tv_permlane16_swap_b32 %18, %19\n\t"
      "s_nop 1\n\t"
      "v_add_f32 %0, %0, %1\n\tv_add_f32 %2, %2, %3\n\t"
      "v_add_f32 %4, %4, %5\n\tv_add_f32 %6, %6, %7\n\t"
      "v_add_f32 %8, %8, %9\n\tv_add_f32 %10, %10, %11\n\t"
      "v_add_f32 %12, %12, %13\n\tv_add_f32 %14, %14, %15\n\t"
      "v_add_f32 %16, %16, %17\n\tv_add_f32 %18, %18, %19\n\t"
      "s_nop 1\n\t"
      "v_permlane32_swap_b32 %0, %2\n\t"
      "v_permlane32_swap_b32 %4, %6\n\t"
      "v_permlane32_swap_b32 %8, %10\n\t"
      "v_permlane32_swap_b32 %12, %14\n\t"
      "v_permlane32_swap_b32 %16, %18\n\t"
      "s_nop 1\n\t"
      "v_add_f32 %0, %0, %2\n\t"
      "v_add_f32 %4, %4, %6\n\t"
      "v_add_f32 %8, %8, %10\n\t"
      "v_add_f32 %12, %12, %14\n\t"
      "v_add_f32 %16, %16, %18"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]), "+v"(r[1][2]), "+v"(r[1][3]), "+v"(r[2][0]), "+v"(r[2][1]), "+v"(r[2][2]), "+v"(r[2][3]), "+v"(r[3][0]), "+v"(r[3][1]), "+v"(r[3][2]), "+v"(r[3][3]), "+v"(r[4][0]), "+v"(r[4][1]), "+v"(r[4][2]), "+v"(r[4][3]));
  }
};
template <>
struct SlotSums<3> {
  float r[3][4];
  __device__ inline void take(const floatx4 (&acc)[3]) {
#pragma unroll
    for (int p = 0; p < 3; p++)
#pragma unroll
      for (int k = 0; k < 4; k++) r[p][k] = acc[p][k];
  }
  // the stages one at a time, for a caller that puts other work (MFMAs of the next tile) between them
  __device__ inline void stage_a() {
    asm volatile(
        "v_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\t"
        "v_permlane16_swap_b32 %4, %5\n\tv_permlane16_swap_b32 %6, %7\n\t"
        "v_permlane16_swap_b32 %8, %9\n\tv_permlane16_swap_b32 %10, %11"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]), "+v"(r[1][2]), "+v"(r[1][3]), "+v"(r[2][0]), "+v"(r[2][1]), "+v"(r[2][2]), "+v"(r[2][3]));
  }
  __device__ inline void stage_b() {
    asm volatile(
        "v_add_f32 %0, %0, %1\n\tv_add_f32 %2, %2, %3\n\t"
        "v_add_f32 %4, %4, %5\n\tv_add_f32 %6, %6, %7\n\t"
        "v_add_f32 %8, %8, %9\n\tv_add_f32 %10, %10, %11"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]), "+v"(r[1][2]), "+v"(r[1][3]), "+v"(r[2][0]), "+v"(r[2][1]), "+v"(r[2][2]), "+v"(r[2][3]));
  }
  __device__ inline void stage_c() {
    asm volatile(
        "v_permlane32_swap_b32 %0, %2\n\t"
        "v_permlane32_swap_b32 %4, %6\n\t"
        "v_permlane32_swap_b32 %8, %10"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]), "+v"(r[1][2]), "+v"(r[1][3]), "+v"(r[2][0]), "+v"(r[2][1]), "+v"(r[2][2]), "+v"(r[2][3]));
  }
  __device__ inline void stage_d() {
    asm volatile(
        "v_add_f32 %0, %0, %2\n\t"
        "v_add_f32 %4, %4, %6\n\t"
        "v_add_f32 %8, %8, %10"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]), "+v"(r[1][2]), "+v"(r[1][3]), "+v"(r[2][0]), "+v"(r[2][1]), "+v"(r[2][2]), "+v"(r[2][3]));
  }
  // all of it at once, right after the MFMAs that produced the accumulators
  __device__ inline void all() {
    asm volatile(
      "s_nop 7\n\ts_nop 3\n\t"
      "v_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\t"
      "v_permlane16_swap_b32 %4, %5\n\tv_permlane16_swap_b32 %6, %7\n\t"
      "v_permlane16_swap_b32 %8, %9\n\tv_permlane16_swap_b32 %10, %11\n\t"
      "s_nop 1\n\t"
      "v_add_f32 %0, %0, %1\n\tv_add_f32 %2, %2, %3\n\t"
      "v_add_f32 %4, %4, %5\n\tv_add_f32 %6, %6, %7\n\t"
      "v_add_f32 %8, %8, %9\n\tv_add_f32 %10, %10, %11\n\t"
      "s_nop 1\n\t"
      "v_permlane32_swap_b32 %0, %2\n\t"
      "v_permlane32_swap_b32 %4, %6\n\t"
      "v_permlane32_swap_b32 %8, %10\n\t"
      "s_nop 1\n\t"
      "v_add_f32 %0, %0, %2\n\t"
      "v_add_f32 %4, %4, %6\n\t"
      "v_add_f32 %8, %8, %10"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]), "+v"(r[1][2]), "+v"(r[1][3]), "+v"(r[2][0]), "+v"(r[2][1]), "+v"(r[2][2]), "+v"(r[2][3]));
  }
};

template <>
struct SlotSums<1> {
  float r[1][4];
  __device__ inline void take(const floatx4 (&acc)[1]) {
#pragma unroll
    for (int p = 0; p < 1; p++)
#pragma unroll
      for (int k = 0; k < 4; k++) r[p][k] = acc[p][k];
  }
  __device__ inline void all() {
    asm volatile(
      "s_nop 7\n\ts_nop 3\n\t"
      "v_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\t"
      "s_nop 1\n\t"
      "v_add_f32 %0, %0, %1\n\tv_add_f32 %2, %2, %3\n\t"
      "s_nop 1\n\t"
      "v_permlane32_swap_b32 %0, %2\n\t"
      "s_nop 1\n\t"
      "v_add_f32 %0, %0, %2"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]));
  }
};
template <>
struct SlotSums<2> {
  float r[2][4];
  __device__ inline void take(const floatx4 (&acc)[2]) {
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int k = 0; k < 4; k++) r[p][k] = acc[p][k];
  }
  __device__ inline void all() {
    asm volatile(
      "s_nop 7\n\ts_nop 3\n\t"
      "v_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\t"
      "v_permlane16_swap_b32 %4, %5\n\tv_permlane16_swap_b32 %6, %7\n\t"
      "s_nop 1\n\t"
      "v_add_f32 %0, %0, %1\n\tv_add_f32 %2, %2, %3\n\t"
      "v_add_f32 %4, %4, %5\n\tv_add_f32 %6, %6, %7\n\t"
      "s_nop 1\n\t"
      "v_permlane32_swap_b32 %0, %2\n\t"
      "v_permlane32_swap_b32 %4, %6\n\t"
      "s_nop 1\n\t"
      "v_add_f32 %0, %0, %2\n\t"
      "v_add_f32 %4, %4, %6"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]), "+v"(r[1][2]), "+v"(r[1][3]));
  }
};
template <>
struct SlotSums<4> {
  float r[4][4];
  __device__ inline void take(const floatx4 (&acc)[4]) {
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
      for (int k = 0; k < 4; k++) r[p][k] = acc[p][k];
  }
  __device__ inline void all() {
    asm volatile(
      "s_nop 7\n\ts_nop 3\n\t"
      "v_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\t"
      "v_permlane16_swap_b32 %4, %5\n\tv_permlane16_swap_b32 %6, %7\n\t"
      "v_permlane16_swap_b32 %8, %9\n\tv_permlane16_swap_b32 %10, %11\n\t"
      "v_permlane16_swap_b32 %12, %13\n\tv_permlane16_swap_b32 %14, %15\n\t"
      "s_nop 1\n\t"
      "v_add_f32 %0, %0, %1\n\tv_add_f32 %2, %2, %3\n\t"
      "v_add_f32 %4, %4, %5\n\tv_add_f32 %6, %6, %7\n\t"
      "v_add_f32 %8, %8, %9\n\tv_add_f32 %10, %10, %11\n\t"
      "v_add_f32 %12, %12, %13\n\tv_add_f32 %14, %14, %15\n\t"
      "s_nop 1\n\t"
      "v_permlane32_swap_b32 %0, %2\n\t"
      "v_permlane32_swap_b32 %4, %6\n\t"
      "v_permlane32_swap_b32 %8, %10\n\t"
      "v_permlane32_swap_b32 %12, %14\n\t"
      "s_nop 1\n\t"
      "v_add_f32 %0, %0, %2\n\t"
      "v_add_f32 %4, %4, %6\n\t"
      "v_add_f32 %8, %8, %10\n\t"
      "v_add_f32 %12, %12, %14"
        : "+v"(r[0][0]), "+v"(r[0][1]), "+v"(r[0][2]), "+v"(r[0][3]), "+v"(r[1][0]), "+v"(r[1][1]), "+v"(r[1][2]), "+v"(r[1][3]), "+v"(r[2][0]), "+v"(r[2][1]), "+v"(r[2][2]), "+v"(r[2][3]), "+v"(r[3][0]), "+v"(r[3][1]), "+v"(r[3][2]), "+v"(r[3][3]));
  }
};

// One k-group of four-row tiles is four MFMAs of sixteen 4 x 4 x 1 blocks each; block l / 4 of
// lane l is (column group (l / 4) % 4, k slot l / 16).  An MFMA can take its A operand, for the four
// blocks of a k slot, from one of them (A broadcast inside groups of four blocks: CBSZ = 2, ABID =
// which).  So lane l = 16 slot + 4 j + r fetches ONE float4 per operand row and tile: tile row r at
// k = 16 j + 4 slot .. + 3 of the wavefront's 64 k -- the wavefront's 64 float4 are the whole
// 4 x 64 piece of the operand, nothing is fetched twice and nothing crosses lanes -- and the MFMA
// of k-group g, step c reads component c with ABID = g: the operands the per-round kernels feed the
// same MFMAs after moving them across lanes.
#define CAVS_MMA4(acc, a, b, abid) acc = __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, acc, 2, abid, 0)

// k-group ABID of an operand fetched that way
template <int ABID>
__device__ inline floatx4 mma4(float a, float b, floatx4 acc) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, acc, 2, ABID, 0);
}

}  // namespace cavs
#endif
