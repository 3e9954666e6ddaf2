// Fused-part path of libhsv: one part's gates multiplied into a dense
// 2^k x 2^k FP64 unitary on the host, applied to the state as a batched
// complex GEMM on the gfx950 matrix cores.
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "gates.hpp"

namespace hsv {

// Scratch device buffer owned by the caller's handle (grown on demand).
struct DeviceScratch {
  void* ptr = nullptr;
  size_t bytes = 0;
  // a buffer the library does not own (the no-allocation entry point's
  // static array): never freed or grown; a larger need is an error
  bool fixed = false;
};

// Launch choices of the BF16-split kernels.
struct BfTune {
  int variant = 2;   // parts of 5..7 qubits: 0 / 1 column-block kernel (1: four
                     // consecutive rows per column in each load), 2 tile kernel
  int tile_tpw = 8;  // tiles of 4096 amplitudes per workgroup, tile kernel
  int tile_order = 4;  // tile kernels: m = the highest m slots outside the tile
                       // vary fastest across workgroups, 0 = natural order
  int part_tpw = 0;  // tiles per workgroup, wide-part kernel (8..14 qubits);
                     // 0: 8 where the step fragments stay in LDS (the next
                     // tile is prefetched during the steps), else 1
  int part13 = 0;    // 13-qubit tiles: 0 = 512 threads, fragments streamed
                     // through LDS, two workgroups per CU; 1 = 1024 threads,
                     // fragments resident, next tile prefetched (when the
                     // steps fit); 2 = as 0, each wave reading the fragments
                     // from L2 straight into registers
};

// Applies the fused unitary of `gates` to the n-qubit state at `amp`
// (dtype HSV_C128 or HSV_C64) on `stream`. mode: hsv_fused_mode.
// `num_cu` sizes the persistent grids of the FP64 / FP32-split kernels.
// live: as in fused_part_launch. pinned: host memory through which a wide BF16
// part is prepared on the device, or null. Returns 0 or a negative
// hsv_status.
int fused_apply(void* amp, int n, int dtype, hipStream_t stream, int num_cu, DeviceScratch* scratch,
                const std::vector<Lowered>& gates, int mode, uint64_t live, std::string* err,
                const BfTune& bf = BfTune(), void* pinned = nullptr, size_t pinned_bytes = 0);

// One part on the BF16-split wide-part kernel (a 12- to 14-qubit tile that
// holds slots 0-4), laid out for its launch.
struct FusedPart {
  struct Step {
    int rbit[5], cbit[9];  // the tile bits of its matrix' index, and the others
    std::vector<cd> U;     // 32 x 32
  };
  int KT = 0;
  uint64_t tmask = 0;
  int slot[14], sslot[14];  // of tile bit j, as loaded and as stored
  bool moves = false, nothing = false;
  std::vector<Step> steps;
  // from fused_parts_check: max |U^H U - I| of each step, the LDS swizzle and
  // the place of the steps' fragments in the scratch (after the tables)
  bool checked = false;
  std::vector<double> uerr;
  uint32_t nimg[14];
  size_t frag_off = 0;
};

// Lays out a part with a qubit layout change: logical qubit q sits in slot
// phys[q] and the pass leaves it in slot phys_after[q]; only qubits of the
// tile may move. tile_qubits: the logical qubits the tile must hold (at
// least those of the gates). pieces: BF16 pieces per value, 2
// (HSV_FUSED_BF16SPLIT) or 3 (HSV_FUSED_BF16X3, 12- and 13-qubit tiles).
// groups: the part's steps (gate indices, identities left out) from
// fused_plan_steps; null or empty: searched here.
int fused_part_prepare(int n, const std::vector<Lowered>& gates, uint64_t tile_qubits, const int* phys,
                       const int* phys_after, int pieces, const std::vector<std::vector<int>>* groups, FusedPart* part,
                       std::string* err);

// Checks the steps of the first parts of a list, swizzles their tables and
// lays out their matrices as fragments, on the device, as many parts as host
// (pinned memory that the kernels write) takes; the parts that are not marked
// checked afterwards go through the same on the host in fused_part_launch.
// The fragments stay in the scratch until it is used for anything else.
int fused_parts_check(hipStream_t stream, DeviceScratch* scratch, void* host, size_t host_bytes, FusedPart* parts,
                      int count, int pieces, std::string* err);

// Runs a part. live_slots: slots whose bit can be 1 in a nonzero amplitude
// (the others hold |0> on the whole state, so tiles with such a bit set are
// zero and are skipped); ~0 when nothing is known.
int fused_part_launch(void* amp, int n, int dtype, hipStream_t stream, DeviceScratch* scratch, const FusedPart& part,
                      uint64_t live_slots, const BfTune& bf, int pieces, std::string* err);

// fused_part_prepare and fused_part_launch, for a single part.
int fused_part_bf_layout(void* amp, int n, int dtype, hipStream_t stream, DeviceScratch* scratch,
                         const std::vector<Lowered>& gates, uint64_t tile_qubits, const int* phys,
                         const int* phys_after, uint64_t live_slots, const BfTune& bf, std::string* err,
                         int pieces = 2);

// The step groups of several wide parts at once, searched on the device with
// the choices of step_groups (partition.hpp, width 16): masks[p][i] = the
// tile bits of part p's i-th gate (0: an identity, in no group). (*groups)[p]
// stays empty where the host's own search is to run: parts too large for the
// kernels, gates on more than k qubits, too little work in all to be worth a
// launch. host: pinned memory that the kernel reads and writes.
int fused_plan_steps(hipStream_t stream, DeviceScratch* scratch, void* host, size_t host_bytes,
                     const std::vector<std::vector<uint64_t>>& masks, int k,
                     std::vector<std::vector<std::vector<int>>>* groups, std::string* err);

// The fused unitary itself (for tests and the cost model): qubits of the
// part (sorted, padded with the lowest free qubits to at least min_qubits)
// and the row-major matrix.
int fused_unitary(int n, const std::vector<Lowered>& gates, std::vector<int>* qubits, std::vector<cd>* U,
                  std::string* err, int min_qubits = 4);

}  // namespace hsv
