// Batched QAOA MaxCut on one MI355X: many instances of uneven qubit counts,
// complex64 states, FP64 expectation values, one hipGraph per batch.
//
// Circuit per instance (n qubits, graph E, p layers): H on every qubit, then
// per layer ZZ(gamma) on every edge -- exp(-i gamma/2 Z_u Z_v), the reference's
// RZZ (basic_gates.hpp:1249-1252) -- and RX(2 beta) on every qubit; output
// <C> with C = sum_edges (1 - Z_u Z_v) / 2.
//
// Schedule. A layer is the diagonal D_l = prod_edges ZZ (looked up by the cut
// size: exp(-i gamma/2 (|E| - 2 cut(x)))), then RX(2 beta) on every qubit. An
// instance of n <= L qubits runs whole in one chunk of LDS. A wider one takes
// p + 1 passes over its state, each on chunks of up to 2^13 amplitudes:
//  * even passes ("low"): contiguous chunks over the L low qubits;
//  * odd passes ("high"): chunks over the n - L high qubits and some of the
//    lowest ones.
// D_l needs RX of layer l - 1 done on every qubit, but can be applied in any
// chunk, and RX on different qubits commute. So pass k finishes layer k - 1 on
// its own half of the qubits (the pass before did the other half), applies
// D_k, and starts layer k on its half: one pass per layer where a pass per
// half and layer would take two. Pass 0 makes the state of the H layer itself
// (nothing is read), and the last pass sums |a_x|^2 cut(x) of what it stores.
// RX(2b) = f M, M = [[1, -it], [-it, 1]], with f = cos b and t = tan b where
// |cos b| >= |sin b|, else f = -i sin b and t = -cot b and an X on the qubit:
// M takes one FMA per component, and f^n of layer l is part of D_l's table. The
// X of a layer act on all qubits at once, which no cut size sees: they are
// left out, and where their number is odd the last two passes put the state
// back in order, each on its half's bits (in the addresses of pass p - 1's
// stores and of pass p's loads).
// cut(x) is a per-instance table over a chunk's bits plus, for the edges that
// leave the chunk, a constant and a weight per bit, all worked out on the host
// (they depend on the graphs alone). The stage kernels are persistent over the
// flattened (instance, chunk) items of a pass. The sequence is captured once
// into a hipGraph; angles are read from device memory, so new parameters need
// no re-capture.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/hsv.h"

// Shared with hsv.hip so that hsv_last_error() reports QAOA failures too.
void hsv_set_last_error(const std::string& msg);

namespace {

int qfail(int code, const std::string& m) {
  hsv_set_last_error(m);
  return code;
}
#define QCHK(expr)                                                                     \
  do {                                                                                 \
    hipError_t e_ = (expr);                                                            \
    if (e_ != hipSuccess) return qfail(HSV_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

constexpr int kMaxEdges = 64;
constexpr int kMaxQaoaQubits = 26;
// High chunks hold an instance's hb = n - L high qubits and its lowest
// low_contig(hb, L, threads) qubits (contiguous runs of 2^that amplitudes): 16
// amplitudes a thread, kStageBBits qubits in all at most, at least kLowContig
// low ones (64-byte runs). Fewer threads take smaller chunks, not longer loops,
// so that a small batch has more of them to run at once: 16 instances of 20
// qubits in 256 threads 503 -> 337 us, 8 of 12 to 14 qubits 135 -> 116 (128
// threads 211 -> 161); a batch that fills the chip, 512 of 12 to 22 qubits,
// 14.8 -> 15.0 ms for the shorter runs.
constexpr int kLowContig = 3;
constexpr int kStageBBits = 13;
inline int low_contig(int hb, int L, int threads) {
  int bits = 4;
  while ((1 << (bits - 4)) < threads) ++bits;
  return std::min(std::max(std::min(kStageBBits, bits) - hb, kLowContig), L);
}

struct alignas(8) cf { float x, y; };

// A layer's table: entry c = f^n exp(-i gamma/2 (|E| - 2c)), c = 0..|E|; in
// entry kRxEntry (t, whether the instance's number of X layers is odd).
constexpr int kRxEntry = kMaxEdges + 1;
constexpr int kPhaseRow = kMaxEdges + 2;

struct Inst {
  uint64_t off;        // first amplitude in the batch buffer
  uint64_t tab[2];     // cut tables of its low and high chunks
  int n;               // qubits
  int ne;              // edges
  int edge_off;        // first edge in the (host) edge arrays
  int p;               // layers
  int angle_off;       // first angle in gamma/beta, first row of the phase tables
  int part_off;        // first cost partial
  int parts;           // cost partials: the chunks of its last pass
  int bits[2];         // qubits in a low / high chunk
  int lc;              // lowest qubits in a high chunk
};

// One chunk of one instance: its first amplitude and what cut(x) adds to the
// chunk's table, per chunk bit (w[0..12]) and in all (w[13]).
struct Item {
  uint64_t off;
  uint32_t inst;
  uint32_t part;       // its cost partial (last pass)
  int8_t w[16];
};

// LDS position of chunk element i: bits 0-2 XOR bits 5-7 and bits 3-4 XOR
// bits 6-7, so that the 64 lanes of a wave reading 8-byte elements spread
// over all bank pairs, for consecutive elements as for the three-bit
// register groups of rx_block (a bijection on [0, 2^bits) for any bits).
__device__ __forceinline__ uint32_t qsw(uint32_t i) { return i ^ ((i >> 5) & 7u) ^ (((i >> 6) & 3u) << 3); }

// M on a pair.
__device__ __forceinline__ void rx_pair(cf& a, cf& b, float t) {
  const float ax = a.x, ay = a.y, bx = b.x, by = b.y;
  a.x = fmaf(t, by, ax);
  a.y = fmaf(-t, bx, ay);
  b.x = fmaf(t, ay, bx);
  b.y = fmaf(-t, ax, by);
}

// M on LDS bit q of a 2^bits block, one pair per thread and step.
__device__ __forceinline__ void rx_lds(cf* s, int bits, int q, float t, int nt) {
  const uint32_t half = 1u << (bits - 1);
  for (uint32_t w = threadIdx.x; w < half; w += nt) {
    const uint32_t lo = w & ((1u << q) - 1);
    const uint32_t i0 = ((w ^ lo) << 1) | lo;
    const uint32_t i1 = i0 | (1u << q);
    cf a = s[qsw(i0)], b = s[qsw(i1)];
    rx_pair(a, b, t);
    s[qsw(i0)] = a;
    s[qsw(i1)] = b;
  }
}

template <int S, int NV>
__device__ __forceinline__ void rx_regs(cf* v, float t) {
#pragma unroll
  for (int r = 0; r < NV; ++r)
    if (!(r & S)) rx_pair(v[r], v[r + S], t);
}

// M on bits [from, bits) of a 2^bits LDS block, three bits per sweep: each
// thread takes the 8 elements of three consecutive bits q0..q0+2 into
// registers, applies M on those of them not done yet and writes them back;
// one barrier per sweep (the block must be in LDS, after a barrier, on entry).
template <int NT>
__device__ __forceinline__ void rx_block(cf* s, int bits, int from, float t) {
  if (bits < 3) {
    for (int q = from; q < bits; ++q) {
      rx_lds(s, bits, q, t, NT);
      __syncthreads();
    }
    return;
  }
  for (int done = from; done < bits;) {
    const int q0 = done < bits - 3 ? done : bits - 3;
    const int first = done - q0;  // 0..2: register bits below it are done
    const uint32_t nw = 1u << (bits - 3);
    for (uint32_t w = threadIdx.x; w < nw; w += NT) {
      const uint32_t lo = w & ((1u << q0) - 1);
      const uint32_t base = ((w ^ lo) << 3) | lo;
      cf v[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) v[r] = s[qsw(base + ((uint32_t)r << q0))];
      if (first == 0) rx_regs<1, 8>(v, t);
      if (first <= 1) rx_regs<2, 8>(v, t);
      rx_regs<4, 8>(v, t);
#pragma unroll
      for (int r = 0; r < 8; ++r) s[qsw(base + ((uint32_t)r << q0))] = v[r];
    }
    __syncthreads();
    done = q0 + 3;
  }
}

// ---- 13-qubit chunks of 512 threads ------------------------------------------
// The chunk lives in registers, 16 amplitudes per thread, and changes layout
// through LDS: which four chunk bits a thread's registers span. A: bits 9-12
// (what a coalesced load or store leaves), B: bits 8-11, C: 0-3, D: 4-7. RX on
// a layout's four bits is register arithmetic; from A, through C and D, to B
// covers all 13 (bit 8 in B) with three writes and three reads of the chunk.
// The swizzle puts the 32 lanes of a half-wave in distinct bank pairs in every
// layout: bits 5-7 onto 0-2 and bit 8 onto 3 and 4.
__device__ __forceinline__ uint32_t sw13(uint32_t j) { return j ^ ((j >> 5) & 7u) ^ ((j >> 8 & 1u) * 24u); }

enum { LAY_A = 9, LAY_B = 8, LAY_C = 0, LAY_D = 4 };  // a layout's lowest register bit
template <int LAY>
__device__ __forceinline__ uint32_t lay_thread() {  // the thread's chunk bits
  uint32_t t = threadIdx.x;
  asm volatile("" : "+v"(t));  // recomputed at each use: hoisted out of the item loop, the layouts' addresses spill
  return (t & ((1u << LAY) - 1)) | ((t >> LAY) << (LAY + 4));
}
// LDS position of register r from its base: in A and B the register bits are
// no swizzled ones (but bit 8, which moves 3 and 4), so they are offsets.
template <int LAY>
__device__ __forceinline__ uint32_t lay_pos(uint32_t b, int r) {
  if constexpr (LAY == LAY_A) return b + ((uint32_t)r << 9);
  if constexpr (LAY == LAY_B) return (r & 1 ? b ^ 24u : b) + ((uint32_t)r << 8);
  return b ^ sw13((uint32_t)r << LAY);
}
template <int LAY>
__device__ __forceinline__ void lay_write(cf* s, const cf* v) {
  const uint32_t b = sw13(lay_thread<LAY>());
#pragma unroll
  for (int r = 0; r < 16; ++r) s[lay_pos<LAY>(b, r)] = v[r];
}
template <int LAY>
__device__ __forceinline__ void lay_read(const cf* s, cf* v) {
  const uint32_t b = sw13(lay_thread<LAY>());
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = s[lay_pos<LAY>(b, r)];
}
// M on the layout's bits from `from` up (t = 0 is the identity, without a branch)
template <int LAY>
__device__ __forceinline__ void lay_rx(cf* v, int from, float t) {
  rx_regs<1, 16>(v, from <= LAY ? t : 0.0f);
  rx_regs<2, 16>(v, from <= LAY + 1 ? t : 0.0f);
  rx_regs<4, 16>(v, from <= LAY + 2 ? t : 0.0f);
  rx_regs<8, 16>(v, from <= LAY + 3 ? t : 0.0f);
}
// the chunk in LDS (after its writes, before a barrier): M on the bits of C
// and D from `from` up; ends on a barrier
__device__ __forceinline__ void sweep_cd(cf* s, int from, float t) {
  __syncthreads();
  cf v[16];
  if (from < 4) {
    lay_read<LAY_C>(s, v);
    lay_rx<LAY_C>(v, from, t);
    lay_write<LAY_C>(s, v);
    __syncthreads();
  }
  if (from < 8) {
    lay_read<LAY_D>(s, v);
    lay_rx<LAY_D>(v, from, t);
    lay_write<LAY_D>(s, v);
    __syncthreads();
  }
}

// cut(x) of the thread's 16 amplitudes in a layout: the chunk table's bytes
// (stored thread by thread, 16 per thread) plus the item's weights, the
// thread's bits summed once and the register bits' sums uniform.
template <int LAY>
__device__ __forceinline__ int lay_cut_thread(const Item& I) {
  const uint32_t t = lay_thread<LAY>();
  int base = I.w[13];
#pragma unroll
  for (int b = 0; b < 13; ++b)
    if (b < LAY || b >= LAY + 4) base += -(int)(t >> b & 1u) & I.w[b];
  return base;
}
template <int LAY>
__device__ __forceinline__ int lay_cut(const Item& I, const uint4& tab, int base, int r) {
  int u = 0;  // uniform
#pragma unroll
  for (int b = 0; b < 4; ++b)
    if (r >> b & 1) u += I.w[LAY + b];
  const uint32_t word = r < 4 ? tab.x : r < 8 ? tab.y : r < 12 ? tab.z : tab.w;
  return (int)(word >> (8 * (r & 3)) & 0xffu) + base + u;
}
template <int LAY>
__device__ __forceinline__ void lay_phase(const Item& I, const uint4& tab, const float2* ph, cf* v) {
  const int base = lay_cut_thread<LAY>(I);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const float2 p = ph[lay_cut<LAY>(I, tab, base, r)];
    const float x = v[r].x, y = v[r].y;
    v[r].x = x * p.x - y * p.y;
    v[r].y = x * p.y + y * p.x;
  }
}
template <int LAY>
__device__ __forceinline__ double lay_cost(const Item& I, const uint4& tab, const cf* v) {
  const int base = lay_cut_thread<LAY>(I);
  double acc = 0.0;
#pragma unroll
  for (int r = 0; r < 16; ++r)
    acc += ((double)v[r].x * v[r].x + (double)v[r].y * v[r].y) * lay_cut<LAY>(I, tab, base, r);
  return acc;
}
// element j of a chunk lies at off + (j & (2^lc - 1)) + (j >> lc) 2^L (low
// chunks: lc = L)
__device__ __forceinline__ uint64_t chunk_at(uint32_t j, int lc, int L) {
  return (j & ((1u << lc) - 1)) + ((uint64_t)(j >> lc) << L);
}
template <int LAY>
__device__ __forceinline__ void lay_load(const cf* st, int lc, int L, uint32_t flip, cf* v) {
  const cf* p = st + chunk_at(lay_thread<LAY>() ^ (flip & ~(15u << LAY)), lc, L);
#pragma unroll
  for (int r = 0; r < 16; ++r) {  // the register bits' offset is uniform
    const cf* q = p + chunk_at((uint32_t)r << LAY ^ (flip & 15u << LAY), lc, L);
    v[r].x = q->x;
    v[r].y = q->y;
  }
}
template <int LAY>
__device__ __forceinline__ void lay_store(cf* st, int lc, int L, uint32_t flip, const cf* v) {
  cf* p = st + chunk_at(lay_thread<LAY>() ^ (flip & ~(15u << LAY)), lc, L);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    cf* q = p + chunk_at((uint32_t)r << LAY ^ (flip & 15u << LAY), lc, L);
    q->x = v[r].x;
    q->y = v[r].y;
  }
}

// sum of a double over the workgroup, at thread 0 (red: one per wave)
template <int NT>
__device__ __forceinline__ double block_sum(double x, double* red) {
  for (int m = 32; m >= 1; m >>= 1) x += __shfl_xor(x, m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0)
    for (int i = 0; i < NT / 64; ++i) t += red[i];
  return t;
}

// Pass k of every instance with p >= k (see the schedule above).
// Bound by the RX arithmetic and the exchanges between register layouts, then
// by HBM: 16 amplitudes a thread and their table offsets take the 128 registers
// of two workgroups a CU (12 spilled at 512 threads). 256 instances of 12 to 22 qubits, p up to 4: 0.51 ms a
// pass, 2.52 ms in all; with a pass per layer and half, one for the initial
// state and one for the cost it was 6.68. 512 instances: 11.1 -> 3.9 ms, flat
// from 2 to 32 workgroups a CU.
template <int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_qaoa_pass(
    cf* __restrict__ st, const Inst* __restrict__ inst, const Item* __restrict__ items, uint32_t nitems, int k, int L,
    const float2* __restrict__ phase, const unsigned char* __restrict__ tabs, double* __restrict__ part) {
  extern __shared__ __align__(16) unsigned char smem[];
  cf* s = reinterpret_cast<cf*>(smem);
  __shared__ float2 ph[kPhaseRow];
  __shared__ int sd[14];
  __shared__ short T1[64], T2[128];
  __shared__ double red[NT / 64];
  const int high = k & 1;
  for (uint32_t it = blockIdx.x; it < nitems; it += gridDim.x) {
    const Item& I = items[it];
    const Inst& Q = inst[I.inst];
    const int bits = Q.bits[high], from = high ? Q.lc : 0, lc = high ? Q.lc : L;
    const bool whole = Q.n <= L, last = whole || k == Q.p;
    const float2* row = phase + (size_t)(Q.angle_off + k) * kPhaseRow;  // layer k's table; k - 1's one row before
    const unsigned char* tab = tabs + Q.tab[high];
    const float amp = (float)(1.0 / std::sqrt((double)(1ull << Q.n)));
    cf* chunk = st + I.off;
    // the X layers' order, put right on this half's bits
    const uint32_t own = (1u << bits) - (1u << from);
    uint32_t flip_in = 0, flip_out = 0;
    if (Q.p > 0 && (whole || k + 1 >= Q.p)) {
      const uint32_t f = phase[(size_t)Q.angle_off * kPhaseRow + kRxEntry].y != 0.0f ? own : 0;
      if (whole || k + 1 == Q.p) flip_out = f;
      else flip_in = f;
    }
    double acc = 0.0;
    if (NT == 512 && bits == 13) {
      const uint4 tb = reinterpret_cast<const uint4*>(tab)[threadIdx.x];
      cf v[16];
      if (k > 0) lay_load<LAY_A>(chunk, lc, L, flip_in, v);
      __syncthreads();  // the previous item's reads of LDS are done
      if (k < Q.p)
        for (int i = threadIdx.x; i <= kRxEntry; i += NT) ph[i] = row[i];
      // layer k - 1 on this half, which leaves layout B (A when only bits 9-12 are its)
      if (k > 0) {
        const float t = row[kRxEntry - kPhaseRow].x;
        lay_rx<LAY_A>(v, from, t);
        if (from <= 8) {
          lay_write<LAY_A>(s, v);
          sweep_cd(s, from, t);
          lay_read<LAY_B>(s, v);
          rx_regs<1, 16>(v, t);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          v[r].x = amp;
          v[r].y = 0.0f;
        }
      }
      __syncthreads();  // ph
      if (from > 8) {
        if (k < Q.p) {
          lay_phase<LAY_A>(I, tb, ph, v);
          lay_rx<LAY_A>(v, from, ph[kRxEntry].x);
        } else {
          acc = lay_cost<LAY_A>(I, tb, v);
        }
        lay_store<LAY_A>(chunk, lc, L, flip_out, v);
      } else {
        for (int l = k; l < Q.p; ++l) {
          const float t = ph[kRxEntry].x;
          lay_phase<LAY_B>(I, tb, ph, v);
          lay_rx<LAY_B>(v, from, t);
          __syncthreads();  // every thread has read its layout, and ph
          lay_write<LAY_B>(s, v);
          sweep_cd(s, from, t);
          lay_read<LAY_A>(s, v);
          rx_regs<8, 16>(v, t);
          if (!whole) break;
          // a whole instance: on to its next layer, or to the cost
          __syncthreads();
          lay_write<LAY_A>(s, v);
          for (int i = threadIdx.x; l + 1 < Q.p && i <= kRxEntry; i += NT)
            ph[i] = row[(size_t)(l + 1 - k) * kPhaseRow + i];
          __syncthreads();
          lay_read<LAY_B>(s, v);
        }
        if (last) {
          acc = lay_cost<LAY_B>(I, tb, v);
          lay_store<LAY_B>(chunk, lc, L, flip_out, v);
        } else {
          lay_store<LAY_A>(chunk, lc, L, flip_out, v);
        }
      }
    } else {
      const uint32_t sz = 1u << bits;
      __syncthreads();
      if (threadIdx.x < 14) sd[threadIdx.x] = I.w[threadIdx.x];
      for (uint32_t j = threadIdx.x; j < sz; j += NT) {
        cf a;
        a.x = amp;
        a.y = 0.0f;
        if (k > 0) a = chunk[chunk_at(j ^ flip_in, lc, L)];
        s[qsw(j)] = a;
      }
      __syncthreads();
      for (int t = threadIdx.x; t < 64 + 128; t += NT) {
        const int i = t < 64 ? t : (t - 64) << 6;  // T1: bits 0-5, T2: bits 6-12 and the constant
        int w = t < 64 ? 0 : sd[13];
        for (int u = 0; u < bits; ++u)
          if (i >> u & 1) w += sd[u];
        if (t < 64) T1[t] = (short)w;
        else T2[t - 64] = (short)w;
      }
      if (k > 0) rx_block<NT>(s, bits, from, row[kRxEntry - kPhaseRow].x);
      for (int l = k; l < Q.p; ++l) {
        __syncthreads();  // the previous layer's reads of ph; T1 and T2
        for (int i = threadIdx.x; i <= kRxEntry; i += NT) ph[i] = row[(size_t)(l - k) * kPhaseRow + i];
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < sz; j += NT) {
          const cf a = s[qsw(j)];
          const float2 p = ph[(int)tab[j] + T1[j & 63] + T2[j >> 6]];
          cf o;
          o.x = a.x * p.x - a.y * p.y;
          o.y = a.x * p.y + a.y * p.x;
          s[qsw(j)] = o;
        }
        __syncthreads();
        rx_block<NT>(s, bits, from, ph[kRxEntry].x);
        if (!whole) break;
      }
      __syncthreads();
      for (uint32_t j = threadIdx.x; j < sz; j += NT) {
        const cf a = s[qsw(j)];
        if (last)
          acc += ((double)a.x * a.x + (double)a.y * a.y) * ((int)tab[j] + T1[j & 63] + T2[j >> 6]);
        chunk[chunk_at(j ^ flip_out, lc, L)] = a;
      }
    }
    if (last) {
      __syncthreads();  // red
      acc = block_sum<NT>(acc, red);
      if (threadIdx.x == 0) part[I.part] = acc;
    }
  }
}

// The phase tables of every (instance, layer): one wave each. owner: the
// instance of each angle.
__global__ __launch_bounds__(64) void k_qaoa_tables(const Inst* __restrict__ inst, const uint32_t* __restrict__ owner,
                                                    const double* __restrict__ gamma, const double* __restrict__ beta,
                                                    float2* __restrict__ phase) {
  const Inst Q = inst[owner[blockIdx.x]];
  const double g = gamma[blockIdx.x], b = beta[blockIdx.x];
  const double c = std::cos(b), sn = std::sin(b);
  const bool sw = std::fabs(sn) > std::fabs(c);
  double f = 1.0;  // f^n up to its power of -i
  for (int i = 0; i < Q.n; ++i) f *= sw ? sn : c;
  const int r = sw ? Q.n & 3 : 0;
  float2* row = phase + (size_t)blockIdx.x * kPhaseRow;
  for (int e = threadIdx.x; e <= Q.ne; e += 64) {
    const double a = -0.5 * g * (double)(Q.ne - 2 * e);
    const double ca = std::cos(a), sa = std::sin(a);
    // times (-i)^n
    const double x = r == 0 ? ca : r == 1 ? sa : r == 2 ? -ca : -sa;
    const double y = r == 0 ? sa : r == 1 ? -ca : r == 2 ? -sa : ca;
    row[e] = make_float2((float)(f * x), (float)(f * y));
  }
  int x = 0;  // layers with an X
  for (int l = threadIdx.x; l < Q.p; l += 64) {
    const double bl = beta[Q.angle_off + l];
    x ^= std::fabs(std::sin(bl)) > std::fabs(std::cos(bl));
  }
  for (int m = 32; m >= 1; m >>= 1) x ^= __shfl_xor(x, m);
  if (threadIdx.x == 0) row[kRxEntry] = make_float2((float)(sw ? -c / sn : sn / c), (float)x);
}

// <C> per instance: its partials, one wave in a fixed order
__global__ __launch_bounds__(64) void k_qaoa_sum(const double* __restrict__ part, const Inst* __restrict__ inst,
                                                 double* __restrict__ out) {
  const Inst Q = inst[blockIdx.x];
  double s = 0.0;
  for (int i = threadIdx.x; i < Q.parts; i += 64) s += part[Q.part_off + i];
  for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

}  // namespace

struct hsv_qaoa_batch {
  int num = 0;
  std::vector<Inst> inst;
  std::vector<unsigned char> eu, ev;
  std::vector<int> layers;
  int pmax = 0;
  int total_angles = 0;
  uint64_t total_amps = 0;
  int L = 12;          // low-chunk bits (tuned)
  int nt = 256;        // threads per workgroup (tuned)
  int grid_per_cu = 4; // persistent workgroups per CU (tuned)
  int num_cu = 256;
  hipStream_t stream = nullptr;
  cf* state = nullptr;
  Inst* d_inst = nullptr;
  double *d_gamma = nullptr, *d_beta = nullptr;
  uint32_t* d_owner = nullptr;       // instance of each angle
  float2* d_phase = nullptr;         // kPhaseRow entries per angle
  // the plan of the current shape: low items | high items | cut tables
  void* d_plan = nullptr;
  double* d_part = nullptr;
  double* h_out = nullptr;  // pinned; the last kernel writes it
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  float last_ms = 0;
};

namespace {

void destroy_graph(hsv_qaoa_batch* b) {
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  b->exec = nullptr;
  b->graph = nullptr;
  if (b->d_plan) (void)hipFree(b->d_plan);
  if (b->d_part) (void)hipFree(b->d_part);
  b->d_plan = nullptr;
  b->d_part = nullptr;
}

// Cut sizes over the `bits` chunk bits of the edges with both ends in the
// chunk (pos[v] = chunk bit of vertex v, or -1), built up bit by bit.
void cut_table(const hsv_qaoa_batch* b, const Inst& I, const int* pos, int bits, unsigned char* cut) {
  cut[0] = 0;
  for (int q = 0; q < bits; ++q) {
    const uint32_t h = 1u << q;
    std::memcpy(cut + h, cut, h);
    for (int e = 0; e < I.ne; ++e) {
      const int u = pos[b->eu[I.edge_off + e]], v = pos[b->ev[I.edge_off + e]];
      if (std::max(u, v) != q || std::min(u, v) < 0) continue;
      const int a = std::min(u, v);
      for (uint32_t y = 0; y < h; ++y) {
        const unsigned char ya = (unsigned char)(y >> a & 1u);
        cut[y] += ya;
        cut[h + y] += 1 - ya;
      }
    }
  }
}

// The fast form of k_qaoa_pass reads a chunk's table thread by thread, 16
// bytes each, in the layout it applies the phases in.
bool fast_chunk(const hsv_qaoa_batch* b, int bits) { return b->nt == 512 && bits == 13; }
void to_layout(int from, const std::vector<unsigned char>& cut, unsigned char* out) {
  const int lay = from <= 8 ? LAY_B : LAY_A;
  for (uint32_t t = 0; t < 512; ++t) {
    const uint32_t jt = (t & ((1u << lay) - 1)) | ((t >> lay) << (lay + 4));
    for (uint32_t r = 0; r < 16; ++r) out[t * 16 + r] = cut[jt | (r << lay)];
  }
}

// The chunks of one instance: what the edges that leave the chunk add to its
// table for each value of the bits outside it.
void add_items(const hsv_qaoa_batch* b, int id, int high, const int* pos, std::vector<Item>* items) {
  const Inst& I = b->inst[id];
  const int bits = I.bits[high];
  const uint64_t chunks = 1ull << (I.n - bits);
  for (uint64_t f = 0; f < chunks; ++f) {
    Item it{};
    const uint64_t base = high ? f << I.lc : f << bits;  // the outside bits are lc..L-1, or L..n-1
    it.off = I.off + base;
    it.inst = (uint32_t)id;
    it.part = (uint32_t)(I.part_off + f);
    for (int e = 0; e < I.ne; ++e) {
      const int u = b->eu[I.edge_off + e], v = b->ev[I.edge_off + e];
      const int pu = pos[u], pv = pos[v];
      const int hu = (int)(base >> u & 1), hv = (int)(base >> v & 1);
      if (pu >= 0 && pv >= 0) continue;
      if (pu < 0 && pv < 0) {
        it.w[13] += (int8_t)(hu ^ hv);
      } else {
        const int a = pu >= 0 ? pu : pv, h = pu >= 0 ? hv : hu;
        it.w[13] += (int8_t)h;
        it.w[a] += (int8_t)(1 - 2 * h);
      }
    }
    items->push_back(it);
  }
}

template <int NT>
void launch_pass(hsv_qaoa_batch* b, const Item* items, uint64_t nitems, int k, size_t lds, const unsigned char* tabs) {
  const int grid = (int)std::min<uint64_t>(nitems, (uint64_t)b->num_cu * b->grid_per_cu);
  hipLaunchKernelGGL((k_qaoa_pass<NT>), grid, NT, lds, b->stream, b->state, b->d_inst, items, (uint32_t)nitems, k, b->L,
                     b->d_phase, tabs, b->d_part);
}

// Builds the items and tables and captures the whole batch into a hipGraph.
int build_graph(hsv_qaoa_batch* b) {
  destroy_graph(b);
  const int L = b->L;
  // instances wider than a low chunk by falling p (those of pass k are a
  // prefix of either item list), then the others, which pass 0 runs whole
  std::vector<int> order(b->num);
  for (int i = 0; i < b->num; ++i) order[i] = i;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
    const Inst &X = b->inst[x], &Y = b->inst[y];
    return (X.n > L) != (Y.n > L) ? X.n > L : X.n > L && X.p > Y.p;
  });
  std::vector<Item> items[2];
  std::vector<unsigned char> tabs;
  std::vector<uint64_t> upto[2];  // items of the instances with p >= k
  upto[0].assign(b->pmax + 2, 0);
  upto[1].assign(b->pmax + 2, 0);
  uint64_t parts = 0;
  int maxbits = 0;
  for (int id : order) {
    Inst& I = b->inst[id];
    const bool whole = I.n <= L;
    const int hb = whole ? 0 : I.n - L;
    I.lc = whole ? I.n : low_contig(hb, L, b->nt);
    I.bits[0] = std::min(I.n, L);
    I.bits[1] = whole ? I.n : I.lc + hb;
    I.part_off = (int)parts;
    I.parts = 1 << (I.n - I.bits[whole ? 0 : I.p & 1]);
    parts += I.parts;
    for (int high = 0; high < (whole ? 1 : 2); ++high) {
      const int bits = I.bits[high];
      int pos[64];
      for (int v = 0; v < 64; ++v)
        pos[v] = !high ? (v < bits ? v : -1) : v < I.lc ? v : v >= L && v < I.n ? I.lc + v - L : -1;
      std::vector<unsigned char> cut(1ull << bits);
      cut_table(b, I, pos, bits, cut.data());
      I.tab[high] = tabs.size();
      tabs.resize(tabs.size() + std::max<size_t>(cut.size(), 16));
      if (fast_chunk(b, bits)) to_layout(high ? I.lc : 0, cut, tabs.data() + I.tab[high]);
      else std::memcpy(tabs.data() + I.tab[high], cut.data(), cut.size());
      add_items(b, id, high, pos, &items[high]);
      maxbits = std::max(maxbits, bits);
      if (!whole)
        for (int k = 0; k <= I.p; ++k) upto[high][k] = items[high].size();
    }
  }
  upto[0][0] = items[0].size();  // pass 0: the whole instances too
  const size_t high_off = items[0].size() * sizeof(Item);
  const size_t tab_off = high_off + items[1].size() * sizeof(Item);
  QCHK(hipMalloc(&b->d_plan, tab_off + tabs.size()));
  auto* plan = static_cast<unsigned char*>(b->d_plan);
  QCHK(hipMemcpy(plan, items[0].data(), high_off, hipMemcpyHostToDevice));
  if (!items[1].empty())
    QCHK(hipMemcpy(plan + high_off, items[1].data(), tab_off - high_off, hipMemcpyHostToDevice));
  QCHK(hipMemcpy(plan + tab_off, tabs.data(), tabs.size(), hipMemcpyHostToDevice));
  QCHK(hipMemcpy(b->d_inst, b->inst.data(), b->inst.size() * sizeof(Inst), hipMemcpyHostToDevice));
  QCHK(hipMalloc(reinterpret_cast<void**>(&b->d_part), parts * sizeof(double)));
  const size_t lds = (size_t(1) << maxbits) * sizeof(cf);

  QCHK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  if (b->total_angles)
    hipLaunchKernelGGL(k_qaoa_tables, b->total_angles, 64, 0, b->stream, b->d_inst, b->d_owner, b->d_gamma, b->d_beta,
                       b->d_phase);
  for (int k = 0; k <= b->pmax; ++k) {
    const uint64_t cnt = upto[k & 1][k];
    if (!cnt) continue;
    const Item* list = reinterpret_cast<const Item*>(plan + (k & 1 ? high_off : 0));
    if (b->nt == 128) launch_pass<128>(b, list, cnt, k, lds, plan + tab_off);
    else if (b->nt == 512) launch_pass<512>(b, list, cnt, k, lds, plan + tab_off);
    else launch_pass<256>(b, list, cnt, k, lds, plan + tab_off);
  }
  hipLaunchKernelGGL(k_qaoa_sum, b->num, 64, 0, b->stream, b->d_part, b->d_inst, b->h_out);
  hipError_t ce = hipStreamEndCapture(b->stream, &b->graph);
  if (ce != hipSuccess) return qfail(HSV_ERR_DEVICE, std::string("graph capture: ") + hipGetErrorString(ce));
  QCHK(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
  return HSV_OK;
}

}  // namespace

extern "C" {

int hsv_qaoa_create(int num_instances, const int* num_qubits, const int* edge_offsets, const int* edges,
                    const int* layers, hsv_qaoa_batch** out) {
  if (!out || num_instances <= 0 || !num_qubits || !edge_offsets || !edges || !layers)
    return qfail(HSV_ERR_ARG, "bad arguments");
  *out = nullptr;
  auto* b = new hsv_qaoa_batch();
  b->num = num_instances;
  uint64_t off = 0;
  int aoff = 0;
  for (int i = 0; i < num_instances; ++i) {
    const int n = num_qubits[i];
    const int e0 = edge_offsets[i], e1 = edge_offsets[i + 1];
    if (n < 1 || n > kMaxQaoaQubits || e1 < e0 || e1 - e0 > kMaxEdges || layers[i] < 0) {
      delete b;
      return qfail(HSV_ERR_ARG, "instance " + std::to_string(i) + ": qubits, edges or layers out of range");
    }
    for (int e = e0; e < e1; ++e) {
      const int u = edges[2 * e], v = edges[2 * e + 1];
      if (u < 0 || v < 0 || u >= n || v >= n || u == v) {
        delete b;
        return qfail(HSV_ERR_ARG, "instance " + std::to_string(i) + ": bad edge");
      }
    }
    Inst I{};
    I.off = off;
    I.n = n;
    I.ne = e1 - e0;
    I.edge_off = (int)b->eu.size();
    I.p = layers[i];
    I.angle_off = aoff;
    for (int e = e0; e < e1; ++e) {
      b->eu.push_back((unsigned char)edges[2 * e]);
      b->ev.push_back((unsigned char)edges[2 * e + 1]);
    }
    b->inst.push_back(I);
    off += 1ull << n;
    aoff += layers[i];
    b->pmax = std::max(b->pmax, layers[i]);
  }
  b->total_amps = off;
  b->total_angles = aoff;
  int dev = 0;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) {
    delete b;
    return qfail(HSV_ERR_DEVICE, "no HIP device");
  }
  b->num_cu = prop.multiProcessorCount;
  if (hipStreamCreate(&b->stream) != hipSuccess) { delete b; return qfail(HSV_ERR_DEVICE, "stream"); }
  if (hipMalloc(reinterpret_cast<void**>(&b->state), off * sizeof(cf)) != hipSuccess ||
      hipMalloc(reinterpret_cast<void**>(&b->d_inst), b->inst.size() * sizeof(Inst)) != hipSuccess ||
      hipMalloc(reinterpret_cast<void**>(&b->d_gamma), std::max(aoff, 1) * sizeof(double)) != hipSuccess ||
      hipMalloc(reinterpret_cast<void**>(&b->d_beta), std::max(aoff, 1) * sizeof(double)) != hipSuccess ||
      hipMalloc(reinterpret_cast<void**>(&b->d_owner), std::max(aoff, 1) * sizeof(uint32_t)) != hipSuccess ||
      hipMalloc(reinterpret_cast<void**>(&b->d_phase), std::max<size_t>(aoff, 1) * kPhaseRow * sizeof(float2)) != hipSuccess ||
      hipHostMalloc(reinterpret_cast<void**>(&b->h_out), b->num * sizeof(double), 0) != hipSuccess) {
    hsv_qaoa_destroy(b);
    return qfail(HSV_ERR_ALLOC, "cannot allocate the batch");
  }
  std::vector<uint32_t> owner;
  for (int i = 0; i < b->num; ++i) owner.insert(owner.end(), b->inst[i].p, (uint32_t)i);
  if (aoff) QCHK(hipMemcpy(b->d_owner, owner.data(), owner.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
  QCHK(hipEventCreate(&b->e0));
  QCHK(hipEventCreate(&b->e1));
  *out = b;
  return HSV_OK;
}

int hsv_qaoa_destroy(hsv_qaoa_batch* b) {
  if (!b) return HSV_OK;
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  destroy_graph(b);
  (void)hipFree(b->state);
  (void)hipFree(b->d_inst);
  (void)hipFree(b->d_gamma);
  (void)hipFree(b->d_beta);
  (void)hipFree(b->d_owner);
  (void)hipFree(b->d_phase);
  if (b->h_out) (void)hipHostFree(b->h_out);
  if (b->e0) (void)hipEventDestroy(b->e0);
  if (b->e1) (void)hipEventDestroy(b->e1);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
  return HSV_OK;
}

int hsv_qaoa_tune(hsv_qaoa_batch* b, const char* key, int value) {
  if (!b || !key) return qfail(HSV_ERR_ARG, "null argument");
  const std::string k = key;
  if (k == "chunk_bits" && value >= 8 && value <= 13) b->L = value;
  else if (k == "threads" && (value == 128 || value == 256 || value == 512)) b->nt = value;
  else if (k == "grid_per_cu" && value >= 1 && value <= 64) b->grid_per_cu = value;
  else return qfail(HSV_ERR_ARG, "unknown QAOA tuning key or value: " + k);
  // a high chunk holds the high qubits and kLowContig low ones: within 64 KB of LDS
  int maxn = 0;
  for (const Inst& I : b->inst) maxn = std::max(maxn, I.n);
  if (kLowContig + maxn - b->L > kStageBBits) return qfail(HSV_ERR_LIMIT, "chunk_bits too small for the widest instance");
  destroy_graph(b);
  return HSV_OK;
}

int hsv_qaoa_set_angles(hsv_qaoa_batch* b, const double* gammas, const double* betas) {
  if (!b || (b->total_angles && (!gammas || !betas))) return qfail(HSV_ERR_ARG, "null argument");
  if (!b->total_angles) return HSV_OK;
  QCHK(hipMemcpyAsync(b->d_gamma, gammas, sizeof(double) * b->total_angles, hipMemcpyHostToDevice, b->stream));
  QCHK(hipMemcpyAsync(b->d_beta, betas, sizeof(double) * b->total_angles, hipMemcpyHostToDevice, b->stream));
  QCHK(hipStreamSynchronize(b->stream));
  return HSV_OK;
}

int hsv_qaoa_run(hsv_qaoa_batch* b, double* expectations) {
  if (!b || !expectations) return qfail(HSV_ERR_ARG, "null argument");
  int maxn = 0;
  for (const Inst& I : b->inst) maxn = std::max(maxn, I.n);
  if (kLowContig + maxn - b->L > kStageBBits) return qfail(HSV_ERR_LIMIT, "chunk_bits too small for the widest instance");
  if (!b->exec)
    if (int rc = build_graph(b)) return rc;
  QCHK(hipEventRecord(b->e0, b->stream));
  QCHK(hipGraphLaunch(b->exec, b->stream));
  QCHK(hipEventRecord(b->e1, b->stream));
  QCHK(hipStreamSynchronize(b->stream));
  QCHK(hipEventElapsedTime(&b->last_ms, b->e0, b->e1));
  std::memcpy(expectations, b->h_out, sizeof(double) * b->num);
  return HSV_OK;
}

int hsv_qaoa_last_ms(hsv_qaoa_batch* b, double* ms) {
  if (!b || !ms) return qfail(HSV_ERR_ARG, "null argument");
  *ms = b->last_ms;
  return HSV_OK;
}

int hsv_qaoa_read_state(hsv_qaoa_batch* b, int instance, double* amps) {
  if (!b || !amps || instance < 0 || instance >= b->num) return qfail(HSV_ERR_ARG, "bad instance");
  const Inst& I = b->inst[instance];
  std::vector<cf> tmp(1ull << I.n);
  QCHK(hipMemcpyAsync(tmp.data(), b->state + I.off, tmp.size() * sizeof(cf), hipMemcpyDeviceToHost, b->stream));
  QCHK(hipStreamSynchronize(b->stream));
  for (size_t i = 0; i < tmp.size(); ++i) {
    amps[2 * i] = tmp[i].x;
    amps[2 * i + 1] = tmp[i].y;
  }
  return HSV_OK;
}

int hsv_qaoa_total_amplitudes(hsv_qaoa_batch* b, uint64_t* out) {
  if (!b || !out) return qfail(HSV_ERR_ARG, "null argument");
  *out = b->total_amps;
  return HSV_OK;
}

}  // extern "C"
