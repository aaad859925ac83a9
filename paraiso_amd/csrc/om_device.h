// Hand-written device templates shared by every generated OM machine (gfx950).
//
// The generator instantiates these for each kernel of an Orthotope Machine:
//   * om_wrap        cyclic index wrap for halo reads
//                    (the reference's `(x + c + n) % n`, Generator/PlanTrans.hs:459-461,481-483),
//   * om_clamp       keeps halo reads of Open (non-periodic) axes inside the grid,
//   * om_max/om_min  exactly std::max/std::min (the reference's CPU Max/Min,
//                    Generator/PlanTrans.hs:690-691): ties and NaNs resolve as there,
//   * om_resident_workgroups  grid size of a persistent (tile-looping) launch,
//   * om_lane*, om_at/om_put, om_turn  register streaming: a neighbour lane's value, a
//                    row's element at a scalar address, 64 cells as a row of bits,
//   * om_block_*     wave64 shuffle tree + LDS combine for Reduce: each
//                    workgroup writes one partial, and a one-workgroup finish
//                    kernel folds the partials in a fixed order, replacing the
//                    reference's serial om_reduce_* (Generator/PlanTrans.hs:719)
//                    with a deterministic tree.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// CUs of the current device.
static inline int om_cus() {
  static int cus = 0;
  if (cus <= 0) {
    int d = 0;
    if (hipGetDevice(&d) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, d) != hipSuccess ||
        cus <= 0)
      cus = 256;
  }
  return cus;
}

// Workgroups a persistent launch starts: as many as the device holds at once (per_cu per
// CU, from the launch's LDS and work-items), a multiple of 8 so that workgroup b, which the
// dispatcher places on XCD b % 8, keeps to that XCD's band of tiles; at most ntiles.
static inline unsigned om_resident_workgroups(unsigned ntiles, int per_cu) {
  unsigned n = ((unsigned)om_cus() * (unsigned)(per_cu > 0 ? per_cu : 1)) & ~7u;
  if (n == 0) n = 8;
  return n < ntiles ? n : ntiles;
}


// Division of a tile index by a tile count d without the division expansion: m is
// floor((2^32 - 1) / d) from the host, so umulhi(x, m) is floor(x / d) or one less for any
// x < 2^31, and one compare corrects it (the operands are uniform: scalar instructions).
static inline unsigned om_udiv_magic(unsigned d) { return d ? 0xFFFFFFFFu / d : 0u; }

__device__ __forceinline__ unsigned om_udiv(unsigned x, unsigned d, unsigned m) {
  const unsigned q = __umulhi(x, m);
  return q + ((q + 1u) * d <= x ? 1u : 0u);
}

// One conditional add and subtract cover -n <= x < 2n.  `wide` (uniform: the host sets it
// when some axis of the grid is shorter than the launch's tile plus its reach) enables the
// remainder for coordinates further out; otherwise the branch around it is scalar.
__device__ __forceinline__ int om_wrap(int x, int n, int wide) {
  x = (x < 0) ? x + n : x;
  x = (x >= n) ? x - n : x;
  if (wide && (unsigned)x >= (unsigned)n) x = ((x % n) + n) % n;
  return x;
}

__device__ __forceinline__ int om_clamp(int x, int n) { return x < 0 ? 0 : (x < n ? x : n - 1); }

template <class T> __device__ __forceinline__ T om_max(T a, T b) { return (a < b) ? b : a; }
template <class T> __device__ __forceinline__ T om_min(T a, T b) { return (b < a) ? b : a; }

// a * b <= 0 ? 0 : (|a| < |b| ? a : b): the median of a, b and 0, and b where one is not a
// number (fast FP32 builds: the same but for a product that underflows to 0, where the limiter
// returns the smaller value as exact arithmetic would).  Three instructions for six.
__device__ __forceinline__ float om_minmod(float a, float b) {
  const float m = __builtin_amdgcn_fmed3f(a, b, 0.0f);
  return __builtin_isunordered(a, b) ? b : m;
}

struct OmSum {
  template <class T> __device__ __forceinline__ T operator()(T a, T b) const { return a + b; }
};
struct OmSumWrap {   // integer sum with two's-complement wrap (order independent)
  __device__ __forceinline__ int operator()(int a, int b) const {
    return (int)((unsigned)a + (unsigned)b);
  }
};
struct OmMin {
  template <class T> __device__ __forceinline__ T operator()(T a, T b) const { return om_min(a, b); }
};
struct OmMax {
  template <class T> __device__ __forceinline__ T operator()(T a, T b) const { return om_max(a, b); }
};

// Fixed-shape reduction of one value per thread of an NT-thread workgroup; every thread
// gets the result.  The xor-shuffle tree and the wave order are fixed, so results are
// bit-reproducible run to run.
template <int NT, class T, class Op>
__device__ __forceinline__ T om_block_reduce(T v, Op op, T* scratch /* >= NT / 64 */) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = op(v, __shfl_xor(v, off, 64));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  T r = scratch[0];
#pragma unroll
  for (int w = 1; w < NT / 64; ++w) r = op(r, scratch[w]);
  return r;   // every thread gets the block result
}

// ---- register streaming (a wave64 owns a strip of the grid, a lane a column of cells)

// The value of the lane D places to the right (left for D < 0): wave-wide DPP moves, one
// VALU instruction per place and 32 bits.  Lanes moved in from outside the wave hold 0 and
// lie in the overlap of neighbouring strips, where nothing is stored.
template <int D> __device__ __forceinline__ int om_lane32(int v) {
  if constexpr (D > 0)
    return om_lane32<D - 1>(__builtin_amdgcn_update_dpp(0, v, 0x130 /* wave_shl:1 */, 0xf, 0xf, true));
  else if constexpr (D < 0)
    return om_lane32<D + 1>(__builtin_amdgcn_update_dpp(0, v, 0x138 /* wave_shr:1 */, 0xf, 0xf, true));
  else
    return v;
}
template <int D> __device__ __forceinline__ int om_lane(int v) { return om_lane32<D>(v); }
template <int D> __device__ __forceinline__ bool om_lane(bool v) { return om_lane32<D>((int)v) != 0; }
template <int D> __device__ __forceinline__ float om_lane(float v) {
  return __builtin_bit_cast(float, om_lane32<D>(__builtin_bit_cast(int, v)));
}
template <int D> __device__ __forceinline__ double om_lane(double v) {
  struct P { int lo, hi; };
  const P p = __builtin_bit_cast(P, v);
  return __builtin_bit_cast(double, P{om_lane32<D>(p.lo), om_lane32<D>(p.hi)});
}

// Element x of the row at a scalar address: the address stays in scalar registers and the
// lane adds a 32-bit byte offset.  Rows of 2^29 cells or more, whose byte offset may not fit,
// take the tile form, or om_far_at where a kernel has no tile form.
template <class T> __device__ __forceinline__ T om_at(const T* row, int x) {
  return *(const T*)((const char*)row + (unsigned)x * (unsigned)sizeof(T));
}
template <class T> __device__ __forceinline__ void om_put(T* row, int x, T v) {
  *(T*)((char*)row + (unsigned)x * (unsigned)sizeof(T)) = v;
}
template <class T> __device__ __forceinline__ T om_far_at(const T* row, int x) { return row[x]; }
template <class T> __device__ __forceinline__ void om_far_put(T* row, int x, T v) { row[x] = v; }

// Lane r's two words become the 64-bit mask: row r of a square of bits (r is a constant after
// unrolling; the masks are scalar).
__device__ int om_writelane(int value, int lane, int old) __asm("llvm.amdgcn.writelane.i32");
__device__ __forceinline__ void om_turn(int r, unsigned long long mask, unsigned& w0, unsigned& w1) {
  w0 = (unsigned)om_writelane((int)(unsigned)mask, r, (int)w0);
  w1 = (unsigned)om_writelane((int)(unsigned)(mask >> 32), r, (int)w1);
}

// A value that every lane holds, in scalar registers, rounded to its type (nothing is
// contracted across it: the same bits as a value read back from memory).
__device__ __forceinline__ int om_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ bool om_uniform(bool v) { return om_uniform((int)v) != 0; }
__device__ __forceinline__ float om_uniform(float v) {
  asm("" : "+v"(v));   // (the compiler sees through readfirstlane of a uniform value)
  return __builtin_bit_cast(float, om_uniform(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double om_uniform(double v) {
  asm("" : "+v"(v));
  struct P { int lo, hi; };
  const P p = __builtin_bit_cast(P, v);
  return __builtin_bit_cast(double, P{om_uniform(p.lo), om_uniform(p.hi)});
}

template <class T, class Op> __device__ __forceinline__ T om_wave_reduce(T v, Op op) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = op(v, __shfl_xor(v, off, 64));
  return v;
}

// Steps along the streaming axis (n long) that one wave takes, for `groups` waves side by
// side: the axis is cut into as many chunks as make the shortest launch, where a chunk costs
// its own steps and a run-up worth `runup` steps, and a SIMD takes as long for a step of its
// waves as for `fill` of them where it holds fewer (issue slots or memory latency that too few
// waves leave unused: 1.2 for the Hydro step, where one wave takes 1.36 us a row and two 2.27;
// 4 where memory bounds).  At most `cap` waves, at least `least` steps.
static inline int om_lane_chunk(int n, unsigned groups, double runup, double fill, unsigned cap,
                                int least, unsigned simds) {
  int best = n;
  double cost = 1e300;
  if (groups == 0) groups = 1;
  for (unsigned k = 1; k <= 8; ++k) {
    unsigned chunks = k * simds / groups;
    if (chunks > cap / groups) chunks = cap / groups;
    if (chunks < 1) chunks = 1;
    int h = (int)((n + chunks - 1) / chunks);
    if (h < least) h = least < n ? least : n;
    const unsigned waves = groups * (unsigned)((n + h - 1) / h);
    const unsigned per = (waves + simds - 1) / simds;
    const double c = ((double)h + runup) * (per > fill ? per : fill);
    if (c < 0.999 * cost) {
      cost = c;
      best = h;
    }
  }
  return best;
}

// Reduce `count` partials in a fixed order.  Thread t keeps eight accumulators: lane
// k folds partials t + (8j + k) NT, so eight independent loads are in flight per thread
// (a one-workgroup reduction of 10^4-10^5 partials is bound by load latency); then the
// eight are folded in order and the workgroup tree finishes.
template <int NT, class T, class Op>
__device__ __forceinline__ T om_partials_reduce(const T* __restrict__ part, int count, T init,
                                                 Op op, T* scratch) {
  T acc[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) acc[k] = init;
  int i = threadIdx.x;
  for (; i + 7 * NT < count; i += 8 * NT) {
    T v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = part[i + k * NT];
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = op(acc[k], v[k]);
  }
  for (int k = 0; i < count; i += NT, ++k) acc[k] = op(acc[k], part[i]);
  T r = acc[0];
#pragma unroll
  for (int k = 1; k < 8; ++k) r = op(r, acc[k]);
  return om_block_reduce<NT>(r, op, scratch);
}
