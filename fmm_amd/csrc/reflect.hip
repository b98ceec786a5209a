// reflect.hip -- the dense M2L by reflection classes (reflect.hpp), on the f64 matrix cores.
#include "reflect.hpp"

#include <algorithm>
#include <cstring>

#include "common.hpp"
#include "kernels.hpp"

namespace fmmh {

const ReflectClasses &reflect_classes() {
  static const ReflectClasses rc = [] {
    ReflectClasses r{};
    int n = 0, pos = 0;
    for (int paired = 0; paired < 8; ++paired) {
      r.run[paired] = n;
      for (int t = 0; t < 64; ++t) {
        const int a = t >> 4, b = (t >> 2) & 3, c = t & 3;
        auto pair = [](int v) { return v == 1 || v == 2; };
        if (a <= 1 && b <= 1 && c <= 1) continue;
        if (((pair(a) ? 4 : 0) | (pair(b) ? 2 : 0) | (pair(c) ? 1 : 0)) != paired) continue;
        r.offset[n] = {a, b, c};
        r.axes[n] = (a > 0 ? 4 : 0) | (b > 0 ? 2 : 0) | (c > 0 ? 1 : 0);
        r.paired[n] = paired;
        r.first[n] = pos;
        pos += 1 << __builtin_popcount(unsigned(paired));
        ++n;
      }
    }
    r.run[8] = n;
    r.first[n] = pos;
    return r;
  }();
  return rc;
}

int ReflectClasses::position(const int d[3], int flip) const {
  int m[3], negative = 0;
  for (int a = 0; a < 3; ++a) {
    const int v = (flip >> (2 - a)) & 1 ? -d[a] : d[a];
    m[a] = v < 0 ? -v : v;
    if (v < 0) negative |= 4 >> a;
  }
  for (int c = 0; c < kReflectClasses; ++c) {
    if (offset[c][0] != m[0] || offset[c][1] != m[1] || offset[c][2] != m[2]) continue;
    require((negative & ~paired[c]) == 0, "M2L schedule: V offset outside the parent's neighbours",
            kUnsupportedLayout);
    int rank = 0;  // among the sign sets of the paired components
    for (int s = 0; s < negative; ++s) rank += (s & ~paired[c]) == 0;
    return first[c] + rank;
  }
  throw Error(kUnsupportedLayout, "M2L schedule: V offset outside the parent's neighbours");
}

// Parity of the coefficient (n, m): odd in z when n - |m| is, in y when it is a sine
// (m < 0), in x when a cosine of odd or a sine of even order.
static int parity_of(int n, int m) {
  const int q = m < 0 ? -m : m;
  const int z = (n - q) & 1, y = m < 0 ? 1 : 0, x = m < 0 ? (q + 1) & 1 : q & 1;
  return 4 * x + 2 * y + z;
}

ReflectLayout::ReflectLayout(int degree, int pad) : p(degree), nc((degree + 1) * (degree + 1)) {
  for (int c = 0; c < 8; ++c) {
    std::vector<int32_t> rows;
    for (int n = 0; n <= p; ++n)
      for (int m = -n; m <= n; ++m)
        if (parity_of(n, m) == c) rows.push_back(n * n + n + m);
    for (int32_t k : rows) {
      perm.push_back(k);
      parity.push_back(uint8_t(c));
    }
    for (size_t i = 0; i < rows.size(); i += 16) {
      for (size_t j = i; j < i + 16; ++j) tile_row.push_back(j < rows.size() ? rows[j] : -1);
      tile_class.push_back(uint8_t(c));
    }
  }
  tiles = int(tile_class.size());
  kp = (nc + pad - 1) / pad * pad;
  perm.resize(kp, -1);
  parity.resize(kp, 0);
}

uint64_t ReflectLayout::steps(int axes, int c, int width) const {
  uint64_t m = 0;
  for (int k = 0; k < nc; ++k)
    if (((parity[k] ^ c) & ~axes & 7) == 0) m |= uint64_t(1) << (k / width);
  return m;
}

namespace dev {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

size_t reflect_table_size(const ReflectLayout &l) { return size_t(l.kp / kReflectChunk) * l.tiles * 256; }

void reflect_table(const ReflectLayout &l, const double *a, double *out) {
  for (int ch = 0; ch < l.kp / kReflectChunk; ++ch)
    for (int t = 0; t < l.tiles; ++t)
      for (int h = 0; h < 2; ++h)
        for (int lane = 0; lane < 64; ++lane)
          for (int q = 0; q < 2; ++q) {
            const int row = l.tile_row[16 * t + (lane & 15)];
            const int k = l.perm[ch * kReflectChunk + 8 * h + 4 * q + (lane >> 4)];
            out[((size_t(ch) * l.tiles + t) * 2 + h) * 128 + 2 * lane + q] =
                row >= 0 && k >= 0 ? a[row + size_t(k) * l.nc] : 0.0;
          }
}

__global__ void k_reflect_sort(int nc, int kp, size_t total, const int32_t *__restrict__ perm,
                               const double *__restrict__ X, double *__restrict__ Xs) {
  for (size_t i = blockIdx.x * size_t(blockDim.x) + threadIdx.x; i < total; i += size_t(gridDim.x) * blockDim.x) {
    const size_t box = i / size_t(kp);
    const int k = perm[i - box * size_t(kp)];
    Xs[i] = k >= 0 ? X[box * size_t(nc) + k] : 0.0;
  }
}

void reflect_sort(hipStream_t s, int nc, int kp, size_t nboxes, const int32_t *perm, const double *X, double *Xs) {
  if (nboxes == 0) return;
  const size_t total = nboxes * size_t(kp);
  const size_t grid = std::min<size_t>((total + 255) / 256, 65536);
  hipLaunchKernelGGL(k_reflect_sort, dim3(unsigned(grid)), dim3(256), 0, s, nc, kp, total, perm, X, Xs);
}

// Waits for this wave's LDS operations, then the workgroup barrier; global loads in flight
// stay in flight (__syncthreads would wait for them too).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

struct ReflectF64 {
  static constexpr int LD = 17;  // row stride (no bank conflicts when written along k)
  double W[2][8][kReflectChunk][LD];
  uint32_t sign[256];  // per sorted coefficient: bits 31, 30, 29 its parities in x, y, z
};

// Bit 31: the sign of a coefficient of parities `sign` (bits 31 .. 29) under the reflection
// of the axes in `flip` (bits 31 .. 29).
__device__ __forceinline__ uint32_t flip_of(uint32_t sign, uint32_t flip) {
  const uint32_t x = sign & flip;
  return x ^ (x << 1) ^ (x << 2);
}

// Units of 64 lanes in one set of the class tables (16 bytes per lane).
__device__ __forceinline__ size_t table_set(const ReflectArgs &a) {
  return size_t(kReflectClasses) * (a.kp / kReflectChunk) * a.tiles * 2;
}
__device__ __forceinline__ size_t table_set16(const ReflectArgs &a) {
  return size_t(kReflectClasses) * (a.kp / kReflectChunk16) * a.tiles * 3;
}

// Small read-only tables through the scalar cache.
template <typename T>
__device__ __forceinline__ T scalar_read(const T *p) {
  return *reinterpret_cast<const __attribute__((address_space(4))) T *>(reinterpret_cast<uintptr_t>(p));
}

__device__ __forceinline__ double signed_one(uint32_t bit) {  // -1 for bit 31 set
  return __hiloint2double(int((bit & 0x80000000u) | 0x3FF00000u), 0);
}

// The butterfly over the paired components PAIRED of one coefficient: v[s], s the negative
// components, becomes W of every parity.  sign: bits 31, 30, 29 the coefficient's parities
// in x, y, z; flip: bit 31 the sign of the coefficient under the target's own reflection.
template <int PAIRED, typename V>
__device__ __forceinline__ void butterfly(V &v, uint32_t sign, uint32_t flip) {
  double f = signed_one(flip);
  if (PAIRED == 0) v[0] *= f;
  uint32_t first = flip;
#pragma unroll
  for (int b = 1; b < 8; b <<= 1) {
    if (!(PAIRED & b)) continue;
    const double e = signed_one((b == 4 ? sign : b == 2 ? sign << 1 : sign << 2) ^ first);
    const bool scale = (PAIRED & (b - 1)) == 0;  // the first component also takes the flip
    first = 0;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      if ((s & b) || (s & ~PAIRED)) continue;
      const double plus = scale ? v[s] * f : v[s], minus = v[s | b];
      v[s] = fma(e, minus, plus);
      v[s | b] = fma(-e, minus, plus);
    }
  }
}

// The classes c0 .. c1 - 1, all of paired components PAIRED: every load and every LDS write
// is unconditional, so the loads of the next step stay in flight over the barrier.
template <int PAIRED, int TPW>
__device__ __forceinline__ void reflect_run(ReflectF64 &sh, int &buf, const ReflectArgs &a, const uint32_t *ids,
                                            uint32_t flip, int c0, int c1, const d2 *__restrict__ tables,
                                            const char *__restrict__ Xs, int nt, const int (&tcls)[TPW],
                                            d4 (&acc)[TPW]) {
  constexpr int NS = 1 << __builtin_popcount(unsigned(PAIRED));
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int nch = a.kp / kReflectChunk;
  const int kk = tid & 15, col = tid >> 4;  // this thread's coefficient and target
  const int g = lane >> 4, n = lane & 15;
  const uint32_t *pos = ids + (scalar_read(a.first + c0) & 0xFFFFu);
  uint32_t id[NS], idn[NS];
  double v[8];
  auto load = [&](const uint32_t (&from)[NS], int ch) {
    int q = 0;
#pragma unroll
    for (int s = 0; s < 8; ++s)
      if (!(s & ~PAIRED))
        v[s] = *reinterpret_cast<const double *>(Xs + (from[q++] + uint32_t(ch * kReflectChunk + kk) * 8u));
  };
#pragma unroll
  for (int q = 0; q < NS; ++q) id[q] = pos[q];
  load(id, 0);
  // the table's operand of a chunk (a tile that skips it reads the chunk's first tile)
  const d2 *t = tables + (size_t(c0) * nch * a.tiles + wave) * 128 + lane;
  uint64_t mask[TPW];
  auto load_masks = [&](int cl) {
    const uint64_t *km = a.kmask + 8 * (scalar_read(a.first + cl) >> 16);
#pragma unroll
    for (int i = 0; i < TPW; ++i) mask[i] = i < nt ? scalar_read(km + tcls[i]) : 0;
  };
  load_masks(c0);
  d2 av[TPW][2];
  uint32_t bits[TPW];
  auto load_table = [&](int i, int ch) {
    bits[i] = uint32_t(mask[i] >> (4 * ch)) & 15u;
    const d2 *ti = t + (bits[i] ? 512 * i : 0);
    av[i][0] = ti[0];
    av[i][1] = ti[64];
  };
#pragma unroll
  for (int i = 0; i < TPW; ++i) load_table(i, 0);
#pragma unroll 1
  for (int cl = c0; cl < c1; ++cl) {
    // the sources of the next class (the last class reads its own again)
    pos += cl + 1 < c1 ? NS : 0;
#pragma unroll
    for (int q = 0; q < NS; ++q) idn[q] = pos[q];
#pragma unroll 1
    for (int ch = 0; ch < nch; ++ch) {
      // the butterflies of this thread's coefficient
      const uint32_t sign = sh.sign[ch * kReflectChunk + kk];
      butterfly<PAIRED>(v, sign, flip_of(sign, flip));
#pragma unroll
      for (int s = 0; s < 8; ++s)
        if (!(s & ~PAIRED)) sh.W[buf][s][kk][col] = v[s];
      // the next step's multipoles
      const int nx = ch + 1 == nch ? 0 : ch + 1;
      if (nx == 0) {
#pragma unroll
        for (int q = 0; q < NS; ++q) id[q] = idn[q];
        load_masks(cl + 1 < c1 ? cl + 1 : cl);
      }
      load(id, nx);
      lds_barrier();
      // every tile's products, and its operand of the next step into the registers they free
      t += size_t(a.tiles) * 128;
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        const double(*w)[ReflectF64::LD] = sh.W[buf][tcls[i] & PAIRED];
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (bits[i] & (3u << (2 * h))) {
            const double b0 = w[8 * h + g][n], b1 = w[8 * h + 4 + g][n];
            acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i][h][0], b0, acc[i], 0, 0, 0);
            acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i][h][1], b1, acc[i], 0, 0, 0);
          }
        load_table(i, nx);
      }
      // the next step fills the other buffer; every wave has read it before this barrier
      buf ^= 1;
    }
  }
}

// One workgroup of four waves per task of 16 target boxes (any in Morton order: a box
// without a source at some reflection has the zero row there).  Per class and chunk of 16
// sorted coefficients every thread forms the butterfly of one (box, coefficient) and puts
// the W of every sign pattern into LDS; the waves then multiply their row tiles (tile t on
// wave t % 4, each of one parity class, so each reads one W) by v_mfma_f64_16x16x4, the table's operand read from L2.  Rows without a partner (an offset
// component 0) skip the chunk's steps of the other parity.
//
// 39.5 x tiles x steps matrix instructions of 64 cycles per 16 boxes bound it; f64 matrix and
// vector instructions do not overlap here, so the butterflies (about an eighth of the cycles)
// add to them.  35 KB of LDS and at most 128 VGPRs: four workgroups per CU cover each other's
// barriers and table loads.  32 and 64 targets per workgroup (half and a quarter of the table
// reads) were slower: 6.3 and 7.7 ms against 5.7 at the same stage of the kernel.  1M points,
// p = 12 (6.0M pairs): 3.0 ms against 8.7 by contraction, 45% -> 59% of the f64 matrix rate.
template <int TPW>
__global__ __launch_bounds__(256, 4) void k_m2l_reflect_f64(ReflectArgs a, uint32_t ntasks,
                                                                const double *__restrict__ tables,
                                                                const double *__restrict__ Xs,
                                                                double *__restrict__ Y, double *__restrict__ S) {
  __shared__ ReflectF64 sh;
  const uint32_t ti = xcd_index(ntasks, 16);
  if (ti >= ntasks) return;
  const ReflectTask task = a.tasks[ti];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (int k = tid; k < a.kp; k += 256) sh.sign[k] = uint32_t(a.parity[k]) << 29;
  // the sources of this thread's target (a row past the task's last takes the last row's)
  const uint32_t mine = task.row0 + min(uint32_t(tid) >> 4, uint32_t(task.nrows) - 1u);
  const uint32_t *ids = a.src + (size_t(mine) * a.sets + task.set) * kReflectPositions;
  const uint32_t flip = uint32_t(a.row_flip[mine]) << 29;
  d4 acc[TPW];
  int tcls[TPW];
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    acc[i] = d4{0.0, 0.0, 0.0, 0.0};
    tcls[i] = wave + 4 * i < a.tiles ? int(a.tile_class[wave + 4 * i]) : 0;
    tcls[i] = __builtin_amdgcn_readfirstlane(tcls[i]);
  }
  const int nt = __builtin_amdgcn_readfirstlane(wave < a.tiles ? (a.tiles - wave + 3) / 4 : 0);
  __syncthreads();
  const d2 *t2 = reinterpret_cast<const d2 *>(tables) + size_t(task.table) * table_set(a) * 64;
  const char *x = reinterpret_cast<const char *>(Xs);
  int buf = 0;
#define FMMH_RUN(P)                                                                         \
  {                                                                                         \
    const int c0 = max(int(task.first), a.run[P]), c1 = min(int(task.last), a.run[P + 1]);  \
    if (c0 < c1) reflect_run<P, TPW>(sh, buf, a, ids, flip, c0, c1, t2, x, nt, tcls, acc);  \
  }
  FMMH_RUN(0)
  FMMH_RUN(1)
  FMMH_RUN(2)
  FMMH_RUN(3)
  FMMH_RUN(4)
  FMMH_RUN(5)
  FMMH_RUN(6)
  FMMH_RUN(7)
#undef FMMH_RUN
  // accumulator element r of lane (g, j): row 4 r + g of the tile, target j
  const uint32_t r = lane & 15;
  if (r >= task.nrows) return;
  const bool slot = task.slot != kNone;
  double *y = slot ? S + size_t(task.slot + r * task.stride) * a.nc : Y + size_t(a.row_out[task.row0 + r]) * a.nc;
  const uint32_t out_flip = uint32_t(a.row_flip[task.row0 + r]) << 29;
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    if (i >= nt) continue;
    const double f = signed_one(flip_of(uint32_t(tcls[i]) << 29, out_flip));
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = a.tile_row[16 * (wave + 4 * i) + 4 * q + (lane >> 4)];
      if (row >= 0) y[row] = slot ? f * acc[i][q] : fma(f, acc[i][q], y[row]);
    }
  }
}

void m2l_reflect_f64(hipStream_t s, const ReflectArgs &a, uint32_t ntasks, const double *tables, const double *Xs,
                     double *Y, double *S) {
  if (ntasks == 0) return;
#define FMMH_REFLECT(N)                                                                                             \
  case N:                                                                                                           \
    hipLaunchKernelGGL(k_m2l_reflect_f64<N>, dim3(xcd_grid(ntasks, 16)), dim3(256), 0, s, a, ntasks, tables, Xs, Y, \
                       S);                                                                                          \
    break;
  switch ((a.tiles + 3) / 4) {
    FMMH_REFLECT(1)
    FMMH_REFLECT(2)
    FMMH_REFLECT(3)
    FMMH_REFLECT(4)
    FMMH_REFLECT(5)
    default:
      break;
  }
#undef FMMH_REFLECT
}

// ---- bf16x3 ----------------------------------------------------------------------------------

size_t reflect_table_size_bf16(const ReflectLayout &l) { return size_t(l.kp / kReflectChunk16) * l.tiles * 3 * 512; }

void reflect_table_bf16(const ReflectLayout &l, const double *a, uint16_t *out) {
  for (int ch = 0; ch < l.kp / kReflectChunk16; ++ch)
    for (int t = 0; t < l.tiles; ++t)
      for (int lane = 0; lane < 64; ++lane)
        for (int e = 0; e < 8; ++e) {
          const int row = l.tile_row[16 * t + (lane & 15)];
          const int k = l.perm[ch * kReflectChunk16 + 8 * (lane >> 4) + e];
          uint16_t s[3] = {0, 0, 0};
          if (row >= 0 && k >= 0) split_bf16x3(a[row + size_t(k) * l.nc], s);
          for (int pl = 0; pl < 3; ++pl)
            out[((size_t(ch) * l.tiles + t) * 3 + pl) * 512 + 8 * lane + e] = s[pl];
        }
}

constexpr int kPlane = 4 * 320;  // bytes of 32 coefficients x 16 targets in bf16, rows of 8 padded apart

struct ReflectBf16 {
  char W[8][3][2][kPlane];  // sign pattern, plane, 16 targets
  uint32_t sign[256];
};

template <int PAIRED, int TPW>
__device__ __forceinline__ void reflect_run16(ReflectBf16 &sh, const ReflectArgs &a, const uint32_t *ids,
                                              uint32_t flip, int c0, int c1, const u4 *__restrict__ tables,
                                              const char *__restrict__ Xs, int t0, int nt, const int (&tcls)[TPW],
                                              double (&sum)[TPW][2][4]) {
  constexpr int NS = 1 << __builtin_popcount(unsigned(PAIRED));
  const int tid = threadIdx.x, lane = tid & 63;
  const int nch = a.kp / kReflectChunk16;
  const int kk = 2 * (tid & 15), col = tid >> 4;  // this thread's two coefficients and target
  char *wp = &sh.W[0][0][col >> 4][(kk >> 3) * 320 + (col & 15) * 16 + (kk & 7) * 2];
  const int rd = (lane >> 4) * 320 + (lane & 15) * 16;
  const uint32_t *pos = ids + (scalar_read(a.first + c0) & 0xFFFFu);
  uint32_t id[NS], idn[NS];
  d2 v[8];
  auto load = [&](const uint32_t (&from)[NS], int ch) {
    int q = 0;
#pragma unroll
    for (int s = 0; s < 8; ++s)
      if (!(s & ~PAIRED))
        v[s] = *reinterpret_cast<const d2 *>(Xs + (from[q++] + uint32_t(ch * kReflectChunk16 + kk) * 8u));
  };
#pragma unroll
  for (int q = 0; q < NS; ++q) id[q] = pos[q];
  load(id, 0);
  const u4 *t = tables + (size_t(c0) * nch * a.tiles + t0) * 192 + lane;
  uint32_t mask[TPW];
  auto load_masks = [&](int cl) {
    const uint64_t *km = a.kmask + 8 * (scalar_read(a.first + cl) >> 16);
#pragma unroll
    for (int i = 0; i < TPW; ++i) mask[i] = i < nt ? uint32_t(scalar_read(km + tcls[i])) : 0u;
  };
  load_masks(c0);
  u4 av[TPW][3];
  bool use[TPW];
  auto load_table = [&](int i, int ch) {
    use[i] = (mask[i] >> ch) & 1u;
    const u4 *ti = t + (use[i] ? 192 * i : 0);
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) av[i][pl] = ti[64 * pl];
  };
#pragma unroll
  for (int i = 0; i < TPW; ++i) load_table(i, 0);
#pragma unroll 1
  for (int cl = c0; cl < c1; ++cl) {
    pos += cl + 1 < c1 ? NS : 0;
#pragma unroll
    for (int q = 0; q < NS; ++q) idn[q] = pos[q];
    f4 acc[TPW][2];
#pragma unroll
    for (int i = 0; i < TPW; ++i) acc[i][0] = acc[i][1] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int ch = 0; ch < nch; ++ch) {
      const uint2 sg = *reinterpret_cast<const uint2 *>(&sh.sign[ch * kReflectChunk16 + kk]);
      {
        double v0[8], v1[8];
#pragma unroll
        for (int s = 0; s < 8; ++s)
          if (!(s & ~PAIRED)) {
            v0[s] = v[s][0];
            v1[s] = v[s][1];
          }
        butterfly<PAIRED>(v0, sg.x, flip_of(sg.x, flip));
        butterfly<PAIRED>(v1, sg.y, flip_of(sg.y, flip));
#pragma unroll
        for (int s = 0; s < 8; ++s)
          if (!(s & ~PAIRED)) v[s] = d2{v0[s], v1[s]};
      }
      lds_barrier();  // the previous chunk's W is read
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        if (s & ~PAIRED) continue;
        const f2 x = {float(v[s][0]), float(v[s][1])};
        const uint32_t hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf2));
        const f2 r1 = {x[0] - __uint_as_float(hi << 16), x[1] - __uint_as_float(hi & 0xFFFF0000u)};
        const uint32_t mid = __builtin_bit_cast(uint32_t, __builtin_convertvector(r1, bf2));
        const f2 r2 = {r1[0] - __uint_as_float(mid << 16), r1[1] - __uint_as_float(mid & 0xFFFF0000u)};
        const uint32_t lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(r2, bf2));
        char *o = wp + s * (3 * 2 * kPlane);
        *reinterpret_cast<uint32_t *>(o) = hi;
        *reinterpret_cast<uint32_t *>(o + 2 * kPlane) = mid;
        *reinterpret_cast<uint32_t *>(o + 4 * kPlane) = lo;
      }
      const int nx = ch + 1 == nch ? 0 : ch + 1;
      if (nx == 0) {
#pragma unroll
        for (int q = 0; q < NS; ++q) id[q] = idn[q];
        load_masks(cl + 1 < c1 ? cl + 1 : cl);
      }
      load(id, nx);
      lds_barrier();
      t += size_t(a.tiles) * 192;
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        if (use[i]) {
          const bf8 ah = __builtin_bit_cast(bf8, av[i][0]), am = __builtin_bit_cast(bf8, av[i][1]),
                    al = __builtin_bit_cast(bf8, av[i][2]);
          const char *w = &sh.W[tcls[i] & PAIRED][0][0][rd];
#pragma unroll
          for (int n = 0; n < 2; ++n) {
            const bf8 bh = __builtin_bit_cast(bf8, *reinterpret_cast<const u4 *>(w + n * kPlane));
            const bf8 bm = __builtin_bit_cast(bf8, *reinterpret_cast<const u4 *>(w + (2 + n) * kPlane));
            const bf8 bl = __builtin_bit_cast(bf8, *reinterpret_cast<const u4 *>(w + (4 + n) * kPlane));
            // smallest terms first
            f4 c = acc[i][n];
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bm, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bh, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bm, c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, c, 0, 0, 0);
            acc[i][n] = c;
          }
        }
        load_table(i, nx);
      }
    }
    // one class's f32 sums into the f64 sums
#pragma unroll
    for (int i = 0; i < TPW; ++i)
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int q = 0; q < 4; ++q) sum[i][n][q] += double(acc[i][n][q]);
  }
}

// The same in bf16x3: one workgroup of eight waves per task of 32 target boxes.  A thread
// forms the butterflies (f64) of two coefficients of one target and splits every W into
// three bf16 (24 bits); the six products above 2^-24 go through v_mfma_f32_16x16x32_bf16,
// summed in f32 within a class and in f64 across the classes.  Wave w has the tiles w TPW ..,
// neighbouring tiles mostly of one parity class.
//
// Vector instructions bound it (58% of the issue cycles at p = 8, the splits most of them,
// the matrix cores at 22% beside them).  62 KB of LDS and 128 VGPRs: two workgroups per CU,
// one's products under the other's splits; at TPW = 2 the f64 sums, touched once a class,
// spill.  1M points, p = 8: 0.58 ms against 1.29 by contraction; 4M points, p = 12, levels 2
// to 5: 1.6 against 2.9.
template <int TPW>
__global__ __launch_bounds__(512, TPW <= 2 ? 4 : 2) void k_m2l_reflect_bf16(ReflectArgs a, uint32_t ntasks,
                                                                            const u4 *__restrict__ tables,
                                                                            const double *__restrict__ Xs,
                                                                            double *__restrict__ Y,
                                                                            double *__restrict__ S) {
  __shared__ ReflectBf16 sh;
  const uint32_t ti = xcd_index(ntasks, 16);
  if (ti >= ntasks) return;
  const ReflectTask task = a.tasks[ti];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (int k = tid; k < a.kp; k += 512) sh.sign[k] = uint32_t(a.parity[k]) << 29;
  const uint32_t mine = task.row0 + min(uint32_t(tid) >> 4, uint32_t(task.nrows) - 1u);
  const uint32_t *ids = a.src + (size_t(mine) * a.sets + task.set) * kReflectPositions;
  const uint32_t flip = uint32_t(a.row_flip[mine]) << 29;
  const int t0 = __builtin_amdgcn_readfirstlane(wave * TPW);
  const int nt = __builtin_amdgcn_readfirstlane(max(0, min(TPW, a.tiles - t0)));
  double sum[TPW][2][4];
  int tcls[TPW];
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int q = 0; q < 4; ++q) sum[i][n][q] = 0.0;
    tcls[i] = __builtin_amdgcn_readfirstlane(i < nt ? int(a.tile_class[t0 + i]) : 0);
  }
  __syncthreads();
  const char *x = reinterpret_cast<const char *>(Xs);
  const u4 *t4 = tables + size_t(task.table) * table_set16(a) * 64;
#define FMMH_RUN(P)                                                                                   \
  {                                                                                                   \
    const int c0 = max(int(task.first), a.run[P]), c1 = min(int(task.last), a.run[P + 1]);            \
    if (c0 < c1)                                                                                      \
      reflect_run16<P, TPW>(sh, a, ids, flip, c0, c1, t4, x, min(t0, a.tiles - 1), nt, tcls, sum);     \
  }
  FMMH_RUN(0)
  FMMH_RUN(1)
  FMMH_RUN(2)
  FMMH_RUN(3)
  FMMH_RUN(4)
  FMMH_RUN(5)
  FMMH_RUN(6)
  FMMH_RUN(7)
#undef FMMH_RUN
  // accumulator element q of lane (g, j): row 4 g + q of the tile, target j
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const uint32_t r = (lane & 15) + 16 * n;
    if (r >= task.nrows) continue;
    const bool slot = task.slot != kNone;
    double *y = slot ? S + size_t(task.slot + r * task.stride) * a.nc : Y + size_t(a.row_out[task.row0 + r]) * a.nc;
    const uint32_t out_flip = uint32_t(a.row_flip[task.row0 + r]) << 29;
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      if (i >= nt) continue;
      const double f = signed_one(flip_of(uint32_t(tcls[i]) << 29, out_flip));
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = a.tile_row[16 * (t0 + i) + 4 * (lane >> 4) + q];
        if (row >= 0) y[row] = slot ? f * sum[i][n][q] : fma(f, sum[i][n][q], y[row]);
      }
    }
  }
}

void m2l_reflect_bf16(hipStream_t s, const ReflectArgs &a, uint32_t ntasks, const uint16_t *tables, const double *Xs,
                      double *Y, double *S) {
  if (ntasks == 0) return;
  const u4 *t4 = reinterpret_cast<const u4 *>(tables);
#define FMMH_REFLECT(N)                                                                                            \
  case N:                                                                                                          \
    hipLaunchKernelGGL(k_m2l_reflect_bf16<N>, dim3(xcd_grid(ntasks, 16)), dim3(512), 0, s, a, ntasks, t4, Xs, Y, S); \
    break;
  switch ((a.tiles + 7) / 8) {
    FMMH_REFLECT(1)
    FMMH_REFLECT(2)
    FMMH_REFLECT(3)
    default:
      break;
  }
#undef FMMH_REFLECT
}

}  // namespace dev
// ---- the operator's side ---------------------------------------------------------------------

// Per target a level costs 56 classes of `tiles` row tiles this way and one product of the
// (p+1)^2 / 16 row tiles per pair by contraction.  At p = 12 (15 tiles against 11) the two
// break even near 50 pairs per box: 4M points' level 6 with 49 takes 2.9 ms against 2.0 in
// bf16x3 and 5.5 against 5.0 in f64, level 5 with 165 takes 1.4 against 2.7 and 3.0 against
// 8.2.  The levels of up to 512 boxes are short of workgroups by contraction and cost launches
// of their own (100,000 points, p = 6: 24 us), so they join the deeper ones' launch, or where
// there are none take the classes from under half of that density on, all of them or none.
std::vector<char> ReflectM2l::levels(int p, const std::vector<uint64_t> &pairs, const std::vector<uint64_t> &boxes) {
  std::vector<char> out(pairs.size(), 0);
  const double per_pair = double(((p + 1) * (p + 1) + 15) / 16), per_box = double(ReflectLayout(p, 16).tiles);
  bool large = false, any = false;
  double small_pairs = 0.0, small_boxes = 0.0;
  std::vector<size_t> small;
  for (size_t l = 0; l < pairs.size(); ++l) {
    if (pairs[l] == 0) continue;
    if (boxes[l] <= 512) {
      small.push_back(l);
      small_pairs += double(pairs[l]);
      small_boxes += double(boxes[l]);
      continue;
    }
    large = true;
    out[l] = double(pairs[l]) * per_pair >= 37.0 * double(boxes[l]) * per_box;
    any = any || out[l];
  }
  if (any || (!large && small_pairs * per_pair >= 16.0 * small_boxes * per_box))
    for (size_t l : small) out[l] = 1;
  return out;
}

bool ReflectM2l::fits(int p, bool mixed, size_t nvec) {
  const ReflectLayout lay(p, mixed ? dev::kReflectChunk16 : dev::kReflectChunk);
  return (nvec + 1) * size_t(lay.kp) * sizeof(double) <= 0xFFFFFFFFu;
}

std::vector<uint16_t> ReflectM2l::class_offsets() {
  std::vector<uint16_t> out;
  for (const auto &d : reflect_classes().offset) out.push_back(uint16_t(offset_index(d[0], d[1], d[2])));
  return out;
}

void ReflectM2l::begin(int p, bool mixed, const std::vector<size_t> &level_vec, int sets) {
  p_ = p;
  mixed_ = mixed;
  level_vec_ = level_vec;
  nvec_ = level_vec.back();
  nlevels_ = int(level_vec.size()) - 1;
  sets_ = sets;
  lay_ = ReflectLayout(p, mixed ? dev::kReflectChunk16 : dev::kReflectChunk);
  level_row_.assign(nlevels_ + 1, 0);
}

uint32_t ReflectM2l::add_tables(const std::function<const double *(int, int)> &table) {
  const size_t sz = mixed_ ? dev::reflect_table_size_bf16(lay_) : dev::reflect_table_size(lay_);
  size_t at = sz * kReflectClasses * ntables_;
  // (after the last chunk a wave reads, and drops, the next chunk's tiles)
  const size_t past = size_t(lay_.tiles + 4) * (mixed_ ? 1536 : 256);
  if (mixed_)
    tables16_h_.resize(at + sz * kReflectClasses * sets_ + past);
  else
    tables_h_.resize(at + sz * kReflectClasses * sets_ + past);
  for (int s = 0; s < sets_; ++s)
    for (int c = 0; c < kReflectClasses; ++c, at += sz) {
      if (mixed_)
        dev::reflect_table_bf16(lay_, table(s, c), tables16_h_.data() + at);
      else
        dev::reflect_table(lay_, table(s, c), tables_h_.data() + at);
    }
  const uint32_t id = ntables_;
  ntables_ += uint32_t(sets_);
  return id;
}

void ReflectM2l::add_row(int level, uint32_t out, int octant, uint32_t tables, const uint16_t *aux, uint32_t n,
                         const std::function<uint32_t(int, uint32_t)> &source) {
  // a target at the lower end of its parent has the offsets -3 .. 2 there: reflected
  static const std::vector<int> where = [] {
    std::vector<int> w(8 * 316, -1);
    for (int o = 0; o < 8; ++o)
      for (int d = 0; d < 316; ++d) {
        int dv[3];
        offset_of_index(d, dv);
        bool seen = true;
        for (int a = 0; a < 3; ++a) seen = seen && dv[a] != (((o >> (2 - a)) & 1) ? -3 : 3);
        if (seen) w[316 * o + d] = reflect_classes().position(dv, 7 & ~o);
      }
    return w;
  }();
  // a row of zeros after the last expansion stands for a source that is not there
  const size_t row_bytes = size_t(lay_.kp) * sizeof(double);
  row_out_h_.push_back(out);
  row_flip_h_.push_back(uint8_t(7 & ~octant));
  row_table_h_.push_back(tables);
  const size_t at = src_h_.size();
  src_h_.resize(at + size_t(sets_) * kReflectPositions, uint32_t(nvec_ * row_bytes));
  for (int s = 0; s < sets_; ++s)
    for (uint32_t e = 0; e < n; ++e) {
      const int pos = where[316 * octant + aux[e]];
      require(pos >= 0, "M2L schedule: V offset outside the parent's neighbours", kUnsupportedLayout);
      src_h_[at + size_t(s) * kReflectPositions + pos] = uint32_t(source(s, e) * row_bytes);
    }
  pairs_ += uint64_t(sets_) * n;
  for (int l = level + 1; l <= nlevels_; ++l) level_row_[l] = static_cast<uint32_t>(row_out_h_.size());
}

void ReflectM2l::finish() {
  const ReflectClasses &rc = reflect_classes();
  // targets per task, and the tasks that run at once: 2 workgroups of 32 or 4 of 16 per CU
  const uint32_t width = mixed_ ? 32 : 16, round = mixed_ ? 512 : 1024;
  // A task walks its classes in sequence.  Tasks beyond a whole number of rounds of the
  // workgroups that run at once would leave most of the GPU idle in the last round, so their
  // classes are split into parts of about equal cost, as many parts as fill the round.  The
  // parts of a row, and its sets, leave their sums in scratch rows that are added in order.
  uint32_t base_tasks = 0;
  for (int l = 0; l < nlevels_; ++l) base_tasks += (level_row_[l + 1] - level_row_[l] + width - 1) / width * uint32_t(sets_);
  const uint32_t whole = base_tasks / round * round;
  const uint32_t parts =
      base_tasks == whole ? 1 : std::min<uint32_t>(28, std::max<uint32_t>(1, round / (base_tasks - whole)));
  // a class costs its products (halved by every component 0) and its butterfly
  std::vector<uint32_t> cost{0};
  for (int c = 0; c < kReflectClasses; ++c)
    cost.push_back(cost.back() + (2u << __builtin_popcount(unsigned(rc.axes[c]))) +
                   uint32_t(rc.first[c + 1] - rc.first[c]));
  std::vector<int> cut{0};
  for (uint32_t q = 1; q < parts; ++q) {
    int c = cut.back() + 1;
    while (c < kReflectClasses && cost[c] * parts < q * cost.back()) ++c;
    cut.push_back(c);
  }
  cut.push_back(kReflectClasses);
  std::vector<dev::ReflectTask> tasks;
  std::vector<uint32_t> red_id, red_off{0}, red_ent;
  uint32_t nscratch = 0, seen = 0;
  level_task_.assign(nlevels_ + 1, 0);
  red_level_.assign(nlevels_ + 1, 0);
  for (int l = 0; l < nlevels_; ++l) {
    for (uint32_t r = level_row_[l]; r < level_row_[l + 1]; r += width) {
      const uint32_t n = std::min<uint32_t>(width, level_row_[l + 1] - r), t = row_table_h_[r];
      const uint32_t np = seen < whole ? 1 : parts, stride = np * uint32_t(sets_);
      seen += uint32_t(sets_);
      if (stride == 1) {
        tasks.push_back(dev::ReflectTask{r, uint16_t(n), 0, kReflectClasses, kNone, 1, t, 0});
        continue;
      }
      for (uint32_t q = 0; q < stride; ++q) {
        const uint32_t set = q / np, part = q % np;
        const int c0 = np == 1 ? 0 : cut[part], c1 = np == 1 ? kReflectClasses : cut[part + 1];
        tasks.push_back(
            dev::ReflectTask{r, uint16_t(n), uint8_t(c0), uint8_t(c1), nscratch + q, stride, t + set, set});
      }
      for (uint32_t k = 0; k < n; ++k) {
        red_id.push_back(row_out_h_[r + k]);
        for (uint32_t q = 0; q < stride; ++q) red_ent.push_back(nscratch++);
        red_off.push_back(static_cast<uint32_t>(red_ent.size()));
      }
    }
    level_task_[l + 1] = static_cast<uint32_t>(tasks.size());
    red_level_[l + 1] = static_cast<uint32_t>(red_id.size());
  }
  slots_ = uint64_t(width) * kReflectPositions * base_tasks;
  std::vector<uint32_t> first;
  for (int c = 0; c <= kReflectClasses; ++c)
    first.push_back(uint32_t(rc.first[c]) | uint32_t(c < kReflectClasses ? rc.axes[c] : 0) << 16);
  std::vector<uint64_t> kmask;
  for (int axes = 0; axes < 8; ++axes)
    for (int c = 0; c < 8; ++c) kmask.push_back(lay_.steps(axes, c, mixed_ ? dev::kReflectChunk16 : 4));
  // every index array in one allocation and one copy
  std::vector<uint8_t> blob;
  auto put = [&](const auto &v) {
    const size_t at = (blob.size() + 63) / 64 * 64, n = v.size() * sizeof(v[0]);
    blob.resize(at + n);
    if (n) std::memcpy(blob.data() + at, v.data(), n);
    return at;
  };
  const size_t o_first = put(first), o_kmask = put(kmask), o_parity = put(lay_.parity), o_rows = put(lay_.tile_row),
               o_class = put(lay_.tile_class), o_perm = put(lay_.perm), o_tasks = put(tasks), o_out = put(row_out_h_),
               o_flip = put(row_flip_h_), o_src = put(src_h_), o_rid = put(red_id), o_roff = put(red_off),
               o_rent = put(red_ent);
  index_.upload(blob);
  auto at = [&](size_t o) { return static_cast<const void *>(index_.ptr + o); };
  perm_ = static_cast<const int32_t *>(at(o_perm));
  red_id_ = static_cast<const uint32_t *>(at(o_rid));
  red_off_ = static_cast<const uint32_t *>(at(o_roff));
  red_ent_ = static_cast<const uint32_t *>(at(o_rent));
  args_.first = static_cast<const uint32_t *>(at(o_first));
  args_.kmask = static_cast<const uint64_t *>(at(o_kmask));
  args_.parity = static_cast<const uint8_t *>(at(o_parity));
  args_.tile_row = static_cast<const int32_t *>(at(o_rows));
  args_.tile_class = static_cast<const uint8_t *>(at(o_class));
  args_.tasks = static_cast<const dev::ReflectTask *>(at(o_tasks));
  args_.row_out = static_cast<const uint32_t *>(at(o_out));
  args_.row_flip = static_cast<const uint8_t *>(at(o_flip));
  args_.src = static_cast<const uint32_t *>(at(o_src));
  scratch_.alloc(size_t(nscratch) * lay_.nc);
  if (mixed_)
    tables16_.upload(tables16_h_);
  else
    tables_.upload(tables_h_);
  sorted_.alloc((nvec_ + 1) * lay_.kp);
  hip_check(hipMemset(sorted_.ptr + nvec_ * lay_.kp, 0, size_t(lay_.kp) * sizeof(double)), "reflection zero row");
  args_.nc = lay_.nc;
  args_.kp = lay_.kp;
  args_.tiles = lay_.tiles;
  std::copy(rc.run.begin(), rc.run.end(), args_.run);
  args_.sets = sets_;
  std::vector<uint32_t>().swap(row_out_h_);
  std::vector<uint32_t>().swap(src_h_);
  std::vector<uint32_t>().swap(row_table_h_);
  std::vector<uint8_t>().swap(row_flip_h_);
  std::vector<double>().swap(tables_h_);
  std::vector<uint16_t>().swap(tables16_h_);
}

size_t ReflectM2l::bytes() const {
  return tables_.bytes() + tables16_.bytes() + sorted_.bytes() + scratch_.bytes() + index_.bytes();
}

void ReflectM2l::launch(hipStream_t s, int first, int last, const double *X, double *Y,
                        const std::function<void(const std::function<void()> &)> &contract) {
  if (level_task_.empty()) return;
  const uint32_t t0 = level_task_[first], t1 = level_task_[last + 1];
  if (t1 == t0) return;
  // the sources are of the targets' levels
  while (!has(first)) ++first;
  while (!has(last)) --last;
  const size_t vec0 = level_vec_[first], vec1 = level_vec_[last + 1];
  dev::reflect_sort(s, lay_.nc, lay_.kp, vec1 - vec0, perm_, X + vec0 * lay_.nc, sorted_.ptr + vec0 * lay_.kp);
  dev::ReflectArgs args = args_;
  args.tasks += t0;
  contract([&] {
    if (mixed_)
      dev::m2l_reflect_bf16(s, args, t1 - t0, tables16_.ptr, sorted_.ptr, Y, scratch_.ptr);
    else
      dev::m2l_reflect_f64(s, args, t1 - t0, tables_.ptr, sorted_.ptr, Y, scratch_.ptr);
  });
  const uint32_t r0 = red_level_[first], r1 = red_level_[last + 1];
  if (r1 > r0)
    dev::reduce_slots(s, p_, r1 - r0, red_id_ + r0, red_off_ + r0, red_ent_, 0, scratch_.ptr,
                      nullptr, Y);
}

}  // namespace fmmh
