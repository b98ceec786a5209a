// reflect.hpp -- the dense M2L by reflection classes: host layout and launch wrappers of
// reflect.hip.
//
// Reflecting an offset in a coordinate plane changes the sign of the harmonics that are odd
// in that coordinate, so T(sigma a) = D_sigma T(a) D_sigma with D_sigma diagonal and +-1
// (the tables of CONVENTIONS §3.12 have this to the last bit).  The offsets are then the
// reflections of 56 classes (|dx|, |dy|, |dz|), and a class's sources share one product:
// with the coefficients sorted by their parities c = (odd in x, y, z),
//   L_r += sum_k T_rk(a) W_c(r)[k],   W_c[k] = sum_sigma chi_c(sigma) chi_c(k)(sigma) M_sigma[k],
// the W a butterfly of the sources' multipoles over the signs sigma.  A component of 1 or 2
// has both signs in a target's list, 3 only one (that of the target's octant, made positive
// by reflecting the target and its sources as a whole), and a component of 0 leaves T_rk = 0
// unless r and k have the same parity in it.  Per target box the products fall from 189
// tables to 39.5 full ones.
#pragma once

#include <hip/hip_runtime.h>

#include <array>
#include <cstdint>
#include <functional>
#include <vector>

#include "devbuf.hpp"

namespace fmmh {

constexpr int kReflectClasses = 56;

// Degree-independent: the classes, sorted by their paired components.
struct ReflectClasses {
  std::array<std::array<int, 3>, kReflectClasses> offset;  // the class's offset, components >= 0
  std::array<int, kReflectClasses> axes;                   // nonzero components: 4 x + 2 y + z
  std::array<int, kReflectClasses> paired;                 // components 1 or 2
  std::array<int, kReflectClasses + 1> first;              // first position of its signs
  std::array<int, 9> run;                                  // first class of every `paired`
  // position (0 .. 188) of offset d of a target whose axes in `flip` are reflected
  int position(const int d[3], int flip) const;
};
constexpr int kReflectPositions = 189;
const ReflectClasses &reflect_classes();

// The coefficients of degree p by parity class: sorted position -> coefficient (-1: padding
// to a multiple of `pad`), and the row tiles of 16 (each of one class).
struct ReflectLayout {
  int p = 0, nc = 0, kp = 0, tiles = 0;
  std::vector<int32_t> perm;        // kp
  std::vector<uint8_t> parity;      // kp
  std::vector<int32_t> tile_row;    // tiles x 16: coefficient or -1
  std::vector<uint8_t> tile_class;  // tiles
  ReflectLayout(int p, int pad);
  // bit s: the sorted positions s width .. s width + width - 1 hold a parity that class c's
  // rows meet when only `axes` are nonzero
  uint64_t steps(int axes, int c, int width) const;
};

namespace dev {

// One workgroup's share: up to 16 (f64) or 32 (bf16x3) target rows from row0 (nrows of them held), classes first ..
// last - 1, added to the boxes' locals or, with slot != kNone, stored in scratch rows
// slot, slot + stride, ...
struct ReflectTask {
  uint32_t row0;
  uint16_t nrows;
  uint8_t first, last;
  uint32_t slot, stride;
  uint32_t table, set;  // its class tables, and the set of sources that they take
};

struct ReflectArgs {
  int nc, kp, tiles;
  int run[9];                    // first class of every set of paired components
  const uint32_t *first;         // 57: first position of every class, its axes << 16
  const uint64_t *kmask;         // [8 axes][8 classes] steps
  const uint8_t *parity;         // kp
  const int32_t *tile_row;       // tiles x 16
  const uint8_t *tile_class;     // tiles
  const ReflectTask *tasks;
  int sets;                      // sets of sources per row
  const uint32_t *row_out;       // target expansions
  const uint8_t *row_flip;       // their reflected axes
  const uint32_t *src;           // rows x sets x 189: byte offset in Xs of the source at every position
};

constexpr int kReflectChunk = 16;  // sorted positions per step of the f64 kernel

// f64 tables of the 56 classes: [class][chunk of 16][tile][half][lane][2]
size_t reflect_table_size(const ReflectLayout &l);
void reflect_table(const ReflectLayout &l, const double *table_colmajor, double *out);
// Xs[box][kp] = X[box][perm], zero in the padding; the kernel also reads a row of zeros that
// stands for a source that is not there
void reflect_sort(hipStream_t s, int nc, int kp, size_t nboxes, const int32_t *perm, const double *X, double *Xs);
// tasks of 16 rows
void m2l_reflect_f64(hipStream_t s, const ReflectArgs &a, uint32_t ntasks, const double *tables, const double *Xs,
                     double *Y, double *S);

// bf16x3: chunks of 32, tables [class][chunk][tile][plane][lane][8]
constexpr int kReflectChunk16 = 32;
size_t reflect_table_size_bf16(const ReflectLayout &l);
void reflect_table_bf16(const ReflectLayout &l, const double *table_colmajor, uint16_t *out);
// tasks of 32 rows
void m2l_reflect_bf16(hipStream_t s, const ReflectArgs &a, uint32_t ntasks, const uint16_t *tables, const double *Xs,
                      double *Y, double *S);

}  // namespace dev
// The levels of an operator whose dense M2L runs by reflection classes.  A row is one real
// target expansion: it adds, for each of `sets` sets of class tables, the products with the
// sources that its V list names for that set (the Laplace operator has one set; a complex
// table is two sets, its real and its imaginary part).
class ReflectM2l {
 public:
  // Which levels take it: V pairs and boxes per level (0 pairs: not asked).
  static std::vector<char> levels(int p, const std::vector<uint64_t> &pairs, const std::vector<uint64_t> &boxes);
  // Whether nvec source expansions fit the kernels' 32-bit byte offsets.
  static bool fits(int p, bool mixed, size_t nvec);
  // (|dx|, |dy|, |dz|) of the classes as offset indices, in the order of add_tables
  static std::vector<uint16_t> class_offsets();

  // level_vec: first expansion of every level, and one past the last level's
  void begin(int p, bool mixed, const std::vector<size_t> &level_vec, int sets);
  // `sets` sets of tables (column-major (p+1)^2 x (p+1)^2, set s of class c at table(s, c));
  // returns their index for add_row
  uint32_t add_tables(const std::function<const double *(int, int)> &table);
  // rows of one level after another, in ascending levels; source(set, e): expansion of V
  // entry e (offset indices aux[0 .. n - 1]) of a target of the given octant
  void add_row(int level, uint32_t out, int octant, uint32_t tables, const uint16_t *aux, uint32_t n,
               const std::function<uint32_t(int, uint32_t)> &source);
  void finish();

  bool has(int level) const { return level + 1 < int(level_task_.size()) && level_task_[level + 1] > level_task_[level]; }
  uint64_t pairs() const { return pairs_; }  // (row, source) pairs, and the column slots issued
  uint64_t slots() const { return slots_; }
  size_t bytes() const;
  // M2L of the levels first .. last: X the multipoles, Y the locals; contract(f) runs the
  // kernel launch f
  void launch(hipStream_t s, int first, int last, const double *X, double *Y,
              const std::function<void(const std::function<void()> &)> &contract);

 private:
  int p_ = 0, nlevels_ = 0, sets_ = 1;
  bool mixed_ = false;
  size_t nvec_ = 0;
  std::vector<size_t> level_vec_;
  uint64_t pairs_ = 0, slots_ = 0;
  ReflectLayout lay_{0, 16};
  dev::ReflectArgs args_{};
  std::vector<uint32_t> row_out_h_, src_h_, row_table_h_, level_row_;
  std::vector<uint8_t> row_flip_h_;
  std::vector<double> tables_h_;
  std::vector<uint16_t> tables16_h_;
  uint32_t ntables_ = 0;
  DevBuf<uint8_t> index_;  // the index arrays, also those of the scratch rows' reduction
  const int32_t *perm_ = nullptr;
  const uint32_t *red_id_ = nullptr, *red_off_ = nullptr, *red_ent_ = nullptr;
  DevBuf<uint16_t> tables16_;
  DevBuf<double> tables_, sorted_, scratch_;
  std::vector<uint32_t> level_task_, red_level_;
};

}  // namespace fmmh
