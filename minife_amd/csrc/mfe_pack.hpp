// Packed stencil values: an exact fixed-point form of the values of a box
// layout (here the symmetric layout's 14 upper slots, mfe_boxsym.hpp).
//
// The layout stores a (block, plane, slot) group as 256 consecutive values,
// one per row of a 16 x 16 block.  For each packed slot the group's values
// are whole multiples k of a power of two q (the largest power of two that
// divides every one of them: the assembled entries are sums of element
// terms, so even the analytically zero ones -- a cube's face neighbours,
// about 1e-9 of the diagonal -- are multiples of the terms' last place).
// The group stores a base kb q and q side by side and each value an unsigned
// field f of W bits: f = 0 stands for +0.0, f = 1 for 1.0 (the padding,
// Dirichlet rows and zeroed columns), and otherwise the value is (kb + f) * q,
// formed as f q + kb q and exact (kb + f is an integer below 2^53, or 2^24
// in FP32, and scaling by a power of two is exact; the plan checks every value).
// kb = kmax - (2^W - 1), so the group's multiples fit W bits when they span at
// most 2^W - 3.  One flag per (block, plane) is 1 when any of its packed values
// is +0.0 or 1.0 (a code can occur), else 0: the SpMV then skips the code tests.
//
// A form gives each slot a width: the cube's slots (every slot but the
// analytically zero ones, NEAR) a narrow width, the NEAR slots the same
// narrow width, a wide one, or none (read at full width from the layout).
// Fields: per (block, plane) and row, the slots are taken in groups of G
// consecutive slots (an SpMV that reads a row's slots in several steps can
// load one group per step); a group's fields follow each other in slot order
// from bit 0 of its first word (a field may straddle two words), and its
// words follow the previous group's.  A (block, plane)'s word w of the
// thread-t row is PW[((block * gz + plane) * words + w) * 256 + t].  The
// widths are compile-time constants of the form, so every load is issued
// without a branch.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>

namespace mfe {

// The forms; kPackNone: the full values.
enum PackForm {
  kPackNone = 0,
  kPackAll16 = 1,          // every slot 16 bits
  kPackCube16Near32 = 2,   // cube 16, near 32 (FP64)
  kPackCube16 = 3,         // cube 16, near at full width
  kPackAll12 = 4,          // every slot 12 bits
  kPackCube12Near24 = 5,   // cube 12, near 24
  kPackAll10 = 6,          // every slot 10 bits
  kPackCube10Near22 = 7    // cube 10, near 22
};
constexpr int kPackForms = 8;
// the field widths whose fits the first pass records (one slot mask per width)
constexpr int kPackWidths[] = {10, 12, 16, 22, 24, 32};
constexpr int kPackNumWidths = 6;

__host__ __device__ constexpr int pack_narrow(int f) {
  return f == kPackAll16 || f == kPackCube16Near32 || f == kPackCube16 ? 16
       : f == kPackAll12 || f == kPackCube12Near24                      ? 12
       : f == kPackAll10 || f == kPackCube10Near22                      ? 10
                                                                         : 0;
}
__host__ __device__ constexpr int pack_wide(int f) {
  return f == kPackCube16Near32 ? 32 : f == kPackCube12Near24 ? 24 : f == kPackCube10Near22 ? 22 : 0;
}
__host__ __device__ constexpr bool pack_all(int f) {
  return f == kPackAll16 || f == kPackAll12 || f == kPackAll10;
}

__host__ __device__ constexpr int pack_rank(unsigned mask, int i) {
  return __builtin_popcount(mask & ((1u << i) - 1u));
}

// NS slots; NEAR: the slots of a cube's analytically zero entries (their
// values span tens of thousands of quanta per group and more, a narrow
// width does not hold them at most sizes); G: slots per group (NS a
// multiple of G).
template <int NS, unsigned NEAR, int G>
struct PackMap {
  static constexpr int kSlots = NS;
  static constexpr unsigned kAll = (1u << NS) - 1u;
  static constexpr unsigned kNear = NEAR;
  static constexpr unsigned kCube = kAll & ~NEAR;
  // bits of slot s (0: read at full width)
  __host__ __device__ static constexpr int width(int f, int s) {
    return !((kAll >> s) & 1u) ? 0
         : !((NEAR >> s) & 1u) || pack_all(f) ? pack_narrow(f)
                                              : pack_wide(f);
  }
  __host__ __device__ static constexpr bool packed(int f, int s) { return width(f, s) > 0; }
  __host__ __device__ static constexpr bool full(int f, int s) { return !packed(f, s); }
  // the slots with a field
  __host__ __device__ static constexpr unsigned mask(int f) {
    unsigned m = 0;
    for (int s = 0; s < NS; ++s)
      if (packed(f, s)) m |= 1u << s;
    return m;
  }
  // bit offset of slot s within its group
  __host__ __device__ static constexpr int gbit(int f, int s) {
    int b = 0;
    for (int u = (s / G) * G; u < s; ++u) b += width(f, u);
    return b;
  }
  __host__ __device__ static constexpr int gwords(int f, int g) {
    return (gbit(f, g * G + G - 1) + width(f, g * G + G - 1) + 31) / 32;
  }
  __host__ __device__ static constexpr int gbase(int f, int g) {
    int b = 0;
    for (int h = 0; h < g; ++h) b += gwords(f, h);
    return b;
  }
  __host__ __device__ static constexpr int words(int f) { return gbase(f, NS / G); }
  // the first word of slot s's field, its shift in it, and whether the field
  // goes on into the next word
  __host__ __device__ static constexpr int word_of(int f, int s) {
    return gbase(f, s / G) + gbit(f, s) / 32;
  }
  __host__ __device__ static constexpr int shift_of(int f, int s) { return gbit(f, s) % 32; }
  __host__ __device__ static constexpr bool straddles(int f, int s) {
    return shift_of(f, s) + width(f, s) > 32;
  }
  // whether word w holds bits of any of slots lo .. lo+cnt-1
  __host__ __device__ static constexpr bool word_needed(int f, int w, int lo, int cnt) {
    for (int s = lo; s < lo + cnt; ++s)
      if (packed(f, s) && (word_of(f, s) == w || (straddles(f, s) && word_of(f, s) + 1 == w)))
        return true;
    return false;
  }
};

// The layout of form F as constant tables (kernels index them with unrolled
// loop counters, so every entry folds to a constant).
constexpr int kPackMaxSlots = 32, kPackMaxWords = 32;
template <typename P, int F>
struct PackLayout {
  int width[kPackMaxSlots] = {}, word[kPackMaxSlots] = {}, shift[kPackMaxSlots] = {};
  bool straddle[kPackMaxSlots] = {};
  unsigned slots_of_word[kPackMaxWords] = {};  // the slots with bits in word w
  int words = 0;
  unsigned mask = 0;  // the slots with a field
  constexpr PackLayout() {
    words = P::words(F);
    mask = P::mask(F);
    for (int s = 0; s < P::kSlots; ++s) {
      width[s] = P::width(F, s);
      if (!width[s]) continue;
      word[s] = P::word_of(F, s);
      shift[s] = P::shift_of(F, s);
      straddle[s] = P::straddles(F, s);
      slots_of_word[word[s]] |= 1u << s;
      if (straddle[s]) slots_of_word[word[s] + 1] |= 1u << s;
    }
  }
  // whether word w holds bits of any of slots lo .. lo+cnt-1
  __host__ __device__ constexpr bool needed(int w, int lo, int cnt) const {
    return (slots_of_word[w] & (((1u << cnt) - 1u) << lo)) != 0u;
  }
};

// The symmetric layout's upper slots u (stencil slot 13 + u): the same-plane
// face neighbours (stencil slots 14, 16) and the next plane's (22) are the
// near-zero ones; one group.
using SymPack = PackMap<14, (1u << 1) | (1u << 3) | (1u << 9), 14>;

// Field of nw bits at bit sh of w[0] (and w[1] when it straddles: a 32-bit
// field does unless sh is 0); nw and sh are constants where the caller's
// loops are unrolled.
__host__ __device__ inline unsigned pack_field(const unsigned* w, int nw, int sh) {
  const unsigned mask = nw >= 32 ? ~0u : (1u << nw) - 1u;
  if (sh + nw <= 32) return (w[0] >> sh) & mask;
  return ((w[0] >> sh) | (w[1] << (32 - sh))) & mask;
}

// The value (kb + f) q of field f from the base kbq = kb q: f q and kb q are
// whole multiples of q and exact, and so is their sum, the stored value (two
// instructions with one scalar operand each; an fma would need a copy of one).
// CODES: the plane may hold +0.0 or 1.0 (the value is computed for every f and
// the codes selected afterwards, so no branch separates the arithmetic from the
// loads of kbq and q); else f >= 2.
template <typename T, bool CODES>
__device__ __forceinline__ T pack_decode(T kbq, T q, unsigned f) {
  const T v = (T)f * q + kbq;
  if constexpr (!CODES) {
    return v;
  } else {
    const T v0 = f == 0u ? T(0) : v;
    return f == 1u ? T(1) : v0;
  }
}

}  // namespace mfe
