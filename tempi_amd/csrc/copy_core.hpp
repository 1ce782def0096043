// copy_core.hpp -- the per-unit strided copy shared by the single-copy
// kernels (kernels.hip) and the batched queue kernel (batch.hip).
//
// A copy is `units` work units; unit u is segment (u % nseg) of row
// (u / nseg).  A group of P lanes moves one unit as U words of W bytes per
// lane, the P lanes touching consecutive words; each thread issues the loads
// of K = units_in_flight(U) units before storing any of them.  Loads and
// stores may sit at any byte address (gfx9 global memory instructions accept
// that), so a row's words are counted from its first byte whatever its
// alignment, and the L % W bytes after the last whole word are the same for
// every row of a copy: one lane moves them as 8, 4, 2 and 1 bytes.
#pragma once

#include "internal.hpp"

#include <hip/hip_runtime.h>

namespace tempi {

// n / d for 32-bit n by multiply-high and shift (Granlund and Montgomery,
// "Division by Invariant Integers using Multiplication", PLDI 1994, fig. 4.1):
// with l = ceil(log2 d) and m = floor(2^32 (2^l - d) / d) + 1,
// n / d = (mulhi(n, m) + n) >> l, the sum taken in 64 bits.
struct FastDiv {
  uint32_t mul = 1;
  uint32_t shift = 0;
  __host__ __device__ __forceinline__ uint32_t div(uint32_t n) const {
    const uint32_t t = (uint32_t)(((uint64_t)n * mul) >> 32);
    return (uint32_t)(((uint64_t)t + n) >> shift);
  }
};

FastDiv make_fastdiv(uint32_t d);

struct KParams {
  const char *src; // first byte of row 0 on the source side
  char *dst;       // first byte of row 0 on the destination side
  int64_t L;       // bytes per row
  uint32_t units;  // rows * nseg
  uint32_t nseg;   // segments per row
  FastDiv segdiv;
  uint32_t words; // L / W
  int32_t nrd;    // row dimensions
  uint32_t cnt[kMaxRowDims];
  FastDiv div[kMaxRowDims];
  int64_t str[kMaxRowDims];
  uint32_t signal; // nonzero: the launch signals its completion (kernels.hip)
  uint32_t tail;   // L % W
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <int W> struct WordT;
template <> struct WordT<16> { typedef u32x4 T; };
template <> struct WordT<12> { typedef u32x3 T; };
template <> struct WordT<8> { typedef u32x2 T; };
template <> struct WordT<4> { typedef uint32_t T; };
template <> struct WordT<2> { typedef uint16_t T; };
template <> struct WordT<1> { typedef uint8_t T; };

// load W bytes from any byte address; NT marks the load nontemporal (the
// line is filled for this access and is first in line for eviction)
template <int W, bool NT>
__device__ __forceinline__ typename WordT<W>::T load_word(const char *p) {
  typedef typename WordT<W>::T T;
  typedef T Tu __attribute__((aligned(1)));
  if constexpr (NT) {
    return __builtin_nontemporal_load(reinterpret_cast<const Tu *>(p));
  } else {
    return *reinterpret_cast<const Tu *>(p);
  }
}

// store W bytes to any byte address
template <int W, bool NT>
__device__ __forceinline__ void store_word(char *p, typename WordT<W>::T v) {
  typedef typename WordT<W>::T T;
  typedef T Tu __attribute__((aligned(1)));
  if constexpr (NT) {
    __builtin_nontemporal_store(v, reinterpret_cast<Tu *>(p));
  } else {
    *reinterpret_cast<Tu *>(p) = v;
  }
}

// byte offset of row `row` on the strided side
__host__ __device__ __forceinline__ int64_t row_offset(const KParams &p,
                                                       uint32_t row) {
  int64_t off = 0;
  uint32_t q = row;
#pragma unroll
  for (int k = 0; k < kMaxRowDims; ++k) {
    if (k >= p.nrd) {
      break;
    }
    if (k == p.nrd - 1) {
      off += (int64_t)q * p.str[k];
      break;
    }
    const uint32_t nq = p.div[k].div(q);
    off += (int64_t)(q - nq * p.cnt[k]) * p.str[k];
    q = nq;
  }
  return off;
}

// Addresses of one work unit, computed before any of the thread's loads.
struct UnitAddr {
  const char *s; // first byte of the row on the source side
  char *d;       // first byte of the row on the destination side
  uint32_t w;    // first word index of this lane
  uint32_t n;    // words of the row (0: nothing to move)
  bool tail;     // this lane moves the row's last L % W bytes
};

// Address phase of work unit `u` (wave-uniform when P == 64).  DIR 0 = pack
// (strided -> packed), 1 = unpack (packed -> strided).  A row's last segment
// holds its tail; the lane that would move the next word moves it.  The
// host-side emulation of a copy (kernels.hip) runs the same code.
template <int P, int W, int U, bool WHOLE, int DIR>
__host__ __device__ __forceinline__ UnitAddr unit_addr(const KParams &p,
                                                       uint32_t u,
                                                       uint32_t lane) {
  const uint32_t row = p.nseg == 1 ? u : p.segdiv.div(u);
  const uint32_t seg = u - row * p.nseg;
  const int64_t soff = row_offset(p, row);
  const int64_t poff = (int64_t)row * p.L;
  UnitAddr a;
  a.s = p.src + (DIR == 0 ? soff : poff);
  a.d = p.dst + (DIR == 0 ? poff : soff);
  a.w = seg * (uint32_t)(P * U) + lane;
  a.n = p.words;
  a.tail = !WHOLE && seg == p.nseg - 1 && lane == p.words % P;
  return a;
}

// Byte offset, within a row's tail of `tail` bytes, of its piece of N bytes
// (N = 8, 4, 2 or 1, present when the bit N of `tail` is set): after the
// larger pieces.
template <int N>
__host__ __device__ constexpr uint32_t tail_at(uint32_t tail) {
  return tail & ~(uint32_t)(2 * N - 1);
}

// The tails of K units in registers, between the load and the store phase.
// `tail` is the same for every row, so the tests of its bits do not diverge.
template <int W> struct TailWords {
  u32x2 v8;
  uint32_t v4;
  uint16_t v2;
  uint8_t v1;
};

template <int W, bool NT>
__device__ __forceinline__ void load_tail(TailWords<W> *t, const char *s,
                                          uint32_t tail) {
  if constexpr (W > 8) {
    if (tail & 8) {
      t->v8 = load_word<8, NT>(s);
    }
  }
  if constexpr (W > 4) {
    if (tail & 4) {
      t->v4 = load_word<4, NT>(s + tail_at<4>(tail));
    }
  }
  if constexpr (W > 2) {
    if (tail & 2) {
      t->v2 = load_word<2, NT>(s + tail_at<2>(tail));
    }
  }
  if (tail & 1) {
    t->v1 = load_word<1, NT>(s + tail_at<1>(tail));
  }
}

template <int W, bool NT>
__device__ __forceinline__ void store_tail(const TailWords<W> &t, char *d,
                                           uint32_t tail) {
  if constexpr (W > 8) {
    if (tail & 8) {
      store_word<8, NT>(d, t.v8);
    }
  }
  if constexpr (W > 4) {
    if (tail & 4) {
      store_word<4, NT>(d + tail_at<4>(tail), t.v4);
    }
  }
  if constexpr (W > 2) {
    if (tail & 2) {
      store_word<2, NT>(d + tail_at<2>(tail), t.v2);
    }
  }
  if (tail & 1) {
    store_word<1, NT>(d + tail_at<1>(tail), t.v1);
  }
}

// s_waitcnt immediate for vmcnt(0) alone on gfx9 (expcnt and lgkmcnt at
// their maxima, 7 and 15, so only the vector memory counter is waited on)
constexpr int kWaitLoads = 0x0F70;

// The words of one unit, held in registers between the load and store phases.
template <int W, int U> struct UnitWords {
  typename WordT<W>::T v[U];
};

// units a thread keeps in flight: enough for four loads per lane
__host__ __device__ constexpr int units_in_flight(int U) {
  return U >= 4 ? 1 : 4 / U;
}

// Move units first, first + stride, ... (K of them, those below `end`) in
// three phases: every unit's addresses, then every load, then every store.
// Keeping the loads in one straight run matters: with the address arithmetic
// of later units between them, the compiler put a wait for the earlier loads
// in front of the later ones (register reuse across the grid-stride loop),
// and each unit paid a full memory round trip of its own.  NTS / NTL:
// nontemporal stores / loads of the body words.
template <int P, int W, int U, bool WHOLE, int DIR, bool NTS, bool NTL,
          int K = units_in_flight(U)>
__device__ __forceinline__ void copy_units(const KParams &p, uint32_t first,
                                           uint32_t stride, uint32_t end,
                                           uint32_t lane) {
  UnitAddr a[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    uint32_t u = first + k * stride;
    if constexpr (P == 64 && K == 1) {
      // wave-uniform: the row arithmetic runs on the scalar unit (with
      // several units in flight their state would overflow the SGPRs)
      u = __builtin_amdgcn_readfirstlane(u);
    }
    if (u < end) {
      a[k] = unit_addr<P, W, U, WHOLE, DIR>(p, u, lane);
    } else {
      a[k].s = nullptr;
      a[k].d = nullptr;
      a[k].w = 0;
      a[k].n = 0;
      a[k].tail = false;
    }
  }
  UnitWords<W, U> v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const uint32_t w = a[k].w + j * P;
      if (w < a[k].n) {
        v[k].v[j] = load_word<W, NTL>(a[k].s + (size_t)w * W);
      }
    }
  }
  TailWords<W> t[K];
  const int64_t tail_off = (int64_t)p.words * W;
  if constexpr (!WHOLE) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (a[k].tail) {
        load_tail<W, NTL>(&t[k], a[k].s + tail_off, p.tail);
      }
    }
  }
  // Every load lands before any store, by one wait in straight-line code.
  // Left to the compiler, the waits sit inside the per-word store
  // conditions; on a path that skips a store its load counts as still
  // pending at the loop back edge, and the next iteration waits for it in
  // the middle of its own loads.
  __builtin_amdgcn_s_waitcnt(kWaitLoads);
#pragma unroll
  for (int k = 0; k < K; ++k) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const uint32_t w = a[k].w + j * P;
      if (w < a[k].n) {
        store_word<W, NTS>(a[k].d + (size_t)w * W, v[k].v[j]);
      }
    }
  }
  if constexpr (!WHOLE) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (a[k].tail) {
        store_tail<W, NTS>(t[k], a[k].d + tail_off, p.tail);
      }
    }
  }
}

constexpr int kBlock = 256;

// The variant list, as X(index, P, W, U, NT): P lanes per row, W-byte words,
// U words per lane per unit, and which side's accesses are nontemporal:
// kPlain none, kLoads the loads, kStrided those of the strided side (a pack's
// loads, an unpack's stores).
enum Nontemporal { kPlain, kLoads, kStrided };
#define TEMPI_VARIANTS(X)                                                      \
  X(0, 8, 16, 2, kStrided)  /* as 5, strided side nontemporal      */          \
  X(1, 64, 16, 4, kPlain)   /* long rows, 4 KiB per unit           */          \
  X(2, 32, 16, 2, kStrided) /* long rows, strided side nontemporal */          \
  X(3, 32, 16, 2, kLoads)   /* long rows, nontemporal loads        */          \
  X(4, 16, 16, 2, kPlain)   /* rows around 256 B - 1 KiB           */          \
  X(5, 8, 16, 2, kPlain)    /* rows around 128 - 256 B             */          \
  X(6, 4, 16, 2, kPlain)    /* rows around 64 - 128 B              */          \
  X(7, 1, 16, 4, kPlain)    /* lane per row, 16-B words            */          \
  X(8, 1, 8, 4, kPlain)     /* lane per row, 8-B words             */          \
  X(9, 1, 4, 4, kPlain)     /* lane per row, 4-B words             */          \
  X(10, 16, 4, 4, kPlain)   /* 4-B words across 16 lanes           */          \
  X(11, 1, 1, 16, kPlain)   /* lane per row, bytes                 */          \
  X(12, 1, 12, 1, kPlain)   /* lane per row, 12-B words (3 floats) */          \
  X(13, 8, 16, 2, kLoads)   /* as 5, nontemporal loads             */          \
  X(14, 4, 16, 2, kStrided) /* as 6, strided side nontemporal      */          \
  X(15, 4, 16, 2, kLoads)   /* as 6, nontemporal loads             */          \
  X(16, 1, 12, 1, kLoads)   /* as 12, nontemporal loads            */          \
  X(17, 4, 8, 1, kLoads)    /* rows of 8 - 32 B, nontemporal loads */          \
  X(18, 1, 8, 4, kLoads)    /* as 8, nontemporal loads             */

// nontemporal stores / loads of a variant's kernel in direction DIR
constexpr bool nt_stores(Nontemporal nt, int dir) {
  return nt == kStrided && dir == 1;
}
constexpr bool nt_loads(Nontemporal nt, int dir) {
  return nt == kLoads || (nt == kStrided && dir == 0);
}

// Work units of one launch stay below 2^31.  The kernels index units with
// 32-bit counters that step by at most (grid * groups * units in flight)
// < 2^28 past the last unit, so no index wraps; launch_copy splits a larger
// copy along its outer row dimensions.
constexpr int64_t kMaxUnits = 1ll << 31;

// work units of a copy with `variant`
int64_t units_of(const Geom &g, int variant);

// Fill the kernel parameters of one copy with `variant`; `whole`: its rows
// are whole words.  A copy of kMaxUnits units or more is reported as
// TEMPI_ERR_UNSUPPORTED.
int fill_kparams(const Geom &g, const char *strided, char *packed, int dir,
                 int variant, KParams *p, bool *whole);

} // namespace tempi
