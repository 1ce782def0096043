// kernels.hip -- gfx950 strided-block pack/unpack kernels and their host-side
// geometry, alignment and launch code.
//
// Every pack or unpack is a set of rows of L bytes (geometry in
// internal.hpp).  A work unit is one segment of one row; a group of P lanes
// of a 64-wide wavefront moves a segment as U words of W bytes per lane, the
// P lanes of a group touching consecutive words so that each load and store
// instruction of the group covers P*W contiguous bytes.  gfx950's global
// loads and stores accept any byte address, so neither side's alignment
// changes how a row is cut: its words start at its first byte and its last
// L % W bytes are a tail of at most four pieces, the same for every row.  An
// earlier form stored only to W-aligned addresses and copied the head and
// tail bytes of each row one by one, every byte its own store and most of
// them a round trip of their own.  Unpacks by the same variant, three buffer
// pairs in turn, the strided side 5 B past a boundary, before and now:
//   2^20 rows of 32 B at a 512-B stride    67.5 -> 28.4 us  (variant 5)
//   2^19 rows of 64 B at a 1777-B stride   44.9 -> 34.4 us  (variant 5)
//   2^17 rows of 256 B at a 700-B stride   27.4 -> 22.5 us  (variant 10)
//   2^16 rows of 512 B at a 3000-B stride  24.7 -> 19.4 us  (variant 10)
// What is left is the traffic of partial lines.
// When L % W == 0 the WHOLE instantiation has no tail.
//
// reference: include/pack_kernels.cuh:19-120 (grid_x_memcpy_aligned,
// pack_2d/unpack_2d) and :350-433 (pack_3d/unpack_3d).  The index map is the
// same -- packed[r*L + x] = strided[start + sum_k idx_k(r)*stride_k + x],
// with the object index as the outermost dimension -- but offsets are 64-bit
// (the reference's `unsigned bi = y*stride1`, :82/:382, wraps past 4 GiB),
// the word width honours the runtime pointers and strides, not only the
// block length and start (:129-157), and the object loop is part of the
// parallel row space instead of a serial loop (:372).
#include "copy_core.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>

namespace tempi {

FastDiv make_fastdiv(uint32_t d) {
  FastDiv f;
  uint32_t l = 0;
  while (l < 32 && (1ull << l) < d) {
    ++l;
  }
  const unsigned __int128 num =
      ((unsigned __int128)1 << 32) * (unsigned __int128)((1ull << l) - d);
  f.mul = (uint32_t)(num / d + 1);
  f.shift = l;
  return f;
}

// Where a signalled copy counts its finished workgroups and reports to the
// host (kernel arguments: read with the copy's own, not through a pointer
// after it).
struct SignalSlots {
  uint32_t *counter; // finished workgroups of the running launch
  uint32_t *flag;    // number of the last completed signal, in pinned host memory
};

// The end of a launch with p.signal set, run by every thread of the
// workgroup: the workgroup's stores are released at system scope (the
// barrier's workgroup-scope fences order the other waves' stores before
// thread 0's release, scopes composing), then counted.  The launch's last
// workgroup resets the counter for the next signalled launch -- launches on
// the library stream never overlap -- and stores the launch's number to the
// host's flag; a workgroup on its own has nothing to count.  The count itself
// is relaxed: the fences before and after it order it, and an ordered one
// would write the L2 back a second time per workgroup (128 workgroups of
// 16 KiB, launch to flag: 11.5 -> 10.7 us).
__device__ __forceinline__ void signal_done(const KParams &p,
                                            const SignalSlots &s) {
  if (!p.signal) {
    return;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (gridDim.x > 1) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
      if (__hip_atomic_fetch_add(s.counter, 1u, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT) +
              1u !=
          gridDim.x) {
        return;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");
      __hip_atomic_store(s.counter, 0u, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    }
    __hip_atomic_store(s.flag, p.signal, __ATOMIC_RELEASE,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// A signal of its own: launched after the work it reports on the same
// stream, which has finished, its stores written back, when this starts.
__global__ void k_signal(uint32_t *flag, uint32_t number) {
  __hip_atomic_store(flag, number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int P, int W, int U, bool WHOLE, int DIR, bool NTS, bool NTL>
__global__ void __launch_bounds__(kBlock)
    k_strided_copy(KParams p, SignalSlots slots) {
  constexpr uint32_t GROUPS = kBlock / P;
  constexpr uint32_t K = units_in_flight(U);
  const uint32_t lane = threadIdx.x % P;
  const uint32_t step = gridDim.x * GROUPS;
  for (uint32_t u = blockIdx.x * GROUPS + threadIdx.x / P; u < p.units;
       u += step * K) {
    copy_units<P, W, U, WHOLE, DIR, NTS, NTL>(p, u, step, p.units, lane);
  }
  signal_done(p, slots);
}

// ---------------------------------------------------------------------------
// variant table
// ---------------------------------------------------------------------------

#define TEMPI_VDESC(I, P, W, U, NT) {P, W, U, nt_stores(NT, 1), nt_loads(NT, 0)},
const VariantDesc kVariants[] = {TEMPI_VARIANTS(TEMPI_VDESC)};
#undef TEMPI_VDESC
const int kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);

typedef void (*KernelFn)(KParams, SignalSlots);

#define TEMPI_KFN(P, W, U, WHOLE, DIR, NT)                                     \
  k_strided_copy<P, W, U, WHOLE, DIR, nt_stores(NT, DIR), nt_loads(NT, DIR)>
#define TEMPI_KROW(I, P, W, U, NT)                                             \
  {{TEMPI_KFN(P, W, U, false, 0, NT), TEMPI_KFN(P, W, U, false, 1, NT)},       \
   {TEMPI_KFN(P, W, U, true, 0, NT), TEMPI_KFN(P, W, U, true, 1, NT)}},

// [variant][whole rows][dir]
static const KernelFn kKernels[][2][2] = {TEMPI_VARIANTS(TEMPI_KROW)};
#undef TEMPI_KROW
#undef TEMPI_KFN
static_assert(sizeof(kKernels) / sizeof(kKernels[0]) ==
                  sizeof(kVariants) / sizeof(kVariants[0]),
              "kernel and variant tables differ");

// ---------------------------------------------------------------------------
// geometry
// ---------------------------------------------------------------------------

int make_geom(const tempi_strided_block &sb, int64_t count, Geom *g) {
  *g = Geom();
  if (sb.ndims < 1 || sb.ndims > TEMPI_MAX_DIMS) {
    return set_error(TEMPI_ERR_ARG, "strided block with %d dimensions",
                     sb.ndims);
  }
  if (count < 0) {
    return set_error(TEMPI_ERR_ARG, "negative count");
  }
  if (sb.strides[0] != 1 && sb.counts[0] > 1) {
    return set_error(TEMPI_ERR_ARG, "strides[0] must be 1");
  }
  std::vector<Dim> dims;
  dims.push_back(Dim{sb.counts[0], 1});
  for (int d = 1; d < sb.ndims; ++d) {
    dims.push_back(Dim{sb.counts[d], sb.strides[d]});
  }
  dims.push_back(Dim{count, sb.extent});
  for (const Dim &x : dims) {
    if (x.count < 0) {
      return set_error(TEMPI_ERR_ARG, "negative dimension count");
    }
    if (x.count == 0) {
      g->start = sb.start;
      return TEMPI_SUCCESS; // nothing to move
    }
  }
  // the packed size bounds every product of counts formed below
  int64_t packed = 1;
  for (const Dim &x : dims) {
    if (__builtin_mul_overflow(packed, x.count, &packed)) {
      return set_error(TEMPI_ERR_ARG, "packed size overflows 64 bits");
    }
  }
  normalize_dims(dims);
  if ((int)dims.size() - 1 > kMaxRowDims) {
    return set_error(TEMPI_ERR_UNSUPPORTED, "%d row dimensions",
                     (int)dims.size() - 1);
  }
  g->start = sb.start;
  g->L = dims[0].count;
  g->nrd = (int)dims.size() - 1;
  g->rows = 1;
  for (int k = 0; k < g->nrd; ++k) {
    g->cnt[k] = dims[k + 1].count;
    g->str[k] = dims[k + 1].stride;
    g->rows *= g->cnt[k];
  }
  return TEMPI_SUCCESS;
}

bool geom_aligned(const Geom &g, const char *strided, const char *packed,
                  int A) {
  if (g.L % A) {
    return false;
  }
  if ((uintptr_t)packed % A || (uintptr_t)(strided + g.start) % A) {
    return false;
  }
  for (int k = 0; k < g.nrd; ++k) {
    if (g.str[k] % A) {
      return false;
    }
  }
  return true;
}

static int max_aligned_word(const Geom &g, const char *strided,
                            const char *packed) {
  for (int W = 16; W > 1; W /= 2) {
    if (geom_aligned(g, strided, packed, W)) {
      return W;
    }
  }
  return 1;
}

// Bytes of the strided side's 128-B lines: a row moves the lines it touches,
// about L + 127 bytes, unless its neighbours share them.
int64_t touched_bytes(const Geom &g) {
  if (g.nrd == 0) {
    return g.L;
  }
  const double L = (double)g.L, apart = std::abs((double)g.str[0]);
  const double bytes =
      (double)g.rows * std::min(L + 127, std::max(L, apart));
  return bytes < 1e18 ? (int64_t)bytes : (int64_t)1e18;
}

// Copies whose strided side touches this much are streamed (below).
constexpr int64_t kStreamBytes = 64ll << 20;
constexpr int64_t kInfinityCache = 256ll << 20;

// the variant nearest to a nontemporal one whose accesses are all cached
static int plain_variant(int v) {
  switch (v) {
  case 0:
  case 13:
    return 5;
  case 2:
  case 3:
    return 4;
  case 14:
  case 15:
    return 6;
  case 16:
    return 12;
  case 17:
  case 18:
    return 8;
  default:
    return v;
  }
}

// The variant for a copy whose strided side touches `touched` bytes, where
// `variant` was picked among the cached ones: itself while that is small
// against the Infinity Cache (256 MiB), else the nontemporal one for the row
// length.  A program touches the strided side once per pass -- a pack's
// source and an unpack's destination are a grid it goes on to compute on --
// while the packed bytes go to the next kernel or to the network, so the
// strided side is kept out of the caches and the packed stores stay in them.
// Pack then unpack of the same bytes, three buffer sets in turn (MI355X, us
// per pass):
//   4 Mi rows of 64 B at 192 B         cached 307, loads + strided stores 231
//   256 Ki rows of 1 KiB at 1072 B     cached 231, loads + strided stores 176
//   512 Ki rows of 64 B at 1777 B      cached 80, loads + strided stores 64,
//                                      loads on both sides 45
//   640 Ki rows of 12 B at 1001 B      cached 61, loads + strided stores 88,
//                                      loads on both sides 38
// Below 64 MiB of lines cached accesses are as fast or up to 10 % faster.
//
// A nontemporal store that covers part of a 64-B sector goes to memory by
// itself, where a cached one waits in the Infinity Cache for its neighbours:
// rows under 16 B never take them, rows that cut sectors only when their lines
// could not stay cached anyway.  Pack then unpack, three buffer sets in turn,
// by the lines of the strided side, cached -> this rule, us:
//   lines of                     300 MiB      600 MiB
//   16-B rows 700 B apart       197 -> 170   396 -> 331
//   64-B rows 192 B apart, 4 B  237 -> 179   482 -> 367
//     past a line
//   144-B rows 200 B apart      313 -> 243   607 -> 610
//   256-B rows 700 B apart      281 -> 216   531 -> 483
//   512-B rows 1088 B apart     284 -> 188   549 -> 459
//   4-KiB rows 8256 B apart     259 -> 255   524 -> 509
// An unpack alone ends later for it, as its stores have reached memory by then,
// where cached ones leave up to 256 MiB of dirty lines to whatever runs next.
// 300 MiB of lines, one unpack after the caches were emptied / one followed by
// a kernel that reads the grid: 64 B at 192 B 37 -> 56 / 106 -> 110, 256 B cut
// 107 -> 143 / 254 -> 194, 4 KiB at 4160 B 94 -> 115 / 185 -> 175.
//
// Short rows that cut sectors below that read the packed stream nontemporal
// instead, which leaves the cache to those lines.  And a line that two
// instructions read nontemporal is fetched twice: rows must be covered by
// one access of a group, or be long.  (600 000 rows of 100 B at 1138 B, 96 B
// in 16-B words and a 4-B tail, one buffer set: cached 68 us per pass, loads
// on both sides 86; 24-B rows as three 8-B words of a lane: 93, as one word
// of three lanes: 64.)
//
// Where several short rows share a line, what counts is how many of them one
// instruction reads: the 12-B words' kernel, a row per lane and four rows in
// flight, or for 16-B rows the 8-B words' reads a line before it is evicted;
// several lanes to a row (15, 17) or one row per lane with its words in turn
// (18) read it again.  The same is seen below 64 MiB in rows under 8 B, which
// are one or two accesses there, from 4 Mi rows on (1 - 2 Mi: from 14 % ahead of
// variant 9 to 12 % behind it).  Pack then unpack, three sets in turn, us:
//   24 MiB in 2-B rows 3 B apart     variant 9 91, 11 103, 12 59
//   40 MiB in 4-B rows 8 B apart     18 88, 16 62, 9 80
//   120 MiB in 8-B rows 12 B apart   17 195, 16 147, 8 149
//   120 MiB in 16-B rows 20 B apart  15 160, 18 129, 7 123
//   24 MiB in 8-B rows 64 B apart    17 143, 18 124, 16 128
// Rows of 12 and 24 B nearly a line apart, each on a line of its own and part
// of its neighbour's, are read cached once the lines outnumber the cache
// (24 B 100 B apart, 500 MiB of lines: loads nontemporal 415, cached 385).
int streamed_variant(int variant, const Geom &g, const char *strided, int dir,
                     int64_t touched) {
  const int plain = plain_variant(variant);
  const int64_t L = g.L, apart = g.nrd ? std::abs(g.str[0]) : 0;
  // several rows to a line, over many lines
  const bool dense = g.nrd && apart < 32 && g.cnt[0] * apart >= 4096;
  const bool word = L == 1 || L == 2 || L == 4 || L == 8;
  if (touched < kStreamBytes) {
    return dense && touched && L < 8 && apart < 24 && g.rows >= 4 << 20 ? 12
                                                                        : plain;
  }
  // the packed address does not matter: the strided one stands in for it
  const bool sectors = geom_aligned(g, strided, strided + g.start, 64);
  const bool stores =
      dir == TEMPI_DIR_UNPACK && L >= 16 &&
      (touched > kInfinityCache || (sectors && touched >= kInfinityCache / 2));
  if (L > 512 || (L % 16 == 0 && L > 128)) {
    return stores ? 2 : 3;
  }
  if (dense && (word || L == 12 || (L < 8 && apart < 16))) {
    return 16;
  }
  if (dense && L == 16) {
    return 18;
  }
  if (L % 16 == 0) {
    return L > 64 ? (stores ? 0 : 13) : (stores ? 14 : 15);
  }
  if (apart >= 96 && apart < 128 && touched > kInfinityCache) {
    return plain;
  }
  return L == 12 ? 16 : L == 24 ? 17 : word ? 18 : plain;
}

int heuristic_variant(const Geom &g, const char *strided, const char *packed,
                      int dir) {
  const int64_t L = g.L;
  int v = 11;
  if (L >= 2048) {
    v = 1;
  } else if (L >= 256) {
    v = 4;
  } else if (L >= 128) {
    v = 5;
  } else if (L >= 64) {
    v = 6;
  } else {
    const int Wa = max_aligned_word(g, strided, packed);
    if (Wa >= 16) {
      v = 7;
    } else if (Wa == 8) {
      v = 8;
    } else if (Wa == 4) {
      // rows of 3 or 6 dwords move as 12-B words
      v = (L % 12 == 0) ? 12 : 9;
    } else if (L >= 16) {
      v = 7;
    }
  }
  return streamed_variant(v, g, strided, dir, touched_bytes(g));
}

// Launched back to back, all variants move a copy of up to 1 MiB at the
// launch cadence (2.2-2.6 us on MI355X), which leaves the selector nothing to
// rank; waited for, the one with the fewest workgroups and the widest words
// that cut no row is seen first.  MPI_Pack, us (workgroups):
//   1024 rows of 256 B   variant 4 10.3 (32), 10 10.3 (64), 1 10.6 (256)
//   8192 rows of 64 B    variant 6 10.6 (64), 4 11.0 (256), 9 11.0 (128)
//   1024 rows of 1 KiB   variant 4 10.6 (64), 1 10.8 (256), 7 10.9 (64)
//   4096 rows of 48 B    variant 6 10.0 (32), 7 10.1 (16), 10 10.5 (256)
//   4096 rows of 24 B    variant 8 10.1 (16), 10 10.8 (256), 4 10.9 (128)
//   300 rows of 12 B     variants 12 9.1 (1), 9 9.6 (2), 4 10.5 (10)
// Rows under 64 B beyond 128 KiB stay with the selector, which has caught up by
// 512 KiB.  Eight row lengths of 4 - 48 B, rule and selector: 128 KiB 10.6 and
// 10.8 us (packs), 11.0 and 11.2 (unpacks); 192 - 256 KiB between 0.8 better
// and 0.3 worse; 512 KiB the same for packs, 11.6 and 11.5 for unpacks (12-B
// rows 12.3 and 11.6).
int latency_variant(const Geom &g) {
  const int64_t L = g.L, bytes = g.L * g.rows;
  if (bytes > (L < 64 ? 128ll << 10 : 1ll << 20)) {
    return -1;
  }
  if (L >= 256) {
    return 4;
  }
  if (L >= 128) {
    return 5;
  }
  if (L >= 64 || L == 48) {
    return 6;
  }
  if (L % 16 == 0) {
    return 7;
  }
  if (L % 8 == 0) {
    return 8;
  }
  if (L % 12 == 0) {
    return 12;
  }
  return L % 4 == 0 || L < 16 ? 9 : 7;
}

// Copies to or from host memory are bound by the link (57 GB/s).  Stores reach
// it from any variant whose words lie together; loads do only where a
// wavefront's lanes read apart from each other -- lane per row, or 16 B per
// lane in dwords -- and not where they read one contiguous KiB, at any grid
// size.  4 MiB unpacked from mapped memory, us (floor 73.3):
//   rows of 64 B    variant 9 78, 7 78, 10 77, 6 101, 8 101
//   rows of 256 B   variant 9 78, 7 78, 4 101, 6 100, 10 103
//   rows of 4 KiB   variant 9 76, 7 77, 1 98, 4 98, 10 101
// Over 55 copies of 0.5 to 15 MiB, rows of 1 B to 4 KiB, the selector, which is
// trained on device memory, unpacked 11.9 % slower than the best variant and
// packed 1.8 %; this rule 1.3 % and 0.7 %.
int link_variant(const Geom &g, int dir) {
  if (g.L * g.rows < 512 << 10) {
    return -1;
  }
  if (dir == TEMPI_DIR_UNPACK) {
    return 9;
  }
  return g.L >= 256 ? 4 : g.L >= 128 ? 5 : g.L >= 32 ? 6 : g.L % 8 ? 9 : 8;
}

int fill_kparams(const Geom &g, const char *strided, char *packed, int dir,
                 int variant, KParams *pp, bool *whole) {
  const VariantDesc &v = kVariants[variant];
  *whole = g.L % v.W == 0;
  const int64_t words = g.L / v.W;
  const int64_t per_unit = (int64_t)v.P * v.U;
  const int64_t nseg = std::max<int64_t>(1, (words + per_unit - 1) / per_unit);
  const int64_t units = g.rows * nseg;
  if (units >= kMaxUnits || words >= (1ll << 32)) {
    return set_error(TEMPI_ERR_UNSUPPORTED,
                     "copy of %lld rows of %lld B exceeds 2^31 work units",
                     (long long)g.rows, (long long)g.L);
  }
  KParams &p = *pp;
  p = KParams{};
  const char *sbase = strided + g.start;
  if (dir == TEMPI_DIR_PACK) {
    p.src = sbase;
    p.dst = packed;
  } else {
    p.src = packed;
    p.dst = const_cast<char *>(sbase);
  }
  p.L = g.L;
  p.units = (uint32_t)units;
  p.nseg = (uint32_t)nseg;
  p.segdiv = make_fastdiv((uint32_t)nseg);
  p.words = (uint32_t)words;
  p.tail = (uint32_t)(g.L % v.W);
  p.nrd = g.nrd;
  for (int k = 0; k < g.nrd; ++k) {
    if (g.cnt[k] >= (1ll << 32)) {
      return set_error(TEMPI_ERR_UNSUPPORTED, "dimension count >= 2^32");
    }
    p.cnt[k] = (uint32_t)g.cnt[k];
    p.div[k] = make_fastdiv((uint32_t)g.cnt[k]);
    p.str[k] = g.str[k];
  }
  return TEMPI_SUCCESS;
}

// Workgroups of one launch of `units` units: one pass over the units, up to
// 256 workgroups per CU.  A grid that loops (16 per CU before) leaves each
// workgroup waiting on its own slowest lines at every turn; pack then unpack,
// three buffer sets in turn, 16 per CU -> one pass:
//   4 Mi rows of 64 B at 192 B      256 -> 232 us
//   1 Mi rows of 256 B at 700 B     289 -> 264
//   256 Ki rows of 1 KiB at 1072 B  193 -> 176
static int64_t grid_of(int variant, uint32_t units, int max_blocks,
                       int cu_count) {
  const int64_t groups = (int64_t)(kBlock / kVariants[variant].P) *
                         units_in_flight(kVariants[variant].U);
  int64_t blocks = ((int64_t)units + groups - 1) / groups;
  const int64_t cap = max_blocks > 0 ? max_blocks : (int64_t)cu_count * 256;
  blocks = std::min<int64_t>(blocks, cap);
  return std::max<int64_t>(blocks, 1);
}

// segments per row of `variant` (the unit count is rows times this)
static int64_t segments_of(const Geom &g, int variant) {
  const VariantDesc &v = kVariants[variant];
  const int64_t per_unit = (int64_t)v.P * v.U;
  return std::max<int64_t>(1, (g.L / v.W + per_unit - 1) / per_unit);
}

int64_t units_of(const Geom &g, int variant) {
  return g.rows * segments_of(g, variant);
}

// Call piece(geometry, strided, packed) for each launch of a copy: rows
// longer than 1 GiB go as 1 GiB pieces, and a copy of kMaxUnits units or
// more is cut along its outer row dimensions -- a run of whole indices of
// the outermost dimension per launch, or one launch per index when a single
// index already holds too many units.
template <class F>
static int split_units(const Geom &g, const char *strided, char *packed,
                       int64_t nseg, F &piece) {
  if (g.rows * nseg < kMaxUnits || g.nrd == 0) {
    return piece(g, strided, packed);
  }
  const int k = g.nrd - 1;
  const int64_t c = g.cnt[k];
  const int64_t inner = g.rows / c;
  Geom sub = g;
  if (inner * nseg < kMaxUnits) {
    const int64_t m = (kMaxUnits - 1) / (inner * nseg);
    for (int64_t o = 0; o < c; o += m) {
      const int64_t n = std::min(m, c - o);
      sub.cnt[k] = n;
      sub.rows = inner * n;
      sub.start = g.start + o * g.str[k];
      int err = piece(sub, strided, packed + o * inner * g.L);
      if (err) {
        return err;
      }
    }
    return TEMPI_SUCCESS;
  }
  sub.nrd = k;
  sub.rows = inner;
  for (int64_t o = 0; o < c; ++o) {
    sub.start = g.start + o * g.str[k];
    int err = split_units(sub, strided, packed + o * inner * g.L, nseg, piece);
    if (err) {
      return err;
    }
  }
  return TEMPI_SUCCESS;
}

template <class F>
static int for_each_launch(const Geom &g, const char *strided, char *packed,
                           int variant, F &&piece) {
  constexpr int64_t kPiece = 1ll << 30;
  if (g.L <= kPiece) {
    return split_units(g, strided, packed, segments_of(g, variant), piece);
  }
  Geom row = g;
  row.nrd = 0;
  row.rows = 1;
  for (int64_t r = 0; r < g.rows; ++r) {
    // strided offset of row r
    int64_t off = g.start, q = r;
    for (int k = 0; k < g.nrd; ++k) {
      off += (q % g.cnt[k]) * g.str[k];
      q /= g.cnt[k];
    }
    for (int64_t x = 0; x < g.L; x += kPiece) {
      row.L = std::min(kPiece, g.L - x);
      row.start = off + x;
      int err = piece(row, strided, packed + r * g.L + x);
      if (err) {
        return err;
      }
    }
  }
  return TEMPI_SUCCESS;
}

// One launch; `signal` > 0: it signals its completion with that number (the
// caller holds the signal's lock).
static int launch_one(const Geom &g, const char *strided, char *packed,
                      int dir, int variant, hipStream_t stream,
                      int max_blocks, uint32_t signal = 0,
                      SignalSlots slots = {}) {
  KParams p;
  bool whole = false;
  int err = fill_kparams(g, strided, packed, dir, variant, &p, &whole);
  if (err) {
    return err;
  }
  const int64_t blocks = grid_of(variant, p.units, max_blocks, device_cu_count());
  KernelFn fn = kKernels[variant][whole ? 1 : 0][dir];
  p.signal = signal;
  void *args[] = {&p, &slots};
  TEMPI_HIP_CHECK(hipLaunchKernel(reinterpret_cast<const void *>(fn),
                                  dim3((unsigned)blocks), dim3(kBlock), args,
                                  0, stream));
  if (in_trial()) {
    ++counters().trial_launches;
  } else if (dir == TEMPI_DIR_PACK) {
    ++counters().pack_kernel_launches;
  } else {
    ++counters().unpack_kernel_launches;
  }
  return TEMPI_SUCCESS;
}

namespace {
thread_local int t_trial_depth = 0;
} // namespace

TrialScope::TrialScope() { ++t_trial_depth; }
TrialScope::~TrialScope() { --t_trial_depth; }
bool in_trial() { return t_trial_depth > 0; }

int launch_copy(const Geom &g, const char *strided, char *packed, int dir,
                int variant, hipStream_t stream, int max_blocks) {
  if (g.rows == 0 || g.L == 0) {
    return TEMPI_SUCCESS;
  }
  if (variant < 0 || variant >= kNumVariants) {
    return set_error(TEMPI_ERR_ARG, "variant %d out of range", variant);
  }
  return for_each_launch(g, strided, packed, variant,
                         [&](const Geom &pg, const char *ps, char *pp) {
                           return launch_one(pg, ps, pp, dir, variant, stream,
                                             max_blocks);
                         });
}

// ---------------------------------------------------------------------------
// waiting for a synchronous copy
// ---------------------------------------------------------------------------
//
// MPI_Pack and MPI_Unpack return when their copy is done.  On MI355X an
// empty kernel's own store reaches the host 5.7 us after its launch begins,
// but hipStreamSynchronize returns after 11.1 us: the rest is the runtime's
// end-of-kernel processing.  A copy of one launch of few workgroups on the
// library stream therefore signals its own completion (KParams::signal) and
// the host spins on the flag.  In larger grids each workgroup's release writes
// its XCD's L2 back and those queue behind each other (counting in 32 leaves
// instead of one counter changes nothing), so a one-thread kernel behind the
// copy stores the flag instead: it starts after the copy's own end-of-kernel
// write-back.  Contiguous copies of 16 KiB per workgroup, launch to the host
// seeing it, us:
//   workgroups               64    128    256    512   1024   2048
//   own signal              8.9   10.7   14.3   21.9   37.2   72.1
//   signal kernel behind    9.9   10.0   10.2   10.8   11.2   17.2
//   hipStreamSynchronize   11.9   12.2   12.5   13.4   14.5   20.8
//
// How few depends on what a write-back finds.  Where the lanes of a row's
// group store next to each other, whole lines; where each lane stores a row of
// its own, lines of which the rest is still to come, and in host memory each
// of those is a write over the link by itself.  Own signal less signal kernel,
// us, median (most) over rows of 4 B - 1 KiB 100 B apart, MPI_Pack and
// MPI_Unpack:
//   workgroups                       16           32           64          128
//   packed on the device, P > 1  -0.7 (-0.4)  -0.5 (-0.2)  -0.3 (0.5)   0.9 (2.7)
//                         P = 1  -0.6 (0.1)   -0.2 (0.5)    0.5 (1.3)   2.2 (3.3)
//   packs to the host,    P > 1  -0.8 (0.4)   -0.6 (0.1)   -0.3 (0.5)   0.2 (2.6)
//                         P = 1  -0.5 (1.0)    1.0 (3.0)    4.4 (15)     15 (44)
//   unpacks from it,      P > 1  -0.4 (0.4)   -0.2 (0.9)    0.2 (1.6)   2.2 (3.2)
//                         P = 1  -0.2 (0.5)    0.2 (0.9)    1.0 (1.9)   2.9 (3.7)

namespace {

// most workgroups of a copy that signals for itself
int64_t own_signal_blocks(const Geom &g, int variant) {
  return kVariants[variant].P > 1 ? 64 : g.host ? 16 : 48;
}

struct SignalState {
  std::mutex mu; // held from a signal's number to its launch
  bool tried = false;
  SignalSlots slots{};       // device addresses: device memory, the flag
  uint32_t *flag = nullptr;  // pinned host memory
  unsigned long long issued = 0; // the last number given to a signal
  int64_t kernels = 0;           // signals sent by a kernel behind their work
  // set after a signalled wait fails: the counter may no longer match the
  // launches, so later copies wait on the stream
  std::atomic<bool> off{false};
};

SignalState &signal_state() {
  static SignalState s;
  return s;
}

// The next signal's number, given for good (the state's lock held).  A number
// that may have reached the device is never given again: were it, the second
// copy's wait would end on the first one's signal.  One whose launch failed is
// skipped, as waits compare with >=, and so are those whose low 32 bits, which
// the kernels store, would read as none.
unsigned long long take_number(SignalState &st) {
  do {
    ++st.issued;
  } while (!(uint32_t)st.issued);
  return st.issued;
}

bool flag_at(const SignalState &st, unsigned long long seq) {
  // fewer than 2^31 signals are ever in flight
  return (int32_t)(__atomic_load_n(st.flag, __ATOMIC_ACQUIRE) -
                   (uint32_t)seq) >= 0;
}

// Counter and flag, allocated once, on the library stream's device (the
// state's lock held); false when they cannot be.
bool signal_ready(SignalState &st) {
  if (st.tried) {
    return st.flag != nullptr && !st.off.load(std::memory_order_relaxed);
  }
  st.tried = true;
  if (env().no_signal) {
    return false;
  }
  // the counter is zeroed on the library stream (which does not wait for the
  // null stream) before the first signalled launch
  hipStream_t s = library_stream();
  void *c = nullptr, *f = nullptr, *fd = nullptr;
  bool ok = hipSuccess == hipMalloc(&c, 256) &&
            hipSuccess == hipMemsetAsync(c, 0, 256, s) &&
            hipSuccess == hipHostMalloc(&f, 256, hipHostMallocMapped |
                                                     hipHostMallocPortable) &&
            hipSuccess == hipHostGetDevicePointer(&fd, f, 0);
  if (ok) {
    __atomic_store_n(static_cast<uint32_t *>(f), 0u, __ATOMIC_RELEASE);
    ok = hipSuccess == hipStreamSynchronize(s);
  }
  if (!ok) {
    (void)hipGetLastError();
    if (c) {
      (void)hipFree(c);
    }
    if (f) {
      (void)hipHostFree(f);
    }
    TEMPI_LOG(LOG_WARN, "no completion signal: synchronous copies wait on the stream");
    return false;
  }
  st.slots = SignalSlots{static_cast<uint32_t *>(c), static_cast<uint32_t *>(fd)};
  st.flag = static_cast<uint32_t *>(f);
  return true;
}

// Spin until signal `seq` arrived.  A launch that never runs to its end
// leaves the flag short, so after 0.2 ms the stream is checked every 0.1 ms:
// finished without the flag is an error, and so is a failed stream.  An
// error switches the signal off.
int wait_signal(SignalState &st, unsigned long long seq) {
  const auto t0 = std::chrono::steady_clock::now();
  double check_at = 2e-4;
  int err = TEMPI_SUCCESS;
  for (;;) {
    if (flag_at(st, seq)) {
      return TEMPI_SUCCESS;
    }
    __builtin_ia32_pause();
    const double el = std::chrono::duration<double>(
                          std::chrono::steady_clock::now() - t0)
                          .count();
    if (el < check_at) {
      continue;
    }
    const hipError_t e = hipStreamQuery(library_stream());
    if (e == hipSuccess) {
      if (flag_at(st, seq)) {
        return TEMPI_SUCCESS;
      }
      err = set_error(TEMPI_ERR_HIP, "a copy ended without its signal");
      break;
    }
    if (e != hipErrorNotReady) {
      (void)hipGetLastError();
      err = set_error(TEMPI_ERR_HIP, "copy failed: %s", hipGetErrorString(e));
      break;
    }
    check_at = el + 1e-4;
  }
  st.off.store(true);
  TEMPI_LOG(LOG_WARN, "completion signal switched off: %s", tempi_last_error());
  (void)hipStreamSynchronize(library_stream());
  return err;
}

bool on_library_device() {
  int dev = -1;
  return hipSuccess == hipGetDevice(&dev) && dev == library_device();
}

// one launch of few enough workgroups, on the library stream's device
bool signal_fits(const Geom &g, int variant, int max_blocks) {
  const int64_t units = units_of(g, variant);
  return g.L <= (1ll << 30) && units < kMaxUnits &&
         grid_of(variant, (uint32_t)units, max_blocks, device_cu_count()) <=
             own_signal_blocks(g, variant) &&
         on_library_device();
}

} // namespace

unsigned long long signal_stream() {
  if (!on_library_device()) {
    return 0;
  }
  SignalState &st = signal_state();
  std::lock_guard<std::mutex> lk(st.mu);
  if (!signal_ready(st)) {
    return 0;
  }
  const unsigned long long n = take_number(st);
  // judged by the launch's own result: hipGetLastError reports, and clears,
  // whatever earlier error of this thread the application has not read yet
  uint32_t number = (uint32_t)n;
  void *args[] = {&st.slots.flag, &number};
  const hipError_t e =
      hipLaunchKernel(reinterpret_cast<const void *>(k_signal), dim3(1),
                      dim3(1), args, 0, library_stream());
  if (e != hipSuccess) {
    (void)hipGetLastError(); // this launch's own
    TEMPI_LOG(LOG_WARN, "signal kernel: %s", hipGetErrorString(e));
    return 0;
  }
  ++st.kernels;
  return n;
}

int launch_copy_signalled(const Geom &g, const char *strided, char *packed,
                          int dir, int variant, int max_blocks,
                          unsigned long long *seq, bool *own) {
  *seq = 0;
  *own = false;
  if (g.rows == 0 || g.L == 0) {
    return TEMPI_SUCCESS;
  }
  if (variant < 0 || variant >= kNumVariants) {
    return set_error(TEMPI_ERR_ARG, "variant %d out of range", variant);
  }
  hipStream_t s = library_stream();
  if (signal_fits(g, variant, max_blocks)) {
    SignalState &st = signal_state();
    std::lock_guard<std::mutex> lk(st.mu);
    if (signal_ready(st)) {
      const unsigned long long n = take_number(st);
      const int err = launch_one(g, strided, packed, dir, variant, s,
                                 max_blocks, (uint32_t)n, st.slots);
      if (!err) {
        *seq = n;
        *own = true;
      }
      return err;
    }
  }
  const int err = launch_copy(g, strided, packed, dir, variant, s, max_blocks);
  if (!err) {
    *seq = signal_stream();
  }
  return err;
}

bool signal_reached(unsigned long long seq) {
  const SignalState &st = signal_state();
  return seq && st.flag && flag_at(st, seq);
}

hipEvent_t mark_library_stream() {
  hipEvent_t ev = nullptr;
  if (hipSuccess == hipEventCreateWithFlags(&ev, hipEventDisableTiming) &&
      hipSuccess == hipEventRecord(ev, library_stream())) {
    return ev;
  }
  (void)hipGetLastError(); // one of these two calls'
  if (ev) {
    (void)hipEventDestroy(ev);
  }
  return nullptr;
}

int poll_signal_or_stream(unsigned long long seq, hipEvent_t ev,
                          uint32_t *polls, bool *done) {
  *done = signal_reached(seq);
  // a signal that does not come is looked after in the stream's own state,
  // every so many polls: the query costs as much as hundreds of them
  if (*done || (seq && ++*polls % 1024)) {
    return TEMPI_SUCCESS;
  }
  const hipError_t q =
      !seq && ev ? hipEventQuery(ev) : hipStreamQuery(library_stream());
  if (q == hipErrorNotReady) {
    return TEMPI_SUCCESS;
  }
  if (q != hipSuccess) {
    (void)hipGetLastError();
    return set_error(TEMPI_ERR_HIP, "copy failed: %s", hipGetErrorString(q));
  }
  *done = !seq || signal_reached(seq);
  return *done ? TEMPI_SUCCESS
               : set_error(TEMPI_ERR_HIP, "a copy ended without its signal");
}

int wait_signal_or_stream(unsigned long long seq, hipEvent_t ev) {
  if (seq) {
    return wait_signal(signal_state(), seq);
  }
  TEMPI_HIP_CHECK(ev ? hipEventSynchronize(ev)
                     : hipStreamSynchronize(library_stream()));
  return TEMPI_SUCCESS;
}

int wait_library_stream() { return wait_signal_or_stream(signal_stream()); }

int launch_copy_wait(const Geom &g, const char *strided, char *packed,
                     int dir, int variant, int max_blocks) {
  unsigned long long seq = 0;
  bool own = false;
  int err = launch_copy_signalled(g, strided, packed, dir, variant, max_blocks,
                                  &seq, &own);
  if (err) {
    // part of the copy may be running
    (void)hipStreamSynchronize(library_stream());
    return err;
  }
  if (g.rows == 0 || g.L == 0) {
    return TEMPI_SUCCESS;
  }
  if ((err = wait_signal_or_stream(seq))) {
    return err;
  }
  if (own) {
    ++counters().signalled_waits;
  }
  return TEMPI_SUCCESS;
}

// ---------------------------------------------------------------------------
// host-side emulation of a copy's memory accesses
// ---------------------------------------------------------------------------
//
// Runs the launches, grid, grid-stride index sequence and unit addresses
// that launch_copy and the kernels would, with the same code for the
// address arithmetic (unit_addr), and records every byte range loaded and
// stored instead of touching memory.  The buffer addresses are numbers
// only; nothing is dereferenced.  It shows on the CPU which bytes a launch
// reads and writes for any variant, alignment and shape.

namespace {

struct Recorder {
  uintptr_t rbase = 0, wbase = 0; // origins of the read and written sides
  int64_t rlo = INT64_MAX, rhi = INT64_MIN, wlo = INT64_MAX, whi = INT64_MIN;
  int64_t nread = 0, nwritten = 0;
  // per-byte store counts over written-side offsets [map_lo, map_lo + size)
  std::vector<uint8_t> map;
  int64_t map_lo = 0;
  bool outside_map = false;
  void read(const char *p, int64_t n) {
    const int64_t o = (int64_t)((uintptr_t)p - rbase);
    rlo = std::min(rlo, o);
    rhi = std::max(rhi, o + n);
    nread += n;
  }
  void write(const char *p, int64_t n) {
    const int64_t o = (int64_t)((uintptr_t)p - wbase);
    wlo = std::min(wlo, o);
    whi = std::max(whi, o + n);
    nwritten += n;
    if (!map.empty()) {
      for (int64_t i = o; i < o + n; ++i) {
        const int64_t j = i - map_lo;
        if (j < 0 || j >= (int64_t)map.size()) {
          outside_map = true;
        } else if (map[(size_t)j] < 255) {
          ++map[(size_t)j];
        }
      }
    }
  }
};

thread_local Recorder *t_rec = nullptr;

// one work unit of one group, all P lanes: the kernels' address phase, then
// the words and tail pieces of the load and store phases
template <int P, int W, int U, bool WHOLE, int DIR>
void emulate_unit(const KParams &p, uint32_t u) {
  for (uint32_t lane = 0; lane < (uint32_t)P; ++lane) {
    const UnitAddr a = unit_addr<P, W, U, WHOLE, DIR>(p, u, lane);
    for (int j = 0; j < U; ++j) {
      const uint32_t w = a.w + (uint32_t)(j * P);
      if (w < a.n) {
        t_rec->read(a.s + (size_t)w * W, W);
        t_rec->write(a.d + (size_t)w * W, W);
      }
    }
    if (!WHOLE && a.tail) {
      const int64_t off = (int64_t)p.words * W;
      const auto piece = [&](uint32_t n, uint32_t at) {
        if (p.tail & n) {
          t_rec->read(a.s + off + at, n);
          t_rec->write(a.d + off + at, n);
        }
      };
      piece(8, 0);
      piece(4, tail_at<4>(p.tail));
      piece(2, tail_at<2>(p.tail));
      piece(1, tail_at<1>(p.tail));
    }
  }
}

typedef void (*EmulateFn)(const KParams &, uint32_t);
#define TEMPI_EROW(I, P, W, U, NT)                                             \
  {{emulate_unit<P, W, U, false, 0>, emulate_unit<P, W, U, false, 1>},          \
   {emulate_unit<P, W, U, true, 0>, emulate_unit<P, W, U, true, 1>}},
const EmulateFn kEmulate[][2][2] = {TEMPI_VARIANTS(TEMPI_EROW)};
#undef TEMPI_EROW

} // namespace

} // namespace tempi

using namespace tempi;

TEMPI_EXPORT int tempi_signals_get(int64_t *numbers, int64_t *kernels) {
  SignalState &st = signal_state();
  std::lock_guard<std::mutex> lk(st.mu);
  if (numbers) {
    *numbers = (int64_t)st.issued;
  }
  if (kernels) {
    *kernels = st.kernels;
  }
  return TEMPI_SUCCESS;
}

// Emulates launch_copy of the copy on the host (see above); `unit_limit`
// bounds the work units emulated in full (beyond it only the launch plan is
// reported).
TEMPI_EXPORT int tempi_copy_emulate(const tempi_strided_block *sb,
                                    int64_t incount, uint64_t strided_addr,
                                    uint64_t packed_addr, int direction,
                                    int variant, int max_blocks, int cu_count,
                                    int64_t unit_limit,
                                    tempi_copy_emulation *out) {
  if (!sb || !out || cu_count <= 0 || max_blocks < 0) {
    return set_error(TEMPI_ERR_ARG, "bad argument");
  }
  int err = check_direction(direction);
  if (err) {
    return err;
  }
  if (variant < 0 || variant >= kNumVariants) {
    return set_error(TEMPI_ERR_ARG, "variant %d out of range", variant);
  }
  Geom g;
  if ((err = make_geom(*sb, incount, &g))) {
    return err;
  }
  *out = tempi_copy_emulation{};
  const char *strided = reinterpret_cast<const char *>((uintptr_t)strided_addr);
  char *packed = reinterpret_cast<char *>((uintptr_t)packed_addr);
  if (g.rows == 0 || g.L == 0) {
    out->exact = 1;
    return TEMPI_SUCCESS;
  }
  // plan: launches and units
  int64_t units_total = 0;
  err = for_each_launch(g, strided, packed, variant,
                        [&](const Geom &pg, const char *, char *) {
                          const int64_t u = pg.rows * segments_of(pg, variant);
                          ++out->launches;
                          out->max_units = std::max(out->max_units, u);
                          units_total += u;
                          return TEMPI_SUCCESS;
                        });
  if (err) {
    return err;
  }
  if (units_total > unit_limit) {
    out->emulated = 0;
    return TEMPI_SUCCESS;
  }
  Recorder rec;
  const bool pack = direction == TEMPI_DIR_PACK;
  rec.rbase = pack ? (uintptr_t)strided : (uintptr_t)packed;
  rec.wbase = pack ? (uintptr_t)packed : (uintptr_t)strided;
  // the bytes the copy must write, each once: the packed stream, or the
  // strided rows (a map of the written side, up to 256 MiB)
  int64_t lo = 0, hi = g.L;
  for (int k = 0; k < g.nrd; ++k) {
    const int64_t reach = (g.cnt[k] - 1) * g.str[k];
    (reach < 0 ? lo : hi) += reach;
  }
  const int64_t map_lo = pack ? 0 : g.start + lo;
  const int64_t map_len = pack ? g.rows * g.L : hi - lo;
  std::vector<uint8_t> want;
  if (map_len <= (256ll << 20)) {
    rec.map.assign((size_t)map_len, 0);
    rec.map_lo = map_lo;
    want.assign((size_t)map_len, 0);
    for (int64_t r = 0; r < g.rows; ++r) {
      int64_t off = pack ? r * g.L : g.start, q = r;
      for (int k = 0; !pack && k < g.nrd; ++k) {
        off += (q % g.cnt[k]) * g.str[k];
        q /= g.cnt[k];
      }
      for (int64_t x = 0; x < g.L; ++x) {
        uint8_t &c = want[(size_t)(off + x - map_lo)];
        c = (uint8_t)std::min(255, c + 1);
      }
    }
  }
  t_rec = &rec;
  err = for_each_launch(
      g, strided, packed, variant,
      [&](const Geom &pg, const char *ps, char *pp) -> int {
        KParams p;
        bool whole = false;
        int e = fill_kparams(pg, ps, pp, direction, variant, &p, &whole);
        if (e) {
          return e;
        }
        const VariantDesc &v = kVariants[variant];
        const EmulateFn fn = kEmulate[variant][whole ? 1 : 0][direction];
        const uint32_t GROUPS = (uint32_t)(kBlock / v.P);
        const uint32_t K = (uint32_t)units_in_flight(v.U);
        const uint32_t blocks =
            (uint32_t)grid_of(variant, p.units, max_blocks, cu_count);
        const uint32_t step = blocks * GROUPS;
        // the kernels' index sequence, in their 32-bit arithmetic
        for (uint32_t b = 0; b < blocks; ++b) {
          for (uint32_t grp = 0; grp < GROUPS; ++grp) {
            for (uint32_t u = b * GROUPS + grp; u < p.units;) {
              for (uint32_t k = 0; k < K; ++k) {
                const uint32_t uu = u + k * step;
                if ((uint64_t)u + (uint64_t)k * step != (uint64_t)uu) {
                  out->wrapped = 1;
                } else if (uu < p.units) {
                  fn(p, uu);
                }
              }
              const uint64_t next = (uint64_t)u + (uint64_t)step * K;
              if (next >= (1ull << 32)) {
                out->wrapped = 1;
                break;
              }
              u = (uint32_t)next;
            }
          }
        }
        return TEMPI_SUCCESS;
      });
  t_rec = nullptr;
  if (err) {
    return err;
  }
  out->emulated = 1;
  out->read_lo = rec.nread ? rec.rlo : 0;
  out->read_hi = rec.nread ? rec.rhi : 0;
  out->write_lo = rec.nwritten ? rec.wlo : 0;
  out->write_hi = rec.nwritten ? rec.whi : 0;
  out->bytes_read = rec.nread;
  out->bytes_written = rec.nwritten;
  out->exact = rec.map.empty() ? -1 : (!rec.outside_map && rec.map == want);
  return TEMPI_SUCCESS;
}

namespace tempi {

// exported for the host-side unit test of the divisor arithmetic
extern "C" __attribute__((visibility("default"))) uint32_t
tempi_fastdiv_check(uint32_t n, uint32_t d) {
  return make_fastdiv(d).div(n);
}

} // namespace tempi
