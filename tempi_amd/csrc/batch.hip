// batch.hip -- many strided copies in one kernel launch.
//
// The reference launches one kernel per MPI_Pack and synchronizes
// (src/internal/packer_2d.cu:101-108).  A batch instead resolves every
// request once, on the host, into the same per-copy parameters the single
// kernels take, uploads them as a device-resident table, and splits each
// request into tiles of one workgroup pass (256 threads, four loads in
// flight per lane: 16 KiB for 16-byte words).  One workgroup takes each tile,
// in address order, each XCD a consecutive range of it (order_tiles); the
// tile's request comes from a tile-to-request table, and a switch runs that
// request's kernel variant.  Heterogeneous shapes -- 12-B halo rows next to
// 2-KiB face rows -- share one launch.
//
// A first version handed tiles out with one atomic counter; every tile then
// paid for a device-scope atomic serialized with all the others (about 30 ns
// each on MI355X), which dominated small and large batches alike.  The
// static assignment has no shared state, so launches need no reset and
// replay from a captured hipGraph unchanged.  Requests inside a batch must
// not write bytes another request reads or writes.
#include "copy_core.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <memory>
#include <new>
#include <vector>

namespace tempi {

namespace {

struct BatchItem {
  int32_t kind;            // 4 * variant + 2 * whole rows + direction + kFour
  uint32_t units_per_tile; // units of one block-pass: groups per block * K
  uint32_t ntiles;         // tiles of this request
  uint32_t pad;
  KParams p;               // after the kind: both in the item's first lines
};

constexpr uint32_t kXcds = 8;

// Lane-per-row variants of one-word units keep four units of a lane in flight
// (kFour) or two.  Among tiles of other requests, in address order, two are
// enough, and four fetch lines before those of their neighbours are done with:
// 254 unpacks of 4-B rows 4 - 516 B apart took 799 us with two, 1 013 us with
// four, 238 of 8-B rows 421 and 509 us.  A batch of few requests has the device
// to itself, and its unpacks take four: the three faces of a 512^3 float grid,
// unpack alone, 8.3 us with two, 7.7 with four (of a 448^3 grid the same).  Its
// packs, whose loads of a line each then queue behind each other, take two
// (8.8 us; 9.4 with four), and so do requests of less than 3/4 of a tile per
// CU, for twice the workgroups (pack + unpack, 320^3, 100 tiles of four: 11.1
// us; 11.6 with four).
__host__ __device__ constexpr bool two_or_four(int P, int U) {
  return P == 1 && units_in_flight(U) > 2;
}

// added to the kind of a request whose lanes take four units instead of two:
// past the other kinds (equal cases would not compile)
constexpr int kFour = 128;

// One block-pass: tile `l` of a request split into `nt` tiles moves K blocks
// of GROUPS units.  RUN: the K * GROUPS units from l * K * GROUPS on, so that
// tiles in address order walk the memory in address order.  Else the blocks
// are nt * GROUPS units apart -- units l*GROUPS + g + k*nt*GROUPS, every unit
// of the request exactly once over the nt tiles: spreading a lane's K units
// across the request measured about 0.2 us faster per launch on MI355X for
// 12-B rows 2 KiB apart (262 144 rows), the same as the single-copy kernels'
// grid-stride order.
template <int P, int W, int U, bool WHOLE, int DIR, bool NTS, bool NTL,
          bool RUN, bool FOUR>
__device__ __forceinline__ void copy_tile(const KParams &p, uint32_t l,
                                          uint32_t nt) {
  constexpr uint32_t GROUPS = kBlock / P;
  constexpr uint32_t K =
      two_or_four(P, U) && !FOUR ? 2 : units_in_flight(U);
  if constexpr (two_or_four(P, U) || !FOUR) {
    copy_units<P, W, U, WHOLE, DIR, NTS, NTL, K>(
        p, l * (RUN ? K * GROUPS : GROUPS) + threadIdx.x / P,
        RUN ? GROUPS : nt * GROUPS, p.units, threadIdx.x % P);
  }
}

template <bool RUN>
__device__ __forceinline__ void run_tile(int kind, const KParams &p,
                                         uint32_t l, uint32_t nt) {
  switch (kind) {
#define TEMPI_BTILE(K, P, W, U, WHOLE, DIR, NT, FOUR)                          \
  case K:                                                                      \
    copy_tile<P, W, U, WHOLE, DIR, nt_stores(NT, DIR), nt_loads(NT, DIR), RUN, \
              FOUR>(p, l, nt);                                                 \
    break;
#define TEMPI_BKINDS(K, P, W, U, NT, FOUR)                                     \
  TEMPI_BTILE(K + 0, P, W, U, false, 0, NT, FOUR)                              \
  TEMPI_BTILE(K + 1, P, W, U, false, 1, NT, FOUR)                              \
  TEMPI_BTILE(K + 2, P, W, U, true, 0, NT, FOUR)                               \
  TEMPI_BTILE(K + 3, P, W, U, true, 1, NT, FOUR)
#define TEMPI_BCASE(I, P, W, U, NT)                                            \
  TEMPI_BKINDS(4 * I, P, W, U, NT, false)                                      \
  TEMPI_BKINDS(4 * I + kFour, P, W, U, NT, true)
    TEMPI_VARIANTS(TEMPI_BCASE)
#undef TEMPI_BCASE
#undef TEMPI_BKINDS
#undef TEMPI_BTILE
  default:
    break;
  }
}

// One tile: the request it belongs to and its index within the request.
struct Tile {
  uint32_t item;
  uint32_t tile;
};

// Workgroups are dispatched round-robin over the XCDs (workgroup b runs on
// XCD b % 8).  The host orders the tile table so that XCD x owns the
// contiguous range [xcd_begin[x], xcd_begin[x+1]) of the tiles in address
// order, an eighth of the traffic: neighbouring tiles, whose rows share lines,
// run at about the same time in one XCD's L2.  The assignment is static: no
// atomics, no state carried between launches.  A grid over its limit loops.
__global__ void __launch_bounds__(kBlock)
    __attribute__((amdgpu_waves_per_eu(5)))
    k_batch(const BatchItem *__restrict__ items,
            const Tile *__restrict__ tiles,
            const uint32_t *__restrict__ xcd_begin, uint32_t ntiles,
            int xcd_split) {
  uint32_t t, end, step;
  if (xcd_split) {
    const uint32_t xcd = blockIdx.x % kXcds;
    step = gridDim.x / kXcds;
    t = xcd_begin[xcd] + blockIdx.x / kXcds;
    end = xcd_begin[xcd + 1];
  } else {
    step = gridDim.x;
    t = blockIdx.x;
    end = ntiles;
  }
  for (; t < end; t += step) {
    // uniform addresses: the tile and its request's parameters are read
    // with scalar loads in place (a private copy of the parameter struct
    // would live in scratch memory)
    const Tile tl = tiles[t];
    const uint32_t r = __builtin_amdgcn_readfirstlane(tl.item);
    const uint32_t l = __builtin_amdgcn_readfirstlane(tl.tile);
    const BatchItem &it = items[r];
    run_tile<true>(it.kind, it.p, l, it.ntiles);
  }
}

// Batches of at most kSmallItems requests pass their tile index in the
// kernel arguments.  k_batch's workgroups wait on three dependent loads
// before their first data load (XCD range, tile record, request parameters);
// here the tile follows from the workgroup index by arithmetic on the
// argument block, leaving one dependent load (the request's parameters).
// The parameters stay in device memory: a back-to-back launch with 2 KiB of
// kernel arguments costs about 0.5 us more than one with a few hundred bytes
// on MI355X, more than the loads it would save.
//
// Padded tile numbering: request r owns tiles [base[r], base[r+1]), a range
// that starts at a multiple of 8 and has 8 * share[r] entries.  Tile T runs
// on XCD T % 8 (the grid is a multiple of 8, so T % 8 == blockIdx.x % 8 on
// every pass), and XCD x takes the request's tiles
// [x * share[r], (x + 1) * share[r]): each XCD gets a contiguous eighth of
// every request.  Padding entries past the request's last tile do nothing.
constexpr int kSmallItems = 8;

struct SmallIndex {
  uint32_t n;                     // requests
  uint32_t end;                   // padded tiles of the whole batch
  uint32_t base[kSmallItems];     // first padded tile of each request
  uint32_t share[kSmallItems];    // tiles of each request per XCD
  uint32_t ntiles[kSmallItems];   // tiles of each request
};

// The index is read through the kernel-argument segment pointer (it is the
// first argument, at offset 0) into registers, every entry unconditionally
// and before the loop: the entries past the last request hold `end`, so no
// test of the request count is needed, and the loads issue together.  (With
// the count tested per entry, or with entries read at a run-time index, the
// compiler chained one scalar load and wait per request in front of the
// first data load, or copied the parameter to scratch memory.)
__global__ void __launch_bounds__(kBlock)
    __attribute__((amdgpu_waves_per_eu(5)))
    k_batch_small(const SmallIndex arg, const BatchItem *__restrict__ items) {
  (void)arg;
  const SmallIndex *ix =
      (const SmallIndex *)__builtin_amdgcn_kernarg_segment_ptr();
  const uint32_t end = ix->end;
  uint32_t base[kSmallItems], share[kSmallItems], ntiles[kSmallItems];
#pragma unroll
  for (int i = 0; i < kSmallItems; ++i) {
    base[i] = ix->base[i];
    share[i] = ix->share[i];
    ntiles[i] = ix->ntiles[i];
  }
  for (uint32_t t = blockIdx.x; t < end; t += gridDim.x) {
    // request r: the last whose range starts at or before t
    uint32_t r = 0, b = base[0], sh = share[0], nt = ntiles[0];
#pragma unroll
    for (int i = 1; i < kSmallItems; ++i) {
      const bool in = t >= base[i];
      r = in ? (uint32_t)i : r;
      b = in ? base[i] : b;
      sh = in ? share[i] : sh;
      nt = in ? ntiles[i] : nt;
    }
    const uint32_t q = t - b;
    const uint32_t l = (q % kXcds) * sh + q / kXcds;
    if (l < nt) {
      const BatchItem &it = items[r];
      run_tile<false>(it.kind, it.p, l, nt);
    }
  }
}

} // namespace

} // namespace tempi

using namespace tempi;

namespace tempi {
namespace {

// What one launch of a batch needs: the grid, the kernel, and where its
// tables sit in device memory.
struct BatchLaunch {
  int grid = 0;
  uint32_t ntiles = 0;
  int xcd_split = 0;
  bool small = false; // k_batch_small with `ix`
  SmallIndex ix{};
  const BatchItem *items = nullptr;
  const Tile *tiles = nullptr;        // tile records, grouped by XCD
  const uint32_t *xcd_begin = nullptr; // first tile of each XCD (kXcds + 1)
};

uint32_t units_per_tile(const VariantDesc &v, bool four) {
  return (uint32_t)(kBlock / v.P) *
         (!four && two_or_four(v.P, v.U) ? 2 : units_in_flight(v.U));
}

void launch_kernel(const BatchLaunch &l, hipStream_t s) {
  if (l.small) {
    hipLaunchKernelGGL(k_batch_small, dim3(l.grid), dim3(kBlock), 0, s, l.ix,
                       l.items);
  } else {
    hipLaunchKernelGGL(k_batch, dim3(l.grid), dim3(kBlock), 0, s, l.items,
                       l.tiles, l.xcd_begin, l.ntiles, l.xcd_split);
  }
}

// One request as the batch resolves it.
struct Req {
  Geom g;
  const char *ds = nullptr; // strided buffer origin (device address)
  char *dp = nullptr;       // first packed byte (device address)
  int dir = 0;
  int variant = 0;
  bool wide = false; // four units per lane where two would be taken
};

// The host image of a batch's device tables (request parameters, tile
// records, XCD range bounds; each section 256-B aligned) and its launch
// shape, with the table pointers left as offsets into the image.
struct BatchPlan {
  std::vector<char> image;
  size_t tl_off = 0, xb_off = 0;
  BatchLaunch launch;
  int n = 0;
};

// The tile records of a batch in the order of the strided side's addresses,
// to windows of 4 KiB, cut into `groups` consecutive ranges of about
// equal cost (begin[x] is the first tile of range x; a range may end inside
// a window).  Requests of a batch share lines -- a halo's faces, edges and
// corners, the low x face of a row and the high one of the row before -- and
// partly written lines: with every request in turn, and an eighth of each on
// every XCD, those lines were fetched by several XCDs, or again after the L2
// had dropped them; now one XCD meets them at about the same time.  MI355X,
// request order -> address order:
//   halo pack + unpack, 64 subdomains of 128^3 doubles   312 -> 276 us
//   36 subdomains of 26^3 floats, radius 1               20.9 -> 7.7 us
//   4 096 random requests from one source of 1.6 GB      5.59 -> 4.33 ms
// (the last with windows of 64 KiB 4.39, of 256 KiB 4.96 ms).
constexpr int kWindowShift = 12; // 4 KiB, wider where they would outnumber the tiles

// [first, last) of the strided addresses a request touches
void strided_range(const Req &q, uintptr_t *first, uintptr_t *last) {
  const uintptr_t a = (uintptr_t)(q.ds + q.g.start);
  *first = a;
  *last = a + (uintptr_t)q.g.L;
  for (int k = 0; k < q.g.nrd; ++k) {
    const int64_t reach = (q.g.cnt[k] - 1) * q.g.str[k];
    (reach < 0 ? *first : *last) += (uintptr_t)reach;
  }
}

// What the tile order needs of each request.  A request's tile l is taken to
// start at `at` + l * `step`: exact for rows at one stride, near enough for
// several dimensions.  Only the order depends on it.
struct Walk {
  int64_t at;   // first tile's position, 12 fraction bits
  int64_t step; // from tile to tile, 12 fraction bits
  float cost;   // tile_cost
};

// What a tile of a request takes of an XCD, in bytes of lines at about 0.67 per
// ns: its lines and packed bytes, but no less than its workgroup's own time.
// Batches of 40 requests of one row length, ns per tile of an XCD, measured
// and as bytes: packs of rows of 16 B - 4 KiB 0.96 to 1.17 of each other (100 B
// 1.33); 1-B rows 2 B apart 12.2 and 2.3 (2 KiB), 4-B rows 5 B apart 14.4 and
// 6.9.  Unpacks whose rows cut sectors take half as much again (64-B rows 65 B
// apart 38 and 25, 256 B 33 and 25), unless their packed bytes are read
// nontemporal (1 000 B 46 and 48).
float tile_cost(const Req &q, uint32_t ntiles) {
  const Geom &g = q.g;
  double bytes = ((double)touched_bytes(g) + (double)g.L * g.rows) / ntiles;
  if (q.dir == TEMPI_DIR_UNPACK && g.L <= 512 &&
      !geom_aligned(g, q.ds, q.ds + g.start, 64)) {
    bytes *= 1.5;
  }
  return (float)std::max(bytes, 8192.0);
}

// The positions are the strided addresses with the memory between the
// requests left out: two grids far apart would otherwise share the windows
// with the gap between them and come out as one window each.  52 packs of 1 280
// rows of 512 B from two grids of 20 MB, us, by the distance of the grids
// (with the gap, ranges ending at windows -> without it, ending anywhere):
//   20 MB 11.8 -> 11.8    16 GiB 16.1 -> 11.8    100 GiB 31.6 -> 11.7
// and 1 000 packs of one 64-KiB region 17.2 -> 11.7.  Returns the length of the
// occupied part.
uint64_t lay_out(const std::vector<Req> &rs, const std::vector<BatchItem> &items,
                 std::vector<Walk> *walk) {
  struct Range {
    uintptr_t first, last;
    size_t r;
  };
  const size_t n = items.size();
  std::vector<Range> ranges(n);
  uintptr_t lo = UINTPTR_MAX, hi = 0;
  for (size_t r = 0; r < n; ++r) {
    Range &q = ranges[r];
    strided_range(rs[r], &q.first, &q.last);
    q.r = r;
    lo = std::min(lo, q.first);
    hi = std::max(hi, q.last);
  }
  // sorted only where gaps may take half of the span or more, told by how many
  // of its 64 parts a request reaches into
  constexpr uintptr_t kParts = 64;
  const uintptr_t part = (hi - lo) / kParts + 1;
  int edges[kParts + 1] = {}, open = 0, occupied = 0;
  for (const Range &q : ranges) {
    ++edges[(q.first - lo) / part];
    --edges[std::min((q.last - 1 - lo) / part + 1, kParts)];
  }
  for (uintptr_t k = 0; k < kParts; ++k) {
    open += edges[k];
    occupied += open > 0;
  }
  const bool gaps = occupied <= (int)kParts / 2;
  if (gaps) {
    std::sort(ranges.begin(), ranges.end(), [](const Range &a, const Range &b) {
      return a.first < b.first;
    });
  }
  constexpr uintptr_t kWindow = (uintptr_t)1 << kWindowShift;
  uintptr_t left_out = lo / kWindow * kWindow, end = gaps ? lo : hi;
  for (const Range &q : ranges) {
    if (q.first > end) {
      left_out += (q.first - end) / kWindow * kWindow;
    }
    end = std::max(end, q.last);
    const BatchItem &it = items[q.r];
    const Geom &g = rs[q.r].g;
    Walk &w = (*walk)[q.r];
    const uint32_t last = it.ntiles - 1;
    const int64_t reach =
        last ? row_offset(it.p, it.p.segdiv.div(last * it.units_per_tile)) : 0;
    w.at = (int64_t)((uintptr_t)(rs[q.r].ds + g.start) - left_out) * 4096;
    w.step = last ? reach * 4096 / (int64_t)last : 0;
    if (g.rows == 1) {
      w.step = (int64_t)((double)g.L * 4096 / it.ntiles);
    }
    w.cost = tile_cost(rs[q.r], it.ntiles);
  }
  return end - left_out;
}

void order_tiles(const std::vector<Req> &rs, const std::vector<BatchItem> &items,
                 uint64_t tiles, int groups, Tile *out, uint32_t *begin) {
  const size_t n = items.size();
  std::vector<Walk> walk(n);
  const uint64_t span = lay_out(rs, items, &walk);
  int shift = kWindowShift;
  while ((span >> shift) > 2 * tiles + 1024) {
    ++shift;
  }
  const int64_t windows = (int64_t)(span >> shift) + 1;
  std::vector<uint32_t> at((size_t)windows + 1, 0);
  const auto window = [&](int64_t pos) {
    return std::min(std::max<int64_t>(pos >> (shift + 12), 0), windows - 1);
  };
  double total = 0;
  for (size_t r = 0; r < n; ++r) {
    int64_t pos = walk[r].at;
    for (uint32_t l = 0; l < items[r].ntiles; ++l, pos += walk[r].step) {
      ++at[(size_t)window(pos) + 1];
    }
    total += (double)walk[r].cost * items[r].ntiles;
  }
  for (int64_t w = 0; w < windows; ++w) {
    at[(size_t)w + 1] += at[(size_t)w];
  }
  for (size_t r = 0; r < n; ++r) {
    int64_t pos = walk[r].at;
    for (uint32_t l = 0; l < items[r].ntiles; ++l, pos += walk[r].step) {
      out[at[(size_t)window(pos)]++] = Tile{(uint32_t)r, l};
    }
  }
  double done = 0;
  int x = 0;
  begin[0] = 0;
  for (uint64_t t = 0; t < tiles && x + 1 < groups; ++t) {
    done += walk[out[t].item].cost;
    while (x + 1 < groups && done >= total * (x + 1) / groups) {
      begin[++x] = (uint32_t)(t + 1);
    }
  }
  while (x + 1 < groups) {
    begin[++x] = (uint32_t)tiles;
  }
}

int plan_tables(const std::vector<Req> &rs, BatchPlan *pl) {
  BatchLaunch &L = pl->launch;
  L = BatchLaunch{};
  std::vector<BatchItem> items;
  std::vector<uint32_t> item_tiles; // tiles of each item
  uint64_t tiles = 0;
  items.reserve(rs.size());
  item_tiles.reserve(rs.size());
  const bool small = rs.size() <= (size_t)kSmallItems;
  for (const Req &r : rs) {
    BatchItem it{};
    bool whole = false;
    int err = fill_kparams(r.g, r.ds, r.dp, r.dir, r.variant, &it.p, &whole);
    if (err) {
      return err;
    }
    it.kind = 4 * r.variant + 2 * (whole ? 1 : 0) + r.dir;
    const VariantDesc &v = kVariants[r.variant];
    const bool four = small ? r.dir == TEMPI_DIR_UNPACK &&
                                  (uint64_t)it.p.units * 4 >=
                                      (uint64_t)units_per_tile(v, true) *
                                          device_cu_count() * 3
                            : r.wide;
    if (four && two_or_four(v.P, v.U)) {
      it.kind += kFour;
    }
    it.units_per_tile = units_per_tile(v, four);
    const uint64_t t = ((uint64_t)it.p.units + it.units_per_tile - 1) /
                       it.units_per_tile;
    tiles += t;
    if (tiles >= (1ull << 31)) {
      return set_error(TEMPI_ERR_UNSUPPORTED, "batch exceeds 2^31 tiles");
    }
    it.ntiles = (uint32_t)t;
    item_tiles.push_back((uint32_t)t);
    items.push_back(it);
  }
  pl->n = (int)items.size();
  L.ntiles = (uint32_t)tiles;
  // One workgroup per tile, dispatched in the tiles' order.  A grid of 8
  // workgroups per CU that looped over them let neighbouring tiles drift
  // apart: halo batches (below) 276 -> 257 us, the random requests 4.51 ->
  // 3.81 ms.
  // (A launch has fewer than 2^32 threads: beyond 2^23 tiles the grid loops.)
  constexpr int64_t cap = 1 << 23;
  if (!items.empty() && small) {
    // tile index in the kernel arguments; only the parameters go to the
    // device table
    SmallIndex &ix = L.ix;
    ix.n = (uint32_t)items.size();
    uint32_t base = 0;
    for (size_t r = 0; r < items.size(); ++r) {
      ix.base[r] = base;
      ix.share[r] = (item_tiles[r] + kXcds - 1) / kXcds;
      ix.ntiles[r] = item_tiles[r];
      base += kXcds * ix.share[r];
    }
    for (size_t r = items.size(); r < (size_t)kSmallItems; ++r) {
      ix.base[r] = base;
    }
    ix.end = base;
    L.small = true;
    L.grid = (int)std::min<int64_t>((int64_t)base, cap);
  } else if ((int64_t)tiles >= 8 * (int64_t)kXcds) {
    L.xcd_split = 1; // the grid follows from the ranges
  } else {
    L.grid = (int)std::max<int64_t>(1, (int64_t)tiles);
  }
  const size_t items_bytes = items.size() * sizeof(BatchItem);
  const size_t tiles_bytes = L.small ? 0 : (size_t)tiles * sizeof(Tile);
  pl->tl_off = (items_bytes + 255) / 256 * 256;
  pl->xb_off = pl->tl_off + (tiles_bytes + 255) / 256 * 256;
  pl->image.assign(pl->xb_off + 256, 0);
  if (!items.empty()) {
    memcpy(pl->image.data(), items.data(), items_bytes);
  }
  uint32_t *begin = reinterpret_cast<uint32_t *>(pl->image.data() + pl->xb_off);
  std::fill(begin, begin + kXcds + 1, (uint32_t)tiles);
  if (tiles_bytes) {
    // grouped by XCD, or one group when the grid is not split
    order_tiles(rs, items, tiles, L.xcd_split ? (int)kXcds : 1,
                reinterpret_cast<Tile *>(pl->image.data() + pl->tl_off), begin);
  }
  if (L.xcd_split) {
    uint32_t most = 0;
    for (uint32_t x = 0; x < kXcds; ++x) {
      most = std::max(most, begin[x + 1] - begin[x]);
    }
    L.grid = (int)std::min<int64_t>((int64_t)most * kXcds, cap);
  }
  return TEMPI_SUCCESS;
}

int plan_batch(const std::vector<Req> &rs, BatchPlan *pl) {
  try {
    return plan_tables(rs, pl);
  } catch (const std::bad_alloc &) {
    return set_error(TEMPI_ERR_NOMEM, "no host memory for the batch tables");
  }
}

// the launch of a plan whose image was copied to device address `dev`
BatchLaunch placed(const BatchPlan &pl, char *dev) {
  BatchLaunch L = pl.launch;
  L.items = reinterpret_cast<const BatchItem *>(dev);
  L.tiles = reinterpret_cast<const Tile *>(dev + pl.tl_off);
  L.xcd_begin = reinterpret_cast<const uint32_t *>(dev + pl.xb_off);
  return L;
}

// Check and resolve the caller's requests: geometry, device addresses and,
// for a request that leaves it to the library (variant -1), the variant
// `pick` returns.  Requests that move nothing are left out; `where` gets
// the caller's index of each resolved request.
struct Resolved {
  std::vector<Req> rs;
  std::vector<int64_t> where;
  int64_t bytes = 0;
};

// the addresses the kernels use for a request's buffers
bool device_buffers(const tempi_batch_request &r, Req *q) {
  void *ds = nullptr, *dp = nullptr;
  if (!device_address(r.strided, &ds) ||
      !device_address(r.packed, &dp, &q->g.host)) {
    return false;
  }
  q->ds = static_cast<const char *>(ds);
  q->dp = static_cast<char *>(dp);
  return true;
}

template <class Buffers, class Pick>
int resolve_requests(const tempi_batch_request *reqs, int64_t n,
                     bool on_device, Buffers &&buffers, Pick &&pick,
                     Resolved *out) {
  // every request is checked before the device is touched
  int err = TEMPI_SUCCESS;
  std::vector<Geom> geoms((size_t)n);
  for (int64_t i = 0; i < n; ++i) {
    if ((err = check_direction(reqs[i].direction)) ||
        (err = make_geom(reqs[i].sb, reqs[i].count, &geoms[(size_t)i]))) {
      return err;
    }
  }
  if (on_device && (err = ensure_runtime())) {
    return err;
  }
  out->rs.reserve((size_t)n);
  out->where.reserve((size_t)n);
  for (int64_t i = 0; i < n; ++i) {
    const tempi_batch_request &r = reqs[i];
    Req q;
    q.g = geoms[(size_t)i];
    if (q.g.rows == 0 || q.g.L == 0) {
      continue;
    }
    if (q.g.L > (1ll << 30)) {
      return set_error(TEMPI_ERR_UNSUPPORTED,
                       "request %lld: rows over 1 GiB are not batched",
                       (long long)i);
    }
    if (!buffers(r, &q)) {
      return set_error(TEMPI_ERR_ARG,
                       "request %lld: buffers must be device-accessible",
                       (long long)i);
    }
    q.dir = r.direction;
    q.variant = r.variant;
    if (q.variant < 0 || q.variant >= kNumVariants) {
      q.variant = pick(q);
    }
    out->bytes += q.g.L * q.g.rows;
    out->rs.push_back(q);
    out->where.push_back(i);
  }
  return TEMPI_SUCCESS;
}

} // namespace
} // namespace tempi

struct tempi_batch {
  int64_t requests = 0;
  int64_t bytes = 0;
  int n = 0;           // items with work
  char *dev = nullptr; // the tables, one allocation
  BatchLaunch launch;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  std::vector<int> variants;
};

static int batch_launch_on(tempi_batch *b, hipStream_t s) {
  if (b->launch.ntiles == 0) {
    return TEMPI_SUCCESS;
  }
  launch_kernel(b->launch, s);
  TEMPI_HIP_CHECK(hipGetLastError());
  return TEMPI_SUCCESS;
}

namespace {

// The device tables and launch shape of a batch of resolved requests.
int build_batch(tempi_batch *b, const std::vector<Req> &rs) {
  hipStream_t s = library_stream();
  BatchPlan pl;
  int err = plan_batch(rs, &pl);
  if (err) {
    return err;
  }
  b->n = pl.n;
  if (hipSuccess != hipMalloc(&b->dev, pl.image.size())) {
    (void)hipGetLastError();
    b->dev = nullptr;
    return set_error(TEMPI_ERR_NOMEM, "batch table allocation failed");
  }
  b->launch = placed(pl, b->dev);
  // one upload, outside any capture
  if (hipSuccess != hipMemcpyAsync(b->dev, pl.image.data(), pl.image.size(),
                                   hipMemcpyHostToDevice, s) ||
      hipSuccess != hipStreamSynchronize(s)) {
    (void)hipGetLastError();
    (void)hipFree(b->dev);
    b->dev = nullptr;
    return set_error(TEMPI_ERR_HIP, "batch table upload failed");
  }
  return TEMPI_SUCCESS;
}

// Tiles of a resolved request (one workgroup pass each) in a batch of more
// than kSmallItems.
uint64_t tiles_of(const Req &q) {
  const uint64_t units = (uint64_t)units_of(q.g, q.variant);
  const uint64_t per_tile = units_per_tile(kVariants[q.variant], q.wide);
  return (units + per_tile - 1) / per_tile;
}

bool fits(const Req &q, int variant) {
  return units_of(q.g, variant) < kMaxUnits;
}

// of the variants that hold a request, the one that splits it into the fewest
// tiles
int fewest_tiles(const Req &q) {
  Req r = q;
  uint64_t best = UINT64_MAX;
  int variant = q.variant;
  for (r.variant = 0; r.variant < kNumVariants; ++r.variant) {
    const uint64_t t = tiles_of(r);
    if (t < best && fits(q, r.variant)) {
      best = t;
      variant = r.variant;
    }
  }
  return variant;
}

// the kernel like `variant` whose units are longer than 12 B or 32 B of a row
int wider(int variant) {
  return variant == 12 ? 7 : variant == 16 ? 13 : variant == 17 ? 15 : variant;
}

// A request is not split, so its units have to stay below kMaxUnits, and the
// rules pick by speed whatever the size: rows of host memory, as units of
// 16 B, reach the limit at 32 GiB.  Returns q.variant or, where it does not
// hold the request, the closed-form rule's or the one of fewest tiles; for a
// variant the caller asked for, the wider one like it.
int fitting_variant(const Req &q, bool asked) {
  if (fits(q, q.variant)) {
    return q.variant;
  }
  if (asked) {
    return wider(q.variant);
  }
  const int rule = heuristic_variant(q.g, q.ds, q.dp, q.dir);
  return fits(q, rule) ? rule : fewest_tiles(q);
}

// The default policy's rule for batches with more tiles than the grid runs at
// once.  The learned selector ranks a copy's variants by the time of the copy
// alone; among other requests what counts is how many bytes a workgroup keeps
// in flight, so the rule takes the variant whose lanes all have a word to
// move and which moves most rows per pass.  Rows under 16 B take the 12-B
// words' kernel whatever their length: a row is one unit of one or two
// accesses there and a lane has two rows in flight, where the other
// lane-per-row kernels hold four words of one row, most of which a short row
// does not have.  Unpacks of rows of 24-47 B take four lanes of 8 B to a
// row, and those and unpacks of rows over 512 B read the packed bytes, which
// nobody reads again, nontemporal: the caches are left to the lines that short
// rows write in part.  Packs gain or lose by nontemporal loads with the size
// of the batch (64 subdomains of 96^3, rows of 8 B, pack + unpack 78 -> 57 us,
// of 12 B 92 -> 111) and do without.  Random requests of 4 KiB - 16 MiB, strides
// up to 512 B past the row, and halo regions (one pack and one unpack, three
// sets of buffers in turn), the former picks (the selector's, or for requests
// under 1 MiB the rule's for single copies) -> this rule on MI355X:
//                                              pack          unpack
//   2 000, rows of 4 B - 4 KiB               2.39 -> 2.24   2.72 -> 1.94 ms
//   the same, all multiples of 16 B apart    2.69 -> 2.36   2.41 -> 2.05 ms
//   2 000, rows of 1 - 224 B, odd lengths    5.51 -> 5.02   8.15 -> 6.54 ms
//   4 000 of up to 1 MiB, rows 1 - 224 B     1.27 -> 0.83   1.94 -> 0.89 ms
//   64 subdomains of 128^3 doubles, radius 3      257 -> 232 us together
// Each length's variant is the best or within 1 % of it over sixteen such
// random batches.  Rows to or from host memory are bound by the link, which
// the dword kernel keeps fullest (48 MiB of 4-KiB rows unpacked at 57.2 GB/s,
// 53.1 with 16-B words; packed 55.5 and 54.4).  Batches of few requests or few
// tiles keep the selector's picks: the three faces of a 512^3 grid took 9.26 us
// with them, 9.91 us with the closed-form rule's.
int saturated_variant(const Geom &g, int dir) {
  const int64_t L = g.L;
  const bool unpack = dir == TEMPI_DIR_UNPACK;
  if (g.host) {
    return 9;
  }
  if (L >= 256) {
    return unpack && L > 512 ? 3 : 4;
  }
  if (L >= 128) {
    return 5;
  }
  if (L >= 48) {
    return 6;
  }
  if (L >= 24) {
    return unpack ? 17 : 7;
  }
  return L < 16 || L >= 20 ? 12 : 7;
}

bool saturated(const std::vector<Req> &rs) {
  if (rs.size() <= (size_t)kSmallItems) {
    return false;
  }
  uint64_t tiles = 0;
  for (const Req &q : rs) {
    tiles += tiles_of(q);
  }
  return tiles > (uint64_t)device_cu_count() * 8;
}

bool asked_for(const tempi_batch_request &r) {
  return r.variant >= 0 && r.variant < kNumVariants;
}

// gives the requests whose variant was left to the library `pick`'s
template <class Pick>
void repick(const tempi_batch_request *reqs, Resolved *q, Pick &&pick) {
  for (size_t k = 0; k < q->rs.size(); ++k) {
    if (!asked_for(reqs[q->where[k]])) {
      q->rs[k].variant = pick(q->rs[k]);
    }
  }
}

void fit_variants(const tempi_batch_request *reqs, Resolved *q) {
  for (size_t k = 0; k < q->rs.size(); ++k) {
    Req &r = q->rs[k];
    r.variant = fitting_variant(r, asked_for(reqs[q->where[k]]));
  }
}

} // namespace

TEMPI_EXPORT int tempi_batch_create(const tempi_batch_request *reqs, int64_t n,
                                    int method, tempi_batch **out) {
  if (!out || (n > 0 && !reqs) || n < 0) {
    return set_error(TEMPI_ERR_ARG, "bad argument");
  }
  *out = nullptr;
  std::unique_ptr<tempi_batch> owner(new tempi_batch());
  tempi_batch *b = owner.get();
  b->requests = n;
  b->variants.assign((size_t)n, -1);
  Resolved q;
  std::vector<Req> &rs = q.rs;
  // the per-copy policy first (in small batches the learned selector's
  // picks for requests under 1 MiB ran the faces of 128^3 - 256^3 float
  // grids 5-28 % faster than the closed-form rule's), then the batch rule
  // for batches that saturate the grid (saturated_variant).  The
  // selector evaluates all the batch's new shapes in one inference first:
  // one launch per shape took 0.14 s to create the 4 096-request batch.
  int err = resolve_requests(
      reqs, n, true, device_buffers, [](const Req &) { return -1; }, &q);
  if (err) {
    return err;
  }
  b->bytes = q.bytes;
  if (method == TEMPI_SELECT_MODEL ||
      (method == TEMPI_SELECT_DEFAULT && model_available())) {
    std::vector<CopyShape> shapes;
    for (const Req &r : rs) {
      if (r.variant < 0) {
        shapes.push_back({r.g, r.ds, r.dp, r.dir});
      }
    }
    model_prefetch(shapes);
  }
  for (Req &r : rs) {
    if (r.variant < 0) {
      r.variant = choose(r.g, r.ds, r.dp, r.dir, method, library_stream(),
                         CopyUse::kInBatch)
                      .variant;
    }
  }
  if (method == TEMPI_SELECT_DEFAULT && saturated(rs)) {
    repick(reqs, &q, [](const Req &r) { return saturated_variant(r.g, r.dir); });
  }
  fit_variants(reqs, &q);
  for (size_t k = 0; k < rs.size(); ++k) {
    b->variants[(size_t)q.where[k]] = rs[k].variant;
  }
  if ((err = build_batch(b, rs))) {
    return err;
  }
  *out = owner.release();
  return TEMPI_SUCCESS;
}

TEMPI_EXPORT int tempi_batch_launch(tempi_batch *b, void *stream) {
  if (!b) {
    return set_error(TEMPI_ERR_ARG, "null batch");
  }
  TraceRange trace("tempi_batch_launch");
  hipStream_t s = stream ? static_cast<hipStream_t>(stream) : library_stream();
  int err = batch_launch_on(b, s);
  if (!err) {
    ++counters().batch_launches;
  }
  return err;
}

namespace {

// A graph of the launches of `n` batches, each depending on the one before
// (kernel nodes added directly: no stream capture).  The batches' device
// tables must outlive the graph.
int build_graph(tempi_batch *const *bs, int64_t n, hipGraph_t *graph,
                hipGraphExec_t *exec, int64_t *nodes) {
  *graph = nullptr;
  *exec = nullptr;
  *nodes = 0;
  TEMPI_HIP_CHECK(hipGraphCreate(graph, 0));
  hipGraphNode_t prev = nullptr;
  int err = TEMPI_SUCCESS;
  for (int64_t i = 0; i < n && !err; ++i) {
    const BatchLaunch &l = bs[i]->launch;
    if (l.ntiles == 0) {
      continue;
    }
    hipKernelNodeParams kp{};
    void *args_small[] = {const_cast<SmallIndex *>(&l.ix),
                          const_cast<const BatchItem **>(&l.items)};
    uint32_t ntiles = l.ntiles;
    int xcd_split = l.xcd_split;
    void *args_big[] = {const_cast<const BatchItem **>(&l.items),
                        const_cast<const Tile **>(&l.tiles),
                        const_cast<const uint32_t **>(&l.xcd_begin), &ntiles,
                        &xcd_split};
    kp.func = l.small ? reinterpret_cast<void *>(&k_batch_small)
                      : reinterpret_cast<void *>(&k_batch);
    kp.gridDim = dim3((unsigned)l.grid);
    kp.blockDim = dim3(kBlock);
    kp.sharedMemBytes = 0;
    kp.kernelParams = l.small ? args_small : args_big;
    kp.extra = nullptr;
    hipGraphNode_t node = nullptr;
    const hipError_t e = hipGraphAddKernelNode(&node, *graph, prev ? &prev : nullptr,
                                               prev ? 1 : 0, &kp);
    if (e != hipSuccess) {
      err = set_error(TEMPI_ERR_HIP, "hipGraphAddKernelNode: %s",
                      hipGetErrorString(e));
      break;
    }
    prev = node;
    ++*nodes;
  }
  if (!err) {
    const hipError_t e = hipGraphInstantiate(exec, *graph, nullptr, nullptr, 0);
    if (e != hipSuccess) {
      err = set_error(TEMPI_ERR_HIP, "hipGraphInstantiate: %s",
                      hipGetErrorString(e));
    }
  }
  if (err) {
    (void)hipGetLastError();
    if (*exec) {
      (void)hipGraphExecDestroy(*exec);
    }
    (void)hipGraphDestroy(*graph);
    *graph = nullptr;
    *exec = nullptr;
  }
  return err;
}

} // namespace

TEMPI_EXPORT int tempi_batch_graph_launch(tempi_batch *b, void *stream) {
  if (!b) {
    return set_error(TEMPI_ERR_ARG, "null batch");
  }
  if (b->launch.ntiles == 0) {
    return TEMPI_SUCCESS;
  }
  TraceRange trace("tempi_batch_graph_launch");
  if (!b->exec) {
    int64_t nodes = 0;
    int err = build_graph(&b, 1, &b->graph, &b->exec, &nodes);
    if (err) {
      return err;
    }
  }
  hipStream_t s = stream ? static_cast<hipStream_t>(stream) : library_stream();
  TEMPI_HIP_CHECK(hipGraphLaunch(b->exec, s));
  ++counters().graph_launches;
  return TEMPI_SUCCESS;
}

struct tempi_graph {
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int64_t nodes = 0;
};

TEMPI_EXPORT int tempi_graph_create(tempi_batch *const *batches, int64_t n,
                                    tempi_graph **out) {
  if (!out || n < 0 || (n > 0 && !batches)) {
    return set_error(TEMPI_ERR_ARG, "bad argument");
  }
  *out = nullptr;
  for (int64_t i = 0; i < n; ++i) {
    if (!batches[i]) {
      return set_error(TEMPI_ERR_ARG, "null batch %lld", (long long)i);
    }
  }
  int err = ensure_runtime();
  if (err) {
    return err;
  }
  std::unique_ptr<tempi_graph> g(new tempi_graph());
  if ((err = build_graph(batches, n, &g->graph, &g->exec, &g->nodes))) {
    return err;
  }
  *out = g.release();
  return TEMPI_SUCCESS;
}

TEMPI_EXPORT int tempi_graph_launch(tempi_graph *g, void *stream) {
  if (!g) {
    return set_error(TEMPI_ERR_ARG, "null graph");
  }
  if (g->nodes == 0) {
    return TEMPI_SUCCESS;
  }
  TraceRange trace("tempi_graph_launch");
  hipStream_t s = stream ? static_cast<hipStream_t>(stream) : library_stream();
  TEMPI_HIP_CHECK(hipGraphLaunch(g->exec, s));
  ++counters().graph_launches;
  return TEMPI_SUCCESS;
}

TEMPI_EXPORT int tempi_graph_destroy(tempi_graph *g) {
  if (!g) {
    return TEMPI_SUCCESS;
  }
  if (g->exec) {
    // the graph may have been launched on any stream
    (void)hipDeviceSynchronize();
    (void)hipGraphExecDestroy(g->exec);
  }
  if (g->graph) {
    (void)hipGraphDestroy(g->graph);
  }
  delete g;
  return TEMPI_SUCCESS;
}

TEMPI_EXPORT int tempi_batch_info(const tempi_batch *b, int64_t *requests,
                                  int64_t *tiles, int64_t *packed_bytes) {
  if (!b) {
    return set_error(TEMPI_ERR_ARG, "null batch");
  }
  if (requests) {
    *requests = b->requests;
  }
  if (tiles) {
    *tiles = b->launch.ntiles;
  }
  if (packed_bytes) {
    *packed_bytes = b->bytes;
  }
  return TEMPI_SUCCESS;
}

TEMPI_EXPORT int tempi_batch_variant(const tempi_batch *b, int64_t i,
                                     int *variant) {
  if (!b || i < 0 || i >= (int64_t)b->variants.size() || !variant) {
    return set_error(TEMPI_ERR_ARG, "bad argument");
  }
  *variant = b->variants[i];
  return TEMPI_SUCCESS;
}

TEMPI_EXPORT int tempi_batch_destroy(tempi_batch *b) {
  if (!b) {
    return TEMPI_SUCCESS;
  }
  if (b->exec || b->dev) {
    // the batch may have been launched on any stream
    (void)hipDeviceSynchronize();
  }
  if (b->exec) {
    (void)hipGraphExecDestroy(b->exec);
  }
  if (b->graph) {
    (void)hipGraphDestroy(b->graph);
  }
  if (b->dev) {
    (void)hipFree(b->dev);
  }
  delete b;
  return TEMPI_SUCCESS;
}

// ---------------------------------------------------------------------------
// the batch entry point that allocates nothing
// ---------------------------------------------------------------------------
//
// tempi_batch_run_noalloc resolves and launches a batch in one call, with
// the request and tile tables in a file-scope device array instead of
// memory the library allocates, for callers that cannot allocate device
// memory.  The array's host-side name is only a stand-in for it: host code
// uses the address hipGetSymbolAddress reports for the current device,
// taken once per device on the first call, and never the name itself.

namespace tempi {
namespace {

// largest table image (request parameters, tile records, XCD bounds) a
// call can place: 4 MiB holds about 4 000 requests over 2^19 tiles (the
// 1 664-request halo batch of 64 subdomains of 128^3 needs 0.5 MiB)
constexpr size_t kScratchBytes = 4u << 20;

struct ScratchSlot {
  std::once_flag once;
  int err = TEMPI_SUCCESS;
  char *ptr = nullptr;             // the array's address on this device
  hipEvent_t uploaded = nullptr;   // the last call's table upload
  std::mutex mu;
  std::vector<char> image;         // that upload's host source
};
constexpr int kMaxDevices = 64;
ScratchSlot g_scratch_slots[kMaxDevices];

} // namespace
} // namespace tempi

static __device__ __align__(256) char scratch[tempi::kScratchBytes];

namespace tempi {
namespace {

int scratch_slot(ScratchSlot **out) {
  int dev = 0;
  TEMPI_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) {
    return set_error(TEMPI_ERR_UNSUPPORTED, "device %d", dev);
  }
  ScratchSlot &sl = g_scratch_slots[dev];
  std::call_once(sl.once, [&sl] {
    void *p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) {
      (void)hipGetLastError();
      sl.err = set_error(TEMPI_ERR_HIP, "hipGetSymbolAddress(scratch): %s",
                         hipGetErrorString(e));
      return;
    }
    e = hipEventCreateWithFlags(&sl.uploaded, hipEventDisableTiming);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      sl.err = set_error(TEMPI_ERR_HIP, "event creation: %s",
                         hipGetErrorString(e));
      return;
    }
    sl.ptr = static_cast<char *>(p);
  });
  if (sl.err != TEMPI_SUCCESS) {
    return set_error(sl.err, "static scratch of device %d is unusable", dev);
  }
  *out = &sl;
  return TEMPI_SUCCESS;
}

} // namespace
} // namespace tempi

namespace {

// The variants and tables of tempi_batch_run_noalloc.  The closed-form rule:
// the learned selector and trial timings would allocate device memory on
// first use.
template <class Buffers>
int plan_noalloc(const tempi_batch_request *reqs, int64_t n, bool on_device,
                 Buffers &&buffers, Resolved *q, BatchPlan *pl) {
  int err = resolve_requests(
      reqs, n, on_device, buffers,
      [](const Req &r) { return heuristic_variant(r.g, r.ds, r.dp, r.dir); }, q);
  if (err || q->rs.empty()) {
    return err;
  }
  if (saturated(q->rs)) {
    repick(reqs, q, [](const Req &r) { return saturated_variant(r.g, r.dir); });
  }
  fit_variants(reqs, q);
  if ((err = plan_batch(q->rs, pl))) {
    return err;
  }
  if (pl->image.size() > kScratchBytes) {
    // as many rows to a tile record as a kernel moves
    for (Req &r : q->rs) {
      r.wide = true;
      if (r.variant != 12) { // four of its units to a lane are as many rows
        r.variant = wider(r.variant);
      }
    }
    repick(reqs, q, fewest_tiles);
    err = plan_batch(q->rs, pl);
  }
  return err;
}

} // namespace

TEMPI_EXPORT int tempi_batch_run_noalloc(const tempi_batch_request *reqs,
                                         int64_t n, void *stream) {
  if ((n > 0 && !reqs) || n < 0) {
    return set_error(TEMPI_ERR_ARG, "bad argument");
  }
  Resolved q;
  BatchPlan pl;
  int err = plan_noalloc(reqs, n, true, device_buffers, &q, &pl);
  if (err || q.rs.empty()) {
    return err;
  }
  if (pl.image.size() > kScratchBytes) {
    return set_error(TEMPI_ERR_UNSUPPORTED,
                     "batch tables of %zu B (%zu requests, %u tiles) exceed "
                     "the %zu B of static scratch",
                     pl.image.size(), q.rs.size(), pl.launch.ntiles,
                     kScratchBytes);
  }
  ScratchSlot *sl = nullptr;
  if ((err = scratch_slot(&sl))) {
    return err;
  }
  TraceRange trace("tempi_batch_run_noalloc");
  hipStream_t s = stream ? static_cast<hipStream_t>(stream) : library_stream();
  std::lock_guard<std::mutex> lk(sl->mu);
  // the previous upload has read its host image (a copy from pageable
  // memory may finish after the call that enqueued it returned)
  TEMPI_HIP_CHECK(hipEventSynchronize(sl->uploaded));
  sl->image.swap(pl.image);
  TEMPI_HIP_CHECK(hipMemcpyAsync(sl->ptr, sl->image.data(), sl->image.size(),
                                 hipMemcpyHostToDevice, s));
  TEMPI_HIP_CHECK(hipEventRecord(sl->uploaded, s));
  launch_kernel(placed(pl, sl->ptr), s);
  TEMPI_HIP_CHECK(hipGetLastError());
  ++counters().batch_launches;
  return TEMPI_SUCCESS;
}

namespace {

// What tempi_batch_run_noalloc would launch for requests whose addresses are
// numbers: the same plan, read back from the tables' host image.
int emulate_batch(const tempi_batch_request *reqs, int64_t n,
                  bool packed_on_host, int32_t *variants,
                  tempi_batch_emulation *out) {
  *out = tempi_batch_emulation{};
  Resolved q;
  BatchPlan pl;
  const int err = plan_noalloc(
      reqs, n, false,
      [&](const tempi_batch_request &r, Req *rq) {
        rq->ds = static_cast<const char *>(r.strided);
        rq->dp = static_cast<char *>(r.packed);
        rq->g.host = packed_on_host;
        return true;
      },
      &q, &pl);
  if (err) {
    return err;
  }
  if (variants) {
    std::fill(variants, variants + n, -1);
    for (size_t k = 0; k < q.rs.size(); ++k) {
      variants[q.where[k]] = q.rs[k].variant;
    }
  }
  out->requests = (int64_t)q.rs.size();
  out->fits_static_tables = pl.image.size() <= kScratchBytes;
  if (q.rs.empty()) {
    out->exact = 1;
    return TEMPI_SUCCESS;
  }
  const BatchLaunch &L = pl.launch;
  out->tiles = L.ntiles;
  out->grid = L.grid;
  const BatchItem *items = reinterpret_cast<const BatchItem *>(pl.image.data());
  std::vector<uint64_t> first(q.rs.size() + 1, 0);
  for (size_t r = 0; r < q.rs.size(); ++r) {
    first[r + 1] = first[r] + items[r].ntiles;
  }
  std::vector<uint8_t> runs(first.back(), 0);
  bool inside = true;
  const auto run = [&](uint32_t xcd, uint32_t r, uint32_t l) {
    if (r >= q.rs.size() || l >= items[r].ntiles) {
      inside = false;
      return;
    }
    runs[first[r] + l] += runs[first[r] + l] < 2;
    ++out->xcd_tiles[xcd];
    out->xcd_cost[xcd] += tile_cost(q.rs[r], items[r].ntiles);
  };
  if (L.small) {
    for (uint32_t r = 0; r < L.ix.n; ++r) {
      for (uint32_t k = 0; k < kXcds * L.ix.share[r]; ++k) {
        const uint32_t l = k % kXcds * L.ix.share[r] + k / kXcds;
        if (l < L.ix.ntiles[r]) {
          run((L.ix.base[r] + k) % kXcds, r, l);
        }
      }
    }
  } else {
    const Tile *tiles = reinterpret_cast<const Tile *>(pl.image.data() + pl.tl_off);
    const uint32_t *begin =
        reinterpret_cast<const uint32_t *>(pl.image.data() + pl.xb_off);
    for (uint32_t x = 0; x < (L.xcd_split ? kXcds : 1u); ++x) {
      const uint32_t end = L.xcd_split ? begin[x + 1] : L.ntiles;
      for (uint32_t t = L.xcd_split ? begin[x] : 0; t < end; ++t) {
        run(L.xcd_split ? x : t % kXcds, tiles[t].item, tiles[t].tile);
      }
    }
  }
  out->exact = inside && std::all_of(runs.begin(), runs.end(),
                                     [](uint8_t c) { return c == 1; });
  return TEMPI_SUCCESS;
}

} // namespace

TEMPI_EXPORT int tempi_batch_emulate(const tempi_batch_request *reqs, int64_t n,
                                     int packed_on_host, int32_t *variants,
                                     tempi_batch_emulation *out) {
  if ((n > 0 && !reqs) || n < 0 || !out) {
    return set_error(TEMPI_ERR_ARG, "bad argument");
  }
  try {
    return emulate_batch(reqs, n, packed_on_host != 0, variants, out);
  } catch (const std::bad_alloc &) {
    return set_error(TEMPI_ERR_NOMEM, "no host memory for the batch plan");
  }
}
