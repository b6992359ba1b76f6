// Node tiles: the products of the scalar-mass (MASS3) and 3x3-block (BSR3)
// layouts with x staged in LDS and no reduction across a wavefront's rows.
//
// What bounds these products: every entry gathers the 3K values of its node,
// 24K bytes against the 12 (MASS3) or 76 (BSR3) bytes of the entry itself.
// Row kernels take them from the caches, 28 times per node; at 1.9M DoF that
// traffic, at 6.5-7 TB/s, was the whole time of the k-column steps.  Here a
// workgroup owns a tile of consecutive node rows (the numbering is spatially
// local), reads each node it references once into LDS (3-4 times its own rows
// instead of 28) and forms the rows from there.
//
// Rows of a tile are sorted by length and cut into slices of 16; four lanes
// share a row.  A "quad" is the next four entries of each of the 16 rows: lane
// 4r + e loads entry e of row r, values and 16-bit list places in unit stride
// without row offsets, and hands them to the row's other lanes by DPP.  With
// K >= 4 each of the four lanes owns one column (groups of four columns per
// workgroup), so sums stay in their lane; with K = 2 and 1 the four lanes are
// 2 columns x 2 and 1 x 4 entries, and one or two DPP additions close a row.
// The row kernels' butterflies cost 24 LDS permutes per row at K = 4.
//
// Long slices (the vertex rows of P2 meshes hold 65 entries, edge rows 19-27)
// are split over several wavefronts with partial sums in LDS added in a fixed
// order, as far as a tile has wavefronts beside one per slice: with one wavefront
// per slice the longest one set the time of the tile.  On a P2 mesh of 60k nodes
// the longest wavefront of a tile carries 6 quads at 128 rows, 8 at 160, 10
// (median; at most 18) at 224, where two can share, and 7 (9) at the stiffness's
// 96 rows of 8 wavefronts.
//
// Measured (FP64 fused Chebyshev step, us; in brackets the fastest of the row
// kernels, LDS tiles and wide layouts, as the autotuner picks it without node
// tiles; one MI355X):
//   DoF        K = 1         K = 2         K = 4         K = 8         K = 16
//   51.5k    4.0 (5.2)     4.5 (6.1)     5.5 (9.2)     8.1 (14.3)   12.7 (26.7)
//   439k    14.8 (20.8)   17.1 (26.0)   24.4 (49.0)   38.8 (91.9)   82.0 (177)
//   1.90M   50.1 (72.0)   69.1 (109)     108 (229)     215 (486)     456 (954)
// At
// 1.9M DoF the step moves 487 MB at K = 4 (counted): 4.5 TB/s, against 5.6 TB/s
// of a copy of that size.  Loads wider than 8 bytes, lists read once per
// wavefront and 64 registers (two workgroups of 16 wavefronts per CU) each
// counted: with 8 wavefronts or spills the same step took 2-4 times as long.  A
// persistent form with the next tile's x in registers was no faster (137 us at
// K = 4), nor was an epilogue through LDS with contiguous stores (143 us).
#include <omp.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <initializer_list>
#include <memory>
#include <new>
#include <numeric>
#include <type_traits>
#include <vector>

#include "nmgpu_device.h"
#include "nmgpu_internal.h"

namespace nmg {

// Place 0 of a tile's nodes in LDS is a node of zeros, which the slots that pad
// a row's quads point at: 0 * x of some node would carry an infinity or NaN
// into rows that do not touch it.
constexpr uint16_t kTileZero = 0;

TilePlan::~TilePlan() {
  for (void* p : {(void*)un, (void*)tcols, (void*)lrow, (void*)eidx, (void*)perm})
    if (p) (void)hipFree(p);
}

// Device memory of M's tiles, within its limit; throws NMG_ENOMEM.
template <class T>
static T* tile_alloc(DevMat& M, size_t count) {
  T* p = nullptr;
  const int64_t bytes = (int64_t)(sizeof(T) * std::max<size_t>(count, 1));
  if ((M.tile_limit >= 0 && M.tile_bytes + bytes > M.tile_limit) || hipMalloc(&p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    throw Error{NMG_ENOMEM, "no memory for node tiles (" + std::to_string(bytes) + " bytes)"};
  }
  M.tile_bytes += bytes;
  return p;
}

template <class T, class A>
static T* to_device(DevMat& M, const std::vector<T, A>& v) {
  T* p = tile_alloc<T>(M, v.size());
  const hipError_t e = hipMemcpy(p, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    (void)hipFree(p);
    NMG_HIP(e);
  }
  return p;
}

// The nodes of one thread's current tile with their places.  calloc: of an array
// over all nodes only the pages around a thread's tiles are ever backed by memory
// (a hash table of the tile's size took 1.6 times as long to lay out 600k nodes).
class NodeTable {
 public:
  explicit NodeTable(int64_t nb) : slot_((Slot*)std::calloc((size_t)nb, sizeof(Slot)), &std::free) {
    if (!slot_) throw std::bad_alloc();
  }
  void clear() { ++now_; }  // at most a tile per node: never wraps
  // whether node c is new, and takes `place`
  bool add(int32_t c, int place) {
    if (slot_.get()[c].epoch == now_) return false;
    slot_.get()[c] = Slot{now_, place};
    return true;
  }
  int operator[](int32_t c) const { return slot_.get()[c].place; }  // of a node that is there

 private:
  struct Slot {
    uint32_t epoch;
    int32_t place;
  };
  std::unique_ptr<Slot, void (*)(void*)> slot_;
  uint32_t now_ = 0;
};

// f(i, thread) for i < n on all threads; std::bad_alloc passes to the caller
// instead of ending the process at the end of the parallel region
template <class F>
static void parallel_for(int64_t n, F&& f) {
  std::atomic<bool> failed{false};
#pragma omp parallel for schedule(dynamic, 16)
  for (int64_t i = 0; i < n; ++i) {
    if (failed) continue;
    try {
      f(i, omp_get_thread_num());
    } catch (const std::bad_alloc&) {
      failed = true;
    }
  }
  if (failed) throw std::bad_alloc();
}

bool tile_layout(int64_t nb, const int64_t* rp, const int32_t* ci, int rows, int cap, int waves, int pack,
                 HostTiles& H) {
  const int spt = rows / kSliceRows;
  if (spt < 1 || spt > waves) return false;  // one wavefront at least per slice
  const int64_t nblk = (nb + rows - 1) / rows;
  int64_t longest = 0;
  for (int64_t r = 0; r < nb; ++r) longest = std::max(longest, rp[r + 1] - rp[r]);
  if (longest + 1 > cap || cap > 65534 || rp[nb] > (int64_t)1 << 28 || nb > (int64_t)1 << 28) return false;
  // cut every aligned run of `rows` rows where its node list would pass cap
  struct Cut {
    int64_t r0, r1;
    std::vector<int32_t> nodes;
  };
  std::vector<std::vector<Cut>> blk(nblk);
  std::vector<std::unique_ptr<NodeTable>> tables((size_t)omp_get_max_threads());
  auto table = [&](int thread) -> NodeTable& {
    if (!tables[thread]) tables[thread].reset(new NodeTable(nb));
    return *tables[thread];
  };
  parallel_for(nblk, [&](int64_t b, int thread) {
    NodeTable& seen = table(thread);
    std::vector<int32_t> fresh;
    const int64_t end = std::min(nb, (b + 1) * rows);
    Cut cur{b * rows, b * rows, {}};
    seen.clear();
    for (int64_t r = b * rows; r < end;) {
      fresh.clear();
      auto see = [&](int32_t c) {
        if (seen.add(c, 0)) fresh.push_back(c);
      };
      for (int64_t k = rp[r]; k < rp[r + 1]; ++k) see(ci[k]);
      see((int32_t)r);  // the row's own x, for the epilogue
      if ((int64_t)(cur.nodes.size() + fresh.size()) > cap) {
        std::sort(cur.nodes.begin(), cur.nodes.end());
        blk[b].push_back(std::move(cur));
        cur = Cut{r, r, {}};
        seen.clear();
        continue;  // the row opens the next tile
      }
      cur.nodes.insert(cur.nodes.end(), fresh.begin(), fresh.end());
      cur.r1 = ++r;
    }
    std::sort(cur.nodes.begin(), cur.nodes.end());
    blk[b].push_back(std::move(cur));
  });
  std::vector<const Cut*> cut;
  for (auto& v : blk)
    for (auto& c : v) cut.push_back(&c);
  const int64_t nt = (int64_t)cut.size();
  H.ntiles = nt;
  H.spt = spt;
  H.lrow.assign(nt * spt * kSliceRows, 0xffff);
  std::vector<int64_t> first(nt + 1, 0);
  H.max_nodes = 0;
  for (int64_t t = 0; t < nt; ++t) {
    first[t + 1] = first[t] + (int64_t)cut[t]->nodes.size();
    H.max_nodes = std::max(H.max_nodes, (int)cut[t]->nodes.size());
  }
  H.tcols.resize(first[nt]);
  std::vector<int2> sd(nt * spt, int2{0, 0});  // per slice {first quad, quads}
  // rows of a tile in order of falling length, 16 to a slice
  parallel_for(nt, [&](int64_t t, int) {
    const Cut& c = *cut[t];
    std::copy(c.nodes.begin(), c.nodes.end(), H.tcols.begin() + first[t]);
    std::vector<int32_t> ord(c.r1 - c.r0);
    std::iota(ord.begin(), ord.end(), (int32_t)c.r0);
    std::stable_sort(ord.begin(), ord.end(),
                     [&](int32_t a, int32_t b) { return rp[a + 1] - rp[a] > rp[b + 1] - rp[b]; });
    for (size_t i = 0; i < ord.size(); ++i) {
      const int64_t s = t * spt + (int64_t)(i / kSliceRows);
      H.lrow[s * kSliceRows + i % kSliceRows] = (uint16_t)(ord[i] - c.r0);
      if (i % kSliceRows == 0) {
        const int nq = (int)((rp[ord[i] + 1] - rp[ord[i]] + 3) / 4);
        sd[s].y = (nq + pack - 1) / pack * pack;
      }
    }
  });
  int64_t q = 0;
  for (auto& s : sd) {
    s.x = (int)q;
    q += s.y;
  }
  if (q * 64 > (int64_t)1 << 30) return false;
  H.quads = q;
  // work units: the slices of a tile cut into runs of at most m quads, m the
  // smallest that leaves no more partial sums (one for each run of a slice after
  // its first) than a full tile has wavefronts to spare: short tiles would
  // otherwise cost every workgroup LDS for up to 15 of them, and with it the
  // second workgroup of a CU (223k DoF, K = 16, 128 rows: 63 us so, 43 now)
  H.un.assign(nt * waves, TileUnit{0, 1, 0, 0, 0, 0, -1, 0});
  H.max_extra = 0;
  for (int64_t t = 0; t < nt; ++t) {
    const Cut& c = *cut[t];
    const int own = (int)(std::lower_bound(c.nodes.begin(), c.nodes.end(), (int32_t)c.r0) - c.nodes.begin());
    const int ns = (int)((c.r1 - c.r0 + kSliceRows - 1) / kSliceRows);
    auto units = [&](int m) {
      int n = 0;
      for (int i = 0; i < ns; ++i) n += std::max(1, (sd[t * spt + i].y + m - 1) / m);
      return n;
    };
    int m = pack;
    while (units(m) - ns > waves - spt) m += pack;
    int u = 0, extra = 0;
    for (int w = 0; w < waves; ++w) {
      H.un[t * waves + w].list = (int)first[t];
      H.un[t * waves + w].nodes = (int)c.nodes.size();
      H.un[t * waves + w].row0 = (int)c.r0;
      H.un[t * waves + w].own = own;
    }
    for (int i = 0; i < ns; ++i) {
      const int2 d = sd[t * spt + i];
      const int np = std::max(1, (d.y + m - 1) / m);
      for (int p = 0; p < np; ++p) {
        TileUnit& w = H.un[t * waves + u++];
        w.q0 = d.x + p * m;
        w.nq = std::min(m, d.y - p * m);
        w.slice = (int)(t * spt + i);
        w.part = p | np << 8 | extra << 16;
      }
      extra += np - 1;
    }
    H.max_extra = std::max(H.max_extra, extra);
  }
  H.eidx.resize(q * 64);
  H.perm.resize(q * 64);
  // Entries of a row in an order that spreads the simultaneous LDS reads of
  // four neighbouring rows over the banks: row i of a slice takes at place e
  // an entry whose node's place in the list is (e + i) mod 4, while it has one
  parallel_for(nt, [&](int64_t t, int thread) {
    const Cut& c = *cut[t];
    NodeTable& local = table(thread);
    local.clear();
    for (size_t i = 0; i < c.nodes.size(); ++i) local.add(c.nodes[i], (int)i);
    struct Placed {
      int32_t k, place;
    };
    std::vector<Placed> by[4];
    for (int64_t s = t * spt; s < (t + 1) * spt; ++s) {
      std::fill_n(H.eidx.begin() + (int64_t)sd[s].x * 64, (int64_t)sd[s].y * 64, kTileZero);
      std::fill_n(H.perm.begin() + (int64_t)sd[s].x * 64, (int64_t)sd[s].y * 64, -1);
      for (int j = 0; j < kSliceRows; ++j) {
        if (H.lrow[s * kSliceRows + j] == 0xffff) continue;
        const int64_t r = c.r0 + H.lrow[s * kSliceRows + j];
        for (auto& b : by) b.clear();
        for (int64_t k = rp[r + 1] - 1; k >= rp[r]; --k) {
          const int place = local[ci[k]];
          by[place & 3].push_back(Placed{(int32_t)k, place});
        }
        for (int64_t e = 0; e < rp[r + 1] - rp[r]; ++e) {
          int cl = (int)((e + j) & 3);
          if (by[cl].empty())
            for (int b = 0; b < 4; ++b)
              if (by[b].size() > by[cl].size()) cl = b;
          const Placed v = by[cl].back();
          by[cl].pop_back();
          const int64_t quad = sd[s].x + e / 4, l = j * 4 + e % 4;
          // the two indices of a pair of quads side by side
          H.eidx[pack == 2 ? quad / 2 * 128 + 2 * l + quad % 2 : quad * 64 + l] = (uint16_t)(v.place + 1);
          H.perm[quad * 64 + l] = v.k;
        }
      }
    }
  });
  return true;
}

// Value slots: MASS3 pairs of quads, [pair][lane][2]; BSR3 [quad], the nine
// values of each lane as 16-byte planes and one plane of the ninth value.
template <class T>
__global__ void tile_values_k(int64_t nslot, int nv, int64_t nbnz, const int32_t* __restrict__ perm,
                              const double* __restrict__ bval, T* __restrict__ out, int flags) {
  constexpr int PW = 16 / (int)sizeof(T);
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nslot; i += (int64_t)gridDim.x * 256) {
    const int32_t k = perm[i];
    const int64_t quad = i >> 6, lane = i & 63;
    if (nv == 1) {
      out[(quad >> 1) * 128 + lane * 2 + (quad & 1)] = k < 0 ? (T)0 : (T)bval[k];
    } else {
      for (int q = 0; q < 9; ++q)
        out[quad * 576 + (q < 8 ? (q / PW) * 64 * PW + lane * PW + q % PW : 512 + lane)] =
            k < 0 ? (T)0 : (T)bval[bidx(k, q, nbnz, flags)];
    }
  }
}

template <class T>
static void write_values(const DevMat& M, const TilePlan& P, T* out, hipStream_t s) {
  const int64_t nslot = P.quads * 64;
  const unsigned grid = (unsigned)std::min<int64_t>(std::max<int64_t>((nslot + 255) / 256, 1), 16384);
  hipLaunchKernelGGL((tile_values_k<T>), dim3(grid), dim3(256), 0, s, nslot, M.layout == L_BSR3 ? 9 : 1, M.nbnz, P.perm,
                     M.bval, out, kflags(M));
  NMG_HIP(hipGetLastError());
}
static size_t value_slots(const DevMat& M, const TilePlan& P) {
  return (size_t)P.quads * 64 * (M.layout == L_BSR3 ? 9 : 1);
}

void refresh_tile_values(DevMat& M, hipStream_t s, bool fp64) {
  for (TileSet& T : M.tset) {
    if (!T.val) continue;
    if (fp64) write_values(M, *T.plan, T.val, s);
    if (!M.bval32) continue;
    float* v = T.val32;
    if (!v) {
      try {
        v = tile_alloc<float>(M, value_slots(M, *T.plan));
      } catch (const Error& e) {
        if (e.code != NMG_ENOMEM) throw;
        continue;  // the FP64 values serve FP32 products too
      }
    }
    write_values(M, *T.plan, v, s);
    if (!T.val32) {
      NMG_HIP(hipStreamSynchronize(s));
      T.val32 = v;
    }
  }
}

void drop_tile_values(DevMat& M) {
  M.touch();
  for (TileSet& T : M.tset) {
    T.use.store(nullptr);
    for (void* p : {(void*)T.val, (void*)T.val32.load()})
      if (p) (void)hipFree(p);
    if (T.val) M.tile_bytes -= (int64_t)(sizeof(double) * value_slots(M, *T.plan));
    if (T.val32) M.tile_bytes -= (int64_t)(sizeof(float) * value_slots(M, *T.plan));
    T.val = nullptr;
    T.val32 = nullptr;
  }
}

void drop_tiles(DevMat& M, int state) {
  drop_tile_values(M);
  for (TileSet& T : M.tset) T.plan.reset();
  M.tile_bytes = 0;
  M.tile_state = state;
}

// Rows of a tile: as few as fill the rounds of 256 tiles, one to a CU, that
// tiles of `most` rows need -- a round begun for a few tiles costs as much as a
// full one (223k DoF, K = 1: 6.9 us with 160 rows, 466 tiles; 9.1 with 144 rows,
// 517 tiles; 56.7k DoF, K = 4: 5.4 us with 80 rows, 237 tiles; 6.1 with 48, 6.5
// with 128).  `most` is what the LDS of two workgroups per CU leaves room for:
// at 24 or 48 bytes a node (K <= 2, FP32 vectors) 224 rows of up to 1400 nodes
// (1.28M DoF, K = 1: 32.4 us, against 34.1 with 192 rows, 42.5 with 128 and 33.0
// with 256), at 96 bytes (K >= 4) 128 rows of up to 700 nodes (K = 4: 64 us,
// against 73 with 192 rows and 67 with 96), or 160 where that leaves two rounds
// (223k DoF, K = 4: 13.5 us against 15.8 with 128); 96 rows for the stiffness
// (439k DoF, K = 1: 62 us against 66 with 128).
static int tile_rows(const DevMat& M, int most) {
  const int64_t round = 256 * std::max<int64_t>(1, (M.nb + 256 * most - 1) / (256 * most));
  return (int)std::min<int64_t>((M.nb + round * kSliceRows - 1) / (round * kSliceRows) * kSliceRows, most);
}

// Scalar masses of few rows take a second plan of twice the rows for K >= 16:
// four workgroups or more share a tile's rows there, one per four columns, and
// half the tiles, with fewer reads of x per row, fill the CUs as well (K = 16:
// 10.6k DoF 8.2 us with 16 rows, 6.1 with 32; 20.1k 9.8 : 7.6; 38.8k 12.4 : 10.7;
// 56.7k 15.2 : 13.5; K = 8 5.1 : 4.6, 5.7 : 5.3, 6.9 : 6.8 and 7.9 : 8.1).
static int deep_rows(const DevMat& M) { return (int)((M.nb + 128 * kSliceRows - 1) / (128 * kSliceRows) * kSliceRows); }
static bool deep_tiles(const DevMat& M) { return M.layout == L_MASS3 && M.nb <= 128 * 160; }

// The smallest node count from which K-column products take the tiles (see
// tile_set), and whether any width can: not with a layout set for each
static int64_t least_rows(const DevMat& M, int K) {
  return M.layout == L_BSR3 ? (K == 1 ? 65536 : 1024) : (K >= 8 ? 1 : 2048);
}
static bool any_width(const DevMat& M) {
  for (int K = 1; K <= 64; K *= 2)
    if (M.nb >= least_rows(M, K) && M.tile_use(K)) return true;
  return false;
}

static void plan_tiles_locked(DevMat& M) {
  if (M.tile_state != TILES_NONE || M.layout == L_CSR || M.nrow != M.ncol ||
      (int64_t)M.h_browptr.size() != M.nb + 1 || !any_width(M))
    return;
  const bool bsr = M.layout == L_BSR3;
  const int rows0 = tile_rows(M, bsr ? 96 : 224);
  const int rows1 = bsr ? rows0 : (deep_tiles(M) ? deep_rows(M) : tile_rows(M, M.nb <= 512 * 160 ? 160 : 128));
  const bool two = rows0 != rows1 || (!bsr && rows0 > 128);
  for (int i = 0; i < (two ? 2 : 1); ++i) {
    HostTiles H;
    const int cap = i == 0 && two && !deep_tiles(M) ? 1400 : 700;
    if (!tile_layout(M.nb, M.h_browptr.data(), M.h_bcol.data(), i == 0 ? rows0 : rows1, cap, bsr ? 8 : 16, bsr ? 1 : 2,
                     H))
      break;
    auto P = std::make_shared<TilePlan>();
    P->ntiles = H.ntiles;
    P->max_nodes = H.max_nodes;
    P->max_extra = H.max_extra;
    P->quads = H.quads;
    P->un = to_device(M, H.un);
    P->tcols = to_device(M, H.tcols);
    P->lrow = to_device(M, H.lrow);
    P->eidx = to_device(M, H.eidx);
    P->perm = to_device(M, H.perm);
    M.tset[i].plan = P;
  }
  M.tile_state = M.tset[0].plan ? TILES_PLANNED : TILES_REFUSED;
}

// The tiles are an option: where their memory does not suffice the matrix keeps
// the row kernels, as for patterns that no tile holds.
template <class F>
static void or_row_kernels(DevMat& M, F&& f) {
  bool ok = false;
  try {
    f();
    ok = true;
  } catch (const std::bad_alloc&) {
  } catch (const Error& e) {
    if (e.code != NMG_ENOMEM) throw;
  }
  if (!ok) drop_tiles(M, TILES_REFUSED);
}

void plan_tiles(DevMat& M) {
  std::lock_guard<std::recursive_mutex> lk(M.mu);
  or_row_kernels(M, [&] { plan_tiles_locked(M); });
}

void build_tiles(DevMat& M, hipStream_t s) {
  std::lock_guard<std::recursive_mutex> lk(M.mu);
  or_row_kernels(M, [&] {
    plan_tiles_locked(M);
    if (M.tile_state != TILES_PLANNED || M.tset[0].val) return;
    for (TileSet& T : M.tset)
      if (T.plan) T.val = tile_alloc<double>(M, value_slots(M, *T.plan));
    M.touch();
    refresh_tile_values(M, s, true);
    NMG_HIP(hipStreamSynchronize(s));
    for (int i = 1; i >= 0; --i)
      if (M.tset[i].plan) M.tset[i].use.store(M.tset[i].plan.get());
  });
}

// The tiles for a K-column product on vectors of `size`-byte values, or null
// for the row kernels: a layout set or tuned explicitly for that width, and
// matrices too small to pay for the list -> x -> LDS chain of a tile (least_rows).
// Measured as the tuner does, tiles : the fastest layout without them, us:
//            stiffness, filter step               scalar mass, Chebyshev step
//   nodes    K = 1        K = 2        K = 4         K = 1      K = 2      K = 4      K = 8
//   458      3.6 : 3.3    4.0 : 3.6    5.0 : 4.3    3.1 : 2.9  3.4 : 3.4  3.9 : 3.5  4.0 : 4.3
//   859      3.7 : 3.3    4.1 : 3.6    5.1 : 4.4    3.3 : 3.0  3.4 : 3.3  4.0 : 3.6  4.1 : 4.3
//   1421     3.7 : 3.4    4.1 : 4.0    5.1 : 5.4    3.2 : 3.4  3.4 : 3.6  4.0 : 3.9  4.1 : 4.8
//   2223     3.8 : 3.9    4.2 : 4.5    5.2 : 6.1    3.3 : 3.6  3.4 : 3.8  4.0 : 4.2  4.7 : 5.3
//   9971     5.0 : 6.1    5.7 : 9.9    7.4 : 14.8   3.6 : 4.4  3.9 : 5.1  4.7 : 7.3  6.4 : 11.0
//   31 016  14.2 : 14.4  14.9 : 23.4  17.2 : 37.8
//   67 539  25.6 : 25.7  28.0 : 44.6  31.6 : 71.1
//   103 363 40.0 : 36.8  43.5 : 66.3  50.6 : 112
//   146 293 64.8 : 73.9  71.5 : 115   81.8 : 180
// (So a single column of stiffness would gain from tiles between some 2 000 and
// 17 000 nodes too; from there to 100 000 neither is ahead throughout.)
static const TileSet* tile_set(const DevMat& M, int K, int size) {
  if (M.layout == L_CSR || !M.tile_use(K)) return nullptr;
  if (M.nb < least_rows(M, K)) return nullptr;
  const int i = M.tset[1].use.load() && (deep_tiles(M) ? K >= 16 : std::min(K, 4) * size > 16) ? 1 : 0;
  return M.tset[i].use.load() ? &M.tset[i] : nullptr;
}

struct TileView {
  const TileUnit* un;
  const int32_t* tcols;
  const uint16_t* lrow;
  const uint16_t* eidx;
};

// element l of p, with the 32-bit byte offset the scalar-base address form takes
template <class T>
__device__ __forceinline__ T* at(T* p, uint32_t l) {
  using C = std::conditional_t<std::is_const_v<T>, const char, char>;
  return reinterpret_cast<T*>(reinterpret_cast<C*>(p) + l * (uint32_t)sizeof(T));
}

// Epilogues on the value at offset o + l of the block vectors (o uniform over
// the wavefront, column c): s is the product there and own the staged x.
struct TEpiStore {
  double* y;
  struct Pre {};
  __device__ __forceinline__ void load(int64_t, uint32_t, int, Pre&) const {}
  __device__ __forceinline__ void store(int64_t o, uint32_t l, int, double s, double, const Pre&) const {
    *at(y + o, l) = s;
  }
};
template <class XT>
struct TEpiCheb {
  const XT* b;
  XT* xm;
  double w, ith;
  struct Pre {
    double b, xm;
  };
  __device__ __forceinline__ void load(int64_t o, uint32_t l, int, Pre& p) const {
    p.b = (double)*at(b + o, l);
    p.xm = (double)*at((const XT*)xm + o, l);
  }
  __device__ __forceinline__ void store(int64_t o, uint32_t l, int, double s, double own, const Pre& p) const {
    *at(xm + o, l) = (XT)(p.xm + w * (own - p.xm + (p.b - s) * ith));
  }
};
struct TEpiFilter {
  const double* vk;
  double* vkm;
  double* y;
  const double* mu;  // per column, or null for mu0
  double mu0, t, cc;
  int first;
  struct Pre {
    double vk, vkm, y;
  };
  __device__ __forceinline__ void load(int64_t o, uint32_t l, int, Pre& p) const {
    p.vk = *at(vk + o, l);
    p.vkm = first ? 0.0 : *at((const double*)vkm + o, l);
    p.y = *at((const double*)y + o, l);
  }
  __device__ __forceinline__ void store(int64_t o, uint32_t l, int c, double s, double, const Pre& p) const {
    const double v = t * (s - cc * p.vk) - p.vkm;
    *at(vkm + o, l) = v;
    *at(y + o, l) = p.y + (mu ? mu[c] : mu0) * v;
  }
};

typedef double d2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void lds_load16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(uintptr_t)g,
                                   (__attribute__((address_space(3))) void*)(uint32_t)(uintptr_t)l, 16, 0, 0);
}

// the values and list places of one lane: a pair of quads (MASS3) or one (BSR3)
template <bool BSR, class VT>
struct Entry;
template <>
struct Entry<false, double> {
  d2 v;
  uint32_t id;
  __device__ __forceinline__ void load(const double* val, const uint16_t* e, int64_t i, int lane) {
    v = *at(reinterpret_cast<const d2*>(val + i * 128), lane);
    id = *at(reinterpret_cast<const uint32_t*>(e + i * 128), lane);
  }
};
template <>
struct Entry<false, float> {
  f2 v;
  uint32_t id;
  __device__ __forceinline__ void load(const float* val, const uint16_t* e, int64_t i, int lane) {
    v = *at(reinterpret_cast<const f2*>(val + i * 128), lane);
    id = *at(reinterpret_cast<const uint32_t*>(e + i * 128), lane);
  }
};
template <>
struct Entry<true, double> {
  d2 w[4];
  double w8;
  int id;
  __device__ __forceinline__ void load(const double* val, const uint16_t* e, int64_t i, int lane) {
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = *at(reinterpret_cast<const d2*>(val + i * 576 + k * 128), lane);
    w8 = *at(val + i * 576 + 512, lane);
    id = *at(e + i * 64, lane);
  }
  __device__ __forceinline__ void get(double* m) const {
#pragma unroll
    for (int k = 0; k < 8; ++k) m[k] = w[k / 2][k % 2];
    m[8] = w8;
  }
};
template <>
struct Entry<true, float> {
  f4 w[2];
  float w8;
  int id;
  __device__ __forceinline__ void load(const float* val, const uint16_t* e, int64_t i, int lane) {
#pragma unroll
    for (int k = 0; k < 2; ++k) w[k] = *at(reinterpret_cast<const f4*>(val + i * 576 + k * 256), lane);
    w8 = *at(val + i * 576 + 512, lane);
    id = *at(e + i * 64, lane);
  }
  __device__ __forceinline__ void get(float* m) const {
#pragma unroll
    for (int k = 0; k < 8; ++k) m[k] = w[k / 4][k % 4];
    m[8] = w8;
  }
};

template <int KG, bool BSR, class VT, class XT, class Epi>
__global__ __launch_bounds__(BSR ? 512 : 1024, BSR ? 4 : 8) void node_tile_k(
    TileView T, const VT* __restrict__ val, const XT* __restrict__ x, int K, int lgroups, int part_off, Epi epi,
    int flags) {
  extern __shared__ double2 tile_lds[];  // a node of zeros (kTileZero), the tile's nodes, partial sums
  char* const xs = reinterpret_cast<char*>(tile_lds);
  double* const partial = reinterpret_cast<double*>(xs + part_off);
  constexpr int NW = BSR ? 8 : 16, TB = 64 * NW;
  constexpr int NV = BSR ? 9 : 1;
  constexpr int QP = BSR ? 1 : 2;            // quads of an Entry
  constexpr int QD = BSR ? 2 : 3;            // entries in flight per lane
  constexpr int SEG = KG * (int)sizeof(XT);  // bytes of one component's columns
  constexpr int NB = 3 * SEG;                // bytes of a node in LDS
  constexpr int UB = SEG >= 16 ? 16 : SEG;   // staged unit
  constexpr int NU = NB / UB, SU = SEG / UB;
  constexpr int SB = NU == 3 ? 3 : 5;        // units per lane and list load
  constexpr int NP = KG == 4 ? 3 : (KG == 2 ? 2 : 1);  // components a lane writes
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qr = lane & 3;
  const int col = KG == 4 ? qr : (KG == 2 ? (qr & 1) : 0);
  auto comp = [&](int p) { return KG == 4 ? p : (KG == 2 ? (qr >> 1) + 2 * p : qr); };
  const int lb = (int)xcd_block(flags);
  const int c0 = (lb & ((1 << lgroups) - 1)) * KG;
  const TileUnit un = T.un[(int64_t)(lb >> lgroups) * NW + wave];

  int lr = 0xffff;  // this lane's row within the tile
  if (un.slice >= 0) lr = (int)T.lrow[(int64_t)un.slice * kSliceRows + (lane >> 2)];
  Entry<BSR, VT> en[QD];
  const int64_t e0 = un.q0 / QP;
  const int ne = un.nq / QP;
#pragma unroll
  for (int u = 0; u < QD; ++u)
    if (u < ne) en[u].load(val, T.eidx, e0 + u, lane);
  char* const xn = xs + NB;
  if (tid < NB / 4) reinterpret_cast<int*>(xs)[tid] = 0;
  // stage x: each wavefront a run of the tile's units, the list read once per
  // SB units and handed to the lanes across the wavefront
  {
    const int total = un.nodes * NU;
    const int per = (total + TB * SB - 1) / (TB * SB) * (64 * SB);
    for (int b0 = wave * per; b0 < (wave + 1) * per && b0 < total; b0 += 64 * SB) {
      const int n0 = b0 / NU;
      const int ln = T.tcols[un.list + min(n0 + lane, un.nodes - 1)];
      uint32_t src[SB];
#pragma unroll
      for (int u = 0; u < SB; ++u) {
        const int t = min(b0 + u * 64 + lane, total - 1);
        const int n = t / NU, part = t - n * NU;
        const int node = __builtin_amdgcn_ds_bpermute((n - n0) * 4, ln);
        src[u] = (uint32_t)(3 * node + part / SU) * (uint32_t)K + (part % SU) * (UB / (int)sizeof(XT));
      }
      if constexpr (UB == 16) {
#pragma unroll
        for (int u = 0; u < SB; ++u)
          if (b0 + u * 64 < total) lds_load16(at(x + c0, src[u]), xn + (size_t)(b0 + u * 64) * 16);
      } else {
        using U = std::conditional_t<UB == 8, double, float>;
        U v[SB];
#pragma unroll
        for (int u = 0; u < SB; ++u) v[u] = *reinterpret_cast<const U*>(at(x + c0, src[u]));
#pragma unroll
        for (int u = 0; u < SB; ++u)
          if (b0 + u * 64 + lane < total) reinterpret_cast<U*>(xn)[b0 + u * 64 + lane] = v[u];
      }
    }
  }
  const int part = un.part & 255, np = (un.part >> 8) & 255, slot = un.part >> 16;
  const int64_t o = 3 * (int64_t)un.row0 * K + c0;
  const uint32_t l0 = (uint32_t)(3 * lr * K + col);
  const bool wr = part == 0 && lr != 0xffff;
  typename Epi::Pre pre[NP];
  if (wr) {
#pragma unroll
    for (int p = 0; p < NP; ++p)
      if (comp(p) < 3) epi.load(o, l0 + comp(p) * K, c0 + col, pre[p]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  double y[3] = {0.0, 0.0, 0.0};
  auto madd = [&](const VT* m, const char* xe) {
    double xv[3];
#pragma unroll
    for (int p = 0; p < 3; ++p) xv[p] = (double)*reinterpret_cast<const XT*>(xe + p * SEG);
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      if constexpr (BSR) {
#pragma unroll
        for (int j = 0; j < 3; ++j) y[p] += (double)m[3 * p + j] * xv[j];
      } else {
        y[p] += (double)m[0] * xv[p];
      }
    }
  };
  const char* const xc = xs + col * (int)sizeof(XT);
  auto step = [&](const VT* m, int id) {
    const int off = id * NB;
    auto one = [&](auto ctrl) {
      constexpr int C = decltype(ctrl)::value;
      VT a[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) a[v] = quad<C>(m[v]);
      madd(a, xc + quad<C>(off));
    };
    if constexpr (KG == 1) {
      madd(m, xc + off);
    } else if constexpr (KG == 2) {
      one(std::integral_constant<int, 0x50>{});
      one(std::integral_constant<int, 0xfa>{});
    } else {
      one(std::integral_constant<int, 0x00>{});
      one(std::integral_constant<int, 0x55>{});
      one(std::integral_constant<int, 0xaa>{});
      one(std::integral_constant<int, 0xff>{});
    }
  };
  // the sums of one quad before the reads of the next: left alone the compiler
  // gathers several quads' reads first and spills
  auto keep = [&] { asm volatile("" : "+v"(y[0]), "+v"(y[1]), "+v"(y[2])); };
  for (int q = 0; q < ne; q += QD) {
#pragma unroll
    for (int u = 0; u < QD; ++u)
      if (q + u < ne) {
        if constexpr (BSR) {
          VT m[9];
          en[u].get(m);
          step(m, en[u].id);
          keep();
        } else {
          const VT m0 = en[u].v[0], m1 = en[u].v[1];
          step(&m0, (int)(en[u].id & 0xffff));
          keep();
          step(&m1, (int)(en[u].id >> 16));
          keep();
        }
        if (q + QD + u < ne) en[u].load(val, T.eidx, e0 + q + QD + u, lane);
      }
  }
  if constexpr (KG == 1) {
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      y[p] += quad<0xb1>(y[p]);
      y[p] += quad<0x4e>(y[p]);
    }
  } else if constexpr (KG == 2) {
#pragma unroll
    for (int p = 0; p < 3; ++p) y[p] += quad<0x4e>(y[p]);
  }
  double sum[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) sum[p] = comp(p) == 0 ? y[0] : (comp(p) == 1 ? y[1] : y[2]);
  if (part_off > 0) {  // some slice of the matrix is split
    if (part > 0) {
#pragma unroll
      for (int p = 0; p < NP; ++p) partial[((slot + part - 1) * NP + p) * 64 + lane] = sum[p];
    }
    __syncthreads();
    if (part == 0)
      for (int i = 0; i < np - 1; ++i)
#pragma unroll
        for (int p = 0; p < NP; ++p) sum[p] += partial[((slot + i) * NP + p) * 64 + lane];
  }
  if (wr) {
#pragma unroll
    for (int p = 0; p < NP; ++p)
      if (comp(p) < 3) {
        const double own = (double)*reinterpret_cast<const XT*>(xc + (un.own + lr + 1) * NB + comp(p) * SEG);
        epi.store(o, l0 + comp(p) * K, c0 + col, sum[p], own, pre[p]);
      }
  }
}

template <int KG, bool BSR, class VT, class XT, class Epi>
static void launch_tile(const DevMat& M, const TilePlan& P, const VT* v, const XT* x, int K, Epi epi, hipStream_t s) {
  int lg = 0;
  while ((KG << lg) < K) ++lg;
  const TileView T{P.un, P.tcols, P.lrow, P.eidx};
  constexpr int NP = KG == 4 ? 3 : (KG == 2 ? 2 : 1);
  // the node of zeros, then the nodes, staged in whole wavefronts of 16 bytes a lane
  size_t lds = 3 * KG * sizeof(XT) + ((size_t)P.max_nodes * 3 * KG * sizeof(XT) + 1023) / 1024 * 1024;
  lds = (lds + 15) / 16 * 16;
  int part_off = 0;  // no slice is split
  if (P.max_extra > 0) {
    part_off = (int)lds;
    lds += (size_t)P.max_extra * 64 * NP * sizeof(double);
  }
  hipLaunchKernelGGL((node_tile_k<KG, BSR, VT, XT, Epi>), dim3((unsigned)(P.ntiles << lg)), dim3(BSR ? 512 : 1024),
                     lds, s, T, v, x, K, lg, part_off, epi, kflags(M));
  NMG_HIP(hipGetLastError());
}

int tile_route(const DevMat& M, int K, int size) {
  const TileSet* T = tile_set(M, K, size);
  return T ? 1 + (int)(T - M.tset) : 0;
}
bool tiles_taken(const DevMat& M, int K) { return tile_route(M, K, 8) > 0; }

template <bool BSR, class XT, class Epi>
static bool tile_product(const DevMat& M, const XT* x, int K, Epi epi, hipStream_t s, bool fp32,
                         std::initializer_list<const void*> others) {
  if (M.layout != (BSR ? L_BSR3 : L_MASS3)) return false;
  const TileSet* T = tile_set(M, K, sizeof(XT));
  if (!T) return false;
  // 32-bit offsets into x, and 16-byte loads (8 at K = 2 in FP32) of its columns
  if ((uint64_t)M.nrow * K * sizeof(XT) >= (uint64_t)1 << 32) return false;
  uintptr_t a = (uintptr_t)x;
  for (const void* p : others) a |= (uintptr_t)p;
  if (a % std::min<size_t>(16, std::min(K, 4) * sizeof(XT))) return false;
  auto go = [&](auto* v) {
    if (K == 1) launch_tile<1, BSR>(M, *T->plan, v, x, K, epi, s);
    else if (K == 2) launch_tile<2, BSR>(M, *T->plan, v, x, K, epi, s);
    else launch_tile<4, BSR>(M, *T->plan, v, x, K, epi, s);
  };
  const float* v32 = fp32 ? T->val32.load() : nullptr;
  if (v32) go(v32);
  else go((const double*)T->val);
  return true;
}

bool k_tile_spmv(int K, const DevMat& M, const double* x, double* y, hipStream_t s, bool fp32) {
  return tile_product<false>(M, x, K, TEpiStore{y}, s, fp32, {y}) ||
         tile_product<true>(M, x, K, TEpiStore{y}, s, fp32, {y});
}
bool k_tile_cheb_step(int K, const DevMat& M, const double* b, const double* xk, double* xm, double w, double ith,
                      hipStream_t s, bool fp32) {
  return tile_product<false>(M, xk, K, TEpiCheb<double>{b, xm, w, ith}, s, fp32, {b, xm});
}
bool k_tile_cheb_step32(int K, const DevMat& M, const float* b, const float* xk, float* xm, double w, double ith,
                        hipStream_t s, bool fp32) {
  return tile_product<false>(M, xk, K, TEpiCheb<float>{b, xm, w, ith}, s, fp32, {b, xm});
}
bool k_tile_filter_step(int K, const DevMat& A, const double* x, const double* vk, double* vkm, double* y,
                        const double* mu, double mu0, double t, double cc, bool first, hipStream_t s, bool fp32) {
  return tile_product<true>(A, x, K, TEpiFilter{vk, vkm, y, mu, mu0, t, cc, first ? 1 : 0}, s, fp32, {vk, vkm, y});
}

}  // namespace nmg
