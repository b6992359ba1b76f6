// Whole Chebyshev solves of small scalar-mass systems in one launch.
//
// Below some 800 (P2) to 1400 (P1) nodes a fused step is nothing but its
// launch: 2.9-3.9 us for 0.1-0.2 us of work.  M (x) I3 does not couple the
// three components, so one workgroup takes one component of one column through
// all steps by itself: two iterates in LDS (16 bytes per node), the
// matrix in registers (2.5 per slot), one workgroup barrier per step and no
// communication between workgroups.
//
// The rows are sorted by length and cut into slices of 16 with four lanes per
// row (long rows: four with 16 lanes), as in nmgpu_tiles.hip; the slices go to
// the 16 wavefronts longest first, each to the least loaded.  A step reads x for
// all of a wavefront's quads eight at a time, adds up each slice, closes it with
// two DPP additions and updates its rows.  For the LDS gather (8 bytes per entry,
// one CU) the entries of four neighbouring rows are ordered on the host such that
// the 16 lanes read together touch different banks where possible.
//
// Measured, us per step of a 60-step solve (one launch per step in brackets):
// 115 P2 nodes 0.46 (2.9), 614 P1 nodes 0.91 (2.9), 556 P2 nodes 1.26 (3.2), 1002
// P1 nodes 1.13 (2.9).  Instruction issue bounds it (about 100 per wavefront
// and step at 614 nodes).  Reading each slice's rows and iterates from LDS at
// its end took 1.06 us at 614 nodes; 32 quads per wavefront spill (2.7 us).
#include <algorithm>
#include <memory>
#include <numeric>
#include <vector>

#include "nmgpu_device.h"
#include "nmgpu_internal.h"

namespace nmg {

constexpr int kSmallWaves = 16;
constexpr int kSmallQuads = 24;  // quads per wavefront that the registers hold
constexpr int kSmallWeights = 8192;  // step weights held; longer solves repeat the last

SmallPlan::~SmallPlan() {
  for (void* p : {(void*)ends, (void*)rows, (void*)eidx, (void*)perm})
    if (p) (void)hipFree(p);
}

bool small_layout(int64_t nb, const int64_t* rp, const int32_t* ci, HostSmall& H) {
  if (nb < 1 || nb > 4096 || rp[nb] > kSmallQuads * kSmallWaves * 64) return false;
  std::vector<int32_t> ord(nb);
  std::iota(ord.begin(), ord.end(), 0);
  auto len = [&](int32_t r) { return rp[r + 1] - rp[r]; };
  std::stable_sort(ord.begin(), ord.end(), [&](int32_t a, int32_t b) { return len(a) > len(b); });
  // slices of 16 rows with four lanes each; rows of more than 32 entries (the
  // vertices of P2 meshes) four to a slice with 16 lanes each
  struct Slice {
    int64_t first;
    int rows, lanes, quads;
  };
  std::vector<Slice> sl;
  for (int64_t r = 0; r < nb;) {
    const int lanes = len(ord[r]) > 32 ? 16 : 4, most = 64 / lanes;
    int n = 0;
    while (n < most && r + n < nb && (lanes == 4 || len(ord[r + n]) > 32)) ++n;
    sl.push_back({r, n, lanes, (int)std::max<int64_t>(1, (len(ord[r]) + lanes - 1) / lanes)});
    r += n;
  }
  std::stable_sort(sl.begin(), sl.end(), [](const Slice& a, const Slice& b) { return a.quads > b.quads; });
  std::vector<int> load(kSmallWaves, 0);
  std::vector<std::vector<Slice>> mine(kSmallWaves);
  for (const Slice& s : sl) {
    const int w = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    load[w] += s.quads;
    mine[w].push_back(s);
  }
  const int most = *std::max_element(load.begin(), load.end());
  H.slices = 0;
  for (auto& m : mine) H.slices = std::max(H.slices, (int)m.size());
  if (most > kSmallQuads || H.slices > 16) return false;
  H.quads = (most + 7) / 8 * 8;
  H.ends.assign(2 * kSmallWaves, 0);
  H.rows.assign((size_t)kSmallWaves * H.slices * kSliceRows, 0xffff);
  // padding points at the zero behind each iterate: 0 * x of any node would carry
  // an infinity or NaN into rows that do not touch it
  H.eidx.assign((size_t)kSmallWaves * H.quads * 64, (uint16_t)nb);
  H.perm.assign((size_t)kSmallWaves * H.quads * 64, -1);
  for (int w = 0; w < kSmallWaves; ++w) {
    int q0 = 0;
    for (size_t i = 0; i < mine[w].size(); ++i) {
      const Slice& s = mine[w][i];
      const int together = 16 / s.lanes;  // rows in the 16 lanes of one LDS pass
      for (int g = 0; g < s.rows; g += together) {
        std::vector<std::vector<int64_t>> left(together);
        for (int j = 0; j < together && g + j < s.rows; ++j) {
          const int32_t r = ord[s.first + g + j];
          H.rows[((size_t)w * H.slices + i) * kSliceRows + (g + j) * s.lanes / 4] = (uint16_t)r;
          for (int64_t k = rp[r]; k < rp[r + 1]; ++k) left[j].push_back(k);
        }
        for (int q = 0; q < s.quads; ++q) {
          uint32_t used = 0;  // banks (8-byte columns) taken in this pass
          for (int e = 0; e < s.lanes; ++e)
            for (int j = 0; j < together; ++j) {
              if (left[j].empty()) continue;
              size_t pick = 0;
              for (size_t c = 0; c < left[j].size(); ++c)
                if (!(used >> (ci[left[j][c]] & 15) & 1)) {
                  pick = c;
                  break;
                }
              const int64_t k = left[j][pick];
              left[j].erase(left[j].begin() + (int64_t)pick);
              used |= 1u << (ci[k] & 15);
              const size_t slot = ((size_t)w * H.quads + q0 + q) * 64 + s.lanes * (g + j) + e;
              H.eidx[slot] = (uint16_t)ci[k];
              H.perm[slot] = (int32_t)k;
            }
        }
      }
      q0 += s.quads;
      H.ends[w] |= 1u << (q0 - 1);
      if (s.lanes == 16) H.ends[kSmallWaves + w] |= 1u << (q0 - 1);
    }
  }
  return true;
}

template <class T>
static T* upload(const std::vector<T>& v) {
  T* p = nullptr;
  NMG_HIP(hipMalloc(&p, sizeof(T) * std::max<size_t>(v.size(), 1)));
  const hipError_t e = hipMemcpy(p, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    (void)hipFree(p);
    NMG_HIP(e);
  }
  return p;
}

void build_small(DevMat& M) {
  std::lock_guard<std::recursive_mutex> lk(M.mu);
  if (M.small || M.layout != L_MASS3 || M.nrow != M.ncol || (int64_t)M.h_browptr.size() != M.nb + 1) return;
  HostSmall H;
  if (!small_layout(M.nb, M.h_browptr.data(), M.h_bcol.data(), H)) return;
  auto P = std::make_shared<SmallPlan>();
  P->quads = H.quads;
  P->slices = H.slices;
  P->ends = upload(H.ends);
  P->rows = upload(H.rows);
  P->eidx = upload(H.eidx);
  P->perm = upload(H.perm);
  M.small = P;
}

SmallWeights::~SmallWeights() {
  if (w) (void)hipFree(w);
}

// The weights live with the matrix, not with the solve: a graph that captured a
// solve then holds buffers of its matrix only.  (In the kernel arguments they
// cost 1.7 us of a 30 us solve; computed in the kernel from w_k = 2 s T_k(s) /
// T_{k+1}(s) they cost nothing, but their rounding, other than the step kernels',
// made a filtered Lanczos run whose residuals end just below its target stop
// with eigenvalues that agree to 4e-12 instead of 1e-13.)
const double* small_weights(DevMat& M, double lmin, double lmax, int deg) {
  constexpr size_t kMost = 64;  // bounds and degrees of one matrix; further solves run step by step
  std::lock_guard<std::recursive_mutex> lk(M.mu);
  if (!M.small) return nullptr;
  for (const auto& W : M.small_w)
    if (W->lmin == lmin && W->lmax == lmax && W->deg == deg) return W->w;
  if (M.small_w.size() >= kMost) return nullptr;
  std::vector<double> w(deg);
  const double sg = (lmax + lmin) / (lmax - lmin);
  double wk = 2.0;
  for (int k = 0; k < deg; ++k) w[k] = wk = 1.0 / (1.0 - wk / (4.0 * sg * sg));
  for (int k = kSmallWeights; k < deg; ++k)
    if (w[k] != w[kSmallWeights - 1]) return nullptr;  // not settled by then: step by step
  w.resize(std::min(deg, kSmallWeights));
  auto W = std::make_unique<SmallWeights>();
  W->lmin = lmin;
  W->lmax = lmax;
  W->deg = deg;
  W->w = upload(w);
  M.small_w.push_back(std::move(W));
  return M.small_w.back()->w;
}

struct SmallView {
  const uint32_t* ends;
  const uint16_t* rows;
  const uint16_t* eidx;
  const int32_t* perm;
  int slices;
};

// Slice sl of a wavefront belongs to the lanes with (lane & 3) == sl & 3: after
// a row's four lanes have its sum, that one keeps it, so the update of up to
// four slices runs once, on all 64 lanes, with b and both iterates of a lane's
// own rows in registers (NS rows for up to 4 NS slices).
template <int QW, int NS, class VT>
__global__ __launch_bounds__(64 * kSmallWaves) void cheb_small_k(SmallView P, const VT* __restrict__ val, int nb, int K,
                                                                 int deg, double ith, const double* __restrict__ wts,
                                                                 const double* __restrict__ b,
                                                                 double* __restrict__ out) {
  // two iterates of nb values and a zero each, then the step weights
  extern __shared__ double small_lds[];
  const int ld = nb + 1;
  char* const xs = reinterpret_cast<char*>(small_lds);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t o = (int64_t)(blockIdx.x % 3) * K + blockIdx.x / 3;  // component, column
  for (int i = tid; i < nb; i += 64 * kSmallWaves) small_lds[i] = b[3 * (int64_t)i * K + o] * ith;
  if (tid < 2) small_lds[tid * ld + nb] = 0.0;
  const uint32_t ends = P.ends[wave], wide = P.ends[kSmallWaves + wave];
  VT v[QW];
  uint32_t id[QW / 2];  // two byte offsets of x
#pragma unroll
  for (int q = 0; q < QW; ++q) {
    const int64_t s = ((int64_t)wave * QW + q) * 64 + lane;
    const int32_t k = P.perm[s];
    v[q] = k < 0 ? (VT)0 : val[k];
    const uint32_t e = (uint32_t)P.eidx[s] * 8;
    id[q / 2] = q % 2 ? id[q / 2] | e << 16 : e;
  }
  int row[NS];
  double bo[NS], xo[NS], mo[NS];
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const int sl = 4 * j + (lane & 3);
    const int r = sl < P.slices ? P.rows[((int64_t)wave * P.slices + sl) * kSliceRows + (lane >> 2)] : 0xffff;
    row[j] = r == 0xffff ? -1 : r;
    bo[j] = row[j] >= 0 ? b[3 * (int64_t)row[j] * K + o] : 0.0;
    xo[j] = bo[j] * ith;
    mo[j] = 0.0;
  }
  // step weights in LDS: a global load per step costs more than the step
  double* const ws = small_lds + 2 * ld;
  for (int i = tid; i < min(deg, kSmallWeights); i += 64 * kSmallWaves) ws[i] = wts[i];
  __syncthreads();
  for (int k = 0; k < deg; ++k) {
    const double w = ws[min(k, kSmallWeights - 1)];
    const uint32_t from = k & 1 ? (uint32_t)ld * 8 : 0;
    double s = 0.0, kept[NS];
    int sl = 0;
#pragma unroll
    for (int j = 0; j < NS; ++j) kept[j] = 0.0;
#pragma unroll
    for (int q0 = 0; q0 < QW; q0 += 8) {
      double xv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        xv[u] = *reinterpret_cast<const double*>(
            xs + from + ((q0 + u) % 2 ? id[(q0 + u) / 2] >> 16 : id[(q0 + u) / 2] & 0xffff));
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        s += (double)v[q0 + u] * xv[u];
        if (ends >> (q0 + u) & 1) {  // uniform over the wavefront: the slice ends here
          s += quad<0xb1>(s);
          s += quad<0x4e>(s);
          if (wide >> (q0 + u) & 1) {  // 16 lanes per row
            s += quad<0x141>(s);
            s += quad<0x140>(s);
          }
          const bool mine = (lane & 3) == (sl & 3);
#pragma unroll
          for (int j = 0; j < NS; ++j)
            if (NS == 1 || sl >> 2 == j) kept[j] = mine ? s : kept[j];
          s = 0.0;
          ++sl;
        }
      }
    }
    char* const to = xs + ((uint32_t)ld * 8 - from);
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const double x = mo[j] + w * (xo[j] - mo[j] + (bo[j] - kept[j]) * ith);
      mo[j] = xo[j];
      xo[j] = x;
      if (row[j] >= 0) reinterpret_cast<double*>(to)[row[j]] = x;
    }
    __syncthreads();
  }
  const double* const x = small_lds + (deg & 1 ? ld : 0);
  for (int i = tid; i < nb; i += 64 * kSmallWaves) out[3 * (int64_t)i * K + o] = x[i];
}

template <int QW, class VT>
static void launch_small_q(const SmallPlan& P, const VT* val, int nb, int K, int deg, double ith, const double* wts,
                           const double* b, double* out, hipStream_t s) {
  const SmallView V{P.ends, P.rows, P.eidx, P.perm, P.slices};
  const size_t lds = (size_t)(nb + 1) * 16 + (size_t)std::min(deg, kSmallWeights) * 8;
  const dim3 grid(3 * (unsigned)K), tb(64 * kSmallWaves);
  if (P.slices <= 4)
    hipLaunchKernelGGL((cheb_small_k<QW, 1, VT>), grid, tb, lds, s, V, val, nb, K, deg, ith, wts, b, out);
  else if (P.slices <= 8)
    hipLaunchKernelGGL((cheb_small_k<QW, 2, VT>), grid, tb, lds, s, V, val, nb, K, deg, ith, wts, b, out);
  else
    hipLaunchKernelGGL((cheb_small_k<QW, 4, VT>), grid, tb, lds, s, V, val, nb, K, deg, ith, wts, b, out);
  NMG_HIP(hipGetLastError());
}

template <class VT>
static void launch_small(const SmallPlan& P, const VT* val, int nb, int K, int deg, double ith, const double* wts,
                         const double* b, double* out, hipStream_t s) {
  switch (P.quads) {
    case 8: launch_small_q<8>(P, val, nb, K, deg, ith, wts, b, out, s); break;
    case 16: launch_small_q<16>(P, val, nb, K, deg, ith, wts, b, out, s); break;
    default: launch_small_q<24>(P, val, nb, K, deg, ith, wts, b, out, s); break;
  }
}

void k_cheb_small(const DevMat& M, int K, int deg, double ith, const double* wts, const double* b, double* out,
                  hipStream_t s, bool fp32) {
  const SmallPlan& P = *M.small;
  if (fp32 && M.bval32) launch_small(P, (const float*)M.bval32, (int)M.nb, K, deg, ith, wts, b, out, s);
  else launch_small(P, (const double*)M.bval, (int)M.nb, K, deg, ith, wts, b, out, s);
}

}  // namespace nmg
