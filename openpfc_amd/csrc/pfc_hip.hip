// pfc_hip.hip -- C-ABI implementation: plans, twiddle tables, size dispatch
// and the launch sequences of the R2C/C2R transforms and the fused PFC step.
#include "../../include/pfc_hip.h"
#include "adjoint_kernels.hpp"
#include "energy_kernels.hpp"
#include "plane.hpp"
#include "variants.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <iterator>
#include <new>
#include <string>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>
#include <vector>

using namespace pfc_amd;


namespace pfc_amd {
// message of the last failed ABI call on this thread (field_io.hip sets it too)
thread_local std::string g_last_error;

// Scratch of pfc_hip_column_max_noalloc: the partial maxima of up to 256
// rows of nx <= 2048 columns (4 MiB), one copy per GPU for the life of the
// process.  Its name is a host-side stand-in for the device array, so host
// code uses only the address col_scratch() obtains on each device.
constexpr long kColScratchDoubles = 256L * 2048;
__device__ __align__(256) double scratch[kColScratchDoubles];
} // namespace pfc_amd

namespace {

using pfc_amd::g_last_error;

int fail(int code, const std::string &msg) {
  g_last_error = msg;
  return code;
}

#define PFC_HIP_TRY(expr, what)                                                \
  do {                                                                         \
    hipError_t e_ = (expr);                                                    \
    if (e_ != hipSuccess)                                                      \
      return fail(PFC_HIP_EDEVICE,                                             \
                  std::string(what) + ": " + hipGetErrorString(e_));           \
  } while (0)

// ---------------------------------------------------------------------------
// Host twiddle tables (long double, rounded once).
// ---------------------------------------------------------------------------
const long double kTwoPi = 6.283185307179586476925286766559005768L;

void unit_root_ld(long m, long n, long double &c, long double &s) {
  m %= n;
  if (m < 0) m += n;
  // exact values on the axes
  if (m == 0) { c = 1; s = 0; return; }
  if (2 * m == n) { c = -1; s = 0; return; }
  if (4 * m == n) { c = 0; s = 1; return; }
  if (4 * m == 3 * n) { c = 0; s = -1; return; }
  long double a = kTwoPi * (long double)m / (long double)n;
  c = cosl(a);
  s = sinl(a);
}

// Line twiddles for the Stockham passes of plan `pid`: exp(-2 pi i q k/(Ns R)).
std::vector<long double> line_twiddles(int n, int pid) {
  std::vector<long double> out; // re, im pairs
  int ns = 1;
  for (int r : radices_for(n, pid)) {
    if (ns > 1) {
      for (int k = 0; k < ns; ++k)
        for (int q = 1; q < r; ++q) {
          long double c, s;
          unit_root_ld((long)q * k, (long)ns * r, c, s);
          out.push_back(c);
          out.push_back(-s);
        }
    }
    ns *= r;
  }
  return out;
}

// exp(-2 pi i k/nx), k = 0..nx/2.
std::vector<long double> real_twiddles(int nx) {
  std::vector<long double> out;
  for (int k = 0; k <= nx / 2; ++k) {
    long double c, s;
    unit_root_ld(k, nx, c, s);
    out.push_back(c);
    out.push_back(-s);
  }
  return out;
}

} // namespace

// ---------------------------------------------------------------------------
// Plan object.
// ---------------------------------------------------------------------------
struct pfc_hip_plan_s {
  int nx = 0, ny = 0, nz = 0, prec = 0, flags = 0;
  int W = 0;        // nx/2 + 1
  int P = 0;        // padded pitch of the plan's own spectrum buffers
  size_t esize = 8; // sizeof(real)
  int device = 0;
  // line twiddles per (length, plan id) and real-FFT twiddles of nx
  std::map<std::pair<int, int>, void *> tw;
  void *wn = nullptr;
  void *work = nullptr; // c2r workspace: W*ny*nz complex
  // fused-step state: natural layout (A, B pitched by P) or transposed
  // layouts T1 (A1, B1) and T2 (A2, B2), W*ny*nz complex each
  void *A = nullptr, *B = nullptr;
  void *C = nullptr; // natural layout with plane kernels: Psi between x/y and z
  void *A1 = nullptr, *B1 = nullptr, *A2 = nullptr, *B2 = nullptr;
  // adjoint workspace: three spectra (of pitch P at most), two real fields, block partials
  void *adj_lam = nullptr, *adj_P = nullptr, *adj_N = nullptr;
  void *adj_a = nullptr, *adj_b = nullptr, *adj_part = nullptr;
  void *adj_zpart = nullptr; // block partials of the fused z pass
  // column maxima (MovingBC): kColParts partial rows of nx, then the result
  void *colmax = nullptr;
  // exp(-2 pi i k/nx) in double for the C2R merge of FP64-butterfly plans
  void *wn64 = nullptr;
  // plane kernels: column and row twiddles and exp(-2 pi i k/nx) in double, within
  // the tables of tw and wn
  const void *plane_tw[2] = {}, *plane_wn = nullptr;
  bool ops_ready = false;
  int model_kind = -1;
  double dt = 0;
  PfcOp op{};    // k-grid, dt, 1/(nx ny nz); eps of the PFC model
  double spacing[3] = {}; // dx, dy, dz of the operators
  TungOp top{};  // Tungsten operator scalars
  double tq[5] = {}; // Tungsten nonlinearity: p3_bar, p4_bar, q3_bar, q4_bar, stabP
  bool mean_split = false; // field holds psi - mean; mean kept in double here
  double mean = 0.0;
  int var[ROLE_COUNT] = {};
  bool chosen[ROLE_COUNT] = {}; // roles set by a caller or the autotuner
  size_t bytes = 0;
  // Batched plans step `batch` fields of these extents stored one after
  // another.  The natural layout steps them all in each launch, reading
  // per-field eps and (3m, 3m^2) from m_eps (double) and m_nl (real type)
  // once `members` is set; the transposed layout steps them one after
  // another (every pass of field 0, then of field 1, ...: a field's spectra
  // stay in the last-level cache between its passes), through one set of
  // T1/T2 buffers, with each field's eps and mean (h_eps, h_mean) as launch
  // arguments.
  int batch = 1;
  void *m_eps = nullptr, *m_nl = nullptr;
  bool members = false;
  std::vector<double> h_eps, h_mean;
  // Bumped by every call that changes a value the step's kernels receive as
  // a launch argument (operators, eps or mean held as scalars, the
  // mean-split mode, variants): a graph captured before such a change
  // replays stale arguments and must be captured again.
  unsigned gen = 0;

  size_t inbox() const { return (size_t)nx * ny * nz; }
  size_t outbox() const { return (size_t)W * ny * nz; }
  size_t padded() const { return (size_t)P * ny * nz; }
  int role_len(int role) const {
    switch (role) {
    case ROLE_X_R2C: case ROLE_X_C2R: return nx / 2;
    case ROLE_COL_Y: return ny;
    case ROLE_COL_Z: case ROLE_PFC_Z: return nz;
    case ROLE_PFC_X: return nx;
    case ROLE_T_X_FWD: return nx;
    case ROLE_T_Y_FWD: case ROLE_T_Y_INV: return ny;
    case ROLE_T_Z: return nz;
    case ROLE_T_X_INV: return nx / 2;
    case ROLE_X_TUNG: case ROLE_T_X_R2C: case ROLE_T_X_TUNG: return nx / 2;
    case ROLE_T_X_FUSE: return nx / 2;
    default: return 0;
    }
  }
  bool transposed() const { return var[ROLE_STEP_LAYOUT] == 0 && t_ok; }
  bool tungsten() const { return model_kind == PFC_HIP_MODEL_TUNGSTEN; }
  int step_passes() const { return tungsten() ? 9 : 5; }
  bool t_ok = false; // transposed step supported for these extents
  // PFC_HIP_FLAG_F64_BUTTERFLIES: single-precision fields whose transposed
  // PFC passes run their butterflies in double (t_variants_xp lists)
  bool xp = false;
  // the plane kernels take these extents (plane_kernels.hpp)
  size_t plane_bytes() const {
    return xp ? 0 : prec == PFC_HIP_F64 ? plane_lds<double>(nx, ny) : plane_lds<float>(nx, ny);
  }
  bool plane_ok() const { return plane_bytes() > 0; }
};

namespace {

int dalloc(pfc_hip_plan_s *p, void **ptr, size_t bytes, const char *what) {
  if (*ptr) return 0;
  hipError_t e = hipMalloc(ptr, bytes ? bytes : 16);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    *ptr = nullptr;
    return fail(PFC_HIP_ENOMEM, std::string("hipMalloc(") + what + ", " +
                                    std::to_string(bytes) +
                                    " bytes): " + hipGetErrorString(e));
  }
  p->bytes += bytes ? bytes : 16;
  return 0;
}

int upload_table(pfc_hip_plan_s *p, void **dst, const std::vector<long double> &v,
                 const char *what) {
  const size_t n = v.size();
  const size_t bytes = n * p->esize;
  if (int rc = dalloc(p, dst, bytes, what)) return rc;
  if (n == 0) return 0;
  if (p->prec == PFC_HIP_F64) {
    std::vector<double> h(n);
    for (size_t i = 0; i < n; ++i) h[i] = (double)v[i];
    PFC_HIP_TRY(hipMemcpy(*dst, h.data(), bytes, hipMemcpyHostToDevice), what);
  } else {
    std::vector<float> h(n);
    for (size_t i = 0; i < n; ++i) h[i] = (float)v[i];
    PFC_HIP_TRY(hipMemcpy(*dst, h.data(), bytes, hipMemcpyHostToDevice), what);
  }
  return 0;
}

// Twiddles of every plan of length n.
int upload_line_tables(pfc_hip_plan_s *p, int n) {
  for (int pid = 0; pid < plan_count(n); ++pid) {
    auto key = std::make_pair(n, pid);
    if (p->tw.count(key)) continue;
    // into the plan's slot, which is freed with the plan if the upload fails
    if (int rc = upload_table(p, &p->tw[key], line_twiddles(n, pid), "line twiddles")) return rc;
  }
  return 0;
}

// exp(-2 pi i k/nx) in double.
int upload_wn64(pfc_hip_plan_s *p) {
  const std::vector<long double> w = real_twiddles(p->nx);
  if (int rc = dalloc(p, &p->wn64, w.size() * sizeof(double), "real twiddles (double)")) return rc;
  std::vector<double> h(w.begin(), w.end());
  PFC_HIP_TRY(hipMemcpy(p->wn64, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice),
              "real twiddles (double)");
  return 0;
}

// Real-FFT twiddles of nx and, with `plane`, what the plane kernels take beside
// them: twiddles of their column (ny) and row (nx/2) plans, where no line plan of
// the same radices has them already, and in single precision the real-FFT twiddles
// in double.  One copy in all, as without the plane kernels: with one for each table
// a 32^3 FP64 stepper took 427 us to make against 339, and an ensemble of seven plans
// 3.05 ms against 2.56 (now within 10 %, and 2.82 ms with its buffers C).
int upload_real_tables(pfc_hip_plan_s *p, bool plane) {
  const bool f64 = p->prec == PFC_HIP_F64;
  std::vector<unsigned char> bytes;
  auto append = [&](const std::vector<long double> &w, bool dbl) { // at a multiple of 16 bytes
    const size_t at = bytes.size();
    auto put = [&](const auto &v) {
      const auto *c = reinterpret_cast<const unsigned char *>(v.data());
      bytes.insert(bytes.end(), c, c + v.size() * sizeof(v[0]));
    };
    if (dbl)
      put(std::vector<double>(w.begin(), w.end()));
    else
      put(std::vector<float>(w.begin(), w.end()));
    bytes.resize((bytes.size() + 15) / 16 * 16);
    return at;
  };
  const std::vector<long double> wn = real_twiddles(p->nx);
  append(wn, f64);
  size_t at[2] = {0, 0}, at_wn = 0;
  for (int row = 0; row < 2 && plane; ++row) {
    const int n = row ? p->nx / 2 : p->ny;
    const int pid = f64 ? plane_pid<double>(row) : plane_pid<float>(row);
    const std::vector<int> radices = radices_for(n, pid);
    for (int i = 0; i < plan_count(n) && !p->plane_tw[row]; ++i)
      if (radices_for(n, i) == radices) p->plane_tw[row] = p->tw.at({n, i});
    if (!p->plane_tw[row]) at[row] = append(line_twiddles(n, pid), f64);
  }
  if (plane && !f64) at_wn = append(wn, true);
  if (int rc = dalloc(p, &p->wn, bytes.size(), "real twiddles")) return rc;
  PFC_HIP_TRY(hipMemcpy(p->wn, bytes.data(), bytes.size(), hipMemcpyHostToDevice),
              "real twiddles");
  const unsigned char *base = (const unsigned char *)p->wn;
  for (int row = 0; row < 2; ++row)
    if (at[row]) p->plane_tw[row] = base + at[row];
  p->plane_wn = base + at_wn;
  return 0;
}

// Twiddles of the double-butterfly plans of length n: double entries at
// plan ids kXpPid + i, whatever the plan's precision.
int upload_line_tables_xp(pfc_hip_plan_s *p, int n) {
  for (int i = 0; i < plan_count_xp(n); ++i) {
    const int pid = kXpPid + i;
    auto key = std::make_pair(n, pid);
    if (p->tw.count(key)) continue;
    const std::vector<long double> v = line_twiddles(n, pid);
    void *d = nullptr;
    if (int rc = dalloc(p, &d, v.size() * sizeof(double), "line twiddles (double)")) return rc;
    p->tw[key] = d;
    if (!v.empty()) {
      std::vector<double> h(v.begin(), v.end());
      PFC_HIP_TRY(hipMemcpy(d, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice),
                  "line twiddles (double)");
    }
  }
  return 0;
}

template <typename T> const cplx<T> *twp(pfc_hip_plan_s *p, int n, int pid) {
  auto it = p->tw.find(std::make_pair(n, pid));
  return it == p->tw.end() ? nullptr : (const cplx<T> *)it->second;
}

template <typename T> TungNl<T> tung_nonlin(const pfc_hip_plan_s *p) {
  return TungNl<T>{(T)p->tq[0], (T)p->tq[1], (T)p->tq[2], (T)p->tq[3], (T)p->tq[4]};
}

// Transposed-step kernel kind of a role, or -1.
int t_kind_of_role(int role) {
  if (role >= ROLE_T_X_FWD && role <= ROLE_T_X_INV) return role - ROLE_T_X_FWD;
  if (role == ROLE_T_X_R2C) return TK_X_R2C;
  if (role == ROLE_T_X_TUNG) return TK_X_TUNG;
  if (role == ROLE_T_X_FUSE) return TK_X_FUSE;
  return -1;
}

template <typename T> Nonlin<T> nonlin_of(bool split, double mean) {
  Nonlin<T> n{};
  n.split = split ? 1 : 0;
  n.c1 = (T)(3.0 * mean);
  n.c2 = (T)(3.0 * mean * mean);
  n.c1d = 3.0 * mean;
  n.c2d = 3.0 * mean * mean;
  return n;
}
template <typename T> Nonlin<T> nonlin(const pfc_hip_plan_s *p) {
  return nonlin_of<T>(p->mean_split, p->mean);
}

void free_all(pfc_hip_plan_s *p) {
  for (auto &kv : p->tw)
    if (kv.second) (void)hipFree(kv.second);
  p->tw.clear();
  void **bufs[] = {&p->wn,      &p->work,  &p->A,     &p->B,     &p->A1,
                   &p->B1,      &p->A2,    &p->B2,    &p->adj_lam, &p->adj_P,
                   &p->adj_N,   &p->adj_a, &p->adj_b, &p->adj_part, &p->m_eps,
                   &p->m_nl,    &p->colmax, &p->wn64, &p->C, &p->adj_zpart};
  for (void **b : bufs) {
    if (*b) (void)hipFree(*b);
    *b = nullptr;
  }
  p->bytes = 0;
}

// Variant list of a transposed-step kind: the double-butterfly passes on a
// PFC_HIP_FLAG_F64_BUTTERFLIES plan (none for the Tungsten kinds and the fused
// boundary there), the plan precision's list otherwise.
template <typename T> const std::vector<TV<T>> &t_list(const pfc_hip_plan_s *p, int kind, int n) {
  if constexpr (std::is_same_v<T, float>) {
    if (p->xp) return t_variants_xp(kind, n);
  }
  return t_variants<T>(kind, n);
}

// Variants of the roles that own an x pass of the natural layout: the row
// kernels, then, where the plane kernels take the extents, one more ("plane")
// that does the y pass of that direction too.
bool plane_role(int role) {
  return role == ROLE_X_R2C || role == ROLE_X_C2R || role == ROLE_PFC_X || role == ROLE_X_TUNG;
}
template <typename T> int row_variant_count(const pfc_hip_plan_s *p, int role) {
  const int n = p->role_len(role);
  switch (role) {
  case ROLE_X_R2C: return (int)xr2c_variants<T>(n).size();
  case ROLE_X_C2R: return (int)xc2r_variants<T>(n).size();
  case ROLE_PFC_X: return (int)pfcx_variants<T>(n).size();
  case ROLE_X_TUNG: return (int)tungx_variants<T>(n).size();
  default: return 0;
  }
}
template <typename T> bool on_plane(const pfc_hip_plan_s *p, int role) {
  return p->plane_ok() && p->var[role] == row_variant_count<T>(p, role);
}

template <typename T> int variant_count(pfc_hip_plan_s *p, int role) {
  const int n = p->role_len(role);
  if (plane_role(role)) {
    const int rows = row_variant_count<T>(p, role);
    return rows > 0 && p->plane_ok() ? rows + 1 : rows;
  }
  if (role == ROLE_STEP_LAYOUT) return p->t_ok && !p->xp ? 2 : 1;
  if (role == ROLE_STEP_FUSE)
    return p->t_ok && !t_list<T>(p, TK_X_FUSE, p->role_len(ROLE_T_X_FUSE)).empty() ? 2 : 1;
  if (t_kind_of_role(role) >= 0) return (int)t_list<T>(p, t_kind_of_role(role), n).size();
  switch (role) {
  case ROLE_COL_Y: case ROLE_COL_Z: return (int)col_variants<T>(n).size();
  case ROLE_PFC_Z: return (int)pfcz_variants<T>(n).size();
  default: return 0;
  }
}

template <typename T> const std::string *variant_name(pfc_hip_plan_s *p, int role, int v) {
  static const std::string layouts[2] = {"transposed", "natural"};
  static const std::string fuse[2] = {"per_step", "fused"};
  static const std::string plane = "plane";
  const int n = p->role_len(role);
  if (v < 0 || v >= variant_count<T>(p, role)) return nullptr;
  if (role == ROLE_STEP_LAYOUT) return &layouts[p->t_ok ? v : 1];
  if (role == ROLE_STEP_FUSE) return &fuse[v];
  if (plane_role(role) && v == row_variant_count<T>(p, role)) return &plane;
  if (t_kind_of_role(role) >= 0) return &t_list<T>(p, t_kind_of_role(role), n)[v].name;
  switch (role) {
  case ROLE_X_R2C: return &xr2c_variants<T>(n)[v].name;
  case ROLE_X_C2R: return &xc2r_variants<T>(n)[v].name;
  case ROLE_COL_Y: case ROLE_COL_Z: return &col_variants<T>(n)[v].name;
  case ROLE_PFC_X: return &pfcx_variants<T>(n)[v].name;
  case ROLE_PFC_Z: return &pfcz_variants<T>(n)[v].name;
  case ROLE_X_TUNG: return &tungx_variants<T>(n)[v].name;
  default: return nullptr;
  }
}

// Column pass along y (axis 1) or z (axis 2) over a (W, ny, nz) array with
// row pitch `pitch`; fields 0/1 in src/dst.
template <typename T>
hipError_t col_pass(pfc_hip_plan_s *p, int axis, int dir, const void *src0,
                    void *dst0, const void *src1, void *dst1, int nfields,
                    int pitch, hipStream_t s) {
  const int role = axis == 1 ? ROLE_COL_Y : ROLE_COL_Z;
  const int n = axis == 1 ? p->ny : p->nz;
  const auto &vs = col_variants<T>(n);
  const auto &v = vs[p->var[role]];
  ColArgs<T> a{};
  a.src[0] = (const cplx<T> *)src0;
  a.dst[0] = (cplx<T> *)dst0;
  a.src[1] = (const cplx<T> *)src1;
  a.dst[1] = (cplx<T> *)dst1;
  a.tw = twp<T>(p, n, v.plan_id);
  a.W = (short)p->W;
  a.s_pos = axis == 1 ? (long)pitch : (long)pitch * p->ny;
  a.s_outer = axis == 1 ? (long)pitch * p->ny : (long)pitch;
  // y columns of a batched plan run over the z planes of every field
  const long n_outer = axis == 1 ? (long)p->nz * p->batch : p->ny;
  return v.fn(dir, a, n_outer, nfields, s);
}

// Arguments of the plane kernels on spectra of row pitch `pitch`.
template <typename T> PlaneArgs<T> plane_args(pfc_hip_plan_s *p, int pitch) {
  PlaneArgs<T> a{};
  a.nl = nonlin<T>(p);
  a.mnl = p->members ? (const T *)p->m_nl : nullptr;
  a.tw_x = (const cplx<T> *)p->plane_tw[1];
  a.tw_y = (const cplx<T> *)p->plane_tw[0];
  a.wn = (const cplx<double> *)p->plane_wn;
  a.nx = p->nx;
  a.ny = p->ny;
  a.nz = p->nz;
  a.pitch = pitch;
  a.nfields = 1;
  a.scale = (T)1;
  return a;
}
template <typename T> hipError_t plane_pass(pfc_hip_plan_s *p, int mode, const PlaneArgs<T> &a,
                                            hipStream_t s) {
  return plane_launch<T>(mode, a, (long)p->nz * p->batch, s);
}

template <typename T>
hipError_t x_c2r_pass(pfc_hip_plan_s *p, const void *in, void *out, int pitch,
                      double scale, hipStream_t s) {
  const int m = p->nx / 2;
  const auto &v = xc2r_variants<T>(m)[p->var[ROLE_X_C2R]];
  XArgs<T> a{};
  a.in = (const T *)in;
  a.out = (T *)out;
  a.tw = twp<T>(p, m, v.plan_id);
  a.wn = (const cplx<T> *)p->wn;
  a.rows = (long)p->ny * p->nz * p->batch;
  a.pitch = pitch;
  a.scale = (T)scale;
  return v.fn(a, s);
}

// Forward x and y passes of one real field into spectra of row pitch `pitch`.
template <typename T>
int r2c_xy(pfc_hip_plan_s *p, const void *in, void *out, int pitch, hipStream_t s) {
  if (on_plane<T>(p, ROLE_X_R2C)) {
    PlaneArgs<T> a = plane_args<T>(p, pitch);
    a.psi_in = (const T *)in;
    a.dst[0] = (cplx<T> *)out;
    PFC_HIP_TRY(plane_pass<T>(p, PL_FWD, a, s), "r2c plane pass");
    return 0;
  }
  const int m = p->nx / 2;
  const auto &v = xr2c_variants<T>(m)[p->var[ROLE_X_R2C]];
  XArgs<T> a{};
  a.in = (const T *)in;
  a.out = (T *)out;
  a.tw = twp<T>(p, m, v.plan_id);
  a.wn = (const cplx<T> *)p->wn;
  a.rows = (long)p->ny * p->nz;
  a.pitch = pitch;
  a.scale = (T)1;
  PFC_HIP_TRY(v.fn(a, s), "r2c x pass");
  if (p->ny > 1)
    PFC_HIP_TRY(col_pass<T>(p, 1, -1, out, out, nullptr, nullptr, 1, pitch, s), "r2c y pass");
  return 0;
}

// Inverse y and x passes of `in` (row pitch `pitch`) into a real field times
// `scale`; the y pass goes through `work` (which may be `in`) off the plane
// kernels.
template <typename T>
int c2r_yx(pfc_hip_plan_s *p, const void *in, void *work, void *out, int pitch, double scale,
           hipStream_t s) {
  if (on_plane<T>(p, ROLE_X_C2R)) {
    PlaneArgs<T> a = plane_args<T>(p, pitch);
    a.src = (const cplx<T> *)in;
    a.psi_out = (T *)out;
    a.scale = (T)scale;
    PFC_HIP_TRY(plane_pass<T>(p, PL_INV, a, s), "c2r plane pass");
    return 0;
  }
  if (p->ny > 1) {
    PFC_HIP_TRY(col_pass<T>(p, 1, +1, in, work, nullptr, nullptr, 1, pitch, s), "c2r y pass");
    in = work;
  }
  PFC_HIP_TRY(x_c2r_pass<T>(p, in, out, pitch, scale, s), "c2r x pass");
  return 0;
}

template <typename T>
int r2c_impl(pfc_hip_plan_s *p, const void *in, void *out, hipStream_t s) {
  hipError_t e;
  if (int rc = r2c_xy<T>(p, in, out, p->W, s)) return rc;
  if (p->nz > 1) {
    e = col_pass<T>(p, 2, -1, out, out, nullptr, nullptr, 1, p->W, s);
    PFC_HIP_TRY(e, "r2c z pass");
  }
  return 0;
}

// C2R through the workspace `work` (outbox complex values; the plan's own,
// allocated on first use, when null).
template <typename T>
int c2r_impl(pfc_hip_plan_s *p, const void *in, void *out, hipStream_t s,
             void *work = nullptr) {
  const void *cur = in;
  hipError_t e;
  if (!work && (p->nz > 1 || p->ny > 1)) {
    if (int rc = dalloc(p, &p->work, p->outbox() * 2 * p->esize, "c2r workspace"))
      return rc;
    work = p->work;
  }
  if (p->nz > 1) {
    e = col_pass<T>(p, 2, +1, cur, work, nullptr, nullptr, 1, p->W, s);
    PFC_HIP_TRY(e, "c2r z pass");
    cur = work;
  }
  return c2r_yx<T>(p, cur, work, out, p->W,
                   1.0 / ((double)p->nx * (double)p->ny * (double)p->nz), s);
}

// z pass of the natural layout (ZMode `mode`): Psi in `in_a`, N or nothing in
// B, result in `out`.
template <typename T>
hipError_t z_natural(pfc_hip_plan_s *p, int mode, void *in_a, void *out, hipStream_t s) {
  const auto &v = pfcz_variants<T>(p->nz)[p->var[ROLE_PFC_Z]];
  PfcZArgs<T> a{};
  a.zero_k0 = (mode == ZM_PFC && p->mean_split) ? 1 : 0;
  a.mode = mode;
  a.A = (cplx<T> *)in_a;
  a.B = (cplx<T> *)p->B;
  a.out = (cplx<T> *)out;
  a.tw = twp<T>(p, p->nz, v.plan_id);
  a.op = p->op;
  a.top = p->top;
  a.meps = p->members ? (const double *)p->m_eps : nullptr;
  a.mstride = (long)p->padded();
  a.s_pos = (long)p->P * p->ny;
  a.pitch = p->P;
  a.W = p->W;
  return v.fn(a, (long)p->ny * p->batch, s);
}

// Forward x and y passes of psi and N(psi) with the row and column kernels into
// spectra of row pitch `pitch`; `between` is called between the two.
template <typename T, typename F>
int pfc_xy_rows(pfc_hip_plan_s *p, const void *psi, void *out_a, void *out_b, int pitch,
                hipStream_t s, F between) {
  const auto &v = pfcx_variants<T>(p->nx)[p->var[ROLE_PFC_X]];
  PfcXArgs<T> a{};
  a.nl = nonlin<T>(p);
  a.mnl = p->members ? (const T *)p->m_nl : nullptr;
  a.mrows = (long)p->ny * p->nz;
  a.psi = (const T *)psi;
  a.outA = (cplx<T> *)out_a;
  a.outB = (cplx<T> *)out_b;
  a.tw = twp<T>(p, p->nx, v.plan_id);
  a.rows = (long)p->ny * p->nz * p->batch;
  a.pitch = pitch;
  PFC_HIP_TRY(v.fn(a, s), "pfc forward x pass");
  between();
  if (p->ny > 1)
    PFC_HIP_TRY(col_pass<T>(p, 1, -1, out_a, out_a, out_b, out_b, 2, pitch, s),
                "pfc forward y pass");
  return 0;
}
template <typename T>
int pfc_xy_rows(pfc_hip_plan_s *p, const void *psi, void *out_a, void *out_b, int pitch,
                hipStream_t s) {
  return pfc_xy_rows<T>(p, psi, out_a, out_b, pitch, s, [] {});
}

// Spectrum that holds Psi between the x/y passes and the z pass of the natural
// layout: the plane kernels leave it in C (a boundary's two blocks of a plane
// both read A), the row kernels in A.
template <typename T> void *natural_psi(pfc_hip_plan_s *p) {
  return on_plane<T>(p, ROLE_PFC_X) ? p->C : p->A;
}

// Plane pass that ends in Psi and N before the z pass: from psi (PL_FWD), or
// from the spectrum the z pass left in A (PL_BND).
template <typename T>
hipError_t plane_fwd(pfc_hip_plan_s *p, int mode, const void *psi, hipStream_t s) {
  PlaneArgs<T> a = plane_args<T>(p, p->P);
  a.psi_in = (const T *)psi;
  a.src = (const cplx<T> *)p->A;
  a.dst[0] = (cplx<T> *)p->C;
  a.dst[1] = (cplx<T> *)p->B;
  a.nfields = 2;
  return plane_pass<T>(p, mode, a, s);
}

// One fused PFC step: 5 launches, 4 or 3 with plane kernels.  `ev` (optional)
// receives 6 events bracketing the 5 passes (a plane pass counts as its x
// pass; the y pass it includes takes no time).
template <typename T>
int step_natural(pfc_hip_plan_s *p, void *psi, hipStream_t s, hipEvent_t *ev) {
  hipError_t e;
  auto mark = [&](int i) {
    if (ev) (void)hipEventRecord(ev[i], s);
  };
  mark(0);
  if (on_plane<T>(p, ROLE_PFC_X)) {
    PFC_HIP_TRY(plane_fwd<T>(p, PL_FWD, psi, s), "pfc forward plane pass");
    mark(1);
  } else {
    if (int rc = pfc_xy_rows<T>(p, psi, p->A, p->B, p->P, s, [&] { mark(1); })) return rc;
  }
  mark(2);
  PFC_HIP_TRY(z_natural<T>(p, ZM_PFC, natural_psi<T>(p), p->A, s), "pfc z pass");
  mark(3);
  if (on_plane<T>(p, ROLE_X_C2R)) {
    mark(4);
    // 1/(nx ny nz) is folded into opL/opN
    if (int rc = c2r_yx<T>(p, p->A, p->A, psi, p->P, 1.0, s)) return rc;
  } else {
    if (p->ny > 1) {
      e = col_pass<T>(p, 1, +1, p->A, p->A, nullptr, nullptr, 1, p->P, s);
      PFC_HIP_TRY(e, "pfc inverse y pass");
    }
    mark(4);
    e = x_c2r_pass<T>(p, p->A, psi, p->P, 1.0, s);
    PFC_HIP_TRY(e, "pfc inverse x pass");
  }
  mark(5);
  return 0;
}

// Whether multi-step PFC runs keep psi on chip between steps with the plane
// kernels: one boundary pass (PL_BND) per step boundary, the arithmetic of
// PL_INV and PL_FWD, so that a run gives the bits of its single steps.
template <typename T> bool plane_steps(pfc_hip_plan_s *p) {
  return !p->transposed() && !p->tungsten() && on_plane<T>(p, ROLE_PFC_X) &&
         on_plane<T>(p, ROLE_X_C2R);
}

// nsteps >= 1 PFC steps of the natural layout on the plane kernels:
// 2*nsteps + 1 launches.
template <typename T> int steps_plane(pfc_hip_plan_s *p, void *psi, int nsteps, hipStream_t s) {
  for (int i = 0; i < nsteps; ++i) {
    PFC_HIP_TRY(plane_fwd<T>(p, i == 0 ? PL_FWD : PL_BND, psi, s), "pfc plane pass");
    PFC_HIP_TRY(z_natural<T>(p, ZM_PFC, natural_psi<T>(p), p->A, s), "pfc z pass");
  }
  return c2r_yx<T>(p, p->A, p->A, psi, p->P, 1.0, s);
}

// Step buffers of the active layout (allocated on first use).
int step_buffers(pfc_hip_plan_s *p) {
  int rc = 0;
  if (p->transposed()) {
    const size_t c = p->outbox() * 2 * p->esize;
    if (!rc) rc = dalloc(p, &p->A1, c, "step T1 psi");
    if (!rc) rc = dalloc(p, &p->B1, c, "step T1 N");
    if (!rc) rc = dalloc(p, &p->A2, c, "step T2 psi");
    if (!rc) rc = dalloc(p, &p->B2, c, "step T2 N");
  } else {
    const size_t c = p->padded() * 2 * p->esize * p->batch;
    if (!rc) rc = dalloc(p, &p->A, c, "step spectrum A");
    if (!rc) rc = dalloc(p, &p->B, c, "step spectrum B");
    const bool plane = p->prec == PFC_HIP_F64 ? on_plane<double>(p, ROLE_PFC_X)
                                              : on_plane<float>(p, ROLE_PFC_X);
    if (!rc && plane && !p->tungsten()) rc = dalloc(p, &p->C, c, "step spectrum C");
  }
  return rc;
}

// Launch arguments of the transposed PFC step of field m of the plan (its
// own eps and mean when the members are set).
template <typename T> TStepArgs<T> pfc_t_args(pfc_hip_plan_s *p, void *psi, int m = 0) {
  TStepArgs<T> a{};
  T *field = (T *)psi + (size_t)m * p->inbox();
  a.psi_in = field;
  a.psi_out = field;
  a.A1 = (cplx<T> *)p->A1;
  a.B1 = (cplx<T> *)p->B1;
  a.A2 = (cplx<T> *)p->A2;
  a.B2 = (cplx<T> *)p->B2;
  // FP64-butterfly kernels read their merge twiddles as double entries
  a.wn = (const cplx<T> *)(p->xp ? p->wn64 : p->wn);
  a.op = p->op;
  a.nl = nonlin<T>(p);
  if (p->members && p->batch > 1) {
    a.op.eps = p->h_eps[(size_t)m];
    a.nl = nonlin_of<T>(p->mean_split, p->h_mean[(size_t)m]);
  }
  a.zero_k0 = p->mean_split ? 1 : 0;
  a.mode = ZM_PFC;
  a.nfields = 2;
  a.nx = p->nx;
  a.ny = p->ny;
  a.nz = p->nz;
  a.W = p->W;
  return a;
}

// Pass k of the transposed PFC step: 0 forward x, 1 forward y, 2 z,
// 3 inverse y, 4 inverse x; 5 the fused step boundary (inverse x of one step
// with the forward x of the next).
constexpr int kTPassRoles[6] = {ROLE_T_X_FWD, ROLE_T_Y_FWD, ROLE_T_Z,
                                ROLE_T_Y_INV, ROLE_T_X_INV, ROLE_T_X_FUSE};
template <typename T>
int t_pass(pfc_hip_plan_s *p, TStepArgs<T> a, int k, hipStream_t s) {
  static const char *what[6] = {"step x forward", "step y forward", "step z pass",
                                "step y inverse", "step x inverse", "step boundary x"};
  const int role = kTPassRoles[k];
  const int n = p->role_len(role);
  const auto &v = t_list<T>(p, t_kind_of_role(role), n)[p->var[role]];
  const cplx<T> *tw = twp<T>(p, v.half ? n / 2 : n, v.plan_id);
  a.tw_x = a.tw_xm = a.tw_y = a.tw_z = tw;
  PFC_HIP_TRY(v.fn(a, s), what[k]);
  return 0;
}

// One transposed PFC step of every field of the plan, field after field.
// `ev` (optional) brackets the passes of field 0: the pass times of one
// field, as for a single plan.
template <typename T>
int step_transposed(pfc_hip_plan_s *p, void *psi, hipStream_t s, hipEvent_t *ev) {
  for (int m = 0; m < p->batch; ++m) {
    auto mark = [&](int i) {
      if (ev && m == 0) (void)hipEventRecord(ev[i], s);
    };
    const TStepArgs<T> a = pfc_t_args<T>(p, psi, m);
    mark(0);
    for (int k = 0; k < 5; ++k) {
      if (int rc = t_pass<T>(p, a, k, s)) return rc;
      mark(k + 1);
    }
  }
  return 0;
}

// Steps a kept-spectrum run may take before Psi is transformed anew.  The kept
// half spectrum is not passed through real space, so on its kx = 0 and nx/2
// planes the part that does not belong to a real field (rounding errors; the C2R
// drops it) is damped or amplified by opL alone, at most exp(g) per step with g
// the largest growth exponent L*dt of a mode.  It starts at the rounding level
// and is harmless while it stays below 1 (its own roundings then stay below the
// field's): runs of at most 8/g steps keep it under 3000 roundings.  g of the PFC
// operator: L(k2) = -k2 (eps + (1 - k2)^2) is positive for some k2 < 1 +
// sqrt(-eps) only.  1 (no kept spectrum) where dt is not positive.
//
// Measured, ms per step of a run, tuned variants, kept spectrum against psi
// transformed anew at a fused boundary (12C) and against single steps (12C + 2R):
//   FP64 1024^3 17.2 / 21.1 / 23.1 (y 3.14, z 5.3 to 6.1 by where its two spectra
//               land in memory, 4.2 in a run's last step, inverse y 3.46, boundary 4.11)
//   FP32 1024^3  9.0 / 11.6 / 12.0 (y 1.60, z 3.03, inverse y 1.75, boundary 2.44)
//   FP64  512^3 2.00 / 2.50 / 2.75,  FP32 512^3 1.07 / 1.34 / 1.42
//   FP64  256^3 .245 / .334 / .363,  FP32 256^3 .134 / .156 / .188
int fused_span(const PfcOp &o) {
  constexpr int kMax = 64;
  if (!(o.dt > 0)) return 1;
  if (o.eps >= 0) return kMax;
  const double top = 1.0 + std::sqrt(-o.eps);
  double g = 0;
  for (int i = 1; i <= 512; ++i) {
    const double k2 = top * i / 512, m = 1.0 - k2;
    g = std::max(g, -k2 * (o.eps + m * m) * o.dt);
  }
  return g * kMax <= 8.0 ? kMax : std::max(1, (int)(8.0 / g));
}

// Whether multi-step PFC runs keep the spectrum and fuse their step
// boundaries (role 16).
template <typename T> bool fused_steps(pfc_hip_plan_s *p) {
  return p->transposed() && !p->tungsten() && p->var[ROLE_STEP_FUSE] == 1 &&
         !t_list<T>(p, TK_X_FUSE, p->role_len(ROLE_T_X_FUSE)).empty();
}

// Events steps_fused records for nsteps steps in runs of at most `span`.
int fused_events(int nsteps, int span) {
  return 1 + 4 * nsteps + (nsteps + span - 1) / span;
}

// nsteps >= 1 PFC steps with fused boundaries, in runs of at most fused_span
// steps: the first step transforms psi and N(psi) (5 passes but the last); the
// following ones transform N alone (boundary x on T1 of A, forward y A1 -> B2,
// z with the kept spectrum in A2, inverse y B2 -> A1); the inverse x ends the
// run.  4*n + 1 launches a run of n.  `ev` (optional) receives one event before
// the first launch and one after each, in order: fused_events of them.
// (Batched plans: the nsteps steps of field 0, then of field 1, ...; `ev`
// brackets those of field 0.)
template <typename T>
int steps_fused(pfc_hip_plan_s *p, void *psi, int nsteps, hipStream_t s, hipEvent_t *ev) {
  for (int m = 0; m < p->batch; ++m) {
    int e = 0;
    auto mark = [&]() {
      if (ev && m == 0) (void)hipEventRecord(ev[e++], s);
    };
    const TStepArgs<T> a = pfc_t_args<T>(p, psi, m);
    const int span = fused_span(a.op);
    mark();
    for (int done = 0; done < nsteps;) {
      const int n = std::min(span, nsteps - done);
      for (int i = 0; i < n; ++i) {
        TStepArgs<T> f = a; // forward y and z of this step
        if (i > 0) {
          f.nfields = 1;
          f.A2 = a.B2;
        }
        TStepArgs<T> z = a;
        z.keep = i + 1 < n;
        z.mode = i > 0 ? ZM_KEEP : z.keep ? ZM_FIRST : ZM_PFC;
        TStepArgs<T> y = a; // inverse y
        if (i > 0 || z.keep) y.A2 = a.B2;
        if (int rc = t_pass<T>(p, a, i == 0 ? 0 : 5, s)) return rc;
        mark();
        if (int rc = t_pass<T>(p, f, 1, s)) return rc;
        mark();
        if (int rc = t_pass<T>(p, z, 2, s)) return rc;
        mark();
        if (int rc = t_pass<T>(p, y, 3, s)) return rc;
        mark();
      }
      if (int rc = t_pass<T>(p, a, 4, s)) return rc;
      mark();
      done += n;
    }
  }
  return 0;
}

// One Tungsten mean-field step (cpu/tungsten_model.hpp:306-366) in the
// natural layout: 9 launches, A holding Psi and B the mean field, then N.
// `mf` (optional) receives psi_MF of the input field.
template <typename T>
int step_tung_natural(pfc_hip_plan_s *p, void *psi, void *mf, hipStream_t s,
                      hipEvent_t *ev) {
  auto mark = [&](int i) {
    if (ev) (void)hipEventRecord(ev[i], s);
  };
  const int m = p->nx / 2;
  const long rows = (long)p->ny * p->nz;
  hipError_t e;
  // a plane pass does the x pass of its slot and the y pass next to it
  const bool pf = on_plane<T>(p, ROLE_X_R2C), pm = on_plane<T>(p, ROLE_X_TUNG),
             pi = on_plane<T>(p, ROLE_X_C2R);
  mark(0);
  if (pf) {
    if (int rc = r2c_xy<T>(p, psi, p->A, p->P, s)) return rc;
  } else {
    const auto &v = xr2c_variants<T>(m)[p->var[ROLE_X_R2C]];
    XArgs<T> a{};
    a.in = (const T *)psi;
    a.out = (T *)p->A;
    a.tw = twp<T>(p, m, v.plan_id);
    a.wn = (const cplx<T> *)p->wn;
    a.rows = rows;
    a.pitch = p->P;
    a.scale = (T)1;
    PFC_HIP_TRY(v.fn(a, s), "tungsten forward x");
  }
  mark(1);
  if (!pf && p->ny > 1) {
    e = col_pass<T>(p, 1, -1, p->A, p->A, nullptr, nullptr, 1, p->P, s);
    PFC_HIP_TRY(e, "tungsten forward y");
  }
  mark(2);
  PFC_HIP_TRY(z_natural<T>(p, ZM_TMF, p->A, p->B, s), "tungsten mean-field z pass");
  mark(3);
  if (!pm && p->ny > 1) {
    e = col_pass<T>(p, 1, +1, p->B, p->B, nullptr, nullptr, 1, p->P, s);
    PFC_HIP_TRY(e, "tungsten mean-field inverse y");
  }
  mark(4);
  if (pm) {
    PlaneArgs<T> a = plane_args<T>(p, p->P);
    a.tnl = tung_nonlin<T>(p);
    a.psi_in = (const T *)psi;
    a.mf_out = (T *)mf;
    a.src = (const cplx<T> *)p->B;
    a.dst[0] = (cplx<T> *)p->B;
    PFC_HIP_TRY(plane_pass<T>(p, PL_TUNG, a, s), "tungsten plane pass");
  } else {
    const auto &v = tungx_variants<T>(m)[p->var[ROLE_X_TUNG]];
    TungXArgs<T> a{};
    a.nl = tung_nonlin<T>(p);
    a.psi = (const T *)psi;
    a.spec = (cplx<T> *)p->B;
    a.mf_out = (T *)mf;
    a.tw = twp<T>(p, m, v.plan_id);
    a.wn = (const cplx<T> *)p->wn;
    a.rows = rows;
    a.pitch = p->P;
    PFC_HIP_TRY(v.fn(a, s), "tungsten fused x pass");
  }
  mark(5);
  if (!pm && p->ny > 1) {
    e = col_pass<T>(p, 1, -1, p->B, p->B, nullptr, nullptr, 1, p->P, s);
    PFC_HIP_TRY(e, "tungsten forward y (N)");
  }
  mark(6);
  PFC_HIP_TRY(z_natural<T>(p, ZM_TCOMB, p->A, p->A, s), "tungsten combine z pass");
  mark(7);
  if (pi) {
    mark(8);
    if (int rc = c2r_yx<T>(p, p->A, p->A, psi, p->P, 1.0, s)) return rc;
  } else {
    if (p->ny > 1) {
      e = col_pass<T>(p, 1, +1, p->A, p->A, nullptr, nullptr, 1, p->P, s);
      PFC_HIP_TRY(e, "tungsten inverse y");
    }
    mark(8);
    PFC_HIP_TRY(x_c2r_pass<T>(p, p->A, psi, p->P, 1.0, s), "tungsten inverse x");
  }
  mark(9);
  return 0;
}

// The Tungsten step on the transposed layouts: 9 launches (T1/T2 buffers A
// for Psi, B for the mean field and then N).
template <typename T>
int step_tung_transposed(pfc_hip_plan_s *p, void *psi, void *mf, hipStream_t s,
                         hipEvent_t *ev) {
  auto mark = [&](int i) {
    if (ev) (void)hipEventRecord(ev[i], s);
  };
  TStepArgs<T> a{};
  a.mode = ZM_PFC;
  a.nfields = 1;
  a.top = p->top;
  a.tnl = tung_nonlin<T>(p);
  a.mf_out = (T *)mf;
  a.psi_in = (const T *)psi;
  a.psi_out = (T *)psi;
  a.A1 = (cplx<T> *)p->A1;
  a.B1 = (cplx<T> *)p->B1;
  a.A2 = (cplx<T> *)p->A2;
  a.B2 = (cplx<T> *)p->B2;
  a.wn = (const cplx<T> *)p->wn;
  a.op = p->op;
  a.nx = p->nx;
  a.ny = p->ny;
  a.nz = p->nz;
  a.W = p->W;
  struct TPass { int role, mode; bool on_b; const char *what; };
  // on_b: the pass reads and writes the B buffers (passed as A1/A2)
  static const TPass passes[9] = {
      {ROLE_T_X_R2C, ZM_PFC, false, "tungsten x forward"},
      {ROLE_T_Y_FWD, ZM_PFC, false, "tungsten y forward"},
      {ROLE_T_Z, ZM_TMF, false, "tungsten mean-field z pass"},
      {ROLE_T_Y_INV, ZM_PFC, true, "tungsten mean-field y inverse"},
      {ROLE_T_X_TUNG, ZM_PFC, false, "tungsten fused x pass"},
      {ROLE_T_Y_FWD, ZM_PFC, true, "tungsten y forward (N)"},
      {ROLE_T_Z, ZM_TCOMB, false, "tungsten combine z pass"},
      {ROLE_T_Y_INV, ZM_PFC, false, "tungsten y inverse"},
      {ROLE_T_X_INV, ZM_PFC, false, "tungsten x inverse"}};
  mark(0);
  for (int k = 0; k < 9; ++k) {
    const TPass &ps = passes[k];
    const int n = p->role_len(ps.role);
    const auto &v = t_list<T>(p, t_kind_of_role(ps.role), n)[p->var[ps.role]];
    TStepArgs<T> b = a;
    b.mode = ps.mode;
    if (ps.on_b) {
      b.A1 = a.B1;
      b.A2 = a.B2;
    }
    b.tw_x = b.tw_xm = b.tw_y = b.tw_z = twp<T>(p, v.half ? n / 2 : n, v.plan_id);
    PFC_HIP_TRY(v.fn(b, s), ps.what);
    mark(k + 1);
  }
  return 0;
}

// One step of the plan's model; `ev` (optional) receives step_passes()+1
// events bracketing the passes; `mf` (Tungsten, optional) receives psi_MF.
template <typename T>
int step_impl(pfc_hip_plan_s *p, void *psi, hipStream_t s, hipEvent_t *ev,
              void *mf = nullptr) {
  if (int rc = step_buffers(p)) return rc;
  if (p->tungsten())
    return p->transposed() ? step_tung_transposed<T>(p, psi, mf, s, ev)
                           : step_tung_natural<T>(p, psi, mf, s, ev);
  return p->transposed() ? step_transposed<T>(p, psi, s, ev)
                         : step_natural<T>(p, psi, s, ev);
}

constexpr unsigned kAdjBlocks = 2048; // blocks of the reduction kernels
// partials of two reductions plus their two sums
constexpr size_t kPartials = 2 * kAdjBlocks + 2;

// Adjoint of one plain PFC step (see adjoint_kernels.hpp).
int adjoint_f64(pfc_hip_plan_s *p, const void *psi, void *lambda, double *dr, hipStream_t s);
int adjoint_f32(pfc_hip_plan_s *p, const void *psi, void *lambda, double *dr, hipStream_t s);

// partial rows of the column maxima (pfc_hip_column_max)
constexpr long kColParts = 256;

constexpr long kColScratch = pfc_amd::kColScratchDoubles;
using pfc_amd::scratch;

// Device address of `scratch` on device `dev` (current), looked up on the
// first call on that device and kept for the process.
constexpr int kMaxDevices = 64;
int col_scratch(int dev, double **out) {
  static std::mutex mu;
  static double *addr[kMaxDevices] = {};
  if (dev < 0 || dev >= kMaxDevices)
    return fail(PFC_HIP_EUNSUPPORTED, "column-max scratch: device index " + std::to_string(dev));
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    void *p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(PFC_HIP_EDEVICE, std::string("hipGetSymbolAddress(column-max scratch): ") +
                                       hipGetErrorString(e));
    addr[dev] = (double *)p;
  }
  *out = addr[dev];
  return 0;
}

// second stage of the column maxima: the maximum of the nparts (<= 256)
// partials, 64 columns a block, 16 slices of the partials side by side.  One
// thread per column walking all 256 partials was a chain of 256 dependent
// loads: 61.6 us for 128 columns, more than a third of a moving-front step of
// 128x64x64; the slices make it 16 loads in flight and a 16-way LDS maximum.
constexpr int kMaxCols = 64, kMaxSlices = 16;
__global__ void __launch_bounds__(kMaxCols *kMaxSlices)
    k_column_max_final(const double *__restrict__ part, int nx, int nparts,
                       double *__restrict__ out) {
  __shared__ double red[kMaxSlices][kMaxCols];
  const int c = threadIdx.x % kMaxCols, sl = threadIdx.x / kMaxCols;
  const int x = blockIdx.x * kMaxCols + c;
  double m = -1.7976931348623157e308; // as the partials start
  if (x < nx) {
#pragma unroll
    for (int i = 0; i < (int)kColParts / kMaxSlices; ++i) {
      const int p = sl + i * kMaxSlices;
      const double v = p < nparts ? part[(long)p * nx + x] : m;
      m = v > m ? v : m;
    }
  }
  red[sl][c] = m;
  __syncthreads();
  if (sl != 0 || x >= nx) return;
#pragma unroll
  for (int i = 1; i < kMaxSlices; ++i) m = red[i][c] > m ? red[i][c] : m;
  out[x] = m;
}

unsigned ic_blocks(long n) {
  return (unsigned)std::min<long>((n + 255) / 256, 1L << 20);
}

// Sum of `n` partials at the start of part, through part[n], on the host.
int sum_partials(double *part, int n, double *out, hipStream_t s) {
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, s, (const double *)part, n, part + n);
  PFC_HIP_TRY(hipGetLastError(), "adjoint reduction");
  PFC_HIP_TRY(hipMemcpyAsync(out, part + n, sizeof(double), hipMemcpyDeviceToHost, s),
              "adjoint reduction copy");
  PFC_HIP_TRY(hipStreamSynchronize(s), "adjoint sync");
  return 0;
}

// Adjoint of one plain PFC step, double fields, with the z transforms and the
// spectral part in one pass (k_adj_z): x and y passes of psi, N(psi) and lambda
// (one plane launch where the plane kernels are on), k_adj_z, inverse y and x with
// the combine (one plane launch).  128^3 FP64: 32 + 27 + 31 us and the reduction's 6,
// against 13 launches of 187 us pass by pass; 20 steps forward and back 4.28 ms
// (6.33 before).
int adjoint_f64(pfc_hip_plan_s *p, const void *psi, void *lambda, double *dr, hipStream_t s) {
  using T = double;
  const size_t cb = p->padded() * 2 * p->esize, rb = p->inbox() * p->esize;
  const int blocks = adj_z_blocks(p->W, p->ny, p->nz);
  const bool pf = on_plane<T>(p, ROLE_PFC_X), pi = on_plane<T>(p, ROLE_X_C2R);
  int rc = 0;
  if (!rc) rc = dalloc(p, &p->adj_lam, cb, "adjoint spectrum");
  if (!rc) rc = dalloc(p, &p->adj_P, cb, "adjoint spectrum");
  if (!rc) rc = dalloc(p, &p->adj_N, cb, "adjoint spectrum");
  if (!rc && !pi) rc = dalloc(p, &p->adj_a, rb, "adjoint field");
  if (!rc && !pi) rc = dalloc(p, &p->adj_b, rb, "adjoint field");
  if (!rc) rc = dalloc(p, &p->adj_zpart, ((size_t)blocks + 1) * sizeof(double), "adjoint partials");
  if (rc) return rc;
  const T mean = p->mean_split ? p->mean : 0.0;
  // lambda takes the same kernel with and without dr: same bits
  const bool all = dr && pf && on_plane<T>(p, ROLE_X_R2C);
  if (dr && pf) {
    PlaneArgs<T> a = plane_args<T>(p, p->P);
    a.psi_in = (const T *)psi;
    a.lam_in = (const T *)lambda;
    a.dst[0] = (cplx<T> *)p->adj_P;
    a.dst[1] = (cplx<T> *)p->adj_N;
    a.dst[2] = (cplx<T> *)p->adj_lam;
    a.nfields = all ? 3 : 2;
    PFC_HIP_TRY(plane_pass<T>(p, PL_FWD, a, s), "adjoint forward plane pass");
  } else if (dr) {
    if ((rc = pfc_xy_rows<T>(p, psi, p->adj_P, p->adj_N, p->P, s))) return rc;
  }
  if (!all && (rc = r2c_xy<T>(p, lambda, p->adj_lam, p->P, s))) return rc;
  AdjZArgs z{};
  z.lam = (const cplx<T> *)p->adj_lam;
  z.P = (cplx<T> *)p->adj_P;
  z.N = (cplx<T> *)p->adj_N;
  z.tw = twp<T>(p, p->nz, adj_z_plan(p->nz));
  z.op = p->op;
  z.partial = (double *)p->adj_zpart;
  z.s_pos = (long)p->P * p->ny;
  z.pitch = p->P;
  z.W = p->W;
  z.want_dr = dr ? 1 : 0;
  PFC_HIP_TRY(adj_z_launch(z, s), "adjoint z pass");
  if (pi) {
    PlaneArgs<T> a = plane_args<T>(p, p->P);
    a.src = (const cplx<T> *)p->adj_P;
    a.src2 = (const cplx<T> *)p->adj_N;
    a.psi_in = (const T *)psi;
    a.psi_out = (T *)lambda;
    a.mean = mean;
    PFC_HIP_TRY(plane_pass<T>(p, PL_ADJ, a, s), "adjoint inverse plane pass");
  } else {
    if (p->ny > 1)
      PFC_HIP_TRY(col_pass<T>(p, 1, +1, p->adj_P, p->adj_P, p->adj_N, p->adj_N, 2, p->P, s),
                  "adjoint inverse y pass");
    PFC_HIP_TRY(x_c2r_pass<T>(p, p->adj_P, p->adj_a, p->P, 1.0, s), "adjoint inverse x pass");
    PFC_HIP_TRY(x_c2r_pass<T>(p, p->adj_N, p->adj_b, p->P, 1.0, s), "adjoint inverse x pass");
    const long n = (long)p->inbox();
    hipLaunchKernelGGL(k_adj_combine<T>, dim3(ic_blocks(n)), dim3(256), 0, s, (const T *)psi,
                       (const T *)p->adj_a, (const T *)p->adj_b, (T *)lambda, n, mean);
    PFC_HIP_TRY(hipGetLastError(), "adjoint combine");
  }
  if (dr) {
    double h = 0;
    if ((rc = sum_partials((double *)p->adj_zpart, blocks, &h, s))) return rc;
    *dr += h / ((double)p->nx * (double)p->ny * (double)p->nz);
  }
  return 0;
}

// The same on single-precision fields, pass by pass: the FP32-mixed trajectory
// returns FP64 tensors that carry the FP32 rounding of exactly these passes.
int adjoint_f32(pfc_hip_plan_s *p, const void *psi, void *lambda, double *dr, hipStream_t s) {
  using T = float;
  const size_t cb = p->padded() * 2 * p->esize, rb = p->inbox() * p->esize;
  int rc = 0;
  if (!rc) rc = dalloc(p, &p->adj_lam, cb, "adjoint spectrum");
  if (!rc) rc = dalloc(p, &p->adj_P, cb, "adjoint spectrum");
  if (!rc) rc = dalloc(p, &p->adj_N, cb, "adjoint spectrum");
  if (!rc) rc = dalloc(p, &p->adj_a, rb, "adjoint field");
  if (!rc) rc = dalloc(p, &p->adj_b, rb, "adjoint field");
  if (!rc) rc = dalloc(p, &p->adj_part, kPartials * sizeof(double), "reduction partials");
  if (rc) return rc;
  const long n = (long)p->inbox();
  PfcOp o = p->op;
  o.scale = 1.0; // the C2R below applies 1/(nx ny nz)
  if (dr) {
    if ((rc = r2c_impl<T>(p, psi, p->adj_P, s))) return rc;
    hipLaunchKernelGGL(k_cube<T>, dim3(ic_blocks(n)), dim3(256), 0, s, (const T *)psi,
                       (T *)p->adj_a, n, nonlin<T>(p));
    PFC_HIP_TRY(hipGetLastError(), "adjoint cube");
    if ((rc = r2c_impl<T>(p, p->adj_a, p->adj_N, s))) return rc;
  }
  if ((rc = r2c_impl<T>(p, lambda, p->adj_lam, s))) return rc;
  hipLaunchKernelGGL(k_adj_spectral<T>, dim3(kAdjBlocks), dim3(256), 0, s, o, p->W,
                     (const cplx<T> *)p->adj_lam, (cplx<T> *)p->adj_P, (cplx<T> *)p->adj_N,
                     (double *)p->adj_part, dr ? 1 : 0);
  PFC_HIP_TRY(hipGetLastError(), "adjoint spectral kernel");
  if (dr) {
    double h = 0;
    if ((rc = sum_partials((double *)p->adj_part, (int)kAdjBlocks, &h, s))) return rc;
    *dr += h / ((double)p->nx * (double)p->ny * (double)p->nz);
  }
  if ((rc = c2r_impl<T>(p, p->adj_P, p->adj_a, s))) return rc;
  if ((rc = c2r_impl<T>(p, p->adj_N, p->adj_b, s))) return rc;
  hipLaunchKernelGGL(k_adj_combine<T>, dim3(ic_blocks(n)), dim3(256), 0, s, (const T *)psi,
                     (const T *)p->adj_a, (const T *)p->adj_b, (T *)lambda, n,
                     (T)(p->mean_split ? p->mean : 0.0));
  PFC_HIP_TRY(hipGetLastError(), "adjoint combine");
  return 0;
}

// Free energy of the plain PFC model (energy_kernels.hpp), summed in double.
template <typename T>
int free_energy_impl(pfc_hip_plan_s *p, const void *psi, double *F, hipStream_t s) {
  int rc = dalloc(p, &p->adj_P, p->padded() * 2 * p->esize, "free-energy spectrum");
  if (!rc) rc = dalloc(p, &p->adj_part, kPartials * sizeof(double), "reduction partials");
  if (rc) return rc;
  if ((rc = r2c_impl<T>(p, psi, p->adj_P, s))) return rc;
  const double npts = (double)p->nx * (double)p->ny * (double)p->nz;
  const double m = p->mean_split ? p->mean : 0.0;
  double *part = (double *)p->adj_part;
  hipLaunchKernelGGL(k_fe_spectral<T>, dim3(kAdjBlocks), dim3(256), 0, s, p->op, p->W,
                     (const cplx<T> *)p->adj_P, npts * m, part);
  PFC_HIP_TRY(hipGetLastError(), "free-energy spectral sum");
  hipLaunchKernelGGL(k_fe_quartic<T>, dim3(kAdjBlocks), dim3(256), 0, s, (const T *)psi,
                     (long)p->inbox(), m, part + kAdjBlocks);
  PFC_HIP_TRY(hipGetLastError(), "free-energy quartic sum");
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, s, (const double *)part,
                     (int)kAdjBlocks, part + 2 * kAdjBlocks);
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, s, (const double *)part + kAdjBlocks,
                     (int)kAdjBlocks, part + 2 * kAdjBlocks + 1);
  PFC_HIP_TRY(hipGetLastError(), "free-energy reduction");
  double h[2] = {0, 0};
  PFC_HIP_TRY(hipMemcpyAsync(h, part + 2 * kAdjBlocks, sizeof(h), hipMemcpyDeviceToHost, s),
              "free-energy copy");
  PFC_HIP_TRY(hipStreamSynchronize(s), "free-energy sync");
  const double dV = p->spacing[0] * p->spacing[1] * p->spacing[2];
  *F = dV * (h[0] / (2.0 * npts) + 0.25 * h[1]);
  return 0;
}

// One 16-byte value per thread: the plain streaming copy of
// pfc_hip_stream_copy.
__global__ void __launch_bounds__(256) k_stream_copy(const uint4 *__restrict__ src,
                                                     uint4 *__restrict__ dst, size_t n) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

// Whether the plane kernels are the default of the x roles: where no ordinary call
// is slower than with the row and column kernels.  One block takes a plane, so they
// need planes enough to keep the CUs busy.  Swept over 2127 extents of up to 2^23
// points (us, plane / row and column kernels; run = step of a multi-step run, one =
// single step):
//   FP64 64x64x64    run 16.0 / 23.5  one 19.4 / 23.7  r2c 14.5 / 17.6  c2r 14.2 / 17.6
//   FP64 128x128x96  run 41.4 / 52.4  one 47.4 / 53.1  r2c 25.4 / 30.1  c2r 24.8 / 28.2
//   FP64 128x128x64  run 36.3 / 44.0  one 41.0 / 44.6  r2c 22.1 / 22.5  c2r 20.9 / 21.5
//   FP64 128x128x32  run 30.6 / 32.9  one 37.1 / 33.5  r2c 19.1 / 18.0  c2r 18.0 / 17.3
//   FP32 96x96x256   run 39.8 / 50.2  one 43.0 / 50.8  r2c 20.7 / 28.1  c2r 19.6 / 26.6
//   FP32 128x128x128 run 35.8 / 45.6  one 40.4 / 46.1  r2c 20.8 / 23.0  c2r 19.9 / 22.1
//   FP32 128x128x48  run 25.0 / 29.3  one 32.5 / 29.8  r2c 16.4 / 17.7  c2r 15.8 / 17.9
//   FP32 512x32x48   run 26.9 / 29.1  one 34.0 / 29.8  r2c 19.2 / 17.7  c2r 16.3 / 17.6
//   FP32 128x192x192 run 67.3 / 68.2  one 74.9 / 69.0  r2c 32.0 / 34.8  c2r 31.3 / 32.1
//   FP32 64x512x128  run 93.9 / 69.3  one 110  / 70.1  r2c 40.9 / 36.2  c2r 41.5 / 33.4
// so, in FP64 and up to 32 KB a plane: from 64 planes on, or where a plane's bytes
// are at most 1600 per plane there is.  Larger FP32 planes against the faster FP32 row
// kernels: at most 1000 up to 80 KB; above that a CU holds one block, so at most 800
// and whole rounds of the 256 CUs (two blocks a plane).  Columns of 512 points run
// one line a wave, in 8- or 16-byte pieces: never.  Above 140 KB the column passes
// are as fast.  Over the extents this takes, single steps gain 1.22 (FP32) and 1.29
// (FP64) times and runs 1.38 and 1.46; five of 1641 lose more than 3 % in some call, 6 %
// at worst (with 64 planes or 1600 bytes for all: 72, and 36 %).
bool plane_variant_default(const pfc_hip_plan_s *p) {
  const size_t b = p->plane_bytes(), nz = (size_t)p->nz;
  if (b == 0 || b > 140 * 1024 || p->ny >= 512) return false;
  if (p->prec == PFC_HIP_F64 || b <= 32 * 1024) return nz >= 64 || b <= 1600 * nz;
  return b <= 80 * 1024 ? b <= 1000 * nz : b <= 800 * nz && nz % 128 == 0;
}

// Default variants by line length, where another variant than the first of a
// role's list measured faster over the grids of that length (role sweeps on
// 256x128x128 to 1024^3 for the transposed roles, 16x1024x64 to 1024^3 for the
// natural ones, both models; the ratio to each sweep's best was 1.00 to 1.05 for
// these and is given below for the first of the list).  What they have in
// common: 128 contiguous bytes per strided access (8 lines of doubles, 16 of
// floats), few wide transposition rounds instead of one per value, non-temporal
// lines, a z table per line; 8 values a thread in double up to 512 points, where
// 16 leave one or two waves per SIMD.  Single precision takes no plan with more
// radix passes (roundings) than the first of its list.
struct DefaultVariant {
  int role, n;
  const char *name;
};
constexpr DefaultVariant kDefaultF64[] = {
    // natural layout
    {ROLE_PFC_Z, 96, "r4x4x6/E12/L8/full"},            // first 1.24
    {ROLE_PFC_Z, 128, "r8x4x4/E8/L8/full"},            // 1.09 to 1.17
    {ROLE_PFC_Z, 256, "r8x8x4/E8/L8/full"},            // 1.22 at 512x32x256
    {ROLE_PFC_Z, 512, "r8x8x8/E8/L4/full"},            // 1.08
    {ROLE_COL_Y, 96, "r4x4x6/E12/L8/full"},            // 1.09
    {ROLE_COL_Y, 512, "r8x8x8/E8/L8/full"},            // 1.05 to 1.09
    {ROLE_COL_Z, 96, "r4x4x6/E12/L8/full"},            // as the y columns
    {ROLE_COL_Z, 512, "r8x8x8/E8/L8/full"},
    {ROLE_PFC_X, 256, "r8x8x4/E8/rows8"},              // 1.03 to 1.06
    {ROLE_X_R2C, 128, "r8x4x4/E8/rows8"},              // 1.14, 1.21
    {ROLE_X_R2C, 256, "r4x4x4x4/E4/rows1"},            // 1.08
    {ROLE_X_C2R, 128, "r8x4x4/E8/rows16"},             // 1.07 to 1.12
    {ROLE_X_C2R, 256, "r4x4x4x4/E4/rows2"},            // 1.02 to 1.11
    // rows of 1024: no line; r16x16x2/E16/rows4 is 2 % ahead from 36864 rows up
    // (C2R 405 | 414 us) and 2 to 6 % behind below (256 rows 16.5 | 15.7)
    {ROLE_X_TUNG, 128, "r8x4x4/E8/rows4"},             // 1.24, 1.52
    {ROLE_X_TUNG, 256, "r4x4x4x4/E4/rows1"},           // 1.05
    // transposed layout
    {ROLE_T_X_FWD, 256, "r4x4x4x4/E4/G8/split/wide/nt"},    // 1.00 to 1.16
    {ROLE_T_X_FWD, 512, "r8x8x8/E8/G8/full/wide/nt"},       // 1.15
    {ROLE_T_X_FWD, 1024, "r16x16x4/E16/G8/split/wide/nt"},  // 1.02, 1.04
    {ROLE_T_Y_FWD, 128, "r8x4x4/E8/G8/split/wide4/nt"},     // 1.06, 1.11
    {ROLE_T_Y_FWD, 256, "r16x16/E16/G8/split/wide4/nt"},    // 1.02 to 1.28
    {ROLE_T_Y_FWD, 512, "r8x8x8/E8/G8/split/wide1/nt"},     // 1.13, 1.16
    {ROLE_T_Y_FWD, 1024, "r16x16x4/E16/G8/split/wide2/nt"}, // 1.08
    {ROLE_T_Z, 128, "r8x4x4/E8/G4/split/mt"},               // 1.29 to 1.44
    {ROLE_T_Z, 256, "r8x8x4/E8/G2/split/pre"},              // 1.13 to 1.26
    {ROLE_T_Z, 512, "r8x8x8/E8/G1/full/mt"},                // 1.25
    {ROLE_T_Z, 1024, "r16x16x4/E16/G1/split/mt"},           // 1.16
    {ROLE_T_Y_INV, 128, "r8x4x4/E8/G8/split/wide4/nt"},     // 1.37
    {ROLE_T_Y_INV, 256, "r16x16/E16/G8/split/wide2"},       // 1.03 to 1.22
    {ROLE_T_Y_INV, 512, "r16x16x2/E16/G8/split/wide2"},     // 1.04, 1.06
    {ROLE_T_Y_INV, 1024, "r16x16x4/E16/G8/split/wide2"},    // 1.01, 1.20
    {ROLE_T_X_INV, 128, "r8x4x4/E8/G8/nt"},                 // 1.01 to 1.25
    {ROLE_T_X_INV, 256, "r8x8x4/E8/G8/nt"},                 // 1.04 to 1.19
    {ROLE_T_X_INV, 512, "r16x16x2/E16/G8/nt"},              // 1.03, 1.07
    {ROLE_T_X_FUSE, 128, "r8x4x4/E8/G8/cols/w4"},           // 1.08
    {ROLE_T_X_FUSE, 256, "r16x16/E16/G8/cols/w2"},          // 1.17
    {ROLE_T_X_FUSE, 512, "r8x8x8/E8/G8/cols/w4"},           // 1.20
    {ROLE_T_X_R2C, 128, "r8x4x4/E8/G8"},                    // 1.06, 1.10
    {ROLE_T_X_TUNG, 128, "r8x4x4/E8/G8/wide"},              // 1.05, 1.15
    {ROLE_T_X_TUNG, 256, "r8x8x4/E8/G8/wide/w4"},           // 1.04
    {ROLE_T_X_TUNG, 512, "r8x8x8/E8/G8/wide/w4"}};          // 1.25 (1024^3)
constexpr DefaultVariant kDefaultF32[] = {
    {ROLE_PFC_Z, 512, "r8x8x8/E8/L8/full"},                  // first 1.13
    {ROLE_PFC_Z, 1024, "r16x16x4/E16/L8/full"},              // 1.77, 2.40
    {ROLE_COL_Y, 512, "r8x8x8/E8/L16/full"},                 // 1.02
    {ROLE_COL_Y, 1024, "r16x16x4/E16/L8/full"},              // 1.06
    {ROLE_COL_Z, 512, "r8x8x8/E8/L16/full"},                 // as the y columns
    {ROLE_COL_Z, 1024, "r16x16x4/E16/L8/full"},
    {ROLE_PFC_X, 256, "r16x16/E16/rows8"},                   // 1.01, 1.11
    {ROLE_T_X_FWD, 256, "r16x16/E16/G16/full/wide/nt"},      // 1.10, 1.27
    {ROLE_T_X_FWD, 512, "r8x8x8/E8/G16/split/wide/nt"},      // 1.07, 1.33
    {ROLE_T_X_FWD, 1024, "r16x16x4/E16/G16/split/wide/nt"},  // 1.11, 1.17
    {ROLE_T_Y_FWD, 256, "r16x16/E16/G16/split/wide2"},       // 1.02 to 1.04
    {ROLE_T_Y_FWD, 512, "r8x8x8/E8/G16/split/wide1/nt"},     // 1.02, 1.05
    {ROLE_T_Y_FWD, 1024, "r16x16x4/E16/G16/split/wide2/nt"}, // 1.20
    {ROLE_T_Z, 128, "r16x8/E16/G8/full/mt"},                 // 1.04 to 1.52
    {ROLE_T_Z, 256, "r16x16/E16/G4/split/mt"},               // 1.29 to 1.36
    {ROLE_T_Z, 512, "r8x8x8/E8/G2/split/mtp"},               // 1.37
    {ROLE_T_Z, 1024, "r16x16x4/E16/G2/split/mtp"},           // 1.73
    {ROLE_T_Y_INV, 128, "r16x8/E16/G16/split/wide2/nt"},     // 1.76, 1.79
    {ROLE_T_Y_INV, 256, "r16x16/E16/G16/split/wide2"},       // 1.24 to 1.34
    {ROLE_T_Y_INV, 512, "r16x16x2/E16/G16/split/wide2"},     // 1.16, 1.21
    {ROLE_T_Y_INV, 1024, "r16x16x4/E16/G16/split/wide2"},    // 1.08
    {ROLE_T_X_INV, 512, "r8x8x8/E8/G16/nt"},                 // 1.05, 1.35
    {ROLE_T_X_FUSE, 128, "r16x8/E16/G8"},                    // 1.04, 1.06
    {ROLE_T_X_FUSE, 512, "r16x16x2/E16/G16/nt"}};            // 1.19, 1.29
// plans with FP64 butterflies
constexpr DefaultVariant kDefaultXp[] = {
    {ROLE_T_X_FWD, 256, "r16x16/E16/xp/G16/full/wide"},         // first 1.11, 1.15
    {ROLE_T_X_FWD, 512, "r8x8x8/E8/xp/G16/split/wide/nt"},      // 1.02
    {ROLE_T_X_FWD, 1024, "r16x16x4/E16/xp/G8/split/wide"},      // 1.13
    {ROLE_T_Y_FWD, 256, "r16x16/E16/xp/G16/split/wide2/nt"},    // 1.11
    {ROLE_T_Y_FWD, 512, "r8x8x8/E8/xp/G16/split/wide2/nt"},     // 1.00, 1.12
    {ROLE_T_Y_FWD, 1024, "r16x16x4/E16/xp/G16/split/wide2/nt"}, // (as 256)
    {ROLE_T_Z, 128, "r8x4x4/E8/xp/G4/split/mt"},                // 1.01 to 1.04
    {ROLE_T_Z, 256, "r16x16/E16/xp/G4/split/mt"},               // 1.31
    {ROLE_T_Z, 512, "r8x8x8/E8/xp/G1/full/mt"},                 // 1.13
    {ROLE_T_Z, 1024, "r16x16x4/E16/xp/G2/split/mtp"},           // 1.2
    {ROLE_T_Y_INV, 128, "r8x4x4/E8/xp/G16/split/wide2/nt"},     // 1.13
    {ROLE_T_Y_INV, 256, "r16x16/E16/xp/G16/split/wide2/nt"},    // 1.08 (in a run)
    {ROLE_T_Y_INV, 512, "r16x16x2/E16/xp/G16/split/wide2"},     // 1.00, 1.06
    {ROLE_T_Y_INV, 1024, "r16x16x4/E16/xp/G16/split/wide2"},
    {ROLE_T_X_INV, 128, "r8x4x4/E8/xp/G16"},                    // 1.03 to 1.15
    {ROLE_T_X_INV, 256, "r16x16/E16/xp/G16"}};                  // 1.05
// Transposed passes of PFC plans whose grids the 256 MB last-level cache holds: so
// many spectra of the plan have to fit.
struct CachedVariant {
  DefaultVariant d;
  int spectra;
};
constexpr size_t kLastLevelCache = 256u << 20;
constexpr CachedVariant kCachedF64[] = {
    {{ROLE_T_X_FWD, 256, "r4x4x4x4/E4/G8/split/wide"}, 3},
    {{ROLE_T_X_FWD, 512, "r8x8x8/E8/G8/full/wide"}, 3},
    {{ROLE_T_Y_FWD, 128, "r8x4x4/E8/G8/split/wide4"}, 3},
    {{ROLE_T_Y_FWD, 256, "r16x16/E16/G8/split/wide4"}, 3},
    {{ROLE_T_Z, 128, "r8x4x4/E8/G4/full"}, 3},
    {{ROLE_T_Z, 256, "r16x16/E16/G4/split"}, 3},
    {{ROLE_T_Z, 512, "r8x8x8/E8/G1/split/pre"}, 3},
    {{ROLE_T_Y_INV, 128, "r8x4x4/E8/G8/split/wide4"}, 3},
    {{ROLE_T_X_INV, 128, "r8x4x4/E8/G8"}, 3},
    {{ROLE_T_X_INV, 256, "r8x8x4/E8/G8"}, 3}};
constexpr CachedVariant kCachedF32[] = {
    {{ROLE_T_X_FWD, 256, "r16x16/E16/G16/split"}, 6},
    {{ROLE_T_X_FWD, 512, "r8x8x8/E8/G16/split/wide"}, 6},
    {{ROLE_T_Y_FWD, 512, "r8x8x8/E8/G16/split"}, 3},
    {{ROLE_T_Z, 128, "r16x8/E16/G8/split"}, 3},
    {{ROLE_T_Z, 256, "r8x8x4/E8/G2/split/pre"}, 3},
    {{ROLE_T_Z, 512, "r8x8x8/E8/G2/split"}, 3},
    {{ROLE_T_Y_INV, 128, "r16x8/E16/G16/split/wide2"}, 3},
    {{ROLE_T_X_INV, 512, "r8x8x8/E8/G16"}, 3}};
constexpr CachedVariant kCachedXp[] = {
    {{ROLE_T_X_FWD, 256, "r16x16/E16/xp/G16/split/wide"}, 3},
    {{ROLE_T_X_FWD, 512, "r8x8x8/E8/xp/G16/split/wide"}, 3},
    {{ROLE_T_X_INV, 256, "r8x8x4/E8/xp/G16"}, 6}};

template <typename T> void pick_variant(pfc_hip_plan_s *p, const DefaultVariant &d) {
  if (p->role_len(d.role) != d.n) return;
  const int nv = variant_count<T>(p, d.role);
  for (int v = 0; v < nv; ++v)
    if (*variant_name<T>(p, d.role, v) == d.name) p->var[d.role] = v;
}

template <typename T, typename Pick> void each_default(const pfc_hip_plan_s *p, Pick pick) {
  if (p->xp)
    std::for_each(std::begin(kDefaultXp), std::end(kDefaultXp), pick);
  else if (sizeof(T) == 8)
    std::for_each(std::begin(kDefaultF64), std::end(kDefaultF64), pick);
  else
    std::for_each(std::begin(kDefaultF32), std::end(kDefaultF32), pick);
}

template <typename T, typename Pick> void each_cached(const pfc_hip_plan_s *p, Pick pick) {
  if (p->xp)
    std::for_each(std::begin(kCachedXp), std::end(kCachedXp), pick);
  else if (sizeof(T) == 8)
    std::for_each(std::begin(kCachedF64), std::end(kCachedF64), pick);
  else
    std::for_each(std::begin(kCachedF32), std::end(kCachedF32), pick);
}

// The transposed passes depend on the footprint and, through it, on the model,
// which the operators set: a non-temporal line is right where the next pass finds
// its grid in HBM anyway and wrong where the last-level cache would hold it.  A PFC
// run keeps three spectra (A2, B2, A1); us of a single step | a step of a run, both
// with every other pass as it is here, plain line against non-temporal:
//   FP64 256x128x128  x fwd 96 / 102 | 71 / 72      x inv 98 / 102 | 71 / 72
//   FP64 256x256x128  x fwd 182 / 192 | 128 / 128   y fwd 182 / 192 | 124 / 128
//   FP64 256x128x256  y inv 189 / 195 | 126 / 132   x inv 185 / 195 | 131 / 132
//   FP32 256x256x128  x fwd 98 / 107 | 77 / 77
//   FP32 512x128x128  x fwd 99 / 104 | 78 / 79      y inv 104 / 104 | 76 / 79
//   FP32 1024x128x128 y inv 194 / 207 | 141 / 147   x inv 198 / 207 | 146 / 147
//   FP32 256x512x128  y fwd 195 / 202 | 138 / 142
//   FP32 with FP64 butterflies 512x256x128 x fwd 208 / 224
// and beyond it FP32 512x512x128 x fwd 376 / 359, FP64 256x256x512 y fwd 554 / 533
// (run).  The FP32 x pass reads a field and writes one spectrum while the previous
// step's lines leave the cache: plain up to 42 MB, at 67 MB 256^3 191 / 188 and
// 512x256x128 197 / 188.  z pass, plain lines against the table form, in a run: FP32 256^3
// 129 / 137, FP64 256x128x128 70 / 75, beyond the cache FP32 256x256x512 254 / 250;
// of the plain FP32 forms, split against full transposition in a single step
// 256x256x128 101 / 107, 1024x128x128 195 / 207 (runs equal), and at 256 points
// tables read ahead 256^3 178 / 188 | 131 / 133.  Tungsten's multipliers cost more
// than the lines: it keeps the forms of large grids.
template <typename T> void transposed_defaults(pfc_hip_plan_s *p) {
  if (!p->t_ok) return;
  const size_t spectrum = p->outbox() * 2 * p->esize;
  for (int r : {ROLE_T_X_FWD, ROLE_T_Y_FWD, ROLE_T_Z, ROLE_T_Y_INV, ROLE_T_X_INV}) {
    if (p->chosen[r]) continue;
    p->var[r] = 0;
    each_default<T>(p, [&](const DefaultVariant &d) {
      if (d.role == r) pick_variant<T>(p, d);
    });
    if (p->tungsten()) continue;
    each_cached<T>(p, [&](const CachedVariant &c) {
      if (c.d.role == r && c.spectra * spectrum <= kLastLevelCache) pick_variant<T>(p, c.d);
    });
  }
}

// The variant each role of a new plan starts with.
template <typename T> void default_variants(pfc_hip_plan_s *p) {
  each_default<T>(p, [&](const DefaultVariant &d) { pick_variant<T>(p, d); });
  transposed_defaults<T>(p);
  for (int r = 0; r < ROLE_COUNT; ++r)
    if (plane_role(r) && row_variant_count<T>(p, r) > 0 && plane_variant_default(p))
      p->var[r] = row_variant_count<T>(p, r);
  p->var[ROLE_STEP_FUSE] = variant_count<T>(p, ROLE_STEP_FUSE) - 1;
}

// Defaults that depend on the model.  A single-precision Tungsten step keeps the
// first variant of every role: a moving front reads the field's column maxima in
// double, which carry the FP32 rounding of exactly these passes (others are as
// accurate, 7.5e-8 against 9.0e-8, but 8e-8 away).
template <typename T> void model_variants(pfc_hip_plan_s *p) {
  if (sizeof(T) == 8 || p->xp) {
    transposed_defaults<T>(p);
    return;
  }
  int kept[ROLE_COUNT];
  std::copy(std::begin(p->var), std::end(p->var), kept);
  if (p->tungsten())
    std::fill(std::begin(p->var), std::end(p->var), 0);
  else
    default_variants<T>(p);
  for (int r = 0; r < ROLE_COUNT; ++r)
    if (p->chosen[r] || r == ROLE_STEP_LAYOUT || r == ROLE_STEP_FUSE) p->var[r] = kept[r];
}

int check_plan(pfc_hip_plan_t p) {
  if (!p) return fail(PFC_HIP_EINVAL, "null plan");
  return 0;
}

// Entry points that act on one field refuse batched plans.
int check_single(pfc_hip_plan_t p, const char *fn) {
  if (int rc = check_plan(p)) return rc;
  if (p->batch > 1)
    return fail(PFC_HIP_EUNSUPPORTED, std::string(fn) + ": not available on a batched plan");
  return 0;
}

int set_device(pfc_hip_plan_t p) {
  int cur = -1;
  if (hipGetDevice(&cur) == hipSuccess && cur == p->device) return 0;
  PFC_HIP_TRY(hipSetDevice(p->device), "hipSetDevice");
  return 0;
}

} // namespace

// ===========================================================================
// C ABI
// ===========================================================================
extern "C" {

int pfc_hip_abi_version(void) { return PFC_HIP_ABI_VERSION; }

const char *pfc_hip_last_error(void) { return g_last_error.c_str(); }

int pfc_hip_plan_create(int nx, int ny, int nz, int precision, int flags,
                        pfc_hip_plan_t *plan) {
  if (!plan) return fail(PFC_HIP_EINVAL, "pfc_hip_plan_create: plan is null");
  *plan = nullptr;
  if (nx < 1 || ny < 1 || nz < 1)
    return fail(PFC_HIP_EINVAL, "pfc_hip_plan_create: extents must be >= 1");
  if (precision != PFC_HIP_F64 && precision != PFC_HIP_F32)
    return fail(PFC_HIP_EINVAL, "pfc_hip_plan_create: unknown precision " +
                                    std::to_string(precision));
  if (flags & ~PFC_HIP_FLAG_F64_BUTTERFLIES)
    return fail(PFC_HIP_EINVAL, "pfc_hip_plan_create: unknown flags " + std::to_string(flags));
  if ((flags & PFC_HIP_FLAG_F64_BUTTERFLIES) && precision != PFC_HIP_F32)
    return fail(PFC_HIP_EINVAL,
                "pfc_hip_plan_create: PFC_HIP_FLAG_F64_BUTTERFLIES needs PFC_HIP_F32");
  if (nx % 2 != 0 || !supported_len(nx / 2) || !supported_len(ny) ||
      !supported_len(nz))
    return fail(PFC_HIP_EUNSUPPORTED,
                "pfc_hip_plan_create: unsupported extents " + std::to_string(nx) +
                    "x" + std::to_string(ny) + "x" + std::to_string(nz) +
                    " (each axis in {1,2,4,...,1024} or {12,24,48,96,192}; nx even with nx/2 "
                    "in the same set)");
  auto *p = new (std::nothrow) pfc_hip_plan_s();
  if (!p) return fail(PFC_HIP_ENOMEM, "pfc_hip_plan_create: host allocation");
  p->nx = nx;
  p->ny = ny;
  p->nz = nz;
  p->prec = precision;
  p->flags = flags;
  p->W = nx / 2 + 1;
  p->esize = precision == PFC_HIP_F64 ? 8 : 4;
  // 128-byte aligned rows for the plan-owned spectra
  const int per128 = (int)(128 / (2 * p->esize));
  p->P = (p->W + per128 - 1) / per128 * per128;
  if (hipGetDevice(&p->device) != hipSuccess) {
    delete p;
    return fail(PFC_HIP_EDEVICE, "pfc_hip_plan_create: no HIP device");
  }
  int rc = 0;
  if (!rc) rc = upload_line_tables(p, nx / 2);
  if (!rc && supported_len(nx)) rc = upload_line_tables(p, nx);
  if (!rc) rc = upload_line_tables(p, ny);
  if (!rc) rc = upload_line_tables(p, nz);
  const bool plane = p->plane_ok() && !(flags & PFC_HIP_FLAG_F64_BUTTERFLIES);
  if (!rc) rc = upload_real_tables(p, plane);
  if (!rc && plane) {
    const hipError_t e = precision == PFC_HIP_F64 ? plane_init<double>() : plane_init<float>();
    if (e != hipSuccess)
      rc = fail(PFC_HIP_EDEVICE, std::string("plane kernels: ") + hipGetErrorString(e));
  }
  if (!rc) {
    bool ok = true;
    for (int r = 0; r < ROLE_COUNT; ++r) {
      if (t_kind_of_role(r) < 0) continue;
      int c = precision == PFC_HIP_F64 ? variant_count<double>(p, r)
                                       : variant_count<float>(p, r);
      ok = ok && c > 0;
    }
    p->t_ok = ok;
  }
  if (!rc && (flags & PFC_HIP_FLAG_F64_BUTTERFLIES)) {
    p->xp = true;
    bool ok = p->t_ok;
    for (int r = ROLE_T_X_FWD; r <= ROLE_T_X_INV && ok; ++r)
      ok = variant_count<float>(p, r) > 0;
    if (!ok) {
      free_all(p);
      delete p;
      return fail(PFC_HIP_EUNSUPPORTED,
                  "pfc_hip_plan_create: PFC_HIP_FLAG_F64_BUTTERFLIES needs the transposed "
                  "step (power-of-two extents, every axis >= 128, nx >= 256), got " +
                      std::to_string(nx) + "x" + std::to_string(ny) + "x" + std::to_string(nz));
    }
    for (int n : {nx, nx / 2, ny, nz})
      if (!rc) rc = upload_line_tables_xp(p, n);
    if (!rc) rc = upload_wn64(p);
  }
  if (rc) {
    free_all(p);
    delete p;
    return rc;
  }
  if (precision == PFC_HIP_F64)
    default_variants<double>(p);
  else
    default_variants<float>(p);
  *plan = p;
  return 0;
}

int pfc_hip_plan_create_batched(int nx, int ny, int nz, int batch, int precision, int flags,
                                pfc_hip_plan_t *plan) {
  if (!plan) return fail(PFC_HIP_EINVAL, "pfc_hip_plan_create_batched: plan is null");
  *plan = nullptr;
  if (batch < 1 || batch > (1 << 16))
    return fail(PFC_HIP_EINVAL, "pfc_hip_plan_create_batched: batch must be in [1, 65536]");
  if ((double)nx * ny * nz * batch > 9.0e18 / 16)
    return fail(PFC_HIP_EINVAL, "pfc_hip_plan_create_batched: too many points");
  if (int rc = pfc_hip_plan_create(nx, ny, nz, precision, flags, plan)) return rc;
  pfc_hip_plan_s *p = *plan;
  p->batch = batch;
  return 0;
}

int pfc_hip_plan_destroy(pfc_hip_plan_t plan) {
  if (!plan) return 0;
  (void)set_device(plan);
  free_all(plan);
  delete plan;
  return 0;
}

int pfc_hip_sizes(pfc_hip_plan_t plan, size_t *inbox, size_t *outbox,
                  size_t *workspace) {
  if (int rc = check_plan(plan)) return rc;
  if (inbox) *inbox = plan->inbox();
  if (outbox) *outbox = plan->outbox();
  if (workspace) *workspace = plan->outbox();
  return 0;
}

int pfc_hip_allocated_bytes(pfc_hip_plan_t plan, size_t *bytes) {
  if (int rc = check_plan(plan)) return rc;
  if (!bytes) return fail(PFC_HIP_EINVAL, "pfc_hip_allocated_bytes: null");
  *bytes = plan->bytes;
  return 0;
}

int pfc_hip_r2c(pfc_hip_plan_t plan, const void *in, void *out, void *stream) {
  if (int rc = check_single(plan, "pfc_hip_r2c")) return rc;
  if (!in || !out) return fail(PFC_HIP_EINVAL, "pfc_hip_r2c: null buffer");
  if (int rc = set_device(plan)) return rc;
  hipStream_t s = (hipStream_t)stream;
  return plan->prec == PFC_HIP_F64 ? r2c_impl<double>(plan, in, out, s)
                                   : r2c_impl<float>(plan, in, out, s);
}

int pfc_hip_c2r(pfc_hip_plan_t plan, const void *in, void *out, void *stream) {
  if (int rc = check_single(plan, "pfc_hip_c2r")) return rc;
  if (!in || !out) return fail(PFC_HIP_EINVAL, "pfc_hip_c2r: null buffer");
  if (int rc = set_device(plan)) return rc;
  hipStream_t s = (hipStream_t)stream;
  return plan->prec == PFC_HIP_F64 ? c2r_impl<double>(plan, in, out, s)
                                   : c2r_impl<float>(plan, in, out, s);
}

// Host-side scalars of the Tungsten operators, in the reference's order
// (tungsten_spectral.hpp:91-101), without contraction into FMAs.
static TungOp tungsten_scalars(const double *q) {
#pragma clang fp contract(off)
  // q = {alpha2, lambda2, farTol, highOrd, Bx, T, T0, stabP, p2_bar, q2_bar}
  TungOp t{};
  t.alpha2 = q[0];
  t.lambda2 = q[1];
  t.rTol = ((-q[0]) * std::log(q[2])) - 1.0;
  t.highOrd = (int)q[3];
  t.c_peak = q[4] * std::exp((-q[5]) / q[6]);
  t.sp2 = q[7] + q[8];
  t.q2 = q[9];
  return t;
}

int pfc_hip_pfc_set_operators(pfc_hip_plan_t plan, int model_kind,
                              const double *params, int nparams, double dt) {
  if (int rc = check_plan(plan)) return rc;
  if (model_kind != PFC_HIP_MODEL_PFC && model_kind != PFC_HIP_MODEL_TUNGSTEN)
    return fail(PFC_HIP_EUNSUPPORTED, "pfc_hip_pfc_set_operators: unknown model " +
                                          std::to_string(model_kind));
  if (model_kind == PFC_HIP_MODEL_PFC && (!params || nparams != 4))
    return fail(PFC_HIP_EINVAL,
                "pfc_hip_pfc_set_operators: PFC needs params {dx, dy, dz, eps}");
  if (model_kind == PFC_HIP_MODEL_TUNGSTEN && plan->batch > 1)
    return fail(PFC_HIP_EUNSUPPORTED,
                "pfc_hip_pfc_set_operators: batched plans run the PFC model only");
  if (model_kind == PFC_HIP_MODEL_TUNGSTEN && plan->xp)
    return fail(PFC_HIP_EUNSUPPORTED, "pfc_hip_pfc_set_operators: PFC_HIP_FLAG_F64_BUTTERFLIES "
                                      "plans run the PFC model only");
  if (model_kind == PFC_HIP_MODEL_TUNGSTEN && (!params || nparams != PFC_HIP_TUNGSTEN_NPARAMS))
    return fail(PFC_HIP_EINVAL,
                "pfc_hip_pfc_set_operators: Tungsten needs " +
                    std::to_string(PFC_HIP_TUNGSTEN_NPARAMS) + " params");
  if (model_kind == PFC_HIP_MODEL_PFC && !supported_len(plan->nx))
    return fail(PFC_HIP_EUNSUPPORTED,
                "pfc_hip_pfc_set_operators: nx unsupported for the fused step");
  const double dx = params[0], dy = params[1], dz = params[2];
  if (!(dx > 0) || !(dy > 0) || !(dz > 0) || !std::isfinite(dt))
    return fail(PFC_HIP_EINVAL, "pfc_hip_pfc_set_operators: bad spacing or dt");
  for (int i = 3; i < nparams; ++i)
    if (!std::isfinite(params[i]))
      return fail(PFC_HIP_EINVAL, "pfc_hip_pfc_set_operators: parameter " +
                                      std::to_string(i) + " is not finite");
  if (model_kind == PFC_HIP_MODEL_TUNGSTEN) {
    const double *q = params + 3;
    if (!(q[0] > 0) || !(q[1] > 0) || !(q[2] > 0) || q[6] == 0.0 || q[3] < 0 ||
        q[3] != std::floor(q[3]) || q[3] > 64)
      return fail(PFC_HIP_EINVAL,
                  "pfc_hip_pfc_set_operators: Tungsten needs alpha2 > 0, lambda2 > 0, "
                  "alpha_farTol > 0, T0 != 0 and an integer alpha_highOrd in [0, 64]");
  }
  if (int rc = set_device(plan)) return rc;
  // kspace.hpp:97-103: f = 2*pi/(d*n); the multipliers are evaluated per
  // mode in the z passes, scaled by the 1/(nx*ny*nz) of the backward transform.
  const double two_pi = 6.283185307179586;
  PfcOp o{};
  o.fx = two_pi / (dx * plan->nx);
  o.fy = two_pi / (dy * plan->ny);
  o.fz = two_pi / (dz * plan->nz);
  o.eps = model_kind == PFC_HIP_MODEL_PFC ? params[3] : 0.0;
  o.dt = dt;
  o.scale = 1.0 / ((double)plan->nx * (double)plan->ny * (double)plan->nz);
  o.nx = plan->nx;
  o.ny = plan->ny;
  o.nz = plan->nz;
  plan->op = o;
  plan->spacing[0] = dx;
  plan->spacing[1] = dy;
  plan->spacing[2] = dz;
  if (model_kind == PFC_HIP_MODEL_TUNGSTEN) {
    plan->top = tungsten_scalars(params + 3);
    for (int i = 0; i < 4; ++i) plan->tq[i] = params[13 + i]; // p3, p4, q3, q4
    plan->tq[4] = params[10];                                  // stabP
  }
  plan->model_kind = model_kind;
  if (plan->prec == PFC_HIP_F64)
    model_variants<double>(plan);
  else
    model_variants<float>(plan);
  if (int rc = step_buffers(plan)) return rc;
  plan->dt = dt;
  plan->ops_ready = true;
  ++plan->gen;
  return 0;
}

int pfc_hip_tungsten_operators(pfc_hip_plan_t plan, void *filterMF, void *expL,
                               void *nW, void *stream) {
  if (int rc = check_single(plan, "pfc_hip_tungsten_operators")) return rc;
  if (!filterMF || !expL || !nW)
    return fail(PFC_HIP_EINVAL, "pfc_hip_tungsten_operators: null buffer");
  if (!plan->ops_ready || !plan->tungsten())
    return fail(PFC_HIP_ESTATE, "pfc_hip_tungsten_operators: Tungsten operators not set");
  if (int rc = set_device(plan)) return rc;
  hipStream_t s = (hipStream_t)stream;
  const unsigned blocks = ic_blocks((long)plan->outbox());
  if (plan->prec == PFC_HIP_F64)
    hipLaunchKernelGGL(k_tung_operators<double>, dim3(blocks), dim3(256), 0, s,
                       plan->op, plan->top, plan->W, (double *)filterMF,
                       (double *)expL, (double *)nW);
  else
    hipLaunchKernelGGL(k_tung_operators<float>, dim3(blocks), dim3(256), 0, s,
                       plan->op, plan->top, plan->W, (float *)filterMF,
                       (float *)expL, (float *)nW);
  PFC_HIP_TRY(hipGetLastError(), "tungsten operator kernel launch");
  return 0;
}

int pfc_hip_pfc_operators(pfc_hip_plan_t plan, void *opL, void *opN,
                          void *stream) {
  if (int rc = check_single(plan, "pfc_hip_pfc_operators")) return rc;
  if (!opL || !opN) return fail(PFC_HIP_EINVAL, "pfc_hip_pfc_operators: null buffer");
  if (!plan->ops_ready || plan->tungsten())
    return fail(PFC_HIP_ESTATE, "pfc_hip_pfc_operators: PFC operators not set");
  if (int rc = set_device(plan)) return rc;
  hipStream_t s = (hipStream_t)stream;
  const unsigned blocks = ic_blocks((long)plan->outbox());
  if (plan->prec == PFC_HIP_F64)
    hipLaunchKernelGGL(k_pfc_operators<double>, dim3(blocks), dim3(256), 0, s,
                       plan->op, plan->W, (double *)opL, (double *)opN);
  else
    hipLaunchKernelGGL(k_pfc_operators<float>, dim3(blocks), dim3(256), 0, s,
                       plan->op, plan->W, (float *)opL, (float *)opN);
  PFC_HIP_TRY(hipGetLastError(), "operator kernel launch");
  return 0;
}

static int step_checks(pfc_hip_plan_t plan, void *psi, int nsteps, const char *fn) {
  if (int rc = check_plan(plan)) return rc;
  if (!psi) return fail(PFC_HIP_EINVAL, std::string(fn) + ": null psi");
  if (nsteps < 0) return fail(PFC_HIP_EINVAL, std::string(fn) + ": nsteps < 0");
  if (!plan->ops_ready)
    return fail(PFC_HIP_ESTATE, std::string(fn) +
                                    ": operators not set (call pfc_hip_pfc_set_operators)");
  if (plan->tungsten() && plan->mean_split)
    return fail(PFC_HIP_EUNSUPPORTED,
                std::string(fn) + ": the mean-split mode applies to the PFC model only");
  return set_device(plan);
}

int pfc_hip_pfc_step(pfc_hip_plan_t plan, void *psi, int nsteps, void *stream) {
  if (int rc = step_checks(plan, psi, nsteps, "pfc_hip_pfc_step")) return rc;
  hipStream_t s = (hipStream_t)stream;
  if (nsteps >= 2) {
    const bool f64 = plan->prec == PFC_HIP_F64;
    if (f64 ? fused_steps<double>(plan) : fused_steps<float>(plan)) {
      if (int rc = step_buffers(plan)) return rc;
      return f64 ? steps_fused<double>(plan, psi, nsteps, s, nullptr)
                 : steps_fused<float>(plan, psi, nsteps, s, nullptr);
    }
    if (f64 ? plane_steps<double>(plan) : plane_steps<float>(plan)) {
      if (int rc = step_buffers(plan)) return rc;
      return f64 ? steps_plane<double>(plan, psi, nsteps, s)
                 : steps_plane<float>(plan, psi, nsteps, s);
    }
  }
  for (int i = 0; i < nsteps; ++i) {
    int rc = plan->prec == PFC_HIP_F64 ? step_impl<double>(plan, psi, s, nullptr)
                                       : step_impl<float>(plan, psi, s, nullptr);
    if (rc) return rc;
  }
  return 0;
}

int pfc_hip_tungsten_step(pfc_hip_plan_t plan, void *psi, int nsteps, void *psiMF,
                          void *stream) {
  if (int rc = step_checks(plan, psi, nsteps, "pfc_hip_tungsten_step")) return rc;
  if (!plan->tungsten())
    return fail(PFC_HIP_ESTATE, "pfc_hip_tungsten_step: Tungsten operators not set");
  if (psiMF && psiMF == psi)
    return fail(PFC_HIP_EINVAL, "pfc_hip_tungsten_step: psiMF must not alias psi");
  hipStream_t s = (hipStream_t)stream;
  for (int i = 0; i < nsteps; ++i) {
    void *mf = (i == nsteps - 1) ? psiMF : nullptr;
    int rc = plan->prec == PFC_HIP_F64 ? step_impl<double>(plan, psi, s, nullptr, mf)
                                       : step_impl<float>(plan, psi, s, nullptr, mf);
    if (rc) return rc;
  }
  return 0;
}

int pfc_hip_pfc_adjoint_step(pfc_hip_plan_t plan, const void *psi_n, void *lambda,
                             double *dr, void *stream) {
  if (int rc = check_single(plan, "pfc_hip_pfc_adjoint_step")) return rc;
  if (!psi_n || !lambda) return fail(PFC_HIP_EINVAL, "pfc_hip_pfc_adjoint_step: null field");
  if (psi_n == lambda)
    return fail(PFC_HIP_EINVAL, "pfc_hip_pfc_adjoint_step: lambda must not alias psi_n");
  if (!plan->ops_ready || plan->model_kind != PFC_HIP_MODEL_PFC)
    return fail(PFC_HIP_ESTATE, "pfc_hip_pfc_adjoint_step: PFC operators not set");
  if (int rc = set_device(plan)) return rc;
  hipStream_t s = (hipStream_t)stream;
  return plan->prec == PFC_HIP_F64 ? adjoint_f64(plan, psi_n, lambda, dr, s)
                                   : adjoint_f32(plan, psi_n, lambda, dr, s);
}

int pfc_hip_pfc_free_energy(pfc_hip_plan_t plan, const void *psi, double *F, void *stream) {
  if (int rc = check_single(plan, "pfc_hip_pfc_free_energy")) return rc;
  if (!psi || !F) return fail(PFC_HIP_EINVAL, "pfc_hip_pfc_free_energy: null argument");
  if (!plan->ops_ready || plan->model_kind != PFC_HIP_MODEL_PFC)
    return fail(PFC_HIP_ESTATE, "pfc_hip_pfc_free_energy: PFC operators not set");
  if (int rc = set_device(plan)) return rc;
  hipStream_t s = (hipStream_t)stream;
  return plan->prec == PFC_HIP_F64 ? free_energy_impl<double>(plan, psi, F, s)
                                   : free_energy_impl<float>(plan, psi, F, s);
}

int pfc_hip_stream_copy(const void *src, void *dst, size_t bytes, void *stream) {
  if (!src || !dst) return fail(PFC_HIP_EINVAL, "pfc_hip_stream_copy: null pointer");
  if (bytes % 16 || (uintptr_t)src % 16 || (uintptr_t)dst % 16)
    return fail(PFC_HIP_EINVAL, "pfc_hip_stream_copy: bytes and pointers must be 16-byte multiples");
  const char *a = (const char *)src, *b = (const char *)dst;
  if (a < b + bytes && b < a + bytes)
    return fail(PFC_HIP_EINVAL, "pfc_hip_stream_copy: src and dst overlap");
  const size_t n = bytes / 16;
  if (n == 0) return 0;
  const size_t blocks = (n + 255) / 256;
  if (blocks > 0x7fffffffu) return fail(PFC_HIP_EINVAL, "pfc_hip_stream_copy: too large");
  hipLaunchKernelGGL(k_stream_copy, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     (const uint4 *)src, (uint4 *)dst, n);
  PFC_HIP_TRY(hipGetLastError(), "pfc_hip_stream_copy");
  return 0;
}

int pfc_hip_pfc_step_timed(pfc_hip_plan_t plan, void *psi, int nsteps,
                           void *stream, double *kernel_ms, int nkernels) {
  if (int rc = step_checks(plan, psi, nsteps, "pfc_hip_pfc_step_timed")) return rc;
  const int np = plan->step_passes();
  if (!kernel_ms || nkernels < np)
    return fail(PFC_HIP_EINVAL, "pfc_hip_pfc_step_timed: kernel_ms needs " +
                                    std::to_string(np) + " entries");
  if (nsteps < 1) return fail(PFC_HIP_EINVAL, "pfc_hip_pfc_step_timed: nsteps < 1");
  hipStream_t s = (hipStream_t)stream;
  const bool f64 = plan->prec == PFC_HIP_F64;
  // with a sixth entry and a fused run: the launches of pfc_hip_pfc_step, whose
  // field 0 remakes its spectrum every `span` steps
  const bool fused = nkernels >= 6 && nsteps >= 2 &&
                     (f64 ? fused_steps<double>(plan) : fused_steps<float>(plan));
  const int span = !fused ? 1
                   : f64  ? fused_span(pfc_t_args<double>(plan, psi, 0).op)
                          : fused_span(pfc_t_args<float>(plan, psi, 0).op);
  const int ne = fused ? fused_events(nsteps, span) : (np + 1) * nsteps;
  std::vector<hipEvent_t> ev((size_t)ne, nullptr);
  int rc = 0;
  for (auto &e : ev) {
    hipError_t he = hipEventCreate(&e);
    if (he != hipSuccess) {
      e = nullptr;
      rc = fail(PFC_HIP_EDEVICE, std::string("hipEventCreate: ") + hipGetErrorString(he));
      break;
    }
  }
  if (!rc && fused) {
    rc = step_buffers(plan);
    if (!rc)
      rc = f64 ? steps_fused<double>(plan, psi, nsteps, s, ev.data())
               : steps_fused<float>(plan, psi, nsteps, s, ev.data());
  } else if (!rc) {
    const int pe = np + 1;
    for (int i = 0; i < nsteps && !rc; ++i)
      rc = f64 ? step_impl<double>(plan, psi, s, &ev[(size_t)pe * i])
               : step_impl<float>(plan, psi, s, &ev[(size_t)pe * i]);
  }
  if (!rc) {
    hipError_t e = hipStreamSynchronize(s);
    if (e != hipSuccess) rc = fail(PFC_HIP_EDEVICE, hipGetErrorString(e));
  }
  auto launch_ms = [&](size_t i) {
    float ms = 0;
    (void)hipEventElapsedTime(&ms, ev[i], ev[i + 1]);
    return (double)ms;
  };
  if (!rc && fused) {
    // launch j of step i of a run is the run's interval 4*i + j; its exit the last.
    // Steps after the first of their run are alike; runs of one step have none.
    const int runs = (nsteps + span - 1) / span;
    const int steady = nsteps - runs, first = steady ? 1 : 0, nmid = steady ? steady : nsteps;
    for (int k = 0; k < 6; ++k) kernel_ms[k] = 0;
    size_t base = 0;
    for (int done = 0; done < nsteps;) {
      const int n = std::min(span, nsteps - done);
      kernel_ms[0] += launch_ms(base) / runs;
      for (int i = first; i < n; ++i) {
        if (i > 0) kernel_ms[5] += launch_ms(base + 4 * i) / steady;
        for (int k = 1; k <= 3; ++k) kernel_ms[k] += launch_ms(base + 4 * i + k) / nmid;
      }
      kernel_ms[4] += launch_ms(base + 4 * n) / runs;
      base += 4 * n + 1;
      done += n;
    }
  } else if (!rc) {
    const int pe = np + 1;
    for (int k = 0; k < np; ++k) kernel_ms[k] = 0;
    for (int i = 0; i < nsteps; ++i)
      for (int k = 0; k < np; ++k) kernel_ms[k] += launch_ms((size_t)pe * i + k) / nsteps;
    if (nkernels > np) kernel_ms[np] = 0;
  }
  for (auto &e : ev)
    if (e) (void)hipEventDestroy(e);
  return rc;
}

int pfc_hip_ic_constant(pfc_hip_plan_t plan, void *psi, double value,
                        void *stream) {
  if (int rc = check_single(plan, "pfc_hip_ic_constant")) return rc;
  if (!psi) return fail(PFC_HIP_EINVAL, "pfc_hip_ic_constant: null psi");
  if (int rc = set_device(plan)) return rc;
  const long n = (long)plan->inbox();
  hipStream_t s = (hipStream_t)stream;
  if (plan->prec == PFC_HIP_F64)
    hipLaunchKernelGGL(k_ic_constant<double>, dim3(ic_blocks(n)), dim3(256),
                       0, s, (double *)psi, n, value);
  else
    hipLaunchKernelGGL(k_ic_constant<float>, dim3(ic_blocks(n)), dim3(256), 0,
                       s, (float *)psi, n, value);
  PFC_HIP_TRY(hipGetLastError(), "ic_constant launch");
  return 0;
}

int pfc_hip_ic_single_seed(pfc_hip_plan_t plan, void *psi, const double *origin3,
                           const double *spacing3, double rho, double amp,
                           double radius, int keep_outside, void *stream) {
  if (int rc = check_single(plan, "pfc_hip_ic_single_seed")) return rc;
  if (!psi || !origin3 || !spacing3)
    return fail(PFC_HIP_EINVAL, "pfc_hip_ic_single_seed: null argument");
  if (int rc = set_device(plan)) return rc;
  SeedArgs a{};
  a.x0 = origin3[0];
  a.y0 = origin3[1];
  a.z0 = origin3[2];
  a.dx = spacing3[0];
  a.dy = spacing3[1];
  a.dz = spacing3[2];
  a.rho = rho;
  a.amp = amp;
  a.r2 = radius * radius;
  a.nx = plan->nx;
  a.ny = plan->ny;
  a.nz = plan->nz;
  a.keep_outside = keep_outside ? 1 : 0;
  const long n = (long)plan->inbox();
  hipStream_t s = (hipStream_t)stream;
  if (plan->prec == PFC_HIP_F64)
    hipLaunchKernelGGL(k_ic_single_seed<double>, dim3(ic_blocks(n)),
                       dim3(256), 0, s, (double *)psi, a);
  else
    hipLaunchKernelGGL(k_ic_single_seed<float>, dim3(ic_blocks(n)), dim3(256),
                       0, s, (float *)psi, a);
  PFC_HIP_TRY(hipGetLastError(), "ic_single_seed launch");
  return 0;
}

int pfc_hip_ic_add_noise(pfc_hip_plan_t plan, void *psi, unsigned long long seed,
                         double lo, double hi, void *stream) {
  if (int rc = check_single(plan, "pfc_hip_ic_add_noise")) return rc;
  if (!psi) return fail(PFC_HIP_EINVAL, "pfc_hip_ic_add_noise: null psi");
  if (int rc = set_device(plan)) return rc;
  const long n = (long)plan->inbox();
  hipStream_t s = (hipStream_t)stream;
  if (plan->prec == PFC_HIP_F64)
    hipLaunchKernelGGL(k_ic_add_noise<double>, dim3(ic_blocks(n)), dim3(256),
                       0, s, (double *)psi, n, seed, lo, hi);
  else
    hipLaunchKernelGGL(k_ic_add_noise<float>, dim3(ic_blocks(n)), dim3(256), 0,
                       s, (float *)psi, n, seed, lo, hi);
  PFC_HIP_TRY(hipGetLastError(), "ic_add_noise launch");
  return 0;
}

int pfc_hip_bc_fixed(pfc_hip_plan_t plan, void *psi, double x0, double dx, double rho_low,
                     double rho_high, double xwidth, double alpha, void *stream) {
  if (int rc = check_single(plan, "pfc_hip_bc_fixed")) return rc;
  if (!psi) return fail(PFC_HIP_EINVAL, "pfc_hip_bc_fixed: null psi");
  if (!std::isfinite(x0) || !std::isfinite(dx) || !std::isfinite(xwidth) ||
      !std::isfinite(alpha))
    return fail(PFC_HIP_EINVAL, "pfc_hip_bc_fixed: non-finite geometry");
  if (int rc = set_device(plan)) return rc;
  FixedBcArgs a{};
  a.x0 = x0;
  a.dx = dx;
  a.xwidth = xwidth;
  a.alpha = alpha;
  a.rho_low = rho_low;
  a.rho_high = rho_high;
  {
#pragma clang fp contract(off)
    a.xpos = ((double)plan->nx * dx) - xwidth; // fixed_bc.hpp: (Lx * dx) - xwidth
  }
  a.nx = plan->nx;
  a.rows = (long)plan->ny * plan->nz;
  const long n = (long)plan->inbox();
  hipStream_t s = (hipStream_t)stream;
  if (plan->prec == PFC_HIP_F64)
    hipLaunchKernelGGL(k_bc_fixed<double>, dim3(ic_blocks(n)), dim3(256), 0, s,
                       (double *)psi, a);
  else
    hipLaunchKernelGGL(k_bc_fixed<float>, dim3(ic_blocks(n)), dim3(256), 0, s,
                       (float *)psi, a);
  PFC_HIP_TRY(hipGetLastError(), "bc_fixed launch");
  return 0;
}

int pfc_hip_ic_seeds(pfc_hip_plan_t plan, void *psi, const double *origin3,
                     const double *spacing3, const double *seeds, int nseeds, int keep_outside,
                     void *stream) {
  if (int rc = check_single(plan, "pfc_hip_ic_seeds")) return rc;
  if (!psi || !origin3 || !spacing3 || (nseeds > 0 && !seeds))
    return fail(PFC_HIP_EINVAL, "pfc_hip_ic_seeds: null argument");
  if (nseeds < 0) return fail(PFC_HIP_EINVAL, "pfc_hip_ic_seeds: nseeds < 0");
  for (int d = 0; d < 3; ++d)
    if (!std::isfinite(origin3[d]) || !(spacing3[d] > 0) || !std::isfinite(spacing3[d]))
      return fail(PFC_HIP_EINVAL, "pfc_hip_ic_seeds: non-finite origin or spacing");
  for (long v = 0; v < 24L * nseeds; ++v)
    if (!std::isfinite(seeds[v]))
      return fail(PFC_HIP_EINVAL, "pfc_hip_ic_seeds: non-finite seed value");
  if (int rc = set_device(plan)) return rc;
  hipStream_t s = (hipStream_t)stream;
  const bool f64 = plan->prec == PFC_HIP_F64;
  if (!keep_outside) {
    const long n = (long)plan->inbox();
    if (f64)
      hipLaunchKernelGGL(k_ic_constant<double>, dim3(ic_blocks(n)), dim3(256), 0, s,
                         (double *)psi, n, 0.0);
    else
      hipLaunchKernelGGL(k_ic_constant<float>, dim3(ic_blocks(n)), dim3(256), 0, s,
                         (float *)psi, n, 0.0);
    PFC_HIP_TRY(hipGetLastError(), "ic_seeds clear");
  }
  const int ext[3] = {plan->nx, plan->ny, plan->nz};
  // last seed first: the first seed holding a point writes it last
  for (int sd = nseeds - 1; sd >= 0; --sd) {
    const double *v = seeds + 24L * sd;
    SeedBoxArgs a{};
    a.x0 = origin3[0];
    a.y0 = origin3[1];
    a.z0 = origin3[2];
    a.dx = spacing3[0];
    a.dy = spacing3[1];
    a.dz = spacing3[2];
    for (int d = 0; d < 3; ++d) a.loc[d] = v[d];
    for (int q = 0; q < 18; ++q) a.q[q] = v[3 + q];
    a.rho = v[21];
    a.r2 = v[22] * v[22];
    a.amp = v[23];
    a.nx = plan->nx;
    a.ny = plan->ny;
    // index box of the sphere, one point of margin each side, clipped
    int lo[3], hi[3];
    bool empty = false;
    for (int d = 0; d < 3; ++d) {
      const double r = std::fabs(v[22]);
      const double f0 = std::floor((v[d] - r - origin3[d]) / spacing3[d]) - 1.0;
      const double f1 = std::ceil((v[d] + r - origin3[d]) / spacing3[d]) + 1.0;
      lo[d] = (int)std::max(0.0, std::min(f0, (double)ext[d]));
      hi[d] = (int)std::min((double)ext[d] - 1.0, std::max(f1, -1.0));
      if (hi[d] < lo[d]) empty = true;
    }
    if (empty) continue;
    a.i0 = lo[0];
    a.j0 = lo[1];
    a.k0 = lo[2];
    a.bx = hi[0] - lo[0] + 1;
    a.by = hi[1] - lo[1] + 1;
    a.nbox = (long)a.bx * a.by * (hi[2] - lo[2] + 1);
    if (f64)
      hipLaunchKernelGGL(k_ic_seed_box<double>, dim3(ic_blocks(a.nbox)), dim3(256), 0, s,
                         (double *)psi, a);
    else
      hipLaunchKernelGGL(k_ic_seed_box<float>, dim3(ic_blocks(a.nbox)), dim3(256), 0, s,
                         (float *)psi, a);
    PFC_HIP_TRY(hipGetLastError(), "ic_seeds launch");
  }
  return 0;
}

int pfc_hip_column_max(pfc_hip_plan_t plan, const void *psi, double *xline, void *stream) {
  if (int rc = check_single(plan, "pfc_hip_column_max")) return rc;
  if (!psi || !xline) return fail(PFC_HIP_EINVAL, "pfc_hip_column_max: null argument");
  if (int rc = set_device(plan)) return rc;
  const int nx = plan->nx;
  const long rows = (long)plan->ny * plan->nz;
  const int parts = (int)std::min<long>(rows, kColParts);
  if (int rc = dalloc(plan, &plan->colmax, ((size_t)kColParts + 1) * nx * sizeof(double),
                      "column maxima"))
    return rc;
  double *part = (double *)plan->colmax;
  double *out = part + (size_t)kColParts * nx;
  hipStream_t s = (hipStream_t)stream;
  const unsigned gx = (unsigned)((nx + 255) / 256);
  if (plan->prec == PFC_HIP_F64)
    hipLaunchKernelGGL(k_column_max_part<double>, dim3(gx, (unsigned)parts), dim3(256), 0, s,
                       (const double *)psi, nx, rows, part);
  else
    hipLaunchKernelGGL(k_column_max_part<float>, dim3(gx, (unsigned)parts), dim3(256), 0, s,
                       (const float *)psi, nx, rows, part);
  PFC_HIP_TRY(hipGetLastError(), "column max (partials)");
  hipLaunchKernelGGL(k_column_max_final, dim3((unsigned)((nx + kMaxCols - 1) / kMaxCols)),
                     dim3(kMaxCols * kMaxSlices), 0, s, (const double *)part, nx,
                     parts, out);
  PFC_HIP_TRY(hipGetLastError(), "column max (final)");
  PFC_HIP_TRY(hipMemcpyAsync(xline, out, (size_t)nx * sizeof(double), hipMemcpyDeviceToHost, s),
              "column max copy");
  PFC_HIP_TRY(hipStreamSynchronize(s), "column max sync");
  return 0;
}

// The same maxima without allocating: partials in the library's static
// scratch, result in the caller's device buffer, nothing waited for.
int pfc_hip_column_max_noalloc(pfc_hip_plan_t plan, const void *psi, double *xline_dev,
                               void *stream) {
  if (int rc = check_single(plan, "pfc_hip_column_max_noalloc")) return rc;
  if (!psi || !xline_dev)
    return fail(PFC_HIP_EINVAL, "pfc_hip_column_max_noalloc: null argument");
  const int nx = plan->nx;
  const long rows = (long)plan->ny * plan->nz;
  const int parts = (int)std::min<long>(rows, kColParts);
  if ((long)parts * nx > kColScratch)
    return fail(PFC_HIP_EINVAL, "pfc_hip_column_max_noalloc: nx = " + std::to_string(nx) +
                                    " needs " + std::to_string((long)parts * nx) +
                                    " doubles of scratch, more than its " +
                                    std::to_string(kColScratch) + " (nx <= " +
                                    std::to_string(kColScratch / kColParts) + ")");
  if (int rc = set_device(plan)) return rc;
  double *part = nullptr;
  if (int rc = col_scratch(plan->device, &part)) return rc;
  hipStream_t s = (hipStream_t)stream;
  const unsigned gx = (unsigned)((nx + 255) / 256);
  if (plan->prec == PFC_HIP_F64)
    hipLaunchKernelGGL(k_column_max_part<double>, dim3(gx, (unsigned)parts), dim3(256), 0, s,
                       (const double *)psi, nx, rows, part);
  else
    hipLaunchKernelGGL(k_column_max_part<float>, dim3(gx, (unsigned)parts), dim3(256), 0, s,
                       (const float *)psi, nx, rows, part);
  PFC_HIP_TRY(hipGetLastError(), "column max (partials)");
  hipLaunchKernelGGL(k_column_max_final, dim3((unsigned)((nx + kMaxCols - 1) / kMaxCols)),
                     dim3(kMaxCols * kMaxSlices), 0, s, (const double *)part, nx,
                     parts, xline_dev);
  PFC_HIP_TRY(hipGetLastError(), "column max (final)");
  return 0;
}

int pfc_hip_bc_moving(pfc_hip_plan_t plan, void *psi, double x0, double dx, double xpos,
                      double rho_low, double rho_high, double xwidth, double alpha,
                      void *stream) {
  if (int rc = check_single(plan, "pfc_hip_bc_moving")) return rc;
  if (!psi) return fail(PFC_HIP_EINVAL, "pfc_hip_bc_moving: null psi");
  if (!std::isfinite(x0) || !std::isfinite(dx) || !(dx > 0) || !std::isfinite(xpos) ||
      !std::isfinite(xwidth) || !std::isfinite(alpha))
    return fail(PFC_HIP_EINVAL, "pfc_hip_bc_moving: non-finite geometry");
  if (int rc = set_device(plan)) return rc;
  MovingBcArgs a{};
  a.x0 = x0;
  a.dx = dx;
  a.xwidth = xwidth;
  a.alpha = alpha;
  a.rho_low = rho_low;
  a.rho_high = rho_high;
  a.nx = plan->nx;
  {
#pragma clang fp contract(off)
    const double Lx = (double)plan->nx;
    a.l = Lx * dx;                 // moving_bc.hpp: l = Lx * dx
    a.xpos = std::fmod(xpos, a.l); // xpos = fmod(m_xpos, l)
  }
  // the columns in a band, by the kernel's own test (host and device round
  // these few operations identically)
  int first = -1, last = -1;
  for (int i = 0; i < plan->nx; ++i) {
#pragma clang fp contract(off)
    const double x = (x0 + ((double)i * dx));
    const double dist = x - a.xpos;
    const bool in = std::fabs(dist) < xwidth ||
                    (a.xpos < xwidth && std::fabs(dist - a.l) < xwidth) ||
                    (a.xpos > a.l - xwidth && std::fabs(dist + a.l) < xwidth);
    if (in) {
      if (first < 0) first = i;
      last = i;
    }
  }
  if (first < 0) return 0;
  a.i0 = first;
  a.bx = last - first + 1;
  a.nbox = (long)a.bx * plan->ny * plan->nz;
  hipStream_t s = (hipStream_t)stream;
  if (plan->prec == PFC_HIP_F64)
    hipLaunchKernelGGL(k_bc_moving<double>, dim3(ic_blocks(a.nbox)), dim3(256), 0, s,
                       (double *)psi, a);
  else
    hipLaunchKernelGGL(k_bc_moving<float>, dim3(ic_blocks(a.nbox)), dim3(256), 0, s,
                       (float *)psi, a);
  PFC_HIP_TRY(hipGetLastError(), "bc_moving launch");
  return 0;
}

// ---------------------------------------------------------------------------
// Launch variants and autotuning.
// ---------------------------------------------------------------------------
int pfc_hip_variant_count(pfc_hip_plan_t plan, int role, int *count) {
  if (int rc = check_plan(plan)) return rc;
  if (!count || role < 0 || role >= ROLE_COUNT)
    return fail(PFC_HIP_EINVAL, "pfc_hip_variant_count: bad role or null count");
  *count = plan->prec == PFC_HIP_F64 ? variant_count<double>(plan, role)
                                     : variant_count<float>(plan, role);
  return 0;
}

const char *pfc_hip_variant_name(pfc_hip_plan_t plan, int role, int index) {
  if (!plan || role < 0 || role >= ROLE_COUNT) return nullptr;
  const std::string *n = plan->prec == PFC_HIP_F64
                             ? variant_name<double>(plan, role, index)
                             : variant_name<float>(plan, role, index);
  return n ? n->c_str() : nullptr;
}

int pfc_hip_variant_get(pfc_hip_plan_t plan, int role, int *index) {
  if (int rc = check_plan(plan)) return rc;
  if (!index || role < 0 || role >= ROLE_COUNT)
    return fail(PFC_HIP_EINVAL, "pfc_hip_variant_get: bad role or null index");
  *index = plan->var[role];
  return 0;
}

int pfc_hip_variant_set(pfc_hip_plan_t plan, int role, int index) {
  if (int rc = check_plan(plan)) return rc;
  if (role < 0 || role >= ROLE_COUNT)
    return fail(PFC_HIP_EINVAL, "pfc_hip_variant_set: bad role");
  int count = 0;
  pfc_hip_variant_count(plan, role, &count);
  if (index < 0 || index >= count)
    return fail(PFC_HIP_EINVAL, "pfc_hip_variant_set: index " + std::to_string(index) +
                                    " out of range (" + std::to_string(count) +
                                    " variants)");
  if (role == ROLE_STEP_LAYOUT && index != plan->var[role]) {
    if (int rc = set_device(plan)) return rc;
    (void)hipDeviceSynchronize();
    void **drop[4] = {&plan->A1, &plan->B1, &plan->A2, &plan->B2};
    void **drop_nat[3] = {&plan->A, &plan->B, &plan->C};
    const size_t tb = plan->outbox() * 2 * plan->esize;
    const size_t nb = plan->padded() * 2 * plan->esize * plan->batch;
    if (index == 1) {
      for (void **b : drop)
        if (*b) { (void)hipFree(*b); *b = nullptr; plan->bytes -= tb; }
    } else {
      for (void **b : drop_nat)
        if (*b) { (void)hipFree(*b); *b = nullptr; plan->bytes -= nb; }
    }
  }
  if (plan->var[role] != index) ++plan->gen;
  plan->var[role] = index;
  plan->chosen[role] = true;
  if ((role == ROLE_STEP_LAYOUT || plane_role(role)) && plan->ops_ready)
    return step_buffers(plan);
  return 0;
}

int pfc_hip_pfc_autotune(pfc_hip_plan_t plan, void *psi, int reps, void *stream,
                         double *times_ms, int max_times) {
  if (int rc = check_plan(plan)) return rc;
  if (!psi || reps < 1)
    return fail(PFC_HIP_EINVAL, "pfc_hip_pfc_autotune: null psi or reps < 1");
  if (!plan->ops_ready)
    return fail(PFC_HIP_ESTATE, "pfc_hip_pfc_autotune: operators not set");
  if (int rc = set_device(plan)) return rc;
  hipStream_t s = (hipStream_t)stream;
  // psi is restored at the end from the c2r workspace (outbox complex >= inbox real)
  if (int rc = dalloc(plan, &plan->work, plan->outbox() * 2 * plan->esize * plan->batch,
                      "c2r workspace"))
    return rc;
  const size_t rbytes = plan->inbox() * plan->esize * plan->batch;
  PFC_HIP_TRY(hipMemcpyAsync(plan->work, psi, rbytes, hipMemcpyDeviceToDevice, s),
              "autotune backup");
  const int np = plan->step_passes();
  std::vector<hipEvent_t> ev((size_t)np + 1, nullptr);
  int rc = 0;
  for (auto &e : ev) {
    hipError_t he = hipEventCreate(&e);
    if (he != hipSuccess) {
      e = nullptr;
      rc = fail(PFC_HIP_EDEVICE, std::string("hipEventCreate: ") + hipGetErrorString(he));
      break;
    }
  }
  // Tuned roles in slot order, with the passes (bit k = pass k of the step)
  // their kernels occupy; the last two slots receive each layout's step time.
  struct RoleSpan { int role, layout; unsigned passes; };
  static const RoleSpan pfc_spans[] = {
      {ROLE_PFC_X, 1, 0x1},   {ROLE_COL_Y, 1, 0xA},    {ROLE_PFC_Z, 1, 0x4},
      {ROLE_X_C2R, 1, 0x10},  {ROLE_T_X_FWD, 0, 0x1},  {ROLE_T_Y_FWD, 0, 0x2},
      {ROLE_T_Z, 0, 0x4},     {ROLE_T_Y_INV, 0, 0x8},  {ROLE_T_X_INV, 0, 0x10}};
  static const RoleSpan tung_spans[] = {
      {ROLE_X_R2C, 1, 0x1},   {ROLE_COL_Y, 1, 0xAA},   {ROLE_PFC_Z, 1, 0x44},
      {ROLE_X_TUNG, 1, 0x10}, {ROLE_X_C2R, 1, 0x100},  {ROLE_T_X_R2C, 0, 0x1},
      {ROLE_T_Y_FWD, 0, 0x22}, {ROLE_T_Z, 0, 0x44},    {ROLE_T_Y_INV, 0, 0x88},
      {ROLE_T_X_TUNG, 0, 0x10}, {ROLE_T_X_INV, 0, 0x100}};
  const RoleSpan *spans = plan->tungsten() ? tung_spans : pfc_spans;
  const int nspans = plan->tungsten() ? (int)(sizeof(tung_spans) / sizeof(RoleSpan))
                                      : (int)(sizeof(pfc_spans) / sizeof(RoleSpan));
  auto run_step = [&](double *pass_ms) -> int {
    int r = plan->prec == PFC_HIP_F64 ? step_impl<double>(plan, psi, s, ev.data())
                                      : step_impl<float>(plan, psi, s, ev.data());
    if (r) return r;
    hipError_t he = hipEventSynchronize(ev[np]);
    if (he != hipSuccess) return fail(PFC_HIP_EDEVICE, hipGetErrorString(he));
    for (int k = 0; k < np; ++k) {
      float ms = 0;
      (void)hipEventElapsedTime(&ms, ev[k], ev[k + 1]);
      pass_ms[k] = ms;
    }
    return 0;
  };
  auto span_ms = [&](const double *pm, unsigned passes) {
    double t = 0;
    for (int k = 0; k < np; ++k)
      if (passes & (1u << k)) t += pm[k];
    return t;
  };
  auto row_variants = [&](int role) {
    return plan->prec == PFC_HIP_F64 ? row_variant_count<double>(plan, role)
                                     : row_variant_count<float>(plan, role);
  };
  // time of one multi-step call (sets rc)
  auto run_ms_of = [&](int n) -> double {
    float ms = 0;
    hipError_t he = hipEventRecord(ev[0], s);
    if (he == hipSuccess) rc = pfc_hip_pfc_step(plan, psi, n, s);
    if (rc) return 1e300;
    if (he == hipSuccess) he = hipEventRecord(ev[1], s);
    if (he == hipSuccess) he = hipEventSynchronize(ev[1]);
    if (he == hipSuccess) he = hipEventElapsedTime(&ms, ev[0], ev[1]);
    if (he != hipSuccess)
      rc = fail(PFC_HIP_EDEVICE, std::string("autotune run: ") + hipGetErrorString(he));
    return rc ? 1e300 : (double)ms;
  };
  int slot = 0;
  double layout_ms[2] = {0, 0};
  // both layouts when the plan has both (natural first, slot order); a
  // double-butterfly plan has the transposed one only
  const bool two = plan->t_ok && !plan->xp;
  const int layouts = two ? 2 : 1;
  for (int li = 0; li < layouts && !rc; ++li) {
    const int layout = two ? 1 - li : (plan->t_ok ? 0 : 1);
    rc = pfc_hip_variant_set(plan, ROLE_STEP_LAYOUT, two ? layout : 0);
    // the row kernels of the natural layout are tuned first (with the y passes
    // they need), the plane kernels set against them below
    int plane_slot[ROLE_COUNT];
    for (int &ps : plane_slot) ps = -1;
    for (int si = 0; si < nspans; ++si)
      if (spans[si].layout == layout && plane_role(spans[si].role) &&
          plan->var[spans[si].role] >= row_variants(spans[si].role))
        plan->var[spans[si].role] = 0;
    for (int si = 0; si < nspans && !rc; ++si) {
      const RoleSpan &sp = spans[si];
      if (sp.layout != layout) continue;
      int count = 0;
      pfc_hip_variant_count(plan, sp.role, &count);
      if (plane_role(sp.role) && count > row_variants(sp.role)) {
        --count;
        plane_slot[sp.role] = slot + count;
        if (times_ms && slot + count < max_times) times_ms[slot + count] = 0.0;
      }
      // Each variant is scored by its fastest rep (interference only adds
      // time); the kTop best are then timed again, round-robin, so that a
      // drift of the clock over the sweep cannot decide between close ones.
      std::vector<double> score((size_t)count, 1e300);
      auto time_variant = [&](int v) {
        plan->var[sp.role] = v;
        double pm[9];
        for (int r = 0; r <= reps && !rc; ++r) { // r == 0 warms up
          rc = run_step(pm);
          if (!rc && r > 0) score[(size_t)v] = std::min(score[(size_t)v], span_ms(pm, sp.passes));
        }
      };
      for (int v = 0; v < count && !rc; ++v) time_variant(v);
      constexpr int kTop = 3;
      std::vector<int> order((size_t)count);
      for (int v = 0; v < count; ++v) order[(size_t)v] = v;
      std::stable_sort(order.begin(), order.end(),
                       [&](int a, int b) { return score[(size_t)a] < score[(size_t)b]; });
      const int top = std::min(kTop, count);
      for (int round = 0; round < 2 && top > 1 && !rc; ++round)
        for (int i = 0; i < top && !rc; ++i) time_variant(order[(size_t)i]);
      int best_v = plan->var[sp.role];
      double best = 1e300;
      for (int v = 0; v < count; ++v) {
        const int idx = slot + v;
        if (times_ms && idx < max_times) times_ms[idx] = score[(size_t)v];
        if (score[(size_t)v] < best) {
          best = score[(size_t)v];
          best_v = v;
        }
      }
      plan->var[sp.role] = best_v;
      slot += count + (plane_slot[sp.role] >= 0 ? 1 : 0);
    }
    // The plane kernels against the tuned row and column kernels, by the time
    // of whole multi-step runs (PFC runs fuse the step boundary when both
    // directions are on them, which no single pass shows): the best of every
    // combination over the roles, starting from all on.
    std::vector<int> pr, row_best;
    for (int si = 0; si < nspans; ++si)
      if (spans[si].layout == layout && plane_slot[spans[si].role] >= 0) {
        pr.push_back(spans[si].role);
        row_best.push_back(plan->var[spans[si].role]);
      }
    if (!rc && !pr.empty()) {
      constexpr int kRun = 4;
      double best = 1e300;
      unsigned best_mask = 0;
      auto apply = [&](unsigned mask) {
        for (size_t i = 0; i < pr.size(); ++i)
          plan->var[pr[i]] = (mask >> i & 1) ? row_variants(pr[i]) : row_best[i];
      };
      for (unsigned m = 1u << pr.size(); m-- > 0 && !rc;) {
        apply(m);
        double t = 1e300;
        for (int r = 0; r <= reps && !rc; ++r) {
          const double ms = run_ms_of(kRun);
          if (r > 0) t = std::min(t, ms / kRun);
        }
        for (size_t i = 0; i < pr.size(); ++i) // reported: the fastest step with the role on
          if ((m >> i & 1) && times_ms && plane_slot[pr[i]] < max_times) {
            double &w = times_ms[plane_slot[pr[i]]];
            w = w > 0 ? std::min(w, t) : t;
          }
        if (t < best) {
          best = t;
          best_mask = m;
        }
      }
      apply(best_mask);
    }
    if (!rc && layout == 0 && !plan->tungsten()) {
      // the fused step boundary of multi-step runs, timed on its own: each
      // variant starts from the T1 spectrum a full step leaves (the pass
      // rewrites T1 in place), one warm-up launch, then `reps` timed ones
      int count = 0;
      pfc_hip_variant_count(plan, ROLE_T_X_FUSE, &count);
      double best = 1e300;
      int best_v = plan->var[ROLE_T_X_FUSE];
      for (int v = 0; v < count && !rc; ++v) {
        plan->var[ROLE_T_X_FUSE] = v;
        double pm[9], fastest = 1e300;
        rc = run_step(pm);
        for (int r = 0; r <= reps && !rc; ++r) {
          hipError_t he = hipEventRecord(ev[0], s);
          if (he != hipSuccess) {
            rc = fail(PFC_HIP_EDEVICE, std::string("autotune event: ") + hipGetErrorString(he));
            break;
          }
          rc = plan->prec == PFC_HIP_F64
                   ? t_pass<double>(plan, pfc_t_args<double>(plan, psi), 5, s)
                   : t_pass<float>(plan, pfc_t_args<float>(plan, psi), 5, s);
          if (rc) break;
          he = hipEventRecord(ev[1], s);
          if (he == hipSuccess) he = hipEventSynchronize(ev[1]);
          if (he != hipSuccess) {
            rc = fail(PFC_HIP_EDEVICE, std::string("autotune sync: ") + hipGetErrorString(he));
            break;
          }
          float ms = 0;
          (void)hipEventElapsedTime(&ms, ev[0], ev[1]);
          if (r > 0) fastest = std::min(fastest, (double)ms);
        }
        if (times_ms && slot + v < max_times) times_ms[slot + v] = fastest;
        if (fastest < best) {
          best = fastest;
          best_v = v;
        }
      }
      plan->var[ROLE_T_X_FUSE] = best_v;
      slot += count;
      // kept-spectrum runs against single steps, by the time of whole runs
      double run_ms[2] = {1e300, 1e300};
      for (int fuse = 0; fuse < 2 && count > 0 && !rc; ++fuse) {
        plan->var[ROLE_STEP_FUSE] = fuse;
        for (int r = 0; r <= reps && !rc; ++r) {
          const double ms = run_ms_of(6);
          if (r > 0) run_ms[fuse] = std::min(run_ms[fuse], ms);
        }
      }
      if (count > 0) plan->var[ROLE_STEP_FUSE] = run_ms[1] < run_ms[0] ? 1 : 0;
    }
    double fastest = 1e300, pm[9];
    for (int r = 0; r <= reps && !rc; ++r) {
      rc = run_step(pm);
      if (!rc && r > 0) fastest = std::min(fastest, span_ms(pm, ~0u));
    }
    // a batched plan's transposed step times its field 0 (the fields run
    // one after another); the natural one times every field at once
    if (layout == 0) fastest *= plan->batch;
    // multi-step runs, where they are faster than single steps (a run covers
    // every field of the plan)
    constexpr int kLayoutRun = 6;
    for (int r = 0; r <= reps && !rc && !plan->tungsten(); ++r) {
      const double ms = run_ms_of(kLayoutRun) / kLayoutRun;
      if (r > 0) fastest = std::min(fastest, ms);
    }
    layout_ms[layout] = fastest;
  }
  if (!rc && two) {
    rc = pfc_hip_variant_set(plan, ROLE_STEP_LAYOUT,
                             layout_ms[0] <= layout_ms[1] ? 0 : 1);
  }
  if (times_ms && slot + 1 < max_times) {
    times_ms[slot] = layout_ms[0];
    times_ms[slot + 1] = layout_ms[1];
  }
  for (auto &e : ev)
    if (e) (void)hipEventDestroy(e);
  ++plan->gen; // the variants of every tuned role may have changed
  std::fill(std::begin(plan->chosen), std::end(plan->chosen), true);
  // psi is restored on every exit path once the backup was enqueued; a
  // failure of the sweep keeps its own code and message
  const std::string sweep_error = rc ? g_last_error : std::string();
  hipError_t he = hipMemcpyAsync(psi, plan->work, rbytes, hipMemcpyDeviceToDevice, s);
  if (he == hipSuccess) he = hipStreamSynchronize(s);
  if (rc) {
    g_last_error = sweep_error + (he == hipSuccess ? std::string(" (psi restored)")
                                                   : std::string(" (psi not restored: ") +
                                                         hipGetErrorString(he) + ")");
    return rc;
  }
  PFC_HIP_TRY(he, "autotune restore");
  return 0;
}

int pfc_hip_pfc_set_members(pfc_hip_plan_t plan, const double *eps, const double *mean,
                            int mean_split) {
  if (int rc = check_plan(plan)) return rc;
  if (!plan->ops_ready || plan->model_kind != PFC_HIP_MODEL_PFC)
    return fail(PFC_HIP_ESTATE, "pfc_hip_pfc_set_members: PFC operators not set");
  if (mean_split && !mean)
    return fail(PFC_HIP_EINVAL, "pfc_hip_pfc_set_members: mean_split needs the means");
  const int nb = plan->batch;
  std::vector<double> e((size_t)nb, plan->op.eps), m((size_t)nb, 0.0);
  for (int b = 0; b < nb; ++b) {
    if (eps) e[(size_t)b] = eps[b];
    if (mean_split) m[(size_t)b] = mean[b];
    if (!std::isfinite(e[(size_t)b]) || !std::isfinite(m[(size_t)b]))
      return fail(PFC_HIP_EINVAL, "pfc_hip_pfc_set_members: value of field " +
                                      std::to_string(b) + " not finite");
  }
  if (int rc = set_device(plan)) return rc;
  if (nb == 1) { // a plain plan: the scalars are the members
    plan->op.eps = e[0];
    plan->mean_split = mean_split != 0;
    plan->mean = m[0];
    ++plan->gen; // launch arguments changed
    return 0;
  }
  if (int rc = dalloc(plan, &plan->m_eps, (size_t)nb * sizeof(double), "field eps")) return rc;
  if (int rc = dalloc(plan, &plan->m_nl, (size_t)nb * 2 * plan->esize, "field means"))
    return rc;
  // (3m, 3m^2) rounded once to the field type, as for a single field
  std::vector<double> c2d((size_t)2 * nb);
  std::vector<float> c2f((size_t)2 * nb);
  for (int b = 0; b < nb; ++b) {
    const double mb = m[(size_t)b];
    c2d[(size_t)2 * b] = 3.0 * mb;
    c2d[(size_t)2 * b + 1] = 3.0 * mb * mb;
    c2f[(size_t)2 * b] = (float)c2d[(size_t)2 * b];
    c2f[(size_t)2 * b + 1] = (float)c2d[(size_t)2 * b + 1];
  }
  // the stream order of later steps is kept by the synchronous copies
  PFC_HIP_TRY(hipDeviceSynchronize(), "pfc_hip_pfc_set_members: sync");
  PFC_HIP_TRY(hipMemcpy(plan->m_eps, e.data(), (size_t)nb * sizeof(double),
                        hipMemcpyHostToDevice),
              "pfc_hip_pfc_set_members: eps upload");
  if (plan->prec == PFC_HIP_F64)
    PFC_HIP_TRY(hipMemcpy(plan->m_nl, c2d.data(), c2d.size() * sizeof(double),
                          hipMemcpyHostToDevice),
                "pfc_hip_pfc_set_members: mean upload");
  else
    PFC_HIP_TRY(hipMemcpy(plan->m_nl, c2f.data(), c2f.size() * sizeof(float),
                          hipMemcpyHostToDevice),
                "pfc_hip_pfc_set_members: mean upload");
  plan->h_eps = e;
  plan->h_mean = m;
  // the natural layout reads eps and the means from device memory; the
  // transposed one takes them, and the mean-split mode, as launch arguments
  ++plan->gen;
  plan->members = true;
  plan->mean_split = mean_split != 0;
  plan->mean = 0.0;
  return 0;
}

int pfc_hip_pfc_set_mean(pfc_hip_plan_t plan, int enable, double mean) {
  if (int rc = check_single(plan, "pfc_hip_pfc_set_mean")) return rc;
  if (enable && plan->tungsten())
    return fail(PFC_HIP_EUNSUPPORTED,
                "pfc_hip_pfc_set_mean: the mean-split mode applies to the PFC model only");
  if (!std::isfinite(mean)) return fail(PFC_HIP_EINVAL, "pfc_hip_pfc_set_mean: mean not finite");
  plan->mean_split = enable != 0;
  plan->mean = enable ? mean : 0.0;
  ++plan->gen;
  return 0;
}

} // extern "C"

namespace pfc_amd {
// Launch-argument generation of a plan (ensemble.hip re-captures its graph
// when a group plan's generation moved since the capture).
unsigned plan_generation(const pfc_hip_plan_s *p) { return p ? p->gen : 0u; }
} // namespace pfc_amd
