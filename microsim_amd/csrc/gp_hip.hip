/*
 * gp_hip.hip -- libgp_hip: the C ABI of include/gp_hip.h over hand-written CDNA4 (gfx950) kernels.
 *
 * Device layout (one handle):
 *   every field component is a plane of rows_x = mesh_x+6 rows; a row holds the halo-inclusive y range
 *   0..mesh_y+5 starting at element kYOff, so the first interior cell y = 3 sits on a 64-element boundary;
 *   the row pitch ps is a multiple of 64 elements. phi (N planes) and mu (NC planes) are ping-ponged,
 *   dphi (N planes) holds delta-phi when it is asked for.
 * A time step (default, gp_cells.h) classifies cells by the phase codes of the current state: k_cbulk updates the
 * bulk cells (streaming mu; phi stays e_b) and lists the interface cells and the delta-phi candidates (its blocks
 * past the tiles add the candidates of the boundary ring); k_dlist_step (k_dlist_c in the compensated mode) evaluates
 * delta-phi of the listed candidates, copies the halo cells whose proxy is a bulk cell, lists the others and folds the
 * statistics of the step before; k_ilist (k_ilist_c) runs the general update of the listed interface cells and of the
 * listed halo cells' proxies; k_stats folds the last step of a run with statistics.
 * GP_PATH=march selects the tiled march (gp_march.h: k_dphi, then k_march near an interface and k_bulk on deep
 * tiles); GP_PATH=twopass the two-pass form (k_phi: delta-phi on x,y in [2, mesh+3]; k_mu: currents and update
 * on the interior), which also runs the smoothing steps and recomputes delta-phi for gp_download. The kernels of both
 * write the halo images of the boundary cells they update.
 * This file holds the C ABI and the host-side handling; the kernels and their launch sequences are templates over
 * (phases, mu fields) in gp_step_impl.h, instantiated once per supported pair by gp_ops.hip.
 * Reference routines replaced: see include/gp_hip.h.
 */
#include <memory>
#include <mutex>

#include "gp_internal.h"
#include "gp_pack.h"
#include "gp_adjoint.h"
#include "gp_cells.h"

using namespace gpk;

namespace {
char g_create_error[512];

/* Scratch of gp_invariants_noalloc: the per-block sums of k_invariants, in a device array the library holds for the
 * life of the process (one copy per GPU). Host code never passes `scratch` itself to a kernel (in host code the
 * name stands for a host-side shadow, not a device address): it uses the device address that hipGetSymbolAddress
 * returned for the current GPU, looked up once per GPU when the first handle is created there. */
static __device__ __align__(256) double scratch[GP_NOALLOC_SCRATCH_DOUBLES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
double *g_scratch_ptr[kMaxDevices];
bool g_scratch_done[kMaxDevices];

/* the device address of `scratch` on GPU `dev` (current), looked up on the first call for that GPU */
int scratch_lookup(int dev, double **out, char *err) {
  if (dev < 0 || dev >= kMaxDevices) return snprintf(err, 512, "device index %d out of range", dev), GP_E_ARG;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_done[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess)
      return snprintf(err, 512, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e)), GP_E_HIP;
    g_scratch_ptr[dev] = (double *)p;
    g_scratch_done[dev] = true;
  }
  *out = g_scratch_ptr[dev];
  return GP_OK;
}
}  // namespace

int gp_fail(gp_handle *h, int code, const char *fmt, ...) {
  char *dst = h ? h->err : g_create_error;
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(dst, 512, fmt, ap);
  va_end(ap);
  return code;
}

/* the kernel set of (N, NC) in the given precision, or NULL when that pair is not instantiated */
static const GpOps *find_ops(int N, int NC, int precision) {
#define GP_FIND_OPS(a, b) \
  if (N == a && NC == b) return gp_ops_##a##_##b(precision);
  GP_COMBOS(GP_FIND_OPS)
#undef GP_FIND_OPS
  return nullptr;
}

/* Tile grid of the single-pass step: 60-cell y-strips by x-segments of 32 rows (16 when that gives fewer than
 * 4096 tiles, to fill the device on small grids); GP_SEG_LEN overrides the segment length. Each segment
 * recomputes two warm-up rows of delta-phi. */
static void march_plan(gp_handle *h) {
  const int64_t mx = h->p.mesh_x, my = h->p.mesh_y;
  const int64_t nstrips = (my + kMarchOut - 1) / kMarchOut;
  int64_t seg = 32;
  if (nstrips * ((mx + seg - 1) / seg) < 4096) seg = 16;
  const char *e = getenv("GP_SEG_LEN");
  if (e && atoi(e) > 0) seg = atoi(e);
  if (seg > mx) seg = mx;
  h->march_seg = (int)seg;
  h->march_nstrips = (int)nstrips;
  h->march_nsegs = (int)((mx + seg - 1) / seg);
  h->march_nwaves = nstrips * h->march_nsegs;
  /* k_cbulk: a tile costs one memory latency plus its rows in turn, so segments are long only when that still gives
   * kCellFill tiles; GP_CELL_SEG overrides (a value below kCellSegMax selects the short segments) */
  const int64_t cstrips = (my + kCellOut - 1) / kCellOut;
  int64_t cseg = cstrips * ((mx + kCellSegMax - 1) / kCellSegMax) >= kCellFill ? kCellSegMax : kCellSegMin;
  const char *ce = getenv("GP_CELL_SEG");
  if (ce && atoi(ce) > 0) cseg = atoi(ce) >= kCellSegMax ? kCellSegMax : kCellSegMin;
  h->cell_seg = (int)cseg;
  h->cell_nstrips = (int)cstrips;
  h->cell_nwaves = cstrips * ((mx + cseg - 1) / cseg);
  h->cell_npad = mx % 4 ? (int)((my + kPadOut - 1) / kPadOut) : 0;
}

/* ------------------------------------------------------------------------------------------------ helpers */

static void stats_reset_host(gp_handle *h, double *s) {
  const int N = h->N, NC = h->NC;
  for (int a = 0; a < N; a++) {
    s[a] = 1.0;      /* phi_max */
    s[N + a] = 0.0;  /* phi_min */
    s[2 * N + 2 * NC + a] = 0.0;
  }
  for (int k = 0; k < NC; k++) {
    s[2 * N + k] = 1.0;       /* mu_max */
    s[2 * N + NC + k] = 1.0;  /* mu_min */
    s[3 * N + 2 * NC + k] = 0.0;
  }
  s[3 * N + 3 * NC] = 0.0;
}

/* grid of the layout kernels: 256 elements of a row by rows (a stride loop past the limit of the y dimension) */
static dim3 pack_grid(int64_t width, int64_t nrows) {
  return dim3((unsigned)((width + 255) / 256), (unsigned)std::min<int64_t>(nrows, 32768));
}

/* `rows` rows of ry doubles go through the staging buffer in runs of whole rows: step(first row, rows, staging) enqueues a
 * run's copy and kernel on the handle's stream, in order, so that a run reuses the buffer after the one before it */
template <class F>
static int staged_rows(gp_handle *h, int64_t rows, F step) {
  const int64_t per = std::max<int64_t>(1, (int64_t)(h->stage_bytes / ((size_t)h->ry * sizeof(double))));
  for (int64_t r = 0; r < rows; r += per) {
    const int rc = step(r, std::min(per, rows - r), (double *)h->clist);
    if (rc) return rc;
  }
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return GP_OK;
}

/* halo-inclusive host planes of a field (0: phi, 1: mu) -> the planes d0 and d1 (unless NULL) in the given form (second
 * parts l0, l1); the halo as the host holds it */
static int rows_to_device(gp_handle *h, int form, void *d0, void *d1, void *l0, void *l1, const double *src, int ncomp) {
  const int64_t ry = h->ry, ps = h->ps;
  return staged_rows(h, ncomp * h->rx, [&](int64_t r, int64_t n, double *st) -> int {
    HIPCHK(h, hipMemcpyAsync(st, src + r * ry, (size_t)(n * ry) * sizeof(double), hipMemcpyHostToDevice, h->stream));
    const dim3 g = pack_grid(ps, n), b(256);
    if (form == PACK_F64) hipLaunchKernelGGL((k_pack<PACK_F64>), g, b, 0, h->stream, st, d0, d1, l0, l1, r, n, ry, ps);
    else if (form == PACK_F32) hipLaunchKernelGGL((k_pack<PACK_F32>), g, b, 0, h->stream, st, d0, d1, l0, l1, r, n, ry, ps);
    else if (form == PACK_DF) hipLaunchKernelGGL((k_pack<PACK_DF>), g, b, 0, h->stream, st, d0, d1, l0, l1, r, n, ry, ps);
    else hipLaunchKernelGGL((k_pack<PACK_C32>), g, b, 0, h->stream, st, d0, d1, l0, l1, r, n, ry, ps);
    HIPCHK(h, hipGetLastError());
    return GP_OK;
  });
}

/* device planes -> halo-inclusive host planes, decoded from the given form (second parts l) */
static int rows_to_host(gp_handle *h, int form, double *dst, const void *s, const void *l, int ncomp) {
  const int64_t ry = h->ry, ps = h->ps;
  return staged_rows(h, ncomp * h->rx, [&](int64_t r, int64_t n, double *st) -> int {
    const dim3 g = pack_grid(ry, n), b(256);
    if (form == PACK_F64) hipLaunchKernelGGL((k_unpack<PACK_F64>), g, b, 0, h->stream, st, s, l, r, n, ry, ps);
    else if (form == PACK_F32) hipLaunchKernelGGL((k_unpack<PACK_F32>), g, b, 0, h->stream, st, s, l, r, n, ry, ps);
    else if (form == PACK_DF) hipLaunchKernelGGL((k_unpack<PACK_DF>), g, b, 0, h->stream, st, s, l, r, n, ry, ps);
    else hipLaunchKernelGGL((k_unpack<PACK_C32>), g, b, 0, h->stream, st, s, l, r, n, ry, ps);
    HIPCHK(h, hipGetLastError());
    HIPCHK(h, hipMemcpyAsync(dst + r * ry, st, (size_t)(n * ry) * sizeof(double), hipMemcpyDeviceToHost, h->stream));
    return GP_OK;
  });
}

/* the stored form of field f of the handle's states */
static int field_form(const gp_handle *h, int f) {
  return h->precision == GP_FP64 ? PACK_F64 : h->precision == GP_FP32 ? PACK_F32 : f == 0 ? PACK_DF : PACK_C32;
}

/* field f of a host state into both state buffers, with the boundary copies */
static int upload_field(gp_handle *h, int f, const double *src) {
  const int ncomp = f == 0 ? h->N : h->NC, form = field_form(h, f);
  const int64_t mx = h->p.mesh_x, my = h->p.mesh_y;
  void *d[2], *l[2] = {nullptr, nullptr};
  for (int b = 0; b < 2; b++) {
    d[b] = f == 0 ? h->phi[b] : h->mu[b];
    if (h->precision == GP_FP32C) l[b] = f == 0 ? (void *)c32_plo(h, b) : (void *)c32_mlo(h, b);
  }
  const int rc = rows_to_device(h, form, d[0], d[1], l[0], l[1], src, ncomp);
  if (rc) return rc;
  const dim3 g((unsigned)((6 * (my + 6) + 6 * mx + 255) / 256), (unsigned)ncomp), b(256);
  if (form == PACK_F64)
    hipLaunchKernelGGL((k_pack_halo<double>), g, b, 0, h->stream, (double *)d[0], (double *)d[1], h->maps, f, h->fs,
                       h->ps, mx, my);
  else
    hipLaunchKernelGGL((k_pack_halo<float>), g, b, 0, h->stream, (float *)d[0], (float *)d[1], h->maps, f, h->fs, h->ps,
                       mx, my);
  if (form == PACK_DF)
    hipLaunchKernelGGL((k_pack_halo<float>), g, b, 0, h->stream, (float *)l[0], (float *)l[1], h->maps, f, h->fs, h->ps,
                       mx, my);
  else if (form == PACK_C32)
    hipLaunchKernelGGL((k_pack_halo<int8_t>), g, b, 0, h->stream, (int8_t *)l[0], (int8_t *)l[1], h->maps, f, h->fs,
                       h->ps, mx, my);
  HIPCHK(h, hipGetLastError());
  return GP_OK;
}

static int validate(const gp_params *p, char *err) {
  if (p->nphases < 2 || p->nphases > GP_MAXP) return snprintf(err, 512, "nphases %d outside [2,%d]", p->nphases, GP_MAXP), GP_E_ARG;
  if (p->ncomp < 2 || p->ncomp - 1 > GP_MAXNC) return snprintf(err, 512, "ncomp %d outside [2,%d]", p->ncomp, GP_MAXNC + 1), GP_E_ARG;
  if (p->mesh_x < 4 || p->mesh_y < 4) return snprintf(err, 512, "mesh must be at least 4x4"), GP_E_ARG;
  if (p->mesh_x > (1 << 20) || p->mesh_y > (1 << 20)) return snprintf(err, 512, "mesh too large"), GP_E_ARG;
  if (p->fn_w != 1 && p->fn_w != 2) return snprintf(err, 512, "fn_w must be 1 (obstacle) or 2 (well)"), GP_E_ARG;
  if (p->fn_aniso != 0 && p->fn_aniso != 1) return snprintf(err, 512, "fn_aniso must be 0 or 1"), GP_E_ARG;
  if (p->fn_aniso == 1 && p->fold != 4) return snprintf(err, 512, "anisotropy type %d not supported (4 only)", p->fold), GP_E_ARG;
  if (!(p->dx > 0 && p->dy > 0 && p->dt > 0 && p->epsilon > 0)) return snprintf(err, 512, "dx, dy, dt, epsilon must be > 0"), GP_E_ARG;
  if (p->solve < 0 || p->solve > 3) return snprintf(err, 512, "unknown solve mode %d", p->solve), GP_E_ARG;
  if (p->solve == GP_SOLVE_BINARY && p->ncomp != 2) return snprintf(err, 512, "BINARY solve needs ncomp = 2"), GP_E_ARG;
  if (p->solve == GP_SOLVE_TERNARY && p->ncomp != 3) return snprintf(err, 512, "TERNARY solve needs ncomp = 3"), GP_E_ARG;
  const int64_t ex[2] = {p->mesh_x + 2, p->mesh_y + 2};
  for (int f = 0; f < 2; f++)
    for (int k = 0; k < 6; k++) {
      if (p->halo_src_x[f][k] < 3 || p->halo_src_x[f][k] > ex[0] || p->halo_src_y[f][k] < 3 || p->halo_src_y[f][k] > ex[1])
        return snprintf(err, 512, "halo map of field %d entry %d points outside the interior", f, k), GP_E_ARG;
    }
  return GP_OK;
}

/* ------------------------------------------------------------------------------------------------ adjoint */

/* the current state into / from a state buffer laid out phi planes then mu planes */
/* (a GP_FP32C state buffer holds the extensions after the planes) */
static int state_save(gp_handle *h, double *dst) {
  const size_t es = esize(h), pb = (size_t)h->N * h->fs * es, mb = (size_t)h->NC * h->fs * es;
  HIPCHK(h, hipMemcpyAsync(dst, h->phi[h->cur], pb, hipMemcpyDeviceToDevice, h->stream));
  HIPCHK(h, hipMemcpyAsync((char *)dst + pb, h->mu[h->cur], mb, hipMemcpyDeviceToDevice, h->stream));
  if (h->precision == GP_FP32C)
    HIPCHK(h, hipMemcpyAsync((char *)dst + pb + mb, h->lo[h->cur], c32_lo_bytes(h), hipMemcpyDeviceToDevice,
                             h->stream));
  return GP_OK;
}
static int state_load(gp_handle *h, const double *src) {
  const size_t es = esize(h), pb = (size_t)h->N * h->fs * es, mb = (size_t)h->NC * h->fs * es;
  HIPCHK(h, hipMemcpyAsync(h->phi[h->cur], src, pb, hipMemcpyDeviceToDevice, h->stream));
  HIPCHK(h, hipMemcpyAsync(h->mu[h->cur], (const char *)src + pb, mb, hipMemcpyDeviceToDevice, h->stream));
  if (h->precision == GP_FP32C)
    HIPCHK(h, hipMemcpyAsync(h->lo[h->cur], (const char *)src + pb + mb, c32_lo_bytes(h), hipMemcpyDeviceToDevice,
                             h->stream));
  h->flags_valid = false;
  h->codes_valid = false;
  h->prev_valid = false;
  return GP_OK;
}

/* The handle's state pointers, bound to stored states (state_save's layout) for a while. direct: steps may run from one
 * stored state into another, which holds when every halo cell is written by a step (a cell without a proxy keeps what an
 * upload left there) and by the cell-classified step, whose output buffer needs no earlier contents. */
struct StateBinding {
  gp_handle *h;
  void *phi[2], *mu[2];
  int8_t *lo[2];
  bool direct, bound = false;
  explicit StateBinding(gp_handle *hh) : h(hh), direct(hh->use_cells && hh->halo_whole) {
    for (int b = 0; b < 2; b++) {
      phi[b] = h->phi[b];
      mu[b] = h->mu[b];
      lo[b] = h->lo[b];
    }
  }
  void bind(int b, double *state) {
    const size_t es = esize(h), pb = (size_t)h->N * h->fs * es, mb = (size_t)h->NC * h->fs * es;
    bound = true;
    h->phi[b] = state;
    h->mu[b] = (char *)state + pb;
    if (h->precision == GP_FP32C) h->lo[b] = (int8_t *)state + pb + mb;
  }
  /* the handle's own buffers again: the codes and flags of the bound states say nothing of them */
  void release() {
    if (!bound) return;
    bound = false;
    for (int b = 0; b < 2; b++) {
      h->phi[b] = phi[b];
      h->mu[b] = mu[b];
      h->lo[b] = lo[b];
    }
    h->codes_valid = h->flags_valid = h->prev_valid = false;
  }
  ~StateBinding() { release(); }
};

/* GP_ADJOINT_CHECK: the smallest index of a non-finite value of g[0, n) into out[0] (atomicMin; stays at ~0 when
 * there is none) and the largest |g| among the finite ones, as the bits of a non-negative double, into out[1] */
static __global__ __launch_bounds__(256) void k_adj_scan(const double *__restrict__ g, int64_t n,
                                                         unsigned long long *out) {
  unsigned long long bad = ~0ull, mx = 0ull;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const double v = g[i];
    if (!isfinite(v)) bad = (unsigned long long)i < bad ? (unsigned long long)i : bad;
    else {
      const unsigned long long b = (unsigned long long)__double_as_longlong(fabs(v));
      mx = b > mx ? b : mx;
    }
  }
  if (bad != ~0ull) atomicMin(&out[0], bad);
  if (mx) atomicMax(&out[1], mx);
}

/* after transposing forward step t (state t -> t + 1): stop with GP_E_NAN at the first non-finite adjoint or theta
 * gradient, naming the cell and the forward state there; every `every` steps print the largest |adjoint| */
static int adj_check(gp_handle *h, int64_t t, int64_t every, const double *phi64, const double *mu64) {
  Adjoint *A = h->adj;
  const int nth = theta_count(h->N, h->NC);
  if (!A->scan) HIPCHK(h, hipMalloc((void **)&A->scan, 4 * sizeof(unsigned long long)));
  const unsigned long long init[4] = {~0ull, 0ull, ~0ull, 0ull};
  HIPCHK(h, hipMemcpyAsync(A->scan, init, sizeof init, hipMemcpyHostToDevice, h->stream));
  const int64_t se = (int64_t)state_elems(h);
  hipLaunchKernelGGL(k_adj_scan, dim3(1024), dim3(256), 0, h->stream, (const double *)A->g[1], se, A->scan);
  hipLaunchKernelGGL(k_adj_scan, dim3(1), dim3(256), 0, h->stream, (const double *)A->gth, (int64_t)nth, A->scan + 2);
  HIPCHK(h, hipGetLastError());
  unsigned long long r[4];
  HIPCHK(h, hipMemcpyAsync(r, A->scan, sizeof r, hipMemcpyDeviceToHost, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  double gmax;
  memcpy(&gmax, &r[1], sizeof gmax);
  if (every > 0 && t % every == 0) fprintf(stderr, "gp adjoint check: step %lld max |adjoint| %.6e\n", (long long)t, gmax);
  if (r[0] == ~0ull && r[2] == ~0ull) return GP_OK;
  if (r[0] == ~0ull)
    return gp_fail(h, GP_E_NAN, "adjoint check: theta gradient %llu non-finite after transposing step %lld",
                   (unsigned long long)r[2], (long long)t);
  const int64_t comp = (int64_t)(r[0] / (unsigned long long)h->fs), c = (int64_t)(r[0] % (unsigned long long)h->fs);
  const int64_t x = (c - kYOff) / h->ps, y = (c - kYOff) % h->ps;
  double ph[P] = {0}, mv[NCM] = {0};
  for (int a = 0; a < h->N; a++)
    HIPCHK(h, hipMemcpy(&ph[a], phi64 + (size_t)a * h->fs + c, sizeof(double), hipMemcpyDeviceToHost));
  for (int k = 0; k < h->NC; k++)
    HIPCHK(h, hipMemcpy(&mv[k], mu64 + (size_t)k * h->fs + c, sizeof(double), hipMemcpyDeviceToHost));
  return gp_fail(h, GP_E_NAN,
                 "adjoint check: non-finite adjoint of %s %lld at cell (x %lld, y %lld) after transposing step %lld "
                 "(largest finite |adjoint| %.3e); state there: phi %.17g %.17g %.17g %.17g, mu %.17g %.17g %.17g",
                 comp < h->N ? "phi" : "mu", (long long)(comp < h->N ? comp : comp - h->N), (long long)x,
                 (long long)y, (long long)t, gmax, ph[0], ph[1], ph[2], ph[3], mv[0], mv[1], mv[2]);
}

/* fold the halo adjoints of A->g[1] into their source cells */
static int adj_fold(gp_handle *h) {
  Adjoint *A = h->adj;
  const dim3 gall((unsigned)((h->ry + 63) / 64), (unsigned)((h->rx + 3) / 4));
  hipLaunchKernelGGL(k_adj_bc, dim3(gall.x, gall.y, 2), dim3(256), 0, h->stream, A->g[1], h->N, h->NC, h->maps, h->fs,
                     h->ps, h->rx, h->ry);
  HIPCHK(h, hipGetLastError());
  return GP_OK;
}

/* ------------------------------------------------------------------------------------------------ frame */

/* temperature of allocated row 0 and the gradient per row, as the serial driver forms them before the loop (t = 0,
 * GPs/microsim_gp.c:77-80) and after step t (:108-111) */
double gp_frame_bottom(const gp_handle *h, int64_t t, double *grad) {
  const gp_params *p = &h->p;
  const double G = (p->tg_deltaT) * p->dy / (p->tg_distance);
  double base;
  if (t == 0) base = (p->tg_offset / p->dy) - (double)h->shift_off;
  else base = (p->tg_offset / p->dy) - (double)h->shift_off + ((p->tg_velocity / p->dy) * ((double)t * p->dt));
  *grad = G;
  return p->tg_base_temp - base * G;
}

/* T of every allocated row before the first step: the t = 0 gradient, then the boundary copies of T that run
 * before the loop (GPs/microsim_gp.c:81-84) */
static int frame_reset(gp_handle *h) {
  h->shift_off = 0;
  h->thermo_valid = false;
  if (!h->p.tempgrady) return GP_OK;
  double G;
  const double tb = gp_frame_bottom(h, 0, &G);
  std::vector<double> T((size_t)h->ry);
  for (int64_t y = 0; y < h->ry; y++) T[y] = tb + (double)y * G;
  for (int k = 0; k < 6; k++) T[h->tp.hy[k]] = T[h->tp.srcT[k]];
  HIPCHK(h, hipMemcpyAsync(h->trow, T.data(), T.size() * sizeof(double), hipMemcpyHostToDevice, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return GP_OK;
}

/* after step t (which has set the new temperature gradient): every 100 steps the moving frame */
static int frame_after_step(gp_handle *h, int64_t t) {
  if (!h->p.shift || t % 100 != 0) return GP_OK;
  const int N = h->N, NC = h->NC, L = N - 1;
  const size_t es = esize(h);
  HIPCHK(h, hipMemsetAsync(h->front, 0, sizeof(int), h->stream));
  const dim3 gf((unsigned)((h->ry - 1 + 63) / 64), (unsigned)((h->p.mesh_x + 3) / 4));
  if (h->precision == GP_FP64)
    hipLaunchKernelGGL((k_front<double>), gf, dim3(256), 0, h->stream,
                       (const double *)h->phi[h->cur] + (size_t)L * h->fs, h->front, h->ps, h->p.mesh_x, h->ry);
  else
    hipLaunchKernelGGL((k_front<float>), gf, dim3(256), 0, h->stream,
                       (const float *)h->phi[h->cur] + (size_t)L * h->fs, h->front, h->ps, h->p.mesh_x, h->ry);
  HIPCHK(h, hipGetLastError());
  int pos = 0;
  HIPCHK(h, hipMemcpyAsync(&pos, h->front, sizeof(int), hipMemcpyDeviceToHost, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  if (pos <= h->p.shiftj) return GP_OK;
  const int64_t sh = pos - h->p.shiftj;
  FillValues fp = {}, fm = {};
  fp.v[L] = 1.0;
  for (int k = 0; k < NC; k++) fm.v[k] = h->p.mu_fill[k];
  const dim3 ga((unsigned)((h->ry + 63) / 64), (unsigned)((h->rx + 3) / 4));
  if (es == sizeof(double)) {
    hipLaunchKernelGGL((k_shift<double>), ga, dim3(256), 0, h->stream, (const double *)h->phi[h->cur],
                       (double *)h->phi[1 - h->cur], N, fp, sh, h->fs, h->ps, h->rx, h->ry);
    hipLaunchKernelGGL((k_shift<double>), ga, dim3(256), 0, h->stream, (const double *)h->mu[h->cur],
                       (double *)h->mu[1 - h->cur], NC, fm, sh, h->fs, h->ps, h->rx, h->ry);
  } else {
    hipLaunchKernelGGL((k_shift<float>), ga, dim3(256), 0, h->stream, (const float *)h->phi[h->cur],
                       (float *)h->phi[1 - h->cur], N, fp, sh, h->fs, h->ps, h->rx, h->ry);
    hipLaunchKernelGGL((k_shift<float>), ga, dim3(256), 0, h->stream, (const float *)h->mu[h->cur],
                       (float *)h->mu[1 - h->cur], NC, fm, sh, h->fs, h->ps, h->rx, h->ry);
  }
  HIPCHK(h, hipGetLastError());
  h->cur = 1 - h->cur;
  if (h->p.tempgrady) {
    /* T moves with the rows; the top rows keep their own */
    std::vector<double> T((size_t)h->ry);
    HIPCHK(h, hipMemcpyAsync(T.data(), h->trow, T.size() * sizeof(double), hipMemcpyDeviceToHost, h->stream));
    HIPCHK(h, hipStreamSynchronize(h->stream));
    for (int64_t y = 0; y + sh <= h->ry - 1; y++) T[y] = T[y + sh];
    HIPCHK(h, hipMemcpyAsync(h->trow, T.data(), T.size() * sizeof(double), hipMemcpyHostToDevice, h->stream));
    HIPCHK(h, hipStreamSynchronize(h->stream));
  }
  h->shift_off += sh;
  h->thermo_valid = false;
  h->codes_valid = false;
  h->flags_valid = false;
  h->prev_valid = false;
  return GP_OK;
}

/* ------------------------------------------------------------------------------------------------ C ABI */

extern "C" {

const char *gp_version(void) { return "gp_hip 0.1 gfx950"; }

const char *gp_last_error(const gp_handle *h) { return h ? h->err : g_create_error; }

int gp_create(const gp_params *params, int precision, gp_handle **out) {
  if (!params || !out) return gp_fail(nullptr, GP_E_ARG, "null argument");
  *out = nullptr;
  int rc = validate(params, g_create_error);
  if (rc) return rc;
  if (precision != GP_FP64 && precision != GP_FP32 && precision != GP_FP32C)
    return gp_fail(nullptr, GP_E_ARG, "unknown precision %d", precision);
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return gp_fail(nullptr, GP_E_NODEV, "no HIP device");
  gp_handle *h = new gp_handle();
  memset(h->err, 0, sizeof h->err);
  h->p = *params;
  h->precision = precision;
  h->N = params->nphases;
  h->NC = params->ncomp - 1;
  h->rx = params->mesh_x + 6;
  h->ry = params->mesh_y + 6;
  h->ps = ((h->ry + kYOff + 63) / 64) * 64;
  h->fs = h->rx * h->ps;
  h->cur = 0;
  h->steps = 0;
  h->ops = find_ops(h->N, h->NC, precision);
  if (!h->ops) {
    delete h;
    return gp_fail(nullptr, GP_E_ARG, "no kernel instantiated for %d phases / %d components", params->nphases, params->ncomp);
  }
  const int64_t hx[6] = {0, 1, 2, h->rx - 3, h->rx - 2, h->rx - 1}, hy[6] = {0, 1, 2, h->ry - 3, h->ry - 2, h->ry - 1};
  for (int f = 0; f < 2; f++)
    for (int k = 0; k < 6; k++) {
      h->maps.sx[f][k] = params->halo_src_x[f][k];
      h->maps.sy[f][k] = params->halo_src_y[f][k];
    }
  for (int k = 0; k < 6; k++) {
    h->maps.hx[k] = (int32_t)hx[k];
    h->maps.hy[k] = (int32_t)hy[k];
  }
  h->halo_whole = true;
  for (int f = 0; f < 2; f++)
    for (int k = 0; k < 6; k++) {
      int bx = 0, by = 0; /* earlier images of the same row or column: a step writes two (halo_source) */
      for (int j = 0; j < k; j++) {
        bx += h->maps.sx[f][j] == h->maps.sx[f][k];
        by += h->maps.sy[f][j] == h->maps.sy[f][k];
      }
      if (bx >= 2 || by >= 2) h->halo_whole = false;
    }
  if (hipGetDevice(&h->device) != hipSuccess) {
    delete h;
    return gp_fail(nullptr, GP_E_NODEV, "hipGetDevice failed");
  }
  {
    /* device address of gp_invariants_noalloc's scratch on this GPU (looked up once per GPU) */
    double *sp = nullptr;
    rc = scratch_lookup(h->device, &sp, g_create_error);
    if (rc) {
      delete h;
      return rc;
    }
  }
  h->nblocks_mu = ((params->mesh_y + kBX - 1) / kBX) * ((params->mesh_x + kBY - 1) / kBY);
  march_plan(h);
  h->nparts_max = std::max(h->nblocks_mu, std::max(2 * h->march_nwaves, 2 * (h->cell_nwaves + h->cell_npad + 4 * (int64_t)kListBlocks)));
  const char *path = getenv("GP_PATH");
  h->use_march = !(path && strcmp(path, "twopass") == 0);
  /* the cell lists and k_cbulk's row offsets are 32-bit: grids beyond that bound (cells_fit, about 46000^2 cells)
   * take the tiled march, which gives the same results */
  h->use_cells = h->use_march && !(path && strcmp(path, "march") == 0) && cells_fit(h->rx, h->ps);
  if ((params->tempgrady || params->shift) && precision == GP_FP32C) {
    delete h;
    return gp_fail(nullptr, GP_E_ARG, "non-isothermal runs and the moving frame run in GP_FP64 or GP_FP32");
  }
  if (params->tempgrady) h->use_march = h->use_cells = false; /* the two-pass kernels carry the row temperatures */
  if (precision == GP_FP32C && !h->use_cells) {
    delete h;
    return gp_fail(nullptr, GP_E_ARG,
                   "the compensated FP32 mode runs the cell-classified step only (GP_PATH selects another path, or the "
                   "grid has 2^31 cells or more)");
  }
  h->prev_valid = false;
  h->fcur = 0;
  h->flags_valid = false;
  h->codes_valid = false;
  const size_t es = precision == GP_FP64 ? 8 : 4;
  const size_t pn = (size_t)h->N * h->fs * es, mn = (size_t)h->NC * h->fs * es;
  hipError_t e = hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking);
  bool ok = e == hipSuccess;
  Arena *mem = h->mem = new Arena();
  for (int b = 0; b < 2; b++) {
    mem->take(&h->phi[b], pn);
    mem->take(&h->mu[b], mn);
    if (precision == GP_FP32C) mem->take(&h->lo[b], c32_lo_bytes(h));
    mem->take(&h->flags[b], sizeof(int) * h->march_nwaves);
    mem->take(&h->codes[b], (size_t)h->rx * h->ps);
  }
  mem->take(&h->dphi, (size_t)h->N * h->fs * dphi_esize(h));
  if (params->tempgrady) {
    const size_t rt = precision == GP_FP64 ? sizeof(RowThermo<double>) : sizeof(RowThermo<float>);
    mem->take(&h->trow, (size_t)h->ry * sizeof(double));
    mem->take(&h->thp, (size_t)h->ry * rt);
    mem->take(&h->thc, (size_t)h->ry * rt);
  }
  if (params->shift) mem->take(&h->front, sizeof(int));
  if (precision == GP_FP32C) mem->take(&h->model64, sizeof(Model<double>));
  mem->take(&h->partials, sizeof(double) * kNStatMax * h->nparts_max);
  mem->take(&h->stats_dev, sizeof(double) * kNStatMax);
  mem->take(&h->inv_dev, sizeof(double) * (GP_MAXNC + 1));
  mem->take(&h->tflags, 2 * (size_t)h->cell_nwaves);
  /* the two cell lists in one piece (8 bytes a cell): between steps it stages the rows of uploads and downloads, the phi
   * planes of a small grid in one run */
  h->stage_bytes = std::max((size_t)h->fs * 2 * sizeof(int32_t),
                            std::min((size_t)h->N * h->fs * sizeof(double), kStageBytes));
  mem->take(&h->clist, h->stage_bytes);
  mem->take(&h->mlist, (size_t)halo_cells(params->mesh_x, params->mesh_y) * 2 * sizeof(uint64_t));
  mem->take(&h->lcount, 6 * sizeof(int));
  h->ccur = 0;
  const size_t msize = precision == GP_FP64 ? sizeof(Model<double>) : sizeof(Model<float>);
  mem->take(&h->model, msize);
  ok = ok && mem->allocate();
  h->ilist = ok ? h->clist + h->fs : nullptr;
  if (!ok) {
    gp_destroy(h);
    return gp_fail(nullptr, GP_E_OOM, "device allocation failed (%zu bytes per phi copy)", pn);
  }
  ok = hipMemsetAsync(h->phi[0], 0, pn, h->stream) == hipSuccess && hipMemsetAsync(h->phi[1], 0, pn, h->stream) == hipSuccess &&
       hipMemsetAsync(h->mu[0], 0, mn, h->stream) == hipSuccess && hipMemsetAsync(h->mu[1], 0, mn, h->stream) == hipSuccess &&
       hipMemsetAsync(h->dphi, 0, (size_t)h->N * h->fs * dphi_esize(h), h->stream) == hipSuccess &&
       hipMemsetAsync(h->lcount, 0, 6 * sizeof(int), h->stream) == hipSuccess;
  h->lsel = 0;
  if (precision == GP_FP64) {
    Model<double> m;
    make_model(params, &m);
    h->pow2 = m.pow2 != 0;
    ok = ok && hipMemcpyAsync(h->model, &m, sizeof m, hipMemcpyHostToDevice, h->stream) == hipSuccess;
    ok = ok && hipStreamSynchronize(h->stream) == hipSuccess;
  } else {
    Model<float> m;
    make_model(params, &m);
    h->pow2 = m.pow2 != 0;
    ok = ok && hipMemcpyAsync(h->model, &m, sizeof m, hipMemcpyHostToDevice, h->stream) == hipSuccess;
    if (precision == GP_FP32C) {
      Model<double> m64;
      make_model(params, &m64);
      ok = ok && hipMemsetAsync(h->lo[0], 0, c32_lo_bytes(h), h->stream) == hipSuccess &&
           hipMemsetAsync(h->lo[1], 0, c32_lo_bytes(h), h->stream) == hipSuccess &&
           hipMemcpyAsync(h->model64, &m64, sizeof m64, hipMemcpyHostToDevice, h->stream) == hipSuccess;
      ok = ok && hipStreamSynchronize(h->stream) == hipSuccess;
    }
    ok = ok && hipStreamSynchronize(h->stream) == hipSuccess;
  }
  if (!ok) {
    gp_destroy(h);
    return gp_fail(nullptr, GP_E_HIP, "device initialisation failed");
  }
  if (params->tempgrady) {
    /* the row coefficients' parameters (gp_frame.h k_thermo) */
    ThermoParams &tp = h->tp;
    tp.Teq = params->Teq;
    for (int k = 0; k < 6; k++) {
      tp.hy[k] = h->maps.hy[k];
      tp.srcT[k] = params->halo_src_T_y[k];
    }
    for (int a = 0; a < GP_MAXP; a++) {
      for (int i = 0; i < GP_MAXNC; i++) {
        tp.Beq[a][i] = params->Beq[a * GP_MAXNC + i];
        tp.dBbdT[a][i] = params->dBbdT[a * GP_MAXNC + i];
        tp.ceq_sol[a][i] = params->ceq_sol[a * GP_MAXNC + i];
        tp.ceq_liq[a][i] = params->ceq_liq[a * GP_MAXNC + i];
        tp.delta_c[a][i] = params->delta_c[a * GP_MAXNC + i];
        for (int j = 0; j < GP_MAXNC; j++) tp.A[a][i][j] = params->A[(a * GP_MAXNC + i) * GP_MAXNC + j];
      }
      tp.delta_T_sol[a] = params->delta_T_sol[a];
      tp.delta_T_liq[a] = params->delta_T_liq[a];
    }
  }
  double s[kNStatMax] = {0};
  stats_reset_host(h, s);
  if (hipMemcpy(h->stats_dev, s, sizeof s, hipMemcpyHostToDevice) != hipSuccess) {
    gp_destroy(h);
    return gp_fail(nullptr, GP_E_HIP, "device initialisation failed");
  }
  *out = h;
  return GP_OK;
}

void gp_destroy(gp_handle *h) {
  if (!h) return;
  /* teardown: errors here have no caller to report to, so they are ignored explicitly */
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  for (auto &r : h->prof) {
    (void)hipEventDestroy(r.second.first);
    (void)hipEventDestroy(r.second.second);
  }
  h->prof.clear();
  delete h->adj;
  delete h->mem;
  for (double *b : h->wide)
    if (b) (void)hipFree(b);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
}

int gp_upload(gp_handle *h, const double *phi, const double *mu) {
  if (!h || !phi || !mu) return h ? gp_fail(h, GP_E_ARG, "null argument") : GP_E_ARG;
  int rc;
  if ((rc = upload_field(h, 0, phi)) || (rc = upload_field(h, 1, mu))) return rc;
  HIPCHK(h, hipMemsetAsync(h->dphi, 0, (size_t)h->N * h->fs * dphi_esize(h), h->stream));
  double s[kNStatMax] = {0};
  stats_reset_host(h, s);
  HIPCHK(h, hipMemcpyAsync(h->stats_dev, s, sizeof s, hipMemcpyHostToDevice, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  h->steps = 0;
  h->prev_valid = false;
  h->flags_valid = false;
  h->codes_valid = false;
  return frame_reset(h);
}

int gp_download(gp_handle *h, double *phi, double *mu, double *dphi) {
  if (!h) return GP_E_ARG;
  int rc;
  const bool c = h->precision == GP_FP32C;
  const void *plo = c ? (const void *)c32_plo(h, h->cur) : nullptr, *mlo = c ? (const void *)c32_mlo(h, h->cur) : nullptr;
  if (phi && (rc = rows_to_host(h, field_form(h, 0), phi, h->phi[h->cur], plo, h->N))) return rc;
  if (mu && (rc = rows_to_host(h, field_form(h, 1), mu, h->mu[h->cur], mlo, h->NC))) return rc;
  if (dphi) {
    if (h->prev_valid) {
      /* single-pass steps do not store delta-phi: recompute the last step's from the previous state */
      if ((rc = h->ops->step(h, MODE_DPHI_PREV))) return rc;
    }
    const int form = dphi_esize(h) == sizeof(double) ? PACK_F64 : PACK_F32;
    if ((rc = rows_to_host(h, form, dphi, h->dphi, nullptr, h->N))) return rc;
  }
  return GP_OK;
}

int gp_upload_fields(gp_handle *h, const gp_cell *cells, int64_t ncells) {
  if (!h || !cells) return h ? gp_fail(h, GP_E_ARG, "null argument") : GP_E_ARG;
  const int64_t n = h->rx * h->ry;
  if (ncells != n) return gp_fail(h, GP_E_ARG, "ncells %lld != rows_x*rows_y %lld", (long long)ncells, (long long)n);
  std::vector<double> phi((size_t)h->N * n), mu((size_t)h->NC * n);
  for (int64_t i = 0; i < n; i++) {
    for (int a = 0; a < h->N; a++) phi[(size_t)a * n + i] = cells[i].phia[a];
    for (int k = 0; k < h->NC; k++) mu[(size_t)k * n + i] = cells[i].compi[k];
  }
  return gp_upload(h, phi.data(), mu.data());
}

int gp_download_fields(gp_handle *h, gp_cell *cells, int64_t ncells) {
  if (!h || !cells) return h ? gp_fail(h, GP_E_ARG, "null argument") : GP_E_ARG;
  const int64_t n = h->rx * h->ry;
  if (ncells != n) return gp_fail(h, GP_E_ARG, "ncells %lld != rows_x*rows_y %lld", (long long)ncells, (long long)n);
  std::vector<double> phi((size_t)h->N * n), mu((size_t)h->NC * n), dphi((size_t)h->N * n), T((size_t)h->ry);
  int rc = gp_download(h, phi.data(), mu.data(), dphi.data());
  if (rc || (rc = gp_get_frame(h, nullptr, T.data()))) return rc;
  for (int64_t i = 0; i < n; i++) {
    cells[i].temperature = T[(size_t)(i % h->ry)];
    for (int a = 0; a < h->N; a++) {
      cells[i].phia[a] = phi[(size_t)a * n + i];
      if (cells[i].deltaphi) cells[i].deltaphi[a] = dphi[(size_t)a * n + i];
    }
    for (int k = 0; k < h->NC; k++) cells[i].compi[k] = mu[(size_t)k * n + i];
  }
  return GP_OK;
}

int gp_smooth(gp_handle *h, int64_t nsteps) {
  if (!h || nsteps < 0) return h ? gp_fail(h, GP_E_ARG, "bad nsteps") : GP_E_ARG;
  step_fn f = h->ops->step;
  {
    ProfScope ps(h, GP_KERNEL_CALL);
    for (int64_t t = 0; t < nsteps; t++) {
      int rc = f(h, MODE_SMOOTH);
      if (rc) return rc;
    }
  }
  if (nsteps > 0) h->prev_valid = false; /* dphi now holds the smoothing increment */
  return GP_OK;
}

int gp_get_stats(gp_handle *h, gp_stats *st) {
  if (!h || !st) return h ? gp_fail(h, GP_E_ARG, "null argument") : GP_E_ARG;
  double s[kNStatMax], inv[GP_MAXNC + 1];
  inv_fn fi = h->ops->invariants;
  int rc = fi(h);
  if (rc) return rc;
  HIPCHK(h, hipMemcpyAsync(s, h->stats_dev, sizeof s, hipMemcpyDeviceToHost, h->stream));
  HIPCHK(h, hipMemcpyAsync(inv, h->inv_dev, sizeof(double) * (h->NC + 1), hipMemcpyDeviceToHost, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  memset(st, 0, sizeof *st);
  const int N = h->N, NC = h->NC;
  for (int a = 0; a < N; a++) {
    st->phi_max[a] = s[a];
    st->phi_min[a] = s[N + a];
    st->rel_change_phi[a] = s[2 * N + 2 * NC + a];
  }
  for (int k = 0; k < NC; k++) {
    st->mu_max[k] = s[2 * N + k];
    st->mu_min[k] = s[2 * N + NC + k];
    st->rel_change_mu[k] = s[3 * N + 2 * NC + k];
  }
  st->nonfinite = (int64_t)s[3 * N + 3 * NC];
  for (int k = 0; k < NC; k++) st->solute[k] = inv[k];
  st->energy = inv[NC];
  st->step = h->steps;
  return GP_OK;
}

int gp_get_frame(gp_handle *h, int64_t *shift_offset, double *T_rows) {
  if (!h) return GP_E_ARG;
  if (shift_offset) *shift_offset = h->shift_off;
  if (T_rows) {
    if (h->p.tempgrady) {
      HIPCHK(h, hipMemcpyAsync(T_rows, h->trow, (size_t)h->ry * sizeof(double), hipMemcpyDeviceToHost, h->stream));
      HIPCHK(h, hipStreamSynchronize(h->stream));
    } else {
      for (int64_t y = 0; y < h->ry; y++) T_rows[y] = h->p.T;
    }
  }
  return GP_OK;
}

int gp_invariants_noalloc(gp_handle *h, const void *phi, const void *mu, double *out, void *stream) {
  if (!h || !phi || !mu || !out) return h ? gp_fail(h, GP_E_ARG, "null argument") : GP_E_ARG;
  const int64_t mx = h->p.mesh_x, my = h->p.mesh_y;
  /* the block sums of k_invariants with one row a thread (64 y-cells by 4 x-rows a block); larger grids take several rows
   * and fewer blocks (invariant_rows), but the bound is the same for every grid */
  const int64_t nblocks = ((my + 63) / 64) * ((mx + 3) / 4);
  const int64_t need = (int64_t)(h->NC + 1) * nblocks;
  if (need > (int64_t)GP_NOALLOC_SCRATCH_DOUBLES)
    return gp_fail(h, GP_E_ARG,
                   "gp_invariants_noalloc: a %lldx%lld grid needs %lld scratch doubles, more than the %lld the library "
                   "holds (GP_NOALLOC_SCRATCH_DOUBLES)",
                   (long long)mx, (long long)my, (long long)need, (long long)GP_NOALLOC_SCRATCH_DOUBLES);
  int dev = -1;
  HIPCHK(h, hipGetDevice(&dev));
  if (dev != h->device)
    return gp_fail(h, GP_E_ARG, "gp_invariants_noalloc: the handle lives on device %d, device %d is current",
                   h->device, dev);
  double *sp = nullptr;
  int rc = scratch_lookup(dev, &sp, h->err);
  if (rc) return rc;
  /* the caller's state is in the reference's plain layout: plane = rows_x * rows_y, row pitch rows_y, no offset */
  return h->ops->invariants_on(h, phi, mu, h->rx * h->ry, h->ry, 0, sp, out,
                               stream ? (hipStream_t)stream : h->stream);
}

int gp_step(gp_handle *h, int64_t nsteps, gp_stats *stats) {
  if (!h || nsteps < 0) return h ? gp_fail(h, GP_E_ARG, "bad nsteps") : GP_E_ARG;
  step_fn f = h->ops->step;
  {
    ProfScope ps(h, GP_KERNEL_CALL);
    const bool framed = h->p.tempgrady || h->p.shift;
    h->stats_pending = false;
    for (int64_t t = 0; t < nsteps; t++) {
      int rc = f(h, h->use_march ? (stats ? MODE_MARCH_STATS : MODE_MARCH) : MODE_TWOPASS);
      if (rc) return rc;
      h->steps++;
      h->prev_valid = h->use_march;
      if (framed && (rc = frame_after_step(h, h->steps))) return rc;
    }
    if (stats && nsteps > 0 && h->use_cells) {
      int rc = f(h, MODE_STATS_FOLD);
      if (rc) return rc;
    }
  }
  if (stats) {
    int rc = gp_get_stats(h, stats);
    if (rc) return rc;
    if (stats->nonfinite) return gp_fail(h, GP_E_NAN, "%lld non-finite values after step %lld", (long long)stats->nonfinite, (long long)h->steps);
  }
  return GP_OK;
}

int gp_theta_count(const gp_handle *h) { return h ? theta_count(h->N, h->NC) : GP_E_ARG; }

int gp_theta_values(const gp_handle *h, double *theta) {
  if (!h || !theta) return GP_E_ARG;
  const gp_params *p = &h->p;
  const int N = h->N, NC = h->NC, L = N - 1;
  int t = 0;
  for (int a = 0; a < N; a++)
    for (int b = a + 1; b < N; b++) {
      theta[t++] = p->dab[a * GP_MAXP + b];
      theta[t++] = p->tau_ab[a * GP_MAXP + b];
      theta[t++] = p->gamma[a * GP_MAXP + b];
    }
  for (int k = 0; k < NC; k++) theta[t++] = p->diffusivity[(L * GP_MAXNC + k) * GP_MAXNC + k];
  theta[t++] = p->tau;
  return GP_OK;
}

int gp_adjoint_forward(gp_handle *h, int64_t nsteps, int64_t every) {
  if (!h || nsteps < 0) return h ? gp_fail(h, GP_E_ARG, "bad nsteps") : GP_E_ARG;
  if (h->p.tempgrady || h->p.shift)
    return gp_fail(h, GP_E_ARG, "the adjoint covers isothermal runs in a fixed frame");
  if (!h->use_march) return gp_fail(h, GP_E_ARG, "the adjoint records single-pass steps (GP_PATH=twopass is set)");
  if (h->fs > 0x7fffffff) return gp_fail(h, GP_E_ARG, "the adjoint indexes cells with 32 bits: grid too large");
  /* the handle takes the recording over when it is whole: after a failure there is none, and a backward sweep is refused
   * (its checkpoints would be null or unwritten) */
  delete h->adj;
  h->adj = nullptr;
  std::unique_ptr<Adjoint> A(new Adjoint());
  if (every <= 0) every = (int64_t)ceil(sqrt((double)(nsteps > 0 ? nsteps : 1)));
  A->nsteps = nsteps;
  A->every = every;
  const int64_t nck = nsteps / every + (nsteps % every != 0);
  /* a count that no device could hold is refused before the host lists its buffers (it would run out of memory first, or
   * their sizes out of 64 bits) */
  size_t free_bytes = 0, device_bytes = 0;
  HIPCHK(h, hipMemGetInfo(&free_bytes, &device_bytes));
  bool fits = (uint64_t)nck <= device_bytes / state_bytes(h);
  if (fits) {
    A->ckpt.resize((size_t)nck);
    for (double *&b : A->ckpt) A->ckpts.take(&b, state_bytes(h));
    fits = A->ckpts.allocate();
  }
  if (!fits) return gp_fail(h, GP_E_OOM, "adjoint: %lld checkpoints do not fit in device memory", (long long)nck);
  for (int64_t k = 0; k < nck; k++) {
    int rc = state_save(h, A->ckpt[(size_t)k]);
    if (!rc) rc = gp_step(h, std::min(every, nsteps - k * every), nullptr);
    if (rc) return rc;
  }
  h->adj = A.release();
  return GP_OK;
}

int gp_adjoint_backward(gp_handle *h, const double *gphi_T, const double *gmu_T, double *gphi_0, double *gmu_0,
                        double *gtheta) {
  if (!h || !gphi_T || !gmu_T || !gphi_0 || !gmu_0 || !gtheta) return h ? gp_fail(h, GP_E_ARG, "null argument") : GP_E_ARG;
  Adjoint *A = h->adj;
  if (!A) return gp_fail(h, GP_E_ARG, "gp_adjoint_forward must run first");
  const int nth = theta_count(h->N, h->NC);
  const size_t se = state_elems(h);
  if (!A->g[0]) {
    Arena &w = A->work;
    const bool other = h->precision != GP_FP64;
    for (double *&g : A->g) w.take(&g, se * sizeof(double));
    w.take(&A->gdphi, (size_t)h->N * h->fs * sizeof(double));
    w.take(&A->gth, sizeof(double) * nth);
    w.take(&A->cbar, (size_t)h->NC * h->fs * sizeof(double));
    w.take(&A->qlist, (size_t)h->fs * sizeof(int32_t));
    w.take(&A->plist, (size_t)h->fs * sizeof(int32_t));
    w.take(&A->counts, 4 * sizeof(int));
    for (int8_t **q : {&A->pcode, &A->bq, &A->cand}) w.take(q, (size_t)h->fs);
    A->seg.resize((size_t)std::max<int64_t>(0, std::min(A->every, A->nsteps) - 1));
    for (double *&b : A->seg) w.take(&b, state_bytes(h));
    if (other) {
      w.take(&A->st64, se * sizeof(double));
      w.take(&A->dphi64, (size_t)h->N * h->fs * sizeof(double));
      w.take(&A->model64, sizeof(Model<double>));
    }
    bool ok = w.allocate() && hipMemsetAsync(w.base(), 0, w.size(), h->stream) == hipSuccess;
    if (ok && other) {
      Model<double> m;
      make_model(&h->p, &m);
      ok = hipMemcpyAsync(A->model64, &m, sizeof m, hipMemcpyHostToDevice, h->stream) == hipSuccess &&
           hipStreamSynchronize(h->stream) == hipSuccess;
    }
    if (!ok) {
      w.reset(); /* a further call starts over */
      A->g[0] = nullptr;
      return gp_fail(h, GP_E_OOM, "adjoint: buffers do not fit in device memory");
    }
  }
  int rc;
  if ((rc = rows_to_device(h, PACK_F64, A->g[1], nullptr, nullptr, nullptr, gphi_T, h->N))) return rc;
  if ((rc = rows_to_device(h, PACK_F64, A->g[1] + (size_t)h->N * h->fs, nullptr, nullptr, nullptr, gmu_T, h->NC))) return rc;
  HIPCHK(h, hipMemsetAsync(A->gth, 0, sizeof(double) * nth, h->stream));
  step_fn f = h->ops->step;
  adj_fn fa = h->ops->adj_step;
  widen_fn fw = h->ops->widen;
  const bool wide = h->precision == GP_FP64;
  /* GP_ADJOINT_CHECK=<n>: scan the adjoint after every transposed step (one synchronisation each) and print its
   * largest magnitude every n steps */
  const char *ck = getenv("GP_ADJOINT_CHECK");
  const bool check = ck && *ck && strcmp(ck, "0") != 0;
  const int64_t check_every = check ? atoll(ck) : 0;
  /* A segment's states S[0 .. n) are its checkpoint and the segment buffers, and the handle steps from one into the next
   * (no copies): its state pointers are bound to them meanwhile and come back on every way out. Nothing of a bound buffer
   * is taken as kept from an earlier step. */
  StateBinding own(h);
  for (int64_t k = (int64_t)A->ckpt.size() - 1; k >= 0; k--) {
    const int64_t n = std::min(A->every, A->nsteps - k * A->every);
    const auto S = [&](int64_t j) { return j == 0 ? A->ckpt[(size_t)k] : A->seg[(size_t)(j - 1)]; };
    if (!own.direct) {
      own.release();
      if ((rc = state_load(h, S(0)))) return rc;
    } else {
      own.bind(h->cur, S(0));
      h->codes_valid = h->flags_valid = false;
    }
    for (int64_t j = 0; j + 1 < n; j++) {
      if (own.direct) own.bind(1 - h->cur, S(j + 1));
      h->prev_valid = false;
      if ((rc = gp_step(h, 1, nullptr))) return rc;
      if (!own.direct && (rc = state_save(h, S(j + 1)))) return rc;
    }
    for (int64_t j = n - 1; j >= 0; j--) {
      ProfScope ps(h, GP_KERNEL_ADJ);
      own.bind(h->cur, S(j));
      if (wide) {
        const double *p64 = (const double *)h->phi[h->cur], *m64 = (const double *)h->mu[h->cur];
        /* the handle is left with delta-phi of the initial state (a sweep stores it at candidates only) */
        if (k == 0 && j == 0) HIPCHK(h, hipMemsetAsync(h->dphi, 0, (size_t)h->N * h->fs * sizeof(double), h->stream));
        if ((rc = h->ops->adj_dphi(h, p64, m64, (double *)h->dphi, h->model))) return rc;
        rc = fa(h, p64, m64, (const double *)h->dphi, h->model);
      } else {
        if ((rc = fw(h))) return rc;
        if ((rc = h->ops->adj_dphi(h, A->st64, A->st64 + (size_t)h->N * h->fs, A->dphi64, A->model64))) return rc;
        rc = fa(h, A->st64, A->st64 + (size_t)h->N * h->fs, A->dphi64, A->model64);
      }
      if (rc) return rc;
      if (check) {
        const double *p64 = wide ? (const double *)h->phi[h->cur] : A->st64;
        const double *m64 = wide ? (const double *)h->mu[h->cur] : A->st64 + (size_t)h->N * h->fs;
        if ((rc = adj_check(h, k * A->every + j, check_every, p64, m64))) return rc;
      }
    }
  }
  own.release();
  if (!A->ckpt.empty() && (rc = state_load(h, A->ckpt[0]))) return rc;
  if ((rc = adj_fold(h))) return rc;
  if ((rc = rows_to_host(h, PACK_F64, gphi_0, A->g[1], nullptr, h->N))) return rc;
  if ((rc = rows_to_host(h, PACK_F64, gmu_0, A->g[1] + (size_t)h->N * h->fs, nullptr, h->NC))) return rc;
  HIPCHK(h, hipMemcpyAsync(gtheta, A->gth, sizeof(double) * nth, hipMemcpyDeviceToHost, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  h->steps = 0; /* the handle holds the initial state again */
  return GP_OK;
}

int gp_profile_enable(gp_handle *h, int enable) {
  if (!h) return GP_E_ARG;
  h->profiling = enable == GP_PROFILE_CALLS ? GP_PROFILE_CALLS : enable ? GP_PROFILE_LAUNCHES : GP_PROFILE_OFF;
  return GP_OK;
}

const char *gp_kernel_name(int kind) {
  static const char *names[GP_NKERNELS] = {"k_phi", "k_mu", "k_stats", "k_march", "k_march_stats", "k_bulk",
                                           "k_dphi", "adj_step", "k_cbulk", "k_ilist", "call", "k_halo"};
  return (kind >= 0 && kind < GP_NKERNELS) ? names[kind] : "?";
}

int gp_profile_read(gp_handle *h, double *avg_ms, int64_t *count) {
  if (!h || !avg_ms || !count) return h ? gp_fail(h, GP_E_ARG, "null argument") : GP_E_ARG;
  HIPCHK(h, hipStreamSynchronize(h->stream));
  double tot[GP_NKERNELS] = {0};
  int64_t cnt[GP_NKERNELS] = {0};
  for (auto &r : h->prof) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, r.second.first, r.second.second) == hipSuccess && r.first >= 0 && r.first < GP_NKERNELS) {
      tot[r.first] += ms;
      cnt[r.first]++;
    }
    (void)hipEventDestroy(r.second.first);
    (void)hipEventDestroy(r.second.second);
  }
  h->prof.clear();
  for (int k = 0; k < GP_NKERNELS; k++) {
    avg_ms[k] = cnt[k] ? tot[k] / (double)cnt[k] : 0.0;
    count[k] = cnt[k];
  }
  return GP_OK;
}

int gp_synchronize(gp_handle *h) {
  if (!h) return GP_E_ARG;
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return GP_OK;
}

}  // extern "C"
