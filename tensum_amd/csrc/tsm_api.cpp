// tsm_api.cpp -- host context and C ABI of libtsm (include/tsm.h).
//
// Owns the device copies of the geometry and of the per-sample state, one HIP
// stream, and the stage loop that replaces the body of FiniteVolume::solve
// (src/fv.cc:2273-2368).  No PyTorch, no MPI: the whole mesh is resident on
// one GPU and every reduction of the reference (dt, residual norm, periodic
// sums) is a device kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "tsm_device.h"
#include "tsm_host.h"
#include "expr.h"
#include "tprog.h"

namespace {
thread_local std::string g_last_error;
int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}
#define HIP_TRY(expr)                                                              \
  do {                                                                             \
    hipError_t _e = (expr);                                                        \
    if (_e != hipSuccess)                                                          \
      return fail(TSM_E_HIP, std::string(#expr) + ": " + hipGetErrorString(_e));  \
  } while (0)
}  // namespace

struct tsm_ctx {
  tsm_params P{};
  int S = 1;
  tsm::Geometry geo;
  hipStream_t st = nullptr;
  int dev = 0;              // device current at tsm_create (holds the buffers and the stream)
  tsm::DevGeo G{};
  tsm::StageArgs A{};
  tsm::StepParams SP{};
  std::vector<void*> allocs;
  double* W[3] = {nullptr, nullptr, nullptr};
  double* V[3] = {nullptr, nullptr, nullptr};  // first entropy variable of W[] (tiled TeCNO)
  double* E[2] = {nullptr, nullptr};
  int cur = 0;              // W[cur] / E[cur] hold the current state
  bool tiled = false;       // LDS-tiled stage kernels in use
  int* bad = nullptr;       // first refused vertex of a state
  bool e_valid = true;      // E[cur] == prim2ent(W[cur])
  tsm::Tiling tiling;
  tsm::StageTab ST{};
  bool two_rings_asked = false;  // tile_fused_gradient on a mesh and scheme it applies to
  double* dtpart = nullptr;
  std::vector<int> perm;    // part-file vertex id -> device vertex id
  const int* d_perm = nullptr;
  // Host memory that kernels write: what a call returns of a few KB arrives with
  // the call's one synchronisation, without copy commands.  Larger answers go
  // through device memory.
  static constexpr size_t PIN = 64 * 1024;
  // States of up to this much go through it too, behind the words of an answer
  // (state_off): a copy between the device and pageable memory is staged by the
  // runtime, 35 to 77 us out for 32 to 135 KB where a kernel and a copy on the host take
  // 13 to 18; from about 256 KB on the memory is pinned for the copy and the two draw
  // level (533 KB: 45 and 35).
  static constexpr size_t PIN_STATE = 512 * 1024;
  size_t state_off = 0;  // of the state in pin, 0 if it takes the copy
  char* pin = nullptr;
  // input bface b, end point k (bface_v[2b+k]) -> offset of its boundary
  // values in a sample's block of G.bstate; device boundary codes
  std::vector<long long> bmap;
  double* force_buf = nullptr;  // per-face force terms and the sum (tsm_forces)
  int* force_sel = nullptr;
  size_t force_cap = 0;
  double* W_keep = nullptr;     // last stage's input states (tsm_keep_stage_state)
  std::vector<int> h_btype;
  double* red = nullptr;   // reduction partials for global / error norms
  size_t red_cap = 0;
  std::vector<double> h_gamma, h_R;
  int nblk_v = 0;
  // captured steps of the tiled path (graph_steps > 0)
  hipGraphExec_t gexec = nullptr;
  int gcur = -1;
  // device copies of the level descriptors of packed multilevel steps
  // (tsm_run_packed with this context first)
  tsm::PackLevel* pack = nullptr;
  size_t pack_cap = 0;
  // time-dependent boundary values (tsm_set_bc_time_expr), re-evaluated
  // before every stage
  tsm::BcTime bt{};

  ~tsm_ctx() {
    if (st) (void)hipStreamSynchronize(st);
    if (pin) (void)hipHostFree(pin);
    if (gexec) (void)hipGraphExecDestroy(gexec);
    for (void* p : allocs) (void)hipFree(p);
    if (st) (void)hipStreamDestroy(st);
  }
  template <class T>
  int alloc(T** p, size_t n) {
    // small arrays share an allocation: a context has some hundred
    const size_t b = (std::max<size_t>(n, 1) * sizeof(T) + 255) & ~(size_t)255;
    if (b > shared_left) {
      void* q = nullptr;
      const bool own = b > SMALL;
      hipError_t e = hipMalloc(&q, own ? b : SHARED);
      if (e != hipSuccess) return fail(TSM_E_HIP, std::string("hipMalloc: ") + hipGetErrorString(e));
      allocs.push_back(q);
      if (own) { *p = (T*)q; return TSM_OK; }
      shared_at = (char*)q;
      shared_left = SHARED;
    }
    *p = (T*)shared_at;
    shared_at += b;
    shared_left -= b;
    return TSM_OK;
  }
  template <class T>
  int upload(const T** dst, const std::vector<T>& src) {
    T* d = nullptr;
    int rc = alloc(&d, src.size());
    if (rc) return rc;
    if (!src.empty()) HIP_TRY(hipMemcpy(d, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice));
    *dst = d;
    return TSM_OK;
  }
  // The same for the many arrays of a new context: small ones go in one copy, with
  // which dst is set (each copy of its own costs some 15 us however small).
  template <class Ptr, class T>
  int upload_later(Ptr* dst, const std::vector<T>& src) {
    static_assert(std::is_same<std::remove_const_t<std::remove_pointer_t<Ptr>>, T>::value, "types");
    const size_t b = src.size() * sizeof(T);
    if (b > SMALL) return upload((const T**)dst, src);
    later.push_back({(const void**)dst, later_bytes.size()});
    later_bytes.resize(later_bytes.size() + ((std::max<size_t>(b, 1) + 255) & ~(size_t)255));
    if (b) std::memcpy(later_bytes.data() + later.back().second, src.data(), b);
    return TSM_OK;
  }
  int upload_now() {
    const char* d = nullptr;
    if (int rc = upload(&d, later_bytes)) return rc;
    for (const auto& q : later) *q.first = d + q.second;
    later.clear();
    later_bytes.clear();
    return TSM_OK;
  }
  static constexpr size_t SMALL = 64 * 1024, SHARED = 1024 * 1024;
  char* shared_at = nullptr;
  size_t shared_left = 0;
  std::vector<std::pair<const void**, size_t>> later;
  std::vector<char> later_bytes;
  // the samples' control blocks on the host
  hipError_t read_ctl(std::vector<tsm::Ctl>& q) {
    const size_t n = S * sizeof(tsm::Ctl);
    hipError_t e;
    if (n <= PIN) {
      tsm::launch_words((long)n, A.ctl, pin, st);
      e = hipStreamSynchronize(st);
      if (e == hipSuccess) std::memcpy(q.data(), pin, n);
    } else {
      e = hipStreamSynchronize(st);
      if (e == hipSuccess) e = hipMemcpy(q.data(), A.ctl, n, hipMemcpyDeviceToHost);
    }
    return e;
  }
  void bind_state() {
    A.W_in = W[cur]; A.W_out = W[cur ^ 1];
    A.V_in = A.V_out = V[cur];
    A.E_in = E[cur]; A.E_out = E[cur ^ 1];
  }
  // Makes W[cur] the state of the CSR kernels' double buffer (W[0]/W[1]) and
  // refreshes the entropy variables they read.
  void csr_ready() {
    state_ready();
    if (!e_valid) {
      for (int s = 0; s < S; ++s) tsm::launch_prim2ent(G, A, s, st);
      e_valid = true;
    }
  }
  // W[cur] in the CSR kernels' double buffer, entropy variables as they are
  void state_ready() {
    if (cur == 2) {
      (void)hipMemcpyAsync(W[0], W[2], 4 * A.cs * sizeof(double), hipMemcpyDeviceToDevice, st);
      cur = 0;
      e_valid = false;
    }
    bind_state();
  }
  // ... with sample s's entropy variables current (single-sample queries: the
  // other samples' stay as they are, so a batch of queries costs one sample each)
  void sample_ready(int s) {
    state_ready();
    if (!e_valid) tsm::launch_prim2ent(G, A, s, st);
  }
};

extern "C" const char* tsm_last_error(void) { return g_last_error.c_str(); }

namespace {

int validate_params(const tsm_params& p) {
  if (!(p.gamma > 1.0)) return fail(TSM_E_ARG, "gamma must be > 1");
  if (!(p.gas_const > 0.0)) return fail(TSM_E_ARG, "gas_const must be > 0");
  if (p.flux < 0 || p.flux > 5) return fail(TSM_E_ARG, "unknown flux scheme");
  if (p.reconstruct < 0 || p.reconstruct > 6) return fail(TSM_E_ARG, "unknown reconstruction");
  if (p.time_scheme < 0 || p.time_scheme > 2)
    return fail(TSM_E_ARG, "time_scheme must be ssprk3 (0), rk4 (1) or heuns (2)");
  if (p.unsteady != 0 && p.unsteady != 1) return fail(TSM_E_ARG, "unsteady must be 0 or 1");
  if (p.strong_bc != 0 && p.strong_bc != 1) return fail(TSM_E_ARG, "strong_bc must be 0 (weak) or 1 (strong)");
  if (p.time_step == 0.0 && p.cfl == 0.0) return fail(TSM_E_ARG, "Either time_step or cfl must be non-zero");
  if (p.time_step > 0.0 && p.cfl > 0.0) return fail(TSM_E_ARG, "both time_step and cfl specified");
  if (p.unsteady && !(p.final_time > 0.0))
    return fail(TSM_E_ARG, "final_time must be positive for unsteady flow");
  if (p.unsteady && p.n_time_stamps <= 0) return fail(TSM_E_ARG, "time_stamps must be > 0");
  if (!p.unsteady && p.max_iter <= 0) return fail(TSM_E_ARG, "max_iter must be > 0");
  if (!(p.min_residue >= 0.0)) return fail(TSM_E_ARG, "min_residue must be >= 0");
  if (p.model == 0 && p.mu_ref > 0.0) return fail(TSM_E_ARG, "mu_ref must be 0 for the model=euler");
  return TSM_OK;
}

}  // namespace

namespace {
// One attempt at a context, with tiles of tb owned vertices (0: the CSR-gather
// kernels; -1: the size of params, to which tb is set).  1: a tile holds more slots
// or faces than the tables address or the stage kernel has LDS or threads for.
int create_with_tiles(const tsm_mesh* mesh, const tsm_params* params, int n_samples, int& tb,
                      tsm_ctx** out);
}  // namespace

extern "C" int tsm_create(const tsm_mesh* mesh, const tsm_params* params, int n_samples,
                          tsm_ctx** out) {
  if (!mesh || !params || !out || n_samples < 1) return fail(TSM_E_ARG, "null argument");
  *out = nullptr;
  int rc = validate_params(*params);
  if (rc) return rc;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    return fail(TSM_E_HIP, "no HIP device visible");
  // tiled stage kernels: every scheme, Euler or Navier-Stokes, with or without
  // the Liou fix; strong boundary conditions keep the CSR kernels.  A mesh with
  // vertices of so many cells that a tile of the wanted size is too large takes
  // smaller tiles, and the CSR kernels if none fits.
  if (params->kernel_path == 0 && !params->strong_bc) {
    if (params->block_fu > tsm::stage_block_max() || params->block_grad > 512)
      return fail(TSM_E_ARG, "tiled kernels: block size out of range");
    int want = -1;
    if ((rc = create_with_tiles(mesh, params, n_samples, want, out)) != 1) return rc;
    for (int tb = want / 2; tb >= 16; tb /= 2)
      if ((rc = create_with_tiles(mesh, params, n_samples, tb, out)) != 1) return rc;
  }
  int csr = 0;
  return create_with_tiles(mesh, params, n_samples, csr, out);
}

namespace {
// Owned vertices per tile where the caller leaves it open: 128, or 112 where viscous
// cells share LDS with gradients: 50 KB then, three tiles per CU instead of two (57
// KB).  A no-slip channel with KEPES-TeCNO Roe and minmod, per step: 257^2 68 us
// against 86, 400^2 119 against 142, 640^2 234 against 281; 96 vertices 69, 140, 269.
// Euler at 513^2: 128 110 us, 112 112.  A quarter of it has to hold a periodic set.
int default_tile(const tsm_params& p, size_t largest_set) {
  if (p.tile_vertices > 0) return p.tile_vertices;
  return p.model == 1 && tsm::stage_has_gradients(p.flux, p.reconstruct) && largest_set <= 112 / 4 ? 112 : 128;
}

int create_with_tiles(const tsm_mesh* mesh, const tsm_params* params, int n_samples, int& tb,
                      tsm_ctx** out) {
  int rc = TSM_OK;
  tsm_ctx* c = new tsm_ctx();
  c->P = *params;
  c->S = n_samples;
  if (hipGetDevice(&c->dev) != hipSuccess) { delete c; return fail(TSM_E_HIP, "hipGetDevice failed"); }
  hipError_t he = hipStreamCreateWithFlags(&c->st, hipStreamNonBlocking);
  if (he != hipSuccess) { delete c; return fail(TSM_E_HIP, "hipStreamCreate failed"); }
  std::string msg;
  int grc = 1;  // median duals: geometry on the device unless the host is asked for
  if (params->cell_type == 0 && !params->host_preprocess) {
    grc = tsm::build_geometry_device(*mesh, c->geo, c->st, msg);
    if (grc < 0) { delete c; return fail(grc, msg); }
  }
  if (grc == 1 && !tsm::build_geometry(*mesh, params->cell_type, c->geo, msg)) {
    delete c;
    return fail(TSM_E_MESH, msg);
  }
  const tsm::Geometry& g = c->geo;
  const int nv = g.nv, nc = g.nc, nf = (int)g.face.size(), nb = (int)g.bface.size();
  bool wall_cells = false;  // Navier-Stokes cells with a non-periodic bface
  if (params->model == 1)
    for (int k = 0; k < nc; ++k) wall_cells = wall_cells || g.cell_has_nonper_bface[k];
  if ((size_t)nf >= (1u << 30) || (size_t)nb >= (1u << 30)) {
    delete c;
    return fail(TSM_E_MESH, "mesh too large for 30-bit face ids");
  }
  // ---- path and vertex numbering -----------------------------------------
  size_t largest_set = 0;
  for (const auto& P : g.periodic) largest_set = std::max(largest_set, P.size());
  if (tb < 0) {
    tb = default_tile(*params, largest_set);
  } else if (tb > 0 && largest_set > (size_t)std::max(4, tb / 4)) {
    delete c;  // a smaller tile than the wanted one that no longer holds a periodic set
    return 1;
  }
  c->tiled = tb > 0;
  std::vector<int> perm(nv), inv(nv);
  tsm::TileGeo dev_tg{};   // device-built tile arrays (dev_tiles)
  bool dev_tiles = false;
  if (c->tiled) {
    if (tb > 256) { delete c; return fail(TSM_E_ARG, "tile_vertices must be <= 256"); }
    if (params->graph_steps < 0 || params->graph_steps > 4096) {
      delete c;
      return fail(TSM_E_ARG, "graph_steps must be in [0, 4096]");
    }
    const bool grad = (params->flux == 0 || params->flux == 1) && params->reconstruct != 0;
    c->two_rings_asked = grad && params->tile_fused_gradient && params->model == 0 &&
                         params->time_scheme == 0 && g.periodic.empty();
    // on the device unless the host is asked for; both give the same arrays
    int trc = 1;
    if (!params->host_preprocess) {
      auto dalloc = [c](void** p, size_t bytes) -> int {
        char* q = nullptr;
        const int r = c->alloc(&q, bytes);
        *p = q;
        return r;
      };
      trc = tsm::build_tiles_device(g, tb, c->tiling, dev_tg, dalloc, c->st, msg);
      if (trc < 0) { delete c; return fail(trc, "tiling: " + msg); }
      if (trc == 2) { delete c; return 1; }
    }
    dev_tiles = trc == 0;
    if (!dev_tiles &&
        (!tsm::build_tiles(g, tb, c->tiling, msg, false) || !tsm::validate_tiles(g, c->tiling, msg))) {
      const bool smaller = c->tiling.too_large;
      delete c;
      return smaller ? 1 : fail(TSM_E_MESH, "tiling: " + msg);
    }
    perm = c->tiling.perm;
    inv = c->tiling.inv;
  } else {
    for (int i = 0; i < nv; ++i) perm[i] = inv[i] = i;
  }
  c->perm = perm;
  if (int e = c->upload_later(&c->d_perm, perm)) { delete c; return e; }
  const size_t state_bytes = 4 * (size_t)nv * sizeof(double);
  if (state_bytes <= tsm_ctx::PIN_STATE) c->state_off = 256;
  const size_t pin_bytes = std::max(tsm_ctx::PIN, c->state_off ? c->state_off + state_bytes : 0);
  if (hipHostMalloc((void**)&c->pin, pin_bytes, hipHostMallocDefault) != hipSuccess) {
    delete c;
    return fail(TSM_E_HIP, "hipHostMalloc");
  }
  // ---- host layout (device vertex ids) -----------------------------------
  std::vector<int> fv(2 * (size_t)nf);
  std::vector<double> fn(2 * (size_t)nf);
  for (int f = 0; f < nf; ++f) {
    fv[2 * f] = perm[g.face[f].v[0]]; fv[2 * f + 1] = perm[g.face[f].v[1]];
    fn[2 * f] = g.face[f].nx; fn[2 * f + 1] = g.face[f].ny;
  }
  // vertex -> face/bface CSR in reference order
  std::vector<int> vfe_ptr(nv + 1, 0), vfe;
  for (int f = 0; f < nf; ++f) { vfe_ptr[fv[2 * f] + 1]++; vfe_ptr[fv[2 * f + 1] + 1]++; }
  for (int b = 0; b < nb; ++b)
    if (!g.bface[b].periodic) { vfe_ptr[perm[g.bface[b].v[0]] + 1]++; vfe_ptr[perm[g.bface[b].v[1]] + 1]++; }
  for (int i = 0; i < nv; ++i) vfe_ptr[i + 1] += vfe_ptr[i];
  vfe.resize(vfe_ptr[nv]);
  {
    std::vector<int> pos(vfe_ptr.begin(), vfe_ptr.end() - 1);
    for (int f = 0; f < nf; ++f) {
      vfe[pos[fv[2 * f]]++] = (int)((0u << 30) | (unsigned)f);
      vfe[pos[fv[2 * f + 1]]++] = (int)((1u << 30) | (unsigned)f);
    }
    for (int b = 0; b < nb; ++b) {
      if (g.bface[b].periodic) continue;
      vfe[pos[perm[g.bface[b].v[0]]]++] = (int)((2u << 30) | (unsigned)b);
      vfe[pos[perm[g.bface[b].v[1]]]++] = (int)((2u << 30) | (unsigned)b);
    }
  }
  // cell -> non-periodic bfaces (bface order)
  std::vector<int> cbf(2 * (size_t)nc, -1);
  for (int b = 0; b < nb; ++b) {
    if (g.bface[b].periodic) continue;
    int cl = g.bface[b].lcell;
    if (cbf[2 * cl] < 0) cbf[2 * cl] = b;
    else if (cbf[2 * cl + 1] < 0) cbf[2 * cl + 1] = b;
    else { delete c; return fail(TSM_E_MESH, "cell with three boundary faces"); }
  }
  std::vector<int> cv(3 * (size_t)nc);
  for (size_t k = 0; k < cv.size(); ++k) cv[k] = perm[g.cell[k]];
  std::vector<int> vc_ptr(nv + 1, 0), vc;
  for (int k = 0; k < nc; ++k)
    for (int j = 0; j < 3; ++j) vc_ptr[cv[3 * k + j] + 1]++;
  for (int i = 0; i < nv; ++i) vc_ptr[i + 1] += vc_ptr[i];
  vc.resize(vc_ptr[nv]);
  {
    std::vector<int> pos(vc_ptr.begin(), vc_ptr.end() - 1);
    for (int k = 0; k < nc; ++k)
      for (int j = 0; j < 3; ++j)
        vc[pos[cv[3 * k + j]]++] = (cbf[2 * k] >= 0) ? (int)(0x80000000u | (unsigned)k) : k;
  }
  std::vector<int> cnb(nc);
  for (int k = 0; k < nc; ++k) cnb[k] = (cbf[2 * k] >= 0) ? 1 : 0;
  std::vector<int> bvv(2 * (size_t)nb), btype(nb);
  std::vector<double> bn(2 * (size_t)nb), bstate(8 * (size_t)nb, 0.0);
  for (int b = 0; b < nb; ++b) {
    bvv[2 * b] = perm[g.bface[b].v[0]]; bvv[2 * b + 1] = perm[g.bface[b].v[1]];
    bn[2 * b] = g.bface[b].nx; bn[2 * b + 1] = g.bface[b].ny;
    btype[b] = g.bface[b].bc;
    for (int i = 0; i < mesh->n_bc; ++i)
      if (mesh->bc_tag[i] == g.bface[b].tag) {
        for (int k = 0; k < 4; ++k)  // both end points take the tag's constant state
          bstate[8 * b + k] = bstate[8 * b + 4 + k] = mesh->bc_state ? mesh->bc_state[4 * i + k] : 0.0;
        if (btype[b] == TSM_BC_NOSLIP && mesh->bc_adiabatic && mesh->bc_adiabatic[i])
          btype[b] = tsm::BC_NOSLIP_ADIABATIC;
      }
  }
  std::vector<double> xs(nv), ys(nv), dca(nv), gfact(nv), wgt(nv);
  std::vector<int> pset(nv);
  for (int i = 0; i < nv; ++i) {
    int o = inv[i];
    xs[i] = g.x[o]; ys[i] = g.y[o]; dca[i] = g.dcarea[o]; wgt[i] = g.weight[o];
    gfact[i] = 1.0 / (6.0 * g.mcarea[o]);
    pset[i] = g.periodic_of[o];
  }
  std::vector<int> pptr(1, 0), pv;
  for (auto& P : g.periodic) { for (int v : P) pv.push_back(perm[v]); pptr.push_back((int)pv.size()); }

  // Navier-Stokes wall cells (src/fv.cc:1236-1312): each cell's boundary edges
  // in its slot order with their bfaces, and per vertex the bfaces, in bface
  // order, whose cell holds the vertex (the order the reference's bface loop
  // adds the cell and wall fluxes in)
  std::vector<int> blc(std::max(nb, 1), -1), cwf(2 * (size_t)nc, -1), cwb(2 * (size_t)nc, -1);
  std::vector<int> vbe_ptr(nv + 1, 0), vbe;
  if (wall_cells) {
    std::vector<int> face_bface(nf, -1);
    {
      std::vector<std::pair<long long, int>> key;
      for (int b = 0; b < nb; ++b) {
        if (g.bface[b].periodic) continue;
        int a0 = g.bface[b].v[0], a1 = g.bface[b].v[1];
        key.push_back({(long long)std::min(a0, a1) * nv + std::max(a0, a1), b});
      }
      std::sort(key.begin(), key.end());
      for (int f = 0; f < nf; ++f) {
        if (g.face[f].type < 0 || g.face[f].periodic) continue;
        int a0 = g.face[f].v[0], a1 = g.face[f].v[1];
        long long k = (long long)std::min(a0, a1) * nv + std::max(a0, a1);
        auto it = std::lower_bound(key.begin(), key.end(), std::make_pair(k, -1));
        if (it == key.end() || it->first != k) { delete c; return fail(TSM_E_MESH, "boundary edge without a bface"); }
        face_bface[f] = it->second;
      }
    }
    for (int k = 0; k < nc; ++k) {
      int t = 0;
      for (int j = 0; j < 3; ++j) {
        // slots keep their indices into the face list as it was before Voronoi
        // duals lost their empty faces (src/grid_preproc.cc:633-647, :811-831);
        // boundary faces come first and are never removed (build_geometry
        // refuses a dual that would lose one), so a slot past the shortened
        // list, like any slot past the boundary faces, is interior
        int f = g.cell_slot_face[3 * k + j];
        if (f < 0 || f >= nf || face_bface[f] < 0) continue;
        if (t == 2) { delete c; return fail(TSM_E_MESH, "cell with three boundary edges"); }
        cwf[2 * k + t] = f;
        cwb[2 * k + t] = face_bface[f];
        ++t;
      }
    }
    for (int b = 0; b < nb; ++b) {
      if (g.bface[b].periodic) continue;
      blc[b] = g.bface[b].lcell;
      for (int j = 0; j < 3; ++j) vbe_ptr[cv[3 * blc[b] + j] + 1]++;
    }
    for (int i = 0; i < nv; ++i) vbe_ptr[i + 1] += vbe_ptr[i];
    vbe.resize(vbe_ptr[nv]);
    std::vector<int> pos(vbe_ptr.begin(), vbe_ptr.end() - 1);
    for (int b = 0; b < nb; ++b) {
      if (g.bface[b].periodic) continue;
      for (int j = 0; j < 3; ++j) {
        int v = cv[3 * blc[b] + j];
        bool on = v == bvv[2 * b] || v == bvv[2 * b + 1];
        vbe[pos[v]++] = (int)((on ? 0x80000000u : 0u) | (unsigned)b);
      }
    }
  }
  if (vbe.empty()) vbe.push_back(0);
  // ---- device ------------------------------------------------------------
  tsm::DevGeo& G = c->G;
  G.nv = nv; G.nf = nf; G.nb = nb; G.nc = nc;
#define UP(field, vec) do { if ((rc = c->upload_later(&G.field, vec))) { delete c; return rc; } } while (0)
  UP(x, xs); UP(y, ys); UP(dcarea, dca); UP(gfact, gfact); UP(weight, wgt);
  UP(carea, g.cell_area);
  UP(fv, fv); UP(fn, fn); UP(vfe_ptr, vfe_ptr); UP(vfe, vfe); UP(vc_ptr, vc_ptr); UP(vc, vc);
  UP(cv, cv); UP(cbf, cbf); UP(cnb, cnb); UP(bv, bvv); UP(bn, bn); UP(btype, btype);
  UP(bstate, bstate); UP(pset, pset); UP(pptr, pptr); UP(pv, pv);
  G.bs_sample = 0;
  c->h_btype = btype;
  if (mesh->n_bface != nb) { delete c; return fail(TSM_E_MESH, "boundary face count changed in preprocessing"); }
  {
    std::vector<std::pair<long long, int>> key(nb);
    for (int b = 0; b < nb; ++b) {
      int a0 = g.bface[b].v[0], a1 = g.bface[b].v[1];
      key[b] = {(long long)std::min(a0, a1) * nv + std::max(a0, a1), b};
    }
    std::sort(key.begin(), key.end());
    c->bmap.assign(2 * (size_t)nb, 0);
    for (int bi = 0; bi < nb; ++bi) {
      int a0 = mesh->bface_v[2 * bi], a1 = mesh->bface_v[2 * bi + 1];
      long long k = (long long)std::min(a0, a1) * nv + std::max(a0, a1);
      auto it = std::lower_bound(key.begin(), key.end(), std::make_pair(k, -1));
      if (it == key.end() || it->first != k) { delete c; return fail(TSM_E_MESH, "bface lost in preprocessing"); }
      const int bd = it->second;
      for (int e = 0; e < 2; ++e)
        c->bmap[2 * bi + e] = 8LL * bd + 4 * (g.bface[bd].v[1] == mesh->bface_v[2 * bi + e] ? 1 : 0);
    }
  }
  UP(blc, blc); UP(cwf, cwf); UP(cwb, cwb); UP(vbe_ptr, vbe_ptr); UP(vbe, vbe);
  if (params->strong_bc) {  // boundary vertices with their bfaces in bface order
    std::vector<std::vector<int>> vb(nv);
    std::vector<unsigned char> noslip(nv, 0);
    for (int b = 0; b < nb; ++b)
      for (int e = 0; e < 2; ++e) {
        const int v = bvv[2 * b + e];
        vb[v].push_back(b);
        if (btype[b] == TSM_BC_NOSLIP || btype[b] == tsm::BC_NOSLIP_ADIABATIC) noslip[v] = 1;
      }
    std::vector<int> sbv, sb_ptr(1, 0), sb;
    for (int v = 0; v < nv; ++v) {
      if (vb[v].empty()) continue;
      sbv.push_back(v);
      sb.insert(sb.end(), vb[v].begin(), vb[v].end());
      sb_ptr.push_back((int)sb.size());
    }
    G.strong = 1;
    G.nsbv = (int)sbv.size();
    if (sbv.empty()) { sbv.push_back(0); sb.push_back(0); }
    UP(sbv, sbv); UP(sb_ptr, sb_ptr); UP(sb, sb); UP(snoslip, noslip);
  }
#undef UP
  if (c->tiled) {
    const tsm::Tiling& T = c->tiling;
    tsm::TileGeo TG{};
    TG.ntiles = T.ntiles; TG.tb = T.tb;
    TG.n_periodic_tiles = T.n_periodic_tiles;
    TG.nhalo = dev_tiles ? dev_tg.nhalo : (int)T.halo.size();
    TG.fu_block = std::max(0, params->block_fu);
    // block_grad has had no kernel of its own since the stage kernel forms the
    // gradients; its range is still checked
    const int bg = std::max(((T.tb + 63) / 64) * 64, std::max(0, params->block_grad));
    tsm::StageTab probe{};
    probe.tb = T.tb; probe.mf = T.max_faces; probe.fu_block = TG.fu_block;
    const int bf = tsm::stage_block(probe);
    if (bf > tsm::stage_block_max()) {  // more faces than its threads take
      delete c;
      return 1;
    }
    if (bf % 64 || bg > 512 || bg % 64) {
      delete c;
      return fail(TSM_E_ARG, "tiled kernels: block size out of range (blocks " + std::to_string(bg) + "/" +
                                 std::to_string(bf) + ")");
    }
#define UT(field, vec) do { if ((rc = c->upload_later(&TG.field, vec))) { delete c; return rc; } } while (0)
    if (dev_tiles) {
      TG.vbeg = dev_tg.vbeg; TG.hbeg = dev_tg.hbeg; TG.halo = dev_tg.halo; TG.fbeg = dev_tg.fbeg;
      TG.bbeg = dev_tg.bbeg; TG.tbf = dev_tg.tbf; TG.gptr = dev_tg.gptr;
      TG.tper = dev_tg.tper; TG.pinfo = dev_tg.pinfo; TG.f_lr = dev_tg.f_lr;
      TG.f_n = dev_tg.f_n; TG.gent = dev_tg.gent;
    } else {
      UT(vbeg, T.vbeg); UT(hbeg, T.hbeg); UT(halo, T.halo); UT(fbeg, T.fbeg); UT(bbeg, T.bbeg);
      UT(tbf, T.tbf); UT(gptr, T.gptr); UT(tper, T.tper);
      UT(pinfo, T.pinfo); UT(f_lr, T.f_lr); UT(f_n, T.f_n); UT(gent, T.gent);
    }
#undef UT
    auto dalloc = [c](void** p, size_t bytes) -> int {
      char* q = nullptr;
      const int r = c->alloc(&q, bytes);
      *p = q;
      return r;
    };
    if ((rc = c->upload_now())) { delete c; return rc; }
    rc = tsm::build_stage_tables(c->G, TG, tsm::stage_has_gradients(params->flux, params->reconstruct),
                                 params->model == 1, wall_cells ? (int)vbe.size() : 0, c->ST, dalloc,
                                 c->st, msg);
    // the static LDS of the kernel and its launches fit beside this much
    if (rc == 0 && tsm::stage_lds(c->ST) > 156 * 1024)
      rc = 1;
    if (rc) {
      delete c;
      return rc == 1 ? 1 : fail(rc, msg);
    }
  }
  tsm::StageArgs& A = c->A;
  const int S = n_samples;
  A.cs = (size_t)S * nv;
  A.fs = (size_t)S * nf;
  A.off = 0;
  c->nblk_v = (nv + 255) / 256;
  const size_t cs = A.cs;
#define AL(ptr, n) do { if ((rc = c->alloc(&(ptr), (n)))) { delete c; return rc; } } while (0)
  AL(c->W[0], 4 * cs); AL(c->W[1], 4 * cs); AL(c->W[2], 4 * cs);
  if (c->tiled && tsm::stage_keeps_var0(params->flux))
    for (auto& v : c->V) AL(v, cs);
  AL(c->E[0], 4 * cs); AL(c->E[1], 4 * cs);
  AL(A.Uold, 4 * cs); AL(A.dE, 8 * cs); AL(A.F, 4 * A.fs); AL(A.R, 4 * cs);
  if (params->time_scheme == 1) AL(A.R2, 4 * cs);
  if (!params->unsteady) AL(A.dtl, cs);  // local time steps (src/fv.cc:1591-1618)
  if (params->liou_fix) AL(A.ssw, cs);
  AL(A.partial, (size_t)S * std::max(c->nblk_v, c->tiling.ntiles) * 4);
  if (c->tiled) AL(c->dtpart, (size_t)S * c->tiling.ntiles);
  AL(c->bad, 1);
#undef AL
  // time stamps of an unsteady run (src/fv.cc:50-60); a steady run has none
  // and no final time (src/parameter.cc:250-252)
  const int n_stamps = params->unsteady ? params->n_time_stamps : 1;
  const double final_time = params->unsteady ? params->final_time : 1.0e20;
  std::vector<double> tst(n_stamps + 1);
  double tdt = final_time / n_stamps;
  for (size_t i = 0; i < tst.size(); ++i) tst[i] = i * tdt;
  c->h_gamma.assign(S, params->gamma);
  c->h_R.assign(S, params->gas_const);
  std::vector<double> gc;  // load_gas
  for (int k = 0; k < S; ++k) { gc.push_back(1.0 / (params->gamma - 1.0)); gc.push_back(1.0 / params->gamma); }
  A.log = nullptr; A.log_cap = 0;
  A.fo = tsm::FluxOpts{params->ev_alpha, params->ev_beta, params->tvb_M, params->nd_active};
  A.vp = tsm::ViscParams{params->mu_ref, params->T_ref, params->T_0, params->omega,
                         params->prandtl, 1.0 / params->prandtl, params->mu_model, params->visc_active,
                         params->heat_active};
  A.ns = params->model == 1;
  A.ns_walls = wall_cells;
  A.heun = params->time_scheme == 2;
  A.scheme = params->time_scheme;
  A.ns_samples = S;
  A.ignore_done = 0;
  c->SP = tsm::StepParams{params->min_residue, final_time, params->time_step,
                          params->cfl, (long long)params->max_iter, params->unsteady, n_stamps};
  std::vector<tsm::Ctl> ctl(S);
  for (auto& q : ctl) { q = tsm::Ctl{}; q.res_total = 1e20; q.counter = 1; q.done = 1; }
#define UA(field, vec) do { if ((rc = c->upload_later(&A.field, vec))) { delete c; return rc; } } while (0)
  UA(tstamps, tst); UA(gamma, c->h_gamma); UA(gasR, c->h_R); UA(gasc, gc); UA(ctl, ctl);
  const bool folds = c->tiled && tsm::stage_ends_step(c->tiling.ntiles, S);
  if (folds) UA(arrive, std::vector<int>(S, 0));
#undef UA
  if ((rc = c->upload_now())) { delete c; return rc; }
  c->bind_state();
  *out = c;
  return TSM_OK;
}
}  // namespace

extern "C" void tsm_destroy(tsm_ctx* c) { delete c; }

extern "C" int tsm_tile_vertices(const tsm_ctx* c) { return !c ? -1 : c->tiled ? c->ST.tb : 0; }

namespace {
// Gives every sample a block of boundary values of its own (they share one
// until a sample's values differ).
int own_bstate(tsm_ctx* c) {
  if (c->G.bs_sample != 0 || c->S == 1) return TSM_OK;
  const int nb = c->G.nb;
  double* all = nullptr;
  int rc = c->alloc(&all, (size_t)c->S * 8 * nb);
  if (rc) return rc;
  HIP_TRY(hipStreamSynchronize(c->st));
  for (int k = 0; k < c->S; ++k)
    HIP_TRY(hipMemcpy(all + (size_t)k * 8 * nb, c->G.bstate, 8 * (size_t)nb * sizeof(double),
                      hipMemcpyDeviceToDevice));
  c->G.bstate = all;
  c->G.bs_sample = 8LL * nb;
  if (c->gexec) { (void)hipGraphExecDestroy(c->gexec); c->gexec = nullptr; }  // captured the old array
  return TSM_OK;
}
}  // namespace

extern "C" int tsm_set_bc_state(tsm_ctx* c, int s, const double* state) {
  if (!c || !state || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  const int nb = c->G.nb;
  std::vector<double> h(8 * (size_t)nb, 0.0);
  for (int bi = 0; bi < nb; ++bi)
    for (int e = 0; e < 2; ++e) {
      const double* q = state + 8 * (size_t)bi + 4 * e;
      const long long o = c->bmap[2 * bi + e];
      const int type = c->h_btype[o / 8];
      for (int k = 0; k < 4; ++k)
        if (!std::isfinite(q[k])) return fail(TSM_E_STATE, "non-finite boundary value at bface " + std::to_string(bi));
      const bool needT = type == TSM_BC_INLET || type == TSM_BC_FARFIELD || type == TSM_BC_NOSLIP;
      const bool needp = type == TSM_BC_INLET || type == TSM_BC_FARFIELD || type == TSM_BC_PRESSURE;
      if ((needT && !(q[0] > 0.0)) || (needp && !(q[3] > 0.0)))
        return fail(TSM_E_STATE, "non-positive boundary T or p at bface " + std::to_string(bi));
      for (int k = 0; k < 4; ++k) h[o + k] = q[k];
    }
  if (c->S > 1) {  // samples stop sharing one block
    int rc = own_bstate(c);
    if (rc) return rc;
  }
  HIP_TRY(hipStreamSynchronize(c->st));
  HIP_TRY(hipMemcpy(const_cast<double*>(c->G.bstate) + (size_t)s * c->G.bs_sample, h.data(),
                    h.size() * sizeof(double), hipMemcpyHostToDevice));
  return TSM_OK;
}

extern "C" int tsm_set_bc_time_expr(tsm_ctx* c, const int* bface_group, int n_groups,
                                    const char* const* expr, int n_const,
                                    const char* const* const_name, const double* const_value) {
  if (!c || n_groups < 0 || (n_groups > 0 && (!bface_group || !expr)) || n_const < 0 ||
      (n_const > 0 && (!const_name || !const_value)))
    return fail(TSM_E_ARG, "bad argument");
  if (n_groups == 0) {
    c->bt = tsm::BcTime{};
    if (c->gexec) { (void)hipGraphExecDestroy(c->gexec); c->gexec = nullptr; }
    return TSM_OK;
  }
  // the reference advances the boundaries' time only in Heun's scheme; the
  // other schemes leave int_step_time unset (src/fv.cc:2294-2299)
  if (c->P.time_scheme != 2 || !c->P.unsteady)
    return fail(TSM_E_ARG, "time-dependent boundary values need an unsteady run with time_scheme heuns");
  std::map<std::string, double> consts;
  for (int k = 0; k < n_const; ++k) {
    if (!const_name[k]) return fail(TSM_E_ARG, "null constant name");
    consts[const_name[k]] = const_value[k];
  }
  // one program per group and field (T, u, v, p), none where no text is given
  std::vector<tsm::Expr> ex(4 * (size_t)n_groups);
  std::vector<int> code, pbeg(4 * (size_t)n_groups, -1);
  for (int g = 0; g < 4 * n_groups; ++g) {
    if (!expr[g] || !expr[g][0]) continue;
    std::string err;
    std::vector<int> pc;
    int depth = 0;
    if (!ex[g].parse(expr[g], consts, err) || !ex[g].time_program(pc, depth, err))
      return fail(TSM_E_ARG, "boundary group " + std::to_string(g / 4) + ": " + err);
    pbeg[g] = (int)code.size();
    code.insert(code.end(), pc.begin(), pc.end());
  }
  // entries: every end point of every bface in a group, each given field
  const int nb = c->G.nb;
  std::vector<int> target, prog, slot;
  std::vector<double> slots;
  for (int bi = 0; bi < nb; ++bi) {
    const int g = bface_group[bi];
    if (g < 0) continue;
    if (g >= n_groups) return fail(TSM_E_ARG, "bface " + std::to_string(bi) + ": group out of range");
    for (int e = 0; e < 2; ++e) {
      const long long o = c->bmap[2 * bi + e];
      const int v = c->geo.bface[o / 8].v[(o % 8) / 4];
      for (int q = 0; q < 4; ++q) {
        const int k = 4 * g + q;
        if (pbeg[k] < 0) continue;
        target.push_back((int)o + q);
        prog.push_back(pbeg[k]);
        slot.push_back((int)slots.size());
        for (int j = 0; j < ex[k].n_time_slots(); ++j)
          slots.push_back(ex[k].time_slot(j, c->geo.x[v], c->geo.y[v]));
      }
    }
  }
  int rc = own_bstate(c);
  if (rc) return rc;
  tsm::BcTime B{};
  B.n = (int)target.size();
  if ((rc = c->upload(&B.target, target)) || (rc = c->upload(&B.prog, prog)) ||
      (rc = c->upload(&B.slot, slot)) || (rc = c->upload(&B.code, code)) ||
      (rc = c->upload(&B.slots, slots)))
    return rc;
  c->bt = B;
  if (c->gexec) { (void)hipGraphExecDestroy(c->gexec); c->gexec = nullptr; }  // captured without them
  // the values at the samples' current time
  tsm::StageArgs A = c->A;
  A.ignore_done = 1;
  tsm::launch_bc_time(c->G, c->bt, A, c->S, 0, c->st);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->st));
  return TSM_OK;
}

extern "C" int tsm_set_sample_material(tsm_ctx* c, int s, double gamma, double R) {
  if (!c || s < 0 || s >= c->S || !(gamma > 1.0) || !(R > 0.0)) return fail(TSM_E_ARG, "bad argument");
  c->h_gamma[s] = gamma; c->h_R[s] = R;
  tsm::launch_set_gas(c->A, s, tsm::Gas{gamma, R, 1.0 / (gamma - 1.0), 1.0 / gamma}, c->st);
  c->bind_state();  // the stored entropy variables are those of the old constants
  if (c->tiled) c->e_valid = false;
  else tsm::launch_prim2ent(c->G, c->A, s, c->st);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->st));
  return TSM_OK;
}

extern "C" int tsm_set_state(tsm_ctx* c, int s, const double* prim) {
  if (!c || !prim || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  const int nv = c->G.nv;
  const size_t off = (size_t)s * nv;
  if (c->tiled) {
    c->state_ready();
    c->e_valid = false;
  } else {
    c->csr_ready();
  }
  const size_t bytes = 4 * (size_t)nv * sizeof(double);
  int* bad = reinterpret_cast<int*>(c->pin);
  double* in;
  if (c->state_off) {
    in = reinterpret_cast<double*>(c->pin + c->state_off);
    std::memcpy(in, prim, bytes);
  } else {
    in = c->W[c->cur == 2 ? 0 : 2];  // free between steps
    HIP_TRY(hipMemcpyAsync(in, prim, bytes, hipMemcpyHostToDevice, c->st));
  }
  tsm::launch_state_put(nv, c->d_perm, in, c->bad, c->W[c->cur] + 4 * off,
                        c->A.W_keep ? c->A.W_keep + 4 * off : nullptr, c->A.ctl + s, c->st);
  tsm::launch_words(sizeof(int), c->bad, bad, c->st);
  // a refused state leaves these too: under bc_scheme strong they are not those of
  // the state (the boundary values imposed on it come after them)
  if (!c->tiled) tsm::launch_prim2ent(c->G, c->A, s, c->st, c->bad);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->st));
  const int i = *bad;
  if (i != INT_MAX) {
    if (!(prim[4 * (size_t)i] > 0.0) || !(prim[4 * (size_t)i + 3] > 0.0) || !std::isfinite(prim[4 * (size_t)i]) ||
        !std::isfinite(prim[4 * (size_t)i + 3]))
      return fail(TSM_E_STATE, "initial temperature and pressure must be positive and finite "
                               "(vertex " + std::to_string(i) + ")");
    return fail(TSM_E_STATE, "initial velocity is not finite (vertex " + std::to_string(i) + ")");
  }
  return TSM_OK;
}

namespace {
// Vertex arrays are array-of-structs with ncomp doubles per vertex.
int download_vec(tsm_ctx* c, const double* base, int ncomp, int s, double* out) {
  const int nv = c->G.nv;
  const size_t off = (size_t)s * nv;
  std::vector<double> aos((size_t)ncomp * nv);
  HIP_TRY(hipStreamSynchronize(c->st));
  HIP_TRY(hipMemcpy(aos.data(), base + (size_t)ncomp * off, aos.size() * sizeof(double),
                    hipMemcpyDeviceToHost));
  for (int i = 0; i < nv; ++i)
    for (int k = 0; k < ncomp; ++k) out[(size_t)ncomp * i + k] = aos[(size_t)ncomp * c->perm[i] + k];
  return TSM_OK;
}
}  // namespace

extern "C" int tsm_get_state(tsm_ctx* c, int s, double* prim) {
  if (!c || !prim || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  const size_t bytes = 4 * (size_t)c->G.nv * sizeof(double);
  const bool small = c->state_off > 0;
  double* out = small ? reinterpret_cast<double*>(c->pin + c->state_off)
                      : c->W[c->cur == 2 ? 0 : 2];  // free between steps
  tsm::launch_state_get(c->G.nv, c->d_perm, c->W[c->cur] + 4 * (size_t)s * c->G.nv, out, c->st);
  HIP_TRY(hipGetLastError());
  if (!small) HIP_TRY(hipMemcpyAsync(prim, out, bytes, hipMemcpyDeviceToHost, c->st));
  HIP_TRY(hipStreamSynchronize(c->st));
  if (small) std::memcpy(prim, out, bytes);
  return TSM_OK;
}

extern "C" int tsm_gradients(tsm_ctx* c, int s, double* dE) {
  if (!c || !dE || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  c->sample_ready(s);
  c->A.ignore_done = 1;
  tsm::launch_gradient_one(c->G, c->A, s, c->st);
  c->A.ignore_done = 0;
  HIP_TRY(hipGetLastError());
  return download_vec(c, c->A.dE, 8, s, dE);
}

extern "C" int tsm_forces(tsm_ctx* c, int s, int force_index, const int* tags, int ntags,
                          double* out) {
  const int nb = c ? c->G.nb : 0;
  if (!c || !out || s < 0 || s >= c->S || ntags < 1 || !tags || force_index < 0 ||
      force_index >= nb)
    return fail(TSM_E_ARG, "bad argument");
  std::vector<int> sel;
  for (int b = 0; b < nb; ++b)
    for (int k = 0; k < ntags; ++k)
      if (c->geo.bface[b].tag == tags[k]) { sel.push_back(b); break; }
  if (sel.empty()) return fail(TSM_E_ARG, "no boundary face has the force's tags");
  if (c->force_cap < sel.size()) {
    int rc = c->alloc(&c->force_buf, 4 * sel.size() + 4);
    if (rc) return rc;
    rc = c->alloc(&c->force_sel, sel.size());
    if (rc) return rc;
    c->force_cap = sel.size();
  }
  c->sample_ready(s);
  HIP_TRY(hipMemcpyAsync(c->force_sel, sel.data(), sel.size() * sizeof(int), hipMemcpyHostToDevice,
                         c->st));
  c->A.ignore_done = 1;
  if (c->P.model == 1) tsm::launch_gradient_one(c->G, c->A, s, c->st);
  c->A.ignore_done = 0;
  tsm::launch_forces(c->G, c->A, s, force_index, c->force_sel, (int)sel.size(), c->P.model == 1,
                     c->force_buf + 4, c->force_buf, c->st);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpyAsync(out, c->force_buf, 4 * sizeof(double), hipMemcpyDeviceToHost, c->st));
  HIP_TRY(hipStreamSynchronize(c->st));
  return TSM_OK;
}

extern "C" int tsm_keep_stage_state(tsm_ctx* c, int on) {
  if (!c) return fail(TSM_E_ARG, "bad argument");
  if (on && !c->A.W_keep) {
    if (!c->W_keep) {
      int rc = c->alloc(&c->W_keep, 4 * c->A.cs);
      if (rc) return rc;
    }
    c->state_ready();
    HIP_TRY(hipMemcpyAsync(c->W_keep, c->W[c->cur], 4 * c->A.cs * sizeof(double),
                           hipMemcpyDeviceToDevice, c->st));
    c->A.W_keep = c->W_keep;
  } else if (!on) {
    c->A.W_keep = nullptr;
  }
  // a captured step graph holds the stage kernels' arguments
  if (c->gexec) { (void)hipGraphExecDestroy(c->gexec); c->gexec = nullptr; }
  HIP_TRY(hipStreamSynchronize(c->st));
  return TSM_OK;
}

namespace {
// Vertex gradients of sample s into its slice of A.dE: of the kept last-stage
// input state (stage) or of the current state.
int sample_gradients(tsm_ctx* c, int s, bool stage) {
  if (stage && !c->A.W_keep)
    return fail(TSM_E_ARG, "the last stage's state is not kept (tsm_keep_stage_state)");
  if (stage) c->state_ready();
  else c->sample_ready(s);
  tsm::StageArgs K = c->A;
  K.ignore_done = 1;
  if (stage) {  // entropy variables of the kept state in the scratch entropy buffer
    K.W_in = c->A.W_keep;
    K.E_in = c->E[c->cur ^ 1];
    tsm::launch_prim2ent(c->G, K, s, c->st);
  }
  tsm::launch_gradient_one(c->G, K, s, c->st);
  HIP_TRY(hipGetLastError());
  return TSM_OK;
}
}  // namespace

extern "C" int tsm_stage_gradients(tsm_ctx* c, int s, double* dE) {
  if (!c || !dE || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  int rc = sample_gradients(c, s, true);
  if (rc) return rc;
  return download_vec(c, c->A.dE, 8, s, dE);
}

extern "C" int tsm_surface(tsm_ctx* c, int s, int stage, const int* tags, int ntags, double* out) {
  const int nb = c ? c->G.nb : 0;
  if (!c || !out || s < 0 || s >= c->S || ntags < 0 || (ntags > 0 && !tags))
    return fail(TSM_E_ARG, "bad argument");
  std::vector<int> sel;
  for (int b = 0; b < nb; ++b)
    for (int k = 0; k < ntags; ++k)
      if (c->geo.bface[b].tag == tags[k]) { sel.push_back(b); break; }
  if (sel.empty()) return TSM_OK;
  if (c->force_cap < sel.size()) {
    int rc = c->alloc(&c->force_buf, 4 * sel.size() + 4);
    if (rc) return rc;
    rc = c->alloc(&c->force_sel, sel.size());
    if (rc) return rc;
    c->force_cap = sel.size();
  }
  int rc = sample_gradients(c, s, stage != 0);
  if (rc) return rc;
  HIP_TRY(hipMemcpyAsync(c->force_sel, sel.data(), sel.size() * sizeof(int), hipMemcpyHostToDevice,
                         c->st));
  tsm::launch_surface(c->G, c->A, s, c->force_sel, (int)sel.size(), c->force_buf, c->st);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpyAsync(out, c->force_buf, 2 * sel.size() * sizeof(double), hipMemcpyDeviceToHost,
                         c->st));
  HIP_TRY(hipStreamSynchronize(c->st));
  return TSM_OK;
}

extern "C" int tsm_residual(tsm_ctx* c, int s, double* R) {
  if (!c || !R || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  c->csr_ready();
  c->A.ignore_done = 1;
  if (c->P.liou_fix) tsm::launch_ssw(c->G, c->A, c->S, c->st);
  tsm::launch_gradient(c->G, c->A, c->S, c->st);
  tsm::launch_flux_update(c->P.flux, c->P.reconstruct, c->G, c->A, c->S, 0, 0, 0, c->st, true, true);
  c->A.ignore_done = 0;
  HIP_TRY(hipGetLastError());
  return download_vec(c, c->A.R, 4, s, R);
}

extern "C" int tsm_compute_dt(tsm_ctx* c, int s, double* dt) {
  if (!c || !dt || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  c->bind_state();
  c->A.ignore_done = 1;
  tsm::launch_dt(c->G, c->A, c->SP, c->S, c->st);
  c->A.ignore_done = 0;
  HIP_TRY(hipGetLastError());
  tsm::Ctl q;
  HIP_TRY(hipStreamSynchronize(c->st));
  HIP_TRY(hipMemcpy(&q, c->A.ctl + s, sizeof(q), hipMemcpyDeviceToHost));
  *dt = q.dt;
  return TSM_OK;
}

namespace {
// One full time step for every live sample with the CSR-gather kernels
// (src/fv.cc:2277-2316).
// dt_ready: the caller already ran the time-step pass (which also stores
// U_old) and may have adjusted dt.
void enqueue_step(tsm_ctx* c, int log_slot, bool dt_ready = false) {
  const int nrk = c->P.time_scheme == 0 ? 3 : (c->P.time_scheme == 1 ? 4 : 2);
  const int mode = c->P.time_scheme == 1 ? 2 : 1;
  c->bind_state();
  if (!dt_ready) tsm::launch_dt(c->G, c->A, c->SP, c->S, c->st);
  if (c->P.liou_fix) tsm::launch_ssw(c->G, c->A, c->S, c->st);
  for (int r = 0; r < nrk; ++r) {
    c->bind_state();
    tsm::launch_bc_time(c->G, c->bt, c->A, c->S, r, c->st);
    tsm::launch_gradient(c->G, c->A, c->S, c->st);
    tsm::launch_flux_update(c->P.flux, c->P.reconstruct, c->G, c->A, c->S, r, r == nrk - 1, mode,
                            c->st, true, true);
    if (c->P.strong_bc) tsm::launch_strong_bc(c->G, c->A, c->S, c->st);
    c->cur ^= 1;
  }
  c->bind_state();
  tsm::launch_step_final(c->G, c->A, c->SP, c->S, log_slot, c->st);
}

// One SSP-RK3 step with the tiled kernels.  W[cur] holds W^n throughout; the
// stages write the two other buffers and the last one writes W^{n+1} back
// in place (each vertex reads its own W^n for U_old before overwriting it).
void enqueue_tiled_step(tsm_ctx* c, int log_slot, hipEvent_t* ev = nullptr) {
  const int ia = (c->cur + 1) % 3, ib = (c->cur + 2) % 3;
  double* Wn = c->W[c->cur];
  // stage buffers: every stage reads W^n for U_old, the last one writes W^{n+1}
  // over it in place; SSP-RK3 and RK4 rotate through two scratch buffers
  const int nrk = c->P.time_scheme == 0 ? 3 : (c->P.time_scheme == 1 ? 4 : 2);
  int ins[4] = {c->cur, ia, ib, ia}, outs[4] = {ia, ib, ia, c->cur};
  if (nrk == 3) outs[2] = c->cur;
  if (nrk == 2) outs[1] = c->cur;
  int e = 0;
  if (c->P.liou_fix) {  // the step's Liou sensor from W^n (src/fv.cc:2281-2285)
    c->A.W_in = Wn;
    tsm::launch_ssw(c->G, c->A, c->S, c->st);
  }
  for (int r = 0; r < nrk; ++r) {
    c->A.W_in = c->W[ins[r]];
    c->A.W_out = c->W[outs[r]];
    c->A.V_in = c->V[ins[r]];
    c->A.V_out = c->V[outs[r]];
    tsm::launch_bc_time(c->G, c->bt, c->A, c->S, r, c->st);
    if (ev) (void)hipEventRecord(ev[e++], c->st);
    tsm::launch_stage(c->P.flux, c->P.reconstruct, c->G, c->ST, c->A, c->SP, Wn, c->dtpart, c->S, r,
                      r == nrk - 1, log_slot, c->st);
  }
  if (ev) (void)hipEventRecord(ev[e++], c->st);
  tsm::launch_step_final_tiled(c->G, c->A, c->SP, c->S, c->ST.ntiles, c->dtpart, log_slot, c->st);
  if (ev) (void)hipEventRecord(ev[e++], c->st);
  c->bind_state();
  c->e_valid = false;
}

// Steps of the current path; the tiled path first forms dt and the loop
// test of the first step with the CSR time-step kernel.
// One HIP graph of graph_steps tiled steps: every kernel argument of a step is
// fixed (the last stage writes W^n in place) and each sample's stop flag lives
// on the device, so the graph replays as it was captured.  Recaptured if the
// state buffer changes.
hipError_t tiled_graph(tsm_ctx* c) {
  if (c->gexec && c->gcur == c->cur) return hipSuccess;
  if (c->gexec) { (void)hipGraphExecDestroy(c->gexec); c->gexec = nullptr; }
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamBeginCapture(c->st, hipStreamCaptureModeThreadLocal);
  if (e != hipSuccess) return e;
  for (int k = 0; k < c->P.graph_steps; ++k) enqueue_tiled_step(c, -1);
  e = hipStreamEndCapture(c->st, &g);
  if (e != hipSuccess) return e;
  e = hipGraphInstantiate(&c->gexec, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (e == hipSuccess) c->gcur = c->cur;
  return e;
}

void enqueue_steps(tsm_ctx* c, long nsteps, bool with_log) {
  if (c->tiled) {
    c->bind_state();
    if (nsteps > 0) tsm::launch_dt(c->G, c->A, c->SP, c->S, c->st);
    long k = 0;
    if (!with_log && c->P.graph_steps > 0 && nsteps >= c->P.graph_steps &&
        tiled_graph(c) == hipSuccess) {
      for (; k + c->P.graph_steps <= nsteps; k += c->P.graph_steps) (void)hipGraphLaunch(c->gexec, c->st);
      c->bind_state();
    }
    for (; k < nsteps; ++k) enqueue_tiled_step(c, with_log ? (int)k : -1);
  } else {
    c->csr_ready();
    for (long k = 0; k < nsteps; ++k) enqueue_step(c, with_log ? (int)k : -1);
  }
}
}  // namespace

extern "C" int tsm_run(tsm_ctx* c, long nsteps, long* done, double* log) {
  if (!c || nsteps < 0) return fail(TSM_E_ARG, "bad argument");
  const int S = c->S;
  std::vector<tsm::Ctl> before(S), after(S);
  HIP_TRY(c->read_ctl(before));
  if (log && nsteps > 0) {
    if (c->A.log_cap < nsteps) {
      double* p = nullptr;
      int rc = c->alloc(&p, (size_t)S * nsteps * 4);
      if (rc) return rc;
      c->A.log = p;
      c->A.log_cap = (int)nsteps;
    }
  }
  enqueue_steps(c, nsteps, log != nullptr);
  HIP_TRY(hipGetLastError());
  HIP_TRY(c->read_ctl(after));
  if (done)
    for (int s = 0; s < S; ++s) done[s] = (long)(after[s].iter - before[s].iter);
  if (log && nsteps > 0) {
    const size_t cap = (size_t)c->A.log_cap;
    std::vector<double> buf((size_t)S * cap * 4);
    HIP_TRY(hipMemcpy(buf.data(), c->A.log, buf.size() * sizeof(double), hipMemcpyDeviceToHost));
    for (int s = 0; s < S; ++s) {
      const long ns = (long)(after[s].iter - before[s].iter);
      for (long k = 0; k < nsteps * 4; ++k)
        log[(size_t)s * nsteps * 4 + k] = (k < ns * 4) ? buf[(size_t)s * cap * 4 + k] : 0.0;
    }
  }
  c->A.log = (log ? c->A.log : c->A.log);
  return TSM_OK;
}

extern "C" int tsm_step(tsm_ctx* c, double t_target, double* dt_out, double* res_out) {
  if (!c) return fail(TSM_E_ARG, "bad argument");
  if (t_target > 0.0 && !c->P.unsteady)
    return fail(TSM_E_ARG, "t_target needs an unsteady run (steady steps use local time steps)");
  const int S = c->S;
  const size_t nc = S * sizeof(tsm::Ctl);
  std::vector<tsm::Ctl> before(S), after(S);
  if (c->A.log_cap < 1) {  // the step's (iter, dt, t, res) rows
    double* p = nullptr;
    int rc = c->alloc(&p, (size_t)S * 4);
    if (rc) return rc;
    c->A.log = p;
    c->A.log_cap = 1;
  }
  // the control blocks before and after and the rows, in one go if they fit
  const size_t nl = (size_t)S * c->A.log_cap * 4 * sizeof(double);
  const bool small = 2 * nc + nl <= tsm_ctx::PIN;
  if (small) tsm::launch_words((long)nc, c->A.ctl, c->pin, c->st);
  else HIP_TRY(c->read_ctl(before));
  if (c->tiled) {
    c->bind_state();
    tsm::launch_dt(c->G, c->A, c->SP, S, c->st);
    if (t_target > 0.0) tsm::launch_clamp_dt(c->A, S, t_target, c->st);
    enqueue_tiled_step(c, 0);
  } else {
    c->csr_ready();
    c->bind_state();
    tsm::launch_dt(c->G, c->A, c->SP, S, c->st);
    if (t_target > 0.0) tsm::launch_clamp_dt(c->A, S, t_target, c->st);
    enqueue_step(c, 0, /*dt_ready=*/true);
  }
  HIP_TRY(hipGetLastError());
  std::vector<double> rows(nl / sizeof(double));
  if (small) {
    tsm::launch_words((long)nc, c->A.ctl, c->pin + nc, c->st);
    tsm::launch_words((long)nl, c->A.log, c->pin + 2 * nc, c->st);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->st));
    std::memcpy(before.data(), c->pin, nc);
    std::memcpy(after.data(), c->pin + nc, nc);
    std::memcpy(rows.data(), c->pin + 2 * nc, nl);
  } else {
    HIP_TRY(c->read_ctl(after));
    HIP_TRY(hipMemcpy(rows.data(), c->A.log, nl, hipMemcpyDeviceToHost));
  }
  for (int s = 0; s < S; ++s) {
    const bool ran = after[s].iter > before[s].iter;
    const double* r = &rows[(size_t)s * c->A.log_cap * 4];
    if (dt_out) dt_out[s] = ran ? r[1] : 0.0;
    if (res_out) res_out[s] = after[s].res_total;
  }
  return TSM_OK;
}

extern "C" int tsm_run_group(tsm_ctx** cs, int n, long nsteps, long* done) {
  if (!cs || n < 1 || nsteps < 0) return fail(TSM_E_ARG, "bad argument");
  std::vector<std::vector<tsm::Ctl>> before(n);
  for (int i = 0; i < n; ++i) {
    tsm_ctx* c = cs[i];
    if (!c) return fail(TSM_E_ARG, "null context in group");
    before[i].resize(c->S);
    HIP_TRY(c->read_ctl(before[i]));
  }
  // A context whose samples are all done takes no further launches: it is looked
  // at after every POLL steps, one look behind so that its stream does not run dry
  // (the launches of a step of finished samples cost 30 us at 64 samples of 129^2).
  constexpr long POLL = 16;
  std::vector<char> idle(n, 0);
  std::vector<int> looks(n, 0);
  struct Events {
    std::vector<hipEvent_t> e;
    ~Events() { for (auto x : e) (void)hipEventDestroy(x); }
  } ev;
  for (int i = 0; i < n; ++i) {
    bool all = true;
    for (const auto& q : before[i]) all = all && q.done;
    idle[i] = all;
    for (int k = 0; k < 2; ++k) {
      hipEvent_t x;
      HIP_TRY(hipEventCreateWithFlags(&x, hipEventDisableTiming));
      ev.e.push_back(x);
    }
  }
  // Interleave the contexts' launches in chunks so every stream has work queued
  // while the others run: levels of different sizes share the GPU.
  const long chunk = 8;
  for (long k0 = 0; k0 < nsteps; k0 += chunk) {
    const long m = std::min(chunk, nsteps - k0);
    for (int i = 0; i < n; ++i) {
      tsm_ctx* c = cs[i];
      if (idle[i]) continue;
      int* flag = reinterpret_cast<int*>(c->pin);
      if (k0 > 0 && k0 % POLL == 0) {
        const int look = looks[i]++;
        if (look > 0) {
          HIP_TRY(hipEventSynchronize(ev.e[2 * i + (look - 1) % 2]));
          if (*static_cast<volatile int*>(flag + (look - 1) % 2)) {
            idle[i] = 1;
            continue;
          }
        }
        tsm::launch_all_done(c->S, c->A.ctl, flag + look % 2, c->st);
        HIP_TRY(hipEventRecord(ev.e[2 * i + look % 2], c->st));
      }
      if (c->tiled) {
        c->bind_state();
        if (k0 == 0) tsm::launch_dt(c->G, c->A, c->SP, c->S, c->st);
        for (long k = 0; k < m; ++k) enqueue_tiled_step(c, -1);
      } else {
        c->csr_ready();
        for (long k = 0; k < m; ++k) enqueue_step(c, -1);
      }
    }
  }
  HIP_TRY(hipGetLastError());
  for (int i = 0; i < n; ++i) {
    tsm_ctx* c = cs[i];
    std::vector<tsm::Ctl> after(c->S);
    HIP_TRY(c->read_ctl(after));
    long tot = 0;
    for (int s = 0; s < c->S; ++s) tot += (long)(after[s].iter - before[i][s].iter);
    if (done) done[i] = tot;
  }
  return TSM_OK;
}

extern "C" int tsm_run_packed(tsm_ctx** cs, int n, long nsteps, long* done) {
  if (!cs || n < 1 || nsteps < 0) return fail(TSM_E_ARG, "bad argument");
  for (int i = 0; i < n; ++i) {
    const tsm_ctx* c = cs[i];
    if (!c) return fail(TSM_E_ARG, "null context in group");
    if (!c->tiled || c->two_rings_asked || c->P.time_scheme != 0 || c->A.ns || c->P.liou_fix)
      return fail(TSM_E_ARG, "packed steps need Euler SSP-RK3 contexts on the tiled kernels, "
                             "without the Liou fix and without tile_fused_gradient");
    if (c->P.flux != cs[0]->P.flux || c->P.reconstruct != cs[0]->P.reconstruct)
      return fail(TSM_E_ARG, "packed contexts must share the flux and the reconstruction");
    for (int j = 0; j < i; ++j)
      if (cs[j] == c) return fail(TSM_E_ARG, "a context appears twice in the group");
  }
  tsm_ctx* c0 = cs[0];
  hipStream_t st = c0->st;
  std::vector<std::vector<tsm::Ctl>> before(n);
  for (int i = 0; i < n; ++i) {
    tsm_ctx* c = cs[i];
    before[i].resize(c->S);
    HIP_TRY(hipStreamSynchronize(c->st));
    HIP_TRY(hipMemcpy(before[i].data(), c->A.ctl, c->S * sizeof(tsm::Ctl), hipMemcpyDeviceToHost));
  }
  // level descriptors of the three stages: every stage reads W^n for U_old and
  // the last writes W^{n+1} over it (the buffer rotation of enqueue_tiled_step)
  std::vector<tsm::PackLevel> lv(3 * (size_t)n);
  tsm::PackPlan plan{};
  for (int r = 0; r < 3; ++r) {
    for (int i = 0; i < n; ++i) {
      tsm_ctx* c = cs[i];
      const int ia = (c->cur + 1) % 3, ib = (c->cur + 2) % 3;
      const int ins[3] = {c->cur, ia, ib}, outs[3] = {ia, ib, c->cur};
      tsm::PackLevel& L = lv[(size_t)r * n + i];
      L.G = c->G;
      L.T = c->ST;
      L.A = c->A;
      L.A.W_in = c->W[ins[r]];
      L.A.W_out = c->W[outs[r]];
      L.A.V_in = c->V[ins[r]];
      L.A.V_out = c->V[outs[r]];
      L.P = c->SP;
      L.Wn = c->W[c->cur];
      L.dtpart = c->dtpart;
      L.S = c->S;
    }
    tsm::pack_plan(&lv[(size_t)r * n], n, c0->P.flux, c0->P.reconstruct, plan);
  }
  if (c0->pack_cap < lv.size()) {
    int rc = c0->alloc(&c0->pack, lv.size());
    if (rc) return rc;
    c0->pack_cap = lv.size();
  }
  HIP_TRY(hipMemcpyAsync(c0->pack, lv.data(), lv.size() * sizeof(tsm::PackLevel),
                         hipMemcpyHostToDevice, st));
  for (int i = 0; i < n; ++i) {  // the first step's dt and loop test, per context
    tsm_ctx* c = cs[i];
    c->bind_state();
    if (nsteps > 0) tsm::launch_dt(c->G, c->A, c->SP, c->S, st);
  }
  for (long k = 0; k < nsteps; ++k) {
    for (int r = 0; r < 3; ++r) {
      const tsm::PackLevel* d = c0->pack + (size_t)r * n;
      tsm::launch_packed_stage(c0->P.flux, c0->P.reconstruct, d, plan, r, r == 2, st);
    }
    tsm::launch_packed_final(c0->pack, plan, st);
  }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(st));
  for (int i = 0; i < n; ++i) {
    tsm_ctx* c = cs[i];
    c->bind_state();
    c->e_valid = false;
    std::vector<tsm::Ctl> after(c->S);
    HIP_TRY(hipMemcpy(after.data(), c->A.ctl, c->S * sizeof(tsm::Ctl), hipMemcpyDeviceToHost));
    long tot = 0;
    for (int s = 0; s < c->S; ++s) tot += (long)(after[s].iter - before[i][s].iter);
    if (done) done[i] = tot;
  }
  return TSM_OK;
}

extern "C" int tsm_time(tsm_ctx* c, int s, double* t, long* iter) {
  if (!c || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  tsm::Ctl q;
  HIP_TRY(hipStreamSynchronize(c->st));
  HIP_TRY(hipMemcpy(&q, c->A.ctl + s, sizeof(q), hipMemcpyDeviceToHost));
  if (t) *t = q.t;
  if (iter) *iter = (long)q.iter;
  return TSM_OK;
}

extern "C" int tsm_bounds(tsm_ctx* c, int s, double* out) {
  if (!c || !out || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  const int nblk = std::max(1, std::min(1024, (c->G.nv + 255) / 256));
  c->state_ready();
  static_assert(8 * 1024 * sizeof(double) <= tsm_ctx::PIN, "the blocks' bounds fit");
  const double* part = reinterpret_cast<const double*>(c->pin);
  tsm::launch_bounds(c->G, c->A, s, reinterpret_cast<double*>(c->pin), nblk, c->st);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->st));
  // T, p, u, v as (min, max); w is zero in two dimensions
  double r[8] = {1.0e20, -1.0e20, 1.0e20, -1.0e20, 1.0e20, -1.0e20, 1.0e20, -1.0e20};
  for (int b = 0; b < nblk; ++b)
    for (int k = 0; k < 4; ++k) {
      r[2 * k] = std::min(r[2 * k], part[8 * (size_t)b + 2 * k]);
      r[2 * k + 1] = std::max(r[2 * k + 1], part[8 * (size_t)b + 2 * k + 1]);
    }
  for (int k = 0; k < 8; ++k) out[k] = r[k];
  out[8] = out[9] = 0.0;
  return TSM_OK;
}

extern "C" int tsm_get_clock(tsm_ctx* c, int s, long* iter, int* counter, double* t, double* res0) {
  if (!c || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  tsm::Ctl q;
  HIP_TRY(hipStreamSynchronize(c->st));
  HIP_TRY(hipMemcpy(&q, c->A.ctl + s, sizeof(q), hipMemcpyDeviceToHost));
  if (iter) *iter = (long)q.iter;
  if (counter) *counter = q.counter;
  if (t) *t = q.t;
  if (res0) *res0 = q.res0;
  return TSM_OK;
}

extern "C" int tsm_set_clock(tsm_ctx* c, int s, long iter, int counter, double t, double res0) {
  if (!c || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  if (iter < 0 || counter < 0 || counter > c->P.n_time_stamps + 1 || !(t >= 0.0) || !std::isfinite(t) ||
      !(res0 > 0.0) || !std::isfinite(res0))
    return fail(TSM_E_ARG, "clock: iter and counter must be >= 0 (counter <= time stamps + 1), t finite "
                           "and >= 0, res0 finite and > 0");
  tsm::Ctl q;
  HIP_TRY(hipStreamSynchronize(c->st));
  HIP_TRY(hipMemcpy(&q, c->A.ctl + s, sizeof(q), hipMemcpyDeviceToHost));
  q.iter = iter; q.counter = counter; q.t = t; q.res0 = res0;
  q.res_total = 1e20; q.reached = 0; q.done = 0;
  HIP_TRY(hipMemcpy(c->A.ctl + s, &q, sizeof(q), hipMemcpyHostToDevice));
  return TSM_OK;
}

extern "C" int tsm_status(tsm_ctx* c, int s, double* v, long* iter, int* counter, int* done) {
  if (!c || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  tsm::Ctl q;
  HIP_TRY(hipStreamSynchronize(c->st));
  HIP_TRY(hipMemcpy(&q, c->A.ctl + s, sizeof(q), hipMemcpyDeviceToHost));
  if (v) { v[0] = q.t; v[1] = q.dt; v[2] = q.res_total; }
  if (iter) *iter = (long)q.iter;
  if (counter) *counter = q.counter;
  if (done) *done = q.done;
  return TSM_OK;
}

extern "C" int tsm_status_all(tsm_ctx* c, double* v, long* iter, int* counter, int* done,
                              double* norms) {
  if (!c) return fail(TSM_E_ARG, "bad argument");
  std::vector<tsm::Ctl> q(c->S);
  HIP_TRY(hipStreamSynchronize(c->st));
  HIP_TRY(hipMemcpy(q.data(), c->A.ctl, q.size() * sizeof(tsm::Ctl), hipMemcpyDeviceToHost));
  for (int s = 0; s < c->S; ++s) {
    if (v) { v[3 * s] = q[s].t; v[3 * s + 1] = q[s].dt; v[3 * s + 2] = q[s].res_total; }
    if (iter) iter[s] = (long)q[s].iter;
    if (counter) counter[s] = q[s].counter;
    if (done) done[s] = q[s].done;
    if (norms)
      for (int k = 0; k < 4; ++k) norms[4 * s + k] = q[s].rn[k];
  }
  return TSM_OK;
}

extern "C" int tsm_residual_norms(tsm_ctx* c, int s, double* norms) {
  if (!c || s < 0 || s >= c->S || !norms) return fail(TSM_E_ARG, "bad argument");
  tsm::Ctl q;
  HIP_TRY(hipStreamSynchronize(c->st));
  HIP_TRY(hipMemcpy(&q, c->A.ctl + s, sizeof(q), hipMemcpyDeviceToHost));
  for (int k = 0; k < 4; ++k) norms[k] = q.rn[k];
  return TSM_OK;
}

namespace {
int ensure_red(tsm_ctx* c, size_t n) {
  if (c->red_cap >= n) return TSM_OK;
  int rc = c->alloc(&c->red, n);
  if (rc) return rc;
  c->red_cap = n;
  return TSM_OK;
}
}  // namespace

extern "C" int tsm_global(tsm_ctx* c, int s, double* ke, double* ent) {
  if (!c || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  int nb = c->nblk_v, rc = ensure_red(c, (size_t)nb * 24);
  if (rc) return rc;
  c->bind_state();
  tsm::launch_global(c->G, c->A, s, c->red, c->st);
  HIP_TRY(hipGetLastError());
  std::vector<double> h((size_t)nb * 2);
  HIP_TRY(hipStreamSynchronize(c->st));
  HIP_TRY(hipMemcpy(h.data(), c->red, h.size() * sizeof(double), hipMemcpyDeviceToHost));
  double K = 0, E = 0;
  for (int b = 0; b < nb; ++b) { K += h[2 * b]; E += h[2 * b + 1]; }
  if (ke) *ke = K;
  if (ent) *ent = E;
  return TSM_OK;
}

extern "C" int tsm_enstrophy(tsm_ctx* c, int s, double* ens) {
  if (!c || !ens || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  const int nb = c->nblk_v;
  int rc = ensure_red(c, (size_t)nb * 24);
  if (rc) return rc;
  c->sample_ready(s);  // gradients of the current state of sample s
  c->A.ignore_done = 1;
  tsm::launch_gradient_one(c->G, c->A, s, c->st);
  c->A.ignore_done = 0;
  tsm::launch_enstrophy(c->G, c->A, s, c->red, c->st);
  HIP_TRY(hipGetLastError());
  std::vector<double> h((size_t)nb);
  HIP_TRY(hipStreamSynchronize(c->st));
  HIP_TRY(hipMemcpy(h.data(), c->red, h.size() * sizeof(double), hipMemcpyDeviceToHost));
  double Z = 0;
  for (int b = 0; b < nb; ++b) Z += h[b];
  *ens = Z;
  return TSM_OK;
}

extern "C" int tsm_error_norms(tsm_ctx* c, int s, const double* exact, double* out) {
  if (!c || !exact || !out || s < 0 || s >= c->S) return fail(TSM_E_ARG, "bad argument");
  const int nv = c->G.nv, nb = c->nblk_v;
  int rc = ensure_red(c, (size_t)nb * 24);
  if (rc) return rc;
  std::vector<double> ex(4 * (size_t)nv);
  for (int i = 0; i < nv; ++i)
    for (int k = 0; k < 4; ++k) ex[4 * (size_t)c->perm[i] + k] = exact[4 * (size_t)i + k];
  double* dex = nullptr;
  HIP_TRY(hipMalloc(&dex, 4 * (size_t)nv * sizeof(double)));
  hipError_t e = hipMemcpy(dex, ex.data(), 4 * (size_t)nv * sizeof(double), hipMemcpyHostToDevice);
  if (e != hipSuccess) { (void)hipFree(dex); return fail(TSM_E_HIP, "upload exact"); }
  c->bind_state();
  tsm::launch_errnorm(c->G, c->A, s, dex, c->red, c->st);
  e = hipGetLastError();
  std::vector<double> h((size_t)nb * 24);
  if (e == hipSuccess) e = hipStreamSynchronize(c->st);
  if (e == hipSuccess) e = hipMemcpy(h.data(), c->red, h.size() * sizeof(double), hipMemcpyDeviceToHost);
  (void)hipFree(dex);
  if (e != hipSuccess) return fail(TSM_E_HIP, hipGetErrorString(e));
  double L1[8] = {0}, L2[8] = {0}, Li[8] = {0};
  for (int b = 0; b < nb; ++b)
    for (int k = 0; k < 8; ++k) {
      L1[k] += h[24 * b + k];
      L2[k] += h[24 * b + 8 + k];
      Li[k] = std::fmax(Li[k], h[24 * b + 16 + k]);
    }
  for (int k = 0; k < 8; ++k) {
    out[3 * k] = L1[k]; out[3 * k + 1] = std::sqrt(L2[k]); out[3 * k + 2] = Li[k];
  }
  return TSM_OK;
}

extern "C" int tsm_geometry_sizes(tsm_ctx* c, int* nf, int* nb) {
  if (!c) return fail(TSM_E_ARG, "bad argument");
  if (nf) *nf = (int)c->geo.face.size();
  if (nb) *nb = (int)c->geo.bface.size();
  return TSM_OK;
}

extern "C" int tsm_geometry(tsm_ctx* c, int* fv, double* fn, double* dc, double* mc) {
  if (!c) return fail(TSM_E_ARG, "bad argument");
  const auto& g = c->geo;
  for (size_t f = 0; f < g.face.size(); ++f) {
    if (fv) { fv[2 * f] = g.face[f].v[0]; fv[2 * f + 1] = g.face[f].v[1]; }
    if (fn) { fn[2 * f] = g.face[f].nx; fn[2 * f + 1] = g.face[f].ny; }
  }
  for (int i = 0; i < g.nv; ++i) {
    if (dc) dc[i] = g.dcarea[i];
    if (mc) mc[i] = g.mcarea[i];
  }
  return TSM_OK;
}

extern "C" int tsm_bench(tsm_ctx* c, int nsteps, double* us) {
  if (!c || nsteps < 1 || !us) return fail(TSM_E_ARG, "bad argument");
  hipEvent_t ev[16];
  for (auto& e : ev) HIP_TRY(hipEventCreate(&e));
  double acc[4] = {0, 0, 0, 0};
  float ms = 0;
  HIP_TRY(hipStreamSynchronize(c->st));
  if (c->tiled) {
    c->bind_state();
    tsm::launch_dt(c->G, c->A, c->SP, c->S, c->st);
    const int nrk = c->P.time_scheme == 0 ? 3 : (c->P.time_scheme == 1 ? 4 : 2);
    for (int k = 0; k < nsteps; ++k) {
      enqueue_tiled_step(c, -1, ev);
      HIP_TRY(hipEventSynchronize(ev[nrk + 1]));
      for (int r = 0; r < nrk; ++r) {
        HIP_TRY(hipEventElapsedTime(&ms, ev[r], ev[r + 1])); acc[2] += ms;
      }
      HIP_TRY(hipEventElapsedTime(&ms, ev[nrk], ev[nrk + 1])); acc[3] += ms;
    }
    us[0] = us[1] = 0.0;
    us[2] = 1e3 * acc[2] / ((double)nrk * nsteps);
    us[3] = 1e3 * acc[3] / nsteps;
  } else {
    c->csr_ready();
    const int nrk = c->P.time_scheme == 0 ? 3 : (c->P.time_scheme == 1 ? 4 : 2);
    const int mode = c->P.time_scheme == 1 ? 2 : 1;
    for (int k = 0; k < nsteps; ++k) {
      c->bind_state();
      HIP_TRY(hipEventRecord(ev[0], c->st));
      tsm::launch_dt(c->G, c->A, c->SP, c->S, c->st);
      HIP_TRY(hipEventRecord(ev[1], c->st));
      if (c->P.liou_fix) tsm::launch_ssw(c->G, c->A, c->S, c->st);
      int e = 2;
      for (int r = 0; r < nrk; ++r) {
        c->bind_state();
        HIP_TRY(hipEventRecord(ev[e++], c->st));
        tsm::launch_gradient(c->G, c->A, c->S, c->st);
        HIP_TRY(hipEventRecord(ev[e++], c->st));
        tsm::launch_flux_update(c->P.flux, c->P.reconstruct, c->G, c->A, c->S, r, r == nrk - 1,
                                mode, c->st, true, false);
        HIP_TRY(hipEventRecord(ev[e++], c->st));
        tsm::launch_flux_update(c->P.flux, c->P.reconstruct, c->G, c->A, c->S, r, r == nrk - 1,
                                mode, c->st, false, true);
        if (c->P.strong_bc) tsm::launch_strong_bc(c->G, c->A, c->S, c->st);
        c->cur ^= 1;
      }
      c->bind_state();
      tsm::launch_step_final(c->G, c->A, c->SP, c->S, -1, c->st);
      HIP_TRY(hipEventRecord(ev[e++], c->st));
      HIP_TRY(hipEventSynchronize(ev[e - 1]));
      HIP_TRY(hipEventElapsedTime(&ms, ev[0], ev[1])); acc[0] += ms;
      for (int r = 0; r < nrk; ++r) {
        HIP_TRY(hipEventElapsedTime(&ms, ev[2 + 3 * r], ev[3 + 3 * r])); acc[1] += ms;
        HIP_TRY(hipEventElapsedTime(&ms, ev[3 + 3 * r], ev[4 + 3 * r])); acc[2] += ms;
        HIP_TRY(hipEventElapsedTime(&ms, ev[4 + 3 * r], ev[(r == nrk - 1) ? e - 1 : 5 + 3 * r])); acc[3] += ms;
      }
    }
    us[0] = 1e3 * acc[0] / nsteps;
    us[1] = 1e3 * acc[1] / (nsteps * (double)nrk);
    us[2] = 1e3 * acc[2] / (nsteps * (double)nrk);
    us[3] = 1e3 * acc[3] / (nsteps * (double)nrk);
  }
  // whole steps without interleaved events
  HIP_TRY(hipEventRecord(ev[14], c->st));
  enqueue_steps(c, nsteps, false);
  HIP_TRY(hipEventRecord(ev[15], c->st));
  HIP_TRY(hipEventSynchronize(ev[15]));
  HIP_TRY(hipEventElapsedTime(&ms, ev[14], ev[15]));
  us[4] = 1e3 * ms / nsteps;
  for (auto& e : ev) (void)hipEventDestroy(e);
  return TSM_OK;
}

extern "C" int tsm_moments(tsm_ctx* c, double* mean, double* m2, double* s2) {
  if (!c) return fail(TSM_E_ARG, "bad argument");
  const int nv = c->G.nv;
  double *dm = nullptr, *dq = nullptr, *dz = nullptr;
  const size_t n = 5 * (size_t)nv;
  HIP_TRY(hipMalloc(&dm, 3 * n * sizeof(double)));
  dq = dm + n;
  dz = dq + n;
  c->bind_state();
  tsm::launch_moments(c->G, c->A, c->S, dm, dq, dz, c->st);
  hipError_t e = hipGetLastError();
  std::vector<double> h(3 * n);
  if (e == hipSuccess) e = hipStreamSynchronize(c->st);
  if (e == hipSuccess) e = hipMemcpy(h.data(), dm, h.size() * sizeof(double), hipMemcpyDeviceToHost);
  (void)hipFree(dm);
  if (e != hipSuccess) return fail(TSM_E_HIP, hipGetErrorString(e));
  double* outs[3] = {mean, m2, s2};
  for (int a = 0; a < 3; ++a) {
    if (!outs[a]) continue;
    for (int i = 0; i < nv; ++i)
      for (int q = 0; q < 5; ++q) outs[a][5 * (size_t)i + q] = h[a * n + 5 * (size_t)c->perm[i] + q];
  }
  return TSM_OK;
}

extern "C" int tsm_probe_density(tsm_ctx* c, int np, const double* px, const double* py,
                                 double* out) {
  if (!c || np < 1 || !px || !py || !out) return fail(TSM_E_ARG, "bad argument");
  // device point location (k_probe_locate: the first cell in cell order that
  // holds the point), then the interpolation of every sample
  const size_t n = (size_t)np;
  double *dpx = nullptr, *dpy = nullptr, *dpw = nullptr, *dout = nullptr;
  int *dpc = nullptr, *dcell = nullptr;
  hipError_t e = hipMalloc(&dpx, 8 * n);
  if (e == hipSuccess) e = hipMalloc(&dpy, 8 * n);
  if (e == hipSuccess) e = hipMalloc(&dpw, 24 * n);
  if (e == hipSuccess) e = hipMalloc(&dout, 8 * n * (size_t)c->S);
  if (e == hipSuccess) e = hipMalloc(&dpc, 12 * n);
  if (e == hipSuccess) e = hipMalloc(&dcell, 4 * n);
  if (e == hipSuccess) e = hipMemcpyAsync(dpx, px, 8 * n, hipMemcpyHostToDevice, c->st);
  if (e == hipSuccess) e = hipMemcpyAsync(dpy, py, 8 * n, hipMemcpyHostToDevice, c->st);
  if (e == hipSuccess) {
    tsm::launch_probe_locate(c->G, np, dpx, dpy, dpc, dpw, dcell, c->st);
    c->bind_state();
    tsm::launch_probes(c->A, c->G.nv, np, dpc, dpw, c->S, dout, c->st);
    e = hipGetLastError();
  }
  std::vector<int> cells(n);
  if (e == hipSuccess) e = hipMemcpyAsync(cells.data(), dcell, 4 * n, hipMemcpyDeviceToHost, c->st);
  if (e == hipSuccess) e = hipMemcpyAsync(out, dout, 8 * n * (size_t)c->S, hipMemcpyDeviceToHost, c->st);
  if (e == hipSuccess) e = hipStreamSynchronize(c->st);
  (void)hipFree(dpx); (void)hipFree(dpy); (void)hipFree(dpw); (void)hipFree(dout);
  (void)hipFree(dpc); (void)hipFree(dcell);
  if (e != hipSuccess) return fail(TSM_E_HIP, hipGetErrorString(e));
  for (int p = 0; p < np; ++p)
    if (cells[p] < 0) return fail(TSM_E_ARG, "probe point " + std::to_string(p) + " outside the mesh");
  return TSM_OK;
}

extern "C" int tsm_probe_density_noalloc(tsm_ctx* c, int np, const double* px, const double* py,
                                         double* out) {
  if (!c || np < 1 || !px || !py || !out) return fail(TSM_E_ARG, "bad argument");
  // scratch layout: px, py, weights (3 per probe), densities (one per probe and
  // sample), corner ids (3 int32 per probe), containing cell (one int32 per
  // probe, -1 outside the mesh); each part 256-byte aligned
  auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
  const size_t n = (size_t)np;
  const size_t o_py = up(8 * n), o_pw = o_py + up(8 * n), o_out = o_pw + up(24 * n);
  const size_t o_pc = o_out + up(8 * n * (size_t)c->S), o_cell = o_pc + up(12 * n);
  const size_t need = o_cell + up(4 * n);
  if (need > tsm::noalloc_scratch_bytes())
    return fail(TSM_E_ARG, "tsm_probe_density_noalloc: " + std::to_string(np) + " probes x " +
                               std::to_string(c->S) + " samples need " + std::to_string(need) +
                               " bytes of scratch, more than its fixed " +
                               std::to_string(tsm::noalloc_scratch_bytes()));
  int prev = -1;
  HIP_TRY(hipGetDevice(&prev));
  if (prev != c->dev) HIP_TRY(hipSetDevice(c->dev));
  struct Restore {  // the caller's device again on every return
    int d, p;
    ~Restore() { if (d != p) (void)hipSetDevice(p); }
  } restore{c->dev, prev};
  void* base = nullptr;
  int he = tsm::noalloc_scratch(&base);
  if (he) return fail(TSM_E_HIP, std::string("hipGetSymbolAddress(scratch): ") +
                                     hipGetErrorString((hipError_t)he));
  char* b = static_cast<char*>(base);
  double* dpx = reinterpret_cast<double*>(b);
  double* dpy = reinterpret_cast<double*>(b + o_py);
  double* dpw = reinterpret_cast<double*>(b + o_pw);
  double* dout = reinterpret_cast<double*>(b + o_out);
  int* dpc = reinterpret_cast<int*>(b + o_pc);
  int* dcell = reinterpret_cast<int*>(b + o_cell);
  HIP_TRY(hipMemcpyAsync(dpx, px, 8 * n, hipMemcpyHostToDevice, c->st));
  HIP_TRY(hipMemcpyAsync(dpy, py, 8 * n, hipMemcpyHostToDevice, c->st));
  tsm::launch_probe_locate(c->G, np, dpx, dpy, dpc, dpw, dcell, c->st);
  HIP_TRY(hipGetLastError());
  c->bind_state();
  tsm::launch_probes(c->A, c->G.nv, np, dpc, dpw, c->S, dout, c->st);
  HIP_TRY(hipGetLastError());
  // the containing cells first (into the caller's output, which is large
  // enough: 8 np S >= 4 np bytes), to report points outside the mesh
  HIP_TRY(hipMemcpyAsync(out, dcell, 4 * n, hipMemcpyDeviceToHost, c->st));
  HIP_TRY(hipStreamSynchronize(c->st));
  const int* cells = reinterpret_cast<const int*>(out);
  for (int p = 0; p < np; ++p)
    if (cells[p] < 0)
      return fail(TSM_E_ARG, "probe point " + std::to_string(p) + " outside the mesh");
  HIP_TRY(hipMemcpyAsync(out, dout, 8 * n * (size_t)c->S, hipMemcpyDeviceToHost, c->st));
  HIP_TRY(hipStreamSynchronize(c->st));
  return TSM_OK;
}

namespace {
// launch(n, a, b, out, stream) over the operands, m results each
template <class F>
int check_operands(long n, const double* a, const double* b, double* out, int m, F&& launch) {
  if (n < 1 || !a || !b || !out) return fail(TSM_E_ARG, "bad argument");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(TSM_E_HIP, "no HIP device visible");
  double* d = nullptr;
  HIP_TRY(hipMalloc(&d, (size_t)(2 + m) * n * sizeof(double)));
  hipError_t e = hipMemcpy(d, a, 8 * (size_t)n, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(d + n, b, 8 * (size_t)n, hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    launch(n, d, d + n, d + 2 * n, nullptr);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(out, d + 2 * n, 8 * (size_t)m * n, hipMemcpyDeviceToHost);
  (void)hipFree(d);
  if (e != hipSuccess) return fail(TSM_E_HIP, hipGetErrorString(e));
  return TSM_OK;
}
}  // namespace

extern "C" int tsm_check_arith(long n, const double* a, const double* b, double* out) {
  return check_operands(n, a, b, out, 4, tsm::launch_check_arith);
}
extern "C" int tsm_check_math(long n, const double* a, const double* b, double* out) {
  return check_operands(n, a, b, out, 6, tsm::launch_check_math);
}

extern "C" int tsm_global_all(tsm_ctx* c, double* ke, double* ent) {
  if (!c) return fail(TSM_E_ARG, "bad argument");
  const int nb = c->nblk_v, S = c->S;
  const size_t n = (size_t)nb * S * 2;
  const bool small = n * sizeof(double) <= tsm_ctx::PIN;
  if (!small)
    if (int rc = ensure_red(c, n)) return rc;  // the context's reduction buffer: no allocation per call
  c->bind_state();
  tsm::launch_global_all(c->G, c->A, S, small ? reinterpret_cast<double*>(c->pin) : c->red, c->st);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->st));
  std::vector<double> big(small ? 0 : n);
  if (!small) HIP_TRY(hipMemcpy(big.data(), c->red, n * sizeof(double), hipMemcpyDeviceToHost));
  const double* h = small ? reinterpret_cast<const double*>(c->pin) : big.data();
  for (int s = 0; s < S; ++s) {
    double K = 0, E = 0;
    for (int b = 0; b < nb; ++b) { K += h[((size_t)s * nb + b) * 2]; E += h[((size_t)s * nb + b) * 2 + 1]; }
    if (ke) ke[s] = K;
    if (ent) ent[s] = E;
  }
  return TSM_OK;
}
