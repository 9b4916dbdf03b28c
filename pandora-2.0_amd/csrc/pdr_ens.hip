// pdr_ens.hip -- batched ensembles of small boxes: many independent
// realisations of uneven sizes advanced together.
//
// A 32^3 box gives a pass a few dozen workgroups, so stepping each member on
// its own leaves most of the 256 CUs idle and pays its kernel launches per step
// per member.  Here every pass of an RK3 stage is one launch over all members of
// one line length (pdr_ens_passes.hip), and the launches of their step are
// captured once into a HIP graph and replayed.  The members of different lengths
// have nothing to wait for in each other: each length's steps run on a stream of
// their own, where one length's kernels fill the CUs that the last workgroups of
// another's leave idle, and the streams meet at the end of a run.  Each member
// runs the device bodies that pdr_step runs for it, with the same arguments; they
// are compiled into other kernels, where the compiler may contract multiply-adds
// differently, so the results agree with pdr_step to rounding.
//
// Scope: members of one precision with the specialised kernels, cubic, line
// lengths 32..256, isotropic with RK3_TIMESTEP = FIXED, no forcing and no
// tracers (the decaying-ensemble case).  Those keep every kernel argument of
// the step constant, which is what makes the step a replayable graph; shear
// frames (per-stage coefficients), CFL steps (a host read of the maximum),
// forcing (per-step draws) and tracers are rejected with PDR_ERR_UNSUPPORTED.
#include <algorithm>
#include <chrono>
#include <cstring>
#include <string>
#include <vector>

#include "pdr_ens_ops.hpp"

namespace {

// The members of one line length.
struct EnsGroup {
  const pdr::EnsOps* ops = nullptr;
  int first = 0, count = 0;  // of the descriptors, which are ordered by length
  hipStream_t stream = nullptr;
  // one RK3 step: `joined` leaves the next step's inverse z pass done (lengths with
  // zz, which then start a run with that pass and end it with `last`)
  hipGraph_t joined = nullptr, last = nullptr;
  hipGraphExec_t joined_exec = nullptr, last_exec = nullptr;
};

}  // namespace

struct pdr_ensemble {
  std::vector<pdr_ctx*> m;
  int prec = 0;
  hipStream_t stream = nullptr;
  pdr::EnsMember* d_mem = nullptr;
  std::vector<EnsGroup> groups;
  int fpb_y = 0, fpb_yf = 0;  // 0: each member's own choice
};

namespace {

using pdr::set_error;

const double kBeta[3] = {0.0, -5.0 / 9.0, -153.0 / 128.0};
const double kGamma[3] = {1.0 / 3.0, 15.0 / 16.0, 8.0 / 15.0};

void ens_release(std::vector<EnsGroup>& groups) {
  for (EnsGroup& q : groups) {
    if (q.stream) (void)hipStreamSynchronize(q.stream);
    for (hipGraphExec_t x : {q.joined_exec, q.last_exec})
      if (x) (void)hipGraphExecDestroy(x);
    for (hipGraph_t x : {q.joined, q.last})
      if (x) (void)hipGraphDestroy(x);
    if (q.stream) (void)hipStreamDestroy(q.stream);
  }
  groups.clear();
}

// Captures one RK3 step of a group: 3 stages of the inverse z pass (where the stage
// before has not done it), the passes of the planes and the z forward + FormF.
hipError_t ens_capture(pdr_ensemble* e, EnsGroup& q, int fpb_y, int fpb_yf, bool joined, hipGraph_t* graph,
                       hipGraphExec_t* exec) {
  const pdr::EnsMember* mem = e->d_mem + q.first;
  hipError_t r = hipStreamBeginCapture(q.stream, hipStreamCaptureModeThreadLocal);
  if (r != hipSuccess) return r;
  hipError_t lr = hipSuccess;
  for (int st = 0; st < 3 && lr == hipSuccess; ++st) {
    if (!q.ops->zz) lr = q.ops->zinv(mem, q.count, q.stream);
    if (lr == hipSuccess) lr = q.ops->mid(mem, q.count, fpb_y, fpb_yf, q.stream);
    if (lr == hipSuccess)
      lr = q.ops->zend(mem, q.count, kBeta[st], kGamma[st], q.ops->zz && (joined || st < 2), q.stream);
  }
  r = hipStreamEndCapture(q.stream, graph);
  if (lr != hipSuccess) return lr;
  if (r != hipSuccess) return r;
  return hipGraphInstantiate(exec, *graph, nullptr, nullptr, 0);
}

// The groups' graphs for a split of the y passes (0: each member's own choice).  They are
// made beside the ones that stand and take their place once all are there, so an
// ensemble whose rebuild fails keeps its graphs and its split.
int ens_build(pdr_ensemble* e, int fpb_y, int fpb_yf) {
  std::vector<EnsGroup> groups;
  const int nm = int(e->m.size());
  std::vector<pdr_ctx*> order = e->m;
  std::stable_sort(order.begin(), order.end(), [](const pdr_ctx* a, const pdr_ctx* b) { return a->g.nx < b->g.nx; });
  std::vector<pdr::EnsMember> h(static_cast<size_t>(nm));
  for (int k = 0; k < nm; ++k) {
    pdr_ctx* c = order[size_t(k)];
    if (k == 0 || c->g.nx != order[size_t(k - 1)]->g.nx) {
      EnsGroup q;
      q.ops = pdr::ens_ops(c->prec, c->g.nx);
      q.first = k;
      if (!q.ops) return set_error(PDR_ERR_UNSUPPORTED, "ensemble: unsupported line length");
      groups.push_back(q);
    }
    ++groups.back().count;
    pdr::EnsMember& d = h[size_t(k)];
    std::memset(&d, 0, sizeof(d));
    d.g = c->g;
    d.cf = pdr::make_coef(c);
    d.dt = c->p.rk3_dt;
    d.norm = 1.0 / (double(c->g.nx) * double(c->g.ny) * double(c->g.nz));
    for (int q = 0; q < 3; ++q) {
      d.u[q] = c->u[q];
      d.rk[q] = c->rk[q];
    }
    d.w1 = c->w1;
    d.w2 = c->w2;
    d.umax = c->umax;
    d.twz = c->tab.twz;
    d.twy = c->tab.twy;
    d.twx = c->tab.twx;
  }
  if (!e->d_mem && hipMalloc(&e->d_mem, sizeof(pdr::EnsMember) * size_t(nm)) != hipSuccess) {
    (void)hipGetLastError();
    e->d_mem = nullptr;
    return set_error(PDR_ERR_NOMEM, "ensemble: device allocation failed");
  }
  hipError_t r = hipMemcpy(e->d_mem, h.data(), sizeof(pdr::EnsMember) * size_t(nm), hipMemcpyHostToDevice);
  for (EnsGroup& q : groups) {
    const pdr_ctx* c = order[size_t(q.first)];
    const int fy = fpb_y ? fpb_y : c->fpb_y, fyf = fpb_yf ? fpb_yf : c->fpb_yf;
    if (r == hipSuccess) r = q.ops->prepare();
    if (r == hipSuccess) r = hipStreamCreateWithFlags(&q.stream, hipStreamNonBlocking);
    if (r == hipSuccess) r = ens_capture(e, q, fy, fyf, false, &q.last, &q.last_exec);
    if (r == hipSuccess && q.ops->zz) r = ens_capture(e, q, fy, fyf, true, &q.joined, &q.joined_exec);
  }
  if (r != hipSuccess) {
    (void)hipGetLastError();
    ens_release(groups);
    return set_error(PDR_ERR_HIP, std::string("ensemble set-up: ") + hipGetErrorString(r));
  }
  ens_release(e->groups);
  e->groups.swap(groups);
  e->fpb_y = fpb_y;
  e->fpb_yf = fpb_yf;
  return PDR_OK;
}

// Queues nsteps steps of every group and waits for them.  The groups take turns, so
// that each has work queued while the others run.
hipError_t ens_steps(pdr_ensemble* e, int nsteps) {
  hipError_t r = hipSuccess;
  for (EnsGroup& q : e->groups)
    if (r == hipSuccess && nsteps > 0 && q.ops->zz) r = q.ops->zinv(e->d_mem + q.first, q.count, q.stream);
  for (int s = 0; s < nsteps && r == hipSuccess; ++s)
    for (EnsGroup& q : e->groups)
      if (r == hipSuccess) r = hipGraphLaunch(q.ops->zz && s + 1 < nsteps ? q.joined_exec : q.last_exec, q.stream);
  for (EnsGroup& q : e->groups) {
    const hipError_t w = hipStreamSynchronize(q.stream);
    if (r == hipSuccess) r = w;
  }
  return r;
}

}  // namespace

extern "C" {

int pdr_ensemble_create(pdr_ensemble** out, pdr_ctx* const* members, int32_t count) {
  if (!out || !members || count < 1) return set_error(PDR_ERR_ARG, "pdr_ensemble_create: bad argument");
  *out = nullptr;
  const int prec = members[0] ? members[0]->prec : 0;
  for (int32_t k = 0; k < count; ++k) {
    const pdr_ctx* c = members[k];
    if (!c) return set_error(PDR_ERR_ARG, "pdr_ensemble_create: null member");
    for (int32_t q = 0; q < k; ++q)
      if (members[q] == c) return set_error(PDR_ERR_ARG, "pdr_ensemble_create: member listed twice");
    const bool ok = c->prec == prec && c->spec && c->fuse_zf && c->g.zc == c->g.nz && c->g.nx == c->g.ny &&
                    c->g.ny == c->g.nz && pdr::ens_ops(prec, c->g.nx) &&
                    c->p.f_type == PDR_F_ISOTROPIC && c->p.rk3_timestep == PDR_RK3_TIMESTEP_FIXED &&
                    !c->forcing && c->np == 0 && c->p.dealiasing == PDR_DEALIASING_TWOTHIRD;
    if (!ok)
      return set_error(PDR_ERR_UNSUPPORTED,
                       "pdr_ensemble_create: members must share the precision and be cubic (32..256 points), "
                       "isotropic, FIXED time step, 2/3 dealiasing, unforced and without tracers");
  }
  pdr_ensemble* e = new pdr_ensemble();
  e->m.assign(members, members + count);
  e->prec = prec;
  if (hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess) {
    (void)hipGetLastError();
    delete e;
    return set_error(PDR_ERR_HIP, "pdr_ensemble_create: stream creation failed");
  }
  int rc = ens_build(e, 0, 0);
  if (rc != PDR_OK) {
    pdr_ensemble_destroy(e);
    return rc;
  }
  *out = e;
  return PDR_OK;
}

int pdr_ensemble_set_split(pdr_ensemble* e, int32_t fpb_y, int32_t fpb_yf) {
  if (!e) return set_error(PDR_ERR_ARG, "null ensemble");
  const bool ok = (fpb_y == 0 || fpb_y == 1 || fpb_y == 2 || fpb_y == 3 || fpb_y == 6) &&
                  (fpb_yf == 0 || fpb_yf == 1 || fpb_yf == 3);
  if (!ok) return set_error(PDR_ERR_ARG, "pdr_ensemble_set_split: fields per workgroup must divide 6 / 3");
  return ens_build(e, fpb_y, fpb_yf);
}

// Times `steps` graph steps for each split of the y passes over workgroups
// (fields per workgroup 1, 2, 3, 6 for the inverse pass and 1, 3 for the
// forward pass), keeps the fastest, and restores every member's state and RK
// registers, so the ensemble is where it was before the call; after an error it has
// the split and the graphs of before as well.
int pdr_ensemble_autotune(pdr_ensemble* e, int32_t steps, int32_t* best_y, int32_t* best_yf) {
  if (!e || steps < 1) return set_error(PDR_ERR_ARG, "pdr_ensemble_autotune: bad argument");
  for (pdr_ctx* c : e->m)
    if (hipStreamSynchronize(c->stream) != hipSuccess)
      return set_error(PDR_ERR_HIP, "pdr_ensemble_autotune: member stream failed");
  // save the state
  size_t total = 0;
  for (pdr_ctx* c : e->m) total += 6 * size_t(c->g.mw) * c->csz;
  char* save = nullptr;
  if (hipMalloc(&save, total) != hipSuccess) {
    (void)hipGetLastError();
    return set_error(PDR_ERR_NOMEM, "pdr_ensemble_autotune: device allocation failed");
  }
  auto copy_state = [&](bool to_save) {
    size_t off = 0;
    hipError_t r = hipSuccess;
    for (pdr_ctx* c : e->m) {
      const size_t b = size_t(c->g.mw) * c->csz;
      void* f[6] = {c->u[0], c->u[1], c->u[2], c->rk[0], c->rk[1], c->rk[2]};
      for (void* a : f) {
        if (r == hipSuccess)
          r = to_save ? hipMemcpyAsync(save + off, a, b, hipMemcpyDeviceToDevice, e->stream)
                      : hipMemcpyAsync(a, save + off, b, hipMemcpyDeviceToDevice, e->stream);
        off += b;
      }
    }
    if (r == hipSuccess) r = hipStreamSynchronize(e->stream);
    return r;
  };
  hipError_t r = copy_state(true);
  const int ys[4] = {1, 2, 3, 6}, yfs[2] = {1, 3};
  double best = 1e30;
  int by = e->fpb_y ? e->fpb_y : 6, byf = e->fpb_yf ? e->fpb_yf : 3;
  bool split = false;  // nothing to tune where every member's planes run as one kernel
  for (const EnsGroup& q : e->groups) split = split || q.ops->split;
  const bool saved = r == hipSuccess;
  std::vector<EnsGroup> before;
  before.swap(e->groups);
  const int before_y = e->fpb_y, before_yf = e->fpb_yf;
  int rc = PDR_OK;
  for (int iy = 0; iy < 4 && split && r == hipSuccess && rc == PDR_OK; ++iy)
    for (int iyf = 0; iyf < 2 && r == hipSuccess && rc == PDR_OK; ++iyf) {
      rc = ens_build(e, ys[iy], yfs[iyf]);
      if (rc != PDR_OK) break;
      r = ens_steps(e, 1);  // warm-up
      const auto t0 = std::chrono::steady_clock::now();
      if (r == hipSuccess) r = ens_steps(e, steps);
      const double s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
      if (r == hipSuccess && s < best) {
        best = s;
        by = ys[iy];
        byf = yfs[iyf];
      }
    }
  if (saved) {
    const hipError_t back = copy_state(false);
    if (r == hipSuccess) r = back;
  }
  (void)hipFree(save);
  if (r == hipSuccess && rc == PDR_OK) rc = ens_build(e, by, byf);
  if (r != hipSuccess || rc != PDR_OK) {
    ens_release(e->groups);
    e->groups.swap(before);
    e->fpb_y = before_y;
    e->fpb_yf = before_yf;
    return r != hipSuccess ? set_error(PDR_ERR_HIP, std::string("pdr_ensemble_autotune: ") + hipGetErrorString(r)) : rc;
  }
  ens_release(before);
  if (best_y) *best_y = by;
  if (best_yf) *best_yf = byf;
  return PDR_OK;
}

int pdr_ensemble_run(pdr_ensemble* e, int32_t tstep0, int32_t nsteps, double* simtime) {
  (void)tstep0;
  if (!e || nsteps < 0 || !simtime) return set_error(PDR_ERR_ARG, "pdr_ensemble_run: bad argument");
  for (pdr_ctx* c : e->m)  // work queued on the members' own streams comes first
    if (hipStreamSynchronize(c->stream) != hipSuccess)
      return set_error(PDR_ERR_HIP, "pdr_ensemble_run: member stream failed");
  if (e->groups.empty()) return set_error(PDR_ERR_STATE, "pdr_ensemble_run: the ensemble has no graphs");
  const hipError_t r = ens_steps(e, nsteps);
  if (r != hipSuccess) return set_error(PDR_ERR_HIP, std::string("pdr_ensemble_run: ") + hipGetErrorString(r));
  for (int32_t s = 0; s < nsteps; ++s)
    // g_RK3Calc: simtime = t + dt after the third stage (src/pg_rk3.f90:82-129)
    for (size_t k = 0; k < e->m.size(); ++k) {
      pdr_ctx* c = e->m[k];
      c->dt = c->p.rk3_dt;
      simtime[k] = simtime[k] + c->dt;
    }
  return PDR_OK;
}

int pdr_ensemble_destroy(pdr_ensemble* e) {
  if (!e) return PDR_OK;
  if (e->stream) (void)hipStreamSynchronize(e->stream);
  ens_release(e->groups);
  if (e->d_mem) (void)hipFree(e->d_mem);
  if (e->stream) (void)hipStreamDestroy(e->stream);
  delete e;
  return PDR_OK;
}

}  // extern "C"
