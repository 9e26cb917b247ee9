// Serving loop of libhdg (include/hdg.h, hdg_server_*): a queue of Poisson
// solves on rectangle meshes, worker slots that each own a context and its
// HIP stream, admission by device-memory budget, per-request latency.
// Host code only; every device operation goes through the C ABI.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <deque>
#include <mutex>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>

#include "../../include/hdg.h"
#include "hdg_arena.h"

namespace {

constexpr int kLookahead = 8;     // queued requests a free slot may pick from
constexpr int kBatchLook = 512;   // queued requests scanned for a batch
struct Pending {
  int64_t id;
  hdg_request req;
  double t_submit;
  size_t foot;
};

struct Done {
  hdg_result res;
  std::vector<double> trace;
};

struct Slot {
  hdg_ctx* ctx = nullptr;
  size_t held = 0;  // device bytes the slot's context holds
  // what the context currently holds
  bool has_mesh = false, has_setup = false;
  int64_t nx = 0, ny = 0;
  double jitter = 0.0;
  uint64_t seed = 0;
  int8_t nt = 0;
  hdg_options opt{};
};

bool same_options(const hdg_options& a, const hdg_options& b) {
  return a.k == b.k && a.quad_degree == b.quad_degree && a.tau == b.tau && a.precision == b.precision &&
         a.rtol == b.rtol && a.maxit == b.maxit && a.schedule == b.schedule && a.precond == b.precond;
}

// requests hdg_batch_* accepts: analytic sources, SINSIN or no error norm
bool batchable(const hdg_request& q) {
  return q.src.kind >= 0 && q.src.kind <= 2 && (q.uex_kind == -1 || q.uex_kind == HDG_UEX_SINSIN);
}

}  // namespace

struct hdg_server {
  int device = 0;
  size_t budget = 0;
  hdg_arena* arena = nullptr;  // the budget as one device allocation (null: device pool)
  std::mutex mu;
  std::condition_variable cv_work, cv_done;
  std::deque<Pending> queue;
  std::unordered_map<int64_t, Done> done;
  std::unordered_map<int64_t, int> open;  // submitted, not yet waited
  size_t reserved = 0, peak = 0;
  bool stopping = false;
  int64_t next_id = 1;
  std::vector<Slot> slots;
  std::vector<std::thread> threads;
  std::vector<double> latency, qwait;
  int64_t completed = 0, failed = 0, cells = 0;
  int batch_max = 1;        // requests per grouped launch (1: one request per slot)
  int64_t batch_cells = 0;  // cell cap of a batch
  double first_start = 1e300, last_done = 0.0;
  std::chrono::steady_clock::time_point t0;
  std::string err;

  double now() const {
    return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  }
};

namespace {

// Runs one request in slot s; returns the result (device bytes filled in).
hdg_result run_request(hdg_server* S, Slot& sl, const Pending& p, std::vector<double>* trace) {
  hdg_result r{};
  r.id = p.id;
  r.t_submit = p.t_submit;
  r.t_start = S->now();
  const hdg_request& q = p.req;
  int st = HDG_OK;
  if (!sl.ctx) {
    st = hdg_create(&sl.ctx, S->device, 0);
    if (st == HDG_OK && S->arena) st = hdg_attach_arena(sl.ctx, S->arena);
  }
  const bool mesh_hit = sl.has_mesh && sl.nx == q.nx && sl.ny == q.ny && sl.jitter == q.jitter &&
                        sl.seed == q.seed;
  if (st == HDG_OK && !mesh_hit) {
    sl.has_mesh = sl.has_setup = false;
    // generated on the device: no host mesh arrays, no upload
    st = hdg_set_rectangle_mesh(sl.ctx, q.nx, q.ny, 0.0, 0.0, 1.0, 1.0, q.jitter, q.seed);
    if (st == HDG_OK) {
      sl.has_mesh = true;
      sl.nx = q.nx;
      sl.ny = q.ny;
      sl.jitter = q.jitter;
      sl.seed = q.seed;
    }
  }
  if (st == HDG_OK && !(sl.has_setup && same_options(sl.opt, q.opt))) {
    sl.has_setup = false;
    st = hdg_setup(sl.ctx, &q.opt);
    if (st == HDG_OK) {
      sl.has_setup = true;
      sl.opt = q.opt;
    }
  }
  hdg_sizes sz{};
  if (st == HDG_OK) st = hdg_query_sizes(sl.ctx, &sz);
  if (st == HDG_OK) st = hdg_set_source(sl.ctx, &q.src);
  // u = 0 on the boundary (every serving problem)
  if (st == HDG_OK) st = hdg_set_dirichlet_boundary(sl.ctx, 0.0);
  hdg_solve_info info{};
  if (st == HDG_OK) st = hdg_run(sl.ctx, &info);
  if (st == HDG_OK && q.uex_kind >= 0) st = hdg_errornorm(sl.ctx, q.uex_kind, nullptr, &r.errornorm);
  if (st == HDG_OK && q.want_trace && trace) {
    trace->resize(sz.n_dofs);
    st = hdg_get_trace(sl.ctx, trace->data());
  }
  size_t used = 0;
  if (sl.ctx) hdg_memory_used(sl.ctx, &used);
  r.status = st;
  r.iters = info.iters;
  r.relres = info.relres;
  r.true_relres = info.true_relres;
  r.n_cells = sz.n_cells;
  r.n_dofs = sz.n_dofs;
  r.device_bytes = used;
  r.t_done = S->now();
  return r;
}

// Records a finished request (lock held).
void record(hdg_server* S, const hdg_result& r, std::vector<double>& trace) {
  if (r.status == HDG_OK) {
    ++S->completed;
    S->cells += r.n_cells;
    S->latency.push_back(r.t_done - r.t_submit);
    S->qwait.push_back(r.t_start - r.t_submit);
    S->first_start = std::min(S->first_start, r.t_start);
    S->last_done = std::max(S->last_done, r.t_done);
  } else {
    ++S->failed;
  }
  Done& d = S->done[r.id];
  d.res = r;
  d.trace.swap(trace);
}

// Runs several requests as one hdg_batch in slot w (lock not held).
void run_batch(hdg_server* S, int w, const std::vector<Pending>& batch) {
  const int n = (int)batch.size();
  std::vector<hdg_request> rq(n);
  for (int i = 0; i < n; ++i) rq[i] = batch[i].req;
  const double t_start = S->now();
  std::vector<hdg_result> res(n);
  std::vector<std::vector<double>> traces(n);
  hdg_batch* b = nullptr;
  int st = hdg_batch_create_in_arena(&b, S->device, 0, n, rq.data(), S->arena);
  double t_run = S->now();
  if (st == HDG_OK) {
    hdg_batch_run(b, res.data());  // per-request statuses in res
    for (int i = 0; i < n; ++i)
      if (rq[i].want_trace && res[i].status == HDG_OK) {
        traces[i].resize(res[i].n_dofs);
        if (hdg_batch_trace(b, i, traces[i].data(), (int64_t)traces[i].size()) != HDG_OK) traces[i].clear();
      }
  } else {
    for (int i = 0; i < n; ++i) {
      std::memset(&res[i], 0, sizeof(hdg_result));
      res[i].status = st;
      res[i].t_done = S->now() - t_run;
    }
  }
  if (b) hdg_batch_destroy(b);
  std::lock_guard<std::mutex> lk(S->mu);
  for (int i = 0; i < n; ++i) {
    hdg_result& r = res[i];
    r.id = batch[i].id;
    r.t_submit = batch[i].t_submit;
    r.t_start = t_start;
    r.t_done = t_run + r.t_done;
    r.slot = w;
    record(S, r, traces[i]);
  }
  S->cv_done.notify_all();
}

void worker(hdg_server* S, int w) {
  Slot& sl = S->slots[w];
  std::unique_lock<std::mutex> lk(S->mu);
  for (;;) {
    if (S->stopping && S->queue.empty()) break;
    // first of the next few queued requests whose footprint fits next to
    // what the other slots hold
    int pick = -1;
    const int look = std::min<int>(kLookahead, (int)S->queue.size());
    for (int j = 0; j < look; ++j) {
      const size_t need = S->reserved - sl.held + S->queue[j].foot;
      if (S->budget == 0 || need <= S->budget) {
        pick = j;
        break;
      }
    }
    if (pick < 0) {
      if (!S->queue.empty() && sl.held > 0) {
        // release this idle slot's device data so that the queue can move
        hdg_ctx* c = sl.ctx;
        sl.ctx = nullptr;
        sl.has_mesh = sl.has_setup = false;
        S->reserved -= sl.held;
        sl.held = 0;
        lk.unlock();
        hdg_destroy(c);
        lk.lock();
        S->cv_work.notify_all();
        continue;
      }
      S->cv_work.wait(lk);
      continue;
    }
    Pending p = S->queue[pick];
    S->queue.erase(S->queue.begin() + pick);
    if (S->batch_max > 1 && batchable(p.req)) {
      // continuous batching: the queued requests with the same options that
      // fit the cell cap and the budget join this one in grouped launches
      std::vector<Pending> batch{p};
      size_t foot = p.foot;
      int64_t cells = 2 * p.req.nx * p.req.ny;
      const size_t base = S->reserved - sl.held;
      for (size_t j = 0; j < S->queue.size() && j < (size_t)kBatchLook && (int)batch.size() < S->batch_max;) {
        const Pending& q = S->queue[j];
        const int64_t qc = 2 * q.req.nx * q.req.ny;
        if (batchable(q.req) && same_options(q.req.opt, p.req.opt) && cells + qc <= S->batch_cells &&
            (S->budget == 0 || base + foot + q.foot <= S->budget)) {
          batch.push_back(q);
          foot += q.foot;
          cells += qc;
          S->queue.erase(S->queue.begin() + j);
        } else {
          ++j;
        }
      }
      // the slot's single-request context gives its memory back first
      hdg_ctx* old_ctx = sl.ctx;
      sl.ctx = nullptr;
      sl.has_mesh = sl.has_setup = false;
      S->reserved = base + foot;
      sl.held = foot;
      S->peak = std::max(S->peak, S->reserved);
      lk.unlock();
      if (old_ctx) hdg_destroy(old_ctx);
      run_batch(S, w, batch);
      lk.lock();
      S->reserved -= sl.held;
      sl.held = 0;
      S->cv_work.notify_all();
      continue;
    }
    S->reserved = S->reserved - sl.held + p.foot;
    sl.held = p.foot;
    S->peak = std::max(S->peak, S->reserved);
    lk.unlock();

    std::vector<double> trace;
    hdg_result r = run_request(S, sl, p, &trace);
    r.slot = w;

    lk.lock();
    // hold what the context really holds from now on
    S->reserved = S->reserved - sl.held + r.device_bytes;
    sl.held = r.device_bytes;
    S->peak = std::max(S->peak, S->reserved);
    if (r.status != HDG_OK) {
      // a failed context may hold partial state: start the slot afresh
      hdg_ctx* c = sl.ctx;
      sl.ctx = nullptr;
      sl.has_mesh = sl.has_setup = false;
      S->reserved -= sl.held;
      sl.held = 0;
      lk.unlock();
      hdg_destroy(c);
      lk.lock();
    }
    record(S, r, trace);
    S->cv_done.notify_all();
    S->cv_work.notify_all();
  }
  lk.unlock();
  if (sl.ctx) hdg_destroy(sl.ctx);
  sl.ctx = nullptr;
}

double percentile(std::vector<double> v, double q) {
  if (v.empty()) return 0.0;
  std::sort(v.begin(), v.end());
  const size_t i = (size_t)std::min<double>((double)v.size() - 1, std::ceil(q * v.size()) - 1);
  return v[i];
}

}  // namespace

extern "C" {

size_t hdg_server_footprint(const hdg_request* q) {
  if (!q || q->nx < 1 || q->ny < 1 || q->opt.k < 1 || q->opt.k > 4) return 0;
  const double nx = (double)q->nx, ny = (double)q->ny;
  const double nn = (nx + 1) * (ny + 1), nc = 2 * nx * ny, nf = nx + ny + 3 * nx * ny;
  const int k = q->opt.k, nu = (k + 1) * (k + 2) / 2, m = 3 * nu, nt = k + 1, ntr = 3 * nt;
  const double N = nf * nt;
  // mesh, face pattern
  double b = 16 * nn + 24 * nc + 8 * nf + 67 * nf;
  // per-cell operators, trace solution and Dirichlet data
  b += 8 * nc * ((double)ntr * ntr + ntr + (double)m * ntr + 2 * m) + N * (1 + 8 + 8);
  if (q->opt.precond == HDG_PC_BLOCK_JACOBI) {
    // assembled trace matrix (face-ELL at most) and rhs, Jacobi blocks, CG vectors
    b += N * (8 * 5 * nt + 8 + 8 * nt + 6 * 8);
  }
  // vertex hierarchy over ~4/3 nn nodes: 9-point stencil, inverse, two
  // vectors (12 doubles) and a mask byte per node
  b += (12.0 * 8 + 1) * nn * 4.0 / 3.0;
  if (q->opt.precond != HDG_PC_BLOCK_JACOBI) {
    // the reduced trace system per grid point (hdg_quad.h)
    b += nn * (8 * (8.0 * nt * nt + 37 * nt + 10) + 2);
    if (q->opt.precision == HDG_MIXED) b += nn * 4 * (7.0 * nt * nt + 13 * nt);
  }
  if (q->src.kind == HDG_SRC_VALUES) b += 8 * nc * 16;
  // allocation granularity and small buffers
  return (size_t)(b * 1.05) + (8u << 20);
}

int hdg_server_create(hdg_server** out, int device, size_t hbm_budget, int slots) {
  if (!out || slots < 1 || slots > 64) return HDG_ERR_ARG;
  hdg_server* S = new hdg_server();
  S->device = device;
  S->budget = hbm_budget;
  S->t0 = std::chrono::steady_clock::now();
  // the slots' contexts allocate from one piece of the budget (a failed
  // allocation of it leaves them on the device pool)
  if (hbm_budget > 0 && hdg_arena_create(&S->arena, device, hbm_budget) != HDG_OK) S->arena = nullptr;
  S->slots.resize(slots);
  for (int w = 0; w < slots; ++w) S->threads.emplace_back(worker, S, w);
  *out = S;
  return HDG_OK;
}

int hdg_server_set_batching(hdg_server* S, int max_requests, int64_t max_cells) {
  if (!S || max_requests < 1 || max_cells < 0) return HDG_ERR_ARG;
  std::lock_guard<std::mutex> lk(S->mu);
  S->batch_max = max_requests;
  S->batch_cells = max_cells > 0 ? max_cells : INT64_MAX;
  return HDG_OK;
}

int hdg_server_submit(hdg_server* S, const hdg_request* req, int64_t* id) {
  if (!S || !req || !id) return HDG_ERR_ARG;
  std::lock_guard<std::mutex> lk(S->mu);
  if (req->nx < 1 || req->ny < 1) {
    S->err = "request mesh must have nx, ny >= 1";
    return HDG_ERR_ARG;
  }
  const size_t foot = hdg_server_footprint(req);
  if (foot == 0) {
    S->err = "unsupported request (k must be 1..4)";
    return HDG_ERR_UNSUPPORTED;
  }
  if (S->budget && foot > S->budget) {
    S->err = "request footprint exceeds the server's HBM budget";
    return HDG_ERR_HBM_BUDGET;
  }
  Pending p{S->next_id++, *req, S->now(), foot};
  // The slots launch every kernel from the host and never capture graphs.
  // A serving run whose slots repeated their set-ups (so that each slot
  // captured and replayed CG graphs from its own thread) ended in a host
  // segmentation fault inside the HIP runtime below hipGraph* calls, also
  // with capture, instantiation, destruction and replay serialised
  // process-wide; the cause is not established, so the path is off here.
  // Results are bitwise those of the captured schedule.
  p.req.opt.schedule |= HDG_SCHEDULE_EAGER;
  *id = p.id;
  S->open[p.id] = 1;
  S->queue.push_back(p);
  S->cv_work.notify_one();
  return HDG_OK;
}

int hdg_server_wait(hdg_server* S, int64_t id, double timeout_s, hdg_result* out) {
  if (!S) return HDG_ERR_ARG;
  std::unique_lock<std::mutex> lk(S->mu);
  if (!S->open.count(id) && !S->done.count(id)) {
    S->err = "unknown request id";
    return HDG_ERR_STATE;
  }
  auto ready = [&] { return S->done.count(id) != 0; };
  if (timeout_s < 0) {
    S->cv_done.wait(lk, ready);
  } else if (!S->cv_done.wait_for(lk, std::chrono::duration<double>(timeout_s), ready)) {
    S->err = "timed out waiting for the request";
    return HDG_ERR_NOT_CONVERGED;
  }
  Done& d = S->done[id];
  if (out) *out = d.res;
  S->open.erase(id);
  if (d.trace.empty()) S->done.erase(id);
  return HDG_OK;
}

int hdg_server_trace(hdg_server* S, int64_t id, double* uhat, int64_t cap) {
  if (!S || !uhat) return HDG_ERR_ARG;
  std::lock_guard<std::mutex> lk(S->mu);
  auto it = S->done.find(id);
  if (it == S->done.end() || it->second.trace.empty()) {
    S->err = "no kept trace for this request (want_trace = 0, not completed, or already taken)";
    return HDG_ERR_STATE;
  }
  if (cap < (int64_t)it->second.trace.size()) {
    S->err = "the trace of request " + std::to_string(id) + " has " + std::to_string(it->second.trace.size()) +
             " doubles, more than the buffer's " + std::to_string(cap);
    return HDG_ERR_ARG;
  }
  std::memcpy(uhat, it->second.trace.data(), sizeof(double) * it->second.trace.size());
  S->done.erase(it);
  return HDG_OK;
}

int hdg_server_stats(hdg_server* S, hdg_server_summary* o) {
  if (!S || !o) return HDG_ERR_ARG;
  std::lock_guard<std::mutex> lk(S->mu);
  std::memset(o, 0, sizeof(*o));
  o->completed = S->completed;
  o->failed = S->failed;
  o->cells = S->cells;
  o->p50_latency = percentile(S->latency, 0.50);
  o->p99_latency = percentile(S->latency, 0.99);
  double sl = 0.0, sw = 0.0;
  for (double v : S->latency) sl += v;
  for (double v : S->qwait) sw += v;
  o->mean_latency = S->latency.empty() ? 0.0 : sl / S->latency.size();
  o->mean_queue_wait = S->qwait.empty() ? 0.0 : sw / S->qwait.size();
  o->busy_seconds = S->completed ? S->last_done - S->first_start : 0.0;
  o->cells_per_second = o->busy_seconds > 0 ? S->cells / o->busy_seconds : 0.0;
  o->peak_reserved = S->peak;
  return HDG_OK;
}

void hdg_server_destroy(hdg_server* S) {
  if (!S) return;
  {
    std::lock_guard<std::mutex> lk(S->mu);
    S->stopping = true;
  }
  S->cv_work.notify_all();
  for (auto& t : S->threads) t.join();
  hdg_arena_destroy(S->arena);
  delete S;
}

const char* hdg_server_last_error(const hdg_server* S) { return S ? S->err.c_str() : "null server"; }

}  // extern "C"
