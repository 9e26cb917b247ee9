// Results on their way to host arrays: kernels that write them in the
// caller's layout straight into pinned memory, and the staging that copies
// finished chunks on while the next ones are written.
//
// Bound by the host link: kernel stores to pinned memory reach 52 GB/s (8 MB,
// any store width), the copy engine 53 GB/s; a pageable hipMemcpy into arrays
// already touched 18 GB/s, into fresh ones 10 (page faults on one core); one
// core copies 12 GB/s, eight 70 (27 into fresh pages).  So the layout change
// costs nothing on the device and no pass on the host, and a few threads
// share the copy out of the pinned chunks.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

#include "hdg_host.h"

namespace hdg {

namespace {

constexpr int kBlock = 256;

__global__ __launch_bounds__(kBlock) void stage_copy_kernel(double* __restrict__ dst, const double* __restrict__ src,
                                                            int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

// Cells [e0, e0 + n) of [q; u] and of the cells' face traces as planes.
// ROWS: q[e nq + i], u[e nu + i], uc[(e nt + t) 3 + lf]; else one plane of n
// values per component (q[i n + e], u[i n + e], uc[(t + nt lf) n + e]).
template <int K, bool ROWS>
__global__ __launch_bounds__(kBlock) void stage_values_kernel(DevMesh m, const double* __restrict__ qu,
                                                              const double* __restrict__ uhat, int64_t e0, int64_t n,
                                                              double* __restrict__ q, double* __restrict__ u,
                                                              double* __restrict__ uc) {
  constexpr int NU = (K + 1) * (K + 2) / 2, NQ = 2 * NU, M = 3 * NU, NT = K + 1;
  if constexpr (ROWS) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int64_t e = i / M;
    if (e < n && (q || u)) {
      const int r = (int)(i - e * M);
      const double v = qu[(e0 + e) * M + r];
      if (r < NQ) {
        if (q) q[e * NQ + r] = v;
      } else if (u) {
        u[e * NU + r - NQ] = v;
      }
    }
    const int64_t ec = i / (3 * NT);
    if (uc && ec < n) {
      const int r = (int)(i - ec * 3 * NT);
      uc[i] = uhat[(int64_t)m.cf[3 * (e0 + ec) + r % 3] * NT + r / 3];
    }
  } else {
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= n) return;
    const double* v = qu + (e0 + e) * M;
    if (q)
#pragma unroll
      for (int i = 0; i < NQ; ++i) q[i * n + e] = v[i];
    if (u)
#pragma unroll
      for (int i = 0; i < NU; ++i) u[i * n + e] = v[NQ + i];
    if (uc)
      for (int lf = 0; lf < 3; ++lf) {
        const double* w = uhat + (int64_t)m.cf[3 * (e0 + e) + lf] * NT;
#pragma unroll
        for (int t = 0; t < NT; ++t) uc[(t + NT * lf) * n + e] = w[t];
      }
  }
}

// n matrices of ntr x ntr, transposed one by one
template <int NTR>
__global__ __launch_bounds__(kBlock) void stage_transpose_kernel(double* __restrict__ dst,
                                                                 const double* __restrict__ src, int64_t n) {
  const int64_t o = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int64_t e = o / (NTR * NTR);
  if (e >= n) return;
  const int r = (int)(o - e * (NTR * NTR));
  dst[o] = src[e * (NTR * NTR) + (r % NTR) * NTR + r / NTR];
}

// block columns of kCscFaces faces each
__global__ __launch_bounds__(kBlock) void csc_count_kernel(DevPattern pat, int64_t nf, int64_t* __restrict__ cnt) {
  static_assert(kCscFaces == kBlock, "one face per thread");
  __shared__ int sh[kBlock / 64];
  const int64_t f = (int64_t)blockIdx.x * kCscFaces + threadIdx.x;
  int v = f < nf ? pat.nslot[f] : 0;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    int s = 0;
    for (int w = 0; w < kBlock / 64; ++w) s += sh[w];
    cnt[blockIdx.x] = s;
  }
}

// Julia's CSC of K (the CSR of K^T: column (g, b) holds rows (f, a) for the
// faces f of row g's pattern, which is structurally symmetric, ascending)
// from the face-ELL values: face blocks [b0, b0 + gridDim.x), pre = block
// columns before each.  A wavefront writes the entries of one face after
// another, side by side.
template <int NT, class I>
__global__ __launch_bounds__(kBlock) void csc_fill_kernel(DevPattern pat, const double* __restrict__ vals, int64_t nf,
                                                          int64_t N, int64_t b0, const int64_t* __restrict__ pre,
                                                          int base, I* __restrict__ colptr, I* __restrict__ rowval,
                                                          double* __restrict__ nzval) {
  __shared__ int off[kCscFaces + 1];
  const int64_t blk = b0 + blockIdx.x, g0 = blk * kCscFaces;
  const int t = threadIdx.x, nfb = (int)min((int64_t)kCscFaces, nf - g0);
  off[t + 1] = t < nfb ? pat.nslot[g0 + t] : 0;
  if (t == 0) off[0] = 0;
  __syncthreads();
  for (int d = 1; d < kCscFaces; d <<= 1) {
    const int v = t + 1 > d ? off[t + 1 - d] : 0;
    __syncthreads();
    off[t + 1] += v;
    __syncthreads();
  }
  // entries before this chunk's first face, and before this block within it
  const int64_t before = pre[blk] * (NT * NT), lead = (pre[blk] - pre[b0]) * (NT * NT);
  if (colptr)
    for (int i = t; i < nfb * NT; i += kBlock) {
      const int j = i / NT, b = i % NT;
      colptr[(int64_t)blockIdx.x * kCscFaces * NT + i] =
          (I)(before + (int64_t)off[j] * (NT * NT) + (off[j + 1] - off[j]) * NT * b + base);
    }
  if (!rowval && !nzval) return;
  for (int j = t >> 6; j < nfb; j += kBlock / 64) {
    const int64_t g = g0 + j, w0 = lead + (int64_t)off[j] * (NT * NT);
    const int ns = off[j + 1] - off[j], per = ns * NT;
    for (int i = t & 63; i < per * NT; i += 64) {
      const int b = i / per, r = i - b * per, s = r / NT, a = r % NT;
      const int64_t f = pat.bcol[kSlots * g + s];
      if (rowval) rowval[w0 + i] = (I)(f * NT + a + base);
      if (nzval) nzval[w0 + i] = vals[(int64_t)(pat.tslot[kSlots * g + s] * NT + b) * N + f * NT + a];
    }
  }
}

unsigned grid_of(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

constexpr size_t kChunk = 4u << 20, kHeadAlign = 4096;
constexpr int kCrew = 8;
// below this much, waking threads costs more than they save (spawning eight
// takes 110 us, one core copies 2 MB in 170)
constexpr size_t kPerThread = 2u << 20;

// Where a chunk's bytes go: bytes[i] from offset off[i] to dst[i].
struct StagePieces {
  static constexpr int kMax = 64;
  int n = 0;
  char* dst[kMax];
  size_t off[kMax], bytes[kMax];
  void add(void* d, size_t o, size_t b) {
    dst[n] = static_cast<char*>(d);
    off[n] = o;
    bytes[n++] = b;
  }
};
// Launches on the stream the kernels that write chunk k to buf and lists its
// pieces; a hipError_t.
using StageFill = int (*)(void* arg, int64_t k, char* buf, StagePieces& out);
// Share t of nshares of a chunk.
void copy_share(const char* buf, const StagePieces& p, int t, int nshares) {
  size_t total = 0;
  for (int i = 0; i < p.n; ++i) total += p.bytes[i];
  size_t lo = total / nshares * t, hi = t + 1 == nshares ? total : total / nshares * (t + 1), at = 0;
  for (int i = 0; i < p.n && at < hi; at += p.bytes[i++]) {
    const size_t a = std::max(lo, at), b = std::min(hi, at + p.bytes[i]);
    if (a < b) std::memcpy(p.dst[i] + (a - at), buf + p.off[i] + (a - at), b - a);
  }
}

// The process's pinned memory for exports, in pieces of two sizes (one chunk,
// or kStageBufs of them, and a head) that are lent to one export each, on any stream or thread.  Pinning costs 0.25-0.3 ms a
// piece whatever its size (30 us where nothing was unpinned before it), more
// than a small export: with pieces of its own, grown twice, a new context's
// first export of 12 x 9 P1 cells took 1.2 ms, now 0.4.  Up to kIdle of each
// size wait for the next export; when the last context and batch go, all but
// one small piece are given back.
constexpr size_t kSmallPiece = kChunk + (64u << 10), kLargePiece = kStageBufs * kChunk + (1u << 20);
constexpr int kIdle = 8;
struct StagePiece {
  char* mem = nullptr;
  size_t bytes = 0;
  int device = -1;
  bool small() const { return bytes <= kSmallPiece; }
};
struct StagePool {
  std::mutex m;
  int owners = 0, n = 0;
  StagePiece idle[2 * kIdle];
};
StagePool& stage_pool() {
  static StagePool* p = new StagePool;  // outlives every owner, static ones too
  return *p;
}

// Memory for a result of `total` bytes and a head of `head` bytes: bufs chunks
// behind the head; 0 or a hipError_t in err.
struct StageLease {
  HostStage& st;
  StagePiece p;
  int err = 0;
  size_t head, chunk, bufs;
  StageLease(HostStage& owner, size_t total, size_t head_bytes) : st(owner) {
    head = (head_bytes + kHeadAlign - 1) / kHeadAlign * kHeadAlign;
    // one buffer for what fits, else kStageBufs chunks
    const size_t one = std::max<size_t>(65536, (total + 4095) / 4096 * 4096);
    chunk = std::min(one, kChunk);
    bufs = total <= chunk ? 1 : kStageBufs;
    hipError_t e = hipSuccess;
    for (hipEvent_t& ev : st.ev)
      if (!ev && e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    const size_t need = head + bufs * chunk;
    int device = 0;
    if (e == hipSuccess) e = hipGetDevice(&device);
    if (e == hipSuccess) {
      StagePool& pool = stage_pool();
      std::lock_guard<std::mutex> lk(pool.m);
      int best = -1;
      for (int i = 0; i < pool.n; ++i)
        if (pool.idle[i].device == device && pool.idle[i].bytes >= need &&
            (best < 0 || pool.idle[i].bytes < pool.idle[best].bytes))
          best = i;
      if (best >= 0) {
        p = pool.idle[best];
        pool.idle[best] = pool.idle[--pool.n];
      }
    }
    if (e == hipSuccess && !p.mem) {
      const size_t mb = 1u << 20, bytes = need <= kSmallPiece ? kSmallPiece : std::max(kLargePiece, (need + mb - 1) / mb * mb);
      e = hipHostMalloc((void**)&p.mem, bytes, hipHostMallocDefault);
      if (e != hipSuccess) p.mem = nullptr;
      p.bytes = bytes;
      p.device = device;
    }
    err = (int)e;
  }
  // after the export: nothing on the device writes the piece any more
  ~StageLease() {
    if (!p.mem) return;
    {
      StagePool& pool = stage_pool();
      std::lock_guard<std::mutex> lk(pool.m);
      int same = 0;
      for (int i = 0; i < pool.n; ++i) same += pool.idle[i].small() == p.small();
      if (same < kIdle) {
        pool.idle[pool.n++] = p;
        return;
      }
    }
    (void)hipHostFree(p.mem);
  }
  StageLease(const StageLease&) = delete;
  StageLease& operator=(const StageLease&) = delete;
  char* chunk_at(int64_t b) const { return p.mem + head + b * chunk; }
};

// A wait of some microseconds: spins, and lets go of the core only when it has
// lasted long.  (Where other threads spin on every core, as a BLAS library's do
// for tens of milliseconds after a product, a thread that yields or sleeps gets
// its core back 3 ms later: with a sleep per chunk and yields between the
// chunks, 54 MB took 45 ms beside such threads; now 3 to 5, and 1.2 without them.)
struct Patience {
  int n = 0;
  void wait() {
    if (++n < 20000)
      __builtin_ia32_pause();
    else
      std::this_thread::yield();
  }
};

// Writes nchunks chunks (total bytes in all) and copies each out while the
// next ones are written; returns when everything has arrived.  A chunk is
// copied in shares, taken by the caller's thread and by those of a crew
// as each is free: nothing waits for a thread that has no core, except to the
// end of a share it has begun.
int staged_out(StageLease& L, hipStream_t s, int64_t nchunks, size_t total, StageFill fill, void* arg) {
  HostStage& st = L.st;
  StagePieces pieces[kStageBufs];
  std::atomic<int64_t> ready{0};  // chunks that have arrived in their buffers
  std::atomic<int64_t> taken{0};  // shares taken, over all chunks
  std::atomic<int64_t> done[kStageBufs] = {};  // shares copied from each buffer
  std::atomic<bool> stop{false};
  std::thread crew[kCrew];
  const int nb = (int)L.bufs;
  const int want = (int)std::min<size_t>({(size_t)kCrew, total / kPerThread,
                                          (size_t)std::max(1u, std::thread::hardware_concurrency() / 2)});
  const int shares = want > 1 ? 2 * kCrew : 1;
  // takes and copies one share of what has arrived
  const auto copy_one = [&]() -> bool {
    int64_t i = taken.load(std::memory_order_relaxed);
    do {
      if (i >= ready.load(std::memory_order_acquire) * shares) return false;
    } while (!taken.compare_exchange_weak(i, i + 1, std::memory_order_relaxed));
    const int b = (int)(i / shares % nb);
    copy_share(L.chunk_at(b), pieces[b], (int)(i % shares), shares);
    done[b].fetch_add(1, std::memory_order_release);
    return true;
  };
  const auto work = [&]() {
    Patience p;
    while (!stop.load(std::memory_order_acquire) && taken.load(std::memory_order_relaxed) < nchunks * shares)
      if (copy_one())
        p = Patience{};
      else
        p.wait();
  };
  const auto launch = [&](int64_t k) {
    StagePieces& p = pieces[k % nb];
    p.n = 0;
    int r = fill(arg, k, L.chunk_at(k % nb), p);
    if (!r) r = (int)hipEventRecord(st.ev[k % nb], s);
    return r;
  };
  int e = 0;
  int64_t launched = 0, arrived = 0, copied = 0;
  while (launched < nchunks && launched < nb && !e)
    if (!(e = launch(launched))) ++launched;
  // the crew starts beside the first chunks
  try {
    for (int t = 1; !e && t < want; ++t) crew[t] = std::thread(work);
  } catch (...) {  // fewer, then
  }
  Patience p;
  while (copied < nchunks && !e) {
    bool moved = false;
    if (arrived < launched) {
      hipError_t q = hipEventQuery(st.ev[arrived % nb]);
      if (q == hipErrorNotReady) {
        (void)hipGetLastError();
        // long work ahead of the export on the stream
        if (p.n > 4000 && copied == arrived) q = hipEventSynchronize(st.ev[arrived % nb]);
      }
      if (q == hipSuccess) {
        ready.store(++arrived, std::memory_order_release);
        moved = true;
      } else if (q != hipErrorNotReady) {
        e = (int)q;
        break;
      }
    }
    if (copy_one()) moved = true;
    if (copied < arrived && done[copied % nb].load(std::memory_order_acquire) == (copied / nb + 1) * shares) {
      ++copied;
      moved = true;
      if (launched < nchunks && !(e = launch(launched))) ++launched;
    }
    if (moved)
      p = Patience{};
    else
      p.wait();
  }
  stop.store(true, std::memory_order_release);
  for (std::thread& t : crew)
    if (t.joinable()) t.join();
  if (e) (void)hipStreamSynchronize(s);
  return e;
}

}  // namespace

HostStage::HostStage() {
  StagePool& pool = stage_pool();
  std::lock_guard<std::mutex> lk(pool.m);
  ++pool.owners;
}

HostStage::~HostStage() {
  StagePiece out[2 * kIdle];
  int n = 0;
  {
    StagePool& pool = stage_pool();
    std::lock_guard<std::mutex> lk(pool.m);
    if (--pool.owners > 0) return;
    int kept = 0;
    for (int i = 0; i < pool.n; ++i)
      if (pool.idle[i].small() && kept == 0)
        pool.idle[kept++] = pool.idle[i];
      else
        out[n++] = pool.idle[i];
    pool.n = kept;
  }
  for (int i = 0; i < n; ++i) (void)hipHostFree(out[i].mem);
}

void stage_free(HostStage& st) {
  for (hipEvent_t& e : st.ev)
    if (e) {
      (void)hipEventDestroy(e);
      e = nullptr;
    }
}

int staged_copy(HostStage& st, hipStream_t s, double* dst, const double* src, int64_t n) {
  std::lock_guard<std::mutex> lk(st.m);
  StageLease L(st, sizeof(double) * n, 0);
  if (L.err) return L.err;
  struct Arg {
    double* dst;
    const double* src;
    int64_t n, per;
    hipStream_t s;
  } a{dst, src, n, (int64_t)(L.chunk / sizeof(double)), s};
  return staged_out(
      L, s, (n + a.per - 1) / a.per, sizeof(double) * n,
      [](void* p, int64_t k, char* buf, StagePieces& out) {
        const Arg& a = *static_cast<Arg*>(p);
        const int64_t i0 = k * a.per, m = std::min(a.per, a.n - i0);
        hipLaunchKernelGGL(stage_copy_kernel, dim3(grid_of(m)), dim3(kBlock), 0, a.s, (double*)buf, a.src + i0, m);
        out.add(a.dst + i0, 0, sizeof(double) * m);
        return (int)hipGetLastError();
      },
      &a);
}

int staged_values(HostStage& st, hipStream_t s, int k, const DevMesh& m, const double* qu, const double* uhat,
                  bool rows, double* q, double* u, double* uc) {
  const int nu = (k + 1) * (k + 2) / 2, nt = k + 1;
  const int per = (q ? 2 * nu : 0) + (u ? nu : 0) + (uc ? 3 * nt : 0);  // doubles per cell
  if (!per) return 0;
  const size_t total = sizeof(double) * per * m.nc;
  std::lock_guard<std::mutex> lk(st.m);
  StageLease L(st, total, 0);
  if (L.err) return L.err;
  struct Arg {
    int k, nu, nt;
    DevMesh m;
    const double *qu, *uhat;
    bool rows;
    double *q, *u, *uc;
    int64_t per;
    hipStream_t s;
  } a{k, nu, nt, m, qu, uhat, rows, q, u, uc, (int64_t)(L.chunk / (sizeof(double) * per)), s};
  return staged_out(
      L, s, (m.nc + a.per - 1) / a.per, total,
      [](void* p, int64_t c, char* buf, StagePieces& out) {
        const Arg& a = *static_cast<Arg*>(p);
        const int64_t nc = a.m.nc, e0 = c * a.per, n = std::min(a.per, nc - e0);
        const int nq = 2 * a.nu, nf = 3 * a.nt;
        double* b = (double*)buf;
        double *q = a.q ? b : nullptr, *u = nullptr, *uc = nullptr;
        if (a.q) b += nq * n;
        if (a.u) u = b, b += a.nu * n;
        if (a.uc) uc = b;
        const auto plane = [&](double* dst, double* src, int w) {
          if (!dst) return;
          const size_t off = (char*)src - buf;
          if (a.rows)
            out.add(dst + e0 * w, off, sizeof(double) * w * n);
          else
            for (int i = 0; i < w; ++i) out.add(dst + nc * i + e0, off + sizeof(double) * n * i, sizeof(double) * n);
        };
        plane(a.q, q, nq);
        plane(a.u, u, a.nu);
        plane(a.uc, uc, nf);
#define VALUES(K)                                                                                             \
  case K:                                                                                                     \
    if (a.rows)                                                                                               \
      hipLaunchKernelGGL((stage_values_kernel<K, true>), dim3(grid_of(n * std::max(nq + a.nu, nf))),          \
                         dim3(kBlock), 0, a.s, a.m, a.qu, a.uhat, e0, n, q, u, uc);                           \
    else                                                                                                      \
      hipLaunchKernelGGL((stage_values_kernel<K, false>), dim3(grid_of(n)), dim3(kBlock), 0, a.s, a.m, a.qu,  \
                         a.uhat, e0, n, q, u, uc);                                                            \
    break;
        switch (a.k) { VALUES(1) VALUES(2) VALUES(3) VALUES(4) }
#undef VALUES
        return (int)hipGetLastError();
      },
      &a);
}

int staged_transposes(HostStage& st, hipStream_t s, int k, double* dst, const double* src, int64_t nc) {
  const int ntr = 3 * (k + 1), w = ntr * ntr;
  const size_t total = sizeof(double) * w * nc;
  std::lock_guard<std::mutex> lk(st.m);
  StageLease L(st, total, 0);
  if (L.err) return L.err;
  struct Arg {
    int k, w;
    double* dst;
    const double* src;
    int64_t nc, per;
    hipStream_t s;
  } a{k, w, dst, src, nc, (int64_t)(L.chunk / (sizeof(double) * w)), s};
  return staged_out(
      L, s, (nc + a.per - 1) / a.per, total,
      [](void* p, int64_t c, char* buf, StagePieces& out) {
        const Arg& a = *static_cast<Arg*>(p);
        const int64_t e0 = c * a.per, n = std::min(a.per, a.nc - e0);
        const dim3 g(grid_of(n * a.w));
        const double* src = a.src + e0 * a.w;
        switch (a.k) {
          case 1: hipLaunchKernelGGL(stage_transpose_kernel<6>, g, dim3(kBlock), 0, a.s, (double*)buf, src, n); break;
          case 2: hipLaunchKernelGGL(stage_transpose_kernel<9>, g, dim3(kBlock), 0, a.s, (double*)buf, src, n); break;
          case 3: hipLaunchKernelGGL(stage_transpose_kernel<12>, g, dim3(kBlock), 0, a.s, (double*)buf, src, n); break;
          case 4: hipLaunchKernelGGL(stage_transpose_kernel<15>, g, dim3(kBlock), 0, a.s, (double*)buf, src, n); break;
        }
        out.add(a.dst + e0 * a.w, 0, sizeof(double) * a.w * n);
        return (int)hipGetLastError();
      },
      &a);
}

namespace {

template <class I>
struct CscArg {
  DevPattern pat;
  const double* vals;
  int64_t nf, N, nblk, per;
  int nt, base;
  const int64_t* pre;
  I *colptr, *rowval;
  double* nzval;
  hipStream_t s;
};

template <class I>
int csc_chunk(void* p, int64_t c, char* buf, StagePieces& out) {
  const CscArg<I>& a = *static_cast<CscArg<I>*>(p);
  const int64_t b0 = c * a.per, b1 = std::min(a.nblk, b0 + a.per);
  const int64_t g0 = b0 * kCscFaces, g1 = std::min(a.nf, b1 * kCscFaces), nt2 = (int64_t)a.nt * a.nt;
  const int64_t w0 = a.pre[b0] * nt2, nw = a.pre[b1] * nt2 - w0, ncol = (g1 - g0) * a.nt;
  // doubles first, so that every plane is aligned
  size_t at = 0;
  double* nz = a.nzval ? (double*)buf : nullptr;
  if (nz) out.add(a.nzval + w0, at, sizeof(double) * nw), at += sizeof(double) * nw;
  I* rv = a.rowval ? (I*)(buf + at) : nullptr;
  if (rv) out.add(a.rowval + w0, at, sizeof(I) * nw), at += sizeof(I) * nw;
  I* cp = a.colptr ? (I*)(buf + at) : nullptr;
  if (cp) out.add(a.colptr + g0 * a.nt, at, sizeof(I) * ncol);
  const dim3 g((unsigned)(b1 - b0));
#define FILL(NT)                                                                                                    \
  case NT:                                                                                                          \
    hipLaunchKernelGGL((csc_fill_kernel<NT, I>), g, dim3(kBlock), 0, a.s, a.pat, a.vals, a.nf, a.N, b0, a.pre,      \
                       a.base, cp, rv, nz);                                                                         \
    break;
  switch (a.nt) { FILL(2) FILL(3) FILL(4) FILL(5) }
#undef FILL
  return (int)hipGetLastError();
}

}  // namespace

template <class I>
int staged_csc(HostStage& st, hipStream_t s, const DevPattern& pat, int nt, int64_t nf, const double* vals, int base,
               I* colptr, I* rowval, double* nzval) {
  if (!colptr && !rowval && !nzval) return 0;
  const int64_t nblk = (nf + kCscFaces - 1) / kCscFaces;
  const size_t face = (size_t)kSlots * nt * nt * ((rowval ? sizeof(I) : 0) + (nzval ? sizeof(double) : 0)) +
                      (colptr ? sizeof(I) * nt : 0);
  const size_t total = face * nf;
  // at least one block of faces per chunk (524 KB at five modes)
  std::lock_guard<std::mutex> lk(st.m);
  StageLease L(st, std::max<size_t>(total, face * kCscFaces), sizeof(int64_t) * (nblk + 1));
  if (L.err) return L.err;
  int64_t* pre = (int64_t*)L.p.mem;
  hipLaunchKernelGGL(csc_count_kernel, dim3((unsigned)nblk), dim3(kBlock), 0, s, pat, nf, pre);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return (int)e;
  int64_t sum = 0;
  for (int64_t b = 0; b <= nblk; ++b) {
    const int64_t n = b < nblk ? pre[b] : 0;
    pre[b] = sum;
    sum += n;
  }
  const int64_t nb = (int64_t)(L.chunk / (face * kCscFaces));
  CscArg<I> a{pat, vals, nf, nf * nt, nblk, nb, nt, base, pre, colptr, rowval, nzval, s};
  const int r = staged_out(L, s, (nblk + nb - 1) / nb, total, csc_chunk<I>, &a);
  if (!r && colptr) colptr[nf * nt] = (I)(sum * nt * nt + base);
  return r;
}
template int staged_csc<int32_t>(HostStage&, hipStream_t, const DevPattern&, int, int64_t, const double*, int,
                                 int32_t*, int32_t*, double*);
template int staged_csc<int64_t>(HostStage&, hipStream_t, const DevPattern&, int, int64_t, const double*, int,
                                 int64_t*, int64_t*, double*);

}  // namespace hdg
