// Host-side helpers shared by the single-problem C ABI (hdg_api.hip) and the
// batches (hdg_batch.hip).  Not part of the public ABI.
#pragma once
#include <mutex>

#include "hdg_internal.h"

namespace hdg {

// Sizes of the vertex hierarchy of an nx x ny rectangle mesh: fills nlev,
// lev[1..nlev-1].nx, ny, n and tail (no device arrays).
void mg_plan_levels(int nx, int ny, MgData& M);

// An owner of exports, a context or a batch: the events of its chunks; its
// concurrent exports take turns.  The pinned memory through which results leave
// for host arrays is the process's, lent to one export at a time.
constexpr int kStageBufs = 3;
struct HostStage {
  std::mutex m;
  hipEvent_t ev[kStageBufs] = {};
  HostStage();
  ~HostStage();
  HostStage(const HostStage&) = delete;
  HostStage& operator=(const HostStage&) = delete;
};
void stage_free(HostStage& st);

// Each returns a hipError_t, the results in place.
// n doubles of device memory to host memory
int staged_copy(HostStage& st, hipStream_t s, double* dst, const double* src, int64_t n);
// q, u and the cells' face traces of order k (any may be null): one row per
// cell, or one column per component
int staged_values(HostStage& st, hipStream_t s, int k, const DevMesh& m, const double* qu, const double* uhat,
                  bool rows, double* q, double* u, double* uc);
// nc matrices of (3 nt)^2, each transposed
int staged_transposes(HostStage& st, hipStream_t s, int k, double* dst, const double* src, int64_t nc);
// CSC of the trace matrix from its face-ELL values, indices from `base`
constexpr int kCscFaces = 256;
template <class I>
int staged_csc(HostStage& st, hipStream_t s, const DevPattern& pat, int nt, int64_t nf, const double* vals, int base,
               I* colptr, I* rowval, double* nzval);

}  // namespace hdg
