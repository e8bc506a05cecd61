// Range check of selection block ids, split into an enqueue and a wait so that the host can
// enqueue the work that follows before it waits.
//
// Reference semantics: nsa/ops/selection/__init__.py:36-42 (a valid id >= the number of blocks is
// an error; negative ids mean "no block").
//
// One kernel reads the ids once and stores 1 into a mapped host word when one is out of range; the
// event recorded behind it is all the host waits for, while the attention enqueued next already
// runs (its kernels skip out-of-range ids, so an error only discards their result).  98,304 ids
// behind an idle GPU: one launch of about 3 us.  The same check as tensor expressions took 12
// launches and 3 waits with the GPU idle in between: attention over 32760 tokens 403 -> 278 us a call
// in a loop of calls, over 1560 tokens (with its pooling and top-k) 161 -> 79 us.
#include <mutex>
#include <vector>

#include "omm_common.h"

namespace omm {
namespace {

constexpr int kCheckThreads = 256;
constexpr int kCheckVec = 4;         // ids per thread and step on a contiguous view
constexpr unsigned kCheckGrid = 256;  // one workgroup per CU: 98,304 ids are 1.5 steps of it

__device__ __forceinline__ void report_bad(int32_t* flag) {
  __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ __launch_bounds__(kCheckThreads) void ids_check_flat_kernel(const int32_t* ids,
                                                                       int64_t n, int32_t limit,
                                                                       int32_t* flag) {
  const int64_t step = static_cast<int64_t>(gridDim.x) * kCheckThreads;
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kCheckThreads + threadIdx.x;
  bool bad = false;
  for (int64_t i = i0; i < n / kCheckVec; i += step) {
    const int4 v = reinterpret_cast<const int4*>(ids)[i];
    bad = bad || v.x >= limit || v.y >= limit || v.z >= limit || v.w >= limit;
  }
  if (i0 < n % kCheckVec) bad = bad || ids[n / kCheckVec * kCheckVec + i0] >= limit;
  if (bad) report_bad(flag);
}

__global__ __launch_bounds__(kCheckThreads) void ids_check_view_kernel(View4<const int32_t> ids,
                                                                       int64_t n1, int64_t n2,
                                                                       int64_t n3, int64_t n,
                                                                       int32_t limit,
                                                                       int32_t* flag) {
  bool bad = false;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kCheckThreads + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * kCheckThreads) {
    const int64_t t = i % n3, r = i / n3, h = r % n2, q = r / n2;
    bad = bad || *ids.at(q / n1, q % n1, h, t) >= limit;
  }
  if (bad) report_bad(flag);
}

// A check in flight: its host word and event, and the device both belong to.
struct Ticket {
  int dev;
  int32_t* host;
  int32_t* word;  // the same word at its device address
  hipEvent_t ev;
};

// Idle tickets, at most kKeep per process; the others are destroyed when they are done.  A
// ticket belongs to one check between begin and end, so threads and streams never share one.
constexpr size_t kKeep = 32;
std::mutex g_mu;
std::vector<Ticket*> g_idle;

void destroy(Ticket* t) {
  (void)hipEventDestroy(t->ev);
  (void)hipHostFree(t->host);
  delete t;
}

void put_back(Ticket* t) {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_idle.size() < kKeep) {
      g_idle.push_back(t);
      return;
    }
  }
  destroy(t);
}

int take(int dev, Ticket** out) {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    for (size_t i = g_idle.size(); i-- > 0;)
      if (g_idle[i]->dev == dev) {
        *out = g_idle[i];
        g_idle[i] = g_idle.back();
        g_idle.pop_back();
        return OMM_OK;
      }
  }
  void *h = nullptr, *d = nullptr;
  hipError_t e = hipHostMalloc(&h, sizeof(int32_t), hipHostMallocMapped | hipHostMallocCoherent);
  if (e != hipSuccess) return set_error(OMM_EHIP, "omm_ids_check: %s", hipGetErrorString(e));
  hipEvent_t ev = nullptr;
  e = hipHostGetDevicePointer(&d, h, 0);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
  if (e != hipSuccess) {
    (void)hipHostFree(h);
    return set_error(OMM_EHIP, "omm_ids_check: %s", hipGetErrorString(e));
  }
  *out = new Ticket{dev, static_cast<int32_t*>(h), static_cast<int32_t*>(d), ev};
  return OMM_OK;
}

int begin(const omm_view4& ids, int64_t num_blocks, hipStream_t s, Ticket** out) {
  const int64_t n = ids.size[0] * ids.size[1] * ids.size[2] * ids.size[3];
  if (n == 0 || num_blocks > 2147483647ll) return OMM_OK;  // no id can be out of range
  int dev = -1;
  const hipError_t de = hipGetDevice(&dev);
  if (de != hipSuccess) return set_error(OMM_EHIP, "omm_ids_check: %s", hipGetErrorString(de));
  Ticket* t = nullptr;
  int rc = take(dev, &t);
  if (rc != OMM_OK) return rc;
  *t->host = 0;
  const int32_t limit = static_cast<int32_t>(num_blocks);
  int64_t run = 1;
  bool flat = (reinterpret_cast<uintptr_t>(ids.data) & 15u) == 0;
  for (int i = 3; i >= 0; --i) {
    flat = flat && (ids.size[i] == 1 || ids.stride[i] == run);
    run *= ids.size[i];
  }
  const int64_t items = flat ? cdiv64(n, kCheckVec) : n;
  const unsigned grid =
      static_cast<unsigned>(std::min<int64_t>(cdiv64(items, kCheckThreads), kCheckGrid));
  if (flat)
    ids_check_flat_kernel<<<grid, kCheckThreads, 0, s>>>(static_cast<const int32_t*>(ids.data), n,
                                                         limit, t->word);
  else
    ids_check_view_kernel<<<grid, kCheckThreads, 0, s>>>(make_view<const int32_t>(ids),
                                                         ids.size[1], ids.size[2], ids.size[3], n,
                                                         limit, t->word);
  rc = check_launch("block id check");
  if (rc == OMM_OK) {
    const hipError_t e = hipEventRecord(t->ev, s);
    if (e != hipSuccess) {
      rc = set_error(OMM_EHIP, "omm_ids_check: %s", hipGetErrorString(e));
      (void)hipStreamSynchronize(s);  // the kernel may still write the ticket's word
    }
  }
  if (rc != OMM_OK) {
    destroy(t);
    return rc;
  }
  *out = t;
  return OMM_OK;
}

}  // namespace
}  // namespace omm

extern "C" int omm_ids_check_begin(const omm_view4* ids, int64_t num_blocks, void* stream,
                                   void** ticket) {
  using namespace omm;
  OMM_REQUIRE(ids != nullptr && ticket != nullptr, OMM_EINVAL, "omm_ids_check: null argument");
  *ticket = nullptr;
  OMM_REQUIRE(num_blocks >= 0, OMM_EINVAL, "omm_ids_check: negative number of blocks");
  for (int i = 0; i < 4; ++i)
    OMM_REQUIRE(ids->size[i] >= 0 && ids->stride[i] >= 0, OMM_EINVAL,
                "omm_ids_check: negative size or stride");
  Ticket* t = nullptr;
  try {
    const int rc = begin(*ids, num_blocks, static_cast<hipStream_t>(stream), &t);
    if (rc != OMM_OK) return rc;
  } catch (const std::exception& e) {
    return set_error(OMM_EHIP, "omm_ids_check: %s", e.what());
  }
  *ticket = t;
  return OMM_OK;
}

extern "C" int omm_ids_check_end(void* ticket, int32_t* bad) {
  using namespace omm;
  OMM_REQUIRE(bad != nullptr, OMM_EINVAL, "omm_ids_check_end: null output");
  *bad = 0;
  if (ticket == nullptr) return OMM_OK;
  Ticket* t = static_cast<Ticket*>(ticket);
  const hipError_t e = hipEventSynchronize(t->ev);
  if (e != hipSuccess)  // the kernel may not have run: neither the word nor the event is reused
    return set_error(OMM_EHIP, "omm_ids_check_end: %s", hipGetErrorString(e));
  *bad = __atomic_load_n(t->host, __ATOMIC_ACQUIRE);
  try {
    put_back(t);
  } catch (const std::exception& ex) {
    destroy(t);
    return set_error(OMM_EHIP, "omm_ids_check_end: %s", ex.what());
  }
  return OMM_OK;
}
