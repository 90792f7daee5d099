// Device buffers of one network (host code; hipMalloc, hipFree and
// hipGetLastError only, so it can be compiled and checked without a GPU).  A
// buffer is never left pointing at memory that is not its own: a growth that
// fails leaves null pointers and no capacity, so the next call allocates
// again, and the loss, which every training call writes whatever its capacity,
// is replaced only once the new buffer is there.
#pragma once
#include <hip/hip_runtime_api.h>
#include <algorithm>
#include <vector>

struct DevPool {
  std::vector<void *> owned;
  template <typename P> hipError_t get(size_t bytes, P *&out) {
    void *q = nullptr;
    out = nullptr;
    const hipError_t e = hipMalloc(&q, bytes ? bytes : 16);
    if (e != hipSuccess) {
      (void)hipGetLastError();         // reported here, not by the next launch's check
      return e;
    }
    owned.push_back(q);
    out = (P *)q;
    return e;
  }
  template <typename P> void drop(P *&p) {
    if (!p) return;
    owned.erase(std::remove(owned.begin(), owned.end(), (void *)p), owned.end());
    (void)hipFree((void *)p);
    p = nullptr;
  }
  void clear() {
    for (void *q : owned) (void)hipFree(q);
    owned.clear();
  }
};

// Batch buffers of k_mlp_rows for up to cap rows (hid: units of all hidden layers).
struct MlpRowBufs {
  int cap = 0;
  short *actT = nullptr, *dzT = nullptr;
  float *act32 = nullptr, *part = nullptr, *losspart = nullptr;
  hipError_t reserve(DevPool &pool, size_t nin_p, size_t hid, int B) {
    if (B <= cap) return hipSuccess;
    pool.drop(actT); pool.drop(dzT); pool.drop(act32); pool.drop(part); pool.drop(losspart);
    cap = 0;
    hipError_t e;
    if ((e = pool.get(sizeof(short) * (nin_p + hid) * B, actT)) != hipSuccess) return e;
    if ((e = pool.get(sizeof(short) * (hid + 16) * B, dzT)) != hipSuccess) return e;
    if ((e = pool.get(sizeof(float) * hid * B, act32)) != hipSuccess) return e;
    if ((e = pool.get(sizeof(float) * (hid + 16) * (B / 16), part)) != hipSuccess) return e;
    if ((e = pool.get(sizeof(float) * (B / 16), losspart)) != hipSuccess) return e;
    cap = B;
    return e;
  }
};

// A data set of up to cap rows: normalised (k_mlp_normalize) and as uploaded.
struct MlpSetBufs {
  int cap = 0;
  float *X = nullptr, *T = nullptr, *xraw = nullptr, *traw = nullptr;
  hipError_t reserve(DevPool &pool, int nin, int nin_p, int nout, int n) {
    if (n <= cap) return hipSuccess;
    pool.drop(X); pool.drop(T); pool.drop(xraw); pool.drop(traw);
    cap = 0;
    hipError_t e;
    if ((e = pool.get(sizeof(float) * (size_t)n * nin_p, X)) != hipSuccess) return e;
    if ((e = pool.get(sizeof(float) * (size_t)n * nout, T)) != hipSuccess) return e;
    if ((e = pool.get(sizeof(float) * (size_t)n * nin, xraw)) != hipSuccess) return e;
    if ((e = pool.get(sizeof(float) * (size_t)n * nout, traw)) != hipSuccess) return e;
    cap = n;
    return e;
  }
};

// The loss of the last step, then those of up to cap steps.
struct MlpLossBuf {
  int cap = -1;
  float *p = nullptr;
  hipError_t reserve(DevPool &pool, int steps) {
    if (steps <= cap) return hipSuccess;
    float *q;
    const hipError_t e = pool.get(sizeof(float) * ((size_t)steps + 1), q);
    if (e != hipSuccess) return e;
    pool.drop(p);
    p = q;
    cap = steps;
    return e;
  }
};
