// Internal host-side types shared by the C ABI translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>
#include <vector>

#include "../../include/qmm.h"

namespace qmm {

constexpr int QMM_MAX_DIM = 8;

size_t dtype_size(qmm_dtype d);

// The object behind a qmm_array handle: an HBM buffer plus shape and dtype.
struct Arr {
  void *data = nullptr;
  bool owned = false;                   // free the buffer with the handle
  hipStream_t alloc_stream = nullptr;   // stream the buffer was allocated on (stream-ordered free)
  int device = -1;                      // an owned buffer's device
  int ndim = 0;
  int shape[QMM_MAX_DIM] = {0};
  qmm_dtype dtype = QMM_BOOL;
  // For a scales array: a copy in the prefill GEMMs' tile-major layout (tiled_bytes bytes,
  // a plain allocation), made at the first prefill call that reads it, complete on the
  // device before it is set, and freed with the handle (release_tiled).
  void *tiled = nullptr;
  size_t tiled_bytes = 0;
  size_t size() const;
  size_t nbytes() const { return size() * dtype_size(dtype); }
};

struct Stream {
  hipStream_t h = nullptr;
};

struct VecArr {
  std::vector<Arr *> items;
};

void latch_error(const char *msg);
int fail(const char *fmt, ...) __attribute__((format(printf, 1, 2)));
int fail_hip(hipError_t e, const char *what);
int finish(int rc);
// Clears an error the HIP runtime holds for this thread from outside the library (at the
// start of every op that launches work).
void begin_op();
int alloc_device(void **p, size_t bytes, hipStream_t st, int *dev_out = nullptr);
// hipMalloc, tried once more after the library's kept buffers are given back; the runtime's
// record of a failure is cleared.
hipError_t malloc_plain(void **p, size_t bytes);
// Scratch for the work that one call enqueues on `st`, kept until the object goes: the
// stream's grow-only workspace, which no other call gets meanwhile, or while the stream is
// being captured and that is too small, a transient allocation released (stream-ordered)
// after the call's kernels.  At most one per call: the workspace's lock is not recursive.
class Scratch {
 public:
  Scratch() = default;
  Scratch(const Scratch &) = delete;
  Scratch &operator=(const Scratch &) = delete;
  ~Scratch();
  int take(hipStream_t st, size_t bytes);             // non-zero, with the error latched, if there is none
  hipError_t try_take(hipStream_t st, size_t bytes);  // the same without latching
  void *get() const { return ptr_; }                  // null before a successful take

 private:
  void *ptr_ = nullptr;
  bool transient_ = false;
  hipStream_t st_ = nullptr;
  std::unique_lock<std::mutex> lk_;
};
Arr *new_arr(const int *shape, int dim, qmm_dtype dtype);
int alloc_arr(qmm_array *res, const std::vector<int> &shape, qmm_dtype dtype, hipStream_t st, Arr **out);
void release_arr(Arr *a);
// Frees the handle's tile-major scale copy, if it has one (waits for the device first).
void release_tiled(Arr *a);
hipStream_t stream_of(qmm_stream s);

}  // namespace qmm
