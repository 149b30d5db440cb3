// The batch driver's host side without a GPU: this program's own definitions of the
// HIP calls stand before the runtime's, launches do nothing and one allocation can be
// refused.  A refused tile must leave the batch at the tile it had.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "euler2d_hip.h"

static int refuse = 0;  // the next hipMalloc fails
static unsigned launched = 0;

struct Dim3 {
  unsigned x, y, z;
};

extern "C" {
int hipMalloc(void **p, size_t n) {
  if (refuse) {
    refuse = 0;
    *p = nullptr;
    return 2;  // hipErrorOutOfMemory
  }
  *p = std::calloc(1, n ? n : 1);
  return *p ? 0 : 2;
}
int hipFree(void *p) {
  std::free(p);
  return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::calloc(1, n);
  return 0;
}
int hipHostFree(void *p) { return hipFree(p); }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) {
  std::memcpy(d, s, n);
  return 0;
}
int hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int, void *) {
  for (size_t k = 0; k < h; ++k)
    std::memcpy(static_cast<char *>(d) + k * dp, static_cast<const char *>(s) + k * sp, w);
  return 0;
}
int hipMemsetAsync(void *d, int v, size_t n, void *) {
  std::memset(d, v, n);
  return 0;
}
int __hipPushCallConfiguration(Dim3 grid, Dim3, size_t, void *) {
  launched = grid.x;
  return 0;
}
int __hipPopCallConfiguration(Dim3 *, Dim3 *, size_t *, void **) { return 0; }
int hipLaunchKernel(const void *, Dim3, Dim3, void **, size_t, void *) { return 0; }
int hipGetDeviceCount(int *n) {
  *n = 1;
  return 0;
}
int hipGetDevice(int *d) {
  *d = 0;
  return 0;
}
int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int *v, int, int) {
  *v = 256;
  return 0;
}
int hipStreamCreateWithFlags(void **s, unsigned) {
  *s = std::malloc(1);
  return 0;
}
int hipStreamDestroy(void *s) { return hipFree(s); }
int hipStreamSynchronize(void *) { return 0; }
int hipEventCreate(void **e) { return hipStreamCreateWithFlags(e, 0); }
int hipEventCreateWithFlags(void **e, unsigned) { return hipStreamCreateWithFlags(e, 0); }
int hipEventDestroy(void *e) { return hipFree(e); }
int hipEventRecord(void *, void *) { return 0; }
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *) {
  *ms = 1.0f;
  return 0;
}
int hipGetLastError() { return 0; }
}

static int waves(e2d_batch *b) {
  long long cells = 0;
  int w = 0, n = 0;
  return e2d_batch_info(b, &cells, &w, &n) ? -1 : w;
}

static unsigned step_blocks(e2d_batch *b) {
  double ms = 0.0;
  int left = 0;
  launched = 0;
  const int rc = e2d_batch_run(b, 1, 0, &ms, &left);
  if (rc) std::printf("run: %s\n", e2d_last_error());
  return rc ? 0u : launched;
}

#define CHECK(c)                                       \
  do {                                                 \
    if (!(c)) {                                        \
      std::printf("line %d: " #c "\n", __LINE__);      \
      return 1;                                        \
    }                                                  \
  } while (0)

int main(int, char **argv) {
  e2d_params p[12];
  int parse = 0;
  CHECK(e2d_params_from_ini(argv[1], &p[0], &parse) == E2D_OK);
  for (e2d_params &q : p) q = p[0];
  e2d_batch *b = nullptr;
  CHECK(e2d_batch_create(p, 2, E2D_PRECISION_FP64, &b) == E2D_OK);
  CHECK(e2d_batch_set_launch(b, E2D_BATCH_LAUNCH_STEPS, 0) == E2D_OK);
  CHECK(e2d_batch_init(b) == E2D_OK);
  CHECK(e2d_batch_set_tile(b, 256) == E2D_OK);  // fewer items: the table keeps its size
  const int w = waves(b);
  const unsigned blocks = step_blocks(b);
  CHECK(w > 0 && blocks > 0);

  refuse = 1;
  CHECK(e2d_batch_set_tile(b, 1) == E2D_ERR_ALLOC && refuse == 0);
  CHECK(waves(b) == w);
  CHECK(step_blocks(b) == blocks);
  CHECK(e2d_batch_set_tile(b, 1) == E2D_OK && waves(b) > w && step_blocks(b) > blocks);
  e2d_batch_destroy(b);

  // the tile that follows the launch mode: neither changes.  Twelve grids on the one
  // queue seen here start in the persistent launch, whose tile is the longer one.
  CHECK(e2d_batch_create(p, 12, E2D_PRECISION_FP64, &b) == E2D_OK);
  const int before = waves(b);
  int mode = -1;
  refuse = 1;
  CHECK(e2d_batch_set_launch(b, E2D_BATCH_LAUNCH_STEPS, 0) == E2D_ERR_ALLOC);
  CHECK(e2d_batch_get_launch(b, &mode) == E2D_OK && mode == E2D_BATCH_LAUNCH_PERSISTENT);
  CHECK(waves(b) == before);
  CHECK(e2d_batch_set_launch(b, E2D_BATCH_LAUNCH_STEPS, 0) == E2D_OK && waves(b) > before);
  e2d_batch_destroy(b);
  std::printf("refused tiles change nothing\n");
  return 0;
}
