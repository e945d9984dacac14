// Graph capture of raycast launches (launch_job_table of
// imagevis3d_amd/csrc/renderer.cpp) on the host, with stand-ins for the HIP
// calls and kernels: one captured graph serves every launch of a kernel
// variant, whatever its jobs' TFs.  Built by tests/test_transfer_host.py; of
// renderer.cpp only what this calls is linked.  TEST INFRASTRUCTURE ONLY.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <vector>

#include "../../imagevis3d_amd/csrc/errors.hpp"
#include "../../imagevis3d_amd/csrc/renderer.hpp"

#define CHECK(c)                                                            \
  do {                                                                      \
    if (!(c)) {                                                             \
      fprintf(stderr, "%s:%d: check failed: %s\n", __FILE__, __LINE__, #c); \
      exit(1);                                                              \
    }                                                                       \
  } while (0)

static int g_graphs = 0;  // instantiated
static tvk::LaunchInfo g_li;

extern "C" {
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = (hipEvent_t)malloc(1);
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = (hipGraph_t)1;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  ++g_graphs;
  *x = (hipGraphExec_t)1;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
}

namespace tvk {
void set_last_error(const std::string&) {}
hipError_t launch_fill_u64(unsigned long long* p, int64_t n, unsigned long long v, hipStream_t) {
  for (int64_t i = 0; i < n; ++i) p[i] = v;
  return hipSuccess;
}
hipError_t launch_background(const JobTable*, hipStream_t) { return hipSuccess; }
hipError_t launch_raycast(const LaunchInfo& li, const JobTable*, hipStream_t) {
  g_li = li;
  return hipSuccess;
}
}  // namespace tvk

using namespace tvk;

// n jobs of one camera: two_d with a 2D TF each, else lit with a 1D TF of
// `entries` entries each
static std::vector<RaycastParams> jobs_of(int n, bool two_d, int entries) {
  static float tfs[64][4];
  static uint32_t masks[64][4];
  std::vector<RaycastParams> jobs((size_t)n);
  for (int k = 0; k < n; ++k) {
    RaycastParams& p = jobs[k];
    memset(&p, 0, sizeof p);
    p.mode = two_d ? 1 : 0;
    p.lighting = 1;
    p.tf = tfs[k];
    p.n_tf = two_d ? 256 : entries;
    p.tf2d_w = two_d ? 256 : 0;
    p.tf2d_h = two_d ? 256 : 0;
    p.tf2d_mask = two_d ? masks[k] : nullptr;
    p.rect_w = p.rect_h = p.tiles_x = p.tiles_y = 4;
    p.width = 100 + k;  // differ: no groups
  }
  return jobs;
}

static int launch(LaunchSlot& sl, const LaunchInfo& li, const std::vector<RaycastParams>& jobs) {
  const int before = g_graphs;
  CHECK(launch_job_table(sl, jobs.data(), (int)jobs.size(), li, 4, 0, nullptr, true) == TVK_OK);
  return g_graphs - before;
}

int main() {
  for (int batch : {8, 4, 2, 1}) {  // 2D TFs: two, then four, one, ten per launch
    LaunchSlot sl;
    CHECK(sl.alloc() == TVK_OK);
    LaunchInfo li;
    li.mode = 1;
    li.batch = batch;
    li.group = 1;
    CHECK(launch(sl, li, jobs_of(2, true, 0)) == 1);
    for (int n : {4, 2, 1, 10, 2, 4}) CHECK(launch(sl, li, jobs_of(n, true, 0)) == 0);
    sl.release();
    printf("OK 2D TFs, batch %d\n", batch);
  }
  {  // lit 1D TFs of any length, alone and several
    LaunchSlot sl;
    CHECK(sl.alloc() == TVK_OK);
    LaunchInfo li;
    li.lighting = 1;
    li.batch = 8;
    li.group = 1;
    li.n_tf_lds = 256;
    CHECK(launch(sl, li, jobs_of(1, false, 256)) == 1);
    for (int n : {4096, 300, 256, 1}) {
      li.n_tf_lds = n;
      CHECK(launch(sl, li, jobs_of(1, false, n)) == 0);
    }
    li.n_tf_lds = 0;
    CHECK(launch(sl, li, jobs_of(3, false, 700)) == 0);
    sl.release();
    printf("OK lit 1D TFs\n");
  }
  {  // another kernel variant has a graph of its own
    LaunchSlot sl;
    CHECK(sl.alloc() == TVK_OK);
    LaunchInfo li;
    li.lighting = 1;
    li.batch = 2;
    li.n_tf_lds = 256;
    CHECK(launch(sl, li, jobs_of(1, false, 256)) == 1 && g_li.n_tf_lds == 256);
    li.n_tf_lds = 300;
    CHECK(launch(sl, li, jobs_of(1, false, 300)) == 1 && g_li.n_tf_lds == 300);
    li.batch = 4;
    CHECK(launch(sl, li, jobs_of(1, false, 300)) == 1 && g_li.n_tf_lds == 0);
    li.lighting = 0;
    CHECK(launch(sl, li, jobs_of(1, false, 300)) == 1 && g_li.n_tf_lds == 300);
    sl.release();
    printf("OK variants\n");
  }
  printf("ALL OK\n");
  return 0;
}
