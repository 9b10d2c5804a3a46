// Error paths of the library's host code on the runtime of host_hip.h; prints
// what does not hold and returns how many.  Usage: error_paths NAME
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <new>
#include <vector>

#include "../../include/heatsim2_amd.h"
#include "host_hip.h"

namespace {
int bad = 0;
void check(bool ok, const char *what, long at) {
  if (ok) return;
  std::printf("%s (failure %ld)\n", what, at);
  bad++;
}

// Aligned arrays that stand for a caller's device arrays
struct Field {
  std::vector<double> v;
  explicit Field(size_t n) : v(n + 2, 1.0) {}
  double *p() { return reinterpret_cast<double *>(((uintptr_t)v.data() + 15) & ~(uintptr_t)15); }
};


struct Plan {
  hs2_plan *p = nullptr;
  std::vector<uint8_t> map;
  Plan(int nz, int ny, int nx) : map((size_t)(nz + 1) * (ny + 1) * (nx + 1), 0) {
    const hs2_grid_desc g{nz, ny, nx, 1e-3, 1e-3, 1e-3, 1e-2};
    if (hs2_plan_create(&g, &p) != HS2_OK) std::printf("hs2_plan_create failed\n");
  }
  ~Plan() { hs2_plan_destroy(p); }
  int set_compact() {
    const double gtab[3] = {0.1, 0.1, 0.1}, mtab[1] = {1.0};
    const uint8_t compute[1] = {1};
    try {
      return hs2_plan_set_compact(p, map.data(), map.data(), map.data(), map.data(), 1, 1, gtab,
                                  mtab, compute);
    } catch (const std::bad_alloc &) {
      return -1;
    }
  }
  int tables() const {
    int a = 0;
    (void)hs2_plan_get_option(p, HS2_OPT_LINE_TABLES, &a);
    return a;
  }
  int step(double *T) {
    return hs2_step(p, T, T, nullptr, nullptr, 0, nullptr, nullptr, nullptr);
  }
};

// What a plan holds is freed whichever allocation of hs2_plan_set_compact
// fails; `arm` makes the n-th fail
void set_compact_frees(void (*arm)(long)) {
  const size_t base = host_hip::live();
  for (long n = 0;; n++) {
    host_hip::clear_error();
    Plan *P = new Plan(8, 6, 40);
    Field T(8 * 6 * 40);
    arm(n);
    const int rc = P->set_compact();
    const bool end = !host_hip::all_used();
    arm(-1);
    if (rc == HS2_OK) check(P->step(T.p()) == HS2_OK, "a plan that was set does not step", n);
    else check(!end, "refused without a failure", n);
    delete P;
    check(host_hip::live() == base, "device memory is not freed", n);
    if (end) return;
  }
}

// Shapes and options are taken whatever memory is left, as before line tables:
// only an optional plane of the x sweep is made then
void set_config_takes(void (*arm)(long)) {
  for (int option = 0; option < 2; option++)
    for (long n = 0;; n++) {
      host_hip::clear_error();
      Plan P(8, 6, 40);
      Field T(8 * 6 * 40);
      check(P.set_compact() == HS2_OK && P.tables() == 7, "no line tables", n);
      const size_t base = host_hip::live();
      int info[14], rc;
      (void)hs2_plan_info(P.p, info);
      arm(n);
      try {
        rc = option ? hs2_plan_set_option(P.p, HS2_OPT_LINE_TABLES, 0)
                    : hs2_plan_set_config(P.p, info[4], info[5], info[10], info[11], info[6],
                                          info[7], info[8], info[9]);
      } catch (const std::bad_alloc &) {
        rc = -1;
      }
      const bool end = !host_hip::all_used();
      arm(-1);
      check(rc == HS2_OK, option ? "hs2_plan_set_option" : "hs2_plan_set_config", n);
      check(P.tables() == 0, "line tables are still on", n);
      check(P.step(T.p()) == HS2_OK, "the plan does not step", n);
      check(end || host_hip::live() == base, "device memory is left from a failed plane", n);
      if (end) break;
    }
}

// Whichever launch of a batch call fails: when it has returned, what its own
// streams still do is behind the caller's stream
void batch_lanes(int graph) {
  const int ninst = 4, K = 4;
  hs2_batch_inst in[ninst];
  for (int i = 0; i < ninst; i++) in[i] = {8 + i, 9, 10, 6 + 5 * i, 0, 1e-3};
  hs2_batch *b = nullptr;
  check(hs2_batch_create(in, ninst, K, &b) == HS2_OK, "hs2_batch_create", 0);
  (void)hs2_batch_set_options(b, graph, 3);
  int64_t sizes[5];
  (void)hs2_batch_layout(b, nullptr, nullptr, sizes);
  const size_t N = (size_t)sizes[0], H = (size_t)sizes[1], W = (size_t)sizes[2];
  Field M(N), gz(N), gy(N), gx(N), T(N), src(N), hist(H), work(W), o[5] = {Field(N), Field(N), Field(N), Field(N), Field(N)};
  std::vector<uint8_t> wbuf(N + 16, 1);
  const uint8_t *w = reinterpret_cast<uint8_t *>(((uintptr_t)wbuf.data() + 15) & ~(uintptr_t)15);
  (void)hs2_batch_set_dense(b, M.p(), w, gz.p(), gy.p(), gx.p());
  int own;
  void *stream = &own;  // any address names a stream of the caller's
  for (int back = 0; back < 2; back++)
    for (long n = 0;; n++) {
      host_hip::clear_error();
      host_hip::fail_launch(n);
      const int rc =
          back ? hs2_batch_backward(b, src.p(), hist.p(), o[0].p(), o[1].p(), o[2].p(), o[3].p(),
                                    o[4].p(), work.p(), W, stream)
               : hs2_batch_forward(b, T.p(), src.p(), hist.p(), work.p(), W, stream);
      const bool end = !host_hip::all_used();
      host_hip::fail_launch(-1);
      check(end ? rc == HS2_OK : rc == HS2_E_HIP, "return value", n);
      check(host_hip::outstanding(stream) == 0,
            back ? "work of hs2_batch_backward is left behind" : "work of hs2_batch_forward is left behind", n);
      if (end) break;
    }
  hs2_batch_destroy(b);
}

// the same for the gradient of a single plan and its second stream
void backward_lanes() {
  const int nz = 8, ny = 9, nx = 10, n = nz * ny * nx, steps = 11, K = 4;
  Plan P(nz, ny, nx);
  Field M(n), gz(n), gy(n), gx(n), ckpt(3 * n), hist(steps * ny * nx), o[5] = {Field(n), Field(n), Field(n), Field(n), Field(n)};
  std::vector<uint8_t> wbuf(n + 16, 1);
  const uint8_t *w = reinterpret_cast<uint8_t *>(((uintptr_t)wbuf.data() + 15) & ~(uintptr_t)15);
  check(hs2_plan_set_dense(P.p, M.p(), w, gz.p(), gy.p(), gx.p()) == HS2_OK, "set_dense", 0);
  const size_t W = hs2_grad_work_best(P.p, steps, K);
  Field work(W);
  int own;
  for (long f = 0;; f++) {
    host_hip::clear_error();
    host_hip::fail_launch(f);
    const int rc = hs2_grad_backward(P.p, steps, K, ckpt.p(), nullptr, nullptr, 0, hist.p(),
                                     o[0].p(), o[1].p(), o[2].p(), o[3].p(), nullptr, o[4].p(),
                                     work.p(), W, &own);
    const bool end = !host_hip::all_used();
    host_hip::fail_launch(-1);
    check(end ? rc == HS2_OK : rc == HS2_E_HIP, "return value", f);
    check(host_hip::outstanding(&own) == 0, "work of hs2_grad_backward is left behind", f);
    if (end) break;
  }
}
}  // namespace

int main(int argc, char **argv) {
  const char *name = argc > 1 ? argv[1] : "";
  if (!std::strcmp(name, "set_compact_host_memory")) set_compact_frees(host_hip::fail_new);
  else if (!std::strcmp(name, "set_compact_device_memory")) set_compact_frees(host_hip::fail_malloc);
  else if (!std::strcmp(name, "set_config_host_memory")) set_config_takes(host_hip::fail_new);
  else if (!std::strcmp(name, "set_config_device_memory")) set_config_takes(host_hip::fail_malloc);
  else if (!std::strcmp(name, "batch_lanes")) batch_lanes(0);
  else if (!std::strcmp(name, "batch_lanes_graphs")) batch_lanes(1);
  else if (!std::strcmp(name, "backward_lanes")) backward_lanes();
  else return 99;
  return bad > 100 ? 100 : bad;
}
