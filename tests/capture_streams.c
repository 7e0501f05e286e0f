/* The order of a pass's launches (csrc/host/plan.c) with the device calls
 * replaced by recorders: prints how many calls name the plan's second stream,
 * of a pass on a plain stream and of one on a stream under capture.
 * Arguments: depth, 1 for the transposed pass. */
#include "../fmbem_gpu_c_amd/csrc/host/plan.c"

static char caller, second;
static int captured, on_second;
static int seen(void *s) {
  on_second += s == &second;
  return FMB_OK;
}

int fmbh_stream_capturing(void *s) { return captured && s == &caller; }
int fmbh_event_record(void *e, void *s) { return seen(s); }
int fmbh_stream_wait(void *s, void *e) { return seen(s); }
int fmbh_begin(const fmb_plan *p, int op, int what, const fmb_c64 *x, int n, void *s) {
  return seen(s);
}
int fmbh_l2p_near(const fmb_plan *p, int op, fmb_c64 *y, int n, int parts, void *s) {
  return seen(s);
}
int fmbh_near_t(const fmb_plan *p, int op, const void *a, const void *b, fmb_c64 *y, int n,
                int parts, void *s) {
  return seen(s);
}
int fmbx_rcr_run(const fmb_plan *p, int op, int kind, int l, int n, void *s) { return seen(s); }
int fmbx_rcr_run_t(const fmb_plan *p, int op, int kind, int l, int n, void *s) { return seen(s); }
int fmbx_m2l_levels(const fmb_plan *p, int op, int trans, int n, int *from, void *s) {
  return seen(s);
}

int main(int argc, char **argv) {
  static fmb_tree t;
  static fmb_plan pl;
  fmb_c64 v = {0, 0};
  t.lmax = argc > 1 ? atoi(argv[1]) : 4;
  pl.tree = &t;
  pl.ready = pl.nrhs_max = 1;
  pl.aux = &second;
  for (captured = 0; captured < 2; captured++) {
    on_second = 0;
    int rc = argc > 2 && atoi(argv[2])
                 ? fmb_matvec_transpose(&pl, FMB_FP64, 3, &v, &v, 1, &caller)
                 : fmb_matvec(&pl, FMB_FP64, &v, &v, 1, &caller);
    printf("%d ", rc ? -1 : on_second);
  }
  return 0;
}
