/* rcr.c -- host planning and dispatch of the rotate-coaxial-rotate
 * translations on the matrix cores (csrc/hip/rcr_kernels.h, rcr_mfma.hip).
 *
 * Every translation kind groups its box pairs into buckets that share one
 * operator:
 *   M2L at level l: the 316 interaction-list offsets (srTransOriginArr /
 *     srTransDestArr, translation.cu:2847-2927), pairs already bucketed by
 *     the tree build;
 *   M2M l -> l-1 and L2L l-1 -> l: the child's octant (the 8 directions of
 *     genSSIdxArrs / genRRIdxArrs, translation.cu:2797-2846, 2928-2969),
 *     one (parent, child) list per level serving both.
 * Buckets are cut into chunks of at most RCR_CHUNK pairs.  The blocks of one
 * translation are split into units (whole blocks when the batch sits in LDS
 * and is updated in place; row groups otherwise) and assigned to the
 * workgroup's waves by longest-processing-time first.
 *
 * The FP32 / FP64 rotation blocks run in even/odd coordinates
 * (csrc/hip/rcr_mfma.hip): degree n's (2n+1)^2 block becomes an even block
 * of n + 1 rows and an odd block of n rows, about half the products, in one
 * unit per degree.  The split-BF16 rotations keep the standard blocks. */
#include <math.h>
#include <pthread.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/file.h>
#include <sys/stat.h>

#include "../fmb_internal.h"
#include "../hip/fmb_hip.h"
#include "host.h"

#define RCR_CHUNK 16
#define RCR_WAVES_MAX 8
#define RCR_GWS_GRID 512

typedef struct {
  int beta, dist;
  double phi;
} rcr_info_t; /* layout of the device OffInfo */

typedef struct {
  int code, cost, aoff; /* aoff: offset of the unit's padded operator block */
  int w;                /* wave the schedule gives it */
} unit_t;

static int by_cost(const void *a, const void *b) {
  const unit_t *x = (const unit_t *)a, *y = (const unit_t *)b;
  if (x->cost != y->cost) return y->cost - x->cost;
  return x->code - y->code;
}

/* units in non-increasing cost order, each to the least-loaded of nw
 * waves; writes the waves' lists back to back as {code, aoff} pairs into
 * out (entry q at out[2q]) and their start entries (nw + 1 values,
 * beginning at base) into off */
static void lpt(unit_t *u, int n, int nw, int base, int *off, int *out) {
  int load[RCR_WAVES_MAX] = {0}, cnt[RCR_WAVES_MAX] = {0};
  qsort(u, n, sizeof(unit_t), by_cost);
  for (int i = 0; i < n; i++) {
    int w = 0;
    for (int q = 1; q < nw; q++)
      if (load[q] < load[w]) w = q;
    load[w] += u[i].cost;
    u[i].w = w;
    cnt[w]++;
  }
  off[0] = base;
  for (int w = 0; w < nw; w++) off[w + 1] = off[w] + cnt[w];
  int fill[RCR_WAVES_MAX];
  for (int w = 0; w < nw; w++) fill[w] = off[w];
  for (int i = 0; i < n; i++) {
    int q = fill[u[i].w]++;
    out[2 * q] = u[i].code;
    out[2 * q + 1] = u[i].aoff;
  }
}

static int tiles(int s) { return (s + 15) / 16; }
static int ksteps(int s) { return (s + 3) / 4; }
static int group_tiles(int nt, int g, int mt, int split) {
  if (!split) return nt;
  return nt - g * mt < mt ? nt - g * mt : mt;
}

/* padded block sizes: rows to a multiple of 16, columns to a multiple of 4 */
static int pad_rows(int s) { return 16 * tiles(s); }
static int pad_cols(int s) { return 4 * ksteps(s); }

/* values of one padded even/odd rotation block of s rows (0 for s = 0) */
static int rot_block(int s) { return s ? pad_rows(s) * pad_cols(s) : 0; }

/* offsets of the padded rotation blocks of degrees n < np (np + 1 values):
 * degree n's even block (n + 1 rows), then its odd block (n rows) */
static void rot_offsets(int np, int *hoff) {
  hoff[0] = 0;
  for (int n = 0; n < np; n++) hoff[n + 1] = hoff[n] + rot_block(n + 1) + rot_block(n);
}

/* offsets of the split-BF16 (standard) rotation blocks n < np (np + 1
 * values): rows padded to 16, K to 32 */
static void rot_offsets_bf(int np, int *hb) {
  hb[0] = 0;
  for (int n = 0; n < np; n++) hb[n + 1] = hb[n] + pad_rows(2 * n + 1) * (((2 * n + 1) + 31) & ~31);
}

/* whether opset op may run mode's rotations in split-BF16 */
static int use_bf(const fmb_plan *pl, int op, int mode) {
  return pl->prm.split_bf16 && pl->ops[op].prec != FMB_FP64 &&
         (mode == FMBH_RCR_LDS || mode == FMBH_RCR_LDSP);  /* not LDSO */
}

/* offsets of the padded coaxial blocks |m| < min(pin, pout) (+1 values) */
static void coax_offsets(int pin, int pout, int *coff) {
  int mn = pin < pout ? pin : pout;
  coff[0] = 0;
  for (int am = 0; am < mn; am++)
    coff[am + 1] = coff[am] + pad_rows(pout - am) * pad_cols(pin - am);
}

/* rotation blocks of degrees n < np: code n*16 + g.  FP32 / FP64: degree
 * n's even (n + 1 rows) and odd (n rows) blocks together; split-BF16: the
 * standard block (2n + 1 rows). */
static int rot_units(int np, int split, int mt, const int *hoff, int bf, unit_t *u) {
  int k = 0;
  for (int n = 0; n < np; n++) {
    int s = bf ? 2 * n + 1 : n + 1, nt = tiles(s), ng = split ? (nt + mt - 1) / mt : 1;
    for (int g = 0; g < ng; g++) {
      u[k].code = n * 16 + g;
      u[k].cost = group_tiles(nt, g, mt, split) * ksteps(s);
      if (!bf) {
        /* the odd block's tiles in this row group */
        int to = split ? tiles(n) - g * mt : tiles(n);
        to = to < 0 ? 0 : (split && to > mt ? mt : to);
        u[k].cost += to * ksteps(n);
      }
      u[k].aoff = hoff[n];
      k++;
    }
  }
  return k;
}

/* coaxial blocks +-am, am < min(pin, pout), processed together (they share
 * the matrix C^{am}): code am*16 + g */
static int coax_units(int pin, int pout, int split, int mt, const int *coff,
                      unit_t *u) {
  int k = 0, mn = pin < pout ? pin : pout;
  for (int am = 0; am < mn; am++) {
    int so = pout - am, si = pin - am, sg = am ? 2 : 1;
    int nt = tiles(so), ng = split ? (nt + mt - 1) / mt : 1;
    for (int g = 0; g < ng; g++) {
      u[k].code = am * 16 + g;
      u[k].cost = 2 * sg * group_tiles(nt, g, mt, split) * ksteps(si);
      u[k].aoff = coff[am];
      k++;
    }
  }
  return k;
}

/* Schedule of one translation shape for nw waves: a header of three offset
 * tables (forward rotation, coaxial, back rotation), nw + 1 entry indices
 * each, giving every wave's units as entries [off[w], off[w+1]); entry q is
 * the int pair {code, operator offset} at [2q, 2q + 1] of the same array.
 * The header is 3 (nw + 1) ints rounded up to even. */
static int build_sched(int pin, int pout, int P, int mode, int mt, int nw, const int *hoff,
                       int bf, const int *coff, int **d_out, int *len, void *stream) {
  int split = mode == FMBH_RCR_GWS, rc;
  if (nw < 1 || nw > RCR_WAVES_MAX)
    return fmb_set_error(FMB_ERR_RANGE, "translation schedule for %d waves", nw);
  const int hdr = (3 * (nw + 1) + 1) & ~1;
  unit_t *u = (unit_t *)malloc(sizeof(unit_t) * 16 * (pin + P + pout));
  if (!u) return fmb_set_error(FMB_ERR_NOMEM, "translation schedule");
  int n1 = rot_units(pin, split, mt, hoff, bf, u);
  int nc = coax_units(pin, pout, split, mt, coff, u + n1);
  int n3 = rot_units(pout, split, mt, hoff, bf, u + n1 + nc);
  int tot = hdr + 2 * (n1 + nc + n3);
  int *h = (int *)calloc(tot, sizeof(int));
  if (!h) {
    free(u);
    return fmb_set_error(FMB_ERR_NOMEM, "translation schedule");
  }
  int base = hdr / 2;
  lpt(u, n1, nw, base, h, h);
  base += n1;
  lpt(u + n1, nc, nw, base, h + nw + 1, h);
  base += nc;
  lpt(u + n1 + nc, n3, nw, base, h + 2 * (nw + 1), h);
  *len = tot;
  rc = fmbh_malloc((void **)d_out, sizeof(int) * tot);
  if (!rc) rc = fmbh_h2d(*d_out, h, sizeof(int) * tot, stream);
  free(u);
  free(h);
  return rc;
}

/* chunks of <= RCR_CHUNK pairs inside each bucket [start[b], start[b+1]) */
static int build_chunks(const int *start, int nbucket, fmb_rcr_tab *tb,
                        void *stream) {
  int npairs = start[nbucket] - start[0], n = 0, rc;
  int *c = (int *)malloc(sizeof(int) * 4 * (npairs / RCR_CHUNK + nbucket + 1));
  if (!c) return fmb_set_error(FMB_ERR_NOMEM, "translation chunks");
  for (int b = 0; b < nbucket; b++)
    for (int s = start[b]; s < start[b + 1]; s += RCR_CHUNK) {
      int e = s + RCR_CHUNK < start[b + 1] ? s + RCR_CHUNK : start[b + 1];
      c[4 * n] = b;
      c[4 * n + 1] = s;
      c[4 * n + 2] = e;
      c[4 * n + 3] = 0;
      n++;
    }
  tb->nchunks = n;
  rc = fmbh_malloc(&tb->d_chunks, sizeof(int) * 4 * (n > 0 ? n : 1));
  if (!rc && n) rc = fmbh_h2d(tb->d_chunks, c, sizeof(int) * 4 * n, stream);
  free(c);
  return rc;
}

/* M2L chunks in tile-major order: pairs of target boxes [tile * T, (tile+1)
 * * T) for every offset, then the next tile; within a (tile, offset) group
 * chunks of at most RCR_CHUNK pairs.  start: the offset buckets of the
 * tree's offset-major pair list, whose targets are in box order inside each
 * bucket. */
static int build_chunks_tiled(const fmb_tree *t, int l, int T, fmb_rcr_tab *tb, void *stream) {
  const int *start = t->h_off_start[l];
  int np = start[FMB_NOFF] - start[0], nbox = t->nbox[l], rc;
  int ntile = (nbox + T - 1) / T;
  int *tg = (int *)malloc(sizeof(int) * (np > 0 ? np : 1));
  /* per (tile, bucket): chunks counted, then placed */
  int *cnt = (int *)calloc((size_t)ntile * FMB_NOFF + 1, sizeof(int));
  int *c = (int *)malloc(sizeof(int) * 4 * (np / RCR_CHUNK + (size_t)ntile * FMB_NOFF + 1));
  if (!tg || !cnt || !c) {
    free(tg);
    free(cnt);
    free(c);
    return fmb_set_error(FMB_ERR_NOMEM, "translation chunks");
  }
  rc = fmbh_d2h(tg, t->d_pair_tgt[l], sizeof(int) * np, stream);
  int n = 0;
  if (!rc) {
    /* group boundaries inside each bucket: runs of one tile */
    for (int b = 0; b < FMB_NOFF; b++)
      for (int s0 = start[b]; s0 < start[b + 1];) {
        int tile = tg[s0] / T, e = s0;
        while (e < start[b + 1] && tg[e] / T == tile) e++;
        cnt[(size_t)tile * FMB_NOFF + b + 1] += (e - s0 + RCR_CHUNK - 1) / RCR_CHUNK;
        s0 = e;
      }
    for (size_t i = 1; i <= (size_t)ntile * FMB_NOFF; i++) cnt[i] += cnt[i - 1];
    for (int b = 0; b < FMB_NOFF; b++)
      for (int s0 = start[b]; s0 < start[b + 1];) {
        int tile = tg[s0] / T, e = s0;
        while (e < start[b + 1] && tg[e] / T == tile) e++;
        int q = cnt[(size_t)tile * FMB_NOFF + b];
        for (int f = s0; f < e; f += RCR_CHUNK, q++) {
          c[4 * q] = b;
          c[4 * q + 1] = f;
          c[4 * q + 2] = f + RCR_CHUNK < e ? f + RCR_CHUNK : e;
          c[4 * q + 3] = 0;
        }
        cnt[(size_t)tile * FMB_NOFF + b] = q;
        s0 = e;
      }
    n = cnt[(size_t)ntile * FMB_NOFF];
  }
  tb->nchunks = n;
  if (!rc) rc = fmbh_malloc(&tb->d_chunks, sizeof(int) * 4 * (n > 0 ? n : 1));
  if (!rc && n) rc = fmbh_h2d(tb->d_chunks, c, sizeof(int) * 4 * n, stream);
  free(tg);
  free(cnt);
  free(c);
  return rc;
}

/* (parent, child) pairs of level l bucketed by the child's octant */
static int octant_pairs(const fmb_tree *t, int l, fmb_rcr_tab *tb, void *stream) {
  int nb = t->nbox[l], rc;
  int *key = (int *)malloc(sizeof(int) * nb), *par = (int *)malloc(sizeof(int) * nb);
  int *sp = (int *)malloc(sizeof(int) * nb), *sc = (int *)malloc(sizeof(int) * nb);
  int start[9] = {0};
  rc = (key && par && sp && sc) ? FMB_OK : fmb_set_error(FMB_ERR_NOMEM, "octant pairs");
  if (!rc) rc = fmbh_d2h(key, t->d_keys[l], sizeof(int) * nb, stream);
  if (!rc) rc = fmbh_d2h(par, t->d_parent[l], sizeof(int) * nb, stream);
  if (!rc) {
    for (int i = 0; i < nb; i++) start[(key[i] & 7) + 1]++;
    for (int o = 0; o < 8; o++) start[o + 1] += start[o];
    int fill[8];
    memcpy(fill, start, sizeof(fill));
    for (int i = 0; i < nb; i++) {
      int o = key[i] & 7, q = fill[o]++;
      sp[q] = par[i];
      sc[q] = i;
    }
    rc = fmbh_malloc((void **)&tb->d_par, sizeof(int) * nb);
  }
  if (!rc) rc = fmbh_malloc((void **)&tb->d_chi, sizeof(int) * nb);
  if (!rc) rc = fmbh_h2d(tb->d_par, sp, sizeof(int) * nb, stream);
  if (!rc) rc = fmbh_h2d(tb->d_chi, sc, sizeof(int) * nb, stream);
  if (!rc) rc = build_chunks(start, 8, tb, stream);
  free(key);
  free(par);
  free(sp);
  free(sc);
  return rc;
}

/* The form with 8 waves beside a shape of the fixed rule (4 waves), for the
 * launches that leave a CU with too few waves to cover the operators' loads.
 * That is, first, every launch of an order whose batches leave room for one
 * workgroup (FP64) or two (FP32) on a CU's LDS: M2L of 327,680 triangles, FP32
 * with nine right-hand sides, 4 -> 8 waves: order 23 39.7 -> 31.7 ms, 31 24.8
 * -> 18.3, 42 19.6 -> 13.4, but 18 62.1 -> 65.1; FP64 with one: 31 5.5 -> 4.8,
 * but 23 8.1 -> 10.5 (an FP64 product occupies its matrix core twice as
 * long).  In the global workspace, FP64 alone, with 8 vectors a batch and
 * blocks in one piece: order 94 3.7 -> 2.7 ms, 62 3.1 -> 2.9, 42 4.8 -> 3.9
 * (FP32 order 62 13.2 -> 13.4).  Second (job_shape), launches that leave half
 * of the 256 CUs empty, with 8 vectors a batch: FP64 M2M of 16 workgroups,
 * order 16, 21 us with 4 waves and 16 vectors, 17 with 8 waves, 13 with 8
 * vectors as well; of 64, order 23, 36 -> 33, but of 204 41 -> 42. */
static int wide_form(fmb_plan *pl, fmb_rcr_tab *tb, int op, const int *hoff, const int *coff,
                     void *stream) {
  const int prec = pl->ops[op].prec, P = tb->P, mode = tb->mode[op];
  if (pl->prm.waves || pl->prm.autotune || tb->bf[op] ||
      (mode != FMBH_RCR_LDS && mode != FMBH_RCR_GWS))
    return FMB_OK;
  int nt = tb->nt[op], mt = tb->mt[op], wide, rc;
  if (mode == FMBH_RCR_GWS) {
    if (prec != FMB_FP64 || pl->prm.rcr_mode == FMB_RCR_MODE_GWS) return FMB_OK;
    nt = 1;
    mt = fmbh_rcr_mt_lds(P, 0) ? fmbh_rcr_mt_lds(P, 0) : 6;
    wide = 1;
  } else {
    const size_t b = fmbh_rcr_lds_bytes(P, prec, nt, tb->sched_len[op]);
    wide = 160 * 1024 / b <= (prec == FMB_FP64 ? 1 : 2);
    if (!wide) nt = 1;
  }
  int *sched = NULL, slen = 0;
  if ((rc = build_sched(tb->pin, tb->pout, P, mode, mt, 8, hoff, 0, coff, &sched, &slen, stream)))
    return rc;
  if (mode == FMBH_RCR_LDS && fmbh_rcr_lds_bytes(P, prec, nt, slen) > 160 * 1024) {
    fmbh_free(sched);
    return FMB_OK;
  }
  tb->nt8[op] = nt;
  tb->mt8[op] = mt;
  tb->wide8[op] = wide;
  tb->d_sched8[op] = sched;
  tb->sched8_len[op] = slen;
  return FMB_OK;
}

/* tile shapes, schedules and padded coaxial blocks of one translation;
 * C: the scaled coaxial matrices of each opset (ncoax of them, order P) */
static int plan_tab(fmb_plan *pl, fmb_rcr_tab *tb, int pin, int pout,
                    void *const *C, int ncoax, const int *hoff, const int *hboff,
                    void *stream) {
  int rc = FMB_OK, mn = pin < pout ? pin : pout;
  tb->pin = pin;
  tb->pout = pout;
  tb->P = pin > pout ? pin : pout;
  int *coff = (int *)malloc(sizeof(int) * (mn + 1));
  int *d_coff = NULL;
  if (!coff) return fmb_set_error(FMB_ERR_NOMEM, "coaxial offsets");
  coax_offsets(pin, pout, coff);
  tb->cpad_stride = (size_t)coff[mn];
  tb->hlen = hoff[tb->P];
  for (int op = 0; op < pl->nops && !rc; op++) {
    fmb_opset *o = &pl->ops[op];
    tb->mode[op] = 0;
    if (pl->prm.rcr_path == FMB_RCR_VALU) continue;
    if ((rc = fmbh_rcr_shape(tb->P, o->prec, &tb->mode[op], &tb->nt[op], &tb->mt[op])))
      break;
    tb->nw[op] = pl->prm.waves ? pl->prm.waves : 4;
    /* a requested workspace mode: GWS always fits; LDSP wherever the rule's
     * LDS batch fits (the same LDS) */
    if (pl->prm.rcr_mode == FMB_RCR_MODE_GWS && tb->mode[op] != FMBH_RCR_GWS) {
      tb->mode[op] = FMBH_RCR_GWS;
      tb->nt[op] = 2;
      tb->mt[op] = 4;
    } else if (pl->prm.rcr_mode == FMB_RCR_MODE_LDSP && tb->mode[op] == FMBH_RCR_LDS) {
      tb->mode[op] = FMBH_RCR_LDSP;
    }
    /* operators in LDS where batch and operators fit (the schedule bound of
     * fmbh_rcr_shape) */
    if ((pl->prm.ldso || pl->prm.rcr_mode == FMB_RCR_MODE_LDSO) && tb->mode[op] != FMBH_RCR_GWS)
      for (int nt = 2; nt >= 1; nt--)
        if (fmbh_rcr_ldso_bytes(tb->P, o->prec, nt, 8 * tb->P + 16, tb->hlen,
                                tb->cpad_stride) <= 160 * 1024) {
          tb->mode[op] = FMBH_RCR_LDSO;
          tb->nt[op] = nt;
          break;
        }
    tb->bf[op] = use_bf(pl, op, tb->mode[op]);
    /* split-BF16 rotations keep the standard blocks: whole 2P - 1 rows */
    if (tb->bf[op] && fmbh_rcr_mt_lds(tb->P, 1)) tb->mt[op] = fmbh_rcr_mt_lds(tb->P, 1);
    if ((rc = build_sched(pin, pout, tb->P, tb->mode[op], tb->mt[op], tb->nw[op],
                          tb->bf[op] ? hboff : hoff, tb->bf[op], coff, &tb->d_sched[op],
                          &tb->sched_len[op], stream)))
      break;
    if ((rc = wide_form(pl, tb, op, hoff, coff, stream))) break;
    if (!d_coff) {
      if ((rc = fmbh_malloc((void **)&d_coff, sizeof(int) * (mn + 1)))) break;
      if ((rc = fmbh_h2d(d_coff, coff, sizeof(int) * (mn + 1), stream))) break;
    }
    size_t bytes = o->csz * tb->cpad_stride * ncoax;
    if ((rc = fmbh_malloc(&tb->d_Cpad[op], bytes))) break;
    pl->bytes += bytes;
    if ((rc = fmbh_pad_coax(o->prec, C[op], ncoax, tb->P, pin, pout, d_coff,
                            tb->cpad_stride, tb->d_Cpad[op], stream)))
      break;
  }
  if (!rc) rc = fmbh_sync(stream);
  fmbh_free(d_coff);
  free(coff);
  return rc;
}

/* ---- target-stationary M2L of low orders (csrc/hip/rcr_ts.hip) ---- */

/* offsets of the table blocks of one class (rotations of degrees n < p) or
 * one distance (coaxial |m| < p), in values; returns their total.  Layouts:
 * k_ts_rot and k_ts_coax. */
static int ts_blocks(int prec, int rot, int p, int *off) {
  int o = 0;
  for (int i = 0; i < p; i++) {
    const int rg = ((rot ? i + 1 : p - i) + 3) / 4; /* row groups */
    off[i] = o;
    if (prec == FMB_FP64)
      o += (rot ? 2 : 4) * rg * 64;
    else
      o += rot ? (rg + 1) / 2 * 256 : 512;
  }
  return o;
}

/* rotation tables and phases of opset o, orders up to FMBH_TS_PMAX */
static int ts_rot_setup(fmb_plan *pl, fmb_opset *o, void *stream) {
  const int P = pl->Pmax < FMBH_TS_PMAX ? pl->Pmax : FMBH_TS_PMAX;
  int hoff[FMBH_TS_PMAX], *d_hoff = NULL, *d_cb = NULL, rc;
  o->ts_P = P;
  o->ts_hstride = ts_blocks(o->prec, 1, P, hoff);
  size_t bytes = o->csz / 2 * (size_t)o->ts_hstride * FMB_NCLASS;
  if ((rc = fmbh_malloc(&o->d_ts_H, bytes))) return rc;
  pl->bytes += bytes;
  rc = fmbh_malloc((void **)&d_hoff, sizeof(int) * P);
  if (!rc) rc = fmbh_malloc((void **)&d_cb, sizeof(int) * FMB_NCLASS);
  if (!rc) rc = fmbh_h2d(d_hoff, hoff, sizeof(int) * P, stream);
  if (!rc) rc = fmbh_h2d(d_cb, pl->class_beta, sizeof(int) * FMB_NCLASS, stream);
  if (!rc)
    rc = fmbh_ts_rot(o->prec, (const double *)pl->ops[0].d_H, pl->Pmax, P, d_cb, d_hoff,
                     o->ts_hstride, o->d_ts_H, stream);
  /* row (offset, parity of n): e^{i m phi} s^(m + n), s = -1 for an offset
   * below its class's direction (dz < 0): the reflection z -> -z multiplies
   * coefficient (n, m) by (-1)^(n + m).  The transposed pass takes the pair
   * of the opposite offset backwards: that offset's angles, conjugated. */
  const size_t n = (size_t)FMB_NOFF * 2 * P;
  double *w = (double *)malloc(sizeof(double) * 2 * n);
  float *f = (float *)malloc(sizeof(float) * 2 * n);
  if (!rc && (!w || !f)) rc = fmb_set_error(FMB_ERR_NOMEM, "phase tables");
  for (int tr = 0; tr < 2 && !rc; tr++) {
    for (int off = 0; off < FMB_NOFF; off++) {
      const int dx = off / 49 - 3, dy = (off / 7) % 7 - 3, dz = off % 7 - 3;
      const double phi = pl->off_phi[tr ? fmb_off_code(-dx, -dy, -dz) : off];
      const int below = tr ? dz > 0 : dz < 0;
      for (int par = 0; par < 2; par++)
        for (int m = 0; m < P; m++) {
          const double s = below && ((m + par) & 1) ? -1.0 : 1.0;
          const size_t i = 2 * (((size_t)off * 2 + par) * P + m);
          w[i] = s * cos(m * phi);
          w[i + 1] = s * (tr ? -sin(m * phi) : sin(m * phi));
        }
    }
    for (size_t i = 0; i < 2 * n; i++) f[i] = (float)w[i];
    if ((rc = fmbh_malloc(&o->d_ts_phase[tr], o->csz * n))) break;
    pl->bytes += o->csz * n;
    rc = fmbh_h2d(o->d_ts_phase[tr], o->prec == FMB_FP64 ? (const void *)w : (const void *)f,
                  o->csz * n, stream);
  }
  free(w);
  free(f);
  if (!rc) rc = fmbh_sync(stream);
  fmbh_free(d_hoff);
  fmbh_free(d_cb);
  return rc;
}

/* schedule: {first, end} of every wave's rotation units, then of its coaxial
 * units, then the units {degree or |m|, table offset}.  Units go by
 * decreasing cost to the least-loaded SIMD (waves w, w + 4, ... share one),
 * and there to the least-loaded wave. */
static int ts_sched(int prec, int p, int **d_out, void *stream) {
  const int nw = prec == FMB_FP64 ? FMBH_TS_WAVES64 : FMBH_TS_WAVES32;
  int off[FMBH_TS_PMAX], h[4 * FMBH_TS_WAVES64 + 4 * FMBH_TS_PMAX], q = 2 * nw, rc;
  unit_t u[FMBH_TS_PMAX];
  const int c1 = prec == FMB_FP64 ? 16 : 8; /* cycles of 4 rows x 1 column */
  for (int st = 0; st < 2; st++) {
    ts_blocks(prec, !st, p, off);
    for (int i = 0; i < p; i++) {
      const int s = st ? p - i : i + 1, rg = (s + 3) / 4;
      u[i].code = i;
      u[i].aoff = off[i];
      /* cycles: the products of both rotations and the rows' loads, phases
       * and sums; the products of the coaxial block */
      u[i].cost = st ? 2 * c1 * rg * s + 20 * s + 100 : 2 * c1 * rg * s + 300 * rg + 300;
    }
    int simd[4] = {0}, load[FMBH_TS_WAVES64] = {0};
    qsort(u, p, sizeof(unit_t), by_cost);
    for (int i = 0; i < p; i++) {
      int b = 0;
      for (int k = 1; k < 4; k++)
        if (simd[k] < simd[b]) b = k;
      int w = b;
      for (int k = b; k < nw; k += 4)
        if (load[k] < load[w]) w = k;
      simd[b] += u[i].cost;
      load[w] += u[i].cost;
      u[i].w = w;
    }
    for (int w = 0; w < nw; w++) {
      h[2 * (st * nw + w)] = q;
      for (int i = 0; i < p; i++)
        if (u[i].w == w) {
          h[2 * q] = u[i].code;
          h[2 * q + 1] = u[i].aoff;
          q++;
        }
      h[2 * (st * nw + w) + 1] = q;
    }
  }
  rc = fmbh_malloc((void **)d_out, sizeof(int) * 2 * q);
  if (!rc) rc = fmbh_h2d(*d_out, h, sizeof(int) * 2 * q, stream);
  return rc;
}

/* Whether an M2L of order p over npairs pairs and nrhs right-hand sides runs
 * target-stationary.  Measured against the offset-batched kernels on trees of
 * 3 to 6 levels (926 to 400,056 pairs a level), as speedups:
 *   FP64, up to 16 right-hand sides: orders 2 to 15 1.1-2.0 (the least on level
 *     2, whose 2,504 pairs had 0.9-1.2 before the launch's split fitted them),
 *     order 16 1.02-1.7.  17 to 100: 1.0-2.0; the worst levels 0.96 (order 16,
 *     17 right-hand sides) and 0.93 (level 2, 33).  Order 18 0.78.
 *   FP32: orders 2 to 14 1.1-2.3, at or under 36,192 vectors 0.85-1.1; order 15
 *     from 16 right-hand sides on 1.0-1.5, order 16 1.1-1.3 where the batches of
 *     a pair fill up, but 0.85-0.98 at 17 to 29 right-hand sides, two batches a
 *     pair, 0.92-1.0 with fewer than 16, and 0.78-0.92 on a level of 926 pairs.
 * (Above order 16 the batch and the sums no longer fit the LDS at a useful
 * size.) */
static int ts_use(int prec, int p, int npairs, int nrhs) {
  if (p > FMBH_TS_PMAX) return 0;
  if (prec == FMB_FP64) return 1;
  if ((double)npairs * nrhs < 40000 || (p > 14 && nrhs < 16)) return 0;
  return p < 16 || (npairs >= 4000 && (nrhs == 16 || nrhs >= 30));
}

/* sums of a workgroup: at most 32 target vectors in 160 KB of LDS, or in the
 * FP32 pass in 80 KB, so that two workgroups share a CU */
static int ts_slots(int prec, int p) {
  const size_t cap = (prec == FMB_FP64 ? 160 : 80) * 1024;
  int s = 32;
  while (s > 1 && fmbh_ts_lds_bytes(p, prec, s) > cap) s--;
  return s;
}

/* schedule, pair lists and coaxial tables of the target-stationary M2L at
 * level l, where its shape was not requested otherwise.  Two lists: groups of
 * as many targets as fill the slots at the most right-hand sides that run so,
 * and at one (passes with fewer right-hand sides than the plan holds). */
static int ts_setup(fmb_plan *pl, int l, fmb_rcr_tab *tb, int op, void *stream) {
  const fmb_tree *t = pl->tree;
  const fmb_plan_params *prm = &pl->prm;
  fmb_opset *o = &pl->ops[op];
  const int p = pl->p[l];
  int rc, coff[FMBH_TS_PMAX], *d_coff = NULL;
  /* 32-bit buffer offsets into the coefficients */
  if ((size_t)t->nbox[l] * pl->nrhs_max * p * p * o->csz >= (1ull << 32)) return FMB_OK;
  if (prm->rcr_mode || prm->waves || prm->ldso || (prm->split_bf16 && op == 1) ||
      prm->m2l_tile != RCR_TILE || prm->m2l_tile_min_mb != RCR_TILE_MIN_MB)
    return FMB_OK;
  int most = pl->nrhs_max; /* the most right-hand sides that a pass may run so */
  while (most && !(t->npairs[l] && ts_use(o->prec, p, t->npairs[l], most))) most--;
  if (!most) return FMB_OK;
  const int S = ts_slots(o->prec, p);
  tb->ts_slots[op] = S;
  for (int i = 0; i < (pl->nrhs_max > 1 ? 2 : 1); i++) {
    const int R = i || pl->nrhs_max == 1 ? 1 : (most < S ? most : S);
    tb->ts_tgrp[op][i] = S / R;
    const size_t bytes = sizeof(int) * (2 * (size_t)t->npairs[l] +
                                        (size_t)FMB_NCLASS * (t->nbox[l] / (S / R) + 1));
    if ((rc = fmbh_ts_lists(t, l, S / R, pl->off_class, &tb->d_ts_pairs[op][i],
                            &tb->d_ts_seg[op][i], stream)))
      return rc;
    pl->bytes += bytes;
  }
  if ((rc = ts_sched(o->prec, p, &tb->d_ts_sched[op], stream))) return rc;
  tb->ts_cstride[op] = ts_blocks(o->prec, 0, p, coff);
  const size_t cb = o->csz / 2 * (size_t)tb->ts_cstride[op] * FMB_NDIST;
  if ((rc = fmbh_malloc(&tb->d_ts_C[op], cb))) return rc;
  pl->bytes += cb;
  rc = fmbh_malloc((void **)&d_coff, sizeof(int) * p);
  if (!rc) rc = fmbh_h2d(d_coff, coff, sizeof(int) * p, stream);
  if (!rc)
    rc = fmbh_ts_coax(o->prec, o->d_Csr[l], p, d_coff, tb->ts_cstride[op], tb->d_ts_C[op], stream);
  if (!rc) rc = fmbh_sync(stream);
  fmbh_free(d_coff);
  return rc;
}

static void ts_job(const fmb_plan *pl, int op, int l, int trans, int nrhs, fmbh_ts_job *job) {
  const fmb_rcr_tab *tb = &pl->rcr[0][l];
  const fmb_opset *o = &pl->ops[op];
  const int S = tb->ts_slots[op];
  /* the list of one right-hand side per group where the other would leave
   * over a quarter of the slots empty */
  int i = 0;
  if (tb->d_ts_pairs[op][1]) {
    const int T = tb->ts_tgrp[op][0], R = S / T < nrhs ? S / T : nrhs;
    i = 4 * T * R < 3 * S && R < 16;
  }
  fmbh_ts_job j;
  j.pairs = tb->d_ts_pairs[op][i];
  j.seg = tb->d_ts_seg[op][i];
  j.npairs = pl->tree->npairs[l];
  j.tgrp = tb->ts_tgrp[op][i];
  j.nbox = pl->tree->nbox[l];
  j.ngroups = (j.nbox + j.tgrp - 1) / j.tgrp;
  j.slots = S;
  j.p = pl->p[l];
  j.phase = o->d_ts_phase[trans];
  j.pstride = o->ts_P;
  j.H = o->d_ts_H;
  j.hstride = o->ts_hstride;
  j.C = tb->d_ts_C[op];
  j.cstride = tb->ts_cstride[op];
  j.cdist = pl->class_dist;
  j.sched = tb->d_ts_sched[op];
  j.in = trans ? o->d_L[l] : o->d_M[l];
  j.out = trans ? o->d_M[l] : o->d_L[l];
  *job = j;
}

static int ts_run(const fmb_plan *pl, int op, int l, int trans, int nrhs, void *stream) {
  fmbh_ts_job j;
  ts_job(pl, op, l, trans, nrhs, &j);
  return fmbh_ts_run(&j, 1, pl->ops[op].prec, nrhs, stream);
}

/* the target-stationary M2L was set up for this pass */
static int ts_ready(const fmb_plan *pl, int op, int l, int nrhs) {
  return pl->rcr[0][l].ts_slots[op] &&
         ts_use(pl->ops[op].prec, pl->p[l], pl->tree->npairs[l], nrhs);
}

/* Whether an FP64 pass on two streams keeps to 4 waves in every launch.  The
 * 8-wave forms fill a CU, so that little runs beside them: where the finest
 * levels have no such form, what they win is less than what the streams then
 * hide.  327,680 triangles, 8 to 16 kHz, nine right-hand sides, 4 against 8
 * waves, with the share of M2L's work (pairs x order^3) in levels of the
 * 8-wave form: 265.6 and 279.0 ms at 0.35, 326.2 and 341.0 at 0.38, 430.5 and
 * 428.0 at 0.64, 700.1 and 683.7 at 0.67; 81,920 triangles 64.6 and 65.2 at
 * 0.31, 153.2 and 144.4 at 0.60, 101.3 and 97.4 at 0.61.  One right-hand side:
 * no difference at 0.35 and 0.38.  A target-stationary finest level fills the
 * CUs itself (1.02 to 1.09 in favour of 8 waves); one stream has nothing to
 * hide (351 ms with 8 waves, 368 with 4, at 0.38).  (FP32, whose batches take
 * half the LDS, gains with 8 waves on either.) */
static int narrow_pass(const fmb_plan *pl, int op, int nrhs, int split) {
  const int L = pl->tree->lmax;
  return split && pl->ops[op].prec == FMB_FP64 && nrhs > 1 && pl->ops[op].wide_share < 0.5 &&
         !pl->rcr[0][L].wide8[op] && !ts_ready(pl, op, L, nrhs);
}

/* tile shape of one launch; split: of a pass on two streams */
static void job_shape(const fmb_plan *pl, const fmb_rcr_tab *tb, int op, int nrhs, int split,
                      fmbh_rcr_job *j) {
  j->mode = tb->mode[op];
  j->bf = tb->bf[op];
  const int v = 8 * tb->nt[op];
  const long wgs = (long)j->nchunks * ((j->chunk_pairs * nrhs + v - 1) / v);
  if (tb->d_sched8[op] && (wgs <= 128 || (tb->wide8[op] && !narrow_pass(pl, op, nrhs, split)))) {
    j->nt = tb->nt8[op];
    j->mt = tb->mt8[op];
    j->nw = 8;
    j->sched = tb->d_sched8[op];
    j->sched_len = tb->sched8_len[op];
    return;
  }
  j->nt = tb->nt[op];
  j->mt = tb->mt[op];
  j->nw = tb->nw[op];
  j->sched = tb->d_sched[op];
  j->sched_len = tb->sched_len[op];
}

/* M2L (M2L^T) of the finest levels that run target-stationary, in one launch;
 * *from: the coarsest level done, lmax + 1 if none.  A level of a few hundred
 * workgroups ends in a round that leaves CUs idle, and each launch sets up its
 * tables again: levels 2 and 3 of 1,280 triangles (FP64) 27 + 41 us apart, 55
 * together. */
int fmbx_m2l_levels(const fmb_plan *pl, int op, int trans, int nrhs, int *from, void *stream) {
  fmbh_ts_job j[FMBH_TS_LEVELS];
  int n = 0, l = pl->tree->lmax;
  for (; l >= 2 && n < FMBH_TS_LEVELS && pl->rcr[0][l].mode[op] && ts_ready(pl, op, l, nrhs); l--)
    ts_job(pl, op, l, trans, nrhs, &j[n++]);
  *from = l + 1;
  return fmbh_ts_run(j, n, pl->ops[op].prec, nrhs, stream);
}

int fmbx_rcr_rot_setup(fmb_plan *pl, void *stream) {
  if (pl->prm.rcr_path == FMB_RCR_VALU) return FMB_OK;
  int rc = FMB_OK;
  /* e^{i m phi} of every bucket, m < Pmax, per opset */
  int nph[3] = {FMB_NOFF, 8, 8};
  for (int q = 0; q < 3 && !rc; q++) {
    double *ph = (double *)malloc(sizeof(double) * 2 * nph[q] * pl->Pmax);
    for (int b = 0; b < nph[q]; b++) {
      double phi = q == 0 ? pl->off_phi[b] : (q == 1 ? pl->m2m_phi[b] : pl->l2l_phi[b]);
      for (int m = 0; m < pl->Pmax; m++) {
        ph[2 * ((size_t)b * pl->Pmax + m)] = cos(m * phi);
        ph[2 * ((size_t)b * pl->Pmax + m) + 1] = sin(m * phi);
      }
    }
    /* cj = 0: e^{i m phi}; cj = 1: e^{-i m phi} for the transposed pass */
    size_t n = (size_t)2 * nph[q] * pl->Pmax;
    for (int cj = 0; cj < 2 && !rc; cj++) {
      if (cj)
        for (size_t i = 1; i < n; i += 2) ph[i] = -ph[i];
      for (int op = 0; op < pl->nops && !rc; op++) {
        fmb_opset *o = &pl->ops[op];
        void **dst = cj ? &o->d_phase_c[q] : &o->d_phase[q];
        rc = fmbh_malloc(dst, o->csz / 2 * n);
        if (rc) break;
        if (o->prec == FMB_FP64) {
          rc = fmbh_h2d(*dst, ph, sizeof(double) * n, stream);
          if (!rc) rc = fmbh_sync(stream);
        } else {
          float *f = (float *)malloc(sizeof(float) * n);
          for (size_t i = 0; i < n; i++) f[i] = (float)ph[i];
          rc = fmbh_h2d(*dst, f, sizeof(float) * n, stream);
          if (!rc) rc = fmbh_sync(stream);
          free(f);
        }
      }
    }
    free(ph);
  }
  for (int op = 0; op < pl->nops && !rc; op++) rc = ts_rot_setup(pl, &pl->ops[op], stream);
  if (rc) return rc;
  /* padded rotation blocks of every polar angle, per opset */
  int *hoff = (int *)malloc(sizeof(int) * (pl->Pmax + 1)), *d_hoff = NULL;
  rot_offsets(pl->Pmax, hoff);
  rc = fmbh_malloc((void **)&d_hoff, sizeof(int) * (pl->Pmax + 1));
  if (!rc) rc = fmbh_h2d(d_hoff, hoff, sizeof(int) * (pl->Pmax + 1), stream);
  for (int op = 0; op < pl->nops && !rc; op++) {
    fmb_opset *o = &pl->ops[op];
    o->hpad_stride = (size_t)hoff[pl->Pmax];
    size_t bytes = o->csz / 2 * o->hpad_stride * pl->nbeta;
    rc = fmbh_malloc(&o->d_Hpad, bytes);
    if (!rc) {
      pl->bytes += bytes;
      /* from the FP64 blocks (opset 0), rounded once */
      rc = fmbh_pad_rot(o->prec, (const double *)pl->ops[0].d_H, pl->nbeta, pl->Pmax, d_hoff,
                        o->hpad_stride, o->d_Hpad, stream);
    }
    /* split-BF16 copies for the FP32 pass */
    if (!rc && use_bf(pl, op, FMBH_RCR_LDS)) {
      int *hb = (int *)malloc(sizeof(int) * (pl->Pmax + 1)), *d_hb = NULL;
      if (!hb) rc = fmb_set_error(FMB_ERR_NOMEM, "split-BF16 offsets");
      if (!rc) {
        rot_offsets_bf(pl->Pmax, hb);
        o->hb_half = (size_t)hb[pl->Pmax];
        size_t hbytes = 2 * sizeof(uint16_t) * o->hb_half * pl->nbeta;
        rc = fmbh_malloc((void **)&d_hb, sizeof(int) * (pl->Pmax + 1));
        if (!rc) rc = fmbh_h2d(d_hb, hb, sizeof(int) * (pl->Pmax + 1), stream);
        if (!rc) rc = fmbh_malloc(&o->d_Hb, hbytes);
        if (!rc) {
          pl->bytes += hbytes;
          rc = fmbh_split_rot((const double *)pl->ops[0].d_H, pl->nbeta, pl->Pmax, d_hb,
                              o->hb_half, o->d_Hb, stream);
        }
        if (!rc) rc = fmbh_sync(stream);
      }
      fmbh_free(d_hb);
      free(hb);
    }
  }
  if (!rc) rc = fmbh_sync(stream);
  fmbh_free(d_hoff);
  free(hoff);
  return rc;
}

/* global workspace of one opset: the largest GWS batch among its
 * translations (at least min_per_wg bytes per workgroup) */
static int size_gws(fmb_plan *pl, int op, size_t min_per_wg) {
  fmb_opset *o = &pl->ops[op];
  size_t need = min_per_wg;
  for (int kind = 0; kind < 3; kind++)
    for (int l = 2; l <= pl->tree->lmax; l++) {
      const fmb_rcr_tab *tb = &pl->rcr[kind][l];
      if (tb->mode[op] != FMBH_RCR_GWS) continue;
      size_t b = fmbh_rcr_gws_bytes(tb->P, o->prec, tb->nt[op]);
      if (b > need) need = b;
    }
  need *= RCR_GWS_GRID;
  o->gws_slot = need;
  /* a second slot for the launches on the plan's second stream */
  if (pl->aux) need *= 2;
  if (need == o->gws_bytes) return FMB_OK;
  fmbh_free(o->d_gws);
  o->d_gws = NULL;
  pl->bytes -= o->gws_bytes;
  o->gws_bytes = 0;
  o->gws_grid = 0;
  if (!need) return FMB_OK;
  int rc = fmbh_malloc(&o->d_gws, need);
  if (rc) return rc;
  o->gws_bytes = need;
  o->gws_grid = RCR_GWS_GRID;
  pl->bytes += need;
  return FMB_OK;
}

/* ---- autotuning of the tile shapes ----
 * Each translation (kind, level) of each opset is timed, on the plan's own
 * box pairs and buffers at nrhs_max right-hand sides, in every valid shape:
 * LDS mode with 8 or 16 vectors per batch (when the batch fits the 160 KB of
 * LDS), and global-workspace mode with 8 or 16 vectors and row groups of
 * 2, 3, 4 or 6 tiles, each with 4 or 8 waves per workgroup, and with
 * split_bf16 the LDS shapes once more with split-BF16 rotations.  The fastest
 * shape (a one-vector warm-up, then one timed run, HIP events on the plan's
 * stream) replaces the fixed rule of fmbh_rcr_shape. */
typedef struct {
  int mode, nt, mt, nw, bf;
} shape_t;

/* bfok: LDS shapes are also tried with split-BF16 rotations */
static int shape_candidates(int P, int bfok, shape_t *c) {
  int n = 0, mt = fmbh_rcr_mt_lds(P, 0);
  static const int mts[4] = {2, 3, 4, 6};
  for (int nw = 4; nw <= 8; nw += 4) {
    for (int bf = 0; bf <= bfok; bf++)
      for (int nt = 1; nt <= 2; nt++) {
        /* split-BF16 rotations keep the standard (2P - 1 row) blocks */
        const int m = fmbh_rcr_mt_lds(P, bf);
        if (m) {
          shape_t v = {FMBH_RCR_LDS, nt, m, nw, bf}, w = {FMBH_RCR_LDSP, nt, m, nw, bf};
          c[n++] = v;
          c[n++] = w;
        }
      }
    for (int nt = 1; nt <= 2; nt++)
      if (mt) {
        shape_t v = {FMBH_RCR_LDSO, nt, mt, nw, 0};
        c[n++] = v;
      }
    for (int nt = 1; nt <= 2; nt++)
      for (int i = 0; i < 4; i++) {
        shape_t v = {FMBH_RCR_GWS, nt, mts[i], nw, 0};
        c[n++] = v;
      }
  }
  return n;
}

/* one launch at one right-hand side (loads the kernel's code object and the
 * operator blocks into the caches), then one timed launch at nrhs_max */
static int time_run(fmb_plan *pl, int op, int kind, int l, void *stream, float *ms) {
  void *e0 = NULL, *e1 = NULL;
  int rc = fmbh_event_create(&e0);
  if (!rc) rc = fmbh_event_create(&e1);
  if (!rc) rc = fmbx_rcr_run(pl, op, kind, l, 1, stream);
  if (!rc) rc = fmbh_event_record(e0, stream);
  if (!rc) rc = fmbx_rcr_run(pl, op, kind, l, pl->nrhs_max, stream);
  if (!rc) rc = fmbh_event_record(e1, stream);
  if (!rc) rc = fmbh_sync(stream);
  if (!rc) rc = fmbh_event_elapsed(e0, e1, ms);
  fmbh_event_destroy(e0);
  fmbh_event_destroy(e1);
  return rc;
}

/* Shapes already tuned, keyed by what the timing depends on: device,
 * precision, kind, orders, chunk count and right-hand sides (a sweep that
 * revisits a level's order reuses its result).  The cache lives for the
 * process and in a text file shared by processes: FMBEM_TUNE_CACHE names it
 * (empty: no file), else $XDG_CACHE_HOME/fmbem/rcr_tiles.txt or
 * $HOME/.cache/fmbem/rcr_tiles.txt.  Each tuned shape is appended as one
 * line under an advisory lock; a process reads the file once, at its first
 * autotuned plan, and a later line for the same key wins. */
typedef struct {
  int prec, kind, pin, pout, nchunks, nrhs, bf;
  shape_t shape;
  float ms;
} tuned_t;
#define TUNE_CACHE 4096
#define TUNE_MAGIC "fmbem-rcr-tile-v2"
#define TUNE_TS 3 /* kind of the target-stationary M2L's entries */
static tuned_t tune_cache[TUNE_CACHE];
static int tune_cached, tune_loaded;
static char tune_dev[64];
static pthread_mutex_t tune_lock = PTHREAD_MUTEX_INITIALIZER;

static int same_key(const tuned_t *c, const tuned_t *key) {
  return c->prec == key->prec && c->kind == key->kind && c->pin == key->pin &&
         c->pout == key->pout && c->nchunks == key->nchunks && c->nrhs == key->nrhs &&
         c->bf == key->bf;
}

/* caller holds tune_lock: replaces an entry of the same key or appends */
static void cache_store(const tuned_t *v) {
  for (int i = 0; i < tune_cached; i++)
    if (same_key(&tune_cache[i], v)) {
      tune_cache[i] = *v;
      return;
    }
  tune_cache[tune_cached < TUNE_CACHE ? tune_cached++ : TUNE_CACHE - 1] = *v;
}

/* the cache file's path, or 0 when there is none */
static int tune_path(char *buf, size_t n) {
  const char *e = getenv("FMBEM_TUNE_CACHE");
  if (e) {
    if (!*e || strlen(e) >= n) return 0;
    strcpy(buf, e);
    return 1;
  }
  const char *x = getenv("XDG_CACHE_HOME"), *h = getenv("HOME");
  int w;
  if (x && *x)
    w = snprintf(buf, n, "%s/fmbem/rcr_tiles.txt", x);
  else if (h && *h)
    w = snprintf(buf, n, "%s/.cache/fmbem/rcr_tiles.txt", h);
  else
    return 0;
  return w > 0 && (size_t)w < n;
}

/* creates the directories leading to path (mkdir -p of its dirname) */
static void make_parents(const char *path) {
  char d[1024];
  size_t n = strlen(path);
  if (n >= sizeof(d)) return;
  memcpy(d, path, n + 1);
  for (char *p = d + 1; *p; p++)
    if (*p == '/') {
      *p = 0;
      mkdir(d, 0755);
      *p = '/';
    }
}

/* reads the file's entries for this device (once per process) */
static void tune_load(void) {
  if (tune_loaded) return;
  tune_loaded = 1;
  if (fmbh_device_tag(tune_dev, sizeof(tune_dev))) tune_dev[0] = 0;
  char path[1024], line[512], magic[32], dev[64];
  if (!tune_path(path, sizeof(path))) return;
  FILE *f = fopen(path, "r");
  if (!f) return;
  flock(fileno(f), LOCK_SH);
  while (fgets(line, sizeof(line), f)) {
    tuned_t v;
    if (sscanf(line, "%31s %63s %d %d %d %d %d %d %d %d %d %d %d %d %f", magic, dev, &v.prec,
               &v.kind, &v.pin, &v.pout, &v.nchunks, &v.nrhs, &v.bf, &v.shape.mode,
               &v.shape.nt, &v.shape.mt, &v.shape.nw, &v.shape.bf, &v.ms) != 15)
      continue;
    if (strcmp(magic, TUNE_MAGIC) || strcmp(dev, tune_dev)) continue;
    if (v.kind == TUNE_TS) { /* a time only */
      if (v.shape.mode == FMB_RCR_MODE_TS && v.ms > 0) cache_store(&v);
      continue;
    }
    /* only shapes this build can launch; split-BF16 only where allowed */
    if (v.shape.mode < FMBH_RCR_LDS || v.shape.mode > FMBH_RCR_LDSO || v.shape.nt < 1 ||
        v.shape.nt > 2 || (v.shape.nw != 4 && v.shape.nw != 8) || v.kind < 0 || v.kind > 2 ||
        (v.shape.mt != 2 && v.shape.mt != 3 && v.shape.mt != 4 && v.shape.mt != 6) ||
        (v.shape.bf && (!v.bf || v.shape.mode == FMBH_RCR_GWS ||
                        v.shape.mode == FMBH_RCR_LDSO)) || !(v.ms >= 0))
      continue;
    cache_store(&v);
  }
  flock(fileno(f), LOCK_UN);
  fclose(f);
}

static void tune_append(const tuned_t *v) {
  char path[1024];
  if (!tune_dev[0] || !tune_path(path, sizeof(path))) return;
  make_parents(path);
  FILE *f = fopen(path, "a");
  if (!f) return;
  flock(fileno(f), LOCK_EX);
  fprintf(f, "%s %s %d %d %d %d %d %d %d %d %d %d %d %d %.4f\n", TUNE_MAGIC, tune_dev,
          v->prec, v->kind, v->pin, v->pout, v->nchunks, v->nrhs, v->bf, v->shape.mode,
          v->shape.nt, v->shape.mt, v->shape.nw, v->shape.bf, v->ms);
  fflush(f);
  flock(fileno(f), LOCK_UN);
  fclose(f);
}

static int cache_find(const tuned_t *key, tuned_t *out) {
  int hit = 0;
  pthread_mutex_lock(&tune_lock);
  tune_load();
  for (int i = 0; i < tune_cached && !hit; i++)
    if (same_key(&tune_cache[i], key)) {
      *out = tune_cache[i];
      hit = 1;
    }
  pthread_mutex_unlock(&tune_lock);
  return hit;
}

static void cache_put(const tuned_t *v) {
  pthread_mutex_lock(&tune_lock);
  cache_store(v);
  tune_append(v);
  pthread_mutex_unlock(&tune_lock);
}

static int autotune(fmb_plan *pl, int op, void *stream) {
  const fmb_tree *t = pl->tree;
  fmb_opset *o = &pl->ops[op];
  int L = t->lmax, rc = FMB_OK;
  /* defined contents for the timing runs */
  for (int l = 2; l <= L && !rc; l++) {
    size_t bytes = (size_t)t->nbox[l] * pl->nrhs_max * pl->p[l] * pl->p[l] * o->csz;
    rc = fmbh_memset(o->d_M[l], 0, bytes, stream);
    if (!rc) rc = fmbh_memset(o->d_L[l], 0, bytes, stream);
  }
  int *hoff = (int *)malloc(sizeof(int) * (pl->Pmax + 1));
  int *hboff = (int *)malloc(sizeof(int) * (pl->Pmax + 1));
  if (!hoff || !hboff) {
    free(hoff);
    free(hboff);
    return fmb_set_error(FMB_ERR_NOMEM, "rotation offsets");
  }
  rot_offsets(pl->Pmax, hoff);
  rot_offsets_bf(pl->Pmax, hboff);
  for (int kind = 0; kind < 3 && !rc; kind++)
    for (int l = (kind ? 3 : 2); l <= L && !rc; l++) {
      fmb_rcr_tab *tb = &pl->rcr[kind][l];
      const fmb_rcr_tab *pairs = kind == 0 ? tb : &pl->rcr[1][l];
      if (!tb->mode[op] || !pairs->nchunks) continue;
      int mn = tb->pin < tb->pout ? tb->pin : tb->pout;
      int *coff = (int *)malloc(sizeof(int) * (mn + 1));
      if (!coff) {
        rc = fmb_set_error(FMB_ERR_NOMEM, "coaxial offsets");
        break;
      }
      coax_offsets(tb->pin, tb->pout, coff);
      tuned_t key = {o->prec, kind, tb->pin, tb->pout, pairs->nchunks, pl->nrhs_max,
                     use_bf(pl, op, FMBH_RCR_LDS), {0, 0, 0, 0, 0}, 0.0f}, hit;
      shape_t c[48];
      int nc;
      float best = 0.0f;
      int cached = cache_find(&key, &hit);
      if (cached) {
        /* only the cached shape, with its recorded time (no timing run) */
        c[0] = hit.shape;
        nc = 1;
        best = 1e30f;
      } else {
        rc = time_run(pl, op, kind, l, stream, &best);
        nc = shape_candidates(tb->P, use_bf(pl, op, FMBH_RCR_LDS), c);
      }
      for (int i = 0; i < nc && !rc; i++) {
        if (c[i].mode == tb->mode[op] && c[i].nt == tb->nt[op] && c[i].mt == tb->mt[op] &&
            c[i].nw == tb->nw[op] && c[i].bf == tb->bf[op])
          continue;
        int *sched = NULL, slen = 0;
        const int bf = c[i].bf;
        if ((rc = build_sched(tb->pin, tb->pout, tb->P, c[i].mode, c[i].mt, c[i].nw,
                              bf ? hboff : hoff, bf, coff, &sched, &slen, stream)))
          break;
        if (c[i].mode == FMBH_RCR_LDS || c[i].mode == FMBH_RCR_LDSP ||
            c[i].mode == FMBH_RCR_LDSO) {
          size_t b = c[i].mode == FMBH_RCR_LDSO
                         ? fmbh_rcr_ldso_bytes(tb->P, o->prec, c[i].nt, slen, tb->hlen,
                                               tb->cpad_stride)
                         : fmbh_rcr_lds_bytes(tb->P, o->prec, c[i].nt, slen);
          if (!b || b > 160 * 1024) {
            fmbh_free(sched);
            continue;
          }
        } else if ((rc = size_gws(pl, op, fmbh_rcr_gws_bytes(tb->P, o->prec, c[i].nt)))) {
          fmbh_free(sched);
          break;
        }
        shape_t prev = {tb->mode[op], tb->nt[op], tb->mt[op], tb->nw[op], tb->bf[op]};
        int *psched = tb->d_sched[op], plen = tb->sched_len[op];
        tb->mode[op] = c[i].mode;
        tb->nt[op] = c[i].nt;
        tb->mt[op] = c[i].mt;
        tb->nw[op] = c[i].nw;
        tb->bf[op] = bf;
        tb->d_sched[op] = sched;
        tb->sched_len[op] = slen;
        float ms = 0.0f;
        /* a cached shape is taken as it is; candidates are timed */
        if (!cached) rc = time_run(pl, op, kind, l, stream, &ms);
        if (!rc && ms < best) {
          best = ms;
          fmbh_free(psched);
        } else {
          tb->mode[op] = prev.mode;
          tb->nt[op] = prev.nt;
          tb->mt[op] = prev.mt;
          tb->nw[op] = prev.nw;
          tb->bf[op] = prev.bf;
          tb->d_sched[op] = psched;
          tb->sched_len[op] = plen;
          fmbh_free(sched);
        }
      }
      if (!rc && cached) best = hit.ms;
      tb->tuned_ms[op] = best;
      if (!rc && !cached) {
        key.shape.mode = tb->mode[op];
        key.shape.nt = tb->nt[op];
        key.shape.mt = tb->mt[op];
        key.shape.nw = tb->nw[op];
        key.shape.bf = tb->bf[op];
        key.ms = best;
        cache_put(&key);
      }
      free(coff);
    }
  free(hoff);
  free(hboff);
  if (!rc) rc = size_gws(pl, op, 0);
  return rc;
}

/* A tuned plan's M2L runs target-stationary where that is faster than the
 * tuned shape too, by its own time at nrhs_max right-hand sides (timed, or
 * from the cache). */
static int ts_tuned(fmb_plan *pl, int op, int l, void *stream) {
  fmb_rcr_tab *tb = &pl->rcr[0][l];
  if (!(tb->tuned_ms[op] > 0) || !ts_ready(pl, op, l, pl->nrhs_max)) return FMB_OK;
  tuned_t key = {pl->ops[op].prec, TUNE_TS, tb->pin, tb->pout, tb->nchunks, pl->nrhs_max, 0,
                 {FMB_RCR_MODE_TS, 2, 0, 0, 0}, 0.0f}, hit;
  if (cache_find(&key, &hit)) {
    key.ms = hit.ms;
  } else {
    int rc = time_run(pl, op, 0, l, stream, &key.ms);
    if (rc) return rc;
    cache_put(&key);
  }
  if (key.ms >= tb->tuned_ms[op]) tb->ts_slots[op] = 0;
  return FMB_OK;
}

/* The tile-major M2L order keeps a tile's sources in its XCD's L2.  It pays
 * where the level's FP64 source coefficients (boxes x right-hand sides x
 * p^2 x 16 bytes) outgrow the GPU's 256 MB last-level (Infinity) cache, the
 * default m2l_tile_min_mb; below that the offset-major order's fuller chunks
 * win (measured: the level-6 and level-7 M2L of the 327,680-triangle sphere
 * at 9 right-hand sides 5-9% faster tile-major; the 20,480- and
 * 81,920-triangle spheres at one right-hand side 6-10% slower per matvec). */
static int m2l_tiled(const fmb_plan *pl, int l) {
  if (pl->prm.m2l_tile <= 0) return 0;
  const size_t p2 = (size_t)pl->p[l] * pl->p[l];
  const size_t bytes = (size_t)pl->tree->nbox[l] * pl->nrhs_max * p2 * 16;
  return bytes > ((size_t)(pl->prm.m2l_tile_min_mb > 0 ? pl->prm.m2l_tile_min_mb : 0) << 20);
}

int fmbx_rcr_setup(fmb_plan *pl, void *stream) {
  const fmb_tree *t = pl->tree;
  int L = t->lmax, rc = FMB_OK;
  for (int kind = 1; kind <= 2; kind++) {
    rcr_info_t info[8];
    for (int o = 0; o < 8; o++) {
      info[o].beta = kind == 1 ? pl->m2m_beta[o] : pl->l2l_beta[o];
      info[o].dist = 0;
      info[o].phi = kind == 1 ? pl->m2m_phi[o] : pl->l2l_phi[o];
    }
    if ((rc = fmbh_malloc(&pl->d_info_oct[kind - 1], sizeof(info)))) return rc;
    if ((rc = fmbh_h2d(pl->d_info_oct[kind - 1], info, sizeof(info), stream))) return rc;
    if ((rc = fmbh_sync(stream))) return rc;
  }
  if (pl->prm.rcr_path != FMB_RCR_VALU) {
    int *hoff = (int *)malloc(sizeof(int) * (pl->Pmax + 1));
    int *hboff = (int *)malloc(sizeof(int) * (pl->Pmax + 1));
    if (!hoff || !hboff) {
      free(hoff);
      free(hboff);
      return fmb_set_error(FMB_ERR_NOMEM, "rotation offsets");
    }
    rot_offsets(pl->Pmax, hoff);
    rot_offsets_bf(pl->Pmax, hboff);
    for (int l = 2; l <= L && !rc; l++) {
      fmb_rcr_tab *tb = &pl->rcr[0][l];
      void *C[2] = {pl->ops[0].d_Csr[l], pl->ops[1].d_Csr[l]};
      tb->tiled = m2l_tiled(pl, l);
      if (tb->tiled)
        rc = build_chunks_tiled(t, l, pl->prm.m2l_tile, tb, stream);
      else
        rc = build_chunks(t->h_off_start[l], FMB_NOFF, tb, stream);
      if (rc) break;
      rc = plan_tab(pl, tb, pl->p[l], pl->p[l], C, FMB_NDIST, hoff, hboff, stream);
    }
    for (int l = 3; l <= L && !rc; l++) {
      fmb_rcr_tab *up = &pl->rcr[1][l], *dn = &pl->rcr[2][l];
      void *Cu[2] = {pl->ops[0].d_Cm2m[l], pl->ops[1].d_Cm2m[l]};
      void *Cd[2] = {pl->ops[0].d_Cl2l[l], pl->ops[1].d_Cl2l[l]};
      if ((rc = octant_pairs(t, l, up, stream))) break;
      if ((rc = plan_tab(pl, up, pl->p[l], pl->p[l - 1], Cu, 1, hoff, hboff, stream))) break;
      rc = plan_tab(pl, dn, pl->p[l - 1], pl->p[l], Cd, 1, hoff, hboff, stream);
    }
    free(hoff);
    free(hboff);
    if (rc) return rc;
  }
  for (int op = 0; op < pl->nops; op++)
    if ((rc = size_gws(pl, op, 0))) return rc;
  if (pl->prm.autotune && pl->prm.rcr_path != FMB_RCR_VALU)
    for (int op = 0; op < pl->nops; op++)
      if ((rc = autotune(pl, op, stream))) return rc;
  /* (last: the autotuner's shapes are those of the offset-batched kernels) */
  if (pl->prm.rcr_path != FMB_RCR_VALU)
    for (int op = 0; op < pl->nops; op++)
      for (int l = 2; l <= L; l++) {
        if ((rc = ts_setup(pl, l, &pl->rcr[0][l], op, stream))) return rc;
        if (pl->prm.autotune && (rc = ts_tuned(pl, op, l, stream))) return rc;
      }
  for (int op = 0; op < pl->nops; op++) {
    double all = 0.0, wide = 0.0;
    for (int l = 2; l <= L; l++) {
      const double w = (double)t->npairs[l] * pl->p[l] * pl->p[l] * pl->p[l];
      all += w;
      if (pl->rcr[0][l].wide8[op]) wide += w;
    }
    pl->ops[op].wide_share = all > 0.0 ? wide / all : 0.0;
  }
  return FMB_OK;
}

void fmbx_rcr_free(fmb_plan *pl) {
  for (int kind = 0; kind < 3; kind++)
    for (int l = 0; l < FMB_MAXLEV; l++) {
      fmb_rcr_tab *tb = &pl->rcr[kind][l];
      fmbh_free(tb->d_chunks);
      fmbh_free(tb->d_par);
      fmbh_free(tb->d_chi);
      for (int op = 0; op < 2; op++) {
        fmbh_free(tb->d_sched[op]);
        fmbh_free(tb->d_sched8[op]);
        fmbh_free(tb->d_Cpad[op]);
        for (int i = 0; i < 2; i++) {
          fmbh_free(tb->d_ts_pairs[op][i]);
          fmbh_free(tb->d_ts_seg[op][i]);
        }
        fmbh_free(tb->d_ts_sched[op]);
        fmbh_free(tb->d_ts_C[op]);
      }
      memset(tb, 0, sizeof(*tb));
    }
  for (int i = 0; i < 2; i++) {
    fmbh_free(pl->d_info_oct[i]);
    pl->d_info_oct[i] = NULL;
  }
}

/* bytes of level l's coefficient array that a pass over nrhs vectors of
 * order p reaches ([box][nrhs][p^2]) */
static size_t coef_bytes(const fmb_plan *pl, const fmb_opset *o, int l, int p, int nrhs) {
  return (size_t)pl->tree->nbox[l] * nrhs * p * p * o->csz;
}

/* kind 0: M2L at level l; 1: M2M level l -> l-1; 2: L2L level l-1 -> l */
int fmbx_rcr_run(const fmb_plan *pl, int op, int kind, int l, int nrhs,
                 void *stream) {
  const fmb_rcr_tab *tb = &pl->rcr[kind][l];
  if (!tb->mode[op]) {
    if (kind == 0) return fmbh_m2l(pl, op, l, nrhs, stream);
    if (kind == 1) return fmbh_m2m(pl, op, l, nrhs, stream);
    return fmbh_l2l(pl, op, l, nrhs, stream);
  }
  if (kind == 0 && ts_ready(pl, op, l, nrhs)) return ts_run(pl, op, l, 0, nrhs, stream);
  const fmb_tree *t = pl->tree;
  const fmb_opset *o = &pl->ops[op];
  const fmb_rcr_tab *pairs = kind == 0 ? tb : &pl->rcr[1][l];
  fmbh_rcr_job j;
  memset(&j, 0, sizeof(j));
  j.Hb = o->d_Hb;
  j.hbstride = 2 * o->hb_half;
  j.hbhalf = o->hb_half;
  j.chunks = pairs->d_chunks;
  j.nchunks = pairs->nchunks;
  j.chunk_pairs = RCR_CHUNK;
  job_shape(pl, tb, op, nrhs, pl->split, &j);
  j.H = o->d_Hpad;
  j.hstride = o->hpad_stride;
  j.C = tb->d_Cpad[op];
  j.cstride = tb->cpad_stride;
  j.P = tb->P;
  j.pin = tb->pin;
  j.pout = tb->pout;
  j.hlen = tb->hlen;
  j.xcd = kind == 0 && tb->tiled && j.mode == FMBH_RCR_LDS;
  j.gws = (pl->aux && stream == pl->aux) ? (char *)o->d_gws + o->gws_slot : o->d_gws;
  j.gws_grid = o->gws_grid;
  j.phase = o->d_phase[kind];
  j.pstride = pl->Pmax;
  if (kind == 0) {
    j.info = pl->d_off_info;
    j.tgt = t->d_pair_tgt[l];
    j.src = t->d_pair_src[l];
    j.in = o->d_M[l];
    j.out = o->d_L[l];
  } else if (kind == 1) {
    j.info = pl->d_info_oct[0];
    j.tgt = pairs->d_par;
    j.src = pairs->d_chi;
    j.in = o->d_M[l];
    j.out = o->d_M[l - 1];
  } else {
    j.info = pl->d_info_oct[1];
    j.tgt = pairs->d_chi;
    j.src = pairs->d_par;
    j.in = o->d_L[l - 1];
    j.out = o->d_L[l];
  }
  /* source level: l (M2L, M2M) or l - 1 (L2L); target level: l or l - 1 */
  j.in_bytes = coef_bytes(pl, o, kind == 2 ? l - 1 : l, j.pin, nrhs);
  j.out_bytes = coef_bytes(pl, o, kind == 1 ? l - 1 : l, j.pout, nrhs);
  return fmbh_rcr(&j, o->prec, nrhs, stream);
}

/* The transposed translations.  The rotation blocks H_n(beta) are symmetric
 * and every coaxial |m| block satisfies C^T = P C P with P = diag((-1)^n),
 * so the transpose of T = Pout H C H Pin (Pin = e^{i m phi},
 * Pout = e^{-i m' phi}) is P (Pin H C' H Pout) P, where C' is C for M2L
 * and, for the scaled M2M / L2L blocks, the other direction's block:
 *   (diag(1/w_{l-1}) RR diag(w_l))^T = P diag(w_l) RR diag(1/w_{l-1}) P.
 * The transposed pass keeps its coefficients multiplied by P, so each
 * transposed translation is the forward kernel with conjugated phases:
 *   kind 0  M2L^T at l: L' (l) -> M' (l), pairs with source and target swapped;
 *   kind 1  M2M^T l-1 -> l: the L2L schedule and blocks, M2M's octant angles;
 *   kind 2  L2L^T l -> l-1: the M2M schedule and blocks, L2L's octant angles. */
int fmbx_rcr_run_t(const fmb_plan *pl, int op, int kind, int l, int nrhs,
                   void *stream) {
  const fmb_rcr_tab *tb = &pl->rcr[kind == 0 ? 0 : (kind == 1 ? 2 : 1)][l];
  if (!tb->mode[op])
    return fmb_set_error(FMB_ERR_ARG,
                         "transposed translations need the matrix-core kernels");
  if (kind == 0 && ts_ready(pl, op, l, nrhs)) return ts_run(pl, op, l, 1, nrhs, stream);
  const fmb_tree *t = pl->tree;
  const fmb_opset *o = &pl->ops[op];
  const fmb_rcr_tab *pairs = kind == 0 ? tb : &pl->rcr[1][l];
  fmbh_rcr_job j;
  memset(&j, 0, sizeof(j));
  j.Hb = o->d_Hb;
  j.hbstride = 2 * o->hb_half;
  j.hbhalf = o->hb_half;
  j.chunks = pairs->d_chunks;
  j.nchunks = pairs->nchunks;
  j.chunk_pairs = RCR_CHUNK;
  job_shape(pl, tb, op, nrhs, pl->split, &j);
  j.H = o->d_Hpad;
  j.hstride = o->hpad_stride;
  j.C = tb->d_Cpad[op];
  j.cstride = tb->cpad_stride;
  j.P = tb->P;
  j.pin = tb->pin;
  j.pout = tb->pout;
  j.hlen = tb->hlen;
  j.xcd = kind == 0 && tb->tiled && j.mode == FMBH_RCR_LDS;
  j.gws = (pl->aux && stream == pl->aux) ? (char *)o->d_gws + o->gws_slot : o->d_gws;
  j.gws_grid = o->gws_grid;
  j.phase = o->d_phase_c[kind];
  j.pstride = pl->Pmax;
  if (kind == 0) {
    j.info = pl->d_off_info;
    j.tgt = t->d_pair_src[l];
    j.src = t->d_pair_tgt[l];
    j.in = o->d_L[l];
    j.out = o->d_M[l];
  } else if (kind == 1) {
    j.info = pl->d_info_oct[0];
    j.tgt = pairs->d_chi;
    j.src = pairs->d_par;
    j.in = o->d_M[l - 1];
    j.out = o->d_M[l];
  } else {
    j.info = pl->d_info_oct[1];
    j.tgt = pairs->d_par;
    j.src = pairs->d_chi;
    j.in = o->d_L[l];
    j.out = o->d_L[l - 1];
  }
  /* source level: l (M2L^T, L2L^T) or l - 1 (M2M^T); target: l or l - 1 */
  j.in_bytes = coef_bytes(pl, o, kind == 1 ? l - 1 : l, j.pin, nrhs);
  j.out_bytes = coef_bytes(pl, o, kind == 2 ? l - 1 : l, j.pout, nrhs);
  return fmbh_rcr(&j, o->prec, nrhs, stream);
}

int fmb_plan_tile_shape(const fmb_plan *pl, int kind, int level, int prec, int *mode,
                        int *nt, int *mt, int *nw, int *bf, double *ms) {
  if (!pl || kind < 0 || kind > 2 || level < 2 || level > pl->tree->lmax ||
      (kind && level < 3))
    return fmb_set_error(FMB_ERR_ARG, "fmb_plan_tile_shape: invalid arguments");
  int op = (prec == FMB_MIXED && pl->nops == 2) ? 1 : 0;
  const fmb_rcr_tab *tb = &pl->rcr[kind][level];
  if (mode) *mode = tb->mode[op];
  if (nt) *nt = tb->nt[op];
  if (mt) *mt = tb->mt[op];
  if (nw) *nw = tb->nw[op];
  if (bf) *bf = tb->bf[op];
  if (ms) *ms = tb->tuned_ms[op];
  return FMB_OK;
}

int fmb_plan_launch_shape(const fmb_plan *pl, int kind, int level, int prec, int nrhs,
                          int *mode, int *nt, int *mt, int *nw, int *bf) {
  if (!pl || !pl->ready || kind < 0 || kind > 2 || level < 2 || level > pl->tree->lmax ||
      (kind && level < 3) || nrhs < 1 || nrhs > pl->nrhs_max)
    return fmb_set_error(FMB_ERR_ARG, "fmb_plan_launch_shape: invalid arguments");
  const int op = (prec == FMB_MIXED && pl->nops == 2) ? 1 : 0;
  const fmb_rcr_tab *tb = &pl->rcr[kind][level];
  fmbh_rcr_job j;
  memset(&j, 0, sizeof(j));
  if (kind == 0 && tb->mode[op] && ts_ready(pl, op, level, nrhs)) {
    j.mode = FMB_RCR_MODE_TS;
    j.nt = 2;
    j.nw = pl->ops[op].prec == FMB_FP64 ? FMBH_TS_WAVES64 : FMBH_TS_WAVES32;
  } else if (tb->mode[op]) {
    j.nchunks = (kind == 0 ? tb : &pl->rcr[1][level])->nchunks;
    j.chunk_pairs = RCR_CHUNK;
    job_shape(pl, tb, op, nrhs, pl->aux != NULL, &j);
  }
  if (mode) *mode = j.mode;
  if (nt) *nt = j.nt;
  if (mt) *mt = j.mt;
  if (nw) *nw = j.nw;
  if (bf) *bf = j.bf;
  return FMB_OK;
}
