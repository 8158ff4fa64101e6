/* Host-side packing of a captured decode step's inputs (CPython extension `_hostprep`).
 *
 * A graph-captured decode step reads its per-step inputs from static device buffers, uploaded
 * from pinned host buffers: token ids, positions and cache slots (int64), the attention plan's row
 * order and context lengths (int32), and the block-table rows (int32). Packing them walks every
 * scheduled sequence; this module does that walk in C, reading the same fields the runner's
 * ScheduledChunk carries (the reference builds the same per-token ids, positions and slots in
 * runner/model_runner.py:162-205).
 *
 *   pack_decode(chunks, block_size, limit, host_i64, host_meta, host_tables, max_blocks, own_slots=False) -> int
 *
 * chunks: the step's scheduled sequences (objects with token_ids, num_computed, num_new,
 * block_table, params). Returns -1 when the step is not a pure greedy decode step within `limit`
 * positions (one new token per sequence at position num_computed == len(token_ids) - 1, params
 * None or greedy) -- nothing is written then; otherwise writes
 *   host_i64[0:b] = ids, [b:2b] = positions, [2b:3b] = slots,
 *   host_meta[0:b] = sequences by position, longest first (ties in batch order),
 *   host_meta[b:2b] = their context lengths (position + 1),
 *   host_tables row r = block-table prefix of plan row r's sequence (the blocks its context uses),
 * and returns 1 when some table row changed, 0 when every row already held its prefix (the host
 * table buffer mirrors the device copy, so unchanged rows need no upload). Every check runs before
 * anything is written: a block table shorter than its context raises RuntimeError, an entry out of
 * int32 range OverflowError, and the buffers are left as they were. With own_slots, a step whose rows do
 * not own their slots (below) returns -1 as well.
 *
 *   rows_own_slots(tables, context_lens, block_size) -> bool
 *
 * Decode rows (int32 tables [rows, width], int32 context lengths [rows]) own their slots when the
 * slot of each row's new token, its table's slot of position context - 1, is no other position of any
 * row's context, its own included. Attention that writes the new keys in the launch that reads
 * the contexts needs this; the same sequence twice in a batch, or a block that is still written
 * to in two tables, breaks it. (Blocks shared as a full prefix do not.)
 *
 *   pack_step(chunks, block_size, tiles, own_rows=0) -> (data, total, sample_idx, layout[, own])
 *
 * Any step (prefill chunks, decodes, both): the flat batch of runner/model_runner.py:162-205 and
 * the attention plan of attention/backends.py:80-98 in one host buffer. `data` (a bytearray) holds
 * int64 [ids | positions | slots] over the `total` new tokens and the flat row of each sampled
 * sequence's last token (sequences whose new tokens end their token list, listed in sample_idx),
 * then the int32 plan parts named in `layout` ((name, shape) pairs, in order):
 *   d_rows, d_ctx [D], d_tables [D, max blocks]: the decode sequences (one new token), longest
 *     context first (ties in batch order), tables padded with block 0;
 *   p_info [P, 3] (flat start, new tokens, cached tokens), p_tables [P, max blocks]: the sequences
 *     with more than one new token, in batch order;
 *   p_work<t> [W, 2] for each tile size t in `tiles`: (prefill sequence, first new token) of every
 *     t-token query tile, the tiles with the most keys (cached + causal) first, ties in sequence
 *     then token order.
 * With own_rows > 0 a fifth item says whether the rows of a step of up to that many decode sequences and
 * no others own their slots (None for other steps).
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>
#include <stdlib.h>
#include <stdio.h>
#include <string.h>

static PyObject *s_token_ids, *s_num_computed, *s_num_new, *s_block_table, *s_params, *s_greedy;

/* An attribute of a scheduled sequence (a dataclass field, or any attribute of that name). */
static PyObject *field(PyObject *obj, PyObject *name) { return PyObject_GetAttr(obj, name); }

static int as_i64(PyObject *o, int64_t *out) {
  long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) return -1;
  *out = (int64_t)v;
  return 0;
}

/* Item i of a list (borrowed) or of another sequence (new reference, released by the caller). */
static PyObject *item(PyObject *seq, Py_ssize_t i, int *owned) {
  if (PyList_Check(seq)) {
    *owned = 0;
    return PyList_GET_ITEM(seq, i);
  }
  *owned = 1;
  return PySequence_GetItem(seq, i);
}

typedef struct {
  int64_t pos;
  int32_t idx;
} Row;

static int by_position(const void *a, const void *b) {
  const Row *x = (const Row *)a, *y = (const Row *)b;
  if (x->pos != y->pos) return x->pos > y->pos ? -1 : 1;  /* longest context first */
  return x->idx < y->idx ? -1 : (x->idx > y->idx);        /* ties in batch order (a stable sort) */
}

/* Whether n decode rows own their slots (see above); -1 without memory. A small open-addressing
 * table maps each row's last block to the row, so the check is one lookup per table entry (64 rows
 * of up to 24 entries: 2.5 us; 256 of up to 250: 65). Negative entries are read as block 0, and not
 * written. */
typedef struct {
  const int32_t *tab;
  int64_t ctx;
} DecRow;

static int own_slots(const DecRow *rows, int64_t n, int64_t bs) {
  uint32_t size = 16, mask;
  while ((int64_t)size < 4 * n) size <<= 1;
  mask = size - 1;
  int32_t *keys = (int32_t *)PyMem_Malloc(2 * (size_t)size * sizeof(int32_t));
  if (keys == NULL) return -1;
  int32_t *who = keys + size;
  memset(keys, 0xff, (size_t)size * sizeof(int32_t)); /* -1: no block */
  int own = 1;
  for (int64_t r = 0; r < n && own; ++r) {
    if (rows[r].ctx < 1) continue;
    const int32_t blk = rows[r].tab[(rows[r].ctx - 1) / bs];
    uint32_t h = ((uint32_t)blk * 2654435761u) & mask;
    while (blk >= 0 && keys[h] >= 0 && keys[h] != blk) h = (h + 1) & mask;
    if (blk < 0 || keys[h] == blk) own = 0; /* (two rows in one last block: the later one reads the earlier's slot) */
    keys[h] = blk;
    who[h] = (int32_t)r;
  }
  for (int64_t r = 0; r < n && own; ++r) {
    const int64_t ctx = rows[r].ctx, need = (ctx + bs - 1) / bs;
    for (int64_t e = 0; e < need; ++e) {
      const int32_t blk = rows[r].tab[e] < 0 ? 0 : rows[r].tab[e];
      uint32_t h = ((uint32_t)blk * 2654435761u) & mask;
      while (keys[h] >= 0 && keys[h] != blk) h = (h + 1) & mask;
      if (keys[h] != blk || (who[h] == r && e == need - 1)) continue;
      if (e * bs + (rows[who[h]].ctx - 1) % bs < ctx) {
        own = 0;
        break;
      }
    }
  }
  PyMem_Free(keys);
  return own;
}

static PyObject *rows_own_slots(PyObject *self, PyObject *args) {
  Py_buffer bt = {0}, bc = {0};
  long long bs_ll;
  if (!PyArg_ParseTuple(args, "y*y*L", &bt, &bc, &bs_ll)) return NULL;
  PyObject *result = NULL;
  DecRow *rows = NULL;
  const int64_t bs = bs_ll, n = (int64_t)(bc.len / sizeof(int32_t));
  const int64_t width = n ? (int64_t)(bt.len / sizeof(int32_t)) / n : 0;
  const int32_t *ctx = (const int32_t *)bc.buf;
  if (bs <= 0 || n * width * (int64_t)sizeof(int32_t) != (int64_t)bt.len) {
    PyErr_SetString(PyExc_ValueError, "rows_own_slots: a positive block_size and tables [rows, width]");
    goto done;
  }
  if ((rows = (DecRow *)PyMem_Malloc((n > 0 ? n : 1) * sizeof(DecRow))) == NULL) {
    PyErr_NoMemory();
    goto done;
  }
  for (int64_t r = 0; r < n; ++r) {
    rows[r].tab = (const int32_t *)bt.buf + r * width;
    rows[r].ctx = ctx[r];
    if (rows[r].ctx > width * bs) {
      PyErr_SetString(PyExc_ValueError, "rows_own_slots: a context is longer than its table row");
      goto done;
    }
  }
  const int own = own_slots(rows, n, bs);
  if (own < 0) PyErr_NoMemory();
  else result = PyBool_FromLong(own);
done:
  PyMem_Free(rows);
  PyBuffer_Release(&bt);
  PyBuffer_Release(&bc);
  return result;
}

typedef struct {
  PyObject *toks, *tab;  /* new references */
  int64_t pos;
  int64_t first;  /* offset of its table prefix in the packed values */
} Seq;

static PyObject *pack_decode(PyObject *self, PyObject *args) {
  PyObject *chunks;
  long long bs_ll, limit_ll, mb_ll;
  Py_buffer bi = {0}, bm = {0}, bt = {0};
  int check_own = 0;
  if (!PyArg_ParseTuple(args, "OLLw*w*w*L|p", &chunks, &bs_ll, &limit_ll, &bi, &bm, &bt, &mb_ll, &check_own)) return NULL;
  PyObject *result = NULL;
  PyObject *fast = NULL;
  Seq *seqs = NULL;
  Row *rows = NULL;
  Py_ssize_t b = 0, made = 0;
  const int64_t bs = bs_ll, limit = limit_ll, mb = mb_ll;
  if (bs <= 0 || mb <= 0) {
    PyErr_SetString(PyExc_ValueError, "pack_decode: block_size and max_blocks must be positive");
    goto done;
  }
  fast = PySequence_Fast(chunks, "pack_decode: chunks must be a sequence");
  if (fast == NULL) goto done;
  b = PySequence_Fast_GET_SIZE(fast);
  if (bi.len < (Py_ssize_t)(3 * b * sizeof(int64_t)) || bm.len < (Py_ssize_t)(2 * b * sizeof(int32_t)) ||
      bt.len < (Py_ssize_t)(b * mb * sizeof(int32_t))) {
    PyErr_SetString(PyExc_ValueError, "pack_decode: host buffers too small for the batch");
    goto done;
  }
  seqs = (Seq *)PyMem_Calloc(b > 0 ? b : 1, sizeof(Seq));
  rows = (Row *)PyMem_Malloc((b > 0 ? b : 1) * sizeof(Row));
  if (seqs == NULL || rows == NULL) {
    PyErr_NoMemory();
    goto done;
  }

  /* Pass 1: every condition and every value, nothing written. */
  int graphable = 1;
  for (Py_ssize_t i = 0; i < b && graphable; ++i) {
    PyObject *s = PySequence_Fast_GET_ITEM(fast, i);
    PyObject *v;
    int64_t num_new, p;
    if ((v = field(s, s_num_new)) == NULL) goto done;
    int rc = as_i64(v, &num_new);
    Py_DECREF(v);
    if (rc < 0) goto done;
    if ((v = field(s, s_num_computed)) == NULL) goto done;
    rc = as_i64(v, &p);
    Py_DECREF(v);
    if (rc < 0) goto done;
    PyObject *toks = field(s, s_token_ids);
    if (toks == NULL) goto done;
    seqs[i].toks = toks;
    made = i + 1;
    const Py_ssize_t ntok = PyObject_Length(toks);
    if (ntok < 0) goto done;
    if (num_new != 1 || p + 1 != (int64_t)ntok || p >= limit || p < 0) {
      graphable = 0;
      break;
    }
    if ((v = field(s, s_params)) == NULL) goto done;
    if (v != Py_None) {
      PyObject *g = PyObject_GetAttr(v, s_greedy);
      Py_DECREF(v);
      if (g == NULL) goto done;
      const int t = PyObject_IsTrue(g);
      Py_DECREF(g);
      if (t < 0) goto done;
      if (!t) {
        graphable = 0;
        break;
      }
    } else {
      Py_DECREF(v);
    }
    PyObject *tab = field(s, s_block_table);
    if (tab == NULL) goto done;
    seqs[i].tab = tab;
    seqs[i].pos = p;
  }
  if (!graphable) {
    result = PyLong_FromLong(-1);
    goto done;
  }
  int64_t total = 0;  /* table entries the contexts use */
  for (Py_ssize_t i = 0; i < b; ++i) {
    const int64_t need = (seqs[i].pos + bs) / bs;
    const Py_ssize_t ntab = PyObject_Length(seqs[i].tab);
    if (ntab < 0) goto done;
    if ((int64_t)ntab < need) {
      PyErr_Format(PyExc_RuntimeError, "block table of %zd blocks is shorter than context %lld", ntab,
                   (long long)(seqs[i].pos + 1));
      goto done;
    }
    if (need > mb) {
      PyErr_Format(PyExc_ValueError, "context %lld needs %lld table entries; the graph holds %lld",
                   (long long)(seqs[i].pos + 1), (long long)need, (long long)mb);
      goto done;
    }
    rows[i].pos = seqs[i].pos;
    rows[i].idx = (int32_t)i;
    seqs[i].first = total;
    total += need;
  }
  /* Values checked before the first write: ids, slots and the table prefixes (int32, packed in
   * vals for the compare-and-write below). */
  int64_t *hi = (int64_t *)bi.buf;
  int32_t *hm = (int32_t *)bm.buf, *ht = (int32_t *)bt.buf;
  int64_t *ids = (int64_t *)PyMem_Malloc((b > 0 ? 2 * b : 1) * sizeof(int64_t));
  int32_t *vals = (int32_t *)PyMem_Malloc((total > 0 ? total : 1) * sizeof(int32_t));
  if (ids == NULL || vals == NULL) {
    PyErr_NoMemory();
    goto fail_ids;
  }
  int64_t *slots = ids + b;
  for (Py_ssize_t i = 0; i < b; ++i) {
    const int64_t p = seqs[i].pos, need = (p + bs) / bs;
    int owned;
    PyObject *t = item(seqs[i].toks, (Py_ssize_t)p, &owned);
    if (t == NULL) goto fail_ids;
    int rc = as_i64(t, &ids[i]);
    if (owned) Py_DECREF(t);
    if (rc < 0) goto fail_ids;
    int32_t *vrow = vals + seqs[i].first;
    for (int64_t e = 0; e < need; ++e) {
      PyObject *x = item(seqs[i].tab, (Py_ssize_t)e, &owned);
      if (x == NULL) goto fail_ids;
      int overflow;
      const long long v = PyLong_AsLongLongAndOverflow(x, &overflow);
      if (owned) Py_DECREF(x);
      if (v == -1 && PyErr_Occurred()) goto fail_ids;
      if (overflow || v < INT32_MIN || v > INT32_MAX) {
        PyErr_SetString(PyExc_OverflowError, "block id out of int32 range");
        goto fail_ids;
      }
      vrow[e] = (int32_t)v;
    }
    slots[i] = (int64_t)vrow[p / bs] * bs + p % bs;
  }
  if (check_own) {
    DecRow *dr = (DecRow *)PyMem_Malloc((b > 0 ? b : 1) * sizeof(DecRow));
    for (Py_ssize_t i = 0; dr != NULL && i < b; ++i) {
      dr[i].tab = vals + seqs[i].first;
      dr[i].ctx = seqs[i].pos + 1;
    }
    const int own = dr != NULL ? own_slots(dr, b, bs) : -1;
    PyMem_Free(dr);
    if (own < 0) PyErr_NoMemory();
    else if (!own) result = PyLong_FromLong(-1);
    if (own <= 0) goto fail_ids;
  }

  /* Pass 2: the writes. */
  qsort(rows, (size_t)b, sizeof(Row), by_position);
  for (Py_ssize_t i = 0; i < b; ++i) {
    hi[i] = ids[i];
    hi[b + i] = seqs[i].pos;
    hi[2 * b + i] = slots[i];
  }
  int changed = 0;
  for (Py_ssize_t r = 0; r < b; ++r) {
    const Py_ssize_t i = rows[r].idx;
    const int64_t need = (seqs[i].pos + bs) / bs;
    hm[r] = (int32_t)i;
    hm[b + r] = (int32_t)(seqs[i].pos + 1);
    const int32_t *src = vals + seqs[i].first;
    if (memcmp(ht + r * mb, src, (size_t)need * sizeof(int32_t)) != 0) {
      memcpy(ht + r * mb, src, (size_t)need * sizeof(int32_t));
      changed = 1;
    }
  }
  PyMem_Free(vals);
  PyMem_Free(ids);
  result = PyLong_FromLong(changed);
  goto done;
fail_ids:
  PyMem_Free(ids);
  PyMem_Free(vals);
done:
  if (seqs != NULL) {
    for (Py_ssize_t i = 0; i < made; ++i) {
      Py_XDECREF(seqs[i].toks);
      Py_XDECREF(seqs[i].tab);
    }
    PyMem_Free(seqs);
  }
  PyMem_Free(rows);
  Py_XDECREF(fast);
  PyBuffer_Release(&bi);
  PyBuffer_Release(&bm);
  PyBuffer_Release(&bt);
  return result;
}

/* ---- pack_step ---------------------------------------------------------------------------- */

typedef struct {
  PyObject *toks, *tab; /* new references */
  int64_t start, n, ntok, flat;
} Chunk;

typedef struct {
  int64_t key;
  int32_t idx;
} Keyed;

static int by_key_desc(const void *a, const void *b) {
  const Keyed *x = (const Keyed *)a, *y = (const Keyed *)b;
  if (x->key != y->key) return x->key > y->key ? -1 : 1;
  return x->idx < y->idx ? -1 : (x->idx > y->idx);
}

static int table_entry(PyObject *tab, int64_t e, int32_t *out) {
  int owned;
  PyObject *x = item(tab, (Py_ssize_t)e, &owned);
  if (x == NULL) return -1;
  int overflow;
  const long long v = PyLong_AsLongLongAndOverflow(x, &overflow);
  if (owned) Py_DECREF(x);
  if (v == -1 && PyErr_Occurred()) return -1;
  if (overflow || v < INT32_MIN || v > INT32_MAX) {
    PyErr_SetString(PyExc_OverflowError, "block id out of int32 range");
    return -1;
  }
  *out = (int32_t)v;
  return 0;
}

/* Rows of padded tables: row r = the first need[r] entries of chunk list[r]'s table, then zeros. */
static int fill_tables(const Chunk *c, const Py_ssize_t *list, Py_ssize_t rows, int64_t bs, int64_t nb, int32_t *dst) {
  for (Py_ssize_t r = 0; r < rows; ++r) {
    const Chunk *k = &c[list[r]];
    const int64_t need = (k->start + k->n + bs - 1) / bs;
    int32_t *row = dst + r * nb;
    for (int64_t e = 0; e < need; ++e)
      if (table_entry(k->tab, e, &row[e]) < 0) return -1;
    for (int64_t e = need; e < nb; ++e) row[e] = 0;
  }
  return 0;
}

static PyObject *shape1(Py_ssize_t a) { return Py_BuildValue("(n)", a); }
static PyObject *shape2(Py_ssize_t a, Py_ssize_t b) { return Py_BuildValue("(nn)", a, b); }

static PyObject *pack_step(PyObject *self, PyObject *args) {
  PyObject *chunks, *tiles_obj;
  long long bs_ll;
  long long own_rows = 0;
  int own = -1; /* not looked at */
  if (!PyArg_ParseTuple(args, "OLO|L", &chunks, &bs_ll, &tiles_obj, &own_rows)) return NULL;
  const int64_t bs = bs_ll;
  PyObject *result = NULL, *fast = NULL, *tiles = NULL, *data = NULL, *sample = NULL, *layout = NULL;
  Chunk *c = NULL;
  Py_ssize_t *dec = NULL, *pre = NULL, made = 0;
  Keyed *work = NULL;
  int32_t *wseq = NULL;
  int64_t *wtile = NULL;
  if (bs <= 0) {
    PyErr_SetString(PyExc_ValueError, "pack_step: block_size must be positive");
    goto done;
  }
  if ((fast = PySequence_Fast(chunks, "pack_step: chunks must be a sequence")) == NULL) goto done;
  if ((tiles = PySequence_Fast(tiles_obj, "pack_step: tiles must be a sequence")) == NULL) goto done;
  const Py_ssize_t b = PySequence_Fast_GET_SIZE(fast), ntiles = PySequence_Fast_GET_SIZE(tiles);
  c = (Chunk *)PyMem_Calloc(b > 0 ? b : 1, sizeof(Chunk));
  dec = (Py_ssize_t *)PyMem_Malloc((b > 0 ? b : 1) * sizeof(Py_ssize_t));
  pre = (Py_ssize_t *)PyMem_Malloc((b > 0 ? b : 1) * sizeof(Py_ssize_t));
  wtile = (int64_t *)PyMem_Malloc((ntiles > 0 ? ntiles : 1) * sizeof(int64_t));
  if (c == NULL || dec == NULL || pre == NULL || wtile == NULL) {
    PyErr_NoMemory();
    goto done;
  }
  for (Py_ssize_t t = 0; t < ntiles; ++t) {
    if (as_i64(PySequence_Fast_GET_ITEM(tiles, t), &wtile[t]) < 0) goto done;
    if (wtile[t] <= 0) {
      PyErr_SetString(PyExc_ValueError, "pack_step: tile sizes must be positive");
      goto done;
    }
  }

  /* Pass 1: fields, checks, sizes. */
  int64_t total = 0, nrows = 0, nb_d = 0, nb_p = 0;
  Py_ssize_t ndec = 0, npre = 0;
  for (Py_ssize_t i = 0; i < b; ++i) {
    PyObject *s = PySequence_Fast_GET_ITEM(fast, i), *v;
    Chunk *k = &c[i];
    if ((v = field(s, s_num_new)) == NULL) goto done;
    int rc = as_i64(v, &k->n);
    Py_DECREF(v);
    if (rc < 0) goto done;
    if ((v = field(s, s_num_computed)) == NULL) goto done;
    rc = as_i64(v, &k->start);
    Py_DECREF(v);
    if (rc < 0) goto done;
    if ((k->toks = field(s, s_token_ids)) == NULL) goto done;
    made = i + 1;
    if ((k->tab = field(s, s_block_table)) == NULL) goto done;
    const Py_ssize_t ntok = PyObject_Length(k->toks);
    if (ntok < 0) goto done;
    k->ntok = ntok;
    if (k->n < 0 || k->start < 0 || k->start + k->n > k->ntok) {
      PyErr_Format(PyExc_ValueError, "sequence %zd schedules tokens [%lld, %lld) of %lld", i, (long long)k->start,
                   (long long)(k->start + k->n), (long long)k->ntok);
      goto done;
    }
    k->flat = total;
    total += k->n;
    if (k->start + k->n == k->ntok) ++nrows;
    if (k->n >= 1) {
      const int64_t need = (k->start + k->n + bs - 1) / bs;
      const Py_ssize_t ntab = PyObject_Length(k->tab);
      if (ntab < 0) goto done;
      if ((int64_t)ntab < need) {
        PyErr_Format(PyExc_RuntimeError, "block table of %zd blocks is shorter than context %lld", ntab,
                     (long long)(k->start + k->n));
        goto done;
      }
      if (k->n == 1) {
        dec[ndec++] = i;
        if (need > nb_d) nb_d = need;
      } else {
        pre[npre++] = i;
        if (need > nb_p) nb_p = need;
      }
    }
    if (total > INT32_MAX || k->start + k->n > INT32_MAX) {
      PyErr_SetString(PyExc_OverflowError, "pack_step: token counts past int32");
      goto done;
    }
  }
  /* Decode rows longest context first, ties in batch order. */
  {
    Keyed *kd = (Keyed *)PyMem_Malloc((ndec > 0 ? ndec : 1) * sizeof(Keyed));
    if (kd == NULL) {
      PyErr_NoMemory();
      goto done;
    }
    for (Py_ssize_t r = 0; r < ndec; ++r) {
      kd[r].key = c[dec[r]].start + 1;
      kd[r].idx = (int32_t)dec[r];
    }
    qsort(kd, (size_t)ndec, sizeof(Keyed), by_key_desc);
    for (Py_ssize_t r = 0; r < ndec; ++r) dec[r] = kd[r].idx;
    PyMem_Free(kd);
  }
  /* Work items per tile size. */
  int64_t nwork = 0;
  for (Py_ssize_t t = 0; t < ntiles; ++t)
    for (Py_ssize_t r = 0; r < npre; ++r) nwork += (c[pre[r]].n + wtile[t] - 1) / wtile[t];
  const int64_t n32 = (ndec ? 2 * ndec + ndec * nb_d : 0) + (npre ? 3 * npre + npre * nb_p + 2 * nwork : 0);
  const int64_t n64 = 3 * total + nrows;
  if ((data = PyByteArray_FromStringAndSize(NULL, (Py_ssize_t)(8 * n64 + 4 * n32))) == NULL) goto done;
  char *base = PyByteArray_AS_STRING(data);
  int64_t *ids = (int64_t *)base, *pos = ids + total, *slots = pos + total, *rows = slots + total;
  int32_t *m32 = (int32_t *)(base + 8 * n64);
  if ((sample = PyList_New(0)) == NULL || (layout = PyList_New(0)) == NULL) goto done;

  /* Pass 2: the flat batch. */
  int64_t rr = 0;
  for (Py_ssize_t i = 0; i < b; ++i) {
    const Chunk *k = &c[i];
    if (k->n >= 1) {
      int32_t blk = 0;
      int64_t cur_block = -1;
      for (int64_t t = 0; t < k->n; ++t) {
        const int64_t p = k->start + t;
        int owned;
        PyObject *x = item(k->toks, (Py_ssize_t)p, &owned);
        if (x == NULL) goto done;
        const int rc = as_i64(x, &ids[k->flat + t]);
        if (owned) Py_DECREF(x);
        if (rc < 0) goto done;
        pos[k->flat + t] = p;
        if (p / bs != cur_block) {
          cur_block = p / bs;
          if (table_entry(k->tab, cur_block, &blk) < 0) goto done;
        }
        slots[k->flat + t] = (int64_t)blk * bs + p % bs;
      }
    }
    if (k->start + k->n == k->ntok) {
      PyObject *ix = PyLong_FromSsize_t(i);
      if (ix == NULL || PyList_Append(sample, ix) < 0) {
        Py_XDECREF(ix);
        goto done;
      }
      Py_DECREF(ix);
      rows[rr++] = k->flat + k->n - 1;
    }
  }

  /* Pass 3: the plan parts. */
#define ADD_PART(name, shape)                                            \
  do {                                                                   \
    PyObject *sh_ = (shape);                                             \
    PyObject *ent_ = sh_ ? Py_BuildValue("(sN)", (name), sh_) : NULL;    \
    if (ent_ == NULL || PyList_Append(layout, ent_) < 0) {               \
      Py_XDECREF(ent_);                                                  \
      goto done;                                                         \
    }                                                                    \
    Py_DECREF(ent_);                                                     \
  } while (0)
  int32_t *w32 = m32;
  if (ndec) {
    for (Py_ssize_t r = 0; r < ndec; ++r) w32[r] = (int32_t)c[dec[r]].flat;
    ADD_PART("d_rows", shape1(ndec));
    w32 += ndec;
    for (Py_ssize_t r = 0; r < ndec; ++r) w32[r] = (int32_t)(c[dec[r]].start + 1);
    ADD_PART("d_ctx", shape1(ndec));
    w32 += ndec;
    if (fill_tables(c, dec, ndec, bs, nb_d, w32) < 0) goto done;
    ADD_PART("d_tables", shape2(ndec, (Py_ssize_t)nb_d));
    if (npre == 0 && ndec <= own_rows) {
      DecRow *dr = (DecRow *)PyMem_Malloc((size_t)ndec * sizeof(DecRow));
      for (Py_ssize_t r = 0; dr != NULL && r < ndec; ++r) {
        dr[r].tab = w32 + r * nb_d;
        dr[r].ctx = c[dec[r]].start + 1;
      }
      own = dr != NULL ? own_slots(dr, ndec, bs) : -1;
      PyMem_Free(dr);
      if (own < 0) {
        PyErr_NoMemory();
        goto done;
      }
    }
    w32 += ndec * nb_d;
  }
  if (npre) {
    for (Py_ssize_t r = 0; r < npre; ++r) {
      const Chunk *k = &c[pre[r]];
      w32[3 * r] = (int32_t)k->flat;
      w32[3 * r + 1] = (int32_t)k->n;
      w32[3 * r + 2] = (int32_t)k->start;
    }
    ADD_PART("p_info", shape2(npre, 3));
    w32 += 3 * npre;
    if (fill_tables(c, pre, npre, bs, nb_p, w32) < 0) goto done;
    ADD_PART("p_tables", shape2(npre, (Py_ssize_t)nb_p));
    w32 += npre * nb_p;
    int64_t most = 0;
    for (Py_ssize_t t = 0; t < ntiles; ++t) {
      int64_t w = 0;
      for (Py_ssize_t r = 0; r < npre; ++r) w += (c[pre[r]].n + wtile[t] - 1) / wtile[t];
      if (w > most) most = w;
    }
    work = (Keyed *)PyMem_Malloc((most > 0 ? most : 1) * sizeof(Keyed));
    wseq = (int32_t *)PyMem_Malloc((most > 0 ? most : 1) * 2 * sizeof(int32_t));
    if (work == NULL || wseq == NULL) {
      PyErr_NoMemory();
      goto done;
    }
    for (Py_ssize_t t = 0; t < ntiles; ++t) {
      const int64_t tile = wtile[t];
      int64_t w = 0;
      for (Py_ssize_t r = 0; r < npre; ++r) {
        const Chunk *k = &c[pre[r]];
        for (int64_t t0 = 0; t0 < k->n; t0 += tile) {
          const int64_t end = t0 + tile < k->n ? t0 + tile : k->n;
          work[w].key = k->start + end; /* cached keys + the causal keys of the tile's last token */
          work[w].idx = (int32_t)w;
          wseq[2 * w] = (int32_t)r;
          wseq[2 * w + 1] = (int32_t)t0;
          ++w;
        }
      }
      qsort(work, (size_t)w, sizeof(Keyed), by_key_desc);
      for (int64_t q = 0; q < w; ++q) {
        w32[2 * q] = wseq[2 * work[q].idx];
        w32[2 * q + 1] = wseq[2 * work[q].idx + 1];
      }
      char name[32];
      snprintf(name, sizeof name, "p_work%lld", (long long)tile);
      ADD_PART(name, shape2((Py_ssize_t)w, 2));
      w32 += 2 * w;
    }
  }
#undef ADD_PART
  result = own_rows > 0 ? Py_BuildValue("(OLOOO)", data, (long long)total, sample, layout,
                                        own < 0 ? Py_None : own ? Py_True : Py_False)
                        : Py_BuildValue("(OLOO)", data, (long long)total, sample, layout);
done:
  if (c != NULL) {
    for (Py_ssize_t i = 0; i < made; ++i) {
      Py_XDECREF(c[i].toks);
      Py_XDECREF(c[i].tab);
    }
    PyMem_Free(c);
  }
  PyMem_Free(dec);
  PyMem_Free(pre);
  PyMem_Free(work);
  PyMem_Free(wseq);
  PyMem_Free(wtile);
  Py_XDECREF(fast);
  Py_XDECREF(tiles);
  Py_XDECREF(data);
  Py_XDECREF(sample);
  Py_XDECREF(layout);
  return result;
}

static PyMethodDef methods[] = {
    {"pack_decode", pack_decode, METH_VARARGS,
     "pack_decode(chunks, block_size, limit, host_i64, host_meta, host_tables, max_blocks, own_slots=False) -> -1 | 0 | 1"},
    {"pack_step", pack_step, METH_VARARGS,
     "pack_step(chunks, block_size, tiles, own_rows=0) -> (data, total, sample_idx, layout[, own])"},
    {"rows_own_slots", rows_own_slots, METH_VARARGS, "rows_own_slots(tables, context_lens, block_size) -> bool"},
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_hostprep", "Decode-step input packing.", -1, methods};

PyMODINIT_FUNC PyInit__hostprep(void) {
  s_token_ids = PyUnicode_InternFromString("token_ids");
  s_num_computed = PyUnicode_InternFromString("num_computed");
  s_num_new = PyUnicode_InternFromString("num_new");
  s_block_table = PyUnicode_InternFromString("block_table");
  s_params = PyUnicode_InternFromString("params");
  s_greedy = PyUnicode_InternFromString("greedy");
  if (!s_token_ids || !s_num_computed || !s_num_new || !s_block_table || !s_params || !s_greedy) return NULL;
  return PyModule_Create(&module);
}
