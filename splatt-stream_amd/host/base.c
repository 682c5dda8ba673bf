/*
 * base.c -- allocation, versions, error mapping, RNG helpers.
 */
#include "host.h"
#include <errno.h>
#include <pthread.h>
#include <stdlib.h>
#include <string.h>

/* src/base.c:42-67: 64-byte aligned allocation, NULL (with a message) on
 * failure. */
void * splatt_malloc(size_t const bytes)
{
  void * ptr = NULL;
  int const rc = posix_memalign(&ptr, 64, bytes ? bytes : 64);
  if(rc != 0) {
    fprintf(stderr, "SPLATT: posix_memalign() of %zu bytes failed (%s).\n",
        bytes, rc == ENOMEM ? "ENOMEM" : "EINVAL");
    return NULL;
  }
  return ptr;
}

void splatt_free(void * ptr)
{
  free(ptr);
}

/* src/mpi_dummy.c:15-34: the non-MPI communicator is rank 0 of 1. */
splatt_comm_info * splatt_alloc_comm_info(void)
{
  splatt_comm_info * ci = (splatt_comm_info *) splatt_malloc(sizeof(*ci));
  if(ci == NULL) {
    return NULL;
  }
  ci->world_rank = 0;
  ci->world_npes = 1;
  return ci;
}

void splatt_free_comm_info(splatt_comm_info * comm_info)
{
  if(comm_info == NULL) {
    return;
  }
  splatt_free(comm_info);
}

int splatt_version_major(void) { return SPLATT_VER_MAJOR; }
int splatt_version_minor(void) { return SPLATT_VER_MINOR; }
int splatt_version_subminor(void) { return SPLATT_VER_SUBMINOR; }

splatt_error_type spl_report(int rc, char const * what)
{
  if(rc == SPD_OK) {
    return SPLATT_SUCCESS;
  }
  fprintf(stderr, "SPLATT: %s failed: %s\n", what, spd_last_error());
  if(rc == SPD_ENOMEM) {
    return SPLATT_ERROR_NOMEMORY;
  }
  return SPLATT_ERROR_BADINPUT;
}

char const * splatt_amd_last_error(void)
{
  return spd_last_error();
}

static int g_mttkrp_dtype = SPD_F64;

int spl_mttkrp_dtype(void) { return g_mttkrp_dtype; }

splatt_error_type splatt_amd_set_mttkrp_precision(int precision)
{
  if(precision != SPLATT_AMD_F64 && precision != SPLATT_AMD_F32) {
    return SPLATT_ERROR_BADINPUT;
  }
  g_mttkrp_dtype = (precision == SPLATT_AMD_F32) ? SPD_F32 : SPD_F64;
  return SPLATT_SUCCESS;
}

splatt_error_type splatt_amd_set_mttkrp_layout(int layout)
{
  if(layout != SPLATT_AMD_LAYOUT_AUTO && layout != SPLATT_AMD_LAYOUT_CSF) {
    return SPLATT_ERROR_BADINPUT;
  }
  spd_mttkrp_set_copies(layout == SPLATT_AMD_LAYOUT_AUTO);
  return SPLATT_SUCCESS;
}

/* src/util.c:15-24: magnitude 3*rand()/RAND_MAX, negated when a second
 * rand() is even. Drawn on the host so the sequence is glibc's. */
static val_t rand_value(int32_t a, int32_t b)
{
  val_t const v = 3.0 * ((val_t) a / (val_t) RAND_MAX);
  return (b % 2 == 0) ? -v : v;
}

val_t spl_rand_val(void)
{
  int32_t const a = rand();
  return rand_value(a, rand());
}

/* n values from a glibc generator state, two draws each (as spl_rand_val).
 * The draws are those of random_r: for the additive feedback generator
 * (TYPE_3, a 128-byte state, what rand() starts with) the step is inlined
 * here with the two state pointers in registers; other types call it. */
void spl_fill_rand_state(struct random_data * rd, double * vals, uint64_t n)
{
  if(rd->rand_type != 3) {
    for(uint64_t i=0; i < n; ++i) {
      int32_t a = 0, b = 0;
      random_r(rd, &a);
      random_r(rd, &b);
      vals[i] = rand_value(a, b);
    }
    return;
  }
  int32_t * fptr = rd->fptr;
  int32_t * rptr = rd->rptr;
  int32_t * const state = rd->state;
  int32_t * const end = rd->end_ptr;
  for(uint64_t i=0; i < n; ++i) {
    uint32_t draw[2];
    for(int k=0; k < 2; ++k) {
      uint32_t const val = (uint32_t) *fptr + (uint32_t) *rptr;
      *fptr = (int32_t) val;
      if(++fptr >= end) {
        fptr = state;
      }
      if(++rptr >= end) {
        rptr = state;
      }
      draw[k] = val >> 1;
    }
    /* negative when the second draw is even, without a branch on it */
    double const sign = (double) ((int32_t) ((draw[1] & 1u) << 1) - 1);
    vals[i] = sign * (3.0 * ((double) draw[0] / (double) RAND_MAX));
  }
  rd->fptr = fptr;
  rd->rptr = rptr;
}

/* One user of the process's generator at a time inside the library: the fills
 * below, and the runtime's start-up, which runs beside it (spd_init). */
static pthread_mutex_t rand_mu = PTHREAD_MUTEX_INITIALIZER;
void spl_rand_lock(void)
{
  pthread_mutex_lock(&rand_mu);
}
void spl_rand_unlock(void)
{
  pthread_mutex_unlock(&rand_mu);
}

#define RAND_WORDS 32     /* the TYPE_3 state: a position and 31 words */
#define RAND_BYTES (RAND_WORDS * sizeof(int32_t))
#define RAND_PROBE 256    /* values a long fill draws with rand() first */
#define RAND_LONG 2048    /* the shortest long fill */

/* True if n successive rand() results of this thread are neighbours in one
 * TYPE_3 sequence: o[i] = o[i-3] + o[i-31], but for a carry out of the lowest
 * bits, which results do not show. A draw of another thread breaks it. */
static int rand_undisturbed(uint32_t const * o, int n)
{
  for(int i=31; i < n; ++i) {
    if(((o[i] - o[i - 3] - o[i - 31]) & 0x7fffffffu) > 1u) {
      return 0;
    }
  }
  return 1;
}

/* Moves the generator from its current state `live` to `cur`, which is not in
 * use. A draw or a seed of another thread meanwhile changes `live`, which is
 * then made current again and moved anew. */
static void rand_move(int32_t * live, char * cur)
{
  int32_t sent[RAND_WORDS];
  for(;;) {
    memcpy(sent, live, RAND_BYTES);
    memcpy(cur, sent, RAND_BYTES);
    setstate(cur);
    if(memcmp(live, sent, RAND_BYTES) == 0) {
      return;
    }
    setstate((char *) live);
  }
}

/* A copy of the process's state, which is out of use while its bytes are
 * copied. 0 if another thread drew or seeded meanwhile (a seed is carried
 * over) or the state is of another type. */
static int rand_copy_state(int32_t * copy)
{
  static int32_t away[RAND_WORDS];     /* in use meanwhile */
  int32_t same[RAND_WORDS];
  struct random_data ra, rs, rc;
  memset(&ra, 0, sizeof(ra));
  memset(&rs, 0, sizeof(rs));
  memset(&rc, 0, sizeof(rc));
  initstate_r(1, (char *) away, RAND_BYTES, &ra);
  initstate_r(1, (char *) same, RAND_BYTES, &rs);
  initstate_r(1, (char *) copy, RAND_BYTES, &rc);
  char * const cur = setstate((char *) away);
  if(cur == NULL) {
    return 0;
  }
  int ok = setstate_r(cur, &rc) == 0 && rc.rand_type == 3;
  if(ok) {
    memcpy(copy, cur, RAND_BYTES);
  }
  setstate(cur);
  if(memcmp(away, same, RAND_BYTES) == 0) {
    return ok;
  }
  /* draws alone lead on from where `away` began; after a seed they do not,
   * and the seeded state is the process's */
  for(int k=0; k < 4096; ++k) {
    int32_t v;
    random_r(&rs, &v);
    if(memcmp(away + 1, same + 1, RAND_BYTES - sizeof(int32_t)) == 0) {
      return 0;
    }
  }
  if(ok) {
    setstate((char *) away);
    rand_move(away, cur);
  }
  return 0;
}

/* Makes `next` the process's state if that is still `seen`. */
static int rand_commit_state(int32_t const * seen, int32_t * next)
{
  char * const cur = setstate((char *) next);
  if(cur == NULL) {
    return 0;
  }
  /* the position comes first; no state array is shorter than the two words */
  if(memcmp(cur, seen, 2 * sizeof(int32_t)) != 0 || memcmp(cur, seen, RAND_BYTES) != 0) {
    setstate(cur);
    return 0;
  }
  rand_move(next, cur);
  return 1;
}

/* Values of the process's rand() sequence, which goes on after them. rand()
 * takes a lock and a call per draw (a stream that adds 90000 rows of rank 32
 * draws 6 million times: 113 ms against 12), so a long fill draws from a copy
 * of the generator's state and then moves the process's state on. The
 * process's state stays in place meanwhile, and another thread may draw from
 * it or seed it as beside a loop over rand(): if the first values show that
 * one does, or the process's next draw is not the copy's first any more, the
 * values are rand()'s. What is left are the two moments in which the state's
 * bytes are copied (about 0.1 us each): a draw of another thread that falls
 * into one may be out of sequence. */
void spl_fill_rand(val_t * vals, idx_t nelems)
{
  static int32_t copy[RAND_WORDS];
  idx_t done = 0;
  int ahead = 0;              /* a draw of the next value is already made */
  int32_t first = 0;
  spl_rand_lock();
  if(nelems >= RAND_LONG) {
    uint32_t o[2 * RAND_PROBE];
    for(; done < RAND_PROBE; ++done) {
      o[2 * done] = (uint32_t) rand();
      o[2 * done + 1] = (uint32_t) rand();
      vals[done] = rand_value((int32_t) o[2 * done], (int32_t) o[2 * done + 1]);
    }
    if(rand_undisturbed(o, 2 * RAND_PROBE) && rand_copy_state(copy)) {
      struct random_data rd, rs;
      int32_t own[RAND_WORDS], seen[RAND_WORDS];
      int32_t expect = 0;
      memset(&rd, 0, sizeof(rd));
      memset(&rs, 0, sizeof(rs));
      initstate_r(1, (char *) own, RAND_BYTES, &rd);
      memcpy(seen, copy, RAND_BYTES);
      setstate_r((char *) copy, &rd);
      spl_fill_rand_state(&rd, vals + done, nelems - done);
      setstate_r((char *) own, &rd);     /* stores the position in copy */
      initstate_r(1, (char *) own, RAND_BYTES, &rs);
      setstate_r((char *) seen, &rs);
      random_r(&rs, &expect);
      setstate_r((char *) own, &rs);
      first = rand();
      ahead = 1;
      if(first == expect && rand_commit_state(seen, copy)) {
        done = nelems;
        ahead = 0;
      }
    }
  }
  if(ahead) {
    vals[done++] = rand_value(first, rand());
  }
  for(; done < nelems; ++done) {
    vals[done] = spl_rand_val();
  }
  spl_rand_unlock();
}
