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
val_t spl_rand_val(void)
{
  val_t v = 3.0 * ((val_t) rand() / (val_t) RAND_MAX);
  if(rand() % 2 == 0) {
    v *= -1;
  }
  return v;
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
      double v = 3.0 * ((double) a / (double) RAND_MAX);
      vals[i] = (b % 2 == 0) ? -v : v;
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

/* Values of the process's rand() sequence, which goes on after them. rand()
 * itself takes a lock and a call per draw (a stream that adds 90000 rows of
 * rank 32 draws 6 million times: 113 ms against 10), so long fills run on the
 * generator's own state: a stand-in state is made current, which stores the
 * position of the caller's in its header, the draws are made from that, and
 * it is made current again. One fill at a time. */
void spl_fill_rand(val_t * vals, idx_t nelems)
{
  static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
  static char standin[128];
  static char own[128];
  idx_t done = 0;
  if(nelems >= 64) {
    pthread_mutex_lock(&mu);
    struct random_data rd;
    memset(&rd, 0, sizeof(rd));
    if(initstate_r(1, own, sizeof(own), &rd) == 0) {
      char * const cur = initstate(1, standin, sizeof(standin));
      if(cur != NULL) {
        if(setstate_r(cur, &rd) == 0) {
          spl_fill_rand_state(&rd, vals, nelems);
          done = nelems;
          /* stores the new position in cur's header */
          setstate_r(own, &rd);
        }
        setstate(cur);
      }
    }
    pthread_mutex_unlock(&mu);
  }
  for(idx_t i=done; i < nelems; ++i) {
    vals[i] = spl_rand_val();
  }
}
