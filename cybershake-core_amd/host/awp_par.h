/*
 * awp_par.h -- a call split over a few host threads.  fn(arg, part, nparts)
 * runs once for every part 0..nparts-1 and must not depend on the others; a
 * thread that cannot be started has its part run by the caller.
 */
#ifndef AWP_PAR_H
#define AWP_PAR_H

#include <pthread.h>
#include <stddef.h>
#include <unistd.h>

#define AWP_PAR_MAX 8

typedef struct {
    void (*fn)(void *, int, int);
    void *arg;
    int part, nparts;
} awp_par_job;

static inline void *awp_par_main(void *p)
{
    awp_par_job *j = (awp_par_job *)p;
    j->fn(j->arg, j->part, j->nparts);
    return NULL;
}

/* threads worth starting for `bytes` of host copying or decoding: one per 2
 * MB (a start costs about 30 us, 2 MB about 200), at most AWP_PAR_MAX and the
 * CPUs online */
static inline int awp_par_threads(size_t bytes)
{
    const long cpus = sysconf(_SC_NPROCESSORS_ONLN);
    size_t n = bytes / ((size_t)2 << 20);
    if (n > AWP_PAR_MAX) n = AWP_PAR_MAX;
    if (cpus > 0 && n > (size_t)cpus) n = (size_t)cpus;
    return n < 1 ? 1 : (int)n;
}

static inline void awp_par(int nparts, void (*fn)(void *, int, int), void *arg)
{
    awp_par_job job[AWP_PAR_MAX];
    pthread_t tid[AWP_PAR_MAX];
    int started[AWP_PAR_MAX] = {0};
    if (nparts > AWP_PAR_MAX) nparts = AWP_PAR_MAX;
    for (int k = 1; k < nparts; ++k) {
        job[k].fn = fn;
        job[k].arg = arg;
        job[k].part = k;
        job[k].nparts = nparts;
        started[k] = pthread_create(&tid[k], NULL, awp_par_main, &job[k]) == 0;
    }
    fn(arg, 0, nparts);
    for (int k = 1; k < nparts; ++k) {
        if (started[k])
            pthread_join(tid[k], NULL);
        else
            fn(arg, k, nparts);
    }
}

#endif
