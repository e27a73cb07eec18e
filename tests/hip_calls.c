/* Loaded before libsevc.so with its symbols global, this stands between that
 * library and the HIP runtime in a test's own process: it notes the calls that
 * tell which way the library went, and can refuse allocations. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
#include <stdio.h>
#include <stdlib.h>

enum { OUT_OF_MEMORY = 2, MOST = 1 << 16 };      /* hipErrorOutOfMemory */

static struct { int kind; void* what; } seen[MOST];
static int n_seen, refuse, more;

static void* real(const char* name) {
    static void* lib;
    if (!lib) lib = dlopen("libamdhip64.so.7", RTLD_NOW);
    void* f = lib ? dlsym(lib, name) : NULL;
    if (!f) {
        fprintf(stderr, "no %s: %s\n", name, dlerror());
        abort();
    }
    return f;
}

static void note(int kind, void* what) {
    if (n_seen < MOST) {
        seen[n_seen].kind = kind;
        seen[n_seen++].what = what;
    }
}

/* The n-th allocation from now on is refused, and the m that follow it. */
void calls_refuse(int n, int m) {
    refuse = n;
    more = m;
}
/* Whether a refusal is still to come. */
int calls_refuse_left(void) { return refuse; }

static int refused(void) {
    if (refuse == 0 || --refuse > 0) return 0;
    if (more > 0) {
        more--;
        refuse = 1;
    }
    return 1;
}

/* Forgets the calls so far; the number of calls; the k-th call. */
void calls_clear(void) { n_seen = 0; }
int calls_count(void) { return n_seen; }
int calls_kind(int k) { return seen[k].kind; }
void* calls_what(int k) { return seen[k].what; }

int hipMalloc(void** p, size_t n) {
    if (refused()) return OUT_OF_MEMORY;
    return ((int (*)(void**, size_t))real("hipMalloc"))(p, n);
}

int hipHostMalloc(void** p, size_t n, unsigned flags) {
    if (refused()) return OUT_OF_MEMORY;
    return ((int (*)(void**, size_t, unsigned))real("hipHostMalloc"))(p, n, flags);
}

int hipMemset(void* p, int v, size_t n) {
    note('M', p);
    return ((int (*)(void*, int, size_t))real("hipMemset"))(p, v, n);
}

int hipGraphLaunch(void* graph, void* stream) {
    note('G', graph);
    return ((int (*)(void*, void*))real("hipGraphLaunch"))(graph, stream);
}

int hipEventRecord(void* event, void* stream) {
    note('R', event);
    return ((int (*)(void*, void*))real("hipEventRecord"))(event, stream);
}

int hipEventSynchronize(void* event) {
    note('S', event);
    return ((int (*)(void*))real("hipEventSynchronize"))(event);
}
