/* Test shim between libphc.so and the HIP runtime: device allocations and
 * graph instantiations that fail on request (the call is refused here and
 * never reaches the runtime), and a record of the live device allocations and
 * of the graphs instantiated.
 * Loaded with RTLD_GLOBAL before libphc.so, so that its calls bind to it. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
#include <stdio.h>
#include <stdlib.h>

enum { OUT_OF_MEMORY = 2 }; /* hipErrorOutOfMemory */

static size_t fail_from = (size_t)-1; /* allocations of at least this many bytes fail */
static int fail_graphs;
static struct { void *p; size_t n; } live[4096];
static size_t peak_call, live_bytes; /* largest request since the last reset, bytes held */
static int refused, instantiated;

static void *real(const char *name)
{
    static void *rt;
    if (!rt) rt = dlopen("libamdhip64.so.7", RTLD_LAZY);
    void *f = rt ? dlsym(rt, name) : NULL;
    if (!f) {
        fprintf(stderr, "hip_faults: no %s in the HIP runtime\n", name);
        abort();
    }
    return f;
}

int hipMalloc(void **p, size_t n)
{
    static int (*f)(void **, size_t);
    if (!f) f = (int (*)(void **, size_t))real("hipMalloc");
    if (n > peak_call) peak_call = n;
    if (n >= fail_from) {
        ++refused;
        return OUT_OF_MEMORY;
    }
    const int st = f(p, n);
    for (size_t i = 0; st == 0 && i < sizeof(live) / sizeof(live[0]); ++i)
        if (!live[i].p) {
            live[i].p = *p;
            live[i].n = n;
            live_bytes += n;
            break;
        }
    return st;
}

int hipFree(void *p)
{
    static int (*f)(void *);
    if (!f) f = (int (*)(void *))real("hipFree");
    for (size_t i = 0; p && i < sizeof(live) / sizeof(live[0]); ++i)
        if (live[i].p == p) {
            live_bytes -= live[i].n;
            live[i].p = NULL;
            break;
        }
    return f(p);
}

int hipGraphInstantiate(void **exec, void *graph, void **node, char *log, size_t size)
{
    static int (*f)(void **, void *, void **, char *, size_t);
    if (!f) f = (int (*)(void **, void *, void **, char *, size_t))real("hipGraphInstantiate");
    if (fail_graphs) {
        ++refused;
        return OUT_OF_MEMORY;
    }
    ++instantiated;
    return f(exec, graph, node, log, size);
}

void hip_faults_set(size_t alloc_from, int refuse_graphs)
{
    fail_from = alloc_from;
    fail_graphs = refuse_graphs;
    refused = 0;
    instantiated = 0;
    peak_call = 0;
}
int hip_faults_graphs(void) { return instantiated; } /* since the last set */
int hip_faults_refused(void) { return refused; }
size_t hip_faults_peak(void) { return peak_call; }
size_t hip_faults_live(void) { return live_bytes; }
