/*
 * fork.c -- sim.mem in forked children.
 *
 * The runtime keeps page-locked memory out of a forked child (VM_DONTFORK on
 * its mapping), so that a child which reads sim.mem, a worker of a pool or one
 * that writes a snapshot, would fault where ordinary memory serves it.  A fork
 * therefore copies the sim.mem of small systems and the child finds the copy at
 * the address, private as any other memory.  Larger ones, whose copy would cost
 * a fork more than 2 ms, stay in the parent alone.
 */
#define _GNU_SOURCE

#include <pthread.h>
#include <string.h>
#include <sys/mman.h>

#include "sf_host.h"

#define SF_FORK_MAX_BYTES 8388608u

static pthread_once_t g_once = PTHREAD_ONCE_INIT;
static struct {
	void *mem, *copy;
	size_t bytes;
} g_copy[SF_MAX_CTX];
static unsigned int g_copies;

static void add_copy(const sf_ctx* c) {
	const size_t bytes = sizeof(float) * (size_t)c->N * c->dof;
	if (!c->host_pinned_base || !bytes || bytes >= SF_FORK_MAX_BYTES) return;
	void* copy = mmap(NULL, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
	if (copy == MAP_FAILED) return;
	memcpy(copy, c->host_mem, bytes);
	g_copy[g_copies].mem = c->host_mem;
	g_copy[g_copies].copy = copy;
	g_copy[g_copies++].bytes = bytes;
}

static void before_fork(void) {
	g_copies = 0;
	sf_ctx_each(add_copy);
}

static void in_parent(void) {
	for (unsigned int k = 0; k < g_copies; ++k) munmap(g_copy[k].copy, g_copy[k].bytes);
	g_copies = 0;
}

static void in_child(void) {
	for (unsigned int k = 0; k < g_copies; ++k)
		mremap(g_copy[k].copy, g_copy[k].bytes, g_copy[k].bytes, MREMAP_MAYMOVE | MREMAP_FIXED, g_copy[k].mem);
	g_copies = 0;
}

static void install(void) { pthread_atfork(before_fork, in_parent, in_child); }

void sf_keep_in_children(void) { pthread_once(&g_once, install); }
