"""The workers that carry products to the host, where threads cannot be made: a
program whose pthread_create fails after the first few (0, 2, or never) still
takes every piece once and ends normally.  On the CPU, with the library's header."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "libmadam_amd", "csrc")

PROGRAM = r"""
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>

#include "madam_workers.hpp"

static std::atomic<int> allowed{0}, made{0};

extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *p)
{
    if (made.load() >= allowed.load()) return EAGAIN;
    ++made;
    using Create = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    return ((Create)dlsym(RTLD_NEXT, "pthread_create"))(t, a, f, p);
}

int main(int, char **argv)
{
    allowed = atoi(argv[1]);
    std::atomic<int> next{0}, sum{0}, workers{0};
    madam::run_workers(8, [&](int) {
        ++workers;
        for (int k = next++; k < 1000; k = next++) sum += k;
    });
    printf("%d %d %d\n", made.load(), workers.load(), sum.load());
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("workers")
    src, exe = d / "w.cpp", d / "w"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(src), "-o", str(exe), "-ldl"])
    return str(exe)


@pytest.mark.parametrize("allowed,threads", [(0, 0), (2, 2), (100, 7)])
def test_pieces_are_taken_with_the_threads_there_are(program, allowed, threads):
    r = subprocess.run([program, str(allowed)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    assert [int(x) for x in r.stdout.split()] == [threads, threads + 1, 499500]
