"""Host work spread over threads (copies to the caller's memory) is done in
full however many threads the system grants.  A probe links the header against
a pthread_create that refuses after a number of calls."""
import os
import subprocess

import pytest

from conftest import ROOT

PROBE = r"""
#include <atomic>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <dlfcn.h>
#include <pthread.h>
#include "hegj_threads.h"
static int granted;
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x) {
    using F = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    if (granted-- <= 0) return EAGAIN;
    return ((F)dlsym(RTLD_NEXT, "pthread_create"))(t, a, f, x);
}
int main(int, char **v) {
    granted = atoi(v[1]);
    std::atomic<size_t> next{0}, done{0};
    hegj::run_on_threads(7, [&](size_t) {
        while (next++ < 1000) done++;
    });
    printf("%zu\n", done.load());
}
"""


@pytest.mark.parametrize("granted", [0, 1, 3, 100])
def test_work_is_done_however_few_threads_start(tmp_path, granted):
    src = tmp_path / "probe.cpp"
    src.write_text(PROBE)
    exe = str(tmp_path / "probe")
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "hegjoin_amd", "csrc"), str(src), "-o", exe,
                    "-ldl", "-lpthread"], check=True)
    r = subprocess.run([exe, str(granted)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "1000\n"
