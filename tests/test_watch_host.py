"""The host's wait on a watched run (csrc/watch_wait.hpp), compiled for the CPU
with the stream replaced by a query that plays a sequence of events."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include "watch_wait.hpp"
// Query k finds states[k] (the last one from then on); just before it answers,
// the words become words[2 k], words[2 k + 1].
extern "C" int wait(int32_t begun, const int32_t *states, const int32_t *words, int32_t n,
                    int32_t *queries) {
  int32_t watch[2] = {0, 0};
  *queries = 0;
  const abm::Waited w = abm::wait_watch(watch, begun, [&] {
    const int k = *queries < n ? *queries : n - 1;
    watch[0] = words[2 * k];
    watch[1] = words[2 * k + 1];
    ++*queries;
    return (abm::StreamState)states[k];
  });
  return (int)w;
}
"""

RUNNING, IDLE, FAILED = range(3)
BEGUN, SETTLED, ERROR, SILENT = range(4)


@pytest.fixture(scope="module")
def wait(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("needs a host C++ compiler")
    d = tmp_path_factory.mktemp("watch")
    src, so = d / "wait.cpp", d / "wait.so"
    src.write_text(SOURCE)
    subprocess.run([cxx, "-std=c++17", "-O2", "-shared", "-fPIC", "-I",
                    os.path.join(REPO, "jaxabm_amd", "csrc"), str(src), "-o", str(so)], check=True)
    f = C.CDLL(str(so)).wait

    def call(begun, events):
        n = len(events)
        states = (C.c_int32 * n)(*[e[0] for e in events])
        words = (C.c_int32 * (2 * n))(*[v for e in events for v in e[1:]])
        queries = C.c_int32()
        return f(begun, states, words, n, C.byref(queries)), queries.value

    return call


@pytest.mark.parametrize("begun", [1, 9])
@pytest.mark.parametrize("events,want", [
    # the run settles between the host's reads and the answer that it is over: the
    # identity step tells the second word alone
    ([(IDLE, 0, 1)], SETTLED),
    ([(RUNNING, 0, 0), (IDLE, 0, 1)], SETTLED),
    # the awaited step begins, and the stream drains, in the same gap
    ([(IDLE, 9, 0)], BEGUN),
    ([(RUNNING, 9, 0)], BEGUN),
    ([(RUNNING, 0, 1)], SETTLED),
    # over without a word: not memory the device can write
    ([(RUNNING, 0, 0), (IDLE, 0, 0)], SILENT),
    ([(RUNNING, 0, 0), (FAILED, 0, 0)], ERROR),
])
def test_wait_ends_as_the_run_does(wait, begun, events, want):
    got, queries = wait(begun, events)
    assert got == want
    assert queries == len(events)
