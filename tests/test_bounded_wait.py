"""The host's bounded wait (neus2_amd/csrc/bounded_wait.h), compiled with the host compiler and run on a clock of the test's own: no GPU needed."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WRAPPERS = """
#include "bounded_wait.h"
#include <cstdint>
struct Steps {  // every reading is `step` later than the one before
	typedef std::chrono::nanoseconds duration;
	typedef std::chrono::time_point<Steps, duration> time_point;
	static int64_t step, at;
	static time_point now() { return time_point(duration(at += step)); }
};
int64_t Steps::step, Steps::at;
extern "C" int poll(int64_t step_ns, int64_t most_ns, int64_t ready_at, int64_t* asked) {
	Steps::step = step_ns;
	Steps::at = 0;
	*asked = 0;
	return n2_poll<Steps>([&]() { return ++*asked >= ready_at; }, std::chrono::nanoseconds(most_ns));
}
"""


@pytest.fixture(scope="module")
def poll(tmp_path_factory):
    d = tmp_path_factory.mktemp("wait")
    src, so = d / "wait.cpp", d / "wait.so"
    src.write_text(WRAPPERS)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "neus2_amd", "csrc"),
                    str(src), "-o", str(so)], check=True, timeout=60)
    f = C.CDLL(str(so)).poll
    f.argtypes = [C.c_int64, C.c_int64, C.c_int64, C.POINTER(C.c_int64)]
    return f


@pytest.mark.parametrize("step_ns", [7, 100, 999_999, 1_000_000, 5_000_000])
def test_a_wait_is_bounded_by_time_and_not_by_questions(poll, step_ns):
    """However long a question takes: those that fit a millisecond, and at least one."""
    asked, most = C.c_int64(), 1_000_000
    questions = -(-most // step_ns)
    assert not poll(step_ns, most, 1 << 60, asked) and asked.value == questions
    for ready_at in {1, questions // 2 + 1, questions}:
        assert poll(step_ns, most, ready_at, asked) and asked.value == ready_at
    assert not poll(step_ns, most, questions + 1, asked)
