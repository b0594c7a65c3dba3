"""The scratch registry (csrc/scratch.cpp) on the CPU: compiled with g++ against a stand-in for the HIP runtime whose allocations fail on demand."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STAND_IN = r"""
#pragma once
#include <stddef.h>
#include <stdlib.h>
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorStreamCaptureUnsupported = 900 };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone = 0 };
typedef struct ihipStream_t* hipStream_t;
extern size_t room, last_request; extern hipError_t last_error;
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { *s = hipStreamCaptureStatusNone; return hipSuccess; }
inline hipError_t hipMalloc(void** p, size_t n) { last_request = n; if (n > room) return last_error = hipErrorOutOfMemory; room -= n; *p = malloc(16); return hipSuccess; }
inline hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipFree(void* p) { free(p); return hipSuccess; }
inline hipError_t hipDeviceSynchronize() { return hipSuccess; }
inline hipError_t hipGetLastError() { const hipError_t e = last_error; last_error = hipSuccess; return e; }
"""
HEAD = r"""
#include <stdio.h>
#include <thread>
#include <vector>
#include "scratch.h"
size_t room, last_request; hipError_t last_error;
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
int main() { void* a = nullptr; void* b = nullptr; hipStream_t st = nullptr;
"""


def run(tmp_path, body, *flags):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STAND_IN)
    (tmp_path / "main.cpp").write_text(HEAD + body + "return 0; }")
    csrc = os.path.join(ROOT, "candle_vllm_amd", "csrc")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", *flags, "-I", str(tmp_path), "-I", csrc, os.path.join(csrc, "scratch.cpp"), str(tmp_path / "main.cpp"),
                        "-o", str(tmp_path / "t")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_a_failed_allocation_leaves_no_error_behind(tmp_path):
    """a caller that falls back launches kernels next and asks hipGetLastError about them: the failure of the allocation must not be there"""
    run(tmp_path, """
    room = 100;
    CHECK(mi355_scratch_get(&a, 7, 1000, st, false) != 0 && !a && last_error == hipSuccess);
    CHECK(mi355_scratch_get(&a, 7, 60, st, false) == 0 && a && last_request == 60 && last_error == hipSuccess);
    """)


def test_growth_doubles_up_to_the_most_and_takes_what_is_asked_where_that_is_all_there_is(tmp_path):
    run(tmp_path, """
    room = 10000;
    CHECK(mi355_scratch_get(&a, 7, 100, st, false, 1000) == 0 && last_request == 100);
    CHECK(mi355_scratch_get(&b, 7, 300, st, false, 1000) == 0 && last_request == 600 && a != b);
    CHECK(mi355_scratch_get(&a, 7, 700, st, false, 1000) == 0 && last_request == 1000);
    CHECK(mi355_scratch_get(&b, 7, 1000, st, false, 1000) == 0 && a == b);
    room = 1500;
    CHECK(mi355_scratch_get(&b, 7, 1200, st, false) == 0 && last_request == 1200 && a != b && last_error == hipSuccess);
    """)


def test_launches_of_two_threads_on_one_stream_take_turns(tmp_path):
    """what a thread enqueues inside a turn is not interleaved with another's (`queue` stands for the stream: a data race without the turn, which the thread
    sanitizer reports as well as the order does)"""
    run(tmp_path, """
    std::vector<int> queue;
    auto work = [&](int me) { for (int i = 0; i < 2000; ++i) { Mi355ScratchTurn turn(12, st); { Mi355ScratchTurn again(12, st); queue.push_back(me); } std::this_thread::yield(); queue.push_back(me); } };
    std::thread one(work, 1), two(work, 2);
    one.join(); two.join();
    CHECK(queue.size() == 8000);
    for (size_t i = 0; i < queue.size(); i += 2) CHECK(queue[i] == queue[i + 1]);
    """, "-fsanitize=thread")
