"""CPU: the CPython binding lets other threads run while the attention call launches
(its launches wait when the stream's queue is full).  The binding is built against
a stub library whose attention call waits for a word another Python thread sets."""

from __future__ import annotations

import ctypes
import importlib.util
import subprocess
import sysconfig
import threading
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

STUB = r"""
#include <chrono>
#include "treemoe_amd.h"
extern "C" {
int tm_op4_argmax_walk(const void*, int, int64_t, int64_t, int64_t, const int64_t*, const int32_t*,
                       const int32_t*, const int32_t*, int64_t, int64_t, int, int32_t*, int64_t*,
                       int64_t*, int64_t*, void*, void*) { return 0; }
int tm_op4_kv_commit(void*, void*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t,
                     const int64_t*, const int64_t*, const int32_t*, int64_t, const int32_t*,
                     int64_t, int64_t, int64_t, int64_t*, void*) { return 0; }
int tm_tree_attention_plan(int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t*,
                           int64_t*) { return 0; }
int tm_stream_capture_id(void*, uint64_t*) { return 0; }
// q: {entered, go}; 0 when `go` is set within two seconds, else 1
int tm_tree_attention(const void* q, int64_t, const void*, const void*, int64_t, void*, void*,
                      int64_t, int64_t, int64_t, const int32_t*, int64_t, int64_t, const int32_t*,
                      int64_t, int, const uint64_t*, int64_t, int64_t, int64_t, int64_t, float,
                      void*, int64_t, int64_t, void*, int64_t, void*) {
  volatile int64_t* w = (volatile int64_t*)q;
  w[0] = 1;
  const auto end = std::chrono::steady_clock::now() + std::chrono::seconds(2);
  while (!w[1])
    if (std::chrono::steady_clock::now() > end) return 1;
  return 0;
}
}
"""


def test_attention_call_releases_the_interpreter(tmp_path):
    (tmp_path / "stub.cpp").write_text(STUB)
    out = tmp_path / ("_tmfast" + sysconfig.get_config_var("EXT_SUFFIX"))
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", f"-I{ROOT / 'include'}",
                    f"-I{sysconfig.get_paths()['include']}", "-o", str(out),
                    str(ROOT / "treemoe_spec_amd" / "csrc" / "pyfast.cpp"),
                    str(tmp_path / "stub.cpp")], check=True)
    spec = importlib.util.spec_from_file_location("_tmfast", out)
    fast = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(fast)
    words = (ctypes.c_int64 * 2)()

    def answer():
        while not words[0]:
            pass
        words[1] = 1

    t = threading.Thread(target=answer)
    t.start()
    args = [ctypes.addressof(words)] + [0] * 27
    args[21] = 1.0
    rc = fast.tree_attention(*args)
    words[0] = 1
    t.join()
    assert rc == 0
