"""A machine whose large prompt passes' buffers do not fit is made all the same, and its prompts take passes of 64 rows: in
a process of its own, a hipMalloc in front of the runtime's reports one of those buffers as out of memory."""
from __future__ import annotations

import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SHIM = """
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
size_t shim_size = 0;
int shim_refused = 0;
int hipMalloc(void **p, size_t n) {
    static int (*real)(void **, size_t);
    if (!real) real = (int (*)(void **, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD), "hipMalloc");
    if (n == shim_size) { shim_refused++; return 2; }
    return real(p, n);
}
"""
SCRIPT = """
import ctypes, json, os, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import torch
torch.cuda.init()
sys.path.insert(0, sys.argv[2])
from conftest import load_sm
sm = load_sm()
out = []
for size in (0, 640 * 2304 * 8):                       # the qkv rows' 64-bit array, 640 rows for 599 positions
    ctypes.c_size_t.in_dll(shim, "shim_size").value = size
    m = sm.Machine(sys.argv[3], max_ctx=601, profile=True)
    m.kernels()
    words = m.stream(sm.prompt_ids(7, 300, 500), 3)
    out.append([words, any(n.startswith("prompt.") and c for n, (c, _) in m.kernels().items())])
    m.close()
print(json.dumps([ctypes.c_int.in_dll(shim, "shim_refused").value, out]))
"""


def test_refused(sm, tmp_path):
    d = sm.layout(sm.convert(sm.random_gpt2(seed=3, vocab=500, n_ctx=700)), str(tmp_path / "layout"))
    src, lib = str(tmp_path / "shim.c"), str(tmp_path / "shim.so")
    with open(src, "w") as f:
        f.write(SHIM)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", lib, src, "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-c", SCRIPT, lib, os.path.dirname(os.path.abspath(__file__)), d], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    refused, (free, short) = json.loads(r.stdout.strip().splitlines()[-1])
    assert refused == 1 and free[1] and not short[1]
    assert free[0] == short[0]
