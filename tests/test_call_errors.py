"""Calls that fail half way (a failure that a shim in front of the runtime makes up): a
batch's sweep between the launches of its groups, a network's gradient between its
copies.  The error comes back once what the call had already put on its streams has
ended, and other work goes on."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
typedef void* P;
static void* hip(const char* name) {
    void* lib = dlopen("libamdhip64.so.7", RTLD_NOW);
    return dlsym(lib, name);
}
static int fail_at = -1, n_call; /* the event record that fails, counted from 0 */
static int n_rec, n_syn;
static P rec[64], syn[64]; /* streams: given work after the fork; waited for */
void shim_arm(int k) { fail_at = k; n_call = n_rec = n_syn = 0; }
int shim_streams(void) { return n_rec; }
int shim_unwaited(void) {
    int n = 0;
    for (int i = 0; i < n_rec; i++) {
        int hit = 0;
        for (int j = 0; j < n_syn; j++) { hit |= syn[j] == rec[i]; }
        n += !hit;
    }
    return n;
}
int hipEventRecord(P ev, P st) {
    if (fail_at >= 0) {
        int k = n_call++;
        if (k > 0) { rec[n_rec++] = st; }
        if (k == fail_at) { fail_at = -1; return 999; }
    }
    return ((int (*)(P, P))hip("hipEventRecord"))(ev, st);
}
static int fail_copy = -1;
void shim_arm_copy(int k) { fail_copy = k; n_rec = n_syn = 0; }
int hipMemcpyAsync(P to, const void* from, size_t n, int kind, P st) {
    if (fail_copy >= 0) {
        rec[0] = st;
        n_rec = 1;
        n_syn = 0;
        if (fail_copy-- == 0) { return 999; }
    }
    return ((int (*)(P, const void*, size_t, int, P))hip("hipMemcpyAsync"))(to, from, n, kind, st);
}
int hipStreamSynchronize(P st) {
    if (n_syn < 64) { syn[n_syn++] = st; }
    return ((int (*)(P))hip("hipStreamSynchronize"))(st);
}
"""

BATCH = r"""
import ctypes as C, sys
shim = C.CDLL(sys.argv[1], C.RTLD_GLOBAL)
from latticednaorigami_amd import abi, systems
from latticednaorigami_amd.sampler import BatchSampler
ss, ts = systems.batch_systems(1600)
a, b = BatchSampler(ss, ts), BatchSampler(ss, ts)
for x in (a, b):
    x.set_kernel(abi.BATCH_LDS)
# event records of a sweep: the fork's, then one after each group on a side stream
shim.shim_arm(2)
try:
    a.sweep(50)
    print("no error")
except abi.LdoError as e:
    print("error", e.code, "streams", shim.shim_streams(), "unwaited", shim.shim_unwaited())
a.close()
b.sweep(50)
print("steps", *[b.observables(k, 1)[0]["step"] for k in (0, 1599)])
b.close()
"""


NETWORK = r"""
import ctypes as C, sys
import numpy as np
shim = C.CDLL(sys.argv[1], C.RTLD_GLOBAL)
import mlp_ref as M
from latticednaorigami_amd import abi
from latticednaorigami_amd.mlp import Mlp
net = Mlp(5, max_batch=40, seed=9)
batch = M.random_batch(np.random.default_rng(3), 33, 5)
first = net.loss_grad(*batch)
# copies of the call: the batch, the losses, the gradients
shim.shim_arm_copy(2)
try:
    net.loss_grad(*batch, want_grads=True)
    print("no error")
except abi.LdoError as e:
    print("error", e.code, "streams", shim.shim_streams(), "unwaited", shim.shim_unwaited())
print("again", net.loss_grad(*batch) == first)
"""


def run(tmp_path, script):
    src, shim = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(shim), str(src), "-ldl"], check=True)
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([ROOT, os.path.join(ROOT, "oracle")]))
    return subprocess.run([sys.executable, "-c", script, str(shim)], env=env, check=True,
                          timeout=100, capture_output=True, text=True).stdout.split("\n")


@pytest.mark.gpu
def test_failed_launch_waits_for_the_groups_before_it(tmp_path):
    print("case: batch of 1600 chains, a failure after its third group", flush=True)
    out = run(tmp_path, BATCH)
    words = out[0].split()
    assert words[0] == "error" and int(words[3]) == 2 and int(words[5]) == 0, out
    assert out[1] == "steps 50 50", out


@pytest.mark.gpu
def test_failed_copy_waits_for_the_copies_before_it(tmp_path):
    print("case: network gradient, a failure at its last copy", flush=True)
    out = run(tmp_path, NETWORK)
    words = out[0].split()
    assert words[0] == "error" and int(words[3]) == 1 and int(words[5]) == 0, out
    assert out[1] == "again True", out
