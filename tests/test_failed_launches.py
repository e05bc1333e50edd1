"""Launches that fail, on the CPU: the library runs against a stand-in for the
HIP runtime (compiled here with gcc) that records every launch and copy and
lets a chosen launch fail, for every launch of a run in turn.

After a failed launch a sort must not go on (its later kernels would index
with tables that were not written), the next sort must clear what the failed
one left in its counters, the caller's planes and ids must be in the same
order, and the items of the failed run must not be used again.
"""
import ctypes
import importlib.util
import json
import os
import re
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

FAKE_HIP = r"""
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
typedef struct { unsigned x, y, z; } dim3_;
static struct { const void *f; const char *name; } fns[16384];
static int nfns, fail_at, count, last;
static char logbuf[1 << 20];
static size_t used;
static struct { dim3_ g, b; size_t sh; void *st; } cfg;
static void put(const char *s) { used += (size_t)snprintf(logbuf + used, sizeof(logbuf) - used, "%s\n", s); }
void fake_reset(int at, int error) { used = 0; logbuf[0] = 0; count = 0; fail_at = at; last = error; }
const char *fake_log(void) { return logbuf; }
void **__hipRegisterFatBinary(const void *d) { (void)d; return (void **)calloc(1, 8); }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *f, char *d, const char *name, unsigned t, void *a, void *b, void *c,
                           void *e, int *w) {
  (void)m; (void)d; (void)t; (void)a; (void)b; (void)c; (void)e; (void)w;
  if (nfns < 16384) { fns[nfns].f = f; fns[nfns++].name = strdup(name); }
}
void __hipRegisterVar(void **m, void *v, char *h, char *d, int e, size_t s, int c, int g) {
  (void)m; (void)v; (void)h; (void)d; (void)e; (void)s; (void)c; (void)g;
}
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t sh, void *st) {
  cfg.g = g; cfg.b = b; cfg.sh = sh; cfg.st = st;
  return 0;
}
int __hipPopCallConfiguration(dim3_ *g, dim3_ *b, size_t *sh, void **st) {
  *g = cfg.g; *b = cfg.b; *sh = cfg.sh; *st = cfg.st;
  return 0;
}
int hipLaunchKernel(const void *f, dim3_ g, dim3_ b, void **args, size_t sh, void *st) {
  (void)g; (void)b; (void)args; (void)sh; (void)st;
  const char *name = "?";
  for (int i = 0; i < nfns; ++i) if (fns[i].f == f) name = fns[i].name;
  if (++count == fail_at) { put("FAILED"); put(name); return last = 719; }
  put(name);
  return 0;
}
int hipGetLastError(void) { int e = last; last = 0; return e; }
const char *hipGetErrorString(int e) { (void)e; return "planted error"; }
int hipMemset(void *p, int v, size_t n) { memset(p, v, n); return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { (void)st; return hipMemcpy(d, s, n, k); }
int hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int k, void *st) {
  char t[64];
  (void)s; (void)sp; (void)dp; (void)w; (void)h; (void)k; (void)st;
  snprintf(t, sizeof(t), "copy to %p", d);
  put(t);
  return 0;
}
int hipDeviceSynchronize(void) { return 0; }
"""


def _child(fake):
    """Runs in a process of its own: prints the logs as JSON."""
    import numpy as np
    F = ctypes.CDLL(fake, mode=ctypes.RTLD_GLOBAL)
    F.fake_log.restype = ctypes.c_char_p
    # the binding alone: the package imports torch, whose own kernels need the real runtime
    spec = importlib.util.spec_from_file_location("_lib", os.path.join(ROOT, "autoquantizer_amd", "_lib.py"))
    _lib = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(_lib)
    L = _lib.lib()

    def log():
        return F.fake_log().decode().split("\n")[:-1]

    keep = []

    def buffer(nbytes):
        a = np.zeros(int(nbytes) + 512, np.uint8)
        keep.append(a)
        return (a.ctypes.data + 255) // 256 * 256

    def sim(dim, n, quant):
        d = _lib.SimDesc()
        d.dim, d.material, d.n_grid, d.bound, d.capacity = dim, _lib.AQ_FLUID, 72 if dim == 2 else 20, 3, n
        d.dx, d.inv_dx, d.dt, d.p_vol, d.p_mass, d.la = 1 / d.n_grid, d.n_grid, 1e-4, 1e-6, 1e-6, 1.0
        d.ncomp, d.storage = 2 * dim + dim * dim + 1, _lib.AQ_STORE_F32
        if quant:
            d.storage, d.nwords = _lib.AQ_STORE_QUANT, d.ncomp
            for c in range(d.ncomp):
                q = d.comps[c]
                q.kind, q.num_bits, q.is_signed, q.bit_offset, q.scale = _lib.AQ_FIXED, 20, 1, 64 * c, 1e-4
        h = ctypes.c_void_p()
        nb = L.aq_sim_workspace_bytes(ctypes.byref(d))
        _lib.check(L.aq_sim_create(ctypes.byref(d), buffer(nb), nb, ctypes.byref(h)))
        return h, buffer(8 * d.ncomp * n), buffer(4 * n), n

    out = {"advance": [], "group": []}

    def follow(sims, fail):
        """After the failed call: the route of a P2G, then of a sort."""
        r = {"fail": fail, "run": log(), "states": [hex(s[1]) for s in sims], "p2g": [], "sort": []}
        for h, state, ids, n in sims:
            F.fake_reset(0, 0)
            _lib.check(L.aq_p2g(h, state, n, None))
            r["p2g"].append(log())
            F.fake_reset(0, 0)
            _lib.check(L.aq_sort(h, state, n, ids, None))
            r["sort"].append(log())
        return r

    for at in range(0, 40):  # 0: no launch fails
        s = sim(2, 300, False)
        F.fake_reset(at, 0)
        rc = L.aq_advance(s[0], s[1], s[3], 4, 0, 2, s[2], None)
        r = follow([s], at)
        r["rc"] = rc
        out["advance"].append(r)
    for at in range(0, 60):
        ss = [sim(2, 300, True), sim(3, 700, True), sim(2, 20, True)]
        nb = L.aq_group_workspace_bytes(3)
        g = ctypes.c_void_p()
        V, I = ctypes.c_void_p * 3, ctypes.c_int64 * 3
        _lib.check(L.aq_group_create(V(*[x[0].value for x in ss]), V(*[x[1] for x in ss]), I(*[x[3] for x in ss]),
                                     V(*[x[2] for x in ss]), 3, buffer(nb), nb, ctypes.byref(g)))
        F.fake_reset(at, 0)
        rc = L.aq_group_advance(g, 4, 0, 2, 0, None)
        r = follow(ss, at)
        r["rc"] = rc
        out["group"].append(r)
        L.aq_group_destroy(g)
    s = sim(2, 300, False)
    F.fake_reset(0, 719)
    out["left"] = {"rc": L.aq_advance(s[0], s[1], s[3], 4, 0, 2, s[2], None), "run": log(),
                   "again": L.aq_advance(s[0], s[1], s[3], 4, 0, 2, s[2], None)}
    F.fake_reset(0, 719)
    out["left"]["sorted"] = L.aq_advance(s[0], s[1], s[3], 4, 0, 2, s[2], None)
    _lib.check(L.aq_p2g(s[0], s[1], s[3], None))
    out["left"]["p2g"] = log()
    print(json.dumps(out))


@pytest.fixture(scope="module")
def logs(tmp_path_factory):
    if shutil.which("gcc") is None:
        pytest.skip("gcc not available")
    d = tmp_path_factory.mktemp("fakehip")
    src, so = d / "fake_hip.c", d / "libfake_hip.so"
    src.write_text(FAKE_HIP)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(so), str(src)], check=True, timeout=120)
    r = subprocess.run([sys.executable, os.path.abspath(__file__), str(so)], capture_output=True, text=True,
                       timeout=600)
    assert r.returncode == 0, r.stderr[-3000:]
    return json.loads(r.stdout.splitlines()[-1])


SORTS = re.compile(r"k_(sort|group)_(keys|counts|count_scan|scan|scatter|finish)")
G2P = re.compile(r"k_tiledI.*?fLb1|k_tiled_groupILi\dELi\dELi\d+ELb1")


def _split(r):
    i = r["run"].index("FAILED")
    return r["run"][:i], r["run"][i + 1], r["run"][i + 2:]


@pytest.mark.parametrize("kind", ["advance", "group"])
def test_runs_reach_every_launch(logs, kind):
    """The sweep covers the whole run, and a run without a failed launch
    returns no error."""
    assert logs[kind][0]["rc"] == 0 and "FAILED" not in logs[kind][0]["run"]
    assert logs[kind][-1]["rc"] == 0  # past the last launch
    n = len(logs[kind][0]["run"])
    for r in logs[kind][1:]:
        assert ("FAILED" in r["run"]) == (r["rc"] < 0) == (r["fail"] <= n), r["fail"]


@pytest.mark.parametrize("kind", ["advance", "group"])
def test_failed_sort_stops_and_is_cleared(logs, kind):
    for r in logs[kind]:
        if r["rc"] == 0:
            continue
        before, failed, after = _split(r)
        if SORTS.search(failed):
            assert not any(SORTS.search(x) for x in after), (r["fail"], after)
        # counters of a sort that did not come to its end
        names = [m.group(2) for m in map(SORTS.search, before + [failed]) if m]
        open_sort = bool(SORTS.search(failed))
        assert names or not open_sort
        for k, s in enumerate(r["sort"]):
            first = ["k_fill_u32" in s[0], "k_fill_u32" in s[1]]
            assert first == [open_sort, open_sort], (r["fail"], k, s)


@pytest.mark.parametrize("kind", ["advance", "group"])
def test_failed_run_leaves_planes_and_ids_in_one_order(logs, kind):
    for r in logs[kind]:
        if r["rc"] == 0:
            continue
        before, failed, after = _split(r)
        # planes of the last complete sort that no G2P has written back: all of a run's, one class of a group's
        last = max([i for i, x in enumerate(before) if "finish" in x], default=-1)
        written = [x for x in before[last + 1:] if G2P.search(x)] if last >= 0 else []
        classes = {re.search(r"k_tiled_groupI(Li\dELi\dELi\d+)", x).group(1) for x in written if "group" in x}
        for k, state in enumerate(r["states"]):
            mine = bool(written) if kind == "advance" else any(c.startswith("Li3" if k == 1 else "Li2") for c in classes)
            want = last >= 0 and not mine
            assert (f"copy to {state}" in after) == want, (r["fail"], k, failed, after)


@pytest.mark.parametrize("kind", ["advance", "group"])
def test_failed_run_drops_the_items(logs, kind):
    for r in logs[kind]:
        for p in r["p2g"]:
            if r["rc"] == 0:
                assert "k_tiled" in p[0]
            else:
                assert "k_p2g" in p[0], (r["fail"], p)


def test_error_left_by_the_caller(logs):
    """An error that an earlier call of the caller left: reported before
    anything is launched, and not again; the items of an earlier sort stay."""
    left = logs["left"]
    assert left["rc"] < 0 and left["run"] == []
    assert left["again"] == 0
    assert left["sorted"] < 0 and "k_tiled" in left["p2g"][0]


if __name__ == "__main__":
    _child(sys.argv[1])
