"""The library's host side on the CPU, with its HIP calls answered by tests/_hip_stub.c in a child process: the tile schedules of
the persistent launches of Q5_K, Q4_K and Q3_K batches, what planning one costs, which calls allocate, copy or wait, which kernel a
Q6_K batch takes, and the launches of device-routed MoE layers."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.skipif(not os.path.isdir("/opt/rocm/include/hip"), reason="no HIP headers")

COMMON = r"""
import ctypes as C, json, os, sys, time
import numpy as np
sys.path.insert(0, os.path.join(ROOT, "stream-_amd"))
import es_hip_quant as E
L, S = E.Lib(), C.CDLL(STUB)
assert L.available(), L.last_error()
counts = (C.c_long * 5).in_dll(S, "counts")
def reset():
    for i in range(5): counts[i] = 0
def job(t, rows, cols, na, k):   # (addresses are never read)
    return dict(type=t, rows=rows, cols=cols, W=(k + 1) << 40, act=1 << 50, astride=cols // 256 * 292, nb=na, y=(k + 1) << 52, ystride=rows)
"""


@pytest.fixture(scope="module")
def child(hiplib, tmp_path_factory):
    so = tmp_path_factory.mktemp("stub") / "stub.so"
    subprocess.run(["gcc", "-O2", "-w", "-shared", "-fPIC", "-I/opt/rocm/include", "-o", str(so), os.path.join(ROOT, "tests", "_hip_stub.c")],
                   check=True)

    def run(code):
        r = subprocess.run([sys.executable, "-c", f"ROOT, STUB = {ROOT!r}, {str(so)!r}\n" + COMMON + code], capture_output=True, text=True,
                           env=dict(os.environ, LD_PRELOAD=str(so)), timeout=300)
        assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
        return json.loads(r.stdout.splitlines()[-1])

    return run


SCHEDULE = r"""
rec = np.dtype([("w", "<u8"), ("act", "<u8"), ("y", "<u8"), ("astride", "<u4"), ("ystride4", "<u4"), ("row_bytes", "<u4"), ("nbk", "<i4"),
                ("t64", "<i4"), ("tok0", "<i4"), ("na", "<i4"), ("rows", "<i4"), ("ntok", "<i4"), ("pad", "<i4")])
bad = []
def check(t, shapes, on):
    L.set_direct_persistent(on)
    p = L.plan([job(t, r, c, na, k) for k, (r, c, na) in enumerate(shapes)])
    n = C.c_size_t.in_dll(S, "copy_bytes").value
    raw = C.string_at(C.c_void_p.in_dll(S, "copy_dst").value, n)
    p.close()
    for T in (64, 128):   # the launch's tile width and grid, from the table's own end
        nt = sum((r + 63) // 64 * ((na + T - 1) // T) for r, _, na in shapes)
        at = (nt * 64 + 255) // 256 * 256
        for grid in (512, 256):
            if at + 4 * (grid + 1) > n: continue
            ptr = np.frombuffer(raw, "<i4", grid + 1, at)
            if ptr[0] == 0 and ptr[-1] == nt and np.all(np.diff(ptr) >= 0): break
        else: continue
        break
    else:
        bad.append([t, shapes, on, "no table"]); return
    tiles = np.frombuffer(raw, rec, nt)
    bb = {E.Q3_K: 110, E.Q4_K: 144, E.Q5_K: 176}[t]
    want = {((k + 1 << 40) + 64 * rt * c // 256 * bb, t0) for k, (r, c, na) in enumerate(shapes) for rt in range((r + 63) // 64)
            for t0 in range(0, na, T)}
    got = [(int(x["w"]), int(x["tok0"])) for x in tiles]
    wg = np.repeat(np.arange(grid), np.diff(ptr))
    xcd = {}
    for x, w in zip(tiles, wg): xcd.setdefault(int(x["w"]), set()).add(int(w) % 8)
    load = np.diff(ptr).reshape(-1, 8)   # [workgroup of the XCD][XCD]
    rts = np.bincount([next(iter(v)) for v in xcd.values()], minlength=8)
    ok = (sorted(got) == sorted(want) and all(len(v) == 1 for v in xcd.values()) and np.all(load.max(0) - load.min(0) <= 1) and
          rts.max() - rts.min() <= 1)
    for x in tiles:
        k = (int(x["w"]) >> 40) - 1
        r, c, na = shapes[k]
        row0 = (int(x["w"]) - (k + 1 << 40)) // (c // 256 * bb)
        ok = ok and x["y"] == (k + 1 << 52) + 4 * (int(x["tok0"]) * r + row0) and x["rows"] == min(64, r - row0)
        ok = ok and x["ntok"] == min(T, na - x["tok0"]) and x["na"] == na and x["nbk"] == c // 256 and x["t64"] == (T == 64 and grid == 512)
    if not ok: bad.append([t, shapes, on, T, grid])
for t in (E.Q3_K, E.Q4_K, E.Q5_K):
    for on in (1, 3) if t != E.Q5_K else (1,):
        for r in (1, 64, 65, 500, 2048, 8192, 8200):
            for na in (33, 64, 65, 128, 129, 512):
                check(t, [(r, 2048, na)], on)
                check(t, [(r, 2048, na), (2 * r + 7, 2048, na)], on)
print(json.dumps(bad))
"""


def test_even_schedules(child):
    """products whose tiles cost the same: every tile once, a row tile's tiles on one XCD, tiles dealt evenly"""
    assert child(SCHEDULE) == []


def test_planning_time(child):
    """a persistent launch of 256 tiles is planned in a few times what the same products' one-workgroup-per-tile launch takes (the
    sorts and heaps of the general schedule made it over 30 times), so a batch that is planned on every call is not bound by it"""
    r = child(r"""
out = []
for on in (3, 1):
    L.set_direct_persistent(on)
    best = 1e9
    for _ in range(200):
        jobs, n = L.make_jobs([job(E.Q5_K, 8192, 2048, 64, k) for k in range(2)])
        t0 = time.perf_counter()
        for _ in range(10): L._L.es_hip_plan_destroy(L._L.es_hip_plan_create(jobs, n))
        best = min(best, (time.perf_counter() - t0) * 1e5)
    out.append(best)
print(json.dumps(out))
""")
    assert r[1] < 8 * r[0] + 5, r


NOALLOC = r"""
def noalloc(t, rows, cols, na):
    return L._L.es_hip_matvec_multi_dev_noalloc(t, 1 << 40, cols, 0, rows, 1 << 50, E.act_bytes(t, cols), na, 1 << 52, rows, None)
"""


def test_noalloc_q6k_limit(child):
    """the no-allocation product's row limit for Q6_K is the tiled kernel's (tables and pre-pass planes of 16, 32 or a multiple of
    64 activations in 32 MiB), whichever kernel serves the call"""
    r = child(NOALLOC + r"""
def ok(nbk, na):
    n = nbk * (16 if na <= 16 else 32 if na <= 32 else (na + 63) // 64 * 64)
    up = lambda v: (v + 255) // 256 * 256
    return 512 + up(n * 256) + up(n * 36) <= 32 << 20
bad = []
for na in (16, 17, 32, 33, 64, 65, 128, 129, 512, 2048):
    edge = next((b for b in range(1, 4097) if not ok(b, na)), 4097)
    for nbk in {1, edge // 2, edge - 2, edge - 1, edge, edge + 1, 4096} - {0}:
        if nbk <= 4096 and (noalloc(E.Q6_K, 64, 256 * nbk, na) == 0) != ok(nbk, na): bad.append([na, nbk])
for na in (1, 5, 8, 15):   # no planes: every row length
    if noalloc(E.Q6_K, 64, 1 << 20, na): bad.append([na])
print(json.dumps(bad))
""")
    assert r == []


def test_noalloc_by_value(child):
    """a no-allocation product that is one job of one launch (and its pre-pass) travels as kernel arguments: nothing is copied, and
    without a pre-pass nothing of the shared scratch is used; only tile schedules (Q3_K and Q4_K on the persistent kernel) are"""
    r = child(NOALLOC + r"""
out = []
for t in (E.Q4_0, E.Q5_0, E.Q8_0, E.Q2_K, E.Q4_K, E.Q6_K):
    for na in (1, 2, 5, 8, 15, 16, 31):
        reset()
        assert noalloc(t, 2048, 2048, na) == 0, L.last_error()
        if counts[0] < 1 or counts[1] or counts[2] or counts[3]: out.append([t, na, list(counts)])
print(json.dumps(out))
""")
    assert r == []


def test_noalloc_q5k_tables(child):
    """Q5_K products: tile tables are copied only where they are short and the per-tile launch is the slower one"""
    r = child(NOALLOC + r"""
out = []
for rows in (64, 2048, 8192, 8256, 32768):
    for na in (1, 8, 63, 64, 65, 128, 512):
        reset()
        assert noalloc(E.Q5_K, rows, 2048, na) == 0, L.last_error()
        if counts[2] != (8 <= na < 64 and rows <= 8192) or C.c_size_t.in_dll(S, "copy_bytes").value > 16384: out.append([rows, na, list(counts)])
print(json.dumps(out))
""")
    assert r == []


Q6K_WAVES = [   # batches faster on the kernel with one wave per superblock: (rows, superblocks, activations) of each product
    [(2048, 3, 5)], [(8192, 8, 5)], [(2048, 24, 5)], [(2048, 28, 7)], [(2048, 32, 9)], [(4096, 32, 6)], [(2048, 3, 8)] * 112, [(8192, 3, 64)],
    [(8192, 3, 128)], [(8192, 8, 128)], [(2048, 32, 64)], [(2048, 32, 256)], [(512, 3, 256)] * 16, [(2048, 3, 5), (512, 8, 2)],
    [(2048, 8, 8), (512, 8, 2)], [(2048, 16, 9), (512, 8, 2)], [(4096, 32, 9), (512, 8, 2)], [(32768, 1, 512)], [(32768, 2, 512)],
    [(2048, 3, n) for n in (17, 25, 33, 41, 50, 60)], [(24158, 12, 9)], [(24050, 12, 9)] * 3, [(52000, 4, 8)] * 3, [(5004, 8, 9)] * 12]
Q6K_OTHERS = [   # ... and faster on the decode or the tiled kernel
    [(512, 28, 5)], [(512, 32, 5)], [(2048, 32, 8)], [(512, 32, 8)] * 4, [(2048, 48, 6)], [(8192, 32, 5)], [(8192, 3, 256)], [(8192, 5, 256)],
    [(32768, 3, 16)], [(32768, 6, 16)], [(2048, 3, 16)] * 64, [(2048, 3, 64)] * 16, [(2048, 8, 5), (512, 8, 2)], [(8192, 8, 8), (512, 8, 2)],
    [(2048, 32, 12), (512, 8, 2)], [(8192, 8, 4)], [(2048, 32, 512)], [(159288, 5, 8)], [(4593, 5, 8)] * 12, [(5809, 7, 8)] * 12, [(8879, 8, 8)] * 12, [(711, 9, 33)] * 12]


def test_q6k_kernel_choice(child):
    """measured batches take the faster kernel (with the choice off, the launches are those of the decode and tiled kernels)"""
    r = child(r"""
shapes = ((C.c_long * 4) * 64).in_dll(S, "shapes")
def launches(batch, on):
    L.set_q6k_persistent(on)
    p = L.plan([job(E.Q6_K, r, 256 * b, na, k) for k, (r, b, na) in enumerate(batch)])
    reset()
    p.run()
    n = counts[0]
    assert 0 < n < 64
    p.close()
    return [list(shapes[i]) for i in range(n)]
def waves(batch): return launches(batch, 1) != launches(batch, 0)
print(json.dumps([[b for b in %r if not waves(b)], [b for b in %r if waves(b)]]))
""" % (Q6K_WAVES, Q6K_OTHERS))
    assert r == [[], []]


def test_q6k_whole_rounds(child):
    """that kernel's workgroups come in whole rounds of the CUs (256) where its waves fill one with a single workgroup: ragged
    batches whose last round was nearly empty"""
    r = child(r"""
shapes = ((C.c_long * 4) * 64).in_dll(S, "shapes")
out = []
for n, rows, nbk, na in ((12, 3461, 22, 11), (5, 6359, 5, 77), (2, 10291, 8, 64), (3, 648, 9, 100)):
    p = L.plan([job(E.Q6_K, rows, 256 * nbk, na, k) for k in range(n)])
    reset()
    p.run()
    if counts[0] != 1 or shapes[0][0] > 256: out.append([n, rows, nbk, na, counts[0], list(shapes[0])])
    p.close()
print(json.dumps(out))
""")
    assert r == []


def test_q6k_pairs_travel_with_their_launch(child):
    """gate and up of a Q6_K FFN of 5 to 64 activations on the kernel with one wave per superblock: no allocation, no copy and no
    wait, on the first call or a later one"""
    r = child(r"""
out = []
for k, na in enumerate((5, 8, 15, 16, 33, 64)):
    for call in range(2):
        reset()
        assert L._L.es_hip_dense_ffn_dev(E.Q6_K, 1 << 40, E.Q6_K, 2 << 40, E.Q6_K, 3 << 40, 2048, 4096, na, 1 << 50, 292 * 8, 1 << 51, 1 << 52,
                                         1 << 53, 2048, None) == 0, L.last_error()
        if counts[0] != 3 or counts[1] or counts[2] or counts[3]: out.append([na, call, list(counts)])
print(json.dumps(out))
""")
    assert r == []


def test_q6k_grid_rows(child):
    """jobs of unequal length as kernel arguments: at most a quarter of the launch's workgroups without a tile"""
    r = child(r"""
shapes = ((C.c_long * 4) * 64).in_dll(S, "shapes")
out = []
for rows, nbk, na in (((2048, 512, 512), 8, 6), ((4096, 1024, 1024), 8, 8), ((2048, 256), 8, 8), ((300, 33, 2500, 16), 4, 8), ((3584, 3584), 8, 6)):
    p = L.plan([job(E.Q6_K, r, 256 * nbk, na, k) for k, r in enumerate(rows)])
    reset()
    p.run()
    least = sum((r + 15) // 16 for r in rows)   # row groups; the largest batch here takes two a workgroup
    x, y = shapes[0][0], shapes[0][1]
    if counts[0] != 1 or x % 8 or y > 8 or x * y > 1.25 * least + 8 * len(rows) or 2 * x * y < least: out.append([rows, nbk, na, counts[0], list(shapes[0])])
    p.close()
print(json.dumps(out))
""")
    assert r == []


def test_decode_grid_rows(child):
    """... and in decode launches: q, k and v of a layer"""
    r = child(r"""
shapes = ((C.c_long * 4) * 64).in_dll(S, "shapes")
out = []
for t, na in ((E.Q6_K, 1), (E.Q3_K, 4), (E.Q4_K, 1), (E.Q2_K, 1)):
    grids = []
    for rows in ((4096, 1024, 1024), (4096,), (1024,)):
        p = L.plan([job(t, r, 4096, na, k) for k, r in enumerate(rows)])
        reset()
        p.run()
        grids.append(shapes[0][0] * shapes[0][1])
        p.close()
    if counts[0] != 1 or grids[0] > 1.1 * (grids[1] + 2 * grids[2]): out.append([t, na, grids])
print(json.dumps(out))
""")
    assert r == []


MOE = r"""
shapes = ((C.c_long * 4) * 64).in_dll(S, "shapes")
def layer(types, n, ff, ne, k, N):   # the launches of a layer of N tokens
    experts = [dict(gate=(1 << 40) + e * (1 << 28), up=(2 << 40) + e * (1 << 28), down=(3 << 40) + e * (1 << 28)) for e in range(ne)]
    ctx = L.moe_ctx(E.MoeArgs(*types, n, ff, experts, np.zeros(1, np.int32), np.zeros((1, k), np.int32), np.zeros((1, k), np.float32)), N, k)
    reset()
    ctx.run(N, 1 << 50, 1 << 51, 1 << 52, E.act_bytes(types[0], n), 1 << 53, n)
    r = [list(shapes[i]) for i in range(counts[0])]
    ctx.close()
    return r
"""


def test_moe_pair_workgroups(child):
    """the pair form's second launch: whole rounds of at most one workgroup per CU while 128 rows a workgroup allow it"""
    r = child(MOE + r"""
bad = []
for n in (1024, 1280, 2048):
    for N in range(1, 17):
        gu, down = layer((E.Q4_K, E.Q4_K, E.Q4_K), n, 512, 128, 4, N)
        rows = -(-n // down[0])
        if down[1] != N or down[0] * N > 256 or rows > 128: bad.append([n, N, down])
print(json.dumps(bad))
""")
    assert r == []


MOE_PAIRS = [   # measured layers faster as pairs: gate/up and down type, n, ff, experts, choices, tokens
    ("Q4_K", "Q6_K", 2048, 768, 128, 8, 1), ("Q4_K", "Q6_K", 2048, 768, 128, 8, 12), ("Q4_K", "Q4_K", 2048, 512, 128, 2, 32),
    ("Q4_K", "Q4_K", 2048, 256, 16, 1, 91), ("Q5_K", "Q6_K", 1536, 1024, 128, 1, 12), ("Q4_K", "Q6_K", 1280, 512, 8, 1, 46),
    ("Q4_0", "Q4_K", 2048, 512, 8, 1, 58), ("Q8_0", "Q6_K", 2048, 256, 16, 1, 60), ("Q4_K", "Q6_K", 2048, 1024, 60, 4, 12)]
MOE_GROUPED = [   # ... and faster grouped
    ("Q4_K", "Q6_K", 2048, 768, 128, 8, 20), ("Q5_K", "Q6_K", 1536, 1024, 128, 1, 21), ("Q5_K", "Q6_K", 1536, 1024, 128, 1, 53),
    ("Q4_K", "Q6_K", 1792, 256, 64, 2, 75), ("Q4_K", "Q6_K", 1792, 768, 60, 2, 20), ("Q4_K", "Q6_K", 2048, 1024, 16, 1, 27), ("Q4_K", "Q4_K", 2048, 512, 128, 2, 80),
    ("Q5_K", "Q6_K", 2048, 512, 60, 1, 75), ("Q4_K", "Q6_K", 2048, 1024, 60, 4, 16)]


def test_moe_form(child):
    """measured layers take the faster form (the pair form is two launches)"""
    r = child(MOE + r"""
def pairs(c):
    t = [E.TYPES[c[0]], E.TYPES[c[0]], E.TYPES[c[1]]]
    return len(layer(t, *c[2:])) == 2
print(json.dumps([[c for c in %r if not pairs(c)], [c for c in %r if pairs(c)]]))
""" % (MOE_PAIRS, MOE_GROUPED))
    assert r == [[], []]
