"""Groups of the sync-free sweep's plan (group_positions of preprocess.cpp).

A workgroup of k_sweep_async takes the next group of eight positions, one per
wave, and runs them side by side; a position waits for its dependencies, and
the workgroup for all of its positions.  On the CPU: the structure of the
groups, and that any number of workgroups finishes them, taken in order.  On
the GPU: a batch large enough for each rule of chain_for (capi.hip) against
the same clouds one by one, bit for bit.
"""

import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

import test_sweep_protocol as protocol
from conftest import PKG, ROOT, load_fixture

pc = PKG.pointcloud
solver = PKG.solver
GROUP = 8

SHIM = """
#include <cstddef>
#include "%s/3d-mfcfd_amd/csrc/preprocess.h"
extern "C" int groups(int n, int m, const int* seq, const long long* ptr, const unsigned* take,
                      const unsigned char* late, int chain, int* slots, unsigned char* late_src) {
    mfcfd::SweepDirPlan p;
    p.seq.assign(seq, seq + m);
    p.take_ptr.assign(ptr, ptr + m + 1);
    p.take.assign(take, take + ptr[m]);
    p.late.assign(late, late + m);
    mfcfd::group_positions(p, n, chain);
    for (std::size_t u = 0; u < p.slots.size(); ++u) slots[u] = p.slots[u];
    for (int u = 0; u < m; ++u) late_src[u] = p.late_src[u];
    return (int)p.slots.size();
}
""" % ROOT


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    d = tmp_path_factory.mktemp("groups")
    src, so = str(d / "groups.cpp"), str(d / "libgroups.so")
    with open(src, "w") as f:
        f.write(SHIM)
    subprocess.run(["g++", "-O2", "-fPIC", "-std=c++17", "-shared", "-o", so, src,
                    os.path.join(ROOT, "3d-mfcfd_amd", "csrc", "preprocess.cpp")], check=True)
    return C.CDLL(so)


def plan_arrays(cl, backup):
    """Per direction: seq, take_ptr, take, late of the cloud's plan."""
    n = cl.n
    f = lambda a: np.ascontiguousarray(a, dtype=np.float64).ravel()
    i = lambda a: np.ascontiguousarray(a, dtype=np.int32).ravel()
    cnt, lists = solver.split_stencils(cl)
    alias, pwa = solver.alias_order(cl)
    cap = 200 * n
    seq, ptr = np.zeros(2 * n, dtype=np.int32), np.zeros(2 * (n + 1), dtype=np.int64)
    take, sizes = np.zeros(2 * cap, dtype=np.uint32), np.zeros(6, dtype=np.int64)
    late = np.zeros(2 * n, dtype=np.uint8)
    rc = protocol.lib().san_sweep_plan_late(n, i(cl.status), i(cl.nbhs), i(cl.conn), i(cnt), i(lists), i(alias),
                                            i(pwa), f(cl.x), f(cl.y), f(cl.z), int(backup), cap, seq, ptr, take,
                                            sizes, late)
    assert rc == 0
    for d in range(2):
        m, _, nt = (int(v) for v in sizes[3 * d:3 * d + 3])
        yield (seq[d * n:d * n + m].copy(), ptr[d * (n + 1):d * (n + 1) + m + 1].copy(),
               take[d * cap:d * cap + nt].copy(), late[d * n:d * n + m].copy())


def run_groups(slots, deps, workgroups):
    """Positions finished before no workgroup can go on."""
    taken, running, done = 0, [], set()
    groups = slots.reshape(-1, GROUP)
    while True:
        while len(running) < workgroups and taken < len(groups):
            running.append([int(u) for u in groups[taken] if u >= 0])
            taken += 1
        moved = False
        for g in running:
            for u in list(g):
                if all(v in done for v in deps[u]):
                    done.add(u)
                    g.remove(u)
                    moved = True
        running = [g for g in running if g]
        if not moved and not (taken < len(groups) and len(running) < workgroups):
            return len(done)


@pytest.mark.parametrize("name,backup", [("implicit_morton", False), ("implicit_backup", True),
                                         ("implicit_supersonic", False)])
@pytest.mark.parametrize("chain", [1, 2, 8])
def test_groups_keep_the_order_and_finish(lib, name, backup, chain):
    cl, _ = load_fixture(name)
    vp = lambda a: a.ctypes.data_as(C.c_void_p)
    linked = 0
    for seq, ptr, take, late in plan_arrays(cl, backup):
        m = len(seq)
        slots, late_src = np.zeros(m + GROUP, dtype=np.int32), np.zeros(m, dtype=np.uint8)
        k = lib.groups(cl.n, m, vp(seq), vp(ptr), vp(take), vp(late), chain, vp(slots), vp(late_src))
        assert k == -(-m // GROUP) * GROUP
        slots = slots[:k]
        assert np.array_equal(np.sort(slots[slots >= 0]), np.arange(m)) and (slots[m:] == -1).all()
        if chain == 1:
            assert np.array_equal(slots[:m], np.arange(m)) and not late_src.any()
        where = np.zeros(m, dtype=np.int64)
        where[slots[:m]] = np.arange(m)
        at = np.full(cl.n, -1)
        at[seq] = np.arange(m)
        deps = []
        for u in range(m):
            e = take[ptr[u]:ptr[u + 1]]
            d = at[(e[(e & 8) != 0] >> 4).astype(np.int64)]
            deps.append(sorted(set(int(v) for v in d)))
            # dependencies: earlier positions, in this group or an earlier one
            assert all(v < u and where[v] // GROUP <= where[u] // GROUP for v in deps[u])
            if late_src[u]:
                v = int(at[int(e[-1] >> 4)])
                assert late[u] > 0 and v == deps[u][-1]
                assert where[v] == where[u] // GROUP * GROUP + late_src[u] - 1
                linked += 1
        for workgroups in (1, 3):
            assert run_groups(slots, deps, workgroups) == m
    assert (linked > 0) == (chain > 1)


@pytest.mark.gpu
@pytest.mark.parametrize("precision,copies,levels", [("fp64", 12, (12, 1e9)), ("fp64", 50, (6, 12)),
                                                     ("fp64", 100, (0, 6)), ("mixed", 110, (6, 12)),
                                                     ("mixed", 200, (0, 6))])
def test_every_chain_rule_gives_the_separate_runs(precision, copies, levels):
    cl = pc.fixture_cloud(900, seed=5, order="morton")
    machs, aoas = np.linspace(0.3, 0.8, copies), np.linspace(-3.0, 6.0, copies)
    prim = [np.tile(pc.freestream_prim(m, a), (cl.n, 1)) for m, a in zip(machs, aoas)]
    bs = solver.BatchSolver([cl] * copies, list(machs), list(aoas), 1.0, mode="implicit", precision=precision)
    info = bs.sweep_info()
    resident = 4096 if precision == "mixed" else 2048
    in_flight = resident * (info["levels_fwd"] + info["levels_bwd"]) / (2.0 * info["swept"])
    print(f"[gpu] {precision}, {copies} clouds of {cl.n}: {in_flight:.1f} levels in flight", flush=True)
    assert levels[0] <= in_flight < levels[1]
    bs.upload("prim", np.concatenate(prim))
    bs.run(1, 4)
    got = bs.split(bs.download("prim"))
    bs.close()
    for b in (0, copies // 2, copies - 1):
        s = solver.Solver(cl, machs[b], aoas[b], 1.0, mode="implicit", precision=precision)
        s.upload("prim", prim[b])
        s.run(1, 4)
        assert np.array_equal(got[b], s.download("prim")), b
        s.close()
