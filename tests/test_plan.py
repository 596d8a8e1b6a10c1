"""The host rules behind the projector kernels' launches (csrc/sq_plan.hpp),
compiled for the CPU: groups of nodes, offsets inside a group and LDS sizes, over
the cube sides and node lists that the kernels accept."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "sqdft_amd", "csrc")
MAXM = 43   # largest cube side the kernels take

SRC = r"""
#include "sq_plan.hpp"
#include <chrono>
#include <cstring>
using namespace sqk;
extern "C" {
int groups(int M, int max_nproj, int n_ip, int w, int n, const int *ts, int nts, const int *nodes, int B, int *out)
{
    size_t t[2] = {(size_t)ts[0], (size_t)ts[1]};
    const std::vector<int> g = make_groups({M, max_nproj, n_ip, w}, n, t, nts, nodes, B);
    std::memcpy(out, g.data(), g.size() * sizeof(int));
    return (int)g.size() - 1;
}
long noalloc_need(int M, int n_ip, int nb, long ng, int rs, int nn)
{
    return (long)NoallocSizes({M, 1, n_ip, 9}, nb, ng, rs, rs == 4, nn).total();
}
long noalloc_cap(int M, int n_ip, int nb, int rs, int nn)
{
    return (long)noalloc_limit({M, 1, n_ip, 9}, nb, rs, rs == 4, nn);
}
long node_bytes(int M, int n_ip, int rs, int nvec, int lists)
{
    return (long)(batch_node_bytes({M, 1, n_ip, 9}, rs, nvec) + batch_list_bytes(lists));
}
int walk(int M, int max_nproj, int w, int ts, int gl_max, int deep12, int deep8, int one12, int one8, long *out)
{
    const ProjDims d{M, max_nproj, 100, w};
    const ProjwUse pw = projw_use(d, ts);
    const int need[2][2] = {{deep12, deep8}, {one12, one8}};
    const ProjwPlan p = projw_plan(M, pw, ts, gl_max, need);
    const long v[9] = {p.shape, p.sz, p.shares, p.pad, (long)p.lds, pw.on ? projw_pu(M, pw, p.pad) : 0,
                       pw.on ? projw_pu(M, pw) : 0, pw.mfma, projw_depths(M, pw, ts).sz[0]};
    std::memcpy(out, v, sizeof v);
    return pw.on;
}
int staged(int M, int ts, int deep, int gl_max, long *out)
{
    const ProjsPlan p = projs_plan(M, ts, deep, gl_max);
    out[0] = p.sz; out[1] = p.shares; out[2] = (long)p.lds;
    return 0;
}
int nlapply(int M, int max_nproj, int n_ip, int gl_max, long *out)
{
    const NlapplyPlan p = nlapply_plan({M, max_nproj, n_ip, 9}, gl_max);
    out[0] = p.fits; out[1] = p.columns; out[2] = (long)p.lds;
    return 0;
}
int planes(int n, int z0, int nz, int *out)
{
    const std::vector<int> v = NodeOrder(n).planes(z0, nz);
    std::memcpy(out, v.data(), v.size() * sizeof(int));
    return (int)v.size();
}
void order(int n, int *nodes, int cnt)
{
    std::vector<int> v(nodes, nodes + cnt);
    NodeOrder(n).sort(v);
    std::memcpy(nodes, v.data(), v.size() * sizeof(int));
}
// seconds to order the whole grid, and to sort it by key
void order_time(int n, double *out)
{
    auto now = [] { return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count(); };
    double t = now();
    const std::vector<int> v = NodeOrder(n).planes(0, n);
    out[0] = now() - t;
    t = now();
    const NodeOrder o(n);
    std::vector<std::pair<unsigned long, int>> k(v.size());
    for (size_t i = 0; i < k.size(); ++i) k[i] = {o.key((int)i), (int)i};
    std::sort(k.begin(), k.end());
    out[1] = now() - t;
}
int nlapply_shares(int M, int max_nproj, int ng) { return nlapply_split({M, max_nproj, 100, 9}, ng); }
int pad(int M) { return group_pad(M); }
int range(int M) { return group_range(M); }
int offset(int m, int M, int dx, int dy, int dz) { return member_offset(m, group_pad(M), M, M * M, M * M * M, dx, dy, dz); }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src, lib = d / "plan.cpp", d / "libplan.so"
    src.write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-fPIC", "-shared", "-I", CSRC, str(src), "-o",
                    str(lib)], check=True)
    d = C.CDLL(str(lib))
    d.noalloc_need.restype = d.noalloc_cap.restype = C.c_long
    d.noalloc_need.argtypes = [C.c_int, C.c_int, C.c_int, C.c_long, C.c_int, C.c_int]
    d.node_bytes.restype = C.c_long
    return d


def iptr(a):
    return a.ctypes.data_as(C.POINTER(C.c_int))


def groups_of(plan, M, np_, w, n, types, nodes):
    nodes = np.ascontiguousarray(nodes, dtype=np.int32)
    ts = np.array(list(types) + [8], dtype=np.int32)
    out = np.zeros(nodes.size + 2, dtype=np.int32)
    ng = plan.groups(M, np_, 100, w, n, iptr(ts), len(types), iptr(nodes), nodes.size, iptr(out))
    return [nodes[out[i]:out[i + 1]] for i in range(ng)]


def node_lists(M):
    """(grid side, nodes): pairs a few rows, columns and planes apart, either one
    first, and a shuffled whole grid."""
    n = 40
    rng = np.random.Generator(np.random.PCG64(M))
    for dx in range(-20, 21):
        for dy in range(0, 21):
            a, b = (20, 1, 7), (20 + dx, 1 + dy, 7 + int(rng.integers(0, 3)))
            p = [(c[2] * n + c[1]) * n + c[0] for c in (a, b)]
            yield n, p if rng.integers(0, 2) else p[::-1]
    yield 9, rng.permutation(9 ** 3)
    yield 9, np.arange(9 ** 3)


@pytest.mark.parametrize("np_,w", [(1, 9), (1, 13), (3, 9), (3, 15)])
@pytest.mark.parametrize("types", [(8,), (4,), (4, 8)])
def test_groups_stay_within_what_the_kernels_walk(plan, np_, w, types):
    for M in range(3, MAXM + 1, 2):
        for n, nodes in node_lists(M):
            gs = groups_of(plan, M, np_, w, n, types, nodes)
            assert np.array_equal(np.concatenate(gs), nodes)
            for g in gs:
                assert 1 <= g.size <= 8
                r = np.stack([g % n, (g // n) % n, g // (n * n)])
                d = r.max(axis=1) - r.min(axis=1)
                assert (M + d[0]) * (M + d[1]) <= (M + 3) ** 2 and d[2] <= 1
                # a member's cube starts at most group_pad values after the corner
                assert d[2] * M * M + d[1] * M + d[0] <= plan.pad(M)


@pytest.mark.parametrize("M", [3, 5, 7, 9, 13, 17, 25, 35, 43])
def test_scalar_offsets_stay_inside_their_resource(plan, M):
    """Whichever members of a group are active: the offset of an active member
    takes its cube to its own vector, that of an idle one is inside the range."""
    rng = np.random.Generator(np.random.PCG64(M))
    pad = plan.pad(M)
    for n, nodes in list(node_lists(M))[::7] + [(9, rng.permutation(9 ** 3)), (9, np.arange(9 ** 3))]:
        for g in groups_of(plan, M, 1, 9, n, (8,), nodes):
            on = rng.integers(0, 2, 8).astype(bool) & (np.arange(8) < g.size)
            if not on.any():
                continue
            start = np.stack([g % n, (g // n) % n, g // (n * n)], axis=1)
            corner = start[on[:g.size]].min(axis=0)
            for m in range(8):
                d = corner - start[min(m, g.size - 1)]
                off = plan.offset(m, M, int(d[0]), int(d[1]), int(d[2]))
                assert 0 <= off < plan.range(M) < 2 ** 28, (n, g, m)
                if on[m]:   # the first point of its cube, seen from the union's corner
                    assert off - (d[2] * M * M + d[1] * M + d[0]) == pad + m * M ** 3


@pytest.mark.parametrize("rs", [8, 4])
@pytest.mark.parametrize("M,n_ip", [(7, 62), (7, 186), (17, 900), (35, 3000), (43, 20000)])
def test_allocation_free_calls_split_only_where_they_must(plan, M, n_ip, rs):
    """A batch that the scratch limit accepts fits whole when its groups are full,
    and up to a quarter of them may hold one node; the limit itself is the sum of
    the buffers in full groups and LCAP + 1 ints a node."""
    up = lambda b: -(-b // 256) * 256   # noqa: E731
    for nb in (1, 2, 7, 8, 9, 64, 1000, 1001, 9133, 60000):
        ng, nn = -(-nb // 8), 4096
        ints = [nb, nb * 512, nb, ng * 1024, ng, 16]
        cap = sum(up(4 * i) for i in ints) + up(8 * nb * n_ip) + up(nb * M ** 3 * rs)
        if rs == 4:
            cap += 2 * up(nb * M ** 3 * rs) + up(nn * rs)
        assert plan.noalloc_cap(M, n_ip, nb, rs, nn) == cap
        assert plan.noalloc_need(M, n_ip, nb, ng, rs, nn) <= cap
        assert plan.noalloc_need(M, n_ip, nb, ng + nb // 4, rs, nn) <= cap


@pytest.mark.parametrize("M,n_ip", [(7, 62), (17, 900), (43, 20000)])
@pytest.mark.parametrize("rs", [8, 4])
def test_batches_budget_for_groups_of_one_node(plan, M, n_ip, rs):
    """A batch is sized for everything it allocates per node: five vectors (one
    more for the forces), projections, four rows of 502 tridiagonal entries, 22
    doubles and 3 ints of scalars, and the lists of a group that holds one node."""
    held = 5 * M ** 3 * rs + 8 * n_ip + 4 * 502 * 8 + 8 * (11 + 8 + 4 + 2) + 4 * 3
    group = 4 * (1024 + 1 + 1)
    assert plan.node_bytes(M, n_ip, rs, 2, 0) >= held + group
    assert plan.node_bytes(M, n_ip, rs, 3, 1) >= held + M ** 3 * rs + group + 4 * (512 + 1)


LDS = 160 * 1024
IMG = 40          # bytes of an image's data in LDS
WIDTHS = {1: (1, 3, 5, 7, 9, 11, 13), 3: (1, 3, 5, 7, 9, 11, 13, 15)}


def up16(b):
    return -(-b // 16) * 16


@pytest.mark.parametrize("np_,ts", [(1, 8), (1, 4), (3, 8)])
def test_walks_whose_slab_and_images_fit_find_room_for_the_columns(plan, np_, ts):
    """k_projw takes every table whose padded slab (one FP64, two FP32 planes) fits
    the LDS beside the longest list's data, with LDS for what its plan stages."""
    out = (C.c_long * 9)()
    for w in WIDTHS[np_]:
        for M in range(max(w, 3), MAXM + 1, 2):
            for gl in list(range(1, 620, 3)) + [700, 1024]:
                assert plan.walk(M, np_, w, ts, gl, 1, 1, 1, 1, out)
                shape, sz, shares, pad, lds, cap, cap_pad, mfma, deep = out
                # the shallowest slab that may be walked
                assert (shape >= 0) == (up16(gl * IMG) + cap_pad * 8 * ts * (1 if mfma else deep) <= LDS), (w, M, gl)
                if shape < 0:
                    continue
                assert sz == deep or up16(gl * IMG) + cap_pad * 8 * ts * deep > LDS
                columns = up16(4 * (M + 3) ** 2)
                assert up16(-(-gl // shares) * IMG) + columns + cap * 8 * ts * sz <= lds <= LDS
                if up16(gl * IMG) + columns + cap_pad * 8 * ts * sz <= LDS - 4 * 49:
                    assert shares == 1 and pad == 1   # shared or unpadded only where it must
                # every union that a group may have fits the capacity
                for dx in range(0, 10):
                    for dy in range(0, 10):
                        ux, uy = M + dx, M + dy
                        if ux * uy > (M + 3) ** 2:
                            continue
                        if not pad:
                            u = ux * uy
                            assert u + (8 - u) % 32 * mfma <= cap


@pytest.mark.parametrize("ts,deep", [(8, 2), (4, 4)])
def test_staged_projections_take_every_list(plan, ts, deep):
    out = (C.c_long * 3)()
    for M in range(3, MAXM + 1, 2):
        for gl in range(1, 1025, 7):
            plan.staged(M, ts, deep, gl, out)
            sz, shares, lds = out
            assert sz in (1, 2, 4) and sz <= deep
            assert up16(-(-gl // shares) * IMG) + (M + 3) ** 2 * 8 * ts * sz <= lds <= LDS, (M, gl)


def test_a_deep_slab_short_of_slots_gives_way_to_one_plane(plan):
    """Matrix-core walks: slots are planned for the deep slab and for one plane."""
    out = (C.c_long * 9)()
    for M, w in ((7, 5), (17, 9), (21, 7), (25, 9)):
        plan.walk(M, 3, w, 8, 200, 12, 18, 12, 18, out)
        deep = out[8]
        assert deep > 1 and (out[0], out[1]) == (0, deep)
        plan.walk(M, 3, w, 8, 200, 13, 19, 12, 18, out)
        assert (out[0], out[1]) == (0, 1)
        plan.walk(M, 3, w, 8, 200, 99, 99, 99, 99, out)
        assert out[0] == -1


@pytest.mark.parametrize("np_", [1, 3, 4, 9])
def test_nonlocal_rows_need_no_room_for_the_columns(plan, np_):
    """k_nlapplyg takes every batch whose loc table and rows fit the LDS, and keeps
    the column table where that fits too."""
    out = (C.c_long * 3)()
    for M in (7, 17, 25, 31, 35, 43):
        for gl in range(1, 1025, 9):
            for n_ip in (1, 900, 3000, 8000, 20000, 40000):
                rows = up16(4 * n_ip) + gl * np_ * 80
                cols = 4 * (M + 3) ** 2
                plan.nlapply(M, np_, n_ip, gl, out)
                assert bool(out[0]) == (rows <= LDS)
                if out[0]:
                    assert rows + cols * out[1] <= out[2] <= LDS
                    assert out[1] or rows + cols + 4 * 49 > LDS


def runs(n, length):
    m = -(-n // length)
    r = np.zeros(n, dtype=int)
    for c in range(m):
        r[c * n // m:(c + 1) * n // m] = c
    return r


def brick_key(n, nodes):
    """Brick z, y, x of the even runs of up to 2, 4 and 4 nodes, then z, y, x."""
    rx, ry, rz = runs(n, 4), runs(n, 2), runs(n, 2)
    x, y, z = nodes % n, (nodes // n) % n, nodes // (n * n)
    return np.lexsort((x, y, z, rx[x], ry[y] // 2, rz[z]))


@pytest.mark.parametrize("n", list(range(1, 20)) + [25, 32])
def test_nodes_are_visited_brick_by_brick(plan, n):
    rng = np.random.Generator(np.random.PCG64(n))
    for z0, nz in {(0, n), (0, 1), (n // 2, n - n // 2), (max(n - 2, 0), min(n, 2)), (n // 3, 1)}:
        out = np.zeros(n ** 3, dtype=np.int32)
        cnt = plan.planes(n, z0, nz, iptr(out))
        ref = np.arange(z0 * n * n, (z0 + nz) * n * n)
        assert cnt == ref.size and np.array_equal(out[:cnt], ref[brick_key(n, ref)])
    for cnt in (0, 1, 2, n ** 3 // 20, n ** 3 // 2, 2 * n ** 3):     # with repeats
        v = rng.integers(0, n ** 3, cnt).astype(np.int32)
        ref = v[brick_key(n, v)]
        plan.order(n, iptr(v), v.size)
        assert np.array_equal(v, ref)


def test_ordering_a_whole_grid_takes_no_sort(plan):
    """96^3 nodes are ordered at every density step, while the GPU waits."""
    t = (C.c_double * 2)()
    best = [1e9, 1e9]
    for _ in range(3):
        plan.order_time(96, t)
        best = [min(a, b) for a, b in zip(best, t)]
    assert 3 * best[0] < best[1], best


def test_shares_of_the_nonlocal_apply(plan):
    """Every share fills the rows again, three times as many for p projectors: fewer
    shares there; at least four points a thread, at least one share."""
    for M in range(3, MAXM + 1, 2):
        for ng in (1, 7, 64, 480, 512, 1024, 4096, 100000):
            s, p = plan.nlapply_shares(M, 1, ng), plan.nlapply_shares(M, 3, ng)
            assert 1 <= p <= s <= max(1, (M + 3) * (M + 1) * M // 2048)
            assert p * ng <= max(3072, ng) and s * ng <= max(6144, ng)
    assert plan.nlapply_shares(35, 1, 1024) == 6 and plan.nlapply_shares(31, 3, 1024) == 3
