"""What the kernel library launches, without a GPU: its host code runs in a child
process behind a recorder of the HIP runtime's launches (tests/native/launch_log.cpp),
with addresses that nothing reads."""

import json
import os
import subprocess
import sys

import pytest

from orion_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import ctypes, json, sys
log = ctypes.CDLL(sys.argv[1])
lib = ctypes.CDLL(sys.argv[2])
log.launch_log_name.restype = log.launch_log_kernel.restype = ctypes.c_char_p
P, Z, D = ctypes.c_void_p, ctypes.c_size_t, ctypes.c_double
lib.orion_gemm_bf16_nt.argtypes = [P, P, P] + [ctypes.c_int] * 4 + [P]
lib.orion_lamb_workspace_bytes.argtypes = [P, ctypes.c_int]
lib.orion_lamb_workspace_bytes.restype = Z
lib.orion_lamb_step.argtypes = [P, ctypes.c_int, D, D, D, D, D, P, Z, P]
AT = 1 << 40                      # an aligned address that nothing reads

def taken():
    out = [(log.launch_log_name(i).decode(), log.launch_log_grid(i), log.launch_log_block(i))
           for i in range(log.launch_log_size())]
    log.launch_log_clear()
    return out
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    if not os.path.exists(_lib.KERNELS_LIB):
        pytest.fail("liborion_kernels.so is not built")
    shim = str(tmp_path_factory.mktemp("launch_log") / "liblaunchlog.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wall",
                    os.path.join(ROOT, "tests", "native", "launch_log.cpp"), "-o", shim],
                   check=True)

    def child(body, *args):
        env = dict(os.environ, LD_PRELOAD=shim)
        out = subprocess.run([sys.executable, "-c", CHILD + body, shim, _lib.KERNELS_LIB,
                              json.dumps(args)], env=env, check=True, capture_output=True,
                             text=True, timeout=120)
        return json.loads(out.stdout)
    return child


GEMM = """
out = []
for m, n, k, cus, stream in json.loads(sys.argv[3])[0]:
    log.launch_log_set_compute_units(cus)
    rc = lib.orion_gemm_bf16_nt(AT, AT, AT, m, n, k, 0, AT if stream is True else stream)
    queries = log.launch_log_queries()
    out.append((rc, taken(), queries))
print(json.dumps(out))
"""

# Workgroups of the tile that measured fastest, by size and compute units of the stream.
GEMM_TILES = [
    # the whole GPU
    (256, 512, 256, 256, 64), (1024, 1024, 1024, 256, 256), (3072, 1024, 1024, 256, 192),
    (2816, 3328, 1856, 256, 143),
    # streams limited to some compute units: 256 x 256 tiles where smaller ones would
    # only take turns (us, 256 x 256 and what the whole GPU's rule takes: 36.8 and 51.4;
    # 13.7 and 23.5; 23.4 and 34.3; 38.3 and 46.6; 8.5 and 20.5; 8.6 and 12.6)
    (2048, 2048, 2048, 64, 64), (1024, 4096, 512, 64, 64), (4096, 2048, 1024, 128, 128),
    (3072, 1024, 1024, 32, 48), (1792, 1024, 192, 32, 28), (2560, 1024, 192, 64, 40),
    # and smaller ones where they still pay (256 x 256 tiles and these: 121 and 31, 121
    # and 23, 60 and 44)
    (512, 512, 8192, 32, 32), (512, 512, 8192, 64, 64), (1792, 768, 3648, 64, 84),
]


def test_gemm_tiles_follow_the_streams_compute_units(run):
    got = run(GEMM, [(m, n, k, cus, True) for m, n, k, cus, _ in GEMM_TILES])
    bad = []
    for case, (rc, launches, _) in zip(GEMM_TILES, got):
        assert rc == 0 and len(launches) == 1
        if launches[0][1] != case[-1]:
            bad.append((case, launches))
    assert not bad


def test_gemm_edge_cases_run_on_the_tiles_that_they_name(run):
    from tests.test_kernels_gpu import EDGE_TILES
    got = run(GEMM, [(*shape, 256, True) for _, shape in EDGE_TILES])
    for (tile, (m, n, k)), (rc, launches, _) in zip(EDGE_TILES, got):
        rows, cols = map(int, tile.split("x"))
        ((name, grid, _),) = launches
        assert rc == 0 and f"tile_kernelILi{rows}ELi{cols}E" in name, (tile, m, n, k, name)
        assert grid == -(-m // rows) * (n // cols)
    assert {m % 96 for tile, (m, _, _) in EDGE_TILES if tile == "96x128"} == {0, 32, 64}


def test_gemm_two_wave_groups_take_uneven_depths_from_nine_k_tiles_on(run):
    from tests.test_kernels_gpu import UNEVEN_DEPTHS
    for depths, tile in ((UNEVEN_DEPTHS, "ILi32ELi64E"), ((64, 192, 320, 448), "ILi64ELi64E")):
        for rc, ((name, _, _),), _ in run(GEMM, [(256, 512, k, 256, True) for k in depths]):
            assert rc == 0 and f"tile_kernel{tile}" in name


def test_gemm_on_limited_streams_by_costs_measured_there(run):
    # 128 x 128 tiles 5 to 18 % faster than the 256 x 256 that the whole GPU's costs ask for
    cases = [(768, 2816, 384, 128, 132), (2048, 1792, 448, 128, 224), (512, 4352, 448, 128, 136),
             (6656, 256, 448, 64, 104), (512, 3840, 384, 64, 120), (768, 1792, 448, 64, 84),
             (256, 2816, 256, 32, 44), (4096, 256, 448, 32, 64), (512, 1536, 320, 32, 48)]
    got = run(GEMM, [(m, n, k, cus, True) for m, n, k, cus, _ in cases])
    for (*_, tiles), (rc, launches, _) in zip(cases, got):
        assert rc == 0 and [grid for _, grid, _ in launches] == [tiles]
        assert "Li128ELi128E" in launches[0][0]


def test_gemm_asks_for_the_compute_units_only_where_they_decide(run):
    (rc, whole, queries), *runtimes_own, (rc_unknown, unknown, _) = run(GEMM, [
        (8192, 8192, 8192, 64, True),       # 256 x 256 tiles on any stream
        (2048, 2048, 2048, 64, None),       # the null, legacy and per-thread streams span
        (2048, 2048, 2048, 64, 1),          # the GPU, and are no handles to ask about
        (2048, 2048, 2048, 64, 2),
        (2048, 2048, 2048, 0, True)])       # a failing query: the whole GPU, and no error left
    assert rc == rc_unknown == 0
    assert queries == 0 and whole[0][1] == 1024
    for status, launches, asked in runtimes_own:
        assert status == 0 and asked == 0 and launches[0][1] == 256
    assert unknown[0][1] == 256


LAMB = """
counts = json.loads(sys.argv[3])[0]
table = (ctypes.c_uint64 * (5 * len(counts)))()
for i, n in enumerate(counts):
    table[5 * i:5 * i + 5] = [AT] * 4 + [n]
size = lib.orion_lamb_workspace_bytes(table, len(counts))
rc = lib.orion_lamb_step(table, len(counts), 0.1, 0.9, 0.999, 1e-6, 0.0, AT, size, None)
print(json.dumps((rc, taken())))
"""


@pytest.mark.parametrize("counts", [
    # the Transformer-XL client's: an embedding of 137 M elements, its bias, one layer's
    [267735 * 512, 267735, 3 * 512 * 512, 512 * 512, 512 * 512, 512, 512, 2048 * 512, 2048,
     2048 * 512, 512, 512, 512],
    [5120 * 4096 - 1, 1], [5120 * 4096], [8192 * 4096 + 1], [3] * 130, [5, 0, 70001]])
def test_no_launch_of_a_lamb_step_is_long(run, counts):
    # a launch once begun cannot be held back: best-effort training has to leave gaps
    rc, launches = run(LAMB, counts)
    assert rc == 0
    for kernel, most in (("lamb_moments", 5120), ("lamb_update", 8192)):
        grids = [grid for name, grid, _ in launches if kernel in name]
        assert max(grids) <= most
        assert sum(grids) == sum(-(-n // 4096) for n in counts)
    ratios = [grid for name, grid, _ in launches if "lamb_ratio" in name]
    assert sum(ratios) == sum(n > 0 for n in counts)


def test_the_passes_of_a_lamb_step_are_launched_as_they_are_built(run):
    # sixteen wavefronts a workgroup in the first pass, four in the second
    _, launches = run(LAMB, [70001])
    assert {name.split("lamb_")[1].split("_")[0]: block for name, _, block in launches} == {
        "moments": 1024, "ratio": 1024, "update": 256}
    source = open(os.path.join(ROOT, "orion_amd", "csrc", "kernels", "lamb.hip")).read()
    for kernel, threads in (("moments", "kMomentsThreads"), ("ratio", "kReduceThreads"),
                            ("update", "kThreads")):
        assert f"__launch_bounds__({threads}) void lamb_{kernel}_kernel" in source


TXL = """
I = ctypes.c_int
class Dims(ctypes.Structure):
    _fields_ = [(n, I) for n in ("layers", "heads", "inner", "q_len", "m_len", "batch")] + [
        ("eps", ctypes.c_float)]
lib.orion_txl_workspace_bytes.argtypes = [P]
lib.orion_txl_workspace_bytes.restype = Z
lib.orion_txl_hidden.argtypes = [P] * 6 + [Z, P, Z, I, P, P, Z, P]
out = []
for layers, heads, inner, q_len, m_len, batch, cus in json.loads(sys.argv[3])[0]:
    log.launch_log_set_compute_units(cus)
    dims = Dims(layers, heads, inner, q_len, m_len, batch, 1e-5)
    size = lib.orion_txl_workspace_bytes(ctypes.byref(dims))
    stride = m_len * batch * 512
    rc = lib.orion_txl_hidden(ctypes.byref(dims), (P * (11 * layers))(*[AT] * (11 * layers)),
                              AT, AT, AT, AT, stride, None, 0, 0, AT, AT, size, AT)
    queries = log.launch_log_queries()
    out.append((rc, taken(), queries))
print(json.dumps(out))
"""


@pytest.mark.parametrize("q_len,batch", [(192, 4), (192, 2), (192, 1), (101, 3), (16, 1), (65, 7)])
def test_no_workgroup_of_a_layers_products_is_empty(run, q_len, batch):
    # the scheduler reads a launch's need of compute units from its number of workgroups
    ((rc, launches, _),) = run(TXL, [(2, 8, 2048, q_len, 192, batch, 256)])
    assert rc == 0
    # rows go to eight, four, or where eight panels hold them two or one groups of workgroups,
    # evenly by 16, and in a group to panels of up to 48, the fewest in all; a panel has 16
    # tasks of each product, and a group as many workgroups, at most its share of 256
    tiles = -(-q_len * batch // 16)
    panels_of = {groups: -(-(-(-tiles // groups)) // 3) for groups in ((8, 4, 2, 1) if tiles <= 24 else (8, 4))}
    groups = min(panels_of, key=lambda groups: groups * panels_of[groups])
    panels, most = panels_of[groups], 256 // groups
    grids = {part: [grid for name, grid, _ in launches if part in name]
             for part in ("panel_gemm_kernelILi64ELi96E", "txl_layer_kernel")}
    assert grids == {"panel_gemm_kernelILi64ELi96E": [-(-q_len * batch // 64) * 3 * 8 * 64 // 96],
                     "txl_layer_kernel": [groups * min(most, panels * 16)] * 2}
    # the smallest group's tasks of the last layer, which has three products
    fewest = -(-(tiles // groups) // 3) * 3 * 16
    assert fewest >= min(most, panels * 16)


@pytest.mark.parametrize("q_len,batch,launches_a_layer", [
    (1, 1, 1), (192, 4, 1), (3840, 1, 1), (3841, 1, 2), (192, 32, 2), (200, 40, 3), (217, 50, 3),
    (65537, 16, 274)])
def test_no_launch_of_a_layers_products_is_long(run, q_len, batch, launches_a_layer):
    # a launch once begun cannot be held back: best-effort inference has to leave gaps
    rows = q_len * batch
    ((rc, _, layer_launches),) = run(TXL[:TXL.index("out = []")] + ROWS, [(q_len, batch)])
    assert rc == 0 and len(layer_launches) == 2 * launches_a_layer
    for layer in (layer_launches[:launches_a_layer], layer_launches[launches_a_layer:]):
        begin = min(at for at, _, _ in layer)
        shares = sorted((at - begin, own) for at, _, own in layer)
        # every row once: means and squares lie 128 bytes to a row
        assert [at for at, _ in shares] == [128 * sum(n for _, n in shares[:i])
                                            for i in range(launches_a_layer)]
        assert sum(own for _, own in shares) == rows and max(own for _, own in shares) <= 3840
        # each with counters of its own: eight of tasks, and three a panel of up to 48 rows
        counters = sorted(at for _, at, _ in layer)
        assert all(b - a >= 128 * (8 + 3 * -(-own // 48)) for a, b, (_, own) in
                   zip(counters, counters[1:], shares))


@pytest.mark.parametrize("inner,q_len,batch,own,ahead", [
    # 192 KiB of the coming weights a workgroup: 6 MiB of a layer, 4.5 of the last
    (2048, 192, 4, 192, [32, 24]), (2048, 16, 1, 8, [32, 24]),
    # as many as attention leaves of 256 compute units
    (2048, 192, 5, 240, [16, 16]), (2048, 128, 8, 256, [0, 0]), (2048, 192, 8, 384, [0, 0]),
    (65536, 192, 4, 192, [64, 64]), (65536, 16, 1, 8, [248, 248])])
def test_weights_read_ahead_follow_attentions_size_on_any_stream(run, inner, q_len, batch, own,
                                                                 ahead):
    # a launch may be issued to another stream than the call names, so that one is not asked
    for rc, launches, queries in run(TXL, [(2, 8, inner, q_len, 192, batch, cus)
                                           for cus in (32, 64, 128, 256)]):
        assert rc == 0 and queries == 0
        assert [grid for name, grid, _ in launches if "attention" in name] == [
            own + more for more in ahead]


def test_no_launch_of_attention_has_more_threads_than_a_grid_can_have(run):
    # many short segments: 2 blocks of queries for each of 6.4 million heads
    ((rc, launches, _),) = run(TXL, [(1, 32, 256, 33, 0, 200_000, 256)])
    assert rc == 0
    attention = [(grid, block) for name, grid, block in launches if "attention" in name]
    assert sum(grid for grid, _ in attention) == 32 * 200_000 * 2
    assert all(grid * block < 1 << 32 for grid, block in attention)


# Where a launch's means and squares lie, its counters and how many rows it has: words of the
# layer kernel's structure.
ROWS = """
log.launch_log_watch(b"txl_layer", 5, 42)
log.launch_log_word.restype = ctypes.c_uint64
((q_len, batch),) = json.loads(sys.argv[3])[0]
dims = Dims(2, 8, 2048, q_len, 0, batch, 1e-5)
size = lib.orion_txl_workspace_bytes(ctypes.byref(dims))
base = 1 << 41
rc = lib.orion_txl_hidden(ctypes.byref(dims), (P * 22)(*[AT] * 22), AT, AT, AT, None, 0, None,
                          0, 0, AT, base, size, None)
launches = [[log.launch_log_word(i, k) for k in (27, 40, 41)] for i in range(log.launch_log_size())
            if log.launch_log_words(i)]
print(json.dumps([(rc, size, [(parts, counters, rows & 0xffffffff)
                              for parts, counters, rows in launches])]))
"""


WORKSPACE = """
log.launch_log_watch(b"txl_layer", 5, 40)          # the structure's first 320 bytes
log.launch_log_word.restype = ctypes.c_uint64
out = []
for base in json.loads(sys.argv[3])[0]:
    dims = Dims(2, 8, 2048, 150, 192, 3, 1e-5)
    size = lib.orion_txl_workspace_bytes(ctypes.byref(dims))
    rc = lib.orion_txl_hidden(ctypes.byref(dims), (P * 22)(*[AT] * 22), AT, AT, AT, AT,
                              192 * 3 * 512, None, 0, 0, AT, base, size, None)
    words = [log.launch_log_word(i, k) for i in range(log.launch_log_size())
             for k in range(log.launch_log_words(i))]
    out.append((rc, size, [w - base for w in words if base <= w < base + size]))
    log.launch_log_clear()
print(json.dumps(out))
"""


def test_a_layers_arrays_begin_on_cache_lines_in_any_workspace(run):
    # caches may hold lines of them that another workgroup has written whole
    bases = [(1 << 41) + at for at in (0, 16, 64, 112, 128, 240)]
    body = TXL[:TXL.index("out = []")] + WORKSPACE
    for base, (rc, size, places) in zip(bases, run(body, bases)):
        assert rc == 0 and len(set(places)) > 10
        assert {(base + at) % 128 for at in places} == {0}
    assert run(body, [(1 << 41) + 8])[0][0] == 3


KERNELS = """
print(json.dumps([log.launch_log_kernel(i).decode() for i in range(log.launch_log_kernels())]))
"""


def test_the_scheduler_knows_the_classes_of_the_clients_kernels(run):
    # by the counters: none of these names tells what bounds its kernel, and a kernel of
    # unknown class passes beside anything
    from orion_amd.profiling import cu_need, rocprof
    names = subprocess.run(["c++filt"], input="\n".join(run(KERNELS)), capture_output=True,
                           check=True, text=True).stdout.split("\n")
    names = {rocprof.short_name(n) for n in names}
    own = {n for n in names if "lamb_" in n or "txl_" in n or "crit_" in n}
    assert len(own) == 12
    assert {n for n in own if cu_need.classify_source(n)[1] != "counters"} == set()
    # a LAMB step reaches 70 and 79 % of the HBM rate in its passes
    assert cu_need.classify("void lamb_moments_kernel") == 0
    assert cu_need.classify("void lamb_update_kernel") == 0
    assert cu_need.classify("crit_logits_kernel") == 1
