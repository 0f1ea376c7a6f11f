"""The library's kernels and host driver, compiled as host C++ against the
CPU emulation of the HIP API in tests/emu (one thread per GPU lane) and run
under AddressSanitizer: every bin variant with rows that fit it in one
chunk and rows spread over several chunks, the global fallbacks, and
out-of-bounds accesses caught on the CPU.  Results are checked against the
host Gustavson product by tests/emu/emu_main.cpp.  Inputs are small:
emulating a 1024-lane workgroup costs a thread per lane."""
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from gpuspgemm_amd import generators as gen
from gpuspgemm_amd.csr import HostCSR

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "emu")
BUILD = os.path.join(EMU, "_build")
EXE = os.path.join(BUILD, "emu_spgemm")
CSRC = os.path.join(ROOT, "gpuspgemm_amd", "csrc")
INT_MAX = 2**31 - 1

import gpuspgemm_amd as g
import oracle

# Compiled variants, read from the library (no GPU needed): symbolic
# (lanes per row, A entries per chunk, table slots) and fused (lanes, chunk,
# capacity).
_SV = g.variant_list(0)
_NV = g.variant_list(1)
SYM = {v["id"]: (v["lanes"], v["chunk"], v["table"]) for v in _SV if not v["max"]}
SYM_MAX = next(v["id"] for v in _SV if v["max"])
NUM = {v["id"]: (v["lanes"], v["chunk"], v["capacity"]) for v in _NV if not v["global"]}
NUM_GLOBAL = next(v["id"] for v in _NV if v["global"])


def build_emu(csrc: str, exe: str) -> None:
    """The emulation build of the kernel and host sources in `csrc`: each
    translation unit compiled by its own g++ process, side by side."""
    srcs = [os.path.join(csrc, f) for f in ("k_rows.hip", "k_sym.hip", "k_symnum.hip", "api.hip")]
    srcs += [os.path.join(EMU, "emu_runtime.cpp"), os.path.join(EMU, "emu_main.cpp")]
    flags = ["-std=c++17", "-O1", "-g", "-fsanitize=address", "-fno-omit-frame-pointer", "-pthread",
             "-Wno-unused-result"]
    inc = ["-I", os.path.join(EMU, "include"), "-I", os.path.join(ROOT, "include"), "-I", csrc,
           "-I", os.path.join(ROOT, "gpuspgemm_amd", "apps")]
    objs = [f"{exe}.{i}.o" for i in range(len(srcs))]
    procs = [subprocess.Popen(["g++", *flags, *inc, "-x", "c++", "-c", s, "-o", o]) for s, o in zip(srcs, objs)]
    codes = [p.wait() for p in procs]
    try:
        assert codes == [0] * len(srcs), f"emulation build failed: {codes}"
        subprocess.run(["g++", *flags, *objs, "-o", exe], check=True)
    finally:
        for o in objs:
            if os.path.exists(o):
                os.remove(o)


@pytest.fixture(scope="module")
def emu():
    os.makedirs(BUILD, exist_ok=True)
    tmp = f".{os.getpid()}"
    build_emu(CSRC, EXE + tmp)
    os.replace(EXE + tmp, EXE)  # parallel test workers may be running the previous build
    return EXE


def run_emu(exe, tmp_path, A, B, *extra, tables=None, env=None):
    fa, fb = tmp_path / "a.csr", tmp_path / "b.csr"
    A.save_to_filename(str(fa))
    B.save_to_filename(str(fb))
    args = [exe, str(fa), str(fb), *extra]
    for phase, text in (tables or {}).items():
        f = tmp_path / f"table{phase}.txt"
        f.write_text(text)
        args += ["--sym-table" if phase == 0 else "--num-table", str(f)]
    res = subprocess.run(args, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=600,
                         env=None if env is None else {**os.environ, **env})
    assert res.returncode == 0, res.stdout[-4000:]
    assert "structure identical" in res.stdout
    return res.stdout


def call(A, B, *extra, tables=None, env=None):
    """One emulator run for run_emu_all."""
    return A, B, extra, tables, env


def run_emu_all(exe, tmp_path, *calls):
    """Independent emulator runs side by side (each emulated workgroup keeps
    only a few host cores busy), each in a directory of its own; their
    outputs in order."""
    def one(i):
        A, B, extra, tables, env = calls[i]
        d = tmp_path / f"run{i}"
        d.mkdir()
        return run_emu(exe, d, A, B, *extra, tables=tables, env=env)
    with ThreadPoolExecutor(len(calls)) as ex:
        return list(ex.map(one, range(len(calls))))


def squares(m, k, seed):
    """k entries per row of A and of B: NIP = k^2, nnz <= k^2."""
    n = max(4 * k, 64)
    return gen.uniform8(m=m, per_row=k, seed=seed, n=n), gen.uniform8(m=n, per_row=k, seed=seed + 1, n=40 * k)


def chunked(m, k, seed):
    """k entries per row of A, one per row of B: NIP = nnz <= k, A rows span k/EC chunks."""
    n = max(4 * k, 64)
    return gen.uniform8(m=m, per_row=k, seed=seed, n=n), gen.uniform8(m=n, per_row=1, seed=seed + 1, n=n)


def rows_for(lanes):
    return 96 if lanes <= 16 else (12 if lanes <= 256 else 3)


def test_uniform_stencil_powerlaw(emu, tmp_path):
    A = gen.uniform8(m=512)
    S = gen.stencil27(g=5).astype(np.float32)
    P = gen.powerlaw(m=1000, seed=5)
    run_emu_all(emu, tmp_path, call(A, A), call(S, S, "--f32"), call(P, P, "--repeat", "2"))


def test_graph_replay(emu, tmp_path):
    """Graph replay on: each repeat multiplies a fresh copy of A with new
    values (new addresses, same launches).  The first call runs eagerly, the
    second captures both phases, the rest replay them; every result must
    equal the host product."""
    A = gen.powerlaw(m=1000, seed=5)
    R = gen.random_csr(200, 150, 0.04, seed=6, empty_rows=0.3)
    Rb = gen.random_csr(150, 120, 0.05, seed=7)
    P = gen.powerlaw(m=600, seed=9)
    out = run_emu_all(emu, tmp_path, call(A, A, "--repeat", "4", "--graphs"),
                      call(R, Rb, "--repeat", "3", "--graphs"),
                      # the server's lanes run eagerly with replay on
                      call(P, P, "--serve", "6", str(1 << 30), "3", "--graphs"))
    assert out[0].count("structure identical") == 4
    assert "graphs captured 2 replayed 4" in out[0]
    assert out[1].count("structure identical") == 3
    assert "graphs captured 2 replayed 2" in out[1]
    assert out[2].count("structure identical") == 6


def test_merged_launches(emu, tmp_path):
    """A fused table with a bin for every variant of the merged small-row
    launch and four bins of the merged longer-row launch: the rows of each
    set's bins share one launch, a workgroup per unit; every result must
    equal the host product."""
    assert sorted(v["id"] for v in _NV if v["merged"] == 0) == [10, 11, 12, 13, 14, 16]
    assert sorted(v["id"] for v in _NV if v["merged"] == 1) == [4, 5, 6, 7, 8]
    table = ("10 4 4\n14 8 8\n11 12 16\n16 16 16\n12 32 32\n13 64 64\n"
             f"4 96 96\n5 160 128\n6 512 256\n7 {INT_MAX} 1024\n{NUM_GLOBAL} {INT_MAX} {INT_MAX}\n")
    A = gen.powerlaw(m=2500, seed=21)
    F = A.astype(np.float32)
    run_emu_all(emu, tmp_path, call(A, A, tables={1: table}), call(F, F, "--f32", tables={1: table}))


def _alternating_units_case():
    """Rows whose symbolic units alternate LDS layouts inside one workgroup
    of the emulated grid (8 workgroups, one XCD slice each): bins of the
    larger-table launch with variants 6, 5, 6 (as in the tuned defaults)
    holding 1, 1 and 22 units of 4 rows, so that workgroup 0 runs a unit of
    each in turn.  B has 16 entries per row; a row of A with k entries has
    NIP 16k."""
    nb = 400
    # columns drawn from 48: rows of C stay short (cheap fused pass), while
    # the symbolic pass still hashes every product
    brows = [np.unique(gen.rand_below(31, 1 + r, np.arange(16), np.full(16, 48))) for r in range(nb)]
    brows = [np.concatenate([x, np.arange(48, 48 + 16 - x.size)]) for x in brows]  # exactly 16 each
    brpt = np.concatenate([[0], np.cumsum([x.size for x in brows])]).astype(np.int32)
    bcol = np.concatenate(brows).astype(np.int32)
    B = HostCSR(nb, 64, brpt, bcol, gen.rand_unit(32, 1, np.arange(bcol.size)) * 2 - 1)
    lengths = [6] * 4 + [12] * 4 + [24] * 88  # NIP 96 (bin of v6), 192 (v5), 384 (v6)
    arows = [np.unique(gen.rand_below(33, 1 + i, np.arange(k), np.full(k, nb)))[:k] for i, k in enumerate(lengths)]
    arows = [np.concatenate([x, np.setdiff1d(np.arange(nb), x)[:k - x.size]]) for x, k in zip(arows, lengths)]
    arows = [np.sort(x) for x in arows]
    rpt = np.concatenate([[0], np.cumsum([x.size for x in arows])]).astype(np.int32)
    col = np.concatenate(arows).astype(np.int32)
    A = HostCSR(len(arows), nb, rpt, col, gen.rand_unit(34, 1, np.arange(col.size)) * 2 - 1)
    table = "".join(f"{v} {cap} {INT_MAX}\n" for v, cap in
                    [(0, 8), (1, 16), (2, 32), (3, 64), (6, 128), (5, 256), (6, 768), (7, 2048), (8, 4096),
                     (SYM_MAX, INT_MAX)])
    return A, B, table


def test_symbolic_units_with_a_wave_held_back(emu, tmp_path):
    """Symbolic units of alternating LDS layouts (variants 6, 5, 6) in one
    workgroup while wave 1 of that workgroup is held back at every wave
    barrier, so the other waves run a unit or two ahead of it: the
    workgroup barrier between units of different layouts must keep them
    off the slots wave 1 still uses, and the result must equal the host
    product.  (Built without that barrier, the same run gives a wrong count
    or an out-of-bounds read only in some runs, so it is not kept as a
    planted-mistake check.)"""
    A, B, table = _alternating_units_case()
    fa, fb, ft = tmp_path / "a.csr", tmp_path / "b.csr", tmp_path / "sym.txt"
    A.save_to_filename(str(fa))
    B.save_to_filename(str(fb))
    ft.write_text(table)
    res = subprocess.run([emu, str(fa), str(fb), "--sym-table", str(ft)], stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, text=True, timeout=600,
                         env=dict(os.environ, EMU_SLOW_WAVE="1:100"))
    assert res.returncode == 0 and "structure identical" in res.stdout, res.stdout[-3000:]


def test_rectangular_and_empty_rows(emu, tmp_path):
    A = gen.random_csr(120, 90, 0.05, seed=1, empty_rows=0.3)
    B = gen.random_csr(90, 70, 0.06, seed=2, empty_rows=0.2)
    run_emu(emu, tmp_path, A, B)


def test_nip_per_row(emu, tmp_path):
    """NIP per row, read through the symbolic bins: a table of one-wide NIP
    ranges (bin b takes the rows of NIP b + 1) counts the rows of every NIP
    up to 14, so a length credited to the wrong row changes a count.  Rows
    of up to six entries sit beside rows of 700 and 1500 entries, whose
    64-row groups take several rounds of the NIP pass, and the 3000 rows
    end in a partial tile.  The debug log gives the counts, the total and
    the maximum; the oracle's NIP per row gives the expected ones."""
    rng = np.random.default_rng(41)
    n = 4096
    b_len = rng.integers(0, 4, n)
    b_rpt = np.concatenate([[0], np.cumsum(b_len)]).astype(np.int32)
    b_col = np.concatenate([np.sort(rng.choice(64, k, replace=False)) for k in b_len]).astype(np.int32)
    B = HostCSR(n, 64, b_rpt, b_col, rng.uniform(-1, 1, b_col.size))
    m = 3000
    a_len = rng.integers(0, 7, m)
    a_len[rng.random(m) < 0.2] = 0
    a_len[[5, 1900, 2990]] = [700, 1500, 40]
    a_rpt = np.concatenate([[0], np.cumsum(a_len)]).astype(np.int32)
    a_col = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in a_len]).astype(np.int32)
    A = HostCSR(m, n, a_rpt, a_col, rng.uniform(-1, 1, a_col.size))
    nip = oracle.nip_rows(A, B)
    caps = list(range(1, 15))
    table = "".join(f"0 {c} {INT_MAX}\n" for c in caps) + f"8 4000 {INT_MAX}\n{SYM_MAX} {INT_MAX} {INT_MAX}\n"
    out = run_emu(emu, tmp_path, A, B, tables={0: table}, env={"SPG_LOG_LEVEL": "debug"})
    want = [int(np.sum(nip == c)) for c in caps]
    want += [int(np.sum((nip > 14) & (nip <= 4000))), int(np.sum(nip > 4000))]
    assert want[-2] >= 2 and sum(want[:14]) > 1500, want
    line = next(x for x in out.splitlines() if "symbolic phase" in x)
    assert f"NIP {int(nip.sum())} (max {int(nip.max())} per row)" in line, line
    got = line.split("rows per symbolic bin [")[1].split("]")[0]
    assert [int(x) for x in got.split()] == want, line


def test_nip_of_dense_tiles(emu, tmp_path):
    """Tiles of dense rows are split over several workgroups of the NIP pass
    (here 1,535 rows of 0 to 90 entries, eight parts of 256 rows): full
    parts, one that the rows end in and two empty ones.  The first empty part
    would start one past A's last row pointer, where AddressSanitizer sees a
    read that is not clamped to the tile's end."""
    rng = np.random.default_rng(43)
    n = 300
    B = gen.random_csr(n, 50, 0.006, seed=44)
    a_len = rng.integers(0, 91, 1535)
    rpt = np.concatenate([[0], np.cumsum(a_len)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in a_len]).astype(np.int32)
    A = HostCSR(1535, n, rpt, col, rng.uniform(-1, 1, col.size))
    assert col.size > 1024 * 16 * 4
    nip = oracle.nip_rows(A, B)
    out = run_emu(emu, tmp_path, A, B, env={"SPG_LOG_LEVEL": "debug"})
    line = next(x for x in out.splitlines() if "symbolic phase" in x)
    assert f"NIP {int(nip.sum())} (max {int(nip.max())} per row)" in line, line


def test_scanned_tile_prefix(emu, tmp_path):
    """The scan stage reads each tile's prefix off one scanned array of tile
    sums, the path of multiplies of 2048 tiles or more, forced here from one
    tile: a product of three tiles and a server's batches of several
    products (each product's prefix starts at its own first tile) must
    equal the host product."""
    env = {"SPG_TILE_PREFIX_MIN": "1"}
    P = gen.powerlaw(m=4500, seed=11)
    Q = gen.powerlaw(m=600, seed=9)
    out = run_emu_all(emu, tmp_path, call(P, P, env=env), call(Q, Q, "--serve", "4", str(1 << 30), "4", env=env))
    assert out[1].count("structure identical") == 4


@pytest.mark.parametrize("variant", sorted(SYM))
def test_symbolic_variant(emu, tmp_path, variant):
    lanes, ec, t = SYM[variant]
    cap = t // 2
    table = {0: f"{variant} {cap} {INT_MAX}\n{SYM_MAX} {INT_MAX} {INT_MAX}\n"}
    m = rows_for(lanes)
    k = int(np.sqrt(cap))
    run_emu_all(emu, tmp_path, call(*squares(m, k, seed=variant), tables=table),
                call(*chunked(m, min(cap, 2 * ec + 1), seed=variant), tables=table))


@pytest.mark.parametrize("variant", sorted(NUM))
def test_fused_variant(emu, tmp_path, variant):
    lanes, ec, p = NUM[variant]
    table = {1: f"{variant} {INT_MAX} {p}\n{NUM_GLOBAL} {INT_MAX} {INT_MAX}\n"}
    m = rows_for(lanes)
    run_emu_all(emu, tmp_path, call(*squares(m, int(np.sqrt(p)), seed=10 + variant), tables=table),
                call(*chunked(m, min(p, 2 * ec + 1), seed=10 + variant), "--f32", tables=table))


WAVE_ROWS = [(0, v) for v, (lanes, _, _) in sorted(SYM.items()) if lanes == 64] + \
            [(1, v) for v, (lanes, _, _) in sorted(NUM.items()) if lanes == 64]


@pytest.mark.parametrize("phase,variant", WAVE_ROWS)
def test_wave_rows_count_entry_starts(emu, tmp_path, phase, variant):
    """Rows of one full wave find each product's A entry by counting entry
    starts in a bitmap: chunks whose products span more than one round
    (symbolic: rows of ~60 entries and NIP near the table size; fused: rows
    of ~120 entries, two chunks, ~2000 products), with B rows of uneven
    length and 40 % of them empty (dropped from the chunk before counting)."""
    if phase == 0:
        _, _, t = SYM[variant]
        table = {0: f"{variant} {t - 1} {INT_MAX}\n{SYM_MAX} {INT_MAX} {INT_MAX}\n"}
        A = gen.random_csr(8, 400, 0.15, seed=60 + variant)
        ncol = 2000
        per_row = 0.8 * (t - 1) / (60 * 0.6)
    else:
        _, _, p = NUM[variant]
        table = {1: f"{variant} {INT_MAX} {p}\n{NUM_GLOBAL} {INT_MAX} {INT_MAX}\n"}
        A = gen.random_csr(8, 400, 0.3, seed=60 + variant)
        ncol = min(p, 400)
        per_row = 2.5 * 64 * 12 / (120 * 0.6)
    B = gen.random_csr(400, ncol, min(0.9, per_row / ncol), seed=70 + variant, empty_rows=0.4)
    run_emu_all(emu, tmp_path, call(A, B, tables=table),
                call(A.astype(np.float32), B.astype(np.float32), "--f32", tables=table))


def _heavy_row_case(draws=9500):
    """A row of 21,525 columns, among the longest that the largest LDS tables
    of both passes hold (16,000 draws: 30,427, more than they hold), plus
    three ordinary rows."""
    nb = 20_000
    r0 = np.unique(gen.rand_below(3, 1, np.arange(draws), np.full(draws, nb)))
    rows = [r0] + [np.unique(gen.rand_below(3, 3 + i, np.arange(3), np.full(3, nb))) for i in range(3)]
    rpt = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    col = np.concatenate(rows).astype(np.int32)
    A = HostCSR(len(rows), nb, rpt, col, gen.rand_unit(3, 9, np.arange(col.size)) * 2 - 1)
    keys = np.unique(np.arange(nb, dtype=np.int64)[:, None] * 200_000
                     + gen.rand_below(4, 1, np.arange(nb * 3), np.full(nb * 3, 200_000)).reshape(nb, 3))
    brpt = np.zeros(nb + 1, dtype=np.int64)
    np.cumsum(np.bincount(keys // 200_000, minlength=nb), out=brpt[1:])
    bcol = (keys % 200_000).astype(np.int32)
    B = HostCSR(nb, 200_000, brpt.astype(np.int32), bcol, gen.rand_unit(4, 2, np.arange(bcol.size)) * 2 - 1)
    return A, B


GLOBAL_TABLES = {0: f"{SYM_MAX} {INT_MAX} {INT_MAX}\n", 1: f"{NUM_GLOBAL} {INT_MAX} {INT_MAX}\n"}


@pytest.mark.parametrize("variant", [v for v, (lanes, _, _) in sorted(NUM.items()) if lanes == 64])
def test_wave_rows_windows_and_wide_offsets(emu, tmp_path, variant):
    """Fused rows of one wave whose chunks of 64 entries hold more products
    than one window of the entry-start bitmap (2048), with entries that
    start before a window and run on into it, A rows of several chunks, and
    rows filled to the variant's capacity; with B's arrays addressed by 32-
    and by 64-bit offsets (SPG_WIDE_MIN)."""
    _, _, p = NUM[variant]
    table = {1: f"{variant} {INT_MAX} {p}\n{NUM_GLOBAL} {INT_MAX} {INT_MAX}\n"}
    A = gen.random_csr(7, 150, 0.9, seed=80 + variant)
    B = gen.random_csr(150, p, 0.5, seed=81 + variant, empty_rows=0.1)
    run_emu_all(emu, tmp_path, call(A, B, tables=table), call(A, B, tables=table, env={"SPG_WIDE_MIN": "0"}),
                call(A.astype(np.float32), B.astype(np.float32), "--f32", tables=table, env={"SPG_WIDE_MIN": "0"}))


def test_wide_offsets_start_where_narrow_ones_end(emu, tmp_path):
    """SPG_WIDE_MIN cannot be raised past the 2^29 entries whose values
    32-bit byte offsets reach."""
    A = gen.uniform8(m=64, per_row=2, seed=3, n=64)
    for value, used in (("2147483647", 1 << 29), (str((1 << 29) + 1), 1 << 29), ("1000", 1000), ("-5", 0)):
        out = run_emu(emu, tmp_path, A, A, env={"SPG_WIDE_MIN": value, "SPG_LOG_LEVEL": "debug"})
        assert f"64-bit offsets from {used} entries of B" in out, out


# fused variants that sort rows of at most `products` in registers
SORTED = [(v, NUM[v][2]) for v in sorted(NUM) if NUM[v][0] == NUM[v][2] or (NUM[v][0] == 64 and NUM[v][2] <= 128)]


@pytest.mark.parametrize("variant,products", SORTED)
@pytest.mark.parametrize("columns", [40, 1 << 25, 1 << 26])
def test_sorted_rows(emu, tmp_path, variant, products, columns):
    """Rows of one product up to the variant's slots and one more (a wave
    with such a row takes the hashed path), empty rows of B inside them,
    repeated columns (40 columns), and column counts at the limits that
    leave no room for the slot number beside the column (2^25 for two
    products a lane, 2^26 for one)."""
    rng = np.random.default_rng(variant)
    lens = [0, 1, 2, 3, 5, 7, 1, 4]
    pool = np.unique(np.r_[0, 1, columns - 1, rng.integers(0, columns, 40)])
    b_rows = [np.sort(rng.choice(pool, size=min(lens[k % 8], len(pool)), replace=False)) for k in range(64)]
    a_rows, per_wave = [], max(1, 64 // NUM[variant][0])
    for total in [products, 1, products - 1, products // 2, products + 1, products, 2, 3]:
        for _ in range(per_wave):  # a row whose products come close to `total`, in random order of B's rows
            row, have = [], 0
            for k in rng.permutation(64):
                if have + len(b_rows[k]) <= total and len(row) < NUM[variant][0]:
                    row.append(k)
                    have += len(b_rows[k])
            a_rows.append(np.sort(row))

    def matrix(rows, n, seed):
        rpt = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
        col = np.concatenate(rows).astype(np.int32)
        return HostCSR(len(rows), n, rpt, col, gen.rand_unit(seed, 1, np.arange(col.size)) * 2 - 1)
    A, B = matrix(a_rows, 64, 95), matrix(b_rows, columns, 96)
    table = {1: f"{variant} {INT_MAX} {NUM[variant][2]}\n{NUM_GLOBAL} {INT_MAX} {INT_MAX}\n"}
    run_emu_all(emu, tmp_path, call(A, B, tables=table), call(A, B, "--f32", tables=table))


@pytest.mark.parametrize("b", [5, 6, 8])
def test_many_products_on_few_columns(emu, tmp_path, b):
    """Dense blocks of b rows: b * b products on b columns.  The default
    tables give such rows to a variant with few lanes to a row (one that
    sorts them needs a lane for each product)."""
    m = 12 * b
    i = np.arange(m)
    col = (i // b * b)[:, None] + np.arange(b)[None, :]
    A = HostCSR(m, m, (np.arange(m + 1) * b).astype(np.int32), col.ravel().astype(np.int32),
                np.random.default_rng(b).uniform(-1, 1, m * b))
    out = run_emu(emu, tmp_path, A, A, env={"SPG_LOG_LEVEL": "debug"})
    fused = next(x for x in out.splitlines() if "fused bins: " in x).split("fused bins: ")[1].split(", ")
    line = next(x for x in out.splitlines() if "symbolic phase" in x)
    rows = [int(x) for x in line.split("rows per fused bin [")[1].split("]")[0].split()]
    taken = [int(fused[k].split()[0][1:]) for k in range(len(rows)) if rows[k]]
    assert sum(rows) == m and [NUM[v][0] for v in taken] == [8], (taken, rows)


@pytest.mark.parametrize("variant", [v["id"] for v in _NV if not v["global"] and v["lanes"] == 256 and v["chunk"] == 64])
def test_group_rows_and_column_counts(emu, tmp_path, variant):
    """Rows that the waves of a workgroup share, filled to one short of the
    variant's capacity, with as many columns as leave room for the table
    slot beside a sorted column (one fewer than 2^32 / slots) and one more,
    where the slots are looked up again."""
    _, _, p = NUM[variant]
    limit = 2**32 // (2 * p)
    table = {1: f"{variant} {INT_MAX} {p}\n{NUM_GLOBAL} {INT_MAX} {INT_MAX}\n"}
    rng = np.random.default_rng(variant)
    calls = []
    for n in (limit - 1, limit):
        pool = np.sort(rng.choice(n - 2, p - 3, replace=False)) + 1
        pool = np.r_[0, pool, n - 1]
        b_rows = [pool[k::40] for k in range(40)] + [pool[:90]] * 3
        rpt = np.concatenate([[0], np.cumsum([len(r) for r in b_rows])]).astype(np.int32)
        col = np.concatenate(b_rows).astype(np.int32)
        B = HostCSR(43, n, rpt, col, rng.uniform(-1, 1, col.size))
        A = HostCSR(2, 43, np.array([0, 43, 63], np.int32), np.r_[0:43, 0:20].astype(np.int32), rng.uniform(-1, 1, 63))
        calls.append(call(A, B, tables=table))
    run_emu_all(emu, tmp_path, *calls)


@pytest.fixture(scope="module")
def wave_share():
    exe = os.path.join(BUILD, "wave_share")
    tmp = f"{exe}.{os.getpid()}"
    os.makedirs(BUILD, exist_ok=True)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address", "-pthread", "-I",
                    os.path.join(EMU, "include"), "-I", CSRC, os.path.join(EMU, "wave_share.cpp"),
                    os.path.join(EMU, "emu_runtime.cpp"), "-o", tmp], check=True)
    os.replace(tmp, exe)
    return exe


@pytest.mark.parametrize("waves", [4, 16])
@pytest.mark.parametrize("entries,b_row", [(40, 3), (64, 5), (130, 4), (250, 3), (733, 4), (300, 9), (300, 20),
                                           (60, 60), (1030, 2), (90, 40)])
def test_waves_share_a_row_evenly(wave_share, waves, entries, b_row):
    """The waves of a workgroup walk a row together (by rounds, by chunks of
    64 entries, and as the rule picks): every product goes to one wave
    once; dealt by rounds, the waves' round counts differ by at most one,
    with one, two or three rounds to a chunk as with many; and the busiest
    wave's chunks read and rounds, as the rule weighs them, are no more
    than in the better of the two ways (for four waves, whose rule only
    looks at the mean, 1.43 times that: its worst over all row lengths)."""
    out = subprocess.run([wave_share, str(waves), str(entries), str(b_row)], stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, text=True, timeout=120)
    assert out.returncode == 0, out.stdout
    cost = {}
    for line in out.stdout.splitlines():
        how, rounds, hits = line.split(":")
        rounds = [int(x) for x in rounds.split()]
        assert len(rounds) == waves and hits.split() == ["1", "1"], line
        if how != "rule":
            chunks = -(-entries // 64)
            cost[how] = max(rounds) + 2 * (chunks if how == "rounds" else -(-chunks // waves))
        if how == "rounds":
            assert max(rounds) - min(rounds) <= 1, line
        if how == "rule":
            picked = rounds
    by = {line.split(":")[0]: [int(x) for x in line.split(":")[1].split()] for line in out.stdout.splitlines()}
    best = min(cost.values())
    # (the rule rounds the average up: one round more is as good)
    bound = (1.43 if waves == 4 else 1.0) * best + 1
    assert any(picked == by[how] and cost[how] <= bound for how in cost), (cost, out.stdout)


# one variant of every kind of row that looks columns up with table_slots: a
# wave, a workgroup, and (fused) a long row's workgroup
PROBED = [(0, min(v for v in SYM if SYM[v][0] == 64)), (0, max(v for v in SYM if SYM[v][0] == 256)),
          (1, min(v for v in NUM if NUM[v][0] == 64)), (1, min(v for v in NUM if NUM[v][:2] == (256, 64))),
          (1, max(v for v in NUM if NUM[v][:2] == (1024, 64)))]


@pytest.mark.parametrize("phase,variant", PROBED)
def test_columns_far_apart(emu, tmp_path, phase, variant):
    """Columns that lie a large power of two apart (as the block indices of a
    flattened tensor) must not share table slots: a product on 64 columns
    2^20 apart takes at most half as many compare-and-swaps again as the
    same product on adjacent columns."""
    if phase == 0:
        table = {0: f"{variant} {SYM[variant][2] // 2 - 1} {INT_MAX}\n{SYM_MAX} {INT_MAX} {INT_MAX}\n"}
    else:
        table = {1: f"{variant} {INT_MAX} {NUM[variant][2]}\n{NUM_GLOBAL} {INT_MAX} {INT_MAX}\n"}
    count, stride = 64, 1 << 20
    rng = np.random.default_rng(variant)
    k = 40
    B = HostCSR(6, count, (np.arange(7) * k).astype(np.int32),
                np.concatenate([np.sort(rng.choice(count, k, replace=False)) for _ in range(6)]).astype(np.int32),
                rng.uniform(-1, 1, 6 * k))
    far = HostCSR(6, (count - 1) * stride + 1, B.rpt, B.col * np.int32(stride), B.val)
    A = HostCSR(2, 6, np.array([0, 6, 11], np.int32), np.r_[0:6, 1:6].astype(np.int32), rng.uniform(-1, 1, 11))
    env = {"EMU_COUNT_CAS": "1"}
    out = run_emu_all(emu, tmp_path, call(A, B, tables=table, env=env), call(A, far, tables=table, env=env))
    near_cas, far_cas = (int(o.split("compare-and-swaps ")[1].split()[0]) for o in out)
    assert far_cas <= 1.5 * near_cas, (near_cas, far_cas)


def test_batch_behind_a_product_without_entries(emu, tmp_path):
    """A batch whose first product has no entries (null arrays): a wave of a
    fused unit that has no row sees item zero, instance zero, and must not
    read that product's B.  Five rows fill the first wave of a unit in part
    and leave the others without one; 20 and 40 products a row too."""
    for i, k in enumerate((2, 4, 6)):
        A = gen.uniform8(m=5, per_row=k, seed=3, n=64)
        B = gen.uniform8(m=64, per_row=k, seed=4, n=640)
        (tmp_path / str(i)).mkdir()
        run_emu(emu, tmp_path / str(i), A, B, "--batch-after-empty")


def test_symbolic_overflow_moves_to_the_largest_table(emu, tmp_path):
    """Workgroup rows of the variant that takes any NIP: 2,049 to 4,000
    distinct columns pass its limit and are counted again by the largest
    table, 2,048 and fewer (one row with 6,000 products on 300 columns)
    stay; rows of B long enough for the waves to share rounds, and short
    ones with enough entries of A for them to share chunks."""
    over = next(v["id"] for v in _SV if v["id"] == SYM_MAX - 1)
    table = {0: f"{over} 100000 {INT_MAX}\n{SYM_MAX} {INT_MAX} {INT_MAX}\n"}

    def matrix(rows, n, seed):
        rpt = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
        col = np.concatenate(rows).astype(np.int32)
        return HostCSR(len(rows), n, rpt, col, gen.rand_unit(seed, 1, np.arange(col.size)) * 2 - 1)

    # long rows of B: row k holds the columns 100 k .. 100 k + 99, the last 60 rows the columns 0 .. 299 in parts
    wide = [np.arange(100 * k, 100 * k + 100) for k in range(40)]
    wide += [np.arange(100 * (k % 3), 100 * (k % 3) + 100) for k in range(60)]
    B = matrix(wide, 4000, 91)
    A = matrix([np.arange(0, 40), np.arange(0, 20), np.r_[0:20, 20], np.arange(40, 100)], 100, 92)
    # one entry a row: 2,048, 2,049 and 300 distinct columns
    B1 = matrix([[k] for k in range(3000)], 3000, 93)
    A1 = matrix([np.arange(2048), np.arange(2049), np.arange(100, 400)], 3000, 94)
    run_emu_all(emu, tmp_path, call(A, B, tables=table), call(A1, B1, "--f32", tables=table))


def test_rows_past_the_counting_table_are_tried_once(emu, tmp_path):
    """24 rows in the bin whose table takes 2,048 columns, three to an
    emulated workgroup: 16 of 2,304 products on about 2,180 columns, two of
    4,800 on about 4,270 and six of 2,400 on 300.  A row that overflows
    takes the next ones of its workgroup with it to the largest-table
    launch, whatever they are, where the shorter ones, more than there are
    workgroups, are counted four at a time.  Every row of C must be right,
    and few products may be counted twice: 1.4 compare-and-swaps for every
    one that a count and a fused pass cannot do without (1.3 so; 1.7 when
    every row was tried until its table was full)."""
    rng = np.random.default_rng(12)
    b_rows = [np.sort(rng.choice(20_000, 48, replace=False)) for _ in range(200)]
    b_rows += [np.sort(rng.choice(300, 48, replace=False)) for _ in range(60)]
    a_rows = []
    for i in range(24):
        if i % 4 == 3:
            a_rows.append(200 + np.sort(rng.choice(60, 50, replace=False)))
        else:
            a_rows.append(np.sort(rng.choice(200, 100 if i in (5, 12) else 48, replace=False)))

    def matrix(rows, n):
        rpt = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
        col = np.concatenate(rows).astype(np.int32)
        return HostCSR(len(rows), n, rpt, col, rng.uniform(-1, 1, col.size))
    A, B = matrix(a_rows, 260), matrix(b_rows, 20_000)
    out = run_emu(emu, tmp_path, A, B, env={"EMU_COUNT_CAS": "1"})
    products, nnz = int(oracle.nip_rows(A, B).sum()), int(oracle.spgemm(A, B).nnz)
    cas = int(out.split("compare-and-swaps ")[1].split()[0])
    assert cas <= 1.4 * (products + nnz), (cas, products, nnz)


def test_global_paths(emu, tmp_path):
    """The heavy-row case first with the default tables, a long row of the
    largest LDS variants, and then with every row forced to the global
    kernels."""
    A, B = _heavy_row_case()
    longest = max(p for _, _, p in NUM.values())
    assert 16384 < int(np.diff(oracle.spgemm(A, B).rpt).max()) <= longest
    run_emu_all(emu, tmp_path, call(A, B), call(A, B, tables=GLOBAL_TABLES))


def test_row_past_the_largest_tables(emu, tmp_path):
    """A row of more columns than the largest count table admits: its waves
    stop, it joins the overflow list, is counted again in global memory (a
    second scan follows) and takes the global fused kernel, with the default
    tables."""
    A, B = _heavy_row_case(draws=16_000)
    assert int(np.diff(oracle.spgemm(A, B).rpt).max()) > max(p for _, _, p in NUM.values())
    out = run_emu(emu, tmp_path, A, B, env={"SPG_LOG_LEVEL": "debug"})
    line = next(x for x in out.splitlines() if "symbolic phase" in x)
    assert "fail bin 1," in line, line
    assert line.split("rows per fused bin [")[1].split("]")[0].split()[-1] == "1", line


def test_noalloc_entry(emu, tmp_path):
    """spg_multiply_noalloc into caller arrays, scratch in the fixed device
    array: a capacity one short of nnz(C) fails with out-of-memory and
    reports the nnz needed, then repeated products match the host; the
    heavy-row case forced to the global kernels carves both global tables
    out of the fixed array too."""
    P = gen.powerlaw(m=1000, seed=5)
    S = gen.stencil27(g=5).astype(np.float32)
    A, B = _heavy_row_case()
    out = run_emu_all(emu, tmp_path, call(P, P, "--noalloc", "--repeat", "2"), call(S, S, "--f32", "--noalloc"),
                      call(A, B, "--noalloc", tables=GLOBAL_TABLES))
    assert out[0].count("structure identical") == 2
    assert "status out of device memory" in out[0]
    assert out[2].count("structure identical") == 1


def test_failed_event_query_is_not_a_failed_multiply(emu, tmp_path):
    """The block cache asks a released block's event whether its work is
    done.  A query that fails (seen on the GPU when the thread that had
    recorded the event was gone) must only pass the block over: the error
    that it leaves with the runtime must not fail the launches that follow."""
    A = gen.uniform8(m=64, per_row=4, seed=3, n=64)
    calls = [call(A, A, "--repeat", "4", env={"EMU_QUERY_ERROR": str(n)}) for n in (1, 2, 3)]
    for out in run_emu_all(emu, tmp_path, *calls):
        assert out.count("structure identical") == 4


def test_server_batches_and_admission(emu, tmp_path):
    """Served form on the CPU: the same product submitted many times to a
    server with a small maximum batch and a budget of about two outputs,
    so batches are split, admitted one after another and run on both
    lanes; every result must equal the host product.  A budget below one
    output must fail every request with out-of-memory."""
    A = gen.powerlaw(m=1000, seed=8)
    C = oracle.spgemm(A, A)
    need = C.nnz * 12
    out = run_emu(emu, tmp_path, A, A, "--serve", "5", str(2 * need + 64), "2")
    assert out.count("structure identical") == 5
    assert "served 5" in out
    res = subprocess.run([emu, str(tmp_path / "a.csr"), str(tmp_path / "b.csr"), "--serve", "2", str(need // 2), "2"],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=600)
    assert res.returncode == 0, res.stdout[-3000:]
    assert res.stdout.count("out of device memory") == 2
