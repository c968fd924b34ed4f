"""The generated code of the down kernels and of the persistent gate/up
kernels, checked on the CPU.

ksl_moe_down streams each wave's weight tiles (with their scale / zero-point
pairs) into registers by ordinary loads, whose waits the compiler places,
reads its activations from LDS and sends its outputs through a per-wave LDS
staging area. The device assembly of csrc/moe_gemm.hip is
built with the library's flags and a few workgroups of the form that a launch
picks (down_kernel up to 256 routed rows, else down_spread_kernel, whose spare
workgroups find the further chunks from the offsets) are run
through tests/gfx950_emu.py: every global, buffer and LDS access must stay in
its buffer (the weights, the tiled layout's trailing pair table, out2,
out3), and no address, stored value or MFMA operand may come from a register
whose load had not landed (the compiler's waits are checked, not assumed).
Shapes: the 256-token layer (one chunk, up to two M tiles), 1024 tokens (four
M tiles, several chunks per expert), a Zipf routing of 1024 tokens (experts of
a few to many chunks), short calls, small / odd I (a 64-K tail group, the
largest I), and a grid planned for fewer rows than there are (several rounds).
Above 8192 routed rows a different kernel runs (moe_rbgemm.hip): ordinary
register loads for its weights, and inline-asm LDS reads of its activation
fragments, whose in-flight windows are checked below on the generated code.
The persistent gate/up kernels (one workgroup per CU walking several expert
column blocks, its consumers publishing row tables in LDS for its producer;
the wide form, above 16 rows per expert, with 64-row passes and the further
chunks appended to the item tables) are run the same way, the item table and
every wave's barrier count checked."""
from __future__ import annotations

import importlib.util
import os
import shutil
import struct
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)
import gfx950_emu as emu  # noqa: E402

ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "knivesysl-diffusion-xe_amd", "csrc")


def _build_flags():
    spec = importlib.util.spec_from_file_location("ksl_build", os.path.join(ROOT, "knivesysl-diffusion-xe_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod.HIPCC, mod.HIP_FLAGS


@pytest.fixture(scope="module")
def down_asm(tmp_path_factory):
    hipcc, flags = _build_flags()
    if not (os.path.exists(hipcc) or shutil.which(hipcc)):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("asm") / "moe_gemm.s")
    res = subprocess.run([hipcc, *flags, "-w", "--cuda-device-only", "-S", os.path.join(CSRC, "moe_gemm.hip"),
                          "-o", out], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-4000:]
    return out


# The launch plan of csrc/moe_gemm.hip (plan_down, kDnWaves, kDnMaxMt,
# launch_down_gl) restated for the emulated launches.
NW, MAX_MT, CUS = 8, 4, 256
DN_SPREAD_FROM = 256  # routed rows above which down_spread_kernel runs


def _plan(E, H, I):
    G = I // 64
    te = H // 16
    nsplit = max(1, min(-(-CUS // E), te))
    tpw = -(-te // nsplit)
    nsplit = -(-te // tpw)
    return nsplit, tpw, MAX_MT * 2 * G * 1024 + NW * 2 * 16 * 80  # activations, then the waves' output staging


def _chunk_of(bid, nsplit, counts):
    """(expert, first row within it, rows, column block) that spare workgroup
    number bid finds (find_row_block<1>, 64-row chunks), or None."""
    j = bid // 8
    blk = j // nsplit * 8 + bid % 8
    for e, m in enumerate(counts):
        n = max(0, -(-(int(m) - 64) // 64))
        if blk < n:
            m0 = (blk + 1) * 64
            return e, m0, min(int(m) - m0, 64), j % nsplit
        blk -= n
    return None


def _routing(E, T, tk, kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "uniform":
        ids = np.stack([rng.permutation(E)[:tk] for _ in range(T)])
    else:
        p = 1.0 / np.arange(1, E + 1) ** 1.1
        p /= p.sum()
        ids = np.stack([rng.choice(E, tk, replace=False, p=p) for _ in range(T)])
    return np.bincount(ids.ravel(), minlength=E)


CASES = [
    # E, H, I, T, tk, routing, layout (0 reference, 1 tiled), workgroups (from
    # E * nsplit on: those that search), row count of the plan (None: the true one)
    (128, 2816, 704, 23, 8, "uniform", 1, (0, 78, 255), None),
    (128, 2816, 704, 32, 8, "zipf", 0, (0, 1, 9), None),
    (128, 2816, 704, 256, 8, "uniform", 1, (0, 77, 255, 256), None),
    (128, 2816, 704, 1024, 8, "uniform", 0, (1, 128, 257), None),
    (128, 2816, 704, 1024, 8, "zipf", 1, (6, 7, 255, 256, 300, 511), None),
    (128, 2816, 704, 300, 8, "zipf", 1, (0, 257), 257),       # spare workgroups go several rounds
    (16, 256, 192, 64, 4, "uniform", 0, (0, 200), None),
    (16, 256, 192, 400, 4, "zipf", 0, (0, 200), 100),         # down_kernel walks chunks of one to four M tiles
    (2, 64, 1024, 64, 2, "uniform", 1, (0, 7), None),
    (2, 64, 1024, 200, 2, "uniform", 1, (0, 7, 8, 20), None),
]


@pytest.mark.parametrize("E,H,I,T,tk,routing,layout,wgs,planned", CASES)
def test_down_kernel_addresses_and_register_flow(down_asm, E, H, I, T, tk, routing, layout, wgs, planned, spread=None):
    G = I // 64
    counts = _routing(E, T, tk, routing, E + H + I)
    offsets = np.concatenate([[0], np.cumsum(counts)])
    nrows = int(counts.sum())
    nsplit, tpw, lds = _plan(E, H, I)
    assert nrows <= 8192  # larger routings run the row-block kernels
    planned = nrows if planned is None else planned
    spread = planned > DN_SPREAD_FROM if spread is None else spread
    first = E * nsplit
    # chunks after an expert's first, a multiple of 8
    grid = first + (-(-(planned // 64) // 8) * 8 * nsplit if spread else 0)
    if planned == nrows:  # one round: every chunk has its workgroup
        found = [_chunk_of(b, nsplit, counts) for b in range(grid - first)] if spread else []
        todo = {(e, m0, min(int(m) - m0, 64), h) for e, m in enumerate(counts) for m0 in range(64, int(m), 64)
                for h in range(nsplit)}
        assert not spread or (todo == {c for c in found if c} and len(todo) == sum(c is not None for c in found))
    name = "18down_spread_kernel" if spread else "11down_kernel"
    fn = f"_ZN3ksl12_GLOBAL__N_1{name}ILi{G // 2}ELb{G % 2}ELi{layout}EEEvNS0_6DnArgsE{'ii' if spread else ''}"
    ins, labels = emu.load_kernel(down_asm, fn)
    dyn = 16 if spread else 0  # find_row_block's static info words come first
    lds += dyn
    bufs, base = {}, 0x7F0000000000

    def alloc(name, size):
        nonlocal base
        bufs[name] = (base, base + size)
        base += ((size + 0xFFFFF) // 0x100000 + 16) * 0x100000
        return bufs[name][0]

    p_out2 = alloc("out2", nrows * I * 2)
    p_off = alloc("offsets", (E + 1) * 4)
    # the tiled layout's buffer: the weights, then the (scale, zero) pair table
    p_q = alloc("dn_q", E * H * I // 2 + (E * H * G * 4 if layout == 1 else 0))
    p_s = alloc("dn_s", E * H * G * 2)
    p_z = alloc("dn_z", E * H * G * 2)
    p_out3 = alloc("out3", nrows * H * 2)
    p_karg = alloc("kernarg", 352)
    p_sz = p_q + E * H * I // 2 if layout == 1 else 0
    # DnArgs (72 bytes), down_spread_kernel's two, then the first hidden argument
    # (the grid's block count)
    karg = struct.pack("<QQQQQQQiiii", p_out2, p_off, p_q, p_s, p_z, p_out3, p_sz, H, I, nsplit, tpw)
    karg += (struct.pack("<ii", first, E) if spread else b"") + struct.pack("<I", grid) + b"\0" * 60
    mem = {p_karg + k: struct.unpack("<I", karg[k:k + 4])[0] for k in range(0, len(karg), 4)}
    mem.update({p_off + 4 * e: int(offsets[e]) for e in range(E + 1)})
    checked = 0
    for wg in wgs:
        assert wg < grid
        waves = [emu.Wave(mem, p_karg, wg, wave_id, bufs, lds) for wave_id in range(NW)]
        emu.run_workgroup(ins, labels, waves)
        for w in waves:
            checked += w.accesses
            assert not w.errors, (wg, w.errors[:4])
        if wg >= first:  # two barriers per chunk (the search, the activations), one for the last search
            n = sum(_chunk_of(b, nsplit, counts) is not None
                    for b in range(wg - first, first + sum(map(int, counts)), grid - first))
            assert [w.barriers for w in waves] == [2 * n + 1] * NW, (wg, n, waves[0].barriers)
    assert checked > 0


SYNTHETIC = """synthetic:
	global_load_dwordx4 v[4:7], v[0:1], off
	v_mov_b64_e32 v[8:9], v[4:5]
	s_waitcnt vmcnt(0)
	global_load_dword v10, v[8:9], off
	s_endpgm
.Lfunc_end0:
"""


def test_emulator_flags_a_copied_in_flight_register(tmp_path):
    """The hazard the checks above exclude, planted in a four-line kernel: a
    loaded register copied before its wait and the copy used as an address."""
    path = tmp_path / "syn.s"
    path.write_text(SYNTHETIC)
    ins, labels = emu.load_kernel(str(path), "synthetic")
    buf = (0x7F0000000000, 0x7F0000100000)
    w = emu.Wave({}, 0x7F0000200000, 0, 0, {"buf": buf, "karg": (0x7F0000200000, 0x7F0000200100)}, 1024)
    w.v[0] = np.uint64(buf[0] & 0xFFFFFFFF) + np.arange(64, dtype=np.uint64) * np.uint64(16)
    w.v[1] = np.uint64(buf[0] >> 32)
    emu.run(ins, labels, w)
    assert any(e[0] == "POISONED ADDRESS load" for e in w.errors), w.errors


@pytest.mark.parametrize("layout", [0, 1])
def test_down_kernel_every_width(down_asm, layout):
    """Every instantiation of both forms (I = 64 .. 1024, with and without a
    64-K tail group) on a small routing: one workgroup each, same checks."""
    for G in range(1, 17):
        for spread in (False, True):
            test_down_kernel_addresses_and_register_flow(down_asm, 4, 128, 64 * G, 48, 2, "uniform", layout, (0, 5), None,
                                                         spread)


# ---- the row-block GEMMs (moe_rbgemm.hip): activation fragments read by asm
@pytest.fixture(scope="module")
def rb_asm(tmp_path_factory):
    hipcc, flags = _build_flags()
    if not (os.path.exists(hipcc) or shutil.which(hipcc)):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("asm") / "moe_rbgemm.s")
    res = subprocess.run([hipcc, *flags, "-w", "--cuda-device-only", "-S", os.path.join(CSRC, "moe_rbgemm.hip"),
                          "-o", out], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-4000:]
    return out


def _codegen_check():
    spec = importlib.util.spec_from_file_location(
        "ksl_codegen_check", os.path.join(ROOT, "knivesysl-diffusion-xe_amd", "codegen_check.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def _ahead_windows(lines):
    return _codegen_check().ahead_windows(lines)


def test_rb_gemm_ahead_reads_stay_untouched_in_flight(rb_asm):
    """Every row-block kernel instance (gate/up and down, both activations and
    both weight layouts): each asm LDS read of the next M tile's activation
    fragment keeps its four destination registers untouched, with no branch,
    until the s_waitcnt lgkmcnt(0) that retires it; seven such reads per
    32-K step of the full-block path."""
    cc = _codegen_check()
    asm = open(rb_asm).read()
    fns = cc.rb_gemm_functions(asm)
    assert len(fns) == 4
    for fn, ins in fns.items():
        reads, bad = cc.ahead_windows(ins)
        # 7 per 32-K step (gate/up: 4 steps per group; down: 4 + 2 for the 64-K tail)
        assert reads > 0 and reads % 7 == 0, (fn, reads)
        assert not bad, (fn, bad[:5])
    assert cc.check_rb_gemm(asm) == []  # what build.py runs before it links


def test_ahead_window_check_flags_a_touched_register():
    """The window check itself: a planted use of an in-flight destination, and
    a branch inside a window, are both reported."""
    ok = ["ds_read_b128 v[4:7], v2 offset:4096 ; ksl-ahead", "v_mfma_f32_16x16x32_f16 v[8:11], v[0:3], v[12:15], v[8:11]",
          "s_waitcnt lgkmcnt(0)", "v_mov_b32 v4, 0"]
    assert _ahead_windows(ok) == (1, [])
    touched = ["ds_read_b128 v[4:7], v2 offset:4096 ; ksl-ahead", "v_mov_b32 v30, v5", "s_waitcnt lgkmcnt(0)"]
    assert len(_ahead_windows(touched)[1]) == 1
    branch = ["ds_read_b128 v[4:7], v2 ; ksl-ahead", "s_cbranch_scc1 .LBB0_1", "s_waitcnt lgkmcnt(0)"]
    assert len(_ahead_windows(branch)[1]) == 1


# ---- gate/up, flowing ring (gateup_flow_kernel, gateup_flow_wide_kernel): one
# persistent workgroup per CU. The launch choice of csrc/moe_gemm.hip
# (launch_gateup, gateup_flow_workgroups, GuFlowShape, launch_gateup_flow,
# gu_flow_fill_table, gu_flow_add_chunks) restated for the emulated launches:
# NC = 11 consumer waves and one producer, ring depth 3, 176 columns per item.
GU_NC, GU_R, GU_MAXITEMS = 11, 3, 64


def _gu_flow_info_off(G, mtx=2):
    slot = 2 * GU_NC * 1024 + 4 * mtx * 1024  # weight blocks + the M tiles' activation blocks
    table = 4 * 16 * GU_NC * G * 2 if mtx == 2 else 5 * 16 * GU_NC * G  # zero-points fp16 or nibbles
    return GU_R * slot + 2 * table + 2 * 16 * mtx * 4


def _gu_flow_lds(G, mtx=2):
    return _gu_flow_info_off(G, mtx) + GU_MAXITEMS * 16


def _gu_flow_room(items, W, nb):
    """Chunks per XCD that every item table has room for beside its own items."""
    return (GU_MAXITEMS - 1 - -(-items // W)) * (W // 8) // nb


def _gu_flow_wide(E, nrows, items, W, nb, H):
    return nrows > 16 * E and _gu_flow_room(items, W, nb) >= 2 and _gu_flow_lds(H // 128, 4) <= 160 * 1024 - 64


def _gu_flow_chunks(w, W, nb, counts):
    """The wide form's further items of workgroup w: (expert, first row within it, rows, column block)."""
    chunks = [(e, m0, min(int(m) - m0, 64)) for e, m in enumerate(counts) for m0 in range(64, int(m), 64)]
    out, q = [], w // 8
    while q // nb * 8 + w % 8 < len(chunks):
        out.append((*chunks[q // nb * 8 + w % 8], q % nb))
        q += W // 8
    return out


def _gu_flow_workgroups(items, H):
    W = CUS - CUS % 8
    G = H // 128
    if items <= CUS or items > W * GU_MAXITEMS or G < 8 or _gu_flow_lds(G) > 160 * 1024 - 64:
        return 0
    return W


def _gu_flow_pair(items, W, nb):
    return items == 2 * W and (W // 8) % nb == 0 and (items // 8) % nb == 0 and W // nb <= 64


def _gu_flow_tiles(w, W, items, nb, counts, pair, cap=1 << 30):
    """Item tiles (expert * nb + column block) of workgroup w; an item has at most cap rows."""
    rm = (lambda b: (b % 8) * (items // 8) + b // 8) if items % 8 == 0 else (lambda b: b)
    tiles = [rm(w + k * W) for k in range(len(range(w, items, W)))]
    if pair:
        n = W // nb
        wj = [8 * nb * (j // 8) + j % 8 for j in range(n)]
        e1 = [rm(x) // nb for x in wj]
        e2 = [rm(x + W) // nb for x in wj]
        m1 = [min(int(counts[e]), cap) for e in e1]
        m2 = [min(int(counts[e]), cap) for e in e2]
        q = w // 8
        b, jm = q % nb, (q // nb) * 8 + w % 8
        r = sum(1 for j in range(n) if m1[j] > m1[jm] or (m1[j] == m1[jm] and e1[j] < e1[jm]))
        order2 = sorted(range(n), key=lambda j: (m2[j], e2[j]))
        tiles[1] = e2[order2[r]] * nb + b
    return tiles


def _sorted_rows(E, T, tk, kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "uniform":
        ids = np.stack([rng.permutation(E)[:tk] for _ in range(T)])
    else:
        p = 1.0 / np.arange(1, E + 1) ** 1.1
        p /= p.sum()
        ids = np.stack([rng.choice(E, tk, replace=False, p=p) for _ in range(T)])
    flat = ids.ravel()
    order = np.argsort(flat, kind="stable").astype(np.int64)
    return np.bincount(flat, minlength=E), order


GU_CASES = [
    # E, H, I, T, tk, routing, workgroups, limit of the wide form (None: the launch's)
    (128, 2816, 704, 256, 8, "uniform", (0, 77, 255), None),   # the 256-token layer: balanced pairs
    (128, 2816, 704, 250, 8, "zipf", (3, 200), None),          # items of many passes, balanced pairs
    (128, 2816, 704, 16, 2, "uniform", (0, 1, 130), None),     # mostly empty items
    (256, 1024, 704, 128, 8, "uniform", (0, 255), None),       # G = 8, the shortest passes; four items each (no pairs)
    (256, 3072, 352, 128, 8, "uniform", (5, 254), None),       # G = 24, the largest LDS, balanced pairs
    (192, 2816, 704, 256, 8, "uniform", (0, 100, 255), None),  # three items per workgroup
    # the wide form
    (128, 2816, 704, 741, 8, "uniform", (0,), None),           # three M tiles, balanced pairs, chunks of a few rows
    (128, 2816, 704, 1024, 8, "zipf", (3, 200), None),         # heavy experts in many chunks, empty ones
    (160, 1024, 704, 700, 8, "zipf", (7, 255), None),          # G = 8; up to three items and the chunks (no pairs)
    (128, 1024, 704, 300, 8, "zipf", (0, 9), 2400),            # as many rows as the limit: whole experts, no chunks
    (128, 1024, 704, 300, 8, "zipf", (0,), 2401),              # one fewer: chunks
]


def test_gateup_chunks_never_overflow_the_item_table():
    """The wide form's tables at the most rows its limit lets through, all of
    one expert or spread so that the chunks are most: less than the table's
    entries before the last, which holds their number."""
    for E, nb in ((128, 4), (65, 4), (512, 4), (72, 64), (9, 64), (5, 64), (257, 1), (4095, 4), (2, 300)):
        items, W = E * nb, 256
        room = _gu_flow_room(items, W, nb)
        if items <= CUS or items > W * GU_MAXITEMS or room < 2:
            continue
        rows = (room - 1) * 8 * 64 - 1
        few = min(E, max(1, rows // 65))
        for counts in ([rows] + [0] * (E - 1), [65] * few + [0] * (E - few), [0] * (E - few) + [rows // few] * few):
            for w in (0, 1, 7, 8, 247, 248, 255):
                n = len(range(w, items, W)) + len(_gu_flow_chunks(w, W, nb, counts))
                assert n < GU_MAXITEMS, (E, nb, w, n)


@pytest.mark.parametrize("E,H,I,T,tk,routing,wgs,limit", GU_CASES)
def test_gateup_flow_kernel_addresses_and_register_flow(down_asm, E, H, I, T, tk, routing, wgs, limit):
    """Every wave of a few workgroups of the form that the launch picks (SiLU):
    the consumers (wave 0 fills the item table, with the balanced second items,
    wave 1 appends the wide form's chunks, and each pass's successor token ids
    go to LDS) and the producer, whose direct global->LDS loads are addressed
    from those tables; all accesses in bounds, no poisoned address or operand,
    LDS within the launch's dynamic size, the item table as restated here (every
    row of every expert and column block in exactly one item), and the same
    number of barriers in every wave."""
    G = H // 128
    nb = I // 176
    items = E * nb
    W = _gu_flow_workgroups(items, H)
    assert W == 256, "the flowing kernel runs for this shape"
    pair = _gu_flow_pair(items, W, nb)
    counts, order = _sorted_rows(E, T, tk, routing, E + H + I + T)
    offsets = np.concatenate([[0], np.cumsum(counts)])
    nrows = T * tk
    assert nrows <= 8192  # larger ones run the row-block kernel
    wide = _gu_flow_wide(E, nrows, items, W, nb, H)
    mtx, cap = 2, 1 << 30
    limit = (_gu_flow_room(items, W, nb) - 1) * 8 * 64 if limit is None else limit
    name, tail = "18gateup_flow_kernel", "iii"
    if wide:
        mtx, name, tail = 4, "23gateup_flow_wide_kernel", "iiiii"
        if nrows < limit:
            cap = 64
    ins, labels = emu.load_kernel(down_asm, f"_ZN3ksl12_GLOBAL__N_1{name}ILi1ELi11EEEvNS0_6GuArgsE{tail}")
    lds = _gu_flow_lds(G, mtx)

    def item_list(w):  # (expert, first row within it, rows, column block)
        out = [(t // nb, 0, min(int(counts[t // nb]), cap), t % nb)
               for t in _gu_flow_tiles(w, W, items, nb, counts, pair, cap)]
        return out + (_gu_flow_chunks(w, W, nb, counts) if cap == 64 else [])

    lists = [item_list(w) for w in range(W)]
    assert max(map(len, lists)) < GU_MAXITEMS
    owned = sorted(((e, b, m0), m) for L in lists for e, m0, m, b in L)
    assert len({k for k, _ in owned}) == len(owned) and {(e, b) for (e, b, _), _ in owned} == \
        {(e, b) for e in range(E) for b in range(nb)}
    assert all(m0 % 64 == 0 and m == min(int(counts[e]) - m0, cap) for (e, b, m0), m in owned)
    assert sum(m for _, m in owned) == nrows * nb
    bufs, base = {}, 0x7F0000000000

    def alloc(name, size):
        nonlocal base
        bufs[name] = (base, base + size)
        base += ((size + 0xFFFFF) // 0x100000 + 16) * 0x100000
        return bufs[name][0]

    p_a16 = alloc("a16", T * H * 2)
    p_rows = alloc("sorted_rows", nrows * 4)
    p_off = alloc("offsets", (E + 1) * 4)
    p_q = alloc("gu_q", E * 2 * I * H // 2)
    p_s = alloc("gu_s", E * 2 * I * G * 2)
    p_z = alloc("gu_z", E * 2 * I * G * 2)
    p_out2 = alloc("out2", nrows * I * 2)
    p_karg = alloc("kernarg", 128)
    early = 1 if nrows >= E else 0
    karg = struct.pack("<QQQQQQQiiiiiiiii", p_a16, p_rows, p_off, p_q, p_s, p_z, p_out2, tk, I, H, early, W, items,
                       int(pair), E, limit)  # (the last two: the wide form's)
    assert len(karg) == 92
    karg += b"\0" * 4
    mem = {p_karg + k: struct.unpack("<I", karg[k:k + 4])[0] for k in range(0, len(karg), 4)}
    mem.update({p_off + 4 * e: int(offsets[e]) for e in range(E + 1)})
    mem.update({p_rows + 4 * r: int(order[r]) for r in range(nrows)})
    info_off = _gu_flow_info_off(G, mtx)

    def lds_i32(lds_map, addr):
        v = 0
        for k in range(4):
            byte, known = lds_map.get(addr + k, (0, False))
            assert known, ("unknown LDS byte", addr + k)
            v |= int(byte) << (8 * k)
        return v - (1 << 32) if v & 0x80000000 else v

    checked = 0
    for wg in wgs:
        assert wg < W
        waves = [emu.Wave(mem, p_karg, wg, wave_id, bufs, lds) for wave_id in range(GU_NC + 1)]
        emu.run_workgroup(ins, labels, waves)
        for w in waves:
            checked += w.accesses
            assert not w.errors, (wg, w.errors[:4])
        for k, (e, m0, m, b) in enumerate(lists[wg]):
            got = [lds_i32(waves[0].lds, info_off + 16 * k + 4 * f) for f in range(4)]
            assert got == [int(offsets[e]) + m0, m, e, b * 176], (wg, k, got)
        if wide:
            assert lds_i32(waves[0].lds, info_off + 16 * (GU_MAXITEMS - 1)) == len(lists[wg])
        # every wave takes the same barriers: the first, one more when the first
        # item has no rows (and a later one has), one per group of each pass
        npass = sum(-(-m // (16 * mtx)) for _, _, m, _ in lists[wg])
        late = 1 if lists[wg][0][2] == 0 and npass > 0 else 0
        assert [w.barriers for w in waves] == [1 + late + npass * G] * (GU_NC + 1), (wg, waves[0].barriers, npass)
    assert checked > 0
