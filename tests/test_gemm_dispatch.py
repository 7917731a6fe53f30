"""The GEMM's dispatch on the CPU, with the fake HIP runtime: which kernels a
call launches and with which pointers, at sizes no GPU test can hold."""
import pytest

import fake_hip


def payload_bytes(n, k, bits):
    return n * (2 << bits) + n * k * bits // 8


def launches(hip, pe, bits, n, k, ms, x_bytes=None):
    """gemm_dev of each M: (layout's group rows, [kernel, rows, first row's LUT and index offset in the weight,
    first row of Y] of each lookup launch, every kernel)."""
    ctx = pe.Context(0)
    w = ctx.upload_dev(fake_hip.Tensor(hip, payload_bytes(n, k, bits)), n, k, bits)
    out = []
    for m in ms:
        x, y = fake_hip.Tensor(hip, m * k * 2), fake_hip.Tensor(hip, m * n * 2)
        hip.clear()
        ctx.gemm_dev(w, x, m, y)
        lk = [ln for ln in hip.launches if ln.lk]
        first = [ln.lk for ln in lk]
        base = min((a.lut for a in first), default=0)
        out.append({"G": first[0].G if first else 0, "kernels": [ln.name for ln in hip.launches],
                    "lk": [[ln.name, ln.lk.N, ln.lk.lut - base, ln.lk.idx - base, (ln.lk.Y - y.address) // 2 % n]
                           for ln in lk],
                    "room": [[hip.room(a.lut), hip.room(a.idx), hip.room(a.X), hip.room(a.Y)] for a in first]})
    return out


# GI weights just below the layout's 2 GiB end, past the bytes a split-block slab takes:
# 4-bit in 32-row groups (2 132 803 584 bytes), 8-bit in 32-row groups (2 139 095 040)
@pytest.mark.parametrize("bits,n,k", [(4, 32768, 130112), (8, 8192, 260608)])
def test_gi_weights_are_never_cut(bits, n, k):
    """The rows of GI weights lie in groups, so a slab's first row is no
    row-multiple from the base: every launch (there may be several, each of some
    tokens) takes them all."""
    for got in fake_hip.call(__name__, "launches", bits, n, k, [17, 300]):
        assert got["G"] == 32 and got["lk"]
        assert all(x[1:] == [n, 0, 0, 0] for x in got["lk"]), got


@pytest.mark.parametrize("bits,n,k", [(4, 33000, 130112), (8, 70000, 32768), (8, 4_200_003, 8)])
def test_split_block_slabs(bits, n, k):
    """Split-block weights past 2 GiB of index or LUT bytes: slabs of whole
    tiles that cover every row once, each launch's bytes below 2 GiB."""
    row, lut = k * bits // 8, 2 << bits
    for got in fake_hip.call(__name__, "launches", bits, n, k, [17, 40]):
        assert got["G"] == 0 and len(got["lk"]) > 1
        at = 0
        for _, rows, lut_at, idx_at, y_at in got["lk"]:
            assert lut_at == at * lut and idx_at == n * lut + at * row and y_at == at
            assert rows * max(row, lut) < 1 << 31 and (rows % 64 == 0 or at + rows == n)
            at += rows
        assert at == n


@pytest.mark.parametrize("bits,n,k,taken", [(4, 3, (1 << 24) - 8, True), (8, 3, (1 << 24) - 8, True),
                                            (4, 3, 1 << 24, False), (8, 3, 1 << 24, False), (4, 70, 1 << 25, False),
                                            (8, 1, 1 << 26, False), (4, 2, 1 << 28, False)])
def test_rows_past_the_offsets_go_to_passes(bits, n, k, taken):
    """64 tokens of x from 2 GiB on, and row tiles past 2 GiB of indices: the
    GEMV passes, which address them by 64-bit pointers."""
    for got in fake_hip.call(__name__, "launches", bits, n, k, [17, 40, 64, 70]):
        assert bool(got["lk"]) == taken and got["kernels"], got
        for x in got["lk"]:
            assert x[1] == n


STREAM = 0x77000  # a stream of the caller's


def plans(hip, pe, bits, n, k, ms, hows):
    """For each M and each of "own", "lent", "capture", "noalloc own", "noalloc lent" (gemm_dev, gemm_dev_noalloc) and
    "gemv own", "gemv lent", "gemv capture": [kernel, grid, K per split] of each launch, and the allocations and frees."""
    ctx = pe.Context(0)
    w = ctx.upload_dev(fake_hip.Tensor(hip, payload_bytes(n, k, bits)), n, k, bits)
    out = []
    for m in ms:
        x, y = fake_hip.Tensor(hip, m * k * 2), fake_hip.Tensor(hip, m * n * 2)
        row = {}
        for how in hows:
            hip.clear()
            stream = None if how.endswith("own") else STREAM
            hip.lib.fake_set_capturing(STREAM if how.endswith("capture") else None)
            if how.startswith("noalloc"):
                ctx.gemm_dev_noalloc(w, x, m, y, stream)
            elif how.startswith("gemv"):
                ctx.gemv_dev(w, x, m, y, stream)
            else:
                ctx.gemm_dev(w, x, m, y, stream)
            row[how] = {"kernels": [[ln.name.replace("prism::", "").replace("void ", "").split("(")[0], ln.grid,
                                     ln.lk.per_split if ln.lk else 0] for ln in hip.launches],
                        "memory": [ln for ln in hip.log() if "malloc" in ln or "free" in ln]}
        out.append(row)
    return out


@pytest.mark.parametrize("bits,n,k", [(4, 4096, 14336), (4, 14336, 4096), (8, 4096, 14336), (4, 2000, 2048)])
def test_noalloc_is_planned_without_a_price_for_scratch(bits, n, k):
    """The static scratch costs nothing, so a caller's stream gets the plan of
    the context's."""
    for row in fake_hip.call(__name__, "plans", bits, n, k, [24, 64, 96, 200, 300], ["own", "noalloc own", "noalloc lent"]):
        assert row["noalloc lent"]["kernels"] == row["noalloc own"]["kernels"] == row["own"]["kernels"]
        assert row["noalloc lent"]["memory"] == []


@pytest.mark.parametrize("bits,n,k", [(4, 14336, 4096), (8, 14336, 4096), (4, 4096, 14336), (8, 1001, 1032), (4, 64, 8192)])
def test_a_captured_call_is_kernels_alone(bits, n, k):
    """Under the capture of a caller's stream nothing is allocated or freed, and
    no kernel needs scratch."""
    ms = [9, 16, 24, 33, 64, 96, 203, 256, 257, 300, 1024, 2048]
    for row in fake_hip.call(__name__, "plans", bits, n, k, ms, ["capture", "gemv capture"]):
        for how in row:
            assert row[how]["memory"] == [] and row[how]["kernels"]
            assert not [x for x in row[how]["kernels"] if "pack" in x[0] or "split_sum" in x[0]], row[how]


@pytest.mark.parametrize("n,k", [(14336, 4096), (4864, 896), (6144, 4096)])
def test_no_split_where_unsplit_is_faster(n, k):
    """4-bit calls of 49..64 tokens on row blocks that fill a good part of the
    CUs: K is not split (14336 x 4096 14.9 us against 22.4 in two splits, 4864
    x 896 5.4 against 8.3), and so a caller's stream allocates nothing."""
    for row in fake_hip.call(__name__, "plans", 4, n, k, [48, 49, 56, 64], ["own", "lent"]):
        for how in row:
            assert [x[0].split("<")[0] for x in row[how]["kernels"]] == ["k_gemm_lookup_x"], row[how]
            assert row[how]["memory"] == []


def _names(row):
    return [x[0].split("<")[0] for x in row["kernels"]]


@pytest.mark.parametrize("n,k,m", [(2752, 1792, 128), (1664, 2088, 99), (4224, 5504, 82), (4608, 3152, 199), (1480, 4224, 181)])
def test_blocks_of_32_tokens_above_64(n, k, m):
    """Matrices of a few thousand rows, over 64 tokens: twice the blocks, of 32
    tokens each, fill the CUs better than blocks of 64 (2752 x 1792, 128 tokens 7.0
    against 9.8 us, 4608 x 3152, 199 tokens 22.7 against 30.5)."""
    for row in fake_hip.call(__name__, "plans", 4, n, k, [m], ["own", "lent"]):
        for how in row:
            assert row[how]["kernels"][0][0].startswith("k_gemm_lookup_x<4, 1"), row[how]


@pytest.mark.parametrize("n,k", [(151936, 896), (65536, 1024)])
def test_tall_matrices_take_register_decode(n, k):
    """An LM head over 33..256 tokens: blocks of k_gemm_w4 fill the CUs several
    times over, where each 64 rows of the lookup GEMM build tables for 448
    index bytes a row (151936 x 896, 64 tokens 34.7 against 65.3 us)."""
    for row in fake_hip.call(__name__, "plans", 4, n, k, [33, 48, 64, 96, 128, 256], ["own", "lent", "capture"]):
        for how in row:
            assert _names(row[how]) == ["k_gemm_w4"], row[how]


def test_the_plans_measured_fastest():
    """The plans that were fastest, or within 1 % of it, when each was measured
    (14336 x 4096 and 4096 x 14336, 4 bits), by kernel and tile."""
    want = {(14336, 4096): {33: "k_gemm_lookup_x<4, 2", 64: "k_gemm_lookup_x<4, 2", 256: "k_gemm_lookup<4, 4, 2",
                            512: "k_gemm_lookup<4, 4, 2", 2048: "k_gemm_lookup<4, 4, 2"},
            (4096, 14336): {24: "k_gemm_lookup_x<4, 1", 203: "k_gemm_lookup_x<4, 2", 1024: "k_gemm_lookup<4, 4, 2"}}
    for (n, k), kernels in want.items():
        for (m, name), row in zip(kernels.items(), fake_hip.call(__name__, "plans", 4, n, k, list(kernels), ["own"])):
            assert any(x[0].startswith(name) for x in row["own"]["kernels"]), (n, k, m, row)


# (bits, N, K, vectors): those that GEMV passes take on a caller's stream and under capture, where K
# is not split, and those that they take everywhere
@pytest.mark.parametrize("bits,n,k,ms,own_too", [
    (4, 256, 8192, [5, 6, 8], True), (4, 256, 8192, [9, 12, 16], False), (8, 256, 8192, [9, 16, 24], False),
    (8, 512, 16384, [5, 8, 9], False), (4, 4096, 4096, [9], True), (8, 1024, 4096, [9, 12], False),
    (4, 4096, 14336, [5, 8, 9], False), (8, 4864, 896, [9, 16], True), (4, 1024, 1024, [5, 8], True)])
def test_passes_where_they_are_faster(bits, n, k, ms, own_too):
    """Few rows of a long K, which the lookup GEMM needs its K splits for (256 x
    8192, 8 bits, 8 vectors on a caller's stream 6.8 us in passes, 22.7 in the
    lookup GEMM), and matrices that one pass of the matrix-core GEMV takes
    (4096 x 4096, 9 vectors 6.9 us against 8.4)."""
    hows = ["gemv lent", "gemv capture", "lent", "capture"] + (["own", "gemv own"] if own_too else [])
    for row in fake_hip.call(__name__, "plans", bits, n, k, ms, hows):
        for how in row:
            assert all(x.startswith("k_gemv_") for x in _names(row[how])) and row[how]["memory"] == [], (how, row[how])


@pytest.mark.parametrize("bits,n,k,ms", [(4, 14336, 4096, [9, 16]), (8, 14336, 4096, [9, 16]), (4, 2048, 2048, [9, 16, 24]),
                                         (4, 896, 4864, [16, 24, 32]), (8, 10752, 1056, [8, 16]), (4, 151936, 896, [17, 32]),
                                         (4, 14592, 13184, [11, 14])])
def test_the_lookup_gemm_where_it_is_faster(bits, n, k, ms):
    """The other side: one round of row blocks, several tile passes, two passes
    of the matrix-core GEMV; on every stream alike."""
    for row in fake_hip.call(__name__, "plans", bits, n, k, ms, ["own", "lent", "capture"]):
        for how in row:
            assert _names(row[how])[0] == "k_gemm_lookup_x", (how, row[how])


def without_memory(hip, pe, n, k, m, stream):
    ctx = pe.Context(0)
    w = ctx.upload_dev(fake_hip.Tensor(hip, payload_bytes(n, k, 4)), n, k, 4)
    x, y = fake_hip.Tensor(hip, m * k * 2), fake_hip.Tensor(hip, m * n * 2)
    hip.lib.fake_refuse(1)
    hip.clear()
    ctx.gemm_dev(w, x, m, y, stream)
    return [[ln.name, ln.lk.P if ln.lk else 0] for ln in hip.launches]


@pytest.mark.parametrize("stream", [None, STREAM])
@pytest.mark.parametrize("n,k,m", [(4096, 14336, 24), (14336, 4096, 300)])
def test_no_memory_for_scratch(n, k, m, stream):
    """A plan whose scratch cannot be had (K split; X packed): the kernel that needs none."""
    launched = fake_hip.call(__name__, "without_memory", n, k, m, stream)
    assert len(launched) == 1 and "k_gemm_lookup_x" in launched[0][0] and not launched[0][1]


@pytest.mark.parametrize("n,k,m,kernel", [(14336, 4096, 512, "k_gemm8"), (14336, 4096, 2048, "k_gemm8"), (14336, 4096, 300, "k_gemm_lookup_x"),
                                          (4096, 4096, 2048, "k_gemm8"), (4096, 4096, 512, "k_gemm_lookup_x"), (151936, 896, 512, "k_gemm8"),
                                          (1001, 1032, 2048, "k_gemm_lookup_x")])
def test_captured_8_bit_prefills(n, k, m, kernel):
    """The kernel without scratch that each was measured fastest on (14336 x
    4096, 2048 tokens 441 us against 577); K % 64 != 0 has one only."""
    for row in fake_hip.call(__name__, "plans", 8, n, k, [m], ["capture"]):
        assert _names(row["capture"]) == [kernel]


def grids(hip, pe, bits, n, k, m, how):
    ctx = pe.Context(0)
    w = ctx.upload_dev(fake_hip.Tensor(hip, payload_bytes(n, k, bits)), n, k, bits)
    x, y = fake_hip.Tensor(hip, m * k * 2), fake_hip.Tensor(hip, m * n * 2)
    hip.clear()
    hip.lib.fake_set_capturing(STREAM if how == "capture" else None)
    ctx.gemm_dev(w, x, m, y, None if how == "own" else STREAM)
    return [[ln.name, ln.grid[0] * ln.threads, ln.lk.M if ln.lk else 0, (ln.lk.Y - y.address) // (2 * n) if ln.lk else 0]
            for ln in hip.launches]


@pytest.mark.parametrize("how", ["own", "lent", "capture"])
@pytest.mark.parametrize("bits,n,k,m", [(8, 151936, 904, 150_001), (4, 151936, 904, 150_001), (8, 1_000_003, 8, 40_000)])
def test_launches_of_less_than_2_32_threads(bits, n, k, m, how):
    """More outputs than one launch has threads for: several, of some tokens each,
    that cover every token once."""
    got = fake_hip.call(__name__, "grids", bits, n, k, m, how)
    assert all(x[1] < 1 << 32 for x in got), got
    at = 0
    for name, _, tokens, first in got:
        if "k_gemm_lookup" in name:
            assert first == at
            at += tokens
    assert at == m
