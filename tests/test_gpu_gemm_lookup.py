"""The lookup GEMM (gemm_lookup.hip) at the edges of its tiles: tokens around
32 / 64 and the group sizes, weight rows around 64 and 128, K that is no
multiple of an iteration, both layouts and bit widths, split K and not.

Bar: max|y - ref| / max|ref| <= 2e-3 per output vector against the oracle,
the repository's parity bar (fp32 sums in another order, one fp16 rounding).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(pe, Y, ref, what):
    for i in range(ref.shape[0]):
        e = pe.rel_err(Y[i], ref[i])
        assert e <= 2e-3, f"{what}: row {i} rel_err {e}"


# (bits, N, K, M, the kernels that run): rows 1 past and short of a 64- / 128-row
# tile, tokens likewise, K with a lone 8 past an iteration, GI group sizes 32 and 40
CASES = [
    (4, 64, 64, 17, "x"), (4, 65, 72, 9, "x"), (4, 127, 1000, 33, "x"), (4, 130, 1096, 48, "x"),
    (4, 200, 2048, 49, "x"), (4, 63, 4096, 64, "x"), (4, 129, 128, 65, "x"), (4, 9100, 2048, 40, "x"),
    (4, 129, 136, 257, "x"), (4, 257, 1000, 300, "x"), (4, 1001, 1032, 513, "x"), (4, 3, 8, 270, "x"),
    (4, 640, 648, 511, "x"), (4, 9100, 2112, 230, "p"), (4, 3584, 2048, 300, "p"),
    # k_gemm_w4 of 2, 4 and 8 token tiles, one K step and more, GI groups of 40
    (4, 40000, 64, 64, "w"), (4, 33000, 128, 33, "w"), (4, 32900, 192, 129, "w"), (4, 32900, 192, 255, "w"), (4, 32900, 512, 255, "w"), (4, 20700, 192, 600, "w"),
    (4, 16500, 512, 300, "w"), (4, 9100, 2112, 400, "w"),
    (8, 64, 32, 17, "x"), (8, 66, 40, 10, "x"), (8, 130, 1000, 33, "x"), (8, 200, 2048, 64, "x"), (8, 9100, 2048, 20, "x"),
    (8, 129, 64, 257, "x"), (8, 255, 72, 290, "x"), (8, 1001, 1032, 300, "x"), (8, 9100, 2048, 200, "p"),
    (8, 5, 8, 266, "x"),
    # packed X over row tiles of 64 and 128 and token tiles of 64 and 128, one iteration of K and more, K split
    (4, 3329, 88, 403, "p"), (4, 12547, 176, 137, "p"), (4, 5309, 896, 198, "p"), (4, 3328, 4760, 282, "p"),
    (4, 8269, 304, 566, "p"), (4, 9321, 2968, 142, "p"), (8, 4235, 64, 791, "p"), (8, 7816, 128, 261, "p"),
    (8, 4678, 144, 441, "p"), (8, 8575, 360, 112, "p"), (8, 5761, 2432, 200, "p"), (8, 972, 2240, 1068, "p"),
    (8, 15645, 208, 627, "p"), (8, 9751, 296, 723, "p"),
]


@pytest.mark.parametrize("bits,N,K,M,kind", CASES)
def test_lookup_gemm_edges(pe, oracle, gpu_ctx, bits, N, K, M, kind):
    t = pe.synth_tensor(N, K, bits, seed=N + K + M)
    w = gpu_ctx.upload_tensor(t)
    X = pe.synth_x(M, K, seed=M)
    Y = gpu_ctx.gemm(w, X)
    ran = gpu_ctx.last_kernels()
    want = {"x": "k_gemm_lookup_x<", "p": "k_gemm_lookup<", "w": "k_gemm_w4<"}[kind]
    assert want in ran, ran
    _check(pe, Y, oracle.gemm(X, t.payload, N, K, bits, threads=8), f"{bits}-bit {M}x{N}x{K} ({ran})")
    w.free()


@pytest.mark.parametrize("bits,batch,N,K", [(4, 12, 300, 1032), (4, 7, 100, 16392), (4, 16, 9000, 4096), (8, 6, 8200, 1064),
                                            (8, 24, 70, 264)])
def test_lookup_gemv_batches(pe, oracle, gpu_ctx, bits, batch, N, K):
    """GEMV batches that the lookup GEMM takes."""
    t = pe.synth_tensor(N, K, bits, seed=N + batch)
    w = gpu_ctx.upload_tensor(t)
    X = pe.synth_x(batch, K, seed=batch)
    Y = gpu_ctx.gemv(w, X)
    assert "k_gemm_lookup_x<" in gpu_ctx.last_kernels()
    _check(pe, Y, oracle.gemm(X, t.payload, N, K, bits, threads=8), f"{bits}-bit gemv x{batch} {N}x{K}")
    w.free()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M", [20, 280])
def test_lookup_gemm_ragged_rows_end(pe, oracle, gpu_ctx, bits, M):
    """Where K is ragged, an iteration's last loads hold the next row's bytes:
    neither an infinite LUT entry that only those bytes select nor an
    infinity at the start of the next token reaches the result."""
    N, K = 70, 72
    t = 1 << bits
    rng = np.random.Generator(np.random.PCG64(bits + M))
    lut = np.sort(rng.normal(0, 0.02, (N, t)), axis=1).astype(np.float16)
    idx = rng.integers(0, t // 2, (N, K), dtype=np.uint8)
    lut[0::2, t // 2:] = np.inf   # even rows: upper half unused and infinite
    lut[1::2, :t // 2] = np.nan   # odd rows the other way round
    idx[1::2] += t // 2
    payload = pe.split_block_payload(lut, idx, bits)
    X = pe.synth_x(M, K, seed=3).copy()
    X[M // 2, :8] = np.float16(np.inf).view(np.uint16)
    w = gpu_ctx.upload(payload, N, K, bits)
    Y = gpu_ctx.gemm(w, X)
    ref = oracle.gemm(X, payload, N, K, bits, threads=4)
    keep = np.arange(M) != M // 2
    assert np.isfinite(Y[keep].view(np.float16)).all()
    _check(pe, Y[keep], ref[keep], "ragged")
    assert np.array_equal(np.isnan(Y[M // 2].view(np.float16)), np.isnan(ref[M // 2].view(np.float16)))
    w.free()


def test_lookup_gemm_scratch_over_streams(pe, gpu_ctx):
    """Packed calls and calls that split K, back to back on three streams and
    the context's own, twice, without a wait between them: each output is, bit
    for bit, that of the call made alone.  (All of them use scratch: packed X of
    up to 8 MB, partials of up to 2 MB.)"""
    import torch
    shapes = {"A": (14336, 4096), "B": (4096, 14336)}
    w = {n: gpu_ctx.upload_tensor(pe.synth_tensor(*s, 4, seed=77)) for n, s in shapes.items()}
    kinds = [("A", 203, "k_pack_x"), ("B", 24, "k_gemm_split_sum"), ("A", 256, "k_pack_x"), ("B", 300, "k_pack_x")]
    streams = [None] + [torch.cuda.Stream() for _ in range(3)]
    calls = []
    for rnd in range(2):
        for i, s in enumerate(streams):
            name, M, kernel = kinds[(i + rnd) % 4]
            X = torch.from_numpy(pe.synth_x(M, shapes[name][1], seed=100 * rnd + i).view(np.int16)).cuda()
            Y = torch.empty((2, M, shapes[name][0]), dtype=torch.int16, device="cuda")
            torch.cuda.synchronize()
            gpu_ctx.gemm_dev(w[name], X, M, Y[0], s)
            assert kernel in gpu_ctx.last_kernels(), gpu_ctx.last_kernels()
            torch.cuda.synchronize()
            calls.append((s, w[name], X, M, Y))
    for s, wt, X, M, Y in calls:
        gpu_ctx.gemm_dev(wt, X, M, Y[1], s)
    torch.cuda.synchronize()
    for i, (_, _, _, M, Y) in enumerate(calls):
        assert torch.equal(Y[0], Y[1]), f"call {i} (M={M})"
    for x in w.values():
        x.free()


def test_lookup_gemm_luts_past_2gib(pe, gpu_ctx):
    """More short 8-bit rows than 31-bit offsets reach LUTs of: the rows around
    the end of the first slab (64-row multiples of 512 bytes below 0x7F000000)
    and the last ones against fp32 torch, 2e-3 as above."""
    import torch
    N, K, M = 4_200_003, 8, 17
    g = torch.Generator(device="cuda").manual_seed(5)
    payload = torch.empty(N * (512 + K), dtype=torch.uint8, device="cuda")
    lut, idx = payload[:N * 512].view(torch.float16).view(N, 256), payload[N * 512:].view(N, K)
    for i in range(0, N, 1 << 20):
        part = lut[i:i + (1 << 20)]
        part.copy_(torch.randn(part.shape, generator=g, device="cuda") * 0.02)
    idx.copy_(torch.randint(0, 256, (N, K), generator=g, device="cuda", dtype=torch.uint8))
    X = torch.randn(M, K, generator=g, device="cuda").half()
    Y = torch.empty(M, N, dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    w = gpu_ctx.upload_dev(payload, N, K, 8)
    gpu_ctx.gemm_dev(w, X, M, Y)
    gpu_ctx.synchronize()
    assert "k_gemm_lookup_x<" in gpu_ctx.last_kernels()
    edge = 0x7F000000 // 512 // 64 * 64
    rows = torch.tensor([0, 1, edge - 1, edge, edge + 1, N - 2, N - 1], device="cuda")
    ref = X.float() @ torch.gather(lut[rows].float(), 1, idx[rows].long()).t()
    assert (Y[:, rows].float() - ref).abs().max() <= 2e-3 * ref.abs().max()
    w.free()


@pytest.mark.parametrize("batch,N,K", [(12, 300, 1032), (40, 256, 8192)])
def test_lookup_gemv_captured(pe, oracle, gpu_ctx, batch, N, K):
    """A GEMV of several vectors captured on the caller's stream: kernels alone,
    no K splits and no memory, and every replay takes the x that is there then,
    with eager calls (which split K at 8192) between the replays."""
    import torch
    t = pe.synth_tensor(N, K, 4, seed=9)
    w = gpu_ctx.upload_tensor(t)
    dX = torch.zeros((batch, K), dtype=torch.int16, device="cuda")
    dY = torch.empty((batch, N), dtype=torch.int16, device="cuda")
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        gpu_ctx.gemv_dev(w, dX, batch, dY, s)
    ran = gpu_ctx.last_kernels()
    assert "k_gemm_lookup_x<" in ran and "split" not in ran, ran
    for i in range(3):
        X = pe.synth_x(batch, K, seed=50 + i)
        dX.copy_(torch.from_numpy(X.view(np.int16)))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        ref = oracle.gemm(X, t.payload, N, K, 4, threads=8)
        _check(pe, dY.cpu().numpy().view(np.uint16), ref, f"replay {i}")
        _check(pe, gpu_ctx.gemv(w, X), ref, f"eager {i}")
    w.free()


# 8 bits, more than 256 tokens: k_gemm8 over GI groups of 40 and over split-block rows, tokens and rows
# that do not fill its 256 x 128 blocks; the unpacked lookup GEMM where that is ahead; 4 bits
@pytest.mark.parametrize("bits,N,K,M,kernel", [(8, 9100, 2048, 520, "k_gemm8<true>"), (8, 8200, 704, 600, "k_gemm8<false>"),
                                               (8, 1001, 1032, 300, "k_gemm_lookup_x<8"), (4, 1001, 1032, 513, "k_gemm_lookup_x<4, 2"), (8, 200, 2048, 70, "k_gemm_lookup_x<8"),
                                               (4, 16500, 512, 300, "k_gemm_w4<4"), (4, 1001, 1032, 270, "k_gemm_lookup_x<4")])
def test_gemm_captured(pe, oracle, gpu_ctx, bits, N, K, M, kernel):
    """gemm_dev captured on the caller's stream: one kernel and no memory; every
    replay takes the X that is there then, with eager calls (which pack X)
    between the replays.  Tokens at the edges of the blocks against the oracle."""
    import torch
    t = pe.synth_tensor(N, K, bits, seed=N)
    w = gpu_ctx.upload_tensor(t)
    dX = torch.zeros((M, K), dtype=torch.int16, device="cuda")
    dY = torch.empty((M, N), dtype=torch.int16, device="cuda")
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        gpu_ctx.gemm_dev(w, dX, M, dY, s)
    ran = gpu_ctx.last_kernels()
    assert ran.startswith(kernel) and "+" not in ran, ran
    rows = sorted({0, 1, 31, 32, 63, 64, 65, 127, 128, 255, 256, 257, 511, 512, M // 2, M - 2, M - 1} & set(range(M)))
    for i in range(3):
        X = pe.synth_x(M, K, seed=70 + i)
        dX.copy_(torch.from_numpy(X.view(np.int16)))
        dY.fill_(-1)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        ref = oracle.gemm(np.ascontiguousarray(X[rows]), t.payload, N, K, bits, threads=8)
        Y = dY.cpu().numpy().view(np.uint16)
        _check(pe, Y[rows], ref, f"replay {i} ({ran})")
        eager = gpu_ctx.gemm(w, X)
        _check(pe, Y, eager, f"replay {i} against eager")
        _check(pe, eager[rows], ref, f"eager {i}")
    del g
    w.free()
