"""The folded contraction kernels over the layouts, edges and launch forms they choose between:
integer inputs, every output bit-exact against a device fp64 product of the operands permuted to
[M][K] x [K][N].  C starts as NaN, so an output that no workgroup writes shows."""
import pytest

pytestmark = pytest.mark.gpu

AXES = ("mh", "ml", "nh", "nl", "kh", "kl")


def _check(torch, mm, ext, orders, seed=0, offsets=(0, 0, 0), pads=(0, 0, 0), **call):
    """Contract integer operands laid out in the given axis orders (`offsets`: elements each tensor
    starts into its buffer; `pads`: elements left free after each run of its innermost axis)."""
    ext = dict(zip(AXES, ext))
    orders = [o.split() for o in orders]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7000 + seed)

    def make(order, off, pad, operand):
        shape = [ext[a] for a in order]
        strides, step = [], 1
        for i in range(len(shape) - 1, -1, -1):
            strides.insert(0, step)
            step *= shape[i]
            if i == len(shape) - 1:
                step += pad
        n = off + sum((s - 1) * t for s, t in zip(shape, strides)) + 1
        if operand:
            # what lies between and before the elements is NaN: it must reach no output
            buf = torch.full((n,), float("nan"), dtype=torch.float16, device="cuda")
            x = buf.as_strided(shape, strides, off)
            x.copy_(torch.randint(-4, 5, shape, generator=gen, device="cuda", dtype=torch.int8))
        else:
            x = torch.full((n,), float("nan"), dtype=torch.float32, device="cuda").as_strided(shape, strides, off)
        return x, dict(zip(order, strides))

    (A, sa), (B, sb), (C, sc) = (make(o, off, pad, t < 2)
                                 for t, (o, off, pad) in enumerate(zip(orders, offsets, pads)))
    d = mm.ContractDesc()
    for f, h in (("m_ext", "m"), ("n_ext", "n"), ("k_ext", "k")):
        getattr(d, f)[0], getattr(d, f)[1] = ext[h + "h"], ext[h + "l"]
    for f, s, h in (("a_m_stride", sa, "m"), ("a_k_stride", sa, "k"), ("b_k_stride", sb, "k"), ("b_n_stride", sb, "n"),
                    ("c_m_stride", sc, "m"), ("c_n_stride", sc, "n")):
        getattr(d, f)[0], getattr(d, f)[1] = s[h + "h"], s[h + "l"]
    M, N, K = (ext[h + "h"] * ext[h + "l"] for h in "mnk")
    print(f"[fold] {ext} {orders} offsets {offsets} pads {pads}", flush=True)
    mm.contract(d, A, B, C, **call)
    torch.cuda.synchronize()
    A2 = A.permute(*[orders[0].index(a) for a in ("mh", "ml", "kh", "kl")]).reshape(M, K).double()
    B2 = B.permute(*[orders[1].index(a) for a in ("kh", "kl", "nh", "nl")]).reshape(K, N).double()
    T = (A2 @ B2).reshape(ext["mh"], ext["ml"], ext["nh"], ext["nl"])
    T = T.permute(*[("mh", "ml", "nh", "nl").index(a) for a in orders[2]]).float()
    assert torch.equal(C, T), f"{int((C != T).sum().item())} of {M * N} outputs differ"
    return d, A, B, C, T


A_MID = "mh kh ml kl"  # K contiguous, k between the m sub-indices
# N-contiguous B beside a K-major A.  (extents mh ml nh nl kh kl; orders of A, B, C.)  kl 64 and 128:
# K tiles inside one block; others per lane, K ending inside the last tile (2 x 8: one tile).  nl 70, 17
# and 2047: the chunk across N.  nh > 1: columns in blocks of 24 or 32.  The last five exchange the
# operands (A m-contiguous, B K-major), number K in its other order (kh innermost), and store C
# m-contiguous; 2048 and up fill rounds of the 256x256, 128x128 and 64x64 tiles.
NCONTIG = [
    ((2, 33, 1, 70, 3, 40), (A_MID, "kh kl nh nl", "mh ml nh nl")),
    ((2, 33, 1, 17, 2, 8), (A_MID, "kh kl nh nl", "mh ml nh nl")),
    ((2, 130, 1, 264, 2, 64), (A_MID, "kh kl nh nl", "mh ml nh nl")),
    ((3, 130, 1, 2047, 2, 128), (A_MID, "kh kl nh nl", "mh ml nh nl")),
    ((2, 130, 3, 24, 2, 128), (A_MID, "nh kh kl nl", "mh ml nh nl")),
    ((2, 300, 9, 32, 5, 24), (A_MID, "kh nh kl nl", "nh mh ml nl")),
    ((2, 300, 9, 32, 5, 24), (A_MID, "kl kh nh nl", "ml mh nl nh")),
    ((8, 256, 1, 2048, 2, 64), (A_MID, "kh kl nh nl", "mh ml nh nl")),
    ((16, 300, 1, 4095, 2, 72), (A_MID, "kh kl nh nl", "mh ml nh nl")),
    ((8, 1024, 1, 4096, 32, 128), (A_MID, "kh kl nh nl", "mh ml nh nl")),
    ((1, 264, 2, 130, 2, 64), ("kh kl mh ml", "nh kh nl kl", "mh ml nh nl")),
    ((1, 263, 2, 130, 3, 40), ("kh kl mh ml", "nh kh nl kl", "nh nl mh ml")),
    ((2, 130, 1, 264, 64, 3), ("mh kl ml kh", "kl kh nh nl", "mh ml nh nl")),
    ((2, 130, 1, 264, 3, 72), (A_MID, "kh kl nh nl", "nh nl mh ml")),
    ((2, 700, 1, 1000, 2, 64), (A_MID, "kh kl nh nl", "nh nl mh ml")),
]


@pytest.mark.parametrize("case", NCONTIG, ids=lambda c: "x".join(map(str, c[0])) + "-" + c[1][2].replace(" ", ""))
def test_fold_n_contiguous(mm, cuda, case):
    _check(cuda, mm, *case)


@pytest.mark.parametrize("pads", [(8, 8, 0), (8, 3, 0), (0, 5, 1), (8, 8, 4)], ids=str)
def test_fold_n_contiguous_padding(mm, cuda, pads):
    """Free elements after A's k runs, B's n rows and C's rows (C rows off 16-byte alignment)."""
    _check(cuda, mm, (2, 300, 1, 261, 3, 72), (A_MID, "kh kl nh nl", "mh ml nh nl"), pads=pads)
    _check(cuda, mm, (2, 300, 1, 264, 3, 128), (A_MID, "kh kl nh nl", "mh ml nh nl"), pads=pads, offsets=(0, 0, 1))


# k blocks that are no multiple of 8, both operands K-major: the chunk at a block's end is zeroed past
# it in LDS (one to seven elements), the last chunk of K gathered.  kl 3 to 9: several blocks in one K
# tile; 63 and 65: one short of and past a tile; kh 1: the only block's end is K's end; one K tile (3 x
# 5, 1 x 13) and many; the 64x64, 128x128 and 256x256 tiles; C n-contiguous, m-contiguous, element by
# element (nl 301, ml 301).  The free elements after each k run are NaN and sit inside the chunks.
PADDED_K = [(2, 130, 3, 70, kh, kl) for kh, kl in
            ((3, 5), (1, 13), (40, 3), (30, 4), (23, 6), (19, 7), (17, 9), (5, 25), (3, 50), (2, 63), (3, 65), (2, 100),
             (1, 1001), (6, 127))] + [
    (2, 301, 3, 301, 3, 25), (8, 256, 8, 256, 3, 50), (16, 300, 13, 315, 2, 100), (16, 512, 16, 512, 3, 25),
    (16, 512, 16, 512, 41, 100)]


@pytest.mark.parametrize("ext", PADDED_K, ids=lambda e: "x".join(map(str, e)))
@pytest.mark.parametrize("c_order", ["mh ml nh nl", "mh nh nl ml"])
def test_fold_padded_k_blocks(mm, cuda, ext, c_order):
    pads = (0, 0, 0) if ext[5] == 100 else (3, 5, 0)
    _check(cuda, mm, ext, (A_MID, "nh kh nl kl", c_order), pads=pads, seed=ext[5])


@pytest.mark.parametrize("kl", [5, 25, 100, 71])
def test_fold_padded_k_blocks_n_contiguous(mm, cuda, kl):
    """The same beside an N-contiguous B, whose k rows past a block's end are not loaded."""
    for nl, pads in ((264, (3, 0, 0)), (261, (1, 7, 0)), (17, (0, 0, 0))):
        _check(cuda, mm, (2, 130, 1, nl, 3, kl), (A_MID, "kh kl nh nl", "mh ml nh nl"), pads=pads, seed=kl)


# the gathering kernel: k runs of 3 one after another in both operands, as given and exchanged (K from 2048);
# an A strided along K beside a K-major B and a B strided along N beside a K-major A; short padded K
GATHERED = [((2, 130, 3, 70, 682, 3), (A_MID, "nh nl kh kl")), ((2, 130, 3, 70, 683, 3), (A_MID, "nh nl kh kl")),
            ((1, 40, 3, 300, 683, 3), (A_MID, "nh nl kh kl")), ((2, 130, 3, 70, 2, 40), ("mh ml kl kh", "nh nl kh kl")),
            ((2, 130, 2, 70, 3, 40), ("mh kh ml kl", "kh kl nl nh")), ((2, 130, 3, 70, 2, 20), (A_MID, "nh kh nl kl")),
            ((2, 130, 1, 264, 2, 20), (A_MID, "kh kl nh nl"))]


@pytest.mark.parametrize("case", GATHERED, ids=lambda c: "x".join(map(str, c[0])))
@pytest.mark.parametrize("c_order", ["mh ml nh nl", "nh nl mh ml", "mh nh nl ml"], ids=lambda o: o.replace(" ", ""))
def test_fold_gathered(mm, cuda, case, c_order):
    _check(cuda, mm, case[0], (*case[1], c_order))


@pytest.mark.parametrize("kl", [40, 64, 100], ids=lambda k: f"kl{k}")
@pytest.mark.parametrize("offsets", [(1, 0, 0), (0, 3, 1), (7, 5, 0)], ids=str)
def test_fold_unaligned_operands(mm, cuda, kl, offsets):
    """K-major operands at 2-byte alignment, rows and blocks at odd strides."""
    _check(cuda, mm, (2, 130, 3, 70, 3, kl), (A_MID, "nh kh nl kl", "mh ml nh nl"), pads=(1, 3, 0), offsets=offsets,
           seed=kl)
    _check(cuda, mm, (2, 130, 1, 264, 3, kl), (A_MID, "kh kl nh nl", "mh ml nh nl"), pads=(1, 1, 0), offsets=offsets,
           seed=kl)


@pytest.mark.parametrize("kl", [96, 128])
@pytest.mark.parametrize("nl", [300, 1030], ids=["given", "exchanged"])
def test_fold_wide(mm, cuda, kl, nl):
    """64-bit addresses (2 GiB from A's first element to its last), K tiles in one block and crossing
    blocks, edges of the 256x256 tile, the operands as given and exchanged for their m-contiguous C."""
    _check(cuda, mm, (8, 140, 1, nl, 4, kl), (A_MID, "nh kh nl kl", "mh nh nl ml"), pads=(1 << 18, 0, 0), seed=nl)
    cuda.cuda.empty_cache()


KM = (A_MID, "nh kh nl kl", "mh nh nl ml")
NM = (A_MID, "kh kl nh nl", "mh ml nh nl")
# K splits, with and without a workspace, on the square tiles: 1, 16, 32, 33, 64 and 65 rows on either side, ends
# of N inside a tile, K blocks per tile, per lane and padded, a split of a partly filled last round (272 tiles
# of 256 x 256); and on the skinny tiles, streams of 64 MiB and more (K tiles inside one block) against 16, 33,
# 17, 64, 30 and 24 rows (the last six; NT loads from 96 MiB)
SPLITS = [((1, 1, 4, 300, 20, 128), KM), ((4, 300, 1, 16, 20, 128), KM), ((4, 301, 1, 32, 33, 72), KM),
          ((3, 11, 4, 300, 20, 100), KM), ((2, 32, 4, 1024, 24, 100), KM), ((5, 13, 4, 300, 20, 128), KM),
          ((1, 16, 1, 1027, 20, 128), NM), ((2, 32, 1, 2045, 31, 72), NM), ((2, 8, 4, 64, 31, 50), (A_MID, "kh nh kl nl",
                                                                                                 "nh mh ml nl")),
          ((2, 100, 4, 100, 40, 128), KM), ((2, 128, 1, 255, 40, 100), NM), ((4, 256, 4, 64, 64, 64), KM),
          ((16, 272, 16, 256, 24, 64), KM), ((128, 64, 1, 16, 50, 128), KM), ((100, 41, 1, 33, 63, 128), KM),
          ((1, 17, 70, 59, 66, 128), KM), ((2, 32, 1, 8200, 32, 128), NM), ((1, 30, 1, 8203, 66, 64), NM),
          ((64, 64, 1, 24, 128, 64), KM)]


@pytest.mark.parametrize("case", SPLITS, ids=lambda c: "x".join(map(str, c[0])))
@pytest.mark.parametrize("ws", [None, False], ids=["workspace", "no_workspace"])
def test_fold_splits(mm, cuda, case, ws):
    d, A, B, C, T = _check(cuda, mm, *case, workspace=ws)
    for _ in range(2):  # the workspace holds the last call's partial sums
        C.fill_(float("nan"))
        mm.contract(d, A, B, C, workspace=ws)
        assert cuda.equal(C, T)


def test_fold_split_small_workspace(mm, cuda):
    """A workspace smaller than the split needs: unsplit, the same values."""
    case = ((4, 300, 1, 16, 20, 128), KM)
    _check(cuda, mm, *case, workspace=cuda.zeros(4096, dtype=cuda.uint8, device="cuda"))


def test_fold_splits_threads_one_stream(mm, cuda):
    """Several host threads contracting on one stream share its workspace: each call's two launches
    stay together, so every thread's output is its own."""
    import threading

    cases = [_check(cuda, mm, (8, 256, 1, 16, 20, 128), KM, seed=s) for s in range(4)]
    stream, wrong = cuda.cuda.current_stream(), []

    def work(d, A, B, C, T):
        for _ in range(50):
            mm.contract(d, A, B, C, stream=stream)
        stream.synchronize()
        if not cuda.equal(C, T):
            wrong.append(int((C != T).sum().item()))

    for _, _, _, C, _ in cases:
        C.fill_(float("nan"))
    threads = [threading.Thread(target=work, args=c) for c in cases]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong


def test_split_entry_points_threads_one_stream(mm, cuda):
    """The C entry points from several host threads on one stream with one workspace, as the header
    allows: a fold, the streaming kernels' splits, a tile split and a persistent grid's last round, each
    with its own values."""
    import ctypes as C
    import threading

    L, ws, st = mm.lib(), cuda.empty(mm.MAX_WORKSPACE_BYTES, dtype=cuda.uint8, device="cuda"), None
    ptr = lambda t: C.c_void_p(t.data_ptr())
    calls = []
    for s in range(2):
        d, A, B, Cd, T = _check(cuda, mm, (8, 256, 1, 16, 20, 128), KM, seed=s)
        calls.append((L.mmm_contract5d_f16f32_ws, (C.byref(d), ptr(A), ptr(B), ptr(Cd), ptr(ws), ws.numel(), st), Cd, T,
                      (d, A, B)))
    for M, N, K in ((16, 4096, 4096), (40, 2048, 4096), (256, 256, 8192), (4608, 4608, 2048)):
        gen = cuda.Generator(device="cuda").manual_seed(M)
        A, B = (cuda.randint(-4, 5, x, generator=gen, device="cuda").half() for x in ((M, K), (K, N)))
        Cd, T = cuda.empty(M, N, device="cuda"), (A.double() @ B.double()).float()
        assert mm.gemm_plan(M, N, K)["workspace_bytes"] > 0
        calls.append((L.mmm_gemm_f16f32_ws, (ptr(A), ptr(B), ptr(Cd), M, N, K, K, N, N, ptr(ws), ws.numel(), st), Cd, T,
                      (A, B)))
    cuda.cuda.synchronize()
    wrong = []

    def work(i, fn, args, Cd, T, keep):
        rc = [fn(*args) for _ in range(100)]
        cuda.cuda.synchronize()
        if any(rc) or not cuda.equal(Cd, T):
            wrong.append(i)

    threads = [threading.Thread(target=work, args=(i, *c)) for i, c in enumerate(calls)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong


@pytest.mark.parametrize("bound", [False, True], ids=["contract", "bind_contract"])
def test_fold_split_graphs_at_once(mm, cuda, bound, monkeypatch):
    """Split contractions captured into two graphs on one stream, replayed at the same time on two
    others beside eager calls on the stream of the capture: each has partial sums of its own."""
    cases = [_check(cuda, mm, (8, 256, 1, 16, 40, 128), KM, seed=s) for s in range(3)]
    side, graphs, own = cuda.cuda.Stream(), [], []
    take = mm._graph_workspace

    def spy(*args):
        t = take(*args)
        own.append((len(graphs), t.data_ptr(), t.numel()))
        return t

    monkeypatch.setattr(mm, "_graph_workspace", spy)
    side.wait_stream(cuda.cuda.current_stream())
    for d, A, B, C, T in cases[:2]:
        g = cuda.cuda.CUDAGraph()
        launch = mm.bind_contract(d, A, B, C, stream=side) if bound else lambda: mm.contract(d, A, B, C)
        with cuda.cuda.graph(g, stream=side):
            launch()
            launch()
        graphs.append(g)
    assert [g for g, _, _ in own] == [0, 0, 1, 1] and all(n > 16 for _, _, n in own)
    assert not {p for g, p, _ in own if g == 0} & {p for g, p, _ in own if g == 1}
    streams = [cuda.cuda.Stream(), cuda.cuda.Stream()]
    d, A, B, C, T = cases[2]
    for i in range(10):
        for c in cases:
            c[3].fill_(float("nan"))
        cuda.cuda.synchronize()
        for s, g in zip(streams, graphs):
            with cuda.cuda.stream(s):
                g.replay()
        with cuda.cuda.stream(side):
            mm.contract(d, A, B, C)
        cuda.cuda.synchronize()
        for j, c in enumerate(cases):
            assert cuda.equal(c[3], c[4]), f"pass {i}: contraction {j}"


# 33 to 64 rows of a row-major GEMM on the fold kernel's skinny tiles: one K tile and K ends inside one,
# odd K and N, a last strip of one column, rows at 2-byte alignment, 256-column strips (odd N, K ending inside a
# chunk and between chunks), one strip, B from 96 MiB (non-temporal); the view's padding is NaN
STREAM64 = [(33, 128, 64, 0), (64, 129, 8, 0), (40, 257, 7, 1), (64, 1000, 1000, 8), (50, 2041, 1031, 3), (33, 16, 9000, 0),
            (57, 16200, 9001, 1), (64, 8192, 16384, 8), (64, 12288, 4096, 0), (35, 17, 100, 2)]
STREAM64 += [(57, 16200, 9001, 8), (57, 16201, 9008, 7), (33, 16398, 8197, 2), (64, 12288, 4160, 0), (64, 20000, 4096, 0)]


# unsplit strips of 64 columns: 256 of them and one more (128-column strips again, 64 ones for K up to 224),
# last strips of 1, 8 and 63 columns, K past and up to the sums per step, odd K and rows
STREAM64 += [(64, 16384, 136, 0), (33, 16385, 264, 0), (48, 16392, 224, 8), (61, 16447, 193, 1), (64, 65, 1100, 0),
             (34, 4104, 2049, 7), (39, 127, 225, 0)]


COLUMNS_256 = [(57, 16200, 9001, 8), (64, 8192, 16384, 8), (57, 16201, 9008, 7), (33, 16398, 8197, 2)]


@pytest.mark.parametrize("shape", STREAM64, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("ws", [None, False], ids=["workspace", "no_workspace"])
def test_gemm_33_to_64_rows(mm, cuda, shape, ws):
    M, N, K, pad = shape
    gen = cuda.Generator(device="cuda").manual_seed(M + N + K)

    def view(rows, cols):
        buf = cuda.full((rows, cols + pad), float("nan"), dtype=cuda.float16, device="cuda")
        x = buf.flatten()[:(rows - 1) * (cols + pad) + cols].as_strided((rows, cols), (cols + pad, 1))
        return x.copy_(cuda.randint(-4, 5, (rows, cols), generator=gen, device="cuda", dtype=cuda.int8))

    A, B = view(M, K), view(K, N)
    C = cuda.full((M, N), float("nan"), dtype=cuda.float32, device="cuda")
    print(f"[gemm 33-64 rows] {shape} workspace {ws is None}", flush=True)
    plan = mm.gemm_plan(M, N, K, lda=K + pad, ldb=N + pad)
    if shape == (64, 12288, 4096, 0):  # with a workspace this one runs on 64x64 tiles: streamed without only
        assert plan["kernel"] == "tile"
    else:
        assert plan["kernel"] == "stream" and plan["stream_columns"] == (256 if shape in COLUMNS_256 else 128)
    mm.gemm(A, B, C, workspace=ws)
    T = (A.double() @ B.double()).float()
    assert cuda.equal(C, T), f"{int((C != T).sum().item())} outputs differ"


@pytest.mark.parametrize("shape", [(64, 4096, 14336), (33, 2048, 28672), (64, 28672, 2048)], ids=lambda s: "x".join(map(str, s)))
def test_gemm_33_to_64_rows_rounding(mm, cuda, shape):
    """2-norm distance from fp64.  A sum of n terms of like size, rounded to 24 bits after each addition,
    is off by about 2^-24 / sqrt(3) * sqrt(n / 2): 2e-7 at the 64 sums or fewer that a K range of these
    shapes and the reduction make with one per K tile; a chain of MFMAs over a range exceeds it."""
    M, N, K = shape
    gen = cuda.Generator(device="cuda").manual_seed(M + N + K)
    A = cuda.empty(M, K, device="cuda").uniform_(-1, 1, generator=gen).half()
    B = cuda.empty(K, N, device="cuda").uniform_(-1, 1, generator=gen).half()
    print(f"[gemm 33-64 rows] rounding {shape}", flush=True)
    T = A.double() @ B.double()
    assert ((mm.gemm(A, B) - T).norm() / T.norm()).item() <= 2e-7


@pytest.mark.parametrize("k", [64, 96, 128])
def test_gemm_33_to_64_rows_rounding_short(mm, cuda, k):
    """Up to ten 32-row K steps: a chain of MFMAs per step.  There is a rounding per 8 products, of partial
    sums of 8, 16, 24 and 32 products in each chain, then of the chains' sums.  A partial sum of s products
    of operands uniform in [-1, 1) is near N(0, s / 9), its rounding uniform in half an ulp either way:
    that gives the distance from fp64 up to a constant of the matrix cores' own, which K = 32 (one chain of
    four) shows.  One chain over each 64-row tile would be 14% (K = 64) or 8% further off; the bound lies
    halfway, and 0.3% is the spread over draws of this size."""
    import math

    def predicted(chains):
        sums, total = [], 0
        for length in chains:
            sums += range(8, length + 1, 8)
            total += length
            sums += [total] if total > length else []
        var = 0.0
        for n in sums:
            sd = math.sqrt(n / 9)
            for e in range(-30, 12):
                inside = math.erf(2.0**(e + 1) / sd / 2**0.5) - math.erf(2.0**e / sd / 2**0.5)
                var += 2.0**(2 * e - 46) / 12 * inside
        return math.sqrt(var / (total / 9))

    def measured(K):
        gen = cuda.Generator(device="cuda").manual_seed(K)
        A = cuda.empty(64, K, device="cuda").uniform_(-1, 1, generator=gen).half()
        B = cuda.empty(K, 16384, device="cuda").uniform_(-1, 1, generator=gen).half()
        T = A.double() @ B.double()
        return ((mm.gemm(A, B, workspace=False) - T).norm() / T.norm()).item()

    print(f"[gemm 33-64 rows] rounding K {k}", flush=True)
    steps, tiles = [32] * (k // 32), [min(64, k - i) for i in range(0, k, 64)]
    bound = (predicted(steps) + predicted(tiles)) / 2 / predicted([32])
    assert measured(k) / measured(32) <= bound


# (blocks, k_lo, blocks and k_lo of the same K in whole chunks): K up to the line between the kernels (2 x 20,
# 8 x 9, 4 x 10) and past it, with sums per K step (4 x 18, 6 x 20), per tile (8 x 25) and per fourth one
@pytest.mark.parametrize("case", [(64, 100, 100, 64), (48, 50, 25, 96), (32, 75, 25, 96), (104, 9, 39, 24), (8, 25, 5, 40),
                                  (6, 20, 5, 24), (4, 18, 3, 24), (2, 20, 1, 40), (8, 9, 3, 24), (4, 10, 1, 40),
                                  (400, 5, 25, 80)], ids=lambda c: f"{c[0]}x{c[1]}")
@pytest.mark.parametrize("form", ["reference", "n_contiguous"])
def test_fold_padded_k_rounding(mm, cuda, case, form):
    """Padded K blocks are no further from fp64 than one chain of MFMAs over the same K in whole chunks
    (0.5%: the spread of a distance over a million outputs)."""
    def distance(kh, kl):
        gen = cuda.Generator(device="cuda").manual_seed(kh * kl)
        a = cuda.empty(2048, kh * kl, device="cuda").uniform_(-1, 1, generator=gen).half()
        b = cuda.empty(kh * kl, 512, device="cuda").uniform_(-1, 1, generator=gen).half()
        T = a.double() @ b.double()
        A = a.reshape(64, 32, kh, kl).permute(0, 2, 1, 3).contiguous()  # [mh][kh][ml][kl]
        d = mm.ContractDesc()
        d.m_ext[:], d.n_ext[:], d.k_ext[:] = (64, 32), (1, 512), (kh, kl)
        d.a_m_stride[:], d.a_k_stride[:] = (kh * 32 * kl, kl), (32 * kl, 1)
        if form == "reference":  # B [n][kh][kl with 8 elements free after it]
            B = cuda.zeros(512, kh, kl + 8, dtype=cuda.float16, device="cuda")
            B[:, :, :kl] = b.t().reshape(512, kh, kl)
            d.b_k_stride[:], d.b_n_stride[:] = (kl + 8, 1), (0, kh * (kl + 8))
        else:
            B = b
            d.b_k_stride[:], d.b_n_stride[:] = (kl * 512, 512), (0, 1)
        d.c_m_stride[:], d.c_n_stride[:] = (32 * 512, 512), (0, 1)
        C = cuda.full((2048, 512), float("nan"), device="cuda")
        mm.contract(d, A, B, C, workspace=False)
        return ((C - T).norm() / T.norm()).item()

    kh, kl, kh8, kl8 = case
    print(f"[fold] rounding {case} {form}", flush=True)
    assert distance(kh, kl) <= 1.005 * distance(kh8, kl8)
