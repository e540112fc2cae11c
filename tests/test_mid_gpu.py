"""The producer / consumer kernel (mid_kernel.h): every tile at its edges, rows that start anywhere in a 128-byte line, K
tails, K parts, pieces lower than the tile. Against the fp64 oracle under "one rounding of the exact value" (half an ulp of the
result, twice, plus 1e-3 for fp32 sums in another order), and bit for bit between equal problems that lie differently in memory:
where a row starts moves its bytes in LDS, not the order of the sums."""
import pytest
import torch

from oracle import oracle
import fsw_weights

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
N_TILES = 36


def assert_one_rounding(out, ref64, dtype, what):
    err = (out.detach().cpu().double() - ref64).abs()
    bound = ref64.abs() * (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10) + 1e-3
    assert not (err > bound).any(), "%s: worst excess %g" % (what, (err - bound).max().item())


def lay(t, pad, offset):
    """The same matrix inside a NaN-filled buffer, rows `pad` elements longer, its start `offset` elements past a 256-byte line."""
    rows, cols = t.shape
    buf = torch.full((rows * (cols + pad) + offset + 128,), float("nan"), dtype=t.dtype, device=DEV)
    view = buf[offset:offset + rows * (cols + pad)].view(rows, cols + pad)[:, :cols]
    view.copy_(t)
    return view


def tile_rows(capi, index):
    """(weight rows, activation rows) of a forced tile, from its name."""
    try:
        assert capi.lib().fsw_set_variant(0, 200 + index) == capi.OK
        name = capi.variant_name(0, 0, 64, 512, 64)
    finally:
        capi.set_variant(0, -1)
    assert name.startswith("mid_")
    return tuple(int(x) for x in name[4:].split("x"))


@pytest.mark.parametrize("index", range(N_TILES))
def test_every_tile_at_its_edges(capi, index):
    """Rows one past the tile in both directions (the second tiles hold one row each), K of less than a line, of whole lines, with a
    tail; gate/up and the plain product; dense rows and rows at every sixteenth of a line beside NaN."""
    bp, bq = tile_rows(capi, index)
    for n, (M, ff, K) in enumerate([(bq + 1, bp // 2 + 4, 200), (bq, bp // 2, 8), (bq - 1, bp // 2 + 3, 328), (bq + 1, bp // 2 - 1, 256)]):
        dtype = torch.float16 if n % 2 else torch.bfloat16
        inp = fsw_weights.make_inputs(M, K, ff, dtype, seed=97 * index + n, x_scale=0.5)
        want = oracle.ref_gateup(inp["X"], inp["W13"], torch.float64)
        plain = inp["X"].double() @ inp["W13"].double().t()
        first = None
        for pad, xo, wo in ((0, 0, 0), (8 * (1 + index % 7), 8 * (1 + n), 8 * (index % 16)), (64 - K % 64, 0, 0)):
            X, W = lay(inp["X"], pad, xo), lay(inp["W13"], pad, wo)
            wide = torch.full((M, ff + 8), float("nan"), dtype=dtype, device=DEV)
            try:
                capi.set_variant(0, 200 + index)
                capi.set_variant(1, 200 + index)
                capi.gateup(X, W, out=wide[:, :ff])
                P = capi.down(X, W)
            finally:
                capi.set_variant(0, -1)
                capi.set_variant(1, -1)
            what = "tile %d (%d x %d) %s pad %d" % (index, bp, bq, (M, ff, K), pad)
            assert torch.isnan(wide[:, ff:]).all(), what
            assert_one_rounding(wide[:, :ff], want, dtype, what)
            assert_one_rounding(P, plain, dtype, what + " plain")
            if M > bq:  # two tiles of rows: no workgroup starts its K walk elsewhere
                first = first if first is not None else (wide.clone(), P)
                assert torch.equal(wide[:, :ff], first[0][:, :ff]) and torch.equal(P, first[1]), what


@pytest.mark.parametrize("index", range(N_TILES))
def test_rings_and_left_out_copies(capi, index):
    """K of 3 .. 13 lines (fewer than a ring holds, as many, a few more: the last of them masked), whole and with a tail, dense and in
    padded rows; weight and activation rows that end 8 rows or more before the tile does, where waves leave copies out."""
    bp, bq = tile_rows(capi, index)
    for lines in range(3, 14):
        M, ff = bq - (8, 9, 17, 31)[lines % 4], bp // 2 - (0, 4, 8, 15)[lines // 4]
        K = 64 * lines - (0, 8, 40)[lines % 3]
        g = torch.Generator(device=DEV).manual_seed(100 * index + lines)
        X = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16)
        W = (torch.randn(2 * ff, K, device=DEV, generator=g) / K ** 0.5).to(torch.bfloat16)
        plain = X.double() @ W.double().t()
        want = plain[:, 0::2] * torch.nn.functional.silu(plain[:, 1::2])
        for pad in (0, (-K) % 64):
            Xp, Wp = lay(X, pad, 0), lay(W, pad, 0)
            try:
                capi.set_variant(0, 200 + index)
                capi.set_variant(1, 200 + index)
                H, P = capi.gateup(Xp, Wp), capi.down(Xp, Wp)
            finally:
                capi.set_variant(0, -1)
                capi.set_variant(1, -1)
            what = "tile %d (%d x %d) %s pad %d" % (index, bp, bq, (M, ff, K), pad)
            assert_one_rounding(H, want.cpu(), torch.bfloat16, what)
            assert_one_rounding(P, plain.cpu(), torch.bfloat16, what + " plain")


@pytest.mark.parametrize("index", range(N_TILES))
def test_long_walks_over_k(capi, index):
    """K of 31 .. 38 lines, where tiles of more than 64 activation rows ask for weight lines in pairs (32 and more), rings are refilled several
    times and whole lines are copied without bounds checks: line counts of both parities around the bound, with and without a tail; dense rows,
    rows of whole lines, rows a multiple of 4 KB apart (walks from different lines), rows at every sixteenth of a line. Weight and activation
    rows that end with the tile, and 8 rows and more before it (waves leave copies out). All tiles of one call and of a call with one row more
    than the tile. One rounding of the exact value, and where no walk starts elsewhere the same bits however the rows lie."""
    bp, bq = tile_rows(capi, index)
    for n, (K, M, ff) in enumerate([(64 * 31, bq, bp // 2), (64 * 32, bq + 1, bp + 3), (64 * 33 - 8, bq - 9, bp // 2 - 4), (64 * 34 - 40, bq, bp),
                                    (64 * 37, bq - 17, bp // 2 - 8), (64 * 37 - 56, bq + 1, bp // 2 + 1), (64 * 38, bq - 31, bp - 15)]):
        dtype = torch.float16 if n % 2 else torch.bfloat16
        g = torch.Generator(device=DEV).manual_seed(100 * index + n)
        X = torch.randn(M, K, device=DEV, generator=g).to(dtype)
        W = (torch.randn(2 * ff, K, device=DEV, generator=g) / K ** 0.5).to(dtype)
        plain = X.double() @ W.double().t()
        want = (plain[:, 0::2] * torch.nn.functional.silu(plain[:, 1::2])).cpu()
        plain, first = plain.cpu(), None
        for pad, xo, wo in ((0, 0, 0), ((-K) % 64 + 64, 0, 0), (-K % 2048, 0, 0), (8 * (1 + index % 7), 8 * (1 + n), 8 * (index % 16))):
            Xp, Wp = lay(X, pad, xo), lay(W, pad, wo)
            try:
                capi.set_variant(0, 200 + index)
                capi.set_variant(1, 200 + index)
                H, P = capi.gateup(Xp, Wp), capi.down(Xp, Wp)
            finally:
                capi.set_variant(0, -1)
                capi.set_variant(1, -1)
            what = "tile %d (%d x %d) %s pad %d" % (index, bp, bq, (M, ff, K), pad)
            assert_one_rounding(H, want, dtype, what)
            assert_one_rounding(P, plain, dtype, what + " plain")
            if M > bq:
                first = first or (H, P)
                assert torch.equal(H, first[0]) and torch.equal(P, first[1]), what


@pytest.mark.parametrize("M", [1, 8, 17, 33, 100, 200, 300])
@pytest.mark.parametrize("D,FF", [(1096, 8008), (1024, 16384), (3000, 4872)])
def test_down_projection_in_parts_of_k(capi, M, D, FF):
    """K parts whose bounds fall inside lines: the parts of one line go to two workgroups and are summed once. H beside NaN, and the
    same numbers from a padded layout."""
    inp = fsw_weights.make_inputs(M, D, FF, torch.bfloat16, seed=M + FF, x_scale=0.5)
    H = torch.randn(M, FF, generator=torch.Generator().manual_seed(M)).to(torch.bfloat16) * 0.3
    ref = oracle.ref_down(H, inp["W2"], torch.float64)
    Y = capi.down(lay(H, 0, 0), lay(inp["W2"], 0, 0))
    assert_one_rounding(Y, ref, torch.bfloat16, "parts %s" % ((M, D, FF),))
    for pad, ho, wo in ((8, 8, 24), (64 - FF % 64, 0, 64)):
        assert_one_rounding(capi.down(lay(H, pad, ho), lay(inp["W2"], pad, wo)), ref, torch.bfloat16, "pad %d" % pad)
    assert torch.equal(capi.mlp(*(inp[k].to(DEV) for k in ("X", "W13", "W2"))), capi.down(
        capi.gateup(inp["X"].to(DEV), inp["W13"].to(DEV)), inp["W2"].to(DEV)))


@pytest.mark.parametrize("tile", [0, 2, 10, 14, 22, 30])
@pytest.mark.parametrize("M,K,ld,spread", [(20, 2048, 2048, True), (20, 2040, 2048, True), (20, 2040, 2112, False), (20, 4088, 4096, True),
                                           (31, 6104, 6144, True)])
def test_workgroups_start_their_walk_over_k_at_different_lines(capi, tile, M, K, ld, spread):
    """All weight rows are the same two, so every workgroup sums the same products: in one order, and to the same float32 bits, if they all
    start at line 0, in different orders if the walk is spread. Off float64 at most what fp32 sums of K products in any order are."""
    gen = torch.Generator(device=DEV).manual_seed(K + M)
    ff = 4096
    X = torch.randn(M, ld, generator=gen, device=DEV).to(torch.bfloat16)[:, :K]
    pair = (torch.randn(2, K, generator=gen, device=DEV) / K ** 0.5).to(torch.bfloat16)
    W = torch.full((2 * ff, ld), float("nan"), dtype=torch.bfloat16, device=DEV)[:, :K]
    W[0::2], W[1::2] = pair[0], pair[1]
    try:
        capi.set_variant(0, 200 + tile)
        H = capi.gateup_f32out(X, W)
    finally:
        capi.set_variant(0, -1)
    assert (H != H[:, :1]).any().item() == spread
    pre = X.double() @ pair.double().t()
    want = (pre[:, 0] * torch.nn.functional.silu(pre[:, 1]))[:, None]
    # a sum of K products whose absolute values add up to S is off by at most (K / 32 + 32) rounding errors of 2^-24 S; the two sums enter the
    # result multiplied by at most 1.1 |up| + |gate| (silu' <= 1.1)
    S = X.double().abs() @ pair.double().abs().t()
    bound = (K / 32 + 32) * 2.0 ** -24 * (S[:, 0] * pre[:, 1].abs() + 1.1 * S[:, 1] * pre[:, 0].abs())[:, None] + 1e-6 * want.abs() + 1e-9
    assert ((H.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("M,D,FF", [(656, 2048, 8192), (999, 1530, 6144), (257, 3072, 12288), (259, 3070, 12288)])
def test_down_projection_of_more_rows_on_narrow_outputs(capi, M, D, FF):
    """Rows past 256 whose parts the 256-row kernel took: H and W2 in rows of whole lines beside NaN, output inside a wider NaN buffer, all of
    the scratch with a guard behind it, less of it refused; against float64 and against the 256-row kernel."""
    L = capi.lib()
    assert capi.variant_name(1, 0, M, D, FF).startswith("splitk_pair16") and capi.variant_name(4, 0, M, D, FF).startswith("mid_")
    H = (torch.randn(M, FF, device=DEV) * 0.3).to(torch.bfloat16)
    W2 = (torch.randn(D, FF, device=DEV) / FF ** 0.5).to(torch.bfloat16)
    ref = (H.double() @ W2.double().t()).cpu()
    Hp, Wp = lay(H, 64, 0), lay(W2, 128, 0)
    nbytes, part = L.fsw_down_workspace_bytes(0, M, D, FF), 4 * M * D
    assert nbytes >= 2 * part
    ws = torch.full((nbytes + 256,), 7, dtype=torch.uint8, device=DEV)
    wide = torch.full((M, D + 8), float("nan"), dtype=torch.bfloat16, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    args = (0, M, D, FF, Hp.data_ptr(), Hp.stride(0), Wp.data_ptr(), Wp.stride(0), wide.data_ptr(), D + 8)
    assert L.fsw_down(*args, ws.data_ptr(), nbytes, stream) == capi.OK
    assert (ws[nbytes:] == 7).all() and torch.isnan(wide[:, D:]).all()
    assert_one_rounding(wide[:, :D], ref, torch.bfloat16, "parts")
    assert L.fsw_down(*args, ws.data_ptr(), nbytes - part, stream) != capi.OK  # refused as before
    try:
        capi.set_variant(1, 5)
        large = capi.down(H, W2)
    finally:
        capi.set_variant(1, -1)
    # either is one rounding of a sum off by fp32 noise: they differ by an ulp where the sum lies next to a tie
    assert ((wide[:, :D].float() - large.float()).abs() <= large.float().abs() * 2.0 ** -7 + 1e-3).all()


@pytest.mark.parametrize("M,D,FF", [(656, 2048, 8192), (300, 2048, 4096), (259, 3070, 12288)])
@pytest.mark.parametrize("h_pad,w_pad,offset", [(8, 24, 0), (64, 64, 8), (0, 40, 24)])
def test_down_projection_on_narrow_outputs_of_rows_that_are_no_whole_lines(capi, M, D, FF, h_pad, w_pad, offset):
    """K of whole lines, which the plan of the scratch goes by, in rows that start anywhere in a line, which the launch goes by: beside NaN,
    exactly the scratch that was asked for with a guard behind it, against float64."""
    L = capi.lib()
    H = (torch.randn(M, FF, device=DEV) * 0.3).to(torch.bfloat16)
    W2 = (torch.randn(D, FF, device=DEV) / FF ** 0.5).to(torch.bfloat16)
    Hp, Wp = lay(H, h_pad, offset), lay(W2, w_pad, offset)
    nbytes = L.fsw_down_workspace_bytes(0, M, D, FF)
    ws = torch.full((nbytes + 256,), 7, dtype=torch.uint8, device=DEV)
    wide = torch.full((M, D + 8), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert L.fsw_down(0, M, D, FF, Hp.data_ptr(), Hp.stride(0), Wp.data_ptr(), Wp.stride(0), wide.data_ptr(), D + 8, ws.data_ptr(), nbytes,
                      torch.cuda.current_stream().cuda_stream) == capi.OK
    assert (ws[nbytes:] == 7).all() and torch.isnan(wide[:, D:]).all()
    assert_one_rounding(wide[:, :D], (H.double() @ W2.double().t()).cpu(), torch.bfloat16, "parts")


def test_down_projection_of_few_rows_runs_without_scratch(capi):
    """Up to 48 rows the weight-streaming kernel needs none: a caller that brings no workspace gets that kernel, not an error."""
    M, D, FF = 20, 2048, 8192
    L = capi.lib()
    assert L.fsw_down_workspace_bytes(0, M, D, FF) > 0 and capi.variant_name(4, 0, M, D, FF).startswith("mid_")
    H = (torch.randn(M, FF, device=DEV) * 0.3).to(torch.bfloat16)
    W2 = (torch.randn(D, FF, device=DEV) / FF ** 0.5).to(torch.bfloat16)
    Y = torch.empty(M, D, dtype=torch.bfloat16, device=DEV)
    assert L.fsw_down(0, M, D, FF, H.data_ptr(), FF, W2.data_ptr(), FF, Y.data_ptr(), D, None, 0,
                      torch.cuda.current_stream().cuda_stream) == capi.OK
    assert_one_rounding(Y, oracle.ref_down(H.cpu(), W2.cpu(), torch.float64), torch.bfloat16, "no scratch")


@pytest.mark.parametrize("M,D,FF", [(121, 336, 904), (90, 488, 1000), (20, 2048, 8192), (16, 5120, 13824)])
def test_down_projection_with_less_scratch_than_its_parts_want(capi, M, D, FF):
    """K parts on the producer / consumer kernel are as many as there is room for: none without a workspace, or with one that is not
    16-byte aligned; fewer in less room. A guard behind the scratch stays as it is."""
    L = capi.lib()
    nbytes = L.fsw_down_workspace_bytes(0, M, D, FF)
    part = 4 * M * D
    assert nbytes >= 2 * part
    H = (torch.randn(M, FF, device=DEV) * 0.3).to(torch.bfloat16)
    W2 = (torch.randn(D, FF, device=DEV) / FF ** 0.5).to(torch.bfloat16)
    ref = (H.double() @ W2.double().T).cpu()
    ws = torch.full((nbytes + 512,), 255, dtype=torch.uint8, device=DEV)
    for offset, size in ((None, 0), (0, part), (8, nbytes), (0, 2 * part), (0, nbytes)):
        Y = torch.empty(M, D, dtype=torch.bfloat16, device=DEV)
        assert L.fsw_down(0, M, D, FF, H.data_ptr(), FF, W2.data_ptr(), FF, Y.data_ptr(), D,
                          None if offset is None else ws.data_ptr() + offset, size,
                          torch.cuda.current_stream().cuda_stream) == capi.OK
        assert (ws[size + 16:] == 255).all()
        assert_one_rounding(Y, ref, torch.bfloat16, "scratch of %d bytes %s" % (size, (M, D, FF)))


@pytest.mark.parametrize("M,d,ff", [(1, 5120, 13824), (16, 3000, 8008), (40, 2048, 8192), (130, 4096, 11008), (200, 3000, 8008),
                                    (300, 3960, 8040), (512, 1024, 2816), (700, 1320, 3000)])
def test_chosen_tiles_against_the_256_row_kernel(capi, M, d, ff):
    """What the dispatcher chooses (pieces lower than the tile included) against the 256-row kernel, which takes any problem: every
    feature, both sums rounded once; and repeated calls bit for bit."""
    assert capi.variant_name(3, 0, M, 2 * ff, d).startswith("mid_")
    inp = fsw_weights.make_inputs(M, d, ff, torch.bfloat16, seed=d, x_scale=1.0)
    X, W = inp["X"].to(DEV), inp["W13"].to(DEV)
    H = capi.gateup(X, W)
    try:
        capi.set_variant(0, 5)
        big = capi.gateup(X, W)
    finally:
        capi.set_variant(0, -1)
    assert ((H.float() - big.float()).abs() <= 2.0 ** -7 * big.float().abs() + 1e-3).all()
    assert all(torch.equal(capi.gateup(X, W), H) for _ in range(3))


@pytest.mark.parametrize("M,d,ff", [(20, 1024, 4104), (257, 520, 2056), (700, 520, 2120), (2049, 264, 1000), (2700, 4096, 3592)])
def test_forward_with_h_in_whole_lines(capi, M, d, ff):
    """With 128 bytes a row more scratch than the query asks for, rows of H are whole lines above 256 rows; what lies between them is
    never read. Scratch full of NaN; against float64, and against the forward on the queried scratch (dense H): the same bits, as no
    sum changes its order."""
    gen = torch.Generator(device=DEV).manual_seed(M + ff)
    X = torch.randn(M, d, generator=gen, device=DEV).to(torch.bfloat16)
    W13 = (torch.randn(2 * ff, d, generator=gen, device=DEV) / d ** 0.5).to(torch.bfloat16)
    W2 = (torch.randn(d, ff, generator=gen, device=DEV) / ff ** 0.5).to(torch.bfloat16)
    queried = capi.mlp_workspace(X, ff)
    ys = []
    for extra in (0, 128 * M - 2, 128 * M):
        ws = torch.full((queried.numel() + extra,), 255, dtype=torch.uint8, device=DEV)
        ys.append(capi.mlp(X, W13, W2, workspace=ws))
    pre = X.double() @ W13.double().T
    H = (pre[:, 0::2] * torch.nn.functional.silu(pre[:, 1::2]))
    oracle.assert_parity(ys[2], (H @ W2.double().T).cpu(), "H in whole lines %s" % ((M, d, ff),))
    assert torch.equal(ys[0], ys[2]) and torch.equal(ys[0], ys[1])


@pytest.mark.parametrize("M,D,FF", [(257, 264, 1032), (371, 2048, 8192), (300, 3000, 8008), (512, 1024, 2816), (700, 2048, 2056),
                                    (1996, 736, 2088)])
def test_fewer_parts_than_there_is_scratch_for(capi, M, D, FF):
    """Above 256 rows the workspace query gives the most parts; the launch may take fewer. Scratch full of NaN, exactly as large as
    the query says, a guard behind it."""
    L = capi.lib()
    H = (torch.randn(M, FF, device=DEV) * 0.3).to(torch.bfloat16)
    W2 = (torch.randn(D, FF, device=DEV) / FF ** 0.5).to(torch.bfloat16)
    nbytes = L.fsw_down_workspace_bytes(0, M, D, FF)
    ws = torch.full((nbytes + 256,), 255, dtype=torch.uint8, device=DEV)
    Y = torch.empty(M, D, dtype=torch.bfloat16, device=DEV)
    assert nbytes > 0 and capi.variant_name(4, 0, M, D, FF).startswith("mid_")
    for _ in range(2):
        assert L.fsw_down(0, M, D, FF, H.data_ptr(), FF, W2.data_ptr(), FF, Y.data_ptr(), D, ws.data_ptr(), nbytes,
                          torch.cuda.current_stream().cuda_stream) == capi.OK
        assert (ws[nbytes:] == 255).all()
        assert_one_rounding(Y, (H.double() @ W2.double().T).cpu(), torch.bfloat16, "parts %s" % ((M, D, FF),))


@pytest.mark.parametrize("M,ff,K", [(1, 4096, 3000), (4, 11008, 4096), (20, 5504, 4096), (33, 3000, 2048)])
def test_float32_output_of_few_rows_keeps_its_short_sums(capi, M, ff, K):
    """skinny_kernel splits K between its waves; the result as it stands in float32 shows the length of the chains. Bit for bit what that
    kernel gives when forced, and within its error of float64: a wave's chain has at most K / (32 * 4) sums of relative error 2^-24
    each, a random walk of sqrt(n) of them; SiLU and the product add about two more roundings. Twice that."""
    inp = fsw_weights.make_inputs(M, K, ff, torch.bfloat16, seed=M + ff, x_scale=1.0)
    X, W = inp["X"].to(DEV), inp["W13"].to(DEV)
    H = capi.gateup_f32out(X, W)
    try:
        capi.set_variant(0, 100)
        few = capi.gateup_f32out(X, W)
    finally:
        capi.set_variant(0, -1)
    assert torch.equal(H, few)
    pre = X.double() @ W.double().T
    ref = pre[:, 0::2] * torch.nn.functional.silu(pre[:, 1::2])
    assert ((H.double() - ref).norm() / ref.norm()).item() <= 2 * 2.0 ** -24 * ((K / 128) ** 0.5 + 2)


@pytest.mark.parametrize("M,ff,K", [(1, 14336, 4096), (4, 14336, 4096), (8, 14336, 4096), (1, 11008, 4096)])
def test_few_rows_of_full_rounds_keep_the_weight_streaming_kernel(capi, M, ff, K):
    """Gate/up of up to 8 rows where the producer / consumer kernel is no faster: the bits of the weight-streaming kernel, whose waves
    sum K in several short chains."""
    inp = fsw_weights.make_inputs(M, K, ff, torch.bfloat16, seed=M + ff, x_scale=1.0)
    X, W = inp["X"].to(DEV), inp["W13"].to(DEV)
    H = capi.gateup(X, W)
    try:
        capi.set_variant(0, 100)
        few = capi.gateup(X, W)
    finally:
        capi.set_variant(0, -1)
    assert torch.equal(H, few)


@pytest.mark.parametrize("M", [12, 16, 24, 32, 48, 64])
@pytest.mark.parametrize("ff,K", [(14336, 4096), (14464, 1024)])
def test_whole_tiles_where_they_fill_a_round(capi, M, ff, K):
    """224 and 226 tiles of 128 weight rows: no pieces, so each feature's sum starts at the K tile it starts at on the forced 128 x 64
    tile (id 4), bit for bit."""
    inp = fsw_weights.make_inputs(M, K, ff, torch.bfloat16, seed=M + ff, x_scale=1.0)
    X, W = inp["X"].to(DEV), inp["W13"].to(DEV)
    H = capi.gateup(X, W)
    try:
        capi.set_variant(0, 4)
        whole = capi.gateup(X, W)
    finally:
        capi.set_variant(0, -1)
    assert torch.equal(H, whole)


@pytest.mark.parametrize("M,ff,K", [(1, 13824, 5120), (4, 5504, 4096), (16, 8192, 3000), (20, 4096, 2048), (40, 3904, 1320)])
def test_few_rows_are_summed_as_finely_as_by_the_weight_streaming_kernel(capi, M, ff, K):
    """The unrounded gate/up product of few rows, on tiles of 32 and 64 activation rows: no further from float64 than the
    weight-streaming kernel, which sums an eighth or a quarter of K in a chain. Both errors are root mean squares over thousands of sums;
    a tenth covers their spread."""
    inp = fsw_weights.make_inputs(M, K, ff, torch.bfloat16, seed=M + ff, x_scale=1.0)
    X, W = inp["X"].to(DEV), inp["W13"].to(DEV)
    pre = X.double() @ W.double().T
    ref = pre[:, 0::2] * torch.nn.functional.silu(pre[:, 1::2])
    error = {}
    for v in (100, 202, 204, 210):  # weight streaming; 64 x 32, 128 x 32, 128 x 64
        try:
            capi.set_variant(0, v)
            H = capi.gateup_f32out(X, W)
        finally:
            capi.set_variant(0, -1)
        error[v] = ((H.double() - ref).norm() / ref.norm()).item()
    assert max(error[v] for v in (202, 204, 210)) <= 1.1 * error[100], error


@pytest.mark.parametrize("M,ff,K", [(17, 1112, 736), (48, 300, 200), (9, 4352, 256), (16, 4400, 264), (14, 1480, 800), (9, 1500, 8), (16, 1000, 896)])
def test_gateup_of_a_short_k_gives_the_bits_of_the_weight_streaming_kernel(capi, M, ff, K):
    """Workgroups of four waves with a K of up to 896 among them: against the kernel forced and the oracle, output inside a wider NaN buffer."""
    inp = fsw_weights.make_inputs(M, K, ff, torch.bfloat16, seed=M + ff, x_scale=1.0)
    X, W = inp["X"].to(DEV), inp["W13"].to(DEV)
    wide = torch.full((M, ff + 8), float("nan"), dtype=torch.bfloat16, device=DEV)
    capi.gateup(X, W, out=wide[:, :ff])
    try:
        capi.set_variant(0, 100)
        few = capi.gateup(X, W)
    finally:
        capi.set_variant(0, -1)
    assert torch.equal(wide[:, :ff], few) and torch.isnan(wide[:, ff:]).all()
    pre = inp["X"].double() @ inp["W13"].double().T
    assert_one_rounding(wide[:, :ff], pre[:, 0::2] * torch.nn.functional.silu(pre[:, 1::2]), torch.bfloat16, "H %s" % ((M, ff, K),))


@pytest.mark.parametrize("M,D,FF", [(17, 512, 1000), (48, 264, 2056), (40, 4104, 520), (16, 4352, 512), (1, 5000, 1000), (9, 4200, 1800)])
def test_down_projection_of_a_short_k_gives_the_bits_of_the_weight_streaming_kernel(capi, M, D, FF):
    """No scratch, no K parts: against the kernel forced and the oracle, output inside a wider NaN buffer."""
    gen = torch.Generator().manual_seed(M + FF)
    H = (torch.randn(M, FF, generator=gen) * 0.5).to(torch.bfloat16)
    W2 = (torch.randn(D, FF, generator=gen) / FF ** 0.5).to(torch.bfloat16)
    wide = torch.full((M, D + 8), float("nan"), dtype=torch.bfloat16, device=DEV)
    capi.down(H.to(DEV), W2.to(DEV), out=wide[:, :D])
    try:
        capi.set_variant(1, 100)
        few = capi.down(H.to(DEV), W2.to(DEV))
    finally:
        capi.set_variant(1, -1)
    assert torch.equal(wide[:, :D], few) and torch.isnan(wide[:, D:]).all()
    assert_one_rounding(wide[:, :D], H.double() @ W2.double().T, torch.bfloat16, "Y %s" % ((M, D, FF),))
