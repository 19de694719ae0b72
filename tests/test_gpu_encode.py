"""Encode side on the GPU against the oracle encoders (needs an MI355X)."""
import numpy as np
import pytest
import torch

from oracle import glq_oracle as O
from tests.gpu_util import DEV, say, t

pytestmark = pytest.mark.gpu


def test_e8_quantize_matches_oracle_indices():
    """Random vectors at several scales, exact ties (the origin, midpoints between table
    rows, lattice points themselves) and the 256-row secondary table: indices bit-equal."""
    from glq_amd import ext
    say("e8 quantize")
    rng = np.random.default_rng(0)
    cb = O.e8_table()
    X = np.concatenate([
        rng.standard_normal((3000, 8)).astype(np.float32),
        (rng.standard_normal((1000, 8)) * 3.0).astype(np.float32),
        (rng.standard_normal((500, 8)) * 0.1).astype(np.float32),
        np.zeros((1, 8), np.float32),
        cb[rng.integers(0, 65536, 300)],
        0.5 * (cb[rng.integers(0, 65536, 300)] + cb[rng.integers(0, 65536, 300)]),
        rng.standard_normal((700, 8)).astype(np.float16).astype(np.float32),
    ])
    dec_ref, idx_ref = O.e8_quantize(X)
    dec, idx = ext.e8_quantize(t(X), t(cb))
    idx = idx.cpu().numpy()
    bad = np.nonzero(idx != idx_ref)[0]
    assert bad.size == 0, (bad[:5], idx[bad[:5]], idx_ref[bad[:5]])
    assert np.array_equal(dec.cpu().numpy(), dec_ref)
    # the walk over the rows, which tables that are not the whole shell table take
    assert np.array_equal(ext.e8_quantize(t(X), t(cb[:65000]))[1].cpu().numpy(), O.e8_quantize(X, cb[:65000])[1])
    # secondary table of the 3 bpw recipe
    _, i2_ref = O.e8_quantize(X[:1000], cb[:256])
    _, i2 = ext.e8_quantize(t(X[:1000]), t(cb[:256]))
    assert np.array_equal(i2.cpu().numpy(), i2_ref)


def test_e8_quantize_residual_stage_and_size():
    from glq_amd import ext
    say("e8 quantize rvq")
    rng = np.random.default_rng(1)
    cb = O.e8_table()
    X = rng.standard_normal((4099, 8)).astype(np.float32)        # ragged against the launch tiling
    d1, i1 = ext.e8_quantize(t(X), t(cb))
    res = (t(X) - d1) * 3.0
    d2, i2 = ext.e8_quantize(res, t(cb))
    r1, j1 = O.e8_quantize(X)
    r2, j2 = O.e8_quantize((X - r1) * np.float32(3.0))
    assert np.array_equal(i1.cpu().numpy(), j1) and np.array_equal(i2.cpu().numpy(), j2)
    again = ext.e8_quantize(t(X), t(cb))[1]
    assert torch.equal(i1, again)


@pytest.mark.parametrize("N,scale", [(1, 1.0), (255, 3.0), (257, 0.3), (5000, 1.5), (20001, 4.0), (70001, 1.0), (40000, 100.0), (262145, 1.0)])
def test_e8_quantize_on_the_shell_table_equals_the_table_walk(N, scale):
    """The search by the table's symmetry against the kernel that walks all rows (pinned on the oracle above through
    tables it does not recognise), at sizes around a workgroup's and past the switch to 512 vectors per workgroup:
    random vectors, exact ties (zeros, equal and opposite entries, midpoints of rows), vectors far outside the table,
    and some that are not finite."""
    from glq_amd import _lib, ext
    say("e8 shell search", N, scale)
    g = torch.Generator().manual_seed(N)
    cb = torch.from_numpy(O.e8_table())
    X = torch.randn(N, 8, generator=g) * scale
    pick = torch.randint(0, N, (8, max(1, N // 50)), generator=g)
    X[pick[0]] = (X[pick[0]] * 2).round() / 2                    # on or near the half-integer grid
    X[pick[1]] = 0.5 * (cb[torch.randint(0, 65536, pick[1].shape, generator=g)] + cb[torch.randint(0, 65536, pick[1].shape, generator=g)])
    X[pick[2], 1] = -X[pick[2], 0]
    X[pick[3]] *= 5.0
    X[pick[4]] = cb[torch.randint(56881, 65536, pick[4].shape, generator=g)] * 1.05
    for j, bad in enumerate((float("nan"), float("inf"), 3e38, 1e-42)):
        X[pick[5, j % pick.shape[1]], j % 8] = bad
    X, cb = X.to(DEV), cb.to(DEV)
    dec, idx = ext.e8_quantize(X, cb)
    norms = (cb * cb).sum(-1)
    walk, wdec = torch.empty_like(idx), torch.empty_like(dec)
    _lib.check(_lib.load().glqh_e8_quantize(X.data_ptr(), cb.data_ptr(), norms.data_ptr(), N, 65536, walk.data_ptr(),
                                            wdec.data_ptr(), torch.cuda.current_stream().cuda_stream))
    assert torch.equal(idx, walk), int((idx != walk).sum())
    assert torch.equal(dec, wdec)
    assert torch.equal(ext.e8_quantize(X, cb, norms)[1], walk)   # the caller's norms
    norms[5] += 0.5                                              # a table that no longer qualifies, same memory
    X, walk, wdec = X[:2000], walk[:2000], wdec[:2000]
    _lib.check(_lib.load().glqh_e8_quantize(X.data_ptr(), cb.data_ptr(), norms.data_ptr(), X.shape[0], 65536, walk.data_ptr(),
                                            wdec.data_ptr(), torch.cuda.current_stream().cuda_stream))
    dec, idx = ext.e8_quantize(X, cb, norms)
    assert torch.equal(idx, walk) and torch.equal(dec, wdec)


def _walk(X, cb, norms):
    """Every row against every vector."""
    from glq_amd import _lib
    idx, dec = torch.empty(X.shape[0], dtype=torch.int64, device=DEV), torch.empty_like(X)
    _lib.check(_lib.load().glqh_e8_quantize(X.data_ptr(), cb.data_ptr(), norms.data_ptr(), X.shape[0], cb.shape[0], idx.data_ptr(),
                                            dec.data_ptr(), torch.cuda.current_stream().cuda_stream))
    return dec, idx


@pytest.mark.parametrize("N,scale", [(63, 20.0), (70001, 2.0), (65600, 20.0), (262200, 6.0)])
def test_e8_quantize_of_many_points_in_reach(N, scale):
    """Where the lists of a workgroup take fewer vectors at a time, are emptied on the way, or run over: all vectors
    outside the table, at each number of vectors to a workgroup, some of whole workgroups with hundreds of points at one
    distance (equal entries, zeros).  The walk's own index and codeword throughout."""
    from glq_amd import ext
    say("e8 shell search, many points", N, scale)
    g = torch.Generator().manual_seed(N)
    X = torch.randn(N, 8, generator=g) * scale
    for first, of in ((0, [1.0, 0, 0, 0, 0, 0, 0, 0]), (N // 4, [1.0] * 8), (N // 2, [1.0, 1.0, 1.0, 1.0, 0, 0, 0, 0]),
                      (3 * N // 4, [3.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0, -1.0])):
        n = min(600, N // 8)
        X[first:first + n] = torch.tensor(of) * (scale * (1 + torch.rand(n, 1, generator=g)))
        X[first + n // 2:first + n] += 1e-5 * torch.randn(n - n // 2, 8, generator=g)
    cb = torch.from_numpy(O.e8_table()).to(DEV)
    X = X.to(DEV)
    dec, idx = ext.e8_quantize(X, cb)
    wdec, walk = _walk(X, cb, (cb * cb).sum(-1))
    assert torch.equal(idx, walk), int((idx != walk).sum())
    assert torch.equal(dec, wdec)


@pytest.mark.parametrize("N,V", [(256, 63), (65600, 256), (262200, 256)])
def test_e8_quantize_on_either_side_of_few_vectors_to_list(N, V):
    """Workgroups with one vector outside the table, with 31, 32 and 33 (the most whose points go to the waves as they are found), and with
    none: the walk's own index and codeword."""
    from glq_amd import ext
    say("e8 shell search, few to list", N)
    g = torch.Generator().manual_seed(N)
    X = torch.randn(N, 8, generator=g) * 0.05
    for i, k in enumerate((1, 31, 32, 33, 0, 48)):
        at = i * 1024 % N + torch.randperm(min(V, 256), generator=g)[:k]
        X[at] = torch.randn(k, 8, generator=g) * 3 + 1
    cb = torch.from_numpy(O.e8_table()).to(DEV)
    X = X.to(DEV)
    dec, idx = ext.e8_quantize(X, cb)
    wdec, walk = _walk(X, cb, (cb * cb).sum(-1))
    assert torch.equal(idx, walk) and torch.equal(dec, wdec), int((idx != walk).sum())


def _changed_table(how):
    cb = torch.from_numpy(O.e8_table()).to(DEV)
    if how == "rows in another order":                           # still the shell table
        return cb[torch.randperm(65536, generator=torch.Generator().manual_seed(1)).to(DEV)].contiguous()
    if how == "fewer rows of norm 12":
        return cb[:60000].contiguous()
    if how == "a row twice, one missing":                        # in number they are as many as before
        cb[300] = cb[40000]
    elif how == "a row of norm 12 twice":
        cb[65535] = cb[60000]
    elif how == "a row off the lattice":
        cb[1234, 0] += 0.25
    elif how == "a row that is not finite":
        cb[50000, 3] = float("nan")
    elif how == "scaled":
        cb *= 2
    return cb


@pytest.mark.parametrize("how", ["rows in another order", "fewer rows of norm 12", "a row twice, one missing", "a row of norm 12 twice",
                                 "a row off the lattice", "a row that is not finite", "scaled"])
@pytest.mark.parametrize("N", [3, 1500])
def test_e8_quantize_reads_its_table_on_every_call(how, N):
    """The same tensor with other contents, written where PyTorch counts no change, and tables that are almost the
    shell table: always the walk's rows."""
    from glq_amd import ext
    say("e8 shell search, changed table", how, N)
    cb = torch.from_numpy(O.e8_table()).to(DEV)
    X = torch.randn(N, 8, generator=torch.Generator().manual_seed(N)) * 1.5
    X[0] = 0.0                                                   # ties
    X[1] = torch.from_numpy(O.e8_table())[40000]
    X = X.to(DEV)
    norms = (cb * cb).sum(-1)
    dec, idx = ext.e8_quantize(X, cb, norms)
    wdec, widx = _walk(X, cb, norms)
    assert torch.equal(idx, widx) and torch.equal(dec, wdec)
    new = _changed_table(how)
    version = cb._version
    cb.data[:new.shape[0]].copy_(new)
    cb2, norms2 = cb[:new.shape[0]], norms[:new.shape[0]]
    norms.data.copy_((cb.data * cb.data).sum(-1))
    assert cb._version == version
    for given in (norms2, None):
        dec, idx = ext.e8_quantize(X, cb2, given)
        wdec, widx = _walk(X, cb2, norms2)
        assert torch.equal(idx, widx) and torch.equal(dec, wdec)


def test_e8_quantize_under_capture():
    """Captured on its first use, replayed on other vectors and with other table contents."""
    from glq_amd import ext
    say("e8 shell search under capture")
    g = torch.Generator().manual_seed(0)
    cb = torch.from_numpy(O.e8_table()).to(DEV)
    norms = (cb * cb).sum(-1)
    X = torch.zeros(700, 8, device=DEV)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        dec, idx = ext.e8_quantize(X, cb, norms)
    for turn in range(4):
        X.copy_(torch.randn(700, 8, generator=g) * (1 + turn))
        if turn == 2:
            cb.copy_(_changed_table("rows in another order"))
            norms.copy_((cb * cb).sum(-1))
        if turn == 3:
            cb.copy_(_changed_table("a row twice, one missing"))
            norms.copy_((cb * cb).sum(-1))
        graph.replay()
        torch.cuda.synchronize()
        wdec, widx = _walk(X, cb, norms)
        assert torch.equal(idx, widx) and torch.equal(dec, wdec), turn


@pytest.mark.parametrize("K", [1, 2, 3, 4])
def test_viterbi_matches_oracle_states(K, golden):
    """Tail-biting Viterbi: the reference's own tiles (golden vectors) and random tiles, state
    sequences and reconstructions bit-equal to the oracle (which is pinned on the reference)."""
    from glq_amd import ext
    say("viterbi", K)
    g = golden("trellis_viterbi")
    rng = np.random.default_rng(K)
    gk = K if f"K{K}_tiles" in g.files else 4           # the reference vectors hold K = 2 and 4
    tiles = np.concatenate([g[f"K{gk}_tiles"].astype(np.float32),
                            rng.standard_normal((5, 256)).astype(np.float32),
                            np.zeros((1, 256), np.float32),
                            (rng.standard_normal((2, 256)) * 3).astype(np.float32)])
    hat_ref, st_ref = O.trellis_quantize_tiles(tiles, K)
    hat, st = ext.trellis_quantize_tiles(t(tiles), K)
    st = st.cpu().numpy()
    bad = np.nonzero((st != st_ref).any(axis=1))[0]
    assert bad.size == 0, ("tiles differ", bad)
    assert np.array_equal(hat.cpu().numpy(), hat_ref)
    if gk == K:                                          # and directly against the reference's states
        assert np.array_equal(st[:6], g[f"K{K}_states"])
    # tail-biting: consecutive states overlap in 16-K bits, also across the wrap
    mask = (1 << (16 - K)) - 1
    assert np.array_equal(st[:, :-1] & mask, st[:, 1:] >> K)
    assert np.array_equal(st[:, -1] & mask, st[:, 0] >> K)
    again = ext.trellis_quantize_tiles(t(tiles), K)[1]
    assert np.array_equal(again.cpu().numpy(), st)


@pytest.mark.parametrize("K", [1, 2, 3, 4])
def test_pack_states_matches_oracle_layout(K):
    """states -> packed kernel layout, bit-equal to the oracle's packer; the HIP dequantizer
    reads the weights back."""
    from glq_amd import ext
    m, n = 64, 192
    say("pack states", K)
    p0 = O.random_packed(m, n, K, seed=K)
    st = O.trellis_states(p0, m, n).astype(np.int32)            # valid tail-biting sequences
    packed = ext.trellis_pack_states(t(st), m, n, K)
    assert np.array_equal(packed.cpu().numpy(), O.pack_layer_from_states(st, m, n, K))
    assert np.array_equal(packed.cpu().numpy(), p0)


def test_quantize_matrix_round_trip():
    """Whole encode path on the GPU: Gaussian matrix -> tiles -> Viterbi -> pack, then the
    decode kernels: decompress equals the encoder's own reconstruction bit for bit, and the
    quantization error is what 4 bpw gives (relative error ~0.07-0.1)."""
    from glq_amd import ext
    say("quantize matrix")
    m, n, K = 64, 128, 4
    W = torch.randn(m, n, generator=torch.Generator().manual_seed(0)) * 0.8934
    packed, recon = ext.trellis_quantize_matrix(W.to(DEV), K)
    Wd = ext.glq_decompress_trellis_3inst_cuda(packed, m, n)
    assert torch.equal(Wd.float(), recon)
    hat_ref, st_ref = O.trellis_quantize_tiles(O.matrix_to_tiles(W.numpy()), K)
    assert np.array_equal(packed.cpu().numpy(), O.pack_layer_from_states(st_ref, m, n, K))
    err = float(((recon.cpu() - W) ** 2).sum() / (W ** 2).sum())
    assert err < 0.02, err


@pytest.mark.parametrize("K,m,n", [(1, 32, 64), (2, 96, 64), (3, 32, 320), (4, 64, 192)])
def test_quantize_matrix_equals_the_tile_route(K, m, n):
    """The entry that reads and writes whole matrices against tiles -> search -> pack -> matrix, bit for bit, with
    inputs that leave a tile's costs tied (a constant block) and large ones."""
    from glq_amd import ext
    say("quantize matrix", K, m, n)
    W = torch.randn(m, n, generator=torch.Generator().manual_seed(K)) * 0.9
    W[:16, :16] = 0.25
    W[16:, 16:] *= 4.0
    W = W.to(DEV)
    packed, recon = ext.trellis_quantize_matrix(W, K)
    hat, states = ext.trellis_quantize_tiles(ext.trellis_matrix_to_tiles(W), K)
    assert torch.equal(packed, ext.trellis_pack_states(states, m, n, K))
    assert torch.equal(recon, ext.trellis_tiles_to_matrix(hat, m, n))
    if K > 1:                                            # the dequantizer takes 2..4 bits
        assert torch.equal(ext.glq_decompress_trellis_3inst_cuda(packed, m, n).float(), recon)


def _search_tiles(n, seed):
    """Gaussian tiles with some that the search on bounds leaves to the exact one or has to compare exactly: constant and
    alternating values, wide ones, inputs that are not finite, few distinct values (ties), tiny ones."""
    g = torch.Generator().manual_seed(seed)
    X = torch.randn(n, 256, generator=g) * 0.8933837
    pick = torch.randperm(n, generator=g)
    special = [torch.full((256,), 0.25), torch.zeros(256), torch.tensor([1.0, -1.0]).repeat(128), torch.randn(256, generator=g) * 3,
               torch.randn(256, generator=g) * 20, (torch.randn(256, generator=g) * 2).round() / 2, torch.randn(256, generator=g) * 1e-3,
               torch.randn(256, generator=g).index_fill(0, torch.tensor([7]), float("inf")), torch.linspace(-16, 16, 256)]
    for j, s in zip(pick[:n // 2].tolist(), special):
        X[j] = s
    return X


@pytest.mark.parametrize("K", [2, 3, 4])
@pytest.mark.parametrize("n", [257, 512, 513, 1025, 2051])
def test_viterbi_on_bounds_equals_the_exact_search(K, n):
    """Every route of the search on lower bounds (one and two tiles a workgroup, an odd last pair, one batch and batches
    that take turns): the states of all tiles step by step on cost rows in memory, of the same tiles searched a few at a
    time, which at 2 and 3 bits is the exact kernel (itself pinned on the oracle above), and of the oracle on some of them."""
    from glq_amd import ext
    say("viterbi on bounds", K, n)
    X = _search_tiles(n, 100 * K + n)
    hat, st = ext.trellis_quantize_tiles(X.to(DEV), K)
    exact = _exact_states(X, K)
    assert torch.equal(st, exact), (st != exact).any(1).nonzero()[:5]
    assert torch.equal(hat.cpu(), torch.from_numpy(O.lut_3inst().astype(np.float32))[exact.cpu().long()])
    few = [ext.trellis_quantize_tiles(c.to(DEV), K) for c in X.split(200)]
    assert torch.equal(st, torch.cat([f[1] for f in few])), (st != torch.cat([f[1] for f in few])).any(1).nonzero()[:5]
    assert torch.equal(hat, torch.cat([f[0] for f in few]))
    if n == 513:
        some = torch.cat([X[:12], X[-4:]])
        _, ref = O.trellis_quantize_tiles(some.numpy(), K)
        got = torch.cat([st[:12], st[-4:]]).cpu().numpy()
        finite = torch.isfinite(some).all(1).numpy()
        assert np.array_equal(got[finite], ref[finite])


def _exact_states(X, K, chunk=256):
    """The search of the oracle's `trellis_quantize_tiles` step by step on cost rows in memory: the single-step kernel (held
    to the reference's step in test_gpu_named_surface.py), lowest states on ties, and the walk back here."""
    from glq_amd import ext
    lut = t(O.lut_3inst())
    lutf, G = lut.float(), 1 << (16 - K)
    state = torch.arange(65536, device=DEV)

    def search(x, over=None):                            # x (b, 256) fp16 -> states (b, 256)
        cost = (lutf - x[:, :1].float()) ** 2
        if over is not None:
            cost = torch.where(state >> K == over[:, None], cost, torch.inf)
        prev = torch.empty(256, x.shape[0], G, dtype=torch.int32, device=DEV)
        for i in range(1, 256):
            cost = ext.viterbi_acs_step(cost, x[:, i].contiguous(), lutf, K, prev[i])
        if over is not None:
            cost = torch.where(state & (G - 1) == over[:, None], cost, torch.inf)
        at = torch.where(cost == cost.min(1, keepdim=True).values, state, 65536).min(1).values
        states = torch.empty(x.shape, dtype=torch.int64, device=DEV)
        for i in range(255, -1, -1):
            states[:, i] = at
            if i:
                at = prev[i].gather(1, (at >> K)[:, None])[:, 0].long()
        return states

    out = []
    for x in X.to(DEV).half().split(chunk):
        out.append(search(x, search(x.roll(128, 1))[:, 128] >> K))
    return torch.cat(out).int()


@pytest.mark.parametrize("K", [2, 3, 4])
@pytest.mark.parametrize("kind", ["decoded", "one value a rounding off", "noise of 1e-5", "noise of 2e-7"])
def test_viterbi_of_decoded_weights(K, kind):
    """Tiles that are decoded tail-biting paths, or nearly: their best path costs nothing or so little that all its bounds in
    fp16 are zero."""
    from glq_amd import ext
    say("viterbi of decoded weights", K, kind)
    n = 300                                              # more than a tile per CU: on bounds at every K
    lut = torch.from_numpy(O.lut_3inst().astype(np.float16))
    X = lut[torch.from_numpy(O.trellis_states(O.random_packed(160, 480, K, seed=K), 160, 480).astype(np.int64))].reshape(n, 256).float()
    g = torch.Generator().manual_seed(K)
    if kind == "one value a rounding off":
        at = X.abs().argsort(1)[torch.arange(n), torch.randint(0, 64, (n,), generator=g)]   # one of the smaller values
        v = X[torch.arange(n), at].half()
        X[torch.arange(n), at] = torch.nextafter(v, torch.full_like(v, 8.0)).float()
    elif kind.startswith("noise"):
        X = X + torch.randn(n, 256, generator=g) * float(kind.split()[-1])
    hat, st = ext.trellis_quantize_tiles(X.to(DEV), K)
    ref = _exact_states(X, K)
    assert torch.equal(st, ref), (st != ref).any(1).nonzero()[:5]
    assert torch.equal(hat.cpu(), lut[ref.long().cpu()].float())
    assert np.array_equal(st[:3].cpu().numpy(), O.trellis_quantize_tiles(X[:3].numpy(), K)[1])
    if kind == "decoded":
        assert torch.equal(hat.cpu(), X)


def _quantize_counts(X, K):
    """States, and how many tiles the search on bounds tried and left (the counts that end its workspace)."""
    from glq_amd import _lib
    lib, n = _lib.load(), X.shape[0]
    X, states, hat = X.to(DEV), torch.empty(n, 256, dtype=torch.int32, device=DEV), torch.empty(n, 256, device=DEV)
    ws = torch.zeros(lib.glqh_trellis_quantize_workspace_bytes(K, n), dtype=torch.uint8, device=DEV)
    _lib.check(lib.glqh_trellis_quantize_tiles(X.data_ptr(), n, K, states.data_ptr(), hat.data_ptr(), ws.data_ptr(), ws.numel(),
                                               torch.cuda.current_stream().cuda_stream))
    return states, *ws[-256:].view(torch.int32)[:2].tolist()


@pytest.mark.parametrize("K", [2, 3, 4])
@pytest.mark.parametrize("kind", ["normal", "wide", "wide among normal", "normal among wide", "ramps"])
def test_viterbi_tiles_on_either_search(K, kind):
    """Which tiles the search on bounds tries, how many it leaves, and the exact states of all of them: normal values (tried,
    and a few in a thousand left), values far beyond the weights' range (not tried), both mixed, a majority (only the
    normal ones) and a minority of normal ones (none), and ramps, which the lists do not hold: not tried to the end."""
    say("viterbi on either search", K, kind)
    n = 2500 if kind == "ramps" else 700
    g = torch.Generator().manual_seed(K)
    X = torch.randn(n, 256, generator=g) * 0.9
    wide = torch.zeros(n, dtype=torch.bool)
    if kind.startswith("wide"):
        wide[:] = kind == "wide"
        wide[::3] = True
    elif kind == "normal among wide":
        wide[:] = True
        wide[::3] = False
    X[wide] *= 7
    if kind == "ramps":
        X = torch.linspace(-3, 3, 256) + X * 1e-3
    states, tried, left = _quantize_counts(X, K)
    if kind == "ramps":
        assert n > tried and left > tried // 2, (tried, left)
    else:
        assert tried == {"normal": n, "wide": 0, "wide among normal": n - int(wide.sum()), "normal among wide": 0}[kind], tried
        assert left <= n // 50, left
    ref = _exact_states(X, K)
    assert torch.equal(states, ref), (states != ref).any(1).nonzero()[:5]


def test_ramps_at_2_bits_are_left_at_their_first_overflow():
    """Slow ramps fill the lists of the walk back: at K = 2 all go to the exact search without a second walk, and come out exact."""
    say("ramps at 2 bits")
    X = torch.linspace(-3, 3, 256) + torch.randn(1024, 256, generator=torch.Generator().manual_seed(2)) * 1e-3
    states, tried, left = _quantize_counts(X, 2)
    assert (tried, left) == (1024, 1024)
    assert torch.equal(states, _exact_states(X, 2))


def test_wide_tiles_at_3_bits_are_left_at_their_first_overflow():
    """Normal values of sigma 2: the lists of the walk back hold most tiles' ways, and at K = 3 the others (6-8 % of those tried; half the
    slack would leave 1 %) go to the exact search without a second walk."""
    say("wide tiles at 3 bits")
    X = torch.randn(2000, 256, generator=torch.Generator().manual_seed(3)) * 2.0
    states, tried, left = _quantize_counts(X, 3)
    assert tried > 1200 and left > tried // 25, (tried, left)
    assert torch.equal(states, _exact_states(X, 3))


def test_tiny_values_at_4_bits_fit_the_lists():
    """Normal values of sigma 1e-4 keep many ways: lists of 768 leave three tiles in ten (of 672 four and more), a call of less
    than twelve tiles a CU without a second walk; the exact states."""
    say("tiny values at 4 bits")
    X = torch.randn(1024, 256, generator=torch.Generator().manual_seed(4)) * 1e-4
    states, tried, left = _quantize_counts(X, 4)
    assert tried == 1024 and 256 <= left <= 384, (tried, left)
    assert torch.equal(states, _exact_states(X, 4))


@pytest.mark.parametrize("K,m,n", [(2, 256, 320), (3, 288, 256), (4, 512, 576)])
def test_quantize_matrix_on_bounds_equals_the_tile_route(K, m, n):
    """More tiles than CUs, whose places in the matrix the lists tell, all but two of them on bounds: the tile route, bit for bit."""
    from glq_amd import ext
    say("quantize matrix on bounds", K, m, n)
    W = torch.randn(m, n, generator=torch.Generator().manual_seed(K)) * 0.9
    W[:16, :16] = 0.25
    W[-16:, 32:48] *= 8
    W = W.to(DEV)
    packed, recon = ext.trellis_quantize_matrix(W, K)
    tiles = ext.trellis_matrix_to_tiles(W)
    states, tried, _ = _quantize_counts(tiles, K)
    assert tried == tiles.shape[0] - 2
    assert torch.equal(packed, ext.trellis_pack_states(states, m, n, K))
    assert torch.equal(recon, ext.trellis_tiles_to_matrix(ext.trellis_quantize_tiles(tiles, K)[0], m, n))
    assert torch.equal(ext.glq_decompress_trellis_3inst_cuda(packed, m, n).float(), recon)


@pytest.mark.parametrize("K,n", [(2, 1025), (3, 2000), (4, 1700), (1, 600), (4, 3)])
def test_viterbi_in_the_least_workspace(K, n, monkeypatch):
    """Where the larger workspace is not to be had: the least one, half of it for many tiles, gives the same states; a byte
    less is refused."""
    from glq_amd import _lib, ext
    say("viterbi least workspace", K, n)
    lib = _lib.load()
    most, least = lib.glqh_trellis_quantize_workspace_bytes(K, n), lib.glqh_trellis_quantize_least_workspace_bytes(K, n)
    assert least < 0.51 * most if K > 1 and n > 1000 else least <= most
    X = _search_tiles(n, n)
    hat, states = ext.trellis_quantize_tiles(X.to(DEV), K)
    W = torch.randn(512, 1024, generator=torch.Generator().manual_seed(K)).to(DEV)
    want = ext.trellis_quantize_matrix(W, K)
    taken, plain = [], ext._ws
    larger = {most} - {least}
    if K > 1:
        larger.add(lib.glqh_trellis_quantize_matrix_workspace_bytes(K, 512, 1024))

    def short(nbytes, device):
        taken.append(nbytes)
        if nbytes in larger:
            raise torch.OutOfMemoryError("short of memory")
        return plain(nbytes, device)

    monkeypatch.setattr(ext, "_ws", short)
    got = ext.trellis_quantize_tiles(X.to(DEV), K)
    assert taken[-1] == least
    assert torch.equal(got[1], states) and torch.equal(got[0], hat)
    assert all(torch.equal(a, b) for a, b in zip(ext.trellis_quantize_matrix(W, K), want))
    monkeypatch.undo()
    ws = torch.empty(least - 1, dtype=torch.uint8, device=DEV)
    x = X.to(DEV)
    with pytest.raises(RuntimeError, match="workspace"):
        _lib.check(lib.glqh_trellis_quantize_tiles(x.data_ptr(), n, K, states.data_ptr(), hat.data_ptr(), ws.data_ptr(), ws.numel(),
                                                   torch.cuda.current_stream().cuda_stream))


@pytest.mark.parametrize("kind,n", [("wide among normal", 3200), ("wide among normal", 8300), ("1500 normal, then ramps", 4300),
                                    ("500 normal, then ramps", 4300), ("ramps", 4200), ("ramps, then wide", 6000)])
def test_viterbi_by_products_over_chips_that_are_not_full(kind, n):
    """At K = 4 a chip of tiles goes through the matrix products only where twelve tiles a CU of it are tried (not 1760 of 3200, whose
    rows then fill 2 GB, nor what 4565 of 8300 leave behind the first chip); one of whose tiles the first pass leaves all
    but three a CU is given up, others are not; the exact states of all tiles throughout."""
    from glq_amd import _lib
    say("viterbi by products, chips not full", kind, n)
    g = torch.Generator().manual_seed(n)
    X = torch.randn(n, 256, generator=g) * 0.9
    ramps = torch.linspace(-3, 3, 256) + torch.randn(n, 256, generator=g) * 1e-3
    wide = n * 9 // 20
    if kind == "wide among normal":
        X[torch.randperm(n, generator=g)[:wide]] *= 7
    elif kind == "ramps, then wide":
        X *= 7
        X[:3200] = ramps[:3200]
    else:
        first = int(kind.split()[0]) if kind != "ramps" else 0
        X[first:] = ramps[first:]
    lib, x = _lib.load(), X.to(DEV)
    states, hat = torch.empty(n, 256, dtype=torch.int32, device=DEV), torch.empty(n, 256, device=DEV)
    ws = torch.full((lib.glqh_trellis_quantize_workspace_bytes(4, n),), 0xA5, dtype=torch.uint8, device=DEV)
    _lib.check(lib.glqh_trellis_quantize_tiles(x.data_ptr(), n, 4, states.data_ptr(), hat.data_ptr(), ws.data_ptr(), ws.numel(),
                                               torch.cuda.current_stream().cuda_stream))
    tried, left = ws[-256:].view(torch.int32)[:2].tolist()
    if kind == "wide among normal":
        assert tried == n - wide and left <= n // 100, (tried, left)
        untouched = int((ws[2200 << 20:3000 << 20] != 0xA5).sum()) == 0   # (a failing assertion would list a tensor compared in it)
        assert untouched == (n == 3200)
    elif kind == "1500 normal, then ramps":
        assert tried == 4096 and 2560 <= left <= 2620, (tried, left)
    else:
        assert (tried, left) == (0, 0), (tried, left)
    ref = _exact_states(X, 4)
    assert torch.equal(states, ref), (states != ref).any(1).nonzero()[:5]


def _quantize_in(X, K, nbytes):
    """States from a workspace of that many bytes, and the last of them that were written."""
    from glq_amd import _lib
    n = X.shape[0]
    x, states, hat = X.to(DEV), torch.empty(n, 256, dtype=torch.int32, device=DEV), torch.empty(n, 256, device=DEV)
    ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=DEV)
    _lib.check(_lib.load().glqh_trellis_quantize_tiles(x.data_ptr(), n, K, states.data_ptr(), hat.data_ptr(), ws.data_ptr(), nbytes,
                                                       torch.cuda.current_stream().cuda_stream))
    changed = (ws.view(-1, 256) != 0xA5).any(1).nonzero()
    return states, 256 * (int(changed[-1]) + 1)


@pytest.mark.parametrize("n", [3072, 4500])
def test_viterbi_between_the_least_workspace_and_the_most(n, monkeypatch):
    """At K = 4 from twelve tiles per CU on: twice the least workspace is used as such (batches of four tiles per CU), the most
    as such, and the least; the exact states from each of them.  The Python entry tries them in turn."""
    from glq_amd import _lib, ext
    say("viterbi between least and most", n)
    lib = _lib.load()
    most, least = lib.glqh_trellis_quantize_workspace_bytes(4, n), lib.glqh_trellis_quantize_least_workspace_bytes(4, n)
    assert 2 * least < most
    X = _search_tiles(n, n)
    ref = _exact_states(X, 4)
    for nbytes, lo, hi in ((most, most, most), (most - 256, 1.9 * least, 2 * least), (2 * least, 1.9 * least, 2 * least),
                           (least, least, least)):
        states, used = _quantize_in(X, 4, nbytes)
        assert lo <= used <= hi, (nbytes, used)
        assert torch.equal(states, ref), (nbytes, (states != ref).any(1).nonzero()[:5])
    taken, plain = [], ext._ws

    def short(nbytes, device):
        taken.append(nbytes)
        if nbytes > 2 * least:
            raise torch.OutOfMemoryError("short of memory")
        return plain(nbytes, device)

    monkeypatch.setattr(ext, "_ws", short)
    assert torch.equal(ext.trellis_quantize_tiles(X.to(DEV), 4)[1], ref)
    assert taken == [most, 2 * least]


def test_viterbi_under_capture():
    """Captured and replayed on other tiles: the launches' batches hand each other their rows through the same memory."""
    from glq_amd import ext
    say("viterbi under capture")
    X = torch.zeros(1100, 256, device=DEV)
    lut = t(O.lut_3inst().astype(np.float32))
    ext.trellis_quantize_tiles(X[:4], 4)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        hat, st = ext.trellis_quantize_tiles(X, 4)
    for turn in range(3):
        X.copy_(_search_tiles(1100, turn))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(st, _exact_states(X, 4)), turn
        assert torch.equal(hat, lut[st.long()]), turn


@pytest.mark.parametrize("n", [3072, 3081, 4396])
def test_viterbi_by_products_equals_the_exact_search(n):
    """Calls that fill the chip at K = 4, whose forward pass is matrix products: the smallest of them, a last workgroup with one
    tile, and a full chip with a rest for the other route; special tiles among them, decoded ones, and some whose best path costs
    about what the bounds are made for, or more.  A few in a thousand may be left to the exact search, not more."""
    say("viterbi by products", n)
    X = _search_tiles(n, n)
    X[-1] = torch.randn(256, generator=torch.Generator().manual_seed(n)) * 0.9   # the last workgroup's, in order and tried
    X[100:140] *= torch.linspace(1, 2.4, 40)[:, None]
    lut = torch.from_numpy(O.lut_3inst().astype(np.float32))
    X[200:260] = lut[torch.from_numpy(O.trellis_states(O.random_packed(96, 160, 4, seed=4), 96, 160).astype(np.int64))].reshape(60, 256)
    X[230:260] += torch.randn(30, 256, generator=torch.Generator().manual_seed(1)) * 1e-3
    states, tried, left = _quantize_counts(X, 4)
    assert tried > n - 40 and left <= n // 100, (tried, left)
    ref = _exact_states(X, 4)
    assert torch.equal(states, ref), (states != ref).any(1).nonzero()[:5]


def test_bounds_of_the_products_are_bounds():
    """What the matrix products leave in the workspace, against the costs in float64: no bound of any group at any stored step
    is above the least cost from the start (beyond the roundings of what moves out of the rows, 2^-24 of it each time), and the
    limit of the walk back is not below the best path's cost.  Normal tiles, tiny ones, decoded paths whose sums cancel to nothing,
    and the largest values that are tried, alone and several."""
    from glq_amd import _lib
    say("bounds of the products")
    n, K, G, levels = 3072, 4, 4096, 128
    g = torch.Generator().manual_seed(11)
    X = torch.randn(n, 256, generator=g) * 0.9
    X[16:24] *= torch.linspace(1.1, 1.7, 8)[:, None]
    X[24:28] *= 0.05
    X[28:32, 100] = torch.tensor([5.98, -5.98, 5.5, -5.0])
    X[32:36, ::64] = 4.98 * torch.tensor([1.0, -1.0, 1.0, -1.0])
    lut = torch.from_numpy(O.lut_3inst().astype(np.float32))
    X[36:44] = lut[torch.from_numpy(O.trellis_states(O.random_packed(32, 64, 4, seed=4), 32, 64).astype(np.int64))].reshape(-1, 256)
    X[40:44] += 1e-3 * torch.randn(4, 256, generator=g)
    lib, x = _lib.load(), X.to(DEV)
    states, hat = torch.empty(n, 256, dtype=torch.int32, device=DEV), torch.empty(n, 256, device=DEV)
    ws = torch.zeros(lib.glqh_trellis_quantize_workspace_bytes(K, n), dtype=torch.uint8, device=DEV)
    _lib.check(lib.glqh_trellis_quantize_tiles(x.data_ptr(), n, K, states.data_ptr(), hat.data_ptr(), ws.data_ptr(), ws.numel(),
                                               torch.cuda.current_stream().cuda_stream))
    assert ws[-256:].view(torch.int32)[:2].tolist() == [n, 0]    # all are tried, in their order, and none left: the rows are as they were
    T = 48
    rows = ws[:levels * n * G * 2].view(torch.float16).view(levels, n, G)
    info = ws[levels * n * G * 2:levels * n * G * 2 + n * 520].view(n, 130, 4)[:T].contiguous()
    pre, over = info[:, :129].contiguous().view(torch.float32)[:, :, 0].double(), info[:, 129].contiguous().view(torch.int32)[:, 0].long()
    group = torch.arange(G, device=DEV)                          # where a row holds a group's bound
    k, a = group >> 8, group & 255
    at = a * 16 + (((k >> 1) ^ (a >> 5 & 7)) << 1) + (k & 1)
    a = at >> 4
    at = ((a & 15) << 4 | a >> 4) << 4 | (at & 15)
    assert torch.equal(at.sort().values, group)
    w, v = lut.to(DEV).double(), x[:T].half().double()
    cost = torch.full((T, 16, G), torch.inf, dtype=torch.float64, device=DEV)   # of states by their high digit and group
    cost[torch.arange(T, device=DEV), :, over] = 0.0
    for i in range(256):
        least = cost.amin(1)
        if i and i % 2 == 0:
            bound, moved = rows[i // 2 - 1, :T][:, at].double(), pre[:, i // 2, None]
            assert float((bound + moved - least - i // 2 * 2 ** -24 * moved).max()) <= 0.0, i
        # state s follows the groups s >> 4
        cost = (least.repeat_interleave(16, 1) + (v[:, i, None] - w) ** 2).view(T, 16, G)
    best = cost.amin(1).gather(1, over[:, None])[:, 0]
    bound, moved = rows[127, :T][:, at].double().gather(1, over[:, None])[:, 0], pre[:, 128]
    assert float((bound + moved - best - 128 * 2 ** -24 * moved).max()) <= 0.0
    lost = 256 * 2 ** -19 + (30 * 2 ** -24 * v * v + 2 ** -24).sum(1)
    room = (bound + moved) * 1.0042 + lost - best
    say("least room under the limit, relative", float((room / best.clamp_min(1e-3)).min()))
    assert float(room.min()) >= 0.0


def test_quantize_matrix_by_products_over_several_chips():
    """2048 x 1088 at K = 4: two chips of tiles one after the other through the same rows, and a rest, read and written in the
    matrix; some tiles left in either chip and some not tried.  The packed exact states."""
    from glq_amd import ext
    say("quantize matrix by products")
    m, n = 2048, 1088
    g = torch.Generator().manual_seed(8)
    X = torch.randn(m * n // 256, 256, generator=g) * 0.9
    X[::40] = torch.linspace(-3, 3, 256) + 1e-3 * torch.randn(X[::40].shape, generator=g)   # ramps show nothing beforehand and fill the lists
    X[5::500] *= 8
    W = ext.trellis_tiles_to_matrix(X.to(DEV), m, n)
    packed, recon = ext.trellis_quantize_matrix(W, 4)
    tiles = ext.trellis_matrix_to_tiles(W)
    states, tried, left = _quantize_counts(tiles.cpu(), 4)
    assert tried == X.shape[0] - 18 and left >= 200, (tried, left)
    ref = _exact_states(X, 4)
    assert torch.equal(tiles.cpu(), X) and torch.equal(states, ref)
    assert torch.equal(packed, ext.trellis_pack_states(ref, m, n, 4))
    assert torch.equal(ext.glq_decompress_trellis_3inst_cuda(packed, m, n).float(), recon)


def test_viterbi_by_products_under_capture():
    """Captured and replayed on other tiles, with eager work between."""
    from glq_amd import ext
    say("viterbi by products under capture")
    n = 3100
    X = torch.zeros(n, 256, device=DEV)
    ext.trellis_quantize_tiles(X[:4], 4)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        _, st = ext.trellis_quantize_tiles(X, 4)
    for turn in range(3):
        X.copy_(_search_tiles(n, turn))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(st, ext.trellis_quantize_tiles(X, 4)[1]), turn
    assert torch.equal(st, _exact_states(X.cpu(), 4))
