"""Shapes with too few tiles to fill the GPU: the forward kernel of 32-query
tiles (csrc/sdpa_f16_fwd_small.hip), its division of a tile's keys over
workgroups, and the edges of both against the oracle."""
import numpy as np
import pytest
import torch

from _common import TOL, Cfg, make_inputs, maxabs, oracle_kw
from test_parity_gpu import _np, _t, run_and_check

pytestmark = pytest.mark.gpu

FWD = [
    # B, S_q, S_kv, D_qk, D_v, causal, dropout; parts of a tile's keys
    (2, 1, 1, 64, 64, False, 0.0, 1),        # one block, one wave
    (3, 33, 97, 40, 72, False, 0.1, 1),      # a block more than the waves, ragged widths
    (2, 129, 129, 128, 128, True, 0.1, 1),   # the diagonal block, a one-row tile
    (1, 31, 1551, 128, 64, False, 0.2, 6),   # parts of unequal length, a ragged tail
    (2, 32, 4096, 32, 128, False, 0.0, 16),  # two blocks per wave
    (5, 2, 3001, 64, 64, False, 1.5, 12),    # every element dropped
    (2, 70, 100, 36, 4, False, 0.1, 1),      # features a multiple of 4 only, on either side
    (2, 33, 2050, 20, 60, False, 0.0, 8),    # the same in parts
    (3, 2881, 1999, 128, 96, False, 0.1, 3),  # the 128-query kernel in parts, ragged
]


@pytest.mark.parametrize("case", FWD, ids=["-".join(map(str, c)) for c in FWD])
def test_small_forward(pkg, O, case):
    B, S_q, S_kv, D_qk, D_v, causal, p, parts = case
    c = Cfg("small_fwd", "f16", B, S_q, S_kv, D_qk, D_v, causal, p, D_qk ** -0.5, 3, 17)
    L = pkg.library()
    rows = parts * B * S_q
    want = 0 if parts == 1 else (rows * D_v * 4 + 255) // 256 * 256 + rows * 8
    dims = (1, B, S_q, S_kv, D_qk, D_v, int(causal))
    assert L.sdpa_hip_fwd_workspace_bytes(*dims) == want
    run_and_check(pkg, O, c)

    # a workspace one byte short, or none, runs undivided: the same bits
    q, k, v = (_t(a) for a in make_inputs(c)[:3])
    outs = []
    for ws_bytes in (want, max(want - 1, 0), 0):
        ws = torch.empty((max(want, 1),), dtype=torch.uint8, device=q.device)
        o = torch.empty((B, S_q, D_v), dtype=q.dtype, device=q.device)
        s = torch.empty((B, S_q), dtype=torch.float32, device=q.device)
        rc = L.sdpa_hip_fwd_ws(1, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), s.data_ptr(),
                               ws.data_ptr(), ws_bytes, B, S_q, S_kv, D_qk, D_v, c.scale, p, int(causal), c.seed,
                               c.offset, torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        torch.cuda.synchronize()
        outs.append((_np(o), _np(s)))
    for a, b in zip(outs[1], outs[2]):
        assert np.array_equal(a, b)
    # Both forms against the oracle at the op's tolerance (they round P~ to
    # half relative to different running maxima, so their bits differ).
    o_ref, s_ref = O.sdpa_fwd_gate(*make_inputs(c)[:3], **oracle_kw(c))
    for o, s in (outs[0], outs[2]):
        assert maxabs(o, o_ref) <= TOL["f16"]["o"] and maxabs(s, s_ref) <= TOL["f16"]["stats"]


F32 = [
    # B, S_q, S_kv, D_qk, D_v, causal, dropout, scale; whether the keys are divided
    (2, 129, 64, 64, 64, False, 0.1, 0.125, False),     # one block, a one-row tile
    (1, 33, 2049, 128, 128, False, 0.0, 0.1, True),     # 32-key blocks, parts, a one-key tail
    (2, 65, 65, 37, 5, True, 0.2, -0.2, False),         # element loads, negated scale
    (2, 200, 200, 32, 128, True, 0.1, 0.0, True),       # scale 0
    (3, 1, 700, 128, 64, False, 1.5, 0.1, True),        # every element dropped
    (1, 17, 8193, 40, 36, False, 0.1, 0.16, False),     # the sequential fp32 sums (more than 8192 keys)
    (1, 33, 8225, 126, 6, False, 0.0, 0.09, False),     # the same with rows of no whole chunks
    (257, 3, 31, 64, 64, False, 0.1, -0.125, False),    # few keys against more than 256 tiles: the fp32 instruction
    (129, 160, 160, 37, 128, True, 0.2, 0.1, False),    # the same, causal, within its lengths
    (260, 2, 161, 64, 33, False, 0.0, 0.125, False),    # one key more than it takes without the mask
]


@pytest.mark.parametrize("case", F32, ids=["-".join(map(str, c)) for c in F32])
def test_f32_forward(pkg, O, case):
    """The fp32 forward on the bf16 matrix cores: o within 1e-5 and, where
    keys are divided, the undivided form as well."""
    B, S_q, S_kv, D_qk, D_v, causal, p, scale, divided = case
    c = Cfg("f32_fwd", "f32", B, S_q, S_kv, D_qk, D_v, causal, p, scale, 3, 17)
    q, k, v, _ = make_inputs(c)
    o_ref, s_ref = O.sdpa_fwd_gate(q, k, v, **oracle_kw(c))
    L = pkg.library()
    want = L.sdpa_hip_fwd_workspace_bytes(0, B, S_q, S_kv, D_qk, D_v, int(causal))
    assert (want > 0) == divided
    t = [_t(a) for a in (q, k, v)]
    for ws_bytes in {want, 0}:
        ws = torch.empty((max(want, 1),), dtype=torch.uint8, device=t[0].device)
        o = torch.empty((B, S_q, D_v), dtype=torch.float32, device=t[0].device)
        s = torch.empty((B, S_q), dtype=torch.float32, device=t[0].device)
        rc = L.sdpa_hip_fwd_ws(0, *(a.data_ptr() for a in t), o.data_ptr(), s.data_ptr(), ws.data_ptr(), ws_bytes,
                               B, S_q, S_kv, D_qk, D_v, scale, p, int(causal), c.seed, c.offset,
                               torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        torch.cuda.synchronize()
        assert maxabs(_np(o), o_ref) <= TOL["f32"]["o"] and maxabs(_np(s), s_ref) <= TOL["f32"]["stats"]


@pytest.mark.parametrize("S_q,S_kv", [(16, 64), (16, 4000), (300, 2000)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_stats_without_values(pkg, dtype, S_q, S_kv):
    """D_v = 0: o is empty, stats are those of the scores (also where other
    value sizes would take the kernel of 32-query tiles or divided keys)."""
    g = torch.Generator().manual_seed(4)
    B = 2 if S_q == 16 else 32
    q, k = (torch.randn((B, n, 64), generator=g).to(dtype).cuda() for n in (S_q, S_kv))
    junk = torch.full((B * S_q,), 777.0, device="cuda")
    del junk  # stats take its place
    o, s = pkg.sdpa(q, k, torch.empty((B, S_kv, 0), dtype=dtype, device="cuda"), scale=0.1)
    ref = torch.logsumexp(torch.bmm(q.double(), k.double().transpose(1, 2).contiguous()) * 0.1, -1)
    assert o.shape == (B, S_q, 0)
    assert (s.double() - ref).abs().max().item() <= TOL["f32"]["stats"]


def test_f32_grid_of_more_threads_than_one_dimension(pkg):
    """2^23 + 5 batch rows of one query and one key: with 512 threads per tile
    more than the 2^32 - 1 threads of a grid dimension.  The one weight is 1,
    so o = v (times 1 / (1 + 1e-6), within the op's 1e-5), dV = dO and dQ = dK = 0,
    each to the rounding of P and of sums of two terms below 40."""
    B = (1 << 23) + 5
    g = torch.Generator(device="cuda").manual_seed(6)
    q, k, v, d_o = (torch.randn((B, 1, 2), generator=g, device="cuda") for _ in range(4))
    o, s = pkg.sdpa(q, k, v, scale=0.5)
    dq, dk, dv = pkg.sdpa_grad(q, k, v, o, s, d_o, scale=0.5)
    assert (o - v).abs().max().item() <= 1e-5
    assert (s - (q * k).sum(2) * 0.5).abs().max().item() <= 1e-4
    assert (dv - d_o).abs().max().item() <= 1e-4
    assert dq.abs().max().item() <= 1e-4 and dk.abs().max().item() <= 1e-4
    # the forward of 512 threads takes more than 160 keys there
    del o, s, dq, dk, dv, v, d_o
    q = q[..., :1].contiguous()
    k, v = (torch.randn((B, 161, 1), generator=g, device="cuda") for _ in range(2))
    o, _ = pkg.sdpa(q, k, v, scale=0.5)
    for i in range(0, B, 1 << 20):
        j = slice(i, i + (1 << 20))
        ref = (torch.softmax(q[j] * k[j] * 0.5, 1) * v[j]).sum(1, keepdim=True)
        assert (o[j] - ref).abs().max().item() <= 1e-5


@pytest.mark.parametrize("dtype,D", [(torch.float16, 64), (torch.float32, 64), (torch.float16, 128)])
def test_workspace_that_cannot_be_had(pkg, monkeypatch, dtype, D):
    """Calls whose tiles would be divided, or whose dS stored, run undivided
    where the memory for it is not there."""
    g = torch.Generator().manual_seed(11)
    q, k, v, d_o = (torch.randn((2, n, D), generator=g).to(dtype).cuda() for n in (16, 3000, 3000, 16))
    o, s = pkg.sdpa(q, k, v, scale=0.1)
    want = (o, s) + pkg.sdpa_grad(q, k, v, o, s, d_o, scale=0.1)
    empty, refused, rows = torch.empty, [], pkg.library().sdpa_hip_bwd_workspace_bytes(2, 16)

    def no_room(size, **kw):
        if kw.get("dtype") is torch.uint8 and size[0] > rows:
            refused.append(size[0])
            raise torch.OutOfMemoryError("no room")
        return empty(size, **kw)

    monkeypatch.setattr(torch, "empty", no_room)
    got = pkg.sdpa(q, k, v, scale=0.1) + pkg.sdpa_grad(q, k, v, o, s, d_o, scale=0.1)
    assert len(refused) == 2
    tol = TOL["f16" if dtype == torch.float16 else "f32"]
    for name, a, b in zip(("o", "stats", "grad", "grad", "grad"), got, want):
        assert (a.float() - b.float()).abs().max().item() <= tol[name] * max(1.0, b.float().abs().max().item())


def test_half4_neighbour_row(pkg):
    """An infinity in a row does not reach the row before it, whose last chunk
    is copied with the first features of that one."""
    g = torch.Generator().manual_seed(2)
    q, k, v = ((torch.rand((1, 64, 12), generator=g) + 0.1).half().cuda() for _ in range(3))
    k[0, 7, 0] = float("-inf")  # key 7 weighs 0; key 6 keeps its weight
    o, s = pkg.sdpa(q, k, v, scale=0.3)
    ref = torch.softmax(q.double().cpu() @ k.double().cpu().transpose(1, 2) * 0.3, -1) @ v.double().cpu()
    assert (o.double().cpu() - ref).abs().max().item() <= 2e-3
    k[0, 7, 0] = 0.5
    v[0, 9, 0] = float("inf")  # dP of key 8 stays finite
    d_o = torch.randn((1, 64, 12), generator=g).half().cuda()
    o = torch.zeros_like(q)
    _, dk, _ = pkg.sdpa_grad(q, k, v, o, s, d_o, scale=0.3)
    assert torch.isfinite(dk[0, 8].float()).all() and not torch.isfinite(dk[0, 9].float()).all()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D_qk,D_v,S_kv", [(36, 60, 50), (64, 64, 50), (12, 60, 1100)])
def test_small_backward_large_dp(pkg, D_qk, D_v, S_kv, causal):
    """A factor dP / (1-p) - delta of 4e8 (dO 30000, v 200: all finite) beside
    weights that are 0, of a gated key and of masked ones, leaves dQ finite
    and within the rounding of dS and of the result to fp16 (2^-10 of the sum
    of its terms' magnitudes; 2^-24 below fp16's normal range, for a dS and for
    the result) and that of the fp32 sums dP and delta, 64 terms of 2^-24 each,
    which cancel in a row of one visible key."""
    if causal and S_kv != 50:
        pytest.skip("one long side only")
    g = torch.Generator().manual_seed(0)
    S_q = 50 if causal else 40
    q, k = torch.randn((1, S_q, D_qk), generator=g).half(), torch.randn((1, S_kv, D_qk), generator=g).half()
    v, d_o = torch.randn((1, S_kv, D_v), generator=g).half(), torch.randn((1, S_q, D_v), generator=g).half()
    q[:, :, 0] = 4
    v *= 0.05  # the factors of the other keys leave dS below 65504
    k[0, 7], v[0, 7] = 0, 200
    k[0, 7, 0] = -60  # a weight of 0
    d_o[0, 25] = 30000
    c = [t.cuda() for t in (q, k, v)]
    o, s = pkg.sdpa(*c, scale=0.2, causal_mask=causal)
    dq, _, _ = pkg.sdpa_grad(*c, o, s, d_o.cuda(), scale=0.2, causal_mask=causal)
    Q, K, V, G, O_, st = (t.double().cpu() for t in (q, k, v, d_o, o, s))
    p = torch.exp(Q @ K.transpose(1, 2) * 0.2 - st[..., None])
    if causal:
        p = p.tril()
    p = torch.where(p <= 1e-6, 0.0, p)
    ds = p * (G @ V.transpose(1, 2) - (G * O_).sum(2, keepdim=True))
    assert 50 < ds[0, 25].abs().max() < 60000 and p[0, 25, 7] == 0
    sums = p * (G.abs() @ V.abs().transpose(1, 2) + (G * O_).abs().sum(2, keepdim=True)) * 2.0 ** -18
    bound = ((ds.abs() * 2.0 ** -10 + sums + 2.0 ** -24) @ K.abs()) * 0.2 + 2.0 ** -24
    assert ((dq.double().cpu() - ds @ K * 0.2).abs() <= bound).all()


@pytest.mark.parametrize("D", [36, 64])
def test_small_dk_of_small_gradients(pkg, D):
    """dK at dropout 0.9 and dO of 1e-3, where most of dS lies near fp16's
    smallest normal value: dS and the result each round to half of 2^-10 at
    most, 2.8e-4 in root mean square, 4e-4 together; twice that."""
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn((4, 512, D), generator=g).half().cuda() for _ in range(3))
    d_o = (torch.randn((4, 512, D), generator=g) * 1e-3).half().cuda()
    kw = dict(dropout=0.9, scale=D ** -0.5)
    keep = pkg.dropout_keep_mask(4, 512, 512, 0.9, 5, 9).double()
    o, s = pkg.sdpa(q, k, v, 5, 9, **kw)
    _, dk, _ = pkg.sdpa_grad(q, k, v, o, s, d_o, 5, 9, **kw)
    Q, K, V, G, O_, st = (t.double() for t in (q, k, v, d_o, o, s))
    p = torch.exp(torch.bmm(Q, K.transpose(1, 2).contiguous()) * D ** -0.5 - st[..., None])
    p = torch.where(p <= 1e-6, 0.0, p)
    dp = torch.bmm(G, V.transpose(1, 2).contiguous()) * keep / (1 - float(np.float32(0.9)))
    ds = p * (dp - (G * O_).sum(2, keepdim=True))
    ref = torch.bmm(ds.transpose(1, 2).contiguous(), Q) * D ** -0.5
    assert ((dk.double() - ref).norm() / ref.norm()).item() <= 8e-4


def test_f32_forward_extreme_keys(pkg):
    """A key of -inf scores weighs 0 (its bf16 parts are NaN past the first),
    and one near the type's lowest value as well; other rows keep their error."""
    g = torch.Generator().manual_seed(1)
    q = (torch.rand((2, 70, 64), generator=g) + 0.1).cuda()
    k, v = torch.randn((2, 70, 64), generator=g).cuda(), torch.randn((2, 70, 64), generator=g).cuda()
    q[0] = 1.0
    k[:, 5] = float("-inf")
    k[:, 40, 3] = -3.4e38
    o, _ = pkg.sdpa(q, k, v, scale=0.125)
    ref = torch.softmax(q.double().cpu() @ k.double().cpu().transpose(1, 2) * 0.125, -1) @ v.double().cpu()
    assert (o.double().cpu() - ref).abs().max().item() <= 1e-5


# D_qk, D_v, S_kv: up to 8192 keys on the bf16 matrix cores (whole chunks and
# element loads, both dQ paths, keys in parts), past that on the fp32 ones.
INF = [(64, 64, 64), (37, 5, 128), (128, 64, 128), (128, 128, 128), (32, 128, 64), (64, 32, 2048), (64, 64, 8256)]


def _same_class(got, ref, tol):
    """Infinite and NaN where the reference is, the rest within tol."""
    got, fin = got.double().cpu(), torch.isfinite(ref)
    assert torch.equal(got[~fin].nan_to_num(nan=7.0), ref[~fin].nan_to_num(nan=7.0))
    assert (got - ref)[fin].abs().max().item() <= tol * max(1.0, ref[fin].abs().max().item())


@pytest.mark.parametrize("D_qk,D_v,S_kv", INF)
def test_f32_forward_infinite_values(pkg, D_qk, D_v, S_kv):
    """An infinite v makes o infinite in its feature (every weight is > 0), and
    a NaN NaN; other features keep their error."""
    g = torch.Generator().manual_seed(8)
    q, k, v = (torch.randn((2, n, d), generator=g) for n, d in ((33, D_qk), (S_kv, D_qk), (S_kv, D_v)))
    v[0, 5, 3] = v[0, 9, 3] = v[1, S_kv - 1, 0] = float("inf")
    v[0, 6, 4] = float("-inf")
    v[0, 7, 2] = float("nan")
    o, s = pkg.sdpa(*(t.cuda() for t in (q, k, v)), scale=0.1)
    x = q.double() @ k.double().transpose(1, 2) * 0.1
    ref = torch.softmax(x, -1) @ v.double()
    assert torch.isinf(ref[0, :, 3:5]).all() and torch.isnan(ref[0, :, 2]).all() and torch.isfinite(ref[0, :, :2]).all()
    _same_class(o, ref, 1e-5)
    assert (s.double().cpu() - torch.logsumexp(x, -1)).abs().max().item() <= TOL["f32"]["stats"]


@pytest.mark.parametrize("what", ["d_o", "v"])
@pytest.mark.parametrize("D_qk,D_v,S_kv", INF)
def test_f32_backward_infinite_values(pkg, D_qk, D_v, S_kv, what):
    """An infinite dO makes dV infinite in its feature, and dS of its row; an
    infinite v makes dS of its key so; dQ and dK take the infinities whose
    factors have one sign, and NaN of the others.  S_q and S_kv fill whole
    tiles: a row of zeros beside an infinity is NaN in 32-row tiles."""
    g = torch.Generator().manual_seed(9)
    S_q = 64
    q, k, v = (torch.randn((2, n, d), generator=g) for n, d in ((S_q, D_qk), (S_kv, D_qk), (S_kv, D_v)))
    q *= 0.5  # every weight well over 1e-6
    d_o = torch.randn((2, S_q, D_v), generator=g)
    q[..., 0], k[..., 0] = q[..., 0].abs() + 0.1, k[..., 0].abs() + 0.1
    o, s = pkg.sdpa(*(t.cuda() for t in (q, k, v)), scale=0.1)
    o = o.cpu()
    if what == "d_o":
        v[0, :, 1] = v[0, :, 1].abs() + 0.1
        d_o[0, 3, 1] = float("inf")
        o[0, 3, 1] = -1.0  # delta -inf: dS of row 3 is +inf
    else:
        d_o[0, :, 3] = d_o[0, :, 3].abs() + 0.1
        v[0, 5, 3] = float("inf")
    got = pkg.sdpa_grad(*(t.cuda() for t in (q, k, v, o)), s, d_o.cuda(), scale=0.1)
    Q, K, V, G, O_, st = (t.double() for t in (q, k, v, d_o, o, s.cpu()))
    p = torch.exp(Q @ K.transpose(1, 2) * 0.1 - st[..., None])
    assert (p > 2e-6).all()
    ds = p * (G @ V.transpose(1, 2) - (G * O_).sum(2, keepdim=True))
    ref = ds @ K * 0.1, ds.transpose(1, 2) @ Q * 0.1, p.transpose(1, 2) @ G
    if what == "d_o":
        assert torch.isinf(ref[2][0, :, 1]).all() and torch.isinf(ref[1][0]).all() and torch.isinf(ref[0][0, 3, 0])
    else:
        assert torch.isinf(ref[0][0]).all() and torch.isinf(ref[1][0, 5, 0]) and torch.isfinite(ref[2]).all()
    for a, b in zip(got, ref):
        _same_class(a, b, TOL["f32"]["grad"])


@pytest.mark.parametrize("D", [64, 37, 128])
def test_f32_backward_extreme_keys(pkg, D):
    """A key of -inf scores weighs 0 in the gradient too: dK and dV of the
    other keys keep their error, its own are 0, and dQ is NaN (0 times -inf)
    in the one feature that holds the infinity."""
    g = torch.Generator().manual_seed(10)
    q, k, v, d_o = (torch.randn((2, 64, D), generator=g) for _ in range(4))
    q[..., 3] = 1.0
    k[0, 5, 3] = float("-inf")
    o, s = pkg.sdpa(*(t.cuda() for t in (q, k, v)), scale=0.1)
    dq, dk, dv = pkg.sdpa_grad(*(t.cuda() for t in (q, k, v)), o, s, d_o.cuda(), scale=0.1)
    Q, K, V, G, O_, st = (t.double().cpu() for t in (q, k, v, d_o, o, s))
    p = torch.exp(Q @ K.transpose(1, 2) * 0.1 - st[..., None])
    assert (p[0, :, 5] == 0).all() and (p > 2e-6).sum() == p.numel() - 64
    ds = p * (G @ V.transpose(1, 2) - (G * O_).sum(2, keepdim=True))
    _same_class(dv, p.transpose(1, 2) @ G, TOL["f32"]["grad"])
    _same_class(dk, ds.transpose(1, 2) @ Q * 0.1, TOL["f32"]["grad"])
    ref = ds @ K.nan_to_num(neginf=0.0) * 0.1
    ref[0, :, 3] = float("nan")
    _same_class(dq, ref, TOL["f32"]["grad"])


BWD = [
    # dtype, B, S_q, S_kv, D_qk, D_v, causal, dropout; parts of a tile in dQ and, fp32, in dK/dV
    ("f16", 2, 97, 65, 64, 64, False, 0.1, 1),      # every wave one query block, a one-key tile
    ("f16", 2, 129, 129, 40, 24, True, 0.1, 1),     # the diagonal blocks, one-row tiles
    ("f16", 1, 257, 31, 32, 64, False, 0.0, 1),     # one key tile, query blocks more than two rounds
    ("f16", 3, 33, 1001, 64, 32, False, 0.2, 4),    # dQ in parts, ragged
    ("f16", 1, 1, 2049, 64, 64, False, 1.5, 8),     # one query; every element dropped
    ("f16", 2, 160, 160, 128, 128, True, 0.2, 1),   # dS path: sub-tiles that are not stored
    ("f16", 1, 98, 225, 128, 32, False, 0.1, 1),    # dS path, ragged on both sides
    ("f16", 1, 129, 70, 24, 72, False, 1.5, 1),     # dS path, every element dropped
    ("f16", 2, 130, 130, 36, 4, True, 0.1, 1),      # features a multiple of 4 only
    ("f16", 2, 35, 1100, 12, 60, False, 0.2, 4),    # the same, dQ in parts
    ("f32", 2, 33, 129, 64, 64, False, 0.1, 3),     # a one-row query block, a one-key tile
    ("f32", 1, 65, 65, 37, 5, True, 0.1, 1),        # element loads, the diagonal
    ("f32", 1, 33, 1100, 64, 64, False, 0.2, 2),    # dQ in parts, ragged
    ("f32", 2, 700, 66, 20, 36, False, 0.1, 2),     # dK/dV in parts
    ("f32", 1, 513, 513, 64, 64, True, 1.5, 2),     # both, the diagonal, every element dropped
    ("f32", 2, 160, 160, 128, 128, True, 0.2, 1),   # dS path
    ("f32", 1, 31, 257, 128, 32, False, 1.5, 1),    # dS path, every element dropped
    ("f32", 1, 17, 8193, 40, 36, False, 0.1, 1),    # the sequential fp32 sums, undivided
    ("f32", 2, 5, 8200, 64, 64, False, 0.1, 2),     # the same for few queries, dQ in parts
    ("f32", 1, 16, 9001, 37, 5, False, 0.0, 2),     # and with element loads
    ("f32", 1, 33, 8225, 128, 64, False, 0.0, 1),   # the same, dS path
    ("f32", 1, 70, 8193, 5, 64, False, 0.2, 1),     # its dK/dV at D <= 64: element loads, a one-key tile
]


@pytest.mark.parametrize("case", BWD, ids=["-".join(map(str, c)) for c in BWD])
def test_small_backward(pkg, O, case):
    dt, B, S_q, S_kv, D_qk, D_v, causal, p, parts = case
    c = Cfg("small_bwd", dt, B, S_q, S_kv, D_qk, D_v, causal, p, D_qk ** -0.5, 5, 23)
    L = pkg.library()
    dims = (1 if dt == "f16" else 0, B, S_q, S_kv, D_qk, D_v, int(causal))
    ds, full = L.sdpa_hip_bwd_workspace_bytes_ds(*dims), L.sdpa_hip_bwd_workspace_bytes_full(*dims)
    if dt == "f16":
        assert full == ds + (parts * B * S_q * D_qk * 4 if parts > 1 else 0)
    else:
        assert (full > ds) == (parts > 1)
    run_and_check(pkg, O, c, fp32_sum_allowance=True)
    # the gradient of another output (o is not this forward's): delta != 0 also where every element is dropped
    q, k, v, d_o = make_inputs(c)
    o, s = pkg.sdpa(_t(q), _t(k), _t(v), c.seed, c.offset, dropout=0.0, scale=c.scale, causal_mask=causal)
    g = pkg.sdpa_grad(_t(q), _t(k), _t(v), o, s, _t(d_o), c.seed, c.offset, dropout=p, scale=c.scale,
                      causal_mask=causal)
    ref = O.sdpa_bwd_gate(q, k, v, _np(o), _np(s), d_o, **oracle_kw(c))
    for a, b in zip(g, ref):
        assert maxabs(_np(a), b) <= TOL[dt]["grad"] * max(1.0, float(np.abs(b.astype(np.float64)).max()))
