"""A NaN among the inputs comes out as NaN wherever plain arithmetic has one, and nowhere else, whether the keys of the
problem are split over workgroups or not."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _plant(what, q, k, v):
    """-> which elements of O are NaN."""
    bad = torch.zeros(q.shape, dtype=torch.bool)
    if what == "query":                 # every score of one row
        q[0, 0, -1] = float("nan")
        bad[0, 0, -1] = True
    elif what == "keys":                # every score of one head
        k[0, -1] = float("nan")
        bad[0, -1] = True
    elif what == "one key":             # one score of every row of a head
        k[0, 0, k.shape[2] // 3, 1] = float("nan")
        bad[0, 0] = True
    else:                               # one column of O
        v[0, 0, -1, 5] = float("nan")
        bad[0, 0, :, 5] = True
    return bad


@pytest.mark.parametrize("what", ["query", "keys", "one key", "value"])
@pytest.mark.parametrize("H,Sq,Sk,D", [
    (2, 1, 2048, 64), (2, 1, 4097, 128), (2, 16, 1000, 128), (2, 600, 1100, 64), (2, 4, 2048, 264), (2, 70, 4096, 512),   # keys split
    (2, 40, 64, 64), (2, 600, 200, 128), (2, 64, 200, 264),      # one workgroup walks all keys: its wavefronts share them, or D > 128
    (80, 100, 200, 64), (80, 100, 1100, 128)])                   # 128-query workgroups of one and of two key groups
def test_nan_stays_nan(what, H, Sq, Sk, D):
    from flame_amd import capi
    print(f"[nan] {what} {H=} {Sq=} {Sk=} {D=}", flush=True)
    g = torch.Generator().manual_seed(Sq + Sk + D)
    q, k, v = (torch.randn((1, H, n, D), generator=g).to(torch.bfloat16) for n in (Sq, Sk, Sk))
    bad = _plant(what, q, k, v)
    sc = D ** -0.5
    want = torch.softmax(q.double() @ k.double().transpose(-1, -2) * sc, dim=-1) @ v.double()
    assert torch.equal(torch.isnan(want), bad)
    dq, dk, dv = (t.cuda() for t in (q, k, v))
    room = capi.attn_fwd(dq, dk, dv, sc)
    none = capi.attn_fwd(dq, dk, dv, sc, workspace=torch.empty(16, dtype=torch.uint8, device="cuda"))
    for name, (o, lse) in (("as the call allocates", room), ("no room for a split", none)):
        o = o.cpu()
        assert torch.equal(torch.isnan(o), bad), name
        assert torch.allclose(o.double()[~bad], want[~bad], atol=2e-2, rtol=1e-2), name
    # a row whose scores hold a NaN has no finite log-sum-exp, split or not
    rows = room[1].cpu(), none[1].cpu()
    assert torch.equal(torch.isfinite(rows[0]), torch.isfinite(rows[1]))
    assert torch.equal(torch.isfinite(rows[0]), torch.ones_like(rows[0], dtype=torch.bool) if what == "value" else ~bad.any(-1).view(rows[0].shape))


@pytest.mark.parametrize("what", ["query", "keys", "one key", "value"])
def test_nan_stays_nan_materialised(what):
    from flame_amd import capi
    print(f"[nan] materialised, {what}", flush=True)
    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn((1, 2, n, 20), generator=g).to(torch.bfloat16) for n in (70, 300, 300))
    bad = _plant(what, q, k, v)
    o, lse = (t.cpu() for t in capi.attn_fwd_materialised(q.cuda(), k.cuda(), v.cuda(), 0.2))
    assert torch.equal(torch.isnan(o), bad)
    want = torch.softmax(q.double() @ k.double().transpose(-1, -2) * 0.2, dim=-1) @ v.double()
    assert torch.allclose(o.double()[~bad], want[~bad], atol=2e-2, rtol=1e-2)
    assert torch.equal(torch.isfinite(lse), torch.ones_like(lse, dtype=torch.bool) if what == "value" else ~bad.any(-1).view(lse.shape))
