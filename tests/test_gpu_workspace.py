"""The decodes write every workspace float they read: a workspace full of NaN gives the bits a zeroed one does.
(The Python entry points hand the library an uninitialised workspace.)  Row counts that do not fill
the kernels' power-of-two row tile, splits of one chunk, exact rows in all their placements."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(g, *shape, dtype=torch.bfloat16):
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def _same(step, need):
    a = step(torch.zeros((need,), device="cuda"))
    b = step(torch.full((need,), float("nan"), device="cuda"))
    assert torch.isfinite(a.float()).all()
    assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,Hkv,rep,Tq,T,window", [
    (1, 1, 1, 1, 33, 1), (1, 3, 3, 1, 200, 40), (2, 4, 3, 2, 1000, 96), (1, 2, 1, 5, 4000, 700),
    (1, 2, 7, 1, 3000, 2000), (16, 8, 4, 1, 2176, 128),       # 16 x 8: one round of packed blocks by class
    (12, 8, 4, 1, 4096, 60),                                  # every slot taken: the window in the packed blocks
])
def test_kivi_decode_any_workspace(dtype, B, Hkv, rep, Tq, T, window):
    import kvq
    g = torch.Generator(device="cuda").manual_seed(T)
    c = kvq.PackedKIVICache.from_context(_rows(g, B, Hkv, T, 128, dtype=dtype), _rows(g, B, Hkv, T, 128, dtype=dtype),
                                         window=window, group_k=64, group_v=64)
    q = _rows(g, B, Hkv * rep, Tq, 128, dtype=dtype)
    size = (B, Hkv * rep, Hkv, Tq, 128, c.n_q, c.n_exact, 64, 64)
    _same(lambda ws: kvq.kivi_decode(q, 0.1, c, workspace=ws), kvq.workspace_floats(*size))

    def scored(ws):
        s = torch.zeros((B, Hkv, c.n_q), device="cuda")
        out = kvq.kivi_decode(q, 0.1, c, workspace=ws, scores=s, score_weight=0.25)
        return torch.cat([out.float().reshape(-1), s.reshape(-1)])
    _same(scored, kvq.score_workspace_floats(*size))
    _same(scored, kvq.workspace_floats(*size))                # the key-rereading score pass


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,Hkv,rep,Tq,T,window", [(1, 1, 3, 1, 150, 10), (2, 3, 1, 6, 1500, 0), (8, 8, 4, 1, 2048, 64),
                                                   (1, 8, 8, 1, 9000, 1500)])
def test_coded_decodes_any_workspace(dtype, B, Hkv, rep, Tq, T, window):
    import kvq
    g = torch.Generator(device="cuda").manual_seed(T + rep)
    K, V = _rows(g, B, Hkv, T, 128, dtype=dtype), _rows(g, B, Hkv, T, 128, dtype=dtype)
    q, Hq = _rows(g, B, Hkv * rep, Tq, 128, dtype=dtype), Hkv * rep
    nb = (T - window) // 64
    w = torch.tensor([2, 4, 8], device="cuda", dtype=torch.int8)[torch.randint(0, 3, (B, Hkv, nb), generator=g, device="cuda")]
    c = kvq.MixedKIVICache.from_context(K, V, w, window=window)
    _same(lambda ws: kvq.mixed_decode(q, 0.1, c, workspace=ws), kvq.mixed_workspace_floats(B, Hq, Hkv, Tq, 128, c.nb, c.n_exact))
    d = kvq.DctCache.from_context(K, V, window=window)
    _same(lambda ws: kvq.dct_decode(q, 0.1, d, workspace=ws), kvq.dct_workspace_floats(B, Hq, Hkv, Tq, 128, d.T, d.n_exact))
    order = torch.rand((B, Hkv, T - window), generator=g, device="cuda").argsort(-1).to(torch.int32)
    n = T - window
    s = kvq.StrataCache.from_context(K, V, window=window, assign=[(8, order[..., :n // 10].contiguous()),
                                                                  (4, order[..., n // 10:n // 2].contiguous()),
                                                                  (2, order[..., n // 2:].contiguous())])
    _same(lambda ws: kvq.strata_decode(q, 0.1, s, workspace=ws),
          kvq.strata_workspace_floats(B, Hq, Hkv, Tq, 128, s.n_exact, [t.n for t in s.tiers], [t.bits for t in s.tiers]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,Hkv,rep,T,last", [(1, 8, 4, 1384, 384), (1, 8, 1, 4352, 384), (2, 3, 2, 700, 200)])
def test_kivi_decode_workspace_sized_once(dtype, B, Hkv, rep, T, last):
    """A workspace of the last step's size serves every step before it, and one that holds the packed splits'
    partials alone serves them all: the window then goes where it needs no partials of its own.  The
    placements agree to rounding (fp32 sums, then one rounding to the output type)."""
    import kvq
    g = torch.Generator(device="cuda").manual_seed(T)
    c = kvq.PackedKIVICache.from_context(_rows(g, B, Hkv, T, 128, dtype=dtype), _rows(g, B, Hkv, T, 128, dtype=dtype),
                                         window=last, group_k=64, group_v=64)
    q = _rows(g, B, Hkv * rep, 1, 128, dtype=dtype)
    size = lambda n: (B, Hkv * rep, Hkv, 1, 128, c.n_q, n, 64, 64)
    end = torch.empty((kvq.workspace_floats(*size(last)),), device="cuda")
    end_s = torch.empty((kvq.score_workspace_floats(*size(last)),), device="cuda")
    few = torch.empty((kvq.workspace_floats(*size(0)),), device="cuda")
    few_s = torch.empty((kvq.score_workspace_floats(*size(0)),), device="cuda")
    atol = 1e-5 if dtype == torch.float32 else 2 ** -8
    for n in sorted({1, 16, 17, 40, 128, last - 1, last}):
        c.n_exact = n
        want, score = kvq.kivi_decode(q, 0.1, c), torch.zeros((B, Hkv, c.n_q), device="cuda")
        assert torch.equal(kvq.kivi_decode(q, 0.1, c, workspace=end), want)
        torch.testing.assert_close(kvq.kivi_decode(q, 0.1, c, workspace=few), want, rtol=0, atol=atol)
        assert torch.equal(kvq.kivi_decode(q, 0.1, c, scores=score), want)
        for ws in (end, end_s, few, few_s):
            s = torch.zeros_like(score)
            torch.testing.assert_close(kvq.kivi_decode(q, 0.1, c, workspace=ws, scores=s), want, rtol=0, atol=atol)
            torch.testing.assert_close(s, score, rtol=1e-5, atol=1e-9)
