"""PackedKIVICache.from_context through kvq_kivi_compress (two launches that write the whole cache) against the
general path (quantise, pack, tile and copy in separate steps, itself held to the oracle by
tests/test_gpu_kivi.py and tests/test_gpu_decode.py): every buffer bit for bit, padding included."""
import pytest
import torch

pytestmark = pytest.mark.gpu

FIELDS = ("kc", "k_lo", "k_sc", "vc", "vmeta", "k_exact", "v_exact")


def _both(K, V, monkeypatch, **kw):
    import kvq
    from kvq import decode
    calls = []
    real = decode._lib.call
    monkeypatch.setattr(decode._lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    got = kvq.PackedKIVICache.from_context(K, V, **kw)
    assert "kvq_kivi_compress" in calls
    monkeypatch.setattr(decode, "_compress_takes", lambda *a: False)
    want = kvq.PackedKIVICache.from_context(K, V, **kw)
    assert calls.count("kvq_kivi_compress") == 1
    monkeypatch.undo()
    for f in FIELDS:
        a, b = getattr(got, f), getattr(want, f)
        assert a.shape == b.shape and a.dtype == b.dtype, f
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), f
    assert (got.n_q, got.n_exact, got.cap_t, got.cap_e, got.ring, got.next_pos) == \
        (want.n_q, want.n_exact, want.cap_t, want.cap_e, want.ring, want.next_pos)


def _rows(B, H, T, dtype, seed, token_major=False):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((B, T, H, 128) if token_major else (B, H, T, 128), generator=g) * 3
    x[..., 5] *= 40.0
    x = x.to(dtype).cuda()
    return x.transpose(1, 2) if token_major else x


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("group_k,group_v", [(32, 128), (64, 64), (128, 32)])
@pytest.mark.parametrize("T,window,ring,extra", [(1, 0, False, 0), (31, 31, False, 3), (129, 128, True, 0),
                                                 (400, 133, True, 70), (1027, 131, False, 5), (2081, 0, False, 300)])
def test_compress_equals_general_path(dtype, group_k, group_v, T, window, ring, extra, monkeypatch):
    K, V = _rows(2, 3, T, dtype, T), _rows(2, 3, T, dtype, T + 1)
    kw = dict(extra_tokens=extra) if ring else dict(extra_tokens=extra, extra_exact=extra)
    if T == 1:                              # a single row's token stride is torch's to choose
        K, V = (torch.empty_strided((2, 3, 1, 128), (384, 128, 128, 1), dtype=dtype, device="cuda").copy_(x) for x in (K, V))
    _both(K, V, monkeypatch, window=window, group_k=group_k, group_v=group_v, ring=ring, **kw)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_compress_views(dtype, monkeypatch):
    K, V = _rows(2, 4, 333, dtype, 1, token_major=True), _rows(2, 4, 350, dtype, 2)[:, :, 9:342]
    _both(K, V, monkeypatch, window=77, group_k=64, group_v=64)
    _both(K[:, 1:3], V[:, :2], monkeypatch, window=128, group_k=32, group_v=32, ring=True, extra_tokens=64)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_compress_extreme_values(dtype, monkeypatch):
    """Constant groups, codes at half-integers, subnormals, values beyond fp16's range, infinities, NaN."""
    K, V = _rows(1, 2, 260, dtype, 4), _rows(1, 2, 260, dtype, 5)
    for x in (K, V):
        x[:, :, 0:64, 0:32] = 1.5
        x[:, :, 64:128, 32:64] = (torch.arange(32, device="cuda") % 31 / 2.0).to(dtype)
        x[:, :, 128:140, 64:80] = 6e-8
        x[:, :, 140:150, 80:90] = 6e4
        if dtype != torch.float16:
            x[:, :, 150, 90:95] = 3e38
        x[:, :, 200, 3], x[:, :, 201, 4], x[:, :, 202, 6] = float("inf"), float("-inf"), float("nan")
    _both(K, V, monkeypatch, window=20, group_k=32, group_v=32)
    _both(K, V, monkeypatch, window=64, group_k=64, group_v=128, ring=True)


def test_other_forms_take_the_general_path():
    """Forms kvq_kivi_compress does not take: other groups, an exact dtype of its own, misaligned and
    repeated rows."""
    from kvq import decode
    x = _rows(1, 2, 96, torch.bfloat16, 6)
    off = torch.empty(2 * 96 * 128 + 1, dtype=torch.bfloat16, device="cuda")[1:].view(1, 2, 96, 128)
    takes = decode._compress_takes
    assert takes(x, x, 64, 64, 64)
    assert not takes(x, x, 16, 64, 64) and not takes(x, x, 64, 16, 64) and not takes(x, x.float(), 64, 64, 64)
    assert not takes(off, x, 64, 64, 64) and not takes(x, x[:, :, :1].expand(1, 2, 96, 128), 64, 64, 64)


# ---- DctCache: the matrix-core encoder, and kvq_dct_compress over views ------------------------------

DCT_FIELDS = ("kc", "ks", "vc", "vs", "k_exact", "v_exact")


def _plain(x, for_values):
    """dct_encode of x through the kernel with one thread per channel, which sums in the fixed order: the rows
    widened to float32 (exact) are the same sums."""
    import kvq
    return kvq.dct_encode(x.float(), for_values)


def _same(a, b, what):
    assert a.shape == b.shape and a.dtype == b.dtype, what
    assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), what


def _dct_rows(kind, dtype, shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(shape, generator=g, device="cuda")
    if kind == "walk":                                   # slow channels: one large coefficient, the rest near zero
        x = x.cumsum(2) * 0.05 + 3.0
    elif kind == "wide":                                 # magnitudes over decades, zeros among them
        x = x * 10.0 ** torch.randint(-6, 4, (*shape[:3], 1), generator=g, device="cuda")
        x = x * (torch.rand(shape, generator=g, device="cuda") > 0.3)
    elif kind == "grid":                                 # few values: coefficients and quotients that tie
        x = torch.randint(-2, 3, shape, generator=g, device="cuda").float() * 0.5
    elif kind == "tiny":                                 # subnormals of both types, scales at the floor
        x = x * 1e-6
    elif kind == "huge":
        x = x * (3e4 if dtype == torch.float16 else 1e36)
    return x.to(dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind", ["noise", "walk", "wide", "grid", "tiny", "huge"])
def test_dct_encode_matrix_cores_equal_fixed_order(dtype, kind):
    import kvq
    x = _dct_rows(kind, dtype, (2, 3, 4096, 128), 7)
    for for_values in (False, True):
        for a, b, f in zip(kvq.dct_encode(x, for_values), _plain(x, for_values), ("codes", "scales")):
            _same(a, b, f)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_dct_encode_non_finite(dtype):
    import kvq
    x = _dct_rows("noise", dtype, (1, 2, 192, 128), 8)
    x[0, 0, 5, 3], x[0, 0, 70, 4], x[0, 1, 130, 9], x[0, 1, 60, 127] = float("inf"), float("-inf"), float("nan"), float("nan")
    x[0, 0, 128:192, 20] = 0
    for for_values in (False, True):
        for a, b, f in zip(kvq.dct_encode(x, for_values), _plain(x, for_values), ("codes", "scales")):
            _same(a, b, f)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T,window,extra", [(1, 0, 0), (63, 0, 2), (64, 0, 0), (200, 9, 5), (4133, 64, 0)])
def test_dct_compress_equals_general_path(dtype, T, window, extra, monkeypatch):
    import kvq
    from kvq import dct
    base = _dct_rows("walk", dtype, (2, T + 3, 3, 128), T)
    for K, V in ((base[:, :T].transpose(1, 2), base[:, 3:].transpose(1, 2)),            # token-major views
                 (base.transpose(1, 2).contiguous()[:, :, 1:T + 1], base[:, :T].transpose(1, 2).contiguous())):
        assert T == 1 or dct._compress_takes(K, V)
        got = kvq.DctCache.from_context(K, V, window=window, extra_exact=extra)
        monkeypatch.setattr(dct, "_compress_takes", lambda *a: False)
        want = kvq.DctCache.from_context(K.float(), V.float(), window=window, extra_exact=extra)
        monkeypatch.undo()
        assert (got.T, got.n_exact) == (want.T, want.n_exact)
        for f in DCT_FIELDS:
            w = getattr(want, f)
            _same(getattr(got, f), w.to(dtype) if f.endswith("exact") else w, f)
