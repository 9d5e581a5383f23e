"""Token steps whose positions go with the launches by value (kvq_exact_append, kvq_kivi_decode_at) against
the same steps with positions on the device and rows copied by torch: equal bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(g, *shape, dtype=torch.float16):
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,Hkv,rep,T,window,extra,steps", [
    (1, 2, 4, 700, 64, 40, (1, 2, 1, 9)),             # window in the packed splits; 9 > 8 tokens: pieces, positions uploaded
    (2, 3, 1, 300, 96, 80, (8, 1, 3)),
    (1, 1, 8, 2000, 900, 8, (1, 1)),                  # window in the merge
    (1, 1, 3, 1500, 1300, 8, (2, 2)),                 # window in exact-row blocks of their own
])
def test_positions_by_value(dtype, B, Hkv, rep, T, window, extra, steps, monkeypatch):
    import kvq
    from kvq import state
    g = torch.Generator(device="cuda").manual_seed(T)
    K, V = _rows(g, B, Hkv, T, 128, dtype=dtype), _rows(g, B, Hkv, T, 128, dtype=dtype)
    a, b = (kvq.KIVIState(K, V, window=window, group_k=32, group_v=64, extra=extra) for _ in (0, 1))
    pos = T
    for t in steps:
        # token-major projections, viewed; the appended rows past the query's position must stay hidden
        k, v = (_rows(g, B, t, Hkv, 128, dtype=dtype).transpose(1, 2) for _ in (0, 1))
        q = _rows(g, B, Hkv * rep, t, 128, dtype=dtype)
        at = torch.arange(pos, pos + t)
        a.append(k, v, at)
        with monkeypatch.context() as m:
            m.setattr(state, "_append_takes", lambda *x: False)
            b.append(k, v, at.cuda())
        for f in ("k_exact", "v_exact"):
            x, y = getattr(a.cache, f), getattr(b.cache, f)
            assert torch.equal(x[:, :, :a.cache.n_exact], y[:, :, :a.cache.n_exact])
        assert torch.equal(a.cache.exact_pos, b.cache.exact_pos) and (a.n, a.cache.n_exact) == (b.n, b.cache.n_exact)
        for shift in (0, -1, 1):                      # earlier positions hide appended rows
            x, y = a.attend(q, 0.1, at + shift), b.attend(q, 0.1, (at + shift).cuda())
            assert torch.isfinite(x.float()).all() and torch.equal(x, y)
        pos += t
    assert torch.equal(a.attend(q, 0.1, list(range(pos - t, pos))), x if t == 0 else a.attend(q, 0.1, at.cuda()))


def test_append_other_forms():
    """Rows of another dtype, one position for several rows, a full buffer."""
    import kvq
    g = torch.Generator(device="cuda").manual_seed(1)
    st = kvq.KIVIState(_rows(g, 1, 2, 100, 128), _rows(g, 1, 2, 100, 128), window=40, group_k=32, group_v=32, extra=6)
    k, v = _rows(g, 1, 2, 2, 128, dtype=torch.float32), _rows(g, 1, 2, 2, 128, dtype=torch.float32)
    st.append(k, v, torch.tensor([100, 101]))
    st.append(k.half(), v.half(), torch.tensor([7]))
    assert st.cache.exact_pos[40:44].tolist() == [100, 101, 7, 7]
    assert torch.equal(st.cache.k_exact[:, :, 40:42], k.half()) and torch.equal(st.cache.v_exact[:, :, 42:44], v.half())
    st.append(k[:, :, :1].half(), v[:, :, :1].half(), 103)
    assert st.cache.exact_pos[44].item() == 103
    with pytest.raises(RuntimeError):
        st.append(k.half(), v.half(), torch.tensor([104, 105]))
    q = _rows(g, 1, 4, 2, 128)
    with pytest.raises(ValueError):
        st.attend(q, 0.1, torch.tensor([1]))
    strided = torch.tensor([103, 0, 104, 0], device="cuda")[::2]
    assert torch.equal(st.attend(q, 0.1, strided), st.attend(q, 0.1, torch.tensor([103, 104])))


def test_step_in_a_graph():
    """A token step captured with host positions replays to the eager result."""
    import kvq
    g = torch.Generator(device="cuda").manual_seed(2)
    st = kvq.KIVIState(_rows(g, 2, 2, 500, 128), _rows(g, 2, 2, 500, 128), window=64, group_k=32, group_v=32, extra=4)
    k, v, q = _rows(g, 2, 2, 1, 128), _rows(g, 2, 2, 1, 128), _rows(g, 2, 8, 1, 128)
    n, e = st.n, st.cache.n_exact

    def step():
        st.n, st.cache.n_exact = n, e
        st.append(k, v, torch.tensor([500]))
        return st.attend(q, 0.1, torch.tensor([500]))
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        step()
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for i in range(4):
        for x in (k, v, q):
            x.copy_(_rows(g, *x.shape))
        graph.replay()
        got = out.clone()
        torch.cuda.synchronize()
        assert torch.equal(got, step())


@pytest.mark.parametrize("B,Hkv,rep,Tq,T,window", [
    (1, 1, 1, 1, 40, 8), (1, 2, 1, 1, 700, 15), (1, 3, 4, 2, 1200, 17), (2, 4, 4, 2, 3001, 96),    # exact-row blocks beside
    (1, 8, 1, 1, 4096, 128), (1, 5, 3, 1, 3000, 250),                                             # up to 48 partials a row
    (12, 8, 4, 1, 4096, 60), (14, 8, 2, 1, 3000, 100),                                            # in the packed blocks
    (1, 1, 2, 1, 5000, 800),                                                                      # in the merge
])
def test_window_placements_match_dense_attention(B, Hkv, rep, Tq, T, window):
    """fp32 steps over packed and exact rows, appended ones causal, wherever the plan attends the window.  The bar is that of
    the packed codes; single exact rows are held by test_every_exact_row_counts_once."""
    import kvq
    g = torch.Generator(device="cuda").manual_seed(T + window)
    f32 = torch.float32
    st = kvq.KIVIState(_rows(g, B, Hkv, T, 128, dtype=f32), _rows(g, B, Hkv, T, 128, dtype=f32), window=window, group_k=32,
                       group_v=32, extra=Tq)
    st.append(_rows(g, B, Hkv, Tq, 128, dtype=f32), _rows(g, B, Hkv, Tq, 128, dtype=f32), torch.arange(T, T + Tq))
    q = _rows(g, B, Hkv * rep, Tq, 128, dtype=f32)
    at = torch.arange(T, T + Tq)
    got, want = st.attend(q, 128 ** -0.5, at), st.reference_attend(q, 128 ** -0.5, at)
    assert float((got - want).abs().max()) <= 2e-3                   # the fp32 bar of every decode


@pytest.mark.parametrize("B,Hkv,rep,Tq,T,n_exact", [
    (1, 8, 1, 1, 4096, 16), (1, 8, 1, 1, 4096, 17), (1, 8, 1, 1, 4096, 128), (1, 8, 1, 1, 4096, 129),    # 16-row blocks beside
    (1, 8, 1, 1, 4240, 272), (1, 8, 1, 1, 4240, 273), (1, 8, 1, 1, 4480, 512), (1, 8, 1, 1, 4481, 513),  # 16 -> 32 rows .. 64
    (2, 3, 4, 2, 900, 33), (1, 5, 3, 1, 700, 250), (1, 1, 8, 1, 300, 31),
    (12, 8, 4, 1, 4096, 60), (14, 8, 2, 1, 3000, 101),                                                   # in the packed blocks
    (16, 8, 4, 1, 2176, 129),                                                                            # beside a class plan
    (1, 1, 2, 1, 5000, 800), (1, 2, 1, 1, 3000, 1300),                                                   # merge; blocks of their own
])
def test_every_exact_row_counts_once(B, Hkv, rep, Tq, T, n_exact):
    """Queries that lean on the exact rows alone (their keys point along the queries, the packed ones away), each
    with its own value: a row lost, counted twice or read from elsewhere moves the output by its share of
    the mass times its distance from the mean, several times the bar.  Against float64 attention over
    the exact rows; the packed rows' mass is below n_q e^-24."""
    import kvq
    g = torch.Generator(device="cuda").manual_seed(n_exact)
    f32 = torch.float32
    u = torch.full((128,), 128 ** -0.5, device="cuda")
    K = 0.02 * _rows(g, B, Hkv, T, 128, dtype=f32) - 12.0 * u
    V = _rows(g, B, Hkv, T, 128, dtype=f32)
    W = n_exact - Tq
    K[:, :, T - W:] += 24.0 * u
    st = kvq.KIVIState(K, V, window=W, group_k=32, group_v=32, extra=Tq)
    k1, v1 = 0.02 * _rows(g, B, Hkv, Tq, 128, dtype=f32) + 12.0 * u, _rows(g, B, Hkv, Tq, 128, dtype=f32)
    at = torch.arange(T, T + Tq)
    st.append(k1, v1, at)
    assert st.cache.n_exact == n_exact
    q = 0.02 * _rows(g, B, Hkv * rep, Tq, 128, dtype=f32) + 1.0 * u
    got = st.attend(q, 1.0, at).transpose(1, 2).double()                                       # (B, Hq, Tq, d)
    ke, ve = (torch.cat(x, 2).double().repeat_interleave(rep, 1) for x in ((K[:, :, T - W:], k1), (V[:, :, T - W:], v1)))
    s = q.double() @ ke.transpose(-1, -2).contiguous()
    hidden = torch.arange(n_exact, device="cuda")[None, :] > W + torch.arange(Tq, device="cuda")[:, None]
    p = s.masked_fill(hidden, float("-inf")).softmax(-1)
    want = p @ ve
    # what the least of the visible rows moves: p_i |v_i - out| in the channel where it shows most
    moved = (p[..., None] * (ve[:, :, None] - want[:, :, :, None]).abs()).amax(-1)
    least = float(moved.masked_fill(hidden, float("inf")).min())
    # the kernel's own error: logits near 12 to 2^-20, sums of at most 1300 products to 1300 2^-24 of their mean size
    err = float((got - want).abs().max())
    print(f"n_exact {n_exact}: err {err:.2e}, least row {least:.2e}", flush=True)
    assert err <= 0.1 * least


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T,n_exact", [(700, 1), (700, 17), (700, 30), (700, 33), (5000, 90), (1400, 1300)])
def test_infinite_value_of_an_exact_row(T, n_exact, dtype):
    """An infinity in a visible exact row's value is its channel's output, and no other channel's: lanes that hold no row
    of a block's last ones, and a merge's slots that hold no partial, must not multiply it by their weight of zero."""
    import kvq
    g = torch.Generator(device="cuda").manual_seed(n_exact)
    for row in {0, n_exact // 2, n_exact - 1}:
        K, V = _rows(g, 1, 2, T, 128, dtype=dtype), _rows(g, 1, 2, T, 128, dtype=dtype)
        V[:, :, T - n_exact + row, 7] = float("inf")
        c = kvq.PackedKIVICache.from_context(K, V, window=n_exact, group_k=32, group_v=32)
        q = _rows(g, 1, 4, 1, 128, dtype=dtype)
        few = torch.empty((kvq.workspace_floats(1, 4, 2, 1, 128, c.n_q, 0, 32, 32),), device="cuda")
        for ws in (None, few)[:1 if n_exact > 1024 else 2]:              # beside the packed blocks, and inside them
            out = kvq.kivi_decode(q, 0.1, c, workspace=ws)
            assert torch.isposinf(out[..., 7]).all() and torch.isfinite(out[..., :7]).all() and torch.isfinite(out[..., 8:]).all()
