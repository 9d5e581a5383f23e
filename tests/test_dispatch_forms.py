"""Which calls the one-launch kernels take: only what they can read and write within the tensors given.  Everything
else goes the general way, where torch refuses what does not fit."""
from dataclasses import replace

import pytest
import torch

from kvq.decode import exact_rows_cache
from kvq.state import PackedState, _append_takes


def _state(cap=12, n=5, dtype=torch.float32):
    k, v = torch.zeros(2, 3, cap, 128, dtype=dtype), torch.zeros(2, 3, cap, 128, dtype=dtype)
    st = PackedState()
    st.cache, st.n, st.n0 = exact_rows_cache(k, v, n, torch.full((cap,), 1 << 62)), n, n
    return st


def test_rows_that_fit_are_taken():
    c = _state().cache
    x = torch.ones(2, 3, 4, 128)
    assert _append_takes(c, x, x)
    assert _append_takes(c, x.transpose(1, 2).contiguous().transpose(1, 2), x)          # token-major


@pytest.mark.parametrize("form", ["dtype", "heads", "narrow", "misaligned", "grad", "channels"])
def test_other_rows_are_left_to_torch(form):
    c = _state().cache
    x = torch.ones(2, 3, 4, 128)
    y = {"dtype": x.half(), "heads": x[:, :1], "narrow": x[..., :64], "grad": x.clone().requires_grad_(),
         "misaligned": torch.ones(2 * 3 * 4 * 128 + 1)[1:].view(2, 3, 4, 128),
         "channels": torch.ones(2, 3, 128, 4).transpose(2, 3)}[form]
    assert not _append_takes(c, y, x) and not _append_takes(c, x, y)


@pytest.mark.parametrize("positions", [lambda p: p[:6], lambda p: p.to(torch.int32), lambda p: p.repeat(2)[::2],
                                       lambda p: p.view(3, 4), lambda p: p.to("meta")])
def test_positions_that_the_kernel_could_not_write(positions):
    """Positions shorter than the row buffers, of another type, layout or device."""
    c = _state().cache
    x = torch.ones(2, 3, 4, 128)
    assert not _append_takes(replace(c, exact_pos=positions(c.exact_pos)), x, x)


def test_value_rows_that_hold_fewer():
    c = _state().cache
    x = torch.ones(2, 3, 4, 128)
    assert not _append_takes(replace(c, v_exact=c.v_exact[:, :, :6].contiguous()), x, x)


def test_positions_too_short_are_refused():
    """As before the one-launch copy: the step after the positions' last raises instead of writing past them."""
    st = _state()
    st.cache = replace(st.cache, exact_pos=st.cache.exact_pos[:7].clone())
    x = torch.ones(2, 3, 2, 128)
    st.append(x, x, torch.tensor([5, 6]))
    assert st.cache.exact_pos.tolist() == [1 << 62] * 5 + [5, 6] and st.cache.n_exact == 7
    with pytest.raises(RuntimeError):
        st.append(x, x, torch.tensor([7, 8]))


def test_contexts_of_two_devices():
    """Keys and values of one device only: the kernels read both sides with one device's stream."""
    from kvq import dct, decode
    x = torch.zeros(1, 2, 96, 128)
    assert decode._compress_takes(x, x, 64, 64, 128) and dct._compress_takes(x, x)
    assert not decode._compress_takes(x, x.to("meta"), 64, 64, 128) and not dct._compress_takes(x, x.to("meta"))
