"""dK and dV leave the dK/dV kernel in 16-byte stores of whole rows where their pointers and strides are multiples of eight
elements, and in 8-byte ones where they are multiples of four: the same bits at the same places, and nothing
written between them."""

import pytest
import torch

from tests.test_attention_direct_gpu import _paged_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,hkv", [(128, 1), (128, 3), (64, 2)])
@pytest.mark.parametrize("n_keys", [256, 200])
def test_wide_and_narrow_stores_write_the_same(gpu, d, hkv, n_keys):
    from dcp_amd.flash_attn_interface import _flash_attn_varlen_backward, _flash_attn_varlen_forward

    bs, hq = 128, 2 * hkv
    rows = [(100, 2, [[[0] * 100, list(range(1, 101))]]), (bs, 2, [[[0] * bs, [n_keys] * bs]])]
    pr = _paged_rows(gpu, rows, bs, hq, hkv, d, seed=d + hkv)
    pr["cu_kv"] = torch.tensor([0, n_keys, 2 * n_keys], dtype=torch.int32, device=gpu)
    k, v = pr["kv"][:, :, 0], pr["kv"][:, :, 1]
    out, lse = torch.empty_like(pr["q"]), torch.empty((hq, len(rows), bs), device=gpu)
    tables = dict(attn_range=pr["rng"], q_block_table=pr["slots"], kv_block_table=pr["kv_table"], out_block_table=pr["slots"])
    _flash_attn_varlen_forward(pr["q"], k, v, pr["cu_q"], pr["cu_kv"], pr["total_q"], bs, 2 * bs, 0.0, d ** -0.5, causal=False,
                               window_size_left=-1, window_size_right=-1, softcap=0.0, alibi_slopes=None,
                               return_softmax=False, out_=out, lse_=lse, **tables)

    def backward(offset, extra):  # dK and dV `offset` elements into rows `extra` elements longer than they are
        shape = (pr["n_dkv"], bs, hkv * d + extra)
        buffers = [torch.full((shape[0] * shape[1] * shape[2] + 8,), 7.0, dtype=torch.bfloat16, device=gpu) for _ in range(2)]
        rows_of = [b[offset : offset + shape[0] * shape[1] * shape[2]].view(shape) for b in buffers]
        dk, dv = (r[:, :, : hkv * d].unflatten(2, (hkv, d)) for r in rows_of)
        _flash_attn_varlen_backward(pr["dout"], pr["q"], k, v, out, lse, torch.empty_like(out), dk, dv, pr["cu_q"], pr["cu_kv"],
                                    pr["total_q"], 2 * n_keys, bs, 2 * bs, 0.0, d ** -0.5, False, -1, -1, 0.0, None, False,
                                    dq_block_table=pr["slots"], dkv_block_table=pr["dkv_table"], **tables)
        for r in rows_of:
            assert (r[:, :, hkv * d :] == 7.0).all(), "written between the rows"
        assert all((b[:offset] == 7.0).all() and (b[offset + shape[0] * shape[1] * shape[2] :] == 7.0).all() for b in buffers)
        return dk.contiguous().view(torch.int16), dv.contiguous().view(torch.int16)

    wide = backward(0, 0)
    assert (wide[0] != torch.tensor(7.0, dtype=torch.bfloat16).view(torch.int16).item()).any()
    for offset, extra in ((4, 0), (0, 4), (4, 12), (0, 8)):
        assert all(torch.equal(a, b) for a, b in zip(wide, backward(offset, extra))), (offset, extra)
