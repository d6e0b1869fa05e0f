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


@pytest.mark.parametrize("mode", [0, 2], ids=["recomputing", "through_ds"])
@pytest.mark.parametrize("d,hkv", [(128, 2), (64, 3)])
@pytest.mark.parametrize("n_keys", [256, 200])
def test_groups_of_a_launch_write_the_same(gpu, mode, d, hkv, n_keys):
    """Groups of rows whose dK and dV go to the caller's unpadded tensors, whole blocks and partly filled ones, and one
    whose go to a slot: whichever of the four pointers and strides makes the stores narrow."""
    from dcp_amd import _lib
    from dcp_amd.flash_attn_interface import _flash_attn_varlen_backward, _flash_attn_varlen_forward

    bs, hq, width = 128, 2 * hkv, hkv * d
    rows = [(100, 2, [[[0] * 100, list(range(1, 101))]]), (bs, 2, [[[0] * bs, [n_keys] * bs]])]
    pr = _paged_rows(gpu, rows, bs, hq, hkv, d, seed=d + hkv)
    pr["cu_kv"] = torch.tensor([0, n_keys, 2 * n_keys], dtype=torch.int32, device=gpu)
    k, v = pr["kv"][:, :, 0], pr["kv"][:, :, 1]
    out, lse = torch.empty_like(pr["q"]), torch.empty((hq, len(rows), bs), device=gpu)
    tables = dict(attn_range=pr["rng"], q_block_table=pr["slots"], kv_block_table=pr["kv_table"], out_block_table=pr["slots"])
    _flash_attn_varlen_forward(pr["q"], k, v, pr["cu_q"], pr["cu_kv"], pr["total_q"], bs, 2 * bs, 0.0, d ** -0.5, causal=False,
                               window_size_left=-1, window_size_right=-1, softcap=0.0, alibi_slopes=None,
                               return_softmax=False, out_=out, lse_=lse, **tables)
    # (kv block, where to, tokens, memory, first visit, visits, all heads, all tiles); an entry of the unpadded tensors is a token
    kv_table, last, slot = pr["host"]["kv_table"].tolist(), n_keys - bs, 2
    groups = torch.tensor([[kv_table[0][0], 0, bs, 1, 0, 1, 0, 0], [kv_table[1][0], bs, bs, 1, 1, 1, 0, 0],
                           [kv_table[0][1], 2 * bs, last, 1, 2, 1, 0, 0], [kv_table[1][1], slot, last, 0, 3, 1, 0, 0]],
                          dtype=torch.int32, device=gpu)
    visits = torch.tensor([[0, 0], [1, 0], [0, 1], [1, 1]], dtype=torch.int32, device=gpu)
    n_tokens = 2 * bs + last

    def memory(n, offset, extra):  # n tokens' rows of `extra` elements more than they have, `offset` elements into memory of 7s
        whole = torch.full((n * (width + extra) + 8,), 7.0, dtype=torch.bfloat16, device=gpu)
        return whole, whole[offset : offset + n * (width + extra)].view(n, width + extra)

    def backward(paged, unpadded):  # each (offset of dK, offset of dV, elements between the rows)
        dk, dv = (memory((slot + 2) * bs, offset, paged[2]) for offset in paged[:2])
        dk2, dv2 = (memory(n_tokens + 1, offset, unpadded[2]) for offset in unpadded[:2])
        view = lambda m: m[1][:, :width].unflatten(1, (hkv, d))
        dq = torch.empty_like(out)
        _flash_attn_varlen_backward(pr["dout"], pr["q"], k, v, out, lse, dq, view(dk).unflatten(0, (slot + 2, bs)),
                                    view(dv).unflatten(0, (slot + 2, bs)), pr["cu_q"], pr["cu_kv"], pr["total_q"], 2 * n_keys, bs,
                                    2 * bs, 0.0, d ** -0.5, False, -1, -1, 0.0, None, False, dq_block_table=pr["slots"],
                                    dkv_block_table=pr["dkv_table"], dkv_groups=(groups, visits, view(dk2), view(dv2), None), **tables)
        written = [m[1][a : a + n, :width].clone().view(torch.int16) for m, a, n in
                   ((dk, slot * bs, last), (dv, slot * bs, last), (dk2, 0, n_tokens), (dv2, 0, n_tokens))]
        for m, a, n in ((dk, slot * bs, last), (dv, slot * bs, last), (dk2, 0, n_tokens), (dv2, 0, n_tokens)):
            m[1][a : a + n, :width] = 7.0
            assert (m[0] == 7.0).all(), "written beside the groups' tokens"
        return written

    lib = _lib.load()
    before = lib.dcp_attn_bwd_select(mode)
    try:
        wide = backward((0, 0, 0), (0, 0, 0))
        seven = torch.tensor(7.0, dtype=torch.bfloat16).view(torch.int16).item()
        assert all((rows_of != seven).any(1).all() for rows_of in wide)
        for paged, unpadded in (((0, 0, 0), (4, 0, 0)), ((0, 0, 0), (0, 4, 0)), ((0, 0, 0), (0, 0, 4)), ((4, 0, 0), (0, 0, 0)),
                                ((0, 4, 0), (0, 0, 0)), ((0, 0, 12), (0, 0, 0)), ((4, 4, 4), (4, 4, 4)), ((0, 0, 8), (0, 0, 16))):
            assert all(torch.equal(a, b) for a, b in zip(wide, backward(paged, unpadded))), (paged, unpadded)
    finally:
        lib.dcp_attn_bwd_select(before)
