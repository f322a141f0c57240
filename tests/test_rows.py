"""q, k, v as column slices of a wider tensor (a layer's split), read in place: the same bits as
their contiguous copies, in every operator and chain form; and which layouts are taken so."""
import numpy as np
import pytest
import torch

from avelang_amd import _native
from avelang_amd import gated_delta_rule as G


def _slices(B, T, Hqk, Hv, K, V, pad=0, device="cpu", seed=0):
    """q, k, v cut from one [B, T, pad + 2 Hqk K + Hv V + pad] tensor as a layer cuts them."""
    gen = torch.Generator().manual_seed(seed)
    y = torch.randn((B, T, 2 * pad + 2 * Hqk * K + Hv * V), generator=gen).to(torch.bfloat16)
    y = y.to(device)[..., pad:y.shape[-1] - pad]
    q, k, v = torch.split(y, [Hqk * K, Hqk * K, Hv * V], dim=-1)
    return q.reshape(B, T, Hqk, K), k.reshape(B, T, Hqk, K), v.reshape(B, T, Hv, V)


def test_layouts_taken_in_place():
    q, k, v = _slices(2, 5, 2, 4, 64, 128, pad=8)
    row = 2 * 2 * 64 + 4 * 128 + 16
    assert G._rows(q, k, v) == (row, row, row)
    assert G._rows(q[:1], k[:1], v[:1]) == (row, row, row)
    assert G._rows(q[:, :1], k[:, :1], v[:, :1]) == (5 * row, 5 * row, 5 * row)
    assert G._rows(*(x.contiguous() for x in (q, k, v))) is None          # nothing to gain
    assert G._rows(q.contiguous(), k, v) == (2 * 64, row, row)
    for bad in (q.transpose(1, 2).contiguous().transpose(1, 2),   # heads not together
                q.flip(1)[..., ::2].repeat_interleave(2, -1)[:, ::2].expand(2, 3, 2, 64)[:, :, ::2],
                q[:, :, :, :1].expand(2, 5, 2, 64),               # elements repeated
                q[:1].expand(2, 5, 2, 64),                        # batches at stride 0
                q[:, :1].expand(2, 5, 2, 64),                     # tokens at stride 0
                _slices(2, 5, 2, 4, 64, 128, pad=4)[0],           # 8-byte alignment
                q[:, ::2]):                                       # batches unevenly spaced
        assert not bad.is_contiguous() and G._row(bad) is None


def test_out_on_the_slices_tensor():
    """An out inside the tensor the slices are cut from is not written beside them: copies."""
    q, k, v = _slices(1, 6, 2, 4, 64, 64)
    flat = q._base.view(-1) if q._base is not None else q.reshape(-1)
    n = 6 * 4 * 64
    for out, taken in ((flat[:n].view(1, 6, 4, 64), False), (flat[-n:].view(1, 6, 4, 64), False),
                       (torch.empty(1, 6, 4, 64, dtype=torch.bfloat16), True), (None, True)):
        q2, k2, v2, rows = G._in_place(q, k, v, out)
        assert (rows is not None) == taken
        assert taken or all(x.is_contiguous() for x in (q2, k2, v2))
        assert all(torch.equal(x, y) for x, y in ((q, q2), (k, k2), (v, v2)))


@pytest.mark.gpu
@pytest.mark.parametrize("decode", [False, True])
def test_out_over_the_slices_gpu(rocm_device, decode):
    from avelang_amd import chunk_gated_delta_rule, fused_recurrent_gated_delta_rule
    op = fused_recurrent_gated_delta_rule if decode else chunk_gated_delta_rule
    B, T = (7, 1) if decode else (1, 130)
    gates = _gates(B, T, 4, rocm_device, False)
    kw = dict(output_final_state=True, use_qk_l2norm_in_kernel=True)
    want, _ = op(*_slices(B, T, 2, 4, 128, 128, device=rocm_device), *gates, **kw)
    q, k, v = _slices(B, T, 2, 4, 128, 128, device=rocm_device)
    n = B * T * 4 * 128
    out = q._base.view(-1)[-n:].view(B, T, 4, 128)
    o, _ = op(q, k, v, *gates, out=out, **kw)
    torch.cuda.synchronize()
    assert o is out and torch.equal(o, want)


def test_refused_rows():
    lib = _native.lib()
    for name in _native.EXPORTS_ROWS:
        assert hasattr(lib, name)
    P = [1 << 40, 2 << 40, 3 << 40]
    gates = [4 << 40, 5 << 40, None, None, None, None, 0, 0, 0, 1.0, 20.0]
    dims = [1, 64, 2, 4, 128, 128, 1]

    def call(p=P, rows=(256, 256, 512), o=6 << 40):
        return lib.gdn_chunk_fwd_rows(*p, *rows, *gates, None, None, o, None, *dims, 0.1, 0,
                                      7 << 40, 0, None)

    assert call() == -4                                            # (only the workspace left)
    for rows in ((255, 256, 512), (256, 260, 512), (256, 256, 504), (1 << 23, 256, 512)):
        assert call(rows=rows) == -2, rows
    assert call(p=[P[0] + 8, P[1], P[2]]) == -2
    assert call(o=P[0] + 2 * 63 * 1024, rows=(1024, 256, 512)) == -5   # inside q's last row
    assert lib.gdn_recurrent_fwd_rows(*P, 256, 256, 511, *gates, None, None, 6 << 40, None, None,
                                      *dims, 1, 0.1, 0, None) == -2


def _gates(B, T, Hv, dev, gated):
    gen = torch.Generator().manual_seed(1)
    a, b = (torch.randn((B, T, Hv), generator=gen).to(dev) for _ in range(2))
    if gated:
        return a.to(torch.bfloat16), b.to(torch.bfloat16), torch.zeros(Hv, device=dev), \
            torch.zeros(Hv, device=dev)
    return -0.1 * torch.nn.functional.softplus(a), torch.sigmoid(b)


@pytest.mark.gpu
@pytest.mark.parametrize("l2", [False, True])
@pytest.mark.parametrize("B,T,Hqk,Hv,K,V", [
    (1, 130, 2, 4, 128, 128), (2, 65, 1, 2, 64, 64), (1, 77, 2, 2, 128, 64),   # state-wave form
    (8, 70, 2, 8, 128, 128),                     # two tiles per workgroup (64 chains)
    (16, 70, 2, 8, 128, 128), (64, 70, 2, 4, 128, 128), (64, 3, 4, 4, 64, 128),   # whole heads
    (1, 4170, 1, 2, 128, 128), (1, 4353, 1, 2, 128, 128)])                     # segments
def test_prefill(rocm_device, B, T, Hqk, Hv, K, V, l2):
    from avelang_amd import chunk_gated_delta_rule, chunk_gated_delta_rule_gated
    qkv = _slices(B, T, Hqk, Hv, K, V, pad=16, device=rocm_device)
    if not l2:
        qkv = (0.05 * qkv[0].float(), 0.05 * qkv[1].float(), qkv[2])
        wide = torch.cat([x.flatten(2).to(torch.bfloat16) for x in qkv], -1)
        qkv = [x.reshape(B, T, h, d) for x, h, d in
               zip(wide.split([Hqk * K, Hqk * K, Hv * V], -1), (Hqk, Hqk, Hv), (K, K, V))]
    assert G._rows(*qkv) is not None
    for op, gated in ((chunk_gated_delta_rule, False), (chunk_gated_delta_rule_gated, True)):
        args = _gates(B, T, Hv, rocm_device, gated)
        kw = dict(output_final_state=True, use_qk_l2norm_in_kernel=l2)
        o, s = op(*qkv, *args, **kw)
        o2, s2 = op(*(x.contiguous() for x in qkv), *args, **kw)
        torch.cuda.synchronize()
        assert o.is_contiguous() and torch.equal(o, o2) and torch.equal(s, s2)
        assert bool(torch.isfinite(o).all()) and bool(o.any())


@pytest.mark.gpu
def test_packed_prefill(rocm_device):
    from avelang_amd import chunk_gated_delta_rule
    qkv = _slices(1, 300, 2, 4, 128, 128, device=rocm_device)
    cu = torch.from_numpy(np.array([0, 100, 100, 163, 300], dtype=np.int32)).to(rocm_device)
    g, beta = _gates(1, 300, 4, rocm_device, False)
    kw = dict(output_final_state=True, cu_seqlens=cu, use_qk_l2norm_in_kernel=True)
    o, s = chunk_gated_delta_rule(*qkv, g, beta, **kw)
    o2, s2 = chunk_gated_delta_rule(*(x.contiguous() for x in qkv), g, beta, **kw)
    torch.cuda.synchronize()
    assert torch.equal(o, o2) and torch.equal(s, s2)


@pytest.mark.gpu
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("B,T,Hqk,Hv,K,V", [(5, 1, 2, 4, 128, 128), (2, 3, 1, 4, 64, 128),
                                            (1, 1, 4, 4, 64, 64), (300, 1, 4, 4, 128, 64)])
def test_decode(rocm_device, B, T, Hqk, Hv, K, V, gated):
    from avelang_amd import (fused_recurrent_gated_delta_rule,
                             fused_recurrent_gated_delta_rule_gated)
    op = fused_recurrent_gated_delta_rule_gated if gated else fused_recurrent_gated_delta_rule
    qkv = _slices(B, T, Hqk, Hv, K, V, pad=8, device=rocm_device)
    args = _gates(B, T, Hv, rocm_device, gated)
    h0 = 0.01 * torch.randn((B + 3, Hv, K, V), device=rocm_device)
    slots = torch.randperm(B + 3)[:B].to(torch.int32).to(rocm_device)
    for idx in (None, slots):
        res = []
        for x in (qkv, [x.contiguous() for x in qkv]):
            pool = (h0 if idx is not None else h0[:B]).clone()
            res.append(op(*x, *args, initial_state=pool, output_final_state=True,
                          use_qk_l2norm_in_kernel=True, ssm_state_indices=idx))
        torch.cuda.synchronize()
        assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
