"""The forward chain's whole-head and segmented forms at the sizes where they
can go wrong: against the CPU oracles, and against the state-wave form.

Which form a call takes depends on its sizes (chain_form in gdn_chunk.hip):
from half a workgroup per compute unit on (K = V = 128; a whole one
otherwise) every (sequence, v-head) is one workgroup, and few long chains are
cut into segments.  Tolerances: the operator's (o 2e-2 absolute + relative,
final state 1e-3, gradients 1e-2 relative Frobenius).
"""
import numpy as np
import pytest
import torch

from avelang_amd import workloads as W
from oracle import cpu as oracle
from oracle import gdn_bwd_ref as RB

pytestmark = pytest.mark.gpu


def _cus(dev):
    return torch.cuda.get_device_properties(dev).multi_processor_count


def _run(wl, dev, l2=False, fn=None, **kw):
    from avelang_amd import chunk_gated_delta_rule
    t = wl.torch(dev)
    r = (fn or chunk_gated_delta_rule)(
        t["q"], t["k"], t["v"], t["g"], t["beta"], initial_state=t["initial_state"],
        output_final_state=True, cu_seqlens=t["cu_seqlens"], use_qk_l2norm_in_kernel=l2, **kw)
    torch.cuda.synchronize()
    return r


def _check(wl, dev, l2=False, what=""):
    o, s = _run(wl, dev, l2)
    a = wl.numpy()
    if l2:
        nrm = lambda x: x / np.sqrt((x * x).sum(-1, keepdims=True) + 1e-6)  # noqa: E731
        a["q"], a["k"] = W._bf16_round(nrm(a["q"])), W._bf16_round(nrm(a["k"]))
    o_ref, s_ref = oracle.run("chunk", **a)
    o, s = o.float().cpu().numpy(), s.cpu().numpy()
    bad = np.abs(o - o_ref) > 2e-2 + 2e-2 * np.abs(o_ref)
    assert not bad.any(), f"{what}: {bad.sum()} / {bad.size} outputs off"
    fro = np.linalg.norm(s - s_ref) / max(np.linalg.norm(s_ref), 1e-30)
    assert fro <= 1e-3, f"{what}: state {fro:.2e}"


@pytest.mark.parametrize("K,V,l2", [(128, 128, False), (128, 128, True), (64, 64, False),
                                    (64, 64, True), (128, 64, False), (64, 128, True)])
@pytest.mark.parametrize("T", [1, 63, 64, 65, 129, 200])
def test_whole_head(rocm_device, K, V, l2, T):
    """Tails of one to 64 tokens, one to four chunks, every head size, GQA 1 / 2 / 4."""
    Hqk, Hv = {1: (4, 4), 63: (1, 4), 64: (2, 4)}.get(T, (2, 4))
    B = -(-_cus(rocm_device) // Hv)
    wl = W.make(B, T, Hqk, Hv, K, V, seed=T, h0_scale=0.01 if T != 65 else 0.0, l2norm=not l2)
    _check(wl, rocm_device, l2, f"K{K} V{V} T{T}")


@pytest.mark.parametrize("chunks,Hqk,Hv", [(1, 1, 1), (1, 1, 3), (3, 3, 6), (127, 1, 3),
                                           (64, 2, 2), (43, 3, 9), (129, 1, 2), (51, 5, 10)])
def test_prep_workgroup_order(rocm_device, chunks, Hqk, Hv):
    """Every (chunk, v-head) once, with (chunk, qk-head) pairs under, at and over multiples of
    the 128 that the prep kernel takes between two v-heads of a pair."""
    _check(W.make(1, 64 * chunks - 5, Hqk, Hv, 128, 128, seed=chunks, h0_scale=0.01), rocm_device)


def _cu(lens):
    return np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)


def _packed(dev, long=0, longs=(), K=128, l2norm=True):
    """Sequences of 0 to 150 tokens (and one of `long`, or some of `longs`) over enough heads for
    the form."""
    Hv = 8 * 128 // K
    n = -(-_cus(dev) // Hv)
    rng = np.random.Generator(np.random.PCG64(5))
    lens = rng.integers(1, 151, size=n)
    lens[3], lens[n // 2] = 0, long or lens[n // 2]
    lens[5:5 + 2 * len(longs):2] = longs
    cu = _cu(lens)
    return W.make(1, int(cu[-1]), 4, Hv, K, K, seed=6, cu_seqlens=cu, l2norm=l2norm)


def test_whole_head_packed(rocm_device):
    _check(_packed(rocm_device), rocm_device, what="packed")


def test_whole_head_packed_with_one_long_sequence(rocm_device):
    """A sequence far over the mean takes state waves, the others stay whole."""
    _check(_packed(rocm_device, long=6011), rocm_device, what="packed, one long")


def _heavy(l2):
    """32 heads: a sequence that is cut, in a batch that fills the GPU (load 24)."""
    cu = _cu([9000, 0, 1, 3500])
    return W.make(1, int(cu[-1]), 16, 32, 128, 128, seed=7, cu_seqlens=cu, l2norm=not l2)


@pytest.mark.parametrize("l2", [False, True])
def test_whole_head_packed_with_one_long_sequence_cut(rocm_device, l2):
    """A sequence far over the load is cut into segments, the others stay whole."""
    _check(_heavy(l2), rocm_device, l2, what="packed, one cut")


# of a load of 3 to 13 chunks: under, at and over the 4 loads that are long, and over the one that
# then takes state waves
_LONGS = [(3000,), (1000, 500, 7, 1500), (3000, 2000), (3000, 2000, 7000), (9000, 4000, 9000, 250)]


@pytest.mark.parametrize("K,l2", [(128, False), (128, True), (64, False)])
@pytest.mark.parametrize("longs", _LONGS)
def test_packed_with_long_sequences(rocm_device, longs, K, l2):
    """Whole heads for the short sequences, state waves for the others."""
    _check(_packed(rocm_device, longs=longs, K=K, l2norm=not l2), rocm_device, l2, str(longs))


@pytest.mark.parametrize("l2", [False, True])
@pytest.mark.parametrize("longs", _LONGS + ["cut"])
def test_training_packed_with_long_sequences(rocm_device, longs, l2):
    from avelang_amd import chunk_gated_delta_rule_bwd, chunk_gated_delta_rule_fwd_save
    wl = _heavy(l2) if longs == "cut" else _packed(rocm_device, longs=longs, l2norm=not l2)
    t = wl.torch(rocm_device)
    o, s = _run(wl, rocm_device, l2)
    o2, s2, ws = _run(wl, rocm_device, l2, fn=chunk_gated_delta_rule_fwd_save)
    assert torch.equal(o, o2) and torch.equal(s, s2)
    args = (t["q"], t["k"], t["v"], t["g"], t["beta"], torch.ones_like(t["v"]))
    kw = dict(initial_state=t["initial_state"], cu_seqlens=t["cu_seqlens"],
              use_qk_l2norm_in_kernel=l2)
    got = chunk_gated_delta_rule_bwd(*args, workspace=ws, saved=True, **kw)
    again = chunk_gated_delta_rule_bwd(*args, **kw)
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(got, again))


@pytest.mark.parametrize("B,T,Hqk,Hv,D,l2,decay", [
    (1, 4096, 1, 2, 128, False, 0.1),      # segments divide the chunks or not,
    (1, 4096 + 1, 2, 2, 128, True, 0.1),   # the last chunk of one token,
    (2, 5000, 1, 2, 128, False, 0.002),    # and states that carry through many segments
    (1, 6200, 2, 4, 64, False, 0.002),
    (2, 4159, 1, 4, 64, True, 0.01),
    (1, 4352, 1, 2, 128, False, 0.002), (1, 4353, 2, 2, 128, True, 0.1)])   # (68 chunks and more)
def test_segments(rocm_device, B, T, Hqk, Hv, D, l2, decay):
    wl = W.make(B, T, Hqk, Hv, D, D, seed=T, decay=decay, h0_scale=0.05, l2norm=not l2)
    _check(wl, rocm_device, l2, f"segments T{T}")


def test_segments_without_an_initial_state(rocm_device):
    _check(W.make(1, 4500, 1, 2, 128, 128, seed=1, decay=0.01, h0_scale=0.0), rocm_device)


@pytest.mark.parametrize("lens", [[9000, 0, 1, 7000], [130, 8200, 5000], [0, 0, 13000],
                                  [13000, 0, 1, 7000]])
def test_segments_packed(rocm_device, lens):
    """Sequences of many, one and no segments."""
    cu = _cu(lens)
    _check(W.make(1, int(cu[-1]), 1, 2, 128, 128, seed=2, cu_seqlens=cu, decay=0.01,
                  h0_scale=0.05), rocm_device, what=str(lens))


@pytest.mark.parametrize("T,Hv,n", [(9000, 2, 2), (400, 8, 64), (3000, 8, 32), (12500, 32, 4)])
def test_violated_cu_seqlens(rocm_device, T, Hv, n):
    """The device contract in segments, whole heads, with long sequences listed and with long ones
    cut: o zero-filled, the final state the initial one."""
    wl = W.make(1, T, 1, Hv, 128, 128, seed=3, cu_seqlens=_cu([T // n] * n))
    t = wl.torch(rocm_device)
    from avelang_amd import chunk_gated_delta_rule
    cu = t["cu_seqlens"].clone()
    cu[1] = T + 5
    out = torch.full_like(t["v"], 7.0)
    _, ht = chunk_gated_delta_rule(t["q"], t["k"], t["v"], t["g"], t["beta"],
                                   initial_state=t["initial_state"], output_final_state=True,
                                   cu_seqlens=cu, out=out)
    torch.cuda.synchronize()
    assert not out.any() and torch.equal(ht, t["initial_state"])


def _training(dev, l2):
    """(workload, what): one of each form."""
    B = -(-_cus(dev) // 4)
    yield W.make(B, 70, 2, 4, 128, 128, seed=8, h0_scale=0.01, l2norm=not l2), "whole"
    yield W.make(1, 4200, 1, 2, 128, 128, seed=9, h0_scale=0.05, decay=0.01,
                 l2norm=not l2), "segments"
    yield W.make(1, 4400, 1, 2, 128, 128, seed=9, h0_scale=0.05, decay=0.01,
                 l2norm=not l2), "segments, of 68 chunks and more"
    yield W.make(1, 6200, 5, 10, 128, 128, seed=9, h0_scale=0.05, decay=0.01,
                 l2norm=not l2), "segments, nine chains and more"


@pytest.mark.parametrize("l2", [False, True])
def test_training_forward_equals_the_plain_one(rocm_device, l2):
    from avelang_amd import chunk_gated_delta_rule_fwd_save
    for wl, what in _training(rocm_device, l2):
        o, s = _run(wl, rocm_device, l2)
        o2, s2, _ = _run(wl, rocm_device, l2, fn=chunk_gated_delta_rule_fwd_save)
        assert torch.equal(o, o2) and torch.equal(s, s2), what


@pytest.mark.parametrize("l2", [False, True])
def test_training_forward_beside_a_plain_one_in_segments(rocm_device, l2):
    """Sizes whose plain forward alone is cut: o and the final state agree to rounding (o within
    two bf16 steps of its size, the state as the forms' own 4e-4 from 64 bits allow)."""
    from avelang_amd import chunk_gated_delta_rule_fwd_save
    wl = W.make(1, 5500, 6, 12, 128, 128, seed=9, h0_scale=0.05, decay=0.01, l2norm=not l2)
    o, s = _run(wl, rocm_device, l2)
    o2, s2, _ = _run(wl, rocm_device, l2, fn=chunk_gated_delta_rule_fwd_save)
    assert not torch.equal(s, s2)
    assert (s2 - s).norm() <= 8e-4 * s.norm()
    assert (o2.float() - o.float()).norm() <= 2 ** -7 * o.float().norm()


def test_gradients(rocm_device):
    """The saved states and deltas of both forms, through the backward; recomputed == saved."""
    from avelang_amd import chunk_gated_delta_rule_bwd, chunk_gated_delta_rule_fwd_save
    for wl, what in _training(rocm_device, False):
        a, t = wl.numpy(), wl.torch(rocm_device)
        rng = np.random.Generator(np.random.PCG64(1))
        do = W._bf16_round(rng.standard_normal(a["v"].shape, dtype=np.float32))
        ref = RB.chunked_bwd(a["q"], a["k"], a["v"], a["g"], a["beta"], do, None,
                             initial_state=a["initial_state"])
        args = (t["q"], t["k"], t["v"], t["g"], t["beta"],
                torch.from_numpy(do).to(device=rocm_device, dtype=torch.bfloat16))
        _, _, ws = _run(wl, rocm_device, fn=chunk_gated_delta_rule_fwd_save)
        got = chunk_gated_delta_rule_bwd(*args, initial_state=t["initial_state"], workspace=ws,
                                         saved=True)
        again = chunk_gated_delta_rule_bwd(*args, initial_state=t["initial_state"])
        torch.cuda.synchronize()
        for name, x, y in zip(("dq", "dk", "dv", "dg", "dbeta", "dh0"), got, again):
            assert torch.equal(x, y), f"{what}: {name} saved != recomputed"
            x = x.double().cpu().numpy()
            rel = np.linalg.norm(x - ref[name]) / np.linalg.norm(ref[name])
            assert rel <= (1e-3 if name == "dh0" else 1e-2), f"{what}: {name} {rel:.2e}"


def test_noalloc_takes_what_fits_without_segments(rocm_device):
    """A problem that gdn_chunk_fwd runs in segments, its workspace with them over the library's
    scratch, without them under it: still accepted, and the same up to rounding."""
    from avelang_amd import _native
    lib = _native.lib()
    wl = W.make(1, 8192, 16, 16, 128, 128, seed=12, h0_scale=0.01)
    assert lib.gdn_chunk_workspace_bytes(1, 8192, 16, 16, 128, 128, 1, 0, 0) > (32 << 20)
    o, s = _run(wl, rocm_device)
    t = wl.torch(rocm_device)
    o2, s2 = torch.full_like(o, 5.0), torch.full_like(s, 5.0)
    rc = lib.gdn_chunk_fwd_noalloc(
        *(t[n].data_ptr() for n in ("q", "k", "v", "g", "beta", "initial_state")), s2.data_ptr(),
        o2.data_ptr(), None, 1, 8192, 16, 16, 128, 128, 1, 128 ** -0.5, 0,
        torch.cuda.current_stream(rocm_device).cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0, lib.gdn_last_error().decode()
    assert (s2 - s).norm() <= 1e-3 * s.norm()
    assert (o2.float() - o.float()).norm() <= 1e-2 * o.float().norm()


@pytest.mark.parametrize("what", ["state waves", "whole heads", "segments"])
@pytest.mark.parametrize("shift", [-30, 20])
def test_q_of_any_magnitude(rocm_device, what, shift):
    """Without l2norm q counts as the caller's bf16, also far outside fp16's range (2^-14 to
    65504): q 2^shift with scale 2^-shift, both exact, gives the same bits in every form."""
    from avelang_amd import chunk_gated_delta_rule
    B = -(-_cus(rocm_device) // 4)
    shape = {"state waves": (1, 200, 2, 4), "whole heads": (B, 130, 2, 4),
             "segments": (1, 4400, 1, 2)}[what]
    t = W.make(*shape, 128, 128, seed=13, h0_scale=0.05, decay=0.01).torch(rocm_device)
    o, o2 = (chunk_gated_delta_rule(t["q"] * 2.0 ** n, t["k"], t["v"], t["g"], t["beta"],
                                    scale=128 ** -0.5 * 2.0 ** -n,
                                    initial_state=t["initial_state"])[0] for n in (0, shift))
    torch.cuda.synchronize()
    assert bool(o.any()) and torch.equal(o, o2)


def _in_place_cases(dev):
    """(workload, l2) at segmented sizes: batched, and packed with cut and uncut sequences, the
    last segments of one chunk and of more."""
    yield W.make(2, 6144 + 1, 1, 2, 128, 128, seed=21, decay=0.01, h0_scale=0.05), False
    yield W.make(1, 6200, 2, 4, 64, 64, seed=22, decay=0.002, h0_scale=0.05, l2norm=False), True
    for lens in ([19000, 0, 1, 7000], [130, 13200, 6000]):
        cu = _cu(lens)
        yield W.make(1, int(cu[-1]), 1, 2, 128, 128, seed=23, cu_seqlens=cu, decay=0.01,
                     h0_scale=0.05, l2norm=False), True
    yield _packed(dev, longs=(3000, 2000, 7000)), False
    yield _heavy(True), True


def _save_workspace(wl, l2, dev):
    from avelang_amd.gated_delta_rule import chunk_bwd_workspace_bytes
    n = chunk_bwd_workspace_bytes(*(wl.dims[x] for x in ("B", "T", "Hqk", "Hv", "K", "V", "N")),
                                  wl.cu_seqlens is not None, l2)
    return torch.empty(n, dtype=torch.uint8, device=dev)


@pytest.mark.parametrize("op", ["plain", "gated", "rows", "save"])
def test_final_state_in_place_of_the_initial_one(rocm_device, op):
    from avelang_amd.gated_delta_rule import _chunk_fwd   # (with the gating, which the public form
    for wl, l2 in _in_place_cases(rocm_device):   # gives no final_state, too)
        t = wl.torch(rocm_device)
        q, k, v = t["q"], t["k"], t["v"]
        if op == "rows":   # column slices of one tensor, read in place
            wide = torch.cat([x.flatten(2) for x in (q, k, v)], -1)
            q, k, v = (x.reshape(y.shape) for x, y in zip(
                wide.split([y[0, 0].numel() for y in (q, k, v)], -1), (q, k, v)))
        g, beta, gate = t["g"], t["beta"], None
        if op == "gated":
            g, beta = g.to(torch.bfloat16), beta.to(torch.bfloat16)
            zero = torch.zeros(v.shape[2], device=rocm_device)
            gate = (zero - 4.0, zero, 1.0, 20.0)
        res = []
        for same in (False, True):
            h0 = t["initial_state"].clone()
            res.append(_chunk_fwd(q, k, v, g, beta, None, h0, True, t["cu_seqlens"], l2, gate=gate,
                                  final_state=h0 if same else None,
                                  save_workspace=_save_workspace(wl, l2, rocm_device)
                                  if op == "save" else None))
            assert not same or res[-1][1] is h0
        torch.cuda.synchronize()
        for x, y in zip(*res):
            assert torch.equal(x, y), (op, wl.dims)


@pytest.mark.parametrize("what", ["state waves", "whole heads", "segments", "segments, 64"])
def test_padding_leaves_the_state(rocm_device, what):
    """Tokens of g = beta = 0 leave every bit of the fp32 state, in every form."""
    from avelang_amd import chunk_gated_delta_rule
    B = -(-_cus(rocm_device) // 4)
    B, T, Hv, D = {"state waves": (1, 200, 4, 128), "whole heads": (B, 130, 4, 128),
                   "segments": (1, 4400, 2, 128), "segments, 64": (2, 5000, 2, 64)}[what]
    t = W.make(B, T, 1, Hv, D, D, seed=14, h0_scale=1.0).torch(rocm_device)
    zero = torch.zeros_like(t["g"])
    _, ht = chunk_gated_delta_rule(t["q"], t["k"], t["v"], zero, zero, output_final_state=True,
                                   initial_state=t["initial_state"])
    torch.cuda.synchronize()
    assert torch.equal(ht, t["initial_state"])


@pytest.mark.parametrize("small,large", [
    (dict(B=1, T=5184, Hqk=2, Hv=4), dict(B=1, T=5248, Hqk=2, Hv=4)),        # segments
    (dict(B=2, T=700, Hqk=16, Hv=32), dict(B=4, T=700, Hqk=16, Hv=32))])     # two tiles, fp16 K
def test_in_the_workspace_of_a_larger_problem(rocm_device, small, large):
    """... whose form needs less, and in the least that the call takes: the same to rounding."""
    from avelang_amd import chunk_workspace_bytes
    size = lambda d: chunk_workspace_bytes(d["B"], d["T"], d["Hqk"], d["Hv"], 128, 128,  # noqa: E731
                                           d["B"], False)
    wl = W.make(**small, K=128, V=128, seed=31, h0_scale=0.05)
    o, s = _run(wl, rocm_device)
    n = -(-small["T"] // 64) * small["B"] * small["Hv"]
    least = 512 + 256 * n + 2 * 6144 * n
    for nbytes in (size(large), least):
        assert least <= nbytes
        ws = torch.full((nbytes + 4096,), 0x5a, dtype=torch.uint8, device=rocm_device)
        o2, s2 = _run(wl, rocm_device, workspace=ws[:nbytes])
        assert bool((ws[nbytes:] == 0x5a).all())
        assert (s2 - s).norm() <= 8e-4 * s.norm()
        assert (o2.float() - o.float()).norm() <= 2 ** -7 * o.float().norm()
    assert least < size(small)
    with pytest.raises(ValueError, match="workspace needs"):
        _run(wl, rocm_device, workspace=ws[:least - 1])


@pytest.mark.parametrize("longs", [(), (3000,), (1000, 500, 7, 1500)])
def test_noalloc_takes_the_same_form_of_a_packed_batch(rocm_device, longs):
    """Long sequences in state waves beside whole heads, in the library's scratch: bit for bit."""
    from avelang_amd import _native
    wl = _packed(rocm_device, longs=longs)
    d, t = wl.dims, wl.torch(rocm_device)
    o, s = _run(wl, rocm_device)
    o2, s2 = torch.full_like(o, 5.0), torch.full_like(s, 5.0)
    rc = _native.lib().gdn_chunk_fwd_noalloc(
        *(t[n].data_ptr() for n in ("q", "k", "v", "g", "beta", "initial_state")), s2.data_ptr(),
        o2.data_ptr(), t["cu_seqlens"].data_ptr(),
        *(d[n] for n in ("B", "T", "Hqk", "Hv", "K", "V", "N")), 128 ** -0.5, 0,
        torch.cuda.current_stream(rocm_device).cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0, _native.last_error()
    assert torch.equal(o, o2) and torch.equal(s, s2)


@pytest.mark.parametrize("K,V", [(128, 128), (64, 64), (128, 64), (64, 128)])
def test_q_rows_of_many_magnitudes(rocm_device, K, V):
    """Whole heads: every token's q times a power of two of its own (2^-6 to 2^6, and 2^-12 to 2^12:
    under and over the 256 where each row takes a scale of its own) gives its o times that (to a
    bf16 rounding of each: P is rounded to fp16, whose subnormals the small rows reach; the scale
    keeps it between them and fp16's largest)."""
    from avelang_amd import chunk_gated_delta_rule
    B = -(-_cus(rocm_device) // 4)
    t = W.make(B, 130, 2, 4, K, V, seed=15, h0_scale=0.05, decay=0.01).torch(rocm_device)
    gen = torch.Generator().manual_seed(1)
    for top in (6, 12):
        f = 2.0 ** torch.randint(-top, top + 1, (B, 130, 1, 1), generator=gen).to(rocm_device)
        o, o2 = (chunk_gated_delta_rule((t["q"].float() * x).to(torch.bfloat16), t["k"], t["v"],
                                        t["g"], t["beta"], scale=K ** -0.5 * 64,
                                        initial_state=t["initial_state"])[0].float()
                 for x in (torch.ones_like(f), f))
        torch.cuda.synchronize()
        off = (o2 - f * o).norm(dim=-1) / (f * o).norm(dim=-1)
        assert off.max() <= 2 ** -7, (top, off.max())


@pytest.mark.parametrize("what", ["state waves", "whole heads", "segments"])
@pytest.mark.parametrize("bad", [float("inf"), float("nan"), 2.0 ** 100])
def test_a_token_of_q_out_of_range_leaves_the_others(rocm_device, what, bad):
    """Without l2norm an inf, NaN or outlier in one token's q changes that token's o alone, in every
    form (its neighbours share the helper wave that scales their rows)."""
    from avelang_amd import chunk_gated_delta_rule
    B = -(-_cus(rocm_device) // 4)
    shape = {"state waves": (1, 200, 2, 4), "whole heads": (B, 130, 2, 4),
             "segments": (1, 4400, 1, 2)}[what]
    t = W.make(*shape, 128, 128, seed=16, h0_scale=0.05, decay=0.01).torch(rocm_device)
    token = 70
    q2 = t["q"].clone()
    q2[:, token, :, 5] = bad
    o, o2 = (chunk_gated_delta_rule(q, t["k"], t["v"], t["g"], t["beta"],
                                    initial_state=t["initial_state"])[0] for q in (t["q"], q2))
    torch.cuda.synchronize()
    others = torch.arange(shape[1], device=rocm_device) != token
    assert torch.equal(o[:, others], o2[:, others])
    if bad == 2.0 ** 100:   # (finite in fp32 sums, out of fp16's P: inf or NaN, never plausible)
        assert not torch.equal(o[:, token], o2[:, token])
