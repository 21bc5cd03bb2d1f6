"""mamba_chunk_scan_combined (Mamba-2's SSD scan) on the GPU against the
float64 oracle (oracle/ssd.py, pinned by tests/test_oracle_ssd.py).

Cases: sequence lengths that are and are not multiples of the 64-step chunk
(one chunk, several, a ragged tail, 2048 steps), headdim 16-64, dstate
16-128, 1, 2 or 4 groups, D per head or per channel, with and without z,
dt_bias, softplus, a dt_limit clamp, initial states and final states;
float32, bfloat16 and float16 storage; every gradient; workgroups walking
1, 2, 4 or 8 heads of a group; chunk states carried by two launches or by
the in-order kernels; opcheck of the two operators; an empty sequence.
Tolerances (unscaled, |got - want| <= atol + rtol |want|): float32 outputs
and final states rtol 1e-4 / atol 1e-5; float32 gradients rtol 1e-3 with
atol 1e-4 for per-element gradients (dx, ddt, dz) and 1e-3 for sums (dA,
dB, dC, dD, ddt_bias, dinitial_states); 16-bit storage 2e-2 / 2e-2, against
the oracle on the same rounded inputs and upstream gradients.
"""

import math

import numpy as np
import pytest
import torch

from conftest import assert_close_report
from oracle import ssd as S

import mamba_cpu

pytestmark = pytest.mark.gpu
DEV = "cuda"
NAMES = ("x", "dt", "A", "B", "C", "D", "z", "dt_bias", "initial_states")


def case(b, l, h, p, g, n, seed=0, D="hp", z=True, bias=True, init=False, dtype=torch.float32):
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen)  # noqa: E731
    c = dict(x=r(b, l, h, p).to(dtype), dt=r(b, l, h) * 0.5 - 1.0,
             A=-torch.exp(torch.rand(h, generator=gen) * math.log(8)),
             B=r(b, l, g, n).to(dtype), C=r(b, l, g, n).to(dtype))
    c["D"] = None if D is None else r(*((h, p) if D == "hp" else (h,)))
    c["z"] = r(b, l, h, p).to(dtype) if z else None
    c["dt_bias"] = torch.rand(h, generator=gen) * 0.5 if bias else None
    c["initial_states"] = r(b, h, p, n) if init else None
    return c


def run(c, grads=True, softplus=True, limit=(0.0, float("inf")), seed=1):
    """out, final states and the gradients of sum(out W) + sum(final V) on
    the GPU, and W, V."""
    dev = {k: None if v is None else v.to(DEV).requires_grad_(grads) for k, v in c.items()}
    out, fin = mamba_cpu.mamba_chunk_scan_combined(**dev, chunk_size=256, dt_softplus=softplus,
                                                   dt_limit=limit, return_final_states=True)
    gen = torch.Generator().manual_seed(seed)
    W = torch.randn(out.shape, generator=gen).to(out.dtype)
    V = torch.randn(fin.shape, generator=gen)
    got = {}
    if grads:
        ((out.float() * W.to(DEV).float()).sum() + (fin * V.to(DEV)).sum()).backward()
        got = {k: v.grad for k, v in dev.items() if v is not None}
    torch.cuda.synchronize()
    return out.detach(), fin.detach(), got, W, V


def check(c, out, fin, got, W, V, softplus=True, limit=(0.0, float("inf")), low=False):
    kw = dict(dt_softplus=softplus, dt_limit=limit)
    want, want_fin = S.ssd_fwd(**c, **kw)
    o_tol = (2e-2, 2e-2) if low else (1e-4, 1e-5)
    assert_close_report(out, want, *o_tol, "out")
    assert_close_report(fin, want_fin, *((2e-2, 2e-2) if low else (1e-4, 1e-5)), "final_states")
    if not got:
        return
    grads = S.ssd_bwd(**c, **kw, dout=W.float(), dfinal_states=V)
    for name, w in zip(NAMES, grads):
        if c[name] is None:
            assert w is None, name
            continue
        if low:
            tol = (2e-2, 2e-2)
        else:
            tol = (1e-3, 1e-4) if name in ("x", "dt", "z") else (1e-3, 1e-3)
        assert_close_report(got[name], w, *tol, f"d{name}")


SHAPES = [
    # b, l, h, p, g, n
    (2, 64, 2, 16, 1, 16),
    (1, 100, 4, 32, 2, 32),
    (2, 130, 4, 64, 1, 128),
    (1, 200, 8, 16, 4, 64),
    (1, 37, 2, 64, 2, 48),
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "b{}l{}h{}p{}g{}n{}".format(*s))
def test_forward_and_gradients_match_oracle(shape):
    c = case(*shape, seed=sum(shape))
    check(c, *run(c))


@pytest.mark.parametrize("opts", [
    dict(D="h", z=False, bias=False, init=True),
    dict(D=None, z=True, bias=True, init=True),
    dict(D="hp", z=False, bias=True, init=False),
], ids=["Dh-noz-init", "noD-z-init", "noz-bias"])
@pytest.mark.parametrize("softplus,limit", [(True, (0.0, float("inf"))), (True, (0.05, 0.6)),
                                            (False, (0.0, float("inf")))], ids=["sp", "sp-clamp", "raw"])
def test_options_match_oracle(opts, softplus, limit):
    c = case(2, 90, 4, 32, 2, 32, seed=5, **opts)
    if not softplus:
        c["dt"] = c["dt"].abs() * 0.3 + 0.05  # a positive step without softplus
    check(c, *run(c, softplus=softplus, limit=limit), softplus=softplus, limit=limit)


def test_raw_negative_steps_are_clamped():
    """Without softplus, a negative raw step is clamped to the default
    dt_limit (0, inf): step 0 and no raw-dt gradient there (mamba_ssm's and
    transformers' semantics; the oracle is pinned against transformers'
    mamba2_chunk_scan in tests/test_oracle_ssd.py)."""
    c = case(2, 150, 4, 32, 2, 32, seed=6, init=True)
    c["dt"] = c["dt"] + 0.8  # about half of dt + dt_bias below 0
    out, fin, got, W, V = run(c, softplus=False)
    check(c, out, fin, got, W, V, softplus=False)
    neg = (c["dt"] + c["dt_bias"][None, None]) < 0
    assert 0.2 < neg.float().mean().item() < 0.8
    assert torch.all(got["dt"].cpu()[neg] == 0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_low_precision_storage(dtype):
    c = case(2, 150, 4, 64, 2, 64, seed=9, dtype=dtype)
    out, fin, got, W, V = run(c)
    assert out.dtype == dtype and got["x"].dtype == dtype and got["B"].dtype == dtype
    check(c, out, fin, got, W, V, low=True)


def test_long_sequence_2048_steps():
    """32 chunks: the state passing over many chunks, forward and backward."""
    c = case(1, 2048, 4, 64, 1, 64, seed=13, init=True)
    check(c, *run(c))


def test_no_grad_forward_equals_training_forward():
    c = case(1, 130, 4, 32, 2, 32, seed=3)
    dev = {k: None if v is None else v.to(DEV) for k, v in c.items()}
    with torch.no_grad():
        a = mamba_cpu.mamba_chunk_scan_combined(**dev, chunk_size=64, dt_softplus=True)
    b = mamba_cpu.mamba_chunk_scan_combined(**{k: None if v is None else v.requires_grad_() for k, v in dev.items()},
                                            chunk_size=64, dt_softplus=True)
    assert torch.equal(a, b.detach())


def test_empty_sequence_passes_the_initial_state_through():
    c = case(2, 0, 2, 16, 1, 16, seed=4, init=True)
    dev = {k: None if v is None else v.to(DEV).requires_grad_() for k, v in c.items()}
    out, fin = mamba_cpu.mamba_chunk_scan_combined(**dev, chunk_size=64, return_final_states=True)
    assert out.shape == (2, 0, 2, 16)
    assert torch.equal(fin, dev["initial_states"])
    V = torch.randn_like(fin)
    (out.sum() + (fin * V).sum()).backward()
    assert torch.equal(dev["initial_states"].grad, V)
    for k in ("A", "D", "dt_bias"):
        assert torch.count_nonzero(dev[k].grad) == 0, k


def test_rejects_unsupported_shapes_and_options():
    c = case(1, 16, 2, 16, 1, 16)
    dev = {k: None if v is None else v.to(DEV) for k, v in c.items()}
    seq = torch.zeros(1, 16, dtype=torch.int32, device=DEV)
    with pytest.raises(ValueError, match="cu_seqlens"):
        mamba_cpu.mamba_chunk_scan_combined(**dev, chunk_size=64, seq_idx=seq, return_varlen_states=True)
    with pytest.raises(ValueError, match="seq_idx"):
        mamba_cpu.mamba_chunk_scan_combined(**dev, chunk_size=64, seq_idx=seq[:, :8])
    bad = dict(dev, x=torch.randn(1, 16, 2, 24, device=DEV), z=None, D=None)
    with pytest.raises(NotImplementedError, match="headdim"):
        mamba_cpu.mamba_chunk_scan_combined(**bad, chunk_size=64)
    with pytest.raises(ValueError):
        mamba_cpu.mamba_chunk_scan_combined(**{k: None if v is None else v.cpu() for k, v in dev.items()},
                                            chunk_size=64)


def run_ops(c, head_block=0, chunk_pass=0, softplus=True, limit=(0.0, float("inf")), seed=1, seq=None):
    """Forward and backward through the operators with the chunk kernels'
    head block and the way chunk states are carried pinned: out, final
    states, the nine gradients of sum(out W) + sum(final V), and W, V.
    seq: packed-sequence ids (batch, seqlen) or None."""
    d = {k: None if v is None else v.to(DEV) for k, v in c.items()}
    if d["D"] is not None and d["D"].dim() == 1:   # the operator takes D per channel
        d["D"] = d["D"][:, None].expand(d["x"].shape[2:]).contiguous()
    args = (d["x"], d["dt"], d["A"], d["B"], d["C"], d["D"], d["z"], d["dt_bias"], d["initial_states"],
            softplus, float(limit[0]), float(limit[1]))
    sq = None if seq is None else torch.as_tensor(seq, dtype=torch.int32).to(DEV)
    out, fin, saved, ysave = torch.ops.mamba_cpu.ssd_fwd(*args, True, head_block, chunk_pass, seq_idx=sq)
    gen = torch.Generator().manual_seed(seed)
    W = torch.randn(out.shape, generator=gen).to(out.dtype)
    V = torch.randn(fin.shape, generator=gen)
    g = torch.ops.mamba_cpu.ssd_bwd(W.to(DEV), V.to(DEV), *args, saved, ysave, head_block, chunk_pass,
                                    seq_idx=sq)
    torch.cuda.synchronize()
    return out, fin, g, W, V


@pytest.mark.parametrize("shape,blocks", [
    ((2, 130, 8, 32, 1, 64), (1, 2, 4, 8)),
    ((1, 200, 8, 16, 2, 32), (2, 4)),
    ((3, 70, 4, 64, 1, 128), (2, 4)),
], ids=["h8g1", "h8g2", "h4n128"])
def test_head_blocks_match_oracle(shape, blocks):
    """Workgroups walking 2, 4 or 8 heads of a group (C B^T shared, dB/dC
    summed over the block's heads in the accumulators, partials per head
    block): every head-block size against the oracle, and the forward
    bitwise equal across sizes (each head's arithmetic is the same)."""
    c = case(*shape, seed=sum(shape) + 1, init=True)
    want = S.ssd_fwd(**c, dt_softplus=True)
    first = None
    for hb in blocks:
        out, fin, g, W, V = run_ops(c, head_block=hb)
        print(f" head_block {hb}")
        assert_close_report(out, want[0], 1e-4, 1e-5, "out")
        assert_close_report(fin, want[1], 1e-4, 1e-5, "final_states")
        wg = S.ssd_bwd(**c, dt_softplus=True, dout=W.float(), dfinal_states=V)
        for name, got, w in zip(NAMES, g, wg):
            tol = (1e-3, 1e-4) if name in ("x", "dt", "z") else (1e-3, 1e-3)
            assert_close_report(got, w, *tol, f"d{name}")
        if first is None:
            first = (out, fin)
        else:
            assert torch.equal(out, first[0]) and torch.equal(fin, first[1])


def check_ops(c, got, softplus=True, limit=(0.0, float("inf")), low=False, seq=None):
    out, fin, g, W, V = got
    kw = dict(dt_softplus=softplus, dt_limit=limit, seq_idx=seq)
    want = S.ssd_fwd(**c, **kw)
    tol = (2e-2, 2e-2) if low else (1e-4, 1e-5)
    assert_close_report(out, want[0], *tol, "out")
    assert_close_report(fin, want[1], *tol, "final_states")
    wg = S.ssd_bwd(**c, **kw, dout=W.float(), dfinal_states=V)
    for name, got_g, w in zip(NAMES, g, wg):
        if c[name] is None:
            continue
        if name == "D" and c["D"].dim() == 1:   # per-channel dD back to the per-head D
            got_g = got_g.sum(-1)
        if low:
            tol = (2e-2, 2e-2)
        else:
            tol = (1e-3, 1e-4) if name in ("x", "dt", "z") else (1e-3, 1e-3)
        assert_close_report(got_g, w, *tol, f"d{name}")


@pytest.mark.parametrize("shape,opts", [
    ((2, 130, 4, 64, 1, 128), dict(init=True)),
    ((1, 200, 8, 16, 4, 64), dict(z=False)),
    ((3, 70, 4, 32, 2, 48), dict(init=True, D="h")),
    ((1, 37, 2, 64, 2, 16), dict(bias=False)),
    ((2, 300, 4, 48, 1, 32), dict(init=True, z=False, D=None)),
], ids=["n128-init", "p16-noz", "n48-init", "n16-short", "p48-noD"])
@pytest.mark.parametrize("chunk_pass", [1, 2], ids=["two-launch", "in-order"])
def test_chunk_passes_match_oracle(shape, opts, chunk_pass):
    """Chunk states carried by the two-launch form (chunk-end states for
    every chunk, then a passing launch) and by the in-order kernels (one
    workgroup per batch row, head and 64-state column block walking the
    chunks, column blocks of 64, 48 and 16 states): forward, final states and
    every gradient against the oracle, with and without initial states, z,
    D and dt_bias."""
    c = case(*shape, seed=sum(shape) + chunk_pass, **opts)
    check_ops(c, run_ops(c, chunk_pass=chunk_pass))


def test_chunk_passes_in_bf16_and_clamped():
    c = case(2, 130, 8, 64, 2, 64, seed=5, init=True, dtype=torch.bfloat16)
    for cp in (1, 2):
        check_ops(c, run_ops(c, chunk_pass=cp, limit=(0.05, 2.0)), limit=(0.05, 2.0), low=True)


def test_chunk_pass_must_be_known():
    c = case(1, 64, 2, 16, 1, 16)
    with pytest.raises(ValueError, match="chunk_pass"):
        run_ops(c, chunk_pass=3)


def test_head_block_must_divide_the_group():
    c = case(1, 64, 6, 16, 2, 16)
    with pytest.raises(ValueError, match="head_block"):
        run_ops(c, head_block=2)   # 3 heads per group


def test_opcheck_ssd_ops():
    c = case(1, 70, 2, 16, 1, 16, seed=6, init=True)
    d = {k: None if v is None else v.to(DEV) for k, v in c.items()}
    if d["D"] is not None and d["D"].dim() == 1:   # the operator takes D per channel
        d["D"] = d["D"][:, None].expand(d["x"].shape[2:]).contiguous()
    args = (d["x"], d["dt"], d["A"], d["B"], d["C"], d["D"], d["z"], d["dt_bias"], d["initial_states"],
            True, 0.0, float("inf"), True)
    torch.library.opcheck(torch.ops.mamba_cpu.ssd_fwd.default, args)
    out, fin, saved, ysave = torch.ops.mamba_cpu.ssd_fwd(*args)
    bargs = (torch.randn_like(out), torch.randn_like(fin)) + args[:12] + (saved, ysave)
    torch.library.opcheck(torch.ops.mamba_cpu.ssd_bwd.default, bargs)


@pytest.mark.parametrize("seqlen", [1, 17, 63, 64, 65, 128, 200])
@pytest.mark.parametrize("headdim,dstate", [(64, 128), (64, 64), (32, 128), (32, 64), (16, 16), (48, 80), (32, 112)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_tile_edges_of_every_product_form(seqlen, headdim, dstate, dtype):
    """The products in bf16 pieces (one to three per operand, by storage type)
    with chunks and tiles cut at every edge: lengths around the 64-step chunk and
    its 32-step halves, the exact 64 x 128 shape and ones padded in headdim,
    dstate or both, single and packed sequences. The pieces carry float32's 24
    bits, so without z (whose saved y is rounded to the storage type) the float32
    results of 16-bit inputs meet the float32 bounds too."""
    rng = np.random.default_rng(seqlen)
    for seq in (None, np.sort(rng.integers(0, 3, (2, seqlen)), axis=1).astype(np.int32)):
        c = case(2, seqlen, 4, headdim, 2, dstate, seed=seqlen + headdim, z=dtype == torch.float32, init=True,
                 dtype=dtype)
        got = run_ops(c, seq=seq)
        check_ops(c, got, low=dtype != torch.float32, seq=seq)
        if dtype != torch.float32:
            _, fin, g, W, V = got
            kw = dict(dt_softplus=True, seq_idx=seq)
            assert_close_report(fin, S.ssd_fwd(**c, **kw)[1], 1e-4, 1e-5, "final_states")
            wg = dict(zip(NAMES, S.ssd_bwd(**c, **kw, dout=W.float(), dfinal_states=V)))
            for name, i, atol in (("dt", 1, 1e-4), ("A", 2, 1e-3), ("D", 5, 1e-3), ("dt_bias", 7, 1e-3)):
                assert_close_report(g[i], wg[name], 1e-3, atol, f"d{name}")


def classes_match(got, want, name, rtol, atol):
    """Infinities of one sign and NaN where want has them, the rest within bounds."""
    got, want = got.detach().cpu().double().numpy(), np.asarray(want, dtype=np.float64)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want), err_msg=name)
    np.testing.assert_array_equal(np.where(np.isinf(got), got, 0), np.where(np.isinf(want), want, 0), err_msg=name)
    ok = np.isfinite(want)
    assert_close_report(got[ok], want[ok], rtol, atol, name)


END_SHAPES = [(1, 130, 4, 64, 1, 128), (1, 130, 4, 32, 2, 64), (1, 100, 4, 48, 1, 80), (2, 130, 8, 16, 1, 16)]


@pytest.mark.parametrize("shape", END_SHAPES, ids=lambda s: "p{}n{}".format(s[3], s[5]))
@pytest.mark.parametrize("chunk_pass", [1, 2], ids=["two-launch", "in-order"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_infinite_values_stay_infinite(shape, chunk_pass, dtype):
    """One infinite value, where the recurrence gives infinities of one sign and
    nothing else: an initial state (the outputs of its row, its final state), a
    final state's gradient (dx of its row, dB of its column), an input x or B
    (the final states it feeds) and an output gradient (the initial state's
    gradient of its row). Everything that the value does not reach is finite."""
    low = dtype != torch.float32
    inf = float("inf")
    otol, gtol = ((2e-2, 2e-2), (2e-2, 2e-2)) if low else ((1e-4, 1e-5), (1e-3, 1e-3))
    for where in ("initial_states", "V", "x", "B", "W"):
        c = case(*shape, seed=3, init=True, dtype=dtype, z=where != "V")
        c["A"] = c["A"] * 0.05   # no decay over the sequence underflows to 0
        gen = torch.Generator().manual_seed(1)
        W = torch.randn(c["x"].shape, generator=gen).to(dtype)
        V = torch.randn(c["initial_states"].shape, generator=gen)
        if where == "initial_states":
            c[where][0, 1, 5, 7] = inf
        elif where == "V":
            V[0, 1, 5, 7] = inf
        elif where == "W":
            W[0, 70, 1, 5] = inf
        else:
            c[where][(0, 70, 1, 5) if where == "x" else (0, 70, 0, 5)] = inf
        out, fin, g = run_with(c, W, V, chunk_pass)
        with np.errstate(invalid="ignore", over="ignore"):
            want, want_fin = S.ssd_fwd(**c, dt_softplus=True)
            wg = dict(zip(NAMES, S.ssd_bwd(**c, dt_softplus=True, dout=W.float(), dfinal_states=V)))
        print(where)
        if where in ("initial_states", "V"):
            classes_match(out, want, "out", *otol)
            for name in ("x", "B"):
                if where == "V" or name == "x":
                    classes_match(g[name], wg[name], f"d{name}", *gtol)
        if where != "W":
            classes_match(fin, want_fin, "final_states", *((1e-4, 1e-4) if not low else otol))
        if where in ("V", "W"):
            classes_match(g["initial_states"], wg["initial_states"], "dinitial_states", *gtol)


def run_with(c, W, V, chunk_pass):
    d = {k: None if v is None else v.to(DEV) for k, v in c.items()}
    args = tuple(d[k] for k in NAMES) + (True, 0.0, float("inf"))
    out, fin, saved, ysave = torch.ops.mamba_cpu.ssd_fwd(*args, True, 0, chunk_pass)
    g = torch.ops.mamba_cpu.ssd_bwd(W.to(DEV), V.to(DEV), *args, saved, ysave, 0, chunk_pass)
    torch.cuda.synchronize()
    return out, fin, dict(zip(NAMES, g))


@pytest.mark.parametrize("shape", END_SHAPES, ids=lambda s: "p{}n{}".format(s[3], s[5]))
@pytest.mark.parametrize("chunk_pass", [1, 2], ids=["two-launch", "in-order"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("scale", [1e-36, 1e-33, 1e37])
def test_values_near_the_ends_of_the_float32_range(shape, chunk_pass, dtype, scale):
    """The scan is linear in (x, initial states), and its gradients in (dout,
    dfinal_states): both scaled to the ends of float32's range, at the upper end
    with one value of each within 2^-8 of the largest, against the oracle. Bound:
    that of the unscaled problem, plus what a value split into bf16 pieces may be
    off at the small end, 2^-134 (ssd_pieces.h), four times."""
    low = dtype != torch.float32
    c = case(*shape, seed=4, init=True, dtype=dtype, z=False, D=None)
    c["A"] = c["A"] * 0.05   # what the decays leave stays of the inputs' size
    gen = torch.Generator().manual_seed(1)
    W = torch.randn(c["x"].shape, generator=gen).to(dtype)
    V = torch.randn(c["initial_states"].shape, generator=gen)
    big = scale > 1
    if big:   # sums of up to 128 products stay in range
        c["B"], c["C"] = (t * 2.0**-7 for t in (c["B"], c["C"]))
    scale = 2.0 ** round(math.log2(scale))
    for fwd in (True, False):
        cc, WW, VV = dict(c), W, V
        if fwd:
            cc["x"], cc["initial_states"] = c["x"] * scale, c["initial_states"] * scale
            WW, VV = W * 0, V * 0
            if big:
                cc["initial_states"][0, 1, 5, 7] = 3.4e38
                if not low:
                    cc["x"][0, 70, 1, 5] = 3.4e38
        else:
            WW, VV = W * scale, V * scale
            cc["x"], cc["initial_states"] = c["x"] * 2.0**-10, c["initial_states"] * 2.0**-10
            if big:
                VV[0, 1, 5, 7] = 3.4e38
                if not low:
                    WW[0, 70, 1, 5] = 3.4e38
        out, fin, g = run_with(cc, WW, VV, chunk_pass)
        if fwd:
            want, want_fin = S.ssd_fwd(**cc, dt_softplus=True)
            pairs = [("out", out, want, 2.0**-8 if low else 1e-5), ("final_states", fin, want_fin, 1e-5)]
        else:
            wg = dict(zip(NAMES, S.ssd_bwd(**cc, dt_softplus=True, dout=WW.float(), dfinal_states=VV)))
            pairs = [("dx", g["x"], wg["x"], 2.0**-8 if low else 1e-5),
                     ("dinitial_states", g["initial_states"], wg["initial_states"], 1e-5)]
        for name, got, ref, tol in pairs:
            got = got.double().cpu().numpy()
            assert np.isfinite(got).all(), name
            err = np.linalg.norm(got / scale - ref / scale) / np.linalg.norm(ref / scale)
            print(name, scale, err)
            assert err <= tol + 2.0**-132 / scale, (name, err)


@pytest.mark.parametrize("headdim,dstate", [(64, 128), (64, 64), (32, 128), (32, 64)])
@pytest.mark.parametrize("z", [False, True], ids=["noz", "z"])
@pytest.mark.parametrize("packed", [False, True])
def test_bf16_chunk_gradients_over_head_blocks(headdim, dstate, z, packed):
    """The chunk gradients of bf16 storage as training runs them: several heads
    to a workgroup (the next head's tiles prefetched, the shared tiles reused, dB
    and dC summed over the block), several chunks and a ragged tail, both ways of
    carrying the states, single and packed sequences. Without z (whose saved y is
    rounded to bf16) the float32 results meet the float32 bounds; each head's dx
    and ddt do not depend on the block."""
    seqlen = 200
    rng = np.random.default_rng(headdim + dstate)
    seq = np.sort(rng.integers(0, 4, (2, seqlen)), axis=1).astype(np.int32) if packed else None
    c = case(2, seqlen, 8, headdim, 1, dstate, seed=headdim + dstate + z, init=True, dtype=torch.bfloat16, z=z)
    want = wg = None
    for chunk_pass in (1, 2):
        first = None
        for hb in (1, 2, 4, 8):
            out, fin, g, W, V = run_ops(c, head_block=hb, chunk_pass=chunk_pass, seq=seq)
            if want is None:
                want = S.ssd_fwd(**c, dt_softplus=True, seq_idx=seq)
                wg = S.ssd_bwd(**c, dt_softplus=True, seq_idx=seq, dout=W.float(), dfinal_states=V)
            print(f" chunk_pass {chunk_pass} head_block {hb}")
            assert_close_report(out, want[0], 2e-2, 2e-2, "out")
            assert_close_report(fin, want[1], 1e-4, 1e-5, "final_states")
            for name, got, w in zip(NAMES, g, wg):
                if c[name] is None:
                    continue
                tol = (2e-2, 2e-2)
                if not z and name in ("dt", "A", "D", "dt_bias", "initial_states"):
                    tol = (1e-3, 1e-4 if name == "dt" else 1e-3)
                assert_close_report(got, w, *tol, f"d{name}")
            if first is None:
                first = (g[0], g[1])
            assert torch.equal(g[0], first[0]) and torch.equal(g[1], first[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("headdim,dstate", [(64, 128), (32, 64), (48, 80)])
def test_parameters_may_start_at_any_element(dtype, headdim, dstate):
    """A, D and dt_bias one element into their buffers give what aligned ones give,
    bit for bit."""
    c = case(1, 130, 4, headdim, 1, dstate, seed=headdim, dtype=dtype)
    gen = torch.Generator().manual_seed(1)
    W = torch.randn(c["x"].shape, generator=gen).to(dtype)
    V = torch.randn(1, 4, headdim, dstate, generator=gen)
    off = dict(c)
    for k in ("A", "D", "dt_bias"):
        buf = torch.zeros(c[k].numel() + 1, device=DEV)
        off[k] = buf[1:].view(c[k].shape)
        off[k].copy_(c[k])
        assert off[k].data_ptr() % 16 == 4
    (out, fin, g), (out1, fin1, g1) = run_with(c, W, V, 1), run_with(off, W, V, 1)
    assert torch.equal(out, out1) and torch.equal(fin, fin1)
    for k, v in g.items():
        assert (v is None and g1[k] is None) or torch.equal(v, g1[k]), k


@pytest.mark.parametrize("headdim,dstate", [(64, 128), (32, 64), (48, 80)])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("chunk_pass", [1, 2], ids=["two-launch", "in-order"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_an_infinite_input_leaves_the_rest_of_its_workgroup(headdim, dstate, packed, chunk_pass, dtype):
    """The last x of one head infinite, four heads to a workgroup: that workgroup does
    its work again in float32, and whatever the value does not enter (the other
    heads' outputs and gradients, its own head's earlier outputs) is the oracle's
    for a finite x, within the bounds of the storage type."""
    seqlen, low = 200, dtype != torch.float32
    rng = np.random.default_rng(headdim)
    seq = np.sort(rng.integers(0, 4, (1, seqlen)), axis=1).astype(np.int32) if packed else None
    c = case(1, seqlen, 4, headdim, 1, dstate, seed=headdim, init=True, dtype=dtype)
    bad = dict(c, x=c["x"].clone())
    bad["x"][0, -1, 1, 5] = float("inf")
    out, fin, g, W, V = run_ops(bad, head_block=4, chunk_pass=chunk_pass, seq=seq)
    want, want_fin = S.ssd_fwd(**c, dt_softplus=True, seq_idx=seq)
    wg = dict(zip(NAMES, S.ssd_bwd(**c, dt_softplus=True, seq_idx=seq, dout=W.float(), dfinal_states=V)))
    tol = (2e-2, 2e-2) if low else (1e-4, 1e-5)
    assert not torch.isfinite(out[0, -1, 1, 5]) and torch.isinf(fin[0, 1, 5]).all()
    out, fin = out.float().cpu().numpy(), fin.float().cpu().numpy()
    out[0, -1, 1, 5], fin[0, 1, 5] = want[0, -1, 1, 5], want_fin[0, 1, 5]
    assert_close_report(out, want, *tol, "out")
    assert_close_report(fin, want_fin, *tol, "final_states")
    rest = [0, 2, 3]
    for name in ("x", "dt", "z"):
        got = dict(zip(NAMES, g))[name].float().cpu().numpy()[:, :, rest]
        assert_close_report(got, wg[name][:, :, rest], *((2e-2, 2e-2) if low else (1e-3, 1e-4)), f"d{name}")
    for name, atol in (("A", 1e-3), ("D", 1e-3), ("dt_bias", 1e-3), ("initial_states", 1e-3)):
        got, ref = dict(zip(NAMES, g))[name].float().cpu().numpy(), wg[name]
        got, ref = (got[:, rest], ref[:, rest]) if name == "initial_states" else (got[rest], ref[rest])
        assert_close_report(got, ref, *((2e-2, 2e-2) if low else (1e-3, atol)), f"d{name}")


@pytest.mark.parametrize("headdim,dstate", [(64, 128), (48, 80)])
@pytest.mark.parametrize("chunk_pass", [1, 2], ids=["two-launch", "in-order"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_outputs_over_inputs_with_an_infinite_value(headdim, dstate, chunk_pass, dtype):
    """The C calls with every output over the input of its shape (out over x, the
    final states over the initial ones, dx over dout, dz over z, ddt over dt, dinit
    over dfinal), one x infinite, four heads to a workgroup: the other heads'
    results are those of separate buffers, and no workgroup does its work twice on
    what it has written. Bound: the storage type's, as the workgroups that do their
    work again add up in another order."""
    import ctypes

    from mamba_cpu import _C

    shape = (1, 200, 4, headdim, 1, dstate)
    low = dtype != torch.float32
    c = case(*shape, seed=headdim, init=True, dtype=dtype, z=True)
    c["x"][0, -1, 1, 5] = float("inf")
    gen = torch.Generator().manual_seed(1)
    W = torch.randn(c["x"].shape, generator=gen).to(dtype)
    V = torch.randn(c["initial_states"].shape, generator=gen)
    stream = torch.cuda.current_stream().cuda_stream

    def call(over):
        d = {k: v.to(DEV).contiguous() for k, v in c.items()}
        dout, dfin = W.to(DEV), V.to(DEV)
        a = _C.SsdArgs()
        for n in NAMES:
            setattr(a, n, d[n].data_ptr())
        a.batch, a.seqlen, a.nheads, a.headdim, a.ngroups, a.dstate = shape
        a.dtype = _C.MCPU_BF16 if low else _C.MCPU_F32
        a.dt_softplus, a.dt_limit_hi, a.head_block, a.chunk_pass = 1, float("inf"), 4, chunk_pass
        place = lambda t: t if over else torch.empty_like(t)  # noqa: E731
        saved = torch.empty(_C.lib.mcpu_ssd_saved_size(ctypes.byref(a)), dtype=torch.uint8, device=DEV)
        out, fin, y = place(d["x"]), place(d["initial_states"]), torch.empty_like(d["x"])
        a.out, a.final_states, a.ysave = out.data_ptr(), fin.data_ptr(), y.data_ptr()
        assert _C.lib.mcpu_ssd_fwd(ctypes.byref(a), saved.data_ptr(), saved.numel(), stream) == _C.MCPU_OK
        res = {"out": out.clone(), "final_states": fin.clone()}
        d["x"].copy_(c["x"])
        d["initial_states"].copy_(c["initial_states"])
        f32 = dict(dtype=torch.float32, device=DEV)
        g = {"dx": place(dout), "ddt": place(d["dt"]), "dz": place(d["z"]), "dinitial_states": place(dfin)}
        rest = {"dA": torch.empty(4, **f32), "dB": torch.empty(d["B"].shape, **f32),
                "dC": torch.empty(d["C"].shape, **f32), "dD": torch.empty(4, headdim, **f32),
                "ddt_bias": torch.empty(4, **f32)}
        a.dout, a.dfinal_states = dout.data_ptr(), dfin.data_ptr()
        for n, t in {**g, **rest}.items():
            setattr(a, n, t.data_ptr())
        ws = torch.empty(_C.lib.mcpu_ssd_bwd_workspace_size(ctypes.byref(a)), dtype=torch.uint8, device=DEV)
        assert _C.lib.mcpu_ssd_bwd(ctypes.byref(a), saved.data_ptr(), saved.numel(), ws.data_ptr(), ws.numel(),
                                   stream) == _C.MCPU_OK
        torch.cuda.synchronize()
        return {**res, **g}

    want, got = call(False), call(True)
    assert torch.isinf(want["final_states"][0, 1, 5]).all() and torch.isinf(got["final_states"][0, 1, 5]).all()
    rest = [0, 2, 3]
    for name, w in want.items():
        heads = (lambda t: t[:, rest]) if "states" in name else (lambda t: t[:, :, rest])
        assert torch.isfinite(heads(w)).all(), name
        assert_close_report(heads(got[name]).float(), heads(w).float().cpu().numpy(),
                            *((2e-2, 2e-2) if low else (1e-3, 1e-4)), name)
