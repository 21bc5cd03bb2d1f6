"""selective_state_update on the GPU.

Mirrors the reference's tests/test_selective_state_update.py (L single steps
equal the full scan; Mamba-2 head layout equals the flattened Mamba-1 layout)
and adds direct comparisons with the float64 oracle for both layouts, grouped
B/C, a bf16 state and state_batch_indices (which the reference rejects).
Tolerance rtol/atol 1e-5 (float32).
"""

import numpy as np
import pytest
import torch

from oracle import numerics as O

from mamba_cpu import selective_scan_fn, selective_state_update

pytestmark = pytest.mark.gpu
DEV = "cuda"


def close(got, want, rtol, atol, name=""):
    np.testing.assert_allclose(got.detach().float().cpu().numpy().astype(np.float64), want,
                               rtol=rtol, atol=atol, err_msg=name)


def test_steps_match_full_scan():
    torch.manual_seed(0)
    batch, dim, seqlen, dstate = 2, 16, 10, 8
    u = torch.randn(batch, dim, seqlen, device=DEV)
    delta = torch.rand(batch, dim, seqlen, device=DEV) * 0.5
    A = -torch.rand(dim, dstate, device=DEV) - 0.5
    B = torch.randn(batch, dstate, seqlen, device=DEV)
    C = torch.randn(batch, dstate, seqlen, device=DEV)
    D = torch.randn(dim, device=DEV)
    z = torch.randn(batch, dim, seqlen, device=DEV)
    dt_bias = torch.rand(dim, device=DEV) * 0.1

    full, last = selective_scan_fn(u, delta, A, B, C, D, z, dt_bias, True, return_last_state=True)
    want, want_last = O.selective_scan_fwd(u, delta, A, B, C, D, z, dt_bias, True)

    state = torch.zeros(batch, dim, dstate, device=DEV)
    steps = [
        selective_state_update(
            state, u[..., t], delta[..., t], A, B[..., t], C[..., t], D, z[..., t], dt_bias, True
        )
        for t in range(seqlen)
    ]
    torch.testing.assert_close(torch.stack(steps, -1), full, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(state, last, rtol=1e-5, atol=1e-5)
    close(torch.stack(steps, -1), want, 1e-5, 1e-5)
    close(state, want_last, 1e-5, 1e-5)


def test_multihead_matches_flattened():
    # Mamba-2 layout with ngroups=1 is Mamba-1 with dim = nheads * headdim.
    torch.manual_seed(0)
    batch, nheads, headdim, dstate = 2, 4, 3, 8
    state = torch.randn(batch, nheads, headdim, dstate, device=DEV)
    x = torch.randn(batch, nheads, headdim, device=DEV)
    dt = torch.rand(batch, nheads, headdim, device=DEV)
    A = -torch.rand(nheads, headdim, dstate, device=DEV)
    B = torch.randn(batch, 1, dstate, device=DEV)
    C = torch.randn(batch, 1, dstate, device=DEV)
    D = torch.randn(nheads, headdim, device=DEV)

    flat_state = state.reshape(batch, -1, dstate).clone()
    out = selective_state_update(state, x, dt, A, B, C, D)
    flat_out = selective_state_update(
        flat_state, x.reshape(batch, -1), dt.reshape(batch, -1), A.reshape(-1, dstate),
        B[:, 0], C[:, 0], D.reshape(-1),
    )
    torch.testing.assert_close(out.reshape(batch, -1), flat_out)
    torch.testing.assert_close(state.reshape(batch, -1, dstate), flat_state)


@pytest.mark.parametrize("multihead", [False, True])
def test_matches_oracle(multihead):
    torch.manual_seed(0)
    b, n = 2, 16
    lead = (4, 8) if multihead else (32,)
    state = torch.randn(b, *lead, n, device=DEV)
    x, dt, z = (torch.randn(b, *lead, device=DEV), torch.rand(b, *lead, device=DEV),
                torch.randn(b, *lead, device=DEV))
    A = -torch.rand(*lead, n, device=DEV) - 0.5
    B = torch.randn(b, 2, n, device=DEV) if multihead else torch.randn(b, n, device=DEV)
    C = torch.randn_like(B)
    D, dt_bias = torch.randn(*lead, device=DEV), torch.rand(*lead, device=DEV)
    want, want_state = O.selective_state_update(state, x, dt, A, B, C, D, z, dt_bias, True)
    out = selective_state_update(state, x, dt, A, B, C, D, z, dt_bias, True)
    close(out, want, 1e-5, 1e-5, "out")
    close(state, want_state, 1e-5, 1e-5, "state")


def test_bf16_state_and_inputs():
    torch.manual_seed(0)
    b, d, n = 3, 40, 16
    state = torch.randn(b, d, n, device=DEV).bfloat16()
    x, dt, z = (torch.randn(b, d, device=DEV).bfloat16(), torch.rand(b, d, device=DEV).bfloat16(),
                torch.randn(b, d, device=DEV).bfloat16())
    A = -torch.rand(d, n, device=DEV) - 0.5
    B, C = torch.randn(b, n, device=DEV), torch.randn(b, n, device=DEV)
    D = torch.randn(d, device=DEV)
    want, want_state = O.selective_state_update(state, x, dt, A, B, C, D, z, None, True)
    out = selective_state_update(state, x, dt, A, B, C, D, z, None, True)
    assert out.dtype == torch.bfloat16 and state.dtype == torch.bfloat16
    close(out, want, 2e-2, 2e-2)
    close(state, want_state, 2e-2, 2e-2)


@pytest.mark.parametrize("heads", [False, True])
def test_state_batch_indices_match_oracle(heads):
    """state_batch_indices (rows of a larger state, one out of range), which
    the reference rejects, against the oracle's restatement of mamba_ssm's
    semantics."""
    torch.manual_seed(5)
    b, h, p, n, rows = 3, 2, 8, 16, 7
    lead = (b, h, p) if heads else (b, h * p)
    prm = (h, p) if heads else (h * p,)
    state = torch.randn((rows,) + lead[1:] + (n,), device=DEV)
    x, z = torch.randn(lead, device=DEV), torch.randn(lead, device=DEV)
    dt = torch.rand(lead, device=DEV)
    A = -torch.rand(prm + (n,), device=DEV) - 0.5
    B = torch.randn((b, 1, n) if heads else (b, n), device=DEV)
    C = torch.randn((b, 1, n) if heads else (b, n), device=DEV)
    D, dtb = torch.randn(prm, device=DEV), torch.rand(prm, device=DEV) * 0.1
    idx = torch.tensor([5, 1, -1], dtype=torch.int32, device=DEV)
    want, want_state = O.selective_state_update(state, x, dt, A, B, C, D, z, dtb, True,
                                                state_batch_indices=idx.cpu().numpy())
    out = selective_state_update(state, x, dt, A, B, C, D, z, dtb, True, state_batch_indices=idx)
    close(out, want, 1e-5, 1e-5, "out")
    close(state, want_state, 1e-5, 1e-5, "state")


def test_rejects_malformed_state_batch_indices():
    s = torch.zeros(1, 4, 2, device=DEV)
    with pytest.raises(ValueError):
        selective_state_update(s, torch.zeros(1, 4, device=DEV), torch.zeros(1, 4, device=DEV),
                               torch.zeros(4, 2, device=DEV), torch.zeros(1, 2, device=DEV),
                               torch.zeros(1, 2, device=DEV),
                               state_batch_indices=torch.zeros(2, dtype=torch.int32, device=DEV))


@pytest.mark.parametrize("n", [8, 16, 24, 32, 48, 64, 96, 100, 128, 200, 256])
@pytest.mark.parametrize("sdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("bcdt", [torch.float32, torch.bfloat16, torch.float16])
def test_state_sizes_types_and_unaligned_views(n, sdt, bcdt):
    """Every lane layout (vectors at 16, 32, 64, 128 and 256 states, one state
    per lane otherwise) with B and C as stored, on views that start one element
    into their buffers, a ragged number of rows, and A both full and expanded
    from per-head values. Bounds: float32 as above (out sums up to 256 terms:
    twice that); 16-bit values carry one rounding, at most 2^-8 of the value."""
    torch.manual_seed(n)
    b, h, p = 3, 2, 19
    state = torch.randn(b * h * p * n + 1, device=DEV).to(sdt)[1:].view(b, h, p, n)
    xdt = torch.float32 if sdt == torch.float32 else bcdt  # with a 16-bit state, B and C of x's type
    x, dt, z = (f(b, h, p, device=DEV).to(xdt) for f in (torch.randn, torch.rand, torch.randn))
    bc = torch.randn(b, 2 * n + 1, device=DEV).to(bcdt)
    B, C = bc[:, 1:n + 1].unsqueeze(1), bc[:, n + 1:].unsqueeze(1)
    D, dtb = torch.randn(h, p, device=DEV), torch.rand(h, p, device=DEV) * 0.1
    for A in (-torch.rand(h, p, n, device=DEV) - 0.5, (-torch.rand(h, device=DEV))[:, None, None].expand(h, p, n)):
        want, want_state = O.selective_state_update(state, x, dt, A, B, C, D, z, dtb, True)
        out = selective_state_update(state, x, dt, A, B, C, D, z, dtb, True)
        close(out, want, 2e-5 if xdt == torch.float32 else 2.0**-8, 2e-5, "out")
        tol = 1e-5 if sdt == torch.float32 else 2.0**-8
        close(state, want_state, tol, 1e-5, "state")


@pytest.mark.parametrize("n,rows_n", [(16, 17), (32, 33), (64, 65), (128, 129), (256, 200)])
@pytest.mark.parametrize("xdt,sdt", [(torch.float32, torch.float32), (torch.bfloat16, torch.float32),
                                     (torch.bfloat16, torch.bfloat16)])
def test_vector_and_row_layouts_sum_alike(n, rows_n, xdt, sdt):
    """<state, C> is one sum whatever layout the size takes: 16 chains over the
    states j, j + 16, ..., added as a tree (what the fused decode steps compute,
    so that their tokens are the unfused model's). Each vector size against a
    neighbouring size of the one-state-per-lane layout, the extra states all
    zero: outputs and states bitwise equal."""
    torch.manual_seed(n)
    b, h, p, m = 3, 4, 21, min(n, rows_n)
    state = torch.randn(b, h, p, m, device=DEV).to(sdt)
    x, dt, z = (f(b, h, p, device=DEV).to(xdt) for f in (torch.randn, torch.rand, torch.randn))
    A = -torch.rand(h, p, m, device=DEV) - 0.5
    B, C = (torch.randn(b, 2, m, device=DEV).to(xdt) for _ in range(2))
    D, dtb = torch.randn(h, p, device=DEV), torch.rand(h, p, device=DEV) * 0.1
    got = []
    for size in (n, rows_n):
        s, a, bb, c = (torch.nn.functional.pad(t, (0, size - m)) for t in (state, A, B, C))
        out = selective_state_update(s, x, dt, a, bb, c, D, z, dtb, True)
        got.append((out, s[..., :m]))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("n", [16, 24, 64, 100, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("groups", [1, 3])
def test_float32_state_with_16_bit_inputs(n, dtype, groups):
    """16-bit x, dt, z, B and C beside a float32 state (a 16-bit model's decode):
    B and C are read as stored, one row per group of heads, so the state keeps the
    float32 bound against the oracle on the same rounded inputs; the output
    carries one rounding of its storage type."""
    torch.manual_seed(n + groups)
    b, h, p = 3, 6, 19
    state = torch.randn(b, h, p, n, device=DEV)
    x, dt, z = (f(b, h, p, device=DEV).to(dtype) for f in (torch.randn, torch.rand, torch.randn))
    B, C = (torch.randn(b, n, groups, device=DEV).to(dtype).transpose(1, 2) for _ in range(2))
    A = -torch.rand(h, p, n, device=DEV) - 0.5
    D, dtb = torch.randn(h, p, device=DEV), torch.rand(h, p, device=DEV) * 0.1
    for Bc, Cc in ((B, C), (B.contiguous(), C.contiguous())):
        s = state.clone()
        want, want_state = O.selective_state_update(s, x, dt, A, Bc, Cc, D, z, dtb, True)
        out = selective_state_update(s, x, dt, A, Bc, Cc, D, z, dtb, True)
        close(out, want, 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11, 2e-5, "out")
        close(s, want_state, 1e-5, 1e-5, "state")
