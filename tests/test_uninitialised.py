"""No result depends on what memory held before: with every allocation filled with NaNs the operators
give the bits they give over zeros."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _scan(batch, dim, length, dstate, groups, act=torch.float32):
    g = torch.Generator().manual_seed(dim + length)

    def r(*shape, dtype=act):
        return torch.randn(shape, generator=g).to(dtype)

    leaves = [r(batch, dim, length), r(batch, dim, length, dtype=torch.float32),
              -r(dim, dstate, dtype=torch.float32).abs() - 0.1, r(batch, groups, dstate, length),
              r(batch, groups, dstate, length), r(dim, dtype=torch.float32), r(batch, dim, length),
              r(dim, dtype=torch.float32)]

    def call(u, dt, A, B, C, D, z, bias):
        from metal_kernelops import selective_scan
        return (selective_scan(u, dt, A, B, C, D, z, bias, True),)

    return leaves, call


def _ssd(batch, length, heads, headdim, groups, dstate, act):
    g = torch.Generator().manual_seed(length)

    def r(*shape, dtype=act):
        return torch.randn(shape, generator=g).to(dtype)

    leaves = [r(batch, length, heads, headdim), r(batch, length, heads, dtype=torch.float32),
              -r(heads, dtype=torch.float32).abs() - 0.1, r(batch, length, groups, dstate),
              r(batch, length, groups, dstate), r(heads, dtype=torch.float32), r(batch, length, heads, headdim)]

    def call(x, dt, A, B, C, D, z):
        from metal_kernelops.cv import mamba2_chunk_scan
        return mamba2_chunk_scan(x, dt, A, B, C, D=D, z=z, dt_softplus=True)

    return leaves, call


def _conv(batch, channels, length, width, act):
    g = torch.Generator().manual_seed(length)
    leaves = [torch.randn(s, generator=g).to(act) for s in ((batch, channels, length), (channels, width), (channels,))]

    def call(x, w, b):
        from metal_kernelops.cv import causal_conv1d_fn
        return (causal_conv1d_fn(x, w, b, "silu"),)

    return leaves, call


def _norm(rows, features, group):
    g = torch.Generator().manual_seed(rows)
    leaves = [torch.randn(s, generator=g) for s in ((rows, features), (features,), (features,), (rows, features))]

    def call(x, w, b, z):
        from metal_kernelops.cv import rmsnorm_gated
        return (rmsnorm_gated(x, w, b, z, group_size=group),)

    return leaves, call


CASES = {
    # lane per (channel, state): whole and ragged lengths, padded states, one and several time runs
    "scan 2x16x48": _scan(2, 16, 48, 16, 2), "scan 1x12x331": _scan(1, 12, 331, 5, 3),
    "scan 1x8x1043": _scan(1, 8, 1043, 16, 1, torch.bfloat16),
    # lane per channel: 32, 20 and 16 states, wavefronts inside a group and across groups, ragged ends
    "scan 1x128x200 n32": _scan(1, 128, 200, 32, 1), "scan 2x64x97 n20": _scan(2, 64, 97, 20, 1),
    "scan 2x24x97 n32": _scan(2, 24, 97, 32, 3), "scan 2x9x203 n16": _scan(2, 9, 203, 16, 3),
    "scan 1x6x1000 n16": _scan(1, 6, 1000, 16, 2, torch.bfloat16),
    "ssd f32": _ssd(2, 133, 4, 24, 2, 40, torch.float32), "ssd bf16": _ssd(1, 300, 4, 64, 1, 128, torch.bfloat16),
    "ssd bf16 long": _ssd(1, 1100, 2, 64, 1, 128, torch.bfloat16), "ssd f16": _ssd(2, 77, 2, 32, 1, 64, torch.float16),
    "conv": _conv(2, 3, 1003, 4, torch.float32), "conv bf16": _conv(1, 5, 520, 3, torch.bfloat16),
    "norm": _norm(37, 320, 64), "norm wide": _norm(5, 9000, 9000),
}


@pytest.mark.parametrize("name", CASES)
def test_results_do_not_depend_on_old_memory(name):
    leaves, call = CASES[name]

    def run(fill):
        args = [t.to(DEV).requires_grad_(True) for t in leaves]
        before = torch.are_deterministic_algorithms_enabled(), torch.utils.deterministic.fill_uninitialized_memory
        # deterministic mode fills what torch.empty allocates: NaN, or 0xff for bytes (a NaN too)
        torch.use_deterministic_algorithms(fill)
        torch.utils.deterministic.fill_uninitialized_memory = fill
        try:
            outs = call(*args)
            grads = torch.autograd.grad(outs, args, [torch.ones_like(o) for o in outs])
        finally:
            torch.use_deterministic_algorithms(before[0])
            torch.utils.deterministic.fill_uninitialized_memory = before[1]
        return [t.detach() for t in outs] + list(grads)

    from metal_kernelops import _native as nat
    plain_workspace = nat.workspace
    nat.workspace = lambda nbytes, device: plain_workspace(nbytes, device).zero_()
    try:
        clean = run(False)
    finally:
        nat.workspace = plain_workspace
    for k, (a, b) in enumerate(zip(clean, run(True))):
        assert torch.isfinite(b.float()).all(), k
        assert torch.equal(a, b), k
