"""GPU parity of the MSA-stack ops against the CPU oracle (gfx950 only).

Same conventions as the pair ops: seeded fp32 draws rounded to bf16 feed both sides, the
oracle runs in fp64 on the module's fp32 parameters, the bare update (``residual=False``) is
compared with rel-RMS <= 1e-2 and max-abs <= 4e-2 * max|ref|, and masking is exact: the
outputs of valid tokens are bitwise independent of the content at masked keys.
"""

from __future__ import annotations

import pytest
import torch

from foldforge_amd import _native, factories
from foldforge_amd.trunk import randomise
from oracle import pairstack as ps
from tests.hip_calls import hip_delta, hip_forward

pytestmark = pytest.mark.gpu

REL_RMS = 1e-2
MAX_ABS = 4e-2


@pytest.fixture(scope="module", autouse=True)
def _device():
    if not torch.cuda.is_available():
        pytest.skip("no GPU in this environment")
    from foldforge_amd import _native

    _native.lib()


def _check(got: torch.Tensor, want: torch.Tensor, what: str) -> None:
    rr = ps.rel_rms(got, want)
    ma = ps.max_abs(got, want)
    ref = want.abs().max().item()
    print(f"{what}: rel_rms={rr:.2e} max_abs={ma:.2e} max_ref={ref:.2e}", flush=True)
    assert rr <= REL_RMS, f"{what}: rel-RMS {rr:.3e}"
    assert ma <= MAX_ABS * ref, f"{what}: max-abs {ma:.3e} vs {MAX_ABS} * {ref:.3e}"


def _inputs(depth: int, n: int, cm: int, lengths, seed: int):
    g = torch.Generator().manual_seed(seed)
    batch = len(lengths)
    m = torch.randn(batch, depth, n, cm, generator=g).bfloat16()
    z = torch.randn(batch, n, n, 128, generator=g).bfloat16()
    mask = torch.zeros(batch, n, dtype=torch.bool)
    for b, length in enumerate(lengths):
        mask[b, :length] = True
    return m, z, mask


def _pwa(cm: int, heads: int, dh: int | None, seed: int):
    m = randomise(factories.msa_pair_weighted_averaging(cm, 128, heads, dh), seed=seed).cuda()
    m.set_backend("hip")
    return m


# d_head 32 is the released models' width; 24 ends MSA rows inside a 128-row output tile; 12 (not a
# multiple of 8) takes the unstaged 8-byte epilogue
@pytest.mark.parametrize("cm,heads,dh", [(64, 8, None), (64, 4, 16), (128, 8, 8), (64, 8, 32), (64, 8, 24),
                                        (64, 16, 12)])
@pytest.mark.parametrize("depth,n,lengths", [(5, 64, [64]), (7, 100, [77]), (3, 130, [130, 41])])
def test_msa_pair_weighted_averaging_matches_oracle(cm, heads, dh, depth, n, lengths):
    msa, z, mask = _inputs(depth, n, cm, lengths, seed=n + cm + heads)
    mod = _pwa(cm, heads, dh, seed=cm + heads)
    assert mod.unsupported(msa.cuda(), z.cuda(), mask.cuda()) is None
    got = hip_delta(mod, msa.cuda(), z.cuda(), mask.cuda()).cpu()
    want = ps.msa_pair_weighted_averaging(msa, z, mask, mod.state_dict(), n_head=heads,
                                          dtype=torch.float64) - msa.double()
    _check(got, want, f"msa_pwa c_m={cm} heads={heads}x{mod.d_hidden} S={depth} n={n} lengths={lengths}")
    full = hip_forward(mod, msa.cuda(), z.cuda(), mask.cuda()).cpu()
    _check(full, want + msa.double(), "msa_pwa residual")


@pytest.mark.parametrize("dh", [8, 16, 32])
@pytest.mark.parametrize("depth,n,lengths", [(1, 1, [1]), (5, 33, [20]), (2, 129, [129, 77]), (9, 200, [200])])
def test_msa_pair_weighted_averaging_of_eight_heads_at_tile_edges(dh, depth, n, lengths):
    """The one-kernel form: MSA rows that do not fill an operand tile (4, 2 or 1 rows), queries past
    the last 32- and 128-query tile."""
    msa, z, mask = _inputs(depth, n, 64, lengths, seed=n + dh)
    mod = _pwa(64, 8, dh, seed=dh + depth)
    want = ps.msa_pair_weighted_averaging(msa, z, mask, mod.state_dict(), n_head=8,
                                          dtype=torch.float64) - msa.double()
    _check(hip_delta(mod, msa.cuda(), z.cuda(), mask.cuda()).cpu(), want, f"msa_pwa 8x{dh} S={depth} n={n}")
    _check(hip_forward(mod, msa.cuda(), z.cuda(), mask.cuda()).cpu(), want + msa.double(), "msa_pwa residual")


@pytest.mark.parametrize("dh", [8, 16, 32])
def test_msa_pair_weighted_averaging_of_eight_heads_rounds_the_gated_average_once(dh):
    """The one-kernel form against its own roundings in 64 bits: values, weights, gate, gate times
    average, the projections' weights and the update in bf16, nothing else. What is left are values
    that fp32 and the hardware's exp2 and reciprocal put on the other side of a rounding, 1 to 2e-4 of
    the update. The update's own rounding (steps u of 5.5e-3 of a value on average) moves a value of
    error e by u with probability e / u, so e shows as sqrt(e u): 0.7 to 1.05e-3, and a second
    rounding of the average (e = 1.66e-3) as 3e-3. The bound lies between the two."""
    depth, n = 9, 200
    msa, z, mask = _inputs(depth, n, 64, [180], seed=dh)
    mod = _pwa(64, 8, dh, seed=dh)
    p = {k: v.double().cpu() for k, v in mod.state_dict().items()}

    def r(x):
        return x.bfloat16().double()

    def norm(x, name):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], p[name + ".weight"], p.get(name + ".bias"), 1e-5)

    x = norm(msa.double(), "ln_msa")[0]  # [S, n, 64]
    logits = (norm(z.double(), "ln_pair") @ p["to_bias.weight"].T)[0].permute(2, 0, 1)  # [8, i, j]
    w = r(logits.masked_fill(~mask[0], float("-inf")).softmax(dim=-1))
    v = r(x @ r(p["to_value.weight"]).T).unflatten(-1, (8, dh))  # [S, j, 8, dh]
    gate = r(torch.sigmoid(x @ r(p["to_gate.weight"]).T))
    average = torch.stack([w[h] @ v[:, :, h] for h in range(8)], dim=2).flatten(2)  # [S, i, 8 dh]
    want = r(r(gate * average) @ r(p["to_out.weight"]).T)
    got = hip_delta(mod, msa.cuda(), z.cuda(), mask.cuda()).cpu()[0].double()
    err = ((got - want).norm() / want.norm()).item()
    print(f"msa_pwa 8x{dh} against its own roundings: {err:.2e}", flush=True)
    assert err <= 1.8e-3


@pytest.mark.parametrize("heads,dh", [(1, 256), (3, 64)])
@pytest.mark.parametrize("n", [1, 31, 65])
def test_msa_pair_weighted_averaging_wide_heads_and_broken_key_runs(heads, dh, n):
    """Heads of 64 channels and more, and tokens that end inside a 32-key run of the values."""
    msa, z, mask = _inputs(3, n, 64, [n], seed=n + dh)
    mod = _pwa(64, heads, dh, seed=dh)
    got = hip_delta(mod, msa.cuda(), z.cuda(), mask.cuda()).cpu()
    want = ps.msa_pair_weighted_averaging(msa, z, mask, mod.state_dict(), n_head=heads,
                                          dtype=torch.float64) - msa.double()
    _check(got, want, f"msa_pwa {heads}x{dh} n={n}")


@pytest.mark.parametrize("cm,heads,dh", [(192, 8, 24), (384, 16, 12), (64, 8, 24)])
@pytest.mark.parametrize("n", [1, 33, 65])
def test_msa_pair_weighted_averaging_does_not_read_what_it_does_not_write(cm, heads, dh, n):
    """On a workspace of NaN the update is that of any other workspace. The values are its first piece,
    ``[heads][S][dh][n padded to 64]``: MSA widths outside the streaming projection's (64, 128, 256)
    leave the padding keys alone instead of projecting copies of the last token."""
    depth = 3
    msa, z, mask = (t.cuda() for t in _inputs(depth, n, cm, [n], seed=n + dh))
    mod = _pwa(cm, heads, dh, seed=dh)
    want = hip_delta(mod, msa, z, mask)
    lib, out = _native.lib(), torch.empty_like(msa)
    size = lib.ffk_msa_pair_weighted_averaging_workspace(1, depth, n, cm, 128, heads, dh)
    ws = torch.full((size,), 255, dtype=torch.uint8, device="cuda")
    p = dict(mod.named_parameters())
    names = ("ln_msa.weight", "ln_msa.bias", "ln_pair.weight", "to_bias.weight", "to_value.weight",
             "to_gate.weight", "to_out.weight")
    status = lib.ffk_msa_pair_weighted_averaging(
        msa.data_ptr(), z.data_ptr(), mask.data_ptr(), *(p[k].data_ptr() for k in names), out.data_ptr(),
        ws.data_ptr(), size, 1, depth, n, cm, 128, heads, dh, 0, mod.ln_msa.eps, mod.ln_pair.eps,
        torch.cuda.current_stream().cuda_stream)
    assert status == 0, lib.ffk_last_error().decode()
    assert torch.equal(out, want)
    np = (n + 63) // 64 * 64
    vt = ws[:heads * depth * dh * np * 2].view(torch.bfloat16).view(heads, depth, dh, np)
    assert torch.isfinite(vt[..., :n].float()).all()
    if cm not in (64, 128, 256):
        assert torch.isnan(vt[..., n:].float()).all()


def test_msa_pair_weighted_averaging_masking_is_exact_and_empty_rows_are_zero():
    depth, n, length = 4, 96, 61
    msa, z, mask = _inputs(depth, n, 64, [length, 0], seed=11)
    mod = _pwa(64, 8, None, seed=12)
    a = hip_delta(mod, msa.cuda(), z.cuda(), mask.cuda()).cpu()
    msa2, z2 = msa.clone(), z.clone()
    msa2[0, :, length:] = 5.0
    z2[0, length:] = -4.0
    z2[0, :, length:] = 9.0
    b = hip_delta(mod, msa2.cuda(), z2.cuda(), mask.cuda()).cpu()
    assert torch.equal(a[0, :, :length], b[0, :, :length])
    assert torch.equal(a[1], torch.zeros_like(a[1]))  # no valid key: zero update


def test_msa_pair_weighted_averaging_full_size_is_finite_and_deterministic():
    depth, n = 512, 384
    msa, z, mask = _inputs(depth, n, 64, [371], seed=21)
    mod = _pwa(64, 8, None, seed=22)
    mc, zc, kc = msa.cuda(), z.cuda(), mask.cuda()
    a = mod(mc, zc, kc)
    b = mod(mc, zc, kc)
    assert torch.isfinite(a.float()).all()
    assert torch.equal(a, b)


@pytest.mark.parametrize("options", [{}, {"parallel": True, "opm_groups": 8, "opm_channel": 8}])
def test_msa_block_overlapped_tracks_are_bitwise_sequential(options):
    """After the outer product mean the MSA block runs its MSA track on a second stream beside
    the pair track: the results equal the sequential order bit for bit (the AF3 order and
    Chai-1's parallel stages with the grouped outer product mean), with every op on ``hip``."""
    from foldforge_amd import dispatch

    n, length, depth, cm, c = 96, 83, 41, 64, 128
    block = randomise(factories.msa_block(cm, c, 4, **options), seed=12).cuda()
    block.set_backend("hip")
    dispatch.set_refusal(block, "error")
    g = torch.Generator().manual_seed(13)
    msa = torch.randn(depth, n, cm, generator=g).bfloat16().cuda()
    z = torch.randn(n, n, c, generator=g).bfloat16().cuda()
    tokens = torch.zeros(n, dtype=torch.bool)
    tokens[:length] = True
    msa_mask = ((torch.rand(depth, n, generator=g) > 0.2) & tokens[None]).float()
    msa_mask[0] = tokens.float()
    pair_mask = (tokens[:, None] & tokens[None, :]).float()
    msa_mask, pair_mask = msa_mask.cuda(), pair_mask.cuda()
    with torch.no_grad():
        block.overlap_tracks = False
        want = block(msa, z, msa_mask, pair_mask)
        block.overlap_tracks = True
        got = block(msa, z, msa_mask, pair_mask)
        again = block(msa, z, msa_mask, pair_mask)
    torch.cuda.synchronize()
    assert dispatch.served_count(block, "hip") == 3 * 8
    for a, b, r in zip(got, want, again):
        assert torch.equal(a, b) and torch.equal(r, b)
