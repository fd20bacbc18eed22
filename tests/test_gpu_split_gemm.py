"""fp32 products in three bf16 parts (csrc/split.h) against float64, at the edges of every tile.

Two bounds.  Element by element a float32 sum of k products is within k * 2^-24 * (|A| |B|) of the
exact one, however its terms are grouped; the parts hold all 24 bits and the dropped products are
below 2^-25 of theirs, inside the same bound.  That worst case would pass a product that lacks a
part, so the errors' root mean square (over everything, each row and each column) is bounded too:
sums over 32 k rounded once each, and eight more roundings where waves or slices meet, every one at
most 2^-25 of the sum, whose own size is |a_row| |b_col| / sqrt(k) for random signs.  A product
without lo parts is at 1e-6 of that, one without mid mid at 2e-7."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from card_playing_gym_amd import _native as nat
from card_playing_gym_amd.nn.kv_cache import stream_handle
from card_playing_gym_amd.nn.train import linear_nt, matmul_nn, matmul_tn
from card_playing_gym_amd.synthetic import StepPlan
from card_playing_gym_amd.nn.trunk import TrunkConfig
from tests.helpers import cache_pair, fill_prefixes, max_err, run_native, run_oracle, twins

pytestmark = pytest.mark.gpu


def bound(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    return a.shape[1] * 2.0**-24 * (a.double().abs() @ b.double().abs())


def assert_fp32(out: torch.Tensor, a: torch.Tensor, b: torch.Tensor, what: str = "") -> None:
    """`out` = a b as fp32 sums over k give it."""

    k, a, b = a.shape[1], a.double(), b.double()
    off = (out.double() - a @ b).abs()
    assert (off <= k * 2.0**-24 * (a.abs() @ b.abs())).all(), what
    z = off / (a.norm(dim=1)[:, None] * b.norm(dim=0)[None, :] / math.sqrt(k))
    bar = 2.0**-25 * math.sqrt(k / 32 + 8)
    for dims, slack in (((0, 1), 1.0), ((0,), 2.0), ((1,), 2.0)):
        rms = z.square().mean(dims).sqrt().max().item()
        few = 1.0 + 3.0 / math.sqrt(math.prod(z.shape[d] for d in dims))  # the spread of a mean of few squares
        assert rms <= slack * few * bar, (what, dims, rms / bar)


def linear(x, w):
    out = torch.empty((x.shape[0], w.shape[0]), device=x.device)
    nat.call("cg_linear", x.data_ptr(), w.data_ptr(), None, out.data_ptr(), x.shape[0], w.shape[0], x.shape[1],
             nat.CG_ACT_NONE, nat.CG_F32, stream_handle(x.device))
    return out


# 16 x 16 tiles, 32 x 32 tiles, staged 64- and 128-row tiles; odd rows, columns and k remainders.
@pytest.mark.parametrize("m, n, k", [(1, 1, 8), (17, 15, 40), (64, 512, 256), (515, 250, 264), (1023, 513, 256),
                                     (2049, 1027, 136), (8200, 1030, 72), (8193, 1024, 1024)])
def test_linear_is_fp32_at_every_tile(device, m, n, k):
    gen = torch.Generator(device=device).manual_seed(m + n + k)
    # magnitudes over forty binades: no part may be scaled away
    x = torch.randn((m, k), generator=gen, device=device) * torch.exp2(torch.randint(-20, 20, (m, 1), generator=gen, device=device).float())
    w = torch.randn((n, k), generator=gen, device=device)
    off = (linear(x, w).double() - x.double() @ w.double().t()).abs()
    assert (off <= bound(x, w.t())).all(), (off / bound(x, w.t())).max()
    assert_fp32(linear(x, w), x, w.t())


@pytest.mark.parametrize("m, n, k", [(64, 256, 256), (1024, 512, 256), (4096, 1024, 64)])
def test_non_finite_operands_behave_as_in_fp32(device, m, n, k):
    gen = torch.Generator(device=device).manual_seed(5)
    x, w = (torch.randn(s, generator=gen, device=device) for s in ((m, k), (n, k)))
    x[3, 5], x[4, 7], x[9, 0], x[m - 1, k - 1] = float("inf"), float("nan"), 3.4e38, -float("inf")
    w[7, 5], w[20, 30], w[n - 1, 0], w[:, 0] = 0.0, -float("inf"), 1.0, 1.0  # inf * 0 and a product past bf16's range
    got = linear(x, w)
    want = x.double().cpu().numpy() @ w.double().cpu().numpy().T
    want = torch.from_numpy(want.astype(np.float32)).to(device)
    assert torch.equal(got.isnan(), want.isnan())
    infinite = want.isinf()
    assert torch.equal(got.isinf(), infinite) and torch.equal(got[infinite], want[infinite])
    fine = want.isfinite()
    torch.testing.assert_close(got[fine], want[fine], rtol=1e-4, atol=1e-3)


# Operand layouts of the training products: k contiguous, rows contiguous, and neither (odd sizes).
@pytest.mark.parametrize("m, n, k", [(4, 4, 4), (128, 64, 32), (132, 260, 36), (129, 67, 33), (1000, 256, 1028),
                                     (13041, 256, 64), (40000, 256, 32), (2048, 40, 256), (9000, 384, 520)])
def test_training_products_are_fp32_in_every_layout(device, m, n, k):
    gen = torch.Generator(device=device).manual_seed(m * n + k)
    randn = lambda *s: torch.randn(s, generator=gen, device=device)  # noqa: E731
    x, w, y = randn(m, k), randn(n, k), randn(m, n)
    for op, a, b, shape in ((linear_nt, x, w, (m, n)), (matmul_nn, y, w, (m, k)), (matmul_tn, y, x, (n, k))):
        out = torch.empty(shape, device=device)
        op(a, b, out)
        left, right = {linear_nt: (a, b.t()), matmul_nn: (a, b), matmul_tn: (a.t(), b)}[op]
        off = (out.double() - left.double() @ right.double()).abs()
        assert (off <= bound(left, right)).all(), op.__name__
        assert_fp32(out, left, right, op.__name__)


# 2^-112 to 2^-126: the lowest part, then the middle one, would end below bf16's smallest number.
SMALL = [2.0**-112, 2.0**-118, 2.0**-124]


@pytest.mark.parametrize("small", SMALL)
@pytest.mark.parametrize("m, n, k", [(64, 512, 256), (515, 250, 264), (1023, 513, 256), (2049, 1027, 136), (8200, 1030, 72)])
def test_linear_of_small_operands(device, m, n, k, small):
    gen = torch.Generator(device=device).manual_seed(m + n + k)
    x, w = torch.randn((m, k), generator=gen, device=device), torch.randn((n, k), generator=gen, device=device)
    x = x.sign() * x.abs().clamp(min=0.25)  # (no subnormal values)
    x[: m // 2] *= small
    assert_fp32(linear(x, w), x, w.t())


@pytest.mark.parametrize("small", SMALL)
@pytest.mark.parametrize("m, n, k", [(132, 260, 36), (1300, 256, 1028), (4096, 64, 256), (13041, 256, 64)])
def test_training_products_of_small_operands(device, m, n, k, small):
    gen = torch.Generator(device=device).manual_seed(m * n + k)
    x, w, y = (torch.randn(s, generator=gen, device=device) for s in ((m, k), (n, k), (m, n)))
    x, y = (t.sign() * t.abs().clamp(min=0.25) * small for t in (x, y))
    for op, a, b, shape in ((linear_nt, x, w, (m, n)), (matmul_nn, y, w, (m, k)), (matmul_tn, y, x / small, (n, k))):
        out = torch.empty(shape, device=device)
        op(a, b, out)
        left, right = {linear_nt: (a, b.t()), matmul_nn: (a, b), matmul_tn: (a.t(), b)}[op]
        assert_fp32(out, left, right, op.__name__)


# Products of few rows, staged tiles, slices over k, and neither operand contiguous.
@pytest.mark.parametrize("m, n, k", [(132, 260, 36), (1300, 256, 1028), (4096, 64, 256), (2051, 66, 130)])
def test_training_products_with_non_finite_operands(device, m, n, k):
    gen = torch.Generator(device=device).manual_seed(m + k)
    x, w, y = (torch.randn(s, generator=gen, device=device) for s in ((m, k), (n, k), (m, n)))
    for t in (x, y):
        t[3, 5], t[4, 7], t[9, 0], t[m - 1, -1] = float("inf"), float("nan"), 3.4e38, -float("inf")
    w[7, 5], w[:, 0] = 0.0, 1.0  # inf * 0 and a product past bf16's range
    plain = torch.randn((m, n), generator=gen, device=device)
    for op, a, b, shape in ((linear_nt, x, w, (m, n)), (matmul_nn, y, w, (m, k)), (matmul_tn, plain, x, (n, k))):
        out = torch.empty(shape, device=device)
        op(a, b, out)
        left, right = {linear_nt: (a, b.t()), matmul_nn: (a, b), matmul_tn: (a.t(), b)}[op]
        want = torch.from_numpy((left.double().cpu().numpy() @ right.double().cpu().numpy()).astype(np.float32)).to(device)
        # (a finite sum past fp32's range may have been so on the way)
        near = want.abs() < 1e38
        assert torch.equal(out.isnan(), want.isnan()), op.__name__
        assert torch.equal(out[want.isinf()], want[want.isinf()]), op.__name__
        terms = torch.nan_to_num(left.double()).abs() @ torch.nan_to_num(right.double()).abs()
        off = (out.double() - want.double()).abs()
        assert (off <= k * 2.0**-23 * terms.clamp(max=1e39))[near].all(), op.__name__


@pytest.mark.parametrize("rows", [40, 1300])
def test_normalising_product_with_non_finite_rows(device, rows):
    """One infinite and one NaN residual row: those games' hidden states are NaN, all others as without them."""

    config = TrunkConfig(d_model=256, n_layers=2, n_heads=8, n_kv_heads=2, d_ff=512)
    model, _ = twins(config, "fp32", device)
    hidden = []
    for value in (0.0, float("inf")):
        cache, ref = cache_pair(config, rows, 16, torch.float32, device)
        rng = np.random.default_rng(rows)
        lengths, slots = rng.integers(1, 12, size=rows), rng.permutation(rows)
        fill_prefixes(cache, ref, lengths, slots, seed=1)
        plan = StepPlan(np.arange(rows) % 509, lengths, slots, np.arange(rows + 1), np.zeros(rows, dtype=np.int64))
        plan.tokens[:2] = 510, 511
        with torch.no_grad():
            model.embedding.weight[510].fill_(1.0)
            model.embedding.weight[511].fill_(1.0)
            model.embedding.weight[510, 3] += value
            model.embedding.weight[511, 3] += value - value
        hidden.append(run_native(model, cache, plan, device, "fp32", packed=False, rows=True)[0])
    assert hidden[1][:2].isnan().all()
    assert torch.equal(hidden[0][2:], hidden[1][2:])


@pytest.mark.parametrize("rows, d_model, d_ff", [(1, 256, 1024), (33, 256, 512), (130, 128, 264), (1300, 256, 1024),
                                                 (2100, 256, 512), (40, 512, 512)])
def test_fp32_step_with_the_normalising_product(device, rows, d_model, d_ff):
    """Decode waves on each side of where the QKV and up products normalise their own rows."""

    config = TrunkConfig(d_model=d_model, n_layers=2, n_heads=8, n_kv_heads=2, d_ff=d_ff)
    model, ref = twins(config, "fp32", device)
    native_cache, ref_cache = cache_pair(config, rows, 16, torch.float32, device)
    rng = np.random.default_rng(rows)
    lengths, slots = rng.integers(0, 12, size=rows), rng.permutation(rows)
    fill_prefixes(native_cache, ref_cache, lengths, slots, seed=1)
    plan = StepPlan(rng.integers(0, 512, size=rows), lengths, slots, np.arange(rows + 1), np.zeros(rows, dtype=np.int64))
    got = run_native(model, native_cache, plan, device, "fp32", packed=False, rows=True)
    want = run_oracle(ref, ref_cache, plan, rows=True)
    assert max(max_err(a, b) for a, b in zip(got, want)) <= 1e-4
