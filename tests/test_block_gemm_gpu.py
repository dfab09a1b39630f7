"""The products of tiles of several shapes (``csrc/kernels/block_gemm.hip``) against 64 bits."""

import pytest
import torch

from vllm_production_stack_amd import ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _rand(*shape, std=1.0):
    return torch.randn(*shape, device="cuda", dtype=torch.float32).mul_(std).to(BF)


def _close(got, want, terms):
    """One rounding to 16 bits, and 32-bit sums of ``terms`` products: 2^-8 of the value and a part of the sum's size."""
    err = (got.double() - want).abs()
    assert bool((err <= want.abs() * 2 ** -8 + 1e-6 * terms ** 0.5).all()), err.max().item()


# a row more and less than tiles of 64, 96, 128 and 192 rows; columns that end inside a tile; one chunk of the reduction, fewer than the
# ring holds, and many; sizes whose costs choose each of the shapes
@pytest.mark.parametrize("m,n,k", [(1, 8, 64), (63, 64, 64), (65, 200, 128), (97, 392, 192), (129, 136, 256), (193, 768, 320),
                                   (1500, 512, 512), (1500, 768, 3072), (3000, 768, 3072), (9000, 768, 3072), (12000, 768, 768),
                                   (6000, 2048, 512)])
@pytest.mark.parametrize("gelu", [False, True])
def test_products_and_epilogues(m, n, k, gelu):
    torch.manual_seed(m + n + k)
    x, w, b, r = _rand(1, m, k), _rand(n, k, std=k ** -0.5), _rand(n), _rand(1, m, n)
    y = x.double() @ w.double().t()
    act = (lambda v: torch.nn.functional.gelu(v)) if gelu else (lambda v: v)
    _close(ops.block_linear(x, [w], [None], gelu), act(y), k)
    _close(ops.block_linear(x, [w], [b], gelu), act(y + b.double()), k)
    want = act(y + b.double()) + r.double()
    _close(ops.block_linear(x, [w], [b], gelu, residual=r), want, k)
    _close(ops.block_linear(x, [w], [b], gelu, residual=r, out=r), want, k)  # in place


def test_three_weights_side_by_side():
    x, ws, bs = _rand(2, 301, 192), [_rand(72, 192, std=0.1) for _ in range(3)], [_rand(72), None, _rand(72)]
    got = ops.block_linear(x, ws, bs)
    want = torch.cat([x.double() @ w.double().t() + (0 if b is None else b.double()) for w, b in zip(ws, bs)], dim=-1)
    _close(got, want, 192)


@pytest.mark.parametrize("stride,t", [(1, 50), (2, 51), (2, 64)])
def test_overlapping_rows_and_rows_of_batches(stride, t):
    """An unfolded convolution: rows that overlap, batches apart, a shared residual, an output with rows between the batches."""
    torch.manual_seed(t)
    b, c, n = 3, 64, 40
    x, w, bias, pos = _rand(b, t + 2, c), _rand(n, 3 * c, std=0.1), _rand(n), _rand(t, n)
    out_t = (t - 1) // stride + 1
    cols = x.as_strided((b, out_t, 3 * c), ((t + 2) * c, stride * c, 1))
    buf = torch.full((b, out_t + 2, n), 7.0, dtype=BF, device="cuda")
    got = ops.block_linear(cols, [w], [bias], True, residual=pos[:out_t], out=buf[:, 1:-1])
    want = torch.nn.functional.gelu(cols.double() @ w.double().t() + bias.double()) + pos[:out_t].double()
    _close(got, want, 3 * c)
    assert bool((buf[:, 0] == 7).all()) and bool((buf[:, -1] == 7).all())


def test_gelu_over_its_range():
    """Values far out on both sides, infinities and NaN: the reduction passes them through (weight 1 in one place)."""
    v = torch.cat([torch.linspace(-14, 14, 8185), torch.tensor([float("inf"), float("-inf"), float("nan"), 0.0, -0.0, 3e38, -3e38])])
    x = torch.zeros(1, v.numel(), 64, device="cuda", dtype=BF)
    x[0, :, 0] = v.to(BF).cuda()
    w = torch.zeros(8, 64, device="cuda", dtype=BF)
    w[:, 0] = 1
    got, z = ops.block_linear(x, [w], [None], True)[0].double(), x[0, :, :1].double()
    want = (z * 0.5 * torch.special.erfc(-z * 0.5 ** 0.5)).expand(-1, 8)  # (1 + erf cancels on the far negative side)
    fin = want.isfinite()
    err = (got - want).abs()[fin]
    assert bool((err <= want[fin].abs() * (2 ** -8 + 2e-5) + 2.0 ** -126).all())
    assert torch.equal(got[~fin].nan_to_num(5.0, 1.0, -1.0), want[~fin].nan_to_num(5.0, 1.0, -1.0))


def test_operands_that_are_left_to_the_caller():
    x, w = _rand(1, 70, 64), _rand(64, 64)
    assert ops.block_linear(x.float(), [w], [None]) is None
    assert ops.block_linear(x, [w.float()], [None]) is None
    assert ops.block_linear(_rand(1, 70, 80), [_rand(64, 80)], [None]) is None        # reduction of no whole chunks
    assert ops.block_linear(x, [_rand(60, 64)], [None]) is None                        # columns of no whole pieces
    assert ops.block_linear(x, [_rand(64, 128)[:, ::2]], [None]) is None
    assert ops.block_linear(_rand(70 * 64 + 1)[1:].view(1, 70, 64), [w], [None]) is None  # rows off their 16 bytes
    assert ops.block_linear(x.cpu(), [w], [None]) is None


@pytest.mark.parametrize("model,windows,frames", [("whisper-base", 1, 3000), ("whisper-tiny", 3, 301), ("whisper-base", 2, 2)])
def test_fused_encoder_against_the_general_one(model, windows, frames, monkeypatch):
    from vllm_production_stack_amd.models.whisper import WHISPER_PRESETS, WhisperModel

    m = WhisperModel(WHISPER_PRESETS[model], BF, torch.device("cuda"))
    m.init_random(3)
    mel = torch.randn(windows, m.cfg.num_mel_bins, frames, device="cuda").tanh()
    assert m._fused_encoder(mel)
    got = m.encode(mel)
    ref = WhisperModel(m.cfg, torch.float32, torch.device("cuda"))
    ref.w = {k: v.float() for k, v in m.w.items()}
    want = ref.encode(mel.to(BF).float())
    monkeypatch.setattr(WhisperModel, "_fused_encoder", lambda self, mel: False)
    general = m.encode(mel)
    err, base = ((v.double() - want.double()).norm() / want.double().norm() for v in (got, general))
    assert got.shape == want.shape and err <= 1.2 * base + 1e-3, (err, base)  # fewer roundings to 16 bits than the general form


@pytest.mark.parametrize("b,t", [(1, 151), (2, 1), (3, 389), (1, 750)])
def test_heads_of_other_widths_on_the_general_path(b, t):
    """16 channels a head (no kernel has them): one window, one position, odd lengths."""
    from vllm_production_stack_amd.models import whisper

    q, k, v = (_rand(b, t, 64) for _ in range(3))
    got = whisper._attend(q, k, v, 4).double()
    qh, kh, vh = (x.double().cpu().view(b, t, 4, 16).transpose(1, 2) for x in (q, k, v))
    p = torch.softmax(qh @ kh.transpose(-1, -2) * 0.25, dim=-1)
    want, size = ((p @ x).transpose(1, 2).reshape(b, t, 64).cuda() for x in (vh, vh.abs()))
    # scores (up to about 6), probabilities and the result are rounded to 16 bits once each
    assert bool(((got - want).abs() <= (2 ** -9 + 6 * 2 ** -8) * size + want.abs() * 2 ** -8).all())
