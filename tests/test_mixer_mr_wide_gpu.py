"""The one-kernel backward of the Hyena-MR mixer in fp32 arithmetic on bf16 tensors, which takes over from the
operator's backward and the featurizer's in sequence at 1024 steps of 32 rows (columns of 64 channels times batch rows
times steps): against that chain at the edges of its steps, channel blocks, taps and runs."""
import pytest
import torch

from savanna_amd import _lib
from test_mixer_mr_gpu import DEV, chain, make

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32


def one_kernel(bs, L, g, dg, hl, kf):
    return _lib.load().gcg_mixer_mr_bwd_scratch_bytes(bs, L, g, dg, hl, kf, _lib.GCG_BF16_F32) == 0


def run(raw, wf, h, dy):
    return _lib.mixer_mr_bwd(*(t.to(DEV) for t in (dy, raw, wf, h)))


def check(got, raw, wf, h, dy):
    """d raw as the chain's, bit for bit.  d wf against its 64-bit sum: one rounding to bf16 (8 significant bits: at most
    2^-8 of the value) and fp32 sums of n terms, sqrt(n) 2^-24 of the terms' norm with a factor of 8.  dh is a sum of
    the chain's terms in another order."""
    raw, wf, h, dy = (t.to(DEV) for t in (raw, wf, h, dy))
    bs, L, g, dg, _ = raw.shape
    _, draw, dwf, dh = chain(raw, wf, h, dy)
    assert torch.equal(got[0], draw)
    f = _lib.dwconv_fwd(raw.reshape(bs, L, 3 * g * dg, 1), wf)
    dfeat, _ = _lib.bwd_interleaved(dy, f.reshape(raw.shape), h)
    df, r = dfeat.double().reshape(bs, L, -1), raw.double().reshape(bs, L, -1)
    kf = wf.shape[-1]
    for k in range(kf):
        back = kf - 1 - k
        terms = df[:, back:] * r[:, :max(L - back, 0)]
        exact, norm = terms.sum((0, 1)), terms.square().sum((0, 1)).sqrt()
        err = (got[1][:, 0, k].double() - exact).abs()
        slack = 8 * (bs * L) ** 0.5 * 2.0 ** -24 * norm + 1e-30
        assert (err <= 2.0 ** -8 * exact.abs() + slack).all(), (k, (err / (2.0 ** -8 * exact.abs() + slack)).max().item())
    scale = dh.double().abs().max()
    assert (got[2].double() - dh.double()).abs().max() <= 1e-5 * scale


@pytest.mark.parametrize("bs,L,g,dg,hl,kf", [
    (1, 1024 * 32, 4, 16, 128, 3),      # the smallest: one column of 1024 steps
    (1, 1023 * 32 + 1, 4, 16, 128, 3),  # its last step holds one row
    (2, 511 * 32 + 31, 3, 16, 128, 3),  # 31 rows, a partial channel block
    (1, 8190, 16, 16, 128, 3),          # 30 rows: the last two rows of d raw are the run's own
    (512, 33, 5, 16, 33, 3),            # two channel blocks, runs of two steps
    (1024, 1, 4, 16, 1 + 8, 2),         # one row
    (1024, 2, 2, 16, 9, 3),
    (1024, 32, 1, 16, 9, 1),            # one tap
    (3, 5003, 20, 16, 128, 2),          # runs of several lengths, a batch that does not divide the chip
    (1, 4096, 11, 48, 128, 3),          # groups that no channel block holds whole: sums in second launches
    (1, 8192, 4, 64, 97, 3),
    (2, 3000, 3, 128, 64, 3),           # groups wider than a channel block
])
def test_against_chain(gcg_lib, bs, L, g, dg, hl, kf):
    assert one_kernel(bs, L, g, dg, hl, kf)
    args = make(bs, L, g, dg, hl, kf, BF, F32, seed=3)
    check(run(*args), *args)


@pytest.mark.parametrize("L,g", [(16236, 256), (3948, 256), (16236, 512)])
def test_chains_of_the_featurizer_gradient(gcg_lib, L, g):
    """d wf of two halves of a sequence that take each other off: dy of the second is the first's with its sign turned,
    and zero at the ends, so what is left of the sum is small and the error of its fp32 additions shows beside the
    rounding to bf16.  (The halves are no multiple of a lane's rows, or the errors would take each other off as well.)
    An addition rounded to nearest is off by 0.4 2^-24 of its result (rms over the mantissas), so a chain of m additions of
    random sign is off by 0.4 2^-24 sqrt(m / 2) of the 2-norm of its terms; the bar is that of chains of 64 rows, and of 16
    terms in the sums above them.  Chains of a run's rows, 512 and 1024 at the first and the last shape, are beyond it."""
    gen = torch.Generator(device=DEV).manual_seed(7)
    half, dg, d = L // 2, 16, 16 * g
    raw = torch.randn(1, half, g, dg, 3, generator=gen, device=DEV).to(BF).repeat(1, 2, 1, 1, 1)
    dy = torch.randn(1, half, g, dg, generator=gen, device=DEV).to(BF)
    dy[:, :256] = 0
    dy[:, -256:] = 0
    dy = torch.cat([dy, -dy], dim=1)
    wf = (torch.randn(3 * d, 1, 3, generator=gen, device=DEV) / 2).to(BF)
    h = torch.randn(g, 1, 128, generator=gen, device=DEV) / 11
    assert one_kernel(1, L, g, dg, 128, 3)
    got = _lib.mixer_mr_bwd(dy, raw, wf, h)[1][:, 0].double()
    f = _lib.dwconv_fwd(raw.reshape(1, L, 3 * d, 1), wf)
    df, r = _lib.bwd_interleaved(dy, f.reshape(raw.shape), h)[0].reshape(L, 3 * d), raw.reshape(L, 3 * d)
    err = terms2 = 0.
    for lo in range(0, 3 * d, 2048):
        for k in range(3):
            terms = df[2 - k:, lo:lo + 2048].double() * r[:L - 2 + k, lo:lo + 2048].double()
            exact = terms.sum(0)
            err += (got[lo:lo + 2048, k] - exact).square().sum().item() - (2.0 ** -9 * exact).square().sum().item() / 3
            terms2 += terms.square().sum().item()
    assert err <= terms2 * (0.4 * 2.0 ** -24) ** 2 * (64 + 16) / 2


@pytest.mark.parametrize("bs,L,g,dg,hl,lc,kf", [
    (2, 4097, 16, 16, 128, 128, 3),
    (1, 8190, 11, 48, 100, 128, 3),     # sums in second launches; a cut filter
    (600, 40, 3, 32, 40, 64, 2),        # runs of two steps, the filter as long as the sequence
    (1, 16384, 16, 16, 9, 128, 1),
])
def test_decayed_filter(gcg_lib, bs, L, g, dg, hl, lc, kf):
    """The filter formed in the kernel, as the module has it: the bits of the explicit filter's, and dw those of its dh."""
    assert one_kernel(bs, L, g, dg, hl, kf)
    raw, wf, _, dy = (t.to(DEV) for t in make(bs, L, g, dg, hl, kf, BF, F32, seed=6))
    w = torch.randn(g, lc, generator=torch.Generator().manual_seed(6)).to(DEV)
    decay = torch.exp(-torch.logspace(0, 2, g)[:, None] * torch.linspace(0, 1, lc)[None]).to(DEV)
    draw, dwf, dw = _lib.mixer_mr_bwd_decay(dy, raw, wf, w, decay, hl, F32)
    want = _lib.mixer_mr_bwd(dy, raw, wf, _lib.filter_decay_fwd(w, decay, hl, F32))
    assert torch.equal(draw, want[0]) and torch.equal(dwf, want[1])
    assert torch.equal(dw, _lib.filter_decay_bwd(want[2], decay))


def test_where_it_starts(gcg_lib):
    assert not one_kernel(1, 1023 * 32, 4, 16, 128, 3) and one_kernel(1, 1023 * 32 + 1, 4, 16, 128, 3)
    lib = _lib.load()
    for code, size in ((_lib.GCG_F32, 4), (_lib.GCG_F16_F32, 2)):        # these keep the chain
        assert lib.gcg_mixer_mr_bwd_scratch_bytes(4, 8192, 16, 16, 128, 3, code) == 3 * 4 * 8192 * 256 * size


@pytest.mark.parametrize("L", [8192 - 5, 8192])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), -3.3e38])
def test_values_without_a_finite_product(gcg_lib, value, L):
    """d raw is finite where the gradient rows it needs are -- its own and the two after it, of the chain's gradient of
    the features, rows past the sequence not among them -- and then equal to the chain's.  (The chain itself may add
    a fourth row times a tap of zero.)"""
    raw, wf, h, dy = (t.to(DEV) for t in make(1, L, 16, 16, 100, 3, BF, F32, seed=4))
    for t in (5, 4000, L - 1):
        raw[0, t, t % 16, 3] = value
    got = run(raw, wf, h, dy)[0]
    f = _lib.dwconv_fwd(raw.reshape(1, L, -1, 1), wf).reshape(raw.shape)
    lost = ~_lib.bwd_interleaved(dy, f, h)[0].isfinite()
    reach = lost.clone()
    reach[:, :-1] |= lost[:, 1:]
    reach[:, :-2] |= lost[:, 2:]
    assert reach.any() and not got[reach].isfinite().any()
    assert not got[~reach].isnan().any()
    want = chain(raw, wf, h, dy)[1]
    same = ~(reach | want.isnan())
    assert torch.equal(got[same], want[same])


def test_graph_replays_match_eager(gcg_lib):
    raw, wf, h, dy = (t.to(DEV) for t in make(2, 8192, 8, 16, 128, 3, BF, F32, seed=5))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        _lib.mixer_mr_bwd(dy, raw, wf, h)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = _lib.mixer_mr_bwd(dy, raw, wf, h)
    for it in range(3):
        raw.normal_()
        dy.normal_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(recorded, _lib.mixer_mr_bwd(dy, raw, wf, h)):
            assert torch.equal(a, b), it
