"""The native binding of the hot entry points against the descriptors built in
Python: a call with its stream named takes the Python path, one without (output
and workspace given) the native one. Same kernels, so equal bytes; and what the
wrapper refuses is refused with the same exception."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
H, HKV, D, RB = 16, 2, 256, 144


def cache(gen, rows, dev):
    c = torch.randint(0, 256, (rows, HKV, 8, 18), generator=gen, device=dev, dtype=torch.uint8)
    c[..., :2] = torch.tensor([0.05], dtype=torch.float16).view(torch.uint8).to(dev)
    return c.view(rows, HKV, RB)


@pytest.fixture
def gen(dev):
    g = torch.Generator(device=dev)
    g.manual_seed(3)
    return g


class Watch:
    """The native binding, with a record of its answers (None: left to Python)."""

    def __init__(self, host):
        self.host, self.answers = host, []

    def __getattr__(self, name):
        def call(*args):
            self.answers.append(getattr(self.host, name)(*args))
            return self.answers[-1]
        return call


@pytest.fixture(autouse=True)
def watch(sqa, monkeypatch):
    w = Watch(sqa._host or sqa._load_host())
    monkeypatch.setattr(sqa, "_host", w)
    return w


def both(call, state, watch):
    """Equal bytes from the native call, which has to answer, and from the Python one."""
    got = []
    for kw in ({}, {"stream": torch.cuda.current_stream()}):
        s = {k: v.clone() for k, v in state.items()}
        watch.answers.clear()
        call(s, **kw)
        assert watch.answers == ([] if kw else [0])
        got.append([v.cpu().numpy().tobytes() for v in s.values()])
    assert got[0] == got[1]


@pytest.mark.parametrize("n_q,strided,masked", [(1, False, True), (1, True, False), (3, True, True), (40, True, True)])
def test_attention_calls(sqa, dev, gen, watch, n_q, strided, masked):
    n_kv = 768
    kc, vc = cache(gen, 1024, dev), cache(gen, 1024, dev)
    wide = torch.randn((n_q, 2 * H, D + 16), generator=gen, device=dev)
    q = wide[:, ::2, :D] if strided else wide[:, :H, :D].contiguous()
    gate = wide[:, 1::2, 3:D + 3] if strided else None
    mask = torch.zeros((n_q, 2 * n_kv), dtype=torch.float16, device=dev)[:, :n_kv] if masked else None
    if masked:
        both(lambda s, **kw: sqa.fill_causal_mask(s["mask"][:, :n_kv], 700, **kw),
             {"mask": torch.zeros((n_q, 2 * n_kv), dtype=torch.float16, device=dev)}, watch)
        sqa.fill_causal_mask(mask, 700)
    ws = torch.empty(sqa.flash_attn_workspace_size(q, kc, n_kv), dtype=torch.uint8, device=dev)
    out = {"out": torch.zeros((n_q, H, D), device=dev)}
    for scale in (None, 0.05):
        both(lambda s, **kw: sqa.flash_attn_ext(q, kc, vc, n_kv, mask=mask, scale=scale, out=s["out"], workspace=ws, **kw), out, watch)
        both(lambda s, **kw: sqa.flash_attn_ext_causal(q, kc, vc, n_kv, 700, gate=gate, scale=scale, out=s["out"],
                                                       workspace=ws, **kw), out, watch)


@pytest.mark.parametrize("n,strided", [(1, False), (5, True)])
def test_producer_cache_and_projection_calls(sqa, dev, gen, watch, n, strided):
    wide = torch.randn((n, 2 * H, D), generator=gen, device=dev)
    src = wide[:, ::2] if strided else wide[:, :H].contiguous()
    w = torch.rand(D, generator=gen, device=dev)
    pos = torch.arange(4 * n, dtype=torch.int32, device=dev)
    rope = sqa.rope_params(64, (11, 11, 10, 0), 1e7)
    idx = torch.arange(2 * n, device=dev)[::2] if strided else torch.arange(n, device=dev)
    k = {"c": cache(gen, 64, dev)}
    for norm in (w, None):
        both(lambda s, **kw: sqa.rope_norm_f32(s["o"], src, norm, 1e-6, pos, rope, **kw),
             {"o": torch.zeros((n, H, D), device=dev)}, watch)
        both(lambda s, **kw: sqa.rope_norm_set_rows_q4_0(s["c"], src[:, :HKV], norm, 1e-6, pos, rope, idx, **kw), k, watch)
    both(lambda s, **kw: sqa.set_rows_q4_0(s["c"], src[:, 0].repeat(1, 2) if not strided else wide.view(n, -1)[:, 5:517],
                                           idx, **kw), k, watch)
    wq = torch.randint(0, 256, (64, 4, 144), generator=gen, device=dev, dtype=torch.uint8)
    wq[..., 1], wq[..., 3] = 0x10, 0x10  # finite fp16 d and dmin
    wq = wq.view(64, 576)[::2] if strided else wq.view(64, 576)
    x, gate = wide.view(n, -1)[:, :1024], wide.view(n, -1)[:, 1024:2048]
    ws = torch.empty(max(1, sqa.out_proj_workspace_size(wq, x)), dtype=torch.uint8, device=dev)
    for g in (gate, None):
        both(lambda s, **kw: sqa.out_proj(wq, x, gate=g, out=s["o"], workspace=ws, **kw),
             {"o": torch.zeros((n, wq.shape[0]), device=dev)}, watch)

    caches = []
    for kw in ({}, {"stream": torch.cuda.current_stream()}):
        kv = sqa.KvCache(2, D, HKV, 64)
        kv.zero_caches()
        kv.begin_step(n)
        rows = src[:, :HKV].reshape(n, -1).contiguous()
        watch.answers.clear()
        kv.append(1, rows, -rows, torch.arange(n, device=dev), **kw)
        assert watch.answers == ([] if kw else [0])
        caches.append([t.cpu().numpy() for t in kv.k + kv.v])
    assert all(np.array_equal(a, b) for a, b in zip(*caches)) and caches[0][1].any()


def test_refusals_are_the_wrappers(sqa, dev, gen, watch):
    kc = cache(gen, 256, dev)
    q = torch.randn((1, H, D), generator=gen, device=dev)
    out, ws = torch.empty_like(q), torch.empty(sqa.flash_attn_workspace_size(q, kc, 256), dtype=torch.uint8, device=dev)
    call = lambda q=q, kc=kc, n_kv=256, ws=ws, **kw: sqa.flash_attn_ext(q, kc, kc, n_kv, out=out, workspace=ws, **kw)
    assert call() is out
    for bad, exc in ((lambda: call(n_kv=257), AssertionError), (lambda: call(kc=kc.view(torch.int8)), AssertionError),
                     (lambda: call(kc=kc[:, :, :72]), AssertionError), (lambda: call(q=q[0]), ValueError),
                     (lambda: call(mask=torch.zeros((1, 256), device=dev)), AssertionError),
                     (lambda: call(max_bias=1), sqa.SqaError), (lambda: call(max_bias=1.0), sqa.SqaError),
                     (lambda: call(ws=ws[:100]), sqa.SqaError), (lambda: call(scale=float("nan")), sqa.SqaError),
                     (lambda: sqa.flash_attn_ext_causal(q, kc, kc, 256, -1, out=out, workspace=ws), sqa.SqaError),
                     (lambda: sqa.set_rows_q4_0(kc, q[0], torch.zeros(16, dtype=torch.int64, device=dev)), AssertionError),
                     (lambda: sqa.rope_norm_f32(out, q, None, 1e-6, torch.zeros(3, dtype=torch.int32, device=dev),
                                                sqa.rope_params(64, (11, 11, 10, 0), 1e7)), sqa.SqaError)):
        watch.answers.clear()
        with pytest.raises(exc):
            bad()
        assert len(watch.answers) == 1 and watch.answers[0] != 0
        assert exc is sqa.SqaError or watch.answers[0] is None


def test_rope_of_another_type_is_refused(sqa, dev):
    src = torch.randn((1, 2, D), device=dev)
    pos = torch.zeros(4, dtype=torch.int32, device=dev)
    idx = torch.zeros(1, dtype=torch.int64, device=dev)
    raw = bytes(sqa.rope_params(64, (11, 11, 10, 0), 1e7))  # the right bytes in the wrong object
    with pytest.raises(TypeError):
        sqa.rope_norm_f32(torch.empty_like(src), src, None, 1e-6, pos, raw)
    with pytest.raises(TypeError):
        sqa.rope_norm_set_rows_q4_0(torch.zeros((4, 2, RB), dtype=torch.uint8, device=dev), src, None, 1e-6, pos, raw, idx)


def test_calls_run_on_the_current_stream(sqa, dev, gen, watch):
    """The native path and the Python one look the stream up by different routes: a
    call inside torch.cuda.stream() has to wait for that stream's work."""
    side = torch.cuda.Stream()
    big, idx = torch.ones(1 << 26, device=dev), torch.arange(4, device=dev)
    for n in (1, 2):  # the second time every kernel is loaded
        src = torch.zeros((4, 512), device=dev)
        want = torch.zeros((8, HKV, RB), dtype=torch.uint8, device=dev)
        sqa.set_rows_q4_0(want, src + n, idx)
        got = torch.zeros_like(want)
        torch.cuda.synchronize()
        watch.answers.clear()
        with torch.cuda.stream(side):
            for _ in range(40):
                big.mul_(1.0)
            src.fill_(n)
            sqa.set_rows_q4_0(got, src, idx)
        side.synchronize()
        assert watch.answers == [0] and torch.equal(got, want)
