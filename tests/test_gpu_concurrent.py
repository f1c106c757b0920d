"""Handles are independent: two optimizer handles bound to two streams,
stepped in an interleaved order with no host wait between them (so their
kernels may overlap on the device), each give exactly the oracle's result
for their own problem.  Also a codec plan and a gradient plan running on a
third stream meanwhile."""
import pytest

import oracle
from oracle import harness as H
from ark_amd.eko import EkoConfig

pytestmark = pytest.mark.gpu


def test_two_handles_on_two_streams():
    import torch
    assert torch.cuda.is_available(), "GPU test run without a GPU"
    from ark_amd import codec, grad
    from ark_amd.optimizer import AdamConfig, AmpConfig, Optimizer
    cfg = AdamConfig(lr=3e-4, beta1=0.9, beta2=0.95, eps=1e-8, weight_decay=0.1, grad_clip=1.0)
    amp = AmpConfig(loss_scale_init=1024.0, loss_scale_max=2.0 ** 24, scale_up_every=2)
    specs = [EkoConfig(n_layers=2, d_model=64, hidden=96, vocab=500).tensors(),
             EkoConfig(n_layers=1, d_model=128, hidden=256, vocab=777).tensors()]
    seeds = [31, 32]
    sig = [[1e-3] * len(s) for s in specs]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    ps, opts, ts, refs = [], [], [], []
    for i in range(2):
        with torch.cuda.stream(streams[i]):
            p = H.gpu_problem(specs[i], seeds[i], cfg.weight_decay, sig[i], 1024.0)
            ps.append(p)
            opts.append(Optimizer(cfg, p, amp))
        t = H.host_problem(specs[i], seeds[i], cfg.weight_decay, sig[i], 1024.0)
        ts.append(t)
        refs.append(oracle.Optimizer(t, opts[i].hp))
    torch.cuda.synchronize()
    # a third stream keeps the device busy with other library work meanwhile
    s3 = torch.cuda.Stream()
    with torch.cuda.stream(s3):
        a16 = torch.randn(1 << 20, device="cuda").half()
        a32 = torch.empty(1 << 20, device="cuda")
        dq = codec.CodecPlan([(a16, a32)], "f16_to_f32")
        x = torch.randn(1 << 20, device="cuda")
        y = torch.randn(1 << 20, device="cuda")
        gp = grad.GradPlan([(x, y)])
    torch.cuda.synchronize()
    for k in range(6):
        for i in (0, 1) if k % 2 else (1, 0):
            with torch.cuda.stream(streams[i]):
                if k:
                    H.gpu_regen_grads(ps[i], seeds[i], sig[i], 1024.0, k)
                opts[i].step_all(cfg.lr)
        with torch.cuda.stream(s3):
            dq.run()
            gp.run()
    torch.cuda.synchronize()
    for i in range(2):
        for k in range(6):
            if k:
                H.host_regen_grads(ts[i], seeds[i], sig[i], 1024.0, k)
            refs[i].step(cfg.lr)
        st = opts[i].get_state()
        assert st.t == refs[i].state.t and st.loss_scale == refs[i].state.loss_scale
        c = H.compare(ps[i], ts[i])
        assert c["w"] == c["m"] == c["v"] == 0, (i, c)
        opts[i].close()
    dq.close(), gp.close()


@pytest.mark.parametrize("source", ["f16", "f32", "units"])
def test_a_norm_pass_that_misses_partials_ends_and_the_next_step_is_whole(source, monkeypatch):
    """The norm pass's finalizer gives a step up after a bounded number of
    looks at the partials (a step of the same handle running at the same time
    may have taken them).  Forced from the host by allowing no second look
    while thousands of blocks are still reading: the step ends, reports the
    error and changes nothing, with and without info; the same handle's next
    steps are, bit for bit, those of a handle that lost none."""
    import torch
    from ark_amd import _abi, grad, synth
    from ark_amd._lib import ArkOptError
    from ark_amd.eko import TensorSpec
    from ark_amd.optimizer import AdamConfig, AmpConfig, Optimizer
    cfg = AdamConfig(lr=3e-4, beta1=0.9, beta2=0.95, eps=1e-8, weight_decay=0.1, grad_clip=1.0)
    amp = AmpConfig(loss_scale_init=1024.0)
    monkeypatch.setenv("ARK_OPT_SUMSQ_SPB", "1")  # 24,415 partials: 47 groups, a tail
    specs = [TensorSpec("a", (100_000_123,), True, False)]
    dt = _abi.GRAD_F16 if source == "f16" else _abi.GRAD_F32
    sets = [synth.problem(specs, 77, 0.1, [1e-3], 1024.0, grad_dtype=dt) for _ in range(2)]
    whole = Optimizer(cfg, sets[1], amp)
    monkeypatch.setenv("ARK_OPT_FIN_POLLS", "0")
    opt = Optimizer(cfg, sets[0], amp)
    plans = []
    if source == "units":
        zero = torch.zeros(specs[0].n, device="cuda")
        plans = [grad.GradPlan([(ps.g(0), zero)]) for ps in sets]

    def step(which, info):
        if plans:
            plans[which].run(final_for=(opt, whole)[which])
        return (opt, whole)[which].step_all(info=info)

    def same():
        return all(torch.equal(getattr(sets[0], k).view(torch.uint8), getattr(sets[1], k).view(torch.uint8))
                   for k in ("w_arena", "g_arena", "m_arena", "v_arena"))

    def state(o):
        return bytes(o.get_state())

    before = state(opt)
    for _ in range(2):
        with pytest.raises(ArkOptError, match="partial sum") as e:
            step(0, True)
        assert e.value.code == _abi.EHIP
        step(0, False)
        torch.cuda.synchronize()
        assert state(opt) == before
    assert same()
    monkeypatch.delenv("ARK_OPT_FIN_POLLS")
    for _ in range(2):
        _, a = step(0, True)
        _, b = step(1, True)
        assert a.applied == 1 and bytes(a) == bytes(b)
    assert same()
    for o in (opt, whole, *plans):
        o.close()
