"""Decode calls: a refused draft count, and calls one after another on one
model, where each takes its own sampler, whatever rounds an earlier call left
captured."""
import pytest

pytestmark = pytest.mark.gpu

CFG = dict(n_layers=2, hidden=256, n_heads=4, n_kv=2, head_dim=128, inter=512, vocab=4096, max_seq=256, rope_theta=1e6,
           eps=1e-6)


@pytest.fixture(scope="module")
def calls(gpu):
    from cmf_amd import synth
    return synth.synth_model(CFG, seed=5, norm_noise=0.1, sigma=0.05), synth.ids(19, 20, CFG["vocab"])


def _decode(m, prompt, *args, **kw):
    m.prefill(prompt)
    return m.decode(*args, **kw)[0].tolist()


# (auto: five speculative rounds, then the last token, whatever the monitor measures)
@pytest.mark.parametrize("spec,n,k", [(False, 16, 4), (True, 24, 3), ("auto", 6, 1)])
def test_each_call_uses_its_sampler(gpu, calls, spec, n, k):
    from cmf_amd import SamplerConfig
    from cmf_amd.model import Model
    sm, prompt = calls
    samplers = [SamplerConfig(0.8, 0.9, 1, 1.0, 0.05), SamplerConfig(1.5, 1.0, 64, 1.0, 0.0), SamplerConfig(0.3, 0.1, 40, 1.0, 0.0)]
    fresh = []
    for s in samplers:
        m = Model(sm)
        fresh.append(_decode(m, prompt, n, sampler=s, seed=77, spec=spec, k=k))
        m.free()
    assert len({tuple(f) for f in fresh}) == len(fresh)
    m = Model(sm)
    for s, want in list(zip(samplers, fresh)) + [(samplers[0], fresh[0])]:
        if spec == "auto":  # (rounds under the monitor replay what a decode of several rounds has captured)
            _decode(m, prompt, 24, sampler=samplers[0], seed=3, spec=True, k=k)
        assert _decode(m, prompt, n, sampler=s, seed=77, spec=spec, k=k) == want
    m.free()


@pytest.mark.parametrize("k", [-1, 0, 9])
def test_bad_draft_count_is_refused(gpu, calls, k):
    from cmf_amd import CmfError
    from cmf_amd.model import Model
    sm, prompt = calls
    m = Model(sm)
    m.prefill(prompt)
    for spec in (True, "auto"):
        with pytest.raises(CmfError, match="k must be 1..8"):
            m.decode(12, spec=spec, k=k)
    assert len(m.decode(12, spec=False, k=k)[0]) == 12  # (plain steps take no drafts)
    m.free()


def test_expert_of_another_codec_after_a_decode(gpu):
    """the one expert of a routed layer, set again in another codec between
    two decodes: the second runs its kernels, not those captured before"""
    import ctypes as C

    from cmf_amd import DT_Q4T, DT_Q8ROW, check, lib, synth
    from cmf_amd.model import Model, _tensor
    moe = dict(n_experts=1, top_k=1, inter=128, layers=[0, 1], router_dtype="q8")
    sms = [synth.synth_model(CFG, seed=31, norm_noise=0.3, sigma=0.08, mtp=False, moe=moe, ffn_dtype=dt) for dt in (DT_Q8ROW, DT_Q4T)]
    prompt = synth.ids(34, 12, CFG["vocab"])
    want = []
    for sm in sms:
        m = Model(sm)
        want.append(_decode(m, prompt, 16, spec=False))
        m.free()
    m = Model(sms[0])
    assert _decode(m, prompt, 16, spec=False) == want[0]
    for layer, li in zip(m.moes, (0, 1)):
        ex, keep = sms[1]["layers"][li]["moe"]["experts"][0], []
        check(lib().cmf_moe_set_expert(layer.h, 0, *(C.byref(_tensor(ex[n], keep)) for n in ("gate", "up", "down"))))
    assert _decode(m, prompt, 16, spec=False) == want[1]
    m.free()


@pytest.mark.parametrize("spec,first", [(False, 470), (True, 470), (True, 506)])
def test_decodes_across_position_steps(gpu, spec, first, monkeypatch):
    """decodes that cross a 512-position step, one after another at shrinking
    and growing contexts, replay captured rounds of their own size: the tokens
    of a model that launches every round eagerly"""
    from cmf_amd import synth
    from cmf_amd.model import Model
    cfg = dict(CFG, max_seq=2400)
    sm = synth.synth_model(cfg, seed=5, norm_noise=0.1, sigma=0.05)
    monkeypatch.setenv("CMF_DECODE_GRAPH", "0")
    eager = Model(sm)
    monkeypatch.delenv("CMF_DECODE_GRAPH")
    m = Model(sm)
    ids = synth.ids(35, 1700, cfg["vocab"])
    for ctx, n in ((first, 60), (1700, 20), (30, 24), (500, 40)):
        assert _decode(m, ids[:ctx], n, spec=spec, k=4) == _decode(eager, ids[:ctx], n, spec=spec, k=4)
    m.free()
    eager.free()
