"""GPU parity of the sampler over full logits with a workspace (the groups' maxima first, then one workgroup over the
groups that can hold a survivor) with the same draw without one (one workgroup over every logit): ids and generator
state equal, at group and workgroup edges, the largest top-k, a history that reorders groups, equal logits, -inf, and
more candidates above the bound than the pool holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["normal", "ties", "ramp", "inf"])
@pytest.mark.parametrize("n", [8191, 8192, 8193, 33000, 151936, 262144])
def test_group_filter_equals_single_workgroup(qh, gpu, n, kind):
    import torch
    g = np.random.default_rng(n)
    x = (g.standard_normal(n) * 3).astype(np.float32)
    if kind == "ties":
        x = np.round(x)
    elif kind == "ramp":  # the largest keys fill whole groups: the pool overflows at the larger top-k
        x = np.sort(x)
    elif kind == "inf":
        x[g.random(n) < 0.9] = -np.inf
    logits = torch.from_numpy(x).to(gpu)
    ws = qh.sample_workspace(n)
    hist = torch.from_numpy(np.concatenate([np.argsort(x)[-40:], g.integers(0, n, 300)]).astype(np.int32)).to(gpu)
    for k, temp, pen, h in ((1, 0.7, 1.1, hist), (20, 0.7, 1.1, hist), (16, 1.3, 1.0, None), (256, 1.5, 1.3, hist),
                            (20, 0.0, 1.2, hist)):
        got = []
        for w in (None, ws):
            state = torch.full((1,), qh.sampler_state(77), dtype=torch.int64, device=gpu)
            p = qh.sampler_params(temperature=temp, top_k=k, top_p=0.95, repeat_penalty=pen)
            ids = [int(qh.sample(logits, p, state, history=h, ws=w)[0]) for _ in range(3)]
            got.append((ids, int(state[0])))
        assert got[0] == got[1], (k, temp, pen)
