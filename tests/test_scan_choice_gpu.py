"""Whole models with recurrences, at sizes at which prompt steps may cut them into pieces: a request gives float32 logits that
are equal bit for bit whether its step runs eagerly, is recorded or is replayed, alone or in a batch; and in bfloat16 the
three choose the same form of the recurrences."""
import pytest
import torch

from conftest import rel_err
from sunusun_cases import _par, _wkv, write_folder

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16]


def _config(heads, dim, width):
    return dict(architecture="Sunusun", vocab=61, width=64, norm=dict(eps=1e-5), logit_scale=0.5, layers=[
        _wkv(heads, dim, 8, ff=96), _par(4, 2, 32, 32, 0.2, 0.2, 64, width, ff=64), _wkv(heads, dim, 8)])


def _prompt(seed, n):
    return torch.randint(0, 61, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


def _step(eng, prompts, cuts=None):
    """Logits of every token of prompts that start together (one of them in portions of the sizes `cuts`)."""
    import bitnet_c_amd as bn
    slots = [eng.new_sequence() for _ in prompts]
    if cuts is None:
        out = eng.step([bn.StepEntry(s, p, range(len(p))) for s, p in zip(slots, prompts)])
    else:
        parts, at = [], 0
        for n in cuts:
            parts.append(eng.step([bn.StepEntry(slots[0], prompts[0][at:at + n], range(n))]))
            at += n
        assert at == len(prompts[0])
        out = torch.cat(parts)
    for s in slots:
        eng.release(s)
    return out


# 200 tokens of one sequence fill a captured step of 256 rows; three sequences of 32 heads one of four
@pytest.mark.parametrize("heads,dim,width,lens", [(2, 64, 96, [200]), (2, 64, 96, [300]), (2, 64, 96, [600]), (32, 8, 40, [70, 90, 96]),
                                                  (32, 8, 40, [8] * 32)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_eager_recorded_and_replayed(tmp_path, monkeypatch, heads, dim, width, lens, dtype):
    import bitnet_c_amd as bn
    from bitnet_c_amd import ops
    taken = []
    for name in ("wkv_scan", "mingru_scan"):
        plain = getattr(ops, name)
        monkeypatch.setattr(ops, name, lambda *a, _f=plain, **kw: (taken.append(kw.get("pieces")) if kw.get("tiles") is not None else None,
                                                                   _f(*a, **kw))[1])
    folder = write_folder(tmp_path / "m", _config(heads, dim, width), 4, dtype)
    wants = 1 + sum(lens) // 257                 # a captured step holds 256 wanted rows: the logits come in as many calls
    eng = bn.Engine.from_folder(folder, dtype=dtype, max_tokens=2 * sum(lens) + 64 * len(lens) + 64, max_slots=len(lens) + 1)
    prompts = [_prompt(i, n) for i, n in enumerate(lens)]

    def request():
        out = []
        for w in range(wants):
            slots = [eng.new_sequence() for _ in prompts]
            out.append(eng.step([bn.StepEntry(s, p, range(w, len(p), wants)) for s, p in zip(slots, prompts)]))
            for s in slots:
                eng.release(s)
        return torch.cat(out)

    first = request()
    forms, built = list(taken), eng.graphs_built
    second, third = request(), request()
    assert eng.graphs_built > built or wants > 1
    assert taken == forms * (len(taken) // len(forms)) and any(taken) == (dtype == torch.bfloat16 and lens in ([200], [300], [600]))
    if dtype == torch.bfloat16:
        assert torch.equal(second, third) and rel_err(second, first) < 0.2
        return
    assert torch.equal(first, second) and torch.equal(first, third)
    if wants == 1:
        alone = torch.cat([_step(eng, [p]) for p in prompts])
        assert torch.equal(alone, first)
    whole = _step(eng, prompts[:1])
    cuts = [2, 3, 64, lens[0] - 69] if lens[0] > 80 else [lens[0] - 2, 2] if lens[0] > 8 else [3, lens[0] - 3]
    assert torch.equal(_step(eng, prompts[:1], cuts), whole)


@pytest.mark.parametrize("heads,dim,width", [(2, 64, 96), (3, 24, 40), (5, 65, 33)])
@pytest.mark.parametrize("graphs", [True, False])
def test_float32_prompts_and_single_tokens_give_the_same_bits(tmp_path, heads, dim, width, graphs):
    import bitnet_c_amd as bn
    folder = write_folder(tmp_path / "m", _config(heads, dim, width), 7, torch.float32)
    eng = bn.Engine.from_folder(folder, dtype=torch.float32, max_tokens=512, use_graphs=graphs)
    prompt = [_prompt(3, 150)]
    whole = _step(eng, prompt)
    for cuts in ([1] * 40 + [110], [130] + [1] * 20, [64, 1, 1, 63, 1, 20]):
        assert torch.equal(_step(eng, prompt, cuts), whole)
