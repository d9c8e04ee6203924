"""Decode steps whose integers follow from the last step's (ops.step_advance) against steps that upload them all."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_advanced_steps_are_uploaded_steps(model_folders, dtype, monkeypatch):
    """Tokens from the device, many steps on end: over a page's edge, on a graph wider than the batch, in changed order, after
    another prompt step, after a step with tokens from the host, in a slot that is used again with the same length.  Which steps
    advance is asserted: those on the same graph, of the same sequences in the same order, one token longer on the same pages."""
    import bitnet_c_amd as bn
    from bitnet_c_amd import ops
    outs, advanced, now = [], [], [None]
    advance = ops.step_advance
    monkeypatch.setattr(ops, "step_advance", lambda *args: (advanced.append(now[0]), advance(*args))[1])
    for on_device in (False, True):
        eng = bn.Engine.from_folder(model_folders("B", dtype), dtype=dtype, max_tokens=4096)
        slots = [eng.new_sequence() for _ in range(3)]
        eng.step([bn.StepEntry(s, [(7 * i + s) % 389 for i in range(n)], []) for s, n in zip(slots, (60, 3, 126))])
        got = []

        def run(sl, k):
            now[0] = k
            toks = [(11 * k + 5 * i) % 389 for i in range(len(sl))]
            if on_device:
                dev = torch.tensor(toks, dtype=torch.int32, device="cuda")
                got.append(eng.step([bn.StepEntry(s, [0], [0]) for s in sl], device_tokens=dev))
            else:
                got.append(eng.step([bn.StepEntry(s, [t], [0]) for s, t in zip(sl, toks)]))

        for k in range(10):
            run(slots, k)
        run(slots[::-1], 10)                              # the same sequences in another order
        run(slots, 11)
        got.append(eng.step([bn.StepEntry(slots[1], [9, 8, 7], [2])]))      # one grows by a prompt step: the others did not
        run(slots, 12)
        run(slots, 13)
        got.append(eng.step([bn.StepEntry(s, [3], [0]) for s in slots]))    # from the host
        run(slots, 14)
        run(slots[:2], 15)
        n = eng.length(slots[0])
        eng.release(slots[0])                             # the slot again, at the length that the graph's integers expect
        again = eng.new_sequence()
        got.append(eng.step([bn.StepEntry(again, [(3 * i) % 389 for i in range(n)], [n - 1])]))
        for k in range(16, 19):
            run([again, slots[1]], k)
        eng.cache.check()
        outs.append(got)
    for i, (a, b) in enumerate(zip(*outs)):
        assert torch.equal(a, b), i
    # not: 0, 10, 11, 12, 15 (another step before them), 2 and 4 (a new page), 16 (the slot's new pages)
    assert advanced == [1, 3, 5, 6, 7, 8, 9, 13, 14, 17, 18]


def test_step_advance_touches_the_sequences_alone():
    from bitnet_c_amd import ops
    for rows, n in ((1, 1), (4, 3), (256, 256), (48, 33)):
        step = torch.arange(7 * rows + 1, dtype=torch.int32)
        toks = 1000 + torch.arange(n, dtype=torch.int32)
        want = step.clone()
        want[:n] = toks
        want[rows:rows + n] += 1
        want[3 * rows:3 * rows + n] += 1
        want[7 * rows] += 1
        dev = step.cuda()
        ops.step_advance(dev, rows, toks.cuda())
        assert torch.equal(dev.cpu(), want)
    with pytest.raises(ops.KernelError):
        ops.step_advance(torch.zeros(7, dtype=torch.int32, device="cuda"), 1, torch.zeros(1, dtype=torch.int32, device="cuda"))
