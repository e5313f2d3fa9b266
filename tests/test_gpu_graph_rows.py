"""Recorded decode steps of three quarters of a bucket's rows: which requests take them, and a batch that shrinks and grows across the line between
the two, step after step against the step in one that is recorded for its size alone."""
import pytest
import torch

from sprout_lm_amd.engine.graphs import sequence_rows


def test_rows():
    assert [sequence_rows(n) for n in (1, 3, 24, 32, 33, 48, 49, 64, 65, 96, 97, 129, 192, 193, 257, 600)] == \
        [1, 4, 32, 32, 48, 48, 64, 64, 96, 96, 128, 192, 192, 256, 512, 1024]


@pytest.mark.gpu
def test_a_batch_crosses_the_line():
    import sprout_lm_amd as S
    from sprout_lm_amd.cli import preset_config
    from sprout_lm_amd.engine import ModelRunner, StepEntry
    from sprout_lm_amd.engine.graphs import DecodeGraphs
    from sprout_lm_amd.sampling.params import SamplingParams
    from sprout_lm_amd.weights.random_init import random_tensors
    config = preset_config("tiny-b")
    plan = S.build_model_plan(config)
    weights = random_tensors(plan.expected_tensors(), 3, dtype=torch.float32, device=torch.device("cuda", 0))
    greedy = SamplingParams(temperature=0.0, ignore_eos=True)

    def generate(sizes, **kw):
        """Tokens of every request, of which sizes[i] take part in step i."""
        runner = ModelRunner(plan, dict(weights), torch.float32, torch.device("cuda", 0), block_size=8, num_blocks=400, max_sequences=64)
        runner._graphs = DecodeGraphs(runner, **kw)
        seqs = [runner.cache.create() for _ in range(max(sizes))]
        rows = [[(7 * i + 3) % 90] for i in range(len(seqs))]
        for n in sizes:
            entries = []
            for i in range(n):
                assert runner.cache.reserve(seqs[i], seqs[i].length + 1)
                entries.append(StepEntry(seqs[i], rows[i][-1:], [0]))
            for row, token in zip(rows, runner._graphs.run(entries, [greedy] * n, [0] * n)):
                row.append(token)
        return rows, runner._graphs

    sizes = [50, 47, 47, 49, 48, 33, 64, 20, 48, 60, 47]
    got, graphs = generate(sizes)
    assert sorted(graphs.graphs) == [(32, 256), (64, 256)]
    pair = graphs.graphs[(64, 256)]
    assert sorted((pair.S, pair.other.S)) == [48, 64] and pair.other.other is None
    # the same with room for a single graph: recorded anew at every change
    assert generate(sizes, max_graphs=1)[0] == got
    # a request's tokens do not depend on who runs beside it
    few, many = generate([40] * 10)[0], generate([64] * 10)[0]
    assert few == many[:40]


class Recorder:
    """Requests of a small model that are answered through `DecodeGraphs`; a step that brings new requests before or after others reads the tokens of
    the step before on the device."""

    def __init__(self, requests, **kw):
        import sprout_lm_amd as S
        from sprout_lm_amd.cli import preset_config
        from sprout_lm_amd.engine import ModelRunner
        from sprout_lm_amd.engine.graphs import DecodeGraphs
        from sprout_lm_amd.sampling.params import SamplingParams
        from sprout_lm_amd.weights.random_init import random_tensors
        device = torch.device("cuda", 0)
        plan = S.build_model_plan(preset_config("tiny-b"))
        self.runner = ModelRunner(plan, random_tensors(plan.expected_tensors(), 3, dtype=torch.float32, device=device), torch.float32, device,
                                  block_size=8, num_blocks=400, max_sequences=64)
        self.graphs = self.runner._graphs = DecodeGraphs(self.runner, **kw)
        self.greedy = SamplingParams(temperature=0.0, ignore_eos=True)
        self.seqs = [self.runner.cache.create() for _ in range(requests)]
        self.rows = [[(7 * i + 3) % 90] for i in range(requests)]

    def launch(self, n, pending=None):
        """A step of the first n requests; those of `pending` have not been read."""
        from sprout_lm_amd.engine import StepEntry
        ahead = 0 if pending is None else min(n, pending.n)
        for seq in self.seqs[:n]:
            assert self.runner.cache.reserve(seq, seq.length + 1)
        entries = [StepEntry(self.seqs[i], [None if i < ahead else self.rows[i][-1]], [0]) for i in range(n)]
        feed = None if pending is None else (pending, [i if i < ahead else -1 for i in range(n)])
        return self.graphs.launch(entries, [self.greedy] * n, [0] * n, feed)

    def read(self, pending):
        for row, token in zip(self.rows, pending.result()):
            row.append(token)


@pytest.mark.gpu
def test_a_step_launched_ahead_across_the_line():
    """The tokens of a step that is not read yet go into one that runs as the bucket's other number of rows, and back."""
    sizes = [50, 47, 49, 50, 33, 64, 40, 48, 60, 47, 47, 64]
    plain, ahead = Recorder(64), Recorder(64)
    pending = None
    for n in sizes:
        plain.read(plain.launch(n))
        following = ahead.launch(n, pending)
        if pending is not None:
            ahead.read(pending)
        pending = following
    ahead.read(pending)
    assert ahead.rows == plain.rows and ahead.graphs.recorded == 2


@pytest.mark.gpu
def test_room_is_made_a_step_at_a_time():
    """The bucket used longest ago gives up one of its two steps where one place is wanted, that used longer ago, then the other."""
    r = Recorder(64, max_graphs=3)
    kept = lambda: [(key[0], g.S, g.other and g.other.S) for key, g in r.graphs.graphs.items()]
    for n in (64, 47, 20):
        r.read(r.launch(n))
    assert kept() == [(64, 48, 64), (32, 32, None)] and r.graphs.recorded == 3
    r.read(r.launch(5))
    assert kept() == [(64, 48, None), (32, 32, None), (8, 8, None)]
    r.read(r.launch(2))
    assert kept() == [(32, 32, None), (8, 8, None), (2, 2, None)]
    r.read(r.launch(50))
    r.read(r.launch(40))      # a step of its bucket's other rows: what is in front stays
    assert kept() == [(2, 2, None), (64, 48, 64)] and r.graphs.recorded == 3
    few = Recorder(64, max_graphs=1)
    for n in (64, 47, 20, 50):
        few.read(few.launch(n))
        assert few.graphs.recorded == 1
    full = Recorder(64)
    for n in (64, 47, 20, 50):
        full.read(full.launch(n))
    assert few.rows == full.rows and full.graphs.recorded == 3
