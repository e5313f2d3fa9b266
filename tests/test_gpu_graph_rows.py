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
